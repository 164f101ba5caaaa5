// race_capi.hip -- the extern "C" boundary declared in include/race_attention.h.
//
// Validates descriptors and pointers on the host (shape, alignment and stride
// checks happen before any launch, so a kernel never sees a shape it does not
// assume), plans the segment decomposition, carves the caller's workspace and
// enqueues the kernels on the caller's stream.  No allocation, no
// synchronisation, no global mutable state besides the thread-local error.
#include <stdarg.h>
#include <stdio.h>

#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>

#include "../../include/race_attention.h"
#include "prefix_mean.hip"
#include "race_kernels.hip"

namespace race {
namespace {

thread_local std::string g_err;

int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

int ok() {
    g_err.clear();
    return RACE_OK;
}

// Workgroups per forward phase of long sequences (256 CUs x 8: several rounds
// of whole segments even out), and the tiles per segment from which that many
// pay.  A segment costs its workgroup's set-up (state row, planes, the first
// tile's load: about 2 tiles' time) and 65 fp64 words a bucket of state written,
// scanned and read again (66 KB a pass at 128 buckets, 4 passes; a tile's rows
// are 24 KB), so shorter sequences run fewer, longer segments: as many
// workgroups as are resident at once (target_blocks).  K=4 L=8 bf16 16 x 16384
// tokens, us: 2048 workgroups of 4 tiles 418 (the scan alone 58), 512 of 16 296;
// 8 x 262001: 2048 of 32 tiles 2080, 512 of 128 1987; K=3 L=8 48 x 4001: 2016 of
// 3 280, 768 of 8 234; fp32 K=4 L=8 8 x 8192: 2048 of 1 433, 256 of 8 282.
constexpr int64_t kTargetBlocks = 2048;
constexpr int64_t kLongSegTiles = 64;
// Up to this many tiles (and slices) in all, segments stay one tile each: not for
// time (of 513 to 1024 tiles of 128 buckets short_tiles would join two), but
// because the state of an automatic forward is there also that of seg_tiles = 1,
// and backward calls with either are used with it.
constexpr int64_t kOneTileBlocks = 1024;
// Workgroups that a launch of the forward and of the backward tile kernels aims
// at, by slice size (8-, 4- and 2-wave workgroups; 256 CUs).  128 buckets: what is
// resident, two per CU in the bf16 forward, one in the backward and in fp32.  Fewer
// buckets: more than is resident where that measured the same or better -- the
// causal bf16 backward holds two workgroups of 64 buckets per CU, and of 32 two
// (k_bwd_out, one wave per SIMD) or three (k_bwd_reduce), the fp32 one of either
// one or two (K=4 L=4 48 x 8192 global: 768 workgroups 350 us, 384 401).
// The non-causal forward of 32 buckets holds six (fp32 four), forward us with
// the causal operator's four (fp32 two) and with these: bf16 K=2 L=5 384 x 785
// 75 -> 70, 576 x 197 54 -> 49, K=3 L=4 32 x 16384 105 -> 98, fp32 48 x 3000
// 82 -> 60.
int64_t target_blocks(bool bf, int SP, bool bwd, bool causal) {
    if (SP == 128) return bf && !bwd ? 512 : 256;
    if (SP == 64) return bf ? 768 : 512;
    if (!bwd && !causal) return bf ? 1536 : 1024;
    return bf ? 1024 : 512;
}
// Longest segment, forward or backward, in 32-token tiles (8192 tokens).
// The bf16 kernels carry B in fp32 MFMA accumulators through a segment:
// k_fwd_reduce and k_bwd_reduce add tile sums from the segment's start,
// and k_bwd_out re-derives B(t) by subtracting them from the fp64 state at
// the segment's end.  Those roundings are relative to the state the walk
// starts from, while B(t) early in a sequence can be far below it (V with a
// non-zero mean makes |B| grow linearly in t), so the walk length must not
// grow with T: long sequences add segments instead.  At 256 tiles the
// walks' error stays below the bf16 operand rounding of B (measured: dK of
// the first tokens equals that of one-tile walks; it grows from 512 tiles).
constexpr int64_t kMaxSegTiles = 256;

struct Plan {
    int SP = 0, S = 0, R = 0, nslice = 1, Spad = 0;
    bool parts = false;  // partial outputs + slice sum (sliced<KB>() instantiations)
    int64_t N = 0, ntiles = 0;
    int nseg = 0, tps = 0;
    int fnseg = 0, fmul = 1;  // forward segments; forward segments per segment of this plan
    size_t esize = 0;
    size_t state_bytes = 0, fws = 0, bws = 0;
    size_t fws_core = 0, bws_core = 0, part_bytes = 0;  // partial-output buffers follow the core
    size_t xpart_bytes = 0;  // sliced dX partials (dproj columns), one buffer each for dQ and dK
    // global normalisation: den partials after the forward workspace; rden
    // and gden [N][T] after the backward workspace, then (sliced) the slices'
    // shares of sum_s P_Q dO.B_s [nslice][N][T]
    size_t gfws = 0, gbws = 0, tok_bytes = 0;
};

// Bucket slices: a workgroup handles SP buckets.  K <= 4 (at most 128 buckets
// in 32 projection columns) runs one slice of the padded bucket count, 32, 64
// or 128; wider tables run ceil(S / SP) slices of 128 (fp32: 32) buckets whose
// partial outputs are summed.
void slice_plan(int dtype, int K, int S, int &SP, int &nslice) {
    if (K <= 4) {
        SP = (S + 31) / 32 * 32;
        if (SP == 96) SP = 128;
        nslice = 1;
        return;
    }
    SP = dtype == RACE_DTYPE_BF16 ? 128 : 32;
    nslice = (S + SP - 1) / SP;
}

// Work-items of a 1-D launch: the dispatch packet counts them in 32 bits.
constexpr int64_t kMaxWorkItems = 0xFFFFFFFFll;

// Workgroups of a launch over nseg segments a stream, as the busiest XCD sees it
// times 8: the workgroups go round the 8 XCDs (32 CUs each), those of a sliced
// launch in groups of the slices of one segment (K=6 L=5, 3 slices, 7 streams of
// 12 segments are 252 workgroups, but 33 on four XCDs: a second round).
int64_t launch_wgs(const Plan &p, int64_t nseg) { return (nseg * p.N + 7) / 8 * 8 * p.nslice; }
// Time, in tiles, of a launch of wgs workgroups that walk `tiles` tiles, r of
// them resident per CU: whole rounds, and a last one with fewer per CU, which
// run faster for it.
double rounds_cost(int64_t wgs, int64_t r, int64_t tiles) {
    const int64_t n = (wgs + 255) / 256, rem = n % r;
    return ((double)(n / r) + (rem ? 0.5 + 0.5 * (double)rem / (double)r : 0.0)) * (double)(tiles + 2);
}

// The causal backward of 128 buckets runs one workgroup per CU: of the joins of 1
// to `most` of fnseg forward segments (tps tiles each) into one backward segment,
// the one whose launch takes the fewest tiles in whole rounds, and those tiles.
double whole_rounds(const Plan &p, int64_t fnseg, int64_t tps, int64_t most, int64_t &join) {
    double cost = 1e300;
    for (int64_t j = 1; j <= most && j <= fnseg; ++j) {
        const int64_t wgs = launch_wgs(p, (fnseg + j - 1) / j);
        const double c = rounds_cost(wgs, 1, j * tps);
        if (c < cost) {
            cost = c;
            join = j;
        }
        if (wgs <= 256) break;  // one round: longer segments only take longer
    }
    return cost;
}

// Tiles per segment of a short sequence: 1 to 4 rounds of target_blocks
// workgroups (non-causal: half of one too, where that saves one-tile segments),
// whichever the cost in tiles -- per round a segment and 2 tiles of set-up, per
// workgroup its state passes (none read per segment by the non-causal operator:
// half) -- says is shortest.  One 8-wave workgroup per CU
// only where that leaves segments of 8 tiles: the backward then still joins
// pairs of forward segments.  With 128 causal buckets the backward's rounds count
// too, at twice the forward's time a tile: one forward segment would leave it no
// choice (K=6 L=5, 3 slices, 96 streams x 1000, us, forward and backward: one
// segment 184 and 530, three 156 and 420).
int64_t short_tiles(const race_desc *d, const Plan &p, int64_t per) {
    int64_t tb = target_blocks(d->dtype == RACE_DTYPE_BF16, p.SP, false, d->causal);
    if (tb < 512 && p.ntiles * per < 8 * tb) tb = 512;
    const double row = 0.018 * p.SP / 128 * (d->causal ? 1.0 : 0.5);
    int64_t best = p.ntiles;
    double cost = 1e300;
    for (const int half : {1, 2, 4, 6, 8}) {
        if (half == 1 && d->causal) continue;
        int64_t nseg = tb * half / (2 * per);
        nseg = nseg < 1 ? 1 : (nseg > p.ntiles ? p.ntiles : nseg);
        const int64_t tps = (p.ntiles + nseg - 1) / nseg;
        nseg = (p.ntiles + tps - 1) / tps;
        double c = (double)((launch_wgs(p, nseg) + tb - 1) / tb) * (double)(tps + 2) + (double)(nseg * per) * row;
        int64_t join;
        if (d->causal && p.SP == 128) c += 2 * whole_rounds(p, nseg, tps, kMaxSegTiles / tps, join);
        if (c < cost) {
            cost = c;
            best = tps;
        }
    }
    return best;
}

// Tiles per backward segment of the non-causal operator (no more segments than the
// forward's).  Backward, us, with one
// residency of segments by target_blocks alone, and with this: K=3 L=8 16 x 65536
// 397, 322; K=6 L=5 (3 slices) 48 x 8192 1178, 802.
int64_t own_tiles(const race_desc *d, const Plan &p, bool capped) {
    const bool bf = d->dtype == RACE_DTYPE_BF16;
    // 64 buckets in bf16: 16-column rows (K = 4) leave LDS for a third workgroup
    const int64_t r = bf && p.SP == 64 ? (d->K == 4 ? 3 : 2) : target_blocks(bf, p.SP, true, false) / 256;
    int64_t best = 0;
    double cost = 1e300;
    // one segment a stream, up to one more than fill four rounds; of the counts
    // that put n workgroups on a CU the largest, whose segments are the shortest
    const int64_t most = 4 * 256 * r / (p.N * p.nslice) + 1;
    for (int64_t n = 0; n <= 8 * r; ++n) {
        int64_t nseg = n ? 256 * n / (8 * p.nslice) * 8 / p.N : 1;
        if (nseg < 1) continue;
        if (nseg > most) nseg = most;
        if (nseg > p.fnseg) nseg = p.fnseg;
        int64_t tl = (p.ntiles + nseg - 1) / nseg;
        if (capped && tl > kMaxSegTiles) tl = kMaxSegTiles;
        const double c = rounds_cost(launch_wgs(p, (p.ntiles + tl - 1) / tl), r, tl);
        if (c < cost) {
            cost = c;
            best = tl;
        }
    }
    return best;
}

// Forward segments per backward segment of the causal operator, at most `most`.
// 128 buckets: whole_rounds.  The others take the fewest segments that fill
// target_blocks; of the counts that leave as many, the smallest, so that the last
// is not a short one.  Backward of 48 streams x 8192,
// us, the fewest that fill one residency and with this: K=6 L=5 2534, 1266, K=7 L=4
// 3230, 1620.
int64_t joined_segments(const race_desc *d, const Plan &p, int64_t per, int64_t most) {
    const int64_t tb = target_blocks(d->dtype == RACE_DTYPE_BF16, p.SP, true, true);
    if (most > p.fnseg) most = p.fnseg;
    int64_t m = (p.fnseg * per + tb - 1) / tb;
    if (p.SP == 128) whole_rounds(p, p.fnseg, p.tps, most, m);
    if (m > most) m = most;
    if (m < 1) return 1;
    const int64_t nb = (p.fnseg + m - 1) / m;
    return (p.fnseg + nb - 1) / nb;
}

// bwd: the backward's plan (longer segments of whole forward ones, at most
// kMaxSegTiles); it rejects an explicit seg_tiles above kMaxSegTiles.
// walks: the automatic plan of a call whose state a backward may walk (every
// call but the no-allocation forward and the probability outputs) caps its
// segments at kMaxSegTiles.
// probs: the probability outputs, which keep no state and run kTargetBlocks
// workgroups at any length.
int make_plan(const race_desc *d, Plan &p, bool bwd = false, bool walks = true, bool probs = false) {
    if (!d) return fail(RACE_E_INVALID, "descriptor is NULL");
    if (d->dtype != RACE_DTYPE_F32 && d->dtype != RACE_DTYPE_BF16)
        return fail(RACE_E_INVALID, "dtype %d is not RACE_DTYPE_F32 or RACE_DTYPE_BF16", d->dtype);
    if (d->M < 1 || d->B < 1 || d->T < 1 || d->H < 1)
        return fail(RACE_E_INVALID, "M, B, T, H must be >= 1 (got %lld, %lld, %lld, %lld)", (long long)d->M,
                    (long long)d->B, (long long)d->T, (long long)d->H);
    if (d->D != D) return fail(RACE_E_UNSUPPORTED, "head dim D=%lld unsupported (this build: D=64)", (long long)d->D);
    // the kernels count tiles of 32 tokens in 32-bit integers
    if (d->T > (1ll << 35))
        return fail(RACE_E_UNSUPPORTED, "T=%lld tokens per sequence unsupported (T <= 2^35)", (long long)d->T);
    if (d->L < 1 || d->K < 1) return fail(RACE_E_INVALID, "L and K must be >= 1 (got L=%d K=%d)", d->L, d->K);
    if (d->K > 8) return fail(RACE_E_UNSUPPORTED, "K=%d hash bits unsupported (K <= 8)", d->K);
    if (d->L * d->K > NCOL)
        return fail(RACE_E_UNSUPPORTED, "L*K=%d projection columns unsupported (L*K <= %d)", d->L * d->K, NCOL);
    if (!(d->eps >= 0.f) || d->eps > 1e30f) return fail(RACE_E_INVALID, "eps must be finite and >= 0");
    if (!d->inv_temp_ptr && (!(d->inv_temp == d->inv_temp) || d->inv_temp > 1e30f || d->inv_temp < -1e30f))
        return fail(RACE_E_INVALID, "inv_temp must be finite");
    if (d->inv_temp_ptr && (uintptr_t)d->inv_temp_ptr % 4)
        return fail(RACE_E_INVALID, "inv_temp_ptr is not 4-byte aligned");
    if (d->planes_m_stride < 0) return fail(RACE_E_INVALID, "planes_m_stride must be >= 0");
    if (d->phases < 0 || d->phases > 7) return fail(RACE_E_INVALID, "phases must be a RACE_PHASE_* bitmask");
    p.R = 1 << d->K;
    p.S = d->L * p.R;
    slice_plan(d->dtype, d->K, p.S, p.SP, p.nslice);
    // (fp32: the rows of 65 to 96 buckets in a workgroup of 128 stay 96, StateRows)
    p.Spad = d->dtype == RACE_DTYPE_F32 && p.nslice == 1 ? (p.S + 31) / 32 * 32 : p.nslice * p.SP;
    p.parts = d->K > 4;
    p.N = d->M * d->B * d->H;
    if (p.N > 65535) return fail(RACE_E_UNSUPPORTED, "M*B*H=%lld streams exceed 65535", (long long)p.N);
    p.ntiles = (d->T + TT - 1) / TT;
    int64_t tps;
    if (d->seg_tiles > 0) {
        if (bwd && d->seg_tiles > kMaxSegTiles)
            return fail(RACE_E_UNSUPPORTED,
                        "seg_tiles=%d exceeds %lld tiles: the backward's fp32 walks of the forward state are "
                        "bounded by the segment length", d->seg_tiles, (long long)kMaxSegTiles);
        tps = d->seg_tiles;
    } else {
        const int64_t per = p.N * p.nslice;  // workgroups per segment index
        int64_t nseg = (kTargetBlocks + per - 1) / per;
        if (nseg > p.ntiles) nseg = p.ntiles;
        tps = (p.ntiles + nseg - 1) / nseg;
        if (tps < kLongSegTiles && !probs && p.ntiles * per > kOneTileBlocks) tps = short_tiles(d, p, per);
        if (walks && tps > kMaxSegTiles) tps = kMaxSegTiles;
    }
    p.tps = (int)(tps < p.ntiles ? tps : p.ntiles);
    const int64_t nseg = (p.ntiles + p.tps - 1) / p.tps;
    if (nseg > (1 << 30)) return fail(RACE_E_UNSUPPORTED, "too many segments");
    // the tile kernels' grids: (nseg, N) of threads_of(SP)-thread workgroups,
    // or (sliced) 1-D over whole blocks of 8 (segment, stream) groups x slices
    const int64_t wgs = p.parts ? (nseg * p.N + 7) / 8 * 8 * p.nslice : nseg;
    if (wgs * threads_of(p.SP) > kMaxWorkItems)
        return fail(RACE_E_UNSUPPORTED, "%lld segments x %lld streams x %d bucket slices exceed one launch's 2^32 "
                    "work-items", (long long)nseg, (long long)p.N, p.nslice);
    p.nseg = (int)nseg;
    p.fnseg = p.nseg;
    p.esize = d->dtype == RACE_DTYPE_BF16 ? 2 : 4;
    const size_t blk = (size_t)p.Spad * SROW;
    p.state_bytes = (size_t)p.N * (p.fnseg + 1) * blk * sizeof(double);
    p.fws_core = align16((size_t)p.N * p.fnseg * blk * sizeof(double));
    if (bwd && d->seg_tiles <= 0) {
        // backward segments of fmul forward ones (one segment when that
        // covers the sequence); explicit seg_tiles keeps the forward's
        // (a segment is at most kMaxSegTiles long: m * tps tiles, or the whole
        // sequence when that is shorter)
        // The non-causal backward reads no state row but the totals, so its
        // segments are its own.
        const int64_t per = p.N * p.nslice;
        const bool capped = walks && p.ntiles > kMaxSegTiles;
        if (!d->causal) {
            p.tps = (int)own_tiles(d, p, capped);
            p.nseg = (int)((p.ntiles + p.tps - 1) / p.tps);
        } else if (const int64_t m = joined_segments(d, p, per, capped ? kMaxSegTiles / p.tps : p.fnseg); m > 1) {
            const int64_t tl = (int64_t)p.tps * m;
            p.fmul = (int)m;
            p.tps = (int)(tl < p.ntiles ? tl : p.ntiles);
            p.nseg = (int)((p.ntiles + p.tps - 1) / p.tps);
        }
    }
    p.bws_core = 2 * (size_t)p.N * p.nseg * blk * sizeof(float) +
                 align16(2 * (size_t)p.N * p.nseg * p.nslice * sizeof(double));
    // k_dx_finish runs one 64-lane wave per 64 tokens of a stream
    if (p.parts && (p.N * ((d->T + 16 * DXF_BLK - 1) / (16 * DXF_BLK)) + 3) / 4 * 256 > kMaxWorkItems)
        return fail(RACE_E_UNSUPPORTED, "M*B*H*T=%lld token-heads exceed one dX launch's 2^32 work-items",
                    (long long)(p.N * d->T));
    const bool f32 = d->dtype == RACE_DTYPE_F32;
    const int parts = p.parts ? p.nslice : 0;  // slices that leave partial outputs
    p.part_bytes = align16((size_t)parts * p.N * d->T * D * p.esize);
    const size_t xesize = xpart_f32(!f32, p.SP, d->K) ? sizeof(float) : p.esize;
    p.xpart_bytes = align16((size_t)parts * p.N * d->T * xcols_of(p.SP, d->K) * xesize);
    p.fws = p.fws_core + p.part_bytes;                         // partial O
    p.bws = p.bws_core + 2 * p.xpart_bytes + p.part_bytes;     // dproj columns for dQ, dK; partial dV
    p.tok_bytes = align16((size_t)p.N * d->T * sizeof(float));
    p.gfws = p.fws + parts * p.tok_bytes;
    p.gbws = p.bws + (2 + parts) * p.tok_bytes;  // + the slices' gsum
    return RACE_OK;
}

// Largest token stride (elements) whose lane byte offsets inside a 32-token
// tile, ((TT - 1) * stride + D) * esize, fit the kernels' 32-bit offsets and
// the 2^31 - 1 byte record size of k_fwd_out's buffer stores.  It also keeps a
// tile's byte stride TT * stride * esize below 2^32, which the kernels' tile
// base addresses (tile index times that stride, a 32 x 32-bit product) need.
int64_t max_token_stride(size_t esize) { return (0x7FFFFFFFll / (int64_t)esize - D) / (TT - 1); }

int check_tensor(const char *name, const void *ptr, const int64_t *st, size_t esize, int64_t T) {
    if (!ptr) return fail(RACE_E_INVALID, "%s is NULL", name);
    if ((uintptr_t)ptr % 16) return fail(RACE_E_INVALID, "%s is not 16-byte aligned", name);
    for (int j = 0; j < 4; ++j) {
        if (st[j] < 0) return fail(RACE_E_INVALID, "%s stride %d is negative", name, j);
        if ((st[j] * (int64_t)esize) % 16)
            return fail(RACE_E_INVALID, "%s stride %d (%lld elements) is not a multiple of 16 bytes", name, j,
                        (long long)st[j]);
    }
    if (T > 1 && st[2] < D)
        return fail(RACE_E_INVALID, "%s token stride %lld overlaps rows", name, (long long)st[2]);
    if (st[2] > max_token_stride(esize))  // lane byte offsets within a 32-token tile are 32-bit
        return fail(RACE_E_UNSUPPORTED, "%s token stride %lld exceeds %lld elements (32-bit tile offsets)", name,
                    (long long)st[2], (long long)max_token_stride(esize));
    return RACE_OK;
}

// A tensor the call writes: as check_tensor, and no two (m, b, t, h) rows
// may share memory through a zero stride or heads closer than D elements
// (workgroups of different streams would race on the same rows).
int check_out(const char *name, const void *ptr, const int64_t *st, size_t esize, const race_desc *d) {
    int rc = check_tensor(name, ptr, st, esize, d->T);
    if (rc) return rc;
    const int64_t sz[4] = {d->M, d->B, d->T, d->H};
    static const char *dim[4] = {"M", "B", "T", "H"};
    for (int j = 0; j < 4; ++j)
        if (sz[j] > 1 && st[j] == 0)
            return fail(RACE_E_INVALID, "%s is written but has stride 0 over %s (size %lld)", name, dim[j],
                        (long long)sz[j]);
    if (d->H > 1 && st[3] < D)
        return fail(RACE_E_INVALID, "%s head stride %lld overlaps rows (< D)", name, (long long)st[3]);
    return RACE_OK;
}

Strides strides_of(const int64_t *s) { return Strides{s[0], s[1], s[2], s[3]}; }

Args base_args(const race_desc *d, const Plan &p, const float *planes) {
    Args a{};
    a.sq = strides_of(d->q_stride);
    a.sk = strides_of(d->k_stride);
    a.sv = strides_of(d->v_stride);
    a.so = strides_of(d->o_stride);
    a.sdo = strides_of(d->do_stride);
    a.sg = strides_of(d->g_stride);
    a.planes = planes;
    a.planes_m_stride = d->planes_m_stride;
    a.M = (int)d->M;
    a.B = (int)d->B;
    a.H = (int)d->H;
    a.L = d->L;
    a.K = d->K;
    a.R = p.R;
    a.S = p.S;
    a.T = d->T;
    a.eps = d->eps;
    a.inv_temp = d->inv_temp;
    a.inv_temp_ptr = d->inv_temp_ptr;
    a.nseg = p.nseg;
    a.tps = p.tps;
    a.fnseg = p.fnseg;
    a.fdrows = p.nseg;
    a.fmul = p.fmul;
    a.nslice = p.nslice;
    a.Spad = p.Spad;
    return a;
}

int launched(const char *what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(RACE_E_LAUNCH, "%s: %s", what, hipGetErrorString(e));
    return ok();
}

bool run_phase(const race_desc *d, int ph) { return d->phases == 0 || (d->phases & ph); }

// Launch grid of the tile kernels (their wg_pos): (nseg, N) unsliced; sliced,
// 1-D over blocks of 8 (segment, stream) groups times the slices.
dim3 tile_grid(const Plan &p) {
    if (!p.parts) return dim3((unsigned)p.nseg, (unsigned)p.N, 1);
    return dim3((unsigned)(((int64_t)p.nseg * p.N + 7) / 8 * 8 * p.nslice), 1, 1);
}

template <typename T>
void slice_sum(const Plan &p, const race_desc *d, const void *part, const int64_t *st, void *out, hipStream_t s) {
    if constexpr (std::is_same<T, bf16>::value) {
        if (p.nslice == 8) {  // the 8-bit slices of 4 tables
            const int64_t n8 = p.N * d->T * (D / 8);
            k_slice_sum8<8><<<elem_blocks(n8), ELEM_THREADS, 0, s>>>((const bf16 *)part, p.N, d->T, (int)d->B,
                                                                     (int)d->H, Strides{st[0], st[1], st[2], st[3]},
                                                                     (bf16 *)out);
            return;
        }
    }
    const int64_t n4 = p.N * d->T * (D / 4);
    k_slice_sum<T><<<elem_blocks(n4), ELEM_THREADS, 0, s>>>((const T *)part, p.nslice, p.N, d->T, (int)d->B, (int)d->H,
                                                                Strides{st[0], st[1], st[2], st[3]}, (T *)out);
}

// dX (dQ, dK, the probability backward's dx) of sliced instantiations from
// the slices' dproj columns
template <typename T>
void dx_finish(const Plan &p, const race_desc *d, const void *part, const Args &a, const int64_t *st, void *out,
               hipStream_t s) {
    const int64_t waves = p.N * ((d->T + 16 * DXF_BLK - 1) / (16 * DXF_BLK));  // one wave per 64 tokens
    if constexpr (std::is_same<T, bf16>::value) {
        // 8-bit hashes, slices of 128 buckets: two slices per table, 8 fp32
        // columns each (the plan gives L <= 4 and 2L slices whenever this holds)
        if (xpart_f32(true, p.SP, d->K)) {
            k_dx_finish8<<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(
                (const float *)part, d->L, a.planes, a.planes_m_stride, (int)d->B, (int)d->H, p.N, d->T,
                Strides{st[0], st[1], st[2], st[3]}, (bf16 *)out);
            return;
        }
    }
    k_dx_finish<T><<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(
        (const T *)part, p.nslice, xcols_of(p.SP, d->K), p.SP, d->K, d->L, a.planes, a.planes_m_stride, (int)d->B,
        (int)d->H, p.N, d->T, Strides{st[0], st[1], st[2], st[3]}, (T *)out);
}

// Whole-tile instantiations (template flag AL of the tile kernels): compiled
// for the causal bf16 slices of 128 buckets at 4 and 8 hash bits and of 32 and
// 64 at 2 to 4, and used when every tile holds TT tokens (T % TT == 0) and
// every bucket of every slice is one of the S buckets, so no load, store or
// probability needs a row or bucket guard.  Those of 32 and 64 buckets walk B in
// fp64 as the general ones do (walk_f64); without the guards the compiler forms
// P_K's lo part with the product that makes P_K, one rounding fewer, so outputs
// differ from the general kernels' (by 3e-5 of 2e-3 and more off 64 bits, either
// way the same).  Forward + backward of
// 48 x 8192, us: K=4 L=4 351 -> 319 (global 354 -> 324), L=2 354 -> 319 (396 ->
// 358), K=3 L=8 390 -> 364, L=4 369 -> 332, K=2 L=16 374 -> 349, L=8 357 -> 323.
// Elsewhere the template argument is false and both branches below launch the
// same kernel.
template <typename T, int SP, int KB> constexpr bool al_compiled() {
    return std::is_same<T, bf16>::value && (SP == 128 ? KB == 4 || KB == 8 : KB >= 2 && KB <= 4);
}
bool whole_tiles(const race_desc *d, const Plan &p) { return d->T % TT == 0 && p.S == p.Spad; }

// The causal F1 operator walks the forward state B back through each backward
// segment (k_bwd_out); its whole-tile bf16 instantiations of 128 buckets do it in fp32, the
// others in fp64 (race_kernels.hip walk_f64).  A table's logits differ by at
// most 2 K |inv_temp| (|tanh| <= 1 per bit), so at most e^(2 K |inv_temp|)
// separates its largest and smallest probability: above K |inv_temp| = 2
// (e^4), or with a temperature on the device, whole tiles take the segment
// sums from the generic k_fwd_reduce (fp64) and walk B in fp64 in the
// whole-tile k_bwd_out.  The forward and the backward of one descriptor choose
// alike.
bool exact_walk(const race_desc *d) {
    return d->causal && (d->inv_temp_ptr != nullptr || (double)d->K * std::fabs((double)d->inv_temp) > 2.0);
}

// Up to TOT_FEW segments leave k_seg_totals' waves one element a lane or none.
template <typename V> void seg_totals(V *dst, int rows, const V *delta, const Plan &p, int elems, hipStream_t s) {
    if (p.nseg <= TOT_FEW)
        k_seg_totals_few<<<dim3((elems + TOT_FEW_THREADS - 1) / TOT_FEW_THREADS, (unsigned)p.N), TOT_FEW_THREADS, 0, s>>>(
            dst, rows, delta, p.nseg, elems);
    else
        k_seg_totals<<<dim3((elems + SCAN_THREADS - 1) / SCAN_THREADS, (unsigned)p.N), SCAN_THREADS * TOT_WAVES, 0, s>>>(
            dst, rows, delta, p.nseg, elems);
}

// Segment scans: the causal operator reads a prefix (forward) or suffix
// (backward) row per segment, the non-causal one only the totals.  With one
// segment its sums are the totals and the reduce kernels write them in place
// (lone_segment): no launch (1536 streams of 197 tokens, K=2 L=5: the two took
// 19 and 16 us of 224).
void fwd_scan(const race_desc *d, const Plan &p, const Args &a, int elems, hipStream_t s) {
    const dim3 grid((elems + SCAN_THREADS - 1) / SCAN_THREADS, (unsigned)p.N);
    if (d->causal)
        k_fwd_scan<<<grid, SCAN_THREADS, 0, s>>>(a.fstate, a.fdelta, p.nseg, elems);
    else if (p.nseg > 1)
        seg_totals(a.fstate + (int64_t)p.nseg * elems, p.nseg + 1, a.fdelta, p, elems, s);
}
void bwd_scan(const race_desc *d, const Plan &p, const Args &a, int elems, hipStream_t s) {
    const dim3 grid((elems + SCAN_THREADS - 1) / SCAN_THREADS, (unsigned)p.N);
    if (d->causal)
        k_bwd_scan<<<grid, SCAN_THREADS, 0, s>>>(a.rstate, a.rdelta, p.nseg, elems);
    else if (p.nseg > 1)
        seg_totals(a.rstate, p.nseg, a.rdelta, p, elems, s);
}

void lone_segment(const race_desc *d, const Plan &p, Args &a, bool bwd) {
    if (d->causal || p.nseg > 1) return;
    if (bwd) {
        a.rdelta = a.rstate;
    } else {  // row 1 of the state's 2
        a.fdelta = a.fstate + (size_t)p.Spad * SROW;
        a.fdrows = 2;
    }
}

template <typename T, int SP, int KB> int fwd_impl(const race_desc *d, const Plan &p, Args a, hipStream_t s) {
    lone_segment(d, p, a, false);
    const dim3 grid = tile_grid(p);
    constexpr bool ALC = al_compiled<T, SP, KB>();
    const bool al = ALC && whole_tiles(d, p);
    if (run_phase(d, RACE_PHASE_REDUCE)) {
        if (al && (SP < 128 || !exact_walk(d)))
            k_fwd_reduce<T, SP, KB, ALC><<<grid, threads_of(SP), 0, s>>>(a);
        else
            k_fwd_reduce<T, SP, KB><<<grid, threads_of(SP), 0, s>>>(a);
    }
    const int elems = p.Spad * SROW;
    if (run_phase(d, RACE_PHASE_SCAN))
        fwd_scan(d, p, a, elems, s);
    if (run_phase(d, RACE_PHASE_OUT)) {
        if (d->causal && al)
            k_fwd_out<T, SP, true, KB, false, ALC><<<grid, threads_of(SP), 0, s>>>(a);
        else if (d->causal)
            k_fwd_out<T, SP, true, KB, false><<<grid, threads_of(SP), 0, s>>>(a);
        else
            k_fwd_out<T, SP, false, KB, false><<<grid, threads_of(SP), 0, s>>>(a);
        if (sliced<KB>()) {
            slice_sum<T>(p, d, a.opart, d->o_stride, a.out, s);
            if (a.den) {
                const int64_t nt = p.N * d->T;
                k_den_sum<<<elem_blocks(nt), ELEM_THREADS, 0, s>>>(a.denpart, p.nslice, nt, a.den);
            }
        }
    }
    return launched("race_fwd");
}

template <typename T, int SP, int KB>
int bwd_impl(const race_desc *d, const Plan &p, Args a, float *grad_inv_temp, hipStream_t s) {
    lone_segment(d, p, a, true);
    const dim3 grid = tile_grid(p);
    constexpr bool ALC = al_compiled<T, SP, KB>();
    const bool al = ALC && whole_tiles(d, p);
    if (run_phase(d, RACE_PHASE_REDUCE)) {
        if (d->causal && al)
            k_bwd_reduce<T, SP, true, KB, false, ALC><<<grid, threads_of(SP), 0, s>>>(a);
        else if (d->causal)
            k_bwd_reduce<T, SP, true, KB, false><<<grid, threads_of(SP), 0, s>>>(a);
        else
            k_bwd_reduce<T, SP, false, KB, false><<<grid, threads_of(SP), 0, s>>>(a);
        if (sliced<KB>()) dx_finish<T>(p, d, a.dqpart, a, d->g_stride, a.dq, s);
    }
    const int elems = p.Spad * SROW;
    if (run_phase(d, RACE_PHASE_SCAN))
        bwd_scan(d, p, a, elems, s);
    if (run_phase(d, RACE_PHASE_OUT)) {
        if (d->causal && al) {
            if constexpr (ALC) {
                if (exact_walk(d))
                    k_bwd_out<T, SP, true, KB, false, true, true><<<grid, threads_of(SP), 0, s>>>(a);
                else
                    k_bwd_out<T, SP, true, KB, false, true><<<grid, threads_of(SP), 0, s>>>(a);
            }
        } else if (d->causal)
            k_bwd_out<T, SP, true, KB, false><<<grid, threads_of(SP), 0, s>>>(a);
        else
            k_bwd_out<T, SP, false, KB, false><<<grid, threads_of(SP), 0, s>>>(a);
        if (sliced<KB>()) {
            dx_finish<T>(p, d, a.dkpart, a, d->g_stride, a.dk, s);
            slice_sum<T>(p, d, a.dvpart, d->g_stride, a.dv, s);
        }
        if (grad_inv_temp) k_temp_sum<<<1, 256, 0, s>>>(a.tpart, 2 * p.N * p.nseg * p.nslice, grad_inv_temp);
    }
    return launched("race_bwd");
}

// Global normalisation (causal): the F1 reduce and scan kernels, then the GN
// readout; its den partials (sliced) are summed with the numerators.  Whole
// tiles run the whole-tile instantiations, as F1 does.
template <typename T, int SP, int KB> int gn_fwd_impl(const race_desc *d, const Plan &p, Args a, hipStream_t s) {
    const dim3 grid = tile_grid(p);
    constexpr bool ALC = al_compiled<T, SP, KB>();
    // the segment sums are F1's (the same kernel): its whole-tile instantiation where it applies
    if (run_phase(d, RACE_PHASE_REDUCE)) {
        if (ALC && whole_tiles(d, p))
            k_fwd_reduce<T, SP, KB, ALC><<<grid, threads_of(SP), 0, s>>>(a);
        else
            k_fwd_reduce<T, SP, KB><<<grid, threads_of(SP), 0, s>>>(a);
    }
    const int elems = p.Spad * SROW;
    if (run_phase(d, RACE_PHASE_SCAN))
        fwd_scan(d, p, a, elems, s);
    if (run_phase(d, RACE_PHASE_OUT)) {
        if (ALC && whole_tiles(d, p))
            k_fwd_out<T, SP, true, KB, true, ALC><<<grid, threads_of(SP), 0, s>>>(a);
        else
            k_fwd_out<T, SP, true, KB, true><<<grid, threads_of(SP), 0, s>>>(a);
        if (sliced<KB>()) {
            const int64_t n4 = p.N * d->T * (D / 4);
            k_slice_sum_gn<T><<<elem_blocks(n4), ELEM_THREADS, 0, s>>>(
                (const T *)a.opart, a.denpart, p.nslice, p.N, d->T, (int)d->B, (int)d->H, strides_of(d->o_stride), (T *)a.out,
                a.den, d->eps);
        }
    }
    return launched("race_fwd_global");
}

// The GN backward: k_bwd_reduce also forms the per-token terms
// (1/max(den, eps) and dL/d den, from out, dout, den, dden) that k_bwd_out reads.
template <typename T, int SP, int KB>
int gn_bwd_impl(const race_desc *d, const Plan &p, Args a, float *grad_beta, hipStream_t s) {
    const dim3 grid = tile_grid(p);
    constexpr bool ALC = al_compiled<T, SP, KB>();
    const bool al = ALC && whole_tiles(d, p);
    if (run_phase(d, RACE_PHASE_REDUCE)) {
        if constexpr (sliced<KB>()) {
            // each slice's share of sum_s P_Q G per token, then rd and gd
            if (al)
                k_bwd_reduce<T, SP, true, KB, true, ALC, true><<<grid, threads_of(SP), 0, s>>>(a);
            else
                k_bwd_reduce<T, SP, true, KB, true, false, true><<<grid, threads_of(SP), 0, s>>>(a);
            const int64_t nt = p.N * d->T;
            k_gn_terms<<<elem_blocks(nt), ELEM_THREADS, 0, s>>>(a.gsum, p.nslice, nt, a.den, a.dden, d->eps, a.rden,
                                                                a.gden);
        }
        if (al)
            k_bwd_reduce<T, SP, true, KB, true, ALC><<<grid, threads_of(SP), 0, s>>>(a);
        else
            k_bwd_reduce<T, SP, true, KB, true><<<grid, threads_of(SP), 0, s>>>(a);
        if (sliced<KB>()) dx_finish<T>(p, d, a.dqpart, a, d->g_stride, a.dq, s);
    }
    const int elems = p.Spad * SROW;
    if (run_phase(d, RACE_PHASE_SCAN))
        bwd_scan(d, p, a, elems, s);
    if (run_phase(d, RACE_PHASE_OUT)) {
        if (al)
            k_bwd_out<T, SP, true, KB, true, ALC><<<grid, threads_of(SP), 0, s>>>(a);
        else
            k_bwd_out<T, SP, true, KB, true><<<grid, threads_of(SP), 0, s>>>(a);
        if (sliced<KB>()) {
            dx_finish<T>(p, d, a.dkpart, a, d->g_stride, a.dk, s);
            slice_sum<T>(p, d, a.dvpart, d->g_stride, a.dv, s);
        }
        if (grad_beta) k_temp_sum<<<1, 256, 0, s>>>(a.tpart, 2 * p.N * p.nseg * p.nslice, grad_beta);
    }
    return launched("race_bwd_global");
}

// Compiled (dtype, slice buckets, hash bits) combinations: every K in 1..8
// with the slice sizes slice_plan() picks (L*K <= 32).
#define RACE_FOR_COMBOS(X)                                                                                          \
    X(bf16, 32, 1) X(bf16, 64, 1) X(bf16, 32, 2) X(bf16, 64, 2) X(bf16, 32, 3) X(bf16, 64, 3) X(bf16, 128, 3)       \
    X(bf16, 32, 4) X(bf16, 64, 4) X(bf16, 128, 4) X(bf16, 128, 5) X(bf16, 128, 6) X(bf16, 128, 7) X(bf16, 128, 8)   \
    X(float, 32, 1) X(float, 64, 1) X(float, 32, 2) X(float, 64, 2) X(float, 32, 3) X(float, 64, 3)                 \
    X(float, 128, 3) X(float, 32, 4) X(float, 64, 4) X(float, 128, 4) X(float, 32, 5) X(float, 32, 6)               \
    X(float, 32, 7) X(float, 32, 8)

template <typename T> int fwd_dispatch(const race_desc *d, const Plan &p, const Args &a, hipStream_t s) {
#define X(TT_, SP_, KB_)                                                                                             \
    if (std::is_same<T, TT_>::value && p.SP == SP_ && d->K == KB_) return fwd_impl<TT_, SP_, KB_>(d, p, a, s);
    RACE_FOR_COMBOS(X)
#undef X
    return fail(RACE_E_UNSUPPORTED, "bucket count / hash bits combination not compiled");
}

template <typename T>
int bwd_dispatch(const race_desc *d, const Plan &p, const Args &a, float *git, hipStream_t s) {
#define X(TT_, SP_, KB_)                                                                                             \
    if (std::is_same<T, TT_>::value && p.SP == SP_ && d->K == KB_) return bwd_impl<TT_, SP_, KB_>(d, p, a, git, s);
    RACE_FOR_COMBOS(X)
#undef X
    return fail(RACE_E_UNSUPPORTED, "bucket count / hash bits combination not compiled");
}

template <typename T> int gn_fwd_dispatch(const race_desc *d, const Plan &p, const Args &a, hipStream_t s) {
#define X(TT_, SP_, KB_)                                                                                             \
    if (std::is_same<T, TT_>::value && p.SP == SP_ && d->K == KB_) return gn_fwd_impl<TT_, SP_, KB_>(d, p, a, s);
    RACE_FOR_COMBOS(X)
#undef X
    return fail(RACE_E_UNSUPPORTED, "bucket count / hash bits combination not compiled");
}

template <typename T> int gn_bwd_dispatch(const race_desc *d, const Plan &p, const Args &a, float *gb, hipStream_t s) {
#define X(TT_, SP_, KB_)                                                                                             \
    if (std::is_same<T, TT_>::value && p.SP == SP_ && d->K == KB_) return gn_bwd_impl<TT_, SP_, KB_>(d, p, a, gb, s);
    RACE_FOR_COMBOS(X)
#undef X
    return fail(RACE_E_UNSUPPORTED, "bucket count / hash bits combination not compiled");
}

// Bucket probabilities (forward) and dP -> dx (backward)
template <typename T, int SP, int KB> int probs_impl(const race_desc *d, const Plan &p, Args a, bool bwd,
                                                     float *grad_inv_temp, hipStream_t s) {
    const dim3 grid = tile_grid(p);
    if (!bwd) {
        k_probs<T, SP, KB, false><<<grid, threads_of(SP), 0, s>>>(a);
        return launched("race_probs");
    }
    k_probs<T, SP, KB, true><<<grid, threads_of(SP), 0, s>>>(a);
    if (sliced<KB>()) dx_finish<T>(p, d, a.dqpart, a, d->g_stride, a.dq, s);
    if (grad_inv_temp) k_temp_sum<<<1, 256, 0, s>>>(a.tpart, p.N * p.nseg * p.nslice, grad_inv_temp);
    return launched("race_probs_bwd");
}

template <typename T>
int probs_dispatch(const race_desc *d, const Plan &p, const Args &a, bool bwd, float *git, hipStream_t s) {
#define X(TT_, SP_, KB_)                                                                                             \
    if (std::is_same<T, TT_>::value && p.SP == SP_ && d->K == KB_) return probs_impl<TT_, SP_, KB_>(d, p, a, bwd, git, s);
    RACE_FOR_COMBOS(X)
#undef X
    return fail(RACE_E_UNSUPPORTED, "bucket count / hash bits combination not compiled");
}

// workspace of race_probs_bwd: temperature partials, then fp32 dx partials (sliced)
size_t probs_ws_core(const Plan &p) { return align16((size_t)p.N * p.nseg * p.nslice * sizeof(double)); }

int check_gn(const race_desc *d) {
    if (d->causal != 1)
        return fail(RACE_E_UNSUPPORTED, "global normalisation is implemented for the causal operator only");
    if (!(d->eps > 0.f)) return fail(RACE_E_INVALID, "eps (the floor of den) must be > 0 for global normalisation");
    return RACE_OK;
}

int check_den(const char *name, const float *p) {
    if (!p) return fail(RACE_E_INVALID, "%s is NULL", name);
    if ((uintptr_t)p % 4) return fail(RACE_E_INVALID, "%s is not 4-byte aligned", name);
    return RACE_OK;
}

// Checks and Args of a backward call (race_bwd, race_bwd_ex)
int bwd_args(const race_desc *d, const Plan &p, const void *q, const void *k, const void *v, const float *planes,
             const void *dout, const void *state, void *dq, void *dk, void *dv, void *ws, size_t ws_bytes, Args &a) {
    int rc;
    if ((rc = check_tensor("q", q, d->q_stride, p.esize, d->T)) || (rc = check_tensor("k", k, d->k_stride, p.esize, d->T)) ||
        (rc = check_tensor("v", v, d->v_stride, p.esize, d->T)) ||
        (rc = check_tensor("dout", dout, d->do_stride, p.esize, d->T)) ||
        (rc = check_out("dq", dq, d->g_stride, p.esize, d)) || (rc = check_out("dk", dk, d->g_stride, p.esize, d)) ||
        (rc = check_out("dv", dv, d->g_stride, p.esize, d)))
        return rc;
    if (!planes) return fail(RACE_E_INVALID, "planes is NULL");
    if (!state) return fail(RACE_E_INVALID, "state is NULL");
    if (!ws || ws_bytes < p.bws)
        return fail(RACE_E_WORKSPACE, "workspace %zu bytes < required %zu", ws_bytes, p.bws);
    a = base_args(d, p, planes);
    a.q = q;
    a.k = k;
    a.v = v;
    a.dout = dout;
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.fstate = (double *)state;
    const size_t blk = (size_t)p.N * p.nseg * p.Spad * SROW;
    a.rdelta = (float *)ws;
    a.rstate = a.rdelta + blk;
    a.tpart = (double *)(a.rstate + blk);  // blk is even: 8-byte aligned
    if (p.parts) {
        float *part = (float *)((char *)ws + p.bws_core);
        a.dqpart = part;
        a.dkpart = (char *)part + p.xpart_bytes;
        a.dvpart = (char *)part + 2 * p.xpart_bytes;
    }
    return RACE_OK;
}

// prefix mean: segment length so that NS * nseg ~ 4096 waves, or (k_pm4_*, rows
// of 16 tokens) ~ 16384 rows of 16 lanes; at most 4096 segments a stream, which
// the scans walk one after the other.
int64_t pm_tseg(int64_t NS, int64_t T, bool rows) {
    int64_t nseg = ((rows ? 16384 : 4096) + NS - 1) / NS;
    if (nseg > 4096) nseg = 4096;
    if (nseg > T) nseg = T;
    if (nseg < 1) nseg = 1;
    const int64_t t = (T + nseg - 1) / nseg;
    return rows ? (t + 15) / 16 * 16 : t;
}
// Whether the k_pm4_* kernels take a call: 16-byte pieces of at most 16 lanes'
// columns.  The scalar arrays need no alignment.
bool pm_rows(int64_t D, const void *a, const void *b, const void *c, const void *d) {
    const uintptr_t m = (uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d;
    return D % 4 == 0 && D <= 64 && m % 16 == 0;
}
size_t pm_workspace(int64_t NS, int64_t T, int64_t D, bool rows) {
    const int64_t tseg = pm_tseg(NS, T, rows), nseg = (T + tseg - 1) / tseg;
    const size_t row = (size_t)(D + 1) * sizeof(double);
    // forward: delta + state; backward adds invA, alpha, rdelta, rstate
    return (size_t)NS * nseg * row + (size_t)NS * (nseg + 1) * row + 2 * (size_t)NS * T * sizeof(double) +
           2 * (size_t)NS * nseg * row;
}

int pm_check(const void *a, const char *na, int64_t NS, int64_t T, int64_t D) {
    if (!a) return fail(RACE_E_INVALID, "%s is NULL", na);
    if (NS < 1 || T < 1 || D < 1) return fail(RACE_E_INVALID, "NS, T, D must be >= 1");
    if (D > 64 * PM_MAXC) return fail(RACE_E_UNSUPPORTED, "D=%lld unsupported (D <= %d)", (long long)D, 64 * PM_MAXC);
    if (NS > 65535) return fail(RACE_E_UNSUPPORTED, "NS=%lld exceeds 65535", (long long)NS);
    return RACE_OK;
}

// ---------------------------------------------------------------- no-allocation forward
// race_fwd_noalloc keeps the forward's segment sums and segment state in one
// file-scope device array instead of caller buffers.  In host code `scratch`
// names a host-side stand-in: kernels get the device address that
// hipGetSymbolAddress returns for the current device (each GPU holds its own
// copy of the array), looked up once per device and cached.
static __device__ __align__(256) unsigned char scratch[RACE_NOALLOC_SCRATCH_BYTES];

std::mutex g_scratch_mu;
constexpr int kMaxDevices = 64;
void *g_scratch_ptr[kMaxDevices];

int scratch_address(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(RACE_E_LAUNCH, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return fail(RACE_E_UNSUPPORTED, "device ordinal %d >= %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(RACE_E_LAUNCH, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return RACE_OK;
}

constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
// What a call is measured by: its state and workspace, and in fp32 the partial
// outputs of slices of 32 buckets also where one workgroup holds all of them and
// there are none.  That keeps the calls that this entry takes, and those it sends
// to race_fwd, what they have been.
size_t noalloc_parts(const race_desc *d, const Plan &p) {
    return d->dtype == RACE_DTYPE_F32 ? align16((size_t)((p.S + 31) / 32) * p.N * d->T * D * sizeof(float)) : p.part_bytes;
}
size_t noalloc_need(const race_desc *d, const Plan &p) {
    return align256(p.state_bytes) + p.fws_core + noalloc_parts(d, p);
}

// Plan of the no-allocation forward: the descriptor's seg_tiles if set, else
// the default segmentation, coarsened (longer segments) until the state and
// the segment sums fit the scratch array.  Returns RACE_E_UNSUPPORTED with the
// bytes needed when even one segment per stream does not fit.
int noalloc_plan(const race_desc *d, race_desc &dd, Plan &p) {
    if (!d) return fail(RACE_E_INVALID, "descriptor is NULL");
    dd = *d;
    int rc = make_plan(&dd, p, false, false);
    if (rc) return rc;
    if (d->seg_tiles <= 0 && noalloc_need(d, p) > RACE_NOALLOC_SCRATCH_BYTES) {
        // state (nseg + 1 rows) and sums (nseg rows) of N * Spad * (D+1) fp64 each
        const size_t row = (size_t)p.N * p.Spad * SROW * sizeof(double);
        const size_t fixed = noalloc_parts(d, p) + row + 512;
        const int64_t nseg = fixed < RACE_NOALLOC_SCRATCH_BYTES
                                 ? (int64_t)((RACE_NOALLOC_SCRATCH_BYTES - fixed) / (2 * row)) : 0;
        dd.seg_tiles = (int32_t)(nseg > 1 ? (p.ntiles + nseg - 1) / nseg : p.ntiles);
        if ((rc = make_plan(&dd, p, false, false))) return rc;
    }
    if (noalloc_need(d, p) > RACE_NOALLOC_SCRATCH_BYTES)
        return fail(RACE_E_UNSUPPORTED,
                    "race_fwd_noalloc: this call needs %zu bytes of scratch (state %zu, segment sums and partial "
                    "outputs %zu); the no-allocation forward holds %zu -- use race_fwd with caller buffers",
                    noalloc_need(d, p), p.state_bytes, p.fws_core + noalloc_parts(d, p),
                    (size_t)RACE_NOALLOC_SCRATCH_BYTES);
    return RACE_OK;
}

} // namespace
} // namespace race

using namespace race;

extern "C" {

size_t race_state_bytes(const race_desc *d) {
    Plan p;
    if (make_plan(d, p) != RACE_OK) return 0;
    ok();
    return p.state_bytes;
}

size_t race_fwd_workspace_bytes(const race_desc *d) {
    Plan p;
    if (make_plan(d, p) != RACE_OK) return 0;
    ok();
    return p.fws;
}

size_t race_bwd_workspace_bytes(const race_desc *d) {
    Plan p;
    if (make_plan(d, p, true) != RACE_OK) return 0;
    ok();
    return p.bws;
}

int race_fwd(const race_desc *d, const void *q, const void *k, const void *v, const float *planes, void *out,
             void *state, void *ws, size_t ws_bytes, void *stream) {
    Plan p;
    int rc = make_plan(d, p);
    if (rc) return rc;
    if ((rc = check_tensor("q", q, d->q_stride, p.esize, d->T)) || (rc = check_tensor("k", k, d->k_stride, p.esize, d->T)) ||
        (rc = check_tensor("v", v, d->v_stride, p.esize, d->T)) || (rc = check_out("out", out, d->o_stride, p.esize, d)))
        return rc;
    if (!planes) return fail(RACE_E_INVALID, "planes is NULL");
    if (!state) return fail(RACE_E_INVALID, "state is NULL");
    if (!ws || ws_bytes < p.fws)
        return fail(RACE_E_WORKSPACE, "workspace %zu bytes < required %zu", ws_bytes, p.fws);
    Args a = base_args(d, p, planes);
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.fstate = (double *)state;
    a.fdelta = (double *)ws;
    a.opart = p.parts ? (void *)((char *)ws + p.fws_core) : nullptr;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return fwd_dispatch<bf16>(d, p, a, s);
    return fwd_dispatch<float>(d, p, a, s);
}

int race_bwd(const race_desc *d, const void *q, const void *k, const void *v, const float *planes,
             const void *dout, const void *state, void *dq, void *dk, void *dv, float *grad_inv_temp, void *ws,
             size_t ws_bytes, void *stream) {
    Plan p;
    int rc = make_plan(d, p, true);
    if (rc) return rc;
    Args a;
    if ((rc = bwd_args(d, p, q, k, v, planes, dout, state, dq, dk, dv, ws, ws_bytes, a))) return rc;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return bwd_dispatch<bf16>(d, p, a, grad_inv_temp, s);
    return bwd_dispatch<float>(d, p, a, grad_inv_temp, s);
}

size_t race_probs_bwd_workspace_bytes(const race_desc *d) {
    Plan p;
    if (make_plan(d, p, false, false, true) != RACE_OK) return 0;
    ok();
    return probs_ws_core(p) + p.xpart_bytes;
}

int race_probs(const race_desc *d, const void *x, const float *planes, float *P, void *stream) {
    Plan p;
    int rc = make_plan(d, p, false, false, true);
    if (rc || (rc = check_tensor("x", x, d->q_stride, p.esize, d->T)) || (rc = check_den("P", P))) return rc;
    if (!planes) return fail(RACE_E_INVALID, "planes is NULL");
    Args a = base_args(d, p, planes);
    a.q = x;
    a.probs = P;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return probs_dispatch<bf16>(d, p, a, false, nullptr, s);
    return probs_dispatch<float>(d, p, a, false, nullptr, s);
}

int race_probs_bwd(const race_desc *d, const void *x, const float *planes, const float *dP, void *dx,
                   float *grad_inv_temp, void *ws, size_t ws_bytes, void *stream) {
    Plan p;
    int rc = make_plan(d, p, false, false, true);
    if (rc || (rc = check_tensor("x", x, d->q_stride, p.esize, d->T)) || (rc = check_den("dP", dP)) ||
        (rc = check_out("dx", dx, d->g_stride, p.esize, d)))
        return rc;
    if (!planes) return fail(RACE_E_INVALID, "planes is NULL");
    const size_t need = probs_ws_core(p) + p.xpart_bytes;
    if (!ws || ws_bytes < need) return fail(RACE_E_WORKSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
    Args a = base_args(d, p, planes);
    a.q = x;
    a.dq = dx;
    a.dprobs = dP;
    a.tpart = (double *)ws;
    a.dqpart = p.parts ? (char *)ws + probs_ws_core(p) : nullptr;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return probs_dispatch<bf16>(d, p, a, true, grad_inv_temp, s);
    return probs_dispatch<float>(d, p, a, true, grad_inv_temp, s);
}

size_t race_fwd_ex_workspace_bytes(const race_desc *d) {
    Plan p;
    if (make_plan(d, p) != RACE_OK) return 0;
    ok();
    return p.gfws;  // den partials per slice, like the global mode
}

} // extern "C"

namespace race {
namespace {

// race_fwd_ex, and with full race_fwd_padded: the weights also on V, out and den
int fwd_ex(const race_desc *d, const void *q, const void *k, const void *v, const float *planes, const float *kmask,
           bool full, void *out, float *den, void *state, void *ws, size_t ws_bytes, void *stream) {
    Plan p;
    int rc = make_plan(d, p);
    if (rc) return rc;
    if (full && !kmask) return fail(RACE_E_INVALID, "kmask is NULL");
    if (d->causal && (kmask || den))
        return fail(RACE_E_UNSUPPORTED, "key weights and den are implemented for the non-causal operator");
    if ((rc = check_tensor("q", q, d->q_stride, p.esize, d->T)) || (rc = check_tensor("k", k, d->k_stride, p.esize, d->T)) ||
        (rc = check_tensor("v", v, d->v_stride, p.esize, d->T)) || (rc = check_out("out", out, d->o_stride, p.esize, d)) ||
        (kmask && (rc = check_den("kmask", kmask))) || (den && (rc = check_den("den", den))))
        return rc;
    if (!planes) return fail(RACE_E_INVALID, "planes is NULL");
    if (!state) return fail(RACE_E_INVALID, "state is NULL");
    const size_t need = den ? p.gfws : p.fws;
    if (!ws || ws_bytes < need) return fail(RACE_E_WORKSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
    Args a = base_args(d, p, planes);
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.kw = kmask;
    a.kwv = full;
    a.den = den;
    a.fstate = (double *)state;
    a.fdelta = (double *)ws;
    a.opart = p.parts ? (void *)((char *)ws + p.fws_core) : nullptr;
    a.denpart = p.parts && den ? (float *)((char *)ws + p.fws) : nullptr;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return fwd_dispatch<bf16>(d, p, a, s);
    return fwd_dispatch<float>(d, p, a, s);
}

int bwd_ex(const race_desc *d, const void *q, const void *k, const void *v, const float *planes, const float *kmask,
           bool full, const void *dout, const float *dden, const void *state, void *dq, void *dk, void *dv,
           float *grad_inv_temp, void *ws, size_t ws_bytes, void *stream) {
    Plan p;
    int rc = make_plan(d, p, true);
    if (rc) return rc;
    if (full && !kmask) return fail(RACE_E_INVALID, "kmask is NULL");
    if (d->causal && (kmask || dden))
        return fail(RACE_E_UNSUPPORTED, "key weights and den are implemented for the non-causal operator");
    if ((kmask && (rc = check_den("kmask", kmask))) || (dden && (rc = check_den("dden", dden)))) return rc;
    Args a;
    if ((rc = bwd_args(d, p, q, k, v, planes, dout, state, dq, dk, dv, ws, ws_bytes, a))) return rc;
    a.kw = kmask;
    a.kwv = full;
    a.dden = dden;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return bwd_dispatch<bf16>(d, p, a, grad_inv_temp, s);
    return bwd_dispatch<float>(d, p, a, grad_inv_temp, s);
}

} // namespace
} // namespace race

extern "C" {

int race_fwd_ex(const race_desc *d, const void *q, const void *k, const void *v, const float *planes,
                const float *kmask, void *out, float *den, void *state, void *ws, size_t ws_bytes, void *stream) {
    return fwd_ex(d, q, k, v, planes, kmask, false, out, den, state, ws, ws_bytes, stream);
}

int race_bwd_ex(const race_desc *d, const void *q, const void *k, const void *v, const float *planes,
                const float *kmask, const void *dout, const float *dden, const void *state, void *dq, void *dk,
                void *dv, float *grad_inv_temp, void *ws, size_t ws_bytes, void *stream) {
    return bwd_ex(d, q, k, v, planes, kmask, false, dout, dden, state, dq, dk, dv, grad_inv_temp, ws, ws_bytes, stream);
}

int race_fwd_padded(const race_desc *d, const void *q, const void *k, const void *v, const float *planes,
                    const float *mask, void *out, float *den, void *state, void *ws, size_t ws_bytes, void *stream) {
    return fwd_ex(d, q, k, v, planes, mask, true, out, den, state, ws, ws_bytes, stream);
}

int race_bwd_padded(const race_desc *d, const void *q, const void *k, const void *v, const float *planes,
                    const float *mask, const void *dout, const float *dden, const void *state, void *dq, void *dk,
                    void *dv, float *grad_inv_temp, void *ws, size_t ws_bytes, void *stream) {
    return bwd_ex(d, q, k, v, planes, mask, true, dout, dden, state, dq, dk, dv, grad_inv_temp, ws, ws_bytes, stream);
}

size_t race_fwd_global_workspace_bytes(const race_desc *d) {
    Plan p;
    if (make_plan(d, p) != RACE_OK) return 0;
    ok();
    return p.gfws;
}

size_t race_bwd_global_workspace_bytes(const race_desc *d) {
    Plan p;
    if (make_plan(d, p, true) != RACE_OK) return 0;
    ok();
    return p.gbws;
}

int race_fwd_global(const race_desc *d, const void *q, const void *k, const void *v, const float *planes, void *out,
                    float *den, void *state, void *ws, size_t ws_bytes, void *stream) {
    Plan p;
    int rc = make_plan(d, p);
    if (rc || (rc = check_gn(d))) return rc;
    if ((rc = check_tensor("q", q, d->q_stride, p.esize, d->T)) || (rc = check_tensor("k", k, d->k_stride, p.esize, d->T)) ||
        (rc = check_tensor("v", v, d->v_stride, p.esize, d->T)) || (rc = check_out("out", out, d->o_stride, p.esize, d)) ||
        (rc = check_den("den", den)))
        return rc;
    if (!planes) return fail(RACE_E_INVALID, "planes is NULL");
    if (!state) return fail(RACE_E_INVALID, "state is NULL");
    if (!ws || ws_bytes < p.gfws)
        return fail(RACE_E_WORKSPACE, "workspace %zu bytes < required %zu", ws_bytes, p.gfws);
    Args a = base_args(d, p, planes);
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.den = den;
    a.fstate = (double *)state;
    a.fdelta = (double *)ws;
    a.opart = p.parts ? (void *)((char *)ws + p.fws_core) : nullptr;
    a.denpart = p.parts ? (float *)((char *)ws + p.fws) : nullptr;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return gn_fwd_dispatch<bf16>(d, p, a, s);
    return gn_fwd_dispatch<float>(d, p, a, s);
}

int race_bwd_global(const race_desc *d, const void *q, const void *k, const void *v, const float *planes,
                    const void *out, const float *den, const void *dout, const float *dden, const void *state,
                    void *dq, void *dk, void *dv, float *grad_beta, void *ws, size_t ws_bytes, void *stream) {
    Plan p;
    int rc = make_plan(d, p, true);
    if (rc || (rc = check_gn(d))) return rc;
    if ((rc = check_tensor("q", q, d->q_stride, p.esize, d->T)) || (rc = check_tensor("k", k, d->k_stride, p.esize, d->T)) ||
        (rc = check_tensor("v", v, d->v_stride, p.esize, d->T)) ||
        (rc = check_tensor("out", out, d->o_stride, p.esize, d->T)) ||
        (rc = check_tensor("dout", dout, d->do_stride, p.esize, d->T)) ||
        (rc = check_out("dq", dq, d->g_stride, p.esize, d)) || (rc = check_out("dk", dk, d->g_stride, p.esize, d)) ||
        (rc = check_out("dv", dv, d->g_stride, p.esize, d)) || (rc = check_den("den", den)) ||
        (dden && (rc = check_den("dden", dden))))
        return rc;
    if (!planes) return fail(RACE_E_INVALID, "planes is NULL");
    if (!state) return fail(RACE_E_INVALID, "state is NULL");
    if (!ws || ws_bytes < p.gbws)
        return fail(RACE_E_WORKSPACE, "workspace %zu bytes < required %zu", ws_bytes, p.gbws);
    Args a = base_args(d, p, planes);
    a.q = q;
    a.k = k;
    a.v = v;
    a.dout = dout;
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.fstate = (double *)state;
    const size_t blk = (size_t)p.N * p.nseg * p.Spad * SROW;
    a.rdelta = (float *)ws;
    a.rstate = a.rdelta + blk;
    a.tpart = (double *)(a.rstate + blk);  // blk is even: 8-byte aligned
    if (p.parts) {
        float *part = (float *)((char *)ws + p.bws_core);
        a.dqpart = part;
        a.dkpart = (char *)part + p.xpart_bytes;
        a.dvpart = (char *)part + 2 * p.xpart_bytes;
    }
    a.out = const_cast<void *>(out);  // read only (the GN per-token terms)
    a.den = const_cast<float *>(den);
    a.dden = dden;
    a.rden = (float *)((char *)ws + p.bws);
    a.gden = (float *)((char *)ws + p.bws + p.tok_bytes);
    a.gsum = p.parts ? (float *)((char *)ws + p.bws + 2 * p.tok_bytes) : nullptr;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return gn_bwd_dispatch<bf16>(d, p, a, grad_beta, s);
    return gn_bwd_dispatch<float>(d, p, a, grad_beta, s);
}

size_t race_prefix_mean_workspace_bytes(int64_t NS, int64_t T, int64_t D) {
    if (NS < 1 || T < 1 || D < 1) return 0;
    // the arrays' alignment, which picks the kernels, is not known here: room for either
    return cmax(pm_workspace(NS, T, D, false), pm_workspace(NS, T, D, true));
}

int race_prefix_mean_fwd(const float *w, const float *v, float *E, int64_t NS, int64_t T, int64_t D, double eps,
                         void *ws, size_t ws_bytes, void *stream) {
    int rc;
    if ((rc = pm_check(w, "w", NS, T, D)) || (rc = pm_check(v, "v", NS, T, D)) || (rc = pm_check(E, "E", NS, T, D)))
        return rc;
    const size_t need = race_prefix_mean_workspace_bytes(NS, T, D);
    if (!ws || ws_bytes < need) return fail(RACE_E_WORKSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
    const bool rows = pm_rows(D, v, E, nullptr, nullptr);
    const int64_t tseg = pm_tseg(NS, T, rows);
    const int nseg = (int)((T + tseg - 1) / tseg);
    double *delta = (double *)ws;
    double *state = delta + NS * nseg * (D + 1);
    hipStream_t s = (hipStream_t)stream;
    const int elems = (int)(D + 1);
    const dim3 grid(nseg, (unsigned)NS), rgrid((unsigned)((NS * pm4_stride(nseg) + PM4_ROWS - 1) / PM4_ROWS)),
        sgrid((elems + PM_SCAN_THREADS - 1) / PM_SCAN_THREADS, (unsigned)NS);
    if (rows)
        k_pm4_reduce<<<rgrid, 16 * PM4_ROWS, 0, s>>>(w, v, delta, NS, T, (int)D, tseg, nseg);
    else
        k_pm_reduce<<<grid, 64, 0, s>>>(w, v, delta, T, (int)D, tseg, nseg);
    k_pm_scan<<<sgrid, PM_SCAN_THREADS, 0, s>>>(state, delta, nseg, elems);
    if (rows)
        k_pm4_out<<<rgrid, 16 * PM4_ROWS, 0, s>>>(w, v, E, state, NS, T, (int)D, tseg, nseg, eps);
    else
        k_pm_out<<<grid, 64, 0, s>>>(w, v, E, state, T, (int)D, tseg, nseg, eps);
    return launched("race_prefix_mean_fwd");
}

int race_prefix_mean_bwd(const float *w, const float *v, const float *gE, float *gW, float *gV, int64_t NS,
                         int64_t T, int64_t D, double eps, void *ws, size_t ws_bytes, void *stream) {
    int rc;
    if ((rc = pm_check(w, "w", NS, T, D)) || (rc = pm_check(v, "v", NS, T, D)) ||
        (rc = pm_check(gE, "gE", NS, T, D)) || (rc = pm_check(gW, "gW", NS, T, D)) ||
        (rc = pm_check(gV, "gV", NS, T, D)))
        return rc;
    const size_t need = race_prefix_mean_workspace_bytes(NS, T, D);
    if (!ws || ws_bytes < need) return fail(RACE_E_WORKSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
    const bool rows = pm_rows(D, v, gE, gV, nullptr);
    const int64_t tseg = pm_tseg(NS, T, rows);
    const int nseg = (int)((T + tseg - 1) / tseg);
    double *delta = (double *)ws;
    double *state = delta + NS * nseg * (D + 1);
    double *invA = state + NS * (nseg + 1) * (D + 1);
    double *alpha = invA + NS * T;
    double *rdelta = alpha + NS * T;
    double *rstate = rdelta + NS * nseg * (D + 1);
    hipStream_t s = (hipStream_t)stream;
    const int elems = (int)(D + 1);
    const dim3 grid(nseg, (unsigned)NS), rgrid((unsigned)((NS * pm4_stride(nseg) + PM4_ROWS - 1) / PM4_ROWS)),
        sgrid((elems + PM_SCAN_THREADS - 1) / PM_SCAN_THREADS, (unsigned)NS);
    if (rows)
        k_pm4_reduce<<<rgrid, 16 * PM4_ROWS, 0, s>>>(w, v, delta, NS, T, (int)D, tseg, nseg);
    else
        k_pm_reduce<<<grid, 64, 0, s>>>(w, v, delta, T, (int)D, tseg, nseg);
    k_pm_scan<<<sgrid, PM_SCAN_THREADS, 0, s>>>(state, delta, nseg, elems);
    if (rows)
        k_pm4_bw_fwd<<<rgrid, 16 * PM4_ROWS, 0, s>>>(w, v, gE, state, invA, alpha, rdelta, NS, T, (int)D, tseg, nseg, eps);
    else
        k_pm_bw_fwd<<<grid, 64, 0, s>>>(w, v, gE, state, invA, alpha, rdelta, T, (int)D, tseg, nseg, eps);
    k_pm_rscan<<<sgrid, PM_SCAN_THREADS, 0, s>>>(rstate, rdelta, nseg, elems);
    if (rows)
        k_pm4_bw_rev<<<rgrid, 16 * PM4_ROWS, 0, s>>>(w, v, gE, invA, alpha, rstate, gW, gV, NS, T, (int)D, tseg, nseg);
    else
        k_pm_bw_rev<<<grid, 64, 0, s>>>(w, v, gE, invA, alpha, rstate, gW, gV, T, (int)D, tseg, nseg);
    return launched("race_prefix_mean_bwd");
}

int race_fwd_noalloc(const race_desc *d, const void *q, const void *k, const void *v, const float *planes,
                     void *out, void *stream) {
    race_desc dd;
    Plan p;
    int rc = noalloc_plan(d, dd, p);
    if (rc) return rc;
    if ((rc = check_tensor("q", q, d->q_stride, p.esize, d->T)) || (rc = check_tensor("k", k, d->k_stride, p.esize, d->T)) ||
        (rc = check_tensor("v", v, d->v_stride, p.esize, d->T)) || (rc = check_out("out", out, d->o_stride, p.esize, d)))
        return rc;
    if (!planes) return fail(RACE_E_INVALID, "planes is NULL");
    void *base = nullptr;
    if ((rc = scratch_address(&base))) return rc;
    Args a = base_args(&dd, p, planes);
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.fstate = (double *)base;
    a.fdelta = (double *)((char *)base + align256(p.state_bytes));
    a.opart = p.parts ? (void *)((char *)a.fdelta + p.fws_core) : nullptr;
    hipStream_t s = (hipStream_t)stream;
    if (d->dtype == RACE_DTYPE_BF16) return fwd_dispatch<bf16>(&dd, p, a, s);
    return fwd_dispatch<float>(&dd, p, a, s);
}

int race_inv_temp(const float *logit, float lo, float hi, float *out, void *stream) {
    int rc;
    if ((rc = check_den("logit", logit)) || (rc = check_den("out", out))) return rc;
    if (!(lo > 0.f) || !(hi >= lo)) return fail(RACE_E_INVALID, "bounds must be 0 < lo <= hi (got %g, %g)", lo, hi);
    k_inv_temp<<<1, 64, 0, (hipStream_t)stream>>>(logit, lo, hi, out);
    return launched("race_inv_temp");
}

const char *race_last_error(void) { return g_err.c_str(); }

int race_abi_version(void) { return 3; }

} // extern "C"
