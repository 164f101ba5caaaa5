// prefix_mean.hip -- gfx950 kernels of the flat causal prefix mean, the
// operator of the reference CPU extension (kernels/cpu/race_pref.cpp:36-220):
//   E[n,t,:] = B_t / (A_t + eps),  A_t = sum_{tau<=t} w,  B_t = sum_{tau<=t} w v
// and its backward.  Accumulation is fp64 as in the reference.  Streams are
// split into token segments; a three-phase scan (segment sums, segment
// prefix, per-segment walk) carries (A, B) across segments.
//
// Two sets of kernels.  k_pm4_*: D <= 64 in whole 16-byte pieces, 16-byte
// aligned arrays; one 16-lane row per (segment, stream), lane l owns columns
// 4l .. 4l+3, and the row's lanes share the per-token scalars of 16 tokens at a
// time.  k_pm_*: any D <= 512 and alignment; one 64-lane wave per (segment,
// stream), lane l owns columns l, l+64, ...
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "race_device.h"

namespace race {

constexpr int PM_MAXC = 8;  // columns per lane -> D <= 512

__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

// per-segment sums of (B, A): delta[ns][seg][0..D) = B, [D] = A
__global__ __launch_bounds__(64) void k_pm_reduce(const float *__restrict__ w, const float *__restrict__ v,
                                                  double *__restrict__ delta, int64_t T, int D, int64_t tseg,
                                                  int nseg) {
    const int64_t ns = blockIdx.y;
    const int seg = blockIdx.x, lane = threadIdx.x;
    const int64_t t0 = seg * tseg, t1 = min(T, t0 + tseg);
    double B[PM_MAXC], A = 0.0;
    for (int c = 0; c < PM_MAXC; ++c) B[c] = 0.0;
    for (int64_t t = t0; t < t1; ++t) {
        const double wt = (double)w[ns * T + t];
        A += wt;
        const float *vt = v + (ns * T + t) * D;
        for (int c = 0; c < PM_MAXC; ++c) {
            const int d = lane + 64 * c;
            if (d < D) B[c] += wt * (double)vt[d];
        }
    }
    double *o = delta + (ns * nseg + seg) * (int64_t)(D + 1);
    for (int c = 0; c < PM_MAXC; ++c) {
        const int d = lane + 64 * c;
        if (d < D) o[d] = B[c];
    }
    if (lane == 0) o[D] = A;
}

// forward walk: E (race_pref.cpp:82-98 order: A += w; inv; B += w v; E = B inv)
__global__ __launch_bounds__(64) void k_pm_out(const float *__restrict__ w, const float *__restrict__ v,
                                               float *__restrict__ E, const double *__restrict__ state, int64_t T,
                                               int D, int64_t tseg, int nseg, double eps) {
    const int64_t ns = blockIdx.y;
    const int seg = blockIdx.x, lane = threadIdx.x;
    const int64_t t0 = seg * tseg, t1 = min(T, t0 + tseg);
    const double *st = state + (ns * (nseg + 1) + seg) * (int64_t)(D + 1);
    double B[PM_MAXC], A = st[D];
    for (int c = 0; c < PM_MAXC; ++c) B[c] = (lane + 64 * c < D) ? st[lane + 64 * c] : 0.0;
    for (int64_t t = t0; t < t1; ++t) {
        const double wt = (double)w[ns * T + t];
        A += wt;
        const double inv = 1.0 / (A + eps);
        const float *vt = v + (ns * T + t) * D;
        float *et = E + (ns * T + t) * D;
        for (int c = 0; c < PM_MAXC; ++c) {
            const int d = lane + 64 * c;
            if (d < D) {
                B[c] += wt * (double)vt[d];
                et[d] = (float)(B[c] * inv);
            }
        }
    }
}

// backward pass 1 (forward walk, race_pref.cpp:161-182): invA[t], alpha[t];
// per-segment sums rdelta[..][0..D) = sum g invA, [D] = sum alpha
__global__ __launch_bounds__(64) void k_pm_bw_fwd(const float *__restrict__ w, const float *__restrict__ v,
                                                  const float *__restrict__ gE, const double *__restrict__ state,
                                                  double *__restrict__ invA, double *__restrict__ alpha,
                                                  double *__restrict__ rdelta, int64_t T, int D, int64_t tseg,
                                                  int nseg, double eps) {
    const int64_t ns = blockIdx.y;
    const int seg = blockIdx.x, lane = threadIdx.x;
    const int64_t t0 = seg * tseg, t1 = min(T, t0 + tseg);
    const double *st = state + (ns * (nseg + 1) + seg) * (int64_t)(D + 1);
    double B[PM_MAXC], bsum[PM_MAXC], A = st[D], asum = 0.0;
    for (int c = 0; c < PM_MAXC; ++c) {
        B[c] = (lane + 64 * c < D) ? st[lane + 64 * c] : 0.0;
        bsum[c] = 0.0;
    }
    for (int64_t t = t0; t < t1; ++t) {
        const double wt = (double)w[ns * T + t];
        A += wt;
        const float *vt = v + (ns * T + t) * D;
        const float *gt = gE + (ns * T + t) * D;
        double dot = 0.0;
        for (int c = 0; c < PM_MAXC; ++c) {
            const int d = lane + 64 * c;
            if (d < D) {
                B[c] += wt * (double)vt[d];
                dot += (double)gt[d] * B[c];
            }
        }
        dot = wave_sum(dot);
        const double iA = 1.0 / (A + eps);
        const double al = -(iA * iA) * dot;
        if (lane == 0) {
            invA[ns * T + t] = iA;
            alpha[ns * T + t] = al;
        }
        asum += al;
        for (int c = 0; c < PM_MAXC; ++c) {
            const int d = lane + 64 * c;
            if (d < D) bsum[c] += (double)gt[d] * iA;
        }
    }
    double *o = rdelta + (ns * nseg + seg) * (int64_t)(D + 1);
    for (int c = 0; c < PM_MAXC; ++c) {
        const int d = lane + 64 * c;
        if (d < D) o[d] = bsum[c];
    }
    if (lane == 0) o[D] = asum;
}

// backward pass 2 (reverse walk, race_pref.cpp:188-216): gW, gV
__global__ __launch_bounds__(64) void k_pm_bw_rev(const float *__restrict__ w, const float *__restrict__ v,
                                                  const float *__restrict__ gE, const double *__restrict__ invA,
                                                  const double *__restrict__ alpha,
                                                  const double *__restrict__ rstate, float *__restrict__ gW,
                                                  float *__restrict__ gV, int64_t T, int D, int64_t tseg,
                                                  int nseg) {
    const int64_t ns = blockIdx.y;
    const int seg = blockIdx.x, lane = threadIdx.x;
    const int64_t t0 = seg * tseg, t1 = min(T, t0 + tseg);
    const double *rs = rstate + (ns * nseg + seg) * (int64_t)(D + 1);
    double beta[PM_MAXC], asuf = rs[D];
    for (int c = 0; c < PM_MAXC; ++c) beta[c] = (lane + 64 * c < D) ? rs[lane + 64 * c] : 0.0;
    for (int64_t t = t1 - 1; t >= t0; --t) {
        const double iA = invA[ns * T + t];
        const float *vt = v + (ns * T + t) * D;
        const float *gt = gE + (ns * T + t) * D;
        float *gvt = gV + (ns * T + t) * D;
        asuf += alpha[ns * T + t];
        const double wt = (double)w[ns * T + t];
        double dot = 0.0;
        for (int c = 0; c < PM_MAXC; ++c) {
            const int d = lane + 64 * c;
            if (d < D) {
                beta[c] += (double)gt[d] * iA;
                dot += beta[c] * (double)vt[d];
                gvt[d] = (float)(wt * beta[c]);
            }
        }
        dot = wave_sum(dot);
        if (lane == 0) gW[ns * T + t] = (float)(asuf + dot);
    }
}

// ------------------------------------------------------------ k_pm4_*
// Bound by memory: the walks read 256-byte rows of v (and gE) and write rows of
// E (gV), a few fp64 operations a byte.  What kept the one-wave walks above at a
// fifth of that is one token's load in flight at a time and, per token, a
// division and a 64-lane fp64 sum in every lane.  Here a row of 16 lanes walks a
// segment 16 tokens at a time: the 16 tokens' loads are issued together, lane j
// holds token j's scalars (A by a scan over the lanes, one division per token),
// and a token's sum over columns is 4 DPP steps.  128 streams x 4096 tokens, D =
// 64, MI355X, us: segment sums 69 -> 24, E 85 -> 46, backward's forward walk 179
// -> 61, reverse walk 177 -> 75: 4.4 to 5.8 TB/s, a large copy's 5.1 (part of v
// stays in the last-level cache between the walks).
constexpr int PM4_ROWS = 16;  // 16-lane rows (segments) per 256-thread workgroup

// lane J of each 16-lane row, in every lane of the row
template <int J> __device__ __forceinline__ float row_lane(float x) { return dpp_f<0x150 + J>(x); }
template <int J> __device__ __forceinline__ double row_lane(double x) { return dpp_d<0x150 + J>(x); }
__device__ __forceinline__ double row_prefix_f64(double x) {
    x += dpp_d<0x111>(x);
    x += dpp_d<0x112>(x);
    x += dpp_d<0x114>(x);
    x += dpp_d<0x118>(x);
    return x;
}
__device__ __forceinline__ double row_suffix_f64(double x) {
    x += dpp_d<0x101>(x);
    x += dpp_d<0x102>(x);
    x += dpp_d<0x104>(x);
    x += dpp_d<0x108>(x);
    return x;
}
// f(integral_constant j) for the tokens j = J0 .. J0+N-1 of 16, or the other way round
template <int J0, int N, bool REV, int J = 0, typename F> __device__ __forceinline__ void each(F &&f) {
    if constexpr (J < N) {
        f(std::integral_constant<int, J0 + (REV ? N - 1 - J : J)>{});
        each<J0, N, REV, J + 1>(f);
    }
}

struct Pm4Pos {
    int64_t ns, t0, t1;  // stream, the segment's tokens
    int seg, l;          // segment; lane in its row (columns 4l ..)
    bool live, col;      // the segment exists; the lane has columns
};
// Rows are numbered over (stream, segment), so that a workgroup's rows all work
// where streams are many and segments few (backward, 16384 x 197, us: segments of
// one stream 4729, these 1092, a wave per segment 1606).  From 4 segments on a
// stream's rows start a new wave: the shorter last segment holds up one wave of a
// stream's, not the next stream's rows too (128 x 197, 13 segments: 26.9 us, not
// 29.4).
__host__ __device__ __forceinline__ int pm4_stride(int nseg) { return nseg < 4 ? nseg : (nseg + 3) / 4 * 4; }
__device__ __forceinline__ Pm4Pos pm4_pos(int64_t NS, int64_t T, int D, int64_t tseg, int nseg) {
    Pm4Pos p;
    const uint32_t row = blockIdx.x * PM4_ROWS + (threadIdx.x >> 4);
    const uint32_t stride = (uint32_t)pm4_stride(nseg);
    p.ns = row / stride;
    p.seg = (int)(row % stride);
    p.l = threadIdx.x & 15;
    p.live = p.ns < NS && p.seg < nseg;
    p.col = 4 * p.l < D;
    p.t0 = p.seg * tseg;
    p.t1 = min(T, p.t0 + tseg);
    return p;
}
// the lane's 4 columns of tokens c .. c+N-1 (zeros past the segment's end and for a lane without columns)
template <int N>
__device__ __forceinline__ void pm4_rows(const float *__restrict__ x, const Pm4Pos &p, int64_t c, int64_t T, int D,
                                         f32x4 (&r)[N]) {
    const float *base = x + (p.ns * T + c) * D + 4 * p.l;
    if (c + N <= p.t1) {
#pragma unroll
        for (int j = 0; j < N; ++j) r[j] = p.col ? *reinterpret_cast<const f32x4 *>(base + j * D) : zero4();
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j)
            r[j] = p.col && c + j < p.t1 ? *reinterpret_cast<const f32x4 *>(base + j * D) : zero4();
    }
}

__global__ __launch_bounds__(256) void k_pm4_reduce(const float *__restrict__ w, const float *__restrict__ v,
                                                    double *__restrict__ delta, int64_t NS, int64_t T, int D,
                                                    int64_t tseg, int nseg) {
    const Pm4Pos p = pm4_pos(NS, T, D, tseg, nseg);
    if (!p.live) return;  // whole rows
    double B[4] = {0.0, 0.0, 0.0, 0.0}, A = 0.0;
    for (int64_t c = p.t0; c < p.t1; c += 16) {
        f32x4 x[16];
        const float wl = c + p.l < p.t1 ? w[p.ns * T + c + p.l] : 0.f;
        pm4_rows(v, p, c, T, D, x);
        A += (double)wl;
        each<0, 16, false>([&](auto J) {
            const double wt = (double)row_lane<J>(wl);
#pragma unroll
            for (int e = 0; e < 4; ++e) B[e] += wt * (double)x[J][e];
        });
    }
    A = row_sum_f64(A);
    double *o = delta + (p.ns * nseg + p.seg) * (int64_t)(D + 1);
    if (p.col)
        for (int e = 0; e < 4; ++e) o[4 * p.l + e] = B[e];
    if (p.l == 0) o[D] = A;
}

__global__ __launch_bounds__(256) void k_pm4_out(const float *__restrict__ w, const float *__restrict__ v,
                                                 float *__restrict__ E, const double *__restrict__ state, int64_t NS,
                                                 int64_t T, int D, int64_t tseg, int nseg, double eps) {
    const Pm4Pos p = pm4_pos(NS, T, D, tseg, nseg);
    if (!p.live) return;
    const double *st = state + (p.ns * (nseg + 1) + p.seg) * (int64_t)(D + 1);
    double B[4], A = st[D];
    for (int e = 0; e < 4; ++e) B[e] = p.col ? st[4 * p.l + e] : 0.0;
    for (int64_t c = p.t0; c < p.t1; c += 16) {
        f32x4 x[16];
        const float wl = c + p.l < p.t1 ? w[p.ns * T + c + p.l] : 0.f;
        pm4_rows(v, p, c, T, D, x);
        const double Al = A + row_prefix_f64((double)wl);
        const double inv = 1.0 / (Al + eps);
        A = row_lane<15>(Al);
        float *base = E + (p.ns * T + c) * D + 4 * p.l;
        each<0, 16, false>([&](auto J) {
            const double wt = (double)row_lane<J>(wl), iv = row_lane<J>(inv);
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                B[e] += wt * (double)x[J][e];
                o[e] = (float)(B[e] * iv);
            }
            if (p.col && c + J < p.t1) *reinterpret_cast<f32x4 *>(base + J * D) = o;
        });
    }
}

// backward pass 1 (as k_pm_bw_fwd)
__global__ __launch_bounds__(256) void k_pm4_bw_fwd(const float *__restrict__ w, const float *__restrict__ v,
                                                    const float *__restrict__ gE, const double *__restrict__ state,
                                                    double *__restrict__ invA, double *__restrict__ alpha,
                                                    double *__restrict__ rdelta, int64_t NS, int64_t T, int D,
                                                    int64_t tseg, int nseg, double eps) {
    const Pm4Pos p = pm4_pos(NS, T, D, tseg, nseg);
    if (!p.live) return;
    const double *st = state + (p.ns * (nseg + 1) + p.seg) * (int64_t)(D + 1);
    double B[4], bsum[4] = {0.0, 0.0, 0.0, 0.0}, A = st[D], asum = 0.0;
    for (int e = 0; e < 4; ++e) B[e] = p.col ? st[4 * p.l + e] : 0.0;
    for (int64_t c = p.t0; c < p.t1; c += 16) {
        const bool tv = c + p.l < p.t1;
        const float wl = tv ? w[p.ns * T + c + p.l] : 0.f;
        const double Al = A + row_prefix_f64((double)wl);
        const double inv = 1.0 / (Al + eps);
        A = row_lane<15>(Al);
        double dl = 0.0;  // lane j: token j's g . B
        auto half = [&](auto H) {  // 8 tokens' rows of both arrays at a time (registers)
            f32x4 x[8], g[8];
            pm4_rows(v, p, c + H, T, D, x);
            pm4_rows(gE, p, c + H, T, D, g);
            each<H, 8, false>([&](auto J) {
                const double wt = (double)row_lane<J>(wl), iv = row_lane<J>(inv);
                double dot = 0.0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    B[e] += wt * (double)x[J - H][e];
                    dot += (double)g[J - H][e] * B[e];
                    if (c + J < p.t1) bsum[e] += (double)g[J - H][e] * iv;  // (inv may be infinite or NaN past the end)
                }
                dot = row_sum_f64(dot);
                dl = p.l == J ? dot : dl;
            });
        };
        half(std::integral_constant<int, 0>{});
        half(std::integral_constant<int, 8>{});
        if (tv) {
            const double al = -(inv * inv) * dl;
            invA[p.ns * T + c + p.l] = inv;
            alpha[p.ns * T + c + p.l] = al;
            asum += al;
        }
    }
    asum = row_sum_f64(asum);
    double *o = rdelta + (p.ns * nseg + p.seg) * (int64_t)(D + 1);
    if (p.col)
        for (int e = 0; e < 4; ++e) o[4 * p.l + e] = bsum[e];
    if (p.l == 0) o[D] = asum;
}

// backward pass 2 (as k_pm_bw_rev)
__global__ __launch_bounds__(256) void k_pm4_bw_rev(const float *__restrict__ w, const float *__restrict__ v,
                                                    const float *__restrict__ gE, const double *__restrict__ invA,
                                                    const double *__restrict__ alpha,
                                                    const double *__restrict__ rstate, float *__restrict__ gW,
                                                    float *__restrict__ gV, int64_t NS, int64_t T, int D, int64_t tseg,
                                                    int nseg) {
    const Pm4Pos p = pm4_pos(NS, T, D, tseg, nseg);
    if (!p.live) return;
    const double *rs = rstate + (p.ns * nseg + p.seg) * (int64_t)(D + 1);
    double beta[4], asuf = rs[D];
    for (int e = 0; e < 4; ++e) beta[e] = p.col ? rs[4 * p.l + e] : 0.0;
    const int64_t last = p.t0 + (p.t1 - 1 - p.t0) / 16 * 16;
    for (int64_t c = last; c >= p.t0; c -= 16) {
        const bool tv = c + p.l < p.t1;
        const int64_t tl = p.ns * T + c + p.l;
        const float wl = tv ? w[tl] : 0.f;
        const double il = tv ? invA[tl] : 0.0, sl = asuf + row_suffix_f64(tv ? alpha[tl] : 0.0);
        asuf = row_lane<0>(sl);
        double dl = 0.0;  // lane j: token j's beta . v
        float *base = gV + (p.ns * T + c) * D + 4 * p.l;
        auto half = [&](auto H) {
            f32x4 x[8], g[8];
            pm4_rows(v, p, c + H, T, D, x);
            pm4_rows(gE, p, c + H, T, D, g);
            each<H, 8, true>([&](auto J) {
                const double wt = (double)row_lane<J>(wl), iv = row_lane<J>(il);
                double dot = 0.0;
                f32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    beta[e] += (double)g[J - H][e] * iv;
                    dot += beta[e] * (double)x[J - H][e];
                    o[e] = (float)(wt * beta[e]);
                }
                if (p.col && c + J < p.t1) *reinterpret_cast<f32x4 *>(base + J * D) = o;
                dot = row_sum_f64(dot);
                dl = p.l == J ? dot : dl;
            });
        };
        half(std::integral_constant<int, 8>{});
        half(std::integral_constant<int, 0>{});
        if (tv) gW[tl] = (float)(sl + dl);
    }
}

// Segment scans (both sets of kernels): exclusive prefix state[ns][seg] (seg <=
// nseg) and exclusive suffix rstate[ns][seg]; the loads of PM_BATCH segments are
// issued together.
constexpr int PM_BATCH = 16, PM_SCAN_THREADS = 64;
__global__ __launch_bounds__(PM_SCAN_THREADS) void k_pm_scan(double *state, const double *delta, int nseg, int elems) {
    const int64_t ns = blockIdx.y;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= elems) return;
    const double *src = delta + ns * nseg * elems + e;
    double *dst = state + ns * (nseg + 1) * elems + e;
    double acc = 0.0;
    int s = 0;
    for (; s + PM_BATCH <= nseg; s += PM_BATCH) {
        double x[PM_BATCH];
#pragma unroll
        for (int j = 0; j < PM_BATCH; ++j) x[j] = src[(int64_t)(s + j) * elems];
#pragma unroll
        for (int j = 0; j < PM_BATCH; ++j) {
            dst[(int64_t)(s + j) * elems] = acc;
            acc += x[j];
        }
    }
    for (; s < nseg; ++s) {
        const double x = src[(int64_t)s * elems];
        dst[(int64_t)s * elems] = acc;
        acc += x;
    }
    dst[(int64_t)nseg * elems] = acc;
}
__global__ __launch_bounds__(PM_SCAN_THREADS) void k_pm_rscan(double *rstate, const double *rdelta, int nseg,
                                                              int elems) {
    const int64_t ns = blockIdx.y;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= elems) return;
    const double *src = rdelta + ns * nseg * elems + e;
    double *dst = rstate + ns * nseg * elems + e;
    double acc = 0.0;
    int s = nseg;
    for (; s >= PM_BATCH; s -= PM_BATCH) {
        double x[PM_BATCH];
#pragma unroll
        for (int j = 0; j < PM_BATCH; ++j) x[j] = src[(int64_t)(s - 1 - j) * elems];
#pragma unroll
        for (int j = 0; j < PM_BATCH; ++j) {
            dst[(int64_t)(s - 1 - j) * elems] = acc;
            acc += x[j];
        }
    }
    for (; s > 0; --s) {
        const double x = src[(int64_t)(s - 1) * elems];
        dst[(int64_t)(s - 1) * elems] = acc;
        acc += x;
    }
}

} // namespace race
