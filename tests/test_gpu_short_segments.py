"""Segment plans of short and medium sequences, and the totals of the
non-causal scans.

Plans (CPU, from the library's buffer sizes): a sequence whose automatic
segments would be short runs about as many workgroups as are resident at once,
never more than the 256-tile walk bound a segment; up to 1024 tiles in all keep
one-tile segments; the causal backward's segments are whole forward ones, the
non-causal one's its own.

Totals (GPU): four waves share a stream's segments; segment counts around the
waves and the 16-load batches, against the fp64 oracle with the parity bars."""
import ctypes

import pytest
import torch

from helpers import TOL, compare, make_case, run_gpu, run_oracle


def _segments(B, T, H, K, L, dtype, causal=1):
    import bench
    from race_attention_amd import _lib
    d = _lib.RaceDesc()
    d.M, d.B, d.T, d.H, d.D, d.L, d.K = 1, B, T, H, 64, L, K
    d.causal, d.dtype, d.eps, d.inv_temp = causal, dtype, 1e-6, 0.125
    lib = _lib.load()
    sb, bw = lib.race_state_bytes(ctypes.byref(d)), lib.race_bwd_workspace_bytes(ctypes.byref(d))
    return bench.scan_bytes(sb, bw, B * H, T, L, K)[2:]


@pytest.mark.parametrize("B,T,H,K,L,fnseg,nseg", [
    (2, 16384, 8, 4, 8, 32, 16),     # 512 forward workgroups, 256 backward ones
    (1, 262001, 8, 4, 8, 64, 32),    # the same, of 128 and 256 tiles
    (1, 1 << 20, 8, 4, 8, 256, 128),  # long: 2048 and 1024
    (4, 4001, 12, 3, 8, 16, 16),     # 64 buckets: 768
    (1, 8192, 4, 4, 8, 256, 64),     # 1024 tiles: one-tile forward segments
    (1, 20, 1, 4, 8, 1, 1),
])
def test_short_sequence_plans(B, T, H, K, L, fnseg, nseg):
    from race_attention_amd import _lib
    assert _segments(B, T, H, K, L, _lib.RACE_DTYPE_BF16) == (fnseg, nseg)


def test_plans_cover_the_sequence_within_the_walk_bound():
    from race_attention_amd import _lib
    for causal in (0, 1):
        for B, H in ((1, 1), (1, 4), (2, 12), (64, 6)):
            for K, L in ((2, 5), (4, 4), (4, 8), (8, 4)):
                for T in (1, 33, 785, 1024, 4097, 30000, 250001):
                    f, b = _segments(B, T, H, K, L, _lib.RACE_DTYPE_BF16, causal)
                    ntiles = -(-T // 32)
                    assert 1 <= b <= f <= ntiles
                    assert -(-ntiles // f) <= 256 and (ntiles <= 256 or -(-ntiles // b) <= 256), (B, H, K, L, T, f, b)


def _plan(B, T, H, K, L, dtype, causal):
    """(forward segments, backward segments) at any K and dtype: what does not
    depend on the segments is taken from a plan of explicit ones."""
    from race_attention_amd import _lib
    lib, N, ntiles = _lib.load(), B * H, -(-T // 32)
    nslice = 1 if K <= 4 else -(-(L << K) // (128 if dtype == _lib.RACE_DTYPE_BF16 else 32))

    def sizes(seg_tiles):
        d = _lib.RaceDesc()
        d.M, d.B, d.T, d.H, d.D, d.L, d.K = 1, B, T, H, 64, L, K
        d.causal, d.dtype, d.eps, d.inv_temp, d.seg_tiles = causal, dtype, 1e-6, 0.125, seg_tiles
        return lib.race_state_bytes(ctypes.byref(d)), lib.race_bwd_workspace_bytes(ctypes.byref(d))

    tiles = min(ntiles, 256)
    known = -(-ntiles // tiles)
    sb, bw = sizes(tiles)
    row = sb // (known + 1)                # fp64 bytes of one segment of all streams
    core = lambda n: n * row + (16 * N * n * nslice + 15) // 16 * 16  # noqa: E731  (two fp32 rows a segment)
    fixed = bw - core(known)
    sb, bw = sizes(0)
    nseg = (bw - fixed) // (row + 16 * N * nslice)
    assert sb % row == 0 and bw == core(nseg) + fixed
    return sb // row - 1, nseg


@pytest.mark.parametrize("N,T,K,L,causal", [
    (48, 8192, 6, 5, 1), (48, 8192, 7, 4, 1),  # 3 and 4 slices
    (96, 1000, 6, 5, 1),                       # the forward leaves the backward a choice
    (7, 47355, 6, 5, 1),                       # groups of 3 slices that no 8 XCDs divide
    (48, 8192, 6, 5, 0), (96, 1000, 6, 5, 0),
])
def test_sliced_backward_takes_about_the_tiles_it_has(N, T, K, L, causal):
    """One workgroup of 128 buckets per CU: whole rounds of the longest segment,
    on the XCD with the most workgroups, within 35% of an even split."""
    from race_attention_amd import _lib
    f, b = _plan(1, T, N, K, L, _lib.RACE_DTYPE_BF16, causal)
    ntiles, nslice = -(-T // 32), -(-(L << K) // 128)
    longest = -(-f // b) * -(-ntiles // f) if causal else -(-ntiles // b)
    rounds = -(-(-(-b * N // 8) * nslice) // 32)
    assert rounds * longest <= 1.35 * ntiles * N * nslice / 256, (f, b, rounds, longest)


@pytest.mark.parametrize("B,T,H,K,L,fnseg,nseg", [
    (1, 8192, 8, 4, 8, 32, 32),    # 8 tiles for each of 256 workgroups of 128 buckets: one residency
    (1, 8160, 8, 4, 8, 64, 32),    # 8 tiles fewer: two rounds, joined in pairs
    (1, 8192, 8, 3, 10, 32, 32),   # 80 of 128 buckets
    (1, 262001, 8, 4, 8, 32, 32),  # segments of 256 tiles, the longest
    (4, 4001, 12, 3, 8, 10, 10),   # 64 buckets: 512
    (1, 8192, 4, 4, 8, 256, 64),   # 1024 tiles: one-tile forward segments
    (2, 4096, 8, 8, 1, 4, 4),      # 8 slices of 32 buckets
    (1, 20, 1, 4, 8, 1, 1),
])
def test_fp32_plans(B, T, H, K, L, fnseg, nseg):
    from race_attention_amd import _lib
    assert _plan(B, T, H, K, L, _lib.RACE_DTYPE_F32, 1) == (fnseg, nseg)


def test_all_plans_cover_the_sequence_within_the_walk_bound():
    from race_attention_amd import _lib
    for dtype in (_lib.RACE_DTYPE_F32, _lib.RACE_DTYPE_BF16):
        for causal in (0, 1):
            for B, H in ((1, 1), (1, 4), (2, 12), (12, 8), (64, 6)):
                for K, L in ((2, 5), (3, 8), (3, 10), (4, 6), (4, 8), (5, 6), (6, 5), (8, 4)):
                    for T in (1, 33, 785, 4097, 8160, 30000, 250001):
                        f, b = _plan(B, T, H, K, L, dtype, causal)
                        ntiles = -(-T // 32)
                        assert 1 <= b <= f <= ntiles, (dtype, causal, B, H, K, L, T, f, b)
                        assert -(-ntiles // f) <= 256 and (ntiles <= 256 or -(-ntiles // b) <= 256)


def test_non_causal_backward_of_64_buckets_takes_whole_rounds():
    """Two workgroups of 64 buckets per CU (K = 4: three): 2048 tiles of 16 streams
    in one round of 512, not in one and a half."""
    from race_attention_amd import _lib
    for K, L, want in ((3, 8, 32), (2, 16, 32), (4, 4, 48)):
        assert _segments(2, 65536, 8, K, L, _lib.RACE_DTYPE_BF16, causal=0)[1] == want


@pytest.mark.gpu
@pytest.mark.parametrize("nseg", [1, 2, 3, 4, 5, 7, 63, 64, 65, 69])
def test_noncausal_totals(dev, nseg):
    for dtype in (torch.float32, torch.bfloat16):
        L, K, T = 5, 2, 32 * nseg - 5
        q, k, v, do, planes = make_case(T=T, H=2, L=L, K=K, dtype=dtype, seed=nseg)
        gpu = run_gpu(q, k, v, do, planes, L=L, K=K, causal=False, inv_temp=0.8, dev=dev, seg_tiles=1)
        ref = run_oracle(q, k, v, do, planes, causal=False, inv_temp=0.8)
        compare(f"totals nseg={nseg} {dtype}", gpu[:4] + (ref[4],), ref, TOL[dtype])


def test_noncausal_backward_segments_are_their_own():
    """384 streams of 10 tiles at 32 buckets: the forward's 3-tile segments are
    no divisor of the backward's 5-tile ones."""
    from race_attention_amd import _lib
    assert _segments(64, 300, 6, 2, 5, _lib.RACE_DTYPE_BF16, causal=0) == (4, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,H,K,L,dtype", [
    (64, 300, 6, 2, 5, torch.bfloat16),  # 4 forward segments, 2 backward ones
    (64, 300, 6, 2, 5, torch.float32),
    (130, 37, 8, 2, 5, torch.bfloat16),  # one segment per stream: the sums are the totals
    (130, 37, 8, 2, 5, torch.float32),
    (65, 40, 16, 8, 2, torch.bfloat16),  # the same, over bucket slices
    (12, 300, 8, 6, 5, torch.bfloat16),  # several over bucket slices
])
def test_noncausal_automatic_segments(dev, B, T, H, K, L, dtype):
    q, k, v, do, planes = make_case(B=B, T=T, H=H, L=L, K=K, dtype=dtype, seed=B)
    gpu = run_gpu(q, k, v, do, planes, L=L, K=K, causal=False, inv_temp=0.8, dev=dev)
    ref = run_oracle(q, k, v, do, planes, causal=False, inv_temp=0.8)
    compare(f"auto {B}x{H}x{T} K={K} {dtype}", gpu[:4] + (ref[4],), ref, TOL[dtype])


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,H,K,L", [
    (12, 1000, 8, 6, 5),  # 3 slices, three forward segments
    (6, 2100, 8, 7, 4),   # 4 slices, joined forward segments
    (1, 9000, 7, 6, 5),   # odd groups
])
def test_causal_automatic_segments_over_slices(dev, B, T, H, K, L):
    q, k, v, do, planes = make_case(B=B, T=T, H=H, L=L, K=K, seed=B)
    gpu = run_gpu(q, k, v, do, planes, L=L, K=K, causal=True, inv_temp=0.125, dev=dev)
    ref = run_oracle(q, k, v, do, planes, causal=True, inv_temp=0.125)
    compare(f"auto {B}x{H}x{T} K={K}", gpu[:4] + (ref[4],), ref, TOL[torch.bfloat16])
