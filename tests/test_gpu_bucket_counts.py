"""Bucket counts at the edges of the workgroup sizes.  Up to 4 hash bits every
bucket of a stream is in one workgroup of 32, 64 or 128 buckets (bf16 and
fp32), whose sigmoid rows hold 16 or 32 projection columns and whose plane
operands are read straight from the planes array: table counts just below and
above each size, a partly empty second column block, one table, planes that
are only 4-byte aligned, and token counts around a tile.

Against the fp64 oracle with the bars of the parity tests (max|a-b|/max|b|:
1e-4 fp32, 2e-2 bf16); eps = 0.5 at T = 1, where the reference's 1e-6 leaves
dq and dk nothing but rounding (see test_gpu_parity.py).  Rows are unit length:
the kernels' tanh is within 1e-7, so dq and dk, which carry 1 - tanh^2, are off
by 2e-7 / (1 - tanh^2) relative where one token and one plane alone set a
tensor's scale -- below 1e-5 at the |x . plane| ~ 1 of unit rows, but 2e-4 was
seen at the |x . plane| ~ 8 of N(0, 1) rows."""
import pytest
import torch

from helpers import TOL, compare, make_case, relerr, run_gpu, run_oracle, to64

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 17), (1, 32), (2, 4), (2, 9), (2, 16), (3, 4), (3, 5), (3, 9), (3, 10), (4, 1), (4, 3), (4, 5)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("K,L", SIZES)
def test_bucket_counts(dev, K, L, dtype):
    for c, (T, causal) in enumerate([(1, True), (33, True), (95, True), (31, False), (70, False)]):
        eps = 0.5 if T == 1 else 1e-6
        q, k, v, do, planes = make_case(T=T, H=2, L=L, K=K, dtype=dtype, seed=100 + c)
        # a planes array that starts 4 bytes into its allocation
        buf = torch.empty(planes.numel() + 1, device=dev)
        buf[1:] = planes.to(dev).flatten()
        gpu = run_gpu(q, k, v, do, buf[1:].view(planes.shape), L=L, K=K, causal=causal, inv_temp=0.5, dev=dev,
                      seg_tiles=2 if T == 95 else 0, eps=eps)
        ref = run_oracle(q, k, v, do, planes, causal=causal, inv_temp=0.5, eps=eps)
        compare(f"K={K} L={L} T={T} causal={causal} {dtype}", gpu, ref, TOL[dtype])


@pytest.mark.parametrize("K,L", [(2, 5), (3, 7), (4, 5)])
def test_bucket_counts_global_fp32(dev, K, L):
    """The global normalisation forms dL/d den from one workgroup's own sums in
    fp32 too."""
    import test_gpu_global as tg
    q, k, v, do, planes = make_case(B=2, T=130, H=2, L=L, K=K, dtype=torch.float32, unit=False, seed=7)
    dden = torch.randn(1, 2, 2, 130, generator=torch.Generator().manual_seed(8))
    gpu = tg._run_gpu(q, k, v, do, dden, planes, L=L, K=K, beta=1.0, dev=dev)
    ref = tg._run_oracle(q, k, v, do, dden, planes, beta=1.0)
    for nm, a, b in zip(("out", "den", "dq", "dk", "dv"), gpu[:5], ref[:5]):
        e = relerr(to64(a), b)
        print(f"[global fp32 K={K} L={L}] {nm} {e:.2e}", flush=True)
        assert e <= TOL[torch.float32], nm


@pytest.mark.parametrize("K,L", [(4, 6), (3, 9)])
@pytest.mark.parametrize("causal", [1, 0])
def test_buffers_of_65_to_96_fp32_buckets(dev, K, L, causal):
    """96 state rows for a workgroup of 128 buckets: buffers of exactly the sizes
    asked for, full of NaN, in front of guard words that stay as they are."""
    import ctypes

    from race_attention_amd import _lib
    from race_attention_amd.functional import _strides4, make_desc
    lib, T, B = _lib.load(), 230, 2
    q, k, v, do, planes = make_case(B=B, T=T, H=3, L=L, K=K, dtype=torch.float32, seed=K)
    x = [t.to(dev) for t in (q, k, v, do)]
    pd = planes.to(dev).contiguous()
    d = make_desc(*x[:3], pd, L=L, K=K, causal=causal, eps=1e-6, inv_temp=0.3, seg_tiles=2)
    d.o_stride = d.do_stride = d.g_stride = _strides4(x[0])
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def buf(n):
        b = torch.full(((n + 7) // 8 + 4096,), float("nan"), dtype=torch.float64, device=dev)
        b[(n + 7) // 8:] = 123.0
        return b, n

    state, wf, wb = [buf(f(ctypes.byref(d))) for f in (lib.race_state_bytes, lib.race_fwd_workspace_bytes,
                                                       lib.race_bwd_workspace_bytes)]
    out, dq, dk, dv = [torch.empty_like(x[0]) for _ in range(4)]
    git = torch.empty((), device=dev)
    _lib.check(lib.race_fwd(ctypes.byref(d), *map(P, x[:3]), P(pd), P(out), P(state[0]), P(wf[0]), wf[1], st), "fwd")
    _lib.check(lib.race_bwd(ctypes.byref(d), *map(P, x[:3]), P(pd), P(x[3]), P(state[0]), P(dq), P(dk), P(dv), P(git),
                            P(wb[0]), wb[1], st), "bwd")
    torch.cuda.synchronize()
    for b, n in (state, wf, wb):
        assert (b[(n + 7) // 8:] == 123.0).all()
    ref = run_oracle(q, k, v, do, planes, causal=bool(causal), inv_temp=0.3)
    gpu = [t.cpu() for t in (out, dq, dk, dv)] + [float(git)]
    compare(f"rows K={K} L={L} causal={causal}", gpu, ref, TOL[torch.float32])
