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
