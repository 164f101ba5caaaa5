"""Whole-tile instantiations of 32 and 64 buckets: causal bf16 at 2 to 4 hash
bits, used when T is a multiple of 32 and the tables fill the workgroup's
buckets.  They do the general kernels' arithmetic without row and bucket guards.

A sequence of T + 1 tokens runs the general kernels (its last tile holds one
row), and what a causal operator gives the first T tokens is that of the first T
alone; with a zero gradient at the last token so are the gradients, whose reverse
sums then only add zeros.  The two are compiled apart, and fp32 expressions that
contract differently (2^-24) move a bf16 rounding now and then: the bar is one
bf16 step of the tensor's largest element, max|a-b| <= 2^-8 max|b|.  T: one tile,
an odd and an even number of tiles in segments of two, and one segment of
several.  And against the fp64 oracle at the parity bar (2e-2 bf16)."""
import pytest
import torch

from helpers import TOL, compare, make_case, relerr, run_gpu, run_oracle, to64

pytestmark = pytest.mark.gpu

STEP = 2.0 ** -8
SIZES = [(2, 8), (2, 16), (3, 4), (3, 8), (4, 2), (4, 4)]


def _pair(T, K, L, seed):
    q, k, v, do, planes = make_case(B=2, T=T + 1, H=2, L=L, K=K, seed=seed)
    do[:, :, T:] = 0
    return q, k, v, do, planes


@pytest.mark.parametrize("K,L", SIZES)
def test_whole_tiles_match_the_general_kernels(dev, K, L):
    from race_attention_amd.functional import race_bwd_raw, race_fwd_raw
    for T, seg in ((32, 1), (96, 2), (128, 2), (160, 5)):
        q, k, v, do, planes = [x.to(dev) for x in _pair(T, K, L, T)]
        got = {}
        for n in (T, T + 1):
            a = [x[:, :, :n].contiguous() for x in (q, k, v)]
            out, st = race_fwd_raw(*a, planes, L=L, K=K, causal=True, inv_temp=0.9, seg_tiles=seg)
            g = race_bwd_raw(*a, planes, do[:, :, :n].contiguous(), st, L=L, K=K, causal=True, inv_temp=0.9,
                             seg_tiles=seg)
            got[n] = [x[:, :, :T] for x in (out, *g[:3])]
        for nm, a, b in zip(("out", "dq", "dk", "dv"), got[T], got[T + 1]):
            e = relerr(to64(a), to64(b))
            print(f"[K={K} L={L} T={T}] {nm} {e:.1e}", flush=True)
            assert e <= STEP, nm


@pytest.mark.parametrize("K,L", SIZES)
def test_whole_tiles_match_the_general_kernels_global(dev, K, L):
    from race_attention_amd.functional import race_global_bwd_raw, race_global_fwd_raw
    for T, seg in ((32, 1), (96, 2), (160, 5)):
        q, k, v, do, planes = [x.to(dev) for x in _pair(T, K, L, T)]
        dden = torch.randn(1, 2, 2, T + 1, generator=torch.Generator().manual_seed(T)).to(dev)
        dden[..., T:] = 0
        got = {}
        for n in (T, T + 1):
            a = [x[:, :, :n].contiguous() for x in (q, k, v)]
            out, den, st = race_global_fwd_raw(*a, planes, L=L, K=K, beta=1.0, seg_tiles=seg)
            g = race_global_bwd_raw(*a, planes, out, den, do[:, :, :n].contiguous(), dden[..., :n].contiguous(), st,
                                    L=L, K=K, beta=1.0, seg_tiles=seg)
            got[n] = [den[..., :T]] + [x[:, :, :T] for x in (out, *g[:3])]
        for nm, a, b in zip(("den", "out", "dq", "dk", "dv"), got[T], got[T + 1]):
            e = relerr(to64(a), to64(b))
            print(f"[global K={K} L={L} T={T}] {nm} {e:.1e}", flush=True)
            assert e <= STEP, nm


@pytest.mark.parametrize("K,L", SIZES)
def test_whole_tiles_oracle(dev, K, L):
    for T, it in ((64, 0.125), (192, 0.9)):
        q, k, v, do, planes = make_case(B=2, T=T, H=2, L=L, K=K, seed=T)
        gpu = run_gpu(q, k, v, do, planes, L=L, K=K, causal=True, inv_temp=it, dev=dev, seg_tiles=2)
        ref = run_oracle(q, k, v, do, planes, causal=True, inv_temp=it)
        compare(f"whole K={K} L={L} T={T}", gpu, ref, TOL[torch.bfloat16])
