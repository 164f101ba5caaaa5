"""The padded estimator in one call (race_fwd_padded / race_bwd_padded) against the
same with the mask's factors on V, the output and den as torch expressions around
race_attention_ex.

A 0/1 mask multiplies without rounding, so outputs and gradients are bit-equal.  A
fractional mask is rounded to the element type by both, but the expressions round
the operator's output (its dV) before the product too: with one rounding more, a
value can come out as the next one, an ulp away -- up to 2^-7 of the value in bf16
(8 significant bits), 2^-23 in fp32 -- and an expand's gradient adds M such values
and rounds their sum: bars of (M + 1) ulps of the largest value."""
import pytest
import torch

from helpers import make_case

pytestmark = pytest.mark.gpu

CASES = [  # K, L, M, T, dtype, expand over M, layout
    (3, 2, 2, 77, torch.bfloat16, True, "contig"),
    (2, 5, 1, 500, torch.bfloat16, False, "bhtd"),
    (4, 4, 1, 64, torch.bfloat16, False, "fused"),
    (4, 8, 1, 33, torch.bfloat16, False, "contig"),
    (8, 2, 1, 90, torch.bfloat16, False, "contig"),   # bucket slices: partial outputs
    (2, 5, 2, 31, torch.float32, True, "contig"),
    (4, 8, 1, 100, torch.float32, False, "fused"),
    (5, 3, 1, 40, torch.float32, False, "contig"),
]


def _run(x, do, dden, planes, mask, K, L, native, with_den):
    from race_attention_amd.functional import race_attention_ex, race_attention_padded
    M = planes.shape[0]
    base = [t.detach().clone().requires_grad_(True) for t in x]
    q, k, v = [t.expand(M, -1, -1, -1, -1) if t.shape[0] != M else t for t in base]
    t = torch.tensor(0.9, device=do.device, requires_grad=True)
    if native:
        r = race_attention_padded(q, k, v, planes, L=L, K=K, inv_temp=t, mask=mask, with_den=with_den)
    else:
        B, T = q.shape[1:3]
        kw = mask.to(torch.float32)
        f = kw.view(1, B, T, 1, 1)
        r = race_attention_ex(q, k, v * f.to(v.dtype), planes, L=L, K=K, inv_temp=t, kmask=kw, with_den=with_den)
        r = (r[0] * f.to(q.dtype), r[1] * kw.view(1, B, 1, T)) if with_den else r * f.to(q.dtype)
    outs = r if with_den else (r,)
    return [*outs, *torch.autograd.grad(outs, (*base, t), (do, dden)[:len(outs)])]


@pytest.mark.parametrize("mask_kind", ["binary", "bool", "fraction"])
@pytest.mark.parametrize("K,L,M,T,dtype,expand,layout", CASES)
def test_padded_equals_expressions(dev, K, L, M, T, dtype, expand, layout, mask_kind):
    q, k, v, do, planes = make_case(M=1 if expand else M, B=3, T=T, H=2, L=L, K=K, dtype=dtype, seed=K + T,
                                    share_planes=M == 1)
    g = torch.Generator().manual_seed(T)
    planes = torch.randn(M, L, K, 64, generator=g).to(dev)
    x = [t.to(dev) for t in (q, k, v)]
    if layout == "bhtd":
        x = [t.permute(0, 1, 3, 2, 4).contiguous().permute(0, 1, 3, 2, 4) for t in x]
    elif layout == "fused":
        big = torch.stack(x, dim=4)
        x = [big[..., j, :] for j in range(3)]
    do = torch.randn(M, 3, T, 2, 64, generator=g).to(dtype).to(dev)
    dden = torch.randn(M, 3, 2, T, generator=g).to(dev)
    mask = torch.rand(3, T, generator=g)
    if mask_kind != "fraction":
        mask = (mask > 0.4)
        mask[0] = True
        mask[1, T // 2:] = False
    mask = mask.to(dev) if mask_kind == "bool" else mask.float().to(dev)
    for with_den in (True, False):
        a = _run(x, do, dden, planes, mask, K, L, True, with_den)
        b = _run(x, do, dden, planes, mask, K, L, False, with_den)
        for j, (u, w) in enumerate(zip(a, b)):
            assert u.shape == w.shape and u.dtype == w.dtype
            if mask_kind != "fraction":
                assert torch.equal(u, w), (j, with_den)
            else:
                bar = (M + 1) * 2.0 ** (-7 if dtype == torch.bfloat16 else -23)
                assert (u.double() - w.double()).abs().max() <= bar * w.double().abs().max(), (j, with_den)


def test_padded_needs_a_mask(dev):
    import ctypes
    from race_attention_amd import _lib
    lib = _lib.load()
    d = _lib.RaceDesc()
    d.M, d.B, d.T, d.H, d.D, d.L, d.K, d.causal, d.dtype, d.eps, d.inv_temp = 1, 1, 8, 1, 64, 2, 3, 0, 1, 1e-6, 0.5
    p = ctypes.c_void_p(256)
    assert lib.race_fwd_padded(ctypes.byref(d), p, p, p, p, None, p, None, p, p, 1 << 30, None) == -1
    d.causal = 1
    assert lib.race_fwd_padded(ctypes.byref(d), p, p, p, p, p, p, None, p, p, 1 << 30, None) == -2
    assert lib.race_bwd_padded(ctypes.byref(d), p, p, p, p, p, p, None, p, p, p, p, None, p, 1 << 30, None) == -2


def test_mask_gradient_through_expressions(dev):
    """A mask that requires a gradient takes the torch expressions: its factors on
    V and the output pass one, as before."""
    from race_attention_amd import classification
    q, k, v, do, _ = make_case(B=2, T=40, H=2, L=2, K=3, dtype=torch.float32, seed=1)
    ace = classification.BatchedACE(64, 3, 2, 1, device=dev).to(dev)
    mask = torch.rand(2, 40, device=dev, requires_grad=True)
    out = ace(k.to(dev), v.to(dev), q.to(dev), mask=mask)
    g, = torch.autograd.grad(out, mask, do.to(dev))
    assert g.shape == mask.shape and g.abs().sum() > 0
    assert torch.allclose(out.detach(), ace(k.to(dev), v.to(dev), q.to(dev), mask=mask.detach()), atol=1e-6)
