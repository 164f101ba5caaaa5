"""The two sets of prefix-mean kernels: 16-lane rows (D <= 64 in whole 16-byte
pieces, 16-byte aligned arrays) and one wave per segment (everything else).
Token counts around the 16-token chunks, column counts around the lanes, streams
and lengths that give one segment and many; every aligned call is repeated with v
and the gradient 4 bytes off (the general kernels), with weights that leave whole
prefixes zero, and with infinities, whose columns alone may be infinite or NaN.

Both sum in fp64 from fp32 values in another order, so E, gW and gV, rounded to
fp32 at the end, agree to a few ulps of fp32: 1e-6 of the largest value (1e-5
against the oracle, as the other prefix-mean tests)."""
import numpy as np
import pytest
import torch

from helpers import relerr

pytestmark = pytest.mark.gpu


def _off(x):
    """The same values, 4 bytes off a 16-byte boundary."""
    buf = torch.empty(x.numel() + 1, device=x.device)
    buf[1:] = x.flatten()
    return buf[1:].view(x.shape)


def _both(w, v, gE, eps):
    from race_attention_amd.functional import prefix_mean_bwd, prefix_mean_fwd
    rows = (prefix_mean_fwd(w, v, eps),) + prefix_mean_bwd(w, v, gE, eps)
    v1, g1 = _off(v), _off(gE)
    general = (prefix_mean_fwd(w, v1, eps),) + prefix_mean_bwd(w, v1, g1, eps)
    return rows, general


@pytest.mark.parametrize("NS,T,D", [(1, 1, 4), (3, 15, 64), (2, 16, 8), (5, 17, 60), (2, 31, 64), (1, 33, 64),
                                    (40, 513, 12), (1, 70001, 64), (3000, 18, 32),
                                    # rows of several streams in one workgroup: 24 and 11 segments a stream, 2, and 1
                                    (700, 600, 64), (1500, 170, 20), (16390, 20, 16), (9001, 37, 64)])
def test_rows_and_general_kernels_agree(dev, oracle, NS, T, D):
    g = torch.Generator().manual_seed(NS + 3 * T + 7 * D)
    w = torch.rand(NS, T, generator=g)
    w[0, : T // 2] = 0.0  # a prefix of zero weight: E = 0 / eps there
    v, gE = torch.randn(NS, T, D, generator=g), torch.randn(NS, T, D, generator=g)
    rows, general = _both(w.to(dev), v.to(dev), gE.to(dev), 1e-6)
    torch.cuda.synchronize()
    ref = (oracle.prefix_mean_flat(w.numpy(), v.numpy(), 1e-6),
           *oracle.prefix_mean_flat_bw(w.numpy(), v.numpy(), gE.numpy(), 1e-6))
    for nm, a, b, r in zip(("E", "gW", "gV"), rows, general, ref):
        assert relerr(a.cpu(), b.cpu()) <= 1e-6 and relerr(a.cpu(), r) <= 1e-5, nm


def test_non_finite_values_stay_in_their_columns(dev):
    g = torch.Generator().manual_seed(4)
    NS, T, D = 3, 50, 16  # the last stream stays finite
    w = torch.rand(NS, T, generator=g).to(dev)
    v, gE = torch.randn(NS, T, D, generator=g).to(dev), torch.randn(NS, T, D, generator=g).to(dev)
    v[0, 37, 5] = float("inf")
    gE[1, 49, 3] = float("nan")
    rows, general = _both(w, v, gE, 1e-6)
    for a, b in zip(rows, general):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)) and torch.equal(torch.isnan(a), torch.isnan(b))
        m = torch.isfinite(b)
        assert np.abs((a - b)[m].cpu().numpy()).max() <= 1e-6 * b[m].abs().max().item()
