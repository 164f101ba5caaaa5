"""The C++ autograd calls (csrc/race_torch.cpp) against the Python Functions,
which make the same C ABI calls: bit-equal outputs and gradients over the forms
an ordinary call takes (layouts, an expand over M, planes of each rank, host and
device temperatures and logits, inputs without gradients, no grad mode), and what
the Python path refuses or converts stays so (shapes, CPU tensors, functorch
transforms, forward-mode AD, integer temperatures, misaligned rows, tensor
subclasses), saved-tensor hooks and the in-place check included."""
import math

import pytest
import torch

from helpers import make_case

pytestmark = pytest.mark.gpu

L, K = 5, 2


def _inputs(dev, dtype=torch.bfloat16, M=1, T=70, layout="contig", seed=3, **kw):
    q, k, v, do, planes = make_case(M=M, B=2, T=T, H=2, L=L, K=K, dtype=dtype, seed=seed, **kw)
    x = [t.to(dev) for t in (q, k, v)]
    if layout == "bhtd":
        x = [t.permute(0, 1, 3, 2, 4).contiguous().permute(0, 1, 3, 2, 4) for t in x]
    elif layout == "fused":
        big = torch.stack(x, dim=4)
        x = [big[..., j, :] for j in range(3)]
    elif layout == "off":  # rows 4 bytes off: copied by either path
        def off(t):
            buf = torch.zeros(t.numel() + 2, dtype=t.dtype, device=dev)
            buf[2:] = t.flatten()
            return buf[2:].view(t.shape).transpose(1, 2).contiguous().transpose(1, 2)
        x = [off(t) for t in x]
    return x, do.to(dev), planes.to(dev)


def _leaves(x):
    return [t.detach().requires_grad_(True) for t in x]


def _equal(a, b):
    for u, w in zip(a, b):
        assert (u is None) == (w is None)
        if u is not None:
            assert u.shape == w.shape and u.dtype == w.dtype and torch.equal(u, w)


def _temps(dev):
    return [0.125, torch.tensor(0.7, device=dev), torch.tensor(0.7, device=dev, dtype=torch.float64)]


@pytest.mark.parametrize("layout", ["contig", "bhtd", "fused", "off"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("causal", [True, False])
def test_operator_equals_python_function(dev, layout, dtype, causal):
    from race_attention_amd.functional import RACEFunction, _native, race_attention
    x, do, planes = _inputs(dev, dtype, layout=layout)
    for pl in (planes, planes[0]):
        for temp in _temps(dev):
            got, ref = [], []
            for fn, res in ((lambda q, k, v, t: race_attention(q, k, v, pl, L=L, K=K, causal=causal, inv_temp=t), got),
                            (lambda q, k, v, t: RACEFunction.apply(q, k, v, pl, t, L, K, causal, 1e-6), ref)):
                q, k, v = _leaves(x)
                t = temp.detach().clone().requires_grad_(True) if torch.is_tensor(temp) else temp
                out = fn(q, k, v, t)
                ins = [q, k, v] + ([t] if torch.is_tensor(t) else [])
                res += [out, *torch.autograd.grad(out, ins, do)]
            _equal(got, ref)
    assert _native("F1", *x, planes, 0.125, None, L, K, causal, False, 1e-6) is not None


def test_expand_partial_gradients_and_no_grad(dev):
    from race_attention_amd.functional import RACEFunction, race_attention
    x, do, planes = _inputs(dev, M=2, expand_m=True, share_planes=False)
    do = do.expand(2, -1, -1, -1, -1)
    base = [t[0].detach().clone() for t in x]
    for need in ((True, True, True), (False, True, False), (True, False, False)):
        res = []
        for native in (True, False):
            b = [t.clone().requires_grad_(n) for t, n in zip(base, need)]
            q, k, v = [t.unsqueeze(0).expand(2, -1, -1, -1, -1) for t in b]
            out = (race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5) if native
                   else RACEFunction.apply(q, k, v, planes, 0.5, L, K, True, 1e-6))
            out.backward(do)
            res.append([out.detach()] + [t.grad for t in b])
        _equal(*res)
    with torch.no_grad():
        out = race_attention(*x, planes, L=L, K=K, causal=True, inv_temp=0.5)
    assert not out.requires_grad and torch.equal(out, res[0][0])


@pytest.mark.parametrize("mask", [None, "float", "bool"])
def test_ex_and_global_and_probs_equal_python(dev, mask):
    from race_attention_amd.functional import (RACEExFunction, RACEGlobalFunction, RACEProbsFunction,
                                               race_attention_ex, race_attention_global, race_bucket_probs)
    x, do, planes = _inputs(dev, torch.float32)
    g = torch.Generator().manual_seed(1)
    m = None if mask is None else (torch.rand(2, 70, generator=g) > 0.3).to(dev)
    m = m.float() if mask == "float" else m
    dden = torch.randn(1, 2, 2, 70, generator=g).to(dev)
    for want in (True, False):
        res = []
        for native in (True, False):
            q, k, v = _leaves(x)
            t = torch.tensor(0.8, device=dev, requires_grad=True)
            r = (race_attention_ex(q, k, v, planes, L=L, K=K, inv_temp=t, kmask=m, with_den=want) if native
                 else RACEExFunction.apply(q, k, v, planes, t, m, L, K, 1e-6, want))
            r = r if isinstance(r, tuple) else (r,)
            outs = r[:2] if want else r[:1]
            res.append([*outs, *torch.autograd.grad(outs, (q, k, v, t), (do, dden)[:len(outs)])])
        _equal(*res)
    for grads in ((do, dden), (do, None), (None, dden)):
        res = []
        for native in (True, False):
            q, k, v = _leaves(x)
            t = torch.tensor(0.8, device=dev, requires_grad=True)
            r = (race_attention_global(q, k, v, planes, L=L, K=K, beta=t) if native
                 else RACEGlobalFunction.apply(q, k, v, planes, t, L, K, 1e-6))
            used = [(o, gr) for o, gr in zip(r, grads) if gr is not None]
            res.append([*r, *torch.autograd.grad([o for o, _ in used], (q, k, v, t), [gr for _, gr in used])])
        _equal(*res)
    dP = torch.randn(1, 2, 2, 70, L, 1 << K, generator=g).to(dev)
    res = []
    for native in (True, False):
        q = _leaves(x)[0]
        t = torch.tensor(0.8, device=dev, requires_grad=True)
        P = (race_bucket_probs(q, planes, L=L, K=K, inv_temp=t) if native
             else RACEProbsFunction.apply(q, planes, t, L, K).view(dP.shape))
        res.append([P, *torch.autograd.grad(P, (q, t), dP)])
    _equal(*res)


@pytest.mark.parametrize("z", [0.0, -0.6931, 2.9, 3.1, -5.0, 100.0, float("nan")])
def test_logit_temperature(dev, z):
    """One launch for 1 / clamp(exp(z), 1e-2, 20) and its gradient against
    torch's expressions, inside and beyond the clamp: exp, a quotient and two
    products, 1e-6 relative (8 ulp)."""
    from race_attention_amd import _lib
    logit = torch.tensor(z, device=dev, requires_grad=True)
    ref = 1.0 / logit.exp().clamp(1e-2, 20.0)
    dref, = torch.autograd.grad(ref, logit)
    out = torch.empty(2, device=dev)
    rc = _lib.load().race_inv_temp(logit.data_ptr(), 1e-2, 20.0, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.testing.assert_close(out, torch.stack([ref.detach(), dref]), rtol=1e-6, atol=0, equal_nan=True)
    assert _lib.load().race_inv_temp(logit.data_ptr(), 0.0, 1.0, out.data_ptr(), None) == -1


def test_module_temperature_equals_expressions(dev):
    """vit.BatchedACE with its logit against the same call with the temperature
    as torch expressions: the inverse temperatures differ by an ulp at most, so
    fp32 results by 1e-5 of the largest value."""
    from race_attention_amd import vit
    from race_attention_amd.functional import RACEFunction
    x, do, planes = _inputs(dev, torch.float32)
    ace = vit.BatchedACE(64, K, L, 1, device=dev).to(dev)
    with torch.no_grad():
        ace.logit_temp.fill_(math.log(0.6))
    res = []
    for native in (True, False):
        q, k, v = _leaves(x)
        out = ace(k, v, q) if native else RACEFunction.apply(q, k, v, ace.planes(), 1.0 / ace.scale(), L, K, False, 1e-6)
        res.append([out, *torch.autograd.grad(out, (q, k, v, ace.logit_temp), do)])
    for a, b in zip(*res):
        assert a.shape == b.shape and (a - b).abs().max() <= 1e-5 * b.abs().max()


def test_refusals_and_conversions_stay(dev):
    from race_attention_amd._lib import RaceError
    from race_attention_amd.functional import race_attention
    x, do, planes = _inputs(dev)
    q, k, v = x
    kw = dict(L=L, K=K, causal=True, inv_temp=0.5)
    ref = race_attention(q, k, v, planes, **kw)
    assert torch.equal(race_attention(q, k, v, planes.double(), **kw), ref)          # planes converted
    assert torch.equal(race_attention(q, k, v, planes, **{**kw, "inv_temp": torch.tensor(0.5)}), ref)  # CPU scalar
    race_attention(q, k, v, planes, **{**kw, "inv_temp": 1})
    with pytest.raises(ValueError):
        race_attention(q, k[:, :, :3], v, planes, **kw)
    with pytest.raises(TypeError):
        race_attention(q, k.float(), v, planes, **kw)
    with pytest.raises(ValueError):
        race_attention(q, k, v, planes[..., :1, :], **kw)
    with pytest.raises(RuntimeError, match="ROCm GPUs only"):
        race_attention(q.cpu(), k.cpu(), v.cpu(), planes.cpu(), **kw)
    with pytest.raises(RaceError, match="hash bits"):
        race_attention(q, k, v, torch.randn(1, 9, 64, device=dev), L=1, K=9, causal=True, inv_temp=0.5)
    assert race_attention(q[:, :, :0], k[:, :, :0], v[:, :, :0], planes, **kw).shape == q[:, :, :0].shape
    one = torch.tensor([0.5], device=dev, requires_grad=True)  # a gradient only for 0-dim temperatures
    with pytest.raises(RuntimeError, match="invalid gradient"):
        race_attention(q, k, v, planes, **{**kw, "inv_temp": one}).sum().backward()
    f = lambda z: race_attention(z, k, v, planes, **kw).float().sum()  # noqa: E731
    with pytest.raises(RuntimeError):
        torch.func.grad(f)(q)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda z: race_attention(z, k, v, planes, **kw))(torch.stack([q, q]))
    with pytest.raises((RuntimeError, NotImplementedError)):
        with torch.autograd.forward_ad.dual_level():
            race_attention(torch.autograd.forward_ad.make_dual(q, torch.ones_like(q)), k, v, planes, **kw)

    class Sub(torch.Tensor):
        pass

    assert torch.equal(race_attention(q.as_subclass(Sub), k, v, planes, **kw).as_subclass(torch.Tensor), ref)


def test_saved_tensor_hooks_and_version_check(dev):
    from race_attention_amd.functional import race_attention
    x, do, planes = _inputs(dev)
    q, k, v = _leaves(x)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.to(dev)):
        out = race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5)
    assert packed.count(q.shape) == 3
    g1 = torch.autograd.grad(out, (q, k, v), do)
    out = race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5)
    _equal(g1, torch.autograd.grad(out, (q, k, v), do))
    # the temperature is copied at the call (an update before the backward is not seen), the inputs are checked
    t = torch.tensor(0.5, device=dev)
    out = race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=t)
    t.fill_(9.0)
    _equal(g1, torch.autograd.grad(out, (q, k, v), do))
    out = race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5)
    with torch.no_grad():
        k.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out, (q, k, v), do)


def test_streams_and_graph_capture(dev):
    """A call on a side stream, and forward + backward captured into a graph and
    replayed on new inputs with eager work between, against eager calls."""
    from race_attention_amd.functional import LogitTemp, race_attention
    x, do, planes = _inputs(dev)
    logit = torch.tensor(-0.3, device=dev, requires_grad=True)

    def step(q, k, v):
        out = race_attention(q, k, v, planes, L=L, K=K, causal=False, inv_temp=LogitTemp(logit, 1e-2, 20.0))
        return (out, *torch.autograd.grad(out, (q, k, v, logit), do))

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        side = step(*_leaves(x))
    torch.cuda.current_stream().wait_stream(s)
    _equal([t.detach() for t in side], [t.detach() for t in step(*_leaves(x))])
    static = _leaves(x)
    with torch.cuda.stream(s):
        for _ in range(2):
            step(*static)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        res = step(*static)
    for rep in range(3):
        new = [torch.nn.functional.normalize(torch.randn(t.shape, device=dev), dim=-1).to(t.dtype) for t in static]
        with torch.no_grad():
            for t, n in zip(static, new):
                t.copy_(n)
        g.replay()
        torch.cuda.synchronize()
        _equal([t.detach().clone() for t in res], [t.detach() for t in step(*_leaves(new))])


@pytest.mark.parametrize("use", ["layer", "layer then exp"])
def test_checkpoint_of_an_operator(dev, use):
    """Non-reentrant checkpointing ends its recomputation with an exception from
    the hook that packs the last saved tensor, which can be the operator's."""
    from torch.utils.checkpoint import checkpoint

    from race_attention_amd.functional import race_attention, race_bucket_probs
    x, do, planes = _inputs(dev)

    def layer(q, k, v):
        out = race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5)
        return out if use == "layer" else out.exp()

    leaves = _leaves(x)
    want = torch.autograd.grad(layer(*leaves), leaves, do)
    _equal(want, torch.autograd.grad(checkpoint(layer, *leaves, use_reentrant=False), leaves, do))
    probs = lambda q: race_bucket_probs(q, planes, L=L, K=K, inv_temp=0.5)
    dP = torch.rand_like(probs(x[0]))
    want = torch.autograd.grad(probs(leaves[0]), leaves[0], dP)
    _equal(want, torch.autograd.grad(checkpoint(probs, leaves[0], use_reentrant=False), leaves[0], dP))


def test_exceptions_keep_their_types(dev):
    from race_attention_amd.functional import race_attention

    class Stop(Exception):
        pass

    def stop(t):
        raise Stop

    x, do, planes = _inputs(dev)
    q, k, v = _leaves(x)
    with torch.autograd.graph.saved_tensors_hooks(stop, lambda t: t), pytest.raises(Stop):
        race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5)
    # the caching allocator's own limit (nothing is asked of the device)
    # an output of 33 GB, more than any block that earlier calls left in the cache, from an expanded input
    big = torch.zeros(1, 1, 16384, 8, 64, device=dev, dtype=torch.bfloat16).expand(1, 2000, -1, -1, -1)
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-9)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            race_attention(big, big, big, planes, L=L, K=K, causal=True, inv_temp=0.5)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    _equal([race_attention(*x, planes, L=L, K=K, causal=True, inv_temp=0.5)],
           [race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5).detach()])


@pytest.mark.parametrize("where", ["class", "instance"])
def test_a_scale_of_the_program_is_used(dev, where):
    """A scale() that a program put in place, in a subclass or on the module."""
    from race_attention_amd import vit
    from race_attention_amd.functional import race_attention
    (q, k, v), do, planes = _inputs(dev)

    class Fixed(vit.BatchedACE):
        def scale(self):
            return 4.0 * self.logit_temp.exp()

    ace = (Fixed if where == "class" else vit.BatchedACE)(d_k=64, K=K, L=L, M=1).to(dev)
    if where == "instance":
        ace.scale = lambda: 4.0 * ace.logit_temp.exp()
    got = ace(k, v, q)
    want = race_attention(q, k, v, ace.planes(), L=L, K=K, causal=False,
                          inv_temp=(1.0 / (4.0 * ace.logit_temp.exp())).detach())
    _equal([got.detach()], [want])
    if where == "instance":  # no upper bound
        ace = vit.BatchedACE(d_k=64, K=K, L=L, M=1, temp_max=None).to(dev)
        assert torch.equal(ace(k, v, q), race_attention(q, k, v, ace.planes(), L=L, K=K, causal=False, inv_temp=1.0))


def test_a_scale_put_on_the_class_and_an_attribute_of_any_name(dev, monkeypatch):
    """A program that replaces BatchedACE.scale itself, and modules that hold an
    attribute named inv_temp: scale() is what counts, in the layer, the padded
    layer and the bucket probabilities."""
    from types import SimpleNamespace

    from race_attention_amd import classification, vit
    from race_attention_amd.buckets import race_bucket_probs_from_qk
    from race_attention_amd.functional import race_attention, race_attention_ex, race_bucket_probs
    (q, k, v), do, planes = _inputs(dev)

    def check(cls, name, scale):
        ace = cls(d_k=64, K=K, L=L, M=1).to(dev)
        ace.inv_temp = torch.tensor(99.0, device=dev)
        kw = dict(L=L, K=K, inv_temp=(1.0 / scale(ace)).detach())
        if name == "vit":
            want = race_attention(q, k, v, ace.planes(), causal=False, **kw)
        else:
            want = race_attention_ex(q, k, v, ace.planes(), **kw)
        _equal([ace(k, v, q).detach()], [want])
        got = race_bucket_probs_from_qk(SimpleNamespace(ace=ace, M=1), q[0], k[0])
        _equal([t.detach() for t in got], [race_bucket_probs(t, ace.planes(), **kw) for t in (q, k)])

    for cls, name in ((vit.BatchedACE, "vit"), (classification.BatchedACE, "padded")):
        check(cls, name, lambda ace: ace.logit_temp.exp())
    monkeypatch.setattr(vit.BatchedACE, "scale", lambda self: 4.0 * self.logit_temp.exp())
    for cls, name in ((vit.BatchedACE, "vit"), (classification.BatchedACE, "padded")):
        check(cls, name, lambda ace: 4.0 * ace.logit_temp.exp())

    class Own:  # any object with planes() and scale()
        L, K, inv_temp = L, K, 99.0
        planes = staticmethod(lambda: planes)
        scale = staticmethod(lambda: torch.tensor(2.0, device=dev))

    got = race_bucket_probs_from_qk(SimpleNamespace(ace=Own, M=1), q[0], k[0])
    _equal(got, [race_bucket_probs(t, planes, L=L, K=K, inv_temp=0.5) for t in (q, k)])


@pytest.mark.parametrize("why", ["absent", "not a library"])
def test_the_python_functions_alone(dev, why, monkeypatch, tmp_path):
    """Where the C++ calls are not built, or do not load, the Python Functions
    make every call; it is said once."""
    import warnings

    from race_attention_amd import _lib, vit
    from race_attention_amd.functional import race_attention, race_attention_global, race_bucket_probs
    (q, k, v), do, planes = _inputs(dev)
    ace = vit.BatchedACE(d_k=64, K=K, L=L, M=1).to(dev)

    def calls():
        a, b, c = _leaves((q, k, v))
        out = race_attention(a, b, c, planes, L=L, K=K, causal=True, inv_temp=0.5)
        layer = ace(b, c, a)  # (no gradient of its temperature: that sums in another order as torch expressions)
        return [out, *torch.autograd.grad(out, (a, b, c), do), *torch.autograd.grad(layer, (a, b, c), do),
                *race_attention_global(q, k, v, planes, L=L, K=K, beta=1.0),
                race_bucket_probs(q, planes, L=L, K=K, inv_temp=0.5)]

    want = calls()
    path = tmp_path / "_race_torch.so"
    if why != "absent":
        path.write_bytes(b"no library")
    monkeypatch.setattr(_lib, "TORCH_PATH", str(path))
    monkeypatch.setattr(_lib, "_calls", None)
    with pytest.warns(RuntimeWarning, match="operator calls go through Python"):
        race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5)
    with warnings.catch_warnings():
        warnings.simplefilter("error", RuntimeWarning)
        _equal(calls(), want)


def test_an_active_dispatch_mode_sees_the_python_call(dev):
    """Under a TorchDispatchMode the Python Functions run, whose allocations and
    conversions the mode sees as ever; a function mode (as set_default_device
    installs) leaves the C++ call in place.  Results are the same."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from race_attention_amd.functional import _native, race_attention
    (q, k, v), do, planes = _inputs(dev)
    want = race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5)
    native = lambda: _native("F1", q, k, v, planes, 0.5, None, L, K, True, False, 1e-6)  # noqa: E731
    seen = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Through(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Log():
        assert native() is None
        _equal([race_attention(q, k, v, planes, L=L, K=K, causal=True, inv_temp=0.5)], [want])
    assert any("empty" in f for f in seen)
    with Through():
        _equal([native()], [want])
    _equal([native()], [want])
