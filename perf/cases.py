"""The work this framework is measured on: RACE attention layers as programs call them.

A case names one layer's sizes and options; ``prepare`` makes what a program holds
before the call (tensors on the GPU, the module with its hyperplanes, the upstream
gradient), ``run`` makes one pass through the public modules and functions, and
``exact`` gives the same outputs in 64 bits from plain torch.  Sizes are heads of
D = 64, tokens T, batch B, heads H, hash bits K, tables L, estimators M.

  forward   causal layer, inference (prefill)                      race.BatchedACE
  causal    causal layer, forward and backward                     race.BatchedACE
  full      non-causal layer with its learnable temperature        vit.BatchedACE
  padded    non-causal layer with a padding mask and the denominator output
                                                                   classification.BatchedACE
  global    causal layer with one normaliser per token             race_attention_global
  probs     bucket probabilities and their gradient                race_bucket_probs
  prefix    flat causal prefix mean, the fp32 CPU operator's form  RACEPrefixMeanFlatFn
"""
import math

import torch

from race_attention_amd import classification, race, vit
from race_attention_amd.functional import RACEPrefixMeanFlatFn, race_attention_global, race_bucket_probs

D = 64
EPS = 1e-6


def _case(name, op, dtype, B, T, H, K, L, M=1):
    case = {"op": op, "dtype": dtype, "B": B, "T": T, "H": H, "K": K, "L": L, "M": M}
    return {"name": name, **case} if name else case


def listed():
    return [
        # prefill of one short prompt in a 12-head decoder: launches and latency
        _case("prompt_forward", "forward", "bf16", 1, 128, 12, 4, 8),
        # a small fp32 encoder layer in training, the smallest training configuration
        _case("encoder_fp32", "full", "fp32", 1, 4096, 4, 2, 5),
        # an ordinary causal training layer: two 16K documents
        _case("causal_16k", "causal", "bf16", 2, 16384, 8, 4, 8),
        # a ViT encoder layer: batch 64 of 784 patches and the class token
        _case("vit_layer", "full", "bf16", 64, 785, 6, 2, 5),
        # the long-context layer: one sequence of a million tokens (the largest)
        _case("causal_1m", "causal", "bf16", 1, 1 << 20, 8, 4, 8),
        # the decoder layer with 8-bit hashes and two independent estimators
        _case("decoder_8bit", "causal", "bf16", 8, 8192, 12, 8, 4, M=2),
        # text batches of a length that is no multiple of anything, 3-bit hashes
        _case("causal_ragged", "causal", "bf16", 4, 4001, 12, 3, 8),
        # the causal layer trained in single precision
        _case("causal_fp32", "causal", "fp32", 1, 8192, 8, 4, 8),
        # globally normalised causal layer with its default 4 bits and 4 tables
        _case("global_8k", "global", "bf16", 4, 8192, 12, 4, 4),
        # padded classification batch with the denominator output, default hashes
        _case("padded_classifier", "padded", "bf16", 32, 500, 8, 3, 2, M=2),
        # bucket probabilities for a hybrid layer, forward and backward
        _case("bucket_probs", "probs", "bf16", 2, 16384, 8, 4, 8),
        # the flat prefix mean over the streams of a 4096-token layer, 16 buckets a head
        _case("prefix_mean", "prefix", "fp32", 1, 4096, 8, 4, 1),
    ]


def _log(rng, lo, hi):
    """A whole number spread over [lo, hi] in its logarithm; one in three is a power of two's multiple of 32."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if rng.random() < 1 / 3:
        return max(lo, min(hi, 32 * max(1, round(x / 32))))
    return max(lo, min(hi, round(x)))


def draw(rng):
    op = rng.choice(["forward", "causal", "causal", "full", "padded", "global", "probs", "prefix"])
    dtype = "fp32" if op == "prefix" or rng.random() < 0.25 else "bf16"
    H = rng.choice([4, 6, 8, 12])
    if op == "prefix":
        # flat streams: heads x buckets of one sequence each
        K = rng.choice([2, 3, 4])
        return _case(None, op, dtype, 1, _log(rng, 200, 8000), H, K, 1)
    K, L = rng.choice([(2, 5), (3, 2), (3, 8), (4, 4), (4, 8), (4, 8)])
    if op == "causal" and dtype == "bf16" and rng.random() < 0.2:
        K, L = 8, 4
    M = 2 if op == "padded" or (K == 8 and rng.random() < 0.5) else 1
    T = _log(rng, *{"forward": (64, 262144), "causal": (500, 262144), "full": (190, 16384), "padded": (100, 2048),
                    "global": (500, 131072), "probs": (500, 65536)}[op])
    # batch: at most about 1.5e9 (fp32: 2e8) token-heads times buckets, and a batch of ordinary size
    budget = (2e8 if dtype == "fp32" else 1.2e9 if K == 8 else 6e8) / (M * H * (L << K))
    T = int(min(T, budget))
    B = max(1, min(rng.choice([1, 2, 4, 8, 16, 32, 64]), int(budget / T)))
    return _case(None, op, dtype, B, T, H, K, L, M)


# ------------------------------------------------------------------ inputs
def _torch_dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _inputs(case, seed):
    """The tensors of a case, from the seed alone (a dict of tensors on the GPU)."""
    g = torch.Generator("cuda").manual_seed(1000003 * int(seed) + 17)
    M, B, T, H, K, L = (case[x] for x in ("M", "B", "T", "H", "K", "L"))
    dt = _torch_dtype(case)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    if case["op"] == "prefix":
        ns = B * H << K
        return {"w": torch.softmax(normal(B * H, 1 << K, T), dim=1).reshape(ns, T), "v": normal(ns, T, D),
                "dout": normal(ns, T, D)}
    unit = torch.nn.functional.normalize
    # independent planes per estimator for M > 1, as the modules draw them
    x = {"planes": normal(M, L, K, D)}
    if case["op"] in ("full", "padded"):
        # Q and K of self-attention come from the same tokens, so a token's key resembles its
        # query, and the layer is trained towards its values: the temperature has a gradient
        # that is not a sum of noise
        h = normal(B, T, H, D)
        q, k, v = h + 0.3 * normal(B, T, H, D), h + 0.3 * normal(B, T, H, D), normal(B, T, H, D)
        if dt is torch.bfloat16:
            q, k, v = unit(q, dim=-1), unit(k, dim=-1), unit(v, dim=-1)
        x.update(q=q.to(dt), k=k.to(dt), v=v.to(dt), dout=(v + 0.1 * normal(B, T, H, D)).to(dt))
        if case["op"] == "padded":
            lengths = torch.randint(T // 4, T + 1, (B, 1), generator=g, device="cuda")
            x["mask"] = (torch.arange(T, device="cuda")[None] < lengths).to(torch.float32)
            x["dden"] = 1e-3 * normal(M, B, T, H)
        return x
    if case["op"] == "probs":
        x["x"] = unit(normal(M, B, T, H, D), dim=-1).to(dt)
        x["dout"] = normal(M, B, H, T, L, 1 << K)
        return x
    for name in ("q", "k", "v"):
        x[name] = unit(normal(M, B, T, H, D), dim=-1).to(dt)
    if case["op"] != "forward":
        x["dout"] = normal(M, B, T, H, D).to(dt)
    if case["op"] == "global":
        x["dden"] = 1e-3 * normal(M, B, H, T)
    return x


def _set_planes(ace, planes):
    """Give a module the case's hyperplanes [M,L,K,D] (its buffer: [D,L*K] shared, [M,D,L*K] otherwise)."""
    M, L, K, _ = planes.shape
    flat = planes.view(M, L * K, D).transpose(1, 2)
    ace.planes_T = flat[0] if ace.share_planes else flat
    return ace


TEMPERATURE = 0.5  # value of the learnable temperature


def prepare(case, seed):
    x = _inputs(case, seed)
    op, M, K, L = case["op"], case["M"], case["K"], case["L"]
    state = {"case": case, **x}
    for name in ("q", "k", "v", "x", "w"):
        if name in x and op != "forward":
            x[name].requires_grad_(True)
    if op in ("forward", "causal"):
        state["ace"] = _set_planes(race.BatchedACE(D, K, L, M, device="cuda", share_planes=M == 1), x["planes"])
    elif op in ("full", "padded"):
        cls = vit.BatchedACE if op == "full" else classification.BatchedACE
        ace = _set_planes(cls(D, K, L, M, device="cuda", share_planes=False), x["planes"]).to("cuda")
        with torch.no_grad():
            ace.logit_temp.fill_(math.log(TEMPERATURE))
        state["ace"] = ace
    elif op == "global":
        state["beta"] = torch.tensor(1.0, device="cuda")
    elif op == "probs":
        state["inv_temp"] = 1.0 / math.sqrt(D)
    return state


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    op, M, K, L = case["op"], case["M"], case["K"], case["L"]
    if op == "forward":
        with torch.no_grad():
            return {"out": state["ace"](state["k"], state["v"], state["q"])}
    if op == "prefix":
        w, v = state["w"], state["v"]
        out = RACEPrefixMeanFlatFn.apply(w, v, EPS)
        dw, dv = torch.autograd.grad(out, (w, v), state["dout"])
        return {"out": out.detach(), "dw": dw, "dv": dv}
    if op == "probs":
        p = race_bucket_probs(state["x"], state["planes"], L=L, K=K, inv_temp=state["inv_temp"])
        dx, = torch.autograd.grad(p, (state["x"],), state["dout"])
        return {"probs": p.detach(), "dx": dx}
    q, k, v = state["q"], state["k"], state["v"]
    if op == "causal":
        out = state["ace"](k, v, q)
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
        return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    if op == "global":
        out, den = race_attention_global(q, k, v, state["planes"], L=L, K=K, beta=state["beta"])
        dq, dk, dv = torch.autograd.grad((out, den), (q, k, v), (state["dout"], state["dden"]))
        return {"out": out.detach(), "den": den.detach(), "dq": dq, "dk": dk, "dv": dv}
    ace = state["ace"]
    Q, Kx, V = (z.unsqueeze(0).expand(M, -1, -1, -1, -1) for z in (q, k, v))
    if op == "full":
        out = ace(Kx, V, Q)
        dq, dk, dv, dtemp = torch.autograd.grad(out, (q, k, v, ace.logit_temp), state["dout"].expand_as(out))
        return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv, "dtemp": dtemp}
    out, den = ace.forward_with_den(Kx, V, Q, mask=state["mask"])
    dq, dk, dv, dtemp = torch.autograd.grad((out, den), (q, k, v, ace.logit_temp),
                                            (state["dout"].expand_as(out), state["dden"]))
    return {"out": out.detach(), "den": den.detach(), "dq": dq, "dk": dk, "dv": dv, "dtemp": dtemp}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Each input read once, each output written once; the operator's own products (projection,
    bucket sums, readout and, for training, their adjoints), as 2 operations a multiply-add."""
    op, M, B, T, H, K, L = (case[x] for x in ("op", "M", "B", "T", "H", "K", "L"))
    e = 2 if case["dtype"] == "bf16" else 4
    S = L << K
    if op == "prefix":
        ns = B * H << K
        return {"bytes": 4 * ns * T * (4 * D + 2), "flops": ns * T * 12 * D}
    th = M * B * T * H
    if op == "probs":
        return {"bytes": th * (2 * D * e + 8 * S), "flops": th * (4 * D * L * K + 8 * S)}
    shared = op in ("full", "padded")  # q, k, v and their gradients have no M dimension
    rows = 3 * B * T * H if shared else 3 * th
    if op == "forward":
        return {"bytes": (rows + th) * D * e, "flops": th * (4 * D * L * K + 4 * S * (D + 1))}
    nbytes = (2 * rows + th + (B * T * H if shared else th)) * D * e
    if op in ("padded", "global"):
        nbytes += 8 * th + (4 * B * T if op == "padded" else 0)
    sums = 4 if op in ("causal", "global") else 2
    return {"bytes": nbytes, "flops": th * (8 * D * L * K + sums * S * (D + 1) + 10 * S * D)}


def tolerance(case):
    """About four times the errors measured against exact(): the prefix mean (64-bit sums) 2.7e-8,
    fp32 layers 1.4e-6, bf16 gradients 6.4e-3 with 4-bit causal hashes and 3.3e-3 elsewhere.  The
    largest single differences are at the first tokens, whose sums hold few keys: 1.9e-4 of the
    value or root mean square in fp32, and that mean square itself in long bf16 sequences."""
    if case["op"] == "prefix":
        return {"rel": 1.2e-7, "max": 1e-6}
    if case["dtype"] == "fp32":
        return {"rel": 6e-6, "max": 1e-3}
    return {"rel": 0.025 if case["op"] in ("causal", "forward") else 0.013, "max": 0.99}


# ------------------------------------------------------------------ the same in 64 bits
def _hash(x, planes, inv_temp, K):
    """x [T,D] -> (P [T,S], th [T,L,K], corners [R,K]) in fp64."""
    L = planes.shape[0]
    th = torch.tanh(x @ planes.reshape(L * K, D).T).view(-1, L, K)
    bits = torch.arange(1 << K, device=x.device)[:, None] >> torch.arange(K - 1, -1, -1, device=x.device)
    corners = 2.0 * (bits & 1).to(torch.float64) - 1.0
    return torch.softmax(inv_temp * (th @ corners.T), dim=-1).reshape(x.shape[0], -1), th, corners


def _hash_grad(dP, P, th, corners, planes, inv_temp):
    """dP [T,S] -> (dx [T,D], d(inv_temp))."""
    T, L, K = th.shape
    P, dP = P.view(T, L, -1), dP.reshape(T, L, -1)
    dz = P * (dP - (P * dP).sum(-1, keepdim=True))
    du = dz @ corners
    return (inv_temp * du * (1 - th * th)).reshape(T, L * K) @ planes.reshape(L * K, D), (du * th).sum()


def _layer(q, k, v, g, planes, inv_temp, K, causal, *, kw=None, dden=None, glob=False, chunk=128):
    """One stream in fp64: q, k, v, g [T,D] (g None: forward only) -> dict of out, den, dq, dk, dv, dit.
    Chunks of tokens: a chunk's own triangle, and the sums of the chunks before (causal) or of all."""
    T = q.shape[0]
    PQ, thq, corners = _hash(q, planes, inv_temp, K)
    PK0, thk, _ = _hash(k, planes, inv_temp, K)
    PK = PK0 if kw is None else PK0 * kw[:, None]
    S = PQ.shape[1]
    n = -(-T // chunk) if causal else 1
    c = chunk if causal else T
    pad = n * c - T

    def cut(x):
        return torch.nn.functional.pad(x, (0, 0, 0, pad)).view(n, c, x.shape[1])

    pq, pk, vc = cut(PQ), cut(PK), cut(v)
    Bsum, Asum = pk.transpose(1, 2).contiguous() @ vc, pk.sum(1, keepdim=True)
    if causal:
        B0, A = Bsum.cumsum(0) - Bsum, Asum.cumsum(0) - Asum + pk.cumsum(1)
        tri = torch.ones(c, c, dtype=torch.float64, device=q.device).tril()
    else:
        B0, A = Bsum, Asum.expand(n, c, S)
    den = (pq * A).sum(-1)
    if glob:
        rd = 1.0 / den.clamp_min(EPS)
        W = pq * rd[..., None]
    else:
        W = pq / (A + EPS)
    out = W @ B0
    if causal:
        sc = (W @ pk.transpose(1, 2).contiguous()) * tri
        out = out + sc @ vc
    res = {"out": out.reshape(n * c, D)[:T], "den": den.reshape(n * c)[:T]}
    if g is None:
        return res
    gc = cut(g)
    h = torch.zeros(n, c, dtype=torch.float64, device=q.device) if dden is None else cut(dden[:, None])[..., 0]
    G = gc @ B0.transpose(1, 2).contiguous()
    if causal:
        m = (gc @ vc.transpose(1, 2).contiguous()) * tri
        G = G + m @ pk
    if glob:
        gd = h - torch.where(den >= EPS, rd * (gc * out).sum(-1), torch.zeros_like(rd))
        dPQ, dA = G * rd[..., None] + gd[..., None] * A, gd[..., None] * pq
    else:
        dPQ = G / (A + EPS)
        dA = -W * dPQ + h[..., None] * pq
        dPQ = dPQ + h[..., None] * A
    Usum, asum = W.transpose(1, 2).contiguous() @ gc, dA.sum(1, keepdim=True)
    if causal:
        U = Usum.flip(0).cumsum(0).flip(0) - Usum
        alpha = asum.flip(0).cumsum(0).flip(0) - asum + dA.flip(1).cumsum(1).flip(1)
        dv = pk @ U + sc.transpose(1, 2).contiguous() @ gc
        dPK = alpha + vc @ U.transpose(1, 2).contiguous() + m.transpose(1, 2).contiguous() @ W
    else:
        dv = pk @ Usum
        dPK = asum + vc @ Usum.transpose(1, 2).contiguous()
    dPK = dPK.reshape(n * c, S)[:T]
    if kw is not None:
        dPK = dPK * kw[:, None]
    res["dv"] = dv.reshape(n * c, D)[:T]
    res["dq"], dit_q = _hash_grad(dPQ.reshape(n * c, S)[:T], PQ, thq, corners, planes, inv_temp)
    res["dk"], dit_k = _hash_grad(dPK, PK0, thk, corners, planes, inv_temp)
    res["dit"] = dit_q + dit_k
    return res


@torch.no_grad()
def exact(case, seed):
    x = {n: t.to(torch.float64) for n, t in _inputs(case, seed).items()}
    op, M, B, T, H, K, L = (case[n] for n in ("op", "M", "B", "T", "H", "K", "L"))
    if op == "prefix":
        A = x["w"].cumsum(1) + EPS
        E = (x["w"][..., None] * x["v"]).cumsum(1) / A[..., None]
        gA = x["dout"] / A[..., None]
        beta = gA.flip(1).cumsum(1).flip(1)
        alpha = -(gA * E).sum(-1).flip(1).cumsum(1).flip(1)
        return {"out": E, "dw": (beta * x["v"]).sum(-1) + alpha, "dv": x["w"][..., None] * beta}
    if op == "probs":
        it = 1.0 / math.sqrt(D)
        P = torch.empty(M, B, H, T, L, 1 << K, dtype=torch.float64, device="cuda")
        dx = torch.empty_like(x["x"])
        for m, b, h in _streams(M, B, H):
            p, th, corners = _hash(x["x"][m, b, :, h], x["planes"][m], it, K)
            P[m, b, h] = p.view(T, L, -1)
            dx[m, b, :, h] = _hash_grad(x["dout"][m, b, h].reshape(T, -1), p, th, corners, x["planes"][m], it)[0]
        return {"probs": P, "dx": dx}
    shared = op in ("full", "padded")
    causal = op in ("forward", "causal", "global")
    # the learnable temperature is an fp32 parameter, log(temperature)
    logit = torch.tensor(math.log(TEMPERATURE), dtype=torch.float32).double().item()
    it = 1.0 / math.exp(logit) if shared else (1.0 if op == "global" else 1.0 / math.sqrt(D))
    out = torch.zeros(M, B, T, H, D, dtype=torch.float64, device="cuda")
    den = torch.zeros(M, B, H, T, dtype=torch.float64, device="cuda")
    grads = {n: torch.zeros_like(x[n]) for n in ("q", "k", "v")} if op != "forward" else {}
    dit = 0.0
    for m, b, h in _streams(M, B, H):
        at = (b, slice(None), h) if shared else (m, b, slice(None), h)
        q, k, v = x["q"][at], x["k"][at], x["v"][at]
        g = x["dout"][at] if op != "forward" else None
        kw = dden = None
        if op == "padded":
            kw = x["mask"][b]
            v, g = v * kw[:, None], g * kw[:, None]  # the mask on V and on the output
            dden = x["dden"][m, b, :, h] * kw        # den's clamp at eps is not met: its tokens have keys
        elif op == "global":
            dden = x["dden"][m, b, h]
        r = _layer(q, k, v, g, x["planes"][m], it, K, causal, kw=kw, dden=dden, glob=op == "global")
        if kw is not None:
            # a padded token's den is clamped at eps and passes no gradient (its dden was masked above)
            r["out"], r["den"], r["dv"] = r["out"] * kw[:, None], (r["den"] * kw).clamp_min(EPS), r["dv"] * kw[:, None]
        out[m, b, :, h], den[m, b, h] = r["out"], r["den"]
        if grads:
            for n in ("q", "k", "v"):
                grads[n][at] += r["d" + n]
            dit = dit + r["dit"]
    res = {"out": out}
    if op == "padded":
        res["den"] = den.permute(0, 1, 3, 2)
    elif op == "global":
        res["den"] = den
    res.update({"d" + n: t for n, t in grads.items()})
    if shared:
        res["dtemp"] = -dit * it  # d(1/exp(z))/dz
    return res


def _streams(M, B, H):
    return [(m, b, h) for m in range(M) for b in range(B) for h in range(H)]
