"""The work that a program using this package has it do, as cases that can be timed and checked.

Kinds of case, each one pass through public entry points on buffers the program keeps:
  forward       flashAttentionForward
  backward      computeD, then flashAttentionBackwardWorkspace (dQ written, workspace kept)
  backward_add  computeD, dQ zeroed, then flashAttentionBackward (the accumulating contract)
  block         both phases of the pre-LN block's attention half through the phase encoder
  products      the sublayer's six matrix products, each through its own entry point
  norm          layernormForward, layernormBackward and residualAdd

listed() holds the cases, draw(rng) gives another one of the same ranges, prepare(case, seed) the
program's state, run(state) one pass, work(case) the bytes and operations a pass cannot do without,
tolerance(case) how far two correct implementations may differ, and exact(case, seed) the same
outputs computed in 64 bits without this package.
"""
import math

import torch

import metalllm_amd as M
import metalllm_amd.glue as G
import metalllm_amd.sublayer as S

LN_EPS = 1e-5
MAX_ELEMS = 16 * 4096 * 16 * 128           # elements of q at the largest listed attention case
MAX_SCORES = 16 * 16 * 4096 * 4096 * 128   # B*H*T*T*D of that case
MAX_ROWS = 32768                           # activation rows of the block, product and norm cases


def listed():
    return [
        # one sequence of the reference's default training shape (it trains on one sequence at a
        # time, T = 256, 384 features, 6 heads): latency of a call
        {"name": "forward one sequence", "kind": "forward", "B": 1, "T": 256, "H": 6, "D": 64, "qk": 1.0},
        # the benchmark's GPT-2-small-like attention, with its peaky rows
        {"name": "forward batch", "kind": "forward", "B": 32, "T": 1024, "H": 12, "D": 64, "qk": 1.5},
        # prefill of one long prompt, 12 heads
        {"name": "forward long prompt", "kind": "forward", "B": 1, "T": 8192, "H": 12, "D": 64, "qk": 1.0},
        # the benchmark's long-context shape, 128-wide heads
        {"name": "forward wide", "kind": "forward", "B": 16, "T": 4096, "H": 16, "D": 128, "qk": 1.0},
        # the training shape with a large batch: many short sequences
        {"name": "backward short batch", "kind": "backward", "B": 128, "T": 256, "H": 6, "D": 64, "qk": 1.0},
        # the benchmark's long-context shape, backward
        {"name": "backward wide", "kind": "backward", "B": 16, "T": 4096, "H": 16, "D": 128, "qk": 1.0},
        # fine-tuning on one document of 47 tiles, five heads: odd sizes, the accumulating contract
        {"name": "backward one document", "kind": "backward_add", "B": 1, "T": 3008, "H": 5, "D": 128, "qk": 1.0},
        # a training step's attention half of a block, one sequence of the default training shape
        {"name": "block one sequence", "kind": "block", "B": 1, "T": 256, "H": 6, "D": 64},
        # the same on a small batch with feature and row counts that are not multiples of 128
        {"name": "block odd", "kind": "block", "B": 3, "T": 320, "H": 5, "D": 64},
        # the benchmark's sublayer shape, ordinary training
        {"name": "block batch", "kind": "block", "B": 8, "T": 2048, "H": 12, "D": 64},
        # the products called one by one, seven heads (448 features)
        {"name": "products", "kind": "products", "B": 4, "T": 960, "H": 7, "D": 64},
        # the norm and the residual around every sublayer, at the benchmark's activation size
        {"name": "norm", "kind": "norm", "R": 16384, "C": 768},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "backward", "backward", "backward_add", "block", "block", "products", "norm"])
    if kind == "norm":
        C = 8 * _log_int(rng, 16, 512)
        return {"kind": kind, "R": _log_int(rng, 64, max(64, min(2 * MAX_ROWS, 32768 * 1024 // C))), "C": C}
    D = rng.choice([64, 64, 128])
    if kind in ("block", "products"):
        T, H = 64 * _log_int(rng, 1, 32), rng.randint(2, 768 // D)
        return {"kind": kind, "B": _log_int(rng, 1, max(1, min(128, MAX_ROWS // T))), "T": T, "H": H, "D": D}
    T, H = 64 * _log_int(rng, 1, 128), rng.randint(1, 16)
    B = _log_int(rng, 1, max(1, min(128, MAX_ELEMS // (T * H * D), MAX_SCORES // (H * T * T * D))))
    return {"kind": kind, "B": B, "T": T, "H": H, "D": D, "qk": rng.choice([1.0, 1.5])}


def _rand(gen, shape, scale=1.0, add=0.0):
    return (torch.randn(shape, generator=gen, device="cuda") * scale + add).to(torch.bfloat16)


def _inputs(case, seed):
    """What the program is given: bf16 tensors (fp32 where an entry point takes fp32)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind == "norm":
        R, C = case["R"], case["C"]
        return {"x": _rand(gen, (R, C)), "dZ": _rand(gen, (R, C)), "gamma": _rand(gen, (C,), 0.1, 1.0),
                "beta": _rand(gen, (C,), 0.1)}
    B, T, H, D = case["B"], case["T"], case["H"], case["D"]
    if kind in ("forward", "backward", "backward_add"):
        shape = (B, T, H, D)
        i = {"q": _rand(gen, shape, case["qk"]), "k": _rand(gen, shape, case["qk"]), "v": _rand(gen, shape)}
        if kind != "forward":
            i["dO"] = _rand(gen, shape)
        return i
    C = H * D
    if kind == "block":
        return {"hidden": _rand(gen, (B, T, C)), "gamma": _rand(gen, (C,), 0.1, 1.0), "beta": _rand(gen, (C,), 0.1),
                "W": _rand(gen, (3, C, C), 0.02), "Wp": _rand(gen, (C, C), 0.02), "dOut": _rand(gen, (B, T, C))}
    i = {n: _rand(gen, (B, T, C)) for n in ("X", "o", "dOut", "dK", "dV")}
    i["dQ"] = torch.randn((B, T, C), generator=gen, device="cuda")
    i["W"], i["Wp"] = _rand(gen, (3, C, C), 0.02), _rand(gen, (C, C), 0.02)
    return i


def prepare(case, seed):
    kind, i = case["kind"], _inputs(case, seed)
    st = dict(i, kind=kind)
    if kind == "norm":
        R, C = case["R"], case["C"]
        st.update(xn=torch.empty_like(i["x"]), out=torch.empty_like(i["x"]), dx=torch.empty_like(i["x"]),
                  res=torch.empty_like(i["x"]), sd=torch.empty(R, device="cuda"), dgamma=torch.empty(C, device="cuda"),
                  dbeta=torch.empty(C, device="cuda"))
        return st
    B, T, H, D = case["B"], case["T"], case["H"], case["D"]
    if kind == "forward":
        st.update(out=torch.empty_like(i["q"]), lse=torch.empty((B, H, T), device="cuda"))
    elif kind in ("backward", "backward_add"):
        # the forward pass has run: its output and logsumexp are in hand
        st["out"], st["lse"] = M.attention_forward(i["q"], i["k"], i["v"])
        st.update(Dv=torch.empty_like(st["lse"]), dQ=torch.empty((B, T, H, D), device="cuda"),
                  dK=torch.empty_like(i["q"]), dV=torch.empty_like(i["q"]))
        if kind == "backward":
            st["ws"] = torch.empty((M.workspace_bytes(B, T, H, D),), dtype=torch.uint8, device="cuda")
    elif kind == "block":
        sub = S.Sublayer(None, *i["W"].unbind(0), i["Wp"], H=H, hidden=i["hidden"], ln_gamma=i["gamma"], ln_beta=i["beta"],
                         ln_eps=LN_EPS)
        sub.dOut.copy_(i["dOut"])
        S.reserve(sub.p)
        st.update(sub=sub, bufs=sub.buffers())
    else:
        C = H * D
        st["p"] = M.AttentionParams.of(B, T, H, D)
        st["qkv"] = torch.empty((3, B, T, C), dtype=torch.bfloat16, device="cuda")
        st.update(out=torch.empty_like(i["X"]), dAttn=torch.empty_like(i["X"]), dX=torch.empty((B, T, C), device="cuda"),
                  dWq=torch.empty((C, C), device="cuda"))
        st.update({n: torch.empty_like(i["Wp"]) for n in ("dWk", "dWv", "dWp")})
    return st


def run(s):
    kind = s["kind"]
    if kind == "forward":
        M.flashAttentionForward(s["q"], s["k"], s["v"], s["out"], s["lse"])
        return {"out": s["out"], "lse": s["lse"]}
    if kind == "backward":
        M.computeD(s["dO"], s["out"], s["Dv"])
        M.flashAttentionBackwardWorkspace(s["dO"], s["Dv"], s["lse"], s["q"], s["k"], s["v"], s["dQ"], s["dK"], s["dV"],
                                          s["ws"])
        return {"D": s["Dv"], "dQ": s["dQ"], "dK": s["dK"], "dV": s["dV"]}
    if kind == "backward_add":
        M.computeD(s["dO"], s["out"], s["Dv"])
        s["dQ"].zero_()  # the entry point adds into dQ
        M.flashAttentionBackward(s["dO"], s["Dv"], s["lse"], s["q"], s["k"], s["v"], s["dQ"], s["dK"], s["dV"])
        return {"D": s["Dv"], "dQ": s["dQ"], "dK": s["dK"], "dV": s["dV"]}
    if kind == "block":
        sub = s["sub"]
        S.encode_phase(0, s["bufs"], sub.p)
        S.encode_phase(1, s["bufs"], sub.p)
        return {"residual": sub.residual, "attn": sub.o, "lse": sub.lse, "dStream": sub.dStream, "dX": sub.dX,
                "dWq": sub.dWq, "dWk": sub.dWk, "dWv": sub.dWv, "dWp": sub.dWp, "dgamma": sub.ln_dgamma,
                "dbeta": sub.ln_dbeta}
    if kind == "products":
        p, W = s["p"], s["W"]
        q, k, v = s["qkv"].unbind(0)
        S.computeQKV(s["X"], q, k, v, W[0], W[1], W[2], p)
        S.projForward(s["o"], s["Wp"], s["out"], p)
        for n in ("dX", "dWq", "dWk", "dWv", "dWp"):  # the gradient products add into these
            s[n].zero_()
        S.projBackwarddW(s["o"], s["dOut"], s["dWp"], p)
        S.projBackwarddX(s["dOut"], s["Wp"], s["dAttn"], p)
        S.computeGradDx(s["dX"], W[0], W[1], W[2], s["dQ"], s["dK"], s["dV"], p)
        S.computeGradDw(s["X"], s["dQ"], s["dK"], s["dV"], s["dWq"], s["dWk"], s["dWv"], p)
        return {n: s[n] for n in ("qkv", "out", "dAttn", "dX", "dWq", "dWk", "dWv", "dWp")}
    G.layernormForward(s["x"], s["xn"], s["out"], s["gamma"], s["beta"], s["sd"], LN_EPS)
    s["dx"].copy_(s["dZ"])  # the backward works in place
    s["dgamma"].zero_()
    s["dbeta"].zero_()
    G.layernormBackward(s["dx"], s["xn"], s["gamma"], s["sd"], s["dgamma"], s["dbeta"])
    G.residualAdd(s["out"], s["x"], s["res"])
    return {n: s[n] for n in ("xn", "out", "sd", "dx", "dgamma", "dbeta", "res")}


def work(case):
    """Causal attention counts half of the dense products: forward 2, backward 5 products' worth of
    B*H*T*T*D (the recomputed scores among them)."""
    kind = case["kind"]
    if kind == "norm":
        R, C = case["R"], case["C"]
        # x in, x_norm and out; dZ in, dx out; res; the weights and column sums are small
        return {"bytes": 12 * R * C + 4 * R + 12 * C, "flops": 30 * R * C}
    B, T, H, D = case["B"], case["T"], case["H"], case["D"]
    e, stat, att = B * T * H * D, B * H * T, B * H * T * T * D
    if kind == "forward":
        return {"bytes": 8 * e + 4 * stat, "flops": 2 * att}
    if kind in ("backward", "backward_add"):
        # q, k, v, out, dO in; dQ (fp32), dK, dV out; lse in, D out
        return {"bytes": 18 * e + 8 * stat, "flops": 5 * att + 2 * e}
    R, C = B * T, H * D
    if kind == "block":
        # hidden and dOut in, residual and dStream out, the outputs kept for the caller (attn, lse,
        # dX); q, k, v, x_norm and their gradients are the path's own but are written for the
        # backward phase, which is another call; weights in and their gradients out
        return {"bytes": (2 + 2 + 2 + 2 + 2 + 4) * R * C + 2 * 5 * R * C + 4 * stat + (8 + 10) * C * C,
                "flops": 24 * R * C * C + 7 * att}
    # X, o, dOut, dK, dV (bf16) and dQ (fp32) in; q, k, v, out, dAttn (bf16) and dX (fp32) out
    return {"bytes": (10 + 4 + 10 + 4) * R * C + (8 + 10) * C * C, "flops": 24 * R * C * C}


def tolerance(case):
    """About four times the largest relative error (2-norm over an output) measured against exact()
    over the ranges: norm 0.0026 (bf16 products summed per column), products 0.0017 (one bf16
    rounding), forward 0.014 (bf16 scores at T = 8192, Q and K times 1.5; 0.003-0.005 with unscaled
    ones), block 0.009. The backward's dK and dV reach 0.019 at T = 8192, where they have been rounded
    to bf16 after each of 128 query tiles; an implementation that does not round there differs from
    one that does by as much, and twice that is allowed."""
    return {"rel": {"norm": 1e-2, "products": 7e-3, "forward": 3e-2, "block": 3e-2, "backward": 4e-2,
                    "backward_add": 4e-2}[case["kind"]]}


def _heads(x):
    """[B, T, H, D] -> iterator of (b, h, [T, D] fp64)."""
    for b in range(x.shape[0]):
        for h in range(x.shape[2]):
            yield b, h


def _attention64(q, k, v, dO=None):
    """Causal attention of [B, T, H, D] inputs in 64 bits, one head at a time; with dO also D and the
    gradients. Returns tensors laid out as the entry points' (outputs in fp32, which holds far more
    digits than the tolerances)."""
    B, T, H, D = q.shape
    f32 = lambda *shape: torch.empty(shape, device="cuda")
    r = {"out": f32(B, T, H, D), "lse": f32(B, H, T)}
    if dO is not None:
        r.update(D=f32(B, H, T), dQ=f32(B, T, H, D), dK=f32(B, T, H, D), dV=f32(B, T, H, D))
    scale = 1.0 / math.sqrt(D)
    mask = torch.ones((T, T), dtype=torch.bool, device="cuda").triu_(1)
    for b, h in _heads(q):
        Q, K, V = (x[b, :, h].double() for x in (q, k, v))
        s = (Q @ K.t()).mul_(scale).masked_fill_(mask, float("-inf"))
        lse = torch.logsumexp(s, 1)
        P = s.sub_(lse[:, None]).exp_()
        O = P @ V
        r["out"][b, :, h], r["lse"][b, h] = O, lse
        if dO is not None:
            g = dO[b, :, h].double()
            Dv = (g * O).sum(1)
            r["D"][b, h], r["dV"][b, :, h] = Dv, P.t() @ g
            dS = (g @ V.t()).sub_(Dv[:, None]).mul_(P).mul_(scale)
            r["dQ"][b, :, h], r["dK"][b, :, h] = dS @ K, dS.t() @ Q
    return r


def _norm64(x, gamma, beta):
    mean = x.mean(-1, keepdim=True)
    sd = ((x - mean).square().mean(-1, keepdim=True) + LN_EPS).sqrt()
    xn = (x - mean) / sd
    return xn, xn * gamma + beta, sd


def _norm_backward64(dZ, xn, gamma, sd):
    d = dZ * gamma
    dx = (d - d.mean(-1, keepdim=True) - xn * (d * xn).mean(-1, keepdim=True)) / sd
    C = dZ.shape[-1]
    return dx, (dZ * xn).reshape(-1, C).sum(0), dZ.reshape(-1, C).sum(0)


def exact(case, seed):
    kind, i = case["kind"], _inputs(case, seed)
    if kind == "forward":
        return _attention64(i["q"], i["k"], i["v"])
    if kind in ("backward", "backward_add"):
        r = _attention64(i["q"], i["k"], i["v"], i["dO"])
        return {n: r[n] for n in ("D", "dQ", "dK", "dV")}
    d = {n: t.double() for n, t in i.items()}
    if kind == "norm":
        xn, out, sd = _norm64(d["x"], d["gamma"], d["beta"])
        dx, dg, db = _norm_backward64(d["dZ"], xn, d["gamma"], sd)
        return {"xn": xn, "out": out, "sd": sd[:, 0], "dx": dx, "dgamma": dg, "dbeta": db, "res": out + d["x"]}
    B, T, H, D = case["B"], case["T"], case["H"], case["D"]
    C, W, Wp = H * D, d["W"], d["Wp"]
    flat = lambda x: x.reshape(B * T, C)
    if kind == "products":
        X, o, g, dQ, dK, dV = (flat(d[n]) for n in ("X", "o", "dOut", "dQ", "dK", "dV"))
        shape = (B, T, C)
        return {"qkv": torch.stack([X @ w for w in W]).view(3, *shape), "out": (o @ Wp).view(shape),
                "dAttn": (g @ Wp.t().contiguous()).view(shape),
                "dX": sum(t @ w.t().contiguous() for t, w in zip((dQ, dK, dV), W)).view(shape),
                "dWq": X.t().contiguous() @ dQ, "dWk": X.t().contiguous() @ dK, "dWv": X.t().contiguous() @ dV,
                "dWp": o.t().contiguous() @ g}
    xn, x, sd = _norm64(d["hidden"], d["gamma"], d["beta"])
    X, g = flat(x), flat(d["dOut"])
    dAttn = g @ Wp.t().contiguous()
    four = lambda t: t.reshape(B, T, H, D)
    a = _attention64(*(four(X @ w) for w in W), four(dAttn))
    o, dQ, dK, dV = (flat(a[n].double()) for n in ("out", "dQ", "dK", "dV"))
    dX = sum(t @ w.t().contiguous() for t, w in zip((dQ, dK, dV), W))
    dh, dg, db = _norm_backward64(dX.view(B, T, C), xn, d["gamma"], sd)
    Xt = X.t().contiguous()
    return {"residual": d["hidden"] + (o @ Wp).view(B, T, C), "attn": o.view(B, T, C), "lse": a["lse"],
            "dStream": dh + d["dOut"], "dX": dX.view(B, T, C), "dWq": Xt @ dQ, "dWk": Xt @ dK, "dWv": Xt @ dV,
            "dWp": o.t().contiguous() @ g, "dgamma": dg, "dbeta": db}
