"""Calls whose buffers share memory: a destination in the memory of an operand that the call, or the
calls of a phase before it, has finished with. The kernels that join several products in one launch
need their destinations apart from what they read; these calls run one product after another and
must give what they give on separate buffers. Feature counts are no multiples of 128 where a joint
launch on 128-wide tiles would need the same (those calls read and write in one launch by contract).
Bars as in test_gpu_sublayer_tile.py."""
import numpy as np
import pytest

import oracle as O
from tests.attn_case import bf16_ulp, f32, to_gpu, to_np
from tests.sublayer_check import bf_err, exact_bf_err, f32_err

pytestmark = pytest.mark.gpu


def bf(rng, shape, scale=1.0):
    return O.f32_to_bf16((rng.standard_normal(shape) * scale).astype(np.float32))


def f64(a):
    return f32(a).astype(np.float64)


@pytest.fixture(scope="module")
def S():
    import metalllm_amd.sublayer as S
    return S


@pytest.mark.parametrize("R,H", [(320, 5), (1024, 3)])
def test_products(gpu, S, R, H):
    import metalllm_amd as M
    C = 64 * H
    print(f"case R={R} C={C}", flush=True)
    rng = np.random.default_rng(R + C)
    X, o, dZ, dK, dV = (bf(rng, (R, C)) for _ in range(5))
    dQ = rng.standard_normal((R, C)).astype(np.float32)
    Ws = [bf(rng, (C, C), 0.05) for _ in range(3)]
    p = M.AttentionParams.of(1, R, H, 64)
    g = lambda a: to_gpu(a, gpu)
    tX, to, tZ, tdQ, tdK, tdV, *tW = (g(a) for a in (X, o, dZ, dQ, dK, dV, *Ws))
    # dX in dQ's memory: dQ + dQ.Wq^T + dK.Wk^T + dV.Wv^T
    dX = tdQ.clone()
    S.computeGradDx(dX, *tW, dX, tdK, tdV, p)
    exact = dQ + dQ.astype(np.float64) @ f64(Ws[0]).T + f64(dK) @ f64(Ws[1]).T + f64(dV) @ f64(Ws[2]).T
    assert f32_err(to_np(dX), exact) <= 1e-5
    # one destination for dKw and dVw: both sums, each rounded to bf16
    old = bf(rng, (C, C), 10.0)
    dWq, dW = g(np.zeros((C, C), np.float32)), g(old)
    S.computeGradDw(tX, tdQ, tdK, tdV, dWq, dW, dW, p)
    assert f32_err(to_np(dWq), f64(X).T @ dQ.astype(np.float64)) <= 1e-4
    first = f64(old) + f64(X).T @ f64(dK)
    both = first + f64(X).T @ f64(dV)
    # half an ulp of each of the two rounded sums, and a tenth for the fp32 sums behind them
    bar = 0.6 * (bf16_ulp(first.astype(np.float32)) + bf16_ulp(both.astype(np.float32))) + 1e-5 * np.abs(both).max()
    assert (np.abs(f64(to_np(dW)) - both) <= bar).all()
    # dQw in dQ's memory, dVw in dV's
    q2, v2 = tdQ.clone(), tdV.clone()
    dWq, dWv, dWk = q2.view(-1)[:C * C].view(C, C), v2.view(-1)[:C * C].view(C, C), g(old)
    S.computeGradDw(tX, q2, tdK, v2, dWq, dWk, dWv, p)
    head = lambda a: a.reshape(-1)[:C * C].reshape(C, C)
    assert f32_err(to_np(dWq), head(dQ) + f64(X).T @ dQ.astype(np.float64)) <= 1e-4
    assert exact_bf_err(to_np(dWk), f64(old) + f64(X).T @ f64(dK)) == 0
    assert exact_bf_err(to_np(dWv), head(f64(dV)) + f64(X).T @ f64(dV)) == 0
    # dProjw in dZ's memory
    z2 = tZ.clone()
    dWp = z2.view(-1)[:C * C].view(C, C)
    S.projBackwarddW(to, z2, dWp, p)
    assert exact_bf_err(to_np(dWp), head(f64(dZ)) + f64(o).T @ f64(dZ)) == 0
    # k in q_w's memory: q is complete by then
    import torch
    mem = torch.empty((max(R, C), C), dtype=torch.bfloat16, device=gpu)
    qw, k = mem[:C], mem[:R]
    qw.copy_(tW[0])
    q, v = (torch.empty((R + 8 * i, C), dtype=torch.bfloat16, device=gpu)[:R] for i in (0, 1))
    S.computeQKV(tX, q, k, v, qw, tW[1], tW[2], p)
    for name, t, r in zip("qkv", (q, k, v), O.computeQKV(X, *Ws, threads=16)):
        bad, mx = bf_err(to_np(t), r)
        assert bad == 0, (name, mx)


# (buffer, buffers whose memory it takes, in a row): each allowed by the order of the phase's calls
REUSE = [("dK", ["attn_out"]), ("dV", ["attn_out"]), ("dK", ["dOut"]), ("dQ", ["attn_out", "dOut"]), ("dX", ["dOut", "attn_out"]),
         ("Dsum", ["dOut"]), ("dKw", ["q_w"]), ("dX", ["q", "k"]), ("dX_bf16", ["dAttn"]), ("dX", ["dQ"])]


@pytest.mark.parametrize("B,T,H", [(3, 320, 5), (2, 256, 6), (1, 64, 1)])
def test_encoder_backward(gpu, S, B, T, H):
    """Phase 1, eager and as a graph, with an output in the memory of buffers that no later call of the
    phase reads, against the same phase on separate buffers. (dX over dQ is read later, by
    computeGradDw: only where the library path runs, from its split of dQ.)"""
    import torch
    C = 64 * H
    rng = np.random.default_rng(B * T + C)
    g = lambda shape, sc=1.0: to_gpu(bf(rng, shape, sc), gpu)
    sub = S.Sublayer(g((B, T, C)), *[g((C, C), 0.05) for _ in range(4)], H=H)
    sub.dOut.copy_(g((B, T, C)))
    sub.encode(0)
    sub.encode(1)
    torch.cuda.synchronize()
    names = dict(dAttn="dO", Dsum="Dv", dQ="dQ", dK="dK", dV="dV", dX="dX", dQw="dWq", dKw="dWk", dVw="dWv", dProjw="dWp",
                 dX_bf16="dXb", attn_out="o", dOut="dOut", q="q", k="k", q_w="Wq")
    keep = {n: getattr(sub, a).clone() for n, a in names.items()}
    for out, into in REUSE:
        if (out, into) == ("dX", ["dQ"]) and C % 128 == 0:
            continue
        print(f"case B={B} T={T} C={C} {out} in {'+'.join(into)}", flush=True)
        inputs = {n: keep[n] for n in ("attn_out", "dOut", "q", "k", "q_w")}
        mem = torch.empty(max(sum(keep[n].nbytes for n in into), keep[out].nbytes), dtype=torch.uint8, device=gpu)
        views, at = {}, 0
        for n in into:
            views[n] = mem[at:at + keep[n].nbytes].view(keep[n].dtype).view(keep[n].shape)
            at += keep[n].nbytes
        views[out] = mem[:keep[out].nbytes].view(keep[out].dtype).view(keep[out].shape)
        b = sub.buffers()
        for n, v in views.items():
            setattr(b, n, v.data_ptr())

        def check(run, what):
            for n, a in names.items():
                if n not in inputs:
                    getattr(sub, a).fill_(float("nan"))
            for n, v in inputs.items():
                (views[n] if n in views else getattr(sub, names[n])).copy_(v)
            run()
            torch.cuda.synchronize()
            for n, a in names.items():
                if n in inputs or n in into:
                    continue
                got, ref = to_np(views.get(n, getattr(sub, a))), to_np(keep[n])
                if got.dtype == np.float32:
                    assert f32_err(got, ref) <= (1e-4 if n == "dQw" else 1e-5), (what, n)
                else:
                    assert bf_err(got, ref)[0] == 0, (what, n)

        check(lambda: S.encode_phase(1, b, sub.p), "eager")
        graph = S.PhaseGraph(1, b, sub.p)
        for _ in range(2):
            check(graph.launch, "graph")
        graph.close()
        for n, v in inputs.items():
            getattr(sub, names[n]).copy_(v)


@pytest.mark.parametrize("B,T,H,D,into", [(2, 512, 4, 128, {"dV": "v"}), (1, 192, 3, 128, {"dQ": "q"}), (3, 576, 4, 128, {"dQ": "v", "dV": "v"}),
                                          (1, 256, 6, 64, {"dV": "v", "dK": "k"}), (2, 128, 3, 64, {"dV": "v", "dK": "k"}),
                                          (1, 192, 5, 64, {"dK": "k"})])
def test_attention_backward(gpu, B, T, H, D, into):
    """flashAttentionBackwardWorkspace with an output in the memory of an input (dQ, twice as long, also
    in dZ's behind it; where dV is in v's as well, dQ in q's and dZ's) against separate buffers: dK and dV
    bit for bit, dQ up to fp32 summation order. At D = 64 flashAttentionBackward as well."""
    import torch
    import metalllm_amd as M
    from tests.attn_case import make_inputs
    print(f"case B={B} T={T} H={H} D={D} {into}", flush=True)
    q, k, v, g = (to_gpu(x, gpu) for x in make_inputs(B, T, H, D, 31))
    out, lse = M.attention_forward(q, k, v)
    Dv = torch.empty_like(lse)
    M.computeD(g, out, Dv)
    ws = torch.empty((M.workspace_bytes(B, T, H, D),), dtype=torch.uint8, device=gpu)
    new = lambda: (torch.zeros((B, T, H, D), device=gpu), torch.empty_like(q), torch.empty_like(q))
    ref = new()
    M.flashAttentionBackwardWorkspace(g, Dv, lse, q, k, v, *ref, ws)
    for entry in ("workspace", "add") if D == 64 else ("workspace",):
        mem = torch.empty((4,) + q.shape, dtype=torch.bfloat16, device=gpu)  # q or v, dZ, then the others
        first = "q" if into.get("dQ") != "v" or "dV" in into else "v"
        i = dict(zip((first, "dZ", "v" if first == "q" else "q", "k"), mem.unbind(0)))
        for n, t in (("q", q), ("k", k), ("v", v), ("dZ", g)):
            i[n].copy_(t)
        dQ, dK, dV = new()
        if "dQ" in into:
            dQ = mem[:2].view(torch.float32).view(q.shape)
        dK, dV = i["k"] if "dK" in into else dK, i["v"] if "dV" in into else dV
        if entry == "workspace":
            M.flashAttentionBackwardWorkspace(i["dZ"], Dv, lse, i["q"], i["k"], i["v"], dQ, dK, dV, ws)
        else:
            M.flashAttentionBackward(i["dZ"], Dv, lse, i["q"], i["k"], i["v"], dQ, dK, dV)
        torch.cuda.synchronize()
        assert torch.equal(dK, ref[1]) and torch.equal(dV, ref[2])
        assert (dQ - ref[0]).abs().max().item() <= 1e-5 * ref[0].abs().max().item()
