"""The sublayer's products on 64 x 64 tiles (sublayer_tile.hip) against the oracle at the sizes where
they can go wrong: row counts that end inside a tile, fewer units of k than waves, feature counts of
one tile and of an odd number of tiles, four and eight waves, row chunks with a second kernel, and the
gradients added into destinations that are not zero. Bars as in test_gpu_sublayer.py: bf16 within one
ulp plus 1e-5 of max, fp32 within 1e-4 of max."""
import numpy as np
import pytest

import oracle as O
from tests.attn_case import f32, to_gpu, to_np
from tests.sublayer_check import bf_err, exact_bf_err, f32_err

pytestmark = pytest.mark.gpu


def bf(rng, shape, scale=1.0):
    return O.f32_to_bf16((rng.standard_normal(shape) * scale).astype(np.float32))


@pytest.mark.parametrize("R,H", [(1, 1), (63, 2), (64, 1), (65, 3), (200, 5), (1344, 7), (2112, 6), (3008, 12)])
def test_row_products(gpu, R, H):
    import torch
    import metalllm_amd as M
    import metalllm_amd.sublayer as S
    C = 64 * H
    print(f"case R={R} C={C}", flush=True)
    rng = np.random.default_rng(R + C)
    X, dQ = bf(rng, (R, C)), (rng.standard_normal((R, C)) * 0.1).astype(np.float32)
    dK, dV = bf(rng, (R, C), 0.1), bf(rng, (R, C), 0.1)
    Ws = [bf(rng, (C, C), 0.05) for _ in range(4)]
    p = M.AttentionParams.of(1, R, H, 64)
    tX, tdQ, tdK, tdV, *tW = (to_gpu(a, gpu) for a in (X, dQ, dK, dV, *Ws))
    # outputs between guard rows that must stay as they are
    def guarded(dtype=torch.bfloat16):
        t = torch.full((R + 2, C), 7.0, dtype=dtype, device=gpu)
        return t, t[1:R + 1]
    (q0, q), (k0, k), (v0, v), (o0, out), (a0, dA) = (guarded() for _ in range(5))
    S.computeQKV(tX, q, k, v, *tW[:3], p)
    S.projForward(tX, tW[3], out, p)
    S.projBackwarddX(tX, tW[3], dA, p)
    x0, dX = guarded(torch.float32)
    S.computeGradDx(dX, *tW[:3], tdQ, tdK, tdV, p)
    for t in (q0, k0, v0, o0, a0, x0):
        assert (t[0] == 7).all() and (t[-1] == 7).all()
    ref = dict(zip(("q", "k", "v"), O.computeQKV(X, *Ws[:3], threads=16)))
    ref["out"] = O.projForward(X, Ws[3], threads=16)
    ref["dA"] = O.projBackwarddX(X, Ws[3], threads=16)
    for name, t in (("q", q), ("k", k), ("v", v), ("out", out), ("dA", dA)):
        bad, mx = bf_err(to_np(t), ref[name])
        print(f"  {name}: beyond bar {bad}, max err {mx:.3g}")
        assert bad == 0
    f = lambda a: f32(a).astype(np.float64)
    exact = 7.0 + dQ.astype(np.float64) @ f(Ws[0]).T + f(dK) @ f(Ws[1]).T + f(dV) @ f(Ws[2]).T
    assert f32_err(to_np(dX), exact) <= 1e-5  # added into 7; fp32 sums of 3 C terms


@pytest.mark.parametrize("R,H", [(64, 1), (128, 3), (448, 5), (1024, 2), (3840, 7), (8192, 1), (4096, 6), (2048, 12)])
def test_weight_gradients(gpu, R, H):
    import torch
    import metalllm_amd as M
    import metalllm_amd.sublayer as S
    C = 64 * H
    print(f"case R={R} C={C}", flush=True)
    rng = np.random.default_rng(2 * R + C)
    X, o, dK, dV, dZ = (bf(rng, (R, C)) for _ in range(5))
    dQ = rng.standard_normal((R, C)).astype(np.float32)
    p = M.AttentionParams.of(1, R, H, 64)
    t = {n: to_gpu(a, gpu) for n, a in dict(X=X, o=o, dK=dK, dV=dV, dZ=dZ, dQ=dQ).items()}
    old = {n: bf(rng, (C, C), 10.0) for n in ("dWk", "dWv", "dWp")}
    oldq = rng.standard_normal((C, C)).astype(np.float32)
    d = {n: to_gpu(a, gpu) for n, a in old.items()}
    dWq = to_gpu(oldq, gpu)
    S.projBackwarddW(t["o"], t["dZ"], d["dWp"], p)
    S.computeGradDw(t["X"], t["dQ"], t["dK"], t["dV"], dWq, d["dWk"], d["dWv"], p)
    f = lambda a: f32(a).astype(np.float64)
    assert f32_err(to_np(dWq), oldq + f(X).T @ dQ.astype(np.float64)) <= 1e-4
    for n, x, g in (("dWk", X, dK), ("dWv", X, dV), ("dWp", o, dZ)):
        assert exact_bf_err(to_np(d[n]), f(old[n]) + f(x).T @ f(g)) == 0, n


@pytest.mark.parametrize("B,T,H,D", [(1, 64, 1, 64), (1, 64, 3, 64), (3, 320, 5, 64), (2, 192, 3, 128), (16, 256, 7, 64),
                                     (64, 128, 1, 64),
                                     (40, 256, 6, 64)])  # projForward on tiles, the other row products not
def test_encoder(gpu, B, T, H, D):
    """Both phases through the encoder against the entry points one by one (bit for bit apart from the
    weight gradients' summation order), and a graph of each against the encoder."""
    import torch
    import metalllm_amd.sublayer as S
    from tests.sublayer_check import WEIGHT_GRADS, check_sublayer, same_up_to_order
    C = H * D
    print(f"case B={B} T={T} C={C} H={H}", flush=True)
    rng = np.random.default_rng(B + T + C)
    X, dOut = to_gpu(bf(rng, (B, T, C)), gpu), to_gpu(bf(rng, (B, T, C)), gpu)
    Ws = [to_gpu(bf(rng, (C, C), 0.05), gpu) for _ in range(4)]
    a, b = (S.Sublayer(X, *Ws, H=H) for _ in range(2))
    a.zero_grads()
    a.forward()
    a.backward(dOut)
    for t in (b.dQ, b.dX, b.dWq, b.dWk, b.dWv, b.dWp):
        t.fill_(float("nan"))
    b.dOut.copy_(dOut)
    b.encode(0)
    b.encode(1)
    names = ("q", "k", "v", "o", "lse", "out", "dO", "Dv", "dQ", "dK", "dV", "dX", "dWq", "dWk", "dWv", "dWp")
    torch.cuda.synchronize()
    got = {n: getattr(b, n).clone() for n in names}
    for n in names:
        assert (same_up_to_order(n, to_np(got[n]), to_np(getattr(a, n))) if n in WEIGHT_GRADS else
                torch.equal(got[n], getattr(a, n))), n
    check_sublayer(b, to_np(dOut), batches=[B - 1], label=f"encoder {(B, T, H, C)}")
    b.capture()
    for _ in range(2):
        for n in names:
            getattr(b, n).fill_(float("nan"))
        b.replay(0)
        b.replay(1)
        torch.cuda.synchronize()
        for n in names:
            assert torch.equal(getattr(b, n), got[n]), n
    b.close()
