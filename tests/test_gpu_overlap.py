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
