"""The gradient products on 128-wide tiles (sublayer_gemm.hip) beyond the sizes that the 64 x 64 tile
kernels take: feature tiles of 128 (256, 512, 640, 1024 features) and row chunks of different lengths,
against 64-bit products; and the phase encoder's launch of computeGradDx and the four weights there,
with the library's row products around it. Bars as in test_gpu_sublayer_tile.py."""
import numpy as np
import pytest

import oracle as O
from tests.attn_case import f32, to_gpu, to_np
from tests.sublayer_check import WEIGHT_GRADS, check_sublayer, exact_bf_err, f32_err, same_up_to_order

pytestmark = pytest.mark.gpu


def bf(rng, shape, scale=1.0):
    return O.f32_to_bf16((rng.standard_normal(shape) * scale).astype(np.float32))


def f64(a):
    return f32(a).astype(np.float64)


@pytest.mark.parametrize("R,H", [(7168, 8), (4480, 10), (1792, 16), (24064, 4)])
def test_dx_and_dw(gpu, R, H):
    import metalllm_amd as M
    import metalllm_amd.sublayer as S
    C = 64 * H
    print(f"case R={R} C={C}", flush=True)
    rng = np.random.default_rng(R + C)
    X, dK, dV = (bf(rng, (R, C)) for _ in range(3))
    dQ = rng.standard_normal((R, C)).astype(np.float32)
    Ws = [bf(rng, (C, C), 0.05) for _ in range(3)]
    p = M.AttentionParams.of(1, R, H, 64)
    tX, tQ, tK, tV, *tW = (to_gpu(a, gpu) for a in (X, dQ, dK, dV, *Ws))
    old = rng.standard_normal((R, C)).astype(np.float32)
    dX = to_gpu(old, gpu)
    S.computeGradDx(dX, *tW, tQ, tK, tV, p)
    d64 = dQ.astype(np.float64)
    exact = old + d64 @ f64(Ws[0]).T + f64(dK) @ f64(Ws[1]).T + f64(dV) @ f64(Ws[2]).T
    assert f32_err(to_np(dX), exact) <= 1e-5
    oq, ok, ov = rng.standard_normal((C, C)).astype(np.float32), bf(rng, (C, C), 10.0), bf(rng, (C, C), 10.0)
    dWq, dWk, dWv = (to_gpu(a, gpu) for a in (oq, ok, ov))
    S.computeGradDw(tX, tQ, tK, tV, dWq, dWk, dWv, p)
    assert f32_err(to_np(dWq), oq + f64(X).T @ d64) <= 1e-4
    assert exact_bf_err(to_np(dWk), f64(ok) + f64(X).T @ f64(dK)) == 0
    assert exact_bf_err(to_np(dWv), f64(ov) + f64(X).T @ f64(dV)) == 0


@pytest.mark.parametrize("R,H", [(18560, 8), (11776, 10), (4608, 16)])
def test_projection_dw(gpu, R, H):
    import metalllm_amd as M
    import metalllm_amd.sublayer as S
    C = 64 * H
    print(f"case R={R} C={C}", flush=True)
    rng = np.random.default_rng(2 * R + C)
    o, dZ, old = bf(rng, (R, C)), bf(rng, (R, C)), bf(rng, (C, C), 10.0)
    dWp = to_gpu(old, gpu)
    S.projBackwarddW(to_gpu(o, gpu), to_gpu(dZ, gpu), dWp, M.AttentionParams.of(1, R, H, 64))
    assert exact_bf_err(to_np(dWp), f64(old) + f64(o).T @ f64(dZ)) == 0


@pytest.mark.parametrize("B,T,H", [(28, 256, 8), (7, 256, 16), (70, 64, 10)])
def test_encoder(gpu, B, T, H):
    """Both phases against the entry points one by one: bit for bit apart from the weight gradients'
    summation order."""
    import torch
    import metalllm_amd.sublayer as S
    C = 64 * H
    print(f"case B={B} T={T} C={C}", flush=True)
    rng = np.random.default_rng(B + C)
    X, dOut = to_gpu(bf(rng, (B, T, C)), gpu), to_gpu(bf(rng, (B, T, C)), gpu)
    W = to_gpu(bf(rng, (4, C, C), 0.05), gpu)  # equally spaced: computeQKV as one batched call
    a, b = (S.Sublayer(X, *W.unbind(0), H=H) for _ in range(2))
    assert S.route(1, b.buffers(), b.p) & 2
    a.zero_grads()
    a.forward()
    a.backward(dOut)
    b.dOut.copy_(dOut)
    b.encode(0)
    b.encode(1)
    torch.cuda.synchronize()
    for n in ("q", "k", "v", "o", "lse", "out", "dO", "Dv", "dQ", "dK", "dV", "dX", *WEIGHT_GRADS):
        x, y = getattr(b, n), getattr(a, n)
        assert torch.equal(x, y) or n in WEIGHT_GRADS and same_up_to_order(n, to_np(x), to_np(y)), n
    check_sublayer(b, to_np(dOut), batches=[B - 1], label=f"encoder {(B, T, H, C)}")
