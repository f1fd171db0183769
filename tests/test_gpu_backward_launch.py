"""The backward's launches by shape: dK/dV and dQ in one launch (whole grids resident, with the dQ
blocks of every second row of ids reversed, by XCD octets and not; more workgroups than are
resident), the stored-dS path at D = 128 beyond two blocks per CU, and the fused kernel of nearly
full rounds of pairs at T = 128 to 256. Every shape goes through both entry points against the oracle at the bars of
test_gpu_parity.py (outputs start as NaN where they are written in full)."""
import numpy as np
import pytest

from tests.attn_case import gpu_backward, gpu_compute_d, gpu_forward, make_inputs, to_gpu
from tests.test_gpu_parity import check_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,D,b_end", [
    (1, 1984, 11, 64, 1),    # 176 + 176 workgroups, ids reversed one by one
    (16, 192, 12, 64, 2),    # 384 + 384, reversed in octets
    (7, 192, 23, 64, 1),     # 322 + 322, last row partial
    (3, 960, 11, 128, 1),    # 264 + 264: more than two per CU, in list order
    (65, 448, 2, 128, 1),    # 520 blocks: dS stored, two-tile dQ ring
    (23, 256, 8, 128, 1),    # 368 blocks: below the line of T < 512 (384)
    (25, 256, 8, 128, 1),    # 400 blocks: above it
    (9, 576, 13, 128, 1),    # 585 blocks: dS stored, four-tile ring, last item 1 of 4 tiles
    (122, 256, 2, 64, 1),    # 244 pairs: the fused kernel, one round 95% full
    (121, 256, 2, 64, 1),    # 242 pairs: the same, 94.5%
    (119, 256, 2, 64, 1),    # 238 pairs: below the line
    (128, 192, 4, 64, 1),    # 512 pairs: the fused kernel, three query tiles, two full rounds
    (205, 128, 5, 64, 1),    # 1025 pairs: 82% of five rounds, below the line
    (244, 128, 5, 64, 1),    # 1220 pairs: the fused kernel, two query tiles, the last of five rounds partly full
])
def test_launch_forms(gpu, B, T, H, D, b_end):
    check_case(gpu, B, T, H, D, 1.0, 211, b_end=b_end)


# D = 128 beyond the lines of the joint launch: dK/dV storing dS, then the dQ ring of two query tiles an
# item (T < 512) or four, with last items of one to all of them
STORED = [(193, 64, 2), (97, 192, 2), (65, 320, 2), (65, 448, 2), (49, 256, 8), (17, 512, 8), (15, 576, 7), (26, 640, 4),
          (22, 704, 4)]


@pytest.mark.parametrize("B,T,H", STORED)
def test_stored_ds(gpu, B, T, H):
    import metalllm_amd.attention as A
    assert A.backward_route(B, T, H, 128, True) == A.STORED
    check_case(gpu, B, T, H, 128, 1.5 if T == 320 else 1.0, 214, b_end=1)


@pytest.mark.parametrize("B,T,H", [(65, 448, 2), (17, 512, 8)])
def test_stored_parts_equal_the_entry_point(gpu, B, T, H):
    """The bench hook's parts 2 and 3 where they store dS: flashAttentionBackwardWorkspace bit for bit."""
    import torch
    import metalllm_amd as M
    q, k, v, g = (to_gpu(x, gpu) for x in make_inputs(B, T, H, 128, 215))
    out, lse = M.attention_forward(q, k, v)
    Dv = torch.empty_like(lse)
    M.computeD(g, out, Dv)
    res = []
    for parts in (False, True):
        ws = torch.full((M.workspace_bytes(B, T, H, 128),), 0x7F, dtype=torch.uint8, device=gpu)
        r = [torch.full(q.shape, float("nan"), device=gpu), torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))]
        if parts:
            M.backward_part(2, g, Dv, lse, q, k, v, *r, workspace=ws)
            assert torch.isnan(r[0]).all()  # dQ comes from the stored dS alone
            M.backward_part(3, g, Dv, lse, q, k, v, *r, workspace=ws)
        else:
            M.flashAttentionBackwardWorkspace(g, Dv, lse, q, k, v, *r, ws)
        res.append(r)
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,T,H", [(247, 256, 2), (241, 192, 2), (244, 128, 5)])
def test_fused_kernel_adds(gpu, B, T, H):
    """flashAttentionBackward's contract in the fused kernel, more pairs than one round: dQ starts at
    values that are not zero and ends at those plus the gradient (one fp32 addition each)."""
    import torch
    import metalllm_amd as M
    import metalllm_amd.attention as A
    assert A.backward_route(B, T, H, 64, False) == A.FUSED
    q, k, v, g = (to_gpu(x, gpu) for x in make_inputs(B, T, H, 64, 213))
    out, lse = M.attention_forward(q, k, v)
    Dv = torch.empty_like(lse)
    M.computeD(g, out, Dv)
    ws = torch.empty((M.workspace_bytes(B, T, H, 64),), dtype=torch.uint8, device=gpu)
    dQ, dK, dV = torch.full((B, T, H, 64), float("nan"), device=gpu), torch.empty_like(q), torch.empty_like(q)
    M.flashAttentionBackwardWorkspace(g, Dv, lse, q, k, v, dQ, dK, dV, ws)
    old = torch.randn((B, T, H, 64), generator=torch.Generator(gpu).manual_seed(5), device=gpu)
    dQ2, dK2, dV2 = old.clone(), torch.empty_like(q), torch.empty_like(q)
    M.flashAttentionBackward(g, Dv, lse, q, k, v, dQ2, dK2, dV2)
    torch.cuda.synchronize()
    assert torch.equal(dQ2, old + dQ)
    assert torch.equal(dK, dK2) and torch.equal(dV, dV2)


def test_short_kernel_agrees_with_both(gpu):
    """One batch of 244 pairs' T = 256 backward (fused kernel) alone (one-launch form): dK and dV bit
    for bit, dQ up to fp32 summation order."""
    q, k, v, g = make_inputs(122, 256, 2, 64, 212)
    out, lse = gpu_forward(q, k, v, gpu)
    Dv = gpu_compute_d(g, out, gpu)
    one = lambda x: np.ascontiguousarray(x[3:4])
    for ws in (False, True):
        full = gpu_backward(g, Dv, lse, q, k, v, gpu, workspace=ws)
        got = gpu_backward(one(g), one(Dv), one(lse), one(q), one(k), one(v), gpu, workspace=ws)
        assert np.array_equal(got[1], full[1][3:4]) and np.array_equal(got[2], full[2][3:4])
        assert np.abs(got[0] - full[0][3:4]).max() <= 1e-5 * np.abs(full[0]).max()
