"""The backward's launches by shape: dK/dV and dQ in one launch (whole grids resident, with the dQ
blocks of every second row of ids reversed, by XCD octets and not; more workgroups than are
resident), the stored-dS path at D = 128 beyond two blocks per CU, and the fused kernel of whole
rounds of T = 256 pairs. Every shape goes through both entry points against the oracle at the bars of
test_gpu_parity.py (outputs start as NaN where they are written in full)."""
import numpy as np
import pytest

from tests.attn_case import gpu_backward, gpu_compute_d, gpu_forward, make_inputs
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
    (122, 256, 2, 64, 1),    # 244 pairs: the fused T = 256 kernel, one round 95% full
    (121, 256, 2, 64, 1),    # 242 pairs: below that line
])
def test_launch_forms(gpu, B, T, H, D, b_end):
    check_case(gpu, B, T, H, D, 1.0, 211, b_end=b_end)


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
