"""Which kernels a backward call runs (host decision, no GPU)."""
import pytest

import metalllm_amd.attention as A

NAMES = ("dZ", "d", "l", "q", "k", "v", "dQ", "dK", "dV")


def at(B, T, H, D, **same):
    """Addresses of the nine buffers right behind one another, with `same` (name=(other, byte offset))."""
    e, stat, pos, r = B * T * H * D, B * H * T, 1 << 40, {}
    for n in NAMES:
        r[n] = pos
        pos += {"d": 4 * stat, "l": 4 * stat, "dQ": 4 * e}.get(n, 2 * e)
    for n, (other, off) in same.items():
        r[n] = r[other] + off
    return [r[n] for n in NAMES]


@pytest.mark.parametrize("B,T,H,D", [(1, 256, 6, 64), (2, 1024, 4, 64), (2, 512, 4, 128), (1, 64, 1, 64)])
def test_joint_launch_needs_outputs_apart(B, T, H, D):
    """Outputs that hold a byte of an input do not go to the joint launch: the kernels are then those of
    the shape alone (fused up to T = 256 at D = 64, else two, with the dS store at D = 128)."""
    e = B * T * H * D
    for ws in (False, True):
        other = A.FUSED if D == 64 and T <= 256 else A.STORED if ws and D == 128 else A.TWO
        assert A.backward_route(B, T, H, D, ws, at(B, T, H, D)) == A.JOINT
        for out in ("dQ", "dK", "dV"):
            for inp in ("dZ", "d", "l", "q", "k", "v"):
                size = 4 * e if out == "dQ" else 2 * e
                for off in (0, 16 - size):  # the input's first bytes: by the output's first, by its last
                    assert A.backward_route(B, T, H, D, ws, at(B, T, H, D, **{out: (inp, off)})) == other, (out, inp, off)


@pytest.mark.parametrize("T,pairs,fused", [
    (256, 239, True), (256, 238, False), (256, 256, True), (256, 257, False), (256, 477, True), (256, 476, False),
    (256, 1367, False), (256, 1379, True), (256, 6144, True), (256, 6, False),
    (192, 256, False), (192, 461, True), (192, 460, False), (192, 768, True), (192, 1824, True), (192, 1612, False),
    (128, 768, False), (128, 1024, True), (128, 1216, True), (128, 1215, False), (128, 2600, False), (128, 2817, True),
    (64, 6144, False), (320, 1024, False)])
def test_fused_kernel_lines(T, pairs, fused):
    """The fused kernel takes the same time for each round of 256 pairs, full or not: it runs where the
    rounds are nearly full, from one round at T = 256, two at 192 and four at 128 on."""
    for ws in (False, True):
        assert A.backward_route(pairs, T, 1, 64, ws) == (A.FUSED if fused else A.JOINT)
        assert A.backward_route(1, T, pairs, 128, ws) != A.FUSED


@pytest.mark.parametrize("B,T,H,stored", [(4, 128, 96, False), (385, 128, 1, True), (16, 512, 8, False), (129, 512, 1, True),
                                          (1, 8192, 8, False), (1, 8192, 9, True), (65, 320, 2, True)])
def test_stored_ds_lines(B, T, H, stored):
    """At D = 128 the workspace entry point stores dS beyond 512 blocks of 128 rows, 384 for T < 512."""
    assert A.backward_route(B, T, H, 128, True) == (A.STORED if stored else A.JOINT)
    assert A.backward_route(B, T, H, 128, False) == A.JOINT


def test_bad_shape():
    with pytest.raises(A.AttentionError):
        A.backward_route(1, 100, 1, 64, True)
