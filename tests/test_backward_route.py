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


def test_bad_shape():
    with pytest.raises(A.AttentionError):
        A.backward_route(1, 100, 1, 64, True)
