"""Which dispatches a phase of the encoder joins in one launch (host decision, no GPU): a joint launch
reads and writes in no order between workgroups, so a buffer that reuses the memory of one the phase
has finished with must send the calls it concerns one after another."""
import pytest

import metalllm_amd as M
import metalllm_amd.sublayer as S

D_JOINED, DPROJW_LAST, TILES = 1, 2, 4
TYPE = {"l": 4, "Dsum": 4, "dQ": 4, "dX": 4, "dQw": 4, "ln_stdev": 4, "ln_dgamma": 4, "ln_dbeta": 4}


def plan(B, T, H, D, block=False):
    """Buffers at addresses of their own (nothing is read through them) and the shape."""
    p = M.AttentionParams.of(B, T, H, D)
    R, C = B * T, H * D
    at, b = 1 << 20, S.SublayerBuffers()
    for n in S.SublayerBuffers.FIELDS:
        if n == "hidden" and not block:
            break
        rows = C if n.endswith("w") or n.endswith("_w") else R
        setattr(b, n, at)
        at += -(-rows * C * TYPE.get(n, 2) // 256) * 256
    return b, p


SHAPES = [(3, 320, 5, 64), (1, 64, 1, 64), (1, 256, 6, 64)]  # tile kernels (the last a multiple of 128)
WIDE = (8, 2048, 12, 64)                                     # 128-wide kernels


@pytest.mark.parametrize("shape", SHAPES)
def test_separate_buffers_join(shape):
    assert S.route(1, *plan(*shape)) == D_JOINED | DPROJW_LAST | TILES
    assert S.route(0, *plan(*shape, block=True)) == 1
    assert S.route(0, *plan(*shape)) == 0


@pytest.mark.parametrize("shape", SHAPES + [WIDE])
@pytest.mark.parametrize("out", ["dAttn", "Dsum", "dQ", "dK", "dV", "dX"])
@pytest.mark.parametrize("into", ["attn_out", "dOut"])
def test_dprojw_first_where_its_operands_are_replaced(shape, out, into):
    """dProjw reads attn_out and dOut: not last when a buffer written before it, or beside it, holds
    any byte of them."""
    b, p = plan(*shape)
    R, C = p.B * p.M, p.N
    for at in (0, 2 * R * C - 16, -16):  # the first bytes, the last ones, the end of `out` in its first
        size = R * C * TYPE.get(out, 2) if out != "Dsum" else 4 * R * p.NH
        setattr(b, out, getattr(b, into) + (at if at >= 0 else 16 - size))
        assert not S.route(1, b, p) & DPROJW_LAST, at
    setattr(b, out, getattr(b, into) + 2 * R * C)  # right behind it
    if out not in ("dQ", "dX"):  # twice as long: these reach the next buffer, no operand of dProjw
        assert S.route(1, b, p) & DPROJW_LAST


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("out,into", [("Dsum", "dOut"), ("Dsum", "proj_w"), ("dAttn", "dOut")])
def test_d_separate(shape, out, into):
    b, p = plan(*shape)
    setattr(b, out, getattr(b, into))
    assert not S.route(1, b, p) & D_JOINED


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("out,into", [("dX", "dQ"), ("dX", "X"), ("dQw", "dQ"), ("dKw", "dK"), ("dVw", "X"), ("dKw", "q_w"),
                                      ("dProjw", "attn_out"), ("dProjw", "dK"), ("dQw", "dOut"), ("dKw", "dVw"), ("dX", "dQw")])
def test_gradient_products_separate(shape, out, into):
    b, p = plan(*shape)
    setattr(b, out, getattr(b, into))
    assert not S.route(1, b, p) & (TILES | DPROJW_LAST) or shape[1] % 128 == 0 and not S.route(1, b, p) & TILES


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("into", ["attn_out", "proj_w"])
def test_residual_separate(shape, into):
    b, p = plan(*shape, block=True)
    b.residual = getattr(b, into)
    assert S.route(0, b, p) == 0
    b.residual = b.hidden  # the same elements, read and written by one thread
    assert S.route(0, b, p) == 1
