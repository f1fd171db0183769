"""layernormBackward where a row is shared by one, two and four waves, with row counts that leave the
last step of a workgroup partly empty, against the oracle at the bars of test_gpu_glue.py; and the
phase encoder's forms (dX cast, ln1 backward and skip add in one kernel; computeD and the residual
add in the projections' launches) bit for bit against the public calls on the encoder's own tensors."""
import numpy as np
import pytest

import oracle as O
from tests import test_gpu_glue as glue_checks
from tests.attn_case import to_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(4099, 1032), (1000, 1536), (515, 2056), (33, 3080), (1, 1024), (17, 512),
                                       # workgroups whose ranges of steps differ by one (ln_bwd_deal)
                                       (3077, 4096), (12281, 64), (12288, 768),
                                       # short rows, of which one lane or two hold all
                                       (12500, 8), (1003, 16), (70001, 24)])
def test_layernorm_row_split(gpu, rows, cols):
    import metalllm_amd.glue as G
    glue_checks.test_layernorm_forward_backward(gpu, G, rows, cols, 1.0)


@pytest.mark.parametrize("B,T,H,C", [(1, 64, 1, 64), (3, 192, 6, 384), (2, 64, 12, 768), (1, 128, 20, 1280), (1, 64, 20, 2560),
                                     (8, 1024, 12, 768), (3, 320, 5, 320), (2, 192, 3, 384),
                                     # ln1's backward in ranges of 3 and 4 steps that end apart (ln_bwd_deal), its rows
                                     # by one wave and by two; the last with ranges that differ by one
                                     (48, 256, 12, 768), (32, 256, 24, 1536), (49, 256, 12, 768)])
def test_block_ends(gpu, B, T, H, C):
    """Also computeD and the residual add where the projections' tiles do them (D = 64; residual at
    every D), against the public calls on the encoder's own dAttn, attn_out and out."""
    import torch
    import metalllm_amd.glue as G
    import metalllm_amd.sublayer as S
    rng = np.random.default_rng(B * T + C)
    bf = lambda shape, sc=1.0, sh=0.0: to_gpu(O.f32_to_bf16((rng.standard_normal(shape) * sc + sh).astype(np.float32)), gpu)
    blk = S.Sublayer(None, *[bf((C, C), 0.02) for _ in range(4)], H=H, hidden=bf((B, T, C), 1.0, 0.3),
                     ln_gamma=bf((C,), 0.1, 1.0), ln_beta=bf((C,), 0.1))
    blk.dOut.copy_(bf((B, T, C)))
    blk.encode(0)
    blk.encode(1)
    d = torch.empty_like(blk.dOut)
    dg, db = torch.zeros(C, device=gpu), torch.zeros(C, device=gpu)
    G.castFloatToBfloat(blk.dX, d)
    G.layernormBackward(d, blk.ln_xnorm, blk.ln_gamma, blk.ln_stdev, dg, db)
    G.residualAdd(d, blk.dOut, d)
    import metalllm_amd as M
    Dv, res = torch.empty_like(blk.Dv), torch.empty_like(blk.residual)
    four = lambda t: t.view(B, T, H, C // H)
    M.computeD(four(blk.dO), four(blk.o), Dv)
    G.residualAdd(blk.hidden, blk.out, res)
    torch.cuda.synchronize()
    assert torch.equal(d, blk.dStream) and torch.equal(res, blk.residual)
    assert torch.equal(Dv.view(torch.int32), blk.Dv.view(torch.int32))
    for a, b in ((blk.ln_dgamma, dg), (blk.ln_dbeta, db)):  # fp32 column sums in atomic order
        assert (a - b).abs().max().item() <= 1e-5 * b.abs().max().item()


def test_residual_in_attn_out(gpu):
    """A forward pass whose residual reuses attn_out's memory: the same residual as with its own buffer
    (the projection's tiles read rows of attn_out that other tiles' residual would have replaced)."""
    import torch
    import metalllm_amd.sublayer as S
    B, T, H, C = 3, 320, 5, 320
    rng = np.random.default_rng(7)
    bf = lambda shape, sc=1.0, sh=0.0: to_gpu(O.f32_to_bf16((rng.standard_normal(shape) * sc + sh).astype(np.float32)), gpu)
    blk = S.Sublayer(None, *[bf((C, C), 0.02) for _ in range(4)], H=H, hidden=bf((B, T, C), 1.0, 0.3),
                     ln_gamma=bf((C,), 0.1, 1.0), ln_beta=bf((C,), 0.1))
    blk.encode(0)
    bufs = blk.buffers()
    shared = torch.empty_like(blk.residual)
    bufs.residual = bufs.attn_out = shared.data_ptr()
    S.encode_phase(0, bufs, blk.p)
    torch.cuda.synchronize()
    assert torch.equal(shared, blk.residual)
