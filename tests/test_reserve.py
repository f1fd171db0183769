"""metalllmSublayerReserve covers every smaller shape (host arithmetic, no GPU): for all calls of at
most R rows and C features, whichever kernels they run, the scratch they need is no more than what is
reserved for (R, C)."""
import numpy as np

import metalllm_amd as M
import metalllm_amd.sublayer as S


def sizes(R, C):
    return S.scratch(M.AttentionParams(R, C, C, 1, 1))


def test_reserve_covers_smaller_shapes():
    rows = sorted({64 * i for i in range(1, 70)} | {128 * i for i in range(20, 140, 3)} | {100, 1000, 8200, 16400, 24576, 32768})
    feats = [8, 64, 128, 192, 200, 256, 320, 384, 448, 512, 576, 640, 768, 896, 1024, 1280]
    need = np.empty((len(rows), len(feats), 2))
    have = np.empty_like(need)
    for i, R in enumerate(rows):
        for j, C in enumerate(feats):
            need[i, j], have[i, j] = sizes(R, C)
    most = np.maximum.accumulate(np.maximum.accumulate(need, 0), 1)  # over smaller R and C
    bad = np.argwhere((most > have).any(-1))
    assert len(bad) == 0, [(rows[i], feats[j]) for i, j in bad[:5]]


def test_reserve_stays_small():
    """4 bytes per element of an activation, and at most 128 per element of a weight but for the row
    chunks of few features (a shape's own need is bounded the same way)."""
    for R, C in ((16384, 768), (32768, 384), (65536, 4096), (2048, 46336), (16384, 8192)):
        _, (split, partial) = sizes(R, C)
        assert 2 * split == 4 * R * C
        assert 4 * partial <= max(128 * C * C, 64 << 20)
