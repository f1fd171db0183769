"""GPU parity: the HIP kernels through the C ABI against the CPU oracle on identical seeded inputs.

Bars: LSE within 1e-3; O within 1e-2 max-abs, where every element
beyond it is listed and must be an output rounding flip (|O| >= 2, whose bf16 spacing 1/64
exceeds the bar, and within one spacing of the oracle's unrounded value); dQ/dK/dV within 2e-2
max-abs relative to max |grad|; computeD bit-exact (the reference's lane-strided sums and the
oracle's butterfly model of simd_sum); causal-mask and index logic exact (row 0 of O equals row 0
of V bit for bit; with V one-hot every future weight is exactly zero). Both backward entry points
are checked: flashAttentionBackward (which adds into dQ, as the reference's atomics do) and
flashAttentionBackwardWorkspace (which writes dQ; from stored dS where test_gpu_backward_launch.py says); their dK/dV must also be
identical to each other, their dQ equal within 1e-5 of max |dQ| (fp32 summation order).
"""
import ctypes
import os

import numpy as np
import pytest

import oracle as O
from tests.attn_case import (bf16_ulp, f32, gpu_backward, gpu_compute_d, gpu_forward, make_inputs, out_error,
                             out_exceptions, rel_to_max, to_gpu, to_np)
from tests.lse_flips import diagnose_row, o_move_bound, rows_beyond

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


def check_case(gpu, B, T, H, D, s, seed, b_end=0, threads=0):
    """Forward, computeD and backward against the oracle; the oracle runs batches [0, b_end)."""
    print(f"case B={B} T={T} H={H} D={D} qk_scale={s} seed={seed} oracle-batches={b_end or B}", flush=True)
    q, k, v, g = make_inputs(B, T, H, D, seed, s)
    nb = b_end or B
    sl = lambda x: np.ascontiguousarray(x[:nb])
    r_out, r_lse, r_of = O.forward_f32(sl(q), sl(k), sl(v), O.opts(threads=threads))
    ref = {"out": r_out, "lse": r_lse}
    out, lse = gpu_forward(q, k, v, gpu)
    lse_err = float(np.abs(lse[:nb] - ref["lse"]).max())
    o_max, _, o_over = out_error(out[:nb], ref["out"])
    flips, unexplained = out_exceptions(out[:nb], r_of)
    print(f"  fwd: lse max err {lse_err:.3g}, O max err {o_max:.3g}, O > 1e-2: {o_over} "
          f"(output rounding flips {len(flips)}, unexplained {len(unexplained)})")
    assert np.isfinite(lse).all() and lse_err <= 1e-3
    assert not unexplained, unexplained[:10]
    # computeD on the GPU's own O; the oracle on the same O must agree bit for bit
    Dfull = gpu_compute_d(g, out, gpu)
    Dr = O.compute_d(sl(g), sl(out))
    assert np.array_equal(Dfull[:nb], Dr), f"computeD differs: {np.abs(Dfull[:nb] - Dr).max()}"
    # backward alone: both sides get the GPU's lse and D
    rQ, rK, rV = O.backward(sl(g), Dr, np.ascontiguousarray(lse[:nb]), sl(q), sl(k), sl(v), O.opts(threads=threads))
    res = []
    for ws in (False, True):
        dQ, dK, dV = gpu_backward(g, Dfull, lse, q, k, v, gpu, workspace=ws)
        errs = {n: rel_to_max(x[:nb], r) for n, x, r in (("dQ", dQ, rQ), ("dK", dK, rK), ("dV", dV, rV))}
        print(f"  bwd{' (workspace)' if ws else ''} rel-to-max:", {n: f"{e:.3g}" for n, e in errs.items()}, flush=True)
        for n, e in errs.items():
            assert e <= 2e-2, n
        res.append((dQ, dK, dV))
    (q0, k0, v0), (q1, k1, v1) = res
    assert np.array_equal(k0, k1) and np.array_equal(v0, v1)
    assert np.abs(q0 - q1).max() <= 1e-5 * np.abs(q0).max()
    if D == 64:  # the workspace entry point stores no dS there: the same kernels, dQ written
        assert np.array_equal(q0, q1)
    return out, lse


CASES = [
    # (B, T, H, D, qk_scale, seed)
    (16, 256, 6, 64, 1.0, 11),    # config 0: the reference default shape
    (2, 512, 2, 128, 1.0, 12),    # D=128
    (1, 1024, 12, 64, 1.5, 13),   # config 2 slice: peaky rows
    (1, 192, 3, 128, 1.5, 14),    # T not a multiple of 128/256, odd head count
    (1, 64, 1, 64, 1.0, 15),      # a single tile
    (3, 320, 1, 64, 1.0, 16),     # 5 tiles, B*H not a multiple of 8
    # few pairs: both backward entry points run the joint launch (the stored-dS rings and the fused
    # kernel, which take many, are in test_gpu_backward_launch.py)
    (4, 448, 2, 128, 1.0, 17),    # 8 pairs: XCD-affine, 7 tiles
    (2, 576, 4, 128, 1.0, 18),    # 8 pairs: XCD-affine, 9 tiles
    (2, 128, 3, 64, 1.5, 19),     # two tiles, peaky
    (1, 192, 5, 64, 1.0, 20),     # three tiles
]


@pytest.mark.parametrize("B,T,H,D,s,seed", CASES)
def test_forward_backward_parity(gpu, B, T, H, D, s, seed):
    check_case(gpu, B, T, H, D, s, seed)


def _sweep_cases(n=14, seed=2024):
    """Seeded shape sweep: T every multiple of 64 up to 640 (few pairs: the persistent forward and the
    joint backward), odd and even head and batch counts (pair counts
    that are and are not multiples of 8), both head sizes and both Q/K scales."""
    rng = np.random.default_rng(seed)
    cases = []
    for i in range(n):
        D = (64, 128)[i % 2]
        T = 64 * int(rng.integers(1, 11))
        B = int(rng.integers(1, 4))
        H = int(rng.integers(1, 9 if T <= 256 else 5))
        cases.append((B, T, H, D, (1.0, 1.5)[int(rng.integers(0, 2))], 100 + i))
    return cases


@pytest.mark.parametrize("B,T,H,D,s,seed", _sweep_cases())
def test_shape_sweep(gpu, B, T, H, D, s, seed):
    check_case(gpu, B, T, H, D, s, seed)


def test_config1_slice_equals_config0(gpu):
    """Config 1 (B=128) on the GPU; its first 16 batches are config 0's inputs bit for bit, and are
    checked against the oracle."""
    out, lse = check_case(gpu, 128, 256, 6, 64, 1.0, 21, b_end=16)
    q0, k0, v0, _ = make_inputs(16, 256, 6, 64, 21)
    out0, lse0 = gpu_forward(q0, k0, v0, gpu)
    assert np.array_equal(out[:16], out0) and np.array_equal(lse[:16], lse0)


@pytest.mark.parametrize("B,H,D,Tp", [(128, 6, 64, 256), (100, 3, 64, 192), (97, 3, 64, 64), (64, 3, 128, 256),
                                      (8, 12, 64, 2048), (16, 4, 128, 2048)])
def test_persistent_forward_equals_per_item_forward(gpu, B, H, D, Tp):
    """The forward runs persistent (each workgroup takes several (pair, query block) items, the next
    item's Q rows and first K tiles loaded during the current item's last step) when there are at
    most two items per resident workgroup (768 at D = 64, 512 at D = 128 on MI355X), otherwise one
    workgroup per item. Causal rows 0..Tp-1 of a T = 2112 sequence depend only on keys 0..Tp-1
    and visit the same key tiles in the same order, so the T = 2112 forward (one workgroup per
    item: its 17 query blocks per pair exceed two per slot in every case here) and the T = Tp
    forward of the prefix (persistent) must agree bit for bit on those rows. At B = 128, H = 6,
    T = 256 each workgroup takes two items; 300 and 291 pairs are not multiples of 8 (one group of
    workgroups), at Tp = 64 an item has one key tile, and the T = 2048 cases are config 4's
    attention shape and its D = 128 counterpart (exactly two items per slot)."""
    print(f"case B={B} H={H} D={D} Tp={Tp}", flush=True)
    q, k, v, _ = make_inputs(B, 2112, H, D, 61)
    out_l, lse_l = gpu_forward(q, k, v, gpu)
    pre = lambda x: np.ascontiguousarray(x[:, :Tp])
    out_s, lse_s = gpu_forward(pre(q), pre(k), pre(v), gpu)
    assert np.array_equal(out_s, out_l[:, :Tp])
    assert np.array_equal(lse_s, lse_l[:, :, :Tp])


ORACLE_FIXTURES = sorted(n[len("oracle_"):-len(".npz")] for n in os.listdir(os.path.join(HERE, "golden"))
                         if n.startswith("oracle_") and n.endswith(".npz"))


@pytest.mark.parametrize("name", ORACLE_FIXTURES)
def test_committed_fixtures(gpu, name):
    """The GPU path on the committed inputs of tests/golden/oracle_<name>.npz against the committed
    oracle outputs (B=1, H=2, T=128, D 64 or 128, normal or peaky): LSE within 1e-3, O within
    max(1e-2, one bf16 spacing), computeD on the stored dO and O bit for bit, and both backward
    entry points on the stored D and LSE within 2e-2 of max |grad|."""
    print(f"fixture {name}", flush=True)
    d = np.load(os.path.join(HERE, "golden", f"oracle_{name}.npz"))
    q, k, v, g = d["q"], d["k"], d["v"], d["dO"]
    out, lse = gpu_forward(q, k, v, gpu)
    assert float(np.abs(lse - d["lse"]).max()) <= 1e-3
    _, beyond, _ = out_error(out, d["out"])
    assert beyond == 0
    assert np.array_equal(gpu_compute_d(g, d["out"], gpu), d["D"])
    for ws in (False, True):
        dQ, dK, dV = gpu_backward(g, d["D"], d["lse"], q, k, v, gpu, workspace=ws)
        for n, x in (("dQ", dQ), ("dK", dK), ("dV", dV)):
            e = rel_to_max(x, d[n])
            print(f"  {n}{' (workspace)' if ws else ''}: rel-to-max {e:.3g}")
            assert e <= 2e-2, n


def test_config2_peaky_slice(gpu):
    """Config 2 (B=32, H=12, T=1024, D=64, Q/K x1.5): two batches checked against the oracle."""
    check_case(gpu, 32, 1024, 12, 64, 1.5, 22, b_end=2)


def test_config3_slice(gpu):
    """Config 3 (B=16, H=16, T=4096, D=128) at B=1: all 16 heads of batch 0 against the oracle."""
    check_case(gpu, 1, 4096, 16, 128, 1.0, 23)


@pytest.mark.parametrize("D", [64, 128])
def test_long_sequence_extends_shorter(gpu, D):
    """T = 8192 (twice config 3's length) against T = 4096 on the same leading rows, both entry
    points of the backward. Causal rows 0..4095 of the forward depend only on keys 0..4095 and
    visit the same tiles in the same order, so O and LSE agree bit for bit; with dO zero on rows
    4096.., those rows have D = 0, dP = 0 and dS = 0, so they add exact zeros to every gradient:
    dQ of rows 0..4095 and dK, dV of keys 0..4095 agree bit for bit with the T = 4096 backward,
    and the rest is zero. The T = 4096 path is checked against the oracle at config 3."""
    B, H, T, Ts = 1, 2, 8192, 4096
    print(f"case T={T} vs {Ts} H={H} D={D}", flush=True)
    q, k, v, g = make_inputs(B, T, H, D, 95)
    g[:, Ts:] = 0
    pre = lambda x: np.ascontiguousarray(x[:, :Ts])
    out_l, lse_l = gpu_forward(q, k, v, gpu)
    out_s, lse_s = gpu_forward(pre(q), pre(k), pre(v), gpu)
    assert np.array_equal(out_s, out_l[:, :Ts]) and np.array_equal(lse_s, lse_l[:, :, :Ts])
    D_l = gpu_compute_d(g, out_l, gpu)
    D_s = gpu_compute_d(pre(g), out_s, gpu)
    assert np.array_equal(D_s, D_l[:, :, :Ts]) and not D_l[:, :, Ts:].any()
    for ws in (False, True):
        dQ_l, dK_l, dV_l = gpu_backward(g, D_l, lse_l, q, k, v, gpu, workspace=ws)
        dQ_s, dK_s, dV_s = gpu_backward(pre(g), D_s, lse_s, pre(q), pre(k), pre(v), gpu, workspace=ws)
        for n, long_, short in (("dQ", dQ_l, dQ_s), ("dK", dK_l, dK_s), ("dV", dV_l, dV_s)):
            assert np.array_equal(long_[:, :Ts], short), n
            assert not f32(long_[:, Ts:]).any(), n


def test_config3_full_size_properties(gpu):
    """Config 3 at full size: row 0 of every head equals V row 0 bit for bit (causal index logic),
    LSE finite, forward and backward deterministic across runs, sum over keys of dV equal to the
    sum over queries of dO (rows of P sum to 1); the workspace backward gives identical dK/dV and
    dQ within fp32 summation order."""
    import torch
    import metalllm_amd as M
    B, T, H, D = 16, 4096, 16, 128
    dev = gpu
    g_ = torch.Generator(device=dev)
    g_.manual_seed(7)
    mk = lambda: torch.randn((B, T, H, D), generator=g_, device=dev).to(torch.bfloat16)
    q, k, v, dO = mk(), mk(), mk(), mk()
    out1, lse1 = M.attention_forward(q, k, v)
    out2, lse2 = M.attention_forward(q, k, v)
    assert torch.equal(out1, out2) and torch.equal(lse1, lse2)
    assert torch.equal(out1[:, 0], v[:, 0])
    assert torch.isfinite(lse1).all()
    dQ1, dK1, dV1, Dv = M.attention_backward(dO, q, k, v, out1, lse1)
    dQ2, dK2, dV2, _ = M.attention_backward(dO, q, k, v, out1, lse1)
    assert torch.equal(dK1, dK2) and torch.equal(dV1, dV2) and torch.equal(dQ1, dQ2)
    ws = torch.empty((M.workspace_bytes(B, T, H, D),), dtype=torch.uint8, device=dev)
    dQ3, dK3, dV3 = torch.empty_like(dQ1), torch.empty_like(dK1), torch.empty_like(dV1)
    M.flashAttentionBackwardWorkspace(dO, Dv, lse1, q, k, v, dQ3, dK3, dV3, ws)
    assert torch.equal(dK1, dK3) and torch.equal(dV1, dV3)
    assert (dQ1 - dQ3).abs().max().item() <= 1e-5 * dQ1.abs().max().item()
    del ws
    sdv = dV1.float().sum(1)
    sdo = dO.float().sum(1)
    assert ((sdv - sdo).abs().max() / sdo.abs().max()).item() < 3e-2


def test_mfma_model_on_random_tiles(gpu):
    """The oracle's matrix-core model reproduces v_mfma_f32_32x32x16_bf16 bit for bit on random
    tiles: N(0,1) operands, scaled operands, mixed magnitudes, and nonzero accumulators."""
    import torch
    lib = ctypes.CDLL(os.path.join(HERE, "golden", "libmfma_probe.so"))
    lib.mfma_probe_run.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_int, ctypes.c_void_p]
    rng = np.random.default_rng(11)
    n = 48
    scale = np.exp(rng.uniform(-6, 6, size=(n, 64, 8)))
    a = O.f32_to_bf16((rng.standard_normal((n, 64, 8)) * scale).astype(np.float32))
    b = O.f32_to_bf16(rng.standard_normal((n, 64, 8)).astype(np.float32))
    c = (rng.standard_normal((n, 64, 16)) * rng.choice([0, 1e-3, 1, 30], size=(n, 1, 1))).astype(np.float32)
    ta, tb, tc = to_gpu(a, gpu), to_gpu(b, gpu), to_gpu(c, gpu)
    assert lib.mfma_probe_run(ta.data_ptr(), tb.data_ptr(), tc.data_ptr(), n, torch.cuda.current_stream().cuda_stream) == 0
    res = to_np(tc)
    orc = O.default()
    A = f32(a)
    Bm = f32(b)
    bad = 0
    for t in range(n):
        Am = np.zeros((32, 16), np.float32)
        Bt = np.zeros((32, 16), np.float32)  # [n][k]
        for l in range(64):
            Am[l % 32, 8 * (l // 32):8 * (l // 32) + 8] = A[t, l]
            Bt[l % 32, 8 * (l // 32):8 * (l // 32) + 8] = Bm[t, l]
        for l in range(64):
            for r in range(16):
                m = 8 * (r // 4) + 4 * (l // 32) + r % 4
                nn = l % 32
                ref = orc.dot(float(c[t, l, r]), Am[m], Bt[nn], O.GEMM_MFMA, O.PASS_SEQ8)
                bad += np.float32(ref) != res[t, l, r]
    assert bad == 0, f"{bad} of {n * 1024} results differ from the model"


def test_backward_dq_contract(gpu):
    """ABI contract. flashAttentionBackward adds the gradient into dQ (the reference's fp32 atomics
    into a caller-zeroed buffer, attention.metal:292-296, model.h:549): with dQ prefilled, the
    result is prefill + gradient, each element one fp32 add of the zero-start result. It writes dK
    and dV in full (stale contents ignored). flashAttentionBackwardWorkspace writes all three in
    full, whatever the stale contents of its outputs or of the workspace. All
    shapes here run the joint launch (the fused kernel's additions are in test_gpu_backward_launch.py).
    At D = 64 the workspace entry point stores no dS, so its dQ equals the zero-start gradient bit for
    bit."""
    import torch
    import metalllm_amd as M
    for T, D in ((256, 64), (192, 64), (512, 64), (256, 128), (512, 128)):
        print(f"case T={T} D={D}", flush=True)
        q, k, v, g = make_inputs(1, T, 2, D, 31)
        tq, tk, tv, tg = (to_gpu(x, gpu) for x in (q, k, v, g))
        out, lse = M.attention_forward(tq, tk, tv)
        Dv = torch.empty((1, 2, T), dtype=torch.float32, device=gpu)
        M.computeD(tg, out, Dv)
        dQ0 = torch.zeros((1, T, 2, D), dtype=torch.float32, device=gpu)
        dK0, dV0 = torch.full_like(tq, float("nan")), torch.full_like(tq, float("nan"))
        M.flashAttentionBackward(tg, Dv, lse, tq, tk, tv, dQ0, dK0, dV0)
        assert torch.isfinite(dQ0).all() and torch.isfinite(dK0.float()).all() and torch.isfinite(dV0.float()).all()
        gen = torch.Generator(device=gpu)
        gen.manual_seed(T)
        prefill = torch.randn((1, T, 2, D), generator=gen, device=gpu) * 3.0
        dQ = prefill.clone()
        dK, dV = torch.full_like(tq, 7.0), torch.full_like(tq, -7.0)
        M.flashAttentionBackward(tg, Dv, lse, tq, tk, tv, dQ, dK, dV)
        assert torch.equal(dQ, prefill + dQ0)
        assert torch.equal(dK, dK0) and torch.equal(dV, dV0)
        ws = torch.full((M.workspace_bytes(1, T, 2, D),), 0x7F, dtype=torch.uint8, device=gpu)
        for fill in (7.0, float("nan")):
            wQ = torch.full_like(dQ0, fill)
            wK, wV = torch.full_like(tq, fill), torch.full_like(tq, -fill)
            M.flashAttentionBackwardWorkspace(tg, Dv, lse, tq, tk, tv, wQ, wK, wV, ws)
            assert torch.isfinite(wQ).all()
            assert (wQ - dQ0).abs().max().item() <= 1e-5 * dQ0.abs().max().item()
            if D == 64:
                assert torch.equal(wQ, dQ0)
            assert torch.equal(wK, dK0) and torch.equal(wV, dV0)


@pytest.mark.parametrize("B,T,H,D", [(1, 64, 1, 64), (2, 128, 3, 128), (1, 64, 2, 128), (2, 192, 4, 128),
                                     (4, 256, 2, 64)])
def test_causal_mask_with_one_hot_v(gpu, B, T, H, D):
    """The causal mask pinned on the GPU (attention.metal:117-120): with V[t] = e_(t mod D), O[i]
    carries the softmax weight of key j in column j mod D, so for rows i < D every column d > i
    (keys that exist only in the future) must be exactly 0, every column d <= i positive, and each
    row must sum to 1 within bf16 rounding. T = 64 and 192 leave the last 128-row block of the
    forward half empty; T = 256 at D = 64 checks rows 0-63 over two key tiles per block."""
    print(f"case B={B} T={T} H={H} D={D}", flush=True)
    q, k, _, _ = make_inputs(B, T, H, D, 51)
    v = np.zeros((B, T, H, D), np.uint16)
    t = np.arange(T)
    v[:, t, :, t % D] = 0x3F80  # bf16 1.0
    out, lse = gpu_forward(q, k, v, gpu)
    A = f32(out)  # [B, T, H, D]
    n = min(T, D)
    for b in range(B):
        for h in range(H):
            P = A[b, :n, h, :n]
            assert (P[np.triu_indices(n, 1)] == 0).all()
            assert (P[np.tril_indices(n)] > 0).all()
    assert np.abs(A.sum(-1) - 1).max() < 1e-2
    r_out, r_lse = O.forward(q, k, v)
    assert np.abs(lse - r_lse).max() <= 1e-3
    assert np.abs(A - f32(r_out)).max() <= 1e-2


@pytest.mark.parametrize("D,s,seed", [(64, 3.0, 71), (128, 3.0, 72), (64, 5.0, 73)])
def test_sharp_attention(gpu, D, s, seed):
    """Q and K scaled by 3 and 5 (score standard deviations of about 9 and 25 against 1 for
    unscaled inputs): the running max moves by far more than the rescale threshold within a row,
    so the O rescale runs with factors far below 1, and most rows put nearly all their weight on
    one key. Forward, computeD and both backward entry points against the oracle at the usual
    bars."""
    check_case(gpu, 1, 512, 2, D, s, seed)


@pytest.mark.parametrize("T,D", [(320, 64), (192, 128)])
def test_uniform_scores_closed_form(gpu, T, D):
    """Q = 0 makes every score 0, so row i attends uniformly to keys 0..i (attention.metal:111-158
    with S = 0): LSE_i = log(i + 1) (the running max is 0 and the row sum counts exact ones) and
    O_i = mean of V_0..V_i, rounded once to bf16 after an fp32 sum."""
    B, H = 1, 2
    print(f"case T={T} D={D}", flush=True)
    _, k, v, _ = make_inputs(B, T, H, D, 81)
    q = np.zeros_like(k)
    out, lse = gpu_forward(q, k, v, gpu)
    ref_lse = np.log(np.arange(1, T + 1, dtype=np.float64))
    assert np.abs(lse.astype(np.float64) - ref_lse[None, None, :]).max() <= 2e-6
    V = f32(v).astype(np.float64)
    mean = np.cumsum(V, axis=1) / np.arange(1, T + 1, dtype=np.float64)[None, :, None, None]
    err = np.abs(f32(out).astype(np.float64) - mean)
    assert (err <= bf16_ulp(mean.astype(np.float32)).astype(np.float64) + 1e-7).all(), float(err.max())


def check_against_plain_order(gpu, B, T, H, D, s, seed, nb, max_rows):
    """GPU forward on seeded inputs; batches [0, nb) against the oracle with the plain sequential
    fp32 order of the reference's matmul2d semantics (GEMM_SEQ), not the matrix-core order the GPU
    executes. Every LSE row beyond 1e-3 must be a diagnosed bf16 rounding flip of a score (the
    exact product within fp32 summation error of a bf16 midpoint; the LSE difference equal to
    what that one-ulp score move produces, at most one step times the flipped key's weight).
    Every O element beyond 1e-2 must be an output rounding flip or lie in such a row, and there
    within the diagnosed move: |O_gpu - O_ref| <= sum over the row's flipped keys j of
    w_j (e^step - 1) |V_j - O_ref| / (1 - sum w_j (1 - e^-step)) plus one bf16 spacing of O_ref
    (the GPU's own output rounding), with O_ref the oracle's unrounded O."""
    print(f"case B={B} T={T} H={H} D={D} qk_scale={s} seed={seed} oracle-batches={nb} (GEMM_SEQ)", flush=True)
    q, k, v, _ = make_inputs(B, T, H, D, seed, s)
    sl = lambda x: np.ascontiguousarray(x[:nb])
    qs, ks, vs = sl(q), sl(k), sl(v)
    r_out, r_lse, r_of = O.forward_f32(qs, ks, vs, O.opts(gemm_model=O.GEMM_SEQ))
    out, lse = gpu_forward(q, k, v, gpu)
    lse = np.ascontiguousarray(lse[:nb])
    rows = rows_beyond(r_lse, lse)
    diag = {}
    for r in rows:
        d = diagnose_row(qs, ks, r_lse, lse, *r, O.GEMM_SEQ, O.GEMM_MFMA)
        print("  diagnosed LSE flip:", {k_: d[k_] for k_ in ("row", "flips", "observed", "explained")}, flush=True)
        assert d["flips"] and abs(d["observed"]) <= d["max_score_step"] * d["flip_weight"] + 5e-5
        diag[r] = d
    print(f"  LSE max err {np.abs(r_lse - lse).max():.3g}; rows beyond 1e-3: {len(rows)}, all diagnosed flips")
    assert len(rows) <= max_rows
    flips, unexplained = out_exceptions(out[:nb], r_of)
    shape = out[:nb].shape  # [B, T, H, D]
    og = f32(out[:nb])
    rof = np.asarray(r_of, np.float32).reshape(shape)
    rest, bounded = [], 0
    for i in unexplained:
        b_, t_, h_, d_ = (int(x) for x in np.unravel_index(i, shape))
        info = diag.get((b_, h_, t_))
        if info is None:
            rest.append(i)
            continue
        move = o_move_bound(info, f32(vs[b_, info["flips"], h_, :]), rof[b_, t_, h_, :])[d_]
        err = abs(float(og[b_, t_, h_, d_]) - float(rof[b_, t_, h_, d_]))
        lim = move + float(bf16_ulp(rof[b_, t_, h_, d_]))
        assert err <= lim, ((b_, t_, h_, d_), err, move, lim)
        bounded += 1
    print(f"  O > 1e-2: output rounding flips {len(flips)}, in LSE-flip rows within the diagnosed move {bounded}, "
          f"other {len(rest)}")
    assert not rest


def test_config2_against_plain_fp32_order(gpu):
    """Config 2 slice (seed 22, batches 0-1, all 12 heads, Q/K x1.5) against the plain fp32 order."""
    check_against_plain_order(gpu, 32, 1024, 12, 64, 1.5, 22, 2, 3)


def test_config3_against_plain_fp32_order(gpu):
    """Config 3 slice (seed 23, batch 0, all 16 heads, T = 4096, D = 128) against the plain fp32
    order; the inputs are config 3's batch 0 (the generator is keyed by index)."""
    check_against_plain_order(gpu, 1, 4096, 16, 128, 1.0, 23, 1, 3)


def test_backward_parts_equal_flash_attention_backward(gpu):
    """The bench hook: part 0 (dK/dV kernel) then part 1 (dQ kernel) is flashAttentionBackward, and
    part 2 then part 3 is flashAttentionBackwardWorkspace, bit for bit (here both the joint launch; parts
    2 and 3 with the dS store are in test_gpu_backward_launch.py)."""
    import torch
    import metalllm_amd as M
    q, k, v, g = make_inputs(2, 512, 3, 128, 41)
    tq, tk, tv, tg = (to_gpu(x, gpu) for x in (q, k, v, g))
    out, lse = M.attention_forward(tq, tk, tv)
    Dv = torch.empty((2, 3, 512), dtype=torch.float32, device=gpu)
    M.computeD(tg, out, Dv)
    ws = torch.empty((M.workspace_bytes(2, 512, 3, 128),), dtype=torch.uint8, device=gpu)
    for first in (0, 2):
        res = []
        for split in (False, True):
            dQ = torch.zeros((2, 512, 3, 128), dtype=torch.float32, device=gpu)  # part 1 adds into dQ
            dK = torch.empty_like(tq)
            dV = torch.empty_like(tq)
            if split:
                M.backward_part(first, tg, Dv, lse, tq, tk, tv, dQ, dK, dV, workspace=ws)
                M.backward_part(first + 1, tg, Dv, lse, tq, tk, tv, dQ, dK, dV, workspace=ws)
            elif first == 0:
                M.flashAttentionBackward(tg, Dv, lse, tq, tk, tv, dQ, dK, dV)
            else:
                M.flashAttentionBackwardWorkspace(tg, Dv, lse, tq, tk, tv, dQ, dK, dV, ws)
            res.append((dQ, dK, dV))
        for a, b in zip(*res):
            assert torch.equal(a, b)


def test_batch_split_is_bit_identical(gpu):
    """Every (batch, head) pair is computed by its own workgroups, so the outputs of one batch must
    not depend on the grid around it. At B = 25, H = 8, T = 1024, D = 64 (200 pairs, 25 per XCD
    group) the forward runs one workgroup per item and the backward kernels run their grids in the
    chunked dispatch order with a short last chunk (forward chunks of 16 pairs: 16 + 9; dK/dV
    chunks of 8: 8 + 8 + 8 + 1); a single batch (8 pairs, one per XCD group) runs the persistent
    forward and one-pair chunks. Batches 0, 12 and 24 run alone must give the same O, LSE, D and
    gradients bit for bit, on both backward entry points."""
    B, T, H, D = 25, 1024, 8, 64
    print(f"case B={B} T={T} H={H} D={D} seed=71 against single batches 0, 12, 24", flush=True)
    q, k, v, g = make_inputs(B, T, H, D, 71)
    out, lse = gpu_forward(q, k, v, gpu)
    Dv = gpu_compute_d(g, out, gpu)
    full = [gpu_backward(g, Dv, lse, q, k, v, gpu, workspace=w) for w in (False, True)]
    for b in (0, 12, 24):
        one = lambda x: np.ascontiguousarray(x[b:b + 1])
        out1, lse1 = gpu_forward(one(q), one(k), one(v), gpu)
        assert np.array_equal(out1, out[b:b + 1]) and np.array_equal(lse1, lse[b:b + 1])
        D1 = gpu_compute_d(one(g), out1, gpu)
        assert np.array_equal(D1, Dv[b:b + 1])
        for w, grads in zip((False, True), full):
            got = gpu_backward(one(g), D1, lse1, one(q), one(k), one(v), gpu, workspace=w)
            for x, y in zip(got, grads):
                assert np.array_equal(x, y[b:b + 1])
