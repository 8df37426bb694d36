"""The mid-size GEMM path (gemm_mid_kernel: tiles through a ring of LDS stages, both weight
layouts, A activations, K of any multiple of 8) against the float64 oracle, at the edges of its
tiles and stages, split and whole, with every epilogue."""
import numpy as np
import pytest
import torch

from oracle import ops_ref as R
from tests.test_gemm_gpu import ACC, ACT, check, dev, h
from vkwr_amd import capi

pytestmark = pytest.mark.gpu

ACTS = {None: capi.ACT_NONE, "tanh": capi.ACT_TANH, "sigmoid": capi.ACT_SIGMOID, "relu2": capi.ACT_RELU_SQUARE}


def run(a, w, layout, gpu, act=None, epi=capi.EPI_NONE, v=None, vf=None, v0=None, ws=None, tile=None, split=None):
    """tile, split: the tile that the launch must take, and whether in K parts."""
    c = torch.full((a.shape[0], w.shape[0] if layout == "nk" else w.shape[1]), float("nan"), device=gpu).half()
    ops = [None if x is None else dev(x, gpu) for x in (v, vf, v0)]
    ta, tw = dev(a, gpu), dev(w, gpu)
    p = [capi.gemm_problem(ta, tw, c, b_layout=capi.GEMM_B_NK if layout == "nk" else capi.GEMM_B_KN,
                           a_act=ACTS[act], epilogue=epi, v=ops[0], v_first=ops[1], v0=ops[2])]
    need = capi.gemm_workspace_bytes(p)
    if tile:
        r = capi.gemm_route(p)
        assert (r.path, r.tile_m, r.tile_n, r.parts > 1) == ("mid", *tile, bool(split)), r
    if ws == "none":
        capi.gemm(p, torch.empty(0, dtype=torch.uint8, device=gpu))
    elif ws == "misaligned":
        capi.gemm(p, torch.empty(need + 64, dtype=torch.uint8, device=gpu)[4:])
    else:
        capi.gemm(p, torch.empty(need, dtype=torch.uint8, device=gpu))
    torch.cuda.synchronize()
    return c


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("M,K,N,tile,split", [
    (129, 8, 8, (64, 64), 0),           # the smallest K and N: one stage, almost all of it past the end
    (129, 72, 136, (64, 64), 0),        # one row, one k chunk, one column chunk into the next
    (255, 64, 128, (64, 64), 0),        # whole stage, whole tiles but for a row
    (333, 480, 1000, (64, 64), 0),      # a ragged last stage after whole ones
    (200, 2048, 2048, (64, 64), 0),     # a whole K, ring wrapped several times
    (700, 8192, 264, (64, 64), 1),      # K in parts, partial planes and the reduce
    (1000, 2048, 2048, (128, 64), 0),   # a ragged last row of tiles
    (520, 2056, 2056, (128, 64), 0),    # ragged everywhere
    (200, 8192, 2048, (128, 64), 1),
    (2304, 4096, 512, (128, 128), 1),
    (300, 2056, 8200, (128, 128), 0),   # ragged everywhere
    (1024, 256, 8192, (256, 128), 0),   # whole
    (129, 8200, 8200, (256, 128), 1),   # ragged everywhere, in parts
    (640, 72, 32776, (128, 256), 0),    # ragged
    (300, 8200, 6152, (128, 256), 1),   # ragged everywhere, in parts
])
def test_mid_vs_oracle(gpu, M, K, N, tile, split, layout):
    a = h(M, K)
    w = h(N, K, scale=0.05) if layout == "nk" else h(K, N, scale=0.05)
    y = run(a, w, layout, gpu, tile=tile, split=split)
    assert torch.equal(y, run(a, w, layout, gpu))  # deterministic
    ref, abs_sum = R.gemm(a, w, layout)
    check(y, ref, ACC * abs_sum, f"{layout} {M}x{K}x{N}")


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("act", ["tanh", "sigmoid", "relu2"])
@pytest.mark.parametrize("M,K,N,tile,split", [
    (130, 96, 2056, (64, 64), 0), (700, 520, 264, (64, 64), 0), (200, 4104, 136, (64, 64), 1),
    (200, 72, 8200, (128, 128), 0), (200, 2056, 2056, (128, 128), 1),
    (129, 72, 16392, (128, 256), 0), (129, 4104, 3080, (128, 256), 1),
])
def test_mid_activations(gpu, M, K, N, tile, split, layout, act):
    """A activations, applied to the staged tile (a ragged stage's excess stays zero); the
    activated operand is rounded to fp16, at the oracle's rounding or its neighbour."""
    a = h(M, K)
    w = h(N, K, scale=0.05) if layout == "nk" else h(K, N, scale=0.05)
    y = run(a, w, layout, gpu, act=act, tile=tile, split=split)
    ref, abs_sum = R.gemm(a, w, layout, a_act=act)
    check(y, ref, (ACC + ACT) * abs_sum, f"{act} {layout} {M}x{K}x{N}")


@pytest.mark.parametrize("M,K,N,tile,split", [
    (130, 96, 264, (64, 64), 0), (700, 8192, 264, (64, 64), 1),  # (in parts: the reduce's epilogue)
    (200, 1032, 4104, (128, 64), 0), (200, 72, 8200, (128, 128), 0), (129, 72, 16392, (256, 128), 0),
    (513, 72, 8200, (128, 256), 0),
])
def test_mid_epilogues(gpu, M, K, N, tile, split):
    a, w = h(M, K), h(N, K, scale=0.5 / K ** 0.5)
    v, vf, v0 = h(M, N), h(M, N), h(N)
    z = R._f(a) @ R._f(w).T
    _, abs_sum = R.gemm(a, w, "nk")
    acc = ACC * abs_sum
    # each epilogue's slope times the accumulation error, and for the sigmoid gate |v_first - v| / 4
    cases = [(capi.EPI_BIAS, z + R._f(v0), acc), (capi.EPI_TANH, np.tanh(z), acc), (capi.EPI_SIGMOID, R.sigmoid(z), acc),
             (capi.EPI_RELU_SQUARE, np.maximum(z, 0) ** 2, 2 * np.abs(z) * acc + acc * acc),
             (capi.EPI_VALUE_RESIDUAL, R._f(v) + (R._f(vf) - R._f(v)) * R.sigmoid(R._f(v0) + z),
              acc * np.abs(R._f(vf) - R._f(v)) + 1e-6)]
    for epi, ref, slack in cases:
        y = run(a, w, "nk", gpu, epi=epi, v=v, vf=vf, v0=v0, tile=tile, split=split)
        check(y, ref.astype(np.float16), slack + 2e-6, f"epilogue {epi} {M}x{K}x{N}")


@pytest.mark.parametrize("ws", ["none", "misaligned"])
def test_mid_workspace(gpu, ws):
    """A shape whose K is split where a workspace is given and which the other paths ran without one:
    it still runs without (unsplit), and with one that is not 16-byte aligned."""
    M, K, N = 700, 8192, 264
    a, w = h(M, K), h(N, K, scale=0.05)
    ref, abs_sum = R.gemm(a, w, "nk")
    check(run(a, w, "nk", gpu, ws=ws), ref, ACC * abs_sum, ws)


@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_mid_ragged_k_keeps_non_finite_weights_in_their_columns(gpu, layout):
    """Inf in the last k of one weight column and NaN in another: those columns only, and the Inf
    stays an Inf (what is staged past K is zeroed in both operands, not only in one)."""
    M, K, N = 200, 72, 136
    a, w = np.abs(h(M, K)) + np.float16(0.5), h(N, K, scale=0.05)
    w[5, K - 1], w[77, K - 1] = np.inf, np.nan
    y = run(a, w if layout == "nk" else np.ascontiguousarray(w.T), layout, gpu).float()
    assert torch.isposinf(y[:, 5]).all() and torch.isnan(y[:, 77]).all()
    rest = [c for c in range(N) if c not in (5, 77)]
    assert torch.isfinite(y[:, rest]).all()


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("M,C,ranks,tile", [
    (999, 2048, (96, 96, 256, 64), (128, 256)),   # three prompts of 333 tokens
    (700, 768, (64, 64, 128, 32), (128, 128)),
    (1000, 4096, (128, 128, 480, 96), (128, 256)),
    (300, 2560, (96, 96, 320, 64), (64, 64)),
])
def test_mid_low_rank_outputs(gpu, M, C, ranks, tile, layout):
    """A prompt's low-rank outputs as the time mix launches them: tanh, none and sigmoid on A, and a value
    residual, in one batch of unequal K."""
    acts, epis = ["tanh", None, "sigmoid", None], [0, 0, 0, capi.EPI_VALUE_RESIDUAL]
    a, w = [h(M, k) for k in ranks], [h(C, k, scale=0.1) for k in ranks]
    v, vf, v0 = h(M, C), h(M, C), h(C)
    keep = [dev(x, gpu) for x in (v, vf, v0)]
    ta, tw = [dev(x, gpu) for x in a], [dev(x if layout == "nk" else x.T, gpu) for x in w]
    c = [torch.full((M, C), float("nan"), device=gpu).half() for _ in ranks]
    probs = [capi.gemm_problem(x, y, z, b_layout=capi.GEMM_B_NK if layout == "nk" else capi.GEMM_B_KN, a_act=ACTS[f],
                               epilogue=e, v=keep[0], v_first=keep[1], v0=keep[2])
             for x, y, z, f, e in zip(ta, tw, c, acts, epis)]
    r = capi.gemm_route(probs)
    assert (r.path, r.tile_m, r.tile_n) == ("mid", *tile), r
    capi.gemm(probs, torch.empty(capi.gemm_workspace_bytes(probs), dtype=torch.uint8, device=gpu))
    torch.cuda.synchronize()
    for i, act in enumerate(acts[:3]):
        ref, abs_sum = R.gemm(a[i], w[i], "nk", a_act=act)
        check(c[i], ref, (ACC + (ACT if act else 0)) * abs_sum, f"problem {i}")
    ref, abs_sum = R.gemm(a[3], w[3], "nk", epi="vres", v=v, v_first=vf, v0=v0)
    # the gate's slope (1/4 of |v_first - v|) times the accumulation error, and the gate's own fp32 rounding
    check(c[3], ref, 0.25 * np.abs(vf.astype(np.float64) - v) * ACC * abs_sum + 2e-6, "value residual")


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("act_shape,shape,tile,split", [
    ((1300, 264, 264), (1300, 264, 2056), (128, 64), 0), ((1000, 72, 136), (1000, 2056, 264), (128, 64), 1),
    ((8, 72, 136), (1000, 72, 8200), (256, 128), 0), ((8, 72, 136), (129, 4104, 8200), (256, 128), 1),
])
def test_mid_activation_beside_a_plain_problem(gpu, act_shape, shape, tile, split, layout):
    """The tiles that a launch takes with an activation on part of it only."""
    probs, want, keep = [], [], []
    for (m, k, n), act in ((act_shape, "sigmoid"), (shape, None)):
        a, w = h(m, k), h(n, k, scale=0.05)
        c = torch.full((m, n), float("nan"), device=gpu).half()
        ta, tw = dev(a, gpu), dev(w if layout == "nk" else w.T, gpu)
        probs.append(capi.gemm_problem(ta, tw, c, b_layout=capi.GEMM_B_NK if layout == "nk" else capi.GEMM_B_KN,
                                       a_act=ACTS[act]))
        ref, abs_sum = R.gemm(a, w, "nk", a_act=act)
        want.append((c, ref, (ACC + (ACT if act else 0)) * abs_sum))
        keep += [ta, tw]
    r = capi.gemm_route(probs)
    assert (r.path, r.tile_m, r.tile_n, r.parts > 1) == ("mid", *tile, bool(split)), r
    capi.gemm(probs, torch.empty(capi.gemm_workspace_bytes(probs), dtype=torch.uint8, device=gpu))
    torch.cuda.synchronize()
    for c, ref, slack in want:
        check(c, ref, slack, f"{shape} {layout}")


def test_mid_batch_of_unequal_k_with_an_empty_problem(gpu):
    """Low-rank outputs: the batch is dealt out longest K first; an empty problem inside it."""
    M, C = 300, 520
    shapes = [(M, 96, C), (M, 264, C), (0, 64, C), (M, 64, C)]
    a = [h(m, k) for m, k, _ in shapes]
    w = [h(n, k, scale=0.05) for _, k, n in shapes]
    ta, tw = [dev(x, gpu) for x in a], [dev(x, gpu) for x in w]
    c = [torch.full((m, n), float("nan"), device=gpu).half() for m, _, n in shapes]
    acts = [capi.ACT_TANH, capi.ACT_SIGMOID, capi.ACT_NONE, capi.ACT_NONE]
    probs = [capi.gemm_problem(x, y, z, a_act=f) for x, y, z, f in zip(ta, tw, c, acts)]
    capi.gemm(probs, torch.empty(capi.gemm_workspace_bytes(probs), dtype=torch.uint8, device=gpu))
    torch.cuda.synchronize()
    for i, act in ((0, "tanh"), (1, "sigmoid"), (3, None)):
        ref, abs_sum = R.gemm(a[i], w[i], "nk", a_act=act)
        check(c[i], ref, (ACC + (ACT if act else 0)) * abs_sum, f"problem {i}")
