"""The decode GEMM's choice of tile by the workgroups it makes (32 x 32 to 128 x 64, eight and four
waves, whole K and K parts) against the float64 oracle, on each side of its lines."""
import numpy as np
import pytest
import torch

from oracle import ops_ref as R
from tests.test_frag_gemm_gpu import ACC, check, h, pack
from vkwr_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (32, 8192, 640),     # 256 tiles of 32 x 32
    (33, 8192, 640),     # 256 of 32 x 64, one row in the second
    (129, 2048, 1152),   # 160 of 32 x 64, a whole number of 16 x 8 steps
    (65, 8192, 640),     # 256 of 64 x 64
    (129, 8192, 640),    # 256 of 128 x 64
    (129, 16384, 640),   # more: 64 x 64 with four waves
    (256, 16392, 1152),  # more: 128 x 64
    (7, 16392, 640),     # one row tile: 32 x 64
    (200, 2056, 96),     # short K: 32 x 64 with four waves
    (129, 1024, 768),    # 32 x 32, 160 workgroups
    (161, 2048, 768),    # K <= 1024: 384 workgroups of 32 x 32
])
def test_whole_k(gpu, M, N, K):
    a, w = h(M, K), h(N, K, scale=0.05)
    pa, pw = pack(a, gpu, M, K), pack(w, gpu, N, K)
    c = torch.full((M, N), float("nan"), dtype=torch.float16, device=gpu)
    capi.frag_gemm([capi.frag_problem(pa, pw, c, M, N, K)])
    ref, abs_sum = R.gemm(a, w, "nk")
    check(c, ref, ACC * abs_sum, f"{M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K,splits", [
    (16, 256, 2048, 4),    # 32 x 32
    (32, 2048, 4096, 8),   # 32 x 64
    (64, 2048, 4096, 8),   # 64 x 64
    (160, 2048, 2048, 4),  # 128 x 64: planes of 192 rows under tiles of 256
    (160, 8192, 512, 1),   # one part
    (200, 8192, 1024, 2),  # more than one round
])
def test_parts(gpu, M, N, K, splits):
    """The sum of the parts; and nothing is written past the planes."""
    a, w = h(M, K), h(N, K, scale=0.05)
    pa, pw = pack(a, gpu, M, K), pack(w, gpu, N, K)
    floats = capi.frag_splitk_workspace_bytes(M, N, splits) // 4
    buf = torch.full((floats + 128 * capi.frag_pad(N),), 7.0, dtype=torch.float32, device=gpu)
    c = torch.full((M, N), float("nan"), dtype=torch.float16, device=gpu)
    capi.frag_gemm_splitk(capi.frag_problem(pa, pw, c, M, N, K), splits, buf[:floats])
    ref, abs_sum = R.gemm(a, w, "nk")
    check(c, ref, ACC * abs_sum, f"{M}x{N}x{K}/{splits}")
    assert (buf[floats:] == 7.0).all()


@pytest.mark.parametrize("M,C,ranks", [
    (8, 768, (64, 64, 128)),       # 32 x 32: all of it in one round
    (65, 1024, (64, 64, 128)),     # short K, more than one round: 32 x 64 with four waves, a step each
    (129, 2048, (96, 96, 256)),
    (256, 4096, (128, 128, 480)),  # K of four steps
])
def test_low_rank_outputs_batch(gpu, M, C, ranks):
    """The decode step's low-rank outputs in one launch (bias, none, none, value residual), K up to 512."""
    ks = [*ranks, 64]
    a, w = [h(M, k) for k in ks], [h(C, k, scale=0.1) for k in ks]
    v, vf, v0, w0 = h(M, C), h(M, C), h(C), h(C)
    tv, tvf, tv0, tw0 = (torch.from_numpy(x).to(gpu) for x in (v, vf, v0, w0))
    pa, pw = [pack(x, gpu, M, k) for x, k in zip(a, ks)], [pack(x, gpu, C, k) for x, k in zip(w, ks)]
    c = [torch.full((M, C), float("nan"), dtype=torch.float16, device=gpu) for _ in ks]
    fp = capi.frag_problem
    capi.frag_gemm([fp(pa[0], pw[0], c[0], M, C, ks[0], epilogue=capi.EPI_BIAS, v0=tw0),
                    fp(pa[1], pw[1], c[1], M, C, ks[1]), fp(pa[2], pw[2], c[2], M, C, ks[2]),
                    fp(pa[3], pw[3], c[3], M, C, ks[3], epilogue=capi.EPI_VALUE_RESIDUAL, v=tv, v_first=tvf, v0=tv0)])
    z, abs_sum = R._f(a[0]) @ R._f(w[0]).T, np.abs(R._f(a[0])) @ np.abs(R._f(w[0])).T
    check(c[0], (z + R._f(w0)).astype(np.float16), ACC * abs_sum, "bias")
    for i in (1, 2):
        ref, abs_sum = R.gemm(a[i], w[i], "nk")
        check(c[i], ref, ACC * abs_sum, f"problem {i}")
    ref, abs_sum = R.gemm(a[3], w[3], "nk", epi="vres", v=v, v_first=vf, v0=v0)
    # the gate's slope (1/4 of |v_first - v|) times the accumulation error, and the gate's own fp32 rounding
    check(c[3], ref, 0.25 * np.abs(R._f(vf) - R._f(v)) * ACC * abs_sum + 2e-6, "value residual")
