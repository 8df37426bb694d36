"""The decode GEMM's choice of tile by the workgroups it makes (32 x 32 to 128 x 64, eight and four
waves, whole K and K parts) against the float64 oracle, on each side of its lines."""
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
