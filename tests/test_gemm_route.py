"""The row-major GEMM's choice between the mid-size and the large-M kernel where both take the launch
([N,K] weights, K in whole stages), on each side of its lines (host only)."""
import ctypes

import pytest

from vkwr_amd import capi

P = ctypes.c_void_p(0x100000)  # never dereferenced


@pytest.mark.parametrize("M,K,N,path,parts", [
    (512, 2048, 2048, "mid", 1), (512, 4096, 16384, "mid", 1), (1000, 4096, 16384, "large", 1),
    # the head at a whole tile of rows: both are bound by the weights, the large-M kernel has less to do
    (256, 768, 65536, "large", 1), (256, 2048, 65536, "large", 1), (255, 2048, 65536, "mid", 1),
    # 256-row tiles all in K parts: the large-M kernel's estimate has nothing on top
    (2100, 8192, 2048, "large", 3), (2304, 8192, 2048, "large", 3), (680, 16384, 4096, "large", 5),
    # ... but with 192-row tiles it does
    (2839, 8192, 2048, "mid", 1), (550, 16384, 4096, "mid", 3), (1024, 16384, 2048, "mid", 4),
])
def test_mid_or_large(M, K, N, path, parts):
    r = capi.gemm_route([capi.GemmProblem(P, P, P, M, N, K, capi.GEMM_B_NK, 0, 0, P, P, P)])
    assert (r.path, r.parts) == (path, parts), r
