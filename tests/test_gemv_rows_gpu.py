"""The [N,K] product of one to four rows: one or two weight rows per wave, one or four chunks of a row
in flight, against the float64 oracle on each side of the lines between them."""
import pytest
import torch

from oracle import ops_ref as R
from tests.test_gemm_gpu import ACC, check, dev, h
from vkwr._ops.v1 import v1_linear_ops as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [
    (1, 8, 8),        # a single chunk
    (2, 512, 41),     # a chunk in every lane; rows left over in the last workgroup
    (1, 96, 4097),    # short K, two rows per wave, an odd number of rows
    (2, 504, 8200),
    (3, 256, 16390),
    (1, 520, 9),      # two chunks in the first lane
    (1, 2056, 4099),  # a second batch of one chunk
    (4, 8192, 1030),  # the activations fill the LDS buffer
    (2, 16384, 33),
    (3, 520, 16385),  # two rows per wave
    (4, 2048, 16384),
])
def test_against_oracle(gpu, M, K, N):
    a, w = h(M, K), h(N, K, scale=0.05)
    y = L.linear_f16_orig(dev(a, gpu), dev(w, gpu))
    ref, abs_sum = R.gemm(a, w, "nk")
    check(y, ref, ACC * abs_sum, f"{M}x{K}x{N}")


@pytest.mark.parametrize("M,K,N,n", [(1, 256, 8192, 4096), (4, 2048, 16384, 2048)])
def test_same_bits_for_both_forms(gpu, M, K, N, n):
    """Rows of a weight that takes two rows per wave, and the same rows by themselves (one)."""
    a, w = dev(h(M, K), gpu), dev(h(N, K, scale=0.05), gpu)
    assert torch.equal(L.linear_f16_orig(a, w)[..., :n], L.linear_f16_orig(a, w[:n].contiguous()))
