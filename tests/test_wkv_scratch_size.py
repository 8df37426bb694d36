"""Scratch of the segmented WKV prefill (host only: the planner reads no memory)."""
import pytest

from vkwr_amd import capi

_bytes = capi._LIB.vkwr_wkv7_fp32_prefill_workspace_bytes


@pytest.mark.parametrize("rows,H", [
    (200, 32),    # too short for segments at any batch
    (2304, 129),  # more than half as many chains as CUs in one sequence
    (2304, 64), (1500, 32), (700, 12), (1023, 3),
    (14000, 64),  # several blocks
])
def test_scratch_for_any_batch_of_so_many_rows(rows, H):
    """Enough for every B, T with B T <= rows, and none or little more than the largest of them takes."""
    most = max(_bytes(B, T, H) for B in range(1, 130) for T in range(1, rows // B + 1))
    got = capi.wkv_prefill_workspace_max(rows, H)
    assert most <= got <= 1.02 * most
