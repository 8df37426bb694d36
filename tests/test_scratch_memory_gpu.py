"""Ops whose scratch makes them faster but that run without it, where torch's allocator has no memory left
for it (a limit of the allocator's own, set on the host)."""
import contextlib
import gc

import pytest
import torch

from tests.wkv_inputs import make_state, make_wkv_inputs
from vkwr_amd import capi

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def no_memory_left():
    """The allocator may reserve nothing more, and what it has cached is taken."""
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
    taken, size = [], 64 << 20
    try:
        while size >= 1 << 18:
            try:
                taken.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            except torch.cuda.OutOfMemoryError:
                size //= 2
        yield
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        taken.clear()


def test_prefill_runs_without_memory_for_its_segments(gpu):
    from vkwr._ops.v1 import v1_wkv_ops as ops

    B, T, H = 1, 1500, 32
    C = H * 64
    ins = [torch.from_numpy(x).to(gpu) for x in make_wkv_inputs(B, T, H, seed=4, dist="realistic")]
    state0 = torch.from_numpy(make_state(B, H, seed=4)).to(gpu)
    slots = torch.arange(B, dtype=torch.int32, device=gpu)
    need = capi._LIB.vkwr_wkv7_fp32_prefill_workspace_bytes(B, T, H)
    assert need > 2 * B * T * C
    plain, plain_state = torch.empty(B, T, C, dtype=torch.float16, device=gpu), state0.clone()
    capi.wkv_slots(B, T, C, H, plain_state, slots, *ins, plain)
    dense, pool, room, room2 = state0.clone(), state0.clone(), torch.empty_like(plain), torch.empty_like(plain)
    with no_memory_left():
        del room  # of y
        y = ops.wkv_forward_fp32(B, T, C, H, dense, *ins)
        del room2
        y2 = ops.wkv_forward_slots_fp32(B, T, C, H, pool, slots, *ins)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            torch.empty(need, dtype=torch.uint8, device=gpu)
    assert torch.equal(y, plain) and torch.equal(dense, plain_state)
    assert torch.equal(y2, plain) and torch.equal(pool, plain_state)


def test_gemm_runs_without_memory_for_its_parts(gpu):
    """[K,N] weights and more than 128 rows: K is split where there is memory for the parts."""
    from vkwr._ops.v1 import v1_linear_ops as L

    M, K, N = 2304, 4096, 512
    g = torch.Generator(device=gpu).manual_seed(1)
    a = torch.randn(M, K, device=gpu, generator=g).half()
    w = (torch.randn(K, N, device=gpu, generator=g) * 0.02).half()
    want, room = L.linear_f16(a, w), torch.empty(M, N, dtype=torch.float16, device=gpu)
    p = [capi.gemm_problem(a, w, room, b_layout=capi.GEMM_B_KN)]
    assert capi.gemm_workspace_bytes(p) > 2 * M * N * 2
    capi.gemm(p, torch.empty(0, dtype=torch.uint8, device=gpu))
    unsplit = room.clone()
    # a batch that its path always needed scratch for still says so
    big_a, big_w = torch.randn(512, 4096, device=gpu).half(), torch.randn(4096, 4096, device=gpu).half()
    room2 = torch.empty(512, 4096, dtype=torch.float16, device=gpu)
    del p
    with no_memory_left():
        del room
        y = L.linear_f16(a, w)
        del room2
        with pytest.raises(torch.cuda.OutOfMemoryError):
            L.linear_f16_orig(big_a, big_w)
    assert torch.equal(y, unsplit)
    assert (want.float() - unsplit.float()).abs().max().item() <= 2.0 ** -9 * want.abs().max().item()
