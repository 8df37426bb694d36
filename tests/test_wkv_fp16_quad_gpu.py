"""The four-wave fp16 recurrence (T > 1, few chains): the oracle's bits around its 16-token staging
chunks, with w0 and the legacy arithmetic, with operands off 16-byte alignment (which take the
one-wave form), and with more chains than it takes."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.wkv_inputs import make_state, make_wkv_inputs

pytestmark = pytest.mark.gpu


def _at_offset(x, off):
    """A copy of x whose first element lies `off` elements past an aligned address."""
    buf = torch.zeros(x.numel() + 16, dtype=x.dtype, device=x.device)
    v = buf[off:off + x.numel()].view(x.shape)
    v.copy_(x)
    return v


@pytest.mark.parametrize("variant", ["seq", "w0", "legacy"])
@pytest.mark.parametrize("B,T,H,odd", [(1, 4, 1, None), (1, 3, 1, None), (2, 15, 3, None), (1, 16, 2, None), (3, 17, 2, None),
                                       (1, 33, 5, None), (2, 19, 2, "y"), (2, 19, 2, "v"), (2, 19, 2, "w"),
                                       (17, 18, 32, None)])
def test_bits(gpu, variant, B, T, H, odd):
    C = H * 64
    ins = make_wkv_inputs(B, T, H, seed=B + T, dist="realistic")
    S0 = make_state(B, H, seed=T, std=0.1, dtype=np.float16)
    el = np.random.default_rng(T).integers(0, 1 << 30, size=B).astype(np.int32)
    w0 = (np.random.default_rng(T).standard_normal(C) * 0.1).astype(np.float16) if variant == "w0" else None
    S_ref = S0.copy()
    y_ref = orc.wkv_fp16(B, T, C, H, S_ref, *ins, el, w0=w0, legacy=variant == "legacy")
    names = "rwkvab"
    d = [_at_offset(torch.from_numpy(x).to(gpu), 1 if n == odd else 0) for n, x in zip(names, ins)]
    y = _at_offset(torch.full((B, T, C), 7.0, dtype=torch.float16, device=gpu), 1 if odd == "y" else 0)
    state, elt = torch.from_numpy(S0).to(gpu), torch.from_numpy(el).to(gpu)
    if variant == "legacy":
        torch.ops.vkwr_rwkv7.forward_seq(B, T, C, H, state, *d, y, elt)
    elif variant == "w0":
        torch.ops.vkwr_v1_wkv.wkv_seq_w0_fp16(B, T, C, H, state, d[0], d[1], torch.from_numpy(w0).to(gpu), *d[2:],
                                              y, elt)
    else:
        torch.ops.vkwr_v1_wkv.wkv_seq_fp16(B, T, C, H, state, *d, y, elt)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint16), y_ref.view(np.uint16))
    assert np.array_equal(state.cpu().numpy().view(np.uint16), S_ref.view(np.uint16))
