"""Slot installs (mlora_install_slot) where the kernel's two ways of walking a slot could differ: 128-bit pieces where
every row starts on a 16-byte boundary, else element by element."""

import pytest
import torch

from helpers import DTYPES


@pytest.mark.gpu
@pytest.mark.parametrize("scaling", [-2.0, float("inf"), float("nan"), 0.0])
@pytest.mark.parametrize("k", [64, 60])  # 60: element by element
@pytest.mark.parametrize("name", list(DTYPES))
def test_padding_beyond_the_rank_is_positive_zero_whatever_the_scaling(name, k, scaling):
    from nanovllm_voxcpm_amd import _hip

    print(f"install {name} K={k} scaling={scaling}", flush=True)
    dtype, slots, n, r, rank, slot = DTYPES[name], 3, 24, 16, 11, 1
    g = torch.Generator().manual_seed(3)
    a_src, b_src = torch.randn(r, k, generator=g).to(dtype), torch.randn(n, r, generator=g).to(dtype)
    a, b = torch.full((slots, r, k), 7.0, dtype=dtype, device="cuda"), torch.full((slots, n, r), 7.0, dtype=dtype, device="cuda")
    _hip.install_slot(a, b, slot, a_src.cuda(), b_src.cuda(), rank, scaling)
    a, b = a.cpu(), b.cpu()
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    assert not a[slot, rank:].contiguous().view(bits).any() and not b[slot, :, rank:].contiguous().view(bits).any()
    assert torch.equal(a[slot, :rank], a_src[:rank])
    want = b_src[:, :rank] * scaling
    assert torch.equal(b[slot, :, :rank].isnan(), want.isnan()) and torch.equal(b[slot, :, :rank].nan_to_num(), want.nan_to_num())
    others = [s for s in range(slots) if s != slot]
    assert (a[others] == 7).all() and (b[others] == 7).all()
