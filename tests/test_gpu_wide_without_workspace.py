"""One launch over 64-token tiles needs no workspace: by name and through AUTO's choice of it, called without one (the host divided by the number
of K parts that fit a workspace, which is none)."""

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["wide", "auto"])
def test_call_without_workspace(form):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    g = torch.Generator().manual_seed(3)
    tokens, rank, k, n = 3000, 64, 1024, 512
    indices = torch.zeros(tokens, dtype=torch.int32, device="cuda")
    a, b = (torch.randn(1, rank, k, generator=g) * 0.02).bfloat16().cuda(), (torch.randn(1, n, rank, generator=g) * 0.1).bfloat16().cuda()
    x, y = torch.randn(tokens, k, generator=g).bfloat16().cuda(), torch.randn(tokens, n, generator=g).bfloat16().cuda()
    out = y.clone()
    _hip.add_lora(out, x, [a], [b], [0], indices, build_segment_plan(indices, 1).workspace, 0.5, _hip.FORMS[form])
    want = y.double() + 0.5 * (x.double() @ a[0].double().T) @ b[0].double().T
    assert torch.allclose(out.double(), want, rtol=1e-2, atol=1e-3)
