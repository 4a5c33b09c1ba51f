"""The sums of the two launches' shrink (csrc/sgmv.hip) against fp64: no further from it than those of the shrink with two chains of its own
(csrc/slab.hip) in the same K parts.  Both add 32 columns a step in fp32, so their rounding errors grow with the square root of a
chain's length: one chain of all of K would be 1.41 times as far off, and ten per cent are ten times what the mean over
131072 sums or more scatters by."""

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("rank,k,slices,parts", [(8, 1024, 1, 1), (16, 2048, 3, 1), (32, 4096, 1, 3), (64, 1024, 3, 1), (64, 8192, 1, 2)])
def test_no_further_from_fp64_than_two_chains(monkeypatch, rank, k, slices, parts):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    print(f"shrink error rank {rank} K {k} {slices} slices {parts} parts", flush=True)
    tokens, width = 131072 // rank, 64
    g = torch.Generator(device="cuda").manual_seed(k + rank)
    x = torch.randn(tokens, k, generator=g, device="cuda").bfloat16()
    a = [(torch.randn(1, rank, k, generator=g, device="cuda") * 0.05).bfloat16() for _ in range(slices)]
    b = [torch.zeros(1, width, rank, device="cuda", dtype=torch.bfloat16) for _ in range(slices)]
    y = torch.zeros(tokens, width * slices, device="cuda", dtype=torch.bfloat16)
    indices = torch.zeros(tokens, dtype=torch.int32, device="cuda")  # (one slot: the sums lie in the tokens' order)
    plan = build_segment_plan(indices, 1)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, slices, rank, torch.bfloat16), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    want = torch.stack([x.double() @ t[0].double().T for t in a], 1)
    errors = []
    try:
        for slab in (0, 2):
            for name, value in (("MLORA_FORCE_FORM", _hip.FORM_SGMV), ("MLORA_SLAB", slab), ("MLORA_SGMV_KSPLIT", parts)):
                monkeypatch.setenv(name, str(value))
            _hip.reload_knobs()
            _hip.add_lora(y, x, a, b, [width * i for i in range(slices)], indices, plan.workspace, 1.0, _hip.FORM_AUTO, scratch)
            sums = scratch[-16 * want.numel():].view(torch.float32).view(4, *want.shape)[:parts].double().sum(0)
            errors.append(((sums - want).norm() / want.norm()).item())
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert 0 < errors[0] <= 1.1 * errors[1] < 1e-6, errors
