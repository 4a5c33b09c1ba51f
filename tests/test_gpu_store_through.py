"""Small tiles whose y leaves at once (csrc/decode.hip, kThrough) hold the bits of those whose y stays in the L2: every instance's rank, one span per
wavefront and two, spans and tiles that end early, K of the staged form and of the general one."""

import pytest
import torch

B16, F16 = torch.bfloat16, torch.float16


@pytest.mark.gpu
@pytest.mark.parametrize("rank, k, widths, dtype", [
    (8, 1024, [8], B16), (16, 2048, [1032, 64], F16), (16, 512, [264], B16), (24, 1024, [520], B16), (32, 1024, [2056], B16), (32, 96, [72], F16),
    (64, 1024, [1024, 256, 256], F16),
])
def test_same_bits(rank, k, widths, dtype, monkeypatch):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    print(f"store through {rank} {k} {widths} {dtype}", flush=True)
    g = torch.Generator().manual_seed(rank + k)
    lengths = [1, 70, 16, 0, 33]
    indices = torch.tensor([i for i, n in enumerate(lengths) for _ in range(n)] + [-1] * 3, dtype=torch.int32, device="cuda")
    tokens, slots = indices.numel(), len(lengths)
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype).cuda() for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype).cuda() for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype).cuda(), torch.randn(tokens, sum(widths), generator=g).to(dtype).cuda()
    plan = build_segment_plan(indices, slots)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    runs = []
    try:
        monkeypatch.setenv("MLORA_DECODE_SHORT", "0")
        for through in (0, 1):
            monkeypatch.setenv("MLORA_DECODE_THROUGH", str(through))
            _hip.reload_knobs()
            out = y.clone()
            _hip.add_lora(out, x, a, b, cols, indices, plan.workspace, 0.75, _hip.FORM_MFMA)
            runs.append(out)
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.equal(*runs) and not torch.equal(runs[0], y)
    assert torch.equal(runs[0][indices < 0], y[indices < 0])
