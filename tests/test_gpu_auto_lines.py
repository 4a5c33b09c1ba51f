"""The form AUTO takes on both sides of the lines between small tiles, the pair and 64-token tiles: its output has the bits of that form called by
name, and is right."""

import types

import pytest
import torch

from test_gpu_parity import _check, _exact

# tokens, slots, rank, K, widths, form
CASES = [
    # one slice: 16-token tiles that fit the chip, and that do not
    (2400, 32, 64, 1024, [1024], "mfma"),
    (4000, 48, 64, 1024, [1024], "wide"),
    (4000, 48, 16, 1024, [1024], "mfma"),
    (4000, 3, 32, 1024, [1024], "mfma"),
    (5000, 3, 32, 1024, [1024], "wide"),
    # segments of fewer than sixteen tokens with many weights, with few, and longer ones
    (1000, 128, 64, 1024, [4096, 4096], "pair"),
    (1000, 128, 16, 1024, [2048, 2048], "mfma"),
    (1100, 16, 64, 1024, [4096, 4096], "sgmv"),
    (1500, 128, 32, 4096, [1024], "pair"),
    (1500, 64, 64, 4096, [1024], "sgmv"),
    (1000, 64, 64, 4096, [1024], "pair"),
    # K = 2048: one launch over 64-token tiles where its workgroups fill their rounds, two above the small tiles' lines
    (6000, 16, 64, 2048, [2048], "wide"),
    (4000, 16, 64, 2048, [2048], "sgmv"),
    (4000, 3, 64, 2048, [2048, 512, 512], "wide"),
    (1500, 16, 64, 2048, [2048], "sgmv"),  # (up to rank 32 AUTO's shrink is another than by name, with other bits)
    (1500, 16, 16, 2048, [2048, 512, 512], "mfma"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_auto_takes_the_form_of_its_side(case):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    tokens, slots, rank, k, widths, form = CASES[case]
    print(f"auto {CASES[case]}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(case)
    indices = (torch.arange(tokens, dtype=torch.int32) * slots // tokens).cuda()
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    a = [(rand(slots, rank, k) * 0.05).bfloat16() for _ in widths]
    b = [(rand(slots, n, rank) * 0.1).bfloat16() for n in widths]
    x, y = rand(tokens, k).bfloat16(), rand(tokens, sum(widths)).bfloat16()
    exact, mag = _exact(types.SimpleNamespace(a=a, b=b, widths=widths), x, y, indices)
    plan = build_segment_plan(indices, slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, torch.bfloat16) + (8 << 20), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    outs = []
    for f in ("auto", form):
        out = y.clone()
        _hip.add_lora(out, x, a, b, cols, indices, plan.workspace, 1.0, _hip.FORMS[f], scratch, active_slots=slots, active_tokens=tokens)
        outs.append(out)
    _check(outs[0], y, exact, mag, indices, f"auto at {CASES[case]}")
    assert torch.equal(*outs)
