"""The form AUTO takes on both sides of the lines that its rules draw by tiles and workgroups: its output has the bits
of that form called by name, and is right."""

import types

import pytest
import torch

from test_gpu_parity import _check, _exact

pytestmark = pytest.mark.gpu

# tokens, slots, slots in use, rank, K, widths, form
CASES = [
    # K = 8192: eight parts per tile over the slots while they fit the chip together, else the pair
    (24, 24, 24, 16, 8192, [2048], "slot"),
    (26, 26, 26, 16, 8192, [2048], "pair"),
    (200, 16, 16, 32, 8192, [2048], "slot"),
    (320, 20, 20, 32, 8192, [2048], "pair"),
    (18, 18, 18, 64, 8192, [2048], "slot"),
    (19, 19, 19, 64, 8192, [2048], "pair"),
    # K parts of buffers of a rank between 32 and 64
    (8, 8, 8, 48, 8192, [2048], "pair"),
    (8, 8, 8, 48, 4096, [1024], "pair"),
    (8, 8, 8, 24, 4096, [1024], "slot"),
    # the pair against 64-token tiles
    (2000, 8, 4, 64, 4096, [1024], "pair"),
    (2100, 8, 4, 64, 4096, [1024], "sgmv"),
    # three slices: a second round of 16-token tiles
    (700, 16, 8, 64, 1024, [1024, 256, 256], "mfma"),
    (1000, 16, 8, 64, 1024, [1024, 256, 256], "wide"),
    (1300, 16, 8, 32, 512, [512, 128, 128], "mfma"),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_auto_takes_the_form_of_its_side(case):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    tokens, slots, used, rank, k, widths, form = CASES[case]
    print(f"auto {CASES[case]}", flush=True)
    g = torch.Generator().manual_seed(case)
    indices = (torch.arange(tokens, dtype=torch.int32) * used // tokens).cuda()
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).bfloat16().cuda() for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).bfloat16().cuda() for n in widths]
    x, y = torch.randn(tokens, k, generator=g).bfloat16().cuda(), torch.randn(tokens, sum(widths), generator=g).bfloat16().cuda()
    exact, mag = _exact(types.SimpleNamespace(a=a, b=b, widths=widths), x, y, indices)
    plan = build_segment_plan(indices, slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, torch.bfloat16) + (8 << 20), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    outs = []
    for f in ("auto", form):
        out = y.clone()
        _hip.add_lora(out, x, a, b, cols, indices, plan.workspace, 1.0, _hip.FORMS[f], scratch, active_slots=used)
        outs.append(out)
    _check(outs[0], y, exact, mag, indices, f"auto at {CASES[case]}")
    assert torch.equal(*outs)
