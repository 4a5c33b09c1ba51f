"""Segment metadata by several workgroups: batches at the edges of what one workgroup holds (512 tokens), against the integer
oracle, and plans of runs against the plan of the same ids in a vector, on every word that a list reaches."""

import pytest
import torch

from test_gpu_parity import test_metadata_bit_exact_random as check_against_the_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,slots,p_neg", [(64, 64, 0.0), (511, 1, 0.0), (512, 64, 0.2), (513, 63, 0.2), (600, 4, 1.0), (1024, 1024, 0.1),
                                                (1025, 2, 0.5), (1537, 16, 0.0)])
def test_edges_of_a_workgroup(tokens, slots, p_neg):
    check_against_the_oracle(tokens, slots, p_neg)


def _reached(workspace, tokens, slots):
    """What the apply kernels may read of a plan."""
    from nanovllm_voxcpm_amd import _hip
    from oracle import segment_meta as oracle

    ws, r4 = workspace.tolist(), lambda v: (v + 3) & ~3
    counts = 16 + r4(tokens)
    small = (counts + r4(slots + 1) + r4(slots + 2) + 31) & ~31
    cap_small, cap_big = ((tokens + 15) // 16 + min(slots, tokens) + 7) & ~7, oracle.big_tile_capacity(tokens, slots)
    big = small + 32 * cap_small
    rows = big + 4 * cap_big
    over = rows + 64 * cap_big
    words = ws[:16] + ws[16 : 16 + ws[_hip.PLAN_NUM_LORA_TOKENS]] + ws[counts : counts + slots + 1] + ws[counts + r4(slots + 1) :][: slots + 2]
    words += ws[small : small + 32 * (ws[_hip.PLAN_TILES_SHORT] + ws[_hip.PLAN_TILES_LONG_SMALL])] + ws[big:rows] + ws[over:]
    for q in range(cap_big):
        if ws[big + 4 * q] >= 0:
            words += ws[rows + 64 * q : rows + 64 * (q + 1)]
    return words


@pytest.mark.parametrize("slots,runs", [
    (4, [(3, 512)]),
    (4, [(3, 200), (1, 0), (3, 313)]),
    (16, [(2, 587), (-1, 63), (7, 0), (15, 1), (2, 700), (-1, 5), (15, 700)]),
    (8, [(9, 0), (1, 3), (8, 2), (1, 700)]),  # (ids of no slot: one in an empty run, one that counts)
    (128, [((5 * i) % 129 - 1, i % 9) for i in range(336)]),
    (1024, [((7 * i) % 1024, 1) for i in range(700)]),
])
def test_plans_of_runs(slots, runs):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.engine.lora_manager import _context_in_one_launch
    from nanovllm_voxcpm_amd.lora_ops import build_segment_plan

    torch.zeros(1, device="cuda")
    ids = [s for s, c in runs for _ in range(c)]
    vector = torch.tensor(ids, dtype=torch.int32, device="cuda")
    want = build_segment_plan(vector, slots).workspace
    assert want[_hip.PLAN_BAD_SLOT].item() == any(s >= slots for s in ids)
    if any(s >= slots for s, _ in runs):  # (a context refuses such ids; the launch itself flags them)
        import ctypes as C

        got = torch.zeros_like(want)
        args = (_hip.MloraMetaArgs * 1)()
        args[0].stream, args[0].num_tokens, args[0].max_slots, args[0].plan = torch.cuda.current_stream().cuda_stream, len(ids), slots, got.data_ptr()
        arrays = [(C.c_int32 * len(runs))(*column) for column in zip(*runs)]
        rc = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int32, C.c_void_p, C.c_void_p, C.c_int32)(_hip.entry_point("mlora_meta_build_runs"))(
            C.cast(args, C.c_void_p), 1, C.cast(arrays[0], C.c_void_p), C.cast(arrays[1], C.c_void_p), len(runs))
        assert rc == 0
    else:
        context = _context_in_one_launch([s for s, _ in runs], [c for _, c in runs], slots, "cuda:0")
        assert context.token_to_slot.tolist() == ids
        got = context.token_to_slot._mlora_plan[0]
    assert _reached(got, len(ids), slots) == _reached(want, len(ids), slots)
