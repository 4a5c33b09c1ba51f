"""What AUTO takes for a call and how it cuts it (mlora_choice of the diagnostic library: host arithmetic, nothing is launched)."""

import ctypes

import pytest
import torch

from nanovllm_voxcpm_amd import _hip

NAMES = {code: name for name, code in _hip.FORMS.items()}


def choice(rows, k, widths, rank, slots, active_slots=0, active_tokens=0, room=8 << 20):
    """(form, K parts, columns per range) of a 16-bit call with `room` bytes of workspace beyond what is asked for."""
    args = _hip.MloraAddArgs()
    args.x = args.y = 1 << 28
    args.x_stride, args.y_stride = k, sum(widths)
    args.token_to_slot, args.plan = 1 << 29, 1 << 30
    args.num_tokens, args.k, args.r, args.num_slots, args.num_slices = rows, k, rank, slots, len(widths)
    args.dtype, args.scaling = _hip.dtype_code(torch.bfloat16), 1.0
    for i, n in enumerate(widths):
        args.slices[i].a, args.slices[i].b, args.slices[i].n, args.slices[i].y_col = 1 << 31, 1 << 32, n, sum(widths[:i])
    args.workspace = 1 << 33
    args.workspace_bytes = _hip.add_workspace_bytes(rows, len(widths), rank, torch.bfloat16) + room
    out = (ctypes.c_int32 * 3)()
    assert _hip.load_diag().mlora_choice(ctypes.byref(args), active_slots, active_tokens, out) == 0
    return NAMES[out[0]], out[1], out[2]


@pytest.mark.parametrize("rows,tokens,k,widths,rank,slots", [
    (1331, 665, 1536, [6144, 6144], 24, 32), (2496, 1872, 4096, [4096, 1024, 1024], 24, 64), (5915, 2070, 1024, [1024], 48, 2),
    (451, 225, 2048, [2048], 64, 8), (973, 340, 1024, [256], 24, 32), (4269, 2134, 1024, [4096, 4096], 48, 100), (1821, 637, 2048, [8192, 8192], 64, 100),
    (1536, 768, 1024, [1024], 64, 64), (329, 164, 1024, [256], 64, 64),
])
def test_rows_known_to_have_no_slot_do_not_count(rows, tokens, k, widths, rank, slots):
    assert choice(rows, k, widths, rank, slots, slots, tokens)[0] == choice(tokens, k, widths, rank, slots, slots, tokens)[0]


def test_nothing_to_do_has_no_form():
    args, out = _hip.MloraAddArgs(), (ctypes.c_int32 * 3)(9, 9, 9)
    assert _hip.load_diag().mlora_choice(ctypes.byref(args), 0, 0, out) == 0 and list(out) == [0, 0, 0]
    args.form = 99
    assert _hip.load_diag().mlora_choice(ctypes.byref(args), 0, 0, out) != 0


@pytest.mark.parametrize("rows,k,widths,rank,slots,parts", [
    (2384, 2560, [2560], 48, 1, 4), (2436, 2048, [2048], 40, 3, 4), (3000, 4096, [16384, 16384], 64, 16, 3),
    (9000, 4096, [1024], 64, 3, 3), (2200, 1920, [7680, 7680], 24, 3, 3),
])
def test_k_parts_need_not_divide_k(rows, k, widths, rank, slots, parts):
    form, got, _ = choice(rows, k, widths, rank, slots, slots, rows)
    assert (form, got) == ("sgmv", parts)


def test_as_many_k_parts_as_the_workspace_holds():
    for held in (1, 2, 3):
        room = (held - 4) * 4 * 2200 * 2 * 24  # of four parts
        assert choice(2200, 1920, [7680, 7680], 24, 3, 3, 2200, room)[:2] == ("sgmv", held)


@pytest.mark.parametrize("rows,k,widths,rank,slots,parts", [
    (5051, 8192, [2048], 32, 3, 3), (4000, 1536, [6144, 6144], 32, 40, 1), (6000, 6144, [1536], 32, 8, 4),
])
def test_parts_up_to_rank_32_by_the_same_cost(rows, k, widths, rank, slots, parts):
    assert choice(rows, k, widths, rank, slots, slots, rows)[:2] == ("sgmv", parts) == choice(rows, k, widths, 48, slots, slots, rows)[:2]


@pytest.mark.parametrize("rows,k,widths,rank,slots,tokens,columns", [
    (9392, 1024, [1024], 64, 8, 0, 512),  # nobody counted: half of the tokens may be without adapter, and all the slot ids but one
    (9392, 1024, [1024], 64, 8, 9392, 1024), (9392, 1024, [1024], 64, 8, 7044, 512),
    (1000, 1024, [1024, 256, 256], 64, 128, 1000, 1024),  # a tile for every slot at least: 512 and 384 workgroups, not 308 and 231
])
def test_columns_of_a_range_by_what_is_known(rows, k, widths, rank, slots, tokens, columns):
    form, _, got = choice(rows, k, widths, rank, slots, slots if tokens else 0, tokens)
    assert (form, got) == ("wide", columns)


@pytest.mark.parametrize("k", [1536, 1792, 2048, 2304, 2560, 3072])
def test_one_launch_or_two_by_the_same_cost_at_every_k(k):
    """Over 64-token tiles from one launch to two as the workgroups of 1024 columns spill, wherever K lies."""
    forms = [choice(rows, k, [k], 64, 3, 3, rows)[0] for rows in range(3000, 9400, 200)]
    assert "sgmv" in forms and ("wide" in forms) == (k <= 2048), forms


def test_sums_that_many_ranges_read_have_their_price():
    assert choice(9392, 1024, [4096, 4096], 64, 8)[:2] == ("sgmv", 1) == choice(9392, 1024, [4096, 4096], 64, 8, 8, 7044)[:2]
    assert choice(9392, 4096, [1024], 64, 8, 8, 7044)[:2] == ("sgmv", 2)


def test_parts_fit_the_fullest_xcd():
    # 82 tiles of three slots: runs of 11 a block, 33 workgroups in three parts on 32 compute units
    assert choice(5160, 8192, [2048], 32, 3, 3, 5160)[:2] == ("sgmv", 4)
    assert choice(5000, 8192, [2048], 32, 3, 3, 5000)[:2] == ("sgmv", 3)


@pytest.mark.parametrize("slots", [1, 5, 100, 1000])
def test_more_slot_ids_than_tiles(slots):
    for rows in (1, 40, 700, 3000):
        choice(rows, 2048, [2048, 2048], 64, slots)


@pytest.mark.parametrize("k", [1536, 1792, 2048, 2304, 2560, 3072])
def test_lines_do_not_depend_on_one_k(k):
    """Small tiles, the pair and 64-token tiles meet at tokens x width and at tokens per slot, whatever K is."""
    width = k * k / 1024 + k
    big = ("sgmv", "wide")
    for rank, limit in ((24, 8.5e6), (48, 8.5e6), (64, 8.5e6), (32, 2.1e7 if k == 2048 else 8.5e6)):
        more = int(limit / width) + 40
        assert choice(more, k, [k], rank, 16, 16, more)[0] in big + (("pair",) if more < 1950 else ())  # (128 tiles)
        assert choice(more - 80, k, [k], rank, 4, 4, more - 80)[0] not in big
    for rank in (24, 32, 48, 64):
        assert choice(2400, k, [4 * k, 4 * k], rank, 128, 128, 2400)[0] == "pair"  # 18.75 tokens to a slot
        assert choice(3000, k, [4 * k, 4 * k], rank, 128, 128, 3000)[0] == "sgmv"
        assert choice(1000, k, [4 * k, 4 * k], rank, 128, 0, 0)[0] == "pair" and choice(1200, k, [4 * k, 4 * k], rank, 128, 0, 0)[0] != "pair"


def test_few_tokens_a_slot_take_the_pair_unless_one_launch_repeats_little():
    assert choice(851, 2048, [2048, 512, 512], 48, 117, 88, 851)[0] == "pair"
    assert choice(1100, 1024, [1024, 256, 256], 64, 128, 128, 1100)[0] == "wide"
