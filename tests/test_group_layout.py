"""How the low-level ops over tiles of a slot are laid over a grid (csrc/group_layout.h, host arithmetic): whatever slots the
tokens have, every token lies in one tile and every tile has a place."""

import ctypes
import random

import numpy as np
import pytest

TILE = 16


def _layout(tokens: int, slots: int, parts: int, extra: int, count: int = 0) -> tuple[int, ...]:
    """(by token, places, slots8, own tiles, narrow width, width of a slot of `count` tokens, its further tiles)."""
    from nanovllm_voxcpm_amd import _hip

    out = (ctypes.c_int32 * 7)()
    _hip.load_diag().mlora_group_layout(tokens, slots, parts, extra, count, out)
    return tuple(out)


def _needed(tokens: int, slots: int, parts: int, extra: int, counts: list[int]) -> int:
    return sum(_layout(tokens, slots, parts, extra, c)[6] for c in counts if c)


def _even(tokens: int, used: int) -> list[int]:
    return [tokens // used + (i < tokens % used) for i in range(used)]


@pytest.mark.parametrize("parts", [1, 4, 12, 32])
@pytest.mark.parametrize("tokens,slots,used", [(64, 32, 9), (300, 64, 25), (255, 64, 64), (512, 64, 40), (96, 32, 19)])
def test_even_batches_over_some_of_the_slots_have_a_place_for_every_tile(tokens, slots, used, parts):
    by_token, places, slots8, tiles, *_ = _layout(tokens, slots, parts, 0)
    assert by_token == 0 and slots8 >= slots
    assert _needed(tokens, slots, parts, 0, _even(tokens, used)) <= places - slots8 * tiles


def test_random_batches_have_a_place_for_every_tile():
    pick = random.Random(5)
    for tokens, slots in [(255, 64), (240, 64), (224, 64), (208, 64), (96, 32)] * 40:
        counts = [0] * slots
        for _ in range(tokens):
            counts[pick.randrange(slots)] += 1
        _, places, slots8, tiles, *_ = _layout(tokens, slots, 4, 1)
        assert _needed(tokens, slots, 4, 1, counts) <= places - slots8 * tiles


def _sizes():
    yield from ((t, s, p) for t in range(1, 81) for s in range(1, t) for p in (1, 7, 40))
    pick = random.Random(6)
    for _ in range(400):
        tokens = pick.randrange(2, 4097)
        yield tokens, pick.randrange(1, min(tokens, 1024)), pick.choice([1, 2, 4, 6, 16, 48, 200])


def test_the_worst_split_of_the_tokens_has_a_place_for_every_tile():
    """A slot's tiles hold its tokens without a gap, and no two slots need more further places than one slot with the tokens of
    both: then the worst split is one slot with all of them, for which there are places."""
    checked = set()
    for tokens, slots, parts in _sizes():
        by_token, places, slots8, tiles, narrow, *_ = _layout(tokens, slots, parts, 1)
        assert by_token == 0 and slots8 > slots and slots8 % 8 == 0 and narrow in (4, 8, TILE)
        assert places - slots8 * tiles >= _layout(tokens, slots, parts, 1, tokens)[6]
        most = min(tokens, 700)
        if any(key[:2] == (tiles, narrow) and key[2] >= most for key in checked):
            continue
        checked.add((tiles, narrow, most))
        further = np.zeros(most + 1, dtype=np.int64)
        for count in range(most + 1):
            width, further[count] = _layout(tokens, slots, parts, 1, count)[5:]
            covered = (tiles + further[count]) * width
            assert covered >= count and (further[count] == 0 or (width == TILE and covered - TILE < count))
        both = np.add.outer(np.arange(most + 1), np.arange(most + 1))
        inside = both <= most
        assert (np.add.outer(further, further)[inside] <= further[both[inside]]).all()


def test_grids_over_the_tokens_have_a_place_for_each():
    for tokens, slots in [(1, 1), (1, 64), (7, 7), (64, 64), (63, 1024)]:
        by_token, places, *_ = _layout(tokens, slots, 4, 0)
        assert by_token == 1 and places == tokens
