"""The low-level shrink and expand over tiles of a slot (csrc/group.hip) at the sizes where they can go wrong: one token,
tiles just filled and one over, more tokens of a slot than it has places for, many slots just above that, slots without tokens, ids that
name no slot, grids over the slots and over the tokens, ranks that are no multiple of eight (shrink) or of a block, ragged and tiny
slices, every element type; where the tiles are forced and where the library chooses."""

import random

import pytest
import torch

B16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

# tokens, slots, rank, K, slice widths, how the tokens are spread, element type, type of the intermediate
CASES = [
    (1, 1, 8, 1024, [4], "even", B16, F32),
    (1, 5, 16, 2048, [64, 60], "none", F16, F32),
    (15, 3, 12, 1024, [256], "one", B16, B16),
    (16, 40, 24, 1024, [260, 8], "one", F16, F16),
    (17, 16, 64, 3072, [512], "one", B16, F32),
    (33, 40, 40, 1024, [100, 1028, 12], "even", B16, F16),
    (64, 2, 33, 1024, [516], "even", F16, F32),
    (100, 7, 1, 9216, [64], "popular", B16, F32),
    (257, 9, 56, 1024, [1032, 256], "popular", B16, F32),
    (512, 3, 16, 1024, [1024, 256, 256], "one", F16, F32),
    (513, 600, 8, 1024, [72], "even", B16, F32),
    (4096, 3, 48, 1024, [8], "popular", B16, B16),
    (900, 64, 32, 1024, [512], "even", B16, F32),
]


def _ids(how: str, tokens: int, slots: int, pick: random.Random) -> list[int]:
    if how == "none":
        return [pick.choice([-1, slots, slots + 7]) for _ in range(tokens)]
    if how == "one":
        return [slots - 1] * tokens
    if how == "popular":
        return [0 if pick.random() < 0.7 else pick.randrange(-1, slots + 1) for _ in range(tokens)]
    return [pick.randrange(-1, slots + 1) for _ in range(tokens)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_ops_over_tiles_against_fp64(case, monkeypatch):
    tokens, slots, rank, k, widths, how, dtype, h_dtype = CASES[case]
    print(f"group ops {CASES[case]}", flush=True)
    # (the tiles wherever they are possible / one workgroup per token)
    _check(_ids(how, tokens, slots, random.Random(case)), slots, rank, k, widths, dtype, h_dtype, case, ("2", "0"), monkeypatch)


# tokens, slot ids, how many of those are in use (0: every token's slot at random over all of them)
UNEVEN = [(64, 32, 9), (300, 64, 25), (255, 64, 0), (208, 64, 0), (96, 32, 0), (130, 24, 9)]


@pytest.mark.gpu
@pytest.mark.parametrize("rank,widths,dtype", [(32, [1024], B16), (64, [1024], F16), (32, [1024, 256, 256], F16), (64, [2048, 2048], B16)])
@pytest.mark.parametrize("tokens,slots,used", UNEVEN)
def test_uneven_batches_where_the_library_chooses(tokens, slots, used, rank, widths, dtype, monkeypatch):
    """Many slots with a token or two more than their own tiles hold at the narrow width."""
    print(f"group ops {(tokens, slots, used, rank, widths, dtype)}", flush=True)
    pick = random.Random(tokens)
    ids = [(t % used) * (slots // used) if used else pick.randrange(slots) for t in range(tokens)]
    pick.shuffle(ids)
    _check(ids, slots, rank, 1024, widths, dtype, F32, tokens, (None, "2"), monkeypatch)  # the library's choice, and the tiles wherever that lies


def _check(ids, slots, rank, k, widths, dtype, h_dtype, seed, uses, monkeypatch):
    """Shrink into a buffer of NaN and expand, with MLORA_GROUP as each of `uses` (None: unset), against fp64."""
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops import lora_expand, lora_shrink

    tokens, g = len(ids), torch.Generator().manual_seed(seed)
    ids = torch.tensor(ids, dtype=torch.int32)
    x = torch.randn(tokens, k + 8, generator=g).to(dtype)[:, :k]
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype) for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype) for n in widths]
    h = (torch.randn(len(widths), tokens, rank, generator=g)).to(h_dtype)
    y = torch.randn(tokens, sum(widths) + 8, generator=g).to(dtype)
    known = (ids >= 0) & (ids < slots)
    slot = torch.where(known, ids, torch.zeros_like(ids)).long()
    got = {}
    try:
        for use in uses:
            monkeypatch.setenv("MLORA_GROUP", use) if use else monkeypatch.delenv("MLORA_GROUP", raising=False)
            _hip.load().mlora_reload_knobs()
            out = torch.full((len(widths), tokens, rank), float("nan"), dtype=h_dtype, device="cuda")
            lora_shrink(x.cuda(), [t.cuda() for t in a], out, ids.cuda(), None, None, None, None, False, 0, 0.5)
            added, written = y.cuda(), y.cuda()
            lora_expand(h.cuda(), [t.cuda() for t in b], added, ids.cuda(), None, None, None, None, False, 0, offset_start=4, add_inputs=True)
            lora_expand(h.cuda(), [t.cuda() for t in b], written, ids.cuda(), None, None, None, None, False, 0, offset_start=4, add_inputs=False)
            got[use] = [t.cpu() for t in (out, added, written)]
    finally:
        monkeypatch.undo()
        _hip.load().mlora_reload_knobs()
    unit = {B16: 2.0**-8, F16: 2.0**-11, F32: 2.0**-24}  # of a rounding
    exact = [t.double() for t in (x, h.to(dtype), y)]
    for out, added, written in got.values():
        col = 4
        assert torch.equal(added[:, :4], y[:, :4]) and torch.equal(written[:, :4], y[:, :4])
        for i, n in enumerate(widths):
            rows = a[i].double()[slot]
            want, size = [0.5 * torch.einsum("tk,trk->tr", v, w) * known[:, None] for v, w in ((exact[0], rows), (exact[0].abs(), rows.abs()))]
            # K sums in fp32, in any order, then one rounding to the output's type (fp16: subnormal below 2^-14)
            assert ((out[i].double() - want).abs() <= k * 2.0**-24 * size + unit[h_dtype] * want.abs() + 2.0**-25).all()
            wide = b[i].double()[slot]
            delta, size = [torch.einsum("tr,tnr->tn", v, w) for v, w in ((exact[1][i], wide), (exact[1][i].abs(), wide.abs()))]
            slack = 2 * rank * 2.0**-24 * size + unit[dtype] * delta.abs() + 2.0**-25  # the product, rounded to the weights' type
            kept = y[:, col : col + n]
            total = exact[2][:, col : col + n] + delta
            assert ((added[:, col : col + n].double() - total).abs() <= slack * 1.01 + unit[dtype] * (total.abs() + slack))[known].all()
            assert ((written[:, col : col + n].double() - delta).abs() <= slack)[known].all()
            assert torch.equal(added[:, col : col + n][~known], kept[~known]) and torch.equal(written[:, col : col + n][~known], kept[~known])
            col += n
        assert torch.equal(added[:, col:], y[:, col:]) and torch.equal(written[:, col:], y[:, col:])
