"""The work this package is used for, as measurable cases.

A serving engine drives the package in three ways, and the cases follow them:

* ``decode`` - one token per running sequence, every call of the step inside one captured graph:
  the batch's slot ids are planned on the host, uploaded, copied into the graph's buffers and the
  graph is replayed (24 layers of stacked projections).
* ``eager`` - prompts (long segments, one adapter each) and chunked-prefill batches that carry
  single-token decodes as well: planned the same way, one ``add_lora`` call per projection and layer.
* ``linears`` - the LoRA linears themselves, base product included, as model code calls them.

Beside them stand the low-level ops (``ops``) and the admission of an adapter into a slot
(``install``).  Sizes are those of the benchmark configurations (hidden 1024, SwiGLU 4096, q|k|v
1024|256|256, ranks 8..64, up to 256 decode streams, prompts of 64..1024 tokens, mixed batches of
8192 tokens over 128 adapters of different rank), of the default adapter (rank 32 on q, k, v, o) and
of a hidden size other than those (2048), with the same proportions.
"""

from __future__ import annotations

import json
import math
import os
import random
import struct
import sys
import tempfile

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "nanovllm-voxcpm_amd"))

from nanovllm_voxcpm_amd.engine.graph_meta import make_graph_domain_buffers, set_graph_lora_contexts  # noqa: E402
from nanovllm_voxcpm_amd.engine.lora_manager import LoRAModelPayload, LoRARuntime, build_lora_context_from_batch_plan  # noqa: E402
from nanovllm_voxcpm_amd.layers.lora import (  # noqa: E402
    LoRAMergedColumnParallelLinear,
    LoRAQKVParallelLinear,
    LoRARowParallelLinear,
    iter_lora_modules,
)
from nanovllm_voxcpm_amd.lora import LoRAMetadata, get_backend  # noqa: E402
from nanovllm_voxcpm_amd.lora_checkpoint import install_lora_payload, load_voxcpm_lora_checkpoint  # noqa: E402
from nanovllm_voxcpm_amd.lora_ops import lora_expand, lora_shrink  # noqa: E402
from nanovllm_voxcpm_amd.utils.context import (  # noqa: E402
    LM_LORA_DOMAIN,
    LORA_DOMAINS,
    LoRAContext,
    get_lora_context,
    reset_lora_context,
    set_lora_context,
)

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed() -> list[dict]:
    return [
        # the smallest step of a server: one running request, the default adapter targets
        dict(name="decode_1_stream", kind="decode", tokens=1, slots=8, rank=32, ranks="full", hidden=1024, layers=24,
             targets="attention", dtype="bf16", without=0.0),
        # the end-to-end benchmark's decode batch: 64 streams, 32 adapters of rank 32 on all linears
        dict(name="decode_64_streams", kind="decode", tokens=64, slots=32, rank=32, ranks="full", hidden=1024, layers=24,
             targets="all", dtype="bf16", without=0.0),
        # the headline decode batch: 256 streams, 32 adapters of rank 16
        dict(name="decode_256_streams", kind="decode", tokens=256, slots=32, rank=16, ranks="full", hidden=1024, layers=24,
             targets="all", dtype="bf16", without=0.0),
        # a wider model, a ragged batch, adapters of different rank, one stream in ten without an adapter
        dict(name="decode_201_streams_wide", kind="decode", tokens=201, slots=48, rank=64, ranks="mixed", hidden=2048, layers=24,
             targets="all", dtype="fp16", without=0.1),
        # one short prompt by itself: launches and host work are all there is
        dict(name="prompt_37_tokens", kind="eager", batch="prompts", tokens=37, sequences=1, slots=8, rank=32, ranks="full",
             hidden=1024, layers=24, targets="all", dtype="bf16", without=0.0),
        # the prefill benchmark: 16 prompts, 8 adapters of rank 64, a quarter of the prompts without an adapter
        dict(name="prefill_9392_tokens", kind="eager", batch="prompts", tokens=9392, sequences=16, slots=8, rank=64, ranks="full",
             hidden=1024, layers=24, targets="all", dtype="bf16", without=0.25),
        # a few prompts of a wider model
        dict(name="prefill_3001_tokens_wide", kind="eager", batch="prompts", tokens=3001, sequences=5, slots=16, rank=16, ranks="full",
             hidden=2048, layers=24, targets="all", dtype="fp16", without=0.0),
        # chunked prefill: two chunks of 2048 tokens and 4096 decodes over 128 adapters of rank 8..64
        dict(name="mixed_8192_tokens", kind="eager", batch="mixed", tokens=8192, sequences=2, slots=128, rank=64, ranks="mixed",
             hidden=1024, layers=24, targets="all", dtype="bf16", without=0.0),
        # model code around it: four layers' LoRA linears on a batch of prompts
        dict(name="linears_1234_tokens", kind="linears", batch="prompts", tokens=1234, sequences=8, slots=16, rank=32, ranks="full",
             hidden=1024, layers=4, targets="all", dtype="bf16", without=0.125),
        # the low-level ops on a decode batch, one layer's projections
        dict(name="ops_256_tokens", kind="ops", batch="prompts", tokens=256, sequences=256, slots=32, rank=16, ranks="full",
             hidden=1024, layers=4, targets="all", dtype="bf16", without=0.0),
        # the plumbing configuration's element type and sizes: 64 tokens, 4 adapters of rank 16
        dict(name="fp32_64_tokens", kind="eager", batch="prompts", tokens=64, sequences=64, slots=4, rank=16, ranks="full",
             hidden=1024, layers=4, targets="all", dtype="fp32", without=0.0),
        # a new request's adapter comes into a slot: pinned fp32 checkpoint payload, ten layers' default targets
        dict(name="install_adapter", kind="install", slots=8, rank=32, hidden=1024, layers=10, dtype="bf16"),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 1e-9))))


def draw(rng: random.Random) -> dict:
    most = max(work(c)["bytes"] for c in listed())
    while True:
        case = _draw(rng)
        if work(case)["bytes"] <= most and _cells(case) <= 5 * 10**9:
            return case


def _draw(rng: random.Random) -> dict:
    kind = rng.choices(["decode", "prompts", "mixed", "linears", "ops", "fp32", "install"], [6, 4, 2, 2, 1, 1, 1])[0]
    hidden = rng.choice([1024, 1024, 2048])
    rank = rng.choice([8, 16, 24, 32, 32, 48, 64])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    without = rng.choice([0.0, 0.0, 0.1, 0.25])
    slots = _log_int(rng, 4, 64)
    ranks = rng.choice(["full", "full", "mixed"])
    targets = rng.choice(["all", "all", "attention"])
    if kind == "decode":
        return dict(kind="decode", tokens=_log_int(rng, 1, 512), slots=slots, rank=rank, ranks=ranks, hidden=hidden, layers=24,
                    targets=targets, dtype=dtype, without=without)
    if kind == "install":
        return dict(kind="install", slots=slots, rank=rank, hidden=hidden, layers=rng.randint(1, 10), dtype=dtype)
    case = dict(kind="eager", batch="prompts", tokens=0, sequences=1, slots=slots, rank=rank, ranks=ranks, hidden=hidden, layers=24,
                targets=targets, dtype=dtype, without=without)
    if kind == "prompts":
        case["tokens"] = _log_int(rng, 16, 9392)
        case["sequences"] = _log_int(rng, max(1, case["tokens"] // 1024), max(1, min(16, case["tokens"] // 16)))
    elif kind == "mixed":
        case.update(batch="mixed", tokens=_log_int(rng, 512, 8192), slots=_log_int(rng, 8, 128), sequences=rng.randint(1, 4))
    elif kind == "linears":
        case.update(kind="linears", tokens=_log_int(rng, 1, 4096), layers=4)
        case["sequences"] = _log_int(rng, max(1, case["tokens"] // 1024), case["tokens"])
    elif kind == "ops":
        case.update(kind="ops", tokens=_log_int(rng, 1, 512), layers=4, ranks="full")
        case["sequences"] = case["tokens"]
    else:
        case.update(tokens=_log_int(rng, 1, 256), dtype="fp32", layers=4, ranks="full")
        case["sequences"] = case["tokens"]
    return case


# ---- shapes and batches ------------------------------------------------------------------------------


def _projections(case: dict) -> dict[str, tuple[int, list[int]]]:
    """Projection -> (K, output column blocks) of one decoder layer."""
    h = case["hidden"]
    every = {"qkv": (h, [h, h // 4, h // 4]), "o": (h, [h]), "gate_up": (h, [4 * h, 4 * h]), "down": (4 * h, [h])}
    return every if case.get("targets") == "all" else {n: every[n] for n in ("qkv", "o")}


def _batch(case: dict, seed: int) -> tuple[list, list[int]]:
    """(adapter id or None, token count) of every sequence of the batch.  The lengths and the
    sequences without an adapter belong to the case, which adapter a sequence uses to the seed."""
    shape, pick = random.Random(71), random.Random(seed)
    if case["kind"] == "decode":
        counts = [1] * case["tokens"]
    elif case["batch"] == "mixed":
        chunk = case["tokens"] // (2 * case["sequences"])
        counts = [chunk] * case["sequences"] + [1] * (case["tokens"] - chunk * case["sequences"])
    else:
        n = case["sequences"]
        share = [shape.uniform(0.12, 1.88) for _ in range(n)]
        left = case["tokens"] - n
        counts = [1 + int(left * s / sum(share)) for s in share]
        counts[-1] += case["tokens"] - sum(counts)
    n, slots = len(counts), case["slots"]
    off = set(shape.sample(range(n), int(case["without"] * n)))
    weights = [1.0 / (i + 1) ** 1.1 for i in range(slots)] if case.get("batch") == "mixed" else None  # few popular adapters
    chosen = pick.choices(range(slots), weights, k=n)
    return [None if i in off else a for i, a in enumerate(chosen)], counts


def _true_ranks(case: dict) -> list[int]:
    choices = [r for r in (8, 16, 32, 64) if r <= case["rank"]]
    pick = random.Random(73)
    return [pick.choice(choices) if case["ranks"] == "mixed" else case["rank"] for _ in range(case["slots"])]


def _activation_sets(case: dict) -> int:
    """How many layers' activations exist side by side (large batches reuse theirs every four layers)."""
    return case["layers"] if case["tokens"] <= 512 else min(4, case["layers"])


def _cells(case: dict) -> int:
    """Elements of the state, which bounds what is drawn."""
    if case["kind"] == "install":
        return 0
    shapes = _projections(case).values()
    weights = sum(case["slots"] * case["rank"] * (len(w) * k + sum(w)) for k, w in shapes)
    return case["layers"] * weights + _activation_sets(case) * case["tokens"] * sum(k + sum(w) for k, w in shapes)


def work(case: dict) -> dict:
    if case["kind"] == "install":
        h, e = case["hidden"], 2
        cells = case["rank"] * (4 * h + (h + h // 2) + h) * case["layers"]
        return {"bytes": cells * (4 + e), "flops": 0}
    ids, counts = _batch(case, 0)
    ranks = _true_ranks(case)
    tokens = sum(c for a, c in zip(ids, counts) if a is not None)
    rank_sum = sum(ranks[a] for a in {a for a in ids if a is not None})
    token_ranks = sum(ranks[a] * c for a, c in zip(ids, counts) if a is not None)
    e = 4 if case["dtype"] == "fp32" else 2
    cells = flops = other = 0
    for k, widths in _projections(case).values():
        s, n = len(widths), sum(widths)
        cells += rank_sum * (s * k + n)
        flops += 2 * token_ranks * (s * k + n)
        if case["kind"] == "linears":  # base product: every row of x and of the output, the base weight
            cells += case["tokens"] * (k + n) + k * n
            flops += 2 * case["tokens"] * k * n
        else:
            cells += tokens * (k + 2 * n)
        if case["kind"] == "ops":  # the intermediate between the two ops, written and read
            other += 2 * 4 * case["tokens"] * s * case["rank"]
    return {"bytes": case["layers"] * (cells * e + other) + 4 * case["tokens"], "flops": case["layers"] * flops}


def tolerance(case: dict) -> dict | str:
    if case["kind"] == "install":
        return "exact"
    # one rounding of the result to the element type; the base product of a linear rounds once more
    rel = {"bf16": 4e-3, "fp16": 5e-4, "fp32": 1e-5}[case["dtype"]]
    return {"rel": 2 * rel if case["kind"] == "linears" else rel, "max": 8 * rel}


# ---- states ------------------------------------------------------------------------------------------


def _normal(gen: torch.Generator, *shape: int, scale: float = 1.0, dtype: torch.dtype) -> torch.Tensor:
    t = torch.randn(shape, generator=gen, device=DEVICE, dtype=dtype)
    return t if scale == 1.0 else t.mul_(scale)


def _runtime(case: dict) -> LoRARuntime:
    """Every adapter registered and resident, adapter i in slot i."""
    runtime = LoRARuntime(max_loras=case["slots"], max_lora_rank=case["rank"])
    for i in range(case["slots"]):
        runtime.register_lora(f"adapter {i}", LoRAModelPayload(modules={}, rank=case["rank"], alpha=32.0))
        runtime.on_sequence_enqueued(i)
    runtime.build_batch_plan(list(range(case["slots"])), [1] * case["slots"], _load)
    return runtime


def _load(slot_id: int, payload: LoRAModelPayload) -> None:
    """The adapters' weights are in the buffers already."""


def _context(state: dict) -> LoRAContext:
    """What an engine does for every batch: sequences -> slots -> device context."""
    plan = state["runtime"].build_batch_plan(state["adapters"], state["counts"], _load)
    return build_lora_context_from_batch_plan(plan, max_slots=state["slots"], device=DEVICE)


def _metadata(context: LoRAContext) -> LoRAMetadata:
    return LoRAMetadata(context.token_to_slot, context.token_indices_sorted_by_slot, context.active_slot_ids,
                        context.num_tokens_per_slot, context.slot_start_offsets, context.no_lora_flag, context.num_active_loras)


def _clear_beyond(ranks: list[int], a: torch.Tensor, b: torch.Tensor) -> None:
    """Slot buffers hold zeros beyond an adapter's own rank."""
    for slot, r in enumerate(ranks):
        if r < a.size(1):
            a[slot, r:] = 0
            b[slot, :, r:] = 0


def prepare(case: dict, seed: int) -> dict:
    if case["kind"] == "install":
        return _prepare_install(case, seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    state = {"kind": case["kind"], "slots": case["slots"], "runtime": _runtime(case)}
    state["adapters"], state["counts"] = _batch(case, seed)
    dtype, ranks = DTYPES[case["dtype"]], _true_ranks(case)
    if case["kind"] == "linears":
        return _prepare_linears(case, state, gen, dtype, ranks)
    state["backend"] = get_backend()
    # the LoRA linears tell the backend the slots' ranks when some are below that of wide buffers
    told = case["rank"] > 16 and min(ranks) < case["rank"]
    state["effective_rank"] = torch.tensor(ranks, dtype=torch.int32, device=DEVICE) if told else None
    sets, slots, rank = _activation_sets(case), case["slots"], case["rank"]
    calls, outputs = [[] for _ in range(case["layers"])], []
    for k, widths in _projections(case).values():
        x = _normal(gen, sets, case["tokens"], k, dtype=dtype)
        y = _normal(gen, sets, case["tokens"], sum(widths), dtype=dtype)
        outputs.append(y)
        for layer in range(case["layers"]):
            a = [_normal(gen, slots, rank, k, scale=0.02, dtype=dtype) for _ in widths]
            b = [_normal(gen, slots, n, rank, scale=0.04, dtype=dtype) for n in widths]  # alpha / r = 2 folded in
            for a_i, b_i in zip(a, b):
                _clear_beyond(ranks, a_i, b_i)
            packed = y[layer % sets]
            calls[layer].append((list(packed.split(widths, dim=-1)), x[layer % sets], a, b, packed))
    state["calls"], state["outputs"] = [c for layer in calls for c in layer], outputs
    if case["kind"] == "ops":
        state["hidden"] = [torch.empty(len(c[2]), case["tokens"], rank, dtype=torch.float32, device=DEVICE) for c in state["calls"]]
    if case["kind"] == "decode":
        _capture(case, state)
    return state


def _apply(state: dict, metadata: LoRAMetadata) -> None:
    backend, ranks = state["backend"], state["effective_rank"]
    for blocks, x, a, b, packed in state["calls"]:
        backend.add_lora(blocks, x, a, b, indices=metadata.token_to_slot, metadata=metadata, scaling=1.0, y_packed=packed,
                         effective_rank=ranks)


def _capture(case: dict, state: dict) -> None:
    """The decode step of this batch size as a graph over fixed metadata buffers."""
    state["vars"] = {"lora_domains": {d: make_graph_domain_buffers(case["tokens"], case["slots"] + 1, DEVICE) for d in LORA_DOMAINS}}
    kept = [y.clone() for y in state["outputs"]]
    _refresh(state)
    _apply(state, _metadata(get_lora_context(LM_LORA_DOMAIN)))
    torch.cuda.synchronize()
    state["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(state["graph"]):
        _apply(state, _metadata(get_lora_context(LM_LORA_DOMAIN)))
    for y, before in zip(state["outputs"], kept):  # the warm-up has added to them
        y.copy_(before)
    reset_lora_context()


def _refresh(state: dict) -> None:
    contexts = {d: LoRAContext() for d in LORA_DOMAINS}
    contexts[LM_LORA_DOMAIN] = _context(state)
    set_graph_lora_contexts(state["vars"], contexts)


def _prepare_linears(case: dict, state: dict, gen: torch.Generator, dtype: torch.dtype, ranks: list[int]) -> dict:
    h, head = case["hidden"], 64
    kw = dict(max_loras=case["slots"], max_lora_rank=case["rank"])
    modules = []
    with torch.device(DEVICE):
        for _ in range(case["layers"]):
            layer = [LoRAQKVParallelLinear(h, head, h // head, h // 4 // head, **kw), LoRARowParallelLinear(h, h, **kw)]
            if case["targets"] == "all":
                layer += [LoRAMergedColumnParallelLinear(h, [4 * h, 4 * h], **kw), LoRARowParallelLinear(4 * h, h, **kw)]
            modules += layer
    x_of = {}
    with torch.no_grad():
        for m in modules:
            m.to(dtype)
            k = m.weight.size(1)
            m.weight.copy_(_normal(gen, *m.weight.shape, scale=k**-0.5, dtype=dtype))
            for slot, r in enumerate(ranks):
                a = _normal(gen, *((m.lora_A.size(0),) if m.lora_A.dim() == 4 else ()), r, k, scale=0.02, dtype=torch.float32)
                widths = getattr(m, "shard_output_sizes", None) or ([m.q_size, m.kv_size, m.kv_size] if hasattr(m, "q_size") else [])
                b = [_normal(gen, n, r, scale=0.02, dtype=torch.float32) for n in widths or [m.weight.size(0)]]
                m.set_slot_lora(slot, a, b if widths else b[0], effective_rank=r, scaling=2.0)
            if k not in x_of:
                x_of[k] = _normal(gen, case["tokens"], k, dtype=dtype)
    state["linears"] = [(m, x_of[m.weight.size(1)]) for m in modules]
    return state


def _write_checkpoint(directory: str, tensors: dict[str, torch.Tensor], rank: int, alpha: float) -> None:
    """A LoRA checkpoint directory: fp32 tensors in the safetensors layout and the adapter's config."""
    header, at = {}, 0
    for name, t in tensors.items():
        header[name] = {"dtype": "F32", "shape": list(t.shape), "data_offsets": [at, at + 4 * t.numel()]}
        at += 4 * t.numel()
    text = json.dumps(header).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(directory, "lora_weights.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        for t in tensors.values():
            f.write(t.numpy().tobytes())
    with open(os.path.join(directory, "lora_config.json"), "w") as f:
        json.dump({"lora_config": {"r": rank, "alpha": alpha}}, f)


def _prepare_install(case: dict, seed: int) -> dict:
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    h, r, head = case["hidden"], case["rank"], 64
    kw = dict(max_loras=case["slots"], max_lora_rank=r)
    model, tensors = torch.nn.Module(), {}
    for i in range(case["layers"]):
        with torch.device(DEVICE):
            layer = torch.nn.Module()
            layer.qkv_proj = LoRAQKVParallelLinear(h, head, h // head, h // 4 // head, **kw)
            layer.o_proj = LoRARowParallelLinear(h, h, **kw)
        model.add_module(f"layer{i}", layer)
        for leaf, n in (("q_proj", h), ("k_proj", h // 4), ("v_proj", h // 4), ("o_proj", h)):
            tensors[f"layer{i}.{leaf}.lora_A"] = _normal(gen, r, h, scale=0.02, dtype=torch.float32).cpu()
            tensors[f"layer{i}.{leaf}.lora_B"] = _normal(gen, n, r, scale=0.02, dtype=torch.float32).cpu()
    model.to(DTYPES[case["dtype"]])
    with tempfile.TemporaryDirectory() as directory:
        _write_checkpoint(directory, tensors, r, 32.0)
        payload = load_voxcpm_lora_checkpoint(directory)
    slot = seed % case["slots"]
    buffers = []
    for m in iter_lora_modules(model):
        if isinstance(m, LoRAQKVParallelLinear):
            buffers += [m.lora_A[:, slot], m.lora_B_q[slot], m.lora_B_k[slot], m.lora_B_v[slot]]
        else:
            buffers += [m.lora_A[slot], m.lora_B[slot]]
    return {"kind": "install", "model": model, "slot": slot, "payload": payload, "loaded": {}, "outputs": buffers}


# ---- one pass ----------------------------------------------------------------------------------------


def run(state: dict):
    kind = state["kind"]
    if kind == "decode":
        _refresh(state)
        state["graph"].replay()
        return state["outputs"]
    if kind == "install":
        install_lora_payload(state["model"], state["slot"], state["payload"], loaded=state["loaded"])
        return state["outputs"]
    context = _context(state)
    if kind == "linears":
        set_lora_context(context)
        with torch.inference_mode():
            outputs = [m(x) for m, x in state["linears"]]
        reset_lora_context()
        return outputs
    metadata = _metadata(context)
    if kind == "ops":
        args = metadata.as_kernel_metadata(metadata.token_to_slot.numel())
        for (_, x, a, b, packed), h in zip(state["calls"], state["hidden"]):
            lora_shrink(x, a, h, *args, 1.0)
            lora_expand(h, b, packed, *args, offset_start=0, add_inputs=True)
        return state["outputs"] + state["hidden"]
    _apply(state, metadata)
    return state["outputs"]
