"""MLORA_NO_FASTCALL=1 keeps every host path to Python, and the Python paths of the low-level ops, batch contexts, slot
installs and LoRA linears enqueue what the C++ ones enqueue: the same bits."""

import random
import types

import pytest
import torch

from nanovllm_voxcpm_amd import _hip


def _keep_to_python(monkeypatch, yes: bool) -> None:
    if yes:
        monkeypatch.setenv("MLORA_NO_FASTCALL", "1")
    else:
        monkeypatch.delenv("MLORA_NO_FASTCALL", raising=False)
    _hip.reload_knobs()
    assert (_hip.load_fastcall() is None) == yes


def test_no_host_path_asks_the_module_that_is_switched_off(monkeypatch):
    from nanovllm_voxcpm_amd.engine.lora_manager import _context_in_one_launch
    from nanovllm_voxcpm_amd.lora import HipLoRABackend
    from nanovllm_voxcpm_amd.lora_checkpoint import install_lora_payload
    from nanovllm_voxcpm_amd.lora_ops import lora_expand, lora_shrink

    def refuse(*_):
        raise AssertionError("the C++ host path was asked")

    names = ("shrink", "expand", "run_totals", "build_context", "install_batch", "create", "call", "call_stacked")
    monkeypatch.setattr(_hip, "_FASTCALL", types.SimpleNamespace(**{n: refuse for n in names}))
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    x, slots = torch.zeros(2, 8), torch.zeros(2, dtype=torch.int32)

    def every_path():
        yield lambda: lora_shrink(x, [torch.zeros(1, 4, 8)], torch.zeros(1, 2, 4), slots, None, None, None, None, False, 1, 1.0)
        yield lambda: lora_expand(torch.zeros(1, 2, 4), [torch.zeros(1, 8, 4)], x, slots, None, None, None, None, False, 1)
        yield lambda: _context_in_one_launch([0], [2], 1, "cuda:0")
        yield lambda: install_lora_payload(torch.nn.Module(), 0, types.SimpleNamespace(modules={}, packed=None))
        yield lambda: HipLoRABackend()._fast_state()

    for off in (False, True):
        if off:
            _keep_to_python(monkeypatch, True)
        for path in every_path():
            try:
                path()
                asked = False
            except AssertionError:
                asked = True
            except RuntimeError as exc:  # (no GPU here: the Python path got as far as that)
                assert "must live on the GPU" in str(exc)
                asked = False
            assert asked is not off


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("tokens,k,rank,widths", [(1, 64, 8, [16]), (256, 1024, 16, [1024, 256, 256]), (33, 100, 12, [40, 7])])
def test_low_level_ops(monkeypatch, dtype, tokens, k, rank, widths):
    from nanovllm_voxcpm_amd.lora_ops import lora_expand, lora_shrink
    from oracle import lora_apply as oracle

    g, slots = torch.Generator().manual_seed(tokens), 5
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, sum(widths) + 3, generator=g).to(dtype)
    a, b = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype) for _ in widths], [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype) for n in widths]
    ids = torch.randint(-1, slots, (tokens,), generator=g, dtype=torch.int32)
    results = []
    for python in (False, True):
        _keep_to_python(monkeypatch, python)
        hidden, out = torch.full((len(widths), tokens, rank), 7.0, device="cuda"), y.cuda()
        meta = (ids.cuda(), None, None, None, None, False, slots)
        lora_shrink(x.cuda(), [t.cuda() for t in a], hidden, *meta, 0.5)
        lora_expand(hidden, [t.cuda() for t in b], out, *meta, offset_start=3, add_inputs=True)
        results.append((hidden.cpu(), out.cpu()))
    assert all(torch.equal(one, other) for one, other in zip(*results))
    want = oracle.lora_shrink(x, a, ids, 0.5, torch.float32)
    assert torch.allclose(results[0][0], want, rtol=1e-5, atol=1e-5 * want.abs().max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["singles", "runs", "none"])
def test_batch_contexts(monkeypatch, name):
    from nanovllm_voxcpm_amd.engine.lora_manager import LoRABatchPlan, build_lora_context_from_batch_plan

    torch.zeros(1, device="cuda")
    slots, counts = {"singles": ([7, -1, 3, 7, 0], [1] * 5), "runs": ([3, -1, 5, 3], [700, 5, 0, 17]), "none": ([-1, 2], [4, 0])}[name]
    built = []
    for python in (False, True):
        _keep_to_python(monkeypatch, python)
        built.append(build_lora_context_from_batch_plan(LoRABatchPlan.from_runs({}, list(slots), list(counts)), max_slots=8, device="cuda:0"))
    for field in ("token_to_slot", "token_indices_sorted_by_slot", "active_slot_ids", "num_tokens_per_slot", "slot_start_offsets"):
        one, other = (getattr(c, field) for c in built)
        assert (one is None) == (other is None) and (one is None or torch.equal(one, other)), field
    assert built[0].no_lora_flag == built[1].no_lora_flag and built[0].num_active_loras == built[1].num_active_loras


@pytest.mark.gpu
@pytest.mark.parametrize("rank", [8, 32, 48])
def test_lora_linears(monkeypatch, rank):
    """Three layers under one context: the first linear of the step looks everything up, the others take add_lora_stacked."""
    from nanovllm_voxcpm_amd.engine.lora_manager import build_lora_context_from_slot_list
    from nanovllm_voxcpm_amd.layers.lora import LoRAMergedColumnParallelLinear, LoRAQKVParallelLinear, LoRARowParallelLinear
    from nanovllm_voxcpm_amd.lora import HipLoRABackend, set_backend_for_testing
    from nanovllm_voxcpm_amd.utils.context import set_lora_context

    pick, g, slots = random.Random(rank), torch.Generator().manual_seed(rank), 4
    kw = dict(max_loras=slots, max_lora_rank=rank)
    layers = []
    for _ in range(3):
        layers += [LoRAQKVParallelLinear(512, 64, 8, 2, **kw), LoRARowParallelLinear(512, 512, **kw), LoRAMergedColumnParallelLinear(512, [512, 512], **kw)]
    x = torch.randn(70, 512, generator=g).bfloat16().cuda()
    with torch.no_grad():
        for m in layers:
            m.cuda().bfloat16()
            m.weight.copy_(torch.randn(m.weight.shape, generator=g) * 0.04)
            for slot in range(slots):
                r = pick.choice([rank, rank // 2])
                a = torch.randn(*m.lora_A.shape[:-3], r, 512, generator=g) * 0.05
                b = [torch.randn(n, r, generator=g) * 0.1 for n in ([512, 128, 128] if hasattr(m, "q_size") else [512, 512] if a.dim() == 3 else [512])]
                m.set_slot_lora(slot, a, b if a.dim() == 3 else b[0], effective_rank=r, scaling=1.5)
    ids = [pick.randrange(-1, slots) for _ in range(70)]
    results = []
    for python in (False, True):
        _keep_to_python(monkeypatch, python)
        backend = HipLoRABackend()
        set_backend_for_testing(backend)
        outs = []
        with torch.no_grad():
            for _ in range(2):  # the second step's weight buffers are known
                set_lora_context(build_lora_context_from_slot_list(ids, max_slots=slots, device="cuda:0"))
                outs += [m(x) for m in layers]
        results.append([t.cpu() for t in outs])
        if python:
            assert backend._fastcall is None
        else:
            handled, passed_on = backend._fastcall.counters(backend._fast_state())
            assert handled >= len(layers) - 1, (handled, passed_on)
    assert all(torch.equal(one, other) for one, other in zip(*results))


@pytest.mark.gpu
@pytest.mark.parametrize("layers,types_", [(1, [torch.bfloat16]), (14, [torch.bfloat16]), (14, [torch.bfloat16, torch.float32, torch.float16])])
def test_slot_installs(monkeypatch, layers, types_):
    """Up to 56 targets, more than one launch's table holds, in buffers and from sources of one element type or of several."""
    from nanovllm_voxcpm_amd.engine.lora_manager import LoRAModelPayload, LoRAModulePayload
    from nanovllm_voxcpm_amd.layers.lora import LoRAQKVParallelLinear, LoRARowParallelLinear, iter_lora_modules
    from nanovllm_voxcpm_amd.lora_checkpoint import install_lora_payload

    g, slots, rank, slot = torch.Generator().manual_seed(layers), 3, 16, 2
    model, modules = torch.nn.Module(), {}
    for i in range(layers):
        layer = torch.nn.Module()
        layer.qkv_proj = LoRAQKVParallelLinear(128, 64, 2, 1, max_loras=slots, max_lora_rank=rank)
        layer.o_proj = LoRARowParallelLinear(128, 128, max_loras=slots, max_lora_rank=rank)
        layer.to("cuda", types_[i % len(types_)])
        model.add_module(f"layer{i}", layer)
        r, source = [16, 5, 8][i % 3], types_[(i // 2) % len(types_)]
        for leaf, widths in (("qkv_proj", [128, 64, 64]), ("o_proj", [128])):
            a = torch.randn(len(widths), r, 128, generator=g).to("cuda", source)
            b = [torch.randn(n, r, generator=g).to("cuda", source) for n in widths]
            modules[f"layer{i}.{leaf}"] = LoRAModulePayload(a if len(b) > 1 else a[0], b if len(b) > 1 else b[0], r, -1.75)
    payload, states = LoRAModelPayload(modules, 16, 32.0), []
    for python in (False, True):
        _keep_to_python(monkeypatch, python)
        for m in iter_lora_modules(model):
            for t in (m.lora_A, *m._b_buffers()):
                t.data.fill_(7.0)
            m.clear_slot_lora(slot)
            for t in (m.lora_A, *m._b_buffers()):
                t.data.fill_(7.0)
        install_lora_payload(model, slot, payload)
        states.append([t.detach().cpu().clone() for m in iter_lora_modules(model)
                       for t in (m.lora_A, *m._b_buffers(), m.effective_lora_rank, m.lora_scaling, m.lora_base_scaling)])
        for name, m in payload.modules.items():
            module = model.get_submodule(name)
            a = module.lora_A[:, slot] if module.lora_A.dim() == 4 else module.lora_A[slot]
            assert torch.equal(a[..., : m.effective_rank, :], m.lora_a.to(a.dtype)) and not a[..., m.effective_rank :, :].any(), name
            for b, src in zip(module._b_buffers(), m.lora_b if isinstance(m.lora_b, list) else [m.lora_b]):
                assert torch.equal(b[slot][:, : m.effective_rank], (src * m.scaling).to(b.dtype)), name
                assert not b[slot][:, m.effective_rank :].any() and (b[:slot] == 7).all(), name
            assert module.effective_lora_rank[slot].item() == m.effective_rank and module.lora_scaling[slot].item() == m.scaling
    assert all(torch.equal(one, other) for one, other in zip(*states))
