"""Decode path of hidden sizes that the projections' norm prologue does not take (2560, 4096, 5120, ...)."""
from __future__ import annotations

import pytest
import torch

from nano_vllm_ascend_amd import _C
from nano_vllm_ascend_amd.block_manager import PagedKVCacheMetadata
from nano_vllm_ascend_amd.config import Qwen3Config
from nano_vllm_ascend_amd.layers import RotaryEmbedding
from nano_vllm_ascend_amd.paged_kv_cache import PagedKVCache
from nano_vllm_ascend_amd.qwen3 import Qwen3ForCausalLM


@pytest.mark.gpu
@pytest.mark.parametrize("rows,hidden", [(1, 32), (5, 2016), (16, 2048), (17, 2560), (40, 4096), (33, 5120), (2, 8192)])
def test_rms_norm_tiled_equals_row_major(device, rows, hidden):
    """The tiled norm against add_rms_norm: the sums of squares are added in another order, so an element may round
    to the neighbouring bf16 value (relative 2^-7)."""
    gen = torch.Generator(device=device).manual_seed(hidden)
    buf = torch.randn((rows, hidden + 8), generator=gen, device=device).bfloat16()
    x, w = buf[:, :hidden], torch.randn(hidden, generator=gen, device=device).bfloat16()
    out = _C.tiled_empty(rows, hidden, device).fill_(7.0)
    _C.rms_norm_tiled(x, w, 1e-6, out)
    ref = torch.empty((rows, hidden), dtype=torch.bfloat16, device=device)
    _C.add_rms_norm(None, x.contiguous(), w, ref, 1e-6)
    torch.cuda.synchronize()
    full = _C.untile(out).float()
    assert bool((full[rows:] == 7.0).all())  # padding rows untouched
    diff = (full[:rows] - ref.float()).abs()
    assert bool((diff <= 2.0 ** -7 * ref.float().abs()).all()) and (diff == 0).float().mean().item() > 0.99


def _model(device, hidden, inter, heads, batch):
    config = Qwen3Config(vocab_size=2048, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=2,
                         num_attention_heads=heads, num_key_value_heads=8)
    with torch.device(device):
        model = Qwen3ForCausalLM(config, 16, 512).to(torch.bfloat16)
    model.model.rotary_emb = RotaryEmbedding(128, 512, 1e6).to(device)  # the table stays in fp32
    model.init_random(3)
    model.eval()
    cache = PagedKVCache(2, batch * 4, 16, 8, 128, torch.bfloat16, device)
    gen = torch.Generator(device=device).manual_seed(5)
    cache.key_cache.normal_(generator=gen)
    cache.value_cache.normal_(generator=gen)
    lens = torch.tensor([1 + (13 * i) % 60 for i in range(batch)])
    tables = torch.arange(batch * 4, dtype=torch.int32).view(batch, 4)
    pos = lens - 1
    slots = tables[torch.arange(batch), pos // 16].long() * 16 + pos % 16
    md = PagedKVCacheMetadata(block_tables=tables.to(device), context_lens=lens.int().to(device),
                              slot_mapping=slots.to(device), positions=pos.to(device), max_context_bound=512,
                              decode_workspace=_C.alloc_paged_decode_workspace(batch, heads, 8, 512, device))
    ids = torch.randint(0, 2048, (batch,), generator=gen, device=device)
    return model, cache, md, ids


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,inter,heads,batch", [(2560, 3072, 32, 7), (4096, 8192, 32, 32), (5120, 2560, 40, 17),
                                                      (4096, 4096, 64, 16), (256, 512, 8, 1), (2560, 9728, 32, 20)])
@torch.inference_mode()
def test_wide_decode_matches_the_library_path(device, hidden, inter, heads, batch):
    model, cache, md, ids = _model(device, hidden, inter, heads, batch)

    def step():
        return model(input_ids_flat=ids, position_ids_flat=md.positions, kv_cache=cache, attn_metadata=md,
                     is_prefill=False).logits.float()

    assert model.decode_wide(batch) and not model.decode_fusable(batch) and not model.decode_wide(33)
    with pytest.MonkeyPatch.context() as m:
        m.setattr(model, "decode_wide", lambda rows: False)
        plain = step()
    before = torch.cuda.memory_allocated()
    wide = step()
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() - before == -(-wide.nbytes // 512) * 512  # nothing but the logits stays
    torch.cuda.synchronize()
    # each of the 2 layers rounds its projections to bf16 six times (1.7e-3 rms each) on either path
    assert ((wide - plain).norm() / plain.norm()).item() < 2e-2


@pytest.mark.gpu
@torch.inference_mode()
def test_wide_decode_takes_the_library_path_for_weights_the_kernels_cannot_read(device):
    model, cache, md, ids = _model(device, 2560, 3072, 32, 4)

    def step():
        return model(input_ids_flat=ids, position_ids_flat=md.positions, kv_cache=cache, attn_metadata=md,
                     is_prefill=False).logits.float()

    wide = step()
    down = model.model.layers[1].mlp.down_weight
    down.data = down.data.t().contiguous().t()  # the same values, column by column
    assert not model.decode_wide(4)
    plain = step()
    torch.cuda.synchronize()
    assert ((wide - plain).norm() / plain.norm()).item() < 2e-2


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["data", "in_place", "state_dict", "load"])
@torch.no_grad()
def test_new_weights_reach_eager_steps_and_captured_graphs(device, change):
    """A wide model reads its weights as they are: after any change of them an eager step and a graph captured before
    give the bits of a model that held the new weights from the start."""
    model, cache, md, ids = _model(device, 2560, 3072, 32, 4)
    other, cache2, md2, _ = _model(device, 2560, 3072, 32, 4)
    other.init_random(4)

    def step(m, kv, meta):
        return m(input_ids_flat=ids, position_ids_flat=meta.positions, kv_cache=kv, attn_metadata=meta,
                 is_prefill=False).logits

    first = step(model, cache, md).float()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(model, cache, md)
    if change == "load":
        model.init_random(4)
    elif change == "state_dict":
        model.load_state_dict(other.state_dict())
    else:
        for p, q in zip(model.parameters(), other.parameters()):
            (p.data if change == "data" else p).copy_(q)
    ref = step(other, cache2, md2).float()
    eager = step(model, cache, md).float()
    torch.cuda.synchronize()
    assert torch.equal(eager, ref) and not torch.equal(ref, first)
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.float(), ref)


@pytest.mark.gpu
@torch.inference_mode()
def test_wide_decode_captured_first_equals_eager(device):
    """A capture before any eager step: the replays, with eager steps between them, give the eager bits."""
    model, cache, md, ids = _model(device, 2560, 9728, 32, 4)

    def step():
        return model(input_ids_flat=ids, position_ids_flat=md.positions, kv_cache=cache, attn_metadata=md,
                     is_prefill=False).logits

    torch.mm(torch.ones(8, 8, device=device).bfloat16(), torch.ones(8, 8, device=device).bfloat16())  # library handle
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        got = out.float()
        eager = step().float()
        torch.cuda.synchronize()
        assert torch.equal(got, eager)


@pytest.mark.gpu
@torch.inference_mode()
def test_wide_decode_on_two_streams_at_once(device):
    """Steps of one model queued on two streams share no workspace: each repeats the bits of a step alone."""
    model, cache, md, ids = _model(device, 2560, 9728, 32, 4)
    cache2 = PagedKVCache(2, 16, 16, 8, 128, torch.bfloat16, device)
    cache2.key_cache.copy_(cache.key_cache)
    cache2.value_cache.copy_(cache.value_cache)
    md2 = PagedKVCacheMetadata(**{**md.__dict__, "decode_workspace": _C.alloc_paged_decode_workspace(4, 32, 8, 512,
                                                                                                     device)})

    def step(kv, meta):
        return model(input_ids_flat=ids, position_ids_flat=meta.positions, kv_cache=kv, attn_metadata=meta,
                     is_prefill=False).logits

    alone = step(cache, md).float()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = []
    for _ in range(6):
        for s, kv, meta in zip(streams, (cache, cache2), (md, md2)):
            with torch.cuda.stream(s):
                outs.append(step(kv, meta))
    torch.cuda.synchronize()
    assert all(torch.equal(o.float(), alone) for o in outs)


@pytest.mark.gpu
@torch.inference_mode()
def test_wide_decode_uses_copies_that_were_built(device, monkeypatch):
    """After build_decode_weights the wide path reads the copies, which a load rewrites."""
    model, cache, md, ids = _model(device, 2560, 9728, 32, 4)

    def step():
        return model(input_ids_flat=ids, position_ids_flat=md.positions, kv_cache=cache, attn_metadata=md,
                     is_prefill=False).logits.float()

    rows = step()
    model.build_decode_weights()
    layouts = []
    inner = _C.skinny_linear

    def spy(*args, **kwargs):
        layouts.append(kwargs.get("w_rows", False))
        return inner(*args, **kwargs)

    monkeypatch.setattr(_C, "skinny_linear", spy)
    tiled = step()
    torch.cuda.synchronize()
    assert layouts and not any(layouts)
    assert ((tiled - rows).norm() / rows.norm()).item() < 2e-2  # other K splits
    model.init_random(4)
    again = step()
    other, cache2, md2, _ = _model(device, 2560, 9728, 32, 4)
    other.init_random(4)
    other.build_decode_weights()
    ref = other(input_ids_flat=ids, position_ids_flat=md2.positions, kv_cache=cache2, attn_metadata=md2,
                is_prefill=False).logits.float()
    torch.cuda.synchronize()
    assert torch.equal(again, ref) and not torch.equal(again, tiled)
