"""Tiled copies of the decode weights while the weights are loaded again (CPU: the copies are plain tensors)."""
from __future__ import annotations

import pytest
import torch

from nano_vllm_ascend_amd import _C
from nano_vllm_ascend_amd.config import Qwen3Config
from nano_vllm_ascend_amd.qwen3 import Qwen3ForCausalLM

CONFIG = Qwen3Config(vocab_size=64, hidden_size=1024, intermediate_size=512, num_hidden_layers=2,
                     num_attention_heads=4, num_key_value_heads=2, tie_word_embeddings=True)


def _model():
    model = Qwen3ForCausalLM(CONFIG, 16, 64).to(torch.bfloat16)
    model.init_random(1)
    return model


def _copies(model):
    out = [(model.lm_head_tiled, model.lm_head)]
    for layer in model.model.layers:
        a, m = layer.self_attn, layer.mlp
        out += [(a.qkv_tiled, a.qkv_weight), (a.o_tiled, a.o_weight), (m.gate_up_tiled, m.gate_up_weight),
                (m.down_tiled, m.down_weight)]
    return out


def _assert_current(model):
    for copy, weight in _copies(model):
        assert copy.of(weight) is not None and torch.equal(_C.untile(copy.of(weight)), weight)


def _assert_never_stale(model):
    for copy, weight in _copies(model):
        assert copy.of(weight) is None or torch.equal(_C.untile(copy.of(weight)), weight)


def _state_dict(seed):
    """HF names; q/k/v and gate/up apart."""
    gen = torch.Generator().manual_seed(seed)
    src = _model()
    sd = {"model.embed_tokens.weight": src.model.embed_tokens, "model.norm.weight": src.model.norm.weight}
    for i, layer in enumerate(src.model.layers):
        a, m, p = layer.self_attn, layer.mlp, f"model.layers.{i}."
        q, k, v = a.qkv_weight.split([a.q_size, a.kv_size, a.kv_size])
        gate, up = m.gate_up_weight.chunk(2)
        for name, t in (("self_attn.q_proj", q), ("self_attn.k_proj", k), ("self_attn.v_proj", v),
                        ("self_attn.o_proj", a.o_weight), ("self_attn.q_norm", a.q_norm.weight),
                        ("self_attn.k_norm", a.k_norm.weight), ("mlp.gate_proj", gate), ("mlp.up_proj", up),
                        ("mlp.down_proj", m.down_weight), ("input_layernorm", layer.input_layernorm.weight),
                        ("post_attention_layernorm", layer.post_attention_layernorm.weight)):
            sd[p + name + ".weight"] = t
    return {n: torch.randn(t.shape, generator=gen).to(torch.bfloat16) for n, t in sd.items()}


@pytest.mark.parametrize("built_in", [True, False], ids=["inference", "normal"])
@pytest.mark.parametrize("loaded_in", [True, False], ids=["inference", "normal"])
def test_loading_rewrites_the_copies_in_place(built_in, loaded_in):
    """Decode builds the copies under inference mode; weights are loaded inside or outside of it."""
    model = _model()
    with torch.inference_mode(built_in):
        model.build_decode_weights()
    storage = [copy.storage.data_ptr() for copy, _ in _copies(model)]
    with torch.inference_mode(loaded_in):
        assert model.load_hf_state_dict(_state_dict(2)) == []
        _assert_current(model)
        model.init_random(3)
        _assert_current(model)
    assert [copy.storage.data_ptr() for copy, _ in _copies(model)] == storage  # captured graphs read these


@pytest.mark.parametrize("mode", [True, False], ids=["inference", "normal"])
def test_failed_load_and_its_retry_leave_no_stale_copy(mode):
    model = _model()
    with torch.inference_mode():
        model.build_decode_weights()
    sd = _state_dict(4)
    bad = {**sd, "model.layers.1.self_attn.o_proj.weight": torch.zeros(3, 5)}
    with torch.inference_mode(mode):
        with pytest.raises(RuntimeError):
            model.load_hf_state_dict(bad)
        _assert_never_stale(model)
        assert model.load_hf_state_dict(sd) == []
        _assert_current(model)


def test_failed_build_is_not_used(monkeypatch):
    """A build that runs out of memory part of the way: no copy of the old weights stays in use."""
    model = _model()
    model.build_decode_weights()
    tile, calls = _C.tile, []

    def failing(w):
        calls.append(w)
        if len(calls) == 3:
            raise torch.OutOfMemoryError("no memory for the third copy")
        return tile(w)

    with monkeypatch.context() as m:
        m.setattr(_C, "tile", failing)
        with pytest.raises(torch.OutOfMemoryError):
            model.init_random(5)
    _assert_never_stale(model)
    assert model.lm_head_tiled.of(model.lm_head) is None  # the next decode builds them
    model.build_decode_weights()
    _assert_current(model)


def _prefill_inputs(device, tokens):
    from nano_vllm_ascend_amd.block_manager import PagedKVCacheMetadata
    from nano_vllm_ascend_amd.paged_kv_cache import PagedKVCache

    cache = PagedKVCache(2, 8, 16, 2, 128, torch.bfloat16, device)
    pos = torch.arange(tokens, device=device)
    md = PagedKVCacheMetadata(
        block_tables=torch.arange(8, dtype=torch.int32, device=device)[None], slot_mapping=pos, positions=pos,
        context_lens=torch.tensor([tokens], dtype=torch.int32, device=device), actual_seq_lengths_q=[tokens],
        actual_seq_lengths_kv=[tokens], query_lens=[tokens], max_query_len=tokens, max_context_len=tokens,
        cu_seqlens_q=torch.tensor([0, tokens], dtype=torch.int32, device=device))
    ids = torch.arange(tokens, device=device) % 64
    return dict(input_ids_flat=ids, position_ids_flat=pos, kv_cache=cache, attn_metadata=md, is_prefill=True)


@pytest.mark.gpu
def test_prefill_and_captured_decode_after_a_failed_and_a_corrected_load(device):
    """A 64-token prefill (which reads the copies) and a decode graph captured before the loads give the bits of a
    model that never held other weights."""
    def cuda_model():
        model = _model().to(device)
        model.model.rotary_emb.cos_sin = model.model.rotary_emb.cos_sin.float()
        return model.eval()

    def decode_inputs(kwargs, lens):
        from nano_vllm_ascend_amd.block_manager import PagedKVCacheMetadata

        n = torch.tensor([lens], device=device)
        md = PagedKVCacheMetadata(block_tables=kwargs["attn_metadata"].block_tables, slot_mapping=n - 1,
                                  positions=n - 1, context_lens=n.int(), max_context_bound=128,
                                  decode_workspace=_C.alloc_paged_decode_workspace(1, 4, 2, 128, device))
        return dict(input_ids_flat=n % 64, position_ids_flat=n - 1, kv_cache=kwargs["kv_cache"], attn_metadata=md,
                    is_prefill=False)

    sd = {n: t.to(device) * 0.05 for n, t in _state_dict(6).items()}
    sd["model.layers.0.self_attn.o_proj.weight"] *= 2
    bad = {**sd, "model.layers.1.self_attn.o_proj.weight": torch.zeros(3, 5, device=device)}
    model, fresh = cuda_model(), cuda_model()
    pre = _prefill_inputs(device, 64)
    with torch.inference_mode():
        model(**pre)
        dec = decode_inputs(pre, 65)
        model(**dec)  # builds the copies
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = model(**dec).logits
    with pytest.raises(RuntimeError):
        model.load_hf_state_dict(bad)
    model.load_hf_state_dict(sd)
    fresh.load_hf_state_dict(sd)
    with torch.inference_mode():
        fresh.build_decode_weights()
        pre2 = _prefill_inputs(device, 64)
        got, ref = model(**pre).logits, fresh(**pre2).logits
        ref_dec = fresh(**decode_inputs(pre2, 65)).logits
        for _ in range(2):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, ref_dec)
    assert torch.equal(got, ref) and bool(got.isfinite().all())
