"""Performance cases of the continuous-batching attention path, through its public entry points.

Kinds of case (the value of ``"kind"``):
  decode    one layer's paged decode attention: ``HipPagedAttention.forward`` over a filled cache, or, with
            ``fused``, ``HipPagedAttention.decode_step`` on the raw projection rows (q/k norm, RoPE, KV store,
            attention), which is what the engine's decode step runs.
  prefill   one layer's causal prefill attention: ``HipBatchPrefillAttention.forward``, on the packed
            activations or, where the prompts have a cached prefix, through the block table.
  block     one layer's whole attention block of a prefill: ``Qwen3Attention.forward`` (qkv projection, q/k norm,
            RoPE, KV store, attention, output projection).
  norm      the decoder's residual add and RMSNorm of a prefill: ``RMSNorm.add_forward``.
  step      one whole decode step of a model by ``DecodeGraphRunner``: the captured graph is replayed on the
            entry's static buffers, as the engine does, and gives logits and the updated cache.

Sequence lengths are fixed by a case's own values, so a case's work does not depend on the seed; tensors and block
tables come from the seed.  Weights are N(0, 0.02) and norm weights N(1, 0.02); cached keys and values and the rows
of a projection are N(0, 1), as normed heads are.
"""
from __future__ import annotations

import math
import random

import torch

from nano_vllm_ascend_amd.block_manager import PagedKVCacheMetadata
from nano_vllm_ascend_amd.config import Qwen3Config
from nano_vllm_ascend_amd.graph import DecodeGraphRunner
from nano_vllm_ascend_amd.layers import HipBatchPrefillAttention, HipPagedAttention, RMSNorm, RotaryEmbedding
from nano_vllm_ascend_amd.paged_kv_cache import PagedKVCache
from nano_vllm_ascend_amd.qwen3 import Qwen3Attention, Qwen3ForCausalLM

D = 128               # head_dim of every configuration
EPS = 1e-6
THETA = 1.0e6
MAX_POSITIONS = 40960
VOCAB = 151936


def listed() -> list[dict]:
    return [
        # The smallest call: one layer's attention of a few short chats; launch latency counts.
        decode("decode_b4_ctx512", 4, 1, 512, bound=512),
        # The framework's headline workload: a decode step of 32 requests in the middle of generation, in the form
        # that the captured step runs it (fused, bound by max_model_len 4096).
        decode("decode_step_b32_ctx2304", 32, 256, 2304, bound=4096, fused=True),
        # The load workload: 100 requests of 2048 prompt tokens, somewhere in their 2048 output tokens.
        decode("decode_b100_ctx4096", 100, 2048, 4096, bound=4096),
        # A model of eight query heads per kv head (Qwen3-32B's ratio) at a middling batch.
        decode("decode_step_gqa8_b16_ctx4096", 16, 512, 4096, hq=64, hkv=8, bound=4096, fused=True),
        # Long documents: a few requests up to the models' 40,960 positions, which also bound the launch.
        decode("decode_b4_ctx40960", 4, 8192, 40960, bound=40960),
        # Prompts of a batch admitted at once, ragged, nothing cached.
        prefill("prefill_b32_2048", 32, 64, 2048),
        # Prompts whose first half is a cached prefix (shared system prompt): the paged route.
        prefill("prefill_prefix_b32_2048", 32, 512, 2048, cached=1024),
        # Two long documents at five query heads per kv head (Qwen3-14B's ratio).
        prefill("prefill_gqa5_b2_12000", 2, 8000, 12000, hq=40, hkv=8),
        # The attention block of the 0.6B shape over 32 short prompts (the published run's 32 x 256).
        block("block_b32_256", 32, 200, 256),
        # Residual add and norm of one prefill batch at a hidden size that is no power of two (Qwen3-4B's).
        norm("norm_12000x2560", 12000, 2560),
        # A whole decode step of Qwen3-0.6B with 8 of its 28 layers: 32 requests, contexts as in the headline workload.
        # (Rounding differences of two correct evaluations grow with depth: 1.3e-2 of the logits at 8 layers,
        # 2.8e-2 at 28.)
        step("step_b32", 32, 256, 2304, layers=8, hidden=1024, inter=3072, hq=16, hkv=8, bound=4096),
        # A few decoder layers and the head of a wider model (hidden 4096, 32 / 8 heads), eight requests.
        step("step_wide_b8", 8, 128, 2048, layers=4, hidden=4096, inter=12288, hq=32, hkv=8, bound=4096),
    ]


def decode(name, batch, lo, hi, hq=16, hkv=8, block_size=128, bound=0, fused=False):
    return _named(name, kind="decode", batch=batch, lo=lo, hi=hi, hq=hq, hkv=hkv, block_size=block_size, bound=bound,
                  fused=fused)


def prefill(name, batch, lo, hi, hq=16, hkv=8, block_size=128, cached=0):
    return _named(name, kind="prefill", batch=batch, lo=lo, hi=hi, hq=hq, hkv=hkv, block_size=block_size,
                  cached=cached)


def block(name, batch, lo, hi, hidden=1024, hq=16, hkv=8, block_size=128, cached=0):
    return _named(name, kind="block", batch=batch, lo=lo, hi=hi, hidden=hidden, hq=hq, hkv=hkv,
                  block_size=block_size, cached=cached)


def norm(name, rows, hidden):
    return _named(name, kind="norm", rows=rows, hidden=hidden)


def step(name, batch, lo, hi, layers, hidden, inter, hq, hkv, block_size=128, bound=4096):
    return _named(name, kind="step", batch=batch, lo=lo, hi=hi, layers=layers, hidden=hidden, inter=inter, hq=hq,
                  hkv=hkv, block_size=block_size, bound=bound)


def _named(name, **case):
    return {"name": name, **case} if name else case


HEADS = [(16, 8), (16, 8), (16, 8), (32, 8), (40, 8), (64, 8), (8, 8), (16, 4), (24, 8), (2, 1)]


def _log(rng, lo, hi) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "block", "norm", "step"])
    hq, hkv = rng.choice(HEADS)
    bs = rng.choice([128, 128, 128, 64, 16, 256])
    if kind == "decode":
        hi = _log(rng, 64, 40960)
        batch = _log(rng, 1, max(1, min(128, 300_000 // hi)))
        lo = rng.choice([1, hi // 2, max(1, hi - 100)])
        bound = rng.choice([0, 4096 * -(-hi // 4096), 40960])
        return decode(None, batch, max(1, lo), hi, hq, hkv, bs, bound, rng.random() < 0.5)
    if kind == "prefill":
        hi = _log(rng, 16, 12000)
        batch = _log(rng, 1, max(1, min(48, 40_000 // hi, 150_000_000 // (hi * hi) + 1)))
        cached = rng.choice([0, 0, 128, 1024])
        return prefill(None, batch, max(1, hi // rng.choice([1, 4, 32])), hi, hq, hkv, bs, cached)
    if kind == "block":
        hi = _log(rng, 8, 2048)
        batch = _log(rng, 1, max(1, min(48, 20_000 // hi)))
        hidden = rng.choice([1024, 2048, 4096])
        return block(None, batch, max(1, hi // rng.choice([1, 4])), hi, hidden, hq, hkv, bs, rng.choice([0, 0, 256]))
    if kind == "norm":
        return norm(None, _log(rng, 1, 40_000), rng.choice([1024, 2048, 2560, 4096, 5120]))
    hidden, inter, heads = rng.choice([(1024, 3072, (16, 8)), (1024, 3072, (16, 8)), (2048, 6144, (16, 8)),
                                       (2560, 9728, (32, 8)), (4096, 12288, (32, 8))])
    hi = _log(rng, 64, 4000)
    return step(None, _log(rng, 1, 128), max(1, hi // 4), hi, rng.randint(2, 6), hidden, inter, heads[0], heads[1],
                128, 4096)


# ------------------------------------------------------------------------------------------------ sizes
def _lens(case) -> list[int]:
    """New tokens (prefill, block) or context lengths (decode, step) of each sequence."""
    rng = random.Random(1_000_003 * case["batch"] + 1_009 * case["lo"] + case["hi"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]


def work(case) -> dict:
    kind = case["kind"]
    if kind == "norm":
        n = case["rows"] * case["hidden"]
        return {"bytes": 2 * (4 * n + case["hidden"]), "flops": 5 * n}
    hq, hkv, lens = case["hq"], case["hkv"], _lens(case)
    total, batch = sum(lens), len(lens)
    if kind == "decode":
        kv_rows = total + (2 * batch if case["fused"] else 0)  # the new token's rows are read and stored
        return {"bytes": 4 * D * hkv * kv_rows + 4 * D * hq * batch + 4 * (-(-total // case["block_size"]) + batch),
                "flops": 4 * D * hq * total}
    if kind == "step":
        h, i, v = case["hidden"], case["inter"], VOCAB
        layer = h * (hq + 2 * hkv) * D + hq * D * h + 3 * h * i
        weights = case["layers"] * layer + v * h
        return {"bytes": 2 * weights + case["layers"] * 4 * D * hkv * (total + batch) + 2 * batch * v,
                "flops": 2 * batch * weights + case["layers"] * 4 * D * hq * total}
    cached = case["cached"]
    pairs = sum(n * cached + n * (n + 1) // 2 for n in lens)
    flops = 4 * D * hq * pairs
    kv_bytes = 4 * D * hkv * (total + cached * batch)
    if kind == "prefill":
        return {"bytes": 4 * D * hq * total + kv_bytes, "flops": flops}
    h = case["hidden"]
    weights = h * (hq + 2 * hkv) * D + hq * D * h
    return {"bytes": 2 * weights + 4 * h * total + kv_bytes, "flops": flops + 2 * total * weights}


def tolerance(case) -> dict:
    """One bf16 rounding of an output is 1.7e-3 rms of its value; an attention's probabilities, and the rows of a
    projection that feeds it, are rounded too.  A whole step rounds several times per layer."""
    if case["kind"] == "norm":
        return {"rel": 5e-3}
    if case["kind"] == "step":
        return {"rel": 3e-2}
    return {"rel": 1e-2}


# ------------------------------------------------------------------------------------------------ states
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, *shape, mean=0.0, std=1.0):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(mean, std, generator=gen)


def _pages(case, lens, seed):
    """A pool that holds every sequence with a block to spare, and its table: distinct blocks in a seeded order."""
    bs = case["block_size"]
    need = [-(-n // bs) for n in lens]
    perm = torch.randperm(sum(need) + 1, generator=torch.Generator().manual_seed(int(seed)))
    width = max(need)
    tables = torch.zeros((len(lens), width), dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        tables[i, :n] = perm[at:at + n].to(torch.int32)
        at += n
    return sum(need) + 1, tables


def _slots(tables, bs, seq, pos):
    return tables[seq, pos // bs].to(torch.int64) * bs + pos % bs


def _kv_cache(gen, case, layers, blocks):
    cache = PagedKVCache(layers, blocks, case["block_size"], case["hkv"], D, torch.bfloat16, torch.device("cuda"))
    cache.key_cache.normal_(generator=gen)
    cache.value_cache.normal_(generator=gen)
    return cache


def _head_norm(gen):
    m = RMSNorm(D, EPS).to(device="cuda", dtype=torch.bfloat16)
    m.weight.data.normal_(1.0, 0.02, generator=gen)
    return m


def _heads(case, qkv):
    """q, k and v as views into the fused projection's rows."""
    t, hq, hkv = qkv.shape[0], case["hq"], case["hkv"]
    return (qkv[:, : hq * D].view(t, hq, D), qkv[:, hq * D : (hq + hkv) * D].view(t, hkv, D),
            qkv[:, (hq + hkv) * D :].view(t, hkv, D))


_ROTARY = {}


def _rotary():
    """The RoPE table, which depends on nothing but the model's constants: every layer of a program shares one."""
    if "table" not in _ROTARY:
        _ROTARY["table"] = RotaryEmbedding(D, MAX_POSITIONS, THETA).to("cuda")
    return _ROTARY["table"]


@torch.no_grad()
def prepare(case, seed) -> dict:
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "block": _prepare_prefill, "norm": _prepare_norm,
            "step": _prepare_step}[case["kind"]](case, seed)


def _prepare_decode(case, seed):
    gen, lens = _generator(seed), _lens(case)
    blocks, tables = _pages(case, lens, seed)
    cache = _kv_cache(gen, case, 1, blocks)
    pos = torch.tensor(lens) - 1
    state = {"case": case, "attn": HipPagedAttention(case["hq"], case["hkv"], D), "cache": cache,
             "heads": _heads(case, _normal(gen, len(lens), (case["hq"] + 2 * case["hkv"]) * D)),
             "tables": tables.cuda(), "context_lens": torch.tensor(lens, dtype=torch.int32).cuda(),
             "positions": pos.cuda(), "bound": max(case["bound"], max(lens)),
             "slots": _slots(tables, case["block_size"], torch.arange(len(lens)), pos).cuda()}
    if case["fused"]:
        state.update(q_norm=_head_norm(gen), k_norm=_head_norm(gen), rotary=_rotary())
    state["workspace"] = state["attn"].workspace(len(lens), state["bound"], torch.device("cuda", 0))
    return state


def _prepare_prefill(case, seed):
    """The packed activations (prefill) or the hidden states and weights (block), and the batch's metadata."""
    gen, lens, cached, bs = _generator(seed), _lens(case), case["cached"], case["block_size"]
    blocks, tables = _pages(case, [n + cached for n in lens], seed)
    cache = _kv_cache(gen, case, 1, blocks)
    ends = torch.tensor([0] + lens).cumsum(0)
    seq = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens))
    pos = torch.arange(int(ends[-1])) - ends[seq] + cached
    slots = _slots(tables, bs, seq, pos)
    md = PagedKVCacheMetadata(
        block_tables=tables.cuda(), context_lens=(torch.tensor(lens, dtype=torch.int32) + cached).cuda(),
        slot_mapping=slots.cuda(), actual_seq_lengths_q=ends[1:].tolist(),
        actual_seq_lengths_kv=[n + cached for n in lens], query_lens=lens, use_paged_prefill=cached > 0,
        cu_seqlens_q=ends.to(torch.int32).cuda(), positions=pos.cuda(), max_query_len=max(lens),
        max_context_len=max(lens) + cached)
    state = {"case": case, "cache": cache, "md": md}
    if case["kind"] == "block":
        config = Qwen3Config(hidden_size=case["hidden"], num_attention_heads=case["hq"],
                             num_key_value_heads=case["hkv"])
        with torch.device("cuda"):
            layer = Qwen3Attention(config, 0, bs, MAX_POSITIONS).to(torch.bfloat16)
        for w in (layer.qkv_weight, layer.o_weight):
            w.data.normal_(0.0, 0.02, generator=gen)
        for n in (layer.q_norm, layer.k_norm):
            n.weight.data.normal_(1.0, 0.02, generator=gen)
        state.update(layer=layer, rotary=_rotary(), hidden=_normal(gen, sum(lens), case["hidden"]))
        return state
    state["attn"] = HipBatchPrefillAttention(case["hq"], case["hkv"], D, bs, MAX_POSITIONS)
    state["heads"] = _heads(case, _normal(gen, sum(lens), (case["hq"] + 2 * case["hkv"]) * D))
    if cached:  # the new tokens' k and v are in the cache before attention runs
        rows = slots.cuda()
        cache.key_cache[0].view(-1, case["hkv"], D)[rows] = state["heads"][1]
        cache.value_cache[0].view(-1, case["hkv"], D)[rows] = state["heads"][2]
    return state


def _prepare_norm(case, seed):
    gen = _generator(seed)
    m = RMSNorm(case["hidden"], EPS).to(device="cuda", dtype=torch.bfloat16)
    m.weight.data.normal_(1.0, 0.02, generator=gen)
    delta, residual = (_normal(gen, case["rows"], case["hidden"]) for _ in range(2))
    return {"case": case, "norm": m, "delta": delta, "residual": residual, "out": torch.empty_like(residual)}


def _prepare_step(case, seed):
    gen, lens, bs = _generator(seed + 1), _lens(case), case["block_size"]
    blocks, tables = _pages(case, lens, seed)
    config = Qwen3Config(vocab_size=VOCAB, hidden_size=case["hidden"], intermediate_size=case["inter"],
                         num_hidden_layers=case["layers"], num_attention_heads=case["hq"],
                         num_key_value_heads=case["hkv"])
    with torch.device("cuda"):
        model = Qwen3ForCausalLM(config, bs, case["bound"]).to(torch.bfloat16)
    model.model.rotary_emb = _rotary()
    model.init_random(seed)
    model.eval()
    cache = _kv_cache(gen, case, case["layers"], blocks)
    runner = DecodeGraphRunner(model, cache, [case["batch"]], max_model_len=case["bound"], block_size=bs)
    ids = torch.randint(0, VOCAB, (case["batch"],), generator=gen, device="cuda")
    entry = runner.entry_for(case["batch"], tables.shape[1], torch.device("cuda", 0), bs)
    pos = torch.tensor(lens) - 1
    entry.buffers["input_ids"].copy_(ids)
    entry.buffers["positions"].copy_(pos)
    entry.buffers["block_tables"][:, : tables.shape[1]].copy_(tables)
    entry.buffers["context_lens"].copy_(torch.tensor(lens, dtype=torch.int32))
    entry.buffers["slot_mapping"].copy_(_slots(tables, bs, torch.arange(len(lens)), pos))
    state = {"case": case, "runner": runner, "entry": entry, "ids": ids, "cache": cache, "model": model}
    with torch.inference_mode():
        runner.replay(entry)  # captures
    return state


# ------------------------------------------------------------------------------------------------ one pass
@torch.inference_mode()
def run(state):
    s = state
    kind = s["case"]["kind"]
    if kind == "norm":
        out = s["norm"].add_forward(s["delta"], s["residual"], s["out"])
        return {"out": out, "residual": s["residual"]}
    if kind == "step":
        s["entry"].buffers["input_ids"].copy_(s["ids"])  # a replay leaves its greedy tokens there
        logits = s["runner"].replay(s["entry"])
        return {"logits": logits, "key_cache": s["cache"].key_cache, "value_cache": s["cache"].value_cache}
    kc, vc = s["cache"].get_physical_cache(0)
    if kind == "block":
        out = s["layer"](s["hidden"], s["rotary"], s["md"].positions, s["cache"], s["md"], True)
        return {"out": out, "key_cache": kc, "value_cache": vc}
    q, k, v = s["heads"]
    if kind == "prefill":
        return {"out": s["attn"](q, k, v, s["md"], kc, vc)}
    if s["case"]["fused"]:
        out = s["attn"].decode_step(q, k, v, s["q_norm"], s["k_norm"], s["rotary"], s["positions"], kc, vc, s["slots"],
                                    s["tables"], s["context_lens"], s["bound"], s["workspace"])
        return {"out": out, "key_cache": kc, "value_cache": vc}
    return {"out": s["attn"](q, kc, vc, s["tables"], s["context_lens"], s["bound"], s["workspace"])}


# ------------------------------------------------------------------------------------------------ in 64 bits
def _rms(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _rope(x, pos):
    """Rotate-half RoPE of [T, heads, D]."""
    freq = THETA ** (-torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)
    angle = pos.to(torch.float64)[:, None] * freq
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., : D // 2], x[..., D // 2 :]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _attend(q, k, v):
    """q [n, Hq, D] are the last n positions of k, v [m, Hkv, D]; causal."""
    n, hq, _ = q.shape
    m, hkv, _ = k.shape
    out = torch.empty_like(q)
    for h in range(hq):
        kh, vh = k[:, h * hkv // hq], v[:, h * hkv // hq].contiguous()
        kt = kh.t().contiguous()
        for r in range(0, n, 4096):
            rows = q[r : r + 4096, h].contiguous()
            s = rows @ kt * D ** -0.5
            seen = torch.arange(m, device="cuda")[None] <= torch.arange(r, r + len(rows), device="cuda")[:, None] + m - n
            out[r : r + 4096, h] = s.masked_fill_(~seen, -math.inf).softmax(-1) @ vh
    return out


def _attend_one(q, k, v):
    """One query row [Hq, D] over k, v [m, Hkv, D]."""
    hq, hkv = q.shape[0], k.shape[1]
    qg = q.view(hkv, hq // hkv, 1, D)
    p = ((qg * k.permute(1, 0, 2)[:, None]).sum(-1) * D ** -0.5).softmax(-1)
    return (p[..., None] * v.permute(1, 0, 2)[:, None]).sum(2).reshape(hq, D)


def _rows(tables, i, n, bs):
    p = torch.arange(n, device="cuda")
    return tables[i, p // bs].long() * bs + p % bs


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "prefill" and work(case)["flops"] > 2e13 or kind == "step" and case["layers"] * case["batch"] > 2000:
        return None
    s = prepare(case, seed)
    if kind == "norm":
        res = s["residual"].double() + s["delta"].double()
        return {"out": _rms(res, s["norm"].weight), "residual": res}
    lens, bs, hkv = _lens(case), case["block_size"], case["hkv"]
    if kind == "step":
        return _exact_step(case, s, lens)
    flat_k, flat_v = (t.view(-1, hkv, D) for t in s["cache"].get_physical_cache(0))
    if kind == "decode":
        q, k, v = (t.double() for t in s["heads"])
        if case["fused"]:
            q = _rope(_rms(q, s["q_norm"].weight), s["positions"])
            k = _rope(_rms(k, s["k_norm"].weight), s["positions"])
        out = torch.empty_like(q)
        for i, n in enumerate(lens):
            rows = _rows(s["tables"], i, n, bs)
            ki, vi = flat_k[rows].double(), flat_v[rows].double()
            if case["fused"]:
                ki[-1], vi[-1] = k[i], v[i]
            out[i] = _attend_one(q[i], ki, vi)
        return {"out": out, "key_cache": None, "value_cache": None} if case["fused"] else {"out": out}
    cached, md = case["cached"], s["md"]
    if kind == "block":
        layer = s["layer"]
        q, k, v = _heads(case, s["hidden"].double() @ layer.qkv_weight.double().t().contiguous())
        q = _rope(_rms(q, layer.q_norm.weight), md.positions)
        k = _rope(_rms(k, layer.k_norm.weight), md.positions)
    else:
        q, k, v = (t.double() for t in s["heads"])
    out = torch.empty_like(q)
    at = 0
    for i, n in enumerate(lens):
        rows = _rows(md.block_tables, i, cached, bs)
        out[at : at + n] = _attend(q[at : at + n], torch.cat((flat_k[rows].double(), k[at : at + n])),
                                   torch.cat((flat_v[rows].double(), v[at : at + n])))
        at += n
    if kind == "prefill":
        return {"out": out}
    out = out.reshape(at, -1) @ s["layer"].o_weight.double().t().contiguous()
    return {"out": out, "key_cache": None, "value_cache": None}


def _exact_step(case, s, lens):
    model, bs, hkv, buf = s["model"], case["block_size"], case["hkv"], s["entry"].buffers

    def linear(x, w):
        return x @ w.double().t().contiguous()

    h = model.model.embed_tokens[s["ids"]].double()
    for l, layer in enumerate(model.model.layers):
        a = layer.self_attn
        q, k, v = _heads(case, linear(_rms(h, layer.input_layernorm.weight), a.qkv_weight))
        q = _rope(_rms(q, a.q_norm.weight), buf["positions"])
        k = _rope(_rms(k, a.k_norm.weight), buf["positions"])
        flat_k, flat_v = (t.view(-1, hkv, D) for t in s["cache"].get_physical_cache(l))
        out = torch.empty_like(q)
        for i, n in enumerate(lens):
            rows = _rows(buf["block_tables"], i, n, bs)
            ki, vi = flat_k[rows].double(), flat_v[rows].double()
            ki[-1], vi[-1] = k[i], v[i]
            out[i] = _attend_one(q[i], ki, vi)
        h = h + linear(out.reshape(len(lens), -1), a.o_weight)
        gate, up = linear(_rms(h, layer.post_attention_layernorm.weight), layer.mlp.gate_up_weight).chunk(2, -1)
        h = h + linear(torch.nn.functional.silu(gate) * up, layer.mlp.down_weight)
    logits = linear(_rms(h, model.model.norm.weight), model.lm_head)
    return {"logits": logits, "key_cache": None, "value_cache": None}
