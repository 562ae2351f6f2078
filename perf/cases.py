"""The framework's work as its users have it done, sized for timing.

`listed()` names the cases, `draw(rng)` gives further ones of the same ranges, `prepare` makes what
a program holds before the call, `run` is one pass through the public entry points, `work` says what
the pass cannot do without, `exact` the same outputs in 64 bits and `tolerance` how far two correct
implementations at the same precision may be apart.

The shapes are the engine's: Qwen2.5-1.5B's attention (12 query heads over 2 kv heads, head dim 128,
16-token cache blocks), its MLP (1536 -> 2 x 8960 -> 1536), its vocabulary (151,936) and the 16-chat
workload of the benchmark; the general kernel's cases are the head dims and types of its tests.
"""
import math
import random
import sys

import numpy as np
import torch

sys.path.insert(0, "my-inference-engine_amd")

from graphs import DecodeGraphs  # noqa: E402
from kernels.fa2 import (FlashAttention2Function, fa2_paged, fa2_paged_varlen,  # noqa: E402
                         fa2_varlen)
from kernels.sample import sample_tokens  # noqa: E402
from kv_cache import KVCache  # noqa: E402
from model import MLP, QWEN25_1P5B, Qwen2ForCausalLM  # noqa: E402

DEV = "cuda"
BLOCK = 16
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
GROWTH = 4096  # tokens a decoding chat may still append in one state of the model case


def listed():
    return [
        # a long prompt in one sequence, the benchmark's headline
        {"name": "prefill_4096", "kind": "dense", "dtype": "bf16", "heads": 12, "kv_heads": 2,
         "rows": 1, "queries": 4096, "keys": 4096, "ragged": False},
        # a padded batch of ordinary prompts of odd lengths, the reference's own call, in fp16
        {"name": "prefill_3x437_fp16", "kind": "dense", "dtype": "fp16", "heads": 12,
         "kv_heads": 2, "rows": 3, "queries": 437, "keys": 437, "ragged": True},
        # 16 sequences of 16 to 1024 tokens packed back to back, without a cache
        {"name": "varlen_16x1024", "kind": "varlen", "dtype": "bf16", "rows": 16, "lo": 16,
         "hi": 1024, "mix": 0},
        # a chat's next message: 150 new tokens over a cached history
        {"name": "followup_150_of_3001", "kind": "followup", "dtype": "bf16", "rows": 1,
         "queries": 150, "keys": 3001},
        # the first step of 16 chats: their prompts packed into one launch over the paged cache
        {"name": "mixed_16_prompts", "kind": "mixed", "dtype": "bf16", "rows": 16, "lo": 32,
         "hi": 1000, "mix": 1},
        # a decode step of many long chats, the benchmark's second headline
        {"name": "decode_64x8192", "kind": "decode", "dtype": "bf16", "rows": 64, "lo": 128,
         "hi": 8192, "mix": 2},
        # one chat's decode step, the smallest call there is
        {"name": "decode_1x1500", "kind": "decode", "dtype": "bf16", "rows": 1, "lo": 1500,
         "hi": 1500, "mix": 3},
        # the reference's CPU-sized call in its own type
        {"name": "fp32_512", "kind": "general", "dtype": "fp32", "heads": 12, "kv_heads": 2,
         "rows": 1, "queries": 512, "keys": 512, "dim": 128, "dim_v": 128},
        # head dim 64, the other size in wide use, a batch of prompts
        {"name": "dim64_4x1000", "kind": "general", "dtype": "bf16", "heads": 12, "kv_heads": 2,
         "rows": 4, "queries": 1000, "keys": 1000, "dim": 64, "dim_v": 64},
        # one layer's MLP in a decode step of 16 chats
        {"name": "mlp_16", "kind": "mlp", "rows": 16},
        # the next token of 16 chats
        {"name": "sample_16", "kind": "sample", "dtype": "bf16", "rows": 16, "vocab": 151936,
         "temperature": 1.0},
        # a whole decode step of 16 chats, replayed from its graph: what serving spends its time on
        {"name": "model_decode_16", "kind": "model", "rows": 16, "lo": 32, "hi": 1000, "mix": 4},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["dense", "varlen", "followup", "mixed", "decode", "general", "mlp",
                       "sample", "model"])
    dtype = rng.choice(["bf16", "fp16"])
    if kind == "dense":
        t = _log(rng, 17, 4095)
        heads, kv_heads = rng.choice([(12, 2), (12, 2), (16, 4), (8, 8)])
        rows = max(1, min(rng.randint(1, 4), 12 * 4096 ** 2 // (heads * t * t)))
        if heads * rows * t * t > 12 * 4096 ** 2:
            heads, kv_heads = 12, 2
        return {"kind": kind, "dtype": dtype, "heads": heads, "kv_heads": kv_heads, "rows": rows,
                "queries": t, "keys": t, "ragged": rows > 1}
    if kind in ("varlen", "mixed"):
        hi = _log(rng, 100, 1100)
        return {"kind": kind, "dtype": dtype, "rows": rng.randint(2, 24), "lo": rng.randint(1, 64),
                "hi": hi, "mix": rng.randint(10, 10 ** 6)}
    if kind == "followup":
        return {"kind": kind, "dtype": dtype, "rows": rng.choice([1, 1, 2]),
                "queries": _log(rng, 5, 700), "keys": _log(rng, 800, 8000)}
    if kind == "decode":
        hi = _log(rng, 200, 8192)
        return {"kind": kind, "dtype": dtype, "rows": _log(rng, 1, 64),
                "lo": rng.randint(1, hi), "hi": hi, "mix": rng.randint(10, 10 ** 6)}
    if kind == "general":
        d = rng.choice([32, 64, 64, 256])
        dtype = rng.choice(["bf16", "fp16", "fp32"])
        if dtype == "fp32":
            d = rng.choice([64, 128])
        t = _log(rng, 60, 1500)
        return {"kind": kind, "dtype": dtype, "heads": 12, "kv_heads": 2, "rows": rng.randint(1, 4),
                "queries": t, "keys": t, "dim": d, "dim_v": d}
    if kind == "mlp":
        return {"kind": kind, "rows": _log(rng, 1, 1024)}
    if kind == "sample":
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp32"]), "rows": rng.randint(1, 32),
                "vocab": _log(rng, 20000, 152000), "temperature": rng.choice([0.7, 1.0, 1.0])}
    hi = _log(rng, 40, 1000)
    return {"kind": "model", "rows": rng.randint(1, 16), "lo": rng.randint(1, 32), "hi": hi,
            "mix": rng.randint(10, 10 ** 6)}


# -- inputs ---------------------------------------------------------------------------------------
def _lens(case):
    r = random.Random(case["mix"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["rows"])]


def _row_keys(case):
    """Keys of each row of a padded batch: the first row is full, the others are shorter."""
    r = random.Random(case["queries"] * 31 + case["rows"])
    n = case["keys"]
    return [n] + [r.randint(max(1, n // 3), n) for _ in range(case["rows"] - 1)]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, dtype, *shape):
    return torch.randn(*shape, generator=g, device=DEV).to(dtype)


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _pool(g, dtype, keys):
    """One layer of a paged cache holding rows of `keys` keys, blocks in a random order:
    (k pool, v pool, block table, lengths)."""
    need = [math.ceil(n / BLOCK) for n in keys]
    total = sum(need) + 8
    perm = torch.randperm(total, generator=g, device=DEV).to(torch.int32)
    table = torch.zeros(len(keys), max(need), dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[at:at + n]
        at += n
    buf = _randn(g, dtype, 2, total * BLOCK, 2, 128)
    return buf[0], buf[1], table, _i32(keys)


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    dtype = DTYPES[case.get("dtype", "bf16")]
    if kind in ("dense", "general"):
        d, dv = case.get("dim", 128), case.get("dim_v", 128)
        B, T, S = case["rows"], case["queries"], case["keys"]
        q = _randn(g, dtype, B, case["heads"], T, d)
        k = _randn(g, dtype, B, case["kv_heads"], S, d)
        v = _randn(g, dtype, B, case["kv_heads"], S, dv)
        return {"kind": "dense", "q": q, "k": k, "v": v,
                "lens": _i32(_row_keys(case)) if case.get("ragged") else None}
    if kind == "varlen":
        lens = _lens(case)
        n = sum(lens)
        return {"kind": kind, "q": _randn(g, dtype, n, 12, 128), "k": _randn(g, dtype, n, 2, 128),
                "v": _randn(g, dtype, n, 2, 128), "longest": max(lens),
                "cu": _i32(np.concatenate([[0], np.cumsum(lens)]).tolist())}
    if kind == "followup":
        kp, vp, table, lens = _pool(g, dtype, [case["keys"]] * case["rows"])
        q = _randn(g, dtype, case["rows"], 12, case["queries"], 128)
        return {"kind": kind, "q": q, "kp": kp, "vp": vp, "table": table, "lens": lens,
                "longest": case["keys"]}
    if kind == "mixed":
        lens = _lens(case)
        kp, vp, table, dev_lens = _pool(g, dtype, lens)
        return {"kind": kind, "q": _randn(g, dtype, sum(lens), 12, 128), "kp": kp, "vp": vp,
                "table": table, "lens": dev_lens, "longest": max(lens),
                "cu": _i32(np.concatenate([[0], np.cumsum(lens)]).tolist())}
    if kind == "decode":
        lens = _lens(case)
        kp, vp, table, dev_lens = _pool(g, dtype, lens)
        return {"kind": kind, "q": _randn(g, dtype, case["rows"], 12, 1, 128), "kp": kp, "vp": vp,
                "table": table, "lens": dev_lens, "longest": max(lens)}
    if kind == "mlp":
        cfg = QWEN25_1P5B
        with torch.device("meta"):
            mlp = MLP(cfg)
        mlp = mlp.to(dtype).to_empty(device=DEV)
        with torch.no_grad():
            for prm in mlp.parameters():
                prm.copy_(_randn(g, dtype, *prm.shape) * 0.02)
        return {"kind": kind, "mlp": mlp, "x": _randn(g, dtype, case["rows"], 1, cfg.hidden_size)}
    if kind == "sample":
        return {"kind": kind, "logits": _randn(g, dtype, case["rows"], case["vocab"]),
                "temperature": case["temperature"], "seed": seed}
    # the model with its cache of `rows` chats and the captured decode step
    cfg, lens = QWEN25_1P5B, _lens(case)
    with torch.device("meta"):
        model = Qwen2ForCausalLM(cfg)
    inv_freq = 1.0 / (cfg.rope_theta ** (torch.arange(0, cfg.head_dim, 2).float() / cfg.head_dim))
    model = model.to(dtype).to_empty(device=DEV).eval()
    model.inv_freq = inv_freq.to(dtype).to(DEV)
    model.init_random(std=0.02, seed=seed)
    # As in a trained model the residual stream outweighs what one layer adds to it, so that a
    # rounding in one layer is not amplified by all that follow (with N(0, 0.02) throughout, the
    # logits of a 16-bit pass are 4% off the same pass in 64 bits; this way 1.3%).
    with torch.no_grad():
        model.embed_tokens.weight.mul_(50)
        for layer in model.layers:
            layer.self_attn.o_proj.weight.mul_((2 * cfg.num_layers) ** -0.5)
            layer.mlp.down_proj.weight.mul_((2 * cfg.num_layers) ** -0.5)
    blocks = sum(math.ceil((n + GROWTH) / BLOCK) for n in lens)
    cache = KVCache(blocks, BLOCK, DEV, dtype, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim)
    cache.buf.normal_(generator=g)
    seqs = [cache.alloc() for _ in lens]
    cache.prepare_packed(seqs, lens)  # the chats' histories: block tables and device lengths
    cache.advance(seqs, lens)
    rows = next(b for b in (1, 2, 4, 8, 16) if b >= len(lens))
    graphs = DecodeGraphs(model, cache, buckets=(rows,))
    tokens = torch.randint(0, cfg.vocab_size, (len(lens),), generator=g, device=DEV).tolist()
    return {"kind": "model", "graphs": graphs, "seqs": seqs, "tokens": tokens}


# -- one pass -------------------------------------------------------------------------------------
def run(state):
    s, kind = state, state["kind"]
    if kind == "dense":
        return FlashAttention2Function.apply(s["q"], s["k"], s["v"], True, s["lens"])
    if kind == "varlen":
        return fa2_varlen(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["longest"], is_causal=True)
    if kind == "followup":
        return fa2_paged(s["q"], s["kp"], s["vp"], s["table"], s["lens"], max_kv_len=s["longest"],
                         is_causal=True)
    if kind == "mixed":
        return fa2_paged_varlen(s["q"], s["kp"], s["vp"], s["cu"], s["table"], s["lens"],
                                s["longest"], max_kv_len=s["longest"])
    if kind == "decode":
        return fa2_paged(s["q"], s["kp"], s["vp"], s["table"], s["lens"], max_kv_len=s["longest"])
    if kind == "mlp":
        with torch.no_grad():
            return s["mlp"](s["x"])
    if kind == "sample":
        return sample_tokens(s["logits"], s["temperature"], s["seed"], 1)
    return s["graphs"].run(s["seqs"], s["tokens"])


# -- what a pass cannot do without ----------------------------------------------------------------
def _pairs(queries, keys):
    """(query, key) pairs of one row under the bottom-right causal mask."""
    first = keys - queries + 1  # keys the first query sees (may be <= 0: it sees none)
    lo = max(first, 1)
    return (lo + keys) * (keys - lo + 1) // 2 if keys >= lo else 0


def work(case):
    kind = case["kind"]
    size = 4 if case.get("dtype") == "fp32" else 2
    if kind in ("dense", "general"):
        d, dv = case.get("dim", 128), case.get("dim_v", 128)
        keys = _row_keys(case) if case.get("ragged") else [case["keys"]] * case["rows"]
        T, H = case["queries"], case["heads"]
        return {"bytes": size * (case["rows"] * H * T * (d + dv)
                                 + sum(keys) * case["kv_heads"] * (d + dv)),
                "flops": 2 * (d + dv) * H * sum(_pairs(T, n) for n in keys)}
    if kind in ("varlen", "mixed"):
        lens = _lens(case)
        return {"bytes": 2 * sum(lens) * 128 * 2 * (12 + 2),
                "flops": 512 * 12 * sum(_pairs(n, n) for n in lens)}
    if kind == "followup":
        return {"bytes": case["rows"] * 512 * (12 * case["queries"] + 2 * case["keys"]),
                "flops": case["rows"] * 512 * 12 * _pairs(case["queries"], case["keys"])}
    if kind == "decode":
        lens = _lens(case)
        return {"bytes": sum(lens) * 1024 + case["rows"] * 12 * 512
                + sum(math.ceil(n / BLOCK) for n in lens) * 4,
                "flops": 512 * 12 * sum(lens)}
    cfg = QWEN25_1P5B
    H, inter = cfg.hidden_size, cfg.intermediate_size
    if kind == "mlp":
        return {"bytes": 2 * (3 * H * inter + 2 * case["rows"] * H),
                "flops": 2 * 3 * H * inter * case["rows"]}
    if kind == "sample":
        return {"bytes": case["rows"] * (case["vocab"] * size + 4), "flops": 0}
    lens, rows = _lens(case), case["rows"]
    qkv = (cfg.num_heads + 2 * cfg.num_kv_heads) * cfg.head_dim
    weights = (cfg.num_layers * (H * qkv + qkv + cfg.num_heads * cfg.head_dim * H + 3 * H * inter
                                 + 2 * H) + cfg.vocab_size * H + H)
    return {"bytes": 2 * weights + cfg.num_layers * 1024 * (sum(lens) + rows)
            + 2 * rows * cfg.vocab_size,
            "flops": 2 * weights * rows + cfg.num_layers * 512 * 12 * (sum(lens) + rows)}


# -- the same in 64 bits --------------------------------------------------------------------------
def _attend(q, k, v, causal=True):
    """One row: q [Hq, T, d], k/v [Hkv, S, *] -> [Hq, T, dv], softmax over the keys each query
    sees, the last query seeing the last key; a query that sees none gives zeros."""
    Hq, T, d = q.shape
    S, n_rep = k.shape[1], Hq // k.shape[0]
    out = torch.zeros(Hq, T, v.shape[-1], dtype=torch.float64, device=q.device)
    hidden = (torch.arange(S, device=q.device)[None, :]
              > torch.arange(T, device=q.device)[:, None] + (S - T)) if causal else None
    for h in range(Hq):
        kk, vv = k[h // n_rep].double(), v[h // n_rep].double()
        s = (q[h].double() @ kk.t().contiguous()) / math.sqrt(d)
        if causal:
            s.masked_fill_(hidden, -math.inf)
        out[h] = torch.nan_to_num(torch.softmax(s, -1)) @ vv
    return out


def _keys_of(pool, table, n):
    """The first n keys of a row of the paged pool, [Hkv, n, d]."""
    slots = (table.long()[:, None] * BLOCK + torch.arange(BLOCK, device=DEV)).reshape(-1)[:n]
    return pool[slots].transpose(0, 1)


def _exact_model(case, s):
    """The decode step in 64 bits: the decoder over the rows' new tokens, their histories read out
    of the cache."""
    graphs, cfg = s["graphs"], QWEN25_1P5B
    model, cache = graphs.model, graphs.cache
    lens, d, half = _lens(case), cfg.head_dim, cfg.head_dim // 2
    f = lambda t: t.detach().double()  # noqa: E731
    ids = torch.tensor(s["tokens"], device=DEV)
    x = f(model.embed_tokens.weight[ids])
    pos = torch.tensor(lens, device=DEV, dtype=torch.float64)
    freq = f(model.inv_freq)  # as the model holds them: the model is in 16 bits as a whole
    ang = torch.cat([pos[:, None] * freq, pos[:, None] * freq], -1)[:, None]  # [B, 1, d]

    def rope(t):
        return t * ang.cos() + torch.cat([-t[..., half:], t[..., :half]], -1) * ang.sin()

    def norm(t, w):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + cfg.rms_norm_eps) * f(w)

    B = len(lens)
    tables = [torch.tensor(cache._block_tables[q], device=DEV) for q in s["seqs"]]
    for i, layer in enumerate(model.layers):
        at = layer.self_attn
        qkv = norm(x, layer.input_layernorm.weight) @ f(at.qkv_proj.weight).t() + f(at.qkv_proj.bias)
        q, k, v = qkv.split([at.q_size, at.kv_size, at.kv_size], -1)
        q = rope(q.view(B, cfg.num_heads, d))
        k, v = rope(k.view(B, cfg.num_kv_heads, d)), v.view(B, cfg.num_kv_heads, d)
        rows = []
        for b, n in enumerate(lens):
            kk = torch.cat([f(_keys_of(cache.k_pool(i), tables[b], n)), k[b][:, None]], 1)
            vv = torch.cat([f(_keys_of(cache.v_pool(i), tables[b], n)), v[b][:, None]], 1)
            rows.append(_attend(q[b][:, None], kk, vv, causal=False).reshape(-1))
        x = x + torch.stack(rows) @ f(at.o_proj.weight).t()
        h = norm(x, layer.post_attention_layernorm.weight) @ f(layer.mlp.gate_up_proj.weight).t()
        gate, up = h.split(cfg.intermediate_size, -1)
        x = x + (gate * torch.sigmoid(gate) * up) @ f(layer.mlp.down_proj.weight).t()
    return norm(x, model.norm.weight) @ f(model.embed_tokens.weight).t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":  # token ids
        return None
    s = prepare(case, seed)
    with torch.no_grad():
        if kind == "model":
            return _exact_model(case, s)
        if kind in ("dense", "general"):
            lens = s["lens"].tolist() if s["lens"] is not None else [case["keys"]] * case["rows"]
            return torch.stack([_attend(s["q"][b], s["k"][b, :, :n], s["v"][b, :, :n])
                                for b, n in enumerate(lens)])
        if kind == "mlp":
            mlp = s["mlp"]
            gate, up = (s["x"].double() @ mlp.gate_up_proj.weight.double().t()).chunk(2, -1)
            return (gate * torch.sigmoid(gate) * up) @ mlp.down_proj.weight.double().t()
        if kind == "varlen":
            cu = s["cu"].tolist()
            rows = [_attend(*(s[t][lo:hi].transpose(0, 1) for t in "qkv"))
                    for lo, hi in zip(cu[:-1], cu[1:])]
            return torch.cat([r.transpose(0, 1) for r in rows])
        lens = s["lens"].tolist()
        kv = [(_keys_of(s["kp"], s["table"][b], n), _keys_of(s["vp"], s["table"][b], n))
              for b, n in enumerate(lens)]
        if kind == "mixed":
            cu = s["cu"].tolist()
            return torch.cat([_attend(s["q"][lo:hi].transpose(0, 1), *kv[b]).transpose(0, 1)
                              for b, (lo, hi) in enumerate(zip(cu[:-1], cu[1:]))])
        return torch.stack([_attend(s["q"][b], *kv[b]) for b in range(case["rows"])])


def tolerance(case):
    """About four times what was seen between two correct passes: the same attention in the two
    work-group shapes of the prefill kernel (bf16 1.4e-3 to 2.6e-3, single values to 0.06; fp16 an
    eighth of that), products summed in another order or rounded elsewhere (the MLP 4e-3 off 64
    bits, the whole model 8e-3 from one order to another), fp32 3e-7."""
    kind, dtype = case["kind"], case.get("dtype", "bf16")
    if kind == "sample":
        return "exact"
    if kind == "model":
        return {"rel": 0.03, "max": 0.3}
    if kind == "mlp":
        return {"rel": 0.012, "max": 0.1}
    if dtype == "fp32":
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 0.01, "max": 0.2} if dtype == "bf16" else {"rel": 0.00125, "max": 0.025}
