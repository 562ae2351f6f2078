"""Qwen2-architecture causal LM whose attention runs on the MI355X paged kernels.

Mirrors the reference's model.py (Qwen2ForCausalLM, model.py:141-207) layer for layer -- fp32
RMSNorm (model.py:43-55), rotate-half RoPE with theta 1e6 (model.py:58-65,148-155), biased q/k/v
projections (model.py:81-84), SwiGLU MLP (model.py:112-120), tied embeddings and last-position
logits (model.py:204-207) -- with two deliberate differences on the GPU path:

  * Attention reads K/V straight from the paged cache inside the kernel (kernels.fa2.fa2_paged)
    instead of gathering a dense copy every layer of every step (KVCache.read, kv_cache.py:117-121,
    called at model.py:97) and then calling the padded kernel (model.py:103).
  * The q/k/v and gate/up projections are single fused GEMMs (one launch instead of three/two).
  * RoPE and the cache write are one HIP launch (kernels.rope.rope_kv_write) instead of the
    elementwise RoPE ops and two index_copy_ (model.py:92,96), with bitwise the same results.
  * Each residual add and the RMSNorm after it are one HIP launch (kernels.model_ops.add_rmsnorm)
    and SiLU x up is one more (kernels.model_ops.silu_mul), instead of about twenty small torch
    launches per layer, with the same rounding points.
  * A step of few tokens (a decode step's rows) runs its projections on hand-written kernels
    (kernels.few_rows) that stream the weights in their own layout and do the norm, RoPE and cache
    write, SwiGLU and residual add of each in the same launch: four launches per layer beside
    attention's, with the same rounding points.
  * For more tokens the gate/up GEMM and the tied lm_head multiply by a cached transposed copy of
    their weight ([in, out] row-major), the layout hipBLASLt has the faster kernels for.  The
    parameters keep the reference's layout; the copy is rebuilt if a weight changes.

forward_mixed() runs one step over rows that append different numbers of tokens -- decoding chats
(one token each) and newly admitted prompts -- packed back to back: every projection, norm and MLP
runs once over all packed tokens, attention goes to the paged decode kernel for the leading
one-token rows and to the paged varlen prefill kernel for the prompt rows, and only each row's last
token reaches the logits.  The reference runs each admitted prompt as a forward of its own
(chat.py:157-185, one per tick, chat.py:247-253) beside the batched decode step.

On CPU tensors the model takes the reference's own fallback (dense read + fp32 SDPA with the
bottom-right mask, model.py:104-107,181-195), which only the CPU tests of the scheduler use; the
attention kernels themselves have no CPU path.
"""
from dataclasses import dataclass

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad

from kernels import few_rows
from kernels.fa2 import fa2_paged, fa2_paged_varlen
from kernels.model_ops import add_rmsnorm, silu_mul
from kernels.rope import rope_kv_write


@dataclass(frozen=True)
class QwenConfig:
    hidden_size: int = 1536
    num_layers: int = 28
    num_heads: int = 12
    num_kv_heads: int = 2
    head_dim: int = 128
    intermediate_size: int = 8960
    vocab_size: int = 151936
    rms_norm_eps: float = 1e-6
    rope_theta: float = 1_000_000.0


QWEN25_1P5B = QwenConfig()  # model.py:18-27


class RMSNorm(nn.Module):
    """Normalise in fp32, scale in the input dtype (model.py:49-55)."""

    def __init__(self, dim, eps):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(dim))
        self.eps = eps

    def forward(self, x):
        if x.is_cuda:
            shape = x.shape
            return add_rmsnorm(x.reshape(-1, shape[-1]), self.weight, self.eps)[1].view(shape)
        dtype = x.dtype
        xf = x.float()
        xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + self.eps)
        return self.weight * xf.to(dtype)


def rotate_half(x):
    x1, x2 = x.chunk(2, dim=-1)
    return torch.cat((-x2, x1), dim=-1)


def apply_rope(q, k, cos, sin):
    return q * cos + rotate_half(q) * sin, k * cos + rotate_half(k) * sin


def transposed(weight):
    """weight.t().contiguous(), cached on the parameter and rebuilt when it is modified."""
    cached = getattr(weight, "_mi_transposed", None)
    if cached is None or cached[0] != weight._version:
        cached = (weight._version, weight.detach().t().contiguous())
        weight._mi_transposed = cached
    return cached[1]


def plain(*modules):
    """Whether the modules are exactly these classes with nothing hooked on and no forward of their
    own, so that a kernel may do their work without calling them."""
    if nn.modules.module._has_any_global_hook():
        return False
    for m in modules:
        d = vars(m)
        if (type(m) not in _PLAIN or "forward" in d or d["_forward_hooks"] or d["_forward_pre_hooks"]
                or d["_backward_hooks"] or d["_backward_pre_hooks"]):
            return False
    return True


def inference(*tensors):
    """Whether nothing would record a gradient, cast the inputs or follow the torch operations (forward
    mode, vmap and other function transforms, tracers, dispatch modes): the fused kernels, launched
    outside torch, would be missing there."""
    return (not (torch.is_grad_enabled() and any(t.requires_grad for t in tensors))
            and not torch.is_autocast_enabled("cuda")
            and forward_ad._current_level < 0 and not torch._C._are_functorch_transforms_active()
            and not torch._C._len_torch_dispatch_stack() and torch._C._get_tracing_state() is None
            and not torch.compiler.is_compiling())


def repeat_kv(x, n_rep):
    if n_rep == 1:
        return x
    b, h, s, d = x.shape
    return x[:, :, None].expand(b, h, n_rep, s, d).reshape(b, h * n_rep, s, d)


def sdpa_fallback(q, k, v, starts, n_rep):
    """The reference's CPU attention: fp32 SDPA over repeat_kv-expanded K/V (model.py:104-107)
    with its mask choice (model.py:181-195).  q [B, Hq, T, d], k/v [B, Hkv, S, d] dense (every row
    padded to S keys); starts[b]: tokens row b held before this step.  When every row starts at
    the same place no mask is built: a fresh prefill (start 0) is SDPA's is_causal, whose top-left
    alignment equals the bottom-right one when T == S, and a one-token step sees every key.
    Otherwise the explicit [B, 1, T, S] bottom-right mask: query i of row b sees key j iff
    j <= starts[b] + i."""
    T, S = q.shape[2], k.shape[2]
    k, v = repeat_kv(k, n_rep), repeat_kv(v, n_rep)
    c0 = starts[0]
    if all(st == c0 for st in starts) and (T == 1 or c0 == 0):
        return F.scaled_dot_product_attention(q, k, v, is_causal=c0 == 0)
    key_pos = torch.arange(S, device=q.device)
    q_pos = (torch.tensor(starts, device=q.device)[:, None]
             + torch.arange(T, device=q.device)[None, :])
    mask = (key_pos[None, None, :] <= q_pos[:, :, None]).unsqueeze(1)
    return F.scaled_dot_product_attention(q, k, v, attn_mask=mask)


class Attention(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.cfg = cfg
        self.q_size = cfg.num_heads * cfg.head_dim
        self.kv_size = cfg.num_kv_heads * cfg.head_dim
        self.qkv_proj = nn.Linear(cfg.hidden_size, self.q_size + 2 * self.kv_size, bias=True)
        self.o_proj = nn.Linear(self.q_size, cfg.hidden_size, bias=False)

    def forward(self, x, cos, sin, cache, layer, meta):
        cfg = self.cfg
        B, T, _ = x.shape
        qkv = self.qkv_proj(x)
        if x.is_cuda:
            # rotated q out, rotated k and v into their cache slots, in one launch
            q = rope_kv_write(qkv.view(B * T, -1), cos[:, 0].reshape(B * T, cfg.head_dim),
                              sin[:, 0].reshape(B * T, cfg.head_dim), meta.slot_mapping32,
                              cache.k_pool(layer), cache.v_pool(layer), cfg.num_heads,
                              cfg.num_kv_heads)
            return self.o_proj(self._attend(q, B, T, cache, layer, meta))
        else:
            q, k, v = qkv.split([self.q_size, self.kv_size, self.kv_size], dim=-1)
            q = q.view(B, T, cfg.num_heads, cfg.head_dim).transpose(1, 2)
            k = k.view(B, T, cfg.num_kv_heads, cfg.head_dim).transpose(1, 2)
            v = v.view(B, T, cfg.num_kv_heads, cfg.head_dim).transpose(1, 2)
            q, k = apply_rope(q, k, cos, sin)
            cache.write(layer, meta, k, v)
            if meta.packed:
                out = self._attend_packed_cpu(q, cache, layer, meta)
                return self.o_proj(out.transpose(1, 2).reshape(B, T, self.q_size))
            k_all, v_all = cache.read(layer, meta)
            out = sdpa_fallback(q, k_all, v_all, meta.starts, cfg.num_heads // cfg.num_kv_heads)
        return self.o_proj(out.transpose(1, 2).reshape(B, T, self.q_size))

    def _attend(self, q, B, T, cache, layer, meta):
        """Attention of the rotated queries q [B * T, Hq * d] over the cache -> [B, T, Hq * d]."""
        cfg = self.cfg
        if meta.packed:
            out = self._attend_packed(q.view(B * T, cfg.num_heads, cfg.head_dim), cache, layer, meta)
            return out.view(B, T, self.q_size)
        q = q.view(B, T, cfg.num_heads, cfg.head_dim).transpose(1, 2)
        out = fa2_paged(q, cache.k_pool(layer), cache.v_pool(layer), meta.block_table,
                        meta.kv_lens, block_size=cache.block_size, max_kv_len=meta.max_kv,
                        is_causal=T > 1)
        return out.transpose(1, 2).reshape(B, T, self.q_size)

    def few_rows_fit(self, x, norm):
        """Whether few_rows_step takes x [tokens, hidden]."""
        qkv, o = self.qkv_proj, self.o_proj
        return (plain(self, norm, qkv, o) and self.cfg.head_dim == few_rows.HEAD_DIM
                and few_rows.linear_fits(x, qkv.weight, norm.weight)
                and qkv.weight.shape[0] == self.q_size + 2 * self.kv_size
                and few_rows.bias_fits(qkv.bias, x, qkv.weight.shape[0])
                and few_rows.weight_fits(o.weight, x, x.shape[1])
                and o.weight.shape[1] == self.q_size and o.bias is None)

    def few_rows_step(self, res, norm, shape, cos, sin, cache, layer, meta):
        """res [tokens, hidden] += attention of norm(res), in three launches and attention's own."""
        cfg = self.cfg
        (B, T, _), n = shape, res.shape[0]
        q = few_rows.qkv_rope(res, norm.weight, cfg.rms_norm_eps, self.qkv_proj.weight, self.qkv_proj.bias,
                              cos[:, 0].reshape(n, cfg.head_dim), sin[:, 0].reshape(n, cfg.head_dim),
                              meta.slot_mapping32, cache.k_pool(layer), cache.v_pool(layer),
                              cfg.num_heads, cfg.num_kv_heads)
        a = self._attend(q, B, T, cache, layer, meta).view(n, self.q_size)
        few_rows.linear(a, self.o_proj.weight, residual=res, out=res)

    def _attend_packed(self, q, cache, layer, meta):
        """q [N, Hq, d] packed queries of a mixed step -> [N, Hq, d]: the leading one-token rows
        through the paged decode kernel, the rest through the paged varlen prefill kernel, both
        writing into one packed output."""
        out = torch.empty_like(q)
        D, B, bs = meta.n_single, len(meta.counts), cache.block_size
        kv_single, kv_multi, q_multi = meta.split()
        kp, vp = cache.k_pool(layer), cache.v_pool(layer)
        if D:
            fa2_paged(q[:D].unsqueeze(2), kp, vp, meta.block_table[:D], meta.kv_lens[:D],
                      block_size=bs, max_kv_len=kv_single, is_causal=False,
                      out=out[:D].unsqueeze(2))
        if D < B:
            fa2_paged_varlen(q, kp, vp, meta.cu_q[D:], meta.block_table[D:], meta.kv_lens[D:],
                             q_multi, block_size=bs, max_kv_len=kv_multi, is_causal=True, out=out)
        return out

    def _attend_packed_cpu(self, q, cache, layer, meta):
        """The dense fallback row by row: q [1, Hq, N, d] -> [1, Hq, N, d] (model.py:181-195)."""
        n_rep = self.cfg.num_heads // self.cfg.num_kv_heads
        outs, c0 = [], 0
        for start, count, table in zip(meta.starts, meta.counts, meta.tables):
            k_all, v_all = cache.read_row(layer, table, start + count)
            mask = (torch.arange(start + count, device=q.device)[None, :]
                    <= start + torch.arange(count, device=q.device)[:, None])
            outs.append(F.scaled_dot_product_attention(
                q[:, :, c0:c0 + count], repeat_kv(k_all[None], n_rep), repeat_kv(v_all[None], n_rep),
                attn_mask=mask))
            c0 += count
        return torch.cat(outs, dim=2)


class MLP(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.inter = cfg.intermediate_size
        self.gate_up_proj = nn.Linear(cfg.hidden_size, 2 * cfg.intermediate_size, bias=False)
        self.down_proj = nn.Linear(cfg.intermediate_size, cfg.hidden_size, bias=False)

    def forward(self, x):
        if x.is_cuda:
            rows = x.reshape(-1, x.shape[-1])
            if few_rows.mlp_pays(*rows.shape) and self.few_rows_fit(rows):
                return few_rows.mlp(rows, self.gate_up_proj.weight,
                                    self.down_proj.weight).view(x.shape)
            gu = rows @ transposed(self.gate_up_proj.weight)
            act = silu_mul(gu).view(*x.shape[:-1], self.inter)
            return self.down_proj(act)
        gu = self.gate_up_proj(x)
        gate, up = gu.split(self.inter, dim=-1)
        return self.down_proj(F.silu(gate) * up)

    def few_rows_fit(self, x, norm=None):
        """Whether few_rows.mlp does this module's work on x [tokens, hidden] (after `norm`)."""
        gu, down = self.gate_up_proj, self.down_proj
        if not plain(gu, down, *((self, norm) if norm is not None else ())):
            return False
        gw, dw = gu.weight, down.weight
        return (gu.bias is None and down.bias is None and inference(x, gw, dw)
                and few_rows.mlp_fits(x, gw, dw, norm.weight if norm is not None else None))


class Block(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.self_attn = Attention(cfg)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.mlp = MLP(cfg)

    def forward(self, x, cos, sin, cache, layer, meta):
        x = x + self.self_attn(self.input_layernorm(x), cos, sin, cache, layer, meta)
        return x + self.mlp(self.post_attention_layernorm(x))


_PLAIN = (nn.Linear, RMSNorm, Attention, MLP, Block)   # what plain() knows


class Qwen2ForCausalLM(nn.Module):
    def __init__(self, cfg=QWEN25_1P5B):
        super().__init__()
        self.cfg = cfg
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(Block(cfg) for _ in range(cfg.num_layers))
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        inv_freq = 1.0 / (cfg.rope_theta ** (torch.arange(0, cfg.head_dim, 2).float() / cfg.head_dim))
        self.register_buffer("inv_freq", inv_freq, persistent=False)

    @torch.no_grad()
    def init_random(self, std=0.02, seed=0):
        """Random weights: N(0, std) for every matrix and bias, ones for the norms."""
        g = torch.Generator(device=self.embed_tokens.weight.device).manual_seed(seed)
        for name, prm in self.named_parameters():
            if name.endswith("layernorm.weight") or name == "norm.weight":
                prm.fill_(1.0)
            else:
                prm.copy_(torch.randn(prm.shape, generator=g, device=prm.device,
                                      dtype=torch.float32).mul_(std).to(prm.dtype))
        return self

    def rope_cos_sin(self, position_ids, dtype):
        # position_ids [B, T] -> cos/sin [B, 1, T, head_dim] (model.py:151-155)
        freqs = position_ids.float()[..., None] * self.inv_freq[None, None, :]
        emb = torch.cat((freqs, freqs), dim=-1)
        return emb.cos()[:, None].to(dtype), emb.sin()[:, None].to(dtype)

    def forward(self, input_ids, cache, seqs):
        """input_ids [B, T] appended to cache sequences `seqs`; returns last-position logits
        [B, 1, vocab] (model.py:157-207)."""
        _, T = input_ids.shape
        meta = cache.prepare(seqs, T)
        logits = self.forward_meta(input_ids, cache, meta)
        cache.advance(seqs, T)
        return logits

    def forward_meta(self, input_ids, cache, meta):
        """The layers over an already prepared step: what a captured decode graph replays, its
        metadata living in static device buffers."""
        _, T = input_ids.shape
        x = self.embed_tokens(input_ids)
        f, starts = self.inv_freq, meta.starts_dev
        if (x.is_cuda and self._own("rope_cos_sin") and f.dtype == x.dtype and x.dtype in (torch.bfloat16, torch.float16)
                and f.shape == (few_rows.HEAD_DIM // 2,) and f.is_contiguous()
                and f.device == starts.device and starts.dtype == torch.int32
                and starts.is_contiguous()):
            cos, sin = few_rows.rope_tables(starts, T, f)
        else:
            position_ids = starts[:, None] + torch.arange(T, device=x.device)[None, :]
            cos, sin = self.rope_cos_sin(position_ids, x.dtype)
        x = self.run_layers(x, cos, sin, cache, meta)
        x, w = x[:, -1:], self.embed_tokens.weight
        rows = x.reshape(-1, x.shape[-1])
        if (x.is_cuda and rows.shape[0] <= few_rows.MAX_NORM_ROWS and plain(self.norm)
                and inference(x, w, self.norm.weight)
                and self._own("lm_head") and few_rows.linear_fits(rows, w, self.norm.weight)):
            return few_rows.linear(rows, w, norm_weight=self.norm.weight,
                                   eps=self.norm.eps).view(*x.shape[:-1], w.shape[0])
        return self.lm_head(self.norm(x))

    def _own(self, name):
        """Whether method `name` is this class's, replaced neither in a subclass nor on the instance."""
        return getattr(self, name) == getattr(Qwen2ForCausalLM, name).__get__(self)

    def lm_head(self, x):
        """Tied-embedding logits (model.py:204-207)."""
        w = self.embed_tokens.weight
        if x.is_cuda:
            rows = x.reshape(-1, x.shape[-1])
            if (few_rows.linear_pays(rows.shape[0], w) and inference(x, w)
                    and few_rows.linear_fits(rows, w)):
                return few_rows.linear(rows, w).view(*x.shape[:-1], w.shape[0])
            return x @ transposed(w)
        return x @ w.T

    def run_layers(self, x, cos, sin, cache, meta):
        """The decoder layers over x [B, T, hidden].  On the GPU each residual add is fused with the
        RMSNorm that follows it (the first layer's input norm has no add; the last layer's MLP
        output is added alone), which is the same arithmetic as Block.forward layer by layer."""
        if not x.is_cuda:
            for layer_idx, layer in enumerate(self.layers):
                x = layer(x, cos, sin, cache, layer_idx, meta)
            return x
        shape, H, eps = x.shape, x.shape[-1], self.cfg.rms_norm_eps
        res = x.reshape(-1, H)
        if self._few_rows_fit(res):
            for i, layer in enumerate(self.layers):
                layer.self_attn.few_rows_step(res, layer.input_layernorm, shape, cos, sin, cache, i,
                                              meta)
                norm, mlp = layer.post_attention_layernorm, layer.mlp
                few_rows.mlp(res, mlp.gate_up_proj.weight, mlp.down_proj.weight, residual=res,
                             norm_weight=norm.weight, eps=eps, out=res)
            return res.view(shape)
        _, h = add_rmsnorm(res, self.layers[0].input_layernorm.weight, eps)
        for i, layer in enumerate(self.layers):
            a = layer.self_attn(h.view(shape), cos, sin, cache, i, meta).reshape(-1, H)
            res, h = add_rmsnorm(res, layer.post_attention_layernorm.weight, eps, y=a,
                                 residual_out=res)
            m = layer.mlp(h.view(shape)).reshape(-1, H)
            if i + 1 < len(self.layers):
                res, h = add_rmsnorm(res, self.layers[i + 1].input_layernorm.weight, eps, y=m,
                                     residual_out=res)
            else:
                res = res + m
        return res.view(shape)

    def _few_rows_fit(self, res):
        """Whether every layer of a step over res [tokens, hidden] runs on the few-row kernels."""
        return (1 <= res.shape[0] <= few_rows.MAX_NORM_ROWS
                and inference(res, *(self.parameters() if torch.is_grad_enabled() else ()))
                and all(layer.self_attn.few_rows_fit(res, layer.input_layernorm)
                        and layer.mlp.few_rows_fit(res, layer.post_attention_layernorm)
                        for layer in self.layers))

    def forward_mixed(self, rows, cache, seqs):
        """One packed step: rows[b] (a list of token ids, at least one) is appended to cache
        sequence seqs[b].  Returns each row's last-token logits [B, vocab]."""
        counts = [len(r) for r in rows]
        meta = cache.prepare_packed(seqs, counts)
        ids = torch.tensor([t for r in rows for t in r], dtype=torch.long)
        if cache.device.type == "cuda":
            ids = ids.pin_memory().to(cache.device, non_blocking=True)
        logits = self.forward_packed(ids, cache, meta)
        cache.advance(seqs, counts)
        return logits

    def forward_packed(self, token_ids, cache, meta):
        """The layers over a prepared mixed step (KVCache.prepare_packed): token_ids [N] are the
        rows' new tokens back to back; returns the rows' last-token logits [B, vocab]."""
        x = self.embed_tokens(token_ids)[None]                      # [1, N, hidden]
        cos, sin = self.rope_cos_sin(meta.positions[None], x.dtype)
        x = self.run_layers(x, cos, sin, cache, meta)
        x = self.norm(x[0, meta.last_idx.long()])
        return self.lm_head(x)
