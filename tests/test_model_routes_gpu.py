"""When the model's few-token kernels may do its modules' and methods' work without calling them."""
import pytest
import torch

from conftest import announce
from kernels import few_rows
from kv_cache import KVCache
from model import QwenConfig, Qwen2ForCausalLM

pytestmark = pytest.mark.gpu
CFG = QwenConfig(hidden_size=256, num_layers=2, num_heads=2, num_kv_heads=1, intermediate_size=512,
                 vocab_size=512)


def make(cfg=CFG):
    return (Qwen2ForCausalLM(cfg).cuda().init_random(std=0.05, seed=0).to(torch.bfloat16).eval()
            .requires_grad_(False))


def decode(model, steps=3, rows=3):
    """Logits of a prompt of 40 tokens and of `steps` single-token steps."""
    cache = KVCache(32, 16, "cuda", next(model.parameters()).dtype, CFG.num_layers, CFG.num_kv_heads,
                    CFG.head_dim)
    seqs = [cache.alloc() for _ in range(rows)]
    g = torch.Generator().manual_seed(1)
    outs = [model(torch.randint(0, CFG.vocab_size, (rows, 40), generator=g).cuda(), cache, seqs)]
    for _ in range(steps):
        outs.append(model(torch.randint(0, CFG.vocab_size, (rows, 1), generator=g).cuda(), cache, seqs))
    return torch.cat(outs, 1)


def close(got, want):
    """The same logits from kernels that sum in another order: a few bf16 roundings apart, which two
    layers carry on."""
    assert torch.isfinite(got).all()
    assert (got - want).abs().max().item() < 0.05 * want.abs().max().item()


def override(model, name, change, on_class):
    """Replace method `name` by one that changes its result; returns the list of its calls."""
    calls, old = [], getattr(type(model), name)

    def new(self, *args):
        calls.append(name)
        return change(old(self, *args))
    if on_class:
        model.__class__ = type("Other", (type(model),), {name: new})
    else:
        setattr(model, name, new.__get__(model))
    return calls


@pytest.mark.parametrize("on_class", [True, False], ids=["subclass", "instance"])
@pytest.mark.parametrize("name,change", [
    ("rope_cos_sin", lambda cs: (cs[0] * 0.5, cs[1] * 0.5)), ("lm_head", lambda y: y + 1)])
def test_overridden_methods_are_called(name, change, on_class):
    announce(f"[gpu] model with its own {name}")
    model = make()
    plain = decode(model)
    calls = override(model, name, change, on_class)
    got = decode(model)
    assert len(calls) == 4   # the prompt's step and the three decode steps
    assert not torch.equal(got, plain)
    if name == "lm_head":
        # logits of about 1: two roundings, before and after the 1 is added, and of the product
        assert (got - 1 - plain).abs().max().item() < 4 * 2.0 ** -8 * plain.abs().max().item() + 2.0 ** -7


def relayout(p, kind):
    """p's values off a 16-byte boundary, as in one flat buffer of parameters, or with a stride."""
    if kind == "offset":
        flat = torch.zeros(p.numel() + 1, dtype=p.dtype, device=p.device)
        flat[1:] = p.detach().flatten()
        return flat[1:].view(p.shape)
    wide = torch.zeros(p.numel(), 2, dtype=p.dtype, device=p.device)
    wide[:, 0] = p.detach().flatten()
    return wide[:, 0]


@pytest.mark.parametrize("kind", ["offset", "strided"])
def test_a_bias_the_kernel_cannot_read_goes_through_the_library(kind):
    announce(f"[gpu] q/k/v bias {kind}")
    model = make()
    plain = decode(model)
    for layer in model.layers:
        qkv = layer.self_attn.qkv_proj
        qkv.bias = torch.nn.Parameter(relayout(qkv.bias, kind), requires_grad=False)
        x = torch.zeros(3, CFG.hidden_size, dtype=qkv.weight.dtype, device="cuda")
        assert not layer.self_attn.few_rows_fit(x, layer.input_layernorm)
    close(decode(model), plain)


class Other(torch.Tensor):
    """A tensor subclass, as quantized or distributed weights are."""


def watch(model, how):
    """Put something on layer 0 that the fused kernels would miss; returns its calls, if it has any."""
    layer, calls = model.layers[0], []
    if how in ("o_proj", "mlp", "post_attention_layernorm"):
        m = {"o_proj": layer.self_attn.o_proj, "mlp": layer.mlp,
             "post_attention_layernorm": layer.post_attention_layernorm}[how]
        m.register_forward_hook(lambda *a: calls.append(how))
    elif how == "forward":
        m = layer.mlp.down_proj
        old = m.forward
        m.forward = lambda x: calls.append(how) or old(x)
    elif how == "grad":
        layer.mlp.down_proj.weight.requires_grad_(True)
    elif how == "subclass":
        w = layer.mlp.down_proj.weight
        layer.mlp.down_proj.weight = torch.nn.Parameter(w.detach().as_subclass(Other),
                                                        requires_grad=False)
    return calls


@pytest.mark.parametrize("how", ["o_proj", "mlp", "post_attention_layernorm", "forward", "grad",
                                 "subclass"])
def test_watched_layers_are_called(how):
    announce(f"[gpu] model layers watched by {how}")
    model = make()
    x = torch.zeros(3, CFG.hidden_size, dtype=torch.bfloat16, device="cuda")
    assert model._few_rows_fit(x) and model.layers[0].mlp.few_rows_fit(x)
    with torch.autocast("cuda", torch.float16):
        assert not model._few_rows_fit(x) and not model.layers[0].mlp.few_rows_fit(x)
    plain = decode(model)
    calls = watch(model, how)
    assert not model._few_rows_fit(x)
    got = decode(model)
    # (a norm's module is not called on the GPU: the layer's own launches do its work)
    if how in ("o_proj", "mlp", "forward"):
        assert len(calls) == 4
    close(got, plain)


def test_the_head_follows_torch_where_torch_is_followed(monkeypatch):
    """Forward mode, vmap, a dispatch mode and autocast see the head's product as they would any other."""
    from torch.utils.flop_counter import FlopCounterMode
    H, V = 768, 512
    model = make(cfg=QwenConfig(hidden_size=H, num_layers=1, num_heads=2, num_kv_heads=1,
                                intermediate_size=512, vocab_size=V))
    w = model.embed_tokens.weight
    x, t = (torch.randn(4, 1, H, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    fused, linear = [], few_rows.linear
    monkeypatch.setattr(few_rows, "linear", lambda *a, **k: fused.append(1) or linear(*a, **k))
    announce("[gpu] head under forward mode, vmap, a dispatch mode and autocast")
    with torch.no_grad():
        want = model.lm_head(x)
        assert len(fused) == 1
        close(torch.func.vmap(model.lm_head)(x), want)
        with FlopCounterMode(display=False) as flops:
            close(model.lm_head(x), want)
        assert flops.get_total_flops() == 2 * 4 * H * V
        with torch.autograd.forward_ad.dual_level():
            y = model.lm_head(torch.autograd.forward_ad.make_dual(x, t))
            tangent = torch.autograd.forward_ad.unpack_dual(y).tangent
            assert tangent is not None
            close(tangent, t @ w.T)
        with torch.autocast("cuda", torch.float16):
            assert model.lm_head(x).dtype == torch.float16
    grad = x.clone().requires_grad_(True)
    model.lm_head(grad).sum().backward()
    assert grad.grad is not None
    assert len(fused) == 1   # none of these
