"""The prefill kernel for head dims 32, 64 and 256 (csrc/fa2_prefill_dims.hip), at shapes the
dispatch gives it, against the fp32 oracle; tolerances as for every 16-bit output of the general
envelope (tests/test_fa2_general_gpu.py)."""
import math

import pytest
import torch

from conftest import announce
from kernels import _lib
from kernels.fa2 import FlashAttention2Function, fa2_forward
from general_rule import DIMS, DIMS_SMALL, on_this_device
from oracle import sdpa
from test_fa2_general_gpu import check_close, rand

pytestmark = pytest.mark.gpu
DTYPES = pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])


# T, S, heads, kv_lens: a last tile of one row, of 127 and of 128; keys one past, one short of and at a
# tile; rows with fewer keys than queries, one key and none; more heads than XCDs, one kv head; one step
# of keys and many.  128-row work-groups at d = 64 and 256; at d = 32 64-row ones but for two shapes.
SHAPES = [(257, 257, (12, 2), [257, 256, 1, 0, 129]), (383, 383, (12, 6), [383, 300, 129, 65]),
          (384, 640, (20, 1), [640, 641 - 257, 100]), (130, 320, (16, 2), [320, 319, 64, 63] * 2),
          (200, 100, (12, 2), [100] * 16), (1025, 1100, (12, 2), [1100, 900]),
          (513, 513, (12, 4), [513, 512, 449, 100]), (1000, 1000, (12, 2), [1000, 999, 513, 100])]
# 64-row work-groups (d <= 64)
SMALL = [(1000, 1000, (12, 2), [1000]), (700, 1300, (6, 6), [1300, 1]), (513, 2000, (12, 1), [1025])]
CASES = ([(d, *shape, DIMS_SMALL if d == 32 and shape[0] not in (200, 1000) else DIMS)
          for d in (32, 64, 256) for shape in SHAPES]
         + [(d, *shape, DIMS_SMALL) for d in (32, 64) for shape in SMALL])


@DTYPES
@pytest.mark.parametrize("causal", [True, False], ids=["causal", "full"])
@pytest.mark.parametrize("d,T,S,heads,lens,which", CASES)
def test_against_the_oracle(d, T, S, heads, lens, which, causal, dtype):
    Hq, Hkv = heads
    B = len(lens)
    assert on_this_device(B, Hq, Hkv, T, S, d) == which
    g = torch.Generator().manual_seed(T + S + d)
    q = torch.randn(B, T, Hq, d, generator=g).to(dtype).transpose(1, 2)   # strided heads
    k, v = rand((B, Hkv, S, d), g, dtype), rand((B, Hkv, S, d), g, dtype)
    for b, n in enumerate(lens):   # padding is never read
        k[b, :, n:] = float("nan")
        v[b, :, n:] = float("inf")
    announce(f"[gpu] prefill dims: d={d} T={T} S={S} heads={heads} causal={causal} {dtype}")
    out, lse = fa2_forward(q.cuda(), k.cuda(), v.cuda(), causal,
                           torch.tensor(lens, dtype=torch.int32, device="cuda"), return_lse=True)
    torch.cuda.synchronize()
    check_close(out, sdpa.attention_ref(q, k, v, causal, lens), dtype, f"d={d}")
    want = sdpa.lse_ref(q, k.nan_to_num(0.), causal, lens)
    fin = torch.isfinite(want)
    assert torch.equal(fin, torch.isfinite(lse.cpu()))
    # the row sum adds P as rounded for the PV product (unit roundoff 2^-8 at most)
    assert (lse.cpu()[fin] - want[fin]).abs().max().item() < math.log1p(2.0 ** -8) + 1e-3


def test_large_scores_move_the_running_maximum():
    # every key's score is 8 above the one before (11.5 in the exponent; past 256, where bf16 holds even
    # numbers, every second one's is 16 above): each tile moves the maximum, and
    # what earlier tiles summed is scaled away
    assert on_this_device(4, 12, 2, 300, 300, 64) == DIMS
    g = torch.Generator().manual_seed(3)
    q = torch.ones(4, 12, 300, 64).bfloat16()
    k = (torch.arange(300).view(1, 1, 300, 1) * torch.ones(4, 2, 300, 64)).bfloat16()
    v = rand((4, 2, 300, 64), g, torch.bfloat16)
    out = FlashAttention2Function.apply(q.cuda(), k.cuda(), v.cuda(), True, None)
    # every output is about one V value, so its rounding to bf16 is not small beside the bars: half a
    # unit is 2^-8 of the value at most and 2^-9 on average
    ref = sdpa.attention_ref(q, k, v, True)
    err = (out.float().cpu() - ref).abs()
    assert (err <= 1e-2 + 2.0 ** -8 * ref.abs()).all()
    assert err.mean().item() < 1e-3 + 2.0 ** -9 * ref.abs().mean().item()


def test_overlapping_key_rows_stay_accepted():
    # a K whose token stride is 0 (one key expanded) is read by the general kernel, as before
    q = torch.randn(4, 12, 300, 64, generator=torch.Generator().manual_seed(5)).bfloat16()
    k = torch.randn(4, 2, 1, 64).bfloat16().cuda().expand(4, 2, 300, 64)
    v = torch.randn(4, 2, 300, 64, generator=torch.Generator().manual_seed(6)).bfloat16()
    out = FlashAttention2Function.apply(q.cuda(), k, v.cuda(), True, None)
    check_close(out, sdpa.attention_ref(q, k.cpu(), v, True), torch.bfloat16, "stride 0")


@pytest.mark.parametrize("d", [32, 64, 256])
@pytest.mark.parametrize("B,T", [(1, 1000), (4, 1000)])
@pytest.mark.parametrize("scale", [-0.125, 0.0])
def test_scales_that_are_not_positive(scale, B, T, d):
    """Negative: the smallest score weighs most; zero: the mean of the visible values."""
    g = torch.Generator().manual_seed(d + T)
    q, k, v = (torch.randn(B, n, T, d, generator=g).bfloat16().cuda() for n in (12, 2, 2))
    o = torch.full_like(q, float("nan"))
    announce(f"[gpu] general entry point, scale {scale}, {B} x {T} x {d}")
    _lib.check(_lib.load().mi_fa2_fwd_general(
        0, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), None, None, B, 12, 2, T, T, d, d,
        *(_lib.strides(t) for t in (q, k, v, o)), None, 1, scale, _lib.stream_of(q)))
    qs = q.float().cpu() * (scale * math.sqrt(d))   # the oracle scales by 1 / sqrt(d)
    check_close(o, sdpa.attention_ref(qs, k.float().cpu(), v.float().cpu(), True), torch.bfloat16, "scale")


@DTYPES
@pytest.mark.parametrize("d", [32, 64, 256])
@pytest.mark.parametrize("B,T", [(1, 1000), (4, 1000)])
@pytest.mark.parametrize("size", [2.0 ** 9, 2.0 ** 15])
def test_scores_past_the_reach_of_the_exponents_fraction(size, B, T, d, dtype):
    """Scores of 2^20 to 2^38, whose rounding alone is more than an exponent holds: each query's largest
    one has all the weight."""
    g = torch.Generator().manual_seed(d)
    q, k, v = (torch.randn(B, n, T, d, generator=g) for n in (12, 2, 2))
    q, k, v = (q.sign() * size).to(dtype), (k.sign() * size).to(dtype), v.to(dtype)
    # scores are whole multiples of size^2: a query's largest stands out by at least 2 of them, or is
    # shared by keys that weigh the same
    announce(f"[gpu] prefill dims: scores of {size}^2, {B} x {T} x {d} {dtype}")
    out = FlashAttention2Function.apply(q.cuda(), k.cuda(), v.cuda(), False, None)
    torch.cuda.synchronize()
    check_close(out, sdpa.attention_ref(q, k, v, False), dtype, "large scores")
