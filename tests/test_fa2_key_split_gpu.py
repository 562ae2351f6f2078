"""The prefill launches whose keys are cut into pieces (few queries over many keys): against the fp32
oracle and against the same call without a workspace, which runs unsplit.

The two round the weights P to 16 bits against different running maxima, each by at most half a unit
(2^-8 of the weight in bf16, 2^-11 in fp16), so the weights of a query differ by at most twice that in
all: 2^-7 (2^-10) of the mean |v| they weigh, about that of the output or of 1, and the log-sum-exps
by as much."""
import math

import pytest
import torch

from conftest import announce
from kernels import _lib
from kernels.fa2 import fa2_forward, fa2_paged
from oracle import sdpa

pytestmark = pytest.mark.gpu
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


def ws_bytes(B, Hq, Hkv, T, S):
    return _lib.load().mi_fa2_fwd_workspace_size(B, Hq, Hkv, T, S, 128)


def unsplit(q, k, v, causal, lens):
    """mi_fa2_fwd without a workspace."""
    (B, Hq, T, d), (Hkv, S) = q.shape, k.shape[1:3]
    o = torch.full_like(q, float("nan"), memory_format=torch.contiguous_format)
    lse = torch.full((B, Hq, T), float("nan"), device=q.device)
    _lib.check(_lib.load().mi_fa2_fwd(
        _lib.DTYPES[q.dtype], q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
        lse.data_ptr(), lens.data_ptr(), B, Hq, Hkv, T, S, d, _lib.strides(q), _lib.strides(k),
        _lib.strides(v), _lib.strides(o), _lib.strides(lse), int(causal), 1 / math.sqrt(d), None, 0,
        _lib.stream_of(q)))
    return o, lse


def check(got, got_lse, want, want_lse, ref):
    u = ULP[got.dtype]
    assert torch.isfinite(got).all()
    assert ((got.float() - want.float()).abs() <= u * want.float().abs().clamp_min(1)).all()
    assert torch.equal(torch.isinf(got_lse), torch.isinf(want_lse))
    seen = ~torch.isinf(want_lse)
    assert ((got_lse - want_lse).abs()[seen] <= u).all()
    err = (got.float().cpu() - ref).abs()
    assert err.max().item() < 1e-2 and err.mean().item() < 1e-3, err.max().item()


# queries: one, of more heads per kv head than the decode takes, two, a ragged last tile, exactly one
# tile of packed rows, several tiles; keys: a few steps, a ragged last one, rows shorter than the
# batch's longest, than their queries, and empty
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("T,heads,lens", [
    (2, (12, 2), [3001]), (150, (12, 2), [3001]), (64, (4, 2), [1153, 40, 0]),
    (128, (1, 1), [8000]), (700, (2, 2), [2048]), (37, (8, 8), [5000, 4999]),
    (33, (17, 1), [1200]), (1, (17, 1), [3001]), (1, (40, 2), [2500, 130, 0])])
def test_padded(T, heads, lens, causal, dtype):
    Hq, Hkv = heads
    B, S = len(lens), max(lens)
    assert ws_bytes(B, Hq, Hkv, T, S) > 0
    g = torch.Generator().manual_seed(T + S)
    q = torch.randn(B, T, Hq, 128, generator=g).to(dtype).transpose(1, 2)   # strided heads
    k, v = (torch.randn(B, Hkv, S, 128, generator=g).to(dtype) for _ in range(2))
    for b, n in enumerate(lens):   # padding must not reach the output
        k[b, :, n:] = float("nan")
        v[b, :, n:] = float("inf")
    announce(f"[gpu] split padded T={T} heads={heads} lens={lens} causal={causal} {dtype}")
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    ln = torch.tensor(lens, dtype=torch.int32, device="cuda")
    got, got_lse = fa2_forward(qd, kd, vd, causal, ln, return_lse=True)
    want, want_lse = unsplit(qd, kd, vd, causal, ln)
    torch.cuda.synchronize()
    check(got, got_lse, want, want_lse, sdpa.attention_ref(q, k, v, causal, lens))


@pytest.mark.parametrize("T", [5, 64, 150])
def test_infinite_values_stay_infinite(T):
    """An inf in a V row every query sees (an overflow in fp16, say) is an inf of its column, whichever
    piece holds it."""
    S, cols = 3001, range(0, 3001, 100)
    assert ws_bytes(1, 12, 2, T, S) > 0
    g = torch.Generator().manual_seed(T)
    q = torch.randn(1, 12, T, 128, generator=g).half()
    k, v = (torch.randn(1, 2, S, 128, generator=g).half() for _ in range(2))
    for i, key in enumerate(cols):
        v[0, :, key, i] = float("inf")
    announce(f"[gpu] split with infinite values T={T}")
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    ln = torch.tensor([S], dtype=torch.int32, device="cuda")
    got, _ = fa2_forward(qd, kd, vd, False, ln, return_lse=True)
    want, _ = unsplit(qd, kd, vd, False, ln)
    torch.cuda.synchronize()
    assert torch.isinf(want[..., :len(cols)]).all() and torch.isfinite(want[..., len(cols):]).all()
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and not torch.isnan(got).any()


@pytest.mark.parametrize("T,lens,block", [(150, [3001], 16), (5, [7777], 16), (90, [2000, 1999], 32),
                                          (60, [4100, 300], 512), (3, [1300, 2], 128)])
def test_paged(T, lens, block):
    B, Hq, Hkv = len(lens), 12, 2
    assert ws_bytes(B, Hq, Hkv, T, max(lens)) > 0
    need = [-(-n // block) for n in lens]
    g = torch.Generator().manual_seed(T + max(lens))
    table = torch.zeros(B, max(need), dtype=torch.int32)
    perm = torch.randperm(sum(need) + 3, generator=g).int()
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[at:at + n]
        at += n
    kp, vp = (torch.randn((sum(need) + 3) * block, Hkv, 128, generator=g).bfloat16() for _ in range(2))
    q = torch.randn(B, Hq, T, 128, generator=g).bfloat16()
    S = max(lens)
    k, v = torch.zeros(B, Hkv, S, 128).bfloat16(), torch.zeros(B, Hkv, S, 128).bfloat16()
    for b, n in enumerate(lens):
        slots = (table[b].long()[:, None] * block + torch.arange(block)).reshape(-1)[:n]
        k[b, :, :n], v[b, :, :n] = kp[slots].transpose(0, 1), vp[slots].transpose(0, 1)
    announce(f"[gpu] split paged T={T} lens={lens} block={block}")
    ln = torch.tensor(lens, dtype=torch.int32, device="cuda")
    got, got_lse = fa2_paged(q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ln, block_size=block,
                             max_kv_len=S, is_causal=True, return_lse=True)
    want, want_lse = unsplit(q.cuda(), k.cuda(), v.cuda(), True, ln)
    torch.cuda.synchronize()
    check(got, got_lse, want, want_lse, sdpa.attention_ref(q, k, v, True, lens))


def test_paged_plans_are_looked_up_by_value():
    """fa2_paged's checked launch arguments are kept per combination of shapes, strides, types and plain
    values: a bound held in a tensor counts by its value at each call, and `out` by its own strides."""
    g = torch.Generator().manual_seed(1)
    kp, vp = (torch.randn(64 * 16, 2, 128, generator=g).bfloat16().cuda() for _ in range(2))
    q = torch.randn(2, 12, 1, 128, generator=g).bfloat16().cuda()
    table = torch.randperm(64, generator=g).int().view(2, 32).cuda()
    lens = torch.tensor([500, 300], dtype=torch.int32, device="cuda")
    want = [fa2_paged(q, kp, vp, table, lens, max_kv_len=n) for n in (512, 128)]
    bound = torch.tensor(512)
    assert torch.equal(fa2_paged(q, kp, vp, table, lens, max_kv_len=bound), want[0])
    bound.fill_(128)   # lengths are clamped to it
    assert torch.equal(fa2_paged(q, kp, vp, table, lens, max_kv_len=bound), want[1])
    wide = torch.zeros(2, 12, 1, 256, dtype=torch.bfloat16, device="cuda")
    out = wide[..., 128:]
    assert fa2_paged(q, kp, vp, table, lens, max_kv_len=512, out=out).data_ptr() == out.data_ptr()
    assert torch.equal(out, want[0]) and (wide[..., :128] == 0).all()
    with pytest.raises(AssertionError):
        fa2_paged(q, kp, vp, table, lens, max_kv_len=513)
    with pytest.raises(AssertionError):
        fa2_paged(q, kp, vp, table, lens.long())
