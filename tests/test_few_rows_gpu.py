"""The few-row projections (csrc/linear_rows.hip, through libmi_model.so) against float64 products of
the same values, and against the unfused launches they replace.

Tolerances, with U the largest relative rounding error of the dtype (half a unit: 2^-8 bf16, 2^-11
fp16): the output's own rounding is U of its value; a value rounded on the way to a sum (the product
before the residual add) moves the result by at most one unit, 2U of that value; values rounded before
the product (the normalised x, the activation) may round to the other neighbour where a sum was taken
in another order, each by 2U: over K independent terms that adds at most the same relative error to
the result's rms, and 5 standard deviations of uniform roundings are 3U of it.  The fp32 sums' own
error (K terms, 2^-24 each) is below 1e-4 of the rms."""
import pytest
import torch

from conftest import announce
from kernels import _lib, few_rows
from kernels.model_ops import add_rmsnorm
from kernels.rope import rope_kv_write

pytestmark = pytest.mark.gpu
DTYPES = pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def rand(*shape, dtype, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


def close(got, want, product=None, inner=False):
    """got against want: product, the value rounded before a residual add; inner, whether values were
    rounded before the product."""
    u, want = U[got.dtype], want.double()
    rms = (want if product is None else product).double().pow(2).mean().sqrt()
    bound = u * want.abs() + (1e-4 + 3 * u * inner) * rms
    if product is not None:
        bound = bound + 2 * u * product.double().abs()
    err = (got.double() - want).abs()
    assert torch.isfinite(got).all()
    assert (err <= bound).all(), (err / bound).max().item()


# rows: one, a part of and the whole of each tile of 16, the last; in: one step (most waves idle),
# uneven shares, the engine's, the last; out: fewer tiles than CUs, more
@DTYPES
@pytest.mark.parametrize("rows,n,k", [(1, 16, 32), (16, 1536, 1536), (17, 48, 96), (33, 4112, 544),
                                      (64, 1536, 2048), (5, 8208, 2048), (48, 2048, 1536)])
def test_linear(dtype, rows, n, k):
    announce(f"[gpu] few-row linear {rows}x{n}x{k} {dtype}")
    x, w = rand(rows, k, dtype=dtype, seed=1), rand(n, k, dtype=dtype, seed=2, scale=k ** -0.5)
    bias, res = rand(n, dtype=dtype, seed=3), rand(rows, n, dtype=dtype, seed=4)
    exact = x.double() @ w.double().t()
    close(few_rows.linear(x, w), exact)
    close(few_rows.linear(x, w, bias=bias), exact + bias.double())
    # strided rows in and out, in place on the residual
    wide = rand(rows, k + 40, dtype=dtype, seed=5)
    wide[:, :k] = x
    out = rand(rows, n + 8, dtype=dtype, seed=6)
    out[:, :n] = res
    got = few_rows.linear(wide[:, :k], w, residual=out[:, :n], out=out[:, :n])
    close(got, exact + res.double(), product=exact)
    if rows <= few_rows.MAX_NORM_ROWS:
        nw = (1 + 0.1 * rand(k, dtype=torch.float32, seed=7)).to(dtype)
        normed = add_rmsnorm(x, nw, 1e-6)[1]
        close(few_rows.linear(x, w, norm_weight=nw, eps=1e-6),
              normed.double() @ w.double().t(), inner=True)


@DTYPES
@pytest.mark.parametrize("rows,hidden,inter", [(1, 32, 32), (16, 1536, 8960), (3, 64, 2080),
                                               (17, 1536, 1024), (64, 2048, 4128), (33, 96, 6176)])
def test_mlp(dtype, rows, hidden, inter):
    announce(f"[gpu] few-row mlp {rows}x{hidden}x{inter} {dtype}")
    x = rand(rows, hidden, dtype=dtype, seed=11)
    gu = rand(2 * inter, hidden, dtype=dtype, seed=12, scale=hidden ** -0.5)
    down = rand(hidden, inter, dtype=dtype, seed=13, scale=inter ** -0.5)

    def exact(x):
        g, u = (x.double() @ gu.double().t()).to(dtype).double().chunk(2, -1)
        act = ((g * torch.sigmoid(g)).to(dtype).double() * u).to(dtype)
        return act.double() @ down.double().t()

    want = exact(x)
    got = few_rows.mlp(x, gu, down)
    close(got, want, inner=True)
    # the sums over K's splits are added in one order, whichever work-group is last
    assert torch.equal(got, few_rows.mlp(x, gu, down))
    if rows <= few_rows.MAX_NORM_ROWS:
        nw = (1 + 0.1 * rand(hidden, dtype=torch.float32, seed=14)).to(dtype)
        res = x.clone()
        few_rows.mlp(res, gu, down, residual=res, norm_weight=nw, eps=1e-6, out=res)
        product = exact(add_rmsnorm(x, nw, 1e-6)[1])
        close(res, product + x.double(), product=product, inner=True)


@DTYPES
@pytest.mark.parametrize("rows,hidden,heads", [(1, 1536, (12, 2)), (16, 1536, (12, 2)),
                                               (7, 96, (4, 4)), (13, 2048, (1, 1))])
def test_qkv_rope_matches_the_separate_launches(dtype, rows, hidden, heads):
    announce(f"[gpu] few-row qkv {rows}x{hidden} heads {heads} {dtype}")
    hq, hkv = heads
    n = (hq + 2 * hkv) * 128
    x, w = rand(rows, hidden, dtype=dtype, seed=21), rand(n, hidden, dtype=dtype, seed=22, scale=hidden ** -0.5)
    bias = rand(n, dtype=dtype, seed=23)
    nw = (1 + 0.1 * rand(hidden, dtype=torch.float32, seed=24)).to(dtype)
    ang = torch.rand(rows, 64, generator=torch.Generator().manual_seed(25)).cuda() * 6.28
    cos, sin = (f(torch.cat([ang, ang], -1)).to(dtype) for f in (torch.cos, torch.sin))
    slots = torch.randperm(64, generator=torch.Generator().manual_seed(26))[:rows].int().cuda()
    slots[-1] = -1 if rows > 1 else slots[-1]      # a padding row writes nothing
    pools = torch.zeros(2, 64, hkv, 128, dtype=dtype, device="cuda")
    q = few_rows.qkv_rope(x, nw, 1e-6, w, bias, cos, sin, slots, pools[0], pools[1], hq, hkv)
    normed = add_rmsnorm(x, nw, 1e-6)[1]
    # the same projection without the rotation, then the rotation's own kernel: the products agree
    # but for the order of the norm's and the product's sums
    qkv = few_rows.linear(normed, w, bias=bias)
    ref = torch.zeros_like(pools)
    want = rope_kv_write(qkv, cos, sin, slots, ref[0], ref[1], hq, hkv)
    # rotated values: two products, each rounded, of a projection that may be a unit apart
    for got, ref_, parts in ((q, want, qkv[:, :hq * 128]), (pools, ref, qkv[:, hq * 128:])):
        close(got, ref_, product=torch.full_like(got, parts.abs().max().item()))
    assert torch.equal(pools[:, 0, 0, 0] == 0, ref[:, 0, 0, 0] == 0)


def test_special_values_stay_in_their_row():
    x = rand(3, 64, dtype=torch.bfloat16, seed=31)
    x[1] = float("nan")
    x[2, 5] = float("inf")
    w = rand(32, 64, dtype=torch.bfloat16, seed=32).abs()
    out = few_rows.linear(x, w)
    assert torch.isfinite(out[0]).all() and torch.isnan(out[1]).all() and torch.isinf(out[2]).all()


def test_a_graph_of_the_mlp_replays_like_the_eager_call():
    x = rand(16, 1536, dtype=torch.bfloat16, seed=41)
    gu = rand(2 * 8960, 1536, dtype=torch.bfloat16, seed=42, scale=0.02)
    down = rand(1536, 8960, dtype=torch.bfloat16, seed=43, scale=0.02)
    few_rows.mlp(x, gu, down)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = few_rows.mlp(x, gu, down)
    for seed in (44, 45, 46):
        x.copy_(rand(16, 1536, dtype=torch.bfloat16, seed=seed))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, few_rows.mlp(x, gu, down)), seed


def test_sizes_outside_the_kernel_are_refused():
    x, w = rand(65, 64, dtype=torch.bfloat16, seed=51), rand(32, 64, dtype=torch.bfloat16, seed=52)
    assert not few_rows.linear_fits(x, w) and few_rows.linear_fits(x[:64], w)
    with pytest.raises(_lib.MiFa2Error, match="rows 65"):
        few_rows.linear(x, w)
    assert not few_rows.linear_fits(x[:17], w, norm=w[0, :64].contiguous())
    assert not few_rows.linear_fits(x[:, :48][:4].contiguous(), w[:, :48].contiguous())


@DTYPES
@pytest.mark.parametrize("starts,T", [([0], 1), ([5, 0, 40000, 131071], 1), ([7, 1023], 300)])
def test_rope_tables_equal_the_torch_chain(starts, T, dtype):
    inv = (1.0 / (1e6 ** (torch.arange(0, 128, 2).float() / 128))).to(dtype).cuda()
    st = torch.tensor(starts, dtype=torch.int32, device="cuda")
    cos, sin = few_rows.rope_tables(st, T, inv)
    pos = st[:, None] + torch.arange(T, device="cuda")[None, :]
    fr = pos.float()[..., None] * inv[None, None, :]
    emb = torch.cat((fr, fr), dim=-1)
    for got, want in ((cos, emb.cos()), (sin, emb.sin())):
        # one rounding apart where the two libraries' fp32 values straddle a 16-bit boundary
        err = (got.float() - want[:, None]).abs()
        assert (err <= U[dtype] * want[:, None].abs() + 1e-6).all(), err.max().item()
