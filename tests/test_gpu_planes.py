"""Rows of 32-bit contexts that their producer stores as three BF16 planes: the bits of the calls on rows of floats."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nv():
    import nvmai_amd
    return nvmai_amd


def _normal(gen, *shape):
    return torch.empty(shape, device="cuda").normal_(0.0, 1.0, generator=gen)


def _planes(x):
    """[rows, 3, k] BF16 by truncation, the smallest part first; infinities in the last one."""
    cut = lambda v: (v.view(torch.int32) & -65536).view(torch.float32)
    hi = cut(x)
    mid = torch.where(torch.isfinite(x), cut(x - hi), 0.0)
    lo = torch.where(torch.isfinite(x), x - hi - mid, 0.0)
    return torch.stack([cut(lo), mid, hi], 1).to(torch.bfloat16)


def _same(a, b):
    """The same bits, whatever NaN it is."""
    return torch.equal(torch.nan_to_num(a, nan=7.0), torch.nan_to_num(b, nan=7.0)) and torch.equal(torch.isnan(a), torch.isnan(b))


# the fewest rows, edges of tiles, products in one launch and in two, cut along k; outputs that end inside a tile
@pytest.mark.parametrize("rows,n,k", [(5, 64, 64), (64, 132, 1024), (65, 1024, 64), (127, 4100, 1024), (700, 1024, 4096), (513, 2816, 1024)])
def test_products(nv, rows, n, k):
    print("planes", rows, n, k, flush=True)
    ctx, ops = nv.Context(0, nv.ACT_FP32), nv.ops
    gen = torch.Generator(device="cuda").manual_seed(rows + n)
    w, x = _normal(gen, n, k).to(torch.bfloat16) * k ** -0.5, _normal(gen, rows, k)
    x[0, 1], x[1, :3] = 0.0, torch.tensor([1e-30, float("inf"), -1e30], device="cuda")
    bias, table = _normal(gen, n).to(torch.bfloat16), _normal(gen, 50, n).to(torch.bfloat16)
    ids = torch.arange(rows, device="cuda", dtype=torch.int32) % 51
    more = [dict(), dict(activation=ops.LINEAR_GELU_ERF), dict(bias=bias), dict(activation=ops.LINEAR_SILU_PAIRS),
            dict(activation=ops.LINEAR_GELU_TANH, mul=table, mul_ids=ids)]
    for e in more:
        cols = n // 2 if e.get("activation") == ops.LINEAR_SILU_PAIRS else n
        y_k = (cols + 63) // 64 * 64
        want, got = torch.zeros((rows, y_k), device="cuda"), torch.zeros((rows, y_k), device="cuda")
        ops.dense_linear(ctx, w, x, y=want, **e)
        ops.dense_linear(ctx, w, _planes(x), y=got, **e)
        assert _same(got, want), e
        out = torch.zeros((rows, 3, y_k), dtype=torch.bfloat16, device="cuda")
        ops.dense_linear(ctx, w, _planes(x), y=out, **e)
        finite = torch.isfinite(want)
        assert torch.equal(torch.where(finite, out[:, 2].float() + out[:, 1].float() + out[:, 0].float(), 0.0), torch.where(finite, want, 0.0)), e
        assert _same(out[:, 2].float()[~finite], want[~finite])
    ctx.close()


@pytest.mark.parametrize("rows,d,k", [(1, 64, 64), (7, 1022, 1024), (33, 1024, 1024), (5, 2050, 2112), (3, 4096, 4096)])
def test_norms(nv, rows, d, k):
    print("planes of norms", rows, d, k, flush=True)
    ctx, ops = nv.Context(0, nv.ACT_FP32), nv.ops
    gen = torch.Generator(device="cuda").manual_seed(d)
    w = lambda: _normal(gen, d).to(torch.bfloat16)
    x, delta, pair, other = _normal(gen, rows, d), _normal(gen, rows, k), (w(), w()), (w(), w())
    calls = [lambda x, out: ops.norm_residual(ctx, x, d, delta, pair, 0.5, other, out), lambda x, out: ops.norm_residual(ctx, x, d, next_norm=other, out=out),
             lambda x, out: ops.rms_residual(ctx, x, d, delta, pair[0], 1.0, other[0], 1.0, out), lambda x, out: ops.rms_residual(ctx, x, d, delta, pair[0], 0.0, out=out)]
    for call in calls:
        a, b, want, got = x.clone(), x.clone(), torch.zeros((rows, k), device="cuda"), torch.zeros((rows, 3, k), dtype=torch.bfloat16, device="cuda")
        call(a, want)
        call(b, got)
        assert torch.equal(a, b) and torch.equal(got[:, 2].float() + got[:, 1].float() + got[:, 0].float(), want)
    ctx.close()


def test_refusals(nv):
    ctx, half, ops = nv.Context(0, nv.ACT_FP32), nv.Context(0, nv.ACT_BF16), nv.ops
    w, x = torch.zeros((66, 64), dtype=torch.bfloat16, device="cuda"), torch.zeros((8, 3, 64), dtype=torch.bfloat16, device="cuda")
    y = torch.zeros((8, 66), device="cuda")
    # fewer than five rows; planes of an odd number of rows of the matrix; a context of 16 bits
    for a, out in ((x[:4], y), (x, torch.zeros((8, 3, 128), dtype=torch.bfloat16, device="cuda"))):
        with pytest.raises(nv.NvmaiError):
            ops.dense_linear(ctx, w, a, y=out)
    e = nv.ops.LinearEpilogue(ops.LINEAR_NONE, None, None, None, 0, 0)
    assert nv.lib.nvmai_hip_dense_linear_planes(half.handle, ops._stream(), w.data_ptr(), 64, x.data_ptr(), 8, 66, 64, y.data_ptr(), 66, None, 0, C.byref(e)) != 0
    ops.dense_linear(ctx, w, x, y=y)
    ctx.close()
    half.close()


def test_rows_of_floats_by_heads(nv):
    # three dimensions do not make planes: [tokens, 3, values] floats are rows of 3 * values
    print("floats by heads", flush=True)
    ctx, ops = nv.Context(0, nv.ACT_FP32), nv.ops
    gen = torch.Generator(device="cuda").manual_seed(3)
    w, norm, x = _normal(gen, 96, 192).to(torch.bfloat16), _normal(gen, 192).to(torch.bfloat16), _normal(gen, 40, 192)
    want, got = torch.zeros((40, 96), device="cuda"), torch.zeros((40, 3, 32), device="cuda")
    ops.dense_linear(ctx, w, x, y=want)
    ops.dense_linear(ctx, w, x.view(40, 3, 64), y=got)
    assert torch.equal(got.view(40, 96), want)
    for call in (lambda out: ops.norm_residual(ctx, x, 192, next_norm=(norm, norm), out=out), lambda out: ops.rms_residual(ctx, x, 192, next_norm=norm, out=out)):
        want, got = torch.zeros((40, 192), device="cuda"), torch.zeros((40, 3, 64), device="cuda")
        call(want), call(got)
        assert torch.equal(got.view(40, 192), want)
    ctx.close()
