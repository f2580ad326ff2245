"""Norms of many rows of 2048, held in registers, against rows at odd addresses, which go value by value: the same bits, in place too and without a weight."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["ACT_BF16", "ACT_FP16"])
@pytest.mark.parametrize("rows", [257, 1027])          # past the form of few rows; a last block that is not full
@pytest.mark.parametrize("weighted", [True, False])
def test_rows_in_registers(act, rows, weighted):
    import nvmai_amd as nv
    from nvmai_amd._lib import check, lib
    print("norms of rows", act, rows, weighted, flush=True)
    ctx, d = nv.Context(0, getattr(nv, act)), 2048
    gen = torch.Generator(device="cuda").manual_seed(rows)
    n = lambda *s: torch.empty(s, device="cuda").normal_(0.0, 1.0, generator=gen).to(ctx.dtype)
    x, delta = n(rows, d), n(rows, d)
    x[3, 5], delta[4, 6] = float("inf"), float("nan")
    weight = n(d).to(torch.bfloat16)
    w = weight.data_ptr() if weighted else None
    s = nv.ops._stream()

    def at(values, off):
        wide = torch.zeros((rows, d + 8), dtype=ctx.dtype, device="cuda")[:, off:off + d]
        return wide.copy_(values)
    out = []
    for off in (0, 1):
        a, b, c, e = at(x, off), at(delta, off), at(x, off), at(x, off)
        to, normed = at(x, off), at(x, off)
        check(lib.nvmai_hip_residual_add_rmsnorm(ctx.handle, s, a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), w, to.data_ptr(), to.stride(0), rows, d, 1e-5), "add")
        check(lib.nvmai_hip_rmsnorm(ctx.handle, s, c.data_ptr(), c.stride(0), w, normed.data_ptr(), normed.stride(0), rows, d, 1e-5), "norm")
        check(lib.nvmai_hip_rmsnorm(ctx.handle, s, e.data_ptr(), e.stride(0), w, e.data_ptr(), e.stride(0), rows, d, 1e-5), "norm")
        torch.cuda.synchronize()
        out.append([v.float() for v in (a, to, normed, e)])
    for held, single in zip(*out):
        assert torch.equal(torch.isnan(held), torch.isnan(single)) and torch.equal(torch.nan_to_num(held, nan=7.0), torch.nan_to_num(single, nan=7.0))
    assert torch.equal(torch.nan_to_num(out[0][2], nan=7.0), torch.nan_to_num(out[0][3], nan=7.0))
    ctx.close()
