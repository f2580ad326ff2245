"""The end of a prompt's layer in one launch against the reduce, the add and the residual add with its norm one after the other: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# less than a piece per thread, one, the next piece's first values, two and four pieces; ranks of one round and of the next
@pytest.mark.parametrize("act", ["ACT_BF16", "ACT_FP16"])
@pytest.mark.parametrize("tokens,top_k,d", [(1, 1, 8), (5, 8, 136), (3, 9, 2048), (2, 8, 2056), (7, 4, 4096), (2, 17, 4104), (2, 8, 8192)])
def test_same_bits_as_three_launches(act, tokens, top_k, d):
    import nvmai_amd as nv
    print("reduce and norm", act, tokens, top_k, d, flush=True)
    ctx = nv.Context(0, getattr(nv, act))
    gen = torch.Generator(device="cuda").manual_seed(d + top_k)
    n = lambda *s: torch.empty(s, device="cuda").normal_(0.0, 1.0, generator=gen).to(ctx.dtype)
    partials, w = n(tokens * top_k, d), torch.empty((tokens, top_k), device="cuda").uniform_(0.0, 1.0, generator=gen).to(torch.float16)
    add, weight = n(tokens, d + 8)[:, :d], n(d).to(torch.bfloat16).view(torch.int16)
    partials[0, 0], add[0, 1] = float("inf"), float("nan")
    wide = n(tokens, d + 16)
    a, b = wide.clone()[:, :d], wide.clone()[:, :d]
    h2 = nv.PrefillMoE(ctx).encode_reduce_token_major(partials, w, tokens, top_k, d)
    want = nv.ops.residual_add_rmsnorm(ctx, a, nv.ops.Elementwise(ctx).encode_residual_add(h2, add.contiguous()), weight, eps=1e-5)
    got = nv.PrefillMoE(ctx).encode_reduce_norm(partials, w, top_k, add, b, weight, 1e-5)
    same = lambda x, y: torch.equal(torch.nan_to_num(x.float(), nan=7.0), torch.nan_to_num(y.float(), nan=7.0)) and torch.equal(torch.isnan(x), torch.isnan(y))
    assert same(a, b) and same(got, want) and (tokens == 1 or bool(torch.isfinite(got[1:]).all()))
    ctx.close()


def test_refusals():
    import nvmai_amd as nv
    ctx = nv.Context(0, nv.ACT_BF16)
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros((2, 2), dtype=torch.float16, device="cuda")
    for d in (12, 8200):
        with pytest.raises(nv.NvmaiError):
            nv.PrefillMoE(ctx).encode_reduce_norm(z(4, d), w, 2, z(2, d), z(2, d), z(d))
    with pytest.raises(nv.NvmaiError):
        nv.PrefillMoE(ctx).encode_reduce_norm(z(4, 16), w, 2, z(2, 20)[:, 2:18], z(2, 16), z(16))
    ctx.close()
