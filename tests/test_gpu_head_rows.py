"""Dense BF16 rows through affine_gemv at every form of the product behind it, outputs at any address."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


# Sums of n products of order n^-1/2, rounded at most n / 16 + 16 times: below 1e-6 of the largest value at these n, twice that; 2^-8 for a
# BF16 output.
@pytest.mark.parametrize("tokens", [1, 2, 4, 5, 16, 17, 64, 65, 200])
@pytest.mark.parametrize("m,n,offset,stride", [(250, 192, 1, 257), (1030, 4096, 0, 1037), (64, 64, 3, 71),
                                               (250, 192, 1, 256), (1030, 2048, 3, 1032), (64, 64, 2, 64)])      # four values at a time but for the address
def test_dense_rows(tokens, m, n, offset, stride):
    import nvmai_amd as nv
    from nvmai_amd._lib import check, lib
    say("dense BF16 rows", tokens, m, n, offset, stride)
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(m + tokens)
    w = (torch.randn((m, n), device="cuda", generator=gen) * n ** -0.5).to(torch.bfloat16)
    x = torch.randn((tokens, n), device="cuda", generator=gen).to(torch.bfloat16)
    want = x.double() @ w.double().T
    y, y32 = torch.full((tokens * stride + offset,), 7.0, device="cuda", dtype=torch.bfloat16), torch.full((tokens * stride + offset,), 7.0, device="cuda")
    check(lib.nvmai_hip_affine_gemv(ctx.handle, torch.cuda.current_stream().cuda_stream, w.data_ptr(), None, None, 16, x.data_ptr(), n, tokens, m, n,
                                    y.data_ptr() + 2 * offset, y32.data_ptr() + 4 * offset, stride), "affine_gemv")
    for got, tol in ((y, 2 ** -8), (y32, 2e-6)):
        assert bool((got[:offset] == 7).all())
        got = got[offset:].view(tokens, stride)
        assert bool((got[:, m:] == 7).all())
        assert float((got[:, :m].double() - want).abs().max() / want.abs().max()) <= tol
