"""One to four input rows at the lines of the rule that gives a wave its rows and steps: no choice changes a bit."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


# 2047, 8191 and 65,535 weight rows stand on the other side of a line each; the rows they share with the next size have the same sums.
@pytest.mark.parametrize("act", ["bf16", "fp32"])
@pytest.mark.parametrize("tokens", [1, 2, 3, 4])
@pytest.mark.parametrize("k", [64, 512, 576, 1024, 1088])
def test_rows_and_steps_of_a_wave(act, tokens, k):
    import nvmai_amd as nv
    say("rows and steps per wave", act, tokens, k)
    ctx = nv.Context(0, nv.ACT_FP32 if act == "fp32" else nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(k)
    w = (torch.randn((65537, k), device="cuda", generator=gen) * k ** -0.5).to(torch.bfloat16)
    x = torch.randn((tokens, k), device="cuda", generator=gen).to(ctx.dtype)
    want = x.double() @ w.double().T
    first = nv.dense_linear(ctx, w[:1001], x, y_f32=torch.empty((tokens, 1001), device="cuda"))
    for n in (2047, 2048, 8191, 8192, 65535, 65536, 65537):
        y = nv.dense_linear(ctx, w[:n], x, y_f32=torch.full((tokens, n + 3), 7.0, device="cuda"))
        assert torch.equal(y[:, :1001], first) and bool((y[:, n:] == 7).all()), n
        # a lane's k / 64 products and six additions of lanes, 2^-24 each: below 2^-22 of the largest value
        assert float((y[:, :n].double() - want[:, :n]).abs().max() / want.abs().max()) <= 2 ** -22, n
