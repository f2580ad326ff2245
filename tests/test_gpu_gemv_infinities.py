"""Infinities at the end of one to four input rows, where a lane's last steps lie past the matrix."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


# Steps of 512 k, two or four at a time: widths below, at and past one turn.  All weights are positive, so that a row with an infinity has infinite outputs.
@pytest.mark.parametrize("tokens", [1, 2, 3, 4])
@pytest.mark.parametrize("k", [64, 512, 576, 1024, 1088, 2048, 2112, 4096])
def test_an_infinite_input_gives_infinite_outputs(tokens, k):
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("infinite inputs", tokens, k)
    n = 70
    gen = torch.Generator(device="cuda").manual_seed(k)
    w = (torch.rand((n, k), device="cuda", generator=gen) + 0.1).to(torch.bfloat16)
    for at in (0, k - 8, k - 1):
        for act, dtype in ((nv.ACT_BF16, torch.bfloat16), (nv.ACT_FP32, torch.float32)):
            ctx = nv.Context(0, act)
            x = torch.randn((tokens, k), device="cuda", generator=gen).to(dtype)
            x[tokens - 1, at] = -float("inf")
            got = [nv.dense_linear(ctx, w, x, y_f32=torch.empty((tokens, n), device="cuda"))]
            if act == nv.ACT_BF16:
                got.append(ops.affine_gemv(ctx, w.view(torch.uint8), None, None, 16, x, n, k, out_f32=True))
            for y in got:
                assert bool((y[-1] == -float("inf")).all()) and bool(y[:-1].isfinite().all()), at
