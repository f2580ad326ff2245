"""The order in which the tiled products add: pieces of eight k, one after another from the first to the last."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


# Every piece holds one value that is not zero, +-2^60 or 1, so that each step of the sum is exact or loses the 1 (far below the bits that a matrix instruction
# keeps): the sum in this order is a number that another order of the pieces does not give.  Weights are one, and two in odd rows: a power of two changes no
# rounding.  32-bit inputs: 64 k are summed from zero, and those sums in their order.  Sizes whose tiles are not cut along k: fewer than four steps of 64 k,
# tiles for every compute unit, or little to gain; (4096, 8200) leaves eight weight rows to a launch of their own.
SIZES = [(65, 4096, 192), (300, 4100, 192), (1000, 2047, 128), (700, 11264, 192), (2047, 8192, 448), (4096, 8200, 320)]


@pytest.mark.parametrize("act,rows,n,k", [(act, *size) for act in ("bf16", "fp32") for size in SIZES] + [("bf16", 1501, 256, 2048)])
def test_pieces_are_added_in_the_order_of_k(act, rows, n, k):
    import nvmai_amd as nv
    say("order of the sums", act, rows, n, k)
    ctx = nv.Context(0, nv.ACT_FP32 if act == "fp32" else nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(rows + k)
    pieces = k // 8
    value = torch.tensor([2.0 ** 60, -2.0 ** 60, 1.0, 1.0], device="cuda")[torch.randint(0, 4, (rows, pieces), device="cuda", generator=gen)]
    at = torch.randint(0, 8, (rows, pieces, 1), device="cuda", generator=gen)
    x = torch.zeros((rows, pieces, 8), device="cuda").scatter_(2, at, value[..., None]).view(rows, k).to(ctx.dtype)
    w = torch.ones((n, k), device="cuda")
    w[1::2] = 2.0

    def total(order):
        whole, part = torch.zeros(rows, device="cuda"), torch.zeros(rows, device="cuda")
        for i in range(pieces):
            part = part + value[:, i // 8 * 8 + order[i % 8]]
            if act == "fp32" and i % 8 == 7:
                whole, part = whole + part, torch.zeros_like(part)
        return whole + part
    want = total(range(8))
    assert not torch.equal(want, total((0, 2, 4, 6, 1, 3, 5, 7)))
    y = nv.dense_linear(ctx, w.to(torch.bfloat16), x, y_f32=torch.empty((rows, n), device="cuda"))
    assert torch.equal(y, want[:, None] * w[:, 0])
