"""Products of 5 to 64 rows: every form of the launch, numbers of steps around the waves' rings (two to four stages, two or four waves), ragged rows and
strides, against the same in 64 bits."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


# k: one step, fewer steps than waves, a ring less one, a ring, several and a rest, the four-wave form (past 2048); n: a tile and a rest, two and four
# row tiles per block
@pytest.mark.parametrize("rows", [5, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(19, 64), (3, 128), (35, 192), (50, 448), (19, 512), (16, 576), (67, 2048), (19, 2112), (45, 8256), (8197, 320), (32771, 128)])
def test_products_of_few_rows(rows, n, k):
    import nvmai_amd as nv
    ctx = nv.Context(0, nv.ACT_BF16)
    say("skinny", rows, n, k)
    gen = torch.Generator(device="cuda").manual_seed(rows * 7 + n + k)
    randn = lambda *s: torch.empty(s, device="cuda").normal_(0.0, 1.0, generator=gen)
    w, x = (randn(n, k + 8) * k ** -0.5).bfloat16()[:, :k], randn(rows, k + 24).bfloat16()[:, :k]
    y, y32 = torch.full((rows, n + 5), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((rows, n + 5), 7.0, device="cuda")
    nv.dense_linear(ctx, w, x, y=y, y_f32=y32)
    want = x.double() @ w.double().T
    # sums of k products in fp32: a few roundings of sums of order one
    assert (y32[:, :n].double() - want).abs().max() < 4e-6 and torch.equal(y32[:, :n].bfloat16(), y[:, :n])
    assert (y[:, n:] == 7).all() and (y32[:, n:] == 7).all()
