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


# every number of partial sums (4, 8 and 16, and 4 for many weight rows), both sides of each step
@pytest.mark.parametrize("n,k", [(300, 1024), (300, 1088), (300, 2048), (300, 2112), (2100, 4160), (2048, 8192), (520, 16384), (8191, 2112), (8192, 2112), (33000, 1088)])
def test_sums_by_size_alone(n, k):
    """The rows of a call choose the waves and tiles of the launch, and change no bit of a row's own sums; these are as close to those in 64 bits as
    their partial sums allow.  P of them, each a chain of c = k / (32 P) matrix instructions, are added in a chain: if every
    one of them rounds by 2^-24 of what it holds, independently, the squares add up to 2^-48 (c + P) / 2 of the outputs'."""
    import nvmai_amd as nv
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    randn = lambda *s: torch.empty(s, device="cuda").normal_(0.0, 1.0, generator=gen)
    w, x = (randn(n, k) * k ** -0.5).bfloat16(), randn(64, k).bfloat16()
    want, first = x.double() @ w.double().T, None
    sums = 4 if n >= 8192 or k <= 1024 else 8 if k <= 2048 else 16
    for rows in (5, 16, 17, 32, 33, 64):
        say("sums", rows, n, k)
        y = torch.zeros((rows, n), device="cuda")
        nv.dense_linear(ctx, w, x[:rows], y_f32=y)
        error = float((y.double() - want[:rows]).norm() / want[:rows].norm())
        assert error < 2 ** -24 * ((k / 32 / sums + sums) / 2) ** 0.5, error
        first = y if first is None else first
        assert torch.equal(y[:5], first)
