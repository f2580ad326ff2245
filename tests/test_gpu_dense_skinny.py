"""Products of 5 to 64 rows: every form of the launch, numbers of steps around the waves' rings (two or four stages, two or four waves) and partial
sums (one to eight per wave), ragged rows and strides, every epilogue, against the same in 64 bits."""
import pytest
import torch

from gpu_util import say
from test_gpu_dense_tiles import KINDS, check, epilogue

pytestmark = pytest.mark.gpu


# k: one step, fewer steps than waves, a ring less one, a ring, several and a rest.  Up to 16 rows: eight weight rows per block in the sizes up to n = 2048 with
# k past 1024; sixteen in two waves (19 x 512, 2049 x 1088, 4097 x 2112) and in four (2049 and 4096 x 2112, 4099 and 8197 x 4160).  More rows: one row tile per block
# with two, four and eight sums per wave, two (8197) and four (32,771) tiles with rings that turn
@pytest.mark.parametrize("rows", [5, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(19, 64), (3, 128), (35, 192), (50, 448), (19, 512), (16, 576), (67, 2048), (19, 2112), (45, 8256), (8197, 320), (32771, 128),
                                 (2048, 1024), (2048, 1088), (2049, 1088), (2048, 2112), (2049, 2112), (4096, 2112), (4097, 2112), (4099, 4160), (8197, 4160), (8197, 1344),
                                 (32771, 1088)])
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


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,n,k", [(5, 38, 1088), (16, 38, 2112), (16, 2046, 4160), (5, 1030, 512), (16, 2054, 2112), (5, 4102, 2112), (17, 2054, 1088), (32, 8198, 320),
                                      (64, 2054, 2112), (40, 8198, 320), (33, 32774, 192)])
def test_epilogues_of_every_form(kind, rows, n, k):
    import nvmai_amd as nv
    say("skinny", kind, rows, n, k)
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    randn = lambda *s: torch.empty(s, device="cuda").normal_(0.0, 1.0, generator=gen)
    w, x = (randn(n, k) * k ** -0.5).bfloat16(), randn(rows, k).bfloat16()
    args, want = epilogue(kind, rows, n, x.double() @ w.double().T)
    m = want.shape[1]
    y, y32 = torch.full((rows, m + m % 2 + 6), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((rows, m + m % 2 + 6), 7.0, device="cuda")
    nv.dense_linear(ctx, w, x, y=y, y_f32=y32, **args)
    check(y32[:, :m], want, 3e-6)           # the sum's 2e-6, and 1e-6 for a GELU or SiLU by hardware exponentials
    assert torch.equal(y32[:, :m].bfloat16(), y[:, :m]) and (y[:, m:] == 7).all() and (y32[:, m:] == 7).all()


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
