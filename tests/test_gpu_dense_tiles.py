"""The tiled products behind dense_linear at the edges of their tiles, rounds and pipelines, against float64 on the device."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


def operands(rows, n, k, dtype, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w = (torch.randn((n, k), device="cuda", generator=gen) * k ** -0.5).to(torch.bfloat16)
    return w, torch.randn((rows, k), device="cuda", generator=gen).to(dtype)


def check(got, want, tol):
    assert float((got.double() - want).abs().max() / want.abs().max()) < tol


# A sum of k products of order k^-1/2 in fp32, rounded at most k / 16 + 16 times: 2^-24 sqrt(k / 16 + 16) of the largest value
# and below 1e-6 at these k; the bound is twice that.
@pytest.mark.parametrize("act", ["bf16", "fp32"])
@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 448])          # one to seven steps: every remainder of a ring of 2, 3, 4 or 5 stages
@pytest.mark.parametrize("rows,n", [(65, 250), (300, 64), (1000, 2047), (300, 8190), (2048, 2170), (2047, 8192)])  # each tile, ragged
def test_tiles(act, k, rows, n):
    import nvmai_amd as nv
    say("dense tiles", act, rows, n, k)
    ctx = nv.Context(0, nv.ACT_FP32 if act == "fp32" else nv.ACT_BF16)
    w, x = operands(rows, n, k, ctx.dtype, rows + n + k)
    want = x.double() @ w.double().T
    stride = n + 5
    y, y32 = torch.full((rows, stride), 7.0, dtype=ctx.dtype, device="cuda"), torch.full((rows, stride), 7.0, device="cuda")
    nv.dense_linear(ctx, w, x, y=y, y_f32=y32)
    check(y32[:, :n], want, 2e-6)
    check(y[:, :n], want, 2e-6 if act == "fp32" else 2 ** -8)
    assert bool((y[:, n:] == 7).all()) and bool((y32[:, n:] == 7).all())


def launches(call):
    """How many launches a call makes, by the nodes of a graph that records it."""
    import ctypes as C
    graph, stream = torch.cuda.CUDAGraph(keep_graph=True), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            call()
    n = C.c_size_t(0)
    assert C.CDLL("libamdhip64.so").hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(n)) == 0
    return n.value


def epilogue(kind, rows, n, want, table_rows=50):
    """The arguments of one kind of epilogue, and float64 sums `want` taken through it."""
    import nvmai_amd as nv
    gen = torch.Generator(device="cuda").manual_seed(12)
    bias, mul = torch.randn(n, device="cuda", generator=gen).to(torch.bfloat16), torch.randn((table_rows, n), device="cuda", generator=gen).to(torch.bfloat16)
    ids = torch.randint(0, table_rows + 2, (rows,), device="cuda", generator=gen, dtype=torch.int32)      # two of them past the table
    gelu = torch.nn.functional.gelu
    if kind == "erf":
        return dict(activation=nv.LINEAR_GELU_ERF), gelu(want)
    if kind == "bias":
        return dict(bias=bias), want + bias.double()
    if kind == "pairs":
        return dict(activation=nv.LINEAR_SILU_PAIRS), torch.nn.functional.silu(want[:, ::2]) * want[:, 1::2]
    if kind == "full":
        table = torch.cat([mul.double(), torch.zeros((2, n), dtype=torch.float64, device="cuda")])
        return dict(bias=bias, activation=nv.LINEAR_GELU_TANH, mul=mul, mul_ids=ids), gelu(want + bias.double(), approximate="tanh") * table[ids.long()]
    return {}, want


KINDS = ["plain", "erf", "bias", "pairs", "full"]


# 2048 rows x 8208: full rounds of large tiles and sixteen weight rows in a launch of their own, from 576 k on; 32-bit rows make
# their planes in a launch before that
@pytest.mark.parametrize("act", ["bf16", "fp32"])
@pytest.mark.parametrize("kind", KINDS)
def test_two_launches_with_every_epilogue(kind, act):
    import nvmai_amd as nv
    say("dense in two launches", kind, act)
    ctx = nv.Context(0, nv.ACT_FP32 if act == "fp32" else nv.ACT_BF16)
    rows, n, k = 2048, 8208, 1024
    w, x = operands(rows, n, k, ctx.dtype, 11)
    args, want = epilogue(kind, rows, n, x.double() @ w.double().T)
    y32 = torch.full((rows, want.shape[1]), 7.0, device="cuda")
    call = lambda: nv.dense_linear(ctx, w, x, y_f32=y32, **args)
    call()
    check(y32, want, 3e-6)              # the sum's 2e-6, and 1e-6 for a GELU or SiLU by hardware exponentials
    assert launches(call) == (3 if act == "fp32" else 2)


# rows: a wave per weight row, the short products, the tiles; strides: four multipliers at once, one by one
@pytest.mark.parametrize("act", ["bf16", "fp32"])
@pytest.mark.parametrize("rows", [3, 40, 200])
@pytest.mark.parametrize("n,stride", [(128, 128), (126, 131)])
def test_a_table_without_rows_multiplies_by_zero(act, rows, n, stride):
    """Nothing of the table is read: what lies there is not a number, and the ids are as large as they can be."""
    import ctypes as C

    import nvmai_amd as nv
    from nvmai_amd._lib import LinearEpilogue, check, lib
    say("multipliers past the table", act, rows, n)
    ctx = nv.Context(0, nv.ACT_FP32 if act == "fp32" else nv.ACT_BF16)
    w, x = operands(rows, n, 64, ctx.dtype, rows)
    table = torch.full((3, stride), float("nan"), device="cuda", dtype=torch.bfloat16)
    table[0] = 2.0
    ids = torch.full((rows,), -1, dtype=torch.int32, device="cuda")
    ids[::2] = 0
    stream = torch.cuda.current_stream().cuda_stream
    for table_rows in (0, 1):
        y = torch.full((rows, n), 7.0, device="cuda")
        e = LinearEpilogue(nv.LINEAR_NONE, None, table.data_ptr(), ids.data_ptr(), stride, table_rows)
        check(lib.nvmai_hip_dense_linear_ex(ctx.handle, stream, w.data_ptr(), 64, x.data_ptr(), 64, rows, n, 64, None, y.data_ptr(), n, C.byref(e)), "dense")
        want = x.double() @ w.double().T * 2.0 * table_rows
        want[1::2] = 0.0
        assert float((y.double() - want).abs().max()) < 1e-5 and bool((y[1::2] == 0).all())


def test_32_bit_values_keep_every_bit():
    """The planes of 32-bit rows hold them exactly: unit rows of the matrix give the inputs back, whatever their size."""
    import nvmai_amd as nv
    ctx = nv.Context(0, nv.ACT_FP32)
    x = torch.randn((70, 64), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    x = x * torch.logspace(-30, 30, 70, device="cuda")[:, None]
    x[0, 0], x[1, 1], x[2, 2], x[3, 3] = float("inf"), float("-inf"), float("nan"), 3.4028234663852886e38
    y = torch.empty((70, 64), device="cuda")
    nv.dense_linear(ctx, torch.eye(64, device="cuda", dtype=torch.bfloat16), x, y_f32=y)
    rest = torch.ones(70, dtype=torch.bool)
    rest[:3] = False                    # an infinity or NaN meets zeros in its row
    assert torch.equal(y[rest.cuda()], x[rest.cuda()])
    one = torch.ones((64, 64), device="cuda", dtype=torch.bfloat16)
    nv.dense_linear(ctx, one, x, y_f32=y)
    assert bool((y[0] == float("inf")).all()) and bool((y[1] == float("-inf")).all()) and bool(y[2].isnan().all())


def test_a_captured_call_without_workspace_still_runs():
    """The planes lie in the workspace; a call that is captured before anything has sized it takes a form without them."""
    import nvmai_amd as nv
    say("captured 32-bit product")
    w, x = operands(100, 200, 256, torch.float32, 5)
    want, y = x.double() @ w.double().T, torch.zeros((100, 200), device="cuda")
    warm, ctx = nv.Context(0, nv.ACT_FP32), nv.Context(0, nv.ACT_FP32)
    nv.dense_linear(warm, w, x, y_f32=torch.empty_like(y))            # loads the module
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            nv.dense_linear(ctx, w, x, y_f32=y)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        check(y, want, 2e-6)


# 2560 rows of 8192 k fill the portion of planes that is made at a time, 47 rows of 475,776, and seven of three million
@pytest.mark.parametrize("rows,n,k", [(2565, 72, 8192), (2560, 8, 8192), (5130, 40, 8192), (100, 24, 475776), (257, 16, 2800000)])
def test_32_bit_rows_in_portions(rows, n, k):
    """Every portion's rows of x, the outputs and the ids; sums of a long k in a total per 64."""
    import nvmai_amd as nv
    say("32-bit rows in portions", rows, n, k)
    ctx = nv.Context(0, nv.ACT_FP32)
    w, x = operands(rows, n, k, torch.float32, k)
    want = torch.cat([x[a:a + 64].double() @ w.double().T for a in range(0, rows, 64)])
    y, y32 = (torch.full((rows, n), 7.0, device="cuda") for _ in range(2))
    nv.dense_linear(ctx, w, x, y=y, y_f32=y32)
    # a total per 64 k: rounded k / 64 times, 2^-24 sqrt(k / 64) of the largest value and below 1.3e-5 at the longest k; twice that
    tol = max(2e-6, 2 * 2 ** -24 * (k / 64) ** 0.5)
    check(y32, want, tol)
    assert torch.equal(y, y32)
    bias, mul = torch.randn(n, device="cuda").to(torch.bfloat16), torch.randn((50, n), device="cuda").to(torch.bfloat16)
    ids = torch.arange(rows, device="cuda", dtype=torch.int32) * 7 % 50
    nv.dense_linear(ctx, w, x, y_f32=y32, bias=bias, activation=nv.LINEAR_GELU_TANH, mul=mul, mul_ids=ids)
    check(y32, torch.nn.functional.gelu(want + bias.double(), approximate="tanh") * mul.double()[ids.long()], 2 * tol)


@pytest.mark.parametrize("act", ["bf16", "fp32"])
@pytest.mark.parametrize("rows", [3, 40, 200, 2000])
def test_gelu_in_32_bit_precision(act, rows):
    """Unit rows of the matrix hand the inputs on, so only the activation rounds.  z/2 (1 + erf(z / sqrt 2)) for z in [-4, 1]: the argument is
    off by 2^-25, erff by two units of 2^-24, the sum rounds by 2^-24 and the product by 2^-23 at most, in all below 6 * 2^-24 of z / 2."""
    import nvmai_amd as nv
    say("gelu", act, rows)
    ctx = nv.Context(0, nv.ACT_FP32 if act == "fp32" else nv.ACT_BF16)
    eye = torch.eye(64, device="cuda", dtype=torch.bfloat16)
    x = (torch.rand((rows, 64), device="cuda", generator=torch.Generator(device="cuda").manual_seed(rows)) * 5.0 - 4.0).to(torch.bfloat16)
    z = x.double()
    y = torch.empty((rows, 64), device="cuda")
    nv.dense_linear(ctx, eye, x.to(ctx.dtype), y_f32=y, activation=nv.LINEAR_GELU_ERF)
    want = 0.5 * z * torch.special.erfc(-z * 0.5 ** 0.5)
    assert bool(((y.double() - want).abs() <= 6 * 2.0 ** -24 * z.abs() / 2).all())
    tanh = torch.empty((rows, 64), device="cuda")
    nv.dense_linear(ctx, eye, x.to(ctx.dtype), y_f32=tanh, activation=nv.LINEAR_GELU_TANH)
    want = torch.nn.functional.gelu(z, approximate="tanh")
    assert bool(((tanh.double() - want).abs() <= 6 * 2.0 ** -24 * z.abs() / 2).all())


# tiles of every size a 32-bit context has, one row a wave
@pytest.mark.parametrize("rows,n", [(3, 70), (70, 70), (700, 500), (2048, 2100)])
def test_infinite_weights_meet_32_bit_rows(rows, n):
    """An infinite weight gives an infinity of the input's sign, NaN only against zero or another infinity: whatever the planes of the
    input are (1.0 has zeros in two of them)."""
    import nvmai_amd as nv
    say("infinite weights", rows, n)
    k, inf = 192, float("inf")
    w, x = operands(rows, n, k, torch.float32, 9)
    x[:, 5] = torch.tensor([1.0, -2.0, 0.1, 0.0, 1e30], device="cuda").repeat(rows)[:rows]
    w[3, 5], w[n - 1, 5], w[n - 1, 70], w[20, 191] = inf, -inf, inf, -inf
    x[2, 100] = inf
    y = torch.empty((rows, n), device="cuda")
    nv.dense_linear(nv.Context(0, nv.ACT_FP32), w, x, y_f32=y)
    want = (x.cpu().double() @ w.cpu().double().T).cuda()
    assert torch.equal(y.isnan(), want.isnan())
    assert torch.equal(y.isinf(), want.isinf()) and torch.equal(y[y.isinf()].double(), want[want.isinf()])
    finite = want.isfinite()
    assert int(finite.sum()) > (n - 4) * (rows - 1) and float((y.double() - want)[finite].abs().max()) < 1e24      # 1e30 among the inputs


@pytest.mark.parametrize("kind", KINDS)
def test_captured_calls_without_workspace_with_every_epilogue(kind):
    """The form without planes, recorded while there is no workspace, ragged at the edges of its tiles of 64."""
    import nvmai_amd as nv
    say("captured 32-bit product", kind)
    rows, n, k = 100, 204, 320
    w, x = operands(rows, n, k, torch.float32, 5)
    args, want = epilogue(kind, rows, n, x.double() @ w.double().T)
    warm, ctx = nv.Context(0, nv.ACT_FP32), nv.Context(0, nv.ACT_FP32)
    y = torch.zeros(want.shape, device="cuda")
    nv.dense_linear(warm, w, x, y_f32=y, **args)                      # loads the module
    check(y, want, 3e-6)
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            nv.dense_linear(ctx, w, x, y_f32=y, **args)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        check(y, want, 3e-6)


@pytest.mark.parametrize("exponent", [-109, -111, -120, -126, -133, -149])
def test_32_bit_values_below_the_planes_range(exponent):
    """Exact down to 2^-110, within 2^-133 below it."""
    import nvmai_amd as nv
    x = ((torch.rand((70, 64), device="cuda", dtype=torch.float64, generator=torch.Generator(device="cuda").manual_seed(1)) + 1) * 2.0 ** exponent).float()
    y = torch.empty((70, 64), device="cuda")
    nv.dense_linear(nv.Context(0, nv.ACT_FP32), torch.eye(64, device="cuda", dtype=torch.bfloat16), x, y_f32=y)
    assert float((y.double() - x.double()).abs().max()) <= (0.0 if exponent > -110 else 2.0 ** -133)


@pytest.mark.parametrize("rows,n,k", [(70, 70, 64), (300, 260, 1088), (2048, 2100, 576)])
def test_32_bit_rows_that_are_not_numbers(rows, n, k):
    """A NaN makes NaN of its own row, whatever weights it meets; the other rows are what they were."""
    import nvmai_amd as nv
    say("32-bit rows that are not numbers", rows, n, k)
    ctx = nv.Context(0, nv.ACT_FP32)
    w, x = operands(rows, n, k, torch.float32, 13)
    clean = nv.dense_linear(ctx, w, x, y_f32=torch.empty((rows, n), device="cuda")).clone()
    bad = sorted({0, 5, 31, 32, rows // 2, rows - 1})
    for j, t in enumerate(bad):
        x[t, (j * 97 + k - 1) % k] = float("nan")
    w[n - 1, 3], w[1, k - 1] = float("inf"), float("-inf")
    y = nv.dense_linear(ctx, w, x, y_f32=torch.empty((rows, n), device="cuda"))
    fine = torch.ones(rows, dtype=torch.bool, device="cuda")
    fine[bad] = False
    assert bool(y[~fine].isnan().all())
    assert torch.equal(y[fine][:, 2:n - 1], clean[fine][:, 2:n - 1])
    assert torch.equal(y[fine, n - 1], torch.sign(x[fine, 3]) * float("inf")) and torch.equal(y[fine, 1], torch.sign(x[fine, k - 1]) * float("-inf"))
