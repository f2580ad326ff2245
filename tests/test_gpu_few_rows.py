"""Three and four input rows against quantized matrices at the lines of the rule that gives them to the matrix cores, and the norm before them."""
import pytest
import torch

from gpu_util import say
from test_gpu_widened import quantized, values

pytestmark = pytest.mark.gpu


# Inputs rounded to eleven bits, sums in fp32: off by 2^-11 of the largest value at most, and half a unit of BF16's last place, 2^-8.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tokens", [3, 4])
@pytest.mark.parametrize("m,n", [(8191, 2048), (8192, 2048), (70, 512), (300, 4096), (1000, 2048)])
def test_products(bits, tokens, m, n):
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("few rows", bits, tokens, m, n)
    ctx = nv.Context(0, nv.ACT_BF16)
    w = quantized(ctx, m, n, bits, m + n)
    x = torch.randn((tokens, n), device="cuda").to(torch.bfloat16)
    want = x.double() @ values(*w, bits).T
    y = ops.affine_gemv(ctx, *w, bits, x, m, n)
    y32 = ops.affine_gemv(ctx, *w, bits, x, m, n, out_f32=True)
    top = float(want.abs().max())
    assert float((y.double() - want).abs().max()) <= (2 ** -8 + 2 ** -11) * top
    assert float((y32.double() - want).abs().max()) <= 2 ** -11 * top


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tokens,m", [(3, 8192), (4, 8192), (4, 100), (3, 100), (4, 16400)])
@pytest.mark.parametrize("with_delta", [False, True])
def test_the_norm_before_them_has_the_bits_of_the_separate_calls(bits, tokens, m, with_delta):
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("few rows behind their norm", bits, tokens, m, with_delta)
    ctx, fresh = nv.Context(0, nv.ACT_BF16), nv.Context(0, nv.ACT_BF16)
    n = 2048
    w = quantized(ctx, m, n, bits, m)
    hidden, delta = (torch.randn((tokens, n), device="cuda").to(torch.bfloat16) for _ in range(2))
    weight = torch.randn(n, device="cuda").to(torch.bfloat16).view(torch.int16)
    want_h = hidden.clone()
    normed = ops.residual_add_rmsnorm(ctx, want_h, delta, weight) if with_delta else ops.RMSNorm(ctx).encode_bf16w(want_h, weight)
    want = ops.affine_gemv(ctx, *w, bits, normed, m, n)
    got_h, scratch = torch.zeros_like(hidden), torch.zeros_like(hidden)
    y = ops.affine_gemv_prenorm(ctx, *w, bits, hidden, delta if with_delta else None, weight, got_h, m, n, normed_scratch=scratch)
    assert torch.equal(got_h, want_h) and torch.equal(y, want)
    # recorded by a context without a workspace, and replayed
    y, stream, graph = torch.zeros_like(want), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            ops.affine_gemv_prenorm(fresh, *w, bits, hidden, delta if with_delta else None, weight, got_h, m, n, y=y, normed_scratch=scratch)
    for _ in range(3):
        y.zero_()
        got_h.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got_h, want_h) and torch.equal(y, want)


# Widths for which the row engine has no instantiation with its inputs in fp16: sums of floats, each of a lane's n / 64 products and the lanes' sums rounded to
# 24 bits, 2^-24 sqrt(n / 64 + 6) = 6e-7 of the value at most at these n (2-norm; inputs rounded to eleven bits as for the matrix cores give 1.2e-6 to 3.7e-6).
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tokens", [3, 4])
@pytest.mark.parametrize("n", [1536, 2560, 3584, 5120])
def test_other_widths_keep_inputs_of_32_bits(bits, tokens, n):
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("few rows, other widths", bits, tokens, n)
    ctx, m = nv.Context(0, nv.ACT_BF16), 300
    w = quantized(ctx, m, n, bits, n)
    x = torch.randn((tokens, n), device="cuda").to(torch.bfloat16)
    want = x.double() @ values(*w, bits).T
    got = ops.affine_gemv(ctx, *w, bits, x, m, n, out_f32=True)
    assert float((got.double() - want).norm() / want.norm()) <= 6e-7


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tokens,m", [(3, 8192), (4, 8192), (4, 100), (3, 100)])
def test_the_norm_before_them_needs_neither_workspace_nor_scratch_rows(bits, tokens, m):
    """A context that has made no call yet records the launches that it makes eagerly, and scratch rows stay as they are."""
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("few rows behind their norm, without workspace", bits, tokens, m)
    ctx, fresh, n = nv.Context(0, nv.ACT_BF16), nv.Context(0, nv.ACT_BF16), 2048
    w = quantized(ctx, m, n, bits, m)
    hidden, delta = (torch.randn((tokens, n), device="cuda").to(torch.bfloat16) for _ in range(2))
    weight = torch.randn(n, device="cuda").to(torch.bfloat16).view(torch.int16)
    want_h = hidden.clone()
    want = ops.affine_gemv(ctx, *w, bits, ops.residual_add_rmsnorm(ctx, want_h, delta, weight), m, n)
    got_h, scratch = torch.zeros_like(hidden), torch.full_like(hidden, 7.0)
    y = ops.affine_gemv_prenorm(ctx, *w, bits, hidden, delta, weight, got_h, m, n, normed_scratch=scratch)
    assert torch.equal(y, want) and bool((scratch == 7).all())
    y, stream, graph = torch.zeros_like(want), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            ops.affine_gemv_prenorm(fresh, *w, bits, hidden, delta, weight, got_h, m, n, y=y)
    for _ in range(3):
        y.zero_()
        got_h.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got_h, want_h) and torch.equal(y, want)


# panels of 2048 and of 1024 values, whole and not; one block of rows and a part of it, every number of them side by side
@pytest.mark.parametrize("bits,below,from_", [(4, 8, 9), (8, 13, 14), (4, 27, 28), (8, 30, 31)])
@pytest.mark.parametrize("m,n", [(10, 2048), (4100, 4096), (8200, 2048), (64, 3072), (64, 512)])
def test_rows_are_the_same_whether_inputs_or_weights_are_requested_first(bits, below, from_, m, n):
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("inputs first", bits, from_, m, n)
    ctx, gen = nv.Context(0, nv.ACT_BF16), torch.Generator(device="cuda").manual_seed(m + n)
    w = nv.quantize_affine(ctx, torch.empty((m, n), device="cuda").normal_(0.0, 0.05, generator=gen).to(torch.bfloat16), bits)
    x = torch.empty((32, n), device="cuda").normal_(0.0, 1.0, generator=gen).to(torch.bfloat16)
    full = 16 if from_ <= 16 else 32
    want = ops.affine_gemv(ctx, *w, bits, x[:below], m, n)
    for tokens in (from_, full - 1, full):
        got = ops.affine_gemv(ctx, *w, bits, x[:tokens], m, n)
        assert torch.equal(got[:below], want), tokens
        if tokens > below:      # a row among others and alone in the last place
            swapped = ops.affine_gemv(ctx, *w, bits, x[:tokens].flip(0).contiguous(), m, n)
            assert torch.equal(swapped.flip(0), got), tokens
    ctx.close()
