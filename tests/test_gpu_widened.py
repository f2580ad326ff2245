"""Dense products over quantized rows whose codes are widened to BF16 once: ragged sizes, odd strides, the form without workspace."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


def values(packed, scales, biases, bits):
    rows = packed.shape[0]
    q = packed.double() if bits == 8 else torch.stack([packed & 15, packed >> 4], -1).reshape(rows, -1).double()
    f = lambda t: t.view(torch.bfloat16).double().view(rows, -1, 1)
    return (q.view(rows, -1, 64) * f(scales) + f(biases)).view(rows, -1)


def quantized(ctx, n, k, bits, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    import nvmai_amd as nv
    return nv.quantize_affine(ctx, (torch.randn((n, k), device="cuda", generator=gen) * k ** -0.5).to(torch.bfloat16), bits)


# The output is rounded to BF16, eight bits: off by half a unit of its last place, 2^-8 of itself at most.  The weights are too, each by 2^-8 of itself at
# most, evenly spread and so 2^-8 3^-1/2 on average: a sum of products by as much of its own size, which over a million sums (five times their mean size
# at most, the largest value five times as well) stays below 2^-9 of the largest value.
TOL = 1.5 * 2 ** -8


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n,k", [(33, 1024, 192), (64, 1030, 1024), (65, 2048, 4096), (130, 1999, 2112), (700, 1024, 2048), (1500, 3000, 1024), (257, 9216, 2048)])
def test_products(bits, rows, n, k):
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("product over quantized rows", bits, rows, n, k)
    ctx = nv.Context(0, nv.ACT_BF16)
    w = quantized(ctx, n, k, bits, rows + n)
    # scales and biases that start on an odd half word
    meta = [torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].copy_(t.view(-1)).view(t.shape) for t in w[1:]]
    x = torch.randn((rows, k + 8), device="cuda").to(torch.bfloat16)[:, :k]
    want = x.double() @ values(*w, bits).T
    y = torch.full((rows, n + 3), 7.0, dtype=torch.bfloat16, device="cuda")
    for _ in range(2):
        ops.MPPPrefillInt4QMM(ctx, bits).encode(w[0], *meta, x, n, k, y=y)
        assert float((y[:, :n].double() - want).abs().max() / want.abs().max()) < TOL
        assert bool((y[:, n:] == 7).all())


def test_a_captured_product_without_workspace_dequantizes_per_tile():
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("captured product over quantized rows")
    warm, ctx = nv.Context(0, nv.ACT_BF16), nv.Context(0, nv.ACT_BF16)
    rows, n, k = 100, 2048, 4096
    w = quantized(warm, n, k, 4, 3)
    x = torch.randn((rows, k), device="cuda").to(torch.bfloat16)
    want = x.double() @ values(*w, 4).T
    y = torch.zeros((rows, n), dtype=torch.bfloat16, device="cuda")
    ops.affine_gemv(warm, *w, 4, x, n, k, y=y)
    ops.affine_gemv(nv.Context(0, nv.ACT_FP16), *w, 4, x.half(), n, k, y=torch.empty_like(x[:, :n].half()))       # loads the other form
    torch.cuda.synchronize()
    for c in (ctx, warm):                                             # without a workspace, and with one
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            with torch.cuda.graph(graph, stream=stream):
                ops.affine_gemv(c, *w, 4, x, n, k, y=y)
        for _ in range(3):
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert float((y.double() - want).abs().max() / want.abs().max()) < TOL


# The two forms round the same values to the same weights (a scale and a bias of eight bits each: the shifted bias of the form per tile is exact) and add in
# another order: sums apart by 2^-20 of their size at most.  Outputs then are, where a sum lies that near the middle of two BF16 values, which are 2^-8 of it
# apart or half that: one output in 2^11, by 2^-8 of itself on average.  In all 2^-5.5 2^-8 of the outputs; not nothing, which would be one form twice.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n,k", [(65, 2048, 4096), (130, 1999, 2112), (700, 1024, 2048), (257, 2048, 4096)])
def test_both_forms_round_alike(bits, rows, n, k):
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("product over quantized rows, both forms", bits, rows, n, k)
    ctx, fresh = nv.Context(0, nv.ACT_BF16), nv.Context(0, nv.ACT_BF16)
    w = quantized(ctx, n, k, bits, n + k)
    x = torch.randn((rows, k), device="cuda").to(torch.bfloat16)
    widened, per_tile = torch.empty((rows, n), dtype=torch.bfloat16, device="cuda"), torch.empty((rows, n), dtype=torch.bfloat16, device="cuda")
    encode = lambda c, y: ops.MPPPrefillInt4QMM(c, bits).encode(*w, x, n, k, y=y)
    encode(ctx, widened)
    torch.cuda.synchronize()
    assert ctx.workspace_bytes >= n * k * 2                           # the form in question
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            encode(fresh, per_tile)
    graph.replay()
    torch.cuda.synchronize()
    assert fresh.workspace_bytes == 0
    a, b = widened.double(), per_tile.double()
    assert 0 < float((a - b).norm() / b.norm()) <= 2 ** -13.5


# The hidden row is rounded to BF16 between the products and the output once more: TOL for each of the two products covers them.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tokens,d,f", [(192, 1024, 256), (333, 2048, 512), (2100, 512, 320)])
def test_shared_expert(bits, tokens, d, f):
    import nvmai_amd as nv
    from nvmai_amd import ops
    say("shared expert over a block of tokens", bits, tokens, d, f)
    ctx = nv.Context(0, nv.ACT_BF16)
    off, stride = nv.expert_offsets(d, f, bits)
    blob = torch.empty(stride, dtype=torch.uint8, device="cuda")
    w = []
    for i, (n, k, wo, so, bo) in enumerate(((f, d, off.gate_w, off.gate_s, off.gate_b), (f, d, off.up_w, off.up_s, off.up_b), (d, f, off.down_w, off.down_s, off.down_b))):
        q = quantized(ctx, n, k, bits, i)
        for t, o in zip(q, (wo, so, bo)):
            flat = t.view(torch.uint8).view(-1)
            blob[o:o + flat.numel()] = flat
        w.append(values(*q, bits))
    x = torch.randn((tokens, d), device="cuda").to(torch.bfloat16)
    xd = x.double()
    want = (torch.nn.functional.silu(xd @ w[0].T) * (xd @ w[1].T)) @ w[2].T
    y = ops.SharedExpertRuntime(ctx, bits).encode(blob, off, x, d, f)
    assert float((y.double() - want).abs().max() / want.abs().max()) < 2 * TOL


@pytest.mark.parametrize("tokens", [131200, 270000])
def test_a_shared_expert_past_offsets_of_32_bits(tokens):
    """f values of 131,200 tokens lie 4.3 GB apart as the dense products count them: the form that dequantizes per tile takes the call; 270,000 in two portions."""
    import nvmai_amd as nv
    from nvmai_amd import ops
    bits, d, f = 4, 2048, 8192
    say("shared expert of many tokens", bits, tokens, d, f)
    ctx = nv.Context(0, nv.ACT_BF16)
    off, stride = nv.expert_offsets(d, f, bits)
    blob = torch.empty(stride, dtype=torch.uint8, device="cuda")
    w = []
    for i, (n, k, wo, so, bo) in enumerate(((f, d, off.gate_w, off.gate_s, off.gate_b), (f, d, off.up_w, off.up_s, off.up_b), (d, f, off.down_w, off.down_s, off.down_b))):
        q = quantized(ctx, n, k, bits, i)
        for t, o in zip(q, (wo, so, bo)):
            flat = t.view(torch.uint8).view(-1)
            blob[o:o + flat.numel()] = flat
        w.append(values(*q, bits))
    x = torch.empty((tokens, d), device="cuda", dtype=torch.bfloat16).normal_()
    y = ops.SharedExpertRuntime(ctx, bits).encode(blob, off, x, d, f)
    at = torch.tensor([0, 1, 65535, 65536, 131071, 131072, 131199, tokens - 7985, tokens - 7984, tokens - 1], device="cuda")
    xd = x[at].double()
    want = (torch.nn.functional.silu(xd @ w[0].T) * (xd @ w[1].T)) @ w[2].T
    assert float((y[at].double() - want).abs().max() / want.abs().max()) < 2 * TOL
