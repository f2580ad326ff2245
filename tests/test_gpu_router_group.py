"""Router, selection and work list of a small batch in one launch against the same steps in their own launches (which a normed row that ends where a row of
the residual stream begins takes): the same experts, weights and sums, with waits that end at once too, and replayed."""
import pytest
import torch

from test_gpu_moe_one import _layer, nv  # noqa: F401

pytestmark = pytest.mark.gpu


def _both(nv, ctx, layer, x, delta, weight):
    """(residual stream, normed rows, output, experts, weights, statistics) in one launch, then in two."""
    moe, out, T, D = nv.MoE(ctx, layer.bits), [], x.shape[0], x.shape[1]
    for over in (False, True):
        # the stream's rows and the normed ones, those in the stream's padding where they are not to be taken in one launch
        rows = torch.zeros((T, 2 * D), dtype=x.dtype, device="cuda")
        rows[:, :D] = x
        hidden = rows[:, :D]
        normed = rows[:, D:] if over else torch.empty_like(x)
        stats = torch.zeros(2, dtype=torch.int32, device="cuda")
        kept, y = torch.empty_like(x), torch.empty_like(x)
        idx = torch.empty((T, layer.top_k), dtype=torch.int32, device="cuda")
        w = torch.empty((T, layer.top_k), dtype=torch.float16, device="cuda")
        moe.decode_layer_prenorm(layer, hidden, delta, weight, kept, normed, y, idx=idx, w=w, stats=stats)
        torch.cuda.synchronize()
        out.append([t.clone().contiguous() for t in (kept, normed, y, idx, w, stats)])
    return out


@pytest.mark.parametrize("act", ["ACT_BF16", "ACT_FP16"])
@pytest.mark.parametrize("looks", [1 << 14, 0])
# tokens of one choosing block and of the next, of several; experts at the edges of a lane's share and of a block of rows; rows of one to eight pieces a lane
@pytest.mark.parametrize("tokens,d,E,k,kind,gated", [
    (1, 512, 40, 3, 4, True), (2, 1024, 256, 8, 16, False), (5, 2048, 256, 8, 16, True), (8, 1024, 257, 7, 16, True), (16, 2048, 255, 8, 8, True), (17, 512, 8, 8, 16, False), (32, 2048, 256, 8, 16, True),
    (33, 256, 40, 3, 4, True), (63, 1024, 512, 4, 16, True)])
def test_one_launch_equals_two(nv, act, looks, tokens, d, E, k, kind, gated):
    print("router and work list", act, looks, tokens, d, E, k, flush=True)
    ctx = nv.Context(0, getattr(nv, act))
    assert nv.lib.nvmai_hip_ctx_wait_limit(ctx.handle, looks) == 0
    gen = torch.Generator(device="cuda").manual_seed(E + tokens)
    layer, keep = _layer(nv, ctx, gen, d, 64, E, k, 8, True, gated, kind, scales=tokens == 16)
    n = lambda *s: torch.empty(s, device="cuda").normal_(0.0, 1.0, generator=gen)
    x, delta = n(tokens, d).to(ctx.dtype), n(tokens, d).to(ctx.dtype)
    weight = (1.0 + 0.1 * n(d)).to(torch.bfloat16).view(torch.int16)
    for one, two in zip(*_both(nv, ctx, layer, x, delta, weight)):
        assert torch.equal(one.view(torch.uint8), two.view(torch.uint8))
    ctx.close()


def test_one_launch_replayed(nv):
    print("router and work list, replayed", flush=True)
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(3)
    layer, keep = _layer(nv, ctx, gen, 1024, 256, 64, 8, 8, True, True)
    x = torch.empty((24, 1024), device="cuda").normal_(0.0, 1.0, generator=gen).to(torch.bfloat16)
    moe, y = nv.MoE(ctx, 8), torch.empty_like(x)
    want = moe.decode_layer(layer, x).clone()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
        moe.decode_layer(layer, x, y)
    for turn in range(4):
        y.zero_()
        graph.replay()
        assert torch.equal(moe.decode_layer(layer, x[:1 + 7 * turn]), want[:1 + 7 * turn]) or turn == 0
        torch.cuda.synchronize()
        assert torch.equal(y, want), turn
    ctx.close()
