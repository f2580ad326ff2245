"""Tiles that several blocks share along k: every epilogue, uneven parts, ragged tiles, replays and other shapes in between."""
import pytest
import torch

from gpu_util import say
from test_gpu_dense_tiles import KINDS, check, epilogue, operands

pytestmark = pytest.mark.gpu


# Tiles of 64 x 64, 128 x 64 and 128 x 128 in 2 .. 12 parts (test_rules.py says which; the last but one in its second launch) and the last size in one; 37, 67 and 129 steps of 64 k leave parts of unequal
# length; one weight row and one token past a tile.  Sums as in the uncut form or of more, shorter chains: below 1e-6 of the largest value at these k (2^-24
# sqrt(k / 16 + 16) of a part), the bound is twice that, and 1e-6 for a GELU or SiLU by hardware exponentials.
SHAPES = [(65, 66, 2368), (129, 250, 4288), (300, 2048, 4288), (700, 2048, 4096), (400, 1000, 8192), (1200, 1000, 8256), (500, 1024, 4096), (70, 66, 16384), (700, 11264, 2048), (65, 64, 128)]


@pytest.mark.parametrize("act", ["bf16", "fp32"])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,n,k", SHAPES)
def test_shared_tiles(act, kind, rows, n, k):
    import nvmai_amd as nv
    say("dense, tiles cut along k", act, kind, rows, n, k)
    ctx = nv.Context(0, nv.ACT_FP32 if act == "fp32" else nv.ACT_BF16)
    w, x = operands(rows, n, k, ctx.dtype, rows + n + k)
    args, want = epilogue(kind, rows, n, x.double() @ w.double().T)
    y = torch.full((rows, want.shape[1] + 7 & ~1), 7.0, device="cuda")
    for _ in range(3):                                                # the tickets are zero again after each
        nv.dense_linear(ctx, w, x, y_f32=y, **args)
        check(y[:, :want.shape[1]], want, 3e-6)
        assert bool((y[:, want.shape[1]:] == 7).all())
        first = y.clone()
        nv.dense_linear(ctx, w[:, :64].contiguous(), x[:, :64].contiguous(), y_f32=y, **args)     # and other tiles in between
        y.copy_(first)
    nv.dense_linear(ctx, w, x, y_f32=y, **args)
    assert torch.equal(y, first)                                      # the order of the sums is fixed


@pytest.mark.parametrize("act", ["bf16", "fp32"])
def test_shared_tiles_in_a_graph(act):
    import nvmai_amd as nv
    say("dense, tiles cut along k, replayed", act)
    ctx = nv.Context(0, nv.ACT_FP32 if act == "fp32" else nv.ACT_BF16)
    rows, n, k = 130, 300, 4096
    w, x = operands(rows, n, k, ctx.dtype, 3)
    y, eager = torch.zeros((rows, n), device="cuda"), torch.zeros((rows, n), device="cuda")
    nv.dense_linear(ctx, w, x, y_f32=eager)
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            nv.dense_linear(ctx, w, x, y_f32=y)
            nv.dense_linear(ctx, w, x, y_f32=y)
    for _ in range(4):
        y.zero_()
        x.copy_(torch.randn_like(x))
        nv.dense_linear(ctx, w, x, y_f32=eager)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager)


def test_infinities_and_nan_in_one_part():
    """A part's sum that is not finite: what the whole sum is."""
    import nvmai_amd as nv
    say("dense, tiles cut along k, infinities")
    rows, n, k = 70, 66, 4096
    for act, dtype in ((nv.ACT_BF16, torch.bfloat16), (nv.ACT_FP32, torch.float32)):
        w, x = operands(rows, n, k, dtype, 5)
        x[3, 4000], x[5, 7], x[5, 4001], x[9, 2000] = float("inf"), float("inf"), float("-inf"), float("nan")
        w[:, [7, 4000, 4001]] = w[:, [7, 4000, 4001]].abs() + 0.01
        y = nv.dense_linear(nv.Context(0, act), w, x, y_f32=torch.empty((rows, n), device="cuda"))
        assert bool((y[3] == float("inf")).all()) and bool(y[5].isnan().all()) and bool(y[9].isnan().all())
        rest = [t for t in range(rows) if t not in (3, 5, 9)]
        check(y[rest], x[rest].double() @ w.double().T, 3e-6)
