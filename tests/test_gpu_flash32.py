"""The 32-bit attention of prompts, sixteen queries to a block, at the edges of its tiles: portions off its sixteen rows, windows that
begin inside a tile, rings that have wrapped, kept first tokens."""
import numpy as np
import pytest

from gpu_util import say
from test_gpu_kemuzen_ops import Window, bar, close
from test_gpu_pakirax_ops import Latent, check_latent

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,keep", [(1, 0), (15, 3), (16, 16), (17, 20), (40, 0), (100, 65)])
@pytest.mark.parametrize("shape,softcap,alibi", [((8, 2, 128, 128), 0.0, True), ((3, 1, 40, 80), 9.0, False), ((2, 2, 64, 16), 0.0, False)])
def test_window_portions_in_a_ring_that_wraps(shape, softcap, alibi, size, keep):
    import nvmai_amd as nv
    say("32-bit window flash", shape, size, keep)
    flash, plain = (Window("float32", *shape, size, keep, softcap, alibi, True, capacity=size + 49) for _ in range(2))
    at = 0
    for n in (16, 17, 50, 31, 33, 16, 48):
        data = flash.rows(at + 1, n)
        want = plain.run(data, nv.row_map(0, at), nv.WINDOW_PLAIN)
        close(flash.run(data, nv.row_map(0, at)), want, bar("float32"), "%d rows at %d" % (n, at))
        at += n


@pytest.mark.parametrize("window", [1, 15, 16, 17, 33, 0])
@pytest.mark.parametrize("heads,nope,rot,vdim", [(8, 128, 64, 128), (3, 16, 16, 80), (1, 112, 48, 64)])
def test_latent_portions_and_windows(heads, nope, rot, vdim, window):
    import nvmai_amd as nv
    say("32-bit latent flash", heads, nope, rot, vdim, window)
    ctx = nv.Context(0, nv.ACT_FP32)
    L = Latent(ctx, np.random.default_rng(window + heads), heads, nope, rot, vdim, 64, window, 150)
    check_latent(ctx, L, L.run([32, 33, 47, 38], 0))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("size,keep", [(None, 0), (17, 3), (40, 20)])
@pytest.mark.parametrize("shape", [(4, 2, 128, 128), (3, 1, 40, 80), (2, 2, 64, 16)])
def test_window_values_that_are_not_numbers_stay_with_the_queries_that_see_them(shape, size, keep, bad):
    """A key's value in one dim, at the edges of a tile, in the kept tokens and behind them: as in the plain form."""
    import nvmai_amd as nv
    n = 75
    for j in (0, 2, 15, 16, 21, 47, 73):
        flash, plain = (Window("float32", *shape, size, keep, 0.0, True, True, capacity=128) for _ in range(2))
        data = flash.rows(j, n, 1.0)
        data[2][j, 0, 1] = bad
        say("32-bit window flash, not numbers", shape, size, keep, j, bad)
        got, want = flash.run(data, nv.row_map(0, 0)), plain.run(data, nv.row_map(0, 0), nv.WINDOW_PLAIN)
        assert np.isnan(want).any() or np.isinf(want).any()
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        fine = np.isfinite(want)
        assert fine[:j].all() and np.abs(got[fine] - want[fine]).max() < bar("float32") * np.abs(want[fine]).max()


@pytest.mark.parametrize("window", [17, 0])
@pytest.mark.parametrize("heads,nope,rot,vdim", [(2, 128, 64, 128), (3, 16, 16, 80), (1, 112, 48, 64)])
def test_latent_rows_that_are_not_numbers_stay_with_the_queries_that_see_them(heads, nope, rot, vdim, window):
    import nvmai_amd as nv
    ctx, n = nv.Context(0, nv.ACT_FP32), 75
    L = Latent(ctx, np.random.default_rng(heads), heads, nope, rot, vdim, 64, window, n)
    want = L.run([n], nv.LATENT_EXPANDED)
    for j in (0, 15, 16, 40, 73):
        say("32-bit latent flash, not numbers", heads, nope, rot, vdim, window, j)
        keep = L.proj[j].clone()
        L.proj[j, L.qc:L.qc + 64] = float("nan")
        got = L.run([n], nv.LATENT_EXPANDED)
        L.proj[j] = keep
        sees = np.array([j <= i and (window == 0 or i - j < window) for i in range(n)])
        assert np.isnan(got[sees]).all() and np.isfinite(got[~sees]).all()
        assert (np.abs(got - want)[~sees] < 2e-6 * np.abs(want).max()).all()


def test_a_captured_latent_prompt_runs_without_room_for_planes():
    """A workspace that holds the keys and values (3.5 MB) but not the planes of their products (1 MB more): recorded without them."""
    import torch

    import nvmai_amd as nv
    say("captured 32-bit latent prompt")
    ctx, n = nv.Context(0, nv.ACT_FP32), 300
    L = Latent(ctx, np.random.default_rng(5), 8, 128, 64, 128, 512, 0, n)
    want = L.run([n], nv.LATENT_EXPANDED)
    small = nv.Context(0, nv.ACT_FP32)
    small.reserve(4 << 20)
    op = nv.LatentAttention(small, L.heads, L.nope, L.rot, L.vdim, L.rank, L.count, L.scale, L.window, L.rotary, L.base, L.eps)
    q, gate = L.q.clone(), L.proj[:, L.qc + L.rank + L.rot:]
    y = torch.zeros((n, L.heads * L.vdim), device="cuda")
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            op.encode(q, gate, L.uk, L.uv, L.cache, nv.row_map(0, 0), y, nv.LATENT_EXPANDED)
    for _ in range(3):
        q.copy_(L.q)                                 # the call rotates it in place
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.abs(y.double().cpu().numpy() - want).max() < 2e-5 * np.abs(want).max()
