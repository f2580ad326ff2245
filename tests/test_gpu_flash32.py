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
