"""The BF16 flash attention of prompts over many tiles: thousands of keys, windows that let a block's waves skip tiles, a last block with one
live wave, every size the kernels are built for, against the forms that load nothing straight into LDS."""
import numpy as np
import pytest

from gpu_util import say
from test_gpu_kemuzen_ops import Window, bar, close
from test_gpu_pakirax_ops import FORMS, Latent

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,size,keep", [(2049, None, 0), (4097, 700, 65), (2081, 64, 3), (4096, 1, 0)])
@pytest.mark.parametrize("shape", [(8, 2, 128, 128), (3, 1, 40, 80), (2, 1, 64, 64), (2, 2, 100, 48), (2, 1, 160, 144)])
def test_windowed(shape, n, size, keep):
    import nvmai_amd as nv
    for softcap, alibi in ((6.0, False), (0.0, True)):
        w = Window("bfloat16", *shape, size, keep, softcap, alibi, True, capacity=n + 63)
        data, more = w.rows(n, n), w.rows(n + 1, 33)
        say("windowed flash, many tiles", shape, n, size, keep, softcap)
        want = w.run(data, nv.row_map(0, 0), nv.WINDOW_PLAIN)
        close(w.run(data, nv.row_map(0, 0), nv.WINDOW_FLASH), want, bar("bfloat16"), "prompt")
        if size:
            want = w.run(more, nv.row_map(0, n), nv.WINDOW_PLAIN)
            close(w.run(more, nv.row_map(0, n), nv.WINDOW_FLASH), want, bar("bfloat16"), "33 rows behind it")


@pytest.mark.parametrize("n,window", [(2049, 0), (4097, 700), (2081, 64), (4096, 1)])
@pytest.mark.parametrize("heads,nope,rot,vdim,rank", [(8, 128, 64, 128, 128), (3, 16, 16, 80, 64), (2, 64, 32, 48, 64), (2, 48, 64, 128, 64),
                                                      (2, 128, 32, 64, 64), (1, 208, 48, 256, 64)])
def test_latent(heads, nope, rot, vdim, rank, n, window):
    import nvmai_amd as nv
    L = Latent(nv.Context(0, nv.ACT_BF16), np.random.default_rng(n + heads), heads, nope, rot, vdim, rank, window, n)
    say("latent flash, many tiles", heads, nope, rot, vdim, n, window)
    want = L.run([n], FORMS["absorbed"])
    for portions in ([n], [n - 33, 33]):
        got = L.run(portions, FORMS["expanded"])
        assert np.abs(got - want).max() < 2e-2 * np.abs(want).max(), portions


# rows and heads on either side of what each form of the launch is for (256 compute units): 64 queries per block up to 448 blocks, 128 by eight waves up
# to 256, by four beyond; waves and groups without a key, one tile, an odd number of tiles
@pytest.mark.parametrize("heads,n", [(16, 33), (16, 65), (16, 1792), (16, 1793), (16, 2048), (24, 1409), (43, 700)])
def test_forms_of_the_launch(heads, n):
    import nvmai_amd as nv
    for softcap, alibi, size in ((6.0, False, None), (0.0, True, 300)):
        w = Window("bfloat16", heads, 1, 128, 128, size, 4, softcap, alibi, True, capacity=n + 63)
        data = w.rows(n, n)
        say("windowed flash, forms", heads, n, softcap)
        close(w.run(data, nv.row_map(0, 0), nv.WINDOW_FLASH), w.run(data, nv.row_map(0, 0), nv.WINDOW_PLAIN), bar("bfloat16"), "prompt")
    L = Latent(nv.Context(0, nv.ACT_BF16), np.random.default_rng(n), heads, 128, 64, 128, 64, 500, n)
    say("latent flash, forms", heads, n)
    want = L.run([n], FORMS["absorbed"])
    got = L.run([n], FORMS["expanded"])
    assert np.abs(got - want).max() < 2e-2 * np.abs(want).max()
