"""Which entry point the calls of 32-bit contexts take: the one on planes where the rows are planes, and only there."""
import types

import pytest
import torch

from nvmai_amd import ops


@pytest.fixture
def calls(monkeypatch):
    """Names and arguments of the library's calls in place of the calls."""
    made = []

    class Lib:
        def __getattr__(self, name):
            return lambda *args: made.append((name, args)) or 0
    monkeypatch.setattr(ops, "lib", Lib())
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    return made


CTX = types.SimpleNamespace(act=ops.ACT_FP32, handle=None)


def test_rows_of_floats_by_heads_are_not_planes(calls):
    # [tokens, heads, values] floats, three heads among them
    w, norm = torch.zeros((8, 192), dtype=torch.bfloat16), torch.zeros(192, dtype=torch.bfloat16)
    x, flat, out = torch.zeros((6, 3, 64)), torch.zeros((6, 192)), torch.zeros((6, 3, 64))
    ops.dense_linear(CTX, w, x, y=torch.zeros((6, 8)))
    ops.dense_linear(CTX, w, flat, y=torch.zeros((6, 2, 4)))
    ops.norm_residual(CTX, flat, 192, next_norm=(norm, norm), out=out)
    ops.rms_residual(CTX, flat, 192, out=out)
    assert [name for name, _ in calls] == ["nvmai_hip_dense_linear", "nvmai_hip_dense_linear", "nvmai_hip_norm_residual", "nvmai_hip_rms_residual"]
    assert calls[0][1][4:7] == (x.data_ptr(), 192, 6) and calls[2][1][-5:-3] == (out.data_ptr(), 192)


def test_planes_take_the_calls_on_planes(calls):
    w, norm = torch.zeros((8, 64), dtype=torch.bfloat16), torch.zeros(64, dtype=torch.bfloat16)
    x, flat = torch.zeros((6, 3, 64), dtype=torch.bfloat16), torch.zeros((6, 64))
    by_heads = torch.zeros((6, 2, 4))
    ops.dense_linear(CTX, w, x, y=torch.zeros_like(x))
    ops.dense_linear(CTX, w, x, y=by_heads)
    ops.norm_residual(CTX, flat, 64, next_norm=(norm, norm), out=x)
    ops.rms_residual(CTX, flat, 64, out=x)
    assert [name for name, _ in calls] == ["nvmai_hip_dense_linear_planes"] * 2 + ["nvmai_hip_norm_residual_planes", "nvmai_hip_rms_residual_planes"]
    assert calls[1][1][8:12] == (by_heads.data_ptr(), 8, None, 0)


def test_a_product_of_planes_has_one_output_and_rows_of_the_matrix(calls):
    w, x, y = torch.zeros((8, 64), dtype=torch.bfloat16), torch.zeros((6, 3, 64), dtype=torch.bfloat16), torch.zeros((6, 8))
    with pytest.raises(AssertionError):
        ops.dense_linear(CTX, w, x, y=y, y_f32=torch.zeros((6, 8)))
    with pytest.raises(AssertionError):
        ops.dense_linear(CTX, w, torch.zeros((6, 3, 128), dtype=torch.bfloat16), y=y)
    assert not calls
    ops.dense_linear(CTX, w, x, y_f32=y)
    assert calls[0][1][8] == y.data_ptr()
