"""One row of each sequence through the recurrent scan with four taps: the same products in the same order as rows taken one after another."""
import pytest
import torch

pytestmark = pytest.mark.gpu
K_HEADS = 2


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("heads,dk,dv,sequences", [(4, 16, 16, 1), (4, 64, 64, 3), (16, 80, 128, 20), (2, 128, 64, 5), (64, 128, 64, 20), (2, 256, 32, 2), (2, 272, 16, 2)])
def test_single_rows_equal_rows_taken_in_runs(kind, heads, dk, dv, sequences):
    """Steps from position 0 over the end of the kept inputs; a run of several rows takes the general form, whose sums it must match bit for bit."""
    import nvmai_amd as nv
    ctx = nv.Context(0, nv.ACT_FP32)
    channels = 2 * K_HEADS * dk + heads * dv
    op = nv.HeadScan(ctx, kind, heads, K_HEADS, dk, dv, 4, 0, channels, channels + heads, dk ** -0.5)
    g = torch.Generator(device="cuda").manual_seed(dk + dv)
    randn = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    conv, bias = (randn(channels, 4) * 0.5).bfloat16(), randn(channels).bfloat16()
    a_log, dt_bias, skip = randn(heads).bfloat16(), randn(heads).bfloat16(), randn(heads).bfloat16()
    runs, steps = op.new_state(sequences), op.new_state(sequences)
    for x in runs + steps:
        x.normal_(generator=g)                          # what lies before position 0 and in other slots is not read
    runs[1].zero_(); steps[1].zero_()
    n = 41
    rows = randn(sequences, n, channels + 2 * heads)
    want, got = torch.empty(sequences, n, heads * dv, device="cuda"), torch.empty(n, sequences, heads * dv, device="cuda")
    weights = (conv, bias, a_log, dt_bias, skip)
    by_heads = lambda x: x.unflatten(1, (heads, dv)).transpose(0, 1)
    starts = [(7 * i) % 9 for i in range(sequences)]    # sequences stand at different positions
    for i in range(sequences):
        for at, count in ([(0, starts[i])] if starts[i] else []) + [(t, min(5, n - t)) for t in range(starts[i], n, 5)]:
            out = by_heads(want[i, at:at + count])
            op.encode(rows[i, at:at + count].contiguous(), *weights, *runs, nv.row_map(i, at), out, nv.SCAN_RECURRENT)
        if starts[i]:
            out = by_heads(got[:starts[i], i].contiguous())
            op.encode(rows[i, :starts[i]].contiguous(), *weights, *steps, nv.row_map(i, 0), out, nv.SCAN_RECURRENT)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    slots = list(range(sequences))[::-1]
    for t in range(n - max(starts)):
        at = [starts[i] + t for i in slots]
        x = torch.stack([rows[i, a] for i, a in zip(slots, at)])
        out = torch.empty(sequences, heads * dv, device="cuda")
        op.encode(x, *weights, *steps, nv.row_map(slots=i32(slots), positions=i32(at)), by_heads(out))
        assert torch.equal(out, torch.stack([want[i, a] for i, a in zip(slots, at)])), (kind, t)
