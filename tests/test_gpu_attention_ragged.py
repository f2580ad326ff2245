"""A ragged batch is dealt out over the device by the sequences' lengths: it gives what every sequence gives in a call of its own."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu

# lengths that fill the blocks unevenly: one sequence has nearly everything, all are equal, most are empty, tiny beside long, many of them
LENGTHS = [[70000, 1], [30000, 30000, 30000], [0, 0, 60007, 0], [1, 2, 3, 4, 5, 6, 7, 40000], [127, 128, 129, 255, 256, 257, 40000], [0, 0],
           [33 * i % 700 for i in range(64)], [900] * 33, [9000] + [33 * i for i in range(63)]]


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("lens", LENGTHS, ids=lambda v: "%dx%d" % (len(v), max(v)))
@pytest.mark.parametrize("heads", [(16, 2), (8, 8)], ids=["gqa", "mha"])
def test_dealt_out_by_length(bits, lens, heads):
    import nvmai_amd as nv
    say("ragged by length", bits, heads, lens[:8])
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(len(lens) + bits)
    (nq, nkv), B, cap = heads, len(lens), max(lens) + 3
    k, v = (nv.KVCache(B, cap, nkv * 256, bits) for _ in range(2))
    for c in (k, v):
        for b in range(B):
            nv.KVCacheQuantizer(ctx).encode(torch.randn((cap, nkv * 256), device="cuda", generator=gen).to(torch.bfloat16), nkv * 256, c.view(b), cap, nkv * 256)
    q = torch.randn((B, nq, 256), device="cuda", generator=gen).to(torch.bfloat16)
    att = nv.Attention(ctx)
    starts = [n // 3 if b % 2 else 0 for b, n in enumerate(lens)]
    one = lambda t: torch.tensor(t, dtype=torch.int32, device="cuda")
    for begin in (None, starts):
        out = att.encode_ragged(q, k, v, 256, nq, nkv, one(lens), cap, kv_starts=None if begin is None else one(begin))
        for b, n in enumerate(lens):
            if n == 0:
                assert not out[b].any()
                continue
            kb, vb = nv.KVCache(1, 1, nkv * 256, bits), nv.KVCache(1, 1, nkv * 256, bits)
            kb.rows, vb.rows = k.rows[b:b + 1], v.rows[b:b + 1]
            want = att.encode_full(q[b:b + 1], kb, vb, 256, nq, nkv, n, kv_start=0 if begin is None else begin[b])[0].float()
            # the same sums in chunks of another length: two roundings to BF16 apart
            assert float((out[b].float() - want).abs().max() / want.abs().max()) < 2 ** -7, b


@pytest.mark.parametrize("lens", [[40000] * 8, [16384] * 48, [8192] * 64, [8191] * 64, [50001] * 3], ids=lambda v: "%dx%d" % (len(v), v[0]))
@pytest.mark.parametrize("heads", [(16, 2), (8, 8)], ids=["gqa", "mha"])
def test_equal_lengths_are_cut_as_an_even_batch(lens, heads):
    """No chunk is longer than in the uniform split, and equal sequences get that split back: the bits of a call that knows the length."""
    import nvmai_amd as nv
    say("ragged with equal lengths", heads, len(lens), lens[0])
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(len(lens))
    (nq, nkv), B, n = heads, len(lens), lens[0]
    k, v = (nv.KVCache(B, n, nkv * 256, 8) for _ in range(2))
    rows = torch.randn((n, nkv * 256), device="cuda", generator=gen).to(torch.bfloat16)
    for c in (k, v):
        for b in range(B):
            nv.KVCacheQuantizer(ctx).encode(rows.roll(b + (c is v), 0), nkv * 256, c.view(b), n, nkv * 256)
    q = torch.randn((B, nq, 256), device="cuda", generator=gen).to(torch.bfloat16)
    att = nv.Attention(ctx)
    got = att.encode_ragged(q, k, v, 256, nq, nkv, torch.tensor(lens, dtype=torch.int32, device="cuda"), n)
    assert torch.equal(got, att.encode_full(q, k, v, 256, nq, nkv, n))
