"""The q/k/v epilogue of heads of 256 in pieces of 8 bytes, of many tokens (a block each) and of few (a block for four heads), against rows at 2-byte boundaries, which go
value by value: the same bits, in rows and in the cache."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["ACT_BF16", "ACT_FP16"])
# heads that end a round of the waves and that do not; rotated parts of less than a wave, of a wave and of the whole head; values normed or not
@pytest.mark.parametrize("heads,kv,rotary,bits,v_norm", [(16, 2, 64, 8, 0), (5, 2, 6, 4, 1), (3, 3, 256, 8, 0), (1, 1, 130, 4, 0), (2, 1, 0, 8, 1)])
def test_many_tokens(act, heads, kv, rotary, bits, v_norm):
    import nvmai_amd as nv
    from nvmai_amd._lib import check
    print("q/k/v epilogue", act, heads, kv, rotary, bits, flush=True)
    ctx, T, hd = nv.Context(0, getattr(nv, act)), 1027, 256
    gen = torch.Generator(device="cuda").manual_seed(heads)
    n = lambda *s: torch.empty(s, device="cuda").normal_(0.0, 1.0, generator=gen)
    width = heads * 2 * hd + 2 * kv * hd
    rows = n(T, width).to(ctx.dtype)
    qw, kw = ((1.0 + 0.1 * n(hd)).to(torch.bfloat16).view(torch.int16) for _ in range(2))
    positions = torch.randint(0, 100000, (T,), device="cuda", dtype=torch.int32, generator=gen)
    out = []
    for step, off in ((T, 0), (100, 0), (T, 1)):
        proj = torch.zeros(T * width + off, dtype=ctx.dtype, device="cuda")[off:].view(T, width)
        proj.copy_(rows)
        q, gate = (torch.zeros((T, heads * hd), dtype=ctx.dtype, device="cuda") for _ in range(2))
        k, v = (torch.zeros((T, kv * hd), dtype=ctx.dtype, device="cuda") for _ in range(2))
        caches = [nv.ops.KVCache(1, T, kv * hd, bits) for _ in range(2)]
        for t in range(0, T, step):
            views = [c.view(0, t) for c in caches]
            at = lambda x: x[t:].data_ptr()
            check(nv.lib.nvmai_hip_attn_qkv_epilogue_kv(ctx.handle, nv.ops._stream(), at(proj), width, 1, qw.data_ptr(), kw.data_ptr(), at(q), at(gate), at(k), at(v),
                                                        kv * hd, C.byref(views[0]), C.byref(views[1]), min(step, T - t), heads, kv, hd, rotary, v_norm,
                                                        at(positions), 0, 1e7, 1e-6), "epilogue")
        torch.cuda.synchronize()
        out.append([x.view(torch.uint8) for x in (q, gate, k, v, caches[0].rows, caches[1].rows)])
    for many, few, single in zip(*out):
        assert torch.equal(many, few) and torch.equal(many, single)
    ctx.close()
