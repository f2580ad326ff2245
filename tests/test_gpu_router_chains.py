"""The router's logits of many tokens against the kernel that takes few, or the oracle where that does not take the row: the
routing does not depend on how many tokens went in together, so the bits are the same."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import act_tensor, dev, gauss, round_act, say

pytestmark = pytest.mark.gpu


# rows and tokens off the tiles of 16, one to eleven chunks a lane, the scaled form, both splits of the chains (few and many tokens)
@pytest.mark.parametrize("act", [0, 1], ids=["bf16", "fp16"])
@pytest.mark.parametrize("experts,d,tokens,scaled", [(2, 256, 64, False), (100, 1280, 65, True), (129, 2816, 79, True), (256, 2048, 4111, False),
                                                     (33, 512, 5000, True)])
def test_logits_of_many_tokens_are_those_of_few(act, experts, d, tokens, scaled):
    import nvmai_amd as nv
    say("router chains", act, experts, d, tokens, scaled)
    ctx = nv.Context(0, act)
    rng = np.random.default_rng(d + tokens)
    w = O.round_bf16(gauss(rng, (experts, d), 0.02))
    x = round_act(gauss(rng, (tokens, d)), act)
    x[1] *= np.float32(2.0 ** -9)
    w[experts // 2, ::3] = 0.0
    host = round_act(x, act)
    x = act_tensor(host, ctx)
    bits = O.bf16_bits(rng.uniform(0.01, 0.04, d).astype(np.float32)) if scaled else None
    eff = dev(bits.view(np.int16)) if scaled else None
    desc, moe = nv.rows_desc(16, dev(O.bf16_bits(w).view(np.int16))), nv.MoE(ctx)
    k = min(8, experts)
    idx, wt, logits = moe.encode_router(desc, x, experts, d, k, eff, want_logits=True)
    for t in (0, 1, 17, tokens - 1) if d > 2048 else ():
        assert np.array_equal(logits[t].cpu().numpy().view(np.uint32), O.router_logits(16, O.bf16_bits(w), None, None, host[t], bits).view(np.uint32))
    for a in range(0, tokens, 1 + tokens // 8) if d <= 2048 else ():
        b = min(a + 40, tokens)
        i2, w2, l2 = moe.encode_router(desc, x[a:b], experts, d, k, eff, want_logits=True)
        assert torch.equal(logits[a:b].view(torch.int32), l2.view(torch.int32)) and torch.equal(idx[a:b], i2) and torch.equal(wt[a:b], w2)
    torch.cuda.synchronize()
    ctx.close()
