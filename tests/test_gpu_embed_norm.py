"""A step's embedding rows and their norm in one launch."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("d,tokens", [(2048, 1), (2048, 5), (2048, 256), (2048, 257), (1024, 3)])
def test_embedding_rows_and_their_norm_have_the_bits_of_the_two_calls(act, bits, d, tokens):
    import nvmai_amd as nv
    from nvmai_amd import ops
    from nvmai_amd._lib import check, lib
    say("embedding rows and their norm", act, bits, d, tokens)
    ctx = nv.Context(0, nv.ACT_BF16 if act == "bf16" else nv.ACT_FP16)
    vocab = 300
    table = nv.quantize_affine(ctx, torch.randn((vocab, d), device="cuda").to(torch.bfloat16), bits)
    ids = torch.randint(0, vocab + 5, (tokens,), device="cuda", dtype=torch.int32)             # some past the table
    ids[0] = vocab - 1
    for weight in (torch.randn(d, device="cuda").to(torch.bfloat16).view(torch.int16), None):
        out, normed = (torch.full((tokens, d + 3), 7.0, device="cuda", dtype=ctx.dtype) for _ in range(2))
        check(lib.nvmai_hip_embed_lookup_rmsnorm(ctx.handle, torch.cuda.current_stream().cuda_stream, *(t.data_ptr() for t in table), bits, ids.data_ptr(), 0,
                                                 tokens, out.data_ptr(), d + 3, d, vocab, 1.25, None if weight is None else weight.data_ptr(),
                                                 normed.data_ptr(), d + 3, 1e-6), "embed_lookup_rmsnorm")
        want = ops.AffineQuantEmbeddingLookup(ctx, bits).encode(*table, ids, d, vocab, out_scale=1.25)
        norm = ops.RMSNorm(ctx)
        after = norm.encode_no_scale(want) if weight is None else norm.encode_bf16w(want, weight)
        assert torch.equal(out[:, :d], want) and torch.equal(normed[:, :d], after)
        assert bool((out[:, d:] == 7).all()) and bool((normed[:, d:] == 7).all())
