"""The MoE block of one token in one launch against the same block in three (which an output in place of the input takes): the same bits, whatever
the shape, with waits that end at once too, replayed, and behind launches of other sizes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nv():
    import nvmai_amd
    return nvmai_amd


def _layer(nv, ctx, gen, d, f, E, k, bits, shared, gated, kind=16, scales=False):
    n = lambda *s, std=0.05: torch.empty(s, device="cuda").normal_(0.0, std, generator=gen).to(torch.bfloat16)
    _, stride = nv.expert_offsets(d, f, bits)
    pool = torch.empty((E + 1, stride), dtype=torch.uint8, device="cuda")
    for e in range(E + 1):
        nv.pack_expert(ctx, n(f, d), n(f, d), n(d, f), bits, pool[e])
    keep = [pool]

    def rows(count, kind):
        if kind == 16:
            keep.append(n(count, d).view(torch.int16))
            return nv.rows_desc(16, keep[-1])
        keep.append(nv.quantize_affine(ctx, n(count, d), kind))
        return nv.rows_desc(kind, *keep[-1])
    router, gate = rows(E, kind), rows(1, 8) if gated else None
    u = lambda count: torch.empty(count, device="cuda").uniform_(0.5, 1.5, generator=gen).to(torch.bfloat16).view(torch.int16)
    more = dict(eff_scale=u(d), per_expert_scale=u(E)) if scales else {}
    keep += list(more.values())
    layer = nv.moe_layer_desc(d, f, E, k, bits, router, pool[:E], pool[E] if shared else None, gate, **more)
    return layer, keep


def _both(nv, ctx, layer, x, stats=True):
    """(output, experts, weights, statistics) in one launch, then in three."""
    moe, out = nv.MoE(ctx, layer.bits), []
    for in_place in (False, True):
        src = x.clone()
        s = torch.zeros(2, dtype=torch.int32, device="cuda")
        y, idx, w = moe.decode_layer(layer, src, src if in_place else torch.empty_like(src), want_routes=True, stats=s)
        torch.cuda.synchronize()
        out.append((y.clone(), idx.clone(), w.clone(), s.clone()))
    return out


@pytest.mark.parametrize("act", ["ACT_BF16", "ACT_FP16"])
@pytest.mark.parametrize("looks", [1 << 14, 0])
# hidden 2048 at 4 and 8 bits, 1024 at 8; rows of the down projection of 16 and 32 pieces; one expert, a lane's share of four or eight scores, its edges
@pytest.mark.parametrize("bits,d,f,E,k,shared,gated,kind,scales", [
    (4, 2048, 512, 256, 8, True, True, 16, False), (8, 2048, 256, 40, 8, True, True, 16, True), (8, 1024, 512, 257, 11, True, False, 8, False),
    (4, 2048, 1024, 9, 8, False, False, 4, False), (8, 2048, 256, 1, 1, True, True, 16, False), (8, 1024, 256, 255, 12, False, False, 16, True),
    (4, 2048, 512, 5, 3, True, True, 16, False)])
def test_one_launch_equals_three(nv, act, looks, bits, d, f, E, k, shared, gated, kind, scales):
    print("one launch", act, looks, bits, d, f, E, k, flush=True)
    ctx = nv.Context(0, getattr(nv, act))
    assert nv.lib.nvmai_hip_ctx_wait_limit(ctx.handle, looks) == 0
    gen = torch.Generator(device="cuda").manual_seed(E + k)
    layer, keep = _layer(nv, ctx, gen, d, f, E, k, bits, shared, gated, kind, scales)
    for row in range(3):
        x = torch.empty((1, d), device="cuda").normal_(0.0, 1.0, generator=gen).to(ctx.dtype)
        if row == 2:
            x[0, ::3] = 0.0
        for one, three in zip(*_both(nv, ctx, layer, x)):
            assert torch.equal(one.view(torch.uint8), three.view(torch.uint8))
    ctx.close()


def test_one_launch_behind_launches_of_other_sizes_and_replayed(nv):
    # the words' numbers go on together whatever the grids, in eager calls and in replays
    print("one launch, replayed", flush=True)
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(1)
    layers = [_layer(nv, ctx, gen, *a) for a in ((2048, 512, 24, 8, 4, True, True), (1024, 512, 300, 4, 8, False, False), (2048, 256, 3, 2, 8, True, False))]
    xs = [torch.empty((1, l.d), device="cuda").normal_(0.0, 1.0, generator=gen).to(torch.bfloat16) for l, _ in layers]
    ys = [torch.empty_like(x) for x in xs]
    want = [_both(nv, ctx, l, x)[1][0] for (l, _), x in zip(layers, xs)]
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            for (l, _), x, y in zip(layers, xs, ys):
                nv.MoE(ctx, l.bits).decode_layer(l, x, y)
    for turn in range(5):
        for y in ys:
            y.zero_()
        graph.replay()
        for (l, _), x, w in zip(layers[turn % 3:], xs[turn % 3:], want[turn % 3:]):
            assert torch.equal(nv.MoE(ctx, l.bits).decode_layer(l, x), w)
        torch.cuda.synchronize()
        for y, w in zip(ys, want):
            assert torch.equal(y, w), turn
    ctx.close()


def test_one_launch_with_scores_that_are_not_numbers(nv):
    # rows of scores with NaN and infinities, on the selection's other path; a NaN anywhere reaches the sums
    print("one launch, NaN", flush=True)
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(2)
    for E in (70, 300):
        layer, keep = _layer(nv, ctx, gen, 1024, 256, E, 8, 8, True, True)
        router = keep[1].view(torch.bfloat16)
        router[::7, 0], router[::11, 1], router[3, :] = float("nan"), float("inf"), 0.0
        for at in ((), (0,), (1,), (0, 1)):
            x = torch.zeros((1, 1024), device="cuda", dtype=torch.bfloat16)
            x[0, 5:9] = torch.tensor([1.0, -2.0, 0.5, 3.0], device="cuda").to(torch.bfloat16)
            for a in at:
                x[0, a] = 1.0
            one, three = _both(nv, ctx, layer, x)
            assert torch.equal(one[1], three[1]) and torch.equal(one[2].view(torch.int16), three[2].view(torch.int16)), (E, at)
            assert torch.equal(torch.isnan(one[0]), torch.isnan(three[0]))
    ctx.close()


@pytest.mark.parametrize("looks", [1 << 14, 0])
def test_output_in_place_of_the_prologues_rows(nv, looks):
    # y over normed or hidden_out takes three launches: the rows of separate buffers, y last
    print("one launch, y over the prologue's rows", looks, flush=True)
    ctx = nv.Context(0, nv.ACT_BF16)
    assert nv.lib.nvmai_hip_ctx_wait_limit(ctx.handle, looks) == 0
    gen = torch.Generator(device="cuda").manual_seed(4)
    row = lambda: torch.empty((1, 2048), device="cuda").normal_(0.0, 1.0, generator=gen).to(torch.bfloat16)
    layer, keep = _layer(nv, ctx, gen, 2048, 512, 64, 8, 4, True, True)
    moe, hidden, delta, weight = nv.MoE(ctx, 4), row(), row(), row()[0]
    h, normed, y = row(), row(), row()
    moe.decode_layer_prenorm(layer, hidden, delta, weight, h, normed, y)
    h2, both = row(), row()
    moe.decode_layer_prenorm(layer, hidden, delta, weight, h2, both, both)
    assert torch.equal(h2, h) and torch.equal(both, y)
    n2, both = row(), row()
    moe.decode_layer_prenorm(layer, hidden, delta, weight, both, n2, both)
    assert torch.equal(n2, normed) and torch.equal(both, y)
    ctx.close()


def test_time_is_booked_under_the_launches_that_are_made(nv):
    # the one launch under a tag of its own; its refusal (an output in place of the input, more tokens) books nothing
    print("one launch, spans", flush=True)
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(5)
    layer, keep = _layer(nv, ctx, gen, 2048, 512, 16, 8, 4, True, True)
    moe = nv.MoE(ctx, 4)
    tags = (nv.PROF_MOE_ONE, nv.PROF_ROUTER, nv.PROF_PHASE1, nv.PROF_PHASE2)
    for tokens, in_place, want in ((1, False, (1, 0, 0, 0)), (1, True, (0, 1, 1, 1)), (2, False, (0, 1, 1, 1)), (4, False, (0, 1, 1, 1))):
        x = torch.zeros((tokens, 2048), dtype=torch.bfloat16, device="cuda")
        ctx.profile_enable(True)
        moe.decode_layer(layer, x, x if in_place else torch.empty_like(x))
        ctx.profile_enable(False)
        assert tuple(ctx.profile_read(tag)[1] for tag in tags) == want, (tokens, in_place)
    ctx.close()


def test_statistics_where_scores_are_not_numbers(nv):
    # experts are chosen again where no score is left that is a number; one token's statistics name its slots and top_k either way, as the three launches do
    print("one launch, statistics", flush=True)
    ctx = nv.Context(0, nv.ACT_BF16)
    gen = torch.Generator(device="cuda").manual_seed(6)
    layer, keep = _layer(nv, ctx, gen, 1024, 256, 12, 8, 8, True, True)
    router = keep[1].view(torch.bfloat16)
    for bad in (0, 1, 5, 12):
        router[:] = 0.01
        router[12 - bad:] = float("nan")
        one, three = _both(nv, ctx, layer, torch.ones((1, 1024), device="cuda", dtype=torch.bfloat16))
        assert torch.equal(one[1], three[1]) and one[3].tolist() == three[3].tolist() == [9, 8], bad
    ctx.close()


@pytest.mark.parametrize("act", ["ACT_BF16", "ACT_FP16"])
@pytest.mark.parametrize("looks", [1 << 14, 0])
@pytest.mark.parametrize("with_delta", [False, True])
@pytest.mark.parametrize("bits,d,f,E,k,shared,gated,kind,scales", [
    (4, 2048, 512, 256, 8, True, True, 16, False), (8, 2048, 512, 30, 8, True, True, 16, True), (8, 1024, 256, 300, 4, False, False, 8, False)])
def test_with_the_norm_before_it(nv, act, looks, with_delta, bits, d, f, E, k, shared, gated, kind, scales):
    # the residual add and the norm inside the launch, as a layer of a decode step takes it, against the norm's own launch and the three
    print("one launch with its norm", act, looks, with_delta, bits, d, f, E, k, flush=True)
    ctx = nv.Context(0, getattr(nv, act))
    assert nv.lib.nvmai_hip_ctx_wait_limit(ctx.handle, looks) == 0
    gen = torch.Generator(device="cuda").manual_seed(E + d)
    layer, keep = _layer(nv, ctx, gen, d, f, E, k, bits, shared, gated, kind, scales)
    row = lambda: torch.empty((1, d), device="cuda").normal_(0.0, 1.0, generator=gen).to(ctx.dtype)
    weight, closing = (torch.empty(d, device="cuda").uniform_(0.5, 1.5, generator=gen).to(torch.bfloat16) for _ in range(2))
    moe, eps = nv.MoE(ctx, bits), 1e-5
    new = lambda: (torch.zeros((1, k), dtype=torch.int32, device="cuda"), torch.zeros((1, k), dtype=torch.float16, device="cuda"), torch.zeros(2, dtype=torch.int32, device="cuda"))
    for turn in range(3):
        hidden, delta = row(), row() if with_delta else None
        stream, stats = hidden.clone(), torch.zeros(2, dtype=torch.int32, device="cuda")
        zero = torch.zeros_like(hidden)
        normed = nv.ops.residual_add_rmsnorm(ctx, stream, delta if with_delta else zero, weight, eps=eps)
        want = normed.clone()
        want, want_idx, want_w = moe.decode_layer(layer, want, want, want_routes=True, stats=stats)
        h, n, y, (idx, w, s) = row(), row(), row(), new()
        moe.decode_layer_prenorm(layer, hidden, delta, weight, h, n, y, eps, idx, w, s)
        for got, wanted in zip((h, n, y, idx, w, s), (stream, normed, want, want_idx, want_w, stats)):
            assert torch.equal(got.view(torch.uint8), wanted.view(torch.uint8)), turn
        # with the end of the layer behind it
        ended = nv.ops.residual_add_rmsnorm(ctx, stream, want, closing, eps=eps)
        h, n, y, (idx, w, s), after = row(), row(), row(), new(), row()
        moe.decode_layer_norms(layer, hidden, delta, weight, h, n, y, closing, after, eps, idx, w, s)
        for got, wanted in zip((h, n, y, after, idx, w, s), (stream, normed, want, ended, want_idx, want_w, stats)):
            assert torch.equal(got.view(torch.uint8), wanted.view(torch.uint8)), turn
    ctx.close()
