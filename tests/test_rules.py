"""Choices between forms of a call that sizes alone decide, compiled for the host."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nvmai_amd", "csrc")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """Answers of one expression of nvmai's rules for a list of values of its variables."""
    def answers(names, rows, expression):
        at = tmp_path_factory.mktemp("rules")
        (at / "rules.cpp").write_text('#include <stdio.h>\n#include "dense_plan.hpp"\n#include "rules.hpp"\nusing namespace nvmai;\nint main() {\n    unsigned %s;\n    while (scanf("%s", %s) == %d) printf("%%lld\\n", (long long)(%s));\n}\n'
                                      % (", ".join(names), "%u " * len(names), ", ".join("&" + n for n in names), len(names), expression))
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", str(at / "rules"), str(at / "rules.cpp")], check=True)
        out = subprocess.run([str(at / "rules")], input="\n".join(" ".join(str(v) for v in r) for r in rows), text=True, check=True, stdout=subprocess.PIPE).stdout
        return [int(v) for v in out.split()]
    return answers


def test_few_rows_take_the_matrix_cores_only_in_place_of_inputs_in_fp16(rule):
    cases = [(b, t, m, n) for b in (4, 8) for t in (3, 4) for m in (1, 8192, 32767, 32768, 248320) for n in range(64, 8193, 64)]
    for (bits, tokens, m, n), taken in zip(cases, rule(("bits", "tokens", "m", "n"), cases, "few_rows_mfma(bits, tokens, m, n)")):
        in_fp16 = n in ((512, 1024, 2048, 4096) if bits == 4 else (256, 512, 1024, 2048))
        assert not taken or (in_fp16 and m < 32768), (bits, tokens, m, n)
        if tokens == 4 and bits == 4 and in_fp16 and m < 32768:
            assert taken


def test_a_shared_expert_is_widened_only_where_both_products_take_its_rows(rule):
    cases = [(t, s, f) for t in (192, 131071, 131072, 140000, 262143, 262144, 600000) for s in (2048, 4096, 8192) for f in (512, 8192, 16384)]
    for (tokens, stride, f), fits, x, act in zip(cases, rule(("t", "s", "f"), cases, "expert_rows_fit(t, s, f)"), rule(("t", "s", "f"), cases, "dense_rows_fit(t, s)"),
                                                 rule(("t", "s", "f"), cases, "dense_rows_fit(t, f)")):
        assert x == (tokens * stride * 4 < 2 ** 32) and act == (tokens * f * 4 < 2 ** 32)
        assert fits == (x and act), (tokens, stride, f)
    assert rule(("t", "s", "f"), [(140000, 2048, 8192)], "expert_rows_fit(t, s, f)") == [0]      # taken, and refused after its first product


def test_a_shared_expert_takes_the_tiles_in_portions_whose_operands_have_offsets_of_32_bits(rule):
    cases = [(s, d, f, b) for d in (64, 1024, 2048, 8192) for s in (d, d + 64, 1 << 24, 1 << 31) for f in (64, 512, 8192, 131072, 1 << 24) for b in (4, 8)]
    for (s, d, f, b), most in zip(cases, rule(("s", "d", "f", "b"), cases, "expert_block_tokens(s, d, f, b)")):
        widest = max(s, d, f) * 2
        assert most * widest < 2 ** 32 and (most + 128) * widest > 2 ** 32 - 2 * widest or (most == 0 and d * f * b // 8 >= 2 ** 32), (s, d, f, b)
    # 270,000 tokens x 8192 had offsets that wrapped: outputs past token 262,143 were other tokens'
    assert rule(("s", "d", "f", "b"), [(2048, 2048, 8192, 4)], "expert_block_tokens(s, d, f, b)") == [262016]


PLAN = "dense_plan(n, rows, k, planes, 256, planes == 3 ? 3 : 5, cut)"


def test_which_tiles_the_cut_sizes_take(rule):
    """The sizes of the test on the device between them take every tile that may be cut, and the fewest and most parts."""
    from test_gpu_dense_cut import SHAPES
    names = ("rows", "n", "k", "planes", "cut")
    for planes, tiles, parts in ((1, {0, 1, 2}, {2, 12}), (3, {0, 1, 2}, {2, 12})):
        cases = [(*shape, planes, 1) for shape in SHAPES]
        got = list(zip(rule(names, cases, PLAN + ".head.tile"), rule(names, cases, PLAN + ".head.parts")))
        assert {t for t, p in got if p > 1} == tiles and parts <= {p for _, p in got}, got
        assert got[-1][1] == 1


def test_parts_have_a_unit_each_and_are_taken_where_they_save_time(rule):
    names = ("rows", "n", "k", "planes", "cut")
    cases = [(r, n, k, p, 1) for r in (5, 20, 65, 130, 300, 700, 1501, 2048, 4096) for n in (64, 250, 1024, 2048, 4160, 8256, 11264) for k in (64, 256, 1024, 2048, 8192, 32768)
             for p in (1, 3) if p == 3 or r > 64]
    value = lambda what, at=cases: rule(names, at, what)
    sizes = ((64, 64), (128, 64), (128, 128), (256, 128), (256, 256))
    whole = value(PLAN + ".ns", [(*c[:4], 0) for c in cases])
    for (rows, n, k, planes, _), first, tile, parts, tail, ns, uncut in zip(cases, value(PLAN + ".first"), value(PLAN + ".head.tile"), value(PLAN + ".head.parts"),
                                                                            value(PLAN + ".tail.parts"), value(PLAN + ".ns"), whole):
        bn, bm = sizes[tile]
        if first < n:                                # two launches: the first fills the units
            assert parts == 1 and (tail == 1 or rows <= 1024)
        if parts > 1:
            assert parts in (2, 3, 4, 6, 8, 12) and 2 * parts <= k // 64
            assert -(-n // bn) * -(-rows // bm) * parts <= 256 and ns <= uncut - (999 if rows > 1024 else 299)
    # what one sum per output is for: prompts of 4096 tokens in portions of 2048, and of 1501
    long = [(2048, n, 2048, 1, 1) for n in (2048, 4160, 8192, 8256)] + [(2048, 2048, 8192, 1, 1), (1501, 256, 2048, 1, 1), (1501, 2048, 5632, 1, 1), (1501, 11264, 2048, 1, 1)]
    assert set(value(PLAN + ".head.parts", long)) == {1}


def test_planes_that_products_share_lie_in_the_room_they_were_given(rule):
    # latents of an expanded attention: keys in steps of 64, beside what the room's own steps of 256 rows and its end at 32,768 leave
    cases = [(rows, k) for k in (*range(64, 1600, 64), 4096, 1 << 20, 1 << 26) for rows in (64, 4096, 14336, 14400, 14464, 14528, 21824, 21888, 32704, *range(32768, 400000, 64 * 13), 43648, 46656,
                                                                             48704, 87360, 349504)]
    names = ("rows", "k")
    at_once = rule(names, cases, "planes_at_once(rows, k)")
    for (rows, k), whole, room in zip(cases, at_once, rule(names, cases, "dense_plane_bytes(rows, k)")):
        assert room <= max(128 << 20, 6 * k) and (not whole or room == 6 * rows * k), (rows, k)
    # past 32,768 rows they had been taken as whole wherever 128 MB hold all of them
    answer = dict(zip(cases, at_once))
    assert answer[32768, 256] and not answer[32768 + 64 * 13, 64] and not answer[46656, 256] and not answer[14400, 1536] and answer[14336, 1536]


def test_rows_that_one_launch_of_the_expert_block_does_not_take(rule):
    # y in the place of any row that the launch reads or stores, whole or by its ends; x, delta, hidden_out and normed apart
    D, at = 2048, dict(x=1 << 20, delta=2 << 20, hidden_out=3 << 20, normed=4 << 20)
    names = ("x", "delta", "hidden", "normed", "y", "d")
    row = lambda a: "Rows16{%s, 4096}" % a
    overlaps = lambda cases: rule(names, cases, "block_overlaps(%s, %s, %s, %s, %s, 1, d)" % tuple(map(row, names[:5])))
    places = tuple(at.values())
    assert overlaps([(*places, p + o, D) for p in places for o in (0, 2 * D - 2, 2 - 2 * D)]) == [1] * 12
    assert overlaps([(*places, p + o, D) for p in places for o in (2 * D, -2 * D)]) == [0] * 8
    assert overlaps([(at["x"], 0, 0, 0, at["x"], D), (at["x"], 0, 0, 0, at["delta"], D)]) == [1, 0]
    # the prologue's rows over what it reads
    assert overlaps([(*(at[k] for k in order), 5 << 20, D) for order in (("x", "delta", "x", "normed"), ("x", "delta", "delta", "normed"), ("x", "delta", "hidden_out", "delta"))]) == [1] * 3
    # several tokens: by the ends of their rows
    several = "rows_overlap(Rows16{x, 4096}, Rows16{y, 4096}, 3, 2048)"
    assert rule(("x", "y"), [(1 << 20, (1 << 20) + 2 * 4096 * 2 + 4094), (1 << 20, (1 << 20) + 2 * 4096 * 2 + 4096)], several) == [1, 0]


def test_inputs_are_requested_first_for_whole_panels_of_nearly_whole_tiles(rule):
    cases = [(b, t, n) for b in (4, 8) for t in range(3, 33) for n in range(512, 8193, 512)]
    for (bits, tokens, n), first in zip(cases, rule(("bits", "tokens", "n"), cases, "gemv_inputs_first(bits, tokens, n)")):
        tile = 16 if tokens <= 16 else 32
        assert not first or (n % (2048 if tile == 16 else 1024) == 0 and tokens > tile // 2), (bits, tokens, n)
        assert first or tokens < tile or n % 2048, (bits, tokens, n)
