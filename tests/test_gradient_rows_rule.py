"""The rule that runs gradient rows one or two a workgroup (csrc/nrc_grad_rows.hpp, host code): its
level-by-level dealing against a workgroup-by-workgroup one, and its choice on launches of both kinds."""
import ctypes as C
import os
import random
import subprocess

import pytest

import grad_rows

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
B = 16384


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rows")
    src = d / "rows.cpp"
    src.write_text('#include "nrc_grad_rows.hpp"\n'
                   'extern "C" bool pairs(const nrc::GradRows *r, unsigned n, unsigned cus) { return nrc::grad_rows_in_pairs<16>(r, n, cus); }\n'
                   'extern "C" unsigned end(const nrc::GradRows *r, unsigned n, unsigned cus, unsigned g, unsigned b, unsigned c) {\n'
                   '  return nrc::grad_launch_end<16>(r, n, cus, g, b, c); }\n')
    so = d / "rows.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared",
                    "-fPIC", "-I", os.path.join(ROOT, "vknrc_amd", "csrc"), str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.pairs.restype = C.c_bool

    def items(rows):
        return (C.c_uint32 * (2 * len(rows)))(*[x for r in rows for x in r])

    return dict(pairs=lambda rows, cus=256: lib.pairs(items(rows), len(rows), cus),
                end=lambda rows, cus, *a: lib.end(items(rows), len(rows), cus, *a))


def test_levels_deal_as_single_workgroups_do(rule):
    rng = random.Random(5)
    for _ in range(300):
        rows = [(rng.choice([1, 2, 63, 64, 65, 128, 255, 256, 257, 700, 1024, rng.randint(1, 1024)]), rng.randint(1, 16))
                for _ in range(rng.randint(1, 16))]
        cus = rng.choice([1, 2, 255, 256, 304, 1000])
        args = (rng.randint(1, 2), rng.randint(0, 12), rng.randint(1, 9))
        assert rule["end"](rows, cus, *args) == grad_rows.launch_end(rows, cus, *args), (rows, cus, args)
        sizes = [(r * c * 64, c) for r, c in rows]
        assert rule["pairs"]([grad_rows.rows_of(*s) for s in sizes]) == grad_rows.in_pairs(sizes)


def test_rows_of_one_length(rule):
    # pairs where they save a round in three, whatever the length: (rows, in pairs)
    for chunks in (2, 3, 4, 8, 12, 16):
        for rows, want in ((1, False), (256, False), (257, True), (288, True), (512, True), (528, False), (640, False),
                           (768, False), (769, True), (1024, True)):
            assert rule["pairs"]([(rows, chunks)]) == want, (rows, chunks)


# launches of several lengths, where single rows took 0.63 to 0.96 of the time of pairs: a count of rows and
# pairs alone would pair them, since 2 ceil(rows / CUs) against ceil(pairs / CUs) says that this saves rounds
@pytest.mark.parametrize("sizes", [
    [(B, 8), (B, 1)], [(B, 1), (B, 8)], [(B, 8)] + [(B, 1)] * 3, [(B, 8)] + [(B, 1)] * 5, [(B, 8)] * 2 + [(B, 1)],
    [(B, 8)] * 4 + [(B, 1)], [(B, 8)] * 7 + [(B, 1)], [(B, 1)] * 2 + [(B, 8)] * 6, [(B, 8)] * 8 + [(4096, 1)],
    [(B, 2), (B, 1)], [(B, 16)] + [(B, 2)] * 6, [(B, 16)] * 9 + [(B, 8)] * 6, [(B, 1)] * 6 + [(B, 4)] * 2])
def test_rows_of_several_lengths_that_pairs_would_slow_down(rule, sizes):
    assert not rule["pairs"]([grad_rows.rows_of(*s) for s in sizes])


# and launches of several lengths where pairs took 0.75 to 0.96 of the time
@pytest.mark.parametrize("sizes", [
    [(64, 2), (B, 1)], [(B, 2)] + [(B, 1)] * 3, [(B, 2)] * 3 + [(B, 1)], [(B, 4)] * 8 + [(B, 1)], [(B, 8)] * 4 + [(B, 1)] * 8,
    [(B, 8)] * 8 + [(B, 1)] * 4, [(B, 4)] * 8 + [(B, 3)] * 3, [(B, 3)] * 3 + [(B, 4)] * 8,
    [(B, 8), (8192, 8), (4096, 8), (B, 8)] * 4])
def test_rows_of_several_lengths_that_pairs_speed_up(rule, sizes):
    assert rule["pairs"]([grad_rows.rows_of(*s) for s in sizes])
