"""The widths a contraction adds its weights in (csrc/widths.h), compiled with
g++ and checked against exact integers at the edges of the ranges: 32-bit staging
while all weights together stay below 2^31, packed tables below 2^32 (unit
weights: up to 2^32 - 1 nonzeros), 32-bit sums in LDS while 8,192 of the largest
weight do, and 64 bits for negative weights."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
B31, B32 = 1 << 31, 1 << 32


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("widths") / "widths_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "pennsylvaniagpugraphclustering_amd",
                                                                             "csrc"),
                           os.path.join(ROOT, "tests", "widths_check.cpp"), "-o", str(exe)])
    return str(exe)


def widths(exe, cases):
    inp = "\n".join(f"{n} {w} {s}" for n, w, s in cases)
    out = subprocess.run([exe], input=inp, capture_output=True, text=True, check=True).stdout.split("\n")
    return [tuple(int(x) for x in line.split()) for line in out if line]


def test_unit_weights(program):
    cases = [(0, 1, 0), (1, 1, 0), (B31 - 1, 1, 0), (B31, 1, 0), (B32 - 2, 1, 0), (B32 - 1, 1, 0), (B32, 1, 0),
             (5 * B32, 1, 0)]
    assert widths(program, cases) == [(1, 1, 1), (1, 1, 1), (1, 1, 1), (0, 1, 1), (0, 1, 1), (0, 1, 1), (0, 0, 1),
                                      (0, 0, 1)]


def test_edges_against_exact_integers(program):
    cases = []
    for nnz in (1, 2, 3, 1000, 31457, 8191, 8192, 8193, 1 << 20, 520768910, 4223269732):
        for bound in (B31, B32):
            for w in ((bound - 1) // nnz, (bound - 1) // nnz + 1):
                cases.append((nnz, max(w, 1), 0))
        for w in ((B32 - 1) // 8192, (B32 - 1) // 8192 + 1, B31 - 1, B31, B32, (1 << 63) - 1, (1 << 64) - 1, 1 << 63):
            cases.append((nnz, w, 0))
    for (nnz, w, _), got in zip(cases, widths(program, cases)):
        small = nnz * w < B31
        assert got == (small, nnz * w < B32, small or 8192 * w < B32), (nnz, w)


def test_known_small_sums(program):
    assert widths(program, [(1 << 30, 1 << 40, 1)]) == [(1, 1, 1)]
