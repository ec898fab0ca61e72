"""Which grids run the compile-time planned Z pass: those whose 32-bit byte
offsets cannot wrap. Thread t of a column addresses plane t of A2 (a plane is
Gy rows of whole 128-byte lines, and one line more) and relies on the buffer's
range, which ends below 4 GiB, to drop what it does not own; a component of the
tensor's octant is one buffer. Both sides of the limit for every planned length,
in both precisions; no GPU is used."""
import ctypes
import os
import re

import pytest

import dda_amd as D

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIMIT = 1 << 32


def _plans():
    """{(length, precision): threads per column}: the general plans as
    plan_list.hpp gives them, the tuned ones at their narrowest (8 points per
    thread, 12 at 48, 96 and 192)."""
    text = open(os.path.join(ROOT, "dda_amd", "csrc", "plan_list.hpp")).read()
    out = {}
    for n, fp32, fp64 in re.findall(r"X\((\d+), \(([\d, ]+)\), \(([\d, ]+)\)\)", text):
        for prec, radices in ((32, fp32), (64, fp64)):
            out[int(n), prec] = int(n) // min(int(r) for r in radices.split(","))
    for n in (32, 48, 64, 96, 128, 192, 256, 512, 1024):
        for prec in (32, 64):
            out[n, prec] = n // (12 if n % 3 == 0 else 8)
    return out


def _threads(grid, precision):
    return D.lib().dda_z_pass_threads((ctypes.c_uint32 * 3)(*grid), precision)


def _fits(gx, gy, gz, precision, threads):
    csz = precision // 4
    line = 128 // csz
    plane = gy * (-(-gx // line) * line) + line
    octant = (gx // 2 + 1) * (gy // 2 + 1) * (gz // 2 + 1)
    return octant * csz < LIMIT and threads * plane * csz < LIMIT


def test_every_length_has_a_plan():
    assert len(_plans()) == 2 * (66 + 9)


# grids whose last thread's offset passes 4 GiB though an eighth of their planes does not
@pytest.mark.parametrize("grid", [(1350, 2016, 500), (900, 3000, 500)])
def test_wide_planes_of_a_three_stage_plan(grid):
    assert not _fits(*grid, 64, 100) and _fits(*grid, 64, 500 // 8 + 1)
    assert _threads(grid, 64) == 0


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("gx", [8, 90, 672, 1350])
def test_z_pass_up_to_its_offsets(gx, precision):
    seen = set()
    for (n, prec), threads in _plans().items():
        if prec != precision:
            continue
        # the largest Gy that fits, by bisection; then around it and well inside
        lo, hi = 2, 1 << 26
        while hi - lo > 2:
            mid = (lo + hi) // 4 * 2
            lo, hi = (mid, hi) if _fits(gx, mid, n, precision, threads) else (lo, mid)
        for gy in (lo // 2, lo, lo + 2, lo + lo // 8, 2 * lo):
            want = _fits(gx, gy, n, precision, threads)
            got = _threads((gx, gy, n), precision)
            assert got == (threads if want else 0), (n, gy, threads)
            seen.add(want)
    assert seen == {True, False}
