"""The order in which the tile table walks the cells of a grid (csrc/brick.h),
compiled for the host and compared with a restatement in unbounded integers:
a permutation of the cells for small grids, and the same cell in the largest
grids a system may have (2^30 cells), where 32-bit products run out first."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "smoothedparticles.jl_amd", "csrc")


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    exe = tmp_path_factory.mktemp("brick") / "brick_order"
    src = os.path.join(ROOT, "tests", "brick_order.cpp")
    # (an overflow wraps, as it does on the device)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fwrapv", "-I", CSRC, src, "-o", str(exe)],
                   check=True)

    def run(L, first, stride, count):
        p = subprocess.run([str(exe), *map(str, (*L, first, stride, count))], capture_output=True,
                           text=True)
        assert p.returncode == 0, f"grid {L}: exit {p.returncode}"
        return [tuple(map(int, line.split())) for line in p.stdout.splitlines()]

    return run


def cell_at(L, r):
    """The cell at rank r: bricks of 4 x 4 x 4 (8 x 8 in one layer), cut to the
    grid, x fastest among the bricks and in each."""
    b = (4, 4, 4) if L[2] > 1 else (8, 8, 1)
    kz, r = divmod(r, b[2] * L[0] * L[1])
    hz = min(b[2], L[2] - kz * b[2])
    ky, r = divmod(r, b[1] * L[0] * hz)
    hy = min(b[1], L[1] - ky * b[1])
    kx, r = divmod(r, b[0] * hy * hz)
    wx = min(b[0], L[0] - kx * b[0])
    iz, r = divmod(r, wx * hy)
    iy, ix = divmod(r, wx)
    return kx * b[0] + ix + L[0] * (ky * b[1] + iy + L[1] * (kz * b[2] + iz))


@pytest.mark.parametrize("L", [(1, 1, 1), (1, 9, 1), (9, 1, 1), (8, 8, 1), (17, 11, 1), (3, 2, 5),
                               (1, 1, 7), (4, 4, 4), (6, 5, 2), (2, 7, 3), (13, 9, 6)])
def test_small_grids(order, L):
    n = L[0] * L[1] * L[2]
    got = order(L, 0, 1, n)
    assert got == [(r, cell_at(L, r)) for r in range(n)]
    assert sorted(c for _, c in got) == list(range(n))


@pytest.mark.parametrize("L", [(478000000, 1, 1), (500000000, 1, 1), (536870912, 1, 1),
                               (1 << 30, 1, 1), (1, 1 << 30, 1), (1, 1, 1 << 30),
                               (250000000, 1, 4), (1, 250000000, 4), (16384, 32767, 2),
                               (32768, 32768, 1), (1023, 1024, 1024), (1 << 28, 2, 2)])
def test_largest_grids(order, L):
    n = L[0] * L[1] * L[2]
    assert n <= 1 << 30
    stride = n // 997
    for first, step, count in ((0, stride, 997), (n - 300, 1, 300)):
        got = order(L, first, step, count)
        assert got == [(r, cell_at(L, r)) for r in range(first, first + step * count, step)]
