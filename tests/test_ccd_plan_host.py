"""The block sums of a mass correction against the room allocated for them.

The final CCD pass leaves one block sum per 256 threads: a line takes 1, 32 or
64 lanes, so a block holds 256, 8 or 4 lines.  Before it, the unlisted lines'
sums take a block per 256 lines and segment.  lsmp_init sizes the buffer by
mass_sums(), which must cover every pass that ccd_plan() lets the launcher make:
of every line, and of any number of listed lines behind the unlisted ones."""
import ctypes as C
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CELLS = os.path.join(HERE, "host_cells")


@pytest.fixture(scope="module")
def plan():
    subprocess.run(["make", "-s", "-C", CELLS], check=True)
    L = C.CDLL(os.path.join(CELLS, "_build", "libccd_plan.so"))
    L.hc_ccd_plan.argtypes = [C.c_int, C.c_int, C.c_long, C.c_int, C.c_int, C.POINTER(C.c_long)]
    L.hc_hsum_blocks.argtypes = [C.c_int, C.c_long]
    L.hc_mass_sums.argtypes = [C.c_int] * 5
    L.hc_hsum_blocks.restype = L.hc_mass_sums.restype = C.c_long
    return L


def blocks(L, dim, n, lines, listed, esz):
    """Blocks of a final pass, from the lanes a line takes."""
    b = C.c_long()
    lanes = L.hc_ccd_plan(dim - 1, n, lines, listed, esz, C.byref(b))
    assert lanes in (1, 32, 64)
    if lanes > 1:
        assert lanes * 17 >= n + 4          # rows of a line in its lanes' registers
    per = 256 // lanes
    assert b.value == -(-lines // per)
    return b.value


def check(L, nx, ny, nz):
    dim = 3 if nz > 1 else 2
    n, lines = (nz, nx * ny) if dim == 3 else (ny, nx)
    seg = L.hc_hsum_segments(n)
    assert 1 <= seg <= 8
    unlisted = -(-lines // 256) * seg
    assert L.hc_hsum_blocks(n, lines) == unlisted
    for esz in (8, 4):
        room = L.hc_mass_sums(dim, nx, ny, nz, esz)
        assert blocks(L, dim, n, lines, 0, esz) <= room, (nx, ny, nz)
        for k in {0, 1, lines // 3, lines - 1, lines}:
            assert unlisted + blocks(L, dim, n, k, 1, esz) <= room, (nx, ny, nz, k)


LONG = [(4097, 541, 1), (8192, 1024, 1), (16384, 1024, 1), (40960, 1084, 1), (40961, 1084, 1), (40960, 1085, 1),
        (32, 600, 600), (20, 700, 700), (8, 600, 541), (4, 4, 600), (200, 200, 1084), (256, 256, 256)]


@pytest.mark.parametrize("grid", LONG, ids=lambda g: "x".join(map(str, g)))
def test_room_for_block_sums(plan, grid):
    check(plan, *grid)


def test_room_for_block_sums_drawn(plan):
    rng = random.Random(7)
    size = lambda top: int(4 * (top / 4) ** rng.random())
    for _ in range(20000):
        check(plan, size(60000), size(3000), 1)
        nx, ny = size(1500), size(1500)
        check(plan, nx, ny, size(min(3000, int(2e9 / (nx * ny)))))


# (direction, cells, bytes a value, lines): the side measured faster; one lane a line
# where many short lines, or lines whose lanes meet in LDS banks, cost more than they save
SIDES = [
    (0, 4, 8, 4096, True), (0, 4, 8, 810000, False), (0, 8, 8, 160000, False), (1, 8, 8, 40000, False),
    (2, 8, 4, 16384, False), (2, 24, 8, 5184, True), (2, 24, 8, 16384, False), (0, 24, 8, 16384, False),
    (1, 48, 8, 40000, False), (0, 80, 8, 160000, False), (0, 64, 4, 160000, True), (0, 128, 8, 810000, True),
    (1, 96, 8, 16384, True), (1, 96, 8, 40000, False), (1, 256, 8, 40000, True), (1, 256, 8, 65536, False),
    (0, 240, 8, 160000, False), (1, 240, 8, 29929, False), (1, 480, 8, 19881, False), (0, 500, 4, 160000, False),
    (0, 700, 8, 40000, False), (0, 700, 4, 40000, True), (1, 700, 8, 10000, True), (1, 700, 8, 19600, False),
    (1, 1000, 4, 19600, False), (0, 2000, 8, 10, False), (1, 1085, 8, 4096, False), (1, 1084, 8, 4096, True),
]


@pytest.mark.parametrize("d,n,esz,lines,wide", SIDES)
def test_lanes_a_line(plan, d, n, esz, lines, wide):
    b = C.c_long()
    assert (plan.hc_ccd_plan(d, n, lines, 0, esz, C.byref(b)) > 1) == wide
    # a list takes 32 or 64 lanes up to 1,084 cells
    assert (plan.hc_ccd_plan(d, n, lines, 1, esz, C.byref(b)) > 1) == (n <= 1084)
