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
    L.hc_ccd_plan.argtypes = [C.c_int, C.c_int, C.c_long, C.c_int, C.POINTER(C.c_long)]
    L.hc_hsum_blocks.argtypes = [C.c_int, C.c_long]
    L.hc_mass_sums.argtypes = [C.c_int] * 4
    L.hc_hsum_blocks.restype = L.hc_mass_sums.restype = C.c_long
    return L


def blocks(L, dim, n, lines, listed):
    """Blocks of a final pass, from the lanes a line takes."""
    b = C.c_long()
    lanes = L.hc_ccd_plan(dim - 1, n, lines, listed, C.byref(b))
    assert lanes in (1, 32, 64)
    if lanes > 1:
        assert lanes * 17 >= n + 4          # rows of a line in its lanes' registers
    per = 256 // lanes
    assert b.value == -(-lines // per)
    return b.value


def check(L, nx, ny, nz):
    dim = 3 if nz > 1 else 2
    n, lines = (nz, nx * ny) if dim == 3 else (ny, nx)
    room = L.hc_mass_sums(dim, nx, ny, nz)
    assert blocks(L, dim, n, lines, 0) <= room, (nx, ny, nz)
    seg = L.hc_hsum_segments(n)
    assert 1 <= seg <= 8
    unlisted = -(-lines // 256) * seg
    assert L.hc_hsum_blocks(n, lines) == unlisted
    for k in {0, 1, lines // 3, lines - 1, lines}:
        assert unlisted + blocks(L, dim, n, k, 1) <= room, (nx, ny, nz, k)


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
