"""The small-tile GEMM's workgroup -> tile map, run on the host: every tile of a grid is computed exactly once, also where the
number of workgroups times the divisor passes 2^32 and a 32-bit reciprocal alone is not exact."""
import os
import random
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "c_host", "tile_order_check.cpp")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("tile_order") / "tile_order_check")
    subprocess.check_call(["hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-std=c++17", SRC, "-o", exe])

    def run(grids):
        text = "".join(f"{n} {m} {tf} {tt}\n" for n, m, tf, tt in grids)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
        assert out[-1] == f"{len(grids)} grids"
        return out[:-1]
    return run


FORMS = ((128, 128), (128, 64), (64, 64))


def test_every_tile_of_small_grids(check):
    assert check([(n, m, *f) for n in range(1, 41) for m in range(1, 41) for f in FORMS]) == []


def test_every_tile_of_grids_beyond_a_32_bit_reciprocal(check):
    # grids on which the reciprocal alone is one too large for some workgroup, then others of that size
    grids = [(5, 30819, 128, 128), (33, 11503, 128, 128), (302, 3810, 128, 128), (1003, 2089, 128, 128)]
    rng = random.Random(3)
    while len(grids) < 60:
        n, m = rng.randrange(1, 4000), rng.randrange(2000, 40000)
        if n * m < 4_000_000 and n * m * m >= 1 << 32:
            grids.append((n, m, *rng.choice(FORMS)))
    assert check(grids) == []


def test_grids_of_more_tiles_than_one_row_of_workgroups_takes(check):
    """Fewer than 2^32 threads along a dimension: 4194304 workgroups of 768."""
    most = 1 << 22
    grids = [(most - 1, 1), (most, 1), (most + 1, 1), (1, most + 1), (5593752, 1), (11187503, 1), (2, 4194305), (3001, 2003)]
    assert check([(n, m, *f) for n, m in grids for f in FORMS]) == []


def test_every_tile_of_the_order_with_the_fewest_bytes(tmp_path):
    exe = str(tmp_path / "cheapest_order_check")
    subprocess.check_call(["hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-std=c++17", os.path.join(os.path.dirname(SRC), "cheapest_order_check.cpp"), "-o", exe])
    rng = random.Random(4)
    grids = [(n, m, *f) for n in range(1, 31) for m in range(1, 61) for f in FORMS] + [(10, 51, 128, 128), (5, 30819, 128, 128), (1003, 2089, 128, 128)]
    grids += [(rng.randrange(1, 300), rng.randrange(1, 3000), *rng.choice(FORMS)) for _ in range(200)]
    text = "".join(f"{n} {m} {tf} {tt}\n" for n, m, tf, tt in grids)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(out) == 1 and int(out[0].split()[0]) > 300, out
