"""The ray kernels' dealing by pairs and blocks of tile rows (compiled for the host):
every tile of a detector exactly once at odd and even counts of tile rows, the
columns through the middle of the detector shared evenly among the 8 XCDs; and the
rules that choose them on both sides of their lines."""
import subprocess

import pytest

from newrecon_amd.build import CSRC, HIPCC

PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "ostr_internal.h"
using namespace ostr;
int main(int, char** argv) {
    const int n = atoi(argv[1]), ti = atoi(argv[2]), tj = atoi(argv[3]);
    const int lg = atoi(argv[4]);
    const int64_t grid = ray_grid(n, ti, tj, lg);
    std::vector<int> seen(n * ti * tj), load(8);
    int64_t all = 0, most = 0;
    for (int64_t w = 0; w < grid; ++w) {
        RayTile t;
        if (!ray_tile((int)w, n, ti, tj, t, lg)) continue;
        if (t.slot < 0 || t.slot >= n || t.ti < 0 || t.ti >= ti || t.tj < 0 || t.tj >= tj) return 1;
        ++seen[(t.slot * ti + t.ti) * tj + t.tj];
        if (t.ti >= ti / 4 && t.ti < ti - ti / 4) ++load[w % 8], ++all;
    }
    for (int s : seen)
        if (s != 1) return 2;
    for (int x : load) most = std::max<int64_t>(most, x);
    printf("%lld %lld %lld %d %d %d %d\\n", (long long)grid, (long long)most, (long long)all,
           ray_by_pairs(16, n, ti, tj), ray_by_pairs(17, n, ti, tj),
           ray_unit_sart(16, n, ti, tj), ray_unit_sart(17, n, ti, tj));
}
"""


@pytest.fixture(scope="module")
def pairs(tmp_path_factory):
    d = tmp_path_factory.mktemp("pairs")
    (d / "t.hip").write_text(PROGRAM)
    subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-host-only", "-I", CSRC, str(d / "t.hip"),
                    "-o", str(d / "t")], check=True, capture_output=True)

    def call(*args):
        r = subprocess.run([str(d / "t")] + [str(a) for a in args], capture_output=True, text=True)
        assert r.returncode == 0, r.returncode
        return [int(v) for v in r.stdout.split()]
    return call


@pytest.mark.parametrize("lg", [1, 4])
@pytest.mark.parametrize("views", [1, 3, 15])
@pytest.mark.parametrize("tiles_j", [1, 2, 23, 24, 25, 33, 127, 128, 416])
@pytest.mark.parametrize("tiles_i", [1, 2, 5, 14, 32])
def test_tiles_and_their_share(pairs, lg, views, tiles_i, tiles_j):
    grid, most, middle, short_walk, long_walk, sart_short, sart_long = pairs(views, tiles_i, tiles_j, lg)
    unit, tiles = 2 ** lg, tiles_i * tiles_j
    # at most the rest of a unit per column and 7 units of all views too many
    assert grid - views * tiles <= views * ((unit - 1) * tiles_i + 7 * unit)
    # even but for a unit of all views on either side of the middle's columns, and a
    # column's last unit, which may be short
    assert most <= middle / 8 + 2 * unit * views + (unit - 1) * views * ((tiles_i + 7) // 8)
    assert short_walk == (tiles_j >= 24 and views * tiles > 2560) and not long_walk
    blocks = tiles_j >= 128 and (tiles > 7000 or views * tiles > 80000)
    assert (sart_short, sart_long) == ((4, 4) if blocks else (short_walk, 0))
