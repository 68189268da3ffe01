"""The ray kernels' work-group to tile mapping (compiled for the host): every tile
of a detector exactly once, for single-geometry launches and batched positions,
and the columns through the middle of the detector (the volume's shadow) shared
evenly among the 8 XCDs, from one row of tiles to many."""
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
    const int64_t grid = ray_grid(n, ti, tj);
    const int tiles = n * ti * tj;
    std::vector<int> seen(tiles), at(tiles), load(8), load_batch(8);
    auto middle = [&](const RayTile& t) { return t.ti >= ti / 4 && t.ti < ti - ti / 4; };
    for (int64_t w = 0; w < grid; ++w) {
        RayTile t;
        if (!ray_tile((int)w, n, ti, tj, t)) continue;
        if (t.slot < 0 || t.slot >= n || t.ti < 0 || t.ti >= ti || t.tj < 0 || t.tj >= tj) return 1;
        ++seen[(t.slot * ti + t.ti) * tj + t.tj];
        if (middle(t)) ++load[w % 8];
    }
    for (int p = 0; p < tiles; ++p) {
        const RayTile t = ray_tile_of_position(p, n, ti, tj);
        if (t.slot < 0 || t.slot >= n || t.ti < 0 || t.ti >= ti || t.tj < 0 || t.tj >= tj) return 2;
        ++at[(t.slot * ti + t.ti) * tj + t.tj];
        int x = 7;  // the XCD whose eighth holds p
        while ((int64_t)tiles * x / 8 > p) --x;
        if (middle(t)) ++load_batch[x];
    }
    int64_t most = 0, most_batch = 0, all = 0;
    for (int x = 0; x < 8; ++x) {
        most = std::max<int64_t>(most, load[x]);
        most_batch = std::max<int64_t>(most_batch, load_batch[x]);
        all += load[x];
    }
    for (int k = 0; k < tiles; ++k)
        if (seen[k] != 1 || at[k] != 1) return 3;
    printf("%lld %lld %lld %lld\\n", (long long)grid, (long long)most, (long long)most_batch, (long long)all);
}
"""


@pytest.fixture(scope="module")
def mapping(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "t.hip").write_text(PROGRAM)
    subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-host-only", "-I", CSRC, str(d / "t.hip"),
                    "-o", str(d / "t")], check=True, capture_output=True)

    def call(*args):
        r = subprocess.run([str(d / "t")] + [str(a) for a in args], capture_output=True, text=True)
        assert r.returncode == 0, r.returncode
        return [int(v) for v in r.stdout.split()]
    return call


@pytest.mark.parametrize("views", [1, 3, 15])
@pytest.mark.parametrize("tiles_j", [1, 2, 3, 5, 8, 9, 10, 15, 16, 20, 23, 24, 25, 32, 33, 416])
@pytest.mark.parametrize("tiles_i", [1, 2, 5, 32])
def test_tiles_and_their_share(mapping, views, tiles_i, tiles_j):
    grid, most, most_batch, middle = mapping(views, tiles_i, tiles_j)
    # at most 7 units of a band or a column too many
    assert grid - views * tiles_i * tiles_j <= 7 * views * tiles_i
    # even to a third (25 bands: 4 on one XCD, 3.125 on average), or to two columns
    # of all views where there are few of them in all
    bar = max(4 / 3 * middle / 8, middle / 8 + 2 * views)
    assert most <= bar and most_batch <= bar
