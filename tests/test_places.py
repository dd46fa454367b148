"""Planes side by side in the backward: the map of workgroups to planes and tiles, compiled for the host.  Workgroup w goes to XCD w % 8, and from the
33rd of an XCD on to compute units that have one already."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sparseattention_amd", "csrc")
PROGRAM = r"""
#include "places.h"
#include <cstdio>
#include <cstdlib>
int main(int, char **a) {
    const int planes = atoi(a[1]), tiles = atoi(a[2]), by_rule = sa::bwd_spread(planes, tiles), total = planes * tiles;
    const int spread = atoi(a[3]) < 0 ? by_rule : atoi(a[3]);
    if (spread == 0 || a[4]) return printf("%d 0\n", spread), 0;
    for (int w = 0; w < total; w++) {
        const sa::SidePlace at = sa::side_place(8 * sa::side_turn(w >> 3, total >> 3) + (w & 7), spread, planes, tiles);
        printf("%d %d\n", at.plane, at.order);
    }
}
"""


@pytest.fixture(scope="module")
def places(tmp_path_factory):
    d = tmp_path_factory.mktemp("places")
    (d / "p.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", str(d / "p.cpp"), "-o", str(d / "p")], check=True)

    def of(*args):
        out = subprocess.run([str(d / "p"), *map(str, args)], check=True, capture_output=True, text=True).stdout
        return [tuple(map(int, ln.split())) for ln in out.splitlines()]
    return of


@pytest.mark.parametrize("planes,tiles,spread", [(76, 8, 4), (44, 12, 4), (132, 8, 12), (12, 16, 12), (12, 67, 4), (36, 11, 36), (4, 33, 4),
                                                 (24, 22, 8), (72, 9, 72), (72, 16, 24), (8, 5, 8), (128, 32, 64), (20, 1, 20), (76, 8, 40), (104, 9, 56), (12, 64, 8)])
def test_every_tile_once_and_the_xcds_alike(places, planes, tiles, spread):
    got = places(planes, tiles, spread)
    assert sorted(got) == [(p, t) for p in range(planes) for t in range(tiles)]
    # causal lists: a tile of order t has tiles - t entries.  What is left over of a row of four orders is all that two XCDs may differ by in a
    # group, and one of the eight workgroups behind the last whole row of eight
    work = [0] * 8
    for w, (_, t) in enumerate(got):
        work[w % 8] += tiles - t
    groups, shared = -(-planes // spread), planes % 8 != 0
    assert max(work) - min(work) <= (groups * 2 if shared and tiles % 4 else 0) + (tiles if planes * tiles % 8 else 0)


# planes of 64 KiB a tile (K and V of 128 keys): as many together as 9 MiB hold, of launches of up to 2048 tiles nine in any case, in groups of even
# size, whatever divides them
@pytest.mark.parametrize("planes,tiles,spread", [(256, 32, 32), (128, 16, 64), (32, 64, 32), (40, 64, 16), (8, 128, 8), (24, 256, 8), (76, 8, 40), (76, 32, 16),
                                                 (132, 8, 68), (44, 12, 44), (104, 8, 104), (72, 16, 72), (4, 128, 4), (12, 64, 12), (40, 32, 40), (16, 32, 16),
                                                 (80, 25, 40), (18, 8, 0), (1, 4096, 0)])
def test_as_many_planes_together_as_the_caches_hold(places, planes, tiles, spread):
    assert places(planes, tiles, -1, 1)[0][0] == spread
    if spread:
        got = places(planes, tiles, -1)
        assert sorted(got) == [(p, t) for p in range(planes) for t in range(tiles)]
        unit = 4 if planes % 8 else 8
        assert spread == unit or spread // unit * tiles * 65536 <= 9 << 20 or planes * tiles <= 2048 and spread // unit <= 9
