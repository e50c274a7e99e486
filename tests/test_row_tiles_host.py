"""The partners that the row pass of H*v reads in LDS for the impurity terms
stay inside the tile, also for the slots of a tile that hold no row (host
walk over all tiles, tests/host/row_tiles.cpp).  The sectors have tiles with
empty slots: more runs of three rows than single rows to fill them up."""
import os
import subprocess

import pytest

from edlib_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def walker(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "row_tiles")
    subprocess.check_call([build.HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I", build.SRC,
                           os.path.join(ROOT, "tests", "host", "row_tiles.cpp"), "-o", out, "-L", build.PKG, "-ledhip",
                           "-Wl,-rpath," + build.PKG])
    return out


@pytest.mark.parametrize("sector", [(9, 3, 4, 5), (11, 3, 6, 5), (14, 3, 7, 7), (14, 3, 6, 7), (14, 3, 8, 7),
                                    (8, 2, 4, 3), (9, 3, 1, 2)])
def test_partners_stay_in_the_tile(walker, sector):
    r = subprocess.run([walker] + [str(x) for x in sector], capture_output=True, text=True, check=True)
    empty, outside, tiles = map(int, r.stdout.split())
    assert tiles > 0
    if sector[0] >= 11:
        assert empty > 0  # the case that is meant
    assert outside == 0
