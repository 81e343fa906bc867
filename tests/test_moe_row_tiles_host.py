"""How the rows of an expert are cut into even tiles (row_tiles.hpp), compiled for the host."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "sglang_amd" / "csrc"
SOURCE = """#define __host__
#define __device__
#include "row_tiles.hpp"
extern "C" void cut(int all, int tiles, int* from, int* units) {
  for (int k = 0; k < tiles; ++k) {
    const sgl_amd::RowTile t = sgl_amd::even_tile(all, tiles, k);
    from[k] = t.from;
    units[k] = t.units;
  }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
@pytest.mark.parametrize("rows", [1, 16, 159, 160, 161, 321, 2500, 3_000_000, 3_400_000, 65535 * 256])
def test_even_tiles_cover_the_rows_of_an_expert(tmp_path, rows):
    """From one row to as many as a launch takes (65535 alignment blocks of 256), for the fewest and the most units of a tile: the tiles follow one another,
    differ by at most a unit and none has more than the most."""
    (tmp_path / "cut.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-fwrapv", "-shared", "-fPIC", f"-I{CSRC}", str(tmp_path / "cut.cpp"), "-o", str(tmp_path / "cut.so")], check=True)
    lib, units = ctypes.CDLL(str(tmp_path / "cut.so")), -(-rows // 16)
    for most in (10, 13, 20):
        tiles = -(-units // most)
        at, size = (ctypes.c_int * tiles)(), (ctypes.c_int * tiles)()
        lib.cut(units, tiles, at, size)
        assert at[0] == 0 and at[tiles - 1] + size[tiles - 1] == units
        assert all(at[k] + size[k] == at[k + 1] for k in range(tiles - 1))
        assert max(size) <= most and max(size) - min(size) <= 1 and min(size) >= 1
