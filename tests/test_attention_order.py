"""The order of the attention tiles, on the CPU: every tile of every head once, longest first on every XCD, heads that share a KV head
together."""
import shutil
import subprocess
from pathlib import Path

import pytest

INCLUDE = Path(__file__).resolve().parent.parent / "pipelink_amd" / "stages" / "attention" / "include"
PROGRAM = r"""
#define FA_ORDER_FN inline
#include "fa_order.hpp"
#include <cstdio>
#include <set>
#include <vector>
int main() {
  for (int batch = 1; batch <= 6; ++batch)
    for (int kv : {1, 2, 3, 4, 5, 8, 12, 16})
      for (int per : {1, 2, 3, 4, 8})
        for (int tiles : {1, 2, 3, 5, 8, 9, 32}) {
          const int q = kv * per, total = batch * q * tiles;
          std::vector<char> seen(total, 0);
          std::vector<int> last(8, tiles), xcd_of(batch * kv, -1);
          for (int i = 0; i < total; ++i) {
            const fa_order::Tile t = fa_order::tile_of(i, batch, q, kv, tiles);
            if (t.tile < 0 || t.tile >= tiles || t.bh < 0 || t.bh >= batch * q || seen[t.tile * batch * q + t.bh]++) return printf("batch %d heads %d / %d tiles %d index %d\n", batch, q, kv, tiles, i), 1;
            if (t.tile > last[i % 8]) return printf("a longer tile later\n"), 1;
            last[i % 8] = t.tile;
            int& x = xcd_of[t.bh / per];
            if (batch * kv % 8 == 0 && x >= 0 && x != i % 8) return printf("a group on two XCDs\n"), 1;
            x = i % 8;
          }
        }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_tile_once_longest_first_and_groups_together(tmp_path):
    (tmp_path / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{INCLUDE}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    res = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


OLD = r"""
#define FA_ORDER_FN inline
#include "fa_order.hpp"
#include <cstdio>
#include <initializer_list>
// the order as it was first written: sets of XCDs by division, head by head where the grid has no eighths
static void first(int index, int batch, int q_heads, int kv_heads, int q_tiles, int& tile, int& bh) {
  const int heads = batch * q_heads, per_kv = q_heads / kv_heads, groups = batch * kv_heads;
  if (heads * q_tiles % 8 != 0) { tile = q_tiles - 1 - index / heads; bh = index % heads; return; }
  const int sets = groups % 8 ? groups & -groups : 8, xcd = index % 8, at = index / 8 * (8 / sets) + xcd / sets;
  const int set_heads = heads / sets, in_level = at % set_heads;
  tile = q_tiles - 1 - at / set_heads;
  bh = (xcd % sets + sets * (in_level / per_kv)) * per_kv + in_level % per_kv;
}
int main() {
  for (int batch = 1; batch <= 6; ++batch)
    for (int kv : {1, 2, 3, 4, 5, 8, 12, 16})
      for (int per : {1, 2, 3, 4, 8})
        for (int tiles : {1, 2, 3, 5, 8, 9, 32})
          for (int i = 0; i < batch * kv * per * tiles; ++i) {
            int tile, bh;
            first(i, batch, kv * per, kv, tiles, tile, bh);
            const fa_order::Tile t = fa_order::tile_of(i, batch, kv * per, kv, tiles);
            if (t.tile != tile || t.bh != bh || t.group != bh / per) return printf("batch %d heads %d / %d tiles %d index %d\n", batch, kv * per, kv, tiles, i), 1;
          }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_the_order_by_shifts_is_the_one_by_divisions(tmp_path):
    (tmp_path / "t.cpp").write_text(OLD)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{INCLUDE}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    res = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


@pytest.mark.parametrize("image", ["linked", "window_linked", "half_linked", "window_half_linked"])
def test_a_workgroup_finds_its_tile_with_four_divisions(image):
    """A division of numbers known at run time is a reciprocal and some ten instructions behind it, in front of everything else."""
    from pipelink_amd.pipec.pack import LLVM_BIN
    from pipelink_amd.stages.attention import build as fa_build

    if not Path("/opt/rocm/bin/hipcc").exists():
        pytest.skip("needs the ROCm toolchain")
    text = subprocess.run([str(LLVM_BIN / "llvm-objdump"), "-d", str(fa_build.images()[image])], capture_output=True, text=True, check=True).stdout
    assert text.count("v_rcp_iflag_f32") <= 4   # three for the tile (heads of a KV head, level, group), one for the output's batch
