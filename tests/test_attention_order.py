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
