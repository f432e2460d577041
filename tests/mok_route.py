"""Which tiles the routed-expert forward runs for given sizes and counts, from the code that the kernel and the host decide it with."""
import collections
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STAGE = os.path.join(ROOT, "pipelink_amd", "stages", "mok")
PROGRAM = r"""
#define MOK_SCHED_FN inline
#define MOK_SCHED_UNIFORM(x) (x)
#include "framework/schedule.hpp"
#include "../../csrc/plk_mok_residues.hpp"
#include <cstdio>
#include <cstdlib>
using namespace mok_framework;
int main(int argc, char** argv) {
  const bool offer = atoi(argv[1]) != 0;
  plk_mok::Dims d;
  d.hidden = atoi(argv[2]), d.intermediate = atoi(argv[3]), d.experts = argc - 4;
  std::vector<int32_t> counts;
  for (int a = 4; a < argc; ++a) counts.push_back(atoi(argv[a])), d.routed_rows += counts.back();
  static Tables tab;
  tab.fill(counts.data(), d.experts);
  MokFrameworkParams g = plk_mok::framework_params(d, 0, 0);
  if (offer) plk_mok::offer_parts(d, g);
  Schedule sched{g, tab, tab.tile_begin[d.experts], g.num_col_tiles_gate_up, g.num_col_tiles_down};
  sched.cut();
  sched.part();
  for (int q = 0; q < NUM_XCD; ++q)
    for (int i = 0, cursor = 0; i < sched.length(q); ++i) {
      const MokGemmTask t = sched.decode(q, i, cursor);
      const bool gate_up = t.op == MOK_GEMM_FWD_ROUTED_GATE_UP;
      const int rows = t.row_end - t.row_begin, cols = (gate_up ? d.intermediate : d.hidden) - t.col_begin;   // as mok::tile_placement
      const char* kind = t.flags & MOK_TASK_QUARTER ? "narrow" : t.flags & MOK_TASK_PART ? "part" : rows <= 32 ? "rows32" : rows <= 64 ? "rows64"
                         : cols <= 64 ? "cols" : "full";
      printf("%s_%s\n", gate_up ? "gate_up" : "down", kind);
    }
}
"""


@functools.lru_cache(None)
def _program() -> str:
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    directory = tempfile.mkdtemp()
    source = os.path.join(directory, "route.cpp")
    with open(source, "w") as f:
        f.write(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{STAGE}", source, "-o", source[:-4]], check=True)
    return source[:-4]


def tiles(H: int, I: int, counts, parts: bool = True) -> collections.Counter:
    """How many tiles of each GEMM are full ones, of few rows (rows32, rows64), of few columns (cols), quarters (narrow) or parts, in a
    launch by the session (``parts``) or by the owners' providers, which offer no parts."""
    out = subprocess.run([_program(), str(int(parts)), str(H), str(I), *(str(int(c)) for c in counts)], check=True, capture_output=True, text=True).stdout
    return collections.Counter(out.split())


def kinds(H: int, I: int, counts, parts: bool = True) -> set[str]:
    return {t.split("_")[-1] for t in tiles(H, I, counts, parts)}
