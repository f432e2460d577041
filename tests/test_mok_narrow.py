"""Column tiles cut in parts for launches of few rows: the schedule and the wait counts on the CPU, the forward on the GPU."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STAGE = os.path.join(ROOT, "pipelink_amd", "stages", "mok")

SCHEDULE = r"""
#define MOK_SCHED_FN inline
#define MOK_SCHED_UNIFORM(x) (x)
#include "framework/schedule.hpp"
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace mok_framework;
int main(int argc, char** argv) {
  const int op = atoi(argv[1]), gu = atoi(argv[2]), dn = atoi(argv[3]);
  std::vector<int32_t> counts;
  for (int a = 4; a < argc; ++a) counts.push_back(atoi(argv[a]));
  const int ne = (int)counts.size();
  // the tables a wave's lanes make: its 64 lanes one after the other, a scan from what the lanes handed in the pass before
  static Tables tab, want;
  want.fill(counts.data(), ne);
  tab.last = tab.claim = 0xA5u;   // the words the launch's end and the queues write are none of the tables'
  std::vector<std::vector<int>> handed(2 * ((ne + 63) / 64), std::vector<int>(64, 0));
  for (int pass = 0; pass < 2; ++pass)   // the second pass has every lane's numbers at hand
    for (int lane = 0; lane < 64; ++lane) {
      int scans = 0, totals = 0;
      tab.fill_by_wave(counts.data(), ne, lane,
        [&](int v) { auto& of = handed.at(scans++); if (!pass) of[lane] = v; int s = 0; for (int l = 0; l <= lane; ++l) s += of[l]; return s; },
        [&](int) { int s = 0; for (int v : handed.at(totals++)) s += v; return s; });
    }
  for (int e = 0; e <= ne; ++e) if (tab.row_begin[e] != want.row_begin[e] || tab.tile_begin[e] != want.tile_begin[e]) { printf("table differs at %d\n", e); return 2; }
  if (tab.last != 0xA5u || tab.claim != 0xA5u) { printf("the tables write the queues' words\n"); return 3; }
  const MokFrameworkParams g{counts.data(), nullptr, ne, op | MOK_FWD_MAY_CUT, gu, dn};
  Schedule sched{g, tab, tab.tile_begin[ne], op == MOK_GEMM_FWD_ROUTED_DOWN ? 0 : gu, op == MOK_GEMM_FWD_ROUTED_GATE_UP ? 0 : dn};
  sched.cut();
  printf("%d %d\n", 1 << sched.gate_up_cut, 1 << sched.down_cut);
  for (int q = 0; q < NUM_XCD; ++q)
    for (int i = 0, cursor = 0; i < sched.length(q); ++i) {
      const MokGemmTask t = sched.decode(q, i, cursor);
      printf("%d %d %d %d %d %d %u\n", t.op, t.expert, t.row_begin, t.row_end, t.col_begin, t.wait_target, t.flags);
    }
}
"""

COUNTS = r"""
#define MOK_COUNT_FN constexpr inline
#include "gemm/load_counts.hpp"
#include <cstdio>
#include <vector>
using namespace mok_gemm_owner::counts;
int main() {
  int bad = 0;
  for (int n = 1; n <= 64; ++n) {
    std::vector<int> seen(n, 0);
    for (int wave = 0; wave < 4; ++wave) {
      const int mine = narrow_slots(wave, n);
      for (int i = 0; i < mine; ++i) { const int s = narrow_slot(wave, i); if (s >= n) { ++bad; continue; } ++seen[s]; }
      for (int ring : {2, 5})
        for (int i = -1; i + 1 < mine; ++i) {
          std::vector<int> order;   // which slot each load is of, in issue order, when the wave waits for slot i + 1
          for (int k = 0; k < mine && k <= (i < 0 ? ring - 1 : i + ring - 1); ++k)
            for (int l = 0; l < 6 + (k % 2 ? 0 : 3); ++l) order.push_back(k);
          int behind = 0;
          for (int k : order) behind += k > i + 1;
          const int got = i < 0 ? narrow_younger(0, ring - 1, mine) : narrow_younger(i + 1, i + ring - 1, mine);
          if (got != behind) { if (bad++ < 5) printf("n %d wave %d ring %d slot %d: %d, not %d\n", n, wave, ring, i + 1, got, behind); }
        }
    }
    for (int s = 0; s < n; ++s) if (seen[s] != 1) { if (bad++ < 5) printf("n %d: slot %d taken %d times\n", n, s, seen[s]); }
  }
  return bad != 0;
}
"""


def _compile(tmp_path, source):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    (tmp_path / "t.cpp").write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{STAGE}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    return str(tmp_path / "t")


def test_narrow_waves_share_the_slots_and_count_their_loads(tmp_path):
    res = subprocess.run([_compile(tmp_path, COUNTS)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


def test_parts_cover_every_column_tile_once(tmp_path):
    exe = _compile(tmp_path, SCHEDULE)
    for op, gu, dn, counts, parts in [(0, 23, 12, [0, 1, 0, 1, 1, 1] + [0] * 26, (1, 4)), (0, 23, 12, [1] * 8 + [0] * 24, (1, 1)),
                                      (0, 23, 12, [1] * 11, (1, 1)), (0, 6, 4, [32, 1, 0, 7], (4, 4)), (0, 6, 4, [33, 1, 0, 7], (1, 1)),
                                      (0, 6, 2, [32, 1, 0, 7], (1, 4)),   # 5 slots of gate/up contraction for 96 tasks
                                      (3, 23, 12, [1, 1], (4, 4)), (5, 23, 12, [1, 1, 1, 1], (1, 4)),
                                      (0, 2, 12, [5] * 22, (1, 1)),   # whole down tiles: the gate/up tiles stay whole too
                                      # layers where quarters were measured slower (us cut / whole 1.2, 1.4, 1.06, 1.05)
                                      (0, 2, 1, [1] * 28 + [0] * 4, (1, 1)), (0, 1, 2, [12, 13] * 16, (1, 1)),
                                      (0, 2, 1, [2, 3] * 4, (1, 1)), (0, 6, 2, [27, 28] * 4, (1, 1)),
                                      # tables of a wave's 64 lanes and more: the totals carried from group to group, an expert of
                                      # too many rows in a later one, down tiles only
                                      *((0, 23, 12, [1] + [0] * (n - 2) + [last], parts) for n in (63, 64, 65, 128, 129, 256)
                                        for last, parts in ((32, (4, 4)), (33, (1, 1)))),
                                      (0, 3, 2, [0, 1, 200, 2] * 64, (1, 1)), (5, 23, 12, ([1] + [0] * 51) * 4 + [0] * 40, (1, 4))]:
        out = subprocess.run([exe, str(op), str(gu), str(dn), *map(str, counts)], check=True, capture_output=True, text=True).stdout.splitlines()
        assert tuple(map(int, out[0].split())) == parts
        want = set()
        for e, c in enumerate(counts):
            first = sum(counts[:e])
            for top, cols, width, p in ((3, gu, 128, parts[0]), (5, dn, 256, parts[1])):
                if c and op in (0, top):
                    target = gu * parts[0] if top == 5 and op == 0 else 0
                    want |= {(top, e, first, first + c, col * (width // p), target, int(p == 4)) for col in range(cols * p)}
        items = [tuple(map(int, line.split())) for line in out[1:]]
        assert len(items) == len(want) and set(items) == want


GRID = r"""
#define MOK_SCHED_FN inline
#define MOK_SCHED_UNIFORM(x) (x)
#include "framework/schedule.hpp"
#include "../../csrc/plk_mok_residues.hpp"
#include <cstdio>
#include <random>
using namespace mok_framework;
int main() {
  std::mt19937 rng(1);
  auto upto = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
  for (int it = 0; it < 200000; ++it) {
    plk_mok::Dims d;
    d.hidden = 64 * upto(1, 48), d.intermediate = 64 * upto(1, 48), d.experts = upto(1, 64), d.pass = upto(0, 2);
    std::vector<int32_t> counts(d.experts);
    const int most = upto(0, 40);
    for (auto& c : counts) { c = rng() % 2 ? upto(0, most) : 0; d.routed_rows += c; }
    if (!d.routed_rows) continue;
    Tables tab;
    tab.fill(counts.data(), d.experts);
    const MokFrameworkParams g = plk_mok::framework_params(d, (uint64_t)(uintptr_t)counts.data(), 0);
    Schedule sched{g, tab, tab.tile_begin[d.experts], d.pass == 2 ? 0 : g.num_col_tiles_gate_up, d.pass == 1 ? 0 : g.num_col_tiles_down};
    sched.cut();
    const long long tasks = sched.gate_up_items() + sched.down_items();
    // the same tasks whatever the host says of them, as long as it says that they may be
    MokFrameworkParams told = g;
    told.op |= MOK_FWD_MAY_CUT;
    Schedule asked{told, tab, sched.row_tiles, sched.gate_up_cols, sched.down_cols};
    asked.cut();
    if (asked.gate_up_cut != sched.gate_up_cut || asked.down_cut != sched.down_cut) { printf("the host does not expect what the kernel cuts\n"); return 1; }
    if (tasks > plk_mok::max_workgroups(d)) { printf("%lld tasks, %lld workgroups\n", tasks, (long long)plk_mok::max_workgroups(d)); return 1; }
  }
  // a layer of 448 x 704, top 2 of 8: nothing is cut from 65 tokens on, and the grid has no room for it
  for (int tokens : {4, 64, 65, 110, 128, 129}) {
    plk_mok::Dims d;
    d.hidden = 448, d.intermediate = 704, d.experts = 8, d.routed_rows = 2 * tokens;
    printf("%d\n", (int)plk_mok::max_workgroups(d));
  }
}
"""


def test_the_grid_has_room_for_the_tasks_and_for_quarters_only_where_they_may_be(tmp_path):
    res = subprocess.run([_compile(tmp_path, GRID)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
    assert list(map(int, res.stdout.split())) == [112, 112, 72, 72, 72, 80]


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs the ROCm toolchain")
def test_the_packages_link_with_the_short_ring(tmp_path):
    """Ring depth 2 is the other value pipelines may bind: the code for parts must leave that link's register allocation possible
    (with parts and whole tiles in one loop the compiler did not survive it)."""
    import json

    from pipelink_amd.pipec import linker, pack
    from pipelink_amd.stages.mok import build as mok_build

    for stage_id, rel in mok_build.STAGES:
        pack.pack_stage(mok_build.HERE / rel, tmp_path / f"{stage_id}.plink")
    pipeline = json.loads((mok_build.HERE / "pipelines_fwd.json").read_text())
    pipeline["pipeline"]["forced_bindings"]["pipelink_mok_gemm_depth"] = 2
    (tmp_path / "pipeline.json").write_text(json.dumps(pipeline))
    link = linker.link(tmp_path / "pipeline.json", tmp_path / "link")
    assert link["bindings"]["pipelink_mok_gemm_depth"] == [2, "forced"] and link["observed"]["calls"] == 0


# one to 32 rows an expert (33: whole tiles); a contraction of one slot, fewer pairs than waves, an odd number of slots, one
# more pair than a ring; columns that end inside a column tile; gate/up and down tiles cut, down tiles only, none; rows of whole
# cache lines (one launch) or not; from `(448, 256` on: quarters of the shortest contractions that are cut
@pytest.mark.gpu
@pytest.mark.parametrize("H,I,counts", [(64, 64, [1]), (128, 320, [32, 0, 5]), (576, 192, [31, 17, 1, 32]), (704, 1088, [2] * 5),
                                        (2880, 2880, [1, 0, 1, 1, 1]), (2880, 2880, [3, 2, 1, 1, 32, 9, 1]), (1536, 2048, [4] * 7),
                                        (448, 704, [33, 2, 1]), (320, 128, [20] * 8),
                                        (448, 256, [16]), (512, 192, [5]), (320, 192, [7]), (576, 384, [9, 0, 31, 1]), (1088, 448, [31, 1]), (1536, 64, [3]),
                                        # more experts than a wave has lanes: the expert of a task found beyond the first 64, parts and none
                                        (512, 512, [0] * 100 + [3] + [0] * 28 + [1]), (256, 192, [1, 0, 2] * 43 + [70]), (128, 128, [1, 0, 2] * 85 + [5])])
def test_forward_of_few_rows_matches_the_oracle(H, I, counts):
    from oracle import moe_ffn
    from pipelink_amd.host import mok_inputs
    from pipelink_amd.host.mok import MoKSession, code_pitch
    from pipelink_amd.stages.mok import build as mok_build
    from test_gpu_moe import TOL, _oracle, _run

    paths = mok_build.images()
    inp = mok_inputs.generate(max(counts) + 3, H, I, len(counts), 1, seed=H + len(counts), counts=counts)
    ref = _oracle(inp)
    ys = []
    for image in ("linked", "one_unit"):
        with MoKSession(paths[image].read_bytes(), str(paths["link_json"])) as sess:
            for launches in (1, 2):
                sess.launches(launches)
                for pitch in (None, code_pitch(I)):
                    hq, hsc, y = _run(sess, inp, H, I, pitch_i=pitch)
                    yy = y.float().numpy()
                    assert not np.isnan(yy).any() and moe_ffn.rel_frobenius(yy, ref["y"]) <= TOL
                    ys.append(yy)
    assert all(np.array_equal(ys[0], other) for other in ys[1:])   # one launch and two, linked and one unit: the same sums


@pytest.mark.gpu
def test_parts_through_the_static_entry_point_and_in_a_graph():
    """Gate/up and down tiles in parts, one launch (rows of whole cache lines) and two, without a session's own buffers: the
    bytes of the plain forward, also on every replay of a captured graph."""
    import json

    import torch
    from pipelink_amd.host import mok_inputs
    from pipelink_amd.host.backend import HipBackend
    from pipelink_amd.host.mok import MoKSession
    from pipelink_amd.stages.mok import build as mok_build
    from test_zz_no_alloc import _device_problem, _poison, _snapshot

    paths = mok_build.images()
    link = json.loads(paths["link_json"].read_text())
    with MoKSession(paths["linked"].read_bytes(), link) as sess, MoKSession(paths["linked"].read_bytes(), link) as fresh:
        cases = [_device_problem(sess, mok_inputs.generate(40, H, I, len(c), 1, seed=H, counts=c), H, I, pitch)
                 for H, I, c, pitch in ((1088, 704, [31, 1, 0, 7], 768), (1088, 704, [31, 1, 0, 7], None), (1536, 64, [3], 128))]
        expected = []
        for prob, out, _ in cases:
            _poison(out)
            sess.forward(prob)
            expected.append(_snapshot(out))
        be = HipBackend(0, 0)
        stream = be.stream_create()
        graph = be.capture(stream, lambda: [fresh.forward_static(prob, stream=stream) for prob, _, _ in cases])
        try:
            for replay in range(4):   # the first turn is the plain call
                for _, out, _ in cases:
                    _poison(out)
                torch.cuda.synchronize()
                if replay:
                    graph.launch(stream)
                    be.synchronize(stream)
                else:
                    for prob, _, _ in cases:
                        sess.forward_static(prob)
                for (_, out, _), want in zip(cases, expected):
                    assert all(torch.equal(g, w) for g, w in zip(_snapshot(out), want)), replay
            assert fresh.status() == 0 and sess.status() == 0
        finally:
            graph.close()
            be.close()
