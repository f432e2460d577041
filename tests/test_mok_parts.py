"""Column tiles as parts of 64 columns, for launches of more rows that leave most of the chip idle: which launches and tasks on the
CPU, the forward on the GPU."""
import subprocess

import numpy as np
import pytest

from test_mok_narrow import _compile

SCHEDULE = r"""
#define MOK_SCHED_FN inline
#define MOK_SCHED_UNIFORM(x) (x)
#include "framework/schedule.hpp"
#include "../../csrc/plk_mok_residues.hpp"
#include <cstdio>
#include <random>
#include <set>
#include <tuple>
using namespace mok_framework;
int main() {
  std::mt19937 rng(2);
  auto upto = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
  int run = 0;
  for (int it = 0; it < 20000; ++it) {
    plk_mok::Dims d;
    d.hidden = 64 * upto(1, 24), d.intermediate = 64 * upto(1, 24), d.experts = upto(1, 20), d.pass = upto(0, 2);
    std::vector<int32_t> counts(d.experts);
    const int most = upto(1, 700);
    for (auto& c : counts) { c = rng() % 4 ? upto(0, most) : 0; d.routed_rows += c; }
    if (!d.routed_rows) continue;
    Tables tab;
    tab.fill(counts.data(), d.experts);
    MokFrameworkParams g = plk_mok::framework_params(d, (uint64_t)(uintptr_t)counts.data(), 0);
    plk_mok::offer_parts(d, g);
    Schedule sched{g, tab, tab.tile_begin[d.experts], d.pass == 2 ? 0 : g.num_col_tiles_gate_up, d.pass == 1 ? 0 : g.num_col_tiles_down};
    sched.cut();
    sched.part();
    const bool parts = sched.down_width == PART_COLS;
    if (parts != (sched.gate_up_width == PART_COLS) || (parts && (sched.down_cut || sched.gate_up_cut))) { puts("half a launch"); return 1; }
    if (parts && d.routed_rows <= 64 * d.experts) { puts("few rows"); return 1; }
    if (!parts) continue;
    ++run;
    std::set<std::tuple<int, int, int, int>> seen;
    long long tasks = 0;
    for (int q = 0; q < NUM_XCD; ++q)
      for (int i = 0, cursor = 0; i < sched.length(q); ++i, ++tasks) {
        const MokGemmTask t = sched.decode(q, i, cursor);
        const bool gu = t.op == MOK_GEMM_FWD_ROUTED_GATE_UP;
        const int cols = gu ? d.intermediate : d.hidden;
        if (t.flags != MOK_TASK_PART || t.col_begin % 64 || t.col_begin >= cols || t.row_end != tab.row_begin[t.expert + 1] ||
            (t.row_begin - tab.row_begin[t.expert]) % 256 || !seen.insert({t.op, t.expert, t.row_begin, t.col_begin}).second) { puts("task"); return 1; }
        if (t.wait_target != (!gu && d.pass == 0 ? d.intermediate / 64 : 0)) { puts("target"); return 1; }
      }
    const long long want = (long long)sched.row_tiles * ((d.pass != 2 ? d.intermediate / 64 : 0) + (d.pass != 1 ? d.hidden / 64 : 0));
    if (tasks != want || tasks > plk_mok::useful_workgroups(d)) { printf("%lld tasks of %lld, %lld workgroups\n", tasks, want, (long long)plk_mok::useful_workgroups(d)); return 1; }
    if (sched.gate_up_items() > CHIP || sched.down_items() > CHIP) { puts("more than one turn"); return 1; }
  }
  printf("%d\n", run);
}
"""


def test_parts_cover_the_columns_once_and_the_grid_has_room_for_them(tmp_path):
    res = subprocess.run([_compile(tmp_path, SCHEDULE)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout) > 1000


# (us whole / parts) where parts are the faster ones, and where they are not: long contractions of several row tiles, 64 output columns
@pytest.mark.parametrize("H,I,counts,parts", [(448, 704, [128] * 8, True), (2048, 512, [130, 90, 100, 80], True), (576, 320, [300, 33, 0, 70, 191], True),
                                              (2880, 2880, [515], False), (2880, 2880, [266, 267], False), (2880, 2880, [73] * 4, False),   # 71.2 / 76.8
                                              (2368, 2304, [853], False), (2880, 2432, [250, 250, 251], False),                            # 63.3 / 68.4
                                              (64, 1728, [429] * 3, False), (64, 1664, [112] * 8, False), (64, 832, [200] * 4, False),         # 32.6 / 37.2
                                              (64, 768, [200] * 4, True), (128, 1728, [429] * 3, True), (1664, 2752, [82] * 4, True)])                                       # 67.3 / 60.4
def test_parts_run_where_they_are_faster(H, I, counts, parts):
    from mok_route import kinds

    assert ("part" in kinds(H, I, counts)) is parts


# rows around a wave's 64, 128 and a tile's 256, experts of few rows and of none among them; columns of one part, an odd number of
# parts and whole column tiles; contractions from one slot to more than a ring; rows of whole cache lines (one launch) and not
@pytest.mark.gpu
@pytest.mark.parametrize("H,I,counts", [(64, 64, [65]), (128, 192, [127, 0, 129]), (448, 704, [128, 64, 200, 65]), (320, 128, [256, 257, 1]),
                                        (256, 640, [511, 3]), (576, 320, [300, 33, 0, 70, 191]), (1088, 448, [100, 90]),
                                        # contractions of 26, 36, 43 and 45 slots, and next to where parts end
                                        (1664, 2752, [82] * 4), (2304, 448, [130, 0, 90, 70]), (192, 2880, [257, 66]), (2880, 192, [300, 1]), (64, 768, [200] * 4)])
def test_forward_in_parts_matches_the_oracle_and_whole_tiles(H, I, counts):
    from mok_route import kinds

    assert kinds(H, I, counts) == {"part"} and "part" not in kinds(H, I, counts, parts=False)
    from oracle import moe_ffn
    from pipelink_amd.host import mok_inputs
    from pipelink_amd.host.mok import MoKSession, code_pitch
    from pipelink_amd.stages.mok import build as mok_build
    from test_gpu_moe import TOL, _oracle, _run

    paths = mok_build.images()
    inp = mok_inputs.generate(max(counts) + 3, H, I, len(counts), 1, seed=H + I, counts=counts)
    ref = _oracle(inp)
    ys = []
    for image in ("linked", "one_unit"):
        with MoKSession(paths[image].read_bytes(), str(paths["link_json"])) as sess:
            for launches in (1, 2):
                sess.launches(launches)
                for pitch in (None, code_pitch(I)):
                    y = _run(sess, inp, H, I, pitch_i=pitch)[2].float().numpy()
                    assert sess.status() == 0 and not np.isnan(y).any() and moe_ffn.rel_frobenius(y, ref["y"]) <= TOL
                    ys.append(y)
    assert all(np.array_equal(ys[0], other) for other in ys[1:])


@pytest.mark.gpu
def test_parts_through_the_static_entry_point_and_in_a_graph():
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
        cases = [_device_problem(sess, mok_inputs.generate(300, 448, 704, len(c), 1, seed=len(c), counts=c), 448, 704, pitch)
                 for c, pitch in (([257, 1, 130], 768), ([257, 1, 130], None))]
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
