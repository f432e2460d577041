// The MoK framework stage's schedule: which tiles a launch has, in which of the eight lists, in which order, and
// item -> task.  Plain C++ on plain integers, so that a host compiler takes it too: the tests enumerate the lists on
// the CPU (every tile of both GEMMs exactly once, gate/up tiles before down tiles, row and column ranges) with
// MOK_SCHED_FN defined empty and MOK_SCHED_UNIFORM(x) as x.
//
// Plays the part of the task decode in campaigns/mok/port/framework/interp_fwd.cu:137-214.
#ifndef PIPELINK_MOK_FRAMEWORK_SCHEDULE_HPP
#define PIPELINK_MOK_FRAMEWORK_SCHEDULE_HPP
#include <stdint.h>
#include "../include/mok_abi.h"
#include "cut.hpp"

#ifndef MOK_SCHED_FN
#define MOK_SCHED_FN __device__ __forceinline__
// wave-uniform by construction; say so, so that the value lives in a scalar register
#define MOK_SCHED_UNIFORM(x) __builtin_amdgcn_readfirstlane(x)
#define MOK_SCHED_COUNT(n, holds) mok_framework::count_by_wave(n, holds)
#endif
#ifndef MOK_SCHED_COUNT
#define MOK_SCHED_COUNT(n, holds) mok_framework::count(n, holds)
#endif

namespace mok_framework {
constexpr int MAX_EXPERTS = 256;
constexpr int NUM_XCD = 8;       // lists
constexpr int TILE_X = 256;      // routed rows of a tile   (the GEMM owner's published facts; the stage source
constexpr int TILE_W = 256;      // weight rows of a tile    checks them against the owner's header)

// how many of the first n numbers a condition holds for: one after the other; by a wave (all of its lanes take part and get
// the answer), where the reads behind the condition are 64 at a time instead of a chain of LDS latencies
template <class Holds>
MOK_SCHED_FN int count(int n, Holds holds) {
  int c = 0;
  for (int i = 0; i < n; ++i) c += holds(i) ? 1 : 0;
  return c;
}
#ifdef __HIP_DEVICE_COMPILE__
template <class Holds>
MOK_SCHED_FN int count_by_wave(int n, Holds holds) {
  int c = 0;
  for (int i = threadIdx.x & 63; i - (int)(threadIdx.x & 63) < n; i += 64)
    c += __builtin_popcountll(__builtin_amdgcn_ballot_w64(i < n && holds(i)));
  return c;
}
#endif

// the schedule's tables in LDS: exclusive prefix sums per expert, and one word of the last workgroup
struct Tables {
  int row_begin[MAX_EXPERTS + 1];
  int tile_begin[MAX_EXPERTS + 1];
  // (nothing here may be written by a workgroup that has no tile and read by it before: no barrier lies between)
  uint32_t last;   // 1 + the list `claim` is of, or 0 if every list has been handed out; in the end: 1 in the workgroup
                   // that leaves the launch last
  uint32_t claim;  // what the list's queue answered this workgroup's last request

  // exclusive prefix sums of rows and row tiles per expert, one expert after the other (what the tests compare the next with)
  MOK_SCHED_FN void fill(const int32_t* tokens_per_expert, int ne) {
    int rows = 0, tiles = 0;
    for (int e = 0; e < ne; ++e) {
      row_begin[e] = rows;
      tile_begin[e] = tiles;
      const int c = tokens_per_expert[e];
      rows += c;
      tiles += (c + TILE_X - 1) / TILE_X;
    }
    row_begin[ne] = rows;
    tile_begin[ne] = tiles;
  }
  // The same by the 64 lanes of one wave, an expert per lane (every workgroup computes its own copy).  `scan` is the
  // inclusive sum over the lanes up to this one, `last_lane` lane 63's value.  fill() by one thread is a chain of `ne`
  // memory reads, one after the other, in front of everything else a launch does: a launch of one token and 32 experts
  // took 54.4 us with it and takes 53.2 us.
  template <class Scan, class Last>
  MOK_SCHED_FN void fill_by_wave(const int32_t* tokens_per_expert, int ne, int lane, Scan scan, Last last_lane) {
    int rows = 0, tiles = 0;
    for (int e0 = 0; e0 < ne; e0 += 64) {
      const int e = e0 + lane;
      const int c = e < ne ? tokens_per_expert[e] : 0, t = (c + TILE_X - 1) / TILE_X;
      const int c_sum = scan(c), t_sum = scan(t);
      if (e < ne) {
        row_begin[e] = rows + c_sum - c;
        tile_begin[e] = tiles + t_sum - t;
      }
      rows += last_lane(c_sum);
      tiles += last_lane(t_sum);
    }
    if (lane == 0) {
      row_begin[ne] = rows;
      tile_begin[ne] = tiles;
    }
  }
};

struct Schedule {
  const MokFrameworkParams& g;
  const Tables& tab;
  int row_tiles;  // of all experts
  int gate_up_cols, down_cols;  // column tiles of the GEMMs this launch runs (0: not run)
  int gate_up_cut = 0, down_cut = 0;  // a column tile is 2^cut tasks (one or four)
  int gate_up_width = TILE_W / 2, down_width = TILE_W;  // columns of a column tile; PART_COLS: every task is a part

  // Narrow tiles, for launches all of whose experts have at most NARROW_ROWS rows (every wave looks at the tables itself):
  // cut_for says whose column tiles are cut in four.
  MOK_SCHED_FN void cut() {
    if (!(g.op & MOK_FWD_MAY_CUT)) return;  // (most launches know here: the tables' sums and the rule took them 0.1 us)
    const Cut c = cut_for(tab.row_begin[g.num_experts], g.num_experts, row_tiles, g.num_col_tiles_gate_up, g.num_col_tiles_down);
    if (MOK_SCHED_UNIFORM(c.down) == 0) return;
    if (MOK_SCHED_COUNT(g.num_experts, [&](int e) { return tab.row_begin[e + 1] - tab.row_begin[e] > NARROW_ROWS; }) != 0) return;
    down_cut = MOK_SCHED_UNIFORM(c.down);
    gate_up_cut = MOK_SCHED_UNIFORM(c.gate_up);
  }
  // Parts of 64 columns, for launches of more rows that leave most of the chip idle: the column tiles are that narrow then.
  MOK_SCHED_FN void part() {
    const int last_gate_up = g.op >> MOK_FWD_LAST_GATE_UP_SHIFT & MOK_FWD_LAST_MASK, last_down = g.op >> MOK_FWD_LAST_DOWN_SHIFT & MOK_FWD_LAST_MASK;
    if (last_gate_up == 0) return;
    const int gu = (g.num_col_tiles_gate_up - 1) * (TILE_W / 2 / PART_COLS) + last_gate_up, d = (g.num_col_tiles_down - 1) * (TILE_W / PART_COLS) + last_down;
    if (!MOK_SCHED_UNIFORM(parts_for(tab.row_begin[g.num_experts], g.num_experts, row_tiles, gu, d))) return;
    if (gate_up_cols) gate_up_cols = gu;
    if (down_cols) down_cols = d;
    gate_up_width = down_width = PART_COLS;
  }
  MOK_SCHED_FN int gate_up_items() const { return row_tiles * gate_up_cols << gate_up_cut; }
  MOK_SCHED_FN int down_items() const { return row_tiles * down_cols << down_cut; }

  // List q: the q-th eighth of the gate/up tiles (all experts' tiles in one sequence: expert by expert, column tile by
  // column tile, row tiles innermost), then the q-th eighth of the down tiles, from its second expert on (`rotated`).
  MOK_SCHED_FN int share(int q, int total) const { return (int)((long long)q * total / NUM_XCD); }
  MOK_SCHED_FN int length(int q) const {
    const int gu = gate_up_items(), d = down_items();
    return share(q + 1, gu) - share(q, gu) + share(q + 1, d) - share(q, d);
  }

  // The down tile list q runs in the place of `item` (launches of both GEMMs): the rest of the expert in whose middle the list
  // begins comes last.  That expert's gate/up tiles are divided alike, some of them the end of the list before, which run last
  // of all gate/up tiles: its down tiles, first in this list, held workgroups for up to a tile's time.  us in the old order /
  // this: 14 tokens of 2880 x 2880, top 4 of 32, 28 experts with rows, 153.6 / 141.0; 10 145.8 / 141.3; 20, 29 experts, 156.6 / 143.0;
  // 2000 264.1 / 261.6; 4000 419.8 / 415.2; 8192 752 / 745.  With 31 of the 32 experts, 20 to 33 tokens, it costs 162.0 / 163.0; 130
  // random layers 0.2 % on average.  (Launches of quarters are one turn of the chip: one token 34.6 / 35.8.  Parts are rotated:
  // 447 random layers 0.6 % longer by it.)
  MOK_SCHED_FN int rotated(int q, int d, int item) const {
    const int first = share(q, d), end = share(q + 1, d);
    const int e = MOK_SCHED_COUNT(g.num_experts, [&](int x) { return tab.tile_begin[x] * down_cols <= first; }) - 1;  // of item `first`
    const int next = MOK_SCHED_UNIFORM(tab.tile_begin[e + 1]) * down_cols;  // the next expert's first item
    if (MOK_SCHED_UNIFORM(tab.tile_begin[e]) * down_cols == first || next >= end) return item;
    const int at = item + next - first;
    return at < end ? at : at - (end - first);
  }

  // item i of list q -> task.  `cursor` is the expert of the item this workgroup decoded last: a workgroup's items
  // come in growing order as long as it stays in one GEMM (down tiles: up to where a rotated list wraps), so the search usually
  // ends where it starts.
  MOK_SCHED_FN MokGemmTask decode(int q, int i, int& cursor) const {
    const int gu = gate_up_items(), d = down_items();
    const int mine = share(q + 1, gu) - share(q, gu);
    const bool gate_up = i < mine;
    int item = gate_up ? share(q, gu) + i : share(q, d) + i - mine;  // in the sequence of its GEMM's items
    if (!gate_up && gu != 0 && down_cut == 0) item = rotated(q, d, item);
    const int cut = gate_up ? gate_up_cut : down_cut;                      // a column tile's parts are neighbours
    const int idx = item >> cut, part = item - (idx << cut);
    const int cols = gate_up ? gate_up_cols : down_cols;
    // last e with tile_begin[e] * cols <= idx: it has row tiles, since tile_begin[e + 1] * cols > idx
    // (a workgroup's next item is usually the same expert's)
    int lo = cursor;
    if (tab.tile_begin[lo] * cols > idx || (lo + 1 < g.num_experts && tab.tile_begin[lo + 1] * cols <= idx))
      lo = MOK_SCHED_COUNT(g.num_experts, [&](int e) { return tab.tile_begin[e] * cols <= idx; }) - 1;
    cursor = lo;
    const int e = MOK_SCHED_UNIFORM(lo);
    const int t0 = tab.tile_begin[e], t1 = tab.tile_begin[e + 1];
    const int local = idx - t0 * cols;
    const int col = local / (t1 - t0);
    const int tile = t0 + local - col * (t1 - t0);  // row tile, counted over all experts
    const int first = tab.row_begin[e] + (tile - tab.tile_begin[e]) * TILE_X;
    const bool both = (g.op & MOK_FWD_OP_MASK) == MOK_FWD_BOTH;
    // wave-uniform by construction; say so, so that the task lives in scalar registers
    MokGemmTask t;
    t.op = gate_up ? MOK_GEMM_FWD_ROUTED_GATE_UP : MOK_GEMM_FWD_ROUTED_DOWN;
    t.expert = e;
    t.row_begin = MOK_SCHED_UNIFORM(first);
    t.row_end = MOK_SCHED_UNIFORM(tab.row_begin[e + 1]);
    t.col_begin = MOK_SCHED_UNIFORM(((col << cut) + part) * ((gate_up ? gate_up_width : down_width) >> cut));
    t.task_idx = MOK_SCHED_UNIFORM(q << 24 | i);
    t.counter_idx = MOK_SCHED_UNIFORM(both ? tile : -1);
    t.wait_target = gate_up ? 0 : gate_up_cols << gate_up_cut;
    t.flags = (uint32_t)MOK_SCHED_UNIFORM(cut != 0 ? MOK_TASK_QUARTER : down_width == PART_COLS ? MOK_TASK_PART : 0);
    return t;
  }
};

}  // namespace mok_framework

#endif
