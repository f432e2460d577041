// When a launch of few rows cuts its column tiles in four.  One rule for the kernel, which knows each expert's rows, and the
// host, which sizes the grid and knows their sum.  Plain constexpr C++ on integers.
#ifndef PIPELINK_MOK_FRAMEWORK_CUT_HPP
#define PIPELINK_MOK_FRAMEWORK_CUT_HPP

namespace mok_framework {
constexpr int NARROW_ROWS = 32;  // routed rows a quarter of a column tile (MOK_TASK_QUARTER) holds at most
constexpr int CHIP = 256;        // workgroups that run at once (one per compute unit)

// a column tile of each GEMM is 2^cut tasks (one or four)
struct Cut {
  int gate_up, down;
};

// A quarter streams a fourth of a tile's weights, at what one compute unit reaches whatever the others do (about 40 GB/s); it
// costs a start, the sum of its waves' parts and an end, and each workgroup more a little at the launch's start and end.  So
// the gain grows with the contraction's slots n and the loss with the launch's tasks after the cut.  us cut / us whole over
// 2746 random layers (contractions of 1 to 45 slots, 1 to 32 active experts, 13 to 60 us), down tiles cut:
//   n 4-5    up to 32 tasks 0.96, 33-64 0.99, 65-128 1.03, 193-256 1.13
//   n 6-7    up to 64 0.95, 65-128 1.00, 193-256 1.04
//   n 8-9    up to 64 0.90, 65-128 0.97 (one of 11 above 1.01), 129-192 1.00, 257-400 1.09
//   n 10-13  up to 128 0.91, 129-192 0.98, 257-400 1.06
//   n 14-19  up to 256 0.88, 257-400 0.95 (up to 1.03)        n 20-45  up to 400 0.79 (0.98 at most)
// and with n of the gate/up GEMM and both cut, against down tiles only: n 4-5 0.97 / 1.00 / 1.06, n 8-9 0.91 / 0.98, n 10-13 up
// to 192 0.91, n 14-45 up to 400 0.80: the same line serves both, and the two lines added where only both together pay.  With
// it 0.902 on average, none above 1.015; the better of the three layouts each time would be 0.891.  (Every launch that fits one
// turn cut, whatever n: up to 1.4.)  More quarters of a GEMM than run at once take a second turn, whose start costs more than
// the finer cut gives: one token of 2880 x 2880, top 4 of 32, is 92 gate/up and 48 down tiles: 53.2 us whole, 44.2 with the
// down tiles cut, 49.4 with both (368 and 192 quarters).
constexpr int cut_line(int slots) { return 16 * slots - 40; }

// row_tiles: of all experts, none of which has more than NARROW_ROWS rows.  (From the numbers of both GEMMs whatever a launch
// runs: one launch and two give the same sums.)  The contraction's slots follow from the other GEMM's columns: 64 a slot, 256
// down columns or 128 gate/up columns a tile.
// `rows` in all: where an expert holds 16 on average, one of them usually holds more than 32, and a grid with room for quarters
// would be idle workgroups (a layer of 448 x 704, top 2 of 8, 110 to 128 tokens: 20.5 us with 72 workgroups, 22.1 with 256).
constexpr Cut cut_for(long long rows, int experts, int row_tiles, int gate_up_cols, int down_cols) {
  Cut c{0, 0};
  if (rows > 16 * (long long)experts) return c;
  const int gate_up = row_tiles * gate_up_cols, down = row_tiles * down_cols;
  const int gate_up_line = cut_line(4 * down_cols - 3), down_line = cut_line(2 * gate_up_cols - 1);
  if (4 * down > CHIP) return c;
  // (the parts of a gate/up tile share cache lines of `hidden`, which only narrow down tiles read at device scope: gate/up tiles
  // are cut only where down tiles are)
  const bool down_pays = gate_up + 4 * down <= down_line;
  const bool both_pay = 4 * gate_up <= CHIP && 4 * gate_up + 4 * down <= gate_up_line + (down_pays ? 0 : down_line);
  if (down_pays || both_pay) c.down = 2;
  if (both_pay) c.gate_up = 2;
  return c;
}

// Launches of more rows: every column tile is parts of 64 columns (MOK_TASK_PART) if all the parts of each GEMM run at once and
// an expert has more than 64 rows on average.  A layer of few column tiles leaves most of the chip idle, and a launch takes as
// long as one tile: its steps, which wait for 16 MFMAs each, and an epilogue of 128 x 128 values a wave.  A part has half the
// MFMAs and epilogue (gate/up) or a quarter (down), spread over waves of 64 rows.  us whole / parts: 448 x 704, top 2 of 8, 257
// tokens 33.4 / 27.6, 509 36.0 / 27.9, 2000 38.3 / 32.3; 256 x 256, top 1 of 4, 300 tokens 23.4 / 19.4; 704 x 448, 600 tokens of
// one expert in four 34.4 / 26.1; 2048 x 512, 400 tokens 45.4 / 40.7; 2880 x 768, 500 tokens 50.1 / 49.9 (long contractions: the
// whole tile's placed loop makes up for it).  With 16 to 64 rows on average tiles are mostly small ones already, which parts only
// make more of: 140 tokens of the first layer 19.6 / 22.4, of 640 x 2560 with 50 rows an expert 27.1 / 34.3.
constexpr int PART_COLS = 64;
constexpr bool parts_for(long long rows, int experts, int row_tiles, int gate_up_parts, int down_parts) {
  return rows > 64 * (long long)experts && row_tiles * gate_up_parts <= CHIP && row_tiles * down_parts <= CHIP;
}
}  // namespace mok_framework

#endif
