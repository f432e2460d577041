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

// A quarter takes a fourth of a tile's steps; it costs a start, the sum of its waves' parts and an end, and each workgroup more a
// little at the launch's start and end.  So the gain grows with the contraction's slots n and the loss with the launch's tasks
// after the cut.  us cut / us whole of 1360 random layers (contractions of 4 to 45 slots, 1 to 32 active experts, 13 to 60 us),
// down tiles cut, by the tasks then:
//   n 4-5    up to 64 tasks 1.04, 65-128 1.05, 129-256 1.11         n 6-7    up to 64 1.00, 65-128 1.01, 129-256 1.09
//   n 8-9    up to 64 0.99, 65-128 1.01, 129-256 1.08               n 10-13  up to 64 1.00, 65-128 1.02, 129-192 1.04
//   n 14-19  up to 64 0.98, 65-128 0.99, 129-192 1.01, 193-256 1.05
//   n 24-31  up to 192 0.96, 193-240 1.00, 241-384 1.02             n 32-39  up to 240 0.94, 241-290 0.97, 290-430 0.99
//   n 40-45  up to 240 0.91, 241-290 0.94, 291-430 0.97
// and cut gate/up tiles against the better of the other two, n of their contraction: n 8-9 up to 64 1.00, 65-128 1.03; n 14-19 up
// to 128 0.98, 129-192 1.02; n 20-45 up to 64 0.90, 65-128 0.93, 129-192 0.98, 193-256 1.01, 257-400 1.07: the same line serves
// both, and the two lines added where only both together pay.  The line lies above where down tiles alone break even between 10
// and 19 slots because of the launches that cut both.  Below 5 slots (three of a narrow tile's four waves have little or nothing to
// multiply) nothing is cut for that contraction: 64 x 64, 4 rows, 11.1 us whole, 12.4 cut; 256 x 128, 3 rows, 12.9 / 15.0; 520
// layers, 320 of them of contractions up to 12 slots, take 1.3 % less on average than with a line of 4 n + 12 from one slot on,
// 17 % at best and 7 % more at worst (one row of 256 x 384).  From 5 to 9 slots small launches of one or two experts gain by
// cutting both: 512 x 256, one row, 15.9 / 14.0.  More quarters of a GEMM than run at once take a second turn, whose start costs more than the finer cut gives.
constexpr int cut_line(int slots) { return slots < 5 ? 0 : slots < 10 ? 4 * slots + 12 : 7 * slots + 40; }
// Where whole tiles take two turns of the chip already, quarters of down tiles that end within them fill the second one evenly:
// 16 experts of 320 x 2432, 36 tokens, 304 + 32 tiles: 32.1 us whole, 29.3 as 304 + 128 tasks.  A third turn loses that: 576 x
// 2880, 112 tokens, 368 + 48: 38.0 whole, 46.2 as 368 + 192.
constexpr bool quarters_fill_the_second_turn(int gate_up, int down) {
  return gate_up + down > CHIP && gate_up + 4 * down <= 2 * CHIP;
}

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
  const bool down_pays = gate_up + 4 * down <= down_line || quarters_fill_the_second_turn(gate_up, down);
  const bool both_pay = 4 * gate_up <= CHIP && 4 * gate_up + 4 * down <= gate_up_line + (down_pays ? 0 : down_line);
  if (down_pays || both_pay) c.down = 2;
  if (both_pay) c.gate_up = 2;
  return c;
}

// Launches of more rows: every column tile is parts of 64 columns (MOK_TASK_PART) where an expert has more than 64 rows on average,
// all the parts of each GEMM run at once, and these take little time in all.  A layer of few column tiles leaves most of the chip
// idle, and a launch takes as long as one tile: its steps, which wait for 16 MFMAs each, and an epilogue of 128 x 128 values a wave.
// A part has half the MFMAs and epilogue (gate/up) or a quarter (down), spread over waves of 64 rows; but a step of it takes a
// little longer than one of the whole tile's placed loop, the more so the more parts ask for loads.  So the gain is a fixed one, and
// the loss grows with the two contractions' steps and with the steps of all parts of a GEMM (row tiles x columns x contraction, the
// same number for either): the line is fitted to us parts - us whole.  us parts / us whole of 836 random layers of 128 to 2880
// columns, 1 to 32 experts, by what is compared with PART_STEPS:
//   up to 3000 0.84 (1.02 at most), 6000 0.90 (1.04), 9000 0.94 (1.04), 11000 0.97 (1.06), 14000 0.99 (1.05), above 1.03 (1.09)
// 448 x 704, top 2 of 8, 257 tokens 33.4 / 27.6, 509 36.0 / 27.9, 2000 38.3 / 32.3; 256 x 256, top 1 of 4, 300 tokens 23.4 / 19.4;
// 704 x 448, 600 tokens of one expert in four 34.4 / 26.1; 2048 x 512, 400 tokens 45.4 / 40.7; 1664 x 2752, 329 rows of four
// experts 67.3 / 60.4 (whole / parts); 2880 x 2880, 515 rows of one expert 71.2 / 76.8.  With 64 output columns the down tiles are
// as narrow already, and whole gate/up tiles take a single step: 41 layers of up to 768 columns of `hidden` 0.97, 50 of more 1.04,
// up to 1.14 (64 x 1728, 1287 rows of three experts 32.6 / 37.2).
// With 16 to 64 rows on average tiles are mostly small ones already, which parts only make more of: 140 tokens of the first layer
// 19.6 / 22.4, of 640 x 2560 with 50 rows an expert 27.1 / 34.3.
constexpr int PART_COLS = 64;
constexpr int PART_STEPS = 14000;
constexpr bool parts_for(long long rows, int experts, int row_tiles, int gate_up_parts, int down_parts) {
  return rows > 64 * (long long)experts && row_tiles * gate_up_parts <= CHIP && row_tiles * down_parts <= CHIP &&
         (down_parts > 1 || gate_up_parts <= 12) &&
         row_tiles * gate_up_parts * down_parts + 120 * (gate_up_parts + down_parts) <= PART_STEPS;
}
}  // namespace mok_framework

#endif
