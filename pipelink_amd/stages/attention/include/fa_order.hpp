// Which tile a workgroup of the flash-attention core takes.  Plain C++ on integers, so that a host compiler takes it too.
#ifndef PIPELINK_FA_ORDER_HPP
#define PIPELINK_FA_ORDER_HPP

#ifndef FA_ORDER_FN
#define FA_ORDER_FN __device__ __forceinline__
#endif

namespace fa_order {
constexpr unsigned XCDS = 8;
struct Tile {
  int tile, bh, group;  // query tile; batch * q_heads + head; batch * kv_heads + KV head
};

// Causal tiles cost in proportion to their position: the latest (longest) tiles of every head come first, so that the grid does
// not end on a few long ones.  Workgroups are dealt to the XCDs in turn, each with an L2 of its own: the query heads that share a
// KV head are kept on one XCD (on 8 / sets of them where the KV heads of the batch are no multiple of 8), where its L2 reads their
// keys and values once.  Dealt head by head, a group of four heads was on four XCDs.  us head by head / this: B 4, 32 / 8 heads, S
// 4096 574 / 550, with a window of 1024 320 / 299; S 1024 58.4 / 54.9; S 512 20.5 / 19.9; B 3, 32 / 4 heads, S 2048 130 / 124; B 4, 16 /
// 16 heads, S 2048, where no heads share and the orders are the same, 91 / 92.  (Group after group, so that an XCD streams one at a
// time, loses the order of lengths: the last 78 / 104, B 3, 8 / 2 heads, S 4096 103 / 131.)
// (The sets are a power of two, and one set is the order head by head: three divisions and shifts.  With a division by each
// of the set counts the smallest launches took 0.2 us more, S 128 of 32 / 8 heads 6.6 / 6.8.)
FA_ORDER_FN Tile tile_of(unsigned index, unsigned batch, unsigned q_heads, unsigned kv_heads, unsigned q_tiles) {
  const unsigned heads = batch * q_heads, groups = batch * kv_heads, per_kv = q_heads / kv_heads;
  // sets: the largest power of two that divides the groups, at most 8 (1 << log_sets); one where the grid has no eighths
  const unsigned log_sets = heads * q_tiles % XCDS ? 0 : __builtin_ctz(groups | XCDS);
  const unsigned xcd = index % XCDS, at = (index / XCDS * XCDS >> log_sets) + (xcd >> log_sets);  // the at-th tile of its set of groups
  const unsigned set_heads = heads >> log_sets, level = at / set_heads, in_level = at - level * set_heads;
  const unsigned of_set = in_level / per_kv, group = (xcd & ((1u << log_sets) - 1)) + (of_set << log_sets);
  return Tile{(int)(q_tiles - 1 - level), (int)(group * per_kv + in_level - of_set * per_kv), (int)group};
}
}  // namespace fa_order

#endif
