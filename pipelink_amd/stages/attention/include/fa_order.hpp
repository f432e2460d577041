// Which tile a workgroup of the flash-attention core takes.  Plain C++ on integers, so that a host compiler takes it too.
#ifndef PIPELINK_FA_ORDER_HPP
#define PIPELINK_FA_ORDER_HPP

#ifndef FA_ORDER_FN
#define FA_ORDER_FN __device__ __forceinline__
#endif

namespace fa_order {
constexpr int XCDS = 8;
struct Tile {
  int tile, bh;  // query tile; batch * q_heads + head
};

// Causal tiles cost in proportion to their position: the latest (longest) tiles of every head come first, so that the grid does
// not end on a few long ones.  Workgroups are dealt to the XCDs in turn, each with an L2 of its own: the query heads that share a
// KV head are kept on one XCD (on 8 / sets of them where the KV heads of the batch are no multiple of 8), where its L2 reads their
// keys and values once.  Dealt head by head, a group of four heads was on four XCDs.  us before / after: B 4, 32 / 8 heads, S 4096
// 546 / 541, with a window of 1024 321 / 289; S 1024 49.1 / 46.2; S 512 18.8 / 17.6; B 3, 32 / 4 heads, S 2048 111 / 108; B 4, 16 / 16
// heads, S 2048, where no heads share, 78.0 / 77.9.  (Group after group, so that an XCD streams one at a time, loses the order of
// lengths: the last 78 / 104, B 3, 8 / 2 heads, S 4096 103 / 131.)
FA_ORDER_FN Tile tile_of(int index, int batch, int q_heads, int kv_heads, int q_tiles) {
  const int heads = batch * q_heads, per_kv = q_heads / kv_heads, groups = batch * kv_heads;
  if (heads * q_tiles % XCDS != 0) return Tile{q_tiles - 1 - index / heads, index % heads};
  const int sets = groups % XCDS ? groups & -groups : XCDS;  // the largest power of two that divides the groups, at most 8
  const int xcd = index % XCDS, at = index / XCDS * (XCDS / sets) + xcd / sets;  // the at-th tile of its set of groups
  const int set_heads = heads / sets, in_level = at % set_heads;
  return Tile{q_tiles - 1 - at / set_heads, (xcd % sets + sets * (in_level / per_kv)) * per_kv + in_level % per_kv};
}
}  // namespace fa_order

#endif
