// Package fa.core: flash-attention forward for one tile of 128 queries of one head; compiled by core_half.hip with
// FA_HALF_TILES, of 64 (half tiles).
//
// Orientation.  Scores are computed transposed, S^T = K . Q^T (keys are the MFMA rows, queries the
// columns), so that a lane holds ONE query (column lane % 32) and 16 of the block's 32 keys: row maxima
// and sums are in-register reductions plus one exchange between lane l and l ^ 32.  The probabilities
// are then, register for register, the B operand of O^T += V^T . P^T -- the contraction index of an MFMA
// is only a summation order, and V^T is read from LDS in the order the registers hold the keys:
//   group g of 16 keys (registers 8g .. 8g+7 of a 32-key score tile), lane half h = lane / 32:
//   elements 0-3 = keys 16g + 4h + 0..3, elements 4-7 = keys 16g + 8 + 4h + 0..3.
// K and V both go global -> LDS as stored (row-major [key][d], the 16-byte chunks of a row permuted so that the
// reads below meet no bank conflict: k_place / v_place).  K rows are the A operand of the first product as they are.  The A operand of the
// second product wants, per lane, four consecutive KEYS at one d -- a column of the V tile: that is what
// ds_read_b64_tr_b16 delivers.  In a group of 16 lanes, lane i hands in the address of 4 consecutive d
// (8 bytes) and lane j receives element j % 4 of the data of lanes j / 4, j / 4 + 4, j / 4 + 8, j / 4 + 12
// (measured with a probe); so lane i points at key kbase + i / 4, d = dbase + 4 (i % 4), and lane j gets keys
// kbase .. kbase + 3 at d = dbase + j.
//
// A tile is a chain of key blocks; a grid that leaves most SIMDs with one wave or none takes as long as the longest chain,
// with nothing beside it.  With half tiles waves 0 and 1 have 32 queries each and the first 32 keys of every block, waves 2
// and 3 the same queries and the other 32 keys: twice the workgroups, each block half as long for a wave.  The two halves
// of a query's sum meet through LDS at the end.  us, whole / half tiles: B 1, 32 heads, S 1152, window 700 (288 tiles) 25.9 /
// 20.6; S 512 causal (128 tiles) 14.5 / 11.8; 8 heads, S 4096 (256 tiles) 82.1 / 60.9; 32 heads, S 2048 (512 tiles) 54.1 /
// 51.8, S 512 of 128 heads (512 tiles) 19.9 / 24.5; B 4, S 4096 (4096 tiles) 550 / 655: with two waves on every SIMD a key block costs its loads twice.
//
// Two LDS buffers per operand: block i + 1 is in flight while block i is multiplied; one barrier per block.
#include <pipelink/stage.hpp>
#ifndef FA_HALF_TILES
#define FA_HALF_TILES 0
#endif
#ifndef PIPELINK_EMIT
#include <hip/hip_runtime.h>
#include <type_traits>
#include "include/fa_abi.h"
#include "include/fa_order.hpp"

extern "C" __device__ int pipelink_fa_kv();  // byte offset of the K / V^T buffers in dynamic LDS
extern "C" __device__ int pipelink_call_mask_key_count(const void* view, int q_first, int q_last);
extern "C" __device__ int pipelink_call_mask_key_begin(const void* view, int q_first, int q_last);
extern "C" __device__ int pipelink_call_mask_all_visible(const void* view, int q_first, int q_last, int k_first, int k_last);
extern "C" __device__ int pipelink_call_mask_visible(const void* view, int q, int k);

extern __shared__ __attribute__((aligned(1024))) unsigned char pipelink_smem[];

namespace fa_core {
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v8f __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int K_BYTES = FA_K_BLOCK * FA_D * 2;     // 16 KB: [64 keys][256 bytes], the same for V
constexpr int BUF_BYTES = 2 * K_BYTES;
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s* lds_v4s;
constexpr float MASKED = -1.0e30f;
constexpr float RESCALE_SLACK = 8.0f;  // log2 units

// Where the 16-byte chunk `chunk` of a key's row stands in its 256-byte LDS row.  K is read one key per lane, 16 lanes
// = 16 consecutive keys at one chunk: the 16 rows must put that chunk in 16 different places.  V is read in columns,
// 32 lanes = 4 consecutive keys x 4 consecutive chunks: the 4 rows must put each group of 4 chunks in a different place.
__device__ __forceinline__ int k_place(int key, int chunk) { return chunk ^ (key & 15); }
__device__ __forceinline__ int v_place(int key, int chunk) { return chunk ^ (4 * (key & 3)); }

// one 64-key block of K or V -> LDS: 64 keys x 256 B; one load instruction of a wave moves 4 keys (1 KB)
template <bool IS_V>
__device__ __forceinline__ void issue_block(__amdgpu_buffer_rsrc_t src, uint32_t first_key_byte, unsigned char* dst, int wave, int lane) {
  const int kr = lane >> 4, pos = lane & 15;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int key = (wave * 4 + j) * 4 + kr;  // 0..63
    const uint32_t off = first_key_byte + (uint32_t)key * (FA_D * 2) + 16u * (uint32_t)(IS_V ? v_place(key, pos) : k_place(key, pos));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_ptr)(dst + (wave * 4 + j) * 1024), 16, (int)off, 0, 0, 0);
  }
}
// The transposing read: in a group of 16 lanes, lane i hands in the address of 4 consecutive d of key kbase + i / 4
// and lane j receives keys kbase .. kbase + 3 at d = dbase + j.  (The parameter is restricted for what inlining makes of it, alias
// scopes on the read: one of which the compiler knows nothing waits for every load into LDS there is, the next block's too.)
__device__ __forceinline__ v4s read_v_piece(const unsigned char* __restrict__ at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(const_cast<unsigned char*>(at)));
}
// A value of this lane and the one of lane ^ 32, without a trip through the LDS: after the swap the first result
// holds the lower half-wave's values in both halves, the second the upper half-wave's.
__device__ __forceinline__ float max_with_other_half(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_with_other_half(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

constexpr bool split = FA_HALF_TILES;
constexpr int TILE_QUERIES = split ? FA_Q_TILE / 2 : FA_Q_TILE;

// one tile; `index` counts them with the longest ones first
__device__ __forceinline__ void attend(const FaCoreParams& p, const pipelink_host_view& view, uint32_t index) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const auto [tile, bh, group] = fa_order::tile_of(index, p.batch, p.q_heads, p.kv_heads, p.seq / TILE_QUERIES);
  const int q0 = tile * TILE_QUERIES, qw = q0 + 32 * (split ? wave & 1 : wave);  // the wave's first query
  const int key0 = split ? 32 * (wave >> 1) : 0;                                 // its first key of every block
  const uint32_t head_bytes = (uint32_t)p.seq * FA_D * 2;
  const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(p.k) + (int64_t)group * p.seq * FA_D, 0, (int)head_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(p.v) + (int64_t)group * p.seq * FA_D, 0, (int)head_bytes, 0x00020000);
  unsigned char* buf = pipelink_smem + pipelink_fa_kv();

  // this lane's query row as the B operand of S^T = K . Q^T: 16 bytes per 16-element step of d
  v8bf qf[8];
  {
    const uint16_t* qrow = p.q + ((int64_t)bh * p.seq + qw + l32) * FA_D;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) qf[kk] = __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(qrow + 16 * kk + 8 * half));
  }
  v16f o[4];  // O^T: [d block][16 d of the block] for this lane's query
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
  float row_max = MASKED, row_sum = 0.0f;
  // (in a register for good: read where it is used, it is loaded again in every block, behind the block's barrier)
  const float scale_log2e = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, p.scale_log2e)));
  bool seen = false;  // this lane's query has met a key it may see (decided on unscaled scores: the scale is the caller's)

  // the mask package says which stretch of keys the tile's queries may see at all: blocks [first_block, blocks)
  const int keys = pipelink_call_mask_key_count(&view, q0, q0 + TILE_QUERIES - 1);
  const int first_block = pipelink_call_mask_key_begin(&view, q0, q0 + TILE_QUERIES - 1) / FA_K_BLOCK;
  const int blocks = (keys + FA_K_BLOCK - 1) / FA_K_BLOCK;
  const int wave_keys = pipelink_call_mask_key_count(&view, qw, qw + 31), wave_begin = pipelink_call_mask_key_begin(&view, qw, qw + 31);
  // Schedule.  Two LDS buffers per operand: block i + 1 is in flight while block i is multiplied; one barrier per
  // block.  LDS reads are issued in batches ahead of the MFMAs that use them (a read costs a few hundred clocks of
  // latency, an MFMA 32): all 16 K fragments of a block before its first score MFMA, the V pieces of the next group
  // of 16 keys before the MFMAs of the present one, those of the first group before the softmax.
  const int li = lane & 15, dgroup = 16 * ((lane >> 4) & 1);  // position in the 16-lane group, the group's first d in a 32-row block
  // LDS addresses, kept few: a K fragment is at [key = 32 t + l32][chunk 2 kk + half] -> this lane's 8 places in
  // its row (the tile t is an immediate offset); a V column piece is at [key][chunk 4 db + c] -> 4 places per lane.
  // (as pointers into both buffers of the pair: the loop adds nothing to them)
  const unsigned char* k_at[2][8];
#pragma unroll
  for (int pb = 0; pb < 2; ++pb)
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) k_at[pb][kk] = buf + pb * BUF_BYTES + (key0 + l32) * (FA_D * 2) + 16 * k_place(l32, 2 * kk + half);
  const int v_key = 4 * half + (li >> 2);  // the key (within a group of 16) this lane points at for the transposing read
  const unsigned char* v_at[2][4];
#pragma unroll
  for (int pb = 0; pb < 2; ++pb)
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const int d = 32 * db + dgroup + 4 * (li & 3);
      v_at[pb][db] = buf + pb * BUF_BYTES + K_BYTES + (key0 + v_key) * (FA_D * 2) + 16 * v_place(v_key, d >> 3) + 2 * (d & 4);
    }
  // the 8 pieces (4 blocks of d x two halves of 8 keys) of the group of 16 keys that starts at key `first`
  auto read_v_group = [&](int pb, int first, v4s (&piece)[8]) {
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      // rows first + v_key and 8 further on: (key & 3) is the same, so is the place in the row
      piece[2 * db] = read_v_piece(v_at[pb][db] + first * (FA_D * 2));
      piece[2 * db + 1] = read_v_piece(v_at[pb][db] + (first + 8) * (FA_D * 2));
    }
  };
  issue_block<false>(kres, (uint32_t)first_block * FA_K_BLOCK * FA_D * 2, buf, wave, lane);
  issue_block<true>(vres, (uint32_t)first_block * FA_K_BLOCK * FA_D * 2, buf + K_BYTES, wave, lane);
  // one block of 64 keys, NT tiles of 32 of them this wave's; PB = (i - first_block) % 2 (the buffer pair) is a compile-time
  // constant so that the address tables are registers
  auto block = [&](int i, auto pair, auto tiles) {
    constexpr int PB = decltype(pair)::value, NT = decltype(tiles)::value;
    // blocks i of K and V have landed, and the buffers of block i - 1 are free.  (The barrier itself waits for no global -> LDS
    // load, and a wave that left the last block early, because none of its queries sees a key of it, has met no other wait.)
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    if (i + 1 < blocks) {
      issue_block<false>(kres, (uint32_t)(i + 1) * FA_K_BLOCK * FA_D * 2, buf + (1 - PB) * BUF_BYTES, wave, lane);
      issue_block<true>(vres, (uint32_t)(i + 1) * FA_K_BLOCK * FA_D * 2, buf + (1 - PB) * BUF_BYTES + K_BYTES, wave, lane);
    }
    const int k0 = i * FA_K_BLOCK + key0;
    if (k0 >= wave_keys || k0 + 32 * NT <= wave_begin) return;  // no query of this wave sees a key of this block: only the loads and the barrier
    // ---- S^T = K . Q^T : NT 32-key tiles -----------------------------------------------------------
    v16f s[NT];
    v4s piece[2][8];
    {
      v4i kf[NT][8];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) kf[t][kk] = *reinterpret_cast<const v4i*>(k_at[PB][kk] + t * 32 * (FA_D * 2));
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(2);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, kf[t][kk]), qf[kk], s[t], 0, 0, 0);
      }
      read_v_group(PB, 0, piece[0]);  // on their way during the softmax
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- mask, online softmax (in units of log2: exp2(x * scale_log2e - max)) -------------------------------
    const int query = qw + l32;
    const bool all = pipelink_call_mask_all_visible(&view, qw, qw + 31, k0, k0 + 32 * NT - 1);
    if (!all) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k0 + 32 * t + 8 * (r / 4) + 4 * half + r % 4;
          if (!pipelink_call_mask_visible(&view, query, key)) s[t][r] = MASKED;
        }
    }
    float block_max = MASKED;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) block_max = fmaxf(block_max, s[t][r]);
    block_max = max_with_other_half(block_max);
    // once a query has seen a key its maximum is a real score, and a masked entry (-1e30) turns into exp2(-huge) = 0
    // by itself
    // The reference point of the exponentials only moves when a score exceeds it by more than 2^RESCALE_SLACK: until
    // then probabilities may be as large as that (harmless in fp32 sums and bf16 operands, and the final division
    // takes it out again), and the accumulated output and sum need no rescaling -- which they otherwise would
    // in most blocks, because some query of the wave sees a new maximum.
    const float top = block_max * scale_log2e;
    const float new_max = top > row_max + RESCALE_SLACK ? top : row_max;
    const float alpha = __builtin_amdgcn_exp2f(row_max - new_max);
    row_max = new_max;
    // a query that has not seen a key yet (a window mask: the block's keys are all too old for it) has no real maximum
    // to lean on: its exponentials are taken against +huge instead, which makes every one of them 0
    seen = seen || block_max > 0.5f * MASKED;
    const float reference = seen ? new_max : -MASKED;
    float block_sum = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r], scale_log2e, -reference));
        s[t][r] = e;
        block_sum += e;
      }
    block_sum = sum_with_other_half(block_sum);
    row_sum = row_sum * alpha + block_sum;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {  // once the maxima have settled nothing needs rescaling
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
    }
    // ---- O^T += V^T . P^T : 2 NT groups of 16 keys, four 32-row blocks of d ----------------------------
    __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int gi = 0; gi < 2 * NT; ++gi) {
      const int t = gi >> 1, g = gi & 1;
      if (gi + 1 < 2 * NT) read_v_group(PB, 16 * (gi + 1), piece[(gi + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      v8f pf;
#pragma unroll
      for (int e = 0; e < 8; ++e) pf[e] = s[t][8 * g + e];
      const v8bf pb = __builtin_convertvector(pf, v8bf);
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const v2i lo2 = __builtin_bit_cast(v2i, piece[gi & 1][2 * db]), hi2 = __builtin_bit_cast(v2i, piece[gi & 1][2 * db + 1]);
        const v4i raw = {lo2.x, lo2.y, hi2.x, hi2.y};
        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, raw), pb, o[db], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
  };
  auto stream = [&](auto tiles) {
    for (int i = first_block; i < blocks; i += 2) {
      block(i, std::integral_constant<int, 0>{}, tiles);
      if (i + 1 < blocks) block(i + 1, std::integral_constant<int, 1>{}, tiles);
    }
  };
  if constexpr (split) {
    stream(std::integral_constant<int, 1>{});
    // the other half of the keys: waves 2 and 3 hand what they have to waves 0 and 1.  A half that has seen no key for a
    // query has no maximum, and nothing to add.
    if (!seen) row_max = MASKED;
    unsigned char* const part = buf + (wave & 1) * (17 * 1024);  // 16 x 1 KB of O^T, then the maxima and the sums
    __syncthreads();  // nobody reads keys or values any more
    if (wave >= 2) {
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const v4f f = {o[db][4 * q4], o[db][4 * q4 + 1], o[db][4 * q4 + 2], o[db][4 * q4 + 3]};
          *reinterpret_cast<v4f*>(part + (4 * db + q4) * 1024 + lane * 16) = f;
        }
      *reinterpret_cast<float*>(part + 16 * 1024 + lane * 8) = row_max;
      *reinterpret_cast<float*>(part + 16 * 1024 + lane * 8 + 4) = row_sum;
    }
    __syncthreads();
    if (wave >= 2) return;
    const float other_max = *reinterpret_cast<const float*>(part + 16 * 1024 + lane * 8);
    const float other_sum = *reinterpret_cast<const float*>(part + 16 * 1024 + lane * 8 + 4);
    const float top = fmaxf(row_max, other_max);
    const float mine = __builtin_amdgcn_exp2f(row_max - top), others = __builtin_amdgcn_exp2f(other_max - top);
    row_sum = row_sum * mine + other_sum * others;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const v4f f = *reinterpret_cast<const v4f*>(part + (4 * db + q4) * 1024 + lane * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[db][4 * q4 + e] = o[db][4 * q4 + e] * mine + f[e] * others;
      }
  } else {
    stream(std::integral_constant<int, 2>{});
  }
  // ---- O[b][query][h][d] = O^T / row_sum, bf16 ------------------------------------------------------------
  const float inv = row_sum > 0.0f ? __builtin_amdgcn_rcpf(row_sum) : 0.0f;
  const int b = (uint32_t)bh / (uint32_t)p.q_heads, h = bh - b * p.q_heads;
  uint16_t* orow = p.o + ((int64_t)b * p.seq + qw + l32) * ((int64_t)p.q_heads * FA_D) + (int64_t)h * FA_D;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const v4f f = {o[db][4 * q4] * inv, o[db][4 * q4 + 1] * inv, o[db][4 * q4 + 2] * inv, o[db][4 * q4 + 3] * inv};
      const v4bf packed = __builtin_convertvector(f, v4bf);
      *reinterpret_cast<v2i*>(orow + 32 * db + 8 * q4 + 4 * half) = __builtin_bit_cast(v2i, packed);
    }
}
}  // namespace fa_core

extern "C" __device__ void fa_core_role_core(const void* params, unsigned variant) {
  (void)variant;
  using namespace fa_core;
  const FaCoreParams& p = *static_cast<const FaCoreParams*>(params);
  const pipelink_host_view view{params, nullptr};
  const uint32_t tiles = (uint32_t)(p.batch * p.q_heads) * (uint32_t)(p.seq / TILE_QUERIES);
  // The image a session is given beside its link may be of the other tile size than the link its grid was made for: whole
  // tiles leave workgroups of a larger grid idle, half tiles take several of a smaller one.
  uint32_t index = blockIdx.x;
  if (index >= tiles) return;
  for (;;) {
    attend(p, view, index);
    if (!split || tiles - index <= gridDim.x) break;
    index += gridDim.x;
    __syncthreads();  // nobody reads this tile's keys, values or partial sums any more
  }
}
#else
#include "include/fa_abi.h"
#endif

#if FA_HALF_TILES
PL_STAGE("fa.core", "0.1.0-half");
#else
PL_STAGE("fa.core", "0.1.0");
#endif
PL_PARAMS(FaCoreParams);
PL_ROLE(core, fa_core_role_core, 4);
PL_TOPOLOGY(false, "static");
PL_VARIANT(0, {});
PL_CALL(mask_key_count, "mask_key_count",
        "extern \"C\" __device__ int pipelink_call_mask_key_count(const void* view, int q_first, int q_last);");
PL_CALL(mask_key_begin, "mask_key_begin",
        "extern \"C\" __device__ int pipelink_call_mask_key_begin(const void* view, int q_first, int q_last);");
PL_CALL(mask_all_visible, "mask_all_visible",
        "extern \"C\" __device__ int pipelink_call_mask_all_visible(const void* view, int q_first, int q_last, int k_first, int k_last);");
PL_CALL(mask_visible, "mask_visible",
        "extern \"C\" __device__ int pipelink_call_mask_visible(const void* view, int q, int k);");
// two buffers of (K block 16 KB + V block 16 KB)
PL_CLAIM("pipelink_fa_kv", "smem", 2 * 2 * (64 * 128 * 2), 1024, "kernel");
PL_USES("pipelink_fa_kv");
// two workgroups per CU (two waves per SIMD, 256 registers per lane each): one multiplies while the other
// is in its softmax or waits at its barrier; 2 x 67.6 KB of LDS fit
PL_FACT("launch.waves_per_simd", 2);
#if FA_HALF_TILES
PL_FACT("fa.core.tile_queries", 64);
#else
PL_FACT("fa.core.tile_queries", 128);
#endif
PL_PRELUDE("include/fa_abi.h");
PL_EMIT_MAIN()
