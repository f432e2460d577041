// Stage package mok.framework: the persistent worker role.  It owns the schedule (which
// workgroup runs which tile, in which order) and calls the GEMM and activation owners
// through link-generated trampolines; it knows nothing of their tile internals beyond the
// published facts TILE_X / TILE_W.
//
// Plays the part of mok_framework_run in campaigns/mok/port/framework/interp_fwd.cu:26-252
// (task decode :137-214, dependency chain gate/up -> act -> down :174-213).  Not carried over: 2-CTA clusters (no
// gfx950 counterpart) and the comm clusters (single GPU).
//
// One launch runs both GEMMs (op MOK_FWD_BOTH) or one of them.  The tiles are in eight lists, one per XCD (workgroup
// id % 8): list q holds the tiles of an eighth of the routed-row tiles -- the gate/up tiles first, then the down tiles
// of the same rows; within each, expert by expert, column tile by column tile, row tiles innermost, so that
// workgroups that run at the same time share a weight tile and one XCD's L2 sees a contiguous run of experts.  A
// workgroup's first two tiles are fixed by its id; after that the list's queue (a word of the workspace) hands the
// tiles out in list order, one atomic per tile, and a workgroup whose list is handed out asks another list that has tiles left
// (the reference asks the cluster launch control for its next tile, interp_fwd.cu:137-160).  Tiles differ in cost
// (full ones, and those of few rows or few columns, which have a placement of their own), and turns of equal length
// leave the workgroups that drew the full ones tiles behind the others.  A down tile reads rows of `hidden` that the
// gate/up tasks of its row tile write (column tiles, or four parts of each): it waits until the row tile's readiness counter
// (MokCounters) has reached their number.  In every list all gate/up tiles come before the first down tile and the queue hands out
// in that order, gate/up tiles wait for nothing, and a workgroup only ever waits while it holds no unfinished tile:
// so the tiles a wait depends on are finished or running, no wait can last, and each is bounded anyway.
//
// Per workgroup the tiles are software-pipelined: the next tile's row tokens and readiness counter are requested
// behind the current tile's first loads (mok_gemm_fwd's `upcoming`), and its first loads are issued between the
// current tile's mainloop and epilogue.
#include <pipelink/stage.hpp>
#ifndef PIPELINK_EMIT
#include "../include/mok_device.hpp"
#include "schedule.hpp"

extern "C" __device__ int pipelink_mok_fw_sched();  // byte offset of the schedule table in dynamic LDS

extern "C" __device__ void pipelink_call_gemm_init(const void* view);
extern "C" __device__ void pipelink_call_gemm_fini(const void* view);
extern "C" __device__ void pipelink_call_act_init(const void* view);
extern "C" __device__ void pipelink_call_gemm_stage(const void* view, const MokGemmTask*, const MokCounters*);
extern "C" __device__ bool pipelink_call_gemm_ready(const void* view, const MokGemmTask*, const MokCounters*);
extern "C" __device__ void pipelink_call_gemm_wait(const void* view, const MokGemmTask*, const MokCounters*);
extern "C" __device__ void pipelink_call_gemm_prefetch(const void* view, const MokGemmTask*, mok::GemmCarry*);
extern "C" __device__ void pipelink_call_gemm_fwd(const void* view, const MokGemmTask*, const MokCounters*, uint32_t*,
                                                  mok::AccFrag*, const mok::GemmCarry*, const MokGemmTask*);
extern "C" __device__ void pipelink_call_gemm_store(const void* view, const MokGemmTask*, const mok::AccFrag*);
extern "C" __device__ void pipelink_call_act_fwd(const void* view, const MokActTask*, const MokCounters*, uint32_t*,
                                                 const mok::AccFrag*);

extern "C" __device__ int pipelink_call_gemm_placement(const void* view, const MokGemmTask*);
extern "C" __device__ void pipelink_call_gemm_fwd_small(const void* view, const MokGemmTask*, const MokCounters*, uint32_t*,
                                                        mok::AccFrag*, const mok::GemmCarry*, const MokGemmTask*);
extern "C" __device__ void pipelink_call_gemm_store_small(const void* view, const MokGemmTask*, const mok::AccFrag*);
extern "C" __device__ void pipelink_call_act_fwd_small(const void* view, const MokActTask*, const MokCounters*, uint32_t*,
                                                       const mok::AccFrag*);

extern __shared__ __attribute__((aligned(1024))) unsigned char pipelink_smem[];

namespace mok_framework {
static_assert(TILE_X == mok::TILE_X && TILE_W == mok::TILE_W, "the schedule's tile is the GEMM owner's");

// Asks a queue for its next number, without waiting for the answer.  (An addition of one lane is made one of a wave by the
// compiler, which has the answer spread over the lanes at once: 1 to 2 us in front of the next tile's first loads.  A wrapping
// increment it leaves alone.)  us with the addition / this, and the two accesses of LDS that waited for everything, back to back on
// one state: one token of 2880 x 2880, top 4 of 32, 36.3 / 34.8; 27 160.1 / 158.2; 128 167.0 / 164.7; 448 x 704, 60 tokens 19.7 / 18.9.  Full tiles keep
// the addition: there the increment's register is the one that makes the next mainloop wait (2000 tokens 277.0 / 279.5).
__device__ __forceinline__ uint32_t take_one(uint32_t* queue) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_atomic_inc32(queue, 0xFFFFFFFFu, __ATOMIC_RELAXED, "agent");
#else
  return __hip_atomic_fetch_add(queue, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
}

// The queue's answer has arrived.  Said where every wave passes: read only behind a branch of thread 0's, it is on its way for
// ever as far as the compiler can tell, and whichever later code writes its register waits, in the next tile's mainloop too.
__device__ __forceinline__ void arrived(uint32_t answer) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" ::"v"(answer));
#else
  (void)answer;
#endif
}

// inclusive sum over the lanes of a full wave: within rows of 16 lanes, then across them
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// A tile with little to multiply (mok::tile_placement): mainloop, the next tile's first loads, epilogue -- what the
// worker's loop does for a full tile, through the owners' exports for the small placement, and in a function of its
// own that is NOT inlined.  The full tile's mainloop uses every register a lane has and depends on where each value
// lives; compiled into the same function, the small tile's code takes registers from it (values kept across the tile
// loop, 100 to 270 of them spilled).  As a call it has an allocation of its own.  Everything goes in and out by value
// so that nothing of the worker's state has to live in memory.
struct SmallTileResult {
  mok::GemmCarry carry;  // of the next tile, if its prefetch was issued
  int early;             // the next tile's prefetch was issued (its rows were complete)
  uint32_t answer;       // thread 0: what the queue answered (the tile after the next)
};
__device__ __attribute__((noinline)) SmallTileResult small_tile(const void* params, MokGemmTask task, MokGemmTask next,
                                                                int32_t* counter_base, uint32_t* status, uint32_t* queue,
                                                                mok::GemmCarry carry) {
  const pipelink_host_view view{params, nullptr};
  const MokCounters counters{counter_base, status};
  // arguments travel in vector registers: say again that these are the same in every lane
  auto uniform = [](MokGemmTask& t) {
    t.op = __builtin_amdgcn_readfirstlane(t.op);
    t.expert = __builtin_amdgcn_readfirstlane(t.expert);
    t.row_begin = __builtin_amdgcn_readfirstlane(t.row_begin);
    t.row_end = __builtin_amdgcn_readfirstlane(t.row_end);
    t.col_begin = __builtin_amdgcn_readfirstlane(t.col_begin);
    t.task_idx = __builtin_amdgcn_readfirstlane(t.task_idx);
    t.counter_idx = __builtin_amdgcn_readfirstlane(t.counter_idx);
    t.wait_target = __builtin_amdgcn_readfirstlane(t.wait_target);
    t.flags = (uint32_t)__builtin_amdgcn_readfirstlane((int)t.flags);
  };
  uniform(task);
  uniform(next);
  uint32_t phase = 0;
  mok::AccFrag acc;
  pipelink_call_gemm_fwd_small(&view, &task, &counters, &phase, &acc, &carry, &next);
  uint32_t answer = 0;
  if (queue && threadIdx.x == 0) answer = take_one(queue);
  const bool early = next.op != 0 && pipelink_call_gemm_ready(&view, &next, &counters);
  if (early) pipelink_call_gemm_prefetch(&view, &next, &carry);
  if (task.op == MOK_GEMM_FWD_ROUTED_GATE_UP) {
    const MokActTask act{MOK_ACT_FWD_ROUTED, task.row_begin, task.row_end, task.col_begin, task.task_idx, task.counter_idx, task.flags};
    pipelink_call_act_fwd_small(&view, &act, &counters, &phase, &acc);
  } else {
    pipelink_call_gemm_store_small(&view, &task, &acc);
  }
  return SmallTileResult{carry, early ? 1 : 0, answer};
}


// The workgroup's tiles.  PARTS: a launch whose column tiles are cut or parts, all of whose tiles are small ones; without it no task is
// a part, and the compiler leaves out what parts need.  One loop for both costs launches without parts 0.2 to 0.7 us (the
// parts' code between the others' and three times the scalar spills): 448 x 704, 160 tokens 20.4 / 20.7 us, 256 x 2048, 250
// tokens 28.6 / 29.7, 27 tokens of 2880 x 2880 163.9 / 165.5.
template <bool PARTS>
__device__ __forceinline__ void run_tiles(const void* params, const MokFrameworkParams& g, Tables& tab, Schedule sched,
                                          const MokCounters& counters) {
  // (what both loops begin with would otherwise move in front of the choice between them, to be kept in registers through the
  // one that is taken; it saved 24 scalar spills)
  if (PARTS) __builtin_amdgcn_sched_barrier(0);
  const pipelink_host_view view{params, nullptr};
  if (!PARTS) {
    sched.gate_up_cut = sched.down_cut = 0;
    sched.gate_up_width = TILE_W / 2;
    sched.down_width = TILE_W;
  }
  uint32_t phase = 0;

  const int q = blockIdx.x % NUM_XCD;
  const int turn = gridDim.x / NUM_XCD;  // the launch grid is a multiple of NUM_XCD: workgroups per list
  const int items = sched.length(q);
  int i = blockIdx.x / NUM_XCD, cursor = 0;
  if (i < items) {
    MokGemmTask task = sched.decode(q, i, cursor);
    // the first tile has no mainloop in front of it to look ahead from
    pipelink_call_gemm_stage(&view, &task, &counters);
    // what was staged has landed for every wave (the barrier itself waits for no global -> LDS load)
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    bool early = false;  // the prefetch of the tile at the loop's head has been issued
    mok::GemmCarry carry;
    // The tile after this one: the workgroup's second turn.  From there on tiles are handed out by the list's queue (a
    // counter in the workspace), one request per tile, made while the tile before the one before is multiplied: tiles
    // differ in cost (full ones, and those with few rows or few columns), and turns of equal length would leave the
    // workgroups that drew the full ones behind the others by several tiles' time.
    // A workgroup whose list has been handed out goes on with another list that has tiles left (the next one first): the
    // lists are cut by number of tiles, not by cost, and whole XCDs would otherwise end a tile or two before others.
    int list = q;       // the list this workgroup asks
    bool asking = true;  // (a workgroup that has found every list handed out asks no more)
    MokGemmTask next = task;
    for (;;) {
      if (!early) {
        if (!pipelink_call_gemm_ready(&view, &task, &counters)) pipelink_call_gemm_wait(&view, &task, &counters);
        pipelink_call_gemm_prefetch(&view, &task, &carry);
        // The mainloop stages the next task where this one's tokens and counter are, and no wave may do that before every
        // wave has read them.  (A tile whose prefetch was early has its predecessor's epilogue and barriers in between.)
        mok::lds_barrier();
      }
      if (i >= 0) {  // the first tile's loads are on their way: the second turn
        if (i + turn < items) next = sched.decode(q, i + turn, cursor);
        else next.op = 0;  // no task: mok_gemm_fwd looks ahead to nothing
        i = -1;
      }
      const bool has_next = next.op != 0;
      const bool asks = has_next && asking;
      uint32_t answer = 0;
      if (PARTS || pipelink_call_gemm_placement(&view, &task) != mok::TILE_FULL) {
        const SmallTileResult res = small_tile(params, task, next, counters.base, counters.status, asks ? g.workspace + MOK_WS_QUEUE + list : nullptr, carry);
        carry = res.carry;
        early = __builtin_amdgcn_readfirstlane(res.early) != 0;
        answer = res.answer;
        ++phase;
      } else {
        mok::AccFrag acc;
        pipelink_call_gemm_fwd(&view, &task, &counters, &phase, &acc, &carry, &next);
        // ask the queue for the tile after the next (one thread); the answer has the epilogue's time to arrive
        if (asks && threadIdx.x == 0)
          answer = __hip_atomic_fetch_add(g.workspace + MOK_WS_QUEUE + list, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // The next tile's first loads fly while this tile's epilogue computes -- unless its rows are not complete yet:
        // then this tile is finished (and counted) first, so that nobody waits for a workgroup that waits.
        early = has_next && pipelink_call_gemm_ready(&view, &next, &counters);
        if (early) pipelink_call_gemm_prefetch(&view, &next, &carry);
        if (task.op == MOK_GEMM_FWD_ROUTED_GATE_UP) {
          const MokActTask act{MOK_ACT_FWD_ROUTED, task.row_begin, task.row_end, task.col_begin, task.task_idx, task.counter_idx, task.flags};
          pipelink_call_act_fwd(&view, &act, &counters, &phase, &acc);
        } else {
          pipelink_call_gemm_store(&view, &task, &acc);
        }
      }
      // the queue's answer goes round the workgroup through LDS; the barrier is one every wave reaches at about the
      // same time (the epilogue has just ended with one)
      arrived(answer);
      if (threadIdx.x == 0) tab.claim = answer;
      mok::lds_barrier();
      MokGemmTask after = next;
      after.op = 0;
      if (asks) {
        int k = 2 * turn + (int)tab.claim;
        if (k >= sched.length(list)) {
          // This list has been handed out.  One look at all the queues says which lists have tiles left (queues only
          // grow: a list that has none never will), then the first of those is asked, and so on.  The workgroup waits for
          // the answer with its next tile in hand: asking the lists one after the other, an atomic each on words all
          // workgroups ask at that time, took up to 20 us (8 tokens: 164 us a launch, now 146; 128 tokens: 175, 168; 1003
          // tokens: 222, 212; 8192 tokens: 787, 786).
          mok::lds_barrier();  // everybody has read the last answer
          if (threadIdx.x < 64) {
            const int other = (list + 1 + (threadIdx.x & (NUM_XCD - 1))) & (NUM_XCD - 1);
            const uint32_t handed = __hip_atomic_load(g.workspace + MOK_WS_QUEUE + other, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t left = (uint32_t)__builtin_amdgcn_ballot_w64(2 * turn + (int)handed < sched.length(other)) & ((1u << NUM_XCD) - 1);
            uint32_t found = 0;
            while (left != 0 && found == 0) {
              const int from = (list + 1 + __builtin_ctz(left)) & (NUM_XCD - 1);
              left &= left - 1;
              uint32_t got = 0;
              if (threadIdx.x == 0) got = __hip_atomic_fetch_add(g.workspace + MOK_WS_QUEUE + from, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              answer = (uint32_t)__builtin_amdgcn_readfirstlane((int)got);
              if (2 * turn + (int)answer < sched.length(from)) found = 1u + (uint32_t)from;
            }
            if (threadIdx.x == 0) {
              tab.claim = answer;
              tab.last = found;
            }
          }
          mok::lds_barrier();
          k = 2 * turn + (int)tab.claim;
          const int from = __builtin_amdgcn_readfirstlane((int)tab.last);
          asking = from != 0;
          if (asking) list = from - 1;
        }
        if (asking) after = sched.decode(list, k, cursor);
      }
      if (!has_next) break;
      task = next;
      next = after;
    }
  }
}

}  // namespace mok_framework

extern "C" __device__ void mok_framework_worker(const void* params, unsigned variant) {
  (void)variant;
  using namespace mok_framework;
  const pipelink_host_view view{params, nullptr};
  const MokFrameworkParams& g = *static_cast<const MokFrameworkParams*>(params);
  Tables& tab = *reinterpret_cast<Tables*>(pipelink_smem + pipelink_mok_fw_sched());
  const int ne = g.num_experts, op = g.op & MOK_FWD_OP_MASK;

  pipelink_call_gemm_init(&view);
  pipelink_call_act_init(&view);

  // exclusive prefix sums of rows and row tiles per expert (every workgroup computes its own copy)
  if (threadIdx.x < 64)
    tab.fill_by_wave(g.tokens_per_expert, ne, threadIdx.x, [](int v) { return wave_scan(v); },
                     [](int v) { return __builtin_amdgcn_readlane(v, 63); });
  __syncthreads();

  Schedule sched{g, tab, tab.tile_begin[ne], op == MOK_GEMM_FWD_ROUTED_DOWN ? 0 : g.num_col_tiles_gate_up,
                 op == MOK_GEMM_FWD_ROUTED_GATE_UP ? 0 : g.num_col_tiles_down};
  sched.cut();
  sched.part();
  const MokCounters counters{op == MOK_FWD_BOTH ? reinterpret_cast<int32_t*>(g.workspace + MOK_WS_COUNTERS) : nullptr,
                             g.workspace + MOK_WS_STATUS};
  const bool small_only = sched.down_cut != 0 || sched.down_width == PART_COLS;  // (every tile is a small one then)
  if (small_only) run_tiles<true>(params, g, tab, sched, counters);
  else run_tiles<false>(params, g, tab, sched, counters);
  pipelink_call_gemm_fini(&view);

  // The last workgroup to leave puts the queues and the counters back to zero for the next launch: by then nobody
  // asks or waits any more.
  if (threadIdx.x == 0) {
    const uint32_t before = __hip_atomic_fetch_add(g.workspace + MOK_WS_FINISHED, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    tab.last = before == gridDim.x - 1 ? 1u : 0u;
  }
  __syncthreads();
  if (tab.last) {
    if (op == MOK_FWD_BOTH)
      for (int w = threadIdx.x; w < sched.row_tiles; w += mok::THREADS)
        __hip_atomic_store(g.workspace + MOK_WS_COUNTERS + w, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x < NUM_XCD) __hip_atomic_store(g.workspace + MOK_WS_QUEUE + threadIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x == 0) {
      __hip_atomic_store(g.workspace + MOK_WS_FINISHED, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(g.workspace + MOK_WS_GAVE_UP, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}
#else  // PIPELINK_EMIT: host-evaluated annotations only
#include "../include/mok_abi.h"
#endif

PL_STAGE("mok.framework", "0.2.0");
PL_PARAMS(MokFrameworkParams);
PL_ROLE(worker, mok_framework_worker, 4);
PL_TOPOLOGY(true, "static");
PL_VARIANT(0, {});
PL_CALL(gemm_init, "mok_gemm_init", "extern \"C\" __device__ void pipelink_call_gemm_init(const void* view);");
PL_CALL(gemm_fini, "mok_gemm_fini", "extern \"C\" __device__ void pipelink_call_gemm_fini(const void* view);");
PL_CALL(act_init, "mok_act_init", "extern \"C\" __device__ void pipelink_call_act_init(const void* view);");
PL_CALL(gemm_stage, "mok_gemm_stage",
        "extern \"C\" __device__ void pipelink_call_gemm_stage(const void* view, const MokGemmTask* task, const MokCounters* counters);");
PL_CALL(gemm_ready, "mok_gemm_ready",
        "extern \"C\" __device__ bool pipelink_call_gemm_ready(const void* view, const MokGemmTask* task, const MokCounters* counters);");
PL_CALL(gemm_wait, "mok_gemm_wait",
        "extern \"C\" __device__ void pipelink_call_gemm_wait(const void* view, const MokGemmTask* task, const MokCounters* counters);");
PL_CALL(gemm_prefetch, "mok_gemm_prefetch",
        "extern \"C\" __device__ void pipelink_call_gemm_prefetch(const void* view, const MokGemmTask* task, mok::GemmCarry* carry);");
PL_CALL(gemm_fwd, "mok_gemm_fwd",
        "extern \"C\" __device__ void pipelink_call_gemm_fwd(const void* view, const MokGemmTask* task, "
        "const MokCounters* counters, uint32_t* phase, mok::AccFrag* acc, const mok::GemmCarry* carry, "
        "const MokGemmTask* upcoming);");
PL_CALL(gemm_store, "mok_gemm_store",
        "extern \"C\" __device__ void pipelink_call_gemm_store(const void* view, const MokGemmTask* task, const mok::AccFrag* acc);");
PL_CALL(act_fwd, "mok_act_fwd",
        "extern \"C\" __device__ void pipelink_call_act_fwd(const void* view, const MokActTask* task, "
        "const MokCounters* counters, uint32_t* phase, const mok::AccFrag* acc);");
PL_CALL(gemm_placement, "mok_gemm_placement",
        "extern \"C\" __device__ int pipelink_call_gemm_placement(const void* view, const MokGemmTask* task);");
PL_CALL(gemm_fwd_small, "mok_gemm_fwd_small",
        "extern \"C\" __device__ void pipelink_call_gemm_fwd_small(const void* view, const MokGemmTask* task, "
        "const MokCounters* counters, uint32_t* phase, mok::AccFrag* acc, const mok::GemmCarry* carry, "
        "const MokGemmTask* upcoming);");
PL_CALL(gemm_store_small, "mok_gemm_store_small",
        "extern \"C\" __device__ void pipelink_call_gemm_store_small(const void* view, const MokGemmTask* task, const mok::AccFrag* acc);");
PL_CALL(act_fwd_small, "mok_act_fwd_small",
        "extern \"C\" __device__ void pipelink_call_act_fwd_small(const void* view, const MokActTask* task, "
        "const MokCounters* counters, uint32_t* phase, const mok::AccFrag* acc);");
// schedule tables: exclusive prefix sums of rows and row tiles for up to 256 experts, and one word more
PL_CLAIM("pipelink_mok_fw_sched", "smem", 2 * (256 + 1) * 4 + 8, 16, "kernel");
PL_USES("pipelink_mok_fw_sched");
// host contract: the schedule's owner
PL_HOST_GROUP("mok.framework.params", "mok_framework");
PL_HOST_ABI_TYPE(3, MokFrameworkParams);
MOK_HOST_SCALARS();
PL_HOST_CHANNEL(1, "tokens_per_expert", 32, "read", "mok.num_local_experts", false);
// status word and readiness counters of a launch: all zero before the first launch, every launch leaves them zero
PL_HOST_CHANNEL(2, "workspace", 32, "write", "mok.workspace_words", false);
PL_FACT("mok.framework.MAX_EXPERTS", 256);
PL_FACT("mok.framework.LISTS", 8);
PL_PRELUDE("../include/mok_abi.h");
PL_PRELUDE("../include/mok_device.hpp");
PL_EMIT_MAIN()
