"""The order in which a workgroup of the MoK framework stages tasks and reads what it staged, on the CPU.

The worker's source is compiled for the host with stand-ins for the GPU's builtins, one lane of one wave, and for the owners'
exports, which print what they do.  Every wave runs the same sequence, each at its own pace: whatever one call writes to the
staged area and another reads must have a workgroup barrier between them."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STAGES = os.path.join(ROOT, "pipelink_amd", "stages", "mok")
CLANG = next((c for c in ("/opt/rocm/lib/llvm/bin/clang++", shutil.which("clang++") or "") if os.path.exists(c)), None)

HIP = r"""
#pragma once
#include <cstdint>
#include <cstdio>
#define __device__
#define __forceinline__ inline
#define __shared__
#define __launch_bounds__(...)
static struct { unsigned x = 0; } threadIdx, blockIdx;
static struct { unsigned x = 256; } blockDim, gridDim;
inline void barrier() { puts("barrier"); }
#define __syncthreads() barrier()
#define __builtin_amdgcn_s_barrier() barrier()
#define __builtin_amdgcn_s_waitcnt(x) ((void)0)
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
#define __builtin_amdgcn_update_dpp(old, v, ...) (old)
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_readlane(v, l) (v)
#define __builtin_amdgcn_ballot_w64(v) ((v) ? 1ull : 0ull)
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, ...) (*(p))
#define __hip_atomic_store(p, v, ...) (*(p) = (v))
template <class T> T added(T* p, T v) { const T old = *p; *p += v; return old; }
#define __hip_atomic_fetch_add(p, v, ...) added(p, v)
"""

PROGRAM = r"""
#define MOK_SCHED_FN inline
#define MOK_SCHED_UNIFORM(x) (x)
#include "framework/framework.hip"
#include <cstdlib>
alignas(1024) unsigned char pipelink_smem[1 << 16];
static int waits, tiles;
extern "C" {
int pipelink_mok_fw_sched() { return 0; }
void pipelink_call_gemm_init(const void*) {}
void pipelink_call_gemm_fini(const void*) {}
void pipelink_call_act_init(const void*) {}
void pipelink_call_gemm_stage(const void*, const MokGemmTask*, const MokCounters*) { puts("write"); }
bool pipelink_call_gemm_ready(const void*, const MokGemmTask* t, const MokCounters*) { puts("read"); return !(waits && t->wait_target > 0); }
void pipelink_call_gemm_wait(const void*, const MokGemmTask*, const MokCounters*) { puts("wait"); }
void pipelink_call_gemm_prefetch(const void*, const MokGemmTask*, mok::GemmCarry*) { puts("read"); }
// a mainloop stages the upcoming task behind its first loads, whatever barriers follow; it ends with one
static void mainloop(const MokGemmTask* next) { ++tiles; if (next->op != 0) puts("write"); barrier(); }
void pipelink_call_gemm_fwd(const void*, const MokGemmTask*, const MokCounters*, uint32_t*, mok::AccFrag*, const mok::GemmCarry*, const MokGemmTask* next) { mainloop(next); }
void pipelink_call_gemm_fwd_small(const void*, const MokGemmTask*, const MokCounters*, uint32_t*, mok::AccFrag*, const mok::GemmCarry*, const MokGemmTask* next) { mainloop(next); }
void pipelink_call_gemm_store(const void*, const MokGemmTask*, const mok::AccFrag*) {}
void pipelink_call_gemm_store_small(const void*, const MokGemmTask*, const mok::AccFrag*) {}
void pipelink_call_act_fwd(const void*, const MokActTask*, const MokCounters*, uint32_t*, const mok::AccFrag*) {}
void pipelink_call_act_fwd_small(const void*, const MokActTask*, const MokCounters*, uint32_t*, const mok::AccFrag*) {}
int pipelink_call_gemm_placement(const void*, const MokGemmTask* t) { puts("placement"); return mok::tile_placement(t->row_end - t->row_begin, 1 << 20, t->flags); }
}
int main(int argc, char** argv) {
  const int rows = atoi(argv[1]), gu = atoi(argv[2]), dn = atoi(argv[3]), workgroups = atoi(argv[4]);
  waits = atoi(argv[5]);
  static uint32_t workspace[1 << 16];
  int32_t tokens = rows;
  MokFrameworkParams g{};
  g.tokens_per_expert = &tokens;
  g.workspace = workspace;
  g.num_experts = 1;
  g.op = MOK_FWD_BOTH | MOK_FWD_MAY_CUT;
  g.num_col_tiles_gate_up = gu;
  g.num_col_tiles_down = dn;
  gridDim.x = workgroups;
  for (blockIdx.x = 0; blockIdx.x < (unsigned)workgroups; ++blockIdx.x) {
    puts("workgroup");
    mok_framework_worker(&g, 0);
  }
  printf("tiles %d\n", tiles);
}
"""


def _worker(d, hip):
    if CLANG is None:
        pytest.skip("needs clang")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(hip)
    (d / "worker.cpp").write_text(PROGRAM)
    subprocess.run([CLANG, "-std=c++17", "-O1", "-w", "-x", "c++", f"-I{d}", f"-I{STAGES}",
                    f"-I{os.path.join(ROOT, 'pipelink_amd', 'pipec', 'include')}", str(d / "worker.cpp"), "-o", str(d / "worker")], check=True)

    def run(*args):
        return subprocess.run([str(d / "worker"), *map(str, args)], check=True, capture_output=True, text=True).stdout.splitlines()
    return run


@pytest.fixture(scope="module")
def trace(tmp_path_factory):
    return _worker(tmp_path_factory.mktemp("worker"), HIP)


# full tiles and small ones, narrow parts of column tiles (8 rows, few tiles); one tile a workgroup and several; down tiles
# whose rows are complete when they are looked at and down tiles that wait
@pytest.mark.parametrize("rows,gu,dn", [(700, 6, 5), (300, 23, 12), (40, 23, 12), (8, 23, 12), (8, 6, 2), (8, 200, 100)])
@pytest.mark.parametrize("workgroups", [8, 24, 256])
@pytest.mark.parametrize("waits", [0, 1])
def test_a_barrier_lies_between_staging_a_task_and_reading_it_and_back(trace, rows, gu, dn, workgroups, waits):
    *events, tiles = trace(rows, gu, dn, workgroups, waits)
    cut = [4 if rows <= 32 and 4 * n <= 256 else 1 for n in (gu, dn)]
    if cut[1] == 1:
        cut[0] = 1
    # launches with parts and launches without have a loop each: only the one without looks whether a tile is a full one
    assert ("placement" in events) == (cut[1] == 1)
    events = [e for e in events if e != "placement"]
    assert tiles == f"tiles {-(-rows // 256) * (gu * cut[0] + dn * cut[1])}"   # every tile has been run
    since = set()   # what has happened to the staged area since the last barrier
    for n, event in enumerate(events):
        if event in ("workgroup", "barrier"):
            since = set()
        elif event != "wait":
            assert not ({"read", "write"} - {event}) & since, (n, events[max(0, n - 8):n + 1])
            since.add(event)


def test_a_wave_waits_for_its_own_staged_loads_before_the_first_tile(tmp_path):
    """What a workgroup's first task stages (no mainloop ends behind it) is waited for in the source itself: the barrier waits for
    no global -> LDS load, whatever the compiler puts in front of it."""
    run = _worker(tmp_path, HIP.replace("s_waitcnt(x) ((void)0)", 's_waitcnt(x) ((x) == 0x0F70 ? (void)puts("landed") : (void)0)'))
    events = run(300, 23, 12, 24, 0)[:-1]
    starts = [n for n, e in enumerate(events) if e == "workgroup"]
    staged = [events.index("write", n) for n in starts]
    assert len(staged) == 24
    assert all(events[n + 1:n + 3] == ["landed", "barrier"] for n in staged)
