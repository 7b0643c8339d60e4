// The chip-resident SOR solve (les_sor_res.hip): plan, buffers and launch.
#pragma once
#include "les_kernels.h"

namespace les {

constexpr int RES_NT = 512;     // threads per workgroup
constexpr int RES_TKMAX = 10;   // most levels per thread
constexpr int RES_TK_KS = 7;    // ... with more than one level block per workgroup (LDS)
constexpr int RES_KWMAX = 128;  // most levels per workgroup
constexpr int RES_JS = 64;      // most groups per row (ip <= 512)

// How the domain is cut: njt x nkt workgroups of rj rows of j and ks * tk levels; ks level
// blocks of tk levels each, one thread per (group of four entries, row, level block).
struct ResPlan {
  int tk = 0;  // 0: the grid does not fit
  int ks = 0, rj = 0, njt = 0, nkt = 0;
  __host__ __device__ int nwg() const { return njt * nkt; }
};

// The queue form: at most one task a workgroup and phase, of RES_NT groups at least (the two fences of
// a task cost more than its sweep does: with tasks of RES_NT groups 300x300x90 took 51 ms).
// The phases are the shifts, then one per sweep (odd jp: two, the seam's copy first).  64 bits:
// any nmaxp is taken.
__host__ __device__ inline unsigned res_queue_blocks(const Dims& d, int nr, int nwg) {
  const unsigned n = ((unsigned)(nr / 4 * d.jp * d.kp) + RES_NT - 1) / RES_NT;
  return n < (unsigned)nwg ? n : (unsigned)nwg;
}
__host__ __device__ inline unsigned long long res_queue_tasks(const Dims& d, int nr, int nwg, int nmaxp) {
  return res_queue_blocks(d, nr, nwg) * (1ull + 2ull * nmaxp * (d.jp % 2 ? 2 : 1));
}

// 2 ms of the 100 MHz clock: other handles' stencils hold CUs for some 0.1 ms at a time (with 0.3 ms a
// few of 1000 solves of eight 150x150x90 handles took the queue form), and that form costs more.
constexpr long RES_WAIT_TICKS = 200000;
// So many solves in a row in the queue form, and the handle leaves this kernel: a few milliseconds
// each at most, while one or two in a row are another kernel's that just ran.
constexpr unsigned RES_GIVE_UP = 16;
constexpr int RES_POLLS = 1 << 22;      // unanswered polls of a sweep's waits: some seconds

struct ResCtl;  // device control block (les_sor_res.hip)

// What a solve tells the host, in pinned host memory
struct ResHost {
  unsigned failed;  // a solve gave up waiting: words of its p are NaN
  unsigned queued;  // solves that took the queue form, their workgroups not all resident in time
  unsigned row;     // ... how many of the last ones in a row
};

// Face slots and control block of one handle (res_alloc / res_free)
struct ResBuf {
  unsigned long long* kslot = nullptr;
  unsigned long long* jslot = nullptr;
  float* seam = nullptr;
  ResCtl* ctl = nullptr;
  ResHost* host = nullptr;
};

ResPlan res_plan(Dims d, int nr, int ncu);
// buffers that serve every plan of pl[0..n) (one at a time: tags of launches only grow)
hipError_t res_alloc(Dims d, int nr, const ResPlan* pl, int n, hipStream_t st, ResBuf& b);
void res_free(ResBuf& b);
size_t res_bytes(Dims d, int nr, const ResPlan* pl, int n);  // device memory of res_alloc
// nmaxp SOR iterations (press.f95:87-115) on the split copy sp.p / sp.r in place.  sub_rhsav: sp.r
// holds the raw rhs; rhsav is taken off every value read and the result written to rout.
// sub_pav: DevScalars::pav_carry is taken off every p value read.  resid_slots (RedBuf::slots, zero):
// with the residual of every iteration (DevScalars::sor, sor_iters) and the early exit; null:
// without.  wait_ticks (100 MHz): how long the workgroups wait for each other to be resident
// before the solve falls back to the queue form; negative: the queue form at once.  polls
// (RES_POLLS): the bound of its later waits.
void launch_sor_resident(hipStream_t st, Dims d, Grid1D g, SplitSOR sp, Physics ph, int nmaxp,
                         DevScalars* sc, int sub_rhsav, int sub_pav, float* rout0, float* rout1,
                         int64_t* resid_slots, const ResPlan& pl, const ResBuf& b, long wait_ticks,
                         int polls);

}  // namespace les
