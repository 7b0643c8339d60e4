// The whole red-black SOR solve of press.f95:87-115 in one launch, with p and rhs held on the
// chip: 256 CUs have 160 KB of LDS and 512 KB of vector registers each, and 8 bytes a cell fit up
// to about 9 million cells (rows of up to 360 cells; 8 million at 400).  Rows from 440 to 512 cells
// fit up to about 4 million, longer ones not at all: a thread's words of a j face are fixed at rows
// of 160 floats a level (res_jn), and a row has at most 64 groups.
//
// A thread owns a group of four consecutive entries of both colours' rows (j, k) over TK
// consecutive levels (the colour-split layout of les_sor.hip): their p and rhs stay in its
// registers for the whole solve.  Updating one colour, it has the cells above and below and the
// nearest east and west ones in its own registers, and reads the rows j + 1 and j - 1 and the
// one further east or west entry of the other colour from LDS, where every thread also keeps a
// copy of its p.  Every cell gets the same FP32 expression with the same operand values as in
// the colour sweeps of les_sor.hip, so the results are the same bit for bit.
//
// Faces between workgroups go through slots in device memory, one 64-bit word per face cell:
// the value and a tag that says which sweep of which launch wrote it.  A reader polls the word
// itself until the tag is the one it needs; there is no separate flag, no fence and no barrier
// between workgroups.  A sweep first publishes what the sweep before left on its faces: the rows
// at the j faces from LDS, their words dealt over the whole workgroup, the k faces from the
// registers.  It then takes the rows across the j faces into LDS (one barrier) and computes; the
// levels at the k faces come last, and the words across them are loaded half a sweep before.
// (Measured and not kept at 300x300x90, where a sweep takes 5.0 us: each row's own threads
// loading their j faces, 6.7 to 8.7 us, their loads queue behind their stores; each row's threads
// publishing level by level, 6.9 us; a flag per face instead of tags, no faster at 8 KB a face.)
// A slot is never overwritten before it is read: a workgroup publishes colour c again two sweeps
// later, and it cannot get there before it has read the words that its neighbour publishes in
// the sweep in between, after the neighbour's last read of the slot.
// Words are relaxed 64-bit atomics, read at agent scope.  A store whose reader is on another XCD
// has agent scope.  A workgroup's neighbours are mostly on its own XCD, whose CUs share one L2:
// for those the store goes only that far (workgroup scope; vector stores write through the CU's
// own cache), which halves the time of an exchange with 16 KB per face (3.1 -> 1.6 us a step for
// 240 workgroups); the agent-scope load bypasses the reader's own cache and finds it in that L2.
// Which XCD a workgroup is on is read from the hardware and shared before the first sweep.
//
// With an odd jp the two rows at the periodic seam have the same colour.  Their images are the
// values before the running sweep (boundp1 follows the colour, press.f95:103-105), so a seam
// row takes the tag of the colour's previous sweep; the j slots are double-buffered then.
//
// All workgroups have to be on the chip together.  They count themselves in first; when they
// are not all there within wait_ticks (another program's kernels hold the CUs), the state word
// goes to RES_QUEUE instead of RES_GO, once for all of them, and the same launch solves through
// a task queue: tasks are taken in order from a counter, a task waits only for tasks before it,
// and those are held by workgroups that are running, so it ends with any number of them
// resident.  No input is overwritten before the decision.  The queue form is slow (50 iterations at
// 300x300x90 11.8 ms, 150x150x90 7.5, 32x24x16 1.4: two agent-scope fences a task and all workgroups
// at two counters); the host is told how many solves took it and leaves this kernel after some.
//
// Bound: instruction issue and the exchange.  Per sweep at 300x300x90 (240 workgroups of 13 rows x
// 9 levels): 2.0 us computing (77 vector instructions a group of four cells, two wavefronts per
// SIMD), 0.9 us more with k faces only, 5.0 us with both; memory is read once and written once
// per solve.  50 iterations, measured with the scatter and gather of p around them: 300x300x90
// 563 us against 50 x 20.5 us for k_sor_iter; 150x150x90 267 against 50 x 11.7; 32x24x16 (one
// workgroup, no exchange: barriers and LDS latency) 133 against 50 x 8.3; the kernel alone at
// 147x133x61 (odd jp) 227 against 100 x (9.2 + 4.9) + 50 x 4.6 in place.
// With the residual (50 iterations): 1080, 700 and 300 us against 2140, 1440 and 1240 for the
// residual-summing sweeps; what it adds is one all-workgroup hop an iteration (about 3 us, on the
// smallest grid) and the sums' instructions.
#include <algorithm>

#include "les_sor_res.h"

namespace les {

constexpr int RES_WGMAX = 1024;  // (no device has that many CUs)
struct ResCtl {
  unsigned arrive, state, done, queued;  // queued: launches that took the queue form
  // low word: the launch's first tag; high: RES_FAILED, a wait was given up in this launch, and the
  // number of launches in a row that took the queue form
  unsigned long long base;
  ResHost* host;    // what the host is told
  unsigned long long ticket, tasks;  // the queue form's (phases x tasks can pass 32 bits)
  // the residual: workgroups that have added their exact sums, last iteration decided from them
  // (times 2, plus 1: stop); each workgroup's sum of an iteration as two tagged words
  unsigned added, decided;
  unsigned long long sums[2][2][RES_WGMAX];
  unsigned xcd[RES_WGMAX];  // the XCD each workgroup of the launch is on
};

namespace {

// LDS entries per level: 10 levels fit only with fewer than RES_NT threads in use
constexpr int res_ns(int tk) { return tk >= RES_TKMAX ? 448 : RES_NT; }

// words of a j face (levels of the workgroup x floats of a row) per thread: enough for rows of
// 160 floats where a workgroup has one level block
constexpr int res_jn(int tk) { return (tk * 160 + RES_NT - 1) / RES_NT; }

typedef unsigned long long u64;
enum { RES_GO = 1, RES_QUEUE = 2 };
constexpr u64 RES_FAILED = 1ull << 63;

struct ResArgs {
  Dims d;
  Grid1D g;
  SplitSOR sp;
  float omega;
  int nmaxp;
  DevScalars* sc;
  int sub_rhsav, sub_pav;
  float* rout[2];
  float pjuge;
  int64_t* slots;  // exact-sum slots of the residual (RedBuf::slots), zero between uses
  ResPlan pl;
  u64 *kslot, *jslot;
  float* seam;
  ResCtl* ctl;
  long wait_ticks;
  int polls;  // most unanswered polls of a sweep's waits
};

template <class T>
__device__ __forceinline__ T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// four face cells: entries 4g .. 4g+3, one word each, 'stride' words apart (lanes next to each
// other read and write words next to each other)
struct Face4 {
  u64 v[4];
};
template <int STRIDE>
__device__ __forceinline__ Face4 face_load(const u64* p) {
  Face4 f;
#pragma unroll
  for (int q = 0; q < 4; ++q) f.v[q] = agent_load(p + q * STRIDE);
  return f;
}
// near: the reader is on this XCD (the branch is uniform)
__device__ __forceinline__ void word_store(u64* p, float v, unsigned tag, bool near) {
  const u64 w = ((u64)tag << 32) | (u64)__float_as_uint(v);
  if (near)
    __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  else
    agent_store(p, w);
}
__device__ __forceinline__ void face_store(u64* p, int stride, float4 x, unsigned tag, bool near) {
  const float v[4] = {x.x, x.y, x.z, x.w};
  if (near) {
#pragma unroll
    for (int q = 0; q < 4; ++q) word_store(p + q * stride, v[q], tag, true);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) word_store(p + q * stride, v[q], tag, false);
  }
}
// A poll left unanswered, and the word read again.  Waits end because every workgroup is resident and a
// sweep waits only for the one before it; 'budget', the polls that a sweep's waits may leave
// unanswered, bounds them all the same (seconds).  A thread that uses it up takes NaN for the
// missing word, which spreads with the sweeps, waits no more, and says so at the end of the solve:
// the host gets an error (ResHost::failed).
__device__ __forceinline__ u64 poll_again(const u64* p, unsigned tag, int& budget) {
  if (--budget > 0) return agent_load(p);
  budget = 0;
  return ((u64)tag << 32) | 0x7fc00000u;
}
// The face's values once all four carry 'tag'.
template <int STRIDE>
__device__ __forceinline__ float4 face_wait(Face4 f, const u64* p, unsigned tag, int& budget) {
  for (;;) {
    bool ok = true;
#pragma unroll
    for (int q = 0; q < 4; ++q) ok = ok && (unsigned)(f.v[q] >> 32) == tag;
    if (ok) break;
    __builtin_amdgcn_s_sleep(1);
    if (--budget > 0) {
      f = face_load<STRIDE>(p);
    } else {
      budget = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) f.v[q] = ((u64)tag << 32) | 0x7fc00000u;
    }
  }
  return make_float4(__uint_as_float((unsigned)f.v[0]), __uint_as_float((unsigned)f.v[1]),
                     __uint_as_float((unsigned)f.v[2]), __uint_as_float((unsigned)f.v[3]));
}

__device__ __forceinline__ float4 sub4(float4 a, float s) {
  return make_float4(a.x - s, a.y - s, a.z - s, a.w - s);
}
__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ void st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
// a copy the compiler cannot see through: keeps addresses derived from it out of registers
// between their uses (they are a few instructions to form again)
__device__ __forceinline__ unsigned opaque(unsigned x) {
  __asm__ volatile("" : "+v"(x));
  return x;
}
__device__ __forceinline__ int opaque_s(int x) {  // the same for a value in a scalar register
  x = __builtin_amdgcn_readfirstlane(x);
  __asm__ volatile("" : "+s"(x));
  return x;
}
// the word at a uniform byte offset plus a thread's (scalar base, 32-bit vector offset)
__device__ __forceinline__ u64* word_at(u64* base, unsigned uni, unsigned mine) {
  return reinterpret_cast<u64*>(reinterpret_cast<char*>(base) + uni + mine);
}
__device__ __forceinline__ unsigned my_xcd() {
  unsigned x;
  __asm__ volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(x));
  return x;
}
// first interior i of colour c in row (j,k)
__device__ __forceinline__ int first_of(int c, int j, int k) { return ((1 + j + k) & 1) == c ? 1 : 2; }

// wait for LDS only: face stores and prefetched face loads stay in flight
__device__ __forceinline__ void lds_only_barrier() {
  __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Exact sum of the residual's terms x = reltmp**2 of one thread and iteration.  Two FP64
// accumulators start at 1.5 * 2^52 units and stay in that binade, so one unit is their last place:
// 2^E0 and 2^E1, E0 = E1 + 45.  The first takes x rounded to its unit, the second what that left,
// which is exact for x a multiple of 2^E1 below 2^(E1 + 89): |left| <= 2^(E1 + 44), and 8 * RES_TKMAX
// terms move either accumulator by less than 2^51 units.  Every x from 2^(E1 + 23) on is such a
// multiple; the others (few, E1 follows the sum of the iteration before) go to the workgroup's
// limbs in LDS one by one, with their group's others.  Four FP64 additions a cell; with integer sums of the terms' 64-bit
// parts an iteration at 300x300x90 took 32.1 us, now 20.0 (10.0 without the residual).
struct SquareAcc {
  double a0, a1;
  int e1;           // uniform
  unsigned lo, hi;  // bit patterns taken: lo <= bits < hi, and zero
  static __device__ __forceinline__ double bias(int e) {  // 1.5 * 2^(52 + e)
    return __longlong_as_double(((long long)(1023 + 52 + e) << 52) | 0x8000000000000ll);
  }
  // E1 for terms up to about 8 times 'sum'
  __device__ __forceinline__ void start(double sum) {
    const int e = (int)((__double_as_longlong(sum) >> 52) & 0x7ff) - 1023;
    e1 = __builtin_amdgcn_readfirstlane(min(max(e + 4 - 89, -149), 39));
    const int l = e1 + 23;
    lo = e1 == -149 ? 1u : l >= -126 ? (unsigned)(l + 127) << 23 : 1u << (l + 149);
    hi = min((unsigned)(e1 + 89 + 127) << 23, 0x7f800000u);
    a0 = bias(e1 + 45);
    a1 = bias(e1);
  }
  // four terms; one outside the range sends all four to the limbs
  __device__ __forceinline__ void add4(const float (&x)[4], u64* limbs) {
    unsigned most = 0u, least = ~0u;  // (zeros pass: least holds bits - 1)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      most = max(most, __float_as_uint(x[q]));
      least = min(least, __float_as_uint(x[q]) - 1u);
    }
    if (most < hi && least >= lo - 1u) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double v = (double)x[q], s = a0 + v;
        a1 += v - (s - a0);
        a0 = s;
      }
    } else {
      TermParts t;
#pragma unroll 1
      for (int q = 0; q < 4; ++q)
        if (split_term(q == 0 ? x[0] : q == 1 ? x[1] : q == 2 ? x[2] : x[3], t)) {
          atomicAdd(&limbs[t.limb], (u64)t.lo);
          atomicAdd(&limbs[t.limb + 1], (u64)t.hi);
        }
    }
  }
  // into the workgroup's units[2]; every lane of the wavefront together
  __device__ __forceinline__ void flush(u64* units) const {
    long long n0 = __double_as_longlong(a0) - __double_as_longlong(bias(e1 + 45));
    long long n1 = __double_as_longlong(a1) - __double_as_longlong(bias(e1));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      n0 += __shfl_xor(n0, o);
      n1 += __shfl_xor(n1, o);
    }
    if (__lane_id() == 0) {
      atomicAdd(&units[0], (u64)n0);
      atomicAdd(&units[1], (u64)n1);
    }
  }
  // one thread: the workgroup's sum, rounded
  __device__ __forceinline__ double value(const u64* units, const u64* limbs) const {
    double v = ldexp((double)(long long)units[0], e1 + 45) + ldexp((double)(long long)units[1], e1);
#pragma unroll
    for (int q = 0; q < NLIMB; ++q) v += ldexp((double)(long long)limbs[q], 32 * q - 149);
    return v;
  }
  // one thread: the workgroup's units into its limbs
  __device__ __forceinline__ void fold(u64* units, u64* limbs) const {
    for (int w = 0; w < 2; ++w) {
      const long long n = (long long)units[w];
      const int off = e1 + (w ? 0 : 45) + 149;
      const long long part[2] = {n & 0xffffffffll, n >> 32};
      for (int q = 0; q < 2; ++q) {
        const int at = (off >> 5) + q;
        const long long y = (long long)((u64)part[q] << (off & 31));
        limbs[at] += (u64)(y & 0xffffffffll);
        if (at + 1 < NLIMB) limbs[at + 1] += (u64)(y >> 32);  // (past the last limb: no bits)
      }
    }
  }
};

// this wavefront's own stores and atomics have reached memory.  What the workgroups exchange about
// the residual is read and written by agent-scope atomics alone, so their order is all that is
// needed; a fence would write the L2 back (the faces kept within an XCD) at every iteration.
__device__ __forceinline__ void mem_done() { __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// One thread: the residual from the limbs (press.f95:97), the iteration's count and the early
// exit (press.f95:114); tells the other workgroups.  Agent scope: another iteration's decision may
// be taken on another XCD.
__device__ inline unsigned res_decide(const ResArgs& a, const int64_t* limbs, unsigned it) {
  const float s = limbs_to_float(limbs);
  const bool stop = s < a.pjuge;
  agent_store(&a.sc->sor, s);
  agent_store(&a.sc->sor_iters, (int)it);
  if (stop) agent_store(&a.sc->sor_done, 1);
  const unsigned dec = 2u * it + (stop ? 1u : 0u);
  mem_done();
  agent_store(&a.ctl->decided, dec);
  mem_done();
  return dec;
}

// The whole workgroup: adds its limbs (in LDS, cleared again) to the slots, and returns whether it
// was the last of 'n' to do so; that one then has all limbs in 'limbs' and the slots are zero.
__device__ inline bool res_add_limbs(const ResArgs& a, u64* lds, unsigned* counter, unsigned n,
                                     int64_t* limbs, unsigned* flag) {
  const int t = threadIdx.x;
  __syncthreads();
  u64* slots = reinterpret_cast<u64*>(a.slots);
  if (t < NLIMB) {
    if (lds[t]) atomicAdd(slots + (blockIdx.x % RED_SLOTS) * NLIMB + t, lds[t]);
    lds[t] = 0;
    mem_done();  // added before counted
  }
  __syncthreads();
  if (t == 0)
    *flag = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == n;
  __syncthreads();
  const bool last = *flag != 0u;
  if (last) {
    for (int q = t; q < RED_SLOTS * NLIMB; q += RES_NT) {
      const u64 v = agent_load(slots + q);
      if (v) {
        atomicAdd(&lds[q % NLIMB], v);
        agent_store(slots + q, (u64)0);
      }
    }
    mem_done();  // cleared before anyone is told
    __syncthreads();
    if (t < NLIMB) {
      limbs[t] = (int64_t)lds[t];
      lds[t] = 0;
    }
  }
  __syncthreads();
  return last;
}

// The last workgroup to leave re-arms the control block for the next launch (stream order makes
// it visible there).
__device__ __forceinline__ void res_leave(const ResArgs& a, bool queued) {
  __syncthreads();
  if (threadIdx.x != 0) return;
  const unsigned n = (unsigned)a.pl.nwg();
  if (atomicAdd(&a.ctl->done, 1u) != n - 1u) return;
  const u64 base = agent_load(&a.ctl->base);
  unsigned row = (unsigned)(base >> 32) & 0x7fffffffu;
  if (base & RES_FAILED) {
    for (int q = 0; a.slots && q < RED_SLOTS * NLIMB; ++q) agent_store(a.slots + q, (int64_t)0);
    agent_store(&a.sc->sor, __builtin_nanf(""));
    __hip_atomic_store(&a.ctl->host->failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (queued || row) {  // (the host's memory is written only where something changes)
    const unsigned total = agent_load(&a.ctl->queued) + (queued ? 1u : 0u);
    row = queued ? (row + 1u) & 0x7fffffffu : 0u;
    agent_store(&a.ctl->queued, total);
    __hip_atomic_store(&a.ctl->host->queued, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&a.ctl->host->row, row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  agent_store(&a.ctl->base, (u64)row << 32 | ((unsigned)base + 2u * (unsigned)a.nmaxp + 2u));
  agent_store(&a.ctl->arrive, 0u);
  agent_store(&a.ctl->ticket, (u64)0);
  agent_store(&a.ctl->tasks, (u64)0);
  agent_store(&a.ctl->added, 0u);
  agent_store(&a.ctl->decided, 0u);
  agent_store(&a.ctl->done, 0u);
  agent_store(&a.ctl->state, 0u);
}

// The same solve through the task queue, on the split copy in device memory.  Phases in order:
// the rhsav / pav shifts, then per sweep (odd jp: a copy of the two seam rows of the colour,
// the values before the sweep, and) the sweep; nb tasks per phase.  A task of
// phase f starts when f * nb tasks have ended.  With the residual, the workgroup that adds the last
// of an iteration's limbs decides before its task ends; after a stop the tasks left are void.
template <bool RESID>
__device__ void res_queue(const ResArgs& a) {
  __shared__ u64 sTask;
  __shared__ unsigned sFlag;
  __shared__ u64 sLimb[NLIMB];
  __shared__ int64_t sSum[NLIMB];
  if (RESID && threadIdx.x < NLIMB) sLimb[threadIdx.x] = 0;
  const Dims& d = a.d;
  const SplitSOR& sp = a.sp;
  const int ng = sp.nr / 4, pl = sp.nr * sp.nj;
  const bool odd = d.jp & 1;
  const unsigned ngroups = (unsigned)(ng * d.jp * d.kp);
  const unsigned nb = res_queue_blocks(d, sp.nr, a.pl.nwg());
  const unsigned chunk = (ngroups + nb - 1) / nb;  // groups of a task
  const unsigned per = odd ? 2u : 1u;
  const u64 ntask = res_queue_tasks(d, sp.nr, a.pl.nwg(), a.nmaxp);
  const float rsh = a.sub_rhsav ? a.sc->rhsav : 0.0f, psh = a.sub_pav ? a.sc->pav_carry : 0.0f;
  const float c2l = a.g.cn2l[0], c2s = a.g.cn2s[0], c3l = a.g.cn3l[0], c3s = a.g.cn3s[0];
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) {
      const u64 n = atomicAdd(&a.ctl->ticket, (u64)1);
      sTask = n;
      if (n < ntask) {
        const u64 need = n / nb * nb;
        while (agent_load(&a.ctl->tasks) < need) {
          if (RESID && (agent_load(&a.ctl->decided) & 1u)) break;
          __builtin_amdgcn_s_sleep(4);
        }
        // An iteration is decided before its last task ends, so with that count seen first every
        // later task sees a stop: 'decided' must not be loaded before 'tasks'.
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (RESID && (agent_load(&a.ctl->decided) & 1u)) sTask = ~(u64)0;
      }
    }
    __syncthreads();
    const u64 n = sTask;
    if (n >= ntask) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    const u64 ph = n / nb;
    const unsigned b = (unsigned)(n - ph * nb);
    ThreadAcc acc;
    acc.init();
    const unsigned end = min((b + 1u) * chunk, ngroups);
    for (unsigned grp_id = b * chunk + threadIdx.x; grp_id < end; grp_id += RES_NT) {
      const int row = (int)(grp_id / (unsigned)ng), g4 = (int)(grp_id - (unsigned)(row * ng));
      const int kk = row / d.jp, j = 1 + row - kk * d.jp, k = 1 + kk;
      const int base = sp.nr * ((j - 1) + sp.nj * (k - 1)) + 4 * g4;
      if (ph == 0) {
        for (int c = 0; c < 2; ++c) {
          if (a.sub_pav) st4(sp.p[c] + base, sub4(ld4(sp.p[c] + base), psh));
          if (a.sub_rhsav) st4(a.rout[c] + base, sub4(ld4(sp.r[c] + base), rsh));
        }
      } else {
        const int c = ((ph - 1u) / per & 1u) ? 0 : 1;
        float* own = sp.p[c];
        if (odd && (ph - 1u) % per == 0u) {  // seam rows before the sweep: j = 1, then j = jp
          if (j == 1) st4(a.seam + sp.nr * (2 * kk) + 4 * g4, ld4(own + base));
          if (j == d.jp) st4(a.seam + sp.nr * (2 * kk + 1) + 4 * g4, ld4(own + base));
        } else {
          const float* po = sp.p[c ^ 1];
          const float* rr = (a.sub_rhsav ? a.rout[c] : sp.r[c]) + base;
          const int f = first_of(c, j, k);
          const float* north = j < d.jp ? po + base + sp.nr
                                        : (odd ? a.seam + sp.nr * (2 * kk) + 4 * g4
                                               : po + base - sp.nr * (d.jp - 1));
          const float* south = j > 1 ? po + base - sp.nr
                                     : (odd ? a.seam + sp.nr * (2 * kk + 1) + 4 * g4
                                            : po + base + sp.nr * (d.jp - 1));
          const float cn1 = sp.cn1k[k], c4l = a.g.cn4l[k - 1], c4s = a.g.cn4s[k - 1];
          for (int q = 0; q < 4; ++q) {
            const int e = 4 * g4 + q, i = f + 2 * e;
            if (i > d.ip) break;
            const float pc = own[base + q];
            const float pe = i == d.ip ? pc : po[base + q + (f == 1 ? 0 : 1)];
            const float pw = i == 1 ? pc : po[base + q - (f == 1 ? 1 : 0)];
            const float pu = k < d.kp ? po[base + q + pl] : pc;
            const float pd = k > 1 ? po[base + q - pl] : pc;
            const float reltmp = a.omega * (cn1 * (c2l * pe + c2s * pw + c3l * north[q] +
                                                   c3s * south[q] + c4l * pu + c4s * pd - rr[q]) -
                                            pc);
            own[base + q] = pc + reltmp;
            if constexpr (RESID) acc.add(reltmp * reltmp, sLimb);
          }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    if constexpr (RESID) {
      acc.flush(sLimb);
      const unsigned it = ph > 0u ? (unsigned)((ph - 1u) / (2u * per)) + 1u : 0u;  // the iteration, from 1
      if (ph > 0u && res_add_limbs(a, sLimb, &a.ctl->added, it * 2u * per * nb, sSum, &sFlag) &&
          threadIdx.x == 0)
        res_decide(a, sSum, it);
    }
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(&a.ctl->tasks, (u64)1);
  }
}

// TK levels per thread; NS: LDS entries per level (threads used, at most RES_NT); KS1: one
// level block per workgroup; RESID: with the residual and the early exit.
template <int TK, int NS, bool KS1, bool RESID>
__global__ __launch_bounds__(RES_NT) void k_sor_resident(ResArgs a) {
  __shared__ float4 sP[2][TK][NS];
  __shared__ float4 sC[KS1 ? TK : RES_KWMAX];  // cn1, cn4l, cn4s of the workgroup's levels
  __shared__ __attribute__((aligned(16))) float sJ[2][res_jn(TK) * RES_NT];  // the rows across the south / north face, one colour
  __shared__ unsigned sCtl[3];
  // the residual's exact sum (by the iteration's parity) and the sum of all workgroups' by wavefront
  __shared__ u64 sLimb[2][RESID ? NLIMB : 1], sUnit[2][2];
  __shared__ double sWave[RES_NT / 64];
  __shared__ int64_t sSum[RESID ? NLIMB : 1];
  const Dims d = a.d;
  const SplitSOR sp = a.sp;
  const int t = threadIdx.x;
  const int njt = a.pl.njt, nkt = a.pl.nkt, ks = KS1 ? 1 : a.pl.ks, rj = a.pl.rj;
  const int nwg = njt * nkt;
  // Workgroups go to the 8 XCDs round-robin; each XCD takes a contiguous share of the cuts, kt
  // fastest, so that most faces are between CUs that share an L2.
  const int turn = (int)blockIdx.x & 7, rem = nwg & 7;
  const int wg = turn * (nwg >> 3) + min(turn, rem) + ((int)blockIdx.x >> 3);
  const int jt = wg / nkt, kt = wg - jt * nkt;

  if (t == 0) {
    unsigned st = RES_GO, st0 = 0u;
    if (a.wait_ticks < 0) {
      st = RES_QUEUE;
    } else if (nwg > 1) {
      agent_store(&a.ctl->xcd[wg], my_xcd());
      // release: the XCD before the count
      if (__hip_atomic_fetch_add(&a.ctl->arrive, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u ==
          (unsigned)nwg)
        __hip_atomic_compare_exchange_strong(&a.ctl->state, &st0, (unsigned)RES_GO, __ATOMIC_ACQ_REL,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const long t0 = (long)wall_clock64();
      while ((st = agent_load(&a.ctl->state)) == 0u) {
        if ((long)wall_clock64() - t0 > a.wait_ticks)
          atomicCAS(&a.ctl->state, 0u, (unsigned)RES_QUEUE);
        else
          __builtin_amdgcn_s_sleep(2);
      }
    }
    sCtl[0] = st;
    sCtl[1] = (unsigned)agent_load(&a.ctl->base);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  if (sCtl[0] != RES_GO) {
    res_queue<RESID>(a);
    res_leave(a, true);
    return;
  }
  const unsigned base_tag = sCtl[1];
  if constexpr (RESID) {
    if (t < 2 * NLIMB) sLimb[t / NLIMB][t % NLIMB] = 0;
    if (t < 4) sUnit[t >> 1][t & 1] = 0;
  }
  SquareAcc acc;

  const int ng = sp.nr >> 2;
  const int blk = rj * ng;  // threads per level block
  const int kb = KS1 ? 0 : t / blk;
  const int tt = t - kb * blk;
  const int row = tt / ng, grp = tt - row * ng;
  const int jA = (int)((long)jt * d.jp / njt), jB = (int)((long)(jt + 1) * d.jp / njt);
  const int nrow = jB - jA;
  const int j = 1 + jA + row;
  const int kw = ks * TK;           // levels per workgroup
  const int kw0 = 1 + kt * kw;      // its first level
  const int k0 = kw0 + kb * TK;     // the thread's first level
  const int nlev = min(TK, d.kp - k0 + 1);
  const bool active = t < ks * blk && row < nrow && nlev > 0;
  const int ltop = (k0 + nlev - 1 == d.kp) ? nlev - 1 : -1;  // the level k = kp, if it has it
  const bool bottom = k0 == 1;
  if (t < kw && kw0 + t <= d.kp) {
    const int k = kw0 + t;
    sC[t] = make_float4(sp.cn1k[k], a.g.cn4l[k - 1], a.g.cn4s[k - 1], 0.0f);
  }
  const float c2l = a.g.cn2l[0], c2s = a.g.cn2s[0], c3l = a.g.cn3l[0], c3s = a.g.cn3s[0];
  const float om = a.omega;

  // the row's first cell of colour C at level l is i = 1 iff s1 == ((C + l) & 1)
  const bool s1 = (1 + j + k0) & 1;
  const bool g0 = grp == 0;
  // the cell i = ip: entry ee of the colour whose rows start at 1 (ip odd) or 2 (ip even)
  const int ee = (d.ip - 1) >> 1;
  const bool ge = grp == (ee >> 2);
  const bool odd_ip = d.ip & 1;
  // image selects for rows of the two phases ([b], b = (C + l) & 1)
  const bool w0[2] = {g0 && !s1, g0 && s1};
  bool eq[2][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const bool e = ge && (ee & 3) == q;
    eq[0][q] = e && (!s1 == odd_ip);
    eq[1][q] = e && (s1 == odd_ip);
  }
  // LDS indices of the rows j+1, j-1 (a lone tile of an even jp wraps around) and of the entry
  // west (rows starting at 1) or east (at 2) of the group, inside the level
  const bool odd_jp = d.jp & 1;
  const bool faceJ = njt > 1 || odd_jp;
  const bool isN = faceJ && active && row == nrow - 1, isS = faceJ && active && row == 0;
  const bool isJ = isN || isS;
  const int tN = row < nrow - 1 ? t + ng : (faceJ ? t : t - ng * (nrow - 1));
  const int tS = row > 0 ? t - ng : (faceJ ? t : t + ng * (nrow - 1));
  const int xw = g0 ? 4 * t : 4 * t - 1, xe = grp == ng - 1 ? 4 * t : 4 * t + 4;
  const int x1 = s1 ? xw : xe, x0 = s1 ? xe : xw;
  // Face slots, in 32-bit byte offsets: k faces [wg][0 below, 1 above][colour][q][RES_NT] words;
  // j faces [wg][buffer][colour][0 south, 1 north][FW] words, the workgroup's levels of a row
  // one after the other.
  constexpr int JN = res_jn(TK);        // words of a j face per thread
  constexpr unsigned FW8 = JN * RES_NT * 8u, KF = 4u * RES_NT * 8u;  // bytes of a face of one colour
  const bool pubD = active && kb == 0 && kt > 0, pubU = active && kb == ks - 1 && kt < nkt - 1;
  const unsigned kslot0 = (unsigned)wg * 4u * KF;
  const int njw = min(kw, d.kp - kw0 + 1) * 4 * ng;  // words of a j face in use
  const int wgS = kt + nkt * (jt == 0 ? njt - 1 : jt - 1);
  const int wgN = kt + nkt * (jt == njt - 1 ? 0 : jt + 1);
  const unsigned nbuf = odd_jp ? 2u : 1u;
  auto jslot = [&](int w, unsigned buf, int c) { return (((unsigned)w * nbuf + buf) * 2u + c) * 2u * FW8; };
  auto bufof = [&](unsigned h2) { return odd_jp ? (h2 >> 1) & 1u : 0u; };  // h2 = h + 2
  // neighbours on this XCD
  auto near = [&](int w) {
    return nwg > 1 && __builtin_amdgcn_readfirstlane(agent_load(&a.ctl->xcd[w])) == my_xcd();
  };
  const bool nearS = near(wgS), nearN = near(wgN);
  const bool nearD = kt > 0 && near(wg - 1), nearU = kt < nkt - 1 && near(wg + 1);
  // This thread's words of a j face are t + i RES_NT; their places in the LDS copy of p (south
  // face: row 0 of the workgroup; north face: its last row, jlast floats further on)
  unsigned jsrc[JN];
#pragma unroll
  for (int i = 0; i < JN; ++i) {
    const int u = min(t + i * RES_NT, njw - 1);
    const int kl = u / (4 * ng), b = KS1 ? 0 : kl / TK, l = kl - b * TK;
    jsrc[i] = (unsigned)((l * NS + b * blk) * 4 + (u - kl * 4 * ng));
  }
  const int jlast = (nrow - 1) * ng * 4;
  const float* const lds_p[2] = {reinterpret_cast<const float*>(&sP[0][0][0]),
                                 reinterpret_cast<const float*>(&sP[1][0][0])};
  // colour c of the rows at the j faces, from LDS (words past njw are not read)
  auto j_publish = [&](auto Cc, unsigned tag, unsigned buf) {
    constexpr int c = decltype(Cc)::value;
    const unsigned o = jslot(wg, buf, c), t8 = opaque(8u * t);
    float v[2][JN];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int i = 0; i < JN; ++i) v[f][i] = lds_p[c][jsrc[i] + (f ? jlast : 0)];
#pragma unroll
    for (int f = 0; f < 2; ++f)
      if (f ? nearN : nearS) {
#pragma unroll
        for (int i = 0; i < JN; ++i)
          word_store(word_at(a.jslot, o + f * FW8 + i * RES_NT * 8u, t8), v[f][i], tag, true);
      } else {
#pragma unroll
        for (int i = 0; i < JN; ++i)
          word_store(word_at(a.jslot, o + f * FW8 + i * RES_NT * 8u, t8), v[f][i], tag, false);
      }
  };

  float4 p[2][TK], r[2][TK];
  const int lstride = sp.nr * sp.nj;
  const int off0 = sp.nr * (j - 1) + 4 * grp + lstride * (k0 - 1);
  if (active) {
    const float psh = a.sub_pav ? a.sc->pav_carry : 0.0f;
    const float rsh = a.sub_rhsav ? a.sc->rhsav : 0.0f;
#pragma unroll
    for (int l = 0; l < TK; ++l) {
      if (l >= nlev) continue;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        p[c][l] = ld4(sp.p[c] + off0 + l * lstride);
        r[c][l] = ld4(sp.r[c] + off0 + l * lstride);
      }
    }
#pragma unroll
    for (int l = 0; l < TK; ++l) {
      if (l >= nlev) continue;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if (a.sub_pav) p[c][l] = sub4(p[c][l], psh);
        if (a.sub_rhsav) {
          r[c][l] = sub4(r[c][l], rsh);
          st4(a.rout[c] + off0 + l * lstride, r[c][l]);
        }
        // the padding past i = ip: zero, so that it stays finite
        const int i0 = first_of(c, j, k0 + l) + 8 * grp;
        float4& x = p[c][l];
        if (i0 > d.ip) x.x = 0.0f;
        if (i0 + 2 > d.ip) x.y = 0.0f;
        if (i0 + 4 > d.ip) x.z = 0.0f;
        if (i0 + 6 > d.ip) x.w = 0.0f;
        sP[c][l][t] = x;
      }
    }
    // the image across k = kp is the cell itself: kept as the other colour's next level
#pragma unroll
    for (int l = 0; l + 1 < TK; ++l)
      if (l == ltop) {
        p[0][l + 1] = p[1][l];
        p[1][l + 1] = p[0][l];
      }
  }
  __syncthreads();

  // the seam's colour 1 as of "sweep -2" (colour 0, "sweep -1", goes out with the first sweep)
  if (odd_jp) j_publish(std::integral_constant<int, 1>{}, base_tag, bufof(0u));

  int budget = a.polls;
  struct Lds {  // a level's operands from LDS
    float4 n, s;
    float x;
  };
  // Levels in the order 1 .. TK-2 (both k neighbours in registers), 0, TK-1: the k faces are
  // needed last, a sweep's time after they were published.
  constexpr auto lv = [](int s) { return TK == 1 ? 0 : (s < TK - 2 ? s + 1 : (s == TK - 2 ? 0 : TK - 1)); };
  constexpr int KL = TK > 2 ? TK / 2 : 0;  // step at which the k faces are loaded
  auto half = [&](auto Cc, unsigned h) {
    constexpr int C = decltype(Cc)::value, O = 1 - C;
    const unsigned tagK = base_tag + 1u + h;  // tag of sweep h - 1
    if (budget > 0) budget = a.polls;
    if (faceJ) {  // publish the rows at the j faces, take those across them into LDS
      j_publish(std::integral_constant<int, O>{}, tagK, bufof(h + 1u));
      const bool seamS = odd_jp && jt == 0, seamN = odd_jp && jt == njt - 1;
      const unsigned inS = jslot(wgS, bufof(seamS ? h : h + 1u), seamS ? C : O) + FW8;
      const unsigned inN = jslot(wgN, bufof(seamN ? h : h + 1u), seamN ? C : O);
      const unsigned tagS = seamS ? tagK - 1u : tagK, tagN = seamN ? tagK - 1u : tagK;
      const unsigned t8 = opaque(8u * t);
      u64 jw[2][JN];
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int i = 0; i < JN; ++i)
          jw[f][i] = agent_load(word_at(a.jslot, (f ? inN : inS) + i * RES_NT * 8u, t8));
      if (pubD) face_store(word_at(a.kslot, kslot0 + O * KF, opaque(8u * tt)), RES_NT, p[O][0], tagK, nearD);
      if (pubU) face_store(word_at(a.kslot, kslot0 + (2 + O) * KF, opaque(8u * tt)), RES_NT, p[O][TK - 1], tagK, nearU);
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int i = 0; i < JN; ++i) {
          while ((unsigned)(jw[f][i] >> 32) != (f ? tagN : tagS) && t + i * RES_NT < njw)
            jw[f][i] = poll_again(word_at(a.jslot, (f ? inN : inS) + i * RES_NT * 8u, t8), f ? tagN : tagS, budget);
          sJ[f][t + i * RES_NT] = __uint_as_float((unsigned)jw[f][i]);
        }
      lds_only_barrier();
    } else {
      if (pubD) face_store(word_at(a.kslot, kslot0 + O * KF, opaque(8u * tt)), RES_NT, p[O][0], tagK, nearD);
      if (pubU) face_store(word_at(a.kslot, kslot0 + (2 + O) * KF, opaque(8u * tt)), RES_NT, p[O][TK - 1], tagK, nearU);
    }
    if (active) {
      const u64 *kd = nullptr, *ku = nullptr;
      Face4 fd, fu;
      auto lds = [&](auto lc) {
        constexpr int l = decltype(lc)::value;
        return Lds{sP[O][l][tN], sP[O][l][tS],
                   reinterpret_cast<const float*>(&sP[O][l][0])[((C + l) & 1) ? x1 : x0]};
      };
      auto level = [&](auto lc, const Lds& m, float4 xn, float4 xs, float4 up, float4 dn) {
        constexpr int l = decltype(lc)::value;
        constexpr int b = (C + l) & 1;
        const float4 xm = p[O][l];
        const float4 pc4 = p[C][l], rr4 = r[C][l];
        const float4 cc = sC[kb * TK + l];
        // z[m], z[m + 1]: the west and east neighbours of the group's cell m.  Rows starting at
        // i = 1 take entries 4g-1 .. 4g+3 of the other colour, rows starting at 2 4g .. 4g+4
        auto sel = [&](float one, float two) { return b ? (s1 ? one : two) : (s1 ? two : one); };
        float z[5] = {sel(m.x, xm.x), sel(xm.x, xm.y), sel(xm.y, xm.z), sel(xm.z, xm.w),
                      sel(xm.w, m.x)};
        const float pcv[4] = {pc4.x, pc4.y, pc4.z, pc4.w}, rv[4] = {rr4.x, rr4.y, rr4.z, rr4.w};
        const float nv[4] = {xn.x, xn.y, xn.z, xn.w}, sv[4] = {xs.x, xs.y, xs.z, xs.w};
        const float uv[4] = {up.x, up.y, up.z, up.w}, dv[4] = {dn.x, dn.y, dn.z, dn.w};
        const bool row1 = b ? s1 : !s1;  // the row's first cell is i = 1
        z[0] = w0[b] ? pcv[0] : z[0];
#pragma unroll
        for (int q = 0; q < 4; ++q) z[q + 1] = eq[b][q] ? pcv[q] : z[q + 1];
        float out[4], sq[4];
        // entries of the group that are cells (the padding past i = ip is none)
        const int ncell = RESID ? ((d.ip - (row1 ? 1 : 2)) >> 1) + 1 - 4 * grp : 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float reltmp =
              om * (cc.x * (c2l * z[q + 1] + c2s * z[q] + c3l * nv[q] + c3s * sv[q] + cc.y * uv[q] +
                            cc.z * dv[q] - rv[q]) -
                    pcv[q]);
          out[q] = pcv[q] + reltmp;
          if constexpr (RESID) sq[q] = q < ncell ? reltmp * reltmp : 0.0f;
        }
        if constexpr (RESID) acc.add4(sq, sLimb[h >> 1 & 1u]);
        const float4 o4 = make_float4(out[0], out[1], out[2], out[3]);
        p[C][l] = o4;
        sP[C][l][t] = o4;
        if constexpr (l + 1 < TK)
          if (l == ltop) p[O][l + 1] = o4;
      };
      auto steps = [&](auto self, auto sc, const Lds& cur) -> void {
        constexpr int s = decltype(sc)::value;
        constexpr int l = lv(s);
        const std::integral_constant<int, l> lc{};
        Lds nxt = cur;
        if constexpr (s + 1 < TK) nxt = lds(std::integral_constant<int, lv(s + 1)>{});
        if constexpr (s == KL) {
          if (pubD) {
            kd = word_at(a.kslot, kslot0 - 4u * KF + (2 + O) * KF, opaque(8u * tt));
            fd = face_load<RES_NT>(kd);
          }
          if (pubU) {
            ku = word_at(a.kslot, kslot0 + 4u * KF + O * KF, opaque(8u * tt));
            fu = face_load<RES_NT>(ku);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (l < nlev) {
          float4 xn = cur.n, xs = cur.s;
          if (isJ) {
            const int o = ((kb * TK + l) * ng + grp) * 4;
            if (isN) xn = ld4(&sJ[1][o]);
            if (isS) xs = ld4(&sJ[0][o]);
          }
          float4 dn, up;
          if constexpr (l > 0) {
            dn = p[O][l - 1];
          } else {
            // below level 0: a face, another level block of this workgroup, or the image
            dn = p[C][0];
            if (pubD)
              dn = face_wait<RES_NT>(fd, kd, tagK, budget);
            else if (!KS1 && !bottom)
              dn = sP[O][TK - 1][max(t - blk, 0)];
          }
          if constexpr (l < TK - 1) {
            up = p[O][l + 1];
          } else {
            up = p[C][l];
            if (pubU)
              up = face_wait<RES_NT>(fu, ku, tagK, budget);
            else if (!KS1 && ltop != TK - 1)
              up = sP[O][0][min(t + blk, NS - 1)];
          }
          level(lc, cur, xn, xs, up, dn);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (s + 1 < TK) self(self, std::integral_constant<int, s + 1>{}, nxt);
      };
      steps(steps, std::integral_constant<int, 0>{}, lds(std::integral_constant<int, lv(0)>{}));
    }
    lds_only_barrier();
  };
  if constexpr (RESID) acc.start(1.0);
  unsigned nexact = 0u;
  for (unsigned it = 0; it < (unsigned)a.nmaxp; ++it) {
    half(std::integral_constant<int, 1>{}, 2u * it);
    half(std::integral_constant<int, 0>{}, 2u * it + 1u);
    if constexpr (RESID) {
      // All workgroups exchange their sums, rounded to FP64, in one hop and add them up alike.
      // Well above pjuge that settles it; near or below it, and after the last iteration (whose
      // residual is kept), the exact sum decides.
      const unsigned par = it & 1u, tag = base_tag + 1u + it;
      acc.flush(sUnit[par]);
      __syncthreads();
      if (t < NLIMB) sLimb[par ^ 1u][t] = 0;
      if (t < 2) sUnit[par ^ 1u][t] = 0;
      double sum = 0.0;
      if (t == 0) {
        sum = acc.value(sUnit[par], sLimb[par]);
        const u64 v = (u64)__double_as_longlong(sum);
        if (nwg > 1) {
          agent_store(&a.ctl->sums[par][0][wg], ((u64)tag << 32) | (v & 0xffffffffull));
          agent_store(&a.ctl->sums[par][1][wg], ((u64)tag << 32) | (v >> 32));
          sum = 0.0;
        }
      }
      for (int w = t; nwg > 1 && w < nwg; w += RES_NT) {
        u64 lo = agent_load(&a.ctl->sums[par][0][w]), hi = agent_load(&a.ctl->sums[par][1][w]);
        while ((unsigned)(lo >> 32) != tag) lo = poll_again(&a.ctl->sums[par][0][w], tag, budget);
        while ((unsigned)(hi >> 32) != tag) hi = poll_again(&a.ctl->sums[par][1][w], tag, budget);
        if (budget <= 0) hi = 0x7ff80000u;  // NaN: to the exact sum's path
        sum += __longlong_as_double((long long)(hi << 32 | (lo & 0xffffffffull)));
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
      if ((t & 63) == 0) sWave[t >> 6] = sum;
      __syncthreads();
      sum = 0.0;
#pragma unroll
      for (int w = 0; w < RES_NT / 64; ++w) sum += sWave[w];
      if (it + 1u == (unsigned)a.nmaxp || !(sum > (double)a.pjuge * (1.0 + 1e-6))) {
        if (t == 0) acc.fold(sUnit[par], sLimb[par]);
        if (res_add_limbs(a, sLimb[par], &a.ctl->added, (unsigned)nwg * ++nexact, sSum, &sCtl[2])) {
          if (t == 0) sCtl[2] = res_decide(a, sSum, it + 1u);
        } else if (t == 0) {
          unsigned dec;
          while ((dec = agent_load(&a.ctl->decided)) >> 1 < it + 1u && budget > 0) {
            --budget;
            __builtin_amdgcn_s_sleep(1);
          }
          sCtl[2] = dec;
        }
        __syncthreads();
        if (sCtl[2] & 1u) break;
      }
      acc.start(sum);
    }
  }

  if (active) {
#pragma unroll
    for (int l = 0; l < TK; ++l) {
      if (l >= nlev) continue;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int i0 = first_of(c, j, k0 + l) + 8 * grp;
        float4 x = p[c][l];
        if (i0 > d.ip) x.x = 0.0f;
        if (i0 + 2 > d.ip) x.y = 0.0f;
        if (i0 + 4 > d.ip) x.z = 0.0f;
        if (i0 + 6 > d.ip) x.w = 0.0f;
        st4(sp.p[c] + off0 + l * lstride, x);
      }
    }
  }
  if (budget <= 0) {
    __hip_atomic_fetch_or(&a.ctl->base, RES_FAILED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);  // before this workgroup is counted as done
  }
  res_leave(a, false);
}

}  // namespace

// The cut with the least estimated time per sweep in us, fitted to the times of 40 cuts of
// 150x150x90 and 96x96x60 and of smaller grids: per level 0.25 plus 0.045 for each wavefront of the
// busiest SIMD; 0.9 for any faces, 0.28 per 1000 words of the k faces, 0.25 and 0.1 per 1000 words
// for j faces, 0.15 where the XCDs' shares cut through a row of workgroups along k.  It prefers cuts
// about as high as they are long: 96x96x60 in 8 levels x 5 rows takes 1.7 us a sweep, in 1 x 32 2.3;
// 150x150x90 in 6 x 13 2.6, in 3 x 25 2.9.
ResPlan res_plan(Dims d, int nr, int ncu) {
  ncu = std::min(ncu, RES_WGMAX);
  ResPlan best;
  double best_cost = 0.0;
  const int ng = nr / 4;
  for (int tk = 1; tk <= RES_TKMAX; ++tk) {
    const int ns = res_ns(tk), maxrows = std::min(d.jp, ns / ng);
    if (maxrows < 1 || ng > RES_JS) continue;
    for (int njt = (d.jp + maxrows - 1) / maxrows; njt <= std::min(ncu, std::max(1, d.jp / 2)); ++njt) {
      const int rj = (d.jp + njt - 1) / njt;
      const int ksmax = tk > RES_TK_KS ? 1 : std::min(std::min(ns / (rj * ng), (d.kp + tk - 1) / tk), RES_KWMAX / tk);
      for (int ks = 1; ks <= ksmax; ++ks) {
        const int nkt = (d.kp + ks * tk - 1) / (ks * tk);
        if ((long)njt * nkt > ncu || 4 * ng * ks * tk > res_jn(tk) * RES_NT) continue;
        const int waves = (rj * ks * ng + 63) / 64;
        const bool fk = nkt > 1, fj = njt > 1 || d.jp % 2;
        const double cost = tk * (0.25 + 0.045 * ((waves + 3) / 4)) + (fk || fj ? 0.9 : 0.0) +
                            (fk ? 0.28e-3 * (8 * rj * ng) : 0.0) +
                            (fj ? 0.25 + 0.1e-3 * (8 * ks * tk * ng) : 0.0) +
                            (fj && njt % 8 ? 0.15 : 0.0) + 1e-4 * njt * nkt;
        if (best.tk == 0 || cost < best_cost) {
          best_cost = cost;
          best.tk = tk;
          best.ks = ks;
          best.rj = rj;
          best.njt = njt;
          best.nkt = nkt;
        }
      }
    }
  }
  return best;
}

namespace {
size_t kwords(const ResPlan* pl, int n) {
  size_t w = 0;
  for (int q = 0; q < n; ++q) w = std::max(w, (size_t)pl[q].nwg() * 2 * 2 * 4 * RES_NT);
  return w;
}
size_t jwords(Dims d, const ResPlan* pl, int n) {
  size_t w = 0;
  for (int q = 0; q < n; ++q)
    w = std::max(w, (size_t)pl[q].nwg() * (d.jp % 2 ? 2 : 1) * 2 * 2 * res_jn(pl[q].tk) * RES_NT);
  return w;
}
size_t seam_floats(Dims d, int nr) { return (size_t)2 * d.kp * nr; }
}  // namespace

size_t res_bytes(Dims d, int nr, const ResPlan* pl, int n) {
  return (kwords(pl, n) + jwords(d, pl, n)) * sizeof(u64) + seam_floats(d, nr) * sizeof(float) + sizeof(ResCtl);
}

hipError_t res_alloc(Dims d, int nr, const ResPlan* pl, int n, hipStream_t st, ResBuf& b) {
  const size_t nk = kwords(pl, n), nj = jwords(d, pl, n), ns = seam_floats(d, nr);
  hipError_t e = hipMalloc(&b.kslot, nk * sizeof(u64));
  if (e == hipSuccess) e = hipMalloc(&b.jslot, nj * sizeof(u64));
  if (e == hipSuccess) e = hipMalloc(&b.seam, ns * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&b.ctl, sizeof(ResCtl));
  if (e == hipSuccess) e = hipHostMalloc(&b.host, sizeof(ResHost), hipHostMallocDefault);
  if (e == hipSuccess) *b.host = ResHost{};
  if (e == hipSuccess) e = hipMemsetAsync(b.kslot, 0, nk * sizeof(u64), st);
  if (e == hipSuccess) e = hipMemsetAsync(b.jslot, 0, nj * sizeof(u64), st);
  ResCtl c0{};
  c0.base = 1u;
  c0.host = b.host;
  if (e == hipSuccess) e = hipMemcpyAsync(b.ctl, &c0, sizeof c0, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) res_free(b);
  return e;
}

void res_free(ResBuf& b) {
  if (b.kslot) hipFree(b.kslot);
  if (b.jslot) hipFree(b.jslot);
  if (b.seam) hipFree(b.seam);
  if (b.ctl) hipFree(b.ctl);
  if (b.host) hipHostFree(b.host);
  b = ResBuf{};
}

namespace {
template <int TK, bool RESID>
void launch_tk(hipStream_t st, const ResArgs& a) {
  constexpr int NS = res_ns(TK);
  const dim3 grid(a.pl.nwg()), blk(RES_NT);
  if (a.pl.ks == 1)
    hipLaunchKernelGGL((k_sor_resident<TK, NS, true, RESID>), grid, blk, 0, st, a);
  if constexpr (TK <= RES_TK_KS)
    if (a.pl.ks > 1) hipLaunchKernelGGL((k_sor_resident<TK, NS, false, RESID>), grid, blk, 0, st, a);
}
template <int TK>
void launch_tk(hipStream_t st, const ResArgs& a) {
  if (a.slots)
    launch_tk<TK, true>(st, a);
  else
    launch_tk<TK, false>(st, a);
}
}  // namespace

void launch_sor_resident(hipStream_t st, Dims d, Grid1D g, SplitSOR sp, Physics ph, int nmaxp,
                         DevScalars* sc, int sub_rhsav, int sub_pav, float* rout0, float* rout1,
                         int64_t* resid_slots, const ResPlan& pl, const ResBuf& b, long wait_ticks,
                         int polls) {
  ResArgs a{d, g, sp, ph.omega, nmaxp, sc, sub_rhsav, sub_pav, {rout0, rout1}, ph.pjuge, resid_slots, pl,
            b.kslot, b.jslot, b.seam, b.ctl, wait_ticks, polls};
  switch (pl.tk) {
    case 1: launch_tk<1>(st, a); break;
    case 2: launch_tk<2>(st, a); break;
    case 3: launch_tk<3>(st, a); break;
    case 4: launch_tk<4>(st, a); break;
    case 5: launch_tk<5>(st, a); break;
    case 6: launch_tk<6>(st, a); break;
    case 7: launch_tk<7>(st, a); break;
    case 8: launch_tk<8>(st, a); break;
    case 9: launch_tk<9>(st, a); break;
    case 10: launch_tk<10>(st, a); break;
    default: break;
  }
}

}  // namespace les
