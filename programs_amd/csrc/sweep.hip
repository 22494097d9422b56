// The one-launch triangular sweeps and factorisations (SweepPlan): DIC /
// DILU of spray-simulation (solv_precond.f90:10-29, solv_direct.f90:11-42)
// and flowlab's factor (solv_m.f90:224-286).  Each row performs the
// reference's operations in its order; only the order between independent
// rows differs, so results equal the sequential loops bit for bit.
//
// A block takes parts of the plan from a ticket counter, in an order in
// which a part only needs values of parts taken before it (no deadlock
// whatever the residency), and runs a part with eight waves:
//   wave 0 computes: it walks the part's chunks (up to 64 rows that do not depend
//     on each other) in order.  All values it reads sit in LDS, its own
//     rows' and the halo's; a wave's LDS operations are in order, so chunk
//     after chunk needs no barrier.  Matrix entries, factor and records are
//     stored by position, so that a chunk's loads are consecutive, and are
//     issued up to eight chunks ahead.  Values that other parts need go to
//     the export buffer at once (agent scope).
//   wave 1 fetches the halo: it polls the export buffer for the values of
//     other parts, in the order in which the chunks need them, puts them
//     into LDS and publishes how many are there.
// All waves load a part's tables and first values into LDS, and store its
// results from there when it is done.
//
// Export slots hold kSweepMark (a signalling NaN: no arithmetic result has
// this pattern) until their value arrives.  A launch marks the buffer of the
// other direction, so no launch is spent on marking.  A halo wave's waits
// are bounded (kSweepSpin polls; 256 once an error is recorded); past the
// bound it records the error, the compute wave runs through what is left on
// what is there and the block stops taking parts.
//
// What bounds it: the chain of chunks a path runs through (LDS read, five
// dependent FP64 operations, LDS write) and the crossings between parts
// (store, poll, reload), not bandwidth.  A chunk is 42 instructions of one
// wave, each at least four cycles: records whose words are LDS addresses as
// they are and are taken apart in the shadow of the LDS reads, a wait loop out
// of line, and loads first issued in the loop's order (else a ring of chunks
// begins by waiting for loads two chunks old) took 15 instructions and those
// waits out: 42 -> 38 us at 24^3, 189 -> 163 at 96^3, 294 -> 250 at 128^3.
// Bricks of 8 x 8 columns, one poll in flight a block and more threads beside
// the chunks took them to 32, 137 and 207 us.  One application of DIC to one
// right-hand side (both sweeps), against the form it replaced (ranges of 4096
// consecutive rows, a level at a time): 24^3 32 us (177), 96^3 137 us (620),
// 128^3 207 us (1232); DILU to three at 128^3 314 us (1823).
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>

#include "ctx.h"
#include "sweep.h"
#include "sweepexec.h"

namespace fvk {

// a compute wave, a halo wave, and six that help to load a part and to store
// it (both sweeps, 24^3 / 96^3 / 128^3: 33.8 / 144 / 233 us with 192 threads)
constexpr int SW_TB = 512;
// chunks whose loads are in flight: at most 8, and at most 56 loads and
// exports (a wave counts 63)
constexpr int sweep_ahead(int MW, int KIND) {
  const int ops = (MW == 8 ? 2 : 1) + MW * (KIND == 2 ? 2 : 1) + (KIND == 0 ? 1 : 0) + 1;
  return ops * 8 <= 56 ? 8 : 56 / ops;
}

struct SweepArgs {
  int P, np, slots, NE, NEo, n, width;
  unsigned shared;            // LDS address of the block's shared scalars
  const int *part, *prow, *ppos, *hsrc;
  const unsigned short *pslot, *rec;
  const double *a, *a2, *c;   // by position
  const double *src, *cr;     // initial values of the rows; backward: their scale
  const int *dix;
  double *dst;
  double *E, *Eo;
  int *ticket, *ticket_o, *err;
  double *crow, *drow, *cpos, *crr;  // factor
  SweepGate gate;
};

// A block's LDS, by byte address from 0 (the kernels have no static LDS, which
// the host checks): values of component q at slot offset + q ld, the halo's
// sources, and the scalars shared by the block's waves at Shared.  Plain
// addresses, so that a record's 16-bit offset is an address as it is.
enum { SH_PART = 0, SH_HAVE = 4, SH_ABORT = 8, kShared = 16 };
template <class T>
using lds_t = __attribute__((address_space(3))) T;
__device__ __forceinline__ double lds_value(unsigned at) { return *(lds_t<double> *)(uintptr_t)at; }
__device__ __forceinline__ void lds_put(unsigned at, double v) { *(lds_t<double> *)(uintptr_t)at = v; }
__device__ __forceinline__ int lds_int(unsigned at) { return *(lds_t<int> *)(uintptr_t)at; }
__device__ __forceinline__ void lds_put(unsigned at, int v) { *(lds_t<int> *)(uintptr_t)at = v; }
__device__ __forceinline__ int lds_get(unsigned at) {
  return __hip_atomic_load((lds_t<int> *)(uintptr_t)at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_post(unsigned at, int v) {
  __hip_atomic_store((lds_t<int> *)(uintptr_t)at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// this wave's LDS operations so far are done
__device__ __forceinline__ void lds_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

typedef const __attribute__((address_space(1))) char *global_p;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
template <class T>
__device__ __forceinline__ T ld_at(global_p base, unsigned byte) {
  return *(const __attribute__((address_space(1))) T *)(base + byte);
}

typedef __attribute__((address_space(1))) char *global_w;
// agent scope, as ld_agent and st_agent
__device__ __forceinline__ unsigned long long ld_agent_at(global_p base, unsigned byte) {
  return __hip_atomic_load((const __attribute__((address_space(1))) unsigned long long *)(base + byte), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_at(global_w base, unsigned byte, double v) {
  __hip_atomic_store((__attribute__((address_space(1))) unsigned long long *)(base + byte),
                     (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// what a lane needs to run its row of a chunk
template <int MW>
struct SweepStage {
  unsigned w[MW <= 4 ? 4 : 6];  // the record's 16-bit words in pairs
  double a[MW], a2[MW], c;
  __device__ __forceinline__ unsigned word(int t) const { return t & 1 ? w[t / 2] >> 16 : w[t / 2] & 0xffffu; }
  __device__ __forceinline__ int need() const { return (int)word(MW <= 4 ? 5 : 9); }
  __device__ __forceinline__ int exp() const { return (int)w[MW <= 4 ? 3 : 5]; }
};

// uniform base pointers of the loads by position (opaque, so that each load
// is one instruction with a scalar base and a 32-bit offset)
template <int MW>
struct SweepBase {
  global_p rec, a[MW], a2[MW], c;
};
__device__ __forceinline__ global_p opaque(const void *p) {
  global_p q = (global_p)p;
  asm volatile("" : "+s"(q));
  return q;
}

// KIND 0: sweep; 1: DIC factor, entries (a a) v; 2: factor, entries (a v) a2
template <int MW, int KIND>
__device__ __forceinline__ void sweep_load(const SweepBase<MW> &B, unsigned bo, SweepStage<MW> &S) {
  const u32x4 x = ld_at<u32x4>(B.rec, bo * (MW <= 4 ? 2u : 4u));
#pragma unroll
  for (int k = 0; k < 4; ++k) S.w[k] = x[k];
  if (MW > 4) {
    const u32x2 y = ld_at<u32x2>(B.rec, bo * 4u + 16u);
    S.w[MW > 4 ? 4 : 0] = y[0];
    S.w[MW > 4 ? 5 : 0] = y[1];
  }
#pragma unroll
  for (int t = 0; t < MW; ++t) {
    S.a[t] = ld_at<double>(B.a[t], bo);
    if (KIND == 2) S.a2[t] = ld_at<double>(B.a2[t], bo);
  }
  if (KIND == 0) S.c = ld_at<double>(B.c, bo);
}

// The chunks of a part.  The groups of kAhead + 1 chunks are straight code
// but for the (rare) wait for the halo, so that the compiler can count the
// loads in flight and waits for the oldest only; a chunk's loads go to the
// stage that the chunk before has freed, while this chunk's LDS reads are
// on their way.
template <bool FWD, int NC, int MW, int KIND>
__device__ __forceinline__ void sweep_compute(const SweepArgs &A, int c0, int nch, unsigned ld) {
  constexpr int kAhead = sweep_ahead(MW, KIND), kRing = kAhead + 1;
  SweepBase<MW> B;
  B.rec = opaque(A.rec);
#pragma unroll
  for (int t = 0; t < MW; ++t) {
    B.a[t] = opaque(A.a + (size_t)t * A.np);
    if (KIND == 2) B.a2[t] = opaque(A.a2 + (size_t)t * A.np);
  }
  if (KIND == 0) B.c = opaque(A.c);
  // lanes beyond the width repeat its last lane: the same row, the same values
  const unsigned lane8 = min((int)threadIdx.x, A.width - 1) * 8u;
  // a power of two, in a vector register: one instruction shifts and adds
  unsigned shift = 31u - __builtin_clz((unsigned)A.width * 8u);
  asm volatile("" : "+v"(shift));
  // byte offset of the j-th chunk in the sweep's direction (clamped to the part's last)
  auto at = [&](int j) {
    const int jj = min(j, nch - 1);
    return ((unsigned)(FWD ? c0 + jj : c0 + nch - 1 - jj) << shift) + lane8;
  };
  SweepStage<MW> S[kRing];
#pragma unroll
  for (int u = 0; u < kAhead; ++u) {
    sweep_load<MW, KIND>(B, at(u), S[u]);
    // in the loop's order: else its waits count on the other order as well
    __builtin_amdgcn_sched_barrier(0);
  }
  int have = 0;
  // the chunk about to run: its LDS addresses and halo need, taken while
  // the reads of the chunk before are on their way
  unsigned off[MW + 1], eoff = 0;
  int nd = 0;
  global_w E[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) E[q] = (global_w)opaque(A.E + (size_t)q * A.NE);
  // (opaque: taken apart here and not between this chunk's write and the next
  // chunk's reads, which is on the chain)
  auto prep = [&](const SweepStage<MW> &Y) {
#pragma unroll
    for (int t = 0; t <= MW; ++t) {
      off[t] = Y.word(t);
      asm volatile("" : "+v"(off[t]));
    }
    eoff = (unsigned)Y.exp() << 3;
    asm volatile("" : "+v"(eoff));
    nd = __builtin_amdgcn_readfirstlane(Y.need());
  };
  auto run = [&](const SweepStage<MW> &X, const SweepStage<MW> &Y, auto ahead) {
    while (__builtin_expect(nd > have, 0)) {
      have = __builtin_amdgcn_readfirstlane(lds_get(A.shared + SH_HAVE));
      // the halo wave gave up: the rest of the part runs on what is there
      if (nd > have && __builtin_amdgcn_readfirstlane(lds_get(A.shared + SH_ABORT))) have = INT_MAX;
    }
    asm volatile("" ::: "memory");
    double acc[NC], v[MW][NC], r[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) acc[q] = lds_value(off[0] + q * ld);
#pragma unroll
    for (int t = 0; t < MW; ++t)
#pragma unroll
      for (int q = 0; q < NC; ++q) v[t][q] = lds_value(off[1 + t] + q * ld);
    __builtin_amdgcn_sched_barrier(0);
    ahead();
    const unsigned own = off[0], eo = eoff;
    prep(Y);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < MW; ++t)
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        if (KIND == 0) acc[q] = acc[q] - X.a[t] * v[t][q];
        else if (KIND == 1) acc[q] = acc[q] - X.a[t] * X.a[t] * v[t][q];
        else acc[q] = acc[q] - X.a[t] * v[t][q] * X.a2[t];
      }
    if (KIND == 0) {
#pragma unroll
      for (int q = 0; q < NC; ++q) lds_put(own + q * ld, r[q] = acc[q] * X.c);
    } else {
      lds_put(own, r[0] = 1.0 / (acc[0] + SMALL));
      lds_put(own + ld, acc[0]);
    }
    if (X.exp() >= 0)
#pragma unroll
      for (int q = 0; q < NC; ++q) st_at(E[q], eo, r[q]);
    __builtin_amdgcn_sched_barrier(0);
  };
  prep(S[0]);
  int j0 = 0;
  for (; j0 + kRing <= nch; j0 += kRing) {
#pragma unroll
    for (int u = 0; u < kRing; ++u)
      run(S[u], S[(u + 1) % kRing],
          [&] { sweep_load<MW, KIND>(B, at(j0 + u + kAhead), S[(u + kAhead) % kRing]); });
  }
  // fewer than kRing chunks are left, all of them loaded
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
    if (j0 + u < nch) run(S[u], S[(u + 1) % kRing], [] {});
}

// The halo of a part: lane l fetches the values l, l + 64, ... of the part's
// list, in the order in which the chunks need them.  One wave with one poll in
// flight: polls are misses to the fabric, and more of them (two waves, several
// polls in flight, two values a lane) delay the answers by more than they save,
// while fewer lanes cannot keep up with the chunks (DIC at 96^3, both sweeps,
// with 192 threads: 141 us; two polls in flight 145; two values a lane 150; two
// waves 151, with two, four, eight polls in flight 156, 187, 279; 32 lanes 199).
template <int NC>
__device__ __forceinline__ void sweep_halo(const SweepArgs &A, int nh, int nr, unsigned ld, unsigned hsrc) {
  if (nh == 0) return;
  const int lane = threadIdx.x & 63;
  auto source = [&](int e) { return (unsigned)lds_int(hsrc + 4u * min(e, nh - 1)) << 3; };
  int cur = lane;  // the value this lane is at; past the last, nothing is asked of the answers
  unsigned src = source(lane), nxt = source(lane + 64);
  int at = 0, pub = 0;  // every lane is at its value number at / 64 or beyond; published
  unsigned spin = 0;
  global_p E[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) E[q] = opaque(A.E + (size_t)q * A.NE);
  for (;;) {
    unsigned long long v[NC];
    bool ready = cur < nh;
#pragma unroll
    for (int q = 0; q < NC; ++q) v[q] = ld_agent_at(E[q], src);
#pragma unroll
    for (int q = 0; q < NC; ++q) ready = ready && v[q] != kSweepMark;
    if (ready) {
      const unsigned o = (unsigned)(nr + cur) * 8u;
#pragma unroll
      for (int q = 0; q < NC; ++q) lds_put(o + q * ld, __longlong_as_double((long long)v[q]));
      cur += 64;
      src = nxt;
      nxt = source(cur + 64);
    }
    // a lane takes one step at most, so `at` takes one at most
    unsigned long long m = __ballot(cur < at + 64);
    at = m ? at : at + 64;
    m = m ? m : __ballot(cur < at + 64);
    const int have = min(nh, at + (m ? __builtin_ctzll(m) : 64));
    if (have > pub) {
      pub = have;
      spin = 0;
      lds_done();
      lds_post(A.shared + SH_HAVE, have);
      if (pub == nh) return;
    } else if (++spin > kSweepSpin ||
               ((spin & 255u) == 0 && __hip_atomic_load(A.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
      __hip_atomic_store(A.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      lds_post(A.shared + SH_ABORT, 1);
      return;
    }
  }
}

template <bool FWD, int NC, int MW, int KIND>
__global__ __launch_bounds__(SW_TB) void k_sweep(SweepArgs A) {
  if (A.gate.done) {
    bool all = true;
    for (int q = 0; q < A.gate.n; ++q) all = all && A.gate.done[q * A.gate.stride];
    if (all) return;
  }
  constexpr int NV = KIND == 0 ? NC : 2;  // values per slot (factor: c and d)
  const unsigned ld = (unsigned)A.slots * 8u;
  const unsigned hsrc = NV * ld;
  const int tid = threadIdx.x, wave = tid >> 6;
  if (KIND == 0) {
    // the other direction's export buffer, for the launch after this one
    const size_t m = (size_t)NC * A.NEo;
    for (size_t i = blockIdx.x * (size_t)SW_TB + tid; i < m; i += (size_t)gridDim.x * SW_TB)
      ((unsigned long long *)A.Eo)[i] = kSweepMark;
    if (blockIdx.x == 0 && tid == 0) *A.ticket_o = 0;
  }
  // Between a barrier and the loop that stores a part, and not after that loop,
  // whose trip count is a thread's own: the compiler may join a branch at the
  // end of a loop's body with one that follows, and threads that skip both then
  // reach the next barrier without a ticket.  The stores hide its latency.
  auto ticket = [&] {
    if (tid == 0) {
      lds_put(A.shared + SH_PART, atomicAdd(A.ticket, 1));
      lds_put(A.shared + SH_HAVE, 0);
    }
  };
  if (tid == 0) lds_put(A.shared + SH_ABORT, 0);
  ticket();
  for (;;) {
    __syncthreads();
    const int o = __builtin_amdgcn_readfirstlane(lds_int(A.shared + SH_PART));
    if (o >= A.P) return;
    const int q = FWD ? o : A.P - 1 - o;
    const int *Q = A.part + 8 * q;
    const int c0 = Q[0], nch = Q[1], r0 = Q[2], nr = Q[3], h0 = FWD ? Q[4] : Q[6], nh = FWD ? Q[5] : Q[7];
    // rows' initial values and the part's tables into LDS
    for (int k0 = tid; k0 < nr; k0 += 4 * SW_TB) {
      int kk[4], row[4];
      unsigned off[4];
      double v[4][NC], s[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        kk[i] = r0 + min(k0 + i * SW_TB, nr - 1);
        off[i] = A.pslot[kk[i]];
        if (FWD) row[i] = A.prow[kk[i]];
        else s[i] = A.cr[kk[i]];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int z = !FWD ? kk[i] : KIND != 0 && A.dix ? A.dix[row[i]] : row[i];
#pragma unroll
        for (int c = 0; c < NC; ++c) v[i][c] = A.src[(size_t)c * A.n + z];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (k0 + i * SW_TB < nr)
#pragma unroll
          for (int c = 0; c < NC; ++c) lds_put(off[i] + c * ld, FWD ? v[i][c] : v[i][c] * s[i]);
    }
    for (int h = tid; h < nh; h += SW_TB) lds_put(hsrc + 4u * h, A.hsrc[h0 + h]);
    if (tid < 2 * NV) lds_put((unsigned)(nr + nh + (tid & 1)) * 8u + (tid >> 1) * ld, 0.0);
    __syncthreads();
    // the halo waves of other blocks poll on the same SIMD
    if (wave == 0) __builtin_amdgcn_s_setprio(3);
    if (wave == 0) sweep_compute<FWD, NC, MW, KIND>(A, c0, nch, ld);
    else if (wave == 1) sweep_halo<NC>(A, nh, nr, ld, hsrc);
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(lds_int(A.shared + SH_ABORT))) return;
    ticket();
    for (int k = tid; k < nr; k += SW_TB) {
      const unsigned off = A.pslot[r0 + k];
      if (KIND == 0) {
        const int z = FWD ? r0 + k : A.prow[r0 + k];
#pragma unroll
        for (int c = 0; c < NC; ++c) A.dst[(size_t)c * A.n + z] = lds_value(off + c * ld);
      } else {
        const int row = A.prow[r0 + k];
        const double c = lds_value(off), d = lds_value(off + ld);
        A.crow[row] = c;
        if (A.drow) A.drow[row] = d;
        A.cpos[A.ppos[r0 + k]] = c;
        A.crr[r0 + k] = A.drow ? d : 1.0 / (c + SMALL);
      }
    }
  }
}

__global__ __launch_bounds__(BS) void k_export_mark(size_t cnt, double *__restrict__ out) {
  for (size_t i = blockIdx.x * (size_t)BS + threadIdx.x; i < cnt; i += (size_t)gridDim.x * BS)
    ((unsigned long long *)out)[i] = kSweepMark;
}

// entry values by position; the factorisation's export buffer and ticket
__global__ __launch_bounds__(BS) void k_sweep_pack(int np, int MW, const int *__restrict__ lval,
                                                   const int *__restrict__ uval, const int *__restrict__ tval,
                                                   const double *__restrict__ vals, const double *__restrict__ tvals,
                                                   double *__restrict__ aL, double *__restrict__ aU,
                                                   double *__restrict__ aT, int NE, double *__restrict__ Ec,
                                                   int *ticket) {
  const size_t i = blockIdx.x * (size_t)BS + threadIdx.x;
  if (i < (size_t)NE) ((unsigned long long *)Ec)[i] = kSweepMark;
  if (i == 0) *ticket = 0;
  if (i >= (size_t)np) return;
  for (int t = 0; t < MW; ++t) {
    const size_t o = (size_t)t * np + i;
    const int l = lval[o], u = uval[o];
    aL[o] = l >= 0 ? vals[l] : 0.0;
    aU[o] = u >= 0 ? vals[u] : 0.0;
    if (tvals) {
      const int x = tval[o];
      aT[o] = x >= 0 ? tvals[x] : 0.0;
    }
  }
}

__global__ __launch_bounds__(BS) void k_sweep_lower(size_t cnt, const int *__restrict__ idx,
                                                    const double *__restrict__ vals, double *__restrict__ a) {
  const size_t i = blockIdx.x * (size_t)BS + threadIdx.x;
  if (i < cnt) a[i] = idx[i] >= 0 ? vals[idx[i]] : 0.0;
}

__global__ __launch_bounds__(BS) void k_sweep_factor_from(int n, const int *__restrict__ prow,
                                                          const int *__restrict__ ppos,
                                                          const double *__restrict__ crow,
                                                          const double *__restrict__ drow, double *__restrict__ cpos,
                                                          double *__restrict__ crr) {
  const int k = blockIdx.x * BS + threadIdx.x;
  if (k >= n) return;
  cpos[ppos[k]] = crow[prow[k]];
  crr[k] = drow[prow[k]];
}

// ---------------------------------------------------------------- host
constexpr int kNoRoom = 1;
static int take(SweepExec &X, void **q, size_t bytes) {
  const hipError_t e = X.deny && X.mem.size() == 8 ? hipErrorOutOfMemory : hipMalloc(q, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    return kNoRoom;
  }
  FVK_HIP(e);
  X.mem.push_back(*q);
  return 0;
}
template <class T>
static int up(SweepExec &X, T **d, const std::vector<T> &v) {
  void *q = nullptr;
  const int rc = take(X, &q, std::max<size_t>(1, v.size()) * sizeof(T));
  if (rc) return rc;
  if (!v.empty()) FVK_HIP(hipMemcpy(q, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  *d = (T *)q;
  return 0;
}
// zeroed; the clear has finished when the build returns (it ends with a wait)
static int room(SweepExec &X, double **d, size_t n, hipStream_t s) {
  void *q = nullptr;
  const int rc = take(X, &q, std::max<size_t>(1, n) * sizeof(double));
  if (rc) return rc;
  FVK_HIP(hipMemsetAsync(q, 0, std::max<size_t>(1, n) * sizeof(double), s));
  *d = (double *)q;
  return 0;
}
static int mark(double *p, size_t cnt, hipStream_t s) {
  k_export_mark<<<(int)std::max<size_t>(1, std::min<size_t>((cnt + BS - 1) / BS, 4096)), BS, 0, s>>>(cnt, p);
  FVK_HIP(hipGetLastError());
  return 0;
}

template <int MW>
static int allow_lds() {
  const void *k[] = {(const void *)k_sweep<true, 1, MW, 0>,  (const void *)k_sweep<true, 2, MW, 0>,
                     (const void *)k_sweep<true, 3, MW, 0>,  (const void *)k_sweep<false, 1, MW, 0>,
                     (const void *)k_sweep<false, 2, MW, 0>, (const void *)k_sweep<false, 3, MW, 0>,
                     (const void *)k_sweep<true, 1, MW, 1>,  (const void *)k_sweep<true, 1, MW, 2>};
  for (const void *f : k) {
    hipFuncAttributes at;
    FVK_HIP(hipFuncGetAttributes(&at, f));
    if (at.sharedSizeBytes) { set_error("a sweep kernel has static LDS"); return FVK_ERR_STATE; }
    FVK_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kSweepLds + kShared));
  }
  return 0;
}

static int exec_build(SweepExec &X, const SweepPlan &p, hipStream_t s) {
  X.n = p.n; X.P = p.P; X.MW = p.MW; X.np = p.np; X.slots = p.slots; X.width = p.width; X.bricks = p.bricks;
  for (int k = 1; k <= 3; ++k) X.lds_[k] = p.lds(k);
  int rc = 0;
#define U(dst, src) if (!rc) rc = up(X, &dst, src)
#define R(dst, cnt) if (!rc) rc = room(X, &dst, cnt, s)
  U(X.part, p.part); U(X.prow, p.prow); U(X.ppos, p.ppos); U(X.pslot, p.pslot); U(X.tval, p.tval);
  const size_t mnp = (size_t)p.MW * p.np;
  for (int k = 0; k < 2; ++k) {
    SweepExec::Dir &D = X.d[k];
    const SweepPlan::Dir &S = p.d[k];
    D.NE = S.NE;
    U(D.rec, S.rec); U(D.val, S.val); U(D.hsrc, S.hsrc);
    R(D.E, (size_t)3 * D.NE); R(D.a, mnp);
    if (!rc) rc = mark(D.E, (size_t)3 * D.NE, s);
  }
  R(X.aT, mnp); R(X.c, p.np); R(X.cr, p.n); R(X.Ec, X.d[0].NE); R(X.t, (size_t)3 * p.n);
  double *tk = nullptr;
  R(tk, 2);
  X.ticket = (int *)tk;
#undef U
#undef R
  if (rc) return rc;
  if ((rc = X.MW == 3 ? allow_lds<3>() : X.MW == 4 ? allow_lds<4>() : allow_lds<8>())) return rc;
  FVK_HIP(hipStreamSynchronize(s));
  return 0;
}

int sweep_exec_build(SweepExec &X, const SweepPlan &p, hipStream_t s) {
  const int rc = exec_build(X, p, s);
  if (rc) {
    (void)hipStreamSynchronize(s);  // clears and marks still queued
    sweep_exec_free(X);
  }
  X.built = rc == 0;
  X.deny = false;
  return rc == kNoRoom ? 0 : rc;
}

void sweep_exec_free(SweepExec &X) {
  for (void *q : X.mem) hipFree(q);
  const int n_cu = X.n_cu, blocks = X.blocks;
  const bool deny = X.deny;
  X = SweepExec();
  X.n_cu = n_cu;
  X.blocks = blocks;
  X.deny = deny;
}

static SweepArgs args(const SweepExec &X, int dir) {
  SweepArgs A;
  const SweepExec::Dir &D = X.d[dir], &O = X.d[1 - dir];
  A.P = X.P; A.np = X.np; A.slots = X.slots; A.NE = D.NE; A.NEo = O.NE; A.n = X.n;
  A.width = X.width;
  A.part = X.part; A.prow = X.prow; A.ppos = X.ppos; A.pslot = X.pslot;
  A.rec = D.rec; A.hsrc = D.hsrc;
  A.a = D.a; A.a2 = nullptr; A.c = X.c; A.src = nullptr; A.cr = X.cr; A.dix = nullptr; A.dst = nullptr;
  A.E = D.E; A.Eo = O.E;
  A.ticket = X.ticket + dir; A.ticket_o = X.ticket + 1 - dir; A.err = nullptr;
  A.crow = A.drow = A.cpos = A.crr = nullptr;
  return A;
}

// Blocks of a launch, at most one a part and as many as can be resident by
// their LDS and 512 threads each.  Of a brick plan no more than one per CU or
// than run at a time (the front through the brick grid is about 2.25 P^(2/3)
// parts wide): those that wait poll.  Fewer than one per CU leave CUs without
// work, and more make little difference (DIC, both sweeps, us, with 128 / 192 /
// 256 / 512 / 1024 blocks: 96^3, 288 bricks, 256 blocks by the rule, 136.5 /
// 136.9 / 138.0 / 138.1 / 137.7; 128^3, 512 bricks, 256: 239 / 213 / 208 / 208 /
// 208; 192^3, 1728 bricks, 324: 630 / 504 / 448 / 447 / 445; 1M triangles, 980
// ranges, 768: 237 / 188 / 164 / 164 / 164).
static int grid(const SweepExec &X, size_t lds) {
  const int fit = X.n_cu * std::max(1, std::min(4, (int)(163840 / (lds + 512))));
  const int front = X.bricks ? std::max(X.n_cu, (int)(2.25 * std::cbrt((double)X.P * X.P))) : fit;
  return std::max(1, std::min({X.P, fit, X.blocks > 0 ? X.blocks : front}));
}

template <bool FWD, int NC, int KIND>
static void launch(const SweepExec &X, const SweepArgs &args, hipStream_t s) {
  const size_t room = (X.lds_[KIND == 0 ? NC : 2] + 15) / 16 * 16, lds = room + kShared;
  const int G = grid(X, lds);
  SweepArgs A = args;
  A.shared = (unsigned)room;
  if (X.MW == 3) k_sweep<FWD, NC, 3, KIND><<<G, SW_TB, lds, s>>>(A);
  else if (X.MW == 4) k_sweep<FWD, NC, 4, KIND><<<G, SW_TB, lds, s>>>(A);
  else k_sweep<FWD, NC, 8, KIND><<<G, SW_TB, lds, s>>>(A);
}

int sweep_pack(SweepExec &X, hipStream_t s, const double *vals, const double *tvals) {
  const int cnt = std::max(X.np, X.d[0].NE);
  k_sweep_pack<<<(cnt + BS - 1) / BS, BS, 0, s>>>(X.np, X.MW, X.d[0].val, X.d[1].val, X.tval, vals, tvals, X.d[0].a,
                                                  X.d[1].a, X.aT, X.d[0].NE, X.Ec, X.ticket + 2);
  FVK_HIP(hipGetLastError());
  return 0;
}

int sweep_lower(SweepExec &X, hipStream_t s, const double *vals, bool transposed) {
  const size_t cnt = (size_t)X.MW * X.np;
  k_sweep_lower<<<(unsigned)((cnt + BS - 1) / BS), BS, 0, s>>>(cnt, transposed ? X.tval : X.d[0].val, vals, X.d[0].a);
  FVK_HIP(hipGetLastError());
  return 0;
}

int sweep_factor(SweepExec &X, hipStream_t s, int kind, const double *diag, const int *dix, double *crow, double *drow,
                 int *err) {
  SweepArgs A = args(X, 0);
  A.src = diag; A.dix = dix; A.err = err; A.E = X.Ec; A.ticket = X.ticket + 2;
  A.crow = crow; A.drow = drow; A.cpos = X.c; A.crr = X.cr;
  // DIC: d - ngn ngn c; DILU: d - ngp c ngn; flowlab: s - a pc a^T
  A.a = kind == SWEEP_DILU ? X.aT : X.d[0].a;
  A.a2 = kind == SWEEP_DILU ? X.d[0].a : X.aT;
  if (kind == SWEEP_DIC) launch<true, 1, 1>(X, A, s);
  else launch<true, 1, 2>(X, A, s);
  FVK_HIP(hipGetLastError());
  return 0;
}

int sweep_factor_from(SweepExec &X, hipStream_t s, const double *crow, const double *drow) {
  k_sweep_factor_from<<<(X.n + BS - 1) / BS, BS, 0, s>>>(X.n, X.prow, X.ppos, crow, drow, X.c, X.cr);
  FVK_HIP(hipGetLastError());
  return 0;
}

int sweep_apply(SweepExec &X, hipStream_t s, int nc, const double *b, double *x, SweepGate gate, int *err) {
  SweepArgs A = args(X, 0), B = args(X, 1);
  A.src = b; A.dst = X.t; A.err = err; A.gate = gate;
  B.src = X.t; B.dst = x; B.err = err; B.gate = gate;
  if (nc == 1) {
    launch<true, 1, 0>(X, A, s);
    launch<false, 1, 0>(X, B, s);
  } else if (nc == 2) {
    launch<true, 2, 0>(X, A, s);
    launch<false, 2, 0>(X, B, s);
  } else {
    launch<true, 3, 0>(X, A, s);
    launch<false, 3, 0>(X, B, s);
  }
  FVK_HIP(hipGetLastError());
  return 0;
}

}  // namespace fvk
