// CG with a diagonal (or no) preconditioner as one resident launch.
//
// On meshes below a quarter million rows an iteration of the launch chain
// ([p, q = A p, p.q], [x, r, z, r.z]) is two kernels of 4 to 6 us whose work
// takes well under 1 us: what they spend is launch, cache maintenance at the
// kernel boundary, and reloading a matrix that has not changed.  Here the
// whole solve is one kernel: every row's entries, its x, r, p and the p of
// its neighbours stay in registers, and per iteration the workgroups of a
// case meet twice, in the p.q and the r.z reduction.
//
// Meeting without a kernel boundary: each workgroup publishes the sums of its
// 64-row groups as one 128-byte line of device-scope stores; every workgroup
// of the case reads all lines, polling the words still holding the unset
// pattern, and adds the groups in the order of the launch chain's reductions
// (so the solve equals the chain bit for bit: same row sums, same partial
// sums, same scalar updates).  A line per workgroup matters: 8-byte words of
// several writers in one line made a meeting of 128 workgroups take 2.3 us,
// a line each 1.0 us (an all-to-all of flags alone; 16 workgroups 0.8 and
// 1.0, 256 workgroups 2.6 and 1.5).  z, the one vector neighbours read, is
// stored at device scope and waited for before the r.z line is published,
// and loaded at device scope.  No fence is needed, and none writes back or
// invalidates an L2.  Each of the two reductions alternates between two
// areas; a line is reset by its owner while the other area is in use (see
// below).
//
// All workgroups must be resident at once.  The host launches at most one
// workgroup per compute unit over all solves in flight on the device
// (ResidentRoom), and every wait is bounded in time: past the bound a
// workgroup raises the abort word, marks its case's state and returns without
// its rows of x, and so does each one that then waits in vain.  At the last
// meeting the others may still find every sum and finish, so the host takes a
// case's result only where the state has stopped and is not marked
// (resident_done); otherwise it solves by launches from the start.
//
// Measured per CG iteration on one MI355X (400 iterations of a solve, 2D
// cavities, Jacobi, FP64), launch chain then resident: 8.8k rows 9.5 to 4.6 us,
// 32k 9.6 to 5.6, 65k 9.9 to 6.1, 130k 15.4 to 7.2, 262k 19.7 to 9.1; a batch
// of four (99k rows) 10.8 to 6.1.  What is left is the two meetings, 1.0 us
// each for the flags alone and about 2 us with the sums, the spread of the
// workgroups and the scalar update; the matrix is read once per solve.
#pragma once

#include "solver_common.h"

namespace xcal {

constexpr int kPersistNT = 512;              // threads per workgroup
constexpr int kPersistWaves = kPersistNT / 64;
constexpr int kPersistLine = 16;             // words of a workgroup's line
constexpr int kPersistWGs = 256;             // most workgroups (lines) of one case
constexpr int kPersistSlots = 2 * kPersistNT;  // most partial-sum slots of one case

// Kernel view of a PersistPlan (persist.hip)
struct PersistK {
  const int4* wg;      // per workgroup: first group, end group, case, its line in the case
  const int2* grp;     // group of at most 64 rows: first row, rows
  const int2* slotA;   // partial-sum slots of p.q: first word in the case's lines, groups
  const int2* slotB;   // of r.z
  const int4* seg;     // per case: slots [x, y) of A, [z, w) of B
  const int4* cwg;     // per case: first workgroup, workgroups, first row, unused
  int batch;           // the order the slots are added in (kb_finalize's or k_finalize's)
  int64_t words;       // kPersistLine x workgroups
  unsigned long long* area;  // 4 areas of `words`: A even, A odd, B even, B odd
  int* abort;
  long long limit;     // ticks of the 100 MHz clock a wait may take
};

// Word of a case's lines that holds its group g (counted from the case's
// first group), at KR rows per thread.
__host__ __device__ constexpr int persist_word(int g, int kr) {
  return g / (kPersistWaves * kr) * kPersistLine + g % (kPersistWaves * kr);
}

constexpr unsigned long long kUnset = ~0ull;  // a NaN no published sum has

template <class T>
__device__ inline T dev_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ inline void dev_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct PersistLDS {
  double word[kPersistWGs * kPersistLine];  // the case's published sums
  double slot[kPersistSlots];
  double own[kPersistLine];  // this workgroup's group sums
  double lds[4];
  double val;
  int stop, fail;
};

// Publishes this wavefront's group sums s (one per row of a thread); returns
// with every wavefront's in L.own.  WAIT: each wavefront first waits for its
// own stores, so that a reader of the line finds them.
template <bool LOCAL, bool WAIT, int KR>
__device__ inline void persist_publish(const double (&s)[KR], unsigned long long* line,
                                       PersistLDS& L) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < KR; ++j) {
    const double w = wave_sum(s[j]);
    if (lane == 0) L.own[wave + kPersistWaves * j] = w;
  }
  if (WAIT && !LOCAL) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (!LOCAL && threadIdx.x < kPersistWaves * KR) {
    unsigned long long b = (unsigned long long)__double_as_longlong(L.own[threadIdx.x]);
    if (b == kUnset) b = kUnset - 1;  // another NaN
    dev_store(line + threadIdx.x, b);
  }
}

// The slots a thread adds up in one reduction (t and t + kPersistNT of the
// case's n), in registers: first group and number of groups of each.
struct PersistSlots {
  int n, g0, c0, g1, c1;
};
__device__ inline PersistSlots persist_slots(const int2* __restrict__ slot, int s0, int s1) {
  const int n = s1 - s0, t = (int)threadIdx.x;
  const int2 a = t < n ? slot[s0 + t] : int2{0, 0};
  const int2 b = t + kPersistNT < n ? slot[s0 + t + kPersistNT] : int2{0, 0};
  return PersistSlots{n, a.x, a.y, b.x, b.y};
}

// Reads the case's nwg lines at `area` into L.word, polling unset words;
// false once a wait was given up.  Every thread of the workgroup calls it.
template <int KR>
__device__ inline bool persist_read(const PersistK& P, int nwg, const unsigned long long* area,
                                    PersistLDS& L) {
  const int t = (int)threadIdx.x;
  // up to four words per thread in flight; a line's unused words are skipped
  const int nw = nwg * kPersistLine;
  const bool used = (t & (kPersistLine - 1)) < kPersistWaves * KR;
  for (int i0 = t; used && i0 < nw; i0 += 4 * kPersistNT) {
    unsigned long long u[4];
    // past the last word: the same word of line 0 again
    auto at = [&](int v) {
      const int i = i0 + v * kPersistNT;
      return i < nw ? i : t & (kPersistLine - 1);
    };
#pragma unroll
    for (int v = 0; v < 4; ++v) u[v] = dev_load(area + at(v));
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = at(v);
      long long t0 = 0;
      for (int spin = 0; u[v] == kUnset; ++spin) {
        // bounded: give up past the limit or when another did, but not on a
        // word that was set while this wavefront was held up
        bool late = false;
        if ((spin & 63) == 63 || P.limit <= 0) {
          const long long now = wall_clock64();
          if (t0 == 0) t0 = now;
          late = now - t0 >= P.limit || dev_load(P.abort) != 0;
        }
        u[v] = dev_load(area + i);
        if (late && u[v] == kUnset) {
          dev_store(P.abort, 1);
          L.fail = 1;
          break;
        }
      }
      L.word[i] = __longlong_as_double((long long)u[v]);
    }
  }
  __syncthreads();
  return L.fail == 0;  // uniform: set before the barrier, never cleared
}

// Total of a reduction from its group sums (L.word, or, LOCAL, L.own), valid
// in thread 0, in the launch chain's order.
template <bool LOCAL, int KR>
__device__ inline double persist_total(const PersistK& P, const PersistSlots& R, PersistLDS& L) {
  const int t = (int)threadIdx.x;
  const double* word = LOCAL ? L.own : L.word;
  auto slot_sum = [&](int g, int c) {  // store_partial's order over a 256-row block
    double v[4], sum = 0.0;
#pragma unroll
    for (int w = 0; w < 4; ++w) v[w] = word[persist_word(w < c ? g + w : g, KR)];
#pragma unroll
    for (int w = 0; w < 4; ++w) sum = w < c ? sum + v[w] : sum;
    return sum;
  };
  if (t < R.n) L.slot[t] = slot_sum(R.g0, R.c0);
  if (t + kPersistNT < R.n) L.slot[t + kPersistNT] = slot_sum(R.g1, R.c1);
  __syncthreads();
  double a = 0.0;
  if (P.batch) {  // wave_sum_segment's order
    if (t < 64) {
      for (int j = t; j < R.n; j += 64) a += L.slot[j];
      a = wave_sum(a);
    }
    return a;
  }
  if (t < kBlock) {  // reduce_partials' order
    for (int j = t; j < R.n; j += kBlock) a += L.slot[j];
    a = wave_sum(a);
    if ((t & 63) == 0) L.lds[t >> 6] = a;
  }
  __syncthreads();
  a = 0.0;
  if (t == 0)
    for (int w = 0; w < kBlock / 64; ++w) a += L.lds[w];
  return a;
}

// A workgroup that leaves before the end of its case's solve marks the state.
__device__ inline void persist_leave(KS* ks) {
  if (threadIdx.x == 0) dev_store(&ks->gave_up, 1);
}

// The resident solve of one case by its workgroups.  LOCAL: the case has one
// workgroup, whose sums and z stay in LDS.
template <bool LOCAL, int G, int KR, class T>
__device__ inline void cg_persist_case(const PersistK& P, const int4 wg, const MatKT<T>& A,
                                       const T* __restrict__ S, T* __restrict__ x,
                                       const T* __restrict__ r, T* z, KS* ks, PersistLDS& L,
                                       T* zl) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  KS k = ks[wg.z];
  if (k.stop != STOP_NONE) return;  // uniform over the case's workgroups
  const int4 seg = P.seg[wg.z], cwg = P.cwg[wg.z];
  const int row0 = cwg.z;  // the case's first row
  const PersistSlots RA = persist_slots(P.slotA, seg.x, seg.y);
  const PersistSlots RB = persist_slots(P.slotB, seg.z, seg.w);
  bool in[KR];
  int32_t row[KR], cnt[KR];
  T av[KR][G], pj[KR][G];
  int32_t col[KR][G];
  T xi[KR], ri[KR], zi[KR], pi[KR], qi[KR], so[KR];
#pragma unroll
  for (int j = 0; j < KR; ++j) {
    const int g = wg.x + wave + kPersistWaves * j;
    const int2 q = P.grp[g < wg.y ? g : wg.x];
    in[j] = g < wg.y && lane < q.y;
    row[j] = in[j] ? q.x + lane : q.x;
    const int32_t k0 = A.rb[row[j]], k1 = A.re[row[j]];
    cnt[j] = (k1 - k0) / kSlice;
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int32_t e = k0 + min(u, cnt[j] - 1) * kSlice;
      col[j][u] = A.colval[e];
      av[j][u] = A.nz[e];
      pj[j][u] = T(0);
    }
    xi[j] = T(0);
    pi[j] = T(0);
    ri[j] = r[row[j]];
    zi[j] = z[row[j]];
    so[j] = S ? S[row[j]] : T(1);
    if (LOCAL) {
      if (in[j]) zl[row[j] - row0] = zi[j];
#pragma unroll
      for (int u = 0; u < G; ++u) col[j][u] -= row0;
    }
  }
  if (LOCAL) __syncthreads();
  // the case's lines of the even areas, and this workgroup's word of them
  unsigned long long* const aA = P.area + (int64_t)cwg.x * kPersistLine;
  unsigned long long* const aB = aA + 2 * P.words;
  const int line = wg.w * kPersistLine;
  int par = 0;
  T zz[KR][G];
  auto gather = [&] {
#pragma unroll
    for (int j = 0; j < KR; ++j)
#pragma unroll
      for (int u = 0; u < G; ++u) zz[j][u] = LOCAL ? zl[col[j][u]] : dev_load(z + col[j][u]);
  };
  gather();
  for (;;) {
    const T beta = (T)k.beta;
    double s[KR];
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      T acc = 0;
#pragma unroll
      for (int u = 0; u < G; ++u) {
        pj[j][u] = zz[j][u] + beta * pj[j][u];
        const T t = av[j][u] * pj[j][u];
        acc = u < cnt[j] ? acc + t : acc;
      }
      qi[j] = acc;
      pi[j] = zi[j] + beta * pi[j];
      s[j] = in[j] ? dd(pi[j], acc) : 0.0;
    }
    unsigned long long *lA = aA + par * P.words, *lB = aB + par * P.words;
    persist_publish<LOCAL, false>(s, lA + line, L);
    if (!LOCAL && !persist_read<KR>(P, cwg.y, lA, L)) return persist_leave(ks + wg.z);
    double tot = persist_total<LOCAL, KR>(P, RA, L);
    if (threadIdx.x == 0) {
      finalize(&k, FIN_CG_PAP, tot, 0.0);
      L.val = k.alpha;
      L.stop = k.stop;
    }
    __syncthreads();
    if (L.stop != STOP_NONE) break;  // uniform over the case
    const T al = (T)L.val;
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      xi[j] = xi[j] + al * pi[j];
      ri[j] = ri[j] + (-al) * qi[j];
      zi[j] = S ? so[j] * ri[j] : ri[j];
      if (in[j]) {
        if (LOCAL) zl[row[j] - row0] = zi[j];
        else dev_store(z + row[j], zi[j]);
      }
      s[j] = in[j] ? dd(ri[j], zi[j]) : 0.0;
    }
    if (!LOCAL && threadIdx.x < kPersistWaves * KR) {
      // Reset this workgroup's lines in the next iteration's areas.  Every
      // workgroup has published this iteration's p.q, so it has read the
      // last iteration's r.z and, before that, its p.q: nobody reads these
      // areas.  The resets and the new z are complete (each wavefront waits
      // for its own) before this workgroup's r.z line is stored, and nobody
      // reads the next iteration's areas or z before having read every r.z
      // line.
      dev_store(aA + (par ^ 1) * P.words + line + threadIdx.x, kUnset);
      dev_store(aB + (par ^ 1) * P.words + line + threadIdx.x, kUnset);
    }
    persist_publish<LOCAL, true>(s, lB + line, L);
    if (!LOCAL && !persist_read<KR>(P, cwg.y, lB, L)) return persist_leave(ks + wg.z);
    gather();  // every new z is there: its loads overlap the sum
    tot = persist_total<LOCAL, KR>(P, RB, L);
    if (threadIdx.x == 0) {
      finalize(&k, FIN_CG_ITER, tot, 0.0);
      L.val = k.beta;
      L.stop = k.stop;
    }
    __syncthreads();
    if (L.stop != STOP_NONE) break;
    k.beta = L.val;
    par ^= 1;
  }
#pragma unroll
  for (int j = 0; j < KR; ++j)
    if (in[j]) x[row[j]] = xi[j];
  if (threadIdx.x == 0 && wg.w == 0) {  // what CG's updates change
    KS* o = ks + wg.z;
    o->gamma = k.gamma;
    o->pAp = k.pAp;
    o->alpha = k.alpha;
    o->beta = k.beta;
    o->rNorm = k.rNorm;
    o->pNorm2 = k.pNorm2;
    o->iter = k.iter;
    o->stop = k.stop;
  }
}

template <int G, int KR, class T>
__global__ void __launch_bounds__(kPersistNT)
    k_cg_persist(PersistK P, MatKT<T> A, const T* __restrict__ S, T* __restrict__ x,
                 const T* __restrict__ r, T* z, KS* ks) {
  __shared__ PersistLDS L;
  __shared__ T zl[KR * kPersistNT];
  const int4 wg = P.wg[blockIdx.x];
  if (threadIdx.x == 0) L.fail = 0;
  __syncthreads();
  if (P.cwg[wg.z].y == 1)
    cg_persist_case<true, G, KR, T>(P, wg, A, S, x, r, z, ks, L, zl);
  else
    cg_persist_case<false, G, KR, T>(P, wg, A, S, x, r, z, ks, L, zl);
}

}  // namespace xcal
