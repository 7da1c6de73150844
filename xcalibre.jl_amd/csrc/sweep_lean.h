// One-workgroup DILU sweeps over every level of a mesh (or of a batch case),
// in one launch: the lean form of the pipelined sweeps (sweep_pipe.h).
//
// A sweep over a mesher's natural numbering is a chain of some 100 to 2000
// short levels, and a level costs what one wavefront issues for it: the
// pipelined body spends about 88 instructions per row and level, half of them
// on addresses (the packed factors' base, width and stride change from level
// to level) and masks.  Here a row is found by its position alone:
//  * entries are stored by position, two per 16-byte load (and a third in an
//    array of its own), so one shifted position addresses every load;
//  * dependencies are 16-bit slots of the LDS ring, packed in one word per
//    row; a missing entry reads a slot that holds zeros, so nothing is masked;
//  * the ring keeps a row's value and its 1/D (forward), so an entry loads
//    neither;
//  * levels are cut into steps of at most one row per thread, padded to whole
//    groups of P steps, so the loop has no remainder (a padding step works the
//    last row again; it was fetched before that row's own step, so an update
//    in place reads what the first one read).
// Loads are issued P steps ahead; `opaque` keeps the compiler from moving
// work on freshly loaded values across steps, where it would wait for them.
//
// 256 threads.  Where every level has at most 256 rows the row-to-thread map
// is the pipelined sweeps', so the dot products match theirs; where some have
// more, k_plan_dots sums them in the launch form's order.  The rows' own sums
// keep the reference's column order, so the sweep equals the sequential loops
// (preconditioners_1_DILU.jl:43-114) bit for bit.
//
// Measured per forward / backward sweep on one MI355X, pipelined or launch
// form then lean: 1600-cell cavity (79 levels) 25 / 25 to 15 / 17 us; 50k-cell
// step (580 levels) 283 / 283 to 94 / 117 us; 256 cavities (511 levels) 162 /
// 159 to 98 / 118 us; 44k-cell natural box (105 levels, 75 launches) about
// 250 / 280 to 50 / 53 us.  About 41 instructions per step and wavefront; a
// step is bound by their issue and the LDS round trip of its dependencies
// (512 and 1024 threads per workgroup measured 60 and 83 us on that box, and
// skipping the barrier between steps of one level 58 us: the branch splits
// the loop's block).
#pragma once

#include <type_traits>

#include "solver_common.h"

namespace xcal {

// Hides a prefetched value's origin until it is used.
template <class V>
__device__ inline void opaque(V& v) {
  asm volatile("" : "+v"(v));
}

// One sweep direction (device arrays of xcal_mesh::Lean).  W entries per row.
struct LeanK {
  const int2* steps;      // first position, rows (0: a padding step); groups of kLeanDepth
  const int32_t* cstep;   // first step of each case (ncase + 1)
  const uint32_t* idx;    // W = 2: one word of two slots per position; W = 3: two words
  int64_t n;              // positions (third entries follow the 2 n pairs)
};

template <class T>
struct alignas(2 * sizeof(T)) LeanVal {  // a row's value and 1/D
  T v, rd;
};

template <int W>
struct LeanIdx {
  uint32_t w[W == 2 ? 1 : 2];
  __device__ inline uint32_t slot(int k) const { return k & 1 ? w[k >> 1] >> 16 : w[k >> 1] & 0xffff; }
};

// A row's static loads: its slots and entries.
template <class T, int W>
struct LeanRow {
  LeanIdx<W> ix;
  T a[W];
};
// Element i of an array below 4 GiB: a 32-bit byte offset from a uniform base
// is one shift, shared by every array of that element size.
template <class V>
__device__ inline V lean_at(const void* base, uint32_t i) {
  return *reinterpret_cast<const V*>(static_cast<const char*>(base) + i * (uint32_t)sizeof(V));
}
template <class V>
__device__ inline void lean_put(V* base, uint32_t i, V v) {
  *reinterpret_cast<V*>(reinterpret_cast<char*>(base) + i * (uint32_t)sizeof(V)) = v;
}
template <class T, int W>
__device__ inline void lean_row(const LeanK& K, const T* __restrict__ a, uint32_t pos,
                                LeanRow<T, W>& R) {
  if constexpr (W == 2) {
    R.ix.w[0] = lean_at<uint32_t>(K.idx, pos);
  } else {
    const uint2 u = lean_at<uint2>(K.idx, pos);
    R.ix.w[0] = u.x;
    R.ix.w[1] = u.y;
  }
  typedef T V2 __attribute__((ext_vector_type(2)));
  const V2 p = lean_at<V2>(a, pos);
  R.a[0] = p.x;
  R.a[1] = p.y;
  if constexpr (W == 3) R.a[2] = lean_at<T>(a + 2 * K.n, pos);
}
template <class T, int W>
__device__ inline void lean_opaque(LeanRow<T, W>& R) {
  opaque(R.ix.w[0]);
  if constexpr (W == 3) opaque(R.ix.w[1]);
#pragma unroll
  for (int k = 0; k < W; ++k) opaque(R.a[k]);
}

// The step loop: fetch(R, p0, cnt) issues a step's loads, gather(R) its
// dependent loads Q steps before it is worked, process(R) works it.
// The table is read through the scalar cache, one step before it is used.
template <int P, int Q, class Rec, class Fetch, class Gather, class Process>
__device__ inline void lean_steps(const int2* table, int ns, Fetch&& fetch, Gather&& gather,
                                  Process&& process) {
  const auto* words = (const __attribute__((address_space(4))) int32_t*)table;
  auto step = [&](int l) {
    l = min(l, ns - 1);
    return int2{words[2 * l], words[2 * l + 1]};
  };
  Rec buf[P];
#pragma unroll
  for (int s = 0; s < P; ++s) fetch(buf[s], step(s));
#pragma unroll
  for (int s = 0; s < Q; ++s) gather(buf[s]);
  int2 nx = step(P);
  for (int l = 0; l < ns; l += P) {
#pragma unroll
    for (int s = 0; s < P; ++s) {
      if (Q > 0) gather(buf[(s + Q) % P]);
      process(buf[s]);
      fetch(buf[s], nx);  // step l + s + P (the last one again past the end)
      nx = step(l + s + P + 1);
      __syncthreads();
    }
  }
}

template <class T, int W>
struct LeanF {
  LeanRow<T, W> r;
  T u, rd;
  int32_t pb;
  uint32_t slot;
};

// y = (I + L D^-1)^-1 u over case positions; y to Yb in backward order.
template <class T, int W, int RING, int P>
__device__ inline void fwd_lean(const LeanK& K, int c, const T* __restrict__ a,
                                const T* __restrict__ rD, const T* __restrict__ u,
                                const int32_t* __restrict__ posb, T* __restrict__ Yb,
                                LeanVal<T>* ring) {
  const int s0 = K.cstep[c], ns = K.cstep[c + 1] - s0;
  if (threadIdx.x == 0) ring[RING] = LeanVal<T>{T(0), T(0)};
  __syncthreads();
  using R = LeanF<T, W>;
  auto fetch = [&](R& r, int2 st) {
    const uint32_t pos = (uint32_t)st.x + min((uint32_t)threadIdx.x, (uint32_t)max(st.y, 1) - 1u);
    lean_row<T, W>(K, a, pos, r.r);
    r.u = lean_at<T>(u, pos);
    r.rd = lean_at<T>(rD, pos);
    r.pb = lean_at<int32_t>(posb, pos);
    r.slot = pos & (RING - 1);
  };
  auto process = [&](R& r) {
    lean_opaque(r.r);
    opaque(r.u);
    opaque(r.rd);
    opaque(r.pb);
    LeanVal<T> d[W];
#pragma unroll
    for (int k = 0; k < W; ++k) d[k] = ring[r.r.ix.slot(k)];
    T sum = 0;
#pragma unroll
    for (int k = 0; k < W; ++k) sum = sum + (r.r.a[k] * d[k].v) * d[k].rd;
    const T y = r.u - sum;
    ring[r.slot] = LeanVal<T>{y, r.rd};
    lean_put(Yb, (uint32_t)r.pb, y);
  };
  lean_steps<P, 0, R>(K.steps + s0, ns, fetch, [](R&) {}, process);
}

template <class T, int W>
struct LeanB {
  LeanRow<T, W> r;
  T yb, d, dv;
  int32_t i;
  uint32_t slot;
  bool own;
};

// z = (D + U)^-1 y in backward order, with the dot products of bwd_row.
template <int DOT, class T, int W, int RING, int P>
__device__ inline void bwd_lean(const LeanK& K, int c, const T* __restrict__ a,
                                const BwdK<T>& Bk, T* ring, double& s0, double& s1) {
  const int b0 = K.cstep[c], ns = K.cstep[c + 1] - b0;
  if (threadIdx.x == 0) ring[RING] = T(0);
  __syncthreads();
  using R = LeanB<T, W>;
  auto fetch = [&](R& r, int2 st) {
    r.own = (int)threadIdx.x < st.y;
    const uint32_t pos = (uint32_t)st.x + min((uint32_t)threadIdx.x, (uint32_t)max(st.y, 1) - 1u);
    lean_row<T, W>(K, a, pos, r.r);
    r.yb = lean_at<T>(Bk.Yb, pos);
    r.d = lean_at<T>(Bk.Db, pos);
    r.i = lean_at<int32_t>(Bk.rows, pos);
    r.slot = pos & (RING - 1);
  };
  auto gather = [&](R& r) {
    opaque(r.i);
    if (DOT != 0) r.dv = lean_at<T>(Bk.dv, (uint32_t)r.i);
  };
  auto process = [&](R& r) {
    lean_opaque(r.r);
    opaque(r.yb);
    opaque(r.d);
    if (DOT != 0) opaque(r.dv);
    T d[W];
#pragma unroll
    for (int k = 0; k < W; ++k) d[k] = ring[r.r.ix.slot(k)];
    T sum = 0;
#pragma unroll
    for (int k = 0; k < W; ++k) sum = sum + r.r.a[k] * d[k];
    const T zi = (r.yb - sum) / r.d;
    ring[r.slot] = zi;
    lean_put(Bk.Z, (uint32_t)r.i, zi);
    const T dvi = DOT != 0 ? r.dv : T(0);
    double a0 = 0.0, a1 = 0.0;
    if (DOT == 1 || DOT == 2) a0 = dd(dvi, zi);
    if (DOT == 3) { a0 = dd(zi, dvi); a1 = dd(zi, zi); }
    if (DOT == 4) { a0 = dd(zi, zi); a1 = dd(dvi, zi); }
    s0 = r.own ? s0 + a0 : s0;
    s1 = r.own ? s1 + a1 : s1;
  };
  lean_steps<P, (P > 2 ? P / 2 : 1), R>(K.steps + b0, ns, fetch, gather, process);
}

template <int W>
struct LeanD {
  LeanRow<double, W> r;
  double d0;
  uint32_t pos;
};

// update_dilu_diagonal!: D_j = a_jj, then D_j -= (a_ij a_ji) / D_i in column
// order; prod holds the products in the entries' layout (0 where missing,
// whose slot holds 1).
template <int W, int RING, int P>
__device__ inline void diag_lean(const LeanK& K, int c, const double* __restrict__ prod, double* D,
                                 double* ring) {
  const int s0 = K.cstep[c], ns = K.cstep[c + 1] - s0;
  if (threadIdx.x == 0) ring[RING] = 1.0;
  __syncthreads();
  using R = LeanD<W>;
  auto fetch = [&](R& r, int2 st) {
    r.pos = (uint32_t)st.x + min((uint32_t)threadIdx.x, (uint32_t)max(st.y, 1) - 1u);
    lean_row<double, W>(K, prod, r.pos, r.r);
    r.d0 = lean_at<double>(D, r.pos);
  };
  auto process = [&](R& r) {
    lean_opaque(r.r);
    opaque(r.d0);
    double Dj = r.d0;
#pragma unroll
    for (int k = 0; k < W; ++k) Dj = Dj - r.r.a[k] / ring[r.r.ix.slot(k)];
    ring[r.pos & (RING - 1)] = Dj;
    lean_put(D, r.pos, Dj);
  };
  lean_steps<P, 0, R>(K.steps + s0, ns, fetch, [](R&) {}, process);
}

// One partial pair per slot of the launch form's backward sweep, from the
// finished z: slot t covers a level launch's workgroup (kind 0: first
// position, rows, workgroup) or a run of small levels (kind 1: first and last
// level), each thread adding the rows it has there in the same order.
template <int DOT, class T>
__global__ void __launch_bounds__(kBlock)
    k_plan_dots(const int4* __restrict__ tab, const int32_t* __restrict__ rows,
                const int32_t* __restrict__ lev_ptr, const T* __restrict__ dv,
                const T* __restrict__ Z, double* partial, const KS* ks) {
  if (ks && stopped(ks)) return;
  const int4 s = tab[blockIdx.x];
  double s0 = 0.0, s1 = 0.0;
  auto add = [&](T dvi, T zi) {
    if (DOT == 1 || DOT == 2) s0 += dd(dvi, zi);
    if (DOT == 3) { s0 += dd(zi, dvi); s1 += dd(zi, zi); }
    if (DOT == 4) { s0 += dd(zi, zi); s1 += dd(dvi, zi); }
  };
  if (s.x == 0) {
    const int x = s.w & 7, l = s.w >> 3;
    const int64_t c0 = (int64_t)s.z * x / 8 / 64 * 64;
    const int64_t end = x == 7 ? s.z : (int64_t)s.z * (x + 1) / 8 / 64 * 64;
    const int64_t t = c0 + (int64_t)l * kBlock + threadIdx.x;
    if (t < end) {
      const int32_t i = rows[s.y + t];
      add(dv[i], Z[i]);
    }
  } else {
    constexpr int U = 8;
    for (int l0 = s.y; l0 < s.z; l0 += U) {
      bool in[U];
      T d[U], z[U];
      int32_t i[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int l = min(l0 + u, s.z - 1);
        const int32_t p = lev_ptr[l], cnt = lev_ptr[l + 1] - p;
        in[u] = l0 + u < s.z && (int)threadIdx.x < cnt;
        i[u] = rows[p + min((int)threadIdx.x, cnt - 1)];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        d[u] = dv[i[u]];
        z[u] = Z[i[u]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (in[u]) add(d[u], z[u]);
    }
  }
  store_partial<kBlock>(s0, s1, partial, blockIdx.x);
}

template <class T, int W, int RING>
__global__ void __launch_bounds__(kLeanBlock)
    k_fwd_lean(LeanK K, const T* __restrict__ a, const T* __restrict__ rD,
               const T* __restrict__ u, const int32_t* __restrict__ posb, T* __restrict__ Yb,
               const KS* ks) {
  __shared__ LeanVal<T> ring[RING + 1];
  if (ks && stopped(ks + blockIdx.x)) return;  // uniform over the workgroup
  fwd_lean<T, W, RING, kLeanDepth>(K, blockIdx.x, a, rD, u, posb, Yb, ring);
}
template <int DOT, class T, int W, int RING>
__global__ void __launch_bounds__(kLeanBlock)
    k_bwd_lean(LeanK K, const T* __restrict__ a, BwdK<T> B, const KS* ks) {
  __shared__ T ring[RING + 1];
  if (ks && stopped(ks + blockIdx.x)) return;
  double s0 = 0.0, s1 = 0.0;
  bwd_lean<DOT, T, W, RING, kLeanDepth>(K, blockIdx.x, a, B, ring, s0, s1);
  if (DOT != 0) store_partial<kLeanBlock>(s0, s1, B.partial, blockIdx.x);
}
template <int W, int RING>
__global__ void __launch_bounds__(kLeanBlock)
    k_diag_lean(LeanK K, const double* __restrict__ prod, double* D) {
  __shared__ double ring[RING + 1];
  diag_lean<W, RING, kLeanDepth>(K, blockIdx.x, prod, D, ring);
}

// Host: calls f(W, RING) with the compile-time form of a lean sweep.
template <class F>
inline void with_lean_form(const xcal_mesh::Lean& L, F&& f) {
  auto go = [&](auto W) {
    if (L.ring == 4096) f(W, std::integral_constant<int, 4096>{});
    else f(W, std::integral_constant<int, 8192>{});
  };
  if (L.w == 2) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 3>{});
}
inline LeanK lean_k(const xcal_mesh* m, const xcal_mesh::Lean& L) {
  return LeanK{L.steps.p, L.cstep.p, L.idx.p, m->n};
}

}  // namespace xcal
