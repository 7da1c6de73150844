// CG with DILU on cone meshes in the split-preconditioned form: two sweeps per
// iteration and no matrix product.
//
// With A = L + Da + U (symmetric) and M = (D + L) D^-1 (D + U), CG on A with
// preconditioner M is CG on (D + L)^-1 A (D + U)^-1 with preconditioner D^-1
// (S. C. Eisenstat, SIAM J. Sci. Stat. Comput. 2, 1981), whose product needs
// one solve with each triangle, because
//   A t = (D + L) t + (D + U) t + (Da - 2 D) t.
// Per iteration, with rho = D (D + L)^-1 r and the direction ph = (D + U) p:
//   backward sweep   ph = rho + beta ph ;  t = (D + U)^-1 ph       (t = p)
//   forward sweep    w = (D + L)^-1 (ph + (Da - 2 D) t) ;  q = D (t + w) ; ph.q/D
//   vectors          x += alpha t ;  rho -= alpha q ;  rho.rho/D  (= r.M^-1 r)
// The iterates, alpha, beta and the stopping norm are the classical form's in
// exact arithmetic; its SpMV (110 MB counted of 374 MB per iteration on the
// 1M-cell box, 27 of 104 us) and its p pass are gone.  With y = D w the
// forward sweep is q = ph + (Da - D) t - sum a_ij w_j, w = q / D - t, so it
// carries no cancelling y.
//
// The sweeps walk the cones of sweep_cone.h (same blocks, positions and
// steps), with each row's loads packed: one 16-byte record (device row, six
// 16-bit cone positions), its entries in pairs (a step's rows are ordered by
// entry count, so pair j holds rows [0, pcnt[j])), and its scalars; a missing
// entry reads an LDS slot that holds 0.  A kernel takes as many pairs as the
// sweep's longest row: one on naturally numbered quadrilaterals, two on
// hexahedra, three on randomly numbered hexahedra.  With three pairs seven
// loads and about 60 issued instructions per row and step against 16 and 110,
// the dependencies read from LDS together instead of one after the other, and
// half the LDS per block.  Stores of rows that another block owns are dropped by the buffer
// store's range check instead of a branch, which would end the loop's block
// and with it exact waits.
//
// The vectors of a solve are in a row order of their own (split_rows): the
// rows of a block together, there by forward, then by backward level.  A
// backward step's rows then lie in one run per forward level inside 16 KB
// instead of in a line each all over the level-major device order, and no
// block's lines are another's.  The residual and 1/D are brought to it once a
// solve and the solution back; the matrix, SpMV and every other solve keep
// the device order (ordering that one by backward level cost SpMV 15%).
//
// Measured on one MI355X, per CG iteration: 1M-cell random box 104 us
// classical (35 + 32 + 27 + 8), 87 split in device order (48 backward, 27
// forward, 12 vectors), 66 in block order (28 + 26 + 11); 343k random box
// 66, 43 and 40; 152k random box in FP32 57, 33 and 31; 308k natural box
// (bands, two pairs) 500 and 346; 67.6k-cell cavity (bands, one pair) in FP64
// 505 and 413, in FP32 403 and 343 (three pairs 482 and 437).  Both sweeps are bound by the step-to-step chain and
// the 1.75 n rows of the cones; 4 steps in flight, 6 and 5 were no faster.
#pragma once

#include "sweep_cone.h"
#include "sweep_lean.h"

namespace xcal {

// Row blocks per workgroup of the streaming vector passes, and their grid.
constexpr int kPFinU = 4;
inline int pfin_grid(int nblk) { return ((nblk + kPFinU - 1) / kPFinU + 7) / 8 * 8; }

constexpr int kSplitGather = 2;  // steps ahead a row's gathers are issued

// Static tables of one direction (xcal_mesh::Cone).
struct SplitK {
  const int32_t* step;  // 8 words per step: first position, rows, poff[3], pcnt[3]
  const int32_t* blk;   // first step of each block (whole groups of kSplitDepth)
  const int32_t* base;  // first position of each block
  const int32_t* hnum;  // halo positions of each block
  const int4* rec;      // per position: row (~row: another block's, or halo), slots 0-1, 2-3, 4-5
  int32_t blk0;
};

// Stores v at element i of an array of n (dropped where `keep` is false).
template <class T>
struct OwnStore {
  __amdgpu_buffer_rsrc_t rs;
  __device__ inline OwnStore(T* p, int64_t n)
      : rs(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)(n * (int64_t)sizeof(T)), 0x00020000)) {}
  __device__ inline void put(bool keep, uint32_t i, T v) const {
    const int off = keep ? (int)(i * (uint32_t)sizeof(T)) : -1;
    if constexpr (sizeof(T) == 8) {
      typedef unsigned int u2 __attribute__((ext_vector_type(2)));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), rs, off, 0, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), rs, off, 0, 0);
    }
  }
};

// A row of a step: record (J = 1: its first half), entry pairs and scalars in
// flight.
template <class T, int NS, int J>
struct SplitRec {
  int row;
  uint32_t w[J];
  T a[2 * J], sc[NS], g0, g1;
  uint32_t lp;
  bool in;
};

// Walks block b's steps.  J entry pairs per row (the most that one has); NS
// scalars per position at `sc`; g0 and, with NG = 2,
// g1 are gathered from G0 and G1 by row; work(R, row, sum) returns the row's
// value.  Halo values come from `halo`.
template <int J, int NS, int NG, class T, class Work>
__device__ inline void split_walk(const SplitK& C, int b, const T* __restrict__ a,
                                  const T* __restrict__ sc, const T* __restrict__ halo,
                                  const T* __restrict__ G0, const T* __restrict__ G1, T* v,
                                  Work&& work) {
  using R = SplitRec<T, NS, J>;
  constexpr int P = kSplitDepth, Q = kSplitGather;
  const int s0 = C.blk[b], ns = C.blk[b + 1] - s0;
  const int32_t base = C.base[b], nh = C.hnum[b];
  for (int32_t p = threadIdx.x; p < nh; p += kConeBlock) v[p] = halo[~C.rec[base + p].x];
  if (threadIdx.x == 0) v[kConeMax] = T(0);
  __syncthreads();
  const auto* words = (const __attribute__((address_space(4))) int32_t*)(C.step + 8 * (int64_t)s0);
  struct Step {
    int32_t r0, cnt, po[J], pc[J];
  };
  auto step = [&](int l) {
    const int o = 8 * min(l, ns - 1);
    Step t;
    t.r0 = words[o];
    t.cnt = words[o + 1];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      t.po[j] = words[o + 2 + j];
      t.pc[j] = words[o + 5 + j];
    }
    return t;
  };
  typedef T V2 __attribute__((ext_vector_type(2)));
  auto fetch = [&](R& r, const Step& st) {
    const uint32_t q = min((uint32_t)threadIdx.x, (uint32_t)max(st.cnt, 1) - 1u);
    const uint32_t pos = (uint32_t)st.r0 + q;
    r.in = (int)threadIdx.x < st.cnt;
    if constexpr (J == 1) {
      const int2 u = lean_at<int2>(C.rec, 2 * pos);
      r.row = u.x;
      r.w[0] = (uint32_t)u.y;
    } else {
      const int4 u = lean_at<int4>(C.rec, pos);
      r.row = u.x;
      r.w[0] = (uint32_t)u.y;
      r.w[1] = (uint32_t)u.z;
      if constexpr (J == 3) r.w[2] = (uint32_t)u.w;
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const V2 p = lean_at<V2>(a, (int)q < st.pc[j] ? (uint32_t)st.po[j] + q : 0u);
      r.a[2 * j] = p.x;
      r.a[2 * j + 1] = p.y;
    }
    if constexpr (NS == 2) {
      const V2 s = lean_at<V2>(sc, pos);
      r.sc[0] = s.x;
      r.sc[1] = s.y;
    } else {
      r.sc[0] = lean_at<T>(sc, pos);
    }
    r.lp = pos - (uint32_t)base;
  };
  auto row = [](const R& r) { return (uint32_t)(r.row ^ (r.row >> 31)); };
  auto gather = [&](R& r) {
    opaque(r.row);
    r.g0 = lean_at<T>(G0, row(r));
    if constexpr (NG == 2) r.g1 = lean_at<T>(G1, row(r));
  };
  auto process = [&](R& r) {
    opaque(r.row);
#pragma unroll
    for (int j = 0; j < J; ++j) opaque(r.w[j]);
#pragma unroll
    for (int k = 0; k < 2 * J; ++k) opaque(r.a[k]);
#pragma unroll
    for (int k = 0; k < NS; ++k) opaque(r.sc[k]);
    opaque(r.g0);
    if constexpr (NG == 2) opaque(r.g1);
    T d[2 * J];
#pragma unroll
    for (int k = 0; k < 2 * J; ++k) d[k] = v[k & 1 ? r.w[k >> 1] >> 16 : r.w[k >> 1] & 0xffff];
    T sum = 0;
#pragma unroll
    for (int k = 0; k < 2 * J; ++k) sum = sum + r.a[k] * d[k];
    v[r.lp] = work(r, row(r), sum);
  };
  R buf[P];
#pragma unroll
  for (int s = 0; s < P; ++s) fetch(buf[s], step(s));
#pragma unroll
  for (int s = 0; s < Q; ++s) gather(buf[s]);
  Step nx = step(P);
  for (int l = 0; l < ns; l += P) {
#pragma unroll
    for (int s = 0; s < P; ++s) {
      gather(buf[(s + Q) % P]);
      process(buf[s]);
      fetch(buf[s], nx);
      nx = step(l + s + P + 1);
      __syncthreads();
    }
  }
}

// Backward sweep: the pending rho.rho/D finalize (kstate; every workgroup),
// then ph = rho + beta pold, t = (D + U)^-1 ph.
template <int J, class T>
__global__ void __launch_bounds__(kConeBlock)
    k_split_bwd(SplitK C, const T* __restrict__ a, const T* __restrict__ rD,
                const T* __restrict__ rho, const T* __restrict__ pold, T* __restrict__ ph, T* t,
                int64_t n, KStep K) {
  __shared__ T v[kConeMax + 1];
  __shared__ double lds[kConeBlock / 64];
  const KS k = kstate(K, lds);
  if (k.stop != STOP_NONE) return;  // uniform over the grid
  const T beta = (T)k.beta;
  const OwnStore<T> sp(ph, n), st(t, n);
  split_walk<J, 1, 2, T>(C, C.blk0 + (int)xcd_block(), a, rD, (const T*)t, rho, pold, v,
                   [&](const SplitRec<T, 1, J>& r, uint32_t i, T sum) {
                     const T p = r.g0 + beta * r.g1;
                     const T z = (p - sum) * r.sc[0];
                     const bool own = r.row >= 0;
                     sp.put(own, i, p);
                     st.put(own, i, z);
                     return z;
                   });
}

// Forward sweep: q = ph + (Da - D) t - sum a_ij w_j, w = q / D - t, and the
// partials of ph.q/D.  sc holds (1/D, Da - D) per position; w goes to `w`
// only where a later band reads it as its halo (w may be null otherwise).
// START: u = ph given alone; rho = y = u - sum a_ij w_j, w = y / D,
// partials of rho.rho/D.
template <bool START, int J, class T>
__global__ void __launch_bounds__(kConeBlock)
    k_split_fwd(SplitK C, const T* __restrict__ a, const T* __restrict__ sc,
                const T* __restrict__ ph, const T* __restrict__ t, T* __restrict__ q, T* w,
                int64_t n, double* partial, const KS* ks) {
  __shared__ T v[kConeMax + 1];
  if (stopped(ks)) return;
  const int b = C.blk0 + (int)xcd_block();
  const OwnStore<T> sq(q, n), sw(w, w ? n : 0);
  double s0 = 0.0;
  split_walk<J, 2, START ? 1 : 2, T>(C, b, a, sc, (const T*)w, ph, t, v,
                   [&](const SplitRec<T, 2, J>& r, uint32_t i, T sum) {
                     const bool own = r.row >= 0;
                     T wi, qi, qd;
                     if (START) {
                       qi = r.g0 - sum;
                       wi = qd = qi * r.sc[0];
                     } else {
                       qi = (r.g0 + r.sc[1] * r.g1) - sum;
                       qd = qi * r.sc[0];
                       wi = qd - r.g1;
                     }
                     sq.put(own, i, qi);
                     if (w) sw.put(own, i, wi);
                     const double d = START ? dd(qi, qd) : dd(r.g0, qd);
                     s0 = own && r.in ? s0 + d : s0;
                     return wi;
                   });
  store_partial<kConeBlock>(s0, 0.0, partial, b);
}

// Vectors: the pending ph.q/D finalize, then x += alpha t, rho -= alpha q and
// the partials of rho.rho/D; kPFinU blocks of consecutive rows a workgroup.
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_split_vec(int64_t n, const T* __restrict__ t, const T* __restrict__ q,
                const T* __restrict__ rD, T* __restrict__ x, T* __restrict__ rho, double* partial,
                KStep K) {
  __shared__ double lds[kBlock / 64];
  int64_t i[kPFinU];
  T xv[kPFinU], tv[kPFinU], rv[kPFinU], qv[kPFinU], dv[kPFinU];
#pragma unroll
  for (int u = 0; u < kPFinU; ++u) {
    const int64_t r = (xcd_block() * kPFinU + u) * kBlock + threadIdx.x;
    i[u] = r < n ? r : -1;
  }
#pragma unroll
  for (int u = 0; u < kPFinU; ++u) {
    const int64_t ii = i[u] >= 0 ? i[u] : 0;
    xv[u] = x[ii];
    tv[u] = t[ii];
    rv[u] = rho[ii];
    qv[u] = q[ii];
    dv[u] = rD[ii];
  }
  const KS k = kstate(K, lds);
  if (k.stop != STOP_NONE) return;  // uniform over the grid
  const T al = (T)k.alpha;
  double s0 = 0.0;
#pragma unroll
  for (int u = 0; u < kPFinU; ++u)
    if (i[u] >= 0) {
      const T r = rv[u] + (-al) * qv[u];
      x[i[u]] = xv[u] + al * tv[u];
      rho[i[u]] = r;
      s0 += dd(r, r * dv[u]);
    }
  store_partial<kBlock>(s0, 0.0, partial, blockIdx.x);
}

// Host: calls f(J) with the entry pairs of a cone's rows.
template <class F>
inline void with_split_pairs(const xcal_mesh::Cone& c, F&& f) {
  if (c.wk <= 2) f(std::integral_constant<int, 1>{});
  else if (c.wk <= 4) f(std::integral_constant<int, 2>{});
  else f(std::integral_constant<int, 3>{});
}
// Host: the kernel view of one direction's tables for the band from blk0.
inline SplitK split_k(const xcal_mesh::Cone& c, int32_t blk0) {
  return SplitK{c.step2.p, c.blk2.p, c.base.p, c.hnum.p, c.rec.p, blk0};
}

}  // namespace xcal
