// Resident CG (persist.h): workgroup plans, admission and launch.
#include <cstdlib>
#include <mutex>

#include "persist.h"

namespace xcal {

// Rows a resident solve may have: at two rows per thread on every one of 256
// compute units, and the 1024 slots of kPersistSlots for one case.  It gains up
// to there (262 144 rows 19.7 to 9.1 us per iteration), so the line is what
// fits.
constexpr int64_t kPersistRows = 1 << 18;
// One row per thread up to this many workgroups, two above: fewer lines to
// read per meeting against more work between them.  Per iteration of a single
// mesh, one row then two: 79 and 40 workgroups 5.83 and 5.99 us, 104 and 52
// 6.15 and 6.07, 128 and 64 6.38 and 6.10, 188 and 94 7.45 and 6.68, 254 and
// 127 7.80 and 7.22.
constexpr int kPersistWide = 64;

struct PersistPlan {
  bool ok = false;
  int nwg = 0, kr = 1;
  int64_t words = 0;
  DBuf<int4> wg, seg, cwg;
  DBuf<int2> grp, slotA, slotB;
};

template <class V>
static void up(DBuf<V>& d, const std::vector<V>& v) {
  d.alloc((int64_t)v.size());
  if (!v.empty())
    XCAL_HIP(hipMemcpy(d.p, v.data(), sizeof(V) * v.size(), hipMemcpyHostToDevice));
}

static int compute_units(int device) {
  int cu = 0;
  XCAL_HIP(hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, device));
  return cu;
}

// Room for resident workgroups on each device (resident.h).  A launch is
// admitted only while all in flight fit the device one per compute unit, so
// admitted launches can never wait for each other.  The file that processes
// share is named by the device's PCI address.
static ResidentRoom* resident_room(int device) {
  static ResidentRoom rooms[64];
  static std::once_flag named[64];
  if (device < 0 || device >= 64) return nullptr;
  std::call_once(named[device], [&] {
    char id[64] = {};
    if (hipDeviceGetPCIBusId(id, sizeof id, device) == hipSuccess && id[0])
      rooms[device].share(std::string("/dev/shm/xcal-resident-") + id);
  });
  return &rooms[device];
}

// Groups of 64 rows, the slots both reductions add them in, and the
// workgroups of each case.  A slot is a 256-row block of the launch chain:
// its row blocks in dispatch order (xblk) for p.q and xcd_row's blocks for
// r.z on a single mesh, the case's blocks for both on a batch mesh.  Not
// built (ok stays false) where a slot does not start on a group, a row is
// wider than row_sum's group, or a case has too many slots.
static std::shared_ptr<PersistPlan> make_plan(const xcal_mesh* m) {
  auto P = std::make_shared<PersistPlan>();
  if (!m->persist_on || m->n > kPersistRows || m->roww > 8) return P;
  std::vector<int2> grp, sa, sb, cgrp;
  std::vector<int4> seg, wg, cwg;
  if (m->batch) {
    const size_t nb = (size_t)m->nblk;
    std::vector<int32_t> r0(nb), r1(nb), cb((size_t)m->ncase + 1);
    XCAL_HIP(hipMemcpy(r0.data(), m->blk_row0.p, 4 * nb, hipMemcpyDeviceToHost));
    XCAL_HIP(hipMemcpy(r1.data(), m->blk_row1.p, 4 * nb, hipMemcpyDeviceToHost));
    XCAL_HIP(hipMemcpy(cb.data(), m->case_blk_d.p, 4 * cb.size(), hipMemcpyDeviceToHost));
    for (int k = 0; k < m->ncase; ++k) {
      const int g0 = (int)grp.size();
      for (int32_t b = cb[k]; b < cb[k + 1]; ++b) {
        const int first = (int)grp.size();
        for (int32_t r = r0[b]; r < r1[b]; r += 64)
          grp.push_back(int2{r, std::min(64, r1[b] - r)});
        sa.push_back(int2{first - g0, (int)grp.size() - first});
      }
      if (cb[k + 1] - cb[k] > kPersistSlots) return P;
      seg.push_back(int4{cb[k], cb[k + 1], cb[k], cb[k + 1]});
      cgrp.push_back(int2{g0, (int)grp.size()});
    }
    sb = sa;
  } else {
    const int64_t n = m->n;
    for (int64_t r = 0; r < n; r += 64) grp.push_back(int2{(int)r, (int)std::min<int64_t>(64, n - r)});
    for (int b = 0; b < m->nxblk; ++b) {
      const int32_t a = m->xblk[2 * b], e = m->xblk[2 * b + 1];
      if (a < e && (a % 64 != 0 || (e % 64 != 0 && e != n) || e - a > kBlock)) return P;
      sa.push_back(a < e ? int2{a / 64, (e - a + 63) / 64} : int2{0, 0});
    }
    const int64_t gr = grid_for(n), q = gr >> 3, rem = gr & 7;
    for (int64_t b = 0; b < gr; ++b) {  // xcd_block
      const int64_t xx = b & 7, blk = xx * q + std::min<int64_t>(xx, rem) + (b >> 3);
      sb.push_back(int2{(int)(4 * blk), (int)std::min<int64_t>(4, (int64_t)grp.size() - 4 * blk)});
    }
    if ((int)sa.size() > kPersistSlots || (int)sb.size() > kPersistSlots) return P;
    seg.push_back(int4{0, (int)sa.size(), 0, (int)sb.size()});
    cgrp.push_back(int2{0, (int)grp.size()});
  }
  // one row per thread while that many workgroups fit, two otherwise
  const int cap = compute_units(m->ctx->device);
  auto count = [&](int kr) {
    int64_t w = 0;
    for (const int2& c : cgrp) w += (c.y - c.x + kPersistWaves * kr - 1) / (kPersistWaves * kr);
    return w;
  };
  P->kr = count(1) <= std::min(cap, kPersistWide) ? 1 : 2;
  if (count(P->kr) > cap) return P;
  for (int k = 0; k < (int)cgrp.size(); ++k) {
    const int w0 = (int)wg.size();
    for (int g = cgrp[k].x; g < cgrp[k].y; g += kPersistWaves * P->kr)
      wg.push_back(int4{g, std::min(g + kPersistWaves * P->kr, cgrp[k].y), k, (int)wg.size() - w0});
    if ((int)wg.size() - w0 > kPersistWGs) return P;
    cwg.push_back(int4{w0, (int)wg.size() - w0, grp[cgrp[k].x].x, 0});
  }
  P->nwg = (int)wg.size();
  P->words = (int64_t)P->nwg * kPersistLine;
  up(P->wg, wg);
  up(P->seg, seg);
  up(P->grp, grp);
  up(P->slotA, sa);
  up(P->slotB, sb);
  up(P->cwg, cwg);
  P->ok = P->nwg > 0;
  return P;
}

static __global__ void __launch_bounds__(kBlock)
    k_persist_reset(unsigned long long* area, int64_t n, int* abort) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) area[i] = kUnset;
  if (i == 0) *abort = 0;
}

// Launches the CG iterations of every case from the state `ks` and the start
// vectors r and z = S r, to each case's stop; x receives the corrections of
// the cases that ran.  False, with nothing launched, where the mesh has no
// plan or the device no room.  The caller reads the states: where a case is
// not resident_done(), waits were given up, and persist_failed() keeps the
// mesh on the launch chain from then on.
template <class T>
bool persist_cg(xcal_eqn* e, const MatKT<T>& A, const T* S, T* x, const T* r, T* z, KS* ks,
                ResidentLease& lease) {
  const xcal_mesh* m = e->mesh;
  if (!m->persist_on || m->ctx->prof_on[0]) return false;
  if (!m->persist) m->persist = make_plan(m);
  const PersistPlan& P = *m->persist;
  if (!P.ok) return false;
  ResidentRoom* room = resident_room(m->ctx->device);
  if (!room || !lease.acquire(*room, P.nwg, compute_units(m->ctx->device))) {
    m->persist_full++;
    return false;
  }
  if (e->parea.n < 4 * P.words + 1) e->parea.alloc(4 * P.words + 1);
  PersistK K;
  K.wg = P.wg.p;
  K.grp = P.grp.p;
  K.slotA = P.slotA.p;
  K.slotB = P.slotB.p;
  K.seg = P.seg.p;
  K.cwg = P.cwg.p;
  K.batch = m->batch ? 1 : 0;
  K.words = P.words;
  K.area = e->parea.p;
  K.abort = (int*)(e->parea.p + 4 * P.words);
  K.limit = m->persist_ticks;
  hipStream_t s = m->ctx->stream;
  hipLaunchKernelGGL(k_persist_reset, dim3(grid_for(4 * P.words)), dim3(kBlock), 0, s, K.area,
                     4 * P.words, K.abort);
  with_row_group(A.rw, [&](auto Gc) {
    constexpr int G = decltype(Gc)::value;
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(P.nwg), dim3(kPersistNT), 0, s, K, A, S, x, r, z, ks);
    };
    if (P.kr == 1) go(k_cg_persist<G, 1, T>);
    else go(k_cg_persist<G, 2, T>);
  });
  XCAL_HIP(hipGetLastError());
  m->persist_runs++;
  return true;
}
template bool persist_cg<double>(xcal_eqn*, const MatKT<double>&, const double*, double*,
                                 const double*, double*, KS*, ResidentLease&);
template bool persist_cg<float>(xcal_eqn*, const MatKT<float>&, const float*, float*, const float*,
                                float*, KS*, ResidentLease&);

void persist_failed(const xcal_mesh* m) {
  m->persist_on = false;
  m->persist_left++;
}
int persist_workgroups(const xcal_mesh* m) {
  return m->persist && m->persist->ok ? m->persist->nwg : 0;
}

// Knobs, read when the mesh is created: XCAL_NO_PERSIST=1 keeps the launch
// chain (as XCAL_NO_FUSE=1 does), XCAL_PERSIST_WAIT_US bounds each wait.
void persist_configure(xcal_mesh* m) {
  const char* off = std::getenv("XCAL_NO_PERSIST");
  m->persist_on = m->fuse && !(off && *off == '1');
  if (const char* w = std::getenv("XCAL_PERSIST_WAIT_US"))
    m->persist_ticks = 100ll * std::max(0, std::atoi(w));
}

}  // namespace xcal
