// Helmholtz particle FMM driver: host octree (the same d3tstrcr tree as the
// Laplace path) -> per-level orders and translation tables -> one upload ->
// the eight steps of hfmm3dparttargmain (src/hfmm3dpart.f:545-1086) and
// hfmm3d_list2 (src/hfmm3drouts.f:153-564) as HIP kernels on one stream ->
// scatter back to the caller's order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <type_traits>
#include <vector>

#include "fmm3d_internal.hpp"
#include "helm_kernels.hip"
#include "helm_tables.hpp"
#include "htria_kernels.hpp"
#include "tria_rules.hpp"
#include "tree_gpu.hpp"
#include "octree.hpp"
#include "plan.hpp"
#include "runtime.hpp"

namespace fmm3d {

namespace {

// The tables in this context's arena: the geometry (rotations, phases, factors)
// of one order, the Gaunt integrals, and the orders and coaxial operators of
// one wavenumber, root box, depth and tolerance.  Each part is replaced when a
// call needs another.
struct HelmCache {
  HelmHostTables H;
  bool valid = false;                        // the operators on the device are H's
  std::shared_ptr<const HostTables> geo;     // the geometry on the device
  std::shared_ptr<const Gaunt> gaunt;        // the integrals on the device
  size_t gI = 0, gD = 0, gL = 0;             // geometry sizes
  size_t o_offrot = 0, o_offdist = 0, o_octrot = 0;
  size_t o_fac = 0, o_offph = 0, o_octph = 0, o_rot = 0, o_rotsd = 0;
  size_t o_rotoff = 0;
  size_t cI = 0, cD = 0, cL = 0, cZ = 0;     // per-call sizes
  size_t o_plev = 0, o_ptrunc = 0, o_sclev = 0, o_coax = 0, o_ztoff = 0, o_zt = 0;
  int m2m_base = 0, l2l_base = 0;
  bool grouped_m2l = false;   // every list-2 order fits its table's tiles
};

template <typename V>
size_t put_aligned(std::vector<V>& to, const std::vector<V>& v, size_t a) {
  const size_t o = to.size();
  to.insert(to.end(), v.begin(), v.end());
  while (to.size() % a) to.push_back(V(0));
  return o;
}

void helm_upload_geometry(Context& ctx, HelmCache& c, const std::shared_ptr<const HostTables>& g) {
  c.geo.reset();
  std::vector<int> I;
  std::vector<double> D;
  std::vector<long> L;
  c.o_offrot = put_aligned(I, g->off_rot, 16);
  c.o_offdist = put_aligned(I, g->off_dist, 16);
  c.o_octrot = put_aligned(I, g->oct_rot, 16);
  c.o_fac = put_aligned(D, g->fac, 8);
  c.o_offph = put_aligned(D, g->off_phase, 8);
  c.o_octph = put_aligned(D, g->oct_phase, 8);
  c.o_rot = put_aligned(D, g->rot, 8);
  c.o_rotsd = put_aligned(D, g->rot_sd, 8);
  c.o_rotoff = put_aligned(L, g->rot_off, 1);
  c.gI = I.size(); c.gD = D.size(); c.gL = L.size();
  void* di = ctx.arena.get("hgeo_i", I.size() * sizeof(int));
  void* dd = ctx.arena.get("hgeo_d", D.size() * sizeof(double));
  void* dl = ctx.arena.get("hgeo_l", L.size() * sizeof(long));
  FMM_HIP(hipMemcpyAsync(di, I.data(), I.size() * sizeof(int), hipMemcpyHostToDevice, ctx.stream));
  FMM_HIP(hipMemcpyAsync(dd, D.data(), D.size() * sizeof(double), hipMemcpyHostToDevice, ctx.stream));
  FMM_HIP(hipMemcpyAsync(dl, L.data(), L.size() * sizeof(long), hipMemcpyHostToDevice, ctx.stream));
  FMM_HIP(hipStreamSynchronize(ctx.stream));
  c.geo = g;
}

void helm_upload_gaunt(Context& ctx, HelmCache& c, const std::shared_ptr<const Gaunt>& g) {
  c.gaunt.reset();
  void* dg = ctx.arena.get("hgaunt_g", g->g.size() * sizeof(double));
  void* dof = ctx.arena.get("hgaunt_o", g->off.size() * sizeof(long));
  FMM_HIP(hipMemcpyAsync(dg, g->g.data(), g->g.size() * sizeof(double), hipMemcpyHostToDevice, ctx.stream));
  FMM_HIP(hipMemcpyAsync(dof, g->off.data(), g->off.size() * sizeof(long), hipMemcpyHostToDevice, ctx.stream));
  FMM_HIP(hipStreamSynchronize(ctx.stream));
  c.gaunt = g;
}

// The tables of the plan H on the device: queues on ctx.stream what this
// context does not hold yet.  H's orders have been checked against what the
// kernels take: a call that is refused queues nothing and keeps the tables of
// the call before it.
HelmCache& helm_upload_tables(Context& ctx, HelmCache& c, HelmHostTables&& plan) {
  c.valid = false;
  c.H = std::move(plan);
  const HelmHostTables& H = c.H;
  if (c.geo != H.geo) helm_upload_geometry(ctx, c, H.geo);
  const auto gaunt = gaunt_for(H.pmax);
  if (c.gaunt != gaunt) helm_upload_gaunt(ctx, c, gaunt);
  const int nd = H.geo->ndist, P1 = H.pmax + 1, nlev = H.nlev;
  std::vector<int> I;
  std::vector<double> D;
  std::vector<long> L;
  c.o_plev = put_aligned(I, H.plev, 16);
  c.o_ptrunc = put_aligned(I, H.ptrunc, 16);
  c.o_sclev = put_aligned(D, H.sclev, 8);
  const size_t o_series = put_aligned(D, H.series, 8);
  c.o_coax = 0;
  auto put_desc = [&](const CoaxDesc& d) { L.push_back(d.base); L.push_back(d.pin); L.push_back(d.pout); };
  for (const auto& d : H.m2l) put_desc(d);
  c.m2m_base = (nlev + 1) * nd;
  for (const auto& d : H.m2m) put_desc(d);
  c.l2l_base = c.m2m_base + nlev + 1;
  for (const auto& d : H.l2l) put_desc(d);
  // grouped M2L: each M2L operator also as complex 4x4 tiles per order am,
  // [row block of n - am][column block of l - am], 16 real parts then 16
  // imaginary parts of [row][column]; every list-2 order must lie within its
  // table's tiles
  std::vector<long> zt_off;
  const long nt = coax_tile_offsets(H, zt_off);
  int mmax = 0;
  for (const CoaxJob& J : H.jobs) mmax = std::max(mmax, std::min(J.pin, J.pout));
  bool ok = true;
  for (int l = 2; l <= nlev && ok; l++)
    for (int code = 0; code < 343 && ok; code++) {
      const int pt = H.ptrunc[(size_t)l * 343 + code];
      if (pt <= 0) continue;
      const CoaxDesc& d = H.m2l[(size_t)l * nd + H.geo->off_dist[code]];
      ok = d.pin == d.pout && pt <= d.pout;
    }
  c.grouped_m2l = ok;
  c.o_ztoff = put_aligned(L, zt_off, 1);
  c.o_zt = (2 * (size_t)H.nz + 7) / 8 * 8;
  c.cI = I.size(); c.cD = D.size(); c.cL = L.size();
  c.cZ = c.o_zt + (size_t)nt;
  // small enough to go through one pinned buffer (the call before this one on
  // the context has finished with it, whichever way it ended: QueuedWork)
  const size_t bI = I.size() * sizeof(int), bD = D.size() * sizeof(double), bL = L.size() * sizeof(long),
               bJ = H.jobs.size() * sizeof(CoaxJob);
  char* h = (char*)ctx.arena.get_host("htab_h", bD + bL + bJ + bI);
  std::memcpy(h, D.data(), bD);
  std::memcpy(h + bD, L.data(), bL);
  std::memcpy(h + bD + bL, H.jobs.data(), bJ);
  std::memcpy(h + bD + bL + bJ, I.data(), bI);
  double* dd = (double*)ctx.arena.get("htab_d", bD);
  long* dl = (long*)ctx.arena.get("htab_l", bL);
  CoaxJob* dj = (CoaxJob*)ctx.arena.get("htab_j", bJ);
  int* di = (int*)ctx.arena.get("htab_i", bI);
  double* dz = (double*)ctx.arena.get("htab_z", c.cZ * sizeof(double));
  FMM_HIP(hipMemcpyAsync(dd, h, bD, hipMemcpyHostToDevice, ctx.stream));
  FMM_HIP(hipMemcpyAsync(dl, h + bD, bL, hipMemcpyHostToDevice, ctx.stream));
  if (bJ) FMM_HIP(hipMemcpyAsync(dj, h + bD + bL, bJ, hipMemcpyHostToDevice, ctx.stream));
  FMM_HIP(hipMemcpyAsync(di, h + bD + bL + bJ, bI, hipMemcpyHostToDevice, ctx.stream));
  if (!H.jobs.empty())
    hipLaunchKernelGGL(k_coax, dim3((unsigned)H.jobs.size(), (unsigned)(mmax + 1)), dim3(256), 0, ctx.stream, dj, dd + o_series,
                       (const long*)ctx.arena.get("hgaunt_o", c.gaunt->off.size() * sizeof(long)),
                       (const double*)ctx.arena.get("hgaunt_g", c.gaunt->g.size() * sizeof(double)), c.gaunt->P + 1,
                       dl + c.o_ztoff, P1, dz, dz + c.o_zt);
  FMM_HIP(hipGetLastError());
  c.valid = true;
  return c;
}

template <typename TN, bool CHG, bool DIP, bool FLD>
void hp2p(const DevPlan& P, const int* items, int n, int kind, double kre, double kim, const double* spos,
          const TN* str, const double* str64, const double* tpos, double* pot, double* fo, hipStream_t s) {
  DevPlan Q = P;
  Q.p2p_items = items;
  Q.n_p2p = n;
  hipLaunchKernelGGL((k_hp2p<TN, CHG, DIP, FLD>), dim3(item_groups(n)), dim3(kP2PBlock * kItemWaves), 0, s, Q, kre, kim,
                     spos, str, str64, tpos, kind, pot, fo);
}

template <typename TN>
void launch_hp2p(const DevPlan& P, const int* items, int n, int kind, double kre, double kim,
                 const double* spos, const TN* str, const double* str64, const double* tpos, int ifcharge, int ifdipole,
                 bool fld, double* pot, double* fo, hipStream_t s) {
  if (n == 0) return;
#define HCASE(C, Dp, F) \
  if (ifcharge == C && ifdipole == Dp && fld == F) return hp2p<TN, C, Dp, F>(P, items, n, kind, kre, kim, spos, str, str64, tpos, pot, fo, s);
  HCASE(1, 0, false) HCASE(1, 0, true) HCASE(0, 1, false) HCASE(0, 1, true) HCASE(1, 1, false) HCASE(1, 1, true)
#undef HCASE
}

// LDS of k_heval3 (L2P) at degree pd
size_t helm_lds_eval(int pd) { return sizeof(double) * 2 * 64 * (size_t)(pd + 2); }

// LDS of the kernels at expansion order p; whether all of it fits
struct HelmLds {
  bool fits = false, form2 = false, m2l = false;
  size_t form = 0, form2_lds = 0, ps = 0;
  int ts = 0, region2 = 0;
};
HelmLds helm_lds(int p, size_t ldsmax) {
  HelmLds W;
  const int K = (p + 1) * (p + 1), Hh = (p + 2) * (p + 3) / 2, Fn = p + 2;
  const size_t per_src = 2 * (size_t)Hh + 2 * (size_t)Fn + 12;
  if (sizeof(double) * (4 * (size_t)K + per_src) > ldsmax) return W;
  const int ts = (int)((ldsmax / sizeof(double) - 4 * (size_t)K) / per_src);
  W.ts = std::max(1, std::min(32, ts));
  W.form = sizeof(double) * (4 * (size_t)K + (size_t)W.ts * per_src);
  // per-thread-sum P2M/P2L: half tables up to degree p+1 held by 256
  // threads x kHFormItems entries, outputs by 256 x kHFormOut
  // (LDS: 64 KB, or what holds 4 sources at order p+1; the kernel picks
  // its tile from what is left after the factor head)
  W.form2 = Hh <= 256 * kHFormItems && K <= 256 * kHFormOut;
  W.form2_lds = std::max<size_t>((size_t)64 * 1024,
                                 hform2_fac_bytes(p) + sizeof(double) * (2 * ((size_t)Hh + Fn) + 8) * 4);
  W.region2 = (int)((W.form2_lds - hform2_fac_bytes(p)) / sizeof(double));
  W.ps = sizeof(double) * 4 * (size_t)K;
  W.m2l = sizeof(double) * 6 * (size_t)K <= ldsmax;
  W.fits = !(W.form2 && W.form2_lds > ldsmax) && W.ps <= ldsmax && helm_lds_eval(p + 1) <= ldsmax;
  return W;
}

}  // namespace

// TN: near-field pair arithmetic (double, or float with FP64 offsets and accumulation)
template <typename TN>
int helm_solve(Context& ctx, const LapCall& c) {
  auto t0 = std::chrono::steady_clock::now();
  double eps;
  int nbox;
  if (!iprec_params(c.iprec, c.ns, c.nt, eps, nbox)) return 32;
  const bool tri = c.tri_dev != nullptr;
  const cplx zk(c.zk_re, c.zk_im);
  // triangle FMM: the near-field rule (of iprec unless the caller names one)
  const std::vector<double>* sym = nullptr;
  if (tri) {
    if (!std::is_same<TN, double>::value) return 128;
    nbox = tri_nbox(c.iprec, c.ns, c.nt);
    sym = &tri_sym_rule(c.tri_nqtri > 0 ? c.tri_nqtri : htri_nqtri(c.iprec));
    if (sym->empty() || sym->size() / 3 > (size_t)kSymRuleMax) return 128;
  }
  const int ns = c.ns, nt = c.nt;
  const Flags f{c.ifcharge ? 1 : 0, c.ifdipole ? 1 : 0, c.ifpot ? 1 : 0, c.iffld ? 1 : 0,
                nt > 0 && c.ifpottarg ? 1 : 0, nt > 0 && c.iffldtarg ? 1 : 0};
  QueuedWork queued(ctx);
  thread_local Octree tree;  // storage reused across calls
  const int* dsperm = nullptr;
  const int* dtperm = nullptr;
  // the interaction lists are built after the first kernels are queued
  if (device_tree_enabled()) {
    if (build_octree_device(ctx, ctx.stream, c.src_dev, ns, c.trg_dev, nt, nbox, tree, &dsperm, &dtperm, false) != 0)
      return 4;
  } else if (build_octree(c.src_host, ns, c.trg_host, nt, nbox, tree, false) != 0) {
    return 4;
  }
  auto t_tree = std::chrono::steady_clock::now();
  // the tables this context holds, or a plan of new ones; nothing is queued
  // for them until the order has been checked
  if (!ctx.helm_tables) ctx.helm_tables = std::make_shared<HelmCache>();
  HelmCache* HC = static_cast<HelmCache*>(ctx.helm_tables.get());
  const bool held = HC->valid && HC->H.zk == zk && HC->H.size == tree.size && HC->H.nlev == tree.nlev && HC->H.eps == eps;
  const size_t ldsmax = max_lds_bytes(ctx);
  int most = kMaxHelmOrder;
  while (most > 0 && !helm_lds(most, ldsmax).fits) most--;
  HelmHostTables plan;
  if (!held && !plan_helm_tables(zk, tree.size, tree.nlev, eps, plan, most)) return 16;
  const int pmax = held ? HC->H.pmax : plan.pmax, K = (pmax + 1) * (pmax + 1);
  const HelmLds W = helm_lds(pmax, ldsmax);
  if (!held) helm_upload_tables(ctx, *HC, std::move(plan));
  const HelmHostTables& H = HC->H;
  thread_local Flat FA, FB, FC;  // plan parts: boxes, near lists, far lists (storage reused)
  FA.I.clear(); FA.D.clear(); FB.I.clear(); FB.D.clear(); FC.I.clear(); FC.D.clear();
  PlanOffsets O;
  build_plan_boxes(tree, f, FA, O, 2);
  auto t1 = std::chrono::steady_clock::now();
  hipStream_t s = ctx.stream;
  Timer tm;
  tm.start(s, 11);
  // plan uploads go through pinned staging buffers so that they do not wait
  // for the kernels already queued
  auto upload_ints = [&](const char* name, const std::vector<int>& v, hipStream_t st) {
    int* h = (int*)ctx.arena.get_host(std::string(name) + "_h", std::max<size_t>(v.size(), 1) * sizeof(int));
    std::memcpy(h, v.data(), v.size() * sizeof(int));
    int* d = (int*)ctx.arena.get(name, std::max<size_t>(v.size(), 1) * sizeof(int));
    FMM_HIP(hipMemcpyAsync(d, h, v.size() * sizeof(int), hipMemcpyHostToDevice, st));
    return d;
  };
  // the near field (P2P) runs on a second stream into its own sums, which
  // the final scatter adds to the far-field sums
  hipStream_t s2 = near_stream(ctx);
  int* dI = upload_ints("plan_i", FA.I, s);
  double* hD = (double*)ctx.arena.get_host("plan_d_h", FA.D.size() * sizeof(double));
  std::memcpy(hD, FA.D.data(), FA.D.size() * sizeof(double));
  double* dD = (double*)ctx.arena.get("plan_d", FA.D.size() * sizeof(double));
  FMM_HIP(hipMemcpyAsync(dD, hD, FA.D.size() * sizeof(double), hipMemcpyHostToDevice, s));
  DevPlan P = make_devplan(tree, pmax, O, dI, dD);
  const int* gi = (const int*)ctx.arena.get("hgeo_i", HC->gI * sizeof(int));
  const double* gd = (const double*)ctx.arena.get("hgeo_d", HC->gD * sizeof(double));
  const long* gl = (const long*)ctx.arena.get("hgeo_l", HC->gL * sizeof(long));
  const int* ti = (const int*)ctx.arena.get("htab_i", HC->cI * sizeof(int));
  const double* td = (const double*)ctx.arena.get("htab_d", HC->cD * sizeof(double));
  const long* tl = (const long*)ctx.arena.get("htab_l", HC->cL * sizeof(long));
  const double* tz = (const double*)ctx.arena.get("htab_z", HC->cZ * sizeof(double));
  DevTables Tb{};
  Tb.p = pmax;
  Tb.off_rot = gi + HC->o_offrot; Tb.off_dist = gi + HC->o_offdist; Tb.oct_rot = gi + HC->o_octrot;
  Tb.fac = gd + HC->o_fac; Tb.off_phase = gd + HC->o_offph; Tb.oct_phase = gd + HC->o_octph;
  Tb.rot = gd + HC->o_rot; Tb.rot_off = gl + HC->o_rotoff;
  HelmDev Hd;
  Hd.kre = zk.real(); Hd.kim = zk.imag();
  Hd.nd = H.geo->ndist;
  Hd.plev = ti + HC->o_plev; Hd.sclev = td + HC->o_sclev; Hd.ptrunc = ti + HC->o_ptrunc;
  Hd.coax = tl + HC->o_coax; Hd.z = tz;
  Hd.rot_sd = gd + HC->o_rotsd;
  Hd.zt = tz + HC->o_zt; Hd.zt_off = tl + HC->o_ztoff;
  const size_t nb = tree.nboxes;
  double* spos = (double*)ctx.arena.get("spos", sizeof(double) * 4 * (size_t)ns);
  double* str64 = (double*)ctx.arena.get("str64", sizeof(double) * 8 * (size_t)ns);
  constexpr bool near32 = sizeof(TN) < sizeof(double);
  float* str32 = near32 ? (float*)ctx.arena.get("str32", sizeof(float) * 8 * (size_t)ns) : nullptr;
  const TN* strn = near32 ? (const TN*)(const void*)str32 : (const TN*)(const void*)str64;
  double* tpos = (double*)ctx.arena.get("tpos", sizeof(double) * 4 * (size_t)std::max(nt, 1));
  double* mp = (double*)ctx.arena.get("mp", sizeof(double) * 2 * K * nb, 16);
  double* lo = (double*)ctx.arena.get("lo", sizeof(double) * 2 * K * nb, 16);
  double* pot_s = (double*)ctx.arena.get("pot_s", sizeof(double) * 2 * (size_t)ns);
  double* fld_s = (double*)ctx.arena.get("fld_s", sizeof(double) * 6 * (size_t)ns);
  double* pot_t = (double*)ctx.arena.get("pot_t", sizeof(double) * 2 * (size_t)std::max(nt, 1));
  double* fld_t = (double*)ctx.arena.get("fld_t", sizeof(double) * 6 * (size_t)std::max(nt, 1));
  double* pot_sn = (double*)ctx.arena.get("pot_sn", sizeof(double) * 2 * (size_t)ns);
  double* fld_sn = (double*)ctx.arena.get("fld_sn", sizeof(double) * 6 * (size_t)ns);
  double* pot_tn = (double*)ctx.arena.get("pot_tn", sizeof(double) * 2 * (size_t)std::max(nt, 1));
  double* fld_tn = (double*)ctx.arena.get("fld_tn", sizeof(double) * 6 * (size_t)std::max(nt, 1));
  const int* sperm = dsperm ? dsperm : dI + O.sperm;
  const int* tperm = dsperm ? dtperm : dI + O.tperm;
  P.src_perm = sperm;
  P.trg_perm = tperm;
  // (triangles: the point strengths are not used -- k_tri_prep forms the
  // triangle densities and quadrature points -- and no dipole vectors are read)
  hipLaunchKernelGGL(k_gather_sources, dim3(blocks(ns, 256)), dim3(256), 0, s, ns, sperm, c.src_dev,
                     c.q_dev, c.ds_dev, c.dv_dev, tri ? 0 : f.ifcharge, tri ? 0 : f.ifdipole, spos, str64, str32);
  if (nt > 0)
    hipLaunchKernelGGL(k_gather_targets, dim3(blocks(nt, 256)), dim3(256), 0, s, nt, tperm, c.trg_dev, tpos);
  auto zero = [&](double* a, size_t n) {
    hipLaunchKernelGGL((k_fill_zero<double>), dim3(std::min<size_t>(blocks(n, 256), 4096)), dim3(256), 0, s, n, a);
  };
  zero(mp, 2 * (size_t)K * nb);
  zero(lo, 2 * (size_t)K * nb);
  zero(pot_s, 2 * (size_t)ns);
  zero(fld_s, 6 * (size_t)ns);
  zero(pot_sn, 2 * (size_t)ns);
  zero(fld_sn, 6 * (size_t)ns);
  if (nt > 0) {
    zero(pot_t, 2 * (size_t)nt);
    zero(fld_t, 6 * (size_t)nt);
    zero(pot_tn, 2 * (size_t)nt);
    zero(fld_tn, 6 * (size_t)nt);
  }
  // triangle FMM: frames and densities in sorted order, and the quadrature
  // points that stand for the triangles in P2M / P2L (their box ranges
  // counted in points)
  const double* fpos = spos;
  const double* fstr = str64;
  double *tgeo = nullptr, *tstr = nullptr;
  int* tri_rng = nullptr;
  if (tri) {
    const std::vector<double> rule = tri_rule(c.iprec, true);
    const int nq = (int)rule.size() / 3;
    tgeo = (double*)ctx.arena.get("tri_geo", sizeof(double) * kTriGeo * (size_t)ns);
    tstr = (double*)ctx.arena.get("tri_str", sizeof(double) * 4 * (size_t)ns);
    double* npos = (double*)ctx.arena.get("tri_npos", sizeof(double) * 4 * (size_t)ns * nq);
    double* nstr = (double*)ctx.arena.get("tri_nstr", sizeof(double) * 8 * (size_t)ns * nq);
    double* hr = (double*)ctx.arena.get_host("tri_rule_h", sizeof(double) * rule.size());
    std::memcpy(hr, rule.data(), sizeof(double) * rule.size());
    double* dr = (double*)ctx.arena.get("tri_rule", sizeof(double) * rule.size());
    FMM_HIP(hipMemcpyAsync(dr, hr, sizeof(double) * rule.size(), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_tri_prep, dim3(blocks(ns, 256)), dim3(256), 0, s, ns, sperm, c.tri_dev, c.q_dev,
                       c.ds_dev, f.ifcharge, f.ifdipole, nq, dr, tgeo, tstr, npos, nstr);
    tri_rng = (int*)ctx.arena.get("tri_ranges", sizeof(int) * 2 * nb);
    hipLaunchKernelGGL(k_scale_ranges, dim3(blocks(nb, 256)), dim3(256), 0, s, (int)nb, P.isrc, P.nsrc, nq, tri_rng,
                       tri_rng + nb);
    fpos = npos;
    fstr = nstr;
  }
  FMM_HIP(hipEventRecord(ctx.aux_ev[0], s));  // inputs gathered, sums zeroed
  tm.mark(1);
  const double* fac = Tb.fac;
  auto form = [&](auto irreg, int nbx, double* out) {
    constexpr bool IR = decltype(irreg)::value;
    if (!nbx) return;
    DevPlan PF = P;  // the current plan (P2L needs list 4), source ranges in points for triangles
    if (tri) {
      PF.isrc = tri_rng;
      PF.nsrc = tri_rng + nb;
    }
    if (!W.form2) {
      hipLaunchKernelGGL((k_hform<IR>), dim3(nbx), dim3(256), W.form, s, PF, Hd, fac, fpos, fstr,
                         f.ifcharge, f.ifdipole, W.ts, out);
    } else if (f.ifcharge && f.ifdipole) {
      hipLaunchKernelGGL((k_hform2<IR, true, true>), dim3(nbx), dim3(256), W.form2_lds, s, PF, Hd, fac, fpos, fstr, W.region2, out);
    } else if (f.ifcharge) {
      hipLaunchKernelGGL((k_hform2<IR, true, false>), dim3(nbx), dim3(256), W.form2_lds, s, PF, Hd, fac, fpos, fstr, W.region2, out);
    } else if (f.ifdipole) {
      hipLaunchKernelGGL((k_hform2<IR, false, true>), dim3(nbx), dim3(256), W.form2_lds, s, PF, Hd, fac, fpos, fstr, W.region2, out);
    }
  };
  // STEP 1: P2M (hfmm3dpart.f:681-757)
  form(std::false_type{}, P.n_p2m, mp);
  tm.mark(2);
  // STEP 3: M2M, bottom-up
  for (size_t g = 0; g < O.m2m_groups.size(); g++) {
    hipLaunchKernelGGL(k_hm2m, dim3(O.m2m_groups[g].second, 8), dim3(256), W.ps, s, P, Tb, Hd,
                       O.m2m_groups[g].first, HC->m2m_base + O.m2m_group_level[g], mp, lo);
    hipLaunchKernelGGL((k_child_sum<double>), dim3(O.m2m_groups[g].second), dim3(256), 0, s, P,
                       O.m2m_groups[g].first, mp, lo);
  }
  tm.mark(3);
  // while the device runs P2M and M2M: list 1 and the P2P plan
  auto t_lists0 = std::chrono::steady_clock::now();
  tree_lists_near(tree);
  build_plan_near(tree, f, FB, O);
  // the P2P work items are addressed explicitly: they must lie in this part
  if (O.p2p0 + 3 * (size_t)O.n_p2p0 > FB.I.size() || O.p2p1 + 3 * (size_t)O.n_p2p1 > FB.I.size())
    throw HipError("plan: P2P work items outside the near-field part of the plan");
  auto t_lists1 = std::chrono::steady_clock::now();
  // STEP 8: P2P (hfmm3dpart.f:1101-1180) on the second stream, once the
  // inputs are gathered; its plan part is uploaded on that stream
  FMM_HIP(hipStreamWaitEvent(s2, ctx.aux_ev[0], 0));
  Timer tn;
  tn.start(s2, 2);
  const int* dIB = upload_ints("plan_ib", FB.I, s2);
  devplan_near(P, O, dIB);
  if (tri && c.far_only) {
    // the far field alone
  } else if (tri && (f.ifcharge || f.ifdipole)) {
    double* hr = (double*)ctx.arena.get_host("htri_rule_h", sizeof(double) * 3 * kSymRuleMax);
    std::memcpy(hr, sym->data(), sizeof(double) * sym->size());
    double* dr = (double*)ctx.arena.get("htri_rule", sizeof(double) * 3 * kSymRuleMax);
    FMM_HIP(hipMemcpyAsync(dr, hr, sizeof(double) * sym->size(), hipMemcpyHostToDevice, s2));
    const HtriParams hp{zk.real(), zk.imag(), std::abs(zk), c.tri_lapc, c.tri_lapd, (int)sym->size() / 3, dr};
    auto tri_near = [&](const int* items, int n, int kind, double* po, double* fo) {
      launch_htri_p2p(P, items, n, f.ifcharge, f.ifdipole, tgeo, tstr, spos, tpos, kind, hp, po, fo, s2);
    };
    tri_near(dIB + O.p2p0, O.n_p2p0, 0, pot_sn, f.iffld ? fld_sn : nullptr);
    tri_near(dIB + O.p2p1, O.n_p2p1, 1, pot_tn, f.iffldtarg ? fld_tn : nullptr);
  } else if (f.ifcharge || f.ifdipole) {
    launch_hp2p<TN>(P, dIB + O.p2p0, O.n_p2p0, 0, Hd.kre, Hd.kim, spos, strn, str64, tpos, f.ifcharge, f.ifdipole,
                    f.iffld != 0, pot_sn, fld_sn, s2);
    launch_hp2p<TN>(P, dIB + O.p2p1, O.n_p2p1, 1, Hd.kre, Hd.kim, spos, strn, str64, tpos, f.ifcharge, f.ifdipole,
                    f.iffldtarg != 0, pot_tn, fld_tn, s2);
  }
  tn.mark(1);
  FMM_HIP(hipEventRecord(ctx.aux_ev[1], s2));  // near field done
  tm.mark(4);
  // while the device runs P2P: lists 2-4 and the far-field plan
  auto t_lists2 = std::chrono::steady_clock::now();
  tree_lists_far(tree);
  build_plan_far(tree, f, FC, O);
  devplan_far(P, O, upload_ints("plan_ic", FC.I, s));
  auto t_lists3 = std::chrono::steady_clock::now();
  // STEP 2: P2L (hfmm3dpart.f:765-830)
  form(std::true_type{}, P.n_p2l, lo);
  tm.mark(5);
  // STEP 4: M2L, grouped by translation class (k_hm2l_grp) when the group's
  // expansions fit LDS and a stage's work items fit one pass, else pair by
  // pair (k_hm2l)
  if (P.n_m2l) {
    GrpShape G;
    if (HC->grouped_m2l) G = grp_shape<double>(pmax, ldsmax);
    if (G.threads > 0) {
      const size_t need = grp_lds_bytes<double>(pmax, G.room, G.teams);
#define HM2L_GRP(NT_, I_) \
  launch_pieces(P.n_m2l, NT_, [&](long first, unsigned count) {                                                     \
    DevPlan Q = P;                                                                                                  \
    Q.m2l_boxes += first;                                                                                           \
    hipLaunchKernelGGL((k_hm2l_grp<NT_, I_>), dim3(count), dim3(NT_), need, s, Q, Tb, Hd, G.room, G.lts, mp, lo);   \
  })
      if (G.threads == 256) HM2L_GRP(256, 1);
      else if (G.items == 1) HM2L_GRP(512, 1);
      else HM2L_GRP(512, 2);
#undef HM2L_GRP
    } else if (W.m2l)
      hipLaunchKernelGGL((k_hm2l<true>), dim3(P.n_m2l), dim3(256), sizeof(double) * 6 * (size_t)K, s, P, Tb, Hd, mp, lo);
    else
      hipLaunchKernelGGL((k_hm2l<false>), dim3(P.n_m2l), dim3(256), W.ps, s, P, Tb, Hd, mp, lo);
  }
  tm.mark(6);
  // STEP 5: L2L, top-down
  for (size_t g = 0; g < O.l2l_groups.size(); g++)
    hipLaunchKernelGGL(k_hl2l, dim3(O.l2l_groups[g].second, 8), dim3(256), W.ps, s, P, Tb, Hd,
                       O.l2l_groups[g].first, HC->l2l_base + O.l2l_group_level[g], lo);
  tm.mark(7);
  // STEP 7: L2P and STEP 6: M2P (list 3), from packed expansions
  {
    const int grad = (f.iffld || f.iffldtarg) ? 1 : 0;
    const bool want_src = f.ifpot || f.iffld, want_trg = f.ifpottarg || f.iffldtarg;
    const int nbx = tree.nboxes;
    // host side: boxes to pack, their entry offsets, the box -> offset maps and
    // the work items (box, kind, first point) in chunks of 64 points
    std::vector<int> hv;                  // m2p slots | l2p slots | m2p pack | l2p pack | items
    std::vector<int> slot_m(nbx, -1), slot_l(nbx, -1), pk_m, off_m, pk_l, off_l, it_m, it_l, red_m;
    int tot_m = 0, tot_l = 0, pdmax = 1;
    auto pdof = [&](int lev) { return H.plev[lev] + grad; };
    auto entries = [&](int lev) { const int pd = pdof(lev); return (pd + 1) * (pd + 2) / 2; };
    auto items = [&](std::vector<int>& it, int b) {
      if (want_src)
        for (int q = 0; q < tree.nsrc[b]; q += 64) { it.push_back(b); it.push_back(0); it.push_back(q); }
      if (want_trg)
        for (int q = 0; q < tree.ntrg[b]; q += 64) { it.push_back(b); it.push_back(1); it.push_back(q); }
    };
    for (int b = 0; b < nbx; b++) {
      const bool has_pts = (want_src && tree.nsrc[b] > 0) || (want_trg && tree.ntrg[b] > 0);
      if (tree.nchild[b] == 0 && tree.level[b] >= 2 && has_pts) {
        slot_l[b] = tot_l;
        pk_l.push_back(b);
        off_l.push_back(tot_l);
        tot_l += entries(tree.level[b]);
        pdmax = std::max(pdmax, pdof(tree.level[b]));
        items(it_l, b);
      }
      if (tree.list[2].count(b) > 0 && has_pts) {
        // list 3 in slices of about kSlice half-table entries: one workgroup per
        // (64 points, slice), the slices summed in order by k_slice_reduce
        constexpr int kSlice = 1024;
        std::vector<int> cuts = {tree.list[2].off[b]};
        int cost = 0;
        for (int k = tree.list[2].off[b]; k < tree.list[2].off[b + 1]; k++) {
          const int j = tree.list[2].idx[k];
          if (tree.level[j] < 2 || tree.nsrc[j] == 0) continue;
          cost += entries(tree.level[j]);
          if (cost >= kSlice && k + 1 < tree.list[2].off[b + 1]) { cuts.push_back(k + 1); cost = 0; }
          if (slot_m[j] >= 0) continue;
          slot_m[j] = tot_m;
          pk_m.push_back(j);
          off_m.push_back(tot_m);
          tot_m += entries(tree.level[j]);
          pdmax = std::max(pdmax, pdof(tree.level[j]));
        }
        cuts.push_back(tree.list[2].off[b + 1]);
        const int nsl = (int)cuts.size() - 1;
        auto slices = [&](int kind, int npts) {
          for (int q = 0; q < npts; q += 64) {
            red_m.push_back(b); red_m.push_back(kind); red_m.push_back(q);
            red_m.push_back((int)(it_m.size() / 5)); red_m.push_back(nsl);
            for (int c = 0; c < nsl; c++) {
              it_m.push_back(b); it_m.push_back(kind); it_m.push_back(q);
              it_m.push_back(cuts[c]); it_m.push_back(cuts[c + 1]);
            }
          }
        };
        if (want_src) slices(0, tree.nsrc[b]);
        if (want_trg) slices(1, tree.ntrg[b]);
      }
    }
    size_t o_sm = 0, o_sl = nbx, o_pm = 2 * (size_t)nbx, o_om = o_pm + pk_m.size(), o_pl = o_om + off_m.size(),
           o_ol = o_pl + pk_l.size(), o_im = o_ol + off_l.size(), o_il = o_im + it_m.size(),
           o_rm = o_il + it_l.size();
    hv.reserve(o_rm + red_m.size());
    for (auto* v : {&slot_m, &slot_l, &pk_m, &off_m, &pk_l, &off_l, &it_m, &it_l, &red_m})
      hv.insert(hv.end(), v->begin(), v->end());
    (void)o_sm;
    int* hh = (int*)ctx.arena.get_host("heval_i_h", std::max<size_t>(hv.size(), 1) * sizeof(int));
    std::memcpy(hh, hv.data(), hv.size() * sizeof(int));
    int* dh = (int*)ctx.arena.get("heval_i", std::max<size_t>(hv.size(), 1) * sizeof(int));
    FMM_HIP(hipMemcpyAsync(dh, hh, hv.size() * sizeof(int), hipMemcpyHostToDevice, s));
    if (!it_l.empty()) {
      double* pack = (double*)ctx.arena.get("hpack_l", sizeof(double) * 16 * (size_t)std::max(tot_l, 1));
      hipLaunchKernelGGL((k_hpack<false>), dim3((unsigned)pk_l.size()), dim3(256), 0, s, P, Hd, fac, lo, dh + o_pl,
                         dh + o_ol, grad, pack);
      hipLaunchKernelGGL((k_heval3<false>), dim3((unsigned)(it_l.size() / 3)), dim3(64), helm_lds_eval(pdmax), s, P, Hd, fac, pack,
                         dh + o_sl, dh + o_il, grad, spos, tpos, f.ifpot, f.iffld, f.ifpottarg, f.iffldtarg, pot_s,
                         fld_s, pot_t, fld_t, (double*)nullptr);
    }
    tm.mark(8);
    if (!it_m.empty() && !pk_m.empty()) {
      double* pack = (double*)ctx.arena.get("hpack_m", sizeof(double) * 16 * (size_t)std::max(tot_m, 1));
      hipLaunchKernelGGL((k_hpack<true>), dim3((unsigned)pk_m.size()), dim3(256), 0, s, P, Hd, fac, mp, dh + o_pm,
                         dh + o_om, grad, pack);
      const size_t nsub = it_m.size() / 5;
      double* partial = (double*)ctx.arena.get("hpart_m", sizeof(double) * 8 * 64 * nsub);
      hipLaunchKernelGGL((k_heval3<true>), dim3((unsigned)nsub), dim3(64), 0, s, P, Hd, fac, pack, dh + o_sm,
                         dh + o_im, grad, spos, tpos, f.ifpot, f.iffld, f.ifpottarg, f.iffldtarg, pot_s, fld_s, pot_t,
                         fld_t, partial);
      hipLaunchKernelGGL(k_slice_reduce, dim3((unsigned)(red_m.size() / 5)), dim3(64), 0, s, dh + o_rm, partial,
                         P.isrc, P.nsrc, P.itrg, P.ntrg, f.ifpot, f.iffld, f.ifpottarg, f.iffldtarg, pot_s, fld_s,
                         pot_t, fld_t);
    }
  }
  tm.mark(9);
  // far + near, scattered back to the caller's order (h3dpsort / h3dfsort)
  FMM_HIP(hipStreamWaitEvent(s, ctx.aux_ev[1], 0));
  auto scatter = [&](int n, int w, const int* perm, const double* far, const double* near, double* out) {
    hipLaunchKernelGGL(k_scatter_sum, dim3(blocks(n, 256)), dim3(256), 0, s, n, w, perm, far, near, out);
  };
  if (f.ifpot) scatter(ns, 1, sperm, pot_s, pot_sn, c.pot_dev);
  if (f.iffld) scatter(ns, 3, sperm, fld_s, fld_sn, c.fld_dev);
  if (f.ifpottarg) scatter(nt, 1, tperm, pot_t, pot_tn, c.pottarg_dev);
  if (f.iffldtarg) scatter(nt, 3, tperm, fld_t, fld_tn, c.fldtarg_dev);
  tm.mark(10);
  FMM_HIP(hipGetLastError());
  queued.wait();
  auto& lt = last_timings();
  lt.assign(13, 0.0);
  auto ms = [](auto a, auto b) { return std::chrono::duration<double, std::milli>(b - a).count(); };
  lt[0] = ms(t0, t1);
  // main stream: upload, P2M, M2M, (near-plan gap), P2L, M2L, L2L, L2P, M2P,
  // wait for the near field + scatter; the P2P time is the second stream's
  auto el = tm.elapsed();
  el.resize(10, 0.0);
  lt[1] = el[0]; lt[2] = el[1]; lt[3] = el[4]; lt[4] = el[2]; lt[5] = el[5];
  lt[6] = el[6]; lt[7] = el[7]; lt[8] = el[8]; lt[9] = tn.elapsed()[0];
  double tot = 0;
  for (auto v : el) tot += v;
  lt[10] = tot + lt[0];
  lt[11] = ms(t0, t_tree);
  lt[12] = ms(t_lists0, t_lists1) + ms(t_lists2, t_lists3);
  return 0;
}

int helm_solve_mode(Context& ctx, const LapCall& c, int mode) {
  mode = c.tri_dev ? 0 : effective_precision(c.iprec, mode);
  last_precision() = mode;
  switch (mode) {
    case 0: return helm_solve<double>(ctx, c);
    case 1: return helm_solve<float>(ctx, c);
  }
  return 128;
}

// h3dpartdirect on the device: identity order, one pass.
int helm_direct(Context& ctx, const LapCall& c) {
  const int ns = c.ns, nt = c.nt;
  hipStream_t s = ctx.stream;
  const size_t nmax = (size_t)std::max(std::max(ns, nt), 1);
  std::vector<int> id(nmax);
  for (size_t i = 0; i < id.size(); i++) id[i] = (int)i;
  int* dperm = (int*)ctx.arena.get("plan_i", id.size() * sizeof(int));
  FMM_HIP(hipMemcpyAsync(dperm, id.data(), id.size() * sizeof(int), hipMemcpyHostToDevice, s));
  double* spos = (double*)ctx.arena.get("spos", sizeof(double) * 4 * (size_t)std::max(ns, 1));
  double* str64 = (double*)ctx.arena.get("str64", sizeof(double) * 8 * (size_t)std::max(ns, 1));
  double* tpos = (double*)ctx.arena.get("tpos", sizeof(double) * 4 * (size_t)std::max(nt, 1));
  double* pot = (double*)ctx.arena.get("pot_s", sizeof(double) * 2 * nmax);
  double* fld = (double*)ctx.arena.get("fld_s", sizeof(double) * 6 * nmax);
  if (ns > 0)
    hipLaunchKernelGGL(k_gather_sources, dim3(blocks(ns, 256)), dim3(256), 0, s, ns, dperm, c.src_dev,
                       c.q_dev, c.ds_dev, c.dv_dev, c.ifcharge ? 1 : 0, c.ifdipole ? 1 : 0, spos, str64,
                       (float*)nullptr);
  // the slices' sums: at most about 16 MB, and none where the points alone fill
  // the chip
  const size_t npart = std::max(c.ifpot || c.iffld ? direct_partial(ns, ns) : 0,
                                c.ifpottarg || c.iffldtarg ? direct_partial(nt, ns) : 0);
  double* partial = npart ? (double*)ctx.arena.get("direct_part", sizeof(double) * npart) : nullptr;
  auto run = [&](int npts, const double* pts, int are_src) {
    if (npts <= 0) return;
    if (ns == 0 || (!c.ifcharge && !c.ifdipole)) {
      hipLaunchKernelGGL((k_fill_zero<double>), dim3(blocks(2 * (size_t)npts, 256)), dim3(256), 0, s, 2 * (size_t)npts, pot);
      hipLaunchKernelGGL((k_fill_zero<double>), dim3(blocks(6 * (size_t)npts, 256)), dim3(256), 0, s, 6 * (size_t)npts, fld);
      return;
    }
    const int nsl = direct_slices(npts, ns);
#define HDCASE(C, D)                                                                                       \
  if ((c.ifcharge ? 1 : 0) == C && (c.ifdipole ? 1 : 0) == D)                                              \
    launch_pieces(blocks(npts, 64), 64 * kDirectWaves, [&](long first, unsigned count) {                   \
      hipLaunchKernelGGL((k_hdirect<C, D>), dim3(count, nsl), dim3(64 * kDirectWaves), 0, s, c.zk_re,      \
                         c.zk_im, ns, spos, str64, npts, (int)(64 * first), pts, are_src, partial, pot, fld); \
    });
    HDCASE(1, 0) HDCASE(0, 1) HDCASE(1, 1)
#undef HDCASE
    if (nsl > 1)
      hipLaunchKernelGGL(k_direct_sum, dim3(blocks(npts, 256)), dim3(256), 0, s, npts, nsl, partial, pot, fld);
  };
  auto copy_out = [&](int npts, int wpot, double* po, int wfld, double* fo) {
    if (wpot) FMM_HIP(hipMemcpyAsync(po, pot, sizeof(double) * 2 * npts, hipMemcpyDeviceToDevice, s));
    if (wfld) FMM_HIP(hipMemcpyAsync(fo, fld, sizeof(double) * 6 * npts, hipMemcpyDeviceToDevice, s));
  };
  if (ns > 0 && (c.ifpot || c.iffld)) {
    run(ns, nullptr, 1);
    copy_out(ns, c.ifpot, c.pot_dev, c.iffld, c.fld_dev);
  }
  if (nt > 0 && (c.ifpottarg || c.iffldtarg)) {
    hipLaunchKernelGGL(k_gather_targets, dim3(blocks(nt, 256)), dim3(256), 0, s, nt, dperm, c.trg_dev, tpos);
    run(nt, tpos, 0);
    copy_out(nt, c.ifpottarg, c.pottarg_dev, c.iffldtarg, c.fldtarg_dev);
  }
  FMM_HIP(hipGetLastError());
  FMM_HIP(hipStreamSynchronize(s));
  return 0;
}

// h3dtriadirect (src/hfmm3dtria.f:1456) on the device: caller's order, one
// pass over all triangles per point, the near-field rule of degree
// c.tri_nqtri.
int htri_direct(Context& ctx, const LapCall& c) {
  const int n = c.ns, nt = c.nt;
  const std::vector<double>& sr = tri_sym_rule(c.tri_nqtri);
  if (sr.empty() || sr.size() / 3 > (size_t)kSymRuleMax) return 128;
  QueuedWork queued(ctx);
  hipStream_t s = ctx.stream;
  double* hr = (double*)ctx.arena.get_host("htri_rule_h", sizeof(double) * 3 * kSymRuleMax);
  std::memcpy(hr, sr.data(), sizeof(double) * sr.size());
  double* dr = (double*)ctx.arena.get("htri_rule", sizeof(double) * 3 * kSymRuleMax);
  FMM_HIP(hipMemcpyAsync(dr, hr, sizeof(double) * sr.size(), hipMemcpyHostToDevice, s));
  const cplx zk(c.zk_re, c.zk_im);
  const HtriParams hp{zk.real(), zk.imag(), std::abs(zk), c.tri_lapc, c.tri_lapd, (int)sr.size() / 3, dr};
  std::vector<int> id((size_t)std::max(n, 1));
  for (size_t i = 0; i < id.size(); i++) id[i] = (int)i;
  int* dperm = (int*)ctx.arena.get("plan_i", id.size() * sizeof(int));
  FMM_HIP(hipMemcpyAsync(dperm, id.data(), id.size() * sizeof(int), hipMemcpyHostToDevice, s));
  double* geo = (double*)ctx.arena.get("tri_geo", sizeof(double) * kTriGeo * (size_t)std::max(n, 1));
  double* tstr = (double*)ctx.arena.get("tri_str", sizeof(double) * 4 * (size_t)std::max(n, 1));
  const int ifc = c.ifcharge ? 1 : 0, ifd = c.ifdipole ? 1 : 0;
  if (n > 0)
    hipLaunchKernelGGL(k_tri_prep, dim3(blocks(n, 256)), dim3(256), 0, s, n, dperm, c.tri_dev, c.q_dev, c.ds_dev,
                       ifc, ifd, 0, (const double*)nullptr, geo, tstr, (double*)nullptr, (double*)nullptr);
  const size_t nmax = (size_t)std::max(std::max(n, nt), 1);
  double* pot = (double*)ctx.arena.get("pot_s", sizeof(double) * 2 * nmax);
  double* fld = (double*)ctx.arena.get("fld_s", sizeof(double) * 6 * nmax);
  auto run = [&](int npts, const double* pts, int centroids, int wpot, double* po, int wfld, double* fo) {
    if (npts <= 0 || !(wpot || wfld)) return;
    if (n == 0 || (!ifc && !ifd)) {
      hipLaunchKernelGGL((k_fill_zero<double>), dim3(blocks(2 * (size_t)npts, 256)), dim3(256), 0, s,
                         2 * (size_t)npts, pot);
      hipLaunchKernelGGL((k_fill_zero<double>), dim3(blocks(6 * (size_t)npts, 256)), dim3(256), 0, s,
                         6 * (size_t)npts, fld);
    } else {
      launch_htri_direct(n, geo, tstr, npts, pts, centroids, hp, ifc, ifd, pot, fld, s);
    }
    if (wpot) FMM_HIP(hipMemcpyAsync(po, pot, sizeof(double) * 2 * npts, hipMemcpyDeviceToDevice, s));
    if (wfld) FMM_HIP(hipMemcpyAsync(fo, fld, sizeof(double) * 6 * npts, hipMemcpyDeviceToDevice, s));
  };
  run(n, c.src_dev, 1, c.ifpot, c.pot_dev, c.iffld, c.fld_dev);
  run(nt, c.trg_dev, 0, c.ifpottarg, c.pottarg_dev, c.iffldtarg, c.fldtarg_dev);
  FMM_HIP(hipGetLastError());
  queued.wait();
  return 0;
}

}  // namespace fmm3d
