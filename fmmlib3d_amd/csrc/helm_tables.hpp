// Host-side pieces of the Helmholtz FMM: spherical Bessel / Hankel series,
// expansion orders (h3dterms), and the per-level translation tables.
#pragma once
#include <cmath>
#include <complex>
#include <memory>
#include <vector>

#include "tables.hpp"

namespace fmm3d {

using cplx = std::complex<double>;

// h3dall (src/helmrouts3d.f:690): hs[i] = h_i(z) sc^i, i = 0..n
void sph_hankel_scaled(int n, cplx z, double sc, cplx* hs);
// jfuns3d (src/cdjseval3d.f:15): fj[i] = j_i(z) / sc^i, i = 0..n; 0 or 8
int sph_bessel_scaled(int n, cplx z, double sc, cplx* fj);

// h3dterms (src/h3dterms.f:28): expansion order for a box of side `size`
int helmholtz_nterms(double size, cplx zk, double eps);
// h3dterms_list2 (src/h3dterms.f:192): 7^3 table by offset code
std::vector<int> helmholtz_itable(double size, cplx zk, double eps);

// One coaxial shift operator, packed by m: for m = 0..min(pin,pout) a
// (pout+1-m) x (pin+1-m) complex block (rows l = m..pout, columns n = m..pin).
struct CoaxDesc {
  long base = 0;   // offset in complex entries into HelmHostTables::z
  int pin = 0, pout = 0;
};

// What one coaxial operator is computed from: its series start at `series` in
// HelmHostTables::series with S = pin + pout: f_s (complex, s = 0..S), base^e
// (e = 0..S), ratio^e (e = 0..max(pin, pout)); mode 0: M2M (R|R), 1: M2L (S|R),
// 2: L2L (R|R); neg: the direction sign is -1.
struct CoaxJob {
  long base = 0;     // as CoaxDesc::base
  long series = 0;   // doubles
  int pin = 0, pout = 0, mode = 0, neg = 0;
  int m2l = -1;      // index of the M2L table this is, or -1
  int pad = 0;
};

// Gaunt integrals G(n,s,l;m) for 0 <= m <= min(n,l), n,l <= P,
// s = |n-l|, |n-l|+2, .., n+l, stored compactly
struct Gaunt {
  int P = -1;
  std::vector<long> off;   // [(m*(P+1)+n)*(P+1)+l]
  std::vector<double> g;
  long at(int m, int n, int l) const { return off[((size_t)m * (P + 1) + n) * (P + 1) + l]; }
};
// those of the next multiple of four from `pmax` on (so that a call's values do
// not depend on the calls before it), the last few kept for the process
std::shared_ptr<const Gaunt> gaunt_for(int pmax);

struct HelmHostTables {
  cplx zk;
  double size = 0, eps = 0;
  int nlev = -1, pmax = 0;
  std::shared_ptr<const HostTables> geo;  // factors, rotations, phases at pmax
  std::vector<int> plev;             // expansion order per level (0 below level 2)
  std::vector<double> sclev;         // rscale per level
  std::vector<int> ptrunc;           // (nlev+1) x 343 list-2 orders
  std::vector<CoaxDesc> m2l;         // (nlev+1) x ndist
  std::vector<CoaxDesc> m2m, l2l;    // per parent level
  std::vector<CoaxJob> jobs;         // one per operator
  std::vector<double> series;        // their series
  long nz = 0;                       // complex entries of all coaxial blocks
};

// build_geometry_tables(p), the last few orders kept for the process
std::shared_ptr<const HostTables> geometry_for(int p);

// The orders, list-2 tables, operator layout and series the Helmholtz FMM
// needs for a tree of root side `size` and depth `nlev`; the blocks are
// computed from the series on the device (k_coax).  Returns false, with nothing
// built, when an order exceeds `most` (what the device's LDS holds).
constexpr int kMaxHelmOrder = 120;
bool plan_helm_tables(cplx zk, double size, int nlev, double eps, HelmHostTables& H, int most = kMaxHelmOrder);
// where the 4x4 tiles of order am of M2L table t start (k_coax), off[t * (pmax + 1)
// + am]; returns their size in doubles
long coax_tile_offsets(const HelmHostTables& H, std::vector<long>& off);

// What k_coax computes and where, also compiled for the host so that the
// sanitizers see it.
#if defined(__HIP__)
#define FMM_HD __host__ __device__
#else
#define FMM_HD
#endif

// offset (complex entries) of the m-block inside a packed coaxial operator
FMM_HD inline long coax_block(int m, int pin, int pout) {
  const long A = pout + 1, B = pin + 1, M = m;
  return M * A * B - (A + B) * M * (M - 1) / 2 + (M - 1) * M * (2 * M - 1) / 6;
}
// entry (l, n) of that block, from J.base on
FMM_HD inline long coax_at(const CoaxJob& J, int m, int n, int l) {
  return J.base + coax_block(m, J.pin, J.pout) + (long)(l - m) * (J.pin + 1 - m) + (n - m);
}
// 4x4 tiles of the m-block: rows n - m, columns l - m
FMM_HD inline int coax_tile_rows(const CoaxJob& J, int m) { return (J.pin - m) / 4 + 1; }
FMM_HD inline int coax_tile_cols(const CoaxJob& J, int m) { return (J.pout - m) / 4 + 1; }
// the real part of (n, l) = (m + row, m + col) in those tiles; the imaginary
// part is 16 further
FMM_HD inline long coax_tile_at(const CoaxJob& J, int m, int row, int col) {
  return 32 * ((long)(row / 4) * coax_tile_cols(J, m) + col / 4) + (row % 4) * 4 + col % 4;
}
// the entry: f the operator's series, g the integrals G(n, s, l; m) of s = |n-l|, ..
FMM_HD inline void coax_entry(const CoaxJob& J, int n, int l, const double* f, const double* g, double& re, double& im) {
  const int S = J.pin + J.pout, s0 = n > l ? n - l : l - n;
  const double *pb = f + 2 * (S + 1), *pr = pb + S + 1;
  re = im = 0.0;
  for (int s = s0; s <= n + l; s += 2) {
    const bool neg = ((((l + s - n) / 2) & 1) != 0) != (J.neg && (s & 1));
    const double c = (neg ? -4.0 : 4.0) * M_PI * sqrt((2.0 * s + 1.0) / (4.0 * M_PI)) * g[(s - s0) / 2];
    const double pw = J.mode == 1 ? pb[n + l - s] : J.mode == 0 ? pb[s - l + n] * pr[n] : pb[s - n + l] * pr[l];
    re += c * pw * f[2 * s];
    im += c * pw * f[2 * s + 1];
  }
}

}  // namespace fmm3d
