// Laplace particle-FMM kernels for gfx950 (MI355X).
//
// Every kernel is templated on the arithmetic type T (double for the FP64
// path, float for the mixed path).  Expansions are packed complex arrays,
// coefficient (n,m) at eidx(n,m), and carry rscale = 1/side of their box, so
// translation tables are level independent.  Conventions match the
// reference's "_trunc" routines (src/laprouts3d.f:12-66 with the (-1)^m
// phase of ylgndrufw): R_n^m = r^n Yhat_n^m, S_n^m = Yhat_n^m / r^{n+1},
// multipole M_n^m = sum q conj(R_n^m(u)), local L_n^m = sum q conj(S_n^m(u))/h.
#include <hip/hip_runtime.h>

#include "kern_common.hpp"
#include "m2l_grp.hpp"

namespace fmm3d {

// ---------------------------------------------------------------------------
// P2M (src/laprouts3d.f:3210, :3835) and P2L (src/laprouts3d.f:3550, :4207;
// IRREG: irregular harmonics at the target box centre, sources taken from the
// boxes of list 4).  One workgroup per (box, range of orders |m| it writes).
//
// Each thread owns up to ITEMS half-table entries (n, a >= 0) of the range and
// accumulates, in registers over every source, for the weights
// w = q, v_x, v_y, v_z the four real sums of w_re, w_im times h_re, h_im, from
// which S^w(n, +-a) = sum_s w_s H_n^{+-a}(u_s) (H^{-a} = conj(H^a)) follow at
// the end; the weights are scalar loads, four sources at a time.  With at most
// 64 (128) entries in all the 256 threads form four (two) groups of GS that
// take the sources in turn and are added in order at the end.
// The harmonics are the scaled ones of FacLayout: a tile of sources is built in
// LDS, one thread per (source, column a) walking n with one dependent FMA per
// degree; columns are stored so that neighbouring lanes (neighbouring a) write
// neighbouring 16-byte slots.  Per-source scalars are computed 64 sources at a
// time.  The sums then go to LDS one weight at a time, and the owner of an
// entry combines the coefficients (n, +-a): charge S^q(n, -m), dipole through
// the derivative factors and degree n-1 (P2M) or n+1 (P2L) and the orders next
// to m, with (v_x -+ i v_y)/2 formed by linearity; a range of a dipole call
// therefore also builds the column on either side of it.
//
// What bounds it is the walk along a column, pt + 1 dependent steps of about ten
// instructions by the lanes that the tile's LDS admits, then the sums' FMAs (16
// per entry and source with dipoles).  So the recurrence has one dependent FMA
// per step (the normalised form had three operations), a range takes only the
// columns it writes, so that a tile holds more sources, and the tile stays near
// 32 KB, for three or four workgroups per CU.  Against the normalised harmonics
// with eight FMAs per weight and the weights read from LDS: dipoles at order 26,
// 200,000 + 180,000 points, P2L 8.5 -> 5.6 ms; 250,000 Plummer points 6.8 -> 4.2
// ms; 1M + 1M uniform, P2M 1.41 -> 1.19 ms (FP32 1.00 -> 0.86 ms).  Measured and
// not kept: two tiles, one built while the other is summed, in 512-thread
// workgroups (5.6 -> 7.6 ms).
// ---------------------------------------------------------------------------
constexpr int kFormBatch = 64;  // sources whose scalars are computed at a time
constexpr int kFormSc = 5;      // scalars per source
constexpr int kFormRanges = 32; // most ranges of orders

// The ranges of orders of one launch: range r writes orders lo[r]..hi[r] and
// builds the columns from[r]..to[r].
struct FormRanges {
  int n = 0;
  short lo[kFormRanges], hi[kFormRanges], from[kFormRanges], to[kFormRanges];
};

// Start of the column after one at `base` of `len` entries, that column being
// the k-th: at a multiple of 8 entries plus k (the 32 LDS banks hold 8 complex
// FP64 values).
__host__ __device__ inline int form_next_col(int base, int len, int k) {
  int c = base + len;
  while ((c & 7) != (k & 7)) c++;
  return c;
}
// entries of one source's row of columns from..to, degrees up to pt
__host__ __device__ inline int form_row(int pt, int from, int to) {
  int c = 0;
  for (int a = from; a <= to; a++) c = form_next_col(c, pt + 1 - a, a + 1 - from);
  return c;
}
// the ranges for degrees up to pt: as many orders each as `cap` entries hold
inline FormRanges form_ranges(int pt, bool dip, int cap) {
  FormRanges R;
  const int halo = dip ? 1 : 0;
  for (int lo = 0; lo <= pt; R.n++) {
    if (R.n == kFormRanges) { R.n = 0; break; }
    const int from = lo - halo < 0 ? 0 : lo - halo;
    int to = from, e = pt + 1 - from;
    while (to < pt && (e + pt - to <= cap || to < lo + halo)) { to++; e += pt + 1 - to; }
    const int hi = to == pt ? pt : to - halo;
    if (e > cap) { R.n = 0; break; }
    R.lo[R.n] = (short)lo; R.hi[R.n] = (short)hi; R.from[R.n] = (short)from; R.to[R.n] = (short)to;
    lo = hi + 1;
  }
  return R;
}
// LDS of k_form2 in T ahead of the tile: recurrence factors of a row, column
// starts, the batch's scalars
__host__ __device__ inline int form_head(int pt, int row) {
  return (row + 8 + 3) / 4 * 4 + (pt + 2 + 3) / 4 * 4 + kFormBatch * kFormSc;
}

// One complex table entry as a single LDS store (16 bytes for double, 8 for
// float; tile rows keep entries at that alignment)
template <typename T>
__device__ __forceinline__ void cst_vec(T* p, int k, C2<T> v) {
  using V2 = typename std::conditional<std::is_same<T, double>::value, double2, float2>::type;
  V2 t;
  t.x = v.re;
  t.y = v.im;
  *reinterpret_cast<V2*>(p + 2 * k) = t;
}

// `region`: the tile's size in T; it also holds one weight's sums at the end
template <typename T, bool IRREG, bool CHG, bool DIP, int GS, int ITEMS>
__global__ __launch_bounds__(256) void k_form2(DevPlan P, const double* __restrict__ fac,
                                               const double* __restrict__ spos, const T* __restrict__ str,
                                               FormRanges R, int region, T* __restrict__ expn) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  using V2 = typename std::conditional<std::is_same<T, double>::value, double2, float2>::type;
  const int p = P.p, K = P.K;
  const int pt = IRREG ? p + 1 : p;
  const FacLayout L(p);
  const int tid = threadIdx.x, rg = blockIdx.y;
  const int lo = R.lo[rg], hi = R.hi[rg], from = R.from[rg], ncol = R.to[rg] - from + 1;
  T* smem = reinterpret_cast<T*>(smem_raw);
  T* beta = smem;
  const int row = form_row(pt, from, from + ncol - 1);
  int* cb = reinterpret_cast<int*>(smem + (row + 8 + 3) / 4 * 4);
  T* scs = smem + form_head(pt, row) - kFormBatch * kFormSc;
  T* tab = smem + form_head(pt, row);
  const int ts = min(kFormBatch, region / (2 * row));
  if (tid == 0) {
    int c = 0;
    for (int k = 0; k < ncol; k++) {
      cb[k] = c;
      c = form_next_col(c, pt + 1 - from - k, k + 1);
    }
  }
  __syncthreads();
  constexpr int G = 256 / GS;
  const int grp = __builtin_amdgcn_readfirstlane(tid / GS), lt = tid - grp * GS;
  int ent[ITEMS], adr[ITEMS];  // owned entries: n << 8 | a (or -1), and their place in a row
#pragma unroll
  for (int q = 0; q < ITEMS; q++) {
    int k = 0, r = lt + q * GS;
    while (k < ncol && r >= pt + 1 - from - k) { r -= pt + 1 - from - k; k++; }
    ent[q] = -1;
    adr[q] = 0;
    if (k < ncol) {
      const int a = from + k, n = a + r;
      ent[q] = n << 8 | a;
      adr[q] = cb[k] + r;
      if (grp == 0) beta[adr[q]] = (T)fac[L.BT + hidx(n, a)];
    }
  }
  const int b = IRREG ? P.p2l_boxes[blockIdx.x] : P.p2m_boxes[blockIdx.x];
  const double ihd = P.inv_side[P.level[b]];
  const T ih = (T)ihd;
  const double cx = P.center[3 * b], cy = P.center[3 * b + 1], cz = P.center[3 * b + 2];
  constexpr int NW = (CHG ? 1 : 0) + (DIP ? 3 : 0), W0 = CHG ? 0 : 1;  // weights, first of q, x, y, z
  T acc[ITEMS][NW][4];
#pragma unroll
  for (int q = 0; q < ITEMS; q++)
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[q][w][e] = T(0);
  const int jbeg = IRREG ? P.l4_off[b] : 0, jend = IRREG ? P.l4_off[b + 1] : 1;
  for (int jj = jbeg; jj < jend; jj++) {
    const int j = IRREG ? P.l4_idx[jj] : b;
    const int s0 = P.isrc[j], sn = P.nsrc[j];
    for (int t0 = 0; t0 < sn; t0 += kFormBatch) {
      const int bn = min(kFormBatch, sn - t0);
      // (the batch before is done with: a barrier ended its last tile)
      if (tid < bn) {
        const double* x = spos + 4 * (size_t)(s0 + t0 + tid);
        const T ux = (T)((x[0] - cx) * ihd), uy = (T)((x[1] - cy) * ihd), uz = (T)((x[2] - cz) * ihd);
        const T r2 = ux * ux + uy * uy + uz * uz;
        T* sc = scs + kFormSc * tid;
        if (IRREG) {
          const T ir2 = T(1) / r2;
          sc[0] = -ux * ir2; sc[1] = -uy * ir2; sc[2] = uz * ir2; sc[3] = ir2; sc[4] = sqrt(ir2);
        } else {
          sc[0] = -ux; sc[1] = -uy; sc[2] = uz; sc[3] = r2; sc[4] = T(1);
        }
      }
      __syncthreads();
      for (int u0 = 0; u0 < bn; u0 += ts) {
        const int tn = min(ts, bn - u0);
        // columns: task = source * ncol + (a - from)
        for (int task = tid; task < tn * ncol; task += 256) {
          const int s = task / ncol, k0 = task - s * ncol, a = from + k0;
          const T* sc = scs + kFormSc * (u0 + s);
          C2<T> w = {sc[0], sc[1]}, r = {sc[4], T(0)}, r0 = {T(0), T(0)};
          const T zz = sc[2], rho = sc[3];
          T* out = tab + 2 * (size_t)(s * row + cb[k0]);
          const T* bt = beta + cb[k0] + 1;
          const int len = pt + 1 - a;
          // four recurrence factors at a time, read ahead of the four steps
          // that use them (the last reads run past the column's, unused)
          T bc[4], bn4[4];
#pragma unroll
          for (int u = 0; u < 4; u++) bc[u] = bt[u];
          for (int e = a; e; e >>= 1) {
            if (e & 1) r = cmul(r, w);
            w = cmul(w, w);
          }
          auto step = [&](int k, T bk) {
            cst_vec(out, k, r);
            const T br = bk * rho;
            C2<T> rn;
            rn.re = fma(zz, r.re, -(br * r0.re));
            rn.im = fma(zz, r.im, -(br * r0.im));
            r0 = r;
            r = rn;
          };
          int k = 0;
          for (; k + 4 <= len; k += 4) {
#pragma unroll
            for (int u = 0; u < 4; u++) bn4[u] = bt[k + 4 + u];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 4; u++) step(k + u, bc[u]);
#pragma unroll
            for (int u = 0; u < 4; u++) bc[u] = bn4[u];
          }
#pragma unroll
          for (int u = 0; u < 3; u++)
            if (k + u < len) step(k + u, bc[u]);
        }
        __syncthreads();
        // sums, four sources' weights at a time (sources past the tile's end
        // read its last weights again, unused)
        for (int s = grp; s < tn; s += 4 * G) {
          T wr[4][NW], wi[4][NW];
#pragma unroll
          for (int v = 0; v < 4; v++) {
            const int sv = s0 + t0 + u0 + min(s + v * G, tn - 1);
            const T* __restrict__ wv = str + 8 * (size_t)(unsigned)__builtin_amdgcn_readfirstlane(sv);
#pragma unroll
            for (int w = 0; w < NW; w++) { wr[v][w] = wv[2 * (W0 + w)]; wi[v][w] = wv[2 * (W0 + w) + 1]; }
          }
#pragma unroll
          for (int v = 0; v < 4; v++) {
            if (s + v * G >= tn) break;
#pragma unroll
            for (int q = 0; q < ITEMS; q++) {
              const V2 hv = *reinterpret_cast<const V2*>(tab + 2 * (size_t)((s + v * G) * row + adr[q]));
#pragma unroll
              for (int w = 0; w < NW; w++) {
                acc[q][w][0] = fma(wr[v][w], hv.x, acc[q][w][0]);
                acc[q][w][1] = fma(wi[v][w], hv.y, acc[q][w][1]);
                acc[q][w][2] = fma(wr[v][w], hv.y, acc[q][w][2]);
                acc[q][w][3] = fma(wi[v][w], hv.x, acc[q][w][3]);
              }
            }
          }
        }
        __syncthreads();
      }
    }
  }
  // one weight at a time: its sums S(n, +a), S(n, -a) to LDS (four values at
  // an entry's place), then into the owners' coefficients (n, a) and (n, -a)
  T co[ITEMS][4], cg[ITEMS][4];
#pragma unroll
  for (int q = 0; q < ITEMS; q++)
#pragma unroll
    for (int e = 0; e < 4; e++) co[q][e] = cg[q][e] = T(0);
  auto sget = [&](int n, int m, T& re, T& im) {
    const int a = m < 0 ? -m : m;
    re = im = T(0);
    if (a > n) return;
    const T* o = tab + 4 * (cb[a - from] + n - a) + (m < 0 ? 2 : 0);
    re = o[0];
    im = o[1];
  };
#pragma unroll
  for (int w = 0; w < NW; w++) {
    for (int g = 0; g < G; g++) {
      if (grp == g) {
#pragma unroll
        for (int q = 0; q < ITEMS; q++) {
          if (ent[q] < 0) continue;
          const T gn = (T)fac[L.GN + hidx(ent[q] >> 8, ent[q] & 255)];
          const T* A = acc[q][w];
          const T v[4] = {gn * (A[0] - A[1]), gn * (A[2] + A[3]), gn * (A[0] + A[1]), gn * (A[3] - A[2])};
          T* o = tab + 4 * adr[q];
#pragma unroll
          for (int e = 0; e < 4; e++) o[e] = g == 0 ? v[e] : o[e] + v[e];
        }
      }
      __syncthreads();
    }
    const int c = W0 + w;  // 0: q, 1..3: v_x, v_y, v_z
    if (grp == 0) {
#pragma unroll
      for (int q = 0; q < ITEMS; q++) {
        const int n = ent[q] >> 8, a = ent[q] & 255;
        if (ent[q] < 0 || a < lo || a > hi || n > p) continue;
#pragma unroll
        for (int sg = 0; sg < 2; sg++) {
          const int km = sg ? a : -a;  // coefficient m = -km
          T re, im;
          if (c == 0) {
            sget(n, km, re, im);
            co[q][2 * sg] = re;
            co[q][2 * sg + 1] = im;
          } else if (IRREG || n >= 1) {
            const int nn = IRREG ? n + 1 : n - 1;
            T &gr = cg[q][2 * sg], &gi = cg[q][2 * sg + 1];
            if (c == 3) {
              const T fa = (T)fac[(IRREG ? L.AS : L.AR) + eidx(n, km)];
              sget(nn, km, re, im);
              gr += fa * re;
              gi += fa * im;
            } else {
              // (v_x - i v_y)/2 with the order one up, (v_x + i v_y)/2 one down
              const T fb = (T)fac[(IRREG ? L.BS : L.BR) + eidx(n, km)] * T(0.5);
              const T fc = (T)fac[(IRREG ? L.CS : L.CR) + eidx(n, km)] * T(0.5);
              T dr, di;
              sget(nn, km + 1, re, im);
              sget(nn, km - 1, dr, di);
              if (c == 1) {
                gr += fb * re + fc * dr;
                gi += fb * im + fc * di;
              } else {
                gr += fb * im - fc * di;
                gi += fc * dr - fb * re;
              }
            }
          }
        }
      }
    }
    __syncthreads();
  }
  if (grp != 0) return;
  const T sc = IRREG ? ih : T(1);
  T* out = expn + 2 * (size_t)b * K;
#pragma unroll
  for (int q = 0; q < ITEMS; q++) {
    const int n = ent[q] >> 8, a = ent[q] & 255;
    if (ent[q] < 0 || a < lo || a > hi || n > p) continue;
#pragma unroll
    for (int sg = 0; sg < 2; sg++) {
      if (sg && a == 0) continue;
      T* o = out + 2 * eidx(n, sg ? -a : a);
      o[0] += (co[q][2 * sg] + cg[q][2 * sg] * ih) * sc;
      o[1] += (co[q][2 * sg + 1] + cg[q][2 * sg + 1] * ih) * sc;
    }
  }
}

// ---------------------------------------------------------------------------
// L2P (src/laprouts3d.f:2772 l3dtaevalall_trunc) and M2P (list 3,
// src/laprouts3d.f:2432 l3dmpevalall_trunc) from packed expansions.  The
// potential and the three gradient sums are
//   pot = sum E H, d/dz = sum Gz H, (d/dx + i d/dy) = sum Gu H, (d/dx - i d/dy) = sum Gd H
// over the harmonics H = R of degree n <= p with
//   Gz(n,m) = AR(n+1,m) L(n+1,m), Gu = BR(n+1,m-1) L(n+1,m-1), Gd = CR(n+1,m+1) L(n+1,m+1)
// for a local L, and H = S of degree n <= p+1 with
//   Gz(n,m) = AS(n-1,m) M(n-1,m), Gu = BS(n-1,m-1) M(n-1,m-1), Gd = CS(n-1,m+1) M(n-1,m+1)
// for a multipole M (zero where an index is outside).  An entry (n, a >= 0) of
// the pack holds, for each X of E, Gz, Gu, Gd and c+- = X(n, +-a) (c- = 0 for
// a = 0), the four reals that take the harmonic h = H_n^a to c+ h + c- conj(h),
//   re: (c+ + c-)_re h_re - (c+ - c-)_im h_im,  im: (c+ + c-)_im h_re + (c+ - c-)_re h_im,
// times the scale of FacLayout's recurrence: kPackEntry values.  Entries are in
// the order of the walk (column a, then n = a..pd); that recurrence's factors
// for degree n + 1 stand once, in the same order, ahead of the packs (with them
// in the entries and the columns padded to an even count the packs took 17%
// more at order 26, 50% at order 2, a fixed workspace held fewer points, and the
// scalar loads straddled their 64-byte lines).  The walk reads both with scalar
// loads, one entry ahead, and pays 16 FMAs and the recurrence's 5 operations per
// entry and point (32 and 9 before, the harmonics normalised and c+ h, c- conj(h)
// taken apart).  VALU bound: 400,000 clustered points at order 39, M2P 11.4 ms
// with normalised harmonics, 8.2 with the factors in the entries, 5.8 so;
// 200,000 + 180,000 at order 26 7.8, 5.7 and 4.1 ms; 1M + 1M uniform, L2P 1.59,
// 1.22 and 1.06 ms (FP32 1.22, 0.74 and 0.70).
// ---------------------------------------------------------------------------
constexpr int kPackEntry = 16;
__host__ __device__ inline int pack_entries(int pd) { return (pd + 1) * (pd + 2) / 2; }
// values ahead of the packs: the factors and one read ahead of the last
__host__ __device__ inline int pack_head(int pd) { return (pack_entries(pd) + 1 + 15) / 16 * 16; }
// values of n packs, with the entry that the walk reads past the last
inline size_t pack_values(int pd, size_t n) { return pack_head(pd) + kPackEntry * ((size_t)pack_entries(pd) * n + 1); }

// coefficients c+- of E, Gz, Gu, Gd at (n, a), as (re, im) pairs, to an entry
template <typename T>
__device__ __forceinline__ void pack_store(T* __restrict__ o, const T (&v)[16], T g) {
#pragma unroll
  for (int x = 0; x < 4; x++) {
    o[4 * x] = g * (v[4 * x] + v[4 * x + 2]);
    o[4 * x + 1] = -g * (v[4 * x + 1] - v[4 * x + 3]);
    o[4 * x + 2] = g * (v[4 * x + 1] + v[4 * x + 3]);
    o[4 * x + 3] = g * (v[4 * x] - v[4 * x + 2]);
  }
}

template <typename T>
__global__ void k_l2p_pack(DevPlan P, const double* __restrict__ fac, const T* __restrict__ lo,
                           T* __restrict__ pack) {
  const int p = P.p, K = P.K;
  const int NE = pack_entries(p);
  FacLayout L(p);
  const size_t total = (size_t)P.n_l2p * NE;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(t / NE);
    const int w = (int)(t - (size_t)i * NE);
    int a = 0, r = w;
    while (r >= p + 1 - a) { r -= p + 1 - a; a++; }
    const int n = a + r;
    if (i == 0) pack[w] = (T)fac[L.BT + hidx(n + 1, a)];
    const T* E = lo + 2 * (size_t)P.l2p_boxes[i] * K;
    T v[16];
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = T(0);
    v[0] = E[2 * eidx(n, a)];
    v[1] = E[2 * eidx(n, a) + 1];
    if (a > 0) { v[2] = E[2 * eidx(n, -a)]; v[3] = E[2 * eidx(n, -a) + 1]; }
    if (n + 1 <= p) {
      const int n1 = n + 1;
      for (int sgn = 0; sgn < (a > 0 ? 2 : 1); sgn++) {
        const int m = sgn ? -a : a;
        const T fz = (T)fac[L.AR + eidx(n1, m)], fu = (T)fac[L.BR + eidx(n1, m - 1)], fd = (T)fac[L.CR + eidx(n1, m + 1)];
        v[4 + 2 * sgn] = fz * E[2 * eidx(n1, m)];
        v[5 + 2 * sgn] = fz * E[2 * eidx(n1, m) + 1];
        v[8 + 2 * sgn] = fu * E[2 * eidx(n1, m - 1)];
        v[9 + 2 * sgn] = fu * E[2 * eidx(n1, m - 1) + 1];
        v[12 + 2 * sgn] = fd * E[2 * eidx(n1, m + 1)];
        v[13 + 2 * sgn] = fd * E[2 * eidx(n1, m + 1) + 1];
      }
    }
    pack_store(pack + pack_head(p) + kPackEntry * t, v, (T)fac[L.GN + hidx(n, a)]);
  }
}

// One pack entry and its factor in scalar registers
template <typename T, bool GRAD>
struct PackRec {
  T c[GRAD ? 16 : 4], b;
  __device__ __forceinline__ void load(const T* __restrict__ o, const T* __restrict__ beta) {
#pragma unroll
    for (int e = 0; e < (GRAD ? 16 : 4); e++) c[e] = o[e];
    b = *beta;
  }
};

// The walk over one pack at a point: w, zz, rho of the recurrence, h00 its
// first value, beta its factors; out (pot, d/dz, U, D) is added to.  Two entries
// at a time, a column of odd length ending on one.  Reads one entry past the
// pack's last.
template <typename T, bool GRAD>
__device__ __forceinline__ void pack_walk(const T* __restrict__ pk, const T* __restrict__ beta, int pd, C2<T> w, T zz,
                                          T rho, T h00, C2<T> (&out)[4]) {
  PackRec<T, GRAD> ra, rb;
  auto arrived = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
  };
  C2<T> hmm = {h00, T(0)}, h, hp;
  auto step = [&](const PackRec<T, GRAD>& r) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < (GRAD ? 4 : 1); x++) {
      out[x].re = fma(r.c[4 * x], h.re, fma(r.c[4 * x + 1], h.im, out[x].re));
      out[x].im = fma(r.c[4 * x + 2], h.re, fma(r.c[4 * x + 3], h.im, out[x].im));
    }
    const T br = r.b * rho;
    C2<T> hn;
    hn.re = fma(zz, h.re, -(br * hp.re));
    hn.im = fma(zz, h.im, -(br * hp.im));
    hp = h;
    h = hn;
  };
  ra.load(pk, beta);
  int e = 0;
  for (int a = 0; a <= pd; a++) {
    if (a > 0) hmm = cmul(w, hmm);
    h = hmm;
    hp = {T(0), T(0)};
    const int end = e + pd + 1 - a;
    for (; e + 1 < end; e += 2) {
      const unsigned u = (unsigned)__builtin_amdgcn_readfirstlane(e);
      const T* __restrict__ o = pk + (size_t)kPackEntry * u;
      const T* __restrict__ bt = beta + u;
      arrived();
      rb.load(o + kPackEntry, bt + 1);
      step(ra);
      arrived();
      ra.load(o + 2 * kPackEntry, bt + 2);
      step(rb);
    }
    if (e < end) {
      const unsigned u = (unsigned)__builtin_amdgcn_readfirstlane(e);
      arrived();
      rb.load(pk + (size_t)kPackEntry * (u + 1), beta + u + 1);
      step(ra);
      arrived();
      ra = rb;
      e++;
    }
  }
}

// One wave per L2P work item (box, kind, first point); the walk over the pack
// is wave uniform.
template <typename T>
__global__ __launch_bounds__(256) void k_l2p2(DevPlan P, const T* __restrict__ pack,
                                               const double* __restrict__ spos, const double* __restrict__ tpos,
                                               int wpot0, int wfld0, int wpot1, int wfld1,
                                               double* __restrict__ pot0, double* __restrict__ fld0,
                                               double* __restrict__ pot1, double* __restrict__ fld1) {
  const int p = P.p;
  // one work item (64 points) per wave
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
  if (w >= P.n_l2pi) return;
  const int ib = P.l2p_items[3 * w], kind = P.l2p_items[3 * w + 1], start = P.l2p_items[3 * w + 2];
  if (ib < 0) return;   // padding item
  const int b = P.l2p_boxes[ib];
  const T* pk = pack + pack_head(p) + (size_t)ib * pack_entries(p) * kPackEntry;
  const T ih = (T)P.inv_side[P.level[b]];
  const double cx = P.center[3 * b], cy = P.center[3 * b + 1], cz = P.center[3 * b + 2];
  const int wp = kind ? wpot1 : wpot0, wf = kind ? wfld1 : wfld0;
  const int n0 = kind ? P.itrg[b] : P.isrc[b];
  const int nn = kind ? P.ntrg[b] : P.nsrc[b];
  const int i = start + (int)(threadIdx.x & 63);
  const bool active = i < nn;
  double x = cx, y = cy, z = cz;
  if (active) {
    const double* q = (kind ? tpos : spos) + 4 * (size_t)(n0 + i);
    x = q[0]; y = q[1]; z = q[2];
  }
  const T ux = (T)((x - cx) * (double)ih), uy = (T)((y - cy) * (double)ih), uz = (T)((z - cz) * (double)ih);
  const T r2 = ux * ux + uy * uy + uz * uz;
  C2<T> out[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
  if (wf)
    pack_walk<T, true>(pk, pack, p, C2<T>{-ux, -uy}, uz, r2, T(1), out);
  else
    pack_walk<T, false>(pk, pack, p, C2<T>{-ux, -uy}, uz, r2, T(1), out);
  if (!active) return;
  const C2<T> pv = out[0], gz = out[1], gu = out[2], gd = out[3];
  const size_t id = (size_t)(n0 + i);
  double* po = kind ? pot1 : pot0;
  double* fo = kind ? fld1 : fld0;
  if (wp) { po[2 * id] += pv.re; po[2 * id + 1] += pv.im; }
  if (wf) {
    // fld = -grad: d/dx = (U+D)/2, d/dy = (U-D)/(2i), d/dz; the gradient in x carries 1/h
    const C2<T> dx = {T(0.5) * (gu.re + gd.re), T(0.5) * (gu.im + gd.im)};
    const C2<T> dy = {T(0.5) * (gu.im - gd.im), -T(0.5) * (gu.re - gd.re)};
    fo[6 * id + 0] -= dx.re * ih; fo[6 * id + 1] -= dx.im * ih;
    fo[6 * id + 2] -= dy.re * ih; fo[6 * id + 3] -= dy.im * ih;
    fo[6 * id + 4] -= gz.re * ih; fo[6 * id + 5] -= gz.im * ih;
  }
}

template <typename T>
__global__ void k_m2p_pack(DevPlan P, const double* __restrict__ fac, const T* __restrict__ mp,
                           const int* __restrict__ boxes, const int* __restrict__ offs, int nbox, int grad,
                           T* __restrict__ pack) {
  const int p = P.p, K = P.K;
  const int pd = grad ? p + 1 : p;
  const int NE = pack_entries(pd);
  FacLayout L(p);
  const size_t total = (size_t)nbox * NE;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(t / NE), w = (int)(t - (size_t)i * NE);
    int a = 0, r = w;
    while (r >= pd + 1 - a) { r -= pd + 1 - a; a++; }
    const int n = a + r;
    if (i == 0) pack[w] = (T)fac[L.BT + hidx(n + 1, a)];
    const T* E = mp + 2 * (size_t)boxes[i] * K;
    auto ef = [&](int off, int n1, int m1, int e) -> T {  // factor * E(n1, m1), zero outside
      if (n1 < 0 || m1 > n1 || m1 < -n1) return T(0);
      return (T)fac[off + eidx(n1, m1)] * E[2 * eidx(n1, m1) + e];
    };
    T v[16];
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = T(0);
    if (n <= p) {
      v[0] = E[2 * eidx(n, a)];
      v[1] = E[2 * eidx(n, a) + 1];
      if (a > 0) { v[2] = E[2 * eidx(n, -a)]; v[3] = E[2 * eidx(n, -a) + 1]; }
    }
    if (grad && n >= 1) {
      const int n1 = n - 1;
      for (int sgn = 0; sgn < (a > 0 ? 2 : 1); sgn++) {
        const int m = sgn ? -a : a;
        for (int e = 0; e < 2; e++) {
          v[4 + 2 * sgn + e] = ef(L.AS, n1, m, e);
          v[8 + 2 * sgn + e] = ef(L.BS, n1, m - 1, e);
          v[12 + 2 * sgn + e] = ef(L.CS, n1, m + 1, e);
        }
      }
    }
    pack_store(pack + pack_head(pd) + kPackEntry * ((size_t)offs[i] + w), v, (T)fac[L.GN + hidx(n, a)]);
  }
}

// M2P: one wave per 64 points of a box and slice of its list 3, the sums
// scaled by 1/h (potential) and 1/h^2 (gradient) of each source box; the
// slice's sums go to `partial` and k_slice_reduce adds the slices in order.
// items: 5 ints per wave (box, kind, first point, first and end position in
// list 3); slot[j]: the pack offset (in entries) of source box j
template <typename T>
__global__ __launch_bounds__(256) void k_m2p_eval(DevPlan P, const T* __restrict__ pack,
                                                  const int* __restrict__ slot, const int* __restrict__ items, int nitems,
                                                  int grad, const double* __restrict__ spos,
                                                  const double* __restrict__ tpos, double* __restrict__ partial) {
  const int pd = grad ? P.p + 1 : P.p;
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
  if (w >= nitems) return;
  const int lane = (int)(threadIdx.x & 63);
  const int* it = items + 5 * w;
  const int b = it[0], kind = it[1], start = it[2], jbeg = it[3], jend = it[4];
  const int n0 = kind ? P.itrg[b] : P.isrc[b];
  const int nn = kind ? P.ntrg[b] : P.nsrc[b];
  const int i = start + lane;
  const bool active = i < nn;
  double x = 0.0, y = 0.0, z = 0.0;
  if (active) {
    const double* q = (kind ? tpos : spos) + 4 * (size_t)(n0 + i);
    x = q[0]; y = q[1]; z = q[2];
  }
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int jj = jbeg; jj < jend; jj++) {
    const int j = P.l3_idx[jj];
    if (P.nsrc[j] == 0) continue;
    const double ihd = P.inv_side[P.level[j]];
    const T ih = (T)ihd;
    // inactive lanes evaluate at a harmless point and are not written
    const T ux = active ? (T)((x - P.center[3 * j]) * ihd) : T(1);
    const T uy = active ? (T)((y - P.center[3 * j + 1]) * ihd) : T(1);
    const T uz = active ? (T)((z - P.center[3 * j + 2]) * ihd) : T(1);
    const T r2 = ux * ux + uy * uy + uz * uz;
    const T ir2 = T(1) / r2, ir = sqrt(ir2);
    C2<T> out[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
    const T* c = pack + pack_head(pd) + kPackEntry * (size_t)slot[j];
    if (grad)
      pack_walk<T, true>(c, pack, pd, C2<T>{-ux * ir2, -uy * ir2}, uz * ir2, ir2, ir, out);
    else
      pack_walk<T, false>(c, pack, pd, C2<T>{-ux * ir2, -uy * ir2}, uz * ir2, ir2, ir, out);
    // pot = sum M S(u)/h ; the gradient w.r.t. x adds another 1/h
    const T sg = ih * ih;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const T sc = v == 0 ? ih : sg;
      acc[2 * v] += (double)(out[v].re * sc);
      acc[2 * v + 1] += (double)(out[v].im * sc);
    }
  }
  double* o = partial + 8 * ((size_t)w * 64 + lane);
#pragma unroll
  for (int e = 0; e < 8; e++) o[e] = acc[e];
}

// ---------------------------------------------------------------------------
// Point-and-shoot translation of one expansion inside a workgroup:
//   A = in * e^{i m phi}           (n <= pin)
//   B = rotate(A)                   (rotation class `rc`)
//   A = zshift(B)  with table Z    (n <= pin -> l <= pout)
//   B = rotate back(A)
//   out += B * e^{-i m phi} * scale
// src/l3dtrans.f:223 (M2M), :868 (M2L), :1676 (L2L) do the same sequence.
// ZMODE 0: Z[m][out][in] ; the same dense (p+1)^3 layout for every shift.
// ---------------------------------------------------------------------------
template <typename T>
__device__ void zshift_block(const double* Z, int p, int pin, int pout, const T* in, T* out) {
  // orders m and -m share the row Z[|m|][l][.]: one thread produces both
  const int Kh = (pout + 1) * (pout + 2) / 2;
  const int P1 = p + 1;
  for (int k = threadIdx.x; k < Kh; k += blockDim.x) {
    int l = (int)((sqrtf(8.0f * k + 1.0f) - 1.0f) * 0.5f);
    while (l * (l + 1) / 2 > k) l--;
    while ((l + 1) * (l + 2) / 2 <= k) l++;
    const int am = k - l * (l + 1) / 2;
    const double* z = Z + ((size_t)am * P1 + l) * P1;
    T pr = 0, pi = 0, qr = 0, qi = 0;
    for (int n = am; n <= pin; n++) {
      const T c = (T)z[n];
      pr += c * in[2 * eidx(n, am)];
      pi += c * in[2 * eidx(n, am) + 1];
      qr += c * in[2 * eidx(n, -am)];
      qi += c * in[2 * eidx(n, -am) + 1];
    }
    out[2 * eidx(l, am)] = pr;
    out[2 * eidx(l, am) + 1] = pi;
    if (am > 0) {
      out[2 * eidx(l, -am)] = qr;
      out[2 * eidx(l, -am) + 1] = qi;
    }
  }
}

template <typename T>
__device__ void point_and_shoot(const DevTables& Tb, int rc, const double* phase, const double* Z,
                                int pin, int pout, const T* in, T* out, T scale, T* A, T* B) {
  const int pm = pin > pout ? pin : pout;
  const int Ki = (pin + 1) * (pin + 1);
  for (int k = threadIdx.x; k < (pm + 1) * (pm + 1); k += blockDim.x) {
    if (k < Ki) {
      int n = (int)sqrtf((float)k);
      while (n * n > k) n--;
      while ((n + 1) * (n + 1) <= k) n++;
      int m = k - n * n - n, am = m < 0 ? -m : m;
      T er = (T)phase[2 * am], ei = (T)phase[2 * am + 1];
      if (m < 0) ei = -ei;
      T xr = in[2 * k], xi = in[2 * k + 1];
      A[2 * k] = xr * er - xi * ei;
      A[2 * k + 1] = xr * ei + xi * er;
    } else {
      A[2 * k] = 0;
      A[2 * k + 1] = 0;
    }
  }
  __syncthreads();
  rotate_block<T>(Tb, rc, pin, A, B, false);
  __syncthreads();
  zshift_block<T>(Z, Tb.p, pin, pout, B, A);
  __syncthreads();
  rotate_block<T>(Tb, rc, pout, A, B, true);
  __syncthreads();
  const int Ko = (pout + 1) * (pout + 1);
  for (int k = threadIdx.x; k < Ko; k += blockDim.x) {
    int n = (int)sqrtf((float)k);
    while (n * n > k) n--;
    while ((n + 1) * (n + 1) <= k) n++;
    int m = k - n * n - n, am = m < 0 ? -m : m;
    T er = (T)phase[2 * am], ei = -(T)phase[2 * am + 1];  // e^{-i m phi}
    if (m < 0) ei = -ei;
    T xr = B[2 * k], xi = B[2 * k + 1];
    out[2 * k] += (xr * er - xi * ei) * scale;
    out[2 * k + 1] += (xr * ei + xi * er) * scale;
  }
  __syncthreads();
}

// M2M into the parents of one level (src/lfmm3drouts.f:195-258), one workgroup
// per child (blockIdx.y): the translated expansion goes to the child's local,
// which is still zero, and k_child_sum adds the children's in order.  A level of
// a deep tree has few parents, and what a translation costs there is the latency
// of its four stages: with one workgroup per parent taking its eight children in
// turn, 400,000 clustered points (p = 39) spent 3.5 ms here and 3.4 in L2L, now
// 1.0 and 0.7; 20,000 points 0.10 ms in each, now 0.03 and 0.02.
template <typename T>
__global__ void k_m2m(DevPlan P, DevTables Tb, int first, const T* __restrict__ mp, T* __restrict__ lo) {
  extern __shared__ unsigned char smem_raw[];
  T* A = reinterpret_cast<T*>(smem_raw);
  T* B = A + 2 * P.K;
  const int b = P.m2m_boxes[first + blockIdx.x], c = blockIdx.y;
  const int p = P.p;
  if (c >= P.nchild[b]) return;
  const int ch = P.child[8 * b + c];
  if (P.nsrc[ch] == 0) return;
  // octant of the child relative to the parent
  const int o = (P.ijk[3 * ch] & 1 ? 0 : 1) | (P.ijk[3 * ch + 1] & 1 ? 0 : 2) | (P.ijk[3 * ch + 2] & 1 ? 0 : 4);
  const double* ph = Tb.oct_phase + (size_t)(o * 2 + 0) * 2 * (p + 1);
  point_and_shoot<T>(Tb, Tb.oct_rot[o * 2 + 0], ph, Tb.z_m2m, p, p, mp + 2 * (size_t)ch * P.K,
                     lo + 2 * (size_t)ch * P.K, T(1), A, B);
}

// L2L for the parents of one level (src/lfmm3drouts.f:498-558), one workgroup
// per child
template <typename T>
__global__ void k_l2l(DevPlan P, DevTables Tb, int first, T* __restrict__ lo) {
  extern __shared__ unsigned char smem_raw[];
  T* A = reinterpret_cast<T*>(smem_raw);
  T* B = A + 2 * P.K;
  const int b = P.l2l_boxes[first + blockIdx.x], c = blockIdx.y;
  const int p = P.p;
  if (c >= P.nchild[b]) return;
  const int ch = P.child[8 * b + c];
  const int o = (P.ijk[3 * ch] & 1 ? 0 : 1) | (P.ijk[3 * ch + 1] & 1 ? 0 : 2) | (P.ijk[3 * ch + 2] & 1 ? 0 : 4);
  const double* ph = Tb.oct_phase + (size_t)(o * 2 + 1) * 2 * (p + 1);
  point_and_shoot<T>(Tb, Tb.oct_rot[o * 2 + 1], ph, Tb.z_l2l, p, p, lo + 2 * (size_t)b * P.K,
                     lo + 2 * (size_t)ch * P.K, T(1), A, B);
}

// M2L over the (pruned) list 2 of each target box (src/lfmm3drouts.f:347-483).
// The target's local accumulates in LDS (the third 2K block) and is added to
// memory once, so HBM sees one read per source multipole and one
// read-modify-write per target.  Without LDS room (LDSACC = false, high
// orders) the local is accumulated in memory directly.
template <typename T, bool LDSACC>
__global__ void k_m2l(DevPlan P, DevTables Tb, const T* __restrict__ mp, T* __restrict__ lo) {
  extern __shared__ unsigned char smem_raw[];
  T* A = reinterpret_cast<T*>(smem_raw);
  T* B = A + 2 * P.K;
  const int b = P.m2l_boxes[blockIdx.x];
  T* acc = LDSACC ? B + 2 * P.K : lo + 2 * (size_t)b * P.K;
  const int p = P.p;
  const T ih = (T)P.inv_side[P.level[b]];
  const size_t zsz = (size_t)(p + 1) * (p + 1) * (p + 1);
  if (LDSACC)
    for (int k = threadIdx.x; k < 2 * P.K; k += blockDim.x) acc[k] = T(0);
  __syncthreads();
  for (int jj = P.l2_off[b]; jj < P.l2_off[b + 1]; jj++) {
    const int j = P.l2_idx[jj];
    int di = P.ijk[3 * j] - P.ijk[3 * b] + 3, dj = P.ijk[3 * j + 1] - P.ijk[3 * b + 1] + 3,
        dk = P.ijk[3 * j + 2] - P.ijk[3 * b + 2] + 3;
    int code = (di * 7 + dj) * 7 + dk;
    int pt = Tb.off_ptrunc[code];
    point_and_shoot<T>(Tb, Tb.off_rot[code], Tb.off_phase + (size_t)code * 2 * (p + 1),
                       Tb.z_m2l + (size_t)Tb.off_dist[code] * zsz, pt, pt,
                       mp + 2 * (size_t)j * P.K, acc, ih, A, B);
  }
  if (LDSACC) {
    T* out = lo + 2 * (size_t)b * P.K;
    for (int k = threadIdx.x; k < 2 * P.K; k += blockDim.x) out[k] += acc[k];
  }
}

// ---------------------------------------------------------------------------
// M2L grouped by translation class (m2l_grp.hpp).
// ---------------------------------------------------------------------------
template <typename T>
struct LapM2LSrc {
  const int *ptrunc, *rot, *dst;
  const T* z;
  long zsize;
  int p;
  __device__ __forceinline__ void geo(int code, int& pt, int& rc, int& dist) const {
    pt = ptrunc[code];
    rc = rot[code];
    dist = dst[code];
  }
  __device__ __forceinline__ const T* ztab(int dist, int am, int q, int& stride) const {
    stride = 16 * ((p - am) / 4 + 1);
    return z + (size_t)dist * zsize + 16 * (grp_tiles(p + 1) - grp_tiles(p + 1 - am) + q);
  }
};
template <typename T>
__device__ __forceinline__ const T* grp_rot_tab(const DevTables& Tb);
template <>
__device__ __forceinline__ const double* grp_rot_tab<double>(const DevTables& Tb) { return Tb.rot_sd; }
template <>
__device__ __forceinline__ const float* grp_rot_tab<float>(const DevTables& Tb) { return Tb.rot_sd_f; }
template <typename T>
__device__ __forceinline__ const T* grp_z_tab(const DevTables& Tb);
template <>
__device__ __forceinline__ const double* grp_z_tab<double>(const DevTables& Tb) { return Tb.z_m2l_t; }
template <>
__device__ __forceinline__ const float* grp_z_tab<float>(const DevTables& Tb) { return Tb.z_m2l_t_f; }

template <typename T, int NT, int ITEMS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(ITEMS == 1 ? 4 : 2))) void k_m2l_grp(DevPlan P, DevTables Tb, int room, int lts, const T* __restrict__ mp,
                                                T* __restrict__ lo) {
  const int b = P.m2l_boxes[xcd_block()];
  const LapM2LSrc<T> S{Tb.off_ptrunc, Tb.off_rot, Tb.off_dist, grp_z_tab<T>(Tb), Tb.zt_size, P.p};
  m2l_grp_box<T, ITEMS, false>(P, b, room, lts, S, Tb.off_phase, grp_rot_tab<T>(Tb), mp, lo,
                               (T)P.inv_side[P.level[b]]);
}

// ---------------------------------------------------------------------------
// M2L with factored rotations.  A rotation by theta about y is
//   d^n(theta) = P Delta^n E(theta) Delta^nT P*,  Delta^n = d^n(pi/2),
//   P = diag(i^m), E = diag(e^{i m theta}),
// so every pair uses the same Delta blocks (they stay in cache) and only a
// diagonal phase depends on the pair; each rotation costs two products with
// Delta instead of one with a per-class matrix streamed from memory.
// Both products read Delta column-wise through d_ab = (-1)^{a-b} d_ba.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int mod4(int m) { return ((m % 4) + 4) % 4; }

// multiply (re, im) by i^r, r = 0..3
template <typename T>
__device__ __forceinline__ void mul_ipow(T& re, T& im, int r) {
  T a = re, b = im;
  if (r == 1) { re = -b; im = a; }
  else if (r == 2) { re = -a; im = -b; }
  else if (r == 3) { re = b; im = -a; }
}

// out_k = sum_m Delta^n_{mk} in_m for every (n, k) with n <= pmax
// (transpose product), then out_k *= e^{i s k theta} (s = +1 or -1).
template <typename T>
__device__ void delta_t_times(const DevTables& Tb, int pmax, const double* e, int s, const T* in, T* out) {
  const int Kt = (pmax + 1) * (pmax + 1);
  for (int idx = threadIdx.x; idx < Kt; idx += blockDim.x) {
    int n = (int)sqrtf((float)idx);
    while (n * n > idx) n--;
    while ((n + 1) * (n + 1) <= idx) n++;
    const int k = idx - n * n - n, dim = 2 * n + 1;
    const double* D = Tb.delta + Tb.delta_off[n];
    T ar = 0, ai = 0;
    for (int m = -n; m <= n; m++) {
      const T d = (T)D[(m + n) * dim + (k + n)];
      ar += d * in[2 * eidx(n, m)];
      ai += d * in[2 * eidx(n, m) + 1];
    }
    const int ak = k < 0 ? -k : k;
    const T er = (T)e[2 * ak];
    T ei = (T)e[2 * ak + 1];
    if ((k < 0) != (s < 0)) ei = -ei;
    out[2 * idx] = ar * er - ai * ei;
    out[2 * idx + 1] = ar * ei + ai * er;
  }
}

// out_a = sum_b Delta^n_{ab} in_b = sum_b (-1)^{a-b} Delta^n_{ba} in_b
template <typename T>
__device__ void delta_times(const DevTables& Tb, int pmax, const T* in, T* out) {
  const int Kt = (pmax + 1) * (pmax + 1);
  for (int idx = threadIdx.x; idx < Kt; idx += blockDim.x) {
    int n = (int)sqrtf((float)idx);
    while (n * n > idx) n--;
    while ((n + 1) * (n + 1) <= idx) n++;
    const int a = idx - n * n - n, dim = 2 * n + 1;
    const double* D = Tb.delta + Tb.delta_off[n];
    T ar = 0, ai = 0;
    for (int b = -n; b <= n; b++) {
      T d = (T)D[(b + n) * dim + (a + n)];
      if ((a - b) & 1) d = -d;
      ar += d * in[2 * eidx(n, b)];
      ai += d * in[2 * eidx(n, b) + 1];
    }
    out[2 * idx] = ar;
    out[2 * idx + 1] = ai;
  }
}

// x_m *= (-i)^m e_m over degrees <= pmax (input factor of a factored rotation)
template <typename T>
__device__ void pre_rot(int pmax, T* x) {
  const int Kt = (pmax + 1) * (pmax + 1);
  for (int idx = threadIdx.x; idx < Kt; idx += blockDim.x) {
    int n = (int)sqrtf((float)idx);
    while (n * n > idx) n--;
    while ((n + 1) * (n + 1) <= idx) n++;
    const int m = idx - n * n - n;
    T re = x[2 * idx], im = x[2 * idx + 1];
    mul_ipow(re, im, mod4(-m));
    if (m > 0 && (m & 1)) { re = -re; im = -im; }
    x[2 * idx] = re;
    x[2 * idx + 1] = im;
  }
}

template <typename T, bool LDSACC>
__global__ void k_m2l_fact(DevPlan P, DevTables Tb, const T* __restrict__ mp, T* __restrict__ lo) {
  extern __shared__ unsigned char smem_raw[];
  T* A = reinterpret_cast<T*>(smem_raw);
  T* B = A + 2 * P.K;
  const int b = P.m2l_boxes[blockIdx.x];
  T* acc = LDSACC ? B + 2 * P.K : lo + 2 * (size_t)b * P.K;
  const int p = P.p;
  const T ih = (T)P.inv_side[P.level[b]];
  const size_t zsz = (size_t)(p + 1) * (p + 1) * (p + 1);
  if (LDSACC)
    for (int k = threadIdx.x; k < 2 * P.K; k += blockDim.x) acc[k] = T(0);
  __syncthreads();
  for (int jj = P.l2_off[b]; jj < P.l2_off[b + 1]; jj++) {
    const int j = P.l2_idx[jj];
    const int di = P.ijk[3 * j] - P.ijk[3 * b] + 3, dj = P.ijk[3 * j + 1] - P.ijk[3 * b + 1] + 3,
              dk = P.ijk[3 * j + 2] - P.ijk[3 * b + 2] + 3;
    const int code = (di * 7 + dj) * 7 + dk;
    const int pt = Tb.off_ptrunc[code];
    const int Ki = (pt + 1) * (pt + 1);
    const double* phase = Tb.off_phase + (size_t)code * 2 * (p + 1);
    const double* e = Tb.rot_e + (size_t)Tb.off_rot[code] * 2 * (p + 1);
    const double* Z = Tb.z_m2l + (size_t)Tb.off_dist[code] * zsz;
    const T* in = mp + 2 * (size_t)j * P.K;
    // A = in e^{i m phi} (-i)^m e_m
    for (int k = threadIdx.x; k < Ki; k += blockDim.x) {
      int n = (int)sqrtf((float)k);
      while (n * n > k) n--;
      while ((n + 1) * (n + 1) <= k) n++;
      const int m = k - n * n - n, am = m < 0 ? -m : m;
      const T er = (T)phase[2 * am];
      const T ei = m < 0 ? -(T)phase[2 * am + 1] : (T)phase[2 * am + 1];
      const T xr = in[2 * k], xi = in[2 * k + 1];
      T re = xr * er - xi * ei, im = xr * ei + xi * er;
      mul_ipow(re, im, mod4(-m));
      if (m > 0 && (m & 1)) { re = -re; im = -im; }
      A[2 * k] = re;
      A[2 * k + 1] = im;
    }
    __syncthreads();
    delta_t_times<T>(Tb, pt, e, +1, A, B);   // B_k = e^{ik theta} sum_m Delta_mk A_m
    __syncthreads();
    delta_times<T>(Tb, pt, B, A);            // A_a = sum_k Delta_ak B_k
    __syncthreads();
    // the rotated vector is e_a i^a A_a; fold those factors into the shift
    for (int k = threadIdx.x; k < Ki; k += blockDim.x) {
      int n = (int)sqrtf((float)k);
      while (n * n > k) n--;
      while ((n + 1) * (n + 1) <= k) n++;
      const int m = k - n * n - n;
      T re = A[2 * k], im = A[2 * k + 1];
      mul_ipow(re, im, mod4(m));
      if (m > 0 && (m & 1)) { re = -re; im = -im; }
      A[2 * k] = re;
      A[2 * k + 1] = im;
    }
    __syncthreads();
    zshift_block<T>(Z, p, pt, pt, A, B);
    __syncthreads();
    pre_rot<T>(pt, B);
    __syncthreads();
    delta_t_times<T>(Tb, pt, e, -1, B, A);   // back rotation: conj(E)
    __syncthreads();
    delta_times<T>(Tb, pt, A, B);
    __syncthreads();
    // acc += e_a i^a B_a e^{-i a phi} / h
    for (int k = threadIdx.x; k < Ki; k += blockDim.x) {
      int n = (int)sqrtf((float)k);
      while (n * n > k) n--;
      while ((n + 1) * (n + 1) <= k) n++;
      const int m = k - n * n - n, am = m < 0 ? -m : m;
      T re = B[2 * k], im = B[2 * k + 1];
      mul_ipow(re, im, mod4(m));
      if (m > 0 && (m & 1)) { re = -re; im = -im; }
      const T er = (T)phase[2 * am];
      const T ei = m < 0 ? (T)phase[2 * am + 1] : -(T)phase[2 * am + 1];
      acc[2 * k] += (re * er - im * ei) * ih;
      acc[2 * k + 1] += (re * ei + im * er) * ih;
    }
    __syncthreads();
  }
  if (LDSACC) {
    T* out = lo + 2 * (size_t)b * P.K;
    for (int k = threadIdx.x; k < 2 * P.K; k += blockDim.x) out[k] += acc[k];
  }
}

// ---------------------------------------------------------------------------
// P2P near field (src/lfmm3dpart.f:1076-1141, lfmm3dpart_direct_self/_targ).
// A work item is 64 evaluation points of a leaf, one per lane; the kP2PSplit waves
// of a workgroup share it and take parts of every source box, their sums added
// in order at the end.  The source loop is
// wave-uniform, so positions and strengths stream through the scalar cache and
// every lane reuses them from SGPRs; the next source is loaded before the
// current pair is computed (p2p_sources).
// Bound: VALU issue, 39 instructions per charge-and-dipole pair in FP64 (a
// 64-lane FP64 one takes 4 cycles, the reciprocal root 16; the clock falls to
// about 1.8 GHz under them) and 38 in FP32.  1M + 1M uniform, charges and
// dipoles, near field alone: FP64 22.4 -> 19.0 ms, FP32 14.5 -> 12.6 ms
// against one wave per item with the loads next to their use (two exposed
// scalar-load waits per pair).  FP32 asks for 6 waves per SIMD, not 8: its
// redo path then spills less (13.1 -> 12.6 ms).  Offsets and r^2
// are formed in FP64 for every precision; with TN = float the rest of the
// pair is FP32, summed in FP32 over runs of at most kFold sources and folded
// into FP64 accumulators, except for the closest pairs (r^2 < rc2, r below
// 1/32 of the leaf side): such a pair dominates the sums at its point, and a
// dipole's v.d can cancel, which multiplies the FP32 rounding of v and d by
// |v||d|/|v.d|.  The FP32 loop only keeps the smallest r^2 of the run (one
// min per pair, no branch, so the loads stay ahead of the arithmetic); a
// point whose run held a close pair drops that run's FP32 sums and runs it
// again with the close pairs in FP64 from the FP64 strengths (redo_run),
// which happens for a few runs only.
// ---------------------------------------------------------------------------

// Waves per work item.  Neighbouring waves read the same sources at about the
// same time, and a small problem's few items still fill the chip: with one
// wave per item 2,000 points took 135 us, 20,000 points 248 us and 250,000
// (FP32) 2.5 ms, with four 59 us, 74 us and 1.4 ms, with sixteen 38 us, 66 us
// and 1.5 ms; 1M + 1M FP32 19.8, 13.0 and 13.3 ms.  It is the same for every
// call: a request's sums must not depend on what else is in its launch.
constexpr int kP2PSplit = 4;

// One source of the pair loop in scalar registers
template <typename TN, bool CHG, bool DIP>
struct SrcRec {
  double x, y, z;
  TN q[2], v[6];
  __device__ __forceinline__ void load(const double* __restrict__ sp, const TN* __restrict__ st) {
    x = sp[0]; y = sp[1]; z = sp[2];
    if (CHG) { q[0] = st[0]; q[1] = st[1]; }
    if (DIP)
#pragma unroll
      for (int k = 0; k < 6; k++) v[k] = st[2 + k];
  }
};

// The pair loop's constants, kept in vector registers over the loop (as
// literals FP64 ones are moved into scalar registers again for every pair)
template <typename TN>
struct PairConst {
  TN c3 = TN(3), c375 = TN(0.375);
  __device__ __forceinline__ PairConst() {
    if constexpr (sizeof(TN) == sizeof(double)) asm volatile("" : "+v"(c3), "+v"(c375));
  }
};

template <typename TN, bool CHG, bool DIP, bool FLD>
struct PairAcc {
  TN pr = 0, pi = 0, fxr = 0, fxi = 0, fyr = 0, fyi = 0, fzr = 0, fzi = 0;
  // pot += q/r + (v.d)/r^3 = (q + (v.d)/r^2)/r;
  // fld += (q + 3 (v.d)/r^2) d/r^3 - v/r^3 = (c d - v)/r^3, d = x_t - x_s
  // returns r^2 in TN
  __device__ __forceinline__ TN add(double xt, double yt, double zt, const SrcRec<TN, CHG, DIP>& s, bool mask,
                                    const PairConst<TN>& pc) {
    const double dxd = xt - s.x, dyd = yt - s.y, dzd = zt - s.z;
    const double r2d = fma(dxd, dxd, fma(dyd, dyd, dzd * dzd));
    const TN dx = (TN)dxd, dy = (TN)dyd, dz = (TN)dzd, r2 = (TN)r2d;
    TN ri = rsqrt_t<TN>(r2, pc.c375);
    if (mask) ri = TN(0);
    const TN ri2 = ri * ri;
    if (!DIP) {
      pr = fma(s.q[0], ri, pr);
      pi = fma(s.q[1], ri, pi);
      if (FLD) {
        const TN ri3 = ri * ri2;
        const TN cr = s.q[0] * ri3, ci = s.q[1] * ri3;
        fxr = fma(cr, dx, fxr); fxi = fma(ci, dx, fxi);
        fyr = fma(cr, dy, fyr); fyi = fma(ci, dy, fyi);
        fzr = fma(cr, dz, fzr); fzi = fma(ci, dz, fzi);
      }
      return r2;
    }
    const TN dotr = fma(s.v[0], dx, fma(s.v[2], dy, s.v[4] * dz));
    const TN doti = fma(s.v[1], dx, fma(s.v[3], dy, s.v[5] * dz));
    const TN ar = CHG ? fma(dotr, ri2, s.q[0]) : dotr * ri2;
    const TN ai = CHG ? fma(doti, ri2, s.q[1]) : doti * ri2;
    pr = fma(ar, ri, pr);
    pi = fma(ai, ri, pi);
    if (FLD) {
      const TN ri3 = ri * ri2, t3 = pc.c3 * ri2;
      const TN cr = CHG ? fma(t3, dotr, s.q[0]) : t3 * dotr;
      const TN ci = CHG ? fma(t3, doti, s.q[1]) : t3 * doti;
      fxr = fma(ri3, fma(cr, dx, -s.v[0]), fxr); fxi = fma(ri3, fma(ci, dx, -s.v[1]), fxi);
      fyr = fma(ri3, fma(cr, dy, -s.v[2]), fyr); fyi = fma(ri3, fma(ci, dy, -s.v[3]), fyi);
      fzr = fma(ri3, fma(cr, dz, -s.v[4]), fzr); fzi = fma(ri3, fma(ci, dz, -s.v[5]), fzi);
    }
    return r2;
  }
  __device__ __forceinline__ void fold_into(double* a) {
    a[0] += (double)pr; a[1] += (double)pi;
    if (FLD) {
      a[2] += (double)fxr; a[3] += (double)fxi; a[4] += (double)fyr;
      a[5] += (double)fyi; a[6] += (double)fzr; a[7] += (double)fzi;
    }
    pr = pi = fxr = fxi = fyr = fyi = fzr = fzi = TN(0);
  }
};

// A run of sources s0..s1-1 again at (xt, yt, zt) after its FP32 sums were
// dropped: the close pairs (r^2 < rc2, not source `self`) in FP64 from the
// FP64 strengths into tot, the rest in FP32 into acc as before.
template <typename TN, bool CHG, bool DIP, bool FLD>
__device__ __forceinline__ void redo_run(PairAcc<TN, CHG, DIP, FLD>& acc, double xt, double yt, double zt,
                                         const double* __restrict__ spos, const TN* __restrict__ str,
                                         const double* __restrict__ str64, int s0, int s1, int self, double rc2,
                                         double* tot) {
  acc = PairAcc<TN, CHG, DIP, FLD>();
  PairAcc<double, CHG, DIP, FLD> c64;
  const PairConst<double> pc64;
  const PairConst<TN> pc;
  for (int s = s0; s < s1; s++) {
    const double* sp = spos + 4 * (size_t)s;
    const double dx = xt - sp[0], dy = yt - sp[1], dz = zt - sp[2];
    if (s != self && fma(dx, dx, fma(dy, dy, dz * dz)) < rc2) {
      SrcRec<double, CHG, DIP> r;
      r.load(sp, str64 + 8 * (size_t)s);
      c64.add(xt, yt, zt, r, false, pc64);
    } else {
      SrcRec<TN, CHG, DIP> r;
      r.load(sp, str + 8 * (size_t)s);
      acc.add(xt, yt, zt, r, s == self, pc);
    }
  }
  c64.fold_into(tot);
}

// The pairs of one point with sources s0..s1-1 (s1 > s0; SELF: source `self`
// is left out).  Two source records are kept: while a pair is computed the
// next source's scalar loads are in flight.  They return out of order, so the
// only wait there is waits for all of them: it stands right before the next
// record's loads are issued, when the one in hand has had a whole pair's
// arithmetic to arrive.  (FP32 instructions that read a scalar register issue
// at half the rate of all-vector ones; FP32 strengths staged in LDS and read
// as vectors were no faster all the same: 12.6 -> 13.4 ms at 1M + 1M.)
template <typename TN, bool CHG, bool DIP, bool FLD, bool SELF>
__device__ __forceinline__ void p2p_sources(PairAcc<TN, CHG, DIP, FLD>& acc, const PairConst<TN>& pc, double x, double y,
                                            double z, const double* __restrict__ spos, const TN* __restrict__ str,
                                            const double* __restrict__ str64, int s0, int s1, int self, double rc2,
                                            double* tot) {
  constexpr bool fold = sizeof(TN) < sizeof(double);
  const TN rc2n = (TN)rc2, kFar = TN(1e30);
  SrcRec<TN, CHG, DIP> ra, rb;
  auto arrived = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
  };
  auto load = [&](SrcRec<TN, CHG, DIP>& r, unsigned s, int k) {  // source s + k
    r.load(spos + 4 * (size_t)s + 4 * k, str + 8 * (size_t)s + 8 * k);
  };
  load(ra, (unsigned)s0, 0);
  for (int c = s0; c < s1; c += (fold ? kFold : (1 << 30))) {
    const int ce = fold ? min(c + kFold, s1) : s1;
    TN mn = kFar;
    auto pair = [&](const SrcRec<TN, CHG, DIP>& r, int s) {
      __builtin_amdgcn_sched_barrier(0);
      const TN r2 = acc.add(x, y, z, r, SELF && s == self, pc);
      if (fold) mn = fmin(mn, SELF && s == self ? kFar : r2);
    };
    // ra holds source s; kFold is even, so it does at every run's start
    int s = c;
    const int lim = min(ce, s1 - 2);
    for (; s < lim; s += 2) {
      // (the index, not pointers, is what the loop carries: carried pointers
      // ended up in vector registers, six readfirstlane per pair)
      const unsigned u = (unsigned)__builtin_amdgcn_readfirstlane(s);
      arrived();
      load(rb, u, 1);
      pair(ra, s);
      arrived();
      load(ra, u, 2);
      pair(rb, s + 1);
    }
    if (s < ce) {  // the last one or two of s0..s1-1: nothing past them is read
      arrived();
      if (s + 1 < ce) {
        load(rb, (unsigned)s, 1);
        pair(ra, s);
        arrived();
        pair(rb, s + 1);
      } else {
        pair(ra, s);
      }
    }
    if (fold) {
      if (mn < rc2n) redo_run(acc, x, y, z, spos, str, str64, c, ce, SELF ? self : -1, rc2, tot);
      acc.fold_into(tot);
    }
  }
}

template <typename TN, bool CHG, bool DIP, bool FLD>
__global__ __launch_bounds__(64 * kP2PSplit) __attribute__((amdgpu_waves_per_eu(sizeof(TN) == 4 ? 6 : 8))) void k_p2p(DevPlan P, const double* __restrict__ spos,
                                             const TN* __restrict__ str, const double* __restrict__ str64,
                                             const double* __restrict__ tpos, double* __restrict__ pot0,
                                             double* __restrict__ fld0, double* __restrict__ pot1,
                                             double* __restrict__ fld1) {
  const int part = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
  const int w = xcd_block();  // one work item per workgroup
  const int b = P.p2p_items[3 * w], kind = P.p2p_items[3 * w + 1], start = P.p2p_items[3 * w + 2];
  double tot[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  bool active = false;
  int me = 0;
  if (b >= 0) {  // not a padding item
    const int n0 = kind ? P.itrg[b] : P.isrc[b];
    const int nn = kind ? P.ntrg[b] : P.nsrc[b];
    const int i = start + lane;
    active = i < nn;
    me = n0 + (active ? i : 0);
    const double* mp = (kind ? tpos : spos) + 4 * (size_t)me;
    const double x = mp[0], y = mp[1], z = mp[2];
    PairAcc<TN, CHG, DIP, FLD> acc;
    const PairConst<TN> pc;
    constexpr bool fold = sizeof(TN) < sizeof(double);
    // FP32 pairs: pairs closer than 1/32 of this leaf's side run in FP64 (on a
    // uniform 1M cube 0.05 such pairs per point; the near-field error of the
    // FP32 pairs falls from 1.5e-7 to 8e-8 of the potential, and on a sphere
    // with a target next to a dipole from 7e-7 to 3e-9)
    const double hside = 1.0 / P.inv_side[P.level[b]];
    const double rc2 = fold ? hside * hside * (1.0 / 1024.0) : 0.0;
    // this wave's part of a box's sources
    auto cut = [&](int s0, int n, int q) { return s0 + (int)((long)n * q / kP2PSplit); };
    // own box first: a source never acts on itself (index test, lfmm3dpart.f:1193)
    if (kind == 0) {
      const int s0 = P.isrc[b], n = P.nsrc[b];
      const int a = cut(s0, n, part), e = cut(s0, n, part + 1);
      if (a < e) p2p_sources<TN, CHG, DIP, FLD, true>(acc, pc, x, y, z, spos, str, str64, a, e, me, rc2, tot);
    }
    const int l0 = P.l1_off[b], l1 = P.l1_off[b + 1];
    for (int jj = kind == 0 ? l0 : l0 - 1; jj < l1; jj++) {  // targets: their own box, then list 1
      const int j = jj < l0 ? b : P.l1_idx[jj];
      const int s0 = P.isrc[j], n = P.nsrc[j];
      const int a = cut(s0, n, part), e = cut(s0, n, part + 1);
      if (a < e) p2p_sources<TN, CHG, DIP, FLD, false>(acc, pc, x, y, z, spos, str, str64, a, e, -1, rc2, tot);
    }
    if (!fold) acc.fold_into(tot);
  }
  add_parts<kP2PSplit, FLD ? 8 : 2>(tot, part, lane);
  if (part > 0) return;
  if (!active) return;
  double* po = kind ? pot1 : pot0;
  po[2 * (size_t)me] += tot[0];
  po[2 * (size_t)me + 1] += tot[1];
  if (FLD) {
    double* fo = kind ? fld1 : fld0;
    for (int k = 0; k < 6; k++) fo[6 * (size_t)me + k] += tot[2 + k];
  }
}

// Direct sum over all sources (l3dpartdirect, src/lfmm3dpart.f:1391): the pair
// arithmetic of the near field in FP64 with every source acting on every point.
// A workgroup takes 64 points, from `first` on, and slice blockIdx.y of the
// sources, each wave a part of the slice (direct_slices); the waves' sums are
// added in order, the slices' by k_direct_sum.  24,001 sources acting on themselves and on 10,007
// targets: 13.4 -> 1.46 ms (the FP64 instructions alone take about 1 ms); one
// wave for 64 points and all sources left two thirds of the SIMDs without a wave,
// and each waited for its own scalar loads.
template <bool CHG, bool DIP>
__global__ __launch_bounds__(64 * kDirectWaves) void k_direct(int ns, const double* __restrict__ spos,
                                                              const double* __restrict__ str, int npts, int first,
                                                              const double* __restrict__ pts, int pts_are_sources,
                                                              double* __restrict__ partial, double* __restrict__ pot,
                                                              double* __restrict__ fld) {
  const int part = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
  first += 64 * (int)blockIdx.x;
  const int i = first + lane;
  const bool active = i < npts;
  const int me = active ? i : 0;
  const double* mp = (pts_are_sources ? spos : pts) + 4 * (size_t)me;
  const double x = mp[0], y = mp[1], z = mp[2];
  const int s0 = direct_cut(ns, part), s1 = direct_cut(ns, part + 1);
  PairAcc<double, CHG, DIP, true> acc;
  const PairConst<double> pc;
  double t[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (s0 < s1) {
    if (pts_are_sources && s0 - first < 64 && s1 > first)  // the points' own sources among them
      p2p_sources<double, CHG, DIP, true, true>(acc, pc, x, y, z, spos, str, str, s0, s1, me, 0.0, t);
    else
      p2p_sources<double, CHG, DIP, true, false>(acc, pc, x, y, z, spos, str, str, s0, s1, -1, 0.0, t);
  }
  acc.fold_into(t);
  add_parts<kDirectWaves, 8>(t, part, lane);
  if (part == 0 && active) direct_store(t, i, npts, partial, pot, fld);
}

}  // namespace fmm3d
