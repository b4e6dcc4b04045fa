// The grouped M2L, shared by Laplace (k_m2l_grp) and Helmholtz (k_hm2l_grp).
//
// List-2 sources of one target whose offsets share (dx^2 + dy^2, dz) share the
// rotation block, the z-shift table and the truncation order; only the
// azimuthal phase differs.  Up to kM2LGroup of them are translated together by
// one workgroup per target, the target's local accumulating in LDS.
//
// Orders m and -m of every expansion are held as their sum s_m = a_m + a_{-m}
// (s_0 = a_0) and difference d_m = a_m - a_{-m}, m >= 1.  The rotation blocks
// obey D[-m][-m'] = D[m][m'], so sums rotate into sums and differences into
// differences, with the blocks D[m][m'] +- D[-m][m'] over m, m' >= 0: half the
// products and half the reads of the product with all orders.  The z-shift is
// the same for m and -m and stays as it is.  Degree n of a member lies in LDS
// as s_0..s_n, d_1..d_n from slot n*n on: one ascending row for each parity
// (slot n*n + parity*n + m).
//
// A work item is four consecutive orders m' (rotation) or degrees l (z-shift);
// its 2 or 4 lanes are (parity) x (pair of members), each lane holding four
// complex outputs of two members: one 4-value table row and two LDS reads feed
// 16 FMAs.  What bounds it is the operand traffic, not the FMAs: per row of a
// tile a wave reads 2 KB of table through L1 and 2 KB of LDS for 16 FMAs (FP64);
// at 1M + 1M points, p = 26, L1's address unit is busy 75% of the time and the
// FMAs issue in half of it.  M2L alone there: 8.4 ms with all orders, one member
// per lane, 4.8 so; FP32 4.7 and 2.3 ms; 400,000 clustered points (p = 39) 7.4
// and 3.4 ms.
#pragma once
#include <hip/hip_runtime.h>

#include "lap_kernels.hpp"

namespace fmm3d {

constexpr int kM2LGroup = 4;   // members per group
constexpr int kM2LChunk = 192; // list-2 entries ordered at a time (list 2 has <= 189)

// ints of the per-index degree table of k_m2l_mfma, kept a multiple of 4 so
// that what follows stays 16-byte aligned
__host__ __device__ inline int grp_kn_ints(int p) { return ((p + 4) * (p + 4) + 3) / 4 * 4; }

// Values per member in LDS: (p+4)^2 complex, padded so that the stride in
// 4-byte words is 8 mod 32 and the members of a work item start in different
// quarters of the 32 LDS banks.
template <typename T>
__host__ __device__ inline int grp_member_stride(int p) {
  const int base = 2 * (p + 4) * (p + 4);
  return sizeof(T) == 8 ? base + ((4 - base) & 15) : base + ((8 - base) & 31);
}

// items (degree n, columns 4q..4q+3) of the degrees below m; in the z-shift
// of order pt the same list enumerates (n = pt - |m|, rows |m|+4q..)
__host__ __device__ inline int grp_items(int m) {
  const int a = m >> 2;
  return (2 * a + (m & 3)) * (a + 1);
}
// sum of (j/4+1)^2 over j < n: 4x4 tiles of the square blocks of those degrees
__host__ __device__ inline int grp_tiles(int n) {
  const int a = n >> 2;
  return 2 * a * (a + 1) * (2 * a + 1) / 3 + (n & 3) * (a + 1) * (a + 1);
}
// ints in front of the values in LDS: seven arrays per list-2 entry, the
// groups (start and size, after four counts), the work items, and (n, m) of
// each pair index n(n+1)/2 + m
__host__ __device__ inline int grp_int_count(int p) {
  return (8 * kM2LChunk + 4 + grp_items(p + 1) + (p + 1) * (p + 2) / 2 + 3) / 4 * 4;
}
// complex values of one team in LDS: phases, the local, a pool for members (of
// the size of `room` members of order p)
template <typename T>
__host__ __device__ inline int grp_pool(int p, int room) { return room * (grp_member_stride<T>(p) / 2); }
template <typename T>
__host__ __device__ inline int grp_team_values(int p, int room) {
  return kM2LGroup * (p + 1) + (p + 1) * (p + 1) + grp_pool<T>(p, room);
}
template <typename T>
__host__ __device__ inline size_t grp_lds_bytes(int p, int room, int teams) {
  return (size_t)grp_int_count(p) * sizeof(int) + 2 * sizeof(T) * (size_t)teams * grp_team_values<T>(p, room);
}
// Members per group of truncation order pt: as many as the pool holds and as
// the team has work items for.  Most list-2 orders are far below p (5 to 8 of
// 14, 9 to 15 of 26), so a pool of two full members holds four of most.
template <typename T>
__device__ inline int grp_members(int pt, int pool, int slots) {
  const int ni = grp_items(pt + 1), ms = grp_member_stride<T>(pt) / 2;
  int g = min(kM2LGroup, pool / ms);
  if (g > 2 && 4 * ni > slots) g = 2;
  return max(g, 1);
}

// Launch shape for order p and the LDS a workgroup may take: threads (0: the
// kernel does not fit), work items per thread, the pool's full-order members,
// log2 of the threads that share a group (a team) and the teams.  A pool of
// four full members instead of two takes 79 KB at p = 26 and leaves two
// workgroups on a CU, with most lanes idle: Helmholtz on a sphere 4.6 ms
// against 3.0, Laplace in a cube FP32 3.3 against 2.3, FP64 4.8 both; a larger
// pool is taken where it costs no workgroup, and two work items per thread where
// one workgroup fills the CU's LDS anyway (p = 39, clusters: 4.0 ms with one
// item, whose groups of high order then hold two members, 3.4 with two).  Small orders put several teams into a
// workgroup, each with its own groups and its own local: what a group costs
// there is the latency of its seven stages, which the teams share (20,000
// points, p = 14: 400 us with one team, 270 us with four).  The shape
// depends on p alone, so a box's sums do not depend on the launch.
struct GrpShape {
  int threads = 0, items = 1, room = 0, lts = 0, teams = 0;
};
template <typename T>
inline GrpShape grp_shape(int p, size_t lds_max) {
  GrpShape s;
  const int lanes = 2 * grp_items(p + 1);
  if (lanes > 1024) return s;
  s.items = lanes > 512 ? 2 : 1;
  s.lts = lanes > 256 ? 9 : lanes > 128 ? 8 : lanes > 64 ? 7 : 6;
  const int threads = s.lts == 8 ? 256 : 512;
  s.teams = threads >> s.lts;
  s.room = grp_lds_bytes<T>(p, 2, s.teams) <= lds_max ? 2 : 1;
  if (grp_lds_bytes<T>(p, s.room, s.teams) > lds_max) return s;
  const size_t fit = lds_max / grp_lds_bytes<T>(p, s.room, s.teams);
  while (s.room < kM2LGroup && lds_max / grp_lds_bytes<T>(p, s.room + 1, s.teams) == fit) s.room++;
  if (fit == 1 && lanes > 256) s.items = 2;
  s.threads = threads;
  return s;
}

template <typename T>
struct __attribute__((aligned(4 * sizeof(T)))) V4 {
  T v[4];
};
template <typename T>
struct __attribute__((aligned(2 * sizeof(T)))) V2 {
  T x, y;
};

// exchange within a quad of lanes (0xB1: lane ^ 1, 0x4E: lane ^ 2)
template <int CTRL>
__device__ __forceinline__ float quad_swap(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double quad_swap(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// two rows of a 4x4 tile, ROW values apart
template <int ROW, typename T>
__device__ __forceinline__ void grp_tab2(V4<T> (&d)[2], const T* __restrict__ t) {
  d[0] = *reinterpret_cast<const V4<T>*>(t);
  d[1] = *reinterpret_cast<const V4<T>*>(t + ROW);
}
// r[4c..4c+3] += d_c * (x, y): x, y the complex values of the two members
template <bool NEG, typename T>
__device__ __forceinline__ void grp_fma_row(T (&r)[16], const V4<T>& d, V2<T> x, V2<T> y) {
  if (NEG) { x.x = -x.x; x.y = -x.y; y.x = -y.x; y.y = -y.y; }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    r[4 * c] = fma(d.v[c], x.x, r[4 * c]);
    r[4 * c + 1] = fma(d.v[c], x.y, r[4 * c + 1]);
    r[4 * c + 2] = fma(d.v[c], y.x, r[4 * c + 2]);
    r[4 * c + 3] = fma(d.v[c], y.y, r[4 * c + 3]);
  }
}

// Four outputs of one parity of degree n, two members: rows m = 0..n of the
// tiles at D (tile stride `stride`), x0/x1 the members' slots of that parity.
// BACK applies the transpose, D^T[m][m'] = (-1)^{m+m'} D[m][m'], but for the
// factor (-1)^{m'}.  d0 holds the first two rows on entry; two buffers of two
// rows each: the next rows are in flight while the current ones are used.
// Rows past n, and m = 0 of the differences, are zero in the table and read
// finite values of neighbouring slots.
template <typename T, bool BACK>
__device__ __forceinline__ void grp_rot_item(const T* __restrict__ D, int stride, int n, const V2<T>* x0,
                                             const V2<T>* x1, V4<T> (&d0)[2], T (&r)[16]) {
  V4<T> d1[2];
  V2<T> a0 = x0[0], a1 = x0[1], b0 = x1[0], b1 = x1[1];
  for (int left = n / 4;; left--) {
    grp_tab2<8>(d1, D + 16);
    const V2<T> a2 = x0[2], a3 = x0[3], b2 = x1[2], b3 = x1[3];
    __builtin_amdgcn_sched_barrier(0);
    grp_fma_row<false>(r, d0[0], a0, b0);
    grp_fma_row<BACK>(r, d0[1], a1, b1);
    const int dx = left > 0 ? 4 : 0;   // (the last pass loads its own rows again)
    D += left > 0 ? stride : 0;
    x0 += dx;
    x1 += dx;
    grp_tab2<8>(d0, D);
    a0 = x0[0]; a1 = x0[1]; b0 = x1[0]; b1 = x1[1];
    __builtin_amdgcn_sched_barrier(0);
    grp_fma_row<false>(r, d1[0], a2, b2);
    grp_fma_row<BACK>(r, d1[1], a3, b3);
    if (left == 0) break;
  }
}

// out_l = sum_{n=am}^{pt} Z[l][n] in_n for l = l0..l0+3 of one order and
// parity, two members.  e: slot of degree am, whose successor at degree n is
// 2n+1+par slots further.  Degrees pt+1..pt+3 of the members are zero.
template <typename T>
__device__ __forceinline__ void grp_z_item(const T* __restrict__ Z, int stride, int am, int par, int nrb,
                                           const V2<T>* x0, const V2<T>* x1, V4<T> (&d0)[2], T (&r)[16]) {
  V4<T> d1[2];
  int e = am * am + par * am + am, st = 2 * am + 1 + par;
  V2<T> a0 = x0[e], b0 = x1[e];
  e += st;
  V2<T> a1 = x0[e], b1 = x1[e];
  for (int left = nrb - 1;; left--) {
    grp_tab2<4>(d1, Z + 8);
    e += st + 2;
    const V2<T> a2 = x0[e], b2 = x1[e];
    e += st + 4;
    const V2<T> a3 = x0[e], b3 = x1[e];
    __builtin_amdgcn_sched_barrier(0);
    grp_fma_row<false>(r, d0[0], a0, b0);
    grp_fma_row<false>(r, d0[1], a1, b1);
    Z += left > 0 ? stride : 0;
    grp_tab2<4>(d0, Z);
    e = left > 0 ? e + st + 6 : 0;
    a0 = x0[e]; b0 = x1[e];
    st += 8;
    e = left > 0 ? e + st : 0;
    a1 = x0[e]; b1 = x1[e];
    __builtin_amdgcn_sched_barrier(0);
    grp_fma_row<false>(r, d1[0], a2, b2);
    grp_fma_row<false>(r, d1[1], a3, b3);
    if (left == 0) break;
  }
}

// The same with a complex table (Helmholtz coaxial shifts): a tile is 16 real
// parts, then 16 imaginary parts.
template <typename T>
__device__ __forceinline__ void grp_fma_row_c(T (&r)[16], const V4<T>& dr, const V4<T>& di, V2<T> x, V2<T> y) {
#pragma unroll
  for (int c = 0; c < 4; c++) {
    r[4 * c] = fma(dr.v[c], x.x, fma(-di.v[c], x.y, r[4 * c]));
    r[4 * c + 1] = fma(dr.v[c], x.y, fma(di.v[c], x.x, r[4 * c + 1]));
    r[4 * c + 2] = fma(dr.v[c], y.x, fma(-di.v[c], y.y, r[4 * c + 2]));
    r[4 * c + 3] = fma(dr.v[c], y.y, fma(di.v[c], y.x, r[4 * c + 3]));
  }
}
template <typename T>
__device__ __forceinline__ void grp_z_item_c(const T* __restrict__ Z, int stride, int am, int par, int nrb,
                                             const V2<T>* x0, const V2<T>* x1, T (&r)[16]) {
  int e = am * am + par * am + am, st = 2 * am + 1 + par;
  V4<T> c0, c1, n0, n1;
  c0 = reinterpret_cast<const V4<T>*>(Z)[0];
  c1 = reinterpret_cast<const V4<T>*>(Z)[4];
  V2<T> a = x0[e], b = x1[e];
  for (int left = nrb - 1;; left--) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const V2<T> ca = a, cb = b;
      if (u < 3) {
        n0 = reinterpret_cast<const V4<T>*>(Z)[u + 1];
        n1 = reinterpret_cast<const V4<T>*>(Z)[u + 5];
        e += st;
      } else {
        Z += left > 0 ? stride : 0;
        n0 = reinterpret_cast<const V4<T>*>(Z)[0];
        n1 = reinterpret_cast<const V4<T>*>(Z)[4];
        e = left > 0 ? e + st : 0;
      }
      st += 2;
      a = x0[e];
      b = x1[e];
      __builtin_amdgcn_sched_barrier(0);
      grp_fma_row_c(r, c0, c1, ca, cb);
      c0 = n0;
      c1 = n1;
    }
    if (left == 0) break;
  }
}

// One target box; a team is 2^lts threads.  Src supplies the operators:
//   geo(code, pt, rc, dist)    truncation order, rotation class, shift class
//   ztab(dist, am, q, &stride) first tile of order am's tile column q
// rtab: per rotation class and degree the tiles of D+ and D-, [row block]
// [column block][row][parity][column]: the two parities of a work item read one
// 64-byte line of L1 (FP64).  mp/lo: packed complex expansions.
template <typename T, int ITEMS, bool CZ, class Src>
__device__ __forceinline__ void m2l_grp_box(const DevPlan& P, int b, int room, int lts, const Src& S,
                                            const double* __restrict__ off_phase, const T* __restrict__ rtab,
                                            const T* __restrict__ mp, T* __restrict__ lo, T scale) {
  extern __shared__ unsigned char smem_raw[];
  const int tid = threadIdx.x, bs = blockDim.x;
  const int p = P.p, P1 = p + 1, K = P1 * P1;
  int* s_key = reinterpret_cast<int*>(smem_raw);
  int* s_box = s_key + kM2LChunk;
  int* s_code = s_box + kM2LChunk;
  int* t_key = s_code + kM2LChunk;
  int* t_box = t_key + kM2LChunk;
  int* t_code = t_box + kM2LChunk;
  int* t_geo = t_code + kM2LChunk;
  int* s_grp = t_geo + kM2LChunk;           // groups: start << 3 | size, after the waves' counts
  int* s_it = s_grp + 4 + kM2LChunk;        // work items n << 8 | q, n ascending
  int* s_nm = s_it + grp_items(P1);         // n << 16 | m of pair n(n+1)/2 + m
  const int TW = grp_team_values<T>(p, room), pool = grp_pool<T>(p, room);
  // (a team is whole waves: what belongs to its group is uniform in a wave)
  const int teams = bs >> lts, team = __builtin_amdgcn_readfirstlane(tid >> lts), tt = tid & ((1 << lts) - 1),
            ts = 1 << lts;
  V2<T>* vals = reinterpret_cast<V2<T>*>(smem_raw + (size_t)grp_int_count(p) * sizeof(int));
  V2<T>* s_ph = vals + team * TW;           // the members' e^{i m phi}
  V2<T>* acc = s_ph + kM2LGroup * P1;
  V2<T>* A = acc + K;
  const V2<T> zero = {T(0), T(0)};
  for (int k = tid; k < teams * TW; k += bs) vals[k] = zero;
  for (int n = tid; n <= p; n += bs) {
    for (int m = 0; m <= n; m++) s_nm[n * (n + 1) / 2 + m] = n << 16 | m;
    for (int q = 0, i0 = grp_items(n); 4 * q <= n; q++) s_it[i0 + q] = n << 8 | q;
  }
  const int rclass = 32 * grp_tiles(P1);    // values per rotation class
  const int off0 = P.l2_off[b], n2 = P.l2_off[b + 1] - off0;
  const int bi = P.ijk[3 * b], bj = P.ijk[3 * b + 1], bk = P.ijk[3 * b + 2];
  for (int c0 = 0; c0 < n2; c0 += kM2LChunk) {
    const int cn = min(kM2LChunk, n2 - c0);
    __syncthreads();
    if (tid < cn) {
      const int j = P.l2_idx[off0 + c0 + tid];
      const int di = P.ijk[3 * j] - bi, dj = P.ijk[3 * j + 1] - bj, dk = P.ijk[3 * j + 2] - bk;
      s_box[tid] = j;
      s_code[tid] = ((di + 3) * 7 + (dj + 3)) * 7 + (dk + 3);
      s_key[tid] = (di * di + dj * dj) * 7 + (dk + 3);
    }
    __syncthreads();
    if (tid < cn) {  // stable rank by key
      const int key = s_key[tid], code = s_code[tid];
      int pt, rc, dist;
      S.geo(code, pt, rc, dist);
      int rank = 0, same = 0, eq = 0;
      for (int t = 0; t < cn; t++) {
        const int kt = s_key[t];
        rank += kt < key;
        eq += kt == key;
        same += kt == key && t < tid;
      }
      rank += same;
      // a group starts at every gm-th entry of a class
      const int gm = grp_members<T>(pt, pool, ITEMS << lts);
      s_grp[4 + rank] = same % gm ? 0 : min(gm, eq - same);
      t_key[rank] = key;
      t_box[rank] = s_box[tid];
      t_code[rank] = code;
      t_geo[rank] = pt << 20 | rc << 10 | dist;
    }
    __syncthreads();
    // the groups in order: each wave counts its starts, then places them
    const int gsz = tid < cn ? s_grp[4 + tid] : 0;
    const unsigned long long starts = __ballot(gsz > 0);
    if (tid < 256 && (tid & 63) == 0) s_grp[tid >> 6] = __popcll(starts);
    __syncthreads();
    if (gsz > 0) {
      int at = __popcll(starts & ((1ull << (tid & 63)) - 1));
      for (int w = 0; w < (tid >> 6); w++) at += s_grp[w];
      s_grp[4 + at] = tid << 3 | gsz;
    }
    __syncthreads();
    const int ng = __builtin_amdgcn_readfirstlane(s_grp[0] + s_grp[1] + s_grp[2] + s_grp[3]);
    for (int gi = team; gi - team < ng; gi += teams) {
      const int grp = __builtin_amdgcn_readfirstlane(gi < ng ? s_grp[4 + gi] : 0);   // (0: an idle team)
      const int s0 = grp >> 3, g = grp & 7;
      const int geo0 = __builtin_amdgcn_readfirstlane(t_geo[s0]);
      const int pt = geo0 >> 20, rc = (geo0 >> 10) & 1023, dist = geo0 & 1023;
      const int MS = grp_member_stride<T>(pt) / 2;
      const int lg = g > 2 ? 2 : 1;         // log2 of the lanes per item
      // item u0 in the first round and NI-1-u0 in the second, which pairs the
      // cheapest items with the most expensive ones
      const int NI = g > 0 ? grp_items(pt + 1) : 0, U0 = ts >> lg;
      const int u0 = tt >> lg, par = tt & 1, jm = g > 2 ? (tt >> 1) & 1 : 0;
      int uq[ITEMS], it[ITEMS];
      uq[0] = u0 < NI ? u0 : -1;
      if (ITEMS > 1) uq[ITEMS - 1] = NI - 1 - u0 >= U0 ? NI - 1 - u0 : -1;
#pragma unroll
      for (int q = 0; q < ITEMS; q++) it[q] = s_it[uq[q] < 0 ? 0 : uq[q]];
      const bool two = 2 * jm + 1 < g;
      V2<T>* x0 = A + 2 * jm * MS;
      V2<T>* x1 = two ? x0 + MS : x0;
      const T* rt[ITEMS];
      int rs[ITEMS];
#pragma unroll
      for (int q = 0; q < ITEMS; q++) {
        const int n = it[q] >> 8, nq = n / 4 + 1;
        rs[q] = 32 * nq;
        rt[q] = rtab + (size_t)rc * rclass + 32 * (grp_tiles(n) + (it[q] & 255)) + 4 * par;
      }
      // (idle lanes load nothing: with most orders truncated they are the most)
      V4<T> d[2] = {};
      if (uq[0] >= 0) grp_tab2<8>(d, rt[0]);
      // (a) members times e^{i m phi}, as sums and differences; the slots of
      // degrees pt+1..pt+3 set to zero
      const int Kp = (pt + 1) * (pt + 1), Kz = (pt + 4) * (pt + 4), Kh = (pt + 1) * (pt + 2) / 2;
      for (int j0 = 0, h0 = tt; j0 < g;) {
        constexpr int U = 4;
        V2<T> xp[U], xm[U];
        V2<double> ph[U];
        int jj[U], nm[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          while (h0 >= Kh) { h0 -= Kh; j0++; }
          jj[u] = j0;
          const int jc = j0 < g ? j0 : g - 1;   // (loads without a branch)
          nm[u] = s_nm[h0];
          const int n = nm[u] >> 16, m = nm[u] & 65535;
          const V2<T>* src = reinterpret_cast<const V2<T>*>(mp) + (size_t)t_box[s0 + jc] * K + n * n + n;
          xp[u] = src[m];
          xm[u] = src[-m];
          ph[u] = reinterpret_cast<const V2<double>*>(off_phase)[(size_t)t_code[s0 + jc] * P1 + m];
          h0 += ts;
        }
#pragma unroll
        for (int u = 0; u < U; u++)
          if (jj[u] < g) {
            const int n = nm[u] >> 16, m = nm[u] & 65535;
            const T er = (T)ph[u].x, ei = (T)ph[u].y;
            V2<T>* out = A + jj[u] * MS + n * n;
            const T ar = xp[u].x * er - xp[u].y * ei, ai = xp[u].x * ei + xp[u].y * er;
            if (m == 0) {
              out[0] = {ar, ai};
            } else {
              const T br = xm[u].x * er + xm[u].y * ei, bi2 = xm[u].y * er - xm[u].x * ei;
              out[m] = {ar + br, ai + bi2};
              out[n + m] = {ar - br, ai - bi2};
            }
            if (n == pt) s_ph[jj[u] * P1 + m] = {er, ei};
          }
      }
      for (int jj = 0; jj < g; jj++)
        for (int k = Kp + tt; k < Kz; k += ts) A[jj * MS + k] = zero;
      __syncthreads();
      T r[ITEMS][16];
      // (b) rotate to the z axis
#pragma unroll
      for (int q = 0; q < ITEMS; q++) {
#pragma unroll
        for (int e = 0; e < 16; e++) r[q][e] = T(0);
        if (uq[q] >= 0) {
          const int n = it[q] >> 8, e0 = n * n + par * n;
          if (q > 0) grp_tab2<8>(d, rt[q]);
          grp_rot_item<T, false>(rt[q], rs[q], n, x0 + e0, x1 + e0, d, r[q]);
        }
      }
      const T* zt[ITEMS];
      int zs[ITEMS];
#pragma unroll
      for (int q = 0; q < ITEMS; q++) zt[q] = S.ztab(dist, pt - min(it[q] >> 8, pt), it[q] & 255, zs[q]);
      d[0] = d[1] = V4<T>{};
      if (!CZ && uq[0] >= 0) grp_tab2<4>(d, zt[0]);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < ITEMS; q++)
        if (uq[q] >= 0) {
          const int n = it[q] >> 8, m0 = 4 * (it[q] & 255), e0 = n * n + par * n;
#pragma unroll
          for (int c = 0; c < 4; c++)
            if (m0 + c <= n && m0 + c >= par) {
              x0[e0 + m0 + c] = {r[q][4 * c], r[q][4 * c + 1]};
              if (two) x1[e0 + m0 + c] = {r[q][4 * c + 2], r[q][4 * c + 3]};
            }
        }
      __syncthreads();
      // (c) shift along z
#pragma unroll
      for (int q = 0; q < ITEMS; q++) {
#pragma unroll
        for (int e = 0; e < 16; e++) r[q][e] = T(0);
        if (uq[q] >= 0) {
          const int t = it[q] >> 8, am = pt - t;
          if (CZ) {
            grp_z_item_c<T>(zt[q], zs[q], am, par, t / 4 + 1, x0, x1, r[q]);
          } else {
            if (q > 0) grp_tab2<4>(d, zt[q]);
            grp_z_item<T>(zt[q], zs[q], am, par, t / 4 + 1, x0, x1, d, r[q]);
          }
        }
      }
      d[0] = d[1] = V4<T>{};
      if (uq[0] >= 0) grp_tab2<8>(d, rt[0]);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < ITEMS; q++)
        if (uq[q] >= 0) {
          const int am = pt - (it[q] >> 8), l0 = am + 4 * (it[q] & 255);
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const int l = l0 + c;
            if (l <= pt && am >= par) {
              x0[l * l + par * l + am] = {r[q][4 * c], r[q][4 * c + 1]};
              if (two) x1[l * l + par * l + am] = {r[q][4 * c + 2], r[q][4 * c + 3]};
            }
          }
        }
      __syncthreads();
      // (d) rotate back, apply the phases e^{-+i m' phi} and sum the members:
      //   s += S cos - i D sin,  d += D cos - i S sin
      // each lane forms both terms of its parity, the two parities exchange
      // the second, and the two pairs of members share the columns
#pragma unroll
      for (int q = 0; q < ITEMS; q++) {
#pragma unroll
        for (int e = 0; e < 16; e++) r[q][e] = T(0);
        if (uq[q] < 0) continue;
        const int n = it[q] >> 8, m0 = 4 * (it[q] & 255), e0 = n * n + par * n;
        if (q > 0) grp_tab2<8>(d, rt[q]);
        grp_rot_item<T, true>(rt[q], rs[q], n, x0 + e0, x1 + e0, d, r[q]);
        const V2<T>* ph = s_ph + 2 * jm * P1;
        V2<T> own[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const int mq = m0 + c <= n ? m0 + c : n;
          V2<T> e1 = ph[mq], e2 = two ? ph[P1 + mq] : zero;
          if (c & 1) { e1.x = -e1.x; e1.y = -e1.y; e2.x = -e2.x; e2.y = -e2.y; }  // (-1)^{m'}
          const T ar = r[q][4 * c], ai = r[q][4 * c + 1], br = r[q][4 * c + 2], bi2 = r[q][4 * c + 3];
          own[c].x = fma(br, e2.x, ar * e1.x);
          own[c].y = fma(bi2, e2.x, ai * e1.x);
          own[c].x += quad_swap<0xB1>(fma(bi2, e2.y, ai * e1.y));
          own[c].y -= quad_swap<0xB1>(fma(br, e2.y, ar * e1.y));
        }
        V2<T>* o = acc + e0 + m0;
        if (g > 2) {
#pragma unroll
          for (int c = 0; c < 2; c++) {
            const V2<T> mine = jm ? own[2 + c] : own[c], give = jm ? own[c] : own[2 + c];
            const T vr = mine.x + quad_swap<0x4E>(give.x), vi = mine.y + quad_swap<0x4E>(give.y);
            const int k = 2 * jm + c;
            if (m0 + k <= n && m0 + k >= par) {
              o[k].x += vr;
              o[k].y += vi;
            }
          }
        } else {
#pragma unroll
          for (int c = 0; c < 4; c++)
            if (m0 + c <= n && m0 + c >= par) {
              o[c].x += own[c].x;
              o[c].y += own[c].y;
            }
        }
      }
      __syncthreads();
    }
  }
  __syncthreads();
  V2<T>* out = reinterpret_cast<V2<T>*>(lo) + (size_t)b * K;
  for (int h = tid; h < (p + 1) * (p + 2) / 2; h += bs) {
    const int n = s_nm[h] >> 16, m = s_nm[h] & 65535, k = n * n + n;
    V2<T> s = zero, dd = zero;
    for (int t = 0; t < teams; t++) {
      const V2<T>* at = vals + t * TW + kM2LGroup * P1 + n * n + m;
      s.x += at[0].x;
      s.y += at[0].y;
      dd.x += at[n].x;
      dd.y += at[n].y;
    }
    if (m == 0) {
      out[k].x += s.x * scale;
      out[k].y += s.y * scale;
    } else {
      const T hs = T(0.5) * scale;
      out[k + m].x += (s.x + dd.x) * hs;
      out[k + m].y += (s.y + dd.y) * hs;
      out[k - m].x += (s.x - dd.x) * hs;
      out[k - m].y += (s.y - dd.y) * hs;
    }
  }
}

}  // namespace fmm3d
