// P2M / P2L of charges in FP64 on the matrix cores (k_form_mfma); k_form2
// (lap_kernels.hip) forms everything else.
#pragma once
#include <hip/hip_runtime.h>

#include "kern_common.hpp"

namespace fmm3d {

// ---------------------------------------------------------------------------
// The sums over sources S(n, +-a) = sum_s q_s H_n^{+-a}(u_s) (see k_form2) are
// products of the harmonics with the charges.  v_mfma_f64_4x4x4 takes its A
// operand as 16 rows (4 blocks of 4) x 4 depths, one value per lane: lane l is
// given column a = a0 + l % 16 of source l / 16 of a group of four, and walks n
// = a, a + 1, .. with the scaled recurrence of FacLayout in registers, so each
// step's harmonic is the operand where it stands and nothing goes through LDS.
// The B operand is q_re, q_im (l % 4 = 0, 1; else 0) of source l / 16, and the
// product adds, for each of the 16 columns, the four sources' h q to the
// accumulators of step k: lane l holds column a0 + 4 (l / 4 % 4) + l / 16,
// weight l % 4, for every step k < S (two doubles each).
// One workgroup of four waves per box; a wave has one block of 16 columns and
// every parts-th group of sources (FormWaves).  Scalars and charges of 64
// sources at a time are staged in LDS by one wave while the others multiply.
// At the end the sums go to LDS, the parts of a block added in order.
//
// A step is 5 FP64 operations and 2 products of 19 cycles for 64 (source,
// column) values; a walk ends at a multiple of four.  At order 39 71% of them are
// used in P2M (820 entries, blocks of 40, 24 and 8 steps), 64% in P2L (861; 44,
// 28 and 12).  400,000 clustered points, order 39: P2L 28.1 -> 7.4 ms, P2M 2.6 ->
// 0.8 ms (with the tables in LDS, k_form2: 12.9 and 1.1 ms).  Dipoles take two
// operands of weights: with both in one wave (one wave per SIMD) 200,000 +
// 180,000 points at order 26 took 4.8 ms for P2L but 0.70 for P2M (k_form2: 5.6
// and 0.34) and 250,000 Plummer points 4.5 and 0.95 ms (k_form2: 4.2, 0.40),
// with a wave per operand 6.0 and 5.5 ms for P2L; they stay with k_form2.
// ---------------------------------------------------------------------------
constexpr int kFormMfmaWaves = 4;
constexpr int kFormMfmaBatch = 64;  // sources staged at a time
constexpr int kFormMfmaRec = 7;     // doubles per staged source: 5 scalars and the charge

// per wave of the workgroup: first column of its block, its part of the
// block's sources and their number
struct FormWaves {
  short a0[kFormMfmaWaves], part[kFormMfmaWaves], parts[kFormMfmaWaves], rounds;
};
// Waves to the blocks of 16 columns, degrees up to pt (at most 4 blocks): one
// each, the rest to the block with the most steps per wave.
inline FormWaves form_waves(int pt) {
  FormWaves W{};
  const int nblk = pt / 16 + 1;
  int n[kFormMfmaWaves] = {0, 0, 0, 0};
  for (int b = 0; b < nblk; b++) n[b] = 1;
  for (int w = nblk; w < kFormMfmaWaves; w++) {
    int best = 0;
    for (int b = 1; b < nblk; b++)
      if ((pt + 1 - 16 * b) * n[best] > (pt + 1 - 16 * best) * n[b]) best = b;
    n[best]++;
  }
  int w = 0;
  for (int b = 0; b < nblk; b++)
    for (int k = 0; k < n[b]; k++, w++) {
      W.a0[w] = (short)(16 * b);
      W.part[w] = (short)k;
      W.parts[w] = (short)n[b];
      W.rounds = (short)(n[b] > W.rounds ? n[b] : W.rounds);
    }
  return W;
}
// LDS doubles: recurrence factors [step][column] and two batches, or at the end
// one weight's sums (4 per half-table entry)
__host__ __device__ inline int form_mfma_lds(int pt) {
  const int run = (pt + 1) * (pt + 1) + 2 * kFormMfmaBatch * kFormMfmaRec, end = 2 * (pt + 1) * (pt + 2);
  return run > end ? run : end;
}

// S: steps held (a multiple of 4, at least pt + 1)
template <bool IRREG, int S>
__global__ __launch_bounds__(64 * kFormMfmaWaves) void k_form_mfma(
    DevPlan P, const double* __restrict__ fac, const double* __restrict__ spos, const double* __restrict__ str,
    FormWaves W, double* __restrict__ expn) {
  extern __shared__ __align__(16) double fsm[];
  const int p = P.p, pt = IRREG ? p + 1 : p, C = pt + 1;
  const FacLayout L(p);
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int NT = 64 * kFormMfmaWaves;
  const int a0 = W.a0[wid], part = W.part[wid], parts = W.parts[wid];
  double* beta = fsm;
  double* stage = fsm + C * C;
  // factor of the step from n = a + k to n + 1 (0 past pt: the walk stays finite)
  for (int e = tid; e < C * C; e += NT) {
    const int k = e / C, a = e - k * C, n = a + k + 1;
    beta[e] = n <= pt ? fac[L.BT + hidx(n, a)] : 0.0;
  }
  const int b = IRREG ? P.p2l_boxes[blockIdx.x] : P.p2m_boxes[blockIdx.x];
  const double ih = P.inv_side[P.level[b]];
  const double cx = P.center[3 * b], cy = P.center[3 * b + 1], cz = P.center[3 * b + 2];
  // source cursor over the boxes of list 4 (P2L) or box b (P2M)
  int jj = IRREG ? P.l4_off[b] : 0, t0 = 0, s0 = 0, sn = 0;
  const int jend = IRREG ? P.l4_off[b + 1] : 1;
  auto open_box = [&] {
    t0 = 0;
    if (jj < jend) {
      const int j = IRREG ? P.l4_idx[jj] : b;
      s0 = P.isrc[j];
      sn = P.nsrc[j];
    }
  };
  // fills a batch (wave `by` loads and stores); returns the number of sources,
  // the slots up to the next multiple of four holding zeros
  auto fill = [&](double* st, int by) {
    int filled = 0, idx = -1;
    while (filled < kFormMfmaBatch && jj < jend) {
      const int take = min(kFormMfmaBatch - filled, sn - t0);
      if (lane >= filled && lane < filled + take) idx = s0 + t0 + lane - filled;
      filled += take;
      t0 += take;
      if (t0 >= sn) {
        jj++;
        open_box();
      }
    }
    if (wid == by && lane < ((filled + 3) & ~3)) {
      double v[kFormMfmaRec] = {0, 0, 0, 0, 0, 0, 0};
      if (idx >= 0) {
        const double* x = spos + 4 * (size_t)idx;
        const double* q = str + 8 * (size_t)idx;
        const double ux = (x[0] - cx) * ih, uy = (x[1] - cy) * ih, uz = (x[2] - cz) * ih;
        const double r2 = ux * ux + uy * uy + uz * uz;
        const double ir2 = IRREG ? 1.0 / r2 : 1.0;
        v[0] = -ux * ir2; v[1] = -uy * ir2; v[2] = uz * ir2;
        v[3] = IRREG ? ir2 : r2;
        v[4] = IRREG ? sqrt(ir2) : 1.0;
        v[5] = q[0]; v[6] = q[1];
      }
      double* o = st + kFormMfmaRec * lane;
#pragma unroll
      for (int k = 0; k < kFormMfmaRec; k++) o[k] = v[k];
    }
    return filled;
  };
  double acc[S][2];
#pragma unroll
  for (int k = 0; k < S; k++) acc[k][0] = acc[k][1] = 0.0;
  const int a = a0 + (lane & 15), len = C - a0;  // this lane's column; steps of the block
  const double* bt = beta + (a <= pt ? a : pt);
  open_box();
  int cur = fill(stage, 0);
  __syncthreads();
  for (int bi = 1; cur > 0; bi++) {
    const double* st = stage + ((bi - 1) & 1) * kFormMfmaBatch * kFormMfmaRec;
    const int nxt = fill(stage + (bi & 1) * kFormMfmaBatch * kFormMfmaRec, bi & (kFormMfmaWaves - 1));
    for (int g = part; 4 * g < cur; g += parts) {
      const double* rec = st + kFormMfmaRec * (4 * g + (lane >> 4));
      C2<double> w = {rec[0], rec[1]}, r = {a <= pt ? rec[4] : 0.0, 0.0};
      const double zz = rec[2], rho = rec[3];
      const double wt = (lane & 3) < 2 ? rec[5 + (lane & 1)] : 0.0;
      for (int e = a; e; e >>= 1) {
        if (e & 1) r = cmul(r, w);
        w = cmul(w, w);
      }
      C2<double> r0 = {0.0, 0.0};
      double bk[3] = {bt[0], bt[(C > 1 ? 1 : 0) * C], bt[(C > 2 ? 2 : C - 1) * C]};  // factors, three steps ahead
#pragma unroll
      for (int k = 0; k < S; k++) {
        if ((k & 3) == 0 && k >= len) break;
        const double br = bk[k % 3] * rho;
        bk[k % 3] = bt[(k + 3 < C ? k + 3 : C - 1) * C];
        acc[k][0] = __builtin_amdgcn_mfma_f64_4x4x4f64(r.re, wt, acc[k][0], 0, 0, 0);
        acc[k][1] = __builtin_amdgcn_mfma_f64_4x4x4f64(r.im, wt, acc[k][1], 0, 0, 0);
        const C2<double> rn = {fma(zz, r.re, -(br * r0.re)), fma(zz, r.im, -(br * r0.im))};
        r0 = r;
        r = rn;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
    cur = nxt;
  }
  // S(n, +a), S(n, -a) to LDS at 4 hidx(n, a), then into the coefficients
  const int ao = a0 + 4 * ((lane >> 2) & 3) + (lane >> 4);  // column of this lane's sums
  for (int rd = 0; rd < W.rounds; rd++) {
    if (part == rd) {
#pragma unroll
      for (int k = 0; k < S; k++) {
        if ((k & 3) == 0 && k >= len) break;
        // lanes of q_re hold the sums of q_re h_re and q_re h_im, their
        // neighbours those of q_im
        const double dr = acc[k][0], di = acc[k][1];
        const double er = __shfl_xor(dr, 1), ei = __shfl_xor(di, 1);
        const int n = ao + k;
        if ((lane & 3) == 0 && n <= pt) {
          const double gn = fac[L.GN + hidx(n, ao)];
          double* o = fsm + 4 * hidx(n, ao);
          const double v[4] = {gn * (dr - ei), gn * (di + er), gn * (dr + ei), gn * (er - di)};
#pragma unroll
          for (int e = 0; e < 4; e++) o[e] = rd == 0 ? v[e] : o[e] + v[e];
        }
      }
    }
    __syncthreads();
  }
  double* out = expn + 2 * (size_t)b * P.K;
  const double sc = IRREG ? ih : 1.0;
  for (int k = tid; k < P.K; k += NT) {
    int n = (int)sqrtf((float)k);
    while (n * n > k) n--;
    while ((n + 1) * (n + 1) <= k) n++;
    const int m = k - n * n - n;  // coefficient (n, m): the sum over H_n^{-m}
    const double* o = fsm + 4 * hidx(n, m < 0 ? -m : m) + (m > 0 ? 2 : 0);
    out[2 * k] += o[0] * sc;
    out[2 * k + 1] += o[1] * sc;
  }
}

}  // namespace fmm3d
