// Device code of the projector bra by sets of matrices (FP64 MFMA).
#pragma once

#include "kernels.h"

namespace octhip {

typedef double d4 __attribute__((ext_vector_type(4)));

// Bra by sets.  A wave takes one group of <= 16 mesh points: its 4 state loads and the
// projector loads of its first 32 projector rows are in flight together, and a product
// A(16 projector rows x 4 points) B(4 points x 16 lanes) serves up to 4 matrices of 4
// projectors.  Lane (kk, ii) supplies A[ii][kk] = P[row ii, point kk] from line step(ii/4) of
// the group (32-byte runs) and gets D[4r+kk][ii]: rows 4r .. 4r+3 are those of step r.  The
// sums go to the wave's part of LDS and the 4 waves are added in a fixed order.  No row of a
// group takes part in a matrix it does not belong to, and operands past its points are zero.
// tid: thread of the BLOCK threads of this block, red: their LDS; a block that is not live
// computes and stores nothing.
// PHASE: the states times the Bloch phases of (point, matrix), which differ by matrix: a
// product per step, of which D rows 4r .. 4r+3 are kept.
template <int TW, bool PHASE>
__device__ __forceinline__ void bra_set_body(const BraMfmaArgs& m, int bl, int lt, double* red, int tid,
                                             bool live) {
  constexpr int TL = 16 * TW;
  static_assert(BRA_SET_GROUPS == BLOCK / 64, "a group per wave");
  const BraArgs& b = m.b;
  const BraSetArgs& a = m.set;
  const int4 blk = a.blk[bl];
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = tid & 63;
  const int kk = ln >> 4, ii = ln & 15;
  const int col = lt * TL + ii * TW, lc = min(col, b.L - TW);  // lanes past a short row: clamped, not stored
  const int sums = blk.w * b.pjmax * TL;      // LDS doubles of a wave
  double* const mine = red + (size_t)wave * sums;
  const KetGroup gr = a.grp[blk.x + min(wave, blk.y - 1)];
  const int n = gr.rows, ns = gr.steps;
  int p[4], row[4];
  double av[2][4];                            // projector rows 0 .. 15 and 16 .. 31
  Vec<TW> bv[4];
  const double* const pt = a.pt + 4 * (size_t)gr.line + (ii & 3);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    p[k] = min(4 * k + kk, n - 1);
    row[k] = a.point[gr.row + p[k]];
    av[0][k] = pt[4 * (size_t)(min(ii >> 2, ns - 1) * n + p[k])];
  }
  if (ns > 4)
#pragma unroll
    for (int k = 0; k < 4; ++k) av[1][k] = pt[4 * (size_t)(min(4 + (ii >> 2), ns - 1) * n + p[k])];
#pragma unroll
  for (int k = 0; k < 4; ++k) bv[k] = ldv<TW>(b.psi + (size_t)row[k] * b.L + lc);
  for (int t = ln; t < sums; t += 64) mine[t] = 0.0;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (wave < blk.y) {
    for (int t0 = 0; t0 < ns; t0 += 4) {      // 16 projector rows at a time
      double x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        x[k] = t0 == 0   ? av[0][k]
               : t0 == 4 ? av[1][k]
                         : pt[4 * (size_t)(min(t0 + (ii >> 2), ns - 1) * n + p[k])];
        x[k] = 4 * k + kk < n ? x[k] : 0.0;
      }
      d4 acc[TW];
      const auto product = [&](const Vec<TW>* v) {
#pragma unroll
        for (int w = 0; w < TW; ++w) acc[w] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int w = 0; w < TW; ++w)
            acc[w] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[k], 4 * k + kk < n ? v[k].v[w] : 0.0, acc[w], 0, 0, 0);
      };
      if constexpr (!PHASE) product(bv);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (t0 + r >= ns) break;
        if constexpr (PHASE) {
          const size_t ent = a.step[gr.step + t0 + r].z;
          Vec<TW> ph[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const double pr = a.phase[2 * (ent + p[k])], pi = a.phase[2 * (ent + p[k]) + 1];
            if constexpr (TW == 2) {
              ph[k].v[0] = zmul_lane(pr, pi, bv[k].v[0], bv[k].v[1], false);
              ph[k].v[1] = zmul_lane(pr, pi, bv[k].v[1], bv[k].v[0], true);
            } else {
              ph[k].v[0] = zmul_lane(pr, pi, bv[k].v[0], __shfl_xor(bv[k].v[0], 1), (col & 1) != 0);
            }
          }
          product(ph);
        }
        // a matrix that holds the point twice adds to its rows twice
        const int sum = t0 == 0 ? gr.sum[r] : a.step[gr.step + t0 + r].y;
        double* const d = mine + (sum + kk) * TL + ii * TW;
        Vec<TW> v = ldv<TW>(d);
#pragma unroll
        for (int w = 0; w < TW; ++w) v.v[w] += acc[w][r];
        stv<TW>(d, v);
      }
    }
  }
  __syncthreads();
  for (int t = tid; t < sums && live; t += BLOCK) {
    const int q = t / TL, slot = q / b.pjmax;
    if (lt * TL + (t - q * TL) >= b.L) continue;
    const double v = (red[t] + red[t + sums]) + (red[t + 2 * (size_t)sums] + red[t + 3 * (size_t)sums]);
    b.partial[((size_t)a.part[blk.z + slot] * b.pjmax + (q - slot * b.pjmax)) * b.L + lt * TL + (t - q * TL)] = v;
  }
}

}  // namespace octhip
