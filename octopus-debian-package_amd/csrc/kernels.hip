// Kernel instances and launchers: fused apply, projector bra (FP64 MFMA and plain).
#include <algorithm>

#include "bra.h"

namespace octhip {

namespace {

template <int N, int IDX, int EPI, int LPT>
int launch_apply_n(ApplyArgs& a, hipStream_t s) {
  const int per = 8 * (a.chunk > 1 ? a.chunk : 1);
  const int grid = ((a.ntiles + per - 1) / per) * per;
  const size_t shmem = (size_t)a.tpts * a.sstride * sizeof(int);
  ProfScope prof("k_apply", s);
  hipLaunchKernelGGL((k_apply<N, IDX, EPI, LPT>), dim3(grid), dim3(BLOCK), shmem, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "k_apply launch: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}

template <int IDX, int EPI, int LPT>
int launch_apply_lpt(ApplyArgs& a, hipStream_t s) {
  switch (a.n) {
    case 25: return launch_apply_n<25, IDX, EPI, LPT>(a, s);
    case 19: return launch_apply_n<19, IDX, EPI, LPT>(a, s);
    case 13: return launch_apply_n<13, IDX, EPI, LPT>(a, s);
    case 7: return launch_apply_n<7, IDX, EPI, LPT>(a, s);
    default: return launch_apply_n<0, IDX, EPI, LPT>(a, s);
  }
}

template <int IDX>
int launch_apply_idx(ApplyArgs& a, int epi, int lpt, hipStream_t s) {
  if (epi == EPI_TAYLOR) return launch_apply_lpt<IDX, EPI_TAYLOR, 2>(a, s);
  if (epi == EPI_TAYLOR_X) return launch_apply_lpt<IDX, EPI_TAYLOR_X, 2>(a, s);
  return lpt == 2 ? launch_apply_lpt<IDX, EPI_STORE, 2>(a, s) : launch_apply_lpt<IDX, EPI_STORE, 1>(a, s);
}

}  // namespace

int launch_apply(ApplyArgs& a, bool lattice, int epi, hipStream_t s) {
  if (a.np <= 0) return OCTHIP_SUCCESS;
  const int lpt = a.L >= 2 ? 2 : 1;
  if (epi != EPI_STORE && lpt != 2) return fail(OCTHIP_ERR_INVALID, "Taylor epilogue needs complex rows");
  int tpp = a.L / lpt;
  if (tpp > 64) tpp = 64;
  int tshift = 0;
  while ((1 << tshift) < tpp) ++tshift;
  a.tpp = tpp;
  a.tshift = tshift;
  const int slots = BLOCK / tpp;
  int iters = a.tile_iters > 0 ? a.tile_iters : 4;
  while (iters > 1 && slots * iters > 256) --iters;
  a.tpts = slots * iters;
  a.sstride = a.n > 0 ? ((a.n + 3) & ~3) : 1;
  a.ntiles = (a.np + a.tpts - 1) / a.tpts;
  if (a.chunk < 1) a.chunk = 1;
  return lattice ? launch_apply_idx<IDX_LATTICE>(a, epi, lpt, s) : launch_apply_idx<IDX_RI>(a, epi, lpt, s);
}

// -------------------------------------------------------------- bra (plain) --
// One workgroup per chunk of <= BRA_CHUNK sphere points of one matrix.  Threads are
// (slice, lane): each slice sums every nsl-th sphere point of the chunk for one lane,
// slices are then added in fixed order through LDS, so results are deterministic.
constexpr int BRA_PJB = 8;  // projectors per register block

__device__ __forceinline__ void bra_plain_body(const BraArgs& b, int c) {
  __shared__ double red[BLOCK * BRA_PJB];
  const int4 ch = b.chunks[c];
  const int4 mi = b.mat_info[ch.x];
  const int npt = mi.x, npj = mi.y, moff = mi.z, mapoff = mi.w;
  const int Lc = b.L < BLOCK ? b.L : BLOCK;
  const int nsl = BLOCK / Lc;
  const int sl = threadIdx.x / Lc;
  const int lc = threadIdx.x - sl * Lc;
  for (int lg = 0; lg < b.L; lg += Lc) {
    const int l = lg + lc;
    for (int jb = 0; jb < npj; jb += BRA_PJB) {
      double acc[BRA_PJB];
#pragma unroll
      for (int jj = 0; jj < BRA_PJB; ++jj) acc[jj] = 0.0;
      for (int q = ch.y + sl; q < ch.z; q += nsl) {
        const int row = b.maps[mapoff + q] - 1;
        double x = b.psi[(size_t)row * b.L + l];
        if (b.pphase) {
          const double xq = b.psi[(size_t)row * b.L + (l ^ 1)];
          x = zmul_lane(b.pphase[2 * (size_t)(mapoff + q)], b.pphase[2 * (size_t)(mapoff + q) + 1], x, xq,
                        (l & 1) != 0);
        }
#pragma unroll
        for (int jj = 0; jj < BRA_PJB; ++jj)
          if (jb + jj < npj) acc[jj] = fma(b.mats[moff + (size_t)(jb + jj) * npt + q], x, acc[jj]);
      }
#pragma unroll
      for (int jj = 0; jj < BRA_PJB; ++jj) red[(sl * BRA_PJB + jj) * Lc + lc] = acc[jj];
      __syncthreads();
      if (sl == 0) {
        for (int jj = 0; jj < BRA_PJB && jb + jj < npj; ++jj) {
          double t = 0.0;
          for (int s2 = 0; s2 < nsl; ++s2) t += red[(s2 * BRA_PJB + jj) * Lc + lc];
          b.partial[((size_t)c * b.pjmax + jb + jj) * b.L + l] = t;
        }
      }
      __syncthreads();
    }
  }
}

__global__ __launch_bounds__(BLOCK) void k_bra_plain(const BraArgs b) { bra_plain_body(b, blockIdx.x); }

// --------------------------------------------------------------- bra (MFMA) --
// D(16 projectors x 16 lanes) += A(16 x 4 sphere points) * B(4 x 16 lanes) with
// v_mfma_f64_16x16x4_f64.  Operand layout (wave64): lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; accumulator element r of lane l is D[4*r + l/16][l%16] (checked on the
// device with an in-bounds probe).
// A comes from the transposed projector table (16 lanes read consecutive doubles of one
// sphere point's row), B from the state rows (16 lanes read 128 contiguous bytes, 256
// with two columns per lane).
// One workgroup per (chunk, lane tile of 16 TW lanes): grids of nchunk * L/(16 TW) blocks
// keep every CU busy; the 4 waves take interleaved groups of 4 sphere points and are
// summed through LDS in a fixed order.  Every load is issued unconditionally (clamped
// indices, zero operands past the chunk end) so the compiler counts them exactly.
// TW = 2: lane ii of a wave loads the 16 bytes of columns 2ii and 2ii+1 of its row (one
// complex value) and feeds two MFMAs, one per column, that share the projector operand:
// each column's sum is the TW = 1 sum, in the same order.
constexpr int BRA_RED = 4 * 16 * 16;  // LDS doubles per accumulator of the wave reduction
template <int TW>
__device__ __forceinline__ void bra_mfma_body(const BraMfmaArgs& m, int c, int lt, double* red) {
  constexpr int KB = 16;                    // MFMA steps (4 sphere points each) per load block
  const BraArgs& b = m.b;
  const int4 ch = b.chunks[c];
  const int4 mi = b.mat_info[ch.x];
  const int npj = mi.y, mapoff = mi.w;
  const int wave = threadIdx.x >> 6;
  const int ln = threadIdx.x & 63;
  const int kk = ln >> 4, ii = ln & 15;
  const int col = lt * 16 * TW + ii * TW;   // first column of this lane
  for (int jb = 0; jb < npj; jb += 16) {
    d4 acc[TW];
#pragma unroll
    for (int w = 0; w < TW; ++w) acc[w] = d4{0.0, 0.0, 0.0, 0.0};
    const int jc = min(jb + ii, npj - 1);
    const bool jok = jb + ii < npj;
    for (int q0 = ch.y + 4 * wave; q0 < ch.z; q0 += KB * 16) {
      int row[KB];
      double av[KB];
      Vec<TW> bv[KB];
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        const int qk = q0 + 16 * k + kk;
        const int qs = qk < ch.z ? qk : ch.y;
        row[k] = b.maps[mapoff + qs] - 1;
        av[k] = m.pt[(size_t)(mapoff + qs) * m.pjs + jc];
      }
#pragma unroll
      for (int k = 0; k < KB; ++k) bv[k] = ldv<TW>(b.psi + (size_t)row[k] * b.L + col);
      if (b.pphase) {
        // Bloch phase of each sphere point on the (re, im) pair: with TW = 2 the lane
        // holds both, otherwise the other one is the neighbouring thread's (lanes ii and
        // ii ^ 1 hold the same point)
#pragma unroll
        for (int k = 0; k < KB; ++k) {
          const int qk = q0 + 16 * k + kk;
          const size_t pi2 = 2 * (size_t)(mapoff + (qk < ch.z ? qk : ch.y));
          if constexpr (TW == 2) {
            const double re = zmul_lane(b.pphase[pi2], b.pphase[pi2 + 1], bv[k].v[0], bv[k].v[1], false);
            const double im = zmul_lane(b.pphase[pi2], b.pphase[pi2 + 1], bv[k].v[1], bv[k].v[0], true);
            bv[k].v[0] = re;
            bv[k].v[1] = im;
          } else {
            const double xq = __shfl_xor(bv[k].v[0], 1);
            bv[k].v[0] = zmul_lane(b.pphase[pi2], b.pphase[pi2 + 1], bv[k].v[0], xq, (col & 1) != 0);
          }
        }
      }
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        const bool ok = q0 + 16 * k + kk < ch.z;
#pragma unroll
        for (int w = 0; w < TW; ++w)
          acc[w] = __builtin_amdgcn_mfma_f64_16x16x4f64((ok && jok) ? av[k] : 0.0, ok ? bv[k].v[w] : 0.0, acc[w],
                                                        0, 0, 0);
      }
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < TW; ++w)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[w * BRA_RED + (wave * 16 + 4 * r + kk) * 16 + ii] = acc[w][r];
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int w = 0; w < TW; ++w)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int jl = 4 * r + kk;
          const double t = (red[w * BRA_RED + (0 * 16 + jl) * 16 + ii] + red[w * BRA_RED + (1 * 16 + jl) * 16 + ii]) +
                           (red[w * BRA_RED + (2 * 16 + jl) * 16 + ii] + red[w * BRA_RED + (3 * 16 + jl) * 16 + ii]);
          const int j = jb + jl;
          if (j < npj) b.partial[((size_t)c * b.pjmax + j) * b.L + col + w] = t;
        }
    }
  }
}

extern __shared__ double2 bra_lds[];
template <bool SETS, bool PHASE>
__device__ __forceinline__ void bra_mfma(const BraMfmaArgs& m, int b) {
  double* const red = reinterpret_cast<double*>(bra_lds);
  const int nlt = mfma_lane_tiles(m.b.L);
  const bool wide = (m.b.L & 31) == 0;
  if constexpr (SETS) {
    if (wide) bra_set_body<2, PHASE>(m, b / nlt, b % nlt, red, threadIdx.x, true);
    else bra_set_body<1, PHASE>(m, b / nlt, b % nlt, red, threadIdx.x, true);
  } else {
    if (wide) bra_mfma_body<2>(m, b / nlt, b % nlt, red);
    else bra_mfma_body<1>(m, b / nlt, b % nlt, red);
  }
}

template <bool SETS, bool PHASE>
__global__ __launch_bounds__(BLOCK) void k_bra_mfma(const BraMfmaArgs m) {
  const int nz = (int)gridDim.x - m.nbra;
  if ((int)blockIdx.x < nz) {
    // the first blocks clear the boundary rows of the batch (boundaries_set), fused into
    // this launch (the bra reads inner rows only); dispatched first, the streaming stores
    // overlap the latency-bound bra blocks instead of trailing them (-4% for the launch)
    for (size_t t = blockIdx.x * (size_t)BLOCK + threadIdx.x; t < m.zcount; t += (size_t)nz * BLOCK)
      m.zf[m.zfirst + t] = 0.0;
    return;
  }
  bra_mfma<SETS, PHASE>(m, (int)blockIdx.x - nz);
}

// Projection row i at 16 lanes, by one wave: scal * the sum of its matrix's parts as four
// interleaved sums, (s0 + s1) + (s2 + s3): lanes 16 q .. 16 q + 15 add parts first + q,
// first + q + 4, ..., loaded together with clamped indices.  (A radius-3 sphere at h = 0.25
// has 29 parts by spheres and about 120 by sets; four sums keep either at one or two round
// trips, so the launch is 4 to 5 us at all sizes.)
__device__ __forceinline__ void bra_reduce_body(const BraReduceArgs& r, int bid, int nblk) {
  constexpr int N = 16;
  const int ln = threadIdx.x & 63, tiles = (r.L + 15) / 16;
  for (int t = bid * (BLOCK / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); t < r.nrow * tiles;
       t += nblk * (BLOCK / 64)) {
    const int i = t / tiles, l0 = (t - i * tiles) * 16, l = min(l0 + (ln & 15), r.L - 1);
    const ProjRow w = r.row[i];
    const int2 p = r.sets ? w.part[1] : w.part[0];
    double s = 0.0;
    for (int c = p.x + (ln >> 4); c < p.y && w.scal >= 0; c += 4 * N) {
      double v[N];
#pragma unroll
      for (int u = 0; u < N; ++u) v[u] = r.partial[((size_t)min(c + 4 * u, p.y - 1) * r.pjmax + w.j) * r.L + l];
#pragma unroll
      for (int u = 0; u < N; ++u)
        if (c + 4 * u < p.y) s += v[u];
    }
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    if (ln < 16 && l0 + ln < r.L) r.proj[(size_t)i * r.L + l] = w.scal < 0 ? 0.0 : s * r.scals[w.scal];
  }
}

__global__ __launch_bounds__(BLOCK) void k_bra_reduce(const BraReduceArgs r) {
  bra_reduce_body(r, blockIdx.x, gridDim.x);
}

}  // namespace octhip

namespace octhip {

int launch_bra(const BraArgs& b, int nchunk, hipStream_t s) {
  if (nchunk <= 0) return OCTHIP_SUCCESS;
  ProfScope prof("k_bra", s);
  hipLaunchKernelGGL(k_bra_plain, dim3(nchunk), dim3(BLOCK), 0, s, b);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "k_bra launch: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}

int launch_bra_mfma(BraMfmaArgs& m, size_t lds, hipStream_t s) {
  if (m.nbra <= 0) return OCTHIP_SUCCESS;
  const int zblocks = m.zf ? (int)std::min<size_t>((m.zcount + BLOCK - 1) / BLOCK, 2048) : 0;
  ProfScope prof("k_bra", s);
  if (m.sets && m.set.phase)
    hipLaunchKernelGGL((k_bra_mfma<true, true>), dim3(m.nbra + zblocks), dim3(BLOCK), lds, s, m);
  else if (m.sets)
    hipLaunchKernelGGL((k_bra_mfma<true, false>), dim3(m.nbra + zblocks), dim3(BLOCK), lds, s, m);
  else
    hipLaunchKernelGGL((k_bra_mfma<false, false>), dim3(m.nbra + zblocks), dim3(BLOCK), lds, s, m);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "k_bra_mfma launch: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}

// One workgroup per (KET_GROUPS groups, lane tile of 16 TW lanes), a group per wave.  MFMA form:
// D(16 rows x 16 lanes) = A(16 rows x 4 projectors) B(4 projectors x 16 lanes); lane (kk, ii)
// supplies A[ii][kk] = P[row ii, kk]
// and B[kk][ii] = proj[kk, col] of the step; accumulator element r of lane (kk, ii) is
// D[4r+kk][ii].  Operands past a group's rows are clamped: their D rows are not stored.
// TW = 2: 32-lane tiles, lane ii computes columns 2ii and 2ii+1 with two MFMAs that share
// the projector operand and stores them as one 16-byte piece (one complex value); each
// column's sum is the TW = 1 sum, in the same order.
// A wave's loads are a chain of round trips (group, then its operands), which is what
// bounds this kernel: a group's record holds its first KET_AHEAD steps, whose operands are
// loaded together, and a wave has one group.
template <int TW, bool PHASE, bool ADD>
__device__ __forceinline__ void ket_mfma_body(const KetArgs& k, int b, int lt) {
  constexpr int TL = 16 * TW;                 // lanes of the tile
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
  const int g = b * KET_GROUPS + wave;
  const int kk = ln >> 4, ii = ln & 15;
  const int col = lt * TL + ii * TW;          // first column of this lane
  const int lc = min(col, k.L - TW);          // (columns past a short row: clamped, not stored)
  if (g >= k.ngrp) return;
  const KetGroup gr = k.grp[g];
  const int n = gr.rows, ns = gr.steps;
  const double* const pt = k.pt + 4 * ((size_t)gr.line + min(ii, n - 1)) + kk;
  const double* const pj = k.proj + (size_t)kk * k.L + lc;
  int p[ADD ? 4 : 1];                         // ADD: mesh rows 4r+kk of the group
  if constexpr (ADD) {
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = k.point[gr.row + min(4 * r + kk, n - 1)];
  }
  d4 acc[TW], tot[TW];
#pragma unroll
  for (int w = 0; w < TW; ++w) acc[w] = tot[w] = d4{0.0, 0.0, 0.0, 0.0};
  int ent = 0;                                // PHASE: first entry of the matrix in acc
  const auto flush = [&]() {
    // tot += the matrix's term of row 4r+kk times conj(its Bloch phase): with TW = 2 the
    // lane holds the (re, im) pair, otherwise lanes ii ^ 1 hold the pair
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const size_t pi2 = 2 * (size_t)(ent + min(4 * r + kk, n - 1));
      const double pr = k.phase[pi2], pi = -k.phase[pi2 + 1];
      if constexpr (TW == 2) {
        tot[0][r] += zmul_lane(pr, pi, acc[0][r], acc[1][r], false);
        tot[1][r] += zmul_lane(pr, pi, acc[1][r], acc[0][r], true);
      } else {
        tot[0][r] += zmul_lane(pr, pi, acc[0][r], __shfl_xor(acc[0][r], 1), (col & 1) != 0);
      }
    }
  };
  Vec<TW> old[ADD ? 4 : 1];
  for (int q0 = 0; q0 < ns; q0 += KET_AHEAD) {
    double av[KET_AHEAD];
    Vec<TW> bv[KET_AHEAD];
#pragma unroll
    for (int u = 0; u < KET_AHEAD; ++u) {
      const int q = min(q0 + u, ns - 1);
      av[u] = pt[4 * (size_t)(q * n)];
      bv[u] = ldv<TW>(pj + (size_t)(q0 == 0 ? gr.proj[u] : k.step[gr.step + q].x) * k.L);
    }
    if constexpr (ADD) {
      if (q0 == 0)
#pragma unroll
        for (int r = 0; r < 4; ++r) old[r] = ldv<TW>(k.out + (size_t)p[r] * k.L + lc);
    }
#pragma unroll
    for (int u = 0; u < KET_AHEAD; ++u) {
      if (q0 + u >= ns) break;
      if constexpr (PHASE) {
        const int4 st = k.step[gr.step + q0 + u];
        if (st.w) {
          if (q0 + u > 0) flush();
          ent = st.z;
#pragma unroll
          for (int w = 0; w < TW; ++w) acc[w] = d4{0.0, 0.0, 0.0, 0.0};
        }
      }
#pragma unroll
      for (int w = 0; w < TW; ++w) acc[w] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv[u].v[w], acc[w], 0, 0, 0);
    }
  }
  if constexpr (PHASE) {
    flush();
#pragma unroll
    for (int w = 0; w < TW; ++w) acc[w] = tot[w];
  }
  if constexpr (ADD && PHASE) {
    if (k.out_phase) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double pr = k.out_phase[2 * (size_t)p[r]], pi = -k.out_phase[2 * (size_t)p[r] + 1];
        const double x0 = old[r].v[0] + acc[0][r];
        old[r].v[0] = 0.0;
        if constexpr (TW == 2) {
          const double x1 = old[r].v[1] + acc[1][r];
          old[r].v[1] = 0.0;
          acc[0][r] = zmul_lane(pr, pi, x0, x1, false);
          acc[1][r] = zmul_lane(pr, pi, x1, x0, true);
        } else {
          acc[0][r] = zmul_lane(pr, pi, x0, __shfl_xor(x0, 1), (col & 1) != 0);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (4 * r + kk < n && col < k.L) {
      Vec<TW> o;
#pragma unroll
      for (int w = 0; w < TW; ++w) o.v[w] = ADD ? old[ADD ? r : 0].v[w] + acc[w][r] : acc[w][r];
      stv<TW>(ADD ? k.out + (size_t)p[ADD ? r : 0] * k.L + col : k.kbuf + (size_t)(gr.row + 4 * r + kk) * k.L + col, o);
    }
  }
}

template <bool PHASE, bool ADD = false>
__device__ __forceinline__ void ket_mfma(const KetArgs& k, int b) {
  const int nlt = mfma_lane_tiles(k.L);
  if ((k.L & 31) == 0) ket_mfma_body<2, PHASE, ADD>(k, b / nlt, b % nlt);
  else ket_mfma_body<1, PHASE, ADD>(k, b / nlt, b % nlt);
}

// plain form (MFMA switched off): a wave per group, one thread per (row, lane)
__device__ __forceinline__ void ket_plain_body(const KetArgs& k, int b) {
  static_assert(KET_GROUPS == BLOCK / 64, "a group per wave");
  const int g = b * KET_GROUPS + (threadIdx.x >> 6);
  if (g < k.ngrp) {
    const KetGroup& gr = k.grp[g];
    const int n = gr.rows, ns = gr.steps;
    for (int t = threadIdx.x & 63; t < n * k.L; t += 64) {
      const int r = t / k.L, l = t - r * k.L;
      double tot = 0.0, acc = 0.0, accq = 0.0;  // accq: the other lane of the (re, im) pair
      int ent = 0;
      for (int q = 0; q <= ns; ++q) {
        const int4 s = q < ns ? k.step[gr.step + q] : make_int4(0, 0, 0, 1);
        if (k.phase && q > 0 && s.w) {
          const size_t pi2 = 2 * (size_t)(ent + r);
          tot += zmul_lane(k.phase[pi2], -k.phase[pi2 + 1], acc, accq, (l & 1) != 0);
          acc = accq = 0.0;
        }
        if (q == ns) break;
        ent = s.z;
        const double* a = k.pt + 4 * (size_t)(gr.line + q * n + r);
        const double* pj = k.proj + (size_t)s.x * k.L;
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = fma(a[j], pj[(size_t)j * k.L + l], acc);
        if (k.phase) {
#pragma unroll
          for (int j = 0; j < 4; ++j) accq = fma(a[j], pj[(size_t)j * k.L + (l ^ 1)], accq);
        }
      }
      k.kbuf[(size_t)(gr.row + r) * k.L + l] = k.phase ? tot : acc;
    }
  }
}

template <bool PHASE, bool ADD>
__global__ __launch_bounds__(BLOCK) void k_ket_mfma(const KetArgs k) { ket_mfma<PHASE, ADD>(k, blockIdx.x); }
__global__ __launch_bounds__(BLOCK) void k_ket_plain(const KetArgs k) { ket_plain_body(k, blockIdx.x); }

int launch_ket(const KetArgs& k, bool mfma, hipStream_t s) {
  const int nblock = ket_blocks(k.ngrp);
  if (nblock <= 0) return OCTHIP_SUCCESS;
  ProfScope prof("k_ket", s);
  const dim3 tiles(nblock * mfma_lane_tiles(k.L));  // 32-lane tiles when the row length allows, else 16
  if (k.out && !mfma) return fail(OCTHIP_ERR_STATE, "ket: no form that adds to the output rows");
  if (k.out && k.phase)
    hipLaunchKernelGGL((k_ket_mfma<true, true>), tiles, dim3(BLOCK), 0, s, k);
  else if (k.out)
    hipLaunchKernelGGL((k_ket_mfma<false, true>), tiles, dim3(BLOCK), 0, s, k);
  else if (mfma && k.phase)
    hipLaunchKernelGGL((k_ket_mfma<true, false>), tiles, dim3(BLOCK), 0, s, k);
  else if (mfma)
    hipLaunchKernelGGL((k_ket_mfma<false, false>), tiles, dim3(BLOCK), 0, s, k);
  else
    hipLaunchKernelGGL(k_ket_plain, dim3(nblock), dim3(BLOCK), 0, s, k);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "k_ket launch: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}

int launch_bra_reduce(const BraReduceArgs& r, hipStream_t s) {
  const int grid = bra_reduce_blocks(r);
  if (grid == 0) return OCTHIP_SUCCESS;
  ProfScope prof("k_bra_reduce", s);
  hipLaunchKernelGGL(k_bra_reduce, dim3(grid), dim3(BLOCK), 0, s, r);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "k_bra_reduce launch: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}

}  // namespace octhip

// ------------------------------------------------------- multi-segment launches --
// One launch over several (system, batch) pairs: segment i owns blocks off[i] ..
// off[i+1]-1 and its argument block args[i]; a block finds its segment by bisection over
// the (uniform) offset table.  Empty segments are skipped by taking the last segment
// whose first block is <= blockIdx.
namespace octhip {
namespace {
__device__ __forceinline__ int segment_of(const int* __restrict__ off, int nseg, int b) {
  int lo = 0, hi = nseg - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// SETS: every pair's bra goes by sets (the other form takes more registers)
template <bool SETS>
__global__ __launch_bounds__(BLOCK) void k_bra_mfma_multi(const BraMfmaArgs* __restrict__ a,
                                                          const int* __restrict__ off, int nseg) {
  const int i = segment_of(off, nseg, blockIdx.x);
  const BraMfmaArgs m = a[i];
  if (SETS || m.sets) bra_mfma<true, false>(m, blockIdx.x - off[i]);
  else bra_mfma<false, false>(m, blockIdx.x - off[i]);
}
__global__ __launch_bounds__(BLOCK) void k_bra_plain_multi(const BraMfmaArgs* __restrict__ a,
                                                           const int* __restrict__ off, int nseg) {
  const int i = segment_of(off, nseg, blockIdx.x);
  bra_plain_body(a[i].b, blockIdx.x - off[i]);
}
__global__ __launch_bounds__(BLOCK) void k_bra_reduce_multi(const BraReduceArgs* __restrict__ a,
                                                            const int* __restrict__ off, int nseg) {
  const int i = segment_of(off, nseg, blockIdx.x);
  bra_reduce_body(a[i], blockIdx.x - off[i], off[i + 1] - off[i]);
}
__global__ __launch_bounds__(BLOCK) void k_ket_mfma_multi(const KetArgs* __restrict__ a,
                                                          const int* __restrict__ off, int nseg) {
  const int i = segment_of(off, nseg, blockIdx.x);
  const KetArgs k = a[i];
  ket_mfma<false>(k, blockIdx.x - off[i]);
}
__global__ __launch_bounds__(BLOCK) void k_ket_plain_multi(const KetArgs* __restrict__ a,
                                                           const int* __restrict__ off, int nseg) {
  const int i = segment_of(off, nseg, blockIdx.x);
  ket_plain_body(a[i], blockIdx.x - off[i]);
}
__global__ __launch_bounds__(BLOCK) void k_zero_multi(const ZeroArgs* __restrict__ a,
                                                      const int* __restrict__ off, int nseg) {
  const int i = segment_of(off, nseg, blockIdx.x);
  const ZeroArgs z = a[i];
  const size_t nb = (size_t)(off[i + 1] - off[i]);
  for (size_t t = (blockIdx.x - off[i]) * (size_t)BLOCK + threadIdx.x; t < z.count; t += nb * BLOCK)
    z.f[z.first + t] = 0.0;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "%s launch: %s", what, hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}
}  // namespace

int launch_multi(int kind, const void* args, const int* off, int nseg, int nblocks, hipStream_t s, size_t lds) {
  if (nblocks <= 0) return OCTHIP_SUCCESS;
  const dim3 g(nblocks), b(BLOCK);
  switch (kind) {
    case MULTI_BRA_MFMA: {
      ProfScope prof("k_bra", s);
      hipLaunchKernelGGL(k_bra_mfma_multi<false>, g, b, lds, s, (const BraMfmaArgs*)args, off, nseg);
      return check_launch("k_bra_mfma_multi");
    }
    case MULTI_BRA_SETS: {
      ProfScope prof("k_bra", s);
      hipLaunchKernelGGL(k_bra_mfma_multi<true>, g, b, lds, s, (const BraMfmaArgs*)args, off, nseg);
      return check_launch("k_bra_mfma_multi");
    }
    case MULTI_BRA_PLAIN: {
      ProfScope prof("k_bra", s);
      hipLaunchKernelGGL(k_bra_plain_multi, g, b, 0, s, (const BraMfmaArgs*)args, off, nseg);
      return check_launch("k_bra_plain_multi");
    }
    case MULTI_BRA_REDUCE: {
      ProfScope prof("k_bra_reduce", s);
      hipLaunchKernelGGL(k_bra_reduce_multi, g, b, 0, s, (const BraReduceArgs*)args, off, nseg);
      return check_launch("k_bra_reduce_multi");
    }
    case MULTI_KET_MFMA: {
      ProfScope prof("k_ket", s);
      hipLaunchKernelGGL(k_ket_mfma_multi, g, b, 0, s, (const KetArgs*)args, off, nseg);
      return check_launch("k_ket_mfma_multi");
    }
    case MULTI_KET_PLAIN: {
      ProfScope prof("k_ket", s);
      hipLaunchKernelGGL(k_ket_plain_multi, g, b, 0, s, (const KetArgs*)args, off, nseg);
      return check_launch("k_ket_plain_multi");
    }
    case MULTI_ZERO: {
      ProfScope prof("k_zero_rows", s);
      hipLaunchKernelGGL(k_zero_multi, g, b, 0, s, (const ZeroArgs*)args, off, nseg);
      return check_launch("k_zero_multi");
    }
    default:
      return fail(OCTHIP_ERR_INVALID, "unknown multi-segment kernel %d", kind);
  }
}
}  // namespace octhip
