// Batched mesh reductions on packed batches (mesh_batch_dotp_vector, mesh_batch_nrm2:
// src/grid/mesh_batch_inc.F90:379-549, 970-1274), the Gram-Schmidt passes of
// mesh_batch_orthogonalization and of the Lanczos exponential, and the elementwise passes of the
// Chebyshev exponential (src/electrons/exponential.F90:766-971); csrc/krylov.hip drives them.
//
// Dot products are deterministic two-stage sums: every workgroup sums a fixed set of rows
// per state column (rows p = b*G + g, b*G + g + nblk*G, ... for its G row groups, then the
// G groups in order through LDS) into one partial per (workgroup, column); a second kernel
// adds the partials in a fixed order and scales by the volume element.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <mutex>
#include <vector>

#include "kernels.h"

namespace octhip {

namespace {

constexpr int DOT_BLOCKS = 512;   // workgroups of the first stage (partials per column)

// columns of a row: complex states (lane pairs) or real lanes
struct Cols {
  int n;   // columns per row
  int cw;  // columns handled side by side by the threads of a workgroup (<= BLOCK)
  int g;   // row groups per workgroup = BLOCK / cw
  int per; // columns per thread = n / cw
};
Cols cols_of(int L, int is_complex) {
  Cols c;
  c.n = is_complex ? L / 2 : L;
  c.cw = std::min(c.n, BLOCK);
  c.g = BLOCK / c.cw;
  c.per = c.n / c.cw;
  return c;
}

// partial[b][c] = sum over the rows of workgroup b of conj(a) * b (complex: two doubles)
__global__ __launch_bounds__(BLOCK) void k_dotp_partial(const double* __restrict__ a, const double* __restrict__ bb,
                                                        int L, int np, int is_complex, int cw, int per,
                                                        double* __restrict__ partial) {
  __shared__ double sre[BLOCK * 4], sim[BLOCK * 4];
  const int G = BLOCK / cw;
  const int c0 = threadIdx.x % cw, g = threadIdx.x / cw;
  const int lsh = __builtin_ctz((unsigned)L);
  double re[4] = {0, 0, 0, 0}, im[4] = {0, 0, 0, 0};
  for (int p = blockIdx.x * G + g; p < np; p += gridDim.x * G) {
    const double* ra = a + ((size_t)p << lsh);
    const double* rb = bb + ((size_t)p << lsh);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k >= per) break;
      const int c = c0 + k * cw;
      if (is_complex) {
        const double ar = ra[2 * c], ai = ra[2 * c + 1], br = rb[2 * c], bi = rb[2 * c + 1];
        re[k] = re[k] + (ar * br + ai * bi);
        im[k] = im[k] + (ar * bi - ai * br);
      } else {
        re[k] = re[k] + ra[c] * rb[c];
      }
    }
  }
  for (int k = 0; k < per && k < 4; ++k) {
    sre[k * BLOCK + threadIdx.x] = re[k];
    sim[k * BLOCK + threadIdx.x] = im[k];
  }
  __syncthreads();
  // column c = c0 + k*cw: sum its G row groups in order
  for (int t = threadIdx.x; t < cw * per; t += BLOCK) {
    const int k = t / cw, cc = t % cw;
    double r = 0.0, i = 0.0;
    for (int gg = 0; gg < G; ++gg) {
      r = r + sre[k * BLOCK + gg * cw + cc];
      i = i + sim[k * BLOCK + gg * cw + cc];
    }
    const int c = cc + k * cw;
    partial[((size_t)blockIdx.x * (cw * per) + c) * 2] = r;
    partial[((size_t)blockIdx.x * (cw * per) + c) * 2 + 1] = i;
  }
}

// out[c] = vol * sum_b partial[b][c] (complex pairs): FIN_G threads per column take every
// FIN_G-th workgroup's partial, then add their sums in order.  One thread per column, a chain of
// 512 dependent additions in a single workgroup, took 122 us for 32 columns; this takes 4 us.
constexpr int FIN_W = 16, FIN_G = 64;  // columns of a workgroup, threads per column
__device__ __forceinline__ void sum_partials(const double* __restrict__ partial, int nblk, int ncol, int c0,
                                             double& re, double& im, double2 (*sh)[FIN_W]) {
  const int w = threadIdx.x % FIN_W, g = threadIdx.x / FIN_W;
  const int c = min(c0 + w, ncol - 1);
  double2 s = make_double2(0.0, 0.0);
  for (int b = g; b < nblk; b += 4 * FIN_G) {
    double2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = reinterpret_cast<const double2*>(partial)[(size_t)min(b + u * FIN_G, nblk - 1) * ncol + c];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (b + u * FIN_G < nblk) {
        s.x = s.x + v[u].x;
        s.y = s.y + v[u].y;
      }
  }
  sh[g][w] = s;
  __syncthreads();
  re = im = 0.0;
  if (g == 0)
    for (int k = 0; k < FIN_G; ++k) {
      re = re + sh[k][w].x;
      im = im + sh[k][w].y;
    }
}

__global__ __launch_bounds__(FIN_W * FIN_G) void k_dotp_final(const double* __restrict__ partial, int nblk, int ncol,
                                                             double vol, double* __restrict__ out) {
  __shared__ double2 sh[FIN_G][FIN_W];
  double re, im;
  sum_partials(partial, nblk, ncol, blockIdx.x * FIN_W, re, im, sh);
  const int c = blockIdx.x * FIN_W + threadIdx.x;
  if (threadIdx.x < FIN_W && c < ncol) {
    out[2 * c] = vol * re;
    out[2 * c + 1] = vol * im;
  }
}

// ---- Gram-Schmidt passes over complex rows (the mesh inner product, per state column) ----
// A workgroup's threads lie side by side over cw columns of its G row groups, as in
// k_dotp_partial; a thread keeps to its columns, so factors are formed once per thread.
// Both passes run at memory speed (two rows per thread in flight, 16-byte pieces): overlaps with
// 4 vectors of 80 MB 77 us (5.1 TB/s), their subtraction with the norm 85 us (5.6 TB/s); with 2
// vectors of 35 MB, from the Infinity Cache, 17 and 22 us (6.1, 6.5 TB/s).
constexpr int GS_MAX = 4;  // vectors per pass
struct GsVecs {
  const double* x[GS_MAX];
};

// partial[b][v * ncol + c] = sum over the rows of workgroup b of conj(x_v) y.  y is read once
// for all vectors (one launch and one pass over y per vector before).
template <int NV>
__global__ __launch_bounds__(BLOCK) void k_gs_dots(const GsVecs xs, const double* __restrict__ y, int L, int np, int cw,
                                                   int per, double* __restrict__ partial) {
  __shared__ double2 sh[NV][BLOCK];
  const int G = BLOCK / cw, ncol = cw * per;
  const int c0 = threadIdx.x % cw, g = threadIdx.x / cw;
  const size_t half = (size_t)L >> 1;
  for (int k = 0; k < per; ++k) {
    const int c = c0 + k * cw;
    double2 s[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) s[v] = make_double2(0.0, 0.0);
    const int step = gridDim.x * G;
    for (int p = blockIdx.x * G + g; p < np; p += 2 * step) {
      // two rows in flight; the second one clamped and left out past the end
      const bool two = p + step < np;
      const size_t o0 = (size_t)p * half + c, o1 = (size_t)(two ? p + step : p) * half + c;
      const double2 y0 = reinterpret_cast<const double2*>(y)[o0], y1 = reinterpret_cast<const double2*>(y)[o1];
      double2 a0[NV], a1[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        a0[v] = reinterpret_cast<const double2*>(xs.x[v])[o0];
        a1[v] = reinterpret_cast<const double2*>(xs.x[v])[o1];
      }
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        s[v].x = s[v].x + (a0[v].x * y0.x + a0[v].y * y0.y);
        s[v].y = s[v].y + (a0[v].x * y0.y - a0[v].y * y0.x);
        if (two) {
          s[v].x = s[v].x + (a1[v].x * y1.x + a1[v].y * y1.y);
          s[v].y = s[v].y + (a1[v].x * y1.y - a1[v].y * y1.x);
        }
      }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) sh[v][threadIdx.x] = s[v];
    __syncthreads();
    if (g < NV) {  // row group v adds vector v's G groups in order (G may be smaller than NV)
      for (int v = g; v < NV; v += G) {
        double2 t = make_double2(0.0, 0.0);
        for (int gg = 0; gg < G; ++gg) {
          t.x = t.x + sh[v][gg * cw + c0].x;
          t.y = t.y + sh[v][gg * cw + c0].y;
        }
        reinterpret_cast<double2*>(partial)[(size_t)blockIdx.x * (NV * ncol) + v * ncol + c] = t;
      }
    }
    __syncthreads();
  }
}

// y = scale[c] y + sum_v coef[v][c] x_v (terms in order; no scaling when scale is null) over the
// np rows, and, when partial is given, partial[b][c] = sum over the rows of workgroup b of |y|^2:
// the subtractions of a Gram-Schmidt step and the norm in one pass over y.  src: read y from
// there (null: in place).
template <int NV>
__global__ __launch_bounds__(BLOCK) void k_gs_update(double* y, const double* src, const GsVecs xs, int L,
                                                     int np, int cw, int per, const double2* __restrict__ scale,
                                                     const double2* __restrict__ coef, double* __restrict__ partial) {
  __shared__ double sh[BLOCK];
  const int G = BLOCK / cw, ncol = cw * per;
  const int c0 = threadIdx.x % cw, g = threadIdx.x / cw;
  const size_t half = (size_t)L >> 1;
  const double2* const in = reinterpret_cast<const double2*>(src ? src : y);
  for (int k = 0; k < per; ++k) {
    const int c = c0 + k * cw;
    double2 f[NV > 0 ? NV : 1];
#pragma unroll
    for (int v = 0; v < NV; ++v) f[v] = coef[(size_t)v * ncol + c];
    const double2 sc = scale ? scale[c] : make_double2(1.0, 0.0);
    double s = 0.0;
    const int step = gridDim.x * G;
    for (int p = blockIdx.x * G + g; p < np; p += 2 * step) {
      const bool two = p + step < np;
      const size_t o[2] = {(size_t)p * half + c, (size_t)(two ? p + step : p) * half + c};
      double2 yv[2], xv[2][NV > 0 ? NV : 1];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        yv[u] = in[o[u]];
#pragma unroll
        for (int v = 0; v < NV; ++v) xv[u][v] = reinterpret_cast<const double2*>(xs.x[v])[o[u]];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (u == 1 && !two) break;
        double2 t = yv[u];
        if (scale) t = make_double2(sc.x * yv[u].x - sc.y * yv[u].y, sc.x * yv[u].y + sc.y * yv[u].x);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          t.x = t.x + (f[v].x * xv[u][v].x - f[v].y * xv[u][v].y);
          t.y = t.y + (f[v].x * xv[u][v].y + f[v].y * xv[u][v].x);
        }
        reinterpret_cast<double2*>(y)[o[u]] = t;
        s = s + (t.x * t.x + t.y * t.y);
      }
    }
    if (partial) {
      sh[threadIdx.x] = s;
      __syncthreads();
      if (g == 0) {
        double t = 0.0;
        for (int gg = 0; gg < G; ++gg) t = t + sh[gg * cw + c0];
        reinterpret_cast<double2*>(partial)[(size_t)blockIdx.x * ncol + c] = make_double2(t, 0.0);
      }
      __syncthreads();
    }
  }
}

// Results and factors of a Gram-Schmidt step, one thread per column.  The vectors are kept with
// norms nrm (1: normalised, or null): x_v = n_v times the unit vector, y = n_y H u.
//   overlaps: ov[v][c] = vol sum / (n_v n_y);  coef[v][c] = -ov[v][c] / n_v;  scale[c] = 1 / n_y
//   (columns >= nst: 0 and 1)
__global__ __launch_bounds__(FIN_W * FIN_G) void k_gs_coefs(const double* __restrict__ partial, int nblk, int ncol,
                                                            int nst, double vol, const double* __restrict__ nx,
                                                            const double* __restrict__ ny, double2* __restrict__ ov,
                                                            double2* __restrict__ coef, double2* __restrict__ scale) {
  __shared__ double2 sh[FIN_G][FIN_W];
  const int v = blockIdx.y, nv = gridDim.y;
  double re, im;
  const int cc = blockIdx.x * FIN_W;
  // the nv vectors' columns lie side by side in a workgroup's partials
  sum_partials(partial, nblk, nv * ncol, v * ncol + cc, re, im, sh);
  const int c = cc + threadIdx.x;
  if (threadIdx.x >= FIN_W || c >= ncol) return;
  const double n0 = nx ? nx[(size_t)v * ncol + c] : 1.0, n1 = ny ? ny[c] : 1.0;
  double2 o = make_double2(vol * re, vol * im);
  if (nx) {
    const double d = n0 * n1;
    o.x = o.x / d;
    o.y = o.y / d;
  }
  const bool on = c < nst;
  ov[(size_t)v * ncol + c] = o;
  coef[(size_t)v * ncol + c] = on ? (nx ? make_double2(-o.x / n0, -o.y / n0) : make_double2(-o.x, -o.y)) : make_double2(0.0, 0.0);
  if (scale && v == 0) scale[c] = make_double2(on && ny ? 1.0 / n1 : 1.0, 0.0);
}

__global__ __launch_bounds__(BLOCK) void k_gs_factors(const double2* __restrict__ ov, int nv, int ncol, int nst,
                                                      double2* __restrict__ coef) {
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  if (i < nv * ncol) coef[i] = i % ncol < nst ? make_double2(-ov[i].x, -ov[i].y) : make_double2(0.0, 0.0);
}

// norm[c] = sqrt(vol sum_b partial), the norm a Krylov vector is kept with (norms below tiny
// count as 1, columns >= nst have 1), and 1 / norm
__global__ __launch_bounds__(FIN_W * FIN_G) void k_gs_norms(const double* __restrict__ partial, int nblk, int ncol,
                                                            int nst, double vol, double tiny, double* __restrict__ norm,
                                                            double* __restrict__ kept, double2* __restrict__ inv) {
  __shared__ double2 sh[FIN_G][FIN_W];
  double re, im;
  sum_partials(partial, nblk, ncol, blockIdx.x * FIN_W, re, im, sh);
  const int c = blockIdx.x * FIN_W + threadIdx.x;
  if (threadIdx.x >= FIN_W || c >= ncol) return;
  const double n = sqrt(vol * re);
  norm[c] = n;
  if (kept) kept[c] = c < nst && !(fabs(n) < tiny) ? n : 1.0;
  if (inv) inv[c] = make_double2(c < nst ? 1.0 / n : 1.0, 0.0);
}

// Chebyshev update in the reference's operation order (exponential.F90:940-947):
// t = Hpsi1 + (-mid) psi1; t = t * (2/span); t = t + zfact psib; t = t + (-1) psi2
__global__ __launch_bounds__(BLOCK) void k_cheby_update(double* __restrict__ out, const double* __restrict__ psi1,
                                                        const double* __restrict__ b, const double* __restrict__ psi2,
                                                        size_t count, double mmid, double two_span, double zr,
                                                        double zi) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    double t = out[i] + mmid * psi1[i];
    t = t * two_span;
    t = t + zmul_lane(zr, zi, b[i], b[i ^ 1], (i & 1) != 0);
    out[i] = t + (-1.0) * psi2[i];
  }
}

// psib = (psi0 + (-1) psi2) * z  (exponential.F90:950-952)
__global__ __launch_bounds__(BLOCK) void k_cheby_final(double* __restrict__ psib, const double* __restrict__ psi0,
                                                       const double* __restrict__ psi2, size_t count, double zr,
                                                       double zi) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    if (i & 1) continue;
    const double tr = psi0[i] + (-1.0) * psi2[i];
    const double ti = psi0[i + 1] + (-1.0) * psi2[i + 1];
    psib[i] = zr * tr - zi * ti;
    psib[i + 1] = zr * ti + zi * tr;
  }
}

unsigned grid_for(size_t count) { return (unsigned)std::min<size_t>((count + BLOCK - 1) / BLOCK, 8192); }

}  // namespace

// Scratch bytes of a dot product of rows of L doubles: DOT_BLOCKS partials + the result.
size_t dotp_scratch_bytes(int L, int is_complex) {
  const Cols c = cols_of(L, is_complex);
  return sizeof(double) * 2 * ((size_t)DOT_BLOCKS * c.n + c.n);
}

// dot[c] = vol * sum_p conj(a(p, c)) b(p, c): partials in scratch, the ncol complex results
// in dest (device) or, when dest is null, at the end of scratch; *result = their address.
int launch_dotp(const double* a, const double* b, int L, int np, int is_complex, double vol, double* scratch,
                hipStream_t s, double** result, double* dest) {
  const Cols c = cols_of(L, is_complex);
  if (c.per > 4) return fail(OCTHIP_ERR_UNSUPPORTED, "dot product: more than %d columns", 4 * BLOCK);
  double* partial = scratch;
  double* out = dest ? dest : scratch + (size_t)2 * DOT_BLOCKS * c.n;
  const int nblk = std::max(1, std::min(DOT_BLOCKS, (np + c.g - 1) / c.g));
  ProfScope prof("k_dotp", s);
  hipLaunchKernelGGL(k_dotp_partial, dim3(nblk), dim3(BLOCK), 0, s, a, b, L, np, is_complex, c.cw, c.per, partial);
  OCTHIP_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_dotp_final, dim3((c.n + FIN_W - 1) / FIN_W), dim3(FIN_W * FIN_G), 0, s, partial, nblk, c.n, vol,
                     out);
  OCTHIP_HIP(hipGetLastError());
  *result = out;
  return OCTHIP_SUCCESS;
}

// workgroups of a Gram-Schmidt pass over np complex rows of L doubles (partials per column)
static int gs_blocks(const Cols& c, int np) { return std::max(1, std::min(DOT_BLOCKS, (np + c.g - 1) / c.g)); }

size_t gs_scratch_bytes(int L) { return sizeof(double) * 2 * (size_t)DOT_BLOCKS * (L / 2) * GS_MAX; }

// ov[v][c] = <x_v|y> / (n_v n_y) of the nv vectors and the factors that subtract them from y
// (k_gs_coefs); partials in scratch (gs_scratch_bytes)
int launch_gs_dots(const double* const* x, int nv, const double* y, int L, int np, int nst, double vol,
                   const double* nx, const double* ny, double* scratch, double* ov, double* coef, double* scale,
                   hipStream_t s) {
  const Cols c = cols_of(L, 1);
  const int nblk = gs_blocks(c, np);
  GsVecs xs{};
  for (int v = 0; v < nv; ++v) xs.x[v] = x[v];
  ProfScope prof("k_dotp", s);
  switch (nv) {
    case 1: hipLaunchKernelGGL(k_gs_dots<1>, dim3(nblk), dim3(BLOCK), 0, s, xs, y, L, np, c.cw, c.per, scratch); break;
    case 2: hipLaunchKernelGGL(k_gs_dots<2>, dim3(nblk), dim3(BLOCK), 0, s, xs, y, L, np, c.cw, c.per, scratch); break;
    case 3: hipLaunchKernelGGL(k_gs_dots<3>, dim3(nblk), dim3(BLOCK), 0, s, xs, y, L, np, c.cw, c.per, scratch); break;
    case 4: hipLaunchKernelGGL(k_gs_dots<4>, dim3(nblk), dim3(BLOCK), 0, s, xs, y, L, np, c.cw, c.per, scratch); break;
    default: return fail(OCTHIP_ERR_INVALID, "Gram-Schmidt pass over %d vectors", nv);
  }
  OCTHIP_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_gs_coefs, dim3((c.n + FIN_W - 1) / FIN_W, nv), dim3(FIN_W * FIN_G), 0, s, scratch, nblk, c.n, nst,
                     vol, nx, ny, reinterpret_cast<double2*>(ov), reinterpret_cast<double2*>(coef),
                     reinterpret_cast<double2*>(scale));
  OCTHIP_HIP(hipGetLastError());
  return OCTHIP_SUCCESS;
}

// y = scale y + sum_v coef[v] x_v per column (src: y read from there); with partial, the |y|^2
// partials that launch_gs_norms sums
int launch_gs_update(double* y, const double* src, const double* const* x, int nv, int L, int np, const double* scale,
                     const double* coef, double* partial, hipStream_t s) {
  const Cols c = cols_of(L, 1);
  const int nblk = gs_blocks(c, np);
  GsVecs xs{};
  for (int v = 0; v < nv; ++v) xs.x[v] = x[v];
  const double2* const sc = reinterpret_cast<const double2*>(scale);
  const double2* const cf = reinterpret_cast<const double2*>(coef);
  ProfScope prof("k_gs_update", s);
  switch (nv) {
    case 0: hipLaunchKernelGGL(k_gs_update<0>, dim3(nblk), dim3(BLOCK), 0, s, y, src, xs, L, np, c.cw, c.per, sc, cf, partial); break;
    case 1: hipLaunchKernelGGL(k_gs_update<1>, dim3(nblk), dim3(BLOCK), 0, s, y, src, xs, L, np, c.cw, c.per, sc, cf, partial); break;
    case 2: hipLaunchKernelGGL(k_gs_update<2>, dim3(nblk), dim3(BLOCK), 0, s, y, src, xs, L, np, c.cw, c.per, sc, cf, partial); break;
    case 3: hipLaunchKernelGGL(k_gs_update<3>, dim3(nblk), dim3(BLOCK), 0, s, y, src, xs, L, np, c.cw, c.per, sc, cf, partial); break;
    case 4: hipLaunchKernelGGL(k_gs_update<4>, dim3(nblk), dim3(BLOCK), 0, s, y, src, xs, L, np, c.cw, c.per, sc, cf, partial); break;
    default: return fail(OCTHIP_ERR_INVALID, "Gram-Schmidt pass over %d vectors", nv);
  }
  OCTHIP_HIP(hipGetLastError());
  return OCTHIP_SUCCESS;
}

// coef[v][c] = -ov[v][c] (columns >= nst: 0)
int launch_gs_factors(const double* ov, int nv, int ncol, int nst, double* coef, hipStream_t s) {
  hipLaunchKernelGGL(k_gs_factors, dim3((nv * ncol + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s,
                     reinterpret_cast<const double2*>(ov), nv, ncol, nst, reinterpret_cast<double2*>(coef));
  OCTHIP_HIP(hipGetLastError());
  return OCTHIP_SUCCESS;
}

int launch_gs_norms(const double* partial, int L, int np, int nst, double vol, double tiny, double* norm, double* kept,
                    double* inv, hipStream_t s) {
  const Cols c = cols_of(L, 1);
  hipLaunchKernelGGL(k_gs_norms, dim3((c.n + FIN_W - 1) / FIN_W), dim3(FIN_W * FIN_G), 0, s, partial, gs_blocks(c, np),
                     c.n, nst, vol, tiny, norm, kept, reinterpret_cast<double2*>(inv));
  OCTHIP_HIP(hipGetLastError());
  return OCTHIP_SUCCESS;
}

int launch_cheby_update(double* out, const double* psi1, const double* b, const double* psi2, size_t count,
                        double mid, double span, std::complex<double> z, hipStream_t s) {
  hipLaunchKernelGGL(k_cheby_update, dim3(grid_for(count)), dim3(BLOCK), 0, s, out, psi1, b, psi2, count, -mid,
                     2.0 / span, z.real(), z.imag());
  OCTHIP_HIP(hipGetLastError());
  return OCTHIP_SUCCESS;
}

int launch_cheby_final(double* psib, const double* psi0, const double* psi2, size_t count, std::complex<double> z,
                       hipStream_t s) {
  hipLaunchKernelGGL(k_cheby_final, dim3(grid_for(count)), dim3(BLOCK), 0, s, psib, psi0, psi2, count, z.real(),
                     z.imag());
  OCTHIP_HIP(hipGetLastError());
  return OCTHIP_SUCCESS;
}

}  // namespace octhip

using namespace octhip;

extern "C" int octhip_mesh_batch_dotp_vector(const double* a, const double* b, int ldf, int np, int is_complex,
                                             double vol, double* dot, void* stream) {
  OCTHIP_RANGE("octhip_mesh_batch_dotp_vector");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(a && b && dot, "null argument");
  OCTHIP_REQUIRE(ldf >= (is_complex ? 1 : 0) && ldf <= MAX_LDF, "ldf=%d outside the packed range", ldf);
  OCTHIP_REQUIRE(np >= 0, "np < 0");
  const int L = 1 << ldf;
  const size_t bytes = dotp_scratch_bytes(L, is_complex);
  Scratch scratch_buf;
  int rc = scratch_buf.get(bytes);
  if (rc) return rc;
  double* const scratch = static_cast<double*>(scratch_buf.ptr());
  hipStream_t s = (hipStream_t)stream;
  double* res = nullptr;
  rc = launch_dotp(a, b, L, np, is_complex, vol, scratch, s, &res, nullptr);
  const int n = is_complex ? L / 2 : L;
  std::vector<double> host(2 * (size_t)n);
  if (!rc) {
    hipError_t e = hipMemcpyAsync(host.data(), res, sizeof(double) * 2 * n, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) rc = fail(OCTHIP_ERR_HIP, "mesh_batch_dotp_vector: %s", hipGetErrorString(e));
  }
  if (rc) {
    (void)hipStreamSynchronize(s);  // nothing may use the buffer once it is back in the pool
    return rc;
  }
  // complex results as (re, im) pairs, real ones as one double per lane
  for (int c = 0; c < n; ++c) {
    if (is_complex) {
      dot[2 * c] = host[2 * c];
      dot[2 * c + 1] = host[2 * c + 1];
    } else {
      dot[c] = host[2 * c];
    }
  }
  return OCTHIP_SUCCESS;
}


// ------------------------------------------------------------ no allocation --
// octhip_mesh_batch_dotp_vector without any allocation: the partials and the results go
// to a fixed device array of this library instead of a per-call buffer.  Its capacity is
// the largest row the library handles (2^MAX_LDF real lanes), 8 MiB + 16 KiB.
namespace {
constexpr size_t NOALLOC_DOUBLES = 2 * ((size_t)DOT_BLOCKS * (1 << MAX_LDF) + (1 << MAX_LDF));
__device__ __align__(256) double scratch[NOALLOC_DOUBLES];

// device address of `scratch` on each device, looked up once with that device current
// (in host code the array's name is not a device address)
constexpr int MAX_DEVICES = 64;
double* scratch_ptr[MAX_DEVICES] = {};
std::mutex scratch_mu;

int scratch_of_current_device(double** out) {
  int dev = 0;
  OCTHIP_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= MAX_DEVICES) return fail(OCTHIP_ERR_UNSUPPORTED, "device %d beyond %d", dev, MAX_DEVICES);
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = scratch_ptr[dev];
  return OCTHIP_SUCCESS;
}
}  // namespace

extern "C" int octhip_mesh_batch_dotp_vector_noalloc(const double* a, const double* b, int ldf, int np, int is_complex,
                                                     double vol, double* dot, void* stream) {
  OCTHIP_RANGE("octhip_mesh_batch_dotp_vector_noalloc");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(a && b && dot, "null argument");
  OCTHIP_REQUIRE(ldf >= (is_complex ? 1 : 0) && ldf <= MAX_LDF, "ldf=%d outside the packed range", ldf);
  OCTHIP_REQUIRE(np >= 0, "np < 0");
  const int L = 1 << ldf;
  OCTHIP_REQUIRE(dotp_scratch_bytes(L, is_complex) <= sizeof(double) * NOALLOC_DOUBLES,
                 "rows of %d doubles need %zu bytes of scratch, more than the %zu available", L,
                 dotp_scratch_bytes(L, is_complex), sizeof(double) * NOALLOC_DOUBLES);
  double* sp = nullptr;
  int rc = scratch_of_current_device(&sp);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  // results as (re, im) pairs straight into the caller's device array (im = 0 for real rows)
  double* res = nullptr;
  return launch_dotp(a, b, L, np, is_complex, vol, sp, s, &res, dot);
}
