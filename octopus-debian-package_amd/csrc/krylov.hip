// Lanczos and Chebyshev exponentials of a packed complex batch
// (exponential_lanczos_batch / exponential_cheby_batch, src/electrons/exponential.F90:766-971)
// and the mesh reductions they use (mesh_batch_nrm2, mesh_batch_orthogonalization,
// src/grid/mesh_batch_inc.F90:970-1274).
//
// The Krylov vectors, the Chebyshev recurrence buffers and the small per-state buffers live
// in a set per (Hamiltonian, stream), like the H-apply's work sets.  The small projected
// problems are solved on the host: the Lanczos matrix of a Hermitian H is Hermitian
// tridiagonal (zheev reads its upper triangle, exponential.F90:829-836), which a diagonal
// unitary turns into a real symmetric tridiagonal matrix; its eigenpairs come from the
// implicit QL iteration with Wilkinson shifts (the tql2 algorithm).
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <vector>

#include "kernels.h"

namespace octhip {
size_t gs_scratch_bytes(int L);
int launch_gs_dots(const double* const* x, int nv, const double* y, int L, int np, int nst, double vol,
                   const double* nx, const double* ny, double* scratch, double* ov, double* coef, double* scale,
                   hipStream_t s);
int launch_gs_update(double* y, const double* src, const double* const* x, int nv, int L, int np, const double* scale,
                     const double* coef, double* partial, hipStream_t s);
int launch_gs_norms(const double* partial, int L, int np, int nst, double vol, double tiny, double* norm, double* kept,
                    double* inv, hipStream_t s);
int launch_gs_factors(const double* ov, int nv, int ncol, int nst, double* coef, hipStream_t s);
int launch_cheby_update(double* out, const double* psi1, const double* b, const double* psi2, size_t count,
                        double mid, double span, std::complex<double> z, hipStream_t s);
int launch_cheby_final(double* psib, const double* psi0, const double* psi2, size_t count, std::complex<double> z,
                       hipStream_t s);
}  // namespace octhip

using namespace octhip;
using cplx = std::complex<double>;

namespace {

constexpr int GS_MAX = 4;        // vectors per Gram-Schmidt pass (csrc/mesh_batch.hip)
constexpr int KCOLS = 1 << (MAX_LDF - 1);  // most complex states of a row

// Device buffers of one stream: nvec batches of np_part rows (Krylov vectors or the
// Chebyshev recurrence) and a small block, in doubles:
//   res    K_RES    overlaps of a step with two vectors (complex), then the norm: one copy to host
//   coef   K_COEF   factors of up to GS_MAX vectors, then `scale`, the scaling (complex)
//   kept   K_KEPT   the norms the two latest Krylov vectors are kept with, by parity
//   part            partial sums
// host is the pinned copy of res, ready an event behind that copy.
struct KrylovBufs {
  double* vec = nullptr;
  double *res = nullptr, *coef = nullptr, *scale = nullptr, *kept = nullptr, *part = nullptr;
  double* host = nullptr;
  hipEvent_t ready = nullptr;
};
constexpr size_t K_RES = 5 * KCOLS, K_COEF = 2 * KCOLS * (GS_MAX + 1), K_KEPT = 2 * KCOLS;

int krylov_bufs(octhip_hamiltonian_s* h, hipStream_t s, int nvec, int ldf, KrylovBufs* out) {
  const size_t L = (size_t)1 << ldf;
  const size_t vec_bytes = sizeof(double) * (size_t)h->kin->np_part * L * nvec;
  const size_t small_bytes = sizeof(double) * (K_RES + K_COEF + K_KEPT) + gs_scratch_bytes(1 << MAX_LDF) / 2;
  octhip_hamiltonian_s::KrylovSet* k = nullptr;
  for (auto& e : h->krylov)
    if (e.s == s) k = &e;
  if (!k) {
    h->krylov.push_back({s, nullptr, 0, nullptr, nullptr, nullptr});
    k = &h->krylov.back();
  }
  if (k->bytes < vec_bytes) {
    dfree(k->vec);
    k->vec = nullptr;
    k->bytes = 0;
    int rc = dalloc((void**)&k->vec, vec_bytes);
    if (rc) return rc;
    k->bytes = vec_bytes;
  }
  if (!k->small) {
    int rc = dalloc((void**)&k->small, small_bytes);
    if (rc) return rc;
  }
  if (!k->host) {
    int rc = halloc((void**)&k->host, sizeof(double) * K_RES);
    if (rc) return rc;
  }
  if (!k->ready) OCTHIP_HIP(hipEventCreateWithFlags(&k->ready, hipEventDisableTiming));
  out->vec = k->vec;
  out->res = k->small;
  out->coef = out->res + K_RES;
  out->scale = out->coef + 2 * KCOLS * GS_MAX;
  out->kept = out->coef + K_COEF;
  out->part = out->kept + K_KEPT;
  out->host = k->host;
  out->ready = k->ready;
  return OCTHIP_SUCCESS;
}

// factors of the nv vectors (states nst.. of the row get 0) and the scaling (1) to the device;
// `host` holds them and has to live until the copies are done
int upload_factors(const std::vector<cplx>& c, int nv, int nst, int ncol, const std::vector<cplx>* scale, double* coef,
                   double* dscale, std::vector<double>& host, hipStream_t s) {
  host.resize(2 * (size_t)ncol * (nv + 1));
  for (int v = 0; v <= nv; ++v)
    for (int i = 0; i < ncol; ++i) {
      const cplx z = v < nv ? (i < nst ? c[(size_t)v * nst + i] : cplx(0.0))
                            : (scale && i < nst ? (*scale)[i] : cplx(1.0));
      host[2 * ((size_t)v * ncol + i)] = z.real();
      host[2 * ((size_t)v * ncol + i) + 1] = z.imag();
    }
  if (nv > 0)
    OCTHIP_HIP(hipMemcpyAsync(coef, host.data(), sizeof(double) * 2 * ncol * nv, hipMemcpyHostToDevice, s));
  OCTHIP_HIP(hipMemcpyAsync(dscale, host.data() + 2 * (size_t)ncol * nv, sizeof(double) * 2 * ncol,
                            hipMemcpyHostToDevice, s));
  return OCTHIP_SUCCESS;
}

// Eigenpairs of the real symmetric tridiagonal matrix (diagonal d[0..n-1], off-diagonal
// e[0..n-2]): implicit QL with Wilkinson shifts (tql2).  z[k*nc + c] = component comp[c] of
// eigenvector k, starting as the identity; a rotation treats every component alike, so a
// caller pays for those it asks for (the components of a vector side by side: rotations of
// all n take the host's vector units).
bool tridiagonal_eigen(int n, std::vector<double>& d, std::vector<double> e, const int* comp, int nc,
                       std::vector<double>& z) {
  z.assign((size_t)n * nc, 0.0);
  for (int c = 0; c < nc; ++c) z[(size_t)comp[c] * nc + c] = 1.0;
  e.resize(n);
  e[n - 1] = 0.0;
  for (int l = 0; l < n; ++l) {
    int iter = 0;
    int m;
    do {
      for (m = l; m < n - 1; ++m) {
        const double dd = std::fabs(d[m]) + std::fabs(d[m + 1]);
        if (std::fabs(e[m]) <= 1e-16 * dd) break;
      }
      if (m != l) {
        if (++iter > 100) return false;
        double g = (d[l + 1] - d[l]) / (2.0 * e[l]);
        double r = std::hypot(g, 1.0);
        g = d[m] - d[l] + e[l] / (g + std::copysign(r, g));
        double sn = 1.0, c = 1.0, p = 0.0;
        int i;
        for (i = m - 1; i >= l; --i) {
          double f = sn * e[i];
          const double b = c * e[i];
          r = std::hypot(f, g);
          e[i + 1] = r;
          if (r == 0.0) {
            d[i + 1] -= p;
            e[m] = 0.0;
            break;
          }
          sn = f / r;
          c = g / r;
          g = d[i + 1] - p;
          r = (d[i] - g) * sn + 2.0 * c * b;
          p = sn * r;
          d[i + 1] = g + p;
          g = c * r - b;
          double* const z0 = z.data() + (size_t)i * nc;
          double* const z1 = z0 + nc;
          for (int k = 0; k < nc; ++k) {
            const double t = z1[k];
            z1[k] = sn * z0[k] + c * t;
            z0[k] = c * z0[k] - sn * t;
          }
        }
        if (r == 0.0 && i >= l) continue;
        d[l] -= p;
        e[l] = g;
        e[m] = 0.0;
      }
    } while (m != l);
  }
  return true;
}

// First column of f(pp * A) for the n x n Hermitian matrix whose upper triangle is
// hm(i, j) = a[i + j*ld] (tridiagonal: the diagonal and the first superdiagonal are read),
// f = exp or phi(x) = (e^x - 1)/x (zlalg_exp / zlalg_phi, src/math/lalg_adv.F90:216-340).
// last: only its last component, which is all that a residual takes.
bool krylov_function(int n, const cplx* a, int ld, cplx pp, bool phi, bool last, cplx* col) {
  std::vector<double> d(n), e(std::max(n - 1, 0));
  std::vector<cplx> ph(n);  // D = diag(ph): A = D T D^H with T real
  ph[0] = 1.0;
  for (int k = 0; k < n; ++k) d[k] = a[k + (size_t)k * ld].real();
  for (int k = 0; k + 1 < n; ++k) {
    const cplx b = a[k + (size_t)(k + 1) * ld];  // A(k, k+1)
    const double m = std::abs(b);
    e[k] = m;
    // T(k, k+1) = conj(ph_k) b ph_{k+1} = |b|
    ph[k + 1] = m > 0.0 ? ph[k] * std::conj(b) / m : ph[k];
  }
  std::vector<int> comp(last ? std::vector<int>{0, n - 1} : std::vector<int>(n));
  if (!last)
    for (int i = 0; i < n; ++i) comp[i] = i;
  const int nc = (int)comp.size();
  std::vector<double> z;
  if (!tridiagonal_eigen(n, d, e, comp.data(), nc, z)) return false;
  std::vector<cplx> f(n);
  for (int k = 0; k < n; ++k) {
    const cplx x = pp * d[k];
    f[k] = phi ? (std::exp(x) - 1.0) / x : std::exp(x);
  }
  for (int c = last ? 1 : 0; c < nc; ++c) {
    cplx s = 0.0;
    for (int k = 0; k < n; ++k) s += z[(size_t)k * nc + c] * f[k] * z[(size_t)k * nc];  // component 0 of eigenvector k
    col[comp[c]] = ph[comp[c]] * s;  // (D U f U^T D^H e_1)_i with ph[0] = 1
  }
  return true;
}

int check_exp_args(octhip_hamiltonian_t h, const double* psi, int ldf, int order) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h && psi, "null argument");
  OCTHIP_REQUIRE(ldf >= 1 && ldf <= MAX_LDF, "exponentials need a complex batch (ldf in 1..%d)", MAX_LDF);
  OCTHIP_REQUIRE(order >= 1 && order <= 256, "order %d outside 1..256", order);
  return OCTHIP_SUCCESS;
}

}  // namespace

namespace octhip {
int krylov_vectors(octhip_hamiltonian_s* h, hipStream_t s, int nvec, int ldf, double** base) {
  KrylovBufs kb;
  int rc = krylov_bufs(h, s, nvec, ldf, &kb);
  if (rc) return rc;
  *base = kb.vec;
  return OCTHIP_SUCCESS;
}

void drop_krylov(octhip_hamiltonian_s* h, hipStream_t s, bool all) {
  for (size_t i = 0; i < h->krylov.size();) {
    if (all || h->krylov[i].s == s) {
      dfree(h->krylov[i].vec);
      dfree(h->krylov[i].small);
      hfree(h->krylov[i].host);
      if (h->krylov[i].ready) (void)hipEventDestroy(h->krylov[i].ready);
      h->krylov.erase(h->krylov.begin() + (long)i);
    } else {
      ++i;
    }
  }
}
}  // namespace octhip

extern "C" int octhip_exponential_lanczos_batch(octhip_hamiltonian_t h, double* psi, int ldf, int nst, double deltat,
                                                int imag_time, int order, double lanczos_tol, const double* inh,
                                                double vol, int* iterations, double* residual, void* stream) {
  OCTHIP_RANGE("octhip_exponential_lanczos_batch");
  int rc = check_exp_args(h, psi, ldf, order);
  if (rc) return rc;
  const int L = 1 << ldf, ncol = L / 2;
  OCTHIP_REQUIRE(nst >= 1 && nst <= ncol, "nst=%d outside 1..%d", nst, ncol);
  OCTHIP_REQUIRE(lanczos_tol > 0.0 && vol > 0.0, "lanczos_tol and vol must be positive");
  hipStream_t s = (hipStream_t)stream;
  const int np = h->np, np_part = h->kin->np_part;
  const size_t rowsz = (size_t)np_part * L;
  KrylovBufs kb;
  rc = krylov_bufs(h, s, order + 1, ldf, &kb);
  if (rc) return rc;
  auto V = [&](int k) { return kb.vec + (size_t)k * rowsz; };  // vb(k + 1)
  const cplx dt = imag_time ? cplx(0.0, deltat) : cplx(deltat, 0.0);
  const cplx pp = cplx(-0.0, -1.0) * dt;  // -i deltat
  const double eps = 2.220446049250313e-16;
  const double tiny = 1e4 * eps;
  const size_t cb = sizeof(double) * ncol;
  double* const norm = kb.res + 4 * (size_t)ncol;     // behind the overlaps with two vectors
  auto kept = [&](int k) { return kb.kept + (size_t)(k & 1) * ncol; };
  auto fetch = [&]() -> int {  // a step's overlaps and norms to the host, an event behind them
    OCTHIP_HIP(hipMemcpyAsync(kb.host, kb.res, 5 * cb, hipMemcpyDeviceToHost, s));
    OCTHIP_HIP(hipEventRecord(kb.ready, s));
    return OCTHIP_SUCCESS;
  };
  // The Krylov vectors are kept unnormalised, W_k = n_k vb(k + 1): the factors 1/n_k go into
  // the next step's overlaps and update, so no pass only scales a vector.  A step is the
  // H-apply, one pass for the overlaps with the two latest vectors, one pass that subtracts
  // them and sums the norm, and one copy of the results to the host; the next H-apply is
  // queued before the host waits for them, so that it runs while the projected problems are
  // solved.  (137,065 points, 16 states, 12 steps: 8.4 -> 1.7 ms against a pass per dot product,
  // subtraction and scaling, each with a copy and a wait.)  The host solves only what a step
  // needs, so that it is done before the H-apply is: the residuals' component from the fourth step
  // on, all components once at the end.
  // vb(1) = inh or psi (inner rows), beta = |vb(1)|
  rc = launch_gs_update(V(0), inh ? inh : psi, nullptr, 0, L, np, nullptr, nullptr, kb.part, s);
  if (!rc) rc = launch_gs_norms(kb.part, L, np, nst, vol, 0.0, norm, kept(0), nullptr, s);
  if (!rc) rc = fetch();
  if (rc) return rc;
  OCTHIP_HIP(hipEventSynchronize(kb.ready));
  std::vector<double> beta(nst);
  bool all_null = true;
  for (int i = 0; i < nst; ++i) {
    beta[i] = kb.host[4 * (size_t)ncol + i];
    if (std::fabs(beta[i]) > 1e-12) all_null = false;
  }
  if (iterations) *iterations = 0;
  if (residual) *residual = 0.0;
  if (all_null) return OCTHIP_SUCCESS;
  const int M = order + 1;  // hamilt(1:M, 1:M) per state, column-major
  std::vector<cplx> hamilt((size_t)nst * M * M, 0.0), expo((size_t)nst * M, 0.0);
  auto H = [&](int st, int i, int j) -> cplx& { return hamilt[(size_t)st * M * M + i + (size_t)j * M]; };
  std::vector<double> res(nst, 0.0), nk((size_t)M * nst, 1.0);  // nk: the norm of every vector kept
  for (int st = 0; st < nst; ++st) nk[st] = beta[st];
  int iter = 1;
  rc = propagator_apply(h, V(0), V(1), ldf, s);
  if (rc) return rc;
  for (; iter <= order; ++iter) {
    // classical Gram-Schmidt against vb(l..iter), l = max(1, iter - 1) (Hermitian H):
    // every overlap first, then the subtractions (mesh_batch_inc.F90:1218-1231)
    const int l = std::max(1, iter - 1), nv = iter - l + 1;
    const double* x[2] = {V(l - 1), V(iter - 1)};
    // the kept norms of the vectors in the order of x: those of an even and an odd vector lie
    // side by side, so an odd-even pair takes the vectors the other way round
    const bool swap = nv == 2 && ((l - 1) & 1);
    if (swap) std::swap(x[0], x[1]);
    rc = launch_gs_dots(x, nv, V(iter), L, np, nst, vol, nv == 2 ? kb.kept : kept(iter - 1), kept(iter - 1), kb.part,
                        kb.res, kb.coef, kb.scale, s);
    if (!rc) rc = launch_gs_update(V(iter), nullptr, x, nv, L, np, kb.scale, kb.coef, kb.part, s);
    if (!rc) rc = launch_gs_norms(kb.part, L, np, nst, vol, tiny, norm, kept(iter), nullptr, s);
    if (!rc) rc = fetch();
    if (!rc && iter < order) rc = propagator_apply(h, V(iter), V(iter + 1), ldf, s);
    if (rc) return rc;
    OCTHIP_HIP(hipEventSynchronize(kb.ready));
    bool happy = true;
    for (int st = 0; st < nst; ++st) {
      for (int j = l; j <= iter; ++j) {
        const int v = swap ? 1 - (j - l) : j - l;
        H(st, j - 1, iter - 1) = cplx(kb.host[2 * ((size_t)v * ncol + st)], kb.host[2 * ((size_t)v * ncol + st) + 1]);
      }
      const double nrm = kb.host[4 * (size_t)ncol + st];
      H(st, iter, iter - 1) = nrm;
      nk[(size_t)iter * nst + st] = nrm >= tiny ? nrm : 1.0;
      if (std::abs(H(st, iter, iter - 1)) >= tiny) happy = false;
    }
    // the residuals decide from the fourth step on; the step that ends the loop reports them
    for (int st = 0; st < nst && (happy || iter > 3 || iter == order); ++st) {
      if (!krylov_function(iter, &H(st, 0, 0), M, pp, inh != nullptr, true, &expo[(size_t)st * M]))
        return fail(OCTHIP_ERR_HIP, "Lanczos: the projected eigenproblem did not converge");
      res[st] = std::abs(H(st, iter, iter - 1) * std::abs(expo[(size_t)st * M + iter - 1]));
    }
    if (happy) break;  // happy breakdown
    if (iter > 3 && *std::max_element(res.begin(), res.end()) < lanczos_tol) break;
  }
  const int used = std::min(iter, order);  // a completed loop adds vb(order+1) with factor 0
  for (int st = 0; st < nst; ++st)
    if (!krylov_function(used, &H(st, 0, 0), M, pp, inh != nullptr, false, &expo[(size_t)st * M]))
      return fail(OCTHIP_ERR_HIP, "Lanczos: the projected eigenproblem did not converge");
  if (iterations) *iterations = used;
  if (residual) *residual = *std::max_element(res.begin(), res.end());
  // inh: psi += deltat nrm V expo(:, 1)  (exponential.F90:883-887); else psi = expo(1,1) psi +
  // sum_{ii >= 2} beta expo(ii,1) vb(ii)  (888-896); GS_MAX vectors per pass
  std::vector<std::vector<double>> staged;
  for (int ii = inh ? 1 : 2; !rc && (ii <= used || (!inh && ii == 2)); ii += GS_MAX) {
    const int nv = std::max(0, std::min(GS_MAX, used - ii + 1));
    std::vector<cplx> c((size_t)nv * nst), first(nst);
    const double* x[GS_MAX] = {};
    for (int v = 0; v < nv; ++v) {
      x[v] = V(ii + v - 1);
      for (int st = 0; st < nst; ++st) {
        const double rb = (inh ? dt.real() * beta[st] : beta[st]) / nk[(size_t)(ii + v - 1) * nst + st];
        const cplx ex = expo[(size_t)st * M + ii + v - 1];
        c[(size_t)v * nst + st] = cplx(rb * ex.real(), rb * ex.imag());
      }
    }
    const bool scaled = !inh && ii == 2;
    for (int st = 0; st < nst; ++st) first[st] = expo[(size_t)st * M];
    staged.emplace_back();
    rc = upload_factors(c, nv, nst, ncol, scaled ? &first : nullptr, kb.coef, kb.scale, staged.back(), s);
    if (!rc && hipEventRecord(kb.ready, s) != hipSuccess) rc = fail(OCTHIP_ERR_HIP, "Lanczos: event record failed");
    if (!rc) rc = launch_gs_update(psi, nullptr, x, nv, L, np, scaled ? kb.scale : nullptr, kb.coef, nullptr, s);
  }
  // the staged factors go out of scope: behind the last upload, or all of the stream's work
  const hipError_t done = rc ? hipStreamSynchronize(s) : hipEventSynchronize(kb.ready);
  if (!rc && done != hipSuccess) rc = fail(OCTHIP_ERR_HIP, "Lanczos: %s", hipGetErrorString(done));
  return rc;
}

extern "C" int octhip_exponential_cheby_batch(octhip_hamiltonian_t h, double* psi, int ldf, double deltat, int order,
                                              double spectral_middle_point, double spectral_half_span,
                                              void* stream) {
  OCTHIP_RANGE("octhip_exponential_cheby_batch");
  int rc = check_exp_args(h, psi, ldf, order);
  if (rc) return rc;
  OCTHIP_REQUIRE(spectral_half_span > 0.0, "spectral_half_span must be positive");
  hipStream_t s = (hipStream_t)stream;
  const int L = 1 << ldf;
  const int np = h->np, np_part = h->kin->np_part;
  const size_t rowsz = (size_t)np_part * L, count = (size_t)np * L;
  KrylovBufs kb;
  rc = krylov_bufs(h, s, 3, ldf, &kb);
  if (rc) return rc;
  // psi0 = psi1 = 0 (batch_set_zero); the copies of the recurrence become buffer rotations
  double* b0 = kb.vec;
  double* b1 = kb.vec + rowsz;
  double* b2 = kb.vec + 2 * rowsz;
  {
    const unsigned grid = (unsigned)std::min<size_t>((3 * rowsz + BLOCK - 1) / BLOCK, 8192);
    hipLaunchKernelGGL(k_zero_rows, dim3(grid), dim3(BLOCK), 0, s, kb.vec, (size_t)0, 3 * rowsz);
    OCTHIP_HIP(hipGetLastError());
  }
  const double x = spectral_half_span * deltat;
  for (int j = order - 1; j >= 0; --j) {
    // psi2 <- psi1, psi1 <- psi0, psi0 <- H psi1 (exponential.F90:936-940)
    double* t = b2;
    b2 = b1;
    b1 = b0;
    b0 = t;
    rc = propagator_apply(h, b1, b0, ldf, s);
    if (rc) return rc;
    static const cplx mi_pow[4] = {cplx(1.0, 0.0), cplx(0.0, -1.0), cplx(-1.0, 0.0), cplx(0.0, 1.0)};
    const cplx two_pow = cplx(2.0 * mi_pow[j & 3].real(), 2.0 * mi_pow[j & 3].imag());
    const double bj = jn(j, x);
    const cplx zfact(two_pow.real() * bj, two_pow.imag() * bj);
    rc = launch_cheby_update(b0, b1, psi, b2, count, spectral_middle_point, spectral_half_span, zfact, s);
    if (rc) return rc;
  }
  // psib = (psi0 - psi2) * exp(-i mid deltat) / 2
  const double ang = spectral_middle_point * deltat;
  const cplx z(0.5 * std::cos(ang), 0.5 * -std::sin(ang));
  return launch_cheby_final(psi, b0, b2, count, z, s);
}

extern "C" int octhip_mesh_batch_nrm2(const double* a, int ldf, int np, int is_complex, double vol, double* nrm2,
                                      void* stream) {
  OCTHIP_REQUIRE(nrm2 != nullptr, "null argument");
  const int L = 1 << (ldf < 0 ? 0 : ldf);
  const int n = is_complex ? L / 2 : L;
  std::vector<double> d(2 * (size_t)n);
  int rc = octhip_mesh_batch_dotp_vector(a, a, ldf, np, is_complex, vol, d.data(), stream);
  if (rc) return rc;
  for (int c = 0; c < n; ++c) nrm2[c] = std::sqrt(is_complex ? d[2 * c] : d[c]);
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_mesh_batch_orthogonalization(int nvec, const double* const* psi, double* phi, int ldf, int nst,
                                                   int np, double vol, int normalize, double* overlap, double* norm,
                                                   void* stream) {
  OCTHIP_RANGE("octhip_mesh_batch_orthogonalization");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(nvec >= 0 && (nvec == 0 || psi) && phi, "bad argument");
  OCTHIP_REQUIRE(ldf >= 1 && ldf <= MAX_LDF, "complex batches only (ldf in 1..%d)", MAX_LDF);
  const int L = 1 << ldf, ncol = L / 2;
  OCTHIP_REQUIRE(nst >= 1 && nst <= ncol && np >= 0, "bad sizes nst=%d np=%d", nst, np);
  hipStream_t s = (hipStream_t)stream;
  // one block: overlaps (nvec), factors of a pass, scaling, norms, partial sums
  const size_t col2 = 2 * (size_t)ncol;
  Scratch buf;
  int rc = buf.get(sizeof(double) * (col2 * (nvec + GS_MAX + 2)) + gs_scratch_bytes(L));
  if (rc) return rc;
  double* const ov = static_cast<double*>(buf.ptr());
  double* const dnorm = ov + col2 * nvec;             // behind the overlaps: one copy to the host
  double* const coef = dnorm + col2;
  double* const scale = coef + col2 * GS_MAX;
  double* const part = scale + col2;
  // Classical Gram-Schmidt: every overlap <psi_k|phi> first, GS_MAX vectors per pass over phi,
  // then phi -= sum_k <psi_k|phi> psi_k, GS_MAX vectors per pass, the last pass summing the norm.
  // (155,331 points, 32 states, 4 vectors with the H-apply before: 1253 -> 343 us.)
  for (int k = 0; k < nvec && !rc; k += GS_MAX) {
    const int nv = std::min(GS_MAX, nvec - k);
    rc = launch_gs_dots(psi + k, nv, phi, L, np, nst, vol, nullptr, nullptr, part, ov + col2 * k, coef, nullptr, s);
  }
  const bool with_norm = norm || normalize;
  for (int k = 0; k < std::max(nvec, 1) && !rc; k += GS_MAX) {
    const int nv = std::min(GS_MAX, nvec - k);
    const bool last = k + GS_MAX >= nvec;
    if (nv == 0 && !with_norm) break;
    // the factors of the last pass are still in coef; earlier ones are formed from the overlaps
    if (nvec > GS_MAX) rc = launch_gs_factors(ov + col2 * k, nv, ncol, nst, coef, s);
    if (!rc) rc = launch_gs_update(phi, nullptr, psi + k, nv, L, np, nullptr, coef, last && with_norm ? part : nullptr, s);
  }
  if (!rc && with_norm) rc = launch_gs_norms(part, L, np, nst, vol, 0.0, dnorm, nullptr, scale, s);
  if (!rc && normalize) rc = launch_gs_update(phi, nullptr, nullptr, 0, L, np, scale, nullptr, nullptr, s);
  std::vector<double> host(col2 * (nvec + 1));
  if (!rc && (overlap || norm)) {
    const hipError_t e = hipMemcpyAsync(host.data(), ov, sizeof(double) * host.size(), hipMemcpyDeviceToHost, s);
    if (e != hipSuccess) rc = fail(OCTHIP_ERR_HIP, "orthogonalization: %s", hipGetErrorString(e));
  }
  const hipError_t e = hipStreamSynchronize(s);  // results on the host, scratch out of use
  if (rc) return rc;
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "orthogonalization: %s", hipGetErrorString(e));
  if (overlap)  // overlap(k, st) = <psi_k|phi_st>, column-major (nvec x nst)
    for (int k = 0; k < nvec; ++k)
      for (int st = 0; st < nst; ++st) {
        overlap[2 * ((size_t)k + (size_t)st * nvec)] = host[col2 * k + 2 * st];
        overlap[2 * ((size_t)k + (size_t)st * nvec) + 1] = host[col2 * k + 2 * st + 1];
      }
  if (norm)
    for (int st = 0; st < nst; ++st) norm[st] = host[col2 * nvec + st];
  return OCTHIP_SUCCESS;
}
