// Hamiltonian handle: local potential, KB projectors, fused apply, Taylor propagator.
#include <algorithm>
#include <complex>
#include <functional>
#include <cstring>

#include "kernels.h"

using namespace octhip;

namespace octhip {
void stencil_args(const octhip_nl_operator_s* op, double factor, ApplyArgs& a);
int launch_bra_mfma(BraMfmaArgs& m, size_t lds, hipStream_t s);
int launch_operator(octhip_nl_operator_s* op, ApplyArgs& a, int epi, hipStream_t s,
                    const BraMfmaArgs* bra = nullptr);
bool operator_takes_bra(const octhip_nl_operator_s* op, const ApplyArgs& a, size_t lds);
int prepare_operator(octhip_nl_operator_s* op, int L, bool nl);
}  // namespace octhip

namespace {

enum { O_POINTS = 0, O_PROJS, O_MATRIX, O_MAP, O_SCAL, O_MIX };

// a graph whose Hamiltonian is destroyed no longer owns work sets (they are freed with it)
void detach_graph(octhip_taylor_graph_t g);

// the work-buffer set of stream s, created empty on first use, and mirrored into h
octhip_hamiltonian_s::WorkSet& workset(octhip_hamiltonian_s* h, hipStream_t s) {
  for (auto& w : h->sets)
    if (w.s == s) return w;
  h->sets.push_back({s, -1, -1, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr, -1});
  return h->sets.back();
}

void bind(octhip_hamiltonian_s* h, const octhip_hamiltonian_s::WorkSet& w) {
  h->d_partial = w.partial;
  h->d_proj = w.proj;
  h->d_ksum = w.ksum;
  h->d_y[0] = w.y0;
  h->d_y[1] = w.y1;
  h->d_y[2] = w.y2;
  h->work_ldf = w.work_ldf;
  h->y_ldf = w.y_ldf;
}

// projector work buffers of stream s for rows of 2^ldf lanes (outgrown ones are retired)
int ensure_work(octhip_hamiltonian_s* h, int ldf, hipStream_t s) {
  auto& w = workset(h, s);
  if (w.work_ldf < ldf) {
    for (void* p : {(void*)w.partial, (void*)w.proj, (void*)w.ksum})
      if (p) h->retired.push_back(p);
    w.partial = w.proj = w.ksum = nullptr;
    w.work_ldf = -1;  // until all three are there: after a failure shorter rows get new ones too
    const size_t L = (size_t)1 << ldf;
    int rc = OCTHIP_SUCCESS;
    if (h->nmat > 0) {
      rc = dalloc((void**)&w.partial, sizeof(double) * partial_doubles(h, L));
      if (!rc) rc = dalloc((void**)&w.proj, sizeof(double) * h->nprow * L);
      if (!rc) rc = dalloc((void**)&w.ksum, sizeof(double) * std::max(h->nslot, 1) * L);
    }
    if (rc) return rc;
    w.work_ldf = ldf;
  }
  bind(h, w);
  return OCTHIP_SUCCESS;
}

// Taylor intermediates of stream s (np rows each)
int ensure_taylor(octhip_hamiltonian_s* h, int ldf, hipStream_t s) {
  auto& w = workset(h, s);
  if (w.y_ldf < ldf) {
    for (void* p : {(void*)w.y0, (void*)w.y1, (void*)w.y2})
      if (p) h->retired.push_back(p);
    w.y0 = w.y1 = w.y2 = nullptr;
    w.y_ldf = -1;
    const size_t bytes = sizeof(double) * ((size_t)h->np << ldf);
    int rc = dalloc((void**)&w.y0, bytes);
    if (!rc) rc = dalloc((void**)&w.y1, bytes);
    if (!rc) rc = dalloc((void**)&w.y2, bytes);
    if (rc) return rc;
    w.y_ldf = ldf;
  }
  bind(h, w);
  return OCTHIP_SUCCESS;
}

// MFMA bra of batch f (L lanes), clearing the boundary rows of zero_bc (optional) on the way
void bra_args(const octhip_hamiltonian_s* h, const double* f, int L, double* zero_bc, BraMfmaArgs& m) {
  const int np = h->kin->np, np_part = h->kin->np_part;
  bra_mfma_args(h, L, h->d_partial, m);
  m.b.psi = f;
  m.zf = zero_bc;
  m.zfirst = (size_t)np * L;
  m.zcount = zero_bc ? (size_t)(np_part - np) * L : 0;
}

// projections from the parts of the bra, and their ket rows into h->d_ksum, or added to out
int run_ket(octhip_hamiltonian_s* h, int L, int pjmax, bool sets, hipStream_t s, double* out = nullptr,
            const double* out_phase = nullptr) {
  BraReduceArgs r;
  r.partial = h->d_partial;
  r.row = h->d_prow;
  r.scals = h->d_scals;
  r.proj = h->d_proj;
  r.L = L;
  r.pjmax = pjmax;
  r.nrow = h->nprow;
  r.sets = sets;
  int rc = launch_bra_reduce(r, s);
  if (rc) return rc;
  KetArgs k;
  ket_args(h, L, h->d_proj, h->d_ksum, k);
  k.out = out;
  k.point = h->d_kpoint;
  k.out_phase = out_phase;
  return launch_ket(k, h->use_mfma, s);
}

// projections of batch f (L lanes) and their ket rows into h->d_ksum; zero_bc (optional) = a batch whose
// boundary rows are cleared on the way (fused into the bra launch when it can be)
int run_bra(octhip_hamiltonian_s* h, const double* f, int L, hipStream_t s, double* zero_bc = nullptr) {
  const int np = h->kin->np, np_part = h->kin->np_part;
  if (h->nchunk == 0) return zero_bc ? zero_boundary(zero_bc, np, np_part, L, s) : OCTHIP_SUCCESS;
  const bool mfma = h->use_mfma && bra_takes_rows(h, L);
  if (zero_bc && !mfma) {
    int rc = zero_boundary(zero_bc, np, np_part, L, s);
    if (rc) return rc;
    zero_bc = nullptr;
  }
  BraMfmaArgs m;
  bra_args(h, f, L, zero_bc, m);
  int rc;
  if (mfma) {
    rc = launch_bra_mfma(m, bra_mfma_lds(h, L), s);
  } else {
    m.b.pjmax = h->max_nprojs;
    rc = launch_bra(m.b, h->nchunk, s);
  }
  if (rc) return rc;
  return run_ket(h, L, m.b.pjmax, mfma && m.sets, s);
}

// H fi into fo with the terms of `a` (a.kslot: the nonlocal one too); zero_bc as in run_bra.
// Where the z-march can take the bra along, the two run in one launch and the ket adds its rows
// to fo afterwards: the bra fills the CUs that the march leaves idle (small systems, the end of
// a launch), and the march reads no ket rows.  The sums keep their order: results are
// bit-identical.  With the bra and the ket in front of the march, and with it: 57,777 points,
// 8 complex states 24.8 -> 20.2 us; 13 real ones on 79,501 points 23.5 -> 19.7; 462,781 points,
// 2 x 32 states 410 -> 380; exponential midpoint, 155,331 points, 48 states 755 -> 689; 8 lanes
// (a bra block per workgroup) 9,843 points 18.0 -> 14.4, 462,781 points 34 -> 30.  Sums of the
// parts by the block that stores the last one instead of a launch of 5 us: 20 -> 44 and 380 ->
// 644 us, every block's release to the other XCDs writes back its L2.  With Bloch phases the march
// leaves the rows of the ket without the conjugate phase, which the ket multiplies after its sum:
// 40^3 cell, 16 states 35.9 -> 32.1 us; 32^3 cell, 4 states 24 -> 21.
int apply_store(octhip_hamiltonian_s* h, ApplyArgs& a, hipStream_t s, double* zero_bc = nullptr) {
  const int L = a.L;
  if (a.kslot && h->use_mfma && bra_by_sets(h) &&
      operator_takes_bra(h->kin, a, bra_mfma_lds(h, L))) {
    BraMfmaArgs m;
    bra_args(h, a.fi, L, zero_bc, m);
    if (!a.out_phase) a.kslot = nullptr;  // else: the rows that the ket multiplies by the phase
    a.ksum = nullptr;
    a.nk = 0;
    int rc = launch_operator(h->kin, a, EPI_STORE, s, &m);
    if (rc) return rc;
    return run_ket(h, L, m.b.pjmax, true, s, a.fo, a.out_phase);
  }
  int rc = OCTHIP_SUCCESS;
  if (a.kslot) rc = run_bra(h, a.fi, L, s, zero_bc);
  else if (zero_bc) rc = zero_boundary(zero_bc, h->kin->np, h->kin->np_part, L, s);
  if (rc) return rc;
  return launch_operator(h->kin, a, EPI_STORE, s);
}

// v_eff(p) = v(p) + (f0 x + f1 y + f2 z): the dipole term of laser_potential
// (src/hamiltonian/lasers.F90:823-853) folded into the local potential once per field.
__global__ void k_veff(double* __restrict__ veff, const double* __restrict__ v,
                       const double* __restrict__ xyz, double f0, double f1, double f2, int np) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x)
    veff[p] = v[p] + (f0 * xyz[3 * (size_t)p] + f1 * xyz[3 * (size_t)p + 1] + f2 * xyz[3 * (size_t)p + 2]);
}

}  // namespace

namespace octhip {
namespace {
int padded(int nprojs) { return (nprojs + 3) / 4 * 4; }
}  // namespace

bool bra_by_sets(const octhip_hamiltonian_s* h) { return h->nsblk > 0; }

bool bra_takes_rows(const octhip_hamiltonian_s* h, int L) { return L >= 16 || bra_by_sets(h); }

size_t partial_doubles(const octhip_hamiltonian_s* h, size_t L) {
  return std::max((size_t)h->nchunk * h->max_nprojs, (size_t)h->set_parts * padded(h->max_nprojs)) * L;
}

int bra_mfma_blocks(const octhip_hamiltonian_s* h, int L) {
  return (bra_by_sets(h) ? h->nsblk : h->nchunk) * mfma_lane_tiles(L);
}

size_t bra_mfma_lds(const octhip_hamiltonian_s* h, int L) {
  const size_t lanes = std::max(L / mfma_lane_tiles(L), 16);
  return sizeof(double) * 4 * lanes * (bra_by_sets(h) ? h->set_sums : 16);
}

void bra_mfma_args(const octhip_hamiltonian_s* h, int L, double* partial, BraMfmaArgs& m) {
  m = BraMfmaArgs();
  m.sets = bra_by_sets(h);
  m.b.L = L;
  m.b.chunks = h->d_chunks;
  m.b.mat_info = h->d_mat_info;
  m.b.mats = h->d_matrices;
  m.b.maps = h->d_maps;
  m.b.partial = partial;
  m.b.pjmax = m.sets ? padded(h->max_nprojs) : h->max_nprojs;
  m.b.pphase = h->has_kpoint ? h->d_pphase : nullptr;
  m.set.grp = h->d_kgrp;
  m.set.step = h->d_kstep;
  m.set.pt = h->d_kpt;
  m.set.point = h->d_kpoint;
  m.set.blk = h->d_sblk;
  m.set.part = h->d_spart;
  m.set.phase = h->has_kpoint ? h->d_kphase : nullptr;
  m.pt = h->d_pt;
  m.pjs = h->pjs;
  m.nbra = bra_takes_rows(h, L) ? bra_mfma_blocks(h, L) : 0;
}

void ket_args(const octhip_hamiltonian_s* h, int L, const double* proj, double* kbuf, KetArgs& k) {
  k = KetArgs();
  k.grp = h->d_kgrp;
  k.ngrp = h->nkgrp;
  k.step = h->d_kstep;
  k.pt = h->d_kpt;
  k.proj = proj;
  k.kbuf = kbuf;
  k.L = L;
  k.phase = h->has_kpoint ? h->d_kphase : nullptr;
}

int zero_boundary(double* f, int np, int np_part, int L, hipStream_t s) {
  const size_t count = (size_t)(np_part - np) * L;
  if (count == 0) return OCTHIP_SUCCESS;
  size_t grid = (count + BLOCK - 1) / BLOCK;
  if (grid > 8192) grid = 8192;
  ProfScope prof("k_zero_rows", s);
  hipLaunchKernelGGL(k_zero_rows, dim3((unsigned)grid), dim3(BLOCK), 0, s, f, (size_t)np * L, count);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "k_zero_rows: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}

// out = v + field . x over the np points (a caller's buffer, e.g. one per stream)
int launch_veff(const octhip_hamiltonian_s* h, double* out, const double field[3], hipStream_t s) {
  if (!h->d_v || !h->d_xyz) return fail(OCTHIP_ERR_STATE, "launch_veff: no local potential or positions");
  const int grid = std::min((h->np + BLOCK - 1) / BLOCK, 4096);
  hipLaunchKernelGGL(k_veff, dim3(grid), dim3(BLOCK), 0, s, out, h->d_v, h->d_xyz, field[0], field[1], field[2],
                     h->np);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "k_veff: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}
}  // namespace octhip

namespace {

int update_veff(octhip_hamiltonian_s* h, hipStream_t s) {
  if (!h->has_field || !h->d_v || !h->d_xyz) return OCTHIP_SUCCESS;
  if (!h->d_veff) {
    int rc = dalloc((void**)&h->d_veff, sizeof(double) * h->np);
    if (rc) return rc;
  }
  const int grid = std::min((h->np + BLOCK - 1) / BLOCK, 4096);
  hipLaunchKernelGGL(k_veff, dim3(grid), dim3(BLOCK), 0, s, h->d_veff, h->d_v, h->d_xyz, h->field[0],
                     h->field[1], h->field[2], h->np);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "k_veff: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}

void fill_terms(const octhip_hamiltonian_s* h, int terms, ApplyArgs& a) {
  if (terms & OCTHIP_TERM_KINETIC) {
    stencil_args(h->kin, -0.5 / h->mass, a);  // factor -1/(2m), hamiltonian_elec_inc.F90:155
  } else {
    stencil_args(h->kin, 0.0, a);
    a.n = 0;  // no stencil term: runtime-size path with zero points
  }
  if ((terms & OCTHIP_TERM_LOCAL_POTENTIAL) && h->d_v) {
    a.v = (h->has_field && h->d_veff) ? h->d_veff : h->d_v;
  }
  if ((terms & OCTHIP_TERM_NON_LOCAL_POTENTIAL) && h->nmat > 0 && h->nslot > 0) {
    a.kslot = h->d_kslot;
    a.ksum = h->d_ksum;
    a.nk = h->nslot;
  }
}

}  // namespace

namespace {
// the phased copy of a k-point apply's input (np_part rows) of stream s
int ensure_ephase(octhip_hamiltonian_s* h, int ldf, hipStream_t s, double** out) {
  auto& w = workset(h, s);
  if (w.ephase_ldf < ldf) {
    if (w.ephase) h->retired.push_back(w.ephase);
    w.ephase = nullptr;
    w.ephase_ldf = -1;
    int rc = dalloc((void**)&w.ephase, sizeof(double) * ((size_t)h->kin->np_part << ldf));
    if (rc) return rc;
    w.ephase_ldf = ldf;
  }
  *out = w.ephase;
  return OCTHIP_SUCCESS;
}

// X(hamiltonian_elec_apply_batch) for a periodic handle or one with Bloch phases
// (src/hamiltonian/hamiltonian_elec_inc.F90:116-154, 243-247): boundaries_set fills the
// boundary rows from their periodic images (times phase_corr when psi carries the phase);
// a psi without the phase is copied with it (epsib, np_part rows) and H psi is multiplied
// by the conjugate phase at the end; the projectors use their Bloch phases; the stencil
// reads the boundary rows as they are.
int periodic_apply(octhip_hamiltonian_s* h, double* psi, double* hpsi, int ldf, int is_complex, int terms,
                   int set_bc, bool has_phase, hipStream_t s) {
  const int L = 1 << ldf;
  const int np = h->np, np_part = h->kin->np_part;
  if (h->has_kpoint && !is_complex) return fail(OCTHIP_ERR_INVALID, "Bloch phases need a complex batch");
  int rc = ensure_work(h, ldf, s);
  if (rc) return rc;
  const double* src = psi;
  const bool set_phase = h->has_kpoint && !has_phase;
  double* e = nullptr;
  if (set_phase) {
    rc = ensure_ephase(h, ldf, s, &e);
    if (rc) return rc;
    src = e;
  }
  if (set_bc && h->periodic && set_phase) {
    rc = launch_periodic_phase(e, psi, h->d_phase, h->d_bnd_src, np, np_part, L, s);
    if (rc) return rc;
  } else {
    if (set_bc) {
      rc = h->periodic ? launch_periodic_bc(psi, h->d_bnd_src, np, h->nbnd, L,
                                            (has_phase && h->has_kpoint) ? h->d_phase_corr : nullptr, s)
                       : zero_boundary(psi, np, np_part, L, s);
      if (rc) return rc;
    }
    if (set_phase) {
      rc = launch_phase(e, psi, h->d_phase, np_part, L, false, s);
      if (rc) return rc;
    }
  }
  ApplyArgs a;
  std::memset(&a, 0, sizeof(a));
  fill_terms(h, terms, a);
  a.fi = src;
  a.fo = hpsi;
  a.L = L;
  a.lim = np_part;  // boundary rows as set above (or by the caller)
  a.out_phase = set_phase ? h->d_phase : nullptr;
  return apply_store(h, a, s);
}

// Ket tables of a handle (KetArgs, BraReduceArgs::row).
struct KetTables {
  std::vector<int> slot, g;
  std::vector<KetGroup> grp;
  std::vector<int4> step, sblk;
  std::vector<ProjRow> prow;
  std::vector<int> point, spart;
  std::vector<double> pt;
  std::vector<int> matrix;  // matrix of each step
};

int padded_projs(const octhip_hamiltonian_s* h, int a) { return (h->offsets[6 * (size_t)a + O_PROJS] + 3) / 4 * 4; }

// blocks of the bra by sets: <= BRA_SET_GROUPS groups and `most` rows of sums
void set_blocks(octhip_hamiltonian_s* h, int most, KetTables& t) {
  const int pj = (h->max_nprojs + 3) / 4 * 4;
  std::vector<int> slot(h->nmat, -1), count(h->nmat, 0), matrix;
  int first_matrix = 0;
  for (size_t i = 0; i < t.grp.size(); ++i) {
    const int s0 = t.grp[i].step, s1 = s0 + t.grp[i].steps;
    int add = 0;
    for (int q = s0; q < s1; ++q) add += t.step[q].w && slot[t.matrix[q]] < 0;
    if (t.sblk.empty() || t.sblk.back().y == BRA_SET_GROUPS || (t.sblk.back().w + add) * pj > most) {
      for (size_t k = first_matrix; k < matrix.size(); ++k) slot[matrix[k]] = -1;
      first_matrix = (int)matrix.size();
      t.sblk.push_back(make_int4((int)i, 0, first_matrix, 0));
    }
    int4& b = t.sblk.back();
    ++b.y;
    int j = 0;
    for (int q = s0; q < s1; ++q) {
      const int a = t.matrix[q];
      if (slot[a] < 0) {
        slot[a] = b.w++;
        matrix.push_back(a);
        ++count[a];
      }
      j = t.step[q].w ? 0 : j + 4;
      t.step[q].y = slot[a] * pj + j;
    }
    h->set_sums = std::max(h->set_sums, b.w * pj);
  }
  // the parts of one matrix are consecutive, in block order
  std::vector<int> first(h->nmat + 1, 0);
  for (int a = 0; a < h->nmat; ++a) first[a + 1] = first[a] + count[a];
  h->set_parts = first[h->nmat];
  size_t row = 0;
  for (int a = 0; a < h->nmat; ++a)
    for (int j = 0; j < padded_projs(h, a); ++j) t.prow[row++].part[1] = make_int2(first[a], first[a + 1]);
  for (int a : matrix) t.spart.push_back(first[a]++);
  h->nsblk = (int)t.sblk.size();
}

// pos, ent: CSR over the mesh points of their sphere points {map index, matrix}, matrix order
void build_ket(octhip_hamiltonian_s* h, const double* matrices, const std::vector<int>& pos,
               const std::vector<int2>& ent, const std::vector<int>& chunk0, KetTables& t) {
  std::vector<int> prow0(h->nmat);
  for (int a = 0; a < h->nmat; ++a) {
    const int* o = h->offsets.data() + 6 * (size_t)a;
    prow0[a] = (int)t.prow.size();
    for (int j = 0; j < padded_projs(h, a); ++j)
      t.prow.push_back(ProjRow{{make_int2(chunk0[a], chunk0[a + 1]), make_int2(0, 0)}, j,
                               j < o[O_PROJS] ? o[O_SCAL] + j : -1});
  }
  h->nprow = (int)t.prow.size();
  // mesh points inside a sphere, by their set of matrices, mesh order within a set
  std::vector<int> pts;
  for (int p = 0; p < h->np; ++p)
    if (pos[p + 1] > pos[p]) pts.push_back(p);
  auto cmp = [&](int p, int q) {  // -1, 0, 1: order of the two points' sets
    for (int i = pos[p], j = pos[q];; ++i, ++j) {
      if (i == pos[p + 1] || j == pos[q + 1]) return (i < pos[p + 1]) - (j < pos[q + 1]);
      if (ent[i].y != ent[j].y) return ent[i].y < ent[j].y ? -1 : 1;
    }
  };
  std::stable_sort(pts.begin(), pts.end(), [&](int p, int q) { return cmp(p, q) < 0; });
  h->nslot = (int)pts.size();
  t.slot.assign(h->np, 0);
  int widest = 0;  // most slots of a set
  for (size_t i = 0, e; i < pts.size(); i = e) {
    for (e = i + 1; e < pts.size() && e < i + 16 && cmp(pts[i], pts[e]) == 0;) ++e;
    const int p0 = pos[pts[i]], ne = pos[pts[i] + 1] - p0, n = (int)(e - i);
    const int step0 = (int)t.step.size(), line0 = (int)(t.pt.size() / 4);
    widest = std::max(widest, ne);
    for (int k = 0; k < ne; ++k) {
      const int a = ent[p0 + k].y;
      const int* o = h->offsets.data() + 6 * (size_t)a;
      const int entry = (int)t.g.size();
      for (size_t r = i; r < e; ++r) t.g.push_back(ent[pos[pts[r]] + k].x);
      for (int j = 0; j < o[O_PROJS]; j += 4) {
        t.step.push_back(make_int4(prow0[a] + j, 0, entry, j == 0));
        t.matrix.push_back(a);
        for (int r = 0; r < n; ++r)
          for (int c = j; c < j + 4; ++c)
            t.pt.push_back(c < o[O_PROJS] ? matrices[o[O_MATRIX] + (size_t)c * o[O_POINTS] + (t.g[entry + r] - o[O_MAP])]
                                          : 0.0);
      }
    }
    KetGroup g = {};
    g.row = (int)i;
    g.rows = n;
    g.steps = (int)t.step.size() - step0;
    g.step = step0;
    g.line = line0;
    t.grp.push_back(g);
    for (size_t r = i; r < e; ++r) t.slot[pts[r]] = (int)r + 1;
  }
  h->nkgrp = (int)t.grp.size();
  t.point = pts;
  // Bra by sets where a set's sums fit a block, unless the rows it reads (groups padded to 16
  // points) with its parts written and read clearly exceed those of the bra by spheres (sets
  // of a few points each).  Without any overlap it reads a tenth more and is still faster
  // (R = 12 sphere x 64 lanes, 16 spheres of radius 1.5 / 4 of them: 14.5 / 13.5 us against
  // 18.0 / 16.1; R = 8 x 16 lanes, 6 spheres: 6.9 against 9.6): more, smaller waves.
  const int pj = (h->max_nprojs + 3) / 4 * 4;
  if (widest * pj <= BRA_SET_ROWS) {
    set_blocks(h, widest * pj <= BRA_SET_ROWS / 2 ? BRA_SET_ROWS / 2 : BRA_SET_ROWS, t);
    const size_t by_sets = 16 * (size_t)h->nkgrp + 2 * (size_t)h->set_parts * pj;
    const size_t by_spheres = ent.size() + 2 * (size_t)h->nchunk * h->max_nprojs;
    if (4 * by_sets >= 5 * by_spheres) h->nsblk = h->set_parts = h->set_sums = 0;
  }
  for (KetGroup& g : t.grp)
    for (int u = 0; u < KET_AHEAD; ++u) {
      const int4 q = t.step[g.step + std::min(u, g.steps - 1)];
      g.proj[u] = q.x;
      g.sum[u] = q.y;
    }
}

}  // namespace

extern "C" int octhip_hamiltonian_create(octhip_nl_operator_t kinetic, double mass, const double* vlocal,
                                         int nmat, const int* offsets, const double* matrices,
                                         const int* maps, const double* scals, octhip_hamiltonian_t* out) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(out != nullptr, "hamiltonian_create: null output handle");
  *out = nullptr;
  OCTHIP_REQUIRE(kinetic != nullptr, "hamiltonian_create: null kinetic operator");
  OCTHIP_REQUIRE(mass > 0.0, "mass must be positive");
  OCTHIP_REQUIRE(nmat >= 0, "nmat < 0");
  OCTHIP_REQUIRE(nmat == 0 || (offsets && matrices && maps && scals), "null projector arrays");
  const int np = kinetic->np;
  // sizes and validation of build_accel's offsets
  size_t matrix_size = 0, total_points = 0, nproj = 0;
  int max_nprojs = 0;
  for (int a = 0; a < nmat; ++a) {
    const int* o = offsets + 6 * (size_t)a;
    OCTHIP_REQUIRE(o[O_POINTS] >= 0 && o[O_PROJS] >= 1, "matrix %d: bad POINTS/PROJS", a);
    OCTHIP_REQUIRE(o[O_MIX] == -1, "matrix %d: mixing matrices (HGH/SOC) are not supported", a);
    OCTHIP_REQUIRE(o[O_MATRIX] >= 0 && o[O_MAP] >= 0 && o[O_SCAL] >= 0, "matrix %d: negative offset", a);
    matrix_size = std::max(matrix_size, (size_t)o[O_MATRIX] + (size_t)o[O_POINTS] * o[O_PROJS]);
    total_points = std::max(total_points, (size_t)o[O_MAP] + o[O_POINTS]);
    nproj = std::max(nproj, (size_t)o[O_SCAL] + o[O_PROJS]);
    max_nprojs = std::max(max_nprojs, o[O_PROJS]);
  }
  for (size_t i = 0; i < total_points; ++i)
    OCTHIP_REQUIRE(maps[i] >= 1 && maps[i] <= np, "map entry %zu = %d outside 1..np", i, maps[i]);
  auto* h = new octhip_hamiltonian_s();
  h->kin = kinetic;
  h->mass = mass;
  h->np = np;
  h->nmat = nmat;
  h->max_nprojs = max_nprojs;
  h->total_points = (int)total_points;
  h->pjs = max_nprojs;
  h->offsets.assign(offsets ? offsets : nullptr, offsets ? offsets + 6 * (size_t)nmat : nullptr);
  hipStream_t s = nullptr;
  int rc = OCTHIP_SUCCESS;
  if (vlocal) rc = upload(&h->d_v, vlocal, (size_t)np, s);
  if (!rc && nmat > 0) {
    std::vector<double> pt(total_points * (size_t)h->pjs, 0.0);
    std::vector<int> cnt(np + 1, 0), chunk0(nmat + 1);
    std::vector<int4> info(nmat), chunks;
    for (int a = 0; a < nmat; ++a) {
      const int* o = offsets + 6 * (size_t)a;
      const int npt = o[O_POINTS], nj = o[O_PROJS];
      info[a] = make_int4(npt, nj, o[O_MATRIX], o[O_MAP]);
      for (int q = 0; q < npt; ++q) {
        for (int j = 0; j < nj; ++j)
          pt[(size_t)(o[O_MAP] + q) * h->pjs + j] = matrices[o[O_MATRIX] + (size_t)j * npt + q];
        cnt[maps[o[O_MAP] + q]]++;  // 1-based -> counts at index p+1
      }
      chunk0[a] = (int)chunks.size();
      for (int q0 = 0; q0 < npt; q0 += BRA_CHUNK)
        chunks.push_back(make_int4(a, q0, std::min(q0 + BRA_CHUNK, npt), (int)chunks.size() - chunk0[a]));
    }
    chunk0[nmat] = (int)chunks.size();
    // CSR of (sphere point, matrix) per mesh point, matrix order preserved
    std::vector<int> pos(np + 1, 0);
    for (int p = 0; p < np; ++p) pos[p + 1] = pos[p] + cnt[p + 1];
    std::vector<int2> ent(pos[np]);
    std::vector<int> fillp(pos.begin(), pos.end() - 1);
    for (int a = 0; a < nmat; ++a) {
      const int* o = offsets + 6 * (size_t)a;
      for (int q = 0; q < o[O_POINTS]; ++q) {
        const int p = maps[o[O_MAP] + q] - 1;
        ent[fillp[p]++] = make_int2(o[O_MAP] + q, a);
      }
    }
    h->nchunk = (int)chunks.size();
    KetTables kt;
    build_ket(h, matrices, pos, ent, chunk0, kt);
    rc = upload(&h->d_kslot, kt.slot.data(), kt.slot.size(), s);
    if (!rc && !kt.grp.empty()) {
      rc = upload(&h->d_kgrp, kt.grp.data(), kt.grp.size(), s);
      if (!rc) rc = upload(&h->d_kstep, kt.step.data(), kt.step.size(), s);
      if (!rc) rc = upload(&h->d_kpt, kt.pt.data(), kt.pt.size(), s);
      h->kg = std::move(kt.g);
      if (!rc && h->nsblk > 0) {
        rc = upload(&h->d_sblk, kt.sblk.data(), kt.sblk.size(), s);
        if (!rc) rc = upload(&h->d_spart, kt.spart.data(), kt.spart.size(), s);
        if (!rc) rc = upload(&h->d_kpoint, kt.point.data(), kt.point.size(), s);
      }
    }
    if (!rc) rc = upload(&h->d_matrices, matrices, matrix_size, s);
    if (!rc) rc = upload(&h->d_maps, maps, total_points, s);
    if (!rc) rc = upload(&h->d_scals, scals, nproj, s);
    if (!rc) rc = upload(&h->d_pt, pt.data(), pt.size(), s);
    if (!rc) rc = upload(&h->d_chunks, chunks.data(), chunks.size(), s);
    if (!rc) rc = upload(&h->d_mat_info, info.data(), info.size(), s);
    if (!rc) rc = upload(&h->d_prow, kt.prow.data(), kt.prow.size(), s);
  }
  if (rc) {
    octhip_hamiltonian_destroy(h);
    return rc;
  }
  *out = h;
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_hamiltonian_destroy(octhip_hamiltonian_t h) {
  if (!h) return OCTHIP_SUCCESS;
  (void)hipDeviceSynchronize();
  dfree(h->d_mat_info);
  dfree(h->d_kslot);
  dfree(h->d_kgrp);
  dfree(h->d_kstep);
  dfree(h->d_prow);
  dfree(h->d_kphase);
  dfree(h->d_sblk);
  dfree(h->d_spart);
  dfree(h->d_kpoint);
  dfree(h->d_kpt);
  dfree(h->d_v);
  dfree(h->d_xyz);
  dfree(h->d_veff);
  dfree(h->d_matrices);
  dfree(h->d_maps);
  dfree(h->d_scals);
  dfree(h->d_pt);
  dfree(h->d_chunks);
  for (auto& w : h->sets)
    for (void* p : {(void*)w.partial, (void*)w.proj, (void*)w.ksum, (void*)w.y0, (void*)w.y1, (void*)w.y2,
                    (void*)w.dpart, (void*)w.dw, (void*)w.ephase})
      dfree(p);
  for (void* p : h->retired) dfree(p);
  dfree(h->d_bnd_src);
  dfree(h->d_phase);
  dfree(h->d_phase_corr);
  dfree(h->d_pphase);
  drop_krylov(h, nullptr, true);
  for (octhip_taylor_graph_t g : h->graphs) detach_graph(g);
  delete h;
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_hamiltonian_set_tuning(octhip_hamiltonian_t h, int key, int value) {
  OCTHIP_REQUIRE(h != nullptr, "null hamiltonian handle");
  if (key == OCTHIP_TUNE_BRA_MODE) {
    OCTHIP_REQUIRE(value == 0 || value == 1, "bra mode must be 0 or 1");
    h->use_mfma = value;
    return OCTHIP_SUCCESS;
  }
  return octhip_nl_operator_set_tuning(h->kin, key, value);  // stencil knobs go to the kinetic operator
}

extern "C" int octhip_hamiltonian_set_potential(octhip_hamiltonian_t h, const double* vlocal, void* stream) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h && vlocal, "null argument");
  hipStream_t s = (hipStream_t)stream;
  if (!h->d_v) {
    int rc = dalloc((void**)&h->d_v, sizeof(double) * h->np);
    if (rc) return rc;
  }
  ++h->changes;
  OCTHIP_HIP(hipMemcpyAsync(h->d_v, vlocal, sizeof(double) * h->np, hipMemcpyHostToDevice, s));
  OCTHIP_HIP(hipStreamSynchronize(s));
  return update_veff(h, s);
}

extern "C" int octhip_hamiltonian_set_dipole_field(octhip_hamiltonian_t h, const double* positions,
                                                   const double* field, void* stream) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h && field, "null argument");
  hipStream_t s = (hipStream_t)stream;
  if (positions) {
    // d_veff keeps its address (captured graphs read it); only the positions are replaced
    ++h->changes;
    dfree(h->d_xyz);
    h->d_xyz = nullptr;
    int rc = upload(&h->d_xyz, positions, 3 * (size_t)h->np, s);
    if (rc) return rc;
  }
  OCTHIP_REQUIRE(h->d_xyz != nullptr, "set_dipole_field: positions never uploaded");
  for (int d = 0; d < 3; ++d) h->field[d] = field[d];
  h->has_field = true;
  return update_veff(h, s);
}

extern "C" int octhip_hamiltonian_release_stream(octhip_hamiltonian_t h, void* stream) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h != nullptr, "null hamiltonian handle");
  const hipStream_t s = (hipStream_t)stream;
  OCTHIP_HIP(hipStreamSynchronize(s));
  drop_workset(h, s);
  drop_krylov(h, s, false);
  return OCTHIP_SUCCESS;
}

namespace {
size_t dev_bytes(const void* p) {
  if (!p) return 0;
  size_t n = 0;
  if (hipMemPtrGetInfo(const_cast<void*>(p), &n) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return n;
}
}  // namespace

extern "C" int octhip_hamiltonian_memory(octhip_hamiltonian_t h, size_t* bytes) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h != nullptr && bytes != nullptr, "null argument");
  size_t data = 0, work = 0, graph = 0, old = 0;
  for (const void* p : {(const void*)h->d_v, (const void*)h->d_xyz, (const void*)h->d_veff,
                        (const void*)h->d_matrices, (const void*)h->d_maps, (const void*)h->d_scals,
                        (const void*)h->d_pt,
                        (const void*)h->d_chunks, (const void*)h->d_mat_info, (const void*)h->d_prow,
                        (const void*)h->d_kslot, (const void*)h->d_kgrp, (const void*)h->d_kstep,
                        (const void*)h->d_kpt, (const void*)h->d_kphase,
                        (const void*)h->d_sblk, (const void*)h->d_spart, (const void*)h->d_kpoint,
                        (const void*)h->d_bnd_src, (const void*)h->d_phase, (const void*)h->d_phase_corr,
                        (const void*)h->d_pphase})
    data += dev_bytes(p);
  for (const auto& w : h->sets) {
    size_t b = 0;
    for (const void* p : {(const void*)w.partial, (const void*)w.proj, (const void*)w.ksum, (const void*)w.y0,
                          (const void*)w.y1, (const void*)w.y2, (const void*)w.dpart, (const void*)w.dw,
                          (const void*)w.ephase})
      b += dev_bytes(p);
    // sets handed to Taylor graphs are kept under negative keys
    if (reinterpret_cast<intptr_t>(w.s) < 0) graph += b;
    else work += b;
  }
  for (const auto& k : h->krylov) work += dev_bytes(k.vec) + dev_bytes(k.small);
  for (const void* p : h->retired) old += dev_bytes(p);
  bytes[0] = data;
  bytes[1] = work;
  bytes[2] = graph;
  bytes[3] = old;
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_hamiltonian_trim(octhip_hamiltonian_t h) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h != nullptr, "null hamiltonian handle");
  // retired buffers belong to no set and no graph; work queued before they were retired
  // may still read them, so wait for the device first
  OCTHIP_HIP(hipDeviceSynchronize());
  for (void* p : h->retired) dfree(p);
  h->retired.clear();
  return OCTHIP_SUCCESS;
}

namespace {
// H psi with the zero boundary (or the boundary rows as they are); reuse: the caller's next
// kernel reads hpsi
int finite_apply(octhip_hamiltonian_s* h, double* psi, double* hpsi, int ldf, int terms, int set_bc, bool reuse,
                 hipStream_t s) {
  const int L = 1 << ldf;
  const octhip_nl_operator_s* op = h->kin;
  int rc = ensure_work(h, ldf, s);
  if (rc) return rc;
  ApplyArgs a;
  std::memset(&a, 0, sizeof(a));
  fill_terms(h, terms, a);
  a.fi = psi;
  a.fo = hpsi;
  a.L = L;
  a.lim = set_bc ? op->np : op->np_part;
  a.reuse = reuse ? 1 : 0;
  // boundaries_set: the boundary rows are cleared inside the bra's launch when there is one
  return apply_store(h, a, s, set_bc ? psi : nullptr);
}
}  // namespace

extern "C" int octhip_hamiltonian_apply_batch(octhip_hamiltonian_t h, double* psi, double* hpsi, int ldf,
                                              int is_complex, int terms, int set_bc, void* stream) {
  OCTHIP_RANGE("octhip_hamiltonian_apply_batch");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h != nullptr, "null hamiltonian handle");
  OCTHIP_REQUIRE(psi && hpsi && psi != hpsi, "bad batch pointers");
  OCTHIP_REQUIRE(ldf >= 0 && ldf <= MAX_LDF, "ldf=%d outside 0..%d", ldf, MAX_LDF);
  OCTHIP_REQUIRE(!is_complex || ldf >= 1, "complex batch needs ldf >= 1");
  hipStream_t s = (hipStream_t)stream;
  if (is_periodic(h)) return periodic_apply(h, psi, hpsi, ldf, is_complex, terms, set_bc, false, s);
  return finite_apply(h, psi, hpsi, ldf, terms, set_bc, false, s);
}

namespace octhip {
int propagator_apply(octhip_hamiltonian_s* h, double* psi, double* hpsi, int ldf, hipStream_t s) {
  if (is_periodic(h)) return periodic_apply(h, psi, hpsi, ldf, 1, OCTHIP_TERM_ALL, 1, true, s);
  return finite_apply(h, psi, hpsi, ldf, OCTHIP_TERM_ALL, 1, true, s);
}
}  // namespace octhip

namespace octhip {
// zfact_k, k = 1..order: zfact *= (-i * deltat) / k (exponential.F90:720-724); deltat ->
// i*deltat in imaginary time (609-619).  z[0] = 1.
void taylor_coefs(double deltat, int imag_time, int order, std::complex<double>* z) {
  const std::complex<double> dt_c = imag_time ? std::complex<double>(0.0, deltat) : std::complex<double>(deltat, 0.0);
  const std::complex<double> mi(-0.0, -1.0);
  const std::complex<double> step(mi.real() * dt_c.real() - mi.imag() * dt_c.imag(),
                                  mi.real() * dt_c.imag() + mi.imag() * dt_c.real());
  z[0] = std::complex<double>(1.0, 0.0);
  for (int k = 1; k <= order; ++k) {
    const std::complex<double> p = z[k - 1];
    const std::complex<double> zz(p.real() * step.real() - p.imag() * step.imag(),
                                  p.real() * step.imag() + p.imag() * step.real());
    z[k] = std::complex<double>(zz.real() / k, zz.imag() / k);
  }
}

// Arguments of the fused pass H `in` for every term, boundary rows of `in` read as zero,
// ket rows taken from `ksum` (a work buffer of the caller's choice).
void h_apply_args(const octhip_hamiltonian_s* h, const double* in, int L, double* ksum, ApplyArgs& a) {
  std::memset(&a, 0, sizeof(a));
  fill_terms(h, OCTHIP_TERM_ALL, a);
  a.fi = in;
  a.L = L;
  a.lim = h->kin->np;
  // fill_terms points ksum at the handle's own buffer, which may not exist yet: the
  // caller's buffer replaces it whenever the nonlocal rows are used
  if (a.kslot) a.ksum = ksum;
}

int prepare_taylor(octhip_hamiltonian_s* h, int ldf, hipStream_t s) {
  int rc = ensure_work(h, ldf, s);
  if (!rc) rc = ensure_taylor(h, ldf, s);
  if (!rc) rc = prepare_operator(h->kin, 1 << ldf, h->nmat > 0 && h->nslot > 0);
  return rc;
}

int set_field(octhip_hamiltonian_s* h, const double field[3], hipStream_t s) {
  for (int d = 0; d < 3; ++d) h->field[d] = field[d];
  h->has_field = true;
  return update_veff(h, s);
}
}  // namespace octhip

extern "C" int octhip_exponential_taylor_batch(octhip_hamiltonian_t h, double* psi, int ldf, double deltat,
                                               int order, int imag_time, void* stream) {
  OCTHIP_RANGE("octhip_exponential_taylor_batch");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h && psi, "null argument");
  OCTHIP_REQUIRE(ldf >= 1 && ldf <= MAX_LDF, "Taylor needs a complex batch (ldf in 1..%d)", MAX_LDF);
  OCTHIP_REQUIRE(order >= 1 && order <= 32, "order %d outside 1..32", order);
  if (is_periodic(h)) return taylor_apply(h, psi, ldf, deltat, order, imag_time, TaylorOptions(), (hipStream_t)stream);
  int rc = prepare_taylor(h, ldf, (hipStream_t)stream);
  if (rc) return rc;
  return taylor_step(h, psi, ldf, deltat, order, imag_time, nullptr, (hipStream_t)stream, nullptr);
}

// ---------------------------------------------------------------- graphs --
struct octhip_taylor_graph_s {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  // the Hamiltonian whose work sets this graph was captured with, and their keys there
  octhip_hamiltonian_s* h = nullptr;
  std::vector<hipStream_t> set_keys;
};

namespace {
void detach_graph(octhip_taylor_graph_t g) {
  g->h = nullptr;
  g->set_keys.clear();
}
}  // namespace

extern "C" int octhip_taylor_graph_create(octhip_hamiltonian_t h, double* const* psi, int nbatch, int ldf,
                                          double deltat, int order, int imag_time, void* stream,
                                          octhip_taylor_graph_t* out) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h && psi && out && nbatch > 0, "bad argument");
  OCTHIP_REQUIRE(ldf >= 1 && ldf <= MAX_LDF, "Taylor needs a complex batch (ldf in 1..%d)", MAX_LDF);
  OCTHIP_REQUIRE(order >= 1 && order <= 32, "order %d outside 1..32", order);
  *out = nullptr;
  if (is_periodic(h))
    return fail(OCTHIP_ERR_UNSUPPORTED, "taylor_graph: periodic handles and Bloch phases run eagerly");
  // Batch b runs on branch b mod nbr of the graph (the capturing stream and up to three
  // more, forked and joined with events), as the reference gives every batch its own
  // stream (src/td/propagation_ops_elec.F90:236): the kernels of different batches
  // overlap, each branch with its own work buffers (measured, 4 batches of 32 states on
  // the R=12 sphere: 4.34 ms per step on one branch, 3.84 on two, 3.75 on four).
  constexpr int MAX_BRANCHES = 4;
  const int nbr = std::min(nbatch, MAX_BRANCHES);
  hipStream_t br[MAX_BRANCHES] = {};      // br[0] is the capturing stream, set below
  hipEvent_t fork = nullptr, join[MAX_BRANCHES] = {};
  auto cleanup = [&]() {
    if (fork) (void)hipEventDestroy(fork);
    for (int k = 1; k < nbr; ++k) {
      if (join[k]) (void)hipEventDestroy(join[k]);
      if (br[k]) (void)hipStreamDestroy(br[k]);
    }
  };
  bool ok = nbr == 1 || hipEventCreateWithFlags(&fork, hipEventDisableTiming) == hipSuccess;
  for (int k = 1; k < nbr && ok; ++k)
    ok = hipStreamCreateWithFlags(&br[k], hipStreamNonBlocking) == hipSuccess &&
         hipEventCreateWithFlags(&join[k], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    cleanup();
    return fail(OCTHIP_ERR_HIP, "taylor_graph_create: stream or event creation failed");
  }
  hipStream_t used = nullptr;
  int rc = capture_graph((hipStream_t)stream,
                       [&](hipStream_t cs) {
                         used = cs;
                         int r = prepare_taylor(h, ldf, cs);
                         for (int k = 1; k < nbr && !r; ++k) r = prepare_taylor(h, ldf, br[k]);
                         return r;
                       },
                       [&](hipStream_t cs) {
                         br[0] = cs;
                         if (nbr > 1) OCTHIP_HIP(hipEventRecord(fork, cs));
                         for (int k = 1; k < nbr; ++k) OCTHIP_HIP(hipStreamWaitEvent(br[k], fork, 0));
                         int r = OCTHIP_SUCCESS;
                         for (int b = 0; b < nbatch && !r; ++b)
                           r = taylor_step(h, psi[b], ldf, deltat, order, imag_time, nullptr, br[b % nbr], nullptr);
                         for (int k = 1; k < nbr; ++k) {
                           OCTHIP_HIP(hipEventRecord(join[k], br[k]));
                           OCTHIP_HIP(hipStreamWaitEvent(cs, join[k], 0));
                         }
                         return r;
                       },
                       out);
  if (rc) {
    // the sets prepared for streams that no longer exist (the branch streams, and the
    // private capturing stream when stream == NULL) go; the caller's stream keeps its own
    for (int k = 1; k < nbr; ++k) drop_workset(h, br[k]);
    if (!stream && used) drop_workset(h, used);
    cleanup();
    return rc;
  }
  // the graph owns the buffers it was captured with (later calls on any stream get
  // others) and frees them when it is destroyed
  octhip_taylor_graph_t g = *out;
  g->h = h;
  for (int k = 0; k < nbr; ++k) {
    const hipStream_t key = pin_workset(h, k == 0 ? used : br[k]);
    if (key) g->set_keys.push_back(key);
  }
  h->graphs.push_back(g);
  cleanup();
  return OCTHIP_SUCCESS;
}

namespace octhip {
// Capture the launches `body` issues on a capturing stream into an instantiated graph.
int capture_graph(hipStream_t s, const std::function<int(hipStream_t)>& prepare,
                  const std::function<int(hipStream_t)>& body, octhip_taylor_graph_t* out) {
  hipStream_t cs = s;
  bool own = false;
  if (!cs) {  // the legacy default stream cannot be captured
    OCTHIP_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    own = true;
  }
  if (prepare) {
    int prc = prepare(cs);
    if (prc) {
      if (own) (void)hipStreamDestroy(cs);
      return prc;
    }
  }
  OCTHIP_HIP(hipStreamSynchronize(cs));
  hipError_t e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) {
    if (own) (void)hipStreamDestroy(cs);
    return fail(OCTHIP_ERR_HIP, "hipStreamBeginCapture: %s", hipGetErrorString(e));
  }
  set_capturing(true);
  int rc = body(cs);
  set_capturing(false);
  hipGraph_t graph = nullptr;
  e = hipStreamEndCapture(cs, &graph);
  if (own) (void)hipStreamDestroy(cs);
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
  auto* g = new octhip_taylor_graph_s();
  g->graph = graph;
  e = hipGraphInstantiate(&g->exec, graph, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    (void)hipGraphDestroy(graph);
    delete g;
    return fail(OCTHIP_ERR_HIP, "hipGraphInstantiate: %s", hipGetErrorString(e));
  }
  *out = g;
  return OCTHIP_SUCCESS;
}

hipStream_t pin_workset(octhip_hamiltonian_s* h, hipStream_t s) {
  for (auto& w : h->sets)
    if (w.s == s) {
      w.s = reinterpret_cast<hipStream_t>(static_cast<intptr_t>(-(++h->graph_sets)));
      return w.s;
    }
  return nullptr;
}

void drop_workset(octhip_hamiltonian_s* h, hipStream_t s) {
  for (size_t i = 0; i < h->sets.size(); ++i) {
    if (h->sets[i].s != s) continue;
    const auto w = h->sets[i];
    for (void* p : {(void*)w.partial, (void*)w.proj, (void*)w.ksum, (void*)w.y0, (void*)w.y1, (void*)w.y2,
                    (void*)w.dpart, (void*)w.dw, (void*)w.ephase})
      dfree(p);
    h->sets.erase(h->sets.begin() + (long)i);
    // the mirrored pointers may name the freed set: they are rebound by the next call
    h->d_partial = h->d_proj = h->d_ksum = h->d_y[0] = h->d_y[1] = h->d_y[2] = nullptr;
    h->work_ldf = h->y_ldf = -1;
    return;
  }
}
}  // namespace octhip

extern "C" int octhip_taylor_graph_launch(octhip_taylor_graph_t g, void* stream) {
  OCTHIP_RANGE("octhip_taylor_graph_launch");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(g != nullptr, "null graph");
  ProfScope prof("taylor_graph", (hipStream_t)stream);
  OCTHIP_HIP(hipGraphLaunch(g->exec, (hipStream_t)stream));
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_taylor_graph_destroy(octhip_taylor_graph_t g) {
  if (!g) return OCTHIP_SUCCESS;
  if (g->h) {
    // launches of the graph may still be running on any stream
    (void)hipDeviceSynchronize();
    for (hipStream_t key : g->set_keys) drop_workset(g->h, key);
    auto& gs = g->h->graphs;
    gs.erase(std::remove(gs.begin(), gs.end(), g), gs.end());
  }
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  delete g;
  return OCTHIP_SUCCESS;
}

namespace octhip {
// One Taylor step in place.  save (optional, order pointers to np-row buffers) receives
// save[0] = psi (boundary cleared) and save[k] = H^k psi for k = 1..order-1: the terms the
// discrete adjoint contracts with the backward states.
int taylor_step(octhip_hamiltonian_s* h, double* psi, int ldf, double deltat, int order, int imag_time,
                double* const* save, hipStream_t s, const double* psi_in, const double* v_override) {
  const int L = 1 << ldf;
  const octhip_nl_operator_s* op = h->kin;
  int rc = prepare_taylor(h, ldf, s);  // the work buffers of stream s (allocated before a capture)
  if (rc) return rc;
  const double* src = psi_in ? psi_in : psi;
  // in place: psi's boundary rows are cleared by the first bra launch (or here when there
  // is no nonlocal term); every pass reads boundary rows as zero (lim = np) in any case.
  // Out of place (psi_in): only the np inner rows of psi are written.
  if (!psi_in && h->nmat == 0) {
    rc = zero_boundary(psi, op->np, op->np_part, L, s);
    if (rc) return rc;
  }
  if (save && save[0] != src)
    OCTHIP_HIP(hipMemcpyAsync(save[0], src, sizeof(double) * op->np * L, hipMemcpyDeviceToDevice, s));
  if (psi_in && order == 1)  // the order-1 axpy works in place on psi
    OCTHIP_HIP(hipMemcpyAsync(psi, psi_in, sizeof(double) * op->np * L, hipMemcpyDeviceToDevice, s));
  std::complex<double> zf[33];
  taylor_coefs(deltat, imag_time, order, zf);
  if (taylor_deferred(order)) {
    // y_k = H y_{k-1} (y_0 = psi) stored for k < order (save[k] when saving); the last
    // pass forms psi + z_1 y_1 + ... + z_order H y_{order-1}, adding the terms in order k,
    // as exponential.F90:733-744 accumulates them order by order.  No accumulator is
    // read and written at the orders in between.
    auto Y = [&](int k) -> double* { return save ? save[k] : h->d_y[k - 1]; };
    for (int k = 1; k <= order; ++k) {
      const double* yin = (k == 1) ? src : Y(k - 1);
      double* const bc = (k == 1 && h->nmat > 0 && !psi_in) ? psi : nullptr;
      ApplyArgs a;
      std::memset(&a, 0, sizeof(a));
      fill_terms(h, OCTHIP_TERM_ALL, a);
      if (v_override) a.v = v_override;
      a.fi = yin;
      a.L = L;
      a.lim = op->np;  // boundary rows are zero: psi's were just cleared, work buffers have none
      a.reuse = 1;
      if (k < order) {
        a.fo = Y(k);
        rc = apply_store(h, a, s, bc);
      } else {
        rc = run_bra(h, yin, L, s, bc);
        if (rc) return rc;
        a.acc = psi;
        a.acc_in = psi_in;  // null: in place
        if (order >= 3) {
          a.ya = Y(1);
          a.car = zf[1].real();
          a.cai = zf[1].imag();
        }
        if (order >= 4) {
          a.yb = Y(2);
          a.cbr = zf[2].real();
          a.cbi = zf[2].imag();
        }
        a.has_c1 = 1;  // the pass's own input y_{order-1}
        a.c1r = zf[order - 1].real();
        a.c1i = zf[order - 1].imag();
        a.c2r = zf[order].real();
        a.c2i = zf[order].imag();
        rc = launch_operator(h->kin, a, EPI_TAYLOR, s);
      }
      if (rc) return rc;
    }
    return OCTHIP_SUCCESS;
  }
  std::complex<double> z, z1;
  for (int k = 1; k <= order; ++k) {
    z = zf[k];
    const double* yin = (k == 1) ? src : (save ? save[k - 1] : h->d_y[(k - 2) & 1]);
    double* yout = (k < order) ? (save ? save[k] : h->d_y[(k - 1) & 1]) : nullptr;
    rc = run_bra(h, yin, L, s, (k == 1 && h->nmat > 0 && !psi_in) ? psi : nullptr);
    if (rc) return rc;
    ApplyArgs a;
    std::memset(&a, 0, sizeof(a));
    fill_terms(h, OCTHIP_TERM_ALL, a);
    if (v_override) a.v = v_override;
    a.fi = yin;
    a.L = L;
    a.lim = op->np;  // boundary rows are zero: psi's were just cleared, work buffers have none
    a.reuse = 1;
    if (order == 1) {
      a.fo = h->d_y[0];
      rc = launch_operator(h->kin, a, EPI_STORE, s);
      if (rc) return rc;
      const size_t count = (size_t)op->np * L;
      size_t grid = std::min<size_t>((count + BLOCK - 1) / BLOCK, 8192);
      ProfScope prof("k_zaxpy", s);
      hipLaunchKernelGGL(k_zaxpy, dim3((unsigned)grid), dim3(BLOCK), 0, s, psi, h->d_y[0], count, z.real(), z.imag());
      OCTHIP_HIP(hipGetLastError());
      break;
    }
    a.yout = yout;
    if (k == 1) {
      a.acc = nullptr;
      z1 = z;
    } else {
      a.acc = psi;
      a.acc_in = (k == 2) ? psi_in : nullptr;  // from the third order on psi holds the sum
      a.has_c1 = (k == 2);
      a.c1r = z1.real();
      a.c1i = z1.imag();
      a.c2r = z.real();
      a.c2i = z.imag();
    }
    rc = launch_operator(h->kin, a, EPI_TAYLOR, s);
    if (rc) return rc;
  }
  return OCTHIP_SUCCESS;
}
}  // namespace octhip

namespace octhip {
namespace {
// density buffers of stream s: nchunk x np partials and the weights of 2^(ldf-1) states
int ensure_density(octhip_hamiltonian_s* h, int nchunk, hipStream_t s, double** dpart, double** dw) {
  auto& w = workset(h, s);
  if (!w.dw) {
    int rc = dalloc((void**)&w.dw, sizeof(double) << (MAX_LDF - 1));
    if (rc) return rc;
  }
  if (nchunk > 0 && w.dchunks < nchunk) {
    if (w.dpart) h->retired.push_back(w.dpart);
    w.dpart = nullptr;
    w.dchunks = 0;
    int rc = dalloc((void**)&w.dpart, sizeof(double) * (size_t)nchunk * h->np);
    if (rc) return rc;
    w.dchunks = nchunk;
  }
  *dpart = w.dpart;
  *dw = w.dw;
  return OCTHIP_SUCCESS;
}

// zfact_k of exponential_taylor_series_batch (src/electrons/exponential.F90:716-720) for a
// complex deltat: zfact_0 (1, or deltat with an inhomogeneous term) and
// zfact_k = zfact_{k-1} (-i deltat) / (k [+1]), with the products written out as the
// oracle does.
void series_coefs(std::complex<double> dt, bool inh, int order, std::complex<double>* z) {
  const double mr = -0.0, mi = -1.0;
  const double sr = mr * dt.real() - mi * dt.imag(), si = mr * dt.imag() + mi * dt.real();
  z[0] = inh ? dt : std::complex<double>(1.0, 0.0);
  for (int k = 1; k <= order; ++k) {
    const int denom = inh ? k + 1 : k;
    const double tr = z[k - 1].real() * sr - z[k - 1].imag() * si;
    const double ti = z[k - 1].real() * si + z[k - 1].imag() * sr;
    z[k] = std::complex<double>(tr / denom, ti / denom);
  }
}

// One series of exponential_taylor_series_batch, kernel by kernel: psi2 = psi (np rows)
// first when given; with inh, psi (psi2) += real(zfact_0) inh and the chain of H-applies
// starts from inh; each order stores y_k = H y_{k-1} and adds zfact_k y_k to psi and
// zfact2_k y_k to psi2 (the reference's axpy per order, 733-744).
int series_generic(octhip_hamiltonian_s* h, double* psi, int ldf, std::complex<double> dt, int order,
                   double* psi2, std::complex<double> dt2, double* inh, hipStream_t s) {
  const int L = 1 << ldf;
  const size_t count = (size_t)h->np * L;
  int rc = prepare_taylor(h, ldf, s);
  if (rc) return rc;
  std::complex<double> z[34], z2[34];
  series_coefs(dt, inh != nullptr, order, z);
  series_coefs(dt2, inh != nullptr, order, z2);
  if (psi2) OCTHIP_HIP(hipMemcpyAsync(psi2, psi, sizeof(double) * count, hipMemcpyDeviceToDevice, s));
  if (inh) {
    rc = launch_daxpy(psi, inh, count, z[0].real(), s);
    if (!rc && psi2) rc = launch_daxpy(psi2, inh, count, z2[0].real(), s);
    if (rc) return rc;
  }
  double* src = inh ? inh : psi;
  // periodic handles: the chain needs np_part rows (its boundary rows are filled from the
  // periodic images by every apply), taken from the stream's Krylov buffers
  double* ychain[2] = {h->d_y[0], h->d_y[1]};
  if (is_periodic(h)) {
    double* base = nullptr;
    rc = krylov_vectors(h, s, 2, ldf, &base);
    if (rc) return rc;
    ychain[0] = base;
    ychain[1] = base + ((size_t)h->kin->np_part << ldf);
  }
  for (int k = 1; k <= order; ++k) {
    double* yin = (k == 1) ? src : ychain[(k - 2) & 1];
    double* yout = ychain[(k - 1) & 1];
    if (is_periodic(h)) {
      rc = propagator_apply(h, yin, yout, ldf, s);
    } else {
      ApplyArgs a;
      std::memset(&a, 0, sizeof(a));
      fill_terms(h, OCTHIP_TERM_ALL, a);
      a.fi = yin;
      a.fo = yout;
      a.L = L;
      a.lim = h->np;
      a.reuse = 1;
      // boundaries_set of the chain's input (its H-apply, set_bc default)
      rc = apply_store(h, a, s, k == 1 ? src : nullptr);
    }
    if (!rc) rc = launch_zaxpy(psi, yout, count, z[k].real(), z[k].imag(), s);
    if (!rc && psi2) rc = launch_zaxpy(psi2, yout, count, z2[k].real(), z2[k].imag(), s);
    if (rc) return rc;
  }
  return OCTHIP_SUCCESS;
}

// The homogeneous series at orders 2..4 with the deferred accumulation: plain H-apply
// passes store y_k = H^k psi (k < order); the last pass forms psi (and psi2 with the
// deltat2 factors, from the same inputs) and, when dpart is given, the density partials of
// the final states.
int series_fused(octhip_hamiltonian_s* h, double* psi, int ldf, std::complex<double> dt, int order,
                 double* psi2, std::complex<double> dt2, double* dpart, const double* dw, hipStream_t s) {
  const int L = 1 << ldf;
  int rc = prepare_taylor(h, ldf, s);
  if (rc) return rc;
  std::complex<double> z[34], z2[34];
  series_coefs(dt, false, order, z);
  series_coefs(dt2, false, order, z2);
  if (h->nmat == 0) {
    rc = zero_boundary(psi, h->np, h->kin->np_part, L, s);
    if (rc) return rc;
  }
  for (int k = 1; k <= order; ++k) {
    const double* yin = (k == 1) ? psi : h->d_y[k - 2];
    double* const bc = (k == 1 && h->nmat > 0) ? psi : nullptr;
    ApplyArgs a;
    std::memset(&a, 0, sizeof(a));
    fill_terms(h, OCTHIP_TERM_ALL, a);
    a.fi = yin;
    a.L = L;
    a.lim = h->np;
    a.reuse = 1;
    if (k < order) {
      a.fo = h->d_y[k - 1];
      rc = apply_store(h, a, s, bc);
      if (rc) return rc;
      continue;
    }
    rc = run_bra(h, yin, L, s, bc);
    if (rc) return rc;
    a.acc = psi;
    if (order >= 3) {
      a.ya = h->d_y[0];
      a.car = z[1].real();
      a.cai = z[1].imag();
      a.dar = z2[1].real();
      a.dai = z2[1].imag();
    }
    if (order >= 4) {
      a.yb = h->d_y[1];
      a.cbr = z[2].real();
      a.cbi = z[2].imag();
      a.dbr = z2[2].real();
      a.dbi = z2[2].imag();
    }
    a.has_c1 = 1;
    a.c1r = z[order - 1].real();
    a.c1i = z[order - 1].imag();
    a.c2r = z[order].real();
    a.c2i = z[order].imag();
    a.d1r = z2[order - 1].real();
    a.d1i = z2[order - 1].imag();
    a.d2r = z2[order].real();
    a.d2i = z2[order].imag();
    a.acc2 = psi2;
    a.dpart = dpart;
    a.dw = dw;
    return launch_operator(h->kin, a, EPI_TAYLOR_X, s);
  }
  return OCTHIP_SUCCESS;
}
}  // namespace

int taylor_apply(octhip_hamiltonian_s* h, double* psi, int ldf, double deltat, int order, int imag_time,
                 const TaylorOptions& o, hipStream_t s) {
  const int L = 1 << ldf;
  const std::complex<double> dt = imag_time ? std::complex<double>(0.0, deltat) : std::complex<double>(deltat, 0.0);
  const std::complex<double> dt2 =
      imag_time ? std::complex<double>(0.0, o.deltat2) : std::complex<double>(o.deltat2, 0.0);
  double* dpart = nullptr;
  double* dw = nullptr;
  int rc = OCTHIP_SUCCESS;
  // periodic handles (psi carries the Bloch phase): plain passes through the periodic apply
  const bool fused = taylor_deferred(order) && !is_periodic(h);
  const bool fuse_density = o.density && fused && !o.inh;
  int nchunk = 0;
  if (o.density) {
    // density partials per lane chunk when the last pass forms them, else none
    ApplyArgs probe;
    std::memset(&probe, 0, sizeof(probe));
    fill_terms(h, OCTHIP_TERM_ALL, probe);
    probe.L = L;
    nchunk = fuse_density ? apply_lane_chunks(h->kin, probe) : 0;
    rc = ensure_density(h, nchunk, s, &dpart, &dw);
    if (rc) return rc;
    OCTHIP_HIP(hipMemcpyAsync(dw, o.weights, sizeof(double) * (L / 2), hipMemcpyHostToDevice, s));
  }
  if (fused) {
    rc = series_fused(h, psi, ldf, dt, order, o.psi2, dt2, fuse_density ? dpart : nullptr, dw, s);
  } else {
    rc = series_generic(h, psi, ldf, dt, order, o.psi2, dt2, nullptr, s);
  }
  if (!rc && o.inh) rc = series_generic(h, psi, ldf, dt, order, o.psi2, dt2, o.inh, s);
  if (rc || !o.density) return rc;
  if (fuse_density) return launch_density_reduce(o.density, dpart, nchunk, h->np, s);
  return launch_density(o.psi2 ? o.psi2 : psi, L, h->np, 1, dw, o.density, s);
}
}  // namespace octhip

extern "C" int octhip_exponential_apply_batch(octhip_hamiltonian_t h, double* psi, int ldf, double deltat,
                                              int order, int imag_time, double* psi2, double deltat2,
                                              double* inh, const double* weights, double* density,
                                              void* stream) {
  OCTHIP_RANGE("octhip_exponential_apply_batch");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h && psi, "null argument");
  OCTHIP_REQUIRE(ldf >= 1 && ldf <= MAX_LDF, "Taylor needs a complex batch (ldf in 1..%d)", MAX_LDF);
  OCTHIP_REQUIRE(order >= 1 && order <= 32, "order %d outside 1..32", order);
  OCTHIP_REQUIRE(psi2 != psi && inh != psi && (!psi2 || psi2 != inh), "psi, psi2 and inh must be distinct");
  OCTHIP_REQUIRE((weights == nullptr) == (density == nullptr), "weights and density go together");
  TaylorOptions o;
  o.psi2 = psi2;
  o.deltat2 = deltat2;
  o.inh = inh;
  o.weights = weights;
  o.density = density;
  return taylor_apply(h, psi, ldf, deltat, order, imag_time, o, (hipStream_t)stream);
}

extern "C" int octhip_density_accumulate(const double* psi, int ldf, int np, int is_complex, const double* weights,
                                         double* density, void* stream) {
  OCTHIP_RANGE("octhip_density_accumulate");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(psi && weights && density, "null argument");
  OCTHIP_REQUIRE(ldf >= (is_complex ? 1 : 0) && ldf <= MAX_LDF, "ldf=%d outside the packed range", ldf);
  OCTHIP_REQUIRE(np >= 0, "np < 0");
  return launch_density(psi, 1 << ldf, np, is_complex ? 1 : 0, weights, density, (hipStream_t)stream);
}

namespace {
// density = 0 over np doubles with a fill kernel (density_calc_init)
int clear_density(double* density, int np, hipStream_t s) {
  const unsigned grid = (unsigned)std::min((np + BLOCK - 1) / BLOCK, 8192);
  hipLaunchKernelGGL(k_zero_rows, dim3(grid), dim3(BLOCK), 0, s, density, (size_t)0, (size_t)np);
  OCTHIP_HIP(hipGetLastError());
  return OCTHIP_SUCCESS;
}

// propagation_ops_elec_exp_apply / _fuse_density_exp_apply over the batches
// (src/td/propagation_ops_elec.F90:213-333): every batch propagated by dt in turn, the
// density of the results accumulated when requested
int exp_apply_batches(octhip_hamiltonian_s* h, double* const* psi, int nbatch, int ldf, double dt, int order,
                      const double* weights, double* density, hipStream_t s) {
  const int pack = 1 << (ldf - 1);
  if (density) {
    int rc = clear_density(density, h->np, s);
    if (rc) return rc;
  }
  for (int b = 0; b < nbatch; ++b) {
    TaylorOptions o;
    if (density) {
      o.weights = weights + (size_t)b * pack;
      o.density = density;
    }
    // k-points: set_phase_corr / unset_phase_corr around the apply
    // (src/td/propagation_ops_elec.F90:238-246)
    int rc = h->has_kpoint ? launch_phase(psi[b], psi[b], h->d_phase, h->np, 1 << ldf, false, s) : 0;
    if (!rc) rc = taylor_apply(h, psi[b], ldf, dt, order, 0, o, s);
    if (!rc && h->has_kpoint) rc = launch_phase(psi[b], psi[b], h->d_phase, h->np, 1 << ldf, true, s);
    if (rc) return rc;
  }
  return OCTHIP_SUCCESS;
}

int check_driver_args(octhip_hamiltonian_s* h, double* const* psi, int nbatch, int ldf, int order,
                      const double* weights, double* density) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h && psi && nbatch > 0, "bad argument");
  OCTHIP_REQUIRE(ldf >= 1 && ldf <= MAX_LDF, "propagators need complex batches (ldf in 1..%d)", MAX_LDF);
  OCTHIP_REQUIRE(order >= 1 && order <= 32, "order %d outside 1..32", order);
  OCTHIP_REQUIRE((weights == nullptr) == (density == nullptr), "weights and density go together");
  for (int b = 0; b < nbatch; ++b) OCTHIP_REQUIRE(psi[b] != nullptr, "batch %d is null", b);
  return OCTHIP_SUCCESS;
}
}  // namespace

extern "C" int octhip_propagator_expmid(octhip_hamiltonian_t h, double* const* psi, int nbatch, int ldf, double dt,
                                        int order, const double* field_mid, const double* weights, double* density,
                                        void* stream) {
  OCTHIP_RANGE("octhip_propagator_expmid");
  int rc = check_driver_args(h, psi, nbatch, ldf, order, weights, density);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (field_mid) {
    OCTHIP_REQUIRE(h->d_xyz != nullptr, "propagator_expmid: positions never uploaded (set_dipole_field)");
    rc = set_field(h, field_mid, s);
    if (rc) return rc;
  }
  return exp_apply_batches(h, psi, nbatch, ldf, dt, order, weights, density, s);
}

extern "C" int octhip_propagator_etrs(octhip_hamiltonian_t h, double* const* psi, int nbatch, int ldf, double dt,
                                     int order, const double* field_old, const double* field_new,
                                     const double* weights, double* density, void* stream) {
  OCTHIP_RANGE("octhip_propagator_etrs");
  int rc = check_driver_args(h, psi, nbatch, ldf, order, weights, density);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  OCTHIP_REQUIRE(!(field_old || field_new) || h->d_xyz != nullptr,
                 "propagator_etrs: positions never uploaded (set_dipole_field)");
  if (field_old) {
    rc = set_field(h, field_old, s);
    if (rc) return rc;
  }
  // dt/2 with H(t - dt), then the Hamiltonian at t and dt/2 with the density
  rc = exp_apply_batches(h, psi, nbatch, ldf, 0.5 * dt, order, nullptr, nullptr, s);
  if (rc) return rc;
  if (field_new) {
    rc = set_field(h, field_new, s);
    if (rc) return rc;
  }
  return exp_apply_batches(h, psi, nbatch, ldf, 0.5 * dt, order, weights, density, s);
}

// ------------------------------------------------------- periodic / k-points --
extern "C" int octhip_hamiltonian_set_periodic(octhip_hamiltonian_t h, const int* bnd_src) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h != nullptr, "null hamiltonian handle");
  // a captured Taylor graph keeps the zero-boundary launches it was built with
  OCTHIP_REQUIRE(h->graphs.empty(), "destroy the Taylor graphs of this Hamiltonian before changing its boundaries");
  const int np = h->np, nb = h->kin->np_part - h->np;
  (void)hipDeviceSynchronize();  // launches in flight may read the old map
  dfree(h->d_bnd_src);
  h->d_bnd_src = nullptr;
  h->nbnd = 0;
  h->periodic = false;
  if (!bnd_src) return OCTHIP_SUCCESS;
  for (int b = 0; b < nb; ++b)
    OCTHIP_REQUIRE(bnd_src[b] >= 0 && bnd_src[b] < np, "boundary row %d: image %d outside 0..np-1", np + b,
                   bnd_src[b]);
  int rc = upload(&h->d_bnd_src, bnd_src, (size_t)nb, nullptr);
  if (rc) return rc;
  h->nbnd = nb;
  h->periodic = true;
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_hamiltonian_set_phases(octhip_hamiltonian_t h, const double* phase, const double* phase_corr,
                                             const double* projector_phases) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h != nullptr, "null hamiltonian handle");
  OCTHIP_REQUIRE(h->graphs.empty(), "destroy the Taylor graphs of this Hamiltonian before setting Bloch phases");
  const int np_part = h->kin->np_part, nb = np_part - h->np;
  (void)hipDeviceSynchronize();
  for (double** p : {&h->d_phase, &h->d_phase_corr, &h->d_pphase, &h->d_kphase}) {
    dfree(*p);
    *p = nullptr;
  }
  h->has_kpoint = false;
  if (!phase) return OCTHIP_SUCCESS;
  OCTHIP_REQUIRE(nb == 0 || phase_corr, "phase_corr is required with the phase (one per boundary row)");
  OCTHIP_REQUIRE(h->nmat == 0 || projector_phases, "projector_phases are required with projectors");
  int rc = upload(&h->d_phase, phase, 2 * (size_t)np_part, nullptr);
  if (!rc && nb > 0) rc = upload(&h->d_phase_corr, phase_corr, 2 * (size_t)nb, nullptr);
  if (!rc && h->nmat > 0) rc = upload(&h->d_pphase, projector_phases, 2 * (size_t)h->total_points, nullptr);
  std::vector<double> by_entry(2 * h->kg.size());
  for (size_t e = 0; e < h->kg.size(); ++e)
    for (int c = 0; c < 2; ++c) by_entry[2 * e + c] = projector_phases[2 * (size_t)h->kg[e] + c];
  if (!rc) rc = upload(&h->d_kphase, by_entry.data(), by_entry.size(), nullptr);
  if (rc) return rc;
  h->has_kpoint = true;
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_hamiltonian_apply_batch_phase(octhip_hamiltonian_t h, double* psi, double* hpsi, int ldf,
                                                    int terms, int set_bc, int psi_has_phase, void* stream) {
  OCTHIP_RANGE("octhip_hamiltonian_apply_batch_phase");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h != nullptr, "null hamiltonian handle");
  OCTHIP_REQUIRE(psi && hpsi && psi != hpsi, "bad batch pointers");
  OCTHIP_REQUIRE(ldf >= 1 && ldf <= MAX_LDF, "a complex batch is needed (ldf in 1..%d)", MAX_LDF);
  OCTHIP_REQUIRE(!psi_has_phase || h->has_kpoint, "psi_has_phase without Bloch phases on the handle");
  OCTHIP_REQUIRE(set_bc || !psi_has_phase || !h->periodic,
                 "a batch with the phase needs set_bc (the phase correction is applied while setting the boundary)");
  hipStream_t s = (hipStream_t)stream;
  if (!is_periodic(h)) return octhip_hamiltonian_apply_batch(h, psi, hpsi, ldf, 1, terms, set_bc, stream);
  return periodic_apply(h, psi, hpsi, ldf, 1, terms, set_bc, psi_has_phase != 0, s);
}

extern "C" int octhip_hamiltonian_base_phase(octhip_hamiltonian_t h, double* psi, const double* src, int ldf, int np,
                                             int conjugate, void* stream) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(h && psi, "null argument");
  OCTHIP_REQUIRE(h->has_kpoint, "no Bloch phases on this handle");
  OCTHIP_REQUIRE(ldf >= 1 && ldf <= MAX_LDF, "a complex batch is needed (ldf in 1..%d)", MAX_LDF);
  OCTHIP_REQUIRE(np >= 0 && np <= h->kin->np_part, "np=%d outside 0..np_part", np);
  return launch_phase(psi, src ? src : psi, h->d_phase, np, 1 << ldf, conjugate != 0, (hipStream_t)stream);
}
