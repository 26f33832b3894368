// nl_operator handle: upload of the run-compressed stencil, lattice rebuild, operate.
#include <algorithm>
#include <climits>
#include <cstring>
#include <deque>

#include <map>
#include <queue>

#include "zmarch.h"

using namespace octhip;

namespace {

// Rebuild lattice coordinates from the run-compressed neighbour table: start at point 0,
// walk every stencil edge p -> p + ri[run(p)][j] assigning coords(p) + points[j], and
// reject the table if any point would receive two different coordinates.
bool rebuild_lattice(int n, const int* pts, const int* ri, const std::vector<int>& rimap, int np,
                     int np_part, std::vector<int>& coords) {
  coords.assign(3 * (size_t)np_part, INT_MIN);
  std::vector<char> seen(np_part, 0);
  std::deque<int> work;
  int visited = 0;
  for (int start = 0; start < np; ++start) {
    if (seen[start]) continue;
    if (start != 0) return false;  // disconnected inner set: no single lattice
    seen[start] = 1;
    coords[0] = coords[1] = coords[2] = 0;
    work.push_back(start);
    while (!work.empty()) {
      const int p = work.front();
      work.pop_front();
      ++visited;
      const int* row = ri + (size_t)rimap[p] * n;
      for (int j = 0; j < n; ++j) {
        const long qq = (long)p + row[j];
        if (qq < 0 || qq >= np_part) return false;
        const int q = (int)qq;
        int c[3];
        for (int d = 0; d < 3; ++d) c[d] = coords[3 * (size_t)p + d] + pts[3 * j + d];
        if (coords[3 * (size_t)q] == INT_MIN) {
          for (int d = 0; d < 3; ++d) coords[3 * (size_t)q + d] = c[d];
        } else {
          for (int d = 0; d < 3; ++d)
            if (coords[3 * (size_t)q + d] != c[d]) return false;
        }
        if (q < np && !seen[q]) {
          seen[q] = 1;
          work.push_back(q);
        }
      }
    }
  }
  if (visited != np) return false;
  for (int q = np; q < np_part; ++q)  // boundary points never reached by any stencil
    if (coords[3 * (size_t)q] == INT_MIN) coords[3 * (size_t)q] = coords[3 * (size_t)q + 1] = coords[3 * (size_t)q + 2] = INT_MIN;
  return true;
}

int build_site_map(octhip_nl_operator_s* op, const int* pts, hipStream_t s) {
  const int np = op->np, np_part = op->np_part, n = op->n;
  const std::vector<int>& c = op->coords;
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
  for (int q = 0; q < np_part; ++q) {
    if (c[3 * (size_t)q] == INT_MIN) continue;
    for (int d = 0; d < 3; ++d) {
      lo[d] = std::min(lo[d], c[3 * (size_t)q + d]);
      hi[d] = std::max(hi[d], c[3 * (size_t)q + d]);
    }
  }
  // pad by the stencil reach so every site + delta of an inner point is inside
  int reach = 0;
  for (int j = 0; j < n; ++j)
    for (int d = 0; d < 3; ++d) reach = std::max(reach, std::abs(pts[3 * j + d]));
  long sz[3];
  for (int d = 0; d < 3; ++d) {
    lo[d] -= reach;
    hi[d] += reach;
    sz[d] = (long)hi[d] - lo[d] + 1;
  }
  const long nsite = sz[0] * sz[1] * sz[2];
  if (nsite > (long)INT_MAX / 2) return fail(OCTHIP_ERR_UNSUPPORTED, "lattice too large (%ld sites)", nsite);
  std::vector<int> cube((size_t)nsite, -1);
  std::vector<int> cidx(np);
  for (int q = 0; q < np_part; ++q) {
    if (c[3 * (size_t)q] == INT_MIN) continue;
    const long site = (c[3 * (size_t)q] - lo[0]) + sz[0] * ((c[3 * (size_t)q + 1] - lo[1]) + sz[1] * (long)(c[3 * (size_t)q + 2] - lo[2]));
    if (cube[site] != -1) return fail(OCTHIP_ERR_INVALID, "two points share lattice site");
    cube[site] = q;
    if (q < np) cidx[q] = (int)site;
  }
  for (int j = 0; j < n; ++j)
    op->dcube[j] = (int)(pts[3 * j] + sz[0] * (pts[3 * j + 1] + sz[1] * (long)pts[3 * j + 2]));
  op->ncube = (size_t)nsite;
  int rc = upload(&op->d_cube, cube.data(), cube.size(), s);
  if (!rc) rc = upload(&op->d_dcube, op->dcube, (size_t)n, s);
  if (rc) return rc;
  return upload(&op->d_cidx, cidx.data(), cidx.size(), s);
}

// The z-march kernel needs the order-4 star in Octopus's point order: x -4..4, then
// y -4..-1,1..4, then z -4..-1,1..4 (src/grid/stencil_star.F90:59-93).
bool is_star4(int n, const int* pts) {
  if (n != 25) return false;
  int j = 0;
  for (int d = 0; d < 3; ++d)
    for (int k = -4; k <= 4; ++k) {
      if (k == 0 && d > 0) continue;
      for (int e = 0; e < 3; ++e)
        if (pts[3 * j + e] != (e == d ? k : 0)) return false;
      ++j;
    }
  return true;
}

// March cube: the inner points' bounding box rounded up to whole ZTX x ZTY column tiles in x
// and y, padded by the stencil reach in x/y and by ZPADZ planes in z; site -> point index.
int build_march(octhip_nl_operator_s* op, hipStream_t s) {
  const int np = op->np, np_part = op->np_part;
  const std::vector<int>& c = op->coords;
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
  for (int q = 0; q < np; ++q)
    for (int d = 0; d < 3; ++d) {
      lo[d] = std::min(lo[d], c[3 * (size_t)q + d]);
      hi[d] = std::max(hi[d], c[3 * (size_t)q + d]);
    }
  op->ntx = (hi[0] - lo[0] + ZTX) / ZTX;
  op->nty = (hi[1] - lo[1] + ZTY) / ZTY;
  op->mx = op->ntx * ZTX + 2 * ZR;
  op->my = op->nty * ZTY + 2 * ZR;
  op->mz = (hi[2] - lo[2] + 1) + 2 * ZPADZ;
  const int ox = lo[0] - ZR, oy = lo[1] - ZR, oz = lo[2] - ZPADZ;
  const size_t nsite = (size_t)op->mx * op->my * op->mz;
  if (nsite > (size_t)INT_MAX / 2) return fail(OCTHIP_ERR_UNSUPPORTED, "march cube too large");
  std::vector<int> mc(nsite, -1);
  op->tile_zlo.assign((size_t)op->ntx * op->nty, INT_MAX);
  op->tile_zhi.assign((size_t)op->ntx * op->nty, -1);
  for (int q = 0; q < np_part; ++q) {
    const int* p = &c[3 * (size_t)q];
    if (p[0] == INT_MIN) continue;
    const long x = p[0] - ox, y = p[1] - oy, z = p[2] - oz;
    if (x < 0 || y < 0 || z < 0 || x >= op->mx || y >= op->my || z >= op->mz) continue;
    mc[(size_t)x + (size_t)op->mx * ((size_t)y + (size_t)op->my * z)] = q;
    if (q < np) {
      const int t = (int)((x - ZR) / ZTX + op->ntx * ((y - ZR) / ZTY));
      op->tile_zlo[t] = std::min(op->tile_zlo[t], (int)z);
      op->tile_zhi[t] = std::max(op->tile_zhi[t], (int)z);
    }
  }
  (void)s;
  op->mcube = std::move(mc);
  return OCTHIP_SUCCESS;
}

}  // namespace

namespace octhip {
int zmarch_resident(int lc, int lpt, int epi, bool nl, bool multi);

constexpr double ZM_OVERHEAD = 6.0;  // an item's prologue and tail, in plane steps
// running workgroups per CU that saturate the chip, of 16 and of 8 lanes
constexpr double ZM_FULL16 = 0.75, ZM_FULL8 = 2.0;

// (tile, z-segment) work items {first record plane, planes} for segment length zs: the z range
// of the mesh is cut into slabs of equal thickness of at most zs planes, and an item is a
// tile's part of a slab.  Neighbouring tiles so start a slab at the same plane and stay
// within a few planes of each other, which keeps their halo rows in L2 (462,781 points, 32
// states: 520 MB read instead of 590 with segments of equal length per tile).  Slab by slab,
// then tile rows.
std::vector<int2> zmarch_items(const octhip_nl_operator_s* op, int zs) {
  int lo = INT_MAX, hi = -1;
  for (size_t t = 0; t < op->tile_zlo.size(); ++t)
    if (op->tile_zhi[t] >= 0) {
      lo = std::min(lo, op->tile_zlo[t]);
      hi = std::max(hi, op->tile_zhi[t]);
    }
  std::vector<int> first(op->tile_zlo.size(), 0);
  int plane = 0;
  for (size_t t = 0; t < op->tile_zlo.size(); ++t) {
    first[t] = plane;
    if (op->tile_zhi[t] >= 0) plane += op->tile_zhi[t] - op->tile_zlo[t] + 9;
  }
  std::vector<int2> items;
  if (hi < 0) return items;
  const long len = hi - lo + 1, nslab = (len + zs - 1) / zs;
  for (long s = 0; s < nslab; ++s) {
    const int a = lo + (int)(len * s / nslab), b = lo + (int)(len * (s + 1) / nslab);
    for (size_t t = 0; t < op->tile_zlo.size(); ++t) {
      if (op->tile_zhi[t] < 0) continue;
      const int z0 = std::max(a, op->tile_zlo[t]), z1 = std::min(b, op->tile_zhi[t] + 1);
      if (z0 < z1) items.push_back(make_int2(first[t] + z0 - op->tile_zlo[t], z1 - z0));
    }
  }
  return items;
}

// bounds of the 8 contiguous parts of equal work of a list of items, one part per XCD
std::vector<size_t> zmarch_cuts(const std::vector<int>& planes) {
  double total = 0.0;
  for (int p : planes) total += p + ZM_OVERHEAD;
  std::vector<size_t> cut(9, 0);
  double sum = 0.0;
  int k = 1;
  for (size_t i = 0; i < planes.size(); ++i) {
    const double w = planes[i] + ZM_OVERHEAD;
    while (k < 8 && sum + 0.5 * w >= total * k / 8.0) cut[k++] = i;
    sum += w;
  }
  while (k <= 8) cut[k++] = planes.size();
  return cut;
}

// Estimated time, in plane steps of a workgroup that has a CU for itself, of a launch over the
// work items of `planes` output planes each, in order, with `resident` workgroups of lc lanes
// per CU.  The items are dealt to the XCDs in contiguous parts of equal work; an XCD starts
// its next item when one ends; an item costs its planes and ZM_OVERHEAD steps (index and row
// prologue, four planes behind the last one); and all workgroups slow down together once more
// than ZM_FULL16 (ZM_FULL8) per CU run (they share LDS, the vector caches and the memory).  Fitted
// to sweeps on MI355X, 16 lanes: 0.47 us per step alone (57,777 points, 8 complex states: 8 planes
// 13.3 us, 12: 15.1, 16: 16.6, 32: 24.5), 462,781 points, 32 states: 12 planes 183 us, 16: 179,
// 24: 175, 32: 172, 48: 175; 155,331 points, 32 states: 8 planes 60 us, 16: 52, 24: 55, 48: 49;
// 64^3 points, 8 real functions: 8 planes 13.8 us, 24: 17.2.
double zmarch_makespan(const std::vector<int>& planes, int lc, int resident) {
  static int ncu = 0;
  if (ncu <= 0 && (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, current_device()) != hipSuccess ||
                   ncu <= 0))
    ncu = 256;
  const size_t slots = (size_t)std::max(ncu / 8, 1) * std::max(resident, 1);
  const double cap = ncu * (lc >= 16 ? ZM_FULL16 * 16.0 / lc : ZM_FULL8 * 8.0 / lc);
  const std::vector<size_t> cut = zmarch_cuts(planes);
  std::priority_queue<std::pair<double, int>, std::vector<std::pair<double, int>>, std::greater<>> ends;
  size_t next[8];
  for (int x = 0; x < 8; ++x)
    for (next[x] = cut[x]; next[x] < std::min(cut[x] + slots, cut[x + 1]); ++next[x])
      ends.push({planes[next[x]] + ZM_OVERHEAD, x});
  double clock = 0.0, time = 0.0;  // steps done by every running workgroup, time passed
  while (!ends.empty()) {
    const auto [end, x] = ends.top();
    time += (end - clock) * std::max(1.0, (double)ends.size() / cap);
    clock = end;
    ends.pop();
    if (next[x] < cut[x + 1]) ends.push({end + planes[next[x]++] + ZM_OVERHEAD, x});
  }
  return time;
}

// Segment lengths tried for a launch.  Longer ones save overlap planes, but neighbouring tiles
// drift apart over a long march and lose each other's halo rows (462,781 points, 32 states: 33
// planes 172 us, 49 planes 174-181; the Taylor pass 311 against 331).
extern const int ZM_SEGS[7];
const int ZM_SEGS[7] = {8, 12, 16, 20, 24, 32, 40};

// Segment length of a launch with nchunk lane chunks of lc lanes: the operator's setting, or
// the one with the smallest estimated time.
int zmarch_zseg(const octhip_nl_operator_s* op, int nchunk, int lc, int resident) {
  if (op->zseg > 0) return op->zseg;
  for (const auto& c : op->zseg_cache)
    if (c.x == nchunk && c.y == lc && c.z == resident) return c.w;
  double best_t = 1e300;
  int best = 8;
  for (int zs : ZM_SEGS) {
    const std::vector<int2> items = zmarch_items(op, zs);
    std::vector<int> planes;
    planes.reserve(items.size() * nchunk);
    for (int c = 0; c < nchunk; ++c)
      for (const int2& it : items) planes.push_back(it.y);
    const double t = zmarch_makespan(planes, lc, resident);
    if (t < best_t) {
      best_t = t;
      best = zs;
    }
  }
  op->zseg_cache.push_back(make_int4(nchunk, lc, resident, best));
  return best;
}

// lane chunk and lanes per thread of a z-march launch over rows of L doubles
void zmarch_shape(const octhip_nl_operator_s* op, int L, int* lc, int* lpt) {
  int c = op->lane_chunk > 0 ? op->lane_chunk : 16;
  int t = op->lanes_per_thread > 0 ? op->lanes_per_thread : 2;
  while (c > 1 && ZNC * c / 2 > 1024) c /= 2;  // 1024 threads per workgroup at most
  if (c > L) c = L;
  if (t > c) t = c;
  if (ZNC * c / t > 1024) t = 2;
  *lc = c;
  *lpt = t;
}

// segment length of a launch of this epilogue (with or without ket rows)
int zmarch_zseg_for(const octhip_nl_operator_s* op, int L, int epi, bool nl) {
  int lc, lpt;
  zmarch_shape(op, L, &lc, &lpt);
  return zmarch_zseg(op, L / lc, lc, zmarch_resident(lc, lpt, epi, nl, false));
}

// Index records of every tile (layout in zmarch.h), built once per operator.  The march cube has at
// most 2^30 sites and a plane of a tile 64 of them, so a plane's number fits an int; the table may
// have more than 2^31 ints (addressed by plane, 32-bit offsets within an item).
int zmarch_records(octhip_nl_operator_s* op) {
  if (op->d_rec) return OCTHIP_SUCCESS;
  size_t planes = 0;
  for (size_t t = 0; t < op->tile_zlo.size(); ++t)
    if (op->tile_zhi[t] >= 0) planes += (size_t)(op->tile_zhi[t] - op->tile_zlo[t] + 9);
  std::vector<int> rec(planes * ZPLANE);
  int* r = rec.data();
  for (size_t t = 0; t < op->tile_zlo.size(); ++t) {
    if (op->tile_zhi[t] < 0) continue;
    const long x0 = (long)(t % op->ntx) * ZTX + ZR, y0 = (long)(t / op->ntx) * ZTY + ZR;
    for (int z = op->tile_zlo[t] - 4; z <= op->tile_zhi[t] + 4; ++z)
      for (int cy = 0; cy < ZTY; ++cy) {
        const int* const row = op->mcube.data() + (size_t)op->mx * ((size_t)(y0 + cy) + (size_t)op->my * (size_t)z) + x0;
        const int* const hrow = row + (long)op->mx * (cy < 4 ? -4 : 4);
        for (int cx = 0; cx < ZTX; ++cx, r += ZREC) {
          r[0] = row[cx] + 1;
          r[1] = row[cx < 4 ? cx - 4 : cx + 4] + 1;
          r[2] = hrow[cx] + 1;
        }
      }
  }
  return upload(&op->d_rec, rec.data(), rec.size(), nullptr);
}

int zmarch_plan(octhip_nl_operator_s* op, int zs, octhip_nl_operator_s::ZPlan** out) {
  int rc = zmarch_records(op);
  if (rc) return rc;
  for (auto& pl : op->plans)
    if (pl.zseg == zs) {
      *out = &pl;
      return OCTHIP_SUCCESS;
    }
  op->plans.push_back({zs, zmarch_items(op, zs), {}});
  *out = &op->plans.back();
  return OCTHIP_SUCCESS;
}

// blockIdx -> work item of `all` in order: part k of zmarch_cuts runs on XCD k (workgroups are
// dealt to XCDs round-robin by blockIdx); entries without planes pad the shorter parts.
std::vector<int4> zmarch_deal(const std::vector<int4>& all) {
  std::vector<int> planes;
  planes.reserve(all.size());
  for (const int4& e : all) planes.push_back(e.y);
  const std::vector<size_t> cut = zmarch_cuts(planes);
  size_t per = 0;
  for (int x = 0; x < 8; ++x) per = std::max(per, cut[x + 1] - cut[x]);
  std::vector<int4> sc(per * 8, make_int4(0, 0, 0, 0));
  for (int x = 0; x < 8; ++x)
    for (size_t i = cut[x]; i < cut[x + 1]; ++i) sc[(i - cut[x]) * 8 + x] = all[i];
  return sc;
}

int zmarch_sched(octhip_nl_operator_s::ZPlan* pl, int nchunk, const int4** out, int* len) {
  for (const auto& e : pl->sched)
    if (e.nchunk == nchunk) {
      *out = e.d;
      *len = e.len;
      return OCTHIP_SUCCESS;
    }
  std::vector<int4> all;
  all.reserve(pl->items.size() * nchunk);
  for (int c = 0; c < nchunk; ++c)
    for (const int2& it : pl->items) all.push_back(make_int4(it.x, it.y, c, 0));
  const std::vector<int4> sc = zmarch_deal(all);
  int4* d = nullptr;
  int rc = upload(&d, sc.data(), sc.size(), nullptr);
  if (rc) return rc;
  pl->sched.push_back({nchunk, d, (int)sc.size()});
  *out = d;
  *len = (int)sc.size();
  return OCTHIP_SUCCESS;
}

int launch_zmarch(const ZArgs& z, int lc, int lpt, int epi, int grid, hipStream_t s);
int launch_zmarch_bra(const ZArgs& z, const BraMfmaArgs& m, int lc, int nz, hipStream_t s);

// The z-march addresses rows with 32-bit byte offsets: every row array it touches (psi
// over np_part rows, the outputs over np, the ket rows) must satisfy
// (rows + 1) * row bytes <= 2^32; larger batches take the gather kernel.
bool zmarch_fits(const octhip_nl_operator_s* op, const ApplyArgs& a) {
  const uint64_t rowb = (uint64_t)a.L * sizeof(double);
  const uint64_t lim = 1ull << 32;
  return (uint64_t)(op->np_part + 1) * rowb <= lim && (!a.kslot || (uint64_t)(a.nk + 1) * rowb <= lim);
}

// Whether the output rows of a pass are stored non-temporally: unless the next pass reads them
// (the powers of a Taylor or Krylov chain) and an array of rows is small enough for the 256 MB
// Infinity Cache to hold what a pass reads and what it writes.  Four passes of a Taylor-4 step,
// cached against non-temporal: rows of 35 MB 147 against 163 us, 59 MB 247 / 260, 80 MB
// 289 / 305, 118 MB 436 / 425, 188 MB 694 / 658, 237 MB 881 / 861.  A lone apply's rows are read
// by its own ket at most, where that adds to them (whole apply): 7 MB 20.5 / 19.8 us, 10 MB 20.9 /
// 20.3, 35 MB 42.1 / 41.6, 50 MB 48.8 / 49.0, 80 MB 63.8 / 64.7, 100 MB 82.2 / 82.4; without a ket
// 59 MB 50.3 / 49.6, 80 MB 53.3 / 50.9, 118 MB 90 / 71, 237 MB 190 / 185.
constexpr double ZM_CACHED_BYTES = 100e6;
int zmarch_nt(const octhip_nl_operator_s* op, const ApplyArgs& a) {
  return a.reuse && (double)op->np * a.L * sizeof(double) <= ZM_CACHED_BYTES ? 0 : 1;
}

// Whether a Taylor pass loads its accumulator and the earlier powers non-temporally: it is the
// last reader of the powers, and where its four row arrays exceed the 256 MB Infinity Cache they
// come from memory anyhow and only push out the halo rows.  Non-temporal against cached, whole
// steps: rows of 20 MB (79,501 points, 16 states) 140 / 136 us; 80 MB (155,331 points, 32-state
// blocks) 682 / 694, order 6 1180 / 1201; 237 MB (462,781 points, 4 x 32 states) 3242 / 3322.
constexpr double ZM_TAYLOR_CACHED_BYTES = 64e6;
int zmarch_ntl(const octhip_nl_operator_s* op, const ApplyArgs& a) {
  return (double)op->np * a.L * sizeof(double) > ZM_TAYLOR_CACHED_BYTES;
}

// Build every lazily created device structure an apply with rows of L doubles needs (both
// epilogues; nl = with ket rows), so that later applies allocate nothing (required before
// a graph capture).
int prepare_operator(octhip_nl_operator_s* op, int L, bool nl) {
  const bool zm = op->zmarch_ok && op->kernel != 1 && op->n == 25;
  if (!zm) return OCTHIP_SUCCESS;
  int lc, lpt;
  zmarch_shape(op, L, &lc, &lpt);
  for (int epi : {EPI_STORE, EPI_TAYLOR, EPI_TAYLOR_X}) {
    if (epi != EPI_STORE && lc < 2) continue;
    octhip_nl_operator_s::ZPlan* pl = nullptr;
    int rc = zmarch_plan(op, zmarch_zseg_for(op, L, epi, nl), &pl);
    if (rc) return rc;
    const int4* sched = nullptr;
    int len = 0;
    rc = zmarch_sched(pl, L / lc, &sched, &len);
    if (rc) return rc;
  }
  // a pass that takes the bra along has no ket rows
  return nl ? prepare_operator(op, L, false) : OCTHIP_SUCCESS;
}

// The z-march writes one density partial per lane chunk of a row, the gather kernel one
// per row (keep in step with launch_operator's kernel choice).
int apply_lane_chunks(const octhip_nl_operator_s* op, const ApplyArgs& a) {
  const bool zm = op->zmarch_ok && op->kernel != 1 && a.n == 25 && zmarch_fits(op, a);
  if (!zm) return 1;
  int lc, lpt;
  zmarch_shape(op, a.L, &lc, &lpt);
  return a.L / lc;
}

// Whether the pass of `a` (EPI_STORE) can take along a bra by sets whose blocks need lds bytes
// each: it goes by the z-march in a shape of k_zmarch_bra, whose windows hold its bra blocks.
bool operator_takes_bra(const octhip_nl_operator_s* op, const ApplyArgs& a, size_t lds) {
  int lc, lpt;
  zmarch_shape(op, a.L, &lc, &lpt);
  return op->zmarch_ok && op->kernel != 1 && a.n == 25 && zmarch_fits(op, a) && (lc == 16 || lc == 8) && lpt == 2 &&
         lds <= sizeof(double) * ZB_RED;
}

// Apply through the best kernel for this operator: z-march for the order-4 star on a
// lattice, the tiled gather otherwise.
int launch_operator(octhip_nl_operator_s* op, ApplyArgs& a, int epi, hipStream_t s, const BraMfmaArgs* bra = nullptr) {
  if (!a.fi || !a.zrow || (a.kslot && !a.ksum && !bra) || (epi == EPI_STORE && !a.fo))
    return fail(OCTHIP_ERR_STATE, "apply: incomplete kernel arguments");
  const bool zm = op->zmarch_ok && op->kernel != 1 && a.n == 25 && zmarch_fits(op, a);
  if (!zm) {
    const int rc = launch_apply(a, op->lattice && a.n > 0, epi, s);
    if (rc || !a.out_phase) return rc;
    return launch_phase(a.fo, a.fo, a.out_phase, a.np, a.L, true, s);
  }
  int lc, lpt;
  zmarch_shape(op, a.L, &lc, &lpt);
  const int zs = zmarch_zseg_for(op, a.L, epi, a.kslot != nullptr && !bra);
  if (lc == 32 && zs > ZM_SEG32)
    return fail(OCTHIP_ERR_INVALID, "z-march: lane chunk 32 (128 KB of LDS) takes z segments of at most %d planes, not %d",
                ZM_SEG32, zs);
  octhip_nl_operator_s::ZPlan* pl = nullptr;
  int rc = zmarch_plan(op, zs, &pl);
  if (rc) return rc;
  if (pl->items.empty() || a.np <= 0) return OCTHIP_SUCCESS;
  const int4* sched = nullptr;
  int len = 0;
  rc = zmarch_sched(pl, a.L / lc, &sched, &len);
  if (rc) return rc;
  ZArgs z;
  z.a = a;
  z.a.nt = zmarch_nt(op, a);
  z.a.ntl = zmarch_ntl(op, a);
  z.rec = op->d_rec;
  z.sched = sched;
  if (bra) return launch_zmarch_bra(z, *bra, lc, len, s);
  // The phased store takes the plan of the plain one: it adds 16 bytes per row.  A chunk of one
  // lane (tuning only) holds no (re, im) pair: its rows get the phase in a pass of their own.
  const bool phased = a.out_phase && lc >= 2;
  rc = launch_zmarch(z, lc, lpt, phased ? EPI_PHASE : epi, len, s);
  if (rc || phased || !a.out_phase) return rc;
  return launch_phase(a.fo, a.fo, a.out_phase, a.np, a.L, true, s);
}
}  // namespace octhip

extern "C" int octhip_nl_operator_create(int n, const double* w, const int* stencil_points, int nri,
                                         const int* ri, const int* rimap_inv, int np, int np_part,
                                         const int* coords, octhip_nl_operator_t* out) {
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(out != nullptr, "nl_operator_create: null output handle");
  *out = nullptr;
  OCTHIP_REQUIRE(n > 0 && n <= MAX_STENCIL, "stencil size %d outside 1..%d", n, MAX_STENCIL);
  OCTHIP_REQUIRE(w && ri && rimap_inv, "nl_operator_create: null descriptor array");
  OCTHIP_REQUIRE(np > 0 && np_part >= np && nri > 0, "bad sizes np=%d np_part=%d nri=%d", np, np_part, nri);
  // rimap from rimap_inv, with the checks nl_operator_build guarantees
  OCTHIP_REQUIRE(rimap_inv[0] == 0 && rimap_inv[nri] == np, "rimap_inv must start at 0 and end at np");
  std::vector<int> rimap(np);
  for (int l = 0; l < nri; ++l) {
    OCTHIP_REQUIRE(rimap_inv[l + 1] > rimap_inv[l], "run %d is empty", l);
    for (int p = rimap_inv[l]; p < rimap_inv[l + 1]; ++p) rimap[p] = l;
  }
  for (int l = 0; l < nri; ++l)
    for (int j = 0; j < n; ++j) {
      const long lo = (long)rimap_inv[l] + ri[(size_t)l * n + j];
      const long hi = (long)rimap_inv[l + 1] - 1 + ri[(size_t)l * n + j];
      OCTHIP_REQUIRE(lo >= 0 && hi < np_part, "ri[%d][%d] reaches outside 0..np_part-1", l, j);
    }
  auto* op = new octhip_nl_operator_s();
  op->n = n;
  op->np = np;
  op->np_part = np_part;
  op->nri = nri;
  op->w.assign(w, w + n);
  if (stencil_points) {
    for (int j = 0; j < n; ++j)
      if (!stencil_points[3 * j] && !stencil_points[3 * j + 1] && !stencil_points[3 * j + 2]) op->center = j;
  }
  hipStream_t s = nullptr;
  int rc = upload(&op->d_ri, ri, (size_t)nri * n, s);
  if (!rc) rc = upload(&op->d_rimap, rimap.data(), rimap.size(), s);
  // inner / outer runs: a run is inner when its last point plus the largest offset is
  // still an inner point (maxp <= np in the reference's 1-based terms)
  {
    std::vector<int> pri[2], pmin[2], pmax[2];
    for (int l = 0; l < nri; ++l) {
      int mx = ri[(size_t)l * n];
      for (int j = 1; j < n; ++j) mx = std::max(mx, ri[(size_t)l * n + j]);
      const int part = (long)rimap_inv[l + 1] + mx <= np ? 0 : 1;
      pri[part].insert(pri[part].end(), ri + (size_t)l * n, ri + (size_t)(l + 1) * n);
      pmin[part].push_back(rimap_inv[l]);
      pmax[part].push_back(rimap_inv[l + 1]);
    }
    for (int part = 0; part < 2 && !rc; ++part) {
      op->part_nri[part] = (int)pmin[part].size();
      if (pmin[part].empty()) continue;
      rc = upload(&op->d_part_ri[part], pri[part].data(), pri[part].size(), s);
      if (!rc) rc = upload(&op->d_part_imin[part], pmin[part].data(), pmin[part].size(), s);
      if (!rc) rc = upload(&op->d_part_imax[part], pmax[part].data(), pmax[part].size(), s);
    }
  }
  if (!rc && stencil_points) {
    bool ok = false;
    if (coords) {
      op->coords.assign(coords, coords + 3 * (size_t)np_part);
      ok = true;
      // verify the caller's coordinates against ri before trusting them
      for (int p = 0; p < np && ok; ++p) {
        const int* row = ri + (size_t)rimap[p] * n;
        for (int j = 0; j < n && ok; ++j) {
          const int q = p + row[j];
          for (int d = 0; d < 3; ++d)
            if (coords[3 * (size_t)q + d] != coords[3 * (size_t)p + d] + stencil_points[3 * j + d]) ok = false;
        }
      }
    } else {
      ok = rebuild_lattice(n, stencil_points, ri, rimap, np, np_part, op->coords);
    }
    if (ok) {
      rc = build_site_map(op, stencil_points, s);
      if (!rc) op->lattice = true;
      if (!rc && is_star4(n, stencil_points)) {
        rc = build_march(op, s);
        if (!rc) op->zmarch_ok = true;
      }
    }
  }
  if (rc) {
    octhip_nl_operator_destroy(op);
    return rc;
  }
  *out = op;
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_nl_operator_destroy(octhip_nl_operator_t op) {
  if (!op) return OCTHIP_SUCCESS;
  dfree(op->d_cidx);
  dfree(op->d_cube);
  dfree(op->d_dcube);
  dfree(op->d_rec);
  for (auto& pl : op->plans)
    for (auto& e : pl.sched) dfree(e.d);
  dfree(op->d_ri);
  dfree(op->d_rimap);
  for (int part = 0; part < 2; ++part) {
    dfree(op->d_part_ri[part]);
    dfree(op->d_part_imin[part]);
    dfree(op->d_part_imax[part]);
  }
  delete op;
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_nl_operator_set_tuning(octhip_nl_operator_t op, int key, int value) {
  OCTHIP_REQUIRE(op != nullptr, "null operator handle");
  switch (key) {
    case OCTHIP_TUNE_KERNEL:
      OCTHIP_REQUIRE(value >= 0 && value <= 2, "kernel %d outside 0..2", value);
      OCTHIP_REQUIRE(value != 2 || op->zmarch_ok, "z-march needs the order-4 star on a lattice");
      op->kernel = value;
      return OCTHIP_SUCCESS;
    case OCTHIP_TUNE_XCD_CHUNK:
      OCTHIP_REQUIRE(value >= 1 && value <= 4096, "xcd_chunk %d outside 1..4096", value);
      op->xcd_chunk = value;
      return OCTHIP_SUCCESS;
    case OCTHIP_TUNE_GATHER_TILE:
      OCTHIP_REQUIRE(value >= 1 && value <= 8, "gather tile %d outside 1..8", value);
      op->tile_iters = value;
      return OCTHIP_SUCCESS;
    case OCTHIP_TUNE_ZSEG:
      OCTHIP_REQUIRE(value >= 0 && value <= 64, "z segment %d outside 0..64 (0 = automatic)", value);
      op->zseg = value;
      return OCTHIP_SUCCESS;
    case OCTHIP_TUNE_LANE_CHUNK:
      OCTHIP_REQUIRE(value == 0 || value == 1 || value == 2 || value == 4 || value == 8 || value == 16 ||
                         value == 32,
                     "lane chunk %d not in {0,1,2,4,8,16,32}", value);
      op->lane_chunk = value;
      return OCTHIP_SUCCESS;
    case OCTHIP_TUNE_LANES_PER_THREAD:
      OCTHIP_REQUIRE(value >= 0 && value <= 2, "lanes per thread %d outside 0..2", value);
      op->lanes_per_thread = value;
      return OCTHIP_SUCCESS;
    default:
      return fail(OCTHIP_ERR_INVALID, "unknown operator tuning key %d", key);
  }
}

extern "C" int octhip_nl_operator_get_tuning(octhip_nl_operator_t op, int key, int* value) {
  OCTHIP_REQUIRE(op != nullptr && value != nullptr, "null argument");
  switch (key) {
    case OCTHIP_TUNE_KERNEL: *value = op->kernel; break;
    case OCTHIP_TUNE_XCD_CHUNK: *value = op->xcd_chunk; break;
    case OCTHIP_TUNE_GATHER_TILE: *value = op->tile_iters; break;
    case OCTHIP_TUNE_ZSEG: *value = op->zseg; break;
    case OCTHIP_TUNE_LANE_CHUNK: *value = op->lane_chunk; break;
    case OCTHIP_TUNE_LANES_PER_THREAD: *value = op->lanes_per_thread; break;
    default: return fail(OCTHIP_ERR_INVALID, "unknown operator tuning key %d", key);
  }
  return OCTHIP_SUCCESS;
}

extern "C" int octhip_nl_operator_uses_lattice(octhip_nl_operator_t op, int* flag) {
  OCTHIP_REQUIRE(op && flag, "null argument");
  *flag = op->lattice ? 1 : 0;
  return OCTHIP_SUCCESS;
}

namespace octhip {
// fill the stencil part of ApplyArgs from an operator handle
void stencil_args(const octhip_nl_operator_s* op, double factor, ApplyArgs& a) {
  a.n = op->n;
  a.np = op->np;
  a.cidx = op->d_cidx;
  a.cube = op->d_cube;
  a.dcp = op->d_dcube;
  a.ri = op->d_ri;
  a.rimap = op->d_rimap;
  for (int j = 0; j < op->n; ++j) {
    a.w[j] = op->w[j] * factor;  // wre = w * factor, src/grid/nl_operator_inc.F90:72-80
    a.dc[j] = op->dcube[j];
  }
  a.zrow = zero_row();
  a.chunk = op->xcd_chunk;
  a.tile_iters = op->tile_iters;
}
}  // namespace octhip

namespace octhip {
// the run-compressed leaf over nri runs given by their ri rows and point ranges
int launch_ri_runs(int n, const double* w, int nri, const int* ri, const int* imin, const int* imax,
                   const double* fi, int ldf, double* fo, hipStream_t s);
}  // namespace octhip

extern "C" int octhip_nl_operator_operate_batch(octhip_nl_operator_t op, const double* fi, double* fo,
                                                int ldf, double factor, int points, void* stream) {
  OCTHIP_RANGE("octhip_nl_operator_operate_batch");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(op != nullptr, "null operator handle");
  OCTHIP_REQUIRE(fi && fo, "null batch pointer");
  OCTHIP_REQUIRE(ldf >= 0 && ldf <= MAX_LDF, "ldf=%d outside 0..%d", ldf, MAX_LDF);
  OCTHIP_REQUIRE(fi != fo, "operate_batch cannot work in place");
  OCTHIP_REQUIRE(points == OCTHIP_OP_ALL || points == OCTHIP_OP_INNER || points == OCTHIP_OP_OUTER,
                 "points=%d is none of OP_INNER, OP_OUTER, OP_ALL", points);
  if (points != OCTHIP_OP_ALL) {
    // the inner or the outer runs only (nl_operator_inc.F90:257-469 with op%inner / op%outer),
    // through the run-compressed leaf: same weights, same summation order per lane
    const int part = points == OCTHIP_OP_INNER ? 0 : 1;
    std::vector<double> wf(op->n);
    for (int j = 0; j < op->n; ++j) wf[j] = op->w[j] * factor;
    return launch_ri_runs(op->n, wf.data(), op->part_nri[part], op->d_part_ri[part], op->d_part_imin[part],
                          op->d_part_imax[part], fi, ldf, fo, (hipStream_t)stream);
  }
  ApplyArgs a;
  std::memset(&a, 0, sizeof(a));
  stencil_args(op, factor, a);
  a.fi = fi;
  a.fo = fo;
  a.L = 1 << ldf;
  a.lim = op->np_part;  // boundary rows are read as the caller set them
  return launch_operator(op, a, EPI_STORE, (hipStream_t)stream);
}

// ------------------------------------------------------- stateless leaf --
namespace {
struct RiWeights {
  double w[MAX_STENCIL];
};

// tpr = min(L, 64) consecutive threads own one run and walk its points, each thread a
// lane (stride tpr) of every point; a 256-thread workgroup covers 256 / tpr runs, so
// short runs (two points on average in Octopus's blocked order) still fill the waves.
// Per lane the sum runs over j in stencil order with fused multiply-adds, as the C leaf.
__global__ __launch_bounds__(BLOCK) void k_operate_ri(int n, const RiWeights w, int nri, const int* __restrict__ ri,
                                                      const int* __restrict__ imin, const int* __restrict__ imax,
                                                      const double* __restrict__ fi, int L, int tshift,
                                                      double* __restrict__ fo) {
  const int tpr = 1 << tshift;
  const int l = (int)(blockIdx.x * (BLOCK >> tshift)) + (int)(threadIdx.x >> tshift);
  if (l >= nri) return;
  const int* row = ri + (size_t)l * n;
  const int i0 = imin[l], i1 = imax[l];
  for (int i = i0; i < i1; ++i)
    for (int k = threadIdx.x & (tpr - 1); k < L; k += tpr) {
      double a = 0.0;
      for (int j = 0; j < n; ++j) a = fma(w.w[j], fi[(size_t)(row[j] + i) * L + k], a);
      fo[(size_t)i * L + k] = a;
    }
}
}  // namespace

namespace octhip {
int launch_ri_runs(int n, const double* w, int nri, const int* ri, const int* imin, const int* imax,
                   const double* fi, int ldf, double* fo, hipStream_t s) {
  if (nri == 0) return OCTHIP_SUCCESS;
  // the weights travel as a kernel argument: nothing is allocated, nothing synchronised
  RiWeights rw;
  for (int j = 0; j < MAX_STENCIL; ++j) rw.w[j] = j < n ? w[j] : 0.0;
  const int tshift = ldf < 6 ? ldf : 6;
  const int runs_per_block = BLOCK >> tshift;
  hipLaunchKernelGGL(k_operate_ri, dim3((nri + runs_per_block - 1) / runs_per_block), dim3(BLOCK), 0, s, n, rw,
                     nri, ri, imin, imax, fi, 1 << ldf, tshift, fo);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(OCTHIP_ERR_HIP, "operate_ri_vec: %s", hipGetErrorString(e));
  return OCTHIP_SUCCESS;
}
}  // namespace octhip

extern "C" int octhip_operate_ri_vec(int n, const double* w, int nri, const int* ri, const int* rimap_inv,
                                     const int* rimap_inv_max, const double* fi, int ldf, double* fo,
                                     void* stream) {
  OCTHIP_RANGE("octhip_operate_ri_vec");
  OCTHIP_REQUIRE_INIT();
  OCTHIP_REQUIRE(n > 0 && n <= MAX_STENCIL && nri >= 0, "bad n=%d or nri=%d", n, nri);
  OCTHIP_REQUIRE(ldf >= 0 && ldf <= MAX_LDF, "ldf=%d outside 0..%d", ldf, MAX_LDF);
  if (nri == 0) return OCTHIP_SUCCESS;
  OCTHIP_REQUIRE(w && ri && rimap_inv && rimap_inv_max && fi && fo, "null argument");
  return launch_ri_runs(n, w, nri, ri, rimap_inv, rimap_inv_max, fi, ldf, fo, (hipStream_t)stream);
}
