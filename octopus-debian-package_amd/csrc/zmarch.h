// 2.5-D "z-march" apply for the order-4 star stencil on a lattice (gfx950).
//
// The gather kernel (k_apply) reads 25 full rows per point, so L2 has to deliver 25x the
// HBM traffic.  Here a workgroup owns an 8x8 tile of lattice columns and one chunk of LC
// lanes, and walks a segment of the tile's z range plane by plane:
//   * the current plane (tile + 4-site halo strips on the four sides) is staged in LDS
//     (double-buffered) as a dense 16x16 window, so that the 16 x and y neighbours of a
//     thread are one base address and compile-time offsets;
//   * z neighbours never leave the registers: a thread keeps its column's values of the 4
//     planes behind, and one partial sum for each of the 4 planes behind.  When plane z
//     arrives it starts its own sum (x and y terms, then z-4..z-1) and adds the +1..+4
//     terms to the four sums behind it; the sum of plane z-4 is then complete.  The terms of
//     every sum still arrive in stencil order, and a plane's own values and its halo are
//     needed at the same step: neighbouring tiles, which run side by side on one XCD, read
//     each other's rows while they are in its L2 (keeping z-4..z+4 resident instead loads a
//     column's own values three planes before its neighbours load them as halo);
//   * the site -> point indices (own column and two halo sites per column) are one 12-byte
//     record per column and plane, loaded a plane ahead of the rows they address;
//   * loads run ahead (depths in ZDepth) in rings with compile-time slots (the z loop is
//     unrolled by 8); every load but the ket rows is unconditional, so the compiler's wait
//     counts stay exact and a step waits only on loads of the steps before it.
// What bounds it (462,781 points, 32 complex states, H-apply with ket rows: 163 us, 518 MB
// read and 237 MB written for 289 + 237 MB of rows): 102 us go to the LDS reads (16 rows of 16
// bytes per output) and the vector memory instructions alone, with every row out of range, and
// the memory traffic overlaps with them only in part.  Measured and not kept: rows two or three
// planes ahead (+1 to +4%), a quad of 2x2 columns per thread (half the LDS reads; 8-byte loads,
// 215-237 us), 8-lane chunks (257 us), the lane chunks of an item side by side (177-200 us).
// Rows go through raw buffer resources (below).  Values follow the gather kernel exactly:
// point q < lim -> its row, anything else -> 0, and the 25 terms are summed in stencil order
// (x -4..4, y -4..-1,1..4, z -4..-1,1..4) with fma, so results are bit-identical to it.
#pragma once

#include "bra.h"

namespace octhip {

constexpr int ZTX = 8, ZTY = 8;       // tile columns along x and y
constexpr int ZR = 4;                 // stencil reach
constexpr int ZNC = ZTX * ZTY;        // own columns of a tile
constexpr int ZHU = 2;                // halo sites per column: 128 for 64 columns
constexpr int ZW = ZTX + 2 * ZR;      // window row length (x)
constexpr int ZS = ZW * (ZTY + 2 * ZR);  // site slots of the window (the 4x4 corners stay unused)
// march-cube padding below/above the inner points in z
constexpr int ZPADZ = 8;
// Index records of a tile: for every plane from 4 below to 4 above its inner points and every
// column, {own, halo 0, halo 1, 0} as point index + 1 (0: no point).  Column (cx, cy) carries the
// halo sites (cx < 4 ? cx - 4 : cx + 4, cy) and (cx, cy < 4 ? cy - 4 : cy + 4) of the tile.
constexpr int ZREC = 4;               // ints per record
constexpr int ZPLANE = ZREC * ZNC;    // ints per plane of a tile

// Prefetch depths in planes: rows (own and halo values) and output-point data (potential,
// ket row, Taylor rows).  One plane each: 85-103 VGPRs, two 512-thread workgroups per CU; deeper
// rings measured slower (rows 2: 166 against 163 us, output-point data 2: 163), also for
// launches of at most one workgroup per CU (rows 3 and output-point data 2, which no longer
// fits 128 VGPRs with ket rows: 57,777 points, 8 complex states 28.9 against 24.8 us for the
// apply; without ket rows 20.4 against 20.2; 64^3 points, 8 real functions 11.1 either way).
struct ZDepth {
  static constexpr int rows = 1, aux = 1;
};

// Raw buffer resources over the row arrays (gfx9 range checking, stride 0): a load whose
// byte offset lies at or beyond num_records returns zeros and such a store is dropped.
// Offsets are 32-bit, row q at q << log2(row bytes), so the point index -1 (and any
// index >= the array's row count) falls out of range: this replaces the zero-row pointer
// selects and keeps every load and store unconditional.  The host sends a batch here only
// when (rows + 1) * row bytes <= 2^32 for every array.
constexpr int ZM_RSRC_DW3 = 0x00020000;  // dword 3 of a raw buffer resource: 32-bit data format
__device__ __forceinline__ __amdgpu_buffer_rsrc_t zrsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, ZM_RSRC_DW3);
}
constexpr int ZM_NT = 2;  // cache-policy operand: non-temporal
template <int LPT, int POLICY = 0>
__device__ __forceinline__ Vec<LPT> bld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  Vec<LPT> v;
  if constexpr (LPT == 2) {
    const double2 t = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, POLICY));
    v.v[0] = t.x;
    v.v[1] = t.y;
  } else {
    v.v[0] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, POLICY));
  }
  return v;
}
// Stores of output rows, cached or non-temporal (cache policy NT).  Rows that the next pass
// finds in the 256 MB Infinity Cache are stored cached; beyond that, non-temporal stores leave
// the XCD's L2 to the input rows that the neighbouring tiles read as their halo (see
// zmarch_nt in nl_operator.hip for the line between them).
template <int LPT>
__device__ __forceinline__ void bst(__amdgpu_buffer_rsrc_t r, uint32_t off, const Vec<LPT>& v, bool nt) {
  if constexpr (LPT == 2) {
    using U4 = decltype(__builtin_amdgcn_raw_buffer_load_b128(r, 0, 0, 0));
    const U4 u = __builtin_bit_cast(U4, make_double2(v.v[0], v.v[1]));
    if (nt) __builtin_amdgcn_raw_buffer_store_b128(u, r, off, 0, ZM_NT);
    else __builtin_amdgcn_raw_buffer_store_b128(u, r, off, 0, 0);
  } else {
    using U2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0));
    const U2 u = __builtin_bit_cast(U2, v.v[0]);
    if (nt) __builtin_amdgcn_raw_buffer_store_b64(u, r, off, 0, ZM_NT);
    else __builtin_amdgcn_raw_buffer_store_b64(u, r, off, 0, 0);
  }
}

// What the threads of a column share (its record, its potential) is loaded as one dword per lane
// and handed round within each quad of lanes by DPP: a dword load occupies the vector memory
// unit 4 cycles instead of 12 or 8 (with the ket rows skipped where a wave has none, 81 cycles
// per plane and wave instead of 104: 462,781 points, 32 states 172 -> 163 us, 155,331 points
// 49 -> 47 us).
template <int K>
__device__ __forceinline__ uint32_t quad_bcast(uint32_t v) {  // lane K of each quad of lanes
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, K * 0x55, 0xf, 0xf, true);
}

struct ZArgs {
  ApplyArgs a;
  const int* __restrict__ rec;       // index records of every tile (ZREC ints each)
  const int4* __restrict__ sched;    // blockIdx -> {first record plane, planes, lane chunk, -}
};

// One work item: `n` output planes of a tile, whose index records start (4 planes below the
// first output plane) at plane rec0 of the table; lane chunk `chunk`.
// za may live in kernel arguments (single operator) or in global memory (one descriptor
// per system of a batched launch): every field is copied to a local once.
template <int LPT, int LC, int EPI, bool NL>
__device__ __forceinline__ void zmarch_body(const ZArgs& za, const int rec0, const int n, const int chunk) {
  constexpr int PAIRS = LC / LPT;    // threads per column
  extern __shared__ double2 zsh2[];  // 16-byte aligned: row chunks move as ds_*_b128
  double* const zsh = reinterpret_cast<double*>(zsh2);
  const ApplyArgs& A = za.a;
  const int a_np = A.np;
  const double* const a_v = A.v;
  double* const a_acc = A.acc;
  const bool a_nt = A.nt != 0, a_ntl = A.ntl != 0;
  double a_w[25];
#pragma unroll
  for (int j = 0; j < 25; ++j) a_w[j] = A.w[j];
  const int kp = threadIdx.x % PAIRS;
  const int col = threadIdx.x / PAIRS;
  const int cx = col % ZTX, cy = col / ZTX;
  const int l = chunk * LC + kp * LPT;         // first lane of this thread
  constexpr bool TAY = EPI == EPI_TAYLOR || EPI == EPI_TAYLOR_X;
  const bool has_acc = TAY && a_acc != nullptr;
  // row q of an array starts at byte q << sh; arrays without a role here get no records
  const int sh = __builtin_ctz((unsigned)A.L) + 3;
  const uint32_t np_bytes = (uint32_t)a_np << sh;
  const auto r_fi = zrsrc(A.fi, (uint32_t)A.lim << sh);
  const auto r_v = zrsrc(a_v, a_v ? (uint32_t)a_np * 8u : 0u);
  // EPI_PHASE without ket rows: rows that a ket is added to later are stored without the phase
  constexpr bool KS = NL || EPI == EPI_PHASE;
  const auto r_ks = zrsrc(A.kslot, KS && A.kslot ? (uint32_t)a_np * 4u : 0u);
  const auto r_k = zrsrc(A.ksum, NL ? (uint32_t)A.nk << sh : 0u);
  const auto r_ai = zrsrc(A.acc_in ? A.acc_in : a_acc, has_acc ? np_bytes : 0u);
  const auto r_fo = zrsrc(A.fo, TAY ? 0u : np_bytes);
  const auto r_ph = zrsrc(A.out_phase, EPI == EPI_PHASE ? (uint32_t)a_np * 16u : 0u);
  const auto r_y = zrsrc(A.yout, (TAY && A.yout) ? np_bytes : 0u);
  const auto r_acc = zrsrc(a_acc, has_acc ? np_bytes : 0u);
  const auto r_ya = zrsrc(A.ya, (has_acc && A.ya) ? np_bytes : 0u);  // earlier powers, last order
  const auto r_yb = zrsrc(A.yb, (has_acc && A.yb) ? np_bytes : 0u);
  // EPI_TAYLOR_X: second accumulator and density partials of this thread's state
  const auto r_a2 = zrsrc(A.acc2, (EPI == EPI_TAYLOR_X && has_acc && A.acc2) ? np_bytes : 0u);
  const auto r_dp = zrsrc(EPI == EPI_TAYLOR_X && A.dpart ? A.dpart + (size_t)chunk * a_np : nullptr,
                          (EPI == EPI_TAYLOR_X && has_acc && A.dpart) ? (uint32_t)a_np * 8u : 0u);
  const double wl = (EPI == EPI_TAYLOR_X && A.dw) ? A.dw[l >> 1] : 0.0;
  const auto r_rec = zrsrc(za.rec + (size_t)rec0 * ZPLANE, (uint32_t)(n + 8) * (uint32_t)(ZPLANE * 4));
  // byte offset of this thread's lanes of row q1 - 1; q1 = 0 (no point) falls out of range
  const uint32_t lrow = (uint32_t)l * 8u - (1u << sh);
  auto roff = [&](uint32_t q1) { return (q1 << sh) + lrow; };
  // byte offset of that point in an array of 2^b bytes per point
  auto poff = [&](uint32_t ro, int b) { return ((ro - lrow) >> (sh - b)) - (1u << b); };
  constexpr uint32_t NONE = ~0u - 7u;  // out of range of the arrays of 4 or 8 bytes per point
  // window slots, in doubles, from the window's corner (so that every offset is positive)
  const int corner = (cy * ZW + cx) * LC + kp * LPT;
  constexpr int own_lds = (ZR * ZW + ZR) * LC;
  const int hx_lds = ((cy + ZR) * ZW + (cx < 4 ? cx : cx + 8)) * LC + kp * LPT;
  const int hy_lds = ((cy < 4 ? cy : cy + 8) * ZW + cx + ZR) * LC + kp * LPT;

  constexpr int RD = ZDepth::rows, AD = ZDepth::aux;
  // (the ket slot of plane 0 is loaded at step 2 - AD)
  static_assert(RD >= 1 && RD <= 3 && AD >= 1 && AD <= 2 && AD <= RD, "prefetch depths");
  // rings, plane P (relative to the first output plane) in slot P mod the ring length:
  //   ov   own values, P in z-4 .. z+RD;    hv  halo values, P in z .. z+RD
  //   part partial sums, P in z-4 .. z-1;   ro  own row offsets, P in z-4 .. z+RD
  //   rec  index records, P in z+RD .. z+RD+2
  //   vr/kr/ar/ra/rb output-point data, P in z-4 .. z-4+AD;  ks  ket slots, P in z-4+AD .. z-3+AD
  struct Rec {
    uint32_t v[PAIRS >= 4 ? 1 : 3];
  };
  Vec<LPT> ov[8], hv[4][ZHU], part[4];
  uint32_t ro[8], ks[4] = {0u, 0u, 0u, 0u};
  Rec rec[4];
  double vr[4];
  uint32_t vd[4];  // QUAD: half of the potential per lane
  Vec<2> ph[EPI == EPI_PHASE ? 4 : 1];  // Bloch phase, QUAD: a quarter of it per lane in pd
  uint32_t pd[EPI == EPI_PHASE ? 4 : 1];
  Vec<LPT> kr[4], ar[TAY ? 4 : 1], ra[TAY ? 4 : 1], rb[TAY ? 4 : 1];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    vr[k] = 0.0;
    vd[k] = 0u;
#pragma unroll
    for (int i = 0; i < LPT; ++i) part[k].v[i] = kr[k].v[i] = 0.0;
  }
  // a quad's lanes share one column when it has at least 4 threads
  constexpr bool QUAD = PAIRS >= 4;
  // record of plane P (planes past the last record read 0)
  auto load_rec = [&](int P) -> Rec {
    Rec r;
    const uint32_t o = (uint32_t)((P + 4) * ZNC + col) * (ZREC * 4u);
    if constexpr (QUAD) {
      r.v[0] = __builtin_amdgcn_raw_buffer_load_b32(r_rec, o + (threadIdx.x & 3) * 4u, 0, 0);
    } else {
      const auto v = __builtin_amdgcn_raw_buffer_load_b96(r_rec, o, 0, 0);
      for (int k = 0; k < 3; ++k) r.v[k] = v[k];
    }
    return r;
  };
  auto own_row = [&](const Rec& r) {
    if constexpr (QUAD) return quad_bcast<0>(r.v[0] << sh) + lrow;
    else return roff(r.v[0]);
  };
  // halo rows, of output planes only
  auto halo_row = [&](const Rec& r, int P, int i) {
    const bool in = P >= 0 && P < n;
    if constexpr (QUAD) {
      const uint32_t o = (in ? r.v[0] : 0u) << sh;
      return (i ? quad_bcast<2>(o) : quad_bcast<1>(o)) + lrow;
    } else {
      return in ? roff(r.v[1 + i]) : lrow;
    }
  };
  {
    Rec r0[4 + RD];
#pragma unroll
    for (int P = -4; P < RD; ++P) r0[P + 4] = load_rec(P);
#pragma unroll
    for (int P = RD; P < RD + 2; ++P) rec[P & 3] = load_rec(P);
#pragma unroll
    for (int P = -4; P < RD; ++P) {
      ro[P & 7] = own_row(r0[P + 4]);
      ov[P & 7] = bld<LPT>(r_fi, ro[P & 7]);
    }
#pragma unroll
    for (int P = 0; P < RD; ++P)
#pragma unroll
      for (int i = 0; i < ZHU; ++i) hv[P & 3][i] = bld<LPT>(r_fi, halo_row(r0[P + 4], P, i));
  }
  const int zend = n + 4;
#pragma nounroll
  for (int z0 = 0; z0 < zend; z0 += 8) {
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const int z = z0 + kk;
      if (z >= zend) return;
      // row of plane z - 4, completed in this step (stores outside the item are dropped)
      const uint32_t qo = z >= 4 ? ro[(kk + 4) & 7] : lrow;
      // ---- stage plane z
      const Vec<LPT> xz = ov[kk & 7];        // own values of planes z and z - 4
      const Vec<LPT> xf = ov[(kk + 4) & 7];
      double* const win = zsh + (kk & 1) * (ZS * LC);
      stv<LPT>(win + corner + own_lds, xz);
      stv<LPT>(win + hx_lds, hv[kk & 3][0]);
      stv<LPT>(win + hy_lds, hv[kk & 3][1]);
      // ---- the +1..+4 terms of the planes behind; plane z - 4 is complete
      Vec<LPT> s = part[kk & 3];
#pragma unroll
      for (int k = 0; k < LPT; ++k) {
        s.v[k] = fma(a_w[24], xz.v[k], s.v[k]);
#pragma unroll
        for (int d = 1; d < 4; ++d)
          part[(kk - d) & 3].v[k] = fma(a_w[20 + d], xz.v[k], part[(kk - d) & 3].v[k]);
      }
      {
        if (a_v) {
          double vv = vr[kk & 3];
          if constexpr (QUAD)
            vv = __builtin_bit_cast(double, (uint64_t)quad_bcast<1>(vd[kk & 3]) << 32 | quad_bcast<0>(vd[kk & 3]));
#pragma unroll
          for (int k = 0; k < LPT; ++k) s.v[k] = fma(vv, xf.v[k], s.v[k]);
        }
        if constexpr (NL) {
#pragma unroll
          for (int k = 0; k < LPT; ++k) s.v[k] = s.v[k] + kr[kk & 3].v[k];
        }
        if constexpr (EPI == EPI_STORE) {
          bst<LPT>(r_fo, qo, s, a_nt);
        } else if constexpr (EPI == EPI_PHASE) {
          double pr = ph[kk & 3].v[0], pi = ph[kk & 3].v[1];
          if constexpr (QUAD) {
            const uint32_t d = pd[kk & 3];
            pr = __builtin_bit_cast(double, (uint64_t)quad_bcast<1>(d) << 32 | quad_bcast<0>(d));
            pi = __builtin_bit_cast(double, (uint64_t)quad_bcast<3>(d) << 32 | quad_bcast<2>(d));
          }
          pi = -pi;
          Vec<LPT> o;
          if constexpr (LPT == 2) {
            o.v[0] = zmul_lane(pr, pi, s.v[0], s.v[1], false);
            o.v[1] = zmul_lane(pr, pi, s.v[1], s.v[0], true);
          } else {
            o.v[0] = zmul_lane(pr, pi, s.v[0], __shfl_xor(s.v[0], 1), (l & 1) != 0);
          }
          if (!NL && ks[kk & 3] != 0u) o = s;
          bst<LPT>(r_fo, qo, o, a_nt);
        } else {
          bst<LPT>(r_y, qo, s, a_nt);  // dropped when there is no yout
          Vec<LPT> av = ar[kk & 3];
          const Vec<LPT> ua = ra[kk & 3], ub = rb[kk & 3];
          // the other lane of each (re, im) pair: in this thread, or the neighbouring one
          auto add = [&](Vec<LPT>& y, double zr, double zi, const Vec<LPT>& x) {
            if constexpr (LPT == 2) {
              const double re = zmul_lane(zr, zi, x.v[0], x.v[1], false);
              const double im = zmul_lane(zr, zi, x.v[1], x.v[0], true);
              y.v[0] = y.v[0] + re;
              y.v[1] = y.v[1] + im;
            } else {
              y.v[0] = y.v[0] + zmul_lane(zr, zi, x.v[0], __shfl_xor(x.v[0], 1), (l & 1) != 0);
            }
          };
          add(av, A.car, A.cai, ua);
          add(av, A.cbr, A.cbi, ub);
          if (A.has_c1) add(av, A.c1r, A.c1i, xf);
          add(av, A.c2r, A.c2i, s);
          bst<LPT>(r_acc, qo, av, a_nt);  // dropped when there is no accumulator
          if constexpr (EPI == EPI_TAYLOR_X) {
            Vec<LPT> dv = av;
            if (A.acc2) {
              // psib2: the same terms with the deltat2 factors, from the same base
              dv = ar[kk & 3];
              add(dv, A.dar, A.dai, ua);
              add(dv, A.dbr, A.dbi, ub);
              if (A.has_c1) add(dv, A.d1r, A.d1i, xf);
              add(dv, A.d2r, A.d2i, s);
            }
            bst<LPT>(r_a2, qo, dv, a_nt);
            // density: |value|^2 of this thread's lanes times its state's weight, summed
            // over the PAIRS consecutive threads of the column (one lane chunk)
            double t = dv.v[0] * dv.v[0];
            if constexpr (LPT == 2) t = t + dv.v[1] * dv.v[1];
            t = wl * t;
#pragma unroll
            for (int off = PAIRS >> 1; off > 0; off >>= 1) t += __shfl_xor(t, off);
            Vec<1> dt;
            dt.v[0] = t;
            bst<1>(r_dp, kp == 0 && z >= 4 ? poff(ro[(kk + 4) & 7], 3) : NONE, dt, false);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- loads, into the registers that the plane staged and the plane completed have left;
      // the ones consumed first in the next step first
      const uint32_t kslot = ks[(kk + AD) & 3];  // of plane z - 4 + AD, loaded two steps ago
      if constexpr (KS) {
        const int P = z - 2 + AD;
        const uint32_t qp = (P >= 0 && P < n) ? poff(ro[(kk + 6 + AD) & 7], 2) : NONE;
        ks[(kk + 2 + AD) & 3] = __builtin_amdgcn_raw_buffer_load_b32(r_ks, qp, 0, 0);
      }
      rec[(kk + RD + 2) & 3] = load_rec(z + RD + 2);
      {
        const int P = z - 4 + AD;
        const bool in = P >= 0 && P < n;
        const uint32_t qp = ro[(kk + 4 + AD) & 7];
        const uint32_t qa = in ? qp : lrow;
        constexpr int M = 3;
        const uint32_t qv = in ? poff(qp, 3) : NONE;
        if constexpr (QUAD) vd[(kk + AD) & M] = __builtin_amdgcn_raw_buffer_load_b32(r_v, qv + (in ? (threadIdx.x & 1) * 4u : 0u), 0, 0);
        else vr[(kk + AD) & M] = bld<1>(r_v, qv).v[0];
        if constexpr (EPI == EPI_PHASE) {
          const uint32_t qh = in ? poff(qp, 4) : ~0u - 15u;
          if constexpr (QUAD) pd[(kk + AD) & M] = __builtin_amdgcn_raw_buffer_load_b32(r_ph, qh + (in ? (threadIdx.x & 3) * 4u : 0u), 0, 0);
          else ph[(kk + AD) & M] = bld<2>(r_ph, qh);
        }
        if constexpr (NL) {
          // most waves have no ket row on a plane
          Vec<LPT> kv;
#pragma unroll
          for (int k = 0; k < LPT; ++k) kv.v[k] = 0.0;
          if (__builtin_amdgcn_ballot_w64(kslot != 0u) != 0ull) kv = bld<LPT>(r_k, roff(kslot));
          kr[(kk + AD) & M] = kv;
        }
        if constexpr (TAY) {
          // zeros (no memory access) without ya / yb; as many loads on either side
          if (a_ntl) {
            ar[(kk + AD) & M] = bld<LPT, ZM_NT>(r_ai, qa);
            ra[(kk + AD) & M] = bld<LPT, ZM_NT>(r_ya, qa);
            rb[(kk + AD) & M] = bld<LPT, ZM_NT>(r_yb, qa);
          } else {
            ar[(kk + AD) & M] = bld<LPT>(r_ai, qa);
            ra[(kk + AD) & M] = bld<LPT>(r_ya, qa);
            rb[(kk + AD) & M] = bld<LPT>(r_yb, qa);
          }
        }
      }
      {
        const Rec& rn = rec[(kk + RD) & 3];
        ro[(kk + RD) & 7] = own_row(rn);
        ov[(kk + RD) & 7] = bld<LPT>(r_fi, ro[(kk + RD) & 7]);
        hv[(kk + RD) & 3][0] = bld<LPT>(r_fi, halo_row(rn, z + RD, 0));
        hv[(kk + RD) & 3][1] = bld<LPT>(r_fi, halo_row(rn, z + RD, 1));
      }
      // ---- start the sum of plane z: x, y, then z-4 .. z-1
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
      Vec<LPT> t;
#pragma unroll
      for (int k = 0; k < LPT; ++k) t.v[k] = 0.0;
      if (z < n && ro[kk & 7] < np_bytes) {
#pragma unroll
        for (int j = 0; j < 17; ++j) {
          const int d = j < 9 ? j - 4 : (j < 13 ? j - 13 : j - 12);
          const Vec<LPT> x = j == 4 ? xz : ldv<LPT>(win + corner + own_lds + (j < 9 ? d : d * ZW) * LC);
#pragma unroll
          for (int k = 0; k < LPT; ++k) t.v[k] = fma(a_w[j], x.v[k], t.v[k]);
          if (j == 4 || j == 8 || j == 12) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int k = 0; k < LPT; ++k) t.v[k] = fma(a_w[17 + d], ov[(kk + 4 + d) & 7].v[k], t.v[k]);
      }
      part[kk & 3] = t;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Workgroups of up to 512 threads are held to 128 VGPRs: two of 512 threads per CU, whose
// loads cover each other's latency.
template <int LPT, int LC, int EPI, bool NL>
__global__ __launch_bounds__(ZNC * LC / LPT, 4) void k_zmarch(const ZArgs za) {
  const int4 sc = za.sched[blockIdx.x];
  if (sc.y <= 0) return;             // padding entry of the schedule (whole workgroup)
  zmarch_body<LPT, LC, EPI, NL>(za, sc.x, sc.y, sc.z);
}

// Several operators (systems) and batches in one launch: sched[b] = {first record plane,
// planes, lane chunk, descriptor}; descriptors zs[] are ZArgs in device memory (their sched is unused).
template <int LPT, int LC, int EPI, bool NL>
__global__ __launch_bounds__(ZNC * LC / LPT, 4) void k_zmarch_multi(const ZArgs* __restrict__ zs,
                                                                   const int4* __restrict__ sched) {
  const int4 sc = sched[blockIdx.x];
  if (sc.y <= 0) return;
  zmarch_body<LPT, LC, EPI, NL>(zs[sc.w], sc.x, sc.y, sc.z);
}

// dynamic LDS bytes of k_zmarch for a lane chunk: two plane windows
constexpr size_t zmarch_shmem(int lc) { return sizeof(double) * 2 * ZS * lc; }

// The stencil pass without ket rows and the bra of the same input in one launch: blocks
// 0 .. nz-1 march, the next ones hold one bra block per BLOCK threads (two at 16 lanes a chunk,
// one at 8), the rest clear boundary rows (BraMfmaArgs::zf).  The ket then adds its rows to the
// output.
constexpr size_t ZB_RED = (size_t)ZS * 16;  // LDS doubles of a bra block
// EPI: EPI_STORE, or EPI_PHASE with the rows of a later ket left without the phase; PHASE: the
// bra takes the states times the Bloch phases of (point, matrix).
template <int LPT, int LC, int EPI, bool PHASE>
__global__ __launch_bounds__(ZNC * LC / LPT, 4) void k_zmarch_bra(const ZArgs za, const BraMfmaArgs m, const int nz) {
  constexpr int NT = ZNC * LC / LPT, PER = NT / BLOCK;  // threads and bra blocks of a workgroup
  static_assert(NT % BLOCK == 0 && PER * ZB_RED * sizeof(double) == zmarch_shmem(LC), "whole bra blocks, their LDS");
  extern __shared__ double2 zsh2[];
  int b = blockIdx.x;
  if (b < nz) {
    const int4 sc = za.sched[b];
    if (sc.y <= 0) return;
    zmarch_body<LPT, LC, EPI, false>(za, sc.x, sc.y, sc.z);
    return;
  }
  b -= nz;
  const int nb = (m.nbra + PER - 1) / PER;
  if (b < nb) {
    const int half = __builtin_amdgcn_readfirstlane(threadIdx.x / BLOCK);
    const int v = PER * b + half, vb = min(v, m.nbra - 1), nlt = mfma_lane_tiles(m.b.L);
    double* const red = reinterpret_cast<double*>(zsh2) + half * ZB_RED;
    if ((m.b.L & 31) == 0) bra_set_body<2, PHASE>(m, vb / nlt, vb % nlt, red, threadIdx.x % BLOCK, v == vb);
    else bra_set_body<1, PHASE>(m, vb / nlt, vb % nlt, red, threadIdx.x % BLOCK, v == vb);
    return;
  }
  b -= nb;
  const size_t stride = (size_t)(gridDim.x - nz - nb) * NT;
  for (size_t t = b * (size_t)NT + threadIdx.x; t < m.zcount; t += stride) m.zf[m.zfirst + t] = 0.0;
}

// Longest segment of a workgroup of 32 lanes.  Its windows take 128 KB of LDS at any segment length,
// so the kernel itself would run longer ones: the limit is part of the interface, from kernels that
// staged index tables in LDS, and what callers see refused stays refused.
constexpr int ZM_SEG32 = 60;

}  // namespace octhip
