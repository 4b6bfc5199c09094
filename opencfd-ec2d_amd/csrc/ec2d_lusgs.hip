// LU-SGS implicit update: du_LU_SGS_2D (sub_LU_SGS.f90:4-108), optionally
// followed by U = U + dU (sub_NS_singlegrid.f90:203-211), for all blocks of
// one mesh level.  Three paths, chosen per level (ec2d_commit's rule, or
// ec2d_autotune):
//
//   split   k_lusgs_prep (every cell in parallel) writes, for each of the two
//           sweeps, a record of all the cell's update needs that does not
//           depend on dU; k_lusgs_sweep runs the two dependent sweeps;
//           k_lusgs_scatter puts dU into the block planes (and U = U + dU);
//   fused   k_lusgs_fused makes the records in the sweep's own workgroup and
//           writes the planes itself (blocks of at most 64 rows);
//   parts   k_lusgs_parts does the same by workgroups of 16 or 32 rows, linked
//           as the split sweeps are (few blocks, any number of rows).
//
// Sweep order.  The forward sweep needs dU(i-1,j) and dU(i,j-1), the backward
// sweep dU(i+1,j) and dU(i,j+1).  Any order that respects these dependencies
// gives the reference's result bit for bit.  Step s handles hyperplane s
// (sub_LU_SGS.f90:25-29, 70-75): row t takes its cell at column offset
// c = s - t.
//
// The sender's side of a cell.  Of the sums dui and duj of a cell, the part
// that comes from one neighbour (sub_LU_SGS.f90:42-58, 85-100) needs that
// neighbour's dU and U + dU, the face's normal and area, and the neighbour's
// spectral radii: nothing of the receiving cell's own solution.  So the lane
// that has just finished a cell forms both of the terms that its cell hands
// on (to the next cell of its row, and to the cell of the next row) and
// passes on these, NV doubles each, instead of dU and U + dU:
//  - p and 1/rho of U + dU are formed once per cell, not once per user;
//  - a neighbour's term crosses lanes in 2 NV register moves instead of 4 NV
//    (and waves and workgroups in NV doubles instead of 2 NV);
//  - F(U).n of a record is the cell's own, so a record is made from the
//    cell's planes and the metrics of its two outgoing faces;
//  - no lane selects: a cell without a neighbour adds the zero that an
//    untouched lane holds (a row's lane before its first cell computes with
//    a neutral record - U = (1, 0, 0, ...), everything else zero - whose
//    outgoing terms are zero).
// A sweep wave issues one instruction at a time, so its step takes as long
// as its instruction count (4 cycles each in FP64); with the neighbour's side
// a step of SA's one-lane form took about 290 vector instructions.
//
// Lanes.  One lane per row (LPC = 1), or two (LPC = 2): lane 2t forms the
// term for the next cell of the row, lane 2t+1 the one for the next row.  The
// terms move one lane up (DPP wave shift): lane 2t then holds its own term
// and row t-1's, forms the sum and hands it to lane 2t+1 (DPP quad permute),
// and both finish the cell with the same bits; with one lane per row, lane t
// receives row t-1's.  The first lane of a wave gets row t-1 through LDS.  Four
// (QuadSlot): each half of the wave has half of the equations.
//
// Divisions.  Every quotient of a sweep has a divisor known before its
// numerator (the diagonal) or shared by three quotients (rho of U + dU).
//   The record holds 1/alfa as yh + yl, good to 2^-104, and a/alfa is
// fma(a, yh, a*yl): one rounding of a value within 2^-104 of the quotient,
// RN(a/alfa) - the value of the reference's division - unless the quotient
// lies that close to a rounding boundary (one in 2^50 of unrelated operands);
// two operations instead of the eleven of a division.
//   rho of a cell that the flow has not reached is within a few units in the
// last place of 1, where quotients do lie next to rounding boundaries.  Its
// three quotients share rcp_n(rho) and take the steps of a division (div_y).
// (RN(1/rho) and two refinements of each quotient: 257 x 65 Euler cells 1.03x a
// pass.)
//
// Scaling.  0.5*(DF*a + Lc*dU) is formed as DF*(0.5 a) + (0.5 Lc)*dU, and
// -0.5*(DF*a - Lc*dU) as DF*(-0.5 a) + (0.5 Lc)*dU, with the factors in the
// record: scaling by a power of two commutes with rounding.
//
// Record layout ("skewed").  A block's records are stored hyperplane by
// hyperplane: the record of the cell that row t handles at step s sits at
// position s*R + t, with R the row count rounded up to whole waves of the
// sweep (the fused launch, one sweep wave: the row count itself),
// S = ncol + nrow - 1 steps and n = S*R + 64 positions per field.  Fields go
// in pairs of doubles, so that every load and store moves 16 bytes per lane:
// the vector memory address path costs the same per lane for 8 and for 16
// bytes, and with 8-byte loads it, not the arithmetic, bounds a block of four
// waves.  Every load of a step is one contiguous run per wave (buffer loads
// with one lane offset and a scalar offset per pair).  The forward record of
// (s, t) belongs to cell (c+1, t+1), the backward record to cell
// (ncol-c, nrow-t): both sweeps use the same index arithmetic.
//
// Per block the records occupy (2*NREC + 2*XP) * n doubles: the forward set,
// the backward set (whose X pairs receive the forward dU from the forward
// sweep), and XP output pairs for the backward dU.  The last 64 positions of
// every field are a trash pad that lanes without a cell to store write to,
// so the sweep's stores are unconditional (a store under a branch makes the
// compiler drain every outstanding load, the prefetch ring included, before
// the next use of a loaded register).
#include "ec2d_device.h"
#include "ec2d_physics.h"
#include <type_traits>

namespace ec2d {

struct LusgsArgs {
  const BlockDesc* blocks;
  const int* block_list;  // blocks of this launch
  const CaseParams* cps;
  double* arena;
  double* sk;             // skewed records of the level
  PlaneMap pm;
  double alfa1;
  int update;             // scatter: 1 also adds dU to U
  int split;              // sweep: workgroups per block (1, 2 or 4: a block's rows split between CUs)
  int dir;                // sweep: 0 both sweeps, 1 forward only, 2 backward only (split launches)
  unsigned long long* gring;  // sweep, split: one ring per boundary between workgroups and direction
  int64_t gstride;        // sweep, split: slots of one ring (at least npad * NV)
  unsigned* tickets;      // parts: per block of the launch, the workgroups that have started (0 between launches)
  int* err;               // sweep, split: set when a cross-workgroup wait ran out of its budget
  int spin_max;           // the budget of a bounded wait, in polls
  int nblk;               // skew: blocks of this launch
  int sk_tiles;           // skew: 16 x 16 tiles per block (the largest block's count)
};

// Field layout of one record set (one sweep direction) of a block.  A
// record has a part of the cell and a part per side (k = 0: the term for the
// next cell of the row, k = 1: the term for the next row).  Both are
// sequences of doubles stored in pairs; in doubles from the set's start:
//   cell's double d of position pos:   (d/2)*2n + 2*pos + d%2
//   side double e of (pos, k):         NSH*n + (e/2)*4n + 2*(2*pos + k) + e%2
// so that a wave's pair loads are contiguous and the two lanes of a cell
// read adjacent pairs of their sides.
template <int NV, bool VISC>
struct RecF {
  // cell: X = Res (forward) or the forward dU (backward), in whole pairs
  // of their own; then U and the reciprocal of the diagonal as yh + yl (a
  // separate one for the SA equation)
  static constexpr int XP = (NV + 1) / 2;
  static constexpr int U = 2 * XP, YH0 = U + NV, YL0 = YH0 + 1, YH4 = YH0 + 2, YL4 = YH0 + 3;
  static constexpr int NSH = 2 * XP + (NV + 2 + (NV == 5 ? 2 : 0) + 1) / 2 * 2;
  // per side: F(U).n, the normal, half the face area (negated: backward), half the
  // inviscid and the viscous spectral radius (padded to whole pairs)
  static constexpr int F = 0, N1 = NV, N2 = NV + 1, A = NV + 2, LC = NV + 3, LV = NV + 4;
  static constexpr int NSDU = NV + 4 + (VISC ? 1 : 0);  // without the padding
  static constexpr int NSD = (NSDU + 1) / 2 * 2;
  static constexpr int NREC = NSH + 2 * NSD;  // doubles per position
};

// The inputs of one record, as logical planes (the block planes they come
// from, or their skewed copies of k_lusgs_skew); U and Res take NV planes.
struct RecIn {
  static constexpr int U = 0;
  template <int NV> static constexpr int RES = NV;
  template <int NV> static constexpr int VOL = 2 * NV;
  template <int NV> static constexpr int DT = 2 * NV + 1;
  template <int NV> static constexpr int LCI = 2 * NV + 2;
  template <int NV> static constexpr int LCJ = 2 * NV + 3;
  template <int NV> static constexpr int LVI = 2 * NV + 4;
  template <int NV> static constexpr int LVJ = 2 * NV + 5;
  template <int NV> static constexpr int NI1 = 2 * NV + 6;
  template <int NV> static constexpr int NI2 = 2 * NV + 7;
  template <int NV> static constexpr int NJ1 = 2 * NV + 8;
  template <int NV> static constexpr int NJ2 = 2 * NV + 9;
  template <int NV> static constexpr int SI = 2 * NV + 10;
  template <int NV> static constexpr int SJ = 2 * NV + 11;
  template <int NV> static constexpr int COUNT = 2 * NV + 12;  // at most NREC of RecF: the skewed copy fits a record set
};

// host side: doubles per position of one record set (RecF<nv, visc>::NREC)
// and of the output pairs
inline int lusgs_rec_doubles(int nv, bool visc) {
  return 2 * ((nv + 1) / 2) + (nv + 2 + (nv == 5 ? 2 : 0) + 1) / 2 * 2 + 2 * ((nv + 4 + (visc ? 1 : 0) + 1) / 2 * 2);
}
inline int lusgs_out_doubles(int nv) { return 2 * ((nv + 1) / 2); }

// operands of one lane for one cell: the cell's part and NS sides (NS = 1:
// the lane's own side k, NS = 2: both)
template <int NV, int NS>
struct Rec {
  double X[NV], U[NV];
  double F[NS][NV], n1[NS], n2[NS], a[NS], Lc[NS], Lv[NS];
  double yh0, yl0, yh4, yl4;  // 1/alfa (SA: and of the SA equation) as yh + yl
};

// what a cell hands on: the term of the next cell of its row and that of the
// next row; with two lanes per cell each lane holds its own side's in j
template <int NV, int LPC>
struct Terms {
  double i[LPC == 1 ? NV : 1], j[NV];
};

// lane l-1 -> lane l (lane 0 receives 0: bound_ctrl)
__device__ __forceinline__ double shr1(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x138, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x138, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// lane l-1 -> lane l; lane 0 receives in
__device__ __forceinline__ double shr1_in(double in, double v) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(in), __double2loint(v), 0x138, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(in), __double2hiint(v), 0x138, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// lane 2t -> lanes 2t, 2t+1 (quad_perm [0,0,2,2])
__device__ __forceinline__ double even_lane(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xA0, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xA0, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
struct D2 {
  double x, y;
};
struct alignas(16) D2a {  // in LDS: one 16-byte read
  double x, y;
};

// one pair of doubles (16 bytes) at voff + soff
__device__ __forceinline__ D2 bload2(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(D2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

__device__ __forceinline__ void bstore2(double x, double y, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  const D2 v = {x, y};
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, voff, soff, 0);
}

// one double (the odd equation's field of the fused launch's X, 8 bytes a position)
__device__ __forceinline__ double bload1(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

__device__ __forceinline__ void bstore1(double x, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), r, voff, soff, 0);
}

// v16: byte offset 16*pos of the lane's position; the field offsets are
// scalar and fixed.  base: byte offset of the record set in the block's
// record region, n16 = 16n (bytes of one pair field); NS = 1 loads side k,
// NS = 2 both sides.
template <int NV, bool VISC, int NS>
__device__ __forceinline__ void load_rec(Rec<NV, NS>& p, __amdgpu_buffer_rsrc_t r, uint32_t base, uint32_t n16,
                                         uint32_t v16, int k) {
  using F = RecF<NV, VISC>;
  double sh[F::NSH];
#pragma unroll
  for (int j = 0; j < F::NSH / 2; j++) {
    const D2 v = bload2(r, v16, base + (uint32_t)j * n16);
    sh[2 * j] = v.x;
    sh[2 * j + 1] = v.y;
  }
#pragma unroll
  for (int m = 0; m < NV; m++) {
    p.X[m] = sh[m];
    p.U[m] = sh[F::U + m];
  }
  p.yh0 = sh[F::YH0];
  p.yl0 = sh[F::YL0];
  if constexpr (NV == 5) {
    p.yh4 = sh[F::YH4];
    p.yl4 = sh[F::YL4];
  } else {
    p.yh4 = p.yh0;
    p.yl4 = p.yl0;
  }
  const uint32_t sb = base + (uint32_t)(F::NSH / 2) * n16;  // side part, at 2*pos + k
#pragma unroll
  for (int h = 0; h < NS; h++) {
    const uint32_t vd = 2u * v16 + (uint32_t)(NS == 1 ? k : h) * 16u;
    double sd[F::NSD];
#pragma unroll
    for (int j = 0; j < F::NSD / 2; j++) {
      const D2 v = bload2(r, vd, sb + (uint32_t)j * 2u * n16);
      sd[2 * j] = v.x;
      sd[2 * j + 1] = v.y;
    }
#pragma unroll
    for (int m = 0; m < NV; m++) p.F[h][m] = sd[F::F + m];
    p.n1[h] = sd[F::N1];
    p.n2[h] = sd[F::N2];
    p.a[h] = sd[F::A];
    p.Lc[h] = sd[F::LC];
    if constexpr (VISC) p.Lv[h] = sd[F::LV];
    else p.Lv[h] = 0.0;
  }
}

// ----------------------------------------------------------------- prep
// The inputs of one record, loaded ahead of its arithmetic: the cell's own
// planes and the metrics of its two outgoing faces.  Forward: the faces to
// (i+1, j) and (i, j+1), whose normals and areas are those of the receiving
// cells (sub_LU_SGS.f90:43-56).  Backward: the receiving cells' normals
// (i-1, j), (i, j-1) with the cell's own areas (sub_LU_SGS.f90:86-99).  The
// defaults are those of the neutral record.
template <int NV>
struct RecSrc {
  double U[NV] = {1.0}, Res[NV] = {};
  double vol = 1.0, dt = 1.0;
  double Lc[2] = {}, Lv[2] = {}, n1[2] = {}, n2[2] = {}, s[2] = {};  // side 0: i, side 1: j
};

// The arithmetic of one record.  SH(d) and SD(k, e) give the destination of
// the cell's double d and of side k's double e (the global skewed records of
// k_lusgs_prep, or an LDS slot of k_lusgs_fused).
// CF: the field numbers of the cell's part.  XB: also write a backward record's
// X (q.Res; the split path's X is where the forward sweep stored it).
template <int NV, bool VISC, bool FWD, bool XB, class CF, class SHF, class SDF>
__device__ __forceinline__ void rec_body(SHF SH, SDF SD, const RecSrc<NV>& q, double g, double alfa1) {
  using F = RecF<NV, VISC>;
#pragma unroll
  for (int m = 0; m < NV; m++) {
    SH(CF::U + m) = q.U[m];
    if constexpr (FWD || XB) SH(m) = q.Res[m];
  }
  // diagonal (sub_LU_SGS.f90:31-39, 76-83)
  double alfa = q.vol / q.dt + 1.0 * (q.Lc[0] + q.Lc[1]) + q.vol * alfa1;
  if constexpr (VISC) alfa = alfa + 2.0 * (q.Lv[0] + q.Lv[1]);
  auto recip = [&](int d, double al) {  // 1/al as yh + yl
    const double y = rcp_rn(al);
    SH(d) = y;
    SH(d + 1) = __builtin_fma(-al, y, 1.0) * y;
  };
  recip(CF::YH0, alfa);
  if constexpr (NV == 5) recip(CF::YH4, alfa + q.Lv[0] + q.Lv[1]);
  const double y = rcp_n(q.U[0]);
  const double p = pressure_y(q.U, y, g);
#pragma unroll
  for (int k = 0; k < 2; k++) {
    double Fo[NV];
    flux_n<NV>(Fo, q.U, y, p, q.n1[k], q.n2[k]);
#pragma unroll
    for (int m = 0; m < NV; m++) SD(k, F::F + m) = Fo[m];
    SD(k, F::N1) = q.n1[k];
    SD(k, F::N2) = q.n2[k];
    SD(k, F::A) = (FWD ? 0.5 : -0.5) * q.s[k];
    SD(k, F::LC) = 0.5 * q.Lc[k];
    if constexpr (VISC) SD(k, F::LV) = q.Lv[k];
  }
}

// block plane slot of a logical input plane
template <int NV>
__device__ __forceinline__ int rec_in_slot(const PlaneMap& pm, int plane) {
  using I = RecIn;
  if (plane < NV) return pm.U + plane;
  if (plane < 2 * NV) return pm.Res + plane - NV;
  switch (plane - 2 * NV) {
    case 0: return pm.vol;
    case 1: return pm.dt;
    case 2: return pm.Lci;
    case 3: return pm.Lcj;
    case 4: return pm.Lvi;
    case 5: return pm.Lvj;
    case 6: return pm.ni1;
    case 7: return pm.ni2;
    case 8: return pm.nj1;
    case 9: return pm.nj2;
    case 10: return pm.si;
    default: return pm.sj;
  }
}

// The inputs of position (c, r) from the block planes: forward cell
// (c+1, r+1), backward cell (ncol-c, nrow-r).  The planes hold the metrics of
// (i+1, j) and (i, j+1) for every cell (1:nx, 1:ny), and of the ghost layer
// (unused values) before the first.
template <int NV, bool VISC, bool FWD>
__device__ __forceinline__ void load_src(RecSrc<NV>& o, const BlockDesc& B, const double* base, const PlaneMap& pm,
                                         int c, int r) {
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  const int i = FWD ? c + 1 : ncol - c;
  const int j = FWD ? r + 1 : nrow - r;
  const int d = FWD ? 1 : -1;
  const int64_t q = pidx(B, i, j), qi = pidx(B, i + d, j), qj = pidx(B, i, j + d);
  auto LD = [&](int slot, int64_t at) { return base[(int64_t)slot * B.plane + at]; };
#pragma unroll
  for (int m = 0; m < NV; m++) {
    o.U[m] = LD(pm.U + m, q);
    if constexpr (FWD) o.Res[m] = LD(pm.Res + m, q);
  }
  o.vol = LD(pm.vol, q);
  o.dt = LD(pm.dt, q);
  o.Lc[0] = LD(pm.Lci, q);
  o.Lc[1] = LD(pm.Lcj, q);
  if constexpr (VISC) {
    o.Lv[0] = LD(pm.Lvi, q);
    o.Lv[1] = LD(pm.Lvj, q);
  }
  o.n1[0] = LD(pm.ni1, qi);
  o.n2[0] = LD(pm.ni2, qi);
  o.s[0] = LD(pm.si, FWD ? qi : q);
  o.n1[1] = LD(pm.nj1, qj);
  o.n2[1] = LD(pm.nj2, qj);
  o.s[1] = LD(pm.sj, FWD ? qj : q);
}

// The same inputs from the skewed copy (k_lusgs_skew: logical plane k of the
// block at sk + k n, a cell at its forward position (i-1 + j-1) R + j-1).
// Backward position (c, r) is the cell whose forward position is
// (ncol-1-c + nrow-1-r) R + nrow-1-r; the cells (i+1, j), (i, j+1) sit R and
// R + 1 further, (i-1, j), (i, j-1) R and R + 1 before.  Lanes of consecutive
// rows read consecutive positions.  A position without a cell keeps the
// neutral record, a face without a receiving cell zero metrics.
template <int NV, bool VISC, bool FWD>
__device__ __forceinline__ void load_src_sk(RecSrc<NV>& o, const BlockDesc& B, const double* __restrict__ sk, int c,
                                            int r) {
  using I = RecIn;
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  o = RecSrc<NV>();
  if (r >= nrow || c < 0 || c >= ncol) return;
  const int64_t R = B.sk_R, n = B.sk_n;
  const int cf = FWD ? c : ncol - 1 - c, rf = FWD ? r : nrow - 1 - r;
  const int64_t p = (int64_t)(cf + rf) * R + rf;
  auto LD = [&](int plane, int64_t at) { return sk[(int64_t)plane * n + at]; };
#pragma unroll
  for (int m = 0; m < NV; m++) {
    o.U[m] = LD(I::U + m, p);
    if constexpr (FWD) o.Res[m] = LD(I::RES<NV> + m, p);
  }
  o.vol = LD(I::VOL<NV>, p);
  o.dt = LD(I::DT<NV>, p);
  o.Lc[0] = LD(I::LCI<NV>, p);
  o.Lc[1] = LD(I::LCJ<NV>, p);
  if constexpr (VISC) {
    o.Lv[0] = LD(I::LVI<NV>, p);
    o.Lv[1] = LD(I::LVJ<NV>, p);
  }
  if (c + 1 < ncol) {
    const int64_t q = FWD ? p + R : p - R;
    o.n1[0] = LD(I::NI1<NV>, q);
    o.n2[0] = LD(I::NI2<NV>, q);
    o.s[0] = LD(I::SI<NV>, FWD ? q : p);
  }
  if (r + 1 < nrow) {
    const int64_t q = FWD ? p + R + 1 : p - R - 1;
    o.n1[1] = LD(I::NJ1<NV>, q);
    o.n2[1] = LD(I::NJ2<NV>, q);
    o.s[1] = LD(I::SJ<NV>, FWD ? q : p);
  }
}

template <int NV, bool VISC, bool FWD>
__device__ __forceinline__ void write_rec(double* __restrict__ rb, int64_t n, int64_t pos, const BlockDesc& B,
                                          const double* base, const PlaneMap& pm, int c, int r, double g,
                                          double alfa1) {
  using F = RecF<NV, VISC>;
  // the cell's double d, side double e of side k (layout of RecF)
  auto SH = [&](int d) -> double& { return rb[(int64_t)(d / 2) * 2 * n + 2 * pos + (d & 1)]; };
  auto SD = [&](int k, int e) -> double& {
    return rb[(int64_t)F::NSH * n + (int64_t)(e / 2) * 4 * n + 2 * (2 * pos + k) + (e & 1)];
  };
  RecSrc<NV> q;
  load_src<NV, VISC, FWD>(q, B, base, pm, c, r);
  rec_body<NV, VISC, FWD, false, F>(SH, SD, q, g, alfa1);
}

// One thread per cell, a wave per 8 x 8 tile of cells (a workgroup per 32
// columns x 8 rows): a load of the block planes touches 8 cache lines per
// wave and a record store about 15 (one per hyperplane through the tile);
// one thread per record position would make the loads walk a diagonal, one
// cache line per lane.
template <int NV, bool VISC>
__global__ __launch_bounds__(256) void k_lusgs_prep(LusgsArgs a) {
  using F = RecF<NV, VISC>;
  const BlockDesc B = a.blocks[a.block_list[blockIdx.y]];
  if (case_frozen(B.case_id)) return;
  const int64_t n = B.sk_n;
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  // tiles of the skewed (step, row) space: a workgroup covers 32 steps x 8
  // rows, a wave 8 x 8, eight lanes one step; its cells (i-1, j-1) =
  // (s - r, r) read 8 consecutive cells of 8 rows, and every record store of
  // the eight lanes of a step fills 8 consecutive positions of both sets
  const int S = B.sk_S;
  const int tiles_s = (S + 31) / 32;
  const int tile = blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int s = (tile % tiles_s) * 32 + wave * 8 + (lane >> 3);  // step
  const int r = (tile / tiles_s) * 8 + (lane & 7);               // j - 1
  const int c = s - r;                                           // i - 1
  const double g = a.cps[B.case_id].gamma;
  const double* base = a.arena + B.base;
  double* fw = a.sk + B.sk_base;
  const int64_t R = B.sk_R;
  if (s < S && r < nrow && c < 0) {
    // a row's lane before its first cell: the neutral record of both sets
    // (the rest of the position keeps the zeros the record arena starts with)
    const int64_t at = (int64_t)(F::U / 2) * 2 * n + 2 * ((int64_t)s * R + r) + (F::U & 1);
    fw[at] = 1.0;
    fw[F::NREC * n + at] = 1.0;
  }
  if (s >= S || r >= nrow || c < 0 || c >= ncol) return;  // other padding positions stay unwritten
  // the cell's forward record at (c, r), its backward record at (ncol-1-c, nrow-1-r)
  const int cb = ncol - 1 - c, rb = nrow - 1 - r;
  write_rec<NV, VISC, true>(fw, n, (int64_t)(c + r) * R + r, B, base, a.pm, c, r, g, a.alfa1);
  write_rec<NV, VISC, false>(fw + F::NREC * n, n, (int64_t)(cb + rb) * R + rb, B, base, a.pm, cb, rb, g, a.alfa1);
}

// The inputs of the fused launch's records in skewed order: logical plane k
// (RecIn) of cell (i, j) goes to sk + k n + (i-1 + j-1) R + j-1 (the
// forward record region, which the fused launch leaves free).  STATIC: the
// mesh planes (vol, normals, face areas), copied once per layout; else the
// planes a residual and an update change (in a main-loop pass the residual
// before the update writes those itself, ResArgs::sk_out, and this copy is
// left out).  A workgroup moves a tile of 16
// steps x 16 rows through LDS: 16 lanes read 16 consecutive cells of a row,
// and 16 lanes write 16 consecutive positions of a step (128 bytes each).
// A row's 16 cells start at column s0 - r, so they straddle two cache lines
// whose other halves the neighbouring tiles of the row read: the grid is
// one-dimensional and XCD-aware (workgroup w runs on XCD w % 8, and XCD x
// takes the contiguous run [x chunk, (x + 1) chunk) of the (block, tile)
// items), so that neighbouring tiles fetch their shared lines into one L2.
template <int NV, bool VISC>
__host__ __device__ constexpr bool skew_plane(int k, bool stat) {
  using I = RecIn;
  const bool is_static = k == I::VOL<NV> || k >= I::NI1<NV>;
  if (!VISC && (k == I::LVI<NV> || k == I::LVJ<NV>)) return false;
  return is_static == stat;
}

template <int NV, bool VISC, bool STATIC>
__global__ __launch_bounds__(256) void k_lusgs_skew(LusgsArgs a) {
  constexpr int NK = RecIn::COUNT<NV>;
  // the planes this launch copies, in order
  constexpr int NC = [] {
    int n = 0;
    for (int k = 0; k < NK; k++) n += skew_plane<NV, VISC>(k, STATIC) ? 1 : 0;
    return n;
  }();
  __shared__ double tile[NC][16][17];  // [plane][row][step], padded against bank conflicts
  const int chunk = (int)gridDim.x / 8;  // the grid is 8 chunk workgroups
  const int w = ((int)blockIdx.x % 8) * chunk + (int)blockIdx.x / 8;
  const int bi = w / a.sk_tiles, ti = w % a.sk_tiles;
  if (bi >= a.nblk) return;
  const BlockDesc B = a.blocks[a.block_list[bi]];
  if (case_frozen(B.case_id)) return;
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  const int S = B.sk_S;
  const int tiles_s = (S + 15) / 16;
  if (ti >= tiles_s * ((nrow + 15) / 16)) return;  // the launch fits the level's largest block
  const int s0 = (ti % tiles_s) * 16, r0 = (ti / tiles_s) * 16;
  const int tid = threadIdx.x;
  const double* __restrict__ base = a.arena + B.base;
  // load: 16 lanes of a row read 16 consecutive cells (step s, cell c = s - r)
  {
    const int rr = tid >> 4, ss = tid & 15, r = r0 + rr, s = s0 + ss, c = s - r;
    if (s < S && r < nrow && c >= 0 && c < ncol) {
      const int64_t q = pidx(B, c + 1, r + 1);
      int j = 0;
#pragma unroll
      for (int k = 0; k < NK; k++)
        if (skew_plane<NV, VISC>(k, STATIC)) tile[j++][rr][ss] = base[(int64_t)rec_in_slot<NV>(a.pm, k) * B.plane + q];
    }
  }
  __syncthreads();
  // store: 16 lanes of a step write 16 consecutive positions s R + r
  {
    const int ss = tid >> 4, rr = tid & 15, r = r0 + rr, s = s0 + ss, c = s - r;
    if (s < S && r < nrow && c >= 0 && c < ncol) {
      double* __restrict__ sk = a.sk + B.sk_base + (int64_t)s * B.sk_R + r;
      int j = 0;
#pragma unroll
      for (int k = 0; k < NK; k++)
        if (skew_plane<NV, VISC>(k, STATIC)) sk[(int64_t)k * B.sk_n] = tile[j++][rr][ss];
    }
  }
}

// The reverse of k_lusgs_skew<..., false> for the planes a residual writes
// (Res, dt, Lci, Lcj and, viscous, Lvi, Lvj; not U, whose planes the update
// keeps): after a main-loop pass whose residual wrote them to the hyperplane
// copy alone (ResArgs::sk_only), this puts them back into their planes.  The
// same tiles, the two phases swapped: 16 lanes of a step read 16 consecutive
// positions, 16 lanes of a row write 16 consecutive cells.  Every block is
// copied, frozen cases included (their copy holds their last residual).
template <int NV, bool VISC>
__host__ __device__ constexpr bool unskew_plane(int k) {
  return skew_plane<NV, VISC>(k, false) && (k < RecIn::U || k >= RecIn::U + NV);
}

template <int NV, bool VISC>
__global__ __launch_bounds__(256) void k_lusgs_unskew(LusgsArgs a) {
  constexpr int NK = RecIn::COUNT<NV>;
  constexpr int NC = [] {
    int n = 0;
    for (int k = 0; k < NK; k++) n += unskew_plane<NV, VISC>(k) ? 1 : 0;
    return n;
  }();
  __shared__ double tile[NC][16][17];
  const int chunk = (int)gridDim.x / 8;
  const int w = ((int)blockIdx.x % 8) * chunk + (int)blockIdx.x / 8;
  const int bi = w / a.sk_tiles, ti = w % a.sk_tiles;
  if (bi >= a.nblk) return;
  const BlockDesc B = a.blocks[a.block_list[bi]];
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  const int S = B.sk_S;
  const int tiles_s = (S + 15) / 16;
  if (ti >= tiles_s * ((nrow + 15) / 16)) return;
  const int s0 = (ti % tiles_s) * 16, r0 = (ti / tiles_s) * 16;
  const int tid = threadIdx.x;
  {
    const int ss = tid >> 4, rr = tid & 15, r = r0 + rr, s = s0 + ss, c = s - r;
    if (s < S && r < nrow && c >= 0 && c < ncol) {
      const double* __restrict__ sk = a.sk + B.sk_base + (int64_t)s * B.sk_R + r;
      int j = 0;
#pragma unroll
      for (int k = 0; k < NK; k++)
        if (unskew_plane<NV, VISC>(k)) tile[j++][rr][ss] = sk[(int64_t)k * B.sk_n];
    }
  }
  __syncthreads();
  {
    const int rr = tid >> 4, ss = tid & 15, r = r0 + rr, s = s0 + ss, c = s - r;
    if (s < S && r < nrow && c >= 0 && c < ncol) {
      double* __restrict__ base = a.arena + B.base;
      const int64_t q = pidx(B, c + 1, r + 1);
      int j = 0;
#pragma unroll
      for (int k = 0; k < NK; k++)
        if (unskew_plane<NV, VISC>(k)) base[(int64_t)rec_in_slot<NV>(a.pm, k) * B.plane + q] = tile[j++][rr][ss];
    }
  }
}

// ----------------------------------------------------------------- sweeps
// The term that a finished cell (dU, W = U + dU, the reciprocal of its density
// and its pressure) hands on through side h of its record: dui or duj of
// sub_LU_SGS.f90:42-58 (forward) or :85-100 (backward) for the receiving cell.
template <int NV, bool VISC, int NS>
__device__ __forceinline__ void side_term(double* v, const Rec<NV, NS>& p, int h, const double* W, const double* du,
                                          double y, double pr) {
  double DF[NV];
  dfn<NV>(DF, W, p.F[h], y, pr, p.n1[h], p.n2[h]);
#pragma unroll
  for (int m = 0; m < NV; m++) {
    v[m] = DF[m] * p.a[h] + p.Lc[h] * du[m];
    if constexpr (VISC) v[m] = v[m] + p.Lv[h] * du[m];
  }
}

// The waves of a block as a pipeline.  Wave w needs, at step s, the terms
// of the last row of wave w-1 at step s-1 and nothing else from other waves,
// so waves do not meet at a barrier per step: wave w-1 puts its last row's
// terms of step s into slot s % RING of an LDS ring and then publishes
// prog = s + 1; wave w reads slot (s-1) % RING.  Its step 0 has no input below it: it
// reads slot RING-1 of the cleared ring, so cons counts that read too and step
// RING-1 is not written before it.  A sweep wave runs turns of
// D steps and looks at the other waves' counters
// once a turn: before a turn that starts at s0 it waits for prog >= s0+D-1
// (its inputs) and for cons >= s0+D+1-RING (the slots it will write), and
// after the turn it publishes cons = s0+D (the inputs of these steps
// taken).  Checked at every step, the counters, the branches around them and
// the selects of the first lane cost each linked wave about 50 instructions a
// step, a quarter of the step.
//   Neither wait can block forever: a wave at s0 has published s0, the wave
// below stops at a turn of at most s0+D-2 when that turn needs more than
// s0, that is when 2D > RING+1; D <= 4 and RING = 16.  The communication
// waves move at most RING/2 steps at a time, under the same rules.  Wave 0
// without an input below it reads a ring of zeros whose prog is at its end,
// the last wave without a consumer writes a ring whose cons is, so that no
// step branches on its place in the block.  Every wave runs the same fixed
// number of steps, so all waits end.
// LDS operations of one wave execute in issue order, so a published counter
// is never seen before the ring data written ahead of it, and a slot is never
// rewritten before the read that cons acknowledges; compiler fences keep
// that order in the instruction stream.  The spins read LDS only and never
// wait for the global-load prefetch.
//
// ring[w] is the input of wave w: its producer is wave w-1 (or, in the upper
// workgroup of a split block, the communication wave), prog[w] that
// producer's progress and cons[w] wave w's consumption.
constexpr int RING = 16;
constexpr int CHAIN_END = 0x7fffffff;
template <int NV, int NW>  // NW: rings (waves and one more)
struct Chain {
  double dump[RING][NV];      // where the lanes below a wave's last one write
  double ring[NW][RING][NV];  // input of wave w: the terms of the row below it
  int prog[NW];               // steps finished by the producer of ring[w]
  int cons[NW];               // inputs that wave w has read, from that of step 0 on
};

__device__ __forceinline__ int lds_get(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_put(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void wait_at_least(const int* p, int v) {
  while (lds_get(p) < v) __builtin_amdgcn_s_sleep(1);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// one cell's result
template <int NV>
struct Out {
  double du[NV], W[NV];
};

// One cell of a sweep from its record p, the terms tm of its row's last cell
// and those of the row below (jin; LPC = 2: lane 2t holds them): its dU and
// U + dU, and in tm the terms it hands on.  LPC = 2: lanes 2t (the term for
// the next cell of the row) and 2t+1 (the term for the next row) share the
// cell; LPC = 1: lane t forms both.
//   Every lane keeps its terms, active or not: an inactive lane's never
// reach an active cell.  Before its first cell a row holds the neutral
// record's zeros; row t+1 at step s+1 sits at the same column offset as
// row t at step s, so it is inactive whenever row t was.
template <int NV, bool VISC, bool FWD, int LPC>
__device__ __forceinline__ void cell_step(const Rec<NV, 3 - LPC>& p, Terms<NV, LPC>& tm, const double* jin, Out<NV>& o,
                                          double g) {
  // (Res + dui) + duj forward, X + (dui + duj) / alfa backward
#pragma unroll
  for (int m = 0; m < NV; m++) {
    const double iin = LPC == 1 ? tm.i[LPC == 1 ? m : 0] : tm.j[m];
    double sum = FWD ? (p.X[m] + iin) + jin[m] : iin + jin[m];
    if constexpr (LPC == 2) sum = even_lane(sum);
    const bool sa = NV == 5 && m == 4;
    const double q = div_hl(sum, sa ? p.yh4 : p.yh0, sa ? p.yl4 : p.yl0);
    o.du[m] = FWD ? q : p.X[m] + q;
    o.W[m] = p.U[m] + o.du[m];
  }
  const double y = rcp_n(o.W[0]);
  const double pr = pressure_y(o.W, y, g);
  if constexpr (LPC == 1) {
    side_term<NV, VISC>(tm.i, p, 0, o.W, o.du, y, pr);
    side_term<NV, VISC>(tm.j, p, 1, o.W, o.du, y, pr);
  } else {
    side_term<NV, VISC>(tm.j, p, 0, o.W, o.du, y, pr);
  }
}

// Scheduling of the block so far: N times one instruction of the kind MASK
// (0x20: memory loads, 0x100: LDS reads), then V vector instructions.  A wave
// that issues a step's loads in one burst waits for the address unit (16
// cycles a load) or the LDS (8) to take them.
template <int MASK, int N, int V>
__device__ __forceinline__ void interleave() {
#pragma unroll
  for (int k = 0; k < N; k++) {
    __builtin_amdgcn_sched_group_barrier(MASK, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x2, V, 0);
  }
}

// One sweep (lanes: the head of this file).
// The records come through a ring of D register sets: step s works on set
// s % D while the loads of step s + D - 1 go into the set that step s - 1 has
// finished with, spread over the step's arithmetic (interleave).  Loads past
// the last step are clamped to it.  The cell's dU
// goes to dst: for the forward sweep the X field of the
// backward record of the same cell, for the backward sweep the output fields.
// LINK: the wave has others to exchange with (not a block of one wave).
template <int NV, bool VISC, bool FWD, int D, int LPC, bool LINK>
__device__ __forceinline__ void sweep(__amdgpu_buffer_rsrc_t rs, uint32_t rec, uint32_t dst, uint32_t n16, int S, int R,
                                      int ncol, int nrow, int t, int k, int lane, int wave, double g, Chain<NV, 17>& ch) {
  using F = RecF<NV, VISC>;
  static_assert(2 * D <= RING + 1 && RING % D == 0, "the turns of linked waves must fit the ring");
  const int npad = (S + D - 1) / D * D;
  // lanes past the block's last row load that row's records: the same cache
  // lines as its own lane, so padding rows cost no memory traffic (their
  // results never reach a cell)
  const int tl = min(t, nrow - 1);
  constexpr int NS = 3 - LPC;
  Terms<NV, LPC> tm = {};
  Rec<NV, NS> set[D];
  auto load_step = [&](Rec<NV, NS>& r, int s) {
    load_rec<NV, VISC, NS>(r, rs, rec, n16, (uint32_t)(min(s, S - 1) * R + tl) * 16u, k);
  };
  // One lane of an active cell stores; every other lane writes its own slot
  // of the trash pad (positions S*R .. S*R+63).  A lane that never stores has
  // a row number that no step reaches.
  const int ts = t < nrow && k == 0 ? t : 0x40000000;
  const uint32_t trash = (uint32_t)(S * R + lane) * 16u;
  const uint32_t dw = FWD ? (uint32_t)(-R * 16) : (uint32_t)(R * 16);
  uint32_t w16 = (uint32_t)(FWD ? (S - 1) * R + (nrow - 1 - t) : t) * 16u;
  // The input of the next step: an LDS broadcast, lane 0 uses it.  The last
  // lane's terms go to the next wave's ring, the other lanes' to the dump (a
  // store without a branch).
  double in[NV];
  const double(*rin)[NV] = ch.ring[wave];
  double(*rout)[NV] = lane == 63 ? ch.ring[wave + 1] : ch.dump;
  int prog = 0, cons = 0;
  auto look = [&] {
    prog = lds_get(&ch.prog[wave]);
    cons = lds_get(&ch.cons[wave + 1]);
  };
  auto read_in = [&](int slot) {
#pragma unroll
    for (int m = 0; m < NV; m++) in[m] = rin[slot][m];
  };
#pragma unroll
  for (int u = 0; u < D - 1; u++) load_step(set[u], u);
  if constexpr (LINK) look();
  for (int s0 = 0; s0 < npad; s0 += D) {
    const int slot0 = s0 & (RING - 1);
    if constexpr (LINK) {
      if (prog < s0 + D - 1) wait_at_least(&ch.prog[wave], s0 + D - 1);
      if (cons < s0 + D + 1 - RING) wait_at_least(&ch.cons[wave + 1], s0 + D + 1 - RING);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      read_in((s0 - 1) & (RING - 1));
    }
#pragma unroll
    for (int u = 0; u < D; u++) {
      const int s = s0 + u;
      load_step(set[(u + D - 1) % D], s + D - 1);
      double jin[NV];
#pragma unroll
      for (int m = 0; m < NV; m++) jin[m] = LINK ? shr1_in(in[m], tm.j[m]) : shr1(tm.j[m]);
      if (LINK && u + 1 < D) read_in(slot0 + u);  // the turn's next step's (its first one's follows the wait)
      Out<NV> o;
      cell_step<NV, VISC, FWD, LPC>(set[u], tm, jin, o, g);
      const uint32_t w = (uint32_t)(s - ts) < (uint32_t)ncol ? w16 : trash;
      w16 += dw;
#pragma unroll
      for (int j = 0; j < (NV + 1) / 2; j++)
        bstore2(o.du[2 * j], 2 * j + 1 < NV ? o.du[2 * j + 1] : 0.0, rs, w, dst + (uint32_t)j * n16);
      if constexpr (LINK) {
#pragma unroll
        for (int m = 0; m < NV; m++) rout[slot0 + u][m] = tm.j[m];
      }
      interleave<0x20, (F::NSH + NS * F::NSD) / 2, LPC == 2 ? 8 : 10>();
      if constexpr (LINK) {
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        lds_put(&ch.prog[wave + 1], s + 1);
        // the counters of the next turn, read early (a stale value only makes
        // it look again)
        if (u == D - 2) look();
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LINK) lds_put(&ch.cons[wave], s0 + D);
  }
}

// ---- a block's rows split between workgroups (one CU each) --------------
// The last compute wave of a workgroup feeds an extra communication wave
// through the LDS ring as if it were the next wave; that wave forwards each
// step's row through global memory to a communication wave of the next
// workgroup, which feeds its first compute wave through the LDS ring.
// Compute waves never poll global memory (a wait on a global load would also
// wait for their record prefetch).  Every step of a sweep has its own global
// slot (steps 0 .. npad-2; the next workgroup never needs the last one), so
// the forwarder only stores: no flow control, no round trip.  A slot double
// holds the sentinel until the forwarder writes the value; the receiver
// polls each double until it differs from the sentinel (every double is its
// own 8-byte handshake, so no ordering between doubles is needed) and, when
// its sweep is done, sets all its slots back to the sentinel for the next
// launch.  The sentinel is a NaN payload that arithmetic never produces (it
// yields the default NaN).  Global waits are bounded: past a.spin_max polls
// the wave sets err and stops waiting for the rest of the sweep, so the
// kernel always ends within one budget (its results are then wrong, and the
// host reports err).  A budget of 0 makes every receiver give up at its
// first slot (the host's way to test the error path).
constexpr unsigned long long GSENT = 0x7FF4DEADBEEF0001ull;
constexpr int SPIN_MAX = 1 << 20;  // the default budget

__device__ __forceinline__ unsigned long long gload(unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void gstore(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sets the global rings to the sentinel once, when the layout is made
__global__ void k_fill_u64(unsigned long long* p, int64_t n, unsigned long long v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// The communication waves have a lane for every double of CK steps (64 / NV, at
// most half the LDS ring).  They move what has arrived, up to CK steps a round trip:
// a row's terms reach the next part a step and a trip later.  (Whole batches of CK:
// 7 links of 513 x 129 SA cells 0.64 -> 0.66 ms a pass, 3 of 257 x 65 Euler 221 -> 226
// us.)
template <int NV>
struct CommLane {
  static constexpr int CK = 64 / NV < RING / 2 ? 64 / NV : RING / 2;
  int kk, f;
  bool on;  // this lane carries double f of step kk of the batch
  __device__ CommLane() : kk((int)(threadIdx.x & 63) / NV), f((int)(threadIdx.x & 63) % NV), on(kk < CK) {}
};

// sending side: take ring[nw] (the last compute wave's row) and store it
template <int NV, int NW>
__device__ void comm_forward(Chain<NV, NW>& ch, int nw, unsigned long long* gr, int npad) {
  const CommLane<NV> c;
  for (int s0 = 0; s0 < npad - 1;) {
    int done;
    while ((done = lds_get(&ch.prog[nw])) <= s0) __builtin_amdgcn_s_sleep(1);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    const int nst = min(min(done, npad - 1) - s0, c.CK);
    const bool on = c.on && c.kk < nst;
    const double v = on ? ch.ring[nw][(s0 + c.kk) & (RING - 1)][c.f] : 0.0;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    lds_put(&ch.cons[nw], s0 + nst + 1);
    if (on) gstore(gr + (s0 + c.kk) * NV + c.f, __builtin_bit_cast(unsigned long long, v));
    s0 += nst;
  }
}

// receiving side: poll the next CK steps at once, feed those that have arrived to
// ring[0]; then reset
template <int NV, int NW>
__device__ void comm_receive(Chain<NV, NW>& ch, unsigned long long* gr, int npad, int* err, int spin_max) {
  const CommLane<NV> c;
  static_assert(CommLane<NV>::CK <= RING, "a batch must fit the LDS ring");
  bool gone = false;  // the other workgroup stopped answering: wait no more
  int tries = 0;
  for (int s0 = 0; s0 < npad - 1;) {
    const int rest = min(c.CK, npad - 1 - s0);
    const bool in = c.on && c.kk < rest;
    unsigned long long x = 0;
    if (in && !gone) x = gload(gr + (s0 + c.kk) * NV + c.f);
    const unsigned long long missing = __ballot(x == GSENT);
    const int nst = missing ? min(rest, (int)__builtin_ctzll(missing) / NV) : rest;
    if (!gone && (nst == 0 ? ++tries >= spin_max : spin_max == 0)) {
      if (c.kk == 0 && c.f == 0) atomicOr(err, 1);
      gone = true;
      continue;
    }
    if (nst == 0) {
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    tries = 0;
    // the slots of steps s0 .. s0+nst-1 are free once wave 0 read step s0+nst-1-RING
    wait_at_least(&ch.cons[0], s0 + nst + 1 - RING);
    if (in && c.kk < nst) ch.ring[0][(s0 + c.kk) & (RING - 1)][c.f] = __builtin_bit_cast(double, x);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    lds_put(&ch.prog[0], s0 + nst);
    s0 += nst;
  }
  // every value of this launch has been read: back to the sentinel
  for (int i = (int)(threadIdx.x & 63); i < (npad - 1) * NV; i += 64) gstore(gr + i, GSENT);
}

// LPC lanes per cell (1 or 2), D register sets of records, MAXT threads at most.
// a.split workgroups per block (blockIdx.x = block * split + part); with a
// split each part has its compute waves, then a receiving communication wave
// (all parts but the first), then a sending one (all parts but the last), and
// the two sweeps are separate launches (a.dir), since the backward sweep of
// one part needs forward results of the others.
template <int NV, bool VISC, int D, int MAXT, int LPC>
__global__ __launch_bounds__(MAXT) void k_lusgs_sweep(LusgsArgs a) {
  using F = RecF<NV, VISC>;
  constexpr bool LINK = MAXT > 64;
  __shared__ Chain<NV, 17> ch[2];  // one per sweep
  const int G = a.split, bi = blockIdx.x / G, half = blockIdx.x % G;  // half: the part of the block
  const BlockDesc B = a.blocks[a.block_list[bi]];
  if (case_frozen(B.case_id)) return;  // every part of the block returns: no part waits on another
  const double g = a.cps[B.case_id].gamma;
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  const int S = B.sk_S, R = B.sk_R;
  const uint32_t n8 = (uint32_t)B.sk_n * 8u, n16 = 2u * n8;  // bytes of a field of doubles, of pairs
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // compute waves holding rows of this part (R is a multiple of split * 64 /
  // LPC); the launch may carry more for the level's tallest block, they sit out
  const int nw = R * LPC / (64 * G);
  const int t = half * (R / G) + (LPC == 2 ? tid >> 1 : tid), k = LPC == 2 ? tid & 1 : 0;
  const bool has_in = half > 0, has_out = half < G - 1;
  for (int q = tid; q < 2 * (int)(sizeof(Chain<NV, 17>) / 8); q += blockDim.x) reinterpret_cast<double*>(ch)[q] = 0.0;
  __syncthreads();
  if (tid < 2) {
    if (!has_in) ch[tid].prog[0] = CHAIN_END;
    if (!has_out) ch[tid].cons[nw] = CHAIN_END;
  }
  __syncthreads();
  // the block's record region: forward set, backward set (its X pairs first),
  // output pairs
  const uint32_t bytes = (uint32_t)((2 * F::NREC + 2 * F::XP) * B.sk_n * 8);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(a.sk + B.sk_base, 0, bytes, 0x00020000);
  const uint32_t fw = 0, bw = F::NREC * n8, out = 2 * F::NREC * n8;
  const int npad = (S + D - 1) / D * D;
  // global ring of boundary b (between parts b and b+1) for sweep direction d
  auto gr = [&](int b, int d) { return a.gring + (((int64_t)bi * (G - 1) + b) * 2 + d) * a.gstride; };
  const bool rcv = has_in && wave == nw, snd = has_out && wave == nw + (has_in ? 1 : 0);
  if (a.dir != 2) {
    if (wave < nw) sweep<NV, VISC, true, D, LPC, LINK>(rs, fw, bw, n16, S, R, ncol, nrow, t, k, lane, wave, g, ch[0]);
    else if (rcv) comm_receive<NV>(ch[0], gr(half - 1, 0), npad, a.err, a.spin_max);
    else if (snd) comm_forward<NV>(ch[0], nw, gr(half, 0), npad);
  }
  // the forward sweep's X before the backward sweep reads it: in one launch
  // only when the block has one workgroup, so a barrier (workgroup scope) does
  if (a.dir == 0) __syncthreads();
  if (a.dir != 1) {
    if (wave < nw) sweep<NV, VISC, false, D, LPC, LINK>(rs, bw, out, n16, S, R, ncol, nrow, t, k, lane, wave, g, ch[1]);
    else if (rcv) comm_receive<NV>(ch[1], gr(half - 1, 1), npad, a.err, a.spin_max);
    else if (snd) comm_forward<NV>(ch[1], nw, gr(half, 1), npad);
  }
}

// ------------------------------------------------- preparation in the sweep
// For levels whose blocks have at most 64 rows (one wave per block, one lane
// per row): k_lusgs_fused does the work of k_lusgs_prep inside the sweep's
// workgroup, so the records never go through HBM.  Wave 0 runs both sweeps
// exactly as k_lusgs_sweep<..., LPC = 1> does (the same cell_step), at the
// highest issue priority of its SIMD; FPROD waves produce the records, each
// every FPROD-th step of the sequence (forward steps 0..npad-1, then backward
// steps 0..npad-1), lane t the cell of row t, from the skewed copy of the
// inputs that k_lusgs_skew (or the residual) made, into a ring of LDS slots.
// A producer loads the inputs of its next record before it waits for a slot,
// so that memory latency is off the records' path.  The
// forward dU goes to the backward records' X in global memory, from where the
// producers take it into the backward records once the sweep wave has turned
// (turned, set behind a fence).  The sweep wave puts the
// backward U + dU (with update; dU without) of eight steps into an LDS
// buffer; the writer wave takes each chunk and stores it to the block planes eight
// consecutive cells of a row at a time: this replaces k_lusgs_scatter
// (stores along a hyperplane, one cache line per lane, hold up whichever
// wave issues them).
//
// The slots hold the records without RecF's padding: 34 doubles of SA, eight
// slots and the buffer take 156 KB of the CU's 160 KB (a six-equation record
// has six slots).  They are filled and released in groups of XD steps, one
// turn of the sweep's loop: it looks at the producers' counters once a turn,
// and a record's LDS offsets are constants of the unrolled loop from one
// address per group.
//
// The writer waits for ob_ready > chunk, reads the chunk, then sets
// ob_taken = chunk + 1; the sweep wave waits for ob_taken >= chunk before
// it writes the chunk's first step, and sets ob_ready after its last.
// Protocol: filled[q] counts the records written into group slot q, consumed
// the steps of the groups that the sweep wave has finished with.  The sweep
// wave waits, before it reads the first record of group G (slot G % NGRP), for
// filled >= XD (G / NGRP + 1); a producer waits, before it writes step g's
// record, for consumed >= XD (g / XD + 1) - NRING.  A producer waits only
// for the sweep wave and the sweep wave only for producers of groups whose
// slots are free, so every wait ends; waits are also bounded
// (a.spin_max polls, then err is set and the wave stops waiting).
template <int NV, bool VISC>
struct FusedSlot {
  using F = RecF<NV, VISC>;
  // the cell's doubles (X without its padding), then side k's from side(k)
  static constexpr int U = NV, YH0 = 2 * NV, YL0 = YH0 + 1, YH4 = YH0 + 2, YL4 = YH0 + 3;
  static constexpr int NSH = 2 * NV + 2 + (NV == 5 ? 2 : 0), NSD = F::NSDU, N = NSH + 2 * NSD;
  static constexpr int side(int k) { return NSH + k * NSD; }
  static constexpr int XD = NV >= 6 ? 2 : 4;     // sweep steps per turn of its loop: one group of slots
  static constexpr int NRING = NV >= 6 ? 6 : 8;  // record slots
  static constexpr int NGRP = NRING / XD;
};
template <int NV, bool VISC>
struct FusedLds {
  using F = FusedSlot<NV, VISC>;
  double rec[F::NRING][F::N][64];  // slot, field, lane
  double ob[8][NV][64];            // the sweep's backward U + dU (update) or dU of eight steps
  int filled[F::NGRP];
  int consumed, turned;
  int ob_ready, ob_taken;          // chunks of eight backward steps put into / taken from ob
};

__device__ __forceinline__ bool wait_bounded(const int* p, int v, int* err, int spin_max) {
  int n = 0;
  while (lds_get(p) < v) {
    if (++n >= spin_max) {
      atomicOr(err, 2);
      return false;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  return true;
}

// The forward dU at a step's backward positions (the backward sweep's X) for
// row r, pairs and, with an odd equation count, a last field of single doubles.
// A lane whose row has no cell at this step reads the nearest row that has
// one: positions without a cell (about (nrow-1)/ncol of the field) are
// never written, and a wave reading them would fetch lines nobody needs;
// such a lane's value never reaches a cell.
template <int NV, bool VISC, int LPC = 1>
__device__ __forceinline__ void load_x(double* x, __amdgpu_buffer_rsrc_t rs, uint32_t bw, uint32_t n16, int st, int r,
                                       int S, int R, int ncol, int nrow) {
  const int sc = min(st, S - 1);
  const int tr = min(max(r, sc - (ncol - 1)), min(sc, nrow - 1));
  const uint32_t pos = (uint32_t)(sc * R + tr);
  if constexpr (LPC == 4) {
    // as the sweep wave stores them: pairs (1, 0), (2, 3), then single doubles
    D2 v = bload2(rs, pos * 16u, bw);
    x[1] = v.x;
    x[0] = v.y;
    v = bload2(rs, pos * 16u, bw + n16);
    x[2] = v.x;
    x[3] = v.y;
#pragma unroll
    for (int m = 4; m < NV; m++) x[m] = bload1(rs, pos * 16u, bw + (uint32_t)(m - 2) * n16);
    return;
  }
#pragma unroll
  for (int j = 0; j < (NV + 1) / 2; j++) {
    if (2 * j + 1 == NV) {
      x[2 * j] = bload1(rs, pos * 8u, bw + (uint32_t)j * n16);
    } else {
      const D2 v = bload2(rs, pos * 16u, bw + (uint32_t)j * n16);
      x[2 * j] = v.x;
      x[2 * j + 1] = v.y;
    }
  }
}

// The writer: each chunk of eight backward steps of ROWS rows (from row0 of
// the backward order) from ob to the block
// planes, every store one aligned 64-byte run (8 cells) of each of 8
// rows.  Row r's cells of a chunk (steps 8ck .. 8ck+7, columns c = step
// - r, plane offset ncol + 1 - c in the row, whose start is 128-byte
// aligned: the pitch is a multiple of 16) straddle two aligned runs.
// Lane = 8 rows x position p of the run (offset mod 8): it reads the one
// step whose cell sits at position p, always the same slot sub of the
// chunk.  Positions 0..q (q = (ncol + 1 + r) mod 8) complete the run they
// fall in and are stored at once; positions q+1..7 start the next run and
// are held one chunk, while the value held from the previous chunk
// completes this one.  A last turn stores the runs held after the final
// chunk.  Every cell is stored exactly once, cells outside the block
// (columns < 0 or >= ncol, rows >= nrow) are skipped.  With update the
// planes are U (U + dU, the update of k_lusgs_scatter; nothing reads the
// dU planes after a main-loop pass, so they are not rewritten), without
// it dU.
template <int NV, int ROWS>
__device__ __forceinline__ void write_planes(double (*ob)[NV][ROWS], int& ob_ready, int& ob_taken, const LusgsArgs& a,
                                             const BlockDesc& B, int row0, int npad, int lane) {
  constexpr int RG = ROWS / 8;
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  double* planes = a.arena + B.base;
  const int p = lane & 7, rl = lane >> 3;
  const int q = (ncol + 1 + rl) & 7;   // rows rl + 8k share it: the pitch and row0 are multiples of 8
  const int sub = (q - p) & 7;
  const bool held = p > q;             // this lane's cell starts the next run
  const int dst = a.update ? a.pm.U : a.pm.dU;
  const int nck = (npad + 7) / 8;
  double keep[RG][NV] = {};
  for (int ck = 0; ck <= nck; ck++) {
    double v[RG][NV];
    if (ck < nck) {
      if (!wait_bounded(&ob_ready, ck + 1, a.err, a.spin_max)) break;
#pragma unroll
      for (int rg = 0; rg < RG; rg++)
#pragma unroll
        for (int m = 0; m < NV; m++) v[rg][m] = ob[sub][m][rg * 8 + rl];
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // the buffer read before it is handed back
      lds_put(&ob_taken, ck + 1);
    } else {
#pragma unroll
      for (int rg = 0; rg < RG; rg++)
#pragma unroll
        for (int m = 0; m < NV; m++) v[rg][m] = 0.0;
    }
#pragma unroll
    for (int rg = 0; rg < RG; rg++) {
      const int r = row0 + rg * 8 + rl;
      // the run's offset in the row: 8 * floor((ncol + 1 + r) / 8) - 8ck + p
      const int off = ((ncol + 1 + r) & ~7) - 8 * ck + p, c = ncol + 1 - off;
      if (r < nrow && c >= 0 && c < ncol) {
        const int64_t qi = (int64_t)(nrow - r + 1) * B.P + off;  // pidx(B, ncol - c, nrow - r)
#pragma unroll
        for (int m = 0; m < NV; m++) planes[(int64_t)(dst + m) * B.plane + qi] = held ? keep[rg][m] : v[rg][m];
      }
#pragma unroll
      for (int m = 0; m < NV; m++) keep[rg][m] = v[rg][m];
    }
  }
}

// The waves of the fused launch: the sweep wave, FPROD producers, the writer,
// and wave 4, which ends at once: a workgroup's waves go to the CU's four SIMDs
// in turn, so waves 0 and 4 share one, and the sweep wave has its SIMD for
// itself (256 SA blocks of 48-64 rows: 0.380 -> 0.368 ms).  A record takes its
// producer about 2 us, most of it memory latency: five producers keep up with
// the sweep, three did not (0.43 ms).
constexpr int FPROD = 5;
constexpr int FUSED_THREADS = 64 * (FPROD + 3);
template <int NV, bool VISC>
__global__ __launch_bounds__(FUSED_THREADS) void k_lusgs_fused(LusgsArgs a) {
  using F = RecF<NV, VISC>;
  using FS = FusedSlot<NV, VISC>;
  constexpr int FRING = FS::NRING, XD = FS::XD, NGRP = FS::NGRP;
  __shared__ FusedLds<NV, VISC> L;
  const BlockDesc B = a.blocks[a.block_list[blockIdx.x]];
  if (case_frozen(B.case_id)) return;
  const double g = a.cps[B.case_id].gamma;
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  const int S = B.sk_S, R = B.sk_R;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = tid < 320 ? tid >> 6 : (tid >> 6) - 1;  // without the idle one
  if (tid < NGRP) L.filled[tid] = 0;
  if (tid == 0) L.consumed = L.turned = L.ob_ready = L.ob_taken = 0;
  __syncthreads();
  if (tid >= 256 && tid < 320) return;  // the sweep wave's SIMD stays free
  const int npad = (S + 3) / 4 * 4;  // whole turns of the sweep
  const int ntot = 2 * npad;
  const uint32_t n8 = (uint32_t)B.sk_n * 8u, n16 = 2u * n8;
  const uint32_t bytes = (uint32_t)((2 * F::NREC + 2 * F::XP) * B.sk_n * 8);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(a.sk + B.sk_base, 0, bytes, 0x00020000);
  const uint32_t bw = F::NREC * n8;
  bool ok = true;
  if (wave == FPROD + 1) {
    write_planes<NV, 64>(L.ob, L.ob_ready, L.ob_taken, a, B, 0, npad, lane);
    return;
  }
  if (wave > 0) {
    // ---- producer: the inputs from their skewed copy (k_lusgs_skew), so
    // that the lanes (rows) of a step read consecutive positions
    const double* skin = a.sk + B.sk_base;
    auto produce = [&](auto fwd_c, int first) {
      constexpr bool fwd = decltype(fwd_c)::value;
      const int gs0 = fwd ? 0 : npad;
      // the inputs of the producer's next two records are in flight while it
      // makes one: a load takes up to 2 us, a sweep step about 0.45
      RecSrc<NV> nx[2];
      auto fetch = [&](RecSrc<NV>& q, int gs, bool x) {
        const int sn = min(gs - gs0, npad - 1);  // past the last step: clamped to it
        load_src_sk<NV, VISC, fwd>(q, B, skin, sn - lane, lane);
        if (!fwd && x) load_x<NV, VISC>(q.Res, rs, bw, n16, sn, lane, S, R, ncol, nrow);
      };
      fetch(nx[0], first, false);
      fetch(nx[1], first + FPROD, false);
      if constexpr (!fwd) {
        // the forward dU, from here on in memory
        ok = wait_bounded(&L.turned, 1, a.err, a.spin_max);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        load_x<NV, VISC>(nx[0].Res, rs, bw, n16, min(first - gs0, npad - 1), lane, S, R, ncol, nrow);
        load_x<NV, VISC>(nx[1].Res, rs, bw, n16, min(first + FPROD - gs0, npad - 1), lane, S, R, ncol, nrow);
      }
      auto record = [&](RecSrc<NV>& n, int gs) {
        const RecSrc<NV> q = n;
        fetch(n, gs + 2 * FPROD, true);
        ok = wait_bounded(&L.consumed, (gs / XD + 1) * XD - FRING, a.err, a.spin_max);
        double* rec = &L.rec[gs % FRING][0][lane];
        auto SH = [&](int d) -> double& { return rec[d * 64]; };
        auto SD = [&](int kk, int e) -> double& { return rec[(FS::side(kk) + e) * 64]; };
        rec_body<NV, VISC, fwd, true, FS>(SH, SD, q, g, a.alfa1);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // the slot's LDS writes done (lgkmcnt 0) before counting it
        if (lane == 0)
          __hip_atomic_fetch_add(&L.filled[(gs / XD) % NGRP], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      };
      int gs = first;
      while (gs < gs0 + npad && ok) {
        record(nx[0], gs);
        gs += FPROD;
        if (gs >= gs0 + npad || !ok) break;
        record(nx[1], gs);
        gs += FPROD;
      }
      return gs;
    };
    const int g1 = produce(std::true_type{}, wave - 1);
    if (ok) produce(std::false_type{}, g1);
    return;
  }
  // ---- the sweep wave: lane t = row t; it issues first on its SIMD
  __builtin_amdgcn_s_setprio(3);
  const int t = lane;
  auto load_lds = [&](Rec<NV, 2>& r, const double* rec) {  // rec: the slot's first field of the lane
#pragma unroll
    for (int m = 0; m < NV; m++) {
      r.X[m] = rec[m * 64];
      r.U[m] = rec[(FS::U + m) * 64];
    }
    r.yh0 = rec[FS::YH0 * 64];
    r.yl0 = rec[FS::YL0 * 64];
    if constexpr (NV == 5) {
      r.yh4 = rec[FS::YH4 * 64];
      r.yl4 = rec[FS::YL4 * 64];
    } else {
      r.yh4 = r.yh0;
      r.yl4 = r.yl0;
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const double* sd = rec + FS::side(h) * 64;
#pragma unroll
      for (int m = 0; m < NV; m++) r.F[h][m] = sd[(F::F + m) * 64];
      r.n1[h] = sd[F::N1 * 64];
      r.n2[h] = sd[F::N2 * 64];
      r.a[h] = sd[F::A * 64];
      r.Lc[h] = sd[F::LC * 64];
      if constexpr (VISC) r.Lv[h] = sd[F::LV * 64];
      else r.Lv[h] = 0.0;
    }
  };
  // One direction of the sweep; the direction is a compile-time constant so
  // that every register array keeps fixed indices.  The next step's record
  // is read from its slot while this step computes.
  int grp = 0, round = 1;  // the group slot of the turn and its use
  auto run_dir = [&](auto fwd_c) {
    constexpr bool fwd = decltype(fwd_c)::value;
    const int gs0 = fwd ? 0 : npad;
    Terms<NV, 1> tm = {};
    // a lane without a cell at a step sends its stores out of the buffer's
    // range, where they are dropped; a row past the block never has a cell
    constexpr uint32_t NOWHERE = 0x80000000u;
    const int ts = t < nrow ? t : 0x40000000;
    uint32_t w8 = (uint32_t)((S - 1) * R + (nrow - 1 - t)) * 8u;  // forward: the cell's X position, falling by R a step
    Rec<NV, 2> rn;
    if (ok) ok = wait_bounded(&L.filled[grp], XD * round, a.err, a.spin_max);
    load_lds(rn, &L.rec[grp * XD][0][t]);
    for (int st = 0; st < npad; st += XD) {
      const double* rec = &L.rec[grp * XD][0][t];
      const int grp1 = grp + 1 == NGRP ? 0 : grp + 1, round1 = grp + 1 == NGRP ? round + 1 : round;
      int pv = 0;  // the next group's count, read a step before it is needed
#pragma unroll
      for (int k = 0; k < XD; k++) {
        const int s = st + k;
        Rec<NV, 2> r = rn;
        // The next step's record.  Its loads are unconditional: a load under
        // a branch makes its registers a phi, which the compiler resolves
        // with copies that wait for the load in flight and so undo the
        // prefetch.  After the direction's last step the slot read is not
        // waited for and its values are never used (the next direction
        // reloads after its own wait).
        if (k == XD - 1) {
          if (s + 1 < npad && ok && pv < XD * round1)
            ok = wait_bounded(&L.filled[grp1], XD * round1, a.err, a.spin_max);
          __atomic_signal_fence(__ATOMIC_SEQ_CST);
          load_lds(rn, &L.rec[grp1 * XD][0][t]);
        } else {
          load_lds(rn, rec + (k + 1) * FS::N * 64);
          if (k == XD - 2) {
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            pv = lds_get(&L.filled[grp1]);
          }
        }
        Out<NV> o;
        double jin[NV];
#pragma unroll
        for (int m = 0; m < NV; m++) jin[m] = shr1(tm.j[m]);
        cell_step<NV, VISC, fwd, 1>(r, tm, jin, o, g);
        interleave<0x100, FS::N / 2, 7>();
        if constexpr (fwd) {
          // dU to the backward records' X (with an odd equation count the
          // last field holds single doubles)
          const bool act = (uint32_t)(s - ts) < (uint32_t)ncol;
          const uint32_t w = act ? 2 * w8 : NOWHERE, wo = act ? w8 : NOWHERE;
          w8 -= (uint32_t)R * 8u;
#pragma unroll
          for (int j = 0; j < F::XP; j++) {
            if (2 * j + 1 == NV) bstore1(o.du[2 * j], rs, wo, bw + (uint32_t)j * n16);
            else bstore2(o.du[2 * j], o.du[2 * j + 1], rs, w, bw + (uint32_t)j * n16);
          }
        } else {
          // U + dU (the record's U is the plane's value; with update) or dU
          // into the output buffer, which the writer wave stores eight steps
          // at a time; npad is a multiple of four, so the last chunk may end
          // after four
          const int b8 = s & 7, ck = s >> 3;
          if (k == 0 || XD < 4)
            if (b8 == 0 && ck > 0 && ok) ok = wait_bounded(&L.ob_taken, ck, a.err, a.spin_max);
          if (a.update) {
#pragma unroll
            for (int m = 0; m < NV; m++) L.ob[b8][m][t] = o.W[m];
          } else {
#pragma unroll
            for (int m = 0; m < NV; m++) L.ob[b8][m][t] = o.du[m];
          }
          if ((k == XD - 1) && (b8 == 7 || s == npad - 1)) {
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_s_waitcnt(0xc07f);  // the chunk's writes done before it is handed over
            lds_put(&L.ob_ready, ck + 1);
          }
        }
      }
      // the group's records have all been read (the last one's values were
      // used by its step)
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      lds_put(&L.consumed, gs0 + st + XD);
      grp = grp1;
      round = round1;
    }
  };
  run_dir(std::true_type{});
  // The forward sweep's stores before the producers' loads: waves of one
  // workgroup, so workgroup scope.  (A device-scope fence also writes back the
  // whole L2.)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  lds_put(&L.turned, 1);
  run_dir(std::false_type{});
}

// ------------------------------------------- the same, in parts of a block's rows
// For levels of few blocks (k parts each, at most one workgroup per CU): each
// part of 16 or 32 rows is a workgroup of its own, linked to the next through
// global memory as the split sweeps' workgroups are, and makes its records in
// LDS as k_lusgs_fused does.  What bounds a single block is the chain of steps,
// so a cell of the sweep wave has two lanes (32 rows) or four (16): of a step of
// four equations' 130 instructions 70 are FP64 with two, of 107 42 with four, in
// which each half of the wave takes half of the equations.  (The split sweeps'
// wave reads its records by 13 memory loads a step, which take it about 7 ns each
// to issue; the LDS reads here 3.)  An update of 257 x 65 cells, four equations,
// 0.19 ms with four lanes, 0.22 with two and with the split sweeps.
//   A producer's 64 lanes make the records of two (four) steps at a time.  LDS
// records come in pairs of doubles, the cell's part by row, the sides' by
// lane, so that the sweep wave's reads are 16 bytes a lane without bank conflicts.
//   A block of one part runs both sweeps in one launch; with several the
// sweeps are separate launches (a.dir), as in k_lusgs_sweep.
template <int NV, bool VISC>
struct PartSlot {
  using F = RecF<NV, VISC>;
  static constexpr int U = NV, YH0 = 2 * NV, YL0 = YH0 + 1, YH4 = YH0 + 2, YL4 = YH0 + 3;
  static constexpr int NSH = 2 * NV + 2 + (NV == 5 ? 2 : 0), NSD = F::NSD;
  static constexpr int SIDE = NSH / 2 * 64, N = SIDE + NSD / 2 * 128;  // doubles of a slot
  static constexpr int XD = 4;                      // sweep steps per turn: one group of slots
  static constexpr int NRING = NV >= 6 ? 12 : 16;   // record slots
  static constexpr int NGRP = NRING / XD;
  // the cell's double d of a row, side k's double e of a row
  __device__ static constexpr int cell(int d, int row) { return d / 2 * 64 + 2 * row + (d & 1); }
  __device__ static constexpr int side(int k, int e, int row) { return SIDE + e / 2 * 128 + 2 * (2 * row + k) + (e & 1); }
};
// Four lanes per cell (parts of 16 rows): lane 32 h + 2 t + k of row t has side k and
// half h of the equations, NP of them: one of the momentum equations, then mass or
// energy, then what the turbulence model adds (one equation: h = 0 only, and half
// 1 computes with whatever is in its place).
template <int NV, bool VISC>
struct QuadSlot {
  using F = RecF<NV, VISC>;
  static constexpr int U = NV, YH0 = 2 * NV, YL0 = YH0 + 1, YH4 = YH0 + 2, YL4 = YH0 + 3;
  static constexpr int NP = NV == 4 ? 2 : 3;
  static constexpr int CY = NP * 64, SIDE = CY + (NV == 5 ? 64 : 32), LANE = SIDE + (VISC ? 192 : 128);
  static constexpr int N = LANE + (NP + 1) / 2 * 128;  // doubles of a slot
  static constexpr int XD = 4;
  static constexpr int NRING = 16;
  static constexpr int NGRP = NRING / XD;
  // half and place of equation m
  __device__ static constexpr int half(int m) { return m == 2 || m == 3 || m == 5; }
  __device__ static constexpr int place(int m) { return m == 1 || m == 2 ? 0 : m < 4 ? 1 : 2; }
  // X and U by (half, row): pairs X0 X1, U0 U1 or X0 X1, X2 U2, U0 U1
  __device__ static constexpr int xu(bool u, int h, int p, int row) {
    const int d = p == 2 ? 2 + u : NP == 2 ? 2 * u + p : 4 * u + p;
    return d / 2 * 64 + 2 * (16 * h + row) + (d & 1);
  }
  __device__ static constexpr int cell(int d, int row) {
    if (d < 2 * NV) return xu(d >= NV, half(d % NV), place(d % NV), row);
    return CY + (d - YH0) / 2 * 32 + 2 * row + ((d - YH0) & 1);
  }
  // F by lane (of three, then the normal's component of the momentum equation);
  // n1 n2, a Lc, Lv by (row, side)
  __device__ static constexpr int side(int k, int e, int row) {
    if (e < NV) return LANE + place(e) / 2 * 128 + 2 * (32 * half(e) + 2 * row + k) + (place(e) & 1);
    const int d = e == F::N1 ? 0 : e == F::N2 ? 1 : e == F::A ? 2 : e == F::LC ? 3 : 4;
    return SIDE + d / 2 * 64 + 2 * (2 * row + k) + (d & 1);
  }
};
template <int NV, bool VISC, int LPC>
using PartSlotOf = std::conditional_t<LPC == 4, QuadSlot<NV, VISC>, PartSlot<NV, VISC>>;
template <int NV, bool VISC, int LPC>
struct PartLds {
  using F = PartSlotOf<NV, VISC, LPC>;
  alignas(16) double rec[F::NRING][F::N];
  double ob[8][NV][64 / LPC];  // the backward U + dU (update) or dU of eight steps
  Chain<NV, 2> ch[2];    // one per sweep
  int filled[F::NGRP];
  int consumed, turned, ob_ready, ob_taken;
  int part;
};
constexpr int PART_PROD = 3;       // producers: waves 1 .. 3 (wave 4 ends at once, see FUSED_THREADS)
constexpr int PART_THREADS = 512;  // then the writer, the receiving and the sending wave

// the value of lane l and of lane l ^ 32: x in the lower lanes, y in the upper
__device__ __forceinline__ void both_halves(double v, double& x, double& y) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
  x = __hiloint2double(hi[0], lo[0]);
  y = __hiloint2double(hi[1], lo[1]);
}

// The sweep wave of a part of 16 rows (lanes: QuadSlot).  A step is a sum, a
// quotient and U + dU per equation of the lane's half, the halves' exchange by
// lane moves, p and F(U).n once per side, and the lane's terms.
template <int NV, bool VISC>
__device__ __forceinline__ void quad_sweeps(const LusgsArgs& a, PartLds<NV, VISC, 4>& L, __amdgpu_buffer_rsrc_t rs,
                                            uint32_t bw, uint32_t n16, int S, int R, int ncol, int nrow, int row0,
                                            int lane, int npad, double g, bool do_f, bool do_b) {
  using PS = QuadSlot<NV, VISC>;
  constexpr int NP = PS::NP, NRING = PS::NRING, XD = PS::XD, NGRP = PS::NGRP;
  const int h = lane >> 5, row = lane >> 1 & 15, k = lane & 1, t = row0 + row;
  struct R4 {
    double X[NP], U[NP], F[NP], yh, yl, yh4, yl4, n1, n2, nA, a, Lc, Lv;
  };
  const int o_xu = 2 * (16 * h + row), o_cy = PS::CY + 2 * row, o_sd = PS::SIDE + 2 * (lane & 31),
            o_ln = PS::LANE + 2 * lane;
  auto load_lds = [&](R4& r, const double* rec) {
    auto pair = [&](int at) { return *reinterpret_cast<const D2a*>(rec + at); };
    D2a v = pair(o_xu);
    r.X[0] = v.x;
    r.X[1] = v.y;
    if constexpr (NP == 3) {
      v = pair(o_xu + 64);
      r.X[NP - 1] = v.x;
      r.U[NP - 1] = v.y;
    }
    v = pair(o_xu + (NP - 1) * 64);
    r.U[0] = v.x;
    r.U[1] = v.y;
    v = pair(o_cy);
    r.yh = v.x;
    r.yl = v.y;
    if constexpr (NV == 5) v = pair(o_cy + 32);
    r.yh4 = v.x;
    r.yl4 = v.y;
    v = pair(o_sd);
    r.n1 = v.x;
    r.n2 = v.y;
    v = pair(o_sd + 64);
    r.a = v.x;
    r.Lc = v.y;
    r.Lv = VISC ? rec[o_sd + (VISC ? 128 : 0)] : 0.0;
    v = pair(o_ln);
    r.F[0] = v.x;
    r.F[1] = v.y;
    if constexpr (NP == 3) {
      v = pair(o_ln + 128);
      r.F[NP - 1] = v.x;
      r.nA = v.y;
    } else {
      r.nA = h ? r.n2 : r.n1;
    }
  };
  constexpr int NREAD = NP + 1 + (NV == 5) + 2 + VISC + NP - 1;
  // this lane's equations, for the planes' chunk buffer
  const int eq[3] = {h ? 2 : 1, h ? 3 : 0, NV == 6 && h ? 5 : 4};
  // in a ring slot: momentum, mass or energy of half 0, of half 1, then the rest
  const int rg = 2 * h, rg2 = NV == 6 ? 4 + h : 4;
  bool ok = true;
  int grp = 0, need = XD;  // the group slot of the turn, its steps when it is full
  const double* rec = L.rec[0];
  auto run_dir = [&](auto fwd_c, int gs0) {
    constexpr bool fwd = decltype(fwd_c)::value;
    Chain<NV, 2>& ch = L.ch[fwd ? 0 : 1];
    double tm[NP] = {};
    constexpr uint32_t NOWHERE = 0x80000000u;  // out of the buffer's range: the store is dropped
    const int ts = t < nrow && k == 0 ? t : 0x40000000;
    uint32_t w16 = (uint32_t)((S - 1) * R + (nrow - 1 - t)) * 16u + (h ? n16 : 0u);
    double in[NP];
    // the last row's terms go to the next part, the others' nowhere (half 1 of five
    // equations has no third)
    const bool out = row == 15 && k == 1;
    double(*rout)[NV] = out ? ch.ring[1] : ch.dump;
    double(*rout2)[NV] = out && !(NV == 5 && h) ? ch.ring[1] : ch.dump;
    auto read_in = [&](int slot) {
      in[0] = ch.ring[0][slot][rg];
      in[1] = ch.ring[0][slot][rg + 1];
      if constexpr (NP == 3) in[NP - 1] = ch.ring[0][slot][rg2];
    };
    int prog = 0, cons = 0, pv = 0;
    auto look = [&] {
      prog = lds_get(&ch.prog[0]);
      cons = lds_get(&ch.cons[1]);
    };
    look();
    R4 rn;
    if (ok) ok = wait_bounded(&L.filled[grp], need, a.err, a.spin_max);
    load_lds(rn, rec);
    for (int st = 0; st < npad; st += XD) {
      const bool wrap = grp == NGRP - 1;
      const int grp1 = wrap ? 0 : grp + 1, need1 = wrap ? need + XD : need;
      const double* rec1 = wrap ? L.rec[0] : rec + XD * PS::N;
      const int slot0 = st & (RING - 1);
      if (prog < st + XD - 1) wait_at_least(&ch.prog[0], st + XD - 1);
      if (cons < st + XD + 1 - RING) wait_at_least(&ch.cons[1], st + XD + 1 - RING);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      read_in((st - 1) & (RING - 1));
#pragma unroll
      for (int u = 0; u < XD; u++) {
        const int s = st + u;
        const R4 r = rn;
        if (u == XD - 1) {
          if (s + 1 < npad && ok && pv < need1)
            ok = wait_bounded(&L.filled[grp1], need1, a.err, a.spin_max);
          __atomic_signal_fence(__ATOMIC_SEQ_CST);
          load_lds(rn, rec1);
        } else {
          load_lds(rn, rec + (u + 1) * PS::N);
        }
        double jin[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
          const double x = shr1(tm[p]);
          jin[p] = row == 0 ? in[p] : x;
        }
        if (u + 1 < XD) read_in(slot0 + u);
        // the reference's order per equation: (Res + dui) + duj forward, X + (dui +
        // duj) / alfa backward (cell_step)
        double du[NP], W[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
          const double sum = even_lane(fwd ? (r.X[p] + tm[p]) + jin[p] : tm[p] + jin[p]);
          const bool sa = NV == 5 && p == 2;
          const double q = div_hl(sum, sa ? r.yh4 : r.yh, sa ? r.yl4 : r.yl);
          du[p] = fwd ? q : r.X[p] + q;
          W[p] = r.U[p] + du[p];
        }
        double C[4];
        both_halves(W[1], C[0], C[3]);
        both_halves(W[0], C[1], C[2]);
        const double y = rcp_n(C[0]);
        const double pr = pressure_y(C, y, g);
        const double un = div_y(C[1] * r.n1 + C[2] * r.n2, C[0], y);
        const double pB = h ? pr : 0.0;
        double Fn[NP];
        Fn[0] = W[0] * un + pr * r.nA;
        Fn[1] = (W[1] + pB) * un;
        if constexpr (NP == 3) Fn[NP - 1] = W[NP - 1] * un;
#pragma unroll
        for (int p = 0; p < NP; p++) {
          tm[p] = (Fn[p] - r.F[p]) * r.a + r.Lc * du[p];
          if constexpr (VISC) tm[p] = tm[p] + r.Lv * du[p];
        }
        rout[slot0 + u][rg] = tm[0];
        rout[slot0 + u][rg + 1] = tm[1];
        if constexpr (NP == 3) rout2[slot0 + u][rg2] = tm[NP - 1];
        interleave<0x100, NREAD, 1>();
        if constexpr (fwd) {
          // (load_x reads them; the third of half 1 lands in a field that only the split
          // sweeps' records have, with five equations unused)
          const uint32_t w = (uint32_t)(s - ts) < (uint32_t)ncol ? w16 : NOWHERE;
          bstore2(du[0], du[1], rs, w, bw);
          if constexpr (NP == 3) bstore1(du[NP - 1], rs, w, bw + 2 * n16);
          w16 -= (uint32_t)R * 16u;
        } else {
          const int b8 = s & 7, ck = s >> 3;
          if (u == 0 && b8 == 0 && ck > 0 && ok) ok = wait_bounded(&L.ob_taken, ck, a.err, a.spin_max);
#pragma unroll
          for (int p = 0; p < NP; p++)
            if (!(NV == 5 && p == 2 && h)) L.ob[b8][eq[p]][row] = a.update ? W[p] : du[p];
          if (u == XD - 1 && (b8 == 7 || s == npad - 1)) {
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_s_waitcnt(0xc07f);  // the chunk's writes done before it is handed over
            lds_put(&L.ob_ready, ck + 1);
          }
        }
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        lds_put(&ch.prog[1], s + 1);
        if (u == XD - 2) {
          look();
          pv = lds_get(&L.filled[grp1]);
        }
      }
      lds_put(&ch.cons[0], st + XD);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      lds_put(&L.consumed, gs0 + st + XD);
      grp = grp1;
      need = need1;
      rec = rec1;
    }
  };
  if (do_f) run_dir(std::true_type{}, 0);
  if (do_f && do_b) {
    // the forward sweep's stores before the producers' loads (see k_lusgs_fused)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    lds_put(&L.turned, 1);
  }
  if (do_b) run_dir(std::false_type{}, do_f ? npad : 0);
}

template <int NV, bool VISC, int LPC>
__global__ __launch_bounds__(PART_THREADS) void k_lusgs_parts(LusgsArgs a) {
  using F = RecF<NV, VISC>;
  using PS = PartSlotOf<NV, VISC, LPC>;
  constexpr int NRING = PS::NRING, XD = PS::XD, NGRP = PS::NGRP;
  constexpr int PART_ROWS = 64 / LPC;
  __shared__ PartLds<NV, VISC, LPC> L;
  const int G = a.split, bi = blockIdx.x / G;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // A block's workgroups take its parts in the order in which they start, so that the
  // part below has always started before one that waits for it, however another
  // process's kernels share the device (by block index alone each could hold the CUs that
  // the other's lower parts need).  The count wraps to 0 with the last of them.
  if (tid == 0) L.part = G > 1 ? (int)atomicInc(a.tickets + bi, (unsigned)(G - 1)) : 0;
  const BlockDesc B = a.blocks[a.block_list[bi]];
  if (case_frozen(B.case_id)) return;  // every part of the block returns: no part waits on another
  const double g = a.cps[B.case_id].gamma;
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  const int nparts = (nrow + PART_ROWS - 1) / PART_ROWS;
  const int S = B.sk_S, R = B.sk_R;
  for (int q = tid; q < 2 * (int)(sizeof(Chain<NV, 2>) / 8); q += PART_THREADS) reinterpret_cast<double*>(L.ch)[q] = 0.0;
  if (tid < NGRP) L.filled[tid] = 0;
  if (tid == 0) {
    L.consumed = L.ob_ready = L.ob_taken = 0;
    L.turned = a.dir == 2 ? 1 : 0;  // a backward launch finds the forward dU in memory
  }
  __syncthreads();
  const int part = __builtin_amdgcn_readfirstlane(L.part);
  if (part >= nparts) return;  // the launch fits the level's tallest block
  const bool has_in = part > 0, has_out = part < nparts - 1;
  const int row0 = part * PART_ROWS;
  if (tid < 2) {
    if (!has_in) L.ch[tid].prog[0] = CHAIN_END;
    if (!has_out) L.ch[tid].cons[1] = CHAIN_END;
  }
  __syncthreads();
  const int npad = (S + XD - 1) / XD * XD;
  const bool do_f = a.dir != 2, do_b = a.dir != 1;
  const uint32_t n8 = (uint32_t)B.sk_n * 8u, n16 = 2u * n8;
  const uint32_t bytes = (uint32_t)((2 * F::NREC + 2 * F::XP) * B.sk_n * 8);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(a.sk + B.sk_base, 0, bytes, 0x00020000);
  const uint32_t bw = F::NREC * n8;
  auto gr = [&](int b, int d) { return a.gring + (((int64_t)bi * (G - 1) + b) * 2 + d) * a.gstride; };
  bool ok = true;
  if (wave == PART_PROD + 1) return;
  if (wave == PART_PROD + 3) {
    if (!has_in) return;
    if (do_f) comm_receive<NV>(L.ch[0], gr(part - 1, 0), npad, a.err, a.spin_max);
    if (do_b) comm_receive<NV>(L.ch[1], gr(part - 1, 1), npad, a.err, a.spin_max);
    return;
  }
  if (wave == PART_PROD + 4) {
    if (!has_out) return;
    if (do_f) comm_forward<NV>(L.ch[0], 1, gr(part, 0), npad);
    if (do_b) comm_forward<NV>(L.ch[1], 1, gr(part, 1), npad);
    return;
  }
  if (wave == PART_PROD + 2) {
    if (do_b) write_planes<NV, PART_ROWS>(L.ob, L.ob_ready, L.ob_taken, a, B, row0, npad, lane);
    return;
  }
  if (wave > 0) {
    // ---- producer: steps LPC q, .., LPC q + LPC - 1 (of PART_ROWS lanes each) of
    // every PART_PROD-th q
    const double* skin = a.sk + B.sk_base;
    const int row = lane % PART_ROWS, half = lane / PART_ROWS, r = row0 + row;
    auto produce = [&](auto fwd_c, int q0) {
      constexpr bool fwd = decltype(fwd_c)::value;
      RecSrc<NV> nx[2];
      auto fetch = [&](RecSrc<NV>& n, int q, bool x) {
        const int sn = min(LPC * q + half, npad - 1);  // past the last step: clamped to it
        load_src_sk<NV, VISC, fwd>(n, B, skin, sn - r, r);
        if (!fwd && x) load_x<NV, VISC, LPC>(n.Res, rs, bw, n16, sn, r, S, R, ncol, nrow);
      };
      int q = wave - 1;
      fetch(nx[0], q, false);
      fetch(nx[1], q + PART_PROD, false);
      if constexpr (!fwd) {
        // the forward dU, from here on in memory
        ok = wait_bounded(&L.turned, 1, a.err, a.spin_max);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        load_x<NV, VISC, LPC>(nx[0].Res, rs, bw, n16, min(LPC * q + half, npad - 1), r, S, R, ncol, nrow);
        load_x<NV, VISC, LPC>(nx[1].Res, rs, bw, n16, min(LPC * (q + PART_PROD) + half, npad - 1), r, S, R, ncol, nrow);
      }
      auto record = [&](RecSrc<NV>& n, int q) {
        const RecSrc<NV> in = n;
        fetch(n, q + 2 * PART_PROD, true);
        const int gs = q0 + LPC * q;  // the first of the steps in the sequence of both sweeps
        ok = wait_bounded(&L.consumed, (gs / XD + 1) * XD - NRING, a.err, a.spin_max);
        double* rec = L.rec[(gs + half) % NRING];
        auto SH = [&](int d) -> double& { return rec[PS::cell(d, row)]; };
        auto SD = [&](int k, int e) -> double& { return rec[PS::side(k, e, row)]; };
        rec_body<NV, VISC, fwd, true, PS>(SH, SD, in, g, a.alfa1);
        if constexpr (LPC == 4 && NV > 4) {
#pragma unroll
          for (int k = 0; k < 2; k++) {
            rec[PS::LANE + 128 + 2 * (2 * row + k) + 1] = in.n1[k];
            rec[PS::LANE + 128 + 2 * (32 + 2 * row + k) + 1] = in.n2[k];
          }
        }
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // the slots' LDS writes done (lgkmcnt 0) before counting them
        if (lane == 0)
          __hip_atomic_fetch_add(&L.filled[(gs / XD) % NGRP], LPC, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      };
      while (LPC * q < npad && ok) {
        record(nx[0], q);
        q += PART_PROD;
        if (LPC * q >= npad || !ok) break;
        record(nx[1], q);
        q += PART_PROD;
      }
    };
    if (do_f) produce(std::true_type{}, 0);
    if (do_b && ok) produce(std::false_type{}, do_f ? npad : 0);
    return;
  }
  // ---- the sweep wave: lanes 2t, 2t+1 = row row0 + t; it issues first on its SIMD
  __builtin_amdgcn_s_setprio(3);
  if constexpr (LPC == 4) {
    quad_sweeps<NV, VISC>(a, L, rs, bw, n16, S, R, ncol, nrow, row0, lane, npad, g, do_f, do_b);
    return;
  } else {
  const int row = lane >> 1, t = row0 + row, k = lane & 1;
  auto load_lds = [&](Rec<NV, 1>& r, const double* rec) {
    const double* cp = rec + 2 * row;
    double c[PS::NSH], e[PS::NSD];
#pragma unroll
    for (int j = 0; j < PS::NSH / 2; j++) {
      const D2a v = *reinterpret_cast<const D2a*>(cp + j * 64);
      c[2 * j] = v.x;
      c[2 * j + 1] = v.y;
    }
    const double* sp = rec + PS::SIDE + 2 * lane;
#pragma unroll
    for (int j = 0; j < PS::NSD / 2; j++) {
      const D2a v = *reinterpret_cast<const D2a*>(sp + j * 128);
      e[2 * j] = v.x;
      e[2 * j + 1] = v.y;
    }
#pragma unroll
    for (int m = 0; m < NV; m++) {
      r.X[m] = c[m];
      r.U[m] = c[PS::U + m];
      r.F[0][m] = e[F::F + m];
    }
    r.yh0 = c[PS::YH0];
    r.yl0 = c[PS::YL0];
    r.yh4 = NV == 5 ? c[NV == 5 ? PS::YH4 : 0] : r.yh0;
    r.yl4 = NV == 5 ? c[NV == 5 ? PS::YL4 : 0] : r.yl0;
    r.n1[0] = e[F::N1];
    r.n2[0] = e[F::N2];
    r.a[0] = e[F::A];
    r.Lc[0] = e[F::LC];
    r.Lv[0] = VISC ? e[VISC ? F::LV : 0] : 0.0;
  };
  int grp = 0, round = 1;  // the group slot of the turn and its use
  auto run_dir = [&](auto fwd_c, int gs0) {
    constexpr bool fwd = decltype(fwd_c)::value;
    Chain<NV, 2>& ch = L.ch[fwd ? 0 : 1];
    Terms<NV, 2> tm = {};
    constexpr uint32_t NOWHERE = 0x80000000u;  // out of the buffer's range: the store is dropped
    const int ts = t < nrow && k == 0 ? t : 0x40000000;
    uint32_t w8 = (uint32_t)((S - 1) * R + (nrow - 1 - t)) * 8u;
    double in[NV];
    double(*rout)[NV] = lane == 63 ? ch.ring[1] : ch.dump;
    auto read_in = [&](int slot) {
#pragma unroll
      for (int m = 0; m < NV; m++) in[m] = ch.ring[0][slot][m];
    };
    int prog = 0, cons = 0, pv = 0;
    auto look = [&] {
      prog = lds_get(&ch.prog[0]);
      cons = lds_get(&ch.cons[1]);
    };
    look();
    Rec<NV, 1> rn;
    if (ok) ok = wait_bounded(&L.filled[grp], XD * round, a.err, a.spin_max);
    load_lds(rn, L.rec[grp * XD]);
    for (int st = 0; st < npad; st += XD) {
      const double* rec = L.rec[grp * XD];
      const int grp1 = grp + 1 == NGRP ? 0 : grp + 1, round1 = grp + 1 == NGRP ? round + 1 : round;
      const int slot0 = st & (RING - 1);
      if (prog < st + XD - 1) wait_at_least(&ch.prog[0], st + XD - 1);
      if (cons < st + XD + 1 - RING) wait_at_least(&ch.cons[1], st + XD + 1 - RING);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      read_in((st - 1) & (RING - 1));
#pragma unroll
      for (int u = 0; u < XD; u++) {
        const int s = st + u;
        const Rec<NV, 1> r = rn;
        // the next step's record (see k_lusgs_fused)
        if (u == XD - 1) {
          if (s + 1 < npad && ok && pv < XD * round1)
            ok = wait_bounded(&L.filled[grp1], XD * round1, a.err, a.spin_max);
          __atomic_signal_fence(__ATOMIC_SEQ_CST);
          load_lds(rn, L.rec[grp1 * XD]);
        } else {
          load_lds(rn, rec + (u + 1) * PS::N);
        }
        double jin[NV];
#pragma unroll
        for (int m = 0; m < NV; m++) jin[m] = shr1_in(in[m], tm.j[m]);
        if (u + 1 < XD) read_in(slot0 + u);
        Out<NV> o;
        cell_step<NV, VISC, fwd, 2>(r, tm, jin, o, g);
#pragma unroll
        for (int m = 0; m < NV; m++) rout[slot0 + u][m] = tm.j[m];
        interleave<0x100, (PS::NSH + PS::NSD) / 2, 1>();
        if constexpr (fwd) {
          const bool act = (uint32_t)(s - ts) < (uint32_t)ncol;
          const uint32_t w = act ? 2 * w8 : NOWHERE, wo = act ? w8 : NOWHERE;
          w8 -= (uint32_t)R * 8u;
#pragma unroll
          for (int j = 0; j < F::XP; j++) {
            if (2 * j + 1 == NV) bstore1(o.du[2 * j], rs, wo, bw + (uint32_t)j * n16);
            else bstore2(o.du[2 * j], o.du[2 * j + 1], rs, w, bw + (uint32_t)j * n16);
          }
        } else {
          const int b8 = s & 7, ck = s >> 3;
          if (u == 0 && b8 == 0 && ck > 0 && ok) ok = wait_bounded(&L.ob_taken, ck, a.err, a.spin_max);
#pragma unroll
          for (int m = 0; m < NV; m++) L.ob[b8][m][row] = a.update ? o.W[m] : o.du[m];
          if (u == XD - 1 && (b8 == 7 || s == npad - 1)) {
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_s_waitcnt(0xc07f);  // the chunk's writes done before it is handed over
            lds_put(&L.ob_ready, ck + 1);
          }
        }
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        lds_put(&ch.prog[1], s + 1);
        if (u == XD - 2) {
          look();
          pv = lds_get(&L.filled[grp1]);
        }
      }
      lds_put(&ch.cons[0], st + XD);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      lds_put(&L.consumed, gs0 + st + XD);
      grp = grp1;
      round = round1;
    }
  };
  if (do_f) run_dir(std::true_type{}, 0);
  if (do_f && do_b) {
    // the forward sweep's stores before the producers' loads (see k_lusgs_fused)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    lds_put(&L.turned, 1);
  }
  if (do_b) run_dir(std::false_type{}, do_f ? npad : 0);
  }
}

// ----------------------------------------------------------------- scatter
template <int NV, bool VISC>
__global__ __launch_bounds__(256) void k_lusgs_scatter(LusgsArgs a) {
  using F = RecF<NV, VISC>;
  const BlockDesc B = a.blocks[a.block_list[blockIdx.y]];
  if (case_frozen(B.case_id)) return;
  const int ncol = B.nx - 1, nrow = B.ny - 1;
  // the tiles of k_lusgs_prep in the backward set's (step, row) space: eight
  // lanes read 8 consecutive output positions, a wave writes 8 cells of 8 rows
  const int S = B.sk_S;
  const int tiles_s = (S + 31) / 32;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int sb = (blockIdx.x % tiles_s) * 32 + wave * 8 + (lane >> 3);
  const int rb = (blockIdx.x / tiles_s) * 8 + (lane & 7);
  const int cb = sb - rb;
  if (sb >= S || rb >= nrow || cb < 0 || cb >= ncol) return;
  const int i = ncol - cb, j = nrow - rb;
  const int64_t n = B.sk_n;
  // the backward record of cell (i, j): position (ncol-i + nrow-j) * R + nrow-j
  const int64_t pos = (int64_t)sb * B.sk_R + rb;
  const double* out = a.sk + B.sk_base + 2 * F::NREC * n + 2 * pos;
  double* base = a.arena + B.base;
  const int64_t q = pidx(B, i, j);
#pragma unroll
  for (int m = 0; m < NV; m++) {
    const double du = out[(int64_t)(m / 2) * 2 * n + (m & 1)];
    base[(int64_t)(a.pm.dU + m) * B.plane + q] = du;
    if (a.update) {
      double* U = base + (int64_t)(a.pm.U + m) * B.plane;
      U[q] = U[q] + du;
    }
  }
}

}  // namespace ec2d
