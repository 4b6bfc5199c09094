// Fused residual kernel: Comput_Residual_one_mesh (sub_Residual.f90:13-107)
// for all blocks of a batch in one launch.
//
// One workgroup computes one TX x TY tile of cells of one block:
//   1. stage U of the tile plus a 2-cell halo from HBM into LDS and turn it
//      into primitives (comput_duvtpckw, sub_Residual.f90:114-152), Sutherland
//      viscosity (get_viscous, :670-689) and, for SA, nu_t
//      (sub_turbulence_SA.f90:24-36); the wall ghost override of Amut_boundary
//      (:180-220) is applied in LDS;
//   2. every i-face and j-face of the tile: reconstruction, rotation, flux,
//      back-rotation, viscous flux (Residual_FVM, :200-455) and the SA face
//      fluxes (sub_turbulence_SA.f90:43-115); results stay in LDS;
//   3. per cell: Res = Fi(i+1)-Fi(i)+Fj(j+1)-Fj(j) (:459-469), the SA
//      residual and source (sub_turbulence_SA.f90:77-168), spectral radii
//      (comput_Lvc, sub_NS_singlegrid.f90:352-388), local time step (comput_dt,
//      :324-348) and this tile's share of Res_max / sum(Res^2).
// HBM traffic per cell: U read once (+halo), Res, dt, Lci, Lcj (Lvi, Lvj)
// written once; faces shared by two tiles are recomputed, never re-read.
#include "ec2d_device.h"
#include "ec2d_physics.h"

namespace ec2d {

struct ResArgs {
  const TileDesc* tiles;
  const int* tile_perm;       // launch order -> logical tile
  const BlockDesc* blocks;
  const CaseParams* cps;
  double* arena;
  double* partials;           // [logical tile][2*NV]: max |Res|, sum Res^2
  unsigned long long* err;    // first cell with T < 1e-5 (block<<40 | j<<20 | i), ~0 if none
  int* cold;                  // per case, in per-case runs: set for a cell with T < 1e-5 (in place of err)
  MeshOpts o;
  PlaneMap pm;
  int clip;                   // apply force_vt_kw to interior nu_t on load
  double* sk_out;             // or null: the changing inputs of the fused LU-SGS in hyperplane order (the
                              // copy k_lusgs_skew makes), written here from the values the epilogue holds
  int sk_only;                // with sk_out: Res, dt, Lci, Lcj, Lvi, Lvj go to the hyperplane copy alone,
                              // not to their planes (k_lusgs_skew's reverse copy restores the planes)
  int write_visc;             // store Amu / Amu_t planes
  int force;                  // coarse multigrid levels, interior cells, variables 1..4, after the norms' values:
                              // 1: QF = QF - Res (comput_force_function), 2: Res = Res + QF (Add_force_function)
  int set_un;                 // also Un = U, variables 1..4, cells 0..nx x 0..ny (Set_Un)
  int closure;                // 1 (SA): take mu_t of interior cells from the closure planes where in range;
                              // 2 (4 equations): mu_t of every ring cell from the closure plane;
                              // 3 (4 equations, Baldwin-Lomax): mu_t of every ring cell from Amu_t as k_bl left it
};

// Small quotients k / D of thread indices without the 32-bit high multiply.
template <int D, int MAX>
__device__ __forceinline__ int div_small(int k) {
  constexpr int M = (65536 + D - 1) / D;
  static_assert((int64_t)(MAX - 1) * M < ((int64_t)1 << 24) && (int64_t)(MAX - 1) * (M * D - 65536) < 65536,
                "the quotient must be exact");
  return __mul24(k, M) >> 16;
}

// One step of the norms' tree over a wave: the sum (maximum) over lanes l and
// l ^ 32 (D = 32) or l ^ 16, of a in the lanes with that bit clear and of b in
// those with it set.
template <int D, class OP>
__device__ __forceinline__ double fold(double a, double b, OP op) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  auto swap = [](uint32_t u, uint32_t v) {
    if constexpr (D == 32) return __builtin_amdgcn_permlane32_swap(u, v, false, false);
    else return __builtin_amdgcn_permlane16_swap(u, v, false, false);
  };
  const auto lo = swap((uint32_t)x, (uint32_t)y), hi = swap((uint32_t)(x >> 32), (uint32_t)(y >> 32));
  return op(__builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]),
            __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]));
}
// the same over lanes l and l ^ 8, 4, 2, 1 by a lane move (after the step of 8 the
// values repeat every 8 lanes, so that a rotation by 4 is l ^ 4)
template <int CTRL, class OP>
__device__ __forceinline__ double fold_dpp(double a, OP op) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0u, (uint32_t)x, CTRL, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0u, (uint32_t)(x >> 32), CTRL, 0xf, 0xf, true);
  return op(a, __builtin_bit_cast(double, (uint64_t)hi << 32 | lo));
}
// N values over the wave in a butterfly's order (steps of 32, 16, ..., 1): value
// m ends in lanes 32 (m & 1) + 16 (m >> 1 & 1) .. + 15 of v[m >> 2].  The first two
// steps fold two values each, so that ten values take 80 instructions and no
// LDS (with a shuffle per step and value: 60 operations and 120 LDS permutes).
template <int N, class OP>
__device__ __forceinline__ void wave_fold(double (&v)[N], OP op) {
  constexpr int N2 = (N + 1) / 2, N4 = (N2 + 1) / 2;
#pragma unroll
  for (int m = 0; m < N2; m++) v[m] = fold<32>(v[2 * m], v[2 * m + 1 < N ? 2 * m + 1 : 2 * m], op);
#pragma unroll
  for (int m = 0; m < N4; m++) {
    double x = fold<16>(v[2 * m], v[2 * m + 1 < N2 ? 2 * m + 1 : 2 * m], op);
    x = fold_dpp<0x128>(x, op);  // row_ror:8
    x = fold_dpp<0x124>(x, op);  // row_ror:4
    x = fold_dpp<0x4e>(x, op);   // quad_perm [2, 3, 0, 1]
    v[m] = fold_dpp<0xb1>(x, op);  // quad_perm [1, 0, 3, 2]
  }
}

// One workgroup per tile of TX x TY cells, one thread per cell.  Instruction
// issue bounds large batches: of 256 SA blocks (3.1e6 cells, 32 x 8 tiles) a
// cell takes 2480 vector instructions, which keep the units busy 69% of 0.35
// ms; its loads and stores alone would take 0.17 ms.  (3284 instructions and
// 0.45 ms with the general divisions, square roots and pow, 64-bit addresses per
// access, a division of each thread index by the halo's width, LDS
// permutes in the norms, Amu / d formed by all users of a cell, and the faces beyond
// one per thread in a pass of their own per direction.)  Tried without gain:
// the next phase's loads ahead of the barrier (0.38 ms), the arguments by uniform
// loads in each phase (0.37 ms: their waits hold up the LDS), wider LDS rows.
//   waves_per_eu: 128 registers, so that the four workgroups that a CU's LDS
// holds do run.
//
// FIX: scheme, reconstruction and flux as compile-time constants, so that the
// compiler drops the other branches of every face; the launch picks it when the
// options match.  All with the original (primitive) reconstruction: MUSCL3 with the van
// Albada limiter in both directions and Roe's flux (1) or AUSM (2), and what a coarse
// level of a V-cycle makes of (1): first order over the i-faces (3).
//   FIX 0, any options: with every loop and reconstruction holding its own copy of
// all schemes and fluxes the code is 108 KB, more than the instruction cache.  Here
// one loop takes both directions in turn and the three reconstructions share the
// schemes (32 KB): 129 x 49 laminar cells with WENO3, HLLC and characteristic
// variables 34 -> 30 us.
template <int TX, int TY, int NV, bool VISC, bool SA, int FIX>
__global__ __launch_bounds__(TX* TY) __attribute__((amdgpu_waves_per_eu(FIX ? 4 : 3))) void k_residual(ResArgs a) {
  constexpr int RW = TX + 4, RH = TY + 4, NT = TX * TY;
  constexpr int CW = TX + 2, CH = TY + 2;  // the viscous quantities are used one cell out
  const int o_scheme = FIX == 3 ? 0 : FIX ? 5 : a.o.scheme, o_gscheme = FIX ? 5 : a.o.global_scheme;
  const int o_flux = FIX == 2 ? 6 : FIX ? 4 : a.o.flux, o_recon = FIX ? 0 : a.o.recon;
  // reciprocals of the constant divisors for div_y (x / Pr, x / Pr_t, x / sigma,
  // x / k^2, x / Ma): the reference's quotients in every comparison, but by trial and
  // not by a theorem, since a y need not be within an ulp of the quotient (1.2e9
  // numerators over 16 such divisors and random ones on the CPU: all correctly rounded)
  constexpr double yPrt = 1.0 / EC2D_PRT, ySig = 1.0 / (2.0 / 3.0), yK2 = 1.0 / (0.41 * 0.41);
  // viscous cases stage T and rebuild p = p00 d T from it (the staging's own
  // expression, so the same value); the cell centres of the viscous
  // gradients are read from their planes, not staged
  __shared__ double sd[RH][RW], su[RH][RW], sv[RH][RW], sp[VISC ? 1 : RH][VISC ? 1 : RW];
  __shared__ double sT[VISC ? RH : 1][VISC ? RW : 1];
  __shared__ double sAm[VISC ? CH : 1][VISC ? CW : 1], sAt[VISC ? CH : 1][VISC ? CW : 1];
  __shared__ double svt[SA ? CH : 1][SA ? CW : 1], snu[SA ? CH : 1][SA ? CW : 1];  // snu: Amu / d
  // face fluxes (SA: two more each): the i-faces' sFi and, after every cell
  // has taken its i-face difference, the j-faces' rows in the same LDS, so
  // that four workgroups of a 32 x 8 SA tile fit on a CU.  The last row of
  // j-faces lies behind sFi: it is made together with the last column of i-faces.
  // (Row pitch TX + 2: the cells of a hyperplane, TY lanes one row and one column
  // apart, read different banks.)
  constexpr int NC = SA ? 6 : 4, NIF = NC * TY * (TX + 2);
  __shared__ double sF[NIF + NC * TX];
  auto& sFi = *reinterpret_cast<double(*)[NC][TY][TX + 2]>(sF);
  auto& sFj = *reinterpret_cast<double(*)[TY + 1][NC][TX]>(sF + 2 * NC * TY);
  __shared__ double sred[2 * NV][NT / 64];

  const int lt = a.tile_perm[blockIdx.x];
  const TileDesc t = a.tiles[lt];
  const BlockDesc B = a.blocks[t.block];
  if (case_frozen(B.case_id)) return;
  const CaseParams cp = a.cps[B.case_id];
  const PlaneMap pm = a.pm;
  const int nx = B.nx, ny = B.ny;
  const double g = cp.gamma;
  double* base = a.arena + B.base;
  // a plane's base is uniform; the place in it is a 32-bit byte offset (a plane
  // has less than 4 GiB), shared by all planes
  int64_t plane = B.plane;
  auto PL = [&](int slot) { return base + (int64_t)slot * plane; };
  // planes' addresses are formed again in each phase: kept through all of them
  // they fill the scalar registers, and each spill takes vector instructions
  auto fresh = [&] { asm volatile("" : "+s"(plane)); };
  auto off = [&](int i, int j) { return ((uint32_t)(j + 1) * (uint32_t)B.P + (uint32_t)(i + 1)) * 8u; };
  auto at = [](double* plane, uint32_t q8) -> double& {
    return *reinterpret_cast<double*>(reinterpret_cast<char*>(plane) + q8);
  };
  const int tid = threadIdx.x;
  const int i0 = t.i0, j0 = t.j0;

  // ---- 1. stage tile + halo ------------------------------------------------
  struct Cell {
    int li, lj, i, j;
    uint32_t q8;
    double u[4 + (SA ? 1 : 0)];
  };
  auto load = [&](Cell& c, int idx) {
    c.lj = div_small<RW, 2 * RW * RH>(idx);
    c.li = idx - __mul24(c.lj, RW);
    c.i = i0 - 2 + c.li;
    c.j = j0 - 2 + c.lj;
    if (c.lj >= RH || c.i < -1 || c.i > nx + 1 || c.j < -1 || c.j > ny + 1) return false;
    c.q8 = off(c.i, c.j);
#pragma unroll
    for (int m = 0; m < 4 + (SA ? 1 : 0); m++) c.u[m] = at(PL(pm.U + m), c.q8);
    return true;
  };
  auto stage = [&](const Cell& c) {
    const int li = c.li, lj = c.lj, i = c.i, j = c.j;
    const uint32_t q8 = c.q8;
    const double d = c.u[0], u1 = c.u[1], u2 = c.u[2], u3 = c.u[3];
    const double yd = rcp_n(d);
    double uu = div_y(u1, d, yd);
    double vv = div_y(u2, d, yd);
    double T = div_n(u3 - 0.5 * d * (uu * uu + vv * vv), cp.Cv * d);
    if (T != T) {  // out of div_n's range: an energy of minus infinity is a cold cell, as for the reference
      uu = u1 / d;
      vv = u2 / d;
      T = (u3 - 0.5 * d * (uu * uu + vv * vv)) / (cp.Cv * d);
    }
    sd[lj][li] = d;
    su[lj][li] = uu;
    sv[lj][li] = vv;
    if constexpr (!VISC) sp[lj][li] = cp.p00 * d * T;
    bool interior = (i >= 1 && i <= nx - 1 && j >= 1 && j <= ny - 1);
    if (interior && T < 1.0e-5) {
      if (a.cold) {
        atomicOr(a.cold + B.case_id, 1);
      } else {
        unsigned long long key = ((unsigned long long)t.block << 40) | ((unsigned long long)j << 20) | (unsigned)i;
        atomicMin(a.err, key);
      }
    }
    if constexpr (VISC) {
      sT[lj][li] = T;
      if (li < 1 || li > RW - 2 || lj < 1 || lj > RH - 2) return;
      const int lc = lj - 1, lr = li - 1;
      bool ring = (i >= 0 && i <= nx && j >= 0 && j <= ny);
      double am = 0.0;
      if (ring) {
        am = div_n(cp.c_am * sqrt_n(T * T * T), cp.Tsb + T);
        if (am != am) am = cp.c_am * sqrt(T * T * T) / (cp.Tsb + T);
      }
      // SST: the model scaled interior Amu by Re and back (sub_turbulence_SST.f90:85, 259)
      if constexpr (NV == 6) {
        if (interior) am = (am * cp.Re) / cp.Re;
      }
      sAm[lc][lr] = am;
      double at_ = 0.0;
      if constexpr (SA) {
        double vt = c.u[SA ? 4 : 0];
        if (a.clip && interior && vt < 0) {
          vt = 1.0e-10;
          at(PL(pm.U + 4), q8) = vt;
        }
        svt[lc][lr] = vt;
        snu[lc][lr] = div_y(am, d, yd);
        if (ring) {
          const double Cv1_3 = 7.1 * 7.1 * 7.1;
          double X = div_n(d * vt, am);
          double X3 = X * X * X;
          double fv1 = div_n(X3, X3 + Cv1_3);
          at_ = fv1 * d * vt;
        }
        if (a.closure && interior && at(PL(pm.clo + 1), q8) != 0.0) at_ = at(PL(pm.clo), q8);
      }
      // SST: mu_t as the model left it (interior and wall ghosts set by
      // k_sst_res, other ghosts untouched)
      if constexpr (NV == 6) at_ = ring ? at(PL(pm.Amu_t), q8) : 0.0;
      // the learned closure as the eddy-viscosity model
      if constexpr (NV == 4) {
        if (a.closure == 2 && ring) at_ = at(PL(pm.clo), q8);
        // Baldwin-Lomax (k_bl wrote every cell, ghosts included, by its own rules)
        if (a.closure == 3 && ring) at_ = at(PL(pm.Amu_t), q8);
      }
      sAt[lc][lr] = at_;
    }
  };
  // two cells' loads at a time
  for (int idx = tid; idx < RW * RH; idx += 2 * NT) {
    Cell c0, c1;
    const bool in0 = load(c0, idx), in1 = load(c1, idx + NT);
    if (in0) stage(c0);
    if (in1) stage(c1);
  }
  __syncthreads();
  // tiles with a ghost cell of the block in the ring
  const bool rim = i0 == 1 || j0 == 1 || i0 + TX > nx - 1 || j0 + TY > ny - 1;
  if (rim && (SA || (NV == 4 && VISC && a.closure == 2))) {
    // Amut_boundary: wall ghost cells of layer 0 take -Amu_t of the adjacent interior cell
    // (sub_turbulence_SA.f90:200-216; the closure's mu_t follows the same rule)
    double* flag = PL(pm.flag);
    for (int idx = tid; idx < CW * CH; idx += NT) {
      const int lj = div_small<CW, CW * CH>(idx), li = idx - lj * CW;
      int i = i0 - 1 + li, j = j0 - 1 + lj;
      if (i < 0 || i > nx || j < 0 || j > ny) continue;
      bool gi = (i == 0 || i == nx) && j >= 1 && j <= ny - 1;
      bool gj = (j == 0 || j == ny) && i >= 1 && i <= nx - 1;
      if (!(gi || gj)) continue;
      if (at(flag, off(i, j)) == 0.0) continue;
      int ii = li, jj = lj;
      if (i == 0 && gi) ii = li + 1;
      else if (gi) ii = li - 1;
      else if (j == 0) jj = lj + 1;
      else jj = lj - 1;
      sAt[lj][li] = -sAt[jj][ii];
    }
    __syncthreads();
  }

  const bool fdm = B.fdm != 0;
  const int LF = 4;
  fresh();
  // ---- 2. the flux through one face: the i-face (jd false) between cells
  // (i-1, j) and (i, j) or the j-face between (i, j-1) and (i, j), (i, j) the
  // tile's cell (fi, fj).  The reference's two loops (sub_Residual.f90:193-455) are
  // the same expressions with the directions exchanged: `back` is the step to the
  // face's other cell, `side` the step along the face.  Of the gradients,
  // exchanging i and j turns the sign of both factors of each product with
  // Ds, which leaves the same bits.  The one sum whose order differs picks it.
  auto face = [&](auto jd, int fi, int fj, double* F) {
    const bool J = jd;
    const int i = i0 + fi, j = j0 + fj;
    if (i > (J ? nx - 1 : nx) || j > (J ? ny : ny - 1)) return false;
    // faces of the finite-difference interior carry no FVM flux, but the SA
    // model's own face loops (sub_turbulence_SA.f90:43-73) cover every face
    const bool skip_fvm = fdm && (i >= LF + 2 && i <= nx - LF - 1) && (j >= LF + 2 && j <= ny - LF - 1);
    if (skip_fvm && !SA) return false;
    const uint32_t q8 = off(i, j);
    const double sl = at(J ? PL(pm.sj) : PL(pm.si), q8), n1 = at(J ? PL(pm.nj1) : PL(pm.ni1), q8),
                 n2 = at(J ? PL(pm.nj2) : PL(pm.ni2), q8);
    // of the cell centres: the difference across the face, and along it that of the
    // mean of its two cells
    double Nx, Ny, Cx, Cy;
    if constexpr (VISC) {
      const uint32_t b8 = J ? (uint32_t)B.P * 8u : 8u, s8 = J ? 8u : (uint32_t)B.P * 8u;
      double *X = PL(pm.x1), *Y = PL(pm.y1);
      Nx = at(X, q8) - at(X, q8 - b8);
      Ny = at(Y, q8) - at(Y, q8 - b8);
      Cx = (at(X, q8 + s8 - b8) + at(X, q8 + s8) - at(X, q8 - b8 - s8) - at(X, q8 - s8)) * 0.25;
      Cy = (at(Y, q8 + s8 - b8) + at(Y, q8 + s8) - at(Y, q8 - b8 - s8) - at(Y, q8 - s8)) * 0.25;
    }
    const int o = __mul24(fj + 2, RW) + fi + 2, back = J ? RW : 1, side = J ? 1 : RW;
    const double *d_ = &sd[0][0] + o, *u_ = &su[0][0] + o, *v_ = &sv[0][0] + o;
    double UL[4], UR[4];
    double F1 = 0.0, F2 = 0.0, F3 = 0.0, F4 = 0.0;
    if (!skip_fvm) {
      double W[4][4], S1[4][4];  // cells -2 back .. back: the variables to reconstruct
      if (o_recon == 0) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int at_ = (k - 2) * back;
          W[k][0] = d_[at_];
          W[k][1] = u_[at_];
          W[k][2] = v_[at_];
          if constexpr (VISC) W[k][3] = cp.p00 * d_[at_] * (&sT[0][0] + o)[at_];
          else W[k][3] = (&sp[0][0] + o)[at_];
        }
      } else {
        double U0[4][4];
        for (int k = 0; k < 4; k++) {
          const uint32_t qk = J ? off(i, j - 2 + k) : off(i - 2 + k, j);
          for (int m = 0; m < 4; m++) U0[k][m] = at(PL(pm.U + m), qk);
        }
        if (o_recon == 1) {
          for (int k = 0; k < 4; k++)
            for (int m = 0; m < 4; m++) W[k][m] = U0[k][m];
        } else {
          to_char(U0, W, S1, g);
        }
      }
      // the j-direction original-variable reconstruction uses the global
      // scheme option, not the mesh's own (sub_Residual.f90:367)
      const int sch = J && o_recon == 0 ? o_gscheme : o_scheme;
      double VL[4], VR[4];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        VL[m] = scheme_fP(W[0][m], W[1][m], W[2][m], W[3][m], sch);
        VR[m] = scheme_fm(W[0][m], W[1][m], W[2][m], W[3][m], sch);
      }
      if (o_recon == 0) {
        for (int m = 0; m < 4; m++) UL[m] = VL[m], UR[m] = VR[m];
      } else if (o_recon == 1) {
        cons_to_prim(VL, UL, g);
        cons_to_prim(VR, UR, g);
      } else {
        char_to_prim(VL, S1, UL, g);
        char_to_prim(VR, S1, UR, g);
      }
      double QL[4], QR[4], F0[4];
      QL[0] = UL[0]; QL[1] = UL[1] * n1 + UL[2] * n2; QL[2] = -UL[1] * n2 + UL[2] * n1; QL[3] = UL[3];
      QR[0] = UR[0]; QR[1] = UR[1] * n1 + UR[2] * n2; QR[2] = -UR[1] * n2 + UR[2] * n1; QR[3] = UR[3];
      face_flux(o_flux, QL, QR, F0, g);
      F1 = -F0[0] * sl;
      F2 = -(F0[1] * n1 - F0[2] * n2) * sl;
      F3 = -(F0[1] * n2 + F0[2] * n1) * sl;
      F4 = -F0[3] * sl;
    }
    if constexpr (VISC) {
      const int oc = __mul24(fj + 1, CW) + fi + 1, cback = J ? CW : 1, cside = J ? 1 : CW;
      const double *Am = &sAm[0][0] + oc, *At = &sAt[0][0] + oc, *T_ = &sT[0][0] + o;
      const int e = J ? j : i, n = J ? ny : nx;
      double am0 = Am[0], amb = Am[-cback], at0 = At[0], atb = At[-cback];
      double Amu1, Amk1;
      if (e == 1 || e == n) {  // the inner cell's alone
        const double am = e == 1 ? am0 : amb, at_ = e == 1 ? at0 : atb;
        Amu1 = am + at_;
        Amk1 = cp.Cp * (div_y(am, cp.Pr, cp.yPr) + div_y(at_, EC2D_PRT, yPrt));
      } else {
        Amu1 = ((amb + am0) + (J ? at0 : atb) + (J ? atb : at0)) * 0.5;
        Amk1 = cp.Cp * (div_y(amb + am0, cp.Pr, cp.yPr) + div_y(atb + at0, EC2D_PRT, yPrt)) * 0.5;
      }
      auto across = [&](const double* w) { return w[0] - w[-back]; };
      auto along = [&](const double* w) { return (w[side - back] + w[side] - w[-back - side] - w[-side]) * 0.25; };
      const double Ds = rcp_rn(Nx * Cy - Cx * Ny);
      const double Nu = across(u_), Nw = across(v_), NT_ = across(T_);
      const double Cu = along(u_), Cw = along(v_), CT = along(T_);
      double ux = (Nu * Cy - Cu * Ny) * Ds, vx = (Nw * Cy - Cw * Ny) * Ds, Tx = (NT_ * Cy - CT * Ny) * Ds;
      double uy = (-Nu * Cx + Cu * Nx) * Ds, vy = (-Nw * Cx + Cw * Nx) * Ds, Ty = (-NT_ * Cx + CT * Nx) * Ds;
      double u1 = (u_[0] + u_[-back]) * 0.5;
      double v1 = (v_[0] + v_[-back]) * 0.5;
      double t11 = ((4.0 / 3.0) * ux - (2.0 / 3.0) * vy) * Amu1;
      double t22 = ((4.0 / 3.0) * vy - (2.0 / 3.0) * ux) * Amu1;
      double t12 = (uy + vx) * Amu1;
      double E1 = u1 * t11 + v1 * t12 + Amk1 * Tx;
      double E2 = u1 * t12 + v1 * t22 + Amk1 * Ty;
      if (!skip_fvm) {
        F2 = F2 + (t11 * n1 + t12 * n2) * sl;
        F3 = F3 + (t12 * n1 + t22 * n2) * sl;
        F4 = F4 + (E1 * n1 + E2 * n2) * sl;
      }
      if constexpr (SA) {
        const double Cb2 = 0.622, SA_sigma = 2.0 / 3.0;
        const double c_diff = 0.5 * (1.0 + Cb2) / SA_sigma;
        const double *vt = &svt[0][0] + oc, *nu = &snu[0][0] + oc;
        double vn1 = u_[-back] * n1 + v_[-back] * n2;
        double vn2 = u_[0] * n1 + v_[0] * n2;
        double vfi = -0.5 * ((vn1 + fabs(vn1)) * vt[-cback] + (vn2 - fabs(vn2)) * vt[0]) * sl;
        double v0 = c_diff * (vt[0] + nu[0] + vt[-cback] + nu[-cback]);
        double Nv = vt[0] - vt[-cback];
        double Cv = (vt[cside - cback] + vt[cside] - vt[-cback - cside] - vt[-cside]) * 0.25;
        double vtx = (Nv * Cy - Cv * Ny) * Ds;
        double vty = (-Nv * Cx + Cv * Nx) * Ds;
        F[4] = vfi + v0 * (vtx * n1 + vty * n2) * sl;
        F[5] = (vtx * n1 + vty * n2) * sl;
      }
    }
    F[0] = F1;
    F[1] = F2;
    F[2] = F3;
    F[3] = F4;
    return true;
  };
  auto put_i = [&](int fi, int fj, const double* F) {
#pragma unroll
    for (int m = 0; m < NC; m++) sFi[m][fj][fi] = F[m];
  };
  auto put_j = [&](int fi, int fj, const double* F) {
#pragma unroll
    for (int m = 0; m < NC; m++) sFj[fj][m][fi] = F[m];
  };
  // The cell of this thread in phases 3a and 3: row-major, or, when the
  // epilogue also writes the hyperplane-order copy (sk_out), along the
  // tile's hyperplanes: TY consecutive lanes take the TY rows of one
  // hyperplane, so that the copy's stores form runs of TY positions.
  const int kd = tid / TY, cjd = tid % TY;
  const int ci = a.sk_out ? (kd - cjd + TX) % TX : tid % TX;
  const int cj = a.sk_out ? cjd : tid / TX;
  const int i = i0 + ci, j = j0 + cj;
  const bool mine = i <= nx - 1 && j <= ny - 1;
  const bool fdm_cell = fdm && (i >= LF + 1 && i <= nx - LF - 1) && (j >= LF + 1 && j <= ny - LF - 1);

  // ---- 3a. each cell's i-face difference (the first terms of Res, in the
  // reference's order), before the j-faces take over the LDS --------------
  double R[NV];
  double r5 = 0.0, v0c = 0.0;  // SA: the cell's v0 of sub_turbulence_SA.f90, kept for phase 3
  auto i_diff = [&] {
    if (mine) {
      if (!fdm_cell) {
  #pragma unroll
        for (int m = 0; m < 4; m++) R[m] = sFi[m][cj][ci + 1] - sFi[m][cj][ci];
      }
      if constexpr (SA) {
        const double SA_sigma = 2.0 / 3.0, Cb2 = 0.622;
        v0c = div_y((svt[cj + 1][ci + 1] + snu[cj + 1][ci + 1]) * Cb2, SA_sigma, ySig);
        r5 = sFi[NC - 2][cj][ci + 1] - sFi[NC - 2][cj][ci] - v0c * (sFi[NC - 1][cj][ci + 1] - sFi[NC - 1][cj][ci]);
      }
    }
  };
  // ---- 2a. i-faces, one per thread, and the TY of the last column; 2b. j-faces
  // and the TX of the last row
  if constexpr (FIX != 0) {
    // one wave takes both remainders in one pass
    for (int f = tid; f < NT + TY + TX; f += NT) {
      double F[6] = {};
      const int x = f - NT;
      const bool J = x >= TY;
      const int fi = x < 0 ? f % TX : J ? x - TY : TX, fj = x < 0 ? f / TX : J ? TY : x;
      if (!face(J, fi, fj, F)) continue;
      if (J) put_j(fi, fj, F);
      else put_i(fi, fj, F);
    }
    __syncthreads();
    fresh();
    i_diff();
    __syncthreads();
    double F[6] = {};
    if (face(std::true_type{}, tid % TX, tid / TX, F)) put_j(tid % TX, tid / TX, F);
    __syncthreads();
  } else {
#pragma unroll 1
    for (int dir = 0; dir < 2; dir++) {
      const bool J = dir != 0;
      for (int f = tid; f < NT + (J ? TX : TY); f += NT) {
        double F[6] = {};
        const int x = f - NT;
        const int fi = x < 0 ? f % TX : J ? x : TX, fj = x < 0 ? f / TX : J ? TY : x;
        if (!face(J, fi, fj, F)) continue;
        if (J) put_j(fi, fj, F);
        else put_i(fi, fj, F);
      }
      __syncthreads();
      if (!J) {
        i_diff();
        __syncthreads();
      }
    }
  }
  fresh();
  // ---- 3. cells ------------------------------------------------------------
  double rmax[NV], rsum[NV];
#pragma unroll
  for (int m = 0; m < NV; m++) { rmax[m] = 0.0; rsum[m] = 0.0; }
  if (mine) {
    const uint32_t q8 = off(i, j), P8 = (uint32_t)B.P * 8u;
    const int li = ci + 2, lj = cj + 2, cr = ci + 1, cc_ = cj + 1;
    const double d = sd[lj][li];
    if (!fdm_cell) {
#pragma unroll
      for (int m = 0; m < 4; m++) R[m] = R[m] + sFj[cj + 1][m][ci] - sFj[cj][m][ci];
    }
    if constexpr (SA) {
      const double SA_sigma = 2.0 / 3.0, Cv1 = 7.1, Cb1 = 0.1355, Cb2 = 0.622, SA_k = 0.41;
      const double Cw1 = Cb1 / (SA_k * SA_k) + (1.0 + Cb2) / SA_sigma, Cw2 = 0.3, Ct3 = 1.3, Ct4 = 0.5;
      const double Cv1_3 = Cv1 * Cv1 * Cv1, Cw3_6 = 2.0 * 2.0 * 2.0 * 2.0 * 2.0 * 2.0;
      double vtc = svt[cc_][cr];
      const double v0 = v0c;
      r5 = r5 + sFj[cj + 1][NC - 2][ci] - sFj[cj][NC - 2][ci] - v0 * (sFj[cj + 1][NC - 1][ci] - sFj[cj][NC - 1][ci]);
      double *X1 = PL(pm.x1), *Y1 = PL(pm.y1);
      double Dix = (at(X1, q8 + 8u) - at(X1, q8 - 8u)) * 0.5;
      double Diy = (at(Y1, q8 + 8u) - at(Y1, q8 - 8u)) * 0.5;
      double Djx = (at(X1, q8 + P8) - at(X1, q8 - P8)) * 0.5;
      double Djy = (at(Y1, q8 + P8) - at(Y1, q8 - P8)) * 0.5;
      double Ds = rcp_rn(Dix * Djy - Djx * Diy);
      double Diu = (su[lj][li + 1] - su[lj][li - 1]) * 0.5;
      double Div = (sv[lj][li + 1] - sv[lj][li - 1]) * 0.5;
      double Dju = (su[lj + 1][li] - su[lj - 1][li]) * 0.5;
      double Djv = (sv[lj + 1][li] - sv[lj - 1][li]) * 0.5;
      double vx = (Div * Djy - Djv * Diy) * Ds;
      double uy = (-Diu * Djx + Dju * Dix) * Ds;
      double S = fabs(vx - uy);
      double dwc = at(PL(pm.dw), q8);
      double X = div_n(d * vtc, sAm[cc_][cr]);
      double X3 = X * X * X;
      double fv1 = div_n(X3, X3 + Cv1_3);
      double fv2 = 1.0 - div_n(X, 1.0 + X * fv1);
      double kd_ = SA_k * dwc;
      double Sd = div_n(fv2 * vtc, kd_ * kd_);
      if (Sd != Sd) Sd = fv2 * vtc / (kd_ * kd_);  // (fmax would drop a NaN: a wall distance whose square overflows)
      double S1 = fmax(S + Sd, EC2D_SP(0.3) * S);
      // S1 is zero in a uniform stream: the full division, whose infinity becomes 10
      double r = fmin(vtc / (S1 * SA_k * SA_k * dwc * dwc), 10.0);
      double gg = r + Cw2 * (r * r * r * r * r * r - r);
      // r has no lower bound (nu_t < 0 inside a Runge-Kutta pass): g^6 beyond
      // pow_sixth's range, up to overflow, takes the general functions
      const double g6 = gg * gg * gg * gg * gg * gg;
      double fw;
      if (g6 < 1.0e37) fw = gg * pow_sixth(div_n(1.0 + Cw3_6, g6 + Cw3_6));
      else fw = gg * pow((1.0 + Cw3_6) / (g6 + Cw3_6), 1.0 / 6.0);
      double ft2 = Ct3 * exp(-(Ct4 * X * X));
      double qv = div_n(vtc, dwc);
      double Q_SA = Cb1 * (1.0 - ft2) * S1 * vtc - (Cw1 * fw - div_y(Cb1 * ft2, SA_k * SA_k, yK2)) * (qv * qv);
      r5 = r5 + Q_SA * at(PL(pm.vol), q8);
      R[4] = r5;
    }
    double Rs[NV];  // Res as stored (with the forcing function on coarse levels)
    if (!fdm_cell) {
#pragma unroll
      for (int m = 0; m < 4; m++) {
        double r = R[m];
        if (a.force == 1) at(PL(pm.QF + m), q8) = at(PL(pm.QF + m), q8) - r;
        else if (a.force == 2) r = r + at(PL(pm.QF + m), q8);
        if (!a.sk_only) at(PL(pm.Res + m), q8) = r;
        Rs[m] = r;
      }
    }
    if constexpr (SA) {
      if (!a.sk_only) at(PL(pm.Res + 4), q8) = R[4];
    }
    if constexpr (NV == 6) {
      // Res(5:6) came from k_sst_res; read for the norms
      R[4] = at(PL(pm.Res + 4), q8);
      R[5] = at(PL(pm.Res + 5), q8);
    }
#pragma unroll
    for (int m = 4; m < NV; m++) Rs[m] = R[m];
    // comput_Lvc
    const uint32_t qi1 = q8 + 8u, qj1 = q8 + P8;
    double s0 = at(PL(pm.vol), q8);
    double si = 0.5 * (at(PL(pm.si), q8) + at(PL(pm.si), qi1));
    double ni1 = 0.5 * (at(PL(pm.ni1), q8) + at(PL(pm.ni1), qi1));
    double ni2 = 0.5 * (at(PL(pm.ni2), q8) + at(PL(pm.ni2), qi1));
    double sj = 0.5 * (at(PL(pm.sj), q8) + at(PL(pm.sj), qj1));
    double nj1 = 0.5 * (at(PL(pm.nj1), q8) + at(PL(pm.nj1), qj1));
    double nj2 = 0.5 * (at(PL(pm.nj2), q8) + at(PL(pm.nj2), qj1));
    double uni = su[lj][li] * ni1 + sv[lj][li] * ni2;
    double unj = su[lj][li] * nj1 + sv[lj][li] * nj2;
    double T;
    if constexpr (VISC) {
      T = sT[lj][li];
    } else {
      const double e = at(PL(pm.U + 3), q8) - 0.5 * d * (su[lj][li] * su[lj][li] + sv[lj][li] * sv[lj][li]);
      T = div_n(e, cp.Cv * d);
      if (T != T) T = e / (cp.Cv * d);
    }
    double cc = div_y(sqrt_n(T), cp.Ma, cp.yMa);
    if (cc != cc) cc = sqrt(T) / cp.Ma;
    double Lci = (fabs(uni) + cc) * si;
    double Lcj = (fabs(unj) + cc) * sj;
    double Lvi = 0.0, Lvj = 0.0;
    if constexpr (VISC) {
      double tmp1 = div_n(g, d) * (div_y(sAm[cc_][cr], cp.Pr, cp.yPr) + div_y(sAt[cc_][cr], EC2D_PRT, yPrt));
      const double y0 = rcp_n(s0);
      Lvi = div_y(tmp1 * si * si, s0, y0);
      Lvj = div_y(tmp1 * sj * sj, s0, y0);
      if (Lvi + Lvj != Lvi + Lvj) {
        tmp1 = g / d * (sAm[cc_][cr] / cp.Pr + sAt[cc_][cr] / EC2D_PRT);
        Lvi = tmp1 * si * si / s0;
        Lvj = tmp1 * sj * sj / s0;
      }
    }
    if (!a.sk_only) {
      if constexpr (VISC) {
        at(PL(pm.Lvi), q8) = Lvi;
        at(PL(pm.Lvj), q8) = Lvj;
      }
      at(PL(pm.Lci), q8) = Lci;
      at(PL(pm.Lcj), q8) = Lcj;
    }
    double dt;
    if (cp.Iflag_local_dt == 0) {
      dt = cp.dt_global;
    } else {
      dt = div_n(cp.CFL * s0, Lci + Lcj + 1.0 * (Lvi + Lvj));
      if (dt != dt) dt = cp.CFL * s0 / (Lci + Lcj + 1.0 * (Lvi + Lvj));
      if (dt > cp.dtmax) dt = cp.dtmax;
      if (dt < cp.dtmin) dt = cp.dtmin;
    }
    if (!a.sk_only) at(PL(pm.dt), q8) = dt;
    if (a.sk_out) {
      // logical plane k of cell (i, j) at k n + (i-1 + j-1) R + j-1 (the
      // layout of k_lusgs_skew): U (nu_t as clipped in the staging), Res,
      // dt, Lci, Lcj and, viscous, Lvi, Lvj
      using I = RecIn;
      const int64_t n = B.sk_n;
      double* so = a.sk_out + B.sk_base;
      const uint32_t p8 = (uint32_t)((i - 1 + j - 1) * B.sk_R + (j - 1)) * 8u;
#pragma unroll
      for (int m = 0; m < NV; m++) {
        double u;
        if (m == 0) u = d;
        else if (SA && m == 4) u = svt[cc_][cr];
        else u = at(PL(pm.U + m), q8);
        at(so + (I::U + m) * n, p8) = u;
        at(so + (I::RES<NV> + m) * n, p8) = Rs[m];
      }
      at(so + I::DT<NV> * n, p8) = dt;
      at(so + I::LCI<NV> * n, p8) = Lci;
      at(so + I::LCJ<NV> * n, p8) = Lcj;
      if constexpr (VISC) {
        at(so + I::LVI<NV> * n, p8) = Lvi;
        at(so + I::LVJ<NV> * n, p8) = Lvj;
      }
    }
    if (!fdm_cell) {
#pragma unroll
      for (int m = 0; m < NV; m++) {
        rmax[m] = fabs(R[m]);
        rsum[m] = R[m] * R[m];
      }
    } else {
#pragma unroll
      for (int m = 4; m < NV; m++) {
        rmax[m] = fabs(R[m]);
        rsum[m] = R[m] * R[m];
      }
    }
    if constexpr (VISC) {
      if (a.write_visc) {
        at(PL(pm.Amu), q8) = sAm[cc_][cr];
        at(PL(pm.Amu_t), q8) = sAt[cc_][cr];
      }
    }
  }
  // the cells (i, j) of the block and its first ghost layer (its corners
  // included) that belong to this tile, a ghost cell to the tile that holds
  // the interior cell next to it (its indices clamped to 1..nx-1, 1..ny-1)
  auto each_own = [&](auto&& f) {
    for (int idx = tid; idx < CW * CH; idx += NT) {
      const int lj = div_small<CW, CW * CH>(idx), li = idx - lj * CW;
      const int i = i0 - 1 + li, j = j0 - 1 + lj;
      if (i < 0 || i > nx || j < 0 || j > ny) continue;
      int ci = min(max(i, 1), nx - 1), cj = min(max(j, 1), ny - 1);
      if (ci < i0 || ci >= i0 + TX || cj < j0 || cj >= j0 + TY) continue;
      f(i, j, lj, li);
    }
  };
  if constexpr (VISC) {
    // mu_t of the first ghost layer (i = 0 or nx, j = 0 or ny, corners
    // included), as the reference's array holds it after Amut_boundary; the
    // output files carry it.  SST and Baldwin-Lomax read these cells from the
    // plane above: the store writes back the value read.
    if (a.write_visc && rim)
      each_own([&](int i, int j, int lj, int li) {
        if (i == 0 || i == nx || j == 0 || j == ny) at(PL(pm.Amu_t), off(i, j)) = sAt[lj][li];
      });
  }
  if (a.set_un) {
    // Set_Un over the cells and the first ghost layer
    each_own([&](int i, int j, int, int) {
      const uint32_t q8 = off(i, j);
#pragma unroll
      for (int m = 0; m < 4; m++) at(PL(pm.Un + m), q8) = at(PL(pm.U + m), q8);
    });
  }
  // ---- tile reduction (fixed tree: wave butterfly, then waves in order) ----
  wave_fold(rmax, [](double x, double y) { return fmax(x, y); });
  wave_fold(rsum, [](double x, double y) { return x + y; });
  const int lane = tid & 63;
  if ((lane & 15) == 0) {
    const int m0 = (lane >> 5) + (lane >> 4 & 1) * 2;  // lanes 0, 32, 16, 48: values 0, 1, 2, 3
#pragma unroll
    for (int k = 0; k < (NV + 3) / 4; k++) {
      if (4 * k + m0 < NV) {
        sred[2 * (4 * k + m0)][tid >> 6] = rmax[k];
        sred[2 * (4 * k + m0) + 1][tid >> 6] = rsum[k];
      }
    }
  }
  __syncthreads();
  if (tid < 2 * NV) {
    double acc = sred[tid][0];
    for (int w = 1; w < NT / 64; w++) acc = (tid & 1) ? acc + sred[tid][w] : fmax(acc, sred[tid][w]);
    a.partials[(int64_t)lt * 2 * NV + tid] = acc;
  }
}

// Deterministic second stage: one workgroup per case reduces its tiles in
// logical order into Res_max(1:NV) and Res_rms(1:NV) = sqrt(sum/Num_Cell).
template <int NV>
__global__ __launch_bounds__(256) void k_norms(const double* partials, const int* case_tile0, const double* ncell,
                                               double* norms, Mail* mail, int mail_case,
                                               const unsigned long long* derr, const int* sweep_err) {
  const int c = blockIdx.x, t0 = case_tile0[c], t1 = case_tile0[c + 1];
  __shared__ double sh[2 * NV][256];
  double acc[2 * NV] = {};
  for (int t = t0 + threadIdx.x; t < t1; t += 256) {
#pragma unroll
    for (int k = 0; k < 2 * NV; k++) {
      const double v = partials[(int64_t)t * 2 * NV + k];
      acc[k] = k & 1 ? acc[k] + v : fmax(acc[k], v);
    }
  }
#pragma unroll
  for (int k = 0; k < 2 * NV; k++) sh[k][threadIdx.x] = acc[k];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  for (int k = threadIdx.x >> 6; k < 2 * NV; k += 4) {
    const bool is_sum = k & 1;
    auto op = [&](double a, double b) { return is_sum ? a + b : fmax(a, b); };
    double v = op(op(sh[k][lane], sh[k][lane + 128]), op(sh[k][lane + 64], sh[k][lane + 192]));
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v = op(v, __shfl_down(v, s));
    if (lane == 0) {
      const int m = k >> 1;
      v = is_sum ? sqrt(v / ncell[c]) : v;
      const int at = is_sum ? 6 + m : m;
      norms[c * 12 + at] = v;
      if (mail && c == mail_case) mail->norms[at] = v;
    }
  }
  if (!mail || c != mail_case) return;
  const int m = threadIdx.x % 6;
  if (threadIdx.x < 12 && m >= NV) mail->norms[threadIdx.x] = norms[c * 12 + threadIdx.x];
  if (threadIdx.x == 0) mail_errors(mail, derr, sweep_err);
}

}  // namespace ec2d

// Run to a residual drop (ec2d_run_to_drop): after the first fine-level
// residual of every main-loop pass, one workgroup per case reduces the
// density's per-tile sums of Res^2 as k_norms does (the same order, so the
// value equals Res_rms(1) of ec2d_res_norms) and decides whether the case
// goes on.  The first check of a run records the reference value r0.  A case
// stops (active = 0, its blocks frozen by every later kernel) when its rms
// falls to drop * r0 (status 1), when the rms of any of its equations is not
// finite (status 2: the NaN guard), or
// has been checked max_iter times (status 3).  iters counts the checks, i.e.
// the residual evaluations of the case's state; the state it stops in has had
// iters - 1 updates in this run.
struct ConvState {
  double r0, last;
  int iters, status;
};

__global__ __launch_bounds__(256) void k_converge(const double* partials, const int* case_tile0, const double* ncell,
                                                  int nv, int* active, ConvState* st, double drop, int max_iter,
                                                  const int* cold) {
  const int c = blockIdx.x;
  if (active[c] == 0) return;
  const int t0 = case_tile0[c], t1 = case_tile0[c + 1];
  __shared__ double sh[256], sh_all[256];
  // acc: the density sum of squares; all: every equation's (non-negative
  // terms, so a NaN or an overflow in any equation leaves it non-finite)
  double acc = 0.0, all = 0.0;
  for (int t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
    const double* pt = partials + (int64_t)t * 2 * nv;
    acc = acc + pt[1];
    for (int m = 0; m < nv; m++) all = all + pt[2 * m + 1];
  }
  sh[threadIdx.x] = acc;
  sh_all[threadIdx.x] = all;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + s];
      sh_all[threadIdx.x] = sh_all[threadIdx.x] + sh_all[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double rms = sqrt(sh[0] / ncell[c]);
    ConvState s = st[c];
    s.iters += 1;
    if (s.iters == 1) s.r0 = rms;
    s.last = rms;
    if (cold[c]) s.status = 4;  // the reference's T < 1e-5 stop, for this case only
    else if (!isfinite(rms) || !isfinite(sh_all[0])) s.status = 2;
    else if (rms <= drop * s.r0) s.status = 1;
    else if (s.iters >= max_iter) s.status = 3;
    if (s.status != 0) active[c] = 0;
    st[c] = s;
  }
}
