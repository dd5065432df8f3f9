// The four split-explicit barotropic schemes of update_ocean_barotropic
// (ocean_barotropic.F90:2829-2843) with barotropic_halo = 1 and no tides,
// geoid, friction, smoothing, blobs or OBC, one template per scheme:
//   <CG=false, PR=false> pred_corr_tropic_depth_bgrid :3225-3579
//   <CG=true,  PR=false> pred_corr_tropic_depth_cgrid :3601-3965
//   <CG=false, PR=true>  pred_corr_tropic_press_bgrid :3989-4329
//   <CG=true,  PR=true>  pred_corr_tropic_press_cgrid :4355-4693
// followed by the tail of update_ocean_barotropic (:2846-2894).
//
// Blocked in time where the domain allows it (k_btv_block, several subcycles a
// launch); otherwise, and with barotropic_subcycles_per_launch = 0, two
// launches per subcycle, each over the data domain:
//   k_btv_velocity  udrho_bt(fstaup1) at every point.  The predicted x
//                   (eta_t_bt or anompb_bt) is recomputed at the points the
//                   pressure gradient needs instead of being stored; the
//                   B-grid's legacy halo update of the prediction and the
//                   C-grid's halo update of udrho_bt are folded in by
//                   computing a rewritten halo point at its cyclic source.
//                   The C-grid Adams-Bashforth Coriolis force of this
//                   subcycle is written (compute points only) into the one
//                   of its three levels the subcycle does not read.
//   k_btv_corrector x_bt(fstaup1) from the new transports, and the time sums
//                   (kept in scratch so that the tail can read a halo
//                   point's source while other threads write the outputs).
// Every value is formed with the reference's operations in its order
// (-ffp-contract=off), so the results equal the CPU restatement bit for bit.
#include "mom_internal.h"

#include <algorithm>

namespace {

constexpr double kEpsln = 1.0e-40;   // shared/constants/constants.F90:123

template <bool CG, bool PR>
struct BtvArgs {
  KDom d;
  // grid (context copies)
  const double *dxu, *dyu, *dxur, *dyur, *dat, *datr, *dxte, *dytn, *f;
  const int *kmt, *kmu;
  // inputs
  const double *x_tau, *xbar_tau, *ud_tau, *forcing, *thick, *tmasken, *patm, *rho_g,
      *dpatm_dt, *pme, *river, *source, *smooth;
  // state: x_bt (2 levels), ud_bt (2 comps x 2 levels), sf, cori1, cori2,
  // coriolis force (2 comps x 3 levels), time sums (x, ud 2 comps)
  double *xb, *ud, *sf, *cori1, *cori2, *cf, *accx, *accu;
  double dtbt, grav, rho0r;
  double c_pred, c_corr;       // predictor / corrector factors of the scheme
  int predict;                 // 0: eta_t_bt(fstaup1) = eta_t_bt(fstau)
  int initsum;
};

__device__ inline double tm1(const int *kmt, int o) { return 1 <= kmt[o] ? 1.0 : 0.0; }

// DIV_UD (ocean_operators.F90:507-608), halo 1; zero on the first row and
// column of the data domain.
template <bool CG, bool PR>
__device__ inline double div_ud(const BtvArgs<CG, PR> &a, const double *u1, const double *u2,
                                int ii, int jj) {
  if (ii == 0 || jj == 0) return 0.0;
  const KDom &d = a.d;
  const int o = ii + d.NI * jj, ojm = o - d.NI, oim = o - 1;
  if (CG) {   // :526-536
    const double uhim = u1[oim] * a.dat[oim] * (1.0 / (a.dxte[oim] + kEpsln));
    const double vhjm = u2[ojm] * a.dat[ojm] * (1.0 / (a.dytn[ojm] + kEpsln));
    const double uh = u1[o] * a.dat[o] * (1.0 / (a.dxte[o] + kEpsln));
    const double vh = u2[o] * a.dat[o] * (1.0 / (a.dytn[o] + kEpsln));
    return ((uh - uhim) + (vh - vhjm)) * a.datr[o];
  }
  const int oimjm = ojm - 1;  // B-grid, :570-605
  const double uh = u1[o] * a.dyu[o], vh = u2[o] * a.dxu[o];
  const double uhjm = u1[ojm] * a.dyu[ojm], vhjm = u2[ojm] * a.dxu[ojm];
  const double uhim = u1[oim] * a.dyu[oim], vhim = u2[oim] * a.dxu[oim];
  const double uhimjm = u1[oimjm] * a.dyu[oimjm], vhimjm = u2[oimjm] * a.dxu[oimjm];
  const double uh_bay = 0.5 * (uh + uhjm);
  const double vh_bax = 0.5 * (vh + vhim);
  const double uhim_bay = 0.5 * (uhim + uhimjm);
  const double vhjm_bax = 0.5 * (vhjm + vhimjm);
  return ((uh_bay - uhim_bay) + (vh_bax - vhjm_bax)) * a.datr[o];
}

// x_bt(fstaup1) after the predictor at data point q (no halo semantics).
template <bool CG, bool PR>
__device__ inline double predicted(const BtvArgs<CG, PR> &a, const double *x0, const double *u1,
                                   const double *u2, int qi, int qj) {
  const int o = qi + a.d.NI * qj;
  if (!a.predict) return x0[o];
  const double dv = div_ud(a, u1, u2, qi, qj);
  const double tmp = PR ? -a.grav * dv : -dv * tm1(a.kmt, o);
  return x0[o] + a.c_pred * (tmp + a.sf[o]);
}

// The field whose gradient drives the transports, at data point q:
// ps_bt = rho_g*eta_t_bt + patm (depth), tmask*anompb_bt (pressure).  The
// B-grid reads the prediction after its legacy halo update (:3383, :4140).
template <bool CG, bool PR>
__device__ inline double drive_p(const BtvArgs<CG, PR> &a, const double *x0, const double *u1,
                                 const double *u2, int qi, int qj) {
  int si = qi, sj = qj;
  if (!CG) halo_source(a.d, qi, qj, si, sj);
  const double xp = predicted(a, x0, u1, u2, si, sj);
  const int o = qi + a.d.NI * qj;
  return PR ? tm1(a.kmt, o) * xp : a.rho_g[o] * xp + a.patm[o];
}

// C-grid Coriolis force at compute point o from the transports u1, u2
// (:3711-3727 and :3838-3851).
__device__ inline void cori_force(const KDom &d, const double *f, const double *u1,
                                  const double *u2, int o, double &F1, double &F2) {
  const int oe = o + 1, os = o - d.NI, ose = os + 1, ow = o - 1, on = o + d.NI, onw = on - 1;
  F1 = 0.25 * (f[o] * (u2[o] + u2[oe]) + f[os] * (u2[os] + u2[ose]));
  F2 = -(0.25 * (f[o] * (u1[o] + u1[on]) + f[ow] * (u1[ow] + u1[onw])));
}

template <bool CG, bool PR>
__global__ void k_btv_init(BtvArgs<CG, PR> a) {
  const KDom &d = a.d;
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const int o = ii + d.NI * jj, P2 = d.P2;
  // itime = 1: fstau = 2, fstaup1 = 1
  a.accx[o] = a.initsum ? a.xbar_tau[o] : a.x_tau[o];
  a.accu[o] = 0.0;
  a.accu[o + P2] = 0.0;
  a.xb[P2 + o] = a.xbar_tau[o];
  a.xb[o] = a.xbar_tau[o];
  a.ud[2 * P2 + o] = a.ud_tau[o];
  a.ud[3 * P2 + o] = a.ud_tau[o + P2];
  const double tm = tm1(a.kmt, o);
  const double s = a.pme[o] + a.river[o] + a.source[o] - a.smooth[o];
  a.sf[o] = PR ? tm * (a.grav * s + a.dpatm_dt[o]) : tm * s;
  if (!CG) {
    const double c1 = 0.5 * a.dtbt * a.f[o];      // :1285-1286
    a.cori1[o] = c1;
    a.cori2[o] = 1.0 / (1.0 + c1 * c1);
  } else {
    double F1 = 0.0, F2 = 0.0;
    if (ii >= 1 && ii <= d.ni && jj >= 1 && jj <= d.nj)
      cori_force(d, a.f, a.ud_tau, a.ud_tau + P2, o, F1, F2);
    for (int lev = 0; lev < 3; ++lev) {
      a.cf[(size_t)P2 * (2 * lev) + o] = F1;
      a.cf[(size_t)P2 * (2 * lev + 1) + o] = F2;
    }
  }
}

// Subcycle itime: levels fstau/fstaup1 (1-based) and the Adams-Bashforth
// levels m0 (written), m1, m2.
template <bool CG, bool PR>
__global__ void k_btv_velocity(BtvArgs<CG, PR> a, int fstau, int fstaup1, int m0, int m1,
                               int m2) {
  const KDom &d = a.d;
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const size_t P2 = (size_t)d.P2;
  const double *x0 = a.xb + P2 * (fstau - 1);
  const double *u1 = a.ud + P2 * (2 * (fstau - 1));
  const double *u2 = u1 + P2;
  double *n1 = a.ud + P2 * (2 * (fstaup1 - 1));
  double *n2 = n1 + P2;
  const int o = ii + d.NI * jj;
  // the point whose transports this thread computes (C-grid: the halo
  // update of udrho_bt(fstaup1), :3895-3897)
  int si = ii, sj = jj;
  if (CG) halo_source(d, ii, jj, si, sj);
  const int os = si + d.NI * sj;
  double g1 = 0.0, g2 = 0.0;
  if (si < d.NI - 1 && sj < d.NJ - 1) {
    const double pc = drive_p(a, x0, u1, u2, si, sj);
    const double pe = drive_p(a, x0, u1, u2, si + 1, sj);
    const double pn = drive_p(a, x0, u1, u2, si, sj + 1);
    if (CG) {   // GRAD_BAROTROPIC_P, C-grid (ocean_operators.F90:664-669)
      g1 = (pe - pc) * (1.0 / (a.dxte[os] + kEpsln)) * a.tmasken[os];
      g2 = (pn - pc) * (1.0 / (a.dytn[os] + kEpsln)) * a.tmasken[P2 + os];
    } else {    // B-grid (:651-660)
      const double pne = drive_p(a, x0, u1, u2, si + 1, sj + 1);
      const double p_fay = 0.5 * (pc + pn);
      const double p_fax = 0.5 * (pc + pe);
      const double pip_fay = 0.5 * (pe + pne);
      const double pjp_fax = 0.5 * (pn + pne);
      const double um = 1 <= a.kmu[os] ? 1.0 : 0.0;
      g1 = (pip_fay - p_fay) * a.dxur[os] * um;
      g2 = (pjp_fax - p_fax) * a.dyur[os] * um;
    }
  }
  const double th1 = a.thick[os], th2 = CG ? a.thick[P2 + os] : th1;
  const double pf1 = PR ? -(a.rho0r * th1 * g1) : -(th1 * g1);
  const double pf2 = PR ? -(a.rho0r * th2 * g2) : -(th2 * g2);
  const double v1 = u1[os], v2 = u2[os];
  double r1, r2;
  if (CG) {
    double acc1 = 0.0, acc2 = 0.0;
    if (si >= 1 && si <= d.ni && sj >= 1 && sj <= d.nj) {
      double F1, F2;
      cori_force(d, a.f, u1, u2, os, F1, F2);
      const double *c1 = a.cf + P2 * (2 * (m1 - 1)), *c2 = a.cf + P2 * (2 * (m2 - 1));
      constexpr double ab0 = 23.0 / 12.0, ab1 = -16.0 / 12.0, ab2 = 5.0 / 12.0;  // :617-619
      acc1 = ab0 * F1 + ab1 * c1[os] + ab2 * c2[os];
      acc2 = ab0 * F2 + ab1 * c1[P2 + os] + ab2 * c2[P2 + os];
      if (os == o) {
        double *c0 = a.cf + P2 * (2 * (m0 - 1));
        c0[o] = F1;
        c0[P2 + o] = F2;
      }
    }
    const double s1 = acc1 + pf1 + a.forcing[os];
    const double s2 = acc2 + pf2 + a.forcing[P2 + os];
    r1 = v1 + a.dtbt * a.tmasken[os] * (PR ? s1 : s1 + 0.0);
    r2 = v2 + a.dtbt * a.tmasken[P2 + os] * (PR ? s2 : s2 + 0.0);
  } else {
    const double fo = a.f[os];
    double t1, t2;
    if (PR) {
      t1 = v1 + a.dtbt * (0.5 * fo * v2 + pf1 + a.forcing[os]);
      t2 = v2 + a.dtbt * (-(0.5 * fo * v1) + pf2 + a.forcing[P2 + os]);
    } else {
      t1 = v1 + a.dtbt * (0.5 * fo * v2 + pf1 + a.forcing[os] + 0.0);
      t2 = v2 + a.dtbt * (-(0.5 * fo * v1) + pf2 + a.forcing[P2 + os] + 0.0);
    }
    r1 = a.cori2[os] * (t1 + a.cori1[os] * t2);
    r2 = a.cori2[os] * (t2 - a.cori1[os] * t1);
  }
  n1[o] = r1;
  n2[o] = r2;
}

template <bool CG, bool PR>
__global__ void k_btv_corrector(BtvArgs<CG, PR> a, int fstau, int fstaup1, double wgt) {
  const KDom &d = a.d;
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const size_t P2 = (size_t)d.P2;
  const double *x0 = a.xb + P2 * (fstau - 1);
  double *x1 = a.xb + P2 * (fstaup1 - 1);
  const double *n1 = a.ud + P2 * (2 * (fstaup1 - 1));
  const double *n2 = n1 + P2;
  const int o = ii + d.NI * jj;
  const double dv = div_ud(a, n1, n2, ii, jj);
  const double tmp = PR ? -a.grav * dv : -dv * tm1(a.kmt, o);
  const double xn = x0[o] + a.c_corr * (tmp + a.sf[o]);
  x1[o] = xn;
  a.accx[o] = a.accx[o] + xn;
  if (wgt == 0.0) {           // barotropic_time_stepping_A
    a.accu[o] = a.accu[o] + n1[o];
    a.accu[P2 + o] = a.accu[P2 + o] + n2[o];
  } else {
    a.accu[o] = a.accu[o] + wgt * n1[o];
    a.accu[P2 + o] = a.accu[P2 + o] + wgt * n2[o];
  }
}

// ---- temporally blocked subcycles -----------------------------------------
// The two-launch form above moves every plane through memory twice a subcycle.
// Here one work-group owns a region of the data domain and advances it nsub
// subcycles with its state in registers, reading and writing the planes once a
// launch.
//
// A wavefront holds neighbouring rows, so x neighbours are DPP lane shifts and
// most y neighbours the thread's own registers; the others go through LDS, one
// row a wavefront and quantity.  The forcing and the thickness are read once a
// subcycle and lie in LDS too.
//
// Grids that do not change along a row (checked at creation) take a row's constants
// by scalar loads (the C-grid pressure instance keeps 75 scalars in lanes of vector
// registers and has 20 B of scratch), so 8 wavefronts of three rows (64 x 24) take at
// most 128 registers and two blocks share a CU: one loads while the other steps.
// Other grids, and the C-grid depth scheme (whose LDS holds two more planes), take
// 16 wavefronts of two rows (64 x 32), one block a CU.  A subcycle is bound by
// its FP64 instructions (C-grid pressure: 87 a point), a launch by loading the
// planes as much.  80 subcycles at 1440x1080, C-grid pressure: 11.4 ms with two
// launches a subcycle, 2.26 ms in 64 x 32 regions with per-point constants and
// edge tests everywhere (130 instructions a point), 1.56 ms so; B-grid pressure 1.03 ms.
//
// Dependencies: a transport needs the transports one point away in each
// direction, x also those of one point west and south.  After nsub subcycles a
// region is exact from nsub + 1 points above its low edges to nsub points below
// its high ones.  On a cyclic-x domain the reference keeps a halo column's own
// values and only overwrites what its halo update covers (B-grid: the predicted
// x, C-grid: the transports, compute rows), so the region runs over the data
// columns 0 .. NI-1, 0, 1, .. and column 0 (NI-1) takes the updated quantity
// from column NI-2 (1), two lanes to the left (right): two more halo lanes a
// side.  A chain of dependencies crosses that seam once if ni > nsub, so
// domains narrower than MIN_NI, and cyclic-y ones, keep the two launches.
constexpr int VX = 64;                 // region columns; rows: R a wavefront, NW wavefronts
constexpr int MIN_NI = 16;             // > the most subcycles a launch takes (12)

__host__ __device__ constexpr int btv_lo(int nsub, bool cyc) { return nsub + 1 + (cyc ? 2 : 0); }
__host__ __device__ constexpr int btv_tx(int nsub, bool cyc) {
  return VX - 2 * nsub - 1 - (cyc ? 4 : 0);
}
__host__ __device__ constexpr int btv_ty(int nsub, int ry) { return ry - 2 * nsub - 1; }

struct BtvBlk {
  const double *xs, *us, *fs;          // state read: x, transports (2), force at two levels (4)
  double *xd, *ud, *fd;                // state written
  const unsigned char *mask;           // bit 0 tmask(k=1), bit 1 umask(k=1)
  const double *rowc;                  // the rows' constants (UNI)
  int s0, nsub, nts, step_a, ntx, ntiles;
  int rev;                             // 1: the tiles in reverse order (see k_bt_block)
};

// A point's constants of the grid.  B-grid: datr, dyu/2, dxu/2, dxur/2, dyur/2,
// cori1, cori2 (:1285-1286), f/2; C-grid: datr, dat, -, 1/(dxte + eps),
// 1/(dytn + eps), -, -, f/4 (the halves and quarters of the averages they
// multiply: powers of two, exact short of the subnormals).
struct RowC {
  double datr, m1, m2, g1, g2, k1, k2, f;
};
template <bool CG, bool PR>
__device__ inline RowC row_const(const BtvArgs<CG, PR> &a, int o) {
  RowC c{};
  c.datr = a.datr[o];
  const double f = a.f[o];
  if (CG) {
    c.m1 = a.dat[o];
    c.g1 = 1.0 / (a.dxte[o] + kEpsln);
    c.g2 = 1.0 / (a.dytn[o] + kEpsln);
    c.f = 0.25 * f;
  } else {
    c.m1 = 0.5 * a.dyu[o]; c.m2 = 0.5 * a.dxu[o];
    c.g1 = 0.5 * a.dxur[o]; c.g2 = 0.5 * a.dyur[o];
    c.k1 = 0.5 * a.dtbt * f;
    c.k2 = 1.0 / (1.0 + c.k1 * c.k1);
    c.f = 0.5 * f;
  }
  return c;
}

// sf and the masks, constant over the subcycles
template <bool CG, bool PR>
__global__ void k_btv_sfmask(BtvArgs<CG, PR> a, unsigned char *__restrict__ mask,
                             double *__restrict__ rowc) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= a.d.NI) return;
  const int o = ii + a.d.NI * jj;
  const double tm = tm1(a.kmt, o);
  const double s = a.pme[o] + a.river[o] + a.source[o] - a.smooth[o];
  a.sf[o] = PR ? tm * (a.grav * s + a.dpatm_dt[o]) : tm * s;
  mask[o] = (unsigned char)((1 <= a.kmt[o] ? 1 : 0) | (1 <= a.kmu[o] ? 2 : 0));
  if (rowc && ii == 0) {
    const RowC c = row_const(a, o);
    double *r = rowc + (size_t)8 * jj;
    r[0] = c.datr; r[1] = c.m1; r[2] = c.m2; r[3] = c.g1; r[4] = c.g2; r[5] = c.k1; r[6] = c.k2;
    r[7] = c.f;
  }
}

template <bool CG, bool PR, int R, int NW>
struct BtvLds {
  static constexpr bool PL = CG && !PR;
  // p and u1 (C) of the wavefronts' first rows, vh and u2 (C) or uh (B) of their last
  double p[NW][VX], v[NW][VX], u1[NW][VX], u2[CG ? NW : 1][VX];
  // forcing (2), thickness (C: 2), C: tmasken (1, a wavefront of three rows); C-grid
  // depth: rho_g, patm
  static constexpr int NC = PL ? 6 : (CG ? (R > 2 ? 5 : 4) : 3);
  double c[NC][R][NW][VX];
};

// EDGE: the region meets the domain's first or last row or column, or the seam; the
// others carry no such tests (two instances: in one, the branches cost registers).
// UNI: the grid does not change along a row; its constants are scalars.
template <bool CG, bool PR, int R, int NW, bool EDGE, bool UNI>
__device__ __forceinline__ void btv_tile(const BtvArgs<CG, PR> &a, const BtvBlk &J, int tx, int ty,
                                         BtvLds<CG, PR, R, NW> &S) {
  const KDom d = a.d;
  const int P2 = d.P2, nsub = J.nsub;
  const bool cyc = d.cyclic_x != 0;
  constexpr bool PL = CG && !PR;
  constexpr bool KL = CG && !PL && R > 2;     // tmasken of the east face in LDS
  auto &s_c = S.c;
  const int lane = threadIdx.x & (VX - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / VX);
  const int wm = max(wave - 1, 0), wp = min(wave + 1, NW - 1);
  const int LX = btv_lo(nsub, cyc), LY = btv_lo(nsub, false);
  const int TX = btv_tx(nsub, cyc), TY = btv_ty(nsub, R * NW);
  const int seq = tx * TX - LX + lane;                    // position in the column sequence
  const int col = cyc ? wrapi(seq, d.NI) : seq;
  const int row0 = ty * TY - LY + R * wave;
  const bool colok = cyc || (seq >= 0 && seq < d.NI);
  // a region that holds the seam of a cyclic-x domain (uniform)
  const int seq0 = tx * TX - LX;
  const bool seam = EDGE && cyc && (seq0 <= 0 || seq0 + VX > d.NI - 2);
  const bool first = J.s0 == 1;
  const double rho0r = a.rho0r, dtbt = a.dtbt, ngrav = -a.grav;
  typedef const __attribute__((address_space(4))) double ConstD;

  auto inside = [&](int q) {
    const int r = R * wave + q, j = row0 + q;
    return colok && j >= 0 && j < d.NJ && lane >= LX && lane < LX + TX && seq < d.NI && r >= LY &&
           r < LY + TY;
  };
  auto div0 = [&](int q) { return EDGE && (col == 0 || row0 + q == 0); };
  auto grad0 = [&](int q) { return EDGE && (col == d.NI - 1 || row0 + q == d.NJ - 1); };
  auto crow = [&](int q) { return row0 + q >= 1 && row0 + q <= d.nj; };
  auto nocomp = [&](int q) { return EDGE && !(crow(q) && col >= 1 && col <= d.ni); };
  // the halo update of a cyclic-x domain's halo columns: from two lanes away
  auto update = [&](int q, double e) {
    const double w = lane_prev(lane_prev(e)), n = lane_next(lane_next(e));
    return !crow(q) ? e : (col == 0 ? w : (col == d.NI - 1 ? n : e));
  };
  bool tmb[R];
  double x[R], u1[R], u2[R], fa1[R], fa2[R], fb1[R], fb2[R], sx[R], su1[R], su2[R];
  double datr[R], m1[R], m2[R], g1c[R], g2c[R], k1[R], k2[R], f[R], sf[R], rg[R], pa[R], um[R];
  double fS = 0.0;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int j = row0 + q;
    const bool present = !EDGE || (colok && j >= 0 && j < d.NJ);
    const int o = present ? col + d.NI * j : 0;
    double c0 = 0.0, c1 = 0.0, c2 = 0.0, c3 = 0.0;
    tmb[q] = false;
    x[q] = u1[q] = u2[q] = fa1[q] = fa2[q] = fb1[q] = fb2[q] = sx[q] = su1[q] = su2[q] = 0.0;
    datr[q] = m1[q] = m2[q] = g1c[q] = g2c[q] = k1[q] = k2[q] = f[q] = 0.0;
    sf[q] = rg[q] = pa[q] = um[q] = 0.0;
    if constexpr (UNI) {
      const int jc = EDGE ? min(max(j, 0), d.NJ - 1) : j;       // uniform
      ConstD *rc = (ConstD *)(unsigned long long)(J.rowc + (size_t)8 * jc);
      datr[q] = rc[0]; m1[q] = rc[1]; g1c[q] = rc[3]; g2c[q] = rc[4]; f[q] = rc[7];
      if (!CG) { m2[q] = rc[2]; k1[q] = rc[5]; k2[q] = rc[6]; }
      if (CG && q == 0) {
        ConstD *rs = (ConstD *)(unsigned long long)(J.rowc + (size_t)8 * max(jc - 1, 0));
        fS = EDGE && j < 1 ? 0.0 : rs[7];
      }
    }
    if (present) {
      const unsigned char mb = J.mask[o];
      tmb[q] = (mb & 1) != 0;
      um[q] = (mb & 2) ? 1.0 : 0.0;
      x[q] = J.xs[o]; u1[q] = J.us[o]; u2[q] = J.us[o + P2];
      sf[q] = a.sf[o];
      // + 0.0 (depth): the forcing is the last term of the sum it is added to
      c0 = PR ? a.forcing[o] : a.forcing[o] + 0.0;
      c1 = PR ? a.forcing[o + P2] : a.forcing[o + P2] + 0.0;
      c2 = PR ? rho0r * a.thick[o] : a.thick[o];
      if (!PR) { rg[q] = a.rho_g[o]; pa[q] = a.patm[o]; }
      if constexpr (!UNI) {
        const RowC c = row_const(a, o);
        datr[q] = c.datr; m1[q] = c.m1; g1c[q] = c.g1; g2c[q] = c.g2; f[q] = c.f;
        if (!CG) { m2[q] = c.m2; k1[q] = c.k1; k2[q] = c.k2; }
        if (CG && q == 0) fS = j >= 1 ? 0.25 * a.f[o - d.NI] : 0.0;
      }
      if (CG) {
        c3 = PR ? rho0r * a.thick[o + P2] : a.thick[o + P2];
        k1[q] = a.tmasken[o]; k2[q] = a.tmasken[o + P2];
        if (!first) {
          fa1[q] = J.fs[o]; fa2[q] = J.fs[o + P2];
          fb1[q] = J.fs[o + 2 * (size_t)P2]; fb2[q] = J.fs[o + 3 * (size_t)P2];
        }
      }
      if (inside(q)) {
        if (first) {
          sx[q] = a.initsum ? a.xbar_tau[o] : a.x_tau[o];
        } else {
          sx[q] = a.accx[o]; su1[q] = a.accu[o]; su2[q] = a.accu[o + P2];
        }
      }
    }
    s_c[0][q][wave][lane] = c0;
    s_c[1][q][wave][lane] = c1;
    s_c[2][q][wave][lane] = c2;
    if constexpr (CG) s_c[3][q][wave][lane] = c3;
    if constexpr (PL) {
      s_c[4][q][wave][lane] = rg[q];
      s_c[5][q][wave][lane] = pa[q];
    }
    if constexpr (KL) s_c[4][q][wave][lane] = k1[q];
  }
  double fW[R];
#pragma unroll
  for (int q = 0; q < R; ++q) fW[q] = UNI ? f[q] : lane_prev(f[q]);

  // the transports through a cell's edges of the rows, those other rows read to LDS
  double uh[R], vh[R], g[R];
  auto share = [&]() {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if (CG) {      // DIV_UD, C-grid (ocean_operators.F90:526-536)
        uh[q] = u1[q] * m1[q] * g1c[q];
        vh[q] = u2[q] * m1[q] * g2c[q];
      } else {
        uh[q] = u1[q] * m1[q];
        vh[q] = u2[q] * m2[q];
      }
    }
    S.v[wave][lane] = vh[R - 1];
    if constexpr (CG) {
      S.u1[wave][lane] = u1[0];
      S.u2[wave][lane] = u2[R - 1];
    } else {
      S.u1[wave][lane] = uh[R - 1];
    }
  };
  // g = the divergence term + sf: what the predictor and the corrector scale
  auto diverge = [&]() {
    double vs = S.v[wm][lane], us = 0.0;
    if constexpr (!CG) {
      us = S.u1[wm][lane];
      vs = vs + lane_prev(vs);                // twice the average, as m2 is half dxu
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      double dv;
      if constexpr (CG) {
        dv = ((uh[q] - lane_prev(uh[q])) + (vh[q] - vs)) * datr[q];
        vs = vh[q];
      } else {         // B-grid (:570-605)
        const double bay = uh[q] + us, bax = vh[q] + lane_prev(vh[q]);
        dv = ((bay - lane_prev(bay)) + (bax - vs)) * datr[q];
        us = uh[q];
        vs = bax;
      }
      if (div0(q)) dv = 0.0;
      const double tmp = PR ? ngrav * dv : (tmb[q] ? -dv : -dv * 0.0);
      g[q] = tmp + sf[q];
    }
  };
  share();
  __syncthreads();
  diverge();

  for (int t = 0; t < nsub; ++t) {
    const int itime = J.s0 + t;
    // A: the prediction and the pressure; C-grid: the Coriolis force, from
    // the transports that the phases B before wrote
    double F1[R], F2[R], p[R + 1];
    if constexpr (CG) {
      const double u1n = S.u1[wp][lane];
      double es = S.u2[wm][lane], fs = fS;
      es = es + lane_next(es);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const double e = u2[q] + lane_next(u2[q]);
        F1[q] = f[q] * e + fs * es;
        const double n = u1[q] + (q + 1 < R ? u1[min(q + 1, R - 1)] : u1n);
        F2[q] = -(f[q] * n + fW[q] * lane_prev(n));
        es = e;
        fs = f[q];
        if (nocomp(q)) F1[q] = F2[q] = 0.0;
        if (itime == 1) {                     // all three levels (:3711-3730)
          fa1[q] = fb1[q] = F1[q];
          fa2[q] = fb2[q] = F2[q];
        }
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      double e = x[q];
      if (a.predict) e = x[q] + a.c_pred * g[q];
      if constexpr (!CG)
        if (seam) e = update(q, e);           // the legacy halo update (:3383, :4140)
      if constexpr (PR)
        p[q] = tmb[q] ? e : e * 0.0;
      else if constexpr (PL)
        p[q] = s_c[4][q][wave][lane] * e + s_c[5][q][wave][lane];
      else
        p[q] = rg[q] * e + pa[q];
    }
    S.p[wave][lane] = p[0];
    __syncthreads();
    // B: pressure gradient and transports
    p[R] = S.p[wp][lane];
    double pe = lane_next(p[0]), fax = p[0] + pe;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double pn = p[q + 1], pne = lane_next(pn);
      double h1, h2;
      const double k1q = KL ? s_c[KL ? 4 : 0][q][wave][lane] : k1[q];
      if constexpr (CG) {    // GRAD_BAROTROPIC_P, C-grid (ocean_operators.F90:664-669)
        h1 = (pe - p[q]) * g1c[q] * k1q;
        h2 = (pn - p[q]) * g2c[q] * k2[q];
      } else {     // B-grid (:651-660), the halves in g1c, g2c
        const double fay = p[q] + pn, pip = pe + pne, pjp = pn + pne;
        h1 = (pip - fay) * g1c[q] * um[q];
        h2 = (pjp - fax) * g2c[q] * um[q];
        fax = pjp;
      }
      pe = pne;
      if (grad0(q)) h1 = h2 = 0.0;
      const double th1 = s_c[2][q][wave][lane], th2 = CG ? s_c[CG ? 3 : 2][q][wave][lane] : th1;
      const double fo1 = s_c[0][q][wave][lane], fo2 = s_c[1][q][wave][lane];
      const double v1 = u1[q], v2 = u2[q];
      if constexpr (CG) {
        constexpr double ab0 = 23.0 / 12.0, ab1 = -16.0 / 12.0, ab2 = 5.0 / 12.0;  // :617-619
        double acc1 = ab0 * F1[q] + ab1 * fa1[q] + ab2 * fb1[q];
        double acc2 = ab0 * F2[q] + ab1 * fa2[q] + ab2 * fb2[q];
        if (nocomp(q)) acc1 = acc2 = 0.0;
        u1[q] = v1 + dtbt * k1q * (acc1 - th1 * h1 + fo1);
        u2[q] = v2 + dtbt * k2[q] * (acc2 - th2 * h2 + fo2);
        if (seam) {                         // the halo update of udrho_bt (:3895-3897)
          u1[q] = update(q, u1[q]);
          u2[q] = update(q, u2[q]);
        }
        fb1[q] = fa1[q]; fb2[q] = fa2[q];
        fa1[q] = F1[q]; fa2[q] = F2[q];
      } else {
        const double r1 = v1 + dtbt * (f[q] * v2 - th1 * h1 + fo1);
        const double r2 = v2 + dtbt * (-(f[q] * v1) - th2 * h2 + fo2);
        u1[q] = k2[q] * (r1 + k1[q] * r2);
        u2[q] = k2[q] * (r2 - k1[q] * r1);
      }
    }
    // the reads of S.v, S.u1, S.u2 of phases C and A are behind the barrier above
    share();
    __syncthreads();
    // C: corrector and time sums
    diverge();
    const double wgt = J.step_a ? 1.0 : (double)(J.nts - itime + 1);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      x[q] = x[q] + a.c_corr * g[q];
      sx[q] = sx[q] + x[q];
      su1[q] = su1[q] + wgt * u1[q];
      su2[q] = su2[q] + wgt * u2[q];
    }
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    if (!inside(q)) continue;
    const int o = col + d.NI * (row0 + q);
    J.xd[o] = x[q];
    J.ud[o] = u1[q];
    J.ud[o + P2] = u2[q];
    if (CG) {
      J.fd[o] = fa1[q];
      J.fd[o + P2] = fa2[q];
      J.fd[o + 2 * (size_t)P2] = fb1[q];
      J.fd[o + 3 * (size_t)P2] = fb2[q];
    }
    a.accx[o] = sx[q];
    a.accu[o] = su1[q];
    a.accu[o + P2] = su2[q];
  }
}

// rows and wavefronts of a region
template <bool CG, bool PR>
__host__ __device__ constexpr int btv_r(bool uni) { return uni && (PR || !CG) ? 3 : 2; }
template <bool CG, bool PR>
__host__ __device__ constexpr int btv_nw(bool uni) { return btv_r<CG, PR>(uni) == 3 ? 8 : 16; }
template <bool CG, bool PR>
__host__ __device__ constexpr int btv_ry(bool uni) {
  return btv_r<CG, PR>(uni) * btv_nw<CG, PR>(uni);
}

template <bool CG, bool PR, bool UNI>
__global__ __launch_bounds__((VX * btv_nw<CG, PR>(UNI)), 4) void k_btv_block(BtvArgs<CG, PR> a,
                                                                          BtvBlk J, int per_xcd) {
  constexpr int R = btv_r<CG, PR>(UNI), NW = btv_nw<CG, PR>(UNI), RY = R * NW;
  __shared__ BtvLds<CG, PR, R, NW> lds;
  const int b = blockIdx.x;
  const int t0 = (b & 7) * per_xcd + (J.rev ? per_xcd - 1 - (b >> 3) : b >> 3);
  if (t0 >= J.ntiles) return;                  // the whole block
  const int tile = strip_tile<8>(t0, J.ntx, J.ntiles / J.ntx);
  const int tx = tile % J.ntx, ty = tile / J.ntx;
  const KDom &d = a.d;
  const bool cyc = d.cyclic_x != 0;
  const int x0 = tx * btv_tx(J.nsub, cyc) - btv_lo(J.nsub, cyc);
  const int y0 = ty * btv_ty(J.nsub, RY) - btv_lo(J.nsub, false);
  if (x0 <= 0 || x0 + VX > d.NI - 2 || y0 <= 0 || y0 + RY > d.NJ - 2)
    btv_tile<CG, PR, R, NW, true, UNI>(a, J, tx, ty, lds);
  else
    btv_tile<CG, PR, R, NW, false, UNI>(a, J, tx, ty, lds);
}

template <bool CG, bool PR>
int btv_tiles(const KDom &d, bool uni, int h) {
  const int TX = btv_tx(h, d.cyclic_x != 0), TY = btv_ty(h, btv_ry<CG, PR>(uni));
  return ((d.NI + TX - 1) / TX) * ((d.NJ + TY - 1) / TY);
}

// Rows of scalar constants, where the grid allows it.
template <bool CG>
bool rows_uniform(const mom_gpu_ctx *ctx) {
  return CG ? ctx->btv_rows_ok : ctx->bt_rows_ok;
}

// nsub = hsub subcycles a launch; the state alternates between two sets of
// planes of ctx->btv (a region reads its neighbours' points).
template <bool CG, bool PR>
int run_blocked(mom_gpu_ctx *ctx, const BtvArgs<CG, PR> &a, int nts, int step_a, int hsub) {
  const KDom &d = a.d;
  const size_t P2 = (size_t)d.P2;
  hipStream_t s = ctx->stream;
  double *w = ctx->btv;
  unsigned char *mask = (unsigned char *)(w + 7 * P2);    // the place of cori1
  double *xb[2] = {w, w + P2}, *ub[2] = {w + 2 * P2, w + 4 * P2};
  double *fb[2] = {w + 8 * P2, w + 18 * P2};              // 4 planes each: 8-11, 18-21
  const bool uni = rows_uniform<CG>(ctx);
  double *rowc = uni ? w + 7 * P2 + (P2 + 7) / 8 : nullptr;   // behind the masks
  hipLaunchKernelGGL((k_btv_sfmask<CG, PR>), dim3((d.NI + 255) / 256, d.NJ), dim3(256), 0, s, a,
                     mask, rowc);
  MOM_LAUNCHED(ctx, "k_btv_sfmask");
  BtvBlk J{a.xbar_tau, a.ud_tau, nullptr, nullptr, nullptr, nullptr, mask, rowc, 1, 0, nts, step_a,
           0, 0, 0};
  const bool cyc = d.cyclic_x != 0;
  for (int which = 0; J.s0 <= nts; J.s0 += hsub, which ^= 1) {
    J.nsub = min(hsub, nts - J.s0 + 1);
    const int TX = btv_tx(J.nsub, cyc), TY = btv_ty(J.nsub, btv_ry<CG, PR>(uni));
    J.ntx = (d.NI + TX - 1) / TX;
    J.ntiles = J.ntx * ((d.NJ + TY - 1) / TY);
    J.xd = xb[which];
    J.ud = ub[which];
    J.fd = fb[which];
    J.rev = uni ? which : 0;
    const int per_xcd = (J.ntiles + 7) / 8;
    if (uni)
      hipLaunchKernelGGL((k_btv_block<CG, PR, true>), dim3(8 * per_xcd), 
                         dim3(VX * btv_nw<CG, PR>(true)), 0, s, a, J, per_xcd);
    else
      hipLaunchKernelGGL((k_btv_block<CG, PR, false>), dim3(8 * per_xcd), 
                         dim3(VX * btv_nw<CG, PR>(false)), 0, s, a, J, per_xcd);
    MOM_LAUNCHED(ctx, "k_btv_block");
    J.xs = J.xd;
    J.us = J.ud;
    J.fs = J.fd;
  }
  return MOM_GPU_OK;
}

// Subcycles a launch: the most with one round of regions, when a launch's time is its
// latency, and 5 or 6 above; no more than the knob, where it is set (it is
// tuned on pred_corr_tropic_depth_bgrid's own kernel, whose regions hold more
// subcycles: 10 a launch at 1440x1080 C-grid pressure are 5.1 ms, 8 2.32).
// 80 subcycles, us alone: scalar rows (two blocks a CU, at most 256 regions, at most
// 10) 90x60 C-grid pressure 254 at 5, 186 at 10; 360x240 256 at 5, 221 at 7, 285 at 8;
// 517x389 388 at 5, 326 at 7, but among the calls of three contexts queued on their
// streams 184 and 211; 1440x1080 1709 at 5, 1748 at 6.  Other regions (one block a
// CU, at most 128, at most 12) 90x60 C-grid depth 291 at 5, 203 at 12; 1440x1080 2167
// at 5, 1993 at 6, 2119 at 7.  Results do not depend on it.
template <bool CG, bool PR>
int blocked_depth(const mom_gpu_ctx *ctx) {
  const int knob = ctx->tune.bt_subcycles_per_launch;
  const bool uni = rows_uniform<CG>(ctx) && btv_r<CG, PR>(true) == 3;
  const int most = uni ? 256 : 128, least = uni ? 5 : 6;
  int h = uni ? 10 : 12;
  while (h > least && btv_tiles<CG, PR>(ctx->kd, uni, h) > most) --h;
  return knob < 0 ? h : std::min(h, knob);
}

// Tail (:2846-2894): the time means, each halo-updated, and
// conv_rho_ud_t = -DIV_UD(udrho(taup1)) halo-updated.
template <bool CG, bool PR>
__device__ inline double mean_ud(const BtvArgs<CG, PR> &a, double rnts, int c, int qi, int qj) {
  int si, sj;
  halo_source(a.d, qi, qj, si, sj);
  return rnts * a.accu[(size_t)a.d.P2 * c + si + a.d.NI * sj];
}

template <bool CG, bool PR>
__global__ void k_btv_tail(BtvArgs<CG, PR> a, double rntsp1, double rnts, double *__restrict__ xbar,
                           double *__restrict__ udrho, double *__restrict__ conv) {
  const KDom &d = a.d;
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const size_t P2 = (size_t)d.P2;
  const int o = ii + d.NI * jj;
  int si, sj;
  halo_source(d, ii, jj, si, sj);
  const int os = si + d.NI * sj;
  xbar[o] = rntsp1 * a.accx[os];
  udrho[o] = rnts * a.accu[os];
  udrho[P2 + o] = rnts * a.accu[P2 + os];
  if (!conv) return;
  // -DIV_UD of the halo-updated mean at the source point
  double dv = 0.0;
  if (si != 0 && sj != 0) {
    const int oim = os - 1, ojm = os - d.NI;
    const double u = mean_ud(a, rnts, 0, si, sj), v = mean_ud(a, rnts, 1, si, sj);
    const double uim = mean_ud(a, rnts, 0, si - 1, sj);
    const double vjm = mean_ud(a, rnts, 1, si, sj - 1);
    if (CG) {
      const double uhim = uim * a.dat[oim] * (1.0 / (a.dxte[oim] + kEpsln));
      const double vhjm = vjm * a.dat[ojm] * (1.0 / (a.dytn[ojm] + kEpsln));
      const double uh = u * a.dat[os] * (1.0 / (a.dxte[os] + kEpsln));
      const double vh = v * a.dat[os] * (1.0 / (a.dytn[os] + kEpsln));
      dv = ((uh - uhim) + (vh - vhjm)) * a.datr[os];
    } else {
      const int oimjm = ojm - 1;
      const double ujm = mean_ud(a, rnts, 0, si, sj - 1);
      const double vim = mean_ud(a, rnts, 1, si - 1, sj);
      const double uimjm = mean_ud(a, rnts, 0, si - 1, sj - 1);
      const double vimjm = mean_ud(a, rnts, 1, si - 1, sj - 1);
      const double uh = u * a.dyu[os], vh = v * a.dxu[os];
      const double uhjm = ujm * a.dyu[ojm], vhjm = vjm * a.dxu[ojm];
      const double uhim = uim * a.dyu[oim], vhim = vim * a.dxu[oim];
      const double uhimjm = uimjm * a.dyu[oimjm], vhimjm = vimjm * a.dxu[oimjm];
      const double uh_bay = 0.5 * (uh + uhjm);
      const double vh_bax = 0.5 * (vh + vhim);
      const double uhim_bay = 0.5 * (uhim + uhimjm);
      const double vhjm_bax = 0.5 * (vhjm + vhimjm);
      dv = ((uh_bay - uhim_bay) + (vh_bax - vhjm_bax)) * a.datr[os];
    }
  }
  conv[o] = -dv;
}

template <bool CG, bool PR>
int run_variant(mom_gpu_ctx *ctx, const mom_gpu_bt_params_t *p, const mom_gpu_bt_variant_t *v) {
  const KDom &d = ctx->kd;
  const size_t P2 = (size_t)d.P2;
  BtvArgs<CG, PR> a{};
  a.d = d;
  a.dxu = ctx->dxu; a.dyu = ctx->dyu; a.dxur = ctx->dxur; a.dyur = ctx->dyur;
  a.dat = ctx->dat; a.datr = ctx->datr; a.dxte = ctx->dxte; a.dytn = ctx->dytn; a.f = ctx->f;
  a.kmt = ctx->kmt; a.kmu = ctx->kmu;
  a.x_tau = v->x_tau; a.xbar_tau = v->x_bar_tau; a.ud_tau = v->udrho_tau;
  a.forcing = v->forcing_bt; a.thick = v->thick; a.tmasken = v->tmasken;
  a.patm = v->patm; a.rho_g = v->rho_g; a.dpatm_dt = v->dpatm_dt;
  a.pme = v->pme; a.river = v->river; a.source = v->source; a.smooth = v->smooth;
  double *w = ctx->btv;
  a.xb = w;               // 2 planes
  a.ud = w + 2 * P2;      // 4
  a.sf = w + 6 * P2;      // 1
  a.cori1 = w + 7 * P2;   // 1
  a.cori2 = w + 8 * P2;   // 1
  a.cf = w + 9 * P2;      // 6
  a.accx = w + 15 * P2;   // 1
  a.accu = w + 16 * P2;   // 2
  a.dtbt = p->dtbt;
  a.grav = v->grav;
  a.rho0r = 1.0 / p->rho0;                                  // ocean_parameters.F90:260
  const double gamma = p->pred_corr_gamma;
  if (PR) {
    a.c_pred = p->dtbt * gamma;                             // dtbt_gamma, :1195
    a.c_corr = p->dtbt;
  } else {
    a.c_pred = p->dtbt * gamma * a.rho0r;                   // dtbt_gamma_rho0r, :1196
    a.c_corr = p->dtbt * a.rho0r;                           // dtbt_rho0r, :1197
  }
  a.predict = (PR && CG) || gamma > 0.0;                    // press_cgrid has no gamma test
  a.initsum = p->initsum_with_bar ? 1 : 0;
  hipStream_t s = ctx->stream;
  const dim3 grid((d.NI + 63) / 64, d.NJ), block(64);
  const int nts = p->nts, hsub = blocked_depth<CG, PR>(ctx);
  const bool blocked = hsub > 0 && !d.cyclic_y && (!d.cyclic_x || d.ni >= MIN_NI);
  ctx->bt_subcycles_used = blocked ? hsub : 0;
  if (blocked) {
    const int rc = run_blocked(ctx, a, nts, p->stepping_a, hsub);
    if (rc) return rc;
  } else {
    hipLaunchKernelGGL((k_btv_init<CG, PR>), grid, block, 0, s, a);
    MOM_LAUNCHED(ctx, "k_btv_init");
    for (int itime = 1; itime <= nts; ++itime) {
      const int fstau = itime % 2 + 1, fstaup1 = (itime + 1) % 2 + 1;
      const int m2 = itime % 3 + 1, m1 = (itime + 1) % 3 + 1, m0 = (itime + 2) % 3 + 1;
      hipLaunchKernelGGL((k_btv_velocity<CG, PR>), grid, block, 0, s, a, fstau, fstaup1,
                         m0, m1, m2);
      const double wgt = p->stepping_a ? 0.0 : (double)(nts - itime + 1);
      hipLaunchKernelGGL((k_btv_corrector<CG, PR>), grid, block, 0, s, a, fstau, fstaup1,
                         wgt);
    }
    MOM_LAUNCHED(ctx, "k_btv_velocity/k_btv_corrector");
  }
  const double rntsp1 = 1.0 / ((double)nts + 1.0);          // :2804
  const double rnts = p->stepping_a ? 1.0 / (double)nts      // :2807-2811
                                    : 2.0 / ((double)nts * (double)(nts + 1));
  hipLaunchKernelGGL((k_btv_tail<CG, PR>), grid, block, 0, s, a, rntsp1, rnts,
                     v->x_bar_taup1, v->udrho_taup1, v->conv_rho_ud_t);
  MOM_LAUNCHED(ctx, "k_btv_tail");
  return MOM_GPU_OK;
}

}  // namespace

int launch_bt_variant(mom_gpu_ctx *ctx, const mom_gpu_bt_params_t *p,
                      const mom_gpu_bt_variant_t *v) {
  if (!ctx->btv) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    MOM_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cs));
    if (cs != hipStreamCaptureStatusNone)
      return mom_fail(ctx, MOM_GPU_ERR_ARG,
                      "update_ocean_barotropic_variant: the first call allocates its state; "
                      "call it once before capturing a graph");
    MOM_HIP(ctx, hipMalloc((void **)&ctx->btv, 22 * (size_t)ctx->kd.P2 * sizeof(double)));
  }
  if (v->cgrid)
    return v->pressure_based ? run_variant<true, true>(ctx, p, v) : run_variant<true, false>(ctx, p, v);
  return v->pressure_based ? run_variant<false, true>(ctx, p, v) : run_variant<false, false>(ctx, p, v);
}
