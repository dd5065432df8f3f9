// Split-explicit barotropic subcycle, B-grid, depth-based vertical
// coordinate: pred_corr_tropic_depth_bgrid (ocean_barotropic.F90:3225-3579)
// with barotropic_halo=1 and use_legacy_barotropic_halos=.true., and the
// time-averaging tail of update_ocean_barotropic (:2804-2811, :2846-2888).
//
// Everything is computed on the data domain, as the reference does.  The one
// halo exchange inside the loop (eta_t_bt after the predictor, :3383) is
// folded into the predictor: on a cyclic-x domain the halo columns of the
// compute rows take the value computed for the interior column they mirror.
#include "mom_internal.h"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace {

struct BtBuf {
  double *eta;    // eta_t_bt, 2 levels
  double *ud;     // udrho_bt, (2 components) x (2 levels)
  double *sf;     // steady_forcing
  double *cori1, *cori2;
};

__device__ inline double *ETA(const BtBuf &b, int P2, int lev) { return b.eta + (size_t)P2 * (lev - 1); }
__device__ inline double *UD(const BtBuf &b, int P2, int c, int lev) {
  return b.ud + (size_t)P2 * ((c - 1) + 2 * (lev - 1));
}

// DIV_UD (ocean_operators.F90:507-608, B-grid, non-legacy order) at the
// data-domain point (ii, jj); zero on the first row and column.
__device__ inline double div_ud(const KDom &d, const double *u1, const double *u2,
                                const double *dxu, const double *dyu, const double *datr,
                                int ii, int jj) {
  if (ii == 0 || jj == 0) return 0.0;
  const int o = ii + d.NI * jj, ojm = o - d.NI, oim = o - 1, oimjm = ojm - 1;
  const double uh = u1[o] * dyu[o], vh = u2[o] * dxu[o];
  const double uhjm = u1[ojm] * dyu[ojm], vhjm = u2[ojm] * dxu[ojm];
  const double uhim = u1[oim] * dyu[oim], vhim = u2[oim] * dxu[oim];
  const double uhimjm = u1[oimjm] * dyu[oimjm], vhimjm = u2[oimjm] * dxu[oimjm];
  const double uh_bay = 0.5 * (uh + uhjm);
  const double vh_bax = 0.5 * (vh + vhim);
  const double uhim_bay = 0.5 * (uhim + uhimjm);
  const double vhjm_bax = 0.5 * (vhjm + vhimjm);
  return ((uh_bay - uhim_bay) + (vh_bax - vhjm_bax)) * datr[o];
}

__global__ void k_bt_init(KDom d, BtBuf b, int initsum, double dtbt,
                          const double *__restrict__ eta_t, const double *__restrict__ eta_bar_tau,
                          const double *__restrict__ ud_tau, const double *__restrict__ pme,
                          const double *__restrict__ river, const double *__restrict__ source,
                          const double *__restrict__ eta_smooth, const double *__restrict__ f,
                          const int *__restrict__ kmt, double *__restrict__ eta_bar,
                          double *__restrict__ ud) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const int o = ii + d.NI * jj, P2 = d.P2;
  eta_bar[o] = initsum ? eta_bar_tau[o] : eta_t[o];
  ud[o] = 0.0;
  ud[o + P2] = 0.0;
  // itime = 1: fstau = mod(1,2)+1 = 2
  ETA(b, P2, 2)[o] = eta_bar_tau[o];
  UD(b, P2, 1, 2)[o] = ud_tau[o];
  UD(b, P2, 2, 2)[o] = ud_tau[o + P2];
  const double tm1 = (1 <= kmt[o]) ? 1.0 : 0.0;
  b.sf[o] = tm1 * (pme[o] + river[o] + source[o] - eta_smooth[o]);
  const double c1 = 0.5 * dtbt * f[o];       // ocean_barotropic.F90:1285-1286
  b.cori1[o] = c1;
  b.cori2[o] = 1.0 / (1.0 + c1 * c1);
}

// predictor for eta (:3365-3376) with the halo update (:3383) folded in
__global__ void k_bt_pred(KDom d, BtBuf b, int fstau, int fstaup1, double c_pred,
                          const double *__restrict__ dxu, const double *__restrict__ dyu,
                          const double *__restrict__ datr, const int *__restrict__ kmt) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const int P2 = d.P2;
  int si = ii;
  if (d.cyclic_x && jj >= 1 && jj <= d.NJ - 2) {
    if (ii == 0) si = d.NI - 2;
    else if (ii == d.NI - 1) si = 1;
  }
  const int os = si + d.NI * jj;
  const double tm1 = (1 <= kmt[os]) ? 1.0 : 0.0;
  const double tmp = -div_ud(d, UD(b, P2, 1, fstau), UD(b, P2, 2, fstau), dxu, dyu, datr, si, jj) * tm1;
  ETA(b, P2, fstaup1)[ii + d.NI * jj] = ETA(b, P2, fstau)[os] + c_pred * (tmp + b.sf[os]);
}

// surface pressure, its B-grid gradient (GRAD_BAROTROPIC_P,
// ocean_operators.F90:631-676) and the momentum update with implicit
// Coriolis (:3394-3486)
__global__ void k_bt_mom(KDom d, BtBuf b, int fstau, int fstaup1, double dtbt,
                         const double *__restrict__ rho_g, const double *__restrict__ patm,
                         const double *__restrict__ thicku, const double *__restrict__ forcing,
                         const double *__restrict__ f, const double *__restrict__ dxur,
                         const double *__restrict__ dyur, const int *__restrict__ kmu) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const int o = ii + d.NI * jj, P2 = d.P2;
  const double *eta = ETA(b, P2, fstaup1);
  double g1 = 0.0, g2 = 0.0;
  if (ii < d.NI - 1 && jj < d.NJ - 1) {
    const int oe = o + 1, on = o + d.NI, one = on + 1;
    const double p = rho_g[o] * eta[o] + patm[o];
    const double pe = rho_g[oe] * eta[oe] + patm[oe];
    const double pn = rho_g[on] * eta[on] + patm[on];
    const double pne = rho_g[one] * eta[one] + patm[one];
    const double p_fay = 0.5 * (p + pn);
    const double p_fax = 0.5 * (p + pe);
    const double pip_fay = 0.5 * (pe + pne);
    const double pjp_fax = 0.5 * (pn + pne);
    const double um = (1 <= kmu[o]) ? 1.0 : 0.0;
    g1 = (pip_fay - p_fay) * dxur[o] * um;
    g2 = (pjp_fax - p_fax) * dyur[o] * um;
  }
  const double pf1 = -(thicku[o] * g1);
  const double pf2 = -(thicku[o] * g2);
  const double u1 = UD(b, P2, 1, fstau)[o], u2 = UD(b, P2, 2, fstau)[o];
  const double t1 = u1 + dtbt * (0.5 * f[o] * u2 + pf1 + forcing[o] + 0.0);
  const double t2 = u2 + dtbt * (-(0.5 * f[o] * u1) + pf2 + forcing[o + P2] + 0.0);
  UD(b, P2, 1, fstaup1)[o] = b.cori2[o] * (t1 + b.cori1[o] * t2);
  UD(b, P2, 2, fstaup1)[o] = b.cori2[o] * (t2 - b.cori1[o] * t1);
}

// corrector (:3497-3505) and the accumulation for the time average
// (:3532-3549)
__global__ void k_bt_corr(KDom d, BtBuf b, int fstau, int fstaup1, double c_corr, int step_a,
                          double wgt, const double *__restrict__ dxu,
                          const double *__restrict__ dyu, const double *__restrict__ datr,
                          const int *__restrict__ kmt, double *__restrict__ eta_bar,
                          double *__restrict__ ud) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const int o = ii + d.NI * jj, P2 = d.P2;
  const double *u1 = UD(b, P2, 1, fstaup1), *u2 = UD(b, P2, 2, fstaup1);
  const double tm1 = (1 <= kmt[o]) ? 1.0 : 0.0;
  const double tmp = -div_ud(d, u1, u2, dxu, dyu, datr, ii, jj) * tm1;
  const double e = ETA(b, P2, fstau)[o] + c_corr * (tmp + b.sf[o]);
  ETA(b, P2, fstaup1)[o] = e;
  eta_bar[o] = eta_bar[o] + e;
  if (step_a) {
    ud[o] = ud[o] + u1[o];
    ud[o + P2] = ud[o + P2] + u2[o];
  } else {
    ud[o] = ud[o] + wgt * u1[o];
    ud[o + P2] = ud[o + P2] + wgt * u2[o];
  }
}

__global__ void k_bt_scale(KDom d, double rntsp1, double rnts, double *__restrict__ eta_bar,
                           double *__restrict__ ud) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const int o = ii + d.NI * jj;
  eta_bar[o] = rntsp1 * eta_bar[o];
  ud[o] = rnts * ud[o];
  ud[o + d.P2] = rnts * ud[o + d.P2];
}

// mpp_update_domains on a cyclic-x single domain: E/W halo columns of the
// compute rows (ncomp planes)
__global__ void k_bt_wrap(KDom d, double *__restrict__ a, int ncomp) {
  const int jj = blockIdx.x * blockDim.x + threadIdx.x + 1;
  if (jj > d.NJ - 2) return;
  for (int c = 0; c < ncomp; ++c) {
    double *p = a + (size_t)d.P2 * c + (size_t)d.NI * jj;
    p[0] = p[d.NI - 2];
    p[d.NI - 1] = p[1];
  }
}

__global__ void k_bt_conv(KDom d, const double *__restrict__ ud, const double *__restrict__ dxu,
                          const double *__restrict__ dyu, const double *__restrict__ datr,
                          double *__restrict__ conv) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  conv[ii + d.NI * jj] = -div_ud(d, ud, ud + d.P2, dxu, dyu, datr, ii, jj);
}

// ---- temporally blocked subcycles -----------------------------------------
// One work-group owns a BRY x BRX region of the data domain and advances it
// nsub subcycles with the state (eta, U) and the accumulators in registers
// and only the exchanged quantities (U*dyu, U*dxu, surface pressure) in
// LDS.  Per subcycle the velocity's exact region shrinks by one point on
// each side (its pressure gradient reaches one point up, the divergence in
// that pressure one point down) and the height, formed from the divergence
// of the new velocity, lags one more point on the low side: after nsub
// subcycles the points from nsub + 1 above the region's low edges to nsub
// below its high edges are exact, an interior of (BRY-2*nsub-1) x
// (BRX-2*nsub-1); the rest is recomputed by the neighbouring groups.  On a
// cyclic-x domain the region addresses the
// periodic images of the compute columns: with the inputs' halo columns
// holding the wrap (what mpp_update_domains leaves), this reproduces the
// reference's evolution of every point, the halo columns of the compute
// rows excepted -- those are rewritten by the tail's halo update anyway.
constexpr int BRX = 64;          // region columns (one wavefront per row)
constexpr int BRY = 32;          // region rows
constexpr int BPT = 2;           // region rows per wavefront
constexpr int BNT = BRX * BRY / BPT;

// the halo a region keeps below its interior, and the interior's extent, for
// nsub subcycles
__host__ __device__ constexpr int bt_lo(int nsub) { return nsub + 1; }
__host__ __device__ constexpr int bt_interior(int n, int nsub) { return n - 2 * nsub - 1; }

// sf: tmask * (pme + river + source - eta_smooth) and mask: bit 0 tmask(k=1),
// bit 1 umask(k=1), formed once per call by k_bt_prep (constant over the
// subcycles) instead of being re-read from their six sources by every launch
struct BtIn {
  const double *rho_g, *patm, *thicku, *forcing, *f;
  const double *dxu, *dyu, *datr, *dxur, *dyur;
  const double *sf;
  const unsigned char *mask;
  const double *rowc;   // per row: datr, dyu/2, dxu/2, dxur/2, dyur/2, cori1, cori2,
                         // f/2 (or null)
  int recip;   // dxur, dyur formed as 1/(dxu + epsln), 1/(dyu + epsln), not loaded
};

constexpr double EPSLN_GRID = 1.0e-40;   // shared/constants/constants.F90:123

// Per data-domain point: bit 0 where dxur or dyur is not, bit for bit, the
// reciprocal ocean_grids.F90:949-951 forms; bit 1 where a metric the blocked
// barotropic multiplies is outside LAND_BOUND in magnitude (or not a number)
// or dxu, dyu, datr carries a sign bit; bit 2 where a metric bt_rows_tile takes from
// its row differs from the row's first point; bit 3 where one of those or of the
// C-grid variants' does.  The host ORs them up.
constexpr double LAND_BOUND = 1.0e100;
__device__ inline bool bounded(double x) { return fabs(x) <= LAND_BOUND; }
__global__ void k_check_recip(KDom d, const double *__restrict__ dxu,
                              const double *__restrict__ dxur, const double *__restrict__ dyu,
                              const double *__restrict__ dyur, const double *__restrict__ datr,
                              const double *__restrict__ f, const double *__restrict__ dat,
                              const double *__restrict__ dxte, const double *__restrict__ dytn,
                              int *__restrict__ bad) {
  auto differ = [](double a, double b) {
    return __builtin_bit_cast(unsigned long long, a) != __builtin_bit_cast(unsigned long long, b);
  };
  const int ii = blockIdx.x * blockDim.x + threadIdx.x;
  const int o = ii + d.NI * blockIdx.y;
  if (ii >= d.NI) return;
  const double rx = 1.0 / (dxu[o] + EPSLN_GRID), ry = 1.0 / (dyu[o] + EPSLN_GRID);
  const bool recip_bad = (__builtin_bit_cast(unsigned long long, rx) !=
                          __builtin_bit_cast(unsigned long long, dxur[o])) ||
                         (__builtin_bit_cast(unsigned long long, ry) !=
                          __builtin_bit_cast(unsigned long long, dyur[o]));
  const bool grid_bad = !(bounded(dxu[o]) && bounded(dyu[o]) && bounded(datr[o]) &&
                          bounded(dxur[o]) && bounded(dyur[o]) && bounded(f[o]) &&
                          !signbit(dxu[o]) && !signbit(dyu[o]) && !signbit(datr[o]));
  const int r = d.NI * blockIdx.y;
  const bool row_bad = differ(dxu[o], dxu[r]) || differ(dyu[o], dyu[r]) ||
                       differ(dxur[o], dxur[r]) || differ(dyur[o], dyur[r]) ||
                       differ(datr[o], datr[r]) || differ(f[o], f[r]);
  const bool crow_bad = row_bad || differ(dat[o], dat[r]) || differ(dxte[o], dxte[r]) ||
                        differ(dytn[o], dytn[r]);
  bad[o] = (recip_bad ? 1 : 0) | (grid_bad ? 2 : 0) | (row_bad ? 4 : 0) | (crow_bad ? 8 : 0);
}

// The per-call inputs that decide whether a point is inert under the
// subcycles (mask bit 2); null in Inert::eta: no point is.
struct Inert {
  const double *eta, *ud, *forcing, *rho_g, *patm, *thicku;
};
// What a call forms once: sf and the masks of every point and, for domains whose
// rows are uniform in x (rowc not null), each row's constants.
struct BtPrep {
  KDom d;
  const double *pme, *river, *source, *eta_smooth;
  const int *kmt, *kmu;
  double *sf;
  unsigned char *mask;
  Inert x;
  const double *datr, *dyu, *dxu, *dxur, *dyur, *f;
  double dtbt;
  double *rowc;
};
__device__ __forceinline__ void bt_prep(const BtPrep &P, int ii, int jj) {
  const KDom &d = P.d;
  const Inert &x = P.x;
  const int o = ii + d.NI * jj;
  const double tm = (1 <= P.kmt[o]) ? 1.0 : 0.0;
  const double s = tm * (P.pme[o] + P.river[o] + P.source[o] - P.eta_smooth[o]);
  P.sf[o] = s;
  const bool t = 1 <= P.kmt[o], u = 1 <= P.kmu[o];
  // inert: both masks 0, forcing and velocity zeros (either sign), sf a
  // zero, the fields multiplied into the pressure bounded
  const size_t P2 = (size_t)d.P2;
  const bool inert = x.eta && !t && !u && s == 0.0 && x.forcing[o] == 0.0 &&
                     x.forcing[o + P2] == 0.0 && x.ud[o] == 0.0 && x.ud[o + P2] == 0.0 &&
                     bounded(x.eta[o]) && bounded(x.rho_g[o]) && bounded(x.patm[o]) &&
                     bounded(x.thicku[o]);
  P.mask[o] = (unsigned char)((t ? 1 : 0) | (u ? 2 : 0) | (inert ? 4 : 0));
  if (P.rowc && ii == 0) {
    double *r = P.rowc + (size_t)8 * jj;
    const double fo = P.f[o], c1 = 0.5 * P.dtbt * fo;     // cori1, cori2 (:1285-1286)
    r[0] = P.datr[o]; r[1] = 0.5 * P.dyu[o]; r[2] = 0.5 * P.dxu[o];
    r[3] = 0.5 * P.dxur[o]; r[4] = 0.5 * P.dyur[o];
    r[5] = c1; r[6] = 1.0 / (1.0 + c1 * c1); r[7] = 0.5 * fo;
  }
}
__global__ void k_bt_prep(BtPrep P) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x;
  if (ii < P.d.NI) bt_prep(P, ii, blockIdx.y);
}
// ensembles: blockIdx.z is the domain
__global__ void k_bt_prep_ens(const BtPrep *__restrict__ Ps) {
  const BtPrep &P = Ps[blockIdx.z];
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii < P.d.NI && jj < P.d.NJ) bt_prep(P, ii, jj);
}

// One launch of the blocked subcycle for one domain: nsub subcycles from s0.
struct BtJob {
  KDom d;
  BtIn in;
  const double *eta_src, *ud_src;
  const double *eb_src, *ub_src;   // the time sums so far (ub_src null: zero, the first launch)
  double *eta_dst, *ud_dst, *eb, *ub;
  int s0, nsub, nts, step_a;
  double dtbt, cp, cc;
  int xbase, xcount, ntx, ntiles, rev;
  const int *land;   // per tile: 1 where bt_tile may take its land path (null: none)
};

// Land path of a tile (a region of ry rows): every point of the region is inert
// (k_bt_prep, mask bit 2).  There the velocity after each momentum phase is +0
// (the pressure gradient is x*0.0, the forcing and the old velocity zeros,
// dtbt > 0, and the Coriolis factors finite), so U*dyu and U*dxu are +0 with
// dxu, dyu >= +0 and the divergence is +0; the corrector adds
// cc*(-0*0.0 + sf) = cc*sf, a signed zero, to eta, and the time sums add eta and
// +0.  The velocity sums start the call at +0 and every subcycle adds +0 to them
// in either path.  The same values as the full path.
__device__ __forceinline__ void bt_land_tile(const BtJob &J, int ry, int x_int0, int y_int0) {
  const KDom d = J.d;
  const bool cyc = d.cyclic_x != 0;
  const int TX = bt_interior(BRX, J.nsub), TY = bt_interior(ry, J.nsub), LO = bt_lo(J.nsub);
  const int lane = threadIdx.x % BRX;
  const int vi = x_int0 - LO + lane;
  const int col = cyc ? 1 + wrapi(vi - 1, d.ni) : vi;
  for (int r = threadIdx.x / BRX; r < ry; r += blockDim.x / BRX) {
    const int j = y_int0 - LO + r;
    const bool inside = (cyc || (vi >= 0 && vi < d.NI)) && j >= 0 && j < d.NJ && lane >= LO &&
                        lane < LO + TX && vi < J.xbase + J.xcount && r >= LO && r < LO + TY;
    if (!inside) continue;
    const int o = col + d.NI * j;
    double e = J.eta_src[o], ebq = J.eb_src[o];
    const double s = J.in.sf[o];
    for (int t = 0; t < J.nsub; ++t) {
      e = e + J.cc * s;
      ebq = ebq + e;
    }
    J.eta_dst[o] = e;
    J.ud_dst[o] = 0.0;
    J.ud_dst[o + d.P2] = 0.0;
    J.eb[o] = ebq;
    if (!J.ub_src) {
      J.ub[o] = 0.0;
      J.ub[o + d.P2] = 0.0;
    }
  }
}

__device__ __forceinline__ void bt_tile(const BtJob &J, int tile) {
  const KDom d = J.d;
  const BtIn &in = J.in;
  const double *__restrict__ eta_src = J.eta_src;
  const double *__restrict__ ud_src = J.ud_src;
  double *__restrict__ eta_dst = J.eta_dst;
  double *__restrict__ ud_dst = J.ud_dst;
  // (a launch after the first reads the sums it writes)
  const double *eb_src = J.eb_src, *ub_src = J.ub_src;
  double *eb = J.eb;
  double *ub = J.ub;
  const int s0 = J.s0, nsub = J.nsub, nts = J.nts, step_a = J.step_a;
  const double dtbt = J.dtbt, cp = J.cp, cc = J.cc;
  const int xbase = J.xbase, xcount = J.xcount, ntx = J.ntx;
  __shared__ double s_ps[BRY][BRX];
  __shared__ double s_uh[BRY][BRX];
  __shared__ double s_vh[BRY][BRX];
  const int TX = bt_interior(BRX, nsub), TY = bt_interior(BRY, nsub), LO = bt_lo(nsub);
  const int tix = tile % ntx, tiy = tile / ntx;
  const int x_int0 = xbase + tix * TX, y_int0 = tiy * TY;
  const int lane = threadIdx.x % BRX, wave = threadIdx.x / BRX;
  const int P2 = d.P2;
  const bool cyc = d.cyclic_x != 0;

  if (J.land && J.land[tile]) {
    bt_land_tile(J, BRY, x_int0, y_int0);
    return;
  }

  int rr[BPT], off[BPT], vj[BPT];
  bool present[BPT], interior[BPT], div0[BPT], grad0[BPT];
  double eta[BPT], u1[BPT], u2[BPT], ebv[BPT], ub1[BPT], ub2[BPT];
  // tmask and umask at k = 1 as lane masks: x*mask is x where the mask is 1
  // and x*0.0 where it is 0 (the same bits as multiplying by the 0/1 double)
  bool tmb[BPT], umb[BPT];
  double sf[BPT], datr[BPT], dyu[BPT], dxu[BPT], rho_g[BPT], patm[BPT], thk[BPT];
  double F1[BPT], F2[BPT], fc[BPT], cori1[BPT], cori2[BPT], dxur[BPT], dyur[BPT];
  const int vi = x_int0 - LO + lane;
  int col = vi;
  bool colok = true;
  if (cyc) col = 1 + wrapi(vi - 1, d.ni);
  else colok = vi >= 0 && vi < d.NI;
#pragma unroll
  for (int q = 0; q < BPT; ++q) {
    const int r = wave + (BNT / BRX) * q;
    rr[q] = r;
    const int j = y_int0 - LO + r;
    vj[q] = j;
    present[q] = colok && j >= 0 && j < d.NJ;
    interior[q] = present[q] && lane >= LO && lane < LO + TX &&
                  vi < xbase + xcount && r >= LO && r < LO + TY;
    div0[q] = (j == 0) || (!cyc && vi == 0);
    grad0[q] = (j == d.NJ - 1) || (!cyc && vi == d.NI - 1);
    const int o = present[q] ? col + d.NI * j : 0;
    off[q] = o;
    if (present[q]) {
      const unsigned char mb = in.mask[o];
      tmb[q] = (mb & 1) != 0;
      sf[q] = in.sf[o];
      datr[q] = in.datr[o]; dyu[q] = in.dyu[o]; dxu[q] = in.dxu[o];
      rho_g[q] = in.rho_g[o]; patm[q] = in.patm[o]; thk[q] = in.thicku[o];
      F1[q] = in.forcing[o]; F2[q] = in.forcing[o + P2]; fc[q] = in.f[o];
      cori1[q] = 0.5 * dtbt * fc[q];
      cori2[q] = 1.0 / (1.0 + cori1[q] * cori1[q]);
      if (in.recip) {
        dxur[q] = 1.0 / (dxu[q] + EPSLN_GRID);
        dyur[q] = 1.0 / (dyu[q] + EPSLN_GRID);
      } else {
        dxur[q] = in.dxur[o]; dyur[q] = in.dyur[o];
      }
      umb[q] = (mb & 2) != 0;
      eta[q] = eta_src[o]; u1[q] = ud_src[o]; u2[q] = ud_src[o + P2];
      ebv[q] = ub1[q] = ub2[q] = 0.0;
      if (interior[q]) {
        ebv[q] = eb_src[o];
        if (ub_src) { ub1[q] = ub_src[o]; ub2[q] = ub_src[o + P2]; }
      }
    } else {
      tmb[q] = umb[q] = false;
      sf[q] = datr[q] = dyu[q] = dxu[q] = rho_g[q] = patm[q] = thk[q] = 0.0;
      F1[q] = F2[q] = fc[q] = cori1[q] = cori2[q] = dxur[q] = dyur[q] = 0.0;
      eta[q] = u1[q] = u2[q] = ebv[q] = ub1[q] = ub2[q] = 0.0;
    }
    s_uh[r][lane] = u1[q] * dyu[q];
    s_vh[r][lane] = u2[q] * dxu[q];
  }
  __syncthreads();

  const int lm = max(lane - 1, 0), lp = min(lane + 1, BRX - 1);
  // The divergence of U*dy, U*dx at each point.  Phase A of a subcycle needs
  // the divergence of the velocity phase C of the previous subcycle formed,
  // from the same LDS values by the same operations, so it is carried over;
  // only the first subcycle of a launch forms it from the loaded velocity.
  double dv[BPT];
#pragma unroll
  for (int q = 0; q < BPT; ++q) {
    const int r = rr[q], rm = max(r - 1, 0);
    dv[q] = 0.0;
    if (!div0[q]) {
      const double uh_bay = 0.5 * (s_uh[r][lane] + s_uh[rm][lane]);
      const double vh_bax = 0.5 * (s_vh[r][lane] + s_vh[r][lm]);
      const double uhim_bay = 0.5 * (s_uh[r][lm] + s_uh[rm][lm]);
      const double vhjm_bax = 0.5 * (s_vh[rm][lane] + s_vh[rm][lm]);
      dv[q] = ((uh_bay - uhim_bay) + (vh_bax - vhjm_bax)) * datr[q];
    }
  }
  for (int t = 0; t < nsub; ++t) {
    const int itime = s0 + t;
    // A: predictor and surface pressure
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const int r = rr[q];
      const double tmp = tmb[q] ? -dv[q] : -dv[q] * 0.0;
      const double es = eta[q] + cp * (tmp + sf[q]);
      s_ps[r][lane] = rho_g[q] * es + patm[q];
    }
    __syncthreads();
    // B: pressure gradient and momentum with implicit Coriolis
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const int r = rr[q], rp = min(r + 1, BRY - 1);
      double g1 = 0.0, g2 = 0.0;
      if (!grad0[q]) {
        const double p = s_ps[r][lane], pe = s_ps[r][lp];
        const double pn = s_ps[rp][lane], pne = s_ps[rp][lp];
        const double p_fay = 0.5 * (p + pn);
        const double p_fax = 0.5 * (p + pe);
        const double pip_fay = 0.5 * (pe + pne);
        const double pjp_fax = 0.5 * (pn + pne);
        const double x1 = (pip_fay - p_fay) * dxur[q];
        const double x2 = (pjp_fax - p_fax) * dyur[q];
        g1 = umb[q] ? x1 : x1 * 0.0;
        g2 = umb[q] ? x2 : x2 * 0.0;
      }
      const double pf1 = -(thk[q] * g1);
      const double pf2 = -(thk[q] * g2);
      const double t1 = u1[q] + dtbt * (0.5 * fc[q] * u2[q] + pf1 + F1[q] + 0.0);
      const double t2 = u2[q] + dtbt * (-(0.5 * fc[q] * u1[q]) + pf2 + F2[q] + 0.0);
      u1[q] = cori2[q] * (t1 + cori1[q] * t2);
      u2[q] = cori2[q] * (t2 - cori1[q] * t1);
      // the previous phase C's reads of s_uh/s_vh finished before the barrier above
      s_uh[r][lane] = u1[q] * dyu[q];
      s_vh[r][lane] = u2[q] * dxu[q];
    }
    __syncthreads();
    // C: corrector and time-average accumulation
    const double wgt = (double)(nts - itime + 1);
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const int r = rr[q], rm = max(r - 1, 0);
      double div = 0.0;
      if (!div0[q]) {
        const double uh_bay = 0.5 * (s_uh[r][lane] + s_uh[rm][lane]);
        const double vh_bax = 0.5 * (s_vh[r][lane] + s_vh[r][lm]);
        const double uhim_bay = 0.5 * (s_uh[r][lm] + s_uh[rm][lm]);
        const double vhjm_bax = 0.5 * (s_vh[rm][lane] + s_vh[rm][lm]);
        div = ((uh_bay - uhim_bay) + (vh_bax - vhjm_bax)) * datr[q];
      }
      dv[q] = div;
      const double tmp = tmb[q] ? -div : -div * 0.0;
      eta[q] = eta[q] + cc * (tmp + sf[q]);
      ebv[q] = ebv[q] + eta[q];
      if (step_a) {
        ub1[q] = ub1[q] + u1[q];
        ub2[q] = ub2[q] + u2[q];
      } else {
        ub1[q] = ub1[q] + wgt * u1[q];
        ub2[q] = ub2[q] + wgt * u2[q];
      }
    }
  }
#pragma unroll
  for (int q = 0; q < BPT; ++q) {
    if (interior[q]) {
      const int o = off[q];
      eta_dst[o] = eta[q];
      ud_dst[o] = u1[q];
      ud_dst[o + P2] = u2[q];
      eb[o] = ebv[q];
      ub[o] = ub1[q];
      ub[o + P2] = ub2[q];
    }
  }
}

// 1 for a tile of nsub subcycles whose whole region (the points bt_tile
// loads) is inert, 0 otherwise: one work-group a tile.
__global__ __launch_bounds__(256) void k_bt_land(KDom d, const unsigned char *__restrict__ mask,
                                                 int ry, int nsub, int xbase, int ntx,
                                                 int ntiles, int *__restrict__ land) {
  const int tile = blockIdx.x;
  if (tile >= ntiles) return;                  // the whole block
  const int TX = bt_interior(BRX, nsub), TY = bt_interior(ry, nsub), LO = bt_lo(nsub);
  const int x_int0 = xbase + (tile % ntx) * TX, y_int0 = (tile / ntx) * TY;
  const int lane = threadIdx.x % BRX;
  const int vi = x_int0 - LO + lane;
  const bool cyc = d.cyclic_x != 0;
  const int col = cyc ? 1 + wrapi(vi - 1, d.ni) : vi;
  const bool colok = cyc || (vi >= 0 && vi < d.NI);
  int ok = 1;
  for (int r = threadIdx.x / BRX; r < ry; r += 256 / BRX) {
    const int j = y_int0 - LO + r;
    if (colok && j >= 0 && j < d.NJ && !(mask[col + d.NI * j] & 4)) ok = 0;
  }
  ok = __syncthreads_and(ok);
  if (threadIdx.x == 0) land[tile] = ok;
}

// bt_tile for a domain whose dxu, dyu, datr, dxur, dyur and f are the same, bit for
// bit, along every row (spherical grids: launch_check_recip).  A row's constants
// are then wavefront-uniform and need no vector register a lane: they lie in scalar
// registers, as far as those reach (the compiler keeps 35 of them in lanes of vector
// registers with three rows a wavefront and 109 with four, whose instance
// also has 12 B of scratch).  x neighbours come by
// lane shifts, y neighbours from the thread's own rows but for one row a
// wavefront each way (LDS).  What bounds it: memory a launch (18 planes once, the
// nine of them that regions share up to twice) against 54 FP64 instructions a
// point and subcycle, so a region wants many subcycles (fewer launches) and few
// redundant points, and two blocks share a CU so that one loads while the other
// steps: 8 wavefronts of 3 rows (64 x 24) or 4 (64 x 32, thickness and forcing in
// LDS).  3600 x 2700, 120 subcycles, ms at the best depth: bt_tile 13.7 (5); one
// block of 16 wavefronts, 2 rows 9.8 (6), 3 rows 8.2 (7), 4 rows 8.1 (10); 12
// wavefronts of 2 rows 11.6 (5), 10 of 3 rows 11.0 (6); 8 of 3 rows 8.4 (6), 8 of
// 4 rows 8.0 (6), 7.8 with every other launch backwards.  517 x 389, 80
// subcycles: 286 us (bt_tile) to 254 alone, 241 to 121 among three states in turn
// (bt_plan).
// The same values as bt_tile, instructions saved:
// - tmask into datr and umask into thicku: x*m is x or a zero of x's sign, as is
//   the product's (a NaN stays one); the pressure force's zero loses its sign in
//   the sum with forcing + 0.0, which is never -0;
// - 0.5*(a + b) and its differences: the halves are in the row constants
//   (a power of two, exact short of the subnormals);
// - the corrector's divergence is the next predictor's.
// Regions inside the domain skip the edge rows' and columns' tests (EDGE).
// Points outside the domain read a clamped place: no value of theirs reaches a
// point inside (the divergence is 0 on the first row and column, the gradient on
// the last).
template <int R, int NW>
struct BtRowsLds {
  // four rows: thickness and forcing in LDS (own lane)
  static constexpr bool CL = R >= 4;
  double p[NW][BRX], u[NW][BRX], v[NW][BRX];
  double c[CL ? 3 : 1][CL ? R : 1][CL ? NW : 1][BRX];
};
template <int R, int NW, bool EDGE>
__device__ __forceinline__ void bt_rows_tile(const BtJob &J, int x_int0, int y_int0,
                                             BtRowsLds<R, NW> &S) {
  constexpr int RY = NW * R;
  constexpr bool CL = BtRowsLds<R, NW>::CL;
  const KDom d = J.d;
  const int nsub = J.nsub, P2 = d.P2;
  const bool cyc = d.cyclic_x != 0;
  auto &s_p = S.p, &s_u = S.u, &s_v = S.v;
  auto &s_c = S.c;
  const int TX = bt_interior(BRX, nsub), TY = bt_interior(RY, nsub), LO = bt_lo(nsub);
  const int lane = threadIdx.x & (BRX - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / BRX);
  const int wm = max(wave - 1, 0), wp = min(wave + 1, NW - 1);
  const int vi = x_int0 - LO + lane;
  int col;
  if (!cyc) {
    col = min(max(vi, 0), d.NI - 1);
  } else if (d.ni >= 2 * BRX) {
    int g = vi - 1;
    g = g < 0 ? g + d.ni : g;
    col = 1 + (g >= d.ni ? g - d.ni : g);
  } else {
    col = 1 + wrapi(vi - 1, d.ni);
  }
  const unsigned cb = (unsigned)col * 8u;
  const bool lin = lane >= LO && lane < LO + TX && vi < J.xbase + J.xcount;
  const int row0 = y_int0 - LO + R * wave;
  typedef const __attribute__((address_space(4))) double ConstD;
  double eta[R], u1[R], u2[R], eb[R], ub1[R], ub2[R], g[R], uh[R], vh[R];
  double sf[R], rg[R], pa[R], th[CL ? 1 : R], F1[CL ? 1 : R], F2[CL ? 1 : R];
  double dm[R];                                                       // datr*tmask
  double hdyu[R], hdxu[R], hdxur[R], hdyur[R], c1[R], c2[R], hf[R];   // uniform
  auto inside = [&](int q) {
    const int r = R * wave + q;
    return lin && row0 + q >= 0 && row0 + q < d.NJ && r >= LO && r < LO + TY;
  };
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int j = row0 + q, jc = min(max(j, 0), d.NJ - 1);      // uniform
    const int ro = d.NI * jc;
    ConstD *rc = (ConstD *)(unsigned long long)(J.in.rowc + (size_t)8 * jc);
    hdyu[q] = rc[1]; hdxu[q] = rc[2]; hdxur[q] = rc[3]; hdyur[q] = rc[4];
    c1[q] = rc[5]; c2[q] = rc[6]; hf[q] = rc[7];
    const unsigned char mb = J.in.mask[ro + col];
    eta[q] = ld_lv(J.eta_src + ro, cb);
    u1[q] = ld_lv(J.ud_src + ro, cb);
    u2[q] = ld_lv(J.ud_src + P2 + ro, cb);
    sf[q] = ld_lv(J.in.sf + ro, cb);
    rg[q] = ld_lv(J.in.rho_g + ro, cb);
    pa[q] = ld_lv(J.in.patm + ro, cb);
    // datr*tmask; thicku*umask; the forcing + 0.0
    dm[q] = rc[0] * ((mb & 1) ? 1.0 : 0.0);
    const double tq = ld_lv(J.in.thicku + ro, cb) * ((mb & 2) ? 1.0 : 0.0),
                 f1q = ld_lv(J.in.forcing + ro, cb) + 0.0,
                 f2q = ld_lv(J.in.forcing + P2 + ro, cb) + 0.0;
    if constexpr (CL) {
      s_c[0][q][wave][lane] = tq;
      s_c[1][q][wave][lane] = f1q;
      s_c[2][q][wave][lane] = f2q;
    } else {
      th[q] = tq; F1[q] = f1q; F2[q] = f2q;
    }
    eb[q] = ub1[q] = ub2[q] = 0.0;
    if (inside(q)) {
      eb[q] = ld_lv(J.eb_src + ro, cb);
      if (J.ub_src) {
        ub1[q] = ld_lv(J.ub_src + ro, cb);
        ub2[q] = ld_lv(J.ub_src + P2 + ro, cb);
      }
    }
  }
  auto share = [&]() {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      uh[q] = u1[q] * hdyu[q];
      vh[q] = u2[q] * hdxu[q];
    }
    s_u[wave][lane] = uh[R - 1];
    s_v[wave][lane] = vh[R - 1];
  };
  // g = -DIV_UD*tmask + sf.  bay(row) = (uh(row) + uh(row - 1))/2 and
  // bax(row) = (vh + vh west)/2; the halves are in dyu and dxu
  auto diverge = [&]() {
    double bx = s_v[wm][lane], um = s_u[wm][lane];
    bx = bx + lane_prev(bx);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double bay = uh[q] + um, bax = vh[q] + lane_prev(vh[q]);
      double dv = ((bay - lane_prev(bay)) + (bax - bx)) * dm[q];
      if (EDGE && (row0 + q == 0 || (!cyc && vi == 0))) dv = 0.0;
      g[q] = sf[q] - dv;
      um = uh[q];
      bx = bax;
    }
  };
  share();
  __syncthreads();
  diverge();
  for (int t = 0; t < nsub; ++t) {
    // A: predictor and surface pressure
    double p[R + 1];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double es = eta[q] + J.cp * g[q];
      p[q] = rg[q] * es + pa[q];
    }
    s_p[wave][lane] = p[0];
    __syncthreads();
    // B: pressure gradient (the halves are in dxur and dyur) and momentum with
    // implicit Coriolis
    p[R] = s_p[wp][lane];
    double pe = lane_next(p[0]), fax = p[0] + pe;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double pne = lane_next(p[q + 1]);
      const double fay = p[q] + p[q + 1], pip = pe + pne, pjp = p[q + 1] + pne;
      double g1 = (pip - fay) * hdxur[q], g2 = (pjp - fax) * hdyur[q];
      if (EDGE && (row0 + q == d.NJ - 1 || (!cyc && vi == d.NI - 1))) g1 = g2 = 0.0;
      double thq, f1q, f2q;
      if constexpr (CL) {
        thq = s_c[0][q][wave][lane]; f1q = s_c[1][q][wave][lane]; f2q = s_c[2][q][wave][lane];
      } else {
        thq = th[q]; f1q = F1[q]; f2q = F2[q];
      }
      const double t1 = u1[q] + J.dtbt * (hf[q] * u2[q] - thq * g1 + f1q);
      const double t2 = u2[q] + J.dtbt * (-(hf[q] * u1[q]) - thq * g2 + f2q);
      u1[q] = c2[q] * (t1 + c1[q] * t2);
      u2[q] = c2[q] * (t2 - c1[q] * t1);
      pe = pne;
      fax = pjp;
    }
    share();      // the previous phase C's reads finished before the barrier above
    __syncthreads();
    // C: corrector and time-average accumulation
    diverge();
#pragma unroll
    for (int q = 0; q < R; ++q) {
      eta[q] = eta[q] + J.cc * g[q];
      eb[q] = eb[q] + eta[q];
    }
    const double wgt = J.step_a ? 1.0 : (double)(J.nts - (J.s0 + t) + 1);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      ub1[q] = ub1[q] + wgt * u1[q];
      ub2[q] = ub2[q] + wgt * u2[q];
    }
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    if (!inside(q)) continue;
    const int ro = d.NI * (row0 + q);
    st_lv(J.eta_dst + ro, cb, eta[q]);
    st_lv(J.ud_dst + ro, cb, u1[q]);
    st_lv(J.ud_dst + P2 + ro, cb, u2[q]);
    st_lv(J.eb + ro, cb, eb[q]);
    st_lv(J.ub + ro, cb, ub1[q]);
    st_lv(J.ub + P2 + ro, cb, ub2[q]);
  }
}

// The tiles: bt_tile, or bt_rows_tile of 8 wavefronts with 3 or 4 rows each
constexpr int BT_ANY = 0, BT_ROWS3 = 3, BT_ROWS4 = 4;
__host__ __device__ constexpr int bt_nw(int tile) { return tile == BT_ANY ? BNT / 64 : 8; }
__host__ __device__ constexpr int bt_ry(int tile) { return tile == BT_ANY ? BRY : 8 * tile; }
template <int T>
__device__ __forceinline__ void bt_any_tile(const BtJob &J, int tile) {
  if constexpr (T == BT_ANY) {
    bt_tile(J, tile);
  } else {
    constexpr int NW = bt_nw(T), RY = bt_ry(T);
    __shared__ BtRowsLds<T, NW> lds;
    const KDom &d = J.d;
    const int LO = bt_lo(J.nsub);
    const int x0 = J.xbase + (tile % J.ntx) * bt_interior(BRX, J.nsub);
    const int y0 = (tile / J.ntx) * bt_interior(RY, J.nsub);
    // a region that meets the first row or column (divergence 0) or the last
    // (gradient 0)
    const bool edge = y0 - LO <= 0 || y0 - LO + RY >= d.NJ ||
                      (!d.cyclic_x && (x0 - LO <= 0 || x0 - LO + BRX >= d.NI));
    if (J.land && J.land[tile]) bt_land_tile(J, RY, x0, y0);
    else if (edge) bt_rows_tile<T, NW, true>(J, x0, y0, lds);
    else bt_rows_tile<T, NW, false>(J, x0, y0, lds);
  }
}

// Tiles in XCD-aware order: blocks are dealt to the 8 XCDs round-robin, so
// each XCD takes per_xcd consecutive positions of the order of 8-wide strips
// (strip_tile) and the halo rows and columns that neighbouring tiles both
// read are fetched into one L2.
template <int T>
__global__ __launch_bounds__(64 * bt_nw(T), 4) void k_bt_block(BtJob J, int per_xcd) {
  const int b = blockIdx.x;
  // bt_rows_tile: every other launch goes backwards, the planes the last tiles of
  // one launch wrote are in the cache for the first tiles of the next (3600x2700,
  // 120 subcycles 8.0 to 7.8 ms; bt_tile, bound by its loads from L2: 15.8 to 16.5)
  const int i = J.rev ? per_xcd - 1 - (b >> 3) : b >> 3;
  const int t = (b & 7) * per_xcd + i;
  if (t >= J.ntiles) return;
  bt_any_tile<T>(J, strip_tile<8>(t, J.ntx, J.ntiles / J.ntx));
}

// Ensemble: launch ell of every domain that still has subcycles; the static
// per-domain part is a device table, the per-launch tile prefix an argument.
constexpr int BT_MAXDOM = 64;
struct BtDom {
  KDom d;
  BtIn in;
  const double *eta_bar_tau, *ud_tau, *eb0;   // the first launch's state and height sum
  double *eta_buf[2], *ud_buf[2];
  double *eb, *ub;
  int nts, step_a;
  double dtbt, cp, cc;
  int xbase, xcount;
};
struct BtLaunch {
  int first[BT_MAXDOM + 1];   // first tile of each domain in this launch
  int ndom, ell, hsub, ry;
};

__device__ __host__ inline void bt_shape(const BtDom &D, const BtLaunch &L, int &nsub, int &ntx,
                                         int &ntiles) {
  const int left = D.nts - L.ell * L.hsub;
  nsub = left < L.hsub ? left : L.hsub;
  if (nsub <= 0) { nsub = 0; ntx = 0; ntiles = 0; return; }
  const int TX = bt_interior(BRX, nsub), TY = bt_interior(L.ry, nsub);
  ntx = (D.xcount + TX - 1) / TX;
  ntiles = ntx * ((D.d.NJ + TY - 1) / TY);
}

// Every domain's tiles in one order, dealt to the XCDs in contiguous runs.
template <int T>
__global__ __launch_bounds__(64 * bt_nw(T), 4) void k_bt_block_ens(const BtDom *__restrict__ doms,
                                                                   BtLaunch L, int per_xcd) {
  const int b = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (b >= L.first[L.ndom]) return;
  int lo = 0, hi = L.ndom - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (L.first[mid] <= b) lo = mid; else hi = mid - 1;
  }
  const BtDom &D = doms[lo];
  BtJob J;
  J.d = D.d;
  J.in = D.in;
  int nsub, ntx, ntiles;
  bt_shape(D, L, nsub, ntx, ntiles);
  const bool first = L.ell == 0;
  J.eta_src = first ? D.eta_bar_tau : D.eta_buf[(L.ell - 1) & 1];
  J.ud_src = first ? D.ud_tau : D.ud_buf[(L.ell - 1) & 1];
  J.eb_src = first ? D.eb0 : D.eb;
  J.ub_src = first ? nullptr : D.ub;
  J.eta_dst = D.eta_buf[L.ell & 1];
  J.ud_dst = D.ud_buf[L.ell & 1];
  J.eb = D.eb;
  J.ub = D.ub;
  J.s0 = L.ell * L.hsub + 1;
  J.nsub = nsub;
  J.nts = D.nts;
  J.step_a = D.step_a;
  J.dtbt = D.dtbt;
  J.cp = D.cp;
  J.cc = D.cc;
  J.xbase = D.xbase;
  J.xcount = D.xcount;
  J.ntx = ntx;
  J.ntiles = ntiles;
  J.rev = 0;
  J.land = nullptr;
  bt_any_tile<T>(J, strip_tile<8>(b - L.first[lo], ntx, ntiles / ntx));
}

// Tail of update_ocean_barotropic (:2804-2811, :2846-2888) from the time sums of
// the blocked subcycles (scratch planes, so that a point may read its neighbours'
// and its cyclic source's): the means, halo columns of the compute rows at
// their cyclic source, and conv_rho_ud_t = -DIV_UD of them, in one pass.  The
// halo columns of the first and last row, which no subcycle touches on a
// cyclic-x domain, hold the initial sums.
struct BtTail {
  KDom d;
  const double *eb0, *eb, *ub;
  double *eta_bar, *ud, *conv;
  double rntsp1, rnts;
  const double *dxu, *dyu, *datr;
};
__device__ __forceinline__ void bt_tail(const BtTail &T, int ii, int jj) {
  const KDom &d = T.d;
  const bool crow = jj >= 1 && jj <= d.NJ - 2;
  // the point whose sums a point takes; -1: none (a halo column the subcycles leave)
  auto source = [&](int i, int j) {
    if (!d.cyclic_x || (i >= 1 && i <= d.ni)) return i + d.NI * j;
    if (j < 1 || j > d.NJ - 2) return -1;
    return (i == 0 ? d.ni : 1) + d.NI * j;
  };
  const int o = ii + d.NI * jj, os = source(ii, jj);
  T.eta_bar[o] = T.rntsp1 * (os >= 0 ? T.eb[os] : T.eb0[o]);
  auto mean = [&](int c, int i, int j) {
    const int q = source(i, j);
    return T.rnts * (q >= 0 ? T.ub[(size_t)d.P2 * c + q] : 0.0);
  };
  const double u = mean(0, ii, jj), v = mean(1, ii, jj);
  T.ud[o] = u;
  T.ud[d.P2 + o] = v;
  if (!T.conv) return;
  // conv at the point, or at its cyclic source
  int si = ii;
  if (d.cyclic_x && crow) si = ii == 0 ? d.ni : (ii == d.NI - 1 ? 1 : ii);
  double dv = 0.0;
  if (si != 0 && jj != 0) {
    const int so = si + d.NI * jj, sm = so - d.NI;
    const double uh = mean(0, si, jj) * T.dyu[so], vh = mean(1, si, jj) * T.dxu[so];
    const double uhjm = mean(0, si, jj - 1) * T.dyu[sm], vhjm = mean(1, si, jj - 1) * T.dxu[sm];
    const double uhim = mean(0, si - 1, jj) * T.dyu[so - 1];
    const double vhim = mean(1, si - 1, jj) * T.dxu[so - 1];
    const double uhimjm = mean(0, si - 1, jj - 1) * T.dyu[sm - 1];
    const double vhimjm = mean(1, si - 1, jj - 1) * T.dxu[sm - 1];
    const double uh_bay = 0.5 * (uh + uhjm);
    const double vh_bax = 0.5 * (vh + vhim);
    const double uhim_bay = 0.5 * (uhim + uhimjm);
    const double vhjm_bax = 0.5 * (vhjm + vhimjm);
    dv = ((uh_bay - uhim_bay) + (vh_bax - vhjm_bax)) * T.datr[so];
  }
  T.conv[o] = -dv;
}
__global__ void k_bt_tail(BtTail T) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x;
  if (ii < T.d.NI) bt_tail(T, ii, blockIdx.y);
}
__global__ void k_bt_tail_ens(const BtTail *__restrict__ Ts) {
  const BtTail &T = Ts[blockIdx.z];
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii < T.d.NI && jj < T.d.NJ) bt_tail(T, ii, jj);
}

// ocean_barotropic_forcing (ocean_barotropic.F90:3058-3141, default namelist,
// B-grid: tmasken = umask): the column sum of accel over the wet U-levels
// plus the surface/bottom stress, on the compute domain; a halo column or
// row takes the value of its cyclic source (what the halo update leaves), a
// closed halo is zero; then the zero friction terms are added, as there.
__global__ void k_bt_forcing(KDom d, const double *__restrict__ accel,
                             const double *__restrict__ smf, const double *__restrict__ bmf,
                             const int *__restrict__ kmu, double *__restrict__ out) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  int si = ii, sj = jj;
  bool valid = true;
  if (jj < 1 || jj > d.nj) {
    if (d.cyclic_y) sj = 1 + wrapi(jj - 1, d.nj); else valid = false;
  }
  if (ii < 1 || ii > d.ni) {
    if (d.cyclic_x) si = 1 + wrapi(ii - 1, d.ni); else valid = false;
  }
  const size_t P2 = (size_t)d.P2, P3 = P2 * (size_t)d.nk;
  const int o = ii + d.NI * jj, os = si + d.NI * sj;
  const int km = valid ? kmu[os] : 0;
  for (int n = 0; n < 2; ++n) {
    double f = 0.0;
    if (valid) {
      double wrk = 0.0;
      for (int k = 1; k <= d.nk; ++k)
        wrk = wrk + (k <= km ? 1.0 : 0.0) * accel[P3 * n + P2 * (size_t)(k - 1) + os];
      f = wrk + (1 <= km ? 1.0 : 0.0) * (smf[P2 * n + os] - bmf[P2 * n + os]);
    }
    out[P2 * n + o] = f + 0.0 + 0.0;
  }
}

struct EtaIn {
  const double *conv, *pme, *river, *source, *dpatm_dt, *ht, *x_taum1;
  const int *kmt;
  double rho0r, grav, rho0grav, dtime;
  int pressure_based;
};

// eta_and_pbot_tendency (ocean_barotropic.F90:2686-2710) at one point.
__device__ inline double eta_tendency(const EtaIn &e, int o) {
  const double tm = 1 <= e.kmt[o] ? 1.0 : 0.0;
  const double sum = e.conv[o] + e.pme[o] + e.river[o] + e.source[o];
  if (!e.pressure_based) return tm * e.rho0r * sum;
  return e.dpatm_dt[o] + e.grav * tm * sum;
}

// eta_and_pbot_tendency then eta_and_pbot_update (:2303-2363): the tendency
// on the data domain; x_taup1 = x_taum1 + dtime*tendency on the compute
// domain and, on halo points the update rewrites, at their cyclic source;
// pressure-based: pbot_t = anompb + rho0grav*ht on the data domain.
__global__ void k_eta_update(KDom d, EtaIn e, double *__restrict__ x_taup1,
                             double *__restrict__ pbot, double *__restrict__ tend) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const int o = ii + d.NI * jj;
  tend[o] = eta_tendency(e, o);
  int si, sj;
  double x;
  if (halo_source(d, ii, jj, si, sj)) {
    const int os = si + d.NI * sj;
    x = e.x_taum1[os] + e.dtime * eta_tendency(e, os);
    x_taup1[o] = x;
  } else {
    x = x_taup1[o];
  }
  if (e.pressure_based) pbot[o] = x + e.rho0grav * e.ht[o];
}

struct ClosureIn {
  const double *eta_bar, *anompb_bar, *patm, *rho_g, *ht;
  const double *dte, *dtw, *dus, *dun, *daur, *dxur, *dyur;
  const double *tmasken, *dxte, *dytn;   // tmasken != NULL: C-grid gradient
  const int *kmu;
  double rho0grav;
  int pressure_based;
};

// The field REMAP_BT_TO_BU is applied to: eta_t_bar, or rho0grav*ht +
// anompb_bar for the pressure-based closure (:2908, :2918).
__device__ inline double remap_src(const ClosureIn &c, int o) {
  return c.pressure_based ? c.rho0grav * c.ht[o] + c.anompb_bar[o] : c.eta_bar[o];
}

// umask(k=1)*REMAP_BT_TO_BU at U point (i, j) (ocean_operators.F90:468-475).
__device__ inline double remap_bu(const KDom &d, const ClosureIn &c, int i, int j) {
  if (i >= d.NI - 1 || j >= d.NJ - 1) return 0.0;
  const int o = i + d.NI * j, oe = o + 1, on = o + d.NI, one = on + 1;
  const double r = (remap_src(c, o) * c.dte[o] * c.dus[o] + remap_src(c, oe) * c.dtw[oe] * c.dus[o]
                    + remap_src(c, on) * c.dte[on] * c.dun[o]
                    + remap_src(c, one) * c.dtw[one] * c.dun[o]) * c.daur[o];
  return (1 <= c.kmu[o] ? 1.0 : 0.0) * r;
}

// ps = rho_g*eta_t_bar + patm (:2970).
__device__ inline double surf_p(const ClosureIn &c, int o) {
  return c.rho_g[o] * c.eta_bar[o] + c.patm[o];
}

// GRAD_BAROTROPIC_P, halo 1, of a pressure given by a point function:
// B-grid (ocean_operators.F90:651-660) or C-grid (:664-669).
template <class P>
__device__ inline void grad_bt(const KDom &d, const ClosureIn &c, int i, int j, P p, double &gx,
                              double &gy) {
  if (i >= d.NI - 1 || j >= d.NJ - 1) {
    gx = 0.0;
    gy = 0.0;
    return;
  }
  const int o = i + d.NI * j, oe = o + 1, on = o + d.NI, one = on + 1;
  if (c.tmasken) {
    const double pc = p(o);
    gx = (p(oe) - pc) * (1.0 / (c.dxte[o] + 1.0e-40)) * c.tmasken[o];
    gy = (p(on) - pc) * (1.0 / (c.dytn[o] + 1.0e-40)) * c.tmasken[(size_t)d.P2 + o];
    return;
  }
  const double pc = p(o), pe = p(oe), pn = p(on), pne = p(one);
  const double p_fay = 0.5 * (pc + pn);
  const double p_fax = 0.5 * (pc + pe);
  const double pip_fay = 0.5 * (pe + pne);
  const double pjp_fax = 0.5 * (pn + pne);
  const double um = 1 <= c.kmu[o] ? 1.0 : 0.0;
  gx = (pip_fay - p_fay) * c.dxur[o] * um;
  gy = (pjp_fax - p_fax) * c.dyur[o] * um;
}

// Closure of update_ocean_barotropic (ocean_barotropic.F90:2906-2921,
// 2956-2985): eta_u (or pbot_u) halo-updated, ps, grad_ps and grad_anompb.
// Neighbour values of ps are recomputed, not read, so one launch suffices.
__global__ void k_bt_closure(KDom d, ClosureIn c, double *__restrict__ eta_u,
                             double *__restrict__ ps, double *__restrict__ grad_ps,
                             double *__restrict__ grad_ab) {
  const int ii = blockIdx.x * blockDim.x + threadIdx.x, jj = blockIdx.y;
  if (ii >= d.NI) return;
  const int o = ii + d.NI * jj;
  int si, sj;
  halo_source(d, ii, jj, si, sj);
  eta_u[o] = remap_bu(d, c, si, sj);
  ps[o] = surf_p(c, o);
  const size_t P2 = (size_t)d.P2;
  double gx, gy;
  grad_bt(d, c, ii, jj, [&](int q) { return surf_p(c, q); }, gx, gy);
  grad_ps[o] = gx;
  grad_ps[P2 + o] = gy;
  if (grad_ab) {
    grad_bt(d, c, ii, jj, [&](int q) { return c.anompb_bar[q]; }, gx, gy);
    grad_ab[o] = gx;
    grad_ab[P2 + o] = gy;
  }
}

}  // namespace

// Sets ctx->bt_recip: whether the context's dxur and dyur are the reciprocals
// the blocked barotropic may form itself (then it loads two planes fewer), and
// the other checks of the grid.
int launch_check_recip(mom_gpu_ctx *ctx) {
  const KDom &d = ctx->kd;
  const size_t n = (size_t)d.P2;
  ctx->bt_recip = 0;
  int *dev = nullptr;
  MOM_HIP(ctx, hipMalloc(&dev, n * sizeof(int)));
  hipLaunchKernelGGL(k_check_recip, dim3((d.NI + 127) / 128, d.NJ), dim3(128), 0, ctx->stream, d,
                     ctx->dxu, ctx->dxur, ctx->dyu, ctx->dyur, ctx->datr, ctx->f, ctx->dat, ctx->dxte,
                     ctx->dytn, dev);
  hipError_t le = hipGetLastError();
  int *host = (int *)malloc(n * sizeof(int));
  hipError_t e1 = host ? hipMemcpyAsync(host, dev, n * sizeof(int), hipMemcpyDeviceToHost,
                                        ctx->stream)
                       : hipErrorOutOfMemory;
  hipError_t e2 = hipStreamSynchronize(ctx->stream);
  (void)hipFree(dev);
  if (le != hipSuccess || e1 != hipSuccess || e2 != hipSuccess) {
    free(host);
    return mom_fail(ctx, MOM_GPU_ERR_HIP, "reciprocal check failed: %s",
                    hipGetErrorString(le != hipSuccess ? le : (e1 != hipSuccess ? e1 : e2)));
  }
  int bad = 0;
  for (size_t q = 0; q < n; ++q) bad |= host[q];
  free(host);
  ctx->bt_recip = (bad & 1) == 0;
  ctx->bt_grid_ok = (bad & 2) == 0;
  // (the rows' constants lie behind the masks in one plane: 64 B a row)
  ctx->bt_rows_ok = (bad & 4) == 0 && d.NI >= 16;
  ctx->btv_rows_ok = (bad & 8) == 0 && d.NI >= 16;
  return MOM_GPU_OK;
}

namespace {
// The planes of ctx->bt as the blocked subcycles use them: 0-5 the state, two
// sets; 6 sf; 7 the masks (a byte a point) and behind them the row constants; 8
// the tiles' land flags (at most one int a point: a tile's interior holds at
// least one); 9-11 the time sums.
struct BtBufs {
  double *eta[2], *ud[2], *sf, *rowc, *eb, *ub;
  unsigned char *mask;
  int *land;
  explicit BtBufs(mom_gpu_ctx *ctx) {
    const size_t P2 = (size_t)ctx->kd.P2;
    double *b = ctx->bt;
    eta[0] = b; eta[1] = b + P2;
    ud[0] = b + 2 * P2; ud[1] = b + 4 * P2;
    sf = b + 6 * P2;
    mask = (unsigned char *)(b + 7 * P2);
    rowc = b + 7 * P2 + (P2 + 7) / 8;
    land = (int *)(b + 8 * P2);
    eb = b + 9 * P2;
    ub = b + 10 * P2;
  }
};

// Tile and subcycles a launch for domains d[0..n) launched together.  Results do
// not depend on either.  rows: every domain's rows are uniform; h: subcycles asked
// for, 0 to choose.
// - While the tiles leave CUs idle a launch's time is its latency, so the deepest
//   launches win: 90 x 60, 80 subcycles, 5 / 10 a launch: 165 / 120 us alone (one
//   call, waited for), 63 / 50 among three states in turn (calls queued on the
//   streams of three contexts, so that one fills what another leaves idle); 360 x
//   240, 5 / 7: 178 / 159, 83 / 81; above one tile a CU, 517 x 389, 5 / 7: 254 / 228
//   but 126 / 144 (a deeper launch does more work a point).  The general tile,
//   one block a CU: 90 x 60, 5 / 12: 256 / 186 and 95 / 69, 360 x 240, 5 / 8:
//   268 / 214 and 122 / 120, past 128 tiles 517 x 389, 5 / 7: 286 / 255, 241 / 240.
// - Three rows a wavefront have the shorter chain (90 x 60, 10 a launch: 120 us
//   against 186), four the fewer redundant points: they win once the 18 planes are
//   larger than the 256 MB cache and every launch is paid in memory traffic (1440
//   x 1080: 933 us with three, 1010 with four; 3600 x 2700: 8404 and 7975), and
//   at depths that leave the lower region no interior.
struct BtPlan {
  int tile, hsub;
};
int bt_tiles(const KDom *const *d, int n, int tile, int h) {
  const int TX = bt_interior(BRX, h), TY = bt_interior(bt_ry(tile), h);
  int t = 0;
  for (int k = 0; k < n; ++k)
    t += (((d[k]->cyclic_x ? d[k]->ni : d[k]->NI) + TX - 1) / TX) * ((d[k]->NJ + TY - 1) / TY);
  return t;
}
BtPlan bt_plan(const KDom *const *d, int n, bool rows, int h) {
  if (!rows) {
    if (h == 0)
      for (h = 12; h > 5 && bt_tiles(d, n, BT_ANY, h) > 128; --h) {}
    return {BT_ANY, h};
  }
  size_t bytes = 0;
  for (int k = 0; k < n; ++k) bytes += (size_t)d[k]->P2 * 18 * sizeof(double);
  const bool large = bytes > (size_t)256 << 20;
  if (h == 0) {
    h = 6;
    if (!large)
      for (h = 10; h > 5 && bt_tiles(d, n, BT_ROWS3, h) > 256; --h) {}
  }
  if (large || h > 10 || (h > 7 && bt_tiles(d, n, BT_ROWS3, h) > 256)) return {BT_ROWS4, h};
  return {BT_ROWS3, h};
}

template <typename F>
void bt_with_tile(int tile, F &&f) {
  if (tile == BT_ANY) f(std::integral_constant<int, BT_ANY>{});
  else if (tile == BT_ROWS3) f(std::integral_constant<int, BT_ROWS3>{});
  else f(std::integral_constant<int, BT_ROWS4>{});
}
}  // namespace

int launch_barotropic_blocked(mom_gpu_ctx *ctx, const mom_gpu_bt_params_t *p,
                              const double *eta_t, const double *eta_bar_tau,
                              const double *ud_tau, const double *forcing, const double *thicku,
                              const double *patm, const double *pme, const double *river,
                              const double *source, const double *eta_smooth,
                              const double *rho_g, double *eta_bar, double *ud, double *conv,
                              int hsub) {
  const KDom &d = ctx->kd;
  const size_t P2 = (size_t)d.P2;
  hipStream_t s = ctx->stream;
  const double rho0r = 1.0 / p->rho0;
  const double c_pred = p->dtbt * p->pred_corr_gamma * rho0r;   // dtbt_gamma_rho0r, :1196
  const double c_corr = p->dtbt * rho0r;                        // dtbt_rho0r, :1197
  const dim3 grid((d.NI + 255) / 256, d.NJ), block(256);
  const BtBufs w(ctx);
  const KDom *const one = &d;
  const BtPlan plan = bt_plan(&one, 1, ctx->bt_rows_ok, hsub);
  hsub = plan.hsub;
  ctx->bt_subcycles_used = hsub;
  // the land path's conditions that do not depend on the data; with at most one
  // tile a CU its tiles would only wait for the others, and forming the flags costs
  // a launch (90x60: 5 us of a step's 154)
  const bool land_ok = bt_tiles(&one, 1, plan.tile, hsub) > 256 && ctx->tune.bt_land_tiles &&
                       ctx->bt_grid_ok && p->dtbt > 0.0 &&
                       std::isfinite(c_pred) && std::isfinite(c_corr);
  const Inert inert = land_ok ? Inert{eta_bar_tau, ud_tau, forcing, rho_g, patm, thicku} : Inert{};
  const double *rowc = ctx->bt_rows_ok ? w.rowc : nullptr;
  hipLaunchKernelGGL(k_bt_prep, grid, block, 0, s,
                     BtPrep{d, pme, river, source, eta_smooth, ctx->kmt, ctx->kmu, w.sf, w.mask,
                            inert, ctx->datr, ctx->dyu, ctx->dxu, ctx->dxur, ctx->dyur, ctx->f,
                            p->dtbt, (double *)rowc});
  MOM_LAUNCHED(ctx, "k_bt_prep");
  const BtIn in{rho_g, patm, thicku, forcing, ctx->f, ctx->dxu, ctx->dyu, ctx->datr, ctx->dxur,
                ctx->dyur, w.sf, w.mask, rowc, ctx->bt_recip};
  int *landp = land_ok ? w.land : nullptr;
  int land_nsub = 0;
  const int xbase = d.cyclic_x ? 1 : 0, xcount = d.cyclic_x ? d.ni : d.NI;
  const int ry = bt_ry(plan.tile);
  const double *eb0 = p->initsum_with_bar ? eta_bar_tau : eta_t;
  const double *eta_src = eta_bar_tau, *ud_src = ud_tau;
  int which = 0;
  for (int s0 = 1; s0 <= p->nts; s0 += hsub) {
    const int nsub = std::min(hsub, p->nts - s0 + 1);
    const int TX = bt_interior(BRX, nsub), TY = bt_interior(ry, nsub);
    const int ntx = (xcount + TX - 1) / TX, nty = (d.NJ + TY - 1) / TY;
    if (landp && nsub != land_nsub) {
      // stream order: the launches that read the previous flags are done
      hipLaunchKernelGGL(k_bt_land, dim3(ntx * nty), dim3(256), 0, s, d, w.mask, ry, nsub, xbase,
                         ntx, ntx * nty, landp);
      MOM_LAUNCHED(ctx, "k_bt_land");
      land_nsub = nsub;
    }
    const BtJob J{d, in, eta_src, ud_src, s0 == 1 ? eb0 : w.eb, s0 == 1 ? nullptr : w.ub,
                  w.eta[which], w.ud[which], w.eb, w.ub, s0, nsub, p->nts, p->stepping_a,
                  p->dtbt, c_pred, c_corr, xbase, xcount, ntx, ntx * nty,
                  plan.tile == BT_ANY ? 0 : which, landp};
    const int per_xcd = (ntx * nty + 7) / 8;
    bt_with_tile(plan.tile, [&](auto t) {
      hipLaunchKernelGGL(k_bt_block<t.value>, dim3(8 * per_xcd), dim3(64 * bt_nw(t.value)), 0, s, J,
                         per_xcd);
    });
    MOM_LAUNCHED(ctx, "k_bt_block");
    eta_src = w.eta[which];
    ud_src = w.ud[which];
    which ^= 1;
  }
  const double nts = (double)p->nts;
  const double rntsp1 = 1.0 / (nts + 1.0);
  const double rnts = p->stepping_a ? 1.0 / nts : 2.0 / (nts * (double)(p->nts + 1));
  hipLaunchKernelGGL(k_bt_tail, grid, block, 0, s,
                     BtTail{d, eb0, w.eb, w.ub, eta_bar, ud, conv, rntsp1, rnts, ctx->dxu, ctx->dyu,
                            ctx->datr});
  MOM_LAUNCHED(ctx, "k_bt_tail");
  return MOM_GPU_OK;
}

int launch_barotropic(mom_gpu_ctx *ctx, const mom_gpu_bt_params_t *p, const double *eta_t,
                      const double *eta_bar_tau, const double *ud_tau, const double *forcing,
                      const double *thicku, const double *patm, const double *pme,
                      const double *river, const double *source, const double *eta_smooth,
                      const double *rho_g, double *eta_bar, double *ud, double *conv) {
  const int knob = ctx->tune.bt_subcycles_per_launch;
  if (knob != 0)
    return launch_barotropic_blocked(ctx, p, eta_t, eta_bar_tau, ud_tau, forcing, thicku, patm,
                                     pme, river, source, eta_smooth, rho_g, eta_bar, ud, conv,
                                     std::max(knob, 0));
  ctx->bt_subcycles_used = 0;
  const KDom &d = ctx->kd;
  const size_t P2 = (size_t)d.P2;
  BtBuf b;
  b.eta = ctx->bt;
  b.ud = ctx->bt + 2 * P2;
  b.sf = ctx->bt + 6 * P2;
  b.cori1 = ctx->bt + 7 * P2;
  b.cori2 = ctx->bt + 8 * P2;
  const double rho0r = 1.0 / p->rho0;
  const double c_pred = p->dtbt * p->pred_corr_gamma * rho0r;   // dtbt_gamma_rho0r, :1196
  const double c_corr = p->dtbt * rho0r;                        // dtbt_rho0r, :1197
  const dim3 grid((d.NI + 255) / 256, d.NJ), block(256);
  hipStream_t s = ctx->stream;
  hipLaunchKernelGGL(k_bt_init, grid, block, 0, s, d, b, p->initsum_with_bar, p->dtbt, eta_t,
                     eta_bar_tau, ud_tau, pme, river, source, eta_smooth, ctx->f, ctx->kmt,
                     eta_bar, ud);
  MOM_LAUNCHED(ctx, "k_bt_init");
  for (int itime = 1; itime <= p->nts; ++itime) {
    const int fstau = (itime + 0) % 2 + 1;
    const int fstaup1 = (itime + 1) % 2 + 1;
    hipLaunchKernelGGL(k_bt_pred, grid, block, 0, s, d, b, fstau, fstaup1, c_pred, ctx->dxu,
                       ctx->dyu, ctx->datr, ctx->kmt);
    hipLaunchKernelGGL(k_bt_mom, grid, block, 0, s, d, b, fstau, fstaup1, p->dtbt, rho_g, patm,
                       thicku, forcing, ctx->f, ctx->dxur, ctx->dyur, ctx->kmu);
    const double wgt = (double)(p->nts - itime + 1);
    hipLaunchKernelGGL(k_bt_corr, grid, block, 0, s, d, b, fstau, fstaup1, c_corr,
                       p->stepping_a, wgt, ctx->dxu, ctx->dyu, ctx->datr, ctx->kmt, eta_bar, ud);
  }
  MOM_LAUNCHED(ctx, "k_bt_subcycle");
  const double nts = (double)p->nts;
  const double rntsp1 = 1.0 / (nts + 1.0);
  const double rnts = p->stepping_a ? 1.0 / nts : 2.0 / (nts * (double)(p->nts + 1));
  hipLaunchKernelGGL(k_bt_scale, grid, block, 0, s, d, rntsp1, rnts, eta_bar, ud);
  const dim3 wg((d.NJ + 255) / 256), wb(256);
  if (d.cyclic_x) {
    hipLaunchKernelGGL(k_bt_wrap, wg, wb, 0, s, d, eta_bar, 1);
    hipLaunchKernelGGL(k_bt_wrap, wg, wb, 0, s, d, ud, 2);
  }
  if (conv) {
    hipLaunchKernelGGL(k_bt_conv, grid, block, 0, s, d, ud, ctx->dxu, ctx->dyu, ctx->datr, conv);
    if (d.cyclic_x) hipLaunchKernelGGL(k_bt_wrap, wg, wb, 0, s, d, conv, 1);
  }
  MOM_LAUNCHED(ctx, "k_bt_tail");
  return MOM_GPU_OK;
}

// Barotropic subcycles of every domain of an ensemble: launch ell advances
// hsub subcycles of each domain that has any left (its own nts, dtbt).
int launch_barotropic_ensemble(mom_gpu_ensemble *e, const mom_gpu_bt_params_t *p,
                               const mom_gpu_bt_fields_t *f) {
  const int nd = (int)e->ctx.size();
  if (nd > BT_MAXDOM) return mom_fail(e->lead, MOM_GPU_ERR_ARG, "ensemble: too many domains");
  const int knob = e->lead->tune.bt_subcycles_per_launch;
  int hsub = knob < 0 ? 0 : knob > 0 ? knob : 4;
  std::vector<BtDom> doms(nd);
  std::vector<BtTail> tails(nd);
  std::vector<BtPrep> preps(nd);
  std::memset((void *)doms.data(), 0, sizeof(BtDom) * nd);
  std::memset((void *)tails.data(), 0, sizeof(BtTail) * nd);
  std::memset((void *)preps.data(), 0, sizeof(BtPrep) * nd);
  int maxNI = 1, maxNJ = 1, nlaunch = 0;
  bool rows = true;                 // every domain's rows are uniform
  std::vector<const KDom *> kds(nd);
  for (int k = 0; k < nd; ++k) {
    rows = rows && e->ctx[k]->bt_rows_ok;
    kds[k] = &e->ctx[k]->kd;
  }
  const BtPlan plan = bt_plan(kds.data(), nd, rows, hsub);
  hsub = plan.hsub;
  for (mom_gpu_ctx *c : e->ctx) c->bt_subcycles_used = hsub;
  for (int k = 0; k < nd; ++k) {
    mom_gpu_ctx *ctx = e->ctx[k];
    const KDom &d = ctx->kd;
    const mom_gpu_bt_fields_t &x = f[k];
    const double rho0r = 1.0 / p[k].rho0;
    const BtBufs w(ctx);
    const double *eb0 = p[k].initsum_with_bar ? x.eta_t_bar_tau : x.eta_t_tau;
    BtPrep &P = preps[k];
    P.d = d;
    P.pme = x.pme; P.river = x.river; P.source = x.source; P.eta_smooth = x.eta_smooth;
    P.kmt = ctx->kmt; P.kmu = ctx->kmu; P.sf = w.sf; P.mask = w.mask;
    P.datr = ctx->datr; P.dyu = ctx->dyu; P.dxu = ctx->dxu; P.dxur = ctx->dxur;
    P.dyur = ctx->dyur; P.f = ctx->f; P.dtbt = p[k].dtbt;
    P.rowc = rows ? w.rowc : nullptr;
    BtDom &D = doms[k];
    D.d = d;
    D.in = BtIn{x.rho_g, x.patm, x.thicku, x.forcing_bt, ctx->f, ctx->dxu, ctx->dyu, ctx->datr,
                ctx->dxur, ctx->dyur, w.sf, w.mask, P.rowc, ctx->bt_recip};
    D.eta_bar_tau = x.eta_t_bar_tau;
    D.ud_tau = x.udrho_tau;
    D.eb0 = eb0;
    D.eta_buf[0] = w.eta[0];
    D.eta_buf[1] = w.eta[1];
    D.ud_buf[0] = w.ud[0];
    D.ud_buf[1] = w.ud[1];
    D.eb = w.eb;
    D.ub = w.ub;
    D.nts = p[k].nts;
    D.step_a = p[k].stepping_a;
    D.dtbt = p[k].dtbt;
    D.cp = p[k].dtbt * p[k].pred_corr_gamma * rho0r;   // dtbt_gamma_rho0r, :1196
    D.cc = p[k].dtbt * rho0r;                          // dtbt_rho0r, :1197
    D.xbase = d.cyclic_x ? 1 : 0;
    D.xcount = d.cyclic_x ? d.ni : d.NI;
    BtTail &T = tails[k];
    T.d = d;
    T.eb0 = eb0;
    T.eb = w.eb;
    T.ub = w.ub;
    T.eta_bar = x.eta_t_bar_taup1;
    T.ud = x.udrho_taup1;
    T.conv = x.conv_rho_ud_t;
    const double nts = (double)p[k].nts;
    T.rntsp1 = 1.0 / (nts + 1.0);
    T.rnts = p[k].stepping_a ? 1.0 / nts : 2.0 / (nts * (double)(p[k].nts + 1));
    T.dxu = ctx->dxu;
    T.dyu = ctx->dyu;
    T.datr = ctx->datr;
    maxNI = std::max(maxNI, d.NI);
    maxNJ = std::max(maxNJ, d.NJ);
    nlaunch = std::max(nlaunch, (p[k].nts + hsub - 1) / hsub);
  }
  // one table: the domains, their preparations, their tails (each 16 B aligned)
  const size_t a16 = 16, sd = (sizeof(BtDom) * nd + a16 - 1) / a16 * a16,
               sp = (sizeof(BtPrep) * nd + a16 - 1) / a16 * a16;
  std::vector<unsigned char> buf(sd + sp + sizeof(BtTail) * nd, 0);
  std::memcpy(buf.data(), doms.data(), sizeof(BtDom) * nd);
  std::memcpy(buf.data() + sd, preps.data(), sizeof(BtPrep) * nd);
  std::memcpy(buf.data() + sd + sp, tails.data(), sizeof(BtTail) * nd);
  const unsigned char *dev = (const unsigned char *)ens_table(e, buf.data(), buf.size());
  if (!dev) return MOM_GPU_ERR_HIP;
  const BtDom *ddev = (const BtDom *)dev;
  const BtPrep *pdev = (const BtPrep *)(dev + sd);
  const BtTail *tdev = (const BtTail *)(dev + sd + sp);
  hipStream_t s = e->lead->stream;
  const dim3 g2((maxNI + 255) / 256, maxNJ, nd), b2(256);
  hipLaunchKernelGGL(k_bt_prep_ens, g2, b2, 0, s, pdev);
  MOM_LAUNCHED(e->lead, "k_bt_prep_ens");
  for (int ell = 0; ell < nlaunch; ++ell) {
    BtLaunch L{};
    L.ndom = nd;
    L.ell = ell;
    L.hsub = hsub;
    L.ry = bt_ry(plan.tile);
    int total = 0;
    for (int k = 0; k < nd; ++k) {
      int nsub, ntx, ntiles;
      bt_shape(doms[k], L, nsub, ntx, ntiles);
      L.first[k] = total;
      total += ntiles;
    }
    L.first[nd] = total;
    if (total == 0) continue;
    const int per_xcd = (total + 7) / 8;
    bt_with_tile(plan.tile, [&](auto t) {
      hipLaunchKernelGGL(k_bt_block_ens<t.value>, dim3(8 * per_xcd), dim3(64 * bt_nw(t.value)), 0,
                         s, ddev, L, per_xcd);
    });
    MOM_LAUNCHED(e->lead, "k_bt_block_ens");
  }
  hipLaunchKernelGGL(k_bt_tail_ens, g2, b2, 0, s, tdev);
  MOM_LAUNCHED(e->lead, "k_bt_tail_ens");
  return MOM_GPU_OK;
}

int launch_bt_forcing(mom_gpu_ctx *ctx, const double *accel, const double *smf, const double *bmf,
                      double *forcing_bt) {
  const KDom &d = ctx->kd;
  hipLaunchKernelGGL(k_bt_forcing, dim3((d.NI + 63) / 64, d.NJ), dim3(64), 0, ctx->stream, d,
                     accel, smf, bmf, ctx->kmu, forcing_bt);
  MOM_LAUNCHED(ctx, "k_bt_forcing");
  return MOM_GPU_OK;
}

int launch_eta_update(mom_gpu_ctx *ctx, int pressure_based, double rho0, double grav,
                      double dtime, const double *conv, const double *pme, const double *river,
                      const double *source, const double *dpatm_dt, const double *ht,
                      const double *x_taum1, double *x_taup1, double *pbot, double *tend) {
  const KDom &d = ctx->kd;
  EtaIn e{conv, pme, river, source, dpatm_dt, ht, x_taum1, ctx->kmt,
          1.0 / rho0, grav, rho0 * grav, dtime, pressure_based};
  hipLaunchKernelGGL(k_eta_update, dim3((d.NI + 63) / 64, d.NJ), dim3(64), 0, ctx->stream, d, e,
                     x_taup1, pbot, tend);
  MOM_LAUNCHED(ctx, "k_eta_update");
  return MOM_GPU_OK;
}

int launch_bt_closure(mom_gpu_ctx *ctx, int pressure_based, double rho0, double grav,
                      const double *eta_bar, const double *anompb_bar, const double *patm,
                      const double *rho_g, const double *ht, const double *tmasken,
                      double *eta_u, double *ps, double *grad_ps, double *grad_ab) {
  const KDom &d = ctx->kd;
  const double *rm = ctx->remap;
  const size_t P2 = (size_t)d.P2;
  ClosureIn c{eta_bar, anompb_bar, patm, rho_g, ht, rm, rm + P2, rm + 2 * P2, rm + 3 * P2,
              rm + 4 * P2, ctx->dxur, ctx->dyur, tmasken, ctx->dxte, ctx->dytn, ctx->kmu,
              rho0 * grav, pressure_based};
  hipLaunchKernelGGL(k_bt_closure, dim3((d.NI + 63) / 64, d.NJ), dim3(64), 0, ctx->stream, d, c,
                     eta_u, ps, grad_ps, grad_ab);
  MOM_LAUNCHED(ctx, "k_bt_closure");
  return MOM_GPU_OK;
}
