// Batched step for Quicker tracers: horz_advect_tracer_quicker
// (ocean_tracer_advect.F90:2538-2653) and vert_advect_tracer_quicker
// (:2981-3031) into th_tendency, with the tracer's tmask_limit
// (ocean_tracer.F90:2788-2892) formed in the kernel from T(tau), then the
// explicit update (ocean_tracer.F90:2341-2350), in one k-marching pass.
//
// Two-level time stepping: T(taum1) = T(tau), one input array.  Every
// value outside the compute domain is read with MOM's halo semantics after
// the halo updates the reference makes (cyclic wrap, zero beyond a closed
// axis), as the batched MDFL pass does.  The arithmetic of every face flux,
// divergence, limit flag and update is the reference's, operation for
// operation, so T(taup1) equals bit for bit the per-tracer sequence
// (compute_tmask_limit, horz_advect_tracer and vert_advect_tracer into a
// zeroed th_tendency, the explicit update) on halo-updated inputs.
//
// Work-group layout as the MDFL pass: 64-wide region rows, one row per
// wavefront, a 2-cell halo (the Quicker stencil reaches i-1..i+2 for the
// face east of i), x neighbours through DPP lane shifts, y neighbours
// through LDS.  The 16 Quicker weights of a column are two-dimensional and
// stay in registers for all levels.
//
// A pass takes two tracers (temperature and salinity first), which share the
// transports, thicknesses and weights; their tmask_limit flags are OR'ed in
// registers.  The pass is latency bound if a level's loads are issued where
// they are used: with them, and two barriers a level, one tracer took 2.2 ms at
// 1440x1080x50 (64 B a cell: 0.9 ms at 5.5 TB/s).  So a level's 3-D inputs are
// issued during the level before, T(k+3) too, and T and the y fluxes have two
// LDS copies by level parity: one barrier a level.  T and S now take 2.0 ms
// together (72 B a cell: 1.0 ms), one tracer 1.4 ms; what is left is the
// reference's arithmetic (360 vector instructions a level and wavefront for
// two tracers) on regions with 12 x 64 of 8 x 60 cells.
#include "mom_internal.h"

#include <vector>

namespace {

constexpr int RX = 64;
constexpr int TX = RX - 4;

__device__ inline double mk(int k, int kmt) { return (k <= kmt) ? 1.0 : 0.0; }
__device__ inline bool outside(double x, double lo, double hi) { return x < lo || x > hi; }

struct QStepJob {
  KDom d;
  const double *T[2];   // T(taum1) = T(tau)
  const double *Tp;     // tmask_limit_ts_same partner's T(tau) (PART)
  double *out[2];       // T(taup1)
  const double *th[2];  // other th_tendency terms, or null
  const double *U, *V, *W, *R, *Rm1, *Rr;
  const int *kmt;
  const double *dyte, *dxtn, *datr, *qw, *qz;
  double dtime, lo[2], hi[2], plo, phi;
  int lwu;              // limit_with_upwind
  int ts;               // G = 2: the two tracers' limit flags are OR'ed
  int ntx, ntiles;
};

// G tracers a pass; PART (G = 1): the flags of a partner tracer, which this
// pass does not advance, are formed from its T(tau) and OR'ed.  TH: some tracer has
// other th_tendency terms; their load sits between the prefetches and the store,
// so a pass without them must not hold it, nor the wait at the join of a branch
// around it, which would be for every prefetch.
template <int G, bool PART, bool TH, int NW>
__global__ __launch_bounds__(RX *NW) void k_quick_step(QStepJob J, int per_xcd) {
  const int b = blockIdx.x;
  const int t = (b & 7) * per_xcd + (b >> 3);
  if (t >= J.ntiles) return;
  const KDom d = J.d;
  constexpr int RY = NW, TY = RY - 4;
  const int tile = strip_tile<8>(t, J.ntx, J.ntiles / J.ntx);
  const int tix = tile % J.ntx, tiy = tile / J.ntx;
  const int lane = threadIdx.x & (RX - 1);
  const int row = __builtin_amdgcn_readfirstlane(threadIdx.x / RX);
  const int gi = tix * TX - 2 + lane, gj = tiy * TY - 2 + row;
  const int nk = d.nk, P2 = d.P2;
  const double dtime = J.dtime;
  // the level stride pinned in scalar registers: the compiler otherwise widens it
  // inside a divergent branch and keeps it, and every level base, per lane
  size_t P2l = (size_t)P2;
  asm volatile("" : "+s"(P2l));
  auto lev = [&](int k) { return P2l * (size_t)k; };

  __shared__ double s_t[2][G][RY][RX];   // T(k) of the region, for y neighbours
  __shared__ double s_tp[PART ? 2 : 1][PART ? RY : 1][RX];
  __shared__ double s_fy[2][G][RY][RX];  // flux through the north face of each point
  __shared__ int s_km[RY][RX];

  int si = gi, sj = gj;
  bool colok = true, rowok = true;
  if (si < 0 || si >= d.ni) {
    if (d.cyclic_x) si = wrapi(si, d.ni); else colok = false;
  }
  if (sj < 0 || sj >= d.nj) {
    if (d.cyclic_y) sj = wrapi(sj, d.nj); else rowok = false;
  }
  const bool ok = colok && rowok;
  const int off = ok ? d2(d, si, sj) : 0;
  const int km = ok ? J.kmt[off] : 0;
  s_km[row][lane] = km;

  // faces this point computes: east face of the point (x), north face (y)
  const bool xface = rowok && lane >= 1 && lane <= RX - 3 && gi >= -1 && gi <= d.ni - 1;
  const bool yface = row >= 1 && row <= RY - 3 && lane >= 2 && lane < RX - 2 && gi < d.ni &&
                     gj >= -1 && gj <= d.nj - 1;
  const bool cell = row >= 2 && row < RY - 2 && lane >= 2 && lane < RX - 2 && gi < d.ni &&
                    gj < d.nj;
  // offset 0 where there is no face (its values are not used)
  const int ox = xface ? d2(d, gi, sj) : 0, oy = yface ? d2(d, gi, gj) : 0;
  // Quicker weights (quicker_init), data-domain planes
  double qx0 = 0.0, qx1 = 0.0, cxp0 = 0.0, cxp1 = 0.0, cxp2 = 0.0, cxn0 = 0.0, cxn1 = 0.0,
         cxn2 = 0.0, dyte = 0.0;
  double qy0 = 0.0, qy1 = 0.0, cyp0 = 0.0, cyp1 = 0.0, cyp2 = 0.0, cyn0 = 0.0, cyn1 = 0.0,
         cyn2 = 0.0, dxtn = 0.0;
  if (xface) {
    const double *w = J.qw + ox;
    qx0 = w[0]; qx1 = w[P2];
    cxp0 = w[plane_at(4, P2)]; cxp1 = w[plane_at(5, P2)]; cxp2 = w[plane_at(6, P2)];
    cxn0 = w[plane_at(7, P2)]; cxn1 = w[plane_at(8, P2)]; cxn2 = w[plane_at(9, P2)];
    dyte = J.dyte[ox];
  }
  if (yface) {
    const double *w = J.qw + oy;
    qy0 = w[plane_at(2, P2)]; qy1 = w[plane_at(3, P2)];
    cyp0 = w[plane_at(10, P2)]; cyp1 = w[plane_at(11, P2)]; cyp2 = w[plane_at(12, P2)];
    cyn0 = w[plane_at(13, P2)]; cyn1 = w[plane_at(14, P2)]; cyn2 = w[plane_at(15, P2)];
    dxtn = J.dxtn[oy];
  }
  const double datr = cell ? J.datr[off] : 0.0;

  // byte offsets within a level: of the point, its east and its north face
  const unsigned bz = (unsigned)off * 8u, bx = (unsigned)ox * 8u, by = (unsigned)oy * 8u;
  const double *Rx = J.Rr ? J.Rr : J.R;
  // the k window of T: km1, k, kp1, min(k+2, nk) (clamped as the reference)
  double t0[G], t1[G], t2[G], t3[G], ft1[G], tp1 = 0.0, tp2 = 0.0;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    t0[g] = t1[g] = t2[g] = t3[g] = ft1[g] = 0.0;
    if (ok) {
      t1[g] = ld_lv(J.T[g], bz);
      t0[g] = t1[g];
      t2[g] = ld_lv(J.T[g] + lev(min(2, nk) - 1), bz);
      t3[g] = ld_lv(J.T[g] + lev(min(3, nk) - 1), bz);
    }
    s_t[1][g][row][lane] = t1[g];
  }
  if constexpr (PART) {
    if (ok) {
      tp1 = ld_lv(J.Tp, bz);
      tp2 = ld_lv(J.Tp + lev(min(2, nk) - 1), bz);
    }
    s_tp[1][row][lane] = tp1;
  }
  double nu = ld_lv(J.U, bx), nv = ld_lv(J.V, by), nw = ld_lv(J.W + P2, bz),
         nm = ld_lv(J.Rm1, bz), nr = ld_lv(Rx, bz);
  __syncthreads();
  // depths of the neighbours the coastal substitutions and limits read
  const int km_w = dpp_prev(km);
  const int km_e = dpp_next(km), km_e2 = dpp_next(km_e);
  const int rm = max(row - 1, 0), rp = min(row + 1, RY - 1), rp2 = min(row + 2, RY - 1);
  const int km_s = s_km[rm][lane], km_n = s_km[rp][lane], km_n2 = s_km[rp2][lane];
  // the vertical weights through the scalar cache: as vector loads each would
  // wait for every load in flight (loads return in order)
  typedef const __attribute__((address_space(4))) double ConstD;
  ConstD *qz = (ConstD *)(unsigned long long)J.qz;

  for (int kk = 1; kk <= nk; ++kk) {
    // the level in a scalar register: scalar level bases and weights
    const int k = __builtin_amdgcn_readfirstlane(kk);
    const int bb = k & 1;
    const int km1 = max(k - 1, 1), kp1 = min(k + 1, nk), p2 = min(k + 2, nk);
    const double u = nu, v = nv, vel_z = nw, rm1 = nm, rxk = nr;
    // the next level's inputs (the last level loads its own again)
    double t4[G], tp3 = 0.0;
    {
      // in the order of their use: a wait for one is then not for a later one, nor
      // for the store that follows
      const size_t pn = lev(min(k, nk - 1)), pw = lev(min(k + 1, nk));
      const size_t p3 = lev(min(k + 3, nk) - 1);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        t4[g] = 0.0;
        if (ok) t4[g] = ld_lv(J.T[g] + p3, bz);
      }
      if constexpr (PART) {
        if (ok) tp3 = ld_lv(J.Tp + lev(p2 - 1), bz);
      }
      nu = ld_lv(J.U + pn, bx);
      nv = ld_lv(J.V + pn, by);
      nw = ld_lv(J.W + pw, bz);
      nm = ld_lv(J.Rm1 + pn, bz);
      nr = ld_lv(Rx + pn, bz);
    }
    const double z0 = qz[k - 1], z1 = qz[k - 1 + nk];                   // quick_z
    const double p0 = qz[k - 1 + 2 * nk], p1 = qz[k - 1 + 3 * nk], p2w = qz[k - 1 + 4 * nk];
    const double n0 = qz[k - 1 + 5 * nk], n1 = qz[k - 1 + 6 * nk], n2 = qz[k - 1 + 7 * nk];
    const double m0 = mk(k, km), me = mk(k, km_e), mn = mk(k, km_n);
    const double mb = (k < nk) ? mk(k + 1, km) : 0.0;
    double te[G], tn[G];
    // tmask_limit(i,j,k) of this point (ocean_tracer.F90:2803-2850, 2858-2869)
    double L[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      te[g] = lane_next(t1[g]);
      tn[g] = s_t[bb][g][rp][lane];
      L[g] = 0.0;
      if (m0 == 1.0 && outside(t1[g], J.lo[g], J.hi[g])) L[g] = m0;
      if (me == 1.0 && outside(te[g], J.lo[g], J.hi[g])) L[g] = m0;
      if (mn == 1.0 && outside(tn[g], J.lo[g], J.hi[g])) L[g] = m0;
      if (k < nk && mb == 1.0 && outside(t2[g], J.lo[g], J.hi[g])) L[g] = m0;
    }
    if constexpr (PART) {
      double Lp = 0.0;
      const double pe = lane_next(tp1), pn = s_tp[bb][rp][lane];
      if (m0 == 1.0 && outside(tp1, J.plo, J.phi)) Lp = m0;
      if (me == 1.0 && outside(pe, J.plo, J.phi)) Lp = m0;
      if (mn == 1.0 && outside(pn, J.plo, J.phi)) Lp = m0;
      if (k < nk && mb == 1.0 && outside(tp2, J.plo, J.phi)) Lp = m0;
      if (L[0] == 1.0 || Lp == 1.0) L[0] = 1.0;
    }
    if constexpr (G == 2) {
      if (J.ts && (L[0] == 1.0 || L[1] == 1.0)) L[0] = L[1] = 1.0;
    }

    double fx[G], fxw[G], fy[G];
    const double velx = dyte * u, vely = dxtn * v;
    const double xpos = 0.5 * (velx + fabs(velx)), xneg = 0.5 * (velx - fabs(velx));
    const double ypos = 0.5 * (vely + fabs(vely)), yneg = 0.5 * (vely - fabs(vely));
    const double eastmsk = m0 * (1.0 - mk(k, km_w));
    const double westmsk = me * (1.0 - mk(k, km_e2));
    const double rnormsk = m0 * (1.0 - mk(k, km_s));
    const double soutmsk = mn * (1.0 - mk(k, km_n2));
#pragma unroll
    for (int g = 0; g < G; ++g) {
      // x flux through the east face of this point (:2590-2606, 2610-2622)
      const double te2 = lane_next(te[g]), tw = lane_prev(t1[g]);
      double f = 0.0;
      if (xface) {
        f = velx * (qx0 * t1[g] + qx1 * te[g]) -
            xpos * (cxp0 * te[g] + cxp1 * t1[g] + cxp2 * (tw * (1.0 - eastmsk) + t1[g] * eastmsk)) -
            xneg * (cxn0 * (te2 * (1.0 - westmsk) + te[g] * westmsk) + cxn1 * te[g] + cxn2 * t1[g]);
        if (J.lwu && L[g] == 1.0) {
          const double up = 0.5 * (u + fabs(u)), un = 0.5 * (u - fabs(u));
          f = dyte * (up * t1[g] + un * te[g]) * m0 * me;
        }
      }
      fx[g] = f;
      fxw[g] = lane_prev(f);
      // y flux through the north face (:2573-2587, 2623-2635)
      fy[g] = 0.0;
      if (yface) {
        const double tn2 = s_t[bb][g][rp2][lane], ts = s_t[bb][g][rm][lane];
        f = vely * (qy0 * t1[g] + qy1 * tn[g]) -
            ypos * (cyp0 * tn[g] + cyp1 * t1[g] + cyp2 * (ts * (1.0 - rnormsk) + t1[g] * rnormsk)) -
            yneg * (cyn0 * (tn2 * (1.0 - soutmsk) + tn[g] * soutmsk) + cyn1 * tn[g] + cyn2 * t1[g]);
        if (J.lwu && L[g] == 1.0) {
          const double up = 0.5 * (v + fabs(v)), un = 0.5 * (v - fabs(v));
          f = dxtn * (up * t1[g] + un * tn[g]) * m0 * mn;
        }
        fy[g] = f;
        s_fy[bb][g][row][lane] = f;
      }
      s_t[bb ^ 1][g][row][lane] = t2[g];
    }
    if constexpr (PART) s_tp[bb ^ 1][row][lane] = tp2;
    // One barrier a level: before it a wavefront writes the copies the next
    // level reads (T) and this update reads (fluxes); the other copies were
    // last read before the previous barrier (T) or are rewritten only after
    // the next one (fluxes).
    __syncthreads();

    if (cell) {
      // vertical flux through the bottom face (:3002-3028)
      const double upos = 0.5 * (vel_z + fabs(vel_z));
      const double uneg = 0.5 * (vel_z - fabs(vel_z));
      const double mkp1 = mk(kp1, km), mkp2 = mk(p2, km);
      const double upmsk = m0 * (1.0 - mk(km1, km));
      const double rr = J.Rr ? rxk : 1.0 / (rxk + 1.0e-40);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const double fys = s_fy[bb][g][row - 1][lane];
        const double res_h = m0 * (fx[g] - fxw[g] + fy[g] - fys) * datr;
        double ft2;
        if (L[g] == 1.0) {
          ft2 = (uneg * t1[g] + upos * t2[g]) * m0 * mkp1;
        } else {
          // kp2 = p2 where that level is wet, else kp1 (:3010)
          const double tkp2 = (mkp2 == 1.0) ? t3[g] : t2[g];
          ft2 = vel_z * (z0 * t1[g] + z1 * t2[g]) -
                uneg * (p0 * t2[g] + p1 * t1[g] + p2w * t0[g]) -
                upos * (n0 * tkp2 + n1 * t2[g] + n2 * (t1[g] * (1.0 - upmsk) + t2[g] * upmsk));
        }
        const double res_v = m0 * (ft1[g] - ft2);
        ft1[g] = ft2;
        const size_t pk = lev(k - 1);
        double th = 0.0;
        if constexpr (TH) th = J.th[g] ? ld_lv(J.th[g] + pk, bz) : 0.0;
        th = th + (-res_h);
        th = th + (-res_v);
        st_lv(J.out[g] + pk, bz, (rm1 * t1[g] + dtime * th) * rr);
      }
    }

    // advance the k window
#pragma unroll
    for (int g = 0; g < G; ++g) {
      t0[g] = t1[g]; t1[g] = t2[g]; t2[g] = t3[g]; t3[g] = t4[g];
    }
    if constexpr (PART) {
      tp1 = tp2;
      tp2 = tp3;
    }
  }
}

template <int G, bool PART, bool TH>
void launch_th(mom_gpu_ctx *ctx, QStepJob J) {
  // two tracers need 162 VGPRs (at 16 wavefronts' 128 they spill: 9.4 ms for the
  // case that takes 5.9 with 12)
  constexpr int NW = G == 2 ? 12 : 16, TY = NW - 4;
  const KDom &d = ctx->kd;
  J.ntx = (d.ni + TX - 1) / TX;
  J.ntiles = J.ntx * ((d.nj + TY - 1) / TY);
  const int per = (J.ntiles + 7) / 8;
  hipLaunchKernelGGL((k_quick_step<G, PART, TH, NW>), dim3(8 * per), dim3(RX * NW), 0, ctx->stream,
                     J, per);
}

template <int G, bool PART>
void launch_one(mom_gpu_ctx *ctx, const QStepJob &J) {
  if (J.th[0] || (G == 2 && J.th[1])) launch_th<G, PART, true>(ctx, J);
  else launch_th<G, PART, false>(ctx, J);
}

}  // namespace

// The Quicker tracers of a batched step (scheme[n] == MOM_ADVECT_QUICKER,
// FP64 only), two a pass.  it/is: 0-based temp/salt indices (-1: none); with
// ts_same their limit flags are OR'ed: they share a pass when both are
// Quicker, otherwise the Quicker one reads the partner's T(tau).
int launch_quicker_step(mom_gpu_ctx *ctx, int ntr, const void *const *T_in, void *const *T_out,
                        const int *scheme, const double *const *th_in, const double *mn,
                        const double *mx, int it, int is, int ts_same, int lwu,
                        const double *u, const double *v, const double *w, const double *rho,
                        const double *rho_taum1, const double *rho_dztr, double dtime) {
  const bool ts = ts_same && it >= 0 && is >= 0;
  std::vector<int> order;        // the pairs that share a pass, then a last single
  const bool pair = ts && it != is && scheme[it] == MOM_ADVECT_QUICKER &&
                    scheme[is] == MOM_ADVECT_QUICKER;
  if (pair) order = {it, is};
  std::vector<int> alone;        // flags from a partner that is not Quicker
  for (int n = 0; n < ntr; ++n) {
    if (scheme[n] != MOM_ADVECT_QUICKER || (pair && (n == it || n == is))) continue;
    if (ts && (n == it || n == is)) alone.push_back(n); else order.push_back(n);
  }
  QStepJob J{};
  J.d = ctx->kd;
  J.U = u; J.V = v; J.W = w; J.R = rho; J.Rm1 = rho_taum1; J.Rr = rho_dztr;
  J.kmt = ctx->kmt;
  J.dyte = ctx->dyte; J.dxtn = ctx->dxtn; J.datr = ctx->datr;
  J.qw = ctx->qw; J.qz = ctx->qzw;
  J.dtime = dtime;
  J.lwu = lwu ? 1 : 0;
  auto take = [&](int q, int n) {
    J.T[q] = (const double *)T_in[n];
    J.out[q] = (double *)T_out[n];
    J.th[q] = th_in ? th_in[n] : nullptr;
    J.lo[q] = mn[n]; J.hi[q] = mx[n];
  };
  for (size_t i = 0; i < order.size(); i += 2) {
    take(0, order[i]);
    J.ts = pair && i == 0;
    if (i + 1 < order.size()) {
      take(1, order[i + 1]);
      launch_one<2, false>(ctx, J);
    } else {
      launch_one<1, false>(ctx, J);
    }
    MOM_LAUNCHED(ctx, "k_quick_step");
  }
  for (int n : alone) {
    const int partner = n == it ? is : it;
    take(0, n);
    J.Tp = (const double *)T_in[partner];
    J.plo = mn[partner]; J.phi = mx[partner];
    launch_one<1, true>(ctx, J);
    MOM_LAUNCHED(ctx, "k_quick_step");
  }
  return MOM_GPU_OK;
}
