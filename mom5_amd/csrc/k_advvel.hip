// Advection velocity on the B-grid: ocean_advection_velocity
// (ocean_core/ocean_advection_velocity.F90:568-672, no blobs, OBC or
// prescribed inflow), T-cell part.
//
// A work-group of sixteen wavefronts owns 63 x 15 columns plus the column west
// and the row south of them, and marches down k; a level's inputs are loaded
// during the level before.  The operators of ocean_core/ocean_operators.F90
// (halo 1) are evaluated point-wise: BAY (:889-902) and BAX (:834-846) average
// the U-cell transport u*dy(x)u*rho_dzu backwards and divide by the T-face
// length; BDX_ET (:945-958) and BDY_NT (:1230-1243) difference the face
// transports backwards.  A point takes its west neighbour's face transport by a
// lane shift and its south neighbour's values through LDS (two copies by level
// parity, one barrier a level), so that each is formed once, as the
// reference's array-valued functions hold it, bit for bit.
//
// Bound by HBM: 32 B read and 32 B written per cell with both outputs and
// rho_dzt_tendency.  A thread per column that read its three neighbours' inputs
// and formed their transports again (twelve loads and four divisions a cell)
// took 2.27 ms at 1440x1080x50; this form 1.26 ms (5.4 GB moved, 4.3 TB/s, what a
// large copy reaches here).  Tiles run row by row in an XCD's share (8-wide strips:
// 1.34 ms).
#include "mom_internal.h"

namespace {

constexpr int AX = 64, AY = 16;      // region: one row a wavefront

struct AdvIn {
  const double *u1, *u2, *rdu, *rtend, *msrc;
};

__global__ __launch_bounds__(AX *AY) void k_adv_vel(
    KDom d, AdvIn in, const double *__restrict__ dyu, const double *__restrict__ dxu,
    const double *__restrict__ dyte, const double *__restrict__ dxtn,
    const double *__restrict__ datr, const int *__restrict__ kmt,
    const double *__restrict__ pme, const double *__restrict__ river,
    double *__restrict__ ue_out, double *__restrict__ vn_out, double *__restrict__ wb,
    double *__restrict__ div_out, int ntx, int ntiles, int per_xcd) {
  const int b = blockIdx.x;
  const int t = (b & 7) * per_xcd + (b >> 3);
  if (t >= ntiles) return;                     // the whole block
  const int tile = strip_tile<32>(t, ntx, ntiles / ntx);
  __shared__ double s_a[2][AY][AX], s_v[2][AY][AX];
  const int lane = threadIdx.x & (AX - 1);
  const int row = __builtin_amdgcn_readfirstlane(threadIdx.x / AX), rs = max(row - 1, 0);
  const int ii = (tile % ntx) * (AX - 1) - 1 + lane, jj = (tile / ntx) * (AY - 1) - 1 + row;
  const bool present = ii >= 0 && ii < d.NI && jj >= 0 && jj < d.NJ;
  const bool out = present && lane >= 1 && row >= 1;
  const bool hw = ii >= 1, hs = jj >= 1;
  const size_t P2 = (size_t)d.P2;
  // a point outside the domain reads point 0 (the values are not used)
  const int o = present ? ii + d.NI * jj : 0;
  const int km = kmt[o];
  const double dyuo = dyu[o], dxuo = dxu[o], dyteo = dyte[o], dxtno = dxtn[o], datro = datr[o];
  double w = -(pme[o] + river[o]);
  if (out) wb[o] = w;
  double u1 = in.u1[o], u2 = in.u2[o], rdu = in.rdu[o];
  double rt = in.rtend ? in.rtend[o] : 0.0, ms = in.msrc ? in.msrc[o] : 0.0;
  for (int k = 0; k < d.nk; ++k) {
    const size_t L = P2 * (size_t)k + o;
    const size_t N = L + (k + 1 < d.nk ? P2 : 0);      // the last level loads itself again
    const double nu1 = in.u1[N], nu2 = in.u2[N], nrdu = in.rdu[N];
    const double nrt = in.rtend ? in.rtend[N] : 0.0, nms = in.msrc ? in.msrc[N] : 0.0;
    // BAX(u2*dxu*rho_dzu)/dxtn, BAY(u1*dyu*rho_dzu)/dyte
    const double a_c = u1 * dyuo * rdu, b_c = u2 * dxuo * rdu;
    const double b_w = lane_prev(b_c);
    const double vn = (hw ? 0.5 * (b_c + b_w) : 0.0) / dxtno;
    const double mv = dxtno * vn;
    s_a[k & 1][row][lane] = a_c;
    s_v[k & 1][row][lane] = mv;
    __syncthreads();
    const double a_s = s_a[k & 1][rs][lane], mv_s = s_v[k & 1][rs][lane];
    const double ue = (hs ? 0.5 * (a_c + a_s) : 0.0) / dyteo;
    const double mu = dyteo * ue, mu_w = lane_prev(mu);
    const double bdx = hw ? (mu - mu_w) * datro : 0.0;
    const double bdy = hs ? (mv - mv_s) * datro : 0.0;
    const double tm = (k + 1 <= km) ? 1.0 : 0.0;
    const double dv = tm * (bdx + bdy);
    w = ((rt - ms) + dv + w) * tm;
    if (out) {
      ue_out[L] = ue;
      vn_out[L] = vn;
      wb[L + P2] = w;
      if (div_out) div_out[L] = dv;
    }
    u1 = nu1; u2 = nu2; rdu = nrdu; rt = nrt; ms = nms;
  }
}

}  // namespace

int launch_adv_vel(mom_gpu_ctx *ctx, const double *u, const double *rho_dzu, const double *pme,
                   const double *river, const double *rtend, const double *msrc, double *ue,
                   double *vn, double *wb, double *div) {
  const KDom &d = ctx->kd;
  const size_t p3 = (size_t)d.P2 * d.nk;
  const int ntx = (d.NI + AX - 2) / (AX - 1), ntiles = ntx * ((d.NJ + AY - 2) / (AY - 1));
  const int per_xcd = (ntiles + 7) / 8;
  hipLaunchKernelGGL(k_adv_vel, dim3(8 * per_xcd), dim3(AX * AY), 0, ctx->stream, d,
                     AdvIn{u, u + p3, rho_dzu, rtend, msrc}, ctx->dyu, ctx->dxu, ctx->dyte,
                     ctx->dxtn, ctx->datr, ctx->kmt, pme, river, ue, vn, wb, div, ntx, ntiles,
                     per_xcd);
  MOM_LAUNCHED(ctx, "k_adv_vel");
  return MOM_GPU_OK;
}
