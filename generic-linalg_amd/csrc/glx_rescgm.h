// glx_rescgm.h -- multishift CG (generic_cg_m.cpp:312-600) on D^dag D with the
// whole system held on the chip, every shift's x_s and p_s included.
//
// What bounds it: a launch per phase takes five launches per iteration and
// moves 64 B per active shift and site through memory.  Here one launch is the
// solve: an iteration is its two chip-wide reductions (glx_restile.h) and one
// D^dag D; the 12 multiply-adds per shift and site of x_s and p_s run while
// the next iteration's <p, Ap> is on its way.  The shifts' recurrences are one
// lane's each.  One row per wave (R = 1): with 16 shifts x_s and p_s take 128
// registers of a lane, so lattices up to 256 tiles of 60 x 8 sites run here.
// The whole solve, 200 x 144, 12 shifts, residuals included: 7.6 ms with a
// launch per phase, 2.1 ms here.
#pragma once

#include "glx_resident.h"

namespace glx {

__global__ __launch_bounds__(kRsThreads) inline void k_rs_cgm(RsGeom g, RsSolve so, RsShiftSet sh_) {
  using T = c128;
  using Sh = RsShared<T, 1>;
  __shared__ Sh sh;
  RsTile<T, 1, 2> t(sh.ex, g, so.ring, so.lines, so.spins);
  RsNormal<T, 1> op(sh, t, so.lk, so.mass);
  const T z = zero_of<T>();
  const bool edge = t.edge, own = t.own;
  auto at = [&](int y) -> int { return y * t.lx + t.xg; };
  T r[1], p[1], ap[1], xs[kRsShifts], ps[kRsShifts];
  if (threadIdx.x == 0) sh.ex.bad = 0;
  const bool lead = t.blk == 0 && threadIdx.x == 0;
  auto give_up = [&]() {
    if (threadIdx.x == 0) so.out->err = 1;
  };
  // lane n of every wave carries shift n
  const int me = t.lane < kRsShifts ? t.lane : 0;
  const double sigma = t.lane < sh_.n ? sh_.shift[me] : 0.0;
  bool active = t.lane < sh_.n;
  c128 zeta{1.0, 0.0}, zeta_p{1.0, 0.0}, beta_s{1.0, 0.0}, alpha_s{0.0, 0.0};

  // ---- r = p = p_s = b (x = 0)
  const T b0 = t.valid ? so.b[at(t.yw)] : z;
  r[0] = p[0] = b0;
#pragma unroll
  for (int n = 0; n < kRsShifts; n++) {
    xs[n] = z;
    ps[n] = b0;
  }
  if (edge) {
#pragma unroll
    for (int h = 0; h < 2; h++) op.hal(RS_RH + h) = op.hal(RS_PH + h) = t.valid ? so.b[at(t.yh[h])] : z;
  }
  int k = 0, c = 0, e = 0;
  double rsq = 0.0, bsqrt = 0.0;
  c128 alpha{0.0, 0.0}, beta{1.0, 0.0};
  const int kmax = so.max_iter - 1;
  auto lane_c = [&](c128 v, int n) { return c128{readlane_d(v.re, n), readlane_d(v.im, n)}; };
  // x_s -= beta_s p_s, and p_s = zeta_s r + alpha_s p_s for the shifts of `more`
  auto shifts = [&](unsigned long long upd, unsigned long long more) {
#pragma unroll
    for (int n = 0; n < kRsShifts; n++) {
      if (!(upd >> n & 1)) continue;
      const c128 bs = lane_c(beta_s, n);
      xs[n] = rs_axpy(c128{-bs.re, -bs.im}, ps[n], xs[n]);
      if (more >> n & 1) {
        const c128 a = lane_c(alpha_s, n), zs = lane_c(zeta, n);
        const T w{a.re * ps[n].re - a.im * ps[n].im, a.re * ps[n].im + a.im * ps[n].re};
        ps[n] = rs_axpy(zs, r[0], w);
      }
    }
  };
  unsigned long long upd = 0, more = 0;
  __syncthreads();
  {
    double n2[1] = {own && t.counts(0) ? norm2(b0) : 0.0};
    t.publish(n2, c);
    if (!t.collect(n2, c)) return give_up();
    c++;
    rsq = n2[0];
    bsqrt = sqrt(rsq);
  }
  for (;; k++) {
    double pap[2] = {0.0, 0.0};
    op.apply(p, ap, [&](int j, T v) {
      if (own && t.counts(j)) {
        pap[0] = p[j].re * v.re + p[j].im * v.im;
        pap[1] = p[j].re * v.im - p[j].im * v.re;
      }
    });
    t.publish(ap, e, pap, c);
    shifts(upd, more);  // (the last iteration's)
    if (!t.collect(ap, [&](int h, T v) { op.hal(RS_APH + h) = v; }, e, pap, c)) return give_up();
    e++;
    c++;
    // ---- beta, and the active shifts' zeta and beta_s (generic_cg_m.cpp:106-122)
    const c128 beta_p = beta;
    beta = cdiv(c128{-rsq, 0.0}, c128{pap[0], pap[1]});
    // ---- r += beta Ap
    r[0] = rs_axpy(beta, ap[0], r[0]);
    double rn[1] = {own && t.counts(0) ? norm2(r[0]) : 0.0};
    t.publish(rn, c);
    if (edge) {
#pragma unroll
      for (int h = 0; h < 2; h++) op.hal(RS_RH + h) = rs_axpy(beta, op.hal(RS_APH + h), op.hal(RS_RH + h));
    }
    if (active) {
      const c128 num = (zeta * zeta_p) * beta_p;
      const c128 sb = sigma * beta;
      const c128 den = (beta * alpha) * (zeta_p - zeta) + (zeta_p * beta_p) * c128{1.0 - sb.re, -sb.im};
      zeta_p = zeta;
      zeta = cdiv(num, den);
      beta_s = cdiv(beta * zeta, zeta_p);
    }
    if (!t.collect(rn, c)) return give_up();
    c++;
    if (lead && so.hist) so.hist[k] = sqrt(rn[0]) / bsqrt;
    // ---- convergence and alpha (generic_cg_m.cpp:139-215)
    upd = __ballot(active);
    if (k % sh_.freq == 0 && active && hypot(zeta.re, zeta.im) * sqrt(rn[0]) < so.eps * bsqrt) active = false;
    more = __ballot(active);
    if (more == 0 || k == kmax) break;
    const double al = rn[0] / rsq;
    alpha = {al, 0.0};
    rsq = rn[0];
    if (active) alpha_s = cdiv((alpha * zeta) * beta_s, zeta_p * beta);
    p[0] = rs_axpy(al, p[0], r[0]);
    if (edge) {
#pragma unroll
      for (int h = 0; h < 2; h++) op.hal(RS_PH + h) = rs_axpy(al, op.hal(RS_PH + h), op.hal(RS_RH + h));
    }
  }
  shifts(upd, 0);
  // ---- the solutions to memory, then every shift's true residual
#pragma unroll
  for (int n = 0; n < kRsShifts; n++)
    if (n < sh_.n && own && t.counts(0))
      rs_put<T>(reinterpret_cast<unsigned long long*>(sh_.x[n] + at(t.yw)), xs[n]);
  {
    double none[1] = {0.0};
    t.publish(none, c);  // (waits for the stores of x first)
    if (!t.collect(none, c)) return give_up();
    c++;
  }
  for (int n0 = 0; n0 < sh_.n; n0 += 4) {
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int q = 0; q < 4 && n0 + q < sh_.n; q++) {
      double s2[2];
      rs_normal_residual<T, 1>(t, so.u64, so.mass, sh_.shift[n0 + q], sh_.x[n0 + q], so.b, at, ap, s2);
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (i == q) v[i] = s2[0];
    }
    t.publish(v, c);
    if (!t.collect(v, c)) return give_up();
    c++;
    if (lead)
      for (int q = 0; q < 4 && n0 + q < sh_.n; q++) sh_.res[n0 + q] = q == 0 ? v[0] : (q == 1 ? v[1] : (q == 2 ? v[2] : v[3]));
  }
  if (lead) {
    so.out->kfinal = k;
    so.out->bsqrt = bsqrt;
    so.out->done = 1;
  }
}

}  // namespace glx
