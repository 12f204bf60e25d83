// glx_reshop.h -- CG and BiCGStab in the reference's order with the whole
// system held on the chip, on the operators of one hop: the Laplacians
// (operators.cpp:28-120, tests/multishift/multishift.cpp:634-672) and the
// staggered D and D^dag (operators.cpp:184-239, :372-441).
//
//   A v(x) = d v(x) + sum_mu [ V_mu(x) v(x+mu) + SB V_mu(x-mu)^* v(x-mu) ],
//
// V the links with the operator's factor and phase (-U for the Laplacians,
// -+ eta U / 2 for D and D^dag) and SB = +1 or -1; the real Laplacian has no
// links.
//
// What bounds it: a launch per iteration spends its time on 4 to 6 dependent
// launches of about 4 us.  Here an iteration is the chain of its chip-wide
// reductions (CG two, BiCGStab three of 1.3 to 2 us each, glx_restile.h) with
// one hop between them; the vectors never leave the registers (FP64 x and the
// shadow residual LDS where a wave holds many rows).  A whole
// solve, a launch per phase against this: real Laplacian 64^2, CG, 149
// iterations, host vectors 2.60 against 0.55 ms; D 256^2, BiCGStab, about 620
// iterations 15.7 against 4.8 ms (25 against 7.7 us per iteration).
#pragma once

#include "glx_restile.h"

namespace glx {

// The operator on a tile: links in registers, the wave boundaries' rows in LDS.
template <class T, int R>
struct RsHopShared {
  T v[2][kRsWaves][2][64];
};

template <class T, int R, int SB>
struct RsHop {
  static constexpr bool kLinks = is_cx<T>::value;
  RsHopShared<T, R>& sh;
  double d;
  T ux[kLinks ? R : 1], uy[kLinks ? R : 1], uyt;

  __device__ __forceinline__ void links(const RsSolve& so, int i, int xg, T& a, T& b) const {
    if constexpr (kLinks) {
      if (!so.u64) {
        a = b = T{so.fx, 0.0};
        return;
      }
      rs_links<double>(RsLinks{so.u64, nullptr, 0}, i, so.fx, (xg & 1) ? so.fy_odd : so.fx, a, b);
    }
  }
  template <class Tile>
  __device__ __forceinline__ RsHop(RsHopShared<T, R>& s, const Tile& t, const RsSolve& so) : sh(s), d(so.diag) {
    ux[0] = uy[0] = uyt = zero_of<T>();
    if constexpr (kLinks) {
#pragma unroll
      for (int j = 0; j < R; j++) {
        ux[j] = uy[j] = zero_of<T>();
        if (t.valid) links(so, (t.yw + j) * t.lx + t.xg, t.xg, ux[j], uy[j]);
      }
      T a;
      if (t.valid) links(so, t.wrapy(t.yw - 1) * t.lx + t.xg, t.xg, a, uyt);
    }
  }
  // A v at one site; uym = V_y(y - 1)
  __device__ __forceinline__ T at(T v, T up, T dn, T x, T y, T uym) const {
    if constexpr (kLinks) {
      const T z = zero_of<T>();
      const T dv{d * v.re, d * v.im};
      if constexpr (SB > 0) {
        const T back = rs_shift<kDwPrev>(rs_maddc(z, x, v));
        return dv + rs_maddc(rs_madd(rs_madd(back, x, rs_shift<kDwNext>(v)), y, dn), uym, up);
      } else {
        const T back = rs_shift<kDwPrev>(rs_msubc(z, x, v));
        return dv + rs_msubc(rs_madd(rs_madd(back, x, rs_shift<kDwNext>(v)), y, dn), uym, up);
      }
    } else {
      return rs_fma(d, v, -((rs_shift<kDwNext>(v) + rs_shift<kDwPrev>(v)) + (dn + up)));
    }
  }
  // out = A v over the wave's rows (rim lanes of v hold the neighbours'
  // columns, `halo` the edge waves' halo row); `buf` alternates between calls
  template <class Tile>
  __device__ __forceinline__ void apply(const Tile& t, const T (&v)[R], T halo, int buf, T (&out)[R]) const {
    sh.v[buf][t.wave][0][t.lane] = v[0];
    sh.v[buf][t.wave][1][t.lane] = v[R - 1];
    __syncthreads();
    const T up = t.top ? halo : sh.v[buf][t.top ? 0 : t.wave - 1][1][t.lane];
    const T below = t.wave == kRsWaves - 1 ? halo : sh.v[buf][t.wave + 1 < kRsWaves ? t.wave + 1 : t.wave][0][t.lane];
#pragma unroll
    for (int j = 0; j < R; j++) {
      if constexpr (kLinks && R >= 4) __builtin_amdgcn_sched_barrier(0);
      const int jl = kLinks ? j : 0;
      out[j] = at(v[j], j ? v[j ? j - 1 : 0] : up, j + 1 < R ? v[j + 1 < R ? j + 1 : j] : below, ux[jl], uy[jl],
                  j ? uy[kLinks && j ? j - 1 : 0] : uyt);
    }
  }
  // r = b - A x from memory (own lanes), with |r|^2 and |b|^2 of the counted
  // rows in s2: a march down the rows, at step i the loads of row i - 1 of the
  // run and A x on the row before it
  template <class Tile>
  __device__ __forceinline__ void residual(const Tile& t, const RsSolve& so, T (&r)[R], double (&s2)[2]) const {
    const T z = zero_of<T>();
    const T* xp = reinterpret_cast<const T*>(so.x);
    const T* bp = reinterpret_cast<const T*>(so.b);
    T xa = z, xb = z, u1x = z, u1y = z, u0y = z;
    s2[0] = s2[1] = 0.0;
#pragma unroll 1
    for (int i = 0; i < R + 2; i++) {
      const int y = t.wrapy(t.yw - 1 + i), k = y * t.lx + t.xg;
      T xc = z, ucx = z, ucy = z;
      if (t.valid) {
        xc = rs_read<T>(reinterpret_cast<const unsigned long long*>(xp + k));
        links(so, k, t.xg, ucx, ucy);
      }
      const T ax = at(xb, xa, xc, u1x, u1y, u0y);
      if (i >= 2) {
        const int j = i - 2;
        T dr = z;
        if (t.own) {
          const T bv = bp[(t.yw + j) * t.lx + t.xg];
          dr = bv - ax;
          if (t.counts(j)) {
            s2[0] += norm2(dr);
            s2[1] += norm2(bv);
          }
        }
#pragma unroll
        for (int jj = 0; jj < R; jj++)
          if (jj == j) r[jj] = dr;
      }
      xa = xb;
      xb = xc;
      u0y = u1y;
      u1x = ucx;
      u1y = ucy;
    }
  }
};

// A per-row vector in registers, or in LDS slots of the thread's own.
template <class T, int R, bool LDS>
struct RsRows {
  T v[R];
  __device__ __forceinline__ T& operator[](int j) { return v[j]; }
  __device__ __forceinline__ explicit RsRows(T (*)[kRsThreads]) {}
};
template <class T, int R>
struct RsRows<T, R, true> {
  T (*m)[kRsThreads];
  __device__ __forceinline__ T& operator[](int j) { return m[j][threadIdx.x]; }
  __device__ __forceinline__ explicit RsRows(T (*q)[kRsThreads]) : m(q) {}
};

__device__ __forceinline__ void rs_dot(double (&s)[2], c128 a, c128 b) {  // s += conj(a) b
  s[0] = __builtin_fma(a.re, b.re, __builtin_fma(a.im, b.im, s[0]));
  s[1] = __builtin_fma(a.re, b.im, __builtin_fma(-a.im, b.re, s[1]));
}
__device__ __forceinline__ void rs_dot(double (&s)[2], double a, double b) { s[0] = __builtin_fma(a, b, s[0]); }
__device__ __forceinline__ void rs_norm(double& s, c128 a) { s = __builtin_fma(a.re, a.re, __builtin_fma(a.im, a.im, s)); }
__device__ __forceinline__ void rs_norm(double& s, double a) { s = __builtin_fma(a, a, s); }

template <class T, int R>
struct RsHcgShared {
  static constexpr bool kX = sizeof(T) == 16 && R >= 6;  // x in LDS
  RsExShared<T, R, 1> ex;
  RsHopShared<T, R> op;
  T x[kX ? R : 1][kRsThreads];
};

// generic_cg.cpp:132-231 (real), :278-382 (complex)
template <class T, int R, int SB>
__global__ __launch_bounds__(kRsThreads) void k_rs_hcg(RsGeom g, RsSolve so) {
  using Sh = RsHcgShared<T, R>;
  __shared__ Sh sh;
  RsTile<T, R, 1> t(sh.ex, g, so.ring, so.lines, so.spins);
  const RsHop<T, R, SB> A(sh.op, t, so);
  RsRows<T, R, Sh::kX> x(sh.x);
  T r[R], p[R], ap[R], rh = zero_of<T>(), ph = rh, aph = rh;
  T* xp = reinterpret_cast<T*>(so.x);
#pragma unroll
  for (int j = 0; j < R; j++) {
    p[j] = zero_of<T>();
    x[j] = t.own ? xp[(t.yw + j) * t.lx + t.xg] : zero_of<T>();
  }
  if (threadIdx.x == 0) sh.ex.bad = 0;
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  auto give_up = [&]() {
    if (threadIdx.x == 0) so.out->err = 1;
  };
  int k = 0, c = 0, e = 0;
  double rsq = 0.0, be = 0.0, bsqrt = 0.0, resSq = 0.0;
  const int kmax = so.max_iter - 1;
  __syncthreads();
  for (bool first = true;; first = false) {
    double s2[2];
    A.residual(t, so, r, s2);
    t.publish(r, e, s2, c);
    if (!t.collect(r, [&](int, T v) { rh = v; }, e, s2, c)) return give_up();
    e++;
    c++;
    if (!first) {
      resSq = s2[0];
      break;
    }
    rsq = s2[0];
    bsqrt = sqrt(s2[1]);
    for (;; k++) {
#pragma unroll
      for (int j = 0; j < R; j++) p[j] = rs_axpy(be, p[j], r[j]);
      ph = rs_axpy(be, ph, rh);
      A.apply(t, p, ph, 0, ap);
      double pap[2] = {0.0, 0.0};
#pragma unroll
      for (int j = 0; j < R; j++)
        if (t.counts(j)) rs_dot(pap, p[j], ap[j]);
      pap[0] = t.own ? pap[0] : 0.0;
      pap[1] = t.own ? pap[1] : 0.0;
      t.publish(ap, e, pap, c);
      if (!t.collect(ap, [&](int, T v) { aph = v; }, e, pap, c)) return give_up();
      e++;
      c++;
      typename Scal<T>::type a, ma;
      if constexpr (is_cx<T>::value) {
        a = cdiv(c128{rsq, 0.0}, c128{pap[0], pap[1]});
        ma = {-a.re, -a.im};
      } else {
        a = rsq / pap[0];
        ma = -a;
      }
      double rn[1] = {0.0};
#pragma unroll
      for (int j = 0; j < R; j++) {
        r[j] = rs_axpy(ma, ap[j], r[j]);
        if (t.counts(j)) rs_norm(rn[0], r[j]);
      }
      rn[0] = t.own ? rn[0] : 0.0;
      t.publish(rn, c);
      rh = rs_axpy(ma, aph, rh);
#pragma unroll
      for (int j = 0; j < R; j++) x[j] = rs_axpy(a, p[j], x[j]);
      if (!t.collect(rn, c)) return give_up();
      c++;
      if (lead && so.hist) so.hist[k] = sqrt(rn[0]) / bsqrt;
      if (sqrt(rn[0]) < so.eps * bsqrt || k == kmax) break;
      be = rn[0] / rsq;
      rsq = rn[0];
    }
    // ---- the solution to memory, for the true residual
#pragma unroll
    for (int j = 0; j < R; j++)
      if (t.own && t.counts(j))
        rs_put<T>(reinterpret_cast<unsigned long long*>(xp + (t.yw + j) * t.lx + t.xg), x[j]);
    double none[1] = {0.0};
    t.publish(none, c);  // (waits for the stores of x first)
    if (!t.collect(none, c)) return give_up();
    c++;
  }
  if (lead) {
    so.out->kfinal = k;
    so.out->resSq = resSq;
    so.out->bsqrt = bsqrt;
    so.out->done = 1;
  }
}

template <int R>
struct RsBicgShared {
  static constexpr bool kX = R >= 4;  // x and r0 in LDS
  RsExShared<c128, R, 1> ex;
  RsHopShared<c128, R> op;
  c128 x[kX ? R : 1][kRsThreads], r0[kX ? R : 1][kRsThreads];
};

// generic_bicgstab.cpp:205-341
template <int R, int SB>
__global__ __launch_bounds__(kRsThreads) void k_rs_bicg(RsGeom g, RsSolve so) {
  using T = c128;
  using Sh = RsBicgShared<R>;
  __shared__ Sh sh;
  RsTile<T, R, 1> t(sh.ex, g, so.ring, so.lines, so.spins);
  const RsHop<T, R, SB> A(sh.op, t, so);
  RsRows<T, R, Sh::kX> x(sh.x), r0(sh.r0);
  const T z = zero_of<T>();
  T r[R], p[R], ap[R], as[R], rh = z, ph = z, aph = z, ash = z;  // (s = r - alpha Ap lies in r)
#pragma unroll
  for (int j = 0; j < R; j++) x[j] = t.own ? so.x[(t.yw + j) * t.lx + t.xg] : z;
  if (threadIdx.x == 0) sh.ex.bad = 0;
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  auto give_up = [&]() {
    if (threadIdx.x == 0) so.out->err = 1;
  };
  int k = 0, c = 0, e = 0;
  double bsqrt = 0.0, resSq = 0.0;
  const int kmax = so.max_iter - 1;
  __syncthreads();
  for (bool first = true;; first = false) {
    double s2[2];
    A.residual(t, so, r, s2);
    t.publish(r, e, s2, c);
    if (!t.collect(r, [&](int, T v) { rh = v; }, e, s2, c)) return give_up();
    e++;
    c++;
    if (!first) {
      resSq = s2[0];
      break;
    }
    bsqrt = sqrt(s2[1]);
    c128 rho{s2[0], 0.0};
#pragma unroll
    for (int j = 0; j < R; j++) {
      r0[j] = r[j];
      p[j] = r[j];
    }
    ph = rh;
    for (;; k++) {
      // ---- alpha = rho / <r0, A p>
      A.apply(t, p, ph, 0, ap);
      double d0[2] = {0.0, 0.0};
#pragma unroll
      for (int j = 0; j < R; j++)
        if (t.counts(j)) rs_dot(d0, r0[j], ap[j]);
      d0[0] = t.own ? d0[0] : 0.0;
      d0[1] = t.own ? d0[1] : 0.0;
      t.publish(ap, e, d0, c);
      if (!t.collect(ap, [&](int, T v) { aph = v; }, e, d0, c)) return give_up();
      e++;
      c++;
      const c128 al = cdiv(rho, c128{d0[0], d0[1]});
      // ---- s = r - alpha Ap, omega = <As, s> / <As, As>
      const c128 mal{-al.re, -al.im};
#pragma unroll
      for (int j = 0; j < R; j++) r[j] = rs_axpy(mal, ap[j], r[j]);
      rh = rs_axpy(mal, aph, rh);
      A.apply(t, r, rh, 1, as);
      double d1[2] = {0.0, 0.0}, n1 = 0.0;
#pragma unroll
      for (int j = 0; j < R; j++)
        if (t.counts(j)) {
          rs_dot(d1, as[j], r[j]);
          rs_norm(n1, as[j]);
        }
      double v4[4] = {t.own ? d1[0] : 0.0, t.own ? d1[1] : 0.0, t.own ? n1 : 0.0, 0.0};
      t.publish(as, e, v4, c);
      if (!t.collect(as, [&](int, T v) { ash = v; }, e, v4, c)) return give_up();
      e++;
      c++;
      const c128 om = cdiv(c128{v4[0], v4[1]}, c128{v4[2], 0.0});
      const c128 mom{-om.re, -om.im};
      // ---- x += alpha p + omega s, r = s - omega As
      double d2[2] = {0.0, 0.0}, n2 = 0.0;
#pragma unroll
      for (int j = 0; j < R; j++) {
        x[j] = rs_axpy(om, r[j], rs_axpy(al, p[j], x[j]));
        r[j] = rs_axpy(mom, as[j], r[j]);
        if (t.counts(j)) {
          rs_norm(n2, r[j]);
          rs_dot(d2, r0[j], r[j]);
        }
      }
      double v5[4] = {t.own ? n2 : 0.0, t.own ? d2[0] : 0.0, t.own ? d2[1] : 0.0, 0.0};
      t.publish(v5, c);
      rh = rs_axpy(mom, ash, rh);
      if (!t.collect(v5, c)) return give_up();
      c++;
      const double rn = v5[0];
      if (lead && so.hist) so.hist[k] = sqrt(rn) / bsqrt;
      if (sqrt(rn) < so.eps * bsqrt || k == kmax) break;
      const c128 rho_new{v5[1], v5[2]};
      const c128 be = cdiv(rho_new, rho) * cdiv(al, om);
      rho = rho_new;
      // ---- p = r + beta (p - omega Ap)
#pragma unroll
      for (int j = 0; j < R; j++) p[j] = rs_axpy(be, rs_axpy(mom, ap[j], p[j]), r[j]);
      ph = rs_axpy(be, rs_axpy(mom, aph, ph), rh);
    }
#pragma unroll
    for (int j = 0; j < R; j++)
      if (t.own && t.counts(j))
        rs_put<T>(reinterpret_cast<unsigned long long*>(so.x + (t.yw + j) * t.lx + t.xg), x[j]);
    double none[1] = {0.0};
    t.publish(none, c);
    if (!t.collect(none, c)) return give_up();
    c++;
  }
  if (lead) {
    so.out->kfinal = k;
    so.out->resSq = resSq;
    so.out->bsqrt = bsqrt;
    so.out->done = 1;
  }
}

}  // namespace glx
