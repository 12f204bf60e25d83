// glx_resident.h -- CG on the staggered normal operator with the whole system
// held on the chip: one launch is one solve.
//
// D^dag D = m^2 - K^2 (operators.cpp:444-453; K as in glx_stencil.h), on the
// full lattice or, for m^2 - D_eo D_oe (operators.cpp:566-588), on even-site
// vectors whose odd lanes hold exact zeros.
//
// What bounds it.  A launch per iteration reads and writes every vector from
// the last-level cache each time (80 - 208 B per site and iteration) and pays
// a kernel boundary (4 us) per launch; the vectors and links of a 1024^2 FP32
// system (40 MB) fit the 128 MB of vector registers.  Here they are loaded
// once; per iteration only tile boundaries and a few sums leave a CU.  What
// remains per iteration is one (single-pass forms) or two (reference order)
// chip-wide reductions of about 2 us (256 blocks; 1.4 us at 64), and the two
// hops' arithmetic.
//
// Work split and exchange: glx_restile.h, with H = 2.  p and r are updated in
// halo lanes and rows as the owner updates them, so only the boundary of Ap is
// exchanged, once per iteration; q = K p on the row next to a tile is formed
// on both sides.
//
// Measured (us per iteration: reference order, single-pass FP64, mixed):
// 64^2 4.1, 2.8, 2.9; 256^2 5.1, 3.5, 3.2; 512^2 6.3, 4.8, 4.0; 1024^2 10.5,
// 10.6, 6.2.  A launch per iteration took 17, 12, 14; 18, 12, 10; 21, 13, 10;
// 38, 30, 14.  (Of an iteration at 256^2, 1.3 us is the round trip of the
// reduction, the rest the latencies of the hops, LDS and block sums.)
//
// Every wait is bounded (RsSolve::spins polls): a block that gives up sets the
// error word and leaves; the others run out of polls as well, nothing of the
// result is used, and the host repeats the solve with a launch per iteration.
// The host launches at most one block per CU and never more resident blocks
// at once than the device has CUs (RsReserve), so all blocks of a launch run
// together unless another process holds the chip.
#pragma once

#include "glx_restile.h"

namespace glx {

// LDS of a block: the first and last row of every wave's run of p and of q
// (v), the reductions' staging and, for FP64, what would not fit the registers:
// x (read and written once per iteration) and the edge waves' halo rows (h).
enum RsHaloVal : int { RS_RH = 0, RS_PH = 2, RS_APH = 4, RS_UXH = 6, RS_UYH, RS_UYHM, RS_NHALO };
template <class T, int R>
struct RsShared {
  static constexpr bool kX = sizeof(T) == 16 && R >= 4;
  // the largest FP64 tile keeps four rows of r and U_y above the run here as
  // well, and p and q share one buffer (with a barrier of their own)
  static constexpr int kR = sizeof(T) == 16 && R > 8 ? 4 : 0;
  static constexpr int kV = kR ? 1 : 2;
  T v[kV][kRsWaves][2][64];
  RsExShared<T, R, 2> ex;
  T x[kX ? R : 1][kX ? kRsThreads : 1];
  T r[kR ? kR : 1][kR ? kRsThreads : 1];
  T uyt[kR ? kRsThreads : 1];
  T h[kX ? 2 : 1][RS_NHALO][kX ? 64 : 1];
};

// D^dag D on a tile: its links, and the edge waves' halo values.
template <class T, int R>
struct RsNormal {
  using Re = typename Real<T>::type;
  using Sh = RsShared<T, R>;
  using Tile = RsTile<T, R, 2>;
  static constexpr int NW = kRsWaves;
  Sh& sh;
  const Tile& t;
  Re m2;
  T ux[R], uy[R], uxm[sizeof(T) == 8 ? R : 1];
  T uyt_reg, hreg[Sh::kX ? 1 : RS_NHALO];

  __device__ __forceinline__ T& hal(int v) {  // (edge waves only)
    if constexpr (Sh::kX) return sh.h[t.top ? 0 : 1][v][t.lane];
    else return hreg[v];
  }
  // U_y of the row above the run
  __device__ __forceinline__ T& uyt() {
    if constexpr (Sh::kR != 0) return sh.uyt[threadIdx.x];
    else return uyt_reg;
  }
  __device__ __forceinline__ T uxm_of(int j) const { return uxm[sizeof(T) == 8 ? j : 0]; }

  // loads the links: the run's, U_y above it and, on the edge waves, those of
  // the nearest row beyond the tile with U_y of the row below it
  __device__ __forceinline__ RsNormal(Sh& sh_, const Tile& t_, const RsLinks& lk, double mass)
      : sh(sh_), t(t_), m2(Re(mass * mass)) {
    const Re ey = (t.xg & 1) ? Re(-0.5) : Re(0.5);
    const T b = zero_of<T>();
    uxm[0] = b;
#pragma unroll
    for (int j = 0; j < R; j++) {
      ux[j] = uy[j] = b;
      if (t.valid) rs_links<Re>(lk, (t.yw + j) * t.lx + t.xg, Re(0.5), ey, ux[j], uy[j]);
      if constexpr (sizeof(T) == 8) uxm[j] = rs_shift<kDwPrev>(ux[j]);
    }
    T a, ux0 = b, uy0 = b, uy1 = b, uyw = b;
    if (t.valid) {
      rs_links<Re>(lk, t.wrapy(t.yw - 1) * t.lx + t.xg, Re(0.5), ey, a, uyw);
      if (t.edge) {
        rs_links<Re>(lk, t.yh[0] * t.lx + t.xg, Re(0.5), ey, ux0, uy0);
        rs_links<Re>(lk, t.yh[1] * t.lx + t.xg, Re(0.5), ey, a, uy1);
        if (!t.top) uy1 = uy[R - 1];
      }
    }
    uyt_reg = b;
    uyt() = uyw;
    if (t.edge || !Sh::kX) {
#pragma unroll
      for (int v = 0; v < RS_UXH; v++) hal(v) = b;
      hal(RS_UXH) = ux0;
      hal(RS_UYH) = uy0;
      hal(RS_UYHM) = uy1;
    }
  }

  // ap = D^dag D p (p with its rim lanes, and the halo rows RS_PH of the edge
  // waves): q = K p in ap, then m^2 p - K q in its place; f(j, ap_j) per row
  template <class F>
  __device__ __forceinline__ void apply(const T (&p)[R], T (&ap)[R], F f) {
    const int lane = t.lane, wave = t.wave;
    const bool top = t.top;
    sh.v[0][wave][0][lane] = p[0];
    sh.v[0][wave][1][lane] = p[R - 1];
    __syncthreads();
    T qh = zero_of<T>(), p0 = qh;
    if (t.edge) {
      p0 = hal(RS_PH);
      const T p1 = hal(RS_PH + 1), uh = hal(RS_UXH);
      qh = rs_hop(p0, top ? p1 : p[R - 1], top ? p[0] : p1, uh, rs_shift<kDwPrev>(uh), hal(RS_UYH), hal(RS_UYHM));
    }
    T up = top ? p0 : sh.v[0][top ? 0 : wave - 1][1][lane];
    T below = wave == NW - 1 ? p0 : sh.v[0][wave + 1 < NW ? wave + 1 : wave][0][lane];
    // (the scheduling fences keep the FP64 rows apart: interleaved, their
    // temporaries spill the links)
#pragma unroll
    for (int j = 0; j < R; j++) {
      if constexpr (Sh::kX) __builtin_amdgcn_sched_barrier(0);
      ap[j] = rs_hop(p[j], j ? p[j ? j - 1 : 0] : up, j + 1 < R ? p[j + 1 < R ? j + 1 : j] : below, ux[j], uxm_of(j),
                     uy[j], j ? uy[j ? j - 1 : 0] : uyt());
    }
    if constexpr (Sh::kV == 1) __syncthreads();
    sh.v[Sh::kV - 1][wave][0][lane] = ap[0];
    sh.v[Sh::kV - 1][wave][1][lane] = ap[R - 1];
    __syncthreads();
    up = top ? qh : sh.v[Sh::kV - 1][top ? 0 : wave - 1][1][lane];
    below = wave == NW - 1 ? qh : sh.v[Sh::kV - 1][wave + 1 < NW ? wave + 1 : wave][0][lane];
#pragma unroll
    for (int j = 0; j < R; j++) {
      if constexpr (Sh::kX) __builtin_amdgcn_sched_barrier(0);
      const T q = ap[j];
      ap[j] = rs_mhop(m2, p[j], q, up, j + 1 < R ? ap[j + 1 < R ? j + 1 : j] : below, ux[j], uxm_of(j), uy[j],
                      j ? uy[j ? j - 1 : 0] : uyt());
      up = q;
      f(j, ap[j]);
    }
  }
};

// out = b - (D^dag D + sigma) x in FP64 from memory (own lanes), with |out|^2
// and |b|^2 of the counted rows in s2: a march down the wave's rows, at step i
// the loads of row i - 2 of the run, q = K x on the row before it, A x on the
// one before that.  at(y): the vectors' index of the lane's column in row y,
// or -1 where a compact vector has none.
template <class T, int R, class At>
__device__ __forceinline__ void rs_normal_residual(const RsTile<T, R, 2>& t, const c128* u64, double mass, double sigma,
                                                   const c128* x, const c128* b, At at, T (&out)[R],
                                                   double (&s2)[2]) {
  const double m2d = mass * mass + sigma;
  const double ed = (t.xg & 1) ? -0.5 : 0.5;
  const c128 z{0.0, 0.0};
  c128 xa = z, xb = z, qa = z, qb = z, u1x = z, u1y = z, u2x = z, u2y = z, u3y = z;
  s2[0] = s2[1] = 0.0;
#pragma unroll 1
  for (int i4 = 0; i4 < R + 4; i4++) {
    const int y = t.wrapy(t.yw - 2 + i4), i = at(y);
    c128 xc = z, ucx = z, ucy = z;
    if (t.valid) {
      if (i >= 0) xc = rs_read<c128>(reinterpret_cast<const unsigned long long*>(x + i));
      rs_links<double>(RsLinks{u64, nullptr, 0}, y * t.lx + t.xg, 0.5, ed, ucx, ucy);
    }
    const c128 qc = rs_hop(xb, xa, xc, u1x, z, u1y, u2y);
    if (i4 >= 4) {
      const c128 ax = rs_mhop(m2d, xa, qb, qa, qc, u2x, z, u2y, u3y);
      const int j = i4 - 4, ib = at(t.yw + j);
      c128 d = z;
      if (t.own && ib >= 0) {
        const c128 bv = b[ib];
        d = bv - ax;
        if (t.counts(j)) {
          s2[0] += norm2(d);
          s2[1] += norm2(bv);
        }
      }
      T dr;
      cvt(dr, d);
#pragma unroll
      for (int jj = 0; jj < R; jj++)
        if (jj == j) out[jj] = dr;
    }
    qa = qb;
    qb = qc;
    xa = xb;
    xb = xc;
    u3y = u2y;
    u2x = u1x;
    u2y = u1y;
    u1x = ucx;
    u1y = ucy;
  }
}

template <class T, int R, int M>
__global__ __launch_bounds__(kRsThreads) void k_rs_cg(RsGeom g, RsSolve so) {
  using Re = typename Real<T>::type;
  using A = typename std::conditional<M == RS_REF, T, Re>::type;  // alpha: complex in the reference's order
  using Sh = RsShared<T, R>;
  __shared__ Sh sh;

  RsTile<T, R, 2> t(sh.ex, g, so.ring, so.lines, so.spins);
  const int lx = t.lx, yw = t.yw, xg = t.xg;
  const bool edge = t.edge, own = t.own;
  // a vector's entry at (xg, y), or -1 where a compact vector has none
  // (the column passes through an empty asm statement, as in RsTile::slot)
  auto at = [&](int y) -> int {
    int x = xg;
    asm volatile("" : "+v"(x));
    if (!so.eo) return y * lx + x;
    return ((x + y) & 1) ? -1 : y * (lx >> 1) + (x >> 1);
  };
  RsNormal<T, R> op(sh, t, so.lk, so.mass);
  T rv_[R - Sh::kR], p[R], ap[R], xr[Sh::kX ? 1 : R];
  auto xref = [&](int j) -> T& {
    if constexpr (Sh::kX) return sh.x[j][threadIdx.x];
    else return xr[j];
  };
  auto rref = [&](int j) -> T& {
    if constexpr (Sh::kR != 0) {
      if (j >= R - Sh::kR) return sh.r[j - (R - Sh::kR)][threadIdx.x];
    }
    return rv_[j < R - Sh::kR ? j : 0];
  };
  auto hal = [&](int v) -> T& { return op.hal(v); };
#pragma unroll
  for (int j = 0; j < R; j++) {
    rref(j) = p[j] = ap[j] = zero_of<T>();
    T x = zero_of<T>();
    if constexpr (M != RS_MIXED) {
      const int i = at(yw + j);
      if (own && i >= 0) x = so.x[i];
    }
    xref(j) = x;
  }
  if (threadIdx.x == 0) sh.ex.bad = 0;

  auto give_up = [&]() {
    if (threadIdx.x == 0) so.out->err = 1;
  };
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;

  int k = 0, c = 0, e = 0;  // iteration, reductions and ring uses so far
  int reliable = 0;
  A a;
  if constexpr (M == RS_REF) a = zero_of<T>();
  else a = Re(0);
  double al = 0.0;  // (single-pass) alpha in FP64
  Re be = Re(0);
  double rsq = 0.0, maxrr = 0.0, bsqrt = 0.0, resSq = 0.0;
  const int kmax = so.max_iter - 1;
  bool first = true;
  __syncthreads();
  for (;;) {
    {
      double s2[2];
      rs_normal_residual<T, R>(t, so.u64, so.mass, 0.0, so.x, so.b, at, ap, s2);
      t.publish(ap, e, s2, c);
      if (!t.collect(ap, [&](int h, T v) { hal(RS_RH + h) = v; }, e, s2, c)) return give_up();
      e++;
      c++;
      if (first) {
        first = false;
        bsqrt = sqrt(s2[1]);
        rsq = maxrr = s2[0];
      } else {
        resSq = s2[0];
        if constexpr (M != RS_MIXED) break;
        reliable++;
        if (resSq == 0.0 || sqrt(resSq) < so.eps * bsqrt || k >= kmax) break;
        // restart the recurrence from it: p = r + beta p with this beta
        be = Re(resSq / rsq);
        a = A{};
        maxrr = resSq;
        k++;
      }
#pragma unroll
      for (int j = 0; j < R; j++) {
        rref(j) = ap[j];
        ap[j] = zero_of<T>();
      }
      if (edge) hal(RS_APH) = hal(RS_APH + 1) = zero_of<T>();
    }

    for (;;) {
    // ---- the vectors' updates, halo copies included
#pragma unroll
    for (int j = 0; j < R; j++) {
      if constexpr (M != RS_REF) {
        xref(j) = rs_axpy(a, p[j], xref(j));
        rref(j) = rs_axpy(-a, ap[j], rref(j));
      }
      p[j] = rs_axpy(be, p[j], rref(j));
    }
    if (edge) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        T rh = hal(RS_RH + h);
        if constexpr (M != RS_REF) hal(RS_RH + h) = rh = rs_axpy(-a, hal(RS_APH + h), rh);
        hal(RS_PH + h) = rs_axpy(be, hal(RS_PH + h), rh);
      }
    }
    constexpr int N1 = M == RS_REF ? 2 : 4;
    double v1[N1];
#pragma unroll
    for (int i = 0; i < N1; i++) v1[i] = 0.0;
    op.apply(p, ap, [&](int j, T v) {
      if (t.counts(j)) {
        const double pr = p[j].re, pi = p[j].im, ar = v.re, ai = v.im;
        v1[0] = __builtin_fma(pr, ar, __builtin_fma(pi, ai, v1[0]));
        if constexpr (M == RS_REF) {
          v1[1] = __builtin_fma(pr, ai, __builtin_fma(-pi, ar, v1[1]));
        } else {
          const T rv = rref(j);
          const double rr = rv.re, ri = rv.im;
          v1[1] = __builtin_fma(ar, ar, __builtin_fma(ai, ai, v1[1]));
          v1[2] = __builtin_fma(ar, rr, __builtin_fma(ai, ri, v1[2]));
          v1[3] = __builtin_fma(rr, rr, __builtin_fma(ri, ri, v1[3]));
        }
      }
    });
#pragma unroll
    for (int i = 0; i < N1; i++) v1[i] = own ? v1[i] : 0.0;
    t.publish(ap, e, v1, c);
    if (!t.collect(ap, [&](int h, T v) { hal(RS_APH + h) = v; }, e, v1, c)) return give_up();
    e++;
    c++;

    // ---- the CG step
    bool stop;
    if constexpr (M == RS_REF) {
      const c128 al = cdiv(c128{rsq, 0.0}, c128{v1[0], v1[1]});
      cvt(a, al);
      const T ma{-a.re, -a.im};
      double v2[1] = {0.0};
#pragma unroll
      for (int j = 0; j < R; j++) {
        const T rv = rs_axpy(ma, ap[j], rref(j));
        rref(j) = rv;
        if (t.counts(j)) v2[0] = __builtin_fma(rv.re, rv.re, __builtin_fma(rv.im, rv.im, v2[0]));
      }
      v2[0] = own ? v2[0] : 0.0;
      t.publish(v2, c);
      if (edge) {
#pragma unroll
        for (int h = 0; h < 2; h++) hal(RS_RH + h) = rs_axpy(ma, hal(RS_APH + h), hal(RS_RH + h));
      }
#pragma unroll
      for (int j = 0; j < R; j++) xref(j) = rs_axpy(a, p[j], xref(j));
      if (!t.collect(v2, c)) return give_up();
      c++;
      const double rn = v2[0];
      if (lead && so.hist) so.hist[k] = sqrt(rn) / bsqrt;
      stop = sqrt(rn) < so.eps * bsqrt || k == kmax;
      be = Re(rn / rsq);
      rsq = rn;
    } else {
      // <p, Ap>, |Ap|^2, <Ap, r>, |r|^2: real parts.  A is Hermitian for any
      // stored links (K is anti-Hermitian in them), so the exact <p, Ap> and
      // alpha are real, and imaginary parts of the sums are rounding alone:
      // the real quotient's error against extended precision is no larger than
      // that of rr / complex <p, Ap> (FP32 p: 1.4e-9 and 1.8e-9 at 64^2, 5.5e-11
      // and 2.5e-10 at 512^2; FP64 equal).  alpha lies in scalar registers: in
      // vector ones it spilled at ten rows.
      // (a zero residual ends the solve: no step)
      rsq = v1[3];
      al = rsq == 0.0 ? 0.0 : readlane_d(rsq / v1[0], 0);
      double rn = rsq - 2.0 * al * v1[2] + al * al * v1[1];
      if (!(rn > 0.0)) rn = 0.0;
      if (rn > maxrr) maxrr = rn;
      const double tol = so.eps * bsqrt;
      stop = rn < tol * tol || k == kmax || rsq == 0.0;
      if (M == RS_MIXED && rn < (so.delta * so.delta) * maxrr) stop = true;
      if (lead && so.hist) so.hist[k] = sqrt(rn) / bsqrt;
      a = Re(al);
      be = Re(rn / rsq);
    }
    if (stop) break;
    k++;
    }

    // ---- the solution to memory, for the true residual: the last step and, in
    // mixed precision, the sum with the FP64 solution in FP64
#pragma unroll
    for (int j = 0; j < R; j++) {
      if constexpr (M == RS_ONE) xref(j) = rs_axpy(a, p[j], xref(j));
      int y = yw;
      asm volatile("" : "+s"(y));
      const int i = at(y + j);
      if (own && i >= 0 && t.counts(j)) {
        unsigned long long* q = reinterpret_cast<unsigned long long*>(so.x + i);
        c128 v;
        cvt(v, xref(j));
        if constexpr (M == RS_MIXED) {
          c128 pj;
          cvt(pj, p[j]);
          v = rs_read<c128>(q) + rs_axpy(al, pj, v);
        }
        rs_put<c128>(q, v);
      }
      if constexpr (M == RS_MIXED) xref(j) = zero_of<T>();
    }
    double none[1] = {0.0};
    t.publish(none, c);  // (waits for the stores of x first)
    if (!t.collect(none, c)) return give_up();
    c++;
  }
  if (lead) {
    so.out->kfinal = k;
    so.out->reliable = reliable;
    so.out->resSq = resSq;
    so.out->bsqrt = bsqrt;
    so.out->done = 1;
  }
}

// ------------------------------------------------------------- host side --
// Settings (process-wide, like the other launch shapes): whether solves may
// run resident, and the polls a wait may take before it gives up.
void set_resident(int on, int spins);
bool resident_on();
int rs_cus();  // CUs of the current device
int resident_spins();
// Solves that ran resident and solves whose resident launch gave up, of the
// process so far.
struct RsCounts {
  long long ran, gave_up;
};
RsCounts resident_counts();
void rs_count(bool gave_up);

// The tiling a system would run resident with on the current device, for an
// operator that reaches `halo` sites and kernels of at most most_rows rows per
// wave; false where it does not fit.
bool rs_plan(int lx, int ly, int halo, int most_rows, RsGeom& g);
constexpr int kRsMostRows = 10;

// Words of the exchange buffers (lines, then ring) of a solve with `words`
// 64-bit words per element.
inline long rs_exchange_words(const RsGeom& g, int words, int halo) {
  const long columns = long(g.nsx) * g.nsy * kRsWaves * g.rows * 2 * halo;
  return long(kRsBufs) * (kRsMaxBlocks * kRsLine + (long(g.lx) * g.ly + columns) * words);
}
// Empties the exchange buffers and clears the result record.
void rs_fill(hipStream_t st, const RsSolve& so, long words);
// Fills, then launches CG on D^dag D or the even/odd Schur operator.
void rs_launch(hipStream_t st, const RsGeom& g, RsMode mode, const RsSolve& so);
// The same for the one-hop operators (glx_reshop.hip): CG on real or complex
// vectors with backward sign sb = 1, BiCGStab on complex vectors with either.
constexpr int kRsMostRowsHop = 8, kRsMostRowsBicg = 6;
void rs_launch_hop_cg(hipStream_t st, const RsGeom& g, bool cplx, const RsSolve& so);
void rs_launch_hop_bicgstab(hipStream_t st, const RsGeom& g, int sb, const RsSolve& so);

// Multishift CG (glx_rescgm.h), its kernel one row per wave.
constexpr int kRsShifts = 16;  // shifts a resident solve may have
struct RsShiftSet {
  int n, freq;  // shifts, iterations between convergence checks
  double shift[kRsShifts];
  c128* x[kRsShifts];
  double* res;  // [n] |(A + shift) x - b|^2
};
bool rs_plan_one_row(int lx, int ly, int halo, RsGeom& g);
void rs_launch_cg_m(hipStream_t st, const RsGeom& g, const RsSolve& so, const RsShiftSet& sh);

// The resident blocks of every solve in flight on a device, over all host
// threads, stay within its CUs and each XCD's, one block each (glx_slots.h): a
// solve waits here until its turn has come and its blocks fit.  Held from before the launch until the stream has drained.
class RsReserve {
 public:
  explicit RsReserve(int blocks);
  ~RsReserve();
  RsReserve(const RsReserve&) = delete;
  RsReserve& operator=(const RsReserve&) = delete;

 private:
  int dev_, slots_;
};

}  // namespace glx
