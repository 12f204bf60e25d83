// glx_state.h -- the scalar state a solve keeps on the device, shared by the
// solver kernels and the resident-system kernels.
#pragma once

#include "glx_common.h"

namespace glx {

constexpr int kMaxShift = 64;

struct SolveState {
  // control word (first 16 bytes, mirrored to the host)
  int k, done, kfinal, n_rem;
  int max_iter, resid_freq, worst_first, n_shift;
  double eps, bsqrt, rsq, rsqNew;
  double beta_r, resSq, maxrr, delta;  // maxrr: single-pass CG: max of |r|^2 since the last reliable update
  int reliable, pending, ko;  // pending: self-finalising single-pass CG; ko: s-step CG launches
  int n_xupd;  // multishift: shifts active before this iteration's check (their x still takes its update)
  c128 alpha, alpha_prev, beta, beta_prev, rho, omega, pap;
  double* hist;
  double* resvec;
  // host-mapped copy of `done` (single-pass CG): the kernels that change
  // `done` also store it here, so the host polls it without a copy command
  int* hdone;
  // multishift
  c128 zeta[kMaxShift], zeta_p[kMaxShift], alpha_s[kMaxShift], beta_s[kMaxShift];
  double shifts[kMaxShift];
  int mapping[kMaxShift];
  int vec[kMaxShift];
  // multishift: sums over the iterations of the shifts whose x_s (n_xupd)
  // and p_s (n_rem after the check) were updated -- the pass's algorithmic
  // bytes are 16 (3 upd_x + upd_p) per site
  long long upd_x, upd_p;
};

struct Mirror {
  int k, done, kfinal, n_rem;
};

template <class T>
__device__ __forceinline__ typename Scal<T>::type as_scal(c128 a) {
  if constexpr (is_cx<T>::value) return a;
  else return a.re;
}

}  // namespace glx
