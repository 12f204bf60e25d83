// glx_rgwalk.h -- how a wave of the resident GCR kernel (glx_resgcr.h) walks
// the staged neighbour values: plain arithmetic, so that it can be checked on
// the host.
//
// Staged values lie [term][site][pitch]; pitch = nc | 1, so where nc is even
// every site ends in a pad that nothing writes.  Wave w contracts the (term,
// column) pairs f = w wf ... of all terms, the first rg_kept of them in groups
// of four without a branch.  Steps beyond the last pair meet zero
// coefficients, and what they read has to be a written column all the same:
// 0 times whatever an unwritten word holds may be a NaN.
#pragma once

namespace glx {

constexpr int kRgWaves = 8;  // waves of a block

constexpr int rg_pitch(int nc) { return nc | 1; }  // colours of a staged site, an odd count for the banks
constexpr int rg_kept(int m) { return m == 1 ? 24 : (m == 2 ? 8 : 4); }  // coefficients kept per entry
// pairs per wave, and the wave's first (the last pair where it has none) and end
constexpr int rg_share(int nf) { return (nf + kRgWaves - 1) / kRgWaves; }
constexpr int rg_first(int nf, int wave) { return wave * rg_share(nf) < nf - 1 ? wave * rg_share(nf) : nf - 1; }
constexpr int rg_end(int nf, int wave) { return (wave + 1) * rg_share(nf) < nf ? (wave + 1) * rg_share(nf) : nf; }

struct RgWalk {
  int nc, tspan, last;
  int c, at;  // the pair's column, and its place for the block's first site
  constexpr RgWalk(int nt, int nc_, int sites, int f0)
      : nc(nc_), tspan(sites * rg_pitch(nc_)), last((nt - 1) * tspan + nc_ - 1), c(f0 % nc_),
        at(f0 / nc_ * tspan + f0 % nc_) {}
  constexpr void step() {
    c++;
    at++;
    if (c == nc) {
      at += tspan - nc;
      c = 0;
    }
    if (at > last) at = last;
  }
};

}  // namespace glx
