// glx_resgcr.hip -- launch shapes of GCR on the chip (glx_resgcr.h).
#include "glx_resgcr.h"

#include <algorithm>

#include "glx_resident.h"

namespace glx {

bool rg_plan(const CsDev& st, RsGcr& g, int& m) {
  // all terms of a stencil with or without the two-link ones
  const bool two = st.terms == (1u << kCsTerms) - 1;
  if (!resident_on() || !st.coef || st.piece != CS_ALL || (!two && st.terms != 0x1Fu)) return false;
  const long v = long(st.lx) * st.ly;
  if (v < 1 || v * st.nc > (1L << 24)) return false;
  const int most = std::min(kRsMaxBlocks, rs_cus());
  for (m = 1; m <= 4; m *= 2) {
    const int s = 64 * m / st.nc;
    if (s < 1 || (v + s - 1) / s > most) continue;
    g.st = st;
    g.sites = s;
    g.nblk = int((v + s - 1) / s);
    g.nt = two ? kCsTerms : 5;
    return true;
  }
  return false;
}

long rg_exchange_words(const RsGcr& g) {
  const long n = long(g.st.lx) * g.st.ly * g.st.nc;
  return kRsBufs * (long(kRsMaxBlocks) * kRsLine + 2 * n + (g.nblk + 1L) * rg_words(g.k0));
}

namespace {
template <int M>
void launch(hipStream_t st, RsGcr& g) {
  constexpr int kLds = 160 * 1024 - 1024;  // (a kilobyte for the kernel's static part)
  int lds = int(sizeof(c128)) * (g.nt * g.sites * rg_pitch(g.st.nc) + (kRsWaves + 1) * 64 * M + rg_words(g.k0) / 2);
  constexpr int one = int(sizeof(c128)) * 64 * M;
  g.held = std::max(0, std::min(kRgDirs, (kLds - lds) / one));
  lds += g.held * one;
  // (the most it may ever be, the same for every solve: the attribute is the
  // function's, and solves of other threads set it too)
  GLX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_rs_gcr<M>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              kLds));
  hipLaunchKernelGGL(k_rs_gcr<M>, dim3(g.nblk), dim3(kRsThreads), lds, st, g);
  GLX_CHECK_LAUNCH();
}
}  // namespace

void rg_launch(hipStream_t st, int m, RsGcr g) {
  RsSolve ex{};
  ex.lines = g.lines;
  ex.out = g.out;
  rs_fill(st, ex, rg_exchange_words(g));
  if (m == 1) launch<1>(st, g);
  else if (m == 2) launch<2>(st, g);
  else launch<4>(st, g);
}

}  // namespace glx
