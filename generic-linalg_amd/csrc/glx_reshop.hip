// glx_reshop.hip -- the instances of the one-hop resident kernels
// (glx_reshop.h) and of the multishift one (glx_rescgm.h).
#include "glx_reshop.h"
#include "glx_rescgm.h"

namespace glx {

namespace {
template <class T>
void hop_cg(hipStream_t st, const RsGeom& g, const RsSolve& so) {
  const dim3 grid(g.nsx * g.nsy), block(kRsThreads);
#define GLX_RS(R)                                                            \
  case R:                                                                    \
    hipLaunchKernelGGL((k_rs_hcg<T, R, 1>), grid, block, 0, st, g, so);      \
    break;
  switch (g.rows) {
    GLX_RS(1)
    GLX_RS(2)
    GLX_RS(3)
    GLX_RS(4)
    GLX_RS(6)
    GLX_RS(8)
    default:
      throw ArgError("no resident kernel for this tiling");
  }
#undef GLX_RS
  GLX_CHECK_LAUNCH();
}
template <int SB>
void hop_bicgstab(hipStream_t st, const RsGeom& g, const RsSolve& so) {
  const dim3 grid(g.nsx * g.nsy), block(kRsThreads);
#define GLX_RS(R)                                                            \
  case R:                                                                    \
    hipLaunchKernelGGL((k_rs_bicg<R, SB>), grid, block, 0, st, g, so);       \
    break;
  switch (g.rows) {
    GLX_RS(1)
    GLX_RS(2)
    GLX_RS(3)
    GLX_RS(4)
    GLX_RS(6)
    default:
      throw ArgError("no resident kernel for this tiling");
  }
#undef GLX_RS
  GLX_CHECK_LAUNCH();
}
}  // namespace

void rs_launch_cg_m(hipStream_t st, const RsGeom& g, const RsSolve& so, const RsShiftSet& sh) {
  rs_fill(st, so, rs_exchange_words(g, 2, 2));
  hipLaunchKernelGGL(k_rs_cgm, dim3(g.nsx * g.nsy), dim3(kRsThreads), 0, st, g, so, sh);
  GLX_CHECK_LAUNCH();
}
void rs_launch_hop_cg(hipStream_t st, const RsGeom& g, bool cplx, const RsSolve& so) {
  rs_fill(st, so, rs_exchange_words(g, cplx ? 2 : 1, 1));
  if (cplx) hop_cg<c128>(st, g, so);
  else hop_cg<double>(st, g, so);
}
void rs_launch_hop_bicgstab(hipStream_t st, const RsGeom& g, int sb, const RsSolve& so) {
  rs_fill(st, so, rs_exchange_words(g, 2, 1));
  if (sb > 0) hop_bicgstab<1>(st, g, so);
  else hop_bicgstab<-1>(st, g, so);
}

}  // namespace glx
