// glx_resident.hip -- the resident-system kernels' instances, launch shapes
// and host-side bookkeeping (glx_resident.h).
#include "glx_resident.h"
#include "glx_slots.h"

#include <algorithm>
#include <atomic>

namespace glx {

namespace {
std::atomic<int> g_on{1};
// a poll takes about a microsecond: a second in all before a wait gives up
constexpr int kSpins = 1 << 20;
std::atomic<int> g_spins{kSpins};
std::atomic<long long> g_ran{0}, g_gave_up{0};

constexpr int kMaxDevices = 64;
int current_device() {
  int d = 0;
  GLX_HIP(hipGetDevice(&d));
  if (d < 0 || d >= kMaxDevices) throw ArgError("device index beyond the resident-solve table");
  return d;
}
int device_cus(int dev) {
  static std::atomic<int> cus[kMaxDevices];
  int n = cus[dev].load();
  if (n == 0) {
    GLX_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    cus[dev].store(n);
  }
  return n;
}

FairSlots& slots(int dev) {
  static FairSlots* s = new FairSlots[kMaxDevices];  // outlives every static user
  return s[dev];
}

__global__ __launch_bounds__(kBlock) void k_rs_fill(unsigned long long* q, long n, RsOut* out) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *out = RsOut{0, 0, 0, 0, 0.0, 0.0};
  for (long i = long(blockIdx.x) * kBlock + threadIdx.x; i < n; i += long(gridDim.x) * kBlock) q[i] = kRsEmpty;
}

}  // namespace

void rs_fill(hipStream_t st, const RsSolve& so, long words) {
  hipLaunchKernelGGL(k_rs_fill, dim3(unsigned(std::min<long>((words + kBlock - 1) / kBlock, 2048))), dim3(kBlock), 0,
                     st, so.lines, words, so.out);
  GLX_CHECK_LAUNCH();
}

namespace {
// rows per wave the kernels are instantiated for
constexpr int kRows[] = {1, 2, 3, 4, 6, 8, 10};

template <class T, int M>
void launch(hipStream_t st, const RsGeom& g, const RsSolve& so) {
  rs_fill(st, so, rs_exchange_words(g, rs_words<T>(), 2));
  const dim3 grid(g.nsx * g.nsy), block(kRsThreads);
#define GLX_RS(R)                                                                              \
  case R:                                                                                      \
    hipLaunchKernelGGL((k_rs_cg<T, R, M>), grid, block, 0, st, g, so);             \
    break;
  switch (g.rows) {
    GLX_RS(1)
    GLX_RS(2)
    GLX_RS(3)
    GLX_RS(4)
    GLX_RS(6)
    GLX_RS(8)
    GLX_RS(10)
    default:
      throw ArgError("no resident kernel for this tiling");
  }
#undef GLX_RS
  GLX_CHECK_LAUNCH();
}
}  // namespace

void set_resident(int on, int spins) {
  g_on.store(on ? 1 : 0);
  g_spins.store(spins > 0 ? spins : kSpins);
}
int rs_cus() { return device_cus(current_device()); }
bool resident_on() { return g_on.load() != 0; }
int resident_spins() { return g_spins.load(); }
RsCounts resident_counts() { return {g_ran.load(), g_gave_up.load()}; }
void rs_count(bool gave_up) { (gave_up ? g_gave_up : g_ran)++; }

bool rs_plan(int lx, int ly, int halo, int most_rows, RsGeom& g) {
  if (lx < 2 * halo || long(lx) * ly > (1L << 24)) return false;
  const int cap = std::min(kRsMaxBlocks, device_cus(current_device()));
  const int nsx = (lx + rs_cols(halo) - 1) / rs_cols(halo);
  for (int r : kRows) {
    if (r > most_rows) break;
    if (ly < kRsWaves * r) break;  // a tile has this many rows
    const int nsy = (ly + kRsWaves * r - 1) / (kRsWaves * r);
    // few rows per wave only while that takes few blocks: the reductions
    // grow with the blocks, the hops with the rows (us per iteration in the
    // reference's order and mixed: 128^2 5.2 and 3.7 at 1 or 2 rows, 5.4 and
    // 4.0 at 4; 256^2 6.2 and 4.1 at 1 row and 160 blocks, 5.9 and 3.9 at 2
    // and 80, 5.9 and 4.4 at 4 and 40; 512^2 7.5 and 4.9 at 3 rows and 198
    // blocks, 7.0 and 4.7 at 4 and 144, 7.4 and 5.2 at 6 and 99; 700^2 8.0 and
    // 5.6 at 6 rows and 180 blocks, 8.6 and 5.8 at 8 and 132)
    const int few = r == 1 ? 64 : (r == 2 ? 128 : (r == 3 ? 160 : kRsMaxBlocks));
    const int most = std::min(cap, few);
    if (long(nsx) * nsy <= most) {
      g = RsGeom{lx, ly, nsx, nsy, r};
      return true;
    }
  }
  return false;
}

bool rs_plan_one_row(int lx, int ly, int halo, RsGeom& g) {
  if (lx < 2 * halo || ly < kRsWaves || long(lx) * ly > (1L << 24)) return false;
  const int nsx = (lx + rs_cols(halo) - 1) / rs_cols(halo), nsy = (ly + kRsWaves - 1) / kRsWaves;
  if (long(nsx) * nsy > std::min(kRsMaxBlocks, device_cus(current_device()))) return false;
  g = RsGeom{lx, ly, nsx, nsy, 1};
  return true;
}

void rs_launch(hipStream_t st, const RsGeom& g, RsMode mode, const RsSolve& so) {
  if (mode == RS_REF) launch<c128, RS_REF>(st, g, so);
  else if (mode == RS_ONE) launch<c128, RS_ONE>(st, g, so);
  else launch<c64, RS_MIXED>(st, g, so);
}

RsReserve::RsReserve(int blocks) : dev_(current_device()), slots_(resident_slots(blocks)) {
  slots(dev_).acquire(slots_, device_cus(dev_));
}
RsReserve::~RsReserve() { slots(dev_).release(slots_); }

}  // namespace glx
