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
// Work split.  Block b owns a tile: one of nsx strips of at most 60 columns
// by one of nsy bands of 8 R rows.  A wave holds R whole rows of its tile in
// registers: lane l <-> column x0 - 2 + l, so lanes 0, 1 and w + 2, w + 3 are
// the neighbours' columns and x-neighbours come by DPP wave shifts;
// y-neighbours are other registers of the lane, or pass through LDS between
// the waves of a block.  The first and last wave also keep the two rows
// beyond the tile.  p and r in those halo lanes and rows are updated like the
// owner's (the same instructions on the same values), so only the ring of Ap
// values has to be exchanged, once per iteration.
//
// Exchange between blocks.  Values are their own flags: a slot holds kRsEmpty
// (a signalling NaN, which arithmetic never returns) until its 64-bit word
// arrives, and the reader polls until every word it needs differs from it.
// All accesses are relaxed agent-scope atomics, so no fence and no store
// acknowledgement lies on the path.  Slots rotate through four buffers: after
// publishing use u the writer empties its slots of use u + 2 (a reduction
// since has shown that every block read their contents, those of use u - 2),
// and waits for those stores before it contributes to the next reduction,
// without which no block polls them.
//
// Reductions: each block stores its sums (FP64) to one 64-byte line; every
// block reads all lines and adds them in the same fixed order, so all blocks
// take the same decisions with the same bits.  A 64-byte line per block
// measured 1.9 us for 256 blocks and one sum, 2.2 us for four sums; eight
// blocks per line 2.9 and 7.8 us.
//
// Ring slots: boundary rows lie by lattice site (whole rows, coalesced);
// boundary columns by block and row, four values side by side, so that a wave
// stores them in whole lines.  With the columns by lattice site as well (two
// 16-byte pieces per row) 1024^2 took 6.97 us per iteration in mixed
// precision and 13.2 us in FP64, against 6.1 and 10.6 us.
//
// Measured (us per iteration: reference order, single-pass FP64, mixed):
// 64^2 4.3, 2.9, 3.2; 256^2 5.3, 3.6, 3.6; 512^2 6.8, 4.6, 4.4; 1024^2 10.6,
// 10.4, 6.1.  A launch per iteration took 17, 12, 14; 18, 12, 10; 21, 13, 10;
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

#include "glx_dwave.h"
#include "glx_sswave.h"
#include "glx_state.h"

namespace glx {

constexpr int kRsWaves = 8;        // waves per block, two per SIMD
constexpr int kRsThreads = 64 * kRsWaves;
constexpr int kRsMaxBlocks = 256;  // blocks (tiles) of a launch
constexpr int kRsLine = 8;         // 64-bit words of a block's reduction line
constexpr int kRsBufs = 4;         // uses the exchange slots rotate through
constexpr int kRsHalo = 2;
constexpr int kRsCols = 64 - 2 * kRsHalo;  // columns a strip may own
constexpr unsigned long long kRsEmpty = 0xFFF4B1D5FFB4B1D5ull;

struct RsGeom {
  int lx, ly;
  int nsx, nsy;  // strips, bands: the grid is nsx * nsy blocks
  int rows;      // R of the kernel that takes it
};

// Links as stored: FP64, FP32, or FP16 with the per-site scale.
struct RsLinks {
  const void* u;
  const float* sc;
  int prec;
};

struct RsOut {
  int err;   // a wait ran out
  int done;  // the solve ended
  int kfinal, reliable;
  double resSq, bsqrt;
};

struct RsSolve {
  c128* x;         // guess in, solution out
  const c128* b;
  const c128* u64; // FP64 links (true residuals)
  RsLinks lk;      // the iteration's links
  double mass, eps, delta;
  int max_iter;
  int eo;          // compact even-site vectors
  int spins;       // polls per wait
  double* hist;    // iterated relative residual per iteration, or null
  unsigned long long* ring;   // [kRsBufs][lx * ly] rows by lattice site, then [kRsBufs][blocks][8 R][4] columns, of T
  unsigned long long* lines;  // [kRsBufs][kRsMaxBlocks][kRsLine]
  RsOut* out;
};

enum RsMode : int {
  RS_REF = 0,    // the reference's order: alpha from <p, Ap>, then |r|^2 by a second reduction
  RS_ONE = 1,    // single-pass: |r_{k+1}|^2 from the recurrence, one reduction
  RS_MIXED = 2,  // single-pass in FP32 with reliable updates in FP64
};

__device__ __forceinline__ unsigned long long rs_load(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void rs_store(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// every store this wave issued has reached memory
__device__ __forceinline__ void rs_stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <class T>
constexpr int rs_words() { return int(sizeof(T) / 8); }
template <class T>
__device__ __forceinline__ void rs_put(unsigned long long* slot, T v) {
  unsigned long long w[rs_words<T>()];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int i = 0; i < rs_words<T>(); i++) rs_store(slot + i, w[i]);
}
template <class T>
__device__ __forceinline__ void rs_empty(unsigned long long* slot) {
#pragma unroll
  for (int i = 0; i < rs_words<T>(); i++) rs_store(slot + i, kRsEmpty);
}
template <class T>
__device__ __forceinline__ T rs_read(const unsigned long long* slot) {
  unsigned long long w[rs_words<T>()];
#pragma unroll
  for (int i = 0; i < rs_words<T>(); i++) w[i] = rs_load(slot + i);
  T v;
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}
template <class T>
__device__ __forceinline__ bool rs_there(const T& v) {
  unsigned long long w[rs_words<T>()];
  __builtin_memcpy(w, &v, sizeof(T));
  bool ok = true;
#pragma unroll
  for (int i = 0; i < rs_words<T>(); i++) ok &= w[i] != kRsEmpty;
  return ok;
}

// Site algebra in explicit fused multiply-adds, so that an owner and a
// neighbour's copy of a value round alike whatever code surrounds them.
__device__ __forceinline__ double rs_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float rs_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// acc + a b, acc - conj(a) b
template <class R>
__device__ __forceinline__ cx<R> rs_madd(cx<R> acc, cx<R> a, cx<R> b) {
  return {rs_fma(a.re, b.re, rs_fma(-a.im, b.im, acc.re)), rs_fma(a.re, b.im, rs_fma(a.im, b.re, acc.im))};
}
template <class R>
__device__ __forceinline__ cx<R> rs_msubc(cx<R> acc, cx<R> a, cx<R> b) {
  return {rs_fma(-a.re, b.re, rs_fma(-a.im, b.im, acc.re)), rs_fma(-a.re, b.im, rs_fma(a.im, b.re, acc.im))};
}
// acc + s b for a real or complex scalar s
template <class R>
__device__ __forceinline__ cx<R> rs_axpy(R s, cx<R> b, cx<R> acc) {
  return {rs_fma(s, b.re, acc.re), rs_fma(s, b.im, acc.im)};
}
template <class R>
__device__ __forceinline__ cx<R> rs_axpy(cx<R> s, cx<R> b, cx<R> acc) {
  return rs_madd(acc, s, b);
}
// the value lane l + 1 (CTRL kDwNext) or l - 1 (kDwPrev) holds; the end lanes read 0
template <int CTRL, class V>
__device__ __forceinline__ V rs_shift(V v) {
  constexpr int N = int(sizeof(V) / 4);
  int w[N];
  __builtin_memcpy(w, &v, sizeof(V));
#pragma unroll
  for (int i = 0; i < N; i++) w[i] = __builtin_amdgcn_update_dpp(0, w[i], CTRL, 0xF, 0xF, true);
  __builtin_memcpy(&v, w, sizeof(V));
  return v;
}

// K v at one site of a run, v(y + 1) = dn, v(y - 1) = up; the links carry K's
// factor 1/2 and eta_y.  FP32 keeps U_x(x - 1) beside the site's own links and
// reads the x-neighbours as DPP operands (sw_hop_x); FP64, which has neither
// the registers nor such operands, moves v(x + 1) and conj(U_x) v to the
// lane that needs them.
__device__ __forceinline__ c64 rs_hop(c64 v, c64 up, c64 dn, c64 ux, c64 uxm, c64 uy, c64 uym) {
  return sw_hop(v, dn, up, ux, uxm, uy, uym);
}
__device__ __forceinline__ c128 rs_hop(c128 v, c128 up, c128 dn, c128 ux, c128, c128 uy, c128 uym) {
  const c128 back = rs_shift<kDwPrev>(rs_msubc(c128{0.0, 0.0}, ux, v));  // -conj(U_x) v of lane l - 1
  return rs_msubc(rs_madd(rs_madd(back, ux, rs_shift<kDwNext>(v)), uy, dn), uym, up);
}
// m2 w - K v
__device__ __forceinline__ c64 rs_mhop(float m2, c64 w, c64 v, c64 up, c64 dn, c64 ux, c64 uxm, c64 uy, c64 uym) {
  return sw_mhop(m2, w, v, dn, up, ux, uxm, uy, uym);
}
__device__ __forceinline__ c128 rs_mhop(double m2, c128 w, c128 v, c128 up, c128 dn, c128 ux, c128 uxm, c128 uy,
                                        c128 uym) {
  const c128 k = rs_hop(v, up, dn, ux, uxm, uy, uym);
  return {rs_fma(m2, w.re, -k.re), rs_fma(m2, w.im, -k.im)};
}

template <class R>
__device__ __forceinline__ void rs_links(const RsLinks& lk, int i, R ey, cx<R>& ux, cx<R>& uy) {
  c128 a, b;
  c64 c, d;
  if (lk.prec == 0) {
    a = static_cast<const c128*>(lk.u)[2 * i];
    b = static_cast<const c128*>(lk.u)[2 * i + 1];
  } else {
    if (lk.prec == 1) {
      c = static_cast<const c64*>(lk.u)[2 * i];
      d = static_cast<const c64*>(lk.u)[2 * i + 1];
    } else {
      const LinksF16 h{static_cast<const HalfLink*>(lk.u), lk.sc};
      h.load(i, c, d);
    }
    cvt(a, c);
    cvt(b, d);
  }
  ux = {R(0.5) * R(a.re), R(0.5) * R(a.im)};
  uy = {ey * R(b.re), ey * R(b.im)};
}

// ------------------------------------------------------------ reductions --
// Sums over the lanes of a wave, four words side by side: lane l ends with
// the total of word l & 3 (in every row of 16 lanes alike).
__device__ __forceinline__ double rs_xor16(double v) {  // v(l) + v(l ^ 16), the lower row first
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const auto lo = __builtin_amdgcn_permlane16_swap(unsigned(b), unsigned(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(unsigned(b >> 32), unsigned(b >> 32), false, false);
  const double a = __longlong_as_double((long long)((unsigned long long)lo[0] | ((unsigned long long)hi[0] << 32)));
  const double c = __longlong_as_double((long long)((unsigned long long)lo[1] | ((unsigned long long)hi[1] << 32)));
  return a + c;
}
__device__ __forceinline__ double rs_xor32(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const auto lo = __builtin_amdgcn_permlane32_swap(unsigned(b), unsigned(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(unsigned(b >> 32), unsigned(b >> 32), false, false);
  const double a = __longlong_as_double((long long)((unsigned long long)lo[0] | ((unsigned long long)hi[0] << 32)));
  const double c = __longlong_as_double((long long)((unsigned long long)lo[1] | ((unsigned long long)hi[1] << 32)));
  return a + c;
}
// lanes of equal l & 3 within a row of 16 (a fixed order per lane)
__device__ __forceinline__ double rs_quads(double v) {
  v += dpp_mov<0x124>(v);         // row_ror:4
  return v + dpp_mov<0x128>(v);   // row_ror:8
}
template <int ND>
__device__ __forceinline__ double rs_wave_words(const double (&v)[ND]) {
  static_assert(ND == 1 || ND == 2 || ND == 4, "words");
  const int lane = threadIdx.x & 63;
  double t;
  if constexpr (ND == 1) {
    t = v[0] + dpp_mov<0xB1>(v[0]);
    t += dpp_mov<0x4E>(t);
  } else {
    // lane parity selects the word; each pair of lanes swaps the other's
    const bool b0 = lane & 1, b1 = lane & 2;
    t = (b0 ? v[1] : v[0]) + dpp_mov<0xB1>(b0 ? v[0] : v[1]);
    if constexpr (ND == 4) {
      const double w = (b0 ? v[3] : v[2]) + dpp_mov<0xB1>(b0 ? v[2] : v[3]);
      t = (b1 ? w : t) + dpp_mov<0x4E>(b1 ? t : w);
    } else {
      t += dpp_mov<0x4E>(t);
    }
  }
  return rs_xor32(rs_xor16(rs_quads(t)));
}
// the eight waves' words (LDS [wave][4]): totals in lanes l & 3
__device__ __forceinline__ double rs_block_words(const double (*w)[4]) {
  const int lane = threadIdx.x & 63;
  static_assert(kRsWaves == 8, "two rows of lanes");
  return rs_xor16(rs_quads(w[(lane >> 2) & 7][lane & 3]));
}

// Adds ND values over the block and stores them to the block's line of
// reduction c, then empties its line of reduction c + 2.
template <int ND>
__device__ __forceinline__ void rs_publish(const double (&v)[ND], double (*sm)[4], unsigned long long* lines, int c) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double t = rs_wave_words<ND>(v);
  if (lane < ND) sm[wave][lane] = t;
  __syncthreads();
  if (wave == 0) {
    const double b = rs_block_words(sm);
    if (lane < ND)
      rs_store(lines + ((c & 3) * kRsMaxBlocks + blockIdx.x) * kRsLine + lane,
               (unsigned long long)__double_as_longlong(b));
    // (all words: reduction c + 2 may have more of them than this one)
    if (lane < 4) rs_store(lines + (((c + 2) & 3) * kRsMaxBlocks + blockIdx.x) * kRsLine + lane, kRsEmpty);
  }
}

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
  T rim[kRsWaves][R][4];  // the run's two columns each side: published, then the neighbours'
  double part[kRsWaves][4], tot[kRsWaves][4];
  int bad;
  T x[kX ? R : 1][kX ? kRsThreads : 1];
  T r[kR ? kR : 1][kR ? kRsThreads : 1];
  T uyt[kR ? kRsThreads : 1];
  T h[kX ? 2 : 1][RS_NHALO][kX ? 64 : 1];
};

template <class T, int R, int M>
__global__ __launch_bounds__(kRsThreads) void k_rs_cg(RsGeom g, RsSolve so) {
  using Re = typename Real<T>::type;
  using A = typename std::conditional<M == RS_REF, T, Re>::type;  // alpha: complex in the reference's order
  using Sh = RsShared<T, R>;
  constexpr int NW = kRsWaves, L = NW * R;
  __shared__ Sh sh;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nblk = gridDim.x, lx = g.lx, ly = g.ly;
  const int sx = blockIdx.x % g.nsx, sy = blockIdx.x / g.nsx;
  const int x0 = int(long(lx) * sx / g.nsx), cols = int(long(lx) * (sx + 1) / g.nsx) - x0;
  // every tile has L rows: the last band begins early and shares rows with
  // the one before it, which alone stores them and counts them in the sums
  const int y0 = min(sy * L, ly - L), shared = sy * L - y0;
  const int yw = y0 + wave * R;  // the wave's first row
  const bool top = wave == 0, edge = top || wave == NW - 1;
  const bool valid = lane < cols + 2 * kRsHalo;
  const bool own = lane >= kRsHalo && lane < cols + kRsHalo;
  const bool rim = valid && !own;                                 // a neighbour's column
  const bool side = own && (lane < 2 * kRsHalo || lane >= cols);  // a column neighbours need
  int xg = (x0 - kRsHalo + lane) % lx;
  xg = valid ? (xg < 0 ? xg + lx : xg) : 0;
  const Re ey = (xg & 1) ? Re(-0.5) : Re(0.5);
  const Re m2 = Re(so.mass * so.mass);
  auto wrapy = [&](int y) {
    y %= ly;
    return y < 0 ? y + ly : y;
  };
  // a vector's entry at (xg, y), or -1 where a compact vector has none
  // (rows and columns pass through empty asm statements here and below, so
  // that the compiler does not keep the addresses of every row in registers)
  auto at = [&](int y) -> int {
    int x = xg;
    asm volatile("" : "+v"(x));
    if (!so.eo) return y * lx + x;
    return ((x + y) & 1) ? -1 : y * (lx >> 1) + (x >> 1);
  };
  // the rows other bands keep as halo rows, as a mask over the wave's rows
  unsigned pub = 0;
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int y = yw + j, t = y % L;
    if (t < 2 || t >= L - 2 || y >= ly - 2 || y == ly - L - 1 || y == ly - L - 2) pub |= 1u << j;
  }
  pub = __builtin_amdgcn_readfirstlane(pub);

  T rv_[R - Sh::kR], p[R], ap[R], ux[R], uy[R], xr[Sh::kX ? 1 : R], uxm[sizeof(T) == 8 ? R : 1];
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
  auto uxm_of = [&](int j) -> T { return uxm[sizeof(T) == 8 ? j : 0]; };
  uxm[0] = zero_of<T>();
#pragma unroll
  for (int j = 0; j < R; j++) {
    rref(j) = p[j] = ap[j] = ux[j] = uy[j] = zero_of<T>();
    T x = zero_of<T>();
    if (valid) {
      rs_links<Re>(so.lk, (yw + j) * lx + xg, ey, ux[j], uy[j]);
      if constexpr (M != RS_MIXED) {
        const int i = at(yw + j);
        if (own && i >= 0) x = so.x[i];
      }
    }
    xref(j) = x;
    if constexpr (sizeof(T) == 8) uxm[j] = rs_shift<kDwPrev>(ux[j]);
  }
  // U_y of the row above the run; on the edge waves the two rows beyond the
  // tile, nearest first (y0 - 1, y0 - 2 or y0 + L, y0 + L + 1), and the
  // nearest one's links with U_y of the row below it
  T uyt_reg = zero_of<T>(), hreg[Sh::kX ? 1 : RS_NHALO];
  auto hal = [&](int v) -> T& {  // (edge waves only)
    if constexpr (Sh::kX) return sh.h[top ? 0 : 1][v][lane];
    else return hreg[v];
  };
  auto uyt = [&]() -> T& {
    if constexpr (Sh::kR != 0) return sh.uyt[threadIdx.x];
    else return uyt_reg;
  };
  const int yh[2] = {wrapy(top ? y0 - 1 : y0 + L), wrapy(top ? y0 - 2 : y0 + L + 1)};
  {
    T a, b = zero_of<T>(), ux0 = b, uy0 = b, uy1 = b, uyw = b;
    if (valid) {
      rs_links<Re>(so.lk, wrapy(yw - 1) * lx + xg, ey, a, uyw);
      if (edge) {
        rs_links<Re>(so.lk, yh[0] * lx + xg, ey, ux0, uy0);
        rs_links<Re>(so.lk, yh[1] * lx + xg, ey, a, uy1);
        if (!top) uy1 = uy[R - 1];
      }
    }
    uyt() = uyw;
    if (edge || !Sh::kX) {
#pragma unroll
      for (int v = 0; v < RS_UXH; v++) hal(v) = b;
      hal(RS_UXH) = ux0;
      hal(RS_UYH) = uy0;
      hal(RS_UYHM) = uy1;
    }
  }
  if (threadIdx.x == 0) sh.bad = 0;

  // ring slots: 32-bit byte offsets from the uniform base
  const unsigned row_bytes = unsigned(lx) * sizeof(T), buf_bytes = unsigned(ly) * row_bytes;
  auto slot = [&](int use, int y) {
    unsigned off = unsigned(xg) * sizeof(T);
    asm volatile("" : "+v"(off));
    off += unsigned(use & 3) * buf_bytes + unsigned(y) * row_bytes;
    return reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(so.ring) + off);
  };
  // The columns neighbours exchange pass through LDS, so that each of the 4 R
  // values of a run is one lane's: lane l moves row l / 4, the run's columns 0,
  // 1, w - 2, w - 1 (published) and -2, -1, w, w + 1 (collected) for l % 4 =
  // 0 .. 3.  Their slots lie by block and row, four in a row, so that a wave
  // stores whole lines.
  const int mrow = lane >> 2, mcol = lane & 3;
  const bool mover = lane < 4 * R;
  const unsigned col_bytes = unsigned(nblk) * unsigned(L * 4 * sizeof(T));
  char* cols_base = reinterpret_cast<char*>(so.ring) + size_t(kRsBufs) * buf_bytes;
  auto col_word = [&](int use, unsigned off) {
    return reinterpret_cast<unsigned long long*>(cols_base + (unsigned(use & 3) * col_bytes + off));
  };
  auto col_off = [&](int blk, int c) { return unsigned((blk * L + wave * R + mrow) * 4 + c) * unsigned(sizeof(T)); };
  const int row0 = blockIdx.x - sx;  // the band's first block
  const int left = row0 + (sx == 0 ? g.nsx - 1 : sx - 1), right = row0 + (sx == g.nsx - 1 ? 0 : sx + 1);
  const unsigned put_off = col_off(blockIdx.x, mcol), get_off = col_off(mcol < 2 ? left : right, mcol ^ 2);
  const int scol = lane < 2 * kRsHalo ? lane - 2 : lane - cols + 2;  // a side lane's column of the four
  const int rcol = lane < kRsHalo ? lane : lane - cols;              // a rim lane's
  // f(slot, j) for the rows of the wave that other bands read
  auto for_rows = [&](int use, auto f) {
    if (pub == 0) return;
    if (own) {
#pragma unroll
      for (int j = 0; j < R; j++)
        if (pub >> j & 1) f(slot(use, yw + j), j);
    }
  };
  auto wave_fence = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // Publishes v (own lanes) as ring use e and the sums as reduction c.
  auto publish = [&](const T(&v)[R], int e, const auto& sums, int c) {
    if (side) {
#pragma unroll
      for (int j = 0; j < R; j++) sh.rim[wave][j][scol] = v[j];
    }
    wave_fence();
    rs_stores_done();  // (the slots emptied since the last reduction)
    if (mover) rs_put<T>(col_word(e, put_off), sh.rim[wave][mrow][mcol]);
    for_rows(e, [&](unsigned long long* q, int j) { rs_put<T>(q, v[j]); });
    rs_publish(sums, sh.part, so.lines, c);
    if (mover) rs_empty<T>(col_word(e + 2, put_off));
    for_rows(e + 2, [&](unsigned long long* q, int) { rs_empty<T>(q); });
  };
  // Collects ring use e into the halo lanes of v and the halo rows hal(h) (RING),
  // and the totals of reduction c over all blocks; false: a wait ran out.
  auto collect = [&](auto ring, T(&v)[R], int h, int e, auto& sums, int c) -> bool {
    constexpr bool RING = decltype(ring)::value;
    constexpr int ND = int(sizeof(sums) / sizeof(double));
    constexpr int J = (kRsMaxBlocks * ND + kRsThreads - 1) / kRsThreads;
    const int l0 = threadIdx.x / ND;
    const unsigned long long* base = so.lines + (c & 3) * kRsMaxBlocks * kRsLine + (lane & (ND - 1));
    const bool need = l0 < nblk;
    unsigned long long q[J];
#pragma unroll
    for (int i = 0; i < J; i++) q[i] = 0;
    T h0 = zero_of<T>(), h1 = h0, m = h0;
    bool ok;
    int it = 0;
    do {
      // (all loads of a round in flight together)
      if (need) {
#pragma unroll
        for (int i = 0; i < J; i++) {
          const int b = l0 + i * (kRsThreads / ND);
          if (i == 0 || b < nblk) q[i] = rs_load(base + b * kRsLine);
        }
      }
      if constexpr (RING) {
        if (edge && valid) {
          h0 = rs_read<T>(slot(e, yh[0]));
          h1 = rs_read<T>(slot(e, yh[1]));
        }
        if (mover) m = rs_read<T>(col_word(e, get_off));
      }
      ok = true;
#pragma unroll
      for (int i = 0; i < J; i++) ok &= q[i] != kRsEmpty;
      if constexpr (RING) ok = ok && rs_there(h0) && rs_there(h1) && rs_there(m);
    } while (!ok && ++it < so.spins);
    if (!ok) sh.bad = 1;
    if constexpr (RING) {
      if (edge) {
        hal(h) = h0;
        hal(h + 1) = h1;
      }
      if (mover) sh.rim[wave][mrow][mcol] = m;
      wave_fence();
      if (rim) {
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = sh.rim[wave][j][rcol];
      }
    }
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < J; i++) t += __longlong_as_double((long long)q[i]);
    if constexpr (ND == 1) t += dpp_mov<0xB1>(t);
    if constexpr (ND <= 2) t += dpp_mov<0x4E>(t);
    t = rs_xor32(rs_xor16(rs_quads(t)));
    if (lane < ND) sh.tot[wave][lane] = t;
    __syncthreads();
    t = rs_block_words(sh.tot);
#pragma unroll
    for (int i = 0; i < ND; i++) sums[i] = readlane_d(t, i);
    return sh.bad == 0;
  };
  auto give_up = [&]() {
    if (threadIdx.x == 0) so.out->err = 1;
  };
  const std::integral_constant<bool, true> with_ring{};
  const std::integral_constant<bool, false> sums_only{};
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;

  int k = 0, c = 0, e = 0;  // iteration, reductions and ring uses so far
  int reliable = 0;
  A a;
  if constexpr (M == RS_REF) a = zero_of<T>();
  else a = Re(0);
  Re be = Re(0);
  double rsq = 0.0, maxrr = 0.0, bsqrt = 0.0, resSq = 0.0;
  const int kmax = so.max_iter - 1;
  bool first = true;
  __syncthreads();
  for (;;) {
    {
      // ---- r = b - A x with FP64 links, a march down the wave's rows: at
      // step t the loads of row t - 2 of the run, q = K x on the row before
      // it, A x on the one before that
      const double m2d = so.mass * so.mass;
      const double ed = (xg & 1) ? -0.5 : 0.5;
      const c128 z{0.0, 0.0};
      c128 xa = z, xb = z, qa = z, qb = z, u1x = z, u1y = z, u2x = z, u2y = z, u3y = z;
      double s2[2] = {0.0, 0.0};
#pragma unroll 1
      for (int t = 0; t < R + 4; t++) {
        const int y = wrapy(yw - 2 + t), i = at(y);
        c128 xc = z, ucx = z, ucy = z;
        if (valid) {
          if (i >= 0) xc = rs_read<c128>(reinterpret_cast<const unsigned long long*>(so.x + i));
          rs_links<double>(RsLinks{so.u64, nullptr, 0}, y * lx + xg, ed, ucx, ucy);
        }
        const c128 qc = rs_hop(xb, xa, xc, u1x, z, u1y, u2y);
        if (t >= 4) {
          const c128 ax = rs_mhop(m2d, xa, qb, qa, qc, u2x, z, u2y, u3y);
          const int j = t - 4, ib = at(yw + j);
          c128 d = z;
          if (own && ib >= 0) {
            const c128 bv = so.b[ib];
            d = bv - ax;
            if (wave * R + j >= shared) {
              s2[0] += norm2(d);
              s2[1] += norm2(bv);
            }
          }
          T dr;
          cvt(dr, d);
#pragma unroll
          for (int jj = 0; jj < R; jj++)
            if (jj == j) ap[jj] = dr;
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
      publish(ap, e, s2, c);
      if (!collect(with_ring, ap, RS_RH, e, s2, c)) return give_up();
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
    sh.v[0][wave][0][lane] = p[0];
    sh.v[0][wave][1][lane] = p[R - 1];

    // ---- q = K p (in ap), then Ap = m^2 p - K q in its place
    __syncthreads();
    T qh = zero_of<T>(), p0 = qh;
    if (edge) {
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
    constexpr int N1 = M == RS_REF ? 2 : 4;
    double v1[N1];
#pragma unroll
    for (int i = 0; i < N1; i++) v1[i] = 0.0;
#pragma unroll
    for (int j = 0; j < R; j++) {
      if constexpr (Sh::kX) __builtin_amdgcn_sched_barrier(0);
      const T q = ap[j];
      const T v = rs_mhop(m2, p[j], q, up, j + 1 < R ? ap[j + 1 < R ? j + 1 : j] : below, ux[j], uxm_of(j), uy[j],
                          j ? uy[j ? j - 1 : 0] : uyt());
      up = q;
      ap[j] = v;
      if (wave * R + j >= shared) {
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
    }
#pragma unroll
    for (int i = 0; i < N1; i++) v1[i] = own ? v1[i] : 0.0;
    publish(ap, e, v1, c);
    if (!collect(with_ring, ap, RS_APH, e, v1, c)) return give_up();
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
        if (wave * R + j >= shared) v2[0] = __builtin_fma(rv.re, rv.re, __builtin_fma(rv.im, rv.im, v2[0]));
      }
      v2[0] = own ? v2[0] : 0.0;
      rs_stores_done();  // (slots and lines emptied since the last reduction)
      rs_publish<1>(v2, sh.part, so.lines, c);
      if (edge) {
#pragma unroll
        for (int h = 0; h < 2; h++) hal(RS_RH + h) = rs_axpy(ma, hal(RS_APH + h), hal(RS_RH + h));
      }
#pragma unroll
      for (int j = 0; j < R; j++) xref(j) = rs_axpy(a, p[j], xref(j));
      if (!collect(sums_only, ap, 0, e, v2, c)) return give_up();
      c++;
      const double rn = v2[0];
      if (lead && so.hist) so.hist[k] = sqrt(rn) / bsqrt;
      stop = sqrt(rn) < so.eps * bsqrt || k == kmax;
      be = Re(rn / rsq);
      rsq = rn;
    } else {
      // <p, Ap>, |Ap|^2, <Ap, r>, |r|^2 (real parts; A is Hermitian)
      // (a zero residual ends the solve: no step)
      rsq = v1[3];
      const double al = rsq == 0.0 ? 0.0 : rsq / v1[0];
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

    // ---- the solution to memory, for the true residual
#pragma unroll
    for (int j = 0; j < R; j++) {
      if constexpr (M != RS_REF) xref(j) = rs_axpy(a, p[j], xref(j));
      int y = yw;
      asm volatile("" : "+s"(y));
      const int i = at(y + j);
      if (own && i >= 0 && wave * R + j >= shared) {
        unsigned long long* q = reinterpret_cast<unsigned long long*>(so.x + i);
        c128 v;
        cvt(v, xref(j));
        if constexpr (M == RS_MIXED) v = rs_read<c128>(q) + v;
        rs_put<c128>(q, v);
      }
      if constexpr (M == RS_MIXED) xref(j) = zero_of<T>();
    }
    rs_stores_done();
    double none[1] = {0.0};
    rs_publish<1>(none, sh.part, so.lines, c);
    if (!collect(sums_only, ap, 0, e, none, c)) return give_up();
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
int resident_spins();

// The tiling a system would run resident with on the current device; false
// where it does not fit.
bool rs_plan(int lx, int ly, RsGeom& g);

// Words of the exchange buffers (lines, then ring) of a solve with `words`
// 64-bit words per element.
inline long rs_exchange_words(const RsGeom& g, int words) {
  const long columns = long(g.nsx) * g.nsy * kRsWaves * g.rows * 4;
  return long(kRsBufs) * (kRsMaxBlocks * kRsLine + (long(g.lx) * g.ly + columns) * words);
}
// Empties the exchange buffers and clears the result record, then launches.
void rs_launch(hipStream_t st, const RsGeom& g, RsMode mode, const RsSolve& so);

// The resident blocks of every solve in flight on a device, over all host
// threads, stay within its CUs, one block each: a solve waits here until its
// blocks fit.  Held from before the launch until the stream has drained.
class RsReserve {
 public:
  explicit RsReserve(int blocks);
  ~RsReserve();
  RsReserve(const RsReserve&) = delete;
  RsReserve& operator=(const RsReserve&) = delete;

 private:
  int dev_, blocks_;
};

}  // namespace glx
