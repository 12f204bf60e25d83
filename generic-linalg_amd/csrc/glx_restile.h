// glx_restile.h -- what the resident-system kernels share (glx_resident.h,
// glx_reshop.h): a lattice held on the chip as tiles, one per block, the
// exchange of tile boundaries between blocks and the chip-wide sums.
//
// Block b owns a tile: one of nsx strips of at most 64 - 2 H columns by one of
// nsy bands of 8 R rows, H the operator's reach.  A wave holds R whole rows of
// its tile in registers: lane l <-> column x0 - H + l, so the first H and the H
// lanes after the strip's own are the neighbours' columns ("rim") and
// x-neighbours come by DPP wave shifts; y-neighbours are other registers of
// the lane, or pass through LDS between the waves of a block.  The first and
// last wave also keep the H rows beyond the tile.  Vectors that are updated by
// axpys are updated in those halo lanes and rows like the owner's (the same
// instructions on the same values), so only operator results have to be
// exchanged.
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
constexpr int rs_cols(int halo) { return 64 - 2 * halo; }  // columns a strip may own
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
  // one-hop operators: the diagonal, and the links' factor in x and on even
  // columns in y (fx) and on odd columns in y (fy_odd)
  double diag, fx, fy_odd;
  int spins;       // polls per wait
  double* hist;    // iterated relative residual per iteration, or null
  unsigned long long* ring;   // [kRsBufs][lx * ly] boundary rows by lattice site, then
                              // [kRsBufs][blocks][8 R][2 H] boundary columns, of T
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
// acc + conj(a) b
template <class R>
__device__ __forceinline__ cx<R> rs_maddc(cx<R> acc, cx<R> a, cx<R> b) {
  return {rs_fma(a.re, b.re, rs_fma(a.im, b.im, acc.re)), rs_fma(a.re, b.im, rs_fma(-a.im, b.re, acc.im))};
}
// acc + s b for a real or complex scalar s
template <class R>
__device__ __forceinline__ cx<R> rs_axpy(R s, cx<R> b, cx<R> acc) {
  return {rs_fma(s, b.re, acc.re), rs_fma(s, b.im, acc.im)};
}
__device__ __forceinline__ double rs_axpy(double s, double b, double acc) { return rs_fma(s, b, acc); }
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
__device__ __forceinline__ void rs_links(const RsLinks& lk, int i, R fx, R fy, cx<R>& ux, cx<R>& uy) {
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
  ux = {fx * R(a.re), fx * R(a.im)};
  uy = {fy * R(b.re), fy * R(b.im)};
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

// Adds ND values over block blk and stores them to the block's line of
// reduction c, then empties its line of reduction c + 2.
template <int ND>
__device__ __forceinline__ void rs_publish(const double (&v)[ND], double (*sm)[4], unsigned long long* lines, int c,
                                           int blk) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double t = rs_wave_words<ND>(v);
  if (lane < ND) sm[wave][lane] = t;
  __syncthreads();
  if (wave == 0) {
    const double b = rs_block_words(sm);
    if (lane < ND)
      rs_store(lines + ((c & 3) * kRsMaxBlocks + blk) * kRsLine + lane,
               (unsigned long long)__double_as_longlong(b));
    // (all words: reduction c + 2 may have more of them than this one)
    if (lane < 4) rs_store(lines + (((c + 2) & 3) * kRsMaxBlocks + blk) * kRsLine + lane, kRsEmpty);
  }
}

// ------------------------------------------------------------------ tile --
// LDS of the exchange: the run's H columns each side (published, then the
// neighbours'), the reductions' staging, and whether a wait of the block ran out.
template <class T, int R, int H>
struct RsExShared {
  T rim[kRsWaves][R][2 * H];
  double part[kRsWaves][4], tot[kRsWaves][4];
  int bad;
};

__device__ __forceinline__ void rs_wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class T, int R, int H>
struct RsTile {
  static constexpr int NW = kRsWaves, L = NW * R;
  using Sh = RsExShared<T, R, H>;
  Sh& sh;
  int lane, wave, blk, nblk, lx, ly;  // blk of nblk: the system's blocks
  int x0, cols, y0, shared;  // shared: the first rows, which the band before stores and counts
  int yw;                    // the wave's first row
  int xg;                    // the lane's column (0 where not valid)
  int yh[H];                 // the edge waves' halo rows, nearest first
  unsigned pub;              // the wave's rows other bands keep as halo rows (a mask)
  bool top, edge, valid, own, rim, side;
  unsigned row_bytes, buf_bytes, col_bytes, put_off, get_off;
  int mrow, mcol, scol, rcol;
  bool mover;
  char* ring;
  unsigned long long* lines;
  int spins;

  __device__ __forceinline__ RsTile(Sh& sh_, const RsGeom& g, unsigned long long* ring_, unsigned long long* lines_,
                                    int spins_, int blk_ = blockIdx.x)
      : sh(sh_), blk(blk_), ring(reinterpret_cast<char*>(ring_)), lines(lines_), spins(spins_) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    nblk = g.nsx * g.nsy;
    lx = g.lx;
    ly = g.ly;
    const int sx = blk % g.nsx, sy = blk / g.nsx;
    x0 = int(long(lx) * sx / g.nsx);
    cols = int(long(lx) * (sx + 1) / g.nsx) - x0;
    // every tile has L rows: the last band begins early and shares rows with
    // the one before it, which alone stores them and counts them in the sums
    y0 = min(sy * L, ly - L);
    shared = sy * L - y0;
    yw = y0 + wave * R;
    top = wave == 0;
    edge = top || wave == NW - 1;
    valid = lane < cols + 2 * H;
    own = lane >= H && lane < cols + H;
    rim = valid && !own;
    side = own && (lane < 2 * H || lane >= cols);
    xg = (x0 - H + lane) % lx;
    xg = valid ? (xg < 0 ? xg + lx : xg) : 0;
#pragma unroll
    for (int h = 0; h < H; h++) yh[h] = wrapy(top ? y0 - 1 - h : y0 + L + h);
    pub = 0;
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int y = yw + j, t = y % L;
      if (t < H || t >= L - H || y >= ly - H || (y < ly - L && y >= ly - L - H)) pub |= 1u << j;
    }
    pub = __builtin_amdgcn_readfirstlane(pub);
    // ring slots: 32-bit byte offsets from the uniform base
    row_bytes = unsigned(lx) * sizeof(T);
    buf_bytes = unsigned(ly) * row_bytes;
    col_bytes = unsigned(nblk) * unsigned(L * 2 * H * sizeof(T));
    // The columns neighbours exchange pass through LDS, so that each of the
    // 2 H R values of a run is one lane's: lane l moves row l / 2H, and the
    // run's first H columns and last H (published) or the H columns on either
    // side of it (collected).
    mrow = lane / (2 * H);
    mcol = lane & (2 * H - 1);
    mover = lane < 2 * H * R;
    const int row0 = blk - sx;  // the band's first block
    const int left = row0 + (sx == 0 ? g.nsx - 1 : sx - 1), right = row0 + (sx == g.nsx - 1 ? 0 : sx + 1);
    put_off = col_off(blk, mcol);
    get_off = col_off(mcol < H ? left : right, mcol ^ H);
    scol = lane < 2 * H ? lane - H : lane - cols + H;  // a side lane's column of the 2 H
    rcol = lane < H ? lane : lane - cols;              // a rim lane's
  }
  __device__ __forceinline__ int wrapy(int y) const {
    y %= ly;
    return y < 0 ? y + ly : y;
  }
  // whether row j of the wave is this block's to store and count
  __device__ __forceinline__ bool counts(int j) const { return wave * R + j >= shared; }
  __device__ __forceinline__ unsigned col_off(int blk, int c) const {
    return unsigned((blk * L + wave * R + mrow) * 2 * H + c) * unsigned(sizeof(T));
  }
  // (the column passes through an empty asm statement here, so that the
  // compiler does not keep the addresses of every row in registers)
  __device__ __forceinline__ unsigned long long* slot(int use, int y) const {
    unsigned off = unsigned(xg) * sizeof(T);
    asm volatile("" : "+v"(off));
    off += unsigned(use & 3) * buf_bytes + unsigned(y) * row_bytes;
    return reinterpret_cast<unsigned long long*>(ring + off);
  }
  __device__ __forceinline__ unsigned long long* col_word(int use, unsigned off) const {
    return reinterpret_cast<unsigned long long*>(ring + size_t(kRsBufs) * buf_bytes +
                                                 (unsigned(use & 3) * col_bytes + off));
  }
  // f(slot, j) for the rows of the wave that other bands read
  template <class F>
  __device__ __forceinline__ void for_rows(int use, F f) const {
    if (pub == 0) return;
    if (own) {
#pragma unroll
      for (int j = 0; j < R; j++)
        if (pub >> j & 1) f(slot(use, yw + j), j);
    }
  }
  // Publishes v (own lanes) as ring use e and the sums as reduction c.
  template <int ND>
  __device__ __forceinline__ void publish(const T (&v)[R], int e, const double (&sums)[ND], int c) {
    if (side) {
#pragma unroll
      for (int j = 0; j < R; j++) sh.rim[wave][j][scol] = v[j];
    }
    rs_wave_fence();
    rs_stores_done();  // (the slots emptied since the last reduction)
    if (mover) rs_put<T>(col_word(e, put_off), sh.rim[wave][mrow][mcol]);
    for_rows(e, [&](unsigned long long* q, int j) { rs_put<T>(q, v[j]); });
    rs_publish(sums, sh.part, lines, c, blk);
    if (mover) rs_empty<T>(col_word(e + 2, put_off));
    for_rows(e + 2, [&](unsigned long long* q, int) { rs_empty<T>(q); });
  }
  // Publishes the sums alone.
  template <int ND>
  __device__ __forceinline__ void publish(const double (&sums)[ND], int c) {
    rs_stores_done();  // (slots and lines emptied since the last reduction)
    rs_publish(sums, sh.part, lines, c, blk);
  }
  // Collects ring use e into the rim lanes of v and, by halo(h, value) on the
  // edge waves, the halo rows (RING), and the totals of reduction c over all
  // blocks; false: a wait ran out.
  template <bool RING, int ND, class F>
  __device__ __forceinline__ bool collect_(T (&v)[R], F halo, int e, double (&sums)[ND], int c) {
    constexpr int J = (kRsMaxBlocks * ND + kRsThreads - 1) / kRsThreads;
    const int l0 = threadIdx.x / ND;
    const unsigned long long* base = lines + (c & 3) * kRsMaxBlocks * kRsLine + (lane & (ND - 1));
    const bool need = l0 < nblk;
    unsigned long long q[J];
#pragma unroll
    for (int i = 0; i < J; i++) q[i] = 0;
    T m = zero_of<T>(), hv[H];
#pragma unroll
    for (int h = 0; h < H; h++) hv[h] = zero_of<T>();
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
#pragma unroll
          for (int h = 0; h < H; h++) hv[h] = rs_read<T>(slot(e, yh[h]));
        }
        if (mover) m = rs_read<T>(col_word(e, get_off));
      }
      ok = true;
#pragma unroll
      for (int i = 0; i < J; i++) ok &= q[i] != kRsEmpty;
      if constexpr (RING) {
        ok = ok && rs_there(m);
#pragma unroll
        for (int h = 0; h < H; h++) ok = ok && rs_there(hv[h]);
      }
    } while (!ok && ++it < spins);
    if (!ok) sh.bad = 1;
    if constexpr (RING) {
      if (edge) {
#pragma unroll
        for (int h = 0; h < H; h++) halo(h, hv[h]);
      }
      if (mover) sh.rim[wave][mrow][mcol] = m;
      rs_wave_fence();
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
  }
  template <int ND, class F>
  __device__ __forceinline__ bool collect(T (&v)[R], F halo, int e, double (&sums)[ND], int c) {
    return collect_<true>(v, halo, e, sums, c);
  }
  template <int ND>
  __device__ __forceinline__ bool collect(double (&sums)[ND], int c) {
    T v[R];
    return collect_<false>(v, [](int, T) {}, 0, sums, c);
  }
};

}  // namespace glx
