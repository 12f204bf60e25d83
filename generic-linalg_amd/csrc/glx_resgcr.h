// glx_resgcr.h -- GCR (generic_gcr.cpp:27-156) on the general Nc-colour stencil
// with the iteration on the chip: one launch runs up to kRgDirs iterations.
//
// What bounds it: the launch-per-phase form takes 6 + k/8 launches and two
// allocations for iteration k, 85 us of them at 32 x 32 x 8 colours where the
// data of an iteration (5 MB of coefficients, some MB of stored directions)
// take 2 us from L2.  Here an iteration is three exchanges between blocks:
//   r to the neighbours; <Ap_j, Ar> of all stored j with |r|^2, summed in two
//   steps (block b adds up the words b, b + nblk, ... of all blocks, so the
//   traffic does not grow with blocks x blocks x k); <Ap, r> with |Ap|^2.
// The convergence test rides on the second, p_{k+1} (needed for x only) is
// formed while the third is on its way.
//
// Whole solves, launch per phase and here, spectral radius 0.6 (45 to 49
// iterations): 8 x 8 x 8 colours 3.9 and 0.39 ms, 32 x 32 x 8 4.3 and 0.46 to
// 0.52, 48 x 48 x 12 with two-link terms 5.2 and 1.07, 64 x 64 x 12 5.0 and
// 1.37, 90 x 90 x 8 (the largest, 253 blocks of 256 entries) 6.2 and 1.23, with
// two-link terms 5.4 and 1.78 ms.  What is left at 32 x 32 x 8, of 10 us per
// iteration: the three exchanges' round trips 5, the stencil's and the
// directions' sums over the waves 3.  Two entries per lane (64 blocks there)
// took 13.4 us where one takes 11.1; A p_j in LDS instead of L2 and columns
// taken four at a time took it from 11.1 to 9.8.
//
// Block b owns S whole sites, 64 M entries at most; lane l of every wave stands
// for the entries l + 64 m.  The eight waves split the contraction indices:
// (term, column) of the stencil, whose coefficients stay in registers as far as
// they fit, and the stored directions in the sums; partial sums meet in LDS.
// Exchange and flags as in glx_restile.h: a slot is kRsEmpty until its word
// arrives; buffers rotate by use, use u + 2 is emptied after reduction u has
// shown that all reads of use u - 2 are over, and those stores are waited for
// before the block contributes to the next sums.
#pragma once

#include "glx_cstencil.h"
#include "glx_restile.h"
#include "glx_rgwalk.h"

namespace glx {

constexpr int kRgDirs = 64;    // iterations (directions) of a launch
constexpr int kRgChunks = 8;   // launches of a solve

struct RsGcr {
  CsDev st;
  int sites, nblk, nt;       // sites per block, blocks, terms
  int k0, max_iter, spins;
  double eps, bsqrt;         // bsqrt: of launches after the first
  c128* x;                   // guess in, solution out
  const c128* b;
  c128* xs;                  // x and r between launches
  c128* rs;
  c128* dir[kRgChunks];      // [kRgDirs][2][n]: p_j, A p_j
  int held;                  // the launch's directions whose A p_j stay in LDS
  double* norms;             // |A p_j|^2
  double* hist;
  unsigned long long* lines;  // [kRsBufs][kRsMaxBlocks][kRsLine]
  unsigned long long* ring;   // [kRsBufs][2 n] r
  unsigned long long* d1;     // [kRsBufs][nblk][words] blocks' sums
  unsigned long long* d2;     // [kRsBufs][words] totals; words = 2 (k0 + kRgDirs + 1)
  RsOut* out;
};

static_assert(kRgWaves == kRsWaves, "the walk's waves");
__host__ __device__ constexpr int rg_words(int k0) { return 2 * (k0 + kRgDirs + 1); }

template <int M>
__global__ __launch_bounds__(kRsThreads) void k_rs_gcr(RsGcr g) {
  constexpr int NW = kRsWaves, EW = 64 * M;           // entries a block may own
  constexpr int Q = (12 * EW + kRsThreads - 1) / kRsThreads;  // staged values per thread
  constexpr int KF = rg_kept(M);
  const int nc = g.st.nc, n = g.st.lx * g.st.ly * nc, pitch = rg_pitch(nc);
  extern __shared__ c128 lds[];
  c128* stage = lds;                                  // [nt][sites][pitch]
  c128* part = stage + g.nt * g.sites * pitch;        // [NW][EW]
  c128* sum = part + NW * EW;                         // [EW]
  c128* beta = sum + EW;                              // [words / 2]
  c128* held = beta + rg_words(g.k0) / 2;             // [g.held][EW]
  __shared__ double tot[NW][4];
  __shared__ int bad;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = blockIdx.x, tid = threadIdx.x;
  const int E = g.sites * nc, i0 = blk * E, ne = min(E, n - i0);
  const int words = rg_words(g.k0), tspan = g.sites * pitch;
  const c128 z{0.0, 0.0};
  if (tid == 0) bad = 0;
  __syncthreads();

  bool has[M];
  int own[M];  // the entry's place in a staged term, without its column: its site's
#pragma unroll
  for (int m = 0; m < M; m++) {
    const int e = lane + 64 * m;
    has[m] = e < ne;
    own[m] = has[m] ? e / nc * pitch : 0;
  }
  // what this thread stages: entry `from` of the vector to place `to`
  int from[Q], to[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int id = tid + q * kRsThreads, t = 1 + id / E, e = id % E;
    const int s = e / nc, c = e - s * nc;
    from[q] = -1;
    to[q] = 0;
    if (t < g.nt && e < ne) {
      const int v = blk * g.sites + s, y = v / g.st.lx, x = v - y * g.st.lx;
      int dx, dy;
      cs_offset(t, dx, dy);
      from[q] = (cs_wrap(y + dy, g.st.ly) * g.st.lx + cs_wrap(x + dx, g.st.lx)) * nc + c;
      to[q] = t * tspan + s * pitch + c;
    }
  }
  // the wave's columns f of all terms': f0 to f1, the first KF kept
  const int nf = g.nt * nc, wf = rg_share(nf);
  const int f0 = rg_first(nf, wave), f1 = rg_end(nf, wave);
  const c128* __restrict__ coef = g.st.coef + i0 + lane;
  c128 kept[KF][M];
#pragma unroll
  for (int q = 0; q < KF; q++)
#pragma unroll
    for (int m = 0; m < M; m++) {
      const int f = wave * wf + q;
      kept[q][m] = f < f1 && has[m] ? coef[size_t(f) * n + 64 * m] : z;
    }

  // sums over the waves of v, by entry, plus add(e), in every wave
  auto meet = [&](c128 (&v)[M], auto add) {
#pragma unroll
    for (int m = 0; m < M; m++) part[wave * EW + lane + 64 * m] = v[m];
    __syncthreads();
    if (tid < EW) {
      c128 s = part[tid];
#pragma unroll
      for (int w = 1; w < NW; w++) s = s + part[w * EW + tid];
      sum[tid] = add(tid, s);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; m++) v[m] = sum[lane + 64 * m];
  };
  // own entries of v into the staged clover term
  auto stage_own = [&](const c128 (&v)[M]) {
    if (wave == 0) {
#pragma unroll
      for (int m = 0; m < M; m++)
        if (has[m]) stage[own[m] + (lane + 64 * m) % nc] = v[m];
    }
  };
  auto apply_staged = [&](c128 (&av)[M]) {
#pragma unroll
    for (int m = 0; m < M; m++) av[m] = z;
    RgWalk w(g.nt, nc, g.sites, f0);
    // four at a time without a branch: columns beyond f1 have zeros
#pragma unroll
    for (int q0 = 0; q0 < KF; q0 += 4) {
      if (f0 + q0 < f1) {
#pragma unroll
        for (int q = q0; q < q0 + 4; q++) {
#pragma unroll
          for (int m = 0; m < M; m++) av[m] = av[m] + kept[q][m] * stage[w.at + own[m]];
          w.step();
        }
      }
    }
#pragma unroll 4
    for (int f = f0 + KF; f < f1; f++) {
#pragma unroll
      for (int m = 0; m < M; m++)
        if (has[m]) av[m] = av[m] + coef[size_t(f) * n + 64 * m] * stage[w.at + own[m]];
      w.step();
    }
    meet(av, [&](int e, c128 a) {
      if (e >= ne) return z;
      if (g.st.shifts) {
        const int s = e / nc, r = e - s * nc, site = blk * g.sites + s;
        const c128 v = stage[s * pitch + r];
        const bool even = ((site % g.st.lx + site / g.st.lx) & 1) == 0;
        if (g.st.shifts & 1) a = a + g.st.shift * v;
        if (g.st.shifts & 2) a = a + ((even ? 1.0 : -1.0) * g.st.eo_shift) * v;
        if (g.st.shifts & 4) a = a + ((r < nc / 2 ? 1.0 : -1.0) * g.st.dof_shift) * v;
      }
      return a;
    });
  };
  // v to the ring as use u
  auto publish = [&](const c128 (&v)[M], int u) {
    if (wave == 0) {
#pragma unroll
      for (int m = 0; m < M; m++)
        if (has[m]) rs_put<c128>(g.ring + (size_t(u & 3) * n + i0 + lane + 64 * m) * 2, v[m]);
    }
    stage_own(v);
  };
  // the neighbours' values of use u
  auto collect = [&](int u) {
    const unsigned long long* src = g.ring + size_t(u & 3) * n * 2;
    c128 v[Q];
    bool ok;
    int it = 0;
    do {
      ok = true;
#pragma unroll
      for (int q = 0; q < Q; q++)
        if (from[q] >= 0) v[q] = rs_read<c128>(src + size_t(from[q]) * 2);
#pragma unroll
      for (int q = 0; q < Q; q++)
        if (from[q] >= 0) ok &= rs_there(v[q]);
    } while (!ok && ++it < g.spins);
    if (!ok) bad = 1;
#pragma unroll
    for (int q = 0; q < Q; q++)
      if (from[q] >= 0) stage[to[q]] = v[q];
    rs_stores_done();  // (the slots emptied since the last reduction)
    __syncthreads();
  };
  // (v0, v1, v2) over the block to its line of use u, by wave 0
  auto publish_line = [&](double v0, double v1, double v2, int u) {
    const double v[4] = {v0, v1, v2, 0.0};
    const double t = rs_wave_words<4>(v);
    if (lane < 4)
      rs_store(g.lines + ((u & 3) * kRsMaxBlocks + blk) * kRsLine + lane,
               (unsigned long long)__double_as_longlong(t));
  };
  auto collect_lines = [&](double (&s)[3], int u) -> bool {
    constexpr int J = kRsMaxBlocks * 4 / kRsThreads;
    const unsigned long long* base = g.lines + (u & 3) * kRsMaxBlocks * kRsLine + (lane & 3);
    unsigned long long q[J];
    bool ok;
    int it = 0;
    do {
      ok = true;
#pragma unroll
      for (int i = 0; i < J; i++) {
        const int bk = (tid >> 2) + i * (kRsThreads / 4);
        q[i] = bk < g.nblk ? rs_load(base + bk * kRsLine) : 0;
      }
#pragma unroll
      for (int i = 0; i < J; i++) ok &= q[i] != kRsEmpty;
    } while (!ok && ++it < g.spins);
    if (!ok) bad = 1;
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < J; i++) t += __longlong_as_double((long long)q[i]);
    t = rs_xor32(rs_xor16(rs_quads(t)));
    if (lane < 4) tot[wave][lane] = t;
    __syncthreads();
    t = rs_block_words(tot);
#pragma unroll
    for (int i = 0; i < 3; i++) s[i] = readlane_d(t, i);
    return bad == 0;
  };
  auto dir = [&](int j, int which) { return g.dir[j / kRgDirs] + size_t(2 * (j % kRgDirs) + which) * n + i0; };
  // A p_j of the block in LDS, or null
  auto held_dir = [&](int j) -> c128* {
    return unsigned(j - g.k0) < unsigned(g.held) ? held + (j - g.k0) * EW : nullptr;
  };
  auto give_up = [&]() {
    if (tid == 0) g.out->err = 1;
  };

  c128 x[M], r[M], p[M], ap[M], ar[M];
  double bb = 0.0;
  int k = g.k0;
  if (k == 0) {
    // r = b - A x
#pragma unroll
    for (int m = 0; m < M; m++) x[m] = has[m] ? g.x[i0 + lane + 64 * m] : z;
    stage_own(x);
#pragma unroll
    for (int q = 0; q < Q; q++)
      if (from[q] >= 0) stage[to[q]] = g.x[from[q]];
    __syncthreads();
    apply_staged(ar);
#pragma unroll
    for (int m = 0; m < M; m++) {
      const c128 bv = has[m] ? g.b[i0 + lane + 64 * m] : z;
      r[m] = bv - ar[m];
      bb += norm2(bv);
    }
  } else {
#pragma unroll
    for (int m = 0; m < M; m++) {
      x[m] = has[m] ? g.xs[i0 + lane + 64 * m] : z;
      r[m] = has[m] ? g.rs[i0 + lane + 64 * m] : z;
    }
  }
  double bsqrt = g.bsqrt;
  const int kend = min(g.max_iter, g.k0 + kRgDirs);
  const bool lead = blk == 0 && tid == 0;
  int u = 0;
  for (;;) {
    publish(r, u);
    // empty what use u + 2 takes (it holds use u - 2's): the reduction of use
    // u - 1 has shown that every block is past it
    if (u >= 2) {
      const int o = (u + 2) & 3;
      for (int i = tid; i < 2 * ne; i += kRsThreads) rs_store(g.ring + (size_t(o) * n + i0) * 2 + i, kRsEmpty);
      unsigned long long* mine = g.d1 + (size_t(o) * g.nblk + blk) * words;
      for (int i = tid; i < 2 * (k - 1); i += kRsThreads) rs_store(mine + i, kRsEmpty);
      for (int j = blk + tid * g.nblk; j <= k - 2; j += g.nblk * kRsThreads) {
        rs_store(g.d2 + size_t(o) * words + 2 * j, kRsEmpty);
        rs_store(g.d2 + size_t(o) * words + 2 * j + 1, kRsEmpty);
      }
      if (tid < 4) rs_store(g.lines + (o * kRsMaxBlocks + blk) * kRsLine + tid, kRsEmpty);
    }
    collect(u);
    apply_staged(ar);

    // ---- <Ap_j, Ar>, two j at a time per wave; |r|^2 and |b|^2
    unsigned long long* mine = g.d1 + (size_t(u & 3) * g.nblk + blk) * words;
    if (wave == NW - 1) {
      double v[2] = {0.0, bb};
#pragma unroll
      for (int m = 0; m < M; m++) v[0] += norm2(r[m]);
      const double t = rs_wave_words<2>(v);
      if (lane < 2) rs_store(mine + 2 * k + lane, (unsigned long long)__double_as_longlong(t));
    }
    for (int j = 2 * wave; j < k; j += 2 * NW) {
      double v[4] = {0.0, 0.0, 0.0, 0.0};
      c128 a[2][M];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int jh = min(j + h, k - 1);
        if (const c128* d = held_dir(jh)) {
#pragma unroll
          for (int m = 0; m < M; m++) a[h][m] = d[lane + 64 * m];
        } else {
          const c128* q = dir(jh, 1);
#pragma unroll
          for (int m = 0; m < M; m++) a[h][m] = has[m] ? q[lane + 64 * m] : z;
        }
      }
#pragma unroll
      for (int m = 0; m < M; m++) {
        const c128 d0 = dotc(a[0][m], ar[m]), d1 = dotc(a[1][m], ar[m]);
        v[0] += d0.re;
        v[1] += d0.im;
        v[2] += d1.re;
        v[3] += d1.im;
      }
      const double t = rs_wave_words<4>(v);
      if (lane < (j + 1 < k ? 4 : 2)) rs_store(mine + 2 * j + lane, (unsigned long long)__double_as_longlong(t));
    }
    // ---- the words this block adds up: beta_j = -<Ap_j, Ar> / |Ap_j|^2
    for (int j = blk + g.nblk * wave; j <= k; j += g.nblk * NW) {
      constexpr int H = kRsMaxBlocks / 32;
      const double nrm = j < k ? g.norms[j] : 1.0;
      const unsigned long long* src = g.d1 + size_t(u & 3) * g.nblk * words + 2 * j + (lane & 1);
      unsigned long long q[H];
      bool ok;
      int it = 0;
      do {
        ok = true;
#pragma unroll
        for (int h = 0; h < H; h++) {
          const int bk = (lane >> 1) + 32 * h;
          q[h] = bk < g.nblk ? rs_load(src + size_t(bk) * words) : 0;
        }
#pragma unroll
        for (int h = 0; h < H; h++) ok &= q[h] != kRsEmpty;
      } while (!ok && ++it < g.spins);
      if (!ok) bad = 1;
      double t = 0.0;
#pragma unroll
      for (int h = 0; h < H; h++) t += __longlong_as_double((long long)q[h]);
      t += dpp_mov<0x4E>(t);
      t = rs_xor32(rs_xor16(rs_quads(t)));
      if (j < k) t = -t / nrm;
      if (lane < 2) rs_store(g.d2 + size_t(u & 3) * words + 2 * j + lane, (unsigned long long)__double_as_longlong(t));
    }
    for (int i = tid; i < 2 * (k + 1); i += kRsThreads) {
      const unsigned long long* src = g.d2 + size_t(u & 3) * words + i;
      unsigned long long q;
      int it = 0;
      do q = rs_load(src);
      while (q == kRsEmpty && ++it < g.spins);
      if (q == kRsEmpty) bad = 1;
      reinterpret_cast<unsigned long long*>(beta)[i] = q;
    }
    __syncthreads();
    if (bad) return give_up();
    const double rr = beta[k].re;
    if (k == 0) {
      bsqrt = sqrt(beta[0].im);
      if (lead) g.out->bsqrt = bsqrt;
    } else {
      if (lead && g.hist) g.hist[k - 1] = sqrt(rr) / bsqrt;
      if (sqrt(rr) < g.eps * bsqrt || k == g.max_iter) break;
    }
    if (k == kend) {
      // the next launch goes on from here
      if (wave == 0) {
#pragma unroll
        for (int m = 0; m < M; m++) {
          if (has[m]) {
            g.xs[i0 + lane + 64 * m] = x[m];
            g.rs[i0 + lane + 64 * m] = r[m];
          }
        }
      }
      return;
    }

    // ---- Ap = Ar + sum beta_j Ap_j
    auto add_memory = [&](c128 (&v)[M], int j0, int which) {
#pragma unroll 4
      for (int j = j0; j < k; j += NW) {
        const c128 bj = beta[j];
        const c128* d = dir(j, which);
#pragma unroll
        for (int m = 0; m < M; m++)
          if (has[m]) v[m] = v[m] + bj * d[lane + 64 * m];
      }
    };
#pragma unroll
    for (int m = 0; m < M; m++) ap[m] = p[m] = z;
    int j = wave;
    if (g.k0 == 0) {
#pragma unroll 2
      for (; j < min(k, g.held); j += NW) {
        const c128 bj = beta[j];
#pragma unroll
        for (int m = 0; m < M; m++) ap[m] = ap[m] + bj * held[j * EW + lane + 64 * m];
      }
    }
    add_memory(ap, j, 1);
    // (each lane's ar is in sum, from apply_staged)
    meet(ap, [&](int e, c128 s) {
      s = e < ne ? s + sum[e] : z;
      if (e < ne) dir(k, 1)[e] = s;
      if (c128* h = held_dir(k)) h[e] = s;
      return s;
    });
    if (wave == 0) {
      c128 d = z;
      double nn = 0.0;
#pragma unroll
      for (int m = 0; m < M; m++) {
        d = d + dotc(ap[m], r[m]);
        nn += norm2(ap[m]);
      }
      publish_line(d.re, d.im, nn, u);
    }
    // ---- p = r + sum beta_j p_j
    add_memory(p, wave, 0);
    meet(p, [](int, c128 s) { return s; });
#pragma unroll
    for (int m = 0; m < M; m++) {
      p[m] = r[m] + p[m];
      if (wave == 0 && has[m]) dir(k, 0)[lane + 64 * m] = p[m];
    }
    double s[3];
    if (!collect_lines(s, u)) return give_up();
    const c128 alpha{s[0] / s[2], s[1] / s[2]};
    if (tid == 0 && k % g.nblk == blk) g.norms[k] = s[2];
#pragma unroll
    for (int m = 0; m < M; m++) {
      r[m] = r[m] - alpha * ap[m];
      x[m] = x[m] + alpha * p[m];
    }
    k++;
    u++;
  }

  // ---- |b - A x|^2
  if (wave == 0) {
#pragma unroll
    for (int m = 0; m < M; m++)
      if (has[m]) g.x[i0 + lane + 64 * m] = x[m];
  }
  publish(x, u + 1);
  collect(u + 1);
  apply_staged(ar);
  if (wave == 0) {
    double v = 0.0;
#pragma unroll
    for (int m = 0; m < M; m++) v += norm2((has[m] ? g.b[i0 + lane + 64 * m] : z) - ar[m]);
    publish_line(v, 0.0, 0.0, u);
  }
  double s[3];
  if (!collect_lines(s, u)) return give_up();
  if (lead) {
    g.out->resSq = s[0];
    g.out->kfinal = k - 1;
    g.out->done = 1;
  }
}

// Blocks and sites per block; false: not a stencil these kernels take.
bool rg_plan(const CsDev& st, RsGcr& g, int& m);
long rg_exchange_words(const RsGcr& g);
// one launch (kRgDirs iterations from g.k0), after clearing the exchange
void rg_launch(hipStream_t st, int m, RsGcr g);

}  // namespace glx
