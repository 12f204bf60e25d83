"""The resident GCR kernel's walk over the staged neighbour values
(glx_rgwalk.h), on the host: every read, those of zero coefficients beyond a
wave's last pair included, is a column that the kernel writes.  With an even
number of colours each staged site ends in a pad that nothing writes (the
pitch is odd); LDS is not cleared between kernels, so a NaN left there by
another kernel would go through 0 * NaN into the solution."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <cstdio>
#include <initializer_list>
#include "glx_rgwalk.h"
using namespace glx;

int main() {
  long bad = 0, reads = 0, pairs = 0;
  for (int m = 1; m <= 4; m *= 2)
    for (int nt : {5, 13})
      for (int nc = 1; nc <= 64 * m; nc++) {
        const int sites = 64 * m / nc, nf = nt * nc, tspan = sites * rg_pitch(nc);
        int next = 0;  // the pairs of all waves, each once and in order
        for (int wave = 0; wave < kRgWaves; wave++) {
          const int f0 = rg_first(nf, wave), f1 = rg_end(nf, wave), kf = rg_kept(m);
          RgWalk w(nt, nc, sites, f0);
          auto read = [&](int f, bool coefficient) {
            const int t = w.at / tspan, c = w.at % tspan;
            bool ok = w.at >= 0 && t < nt && c < nc;
            if (coefficient) {
              ok = ok && f == next && t == f / nc && c == f % nc;
              next++;
              pairs++;
            }
            if (!ok && bad++ < 10) std::printf("m %d terms %d colours %d wave %d pair %d: word %d\n", m, nt, nc, wave, f, w.at);
            reads++;
            w.step();
          };
          // (coefficients: the kernel's kept[q] is zero unless wave * share + q < f1)
          for (int q0 = 0; q0 < kf; q0 += 4)
            if (f0 + q0 < f1)
              for (int q = q0; q < q0 + 4; q++) read(f0 + q, wave * rg_share(nf) + q < f1);
          for (int f = f0 + kf; f < f1; f++) read(f, true);
        }
        if (next != nf && bad++ < 10) std::printf("m %d terms %d colours %d: %d of %d pairs\n", m, nt, nc, next, nf);
      }
  std::printf("%ld reads, %ld pairs, %ld bad\n", reads, pairs, bad);
  return bad != 0;
}
"""


def test_every_read_is_a_written_column(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "generic-linalg_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
