"""The serving engine's estimate of a solve's device memory against the split
rules of the launches (m2l_split.h): level arrays and the partial sums of any
number of targets must fit in it without its tables term and its slack.

The estimate is internal to serve.cpp, so a small program is built around the
source and linked to the library; it touches no device."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "serve.cpp"
using namespace wbfmm;

static unsigned chunks(unsigned nt, unsigned per, bool even) {
  if (!even) return (nt + per - 1) / per;
  unsigned n = 0;
  for (unsigned c = 0; c < 8; c++) n += (nt / 8 + (c < nt % 8) + per - 1) / per;
  return n;
}

int main() {
  int bad = 0, cases = 0;
  for (int helm = 0; helm < 2; helm++)
    for (int precision = 32; precision <= 64; precision += 32)
      for (int depth = 2; depth <= 6; depth++)
        for (int order : {2, 5, 8, 13, 16, 20, 24, 27, 30, 40}) {
          if (!helm && order > 24) continue;
          wbfmm_serve_request_t r{};
          Plan p;
          r.problem = helm ? WBFMM_PROBLEM_HELMHOLTZ : WBFMM_PROBLEM_LAPLACE;
          r.k = 1.0;
          r.nsrc = 1000;
          r.fstr = 8;
          p.precision = precision;
          p.depth = depth;
          p.D = 1.0;
          p.lmax = order;
          for (int l = 0; l <= depth; l++) p.orders[l] = order;
          const size_t fp = footprint(r, p) - table_bytes(r.problem, p) - ((size_t)16 << 20);
          size_t arrays = 0, part = 0;
          for (int l = 1; l <= depth; l++) {
            const unsigned nb = 1u << (3 * l);
            const size_t C = (size_t)(order + 1) * (order + 1);
            const size_t one = C * (helm ? 2 : 1) * (precision == 32 ? 4 : 8);
            arrays += 2 * one * nb;
            for (unsigned nt = 1; l >= 2 && nt <= nb; nt += nt < 600 ? 1 : nt / 64)
              for (int even = 0; even < 2; even++) {
                if (!even && nt > nb / 8) continue;   // one class holds an eighth of a level
                const unsigned n16 = chunks(nt, 16, even), n8 = chunks(nt, 8, even);
                const int s = m2l_nsplit(l, helm ? n8 : n16, one);
                if (s > 1) part = std::max(part, (size_t)s * nt * one);
                if (helm) {   // orders above 27 and levels of two orders, in FP64
                  const int w = wide_nsplit(n8), u = wide_m2m_nsplit((nt + 7) / 8);
                  if (w > 1) part = std::max(part, (size_t)w * nt * C * 16);
                  if (u > 1) part = std::max(part, (size_t)u * nt * C * 16);
                }
              }
          }
          cases++;
          if (fp < arrays + part) {
            bad++;
            printf("helm %d precision %d depth %d order %d: %.1f MB estimated, %.1f needed\n", helm,
                   precision, depth, order, fp / 1e6, (arrays + part) / 1e6);
          }
        }
  printf("%d cases, %d too small\n", cases, bad);
  return bad != 0;
}
"""


def test_estimate_holds_the_split_partials(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    lib = os.path.join(ROOT, "wbfmm_amd")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(lib, "csrc"), "-o", str(exe), str(src), "-L", lib,
                        "-l:libwbfmm.so", "-Wl,-rpath," + lib, "-Wl,--allow-shlib-undefined"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
