"""The planner's tile tables on the CPU, through a program linked to the library:
the parts of every tile that the FP64 GEMM cuts along K cover the tile's
contracted values once, in order, and each joined tile has at least one part,
also where block pairs without values (sectors of size zero) make up a block.
"""
import os
import shutil
import subprocess

import pytest

from helpers import ROOT

PKG = os.path.join(ROOT, "itensors.jl_amd")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "itg_plan.h"
using namespace itg;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

// groups: M N, number of pairs, then their K
int main(int argc, char** argv) {
  ExecPlan ep;
  ep.ta = std::atoi(argv[1]);
  ep.tb = std::atoi(argv[2]);
  const bool want = std::atoi(argv[3]) != 0;
  int64_t off_a = 0, off_b = 0, off_c = 0;
  for (int i = 4; i < argc;) {
    GemmGroup g{};
    g.M = std::atoi(argv[i++]);
    g.N = std::atoi(argv[i++]);
    g.ldc = g.M;
    g.off_c = off_c;
    off_c += (int64_t)g.M * g.N;
    g.p0 = (int32_t)ep.h_pairs.size();
    for (int n = std::atoi(argv[i++]); n > 0; --n) {
      GemmPair p{};
      p.K = std::atoi(argv[i++]);
      p.off_a = off_a;
      p.off_b = off_b;
      p.lda = ep.ta ? p.K : g.M;
      p.ldb = ep.tb ? g.N : p.K;
      off_a += (int64_t)g.M * p.K;
      off_b += (int64_t)g.N * p.K;
      p.alpha_re = 1.0;
      ep.h_pairs.push_back(p);
    }
    g.p1 = (int32_t)ep.h_pairs.size();
    set_first_pair(&g, ep.h_pairs.data());
    ep.h_groups.push_back(g);
  }
  TileForm form[2];
  PartTables pt;
  const std::vector<GemmTile> whole = xcd_tile_table(ep, form, &pt);
  CHECK(whole.size() % 8 == 0);
  CHECK(!want || form[0] == TileForm::kParts);
  if (pt.tiles.empty()) return 0;
  size_t live = 0, cut = 0;
  std::vector<int> uses(pt.groups.size(), 0);
  for (const GemmTile& t : whole) live += t.g >= 0;
  for (const GemmTile& t : pt.tiles) {
    if (t.g < 0) continue;
    CHECK((size_t)t.g < pt.groups.size());
    ++uses[(size_t)t.g];
    if (pt.groups[(size_t)t.g].part) ++cut; else --live;
  }
  CHECK(live == pt.joins.size());  // every tile is left whole or joined
  size_t g = ep.h_groups.size();
  int64_t at = 0;
  for (const GemmJoin& J : pt.joins) {
    CHECK(J.S >= 1);
    CHECK(J.poff == at);
    at += (int64_t)J.S * J.M * J.N;
    // the tile's group: the one whose block holds its first element
    size_t o = 0;
    while (o + 1 < ep.h_groups.size() && ep.h_groups[o + 1].off_c <= J.off_c) ++o;
    const GemmGroup& G = ep.h_groups[o];
    const int m0 = (int)((J.off_c - G.off_c) % G.ldc), n0 = (int)((J.off_c - G.off_c) / G.ldc);
    int p = G.p0, k = 0;
    for (int s = 0; s < J.S; ++s, ++g) {
      const GemmGroup& h = pt.groups[g];
      CHECK(uses[g] == 1 && h.part && h.M == J.M && h.N == J.N && h.ldc == J.M);
      CHECK(h.off_c == J.poff + (int64_t)s * J.M * J.N && h.p1 > h.p0 && h.pf == h.p0);
      for (int q = h.p0; q < h.p1; ++q) {
        const GemmPair& y = pt.pairs[(size_t)q];
        while (p < G.p1 && k == ep.h_pairs[(size_t)p].K) ++p, k = 0;
        CHECK(p < G.p1);
        const GemmPair& x = ep.h_pairs[(size_t)p];
        CHECK(y.K > 0 && k + y.K <= x.K && y.lda == x.lda && y.ldb == x.ldb);
        CHECK(y.off_a == x.off_a + (ep.ta ? k + (int64_t)m0 * x.lda : (int64_t)k * x.lda + m0));
        CHECK(y.off_b == x.off_b + (ep.tb ? (int64_t)k * x.ldb + n0 : k + (int64_t)n0 * x.ldb));
        CHECK(k + y.K == x.K || y.K % 16 == 0);
        k += y.K;
      }
    }
    while (p < G.p1 && k == ep.h_pairs[(size_t)p].K) ++p, k = 0;
    CHECK(p == G.p1);
  }
  CHECK(at == pt.elems && g == pt.groups.size() && cut == g - ep.h_groups.size());
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(cxx):
        pytest.skip("needs hipcc")
    d = tmp_path_factory.mktemp("tiles")
    (d / "tiles.cpp").write_text(PROGRAM)
    libdir = os.path.join(PKG, "itg")
    subprocess.run([cxx, "-std=c++17", "-O1", "--offload-host-only",
                    "-I" + os.path.join(PKG, "csrc"), "-c", "-x", "hip", str(d / "tiles.cpp"),
                    "-o", str(d / "tiles.o")], check=True)
    subprocess.run([cxx, str(d / "tiles.o"), os.path.join(libdir, "libitg.so"),
                    "-Wl,-rpath," + libdir, "-o", str(d / "tiles")], check=True)
    return str(d / "tiles")


def group(M, N, *ks):
    return [M, N, len(ks), *ks]


CASES = {
    "one block": (1, group(1500, 1500, 1500)),
    "edges": (1, group(3001, 1777, 2049)),
    "pairs": (1, group(1500, 1500, 17, 31, 640, 3, 200, 609)),
    "empty pairs between": (1, group(1500, 1500, 0, 860, 0, 0, 640, 0)),
    "empty block of many pairs": (1, group(1500, 1500, 1500) + group(64, 64, *[0] * 400)),
    "empty edge block": (1, group(1500, 1500, 1500) + group(700, 33, *[0] * 2000)),
    "only empty": (0, group(700, 330, *[0] * 1000)),
    "small": (0, group(40, 50, 60)),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
def test_parts_cover_their_tiles(program, name, ta, tb):
    want, groups = CASES[name]
    r = subprocess.run([program, str(ta), str(tb), str(want)] + [str(x) for x in groups],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
