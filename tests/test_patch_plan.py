"""The plan of the fused constraint sweep (csrc/patch_plan.cpp) on the CPU: sweeping every
patch by itself leaves its own vertices as a color-by-color pass over the whole mesh does.
A constraint is stood in for by an exact function of its id and all its vertices' values, so
any missing, extra or misordered constraint changes the result."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

from xrtailor_amd import scenes

CSRC = Path(__file__).resolve().parent.parent / "xrtailor_amd" / "csrc"

DRIVER = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "patch_plan.h"
#include "topology.h"
using namespace xrt;
static uint64_t Mix(uint64_t z) { return SplitMix64(&z); }
static void Solve(uint64_t* x, const int* v, int arity, uint64_t id) {
  uint64_t h = Mix(id);
  for (int a = 0; a < arity; ++a) h = Mix(h ^ x[v[a]]);
  for (int a = 0; a < arity; ++a) x[v[a]] = Mix(x[v[a]] + h + a);
}
int main(int argc, char** argv) {
  const int mode = atoi(argv[1]), target = atoi(argv[2]), max_local = atoi(argv[3]), first = atoi(argv[4]);
  const double max_work = atof(argv[5]);
  int nv, nt;
  if (scanf("%d %d", &nv, &nt) != 2) return 2;
  std::vector<float> pos(3 * nv);
  std::vector<int32_t> tris(3 * nt);
  for (auto& p : pos) if (scanf("%f", &p) != 1) return 2;
  for (auto& t : tris) if (scanf("%d", &t) != 1) return 2;
  const auto edges = BuildEdges(tris.data(), nt);
  const auto bends = BuildBends(tris.data(), nt, edges);
  const std::vector<int32_t>* sets[3] = {&tris, &edges, &bends};
  const int arity[3] = {3, 2, 4};
  std::vector<PatchFamily> fam;
  for (int k = first; k < 3; k += first == 0 ? 2 : 1) {  // strain + bends, or edges + bends
    const int n = static_cast<int>(sets[k]->size()) / arity[k];
    int nc = 0;
    const auto col = ColorConstraints(sets[k]->data(), arity[k], n, nv, 7, mode, &nc);
    PatchFamily F;
    F.arity = arity[k];
    F.coloff.assign(nc + 1, 0);
    for (int c : col) F.coloff[c + 1]++;
    for (int c = 0; c < nc; ++c) F.coloff[c + 1] += F.coloff[c];
    std::vector<int32_t> fill(F.coloff.begin(), F.coloff.end() - 1);
    F.cons.resize(sets[k]->size());
    for (int i = 0; i < n; ++i) {
      const int p = fill[col[i]]++;
      for (int a = 0; a < arity[k]; ++a) F.cons[arity[k] * p + a] = (*sets[k])[arity[k] * i + a];
    }
    fam.push_back(F);
  }
  std::vector<uint64_t> x(nv);
  for (int i = 0; i < nv; ++i) x[i] = Mix(i + 1);
  const std::vector<uint64_t> start = x;
  uint64_t id = 0;
  std::vector<uint64_t> base;
  for (const auto& F : fam) {
    base.push_back(id);
    const int n = static_cast<int>(F.cons.size()) / F.arity;
    for (int p = 0; p < n; ++p) Solve(x.data(), &F.cons[F.arity * p], F.arity, id + p);
    id += n;
  }
  std::vector<Patch> plan;
  const int n_total = argc > 6 ? atoi(argv[6]) : 0;  // > 0: the sizes of such a context on 256 CUs
  if (!(n_total > 0 ? CutInstance(pos.data(), nv, fam, ChoosePatchSizes(n_total, 256), max_local,
                                  max_work, &plan)
                    : BuildPatches(pos.data(), nv, fam, target, max_local, max_work, &plan))) {
    printf("no plan\n");
    return plan.empty() ? 42 : 11;
  }
  std::vector<int> owned(nv, 0), owner(id, 0);
  size_t work = 0, most = 0;
  for (const auto& P : plan) {
    most = std::max(most, P.verts.size());
    std::vector<uint64_t> loc;
    for (int v : P.verts) loc.push_back(start[v]);
    for (size_t f = 0; f < fam.size(); ++f) {
      const int ar = fam[f].arity;
      if (static_cast<int>(P.coloff[f].size()) != std::max(fam[f].colors(), 0) + 1) return 3;
      for (size_t e = 0; e < P.cons[f].size(); ++e) {
        int v[4];
        const int p = P.cons[f][e] & 0x7fffffff;
        for (int a = 0; a < ar; ++a) {
          v[a] = P.local[f][ar * e + a];
          if (v[a] >= static_cast<int>(P.verts.size()) || P.verts[v[a]] != fam[f].cons[ar * p + a]) return 4;
        }
        if (P.cons[f][e] < 0) owner[base[f] + p]++;
        Solve(loc.data(), v, ar, base[f] + p);
        ++work;
      }
      for (size_t c = 0; c + 1 < P.coloff[f].size(); ++c) {  // one color at a time, no shared vertex
        std::vector<int> seen(P.verts.size(), 0);
        for (int e = P.coloff[f][c]; e < P.coloff[f][c + 1]; ++e) {
          const int p = P.cons[f][e] & 0x7fffffff;
          if (p < fam[f].coloff[c] || p >= fam[f].coloff[c + 1]) return 5;
          for (int a = 0; a < ar; ++a)
            if (seen[P.local[f][ar * e + a]]++) return 6;
        }
      }
    }
    for (int i = 0; i < P.n_own; ++i) {
      owned[P.verts[i]]++;
      if (loc[i] != x[P.verts[i]]) return 7;
    }
  }
  for (int o : owned) if (o != 1) return 8;
  for (int o : owner) if (o != 1) return 9;
  if (static_cast<int>(most) > max_local) return 10;
  if (id && static_cast<double>(work) > max_work * id) return 12;
  printf("patches %zu work %.2f largest %zu\n", plan.size(), id ? double(work) / id : 0.0, most);
  return 0;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(DRIVER)
    exe = d / "plan"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", f"-I{CSRC}", str(d / "main.cpp"),
                    str(CSRC / "patch_plan.cpp"), str(CSRC / "topology.cpp"), "-o", str(exe)],
                   check=True)
    return exe


def _mesh(kind):
    if kind == "grid":
        return scenes.grid(33, 1.0)
    if kind.startswith("grid"):
        return scenes.grid(int(kind[4:]), 1.0)
    if kind == "strip":
        pos, tris = scenes.grid(41, 1.0)
        keep = np.all(tris < 5 * 41, axis=1)
        return pos[:5 * 41], tris[keep]
    if kind == "tube":
        return scenes.tube(24, 17, 0.2, 0.6)
    if kind == "ball":
        return scenes.icosphere(3, 1.0)
    if kind == "triangle":
        return np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0.0]]), np.array([[0, 1, 2]], np.int32)
    rng = np.random.RandomState(3)  # faces between random vertices: no locality, edges of > 2 faces
    tris = np.array([rng.choice(60, 3, replace=False) for _ in range(80)], np.int32)
    return rng.rand(60, 3), tris


def _run(driver, kind, mode, target, max_local, first, max_work, n_total=0):
    pos, tris = _mesh(kind)
    text = f"{len(pos)} {len(tris)}\n" + " ".join(f"{v:.9g}" for v in np.ravel(pos)) + "\n" + \
        " ".join(str(v) for v in np.ravel(tris)) + "\n"
    r = subprocess.run([str(driver), *map(str, (mode, target, max_local, first, max_work, n_total))],
                       input=text, capture_output=True, text=True)
    print(r.stdout.strip())
    return r.returncode


@pytest.mark.parametrize("kind", ["grid", "strip", "tube", "ball", "triangle", "random"])
@pytest.mark.parametrize("mode,target,max_local,first", [
    (0, 64, 10240, 1), (0, 200, 10240, 0), (1, 100, 10240, 1), (0, 5000, 10240, 1),
    (0, 300, 700, 1), (0, 1, 10240, 1)])
def test_sweeping_patches_equals_the_color_order(driver, kind, mode, target, max_local, first):
    assert _run(driver, kind, mode, target, max_local, first, 1e9) == 0


def test_no_plan_beyond_the_work_or_size_limit(driver):
    assert _run(driver, "grid", 0, 64, 10240, 1, 2.0) == 42   # needs six times the constraints
    assert _run(driver, "grid", 0, 64, 50, 1, 1e9) == 42      # one vertex needs more than 50
    assert _run(driver, "grid", 0, 2000, 10240, 1, 1.0) == 0  # one patch: nothing twice


# cloths of 40,960 vertices and more in contexts where an instance of their size is to stay whole
# (more vertices than that per CU), and around; 5,851 vertices hold the reverse sweep's adjoints
@pytest.mark.parametrize("kind,copies", [("grid203", 204), ("grid203", 210), ("grid256", 216),
                                         ("grid100", 1000), ("grid203", 1)])
@pytest.mark.parametrize("first,max_local", [(1, 10240), (0, 10240), (1, 5851)])
def test_instances_of_any_size_get_a_plan(driver, kind, copies, first, max_local):
    n_total = copies * int(kind[4:]) ** 2
    assert _run(driver, kind, 0, 0, max_local, first, 6.0, n_total) == 0
