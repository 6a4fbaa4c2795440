#include "patch_plan.h"

#include <algorithm>
#include <cstddef>
#include <limits>

namespace xrt {
namespace {

// cuts v[b, e) into `parts` pieces of nearly equal size along its longest axis, recursively
void Bisect(const float* pos, std::vector<int32_t>& v, int b, int e, int parts,
            std::vector<std::vector<int32_t>>* out) {
  if (parts <= 1 || e - b <= 1) {
    out->emplace_back(v.begin() + b, v.begin() + e);
    return;
  }
  float lo[3], hi[3];
  for (int k = 0; k < 3; ++k) {
    lo[k] = std::numeric_limits<float>::max();
    hi[k] = -lo[k];
  }
  for (int i = b; i < e; ++i)
    for (int k = 0; k < 3; ++k) {
      const float x = pos[3 * static_cast<size_t>(v[i]) + k];
      lo[k] = std::min(lo[k], x);
      hi[k] = std::max(hi[k], x);
    }
  int axis = 0;
  for (int k = 1; k < 3; ++k)
    if (hi[k] - lo[k] > hi[axis] - lo[axis]) axis = k;
  const int left = parts / 2;
  const int mid = b + static_cast<int>(static_cast<int64_t>(e - b) * left / parts);
  std::nth_element(v.begin() + b, v.begin() + mid, v.begin() + e, [&](int32_t p, int32_t q) {
    const float x = pos[3 * static_cast<size_t>(p) + axis], y = pos[3 * static_cast<size_t>(q) + axis];
    return x < y || (x == y && p < q);
  });
  Bisect(pos, v, b, mid, left, out);
  Bisect(pos, v, mid, e, parts - left, out);
}

}  // namespace

bool BuildPatches(const float* pos, int nv, const std::vector<PatchFamily>& families, int target,
                  int max_local, double max_work, std::vector<Patch>* out) {
  out->clear();
  if (nv <= 0) return true;
  max_local = std::min(max_local, 65535);
  // per family: the constraint of each color that vertex v is in, at [v * colors + c] (-1: none),
  // and the last patch that listed each constraint
  std::vector<std::vector<int32_t>> at(families.size()), seen(families.size());
  for (size_t f = 0; f < families.size(); ++f) {
    const PatchFamily& F = families[f];
    const size_t nc = static_cast<size_t>(std::max(F.colors(), 0));
    at[f].assign(nc * nv, -1);
    seen[f].assign(F.cons.size() / F.arity, -1);
    for (size_t c = 0; c < nc; ++c)
      for (int p = F.coloff[c]; p < F.coloff[c + 1]; ++p)
        for (int a = 0; a < F.arity; ++a)
          at[f][F.cons[static_cast<size_t>(F.arity) * p + a] * nc + c] = p;
  }
  double budget = 0.0;  // listed constraints left
  for (const PatchFamily& F : families) budget += max_work * static_cast<double>(F.cons.size()) / F.arity;
  std::vector<int32_t> all(nv);
  for (int i = 0; i < nv; ++i) all[i] = i;
  std::vector<std::vector<int32_t>> todo;
  Bisect(pos, all, 0, nv, std::max(1, (nv + target - 1) / std::max(target, 1)), &todo);
  std::reverse(todo.begin(), todo.end());
  std::vector<int32_t> local(nv, -1);  // mark of the needed vertices, then their patch-local index
  std::vector<int32_t> list, start;    // listed constraints, last color first; color starts
  for (int32_t id = 0; !todo.empty(); ++id) {
    std::vector<int32_t> need = std::move(todo.back());
    todo.pop_back();
    std::sort(need.begin(), need.end());
    const int n_own = static_cast<int>(need.size());
    for (int32_t v : need) local[v] = 0;
    list.clear();
    start.clear();
    bool fits = true;
    for (int f = static_cast<int>(families.size()) - 1; f >= 0 && fits; --f) {
      const PatchFamily& F = families[f];
      const int32_t* of = at[f].data();
      const size_t nc = static_cast<size_t>(std::max(F.colors(), 0));
      for (size_t c = nc; c-- > 0 && fits;) {
        const size_t first = list.size();
        start.push_back(static_cast<int32_t>(first));
        for (int32_t v : need) {
          const int32_t p = of[v * nc + c];
          if (p < 0 || seen[f][p] == id) continue;
          seen[f][p] = id;
          list.push_back(p);
        }
        // (the vertices that join here have no other constraint of this color)
        for (size_t i = first; i < list.size(); ++i)
          for (int a = 0; a < F.arity; ++a) {
            const int32_t v = F.cons[static_cast<size_t>(F.arity) * list[i] + a];
            if (local[v] < 0) {
              local[v] = 0;
              need.push_back(v);
            }
          }
        fits = static_cast<int>(need.size()) <= max_local;
        budget -= static_cast<double>(list.size() - first);
      }
    }
    if (budget < 0.0) {
      out->clear();
      return false;
    }
    if (!fits) {
      for (int32_t v : need) local[v] = -1;
      if (n_own <= 1) {
        out->clear();
        return false;
      }
      std::vector<int32_t> own(need.begin(), need.begin() + n_own);
      std::vector<std::vector<int32_t>> halves;
      Bisect(pos, own, 0, n_own, 2, &halves);
      for (auto it = halves.rbegin(); it != halves.rend(); ++it) todo.push_back(std::move(*it));
      continue;
    }
    std::sort(need.begin() + n_own, need.end());
    for (size_t i = 0; i < need.size(); ++i) local[need[i]] = static_cast<int32_t>(i);
    Patch P;
    P.n_own = n_own;
    P.coloff.resize(families.size());
    P.cons.resize(families.size());
    P.local.resize(families.size());
    size_t k = start.size();  // the colors were listed last first
    for (size_t f = 0; f < families.size(); ++f) {
      const PatchFamily& F = families[f];
      P.coloff[f].push_back(0);
      for (int c = 0; c < F.colors(); ++c) {
        --k;
        const size_t e = k + 1 < start.size() ? start[k + 1] : list.size();
        for (size_t i = start[k]; i < e; ++i) {
          const int32_t* v = &F.cons[static_cast<size_t>(F.arity) * list[i]];
          const uint32_t own = local[v[0]] < n_own ? 0x80000000u : 0u;
          P.cons[f].push_back(static_cast<int32_t>(static_cast<uint32_t>(list[i]) | own));
          for (int a = 0; a < F.arity; ++a) P.local[f].push_back(static_cast<uint16_t>(local[v[a]]));
        }
        P.coloff[f].push_back(static_cast<int32_t>(P.cons[f].size()));
      }
    }
    for (int32_t v : need) local[v] = -1;
    P.verts = std::move(need);
    out->push_back(std::move(P));
  }
  return true;
}

// Own vertices per patch: what gives 4 of 5 CUs a patch, down to 256 vertices, where the
// ring of neighbors already quadruples the stretch work of a grid, and up to 4096 (a grid's
// patch then needs 117 KB of LDS, 1.4x the stretch and 1.2x the bend work).  ms per frame at
// 144 / 256 / 400 / 1024 / 2304 / 4096 own vertices: one 64 x 64 cloth 2.22 / 2.28 / 2.40 /
// 2.75 / 3.51 / 4.43, 16 garments (93 k vertices) - / 10.3 / 8.25 / 8.66 / 9.67 / 10.5, 256
// cloths (2.53 M vertices) 115 / 108 / 75 / 44.6 / 29.3 / 23.7.  An instance stays whole
// (nothing is solved twice) when there are patches enough without cutting it, and below
// 1200 vertices, where a color takes one or two rounds of one workgroup anyway.
PatchSizes ChoosePatchSizes(int n_total, int cu_count) {
  const int per_cu = n_total / std::max(1, cu_count * 4 / 5);
  return PatchSizes{std::min(4096, std::max(256, per_cu)), std::max(1200, per_cu)};
}

bool CutInstance(const float* pos, int nv, const std::vector<PatchFamily>& families, PatchSizes sizes,
                 int max_local, double max_work, std::vector<Patch>* out) {
  // (BuildPatches halves what a workgroup cannot hold, however large the instance is)
  if (nv <= sizes.whole) return BuildPatches(pos, nv, families, nv, max_local, max_work, out);
  for (int target = sizes.cut; target < 40960; target *= 4)
    if (BuildPatches(pos, nv, families, target, max_local, max_work, out)) return true;
  return false;
}

}  // namespace xrt
