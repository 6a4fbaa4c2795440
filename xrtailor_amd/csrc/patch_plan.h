// Host-side plan of the fused constraint sweep (patch.h): the vertices of an instance are cut
// into compact patches, and each patch lists the constraints it has to solve, color by
// color, so that its own vertices come out of the whole sweep exactly as a color-by-color
// pass over the instance leaves them.
//
// The lists follow from the dependencies: going through the colors backwards with the set of
// vertices whose value is needed (at first the patch's own), every constraint of the color
// that touches the set is listed and its other vertices join the set.  A constraint that
// crosses a patch boundary is therefore listed by every patch that needs it; each solves it on
// the same inputs with the same result, and one of them (the patch that owns the
// constraint's first vertex) is its owner.  Within a color no two constraints share a vertex,
// so a vertex is in at most one constraint of a color.
#pragma once
#include <cstdint>
#include <vector>

namespace xrt {

// One kind of constraints in color-sorted order: constraint p has the vertices
// cons[arity * p ..], color c holds the positions [coloff[c], coloff[c + 1]).
struct PatchFamily {
  int arity = 0;
  std::vector<int32_t> cons;
  std::vector<int32_t> coloff;
  int colors() const { return static_cast<int>(coloff.size()) - 1; }
};

struct Patch {
  int n_own = 0;               // the first n_own of verts are the patch's own vertices
  std::vector<int32_t> verts;  // instance-local ids: own, then the others, each ascending
  // per family: entries of every color one after the other, coloff[f][c] their offsets
  std::vector<std::vector<int32_t>> coloff;
  std::vector<std::vector<int32_t>> cons;   // constraint position; bit 31: this patch owns it
  std::vector<std::vector<uint16_t>> local; // arity patch-local vertex indices per entry
};

// Patches of about `target` own vertices over `nv` vertices at `pos` (3 floats each), the
// families swept in the given order.  A patch whose vertices exceed max_local is cut again.
// False (and no plan) when even single vertices need more, or when the patches together list
// more than max_work times the constraints (a mesh without locality).
bool BuildPatches(const float* pos, int nv, const std::vector<PatchFamily>& families, int target,
                  int max_local, double max_work, std::vector<Patch>* out);

// How a context's instances are cut: one of up to `whole` vertices stays whole (as far as
// max_local allows), a larger one gets patches of about `cut` own vertices.
struct PatchSizes {
  int cut, whole;
};
PatchSizes ChoosePatchSizes(int n_total, int cu_count);

// BuildPatches for one instance at these sizes.  A mesh with little locality gets larger patches,
// or none.
bool CutInstance(const float* pos, int nv, const std::vector<PatchFamily>& families, PatchSizes sizes,
                 int max_local, double max_work, std::vector<Patch>* out);

}  // namespace xrt
