// Fused constraint sweep: every stretch and bend color of an iteration in one launch.
//
// One workgroup takes a patch of an instance (patch_plan.h): it stages the patch's vertices
// and the ring of neighbors that their results depend on in LDS, solves the listed
// constraints color by color between workgroup barriers, and writes its own vertices to the
// other of two position buffers (its neighbors' workgroups still read the first).  A
// constraint near a boundary is solved by several patches, each on the same inputs in the
// same order, so the result is that of a color-by-color pass bit for bit.
//
// HBM layout (all patches concatenated):
//   verts   int32[]      global vertex ids of a patch: own, then neighbors
//   off     int32[]      per patch NS + 1 + NB + 1 offsets of its colors into srec / brec
//   srec    int4[]       stretch entry: local indices (16 + 16 bits), rest length,
//                        compliance, constraint (bit 31: this patch owns it)
//   slam    float[]      the entry's multiplier (every patch keeps its own copy)
//   brec    int4[]       bend entry: local indices (4 x 16 bits), rest angle, compliance
//   bcon    int32[]      the bend entry's element (bit 31: owned), read by the taped sweep
// and for the quality mode's constraints, in a plan of their own
//   frec    int4[]       strain entry: local indices (2 x 16 bits, 32 bits), rest area
//   finv    float4[]     its inverse rest matrix
//   irec    int4[]       isometric bending entry: local indices (4 x 16 bits), coefficient,
//                        element (bit 31: owned); iK float4[], ilam float[] its weights and
//                        multiplier
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "contact.h"
#include "device.h"

namespace xrt {

struct PatchDev {
  int32_t vbeg, n_own, n_loc;  // verts[vbeg, vbeg + n_loc)
  int32_t off;                 // the patch's color offsets
  int32_t inst;
};

constexpr int kPatchMaxOffsets = 128;  // stretch + bend colors + 2 that a sweep can hold

struct PatchArgs {
  const PatchDev* patch;
  const int32_t* verts;
  const int32_t* off;
  const int4* srec;
  float* slam;
  const int4* brec;
  const int32_t* bcon;
  float* slam_out;  // multipliers by constraint, written in the last iteration
  int n, ns, nb;    // patches, stretch colors, bend colors
};

struct PatchFemArgs {
  const PatchDev* patch;
  const int32_t* verts;
  const int32_t* off;
  const int4* frec;
  const float4* finv;
  const int4* irec;
  const float4* iK;
  float* ilam;
  float* ilam_out;
  int n, nf, nb;
};

// What a sweep does beside the constraints: ground plane and vertex-face contacts after them
// (before any later operator of the iteration), tape of the operators' inputs (see adjoint.h; null: none)
struct PatchSweep {
  const float4* x;   // input positions
  float4* out;       // output positions (not x)
  const float4* x0;  // start of the substep (ground friction)
  int iter, last;    // iteration; 1 in the substep's last one
  int ground;
  float4* tape_s;
  float4* tape_b;
  float4* tape_g;
  // the vertex-face solves against the obstacles (null: they follow as a launch of their own),
  // with the tape of the positions before and after them
  const InstContactDev* ic;
  float mu, inv_ns;
  float4* tape_c;
  float4* tape_e;
};

hipError_t LaunchPatchSweep(hipStream_t s, const PatchArgs& a, const PatchSweep& w,
                            const StepConsts& k, const BendMode& m, int threads, size_t lds_bytes);
hipError_t LaunchPatchFem(hipStream_t s, const PatchFemArgs& a, const PatchSweep& w,
                          const StepConsts& k, const FemConsts& fk, int threads, size_t lds_bytes);
hipError_t ConfigurePatchSweep(size_t lds_bytes);
// the entries' compliances from the constraints sc (after they changed)
hipError_t LaunchPatchCompliance(hipStream_t s, const StretchC* sc, int4* srec, int n);

}  // namespace xrt
