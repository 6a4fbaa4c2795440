// The vertex-face contact solve of one vertex, run by the collider kernels and at the end of the
// fused constraint sweep.
#pragma once
#include "bvh.h"
#include "contact.h"
#include "contact_math.h"

namespace xrt {
namespace cm {

// SolveVFDCD_Kernel / SolveVFCCD_Kernel (PBDCollision.cu:54-76,280-300)
// VF solve: push along the pred face normal to the contact point (+offset), then, with
// fr.mu > 0, ComputeFriction (ClothSolverHelper.cu:156-169) on that correction: the part of
// the vertex's substep displacement (x - x0) relative to the obstacle face's (its vertices'
// mean frame displacement / substeps) that is tangential to the normal is removed, at most
// mu x |correction|.  The reference applies no friction on mesh contacts; mu = 0 is its
// behaviour.
// True when xi, vertex i's position, was pushed.
__device__ __forceinline__ bool VfSolveVertex(float4& xi, int i, const BvhView& t,
                                              const int32_t* __restrict__ face,
                                              const float4* __restrict__ q, float offset,
                                              const VfFriction& fr) {
  XRT_NO_FMA
  const int f = face[i];
  if (f < 0) return false;
  const int4 tr = t.tris[f];
  const F3 nrm = FaceNormal(L3(t.pred[tr.x]), L3(t.pred[tr.y]), L3(t.pred[tr.z]));
  const float lam = D(nrm, S(L3(xi), L3(q[i]))) - offset;
  if (!(lam < 0)) return false;
  float fx = 0.0f, fy = 0.0f, fz = 0.0f;
  if (fr.mu > 0.0f) {
    const float4 a0 = fr.o_x0[tr.x], b0 = fr.o_x0[tr.y], c0 = fr.o_x0[tr.z];
    const float4 a1 = fr.o_x[tr.x], b1 = fr.o_x[tr.y], c1 = fr.o_x[tr.z];
    const float ox = ((a1.x - a0.x) + (b1.x - b0.x) + (c1.x - c0.x)) / 3.0f * fr.inv_ns;
    const float oy = ((a1.y - a0.y) + (b1.y - b0.y) + (c1.y - c0.y)) / 3.0f * fr.inv_ns;
    const float oz = ((a1.z - a0.z) + (b1.z - b0.z) + (c1.z - c0.z)) / 3.0f * fr.inv_ns;
    const float4 p0 = fr.x0[i];
    const float rx = (xi.x - p0.x) - ox, ry = (xi.y - p0.y) - oy, rz = (xi.z - p0.z) - oz;
    const float rn = rx * nrm.x + ry * nrm.y + rz * nrm.z;
    const float tx = rx - nrm.x * rn, ty = ry - nrm.y * rn, tz = rz - nrm.z * rn;
    const float tl = sqrtf(tx * tx + ty * ty + tz * tz);
    if (tl > 0.0f) {
      const float s = fminf(-lam * fr.mu / tl, 1.0f);
      fx = -tx * s;
      fy = -ty * s;
      fz = -tz * s;
    }
  }
  xi.x += -lam * nrm.x + fx;
  xi.y += -lam * nrm.y + fy;
  xi.z += -lam * nrm.z + fz;
  return true;
}

}  // namespace cm
}  // namespace xrt
