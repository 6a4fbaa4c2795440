#include "patch.h"

#include "contact_solve.h"
#include "elements.h"
#include "fem.h"

namespace xrt {
namespace {

// LDS is all that the waves of a workgroup share between two colors: the global loads of the
// next color's records stay in flight across the barrier
__device__ __forceinline__ void LdsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The patch's color offsets, one per lane (two registers): reading one costs no load and
// gives every lane the same scalar.
struct LaneOffsets {
  int lo, hi;
  __device__ __forceinline__ LaneOffsets(const int32_t* __restrict__ off, int n) {
    const int lane = static_cast<int>(threadIdx.x) & 63;
    lo = lane < n ? off[lane] : 0;
    hi = lane + 64 < n ? off[lane + 64] : 0;
  }
  __device__ __forceinline__ int operator[](int i) const {  // i: the same in every lane
    return i < 64 ? __builtin_amdgcn_readlane(lo, i) : __builtin_amdgcn_readlane(hi, i - 64);
  }
};

// One family of entries, its colors at off[o0 ..]: walked as (color, round) steps with a
// workgroup barrier after each color.  load(e) gives entry e's record, one step ahead of its
// use, so that a color waits for LDS and arithmetic only; solve(e, record) projects it.
template <class Load, class Solve>
__device__ __forceinline__ void SweepColors(const LaneOffsets& off, int o0, int colors, Load&& load,
                                            Solve&& solve) {
  using Rec = decltype(load(0));
  const int tid = threadIdx.x, bs = blockDim.x;
  int c = 0, beg = off[o0], end = off[o0 + 1];
  Rec rec{};
  if (beg + tid < end) rec = load(beg + tid);
  while (c < colors) {
    const int e = beg + tid;
    const bool more = beg + bs < end;        // another round of this color
    const int nbeg = more ? beg + bs : end;  // (colors lie one after the other)
    const int nend = more ? end : (c + 1 < colors ? off[o0 + c + 2] : nbeg);
    Rec next{};
    if (nbeg + tid < nend) next = load(nbeg + tid);
    if (e < end) solve(e, rec);
    if (!more) {
      if (nbeg > off[o0 + c]) LdsBarrier();  // (nothing to wait for after an empty color)
      ++c;
    }
    beg = nbeg;
    end = nend;
    rec = next;
  }
}

// the patch's vertices into LDS
__device__ __forceinline__ void StageVertices(float4* X, const float4* __restrict__ x,
                                              const int32_t* __restrict__ verts, int n) {
  const int tid = threadIdx.x, bs = blockDim.x;
  for (int v0 = tid; v0 < n; v0 += 4 * bs) {
    int g[4];
    float4 p[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) g[u] = v0 + u * bs < n ? verts[v0 + u * bs] : verts[v0];
#pragma unroll
    for (int u = 0; u < 4; ++u) p[u] = x[g[u]];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (v0 + u * bs < n) X[v0 + u * bs] = p[u];
  }
  LdsBarrier();
}

// The patch's own vertices out of LDS, through the ground plane and the vertex-face contacts when
// they come next: both concern one vertex at a time, and as launches of their own they cost 2 to 4
// us and a gap each (8 cloths landing: 5 us less of an iteration).
template <bool kTape>
__device__ __forceinline__ void WriteOwn(const float4* X, const PatchSweep& w, const StepConsts& k,
                                         const PatchDev& p, const int32_t* __restrict__ verts) {
  for (int v = threadIdx.x; v < p.n_own; v += blockDim.x) {
    const int g = verts[v];
    float4 x = X[v];
    if (w.ground) {
      if constexpr (kTape) w.tape_g[g] = x;
      if (x.w > kEps && x.y < k.ground_y) x = GroundVertex(x, w.x0[g], k.ground_y, k.friction);
    }
    if (w.ic) {
      const InstContactDev& c = w.ic[p.inst];
      if constexpr (kTape) w.tape_c[g] = x;
      if (c.has_obs) {
        const VfFriction fr{w.x0 + c.vbeg, c.o_x0, c.o_x, w.inv_ns, w.mu};
        cm::VfSolveVertex(x, g - c.vbeg, c.obvh, c.rt_face, c.rt_q, 0.0f, fr);
        cm::VfSolveVertex(x, g - c.vbeg, c.obvh, c.vf_face, c.vf_q, 1e-3f, fr);
      }
      if constexpr (kTape) w.tape_e[g] = x;
    }
    w.out[g] = x;
  }
}

__device__ __forceinline__ int Lo16(int v) { return v & 0xffff; }
__device__ __forceinline__ int Hi16(int v) { return static_cast<int>(static_cast<uint32_t>(v) >> 16); }

struct StretchEntry {
  int4 r;
  float lam;
};

// Replaces one launch per color (20 on a grid): those were bound by the launches in small
// contexts (about 5 us each for 2.5 us of work) and by sweeping the positions through L2 in
// large ones.  Here a color costs a workgroup barrier, LDS gathers and arithmetic; the sweep is
// bound by the projections' instructions (about 110 per stretch, 400 per bend, most of them
// correctly rounded divisions and roots) and, with few patches, by their latency.  Measured
// per iteration, launches per color -> sweep: one 64 x 64 cloth 59 -> 22 us (one persistent
// workgroup: 41 us), 64 k vertices of garments 60 us less of 131, 256 cloths with 2.53 M
// vertices 450 -> 206 us.
template <bool kTape>
__global__ __launch_bounds__(1024) void PatchSweepKernel(PatchArgs a, PatchSweep w, StepConsts k,
                                                         BendMode m) {
  extern __shared__ float4 X[];
  const PatchDev p = a.patch[blockIdx.x];
  const LaneOffsets off(a.off + p.off, a.ns + a.nb + 2);
  const int32_t* __restrict__ verts = a.verts + p.vbeg;
  StageVertices(X, w.x, verts, p.n_loc);
  SweepColors(
      off, 0, a.ns,
      [&](int e) {
        return StretchEntry{a.srec[e], w.iter > 0 ? a.slam[e] : 0.0f};
      },
      [&](int e, StretchEntry& s) {
        const int i0 = Lo16(s.r.x), i1 = Hi16(s.r.x);
        const StretchC sc{i0, i1, __int_as_float(s.r.y), __int_as_float(s.r.z)};
        float4 xa = X[i0], xb = X[i1];
        if constexpr (kTape) {
          if (s.r.w < 0) {
            const int64_t q = s.r.w & 0x7fffffff;
            w.tape_s[2 * q] = make_float4(xa.x, xa.y, xa.z, s.lam);
            w.tape_s[2 * q + 1] = xb;
          }
        }
        if (StretchSolve(xa, xb, sc, s.lam, k.inv_dt2)) {
          X[i0] = xa;
          X[i1] = xb;
        }
        a.slam[e] = s.lam;
        if (w.last && s.r.w < 0) a.slam_out[s.r.w & 0x7fffffff] = s.lam;
      });
  if (k.solve_bending)
    SweepColors(
        off, a.ns + 1, a.nb, [&](int e) { return a.brec[e]; },
        [&](int e, const int4& r) {
          const int i0 = Lo16(r.x), i1 = Hi16(r.x), i2 = Lo16(r.y), i3 = Hi16(r.y);
          float4 x1 = X[i0], x2 = X[i1], x3 = X[i2], x4 = X[i3];
          if constexpr (kTape) {
            const int q = a.bcon[e];
            if (q < 0) {
              float4* t = w.tape_b + 3 * static_cast<int64_t>(q & 0x7fffffff);
              t[0] = make_float4(x1.x, x1.y, x1.z, x2.x);
              t[1] = make_float4(x2.y, x2.z, x3.x, x3.y);
              t[2] = make_float4(x3.z, x4.x, x4.y, x4.z);
            }
          }
          if (BendSolve(x1, x2, x3, x4, make_float2(__int_as_float(r.z), __int_as_float(r.w)),
                        k.inv_dt2, m)) {
            X[i0] = x1;
            X[i1] = x2;
            X[i2] = x3;
            X[i3] = x4;
          }
        });
  WriteOwn<kTape>(X, w, k, p, verts);
}

struct StrainEntry {
  int4 r;
  float4 inv;
};
struct IsoEntry {
  int4 r;
  float4 K;
  float lam;
};

// The same for the quality mode's constraints: strain over the face colors, then isometric
// bending over the hinge colors.
__global__ __launch_bounds__(1024) void PatchFemKernel(PatchFemArgs a, PatchSweep w, StepConsts k,
                                                       FemConsts fk) {
  extern __shared__ float4 X[];
  const PatchDev p = a.patch[blockIdx.x];
  const LaneOffsets off(a.off + p.off, a.nf + a.nb + 2);
  const int32_t* __restrict__ verts = a.verts + p.vbeg;
  StageVertices(X, w.x, verts, p.n_loc);
  SweepColors(
      off, 0, a.nf, [&](int e) { return StrainEntry{a.frec[e], a.finv[e]}; },
      [&](int, const StrainEntry& s) {
        const StrainC c{Lo16(s.r.x), Hi16(s.r.x), s.r.y, __int_as_float(s.r.z),
                        {s.inv.x, s.inv.y, s.inv.z, s.inv.w}};
        StrainProject(X, c, fk);
      });
  if (k.solve_bending)
    SweepColors(
        off, a.nf + 1, a.nb,
        [&](int e) { return IsoEntry{a.irec[e], a.iK[e], w.iter > 0 ? a.ilam[e] : 0.0f}; },
        [&](int e, IsoEntry& s) {
          IsoProject(X, make_int4(Lo16(s.r.x), Hi16(s.r.x), Lo16(s.r.y), Hi16(s.r.y)), s.K,
                     __int_as_float(s.r.z), &s.lam, w.iter, fk);
          a.ilam[e] = s.lam;
          if (w.last && s.r.w < 0) a.ilam_out[s.r.w & 0x7fffffff] = s.lam;
        });
  WriteOwn<false>(X, w, k, p, verts);
}

__global__ __launch_bounds__(256) void PatchComplianceKernel(const StretchC* __restrict__ sc,
                                                             int4* __restrict__ srec, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) srec[i].z = __float_as_int(sc[srec[i].w & 0x7fffffff].compliance);
}
}  // namespace

hipError_t LaunchPatchSweep(hipStream_t s, const PatchArgs& a, const PatchSweep& w,
                            const StepConsts& k, const BendMode& m, int threads,
                            size_t lds_bytes) {
  if (a.n <= 0) return hipSuccess;
  if (threads < 64 || threads > 1024 || threads % 64) return hipErrorInvalidValue;
  if (w.tape_s)
    PatchSweepKernel<true><<<a.n, threads, lds_bytes, s>>>(a, w, k, m);
  else
    PatchSweepKernel<false><<<a.n, threads, lds_bytes, s>>>(a, w, k, m);
  return hipGetLastError();
}

hipError_t LaunchPatchFem(hipStream_t s, const PatchFemArgs& a, const PatchSweep& w,
                          const StepConsts& k, const FemConsts& fk, int threads,
                          size_t lds_bytes) {
  if (a.n <= 0) return hipSuccess;
  if (threads < 64 || threads > 1024 || threads % 64) return hipErrorInvalidValue;
  PatchFemKernel<<<a.n, threads, lds_bytes, s>>>(a, w, k, fk);
  return hipGetLastError();
}

hipError_t ConfigurePatchSweep(size_t lds_bytes) {
  const void* fns[3] = {reinterpret_cast<const void*>(&PatchSweepKernel<false>),
                        reinterpret_cast<const void*>(&PatchSweepKernel<true>),
                        reinterpret_cast<const void*>(&PatchFemKernel)};
  for (const void* f : fns) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             static_cast<int>(lds_bytes));
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t LaunchPatchCompliance(hipStream_t s, const StretchC* sc, int4* srec, int n) {
  if (n <= 0) return hipSuccess;
  PatchComplianceKernel<<<(n + 255) / 256, 256, 0, s>>>(sc, srec, n);
  return hipGetLastError();
}

}  // namespace xrt
