#include "patch.h"

#include "elements.h"

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
  const int tid = threadIdx.x, bs = blockDim.x;
  const LaneOffsets off(a.off + p.off, a.ns + a.nb + 2);
  const int32_t* __restrict__ verts = a.verts + p.vbeg;

  // the entries are walked as (color, round) steps; each step's records are loaded one step
  // ahead, so a color waits for LDS and arithmetic only
  int c = 0, beg = off[0], end = off[1];
  int4 rec = make_int4(0, 0, 0, 0);
  float lam = 0.0f;
  if (a.ns > 0 && beg + tid < end) {
    rec = a.srec[beg + tid];
    if (w.iter > 0) lam = a.slam[beg + tid];
  }
  for (int v0 = tid; v0 < p.n_loc; v0 += 4 * bs) {
    int g[4];
    float4 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) g[u] = v0 + u * bs < p.n_loc ? verts[v0 + u * bs] : verts[v0];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = w.x[g[u]];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (v0 + u * bs < p.n_loc) X[v0 + u * bs] = x[u];
  }
  LdsBarrier();
  while (c < a.ns) {
    const int e = beg + tid;
    const bool more = beg + bs < end;          // another round of this color
    const int nbeg = more ? beg + bs : end;    // (colors lie one after the other)
    const int nend = more ? end : (c + 1 < a.ns ? off[c + 2] : nbeg);
    int4 nrec = make_int4(0, 0, 0, 0);
    float nlam = 0.0f;
    if (nbeg + tid < nend) {
      nrec = a.srec[nbeg + tid];
      if (w.iter > 0) nlam = a.slam[nbeg + tid];
    }
    if (e < end) {
      const int i0 = rec.x & 0xffff, i1 = static_cast<int>(static_cast<uint32_t>(rec.x) >> 16);
      const StretchC sc{i0, i1, __int_as_float(rec.y), __int_as_float(rec.z)};
      float4 xa = X[i0], xb = X[i1];
      if constexpr (kTape) {
        if (rec.w < 0) {
          const int q = rec.w & 0x7fffffff;
          w.tape_s[2 * q] = make_float4(xa.x, xa.y, xa.z, lam);
          w.tape_s[2 * q + 1] = xb;
        }
      }
      if (StretchSolve(xa, xb, sc, lam, k.inv_dt2)) {
        X[i0] = xa;
        X[i1] = xb;
      }
      a.slam[e] = lam;
      if (w.last && rec.w < 0) a.slam_out[rec.w & 0x7fffffff] = lam;
    }
    if (!more) {
      if (nbeg > off[c]) LdsBarrier();  // (nothing to wait for after an empty color)
      ++c;
    }
    beg = nbeg;
    end = nend;
    rec = nrec;
    lam = nlam;
  }
  if (k.solve_bending && a.nb > 0) {
    const int b0 = a.ns + 1;
    c = 0;
    beg = off[b0];
    end = off[b0 + 1];
    rec = make_int4(0, 0, 0, 0);
    if (beg + tid < end) rec = a.brec[beg + tid];
    while (c < a.nb) {
      const int e = beg + tid;
      const bool more = beg + bs < end;
      const int nbeg = more ? beg + bs : end;
      const int nend = more ? end : (c + 1 < a.nb ? off[b0 + c + 2] : nbeg);
      int4 nrec = make_int4(0, 0, 0, 0);
      if (nbeg + tid < nend) nrec = a.brec[nbeg + tid];
      if (e < end) {
        const int i0 = rec.x & 0xffff, i1 = static_cast<int>(static_cast<uint32_t>(rec.x) >> 16);
        const int i2 = rec.y & 0xffff, i3 = static_cast<int>(static_cast<uint32_t>(rec.y) >> 16);
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
        if (BendSolve(x1, x2, x3, x4, make_float2(__int_as_float(rec.z), __int_as_float(rec.w)),
                      k.inv_dt2, m)) {
          X[i0] = x1;
          X[i1] = x2;
          X[i2] = x3;
          X[i3] = x4;
        }
      }
      if (!more) {
        if (nbeg > off[b0 + c]) LdsBarrier();
        ++c;
      }
      beg = nbeg;
      end = nend;
      rec = nrec;
    }
  }
  for (int v = tid; v < p.n_own; v += bs) {
    const int g = verts[v];
    float4 x = X[v];
    if (w.ground) {
      if constexpr (kTape) w.tape_g[g] = x;
      if (x.w > kEps && x.y < k.ground_y) x = GroundVertex(x, w.x0[g], k.ground_y, k.friction);
    }
    w.out[g] = x;
  }
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

hipError_t ConfigurePatchSweep(size_t lds_bytes) {
  const void* fns[2] = {reinterpret_cast<const void*>(&PatchSweepKernel<false>),
                        reinterpret_cast<const void*>(&PatchSweepKernel<true>)};
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
