// Device-side LBVH helpers shared by the build / query kernels and the contact kernels
// (header-only: every translation unit inlines its own copy).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "bvh.h"
#include "device.h"

namespace xrt {

constexpr int kMaxHits = 256;  // LBVH_MAX_BUFFER_SIZE (xrtailor/include/xrtailor/core/Common.cuh:24)

// MathFunctions::min / max (xrtailor/include/xrtailor/math/MathFunctions.cuh:24-51)
__device__ __forceinline__ float Mn(float a, float b) { return a < b ? a : b; }
__device__ __forceinline__ float Mx(float a, float b) { return a > b ? a : b; }

__device__ __forceinline__ Box MergeBox(const Box& a, const Box& b) {
  return Box{make_float4(Mn(a.lo.x, b.lo.x), Mn(a.lo.y, b.lo.y), Mn(a.lo.z, b.lo.z), 0.0f),
             make_float4(Mx(a.hi.x, b.hi.x), Mx(a.hi.y, b.hi.y), Mx(a.hi.z, b.hi.z), 0.0f)};
}

// Bounds::Overlap(p): strict containment (xrtailor/src/physics/broad_phase/Bounds.cu:130-136)
__device__ __forceinline__ bool OverlapPoint(const Box& b, float4 p) {
  return p.x > b.lo.x && p.x < b.hi.x && p.y > b.lo.y && p.y < b.hi.y && p.z > b.lo.z &&
         p.z < b.hi.z;
}

__device__ __forceinline__ bool GetIntersection(float d1, float d2, float4 p1, float4 p2,
                                                float4& hit) {  // Bounds.cu:139-147
  if ((d1 * d2) >= 0.0f) return false;
  if (d1 == d2) return false;
  const float s = -d1 / (d2 - d1);
  hit = make_float4(p1.x + (p2.x - p1.x) * s, p1.y + (p2.y - p1.y) * s, p1.z + (p2.z - p1.z) * s,
                    0.0f);
  return true;
}

__device__ __forceinline__ bool InBox(float4 h, const Box& b, int axis) {  // Bounds.cu:149-158
  if (axis == 1 && h.z > b.lo.z && h.z < b.hi.z && h.y > b.lo.y && h.y < b.hi.y) return true;
  if (axis == 2 && h.z > b.lo.z && h.z < b.hi.z && h.x > b.lo.x && h.x < b.hi.x) return true;
  if (axis == 3 && h.x > b.lo.x && h.x < b.hi.x && h.y > b.lo.y && h.y < b.hi.y) return true;
  return false;
}

// Bounds::Overlap(p1, p2, hit): segment vs box (Bounds.cu:160-191)
__device__ __forceinline__ bool OverlapSegment(const Box& b, float4 p1, float4 p2) {
  if (p2.x < b.lo.x && p1.x < b.lo.x) return false;
  if (p2.x > b.hi.x && p1.x > b.hi.x) return false;
  if (p2.y < b.lo.y && p1.y < b.lo.y) return false;
  if (p2.y > b.hi.y && p1.y > b.hi.y) return false;
  if (p2.z < b.lo.z && p1.z < b.lo.z) return false;
  if (p2.z > b.hi.z && p1.z > b.hi.z) return false;
  if (OverlapPoint(b, p1)) return true;
  float4 h;
  return (GetIntersection(p1.x - b.lo.x, p2.x - b.lo.x, p1, p2, h) && InBox(h, b, 1)) ||
         (GetIntersection(p1.y - b.lo.y, p2.y - b.lo.y, p1, p2, h) && InBox(h, b, 2)) ||
         (GetIntersection(p1.z - b.lo.z, p2.z - b.lo.z, p1, p2, h) && InBox(h, b, 3)) ||
         (GetIntersection(p1.x - b.hi.x, p2.x - b.hi.x, p1, p2, h) && InBox(h, b, 1)) ||
         (GetIntersection(p1.y - b.hi.y, p2.y - b.hi.y, p1, p2, h) && InBox(h, b, 2)) ||
         (GetIntersection(p1.z - b.hi.z, p2.z - b.hi.z, p1, p2, h) && InBox(h, b, 3));
}

// Bounds::Overlap(b, thickness) = Overlap(b.Dilate(thickness)) (Bounds.cu:96-128)
__device__ __forceinline__ bool OverlapDilated(const Box& rhs, const Box& lhs, float th) {
  const float lx = lhs.lo.x - th, ly = lhs.lo.y - th, lz = lhs.lo.z - th;
  const float hx = lhs.hi.x + th, hy = lhs.hi.y + th, hz = lhs.hi.z + th;
  if (rhs.lo.x > hx || rhs.hi.x < lx) return false;
  if (rhs.lo.y > hy || rhs.hi.y < ly) return false;
  if (rhs.lo.z > hz || rhs.hi.z < lz) return false;
  return true;
}

// ------------------------------------------------------------------------------------
// Per-element bodies of the refit / traversal kernels, shared by the single-tree kernels
// (bvh.hip) and the multi-instance ones (contact.hip) so both run the same arithmetic.

// RefitExternalNodeMidstep (BVH.cu:770-818) / Update: pred = x1 + tol n1 (or x)
__device__ __forceinline__ void RefitPredBody(const float4* __restrict__ x1,
                                              const float4* __restrict__ n1, float tol, int i,
                                              float4* __restrict__ pred) {
  const float4 p = x1[i];
  if (n1) {
    const float4 n = n1[i];
    pred[i] = make_float4(p.x + tol * n.x, p.y + tol * n.y, p.z + tol * n.z, 0.0f);
  } else {
    pred[i] = make_float4(p.x, p.y, p.z, 0.0f);
  }
}

// leaf i's box, grown by its 3 corners of pa (midstep) or by Face::ComputeBounds(ccd) of pa
// [and pb]
__device__ __forceinline__ Box GrownLeaf(const BvhView& t, const float4* pa, const float4* pb, int i) {
  const int ni = t.nf - 1;
  const int4 f = t.tris[t.nodes[ni + i].w];
  const Box b = t.box[ni + i];
  float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
  float4 hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
  const int vid[3] = {f.x, f.y, f.z};
  for (int c = 0; c < 3; ++c) {
    const float4 p = pa[vid[c]];
    lo.x = Mn(lo.x, p.x); lo.y = Mn(lo.y, p.y); lo.z = Mn(lo.z, p.z);
    hi.x = Mx(hi.x, p.x); hi.y = Mx(hi.y, p.y); hi.z = Mx(hi.z, p.z);
    if (pb) {
      const float4 q = pb[vid[c]];
      lo.x = Mn(lo.x, q.x); lo.y = Mn(lo.y, q.y); lo.z = Mn(lo.z, q.z);
      hi.x = Mx(hi.x, q.x); hi.y = Mx(hi.y, q.y); hi.z = Mx(hi.z, q.z);
    }
  }
  return MergeBox(b, Box{lo, hi});
}

// A node's box and its traversal record: the box with lo.w = left child (internal node) or
// -(object + 1) (leaf) and hi.w = escape, so that one 32-byte load serves a visit.  Every merge
// writes both, so the records are current whenever the boxes are.
__device__ __forceinline__ void StoreNode(const BvhView& t, int node, Box b, int code, int escape) {
  t.box[node] = b;
  b.lo.w = __int_as_float(code);
  b.hi.w = __int_as_float(escape);
  t.packed[node] = b;
}

// Boxes of the internal nodes from the leaves up, in two launches.
//
// An internal node of the radix tree covers a contiguous range of leaves and has the number of
// one end of it.  So a workgroup that takes kMergeChunk consecutive leaves can merge every
// node whose range lies within them out of LDS: the second child to arrive at a node (a
// counter in LDS) merges the two.  What is left are the nodes over chunk boundaries, a few
// percent; one workgroup per tree merges them the same way through L2 (MergeTop), starting
// from the roots of the chunks' subtrees, which MergeChunk lists in t.lvl (chunk c's at
// [kMergeChunk c ..), their number at nf + c).  The boxes are unions (min / max), so the
// order of the merges changes nothing; a leaf that only grows keeps every old box inside
// the new one.  One workgroup merging a whole tree depth by depth (as before) took 716 us for
// the 130,050 faces of a 256 x 256 cloth and a climb over all leaves with device-wide fences
// 435 us for 64,082; the two launches take 256 us and 89 us.
constexpr int kMergeChunk = 1024;  // leaves per workgroup, one per thread

struct MergeShared {
  float box[6][2 * kMergeChunk];  // leaves of the chunk, then its internal nodes
  int parent[kMergeChunk], left[kMergeChunk], right[kMergeChunk], escape[kMergeChunk];
  int count[kMergeChunk];
  int roots;
};

// leaf_box(i): the box of leaf slot i (called once per leaf); a workgroup of kMergeChunk threads
template <class LeafBox>
__device__ __forceinline__ void MergeChunk(const BvhView& t, int chunk, MergeShared& m,
                                           LeafBox&& leaf_box) {
  const int nf = t.nf, ni = nf - 1, cb = chunk * kMergeChunk;
  const int tid = threadIdx.x, i = cb + tid;
  if (i < ni) {
    const int4 nd = t.nodes[i];
    m.parent[tid] = nd.x;
    m.left[tid] = nd.y;
    m.right[tid] = nd.z;
    m.escape[tid] = t.escape[i];
    t.flags[i] = 0;
  }
  m.count[tid] = 0;
  if (tid == 0) m.roots = 0;
  auto put = [&](int k, const Box& b) {
    m.box[0][k] = b.lo.x; m.box[1][k] = b.lo.y; m.box[2][k] = b.lo.z;
    m.box[3][k] = b.hi.x; m.box[4][k] = b.hi.y; m.box[5][k] = b.hi.z;
  };
  auto get = [&](int k) {
    return Box{make_float4(m.box[0][k], m.box[1][k], m.box[2][k], 0.0f),
               make_float4(m.box[3][k], m.box[4][k], m.box[5][k], 0.0f)};
  };
  int node = ni + i, p = -1;
  if (i < nf) {
    const int4 nd = t.nodes[node];
    p = nd.x;
    const Box b = leaf_box(i);
    StoreNode(t, node, b, -(nd.w + 1), t.escape[node]);
    put(tid, b);
  }
  __syncthreads();
  int stop = -1, at = -1;  // the node this thread stopped with, the parent it waits at (-1: outside)
  while (p >= 0) {         // (a climb passes each node of the chunk at most once)
    const int lp = p - cb;
    if (lp < 0 || lp >= kMergeChunk) {
      stop = node;
      break;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    const int old = atomicAdd(&m.count[lp], 1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (old == 0) {
      stop = node;
      at = lp;
      break;
    }
    // a child is a leaf (number ni + slot) or an internal node, of this chunk either way
    const int l = m.left[lp], r = m.right[lp];
    const Box b = MergeBox(get(l >= ni ? l - ni - cb : kMergeChunk + l - cb),
                           get(r >= ni ? r - ni - cb : kMergeChunk + r - cb));
    put(kMergeChunk + lp, b);
    StoreNode(t, p, b, l, m.escape[lp]);
    node = p;
    p = m.parent[lp];
  }
  __syncthreads();
  // stopped for good where no second child of this chunk arrived
  if (stop >= 0 && (at < 0 || m.count[at] == 1)) t.lvl[cb + atomicAdd(&m.roots, 1)] = stop;
  __syncthreads();
  if (tid == 0) t.lvl[nf + chunk] = m.roots;
}

// The nodes over chunk boundaries, by one workgroup of 1024 threads after every chunk of the tree.
// A chunk lists some 20 roots and every climb is a chain of L2 round trips, so the roots of 1024
// chunks at a time are numbered through and taken by all threads (a wave per chunk left two
// thirds of the lanes idle and took 231 us for 130 k faces, this 76 us).
__device__ __forceinline__ void MergeTop(const BvhView& t) {
  const int nf = t.nf, ni = nf - 1;
  const int chunks = (nf + kMergeChunk - 1) / kMergeChunk;
  if (chunks <= 1) return;
  __shared__ int start[1024], wave_sum[16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int c0 = 0; c0 < chunks; c0 += 1024) {
    const int n = c0 + tid < chunks ? t.lvl[nf + c0 + tid] : 0;
    int inc = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(inc, d, 64);
      if (lane >= d) inc += v;
    }
    __syncthreads();  // the last round's readers of start and wave_sum are done
    if (lane == 63) wave_sum[w] = inc;
    __syncthreads();
    int before = 0, total = 0;
    for (int j = 0; j < 16; ++j) {
      before += j < w ? wave_sum[j] : 0;
      total += wave_sum[j];
    }
    start[tid] = before + inc - n;
    __syncthreads();
    for (int r = tid; r < total; r += 1024) {
      int c = 0;  // the last chunk that starts at or before r (empty ones start with their next)
#pragma unroll
      for (int step = 512; step > 0; step >>= 1)
        if (start[c + step] <= r) c += step;
      int node = t.lvl[(c0 + c) * kMergeChunk + (r - start[c])];
      Box b = t.box[node];
      int p = t.nodes[node].x;
      for (int level = 0; p >= 0 && p < ni && level < nf; ++level) {
        const int4 nd = t.nodes[p];  // on their way during the atomic
        const int esc = t.escape[p];
        __threadfence_block();
        if (atomicAdd(&t.flags[p], 1) == 0) break;
        __threadfence_block();
        const bool left = nd.y == node;  // the other child's box is the one load left
        const Box other = t.box[left ? nd.z : nd.y];
        b = left ? MergeBox(b, other) : MergeBox(other, b);
        StoreNode(t, p, b, nd.y, esc);
        node = p;
        p = nd.x;
      }
    }
  }
}

// the stackless pair traversal (CountPairs_Kernel / FindPairs_Kernel, BVH.cu:1149-1227) over
// the traversal records: on_leaf(rhs object) for every rhs leaf overlapping lb dilated by th
template <class OnLeaf>
__device__ __forceinline__ void TraversePacked(const Box* __restrict__ pk, int nf, const Box& lb,
                                               float th, OnLeaf&& on_leaf) {
  int node = 0;
  const int max_steps = 2 * nf;  // each node is visited at most once
  for (int step = 0; node != -1 && step < max_steps; ++step) {
    const Box b = pk[node];
    const int code = __float_as_int(b.lo.w), esc = __float_as_int(b.hi.w);
    if (OverlapDilated(b, lb, th)) {
      if (code < 0) {
        on_leaf(-code - 1);
        node = esc;
      } else {
        node = code;
      }
    } else {
      node = esc;
    }
  }
}

// TraversePacked with the face record of every leaf slot (lf[j], leaf node nf - 1 + j)
// loaded beside the node's record, so a hit's face data costs no dependent load:
// on_leaf(rhs object, its face record) in the same order
template <class OnLeaf>
__device__ __forceinline__ void TraversePackedFace(const Box* __restrict__ pk,
                                                   const int4* __restrict__ lf, int nf,
                                                   const Box& lb, float th, OnLeaf&& on_leaf) {
  const int ni = nf - 1;
  int node = 0;
  const int max_steps = 2 * nf;
  for (int step = 0; node != -1 && step < max_steps; ++step) {
    const Box b = pk[node];
    const int4 f = node >= ni ? lf[node - ni] : make_int4(0, 0, 0, 0);
    const int code = __float_as_int(b.lo.w), esc = __float_as_int(b.hi.w);
    if (OverlapDilated(b, lb, th)) {
      if (code < 0) {
        on_leaf(-code - 1, f);
        node = esc;
      } else {
        node = code;
      }
    } else {
      node = esc;
    }
  }
}

// A tree against itself, each couple of leaves once: lb is the record of leaf slot `slot`, and
// the traversal enters at its escape, where the depth-first order goes on to the leaves of
// higher slots.  on_leaf(rhs object, its face record, fwd, rev) for every such leaf that
// TraversePackedFace would report for lb (fwd) or would report lb for (rev).  The two differ
// only by the rounding of the dilation, so the nodes are tested with a box grown by more than
// that rounding, and the exact tests are made at the leaves that are left.
template <class OnLeaf>
__device__ __forceinline__ void TraversePackedAfter(const Box* __restrict__ pk,
                                                    const int4* __restrict__ lf, int nf,
                                                    const Box& lb, float th, OnLeaf&& on_leaf) {
  const int ni = nf - 1;
  constexpr float kUlps = 4.76837158203125e-7f;  // 2^-21
  Box wide = lb;
  wide.lo.x -= kUlps * (fabsf(lb.lo.x) + fabsf(th));
  wide.lo.y -= kUlps * (fabsf(lb.lo.y) + fabsf(th));
  wide.lo.z -= kUlps * (fabsf(lb.lo.z) + fabsf(th));
  wide.hi.x += kUlps * (fabsf(lb.hi.x) + fabsf(th));
  wide.hi.y += kUlps * (fabsf(lb.hi.y) + fabsf(th));
  wide.hi.z += kUlps * (fabsf(lb.hi.z) + fabsf(th));
  int node = __float_as_int(lb.hi.w);
  const int max_steps = 2 * nf;
  for (int step = 0; node != -1 && step < max_steps; ++step) {
    const Box b = pk[node];
    const int4 f = node >= ni ? lf[node - ni] : make_int4(0, 0, 0, 0);
    const int code = __float_as_int(b.lo.w), esc = __float_as_int(b.hi.w);
    if (OverlapDilated(b, wide, th)) {
      if (code < 0) {
        const bool fwd = OverlapDilated(b, lb, th), rev = OverlapDilated(lb, b, th);
        if (fwd || rev) on_leaf(-code - 1, f, fwd, rev);
        node = esc;
      } else {
        node = code;
      }
    } else {
      node = esc;
    }
  }
}

// CountPairs_Kernel (BVH.cu:1149-1179): rhs leaves overlapping lhs leaf id dilated by th
__device__ __forceinline__ uint32_t CountPairsBody(const BvhView& l, const BvhView& r, float th,
                                                   int id) {
  uint32_t c = 0;
  TraversePacked(r.packed, r.nf, l.packed[l.nf - 1 + id], th, [&](int) { ++c; });
  return c;
}

// FindPairs_Kernel (BVH.cu:1189-1227): leaf id's pairs fill [lo, lo + n) backwards; only
// slots below cap are written
__device__ __forceinline__ void FindPairsBody(const BvhView& l, const BvhView& r, float th, int id,
                                              int64_t lo, uint32_t n, int2* __restrict__ pairs,
                                              int64_t cap) {
  const Box lb = l.packed[l.nf - 1 + id];
  const int lobj = -__float_as_int(lb.lo.w) - 1;
  int64_t index = lo + n - 1;
  TraversePacked(r.packed, r.nf, lb, th, [&](int robj) {
    if (index >= lo && index < cap) pairs[index] = make_int2(lobj, robj);
    --index;
  });
}

// UpdateNodeNormals (xrtailor/src/physics/PhysicsMeshHelper.cu:196-210,282-295) for vertex
// v as a gather over a corner CSR in ascending face order (deterministic)
__device__ __forceinline__ float4 VertexNormalBody(const float4* __restrict__ x,
                                                   const int4* __restrict__ tris,
                                                   const int32_t* __restrict__ vptr,
                                                   const int32_t* __restrict__ corner, int v) {
  float sx = 0.0f, sy = 0.0f, sz = 0.0f;
  for (int k = vptr[v]; k < vptr[v + 1]; ++k) {
    const int c = corner[k];
    const int4 t = tris[c / 3];
    const int j = c % 3;
    const int a = j == 0 ? t.x : (j == 1 ? t.y : t.z);
    const int b = j == 0 ? t.y : (j == 1 ? t.z : t.x);
    const int d = j == 0 ? t.z : (j == 1 ? t.x : t.y);
    const float4 p = x[a], pb = x[b], pd = x[d];
    const float e0x = pb.x - p.x, e0y = pb.y - p.y, e0z = pb.z - p.z;
    const float e1x = pd.x - p.x, e1y = pd.y - p.y, e1z = pd.z - p.z;
    const float den = (e0x * e0x + e0y * e0y + e0z * e0z) * (e1x * e1x + e1y * e1y + e1z * e1z);
    const float cx = e0y * e1z - e0z * e1y, cy = e0z * e1x - e0x * e1z, cz = e0x * e1y - e0y * e1x;
    sx = sx + cx / den;
    sy = sy + cy / den;
    sz = sz + cz / den;
  }
  const float l = sqrtf(sx * sx + sy * sy + sz * sz);
  return make_float4(sx / l, sy / l, sz / l, 0.0f);
}

// ------------------------------------------------------------ radix sort bodies
// (256-thread workgroups; a tile of kSortTile keys per workgroup)
constexpr int kSortBlock = 256;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortBlock * kSortItems;

// Stable LSD radix sort of (key, value), 8-bit digits: per-tile histograms, one
// exclusive scan over the digit-major table, then a scatter whose in-tile ranks come
// from wave64 ballots (lanes with equal digits), so equal keys keep their input order.
__device__ __forceinline__ void RadixHistBody(const uint32_t* __restrict__ keys, int n, int shift,
                                              int nblocks, uint32_t* __restrict__ hist, int blk) {
  __shared__ uint32_t cnt[256];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const int base = blk * kSortTile;
  for (int r = 0; r < kSortItems; ++r) {
    const int i = base + r * kSortBlock + threadIdx.x;
    if (i < n) atomicAdd(&cnt[(keys[i] >> shift) & 255u], 1u);
  }
  __syncthreads();
  hist[threadIdx.x * nblocks + blk] = cnt[threadIdx.x];
}

__device__ __forceinline__ void RadixScatterBody(
    const uint32_t* __restrict__ kin, const int32_t* __restrict__ vin, uint32_t* __restrict__ kout,
    int32_t* __restrict__ vout, int n, int shift, int nblocks, const uint32_t* __restrict__ offs,
    int blk) {
  __shared__ uint32_t run[256];
  __shared__ uint32_t wc[kSortBlock / 64][256];
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  run[t] = offs[t * nblocks + blk];
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int base = blk * kSortTile;
  for (int r = 0; r < kSortItems; ++r) {
    for (int k = 0; k < kSortBlock / 64; ++k) wc[k][t] = 0u;
    __syncthreads();
    const int i = base + r * kSortBlock + t;
    const bool valid = i < n;
    const uint32_t key = valid ? kin[i] : 0u;
    const uint32_t d = (key >> shift) & 255u;
    uint64_t peers = __ballot(valid);
    for (int bit = 0; bit < 8; ++bit) {
      const uint64_t bb = __ballot(valid && ((d >> bit) & 1u));
      peers &= ((d >> bit) & 1u) ? bb : ~bb;
    }
    const uint32_t rank = static_cast<uint32_t>(__popcll(peers & lt));
    if (valid && (peers & lt) == 0) wc[w][d] = static_cast<uint32_t>(__popcll(peers));
    __syncthreads();
    {  // per digit: ordered prefix over the waves of this round
      uint32_t acc = run[t];
      for (int k = 0; k < kSortBlock / 64; ++k) {
        const uint32_t c = wc[k][t];
        wc[k][t] = acc;
        acc += c;
      }
      run[t] = acc;
    }
    __syncthreads();
    if (valid) {
      const uint32_t pos = wc[w][d] + rank;
      if (pos < static_cast<uint32_t>(n)) {  // always true when histogram and scatter agree
        kout[pos] = key;
        vout[pos] = vin[i];
      }
    }
    __syncthreads();
  }
}

// exclusive scan of n uint32 in place by one 1024-thread workgroup; *total (if given)
// receives the sum.  4096 elements a step, neighboring threads on neighboring elements: a
// contiguous run per thread took 33 us a scan of a 64 k face tree's sort and pair counts, this
// 11 us.
__device__ __forceinline__ void BlockExclusiveScan(uint32_t* __restrict__ a, int n,
                                                   int32_t* __restrict__ total) {
  constexpr int kRows = 4, kWaves = 16;
  __shared__ uint32_t sums[kRows * kWaves];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  uint32_t carry = 0;
  for (int base = 0; base < n; base += kRows * 1024) {
    uint32_t v[kRows], inc[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int i = base + r * 1024 + t;
      v[r] = inc[r] = i < n ? a[i] : 0u;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        const uint32_t u = __shfl_up(inc[r], d, 64);
        if (lane >= d) inc[r] += u;
      }
    if (lane == 63)
#pragma unroll
      for (int r = 0; r < kRows; ++r) sums[r * kWaves + w] = inc[r];
    __syncthreads();
    // every wave scans the 64 sums for itself, in the order of the elements
    const uint32_t own = sums[lane];
    uint32_t scan = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t u = __shfl_up(scan, d, 64);
      if (lane >= d) scan += u;
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int i = base + r * 1024 + t;
      const uint32_t before = __shfl(scan - own, r * kWaves + w, 64);
      if (i < n) a[i] = carry + before + inc[r] - v[r];
    }
    carry += __shfl(scan, 63, 64);
    __syncthreads();  // sums is written again
  }
  if (t == 1023 && total) *total = static_cast<int32_t>(carry);
}

// QueryDeviceStackless (xrtailor/src/physics/broad_phase/lbvh/BVH.cu:957-1021): visits the
// leaves whose boxes contain p (segment == false) or meet segment p->q, in traversal order,
// calling f(object) for at most kMaxHits of them; one traversal record per visit.
template <bool kSegment, class F>
__device__ __forceinline__ int StacklessQuery(const Box* __restrict__ pk, int nf, float4 p,
                                                    float4 q, F&& f) {
  int node = 0, found = 0;
  const int max_steps = 2 * nf;
  for (int step = 0; node != -1 && step < max_steps; ++step) {
    if (found >= kMaxHits) break;
    const Box bx = pk[node];
    const int code = __float_as_int(bx.lo.w), esc = __float_as_int(bx.hi.w);
    const bool hit = kSegment ? OverlapSegment(bx, p, q) : OverlapPoint(bx, p);
    if (hit) {
      if (code < 0) {
        f(-code - 1);
        ++found;
        node = esc;
      } else {
        node = code;
      }
    } else {
      node = esc;
    }
  }
  return found;
}

}  // namespace xrt
