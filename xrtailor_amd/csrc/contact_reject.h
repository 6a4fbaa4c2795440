// Sign parts of the repulsion's inside tests, and cheap tests that reject most items before
// them.
//
// An edge pair passes only if the common perpendicular of the two lines meets both segments, a
// vertex-face pair only if the vertex projects into the face; VfSigns and EESigns decide that
// by the signs of triple products with normalised directions, all in FP32.  Without the
// normalisations the same signs follow from two products.  With N = ea x eb, q = N.N, d = y0 - x0:
//   a0, a1 ~ p + q, -p   with p = N.(eb x d):  one strict sign only if -q < p < 0
//   b0, b1 ~ r + q, -r   with r = N.(ea x d):  one strict sign only if -q < r < 0
// and for a vertex x against y0, y1, y2 with e1 = y1 - y0, e2 = y2 - y0, N = e1 x e2, d = y0 - x:
//   b2, b1, b0 ~ s, t, q - s - t   with s = N.(d x e1), t = N.(e2 x d): one strict sign only
//   if s > 0, t > 0 and s + t < q
// EeReject / VfReject are true only where a product is beyond its bound by more than E, the
// rounding of both evaluations; NaN or infinite values compare false: nothing is rejected.  With
// u = 2^-24, S = |ea| + |eb| + |d| (no difference of two of the four points is longer), every
// difference off by u relative, a product of three by 6 u, and la = |ea|, lb = |eb|:
//   EE: with m = eb x d (p) or ea x d (r), |N| <= la lb.  EESigns takes a1, b1 as a cross product
//   of length |m| and a0, b0 as one of at most |m| + |N|, off by 6 u S^2, times the normal, off by
//   20 u (unit directions 6 u each); scaled by la lb that is 6 u |N| S^2 + 20 u la lb (|m| + |N|).
//   The products here are off by 9 u la lb |m| + 6 u lb |d| |N| (p, r) and 15 u la lb |N| (q).
//   In all less than u (17 |N| S^2 + 29 la lb |m|); E = u (144 |N| T + 32 L |m|) with L = la^2 + lb^2
//   >= 2 la lb, T = L + |d|^2 >= S^2 / 3 is more than twice that, and 0.01 u L T covers the
//   rounding of |N| >= 1e-3 la lb and of |m| themselves.  The bound shrinks with N and m: edges in
//   one line, two apart on a grid line, are rejected too (with 96 u L T instead, 3.8 % of the items
//   of 256 draped grids stayed open where 1.3 % pass EESigns).
//   VF: the products are off by 16 u la lb S^2 and those of VfSigns, scaled by la lb, by
//   48 u la lb S^2; E = 96 u L T >= 64 u la lb S^2.
// and 1e-30 for products that underflow.
// Both tests also fail where the two directions are parallel, |ua x ub|^2 < 1e-6; they are
// rejected for it below 0.99e-6 (the rounding of both sides is 0.3 %).
// Both are the same test with the two edges exchanged (p and r change places), so one answer
// holds for an edge couple in either order.
// A rejected item costs about 60 instructions instead of 225, and what is left open three
// dependent rounds of gathers more.
#pragma once
#include <cmath>

#include "contact_math.h"

namespace xrt {
namespace cm {

constexpr float kUnit = 1.0f / 16777216.0f;
constexpr float kRejectErr = 192.0f * 0.5f / 16777216.0f;

// within an ulp (the bounds have room for it)
__device__ __forceinline__ float RootUp(float v) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_sqrtf(v);
#else
  return std::sqrt(v);
#endif
}

__device__ __forceinline__ bool EeReject(F3 x0, F3 x1, F3 y0, F3 y1) {
  const F3 ea = S(x1, x0), eb = S(y1, y0), d = S(y0, x0);
  const F3 n = C(ea, eb);
  const float q = D(n, n), la = D(ea, ea), lb = D(eb, eb);
  const F3 mb = C(eb, d), ma = C(ea, d);
  const float l = la + lb, t = l + D(d, d);
  const float e = kUnit * (144.0f * RootUp(q) * t + 0.01f * l * t) + 1e-30f;
  const float f = 32.0f * kUnit * l;
  const float p = D(n, mb), r = D(n, ma);
  const float ep = e + f * RootUp(D(mb, mb)), er = e + f * RootUp(D(ma, ma));
  return p > ep || r > er || p + q < -ep || r + q < -er || q + 1e-30f < 0.99e-6f * la * lb;
}

__device__ __forceinline__ bool VfReject(F3 x, F3 y0, F3 y1, F3 y2) {
  const F3 e1 = S(y1, y0), e2 = S(y2, y0), d = S(y0, x);
  const F3 n = C(e1, e2);
  const float q = D(n, n), la = D(e1, e1), lb = D(e2, e2);
  const float e = kRejectErr * (la + lb) * (la + lb + D(d, d)) + 1e-30f;
  const float s = D(n, C(d, e1)), t = D(n, C(e2, d));
  return s < -e || t < -e || s + t > q + e || q + 1e-30f < 0.99e-6f * la * lb;
}

// The inside test of EvaluateVFProximity on the current state, which rejects most pairs;
// it is evaluated before the start-of-substep side (both are pure, so the order does not
// change any result).  It is SignedVF's weights with an early exit: min(-w1, -w2, -w3) >=
// 1e-6 needs b0, b1, b2 of one strict sign (a NaN or a zero weight cannot pass either), so
// that is checked before the divisions, on the same expressions.  VfSigns is the part
// before the divisions (num receives b0, b1, b2), VfWeights the divisions and the bound.
__device__ __forceinline__ bool VfSigns(int node, int4 tr, bool self, F3 x, F3 y0, F3 y1, F3 y2,
                                        float4& num) {
  if (self && (node == tr.x || node == tr.y || node == tr.z)) return false;
  F3 n = C(Nz(S(y1, y0)), Nz(S(y2, y0)));
  if (D(n, n) < 1e-6f) return false;  // degenerate: weights 0
  n = Nz(n);
  const float b0 = Mixed(S(y1, x), S(y2, x), n);
  const float b1 = Mixed(S(y2, x), S(y0, x), n);
  const float b2 = Mixed(S(y0, x), S(y1, x), n);
  if (!((b0 > 0 && b1 > 0 && b2 > 0) || (b0 < 0 && b1 < 0 && b2 < 0))) return false;
  num = make_float4(b0, b1, b2, 0.0f);
  return true;
}

// EvaluateEEProximity (PBDRepulsion.cu:411-468) of the edges with vertices a (cloth) and
// b (obstacle or cloth); ua, ub: their unit directions in the current state,
// Nz(x_a.y - x_a.x).  The edge ids, ids() = (e0, e1), are needed only by the pairs that
// pass the inside test.
// The inside test of EvaluateEEProximity (PBDRepulsion.cu:411-468) on the current state of
// the edges with vertices a (cloth) and b (obstacle or cloth): x0, x1, y0, y1 are their
// positions, ua, ub their unit directions Nz(x_a.y - x_a.x).  True, with SignedEE's weights
// in bw, when the barycentric part passes; InEdge and the response follow in EEResponse.
// The weights take early exits: an accepted pair has every weight > 0 (a NaN weight fails
// InEdge or leaves another weight <= 0), which needs a0, a1 and b0, b1 each of one strict
// sign, checked before the divisions on the same expressions.  EESigns is the part before
// the divisions (num receives a0, a1, b0, b1), EEWeights the divisions and the lower bound.
__device__ __forceinline__ bool EESigns(int2 a, int2 b, F3 x0, F3 x1, F3 y0, F3 y1, bool self,
                                        F3 ua, F3 ub, float4& num) {
  if (self && (a.x == b.x || a.x == b.y || a.y == b.x || a.y == b.y)) return false;
  const F3 ncur = C(ua, ub);
  if (D(ncur, ncur) < 1e-6f) return false;  // degenerate: weights 0
  const F3 d00 = S(y0, x0), d01 = S(y1, x0), d10 = S(y0, x1), d11 = S(y1, x1);
  const float a0 = Mixed(d11, d10, ncur), a1 = Mixed(d00, d01, ncur);
  if (!((a0 > 0 && a1 > 0) || (a0 < 0 && a1 < 0))) return false;
  // b0 = Mixed(S(x0, y1), S(x1, y1), ncur) and b1 = Mixed(S(x1, y0), S(x0, y0), ncur): both
  // differences negated, which leaves every nonzero result the same bits (rounding is
  // symmetric; only the sign of an exact zero can differ, and zero fails the test either way)
  const float b0 = Mixed(d01, d11, ncur), b1 = Mixed(d10, d00, ncur);
  if (!((b0 > 0 && b1 > 0) || (b0 < 0 && b1 < 0))) return false;
  num = make_float4(a0, a1, b0, b1);
  return true;
}

}  // namespace cm
}  // namespace xrt
