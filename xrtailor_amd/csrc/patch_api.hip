// The fused constraint sweeps' plan (built on the host at xrt_start) and their launch.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "context.h"
#include "patch.h"
#include "patch_plan.h"

namespace xrt {
namespace {

constexpr int kPatchMaxVerts = 10240;  // 160 KB of LDS
constexpr double kPatchMaxWork = 6.0;  // listed constraints / constraints

// families of an instance: its stretch edges and bend elements in color-sorted order
std::vector<PatchFamily> Families(const HostInstance& h) {
  std::vector<PatchFamily> f(2);
  f[0].arity = 2;
  f[0].coloff = h.s_coloff;
  f[0].cons.resize(2 * static_cast<size_t>(h.ne()));
  for (int p = 0; p < h.ne(); ++p)
    for (int a = 0; a < 2; ++a) f[0].cons[2 * static_cast<size_t>(p) + a] = h.edges[2 * h.s_order[p] + a];
  f[1].arity = 4;
  f[1].coloff = h.b_coloff;
  f[1].cons.resize(4 * static_cast<size_t>(h.nb()));
  for (int p = 0; p < h.nb(); ++p)
    for (int a = 0; a < 4; ++a) f[1].cons[4 * static_cast<size_t>(p) + a] = h.bends[4 * h.b_order[p] + a];
  return f;
}

// fn(0) .. fn(n - 1) on up to 16 threads; false when one returned false or threw (the
// others are then skipped).  Nothing leaves it by exception.
template <class F>
bool ParallelFor(int n, F&& fn) {
  std::atomic<int> next{0};
  std::atomic<bool> ok{true};
  auto work = [&]() {
    try {
      for (int i = next++; i < n && ok; i = next++)
        if (!fn(i)) ok = false;
    } catch (...) {
      ok = false;
    }
  };
  const int nt = std::min({n, 16, static_cast<int>(std::thread::hardware_concurrency())});
  std::vector<std::thread> pool;
  try {
    pool.reserve(std::max(nt, 1));
    for (int t = 1; t < nt; ++t) pool.emplace_back(work);
  } catch (...) {  // fewer helpers than asked for
  }
  work();
  for (auto& t : pool) t.join();
  return ok;
}

}  // namespace

int PatchPrepare(xrt_ctx* ctx) {
  PatchData& P = ctx->patches;
  P.ready = false;
  const int ni = static_cast<int>(ctx->inst.size());
  int ns = 0, nb = 0;
  for (const HostInstance& h : ctx->inst) {
    ns = std::max(ns, h.s_ncol);
    nb = std::max(nb, h.b_ncol);
  }
  if (ns + nb == 0 || ns + nb + 2 > kPatchMaxOffsets) return XRT_OK;
  const int max_local = static_cast<int>(
      std::min<size_t>(kPatchMaxVerts, std::min<size_t>(ctx->max_lds, 160 * 1024) / sizeof(float4)));
  // Own vertices per patch: what gives 4 of 5 CUs a patch, down to 256 vertices, where the
  // ring of neighbors already quadruples the stretch work of a grid, and up to 4096 (a grid's
  // patch then needs 117 KB of LDS, 1.4x the stretch and 1.2x the bend work).  ms per frame at
  // 144 / 256 / 400 / 1024 / 2304 / 4096 own vertices: one 64 x 64 cloth 2.22 / 2.28 / 2.40 /
  // 2.75 / 3.51 / 4.43, 16 garments (93 k vertices) - / 10.3 / 8.25 / 8.66 / 9.67 / 10.5, 256
  // cloths (2.53 M vertices) 115 / 108 / 75 / 44.6 / 29.3 / 23.7.  An instance stays whole
  // (nothing is solved twice) when there are patches enough without cutting it, and below
  // 1200 vertices, where a color takes one or two rounds of one workgroup anyway.
  const int per_cu = ctx->wide.n_total / std::max(1, ctx->cu_count * 4 / 5);
  const int cut = std::min(4096, std::max(256, per_cu)), whole = std::max(1200, per_cu);
  std::vector<std::vector<Patch>> plan(ni);
  const bool built = ParallelFor(ni, [&](int i) {
    const HostInstance& h = ctx->inst[i];
    const std::vector<PatchFamily> fam = Families(h);
    // a mesh with little locality gets larger patches, or none
    for (int target = h.nv <= whole ? h.nv : cut; target < 4 * kPatchMaxVerts; target *= 4)
      if (BuildPatches(h.rest_pos.data(), h.nv, fam, target, max_local, kPatchMaxWork, &plan[i]))
        return true;
    return false;
  });
  if (!built) return XRT_OK;
  std::vector<PatchDev> dev;
  std::vector<int32_t> verts, off, bcon;
  std::vector<int4> srec, brec;
  size_t max_loc = 0, max_color = 0;
  for (int i = 0; i < ni; ++i) {
    const HostInstance& h = ctx->inst[i];
    for (const Patch& q : plan[i]) {
      PatchDev d;
      d.vbeg = static_cast<int32_t>(verts.size());
      d.n_own = q.n_own;
      d.n_loc = static_cast<int32_t>(q.verts.size());
      d.off = static_cast<int32_t>(off.size());
      dev.push_back(d);
      max_loc = std::max(max_loc, q.verts.size());
      for (int32_t v : q.verts) verts.push_back(h.desc.vbeg + v);
      auto offsets = [&](int f, int n, size_t base) {
        for (int c = 0; c <= n; ++c) {
          const int cc = std::min<int>(c, static_cast<int>(q.coloff[f].size()) - 1);
          off.push_back(static_cast<int32_t>(base) + q.coloff[f][cc]);
          if (c > 0) max_color = std::max<size_t>(max_color, off[off.size() - 1] - off[off.size() - 2]);
        }
      };
      offsets(0, ns, srec.size());
      offsets(1, nb, brec.size());
      for (size_t e = 0; e < q.cons[0].size(); ++e) {
        const int p = q.cons[0][e] & 0x7fffffff;
        const int o = h.s_order[p];
        const uint32_t ij = q.local[0][2 * e] | static_cast<uint32_t>(q.local[0][2 * e + 1]) << 16;
        int4 r;
        r.x = static_cast<int>(ij);
        std::memcpy(&r.y, &h.rest_len[o], 4);
        std::memcpy(&r.z, &h.s_comp[o], 4);
        r.w = static_cast<int>(static_cast<uint32_t>(h.sbeg + p) | (q.cons[0][e] & 0x80000000u));
        srec.push_back(r);
      }
      for (size_t e = 0; e < q.cons[1].size(); ++e) {
        const int p = q.cons[1][e] & 0x7fffffff;
        const int o = h.b_order[p];
        const uint16_t* l = &q.local[1][4 * e];
        int4 r;
        r.x = static_cast<int>(l[0] | static_cast<uint32_t>(l[1]) << 16);
        r.y = static_cast<int>(l[2] | static_cast<uint32_t>(l[3]) << 16);
        std::memcpy(&r.z, &h.theta[o], 4);
        std::memcpy(&r.w, &h.b_comp[o], 4);
        brec.push_back(r);
        bcon.push_back(static_cast<int>(static_cast<uint32_t>(h.bbeg + p) | (q.cons[1][e] & 0x80000000u)));
      }
    }
  }
  if (std::max({verts.size(), srec.size(), brec.size()}) > static_cast<size_t>(INT32_MAX)) return XRT_OK;
  hipStream_t s = ctx->stream;
  // block b takes patch b: the patches with most work first, so that the last ones to start are then the short ones (256 cloths: 23.7 ->
  // 21.6 ms per frame)
  {
    auto entries = [&](const PatchDev& d) {  // a bend costs about four stretches
      const int32_t* o = &off[d.off];
      return (o[ns] - o[0]) + 4 * static_cast<int64_t>(o[ns + 1 + nb] - o[ns + 1]);
    };
    std::stable_sort(dev.begin(), dev.end(), [&](const PatchDev& a, const PatchDev& b) {
      return entries(a) > entries(b);
    });
  }
  P.n = static_cast<int>(dev.size());
  P.split = P.n > ni;
  P.ns = ns;
  P.nb = nb;
  P.lds_bytes = sizeof(float4) * max_loc;
  P.threads = static_cast<int>(std::min<size_t>(1024, std::max<size_t>(64, (max_color + 63) / 64 * 64)));
  hipError_t e = P.patch.Upload(dev, s);
  if (e == hipSuccess) e = P.verts.Upload(verts, s);
  if (e == hipSuccess) e = P.off.Upload(off, s);
  if (e == hipSuccess) e = P.srec.Upload(srec, s);
  if (e == hipSuccess) e = P.brec.Upload(brec, s);
  if (e == hipSuccess) e = P.bcon.Upload(bcon, s);
  if (e == hipSuccess) e = P.slam.Alloc(std::max<size_t>(srec.size(), 1));
  if (e == hipSuccess) e = P.alt.Alloc(std::max<size_t>(ctx->x.n, 1));
  if (e != hipSuccess) {  // no memory left for the plan: the colors run as launches of their own
    P.patch.Free();
    P.verts.Free();
    P.off.Free();
    P.srec.Free();
    P.brec.Free();
    P.bcon.Free();
    P.slam.Free();
    P.alt.Free();
    (void)hipGetLastError();
    return e == hipErrorOutOfMemory ? XRT_OK : XRT_ERR_HIP;
  }
  if (P.lds_bytes > 64 * 1024) XRT_CHECK_HIP(ConfigurePatchSweep(P.lds_bytes));
  P.ready = true;
  return XRT_OK;
}

int PatchIter(xrt_ctx* ctx, const StepConsts& k, const BendMode& m, int it, bool ground,
              float4* tape_s, float4* tape_b, float4* tape_g) {
  PatchData& P = ctx->patches;
  PatchArgs a{P.patch.ptr, P.verts.ptr, P.off.ptr, P.srec.ptr, P.slam.ptr, P.brec.ptr, P.bcon.ptr,
              ctx->slam.ptr, P.n, P.ns, P.nb};
  float4* out = ctx->xcur == ctx->x.ptr ? P.alt.ptr : ctx->x.ptr;
  PatchSweep w{ctx->xcur, out, ctx->x0.ptr, it, it + 1 == k.iterations ? 1 : 0, ground ? 1 : 0,
               tape_s, tape_b, tape_g};
  const int threads = ctx->tuning.wide_per_thread == 2 ? std::max(64, (P.threads / 2 + 63) / 64 * 64)
                                                       : P.threads;
  XRT_CHECK_HIP(LaunchPatchSweep(ctx->stream, a, w, k, m, threads, P.lds_bytes));
  ctx->xcur = out;
  return XRT_OK;
}

int PatchRefreshCompliance(xrt_ctx* ctx) {
  PatchData& P = ctx->patches;
  if (!P.ready) return XRT_OK;
  XRT_CHECK_HIP(LaunchPatchCompliance(ctx->stream, ctx->sc.ptr, P.srec.ptr,
                                      static_cast<int>(P.srec.n)));
  return XRT_OK;
}

}  // namespace xrt
