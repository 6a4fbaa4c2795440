// The fused constraint sweeps' plan (built on the host at xrt_start) and their launch.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <new>
#include <thread>

#include "context.h"
#include "adjoint.h"
#include "patch.h"
#include "patch_plan.h"

namespace xrt {
namespace {

constexpr size_t kPatchMaxLds = 160 * 1024;
constexpr int kPatchMaxVerts = kPatchMaxLds / sizeof(float4);
constexpr double kPatchMaxWork = 6.0;  // listed constraints / constraints

// constraints of `arity` vertices in sorted order: position p is cons[order[p]]
PatchFamily Family(int arity, const std::vector<int32_t>& cons, const std::vector<int32_t>& order,
                   const std::vector<int32_t>& coloff) {
  PatchFamily f;
  f.arity = arity;
  f.coloff = coloff;
  f.cons.resize(order.size() * arity);
  for (size_t p = 0; p < order.size(); ++p)
    std::copy_n(&cons[static_cast<size_t>(order[p]) * arity], arity, &f.cons[p * arity]);
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

int Pack16(int a, int b) { return static_cast<int>(static_cast<uint32_t>(a) | static_cast<uint32_t>(b) << 16); }
int Bits(float v) {
  int r;
  std::memcpy(&r, &v, 4);
  return r;
}
// constraint position p of a patch (bit 31: owned) as an index over all instances
int Global(int p, int beg) {
  return static_cast<int>((static_cast<uint32_t>(p & 0x7fffffff) + static_cast<uint32_t>(beg)) |
                          (static_cast<uint32_t>(p) & 0x80000000u));
}

// The plan of every instance from its two families; entry0 / entry1 (instance, position with
// the owner bit, local indices) append one entry's records.  True with D filled (on the
// host side in `dev`, `verts`, `off`), false when there is no plan, for want of host memory too.
struct HostPlan {
  std::vector<PatchDev> dev;
  std::vector<int32_t> verts, off;
};
template <class Families, class Entry0, class Entry1>
bool MakePlan(xrt_ctx* ctx, int c0, int c1, Families&& families, Entry0&& entry0, Entry1&& entry1,
              PatchPlanDev& D, HostPlan& H, size_t vert_bytes = sizeof(float4),
              bool hinges_first = false) try {
  if (c0 + c1 == 0 || c0 + c1 + 2 > kPatchMaxOffsets) return false;
  const int ni = static_cast<int>(ctx->inst.size());
  const int max_local = static_cast<int>(
      std::min<size_t>(kPatchMaxVerts, std::min<size_t>(ctx->max_lds, kPatchMaxLds) / vert_bytes));
  const PatchSizes sizes = ChoosePatchSizes(ctx->wide.n_total, ctx->cu_count);
  std::vector<std::vector<Patch>> plan(ni);
  const bool built = ParallelFor(ni, [&](int i) {
    const HostInstance& h = ctx->inst[i];
    const std::vector<PatchFamily> fam = families(i);
    return CutInstance(h.rest_pos.data(), h.nv, fam, sizes, max_local, kPatchMaxWork, &plan[i]);
  });
  if (!built) return false;
  size_t max_loc = 0, n0 = 0, n1 = 0;
  int max_color = 0;
  for (int i = 0; i < ni; ++i) {
    for (const Patch& q : plan[i]) {
      PatchDev d;
      d.vbeg = static_cast<int32_t>(H.verts.size());
      d.n_own = q.n_own;
      d.n_loc = static_cast<int32_t>(q.verts.size());
      d.off = static_cast<int32_t>(H.off.size());
      d.inst = i;
      H.dev.push_back(d);
      max_loc = std::max(max_loc, q.verts.size());
      for (int32_t v : q.verts) H.verts.push_back(ctx->inst[i].desc.vbeg + v);
      for (int f = 0; f < 2; ++f) {
        const size_t base = f == 0 ? n0 : n1;
        if (base + q.cons[f].size() > static_cast<size_t>(INT32_MAX)) return false;
        for (int c = 0; c <= (f == 0 ? c0 : c1); ++c) {
          const int cc = std::min<int>(c, static_cast<int>(q.coloff[f].size()) - 1);
          H.off.push_back(static_cast<int32_t>(base) + q.coloff[f][cc]);
          if (c > 0) max_color = std::max(max_color, H.off.back() - H.off[H.off.size() - 2]);
        }
      }
      const int a0 = q.cons[0].empty() ? 0 : static_cast<int>(q.local[0].size() / q.cons[0].size());
      const int a1 = q.cons[1].empty() ? 0 : static_cast<int>(q.local[1].size() / q.cons[1].size());
      for (size_t e = 0; e < q.cons[0].size(); ++e) entry0(i, q.cons[0][e], &q.local[0][a0 * e]);
      for (size_t e = 0; e < q.cons[1].size(); ++e) entry1(i, q.cons[1][e], &q.local[1][a1 * e]);
      n0 += q.cons[0].size();
      n1 += q.cons[1].size();
    }
    plan[i].clear();
    plan[i].shrink_to_fit();
  }
  if (H.verts.size() > static_cast<size_t>(INT32_MAX)) return false;
  // block b takes patch b: the patches with most work first, so that the last ones to start
  // are the short ones (256 cloths: 23.7 -> 21.6 ms per frame)
  auto entries = [&](const PatchDev& d) {  // a hinge costs about four edges
    const int32_t* o = &H.off[d.off];
    const int64_t n0 = o[c0] - o[0], n1 = o[c0 + 1 + c1] - o[c0 + 1];
    return hinges_first ? 4 * n0 + n1 : n0 + 4 * n1;
  };
  std::stable_sort(H.dev.begin(), H.dev.end(), [&](const PatchDev& a, const PatchDev& b) {
    return entries(a) > entries(b);
  });
  D.n = static_cast<int>(H.dev.size());
  D.split = D.n > ni;
  D.c0 = c0;
  D.c1 = c1;
  D.lds_bytes = vert_bytes * max_loc;
  D.threads = std::min(1024, std::max(64, (max_color + 63) / 64 * 64));
  return true;
} catch (const std::bad_alloc&) {
  return false;
}

hipError_t UploadPlan(xrt_ctx* ctx, PatchPlanDev& D, const HostPlan& H) {
  hipError_t e = D.patch.Upload(H.dev, ctx->stream);
  if (e == hipSuccess) e = D.verts.Upload(H.verts, ctx->stream);
  if (e == hipSuccess) e = D.off.Upload(H.off, ctx->stream);
  if (e == hipSuccess && !ctx->patches.alt.ptr) e = ctx->patches.alt.Alloc(std::max<size_t>(ctx->x.n, 1));
  return e;
}

// a plan whose buffers did not fit is dropped: the colors then run as launches of their own
template <class... Bufs>
int FinishPlan(PatchPlanDev& D, hipError_t e, hipError_t (*configure)(size_t), Bufs&... bufs) {
  if (e == hipSuccess && D.lds_bytes > 64 * 1024) e = configure(kPatchMaxLds);
  if (e == hipSuccess) {
    D.ready = true;
    return XRT_OK;
  }
  (bufs.Free(), ...);
  D.patch.Free();
  D.verts.Free();
  D.off.Free();
  (void)hipGetLastError();
  if (e == hipErrorOutOfMemory) return XRT_OK;
  SetError(std::string("constraint sweep plan: ") + hipGetErrorString(e));
  return XRT_ERR_HIP;
}

}  // namespace

int PatchPrepare(xrt_ctx* ctx) {
  PatchData& P = ctx->patches;
  P.xpbd.ready = false;
  P.xpbd.tried = true;
  int ns = 0, nb = 0;
  for (const HostInstance& h : ctx->inst) {
    ns = std::max(ns, h.s_ncol);
    nb = std::max(nb, h.b_ncol);
  }
  HostPlan H;
  std::vector<int4> srec, brec;
  std::vector<int32_t> bcon;
  const bool made = MakePlan(
      ctx, ns, nb,
      [&](int i) {
        const HostInstance& h = ctx->inst[i];
        return std::vector<PatchFamily>{Family(2, h.edges, h.s_order, h.s_coloff),
                                        Family(4, h.bends, h.b_order, h.b_coloff)};
      },
      [&](int i, int p, const uint16_t* l) {
        const HostInstance& h = ctx->inst[i];
        const int o = h.s_order[p & 0x7fffffff];
        srec.push_back(make_int4(Pack16(l[0], l[1]), Bits(h.rest_len[o]), Bits(h.s_comp[o]),
                                 Global(p, h.sbeg)));
      },
      [&](int i, int p, const uint16_t* l) {
        const HostInstance& h = ctx->inst[i];
        const int o = h.b_order[p & 0x7fffffff];
        brec.push_back(make_int4(Pack16(l[0], l[1]), Pack16(l[2], l[3]), Bits(h.theta[o]),
                                 Bits(h.b_comp[o])));
        bcon.push_back(Global(p, h.bbeg));
      },
      P.xpbd, H);
  if (!made) return XRT_OK;
  hipStream_t s = ctx->stream;
  hipError_t e = UploadPlan(ctx, P.xpbd, H);
  if (e == hipSuccess) e = P.srec.Upload(srec, s);
  if (e == hipSuccess) e = P.brec.Upload(brec, s);
  if (e == hipSuccess) e = P.bcon.Upload(bcon, s);
  if (e == hipSuccess) e = P.slam.Alloc(std::max<size_t>(srec.size(), 1));
  return FinishPlan(P.xpbd, e, ConfigurePatchSweep, P.srec, P.brec, P.bcon, P.slam);
}

int PatchPrepareFem(xrt_ctx* ctx) {
  PatchData& P = ctx->patches;
  const FemData& F = ctx->fem;
  P.fem.ready = false;
  P.fem.tried = true;
  int nf = 0, nb = 0;
  for (size_t i = 0; i < ctx->inst.size(); ++i) {
    nf = std::max(nf, F.inst[i].ncol);
    nb = std::max(nb, ctx->inst[i].b_ncol);
  }
  HostPlan H;
  std::vector<int4> frec, irec;
  std::vector<float4> finv, iK;
  const bool made = MakePlan(
      ctx, nf, nb,
      [&](int i) {
        const HostInstance& h = ctx->inst[i];
        return std::vector<PatchFamily>{Family(3, h.tris, F.inst[i].order, F.inst[i].coloff),
                                        Family(4, h.bends, h.b_order, h.b_coloff)};
      },
      [&](int i, int p, const uint16_t* l) {
        const StrainC& c = F.host_sc[F.inst[i].fbeg + (p & 0x7fffffff)];
        frec.push_back(make_int4(Pack16(l[0], l[1]), l[2], Bits(c.area), 0));
        finv.push_back(make_float4(c.inv[0], c.inv[1], c.inv[2], c.inv[3]));
      },
      [&](int i, int p, const uint16_t* l) {
        const int b = ctx->inst[i].bbeg + (p & 0x7fffffff);
        irec.push_back(make_int4(Pack16(l[0], l[1]), Pack16(l[2], l[3]), Bits(F.host_c[b]),
                                 Global(p, ctx->inst[i].bbeg)));
        iK.push_back(F.host_k[b]);
      },
      P.fem, H);
  if (!made) return XRT_OK;
  hipStream_t s = ctx->stream;
  hipError_t e = UploadPlan(ctx, P.fem, H);
  if (e == hipSuccess) e = P.frec.Upload(frec, s);
  if (e == hipSuccess) e = P.finv.Upload(finv, s);
  if (e == hipSuccess) e = P.irec.Upload(irec, s);
  if (e == hipSuccess) e = P.iK.Upload(iK, s);
  if (e == hipSuccess) e = P.ilam.Alloc(std::max<size_t>(irec.size(), 1));
  return FinishPlan(P.fem, e, ConfigurePatchSweep, P.frec, P.finv, P.irec, P.iK, P.ilam);
}

// The reverse sweep's plan (built when the first adjoint begins): what a vertex's adjoint depends
// on in the reversed order of the colors.
int PatchPrepareAdj(xrt_ctx* ctx) {
  PatchData& P = ctx->patches;
  if (P.adj.tried) return XRT_OK;
  P.adj.tried = true;
  const size_t ni = ctx->inst.size();
  int ns = 0, nb = 0;
  for (const HostInstance& h : ctx->inst) {
    ns = std::max(ns, h.s_ncol);
    nb = std::max(nb, h.b_ncol);
  }
  // color-sorted positions in reversed color order, and that order's color offsets
  auto reversed = [](const std::vector<int32_t>& coloff, std::vector<int32_t>& pos,
                     std::vector<int32_t>& off) {
    pos.clear();
    off.assign(1, 0);
    for (size_t c = coloff.size(); c-- > 1;) {
      for (int32_t p = coloff[c - 1]; p < coloff[c]; ++p) pos.push_back(p);
      off.push_back(static_cast<int32_t>(pos.size()));
    }
  };
  auto orders = [](const std::vector<int32_t>& pos, const std::vector<int32_t>& order) {
    std::vector<int32_t> o(pos.size());
    for (size_t k = 0; k < pos.size(); ++k) o[k] = order[pos[k]];
    return o;
  };
  std::vector<std::vector<int32_t>> spos(ni), bpos(ni);
  std::vector<int2> sent;
  std::vector<int4> bent;
  HostPlan H;
  const bool made = MakePlan(
      ctx, nb, ns,
      [&](int i) {
        const HostInstance& h = ctx->inst[i];
        std::vector<int32_t> soff, boff;
        reversed(h.s_coloff, spos[i], soff);
        reversed(h.b_coloff, bpos[i], boff);
        return std::vector<PatchFamily>{Family(4, h.bends, orders(bpos[i], h.b_order), boff),
                                        Family(2, h.edges, orders(spos[i], h.s_order), soff)};
      },
      [&](int i, int p, const uint16_t* l) {
        const int q = bpos[i][p & 0x7fffffff] | (p & static_cast<int>(0x80000000u));
        bent.push_back(make_int4(Pack16(l[0], l[1]), Pack16(l[2], l[3]), Global(q, ctx->inst[i].bbeg), 0));
      },
      [&](int i, int p, const uint16_t* l) {
        const int q = spos[i][p & 0x7fffffff] | (p & static_cast<int>(0x80000000u));
        sent.push_back(make_int2(Pack16(l[0], l[1]), Global(q, ctx->inst[i].sbeg)));
      },
      P.adj, H, kPatchAdjVertBytes, true);
  if (!made) return XRT_OK;
  hipStream_t s = ctx->stream;
  hipError_t e = P.adj.patch.Upload(H.dev, s);
  if (e == hipSuccess) e = P.adj.verts.Upload(H.verts, s);
  if (e == hipSuccess) e = P.adj.off.Upload(H.off, s);
  if (e == hipSuccess) e = P.bent.Upload(bent, s);
  if (e == hipSuccess) e = P.sent.Upload(sent, s);
  if (e == hipSuccess) e = P.glam.Alloc(std::max<size_t>(sent.size(), 1));
  if (e == hipSuccess) e = P.gx_alt.Alloc(ctx->x0.n);
  return FinishPlan(P.adj, e, ConfigurePatchAdj, P.bent, P.sent, P.glam, P.gx_alt);
}

int PatchAdjIter(xrt_ctx* ctx, const StepConsts& k, const BendMode& m, bool first,
                 const float4* tape_b, const float4* tape_s) {
  PatchData& P = ctx->patches;
  AdjointData& A = *ctx->adj;
  const PatchPlanDev& D = P.adj;
  const PatchAdjArgs a{D.patch.ptr, D.verts.ptr, D.off.ptr, P.bent.ptr,   P.sent.ptr,
                       ctx->bpar.ptr, ctx->sc.ptr, ctx->x0.ptr, A.gx.ptr, P.gx_alt.ptr,
                       P.glam.ptr,  A.gcomp.ptr, A.gbcomp.ptr, D.n, D.c0, D.c1};
  XRT_CHECK_HIP(LaunchPatchAdj(ctx->stream, a, k.inv_dt2, m, k.solve_bending ? 1 : 0, first ? 1 : 0,
                               tape_b, tape_s, D.threads, D.lds_bytes));
  std::swap(A.gx.ptr, P.gx_alt.ptr);
  return XRT_OK;
}

const PatchPlanDev& PatchPlanOf(const xrt_ctx* ctx) {
  return FemOn(ctx) ? ctx->patches.fem : ctx->patches.xpbd;
}

int PatchIter(xrt_ctx* ctx, const StepConsts& k, const BendMode& m, int it, bool ground,
              bool contacts, const PatchTape& t) {
  PatchData& P = ctx->patches;
  const PatchPlanDev& D = PatchPlanOf(ctx);
  float4* out = ctx->xcur == ctx->x.ptr ? P.alt.ptr : ctx->x.ptr;
  const PatchSweep w{ctx->xcur, out, ctx->x0.ptr, it, it + 1 == k.iterations ? 1 : 0,
                     ground ? 1 : 0, t.s, t.b, t.g, contacts ? ctx->ic.ptr : nullptr,
                     ctx->params.contact_friction,
                     1.0f / static_cast<float>(ctx->params.num_substeps), t.c, t.e};
  const int threads = ctx->tuning.wide_per_thread == 2 ? std::max(64, (D.threads / 2 + 63) / 64 * 64)
                                                       : D.threads;
  if (FemOn(ctx)) {
    const PatchFemArgs a{D.patch.ptr, D.verts.ptr, D.off.ptr,  P.frec.ptr,
                         P.finv.ptr,  P.irec.ptr,  P.iK.ptr,   P.ilam.ptr,
                         ctx->fem.iso_lam.ptr,     D.n, D.c0, D.c1};
    XRT_CHECK_HIP(LaunchPatchFem(ctx->stream, a, w, k, FemConstsOf(ctx->params), threads, D.lds_bytes));
  } else {
    const PatchArgs a{D.patch.ptr, D.verts.ptr, D.off.ptr, P.srec.ptr, P.slam.ptr, P.brec.ptr,
                      P.bcon.ptr, ctx->slam.ptr, D.n, D.c0, D.c1};
    XRT_CHECK_HIP(LaunchPatchSweep(ctx->stream, a, w, k, m, threads, D.lds_bytes));
  }
  ctx->xcur = out;
  return XRT_OK;
}

int PatchRefreshCompliance(xrt_ctx* ctx) {
  PatchData& P = ctx->patches;
  if (!P.xpbd.ready) return XRT_OK;
  XRT_CHECK_HIP(LaunchPatchCompliance(ctx->stream, ctx->sc.ptr, P.srec.ptr,
                                      static_cast<int>(P.srec.n)));
  return XRT_OK;
}

}  // namespace xrt
