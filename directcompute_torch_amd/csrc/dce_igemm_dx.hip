// The input gradient GEMM of the convolutions: filters (rows c) x G patches
// (rows = input pixels).  On bf16 parts (dce_igemm_parts.h) or, for few
// channels, on fp32 MFMAs (dce_igemm.h).
#include "dce_igemm_parts.h"

namespace dce {

template <bool S1, bool BLK>
struct DxRun {
  const float* wt;
  const float* gn;
  float* dx;
  float* part;
  ConvGeom g;
  uint32_t splits;
  template <int MT, int NT, int KT>
  int occ(bool split) const {
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPixRK<NT, KT, false, S1, BLK>;
    return split ? occupancy(k_igemm<MT, NT, KT, LA, LB, EpiRowMajor>)
                 : occupancy(k_igemm<MT, NT, KT, LA, LB, EpiNCHW>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    const uint32_t OCp = pad4(g.OC), KK = g.k * g.k, kdim = KK * OCp;
    const uint32_t HW = g.H * g.W, N = g.B * HW;
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPixRK<NT, KT, false, S1, BLK>;
    const typename LA::Params pa{wt, kdim, g.C, kdim, g.C * kdim};
    const typename LB::Params pb{gn, g.OH, g.OW, OCp, g.k, g.s, g.p, g.W, HW, N, kdim,
                                 g.B * g.OH * g.OW * OCp, make_fastdiv(HW), make_fastdiv(g.W),
                                 make_fastdiv(BLK ? KK : OCp), make_fastdiv(g.k)};
    const uint32_t kt = cdiv(kdim, KT);
    const EpiNCHW::Params pe{dx, nullptr, g.C, HW, N, 0, make_fastdiv(HW)};
    if (splits > 1) {
      const EpiRowMajor::Params pr{part, g.C, N, N, g.C * N};
      return launch<MT, NT, KT, LA, LB, EpiRowMajor>(pa, pb, pr, g.C, N, kt, splits,
                                                    "conv_backward_input") &&
             split_nchw(part, nullptr, dx, g.C, N, HW, splits, 0);
    }
    return launch<MT, NT, KT, LA, LB, EpiNCHW>(pa, pb, pe, g.C, N, kt, 1, "conv_backward_input");
  }
};

// One sub-pixel phase of a strided dX (s > 1).  The input pixels (b, ph +
// s*a, pw + s*c) receive only the taps kh = rh + s*jh (jh < nh), kw = rw +
// s*jw (jw < nw) with rh = (ph + p) mod s, whose output pixels are (a + qh -
// jh, c + qw - jw), qh = (ph + p - rh) / s: a stride-1 gather over the
// phase's own GH x GW grid with an nh x nw kernel.
struct PhaseGeom {
  uint32_t ph, pw, rh, rw, nh, nw, qh, qw, GH, GW;
};

template <class LA, class LB, bool BLK>
static void dx_phase_params(const float* wt, const float* gn, float* dx, const ConvGeom& g,
                            const PhaseGeom& q, typename LA::Params& pa, typename LB::Params& pb,
                            EpiNCHWPhase::Params& pe) {
  const uint32_t OCp = pad4(g.OC), KK = q.nh * q.nw, kdim = KK * OCp;
  const uint32_t GHW = q.GH * q.GW, N = g.B * GHW;
  pa = {wt, kdim, g.C, kdim, g.C * kdim};
  pb = {gn, g.OH, g.OW, OCp, q.nw, 1, q.qh, q.GW, GHW, N, kdim,
        g.B * g.OH * g.OW * OCp, make_fastdiv(GHW), make_fastdiv(q.GW),
        make_fastdiv(BLK ? KK : OCp), make_fastdiv(q.nw), int(q.qw) - int(q.qh)};
  pe = {dx, g.C, g.H, g.W, q.GW, GHW, N, g.s, q.ph, q.pw, make_fastdiv(GHW), make_fastdiv(q.GW)};
}
template <bool BLK>
struct DxPhaseRun {
  const float* wt;
  const float* gn;
  float* dx;
  ConvGeom g;
  PhaseGeom q;
  template <int MT, int NT, int KT>
  int occ(bool) const {
    return occupancy(
        k_igemm<MT, NT, KT, LdDenseRK<MT, KT>, LdPixRK<NT, KT, false, true, BLK>, EpiNCHWPhase>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPixRK<NT, KT, false, true, BLK>;
    typename LA::Params pa;
    typename LB::Params pb;
    EpiNCHWPhase::Params pe;
    dx_phase_params<LA, LB, BLK>(wt, gn, dx, g, q, pa, pb, pe);
    const uint32_t kdim = q.nh * q.nw * pad4(g.OC), N = g.B * q.GH * q.GW;
    return launch<MT, NT, KT, LA, LB, EpiNCHWPhase>(pa, pb, pe, g.C, N, cdiv(kdim, KT), 1,
                                                    "conv_backward_input");
  }
};

// dX on parts at stride 1 (the phase fields unused), or one phase.
template <class EPI>
struct DxPartsRun {
  const float* wt;
  const float* gn;
  float* dx;
  float* part;
  ConvGeom g;
  uint32_t splits;
  PhaseGeom q;
  static constexpr bool PHASE = std::is_same<EPI, PEpiPhase>::value;
  template <int MT, int NT>
  int occ(bool split) const {
    return split ? occupancy(k_gemm_parts<MT, NT, PRows<MT>, PPix<NT>, PEpiRowMajor>)
                 : occupancy(k_gemm_parts<MT, NT, PRows<MT>, PPix<NT>, EPI>);
  }
  template <int MT, int NT>
  bool run() const {
    const uint32_t no = pad16(g.OC) / 16, KK = PHASE ? q.nh * q.nw : g.k * g.k, kt = KK * no;
    const uint32_t GW = PHASE ? q.GW : g.W, GHW = PHASE ? q.GH * q.GW : g.H * g.W, N = g.B * GHW;
    const uint32_t kw = PHASE ? q.nw : g.k;
    const char* what = "conv_backward_input";
    using LA = PRows<MT>;
    using LB = PPix<NT>;
    const typename LA::Params pa{wt, g.C, kt, g.C * kt * 24};
    const typename LB::Params pb{gn, g.OH, g.OW, no, kw, PHASE ? q.qh : g.p, GW, GHW, N,
                                 uint32_t(parts_floats(size_t(g.B) * g.OH * g.OW, g.OC)),
                                 make_fastdiv(GHW), make_fastdiv(GW), make_fastdiv(KK),
                                 make_fastdiv(kw), PHASE ? int(q.qw) - int(q.qh) : 0};
    if constexpr (PHASE) {
      const EpiNCHWPhase::Params pe{dx, g.C, g.H, g.W, GW, GHW, N, g.s, q.ph, q.pw, pb.dGridHW,
                                    pb.dGridW};
      return launch_parts<MT, NT, LA, LB, PEpiPhase>(pa, pb, pe, g.C, N, kt, 1, what);
    } else {
      if (splits > 1) {
        const EpiRowMajor::Params pr{part, g.C, N, N, g.C * N};
        return launch_parts<MT, NT, LA, LB, PEpiRowMajor>(pa, pb, pr, g.C, N, kt, splits, what) &&
               split_nchw(part, nullptr, dx, g.C, N, GHW, splits, 0);
      }
      const EpiNCHW::Params pe{dx, nullptr, g.C, GHW, N, 0, pb.dGridHW};
      return launch_parts<MT, NT, LA, LB, PEpiNCHW>(pa, pb, pe, g.C, N, kt, 1, what);
    }
  }
};

static PhaseGeom phase_geom(const ConvGeom& g, uint32_t ph, uint32_t pw) {
  const uint32_t s = g.s;
  PhaseGeom q{};
  q.ph = ph;
  q.pw = pw;
  q.GH = ph < g.H ? cdiv(g.H - ph, s) : 0;
  q.GW = pw < g.W ? cdiv(g.W - pw, s) : 0;
  q.rh = (ph + g.p) % s;
  q.rw = (pw + g.p) % s;
  q.nh = q.rh < g.k ? cdiv(g.k - q.rh, s) : 0;
  q.nw = q.rw < g.k ? cdiv(g.k - q.rw, s) : 0;
  q.qh = (ph + g.p - q.rh) / s;
  q.qw = (pw + g.p - q.rw) / s;
  return q;
}

// The phases of a stride-2 dX that some tap reaches, in one launch.
struct DxPhases {
  ConvGeom g;
  PhaseGeom q[4];
  uint32_t n, cols, kmax;  // phases, their pixels together, the longest dot product
  bool empty;              // pixels that no tap reaches
  const float* gn;
  float* dx;
  const float* wt[4];
  uint32_t splits;
  float* part;  // splits > 1: partials, each laid out as dx
  DxPhases(const ConvGeom& geom, bool parts) : g(geom), n(0), cols(0), kmax(0), empty(false) {
    for (uint32_t i = 0; i < 4; ++i) {
      const PhaseGeom f = phase_geom(g, i / 2, i % 2);
      if (f.GH * f.GW == 0) continue;
      if (f.nh * f.nw == 0) {
        empty = true;
        continue;
      }
      q[n++] = f;
      cols += g.B * f.GH * f.GW;
      kmax = std::max(kmax, f.nh * f.nw * (parts ? pad16(g.OC) : pad4(g.OC)));
    }
  }
  // f(i, phase, columns) fills product i; returns the workgroups of them all.
  template <class A, class F>
  uint32_t fill(A& a, uint32_t MT, uint32_t NT, F&& f) const {
    a.gm = cdiv(g.C, MT);
    uint32_t wgs = 0;
    for (uint32_t i = 0; i < 4; ++i) {
      a.first[i] = i < n ? wgs : 0xFFFFFFFFu;
      if (i >= n) continue;
      const uint32_t N = g.B * q[i].GH * q[i].GW;
      f(i, q[i], N);
      wgs += a.gm * cdiv(N, NT);
    }
    return wgs;
  }
};
struct DxMultiParts : DxPhases {
  using DxPhases::DxPhases;
  using EPI = PEpiPhase;
  template <int MT, int NT>
  int occ(bool) const {
    return occupancy(k_gemm_parts_multi<MT, NT, PRows<MT>, PPix<NT>, EPI>);
  }
  template <int MT, int NT>
  bool run() const {
    Multi<PRows<MT>, PPix<NT>, EPI> a{};
    const uint32_t no = pad16(g.OC) / 16;
    const uint32_t wgs = fill(a, MT, NT, [&](uint32_t i, const PhaseGeom& f, uint32_t N) {
      const uint32_t KK = f.nh * f.nw, GHW = f.GH * f.GW;
      a.ktiles[i] = KK * no;
      a.pa[i] = {wt[i], g.C, KK * no, g.C * KK * no * 24};
      a.pb[i] = {gn, g.OH, g.OW, no, f.nw, f.qh, f.GW, GHW, N,
                 uint32_t(parts_floats(size_t(g.B) * g.OH * g.OW, g.OC)), make_fastdiv(GHW),
                 make_fastdiv(f.GW), make_fastdiv(KK), make_fastdiv(f.nw), int(f.qw) - int(f.qh)};
      a.pe[i] = {splits > 1 ? part : dx, g.C,  g.H,  g.W,  f.GW, GHW, N, g.s, f.ph, f.pw,
                 a.pb[i].dGridHW,        a.pb[i].dGridW};
    });
    const uint32_t values = g.B * g.C * g.H * g.W;
    hipLaunchKernelGGL((k_gemm_parts_multi<MT, NT, PRows<MT>, PPix<NT>, EPI>),
                       dim3(wgs * splits), dim3(kThreads), 0, stream(), a, wgs, splits, values);
    return check_launch("conv_backward_input") &&
           (splits == 1 || split_sum(part, dx, values, splits));
  }
};
template <bool BLK>
struct DxMulti : DxPhases {
  using DxPhases::DxPhases;
  template <int MT, int NT, int KT>
  int occ(bool) const {
    return occupancy(k_igemm_multi<MT, NT, KT, LdDenseRK<MT, KT>, LdPixRK<NT, KT, false, true, BLK>,
                                   EpiNCHWPhase>);
  }
  template <int MT, int NT, int KT>
  bool run() const {
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPixRK<NT, KT, false, true, BLK>;
    Multi<LA, LB, EpiNCHWPhase> a{};
    const uint32_t wgs = fill(a, MT, NT, [&](uint32_t i, const PhaseGeom& f, uint32_t N) {
      a.ktiles[i] = cdiv(f.nh * f.nw * pad4(g.OC), KT);
      dx_phase_params<LA, LB, BLK>(wt[i], gn, dx, g, f, a.pa[i], a.pb[i], a.pe[i]);
    });
    hipLaunchKernelGGL((k_igemm_multi<MT, NT, KT, LA, LB, EpiNCHWPhase>), dim3(wgs), dim3(kThreads),
                       0, stream(), a);
    return check_launch("conv_backward_input");
  }
};
// Their filters are re-laid by one launch too; phases that no tap reaches (k =
// 1) are zero.
template <class R>
static bool phases_in_one(R& r, const TileCfg& c, const float* w, float* wt, const float* gn,
                          float* dx, float* part, bool parts) {
  const ConvGeom& g = r.g;
  const uint32_t OCp = parts ? pad16(g.OC) : pad4(g.OC);
  WPerm4 pw{};
  float* at = wt;
  for (uint32_t i = 0; i < r.n; ++i) {
    const PhaseGeom& q = r.q[i];
    const uint32_t KK = q.nh * q.nw;
    pw.p[i] = WPerm{w, at, g.OC, g.C, KK, OCp, KK * OCp, 1, blocked_k(OCp) ? 1 : 0, q.nw, g.k, 2,
                    q.rh, q.rw, parts ? 1u : 0u};
    r.wt[i] = at;
    at += parts ? parts_floats(size_t(g.C) * KK, g.OC) : size_t(g.C) * KK * OCp;
  }
  r.gn = gn;
  r.dx = dx;
  r.splits = c.splits;
  r.part = part;
  if (r.empty && !fill_zero(dx, size_t(g.B) * g.C * g.H * g.W)) return false;
  if (r.n == 0) return true;
  if (!permute_w4(pw)) return false;
  if constexpr (std::is_same<R, DxMultiParts>::value)
    return parts_dispatch(c, r);
  else
    return tiles_dispatch16(c, r);
}

// dX of a strided convolution as its s*s sub-pixel phases: every input pixel
// multiplies only the taps that reach it, where the strided gather walks all
// k*k taps for every pixel and finds all but about 1/s^2 of them out of
// step.  Each phase gets its own filter re-layout (into wt, C * k*k * OCp
// floats) and GEMM, unsplit; phases that no tap reaches (k < s) are zero.
static bool dx_phases(const float* w, float* wt, const float* gn, float* dx, const ConvGeom& g,
                      bool parts) {
  const uint32_t s = g.s, OCp = parts ? pad16(g.OC) : pad4(g.OC);
  const bool blk = blocked_k(OCp);
  bool empty = false;
  for (uint32_t ph = 0; ph < s; ++ph)
    for (uint32_t pw = 0; pw < s; ++pw) {
      const PhaseGeom q = phase_geom(g, ph, pw);
      empty |= q.GH * q.GW > 0 && q.nh * q.nw == 0;
    }
  if (empty && !fill_zero(dx, size_t(g.B) * g.C * g.H * g.W)) return false;
  for (uint32_t ph = 0; ph < s; ++ph)
    for (uint32_t pw = 0; pw < s; ++pw) {
      const PhaseGeom q = phase_geom(g, ph, pw);
      if (q.GH * q.GW == 0 || q.nh * q.nw == 0) continue;
      const uint32_t KK = q.nh * q.nw, kdim = KK * OCp, N = g.B * q.GH * q.GW;
      if (!permute_w(WPerm{w, wt, g.OC, g.C, KK, OCp, kdim, 1, blk ? 1 : 0, q.nw, g.k, s, q.rh,
                           q.rw, parts ? 1u : 0u}))
        return false;
      if (parts) {
        const DxPartsRun<PEpiPhase> run{wt, gn, dx, nullptr, g, 1, q};
        const TileCfg t = parts_choose("DCE_TUNE_DX", g.C, N, kdim, 1, true,
                                       [&](const TileCfg& v) { return parts_occ(v, run); });
        if (!parts_dispatch(t, run)) return false;
        continue;
      }
      TileCfg c = choose(
          "DCE_TUNE_DX", g.C, N, kdim, 1, true,
          [&](const TileCfg& t) {
            return blk ? tiles_occ16(t, DxPhaseRun<true>{}) : tiles_occ16(t, DxPhaseRun<false>{});
          },
          true);
      narrow_short_k(c, "DCE_TUNE_DX", g.C, N, kdim);
      c.splits = 1;
      const bool ok = blk ? tiles_dispatch16(c, DxPhaseRun<true>{wt, gn, dx, g, q})
                          : tiles_dispatch16(c, DxPhaseRun<false>{wt, gn, dx, g, q});
      if (!ok) return false;
    }
  return true;
}

// The whole gather.
static TileCfg dx_choose(const ConvGeom& g, bool parts) {
  const uint32_t N = g.B * g.H * g.W;
  const bool s1 = g.s == 1;
  if (parts)  // s1: conv_dx_plan takes the phases otherwise
    return parts_choose("DCE_TUNE_DX", g.C, N, g.k * g.k * pad16(g.OC), 8, true,
                        [&](const TileCfg& t) { return parts_occ(t, DxPartsRun<PEpiNCHW>{}); });
  const uint32_t OCp = pad4(g.OC), kdim = g.k * g.k * OCp;
  const bool blk = blocked_k(OCp);
  TileCfg c = choose(
      "DCE_TUNE_DX", g.C, N, kdim, 8, true,
      [&](const TileCfg& t) { return conv_variant_occ<DxRun>(s1, blk, t); }, true);
  narrow_short_k(c, "DCE_TUNE_DX", g.C, N, kdim);
  return c;
}
// All phases of a stride-2 dX.
static TileCfg dx_choose_phases(const ConvGeom& g, bool parts) {
  if (parts) {
    const DxMultiParts r(g, true);
    return parts_choose("DCE_TUNE_DX", g.C, r.cols, r.kmax, r.empty ? 1 : 8, true,
                        [&](const TileCfg& v) { return parts_occ(v, r); });
  }
  const DxPhases r(g, false);
  auto go = [&](const auto& run) {
    TileCfg c = choose("DCE_TUNE_DX", g.C, r.cols, r.kmax, 1, true,
                       [&](const TileCfg& t) { return tiles_occ16(t, run); }, true);
    narrow_short_k(c, "DCE_TUNE_DX", g.C, r.cols, r.kmax);
    c.splits = 1;
    return c;
  };
  return blocked_k(pad4(g.OC)) ? go(DxMulti<true>(g, false)) : go(DxMulti<false>(g, false));
}

// How a dX runs.  At stride 3 or more as sub-pixel phases (dx_phases), each with
// its own filter re-layout and no split: the strided gather would walk s^2 times
// the taps that reach a pixel (AlexNet c1's dX at b128: 18.0 -> 1.24 ms).  At
// stride 2 the four phases share one launch.  On parts they are always taken (12
// x 37 x 61 x 45 -> 70, k5: dX 78 -> 32 us), split where few pixels meet long dot
// products (forward and backward, gather on fp32 MFMAs, unsplit and split
// phases: 7 x 137 x 6 x 7 -> 505, k3 65, 97 and 56, 1 x 56 x 7 x 31 -> 384, k7
// 175, 211 and 80, 32 x 39 x 6 x 10 -> 287, k3 60, 78 and 52 us).  On fp32 MFMAs they are unsplit (forward and backward, gather ->
// phases; B x C x H x W -> OC): 128 x 8 x 100 x 90 -> 40, k3 338 -> 229, 32 x 16
// x 112 x 112 -> 24, k3 102 -> 85, 20 x 160 x 160 -> 31, k5 75 -> 58, 64 x 128 x
// 28 x 28 -> 256, k1 104 -> 84 us.  Not where the gather splits its k * k taps so
// often that the largest phase's unsplit taps, (k + 1) / 2 squared, make the
// longer chain (30 x 9 x 9 -> 384, k5 79 -> 131, 128 x 30 x 7 x 7 -> 384, k5 149
// -> 180 us), nor where the products saved do not pay for the launches added, the
// filters' and for k = 1 the zeros' (8 x 16 x 64 x 64 -> 24, k3 37 -> 41, 16 x 64
// x 56 x 56 -> 128, k1 alone 76 -> 88 us), nor under short dot products, where
// the phases' stores, every second float of a row, bound them (48 x 390 x 118 x
// 16 -> 4, k2 163 -> 226, 67 x 55 x 182 x 67 -> 6, k3 319 -> 384, 27 x 220 x 49 x
// 35 -> 9, k3 99 -> 110; but 83 x 20 x 137 x 68 -> 48, k2 229 -> 196, 6 x 10 x 129
// x 146 -> 21, k3 52 -> 49 and, over few channels, 112 x 9 x 26 x 145 -> 9, k3 70
// -> 64 us).
DxPlan conv_dx_plan(const ConvGeom& g, bool parts) {
  DxPlan p{g.s >= 3 || (parts && g.s == 2), {128, 128, 16, 1}, 0};
  if (g.s == 1 || !p.phased) {
    p.cfg = dx_choose(g, parts);
    const uint32_t KK = g.k * g.k, kp = (g.k + 1) / 2;
    const double products = double(g.C) * g.B * g.H * g.W * KK * pad4(g.OC);
    p.phased = g.s == 2 && p.cfg.splits * kp * kp <= KK && products >= (g.k == 1 ? 8e8 : 2e8) &&
               KK * pad4(g.OC) >= (g.C > 16 ? 180u : 100u);
  }
  if (g.s == 2 && p.phased) p.cfg = dx_choose_phases(g, parts);
  if (p.cfg.splits > 1) p.part = size_t(p.cfg.splits) * g.C * g.B * g.H * g.W;
  return p;
}
bool conv_dx(const DxPlan& p, const float* w, float* wt, const float* gn, float* dx, float* part,
             const ConvGeom& g, bool parts) {
  if (p.phased && g.s == 2) {
    if (parts) {
      DxMultiParts r(g, true);
      return phases_in_one(r, p.cfg, w, wt, gn, dx, part, true);
    }
    auto go = [&](auto&& r) { return phases_in_one(r, p.cfg, w, wt, gn, dx, part, false); };
    return blocked_k(pad4(g.OC)) ? go(DxMulti<true>(g, false)) : go(DxMulti<false>(g, false));
  }
  if (p.phased) return dx_phases(w, wt, gn, dx, g, parts);
  if (parts) {
    if (g.s != 1) {
      set_error("conv_backward_input: a strided gather has no kernel on parts");
      return false;
    }
    return parts_dispatch(p.cfg, DxPartsRun<PEpiNCHW>{wt, gn, dx, part, g, p.cfg.splits, {}});
  }
  return conv_variant<DxRun>(g.s == 1, blocked_k(pad4(g.OC)), p.cfg, wt, gn, dx, part, g,
                             p.cfg.splits);
}

}  // namespace dce
