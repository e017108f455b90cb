// The filter gradient GEMM of the convolutions: dW = G (rows oc) x x-taps
// (rows (kh, kw, c)), both with k = output pixel.  On bf16 parts
// (dce_igemm_parts.h) or, for few channels, on fp32 MFMAs (dce_igemm.h).
#include "dce_igemm_parts.h"

namespace dce {

// `trans` swaps the operands (taps as output rows) for layers with fewer taps
// x channels than output channels, so the narrow tiles cover the short axis.
struct DwRun {
  const float* gn;  // G: NHWC, or G_pad for the stride-phase layout
  const float* xn;
  float* part;
  ConvGeom g;
  uint32_t splits;
  bool trans;
  bool pk;  // xn is the channel-packed copy: taps (kh, kw, c) with C unpadded
  bool ps;  // xn is the stride-phase copy, gn G_pad: taps (c, kh, kw), padded pixels
  template <int MT, int NT, int KT>
  int occ(bool) const {
    if (ps)
      return trans ? occupancy(k_igemm<MT, NT, KT, LdPsRK<MT, KT>, LdGPadRK<NT, KT>, EpiRowMajor>)
                   : occupancy(k_igemm<MT, NT, KT, LdGPadRK<MT, KT>, LdPsRK<NT, KT>, EpiRowMajor>);
    if (pk)
      return trans ? occupancy(k_igemm<MT, NT, KT, LdPkKR<MT, KT>, LdGradKR<NT, KT>, EpiRowMajor>)
                   : occupancy(k_igemm<MT, NT, KT, LdGradKR<MT, KT>, LdPkKR<NT, KT>, EpiRowMajor>);
    return trans ? occupancy(k_igemm<MT, NT, KT, LdXTapKR<MT, KT>, LdGradKR<NT, KT>, EpiRowMajor>)
                 : occupancy(k_igemm<MT, NT, KT, LdGradKR<MT, KT>, LdXTapKR<NT, KT>, EpiRowMajor>);
  }
  template <int MT, int NT, int KT, class LX>
  bool go(const typename LX::Params& px, uint32_t N) {
    const uint32_t OCp = pad4(g.OC), npix = g.B * g.OH * g.OW;
    const GradKRParams pg{gn, OCp, npix, npix * OCp};
    const uint32_t zs = 4 * cdiv(size_t(g.OC) * N, 4);  // split stride of the partials
    if (trans) {
      const EpiRowMajor::Params pe{part, N, g.OC, g.OC, zs};
      return launch<MT, NT, KT, LX, LdGradKR<NT, KT>, EpiRowMajor>(
          px, pg, pe, N, g.OC, cdiv(npix, KT), splits, "conv_backward_filter");
    }
    using LB = typename std::conditional<std::is_same<LX, LdPkKR<MT, KT>>::value, LdPkKR<NT, KT>,
                                         LdXTapKR<NT, KT>>::type;
    const EpiRowMajor::Params pe{part, g.OC, N, N, zs};
    return launch<MT, NT, KT, LdGradKR<MT, KT>, LB, EpiRowMajor>(
        pg, px, pe, g.OC, N, cdiv(npix, KT), splits, "conv_backward_filter");
  }
  template <int MT, int NT, int KT>
  bool run_ps() {
    const PsParams px = ps_params(xn, g);
    const GPadParams pg{gn, g.OC, px.OHWp, px.npix, g.B * g.OC * px.OHWp, px.dOHWp};
    const uint32_t N = px.kdim, zs = 4 * cdiv(size_t(g.OC) * N, 4), kt = cdiv(px.npix, KT);
    if (trans) {
      const EpiRowMajor::Params pe{part, N, g.OC, g.OC, zs};
      return launch<MT, NT, KT, LdPsRK<MT, KT>, LdGPadRK<NT, KT>, EpiRowMajor>(
          px, pg, pe, N, g.OC, kt, splits, "conv_backward_filter");
    }
    const EpiRowMajor::Params pe{part, g.OC, N, N, zs};
    return launch<MT, NT, KT, LdGPadRK<MT, KT>, LdPsRK<NT, KT>, EpiRowMajor>(
        pg, px, pe, g.OC, N, kt, splits, "conv_backward_filter");
  }
  template <int MT, int NT, int KT>
  bool run() {
    const uint32_t KK = g.k * g.k, OHW = g.OH * g.OW, npix = g.B * OHW;
    if (ps) return run_ps<MT, NT, KT>();
    if (pk) return go<MT, NT, KT, LdPkKR<MT, KT>>(pk_params(xn, g), KK * g.C);
    const uint32_t Cp = pad4(g.C), N = KK * Cp;
    const XTapParams px{xn, g.H, g.W, Cp, g.k, g.s, g.p, g.OW, OHW, npix, N,
                        g.B * g.H * g.W * Cp, make_fastdiv(OHW), make_fastdiv(g.OW),
                        make_fastdiv(Cp), make_fastdiv(g.k)};
    return go<MT, NT, KT, LdXTapKR<MT, KT>>(px, N);
  }
};

// On parts: channels padded to 16, taps (kh, kw, c) with c over pad16(C).
struct DwPartsRun {
  const float* gn;
  const float* xn;
  float* part;
  ConvGeom g;
  uint32_t splits;
  bool trans;
  // Layers on parts have at least 200 taps x channels: no 32-row tile of taps.
  template <int MT, int NT>
  int occ(bool) const {
    if constexpr (MT > 32)
      if (trans) return occupancy(k_gemm_parts<MT, NT, PTap<MT>, PGrad<NT>, PEpiRowMajor>);
    return occupancy(k_gemm_parts<MT, NT, PGrad<MT>, PTap<NT>, PEpiRowMajor>);
  }
  template <int MT, int NT>
  bool run() {
    const uint32_t OHW = g.OH * g.OW, npix = g.B * OHW, nc = pad16(g.C) / 16, no = pad16(g.OC) / 16;
    const uint32_t N = g.k * g.k * nc * 16, zs = 4 * cdiv(size_t(g.OC) * N, 4), kt = cdiv(npix, 16);
    const uint32_t fg = uint32_t(parts_floats(npix, g.OC));
    const uint32_t fx = uint32_t(parts_floats(size_t(g.B) * g.H * g.W, g.C));
    if (trans) {
      if constexpr (MT > 32) {
        const typename PTap<MT>::Params px{xn, g.H, g.W, nc, g.k, g.s, g.p, g.OW, OHW, npix, N, fx,
                                           make_fastdiv(OHW), make_fastdiv(g.OW),
                                           make_fastdiv(16 * nc), make_fastdiv(g.k)};
        const typename PGrad<NT>::Params pg{gn, no, npix, fg};
        const PEpiRowMajor::Params pe{part, N, g.OC, g.OC, zs};
        return launch_parts<MT, NT, PTap<MT>, PGrad<NT>, PEpiRowMajor>(px, pg, pe, N, g.OC, kt, splits,
                                                                       "conv_backward_filter");
      }
      set_error("conv_backward_filter: %u taps x channels on a %d-row tile", N, MT);
      return false;
    }
    const typename PGrad<MT>::Params pg{gn, no, npix, fg};
    const typename PTap<NT>::Params px{xn, g.H, g.W, nc, g.k, g.s, g.p, g.OW, OHW, npix, N, fx,
                                       make_fastdiv(OHW), make_fastdiv(g.OW), make_fastdiv(16 * nc),
                                       make_fastdiv(g.k)};
    const PEpiRowMajor::Params pe{part, g.OC, N, N, zs};
    return launch_parts<MT, NT, PGrad<MT>, PTap<NT>, PEpiRowMajor>(pg, px, pe, g.OC, N, kt, splits,
                                                                   "conv_backward_filter");
  }
};

// M x N: the product's shape (rows x columns, transposed when `trans`).  A
// grid of a few tiles gets more split-K slices, so that the whole chip works
// on it.
TileCfg conv_dw_choose(uint32_t M, uint32_t N, uint32_t kdim, bool trans, bool pk, bool ps,
                       bool parts) {
  const uint32_t ntiles = cdiv(M, pick_tile_m(M)) * cdiv(N, pick_tile(N));
  const uint32_t most = ntiles <= 4 ? 1024 : 256;
  if (parts) {
    DwPartsRun r{};
    r.trans = trans;
    return parts_choose("DCE_TUNE_DW", M, N, kdim, most, false,
                        [&](const TileCfg& t) { return parts_occ(t, r); });
  }
  DwRun r{};
  r.trans = trans;
  r.pk = pk;
  r.ps = ps;
  return choose(
      "DCE_TUNE_DW", M, N, kdim, most, false,
      [&](const TileCfg& t) { return tiles_occ<true>(t, r); }, false, true, !ps && !pk);
}
bool conv_dw_gemm(const TileCfg& c, const float* gn, const float* xn, float* part,
                  const ConvGeom& g, bool trans, bool pk, bool ps, bool parts) {
  if (parts) return parts_dispatch(c, DwPartsRun{gn, xn, part, g, c.splits, trans});
  return tiles_dispatch<true>(c, DwRun{gn, xn, part, g, c.splits, trans, pk, ps});
}

}  // namespace dce
