// The flagged dense GEMM of MatMulAlloc (implicit GEMM of dce_igemm.h).
#include "dce_igemm.h"

namespace dce {

// ----------------------------------------------------------------- GEMM
template <bool AT, bool BT>
struct GemmRun {
  const float *a, *b;
  float* c;
  uint32_t M, K, N, splits;
  uint32_t lda, ldb, kdA, kdB;  // row strides and K extents as stored (padded)
  float* part;                  // split-K partials (splits > 1)
  // A[m][k]: stored M x K (ROWK) or K x M (KROW); B[n][k]: stored N x K (ROWK) or K x N (KROW).
  template <int MT, int KT>
  using LAt = typename std::conditional<AT, LdDenseKR<MT, KT>, LdDenseRK<MT, KT>>::type;
  template <int NT, int KT>
  using LBt = typename std::conditional<BT, LdDenseRK<NT, KT>, LdDenseKR<NT, KT>>::type;
  template <int MT, int NT, int KT>
  int occ(bool) const {
    return occupancy(k_igemm<MT, NT, KT, LAt<MT, KT>, LBt<NT, KT>, EpiRowMajor>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    using LA = LAt<MT, KT>;
    using LB = LBt<NT, KT>;
    const typename LA::Params pa{a, lda, AT ? lda : M, kdA, (AT ? K : M) * lda};
    const typename LB::Params pb{b, ldb, BT ? N : ldb, kdB, (BT ? N : K) * ldb};
    const uint32_t kt = cdiv(std::max(kdA, kdB), KT);
    const EpiRowMajor::Params pe{c, M, N, N, M * N};
    if (splits > 1) {
      const EpiRowMajor::Params pr{part, M, N, N, M * N};
      return launch<MT, NT, KT, LA, LB, EpiRowMajor>(pa, pb, pr, M, N, kt, splits, "gemm") &&
             split_sum(part, c, M * N, splits);
    }
    return launch<MT, NT, KT, LA, LB, EpiRowMajor>(pa, pb, pe, M, N, kt, 1, "gemm");
  }
};

bool gemm(const float* a, const float* b, float* c, uint32_t M, uint32_t K, uint32_t N,
          uint32_t flags) {
  if (K == 0) return fill_zero(c, size_t(M) * N);
  const bool aT = flags & 1, bT = flags & 2;
  if (!operand_fits(size_t(M) * pad4(K), "gemm") || !operand_fits(size_t(K) * pad4(N), "gemm") ||
      !operand_fits(size_t(pad4(M)) * K, "gemm") || !operand_fits(size_t(N) * pad4(K), "gemm"))
    return false;
  // The dense loaders read whole quads along each operand's contiguous axis:
  // a stride that is not a multiple of 4 (or an unaligned base) gets a
  // zero-padded copy.
  const uint32_t aRows = aT ? K : M, aCols = aT ? M : K;
  const uint32_t bRows = bT ? N : K, bCols = bT ? K : N;
  const bool padA = (aCols % 4) || !aligned16(a), padB = (bCols % 4) || !aligned16(b);
  auto gemm_occ = [&](const TileCfg& t) {
    if (!aT && !bT) return tiles_occ(t, GemmRun<false, false>{});
    if (!aT && bT) return tiles_occ(t, GemmRun<false, true>{});
    if (aT && !bT) return tiles_occ(t, GemmRun<true, false>{});
    return tiles_occ(t, GemmRun<true, true>{});
  };
  TileCfg cfg = choose("DCE_TUNE_GEMM", M, N, pad4(K), 16, true, gemm_occ);
  // A grid that leaves CUs idle (small GEMMs such as AlexNet's fc3) runs
  // faster on 64 x 64 tiles 32 deep, at split counts that fill the chip:
  // fc3 forward 34 -> 22 us, its dA 29 -> 24 us in a sweep of every tile
  // and split count on MI355X.
  const uint32_t cus = uint32_t(num_cus());
  auto wgs = [&](const TileCfg& t) {
    return cdiv(M, uint32_t(t.MT)) * cdiv(N, uint32_t(t.NT)) * t.splits;
  };
  if (!getenv("DCE_TUNE_GEMM") && wgs(cfg) < cus && M >= 64 && N >= 64) {
    const uint32_t kt32 = cdiv(pad4(K), 32u);
    TileCfg alt{64, 64, 32, 1};
    const uint32_t t64 = cdiv(M, 64u) * cdiv(N, 64u);
    // The fewest splits that fill every CU, keeping at least 8 K tiles each.
    while (t64 * alt.splits < cus && alt.splits < 16 && kt32 / (alt.splits + 1) >= 8) alt.splits++;
    if (wgs(alt) > wgs(cfg)) cfg = alt;
  }
  // Skinny products with long dot products (a linear layer's forward and
  // input gradient at batch 128): 64 x 64 tiles 32 deep over about 1024
  // workgroups beat the 128 x 128 split-K choice (AlexNet fc1 forward 104 ->
  // 97 us, fc2 forward 56 -> 50 us, fc2 input gradient 53 -> 49 us in a sweep
  // of tiles and split counts on MI355X; wider grids, such as fc1's input
  // gradient with 288 such tiles, keep the model's choice).
  if (!getenv("DCE_TUNE_GEMM") && M <= 128 && pad4(K) >= 4096) {
    const uint32_t t64 = cdiv(M, 64u) * cdiv(N, 64u), kt32 = cdiv(pad4(K), 32u);
    if (t64 >= 64 && t64 <= 256) {
      TileCfg alt{64, 64, 32, std::max(1u, std::min(16u, 1024u / t64))};
      while (alt.splits > 1 && kt32 / alt.splits < 8) alt.splits--;
      cfg = alt;
    }
  }
  const size_t nA = padA ? al64(size_t(aRows) * pad4(aCols)) : 0;
  const size_t nB = padB ? al64(size_t(bRows) * pad4(bCols)) : 0;
  const size_t nP = cfg.splits > 1 ? size_t(cfg.splits) * M * N : 0;
  float* ws = (nA + nB + nP) ? workspace(nA + nB + nP) : nullptr;
  if ((nA + nB + nP) && !ws) return false;
  const float* ap = a;
  const float* bp = b;
  if (padA) {
    if (!pad_cols(a, ws, aRows, aCols, pad4(aCols))) return false;
    ap = ws;
  }
  if (padB) {
    if (!pad_cols(b, ws + nA, bRows, bCols, pad4(bCols))) return false;
    bp = ws + nA;
  }
  float* part = cfg.splits > 1 ? ws + nA + nB : nullptr;
  const uint32_t lda = pad4(aCols), ldb = pad4(bCols);
  // K extents: a ROWK operand's k axis is its padded row (zeros past K); a
  // KROW operand's k axis is its row count K.
  const uint32_t kdA = aT ? K : lda, kdB = bT ? ldb : K;
  bool ok;
  {
    ProfScope prof("gemm", 2.0 * M * N * double(K),
                   4.0 * (double(M) * K + double(K) * N + double(M) * N));
    if (!aT && !bT)
      ok = tiles_dispatch(cfg, GemmRun<false, false>{ap, bp, c, M, K, N, cfg.splits, lda, ldb, kdA, kdB, part});
    else if (!aT && bT)
      ok = tiles_dispatch(cfg, GemmRun<false, true>{ap, bp, c, M, K, N, cfg.splits, lda, ldb, kdA, kdB, part});
    else if (aT && !bT)
      ok = tiles_dispatch(cfg, GemmRun<true, false>{ap, bp, c, M, K, N, cfg.splits, lda, ldb, kdA, kdB, part});
    else
      ok = tiles_dispatch(cfg, GemmRun<true, true>{ap, bp, c, M, K, N, cfg.splits, lda, ldb, kdA, kdB, part});
  }
  return ok;
}

}  // namespace dce
