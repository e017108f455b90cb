// The flagged dense GEMM of MatMulAlloc: on fp32 MFMAs (dce_igemm.h),
// large A B^T products on bf16 parts (dce_igemm_parts.h).
#include "dce_igemm_parts.h"

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

// --------------------------------------------------------- A B^T on bf16 parts
// The input gradient of a linear layer, dX = dY W^T.  Large ones are bound by
// the fp32 MFMAs, at twice the time that reading W takes; as in the
// convolutions' backward, six bf16 products stand for one fp32 product.  W is
// read once by each row of tiles, so both operands are split on their way from
// registers into LDS.  128 x 4096 x 9216: 90 -> 74 us; 512 x 4096 x 9216: 355 -> 269 us;
// error against float64 4.4e-7 -> 1.5e-7 (over 2048: 2.9e-7 -> 1.2e-7).
//
// Not taken for A^T B (the filter gradient: both operands split by a pass
// 107 -> 106 us at 9216 x 128 x 4096, 46 -> 56 us at 4096 x 128 x 4096; its
// eight steps of 16 do not cover the loads and the store) nor for A B (the
// forward: 96 -> 83 us at 128 x 9216 x 4096, but another rounding there turns
// ReLU decisions).

// Rows [rows][kd] of an fp32 matrix, split between registers and stage; a
// thread takes 8 values of one row.  kd is a multiple of 4, the base is
// 16-byte aligned.
template <int R>
struct DSplit {
  using St = PStage<R, false>;
  struct Params {
    const float* p;
    uint32_t rows, kd, n;
  };
  struct Regs {
    f4 v[2];
  };
  static_assert(2 * R <= kThreads, "at most one group of 8 per thread");
  BRes b;
  uint32_t base, kd, k0;
  int slot;        // of the h part; -1: none
  uint32_t least;  // parts_key of the values stored as FINITE
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int t) {
    b.init(P.p, P.n);
    kd = P.kd;
    const int row = t / 2, half = t & 1;
    k0 = 8 * half;
    base = row < R && row0 + row < P.rows ? (row0 + row) * P.kd + k0 : kOob;
    slot = row < R ? row * 6 + (half ^ St::rhalf(row)) : -1;
    least = 0xffffffffu;
  }
  __device__ __forceinline__ void load(uint32_t kt, uint32_t ke, Regs& r) const {
    const uint32_t k = kt * 16 + k0, o = base + kt * 16;
    const bool ok = kt < ke && base != kOob;
    r.v[0] = b.ld4(ok && k < kd ? o : kOob);
    r.v[1] = b.ld4(ok && k + 4 < kd ? o + 4 : kOob);
  }
  template <bool FINITE>
  __device__ __forceinline__ void store(const Regs& r, char* S) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = r.v[e / 4][e % 4];
      if (FINITE) least = min(least, parts_key(x[e]));
    }
    uint4 q[3];
    split_parts8<FINITE>(x, q);
    if (slot < 0) return;
#pragma unroll
    for (int p = 0; p < 3; ++p) reinterpret_cast<uint4*>(S)[slot + 2 * p] = q[p];
  }
};

// As gemm_parts_tile, with both operands through registers and their loads two
// steps ahead: B streams from HBM, and with one step in flight (8 KB a
// workgroup) the latency of its loads would bound the kernel.
template <int MT, int NT>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
    k_dense_parts(const typename DSplit<MT>::Params pa, const typename DSplit<NT>::Params pb,
                  const EpiRowMajor::Params pe, TileGrid tg, uint32_t ktiles, uint32_t splits) {
  using LA = DSplit<MT>;
  using LB = DSplit<NT>;
  using SA = typename LA::St;
  using SB = typename LB::St;
  constexpr int WM = MT / 2, WN = NT / 2, FM = WM / 32, FN = WN / 32;
  constexpr int STAGE = SA::BYTES + SB::BYTES;
  __shared__ __attribute__((aligned(16))) char S[2 * STAGE];
  uint32_t mt, nt, z;
  tile_coords(tg, mt, nt, z);
  const uint32_t m0 = mt * MT, n0 = nt * NT;
  const uint32_t kb = uint32_t((uint64_t(ktiles) * z) / splits);
  const uint32_t ke = uint32_t((uint64_t(ktiles) * (z + 1)) / splits);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave / 2, wn = wave % 2;
  LA la;
  LB lb;
  la.init(pa, m0, tid);
  lb.init(pb, n0, tid);
  f16v acc[FM][FN];

  auto k_loop = [&](auto fp32) {
    constexpr bool FP32 = decltype(fp32)::value;
    f16v lo[FM][FN];
    parts_zero(acc);
    parts_zero(lo);
    typename LA::Regs ra[2];
    typename LB::Regs rb[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      la.load(kb + s, ke, ra[s]);
      lb.load(kb + s, ke, rb[s]);
    }
    la.template store<!FP32>(ra[0], S);
    lb.template store<!FP32>(rb[0], S + SA::BYTES);
    __syncthreads();
    // Step kt from stage `cur`, whose registers then take step kt + 2.
    auto step = [&](uint32_t kt, auto curc) {
      constexpr int cur = decltype(curc)::value;
      const char* Ac = S + cur * STAGE;
      la.load(kt + 2, ke, ra[cur]);
      lb.load(kt + 2, ke, rb[cur]);
      __builtin_amdgcn_sched_barrier(0);
      u4v a[FM][3], b[FN][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int j = 0; j < FN; ++j) b[j][p] = SB::frag(Ac + SA::BYTES, p, wn * WN + 32 * j, lane);
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i][p] = SA::frag(Ac, p, wm * WM + 32 * i, lane);
      }
      parts_mma<FP32>(a, b, acc, lo);
      la.template store<!FP32>(ra[cur ^ 1], S + (cur ^ 1) * STAGE);
      lb.template store<!FP32>(rb[cur ^ 1], S + (cur ^ 1) * STAGE + SA::BYTES);
      __syncthreads();
    };
    for (uint32_t kt = kb; kt < ke; kt += 2) {
      step(kt, std::integral_constant<int, 0>{});
      if (kt + 1 < ke) step(kt + 1, std::integral_constant<int, 1>{});
    }
    if constexpr (!FP32) parts_join(acc, lo);
  };
  k_loop(std::false_type{});
  if (__syncthreads_or(parts_bad(acc) || min(la.least, lb.least) < kTinyKey))
    k_loop(std::true_type{});
  parts_store<PEpiRowMajor>(pe, acc, m0 + wm * WM, n0 + wn * WN, z, lane);
}

struct DensePartsRun {
  const float *a, *b;
  float *c, *part;
  uint32_t M, K, N, ld, splits;
  template <int MT, int NT>
  int occ(bool) const {
    return occupancy(k_dense_parts<MT, NT>);
  }
  template <int MT, int NT>
  bool run() const {
    const uint32_t kt = cdiv(K, 16);
    const typename DSplit<MT>::Params pa{a, M, ld, M * ld};
    const typename DSplit<NT>::Params pb{b, N, ld, N * ld};
    const EpiRowMajor::Params pe{splits > 1 ? part : c, M, N, N, M * N};
    const TileGrid tg{cdiv(M, MT), cdiv(N, NT), xcd_order() ? 1u : 0u};
    hipLaunchKernelGGL((k_dense_parts<MT, NT>), dim3(tg.gm * tg.gn * splits), dim3(kThreads), 0,
                       stream(), pa, pb, pe, tg, kt, splits);
    return check_launch("gemm") && (splits == 1 || split_sum(part, c, M * N, splits));
  }
};
#define DCE_DENSE_TILES DCE_T(128, 128) DCE_T(128, 64) DCE_T(64, 128) DCE_T(64, 64)
template <class F>
static bool dense_dispatch(const TileCfg& c, F&& f) {
#define DCE_T(a, b) \
  if (c.MT == a && c.NT == b) return f.template run<a, b>();
  DCE_DENSE_TILES
#undef DCE_T
  set_error("gemm: unsupported tile %dx%d", c.MT, c.NT);
  return false;
}
template <class F>
static int dense_occ(const TileCfg& c, const F& f) {
#define DCE_T(a, b) \
  if (c.MT == a && c.NT == b) return f.template occ<a, b>(c.splits > 1);
  DCE_DENSE_TILES
#undef DCE_T
  return 1;
}

// More than one 64-row tile and at least 2e9 products: 96 x 4096 x 4096 41 and
// 41, 200 x 4096 x 4096 85 -> 64, 320 x 9000 x 700 (rows x columns x K) 57 ->
// 43, 512 x 1500 x 4096 64 -> 53 us; 256 x 2048 x 2048 (33 -> 34) and 200 x 700
// x 900 (12.5 -> 14.4 us) stay on fp32 MFMAs.  Over many rows the dot products
// have to be long as well: 500 x 4000 x 1200 loses (54 -> 59 us).
static bool dense_on_parts(uint32_t M, uint32_t K, uint32_t N, bool aT, bool bT) {
  return !aT && bT && M > 64 && K >= (M > 384 ? 2048u : 512u) && double(M) * N * K >= 2e9 &&
         size_t(M) * N < kOob;
}

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
  const bool parts = dense_on_parts(M, K, N, aT, bT);
  TileCfg cfg = parts ? parts_choose("DCE_TUNE_GEMM", M, N, K, 16, true,
                                     [&](const TileCfg& t) { return dense_occ(t, DensePartsRun{}); })
                      : choose("DCE_TUNE_GEMM", M, N, pad4(K), 16, true, gemm_occ);
  // A grid that leaves CUs idle (small GEMMs such as AlexNet's fc3) runs
  // faster on 64 x 64 tiles 32 deep, at split counts that fill the chip:
  // fc3 forward 34 -> 22 us, its dA 29 -> 24 us in a sweep of every tile
  // and split count on MI355X.
  const uint32_t cus = uint32_t(num_cus());
  auto wgs = [&](const TileCfg& t) {
    return cdiv(M, uint32_t(t.MT)) * cdiv(N, uint32_t(t.NT)) * t.splits;
  };
  if (!parts && !getenv("DCE_TUNE_GEMM") && wgs(cfg) < cus && M >= 64 && N >= 64) {
    const uint32_t kt32 = cdiv(pad4(K), 32u);
    TileCfg alt{64, 64, 32, 1};
    const uint32_t t64 = cdiv(M, 64u) * cdiv(N, 64u);
    // The fewest splits that fill every CU, keeping at least 8 K tiles each.
    while (t64 * alt.splits < cus && alt.splits < 16 && kt32 / (alt.splits + 1) >= 8) alt.splits++;
    if (wgs(alt) > wgs(cfg)) cfg = alt;
  }
  // A^T B over few rows (a linear layer's filter gradient): a 128 x 128 tile is
  // 16 steps at most, and a last batch of four workgroups a CU that is not full
  // costs as much as a full one.  64 x 128 tiles halve what is lost: 9216 x
  // 128 x 4096 (rows x K x columns; 2.25 batches) 106 -> 99 us, 5120 x 128 x
  // 4096 70 -> 57, 9216 x 250 x 1000 54 -> 46, 4608 x 37 x 4096 32 -> 25 us.
  // Grids that fill their batches stay (4096 x 128 x 4096 42 -> 44, 8192 x 250
  // x 4096 137 -> 139 us).  The order of every sum is the same.
  if (!getenv("DCE_TUNE_GEMM") && aT && !bT && K <= 256 && cfg.splits == 1 && cfg.MT == 128 &&
      cfg.NT == 128) {
    const uint32_t t = wgs(cfg), batch = cus * uint32_t(gemm_occ(cfg));
    if (double(cdiv(t, batch)) * batch > 1.1 * t) cfg.MT = 64;
  }
  // Skinny products with long dot products (a linear layer's forward and
  // input gradient at batch 128): 64 x 64 tiles 32 deep over about 1024
  // workgroups beat the 128 x 128 split-K choice (AlexNet fc1 forward 104 ->
  // 97 us, fc2 forward 56 -> 50 us, fc2 input gradient 53 -> 49 us in a sweep
  // of tiles and split counts on MI355X; wider grids, such as fc1's input
  // gradient with 288 such tiles, keep the model's choice).
  if (!parts && !getenv("DCE_TUNE_GEMM") && M <= 128 && pad4(K) >= 4096) {
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
    if (parts)
      ok = dense_dispatch(cfg, DensePartsRun{ap, bp, c, part, M, K, N, lda, cfg.splits});
    else if (!aT && !bT)
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
