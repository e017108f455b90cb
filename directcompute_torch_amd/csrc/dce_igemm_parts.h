// fp32 products on the bf16 matrix cores: the implicit GEMM of the
// convolutions' backward passes (dce_igemm_dw.hip, dce_igemm_dx.hip) and the
// linear layers' input gradient (dce_igemm_dense.hip).
//
// A float has a 24-bit significand and three bf16 have 3 x 8: x = h + m + l
// exactly, each part what the ones before it leave, rounded to nearest.  Of the
// nine part products the six largest are kept, as G. Henry, P. T. P. Tang and A.
// Heinecke do ("Leveraging the bfloat16 artificial intelligence datatype for
// higher-precision computations", 2019).  gfx950 runs bf16 MFMAs at 16 times the
// fp32 rate (1017 against 64 flops per cycle and SIMD), so six of them take 3/8
// of the fp32 MFMA's time.
//
// Nearest, because |m| <= 2^-8 |x| and |l| <= 2^-17 |x| then have either sign:
// the dropped m*l, l*m and l*l are at most 2^-24 of the product and average
// out.  Cut-off parts drop up to 2^-21, always towards zero: 4e-8 of the result
// at any length, and 2.4 times the fp32 error in sums of a few terms.
//
// The five smaller products have an accumulator of their own and the two are
// added once, at the end.  The large one then sums 16-bit products, whose low
// bits survive for many terms, and the small one's roundings are 2^-8 of the
// result's.  A bf16 MFMA cuts its addends off at the largest one's scale, always
// downwards: small products summed with the large ones drift by 3e-7 of the
// result over 2^17 steps.
//
// Error against float64 (2-norm, normal operands), with v_mfma_f32_16x16x4_f32
// and on parts: one product 2.5e-8 and 2.6e-8, 16 terms of 4096 6.3e-8 and
// 5.8e-8, 576 terms 4.1e-7 and 7.9e-8, 4096 4.4e-7 and 1.5e-7, 25088 in splits
// 2.1e-7 and 1.3e-7; gradients of which one value in 2000 survives a mask 5.6e-8
// and 5.6e-8 (dW), 2.9e-8 and 2.6e-8 (dX).
//
// The operands are split once, by the pass that re-lays them out anyway, and
// kept in memory as parts: the 16 channels of a block as 16 h, 16 m, 16 l (96
// bytes).  Split inside the GEMM instead, each element is split again for
// every tile that reads it, and the vector unit bounds the kernel: with the
// split after the LDS read 8.1 vector instructions per MFMA and the matrix
// unit 37 % busy (64 -> 128 channels, 56 x 56, b128: dW 433 us), with the split
// before the LDS write and one LDS stage 476 us, with fp32 MFMAs 495 us, split
// once and kept 343 us (matrix unit 50 % busy, address unit 73 %).
//
// An operand without three bf16 parts (infinite, NaN, so large that it rounds to
// infinity, or not zero and below 2^-110 = 8e-34) is kept as a NaN and its own
// two halves.  Such an operand, or a product that overflows, leaves a NaN or an
// infinity in the accumulator: that tile is computed again with fp32 MFMAs on
// the values themselves.
//
// The forward passes stay on fp32 MFMAs: their values decide ReLU masks and
// max-pool routes, so another rounding there sends a few gradient elements of
// every step another way.
#pragma once
#include "dce_igemm.h"

namespace dce {

using u4v = uint32_t __attribute__((ext_vector_type(4)));
using s4v = short __attribute__((ext_vector_type(4)));
using bf8 = __bf16 __attribute__((ext_vector_type(8)));
using f16v = float __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f16v mfma_bf16(const u4v& a, const u4v& b, const f16v& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a),
                                                 __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

constexpr uint32_t kBlkBytes = 96;               // 16 channels: h, m, l
constexpr uint32_t kOobBytes = kOob * 4u;

// ---------------------------------------------------------------------------
// LDS stage of one operand's 16-deep step, filled by direct 16-byte loads
// (slot s = thread + 256 * load):
//   ROWK  [row][6]             a row's h, m, l of 8 + 8 k, as in memory, so
//                              that consecutive lanes read 96-byte runs
//   KROW  [plane][k][R / 8]    a quad = 8 consecutive rows of one k, read
//                              back transposed (ds_read_b64_tr_b16)
// A fragment read should cover all 64 banks once: ROWK rows 8 apart (which
// share banks) hold their two k halves in opposite order, and KROW quads are
// XOR-swizzled by k, for the 32 rows at 4 k's of a transposed read.
// ---------------------------------------------------------------------------
template <int R, bool KROW>
struct PStage {
  static_assert(R == 32 || R == 64 || R == 128, "rows of a tile");
  static constexpr int QP = 2 * R;  // quads per part
  static constexpr int LOADS = (3 * QP + kThreads - 1) / kThreads;
  static constexpr int BYTES = 3 * QP * 16;
  static constexpr int RQ = R / 8;
  // Different source rows of a thread (ROWK: one per load), and load i's.
  static constexpr int UN = !KROW ? LOADS : QP > kThreads ? QP / kThreads : 1;
  __device__ static constexpr int un(int i) { return !KROW ? i : UN == 1 ? 0 : i % UN; }
  __device__ static __forceinline__ int swz(int k) {
    return R >= 128 ? 4 * (k & 3) : R == 64 ? 4 * ((k >> 1) & 1) : 0;
  }
  __device__ static __forceinline__ int rhalf(int row) { return (row >> 3) & 1; }
  // ROWK: row of thread t's load i, and byte in its 96-byte block.
  __device__ static __forceinline__ int row(int t, int i) { return (t + kThreads * i) / 6; }
  __device__ static __forceinline__ uint32_t byte(int t, int i) {
    const int s = t + kThreads * i, rw = s / 6;
    return uint32_t((s - 6 * rw) ^ rhalf(rw)) * 16;
  }
  // KROW: k and (swizzled back) row quad of the thread's source row un.
  __device__ static __forceinline__ int kk(int t, int u) { return (t + kThreads * u) % QP / RQ; }
  __device__ static __forceinline__ int rq(int t, int u) {
    return ((t + kThreads * u) % QP % RQ) ^ swz(kk(t, u));
  }
  __device__ static __forceinline__ uint32_t part(int t, int i) {
    if (!KROW) return 0;
    return QP % kThreads == 0 ? uint32_t(i / UN) : uint32_t((t + kThreads * i) / QP);
  }
  __device__ static __forceinline__ bool active(int t, int i) {
    return (3 * QP) % kThreads == 0 || t + kThreads * i < 3 * QP;
  }
  // Fragment: 32 rows from rb, 8 k per lane (k = 8 * (lane / 32) + e).
  __device__ static __forceinline__ u4v frag(const char* S, int p, int rb, int lane) {
    const int half = lane >> 5;
    if constexpr (!KROW) {
      const int rw = rb + (lane & 31);
      return *reinterpret_cast<const u4v*>(S + (rw * 6 + 2 * p + (half ^ rhalf(rw))) * 16);
    } else {
      const int j = lane & 15, col = rb + (lane & 16) + 4 * (j & 3);
      u4v v;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int k = 8 * half + 4 * e + (j >> 2);
        const int off = (p * QP + k * RQ + ((col >> 3) ^ swz(k))) * 16 + (col & 7) * 2;
        const s4v w = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s4v*)(S + off));
        const uint64_t u = __builtin_bit_cast(uint64_t, w);
        v[2 * e] = uint32_t(u);
        v[2 * e + 1] = uint32_t(u >> 32);
      }
      return v;
    }
  }
};

// Common to the loaders: off(kt, un) is the byte offset of the thread's quad
// (KROW: of its h part), or past the buffer for zeros.
template <int R, bool KROW>
struct PLoader {
  using St = PStage<R, KROW>;
  BRes b;
  int tid, wave;
  __device__ __forceinline__ void base_init(const float* p, uint32_t n, int t) {
    b.init(p, n);
    tid = t;
    wave = __builtin_amdgcn_readfirstlane(t >> 6);
  }
  template <class L>
  __device__ __forceinline__ void issue(const L& l, uint32_t kt, char* S) const {
    uint32_t o[St::UN];
#pragma unroll
    for (int u = 0; u < St::UN; ++u) o[u] = l.off(kt, u);
#pragma unroll
    for (int i = 0; i < St::LOADS; ++i) {
      if (!St::active(tid, i)) break;
      b.ld16_lds(o[St::un(i)] + St::part(tid, i) * 32u, S + (wave * 64 + i * kThreads) * 16);
    }
  }
};

// Dense rows [rows][kblk] (the filters).
template <int R>
struct PRows : PLoader<R, false> {
  using St = PStage<R, false>;
  static constexpr bool KROW = false;
  struct Params {
    const float* p;
    uint32_t rows, kblk, n;
  };
  uint32_t base[St::UN], kblk;
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int t) {
    this->base_init(P.p, P.n, t);
    kblk = P.kblk;
#pragma unroll
    for (int u = 0; u < St::UN; ++u) {
      const uint32_t row = row0 + St::row(t, u);
      base[u] = row < P.rows ? row * P.kblk * kBlkBytes + St::byte(t, u) : kOobBytes;
    }
  }
  __device__ __forceinline__ uint32_t off(uint32_t kt, int u) const {
    return kt < kblk && base[u] != kOobBytes ? base[u] + kt * kBlkBytes : kOobBytes;
  }
};

// G patches for dX at stride 1 (a layer, or a sub-pixel phase): rows = input
// pixels, K tile kt = (channel block, tap); LdPixRK's blocked order.
template <int R>
struct PPix : PLoader<R, false> {
  using St = PStage<R, false>;
  static constexpr bool KROW = false;
  struct Params {
    const float* src;
    uint32_t srcH, srcW, nblk, k, p, gridW, gridHW, N, n;
    FastDiv dGridHW, dGridW, dKK, dK;
    int pwd;  // the column origin is c + p + pwd
  };
  uint32_t srcH, srcW, nblk, k;
  FastDiv dKK, dK;
  uint32_t qbase[St::UN];
  int r0[St::UN], c0[St::UN];
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int t) {
    this->base_init(P.src, P.n, t);
    srcH = P.srcH;
    srcW = P.srcW;
    nblk = P.nblk;
    k = P.k;
    dKK = P.dKK;
    dK = P.dK;
#pragma unroll
    for (int u = 0; u < St::UN; ++u) {
      const uint32_t n = row0 + St::row(t, u);
      const uint32_t bb = fdiv(n, P.dGridHW), rem = n - bb * P.gridHW;
      const uint32_t a = fdiv(rem, P.dGridW), c = rem - a * P.gridW;
      r0[u] = n < P.N ? int(a + P.p) : (1 << 20);  // past the grid: no tap is in the image
      c0[u] = int(c + P.p) + P.pwd;
      // Offset of tap (0, 0), modulo 2^32 (the origin may lie in the padding).
      qbase[u] = (bb * P.srcH * P.srcW + uint32_t(r0[u]) * P.srcW + uint32_t(c0[u])) * P.nblk *
                     kBlkBytes +
                 St::byte(t, u);
    }
  }
  __device__ __forceinline__ uint32_t off(uint32_t kt, int u) const {
    const uint32_t cb = fdiv(kt, dKK), khw = kt - cb * dKK.d;
    const uint32_t kh = fdiv(khw, dK), kw = khw - kh * k;
    const int h = r0[u] - int(kh), w = c0[u] - int(kw);
    const bool ok = cb < nblk && uint32_t(h) < srcH && uint32_t(w) < srcW;
    return ok ? qbase[u] + (cb * kBlkBytes - (kh * srcW + kw) * nblk * kBlkBytes) : kOobBytes;
  }
};

// G rows for dW: rows = output channels, k = flat output pixel.
template <int R>
struct PGrad : PLoader<R, true> {
  using St = PStage<R, true>;
  static constexpr bool KROW = true;
  struct Params {
    const float* p;
    uint32_t nblk, npix, n;
  };
  uint32_t base[St::UN], kk[St::UN], npix, nblk;
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int t) {
    this->base_init(P.p, P.n, t);
    npix = P.npix;
    nblk = P.nblk;
#pragma unroll
    for (int u = 0; u < St::UN; ++u) {
      kk[u] = St::kk(t, u);
      const uint32_t col = row0 + 8u * St::rq(t, u);
      base[u] = col < P.nblk * 16 ? (kk[u] * P.nblk + col / 16) * kBlkBytes + ((col >> 3) & 1) * 16
                                  : kOobBytes;
    }
  }
  __device__ __forceinline__ uint32_t off(uint32_t kt, int u) const {
    return kt * 16 + kk[u] < npix && base[u] != kOobBytes
               ? base[u] + kt * (16 * nblk * kBlkBytes)
               : kOobBytes;
  }
};

// x taps for dW: rows n = (kh, kw, c), c over the padded channels; k = flat
// output pixel.
template <int R>
struct PTap : PLoader<R, true> {
  using St = PStage<R, true>;
  static constexpr bool KROW = true;
  struct Params {
    const float* x;
    uint32_t H, W, nblk, k, s, p, OW, OHW, npix, N, n;
    FastDiv dOHW, dOW, dC, dK;  // dC: 16 * nblk
  };
  uint32_t H, W, s, OW, OHW, npix, pixBytes;
  FastDiv dOHW, dOW;
  uint32_t chan[St::UN], kk[St::UN];
  int kh[St::UN], kw[St::UN];
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int t) {
    this->base_init(P.x, P.n, t);
    H = P.H;
    W = P.W;
    s = P.s;
    OW = P.OW;
    OHW = P.OHW;
    npix = P.npix;
    pixBytes = P.nblk * kBlkBytes;
    dOHW = P.dOHW;
    dOW = P.dOW;
#pragma unroll
    for (int u = 0; u < St::UN; ++u) {
      kk[u] = St::kk(t, u);
      const uint32_t n = row0 + 8u * St::rq(t, u);
      const uint32_t khw = fdiv(n, P.dC), c = n - khw * P.dC.d;
      const uint32_t a = fdiv(khw, P.dK);
      chan[u] = (c / 16) * kBlkBytes + ((c >> 3) & 1) * 16;
      // A row past the taps gets an offset no pixel can bring into the image.
      kh[u] = n < P.N ? int(a) - int(P.p) : -(1 << 20);
      kw[u] = int(khw - a * P.k) - int(P.p);
    }
  }
  __device__ __forceinline__ uint32_t off(uint32_t kt, int u) const {
    const uint32_t pix = kt * 16 + kk[u];
    const uint32_t bb = fdiv(pix, dOHW), rem = pix - bb * OHW;
    const uint32_t oh = fdiv(rem, dOW), ow = rem - oh * OW;
    const int ih = int(oh * s) + kh[u], iw = int(ow * s) + kw[u];
    const bool ok = pix < npix && uint32_t(ih) < H && uint32_t(iw) < W;
    return ok ? ((bb * H + uint32_t(ih)) * W + uint32_t(iw)) * pixBytes + chan[u] : kOobBytes;
  }
};

// ---------------------------------------------------------------------------
// Epilogues: a lane stores quads of four consecutive columns n of one row m
// (the MFMAs take the B fragment first and accumulate C transposed).
// ---------------------------------------------------------------------------
struct PEpiRowMajor {
  using Params = EpiRowMajor::Params;
  __device__ static __forceinline__ void quad(const Params& p, uint32_t m, uint32_t n, uint32_t z,
                                              const f4& v) {
    if (m >= p.M || n >= p.N) return;
    float* dst = p.c + size_t(z) * p.splitStride + size_t(m) * p.ldc + n;
    if (((p.ldc | p.splitStride) & 3) == 0 && n + 3 < p.N) {
      *reinterpret_cast<f4*>(dst) = v;
      return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.N) dst[e] = v[e];
  }
};
struct PEpiNCHW {
  using Params = EpiNCHW::Params;
  __device__ static __forceinline__ void quad(const Params& p, uint32_t m, uint32_t n, uint32_t,
                                              const f4& v) {
    if (m >= p.M || n >= p.N) return;
    uint32_t b = fdiv(n, p.dHW), pix = n - b * p.HW;
    if (pix + 3 < p.HW && n + 3 < p.N) {
      stu(p.out + (size_t(b) * p.M + m) * p.HW + pix, v);
      return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (n + e < p.N) p.out[(size_t(b) * p.M + m) * p.HW + pix] = v[e];
      if (++pix == p.HW) {
        pix = 0;
        ++b;
      }
    }
  }
};
struct PEpiPhase {
  using Params = EpiNCHWPhase::Params;
  __device__ static __forceinline__ void quad(const Params& p, uint32_t m, uint32_t n, uint32_t,
                                              const f4& v) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (m < p.M && n + e < p.N) p.out[EpiNCHWPhase::at(p, n + e, m)] = v[e];
  }
};

// hi + lo += a b for one 16-deep step: six bf16 products, or (FP32) the values put
// together again and multiplied in fp32, into hi alone.
template <bool FP32, int FM, int FN>
__device__ __forceinline__ void parts_mma(const u4v (&a)[FM][3], const u4v (&b)[FN][3],
                                          f16v (&hi)[FM][FN], f16v (&lo)[FM][FN]) {
  if constexpr (!FP32) {
    auto product = [&](int pb, int pa, f16v (&acc)[FM][FN]) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma_bf16(b[j][pb], a[i][pa], acc[i][j]);
    };
    product(1, 1, lo);
    product(0, 2, lo);
    product(2, 0, lo);
    product(0, 1, lo);
    product(1, 0, lo);
    product(0, 0, hi);
  } else {
    // Lane halves hold k = e and 8 + e: two k per fp32 MFMA.
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      auto word = [&](const u4v (&f)[3]) {
        uint32_t x[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) x[p] = e & 1 ? f[p][e / 2] & 0xffff0000u : f[p][e / 2] << 16;
        return parts_value(x[0], x[1], x[2]);
      };
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          hi[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(word(b[j]), word(a[i]), hi[i][j], 0, 0, 0);
    }
  }
}
template <int FM, int FN>
__device__ __forceinline__ void parts_zero(f16v (&acc)[FM][FN]) {
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
}
template <int FM, int FN>
__device__ __forceinline__ void parts_join(f16v (&hi)[FM][FN], const f16v (&lo)[FM][FN]) {
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) hi[i][j] += lo[i][j];
}
// Does the tile hold an infinity or a NaN?
template <int FM, int FN>
__device__ __forceinline__ bool parts_bad(const f16v (&acc)[FM][FN]) {
  // x * 0 is NaN for an infinity or a NaN.
  float bad = 0.f;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) bad = fmaf(acc[i][j][v], 0.f, bad);
  return bad != bad;
}
template <class EPI, int FM, int FN>
__device__ __forceinline__ void parts_store(const typename EPI::Params& pe, const f16v (&acc)[FM][FN],
                                            uint32_t m0, uint32_t n0, uint32_t z, int lane) {
  // Block (i, j): row m = lane % 32, columns 8q + 4 * (lane / 32) + 0 .. 3.
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        EPI::quad(pe, m0 + 32 * i + (lane & 31),
                  n0 + 32 * j + 8 * q + 4 * (lane >> 5), z,
                  f4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                     acc[i][j][4 * q + 3]});
}

// ---------------------------------------------------------------------------
// The kernel: 256 threads, waves 2 x 2 (1 x 4 when the tile is four times as
// wide as high, or 32 rows high) over an MT x NT tile of 32 x 32 blocks; K in
// steps of 16 through two LDS stages with one barrier per step, the next
// step's direct loads in flight while the current one is multiplied.
// ---------------------------------------------------------------------------
template <int MT, int NT, class LA, class LB>
struct PTile {
  static constexpr int BYTES = LA::St::BYTES + LB::St::BYTES;
};
template <int MT, int NT, class LA, class LB, class EPI>
__device__ __forceinline__ void gemm_parts_tile(char* S, const typename LA::Params& pa,
                                                const typename LB::Params& pb,
                                                const typename EPI::Params& pe, uint32_t m0,
                                                uint32_t n0, uint32_t z, uint32_t kb, uint32_t ke) {
  using SA = typename LA::St;
  using SB = typename LB::St;
  constexpr int WGM = MT == 32 ? 1 : 2, WGN = 4 / WGM;
  constexpr int WM = MT / WGM, WN = NT / WGN, FM = WM / 32, FN = WN / 32;
  static_assert(FM >= 1 && FN >= 1, "32 x 32 blocks");
  constexpr int STAGE = PTile<MT, NT, LA, LB>::BYTES;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, wm = wave / WGN, wn = wave % WGN;
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
    if (kb < ke) {
      la.issue(la, kb, S);
      lb.issue(lb, kb, S + SA::BYTES);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (uint32_t kt = kb; kt < ke; ++kt) {
      const int cur = int(kt - kb) & 1;
      const char* Ac = S + cur * STAGE;
      const char* Bc = Ac + SA::BYTES;
      // Fragments first: a direct load in flight would make the compiler
      // wait for it before any LDS read.
      u4v a[FM][3], b[FN][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int j = 0; j < FN; ++j) b[j][p] = SB::frag(Bc, p, wn * WN + 32 * j, lane);
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i][p] = SA::frag(Ac, p, wm * WM + 32 * i, lane);
      }
      if (kt + 1 < ke) {
        la.issue(la, kt + 1, S + (cur ^ 1) * STAGE);
        lb.issue(lb, kt + 1, S + (cur ^ 1) * STAGE + SA::BYTES);
      }
      parts_mma<FP32>(a, b, acc, lo);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
    if constexpr (!FP32) parts_join(acc, lo);
  };
  k_loop(std::false_type{});
  if (__syncthreads_or(parts_bad(acc))) k_loop(std::true_type{});
  parts_store<EPI>(pe, acc, m0 + wm * WM, n0 + wn * WN, z, lane);
}

template <int MT, int NT, class LA, class LB, class EPI>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
    k_gemm_parts(const typename LA::Params pa, const typename LB::Params pb,
                 const typename EPI::Params pe, TileGrid tg, uint32_t ktiles, uint32_t splits) {
  __shared__ __attribute__((aligned(16))) char S[2 * PTile<MT, NT, LA, LB>::BYTES];
  uint32_t mt, nt, z;
  tile_coords(tg, mt, nt, z);
  gemm_parts_tile<MT, NT, LA, LB, EPI>(S, pa, pb, pe, mt * MT, nt * NT, z,
                                       uint32_t((uint64_t(ktiles) * z) / splits),
                                       uint32_t((uint64_t(ktiles) * (z + 1)) / splits));
}

// Up to four products in one launch, as k_igemm_multi; their K in `splits`, the
// partials `zstride` floats apart.
template <int MT, int NT, class LA, class LB, class EPI>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
    k_gemm_parts_multi(const Multi<LA, LB, EPI> a, uint32_t wgs, uint32_t splits,
                       uint32_t zstride) {
  __shared__ __attribute__((aligned(16))) char S[2 * PTile<MT, NT, LA, LB>::BYTES];
  const uint32_t all = xcd_block_id(), z = all / wgs, id = all - z * wgs;
  typename LA::Params pa = a.pa[0];
  typename LB::Params pb = a.pb[0];
  typename EPI::Params pe = a.pe[0];
  uint32_t kt = a.ktiles[0], t = id;
#pragma unroll
  for (int i = 1; i < kMulti; ++i)
    if (id >= a.first[i]) {
      pa = a.pa[i];
      pb = a.pb[i];
      pe = a.pe[i];
      kt = a.ktiles[i];
      t = id - a.first[i];
    }
  pe.out += size_t(z) * zstride;
  gemm_parts_tile<MT, NT, LA, LB, EPI>(S, pa, pb, pe, t % a.gm * MT, t / a.gm * NT, 0,
                                       uint32_t((uint64_t(kt) * z) / splits),
                                       uint32_t((uint64_t(kt) * (z + 1)) / splits));
}

template <int MT, int NT, class LA, class LB, class EPI>
static bool launch_parts(const typename LA::Params& pa, const typename LB::Params& pb,
                         const typename EPI::Params& pe, uint32_t M, uint32_t N, uint32_t ktiles,
                         uint32_t splits, const char* what) {
  const TileGrid tg{cdiv(M, MT), cdiv(N, NT), xcd_order() ? 1u : 0u};
  hipLaunchKernelGGL((k_gemm_parts<MT, NT, LA, LB, EPI>), dim3(tg.gm * tg.gn * splits),
                     dim3(kThreads), 0, stream(), pa, pb, pe, tg, ktiles, splits);
  return check_launch(what);
}

#define DCE_PARTS_TILES \
  DCE_T(128, 128) DCE_T(128, 64) DCE_T(64, 128) DCE_T(64, 64) DCE_T(32, 128)
// Tile and split choice: the least estimated microseconds.  As est_us
// (dce_igemm.h), the workgroups spread evenly over the CUs and each CU runs its
// n in batches of at most the kernel's occupancy; a step (16 k) of a batch of r
// takes lat + r * step, fitted per tile to sweeps of the AlexNet and UNet
// layers and the 64 -> 128 channel 56 x 56 one: 128 x 128 takes 0.95 us alone
// on its CU and 1.40 us in pairs, 64 x 128 0.8 us in pairs and 1.4 us in fours,
// the small tiles 0.65 - 0.8 us up to three at a time.  The fits are from
// kernels that added the small products to the accumulator after every step;
// without those adds every tile is some 5 % faster, and the AlexNet layers
// reach 172 - 260 TFLOP/s with the choices made.
struct PartsTile {
  int MT, NT;
  double lat, step;
};
constexpr PartsTile kPartsTiles[] = {{128, 128, 0.50, 0.45}, {128, 64, 0.30, 0.28},
                                     {64, 128, 0.30, 0.28},  {64, 64, 0.35, 0.15},
                                     {32, 128, 0.50, 0.11}};
template <class OccFn>
static TileCfg parts_choose(const char* var, uint32_t M, uint32_t N, uint32_t kdim,
                            uint32_t max_splits, bool dense_out, OccFn&& occ) {
  const uint32_t ktiles = cdiv(kdim, 16), cus = uint32_t(num_cus());
  TileCfg o{0, 0, 16, 1};
  const bool tuned = tune_override(var, o);
  TileCfg best{128, 128, 16, 1};
  double bestT = 0;
  for (const auto& t : kPartsTiles) {
    TileCfg c{t.MT, t.NT, 16, 1};
    if (c.MT == 32 && M > 32) continue;
    // A tune override with a tile of the fp32 kernel sets the splits alone.
    bool have = false;
    for (const auto& u : kPartsTiles) have |= u.MT == o.MT && u.NT == o.NT;
    if (tuned && have && (c.MT != o.MT || c.NT != o.NT)) continue;
    const uint32_t tiles = cdiv(M, uint32_t(c.MT)) * cdiv(N, uint32_t(c.NT)), oc = uint32_t(occ(c));
    const uint32_t smax = std::max<uint32_t>(1, std::min(max_splits, ktiles / 8));
    for (uint32_t sp = 1; sp <= smax; ++sp) {
      if (tuned && sp != std::min(smax, o.splits)) continue;
      const uint32_t n = cdiv(tiles * sp, cus), full = n / oc, rem = n - full * oc;
      const double kps = double(ktiles) / sp;
      double T = kps * full * (t.lat + oc * t.step);
      if (rem) T += kps * (t.lat + rem * t.step);
      if (sp > 1 || !dense_out) T += 4.0 + 2.0 * sp * double(M) * N * 4.0 / kFinishBytesPerUs;
      if (bestT == 0 || T < bestT) {
        bestT = T;
        best = c;
        best.splits = sp;
      }
    }
  }
  if (const char* e = getenv("DCE_TUNE_LOG")) {
    if (*e && *e != '0')
      fprintf(stderr, "[dcengine] %s parts M=%u N=%u K=%u -> %dx%d splits %u (occupancy %d) est %.1f us\n",
              var, M, N, kdim, best.MT, best.NT, best.splits, occ(best), bestT);
  }
  return best;
}

template <class F>
static bool parts_dispatch(const TileCfg& c, F&& f) {
#define DCE_T(a, b) \
  if (c.MT == a && c.NT == b) return f.template run<a, b>();
  DCE_PARTS_TILES
#undef DCE_T
  set_error("igemm: unsupported tile %dx%d", c.MT, c.NT);
  return false;
}
template <class F>
static int parts_occ(const TileCfg& c, const F& f) {
#define DCE_T(a, b) \
  if (c.MT == a && c.NT == b) return f.template occ<a, b>(c.splits > 1);
  DCE_PARTS_TILES
#undef DCE_T
  return 1;
}

}  // namespace dce
