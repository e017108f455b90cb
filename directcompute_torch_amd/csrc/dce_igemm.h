// fp32 implicit GEMM on CDNA4 matrix cores (v_mfma_f32_16x16x4_f32) for the
// convolution forward, filter gradient (dW), input gradient (dX) and the
// flagged dense GEMM of MatMulAlloc.
//
//   C[m, n] = sum_k A[m, k] * B[n, k]
//
// Workgroup: 256 threads = 4 wave64 owning an MT x NT output tile: for MT in
// {64, 128} the waves sit 2x2, each with an (MT/2) x (NT/2) block of 16x16
// accumulators; for the narrow tiles MT in {16, 32} (few output channels)
// they sit 1x4, each with an MT x (NT/4) block, or (KT = 64) each wave takes
// the whole tile over its own 16-deep slice of every K tile.  K advances in
// tiles of KT (16, 32 or 64) through a double buffered LDS stage with one
// barrier per tile; the next tile's global loads are in flight while the
// current one is multiplied.
//
// Every global load is a (predicated) 16-byte load of four consecutive
// elements ("quad"), into registers or straight into LDS.  An operand is
// staged in LDS in one of two layouts:
//   ROWK  [row][k], quads along k  (row stride KT)       -> ds_read_b128
//   KROW  [k][row], quads along rows                     -> 4 x ds_read_b32
// Both feed the MFMA with the same k order: in MFMA s of a 16-wide k slice,
// lane l (r = l % 16, g = l / 16) supplies A[r][4g + s] and B[4g + s][r], so
// the four MFMAs together cover k 0..15 (the matrix unit sums over g).  ROWK
// rows are unpadded with their quads XOR-swizzled by row; KROW rows at least
// 64 wide are unpadded and swizzled by k where the loader allows it, the
// others padded by 4 floats (see Stage).  A wave with 2 or 4 fragments of a KROW operand
// interleaves them row by row, so that one ds_read_b64 / b128 per k serves
// all of them (Stage::frags_rif).
//
// Convolutions work on channel-innermost ("NHWC", channels padded to a
// multiple of 4) copies of their activations so that a quad is four
// consecutive channels of one pixel:
//   forward  A = filters [oc][(kh,kw,c)]      ROWK   B = x patches, rows = output pixels   ROWK
//   dX       A = filters [c][(kh,kw,oc)]      ROWK   B = G patches, rows = input pixels    ROWK
//   dW       A = G rows oc, k = pixels        KROW   B = x taps, rows (kh,kw,c), k = pixels KROW
// where G = dy masked by the ReLU output (y <= 0 -> 0), produced once per
// backward by a transpose pass that also reduces the bias gradient.  No
// im2col / col2im buffer exists; the NHWC copy of x is what ConvForwardFused
// hands back as its "im2col" handle.  Two layer kinds take other operands:
// pointwise (1x1, stride 1) layers multiply the NCHW planes in place, and
// layers with fewer than 4 input channels read a stride-phase copy of x
// (stride-phase section below).
// Split-K writes partial tiles (split z is the slowest index of the tile
// numbering) that a second pass sums in a fixed order; nothing uses atomics,
// so results are deterministic.
#pragma once
#include "dce_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <type_traits>

namespace dce {

constexpr int kThreads = 256;
static inline uint32_t cdiv(uint64_t a, uint64_t b) { return uint32_t((a + b - 1) / b); }

// ---------------------------------------------------------------------------
// LDS stage geometry of one operand.
// ---------------------------------------------------------------------------
template <int R, int KT, bool KROW, bool SWZOK = true>
struct Stage {
  // ROWK rows are KT floats, unpadded.  Measured with an LDS probe on gfx950
  // (64 banks): 16-byte stores of the loaders' ROWK pattern (KQ quads of
  // consecutive rows) run 15% slower with a +4 pad than without, while the
  // fragment reads (one quad of 16 consecutive rows) cost the same either way.
  // KROW rows of at least 64 floats (SWZ, when the loader opts in) are
  // unpadded too, with the row-quad index XOR-swizzled by k (fk): a fragment
  // read takes one float of 16 consecutive rows at 4 k's 4 apart, which the
  // swizzle spreads over all 64 banks (unswizzled, k rows R floats apart
  // would share banks).  Other KROW rows keep a +4 pad.  Unpadded stages take
  // direct global-to-LDS loads, the conv dW operands included (the G rows
  // and the per-quad tap rows of x: AlexNet's conv backward 112.3 -> 113.0
  // -> 113.7 TFLOP/s as each went direct).
  static constexpr bool SWZ = KROW && SWZOK && R >= 64;
  static constexpr int LD = KROW ? (SWZ ? R : R + 4) : KT;
  static constexpr int SIZE = KROW ? KT * LD : R * LD;
  static constexpr int KQ = KT / 4;
  static constexpr int RQ = R / 4;
  // NQ quads per stage.  A narrow operand (NQ < kThreads) is staged by the
  // first NQ threads, one quad each; the others load and store nothing.
  static constexpr int NQ = R * KT / 4;
  static_assert(NQ % kThreads == 0 || kThreads % NQ == 0, "tile must split evenly over the workgroup");
  static constexpr bool PART = NQ < kThreads;
  static constexpr int Q = PART ? 1 : NQ / kThreads;
  __device__ static __forceinline__ bool active(int t) { return !PART || t < NQ; }
  // Quad i of thread t.  ROWK: consecutive lanes take consecutive k-quads of
  // one row; KROW: consecutive lanes take consecutive row-quads of one k.
  // kThreads is a multiple of KQ and RQ, so quad i sits DROW rows (ROWK) or
  // DK k-steps (KROW) past quad 0, and DLDS floats past it in LDS.
  static constexpr int DROW = KROW ? 0 : kThreads / KQ;
  static constexpr int DK = KROW ? kThreads / RQ : 0;
  static constexpr int DLDS = KROW ? DK * LD : DROW * LD;
  // ROWK quad swizzle: logical k-quad q of row `row` sits at physical quad
  // q ^ fr(row).  A fragment read takes quad q of 16 consecutive rows; rows
  // are KT floats, so 64 / KT consecutive rows fill the 64 banks once and the
  // unswizzled quads of rows 64 / KT apart share banks (4-way conflicts at
  // KT = 16, 16-way at KT = 64).  fr spreads the 16 rows over all 64 banks.
  // Thread t still owns the 16-byte slot t of its row group (the direct
  // loads' lane order); it loads the logical quad that belongs there.
  static_assert(KROW || (KT <= 64 && 64 % KT == 0), "ROWK swizzle period");
  static_assert(KROW || Q == 1 || DROW % 16 == 0, "fr is periodic in 16 rows");
  __device__ static __forceinline__ int fr(int row) { return (row / (64 / KT)) % KQ; }
  __device__ static __forceinline__ int qrow(int t, int i) {
    return KROW ? 4 * (t % RQ) : t / KQ + DROW * i;
  }
  // Logical k offset of the data in thread t's quad i (DROW is a multiple of
  // fr's 16-row period, so it is the same for every i).
  __device__ static __forceinline__ int qk(int t, int i) {
    return KROW ? t / RQ + DK * i : 4 * ((t % KQ) ^ fr(t / KQ));
  }
  __device__ static __forceinline__ int lds_off(int t) {
    return KROW ? qk(t, 0) * LD + qrow(t, 0) : qrow(t, 0) * LD + 4 * (t % KQ);
  }
  // SWZ: logical row quad rq of k row k sits at physical quad rq ^ fk(k).
  __device__ static __forceinline__ int fk(int k) { return 4 * ((k >> 2) & 3); }
  // The logical first row of quad i of thread t (its physical slot is
  // lds_off(t) + i * DLDS): KROW rows are swizzled back from the slot.
  __device__ static __forceinline__ int qrow_data(int t, int i) {
    if (!SWZ) return qrow(t, i);
    return 4 * ((t % RQ) ^ fk(qk(t, i)));
  }
  static constexpr bool kRow = KROW;
  // KROW, F = 2 or 4 fragments read together ("row-interleaved"): fragment i
  // takes rows rb + F*rho + i (rho = 0..15), so lane (r, g) finds the F
  // fragments' values at k = kb + 4g + s in F consecutive floats of one k row
  // (inside one row quad, so the SWZ swizzle moves them together): one
  // ds_read_b64 / b128 per s instead of F ds_read_b32.  The epilogues map the
  // accumulator rows back (frow).
  template <int F>
  __device__ static __forceinline__ void frags_rif(const float* S, int rb, int r, int g, int kb,
                                                   f4 (&out)[F]) {
    static_assert(KROW && (F == 2 || F == 4), "row-interleaved fragments: KROW, F in {2, 4}");
    const int row = rb + F * r;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = kb + 4 * g + s;
      const float* p = S + k * LD + (SWZ ? 4 * ((row >> 2) ^ fk(k)) + (row & 3) : row);
      if constexpr (F == 4) {
        const f4 v = *reinterpret_cast<const f4*>(p);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i][s] = v[i];
      } else {
        const f2 v = *reinterpret_cast<const f2*>(p);
        out[0][s] = v[0];
        out[1][s] = v[1];
      }
    }
  }
  // MFMA operand of 16 rows starting at rb, k slice kb: components s = 0..3.
  __device__ static __forceinline__ f4 frag(const float* S, int rb, int r, int g, int kb) {
    if (!KROW) return *reinterpret_cast<const f4*>(S + (rb + r) * LD + 4 * ((kb / 4 + g) ^ fr(rb + r)));
    f4 v;
    const int row = rb + r;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = kb + 4 * g + s;
      v[s] = SWZ ? S[k * LD + 4 * ((row >> 2) ^ fk(k)) + (row & 3)] : S[k * LD + row];
    }
    return v;
  }
};

template <class St>
struct LoaderBase {
  static constexpr int Q = St::Q;
  // LDSD: the operand goes global -> LDS directly (buffer_load ... lds).  Only
  // the unpadded [row][k] stages qualify: there a wave's 64 quads of one load
  // are 64 consecutive 16-byte LDS slots in lane order (lds_off(t) = 4 t).
  static constexpr bool LDSD = false;
  // As the B operand: accumulate C transposed (MFMA B fragment first).
  static constexpr bool kTransAcc = false;
  int lds0, wbase;
  bool act;
  __device__ __forceinline__ void base_init(int tid) {
    lds0 = St::lds_off(tid);
    // Wave-uniform, so M0 of the direct loads is set with scalar arithmetic.
    wbase = __builtin_amdgcn_readfirstlane(St::lds_off(tid & ~63));
    act = St::active(tid);
  }
  __device__ __forceinline__ void store(float* S, const f4 (&r)[Q]) const {
    if (St::PART && !act) return;
#pragma unroll
    for (int i = 0; i < Q; ++i) *reinterpret_cast<f4*>(S + lds0 + i * St::DLDS) = r[i];
  }
};

__device__ __forceinline__ f4 zero4() { return f4{0.f, 0.f, 0.f, 0.f}; }

// ---------------------------------------------------------------------------
// Dense operands.  Preconditions (the host pads copies to meet them): 16-byte
// aligned base, ld % 4 == 0, and kdim (ROWK) / rows (KROW) a multiple of 4, so
// a quad is either wholly inside the matrix or wholly padding.
// ---------------------------------------------------------------------------
// [rows][kdim] row-major (ROWK).
template <int R, int KT>
struct LdDenseRK : LoaderBase<Stage<R, KT, false>> {
  using St = Stage<R, KT, false>;
  static constexpr bool KROW = false;
  using LoaderBase<St>::Q;
  struct Params {
    const float* p;
    uint32_t ld, rows, kdim, n;  // n: floats in the buffer
  };
  BRes b;
  uint32_t kdim, kq;
  uint32_t base[Q];
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int tid) {
    this->base_init(tid);
    b.init(P.p, P.n);
    kdim = P.kdim;
    kq = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t row = row0 + St::qrow(tid, i);
      base[i] = (this->act && row < P.rows) ? row * P.ld + kq : kOob;
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    const uint32_t k0 = kt * KT;
    const bool kok = k0 + kq < kdim;
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = b.ld4(kok ? base[i] + k0 : kOob);
  }
  static constexpr bool LDSD = true;
  __device__ __forceinline__ void issue_lds(uint32_t kt, float* S) const {
    if (St::PART && !this->act) return;  // whole waves (NQ is a multiple of 64)
    const uint32_t k0 = kt * KT;
    const bool kok = k0 + kq < kdim;
#pragma unroll
    for (int i = 0; i < Q; ++i) b.ld4_lds(kok ? base[i] + k0 : kOob, S + this->wbase + i * St::DLDS);
  }
};

// [kdim][rows] k-major (KROW).
template <int R, int KT>
struct LdDenseKR : LoaderBase<Stage<R, KT, true>> {
  using St = Stage<R, KT, true>;
  static constexpr bool KROW = true;
  using LoaderBase<St>::Q;
  struct Params {
    const float* p;
    uint32_t ld, rows, kdim, n;
  };
  BRes b;
  uint32_t kdim, ld, kk0;
  uint32_t base[Q];  // quad i's offset at k tile 0, or kOob for rows past the matrix
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int tid) {
    this->base_init(tid);
    b.init(P.p, P.n);
    kdim = P.kdim;
    ld = P.ld;
    kk0 = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t row = row0 + St::qrow_data(tid, i);
      base[i] = (this->act && row < P.rows) ? (kk0 + St::DK * i) * P.ld + row : kOob;
    }
  }
  __device__ __forceinline__ void offsets(uint32_t kt, uint32_t (&o)[Q]) const {
    const uint32_t k0 = kt * KT;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t k = k0 + kk0 + St::DK * i;
      o[i] = k < kdim ? base[i] + k0 * ld : kOob;
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = b.ld4(o[i]);
  }
  static constexpr bool LDSD = St::SWZ;
  __device__ __forceinline__ void issue_lds(uint32_t kt, float* S) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) b.ld4_lds(o[i], S + this->wbase + i * St::DLDS);
  }
};

// ---------------------------------------------------------------------------
// NCHW operands of the pointwise (1 x 1, stride 1, no padding) convolutions,
// read in place: a pixel n = b*HW + pix of channel ch is src[(b*Ch + ch)*HW
// + pix].  HW % 4 == 0, so four consecutive pixels (a quad) lie in one image.
// ---------------------------------------------------------------------------
// KROW: rows = pixels n, k = channel (zero for k >= Ch or n >= N).
struct NchwKRParams {
  const float* src;
  uint32_t Ch, HW, N, n;
  FastDiv dHW;
};
template <int R, int KT>
struct LdNchwKR : LoaderBase<Stage<R, KT, true>> {
  using St = Stage<R, KT, true>;
  static constexpr bool KROW = true;
  static constexpr bool kTransAcc = true;  // pixel columns: quad stores
  using LoaderBase<St>::Q;
  using Params = NchwKRParams;
  BRes b;
  uint32_t Ch, HW, kk0;
  uint32_t base[Q];  // quad i's offset at channel 0, or kOob past the pixels
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int tid) {
    this->base_init(tid);
    b.init(P.src, P.n);
    Ch = P.Ch;
    HW = P.HW;
    kk0 = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t n = row0 + St::qrow_data(tid, i);
      const uint32_t bb = fdiv(n, P.dHW);
      base[i] = (this->act && n < P.N) ? bb * P.Ch * P.HW + (n - bb * P.HW) : kOob;
    }
  }
  __device__ __forceinline__ void offsets(uint32_t kt, uint32_t (&o)[Q]) const {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t ch = kt * KT + kk0 + St::DK * i;
      o[i] = (base[i] != kOob && ch < Ch) ? base[i] + ch * HW : kOob;
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = b.ld4(o[i]);
  }
  static constexpr bool LDSD = St::SWZ;
  __device__ __forceinline__ void issue_lds(uint32_t kt, float* S) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) b.ld4_lds(o[i], S + this->wbase + i * St::DLDS);
  }
};

// ROWK: rows = channels, k = pixel n over the batch (the pointwise dW
// operands).  Row `onesRow` (when below R rows of the grid) reads 1 for
// every k < K, from a 4-float buffer of ones: the dW GEMM then yields the
// bias gradient, sum over k of the other operand, as its extra column.
struct NchwRKParams {
  const float* src;
  const float* ones;
  uint32_t Ch, HW, K, n, onesRow;
  FastDiv dHW;
};
template <int R, int KT>
struct LdNchwRK : LoaderBase<Stage<R, KT, false>> {
  using St = Stage<R, KT, false>;
  static constexpr bool KROW = false;
  using LoaderBase<St>::Q;
  using Params = NchwRKParams;
  BRes b, bo;
  uint32_t Ch, HW, K, kq;
  FastDiv dHW;
  uint32_t rowoff[Q];  // quad i's channel offset ch * HW, or kOob past the channels
  bool one[Q];
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int tid) {
    this->base_init(tid);
    b.init(P.src, P.n);
    bo.init(P.ones, 4);
    Ch = P.Ch;
    HW = P.HW;
    K = P.K;
    dHW = P.dHW;
    kq = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t r = row0 + St::qrow(tid, i);
      one[i] = this->act && r == P.onesRow;
      rowoff[i] = (this->act && r < P.Ch) ? r * P.HW : kOob;
    }
  }
  // The thread's quads share their k (ROWK): one image / pixel split per tile.
  __device__ __forceinline__ void offsets(uint32_t kt, uint32_t (&o)[Q]) const {
    const uint32_t k0 = kt * KT + kq;
    const uint32_t bb = fdiv(k0, dHW);
    const uint32_t img = bb * Ch * HW + (k0 - bb * HW);
#pragma unroll
    for (int i = 0; i < Q; ++i) o[i] = (rowoff[i] != kOob && k0 < K) ? img + rowoff[i] : kOob;
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    uint32_t o[Q];
    offsets(kt, o);
    const bool kin = kt * KT + kq < K;
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = one[i] ? bo.ld4(kin ? 0u : kOob) : b.ld4(o[i]);
  }
  static constexpr bool LDSD = true;
  __device__ __forceinline__ void issue_lds(uint32_t kt, float* S) const {
    if (St::PART && !this->act) return;  // whole waves (NQ is a multiple of 64)
    uint32_t o[Q];
    offsets(kt, o);
    const bool kin = kt * KT + kq < K;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      float* dst = S + this->wbase + i * St::DLDS;
      if (one[i])
        bo.ld4_lds(kin ? 0u : kOob, dst);
      else
        b.ld4_lds(o[i], dst);
    }
  }
};

// ---------------------------------------------------------------------------
// Pixel-row gather over an NHWC source (ROWK): rows = pixels of a grid
// (b, a, c); k runs over the taps (kh, kw) and the Cp source channels (Cp the
// padded channel count, Cp % 4 == 0) in one of two orders:
//   flat    (BLK false): k = (kh * k + kw) * Cp + ch;
//   blocked (BLK true, Cp % kCB == 0, KT == kCB):
//           k = (cb * KK + kh * k + kw) * kCB + ci, ch = cb * kCB + ci.
// The blocked order makes a K tile one tap of one channel block, so a block's
// slice of the source stays in L1 while all KK taps walk over it (the flat
// order re-fetches each source pixel once per tap when Cp is large).  Within
// a thread, all quads share their k (ROWK), so the tap decomposition is done
// once per K tile.
//   FWD: source = x, rows = output pixels, tap reads x[b, a*s + kh - p, c*s + kw - p].
//   !FWD (dX): source = G, rows = input pixels, tap reads G[b, oh, ow] with
//        oh*s == a + p - kh exactly (S1: s == 1, no divisibility test).
//        A strided dX runs as s*s sub-pixel phases, each an S1 gather over
//        its own grid of input pixels with nh x nw taps (k = nw) and the
//        column origin shifted by pwd (dx_phase_params).
// ---------------------------------------------------------------------------
constexpr int kCB = 16;

template <int R, int KT, bool FWD, bool S1, bool BLK>
struct LdPixRK : LoaderBase<Stage<R, KT, false>> {
  static_assert(!BLK || KT == kCB, "blocked order: one K tile per (channel block, tap)");
  static_assert(!Stage<R, KT, false>::PART, "pixel operands fill the workgroup");
  using St = Stage<R, KT, false>;
  static constexpr bool KROW = false;
  using LoaderBase<St>::Q;
  struct Params {
    const float* src;
    uint32_t srcH, srcW, Cp, k, s, p;
    uint32_t gridW, gridHW, N, kdim, n;
    FastDiv dGridHW, dGridW, dInner, dK;  // dInner: KK (blocked) or Cp (flat)
    int pwd;  // dX: the column origin is c + p + pwd (0 but for the sub-pixel phases)
  };
  // FAST (blocked order, forward or stride-1 dX): the K tile's tap and
  // channel block are wave-uniform, so a quad's source offset is a per-quad
  // constant qbase plus a uniform tap term -- no per-tile multiplies.
  static constexpr bool FAST = BLK && (FWD || S1);
  static constexpr bool kTransAcc = true;  // pixel columns: quad stores (measured faster)
  BRes b;
  uint32_t srcH, srcW, Cp, k, s, kdim, kq;
  FastDiv dInner, dK;
  uint32_t pbase[Q], qbase[Q];
  int r0[Q], c0[Q];
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int tid) {
    this->base_init(tid);
    b.init(P.src, P.n);
    srcH = P.srcH;
    srcW = P.srcW;
    Cp = P.Cp;
    k = P.k;
    s = P.s;
    kdim = P.kdim;
    dInner = P.dInner;
    dK = P.dK;
    kq = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t n = row0 + St::qrow(tid, i);
      const uint32_t bb = fdiv(n, P.dGridHW);
      const uint32_t rem = n - bb * P.gridHW;
      const uint32_t a = fdiv(rem, P.dGridW);
      const uint32_t c = rem - a * P.gridW;
      pbase[i] = bb * P.srcH * P.srcW;
      if (FWD) {
        r0[i] = int(a * P.s) - int(P.p);
        c0[i] = int(c * P.s) - int(P.p);
      } else {
        r0[i] = int(a + P.p);
        c0[i] = int(c + P.p) + P.pwd;
      }
      // A row past the grid gets an origin no tap can bring into the image.
      if (n >= P.N) r0[i] = FWD ? -(1 << 20) : (1 << 20);
      // Offset of tap (0, 0), channel kq, modulo 2^32 (the origin may lie
      // in the padding); only in-image taps are ever used.
      qbase[i] = (pbase[i] + uint32_t(r0[i]) * P.srcW + uint32_t(c0[i])) * P.Cp + kq;
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    uint32_t off[Q];
    offsets(kt, off);
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = b.ld4(off[i]);
  }
  static constexpr bool LDSD = true;
  __device__ __forceinline__ void issue_lds(uint32_t kt, float* S) const {
    uint32_t off[Q];
    offsets(kt, off);
#pragma unroll
    for (int i = 0; i < Q; ++i) b.ld4_lds(off[i], S + this->wbase + i * St::DLDS);
  }
  __device__ __forceinline__ void offsets(uint32_t kt, uint32_t (&o)[Q]) const {
    if constexpr (FAST) {
      const uint32_t cb = fdiv(kt, dInner);
      const uint32_t khw = kt - cb * dInner.d;
      const uint32_t kh = fdiv(khw, dK);
      const uint32_t kw = khw - kh * k;
      const bool kok = cb * kCB < Cp;  // Cp % kCB == 0: the whole tile or none
      const uint32_t tap = (kh * srcW + kw) * Cp;
      const uint32_t toff = FWD ? cb * kCB + tap : cb * kCB - tap;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int h = FWD ? r0[i] + int(kh) : r0[i] - int(kh);
        const int w = FWD ? c0[i] + int(kw) : c0[i] - int(kw);
        const bool ok = kok && uint32_t(h) < srcH && uint32_t(w) < srcW;
        o[i] = ok ? qbase[i] + toff : kOob;
      }
      return;
    }
    uint32_t khw, ch;
    bool kok;
    if (BLK) {
      const uint32_t cb = fdiv(kt, dInner);
      khw = kt - cb * dInner.d;
      ch = cb * kCB + kq;
      kok = ch < Cp;
    } else {
      const uint32_t kk0 = kt * KT + kq;
      khw = fdiv(kk0, dInner);
      ch = kk0 - khw * Cp;
      kok = kk0 < kdim;
    }
    const uint32_t kh = fdiv(khw, dK);
    const uint32_t kw = khw - kh * k;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      int h, w;
      bool ok = kok;
      if (FWD) {
        h = r0[i] + int(kh);
        w = c0[i] + int(kw);
      } else if (S1) {
        h = r0[i] - int(kh);
        w = c0[i] - int(kw);
      } else {
        const int hs = r0[i] - int(kh), ws = c0[i] - int(kw);
        ok = ok && hs >= 0 && ws >= 0;
        h = int(uint32_t(hs) / s);
        w = int(uint32_t(ws) / s);
        ok = ok && uint32_t(h) * s == uint32_t(hs) && uint32_t(w) * s == uint32_t(ws);
      }
      ok = ok && uint32_t(h) < srcH && uint32_t(w) < srcW;
      o[i] = ok ? (pbase[i] + uint32_t(h) * srcW + uint32_t(w)) * Cp + ch : kOob;
    }
  }
};

// ---------------------------------------------------------------------------
// dW operands (KROW, k = flat output pixel over the batch).
// ---------------------------------------------------------------------------
// A: G rows oc, element (oc, pix) = G_nhwc[pix*OCp + oc].
struct GradKRParams {
  const float* g;
  uint32_t OCp, npix, n;
};
template <int R, int KT>
struct LdGradKR : LoaderBase<Stage<R, KT, true>> {
  using St = Stage<R, KT, true>;
  static constexpr bool KROW = true;
  using LoaderBase<St>::Q;
  using Params = GradKRParams;
  BRes b;
  uint32_t OCp, npix, kk0;
  uint32_t base[Q];  // quad i's offset at k tile 0, or kOob for channels past OCp
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int tid) {
    this->base_init(tid);
    b.init(P.g, P.n);
    OCp = P.OCp;
    npix = P.npix;
    kk0 = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t oc = row0 + St::qrow_data(tid, i);
      base[i] = (this->act && oc < P.OCp) ? (kk0 + St::DK * i) * P.OCp + oc : kOob;
    }
  }
  __device__ __forceinline__ void offsets(uint32_t kt, uint32_t (&o)[Q]) const {
    const uint32_t p0 = kt * KT;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t pix = p0 + kk0 + St::DK * i;
      o[i] = pix < npix ? base[i] + p0 * OCp : kOob;
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = b.ld4(o[i]);
  }
  static constexpr bool LDSD = St::SWZ;
  __device__ __forceinline__ void issue_lds(uint32_t kt, float* S) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) b.ld4_lds(o[i], S + this->wbase + i * St::DLDS);
  }
};

// B: x taps, rows n = (kh, kw, c) (c fastest, Cp), element (n, pix) =
// x_nhwc[b, oh*s + kh - p, ow*s + kw - p, c] or 0 outside the image.
struct XTapParams {
  const float* x;
  uint32_t H, W, Cp, k, s, p, OW, OHW, npix, N, n;
  FastDiv dOHW, dOW, dCp, dK;
};
template <int R, int KT>
struct LdXTapKR : LoaderBase<Stage<R, KT, true>> {
  using St = Stage<R, KT, true>;
  static constexpr bool KROW = true;
  using LoaderBase<St>::Q;
  using Params = XTapParams;
  BRes b;
  uint32_t H, W, Cp, s, OW, OHW, npix, kk0;
  FastDiv dOHW, dOW;
  // Quad i's tap row: channel offset and tap origin (kh, kw); with the
  // swizzled stage the quads of one thread sit on different tap rows.
  uint32_t off[Q];
  int kh[Q], kw[Q];
  __device__ __forceinline__ void init(const Params& P, uint32_t row0, int tid) {
    this->base_init(tid);
    b.init(P.x, P.n);
    H = P.H;
    W = P.W;
    Cp = P.Cp;
    s = P.s;
    OW = P.OW;
    OHW = P.OHW;
    npix = P.npix;
    dOHW = P.dOHW;
    dOW = P.dOW;
    kk0 = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t n = row0 + St::qrow_data(tid, i);
      const uint32_t khw = fdiv(n, P.dCp);
      off[i] = n - khw * P.Cp;
      const uint32_t a = fdiv(khw, P.dK);
      kh[i] = int(a) - int(P.p);
      kw[i] = int(khw - a * P.k) - int(P.p);
      // A row past the taps (or a thread that stages nothing) gets an offset
      // no pixel can bring into the image.
      if (n >= P.N || !this->act) kh[i] = -(1 << 20);
    }
  }
  __device__ __forceinline__ void offsets(uint32_t kt, uint32_t (&o)[Q]) const {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t pix = kt * KT + kk0 + St::DK * i;
      const uint32_t bb = fdiv(pix, dOHW);
      const uint32_t rem = pix - bb * OHW;
      const uint32_t oh = fdiv(rem, dOW);
      const uint32_t ow = rem - oh * OW;
      const int ih = int(oh * s) + kh[i];
      const int iw = int(ow * s) + kw[i];
      const bool ok = pix < npix && uint32_t(ih) < H && uint32_t(iw) < W;
      o[i] = ok ? ((bb * H + uint32_t(ih)) * W + uint32_t(iw)) * Cp + off[i] : kOob;
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = b.ld4(o[i]);
  }
  static constexpr bool LDSD = St::SWZ;
  __device__ __forceinline__ void issue_lds(uint32_t kt, float* S) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) b.ld4_lds(o[i], S + this->wbase + i * St::DLDS);
  }
};

// ---------------------------------------------------------------------------
// Channel-packed source for convolutions over C < 4 channels: x copied by
// k_to_pk to [B][Hp][Wp][C] (Hp = H + 2p, Wp = W + 2p, zero border), and the
// unpadded tap order t = kh * kC + j with kC = k * C, j = kw * C + c (kdim =
// k * kC; the NHWC layout would pad C to 4 and waste up to 3/4 of the
// tap axis).  For every output pixel a kernel row's kC values are contiguous,
// so a quad of 4 consecutive t is one 16-byte load (4-byte aligned) unless it
// runs past the end of its kernel row (j + 3 >= kC): its tail then comes from
// a second load at the next kernel row, shifted so that element e lines up
// (from t's row origin + rowp - (kC - j)).  Tail elements past the last
// kernel row read as zeros.
// ---------------------------------------------------------------------------
struct PkParams {
  const float* src;
  uint32_t rowp, imgp, C, k, s, kC, kdim;  // rowp = Wp * C, imgp = Hp * Wp * C
  uint32_t OW, OHW, npix, n;               // n: floats in the copy
  FastDiv dOHW, dOW, dKC;
};

// Offset of output pixel pix's window origin in the packed copy.
__device__ __forceinline__ uint32_t pk_origin(const PkParams& P, uint32_t pix) {
  const uint32_t bb = fdiv(pix, P.dOHW);
  const uint32_t rem = pix - bb * P.OHW;
  const uint32_t oh = fdiv(rem, P.dOW);
  const uint32_t ow = rem - oh * P.OW;
  return bb * P.imgp + oh * P.s * P.rowp + ow * P.s * P.C;
}

// Quad of taps t..t+3 at a window origin: o1 = t's offset from the origin,
// o2 = the shifted next-row offset (kOob: none), m = elements left in t's row.
__device__ __forceinline__ f4 pk_quad(const BRes& b, bool ok, uint32_t org, uint32_t o1,
                                      uint32_t o2, uint32_t m) {
  f4 v = b.ld4(ok && o1 != kOob ? org + o1 : kOob);
  if (m < 4) {
    const f4 w = b.ld4(ok && o2 != kOob ? org + o2 : kOob);
#pragma unroll
    for (int e = 1; e < 4; ++e)
      if (uint32_t(e) >= m) v[e] = w[e];
  }
  return v;
}

// Row-origin offsets of tap t (shared by the two loaders below).
__device__ __forceinline__ void pk_tap(const PkParams& P, uint32_t t, uint32_t& o1, uint32_t& o2,
                                       uint32_t& m) {
  if (t >= P.kdim) {
    o1 = o2 = kOob;
    m = 4;
    return;
  }
  const uint32_t kh = fdiv(t, P.dKC), j = t - kh * P.kC;
  m = P.kC - j;
  o1 = kh * P.rowp + j;
  o2 = (m < 4 && kh + 1 < P.k) ? (kh + 1) * P.rowp - m : kOob;
}

// Forward B operand (ROWK): rows = output pixels, k = packed taps.  All quads
// of a thread share their taps, so the tap split is done once per K tile.
template <int R, int KT>
struct LdPkRK : LoaderBase<Stage<R, KT, false>> {
  static_assert(!Stage<R, KT, false>::PART, "pixel operands fill the workgroup");
  using St = Stage<R, KT, false>;
  static constexpr bool KROW = false;
  using LoaderBase<St>::Q;
  using Params = PkParams;
  BRes b;
  PkParams P;
  uint32_t kq;
  uint32_t org[Q];
  bool ok[Q];
  __device__ __forceinline__ void init(const Params& p, uint32_t row0, int tid) {
    this->base_init(tid);
    P = p;
    b.init(p.src, p.n);
    kq = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t pix = row0 + St::qrow(tid, i);
      ok[i] = pix < p.npix;
      org[i] = ok[i] ? pk_origin(p, pix) : 0u;
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    uint32_t o1, o2, m;
    pk_tap(P, kt * KT + kq, o1, o2, m);
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = pk_quad(b, ok[i], org[i], o1, o2, m);
  }
};

// dW operand (KROW): rows = packed taps, k = output pixels.  A thread's quads
// keep their taps for the whole K loop; the pixel walks.
template <int R, int KT>
struct LdPkKR : LoaderBase<Stage<R, KT, true, false>> {
  using St = Stage<R, KT, true, false>;
  static constexpr bool KROW = true;
  using LoaderBase<St>::Q;
  using Params = PkParams;
  BRes b;
  PkParams P;
  uint32_t kk0;
  uint32_t o1[Q], o2[Q], m[Q];
  __device__ __forceinline__ void init(const Params& p, uint32_t row0, int tid) {
    this->base_init(tid);
    P = p;
    b.init(p.src, p.n);
    kk0 = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      pk_tap(p, this->act ? row0 + St::qrow_data(tid, i) : p.kdim, o1[i], o2[i], m[i]);
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t pix = kt * KT + kk0 + St::DK * i;
      const bool ok = pix < P.npix;
      r[i] = pk_quad(b, ok, ok ? pk_origin(P, pix) : 0u, o1[i], o2[i], m[i]);
    }
  }
};

// ---------------------------------------------------------------------------
// Stride-phase copy for convolutions over C < 4 channels with stride S <= 4
// (k_to_ps): xs[((b*Hp + r)*C + c)*S + ph][col] = x[b][c][r - p][col*S + ph
// - p] (zero outside the image), rows of Ncol floats (Ncol % 4 == 0), Hp =
// H + 2p.  The output pixels form a padded grid (b, oh, ow) with ow < OWp =
// pad4(OW); the extra columns are computed and dropped (their G is zero).
// Tap t = (c*k + kh)*k + kw of output pixel (b, oh, ow) reads
//   xs[pixel part (b*Hp + oh*S)*RS + ow] + [tap part (kh*C + c)*S*Ncol +
//   (kw % S)*Ncol + kw / S],  RS = C*S*Ncol,
// so four consecutive output pixels of one tap are four consecutive floats:
// a quad never straddles anything (taps or pixels), unlike the channel-packed
// layout whose tap quads straddle kernel rows.  Quads start at 4-byte
// alignment (kw / S); the GPU runs with unaligned access enabled.
// ---------------------------------------------------------------------------
struct PsParams {
  const float* src;
  uint32_t RS, Hp, S, Ncol, C, k, KK, kdim;  // kdim = C*KK taps
  uint32_t OWp, OHWp, npix, n;               // npix = B*OHWp padded pixels; n: floats
  FastDiv dOHWp, dOWp, dKK, dK, dS;
};

__device__ __forceinline__ uint32_t ps_pixel(const PsParams& P, uint32_t n) {
  const uint32_t b = fdiv(n, P.dOHWp), rem = n - b * P.OHWp;
  const uint32_t oh = fdiv(rem, P.dOWp), ow = rem - oh * P.OWp;
  return (b * P.Hp + oh * P.S) * P.RS + ow;
}
__device__ __forceinline__ uint32_t ps_tap(const PsParams& P, uint32_t t) {
  const uint32_t c = fdiv(t, P.dKK), r = t - c * P.KK;
  const uint32_t kh = fdiv(r, P.dK), kw = r - kh * P.k;
  const uint32_t cq = fdiv(kw, P.dS), ph = kw - cq * P.S;
  return ((kh * P.C + c) * P.S + ph) * P.Ncol + cq;
}

// Forward B operand (KROW): rows = padded output pixels, k = taps.  A
// thread's quads share one row quad (4 pixels, fixed for the K loop).
template <int R, int KT>
struct LdPsKR : LoaderBase<Stage<R, KT, true, false>> {
  using St = Stage<R, KT, true, false>;
  static constexpr bool KROW = true;
  static constexpr bool kTransAcc = true;  // pixel columns: quad stores (measured faster)
  using LoaderBase<St>::Q;
  using Params = PsParams;
  BRes b;
  PsParams P;
  uint32_t kk0, pbase;
  __device__ __forceinline__ void init(const Params& p, uint32_t row0, int tid) {
    this->base_init(tid);
    P = p;
    b.init(p.src, p.n);
    kk0 = St::qk(tid, 0);
    const uint32_t n0 = row0 + St::qrow_data(tid, 0);
    pbase = (this->act && n0 < p.npix) ? ps_pixel(p, n0) : kOob;
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t t = kt * KT + kk0 + St::DK * i;
      r[i] = b.ld4(pbase != kOob && t < P.kdim ? pbase + ps_tap(P, t) : kOob);
    }
  }
};

// dW operand (ROWK): rows = taps (fixed per thread), k = padded pixels.
template <int R, int KT>
struct LdPsRK : LoaderBase<Stage<R, KT, false>> {
  using St = Stage<R, KT, false>;
  static constexpr bool KROW = false;
  using LoaderBase<St>::Q;
  using Params = PsParams;
  BRes b;
  PsParams P;
  uint32_t kq;
  uint32_t toff[Q];
  __device__ __forceinline__ void init(const Params& p, uint32_t row0, int tid) {
    this->base_init(tid);
    P = p;
    b.init(p.src, p.n);
    kq = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t t = row0 + St::qrow(tid, i);
      toff[i] = (this->act && t < p.kdim) ? ps_tap(p, t) : kOob;
    }
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    const uint32_t k0 = kt * KT + kq;
    const uint32_t pb = k0 < P.npix ? ps_pixel(P, k0) : kOob;
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = b.ld4(pb != kOob && toff[i] != kOob ? pb + toff[i] : kOob);
  }
};

// dW operand (ROWK, direct to LDS): rows = output channels, k = padded
// pixels of the masked gradient G_pad[b][oc][oh][OWp] (k_mask_pad).  OHWp is
// a multiple of 4, so a pixel quad is 16-byte aligned and inside one image.
struct GPadParams {
  const float* g;
  uint32_t OC, OHWp, npix, n;
  FastDiv dOHWp;
};
template <int R, int KT>
struct LdGPadRK : LoaderBase<Stage<R, KT, false>> {
  using St = Stage<R, KT, false>;
  static constexpr bool KROW = false;
  using LoaderBase<St>::Q;
  using Params = GPadParams;
  BRes b;
  GPadParams P;
  uint32_t kq;
  uint32_t ocoff[Q];
  __device__ __forceinline__ void init(const Params& p, uint32_t row0, int tid) {
    this->base_init(tid);
    P = p;
    b.init(p.g, p.n);
    kq = St::qk(tid, 0);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const uint32_t oc = row0 + St::qrow(tid, i);
      ocoff[i] = (this->act && oc < p.OC) ? oc * p.OHWp : kOob;
    }
  }
  __device__ __forceinline__ void offsets(uint32_t kt, uint32_t (&o)[Q]) const {
    const uint32_t k0 = kt * KT + kq;
    const uint32_t bb = fdiv(k0, P.dOHWp);
    const uint32_t base = k0 < P.npix ? bb * P.OC * P.OHWp + (k0 - bb * P.OHWp) : kOob;
#pragma unroll
    for (int i = 0; i < Q; ++i) o[i] = base != kOob && ocoff[i] != kOob ? base + ocoff[i] : kOob;
  }
  __device__ __forceinline__ void load(uint32_t kt, f4 (&r)[Q]) const {
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) r[i] = b.ld4(o[i]);
  }
  static constexpr bool LDSD = true;
  __device__ __forceinline__ void issue_lds(uint32_t kt, float* S) const {
    if (St::PART && !this->act) return;  // whole waves (NQ is a multiple of 64)
    uint32_t o[Q];
    offsets(kt, o);
#pragma unroll
    for (int i = 0; i < Q; ++i) b.ld4_lds(o[i], S + this->wbase + i * St::DLDS);
  }
};

// ---------------------------------------------------------------------------
// Epilogues.  The accumulator layout depends on the MFMA operand order, a
// per-kernel choice (TACC, a trait of the B loader: whichever measured faster
// for that kernel's instruction schedule).  Lane l of wave (wm, wn) holds,
// for block (i, j) and register v, with r = l % 16, g = l / 16:
//   TACC false:  C[m0 + wm*16FM + 16i + 4g + v][n0 + wn*16FN + 16j + r]
//                (four consecutive rows of one column: four scalar stores);
//   TACC true:   C[m0 + wm*16FM + 16i + r][n0 + wn*16FN + 16j + 4g + v]
//                (B fragment first: four consecutive columns of one row,
//                 16 contiguous bytes of a row-major C: one quad store).
// With row-interleaved fragments (RA for the A operand, RB for B; see
// Stage::frags_rif) the wave-local row 16i + rho of fragment i becomes
// F*rho + i (frow).  RB is only used without TACC: lane (r, g) then holds FN
// consecutive columns FN*r .. FN*r + FN - 1 of each of its rows (j = 0 ..
// FN - 1), which EpiRowMajor stores as one FN-float vector.
// ---------------------------------------------------------------------------
template <bool RIF, int F>
__device__ __forceinline__ uint32_t frow(int i, int rho) {
  return RIF ? uint32_t(F * rho + i) : uint32_t(16 * i + rho);
}
__device__ __forceinline__ float epi_act(float z, uint32_t act) {
  if (act == 1) return fmaxf(z, 0.f);
  if (act == 2) return tanhf(z);
  return z;
}

struct EpiRowMajor {
  struct Params {
    float* c;
    uint32_t M, N, ldc, splitStride;
  };
  template <int MT, int NT, int FM, int FN, bool TACC, bool RA, bool RB>
  __device__ static __forceinline__ void store(const Params& p, const f4 (&acc)[FM][FN],
                                               uint32_t m0, uint32_t n0, uint32_t z, int wm,
                                               int wn, int lane) {
    float* c = p.c + size_t(z) * p.splitStride;
    const int r = lane & 15, g = lane >> 4;
    if constexpr (!TACC && RB) {
      // FN consecutive columns per row: one FN-float store (rows aligned to
      // FN floats, uniform over the launch).
      const bool vec = ((p.ldc | p.splitStride) & (FN - 1)) == 0 &&
                       (reinterpret_cast<uintptr_t>(p.c) & (4 * FN - 1)) == 0;
      const uint32_t n = n0 + wn * (FN * 16) + FN * r;
      if (n >= p.N) return;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const uint32_t m = m0 + wm * (FM * 16) + frow<RA, FM>(i, 4 * g + v);
          if (m >= p.M) continue;
          float* dst = c + size_t(m) * p.ldc + n;
          if (vec && n + FN - 1 < p.N) {
            if constexpr (FN == 4)
              *reinterpret_cast<f4*>(dst) = f4{acc[i][0][v], acc[i][1][v], acc[i][2][v], acc[i][3][v]};
            else
              *reinterpret_cast<f2*>(dst) = f2{acc[i][0][v], acc[i][1][v]};
          } else {
#pragma unroll
            for (int j = 0; j < FN; ++j)
              if (n + j < p.N) dst[j] = acc[i][j][v];
          }
        }
      }
      return;
    }
    if constexpr (!TACC) {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const uint32_t n = n0 + wn * (FN * 16) + j * 16 + r;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const uint32_t m = m0 + wm * (FM * 16) + frow<RA, FM>(i, 4 * g + v);
            if (m < p.M && n < p.N) c[m * p.ldc + n] = acc[i][j][v];
          }
        }
      }
      return;
    }
    // Quad stores need 16-byte aligned rows (uniform over the launch).
    const bool vec =
        ((p.ldc | p.splitStride) & 3) == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15) == 0;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const uint32_t m = m0 + wm * (FM * 16) + frow<RA, FM>(i, r);
      if (m >= p.M) continue;
      float* row = c + size_t(m) * p.ldc;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const uint32_t n = n0 + wn * (FN * 16) + j * 16 + 4 * g;
        if (vec && n + 3 < p.N) {
          *reinterpret_cast<f4*>(row + n) = acc[i][j];
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (n + v < p.N) row[n + v] = acc[i][j][v];
        }
      }
    }
  }
};

// NCHW output: out[b][m][pix] for n = b*HW + pix; optional bias + activation
// (0 identity, 1 ReLU, 2 tanh), as nn_conv_reshape.hlsl:23-26.  With TACC a
// lane's four columns are four consecutive pixels of one plane unless they
// cross an image boundary; the quad is stored at 4-byte alignment (planes of
// odd size; unaligned access is on).
struct EpiNCHW {
  struct Params {
    float* out;
    const float* bias;
    uint32_t M, HW, N, act;
    FastDiv dHW;
  };
  template <int MT, int NT, int FM, int FN, bool TACC, bool RA, bool RB>
  __device__ static __forceinline__ void store(const Params& p, const f4 (&acc)[FM][FN],
                                               uint32_t m0, uint32_t n0, uint32_t, int wm,
                                               int wn, int lane) {
    const int r = lane & 15, g = lane >> 4;
    if constexpr (!TACC) {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const uint32_t n = n0 + wn * (FN * 16) + frow<RB, FN>(j, r);
        const uint32_t b = fdiv(n, p.dHW);
        const uint32_t base = b * p.M * p.HW + (n - b * p.HW);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const uint32_t m = m0 + wm * (FM * 16) + frow<RA, FM>(i, 4 * g + v);
            if (m < p.M && n < p.N)
              p.out[base + m * p.HW] = epi_act(acc[i][j][v] + (p.bias ? p.bias[m] : 0.f), p.act);
          }
        }
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const uint32_t n = n0 + wn * (FN * 16) + j * 16 + 4 * g;
      if (n >= p.N) continue;
      const uint32_t b = fdiv(n, p.dHW);
      const uint32_t pix = n - b * p.HW;
      const bool quad = pix + 3 < p.HW && n + 3 < p.N;
      const size_t base = size_t(b) * p.M * p.HW + pix;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const uint32_t m = m0 + wm * (FM * 16) + frow<RA, FM>(i, r);
        if (m >= p.M) continue;
        const float bias = p.bias ? p.bias[m] : 0.f;
        f4 z;
#pragma unroll
        for (int v = 0; v < 4; ++v) z[v] = epi_act(acc[i][j][v] + bias, p.act);
        if (quad) {
          stu(p.out + base + size_t(m) * p.HW, z);
        } else {
          uint32_t bb = b, pp = pix;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            if (n + v < p.N) p.out[(size_t(bb) * p.M + m) * p.HW + pp] = z[v];
            if (++pp == p.HW) {
              pp = 0;
              ++bb;
            }
          }
        }
      }
    }
  }
};

// NCHW output over a padded pixel grid (n = b*OHWp + oh*OWp + ow, ow < OWp,
// OWp % 4 == 0, so a TACC lane's four columns share one padded row): columns
// with ow >= OW are dropped; otherwise as EpiNCHW.
struct EpiNCHWPad {
  struct Params {
    float* out;
    const float* bias;
    uint32_t M, OHW, OW, OWp, OHWp, N, act;
    FastDiv dOHWp, dOWp;
  };
  template <int MT, int NT, int FM, int FN, bool TACC, bool RA, bool RB>
  __device__ static __forceinline__ void store(const Params& p, const f4 (&acc)[FM][FN],
                                               uint32_t m0, uint32_t n0, uint32_t, int wm,
                                               int wn, int lane) {
    static_assert(!(TACC && RB), "row-interleaved B fragments are not used with TACC");
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const uint32_t n = n0 + wn * (FN * 16) + (TACC ? j * 16 + 4 * g : frow<RB, FN>(j, r));
      const uint32_t b = fdiv(n, p.dOHWp), rem = n - b * p.OHWp;
      const uint32_t oh = fdiv(rem, p.dOWp), ow = rem - oh * p.OWp;
      if (n >= p.N || ow >= p.OW) continue;
      const size_t base = size_t(b) * p.M * p.OHW + oh * p.OW + ow;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        if constexpr (!TACC) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const uint32_t m = m0 + wm * (FM * 16) + frow<RA, FM>(i, 4 * g + v);
            if (m < p.M)
              p.out[base + size_t(m) * p.OHW] =
                  epi_act(acc[i][j][v] + (p.bias ? p.bias[m] : 0.f), p.act);
          }
        } else {
          const uint32_t m = m0 + wm * (FM * 16) + frow<RA, FM>(i, r);
          if (m >= p.M) continue;
          const float bias = p.bias ? p.bias[m] : 0.f;
          f4 z;
#pragma unroll
          for (int v = 0; v < 4; ++v) z[v] = epi_act(acc[i][j][v] + bias, p.act);
          float* dst = p.out + base + size_t(m) * p.OHW;
          if (ow + 3 < p.OW) {
            stu(dst, z);
          } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
              if (ow + v < p.OW) dst[v] = z[v];
          }
        }
      }
    }
  }
};

// One sub-pixel phase of a strided dX: columns n = b*GHW + a*GW + c of the
// phase's pixel grid go to out[b][m][ph + s*a][pw + s*c] (NCHW, H x W
// planes).  Consecutive columns land s floats apart, so every value is its
// own store.
struct EpiNCHWPhase {
  struct Params {
    float* out;
    uint32_t M, H, W, GW, GHW, N, s, ph, pw;
    FastDiv dGHW, dGW;
  };
  __device__ static __forceinline__ size_t at(const Params& p, uint32_t n, uint32_t m) {
    const uint32_t b = fdiv(n, p.dGHW), rem = n - b * p.GHW;
    const uint32_t a = fdiv(rem, p.dGW), c = rem - a * p.GW;
    return (size_t(b) * p.M + m) * p.H * p.W + size_t(p.ph + p.s * a) * p.W + p.pw + p.s * c;
  }
  template <int MT, int NT, int FM, int FN, bool TACC, bool RA, bool RB>
  __device__ static __forceinline__ void store(const Params& p, const f4 (&acc)[FM][FN],
                                               uint32_t m0, uint32_t n0, uint32_t, int wm,
                                               int wn, int lane) {
    static_assert(!(TACC && RB), "row-interleaved B fragments are not used with TACC");
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          // TACC: row 16i + r, column 16j + 4g + v; else row 16i + 4g + v, column 16j + r
          const uint32_t m = m0 + wm * (FM * 16) + (TACC ? frow<RA, FM>(i, r) : frow<RA, FM>(i, 4 * g + v));
          const uint32_t n = n0 + wn * (FN * 16) + (TACC ? j * 16 + 4 * g + v : frow<RB, FN>(j, r));
          if (m < p.M && n < p.N) p.out[at(p, n, m)] = acc[i][j][v];
        }
  }
};

// EpiNCHW that also leaves the batch-norm statistics of the values it stores:
// for each output row m (a channel) the sums of z and z*z over the tile's
// columns below N, as doubles at stats[(m * pieces + nt) * 2 + {0, 1}] with
// nt the tile's column index: one piece per column tile, the layout of the
// BN statistics' partial sums.  The transposed-accumulation form only (the
// pixel and pointwise GEMMs): a lane's row is fixed per fragment, so it
// stores each quad as EpiNCHW does and adds its (at most 16) values of the
// row in float; the lanes' float pairs go to LDS (the A stages, free after
// the main loop's last barrier) and after one barrier a thread per row adds
// them in double in a fixed order (the same bits on every run).  The row's
// bias is loaded once for both uses.
struct EpiNCHWStats {
  static constexpr bool kStats = true;
  struct Params {
    EpiNCHW::Params o;
    double* stats;
    uint32_t pieces;
  };
  // All WGN waves of the workgroup call this.  lds: WGN * 4 * MT float2.
  template <int MT, int NT, int FM, int FN, bool TACC, bool RA, bool RB, int WGN>
  __device__ static __forceinline__ void store_stats(const Params& p, const f4 (&acc)[FM][FN],
                                                     uint32_t m0, uint32_t n0, int wm, int wn,
                                                     int lane, float* lds) {
    static_assert(TACC && WGN > 1, "pixel-column GEMMs with several waves per row block");
    const EpiNCHW::Params& o = p.o;
    const int r = lane & 15, g = lane >> 4;
    float2* red = reinterpret_cast<float2*>(lds);
    uint32_t m[FM];
    float bv[FM], f0[FM], f1[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      m[i] = m0 + wm * (FM * 16) + frow<RA, FM>(i, r);
      bv[i] = o.bias && m[i] < o.M ? o.bias[m[i]] : 0.f;
      f0[i] = f1[i] = 0.f;
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const uint32_t n = n0 + wn * (FN * 16) + j * 16 + 4 * g;
      const uint32_t b = fdiv(n, o.dHW);
      const uint32_t pix = n - b * o.HW;
      const bool quad = pix + 3 < o.HW && n + 3 < o.N;
      const size_t base = size_t(b) * o.M * o.HW + pix;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        f4 z;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          z[v] = epi_act(acc[i][j][v] + bv[i], o.act);
          const float zz = m[i] < o.M && n + v < o.N ? z[v] : 0.f;
          f0[i] += zz;
          f1[i] = fmaf(zz, zz, f1[i]);
        }
        if (m[i] >= o.M || n >= o.N) continue;
        if (quad) {
          stu(o.out + base + size_t(m[i]) * o.HW, z);
        } else {
          uint32_t bb = b, pp = pix;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            if (n + v < o.N) o.out[(size_t(bb) * o.M + m[i]) * o.HW + pp] = z[v];
            if (++pp == o.HW) {
              pp = 0;
              ++bb;
            }
          }
        }
      }
    }
    // Lane (r, g) of wave (wm, wn) holds row wm*WM + frow(i, r): slot
    // (wn * 4 + g) of that row.
#pragma unroll
    for (int i = 0; i < FM; ++i)
      red[(wn * 4 + g) * MT + wm * (FM * 16) + frow<RA, FM>(i, r)] = float2{f0[i], f1[i]};
    __syncthreads();
    const int t = threadIdx.x;
    if (t < MT && m0 + t < o.M) {
      double s0 = 0, s1 = 0;
#pragma unroll
      for (int w = 0; w < WGN * 4; ++w) {
        const float2 e = red[w * MT + t];
        s0 += double(e.x);
        s1 += double(e.y);
      }
      double* d = p.stats + (size_t(m0 + t) * p.pieces + n0 / NT) * 2;
      d[0] = s0;
      d[1] = s1;
    }
  }
};
template <class E, class = void>
struct EpiStats : std::false_type {};
template <class E>
struct EpiStats<E, std::void_t<decltype(E::kStats)>> : std::true_type {};

// ---------------------------------------------------------------------------
// The kernel.
// ---------------------------------------------------------------------------
// Tile order.  The dispatcher hands consecutive workgroup ids to the eight
// XCDs in turn, and each XCD has its own L2.  With `xcd` set, the ids are
// renumbered so that each XCD receives a contiguous run of logical tiles; the
// logical order is m-tile fastest, then n-tile, then split, so the tiles that
// read the same operand rows (the same n-tile, or the same split's K range)
// run on one XCD at about the same time.
struct TileGrid {
  uint32_t gm, gn, xcd;
};
__device__ __forceinline__ void tile_coords(const TileGrid& tg, uint32_t& mt, uint32_t& nt,
                                            uint32_t& z) {
  const uint32_t id = tg.xcd ? xcd_block_id() : blockIdx.x;
  mt = id % tg.gm;
  const uint32_t t = id / tg.gm;
  nt = t % tg.gn;
  z = t / tg.gn;
}

// Occupancy floor: the 128 x 128 tile holds 64 accumulator registers per
// lane, and four workgroups per CU (the LDS limit) need the rest of the
// register file to fit in 64 more.
template <int MT, int NT>
constexpr int igemm_min_waves() {
  return MT * NT == 128 * 128 ? 4 : (MT * NT == 256 * 128 ? 2 : 1);
}

// One MT x NT tile at (m0, n0) over the K tiles [kb, ke); As and Bs are two LDS
// stages of each operand.
template <int MT, int NT, int KT, class LA, class LB, class EPI>
__device__ __forceinline__ void igemm_tile(float* As, float* Bs, const typename LA::Params& pa,
                                           const typename LB::Params& pb,
                                           const typename EPI::Params& pe, uint32_t m0, uint32_t n0,
                                           uint32_t z, uint32_t kb, uint32_t ke) {
  using SA = typename LA::St;
  using SB = typename LB::St;
  // WKS (narrow tiles, MT <= 32 with KT = 64): the four waves split every K
  // tile, each computing the whole MT x NT tile over its own 16-k slice, and
  // the four partial tiles are added in wave order at the end.  A barrier
  // then covers four times the MFMA work of the 1 x 4 wave grid at KT = 16.
  constexpr bool WKS = MT <= 32 && KT == 64;
  constexpr int WGM = WKS ? 1 : (MT >= 64 ? 2 : 1), WGN = WKS ? 1 : 4 / WGM;  // wave grid
  constexpr int WM = MT / WGM, WN = NT / WGN, FM = WM / 16, FN = WN / 16;
  static_assert(FM >= 1 && FN >= 1 && WM % 16 == 0 && WN % 16 == 0, "tile too small");
  static_assert(!WKS || 3 * FM * FN * 256 <= 2 * SB::SIZE, "wave partials fit the B stages");

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = WKS ? 0 : wave / WGN, wn = WKS ? 0 : wave % WGN;  // WKS: every wave the whole tile

  LA la;
  LB lb;
  la.init(pa, m0, tid);
  lb.init(pb, n0, tid);
  f4 ra[LA::Q], rb[LB::Q];

  f4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = zero4();

  constexpr bool DA = LA::LDSD, DB = LB::LDSD;
  constexpr bool TACC = LB::kTransAcc;
  // Row-interleaved fragments for [k][row] operands read 2 or 4 fragments at
  // a time (B only without TACC, whose quad stores need 16-row fragments).
  constexpr bool RA = SA::kRow && (FM == 2 || FM == 4);
  constexpr bool RB = SB::kRow && !TACC && (FN == 2 || FN == 4);
  const int r = lane & 15, g = lane >> 4;
  // Fragments of one 16-deep k slice of LDS stage `cur`, and its MFMAs.
  struct Frags {
    f4 a[FM], b[FN];
  };
  auto read_slice = [&](int cur, int ks, Frags& f) {
    const float* Ac = As + cur * SA::SIZE;
    const float* Bc = Bs + cur * SB::SIZE;
    if constexpr (RA) {
      SA::template frags_rif<FM>(Ac, wm * WM, r, g, ks, f.a);
    } else {
#pragma unroll
      for (int i = 0; i < FM; ++i) f.a[i] = SA::frag(Ac, wm * WM + i * 16, r, g, ks);
    }
    if constexpr (RB) {
      SB::template frags_rif<FN>(Bc, wn * WN, r, g, ks, f.b);
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j) f.b[j] = SB::frag(Bc, wn * WN + j * 16, r, g, ks);
    }
  };
  auto mfma_slice = [&](const Frags& f) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          // TACC: B first, the block accumulates C transposed (see the epilogues).
          acc[i][j] = TACC ? __builtin_amdgcn_mfma_f32_16x16x4f32(f.b[j][s], f.a[i][s], acc[i][j], 0, 0, 0)
                           : __builtin_amdgcn_mfma_f32_16x16x4f32(f.a[i][s], f.b[j][s], acc[i][j], 0, 0, 0);
  };
  if (kb < ke) {
    if constexpr (DA) la.issue_lds(kb, As); else la.load(kb, ra);
    if constexpr (DB) lb.issue_lds(kb, Bs); else lb.load(kb, rb);
    if constexpr (!DA) la.store(As, ra);
    if constexpr (!DB) lb.store(Bs, rb);
  }
  if constexpr (DA || DB) __builtin_amdgcn_s_waitcnt(0);  // the direct loads have landed
  __syncthreads();

  for (uint32_t kt = kb; kt < ke; ++kt) {
    const int cur = int(kt - kb) & 1;
    const bool more = kt + 1 < ke;
    // The first slice's fragments are read before the next tile's loads are
    // issued: a direct load into LDS that is still in flight would otherwise
    // make the compiler wait for it before any LDS read.
    Frags f0;
    read_slice(cur, WKS ? 16 * wave : 0, f0);
    // Next tile: register staging, or straight into the other LDS stage (its
    // readers finished before the previous barrier).
    if (more) {
      if constexpr (DA) la.issue_lds(kt + 1, As + (cur ^ 1) * SA::SIZE); else la.load(kt + 1, ra);
      if constexpr (DB) lb.issue_lds(kt + 1, Bs + (cur ^ 1) * SB::SIZE); else lb.load(kt + 1, rb);
    }
    mfma_slice(f0);
    if constexpr (!WKS) {
#pragma unroll
      for (int ks = 16; ks < KT; ks += 16) {
        Frags f;
        read_slice(cur, ks, f);
        mfma_slice(f);
      }
    }
    // Every MFMA of the tile is issued before the wait for the next tile's
    // loads and the barrier (the scheduler would otherwise hoist them above
    // part of the MFMAs, and a wave would stall on the loads with MFMA work
    // still unissued).
    __builtin_amdgcn_sched_barrier(0);
    if (more) {
      if constexpr (!DA) la.store(As + (cur ^ 1) * SA::SIZE, ra);
      if constexpr (!DB) lb.store(Bs + (cur ^ 1) * SB::SIZE, rb);
    }
    if constexpr (DA || DB) __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  if constexpr (WKS) {
    // Waves 1-3 park their partial tiles in the (now idle) B stages; wave 0
    // adds them in wave order and stores the tile.
    f4* red = reinterpret_cast<f4*>(Bs);
    if (wave != 0) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) red[((wave - 1) * FM * FN + i * FN + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] += red[(w * FM * FN + i * FN + j) * 64 + lane];
  }
  if constexpr (EpiStats<EPI>::value) {
    static_assert(WGN * 4 * MT * 8 <= 2 * SA::SIZE * 4, "the statistics' lane sums fit the A stages");
    EPI::template store_stats<MT, NT, FM, FN, TACC, RA, RB, WGN>(pe, acc, m0, n0, wm, wn, lane, As);
  } else {
    EPI::template store<MT, NT, FM, FN, TACC, RA, RB>(pe, acc, m0, n0, z, wm, wn, lane);
  }
}

template <int MT, int NT, int KT, class LA, class LB, class EPI>
__global__ void __launch_bounds__(kThreads)
    __attribute__((amdgpu_waves_per_eu(igemm_min_waves<MT, NT>())))
    k_igemm(const typename LA::Params pa, const typename LB::Params pb,
            const typename EPI::Params pe, TileGrid tg, uint32_t ktiles, uint32_t splits) {
  __shared__ __attribute__((aligned(16))) float As[2 * LA::St::SIZE];
  __shared__ __attribute__((aligned(16))) float Bs[2 * LB::St::SIZE];
  uint32_t mt, nt, z;
  tile_coords(tg, mt, nt, z);
  igemm_tile<MT, NT, KT, LA, LB, EPI>(As, Bs, pa, pb, pe, mt * MT, nt * NT, z,
                                      uint32_t((uint64_t(ktiles) * z) / splits),
                                      uint32_t((uint64_t(ktiles) * (z + 1)) / splits));
}

// Up to four independent products of one shape of tile in one launch (the
// sub-pixel phases of a stride-2 dX, each a quarter of the chip's work).
constexpr int kMulti = 4;
template <class LA, class LB, class EPI>
struct Multi {
  typename LA::Params pa[kMulti];
  typename LB::Params pb[kMulti];
  typename EPI::Params pe[kMulti];
  uint32_t ktiles[kMulti], gm, first[kMulti + 1];  // first workgroup of each product
};
template <int MT, int NT, int KT, class LA, class LB, class EPI>
__global__ void __launch_bounds__(kThreads)
    __attribute__((amdgpu_waves_per_eu(igemm_min_waves<MT, NT>())))
    k_igemm_multi(const Multi<LA, LB, EPI> a) {
  __shared__ __attribute__((aligned(16))) float As[2 * LA::St::SIZE];
  __shared__ __attribute__((aligned(16))) float Bs[2 * LB::St::SIZE];
  const uint32_t id = xcd_block_id();
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
  igemm_tile<MT, NT, KT, LA, LB, EPI>(As, Bs, pa, pb, pe, t % a.gm * MT, t / a.gm * NT, 0, 0, kt);
}

// Filters in the K order of the pixel loaders (flat or blocked), zero for
// padding channels; `inner` is the padded channel count the K axis runs over
// (Cp for the forward, OCp for dX):
// mode 0 (forward A): out[oc][kk] = w[oc][c][khw]   with c  = channel of kk
// mode 1 (dX A):      out[c][kk]  = w[oc][c][khw]   with oc = channel of kk
// where kk = khw*inner + ch (flat) or (cb*KK + khw)*kCB + ci, ch = cb*kCB + ci
// (blocked).  Rows are ld >= KK*inner floats apart, zero past KK*inner; size
// rows * ld, rows = OC (mode 0) or C (mode 1).  The packed forward (C < 4
// channels) uses the flat order with inner = C and ld = pad4(KK*C).
// With vw != 0 the K order runs over the taps of one sub-pixel phase of a
// strided dX: virtual tap v = jh * vw + jw is the filter tap (rh + s*jh,
// rw + s*jw) of a kk x kk filter, and KK counts the phase's taps.
struct WPerm {
  const float* w;  // null: nothing to re-lay
  float* out;
  uint32_t OC, C, KK, inner, ld;
  int mode, blocked;
  uint32_t vw, kk, s, rh, rw;
  // Blocked order with inner % 16 == 0: out as bf16 parts, 96 bytes per
  // block of 16 k (split_pair).
  uint32_t parts;
  uint32_t blocks() const { return w ? cdiv(size_t(mode == 0 ? OC : C) * ld, 256) : 0; }
};

struct BwdSide {
  const float* dbPart;  // bias-gradient partials [OC][dbRows]
  float* db;
  uint32_t dbRows, nRow;  // nRow = OC, or 0 for no bias gradient
};

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
// Operands are read through buffer resources addressed by 32-bit float
// offsets below kOob.
static bool operand_fits(size_t floats, const char* what) {
  if (floats < kOob) return true;
  set_error("%s: operand of %zu floats exceeds the implicit-GEMM limit of %u floats (2 GiB)", what,
            floats, kOob);
  return false;
}

struct TileCfg {
  int MT, NT, KT;
  uint32_t splits;
};

// Tuning overrides: DCE_TUNE_<FWD|DW|DX|GEMM>="MT,NT,KT,splits" replaces the
// heuristic choice for that GEMM family (read on every call).
static bool tune_override(const char* var, TileCfg& c) {
  const char* e = getenv(var);
  if (!e || !*e) return false;
  int a, b, k;
  unsigned sp;
  if (sscanf(e, "%d,%d,%d,%u", &a, &b, &k, &sp) != 4) return false;
  c = TileCfg{a, b, k, sp ? sp : 1u};
  return true;
}

// XCD-contiguous tile order (on unless DCE_XCD=0; read on every call).
static bool xcd_order() {
  const char* e = getenv("DCE_XCD");
  return !(e && *e && atoi(e) == 0);
}

// 128 unless 64 wastes clearly less padding (8 % or more of the extent: the
// 576 taps x channels of a 3x3 conv over 64 channels run 11 % padding MFMA
// work on 128-wide dW tiles, and 64-wide ones measured 7 % faster on the
// 128 x 64 x 56 x 56 conv's dW, 3 % on UNet's 64-channel layers).
static int pick_tile(uint32_t extent) {
  const uint64_t w128 = uint64_t(cdiv(extent, 128)) * 128, w64 = uint64_t(cdiv(extent, 64)) * 64;
  return (w128 * 100 > w64 * 108) ? 64 : 128;
}

// Rows of the output tile (the channel axis): the narrow 16- and 32-row tiles
// for up to 16 / 32 channels, where a 64-row tile would feed the matrix unit
// mostly zero rows.
static int pick_tile_m(uint32_t M) {
  if (M <= 16) return 16;
  if (M <= 32) return 32;
  return pick_tile(M);
}

// Workgroups of one kernel instantiation that fit on a CU at once.
template <class Kern>
static int occupancy(Kern kernel) {
  static std::map<const void*, int> cache;
  const void* key = reinterpret_cast<const void*>(kernel);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kThreads, 0) != hipSuccess || n < 1)
    n = 1;
  cache[key] = n;
  return n;
}

// Estimated microseconds of one launch plus its split-K finish, used to pick
// the split count.  The W = tiles * splits workgroups are spread evenly over
// the CUs; the busiest CU gets n = ceil(W / CUs) of them and runs them in
// batches of at most `occ` (the kernel's workgroups per CU).  In a batch of r
// workgroups one K tile takes max(kLatencyUs, r * tm), where tm is the K
// tile's MFMA time for a lone workgroup (MT*NT*KT*2 flops at the CU's
// 614 GFLOP/s fp32 matrix peak) and kLatencyUs the latency-bound floor, so a
// short last batch costs less than a full one.  Split partials cost
// 2 * splits * M * N * 4 bytes at kFinishBytesPerUs.  The constants were
// fitted to a sweep of every split count of the AlexNet convolutions on
// MI355X: the choices are within 1 % of the best measured configurations.
constexpr double kCuFlopsPerUs = 614.4e3;
constexpr double kLatencyUs = 2.0;
constexpr double kFinishBytesPerUs = 3.0e6;
static double est_us(uint32_t M, uint32_t N, uint32_t kdim, const TileCfg& c, int occ,
                     bool partials) {
  const uint32_t cus = uint32_t(num_cus());
  const uint32_t tiles = cdiv(M, uint32_t(c.MT)) * cdiv(N, uint32_t(c.NT));
  const uint32_t n = cdiv(tiles * c.splits, cus);
  const uint32_t full = n / uint32_t(occ), rem = n - full * uint32_t(occ);
  const double kps = double(cdiv(kdim, uint32_t(c.KT))) / c.splits;
  const double tm = double(c.MT) * c.NT * c.KT * 2.0 / kCuFlopsPerUs;
  double T = kps * full * std::max(kLatencyUs, occ * tm);
  if (rem > 0) T += kps * std::max(kLatencyUs, rem * tm);
  if (partials) T += 2.0 * c.splits * double(M) * N * 4.0 / kFinishBytesPerUs;
  return T;
}

// Tile / split choice for an M x N output with kdim-long dot products.  The
// tile is 128 or 64 per axis (pick_tile); the split count minimises est_us
// over 1..max_splits with at least 8 K tiles per split.  `occ(cfg)` gives the
// occupancy of the kernel that cfg launches; `dense_out` says the unsplit
// launch writes the final output (no partial buffer).
template <class OccFn>
static TileCfg choose(const char* var, uint32_t M, uint32_t N, uint32_t kdim, uint32_t max_splits,
                      bool dense_out, OccFn&& occ, bool kt16_only = false,
                      bool narrow_ksplit = false, bool narrow32 = false) {
  TileCfg c{pick_tile_m(M), pick_tile(N), 16, 1};
  if (kt16_only && c.MT < 64) c.NT = 128;  // the pixel GEMMs' narrow tiles are 128 or 256 wide
  if (narrow_ksplit && c.MT < 64) {
    // Narrow tiles with the waves splitting K: 64 columns (a wave then holds
    // the whole tile's accumulators; 128 would cost registers and occupancy),
    // or 32 (narrow32) when 64 pads the columns by 8 % more: the 144 and 288
    // taps x channels of 3x3 convs over 16 and 32 channels.
    const uint64_t w64 = uint64_t(cdiv(N, 64)) * 64, w32 = uint64_t(cdiv(N, 32)) * 32;
    c.NT = (narrow32 && w64 * 100 > w32 * 108) ? 32 : 64;
    c.KT = 64;
  }
  const uint32_t ktiles = cdiv(kdim, uint32_t(c.KT));
  if (tune_override(var, c)) {
    if (kt16_only) c.KT = 16;
    c.splits = std::max<uint32_t>(1, std::min<uint32_t>(c.splits, cdiv(kdim, uint32_t(c.KT))));
    return c;
  }
  const uint32_t smax = std::max<uint32_t>(1, std::min(max_splits, ktiles / 8));
  double best = 0;
  uint32_t bestS = 1;
  for (uint32_t sp = 1; sp <= smax; ++sp) {
    TileCfg t = c;
    t.splits = sp;
    const double e = est_us(M, N, kdim, t, occ(t), sp > 1 || !dense_out);
    if (sp == 1 || e < best) {
      best = e;
      bestS = sp;
    }
  }
  c.splits = bestS;
  // A 128 x 256 tile (two workgroups per CU) beats 128 x 128 (four) on the
  // pixel-row GEMMs whose rows fill whole 128-row tiles, that need split K to
  // fill the chip and whose 128 x 256 grid still gives every CU about two
  // workgroups: AlexNet b128 c4 / c5 forward and c5 dX (510 workgroups) 3-5 %
  // faster at the same split count.  Unsplit ones (c3 forward, the 56x56
  // single conv) run as fast or slower on it, and small grids (UNet's 32x32
  // and 16x16 levels: 64-384 workgroups) lose up to half their speed.
  if (kt16_only && c.MT == 128 && c.NT == 128 && M % 128 == 0 && c.splits >= 2 &&
      uint64_t(cdiv(M, 128)) * cdiv(N, 256) * c.splits * 8 >= uint64_t(num_cus()) * 15)
    c.NT = 256;
  if (const char* e = getenv("DCE_TUNE_LOG")) {
    if (*e && *e != '0')
      fprintf(stderr, "[dcengine] %s M=%u N=%u K=%u -> %dx%dx%d splits %u (occupancy %d)\n", var, M,
              N, kdim, c.MT, c.NT, c.KT, c.splits, occ(c));
  }
  return c;
}

// Pixel-row GEMMs (forward, dX) of convolutions with few channels on small
// images: at most 128 output rows, dot products of at most 1152 (128
// channels x 3 x 3) and at most 131072 pixels (UNet-base16 b8 below the
// 256^2 level).  The cost model prices their K tiles at its 2 us latency
// floor and splits them 4-7 ways or runs them on 128-row tiles (M = 96);
// measured, unsplit 32-row tiles over more workgroups are 10-20 % faster
// (UNet levels 1-3: 36-41 -> 31-36 us per layer, M = 96 dX 92 -> 73 us).
// An override through DCE_TUNE_* keeps its tile.
static void narrow_short_k(TileCfg& c, const char* var, uint32_t M, uint32_t N, uint32_t kdim) {
  if (const char* e = getenv(var))
    if (*e) return;
  if (M > 128 || kdim > 1152 || N > 131072) return;
  c = TileCfg{M <= 16 ? 16 : 32, 128, 16, 1};
}

template <int MT, int NT, int KT, class LA, class LB, class EPI>
static bool launch(const typename LA::Params& pa, const typename LB::Params& pb,
                   const typename EPI::Params& pe, uint32_t M, uint32_t N, uint32_t ktiles,
                   uint32_t splits, const char* what) {
  const TileGrid tg{cdiv(M, MT), cdiv(N, NT), xcd_order() ? 1u : 0u};
  const uint32_t nwg = tg.gm * tg.gn * splits;
  hipLaunchKernelGGL((k_igemm<MT, NT, KT, LA, LB, EPI>), dim3(nwg), dim3(kThreads), 0, stream(),
                     pa, pb, pe, tg, ktiles, splits);
  return check_launch(what);
}

// Dispatch a functor over the (MT, NT) tile shapes: 64/128 square-ish tiles at
// two KT depths and the narrow MT = 16/32 tiles at KT = 16 (1 x 4 wave grid)
// or KT = 64 (waves split the K tile).  NARROW32: also 32 columns at KT = 64
// (the conv dW of few output channels over 16 or 32 input channels).
template <bool NARROW32 = false, class F>
static bool tiles_dispatch(const TileCfg& c, F&& f) {
#define DCE_T(a, b, k) \
  if (c.MT == a && c.NT == b && c.KT == k) return f.template run<a, b, k>();
  DCE_T(128, 128, 32) DCE_T(128, 64, 32) DCE_T(64, 128, 32) DCE_T(64, 64, 32)
  DCE_T(256, 128, 16) DCE_T(128, 256, 16)
  DCE_T(128, 128, 16) DCE_T(128, 64, 16) DCE_T(64, 128, 16) DCE_T(64, 64, 16)
  DCE_T(32, 128, 16) DCE_T(32, 64, 16) DCE_T(16, 128, 16) DCE_T(16, 64, 16)
  DCE_T(32, 128, 64) DCE_T(32, 64, 64) DCE_T(16, 128, 64) DCE_T(16, 64, 64)
  if constexpr (NARROW32) {
    DCE_T(32, 32, 64) DCE_T(16, 32, 64)
  }
#undef DCE_T
  set_error("igemm: unsupported tile %dx%dx%d", c.MT, c.NT, c.KT);
  return false;
}

// The KT = 16 shapes of the pixel-row GEMMs (forward, dX): the narrow tiles
// come with 128 or 256 pixel columns.
template <class F>
static bool tiles_dispatch16(const TileCfg& c, F&& f) {
#define DCE_T(a, b) \
  if (c.MT == a && c.NT == b && c.KT == 16) return f.template run<a, b, 16>();
  DCE_T(256, 128) DCE_T(128, 256)
  DCE_T(128, 128) DCE_T(128, 64) DCE_T(64, 128) DCE_T(64, 64)
  DCE_T(32, 256) DCE_T(32, 128) DCE_T(16, 256) DCE_T(16, 128)
#undef DCE_T
  set_error("igemm: unsupported tile %dx%dx%d", c.MT, c.NT, c.KT);
  return false;
}
template <class F>
static int tiles_occ16(const TileCfg& c, const F& f) {
#define DCE_T(a, b) \
  if (c.MT == a && c.NT == b && c.KT == 16) return f.template occ<a, b, 16>(c.splits > 1);
  DCE_T(256, 128) DCE_T(128, 256)
  DCE_T(128, 128) DCE_T(128, 64) DCE_T(64, 128) DCE_T(64, 64)
  DCE_T(32, 256) DCE_T(32, 128) DCE_T(16, 256) DCE_T(16, 128)
#undef DCE_T
  return 1;
}

// Occupancy of the kernel a functor would launch for cfg.
template <bool NARROW32 = false, class F>
static int tiles_occ(const TileCfg& c, const F& f) {
#define DCE_T(a, b, k) \
  if (c.MT == a && c.NT == b && c.KT == k) return f.template occ<a, b, k>(c.splits > 1);
  DCE_T(128, 128, 32) DCE_T(128, 64, 32) DCE_T(64, 128, 32) DCE_T(64, 64, 32)
  DCE_T(256, 128, 16) DCE_T(128, 256, 16)
  DCE_T(128, 128, 16) DCE_T(128, 64, 16) DCE_T(64, 128, 16) DCE_T(64, 64, 16)
  DCE_T(32, 128, 16) DCE_T(32, 64, 16) DCE_T(16, 128, 16) DCE_T(16, 64, 16)
  DCE_T(32, 128, 64) DCE_T(32, 64, 64) DCE_T(16, 128, 64) DCE_T(16, 64, 64)
  if constexpr (NARROW32) {
    DCE_T(32, 32, 64) DCE_T(16, 32, 64)
  }
#undef DCE_T
  return 1;
}

static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
static inline size_t al64(size_t n) { return (n + 63) & ~size_t(63); }

// ---------------------------------------------------------------------------
// Shared by the GEMM families (dce_igemm*.hip).
// ---------------------------------------------------------------------------
inline uint32_t pad16(uint32_t c) { return (c + 15u) & ~15u; }
// Floats of a [rows][pad16(c)] array of bf16 parts (96 bytes per 16 values).
inline size_t parts_floats(size_t rows, uint32_t c) { return rows * (pad16(c) / 16) * 24; }
// The bf16 parts (dce_igemm_parts.h) of two values, the first in the low half of
// each word.  Every part is what the ones before it leave, rounded to nearest
// even.  A value that rounds to infinity, an infinity or a NaN gets a NaN or
// infinite part.
using bf2 = __bf16 __attribute__((ext_vector_type(2)));
struct Parts2 {
  uint32_t h, m, l;
};
__device__ __forceinline__ uint32_t bf16_pair(float x, float y) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x, y}, bf2));
}
__device__ __forceinline__ Parts2 split_pair(float x, float y) {
  const uint32_t h = bf16_pair(x, y);
  const float rx = x - __uint_as_float(h << 16), ry = y - __uint_as_float(h & 0xffff0000u);
  const uint32_t m = bf16_pair(rx, ry);
  return Parts2{h, m, bf16_pair(rx - __uint_as_float(m << 16), ry - __uint_as_float(m & 0xffff0000u))};
}
// Below 2^-110 the last bits of a float leave the bf16 range, from 0x7f7f8000 on
// it rounds to infinity: x has no three bf16 parts then.  It is kept as a NaN,
// then its own upper and lower half (parts_value puts it together again).
// `key` is the magnitude's bits, shifted so that zero, which has parts, is the
// largest.
__device__ __forceinline__ uint32_t parts_key(float x) { return (__float_as_uint(x) << 1) - 1u; }
constexpr uint32_t kTinyKey = 2 * 0x08800000u - 1, kHugeKey = 2 * 0x7f7f8000u - 1;
__device__ __forceinline__ bool parts_raw(float x) {
  const uint32_t k = parts_key(x);
  return k < kTinyKey || (k >= kHugeKey && k != 0xffffffffu);
}
// Parts of 8 values as one 16-byte quad per part.  FINITE: nothing is raw (a
// value at the upper end that is gets a NaN part).
template <bool FINITE>
__device__ __forceinline__ void split_parts8(const float (&x)[8], uint4 (&out)[3]) {
  uint32_t q[3][4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const Parts2 p = split_pair(x[2 * e], x[2 * e + 1]);
    q[0][e] = p.h;
    q[1][e] = p.m;
    q[2][e] = p.l;
  }
  if constexpr (!FINITE) {
    uint32_t least = 0xffffffffu, most = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t k = parts_key(x[e]);
      least = min(least, k);
      most = max(most, k + 1u);
    }
    if (least < kTinyKey || most > kHugeKey) {  // hardly ever
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (!parts_raw(x[e])) continue;
        const uint32_t u = __float_as_uint(x[e]), at = 16 * (e & 1), keep = 0xffff0000u >> at;
        q[0][e / 2] = (q[0][e / 2] & keep) | (0x7fffu << at);
        q[1][e / 2] = (q[1][e / 2] & keep) | ((u >> 16) << at);
        q[2][e / 2] = (q[2][e / 2] & keep) | ((u & 0xffffu) << at);
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) out[p] = uint4{q[p][0], q[p][1], q[p][2], q[p][3]};
}
// A value from its parts (each in the upper half of a word).
__device__ __forceinline__ float parts_value(uint32_t h, uint32_t m, uint32_t l) {
  const float x = __uint_as_float(h);
  return x == x ? (x + __uint_as_float(m)) + __uint_as_float(l) : __uint_as_float(m | l >> 16);
}

bool permute_w(const WPerm& pw);
// Four filter re-layouts in one launch (null w: none).
struct WPerm4 {
  WPerm p[4];
};
bool permute_w4(const WPerm4& pw);
// Zero-padded copy of a row-major [rows][cols] matrix to row stride ldp.
bool pad_cols(const float* in, float* out, uint32_t rows, uint32_t cols, uint32_t ldp);
// Split-K finishes: NCHW output (bias, activation), row-major output.
bool split_nchw(const float* part, const float* bias, float* out, uint32_t M, uint32_t N,
                uint32_t HW, uint32_t splits, uint32_t act);
bool split_sum(const float* part, float* c, uint32_t n, uint32_t splits);

struct PsGeom {
  uint32_t Hp, OWp, OHWp, Ncol, RS;
  size_t floats;
};
PsGeom ps_geom(const ConvGeom& g);
PsParams ps_params(const float* src, const ConvGeom& g);
PkParams pk_params(const float* src, const ConvGeom& g);

// The conv backward's GEMMs: dW split partials and dX.  With `parts` G, x and
// the filters come as bf16 parts (dce_igemm_parts.h), otherwise as fp32.
TileCfg conv_dw_choose(uint32_t M, uint32_t N, uint32_t kdim, bool trans, bool pk, bool ps,
                       bool parts);
bool conv_dw_gemm(const TileCfg& c, const float* gn, const float* xn, float* part,
                  const ConvGeom& g, bool trans, bool pk, bool ps, bool parts);
struct DxPlan {
  bool phased;   // as sub-pixel phases, which re-lay the filters themselves (w -> wt)
  TileCfg cfg;   // of the one launch (stride 3 or more: chosen per phase)
  size_t part;   // floats of split partials
};
DxPlan conv_dx_plan(const ConvGeom& g, bool parts);
bool conv_dx(const DxPlan& p, const float* w, float* wt, const float* gn, float* dx, float* part,
             const ConvGeom& g, bool parts);

// K order: blocked when the padded channel count is a multiple of kCB (no
// extra padding then), flat otherwise.
static inline bool blocked_k(uint32_t Cp) { return Cp % kCB == 0; }

// Run F<S1, BLK> for the runtime (stride == 1, blocked) pair.
template <template <bool, bool> class F, class... A>
static bool conv_variant(bool s1, bool blk, const TileCfg& c, A&&... a) {
  if (s1 && blk) return tiles_dispatch16(c, F<true, true>{a...});
  if (s1) return tiles_dispatch16(c, F<true, false>{a...});
  if (blk) return tiles_dispatch16(c, F<false, true>{a...});
  return tiles_dispatch16(c, F<false, false>{a...});
}
template <template <bool, bool> class F>
static int conv_variant_occ(bool s1, bool blk, const TileCfg& c) {
  if (s1 && blk) return tiles_occ16(c, F<true, true>{});
  if (s1) return tiles_occ16(c, F<true, false>{});
  if (blk) return tiles_occ16(c, F<false, true>{});
  return tiles_occ16(c, F<false, false>{});
}

}  // namespace dce
