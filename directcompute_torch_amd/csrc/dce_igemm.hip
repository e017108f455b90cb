// Convolutions on the implicit GEMM of dce_igemm.h: layout passes, split-K
// finishes, the forward, the pointwise backward and the backward's host side
// (its dW and dX GEMMs are in dce_igemm_dw.hip and dce_igemm_dx.hip, the
// dense products in dce_igemm_dense.hip).
#include "dce_igemm.h"

namespace dce {

// ---------------------------------------------------------------------------
// Side kernels: NHWC transpose (+ ReLU mask + bias-gradient partials),
// filter re-layouts, split-K sums.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void permute_w_elem(const WPerm& pw, uint32_t i) {
  const float* __restrict__ w = pw.w;
  float* __restrict__ out = pw.out;
  const uint32_t OC = pw.OC, C = pw.C, KK = pw.KK, inner = pw.inner, ld = pw.ld;
  const int mode = pw.mode, blocked = pw.blocked;
  const uint32_t kdim = KK * inner;
  const uint32_t rows = mode == 0 ? OC : C;
  if (i >= rows * ld) return;
  const uint32_t r = i / ld, kk = i - r * ld;
  if (kk >= kdim) {  // row pitch padding
    out[i] = 0.f;
    return;
  }
  uint32_t khw, ch;
  if (blocked) {
    const uint32_t blk = kk / kCB, ci = kk - blk * kCB;
    const uint32_t cb = blk / KK;
    khw = blk - cb * KK;
    ch = cb * kCB + ci;
  } else {
    khw = kk / inner;
    ch = kk - khw * inner;
  }
  uint32_t wk = khw, wKK = KK;
  if (pw.vw) {
    const uint32_t jh = khw / pw.vw, jw = khw - jh * pw.vw;
    wk = (pw.rh + pw.s * jh) * pw.kk + pw.rw + pw.s * jw;
    wKK = pw.kk * pw.kk;
  }
  float v;
  if (mode == 0)
    v = ch < C ? w[(r * C + ch) * wKK + wk] : 0.f;
  else
    v = ch < OC ? w[(ch * C + r) * wKK + wk] : 0.f;
  if (!pw.parts) {
    out[i] = v;
    return;
  }
  const Parts2 q = split_pair(v, 0.f);
  const uint32_t u = __float_as_uint(v);
  const bool raw = parts_raw(v);
  uint16_t* o = reinterpret_cast<uint16_t*>(out) + (size_t(r) * (ld / 16) + kk / 16) * 48 + kk % 16;
  o[0] = uint16_t(raw ? 0x7fffu : q.h);
  o[16] = uint16_t(raw ? u >> 16 : q.m);
  o[32] = uint16_t(raw ? u : q.l);
}

__global__ void k_permute_w(WPerm pw) { permute_w_elem(pw, blockIdx.x * blockDim.x + threadIdx.x); }

bool permute_w(const WPerm& pw) {
  hipLaunchKernelGGL(k_permute_w, dim3(pw.blocks()), dim3(256), 0, stream(), pw);
  return check_launch("permute_w");
}

__global__ void k_permute_w4(WPerm4 q) {
  uint32_t b = blockIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const WPerm& pw = q.p[i];
    const uint32_t rows = pw.mode == 0 ? pw.OC : pw.C;
    const uint32_t nb = pw.w ? (rows * pw.ld + 255) / 256 : 0;
    if (b < nb) {
      permute_w_elem(pw, b * 256 + threadIdx.x);
      return;
    }
    b -= nb;
  }
}
bool permute_w4(const WPerm4& q) {
  uint32_t n = 0;
  for (const WPerm& p : q.p) n += p.blocks();
  hipLaunchKernelGGL(k_permute_w4, dim3(n), dim3(256), 0, stream(), q);
  return check_launch("permute_w");
}

// out[((b*HW) + p)*Cp + c] = (c < C) ? in[(b*C + c)*HW + p] masked : 0.
// Block: CB channels x PB = 2048 / CB pixels through LDS (CB = 16 for tensors
// of at most 16 channels, 32 otherwise, so few-channel tensors do not leave
// half the block idle).  dbPart[c][b*npb + block]: the masked values of
// channel c summed over the block's pixels.
// Loads are 16-byte quads of 4 pixels of one channel row and stores 16-byte
// quads of 4 channels of one pixel (Cp % 4 == 0 keeps those aligned).  Plane
// rows of odd length leave the load quads only 4-byte aligned; the GPU runs
// with unaligned access enabled.  A quad that would cross the end of its row
// is read dword by dword.
// Workgroups past the first nMain re-lay filters instead (pw: the forward's
// filter permutation, which then costs no launch of its own).
// BNDX: `in` is the dy of a batch norm and `y` its input x; the values
// transposed are that batch norm's dx (bn_dx_elem), which the kernel also
// stores in NCHW to bn.dx: batchnorm_backward_dx and the transpose pass of
// the conv below it in one pass.
struct BnDxArgs {
  const float* mean;
  const float* var;
  const float* gamma;
  const float* dg;
  const float* db;
  float* dx;
  float eps, m;
};
// A thread's parts of 8 channels, in the order of memory (quad i of group g =
// threadIdx.x: block g / 2, part i, half g % 2), so that consecutive threads then
// store consecutive quads (32-byte runs, which a thread's own quads would make,
// took longer).
__device__ __forceinline__ void stage_parts8(const float (&x)[8], uint4* qs) {
  uint4 w[3];
  split_parts8<false>(x, w);
  const int gr = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 3; ++i) qs[gr / 2 * 6 + 2 * i + (gr & 1)] = w[i];
  __syncthreads();
}

// The forward's channel-innermost copy of x as bf16 parts, 256 groups of 8
// channels a workgroup.
struct XSplit {
  const float* src;  // null: no job
  float* dst;
  uint32_t groups, nblk, Cp;
  FastDiv dGroups;  // of a pixel: 2 * nblk
  uint32_t blocks() const { return src ? cdiv(groups, 256) : 0; }
};
__device__ __forceinline__ void xsplit_block(const XSplit& q, uint32_t blk, uint4* qs) {
  const uint32_t g = blk * 256 + threadIdx.x, pix = fdiv(g, q.dGroups);
  const uint32_t c = 8 * (g - pix * q.dGroups.d);
  const float* src = q.src + size_t(pix) * q.Cp + c;
  f4 v[2] = {zero4(), zero4()};
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (g < q.groups && c + 4 * i < q.Cp) v[i] = *reinterpret_cast<const f4*>(src + 4 * i);
  const float x[8] = {v[0][0], v[0][1], v[0][2], v[0][3], v[1][0], v[1][1], v[1][2], v[1][3]};
  stage_parts8(x, qs);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const uint32_t s = threadIdx.x + 256 * j;
    if (blk * 768 + s < 3 * q.groups)
      reinterpret_cast<uint4*>(q.dst)[size_t(blk) * 768 + s] = qs[s];
  }
}
__global__ void __launch_bounds__(256) k_xsplit(const XSplit q) {
  __shared__ uint4 qs[768];
  xsplit_block(q, blockIdx.x, qs);
}
static bool xsplit(const XSplit& q) {
  ProfScope prof("x_parts", 0, 4.0 * double(q.groups) * 8 * 2.5);
  hipLaunchKernelGGL(k_xsplit, dim3(q.blocks()), dim3(256), 0, stream(), q);
  return check_launch("xsplit");
}

// PARTS (CB = 32): out as bf16 parts, [pixel][nblk][h, m, l of 16 channels]; the
// workgroups past the filters' split a kept copy of x (xs).
template <int CB, bool BNDX, bool PARTS>
__global__ void __launch_bounds__(256)
    k_to_nhwc(const float* __restrict__ in, const float* __restrict__ y, float* __restrict__ out,
              float* __restrict__ dbPart, uint32_t C, uint32_t HW, uint32_t Cp, uint32_t npb,
              uint32_t ncb, uint32_t nB, uint32_t nMain, WPerm pw, uint32_t nblk, uint32_t nPerm,
              XSplit xs, BnDxArgs bn) {
  static_assert(!PARTS || CB == 32, "parts: one group of 8 channels per thread");
  __shared__ uint4 qs[PARTS ? 768 : 1];
  if (blockIdx.x >= nMain) {
    const uint32_t e = blockIdx.x - nMain;
    if (!PARTS || e < nPerm)
      permute_w_elem(pw, e * 256 + threadIdx.x);
    else
      xsplit_block(xs, e - nPerm, qs);
    return;
  }
  constexpr int PB = 2048 / CB, PQ = PB / 4;  // pixels per block, pixel quads per row
  constexpr int CR = 256 / PQ;                // channel rows per load pass
  constexpr int PR = 256 / (CB / 4);          // pixels per store pass
  static_assert(CR * 2 == CB && PR * 2 == PB, "two load and two store passes");
  __shared__ float t[CB][PB + 1];
  // 1-D grid over (pixel block, channel block, image), pixel block fastest,
  // in XCD-contiguous order: a plane row's neighbouring blocks share its
  // partial cache lines.
  const uint32_t id = xcd_block_id(nMain);
  const uint32_t pb = id % npb, rest = id / npb;
  const uint32_t c0 = (rest % ncb) * CB, p0 = pb * PB, b = rest / ncb;
  const int tid = threadIdx.x;
  // Branch-free loads through buffer resources (elements outside the tile's
  // channels / pixels read at kOob, i.e. zero): all of a thread's loads are
  // in flight together.  Callers admit tensors below kOob floats.
  BRes bi, by;
  const uint32_t n = nB * C * HW;
  bi.init(in, n);
  by.init(y ? y : in, n);
  const int pq = tid % PQ;  // pixel quad of the load phase
  f4 v[2], m[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t c = c0 + tid / PQ + CR * j, p = p0 + 4 * pq;
    const uint32_t row = (b * C + c) * HW;
    if (c < C && p + 3 < HW) {
      v[j] = bi.ld4(row + p);
      m[j] = y ? by.ld4(row + p) : f4{1.f, 1.f, 1.f, 1.f};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t off = (c < C && p + e < HW) ? row + p + e : kOob;
        v[j][e] = bi.ld1(off);
        m[j][e] = y ? by.ld1(off) : 1.f;
      }
    }
  }
  if constexpr (BNDX) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t c = c0 + tid / PQ + CR * j, p = p0 + 4 * pq;
      if (c >= C) {
        v[j] = zero4();
        continue;
      }
      const float mu = bn.mean[c], rstd = 1.0f / sqrtf(bn.var[c] + bn.eps);
      const float g = bn.gamma[c], dg = bn.dg[c], db = bn.db[c];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[j][e] = p + e < HW ? bn_dx_elem(m[j][e], v[j][e], mu, rstd, g, dg, db, bn.m) : 0.f;
      float* dst = bn.dx + (size_t(b) * C + c) * HW + p;
      if (p + 3 < HW) {
        stu(dst, v[j]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (p + e < HW) dst[e] = v[j][e];
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) t[tid / PQ + CR * j][4 * pq + e] = v[j][e];
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        // ReLU mask: y <= 0 zeroes the gradient (a NaN y keeps it).
        t[tid / PQ + CR * j][4 * pq + e] = m[j][e] <= 0.f ? 0.f : v[j][e];
  }
  __syncthreads();
  if (dbPart != nullptr && tid < 8 * CB) {
    // 8 lanes per channel, PB / 8 pixels each, then a fixed butterfly.
    const int cl = tid >> 3, part = tid & 7;
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < PB / 8; ++q) s += t[cl][part * (PB / 8) + q];
    s = group8_reduce(s);
    if (part == 0 && c0 + cl < C)
      dbPart[size_t(c0 + cl) * nB * npb + size_t(b) * npb + pb] = s;
  }
  if constexpr (PARTS) {
    constexpr int GP = CB / 8, QB = CB / 16 * 6;  // groups and quads of a pixel
    {
      const int pl = tid / GP, gr = tid % GP;
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = t[8 * gr + e][pl];
      stage_parts8(x, qs);
    }
    const uint32_t qn = min(uint32_t(QB), 6 * (nblk - c0 / 16));  // quads inside the channels
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const uint32_t s = tid + 256 * j, pl = s / QB, q = s - pl * QB, p = p0 + pl;
      if (p < HW && q < qn)
        *reinterpret_cast<uint4*>(reinterpret_cast<char*>(out) +
                                  ((size_t(b) * HW + p) * nblk + c0 / 16) * 96 + q * 16) = qs[s];
    }
    return;
  }
  const int cq = tid % (CB / 4);  // channel quad of the store phase
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int pl = tid / (CB / 4) + PR * j;
    const uint32_t c = c0 + 4 * cq, p = p0 + pl;
    const f4 q = {t[4 * cq][pl], t[4 * cq + 1][pl], t[4 * cq + 2][pl], t[4 * cq + 3][pl]};
    if (p < HW && c < Cp) *reinterpret_cast<f4*>(out + (size_t(b) * HW + p) * Cp + c) = q;
  }
}

// Few channels (Cp <= 8): one thread per pixel reads its C channel values
// (coalesced across threads per channel) and stores Cp/4 quads.
__global__ void k_to_nhwc_small(const float* __restrict__ in, float* __restrict__ out, uint32_t C,
                                uint32_t HW, uint32_t Cp, uint32_t npix, FastDiv dHW) {
  const uint32_t n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= npix) return;
  const uint32_t b = fdiv(n, dHW), p = n - b * HW;
  const float* src = in + size_t(b) * C * HW + p;
  f4* dst = reinterpret_cast<f4*>(out + size_t(n) * Cp);
  for (uint32_t q = 0; q < Cp / 4; ++q) {
    f4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (4 * q + e < C) ? src[size_t(4 * q + e) * HW] : 0.f;
    dst[q] = v;
  }
}

// out[c] = sum of the `rows` partials of channel c (stored contiguously,
// part[c*rows + r]): 256 strided per-thread sums, then a fixed tree.  One
// 256-thread block per channel.
__device__ __forceinline__ void rowsum_block(const float* __restrict__ part,
                                             float* __restrict__ out, uint32_t rows,
                                             uint32_t c) {
  __shared__ float sh[4];
  const float* p = part + size_t(c) * rows;
  float s = 0.f;
#pragma unroll 8
  for (uint32_t r = threadIdx.x; r < rows; r += 256) s += p[r];
  s = wave_reduce(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[c] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ void __launch_bounds__(256)
    k_rowsum(const float* __restrict__ part, float* __restrict__ out, uint32_t rows) {
  rowsum_block(part, out, rows, blockIdx.x);
}


// Deterministic split-K sum: out[i] = sum_z part[z*n + i] in z order.
__global__ void k_splitk_sum(const float* __restrict__ part, float* __restrict__ out, uint32_t n,
                             uint32_t splits) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (uint32_t z = 0; z < splits; ++z) s += part[size_t(z) * n + i];
  out[i] = s;
}

// Quad form of k_splitk_sum for n % 4 == 0 (same summation order).
// Sum of the split partials p[0], p[zs], p[2 zs], ... in split order; the
// loads of each group of up to four are issued before its adds (the finishes
// run at 2 - 3 splits, which a one-at-a-time loop would serialise).
__device__ __forceinline__ f4 sum_splits4(const f4* __restrict__ p, size_t zs, uint32_t splits) {
  f4 s = {0.f, 0.f, 0.f, 0.f};
  uint32_t z = 0;
  for (; z + 3 < splits; z += 4) {
    const f4 a = p[z * zs], b = p[(z + 1) * zs], c = p[(z + 2) * zs], d = p[(z + 3) * zs];
    s += a;
    s += b;
    s += c;
    s += d;
  }
  const uint32_t rem = splits - z;  // uniform across the grid
  if (rem == 3) {
    const f4 a = p[z * zs], b = p[(z + 1) * zs], c = p[(z + 2) * zs];
    s += a;
    s += b;
    s += c;
  } else if (rem == 2) {
    const f4 a = p[z * zs], b = p[(z + 1) * zs];
    s += a;
    s += b;
  } else if (rem == 1) {
    s += p[z * zs];
  }
  return s;
}
__global__ void __launch_bounds__(256)
    k_splitk_sum4(const f4* __restrict__ part, f4* __restrict__ out, uint32_t nq,
                  uint32_t splits) {
  const uint32_t q = blockIdx.x * 256 + threadIdx.x;
  if (q >= nq) return;
  out[q] = sum_splits4(part + q, nq, splits);
}

// dW finalize: dw[oc][c][khw] = sum_z part[z][oc][khw*Cp + c], or with
// `trans` (the GEMM ran with taps as rows) sum_z part[z][khw*Cp + c][oc].
// Quad form: thread (quad q, slice w) sums the 16-byte quads part[z][4q..]
// over z = w, w + SL, w + 2 SL, ... (four loads in flight); with SL > 1 the
// SL slice sums are then added in slice order through LDS, so the result is
// deterministic.  SL (1, 4 or 16) is chosen from the quad count alone, which
// keeps enough loads in flight when few quads take many splits.  Elements
// i = 4q + j are stored in storage order of the partials; Cp is the channel
// stride of the tap axis (pad4(C), or C for the packed layout), and each
// split's partials start 4 * ceil(OC*KK*Cp / 4) floats apart.  Padding
// channels (c >= C) and the tail past OC*KK*Cp are dropped.
//
// The same launch carries the conv backward's bias-gradient sum as side.nRow
// extra blocks after the nMain finishing blocks (rowsum_block), so that it
// costs no launch of its own; the two jobs touch disjoint buffers.
//
// dbCol (not null, KK == 1, !trans): the tap axis' column C holds the bias
// gradient (a GEMM operand row of ones), written to dbCol[oc].
template <int SL>
__global__ void __launch_bounds__(256)
    k_dw_final(const f4* __restrict__ part, float* __restrict__ dw, uint32_t OC, uint32_t C,
               uint32_t KK, uint32_t Cp, uint32_t splits, uint32_t trans, uint32_t nMain,
               BwdSide side, float* __restrict__ dbCol, WPerm pw) {
  if (blockIdx.x >= nMain) {
    // Extra blocks: the bias-gradient sum (one per channel), then a filter
    // re-layout riding in this launch.
    const uint32_t e = blockIdx.x - nMain;
    if (e < side.nRow)
      rowsum_block(side.dbPart, side.db, side.dbRows, e);
    else
      permute_w_elem(pw, (e - side.nRow) * 256 + threadIdx.x);
    return;
  }
  constexpr uint32_t QB = 256 / SL;
  __shared__ f4 sh[SL][QB];
  const uint32_t N = KK * Cp, total = OC * N, nq = (total + 3) / 4;
  const uint32_t lq = threadIdx.x % QB, w = threadIdx.x / QB;
  const uint32_t q = blockIdx.x * QB + lq;
  f4 s = {0.f, 0.f, 0.f, 0.f};
  if (q < nq) {
    const size_t zs = nq;
    uint32_t z = w;
    // Eight loads in flight, added in z order.
    for (; z + 7 * SL < splits; z += 8 * SL) {
      f4 t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = part[(z + u * SL) * zs + q];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += t[u];
    }
    for (; z + 3 * SL < splits; z += 4 * SL) {
      const f4 a = part[z * zs + q], b = part[(z + SL) * zs + q];
      const f4 c = part[(z + 2 * SL) * zs + q], d = part[(z + 3 * SL) * zs + q];
      s += a;
      s += b;
      s += c;
      s += d;
    }
    for (; z < splits; z += SL) s += part[z * zs + q];
  }
  if constexpr (SL > 1) {
    sh[w][lq] = s;
    __syncthreads();
    if (w != 0) return;
    s = sh[0][lq];
#pragma unroll
    for (int k = 1; k < SL; ++k) s += sh[k][lq];
  }
  if (q >= nq) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t i = 4 * q + j;
    if (i >= total) break;
    uint32_t oc, n;
    if (trans) {
      n = i / OC;
      oc = i - n * OC;
    } else {
      oc = i / N;
      n = i - oc * N;
    }
    const uint32_t khw = n / Cp, c = n - khw * Cp;
    if (c < C)
      dw[(size_t(oc) * C + c) * KK + khw] = s[j];
    else if (dbCol && c == C)
      dbCol[oc] = s[j];
  }
}

// Slices per quad for k_dw_final: the fewest (1, 4, 16) that give about
// 128 K threads, never more than the splits.
static uint32_t dw_final_slices(uint32_t nq, uint32_t splits) {
  uint32_t sl = 1;
  while (sl < 16 && size_t(nq) * sl < 131072 && sl * 4 <= splits) sl *= 4;
  return sl;
}

static bool dw_final(const float* part, float* dw, uint32_t OC, uint32_t C, uint32_t KK,
                     uint32_t Cp, uint32_t splits, bool trans, BwdSide side = BwdSide{},
                     float* dbCol = nullptr, const WPerm& pw = WPerm{}) {
  const uint32_t nq = cdiv(size_t(OC) * KK * Cp, 4), sl = dw_final_slices(nq, splits);
  const f4* p4 = reinterpret_cast<const f4*>(part);
  const uint32_t tr = trans ? 1u : 0u;
  const uint32_t nMain = cdiv(nq, 256u / sl);
  const dim3 grid(nMain + side.nRow + pw.blocks());
  if (sl == 1)
    hipLaunchKernelGGL(k_dw_final<1>, grid, dim3(256), 0, stream(), p4, dw, OC, C, KK, Cp, splits,
                       tr, nMain, side, dbCol, pw);
  else if (sl == 4)
    hipLaunchKernelGGL(k_dw_final<4>, grid, dim3(256), 0, stream(), p4, dw, OC, C, KK, Cp, splits,
                       tr, nMain, side, dbCol, pw);
  else
    hipLaunchKernelGGL(k_dw_final<16>, grid, dim3(256), 0, stream(), p4, dw, OC, C, KK, Cp,
                       splits, tr, nMain, side, dbCol, pw);
  return check_launch("dw_final");
}

// Split-K finish for an NCHW output: out[b][m][pix] = act(sum_z part[z][m][n]
// + bias[m]) for n = b*HW + pix, z summed in order (deterministic).
__global__ void k_splitk_nchw(const float* __restrict__ part, const float* __restrict__ bias,
                              float* __restrict__ out, uint32_t M, uint32_t N, uint32_t HW,
                              uint32_t splits, uint32_t act) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * N) return;
  const uint32_t m = i / N, n = i - m * N;
  float z = 0.f;
  for (uint32_t k = 0; k < splits; ++k) z += part[size_t(k) * M * N + i];
  if (bias) z += bias[m];
  if (act == 1)
    z = fmaxf(z, 0.f);
  else if (act == 2)
    z = tanhf(z);
  const uint32_t b = n / HW, pix = n - b * HW;
  out[(size_t(b) * M + m) * HW + pix] = z;
}

// Quad form of k_splitk_nchw for N % 4 == 0: 16-byte partial loads, four in
// flight, z still summed in order (same bits as the scalar form).  The four
// elements of a quad lie in one row m and may straddle an image boundary.
__global__ void __launch_bounds__(256)
    k_splitk_nchw4(const f4* __restrict__ part, const float* __restrict__ bias,
                   float* __restrict__ out, uint32_t M, uint32_t N, uint32_t HW, uint32_t splits,
                   uint32_t act) {
  const uint32_t q = blockIdx.x * 256 + threadIdx.x;
  const uint32_t nq = M * (N / 4);
  if (q >= nq) return;
  f4 s = sum_splits4(part + q, nq, splits);
  const uint32_t m = (4 * q) / N, n0 = 4 * q - m * N;
  uint32_t b = n0 / HW, pix = n0 - b * HW;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float v = s[j];
    if (bias) v += bias[m];
    if (act == 1)
      v = fmaxf(v, 0.f);
    else if (act == 2)
      v = tanhf(v);
    s[j] = v;
  }
  if (pix + 3 < HW) {
    // The quad lies in one plane: one 16-byte store (4-byte aligned for planes
    // of odd size; unaligned access is on).
    stu(out + (size_t(b) * M + m) * HW + pix, s);
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    out[(size_t(b) * M + m) * HW + pix] = s[j];
    if (++pix == HW) {
      pix = 0;
      ++b;
    }
  }
}

// k_splitk_nchw that also leaves the batch-norm statistics of what it
// stores (as EpiNCHWStats): block (piece, m) finishes columns
// [piece * kStatsSpan, (piece + 1) * kStatsSpan) of row m, with the same sum
// order as k_splitk_nchw / k_splitk_nchw4 (the same bits of y), and writes
// the double sums of z and z*z over them to stats[(m * pieces + piece) * 2].
// Q4 (N % 4 == 0, 16-byte aligned partials): thread t takes the quad of
// columns 4t .. 4t + 3 of the block's span, as k_splitk_nchw4 does.
constexpr uint32_t kStatsSpan = 1024;
template <bool Q4>
__global__ void __launch_bounds__(256)
    k_splitk_nchw_stats(const float* __restrict__ part, const float* __restrict__ bias,
                        float* __restrict__ out, uint32_t M, uint32_t N, uint32_t HW,
                        uint32_t splits, uint32_t act, double* __restrict__ stats,
                        uint32_t pieces, FastDiv dHW) {
  __shared__ double sh[4];
  const uint32_t m = blockIdx.y, piece = blockIdx.x;
  const float bv = bias ? bias[m] : 0.f;
  double a0 = 0.0, a1 = 0.0;
  if constexpr (Q4) {
    const uint32_t n0 = piece * kStatsSpan + 4 * threadIdx.x;
    if (n0 < N) {
      const size_t nq = size_t(M) * (N / 4);
      f4 z = sum_splits4(reinterpret_cast<const f4*>(part) + (size_t(m) * N + n0) / 4, nq, splits);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        z[e] = epi_act(z[e] + bv, act);
        a0 += double(z[e]);
        a1 += double(z[e]) * double(z[e]);
      }
      uint32_t b = fdiv(n0, dHW), pix = n0 - b * HW;
      if (pix + 3 < HW) {
        stu(out + (size_t(b) * M + m) * HW + pix, z);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          out[(size_t(b) * M + m) * HW + pix] = z[e];
          if (++pix == HW) {
            pix = 0;
            ++b;
          }
        }
      }
    }
  } else {
#pragma unroll
    for (uint32_t u = 0; u < kStatsSpan / 256; ++u) {
      const uint32_t n = piece * kStatsSpan + u * 256 + threadIdx.x;
      if (n >= N) break;
      const size_t i = size_t(m) * N + n;
      float z = 0.f;
      for (uint32_t k = 0; k < splits; ++k) z += part[size_t(k) * M * N + i];
      z = epi_act(z + bv, act);
      const uint32_t b = fdiv(n, dHW), pix = n - b * HW;
      out[(size_t(b) * M + m) * HW + pix] = z;
      a0 += double(z);
      a1 += double(z) * double(z);
    }
  }
  const double s0 = block_sum256(a0, sh);
  const double s1 = block_sum256(a1, sh);
  if (threadIdx.x == 0) {
    double* d = stats + (size_t(m) * pieces + piece) * 2;
    d[0] = s0;
    d[1] = s1;
  }
}

// Zero-padded copy of a row-major [rows][cols] matrix to row stride ldp.
__global__ void k_pad_cols(const float* __restrict__ in, float* __restrict__ out, uint32_t rows,
                           uint32_t cols, uint32_t ldp) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(rows) * ldp) return;
  const uint32_t r = uint32_t(i / ldp), c = uint32_t(i - size_t(r) * ldp);
  out[i] = c < cols ? in[size_t(r) * cols + c] : 0.f;
}

bool pad_cols(const float* in, float* out, uint32_t rows, uint32_t cols, uint32_t ldp) {
  hipLaunchKernelGGL(k_pad_cols, dim3(cdiv(size_t(rows) * ldp, 256)), dim3(256), 0, stream(), in,
                     out, rows, cols, ldp);
  return check_launch("pad_cols");
}

static bool split_nchw_stats(const float* part, const float* bias, float* out, uint32_t M,
                             uint32_t N, uint32_t HW, uint32_t splits, uint32_t act,
                             double* stats, uint32_t pieces) {
  if (N % 4 == 0 && aligned16(part))
    hipLaunchKernelGGL(k_splitk_nchw_stats<true>, dim3(pieces, M), dim3(256), 0, stream(), part,
                       bias, out, M, N, HW, splits, act, stats, pieces, make_fastdiv(HW));
  else
    hipLaunchKernelGGL(k_splitk_nchw_stats<false>, dim3(pieces, M), dim3(256), 0, stream(), part,
                       bias, out, M, N, HW, splits, act, stats, pieces, make_fastdiv(HW));
  return check_launch("splitk_nchw");
}
bool split_nchw(const float* part, const float* bias, float* out, uint32_t M, uint32_t N,
                       uint32_t HW, uint32_t splits, uint32_t act) {
  if (N % 4 == 0 && aligned16(part))
    hipLaunchKernelGGL(k_splitk_nchw4, dim3(cdiv(size_t(M) * (N / 4), 256)), dim3(256), 0,
                       stream(), reinterpret_cast<const f4*>(part), bias, out, M, N, HW, splits,
                       act);
  else
    hipLaunchKernelGGL(k_splitk_nchw, dim3(cdiv(size_t(M) * N, 256)), dim3(256), 0, stream(),
                       part, bias, out, M, N, HW, splits, act);
  return check_launch("splitk_nchw");
}

// Deterministic split-K sum of row-major partials into c (n elements).
bool split_sum(const float* part, float* c, uint32_t n, uint32_t splits) {
  if (n % 4 == 0 && aligned16(part) && aligned16(c))
    hipLaunchKernelGGL(k_splitk_sum4, dim3(cdiv(n / 4, 256u)), dim3(256), 0, stream(),
                       reinterpret_cast<const f4*>(part), reinterpret_cast<f4*>(c), n / 4, splits);
  else
    hipLaunchKernelGGL(k_splitk_sum, dim3(cdiv(n, 256u)), dim3(256), 0, stream(), part, c, n,
                       splits);
  return check_launch("splitk_sum");
}

// ----------------------------------------------------------- NHWC copies
size_t nhwc_floats(uint32_t B, uint32_t C, uint32_t H, uint32_t W) {
  return size_t(B) * H * W * pad4(C);
}

// Bias-gradient partial rows per channel of the transpose pass (the pixel
// blocks of every plane): 128-pixel blocks for up to 16 channels, else 64.
static uint32_t to_nhwc_rows(uint32_t B, uint32_t Cp, uint32_t HW) {
  return B * (Cp <= 16 ? cdiv(HW, 128) : cdiv(HW, 64));
}

// parts: out is bf16 parts (C > 16); xs rides in that launch.
static bool to_nhwc_masked(const float* in, const float* y, float* out, float* dbPart,
                           uint32_t B, uint32_t C, uint32_t HW, uint32_t* npbOut,
                           const WPerm& pw = WPerm{}, bool parts = false,
                           const XSplit& xs = XSplit{}) {
  const uint32_t Cp = pad4(C), nblk = pad16(C) / 16;
  // Family "conv_grad_nhwc": the masked dy -> G pass of the conv backward
  // (reads dy and y, writes G); "nhwc": a plain copy of an activation.
  ProfScope prof(y ? "conv_grad_nhwc" : "nhwc", 0,
                 4.0 * double(B) * HW * ((y ? 2.0 : 1.0) * C + (parts ? 24 * nblk : Cp)) +
                     4.0 * double(xs.groups) * 8 * 2.5);
  if (Cp <= 8 && !y && !dbPart) {
    const uint32_t npix = B * HW;
    hipLaunchKernelGGL(k_to_nhwc_small, dim3(cdiv(npix, 256)), dim3(256), 0, stream(), in, out, C,
                       HW, Cp, npix, make_fastdiv(HW));
    return check_launch("to_nhwc") && (!pw.w || permute_w(pw));
  }
  const uint32_t npb = cdiv(HW, Cp <= 16 ? 128 : 64), ncb = Cp <= 16 ? 1 : cdiv(Cp, 32);
  const uint32_t nMain = npb * ncb * B, nPerm = pw.blocks();
  if (npbOut) *npbOut = npb;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nMain + nPerm + xs.blocks()), dim3(256), 0, stream(), in, y,
                       out, dbPart, C, HW, Cp, npb, ncb, B, nMain, pw, nblk, nPerm, xs, BnDxArgs{});
  };
  if (parts)
    go(k_to_nhwc<32, false, true>);
  else if (Cp <= 16)
    go(k_to_nhwc<16, false, false>);
  else
    go(k_to_nhwc<32, false, false>);
  return check_launch("to_nhwc");
}

uint32_t bn_dx_g_rows(uint32_t B, uint32_t C, uint32_t HW) { return to_nhwc_rows(B, pad4(C), HW); }

bool bn_dx_g(const float* x, const float* dy, const float* mean, const float* var,
             const float* gamma, const float* dg, const float* db, float eps, float* dx,
             uint32_t layout, float* g, float* dbPart, uint32_t B, uint32_t C, uint32_t HW) {
  const uint32_t Cp = pad4(C), nblk = pad16(C) / 16;
  const bool parts = layout == kGLayoutParts;
  if (uint64_t(B) * C * HW >= kOob || uint64_t(B) * HW * (parts ? 24 * nblk : Cp) >= kOob)
    return false;
  ProfScope prof("bn_bwd_dx", 0, 4.0 * double(B) * HW * (3.0 * C + (parts ? 24 * nblk : Cp)));
  const BnDxArgs bn{mean, var, gamma, dg, db, dx, eps, float(uint64_t(B) * HW)};
  // The same blocks (and bias partials) as the conv backward's transpose pass.
  const uint32_t npb = cdiv(HW, Cp <= 16 ? 128 : 64), ncb = Cp <= 16 ? 1 : cdiv(Cp, 32);
  const uint32_t nMain = npb * ncb * B;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nMain), dim3(256), 0, stream(), dy, x, g, dbPart, C, HW, Cp,
                       npb, ncb, B, nMain, WPerm{}, nblk, 0u, XSplit{}, bn);
  };
  if (parts)
    go(k_to_nhwc<32, true, true>);
  else if (Cp <= 16)
    go(k_to_nhwc<16, true, false>);
  else
    go(k_to_nhwc<32, true, false>);
  return check_launch("batchnorm_backward_dx");
}

bool to_nhwc(const float* x, float* out, uint32_t B, uint32_t C, uint32_t H, uint32_t W) {
  return to_nhwc_masked(x, nullptr, out, nullptr, B, C, H * W, nullptr);
}

// Channel-packed, zero-padded copy (fewer than four channels): out[((b*Hp +
// h)*Wp + w)*C + c] = x[b][c][h - p][w - p], zero in the border.  A thread
// takes 4 consecutive padded pixels of one row: one 16-byte load per channel
// (4-byte aligned: unaligned access is on) where the 4 source columns lie in
// the image, else element loads, and C 16-byte stores (the 4*C outputs are
// contiguous and 16-byte aligned when Wp % 4 == 0; otherwise element stores).
template <int C>
__global__ void k_to_pk(const float* __restrict__ x, float* __restrict__ out, uint32_t H,
                        uint32_t W, uint32_t p, uint32_t Hp, uint32_t Wp, uint32_t WQ, uint32_t nq,
                        FastDiv dWQ, FastDiv dHp) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nq) return;
  const uint32_t t = fdiv(i, dWQ), wq = i - t * WQ;  // t = b * Hp + h
  const uint32_t b = fdiv(t, dHp), h = t - b * Hp;
  const uint32_t w0 = 4 * wq, ih = h - p;  // ih wraps when in the border
  const int iw0 = int(w0) - int(p);
  const bool rowin = ih < H;
  const bool fullin = rowin && iw0 >= 0 && iw0 + 4 <= int(W);
  float o[4 * C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const float* src = x + ((size_t(b) * C + c) * H + (rowin ? ih : 0)) * W;
    f4 q;
    if (fullin) {
      q = ldu<f4>(src + iw0);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int iw = iw0 + e;
        q[e] = (rowin && iw >= 0 && iw < int(W)) ? src[iw] : 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e * C + c] = q[e];
  }
  float* dst = out + (size_t(t) * Wp + w0) * C;
  if (Wp % 4 == 0) {
#pragma unroll
    for (int k = 0; k < C; ++k) *reinterpret_cast<f4*>(dst + 4 * k) = f4{o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (w0 + e < Wp) {
#pragma unroll
        for (int c = 0; c < C; ++c) dst[e * C + c] = o[e * C + c];
      }
  }
}

// Stride-phase copy (see PsParams): thread (b, r, c, column quad cq) reads
// the 4*S consecutive source elements of padded row r from column 4*cq*S - p
// (16-byte loads at 4-byte alignment where they lie in the image, element
// loads at its edges) and stores one 16-byte quad per phase.
template <int S>
__global__ void __launch_bounds__(256)
    k_to_ps(const float* __restrict__ x, float* __restrict__ out, uint32_t C, uint32_t H,
            uint32_t W, uint32_t p, uint32_t Hp, uint32_t Ncol, uint32_t nq, FastDiv dNQ,
            FastDiv dC, FastDiv dHp) {
  const uint32_t i = xcd_block_id() * 256 + threadIdx.x;  // neighbouring rows share an L2
  if (i >= nq) return;
  const uint32_t NQ = dNQ.d;
  const uint32_t t = fdiv(i, dNQ), cq = i - t * NQ;     // t = (b*Hp + r)*C + c
  const uint32_t u = fdiv(t, dC), c = t - u * C;        // u = b*Hp + r
  const uint32_t b = fdiv(u, dHp), r = u - b * Hp;
  const uint32_t ih = r - p;                            // wraps in the border
  const int iw0 = int(4 * cq * S) - int(p);
  const bool rowin = ih < H;
  const float* src = x + ((size_t(b) * C + c) * H + (rowin ? ih : 0)) * W;
  float v[4 * S];
  if (rowin && iw0 >= 0 && iw0 + 4 * S <= int(W)) {
#pragma unroll
    for (int q = 0; q < S; ++q) {
      const f4 a = ldu<f4>(src + iw0 + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * q + e] = a[e];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4 * S; ++j) {
      const int iw = iw0 + j;
      v[j] = (rowin && iw >= 0 && iw < int(W)) ? src[iw] : 0.f;
    }
  }
  float* dst = out + size_t(t) * S * Ncol + 4 * cq;
#pragma unroll
  for (int ph = 0; ph < S; ++ph)
    *reinterpret_cast<f4*>(dst + ph * Ncol) = f4{v[ph], v[S + ph], v[2 * S + ph], v[3 * S + ph]};
}

// Masked gradient on the padded pixel grid for the stride-phase dW GEMM:
// G_pad[b][oc][oh][ow] = dy masked by y (y <= 0 -> 0; a NaN y keeps it) for
// ow < OW, 0 for OW <= ow < OWp.  Block = one chunk of up to kMaskChunk
// padded elements of one (b, oc) plane, four 16-byte quads per thread (all
// loaded before any is stored); dbPart[oc][b*nchunk + chunk] = the block's
// sum of the masked values (thread, wave, then wave order).
constexpr uint32_t kMaskChunk = 4096;
__global__ void __launch_bounds__(256)
    k_mask_pad(const float* __restrict__ dy, const float* __restrict__ y, float* __restrict__ g,
               float* __restrict__ dbPart, uint32_t OC, uint32_t OH, uint32_t OW, uint32_t OWp,
               uint32_t nchunk, uint32_t nB, FastDiv dChunk, FastDiv dOWp) {
  __shared__ float sh[4];
  // XCD-contiguous numbering: neighbouring chunks share the cache lines of
  // rows of odd length, and then share an L2.
  const uint32_t id = xcd_block_id();
  const uint32_t plane = fdiv(id, dChunk), chunk = id - plane * nchunk;
  const uint32_t OHWp = OH * OWp;
  const float* dyp = dy + size_t(plane) * OH * OW;
  const float* yp = y ? y + size_t(plane) * OH * OW : nullptr;
  // Every quad is one 16-byte load (4-byte aligned; unaligned access is on),
  // issued back to back with no branch between them: a quad that would run
  // past its row (or a thread past the plane) loads the 4 elements ending at
  // the row's last one (at the plane's start) and shifts them into place,
  // zero-filling.  Rows of fewer than 4 elements take element loads.
  f4 v[4], m[4];
  uint32_t e[4];
  if (OW >= 4) {
    uint32_t shift[4], src[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      e[j] = chunk * kMaskChunk + 4 * (threadIdx.x + 256 * j);
      const uint32_t ej = e[j] < OHWp ? e[j] : 0u;
      const uint32_t oh = fdiv(ej, dOWp), ow = ej - oh * OWp;
      shift[j] = ow + 4 <= OW ? 0u : ow + 4 - OW;  // 1..3 for a row's last quad
      src[j] = oh * OW + ow - shift[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = ldu<f4>(dyp + src[j]);
      m[j] = yp ? ldu<f4>(yp + src[j]) : f4{1.f, 1.f, 1.f, 1.f};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t d = shift[j];
      const f4 a = v[j], b = m[j];
      v[j] = f4{d == 0 ? a[0] : d == 1 ? a[1] : d == 2 ? a[2] : a[3],
                d == 0 ? a[1] : d == 1 ? a[2] : d == 2 ? a[3] : 0.f,
                d == 0 ? a[2] : d == 1 ? a[3] : 0.f, d == 0 ? a[3] : 0.f};
      m[j] = f4{d == 0 ? b[0] : d == 1 ? b[1] : d == 2 ? b[2] : b[3],
                d == 0 ? b[1] : d == 1 ? b[2] : d == 2 ? b[3] : 1.f,
                d == 0 ? b[2] : d == 1 ? b[3] : 1.f, d == 0 ? b[3] : 1.f};
      if (e[j] >= OHWp) v[j] = f4{0.f, 0.f, 0.f, 0.f};
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      e[j] = chunk * kMaskChunk + 4 * (threadIdx.x + 256 * j);
      v[j] = m[j] = f4{0.f, 0.f, 0.f, 0.f};
      if (e[j] >= OHWp) continue;
      const uint32_t oh = fdiv(e[j], dOWp), ow = e[j] - oh * OWp;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[j][q] = ow + q < OW ? dyp[oh * OW + ow + q] : 0.f;
        m[j][q] = (yp && ow + q < OW) ? yp[oh * OW + ow + q] : 1.f;
      }
    }
  }
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int q = 0; q < 4; ++q) v[j][q] = m[j][q] <= 0.f ? 0.f : v[j][q];
    if (e[j] < OHWp) *reinterpret_cast<f4*>(g + size_t(plane) * OHWp + e[j]) = v[j];
    sum += (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
  }
  if (dbPart == nullptr) return;
  sum = wave_reduce(sum);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t b = plane / OC, oc = plane - b * OC;
    dbPart[size_t(oc) * nB * nchunk + size_t(b) * nchunk + chunk] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  }
}

// Layout of the conv input copy: channel-innermost (C >= 4), stride-phase
// (C < 4, stride <= 4) or channel-packed (C < 4, larger strides).
bool ps_x(const ConvGeom& g) { return g.C < 4 && g.s <= 4; }
// Pointwise convolutions (1 x 1, stride 1, no padding, planes of a multiple
// of 4 pixels, at least 4 channels) read x, dy and write y, dx in NCHW: the
// GEMMs take the planes as they are, with no channel-innermost copy.
bool pw_x(const ConvGeom& g) {
  return g.k == 1 && g.s == 1 && g.p == 0 && (g.H * g.W) % 4 == 0 && g.C >= 4;
}
bool packed_x(const ConvGeom& g) { return g.C < 4 && g.s > 4; }
// Does the backward run on bf16 parts (dce_igemm_parts.h)?  The parts cost
// traffic (the forward's copy of x split to 6 bytes a value, G written and read
// as 6 instead of 4), which C * OC * k * k products per pixel have to pay for:
// 3 x 3 layers over 32 -> 32 and 32 -> 64 channels lose (forward and backward on
// fp32 and on parts 111 and 114 us at 8 x 128 x 128, 70 and 73 at 8 x 64 x 64),
// 96 -> 32 and 64 -> 64 gain (246 and 228, 104 and 94 us), 384 -> 256 at 13 x
// 13, b128: 942 and 714 us.
bool conv_parts(const ConvGeom& g) {
  if (g.C < 32 || g.OC < 32) return false;
  // dW over less than one 16-deep step gains nothing, and a sum of one product is
  // the one that parts round worse (2.6e-8 against 2.5e-8).
  if (g.B * g.OH * g.OW < 16) return false;
  const double products = double(g.k) * g.k * g.C * g.OC, x = double(g.B) * g.C * g.H * g.W;
  if (products < 210.0 * (g.C + g.OC)) return false;
  // At stride 3 and more an output pixel stands for s * s pixels of x.  Where
  // their parts are real traffic they have to be paid for too (118 x 289 x 15 x
  // 108 -> 88, k3 s4 583 on fp32, 649 us on parts; 53 x 56 x 93 x 94 -> 510, k3
  // s4 687 and 751); smaller layers are bound by launches and latency and gain
  // 9 % over 96 shapes (from -43 to +6 %).
  if (g.s >= 3 && x >= 1e7 && products < 210.0 * (x / (double(g.B) * g.OH * g.OW) + g.OC))
    return false;
  return parts_floats(size_t(g.B) * g.H * g.W, g.C) < kOob &&
         parts_floats(size_t(g.B) * g.OH * g.OW, g.OC) < kOob &&
         parts_floats(size_t(g.C) * g.k * g.k, g.OC) < kOob;
}

PsGeom ps_geom(const ConvGeom& g) {
  PsGeom q;
  q.Hp = g.H + 2 * g.p;
  q.OWp = pad4(g.OW);
  q.OHWp = g.OH * q.OWp;
  // Columns: the padded image, and every quad a padded output row's taps
  // read (up to OWp - 1 + (k - 1) / S).
  const uint32_t cols = std::max(cdiv(g.W + 2 * g.p, g.s), q.OWp + (g.k - 1) / g.s);
  q.Ncol = pad4(cols);
  q.RS = g.C * g.s * q.Ncol;
  q.floats = size_t(g.B) * q.Hp * q.RS;
  return q;
}

size_t xcopy_floats(const ConvGeom& g) {
  if (pw_x(g)) return 4;  // no copy: a placeholder handle
  if (ps_x(g)) return ps_geom(g).floats;
  if (!packed_x(g)) return nhwc_floats(g.B, g.C, g.H, g.W);
  return size_t(g.B) * (g.H + 2 * g.p) * (g.W + 2 * g.p) * g.C;
}

// Floats of the copy of x that the backward's general path reads: the kept one,
// or one it builds (on parts always: the kept copy is the forward's, fp32, so
// that a forward whose backward never comes pays nothing for it; a pointwise
// layer that takes the general path, for its ReLU mask, has kept none).
static size_t xbuild_floats(const ConvGeom& g) {
  if (conv_parts(g)) return parts_floats(size_t(g.B) * g.H * g.W, g.C);
  return pw_x(g) ? nhwc_floats(g.B, g.C, g.H, g.W) : xcopy_floats(g);
}

uint32_t xcopy_tag(const ConvGeom& g) {
  if (pw_x(g)) return 0x40000u;
  if (ps_x(g)) return 0x20000u + g.p + (g.s << 8) + (g.k << 12);
  return packed_x(g) ? 0x10000u + g.p : pad4(g.C);
}

static bool to_ps(const float* x, float* out, const ConvGeom& g) {
  const PsGeom q = ps_geom(g);
  const uint32_t NQ = q.Ncol / 4, nq = g.B * q.Hp * g.C * NQ;
  ProfScope prof("nhwc", 0, 4.0 * (double(g.B) * g.C * g.H * g.W + double(q.floats)));
  const dim3 grid(cdiv(nq, 256));
  const FastDiv fNQ = make_fastdiv(NQ), fC = make_fastdiv(g.C), fHp = make_fastdiv(q.Hp);
#define DCE_PS(S_)                                                                            \
  if (g.s == S_)                                                                              \
    hipLaunchKernelGGL(k_to_ps<S_>, grid, dim3(256), 0, stream(), x, out, g.C, g.H, g.W, g.p, \
                       q.Hp, q.Ncol, nq, fNQ, fC, fHp);
  DCE_PS(1) DCE_PS(2) DCE_PS(3) DCE_PS(4)
#undef DCE_PS
  return check_launch("to_ps");
}

PsParams ps_params(const float* src, const ConvGeom& g) {
  const PsGeom q = ps_geom(g);
  const uint32_t KK = g.k * g.k;
  return PsParams{src, q.RS, q.Hp, g.s, q.Ncol, g.C, g.k, KK, g.C * KK, q.OWp, q.OHWp,
                  g.B * q.OHWp, uint32_t(q.floats), make_fastdiv(q.OHWp), make_fastdiv(q.OWp),
                  make_fastdiv(KK), make_fastdiv(g.k), make_fastdiv(g.s)};
}

// G_pad (and, with dbPart, the bias-gradient partials: OC rows of
// B * nchunk); returns nchunk.
static uint32_t mask_pad(const float* dy, const float* y, float* gp, float* dbPart,
                         const ConvGeom& g, bool* ok) {
  const PsGeom q = ps_geom(g);
  const uint32_t nchunk = cdiv(q.OHWp, kMaskChunk), planes = g.B * g.OC;
  ProfScope prof("conv_grad_nhwc", 0, 4.0 * (2.0 * g.B * g.OC * g.OH * g.OW + double(planes) * q.OHWp));
  hipLaunchKernelGGL(k_mask_pad, dim3(planes * nchunk), dim3(256), 0, stream(), dy, y, gp, dbPart,
                     g.OC, g.OH, g.OW, q.OWp, nchunk, g.B, make_fastdiv(nchunk),
                     make_fastdiv(q.OWp));
  *ok = check_launch("mask_pad");
  return nchunk;
}

static bool to_pk(const float* x, float* out, const ConvGeom& g) {
  const uint32_t Hp = g.H + 2 * g.p, Wp = g.W + 2 * g.p, npix = g.B * Hp * Wp;
  const uint32_t WQ = cdiv(Wp, 4), nq = g.B * Hp * WQ;
  ProfScope prof("nhwc", 0, 4.0 * (double(g.B) * g.C * g.H * g.W + double(npix) * g.C));
  const dim3 grid(cdiv(nq, 256));
  const FastDiv fWQ = make_fastdiv(WQ), fHp = make_fastdiv(Hp);
  if (g.C == 1)
    hipLaunchKernelGGL(k_to_pk<1>, grid, dim3(256), 0, stream(), x, out, g.H, g.W, g.p, Hp, Wp, WQ,
                       nq, fWQ, fHp);
  else if (g.C == 2)
    hipLaunchKernelGGL(k_to_pk<2>, grid, dim3(256), 0, stream(), x, out, g.H, g.W, g.p, Hp, Wp, WQ,
                       nq, fWQ, fHp);
  else
    hipLaunchKernelGGL(k_to_pk<3>, grid, dim3(256), 0, stream(), x, out, g.H, g.W, g.p, Hp, Wp, WQ,
                       nq, fWQ, fHp);
  return check_launch("to_pk");
}

PkParams pk_params(const float* src, const ConvGeom& g) {
  const uint32_t Hp = g.H + 2 * g.p, Wp = g.W + 2 * g.p, OHW = g.OH * g.OW, kC = g.k * g.C;
  return PkParams{src, Wp * g.C, Hp * Wp * g.C, g.C, g.k, g.s, kC, g.k * kC, g.OW, OHW,
                  g.B * OHW, uint32_t(xcopy_floats(g)), make_fastdiv(OHW), make_fastdiv(g.OW),
                  make_fastdiv(kC)};
}

// ----------------------------------------------------------- conv forward
// Output pixels as GEMM columns: split-K partials go to a row-major [M][N]
// workspace and k_splitk_nchw finishes (bias, activation, NCHW scatter).
template <bool S1, bool BLK>
struct FwdRun {
  const float* wp;
  const float* xn;
  const float* bias;
  float* y;
  float* part;
  ConvGeom g;
  uint32_t act, splits;
  double* stats;  // stride 1: BN statistics of y (pieces as stats_buffer sets them)
  uint32_t pieces;
  template <int MT, int NT, int KT>
  int occ(bool split) const {
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPixRK<NT, KT, true, S1, BLK>;
    return split ? occupancy(k_igemm<MT, NT, KT, LA, LB, EpiRowMajor>)
                 : occupancy(k_igemm<MT, NT, KT, LA, LB, EpiNCHW>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    const uint32_t Cp = pad4(g.C), KK = g.k * g.k, kdim = KK * Cp;
    const uint32_t OHW = g.OH * g.OW, N = g.B * OHW;
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPixRK<NT, KT, true, S1, BLK>;
    const typename LA::Params pa{wp, kdim, g.OC, kdim, g.OC * kdim};
    const typename LB::Params pb{xn, g.H, g.W, Cp, g.k, g.s, g.p, g.OW, OHW, N, kdim,
                                 g.B * g.H * g.W * Cp, make_fastdiv(OHW), make_fastdiv(g.OW),
                                 make_fastdiv(BLK ? KK : Cp), make_fastdiv(g.k)};
    const uint32_t kt = cdiv(kdim, KT);
    const EpiNCHW::Params pe{y, bias, g.OC, OHW, N, act, make_fastdiv(OHW)};
    if (splits > 1) {
      const EpiRowMajor::Params pr{part, g.OC, N, N, g.OC * N};
      return launch<MT, NT, KT, LA, LB, EpiRowMajor>(pa, pb, pr, g.OC, N, kt, splits,
                                                    "conv_forward") &&
             (stats ? split_nchw_stats(part, bias, y, g.OC, N, OHW, splits, act, stats, pieces)
                    : split_nchw(part, bias, y, g.OC, N, OHW, splits, act));
    }
    if constexpr (S1) {
      if (stats) {
        const EpiNCHWStats::Params ps{pe, stats, pieces};
        return launch<MT, NT, KT, LA, LB, EpiNCHWStats>(pa, pb, ps, g.OC, N, kt, 1,
                                                        "conv_forward");
      }
    }
    return launch<MT, NT, KT, LA, LB, EpiNCHW>(pa, pb, pe, g.OC, N, kt, 1, "conv_forward");
  }
};

// Forward over the channel-packed copy (C < 4): K runs over the unpadded
// taps (kh, kw, c), filters padded to pad4(KK * C) per row.
struct FwdPkRun {
  const float* wp;
  const float* xp;
  const float* bias;
  float* y;
  float* part;
  ConvGeom g;
  uint32_t act, splits;
  template <int MT, int NT, int KT>
  int occ(bool split) const {
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPkRK<NT, KT>;
    return split ? occupancy(k_igemm<MT, NT, KT, LA, LB, EpiRowMajor>)
                 : occupancy(k_igemm<MT, NT, KT, LA, LB, EpiNCHW>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    const uint32_t kdim = pad4(g.k * g.k * g.C);
    const uint32_t OHW = g.OH * g.OW, N = g.B * OHW;
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPkRK<NT, KT>;
    const typename LA::Params pa{wp, kdim, g.OC, kdim, g.OC * kdim};
    const PkParams pb = pk_params(xp, g);
    const uint32_t kt = cdiv(kdim, KT);
    const EpiNCHW::Params pe{y, bias, g.OC, OHW, N, act, make_fastdiv(OHW)};
    if (splits > 1) {
      const EpiRowMajor::Params pr{part, g.OC, N, N, g.OC * N};
      return launch<MT, NT, KT, LA, LB, EpiRowMajor>(pa, pb, pr, g.OC, N, kt, splits,
                                                    "conv_forward") &&
             split_nchw(part, bias, y, g.OC, N, OHW, splits, act);
    }
    return launch<MT, NT, KT, LA, LB, EpiNCHW>(pa, pb, pe, g.OC, N, kt, 1, "conv_forward");
  }
};

// Forward over the stride-phase copy (C < 4, stride <= 4): K runs over the
// taps (c, kh, kw), the filters' own order (rows padded to pad4(C*KK)); the
// columns are the padded pixel grid, written through EpiNCHWPad (no split).
struct FwdPsRun {
  const float* wp;
  const float* xs;
  const float* bias;
  float* y;
  ConvGeom g;
  uint32_t act;
  template <int MT, int NT, int KT>
  int occ(bool) const {
    return occupancy(k_igemm<MT, NT, KT, LdDenseRK<MT, KT>, LdPsKR<NT, KT>, EpiNCHWPad>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    const uint32_t kdim = pad4(g.C * g.k * g.k);
    using LA = LdDenseRK<MT, KT>;
    using LB = LdPsKR<NT, KT>;
    const typename LA::Params pa{wp, kdim, g.OC, kdim, g.OC * kdim};
    const PsParams pb = ps_params(xs, g);
    const EpiNCHWPad::Params pe{y, bias, g.OC, g.OH * g.OW, g.OW, pb.OWp, pb.OHWp, pb.npix, act,
                                pb.dOHWp, pb.dOWp};
    return launch<MT, NT, KT, LA, LB, EpiNCHWPad>(pa, pb, pe, g.OC, pb.npix, cdiv(kdim, KT), 1,
                                                  "conv_forward");
  }
};

static bool conv_forward_ps(const float* x, float* keep, const float* w, const float* bias,
                            float* y, const ConvGeom& g, uint32_t act) {
  const PsGeom q = ps_geom(g);
  const uint32_t taps = g.C * g.k * g.k, kdim = pad4(taps), N = g.B * q.OHWp;
  if (!operand_fits(q.floats, "conv_forward") || !operand_fits(size_t(g.OC) * kdim, "conv_forward"))
    return false;
  TileCfg cfg = choose("DCE_TUNE_FWD", g.OC, N, kdim, 1, true,
                       [&](const TileCfg& t) { return tiles_occ16(t, FwdPsRun{}); }, true);
  cfg.splits = 1;  // the padded-grid epilogue writes the output directly
  const size_t nw = al64(size_t(g.OC) * kdim);
  float* ws = workspace(nw + (keep ? 0 : al64(q.floats)));
  if (!ws) return false;
  float* xs = keep ? keep : ws + nw;
  if (!to_ps(x, xs, g)) return false;
  if (!pad_cols(w, ws, g.OC, taps, kdim)) return false;
  ProfScope prof("conv_fwd", 2.0 * g.OC * taps * double(g.B) * g.OH * g.OW,
                 4.0 * (double(g.B) * g.C * g.H * g.W + double(g.B) * g.OC * g.OH * g.OW));
  return tiles_dispatch16(cfg, FwdPsRun{ws, xs, bias, y, g, act});
}

// Pointwise forward: y[oc][n] = sum_c w[oc][c] x[c][n] over the pixels n =
// b*HW + pix of NCHW x, filters padded to pad4(C) per row.
struct FwdPwRun {
  const float* wp;
  const float* x;
  const float* bias;
  float* y;
  float* part;
  ConvGeom g;
  uint32_t act, splits;
  double* stats;  // BN statistics of y (pieces as stats_buffer sets them)
  uint32_t pieces;
  template <int MT, int NT, int KT>
  int occ(bool split) const {
    using LA = LdDenseRK<MT, KT>;
    using LB = LdNchwKR<NT, KT>;
    return split ? occupancy(k_igemm<MT, NT, KT, LA, LB, EpiRowMajor>)
                 : occupancy(k_igemm<MT, NT, KT, LA, LB, EpiNCHW>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    const uint32_t Cp = pad4(g.C), HW = g.H * g.W, N = g.B * HW;
    using LA = LdDenseRK<MT, KT>;
    using LB = LdNchwKR<NT, KT>;
    const typename LA::Params pa{wp, Cp, g.OC, Cp, g.OC * Cp};
    const NchwKRParams pb{x, g.C, HW, N, g.B * g.C * HW, make_fastdiv(HW)};
    const uint32_t kt = cdiv(Cp, KT);
    const EpiNCHW::Params pe{y, bias, g.OC, HW, N, act, make_fastdiv(HW)};
    if (splits > 1) {
      const EpiRowMajor::Params pr{part, g.OC, N, N, g.OC * N};
      return launch<MT, NT, KT, LA, LB, EpiRowMajor>(pa, pb, pr, g.OC, N, kt, splits,
                                                    "conv_forward") &&
             (stats ? split_nchw_stats(part, bias, y, g.OC, N, HW, splits, act, stats, pieces)
                    : split_nchw(part, bias, y, g.OC, N, HW, splits, act));
    }
    if (stats) {
      const EpiNCHWStats::Params ps{pe, stats, pieces};
      return launch<MT, NT, KT, LA, LB, EpiNCHWStats>(pa, pb, ps, g.OC, N, kt, 1, "conv_forward");
    }
    return launch<MT, NT, KT, LA, LB, EpiNCHW>(pa, pb, pe, g.OC, N, kt, 1, "conv_forward");
  }
};

// The buffer for the BN statistics of a conv forward's output when its GEMM
// leaves them (pixel GEMMs at stride 1 and pointwise GEMMs, no activation):
// one piece per column tile, or per kStatsSpan columns of the split-K finish.
static double* stats_buffer(ConvStatsReq* st, const TileCfg& cfg, uint32_t N, uint32_t act,
                            bool able) {
  if (!st || act != 0 || !able) return nullptr;
  const uint32_t pieces = cfg.splits > 1 ? cdiv(N, kStatsSpan) : cdiv(N, cfg.NT);
  double* d = st->get(st->ctx, pieces);
  if (d) st->pieces = pieces;
  return d;
}

// Pointwise products with dot products of at most 32 (expand forward,
// project dX): streaming-bound, one K tile or two per output tile.  For up to
// 160 output rows, unsplit 32-row tiles (rows filled exactly or nearly, more
// workgroups in flight) measured faster than the 64- and 128-row choices
// (MobileNetV2 b64: 96 x 200704 x 24 dX 37.6 -> 26.7 us, 144 x 200704 x 24
// forward and dX 46.2 -> 42.6 and 43.6 -> 39.9 us, 96 x 802816 x 16 forward
// 110.3 -> 107.4 us); at 192 rows (x 50176 x 32) they were no faster (dX)
// or 5 % slower (forward), so the rule stops at 160.  An override through
// DCE_TUNE_* keeps its tile.
static void narrow_pw(TileCfg& c, const char* var, uint32_t M, uint32_t kdim) {
  if (const char* e = getenv(var))
    if (*e) return;
  if (M <= 32 || M > 160 || kdim > 32) return;
  c = TileCfg{32, 128, 16, 1};
}

static bool conv_forward_pw(const float* x, const float* w, const float* bias, float* y,
                            const ConvGeom& g, uint32_t act, ConvStatsReq* st) {
  const uint32_t Cp = pad4(g.C), N = g.B * g.H * g.W;
  if (!operand_fits(size_t(g.B) * g.C * g.H * g.W, "conv_forward")) return false;
  TileCfg cfg = choose(
      "DCE_TUNE_FWD", g.OC, N, Cp, 8, true,
      [&](const TileCfg& t) { return tiles_occ16(t, FwdPwRun{}); }, true);
  narrow_pw(cfg, "DCE_TUNE_FWD", g.OC, Cp);
  // Filters [OC][C] are already the A operand when C % 4 == 0 (16-byte rows).
  const bool wDirect = g.C % 4 == 0 && aligned16(w);
  const size_t nw = wDirect ? 0 : al64(size_t(g.OC) * Cp);
  const size_t nP = cfg.splits > 1 ? size_t(cfg.splits) * g.OC * N : 0;
  float* ws = (nw + nP) ? workspace(nw + nP) : nullptr;
  if ((nw + nP) && !ws) return false;
  if (!wDirect && !permute_w(WPerm{w, ws, g.OC, g.C, 1, Cp, Cp, 0, 0})) return false;
  ProfScope prof("conv_fwd", 2.0 * g.OC * g.C * double(N),
                 4.0 * (double(g.B) * g.C * g.H * g.W + double(g.B) * g.OC * g.OH * g.OW));
  double* stats = stats_buffer(st, cfg, N, act, true);
  return tiles_dispatch16(cfg, FwdPwRun{wDirect ? w : ws, x, bias, y, ws ? ws + nw : nullptr, g,
                                        act, cfg.splits, stats, st ? st->pieces : 0});
}

bool conv_forward(const float* x, float* x_nhwc_keep, const float* w, const float* bias,
                  float* y, const ConvGeom& g, uint32_t act, ConvStatsReq* st) {
  if (st) st->pieces = 0;
  if (pw_x(g)) return conv_forward_pw(x, w, bias, y, g, act, st);
  if (ps_x(g)) return conv_forward_ps(x, x_nhwc_keep, w, bias, y, g, act);
  const bool pk = packed_x(g);
  const uint32_t Cp = pad4(g.C), KK = g.k * g.k, kdim = pk ? pad4(KK * g.C) : KK * Cp;
  const bool blk = !pk && blocked_k(Cp), s1 = g.s == 1;
  const size_t nx = xcopy_floats(g);
  const uint32_t N = g.B * g.OH * g.OW;
  if (!operand_fits(nx, "conv_forward") || !operand_fits(size_t(g.OC) * kdim, "conv_forward"))
    return false;
  TileCfg cfg = choose(
      "DCE_TUNE_FWD", g.OC, N, kdim, 8, true,
      [&](const TileCfg& t) {
        return pk ? tiles_occ16(t, FwdPkRun{}) : conv_variant_occ<FwdRun>(s1, blk, t);
      },
      true);
  if (!pk) narrow_short_k(cfg, "DCE_TUNE_FWD", g.OC, N, kdim);
  const size_t nw = al64(size_t(g.OC) * kdim);
  const size_t nxs = x_nhwc_keep ? 0 : al64(nx);
  const size_t nP = cfg.splits > 1 ? size_t(cfg.splits) * g.OC * N : 0;
  float* ws = workspace(nw + nxs + nP);
  if (!ws) return false;
  float* wp = ws;
  float* xn = x_nhwc_keep ? x_nhwc_keep : ws + nw;
  float* part = ws + nw + nxs;
  // The filter re-layout rides in the NHWC copy's launch.
  const WPerm fwdPerm{w, wp, g.OC, g.C, KK, pk ? g.C : Cp, kdim, 0, blk ? 1 : 0};
  if (pk ? !(to_pk(x, xn, g) && permute_w(fwdPerm))
         : !to_nhwc_masked(x, nullptr, xn, nullptr, g.B, g.C, g.H * g.W, nullptr, fwdPerm))
    return false;
  const double fl = 2.0 * g.OC * g.C * KK * double(g.B) * g.OH * g.OW;
  {
    ProfScope prof("conv_fwd", fl,
                   4.0 * (double(g.B) * g.C * g.H * g.W + double(g.B) * g.OC * g.OH * g.OW));
    double* stats = stats_buffer(st, cfg, N, act, !pk && s1);
    const bool ok =
        pk ? tiles_dispatch16(cfg, FwdPkRun{wp, xn, bias, y, part, g, act, cfg.splits})
           : conv_variant<FwdRun>(s1, blk, cfg, wp, xn, bias, y, part, g, act, cfg.splits,
                                  stats, st ? st->pieces : 0u);
    if (!ok) return false;
  }
  return true;
}

// ----------------------------------------------------------- conv backward
// Fraction of an M x N tile grid's area that is real output.
static double tile_fill(uint32_t M, uint32_t N) {
  const double mt = pick_tile_m(M), nt = pick_tile(N);
  return double(M) * N / (std::ceil(M / mt) * mt * std::ceil(N / nt) * nt);
}

// filters re-laid [c][pad4(OC)]).
// WK: the A operand is the filters themselves, [OC][C] read as [k = oc][row
// = c] (C % 4 == 0); otherwise their re-layout [C][pad4(OC)].
template <bool WK>
struct DxPwRun {
  const float* wt;
  const float* dy;
  float* dx;
  float* part;
  ConvGeom g;
  uint32_t splits;
  template <int MT, int KT>
  using LAt = typename std::conditional<WK, LdDenseKR<MT, KT>, LdDenseRK<MT, KT>>::type;
  template <int MT, int NT, int KT>
  int occ(bool split) const {
    using LA = LAt<MT, KT>;
    using LB = LdNchwKR<NT, KT>;
    return split ? occupancy(k_igemm<MT, NT, KT, LA, LB, EpiRowMajor>)
                 : occupancy(k_igemm<MT, NT, KT, LA, LB, EpiNCHW>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    const uint32_t OCp = pad4(g.OC), HW = g.H * g.W, N = g.B * HW;
    using LA = LAt<MT, KT>;
    using LB = LdNchwKR<NT, KT>;
    const typename LA::Params pa = WK ? typename LA::Params{wt, g.C, g.C, g.OC, g.OC * g.C}
                                      : typename LA::Params{wt, OCp, g.C, OCp, g.C * OCp};
    const NchwKRParams pb{dy, g.OC, HW, N, g.B * g.OC * HW, make_fastdiv(HW)};
    const uint32_t kt = cdiv(OCp, KT);
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

// Pointwise dW: dw[oc][c] = sum_n dy[oc][n] x[c][n]; with db, x gets a row of
// ones (column C of the product is the bias gradient, written by the finish).
struct DwPwRun {
  const float* dy;
  const float* x;
  float* part;
  ConvGeom g;
  uint32_t N, splits;  // N = C, or C + 1 with the ones row
  bool trans;          // input channels as the product's rows (partials [z][c][oc])
  template <int MT, int NT, int KT>
  int occ(bool) const {
    return occupancy(k_igemm<MT, NT, KT, LdNchwRK<MT, KT>, LdNchwRK<NT, KT>, EpiRowMajor>);
  }
  template <int MT, int NT, int KT>
  bool run() {
    const uint32_t HW = g.H * g.W, K = g.B * HW;
    const NchwRKParams pa{dy, ones4(), g.OC, HW, K, g.B * g.OC * HW, 0xFFFFFFFFu, make_fastdiv(HW)};
    const NchwRKParams pb{x, ones4(), g.C, HW, K, g.B * g.C * HW, N > g.C ? g.C : 0xFFFFFFFFu,
                          make_fastdiv(HW)};
    const uint32_t zs = 4 * cdiv(size_t(g.OC) * N, 4);
    if (trans) {
      const EpiRowMajor::Params pe{part, N, g.OC, g.OC, zs};
      return launch<MT, NT, KT, LdNchwRK<MT, KT>, LdNchwRK<NT, KT>, EpiRowMajor>(
          pb, pa, pe, N, g.OC, cdiv(K, KT), splits, "conv_backward_filter");
    }
    const EpiRowMajor::Params pe{part, g.OC, N, N, zs};
    return launch<MT, NT, KT, LdNchwRK<MT, KT>, LdNchwRK<NT, KT>, EpiRowMajor>(
        pa, pb, pe, g.OC, N, cdiv(K, KT), splits, "conv_backward_filter");
  }
};

static bool conv_backward_pw(const float* dy, const float* x, const float* w, float* dw,
                             float* db, float* dx, const ConvGeom& g) {
  const uint32_t OCp = pad4(g.OC), HW = g.H * g.W, N = g.B * HW;
  const double fl = 2.0 * g.OC * g.C * double(N);
  ProfScope profAll("conv_bwd", fl * ((dw ? 1 : 0) + (dx ? 1 : 0)), 0.0);
  const uint32_t Ndw = g.C + (db ? 1u : 0u);
  TileCfg dwc{128, 128, 16, 1}, dxc{128, 128, 16, 1};
  size_t nP = 0, nW = 0, nQ = 0;
  // dW orientation with the fuller tile grid: expand layers (many more
  // output than input channels) put the few input channels on the narrow
  // rows.
  const bool dwT = tile_fill(Ndw, g.OC) > tile_fill(g.OC, Ndw) * 1.25;
  if (dw) {
    const uint32_t dM = dwT ? Ndw : g.OC, dN = dwT ? g.OC : Ndw;
    const uint32_t ntiles = cdiv(dM, pick_tile_m(dM)) * cdiv(dN, pick_tile(dN));
    dwc = choose(
        "DCE_TUNE_DW", dM, dN, N, ntiles <= 4 ? 1024 : 256, false,
        [&](const TileCfg& t) { return tiles_occ(t, DwPwRun{}); }, false, true);
    nP = al64(size_t(dwc.splits) * 4 * cdiv(size_t(g.OC) * Ndw, 4));
  }
  const bool wk = g.C % 4 == 0 && aligned16(w);  // dX reads the filters in place
  if (dx) {
    dxc = choose(
        "DCE_TUNE_DX", g.C, N, OCp, 8, true,
        [&](const TileCfg& t) {
          return wk ? tiles_occ16(t, DxPwRun<true>{}) : tiles_occ16(t, DxPwRun<false>{});
        },
        true);
    narrow_pw(dxc, "DCE_TUNE_DX", g.C, OCp);
    nW = wk ? 0 : al64(size_t(g.C) * OCp);
    nQ = dxc.splits > 1 ? size_t(dxc.splits) * g.C * N : 0;
  }
  float* ws = (nP + nW + nQ) ? workspace(nP + nW + nQ) : nullptr;
  if ((nP + nW + nQ) && !ws) return false;
  float* part = ws;
  float* wt = ws ? ws + nP : nullptr;
  float* qpart = wt ? wt + nW : nullptr;
  if (dw) {
    ProfScope prof("conv_dw", fl, 4.0 * (double(N) * g.OC + double(N) * g.C));
    if (!tiles_dispatch(dwc, DwPwRun{dy, x, part, g, Ndw, dwc.splits, dwT}) ||
        !dw_final(part, dw, g.OC, g.C, 1, Ndw, dwc.splits, dwT, BwdSide{}, db))
      return false;
  }
  if (dx) {
    if (!wk && !permute_w(WPerm{w, wt, g.OC, g.C, 1, OCp, OCp, 1, 0})) return false;
    ProfScope prof("conv_dx", fl, 4.0 * (double(N) * g.OC + double(N) * g.C));
    const bool ok = wk ? tiles_dispatch16(dxc, DxPwRun<true>{w, dy, dx, qpart, g, dxc.splits})
                       : tiles_dispatch16(dxc, DxPwRun<false>{wt, dy, dx, qpart, g, dxc.splits});
    if (!ok) return false;
  }
  return true;
}

uint32_t conv_g_layout(const ConvGeom& g) {
  return ps_x(g) ? kGLayoutPad : conv_parts(g) ? kGLayoutParts : kGLayoutNhwc;
}
bool conv_g_nhwc_pass(const ConvGeom& g) { return !ps_x(g) && !pw_x(g); }
uint32_t conv_g_pad_width(const ConvGeom& g) { return ps_geom(g).OWp; }

bool conv_backward(const float* dy, const float* y, const float* x, const float* x_nhwc,
                   const float* w, float* dw, float* db, float* dx, const ConvGeom& g,
                   const PreG* pre) {
  // Pointwise layers with no ReLU mask (and dW requested whenever db is: the
  // bias gradient is the dW product's ones column) read NCHW in place.
  if (pw_x(g)) {
    if (!y && (dw || !db)) {
      if (!operand_fits(size_t(g.B) * g.C * g.H * g.W, "conv_backward") ||
          !operand_fits(size_t(g.B) * g.OC * g.H * g.W, "conv_backward"))
        return false;
      return conv_backward_pw(dy, x, w, dw, db, dx, g);
    }
    x_nhwc = nullptr;  // the forward kept no copy: the general path builds its own
  }
  // Parts: G, x and the dX filters as bf16 parts, channels padded to 16.
  const bool parts = conv_parts(g);
  const uint32_t Cp = parts ? pad16(g.C) : pad4(g.C), OCp = parts ? pad16(g.OC) : pad4(g.OC);
  const uint32_t KK = g.k * g.k;
  const uint32_t OHW = g.OH * g.OW, npix = g.B * OHW, HW = g.H * g.W;
  const size_t gFloats = parts ? parts_floats(npix, g.OC) : size_t(npix) * OCp;
  const size_t wFloats = parts ? parts_floats(size_t(g.C) * KK, g.OC) : size_t(g.C) * KK * OCp;
  if (!operand_fits(gFloats, "conv_backward") ||
      !operand_fits(xbuild_floats(g), "conv_backward") || !operand_fits(wFloats, "conv_backward"))
    return false;
  // Workspace carve-up: G (NHWC) and / or G_pad, db partials, the copy of x
  // if not kept by the forward, dW split-K partials, dX filters, dX split-K
  // partials.  Fewer than four input channels: x is stride-phase split (or,
  // for strides above 4, channel-packed) and the dW tap axis runs over KK * C
  // unpadded taps (Cx = C), otherwise over KK * pad4(C).
  const bool pk = packed_x(g), ps = ps_x(g);
  const uint32_t Cx = (pk || ps) ? g.C : Cp;
  const uint32_t npb = cdiv(OHW, 64);
  // The whole call as one family: the masked transpose of dy, the bias-grad
  // sum, any rebuilt copy of x, the filter re-layout and the split-K finishes
  // count with the GEMMs' FLOPs.
  const double callFlops = 2.0 * g.OC * g.C * KK * double(npix) * ((dw ? 1 : 0) + (dx ? 1 : 0));
  ProfScope profAll("conv_bwd", callFlops, 0.0);
  // The stride-phase dW reads the masked gradient on the padded pixel grid
  // (G_pad, which also yields the bias-gradient partials); dX reads the NHWC
  // G of the transpose pass.  Other layouts use the NHWC G for both.
  const PsGeom q = ps ? ps_geom(g) : PsGeom{};
  const bool useGpad = ps && (dw || (db && !dx)), useGnhwc = !ps || dx;
  // A G_pad made by dy's producer (with its bias-gradient partials) replaces
  // the masking pass that makes it.
  const bool preG = pre && pre->layout == kGLayoutPad && useGpad;
  // An NHWC G made by dy's producer (the batch-norm backward; no ReLU mask)
  // replaces the transpose pass.
  const bool preGn =
      pre && pre->layout == (parts ? kGLayoutParts : kGLayoutNhwc) && !ps && !y;
  const uint32_t nchunk = ps ? cdiv(q.OHWp, kMaskChunk) : 0;
  const uint32_t dbRows = useGpad ? g.B * nchunk : g.B * npb;
  const uint32_t dwK = ps ? g.B * q.OHWp : npix;  // dW GEMM K extent (pixels)
  const size_t nG = (useGnhwc && !preGn) ? al64(gFloats) : 0;
  const size_t nGp = (useGpad && !preG) ? al64(size_t(g.B) * g.OC * q.OHWp) : 0;
  const size_t nDb = (db && !preG && !preGn) ? al64(size_t(dbRows) * g.OC) : 0;
  const size_t nX = (dw && (parts || !x_nhwc)) ? al64(xbuild_floats(g)) : 0;
  if (ps && !operand_fits(nGp, "conv_backward")) return false;
  TileCfg dwc{128, 128, 16, 1};
  size_t nP = 0, nW = 0, nQ = 0;
  bool dwT = false;
  if (dw) {
    // Orientation with the fuller tile grid; a grid of a few tiles gets more
    // split-K slices so that the whole chip works on it.
    const uint32_t taps = KK * Cx;
    dwT = tile_fill(taps, g.OC) > tile_fill(g.OC, taps) * 1.25;
    const uint32_t dM = dwT ? taps : g.OC, dN = dwT ? g.OC : taps;
    dwc = conv_dw_choose(dM, dN, dwK, dwT, pk, ps, parts);
    nP = al64(size_t(dwc.splits) * 4 * cdiv(size_t(g.OC) * taps, 4));
  }
  DxPlan dxp{};
  if (dx) {
    dxp = conv_dx_plan(g, parts);
    nQ = dxp.part;
  }
  if (dx) nW = al64(wFloats);
  float* ws = workspace(nG + nGp + nDb + nX + nP + nW + nQ);
  if (!ws) return false;
  float* gn = ws;
  float* gp = gn + nG;
  float* dbPart = db ? gp + nGp : nullptr;
  float* xs = gp + nGp + nDb;
  float* part = xs + nX;
  float* wt = part + nP;
  float* qpart = wt + nW;
  if (preG) {
    gp = const_cast<float*>(pre->g);
    if (db) dbPart = const_cast<float*>(pre->db);
  }
  if (preGn) {
    gn = const_cast<float*>(pre->g);
    if (db) dbPart = const_cast<float*>(pre->db);
  }

  if (useGpad && !preG) {
    bool ok = false;
    mask_pad(dy, y, gp, dbPart, g, &ok);
    if (!ok) return false;
  }
  // The dX filter re-layout rides in the G pass launch (dX always has the
  // NHWC G), the bias-gradient sum in the dW finishing launch.
  const WPerm dxPerm{w, wt, g.OC, g.C, KK, OCp, KK * OCp, 1, dx && blocked_k(OCp) ? 1 : 0,
                     0, 0, 0, 0, 0, parts ? 1u : 0u};
  // On parts the kept copy of x is split in that launch too, or by itself.
  XSplit xsJob{};
  if (dw && parts && x_nhwc) {
    const uint32_t nblk = pad16(g.C) / 16;
    xsJob = XSplit{x_nhwc, xs, g.B * HW * 2 * nblk, nblk, pad4(g.C), make_fastdiv(2 * nblk)};
  }
  uint32_t npbGot = npb;
  if (useGnhwc && !preGn &&
      !to_nhwc_masked(dy, y, gn, useGpad ? nullptr : dbPart, g.B, g.OC, OHW, &npbGot,
                      dx && !dxp.phased ? dxPerm : WPerm{}, parts, xsJob))
    return false;
  if (preGn && xsJob.src && !xsplit(xsJob)) return false;
  // With the producer's G the dX filter re-layout rides in the dW finish
  // (which runs before dX), or runs by itself when no dW is asked for.
  const bool permInFinish = preGn && dx && !dxp.phased && dw;
  if (preGn && dx && !dxp.phased && !dw && !permute_w(dxPerm)) return false;
  const uint32_t dbRowsGot =
      (preG || preGn) ? pre->dbRows : (useGpad ? dbRows : g.B * npbGot);
  if (db && !dw) {
    hipLaunchKernelGGL(k_rowsum, dim3(g.OC), dim3(256), 0, stream(), dbPart, db, dbRowsGot);
    if (!check_launch("bias_grad")) return false;
  }
  auto dx_chain = [&]() {
    ProfScope prof("conv_dx", 2.0 * g.OC * g.C * KK * double(npix),
                   4.0 * (double(npix) * OCp + double(g.B) * g.C * g.H * g.W));
    return conv_dx(dxp, w, wt, gn, dx, qpart, g, parts);
  };
  auto dw_gemm = [&]() {
    const float* xn = xsJob.src ? xs : x_nhwc;
    if (!xn) {
      const bool built = ps ? to_ps(x, xs, g)
                         : pk ? to_pk(x, xs, g)
                              : to_nhwc_masked(x, nullptr, xs, nullptr, g.B, g.C, HW, nullptr,
                                               WPerm{}, parts);
      if (!built) return false;
      xn = xs;
    }
    ProfScope prof("conv_dw", 2.0 * g.OC * g.C * KK * double(npix),
                   4.0 * (double(npix) * OCp + double(g.B) * g.H * g.W * Cp + double(g.OC) * KK * Cp));
    return conv_dw_gemm(dwc, ps ? gp : gn, xn, part, g, dwT, pk, ps, parts);
  };
  auto dw_finish = [&]() {
    BwdSide side{};
    if (db) {
      side.dbPart = dbPart;
      side.db = db;
      side.dbRows = dbRowsGot;
      side.nRow = g.OC;
    }
    // The stride-phase taps are already in the filters' (c, kh, kw) order:
    // the finish is a plain split sum (one channel of C*KK taps).
    return ps ? dw_final(part, dw, g.OC, 1, KK * g.C, 1, dwc.splits, dwT, side)
              : dw_final(part, dw, g.OC, g.C, KK, Cx, dwc.splits, dwT, side, nullptr,
                         permInFinish ? dxPerm : WPerm{});
  };
  if (dw && !(dw_gemm() && dw_finish())) return false;
  if (dx && !dx_chain()) return false;
  return true;
}

}  // namespace dce
