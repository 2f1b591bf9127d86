// ss_gemm.h - block-quantized matrix x token-block products on MFMA (gfx950),
// for prompts: Y[t] = W X[t] over T tokens at once (layer_scheduler.c:681-803
// evaluates a prompt layer by layer; every token of a layer multiplies the
// same matrices).
//
// The products run on v_mfma_f32_32x32x16_f16 for every block format (Q4_0,
// Q8_0, Q4_1, Q5_1, Q8_1, the K-quants; Q5_0 as Q8_0): the codes are exact
// fp16 integers from a magic number (bits 0x6400 | u are 1024 + u; the
// subtraction of the offset is exact), x is split into two fp16 parts under a
// power-of-two scale per token and 256 columns (the largest |x s| in [2^13,
// 2^14), so xh + xl is within 2^-23 |x| of x), every block's fp32 result is
// scaled by its A into fp32 accumulators. The RMSNorm scale 1/rms of each
// token multiplies its outputs (tensor.c:114-131 applies it to x).
//
// Two kernels share the arithmetic. k_gemm_ks, for short prompts, splits the
// columns over the 8 waves of a workgroup and takes x straight into
// registers; k_gemm_rs, for longer ones, has several waves read the same x
// from LDS. pick_shape() chooses.
//
// MFMA operands: lane l supplies A[l%32][8(l/32) + i] (x: token l%32) and
// B[8(l/32) + i][l%32] (codes: row l%32), i = 0..7, and receives
// D[8(j/4) + 4(l/32) + j%4][l%32] (token, row) in register j = 0..15. Step h
// = 0, 1 of a block covers its columns 16h .. 16h + 15 (its two 16-weight
// groups); slot i of lane half kg is column 16h + 8kg + 4(i/4) + p(i%4), p =
// 0, 2, 1, 3: the order in which masking a code word gives fp16 pairs.
//
// K-quants other than Q6_K: weight = d * (sc * q) - dmin * m (Q3_K: d *
// (s - 32)(q - 4), no minimum) with sc * q an integer of at most 2048, exact
// in fp16. The codes are multiplied by their integer scale as fp16 pairs, a
// whole unit (one super-block) runs as one chain of MFMAs, and d multiplies
// its result once instead of every block's. The minima are one more MFMA per
// unit (m exact, the unit's sums of x in two fp16 parts), times dmin. Q4_1
// and Q5_1 take their minima the same way (m is an fp16).

#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>

#include "ss_device.h"
#include "ss_kernels.h"

namespace ssk {

// k_gemm_ks on matrices of one or two units (ss_gemm_few.hip), x split already.
hipError_t launch_gemm_few(int epi, const GemmArgs& a, int nu, hipStream_t s);

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// Every 32-weight block is sum_g (A_g * sum c x - B_g * sum x) over its two
// 16-weight groups g, c being the stored code (an exact fp16 integer) and A,
// B exact fp32:
//   Q4_0, Q8_0: A = d, B = 0 (Q4_0 codes are nibble - 8)
//   Q4_1, Q5_1: A = d, B = -m (nibbles; 5-bit codes as int8)
//   Q8_1:       A = fp32 d, B = 0
//   K-quants:   kq_affine (Q4_K and Q5_K one (A, B) pair per block; Q2_K,
//               Q3_K and Q6_K one per 16-weight group)
// kLay: the code layout (2: nibbles as Q4_0's, 8: int8 codes as Q8_0's).
template <int QT>
struct PQ {
  static constexpr int kLay = code_bytes_of(QT) == 16 ? 2 : 8;
};

// A of a block from its scale entry e (16 bits, or 32 for Q4_1 / Q5_1 / Q8_1)
template <int QT>
__device__ __forceinline__ float block_scale(uint32_t e) {
  static_assert(!is_kq(QT), "the K-quants' scales: kq_affine, int_scale");
  if constexpr (QT == kQ8_1) return __uint_as_float(e);
  return h2f((uint16_t)(e & 0xffffu));
}

// a * x + y
__device__ __forceinline__ v16f fma16(float a, v16f x, v16f y) { return __builtin_elementwise_fma(v16f(a), x, y); }

constexpr int kSW = 8;            // waves per workgroup
constexpr int kSUnit = 8;         // 32-column blocks of a unit (2 tiles, one super-block)
constexpr int kSTok = 32;         // tokens of a tile
constexpr float kSumScale = 1.0f / 32.0f;   // |x s_t| < 2^14, so a block's sum times this is below 2^14 too

// MFMA steps of a unit's minima (8 sums each): none, one per block, one per 16-weight group
template <int QT>
constexpr int sum_steps() {
  return QT == kQ2K ? 2 : QT == kQ4_1 || QT == kQ5_1 || QT == kQ4K || QT == kQ5K ? 1 : 0;
}
// the integer scale is multiplied into the codes
template <int QT>
constexpr bool folded() { return QT == kQ2K || QT == kQ3K || QT == kQ4K || QT == kQ5K; }

__host__ __device__ constexpr int slot_col_ks(int i) {   // column of slot i (i < 8) within a lane half's 8
  return 4 * (i >> 2) + ((i & 1) << 1 | ((i >> 1) & 1));
}

// The split x of ntile token tiles and nu units: the fragments, then per
// (tile, unit) of 32 tokens the inverse scales, the sums of squares, and the
// block sums' fragments.
struct KsView {
  uint4* x;        // fragment (tile, block, step, part): 64 chunks of 16 bytes
  float* inv;      // [tile][unit][32]
  float* ssq;      // [tile][unit][32]
  uint4* sum;      // fragment (tile, unit, step): 64 chunks
};
__host__ __device__ inline KsView ks_view(uint16_t* xs, int ntile, int nu) {
  KsView v;
  v.x = reinterpret_cast<uint4*>(xs);
  v.inv = reinterpret_cast<float*>(v.x + (size_t)ntile * nu * kSUnit * 4 * 64);
  v.ssq = v.inv + (size_t)ntile * nu * kSTok;
  v.sum = reinterpret_cast<uint4*>(v.ssq + (size_t)ntile * nu * kSTok);
  return v;
}

// One wave: 8 tokens (lane % 8) x the 8 blocks (lane / 8) of unit blockIdx.y
// of x (times nw). The unit's inverse scale 1/s per token (the largest |x s|
// of the unit lies in [2^13, 2^14)) and its sum of squares of x, then x s as
// two fp16 parts in fragment order: part p of step h of block b is the 1 KB
// fragment 2h + p of (tile, b), lane half kg and token t%32 at chunk 32 kg +
// t%32. So 8 lanes write 128 contiguous bytes, and no reduction leaves the
// wave. Blocks past the row are zero; tokens past T are not written (nor
// used). SUMS: also the sums of each block (1) or 16-column group (2), times
// kSumScale, as two fp16 parts: fragment (tile, unit, step), part and token
// as kg and token above, 8 sums each.
template <int SUMS>
__global__ void __launch_bounds__(64) k_split_ks(const float* __restrict__ x, int ldx, const float* __restrict__ nw,
                                                 int T, int nb, KsView o) {
  const int lane = threadIdx.x, b = lane >> 3;
  const int t = blockIdx.x * 8 + (lane & 7), unit = blockIdx.y, nu = gridDim.y;
  const int blk = unit * kSUnit + b, tile = t / kSTok, tok = t % kSTok;
  const bool in = t < T && blk < nb;
  float u[32], ss = 0.f, mx = 0.f;
  {
    const float4* xq = reinterpret_cast<const float4*>(x + (size_t)min(t, T - 1) * ldx + 32 * min(blk, nb - 1));
    const float4* wq = nw ? reinterpret_cast<const float4*>(nw + 32 * min(blk, nb - 1)) : xq;
    float4 xv[8], wv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) xv[i] = xq[i];
#pragma unroll
    for (int i = 0; i < 8; ++i) wv[i] = wq[i];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
      const float w[4] = {wv[i].x, wv[i].y, wv[i].z, wv[i].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float v = in ? a[k] : 0.f;
        ss = fmaf(v, v, ss);
        u[4 * i + k] = nw ? v * w[k] : v;
        mx = fmaxf(mx, fabsf(u[4 * i + k]));
      }
    }
  }
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) {
    ss += __shfl_xor(ss, off, kWave);
    mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
  }
  int e = 0;
  if (mx > 0.f && mx <= 3.0e38f) frexpf(mx, &e);        // mx < 2^e
  e = max(e, -100);                                     // (2^(14 - e) stays finite)
  const float sc = ldexpf(1.0f, 14 - e);                // largest |x s| in [2^13, 2^14)
  if (t >= T) return;
  const size_t at = (size_t)tile * nu + unit;
  if (b == 0) {
    o.inv[at * kSTok + tok] = ldexpf(1.0f, e - 14);
    o.ssq[at * kSTok + tok] = ss;
  }
  uint4* q = o.x + (at * kSUnit + b) * 4 * kWave + tok;
  float sum[2] = {0.f, 0.f};
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int kg = 0; kg < 2; ++kg) {
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float v0 = u[16 * h + 8 * kg + slot_col_ks(2 * k)] * sc;
        const float v1 = u[16 * h + 8 * kg + slot_col_ks(2 * k + 1)] * sc;
        const _Float16 p = (_Float16)v0, r = (_Float16)v1;
        const _Float16 lp = (_Float16)(v0 - (float)p), lr = (_Float16)(v1 - (float)r);
        hi[k] = __builtin_bit_cast(uint32_t, h2{p, r});
        lo[k] = __builtin_bit_cast(uint32_t, h2{lp, lr});
        if constexpr (SUMS > 0) sum[SUMS == 2 ? h : 0] += ((float)p + (float)lp) + ((float)r + (float)lr);
      }
      q[(2 * h) * kWave + 32 * kg] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
      q[(2 * h + 1) * kWave + 32 * kg] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
#pragma unroll
  for (int g = 0; g < SUMS; ++g) {
    const int i = SUMS * b + g;   // sum i of the unit
    const float v = sum[g] * kSumScale;
    const _Float16 p = (_Float16)v;
    const _Float16 r = (_Float16)(v - (float)p);
    uint16_t* z = reinterpret_cast<uint16_t*>(o.sum + (at * SUMS + i / 8) * kWave + tok) + i % 8;
    z[0] = __builtin_bit_cast(uint16_t, p);
    z[32 * 8] = __builtin_bit_cast(uint16_t, r);
  }
}

// A lane's 8 codes of step h of a block as exact fp16 values in slot order.
// Nibble layout: words 2kg and 2kg+1 of the block's chunk serve both steps
// (low nibbles, then high). int8 layout: words 4h + 2kg and + 1.
// magic: 0x64006400 in a vector register, so that mask and or are one
// instruction (it takes one constant beside its registers).
template <int QT>
__device__ __forceinline__ v8h codes_ks(uint2 w, int h, uint32_t magic) {
  v4u r;
  const uint32_t q[2] = {w.x, w.y};
  if constexpr (PQ<QT>::kLay == 2) {
    // Q4_0: nibble - 8; Q3_K: its code + 4 - 4; the others' nibble as it is
    constexpr float kOff = QT == 2 ? -1032.0f : QT == kQ3K ? -1028.0f : -1024.0f;
    const h2 off = {(_Float16)kOff, (_Float16)kOff};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      r[k] = __builtin_bit_cast(
          uint32_t, __builtin_bit_cast(h2, ((q[k >> 1] >> (8 * (k & 1) + 4 * h)) & 0x000F000Fu) | magic) + off);
  } else {
    const h2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // bytes 0, 2 (k even) or 1, 3 of the word, each below a 0x64
      const uint32_t u = q[k >> 1] ^ 0x80808080u;
      r[k] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, __builtin_amdgcn_perm(magic, u, k & 1 ? 0x05030501u : 0x05020500u)) + off);
    }
  }
  return __builtin_bit_cast(v8h, r);
}
// times an integer scale (the products are integers of at most 2048: exact)
__device__ __forceinline__ v8h times(v8h c, int sc) {
  const h2 s = {(_Float16)sc, (_Float16)sc};
  v4u r = __builtin_bit_cast(v4u, c);
#pragma unroll
  for (int k = 0; k < 4; ++k) r[k] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, (uint32_t)r[k]) * s);
  return __builtin_bit_cast(v8h, r);
}
// the integer scale of 16-weight group h from a block's scale entry (kq_affine)
template <int QT>
__device__ __forceinline__ int int_scale(uint32_t e, int h) {
  if constexpr (QT == kQ2K) return (int)((e >> (8 * h)) & 15u);
  if constexpr (QT == kQ3K) return (int)((e >> (8 * h)) & 0xffu) - 32;
  return (int)(e & 0xffu);
}

// One unit's codes and scale entries of one 32-row tile: lane (row n = l%32,
// half kg).
template <int QT>
struct KCodes {
  static constexpr int kQ = PQ<QT>::kLay == 2 ? 1 : 2;
  uint2 q[kSUnit][kQ];
};
template <int QT>
struct KScale {
  static constexpr int kE = is_wide(QT) ? kSUnit : kSUnit / 2;
  uint32_t e[kE];   // entries of (block b, both tiles)
  uint32_t su;      // K-quants: the unit is one super-block
  __device__ __forceinline__ uint32_t entry(int k) const {
    if constexpr (is_wide(QT)) return e[k];
    return k / kTB ? e[k % kTB] >> 16 : e[k % kTB] & 0xffffu;
  }
};

// The planes of one 32-row tile (row groups gb and gb + 1 of the matrix) as
// buffer views: a lane's offset is loop-invariant, the tile and unit a scalar.
template <int QT>
struct KView {
  static constexpr int kQB = QTraits<QT>::kQB, kEB = is_wide(QT) ? 4 : 2;
  __amdgpu_buffer_rsrc_t q, e, su;
  uint32_t qo, eo, so;
  int ntk;
  __device__ __forceinline__ void init(const PackedMat& w, int gb, int ngroups, int ntk_, int n, int kg) {
    ntk = ntk_;
    gb = min(gb, ngroups - 1);
    const int g = min(n / kRG, ngroups - 1 - gb);   // a missing second group: the first again, not stored
    const uint32_t qg = (uint32_t)ntk * kWave * kQB;
    const uint32_t eg = (uint32_t)((ntk + kUT - 1) / kUT) * kWave * kUT * kEB;
    const uint32_t sg = (uint32_t)(ntk / 2) * kRG * 4;
    q = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(w.qs) + (size_t)gb * qg, (short)0, (int)(2 * qg), kBufferFlags);
    e = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(w.ds)) + (size_t)gb * eg, (short)0, (int)(2 * eg), kBufferFlags);
    if constexpr (is_kq(QT))
      su = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(w.su)) + (size_t)gb * sg, (short)0, (int)(2 * sg), kBufferFlags);
    qo = g * qg + (n % kRG) * kQB + 8 * kg;
    eo = g * eg + (n % kRG) * kUT * kEB;
    so = g * sg + (n % kRG) * 4;
  }
};

typedef unsigned int v2u __attribute__((ext_vector_type(2)));

// tile h (blocks 4h .. 4h + 3) of unit u, or with h = -1 both
template <int QT>
__device__ __forceinline__ void load_codes(KCodes<QT>& f, const KView<QT>& w, int u, int h) {
  constexpr int kQB = KView<QT>::kQB;
#pragma unroll
  for (int k = 0; k < kSUnit; ++k) {
    if (h >= 0 && k / kTB != h) continue;
    // a tile past the row (the last unit's) reloads the last one: its x is zero
    const int t = min(2 * u + k / kTB, w.ntk - 1);
#pragma unroll
    for (int i = 0; i < KCodes<QT>::kQ; ++i) {
      const v2u v = __builtin_amdgcn_raw_buffer_load_b64(w.q, w.qo + (k % kTB) * kRG * kQB + 16 * i, t * kWave * kQB, 0);
      f.q[k][i] = make_uint2(v.x, v.y);
    }
  }
}
template <int QT>
__device__ __forceinline__ void load_scales(KScale<QT>& f, const KView<QT>& w, int u) {
  constexpr int kEB = KView<QT>::kEB;
  const int es = ((2 * u / kUT) * kWave * kUT + 2 * u % kUT) * kEB;
#pragma unroll
  for (int b = 0; b < kTB; ++b) {
    if constexpr (is_wide(QT)) {
      const v2u v = __builtin_amdgcn_raw_buffer_load_b64(w.e, w.eo + b * kRG * kUT * kEB, es, 0);
      f.e[b] = v.x;
      f.e[kTB + b] = v.y;
    } else {
      f.e[b] = __builtin_amdgcn_raw_buffer_load_b32(w.e, w.eo + b * kRG * kUT * kEB, es, 0);
    }
  }
  f.su = 0u;
  if constexpr (is_kq(QT)) f.su = __builtin_amdgcn_raw_buffer_load_b32(w.su, w.so, u * kRG * 4, 0);
}

// The minima of a unit as an MFMA operand: sum i of the unit times its m, in
// both lane halves (the sums' two parts).
template <int QT, int S>
__device__ __forceinline__ void unit_minima(const KScale<QT>& w, v8h (&mv)[S]) {
#pragma unroll
  for (int s = 0; s < sum_steps<QT>(); ++s)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t e = w.entry(QT == kQ2K ? (8 * s + j) / 2 : j);
      if constexpr (QT == kQ2K)
        mv[s][j] = (_Float16)(int)((e >> (8 * (j & 1) + 4)) & 15u);
      else if constexpr (is_wide(QT))
        mv[s][j] = __builtin_bit_cast(_Float16, (uint16_t)(e >> 16));
      else
        mv[s][j] = (_Float16)(int)(e >> 8);
    }
}
// acc += (part * d + mins * f) / s for the 16 tokens of a lane half, whose
// inverse scales are inv[8 (j/4) + j%4]
template <int QT>
__device__ __forceinline__ void unit_scale(v16f& acc, const v16f& part, const v16f& mins, float d, float f,
                                           const float* inv, bool live) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 s4 = *reinterpret_cast<const float4*>(inv + 8 * q);
    const float s[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int j = 4 * q + c;
      float v = part[j];
      if constexpr (folded<QT>()) v *= d;
      if constexpr (sum_steps<QT>() > 0) v = fmaf(f, mins[j], v);
      if (live) acc[j] = fmaf(s[c], v, acc[j]);
    }
  }
}

// One wave's products of a 32-row tile with TT token tiles, block by block.
// A block is 4 TT MFMAs; the matrix core takes 32 cycles for each, in which
// the wave can issue 8 other vector instructions, so what a block needs
// besides is put between them: the codes of the next block, the scaling of
// the first token tiles' products while the last one's run, and the scaling
// of the last one's of the block before.
template <int QT, int TT>
struct Pipe {
  v16f part[TT];   // the unit's sums, to be scaled by 1/s (and d)
  v8h c0, c1;      // codes of the block to come
  v16f p;          // the last token tile's product of the block before, not yet scaled
  float A;         // and its scale
  uint32_t magic;

  static constexpr bool kDelay = !folded<QT>() && QT != kQ6K;   // p and A are used
  __device__ __forceinline__ void codes(const KCodes<QT>& q, const KScale<QT>& w, int blk, v8h& n0, v8h& n1) const {
    n0 = codes_ks<QT>(q.q[blk][0], 0, magic);
    n1 = codes_ks<QT>(q.q[blk][KCodes<QT>::kQ - 1], 1, magic);
    if constexpr (folded<QT>()) {
      n0 = times(n0, int_scale<QT>(w.entry(blk), 0));
      n1 = times(n1, int_scale<QT>(w.entry(blk), 1));
    }
  }
  __device__ __forceinline__ void init(const KCodes<QT>& q, const KScale<QT>& w) {
    magic = 0x64006400u;
    asm("" : "+v"(magic));
    codes(q, w, 0, c0, c1);
  }
  // block BLK of the unit with scales w and x fragments x; wc: the unit's
  // codes, qn, wn: codes and scales of the unit after it
  template <int BLK>
  __device__ __forceinline__ void block(const KCodes<QT>& wc, const KScale<QT>& w, const KCodes<QT>& qn, const KScale<QT>& wn,
                                        const v8h (&x)[TT][4]) {
    v8h n0, n1;
    if constexpr (BLK + 1 < kSUnit)
      codes(wc, w, BLK + 1, n0, n1);
    else
      codes(qn, wn, 0, n0, n1);
    if constexpr (QT == kQ6K) {   // one scale per 16-weight group
      float S[2], Z[2];
      kq_affine<QT>(w.entry(BLK), w.su, S, Z);
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        v16f q = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt][0], c0, v16f{}, 0, 0, 0);
        v16f r = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt][2], c1, v16f{}, 0, 0, 0);
        q = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt][1], c0, q, 0, 0, 0);
        r = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt][3], c1, r, 0, 0, 0);
        part[tt] = fma16(S[1], r, BLK > 0 ? fma16(S[0], q, part[tt]) : q * S[0]);
      }
    } else {
      v16f q[TT];
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        q[tt] = folded<QT>() && BLK > 0 ? part[tt] : v16f{};
        q[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt][0], c0, q[tt], 0, 0, 0);
        q[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt][1], c0, q[tt], 0, 0, 0);
        q[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt][2], c1, q[tt], 0, 0, 0);
        q[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt][3], c1, q[tt], 0, 0, 0);
      }
      if constexpr (folded<QT>()) {
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) part[tt] = q[tt];
      } else {
        if constexpr (BLK > 0) add_last<BLK>();
        const float S = block_scale<QT>(w.entry(BLK));
#pragma unroll
        for (int tt = 0; tt + 1 < TT; ++tt) part[tt] = BLK > 0 ? fma16(S, q[tt], part[tt]) : q[tt] * S;
        p = q[TT - 1];
        A = S;
      }
    }
    c0 = n0;
    c1 = n1;
    constexpr int kValu = (24 + (folded<QT>() ? 10 : QT == kQ6K ? 32 * TT : 16 * TT)) / (4 * TT);
#pragma unroll
    for (int i = 0; i < 4 * TT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // an MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);   // then vector instructions
    }
    // the sums stay where they are: the compiler would otherwise put off the
    // scaling of several blocks
    if constexpr (!folded<QT>()) {
      if constexpr (TT == 2 && (BLK > 0 || QT == kQ6K))
        asm volatile("" : "+v"(part[0]), "+v"(part[TT - 1]));
      else if constexpr (TT == 2 || BLK > 0 || QT == kQ6K)
        asm volatile("" : "+v"(part[0]));
      if constexpr (kDelay) asm volatile("" : "+v"(p));
    }
  }
  template <int BLK>
  __device__ __forceinline__ void add_last() {   // block BLK - 1's last product
    part[TT - 1] = BLK > 1 ? fma16(A, p, part[TT - 1]) : p * A;
  }
  // The unit is done: acc += its sums, scaled, with its minima. sum: the
  // fragments of its block sums; inv: the inverse scales of the lane half's
  // tokens, 8 (j/4) + j%4 for register j of token tile 0, stride ld per tile.
  template <int S>
  __device__ __forceinline__ void finish(v16f (&acc)[TT], const KScale<QT>& w, const v8h (&sum)[S][TT], const float* inv,
                                         int ld, bool live) {
    if constexpr (kDelay) add_last<kSUnit>();
    const float d = folded<QT>() ? h2f((uint16_t)(w.su & 0xffffu)) : 1.f, dm = h2f((uint16_t)(w.su >> 16));
    v8h mv[S];
    unit_minima<QT>(w, mv);
    const float fm = is_wide(QT) ? 32.0f : -32.0f * dm;   // Q4_1, Q5_1: + m
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      v16f r = v16f{};
#pragma unroll
      for (int s = 0; s < sum_steps<QT>(); ++s) r = __builtin_amdgcn_mfma_f32_32x32x16_f16(sum[s][tt], mv[s], r, 0, 0, 0);
      unit_scale<QT>(acc[tt], part[tt], r, d, fm, inv + tt * ld, live);
    }
  }
};

// Codes of one unit, and the fragments of its block sums.
template <int QT, int TT>
struct KWork {
  KCodes<QT> q;
  KScale<QT> w;
  v8h sum[sum_steps<QT>() > 0 ? sum_steps<QT>() : 1][TT];
};

// ---- short prompts: the columns split over the waves ------------------------
// A workgroup of 8 waves owns 32 rows x 32 tokens (NMAT 2: of both matrices,
// the first half of the waves taking w (gate), the second w2 (up)); wave w
// takes the units w, w + 8, ... (w + 4). A wave shares nothing with another
// until the end: no barrier and no LDS in the loop, x and codes straight into
// registers. At the end the partial sums of every output are added in LDS in
// wave order. What bounds it at these sizes is the latency of the chain codes
// -> x -> products -> sum, not a rate: a 4096 x 4096 Q4_0 matrix takes 10 us
// per round of workgroups (32 to 64 tokens: 14.4 and 15.9 us with the split,
// 46.4 us with the 64-row workgroups that staged x in LDS for every matrix
// before; Q4_K at 77 tokens 58 -> 26.5 us).
constexpr int kKsUnits = 128;   // units whose inverse scales go through LDS; past them, from memory

template <int QT, int NMAT, int EPI, int KW>
__global__ void __launch_bounds__(KW * 64, 2) k_gemm_ks(const GemmArgs a, int nu) {
  constexpr int SUMS = sum_steps<QT>();
  constexpr int KS = KW / NMAT;   // column slices
  constexpr int kThreads = KW * 64, kPer = 1024 / kThreads;   // outputs of a tile per thread
  __shared__ float red[KW][16][kWave];
  __shared__ float rn[kThreads];
  constexpr int kUnits = KW < kSW ? KS : kKsUnits;
  __shared__ float inv_lds[kUnits * kSTok];   // [nu][32]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slice = wave % KS;
  const int n = lane & 31, kg = lane >> 5;
  const int ntk = ((a.cols >> 5) + kTB - 1) / kTB;
  const int ngroups = (a.rows + kRG - 1) / kRG;
  const int row0 = blockIdx.x * 32;
  const int tile = blockIdx.y, ntile = (a.T + kSTok - 1) / kSTok;
  const KsView xs = ks_view(a.xs, ntile, nu);

  KView<QT> wv;
  wv.init(NMAT == 2 && wave >= KS ? a.w2 : a.w, row0 / kRG, ngroups, ntk, n, kg);

  // this workgroup's token tile as buffer views: a lane whose token is past T
  // has an offset past the view and reads zero without touching memory
  const size_t at = (size_t)tile * nu;
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc(xs.x + at * kSUnit * 4 * kWave, (short)0, nu * kSUnit * 4096, kBufferFlags);
  __amdgpu_buffer_rsrc_t sr;
  if constexpr (SUMS > 0) sr = __builtin_amdgcn_make_buffer_rsrc(xs.sum + at * SUMS * kWave, (short)0, nu * SUMS * 1024, kBufferFlags);
  const uint32_t xo = tile * kSTok + n < a.T ? lane * 16u : 0x7fffff00u;
  struct Frags {
    v8h v[1][4];   // (step, part) fragments of one block
  };
  auto load_x = [&](Frags& f, int blk) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      f.v[0][i] = __builtin_bit_cast(v8h, __builtin_amdgcn_raw_buffer_load_b128(xr, xo + i * 1024, blk * 4096, 0));
  };
  // two units of codes, used in turn: each is refilled with the unit two
  // turns on as soon as it is used up
  KWork<QT, 1> wa, wb;
  auto load_w = [&](KWork<QT, 1>& f, int u) {
    u = min(u, nu - 1);   // past the end: reloaded, not used
    load_scales<QT>(f.w, wv, u);
    load_codes<QT>(f.q, wv, u, -1);
#pragma unroll
    for (int s = 0; s < SUMS; ++s)
      f.sum[s][0] = __builtin_bit_cast(v8h, __builtin_amdgcn_raw_buffer_load_b128(sr, xo, (u * SUMS + s) * 1024, 0));
  };
  v16f acc[1] = {v16f{}};
  Frags xa, xb;   // blocks of even and odd index
  const int u0 = min(slice, nu - 1);
  load_w(wa, u0);
  load_x(xa, u0 * kSUnit);
  load_x(xb, u0 * kSUnit + 1);
  load_w(wb, u0 + KS);
  // while those are in flight: the inverse scales into LDS, and each token's
  // sum of squares (thread: token tid % 32, units tid / 32, + KW * 2, ...)
  {
    float ss = 0.f;
    for (int i = tid; i < nu * kSTok; i += kThreads) {
      if (nu <= kUnits) inv_lds[i] = xs.inv[at * kSTok + i];
      ss += xs.ssq[at * kSTok + i];
    }
    rn[tid] = ss;
  }
  __syncthreads();
  Pipe<QT, 1> pipe;
  pipe.init(wa.q, wa.w);
  auto unit = [&](int u, KWork<QT, 1>& f, const KWork<QT, 1>& next) {
    const int un = min(u + KS, nu - 1);
    auto blocks = [&](auto kc) {   // blocks 2k and 2k + 1, then the x two on
      constexpr int k = 2 * decltype(kc)::value;
      pipe.template block<k>(f.q, f.w, next.q, next.w, xa.v);
      load_x(xa, k + 2 < kSUnit ? u * kSUnit + k + 2 : un * kSUnit);
      __builtin_amdgcn_sched_barrier(0);
      pipe.template block<k + 1>(f.q, f.w, next.q, next.w, xb.v);
      load_x(xb, k + 3 < kSUnit ? u * kSUnit + k + 3 : un * kSUnit + 1);
      __builtin_amdgcn_sched_barrier(0);
    };
    blocks(std::integral_constant<int, 0>{});
    blocks(std::integral_constant<int, 1>{});
    blocks(std::integral_constant<int, 2>{});
    blocks(std::integral_constant<int, 3>{});
    if (nu <= kUnits)
      pipe.finish(acc, f.w, f.sum, inv_lds + u * kSTok + 4 * kg, 0, true);
    else
      pipe.finish(acc, f.w, f.sum, xs.inv + (at + u) * kSTok + 4 * kg, 0, true);
    load_w(f, u + 2 * KS);
  };
  int u = slice;
#pragma unroll 1
  for (; u + KS < nu; u += 2 * KS) {   // (no branch inside: the compiler then counts the loads exactly)
    unit(u, wa, wb);
    unit(u + KS, wb, wa);
  }
  if (u < nu) unit(u, wa, wb);

  // the slices' partial sums, added in slice order: output tid + kThreads k of
  // the tile is register j = wave + KW k, lane `lane`
#pragma unroll
  for (int j = 0; j < 16; ++j) red[wave][j][lane] = acc[0][j];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int j = wave + KW * k;
    float v[NMAT];
#pragma unroll
    for (int m = 0; m < NMAT; ++m) {
      v[m] = 0.f;
#pragma unroll
      for (int q = 0; q < KS; ++q) v[m] += red[m * KS + q][j][lane];
    }
    const int tok = 8 * (j >> 2) + 4 * kg + (j & 3), t = tile * kSTok + tok, row = row0 + n;
    if (t >= a.T || row >= a.rows) continue;
    float scale = 1.f;   // the RMSNorm scale of tensor.c:114-131
    if (a.nw) {
      float ss = 0.f;
#pragma unroll
      for (int q = 0; q < 2 * KW; ++q) ss += rn[q * kSTok + tok];
      scale = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
    }
    float* yp = a.y + (size_t)t * a.ldy + row;
    const float y = v[0] * scale;
    if constexpr (EPI == EPI_SWIGLU)
      *yp = v[NMAT - 1] * scale * (a.act == 1 ? gelu_tanh(y) : silu(y));   // layer_scheduler.c:529-547
    else if constexpr (EPI == EPI_ADD)
      *yp += y;
    else
      *yp = y;
  }
}

// ---- longer prompts: x shared through LDS -----------------------------------
// The same products for more tokens. A workgroup of 8 waves owns RW row
// tiles (32 rows each; NMAT 2: RW / 2 of each matrix) x 64 tokens, its waves
// being KG = 8 / RW column groups of RW row tiles: column group g takes the
// units g, g + KG, .... The RW waves of a group read the same x, so it goes
// through LDS: 32 KB per stage for all groups (SB = RW / 2 blocks of each
// group's unit), by direct global-to-LDS loads, four stages in four arrays
// named at compile time, three of them in flight ahead of the one in use.
// One barrier per stage: past it every wave's loads of the next stage have
// landed, and every wave has the last of the stage before in registers, so
// that its array can be refilled. The counts of wait_loads hold only while the
// compiler issues the code loads counted beside the stages': one more waits
// for more, one fewer would let x be read before it is here. A test without a
// GPU reads the compiled loops for it (at most two stages in flight at a
// barrier). With RW 4 the compiler waits for everything once per unit besides,
// where the next unit's scales are first used: no counted wait comes between
// their load and that.
//
// Bound: the vector and matrix instructions of two waves per SIMD. A block of
// 8 waves takes 0.30 us with nothing but its LDS reads, MFMAs and vector
// instructions, 0.36 us with the whole chip busy (the clock drops), and about
// 0.45 us here; a round of workgroups adds the first loads and the last sum.
// 512 tokens, split included, against 64-row (128-row) workgroups of 16x16x32
// MFMAs with one tile of x ahead and a full drain per barrier: Q4_0 4096 x
// 4096 71.8 -> 49.7 us, 11008 x 4096 149 -> 124 us, 4096 x 11008 164 -> 117
// us; Q4_K 4096 x 4096 93 -> 53.5 us.
constexpr int kRsUnits = 112;   // columns / 256 at most (the inverse scales' share of LDS)

template <int N>
__device__ __forceinline__ void wait_loads() {   // all but the N youngest loads, and every LDS access
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));   // the builtin: the compiler counts it
}

template <int QT, int NMAT, int EPI, int RW>
__global__ void __launch_bounds__(kSW * 64) k_gemm_rs(const GemmArgs a, int nu) {
  constexpr int KG = kSW / RW, SB = RW / 2, NS = kSUnit / SB, TT = 2;
  constexpr int RT = RW / NMAT;   // row tiles of each matrix
  constexpr int SUMS = sum_steps<QT>();
  static_assert(RW >= 2 && NS % 4 == 0, "whole turns of the four stages per unit");
  // vector memory instructions of a unit's two loads of codes
  constexpr bool kSumLate = is_wide(QT);   // the block sums at the unit's end (Q4_1, Q5_1: registers)
  // and Q5_1's scales not before its unit begins: with a second set in
  // registers the accumulators went through scratch memory every unit (14336 x
  // 4096 at 77 / 200 / 512 tokens: 91, 178 and 320 us)
  constexpr bool kScaleLate = QT == kQ5_1;
  constexpr int kN1 = (kScaleLate ? 0 : kTB) + (is_kq(QT) ? 1 : 0) + kTB * KCodes<QT>::kQ + (kSumLate ? 0 : SUMS * TT), kN2 = kTB * KCodes<QT>::kQ;
  constexpr int kStage = 2048;   // 16-byte chunks
  __shared__ v4u s0[kStage], s1[kStage], s2[kStage], s3[kStage];
  __shared__ float rn[TT * kSTok], psum[TT][kSW][kSTok];
  __shared__ float inv_lds[TT * kRsUnits * kSTok];   // [TT][nu][32]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rt = wave % RW, kgrp = wave / RW;
  const int n = lane & 31, kg = lane >> 5;
  const int ntk = ((a.cols >> 5) + kTB - 1) / kTB;
  const int ngroups = (a.rows + kRG - 1) / kRG;
  const int row0 = blockIdx.x * 32 * RT;
  const int tile0 = blockIdx.y * TT, ntile = (a.T + kSTok - 1) / kSTok;
  const KsView xs = ks_view(a.xs, ntile, nu);

  KView<QT> wv;
  wv.init(NMAT == 2 && rt >= RT ? a.w2 : a.w, (row0 + 32 * (rt % RT)) / kRG, ngroups, ntk, n, kg);
  __amdgpu_buffer_rsrc_t sr[TT];
  if constexpr (SUMS > 0) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
      sr[tt] = __builtin_amdgcn_make_buffer_rsrc(xs.sum + (size_t)min(tile0 + tt, ntile - 1) * nu * SUMS * kWave, (short)0,
                                                 nu * SUMS * 1024, kBufferFlags);
  }
  const int nit = (nu + KG - 1) / KG;
  auto unit_of = [&](int it) { return min(kgrp + it * KG, nu - 1); };
  // this wave's 4 of the stage's fragments: 8 SB per group, (tt, block, i)
  auto issue = [&](int u, int stage, v4u* buf) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int f = 4 * rt + k, tt = f / (4 * SB), b = f / 4 % SB, i = f % 4;
      const uint4* src = xs.x + ((((size_t)min(tile0 + tt, ntile - 1) * nu + u) * kSUnit + stage * SB + b) * 4 + i) * kWave + lane;
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)src, (lds_ptr_t)&buf[(kgrp * 8 * SB + f) * kWave], 16, 0, 0);
    }
  };

  v16f acc[TT];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) acc[tt] = v16f{};
  // One unit of codes: its first tile is refilled with the next unit's after
  // block 3, with that unit's scales and this one's block sums, its second
  // tile after block 7 (a second unit in registers would spill)
  KCodes<QT> q;
  KScale<QT> w, wn;
  v8h sum[SUMS > 0 ? SUMS : 1][TT];
  auto load_sums = [&](int it) {
#pragma unroll
    for (int s = 0; s < SUMS; ++s)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
        sum[s][tt] = __builtin_bit_cast(
            v8h, __builtin_amdgcn_raw_buffer_load_b128(sr[tt], lane * 16, (unit_of(it) * SUMS + s) * 1024, 0));
  };
  auto load_first = [&](int it) {
    asm volatile("" ::: "memory");   // the count of wait_loads: not before the loads ahead, not after those behind
    load_codes<QT>(q, wv, unit_of(it + 1), 0);
    if constexpr (!kScaleLate) load_scales<QT>(wn, wv, unit_of(it + 1));
    if constexpr (!kSumLate) load_sums(it);
    asm volatile("" ::: "memory");
  };
  auto load_second = [&](int it) {
    asm volatile("" ::: "memory");
    load_codes<QT>(q, wv, unit_of(it + 1), 1);
    asm volatile("" ::: "memory");
  };
  load_codes<QT>(q, wv, unit_of(0), -1);
  load_scales<QT>(w, wv, unit_of(0));
  issue(unit_of(0), 0, s0);
  issue(unit_of(0), 1, s1);
  issue(unit_of(0), 2, s2);
  issue(unit_of(0), 3, s3);
  // inverse scales and sums of squares: as in k_gemm_ks
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
    const size_t at = (size_t)min(tile0 + tt, ntile - 1) * nu * kSTok;
    float ss = 0.f;
    for (int i = tid; i < nu * kSTok; i += kSW * 64) {
      inv_lds[tt * nu * kSTok + i] = xs.inv[at + i];
      ss += xs.ssq[at + i];
    }
    ss += __shfl_xor(ss, 32, kWave);
    if (lane < kSTok) psum[tt][wave][lane] = ss;
  }
  vm_drain();        // every load so far, the four stages among them
  __syncthreads();
  if (tid < TT * kSTok) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < kSW; ++i) ss += psum[tid / kSTok][i][tid % kSTok];
    // the RMSNorm scale of tensor.c:114-131 (read after the loop's barriers)
    rn[tid] = a.nw ? 1.0f / sqrtf(ss / (float)a.cols + a.eps) : 1.0f;
  }
  // x fragments of one block: read from LDS while the block before is used
  struct Frags {
    v8h v[TT][4];
  };
  Frags fa, fb;
  auto read = [&](Frags& x, const v4u* buf, int b) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        x.v[tt][i] = __builtin_bit_cast(v8h, buf[(kgrp * 8 * SB + (tt * SB + b) * 4 + i) * kWave + lane]);
    __builtin_amdgcn_sched_barrier(0);
  };
  read(fa, s0, 0);
  Pipe<QT, TT> pipe;
  pipe.init(q, w);
#pragma unroll 1
  for (int it = 0; it < nit; ++it) {
    const int u = unit_of(it);
    // a group without a unit in the last turn: its sums are dropped
    const bool live = kgrp + it * KG < nu;
    // stage k of the unit from cur (its first block's x read already), the
    // next stage in nxt: past the barrier, cur is read by no one any more
    // (every wave has its last block in registers) and takes the stage four on
    auto stage = [&](auto kc, v4u* cur, const v4u* nxt) {
      constexpr int k = decltype(kc)::value;
      if constexpr (SB == 2) {
        // the first block's x (read a block ago) is here: said before the next
        // reads, or the compiler waits for those too
        __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
        read(fb, cur, 1);
        pipe.template block<k * SB>(q, w, q, wn, fa.v);
        __builtin_amdgcn_sched_barrier(0);
      }
      // the next stage was requested three stages ago; since then two more
      // (4 loads each) and the codes loaded at the end of the three stages
      // before this one
      constexpr int kEnd1 = NS / 2 - 1, kEnd2 = NS - 1;   // the stages that end with them
      constexpr auto among = [](int e) { return e == (k + NS - 1) % NS || e == (k + NS - 2) % NS || e == (k + NS - 3) % NS; };
      wait_loads<8 + (among(kEnd1) ? kN1 : 0) + (among(kEnd2) ? kN2 : 0)>();
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if constexpr (k + 4 < NS)
        issue(u, k + 4, cur);
      else
        issue(unit_of(it + 1), k + 4 - NS, cur);
      asm volatile("" ::: "memory");
      if constexpr (SB == 2) {
        read(fa, nxt, 0);
        pipe.template block<k * SB + 1>(q, w, q, wn, fb.v);
      } else if constexpr (k % 2 == 0) {
        read(fb, nxt, 0);
        pipe.template block<k>(q, w, q, wn, fa.v);
      } else {
        read(fa, nxt, 0);
        pipe.template block<k>(q, w, q, wn, fb.v);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (k == NS / 2 - 1) load_first(it);
    };
    auto turn = [&](auto qc) {   // four stages
      constexpr int q = 4 * decltype(qc)::value;
      stage(std::integral_constant<int, q>{}, s0, s1);
      stage(std::integral_constant<int, q + 1>{}, s1, s2);
      stage(std::integral_constant<int, q + 2>{}, s2, s3);
      stage(std::integral_constant<int, q + 3>{}, s3, s0);
    };
    turn(std::integral_constant<int, 0>{});
    if constexpr (NS == 8) turn(std::integral_constant<int, 1>{});
    if constexpr (kSumLate) load_sums(it);   // (not among the counted: wait_loads then waits for more)
    load_second(it);
    pipe.finish(acc, w, sum, inv_lds + u * kSTok + 4 * kg, nu * kSTok, live);
    if constexpr (kScaleLate)
      load_scales<QT>(w, wv, unit_of(it + 1));   // (nor these)
    else
      w = wn;
  }

  // the column groups' sums of each row tile, added in group order
  vm_drain();
  __syncthreads();
  float* red[TT] = {reinterpret_cast<float*>(s0), reinterpret_cast<float*>(s1)};   // [wave][16][64]
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int j = 0; j < 16; ++j) red[tt][(wave * 16 + j) * kWave + lane] = acc[tt][j];
  __syncthreads();
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int q = 0; q < 2 * RT; ++q) {   // row tile q / 2, register j, lane
      const int j = wave + kSW * (q & 1), r = q >> 1;
      const int tok = 8 * (j >> 2) + 4 * kg + (j & 3), t = (tile0 + tt) * kSTok + tok;
      const int row = row0 + 32 * r + n;
      if (t >= a.T || row >= a.rows) continue;
      float v[NMAT];
#pragma unroll
      for (int m = 0; m < NMAT; ++m) {
        v[m] = 0.f;
#pragma unroll
        for (int g = 0; g < KG; ++g) v[m] += red[tt][((g * RW + m * RT + r) * 16 + j) * kWave + lane];
        v[m] *= rn[tt * kSTok + tok];
      }
      float* yp = a.y + (size_t)t * a.ldy + row;
      if constexpr (EPI == EPI_SWIGLU)
        *yp = v[NMAT - 1] * (a.act == 1 ? gelu_tanh(v[0]) : silu(v[0]));   // layer_scheduler.c:529-547
      else if constexpr (EPI == EPI_ADD)
        *yp += v[0];
      else
        *yp = v[0];
    }
}

}  // namespace
}  // namespace ssk
