// ss_flash.h - causal attention of a prompt's rows on MFMA (gfx950).
//
// The reference evaluates a prompt token by token, each token attending to
// positions 0..its own over the fp16 cache (layer_scheduler.c:415-468, called
// per token from ss_scheduler_prefill, :681-803). Here the tokens of a prompt
// chunk attend together, 32 query rows of one KV head to a tile (row r: token
// r / G, head r % G), on v_mfma_f32_32x32x16_f16.
//
// Operand layout of v_mfma_f32_32x32x16_f16 (checked on the device by the
// prompt products): lane l supplies A[l%32][8(l/32) + i] and B[8(l/32) + i][l%32],
// i = 0..7, and receives D[8(j/4) + 4(l/32) + j%4][l%32], j = 0..15.
//
// Each wave owns 32 query rows and, per 32-key block, computes transposed
// tiles: S^T = K Q^T (A = the keys' K rows, B = Q^T), so lane (n, h) = (l%32,
// l/32) receives scores of query row n, and O^T = V^T P^T (A = V^T, B = P^T),
// whose B operand is exactly the scores' D registers once row 16c + 8b + 4h + i
// of the S^T tile is key 16c + 8h + 4b + i: elements 8c..8c+7 of lane (n, h)
// are then keys 16c + 8h + 0..7 of query row n, the B layout. A row's softmax
// statistics live in lanes n and n + 32 (one v_permlane32_swap per reduction).
//
// Precision: K and V are fp16 in the cache (exact MFMA operands). q, times the
// softmax's scale and log2(e) (that product to 2^-48), is scaled per row by a
// power of two (its largest magnitude to [2^13, 2^14)) and held as two fp16
// parts, to 2^-23 of the value; P (times 2^12) is held the same way; each
// product is two MFMAs accumulating in fp32. The softmax is the online form
// (running maximum and sum per row) in fp32, in base 2; maxima are whole
// numbers, so moving one is exact, and one may lag the true maximum by up to 3
// (P <= 2^3: 2^15 after the scale, inside fp16's range), so most blocks skip
// rescaling O. What else rounds are the sums, in two forms. FULL adds a
// score's high parts in two chains and a block's share of O from zero: each
// sum rounds a few times per block, and over 4 to 7 tokens (fp16) and 4 to 64
// (int8), contexts 4 to 4008 and every head dimension its error against 64
// bits is that of the attention of single tokens, which sums in fp32
// throughout (0.98 and 0.89 of it, geometric means; 1.8 and 1.4 with one chain
// of sixteen MFMAs per score, a scale rounded to fp32 and weights' exponents
// up to 15). It is used where such tokens would otherwise be attended one by
// one. The other form runs longer fp16 prompts: the score's parts in one
// chain, the low ones first, and O one chain over all blocks (1.2 of that
// error, up to 1.8 at 4000 positions; 100 tokens over 3000, 32 heads on 8,
// head_dim 128: 38 us, FULL 43).
//
// Bound and split. At 32 rows per wave one LDS operand read feeds two MFMAs of
// 32 cycles, so a block is 1024 matrix cycles per wave at head_dim 128 against
// 512 of LDS and about as many of softmax as of products. A workgroup is RT row
// tiles x KG key groups, the groups taking every KG-th block and merged through
// LDS at the end, so a short prompt over a long prefix walks KG times fewer
// steps. With 16 rows per wave, four waves walking all keys and V transposed
// in registers, 512 tokens over 1536 (32 heads on 8, head_dim 128) took 94 us
// and 77 over 1000 50 us; now 41 and 18, the first 1.6 times what a large
// fp16 product takes for the same operations. At head_dim 256 the O and q of
// 32 rows would leave one wave per SIMD pair, so DS = 2 waves share a row tile:
// each scores half of the head dimension and the halves are added through LDS,
// and each holds half of O (64 tokens over 700, 16 heads on 8: 31 us; one
// wave 44; before 60).
//
// Staging, per block and key group, double buffered, by direct global-to-LDS
// loads: K rows in tile-row order (16-byte chunk c of row r at slot c ^ kswz),
// V rows as they are (chunk c at slot c ^ vswz(key)), read transposed by
// ds_read_b64_tr_b16 (lane i of 16 addresses key i/4, dims 4(i%4)..+3, and
// receives dim i of the four keys). Both swizzles spread a read over all banks.
//
// An int8 cache's codes are exact in fp16: a block passes through registers,
// where codes become fp16 (requested before the current block's products,
// written to LDS after them), a position's K scale multiplies its scores and
// its V scale the weights after the row's sum took them. Weight times V scale
// has no bound of its own, so each row also keeps the binary exponent of its
// largest one (lagging by 2 at most) and holds P, and so O, relative to that:
// a row's precision depends on the positions it sees alone. A position the row
// does not see has V scale 0 (its own may be infinite).

#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>

#include "ss_device.h"
#include "ss_kernels.h"

namespace ssk {

// The FULL form's launches (ss_flash_full.hip): RT, KG as launch_attention_rows chose them.
hipError_t launch_flash_full(int head_dim, int rt, int kg, int group, int kv_type, const AttnArgs& a, hipStream_t s);

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(3))) v4s* lds_v4s_t;
typedef __attribute__((address_space(1))) void* gbl_ptr_t;

constexpr int kBlk = 32;            // keys per block, query rows per tile
constexpr float kLog2e = 1.44269504088896340736f, kLog2eLow = 1.92596299e-8f;   // log2 e = their sum
constexpr float kPExp = 12.0f, kPScale = 4096.0f;   // P is held times 2^12
constexpr float kLag = 3.0f;        // the running maximum's lag (base 2)
constexpr float kLagX = 2.0f;       // int8: the lag of the exponent of weight times V scale

// the value of the lane with the same query row (lane ^ 32) joined to this one's
__device__ __forceinline__ float max_pair(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_pair(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// 2^e of a whole number (or -inf: 0)
__device__ __forceinline__ float pow2(float e) { return ldexpf(1.0f, (int)fmaxf(e, -200.f)); }

// hi + lo = v (to 2^-23 of |v| for normal values) as two fp16 vectors
__device__ __forceinline__ void split8(const float* v, v8h& hi, v8h& lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const _Float16 h = (_Float16)v[i];
    hi[i] = h;
    lo[i] = (_Float16)(v[i] - (float)h);
  }
}

// 8 int8 codes -> fp16, exact: 1024 + (code + 128) by placing the byte, less 1152
__device__ __forceinline__ v4u codes8(uint32_t lo, uint32_t hi) {
  const v2h off = {(_Float16)1152.f, (_Float16)1152.f};
  v4u r;
  lo ^= 0x80808080u;
  hi ^= 0x80808080u;
  r[0] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u)) - off);
  r[1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u)) - off);
  r[2] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u)) - off);
  r[3] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u)) - off);
  return r;
}

// tile row -> key of the block: bits 2 and 3 change places (its own inverse)
__host__ __device__ constexpr int tile_key(int r) { return (r & 19) | ((r & 4) << 1) | ((r & 8) >> 1); }
// slot swizzles (16-byte chunks of a row of CH): 16 neighbouring tile rows take
// 16 places of 256 bytes; the 4 keys of a transposed read take 4 groups of 4
template <int CH> __device__ __forceinline__ int kswz(int row) { return CH == 8 ? (row >> 1) & 7 : row & 15; }
template <int CH> __device__ __forceinline__ int vswz(int key) { return CH == 8 ? 2 * (key & 2) : 4 * (key & 3); }

// One query row over positions 0..lim of the fp16 cache by one wave in fp32: 64
// keys at a time, one per lane, then their V rows, lane l taking dimensions l,
// l + 64, ... For the rows a tile's products cannot serve: a V that is not
// finite reaches, as 0 * inf, rows that do not see its position. (Finite
// launches pay one test per output: 180 shapes take 0.999 of what they took
// without, geometric mean. 512 tokens over 1536 that all see a NaN, 32 heads on
// 8, head_dim 128: 2.1 ms.)
template <int HD>
__device__ __forceinline__ void one_row(const AttnArgs& a, const float* q, const uint16_t* kc, const uint16_t* vc, int lim,
                                        float* out) {
  constexpr int ND = HD / kWave;
  const int lane = threadIdx.x & 63;
  float m = -INFINITY, l = 0.f, o[ND] = {};
#pragma unroll 1
  for (int k0 = 0; k0 <= lim; k0 += kWave) {
    float s = -INFINITY;
    if (k0 + lane <= lim) {
      const uint16_t* kr = kc + (size_t)(k0 + lane) * HD;
      s = 0.f;
#pragma unroll 1
      for (int i = 0; i < HD; i += 8) {
        const v8h kv = *reinterpret_cast<const v8h*>(kr + i);
#pragma unroll
        for (int k = 0; k < 8; ++k) s = fmaf(q[i + k], (float)kv[k], s);
      }
      s *= a.scale;
      if (a.softcap > 0.f) s = softcap(s, a);
    }
    const float mn = fmaxf(m, wave_max(s));
    const float mo = mn == -INFINITY ? 0.f : mn;
    const float p = expf(s - mo), corr = expf(m - mo);
    l = l * corr + wave_sum(p);
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d] *= corr;
    const int nk = min(kWave, lim + 1 - k0);
#pragma unroll 1
    for (int j = 0; j < nk; j += 8) {   // (past the last: the last again, not added)
      float pj[8], v[8][ND];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int ju = min(j + u, nk - 1);
        pj[u] = __shfl(p, ju, kWave);
#pragma unroll
        for (int d = 0; d < ND; ++d) v[u][d] = h2f(vc[(size_t)(k0 + ju) * HD + lane + kWave * d]);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (j + u < nk) {
#pragma unroll
          for (int d = 0; d < ND; ++d) o[d] = fmaf(pj[u], v[u][d], o[d]);
        }
    }
    m = mn;
  }
#pragma unroll
  for (int d = 0; d < ND; ++d) out[lane + kWave * d] = o[d] / l;
}

template <int HD, int G, int RT, int KG, int DS, bool Q8, bool FULL>
__global__ void __launch_bounds__(RT * KG * DS * 64) k_flash_rows(const AttnArgs a) {
  constexpr int CH = HD / 8;             // 16-byte chunks per row
  constexpr int NC = HD / 16 / DS;       // a wave's 16-wide slices of the head dimension
  constexpr int NDT = HD / 32 / DS;      // and 32-dim tiles of O^T
  constexpr int NT = RT * KG * DS * 64;
  constexpr int kGrp = kBlk * CH;        // chunks of one key group's block
  constexpr int kLoads = kGrp / (64 * RT * DS);   // direct loads per wave, K and V each
  static_assert(HD == 64 || HD == 128 || HD == 256, "head_dim 64, 128 or 256");
  static_assert(kBlk % G == 0 && RT <= 2 && KG % 2 == 0 && kGrp % (64 * RT * DS) == 0, "shape");

  // two buffers of each, as separate arrays: the loop names them at compile
  // time, so the compiler can tell the buffer being read from the one the
  // direct global-to-LDS loads of the next block fill, and does not wait for
  // those loads before the current block's reads
  __shared__ v4u ks0[KG * kGrp], ks1[KG * kGrp];
  __shared__ v4u vs0[KG * kGrp], vs1[KG * kGrp];
  __shared__ float xs[DS > 1 ? RT * KG * DS : 1][DS > 1 ? 16 * 64 : 1];   // the waves' shares of S^T
  __shared__ float sc0[Q8 ? KG : 1][64], sc1[Q8 ? KG : 1][64];   // int8: the block's K scales, then its V scales
  __shared__ float gm[KG][RT * 32], gl[KG][RT * 32];   // each group's maximum and sum of a row

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ds = wave % DS, rt = wave / DS % RT, g = wave / (DS * RT);
  const int n = lane & 31, h = lane >> 5;
  // neighbouring workgroups take the KV heads in turn, so the workgroups of
  // one head meet in one XCD's L2; the longest prefixes come first
  const int kvh = blockIdx.x % a.n_kv_heads;
  const int row0 = (gridDim.x / a.n_kv_heads - 1 - blockIdx.x / a.n_kv_heads) * (RT * 32);

  // this lane's query row: token z, head hq of the KV head's group
  const int row = row0 + 32 * rt + n;
  const int z = row / G, hq = row % G;
  const int lim = a.pos0 + z;   // last position the row sees (rows past the last token are not stored)
  // positions 0..ctx-1 serve every token of the workgroup; wmin..wmax are this wave's rows' limits
  const int ctx = a.pos0 + min((row0 + RT * 32 - 1) / G, a.n_tok - 1) + 1;
  const int wmin = a.pos0 + (row0 + 32 * rt) / G, wmax = min(wmin + 32 / G, ctx) - 1;
  const int nstep = (ctx + KG * kBlk - 1) / (KG * kBlk);

  const bool cap = a.softcap > 0.f;
  float qv[NC][8];
  float amax = 0.f;
  {
    const float* qp = a.q + (size_t)min(z, a.n_tok - 1) * a.tok_q + ((size_t)kvh * G + hq) * HD + 8 * h;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const float4 x0 = *reinterpret_cast<const float4*>(qp + 16 * (ds * NC + c));
      const float4 x1 = *reinterpret_cast<const float4*>(qp + 16 * (ds * NC + c) + 4);
      qv[c][0] = x0.x, qv[c][1] = x0.y, qv[c][2] = x0.z, qv[c][3] = x0.w;
      qv[c][4] = x1.x, qv[c][5] = x1.y, qv[c][6] = x1.z, qv[c][7] = x1.w;
    }
  }
  const size_t head_base = (size_t)kvh * a.max_seq * HD;
  const uint16_t* kc = static_cast<const uint16_t*>(a.kc) + (Q8 ? 0 : head_base);
  const uint16_t* vc = static_cast<const uint16_t*>(a.vc) + (Q8 ? 0 : head_base);

  // this group's block of a step -> LDS, each of its RT * DS waves a share
  // (positions past ctx - 1 reload ctx - 1: finite, masked)
  auto stage = [&](int step, v4u* kd, v4u* vd) {
    const int kb = (step * KG + g) * kBlk;
    if (kb >= ctx) return;
    int ln = lane;
    if (HD == 256) asm volatile("" : "+v"(ln));   // places computed again each step, not kept in registers
#pragma unroll
    for (int k = 0; k < kLoads; ++k) {
      const int base = ((rt * DS + ds) * kLoads + k) * 64;
      const int r = (base + ln) / CH, slot = (base + ln) % CH;
      const int pk = min(kb + tile_key(r), ctx - 1);
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)(kc + (size_t)pk * HD + 8 * (slot ^ kswz<CH>(r))),
                                       (lds_ptr_t)&kd[g * kGrp + base], 16, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < kLoads; ++k) {
      const int base = ((rt * DS + ds) * kLoads + k) * 64;
      const int r = (base + ln) / CH, slot = (base + ln) % CH;
      const int pv = min(kb + r, ctx - 1);
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)(vc + (size_t)pv * HD + 8 * (slot ^ vswz<CH>(r))),
                                       (lds_ptr_t)&vd[g * kGrp + base], 16, 0, 0);
    }
  };
  // an int8 block passes through registers: 16 codes are two chunks of fp16
  constexpr int kQLoads = Q8 ? kLoads / 2 : 1, kQRow = HD / 16;
  static_assert(kLoads % 2 == 0, "pairs of chunks");
  v4u kq[kQLoads], vq[kQLoads];
  float qsc = 0.f;
  auto load_q = [&](int step) {
    const int kb = (step * KG + g) * kBlk;
    if (kb >= ctx) return;
    const int8_t* k8 = static_cast<const int8_t*>(a.kc) + head_base;
    const int8_t* v8 = static_cast<const int8_t*>(a.vc) + head_base;
#pragma unroll
    for (int k = 0; k < kQLoads; ++k) {
      const int i = ((rt * DS + ds) * kQLoads + k) * 64 + lane;
      const int pk = min(kb + tile_key(i / kQRow), ctx - 1), pv = min(kb + i / kQRow, ctx - 1);
      kq[k] = *reinterpret_cast<const v4u*>(k8 + (size_t)pk * HD + 16 * (i % kQRow));
      vq[k] = *reinterpret_cast<const v4u*>(v8 + (size_t)pv * HD + 16 * (i % kQRow));
    }
    qsc = (h ? a.vs : a.ks)[min(kb + n, ctx - 1)];
  };
  auto store_q = [&](int step, v4u* kd, v4u* vd, float (*scd)[64]) {
    if ((step * KG + g) * kBlk >= ctx) return;
#pragma unroll
    for (int k = 0; k < kQLoads; ++k) {
      const int i = ((rt * DS + ds) * kQLoads + k) * 64 + lane;
      const int r = i / kQRow, c = 2 * (i % kQRow);
      v4u* kr = kd + g * kGrp + r * CH;
      v4u* vr = vd + g * kGrp + r * CH;
      kr[c ^ kswz<CH>(r)] = codes8(kq[k][0], kq[k][1]);
      kr[(c + 1) ^ kswz<CH>(r)] = codes8(kq[k][2], kq[k][3]);
      vr[c ^ vswz<CH>(r)] = codes8(vq[k][0], vq[k][1]);
      vr[(c + 1) ^ vswz<CH>(r)] = codes8(vq[k][2], vq[k][3]);
    }
    if (rt == 0 && ds == 0) scd[g][lane] = qsc;
  };
  // the staged loads have landed and the other buffer's reads are done, for
  // this wave, and for the others where waves share the staging
  auto turn = [&] {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    if (RT * DS > 1) __syncthreads();
  };

  if (Q8) {
    load_q(0);
    store_q(0, ks0, vs0, sc0);
  } else {
    stage(0, ks0, vs0);
  }

  // q as the B operand of S^T: lane (n, h) holds q[16c + 8h + i] of row n
  v8h qh[NC], ql[NC];
  float qscale;
  {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(qv[c][i]));
    amax = max_pair(amax);
    if (DS > 1) {   // the row's other half counts too
      xs[wave][lane] = amax;
      __syncthreads();
      amax = fmaxf(amax, xs[wave ^ 1][lane]);
    }
    int e = 0;
    // q times the softmax's scale (and log2 e), as sh + sl, keeps what its two
    // parts hold
    const float c0 = cap ? a.scale : a.scale * kLog2e;
    const float c1 = cap ? 0.f : __builtin_fmaf(a.scale, kLog2e, -c0) + a.scale * kLog2eLow;
    frexpf(amax * c0, &e);
    const int shift = min(max(14 - e, -100), 100);
    const float sh = ldexpf(c0, shift), sl = ldexpf(c1, shift);
    qscale = ldexpf(1.0f, -shift);   // S^T holds the scores * 2^shift
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float p = qv[c][i] * sh;
        asm("" : "+v"(p));   // one value for both parts (see the weights below)
        const _Float16 hi = (_Float16)p;
        qh[c][i] = hi;
        ql[c][i] = (_Float16)__builtin_fmaf(qv[c][i], sl, __builtin_fmaf(qv[c][i], sh, -(float)hi));
      }
  }
  const float qs = cap ? kLog2e : qscale;   // scores of the tile -> base-2 exponents

  v16f o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = v16f{};
  float m = -INFINITY, l = 0.f;   // l: this lane's share of the row's sum, times 2^12 (int8: the sum)
  float ex = -INFINITY;           // int8: the exponent O is held relative to, times 2^12

  // transposed V read: lane's key of 4 and its 8 bytes of a 32-dim tile
  const int vkey = 8 * h + ((lane >> 2) & 3);
  const int vch = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);

  auto step = [&](int st, const v4u* kall, const v4u* vall, const float (*scl)[64], v4u* knxt, v4u* vnxt,
                  float (*scn)[64]) {
    if (st + 1 < nstep) {
      if (Q8) load_q(st + 1);
      else stage(st + 1, knxt, vnxt);
    }
    const int kb = (st * KG + g) * kBlk;
    const v4u* kcur = kall + g * kGrp;
    const v4u* vcur = vall + g * kGrp;
    v16f acc = v16f{};
    if (kb <= wmax) {
      auto read_k = [&](int c) {
        return __builtin_bit_cast(v8h, kcur[n * CH + ((2 * (ds * NC + c) + h) ^ kswz<CH>(n))]);
      };
      // slices c0 .. c0 + N - 1 in one chain, the low parts first: what rounds then is the small sum
      auto chain = [&](auto nc, int c0, v16f d) {
        constexpr int N = decltype(nc)::value;
        v8h kv[N];
#pragma unroll
        for (int c = 0; c < N; ++c) {
          kv[c] = read_k(c0 + c);
          d = __builtin_amdgcn_mfma_f32_32x32x16_f16(kv[c], ql[c0 + c], d, 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < N; ++c) d = __builtin_amdgcn_mfma_f32_32x32x16_f16(kv[c], qh[c0 + c], d, 0, 0, 0);
        return d;
      };
      if constexpr (FULL) {
        constexpr std::integral_constant<int, NC / 2> half;
        const v16f first = chain(half, 0, v16f{});
        acc = first + chain(half, NC / 2, v16f{});
      } else {
        acc = chain(std::integral_constant<int, NC>{}, 0, v16f{});
      }
    }
    if (DS > 1) {   // the sum of the two waves' shares, the same in both
#pragma unroll
      for (int j = 0; j < 16; ++j) xs[wave][64 * j + lane] = acc[j];
      __syncthreads();
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[j] += xs[wave ^ 1][64 * j + lane];
    }
    if (kb <= wmax) {
      // element j is key kb + 16(j/8) + 8h + j%8 of row n
      float sc[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) sc[j] = Q8 ? acc[j] * scl[g][16 * (j / 8) + 8 * h + j % 8] : acc[j];
      float vsc[Q8 ? 16 : 1];
      if constexpr (Q8) {
#pragma unroll
        for (int j = 0; j < 16; ++j) vsc[j] = scl[g][32 + 16 * (j / 8) + 8 * h + j % 8];
      }
      if (cap) {   // (q . k) / sqrt(hd), softcapped (layer_scheduler.c:442-448)
#pragma unroll
        for (int j = 0; j < 16; ++j) sc[j] = softcap(sc[j] * qscale, a);
      }
      if (kb + kBlk - 1 > wmin) {   // causal limit
#pragma unroll
        for (int j = 0; j < 16; ++j)
          if (kb + 16 * (j / 8) + 8 * h + j % 8 > lim) {
            sc[j] = -INFINITY;
            if constexpr (Q8) vsc[j] = 0.f;
          }
      }
      float bmax = sc[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) bmax = fmaxf(bmax, sc[j]);
      bmax = max_pair(bmax) * qs;
      if (__any(bmax > m + kLag)) {
        const float mn = ceilf(fmaxf(m, bmax));
        const float corr = pow2(m - (mn == -INFINITY ? 0.f : mn));
        l *= corr;
        if constexpr (!Q8) {
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) o[dt] *= corr;
        }
        m = mn;
      }
      const float mo = m == -INFINITY ? 0.f : m;   // nothing seen yet: weights stay 0
      float pv[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) pv[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[j], qs, -mo));   // layer_scheduler.c:450-458
      {
        float t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = pv[j] + pv[j + 8];
        l += ((t[0] + t[4]) + (t[1] + t[5])) + ((t[2] + t[6]) + (t[3] + t[7]));
      }
      if constexpr (Q8) {
        float bx = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          pv[j] *= vsc[j];
          bx = fmaxf(bx, pv[j]);
        }
        bx = max_pair(bx);   // below 2^(e + 1)
        const float t = m + (float)max((int)(__float_as_uint(bx) >> 23) - 127, -100);
        if (__any(bx > 0.f && t > ex + kLagX)) {
          const float en = bx > 0.f ? fmaxf(ex, t) : ex;
          const float corr = en == ex ? 1.f : pow2(ex - en);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) o[dt] *= corr;
          ex = en;
        }
        const int up = (int)fminf(kPExp + m - ex, 126.f);   // (past 126 with every pv 0 only)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          pv[j] = ldexpf(pv[j], up);
          // rounded to fp32 before it is split: as a factor of the split's
          // conversions it would give hi two values, one to multiply and
          // another to take lo from, an fp16 step apart where they round to
          // different sides
          asm("" : "+v"(pv[j]));
        }
      }
      if constexpr (!Q8) {
#pragma unroll
        for (int j = 0; j < 16; ++j) pv[j] *= kPScale;   // (exact: part of the split's conversions)
      }
      v8h ph[2], pl[2];
      split8(pv, ph[0], pl[0]);
      split8(pv + 8, ph[1], pl[1]);
      // O^T += V^T P^T
      auto read_v = [&](int c, int dt) {
        union { v4s t[2]; v8h v; } vv;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int key = 16 * c + 4 * u + vkey;
          const v4u* p = &vcur[key * CH + ((4 * (ds * NDT + dt) + vch) ^ vswz<CH>(vkey))];
          vv.t[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t)(reinterpret_cast<const v4s*>(p) + (lane & 1)));
        }
        return vv.v;
      };
      if constexpr (FULL) {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          const v8h v0 = read_v(0, dt), v1 = read_v(1, dt);
          v16f r = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, pl[0], v16f{}, 0, 0, 0);
          r = __builtin_amdgcn_mfma_f32_32x32x16_f16(v1, pl[1], r, 0, 0, 0);
          r = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, ph[0], r, 0, 0, 0);
          r = __builtin_amdgcn_mfma_f32_32x32x16_f16(v1, ph[1], r, 0, 0, 0);
          o[dt] += r;
        }
      } else {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const v8h v = read_v(c, dt);
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, ph[c], o[dt], 0, 0, 0);
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, pl[c], o[dt], 0, 0, 0);
          }
      }
    }
    if (Q8 && st + 1 < nstep) store_q(st + 1, knxt, vnxt, scn);
    turn();
  };
  turn();
#pragma unroll 1
  for (int st = 0; st < nstep; st += 2) {
    step(st, ks0, vs0, sc0, ks1, vs1, sc1);
    if (st + 1 < nstep) step(st + 1, ks1, vs1, sc1, ks0, vs0, sc0);
  }

  // the groups' rows -> one: every group's O at the common maximum through
  // LDS (the staging buffers: RT * KG tiles of 32 rows x HD floats, KG / 2 in
  // each), then summed row by row   (layer_scheduler.c:460-466)
  l = sum_pair(l);
  if (h == 0 && ds == 0) {
    gm[g][32 * rt + n] = m;
    gl[g][32 * rt + n] = l;
  }
  __syncthreads();
  {
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < KG; ++k) mx = fmaxf(mx, gm[k][32 * rt + n]);
    float lt = 0.f;
#pragma unroll
    for (int k = 0; k < KG; ++k) {
      const float mk = gm[k][32 * rt + n];
      lt += mk == -INFINITY ? 0.f : gl[k][32 * rt + n] * __builtin_amdgcn_exp2f(mk - mx);
    }
    // (a row whose scores are all -inf keeps its 0 / 0)
    const float f = (m == -INFINITY ? 0.f : pow2((Q8 ? ex : m) - kPExp - mx)) / lt;
    auto bank = [&](int w) { return w == 0 ? ks0 : w == 1 ? vs0 : w == 2 ? ks1 : vs1; };
    const int tile = wave / DS;
    float4* dst = reinterpret_cast<float4*>(bank(tile / (KG / 2))) + (tile % (KG / 2)) * (32 * HD / 4);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q)   // dims 32dt + 8q + 4h .. +3 of row n
        dst[n * (HD / 4) + ((8 * (ds * NDT + dt) + 2 * q + h) ^ (n & 15))] =
            make_float4(o[dt][4 * q] * f, o[dt][4 * q + 1] * f, o[dt][4 * q + 2] * f, o[dt][4 * q + 3] * f);
    __syncthreads();
    static_assert(RT * 32 * (HD / 4) % NT == 0, "every lane of a wave takes each turn");
    float odd = 0.f;   // NaN: some output of this thread is not finite
    for (int i = tid; i < RT * 32 * (HD / 4); i += NT) {
      const int r = i / (HD / 4), c = i % (HD / 4);
      const int zr = (row0 + r) / G, hr = (row0 + r) % G;
      const bool live = zr < a.n_tok;
      float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int k = 0; k < KG; ++k) {
        const int w = k * RT + r / 32;
        const float4* src = reinterpret_cast<const float4*>(bank(w / (KG / 2))) + (w % (KG / 2)) * (32 * HD / 4);
        const float4 v = src[(r % 32) * (HD / 4) + (c ^ (r & 15))];
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
        s.w += v.w;
      }
      if (live) *reinterpret_cast<float4*>(a.out + (size_t)zr * a.tok_o + ((size_t)kvh * G + hr) * HD + 4 * c) = s;
      // (inf - inf and NaN - NaN are NaN)
      if (!Q8 && live) odd += (s.x - s.x) + (s.y - s.y) + (s.z - s.z) + (s.w - s.w);
    }
    // fp16: rows that are not finite, again, each over the positions it sees
    // alone (layer_scheduler.c:415-468 reads no others). A row's HD / 4 threads
    // are neighbours in one wave.
    if (!Q8 && __ballot(odd != odd)) {
      vm_drain();   // this wave's stores
#pragma unroll 1
      for (int i = tid; i < RT * 32 * (HD / 4); i += NT) {
        const int r = i / (HD / 4), z = (row0 + r) / G;
        float* op = a.out + (size_t)z * a.tok_o + ((size_t)kvh * G + (row0 + r) % G) * HD;
        float d = 0.f;
        if (z < a.n_tok)
          for (int k = 0; k < 4; ++k) d += op[4 * (i % (HD / 4)) + k] - op[4 * (i % (HD / 4)) + k];
        uint64_t bad = __ballot(d != d);
        while (bad) {
          const int at = __ffsll((unsigned long long)bad) - 1, rb = __shfl(r, at, kWave);
          bad &= ~(((HD / 4 < 64 ? 1ull << (HD / 4 % 64) : 0ull) - 1) << (at / (HD / 4) * (HD / 4)));
          const int zb = (row0 + rb) / G;
          const size_t head = ((size_t)kvh * G + (row0 + rb) % G) * HD;
          one_row<HD>(a, a.q + (size_t)zb * a.tok_q + head, kc, vc, a.pos0 + zb, a.out + (size_t)zb * a.tok_o + head);
        }
      }
    }
  }
}

template <int HD, int RT, int KG, int DS, bool Q8, bool FULL>
hipError_t launch_flash(int group, const AttnArgs& a, hipStream_t s) {
  const int64_t tiles = ((int64_t)a.n_tok * group + 32 * RT - 1) / (32 * RT);
  if (tiles * a.n_kv_heads > INT32_MAX) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(tiles * a.n_kv_heads)), block(RT * KG * DS * 64);
  switch (group) {
    case 1: hipLaunchKernelGGL((k_flash_rows<HD, 1, RT, KG, DS, Q8, FULL>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_flash_rows<HD, 2, RT, KG, DS, Q8, FULL>), grid, block, 0, s, a); break;
    case 4: hipLaunchKernelGGL((k_flash_rows<HD, 4, RT, KG, DS, Q8, FULL>), grid, block, 0, s, a); break;
    case 8: hipLaunchKernelGGL((k_flash_rows<HD, 8, RT, KG, DS, Q8, FULL>), grid, block, 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace
}  // namespace ssk
