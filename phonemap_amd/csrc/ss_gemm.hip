// ss_gemm.hip - launches of the prompt products (ss_gemm.h): the split of x, the
// workgroup shape, and the kernels of matrices of more than 512 columns.

#include "ss_gemm.h"

#include <atomic>

namespace ssk {
namespace {

// Sum of squares of each token's x (one workgroup per token), for the
// embedding's RMSNorm scale.
__global__ void __launch_bounds__(256) k_sumsq(const float* __restrict__ x, int ldx, int cols,
                                               float* __restrict__ ssq) {
  __shared__ float red[4];
  const float* xt = x + (size_t)blockIdx.x * ldx;
  float ss = 0.f;
  for (int c = threadIdx.x * 4; c < cols; c += 1024) {
    const float4 v = *reinterpret_cast<const float4*>(xt + c);
    ss = fmaf(v.x, v.x, ss);
    ss = fmaf(v.y, v.y, ss);
    ss = fmaf(v.z, v.z, ss);
    ss = fmaf(v.w, v.w, ss);
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  if (threadIdx.x == 0) ssq[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// launches per epilogue and kernel (k_gemm_ks, k_gemm_rs)
std::atomic<int64_t> g_gemm_launches[kGemmVariants];
template <int EPI>
void count_launch(int kernel) {
  constexpr int slot = EPI == EPI_STORE ? 0 : EPI == EPI_ADD ? 1 : 2;
  g_gemm_launches[2 * slot + kernel].fetch_add(1, std::memory_order_relaxed);
}

template <int QT, int NMAT, int EPI>
hipError_t launch_ks(const GemmArgs& a, int nu, hipStream_t s) {
  count_launch<EPI>(0);
  if (nu <= 2) return launch_gemm_few(EPI, a, nu, s);
  const dim3 grid((a.rows + 31) / 32, (a.T + kSTok - 1) / kSTok);
  hipLaunchKernelGGL((k_gemm_ks<QT, NMAT, EPI, kSW>), grid, dim3(kSW * 64), 0, s, a, nu);
  return hipGetLastError();
}

template <int QT, int NMAT, int EPI, int RW>
hipError_t launch_rs(const GemmArgs& a, int nu, hipStream_t s) {
  count_launch<EPI>(1);
  const int rows = 32 * RW / NMAT;
  const dim3 grid((a.rows + rows - 1) / rows, (a.T + 2 * kSTok - 1) / (2 * kSTok));
  hipLaunchKernelGGL((k_gemm_rs<QT, NMAT, EPI, RW>), grid, dim3(kSW * 64), 0, s, a, nu);
  return hipGetLastError();
}

// The workgroup shape: 1 for k_gemm_ks, else k_gemm_rs's RW. Every shape runs
// one workgroup per compute unit at a time, so a launch takes its rounds of
// workgroups times what one round takes: at 4096 columns 10 us (two matrices
// 18: half the waves for each), 24 us (RW 2) and 38 us (RW 4), and in the
// same ratio at others. The least of the three was the fastest measured at
// every token count from 8 to 512 of 4096, 11008 and 1024 rows but for ties
// (4096 rows, 77 / 128 / 256 / 512 tokens: 25.1, 27.1, 48.8, 89.3 us with 1;
// 26.3, 27.3, 32.7, 58.3 with 2; 36.8, 37.5, 40.9, 49.7 with 4).
// rw: the most row tiles the type has.
//
// Up to 512 columns k_gemm_ks has a wave per unit and matrix, so 8 / nu
// workgroups of one matrix run on a compute unit at a time. One unit: always
// (Q8_0 8192 x 256, 33 / 512 tokens: 9.3 and 20.4 us; with 8 waves of which one
// works 14.4, with RW 4 24.8). Two: a round takes 4.5 to 6 us, RW 2's at least
// as long and RW 4's 6.5 (8192 x 512, 512 tokens: 31.4 us, RW 4 25.6; 4100 x
// 512, 100 tokens: 10.6 and 14.3).
int pick_shape(int rows, int T, int nmat, int nu, int rw, int n_cu) {
  auto rounds = [&](int r, int t, int per_cu = 1) {
    const long wg = (long)((rows + r - 1) / r) * ((T + t - 1) / t), slots = (long)per_cu * n_cu;
    return (wg + slots - 1) / slots;
  };
  if (nu == 1) return 1;
  if (nu == 2) {
    const long c1 = rounds(32, 32, 4 / nmat) * 50, c2 = rounds(64 / nmat, 64) * 52, c4 = rounds(128 / nmat, 64) * 65;
    if (c1 <= c2 && (rw < 4 || c1 <= c4)) return 1;
    return rw < 4 || c2 <= c4 ? 2 : 4;
  }
  const long c1 = rounds(32, 32) * (nmat == 2 ? 18 : 10);
  const long c2 = rounds(64 / nmat, 64) * 24, c4 = rounds(128 / nmat, 64) * 38;
  if (nu > kRsUnits || (c1 <= c2 && (rw < 4 || c1 <= c4))) return 1;
  return rw < 4 || c2 <= c4 ? 2 : 4;
}
// Q4_1 and Q5_1 (a scale and a minimum of 16 bits per block) run with at most
// RW 2: RW 4 would keep 1040 bytes per lane of Q5_1 in scratch memory
constexpr int most_row_tiles(int qt) { return qt == kQ4_1 || qt == kQ5_1 ? 2 : 4; }

template <int QT, int NMAT, int EPI>
hipError_t launch_shape(const GemmArgs& a, int nu, hipStream_t s) {
  constexpr int RW = most_row_tiles(QT);
  switch (pick_shape(a.rows, a.T, NMAT, nu, RW, a.n_cu)) {
    case 1: return launch_ks<QT, NMAT, EPI>(a, nu, s);
    case 2: return launch_rs<QT, NMAT, EPI, 2>(a, nu, s);
    default: return launch_rs<QT, NMAT, EPI, RW>(a, nu, s);
  }
}

template <int QT>
hipError_t launch_type(int epi, const GemmArgs& a, hipStream_t s) {
  const int nb = a.cols / 32, nu = (nb + kSUnit - 1) / kSUnit;
  const KsView v = ks_view(a.xs, (a.T + kSTok - 1) / kSTok, nu);
  hipLaunchKernelGGL(k_split_ks<sum_steps<QT>()>, dim3((a.T + 7) / 8, nu), dim3(64), 0, s, a.x, a.ldx, a.nw, a.T, nb, v);
  if (hipError_t e = hipGetLastError()) return e;
  switch (epi) {
    case EPI_STORE: return launch_shape<QT, 1, EPI_STORE>(a, nu, s);
    case EPI_ADD: return launch_shape<QT, 1, EPI_ADD>(a, nu, s);
    default: return launch_shape<QT, 2, EPI_SWIGLU>(a, nu, s);
  }
}

}  // namespace

void gemm_launch_counts(int64_t* out, int n) {
  for (int i = 0; i < n && i < kGemmVariants; ++i) out[i] = g_gemm_launches[i].load(std::memory_order_relaxed);
}

int gemm_shape(int rows, int T, int nmat, int cols, int type, int n_cu) {
  return pick_shape(rows, T, nmat, (cols / 32 + kSUnit - 1) / kSUnit, most_row_tiles(dev_type(type)), n_cu);
}

hipError_t launch_sumsq(const float* x, int cols, int T, float* ssq, hipStream_t s) {
  if (T <= 0 || cols <= 0 || cols % 4) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_sumsq, dim3(T), dim3(256), 0, s, x, cols, cols, ssq);
  return hipGetLastError();
}

hipError_t launch_gemm(int epi, const GemmArgs& a, hipStream_t s) {
  if (a.T <= 0 || a.rows <= 0 || a.cols <= 0 || a.cols % 32 || a.ldy < a.rows || a.ldx < a.cols || a.ldx % 4 || !a.xs ||
      a.n_cu <= 0)
    return hipErrorInvalidValue;
  if (epi != EPI_STORE && epi != EPI_ADD && epi != EPI_SWIGLU) return hipErrorInvalidValue;
  const int t = dev_type(a.type);
  if (is_kq(t) && a.cols % 256) return hipErrorInvalidValue;   // whole super-blocks
  switch (t) {
    case 2: return launch_type<2>(epi, a, s);
    case 8: return launch_type<8>(epi, a, s);
    case kQ4_1: return launch_type<kQ4_1>(epi, a, s);
    case kQ5_1: return launch_type<kQ5_1>(epi, a, s);
    case kQ8_1: return launch_type<kQ8_1>(epi, a, s);
    case kQ2K: return launch_type<kQ2K>(epi, a, s);
    case kQ3K: return launch_type<kQ3K>(epi, a, s);
    case kQ4K: return launch_type<kQ4K>(epi, a, s);
    case kQ5K: return launch_type<kQ5K>(epi, a, s);
    case kQ6K: return launch_type<kQ6K>(epi, a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ssk
