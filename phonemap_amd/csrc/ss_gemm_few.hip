// ss_gemm_few.hip - k_gemm_ks (ss_gemm.h) on matrices of up to 512 columns, with a
// wave per unit and matrix. A source of its own, so that a process loads these
// kernels' code (1.2 MB, 2 ms) when it first meets such a matrix and other
// prompts do not wait for it.

#include "ss_gemm.h"

namespace ssk {
namespace {

template <int QT, int NMAT, int EPI>
hipError_t launch_units(const GemmArgs& a, int nu, hipStream_t s) {
  const dim3 grid((a.rows + 31) / 32, (a.T + kSTok - 1) / kSTok);
  if (nu == 1)
    hipLaunchKernelGGL((k_gemm_ks<QT, NMAT, EPI, NMAT>), grid, dim3(NMAT * 64), 0, s, a, nu);
  else
    hipLaunchKernelGGL((k_gemm_ks<QT, NMAT, EPI, 2 * NMAT>), grid, dim3(2 * NMAT * 64), 0, s, a, nu);
  return hipGetLastError();
}
template <int QT>
hipError_t launch_epi(int epi, const GemmArgs& a, int nu, hipStream_t s) {
  switch (epi) {
    case EPI_STORE: return launch_units<QT, 1, EPI_STORE>(a, nu, s);
    case EPI_ADD: return launch_units<QT, 1, EPI_ADD>(a, nu, s);
    default: return launch_units<QT, 2, EPI_SWIGLU>(a, nu, s);
  }
}

}  // namespace

hipError_t launch_gemm_few(int epi, const GemmArgs& a, int nu, hipStream_t s) {
  switch (dev_type(a.type)) {
    case 2: return launch_epi<2>(epi, a, nu, s);
    case 8: return launch_epi<8>(epi, a, nu, s);
    case kQ4_1: return launch_epi<kQ4_1>(epi, a, nu, s);
    case kQ5_1: return launch_epi<kQ5_1>(epi, a, nu, s);
    case kQ8_1: return launch_epi<kQ8_1>(epi, a, nu, s);
    case kQ2K: return launch_epi<kQ2K>(epi, a, nu, s);
    case kQ3K: return launch_epi<kQ3K>(epi, a, nu, s);
    case kQ4K: return launch_epi<kQ4K>(epi, a, nu, s);
    case kQ5K: return launch_epi<kQ5K>(epi, a, nu, s);
    case kQ6K: return launch_epi<kQ6K>(epi, a, nu, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ssk
