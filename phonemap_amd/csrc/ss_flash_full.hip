// ss_flash_full.hip - the prompt rows' attention in the FULL form (ss_flash.h):
// int8 caches, and fp16 prompts of few tokens. A source of its own, so that a
// process loads these kernels' code (0.9 MB, about 3 ms) when it first needs
// them and longer fp16 prompts do not wait for it.

#include "ss_flash.h"

namespace ssk {
namespace {

template <int HD, int RT, int KG, int DS = 1>
hipError_t launch_kv(int group, int kv_type, const AttnArgs& a, hipStream_t s) {
  return kv_type ? launch_flash<HD, RT, KG, DS, true, true>(group, a, s)
                 : launch_flash<HD, RT, KG, DS, false, true>(group, a, s);
}

}  // namespace

hipError_t launch_flash_full(int head_dim, int rt, int kg, int group, int kv_type, const AttnArgs& a, hipStream_t s) {
  if (head_dim == 64) return kg == 2 ? launch_kv<64, 1, 2>(group, kv_type, a, s) : launch_kv<64, 1, 4>(group, kv_type, a, s);
  if (head_dim == 256) return launch_kv<256, 1, 2, 2>(group, kv_type, a, s);
  if (kg == 2) return launch_kv<128, 1, 2>(group, kv_type, a, s);
  if (rt == 1) return launch_kv<128, 1, 4>(group, kv_type, a, s);
  return kv_type ? launch_flash<128, 2, 4, 1, true, true>(group, a, s) : hipErrorInvalidValue;
}

}  // namespace ssk
