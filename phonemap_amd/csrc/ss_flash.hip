// ss_flash.hip - launches of the prompt rows' attention (ss_flash.h): the shape
// rule, and the fp16 kernels of prompts of kFullRows tokens or more.

#include "ss_flash.h"

namespace ssk {
namespace {

constexpr int kFullRows = 8;   // fp16 launches of fewer tokens, and all int8 ones, sum in the FULL form

template <int HD, int RT, int KG, int DS = 1>
hipError_t launch_shape(int group, int kv_type, const AttnArgs& a, hipStream_t s) {
  if (kv_type || a.n_tok < kFullRows) return launch_flash_full(HD, RT, KG, group, kv_type, a, s);
  return launch_flash<HD, RT, KG, DS, false, false>(group, a, s);
}

}  // namespace

hipError_t launch_attention_rows(int head_dim, int group, int kv_type, const AttnArgs& a, hipStream_t s) {
  if (a.n_tok < 1 || a.n_kv_heads < 1 || a.max_seq < 1 || !a.q || !a.out || !a.kc || !a.vc ||
      (kv_type && (!a.ks || !a.vs)) || a.tok_q % 4 ||
      a.tok_o % 4 || a.n_cu <= 0)
    return hipErrorInvalidValue;
  // Up to 64 keys: two key groups, one step (32 heads x 32 tokens at head_dim
  // 128: 6.5 us, with four groups 7.8). More row tiles than compute units at
  // head_dim 128: two tiles share a workgroup's staging (512 tokens over 1536,
  // 32 heads on 8: 41 us against 55 with one; 77 tokens over 1000, 80 tiles:
  // 18 against 23 the other way round). head_dim 64 keeps one tile, as two
  // such workgroups fit a compute unit (2000 tokens, 8 heads: 22 against 24).
  // head_dim 256 has LDS for two key groups only.
  const bool two_blocks = (int64_t)a.pos0 + a.n_tok <= 2 * kBlk;
  const int64_t tiles = ((int64_t)a.n_tok * group + 31) / 32 * a.n_kv_heads;
  if (head_dim == 64) return two_blocks ? launch_shape<64, 1, 2>(group, kv_type, a, s) : launch_shape<64, 1, 4>(group, kv_type, a, s);
  if (head_dim == 128) {
    if (two_blocks) return launch_shape<128, 1, 2>(group, kv_type, a, s);
    return tiles > a.n_cu && (kv_type || a.n_tok >= kFullRows) ? launch_shape<128, 2, 4>(group, kv_type, a, s) : launch_shape<128, 1, 4>(group, kv_type, a, s);
  }
  if (head_dim == 256) return launch_shape<256, 1, 2, 2>(group, kv_type, a, s);   // Gemma
  return hipErrorInvalidValue;
}

}  // namespace ssk
