// Table of the fp16 / bf16 attention forward (attn_fwd.h).
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

#define TX_ATTN_BLOCKS(C, HD, BF)                                                          \
{{attn_fwd_kernel<C, HD, BF, 128, 64>, attn_fwd_kernel<C, HD, BF, 128, 32>},    \
 {attn_fwd_kernel<C, HD, BF, 64, 64>, attn_fwd_kernel<C, HD, BF, 64, 32>}}
#define TX_ATTN_DTYPES(C, HD) {TX_ATTN_BLOCKS(C, HD, false), TX_ATTN_BLOCKS(C, HD, true)}
// [causal][head_dim 16 / 32 / 64 / 128 / 256][bf16][BLOCK_M 64][BLOCK_N 32]
const AttnFn kAttn[2][5][2][2][2] = {
    {TX_ATTN_DTYPES(false, 16), TX_ATTN_DTYPES(false, 32), TX_ATTN_DTYPES(false, 64),
     TX_ATTN_DTYPES(false, 128), TX_ATTN_DTYPES(false, 256)},
    {TX_ATTN_DTYPES(true, 16), TX_ATTN_DTYPES(true, 32), TX_ATTN_DTYPES(true, 64),
     TX_ATTN_DTYPES(true, 128), TX_ATTN_DTYPES(true, 256)}};
#undef TX_ATTN_DTYPES
#undef TX_ATTN_BLOCKS

// (head dim 128 has no 32 x 4: its slots would take 256 KiB)
#define TX_ATTN_KS(C, HD, BM, KS)                                                           \
  {attn_fwd_ks_kernel<C, HD, false, BM, KS>, attn_fwd_ks_kernel<C, HD, true, BM, KS>}
#define TX_ATTN_KSD(C, BM, KS)                                                              \
  {TX_ATTN_KS(C, 16, BM, KS), TX_ATTN_KS(C, 32, BM, KS), TX_ATTN_KS(C, 64, BM, KS),         \
   TX_ATTN_KS(C, 128, BM, KS)}
const AttnFn kAttnKs[3][2][4][2] = {
    {TX_ATTN_KSD(false, 128, 2), TX_ATTN_KSD(true, 128, 2)},
    {TX_ATTN_KSD(false, 64, 2), TX_ATTN_KSD(true, 64, 2)},
    {{TX_ATTN_KS(false, 16, 32, 4), TX_ATTN_KS(false, 32, 32, 4), TX_ATTN_KS(false, 64, 32, 4),
      {nullptr, nullptr}},
     {TX_ATTN_KS(true, 16, 32, 4), TX_ATTN_KS(true, 32, 32, 4), TX_ATTN_KS(true, 64, 32, 4),
      {nullptr, nullptr}}}};
#undef TX_ATTN_KSD
#undef TX_ATTN_KS

} // namespace txk
