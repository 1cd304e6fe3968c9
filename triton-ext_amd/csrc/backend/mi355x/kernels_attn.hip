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

#define TX_ATTN_KS(C, HD)                                                                   \
  {attn_fwd_ks_kernel<C, HD, false, 32, 4>, attn_fwd_ks_kernel<C, HD, true, 32, 4>}
const AttnFn kAttnKs[2][3][2] = {
    {TX_ATTN_KS(false, 16), TX_ATTN_KS(false, 32), TX_ATTN_KS(false, 64)},
    {TX_ATTN_KS(true, 16), TX_ATTN_KS(true, 32), TX_ATTN_KS(true, 64)}};
#undef TX_ATTN_KS

} // namespace txk
