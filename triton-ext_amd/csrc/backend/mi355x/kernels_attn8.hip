// Table of the e5m2 attention forward (attn_fwd8.h).
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

// [causal][head_dim 16 / 32 / 64 / 128 / 256][BLOCK_M 64][BLOCK_N 32]
#define TX_ATTN8_BLOCKS(C, HD)                                                             \
{{attn_fwd8_kernel<C, HD, 128, 64>, attn_fwd8_kernel<C, HD, 128, 32>},          \
 {attn_fwd8_kernel<C, HD, 64, 64>, attn_fwd8_kernel<C, HD, 64, 32>}}
const AttnFn kAttn8[2][5][2][2] = {
    {TX_ATTN8_BLOCKS(false, 16), TX_ATTN8_BLOCKS(false, 32), TX_ATTN8_BLOCKS(false, 64),
     TX_ATTN8_BLOCKS(false, 128), TX_ATTN8_BLOCKS(false, 256)},
    {TX_ATTN8_BLOCKS(true, 16), TX_ATTN8_BLOCKS(true, 32), TX_ATTN8_BLOCKS(true, 64),
     TX_ATTN8_BLOCKS(true, 128), TX_ATTN8_BLOCKS(true, 256)}};
#undef TX_ATTN8_BLOCKS

} // namespace txk
