// Tables of the 16-bit decode kernel (decode16.h): strips of 64 columns.
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

// The 16-bit decode kernel by [B K-major][bf16][slice rows / 16 - 1], slices
// of 16 .. 96 rows.
#define TX_D16_SLICES(BF, BT)                                                                  \
  {decode16_kernel<16, BF, BT>, decode16_kernel<32, BF, BT>, decode16_kernel<48, BF, BT>,      \
   decode16_kernel<64, BF, BT>, decode16_kernel<80, BF, BT>, decode16_kernel<96, BF, BT>}
const Decode16KernelFn kDecode16Kernels[2][2][kDec16MaxM / 16] = {
    {TX_D16_SLICES(false, false), TX_D16_SLICES(true, false)},
    {TX_D16_SLICES(false, true), TX_D16_SLICES(true, true)}};
#undef TX_D16_SLICES

} // namespace txk
