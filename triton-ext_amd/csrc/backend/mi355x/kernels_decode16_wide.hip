// Tables of the 16-bit decode kernel (decode16.h): strips of 128 columns.
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

// The 16-bit decode kernel with strips of 128 columns, slices of 16 .. 80 rows.
#define TX_D16W_SLICES(BF, BT)                                                                 \
  {decode16_kernel<16, BF, BT, 128>, decode16_kernel<32, BF, BT, 128>,                         \
   decode16_kernel<48, BF, BT, 128>, decode16_kernel<64, BF, BT, 128>,                         \
   decode16_kernel<80, BF, BT, 128>}
const Decode16KernelFn kDecode16WideKernels[2][2][kDec16WideMaxM / 16] = {
    {TX_D16W_SLICES(false, false), TX_D16W_SLICES(true, false)},
    {TX_D16W_SLICES(false, true), TX_D16W_SLICES(true, true)}};
#undef TX_D16W_SLICES

} // namespace txk
