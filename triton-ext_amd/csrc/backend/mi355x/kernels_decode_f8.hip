// Tables of the 8-bit ring decode kernel (decode_f8.h): unscaled fp8.
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

// The 8-bit ring decode kernel: unscaled fp8 by [B K-major][A e4m3 / e5m2]
// [B e4m3 / e5m2][slice of 16, 32, 48, 64 rows], block-scaled (e4m3) by
// [B K-major][slice], int8 with B K-major (int32 C or W8A8) by slice.
#define TX_DF8_SLICES(SC, FA, FB, BT, I8)                                                  \
  {decode_f8_kernel<16, SC, FA, FB, BT, I8>, decode_f8_kernel<32, SC, FA, FB, BT, I8>,     \
   decode_f8_kernel<48, SC, FA, FB, BT, I8>, decode_f8_kernel<64, SC, FA, FB, BT, I8>}
const DecodeF8KernelFn kDecodeF8Kernels[2][2][2][4] = {
    {{TX_DF8_SLICES(false, 0, 0, false, false), TX_DF8_SLICES(false, 0, 1, false, false)},
     {TX_DF8_SLICES(false, 1, 0, false, false), TX_DF8_SLICES(false, 1, 1, false, false)}},
    {{TX_DF8_SLICES(false, 0, 0, true, false), TX_DF8_SLICES(false, 0, 1, true, false)},
     {TX_DF8_SLICES(false, 1, 0, true, false), TX_DF8_SLICES(false, 1, 1, true, false)}}};
#undef TX_DF8_SLICES

} // namespace txk
