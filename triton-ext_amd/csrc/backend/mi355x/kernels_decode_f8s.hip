// Tables of the 8-bit ring decode kernel (decode_f8.h): block-scaled fp8, int8, MX.
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

#define TX_DF8_SLICES(SC, FA, FB, BT, I8)                                                  \
  {decode_f8_kernel<16, SC, FA, FB, BT, I8>, decode_f8_kernel<32, SC, FA, FB, BT, I8>,     \
   decode_f8_kernel<48, SC, FA, FB, BT, I8>, decode_f8_kernel<64, SC, FA, FB, BT, I8>}
const DecodeF8KernelFn kDecodeF8ScaledKernels[2][4] = {TX_DF8_SLICES(true, 0, 0, false, false),
                                                       TX_DF8_SLICES(true, 0, 0, true, false)};
const DecodeF8KernelFn kDecodeI8KmajorKernels[4] = TX_DF8_SLICES(false, 0, 0, true, true);
#undef TX_DF8_SLICES
// MX operands: fp8 by [A e4m3 / e5m2][B e4m3 / e5m2][slice], and e2m1 by slice.
#define TX_DMX_SLICES(FA, FB)                                                              \
  {decode_f8_kernel<16, false, FA, FB, false, false, true>,                                \
   decode_f8_kernel<32, false, FA, FB, false, false, true>,                                \
   decode_f8_kernel<48, false, FA, FB, false, false, true>,                                \
   decode_f8_kernel<64, false, FA, FB, false, false, true>}
const DecodeF8KernelFn kDecodeMx8Kernels[2][2][4] = {
    {TX_DMX_SLICES(0, 0), TX_DMX_SLICES(0, 1)}, {TX_DMX_SLICES(1, 0), TX_DMX_SLICES(1, 1)}};
const DecodeF8KernelFn kDecodeMx4Kernels[4] = TX_DMX_SLICES(4, 4);
#undef TX_DMX_SLICES

} // namespace txk
