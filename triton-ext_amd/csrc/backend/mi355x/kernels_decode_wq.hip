// Tables of the 16-bit decode kernel (decode16.h) with B upcast in registers.
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

// The 16-bit decode kernel with B upcast in registers, strips of 128 columns, slices of 16 ..
// 96 rows: B e2m1 / e4m3 / e5m2 under e8m0 scales, e2m1 under e4m3 scales.
#define TX_DWQ_SLICES(WQ)                                                                      \
  {decode16_kernel<16, true, false, 128, WQ>, decode16_kernel<32, true, false, 128, WQ>,       \
   decode16_kernel<48, true, false, 128, WQ>, decode16_kernel<64, true, false, 128, WQ>,       \
   decode16_kernel<80, true, false, 128, WQ>, decode16_kernel<96, true, false, 128, WQ>}
const Decode16KernelFn kDecodeWqKernels[4][kDec16MaxM / 16] = {
    TX_DWQ_SLICES(WQ_MX_E2M1), TX_DWQ_SLICES(WQ_MX_E4M3), TX_DWQ_SLICES(WQ_MX_E5M2),
    TX_DWQ_SLICES(WQ_NV_E2M1)};
#undef TX_DWQ_SLICES

} // namespace txk
