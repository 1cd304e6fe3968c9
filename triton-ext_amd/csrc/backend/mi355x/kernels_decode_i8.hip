// Tables of the W8A8 decode kernels (decode_i8.h, decode_rows_i8.h).
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

const DecodeKernelFn kDecodeKernels[4] = {decode_i8_kernel<1>, decode_i8_kernel<2>,
                                           decode_i8_kernel<3>, decode_i8_kernel<4>};
// The row-parallel decode kernel by slice height (64, 128, 256 rows): rings
// of 6, 4 and 3 slots of 24, 32 and 48 KiB (a 128-row batch: B's 16 KiB and
// the slice's A).
// [B K-major][slice of 64, 128, 256 rows]
const DecodeKernelFn kDecodeRowsKernels[2][3] = {
    {decode_rows_i8_kernel<64, 6>, decode_rows_i8_kernel<128, 4>, decode_rows_i8_kernel<256, 3>},
    {decode_rows_i8_kernel<64, 6, true>, decode_rows_i8_kernel<128, 4, true>,
     decode_rows_i8_kernel<256, 3, true>}};

} // namespace txk
