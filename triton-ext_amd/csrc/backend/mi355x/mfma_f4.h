// The fp4 form of gfx950's scaled MFMA, shared by the 256x256 tile and the
// 8-bit ring decode kernel.
#pragma once

#include "gemm_tile.h"

namespace txk {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

// The fp4 form of the scaled MFMA reads 4-dword operands: the intrinsic's
// v4i32 overload, called by its LLVM name (the clang builtin is declared for
// 8-dword operands only).
extern "C" __device__ f32x4_t txk_mfma_scale_16x16x128_f4(i32x4_t, i32x4_t, f32x4_t, int, int,
                                                          int, int, int, int)
    __asm("llvm.amdgcn.mfma.scale.f32.16x16x128.f8f6f4.v4i32.v4i32");

} // namespace txk
