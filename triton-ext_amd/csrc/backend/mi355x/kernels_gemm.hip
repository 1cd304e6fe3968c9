// Table of the GEMM tiles.
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

#define TX_GEMM(OP, BM, BN, BK, WM, WN, EPI)                                   \
  GemmConfig {                                                                 \
    OP, BM, BN, BK, WM, WN, EPI, gemm_tile_kernel<OP, BM, BN, BK, WM, WN, EPI>,\
        0, GemmTile<OP, BM, BN, BK, WM, WN, EPI>::LDS_BYTES, 0                 \
  }
#define TX_GEMM_DMA_S(OP, BM, BN, BK, WM, WN, ST, EPI)                         \
  GemmConfig {                                                                 \
    OP, BM, BN, BK, WM, WN, EPI,                                               \
        gemm16_dma_kernel<OP, BM, BN, BK, WM, WN, ST, EPI>, 0, 0, 1            \
  }
#define TX_GEMM_DMA(OP, BM, BN, BK, WM, WN, EPI)                               \
  TX_GEMM_DMA_S(OP, BM, BN, BK, WM, WN, 2, EPI)

#define TX_GEMM_W4(OP, EPI)                                                    \
  GemmConfig { OP, 256, 256, 64, 2, 2, EPI, gemm16_w4_kernel<OP, EPI, 4>, 0, 0, 2 }
#define TX_GEMM_W4T(OP, EPI)                                                   \
  GemmConfig { OP, 256, 256, 64, 2, 2, EPI, gemm16_w4_kernel<OP, EPI, 4, true>, 1, 0, 2 }
#define TX_GEMM_8(OP, EPI)                                                     \
  GemmConfig { OP, 256, 256, 128, 2, 4, EPI, gemm8_w4_kernel<OP, EPI>, 0, 0, 5 }
// MX (tl.dot_scaled) tiles: MFMA format codes FA, FB (0 e4m3, 1 e5m2,
// 4 e2m1); BK in elements (128 bytes of K per step).
#define TX_GEMM_MX(FA, FB, BK, EPI)                                            \
  GemmConfig {                                                                 \
    OP_F8, 256, 256, BK, 2, 4, EPI, gemm8_w4_kernel<OP_F8, EPI, FA, FB>, 0, 0, \
        5, (FA) | ((FB) << 4)                                                  \
  }
// Unscaled fp8 with e5m2 operands (MFMA format codes FA, FB; fp32 C).
#define TX_GEMM_8F(FA, FB)                                                     \
  GemmConfig {                                                                 \
    OP_F8, 256, 256, 128, 2, 4, EPI_F32, gemm8_w4_kernel<OP_F8, EPI_F32, FA, FB>, \
        0, 0, 5, (FA) | ((FB) << 4)                                            \
  }
// The same with B K-major (TX_FLAG_B_KMAJOR): every 8-bit epilogue but MX's.
#define TX_GEMM_8T(OP, EPI)                                                    \
  GemmConfig { OP, 256, 256, 128, 2, 4, EPI, gemm8_w4_kernel<OP, EPI, 0, 0, true>, 1, 0, 5 }
#define TX_GEMM_8FT(FA, FB)                                                    \
  GemmConfig {                                                                 \
    OP_F8, 256, 256, 128, 2, 4, EPI_F32, gemm8_w4_kernel<OP_F8, EPI_F32, FA, FB, true>, \
        1, 0, 5, (FA) | ((FB) << 4)                                            \
  }
#define TX_GEMM_8N(OP, EPI)                                                    \
  GemmConfig { OP, 256, 224, 128, 4, 2, EPI, gemm8_n224_kernel<OP, EPI>, 0, 0, 5 }

// Every (operands, tile, epilogue) instantiated; findGemmConfig takes the
// entry that matches a plan exactly.
const GemmConfig kGemmConfigs[] = {
    // bf16 / fp16 operands, 256x256x64 tiles of 4 waves
    TX_GEMM_W4(OP_BF16, EPI_BF16),
    TX_GEMM_W4(OP_BF16, EPI_F32),
    TX_GEMM_W4(OP_F16, EPI_F32),
    TX_GEMM_W4(OP_F16, EPI_F16),
    // the same with B K-major (TX_FLAG_B_KMAJOR)
    TX_GEMM_W4T(OP_BF16, EPI_BF16),
    TX_GEMM_W4T(OP_BF16, EPI_F32),
    TX_GEMM_W4T(OP_F16, EPI_F32),
    TX_GEMM_W4T(OP_F16, EPI_F16),
    // bf16 / fp16 operands, 128x128x64 tiles: direct-to-LDS staging, 64-bit
    // addresses (operands spanning 2 GiB or more); two stages, two
    // workgroups per CU (three or four stages leave one: 32.3 -> 25.6% of
    // peak at bf16 4096^3)
    TX_GEMM_DMA(OP_BF16, 128, 128, 64, 2, 2, EPI_BF16),
    TX_GEMM_DMA(OP_BF16, 128, 128, 64, 2, 2, EPI_F32),
    TX_GEMM_DMA(OP_F16, 128, 128, 64, 2, 2, EPI_F32),
    TX_GEMM_DMA(OP_F16, 128, 128, 64, 2, 2, EPI_F16),
    // 64x64x32 tiles (the reference's BLOCK of config 0): direct-to-LDS
    // staging, three stages (measured at fp16 512^3: 2 / 3 / 4 / 5 stages
    // 8.35 / 7.40 / 7.83 / 8.71 us; register staging 9.05 us)
    TX_GEMM_DMA_S(OP_BF16, 64, 64, 32, 2, 2, 3, EPI_BF16),
    TX_GEMM_DMA_S(OP_BF16, 64, 64, 32, 2, 2, 3, EPI_F32),
    TX_GEMM_DMA_S(OP_F16, 64, 64, 32, 2, 2, 3, EPI_F32),
    TX_GEMM_DMA_S(OP_F16, 64, 64, 32, 2, 2, 3, EPI_F16),
    // int8 / fp8 operands, 256x256x128 tiles of 8 waves (gemm8_w4.h)
    TX_GEMM_8(OP_I8, EPI_I32),
    TX_GEMM_8(OP_I8, EPI_ROWCOL_BF16),
    TX_GEMM_8(OP_F8, EPI_BLOCK128_BF16),
    TX_GEMM_8(OP_F8, EPI_BLOCK128_F32),
    TX_GEMM_8(OP_F8, EPI_F32),
    // fp8 tt.dot with e5m2 on either side (the tutorial's p . v with fp8e5 p)
    TX_GEMM_8F(1, 1),
    TX_GEMM_8F(0, 1),
    TX_GEMM_8F(1, 0),
    // the same with B K-major (q . k^T, or weights kept [out][in])
    TX_GEMM_8T(OP_I8, EPI_I32),
    TX_GEMM_8T(OP_I8, EPI_ROWCOL_BF16),
    TX_GEMM_8T(OP_F8, EPI_BLOCK128_BF16),
    TX_GEMM_8T(OP_F8, EPI_BLOCK128_F32),
    TX_GEMM_8T(OP_F8, EPI_F32),
    TX_GEMM_8FT(1, 1),
    TX_GEMM_8FT(0, 1),
    TX_GEMM_8FT(1, 0),
    // MX: e8m0-scaled fp8 (e4m3 / e5m2 in any mix) and fp4 (gemm8_w4.h)
    TX_GEMM_MX(0, 0, 128, EPI_MX_F32),
    TX_GEMM_MX(0, 0, 128, EPI_MX_BF16),
    TX_GEMM_MX(0, 1, 128, EPI_MX_F32),
    TX_GEMM_MX(0, 1, 128, EPI_MX_BF16),
    TX_GEMM_MX(1, 0, 128, EPI_MX_F32),
    TX_GEMM_MX(1, 0, 128, EPI_MX_BF16),
    TX_GEMM_MX(1, 1, 128, EPI_MX_F32),
    TX_GEMM_MX(1, 1, 128, EPI_MX_BF16),
    TX_GEMM_MX(4, 4, 256, EPI_MX_F32),
    TX_GEMM_MX(4, 4, 256, EPI_MX_BF16),
    // the same with 256x224 tiles (gemm8_n224.h)
    TX_GEMM_8N(OP_I8, EPI_I32),
    TX_GEMM_8N(OP_I8, EPI_ROWCOL_BF16),
    TX_GEMM_8N(OP_F8, EPI_BLOCK128_BF16),
    TX_GEMM_8N(OP_F8, EPI_BLOCK128_F32),
    TX_GEMM_8N(OP_F8, EPI_F32),
    // int8 operands, int32 accumulation, 128x128x128 register-staged tiles
    TX_GEMM(OP_I8, 128, 128, 128, 2, 2, EPI_I32),
    TX_GEMM(OP_I8, 128, 128, 128, 2, 2, EPI_ROWCOL_BF16),
    // fp8 e4m3 operands, fp32 accumulation, 128x128x128 register-staged tiles
    TX_GEMM(OP_F8, 128, 128, 128, 2, 2, EPI_BLOCK128_BF16),
    TX_GEMM(OP_F8, 128, 128, 128, 2, 2, EPI_BLOCK128_F32),
    TX_GEMM(OP_F8, 128, 128, 128, 2, 2, EPI_F32),
};
static_assert(sizeof(kGemmConfigs) / sizeof(kGemmConfigs[0]) == kNumGemmConfigs,
              "kernels.h states the table's length");

const UpcastKernelFn kUpcastKernels[2][4] = {
    {mx_upcast_a_kernel<0>, mx_upcast_a_kernel<1>, mx_upcast_a_kernel<4>,
     mx_upcast_a_kernel<4, true>},
    {mx_upcast_b_kernel<0>, mx_upcast_b_kernel<1>, mx_upcast_b_kernel<4>,
     mx_upcast_b_kernel<4, true>}};
const SplitReduceFn kSplitReduceKernels[4] = {splitk_reduce_kernel<2>, splitk_reduce_kernel<4>,
                                              splitk_reduce_kernel<8>, splitk_reduce_kernel<16>};

} // namespace txk
