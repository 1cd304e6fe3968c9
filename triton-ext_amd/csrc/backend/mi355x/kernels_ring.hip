// Table of the 128x128 deep-ring tiles (gemm_ring.h).
// (One of the backend's translation units of kernels; kernels.h declares the
// tables, so that the units compile side by side.)

#include "kernels.h"

namespace txk {

// BK in elements: a ring step of 128 bytes of K.
#define TX_RING(OP, EPI, BK)                                                               \
  GemmConfig { OP, 128, 128, BK, 2, 4, EPI, gemm_ring_kernel<OP, EPI>, 0, 0, 6 }
#define TX_RINGT(OP, EPI, BK)                                                              \
  GemmConfig { OP, 128, 128, BK, 2, 4, EPI, gemm_ring_kernel<OP, EPI, 0, 0, true>, 1, 0, 6 }
#define TX_RINGF(EPI, FA, FB, BK)                                                          \
  GemmConfig {                                                                             \
    OP_F8, 128, 128, BK, 2, 4, EPI, gemm_ring_kernel<OP_F8, EPI, FA, FB>, 0, 0, 6,          \
        (FA) | ((FB) << 4)                                                                 \
  }
#define TX_RINGFT(FA, FB)                                                                  \
  GemmConfig {                                                                             \
    OP_F8, 128, 128, 128, 2, 4, EPI_F32, gemm_ring_kernel<OP_F8, EPI_F32, FA, FB, true>, 1, \
        0, 6, (FA) | ((FB) << 4)                                                           \
  }

const GemmConfig kRingConfigs[] = {
    TX_RING(OP_BF16, EPI_BF16, 64),
    TX_RING(OP_BF16, EPI_F32, 64),
    TX_RING(OP_F16, EPI_F16, 64),
    TX_RING(OP_F16, EPI_F32, 64),
    TX_RINGT(OP_BF16, EPI_BF16, 64),
    TX_RINGT(OP_BF16, EPI_F32, 64),
    TX_RINGT(OP_F16, EPI_F16, 64),
    TX_RINGT(OP_F16, EPI_F32, 64),
    TX_RING(OP_I8, EPI_I32, 128),
    TX_RING(OP_I8, EPI_ROWCOL_BF16, 128),
    TX_RINGT(OP_I8, EPI_I32, 128),
    TX_RINGT(OP_I8, EPI_ROWCOL_BF16, 128),
    TX_RING(OP_F8, EPI_BLOCK128_BF16, 128),
    TX_RING(OP_F8, EPI_BLOCK128_F32, 128),
    TX_RINGT(OP_F8, EPI_BLOCK128_BF16, 128),
    TX_RINGT(OP_F8, EPI_BLOCK128_F32, 128),
    TX_RINGF(EPI_F32, 0, 0, 128),
    TX_RINGF(EPI_F32, 0, 1, 128),
    TX_RINGF(EPI_F32, 1, 0, 128),
    TX_RINGF(EPI_F32, 1, 1, 128),
    TX_RINGFT(0, 0),
    TX_RINGFT(0, 1),
    TX_RINGFT(1, 0),
    TX_RINGFT(1, 1),
    TX_RINGF(EPI_MX_F32, 0, 0, 128),
    TX_RINGF(EPI_MX_F32, 0, 1, 128),
    TX_RINGF(EPI_MX_F32, 1, 0, 128),
    TX_RINGF(EPI_MX_F32, 1, 1, 128),
    TX_RINGF(EPI_MX_F32, 4, 4, 256),
    TX_RINGF(EPI_MX_BF16, 0, 0, 128),
    TX_RINGF(EPI_MX_BF16, 0, 1, 128),
    TX_RINGF(EPI_MX_BF16, 1, 0, 128),
    TX_RINGF(EPI_MX_BF16, 1, 1, 128),
    TX_RINGF(EPI_MX_BF16, 4, 4, 256),
};
static_assert(sizeof(kRingConfigs) / sizeof(kRingConfigs[0]) == kNumRingConfigs,
              "kernels.h states the table's length");

} // namespace txk
