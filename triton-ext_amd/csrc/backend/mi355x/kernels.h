// The backend's kernels as its launch layer sees them: every kernel header
// (argument structs, launch constants) and the tables of kernel instances,
// which kernels_*.hip define.
#pragma once

#include <hip/hip_runtime.h>

#include "attn_fwd.h"
#include "attn_fwd8.h"
#include "decode16.h"
#include "decode_f8.h"
#include "decode_i8.h"
#include "decode_rows_i8.h"
#include "gemm16_dma.h"
#include "gemm16_w4.h"
#include "gemm8_n224.h"
#include "gemm8_w4.h"
#include "gemm_ring.h"
#include "gemm_tile.h"
#include "mx_upcast.h"
#include "splitk_reduce.h"

namespace txk {

typedef void (*GemmKernelFn)(GemmArgs);

struct GemmConfig {
  int op, bm, bn, bk, wm, wn, epi;
  GemmKernelFn fn;
  int bt;        // B K-major (TX_FLAG_B_KMAJOR)
  int lds_bytes; // dynamic LDS (0 for kernels with static LDS)
  int dma;       // 0: register-staged (gemm_tile.h), 1: direct-to-LDS
                 // staging with 64-bit addresses (gemm16_dma.h), 2: 16-bit
                 // 256x256 tile (gemm16_w4.h), 5: 8-bit 256x256x128 and
                 // 256x224x128 tiles (gemm8_w4.h, gemm8_n224.h), 6: 128x128
                 // tiles on a deep ring (gemm_ring.h, kRingConfigs); 2, 5 and
                 // 6 address A and B through 32-bit buffer offsets
  int fmt;       // MX operand formats: MFMA code of A | code of B << 4
};

// Every (operands, tile, epilogue) instantiated, and the 128x128 ring tiles
// that serve 256x256 tile plans with TX_FLAG_TILES_128.
constexpr int kNumGemmConfigs = 52, kNumRingConfigs = 34;
extern const GemmConfig kGemmConfigs[kNumGemmConfigs];
extern const GemmConfig kRingConfigs[kNumRingConfigs];

// The kernels launched right before and after a tile, in the tiles' own unit
// (code object): the upcast of an MX operand by [B side][format e4m3, e5m2,
// e2m1, e2m1 with e4m3 scales], and the split-K reduction of 2, 4, 8, 16 ranges.
typedef void (*UpcastKernelFn)(UpcastArgs);
typedef void (*SplitReduceFn)(SplitReduceArgs);
extern const UpcastKernelFn kUpcastKernels[2][4];
extern const SplitReduceFn kSplitReduceKernels[4];

typedef void (*DecodeKernelFn)(DecodeArgs);
typedef void (*DecodeF8KernelFn)(DecodeF8Args);
typedef void (*Decode16KernelFn)(Decode16Args);
typedef void (*AttnFn)(AttnArgs);
extern const DecodeKernelFn kDecodeKernels[4];
extern const DecodeKernelFn kDecodeRowsKernels[2][3];
extern const DecodeF8KernelFn kDecodeF8Kernels[2][2][2][4];
extern const DecodeF8KernelFn kDecodeF8ScaledKernels[2][4];
extern const DecodeF8KernelFn kDecodeI8KmajorKernels[4];
extern const DecodeF8KernelFn kDecodeMx8Kernels[2][2][4];
extern const DecodeF8KernelFn kDecodeMx4Kernels[4];
extern const Decode16KernelFn kDecode16Kernels[2][2][kDec16MaxM / 16];
extern const Decode16KernelFn kDecode16WideKernels[2][2][kDec16WideMaxM / 16];
extern const Decode16KernelFn kDecodeWqKernels[4][kDec16MaxM / 16];
extern const AttnFn kAttn[2][5][2][2][2];
extern const AttnFn kAttn8[2][5][2][2];
// The same with 4 groups of waves that share 32 rows and split the keys:
// [causal][head_dim 16 / 32 / 64][bf16].
extern const AttnFn kAttnKs[2][3][2];

} // namespace txk
