// bf16 / fp16 small-M dot (decode shape) for gfx950:
//   C[m][n] = sum_k A[m][k] * B[k][n]
// with A [M,K] (M <= 96) and B [K,N] row-major, both bf16 or both fp16,
// fp32 accumulation, and C in the operands' type (rounded to nearest even)
// or in fp32 (C = sum, or C += sum for tl.dot's acc).
//
// A dot with a few rows of A reads all of B once and does 2 M FLOPs per
// element of B, so it is HBM-bound; the GEMM tiles would leave most of a
// 64-row tile empty and cover N with a handful of workgroups.  Here a
// workgroup owns a strip of 64 columns (128-byte rows of B), the slice of
// SR = 16 ceil(M / 16) rows and a range of K (split-K), so strips x splits
// workgroups stream B once between them:
//  * B's batches of 128 K rows (16 KiB) go through one LDS ring shared by the
//    4 waves: each wave issues 4 of a batch's 16 direct-to-LDS loads
//    (non-temporal: each byte is read once), waits for its own loads
//    (s_waitcnt vmcnt) and one s_barrier per batch makes the whole batch
//    visible.  The same barrier tells every wave that the slot read one batch
//    earlier is free; the batch S - 1 ahead is loaded into it.
//  * A's rows of the batch (SR x 256 bytes) go into the same slot, a quarter
//    loaded by each wave, each load 4 whole rows; 16-byte chunk c of row r
//    sits at c ^ (r & 15), so the 16 rows one quarter-wave reads with
//    ds_read_b128 fall in 16 bank groups.
//  * B rows are N-contiguous and the MFMA wants K-contiguous elements per
//    column: ds_read_b64_tr_b16 transposes on the LDS read (within a 16-lane
//    group, lane L reads row L / 4, columns 4 (L % 4) .. +3 of a 16-column
//    block; lane i receives column i's 4 K-consecutive elements).  B's
//    16-byte chunk c of row r sits at c ^ (r & 7).
//  * Wave w owns columns 16 w .. 16 w + 15 of the strip for every row of the
//    slice (slices past 64 rows read tiles 4 .. T - 1 in a second block of
//    LDS reads), so every wave has MFMA work at any M:
//    v_mfma_f32_16x16x32_{bf16,f16} with the roles swapped (MFMA A := B
//    columns, MFMA B := A rows), so lane l holds row 16 t + l % 16 at the 4
//    consecutive columns 16 w + 4 (l / 16) .. +3.  No cross-wave reduction:
//    the waves own disjoint outputs.
//  * Split-K: decode_i8.h's exchange (SC1 stores of the fp32 partial, an
//    arrival counter per strip that the last arrival resets; the last
//    arrival gathers).  Partials are kept in lane order, 1 KiB per (wave,
//    row tile).  fp32 addition depends on order, so the last arrival adds
//    the splits' partials in split order 0, 1, .. (its own from registers at
//    its place): the result does not depend on which split arrives last.
//
// K loop in LoopSplit form: batches below k_main_batches load unmasked; the
// rest send B rows >= K, B chunks at or past N and A rows >= M to the
// zero-filled chunk.  An A chunk that crosses K is loaded whole and its
// elements past K are zeroed in registers (they would meet B's zero rows,
// but a row's padding may hold Inf or NaN, and Inf * 0 is NaN).
//
// BT: B stored K-major ([N][K] row-major, row stride ldb; q . k^T with k
// row-major, or a weight kept [out][in]).  A strip is then 64 rows of that
// storage, staged like A's rows (256 bytes of a batch each, chunk c of row r
// at c ^ (r & 15)), and the wave's fragment of columns 16 w .. 16 w + 15 is
// read with ds_read_b128 like an A tile: lane l gets column 16 w + l % 16 at
// K 8 (l / 16) .. +7 of the step, the K indices of the A fragment it meets.
// B's chunk that crosses K is loaded whole too, and zeroed in registers like
// A's.  Each strip starts its split's batches at its own batch (strip mod the
// split's batch count), so its fp32 sums can differ from the row-major form's
// in the last bits.
//
// W = 128: strips of 128 columns, for slices up to 80 rows (three slots of
// 32 KiB of B and the slice's A rows fit the LDS).  Every strip reads all of
// A, so A's re-reads are M / W of B's bytes, and wider strips halve them.
// The batch's B is stored as two 64-column halves in the layout above, and
// wave w owns 16-column blocks 2 w and 2 w + 1 (the second block's B
// fragments read in a block of their own); in K-major B, storage rows
// 32 w .. 32 w + 31.
//
// WQ: B in a microscaled format with bf16 A (tl.dot_scaled's weight-only
// form): e2m1 (packed rows [K/2][N]), e4m3 or e5m2 ([K][N]) with e8m0 scales
// per 32 K, or e2m1 with e4m3 scales per 16 K, scales [N][K / 32 or 16].
// Triton upcasts the scaled operand to bf16 and runs the bf16 dot; here each
// wave upcasts its B fragments in registers on the way to the MFMA (W = 128
// strips), so B is read once in its own bytes instead of being written to
// memory and read back as bf16.  The K order of the MFMAs is the plain
// kernel's, their fp32 sums run in two chains that take 4 batches (512 K) each in
// turn (halves of 5 to 7): up to 4 batches a split they are those of the bf16 dot of the upcast
// operand, and past it no less exact than those of the upcast and the bf16
// tile, which splits K further (bf16 x e4m3 22x6656x7296 against 64 bits: that
// 1.03e-7, one chain 1.36e-7, two 1.01e-7).  4 splits or more are added in halves
// (16 of bf16 x e2m1 16x704x8128: that 6.4e-8, one row 7.5e-8, halves 6.1e-8).
//  * B's batch is 128 K: 64 packed rows or 128 byte rows of 128 bytes, 16-byte
//    chunk c of row r at c ^ swz(r).  ds_read_b64_tr_b8 hands a lane 8 rows of
//    one column, and the 8 rows are the addressing lanes' choice: e2m1 takes
//    rows 4 G .. +3 of two K steps at once (a step is 16 packed rows, one
//    dword its 8 elements), fp8 rows 8 G .. +7 of one.
//  * Upcast: v_cvt_scalef32_pk_bf16_* converts pairs under one scale where
//    the scale exponent lies in [17, 239], where the product is exact; a batch
//    with another scale in any of the wave's lanes decodes to fp32 pairs
//    (exact, as is their ldexp short of overflow) and rounds once.  e4m3
//    scales (not powers of two) multiply the fp32 pair; the product is exact
//    in bf16.
//  * One wave a SIMD and little to load, so a batch's own serial chain bounds it
//    (bf16 x e2m1, 16 x 8192 x 16384: 0.87 us a batch of 128 K, of which its
//    loads are 0.15).  Hence one block of LDS reads and one wait a batch rather
//    than three, one branch for the upcast rather than one a fragment, load
//    addresses kept and advanced rather than worked out, and a loop that is not
//    unrolled by the ring (its code holds both upcasts): 0.55 us a batch.  M =
//    32, N = K = 8192: 23.9 -> 19.3 us (e2m1), 25.2 -> 19.9 (e4m3); with two
//    chains of sums 19.6 -> 19.4 (e2m1).
//  * Scales are staged per segment of 128 groups like decode_f8.h's MX form;
//    columns past N and groups past K take a unit scale (their codes are 0).
#pragma once

#include <type_traits>

#include "decode_i8.h"
#include "mx_upcast.h"

namespace txk {

// B's format in the 16-bit decode kernel: A's type, or microscaled (WQ).
enum { WQ_NONE = 0, WQ_MX_E2M1, WQ_MX_E4M3, WQ_MX_E5M2, WQ_NV_E2M1 };
#define tx_unit_scales TX_TU_CAT(tx_unit_scales, TX_TU)
__device__ uint32_t tx_unit_scales[2] = {0x7f7f7f7fu, 0x38383838u}; // e8m0 2^0; e4m3 1.0

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

constexpr int kDec16StripN = 64;                                   // columns: 128-byte rows
constexpr int kDec16WideMaxM = 80; // strips of 128 columns: slices up to 80 rows (3 slots)
constexpr int kDec16BatchK = 128;                                  // K rows a batch
constexpr int kDec16MaxM = 96;                                     // one slice of 96 rows
constexpr int64_t kDec16MaxStrips = kDecodeCounterBytes / 4;       // one counter per strip

struct Decode16Args {
  const uint16_t *A;
  const uint16_t *B;
  void *C;
  int32_t c_f32; // C is fp32 (else the operands' 16-bit type)
  int32_t acc_c; // fp32 C: add the sums to C's contents (tl.dot's acc)
  int32_t M, N, K;
  int64_t lda, ldb, ldc; // row strides in elements
  int32_t ksplit;
  int32_t batches_per_split;
  int32_t k_main_batches; // batches with every K row < K (unmasked)
  float *partials;        // [ksplit][strips][4 waves][SR / 16][64 lanes][4] fp32
  uint32_t *counters;     // [strips] arrival counters
  const uint8_t *sb;      // WQ: scales [N][sb_ld]
  int32_t sb_ld;
};

// Bytes of one split's partials: every strip's SR x W fp32 sums.
__host__ __device__ constexpr int64_t decode16_split_bytes(int64_t strips, int sr,
                                                           int w = kDec16StripN) {
  return strips * sr * w * 4;
}

template <int SR, int W = kDec16StripN, int WQ = WQ_NONE> struct Decode16Cfg {
  static_assert(W == 64 || W == 128, "strips of 64 or 128 columns");
  static constexpr bool FP4 = WQ == WQ_MX_E2M1 || WQ == WQ_NV_E2M1;
  // WQ: scale groups a batch, batches a segment, scale bytes staged
  static constexpr int GPB = WQ == WQ_NV_E2M1 ? 8 : 4, SEG_B = 128 / GPB;
  static constexpr int WQS_BYTES = WQ ? W * 35 * 4 : 0;
  static constexpr int T = SR / 16;                         // 16-row tiles
  static constexpr int JB = W / 64;                         // 16-column blocks a wave
  static constexpr int A_OFF = FP4 ? kDec16BatchK / 2 * W : WQ ? kDec16BatchK * W
                                                              : kDec16BatchK * 2 * W; // B's batch first
  static constexpr int SLOT = A_OFF + SR * kDec16BatchK * 2; // then SR rows of 256 bytes
  static constexpr int S_FIT = (158 * 1024 - WQS_BYTES) / SLOT;
  static constexpr int S = S_FIT > 8 ? 8 : S_FIT;
  static constexpr int B_LOADS = A_OFF / 1024 / kDecodeWaves;                  // 4 (W = 64)
  static constexpr int A_LOADS = SR * kDec16BatchK * 2 / 1024 / kDecodeWaves; // SR / 16
  static constexpr int VPB = B_LOADS + A_LOADS;
  static_assert(SR % 16 == 0 && SR >= 16 && SR <= kDec16MaxM, "slices of 16 .. 96 rows");
  static_assert(S >= 3 && (S - 2) * VPB <= 63, "ring depth; vmcnt is 6 bits");
  static_assert(!WQ || (W == 128 && (S - 1) * VPB + (W * 35 + 255) / 256 <= 63),
                "WQ: strips of 128 columns; vmcnt is 6 bits");
  // WQ: the chunk swizzle of B's row r: distinct over the 8 rows of a
  // transposed read (e2m1: rows r and r + 16 of 4 consecutive r)
  __device__ __forceinline__ static int swz(int r) {
    return FP4 ? (r & 3) | ((r >> 2) & 4) : r & 7;
  }
};

// Operands of two K steps (32 rows each, KS and KS + 1) of a batch: the
// wave's B fragments (two transposed reads a step, at `blo` / `bhi` and
// +4 KiB for the second step) and its T A fragments (ds_read_b128 at `a0` /
// `a1`, +4 KiB per 16-row tile), waiting for them before the block ends.
// Outputs are early-clobber: a read lands while later reads of the block
// still use their address registers.
#define TX_D16_TR                                                                           \
  "ds_read_b64_tr_b16 %0, %[blo]\n\tds_read_b64_tr_b16 %1, %[bhi]\n\t"                      \
  "ds_read_b64_tr_b16 %2, %[blo] offset:4096\n\tds_read_b64_tr_b16 %3, %[bhi] offset:4096\n\t"
#define TX_D16_OUT "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1])
#define TX_D16_IN [blo] "v"(blo), [bhi] "v"(bhi), [a0] "v"(a0), [a1] "v"(a1)
template <int T>
__device__ __forceinline__ void dec16_read_pair(uint32_t blo, uint32_t bhi, uint32_t a0,
                                                uint32_t a1, v2i_t (&lo)[2], v2i_t (&hi)[2],
                                                i32x4_t (&a)[2][T]) {
  if constexpr (T == 1)
    asm volatile(TX_D16_TR "ds_read_b128 %4, %[a0]\n\tds_read_b128 %5, %[a1]\n\t"
                           "s_waitcnt lgkmcnt(0)"
                 : TX_D16_OUT, "=&v"(a[0][0]), "=&v"(a[1][0])
                 : TX_D16_IN
                 : "memory");
  else if constexpr (T == 2)
    asm volatile(TX_D16_TR "ds_read_b128 %4, %[a0]\n\tds_read_b128 %5, %[a0] offset:4096\n\t"
                           "ds_read_b128 %6, %[a1]\n\tds_read_b128 %7, %[a1] offset:4096\n\t"
                           "s_waitcnt lgkmcnt(0)"
                 : TX_D16_OUT, "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1])
                 : TX_D16_IN
                 : "memory");
  else if constexpr (T == 3)
    asm volatile(TX_D16_TR "ds_read_b128 %4, %[a0]\n\tds_read_b128 %5, %[a0] offset:4096\n\t"
                           "ds_read_b128 %6, %[a0] offset:8192\n\t"
                           "ds_read_b128 %7, %[a1]\n\tds_read_b128 %8, %[a1] offset:4096\n\t"
                           "ds_read_b128 %9, %[a1] offset:8192\n\t"
                           "s_waitcnt lgkmcnt(0)"
                 : TX_D16_OUT, "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[1][0]),
                   "=&v"(a[1][1]), "=&v"(a[1][2])
                 : TX_D16_IN
                 : "memory");
  else
    asm volatile(TX_D16_TR "ds_read_b128 %4, %[a0]\n\tds_read_b128 %5, %[a0] offset:4096\n\t"
                           "ds_read_b128 %6, %[a0] offset:8192\n\t"
                           "ds_read_b128 %7, %[a0] offset:12288\n\t"
                           "ds_read_b128 %8, %[a1]\n\tds_read_b128 %9, %[a1] offset:4096\n\t"
                           "ds_read_b128 %10, %[a1] offset:8192\n\t"
                           "ds_read_b128 %11, %[a1] offset:12288\n\t"
                           "s_waitcnt lgkmcnt(0)"
                 : TX_D16_OUT, "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]),
                   "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[1][2]), "=&v"(a[1][3])
                 : TX_D16_IN
                 : "memory");
}
#undef TX_D16_IN
#undef TX_D16_OUT
#undef TX_D16_TR

// The same with B K-major: two K steps' B fragments (ds_read_b128 at `b0` /
// `b1`) and the T A fragments of each.
#define TX_D16K_T(t, off)                                                                  \
  "ds_read_b128 %[x0" #t "], %[a0] offset:" #off "\n\tds_read_b128 %[x1" #t "], %[a1] offset:" #off \
  "\n\t"
#define TX_D16K_O(t) [x0##t] "=&v"(a[0][t]), [x1##t] "=&v"(a[1][t])
#define TX_D16K_HEAD "ds_read_b128 %[y0], %[b0]\n\tds_read_b128 %[y1], %[b1]\n\t"
#define TX_D16K_BO [y0] "=&v"(bq[0]), [y1] "=&v"(bq[1])
#define TX_D16K_IN [b0] "v"(b0), [b1] "v"(b1), [a0] "v"(a0), [a1] "v"(a1)
template <int T>
__device__ __forceinline__ void dec16_read_pair_kmajor(uint32_t b0, uint32_t b1, uint32_t a0,
                                                       uint32_t a1, i32x4_t (&bq)[2],
                                                       i32x4_t (&a)[2][T]) {
  if constexpr (T == 1)
    asm volatile(TX_D16K_HEAD TX_D16K_T(0, 0) "s_waitcnt lgkmcnt(0)"
                 : TX_D16K_BO, TX_D16K_O(0)
                 : TX_D16K_IN
                 : "memory");
  else if constexpr (T == 2)
    asm volatile(TX_D16K_HEAD TX_D16K_T(0, 0) TX_D16K_T(1, 4096) "s_waitcnt lgkmcnt(0)"
                 : TX_D16K_BO, TX_D16K_O(0), TX_D16K_O(1)
                 : TX_D16K_IN
                 : "memory");
  else if constexpr (T == 3)
    asm volatile(TX_D16K_HEAD TX_D16K_T(0, 0) TX_D16K_T(1, 4096) TX_D16K_T(2, 8192)
                 "s_waitcnt lgkmcnt(0)"
                 : TX_D16K_BO, TX_D16K_O(0), TX_D16K_O(1), TX_D16K_O(2)
                 : TX_D16K_IN
                 : "memory");
  else
    asm volatile(TX_D16K_HEAD TX_D16K_T(0, 0) TX_D16K_T(1, 4096) TX_D16K_T(2, 8192)
                 TX_D16K_T(3, 12288) "s_waitcnt lgkmcnt(0)"
                 : TX_D16K_BO, TX_D16K_O(0), TX_D16K_O(1), TX_D16K_O(2), TX_D16K_O(3)
                 : TX_D16K_IN
                 : "memory");
}
#undef TX_D16K_IN
#undef TX_D16K_BO
#undef TX_D16K_HEAD
#undef TX_D16K_O
#undef TX_D16K_T

// The A fragments of row tiles 4 .. 4 + N - 1 of two K steps (slices past 64
// rows): ds_read_b128 at a0 / a1 + 16 KiB, +4 KiB per tile.
#define TX_D16M_T(t, off)                                                                  \
  "ds_read_b128 %[p0" #t "], %[a0] offset:" #off "\n\tds_read_b128 %[p1" #t "], %[a1] offset:" #off \
  "\n\t"
#define TX_D16M_O(t) [p0##t] "=&v"(x[0][t]), [p1##t] "=&v"(x[1][t])
#define TX_D16M_IN [a0] "v"(a0), [a1] "v"(a1)
template <int N>
__device__ __forceinline__ void dec16_read_more(uint32_t a0, uint32_t a1, i32x4_t (&x)[2][N]) {
  if constexpr (N == 1)
    asm volatile(TX_D16M_T(0, 16384) "s_waitcnt lgkmcnt(0)" : TX_D16M_O(0) : TX_D16M_IN : "memory");
  else if constexpr (N == 2)
    asm volatile(TX_D16M_T(0, 16384) TX_D16M_T(1, 20480) "s_waitcnt lgkmcnt(0)"
                 : TX_D16M_O(0), TX_D16M_O(1)
                 : TX_D16M_IN
                 : "memory");
  else if constexpr (N == 3)
    asm volatile(TX_D16M_T(0, 16384) TX_D16M_T(1, 20480) TX_D16M_T(2, 24576)
                 "s_waitcnt lgkmcnt(0)"
                 : TX_D16M_O(0), TX_D16M_O(1), TX_D16M_O(2)
                 : TX_D16M_IN
                 : "memory");
  else
    asm volatile(TX_D16M_T(0, 16384) TX_D16M_T(1, 20480) TX_D16M_T(2, 24576)
                 TX_D16M_T(3, 28672) "s_waitcnt lgkmcnt(0)"
                 : TX_D16M_O(0), TX_D16M_O(1), TX_D16M_O(2), TX_D16M_O(3)
                 : TX_D16M_IN
                 : "memory");
}
#undef TX_D16M_IN
#undef TX_D16M_O
#undef TX_D16M_T

template <bool BF>
__device__ __forceinline__ f32x4_t mfma16x16x32(const i32x4_t &a, const i32x4_t &b,
                                                const f32x4_t &c) {
  if constexpr (BF) {
    typedef __bf16 v8_t __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8_t, a),
                                                   __builtin_bit_cast(v8_t, b), c, 0, 0, 0);
  } else {
    typedef _Float16 v8_t __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8_t, a),
                                                  __builtin_bit_cast(v8_t, b), c, 0, 0, 0);
  }
}

// Zero the 16-bit elements of a fragment at K index `k` .. k + 7 that lie at
// or past K (the chunk that crosses K, in the tail batch).
__device__ __forceinline__ i32x4_t dec16_mask_k(const i32x4_t &v, int64_t k, int64_t K) {
  const int w[4] = {v[0], v[1], v[2], v[3]};
  int o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t lo = k + 2 * i < K ? 0xffffu : 0u;
    const uint32_t hi = k + 2 * i + 1 < K ? 0xffff0000u : 0u;
    o[i] = (int)((uint32_t)w[i] & (lo | hi));
  }
  return i32x4_t{o[0], o[1], o[2], o[3]};
}

// B-only reads of two K steps for a wave's second column block (strips of
// 128 columns): row-major, transposed reads at blo / bhi and +4 KiB;
// K-major, ds_read_b128 at b0 / b1.
__device__ __forceinline__ void dec16_read_b_pair(uint32_t blo, uint32_t bhi, v2i_t (&lo)[2],
                                                  v2i_t (&hi)[2]) {
  asm volatile("ds_read_b64_tr_b16 %0, %[blo]\n\tds_read_b64_tr_b16 %1, %[bhi]\n\t"
               "ds_read_b64_tr_b16 %2, %[blo] offset:4096\n\t"
               "ds_read_b64_tr_b16 %3, %[bhi] offset:4096\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1])
               : [blo] "v"(blo), [bhi] "v"(bhi)
               : "memory");
}
__device__ __forceinline__ void dec16_read_bk_pair(uint32_t b0, uint32_t b1, i32x4_t (&bq)[2]) {
  asm volatile("ds_read_b128 %0, %[b0]\n\tds_read_b128 %1, %[b1]\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(bq[0]), "=&v"(bq[1])
               : [b0] "v"(b0), [b1] "v"(b1)
               : "memory");
}

// WQ: a batch's operands of up to 4 row tiles in one block of LDS reads: both
// column blocks' staged scale dwords (three from an aligned address, of which
// the batch's bytes are cut at the row's misalignment), their NB transposed
// reads of B (e2m1: 2, both steps' dwords in one; fp8: 4, one a step; 4 KiB
// apart) and the T row tiles of A of the 4 K steps.
#define TX_DWQ_S                                                                           \
  "ds_read2_b32 %[p0], %[s0] offset0:0 offset1:1\n\tds_read2_b32 %[p1], %[s1] offset0:0 offset1:1\n\t" \
  "ds_read_b32 %[r0], %[s0] offset:8\n\tds_read_b32 %[r1], %[s1] offset:8\n\t"
#define TX_DWQ_B(h, off)                                                                   \
  "ds_read_b64_tr_b8 %[y0" #h "], %[b0] offset:" #off "\n\tds_read_b64_tr_b8 %[y1" #h            \
  "], %[b1] offset:" #off "\n\t"
#define TX_DWQ_A(t, off)                                                                   \
  "ds_read_b128 %[x0" #t "], %[a0] offset:" #off "\n\tds_read_b128 %[x1" #t "], %[a1] offset:" #off \
  "\n\tds_read_b128 %[x2" #t "], %[a2] offset:" #off "\n\tds_read_b128 %[x3" #t                \
  "], %[a3] offset:" #off "\n\t"
#define TX_DWQ_BO(h) [y0##h] "=&v"(bq[0][h]), [y1##h] "=&v"(bq[1][h])
#define TX_DWQ_AO(t)                                                                       \
  [x0##t] "=&v"(a[0][t]), [x1##t] "=&v"(a[1][t]), [x2##t] "=&v"(a[2][t]), [x3##t] "=&v"(a[3][t])
#define TX_DWQ_ASM(B, BO, A, ...)                                                          \
  asm volatile(TX_DWQ_S B A "s_waitcnt lgkmcnt(0)"                                          \
               : [p0] "=&v"(p0), [p1] "=&v"(p1), [r0] "=&v"(v[0][2]), [r1] "=&v"(v[1][2]), BO, \
                 __VA_ARGS__                                                               \
               : [s0] "v"(s0), [s1] "v"(s1), [b0] "v"(b0), [b1] "v"(b1), [a0] "v"(a0),       \
                 [a1] "v"(a1), [a2] "v"(a2), [a3] "v"(a3)                                   \
               : "memory")
#define TX_DWQ_T(B, BO)                                                                    \
  if constexpr (T == 1)                                                                    \
    TX_DWQ_ASM(B, TX_DWQ_C(BO), TX_DWQ_A(0, 0), TX_DWQ_AO(0));                              \
  else if constexpr (T == 2)                                                               \
    TX_DWQ_ASM(B, TX_DWQ_C(BO), TX_DWQ_A(0, 0) TX_DWQ_A(1, 4096), TX_DWQ_AO(0), TX_DWQ_AO(1)); \
  else if constexpr (T == 3)                                                               \
    TX_DWQ_ASM(B, TX_DWQ_C(BO), TX_DWQ_A(0, 0) TX_DWQ_A(1, 4096) TX_DWQ_A(2, 8192),         \
               TX_DWQ_AO(0), TX_DWQ_AO(1), TX_DWQ_AO(2));                                   \
  else                                                                                     \
    TX_DWQ_ASM(B, TX_DWQ_C(BO),                                                             \
               TX_DWQ_A(0, 0) TX_DWQ_A(1, 4096) TX_DWQ_A(2, 8192) TX_DWQ_A(3, 12288),       \
               TX_DWQ_AO(0), TX_DWQ_AO(1), TX_DWQ_AO(2), TX_DWQ_AO(3))
#define TX_DWQ_BO2 TX_DWQ_BO(0), TX_DWQ_BO(1)
#define TX_DWQ_BO4 TX_DWQ_BO2, TX_DWQ_BO(2), TX_DWQ_BO(3)
template <int T, int NB>
__device__ __forceinline__ void decwq_read(uint32_t s0, uint32_t s1, uint32_t b0, uint32_t b1,
                                           uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3,
                                           uint32_t (&v)[2][3], v2i_t (&bq)[2][NB],
                                           i32x4_t (&a)[4][T]) {
  v2i_t p0, p1;
  if constexpr (NB == 2) {
#define TX_DWQ_C(x) TX_DWQ_BO2
    TX_DWQ_T(TX_DWQ_B(0, 0) TX_DWQ_B(1, 4096), 0);
#undef TX_DWQ_C
  } else {
#define TX_DWQ_C(x) TX_DWQ_BO4
    TX_DWQ_T(TX_DWQ_B(0, 0) TX_DWQ_B(1, 4096) TX_DWQ_B(2, 8192) TX_DWQ_B(3, 12288), 0);
#undef TX_DWQ_C
  }
  v[0][0] = p0.x, v[0][1] = p0.y;
  v[1][0] = p1.x, v[1][1] = p1.y;
}
#undef TX_DWQ_S
#undef TX_DWQ_B
#undef TX_DWQ_A
#undef TX_DWQ_BO
#undef TX_DWQ_AO
#undef TX_DWQ_ASM
#undef TX_DWQ_T
#undef TX_DWQ_BO2
#undef TX_DWQ_BO4

// Elements 2 i and 2 i + 1 of 8 codes of a column (e2m1: a dword; fp8: two) in fp32.
typedef float f32x2_t __attribute__((ext_vector_type(2)));
template <int FMT, int I> __device__ __forceinline__ f32x2_t decwq_pair(uint32_t w0, uint32_t w1) {
  if constexpr (FMT == 4)
    return __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w0, 1.0f, I);
  else if constexpr (FMT == 1)
    return __builtin_amdgcn_cvt_scalef32_pk_f32_bf8(I < 2 ? w0 : w1, 1.0f, (I & 1) != 0);
  else
    return __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(I < 2 ? w0 : w1, 1.0f, (I & 1) != 0);
}

// One MFMA operand of B: 8 codes under one scale byte, as 8 bf16.  HW: the
// scale lies in the pair conversion's exact range (MX).
template <int WQ, bool HW>
__device__ __forceinline__ i32x4_t decwq_upcast(uint32_t w0, uint32_t w1, uint32_t s) {
  constexpr int FMT = WQ == WQ_MX_E4M3 ? 0 : WQ == WQ_MX_E5M2 ? 1 : 4;
  if constexpr (WQ != WQ_NV_E2M1 && HW) {
    const float f = __builtin_bit_cast(float, s << 23);
    if constexpr (FMT == 4)
      return i32x4_t{(int)mx_cvt_pair<4, 0>(w0, f), (int)mx_cvt_pair<4, 1>(w0, f),
                     (int)mx_cvt_pair<4, 2>(w0, f), (int)mx_cvt_pair<4, 3>(w0, f)};
    else
      return i32x4_t{(int)mx_cvt_pair<FMT, 0>(w0, f), (int)mx_cvt_pair<FMT, 1>(w0, f),
                     (int)mx_cvt_pair<FMT, 0>(w1, f), (int)mx_cvt_pair<FMT, 1>(w1, f)};
  } else {
    const float f = __builtin_amdgcn_cvt_f32_fp8((int)s, 0); // NV: the e4m3 scale
    auto pair = [&](f32x2_t v) {
      if constexpr (WQ == WQ_NV_E2M1)
        return (int)pk_bf16_rne(v.x * f, v.y * f);
      const float x = __builtin_amdgcn_ldexpf(v.x, (int)s - 127);
      const float y = __builtin_amdgcn_ldexpf(v.y, (int)s - 127);
      const float nan = __builtin_nanf("");
      return (int)pk_bf16_rne(s == 255 ? nan : x, s == 255 ? nan : y);
    };
    return i32x4_t{pair(decwq_pair<FMT, 0>(w0, w1)), pair(decwq_pair<FMT, 1>(w0, w1)),
                   pair(decwq_pair<FMT, 2>(w0, w1)), pair(decwq_pair<FMT, 3>(w0, w1))};
  }
}

template <int SR, bool BF, bool BT = false, int W = kDec16StripN, int WQ = WQ_NONE>
__global__ void __launch_bounds__(kDecodeWaves * 64, 1) decode16_kernel(Decode16Args p) {
  static_assert(!WQ || (BF && !BT && W == 128), "WQ: bf16 A, row-major B, strips of 128");
  typedef Decode16Cfg<SR, W, WQ> Cfg;
  constexpr int S = Cfg::S, SLOT = Cfg::SLOT, T = Cfg::T, JB = Cfg::JB;
  __shared__ __attribute__((aligned(1024))) uint8_t ring[S * SLOT];
  __shared__ uint32_t last_flag;
  __shared__ __attribute__((aligned(256))) uint8_t wqs[WQ ? (Cfg::WQS_BYTES + 255) / 256 * 256 : 4];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = lane >> 4, L = lane & 15;
  // Workgroup -> (strip, split): consecutive workgroups are adjacent strips
  // of one split, so the workgroups running at once read whole stretches of
  // B's rows.
  const int strips = (p.N + W - 1) / W;
  const int strip = blockIdx.x % strips, split = blockIdx.x / strips;
  const int64_t n0 = (int64_t)strip * W;
  const bool n_edge = n0 + W > p.N;

  const int total_batches = (p.K + kDec16BatchK - 1) / kDec16BatchK;
  const int b_begin = split * p.batches_per_split;
  int b_end = b_begin + p.batches_per_split;
  if (b_end > total_batches)
    b_end = total_batches;
  const int nb = b_end > b_begin ? b_end - b_begin : 0; // the same for every wave
  // K-major B: each strip walks its split's batches from its own starting
  // batch (strip mod nb), so the workgroups running at once read rows of B's
  // storage at different K offsets, not all at one offset of rows ldb apart.
  const int rot = BT && nb > 0 ? strip % nb : 0;
  auto batch = [&](int i) { // the split's i-th batch to run (i < nb)
    if constexpr (!BT)
      return b_begin + i;
    const int j = i + rot;
    return b_begin + (j >= nb ? j - nb : j);
  };

  // Loads of the split's batch i into `slot`: B rows 32 wave .. +31 of the
  // batch (load u: rows 8 q .. 8 q + 7, q = 4 wave + u, lane l' fetching
  // chunk (l' % 8) ^ (row & 7) of row 8 q + l' / 8; K-major B: storage rows
  // n0 + 4 q .. +3, lane l' fetching chunk (l' % 16) ^ (row & 15) of row
  // 4 q + l' / 16, as for A) and A rows 4 q .. 4 q + 3 (q = A_LOADS wave + u,
  // lane l' fetching chunk (l' % 16) ^ (row & 15) of row 4 q + l' / 16).  No loaded VGPR is live across the loop (with
  // direct-to-LDS loads pending the compiler could only wait for one with
  // vmcnt(0)).  For i >= nb every load reads the zero chunk, so each step
  // issues the same loads.
  auto issue = [&](int i, uint8_t *slot) {
    const bool live = i < nb;
    const int b = live ? batch(i) : b_begin + i;
    const int64_t k0 = (int64_t)b * kDec16BatchK;
    const bool mask = !live || n_edge || b >= p.k_main_batches;
#pragma unroll
    for (int u = 0; u < Cfg::B_LOADS; ++u) {
      const int q = Cfg::B_LOADS * wave + u;
      const void *src;
      if constexpr (BT) {
        const int r = 4 * q + (lane >> 4);
        const int c = (lane & 15) ^ (r & 15);
        const int64_t n = n0 + r, k = k0 + 8 * c;
        src = p.B + n * p.ldb + k;
        if (mask && (!live || n >= p.N || k >= p.K))
          src = tx_zero_chunk;
      } else {
        // Strips of 128 columns: load q >= 16 fills the second 16 KiB, the
        // batch's columns 64 .. 127 in the same layout.
        const int row = 8 * (q & 15) + (lane >> 3);
        const int c = (lane & 7) ^ (row & 7);
        const int64_t k = k0 + row, n = n0 + 64 * (q >> 4) + 8 * c;
        src = p.B + k * p.ldb + n;
        if (mask && (!live || k >= p.K || n >= p.N))
          src = tx_zero_chunk;
      }
      dma16_stream(src, (lds_void *)(slot + q * 1024)); // B is read once
    }
#pragma unroll
    for (int u = 0; u < Cfg::A_LOADS; ++u) {
      const int q = Cfg::A_LOADS * wave + u;
      const int r = 4 * q + (lane >> 4);
      const int c = (lane & 15) ^ (r & 15);
      const int64_t k = k0 + 8 * c;
      const void *src = p.A + (int64_t)r * p.lda + k;
      if (!live || r >= p.M || (b >= p.k_main_batches && k >= p.K))
        src = tx_zero_chunk;
      dma16(src, (lds_void *)(slot + Cfg::A_OFF + q * 1024)); // A: re-read by every strip
    }
  };

  f32x4_t acc[JB][T]; // [column block][row tile]
#pragma unroll
  for (int jj = 0; jj < JB; ++jj)
#pragma unroll
    for (int t = 0; t < T; ++t)
      acc[jj][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // Per-lane LDS offsets within a slot.  B, K step ks: rows 32 ks + 8 G +
  // L / 4 (lo) and +4 (hi), columns 16 wave + 4 (L % 4) .. +3, i.e. chunk
  // 2 wave + (L % 4) / 2, byte 8 (L % 2); the swizzle takes row & 7, which
  // is L / 4 for lo and L / 4 + 4 for hi in every step, so a step is +4 KiB.
  // A, step ks, tile t: row 16 t + L, chunk (4 ks + G) ^ L: +4 KiB per tile.
  // Column block jj of the wave is block J = JB wave + jj of the strip: in
  // row-major B, the 16 KiB half J / 4 and there block J % 4.
  uint32_t b_lo[JB], b_hi[JB];
#pragma unroll
  for (int jj = 0; jj < JB; ++jj) {
    const int J = JB * wave + jj;
    const int cb = 2 * (J & 3) + ((L & 3) >> 1);
    b_lo[jj] = (J >> 2) * 16384 + (L >> 2) * 128 + ((cb ^ (L >> 2)) << 4) + 8 * (L & 1) +
               8 * G * 128;
    b_hi[jj] = b_lo[jj] + 4 * 128 - ((cb ^ (L >> 2)) << 4) + ((cb ^ ((L >> 2) + 4)) << 4);
  }
  // K-major B, step ks: storage row 16 J + L, chunk (4 ks + G) ^ L.
  uint32_t a_k[4], bk_k[JB][4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    a_k[ks] = Cfg::A_OFF + L * 256 + (((4 * ks + G) ^ L) << 4);
#pragma unroll
    for (int jj = 0; jj < JB; ++jj)
      bk_k[jj][ks] = (16 * (JB * wave + jj) + L) * 256 + (((4 * ks + G) ^ L) << 4);
  }

  // WQ: a segment's scales of the strip's columns, `pitch` dwords a column from
  // its first byte rounded down (decode_f8.h's MX form).
  const int seg_groups = (nb < Cfg::SEG_B ? nb : Cfg::SEG_B) * Cfg::GPB;
  const int pitch = WQ ? ((seg_groups + 3 + 3) / 4 + 1) | 1 : 1; // <= 35: the last read's third dword
  auto stage_scales = [&](int i0) {
    const int64_t g0 = (int64_t)(b_begin + i0) * Cfg::GPB;
    const int items = W * pitch;
    const int64_t bytes = ((int64_t)p.N * p.sb_ld + 3) & ~3ll;
    for (int q0 = 64 * wave; q0 < items; q0 += 64 * kDecodeWaves) {
      const int q = q0 + lane, r = q / pitch, dw = q - r * pitch;
      const int64_t at = (((n0 + r) * p.sb_ld + g0) & ~3ll) + 4 * dw;
      const void *src = p.sb + at;
      // (whole dwords: each holds at least one byte of the array)
      if (q >= items || n0 + r >= p.N || at >= bytes)
        src = &tx_unit_scales[WQ == WQ_NV_E2M1];
      __builtin_amdgcn_global_load_lds(src, (lds_void *)(wqs + 4 * q0), 4, 0, 0);
    }
  };
  // This lane's column of each block: its staged row and misalignment, and its
  // first transposed read (a K step pair is +4 KiB, fp8 +8 KiB).
  uint32_t xs[2] = {0, 0}, mis[2] = {0, 0}, wq_b[2] = {0, 0};
  if constexpr (WQ != WQ_NONE) {
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      const int J = 2 * wave + jj, r = L >> 1;
      xs[jj] = lds_addr(wqs) + 4u * (uint32_t)((16 * J + L) * pitch);
      mis[jj] = ((uint32_t)(n0 + 16 * J + L) * (uint32_t)p.sb_ld) & 3u; // (g0 is a multiple of 4)
      const int row = Cfg::FP4 ? 4 * G + (r & 3) + 16 * (r >> 2) : 8 * G + r;
      wq_b[jj] = row * 128 + ((J ^ Cfg::swz(row)) << 4) + 8 * (L & 1);
    }
  }

  auto consume = [&](const uint8_t *slot, int i) {
    const uint32_t base = lds_addr(slot);
    const int b = batch(i);
    const bool tail = b >= p.k_main_batches;
    const int64_t k0 = (int64_t)b * kDec16BatchK;
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
      constexpr int T4 = T < 4 ? T : 4; // tiles the first read block brings
      i32x4_t bq[JB][2];
      i32x4_t a4[2][T4];
      if constexpr (BT) {
        dec16_read_pair_kmajor<T4>(base + bk_k[0][2 * pr], base + bk_k[0][2 * pr + 1],
                                   base + a_k[2 * pr], base + a_k[2 * pr + 1], bq[0], a4);
        if constexpr (JB == 2)
          dec16_read_bk_pair(base + bk_k[1][2 * pr], base + bk_k[1][2 * pr + 1], bq[1]);
      } else {
        v2i_t lo[JB][2], hi[JB][2];
        dec16_read_pair<T4>(base + b_lo[0] + pr * 8192, base + b_hi[0] + pr * 8192,
                            base + a_k[2 * pr], base + a_k[2 * pr + 1], lo[0], hi[0], a4);
        if constexpr (JB == 2)
          dec16_read_b_pair(base + b_lo[1] + pr * 8192, base + b_hi[1] + pr * 8192, lo[1],
                            hi[1]);
#pragma unroll
        for (int jj = 0; jj < JB; ++jj)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            bq[jj][h] = i32x4_t{lo[jj][h].x, lo[jj][h].y, hi[jj][h].x, hi[jj][h].y};
      }
      i32x4_t a[2][T];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < T4; ++t)
          a[h][t] = a4[h][t];
      if constexpr (T > 4) { // slices past 64 rows: tiles 4 .. T - 1
        i32x4_t am[2][T - 4];
        dec16_read_more<T - 4>(base + a_k[2 * pr], base + a_k[2 * pr + 1], am);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 4; t < T; ++t)
            a[h][t] = am[h][t - 4];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        i32x4_t bf[JB];
#pragma unroll
        for (int jj = 0; jj < JB; ++jj)
          bf[jj] = bq[jj][h];
        if (tail) {
          const int64_t k = k0 + 32 * (2 * pr + h) + 8 * G;
#pragma unroll
          for (int t = 0; t < T; ++t)
            a[h][t] = dec16_mask_k(a[h][t], k, p.K);
          if constexpr (BT) {
#pragma unroll
            for (int jj = 0; jj < JB; ++jj)
              bf[jj] = dec16_mask_k(bf[jj], k, p.K);
          }
        }
#pragma unroll
        for (int jj = 0; jj < JB; ++jj)
#pragma unroll
          for (int t = 0; t < T; ++t)
            acc[jj][t] = mfma16x16x32<BF>(bf[jj], a[h][t], acc[jj][t]);
      }
    }
  };

  // WQ loads: as above, but each lane keeps the addresses of its loads of the
  // next batch and adds a step to them (0 where it reads the zero chunk: rows of
  // A >= M, columns of B >= N); batches are issued in order.
  const uint8_t *wq_src[Cfg::VPB];
  int64_t wq_step[Cfg::VPB];
  auto wq_row = [&](int u) { // load u's row of B's batch
    return 8 * (Cfg::B_LOADS * wave + u) + (lane >> 3);
  };
  auto wq_chunk = [&](int u) { // load u's 16-byte chunk of A's batch
    const int r = 4 * (Cfg::A_LOADS * wave + u) + (lane >> 4);
    return (lane & 15) ^ (r & 15);
  };
  if constexpr (WQ != WQ_NONE) {
    constexpr int ROWS = Cfg::FP4 ? 64 : 128;
#pragma unroll
    for (int u = 0; u < Cfg::B_LOADS; ++u) { // rows 8 q .. +7 of the batch's 64 or 128
      const int row = wq_row(u), c = (lane & 7) ^ Cfg::swz(row);
      const int64_t k = (int64_t)b_begin * ROWS + row, n = n0 + 16 * c;
      const bool in = n < p.N;
      wq_src[u] = in ? reinterpret_cast<const uint8_t *>(p.B) + k * p.ldb + n
                     : (const uint8_t *)tx_zero_chunk;
      wq_step[u] = in ? ROWS * p.ldb : 0;
    }
#pragma unroll
    for (int u = 0; u < Cfg::A_LOADS; ++u) {
      const int r = 4 * (Cfg::A_LOADS * wave + u) + (lane >> 4);
      const int64_t k = (int64_t)b_begin * kDec16BatchK + 8 * wq_chunk(u);
      const bool in = r < p.M;
      wq_src[Cfg::B_LOADS + u] =
          in ? reinterpret_cast<const uint8_t *>(p.A + (int64_t)r * p.lda + k)
             : (const uint8_t *)tx_zero_chunk;
      wq_step[Cfg::B_LOADS + u] = in ? kDec16BatchK * 2 : 0;
    }
  }
  auto wq_issue = [&](int i, uint8_t *slot) {
    const int b = b_begin + i;
    auto load = [&](int u, const void *src) {
      if (u < Cfg::B_LOADS) // B is read once
        dma16_stream(src, (lds_void *)(slot + (Cfg::B_LOADS * wave + u) * 1024));
      else // A: re-read by every strip
        dma16(src, (lds_void *)(slot + Cfg::A_OFF +
                                (Cfg::A_LOADS * wave + u - Cfg::B_LOADS) * 1024));
    };
    if (i < nb && b < p.k_main_batches) {
#pragma unroll
      for (int u = 0; u < Cfg::VPB; ++u)
        load(u, wq_src[u]);
    } else { // past the split: zeros; K's end: rows or chunks past K too
#pragma unroll
      for (int u = 0; u < Cfg::VPB; ++u) {
        const int64_t k = (int64_t)b * kDec16BatchK +
                          (u < Cfg::B_LOADS ? (Cfg::FP4 ? 2 : 1) * wq_row(u)
                                            : 8 * wq_chunk(u - Cfg::B_LOADS));
        load(u, i < nb && k < p.K ? wq_src[u] : (const uint8_t *)tx_zero_chunk);
      }
    }
#pragma unroll
    for (int u = 0; u < Cfg::VPB; ++u)
      wq_src[u] += wq_step[u];
  };
  auto wq_consume = [&](const uint8_t *slot, int i, f32x4_t (&sums)[JB][T]) {
    constexpr int T4 = T < 4 ? T : 4, NB = Cfg::FP4 ? 2 : 4;
    const uint32_t base = lds_addr(slot);
    const int b = b_begin + i;
    const bool tail = b >= p.k_main_batches;
    const uint32_t at = (uint32_t)(i % Cfg::SEG_B) * Cfg::GPB;
    uint32_t v[2][3];
    v2i_t w[2][NB];
    i32x4_t a[4][T4];
    decwq_read<T4, NB>(xs[0] + at, xs[1] + at, base + wq_b[0], base + wq_b[1], base + a_k[0],
                       base + a_k[1], base + a_k[2], base + a_k[3], v, w, a);
    uint32_t sc[2][4]; // the scale byte of block jj at K step ks
    bool odd = false;
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      uint32_t d0 = __builtin_amdgcn_alignbyte(v[jj][1], v[jj][0], mis[jj]);
      uint32_t d1 = __builtin_amdgcn_alignbyte(v[jj][2], v[jj][1], mis[jj]);
      if (tail) { // groups at or past the row's last
        const int left = p.sb_ld - b * Cfg::GPB; // > 0
        const uint32_t unit = WQ == WQ_NV_E2M1 ? 0x38383838u : 0x7f7f7f7fu;
        const uint32_t k0m = left >= 4 ? ~0u : (1u << (8 * left)) - 1;
        const uint32_t k1m = left >= 8 ? ~0u : left <= 4 ? 0u : (1u << (8 * (left - 4))) - 1;
        d0 = (d0 & k0m) | (unit & ~k0m);
        d1 = (d1 & k1m) | (unit & ~k1m);
      }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        if constexpr (WQ == WQ_NV_E2M1) { // group 2 ks + G / 2 of the batch's 8
          sc[jj][ks] = ((ks < 2 ? d0 : d1) >> (16 * (ks & 1) + 8 * (G >> 1))) & 0xff;
        } else {
          sc[jj][ks] = (d0 >> (8 * ks)) & 0xff;
          odd = odd || sc[jj][ks] - kHwScaleLo > kHwScaleHi - kHwScaleLo;
        }
      }
    }
    auto products = [&](auto hw) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        i32x4_t bf[2];
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
          const uint32_t w0 = Cfg::FP4 ? (ks & 1 ? w[jj][ks / 2].y : w[jj][ks / 2].x)
                                       : w[jj][NB == 4 ? ks : 0].x;
          const uint32_t w1 = Cfg::FP4 ? 0 : w[jj][NB == 4 ? ks : 0].y;
          bf[jj] = decwq_upcast<WQ, decltype(hw)::value>(w0, w1, sc[jj][ks]);
        }
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
          for (int t = 0; t < T4; ++t)
            sums[jj][t] = mfma16x16x32<BF>(bf[jj], a[ks][t], sums[jj][t]);
        if constexpr (T > 4) { // slices past 64 rows: tiles 4 .. T - 1, two steps a read
          if (ks & 1)
            continue;
          i32x4_t am[2][T - 4], bn[2];
          dec16_read_more<T - 4>(base + a_k[ks], base + a_k[ks + 1], am);
#pragma unroll
          for (int jj = 0; jj < 2; ++jj) {
            const uint32_t w0 = Cfg::FP4 ? w[jj][ks / 2].y : w[jj][NB == 4 ? ks + 1 : 0].x;
            const uint32_t w1 = Cfg::FP4 ? 0 : w[jj][NB == 4 ? ks + 1 : 0].y;
            bn[jj] = decwq_upcast<WQ, decltype(hw)::value>(w0, w1, sc[jj][ks + 1]);
          }
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
              for (int t = 4; t < T; ++t)
                sums[jj][t] =
                    mfma16x16x32<BF>(h ? bn[jj] : bf[jj], am[h][t - 4], sums[jj][t]);
        }
      }
    };
    if (WQ != WQ_NV_E2M1 && __any(odd)) // one branch a batch
      products(std::false_type());
    else
      products(std::true_type());
  };

  // Prologue: S - 1 batches in flight; batch i uses slot i % S.  (WQ: the
  // first segment's scales before them.)
  if constexpr (WQ != WQ_NONE) {
    stage_scales(0);
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
      wq_issue(s, ring + s * SLOT);
    // The loop below, unrolled by the two chains only: a batch's code holds both
    // upcasts.
    f32x4_t acc2[JB][T];
#pragma unroll
    for (int jj = 0; jj < JB; ++jj)
#pragma unroll
      for (int t = 0; t < T; ++t)
        acc2[jj][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int chain = nb > 4 && nb < 8 ? (nb + 1) / 2 : 4; // batches a turn
    int s = 0, sl = S - 1;
    auto run = [&](int i, f32x4_t (&sums)[JB][T]) {
      for (const int end = i + chain < nb ? i + chain : nb; i < end; ++i) {
        if (i > 0 && i % Cfg::SEG_B == 0) { // every wave has read the segment before
          asm volatile("s_barrier" ::: "memory");
          stage_scales(i);
          wait_vmcnt<0>();
        }
        wait_vmcnt<(S - 2) * Cfg::VPB>();
        asm volatile("s_barrier" ::: "memory");
        wq_issue(i + S - 1, ring + sl * SLOT);
        wq_consume(ring + s * SLOT, i, sums);
        s = s + 1 == S ? 0 : s + 1;
        sl = sl + 1 == S ? 0 : sl + 1;
      }
    };
    for (int i = 0; i < nb; i += 2 * chain) {
      run(i, acc);
      run(i + chain, acc2);
    }
#pragma unroll
    for (int jj = 0; jj < JB; ++jj)
#pragma unroll
      for (int t = 0; t < T; ++t)
        acc[jj][t] += acc2[jj][t];
    goto k_loop_done;
  }
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    issue(s, ring + s * SLOT);
  // Main loop, unrolled by S so slot addresses are static; left at the first
  // batch past nb.  At batch i: wait for this wave's loads of batch i (the
  // S - 2 batches after it stay in flight), barrier (every wave's loads of
  // batch i have landed and every wave has read batch i - 1's slot), issue
  // batch i + S - 1 into that slot, then the MFMAs of batch i.
  for (int i0 = 0;; i0 += S) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int i = i0 + s;
      if (i >= nb)
        goto k_loop_done;
      wait_vmcnt<(S - 2) * Cfg::VPB>();
      asm volatile("s_barrier" ::: "memory");
      issue(i + S - 1, ring + ((s + S - 1) % S) * SLOT);
      consume(ring + s * SLOT, i);
    }
  }
k_loop_done:
  __builtin_amdgcn_s_waitcnt(0); // the zero-chunk loads past nb have landed

  // C for this lane and column block jj: row 16 t + L, columns
  // n0 + 16 (JB wave + jj) + 4 G .. +3 (one 8-byte store in 16-bit C, 16
  // bytes in fp32; single elements where the quad crosses N).
  auto epilogue = [&](const f32x4_t (&sum)[T], int jj) {
    const int64_t col = n0 + 16 * (JB * wave + jj) + 4 * G;
    if (col >= p.N)
      return;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int m = 16 * t + L;
      if (m >= p.M)
        continue;
      const float f[4] = {sum[t][0], sum[t][1], sum[t][2], sum[t][3]};
      if (p.c_f32) {
        float *c = static_cast<float *>(p.C) + (int64_t)m * p.ldc + col;
        if (col + 4 <= p.N) {
          f32x4_t v = sum[t];
          if (p.acc_c)
            v += *reinterpret_cast<const f32x4_t *>(c);
          *reinterpret_cast<f32x4_t *>(c) = v;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (col + r < p.N)
              c[r] = p.acc_c ? c[r] + f[r] : f[r];
        }
      } else {
        uint16_t *c = static_cast<uint16_t *>(p.C) + (int64_t)m * p.ldc + col;
        if (col + 4 <= p.N) {
          uint2 w;
          w.x = BF ? pk_bf16_rne(f[0], f[1]) : pk_f16_rne(f[0], f[1]);
          w.y = BF ? pk_bf16_rne(f[2], f[3]) : pk_f16_rne(f[2], f[3]);
          *reinterpret_cast<uint2 *>(c) = w;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (col + r < p.N)
              c[r] = BF ? f32_to_bf16_rne(f[r]) : f32_to_f16_rne(f[r]);
        }
      }
    }
  };
  if (p.ksplit == 1) {
#pragma unroll
    for (int jj = 0; jj < JB; ++jj)
      epilogue(acc[jj], jj);
    return;
  }

  // Publish this split's partial, count arrivals for the strip, and let the
  // last arrival gather: decode_i8.h's protocol and SC1 cache policy (data
  // crosses workgroups only through the device-coherent level; every store
  // is acknowledged before the barrier that precedes the counter increment;
  // the last workgroup loads only after its increment has returned).
  constexpr int kSC1 = 16;
  const int64_t split_bytes = decode16_split_bytes(strips, SR, W);
  auto part_rsrc = [&](int q) {
    return __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<uint8_t *>(p.partials) + (int64_t)q * split_bytes, 0, (int)split_bytes,
        0x00020000);
  };
  // 1 KiB blocks in lane order: column block jj, row tile t at blk0 + jj T + t.
  const int blk0 = (strip * kDecodeWaves + wave) * JB * T;
  {
    const auto mine = part_rsrc(split);
#pragma unroll
    for (int jj = 0; jj < JB; ++jj)
#pragma unroll
      for (int t = 0; t < T; ++t)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i_t, acc[jj][t]), mine,
                                               ((blk0 + jj * T + t) << 10) + 16 * lane, 0,
                                               kSC1);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0) {
    uint32_t *const ctr = &p.counters[strip];
    const uint32_t old =
        __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = old + 1 == (uint32_t)p.ksplit;
    if (last) // every split has arrived: none touches the counter again
      __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *reinterpret_cast<volatile uint32_t *>(&last_flag) = last;
  }
  __syncthreads();
  if (!*reinterpret_cast<volatile uint32_t *>(&last_flag))
    return;
  // Last arrival: sum = partial 0 + partial 1 + .. in split order (WQ: 4 or more in
  // halves), its own from registers; NQ splits' loads in flight before any is used.
  f32x4_t sum[JB][T];
#pragma unroll
  for (int jj = 0; jj < JB; ++jj)
#pragma unroll
    for (int t = 0; t < T; ++t)
      sum[jj][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  [[maybe_unused]] f32x4_t low[JB][T]; // WQ: the first half of 4 splits or more
  constexpr int NQ = 4 / JB;
  for (int q0 = 0; q0 < p.ksplit; q0 += NQ) {
    if constexpr (WQ != WQ_NONE) {
      if (q0 == p.ksplit / 2 && q0 > 1) {
#pragma unroll
        for (int jj = 0; jj < JB; ++jj)
#pragma unroll
          for (int t = 0; t < T; ++t) {
            low[jj][t] = sum[jj][t];
            sum[jj][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
    v4i_t v[NQ][JB][T];
#pragma unroll
    for (int qq = 0; qq < NQ; ++qq)
      if (q0 + qq < p.ksplit && q0 + qq != split) {
        const auto r = part_rsrc(q0 + qq);
#pragma unroll
        for (int jj = 0; jj < JB; ++jj)
#pragma unroll
          for (int t = 0; t < T; ++t)
            v[qq][jj][t] = __builtin_amdgcn_raw_buffer_load_b128(
                r, ((blk0 + jj * T + t) << 10) + 16 * lane, 0, kSC1);
      }
#pragma unroll
    for (int qq = 0; qq < NQ; ++qq)
      if (q0 + qq < p.ksplit)
#pragma unroll
        for (int jj = 0; jj < JB; ++jj)
#pragma unroll
          for (int t = 0; t < T; ++t)
            sum[jj][t] +=
                q0 + qq == split ? acc[jj][t] : __builtin_bit_cast(f32x4_t, v[qq][jj][t]);
  }
  if constexpr (WQ != WQ_NONE) {
    if (p.ksplit > 2) {
#pragma unroll
      for (int jj = 0; jj < JB; ++jj)
#pragma unroll
        for (int t = 0; t < T; ++t)
          sum[jj][t] += low[jj][t];
    }
  }
#pragma unroll
  for (int jj = 0; jj < JB; ++jj)
    epilogue(sum[jj], jj);
}

} // namespace txk
