// arith_intensity extension: libarith_intensity.so.
//
// The task names an "arithmetic-intensity pass" that the reference snapshot
// does not contain, so this extension has no reference source to follow.  It
// classifies a dot by its algorithmic work (every operand read once, the
// output written once, scales read once) against MI355X's roofline and
// recommends a tile from the set the mi355x_dot backend instantiates.
//
// MI355X public dense peaks: bf16/fp16 MFMA 2516.6 TFLOP/s (256 CUs x
// 2.4 GHz x 4096 FLOP/clk/CU), fp8 and int8 5033.2 T(FL)OP/s, fp4 10066.4
// TFLOP/s, HBM3E 8 TB/s.

#include "triton_ext/TritonExtPassInfra.h"
#include "triton_ext/tx_dot.h"
#include "triton_ext/tx_passes.h"

#include <climits>
#include <cmath>
#include <cstdint>

namespace {

constexpr double kPeak16 = 2516.6e12;
constexpr double kPeak8 = 5033.2e12;
constexpr double kPeak4 = 10066.4e12;
constexpr double kPeakF32 = 157.3e12;
constexpr double kHbm = 8.0e12;
constexpr int kCUs = 256;

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

struct Tile {
  int32_t bm, bn, bk;
  bool tiles128 = false; // TX_FLAG_TILES_128: the 256x256 plan on 128x128 tiles
};

// Estimated time of a tiled dot, in us.  A round of n workgroups (at most one,
// or `occ`, a CU) takes `per + steps * (s0 + s1 * n / CUs)`: a K step is
// slower the more CUs load and draw power at once.  Fitted to back-to-back
// launches on one MI355X, measured / estimated in us:
//   bf16 256x256x64:  4096^3 104 / 106, 3072^3 61 / 70, M = 512 N = K = 8192 (split 4) 82 / 82;
//   bf16 128x128:     M = 1000 N = K = 4000 39.4 / 39.6, 3072^3 78 / 79, 2048^3 22 / 23;
//   bf16 64x64x32:    512^3 7.4 / 9, 1024^3 18 / 19;
//   W8A8 256x256x128: 3072^3 39 / 43, M = 512 N = K = 8192 (split 4) 54 / 61;
//   W8A8 128x128:     M = 512 N = K = 8192 40 / 41, 3072^3 50 / 46;
//   fp8 block-scaled  256: M = 1024 N = K = 7168 73 / 77, 128: 79 / 80, M = 512 40 / 43;
//   mxfp8             256: M = 1024 N = 8192 K = 4096 53 / 54, 128: 53 / 52;
//   mxfp4             256: the same shape 33 / 34, 128: 36 / 39; 2048x2800x8192 61 / 56, 66 / 61.
struct Rate {
  double launch, per, s0, s1;
  int occ; // workgroups a CU
};
constexpr Rate k256x16{4.5, 2.5, 1.00, 0.55, 1}, k128x16{4.0, 2.2, 0.33, 0.20, 1};
constexpr Rate k64x16{2.0, 0.5, 0.33, 0.20, 4}, k128dma{3.0, 0.5, 0.90, 0.40, 2};
constexpr Rate k256x8{5.0, 3.0, 1.05, 0.70, 1}, k128x8{4.0, 2.2, 0.33, 0.22, 1};
constexpr Rate k128f8b{4.0, 2.2, 0.40, 0.27, 1};
constexpr Rate k256mx8{5.0, 3.0, 1.15, 0.55, 1}, k128mx8{4.0, 2.2, 0.40, 0.28, 1};
constexpr Rate k256mx4{5.0, 3.0, 1.20, 0.90, 1}, k128mx4{4.0, 2.2, 0.53, 0.43, 1};

double estimate(const Rate &r, int64_t bm, int64_t bn, int64_t bk, int64_t split, int64_t M,
                int64_t N, int64_t K) {
  const int64_t n = cdiv(M, bm) * cdiv(N, bn) * split;
  const double steps = (double)cdiv(cdiv(K, bk), split);
  const int64_t cap = (int64_t)kCUs * r.occ, full = n / cap, rem = n % cap;
  auto round = [&](int64_t wgs) {
    return r.per + steps * (r.s0 + r.s1 * (wgs < kCUs ? (double)wgs / kCUs : 1.0));
  };
  double us = r.launch + (double)full * round(cap) + (rem ? round(rem) : 0.0);
  // The reduction: its partials written and read at about 6 TB/s from a whole
  // round of workgroups; those of a part of one are mostly hidden (fp8
  // 2048x2800x8192, 176 workgroups: 63 us in all, of which the ranges take 57;
  // bf16 1000x8192x4096, 256: 78 of which 57).
  if (split > 1) {
    const double f = n < kCUs ? (double)n / kCUs : 1.0;
    us += 3.0 + f * f * 8.0 * (double)split * (double)M * (double)N / 6e6;
  }
  return us;
}

// The 256x256 tile of a dot: on 256x256 or on 128x128 tiles (TX_FLAG_TILES_128).
// bk: elements of 128 bytes of K; split256: the 256x256 tiles may split K.
Tile choose256(const Rate &r256, const Rate &r128, int32_t bk, bool split256, int64_t M, int64_t N,
               int64_t K, bool can128, double *us) {
  Tile t{256, 256, bk};
  const int64_t steps = cdiv(K, bk);
  const int64_t s256 = split256 ? tx_gemm_split_k(cdiv(M, 256) * cdiv(N, 256), steps) : 1;
  *us = estimate(r256, 256, 256, bk, s256, M, N, K);
  if (!can128)
    return t;
  const double u128 = estimate(r128, 128, 128, bk,
                               tx_ring_split_k(cdiv(M, 128) * cdiv(N, 128), steps), M, N, K);
  if (u128 < *us) {
    t.tiles128 = true;
    *us = u128;
  }
  return t;
}

} // namespace

extern "C" int32_t tx_gemm_split_k(int64_t tiles, int64_t ksteps) {
  int32_t s = 1;
  while (s < 16 && tiles * s * 2 <= kCUs && ksteps / (s * 2) >= 8)
    s *= 2;
  return s;
}

extern "C" int32_t tx_ring_split_k(int64_t tiles128, int64_t ksteps) {
  return tx_gemm_split_k(tiles128, ksteps); // the same rule on its own tiles
}

extern "C" int32_t tx_dtype_bits(int32_t dtype) {
  switch (dtype) {
  case TX_F32: return 32;
  case TX_F16: return 16;
  case TX_BF16: return 16;
  case TX_I8: return 8;
  case TX_F8E4M3: return 8;
  case TX_I32: return 32;
  case TX_F8E5M2: return 8;
  case TX_F4E2M1: return 4;
  default: return 0;
  }
}

extern "C" int32_t tx_dtype_size(int32_t dtype) {
  const int32_t b = tx_dtype_bits(dtype);
  return b % 8 ? 0 : b / 8;
}

extern "C" double tx_mi355x_peak_flops(int32_t dtype) {
  switch (dtype) {
  case TX_F16:
  case TX_BF16: return kPeak16;
  case TX_I8:
  case TX_F8E4M3:
  case TX_F8E5M2: return kPeak8;
  case TX_F4E2M1: return kPeak4;
  case TX_F32: return kPeakF32;
  default: return 0.0;
  }
}

extern "C" double tx_mi355x_peak_bw(void) { return kHbm; }

extern "C" int tx_dot_operand_spans(const tx_dot_desc *d, int64_t *a_bytes, int64_t *b_bytes) {
  if (!d || !a_bytes || !b_bytes)
    return TX_ERR_INVALID;
  const int32_t ba = tx_dtype_bits(d->a_type), bb = tx_dtype_bits(d->b_type);
  if (!ba || !bb)
    return TX_ERR_INVALID;
  const bool bt = (d->flags & TX_FLAG_B_KMAJOR) != 0;
  const int64_t lda = d->lda ? d->lda : d->K;
  const int64_t ldb = d->ldb ? d->ldb : (bt ? d->K : d->N);
  // ((rows - 1) * ld + len) elements of `bits` bits, in 128-bit arithmetic
  auto span = [](int64_t rows, int64_t ld, int64_t len, int32_t bits) -> int64_t {
    if (rows <= 0 || len <= 0)
      return 0;
    const __int128 e = (__int128)(rows - 1) * ld + len;
    const __int128 b = (e * bits + 7) / 8;
    return b > (__int128)INT64_MAX ? INT64_MAX : (int64_t)b;
  };
  *a_bytes = span(d->M, lda, d->K, ba);
  if (bt)
    *b_bytes = span(d->N, ldb, d->K, bb);
  else if (bb == 4) // packed rows of two K values: K / 2 rows of ldb bytes
    *b_bytes = span((d->K + 1) / 2, ldb, d->N, 8);
  else
    *b_bytes = span(d->K, ldb, d->N, bb);
  return TX_OK;
}

extern "C" int32_t tx_ring_reaches(const tx_dot_desc *d) {
  if (!d || cdiv(d->M, 128) * cdiv(d->N, 128) >= ((int64_t)1 << 23))
    return 0;
  if (d->flags & TX_FLAG_B_KMAJOR)
    return 1;
  const bool packed = tx_dtype_bits(d->b_type) == 4; // ldb: bytes of a row of two K values
  const int64_t rows = packed ? (d->K + 1) / 2 : d->K, ldb = d->ldb ? d->ldb : d->N;
  const __int128 bytes =
      (__int128)(rows + 128) * ldb * (packed ? 1 : tx_dtype_bits(d->b_type) / 8);
  return bytes < (__int128)1 << 32;
}

namespace {

// tx_arith_intensity; *tiles128: the chosen tile runs on 128x128 tiles.
int analyse(const tx_dot_desc *d, tx_ai_report *out, bool *tiles128) {
  if (!d || !out)
    return TX_ERR_INVALID;
  *out = tx_ai_report{};
  const int32_t ba = tx_dtype_bits(d->a_type), bb = tx_dtype_bits(d->b_type),
                bc = tx_dtype_bits(d->c_type);
  if (!ba || !bb || !bc || d->M < 0 || d->N < 0 || d->K < 0)
    return TX_ERR_INVALID;
  const double sa = ba / 8.0, sb = bb / 8.0, sc = bc / 8.0; // bytes per element
  const double M = (double)d->M, N = (double)d->N, K = (double)d->K;
  double scaleBytes = 0.0;
  if (d->scale_mode == TX_SCALE_ROWCOL)
    scaleBytes = 4.0 * (M + N);
  else if (d->scale_mode == TX_SCALE_BLOCK128)
    scaleBytes = 4.0 * (M * cdiv(d->K, 128) +
                        (double)cdiv(d->K, 128) * cdiv(d->N, 128));
  else if (d->scale_mode == TX_SCALE_MX32 || d->scale_mode == TX_SCALE_NV16)
    // one scale byte per 32 K (e8m0) or 16 K (e4m3); a bf16 side has none
    scaleBytes = ((ba == 16 ? 0.0 : M) + (bb == 16 ? 0.0 : N)) *
                 (double)cdiv(d->K, d->scale_mode == TX_SCALE_NV16 ? 16 : 32);
  out->flops = 2.0 * M * N * K;
  // C once, twice when accumulating into it (read, then written)
  const double cPasses = (d->flags & TX_FLAG_ACCUMULATE) ? 2.0 : 1.0;
  out->bytes = M * K * sa + K * N * sb + cPasses * M * N * sc + scaleBytes;
  out->intensity = out->bytes > 0 ? out->flops / out->bytes : 0.0;
  // a mixed product runs at the rate of its wider operand
  out->peak_flops = ba >= bb ? tx_mi355x_peak_flops(d->a_type)
                             : tx_mi355x_peak_flops(d->b_type);
  if (d->scale_mode == TX_SCALE_NV16) // e4m3 scales run on the bf16 tile
    out->peak_flops = tx_mi355x_peak_flops(TX_BF16);
  out->peak_bw = kHbm;
  out->ridge = out->peak_flops / out->peak_bw;
  out->bound = out->intensity > out->ridge ? TX_BOUND_MFMA : TX_BOUND_HBM;
  double tc = out->peak_flops > 0 ? out->flops / out->peak_flops : 0.0;
  double tm = out->bytes / out->peak_bw;
  out->roofline_us = 1e6 * (tc > tm ? tc : tm);

  Tile t{d->block_m, d->block_n, d->block_k};
  if (t.bm <= 0 || t.bn <= 0 || t.bk <= 0) {
    // Operands as the tile reads them (an upcast MX side: packed bf16), and
    // whether the 256-wide tiles (32-bit buffer offsets) can address them.
    const bool upcast = (d->scale_mode == TX_SCALE_MX32 && (ba == 16 || bb == 16)) ||
                        d->scale_mode == TX_SCALE_NV16;
    tx_dot_desc e = *d;
    if (upcast) {
      if (e.a_type != TX_BF16)
        e.a_type = TX_BF16, e.lda = 0;
      if (e.b_type != TX_BF16)
        e.b_type = TX_BF16, e.ldb = TX_MX_UPCAST_LD(d->N);
    }
    int64_t spanA = 0, spanB = 0;
    tx_dot_operand_spans(&e, &spanA, &spanB);
    // The decode kernels' epilogues: W8A8 (row x column scales, bf16 C) and
    // the plain int8 -> int32 dot (no scales, int32 C), N up to their 4096
    // column strips; B row-major, or K-major on the row kernel (M > 48: the
    // 8-bit ring decode kernel takes K-major B below that).  Both stream B
    // once with split-K.
    const bool decode =
        d->a_type == TX_I8 && d->b_type == TX_I8 &&
        (!(d->flags & TX_FLAG_B_KMAJOR) || d->M > 48) && d->N <= (int64_t)4096 * 128 &&
        ((d->scale_mode == TX_SCALE_ROWCOL && d->c_type == TX_BF16) ||
         (d->scale_mode == TX_SCALE_NONE && d->c_type == TX_I32));
    // The 16-bit decode kernel: both operands bf16 or both fp16, no scales,
    // C in their type or fp32, B row-major or K-major, M <= 96, N up to its
    // 16384 strips of 64 columns.  It streams B once with split-K.  Each wave
    // reads every row of the slice from LDS, so its time grows with M: at
    // N = K = 8192 bf16, M = 64 / 80 / 96 33.0 / 34.9 / 45.5 us against the
    // 256x256 tiles with split-K's 46.6 / 48.0 / 49.1, from which the bound at 96
    // was drawn, and the 128x128 ring tiles' 33.8 / 34.6 / 35.2.
    const bool decode16 =
        (d->a_type == TX_BF16 || d->a_type == TX_F16) && d->b_type == d->a_type &&
        d->scale_mode == TX_SCALE_NONE && (d->c_type == d->a_type || d->c_type == TX_F32) &&
        d->M <= 96 && d->N <= (int64_t)16384 * 64;
    // The 8-bit ring decode kernel, B row-major or K-major: fp8 x fp8 with
    // fp32 C, e4m3 x e4m3 with 128-block scales and bf16 / fp32 C, M <= 64;
    // with B K-major also int8 -> int32 and W8A8, M <= 48 (the row kernel's
    // 32 x 32 x 32 products take M = 64: W8A8 22.4 against 26.8 us at
    // N = K = 8192); MX operands (fp8 pairs or e2m1 on both sides) with bf16 /
    // fp32 C; N up to its 16384 strips of 128 columns.
    const bool fp8a = d->a_type == TX_F8E4M3 || d->a_type == TX_F8E5M2;
    const bool fp8b = d->b_type == TX_F8E4M3 || d->b_type == TX_F8E5M2;
    const bool kmajor = (d->flags & TX_FLAG_B_KMAJOR) != 0;
    const bool decode_f8 =
        d->M <= 64 && d->N <= (int64_t)16384 * 128 &&
        ((fp8a && fp8b && d->scale_mode == TX_SCALE_NONE && d->c_type == TX_F32) ||
         (d->scale_mode == TX_SCALE_BLOCK128 && d->a_type == TX_F8E4M3 &&
          d->b_type == TX_F8E4M3 && (d->c_type == TX_BF16 || d->c_type == TX_F32)) ||
         (kmajor && d->a_type == TX_I8 && d->b_type == TX_I8 && d->M <= 48 &&
          ((d->scale_mode == TX_SCALE_NONE && d->c_type == TX_I32) ||
           (d->scale_mode == TX_SCALE_ROWCOL && d->c_type == TX_BF16))));
    const bool decode_mx = d->scale_mode == TX_SCALE_MX32 && !upcast && !kmajor && d->M <= 64 &&
                           d->N <= (int64_t)16384 * 128 &&
                           (d->c_type == TX_BF16 || d->c_type == TX_F32);
    // The 16-bit decode kernel with B upcast in registers: bf16 A (or e2m1 A
    // under e4m3 scales), B scaled, M <= 96; K of two batches or more.
    const bool decode_wq = upcast && d->b_type != TX_BF16 &&
                           (d->a_type == TX_BF16 || d->scale_mode == TX_SCALE_NV16) &&
                           d->M <= 96 && d->K >= 256 && d->N <= (int64_t)16384 * 128 &&
                           (d->c_type == TX_BF16 || d->c_type == TX_F32);
    // Operands the 32-bit-offset tiles reach, and the 128x128 ring tiles too.
    const bool span32 = spanA < TX_SPAN32_LIMIT && spanB < TX_SPAN32_LIMIT;
    const bool can128 = span32 && tx_ring_reaches(&e);
    const bool mx = d->scale_mode == TX_SCALE_MX32;
    double us = 0.0;
    // The 16-bit tiles: 256x256 (or 128x128) against 64x64, which only
    // launch-bound sizes still take; operands past 2 GiB the tiles with 64-bit
    // addresses.
    auto tile16 = [&]() -> Tile {
      if (!span32) {
        const double u128 = estimate(k128dma, 128, 128, 64, 1, d->M, d->N, d->K);
        return u128 <= estimate(k64x16, 64, 64, 32, 1, d->M, d->N, d->K) ? Tile{128, 128, 64}
                                                                        : Tile{64, 64, 32};
      }
      const Tile t256 = choose256(k256x16, k128x16, 64, true, d->M, d->N, d->K, can128, &us);
      if (!kmajor && estimate(k64x16, 64, 64, 32, 1, d->M, d->N, d->K) < us)
        return Tile{64, 64, 32};
      return t256;
    };
    if (decode_wq)
      t = Tile{(int32_t)(16 * cdiv(d->M > 0 ? d->M : 1, 16)), 128, 128};
    else if (upcast)
      t = tile16(); // MX x bf16: the bf16 dot's tile
    else if (decode_mx)
      t = Tile{(int32_t)(16 * cdiv(d->M > 0 ? d->M : 1, 16)), 128, ba == 4 ? 256 : 128};
    else if (mx) // (its 256x256 tiles do not split K)
      t = ba == 4 ? choose256(k256mx4, k128mx4, 256, false, d->M, d->N, d->K, can128, &us)
                  : choose256(k256mx8, k128mx8, 128, false, d->M, d->N, d->K, can128, &us);
    else if (decode_f8)
      t = Tile{(int32_t)(16 * cdiv(d->M > 0 ? d->M : 1, 16)), 128, 128};
    else if (decode16) {
      // Every strip reads all of A, so A's re-reads are M / W of B's bytes.
      // Strips of W = 128 columns halve them: at N = K = 8192 bf16 M = 48 / 64
      // / 80 31.3 / 34.0 / 38.0 us against 35.0 / 39.6 / 45.3 with 64 (B
      // K-major: M = 32 28.5 against 31.8), about equal at M = 16; M = 64 at
      // N = 16384 / 28672 57.1 / 100.2 against 68.4 / 129.9.  With B under
      // 2^25 elements the wider strips double the split (and its partials) or
      // halve the workgroups, and lose: M = 64 at N = K = 4096 18.2 against
      // 16.4 us, at N = 2048 22.0 against 17.9.  Their ring holds slices up
      // to 80 rows.  Slices of 16 rows gain from them at N >= 16384, where 64
      // columns make 256 strips or more: M = 16 at N = 28672, K = 8192 77.6
      // against 93.0 us (B K-major 73.6 / 87.4), at N = 16384, K = 4096 26.6
      // against 28.9 (K-major 29.3 / 37.0); at N = K = 8192 they tie.
      const int32_t rows = (int32_t)(16 * cdiv(d->M > 0 ? d->M : 1, 16));
      const int64_t nk = d->N * d->K;
      const bool wide = (rows >= 32 && rows <= 80 && nk >= ((int64_t)1 << 25)) ||
                        (rows == 16 && d->N >= 16384 && nk >= ((int64_t)1 << 26));
      t = Tile{rows, wide ? 128 : 64, 128};
    }
    else if (sa == 2)
      t = tile16();
    else if (decode && d->M <= 256)
      // W8A8 decode (M <= 256, N up to its 4096 column strips; past it the
      // 8-bit tiles with split-K: at N = K = 8192 M = 384 57.5 us, 512 63.9 on
      // the 256x256 ones, against 76.0 and 78.7 for the row kernel's slices of
      // 256.  The bound is theirs: back to back, M = 96 / 128 / 192 / 256 take
      // 26.0 / 26.4 / 38.1 / 38.6 here, 32.5 / 37.4 / 40.3 / 45.0 on them and
      // 25.7 / 27.8 / 32.7 / 36.8 on the 128x128 ring tiles), 128-column strips.  Up to M = 48 one row slice and 64-row K batches split among
      // the waves; beyond, row slices whose waves all take every 128-row K
      // batch: of 64 rows up to M = 128, of 128 past it.  Measured at
      // N = K = 8192, in us: M = 32 20.1 / 22.1-22.7 (slices of 64), 48 22.0 /
      // 22.2-22.5, 64 25.2 / 22.3-22.9, 96 29.4 (64) / 31.2-32.0 (128), 128
      // 29.6 / 30.5, 192 53.5 / 43.7-44.8, 256 44.8 / 42.6.
      t = d->M > 128 ? Tile{128, 128, 128}
          : d->M > 48 ? Tile{64, 128, 128}
                      : Tile{(int32_t)(16 * cdiv(d->M > 0 ? d->M : 1, 16)), 128, 64};
    else if (!span32) // the register-staged tile: 64-bit addresses
      t = Tile{128, 128, 128};
    else
      t = choose256(k256x8, d->scale_mode == TX_SCALE_BLOCK128 ? k128f8b : k128x8, 128, true, d->M,
                    d->N, d->K, can128, &us);
  }
  if (tiles128)
    *tiles128 = t.tiles128;
  out->block_m = t.bm;
  out->block_n = t.bn;
  out->block_k = t.bk;
  out->tile_intensity = 2.0 * t.bm * t.bn / ((double)(t.bm + t.bn) * sa);
  return TX_OK;
}

} // namespace

extern "C" int tx_arith_intensity(const tx_dot_desc *d, tx_ai_report *out) {
  return analyse(d, out, nullptr);
}

namespace {

// Pass body: classification and tile choice for one dot.
int txArithIntensityRun(tx_dot_plan *plan) {
  tx_ai_report r;
  bool tiles128 = false;
  int rc = analyse(&plan->desc, &r, &tiles128);
  if (rc != TX_OK)
    return rc;
  if (tiles128)
    plan->desc.flags |= TX_FLAG_TILES_128;
  plan->flops = r.flops;
  plan->bytes = r.bytes;
  plan->intensity = r.intensity;
  plan->peak_flops = r.peak_flops;
  plan->peak_bw = r.peak_bw;
  plan->ridge = r.ridge;
  plan->roofline_us = r.roofline_us;
  plan->tile_intensity = r.tile_intensity;
  plan->bound = r.bound;
  plan->desc.block_m = r.block_m;
  plan->desc.block_n = r.block_n;
  plan->desc.block_k = r.block_k;
  plan->passes_run += 1;
  return TX_OK;
}

} // namespace

#define TRITON_EXT_ARG "tx-arith-intensity"
#define TRITON_EXT_RUN txArithIntensityRun
#include "../../infra/TritonExtPass.inc"
