// 128x128 tile kernel on a deep LDS ring, for dots whose 256x256 tiles leave
// CUs idle (a few hundred rows, or N and K of a few thousand): bf16 / fp16,
// int8, fp8 (e4m3 / e5m2 in any mix, unscaled or 128-block-scaled) and MX
// operands, B row-major or K-major, every epilogue of those dots.
//
// One workgroup of 8 waves (2 x 4 waves of 64x32, two a SIMD) fills a CU's LDS
// with a ring of S = 4 slots, each 128 bytes of K: 16 KiB of A, 16 KiB of B
// and the step's scales.  Why this shape: with one workgroup a CU nothing else
// hides a load's latency, so three to four steps (96-128 KiB) are kept in
// flight, against the one to two steps of the 256x256 tile.  Eight waves
// rather than four of 64x64: one wave a SIMD reads LDS at about half the rate
// of two (106 against 210 B/clk of ds_read_b128, 45 against 115 of the
// transposed reads), and four waves took 36.5 us for the reads and MFMAs alone
// of bf16 1024x4096x4096 (64 steps), more than its loads (27.1 us).  A wave's
// fragments of step i + 1 are read into a second set of registers around step
// i's MFMAs.  Step i:
//     wait: own loads of step i + 1 landed, own fragment reads of step i done
//     s_barrier      (so every wave's are: slot i + 1 is whole, slot i free)
//     loads of step i + S into slot i; fragment reads of step i + 1
//     MFMAs of step i
// What bounds it: the bytes a CU can load (32 KiB a step for 4.2 (8-bit) or
// 2.1 (16-bit) MFLOP), 1.4 to 2 times the 256x256 tile's per FLOP.
//
// Staging is the 256x256 tiles': asm buffer loads into LDS with a lane's byte
// offset kept per tile, the K step in the scalar offset, out-of-range offsets
// (rows of A >= M, columns of B >= N, K chunks >= K, steps past the range)
// reading zeros.  A chunk that crosses K is loaded whole and its bytes past K
// are zeroed in the fragment registers in the masked steps (not for MX, whose
// chunks never cross, nor A of a row-major int8 dot, where junk meets zeros).
// Slot layout, 16-byte chunk c of row r at c ^ swizzle(r):
//   A, and K-major B: [128][128 B], swizzle (r >> 1) & 7: the 16 rows a
//     quarter-wave reads with ds_read_b128 fall in 16 bank groups;
//   B 8-bit: [128 K][128 B], (r >> 1) & 3 and, as bit 2, the row bit that
//     tells neighbouring lane groups apart, so that one ds_read_b64_tr_b8
//     (4 groups of 8 rows) covers every bank group twice;
//   B 16-bit: [64 K][256 B], the same on chunk pairs with r & 3 and bit 3.
// Fragment order: 8-bit lanes hold K bytes 32 (l / 16) .. +31 of a step, MX
// and 16-bit ones chunks l / 16 and 4 + l / 16 (the scaled MFMA's true order;
// for 16 bits K steps 0 and 1 of 32 elements).  MFMA roles are swapped as on
// the other tiles: lane l ends with C row l % 16 at 4 consecutive columns.
//
// Sums: with fp32 C from 16-bit or e2m1 operands the accumulators are emptied
// into a second set every 8 steps, so no chain of additions is longer than 8
// steps or their number.  A range here is up to 8 times the one the 256x256
// tile's own split would take, and one chain over it doubled the error (bf16
// 860x1856x4928 against 64 bits: 3.0e-7, that tile 1.5e-7, this 1.3e-7).  fp8
// operands' error is the MFMA's own sum of 32 products (1.29e-5 either way,
// K = 2048 to 8192), and there the second set costs 6 % of the time.
//
// The plan is the 256x256 tile's (TX_FLAG_TILES_128): its block_k is one ring
// step.  Split-K ranges are whole steps; a range's partial C is 32-bit, summed
// by splitk_reduce.h.
#pragma once

#include <type_traits>

#include "decode_f8.h"
#include "gemm8_w4.h"

namespace txk {

template <int OP, int EPI, int FA = 0, int FB = 0, bool BT = false> struct GemmRing {
  static constexpr int BM = 128, BN = 128, NW = 8, WTM = 64, WTN = 32, FM = 4, FN = 2,
                       S = 4;
  static constexpr bool B16 = OP == OP_BF16 || OP == OP_F16, INT = OP == OP_I8;
  static constexpr int ELT = B16 ? 2 : 1;
  static constexpr bool SCALED = EPI == EPI_BLOCK128_BF16 || EPI == EPI_BLOCK128_F32;
  static constexpr bool MX = EPI == EPI_MX_F32 || EPI == EPI_MX_BF16;
  static constexpr bool F4 = MX && FA == 4;
  static constexpr bool W32 = EPI == EPI_F32 || EPI == EPI_I32 || EPI == EPI_BLOCK128_F32 ||
                              EPI == EPI_MX_F32; // 32-bit C
  static constexpr bool CHAINS = W32 && (B16 || F4); // sums in two levels
  static constexpr int SG = F4 ? 8 : 4, NSD = F4 ? 4 : 2, RS = 4 * NSD; // MX (gemm8_w4.h)
  static constexpr int A_BYTES = 16384, SA_OFF = 32768;
  static constexpr int SB_OFF = SA_OFF + (MX ? BM * RS : SCALED ? BM * 4 : 0);
  static constexpr int SLOT = SB_OFF + (MX ? BN * RS : SCALED ? 1536 : 0);
  static constexpr int SC_LOADS = MX ? NSD / 2 : SCALED ? 1 : 0; // scale loads a wave and step
  static constexpr int LD = 16 / NW; // loads of A, and of B, a wave and step
  static constexpr int VPB = 2 * LD + SC_LOADS;
  static constexpr uint32_t kOOB = 0x80000000u;
  static_assert(S * SLOT <= 160 * 1024 && SLOT % 128 == 0, "ring in LDS; offsets keep bits 0-6");
  static_assert((S - 1) * VPB <= 63, "vmcnt is 6 bits");
  static_assert(!BT || !MX, "K-major B: not the MX forms");
  typedef std::conditional_t<INT, i32x4_t, f32x4_t> Acc;
  typedef Gemm8W4<B16 ? OP_F8 : OP, B16 ? EPI_F32 : EPI, B16 ? 0 : FA, B16 ? 0 : FB,
                  !MX && BT> W8; // the 8-bit tile's MFMA forms

  // This lane's byte offsets of the wave's 2 + 2 loads of a step (kOOB: a row
  // or column outside the matrix) and of its scale loads.
  struct Offsets {
    uint32_t a[LD], b[LD], s[SC_LOADS ? SC_LOADS : 1];
  };
  // Row and swizzled chunk of load j (1 KiB) of a [128][128 B] operand.
  __device__ __forceinline__ static void at128(int j, int lane, int &row, int &c) {
    row = 8 * j + (lane >> 3);
    c = (lane & 7) ^ ((row >> 1) & 7);
  }
  __device__ __forceinline__ static void offsets(const GemmArgs &p, int64_t m0, int64_t n0,
                                                 Offsets &o) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lda = (uint32_t)(p.lda * ELT), ldb = (uint32_t)(p.ldb * ELT);
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const int j = LD * wave + i;
      int row, c;
      at128(j, lane, row, c);
      o.a[i] = m0 + row < p.M ? (uint32_t)(m0 + row) * lda + 16u * c : kOOB;
      if constexpr (BT) {
        o.b[i] = n0 + row < p.N ? (uint32_t)(n0 + row) * ldb + 16u * c : kOOB;
      } else if constexpr (B16) {
        const int k = 4 * j + (lane >> 4);
        const int cb = (lane & 15) ^ (((k & 3) | (((k >> 3) & 1) << 2)) << 1);
        o.b[i] = n0 + 8 * cb < p.N ? (uint32_t)k * ldb + (uint32_t)n0 * 2u + 16u * cb : kOOB;
      } else {
        const int k = 8 * j + (lane >> 3);
        const int cb = (lane & 7) ^ (((k >> 1) & 3) | (((k >> (MX ? 4 : 5)) & 1) << 2));
        o.b[i] = n0 + 16 * cb < p.N ? (uint32_t)k * ldb + (uint32_t)n0 + 16u * cb : kOOB;
      }
    }
    if constexpr (MX) { // rows of A's scales, then of B's: dword q % NSD of row q / NSD
#pragma unroll
      for (int t = 0; t < SC_LOADS; ++t) {
        const int q = (wave * SC_LOADS + t) * 64 + lane, r = q / NSD;
        const bool is_a = r < BM;
        const int64_t g = is_a ? m0 + r : n0 + r - BM;
        o.s[t] = g < (is_a ? p.M : p.N)
                     ? (((uint32_t)g * (uint32_t)p.sa_ld) & ~3u) + 4u * (uint32_t)(q % NSD)
                     : kOOB;
      }
    }
    if constexpr (SCALED) { // waves 0, 1: sa of 64 rows; wave 2: sb; the others: zeros
      const int64_t gm = m0 + 64 * wave + lane;
      o.s[0] = wave < 2 ? (gm < p.M ? (uint32_t)gm * (uint32_t)(p.sa_ld * 4) : kOOB)
               : wave == 2 && lane == 0 ? (uint32_t)(n0 >> 7) * 4u : kOOB;
    }
  }

  struct Rsrc {
    i32x4_t a, b, sa, sb;
  };

  // Loads of K step kt (128 bytes of K) into the slot at LDS address st.
  // MASKED: chunks past K, and every load of a step past the range (!live),
  // read zeros.
  template <bool MASKED>
  __device__ __forceinline__ static void issue(const GemmArgs &p, const Offsets &o, const Rsrc &r,
                                               int kt, bool live_, uint32_t st) {
    const bool live = !MASKED || live_;
    typedef Gemm16W4<OP_BF16, EPI_F32, 4> W;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t k0 = (uint32_t)kt * 128u; // bytes of K
    const uint32_t kb = (uint32_t)(p.K * ELT);
    const uint32_t sb = BT ? k0 : (uint32_t)((int64_t)kt * (128 / ELT) * p.ldb * ELT);
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      uint32_t v = o.a[i];
      if constexpr (MASKED) {
        int row, c;
        at128(LD * wave + i, lane, row, c);
        v = live && k0 + 16u * c < kb ? v : kOOB;
      }
      W::buffer_lds16(v, r.a, live ? k0 : 0u, st + (LD * wave + i) * 1024);
    }
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      uint32_t v = o.b[i];
      if constexpr (MASKED) {
        int row, c;
        at128(LD * wave + i, lane, row, c);
        v = live && (!BT || k0 + 16u * c < kb) ? v : kOOB;
      }
      W::buffer_lds16(v, r.b, live ? sb : 0u, st + A_BYTES + (LD * wave + i) * 1024);
    }
    if constexpr (MX) {
#pragma unroll
      for (int t = 0; t < SC_LOADS; ++t) {
        const int q0 = (wave * SC_LOADS + t) * 64; // whole loads of A's or of B's rows
        W8::buffer_lds4(live ? o.s[t] : kOOB, q0 < BM * NSD ? r.sa : r.sb,
                        live ? (uint32_t)(kt * SG) : 0u, st + SA_OFF + q0 * 4);
      }
    }
    if constexpr (SCALED)
      W8::buffer_lds4(live ? o.s[0] : kOOB, wave < 2 ? r.sa : r.sb,
                      !live ? 0u : wave < 2 ? (uint32_t)kt * 4u : (uint32_t)(kt * p.sb_ld * 4),
                      st + (wave < 2 ? SA_OFF + 256 * wave : SB_OFF + 256 * (wave - 2)));
  }

  // A wave's operands of one step.
  struct Frags {
    i32x4_t a[FM][2], b[FN][2];
    float s[SCALED ? FM : 1];             // sa * sb of the lane's row
    int sxa[MX ? FM : 1], sxb[MX ? FN : 1]; // MX scale operands
  };
  // Per-lane LDS offsets within a slot.
  struct Bases {
    uint32_t a, b, xa, xb;
  };
  __device__ __forceinline__ static void bases(const GemmArgs &p, int64_t m0, int64_t n0, int wm,
                                               int wn, Bases &bs) {
    const int lane = threadIdx.x & 63, G = lane >> 4, L = lane & 15;
    const int c0 = (MX || B16) ? G : 2 * G; // first chunk; the second is ^ 4 or ^ 1
    bs.a = (wm * WTM + L) * 128 + ((c0 ^ (L >> 1)) << 4);
    if constexpr (BT)
      bs.b = A_BYTES + (wn * WTN + L) * 128 + ((c0 ^ (L >> 1)) << 4);
    else if constexpr (B16) // rows 32 ks + 8 G + L / 4 (+4), columns 32 wn + 16 j + 4 (L % 4)
      bs.b = A_BYTES + (8 * G + (L >> 2)) * 256 +
             (((4 * wn + ((L & 3) >> 1)) ^ (((L >> 2) | ((G & 1) << 2)) << 1)) << 4) + 8 * (L & 1);
    else // rows 32 G (MX: 16 G) + L / 2, chunk 2 wn + j
      bs.b = A_BYTES + ((MX ? 16 : 32) * G + (L >> 1)) * 128 +
             (((2 * wn) ^ (((L >> 2) & 3) | ((G & 1) << 2))) << 4) + 8 * (L & 1);
    if constexpr (MX) { // scale bytes: the row's misalignment, then its group
      const uint32_t sld = (uint32_t)p.sa_ld;
      const int ra = wm * WTM + L, cb = wn * WTN + L;
      bs.xa = SA_OFF + ra * RS + (((uint32_t)(m0 + ra) * sld) & 3u) + G;
      bs.xb = SB_OFF + cb * RS + (((uint32_t)(n0 + cb) * sld) & 3u) + G;
    }
  }

  typedef __attribute__((address_space(3))) i32x4_t lds_i32x4;
  typedef __attribute__((address_space(3))) float lds_f32;
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  __device__ __forceinline__ static i32x4_t read16(uint32_t a) {
    return *(const lds_i32x4 *)(uintptr_t)a;
  }
  __device__ __forceinline__ static int read_sx(uint32_t a) {
    int v = *(const lds_u8 *)(uintptr_t)a;
    if constexpr (F4)
      v |= (int)*(const lds_u8 *)(uintptr_t)(a + 4) << 8;
    return v;
  }
  __device__ __forceinline__ static void read(const Bases &bs, uint32_t st, int wm, Frags &f) {
    const int L = threadIdx.x & 15;
    constexpr uint32_t X = (MX || B16) ? 64u : 16u;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (BT) {
        f.b[j][0] = read16(st + bs.b + 2048 * j);
        f.b[j][1] = read16((st + bs.b + 2048 * j) ^ X);
      } else if constexpr (B16) {
        typedef __attribute__((address_space(3))) i16x4_t lds_t;
        const uint32_t a = st + (bs.b ^ (32u * j));
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const v2i_t lo = __builtin_bit_cast(
              v2i_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t *)(uintptr_t)(a + 8192 * ks)));
          const v2i_t hi = __builtin_bit_cast(
              v2i_t,
              __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t *)(uintptr_t)(a + 8192 * ks + 1024)));
          f.b[j][ks] = i32x4_t{lo.x, lo.y, hi.x, hi.y};
        }
      } else {
        typedef __attribute__((address_space(3))) v2i_t lds_t;
        const uint32_t a = st + (bs.b ^ (16u * j));
        v2i_t v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[q] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
              (lds_t *)(uintptr_t)(a + 128 * (MX ? (q & 1) * 8 + (q >> 1) * 64 : q * 8)));
        f.b[j][0] = i32x4_t{v[0].x, v[0].y, v[1].x, v[1].y};
        f.b[j][1] = i32x4_t{v[2].x, v[2].y, v[3].x, v[3].y};
      }
      if constexpr (MX)
        f.sxb[j] = read_sx(st + bs.xb + 16 * RS * j);
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      f.a[i][0] = read16(st + bs.a + 2048 * i);
      f.a[i][1] = read16((st + bs.a + 2048 * i) ^ X);
      if constexpr (MX)
        f.sxa[i] = read_sx(st + bs.xa + 16 * RS * i);
      if constexpr (SCALED)
        f.s[i] = *(const lds_f32 *)(uintptr_t)(st + SA_OFF + 4 * (wm * WTM + 16 * i + L)) *
                 *(const lds_f32 *)(uintptr_t)(st + SB_OFF);
    }
  }
  // A masked step: bytes at or past K zeroed, MX groups past K / 32 neutral.
  __device__ __forceinline__ static void mask(const GemmArgs &p, int kt, Frags &f) {
    const int G = (threadIdx.x & 63) >> 4;
    if constexpr (MX) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
        f.sxa[i] = W8::tail_sx(f.sxa[i], kt, p.sa_ld);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        f.sxb[j] = W8::tail_sx(f.sxb[j], kt, p.sa_ld);
    } else if constexpr (!INT || BT) {
      const int64_t kb = p.K * ELT, k0 = (int64_t)kt * 128 + 16 * (B16 ? G : 2 * G);
      constexpr int H = B16 ? 64 : 16; // the second chunk, in bytes of K
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        f.a[i][0] = dec8_mask_k(f.a[i][0], k0, kb);
        f.a[i][1] = dec8_mask_k(f.a[i][1], k0 + H, kb);
      }
      if constexpr (BT) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          f.b[j][0] = dec8_mask_k(f.b[j][0], k0, kb);
          f.b[j][1] = dec8_mask_k(f.b[j][1], k0 + H, kb);
        }
      }
    }
  }

  __device__ __forceinline__ static i32x8_t join(const i32x4_t (&v)[2]) {
    return i32x8_t{v[0][0], v[0][1], v[0][2], v[0][3], v[1][0], v[1][1], v[1][2], v[1][3]};
  }
  __device__ __forceinline__ static void pin(Acc &v) { asm volatile("" : "+v"(v)); }
  __device__ __forceinline__ static void products(const Frags &f, Acc (&acc)[FM][FN]) {
    if constexpr (B16) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = mfma16x16x32<OP == OP_BF16>(f.b[j][ks], f.a[i][ks], acc[i][j]);
    } else if constexpr (INT) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = mfma_i8_16(f.b[j][h], f.a[i][h], acc[i][j]);
    } else if constexpr (SCALED) {
      // a row block's products, then the scale FMAs of the block before it,
      // which have had these MFMAs' time to finish
      Acc P[FN], Q[FN];
#pragma unroll
      for (int i = 0; i <= FM; ++i) {
        if (i < FM) {
#pragma unroll
          for (int j = 0; j < FN; ++j)
            Q[j] = W8::mma(join(f.b[j]), join(f.a[i < FM ? i : 0]), Acc{0, 0, 0, 0});
        }
        if (i > 0) {
#pragma unroll
          for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              acc[i - 1][j][r] = __builtin_fmaf(P[j][r], f.s[i - 1], acc[i - 1][j][r]);
            pin(acc[i - 1][j]);
          }
        }
#pragma unroll
        for (int j = 0; j < FN; ++j)
          P[j] = Q[j];
      }
    } else {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          if constexpr (MX)
            acc[i][j] = W8::mma_mx(join(f.b[j]), join(f.a[i]), acc[i][j], f.sxb[j], f.sxa[i]);
          else
            acc[i][j] = W8::mma(join(f.b[j]), join(f.a[i]), acc[i][j]);
        }
    }
  }

  // C through LDS (the ring is free once every wave is past the K loop): the
  // tile leaves in whole rows, 16-byte chunk c of row r staged at c ^ (r & 15).
  __device__ __forceinline__ static void epilogue(const GemmArgs &p, void *C, int64_t m0,
                                                  int64_t n0, int wm, int wn,
                                                  const Acc (&acc)[FM][FN], uint32_t lds0) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v2u lds_v2u;
    typedef __attribute__((address_space(3))) v4u lds_v4u;
    const int lane = threadIdx.x & 63, t = threadIdx.x, G = lane >> 4, L = lane & 15;
    constexpr int ROWB = W32 ? 512 : 256, CH = ROWB / 16, EPC = W32 ? 4 : 8; // elements a chunk
    __syncthreads();
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int r = wm * WTM + 16 * i + L;
      float sar = 1.f;
      if constexpr (EPI == EPI_ROWCOL_BF16)
        sar = m0 + r < p.M ? p.sa[m0 + r] : 0.f;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = wn * WTN + 16 * j + 4 * G;
        const Acc &v = acc[i][j];
        if constexpr (W32) {
          *(lds_v4u *)(uintptr_t)(lds0 + r * ROWB + (((col >> 2) ^ (r & 15)) << 4)) =
              __builtin_bit_cast(v4u, v);
        } else {
          float f[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if constexpr (EPI == EPI_ROWCOL_BF16) {
#pragma clang fp contract(off)
              f[q] = ((float)v[q] * sar) * p.sb[n0 + col + q < p.N ? n0 + col + q : 0];
            } else {
              f[q] = (float)v[q];
            }
          }
          const v2u w = EPI == EPI_F16 ? v2u{pk_f16_rne(f[0], f[1]), pk_f16_rne(f[2], f[3])}
                                       : v2u{pk_bf16_rne(f[0], f[1]), pk_bf16_rne(f[2], f[3])};
          *(lds_v2u *)(uintptr_t)(lds0 + r * ROWB + (((col >> 3) ^ (r & 15)) << 4) +
                                  (col & 7) * 2) = w;
        }
      }
    }
    __syncthreads();
#pragma unroll 4
    for (int q = 0; q < BM * CH / (64 * NW); ++q) {
      const int idx = q * 64 * NW + t, r = idx / CH, ch = idx % CH;
      const int64_t row = m0 + r, col = n0 + ch * EPC;
      const v4u v = *(const lds_v4u *)(uintptr_t)(lds0 + r * ROWB + ((ch ^ (r & 15)) << 4));
      if (row >= p.M || col >= p.N)
        continue;
      const bool whole = col + EPC <= p.N;
      if constexpr (W32) {
        typedef std::conditional_t<INT, int32_t, float> E;
        E *c = static_cast<E *>(C) + row * p.ldc + col;
        Acc s = __builtin_bit_cast(Acc, v);
        if (whole) {
          if (p.accumulate)
            s += *reinterpret_cast<const Acc *>(c);
          *reinterpret_cast<Acc *>(c) = s;
        } else {
          const E e[4] = {s[0], s[1], s[2], s[3]};
#pragma unroll
          for (int x = 0; x < 4; ++x)
            if (col + x < p.N)
              c[x] = p.accumulate ? c[x] + e[x] : e[x];
        }
      } else {
        uint16_t *c = static_cast<uint16_t *>(C) + row * p.ldc + col;
        if (whole) {
          *reinterpret_cast<v4u *>(c) = v;
        } else {
          const unsigned w[4] = {v[0], v[1], v[2], v[3]};
#pragma unroll
          for (int x = 0; x < 8; ++x)
            if (col + x < p.N)
              c[x] = (uint16_t)(w[x / 2] >> (16 * (x & 1)));
        }
      }
    }
  }

  __device__ __forceinline__ static void run(const GemmArgs &p, int64_t m0, int64_t n0,
                                             uint8_t *smem) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const int all = (int)((p.K * ELT + 127) / 128), main = p.k_main_steps;
    const int z = blockIdx.y; // this workgroup's K range
    const int k_begin = z * p.split_steps;
    const int k_end = z + 1 < p.split_k ? k_begin + p.split_steps : all;
    const int n = k_end - k_begin;
    void *C = p.split_k > 1 ? static_cast<uint8_t *>(p.C) + (int64_t)z * p.M * p.ldc * 4 : p.C;
    const uint32_t lds0 = lds_addr(smem);
    // Ranges end at the 16-byte chunk holding each operand's last element.
    const int64_t kb = p.K * ELT;
    Rsrc r;
    r.a = make_rsrc(p.A, (uint32_t)((p.M - 1) * p.lda * ELT + ((kb + 15) & ~15ll)));
    r.b = BT ? make_rsrc(p.B, (uint32_t)((p.N - 1) * p.ldb * ELT + ((kb + 15) & ~15ll)))
             : make_rsrc(p.B, (uint32_t)((p.K - 1) * p.ldb * ELT + ((p.N * ELT + 15) & ~15ll)));
    r.sa = r.sb = i32x4_t{0, 0, 0, 0};
    if constexpr (SCALED) {
      r.sa = make_rsrc(p.sa, (uint32_t)(p.M * p.sa_ld * 4));
      r.sb = make_rsrc(p.sb, (uint32_t)(((p.K + 127) / 128) * p.sb_ld * 4));
    }
    if constexpr (MX) { // whole dwords: each holds at least one byte of the array
      r.sa = make_rsrc(p.sa, (uint32_t)((p.M * p.sa_ld + 3) & ~3ll));
      r.sb = make_rsrc(p.sb, (uint32_t)((p.N * p.sa_ld + 3) & ~3ll));
    }
    Offsets o;
    offsets(p, m0, n0, o);
    Bases bs;
    bases(p, m0, n0, wm, wn, bs);
    Acc acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        acc[i][j] = Acc{0, 0, 0, 0};
    Acc sum[CHAINS ? FM : 1][FN];
    if constexpr (CHAINS) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          sum[i][j] = Acc{0, 0, 0, 0};
    }
    auto slot = [&](int i) { return lds0 + (uint32_t)((unsigned)i % S) * SLOT; };
    auto issue_step = [&](int i) { // ring step i of the range into slot i % S
      const int kt = k_begin + i;
      if (i >= n || kt >= main)
        issue<true>(p, o, r, kt, i < n, slot(i));
      else
        issue<false>(p, o, r, kt, true, slot(i));
    };
    if (n > 0) {
#pragma unroll
      for (int s = 0; s < S; ++s)
        issue_step(s);
      wait_vmcnt<(S - 1) * VPB>();
      asm volatile("s_barrier" ::: "memory");
      Frags f[2];
      read(bs, slot(0), wm, f[0]);
      // (The reads of step i + 1 are unconditional: past the range they bring
      // values that are not used, and the block stays one scheduling region.)
      auto step = [&](int i, Frags &cur, Frags &next, auto masked) {
        // own reads of step i done, own loads of step i + 1 landed
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_vmcnt<(S - 2) * VPB>();
        asm volatile("s_barrier" ::: "memory");
        issue_step(i + S);
        if (decltype(masked)::value && k_begin + i >= main)
          mask(p, k_begin + i, cur);
        read(bs, slot(i + 1), wm, next);
        products(cur, acc);
      };
      const int nu = (main < k_end ? main : k_end) - k_begin; // unmasked steps
      int i = 0;
      for (; i + 1 < nu; i += 2) {
        step(i, f[0], f[1], std::false_type());
        step(i + 1, f[1], f[0], std::false_type());
        if constexpr (CHAINS) {
          if ((i & 6) == 6) {
#pragma unroll
            for (int x = 0; x < FM; ++x)
#pragma unroll
              for (int y = 0; y < FN; ++y) {
                sum[x][y] += acc[x][y];
                acc[x][y] = Acc{0, 0, 0, 0};
              }
          }
        }
      }
      for (; i < n; i += 2) {
        step(i, f[0], f[1], std::true_type());
        if (i + 1 < n)
          step(i + 1, f[1], f[0], std::true_type());
      }
      __builtin_amdgcn_s_waitcnt(0); // the zero loads past the range have landed
    }
    if constexpr (CHAINS) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] += sum[i][j];
    }
    epilogue(p, C, m0, n0, wm, wn, acc, lds0);
  }
};

template <int OP, int EPI, int FA = 0, int FB = 0, bool BT = false>
__global__ void __launch_bounds__(512, 1) gemm_ring_kernel(GemmArgs p) {
  typedef GemmRing<OP, EPI, FA, FB, BT> R;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[R::S * R::SLOT];
  // Workgroups go round-robin to the 8 XCDs: give each XCD a run of tiles,
  // walked in groups of group_m tile rows (tile_coords, for any tile count).
  const int nwg = gridDim.x, b = blockIdx.x, per = nwg / 8, rem = nwg % 8, x = b % 8;
  const int t = x * per + (x < rem ? x : rem) + b / 8;
  const int width = p.group_m * p.tiles_n, group = t / width, first = group * p.group_m;
  const int gsz = p.tiles_m - first < p.group_m ? p.tiles_m - first : p.group_m;
  const int q = t - group * width;
  R::run(p, (int64_t)(first + q % gsz) * R::BM, (int64_t)(q / gsz) * R::BN, smem);
}

} // namespace txk
