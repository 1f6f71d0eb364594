// X rows times 32 int8 weight rows per wave, summed in the order of the
// multi-token GEMMs (gemm_wide.h): the same fp16 weights, the same
// v_mfma_f32_32x32x16_f16 chain over k, so the fp32 sums have the same bits as
// the rows of those GEMMs.
//
// For one live X row the GEMMs spend a stage's round trip, a barrier and 32 or
// 64 rows of X on every 64 of K.  Here a wave works alone: codes, scales and X
// of 512 k come to its own ring in LDS by direct loads, the whole of a K that
// fits issued at once, and a stage's 16 chunks are one straight run of LDS
// reads, dequantisation (~28 vector instructions per 32 k) and matrix ops.
#pragma once

#include "gemm_core.h"
#include "lds_dma.h"

namespace lemoq_gemm {

constexpr int RW_COLS = 32;  // weight rows per wave

// PAIR: group % 64 == 0 and K % 64 == 0; otherwise K % 16 == 0 and group % 16
// == 0.  XR: 1, every weight row times the one X row; 8, weight row c times X
// row c / 4.
template <bool PAIR, int XR>
struct RowDot {
  static constexpr int KS = 512, CH = KS / 32;                   // k and 32-k chunks of a stage
  static constexpr int UNIT = PAIR ? 64 : 16, SU = KS / UNIT;    // k of a scale, and scales of a row and stage
  static constexpr int WB = RW_COLS * KS, XB = XR * KS * 2, SB = RW_COLS * SU * 4;
  static constexpr int STAGE = WB + XB + SB;                     // bytes: codes, X, scales (a dword each)
  static constexpr int WL = WB / 1024, XL = XB / 1024;           // direct loads of a stage's codes, its X ...
  static constexpr int NL = WL + XL + SU / 2;                    // ... and all of it
  static constexpr int RING = XR > 1 ? 2 : PAIR ? 4 : 3;         // two waves of XR 1, three of XR 8 to a CU
  static constexpr int LDS = RING * STAGE;
  static constexpr int AHEAD = 3;                                // chunks read from LDS ahead of their matrix ops

  struct Chunk {  // 32 k in registers
    u32x4 c;
    h8v x[2];
    uint32_t s;
  };
  uint8_t* lds;         // this wave's ring
  const int8_t* w[4];   // codes of tile row 8 p + lane / 8
  const uint16_t* sc;   // scales of tile row lane % 32
  const uint16_t* x[2]; // X row 4 p + lane / 16 (XR 8)
  int K, ng;
  float per_unit;       // groups per unit

  // row(c): the weight row of tile row c.  X row r at x + r * x_ld, r < x_rows <= XR (the last one beyond).
  template <class Row>
  __device__ __forceinline__ RowDot(uint8_t* lds_, const uint16_t* x_, int64_t x_ld, int x_rows,
                                    const int8_t* codes, const uint16_t* scale, int K_, int group, const Row& row)
      : lds(lds_), K(K_), ng(K_ / group), per_unit(1.0f / (float)(group / UNIT)) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int p = 0; p < 4; ++p) w[p] = codes + row(8 * p + (lane >> 3)) * (int64_t)K;
    sc = scale + row(lane & 31) * (int64_t)ng;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int r = XR == 1 ? 0 : 4 * p + (lane >> 4);
      x[p] = x_ + (r < x_rows ? r : x_rows - 1) * x_ld;
    }
  }

  // Stage s to ring buffer b: per 128 k the 32 rows' codes (16-byte piece c of
  // row r at c ^ (r / 2 % 8)) and, XR 8, the X rows (piece c of row r at c ^ r),
  // so that the lanes that read one piece of all rows hit different banks; XR 1, X
  // as it is.  Past K the last pieces are read again (and not used).
  __device__ __forceinline__ void load(int s, int b) const {
    const int lane = threadIdx.x & 63;
    const uint32_t to = lds_addr(lds) + (uint32_t)(b * STAGE);
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      const int r = 8 * (i & 3) + (lane >> 3), k = KS * s + 128 * (i >> 2) + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
      dma16(to + 1024u * i, (uint64_t)(uintptr_t)(w[i & 3] + (k < K ? k : K - 16)));
    }
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int k = KS * s + (XR == 1 ? 8 * lane : 128 * (i >> 1) + ((lane & 15) ^ (4 * (i & 1) + (lane >> 4))) * 8);
      dma16(to + (uint32_t)(WB + 1024 * i), (uint64_t)(uintptr_t)(x[i & 1] + (k < K ? k : K - 8)));
    }
#pragma unroll
    for (int q = 0; q < SU / 2; ++q) {
      // the unit's group: a division by multiplication, exact for these few units
      // (half a unit is far more than the product's error)
      const int u = s * SU + 2 * q + (lane >> 5);
      const int g = (int)(((float)u + 0.5f) * per_unit);
      dma2(to + (uint32_t)(WB + XB + 256 * q), (uint64_t)(uintptr_t)(sc + (g < ng ? g : ng - 1)));
    }
  }
  // At most n whole stages of this wave's loads are in flight (vmcnt counts to 63).
  __device__ __forceinline__ static void wait(int n) {
    if (n == 0)
      asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    else if (n == 1)
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"(NL) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * NL < 63 ? 2 * NL : 63) : "memory");
  }

  __device__ __forceinline__ void read(Chunk& f, const uint8_t* st, int ch) const {
    const int lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    f.c = *reinterpret_cast<const u32x4*>(st + 4096 * (ch >> 2) + l32 * 128 +
                                          ((2 * (ch & 3) + half) ^ ((l32 >> 1) & 7)) * 16);
    const int r = l32 >> 2;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      f.x[j] = *reinterpret_cast<const h8v*>(
          st + WB + (XR == 1 ? (4 * ch + 2 * half + j) * 16
                             : 2048 * (ch >> 2) + r * 256 + ((4 * (ch & 3) + 2 * half + j) ^ r) * 16));
    f.s = reinterpret_cast<const uint32_t*>(st + WB + XB)[32 * (PAIR ? ch >> 1 : 2 * ch + half) + l32];
  }
  __device__ __forceinline__ static void mul(const Chunk& f, f32x16& acc) {
    u32x4 lo, hi;
    dequant16(f.c, f.s * 0x10001u, lo, hi);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[0], h8_of(lo), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[1], h8_of(hi), acc, 0, 0, 0);
  }

  // The sums: XR 1, x . w of weight row lane % 32 in every register; XR 8, the
  // products of X row r in registers and halves 4 r .. 4 r + 3 of acc_row.
  __device__ __forceinline__ f32x16 dot() const {
    f32x16 acc = (f32x16){};
    const int nst = (K + KS - 1) / KS, whole = K / KS;
    for (int s = 0; s < RING && s < nst; ++s) load(s, s);
    int b = 0;
    for (int s = 0; s < whole; ++s) {
      wait(min(nst - 1 - s, RING - 1));
      const uint8_t* st = lds + b * STAGE;
      Chunk f[CH];
#pragma unroll
      for (int ch = 0; ch < AHEAD; ++ch) read(f[ch], st, ch);
#pragma unroll
      for (int ch = 0; ch < CH; ++ch) {
        if (ch + AHEAD < CH) read(f[ch + AHEAD], st, ch + AHEAD);
        __builtin_amdgcn_sched_barrier(0);  // or the compiler moves the reads to their uses
        mul(f[ch], acc);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (s + RING < nst) {
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // the stage is in registers
        load(s + RING, b);
      }
      b = b == RING - 1 ? 0 : b + 1;
    }
    if (whole < nst) {
      wait(0);
      const int left = K - KS * whole, half = (threadIdx.x >> 5) & 1;
      for (int ch = 0; 32 * ch < left; ++ch) {
        Chunk f;
        read(f, lds + b * STAGE, ch);
        if (!PAIR && 32 * ch + 16 * half >= left) f.s = 0u, f.x[0] = f.x[1] = (h8v){};
        mul(f, acc);
      }
    }
    return acc;
  }
};

}  // namespace lemoq_gemm
