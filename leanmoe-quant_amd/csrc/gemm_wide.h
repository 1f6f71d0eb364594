// Matrix-core main loop of the prefill GEMMs on quantised weights (X W^T, X
// fp16 rows, W codes with group scales), both operands brought to LDS by
// direct loads.
//
// A block of WN waves computes up to 32 MF rows x 32 FN WN weight rows with
// v_mfma_f32_32x32x16_f16; every wave takes all of the block's rows and its
// own 32 FN weight rows.  K advances in stages of 64 through a ring of RING
// LDS buffers filled by global_load_lds_dwordx4: X as fp16, W as its codes.
// There are no staging registers, and the codes become the fp16 weights of the
// reference's multi-token arm (fp16 of code * scale, (code - zero) * scale or
// e2m1 * 2^(X - 127)) in registers, once per wave that uses them.
#pragma once

#include <type_traits>

#include "gemm_core.h"
#include "lds_dma.h"

namespace lemoq_gemm {

// Weight formats (LEMOQ_QFMT_*): BITS per code; how the 16 codes of a lane's
// half chunk (u32x4 or uint2, code i at bit BITS * i) and the raw scale and
// zero of their group become 16 fp16 weights; VALU, about how many
// instructions that takes.
struct WideW8 {  // int8, fp16 scale
  static constexpr int BITS = 8, VALU = 28;
  static constexpr bool ZERO = false;
  using Codes = u32x4;
  static __device__ __forceinline__ void weights(const u32x4 c, uint32_t s, uint32_t, u32x4& lo, u32x4& hi) {
    dequant16(c, s * 0x10001u, lo, hi);
  }
};
struct WideW4 {  // int4, fp16 scale; as WideW8, the pair of a byte by one permute, one mask and one exact fma
  static constexpr int BITS = 4, VALU = 32;
  static constexpr bool ZERO = false;
  using Codes = uint2;
  static __device__ __forceinline__ void weights(const uint2 c, uint32_t s, uint32_t, u32x4& lo, u32x4& hi) {
    const f16x2 sc = as_h2(s * 0x10001u);
    const f16x2 mul = {(f16)1.0f, (f16)0.0625f}, sub = {(f16)-1032.0f, (f16)-72.0f};
    uint32_t o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t w = i < 4 ? c.x : c.y;
      // 1024 + u and 1024 + 16 u of the offset-binary nibbles u = code + 8
      const uint32_t t = __builtin_amdgcn_perm(0u, w, 0x0C000C00u + 0x00010001u * (uint32_t)(i & 3));
      const f16x2 v = __builtin_elementwise_fma(as_h2((t & 0x00F0000Fu) ^ 0x64806408u), mul, sub);
      o[i] = __builtin_bit_cast(uint32_t, v * sc);
    }
    lo = (u32x4){o[0], o[1], o[2], o[3]};
    hi = (u32x4){o[4], o[5], o[6], o[7]};
  }
};
// The other formats in fp32, as the reference's dequantised weight.
__device__ __forceinline__ void wide_round16(const float (&v)[16], u32x4& lo, u32x4& hi) {
  uint32_t o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = __builtin_bit_cast(uint32_t, f2h2(v[2 * i], v[2 * i + 1]));
  lo = (u32x4){o[0], o[1], o[2], o[3]};
  hi = (u32x4){o[4], o[5], o[6], o[7]};
}
struct WideW8Asym {  // uint8, fp16 scale and zero
  static constexpr int BITS = 8, VALU = 58;
  static constexpr bool ZERO = true;
  using Codes = u32x4;
  static __device__ __forceinline__ void weights(const u32x4 c, uint32_t s, uint32_t z, u32x4& lo, u32x4& hi) {
    const uint32_t w[4] = {c.x, c.y, c.z, c.w};
    const float sf = h2f((uint16_t)s), zf = h2f((uint16_t)z);
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = ((float)((w[i >> 2] >> (8 * (i & 3))) & 0xFFu) - zf) * sf;
    wide_round16(v, lo, hi);
  }
};
struct WideW4Asym {  // uint4, fp16 scale and zero
  static constexpr int BITS = 4, VALU = 64;
  static constexpr bool ZERO = true;
  using Codes = uint2;
  static __device__ __forceinline__ void weights(const uint2 c, uint32_t s, uint32_t z, u32x4& lo, u32x4& hi) {
    const float sf = h2f((uint16_t)s), zf = h2f((uint16_t)z);
    float v[16];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const uint32_t w = d ? c.y : c.x, even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        v[8 * d + 2 * b] = ((float)((even >> (8 * b)) & 0xFFu) - zf) * sf;
        v[8 * d + 2 * b + 1] = ((float)((odd >> (8 * b)) & 0xFFu) - zf) * sf;
      }
    }
    wide_round16(v, lo, hi);
  }
};
struct WideMx4 {  // E2M1, E8M0 byte: X = 0 is 2^-127, X = 255 overflows to +inf
  static constexpr int BITS = 4, VALU = 48;
  static constexpr bool ZERO = false;
  using Codes = uint2;
  static __device__ __forceinline__ void weights(const uint2 c, uint32_t s, uint32_t, u32x4& lo, u32x4& hi) {
    const float sf = as_f32(s == 0u ? 0x00400000u : s << 23);
    float v[16];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const uint32_t w = d ? c.y : c.x;
      const f16x2 p[4] = {__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0),
                          __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1),
                          __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2),
                          __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3)};
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        v[8 * d + 2 * b] = (float)p[b].x * sf;
        v[8 * d + 2 * b + 1] = (float)p[b].y * sf;
      }
    }
    wide_round16(v, lo, hi);
  }
};

template <class Q_, int MF_, int FN_, int WN_, int RING_, int MAXG_>
struct WideGeo {
  using Q = Q_;
  static constexpr int MF = MF_, FN = FN_, WN = WN_, RING = RING_;
  static constexpr int MAXG = MAXG_;             // scale groups along K that fit beside the ring
  static constexpr int NT = 64 * WN;             // threads
  static constexpr int BM = 32 * MF, BN = 32 * FN * WN;
  static constexpr int RB = BK * Q::BITS / 8;    // code bytes of a row and stage
  static constexpr int LPR = RB / 16;            // lanes that load them
  static constexpr int XB = BM * BK * 2;         // X bytes of a stage
  static constexpr int STAGE = XB + BN * RB;     // and the codes
  static constexpr int SCALES = RING * STAGE;    // byte offset of the scales [group][BN], then the zeros
  static constexpr int LDS = SCALES + MAXG * BN * 2 * (Q::ZERO ? 2 : 1);
  static constexpr int CR = 64 / LPR * WN;       // weight rows of a pass of code loads
  static constexpr int XP = BM / (8 * WN);       // direct loads per wave and stage: X rows (all MF) ...
  static constexpr int CP = BN / CR;             // ... and codes
  static_assert(BM % (8 * WN) == 0 && 4 % WN == 0 && BN % CR == 0, "whole passes of loads");
};

// A lane's sources: byte offsets from the (block-uniform) bases xb and cb, or,
// for gathered X rows (GATHER), addresses in xo and no xb; for rows too long for
// 32-bit offsets (FAR, with GATHER) addresses in co too, and no cb.
template <class G, bool GATHER, bool FAR = false>
struct WideSrc {
  static_assert(GATHER || !FAR, "far rows");
  const uint8_t* xb;
  const uint8_t* cb;
  std::conditional_t<GATHER, uint64_t, uint32_t> xo[G::XP];  // pass p: tile row 8 WN p + 8 wave + lane / 8
  std::conditional_t<FAR, uint64_t, uint32_t> co[G::CP];     // pass p: weight row wide_c_row
};

// Tile row of this lane in pass p of the X / code loads, and the 16-byte
// chunk it fetches.  A load writes lane l's 16 bytes at LDS base + 16 l, so
// rows lie back to back (128 B of X, 64 or 32 B of codes) and the chunk is
// XORed with the row (X: (row >> 1) & 7, codes: (row >> 2) & 3 or (row >> 3) &
// 1): 16 lanes that read one chunk of 16 consecutive rows then hit 16
// different bank groups (4-bit codes, 8 bytes a lane: half as many).
template <class G>
__device__ __forceinline__ int wide_x_row(int p, int wave, int lane) {
  return 8 * G::WN * p + 8 * wave + (lane >> 3);
}
__device__ __forceinline__ uint32_t wide_x_chunk(int row, int lane) {
  return (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
}
template <class G>
__device__ __forceinline__ int wide_c_row(int p, int wave, int lane) {
  return G::CR * p + 64 / G::LPR * wave + lane / G::LPR;
}
template <class G>
__device__ __forceinline__ int wide_c_swizzle(int row) {
  return G::LPR == 4 ? (row >> 2) & 3 : (row >> 3) & 1;
}
template <class G>
__device__ __forceinline__ uint32_t wide_c_chunk(int row, int lane) {
  return (uint32_t)(((lane % G::LPR) ^ wide_c_swizzle<G>(row)) * 16);
}

// This wave's LDS reads are done and at most N of its direct loads are in
// flight, in every wave of the block.
template <int N>
__device__ __forceinline__ void wide_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

// The K loop over nst stages of a block with NF fragments of 32 rows; cpg
// 32-k chunks share a scale group (WideW8: an even number).  This wave's weight rows are the fragments at
// tile rows b_row0[0 .. FN-1].  `put_scales(g0)` writes the block's scales of
// groups g0 .. g0 + MAXG - 1 to LDS: for g0 = 0 once the first loads are out,
// then whenever a long K has used up the MAXG that fit.  On return no direct load is in
// flight, and a barrier frees the LDS.
template <class G, int NF, bool GATHER, bool FAR, class PutScales>
__device__ __forceinline__ void wide_mainloop(f32x16 (&acc)[G::MF][G::FN], const WideSrc<G, GATHER, FAR>& src, int nst,
                                              int cpg, uint8_t* lds, const int (&b_row0)[G::FN],
                                              const PutScales& put_scales) {
  using Q = typename G::Q;
  constexpr int FN = G::FN, R = G::RING;
  constexpr int XP = (32 * NF + 8 * G::WN - 1) / (8 * G::WN), VM = XP + G::CP;  // loads per wave and stage
  constexpr int DQ_VALU = Q::VALU * FN;                                              // of one chunk's dequantisation
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const uint32_t lds0 = lds_addr(lds);
  const int last = nst - 1;
  auto load = [&](int p, int buf, int stage) {
    const uint32_t to = lds0 + (uint32_t)(buf * G::STAGE);
    if (p < XP) {
      const uint32_t row = to + (uint32_t)(8 * G::WN * p + 8 * wave) * 128u;
      if constexpr (FAR)
        dma16(row, src.xo[p] + (uint64_t)stage * (BK * 2));
      else if constexpr (GATHER)
        dma16(row, src.xo[p] + (uint32_t)stage * (BK * 2));
      else
        dma16(row, src.xo[p], src.xb + (int64_t)stage * (BK * 2));
    } else {
      const uint32_t row = to + (uint32_t)(G::XB + (G::CR * (p - XP) + 64 / G::LPR * wave) * G::RB);
      if constexpr (FAR)
        dma16(row, src.co[p - XP] + (uint64_t)stage * G::RB);
      else
        dma16(row, src.co[p - XP], src.cb + (int64_t)stage * G::RB);
    }
  };
  // the ring starts with stages 0 .. R - 1 (clamped: a re-read is harmless)
#pragma unroll
  for (int b = 0; b < R; ++b)
#pragma unroll
    for (int p = 0; p < VM; ++p) load(p, b, b < last ? b : last);
  put_scales(0);
  wide_wait<(R - 1) * VM>();

  // LDS byte offsets of this lane's reads within a stage
  const int sx = (l32 >> 1) & 7, sb = wide_c_swizzle<G>(l32);
  uint32_t xa[4], ca[2];  // 16-k step q; 32-k chunk c
#pragma unroll
  for (int q = 0; q < 4; ++q) xa[q] = (uint32_t)(l32 * 128 + (((4 * (q >> 1) + 2 * half + (q & 1)) ^ sx) * 16));
#pragma unroll
  for (int c = 0; c < 2; ++c)  // 16 codes: one 16-byte chunk, or half of one
    ca[c] = (uint32_t)(G::XB + l32 * G::RB + (G::LPR == 4 ? ((2 * c + half) ^ sb) * 16 : (c ^ sb) * 16 + half * 8));
  const uint16_t* sc = reinterpret_cast<const uint16_t*>(lds + G::SCALES) + l32;

  h8v a[3][NF];      // X fragments of 16-k steps
  typename Q::Codes codes[FN];  // codes of a 32-k chunk
  h8v b[FN][2];                 // the chunk's weights, [n][16-k step]
  uint32_t s16[FN], z16[FN];    // the group's scales and zeros
  auto read_a = [&](h8v(&d)[NF], uint32_t base, int q) {
#pragma unroll
    for (int i = 0; i < NF; ++i) d[i] = *reinterpret_cast<const h8v*>(lds + base + xa[q] + 4096 * i);
  };
  auto read_c = [&](uint32_t base, int c) {
#pragma unroll
    for (int n = 0; n < FN; ++n)
      codes[n] = *reinterpret_cast<const typename Q::Codes*>(lds + base + ca[c] + b_row0[n] * G::RB);
  };
  auto read_s = [&](int g) {
#pragma unroll
    for (int n = 0; n < FN; ++n) {
      s16[n] = sc[g * G::BN + b_row0[n]];
      z16[n] = Q::ZERO ? sc[(G::MAXG + g) * G::BN + b_row0[n]] : 0;
    }
  };
  auto dq = [&](h8v(&o)[FN][2]) {
#pragma unroll
    for (int n = 0; n < FN; ++n) {
      u32x4 lo, hi;
      Q::weights(codes[n], s16[n], z16[n], lo, hi);
      o[n][0] = h8_of(lo);
      o[n][1] = h8_of(hi);
    }
  };
  auto mm1 = [&](const h8v(&d)[NF], int j, int i) {
#pragma unroll
    for (int n = 0; n < FN; ++n) acc[i][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(d[i], b[n][j], acc[i][n], 0, 0, 0);
  };
  auto mm = [&](const h8v(&d)[NF], int j) {
#pragma unroll
    for (int i = 0; i < NF; ++i) mm1(d, j, i);
  };
  // one 16-k step with the next chunk's dequantisation between its matrix ops
  auto mm_dq = [&](const h8v(&d)[NF], int j) {
    h8v nb[FN][2];
    dq(nb);
    mm(d, j);
#pragma unroll
    for (int i = 0; i < FN * NF; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                      // one matrix op
      __builtin_amdgcn_sched_group_barrier(0x2, DQ_VALU / (FN * NF), 0);    // its share of the VALU work
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < FN; ++n) b[n][0] = nb[n][0], b[n][1] = nb[n][1];
  };
  // the rest of a stage's reads and its first two 16-k steps
  int buf = 0, gi = 0, gc = 0, g0 = 0;
  auto advance = [&]() {  // to the next chunk's scale group
    if (++gc == cpg) gc = 0, ++gi;
  };
  auto front = [&](uint32_t base) {
    advance();
    if constexpr (!std::is_same_v<Q, WideW8>) read_s(gi);
    read_a(a[1], base, 1);
    read_c(base, 1);
    __builtin_amdgcn_sched_barrier(0);
    mm(a[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    read_a(a[0], base, 2);
    read_a(a[2], base, 3);
    __builtin_amdgcn_sched_barrier(0);
    mm_dq(a[1], 1);
  };
  // From stage s to s + 1: the last two 16-k steps of s run after the barrier
  // that hands over its buffer, over the first reads of s + 1.
  auto next = [&](int s, auto more) {
    constexpr bool MORE = decltype(more)::value;
    wide_wait<MORE ? (R - 2) * VM : 0>();  // stage s is read by all, stage s + 1 has landed for all
    const int freed = buf;
    buf = buf == R - 1 ? 0 : buf + 1;
    advance();
    if (gi == G::MAXG) {  // every wave has read its last scales before the barrier above
      gi = 0, g0 += G::MAXG;
      put_scales(g0);
      wide_wait<0>();
    }
    const uint32_t base = (uint32_t)(buf * G::STAGE);
    read_s(gi);
    read_c(base, 0);
    __builtin_amdgcn_sched_barrier(0);
    int p = 0;
#pragma unroll
    for (int i = 0; i < NF; ++i) {  // stage s + R's loads go out between the matrix ops
      mm1(a[0], 0, i);
      if constexpr (MORE) {
        const int end = ((i + 1) * VM) / NF;
#pragma unroll
        for (int pp = 0; pp < VM; ++pp)
          if (pp >= p && pp < end) load(pp, freed, s + R);
        p = end;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    read_a(a[0], base, 0);
    __builtin_amdgcn_sched_barrier(0);
    mm_dq(a[2], 1);
    front(base);
  };
  read_s(0);
  read_c(0, 0);
  read_a(a[0], 0, 0);
  dq(b);
  front(0);
  int s = 0;
  for (; s < nst - R; ++s) next(s, std::true_type{});
  for (; s < nst - 1; ++s) next(s, std::false_type{});
  if (nst == 1) wide_wait<0>();  // the ring's re-reads (the last `next` waits for them otherwise): the caller reuses the LDS
  mm(a[0], 0);
  mm(a[2], 1);
}

// The block's scales (and zeros): thread t owns tile weight row t % BN, whose
// fp16 scales start at `row` (zeros at `zrow`; bytes for WideMx4), ng of them;
// g_base is a multiple of MAXG.  With `vec` (ng a multiple of 8, rows 16-byte
// aligned) the scales move as 16-byte chunks, the first two per thread loaded
// at construction so that their latency is under the first direct loads.
template <class G>
struct WideScales {
  static constexpr int TPR = G::NT / G::BN;  // threads per weight row
  static_assert(G::NT % G::BN == 0 && G::MAXG % 8 == 0, "scale rows");
  using Raw = std::conditional_t<std::is_same_v<typename G::Q, WideMx4>, uint8_t, uint16_t>;
  const Raw *row, *zrow;
  int ng, vec;
  u32x4 pre[2];
  __device__ __forceinline__ WideScales(const Raw* row_, const Raw* zrow_, int ng_, int vec_)
      : row(row_), zrow(zrow_), ng(ng_), vec(vec_) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = part() + TPR * i;
      pre[i] = vec && 8 * c < ng ? *reinterpret_cast<const u32x4*>(row + 8 * c) : (u32x4){0u, 0u, 0u, 0u};
    }
  }
  __device__ static int part() { return TPR > 1 ? (int)threadIdx.x / G::BN : 0; }
  __device__ __forceinline__ void put(uint8_t* lds, int g_base) const {
    uint16_t* to = reinterpret_cast<uint16_t*>(lds + G::SCALES) + (int)threadIdx.x % G::BN;
    const int n = ng - g_base < G::MAXG ? ng - g_base : G::MAXG;
    if constexpr (G::Q::ZERO)
      for (int g = part(); g < n; g += TPR) to[(G::MAXG + g) * G::BN] = zrow[g_base + g];
    if (!vec) {
      for (int g = part(); g < n; g += TPR) to[g * G::BN] = row[g_base + g];
      return;
    }
    auto chunk = [&](int c, const u32x4 v) {
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) to[(8 * c + j) * G::BN] = (uint16_t)(w[j >> 1] >> (16 * (j & 1)));
    };
    int c = part();
    if (g_base == 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i, c += TPR)
        if (8 * c < n) chunk(c, pre[i]);
    }
    for (; 8 * c < n; c += TPR) chunk(c, *reinterpret_cast<const u32x4*>(row + g_base + 8 * c));
  }
};

// Runs f(NF) (an integral constant) for nf = 1 .. MF fragments.
template <int MF, class F>
__device__ __forceinline__ void wide_dispatch(int nf, const F& f) {
  if constexpr (MF > 1) {
    if (nf < MF) return wide_dispatch<MF - 1>(nf, f);
  }
  f(std::integral_constant<int, MF>{});
}

}  // namespace lemoq_gemm
