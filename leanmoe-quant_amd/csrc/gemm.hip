// Batched (prefill) GEMM on the gfx950 matrix cores: Y = X W^T with X (M, K)
// fp16 and W (N, K) either w8 (int8 codes + fp16 scales per group of 128
// along K) or fp16, fp32 accumulation.
//
// The w8 path dequantises W exactly as the reference's separate path does
// before its F.linear (QuantLinear.forward for T > 1, src/lemoq/quant/
// linear.py:365-395, 471-480): w = fp16(code * scale_fp16) -- the exact
// code, converted to fp16, times the fp16 scale in one fp16 rounding
// (v_pk_mul_f16).
//
// Tiling: w8 weights run on the direct-load main loop of gemm_wide.h, in one
// of three block shapes chosen by how the tiles fill the CUs (tile_pick), one row
// of them on row_gemm.h's wave per 32 columns; fp16 weights on the
// register-staged pipeline of gemm_core.h.  Tiles are numbered
// n-major (consecutive tiles share the weight tile) and each XCD takes a
// contiguous range of them.
//
// Rows: X row m may be gathered (x_rows[m]); the output is fp16 rows with an
// optional fp16 residual added in one rounding (torch's fp16 add).  Rows and
// columns beyond M/N are clamped on load and not stored.  When the output
// (and residual) rows are 16-byte aligned, the block stages its fp16 tile in
// LDS and writes whole row segments in 16-byte chunks; otherwise each lane
// stores its own elements.
#include "gemm_wide.h"
#include "row_gemm.h"

#include <mutex>

namespace {

using namespace lemoq_gemm;

struct GemmArgs {
  const uint16_t* x;       // (rows, x_ld) fp16
  int64_t x_ld;
  const int32_t* x_rows;   // optional gather (M)
  int64_t M, N, K;
  const uint8_t* codes;    // quantised: (N, K) codes, K / 2 bytes a row at 4 bits
  const void* scale;       // quantised: (N, K/group) fp16 (E8M0 bytes for MXFP4)
  const void* zero;        // asymmetric: (N, K/group) fp16
  const uint16_t* w16;     // fp16 weights (N, K) (when codes == nullptr)
  int group;
  uint16_t* y16;           // fp16 out (M, y_ld)
  int64_t y_ld;
  const uint16_t* resid;   // optional fp16 residual (M, resid_ld)
  int64_t resid_ld;
  int splits;              // K ranges (blockIdx.y); > 1 writes fp32 partials
  float* part;             // (splits, M, N) fp32 partials when splits > 1
  int row_out;             // fp16 rows written as 16-byte chunks (set by the host)
  int scale_vec;           // quantised: scale rows move as 16-byte chunks (set by the host)
  int row_tiles;           // quantised: row tiles, the 32-row fragments dealt evenly over them (set by the host)
};

// fp16 residual added to 8 fp16 values, one rounding each (torch's fp16 add).
__device__ __forceinline__ u32x4 add_resid8(const u32x4 v, const u32x4 rv) {
  const uint32_t in[4] = {v.x, v.y, v.z, v.w}, ri[4] = {rv.x, rv.y, rv.z, rv.w};
  uint32_t o[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint16_t lo = hadd_round(h2f((uint16_t)(in[q] & 0xFFFFu)), (uint16_t)(ri[q] & 0xFFFFu));
    const uint16_t hi = hadd_round(h2f((uint16_t)(in[q] >> 16)), (uint16_t)(ri[q] >> 16));
    o[q] = (uint32_t)lo | ((uint32_t)hi << 16);
  }
  return (u32x4){o[0], o[1], o[2], o[3]};
}

// fp16 weights.
template <int BM, int BN, int WM = 2>
__global__ __launch_bounds__(128 * WM) void gemm_kernel(const GemmArgs a) {
  using TL = Tile<BM, BN, WM, 2>;
  __shared__ __align__(16) uint16_t lds[TL::LDS_ELEMS];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int half = lane >> 5, l32 = lane & 31;
  const int64_t nbm = (a.M + BM - 1) / BM, nbn = (a.N + BN - 1) / BN;
  const int64_t tile = xcd_tile(blockIdx.x, nbm * nbn);
  const int64_t m0 = (tile % nbm) * BM, n0 = (tile / nbm) * BN;
  const int z = blockIdx.y;
  const int64_t klen = a.K / a.splits, kb = z * klen;  // this block's K range

  Sources<TL> src;
#pragma unroll
  for (int i = 0; i < TL::A_CH; ++i) {
    int64_t m = m0 + TL::a_row(t, i);
    m = m < a.M ? m : a.M - 1;
    const int64_t row = a.x_rows ? (int64_t)a.x_rows[m] : m;
    src.a[i] = a.x + row * a.x_ld + kb + TL::a_col(t, i);
  }
#pragma unroll
  for (int i = 0; i < TL::B_CH; ++i) {
    int64_t n = n0 + TL::b_row(t, i);
    n = n < a.N ? n : a.N - 1;
    src.b[i] = a.w16 + n * a.K + kb + TL::b_col(t, i);
  }
  const int wm = wave >> 1, wn = wave & 1;  // WM x 2 waves
  int b_row0[TL::FN];
#pragma unroll
  for (int j = 0; j < TL::FN; ++j) b_row0[j] = wn * (BN / 2) + 32 * j;
  Acc<TL::FM, TL::FN> acc;
  block_mainloop2<TL>(acc, src, klen, lds, wm * (BM / WM), b_row0);

  if (a.row_out) {  // block-uniform
    // fp16(acc) into the (then idle) stage buffers as a BM x BN row-major
    // tile, then each row segment goes out in 16-byte chunks with the
    // residual added per chunk: the same roundings as the per-element path.
    constexpr int OP = BN + 8, CPR = BN / 8, RPI = TL::NT / CPR;
    static_assert(BM * OP <= TL::LDS_ELEMS && TL::NT % CPR == 0, "output tile");
    __syncthreads();  // every wave has read its last stage from LDS
#pragma unroll
    for (int i = 0; i < TL::FM; ++i)
#pragma unroll
      for (int j = 0; j < TL::FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          lds[(wm * (BM / WM) + 32 * i + acc_row(r, half)) * OP + wn * (BN / 2) + 32 * j + l32] =
              f2h(acc.v[i][j][r]);
    __syncthreads();
    const int c8 = (t % CPR) * 8;
    const int64_t n = n0 + c8;
    if (n >= a.N) return;  // N % 8 == 0: a chunk is wholly inside or outside
    const int rows = (int)(a.M - m0 < BM ? a.M - m0 : BM);
    for (int row = t / CPR; row < rows; row += RPI) {
      u32x4 v = *reinterpret_cast<const u32x4*>(lds + row * OP + c8);
      if (a.resid) v = add_resid8(v, *reinterpret_cast<const u32x4*>(a.resid + (m0 + row) * a.resid_ld + n));
      *reinterpret_cast<u32x4*>(a.y16 + (m0 + row) * a.y_ld + n) = v;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < TL::FM; ++i)
#pragma unroll
    for (int j = 0; j < TL::FN; ++j) {
      const int64_t n = n0 + wn * (BN / 2) + 32 * j + l32;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t m = m0 + wm * (BM / WM) + 32 * i + acc_row(r, half);
        if (m >= a.M || n >= a.N) continue;
        if (a.part) {
          a.part[((int64_t)z * a.M + m) * a.N + n] = acc.v[i][j][r];
          continue;
        }
        uint16_t o = f2h(acc.v[i][j][r]);
        if (a.resid) o = hadd_round(h2f(o), a.resid[m * a.resid_ld + n]);
        a.y16[m * a.y_ld + n] = o;
      }
    }
}

// Split-K finish: y = fp16(sum over z of part[z]) in z order (+ residual).
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int splits, int64_t M,
                                                           int64_t N, uint16_t* __restrict__ y, int64_t y_ld,
                                                           const uint16_t* __restrict__ resid, int64_t resid_ld) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * N) return;
  const int64_t m = idx / N, n = idx - m * N;
  float v = 0.0f;
  for (int z = 0; z < splits; ++z) v += part[z * M * N + idx];
  uint16_t o = f2h(v);
  if (resid) o = hadd_round(h2f(o), resid[m * resid_ld + n]);
  y[m * y_ld + n] = o;
}

// Quantised weights: one block per (row tile, BN columns) on gemm_wide.h's main loop.
// Bound by the chip's power and the matrix units at many rows, by the latency
// of the K loop's stages at few (about 0.35 us a stage of 64).  On 6144 x 2048
// and 2048 x 2048 weights against the register-staged 256 x 128, 128 x 128 and
// 64 x 64 tiles before, us (MI355X): 6144 columns, 75 rows 14.2 -> 12.9, 317
// 19.5 -> 15.9, 700 43.9 -> 28.3, 1024 36.3 -> 34.6, 2048 73.4 -> 62, 4096 126
// -> 104; 2048 columns, 75 rows 14.3 -> 12.8, 1024 21.6 -> 18.6, 1500 29.5 ->
// 24.6, 4096 46.5 -> 45.6.  Bit-identical: the same products in the same order.
// The other formats (4-bit, asymmetric, MXFP4) were dequantised to an fp16
// weight first and then multiplied: 6144 x 2048 4-bit weights, 317 rows, 37.1
// -> 18.1 us.
template <class G, bool GATHER, bool FAR = false>
__global__ __launch_bounds__(G::NT, 2) void gemm_q_kernel(const GemmArgs a) {
  constexpr int OP = G::BN + 8;  // pitch of the output tile that the idle ring holds at the end (fp16)
  __shared__ __align__(1024) uint8_t lds[G::LDS > G::BM * OP * 2 ? G::LDS : G::BM * OP * 2];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int64_t nbn = (a.N + G::BN - 1) / G::BN;
  const int64_t tile = xcd_tile(blockIdx.x, a.row_tiles * nbn);
  const int64_t tm = tile % a.row_tiles, n0 = tile / a.row_tiles * G::BN;
  const int64_t frags = (a.M + 31) >> 5, fq = frags / a.row_tiles, fr = frags % a.row_tiles;
  const int64_t m0 = 32 * (tm * fq + (tm < fr ? tm : fr));
  const int nf = (int)(fq + (tm < fr ? 1 : 0));
  const int rows = (int)(a.M - m0 < 32 * nf ? a.M - m0 : 32 * nf);
  const int64_t ng = a.K / a.group;
  // weight row of tile row r, from n0 (clamped: columns past N are not stored)
  auto wrow = [&](int r) { return n0 + r < a.N ? r : (int)(a.N - 1 - n0); };
  using Raw = typename WideScales<G>::Raw;
  const int64_t srow = (n0 + wrow(t % G::BN)) * ng;
  const WideScales<G> sc(reinterpret_cast<const Raw*>(a.scale) + srow, reinterpret_cast<const Raw*>(a.zero) + srow,
                         (int)ng, a.scale_vec);
  WideSrc<G, GATHER, FAR> src;
#pragma unroll
  for (int p = 0; p < G::XP; ++p) {
    const int r = wide_x_row<G>(p, wave, lane);
    const int m = r < rows ? r : rows - 1;
    if constexpr (GATHER) {
      const int64_t row = a.x_rows ? (int64_t)a.x_rows[m0 + m] : m0 + m;
      src.xo[p] = (uint64_t)(uintptr_t)(a.x + row * a.x_ld) + wide_x_chunk(r, lane);
    } else {
      src.xo[p] = (uint32_t)(m * (2 * a.x_ld)) + wide_x_chunk(r, lane);
    }
  }
  src.xb = reinterpret_cast<const uint8_t*>(a.x + m0 * a.x_ld);
  const int64_t row_bytes = a.K * G::Q::BITS / 8;
  src.cb = a.codes + n0 * row_bytes;
#pragma unroll
  for (int p = 0; p < G::CP; ++p) {
    const int r = wide_c_row<G>(p, wave, lane);
    if constexpr (FAR)
      src.co[p] = (uint64_t)(uintptr_t)(src.cb + wrow(r) * row_bytes) + wide_c_chunk<G>(r, lane);
    else
      src.co[p] = (uint32_t)(wrow(r) * row_bytes) + wide_c_chunk<G>(r, lane);
  }
  int b_row0[G::FN];
#pragma unroll
  for (int j = 0; j < G::FN; ++j) b_row0[j] = 32 * (G::FN * wave + j);
  f32x16 acc[G::MF][G::FN];
#pragma unroll
  for (int i = 0; i < G::MF; ++i)
#pragma unroll
    for (int j = 0; j < G::FN; ++j) acc[i][j] = (f32x16){};
  wide_dispatch<G::MF>(nf, [&](auto nfc) {
    wide_mainloop<G, decltype(nfc)::value, GATHER, FAR>(acc, src, (int)(a.K / BK), a.group / 32, lds, b_row0,
                                                        [&](int g0) { sc.put(lds, g0); });
  });
  if (a.row_out) {  // as gemm_kernel: through LDS (the idle ring), 16-byte chunks of whole rows
    constexpr int CPR = G::BN / 8, RPI = G::NT / CPR;
    static_assert(G::NT % CPR == 0, "output tile");
    uint16_t* o = reinterpret_cast<uint16_t*>(lds);
    __syncthreads();  // every wave has read its last stage from LDS
#pragma unroll
    for (int i = 0; i < G::MF; ++i) {
      if (i >= nf) break;
#pragma unroll
      for (int j = 0; j < G::FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[(32 * i + acc_row(r, half)) * OP + b_row0[j] + l32] = f2h(acc[i][j][r]);
    }
    __syncthreads();
    const int c8 = (t % CPR) * 8;
    const int64_t n = n0 + c8;
    if (n >= a.N) return;  // N % 8 == 0: a chunk is wholly inside or outside
    for (int row = t / CPR; row < rows; row += RPI) {
      u32x4 v = *reinterpret_cast<const u32x4*>(o + row * OP + c8);
      if (a.resid) v = add_resid8(v, *reinterpret_cast<const u32x4*>(a.resid + (m0 + row) * a.resid_ld + n));
      *reinterpret_cast<u32x4*>(a.y16 + (m0 + row) * a.y_ld + n) = v;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < G::MF; ++i) {
    if (i >= nf) break;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 32 * i + acc_row(r, half);
      if (row >= rows) continue;
#pragma unroll
      for (int j = 0; j < G::FN; ++j) {  // a row's neighbouring segments one after the other
        const int64_t n = n0 + b_row0[j] + l32;
        if (n >= a.N) continue;
        uint16_t o = f2h(acc[i][j][r]);
        if (a.resid) o = hadd_round(h2f(o), a.resid[(m0 + row) * a.resid_ld + n]);
        a.y16[(m0 + row) * a.y_ld + n] = o;
      }
    }
  }
}

// One row of int8 weights: a wave per 32 columns (row_gemm.h), the same bits as
// the tiles below, which for one row leave most of the chip idle (16 blocks of 64
// x 128 on 2048 columns) and pay 0.4 us a stage.  One row / the tiles, us (weights
// from memory): K 2048, 64 columns 8.6 / 12.9, 2048 9.0 / 13.9, 6144 9.4 / 14.0,
// 16384 13.5 / 15.7, 20480 21.2 / 15.9; K 512, 2048 columns 3.9 / 5.8, 16384 5.4 /
// 6.7, 32768 8.7 / 7.7; K 4096, 4096 columns 15.8 / 24.2, 16384 23.0 / 26.8, 24576
// 38.6 / 30.3; K 8192, 8192 columns 31 / 46.  The rings let two blocks share a CU:
// above 512 blocks the tiles are the faster form.
constexpr int64_t ROW_MAX_N = 512 * RW_COLS;
__global__ __launch_bounds__(64) void gemm_w8_row_kernel(const GemmArgs a) {
  using Dot = RowDot<true, 1>;
  __shared__ __align__(1024) uint8_t lds[Dot::LDS];
  const int lane = threadIdx.x;
  const int64_t n0 = (int64_t)blockIdx.x * RW_COLS, n = n0 + (lane & 31);
  const int64_t m = a.x_rows ? (int64_t)a.x_rows[0] : 0;
  const Dot d(lds, a.x + m * a.x_ld, 0, 1, reinterpret_cast<const int8_t*>(a.codes),
              reinterpret_cast<const uint16_t*>(a.scale), (int)a.K, a.group,
              [&](int c) { return n0 + c < a.N ? n0 + c : a.N - 1; });
  uint16_t o = f2h(d.dot()[0]);
  if (lane >= 32 || n >= a.N) return;
  if (a.resid) o = hadd_round(h2f(o), a.resid[n]);
  a.y16[n] = o;
}

// Block shapes: two blocks per CU each (at most 80 KB of LDS).
template <class Q>
using QWide = WideGeo<Q, 4, 2, 4, 2, Q::ZERO ? 16 : 32>;   // 128 x 256
template <class Q>
using QMid = WideGeo<Q, 4, 1, 4, 3, Q::ZERO ? 16 : 32>;    // 128 x 128
template <class Q>
using QSmall = WideGeo<Q, 2, 1, 4, 4, Q::ZERO ? 16 : 32>;  // 64 x 128

// The shape and rows per tile with the least estimated time: a tile that has
// a CU to itself takes `one`, and every further tile of a CU adds `more`.  They
// rank the shapes and predict no time: measured at K = 2048 with CUs to spare
// (us), where a full round of 256 tiles takes longer (128 x 256: 40 us against 31)
// in every shape, and the stores at the end do not grow with K as the loop does.
// Few rows per tile cost matrix work for the weights' dequantisation, many leave
// CUs idle.  Rows that go out element by element (unaligned) cost every tile its
// 2-byte stores, the wide tiles most (one_e, more_e): 4099 columns, K = 1024, 512
// rows 17.1 us with the constants of aligned rows, 15.1 with these; 1500 rows 26.1
// / 24.2.  Of 198 sizes (K 1024, 2048, 4096; 1024 to 6144 columns, aligned or not;
// 32 to 4096 rows) with all five candidates timed, the one picked is within 4% of
// the best at 194; the others are 5, 7, 7 and 10% off (unaligned, 700 to 3000 rows).
struct TilePick {
  int shape, rows;
};
TilePick tile_pick(int64_t M, int64_t N, bool row_out) {
  struct Cand {
    int shape, rows, bn;
    double one, more;      // rows that go out in 16-byte chunks
    double one_e, more_e;  // element by element
  };
  static const Cand cand[] = {{0, 128, 256, 31.0, 31.0, 41.0, 35.0}, {0, 96, 256, 28.0, 27.0, 30.0, 28.0},
                              {1, 128, 128, 21.0, 20.0, 23.0, 20.0}, {2, 64, 128, 15.5, 13.5, 16.8, 11.4},
                              {2, 32, 128, 13.2, 9.8, 14.2, 9.8}};
  TilePick best{2, 32};
  double best_t = 0.0;
  for (const Cand& c : cand) {
    const int64_t tiles = ((M + c.rows - 1) / c.rows) * ((N + c.bn - 1) / c.bn);
    const int64_t per_cu = (tiles + 255) / 256;
    const double one = row_out ? c.one : c.one_e, all = per_cu * (row_out ? c.more : c.more_e);
    const double t = all > one ? all : one;
    if (best_t == 0.0 || t < best_t) best = {c.shape, c.rows}, best_t = t;
  }
  return best;
}

constexpr int64_t NEAR_K = 1LL << 23;  // a tile's 256 rows of codes have 32-bit offsets

template <class Q, bool GATHERS>
int launch_q(GemmArgs a, hipStream_t st) {
  if constexpr (std::is_same_v<Q, WideW8>) {
    if (a.M == 1 && a.N <= ROW_MAX_N && a.K <= NEAR_K) {
      hipLaunchKernelGGL(gemm_w8_row_kernel, dim3((unsigned)((a.N + RW_COLS - 1) / RW_COLS)), dim3(64), 0, st, a);
      LEMOQ_CHECK_LAUNCH();
    }
  }
  const int64_t ng = a.K / a.group;
  a.scale_vec = !std::is_same_v<Q, WideMx4> && ng % 8 == 0 && lemoq_aligned16(a.scale);
  if constexpr (std::is_same_v<Q, WideW8>) {
    if (a.K > NEAR_K) {  // longer rows: 64-bit row addresses, one block shape
      using G = QMid<Q>;
      a.row_tiles = (int)((a.M + G::BM - 1) / G::BM);
      hipLaunchKernelGGL((gemm_q_kernel<G, true, true>), dim3((unsigned)(a.row_tiles * ((a.N + G::BN - 1) / G::BN))),
                         dim3(G::NT), 0, st, a);
      LEMOQ_CHECK_LAUNCH();
    }
  }
  const TilePick pick = tile_pick(a.M, a.N, a.row_out != 0);
  a.row_tiles = (int)((a.M + pick.rows - 1) / pick.rows);
  // 64-bit row addresses for gathered rows, and for strides beyond a tile's 32-bit offsets
  const bool gather = GATHERS && (a.x_rows || a.x_ld >= (1LL << 22));
  auto go = [&](auto geo) {
    using G = decltype(geo);
    const int64_t blocks = a.row_tiles * ((a.N + G::BN - 1) / G::BN);
    if (gather)
      hipLaunchKernelGGL((gemm_q_kernel<G, GATHERS>), dim3((unsigned)blocks), dim3(G::NT), 0, st, a);
    else
      hipLaunchKernelGGL((gemm_q_kernel<G, false>), dim3((unsigned)blocks), dim3(G::NT), 0, st, a);
    LEMOQ_CHECK_LAUNCH();
  };
  if (pick.shape == 0) return go(QWide<Q>{});
  if (pick.shape == 1) return go(QMid<Q>{});
  return go(QSmall<Q>{});
}

int launch_f16(const GemmArgs& a, hipStream_t st) {
  if (a.splits > 1) {  // small grids: 64 x 64 tiles, one K range per blockIdx.y, then the ordered sum
    const int64_t tiles = ((a.M + 63) / 64) * ((a.N + 63) / 64);
    hipLaunchKernelGGL((gemm_kernel<64, 64>), dim3((unsigned)tiles, (unsigned)a.splits), dim3(256), 0, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    if (!a.y16) return LEMOQ_OK;  // partials only: the consumer sums them
    const int64_t n = a.M * a.N;
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a.part, a.splits,
                       a.M, a.N, a.y16, a.y_ld, a.resid, a.resid_ld);
    LEMOQ_CHECK_LAUNCH();
  }
  // Measured on the OLMoE linears (qkv, o_proj at 1 to 4096 rows): 256 x 128 tiles of 8
  // waves (each wave 64 x 64, the B tile shared by 4 row waves) are fastest while they give
  // at least 192 blocks; then 128 x 128 (8 waves of 32 x 64) from 256 blocks; below that, and
  // for fewer rows than a tile (padding rows cost matrix work), 64 x 64 tiles of 4 waves.
  const int64_t t256 = ((a.M + 255) / 256) * ((a.N + 127) / 128);
  const int64_t t128 = ((a.M + 127) / 128) * ((a.N + 127) / 128);
  if (a.M >= 256 && t256 >= 192) {
    hipLaunchKernelGGL((gemm_kernel<256, 128, 4>), dim3((unsigned)t256), dim3(512), 0, st, a);
  } else if (a.M >= 128 && t128 >= 256) {
    hipLaunchKernelGGL((gemm_kernel<128, 128, 4>), dim3((unsigned)t128), dim3(512), 0, st, a);
  } else {
    const int64_t small = ((a.M + 63) / 64) * ((a.N + 63) / 64);
    hipLaunchKernelGGL((gemm_kernel<64, 64>), dim3((unsigned)small), dim3(256), 0, st, a);
  }
  LEMOQ_CHECK_LAUNCH();
}

int launch_gemm(GemmArgs a, hipStream_t st, int fmt = LEMOQ_QFMT_W8) {
  // 16-byte row stores need 16-byte aligned rows of the output (and residual)
  a.row_out = a.splits == 1 && a.y16 && lemoq_aligned16(a.y16) && a.y_ld % 8 == 0 && a.N % 8 == 0 &&
              (!a.resid || (lemoq_aligned16(a.resid) && a.resid_ld % 8 == 0));
  switch (a.codes ? fmt : -1) {
    case LEMOQ_QFMT_W8: return launch_q<WideW8, true>(a, st);
    case LEMOQ_QFMT_W8_ASYM: return launch_q<WideW8Asym, false>(a, st);
    case LEMOQ_QFMT_W4: return launch_q<WideW4, false>(a, st);
    case LEMOQ_QFMT_W4_ASYM: return launch_q<WideW4Asym, false>(a, st);
    case LEMOQ_QFMT_MXFP4: return launch_q<WideMx4, false>(a, st);
    default: return launch_f16(a, st);
  }
}

int check_gemm(const GemmArgs& a, int group_step = 64) {
  if (!a.x || (!a.codes && !a.w16) || (a.codes && !a.scale) || (!a.y16 && (a.splits == 1 || a.resid)))
    return LEMOQ_ERR_NULL;
  if (a.M <= 0 || a.N <= 0 || a.K <= 0 || a.M > (1LL << 24) || a.N > (1LL << 24)) return LEMOQ_ERR_SHAPE;
  if (((a.M + 63) / 64) * ((a.N + 63) / 64) > 0x7fffffffLL) return LEMOQ_ERR_SHAPE;
  if (a.K % 64 != 0 || a.x_ld < a.K || a.x_ld % 8 != 0 || (a.y16 && a.y_ld < a.N)) return LEMOQ_ERR_SHAPE;
  if (a.codes && (a.group <= 0 || a.group % group_step != 0 || a.K % a.group != 0)) return LEMOQ_ERR_UNSUPPORTED;
  if (a.resid && a.resid_ld < a.N) return LEMOQ_ERR_SHAPE;
  if (a.splits < 1 || a.splits > 64 || a.K % (64LL * a.splits) != 0) return LEMOQ_ERR_SHAPE;
  if (a.splits > 1 && (!a.part || a.M * a.N > (1LL << 31)))
    return a.part ? LEMOQ_ERR_SHAPE : LEMOQ_ERR_NULL;
  if (!lemoq_aligned16(a.x) || (a.codes && !lemoq_aligned16(a.codes)) || (a.w16 && !lemoq_aligned16(a.w16)))
    return LEMOQ_ERR_ALIGN;
  return LEMOQ_OK;
}

}  // namespace

extern "C" int lemoq_gemm_w8(const uint16_t* x, int64_t M, int64_t K, int64_t x_ld, const int32_t* x_rows,
                             const int8_t* codes, const uint16_t* scale, int64_t N, int64_t group,
                             uint16_t* y, int64_t y_ld, const uint16_t* residual, int64_t residual_ld,
                             void* stream) {
  GemmArgs a{};
  a.x = x; a.x_ld = x_ld; a.x_rows = x_rows; a.M = M; a.N = N; a.K = K;
  a.codes = reinterpret_cast<const uint8_t*>(codes); a.scale = scale; a.w16 = nullptr; a.group = (int)group;
  a.y16 = y; a.y_ld = y_ld;
  a.resid = residual; a.resid_ld = residual_ld;
  a.splits = 1; a.part = nullptr;
  if (!y || !codes) return LEMOQ_ERR_NULL;
  const int rc = check_gemm(a);
  if (rc != LEMOQ_OK) return rc;
  return launch_gemm(a, lemoq_stream(stream));
}

extern "C" int lemoq_gemm_q(const uint16_t* x, int64_t M, int64_t K, int64_t x_ld, const void* qweight, int fmt,
                            const void* scale, const void* zero, int64_t N, int64_t group, uint16_t* y, int64_t y_ld,
                            void* stream) {
  if (fmt < LEMOQ_QFMT_W8 || fmt > LEMOQ_QFMT_MXFP4) return LEMOQ_ERR_UNSUPPORTED;
  const bool asym = fmt == LEMOQ_QFMT_W8_ASYM || fmt == LEMOQ_QFMT_W4_ASYM;
  if (!y || !qweight || (asym && !zero)) return LEMOQ_ERR_NULL;
  if (fmt == LEMOQ_QFMT_MXFP4 && group != 32) return LEMOQ_ERR_UNSUPPORTED;
  if (x_ld >= (1LL << 22) || K > NEAR_K) return LEMOQ_ERR_SHAPE;  // a tile's rows are addressed by 32-bit offsets
  GemmArgs a{};
  a.x = x; a.x_ld = x_ld; a.M = M; a.N = N; a.K = K;
  a.codes = reinterpret_cast<const uint8_t*>(qweight); a.scale = scale; a.zero = asym ? zero : nullptr;
  a.group = (int)group; a.y16 = y; a.y_ld = y_ld; a.splits = 1;
  const int rc = check_gemm(a, fmt == LEMOQ_QFMT_W8 ? 64 : 32);
  if (rc != LEMOQ_OK) return rc;
  return launch_gemm(a, lemoq_stream(stream), fmt);
}

extern "C" int lemoq_gemm_f16(const uint16_t* x, int64_t M, int64_t K, int64_t x_ld, const uint16_t* w,
                              int64_t N, uint16_t* y, int64_t y_ld, void* stream) {
  GemmArgs a{};
  a.x = x; a.x_ld = x_ld; a.x_rows = nullptr; a.M = M; a.N = N; a.K = K;
  a.codes = nullptr; a.scale = nullptr; a.w16 = w; a.group = 0;
  a.y16 = y; a.y_ld = y_ld;
  a.resid = nullptr; a.resid_ld = 0;
  a.splits = 1; a.part = nullptr;
  if (!y || !w) return LEMOQ_ERR_NULL;
  const int rc = check_gemm(a);
  if (rc != LEMOQ_OK) return rc;
  return launch_gemm(a, lemoq_stream(stream));
}

// ---------------------------------------------------------------------------
// lemoq_gemm_f16_splitk_noalloc: the same launches with the split partials in
// a fixed device array instead of a caller workspace, so the call allocates
// nothing.  The array's host-side name is not a device address: its address
// on each device comes from hipGetSymbolAddress, taken once per device (with
// that device current) on the first call there, and only that pointer is
// handed to the kernels.
// ---------------------------------------------------------------------------
static __device__ __align__(256) float scratch[LEMOQ_SPLITK_SCRATCH_FLOATS];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float* g_scratch_ptr[kMaxDevices] = {};

// This device's copy of `scratch` (looked up once per device).
int scratch_ptr(float** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return LEMOQ_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return LEMOQ_ERR_NULL;
    g_scratch_ptr[dev] = static_cast<float*>(p);
  }
  *out = g_scratch_ptr[dev];
  return LEMOQ_OK;
}

}  // namespace

extern "C" int lemoq_gemm_f16_splitk_noalloc(const uint16_t* x, int64_t M, int64_t K, int64_t x_ld,
                                             const uint16_t* w, int64_t N, uint16_t* y, int64_t y_ld,
                                             int64_t splits, void* stream) {
  GemmArgs a{};
  a.x = x; a.x_ld = x_ld; a.x_rows = nullptr; a.M = M; a.N = N; a.K = K;
  a.codes = nullptr; a.scale = nullptr; a.w16 = w; a.group = 0;
  a.y16 = y; a.y_ld = y_ld;
  a.resid = nullptr; a.resid_ld = 0;
  // y is required: the partials stay in the library's array, which the caller cannot read
  if (!y || !w) return LEMOQ_ERR_NULL;
  if (splits < 1 || splits > 64) return LEMOQ_ERR_SHAPE;
  if (M <= 0 || N <= 0 || M > (1LL << 24) || N > (1LL << 24)) return LEMOQ_ERR_SHAPE;
  if (splits > 1 && M * N > LEMOQ_SPLITK_SCRATCH_FLOATS / splits) return LEMOQ_ERR_CAPACITY;
  a.splits = (int)splits;
  a.part = nullptr;
  if (splits > 1) {
    const int rc = scratch_ptr(&a.part);
    if (rc != LEMOQ_OK) return rc;
  }
  const int rc = check_gemm(a);
  if (rc != LEMOQ_OK) return rc;
  return launch_gemm(a, lemoq_stream(stream));
}

extern "C" int lemoq_gemm_f16_splitk(const uint16_t* x, int64_t M, int64_t K, int64_t x_ld, const uint16_t* w,
                                     int64_t N, uint16_t* y, int64_t y_ld, int64_t splits, float* workspace,
                                     void* stream) {
  GemmArgs a{};
  a.x = x; a.x_ld = x_ld; a.x_rows = nullptr; a.M = M; a.N = N; a.K = K;
  a.codes = nullptr; a.scale = nullptr; a.w16 = w; a.group = 0;
  a.y16 = y; a.y_ld = y_ld;
  a.resid = nullptr; a.resid_ld = 0;
  if ((!y && splits == 1) || !w) return LEMOQ_ERR_NULL;
  if (splits < 1 || splits > 64) return LEMOQ_ERR_SHAPE;
  a.splits = (int)splits;
  // one split is lemoq_gemm_f16: the workspace is not used (a non-null part
  // would make the kernel write partials instead of y)
  a.part = splits > 1 ? workspace : nullptr;
  if (splits > 1 && !lemoq_aligned16(workspace)) return workspace ? LEMOQ_ERR_ALIGN : LEMOQ_ERR_NULL;
  const int rc = check_gemm(a);
  if (rc != LEMOQ_OK) return rc;
  return launch_gemm(a, lemoq_stream(stream));
}
