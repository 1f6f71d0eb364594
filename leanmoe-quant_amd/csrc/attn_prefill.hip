// Causal self-attention over the prompt (prefill) on the matrix cores.
//
// The reference prefills through HF's attention with the sdpa backend (the
// decode core replacement only takes q_len == 1; src/lemoq/kernels/
// attn_decode.py:836-1017): softmax(q k^T / sqrt(D) + causal mask) v over the
// fp16 q, k, v of the prompt, fp32 inside, fp16 out.  This kernel computes
// the same with an online softmax (flash-attention order), fp32 statistics
// and accumulators; P is rounded to fp16 for the P V product (as flash
// kernels do).
//
// Layout per wave: 32 queries.  S^T = K Q^T puts one query per lane column
// (accumulator register r of lane l holds key 8*(r/4) + 4*(l/32) + r%4 of the
// 32-key fragment, query l % 32), so the running max and sum of a query are a
// lane-local reduction plus one exchange with lane l ^ 32, and the
// probabilities are already the B operand of O^T = V^T P^T (with the key
// order of that register layout used for the k index of both operands).
//
// A block of NW waves shares key tiles of KT = 8192 / D keys staged in LDS, K
// and V row-major as they lie in memory; the V^T operand is formed by the LDS's
// transposing reads.  Each wave owns 32 queries; with a key split KS = 2, two
// waves own the same 32 queries and take the two halves of every tile, and
// their online-softmax states are merged through LDS at the end (more blocks
// for short prompts).  The tile after the current one goes straight to the
// other half of a double buffer (global_load_lds_dwordx4) while the current one
// is used; one barrier per tile.  Blocks are launched heaviest (latest queries)
// first, or paired with complementary work on one CU (attn_block_of).
//
// Bound by the vector unit: per 64-key tile of head_dim 128 a wave issues 32
// matrix ops (1024 clocks) against 33 quarter-rate exponentials and ~250 other
// vector instructions (~1500), and the two waves of a SIMD overlap the two.
// Tiles that went through registers, V transposed there by v_perm and stored
// 8 bytes at a time, cost a further ~100 vector instructions, 64 LDS stores and
// 48 registers a tile: 16 heads of 128, T 75 6.4 -> 5.6 us, 1024 23.8 -> 23.6,
// 2048 56 -> 48, 4096 120 -> 103 (0.66 PFLOP/s), 8192 490 -> 426; head_dim 64
// at T 5000 166 -> 157, 256 at T 4096 508 -> 474; the same bits.  Next tile's
// scores under this tile's softmax needs more than 256 registers (T 4096: 150
// us); eight waves with a key split of 4 is slower below T 300 and above T 1024.
#include "lds_dma.h"

namespace {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ h8v h8_of(const u32x4 v) { return __builtin_bit_cast(h8v, v); }

// 2^x by v_exp_f32 alone, for the softmax numerators and the running-max
// rescale.  Results below 2^-126 flush to 0 where exp2f returns denormals; p
// is rounded to fp16 (smallest subnormal 2^-24) before P.V and every running
// sum it enters is >= 1, so no output changes.  exp2f's denormal path costs
// four more instructions per score.
__device__ __forceinline__ float exp2_flush(float x) { return __builtin_amdgcn_exp2f(x); }

template <int D, int NW, int KS = 1>
struct AttnGeom {
  static constexpr int THREADS = 64 * NW;
  static constexpr int QG = NW / KS;               // query fragments per block
  static constexpr int QB = 32 * QG;               // queries per block
  static constexpr int KT = 8192 / D;              // keys per tile
  static constexpr int NS = KT / 32;               // S fragments per tile
  static constexpr int NSW = NS / KS;              // S fragments per wave per tile
  static_assert(NS % KS == 0 && NW % KS == 0, "key split");
  static constexpr int DF = D / 32;                // output fragments
  static constexpr int ROW = 2 * D;                // bytes of a K or V row in LDS, rows back to back
  static constexpr int CPR = D / 8;                // 16-byte chunks of a row
  static constexpr int RPL = 64 / CPR;             // rows of one direct load (64 lanes x 16 bytes)
  static constexpr int PASSES = KT / RPL / NW;     // direct loads per wave for a tile's K (and V)
  static constexpr int KB = KT * ROW;              // bytes of a K (or V) tile
  static constexpr int BUF = 2 * KB;               // one LDS buffer: K then V
  // Chunk c of row r sits at chunk c ^ kswz(r) (K) or c ^ vswz(r) (V).  K: 16
  // lanes reading one chunk of 16 rows hit 16 different bank groups; V: the
  // four rows x 64 bytes that 32 lanes of a transposing read touch lie in
  // different quarters of the banks.
  __device__ static int kswz(int r) { return D == 64 ? (r >> 1) & 7 : r & 15; }
  __device__ static int vswz(int r) { return D == 64 ? 4 * ((r >> 1) & 1) : 4 * (r & 3); }
  static_assert(PASSES >= 1 && KT % (RPL * NW) == 0, "tile split");
};

// The K and V rows [k0, k0 + KT) to an LDS buffer by direct loads, this wave's
// share; rows past the prompt read its last row.
template <class G>
__device__ __forceinline__ void attn_load(uint32_t buf, const uint16_t* __restrict__ kh,
                                          const uint16_t* __restrict__ vh, int64_t k0, int64_t T, int wave, int lane) {
  const uint8_t* kb = reinterpret_cast<const uint8_t*>(kh) + k0 * G::ROW;
  const uint8_t* vb = reinterpret_cast<const uint8_t*>(vh) + k0 * G::ROW;
  const int left = T - 1 - k0 < G::KT ? (int)(T - 1 - k0) : G::KT;  // >= 0: tiles start inside the prompt
#pragma unroll
  for (int p = 0; p < G::PASSES; ++p) {
    const int first = G::RPL * (G::PASSES * wave + p);
    const int row = first + lane / G::CPR, c = lane % G::CPR;
    const int src = row < left ? row : left;
    const uint32_t ko = (uint32_t)(src * G::ROW + (c ^ G::kswz(row)) * 16);
    const uint32_t vo = (uint32_t)(src * G::ROW + (c ^ G::vswz(row)) * 16);
    const uint32_t to = buf + (uint32_t)(first * G::ROW);
    dma16(to, ko, kb);
    dma16(to + G::KB, vo, vb);
  }
}

// This wave's LDS reads and direct loads are done, in every wave of the block.
__device__ __forceinline__ void attn_wait() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
}

// 4 fp16 of the column that this lane names in a 4 x 16 tile of LDS: lane i of
// 16 passes the address of row i / 4, columns 4 (i % 4) .. + 3, and receives
// column i of the four rows.
__device__ __forceinline__ uint2 lds_read_tr(const uint8_t* p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
}

// Query blocks and heads over the grid.  Two-dimensional: blockIdx.x is the
// query block's rank (0 = the latest prompt rows, the most keys), blockIdx.y
// the head.  PAIRED (an even number of heads): a 1-D grid whose first half
// takes heads 0 .. heads/2 - 1 latest-first and whose second half takes the
// other heads earliest-first, so blocks b and b + grid/2, which the dispatcher
// places on the same compute unit when the whole grid is resident at two
// blocks per CU, carry complementary numbers of key tiles (16 heads of 128:
// T 4096 131 -> 103 us, T 8192 474 -> 436).
template <bool PAIRED>
__device__ __forceinline__ void attn_block_of(int64_t nqb, int heads, int& h, int64_t& rank) {
  if constexpr (PAIRED) {
    const int64_t L = blockIdx.x, half_grid = nqb * (heads / 2);
    if (L < half_grid) {
      h = (int)(L / nqb);
      rank = L % nqb;
    } else {
      h = heads / 2 + (int)((L - half_grid) / nqb);
      rank = nqb - 1 - (L - half_grid) % nqb;
    }
  } else {
    h = blockIdx.y;
    rank = blockIdx.x;
  }
}

template <int D, int NW, int KS, bool PAIRED>
__device__ __forceinline__ void attn_prefill_body(
    const uint16_t* __restrict__ q, int64_t q_ld, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, int64_t kv_head_stride, int64_t T, float qk_scale,
    uint16_t* __restrict__ out, int64_t out_ld, int heads) {
  using G = AttnGeom<D, NW, KS>;
  __shared__ __align__(1024) uint8_t lds[2 * G::BUF];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int qfrag = wave % G::QG, kpart = wave / G::QG;  // kpart: which NSW-fragment slice of each tile
  const int64_t nqb = (T + G::QB - 1) / G::QB;
  int h;
  int64_t rank;
  attn_block_of<PAIRED>(nqb, heads, h, rank);
  const int64_t q0 = (nqb - 1 - rank) * G::QB;
  const int64_t qw = q0 + 32 * qfrag;
  const int64_t qi = qw + l32;
  const int64_t qc = qi < T ? qi : T - 1;

  // Q^T operand: lane half h holds dims 32j + 16h + [0, 16) of its query.
  h8v qf[G::DF][2];
  {
    const uint16_t* qp = q + qc * q_ld + (int64_t)h * D + 16 * half;
#pragma unroll
    for (int j = 0; j < G::DF; ++j) {
      qf[j][0] = h8_of(*reinterpret_cast<const u32x4*>(qp + 32 * j));
      qf[j][1] = h8_of(*reinterpret_cast<const u32x4*>(qp + 32 * j + 8));
    }
  }
  const uint16_t* kh = k + (int64_t)h * kv_head_stride;
  const uint16_t* vh = v + (int64_t)h * kv_head_stride;

  float m = -INFINITY, l = 0.0f;
  f32x16 o[G::DF];
#pragma unroll
  for (int f = 0; f < G::DF; ++f) o[f] = (f32x16){};

  const int64_t kend = T < q0 + G::QB ? T : q0 + G::QB;
  const int64_t ntile = (kend + G::KT - 1) / G::KT;
  const uint32_t lds0 = lds_addr(lds);
  attn_load<G>(lds0, kh, vh, 0, T, wave, lane);
  // V^T fragment f: lane 16 g + i reads dims 32 f + 16 (g % 2) + 4 (i % 4) of
  // key 4 half + i / 4 (+ the step's first key): its byte offset in a tile
  const int vkey = 4 * half + ((lane & 15) >> 2);
  uint32_t va[G::DF];
#pragma unroll
  for (int f = 0; f < G::DF; ++f)
    va[f] = (uint32_t)(vkey * G::ROW + ((4 * f + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ G::vswz(vkey)) * 16 +
                       8 * (lane & 1));
  for (int64_t it = 0; it < ntile; ++it) {
    const int64_t k0 = it * G::KT;
    attn_wait();  // tile it has landed, tile it - 1 is read by all
    if (it + 1 < ntile) attn_load<G>(lds0 + (uint32_t)(((it + 1) & 1) * G::BUF), kh, vh, k0 + G::KT, T, wave, lane);
    const uint8_t* ks = lds + (it & 1) * G::BUF;
    const uint8_t* vt = ks + G::KB;
    const int64_t kw = k0 + 32 * G::NSW * kpart;  // first key of this wave's slice of the tile
    if (kw <= qw) {  // wave-uniform: the slice holds a key at or before every query of the wave
      f32x16 s[G::NSW];
#pragma unroll
      for (int sf = 0; sf < G::NSW; ++sf) s[sf] = (f32x16){};
      // the NSW accumulation chains are interleaved (independent neighbours)
#pragma unroll
      for (int j = 0; j < G::DF; ++j)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int sf = 0; sf < G::NSW; ++sf) {
            const h8v kf = *reinterpret_cast<const h8v*>(
                ks + (32 * (G::NSW * kpart + sf) + l32) * G::ROW + ((4 * j + 2 * half + hh) ^ G::kswz(l32)) * 16);
            s[sf] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[j][hh], s[sf], 0, 0, 0);
          }
      float mx = -INFINITY;
      // Masks are needed only where the slice reaches past the wave's first
      // query or past the prompt (wave-uniform test); there the key offset
      // from this lane's query fits 32 bits.
      const int64_t kend_w = kw + 32 * G::NSW;
      if (kend_w - 1 <= qw && kend_w <= T) {
#pragma unroll
        for (int sf = 0; sf < G::NSW; ++sf)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            s[sf][r] *= qk_scale;
            mx = fmaxf(mx, s[sf][r]);
          }
      } else {
        const int lim = (int)((T < qi + 1 ? T : qi + 1) - kw);  // keys kw + j with j < lim are valid
#pragma unroll
        for (int sf = 0; sf < G::NSW; ++sf)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int j = 32 * sf + 8 * (r / 4) + 4 * half + (r % 4);
            s[sf][r] = j < lim ? s[sf][r] * qk_scale : -INFINITY;
            mx = fmaxf(mx, s[sf][r]);
          }
      }
      mx = fmaxf(mx, xor32_get(mx, lane));
      // key kw <= qw <= qi is valid for every query of a wave with stored outputs
      // (qw < T), so mn is finite there; waves wholly past the prompt store nothing
      const float mn = fmaxf(m, mx);
      const float alpha = exp2_flush(m - mn);
      float ps = 0.0f;
      h8v pb[2 * G::NSW];
#pragma unroll
      for (int sf = 0; sf < G::NSW; ++sf) {
        uint32_t pk[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float p0 = exp2_flush(s[sf][2 * i] - mn), p1 = exp2_flush(s[sf][2 * i + 1] - mn);
          ps += p0 + p1;
          const f16x2 hp = {(f16)p0, (f16)p1};  // one v_cvt_pk_f16_f32 (round to nearest even)
          pk[i] = __builtin_bit_cast(uint32_t, hp);
        }
        pb[2 * sf] = h8_of((u32x4){pk[0], pk[1], pk[2], pk[3]});
        pb[2 * sf + 1] = h8_of((u32x4){pk[4], pk[5], pk[6], pk[7]});
      }
      l = l * alpha + ps;
      m = mn;
      // rescale only when some query's running max moved (wave-uniform test)
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
        for (int f = 0; f < G::DF; ++f)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[f][r] *= alpha;
      }
#pragma unroll
      for (int qq = 0; qq < 2 * G::NSW; ++qq) {
        const int kb = 32 * (G::NSW * kpart + qq / 2) + 16 * (qq % 2);
#pragma unroll
        for (int f = 0; f < G::DF; ++f) {
          const uint2 a0 = lds_read_tr(vt + va[f] + kb * G::ROW);        // keys kb + 4 half ..
          const uint2 a1 = lds_read_tr(vt + va[f] + (kb + 8) * G::ROW);  // and kb + 8 + 4 half ..
          o[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(h8_of((u32x4){a0.x, a0.y, a1.x, a1.y}), pb[qq], o[f], 0, 0, 0);
        }
      }
    }
  }

  if constexpr (KS == 2) {
    attn_wait();  // the tile buffers are free
    // Merge the two key slices of each query fragment: slice 1 publishes m, its lane's
    // partial l and o, transposed so consecutive lanes hit consecutive banks;
    // slice 0 combines in a fixed order.
    constexpr int NV = 16 * G::DF + 2;
    float* mrg = reinterpret_cast<float*>(lds) + qfrag * NV * 64;
    if (kpart == 1) {
      mrg[lane] = m;
      mrg[64 + lane] = l;
#pragma unroll
      for (int f = 0; f < G::DF; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) mrg[(2 + 16 * f + r) * 64 + lane] = o[f][r];
    }
    __syncthreads();
    if (kpart == 1) return;
    const float mb = mrg[lane], lb = mrg[64 + lane];
    const float mm = fmaxf(m, mb);  // m is finite: slice 0 always holds key 0 for this fragment
    const float fa = exp2f(m - mm), fb = exp2f(mb - mm);
    l = l * fa + lb * fb;
#pragma unroll
    for (int f = 0; f < G::DF; ++f)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[f][r] = o[f][r] * fa + mrg[(2 + 16 * f + r) * 64 + lane] * fb;
  }
  const float lt = l + xor32_get(l, lane);
  const float inv = 1.0f / lt;
  if (qi >= T) return;
  uint16_t* op = out + qi * out_ld + (int64_t)h * D + 4 * half;
#pragma unroll
  for (int f = 0; f < G::DF; ++f)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint32_t lo = (uint32_t)f2h(o[f][4 * b] * inv) | ((uint32_t)f2h(o[f][4 * b + 1] * inv) << 16);
      const uint32_t hi = (uint32_t)f2h(o[f][4 * b + 2] * inv) | ((uint32_t)f2h(o[f][4 * b + 3] * inv) << 16);
      *reinterpret_cast<uint2*>(op + 32 * f + 8 * b) = make_uint2(lo, hi);
    }
}

// Two waves per SIMD need at most 256 registers a lane: met without spills
// for head_dim 128 with 4-wave blocks (two blocks fit the LDS of a CU).
template <int D, int NW, int KS, bool PAIRED>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void attn_prefill_kernel_occ2(
    const uint16_t* __restrict__ q, int64_t q_ld, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, int64_t kv_head_stride, int64_t T, float qk_scale,
    uint16_t* __restrict__ out, int64_t out_ld, int heads) {
  attn_prefill_body<D, NW, KS, PAIRED>(q, q_ld, k, v, kv_head_stride, T, qk_scale, out, out_ld, heads);
}

template <int D, int NW, int KS, bool PAIRED>
__global__ __launch_bounds__(64 * NW) void attn_prefill_kernel(
    const uint16_t* __restrict__ q, int64_t q_ld, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, int64_t kv_head_stride, int64_t T, float qk_scale,
    uint16_t* __restrict__ out, int64_t out_ld, int heads) {
  attn_prefill_body<D, NW, KS, PAIRED>(q, q_ld, k, v, kv_head_stride, T, qk_scale, out, out_ld, heads);
}

template <int D, int NW, int KS, bool PAIRED>
void launch_attn_grid(const uint16_t* q, int64_t q_ld, const uint16_t* k, const uint16_t* v,
                      int64_t kv_head_stride, int64_t T, int64_t heads, float qk_scale, uint16_t* out,
                      int64_t out_ld, hipStream_t st) {
  constexpr int QB = 32 * NW / KS;
  const int64_t nqb = (T + QB - 1) / QB;
  const dim3 grid = PAIRED ? dim3((unsigned)(nqb * heads)) : dim3((unsigned)nqb, (unsigned)heads);
  if constexpr (D == 128 && NW == 4)
    hipLaunchKernelGGL((attn_prefill_kernel_occ2<D, NW, KS, PAIRED>), grid, dim3(64 * NW), 0, st, q, q_ld, k, v,
                       kv_head_stride, T, qk_scale, out, out_ld, (int)heads);
  else
    hipLaunchKernelGGL((attn_prefill_kernel<D, NW, KS, PAIRED>), grid, dim3(64 * NW), 0, st, q, q_ld, k, v,
                       kv_head_stride, T, qk_scale, out, out_ld, (int)heads);
}

// 128-query blocks of an even number of heads run the paired grid.
template <int D, int NW, int KS>
void launch_attn(const uint16_t* q, int64_t q_ld, const uint16_t* k, const uint16_t* v, int64_t kv_head_stride,
                 int64_t T, int64_t heads, float qk_scale, uint16_t* out, int64_t out_ld, hipStream_t st) {
  constexpr int QB = 32 * NW / KS;
  const int64_t nqb = (T + QB - 1) / QB;
  if (KS == 1 && heads % 2 == 0 && nqb * heads <= 0x7fffffffLL)
    launch_attn_grid<D, NW, KS, true>(q, q_ld, k, v, kv_head_stride, T, heads, qk_scale, out, out_ld, st);
  else
    launch_attn_grid<D, NW, KS, false>(q, q_ld, k, v, kv_head_stride, T, heads, qk_scale, out, out_ld, st);
}

template <int D>
void launch_attn_d(const uint16_t* q, int64_t q_ld, const uint16_t* k, const uint16_t* v, int64_t kv_head_stride,
                   int64_t T, int64_t heads, float qk_scale, uint16_t* out, int64_t out_ld, hipStream_t st) {
  // 128 queries per 4-wave block once that gives two blocks per compute unit;
  // below that, 64 queries per block with each tile's keys split between
  // wave pairs (twice the blocks, half the keys per wave).  16 heads of 128,
  // unsplit / split: T 1024 27.5 / 23.6 us, 2048 50.4 / 48.2, 3000 86.4 / 84.5,
  // 4096 (512 blocks) 103 / 160.
  if constexpr (D > 128) {  // one 32-key fragment per tile: nothing to split
    launch_attn<D, 4, 1>(q, q_ld, k, v, kv_head_stride, T, heads, qk_scale, out, out_ld, st);
  } else {
    if (((T + 127) / 128) * heads >= 512)
      launch_attn<D, 4, 1>(q, q_ld, k, v, kv_head_stride, T, heads, qk_scale, out, out_ld, st);
    else
      launch_attn<D, 4, 2>(q, q_ld, k, v, kv_head_stride, T, heads, qk_scale, out, out_ld, st);
  }
}

}  // namespace

extern "C" int lemoq_attn_prefill_f16(const uint16_t* q, int64_t q_ld, const uint16_t* k, const uint16_t* v,
                                      int64_t kv_head_stride, int64_t T, int64_t heads, int64_t head_dim,
                                      float qk_scale, uint16_t* out, int64_t out_ld, void* stream) {
  if (!q || !k || !v || !out) return LEMOQ_ERR_NULL;
  if (T <= 0 || T > (1LL << 30) || heads <= 0 || heads > 65535) return LEMOQ_ERR_SHAPE;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) return LEMOQ_ERR_UNSUPPORTED;
  if (q_ld < heads * head_dim || out_ld < heads * head_dim || q_ld % 8 != 0 || out_ld % 4 != 0 ||
      kv_head_stride < T * head_dim || kv_head_stride % 8 != 0)
    return LEMOQ_ERR_SHAPE;
  if (!lemoq_aligned16(q) || !lemoq_aligned16(k) || !lemoq_aligned16(v) ||
      (reinterpret_cast<uintptr_t>(out) & 7u) != 0)
    return LEMOQ_ERR_ALIGN;
  hipStream_t st = lemoq_stream(stream);
  switch (head_dim) {
    case 64: launch_attn_d<64>(q, q_ld, k, v, kv_head_stride, T, heads, qk_scale, out, out_ld, st); break;
    case 128: launch_attn_d<128>(q, q_ld, k, v, kv_head_stride, T, heads, qk_scale, out, out_ld, st); break;
    default: launch_attn_d<256>(q, q_ld, k, v, kv_head_stride, T, heads, qk_scale, out, out_ld, st); break;
  }
  LEMOQ_CHECK_LAUNCH();
}
