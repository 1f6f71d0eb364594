// The MoE block of one row in the arithmetic of the multi-token block
// (moe_prefill.hip): weights rounded to fp16 before the dots, fp32 sums in the
// grouped GEMMs' order (row_gemm.h), fp16 gate, up, silu and product, fp16
// expert outputs times the fp16 routing weight, added in fp16 in ascending
// expert order.  It serves the one row that the last layer of a prefill needs,
// with the bits of the sort, the grouped GEMMs and the combine.
//
// gate/up:  grid (ceil(F / 32), top_k), two waves: wave 0 the 32 gate rows,
//           wave 1 the matching up rows, joined through LDS.
// down:     grid ceil(H / 4), one wave: 4 rows of 8 slots at a time, a tile row
//           each, times the slots' own X rows; the slots' results are added
//           through LDS.
//
// Both are bound by the latency of a weight stream (34 and 17 MB at H 2048, F 1024,
// top 8) and the chain over k behind it; the grouped GEMMs add a stage's round
// trip through LDS on every 64 k.  gate/up and down / sort, grouped gate/up and
// down and combine, us (weights from memory): H 2048, F 1024, 8 of 64 experts 22.8 /
// 44.2, one of them 16.2 / 40.8; H 1024, F 512, 8 of 32 12.7 / 29.5; H 512, F 1024,
// 8 of 64 12.8 / 29.4; H 4096, F 1024, 8 of 24 40.0 / 71.2.  In the order of the
// one-token GEMVs (moe.hip) the two take 15 us, with other fp32 sums.
#include "row_gemm.h"

namespace {

using namespace lemoq_gemm;

struct RowGateUpArgs {
  const uint16_t* x;
  const int8_t* codes;     // (E, 2F, H)
  const uint16_t* scale;
  const int64_t* ids;      // given experts (PL = 0), and their fp32 weights
  const float* w_in;
  const uint16_t* logits;  // routed form (PL > 0): (E) fp16 router logits
  int top_k, norm;
  int64_t* ids_out;        // routed form: the selected ids
  uint16_t* w_out;         // fp16 routing weights
  int E, F, H, group;
  uint16_t* act;           // (top_k, F)
};

template <int PL, bool PAIR>
__global__ __launch_bounds__(128) void moe_row_gate_up_kernel(const RowGateUpArgs a) {
  using Dot = RowDot<PAIR, 1>;
  __shared__ __align__(1024) uint8_t lds[2 * Dot::LDS];
  __shared__ uint16_t up[RW_COLS];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, slot = blockIdx.y;
  const bool publish = blockIdx.x == 0 && slot == 0;
  int64_t e;
  if constexpr (PL > 0) {
    // both waves rank the logits: every block up to its own slot, block (0, 0) all of them
    float z[PL], w;
    int id;
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      const int at = lane + 64 * i;
      z[i] = at < a.E ? h2f(a.logits[at]) : -INFINITY;
    }
    const int rounds = publish ? a.top_k : slot + 1;
    wave_route<PL>(z, a.E, a.top_k, a.norm != 0, id, w, rounds);
    if (publish && wave == 0 && lane < rounds) {
      a.ids_out[lane] = (int64_t)id;
      a.w_out[lane] = f2h(w);
    }
    e = __builtin_amdgcn_readlane(id, slot);
  } else {
    e = a.ids[slot];
    if (publish && wave == 0 && lane < a.top_k) a.w_out[lane] = f2h(a.w_in[lane]);
  }
  const int n = blockIdx.x * RW_COLS + l32;
  const bool ev = e >= 0 && e < a.E;  // an invalid expert id yields a zero row
  float v = 0.0f;
  if (ev) {  // block-uniform
    const int n0 = blockIdx.x * RW_COLS;
    const Dot d(lds + wave * Dot::LDS, a.x, 0, 1, a.codes, a.scale, a.H, a.group, [&](int c) {
      return e * 2 * a.F + wave * a.F + (n0 + c < a.F ? n0 + c : a.F - 1);
    });
    v = d.dot()[0];
  }
  if (wave == 1 && lane < 32) up[lane] = f2h(v);
  __syncthreads();
  if (wave == 0 && lane < 32 && n < a.F) {
    const float g = h2f(f2h(v));
    a.act[(int64_t)slot * a.F + n] = f2h(h2f(f2h(g / (1.0f + expf(-g)))) * h2f(up[lane]));
  }
}

template <bool PAIR>
__global__ __launch_bounds__(64) void moe_row_down_kernel(
    const uint16_t* __restrict__ act, const int8_t* __restrict__ codes, const uint16_t* __restrict__ scale,
    const int64_t* __restrict__ ids, const uint16_t* __restrict__ top_w, int top_k, int E, int H, int F, int group,
    const uint16_t* resid, uint16_t* out) {
  using Dot = RowDot<PAIR, 8>;
  constexpr int R = 4;
  __shared__ __align__(1024) uint8_t lds[Dot::LDS];
  __shared__ float part[64][R];  // by place in the sum
  const int lane = threadIdx.x, l32 = lane & 31, n0 = blockIdx.x * R;
  // lane l knows slot l: its expert, and its place in the sum (ascending expert
  // id, slot order among equal ids)
  const int64_t id = ids[lane < top_k ? lane : top_k - 1];
  const bool valid = id >= 0 && id < E;
  const int mine = valid ? (int)id : 0;
  const float w = valid && lane < top_k ? h2f(top_w[lane]) : 0.0f;
  int at = 0;
  for (int s = 0; s < top_k; ++s) {
    const int64_t o = ids[s];
    at += o < id || (o == id && s < lane) ? 1 : 0;
  }
  for (int s0 = 0; s0 < top_k; s0 += 8) {
    const Dot d(lds, act + (int64_t)s0 * F, F, top_k - s0, codes, scale, F, group, [&](int c) {
      const int n = n0 + c % R;
      return (int64_t)__shfl(mine, s0 + c / R, 64) * H + (n < H ? n : H - 1);
    });
    const f32x16 acc = d.dot();
    // tile row c of slot s = c / 4: rows 4 s .. 4 s + 3 of the result, in half s % 2
    const float lo = l32 & 8 ? acc[4] : acc[0], hi = l32 & 8 ? acc[12] : acc[8];
    const float v = l32 & 16 ? hi : lo;
    const int slot = s0 + l32 / R;
    const float ws = __shfl(w, slot & 63, 64);
    const int place = __shfl(at, slot & 63, 64), ok = __shfl((int)valid, slot & 63, 64);
    if (slot < top_k && (lane >> 5) == ((l32 >> 2) & 1)) part[place][l32 % R] = ok ? h2f(f2h(h2f(f2h(v)) * ws)) : 0.0f;
    __syncthreads();
  }
  const int n = n0 + lane;
  if (lane < R && n < H) {
    float v = 0.0f;
    for (int i = 0; i < top_k; ++i) v = h2f(f2h(v + part[i][lane]));
    out[n] = resid ? hadd_round(v, resid[n]) : f2h(v);
  }
}

int check_row(const void* x, const int8_t* codes, const uint16_t* scale, int64_t top_k, int64_t E, int64_t N, int64_t K,
              int64_t group) {
  if (!x || !codes || !scale) return LEMOQ_ERR_NULL;
  if (top_k <= 0 || top_k > 64 || E <= 0 || N <= 0 || K <= 0) return LEMOQ_ERR_SHAPE;
  if (K > 8192 || K % 16 != 0 || group <= 0 || group % 16 != 0 || K % group != 0) return LEMOQ_ERR_UNSUPPORTED;
  if (E * N * K >= (int64_t)1 << 40) return LEMOQ_ERR_SHAPE;
  if (!lemoq_aligned16(codes) || !lemoq_aligned16(x)) return LEMOQ_ERR_ALIGN;
  return LEMOQ_OK;
}

template <int PL>
int launch_gate_up(const RowGateUpArgs& a, void* stream) {
  const dim3 grid((unsigned)((a.F + RW_COLS - 1) / RW_COLS), (unsigned)a.top_k);
  if (a.group % 64 == 0)  // and so H
    hipLaunchKernelGGL((moe_row_gate_up_kernel<PL, true>), grid, dim3(128), 0, lemoq_stream(stream), a);
  else
    hipLaunchKernelGGL((moe_row_gate_up_kernel<PL, false>), grid, dim3(128), 0, lemoq_stream(stream), a);
  LEMOQ_CHECK_LAUNCH();
}

}  // namespace

extern "C" int lemoq_moe_gate_up_w8_dq(const uint16_t* x, const int8_t* codes, const uint16_t* scale,
                                       const int64_t* ids, const float* top_w32, int64_t top_k, int64_t num_experts,
                                       int64_t ffn, int64_t hidden, int64_t group, uint16_t* act, uint16_t* top_w,
                                       void* stream) {
  if (!ids || !top_w32 || !act || !top_w) return LEMOQ_ERR_NULL;
  const int rc = check_row(x, codes, scale, top_k, num_experts, 2 * ffn, hidden, group);
  if (rc) return rc;
  return launch_gate_up<0>({x, codes, scale, ids, top_w32, nullptr, (int)top_k, 0, nullptr, top_w, (int)num_experts,
                            (int)ffn, (int)hidden, (int)group, act}, stream);
}

extern "C" int lemoq_moe_gate_up_w8_routed_dq(const uint16_t* x, const int8_t* codes, const uint16_t* scale,
                                              const uint16_t* router_logits, int64_t top_k, int norm_topk_prob,
                                              int64_t num_experts, int64_t ffn, int64_t hidden, int64_t group,
                                              uint16_t* act, int64_t* top_i, uint16_t* top_w, void* stream) {
  if (!router_logits || !act || !top_i || !top_w) return LEMOQ_ERR_NULL;
  const int rc = check_row(x, codes, scale, top_k, num_experts, 2 * ffn, hidden, group);
  if (rc) return rc;
  if (top_k > num_experts) return LEMOQ_ERR_SHAPE;
  if (num_experts > 256) return LEMOQ_ERR_UNSUPPORTED;
  const RowGateUpArgs a = {x, codes, scale, nullptr, nullptr, router_logits, (int)top_k, norm_topk_prob ? 1 : 0, top_i,
                           top_w, (int)num_experts, (int)ffn, (int)hidden, (int)group, act};
  return num_experts <= 64 ? launch_gate_up<1>(a, stream) : launch_gate_up<4>(a, stream);
}

extern "C" int lemoq_moe_down_w8_dq(const uint16_t* act, const int8_t* codes, const uint16_t* scale,
                                    const int64_t* ids, const uint16_t* top_w, int64_t top_k, int64_t num_experts,
                                    int64_t hidden, int64_t ffn, int64_t group, const uint16_t* residual,
                                    uint16_t* out, void* stream) {
  if (!ids || !top_w || !out) return LEMOQ_ERR_NULL;
  const int rc = check_row(act, codes, scale, top_k, num_experts, hidden, ffn, group);
  if (rc) return rc;
  const dim3 grid((unsigned)((hidden + 3) / 4));
  if (group % 64 == 0)
    hipLaunchKernelGGL((moe_row_down_kernel<true>), grid, dim3(64), 0, lemoq_stream(stream), act, codes, scale, ids,
                       top_w, (int)top_k, (int)num_experts, (int)hidden, (int)ffn, (int)group, residual, out);
  else
    hipLaunchKernelGGL((moe_row_down_kernel<false>), grid, dim3(64), 0, lemoq_stream(stream), act, codes, scale, ids,
                       top_w, (int)top_k, (int)num_experts, (int)hidden, (int)ffn, (int)group, residual, out);
  LEMOQ_CHECK_LAUNCH();
}
