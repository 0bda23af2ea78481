// Selection of a token's experts, shared by the launches that need it (moe_aux.hip, moe_decode.hip).
#pragma once
#include "qlinear_common.hpp"

namespace qlin {

// ---------------------------------------------------------------- top-k
// One wavefront per token.  Expert e lives in lane e % 64, slot e / 64.  The
// selection runs on the logits (softmax is monotone): K rounds of wave-wide
// argmax where the LOWEST index wins ties, then the selected probabilities are
// renormalised.  The logits are 16-bit values, so a round is one 32-bit wave
// maximum over keys (order-preserving 16 logit bits << 16 | 0xFFFF - index),
// reduced with DPP inside rows of 16 lanes and v_readlane across the four rows;
// the winner's logit is recovered from the key itself.
constexpr int kTopkSlots = 16;                       // up to 1024 experts

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
  return o > v ? o : v;
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = dpp_max_u32<0xB1>(v);
  v = dpp_max_u32<0x4E>(v);
  v = dpp_max_u32<0x141>(v);
  v = dpp_max_u32<0x140>(v);
  uint32_t r = 0;
#pragma unroll
  for (int row = 0; row < 4; ++row) {
    const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)v, row * 16);
    r = o > r ? o : r;
  }
  return r;
}
// 16-bit float pattern (fp16 or bf16) -> unsigned, monotone, and back; the smallest key, 0, is kept for
// "no value" (it would be the pattern of the negative NaN with every bit set)
// -0 is ordered as +0: a float compare calls them equal, and then the lowest index wins the tie
__device__ __forceinline__ uint32_t f16_order(uint32_t b) {
  b = b == 0x8000u ? 0u : b;
  return (b & 0x8000u) ? (~b & 0xFFFFu) : (b | 0x8000u);
}
__device__ __forceinline__ uint32_t f16_unorder(uint32_t u) { return (u & 0x8000u) ? (u & 0x7FFFu) : (~u & 0xFFFFu); }
template <class Act, int SLOTS>
__device__ __forceinline__ void moe_topk_body(const typename Act::elem* __restrict__ logits,
                                              typename Act::elem* __restrict__ top_w,
                                              int32_t* __restrict__ top_ids, int T, int E,
                                              int K, int renorm,
                                              const float* __restrict__ expert_scale,
                                              const typename Act::v8* __restrict__ gate_x,
                                              const typename Act::v8* __restrict__ gate_w,
                                              float* __restrict__ gate_out, int H8, int t) {
  const int lane = threadIdx.x & 63;
  if (t >= T) return;
  // optional second result of the same wavefront: gate_out[t] = sigmoid(gate_x[t, :] . gate_w[:]) (the
  // shared expert's gate of the fused decode ops); its loads are in flight while the selection runs
  float gate_acc = 0.f;
  if (gate_out) {
    // four steps' loads are requested together (indices held inside the row, the surplus is not added)
    for (int c0 = lane; c0 < H8; c0 += 256) {
      typename Act::v8 a[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = min(c0 + 64 * u, H8 - 1);
        a[u] = gate_x[(size_t)t * H8 + c];
        b[u] = gate_w[c];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (c0 + 64 * u < H8) {
#pragma unroll
          for (int e = 0; e < 8; ++e) gate_acc += Act::to_f32(a[u][e]) * Act::to_f32(b[u][e]);
        }
      }
    }
  }
  const typename Act::elem* row = logits + (size_t)t * E;
  float v[SLOTS];
  uint32_t key[SLOTS];                               // selection keys; 0 = taken or past E
  float mx = -INFINITY;
  // unconditional loads (index held inside the row): with a branch per slot every load waits for the
  // one before
  typename Act::elem raws[SLOTS];
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) raws[s] = row[min(s * 64 + lane, E - 1)];
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const int e = s * 64 + lane;
    const typename Act::elem raw = raws[s];
    v[s] = e < E ? Act::to_f32(raw) : -INFINITY;
    key[s] = e < E ? (f16_order((uint32_t)__builtin_bit_cast(uint16_t, raw)) << 16) | (0xFFFFu - (uint32_t)e) : 0u;
    mx = fmaxf(mx, v[s]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) sum += (s * 64 + lane < E) ? __expf(v[s] - mx) : 0.f;
  sum = wave_sum(sum);

  float my_w = 0.f;                                  // lane r keeps the r-th pick
  int my_id = 0;
  float sel_sum = 0.f;
  for (int r = 0; r < K; ++r) {
    uint32_t best = 0;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) best = key[s] > best ? key[s] : best;
    best = wave_max_u32(best);
    const int cand = (int)(0xFFFFu - (best & 0xFFFFu));
    const float wbest = Act::to_f32(__builtin_bit_cast(typename Act::elem, (uint16_t)f16_unorder(best >> 16)));
    // remove the winner from its owner lane
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
      if (s * 64 + lane == cand) key[s] = 0u;
    const float p = __expf(wbest - mx) / sum;
    sel_sum += p;
    if (lane == r) { my_w = p; my_id = cand; }
  }
  if (lane < K) {
    const float w = renorm ? my_w / sel_sum : my_w;
    typename Act::elem w16 = Act::from_f32(w);
    // optional factor per selected expert, applied to the rounded weight and rounded again
    if (expert_scale) w16 = Act::from_f32(Act::to_f32(w16) * expert_scale[my_id]);
    top_w[(size_t)t * K + lane] = w16;
    top_ids[(size_t)t * K + lane] = my_id;
  }
  if (gate_out) {
    gate_acc = wave_sum(gate_acc);
    if (lane == 0) gate_out[t] = 1.0f / (1.0f + __expf(-gate_acc));
  }
}

}  // namespace qlin
