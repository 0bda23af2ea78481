// The fused MoE decode step in two launches, where these are ahead of one GEMV launch per projection (mi_moe_decode_plan).
//
// mi_moe_gate_up_topk_fp8_block: routing, and the gate_up rows of the selected experts and of the shared expert.  Bound: the round
// trips logits -> weights and the weight stream.  Selecting took a launch of its own, a round trip and a launch's start ahead of
// the weights; a wavefront here picks the experts of its own rows (as many rounds of the selection as they are down the list; none
// for the shared expert's rows), and one more workgroup per token writes the selection for the launch that follows.  A
// wavefront owns consecutive rows of (route, row), all of them in flight, against x in its registers.
//
// mi_moe_down_sum_fp8_block: the down projections of a token's routes and of the shared expert, SiLU(gate) x up on the way in,
// and their weighted sum:
//
//   out[t][n] = sum_j w[t][j] (a[t][j] . W2[ids[t][j]][n]) + gate[t] (a[shared t] . W2shared[n]),   a = act(gate_up row)
//
// Bound: one round trip (ids -> weights) and the weight stream.  With a route per workgroup and a launch for the sum it was two
// dependent launches, and the routes' rows went through memory.  A wavefront owns output rows: the k + 1 weight rows that make up
// an output are one sequence of 16-byte pieces over its lanes (9 x 768 bytes: 6.75 loads per lane, all of them in flight before
// the activations are staged), every lane scales its partial sums itself, and one reduction ends the row.  Sums stay in fp32
// until the output's rounding.
//
// The step, 128 experts, top 8, H = 2048, I = 768, bf16, us: four launches / the sum in the down launch / two launches: one token
// 21.5 / 18.7 / 14.4, two 31.1 / 27.0 / 22.2, four 48.6 / 42.6 / 35, eight 71.8 / 67.6 / 64, twelve 118.4 / 109.5 / 92.
#include "qlinear_common.hpp"
#include "gemv_rows.hpp"
#include "moe_topk.hpp"
#include "../../include/mi355x_qlinear.h"

namespace qlin {

struct GateUpArgs {
  const void* x;              // [T, H]
  const void* logits;         // [T, E]
  const void* gate_w;         // [H]
  const void *w, *shared_w;   // [E, 2 I, H], [2 I, H]
  const float *scale, *shared_scale;
  void* out;                  // [T k + T, 2 I]
  int32_t* ids;               // [T, k]
  void* top_w;                // [T, k]
  float* gate;                // [T]
  int T, k, E, H, N;          // N = 2 I
};

constexpr int kGateWaves = 8;

// NI: 1024-byte pieces of a weight row; RP: consecutive rows of the sequence (route, row) per wavefront, all in flight
template <class Act, int SLOTS, int NI, int RP>
__global__ __launch_bounds__(64 * kGateWaves) void gate_up_topk_kernel(const GateUpArgs p) {
  using Elem = typename Act::elem;
  using V8 = typename Act::v8;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = blockIdx.y, k = p.k, E = p.E, H = p.H, N = p.N;
  if (blockIdx.x == gridDim.x - 1) {                  // this one hands the selection and the shared expert's gate on
    if (wave == 0)
      moe_topk_body<Act, SLOTS>((const Elem*)p.logits, (Elem*)p.top_w, p.ids, p.T, E, k, 1, nullptr, (const V8*)p.x, (const V8*)p.gate_w,
                                p.gate, H >> 3, t);
    return;
  }
  const int rows = (k + 1) * N, q0 = (blockIdx.x * kGateWaves + wave) * RP;
  if (q0 >= rows) return;
  const int pieces = H >> 4;                          // 16-byte pieces of a weight row
  u32x4 xv[NI][2];
  Elem raws[SLOTS];
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) raws[s] = ((const Elem*)p.logits)[(size_t)t * E + min(s * 64 + lane, E - 1)];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int c = i * 64 + lane;
    const u32x4* src = reinterpret_cast<const u32x4*>((const Elem*)p.x + (size_t)t * H) + 2 * (c < pieces ? c : pieces - 1);
    xv[i][0] = src[0];
    xv[i][1] = src[1];
  }
  // the experts of this wavefront's first and last row: as many rounds of the selection as they are down the list
  const int r0 = q0 / N, q1 = min(q0 + RP, rows) - 1, r1 = q1 / N;
  int e0 = 0, e1 = 0;
  {
    uint32_t key[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      const int e = s * 64 + lane;
      key[s] = e < E ? (f16_order((uint32_t)__builtin_bit_cast(uint16_t, raws[s])) << 16) | (0xFFFFu - (uint32_t)e) : 0u;
    }
    for (int r = 0; r <= min(r1, k - 1); ++r) {
      if (r0 >= k) break;                             // shared expert's rows only
      uint32_t best = 0;
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) best = key[s] > best ? key[s] : best;
      best = wave_max_u32(best);
      const int cand = __builtin_amdgcn_readfirstlane((int)(0xFFFFu - (best & 0xFFFFu)));
#pragma unroll
      for (int s = 0; s < SLOTS; ++s)
        if (s * 64 + lane == cand) key[s] = 0u;
      if (r == r0) e0 = cand;
      e1 = cand;
    }
  }
  u32x4 wv[RP][NI];
  float f[RP][NI];
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    const int q = min(q0 + j, q1), r = q >= r1 * N ? r1 : r0, n = q - r * N;
    const size_t e = (size_t)(r == r1 ? e1 : e0);
    const unsigned char* w = (r >= k ? (const unsigned char*)p.shared_w : (const unsigned char*)p.w + e * (size_t)N * H) + (size_t)n * H;
    const float* sc = (r >= k ? p.shared_scale : p.scale + e * (size_t)(N >> 7) * (H >> 7)) + (size_t)(n >> 7) * (H >> 7);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int c = i * 64 + lane < pieces ? i * 64 + lane : pieces - 1;
      wv[j][i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w) + c);
      f[j][i] = sc[c >> 3];
    }
  }
  float mine = 0.0f;                                  // lane j: row q0 + j
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const u32x4 b0 = __builtin_bit_cast(u32x4, fp8x8_to_act<Act>(wv[j][i][0], wv[j][i][1]));
      const u32x4 b1 = __builtin_bit_cast(u32x4, fp8x8_to_act<Act>(wv[j][i][2], wv[j][i][3]));
      float d = 0.0f;
#pragma unroll
      for (int m = 0; m < 4; ++m) d = Dot2<Act>::run(b0[m], xv[i][0][m], d);
#pragma unroll
      for (int m = 0; m < 4; ++m) d = Dot2<Act>::run(b1[m], xv[i][1][m], d);
      acc += i * 64 + lane < pieces ? d * f[j][i] : 0.0f;
    }
    acc = wave_sum(acc);
    mine = lane == j ? acc : mine;
  }
  const int q = q0 + lane;
  if (lane < RP && q <= q1)
    ((Elem*)p.out)[q < k * N ? (size_t)t * k * N + q : ((size_t)p.T * k + t) * N + (q - k * N)] = Act::from_f32(mine);
}

template <class Act, int SLOTS, int NI>
static void launch_gate_up2(const GateUpArgs& p, hipStream_t st) {
  auto go = [&](auto rp) {
    constexpr int RP = decltype(rp)::value;
    const int per = kGateWaves * RP;
    hipLaunchKernelGGL((gate_up_topk_kernel<Act, SLOTS, NI, RP>), dim3((unsigned)(((p.k + 1) * p.N + per - 1) / per + 1), (unsigned)p.T),
                       dim3(64 * kGateWaves), 0, st, p);
  };
  // rows per wavefront 2 / 4 / 8, us for the whole step: one token 14.2 / 14.5 / 14.9, four 36.0 / 34.4 / 36.0, twelve 97.7 / 92.0 / 94.2
  if (p.T == 1) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
}
template <class Act, int NI>
static void launch_gate_up1(const GateUpArgs& p, hipStream_t st) {
  if (p.E <= 128) launch_gate_up2<Act, 2, NI>(p, st);
  else if (p.E <= 256) launch_gate_up2<Act, 4, NI>(p, st);
  else if (p.E <= 512) launch_gate_up2<Act, 8, NI>(p, st);
  else launch_gate_up2<Act, 16, NI>(p, st);
}
template <class Act>
static int launch_gate_up(const GateUpArgs& p, hipStream_t st) {
  if (p.H <= 1024) launch_gate_up1<Act, 1>(p, st);
  else if (p.H <= 2048) launch_gate_up1<Act, 2>(p, st);
  else launch_gate_up1<Act, 4>(p, st);
  return launch_status();
}

struct DownSumArgs {
  const void* gu;             // [T k + T, 2 I]: routes in pair order, then the shared expert's rows
  const void *w, *shared_w;
  const float *scale, *shared_scale;
  const int32_t* ids;         // [T, k]
  const void* route_weight;   // [T, k], activation type
  const float* gate;          // [T]
  void* out;                  // [T, H]
  int T, k, E, H, I;
};

constexpr int kDownWaves = 8, kDownPieces = 8;        // wavefronts per workgroup, pieces in flight per lane and row

template <class Act, int RPW>                         // output rows per wavefront
__global__ __launch_bounds__(64 * kDownWaves) void down_sum_kernel(const DownSumArgs p) {
  using Elem = typename Act::elem;
  using V8 = typename Act::v8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];        // [k + 1][I] activations
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t = blockIdx.y, k = p.k, H = p.H, I = p.I;
  const int n0 = (blockIdx.x * kDownWaves + wave) * RPW;
  const unsigned per = (unsigned)I >> 4, total = per * (unsigned)(k + 1);      // 16-byte pieces of a route's row, of an output row
  u32x4 wv[RPW][kDownPieces];
  float f[RPW][kDownPieces];                          // block scale x routing weight (or the shared expert's gate)
  // request the pieces [s0, + 64 x kDownPieces); rows past H and pieces past the end repeat valid ones
  auto request = [&](unsigned s0) __attribute__((always_inline)) {
    unsigned s[kDownPieces], r[kDownPieces];
    int e[kDownPieces];
#pragma unroll
    for (int i = 0; i < kDownPieces; ++i) {
      s[i] = s0 + i * 64 + lane;
      if (s[i] >= total) s[i] = total - 1;
      r[i] = s[i] / per;
      e[i] = p.ids[(size_t)t * k + (r[i] < (unsigned)k ? r[i] : (unsigned)k - 1)];
    }
#pragma unroll
    for (int i = 0; i < kDownPieces; ++i) {
      const bool shared = r[i] >= (unsigned)k;
      const unsigned c = s[i] - r[i] * per;
      const size_t ex = (size_t)(e[i] < 0 ? 0 : (e[i] >= p.E ? p.E - 1 : e[i]));   // ids outside the stack are held into it
      const unsigned char* w = shared ? (const unsigned char*)p.shared_w : (const unsigned char*)p.w + ex * (size_t)H * I;
      const float* sc = shared ? p.shared_scale : p.scale + ex * (size_t)(H >> 7) * (I >> 7);
#pragma unroll
      for (int q = 0; q < RPW; ++q) {
        const int n = n0 + q < H ? n0 + q : H - 1;
        wv[q][i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w + (size_t)n * I + c * 16));
        f[q][i] = sc[(size_t)(n >> 7) * (I >> 7) + (c >> 3)];
      }
    }
#pragma unroll
    for (int i = 0; i < kDownPieces; ++i) {
      const bool shared = r[i] >= (unsigned)k;
      const float m = shared ? p.gate[t] : Act::to_f32(((const Elem*)p.route_weight)[(size_t)t * k + (shared ? 0 : r[i])]);
#pragma unroll
      for (int q = 0; q < RPW; ++q) f[q][i] *= m;
    }
  };
  float acc[RPW];
#pragma unroll
  for (int q = 0; q < RPW; ++q) acc[q] = 0.0f;
  auto multiply = [&](unsigned s0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kDownPieces; ++i) {
      unsigned s = s0 + i * 64 + lane;
      const bool mine = s < total;                    // selected, not multiplied by 0: what is repeated may be infinite
      if (!mine) s = total - 1;
      const u32x4 a0 = *reinterpret_cast<const u32x4*>(smem + (size_t)s * 32), a1 = *reinterpret_cast<const u32x4*>(smem + (size_t)s * 32 + 16);
#pragma unroll
      for (int q = 0; q < RPW; ++q) {
        const u32x4 b0 = __builtin_bit_cast(u32x4, fp8x8_to_act<Act>(wv[q][i][0], wv[q][i][1]));
        const u32x4 b1 = __builtin_bit_cast(u32x4, fp8x8_to_act<Act>(wv[q][i][2], wv[q][i][3]));
        float d = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) d = Dot2<Act>::run(b0[j], a0[j], d);
#pragma unroll
        for (int j = 0; j < 4; ++j) d = Dot2<Act>::run(b1[j], a1[j], d);
        acc[q] = mine ? __builtin_fmaf(d, f[q][i], acc[q]) : acc[q];
      }
    }
  };
  request(0);
  // SiLU(gate) x up of the k + 1 rows: fp32 inside, one rounding, as silu_mul_kernel computes it
  const unsigned pieces = (unsigned)I >> 3;           // of 8 elements
  for (unsigned i = tid; i < pieces * (unsigned)(k + 1); i += 64 * kDownWaves) {
    const unsigned r = i / pieces, c = i - r * pieces;
    const size_t row = r < (unsigned)k ? (size_t)t * k + r : (size_t)p.T * k + t;
    const u32x4* src = reinterpret_cast<const u32x4*>((const Elem*)p.gu + row * 2 * I) + c;
    const V8 g8 = as_v8<V8>(src[0]), u8 = as_v8<V8>(src[pieces]);
    V8 o8;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float g = Act::to_f32(g8[j]), u = Act::to_f32(u8[j]);
      o8[j] = Act::from_f32(g / (1.0f + expf(-g)) * u);
    }
    *reinterpret_cast<u32x4*>(smem + (size_t)i * 16) = __builtin_bit_cast(u32x4, o8);
  }
  __syncthreads();
  multiply(0);
  for (unsigned s0 = 64 * kDownPieces; s0 < total; s0 += 64 * kDownPieces) {
    request(s0);
    multiply(s0);
  }
#pragma unroll
  for (int q = 0; q < RPW; ++q) {
    const float v = wave_sum(acc[q]);
    if (lane == 0 && n0 + q < H) ((Elem*)p.out)[(size_t)t * H + n0 + q] = Act::from_f32(v);
  }
}

template <class Act>
static int launch_down_sum(const DownSumArgs& p, hipStream_t st) {
  const size_t lds = (size_t)(p.k + 1) * p.I * 2;
  // A workgroup stages all of its token's activations: a row per wavefront while these fit the chip in one round, else more rows share
  // the staging.  1 / 2 / 4 rows, us for the whole step (sizes as above): one token 18.7 / 19.7 / 22.8, two 28.5 / 27.0 / 29.2, three
  // 37.7 / 38.5 / 34.8, eight 76.5 / 74.0 / 66.9.
  auto go = [&](auto rpw) {
    constexpr int RPW = decltype(rpw)::value;
    hipLaunchKernelGGL((down_sum_kernel<Act, RPW>), dim3((unsigned)((p.H + kDownWaves * RPW - 1) / (kDownWaves * RPW)), (unsigned)p.T),
                       dim3(64 * kDownWaves), lds, st, p);
  };
  const int cus = device_cu_count(), groups = (p.H + kDownWaves - 1) / kDownWaves * p.T;
  if (groups <= cus) go(std::integral_constant<int, 1>{});
  else if (groups <= 2 * cus) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
  return launch_status();
}

// ---------------------------------------------------------------- which launches
constexpr int kRoutedPairs = 96;                      // (token, route) pairs up to which one GEMV runs per route
constexpr int kGateUpColumns = 4096;                  // x of gate_up_topk_kernel is held in registers
constexpr long long kDownSumBytes = 64 * 1024;        // a token's activations of down_sum_kernel are held in LDS

// The two launches above against the row GEMV's (gemv_rows.hpp, with mi_moe_topk and mi_moe_combine_shared), each half on its own: 4421 problems (17
// sizes, H 256 .. 5120, I 128 .. 8192, E 8 .. 512, top 1 .. 32, fp16 and bf16) of up to 96 pairs.  By these lines the step takes 0.51 to 1.04 of
// the four launches' time (0.86 in the mean; the best choice for each 0.82), 1.02 and more on 8; the two launches everywhere 0.51 to 2.22.  On 1965 problems
// of seven other sizes it takes at most 1.03 (0.85 in the mean, best 0.80; the two launches up to 2.11).
//
// Gate_up: ahead up to three tokens, which read hardly any matrix twice.  With more, every token reads the shared expert and, with few
// experts, those of others again; the row GEMV puts the same rows of all routes on the same XCD where its workgroups per route are a
// multiple of 4, and reads them from that XCD's L2: E = 8, top 1, H = 4096, I = 1536, gate_up launches in a step of 32 tokens 123 / 166 us (row
// GEMV / this), of 12 tokens 82 / 76; top 8 of 8, H = 2048, I = 768, 8 tokens 60 / 65.  Every wavefront selects by itself: the rounds times the keys
// per lane are bounded (top 32 of 512, H = 1024, I = 512, one token 33 / 41).
static bool gate_up_topk_pays(int T, int k, int E, int H) {
  const int keys = E <= 128 ? 2 : E <= 256 ? 4 : E <= 512 ? 8 : 16;
  if (H > kGateUpColumns || k * keys > 64) return false;
  if (T <= 3) return true;
  const int routes = T * (k + 1), per_route = (2 * device_cu_count() + routes - 1) / routes;
  return k >= 4 && (per_route % 4 != 0 || T * k <= E);
}

// Down: every workgroup stages the token's activations, and a lane has 8 pieces of a row in flight.  Ahead while one batch of pieces makes the
// row (a second one is a second round trip; short rows per route are worse for the row GEMV, whose spans are 1024 wide) and the
// workgroups are few rounds of the chip, fewer where the activations are long, more where the row fills the lanes (top 8 and more).
// Step's time with row GEMVs and sum / with this, us: top 1 of 8, H = 4096, I = 512, 64 tokens 130 / 268; top 8 of 128, H = 2048, I = 768, one token
// 20.3 / 18.2, 12 tokens 119 / 108; top 3 of 8, H = 2176, I = 2048, two tokens 26.1 / 27.6; top 8 of 64, H = 2048, I = 256, 12 tokens 71 / 52.
static bool down_sum_pays(int T, int k, int H, int I) {
  const long long pieces = (long long)(k + 1) * (I / 16), groups = (long long)T * ((H + kDownWaves - 1) / kDownWaves);
  const long long cus = device_cu_count(), batch = 64 * kDownPieces;
  if ((long long)(k + 1) * I * 2 > kDownSumBytes || (pieces > batch && I > 640)) return false;
  return groups <= 2 * cus || (groups <= 4 * cus && I <= 1536) || (groups <= 12 * cus && k >= 8 && pieces <= batch);
}

}  // namespace qlin

using namespace qlin;

extern "C" {

int mi_moe_decode_plan(int T, int topk, int num_experts, int H, int I, int* plan) {
  if (!plan) return MI_ERR_ARG;
  if (T < 0 || topk < 1 || num_experts < 1 || H < 1 || I < 1) return MI_ERR_SHAPE;
  *plan = 0;
  if ((long long)T * topk > kRoutedPairs) return MI_OK;
  *plan = MI_DECODE_ROUTED;
  if (topk > 64 || num_experts > 64 * kTopkSlots || topk > num_experts || (H % 128) || (I % 128)) return MI_OK;
  if (gate_up_topk_pays(T, topk, num_experts, H)) *plan |= MI_DECODE_GATE_UP_TOPK;
  if (down_sum_pays(T, topk, H, I)) *plan |= MI_DECODE_DOWN_SUM;
  return MI_OK;
}

int mi_moe_gate_up_topk_fp8_block(const void* x, const void* logits, const void* gate_weight, const void* w, const float* w_scale,
                                  const void* shared_w, const float* shared_scale, void* gate_up, int32_t* top_ids, void* top_w, float* gate,
                                  int T, int topk, int num_experts, int H, int I, int act_dtype, void* stream) {
  if (!x || !logits || !gate_weight || !w || !w_scale || !shared_w || !shared_scale || !gate_up || !top_ids || !top_w || !gate) return MI_ERR_ARG;
  if (act_dtype != DT_F16 && act_dtype != DT_BF16) return MI_ERR_ARG;
  if (T < 0 || T > 65535 || num_experts < 1 || num_experts > 64 * kTopkSlots || topk < 1 || topk > 64 || topk > num_experts) return MI_ERR_SHAPE;
  if (H <= 0 || I <= 0 || (H % 128) || (I % 128) || (long long)(topk + 1) * 2 * I >= (1LL << 31)) return MI_ERR_SHAPE;
  if (H > kGateUpColumns) return MI_ERR_LIMIT;
  if (!T) return MI_OK;
  const GateUpArgs p{x, logits, gate_weight, w, shared_w, w_scale, shared_scale, gate_up, top_ids, top_w, gate, T, topk, num_experts, H, 2 * I};
  return act_dtype == DT_F16 ? launch_gate_up<ActF16>(p, (hipStream_t)stream) : launch_gate_up<ActBF16>(p, (hipStream_t)stream);
}

int mi_moe_down_sum_fp8_block(const void* gate_up, const void* w, const float* w_scale, const void* shared_w, const float* shared_scale,
                              const int32_t* top_ids, const void* top_w, const float* gate, void* out, int T, int topk, int num_experts,
                              int H, int I, int act_dtype, void* stream) {
  if (!gate_up || !w || !w_scale || !shared_w || !shared_scale || !top_ids || !top_w || !gate || !out) return MI_ERR_ARG;
  if (act_dtype != DT_F16 && act_dtype != DT_BF16) return MI_ERR_ARG;
  if (T < 0 || T > 65535 || topk < 1 || num_experts < 1 || H <= 0 || I <= 0 || (H % 128) || (I % 128)) return MI_ERR_SHAPE;
  if ((long long)(topk + 1) * I * 2 > kDownSumBytes) return MI_ERR_LIMIT;
  if (!T) return MI_OK;
  const DownSumArgs p{gate_up, w, shared_w, w_scale, shared_scale, top_ids, top_w, gate, out, T, topk, num_experts, H, I};
  return act_dtype == DT_F16 ? launch_down_sum<ActF16>(p, (hipStream_t)stream) : launch_down_sum<ActBF16>(p, (hipStream_t)stream);
}

}  // extern "C"
