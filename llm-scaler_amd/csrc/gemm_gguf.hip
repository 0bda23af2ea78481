// Prefill GEMMs on the GGUF formats Q4_0, Q8_0, Q5_K and Q6_K (repacked) for more than 64 activation
// rows: the tiled matrix-core GEMM of gemm_tiled.hpp, which reads and dequantizes a weight once per
// 128 or 256 rows of x; the weight-streaming kernel does it once per 64 (M=500, K=N=5120, Q6_K:
// 168 us streaming, 66 us tiled).
#include "gemm_tiled.hpp"
#include "../../include/mi355x_qlinear.h"

namespace qlin {

template <class Act, int BN> using WQ40 = WGguf<Act, BN, GT_Q40>;
template <class Act, int BN> using WQ80 = WGguf<Act, BN, GT_Q80>;
template <class Act, int BN> using WQ5K = WGguf<Act, BN, GT_Q5K>;
template <class Act, int BN> using WQ6K = WGguf<Act, BN, GT_Q6K>;

}  // namespace qlin

using namespace qlin;

extern "C" {

int mi_gemm_gguf_tiled_ws(int fmt, const void* x, const void* w, const void* qh, const void* scale, const void* qmin,
                          void* out, void* workspace, long long workspace_bytes, int M, int N, int K, void* stream) {
  if (!x || !w || !scale || !out) return MI_ERR_ARG;
  if (fmt < GT_Q40 || fmt > GT_Q6K) return MI_ERR_ARG;
  if ((fmt == GT_Q5K || fmt == GT_Q6K) && !qh) return MI_ERR_ARG;
  if (fmt == GT_Q5K && !qmin) return MI_ERR_ARG;
  if (M < 0 || N < 0 || K <= 0 || (K % (fmt == GT_Q5K || fmt == GT_Q6K ? 512 : 128))) return MI_ERR_SHAPE;
  if ((uint64_t)(M + 15) * (uint64_t)K * 2 >= (1ull << 31) || (uint64_t)N * (uint64_t)K >= (1ull << 31)) return MI_ERR_SHAPE;
  if (!M || !N) return MI_OK;
  if (!workspace || workspace_bytes < (long long)((M + 15) & ~15) * K * 2) return MI_ERR_ARG;
  GemmArgs p{};
  p.w = w; p.qh = qh; p.scale = scale; p.zp = qmin; p.out = out; p.M = M; p.N = N; p.K = K;
  hipStream_t st = (hipStream_t)stream;
  switch (fmt) {
    case GT_Q40: return run_gemm_tiled<ActF16, WQ40>(p, x, workspace, workspace_bytes, st);
    case GT_Q80: return run_gemm_tiled<ActF16, WQ80>(p, x, workspace, workspace_bytes, st);
    case GT_Q5K: return run_gemm_tiled<ActF16, WQ5K>(p, x, workspace, workspace_bytes, st);
    default: return run_gemm_tiled<ActF16, WQ6K>(p, x, workspace, workspace_bytes, st);
  }
}

}  // extern "C"
