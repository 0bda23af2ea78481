// Prefill GEMMs on the GGUF formats Q4_0, Q8_0, Q5_K and Q6_K (repacked) for more than 64 activation
// rows: the tiled matrix-core GEMM of gemm_tiled.hpp, which reads and dequantizes a weight once per
// 128 to 256 rows of x; the weight-streaming kernel does it once per 64 (M=500, K=N=5120, Q6_K:
// 168 us streaming, 45 us tiled).
#include "gemm_tiled.hpp"
#include "../../include/mi355x_qlinear.h"

namespace qlin {

template <class Act, int BN> using WQ40 = WGguf<Act, BN, GT_Q40>;
template <class Act, int BN> using WQ80 = WGguf<Act, BN, GT_Q80>;
template <class Act, int BN> using WQ5K = WGguf<Act, BN, GT_Q5K>;
template <class Act, int BN> using WQ6K = WGguf<Act, BN, GT_Q6K>;

// 65 .. 128 rows: up to which K two passes of the weight-streaming kernels are ahead.  They are at their best where the
// weight gives a CU one 16-row block or a little less or more, and on short rows, which the tiles' pipeline does not
// amortise; the K-sliced kernel takes Q4_0 and Q8_0 further than the others.  Streaming / tiled in us (M x N x K):
// Q6_K 112 x 4096 x 1024 10.2 / 15.4, 112 x 3072 x 2560 15.8 / 18.3, 112 x 1024 x 2048 12.3 / 11.9, 80 x 10240 x 1024 20.0 / 11.9,
// 80 x 1024 x 1024 11.8 / 9.9, 128 x 1048 x 1024 10.1 / 12.1; Q8_0 80 x 4096 x 3072 14.6 / 18.6, 128 x 1024 x 3072 16.1 / 12.2;
// Q4_0 80 x 4096 x 4096 16.7 / 19.3, 128 x 1024 x 4096 19.3 / 13.0.  Of 663 problems that take the tiles (N 256 .. 10240, K 512 .. 4096) 64
// are slower there by more than 3 %, at most 1.19 times.  The line was drawn before the tall tiles, on the safe side of them now: of 537
// that stream, 168 would be faster on the tiles by more than 3 %, at most 1.55 times (Q8_0 115 x 10168 x 1152 18.7 / 12.0).
static int stream_k(int fmt, long M, long N) {
  const long cus = device_cu_count_gemm();
  const bool one_block = N >= 8 * cus && N <= 16 * cus;
  if (fmt == GT_Q40) return one_block && M <= 96 ? 4096 : 3072;
  if (fmt == GT_Q80) return one_block ? 3072 : 2048;
  if (one_block) return M <= 96 ? 2560 : 3072;
  if (M <= 96 || N > 32 * cus) return 0;
  return N < 8 * cus ? 1024 : 1536;
}

}  // namespace qlin

using namespace qlin;

extern "C" {

int mi_gemm_gguf_tiled_pays(int fmt, int M, int N, int K, int* pays) {
  if (!pays || fmt < 2 || fmt > GT_Q6K) return MI_ERR_ARG;
  if (M < 0 || N < 0 || K <= 0) return MI_ERR_SHAPE;
  *pays = M > 64 && N && K % 128 == 0;
  if (fmt == 2) return MI_OK;
  if ((uint64_t)(M + 15) * (uint64_t)K * 2 >= (1ull << 31) || (uint64_t)N * (uint64_t)K >= (1ull << 31)) *pays = 0;
  if ((fmt == GT_Q5K || fmt == GT_Q6K) && K % 512) *pays = 0;
  if (M <= 128 && K <= stream_k(fmt, M, N)) *pays = 0;
  return MI_OK;
}

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
