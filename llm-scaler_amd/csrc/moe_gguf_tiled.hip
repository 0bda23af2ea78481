// Grouped GGUF MoE GEMMs over chunks (mi_moe_gguf_grouped's operands) for prompts: the chunks of an expert that
// follow each other are merged into M-tiles and run through the tiled matrix-core GEMM, which dequantizes a weight
// once per tile; the chunk kernel (moe_gguf_grouped.hip) does it once per 64 rows and wavefront.
//   1. one workgroup turns the chunk list into a table of M-tiles {expert, first row, rows, first 16-row
//      activation block} and a table of activation blocks;
//   2. the rows of x are gathered (token list) and re-tiled into MFMA operand order per block;
//   3. the GEMM runs one workgroup per (M-tile, N-tile); gate and up are two stacks of one launch.
#include "gemm_tiled.hpp"
#include "../../include/mi355x_qlinear.h"

namespace qlin {

// 256 x 128, two workgroups per CU, like the FP8 experts' tiles (a wavefront skips the row tiles past the chunk's last).  Layer with top 8
// of 128 experts, H = 2048, I = 768, 256 x 256 (one workgroup per CU) / 256 x 128, us: 1000 tokens 259 / 235, 1500 292 / 270, 2048 332 / 310.
constexpr int kGgufBM = 256, kGgufBN = 128;
constexpr int kChunkRows = 64;                        // rows of a chunk that count
constexpr int kChunkMapThreads = 1024;

template <class Act, int BN> using WQ5P = WGguf<Act, BN, GT_Q5P>;
template <class Act, int BN> using WQ6P = WGguf<Act, BN, GT_Q6P>;

// Chunk i continues chunk i - 1 when that one is full and i goes on behind it with the same expert; a run of
// continuing chunks is cut into tiles of kGgufBM rows.  Thread t owns `per` consecutive chunks; runs across threads
// are found with a running maximum of the run starts, the places of tiles and blocks with two exclusive scans.
// One workgroup and no bandwidth to speak of: what it costs is the chain of dependent reads, a chunk and its neighbours up to
// kPerTile ahead, several times over.  So the list is read once, in order, into one byte per chunk in LDS (rows, and whether it
// continues), and the chain runs there.  Before / after, alone: 8.4 / 6.1 us for 128 experts' prompts of
// 2048 tokens, that layer 319 / 316; down launch of 2560 chunks 346 / 335, of 6400 821 / 783, up to 1024 no difference.
__global__ __launch_bounds__(kChunkMapThreads) void chunk_tile_map_kernel(const int32_t* __restrict__ chunks, int n, int E,
                                                                          int out_rows, int32_t* __restrict__ g_tile,
                                                                          int32_t* __restrict__ blk, int32_t* __restrict__ counts) {
  constexpr int kPerTile = kGgufBM / kChunkRows;
  __shared__ int s_a[kChunkMapThreads / 64], s_b[kChunkMapThreads / 64], s_c[kChunkMapThreads / 64];
  extern __shared__ __align__(16) uint8_t s_info[];   // n bytes: rows that count (0: skipped), kContinues
  constexpr int kContinues = 128;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int per = (n + kChunkMapThreads - 1) / kChunkMapThreads;
  const int i0 = min(tid * per, n), i1 = min(i0 + per, n);
  auto live = [&](int e, int t0, int nt) {
    return nt <= 0 || e < 0 || e >= E || t0 < 0 || t0 >= out_rows ? 0 : min(min(nt, kChunkRows), out_rows - t0);
  };
  for (int i = tid; i < n; i += kChunkMapThreads) {
    const int j = max(i - 1, 0);
    const int e = chunks[3 * i], t0 = chunks[3 * i + 1], r = live(e, t0, chunks[3 * i + 2]);
    const int pe = chunks[3 * j], pt0 = chunks[3 * j + 1], pr = live(pe, pt0, chunks[3 * j + 2]);
    const bool c = i > 0 && r > 0 && pr == kChunkRows && e == pe && t0 - kChunkRows == pt0;
    s_info[i] = (uint8_t)(r | (c ? kContinues : 0));
  }
  __syncthreads();
  auto rows = [&](int i) { return s_info[i] & (kContinues - 1); };
  auto continues = [&](int i) { return s_info[i] >= kContinues; };
  // last run start in the own chunks, then the last one before them
  int last = -1;
  for (int i = i0; i < i1; ++i)
    if (!continues(i)) last = i;
  int m = last;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(m, off);
    if (lane >= off) m = max(m, o);
  }
  if (lane == 63) s_a[w] = m;
  int before = __shfl_up(m, 1);
  if (lane == 0) before = -1;
  __syncthreads();
  for (int i = 0; i < w; ++i) before = max(before, s_a[i]);
  // tiles and blocks that start in the own chunks
  auto tile_rows = [&](int i) {
    int r = rows(i);
    for (int k = 1; k < kPerTile && i + k < n && continues(i + k); ++k) r += rows(i + k);
    return r;
  };
  auto starts = [&](int i, int& run) {
    if (!continues(i)) run = i;
    return rows(i) > 0 && (i - run) % kPerTile == 0;
  };
  int tiles = 0, blocks = 0, run = before;
  for (int i = i0; i < i1; ++i)
    if (starts(i, run)) {
      ++tiles;
      blocks += (tile_rows(i) + 15) >> 4;
    }
  int it = tiles, ib = blocks;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int ot = __shfl_up(it, off), ob = __shfl_up(ib, off);
    if (lane >= off) { it += ot; ib += ob; }
  }
  if (lane == 63) { s_b[w] = it; s_c[w] = ib; }
  __syncthreads();
  int at = it - tiles, ab = ib - blocks, all_t = 0, all_b = 0;
  for (int i = 0; i < kChunkMapThreads / 64; ++i) {
    if (i < w) { at += s_b[i]; ab += s_c[i]; }
    all_t += s_b[i]; all_b += s_c[i];
  }
  run = before;
  for (int i = i0; i < i1; ++i)
    if (starts(i, run)) {
      const int r = tile_rows(i), t0 = chunks[3 * i + 1];
      int32_t* t = g_tile + 4 * at;
      t[0] = chunks[3 * i]; t[1] = t0; t[2] = r; t[3] = ab;
      ++at;
      for (int b = 0; b * 16 < r; ++b, ++ab) {
        blk[2 * ab] = t0 + 16 * b;
        blk[2 * ab + 1] = min(16, r - 16 * b);
      }
    }
  if (tid == 0) { counts[0] = all_t; counts[1] = all_b; }
}

// {re-tiled x, tile table, block table, counts}: at most one tile per chunk, four blocks per chunk
struct ChunkLayout { long long tile_off, blk_off, cnt_off, total; };
static inline ChunkLayout chunk_layout(long long n, long long K) {
  ChunkLayout L;
  L.tile_off = (n * kChunkRows * K * 2 + 255) & ~255LL;
  L.blk_off = L.tile_off + ((n * 16 + 255) & ~255LL);
  L.cnt_off = L.blk_off + ((n * (kChunkRows / 16) * 8 + 255) & ~255LL);
  L.total = L.cnt_off + 256;
  return L;
}

template <template <class, int> class FMT>
static int launch_chunk_gemm(GemmArgs p, int nmat, int max_tiles, hipStream_t st) {
  using F = FMT<ActF16, kGgufBN>;
  p.tiles_m = (max_tiles + 7) / 8 * 8;                // whole rounds of the 8 XCDs (surplus workgroups exit)
  p.tiles_n = nmat * ((p.N + kGgufBN - 1) / kGgufBN);
  if ((long long)p.tiles_m * p.tiles_n >= (1LL << 31)) return MI_ERR_SHAPE;
  auto kern = gemm_tiled_kernel<ActF16, F, kGgufBM, kGgufBN, true, false, false, 2, 4>;
  constexpr size_t lds = TileLds<F>::kBytes;
  static_assert(lds <= 64 * 1024, "more dynamic LDS has to be asked for");
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_m * p.tiles_n)), dim3(256), lds, st, p);
  return launch_status();
}

// Which of the two kernels a chunk list takes, from what the host knows of it: its length, not its contents.  A list
// that covers its buffer holds out_rows rows in chunks of which at most one per expert is not full.  Where the buffer is
// larger than the list can cover, its rows are at least those of the full chunks; where the list is longer, its chunks do
// not merge.  The experts' tiles follow from the chunks as on average for independent remainders.
// Time in us.  Tiled: tables and re-tiling, then a chain of K / 64 steps per round of one workgroup per CU, and the
// multiplications of the live rows.  Chunks: a chain of K steps, and a part per chunk and per 64 rows for every million
// weights.  The constants are a fit to a tile of 256 columns with one workgroup per CU, which the tiles of 128 columns outrun; a fit to
// those misjudges sizes that it was not made from (left-out sizes: 10 to 21 % of the launches go to tiles that are over 3 % slower), so these constants stay and the margin is
// what moves for the down launches: 0.95 up, 1.05 down.  The down margin was picked on 1242 launches (1 .. 256 experts, H 1024 .. 4096,
// I 512 .. 2048, 8 .. 400 rows per expert; even, drawn and skewed counts) and checked on 1053 of nine other sizes: it moves 30 of these to the
// tiles, 0.62 to 0.98 of the chunks' time and one 1.02; all picks together are never more than 1.02, and 179 launches that stay on chunks
// would be faster by more than 3 %, at most 2.35 times.  At 1.1 the down tiles are up to 1.28 times slower, and the up launch of 256 experts,
// H = 2048, I = 512 and 60 rows is 176 on tiles against 159 for even counts.
// Chunks / tiles in us, up and Q5_K down launch, drawn counts: E = 128, H = 2048, I = 768, 60 rows per expert 143 / 130, 103 / 83, 96 rows
// 219 / 153, 158 / 94, 256 rows 449 / 321, 330 / 186; E = 256, H = 2048, I = 512, 60 rows 175 / 176, 140 / 121, 96 rows 294 / 225, 232 / 141;
// E = 12, H = 4096, I = 1024, 60 rows 57 / 53, 31 / 36, 112 rows 99 / 61, 57 / 40.
static bool chunk_tiles_pay(bool up, long long n, long long out_rows, long long E, long long N, long long K, long long nmat) {
  if (kChunkRows * n > out_rows + kChunkRows * E) return false;
  const long long rows = out_rows <= kChunkRows * n ? out_rows : std::max(n, kChunkRows * (n - E));
  const long long used = std::min(E, n), m_tiles = std::min(n, std::max(used, (2 * n + 3 * used + 7) / 8));
  const long long cus = device_cu_count_gemm(), n_tiles = nmat * ((N + 255) / 256);
  const double rounds = (double)((m_tiles * n_tiles + cus - 1) / cus), full = (double)(rows * n_tiles) / (double)(kGgufBM * cus);
  const double steps = (double)(K / 64), weights = (double)(nmat * N * K) / 1e6, r64 = (double)rows / kChunkRows;
  const double tiled = up ? 17.0 + steps * (0.97 * rounds + 1.64 * full) : 18.0 + steps * (1.11 * rounds + 2.16 * full);
  const double chunks = up ? 7.0 + 0.41 * steps + weights * (0.12 * (double)n + 0.18 * r64)
                           : 9.0 + 0.41 * steps + weights * (0.21 * (double)n + 0.18 * r64);
  return tiled < (up ? 0.95 : 1.05) * chunks;
}

}  // namespace qlin

using namespace qlin;

extern "C" {

int mi_moe_gguf_grouped_tiled_pays(int fmt, int nmat, int num_chunks, int out_rows, int num_experts, int N, int K, int* pays) {
  if (!pays) return MI_ERR_ARG;
  if ((fmt != 2 && fmt != 5 && fmt != 6) || nmat < 1 || nmat > 2 || num_experts < 1) return MI_ERR_ARG;
  if (num_chunks < 0 || out_rows < 0 || N < 0 || K <= 0) return MI_ERR_SHAPE;
  long long bytes = 0;
  *pays = !(nmat == 2 && fmt != 2) && mi_moe_gguf_grouped_tiled_workspace(num_chunks, K, &bytes) == MI_OK && num_chunks && N &&
          chunk_tiles_pay(fmt == 2, num_chunks, out_rows, num_experts, N, K, nmat);
  return MI_OK;
}

int mi_moe_gguf_grouped_tiled_workspace(int num_chunks, int K, long long* bytes) {
  if (!bytes) return MI_ERR_ARG;
  if (num_chunks < 0 || K <= 0 || (K % 128)) return MI_ERR_SHAPE;
  if ((long long)num_chunks * kChunkRows * K * 2 >= (1LL << 31)) return MI_ERR_SHAPE;
  *bytes = chunk_layout(num_chunks, K).total;
  return MI_OK;
}

int mi_moe_gguf_grouped_tiled_ws(int fmt, const void* x, int x_rows, const int32_t* tok_ids, int nmat, const void* const* ql,
                                 const void* const* qh, const void* const* scale, const void* const* qmin, void* out,
                                 long long out_stride, int out_rows, const int32_t* chunks, int num_chunks, int num_experts,
                                 int N, int K, void* workspace, long long workspace_bytes, void* stream) {
  if (!x || !ql || !scale || !out || !chunks) return MI_ERR_ARG;
  if (fmt != 2 && fmt != 5 && fmt != 6) return MI_ERR_ARG;
  if (nmat < 1 || nmat > 2 || (nmat == 2 && fmt != 2) || num_experts < 1) return MI_ERR_ARG;
  if (x_rows < 0 || out_rows < 0 || num_chunks < 0 || N < 0) return MI_ERR_SHAPE;
  long long need = 0;
  if (const int rc = mi_moe_gguf_grouped_tiled_workspace(num_chunks, K, &need)) return rc;
  if (out_stride < (long long)nmat * N || out_stride >= (1LL << 31)) return MI_ERR_SHAPE;
  if ((uint64_t)N * (uint64_t)K >= (1ull << 31) || (uint64_t)x_rows * (uint64_t)K * 2 >= (1ull << 31)) return MI_ERR_SHAPE;
  for (int i = 0; i < nmat; ++i) {
    if (!ql[i] || !scale[i]) return MI_ERR_ARG;
    if (fmt != 6 && (!qmin || !qmin[i])) return MI_ERR_ARG;
    if (fmt != 2 && (!qh || !qh[i])) return MI_ERR_ARG;
  }
  if (!num_chunks || !N || !out_rows || !x_rows) return MI_OK;
  if (!workspace || workspace_bytes < need) return MI_ERR_ARG;
  const ChunkLayout L = chunk_layout(num_chunks, K);
  char* ws = (char*)workspace;
  int32_t *tile = (int32_t*)(ws + L.tile_off), *blk = (int32_t*)(ws + L.blk_off), *cnt = (int32_t*)(ws + L.cnt_off);
  hipStream_t st = (hipStream_t)stream;
  if (num_chunks > 64 * 1024) {                       // fewer than 131072: K is at least 128 and the re-tiled rows stay below 2 GiB
    static const int raised = hipFuncSetAttribute(reinterpret_cast<const void*>(chunk_tile_map_kernel),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024) == hipSuccess ? MI_OK : MI_ERR_LAUNCH;
    if (raised != MI_OK) return raised;
  }
  hipLaunchKernelGGL(chunk_tile_map_kernel, dim3(1), dim3(kChunkMapThreads), (size_t)num_chunks, st, chunks, num_chunks, num_experts, out_rows, tile,
                     blk, cnt);
  const int Q = K / 32, max_blocks = num_chunks * (kChunkRows / 16);
  hipLaunchKernelGGL(pack_x_grouped_kernel<true>, dim3((unsigned)max_blocks * ((Q + kPackQ - 1) / kPackQ)), dim3(256), 0, st,
                     (const uint16_t*)x, tok_ids, blk, cnt, (u32x4*)ws, x_rows, K, Q, 1);
  GemmArgs p{};
  const long long nk = (long long)N * K;
  p.x = ws; p.w = ql[0]; p.scale = scale[0]; p.out = out; p.M = out_rows; p.N = N; p.K = K;
  p.zp = fmt != 6 ? qmin[0] : nullptr;
  p.qh = fmt != 2 ? qh[0] : nullptr;
  if (nmat == 2) { p.w1 = ql[1]; p.scale1 = scale[1]; p.zp1 = qmin[1]; }
  p.g_tile = tile; p.g_count = cnt;
  p.g_w_stride = nk / 2;
  p.g_s_stride = fmt == 6 ? nk / 8 : nk / 16;
  p.g_z_stride = nk / 16;
  p.g_h_stride = fmt == 5 ? nk / 8 : nk / 4;
  p.x_blocks = max_blocks; p.out_rows = out_rows; p.out_ld = (int)out_stride;
  if (fmt == 2) return launch_chunk_gemm<WQ4K>(p, nmat, num_chunks, st);
  return fmt == 5 ? launch_chunk_gemm<WQ5P>(p, nmat, num_chunks, st) : launch_chunk_gemm<WQ6P>(p, nmat, num_chunks, st);
}

}  // extern "C"
