// Prefill GEMM for gfx950 on quantized weights: out[M,N] = x[M,K] @ dequant(w[N,K])^T with
// fp16 / bf16 activations, templated on the weight format (INT4 group 128, FP8 E4M3 with
// per-channel / per-tensor / 128x128 block scales, GGUF Q4_K in its repacked representation).
//
// MFMA-bound regime (M in the hundreds or thousands).  A workgroup of 4 wavefronts (2 x 2; 4 x 1 on
// the tall, narrow tiles of problems that do not fill the chip otherwise, see gemm_small_tile)
// owns a BM x BN output tile; each wavefront computes a sub-tile of it with
// v_mfma_f32_16x16x32_{bf16,f16}, accumulators in the AGPR half of the register file.  Large
// tiles are limited by the matrix pipe, tall ones by what a CU moves per step (measured with eight wavefronts: LDS reads 230 to
// 290 B/ns, LDS writes 185, L1 148, L2 132 to 145), so only the operand that has to be shared goes through LDS:
//   * weights: each 64-wide K step of the BN weight rows is loaded once per workgroup (128-bit
//     loads), dequantized to the activation type in registers and written to a double-buffered
//     LDS tile (row pitch 144 B, so the 16 rows of an MFMA operand read fall into distinct
//     banks); every weight is dequantized once per workgroup and reused by all BM rows;
//   * activations: never touch LDS.  A small pre-pass re-tiles x into MFMA operand order (one
//     1 KiB block per 16 rows x 32 k, lane l's 16 bytes at l * 16), so that a wavefront fetches
//     an operand with one fully contiguous 128-bit load per lane straight from global memory /
//     L2 into a 4-deep register ring, 3 K steps of 32 ahead of its use.  (Read from the
//     row-major matrix, the 64 lanes of an operand hit 64 different 16-byte pieces of 16 rows
//     and the texture addresser becomes the bottleneck.)  The re-tiled copy lives in a caller-
//     provided workspace of roundup(M, 16) * K * 2 bytes.
// The dequantization is cut into small pieces that are placed behind individual MFMAs, so the
// vector ALU works in the shadow of the matrix pipe.  One barrier per 64-wide K step.  The
// weights are the MFMA A operand, so a lane ends up with 4 consecutive output columns of one
// row and stores them as 8 bytes.
//
// A weight format is a policy class: how a 64-wide K step of a weight row is cut into chunks (16
// bytes; 8 for nibbles on narrow tiles), which side loads (scales, zero-points, mins) a chunk needs, the dequantization of a
// chunk as a sequence of small pieces, and an optional factor on the finished sums.
#pragma once
#include "qlinear_common.hpp"
#include <algorithm>
#include <type_traits>
#include <utility>

namespace qlin {

struct GemmArgs {
  const void* x;              // activations re-tiled into MFMA operand order (the workspace)
  const void* w;
  const void* scale;
  const void* zp;             // int4: zero-points (may be null); Q4_K / Q5_K: mins
  const void* qh;             // Q5_K / Q6_K: high bits
  void* out;
  int M, N, K;
  int tiles_m, tiles_n;
  int xcd_m;                  // dense launches: the 8 XCDs form an xcd_m x (8 / xcd_m) grid over the tiles (0: none)
  int scale_mode;             // fp8: 0 = per output channel, 1 = per tensor / expert, 2 = 128x128 blocks,
                              // 3 = two per expert: weight rows below n_half, rows from n_half on
  int scale_f16;              // fp8 per channel: the scales are fp16 instead of fp32
  // Grouped launch (GROUPED kernels): M-tile i of the grid belongs to expert g_tile[4 i] and covers
  // the rows [g_tile[4 i + 1], + g_tile[4 i + 2]) of the expert-sorted order; its activations
  // start at 16-row block g_tile[4 i + 3] of the re-tiled copy (every expert's rows are padded
  // to whole blocks there).  g_count[0] = number of M-tiles; M = rows of x (all experts).
  // The matrices of expert e start e * g_w_stride bytes into w and e * g_s_stride bytes into
  // scale.  out rows: sorted position, or out_map[position]; optional factor row_weight[row].
  const int32_t* g_tile;
  const int32_t* g_count;
  long long g_w_stride, g_s_stride;
  long long g_z_stride, g_h_stride;   // GGUF stacks: mins, high bits
  const void *w1, *scale1, *zp1;      // a second stack of matrices (w1 set): N-tiles from tiles_n / 2 on take it, output columns N ..
  int out_ld;                 // GROUPED: columns of a row of out (0: the output columns)
  const int32_t* out_map;
  const void* row_weight;
  int x_blocks;               // 16-row blocks in the re-tiled activations
  int n_half;                 // FUSE: weight row n (gate) pairs with row n + n_half (up); N = 2 n_half
  int gelu;                   // FUSE: tanh-GELU instead of SiLU
  int out_rows;               // rows of out (bounds mapped rows)
  int splits, split_steps;    // SPLIT: the 64-wide steps of K go to `splits` workgroups per tile, split_steps (even) each
  float* partial;             // SPLIT: fp32 sums, [split][tile][wave][column tile][row tile][lane][4]
  int out_packed;             // GROUPED: out is written in the re-tiled operand order of x (16-row blocks of the
                              // tile table, n_out / 32 steps each) for a following grouped GEMM; out_rows = 16 x blocks
};

// MFMA with the accumulator pinned to the AGPR half of the register file and updated in place.
// Left to the register allocator, the 224-256 accumulator registers of a 128 x 128 wave tile
// get split and copied around the loop; the constraint keeps them where they are.  The compiler does
// not know that this is an MFMA and keeps no distance from it: the operands of every call come from LDS /
// global loads (never from a vector-ALU result), and the body of the K loop ends in an explicit wait, so that it lies
// before whatever the register allocator does with the accumulators behind the loop.
template <class Act>
__device__ __forceinline__ void mfma_agpr(f32x4& acc, u32x4 a, u32x4 b) {
  if constexpr (Act::dt == DT_F16)
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// What a weight costs on its way into LDS: one conversion per pair of weights, the other formats, high bits in an array of their own.
enum class GemmDecode { kCheap, kMid, kDear };

constexpr int kBK = 64;
constexpr int kPitch = kBK + 8;                      // elements per LDS row (144 bytes)

// Exact integers as fp16 pairs, one instruction per pair.  Nibbles in bytes: a byte 0..15 read as an E4M3 code is
// n * 2^-9 (the subnormals and the first binade, same spacing).  Bytes: 0x6400 | u is 1024 + u.
__device__ __forceinline__ f16x2 nibbles_f16(uint32_t bytes, bool high) {
  return __builtin_bit_cast(f16x2, high ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(bytes, 512.0f, true)
                                        : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(bytes, 512.0f, false));
}
__device__ __forceinline__ f16x2 planted_f16(uint32_t bytes, bool high) {
  return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, bytes, high ? 0x04030402u : 0x04010400u));
}
// (s0 s1)(s2 s3), (m0 m1)(m2 m3) -> (s0 m0)(s1 m1)(s2 m2)(s3 m3)
__device__ __forceinline__ u32x4 scale_min_pairs(u32x2 s, u32x2 m) {
  return u32x4{__builtin_amdgcn_perm(m[0], s[0], 0x05040100u), __builtin_amdgcn_perm(m[0], s[0], 0x07060302u),
               __builtin_amdgcn_perm(m[1], s[1], 0x05040100u), __builtin_amdgcn_perm(m[1], s[1], 0x07060302u)};
}
template <int DW> using Dwords = std::conditional_t<DW == 4, u32x4, u32x2>;
template <int DW>
__device__ __forceinline__ void load_dwords(Dwords<DW>& v, const __amdgpu_buffer_rsrc_t& r, uint32_t off, uint32_t soff) {
  if constexpr (DW == 4) v = __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0);
  else v = __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0);
}
__device__ __forceinline__ f16x2 both(float v) { return f16x2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ f16x2 both_bits(uint32_t v) { return __builtin_bit_cast(f16x2, (v & 0xffffu) * 0x10001u); }
__device__ __forceinline__ uint32_t bits(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }

// ------------------------------------------------------------------ INT4 group 128
// 32 nibbles per 16-byte chunk, two chunks per row and step; fp16 scale and optional zero-point
// byte per group of 128.  A nibble 0..15 read as an E4M3 code is nib * 2^-9 (codes below 16 are
// the subnormals and the first binade, same spacing), so one v_cvt_pk_f32_fp8 turns two nibbles
// into floats; fma(nib * 2^-9, 512 s, -z s) in fp32 is exact ((nib - z) * s has at most 16
// significant bits), then one RNE to the activation type: the same value as rne((nib - z) * s),
// only the sign of a zero can differ from the subtract-then-multiply form, which no product
// notices.  fp16 activations take the same value from packed fp16: n - z is exact and the product is
// rounded once; the pairs are (0 2)(1 3)(4 6)(5 7) of a dword's 8 nibbles, and x is re-tiled in that order.
template <class Act, int BN>
struct WInt4 {
  static constexpr int CPR = BN <= 64 ? 4 : 2;        // chunks per row and 64-wide step: 8 bytes each on narrow tiles,
  static constexpr int DW = 8 / CPR;                  // so that every thread has one; dwords per chunk
  static constexpr double kWeightBytesPerK = 0.5;
  static constexpr int B_CH = (BN * CPR + 255) / 256; // chunks per thread
  static constexpr int kEntry = 4;                    // bytes per row of a scale table: scale, zero-point (see gemm_tiled_kernel)
  static constexpr bool kHalfEntry = false;
  static constexpr int LPC = 1;                       // load instructions per chunk
  static constexpr int kPieces = B_CH * DW * 8;        // 8 pieces per packed dword of 8 nibbles
  static constexpr GemmDecode kDecode = GemmDecode::kMid;
  static constexpr bool kOutScale = false;
  static constexpr bool kHalf = Act::dt == DT_F16;
  static constexpr bool kPermK = kHalf;
  struct Res {
    __amdgpu_buffer_rsrc_t wr, sr, zr;
    bool has_zp;
    int Kg;
  };
  struct Stage {
    Dwords<DW> b[B_CH];
  };
  struct Side { uint32_t s, z; };                     // a row's fp16 scale bits and zero-point of 128 k
  struct Dq {
    uint32_t e, o;
    f32x2 fe, fo;
    f16x2 te, to, sh[B_CH], nz[B_CH];                 // fp16: scale and -z
    u32x4 outv;
    float sf[B_CH], nzs[B_CH];                        // bf16: 512 * scale and -z * scale (exact)
  };
  static __device__ __forceinline__ Res make(const GemmArgs& p, int = 0) {
    Res r;
    r.Kg = p.K >> 7;
    r.wr = make_rsrc(p.w, (uint32_t)p.N * ((uint32_t)p.K >> 1));
    r.sr = make_rsrc(p.scale, (uint32_t)p.N * (uint32_t)r.Kg * 2u);
    r.zr = make_rsrc(p.zp, p.zp ? (uint32_t)p.N * (uint32_t)r.Kg : 0u);
    r.has_zp = p.zp != nullptr;
    return r;
  }
  // byte offset of chunk kc of row n at k = 0
  static __device__ __forceinline__ uint32_t chunk_addr(Res&, int, int n, int kc, int K) {
    return (uint32_t)n * ((uint32_t)K >> 1) + (uint32_t)(kc * DW * 4);
  }
  static __device__ __forceinline__ void load1(const Res& r, Stage& st, const uint32_t (&boff)[B_CH], int kt, uint32_t dead, int i) {
    load_dwords<DW>(st.b[i], r.wr, boff[i] | dead, (uint32_t)kt * (kBK / 2));
  }
  static __device__ __forceinline__ void side_load(const Res& r, Side& d, int n, int pair, uint32_t dead) {
    d.s = __builtin_amdgcn_raw_buffer_load_b16(r.sr, (uint32_t)n * (uint32_t)r.Kg * 2u | dead, (uint32_t)pair * 2u, 0);
    // without zero-points the resource is empty and the load returns 0
    d.z = __builtin_amdgcn_raw_buffer_load_b8(r.zr, (uint32_t)n * (uint32_t)r.Kg | dead, (uint32_t)pair, 0);
  }
  static __device__ __forceinline__ void side_store(const Side& d, unsigned char* at) { *reinterpret_cast<uint32_t*>(at) = d.s | d.z << 16; }
  static __device__ __forceinline__ void begin(const Res& r, const uint32_t (&v)[B_CH], Dq& q) {
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const _Float16 sc = __builtin_bit_cast(_Float16, (uint16_t)v[i]);
      const float z = r.has_zp ? (float)(v[i] >> 16) : 8.0f;
      if constexpr (kHalf) {
        q.sh[i] = f16x2{sc, sc};
        q.nz[i] = both(-z);
      } else {
        q.sf[i] = (float)sc * 512.0f;
        q.nzs[i] = -z * (float)sc;
      }
    }
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (Act::dt == DT_F16) {
      const f16x2 r = {(_Float16)a, (_Float16)b};
      return __builtin_bit_cast(uint32_t, r);
    } else {
      const bf16x2 r = {(__bf16)a, (__bf16)b};
      return __builtin_bit_cast(uint32_t, r);
    }
  }
  // piece I of the stage; dst[i] = LDS address of chunk i's output in the target buffer
  static __device__ __forceinline__ void piece(const Stage& st, Dq& q, int I, unsigned char* const (&dst)[B_CH]) {
    const int dword = I >> 3, part = I & 7;
    const int i = dword / DW, dw = dword % DW;
    auto pair = [&](float a, float b) {
      return pack2(__builtin_fmaf(a, q.sf[i], q.nzs[i]), __builtin_fmaf(b, q.sf[i], q.nzs[i]));
    };
    if (part == 0) {
      const uint32_t w = st.b[i][dw];
      q.e = w & 0x0F0F0F0Fu;
      q.o = (w >> 4) & 0x0F0F0F0Fu;
    } else if (part == 7) {
      *reinterpret_cast<u32x4*>(dst[i] + dw * 16) = q.outv;
    } else if constexpr (kHalf) {
      const f16x2 s = q.sh[i], nz = q.nz[i];
      if (part == 1 || part == 4) {
        q.te = nibbles_f16(q.e, part == 4);
        q.to = nibbles_f16(q.o, part == 4);
      } else if (part == 2 || part == 5) q.outv[part == 5 ? 2 : 0] = bits((q.te + nz) * s);
      else q.outv[part == 6 ? 3 : 1] = bits((q.to + nz) * s);
    } else if (part == 1) {
      q.fe = __builtin_amdgcn_cvt_pk_f32_fp8((int)q.e, false);
      q.fo = __builtin_amdgcn_cvt_pk_f32_fp8((int)q.o, false);
    } else if (part == 4) {
      q.fe = __builtin_amdgcn_cvt_pk_f32_fp8((int)q.e, true);
      q.fo = __builtin_amdgcn_cvt_pk_f32_fp8((int)q.o, true);
    } else if (part == 2) q.outv[0] = pair(q.fe[0], q.fo[0]);
    else if (part == 3) q.outv[1] = pair(q.fe[1], q.fo[1]);
    else if (part == 5) q.outv[2] = pair(q.fe[0], q.fo[0]);
    else q.outv[3] = pair(q.fe[1], q.fo[1]);
  }
  static __device__ __forceinline__ float out_scale(const Res&, const GemmArgs&, int) { return 1.0f; }
};

// ------------------------------------------------------------------ GGUF Q4_K (repacked)
// The int4 nibble layout with an fp16 scale and an fp16 min per 32 k = per chunk:
// w = fp16(fp16(nib * scale) - min), the product rounded before the subtraction (two roundings,
// as the dense dequantization does): one conversion, one packed product and one packed difference per
// pair of weights.  fp16 activations only; pairs and x in the order of INT4's fp16 form.
template <class Act, int BN>
struct WQ4K {
  static_assert(Act::dt == DT_F16, "Q4_K runs in fp16");
  static constexpr int CPR = BN <= 64 ? 4 : 2;        // chunks per row and 64-wide step: 8 bytes each on narrow tiles,
  static constexpr int DW = 8 / CPR;                  // so that every thread has one; dwords per chunk
  static constexpr double kWeightBytesPerK = 0.5;
  static constexpr int B_CH = (BN * CPR + 255) / 256;
  static constexpr int kEntry = 16, LPC = 1;
  static constexpr bool kHalfEntry = false;
  struct Side { u32x2 s, m; };                        // a row's scales and mins of 128 k
  static constexpr int PPD = 8;                       // pieces per dword of 8 nibbles
  static constexpr int kPieces = B_CH * DW * PPD;
  static constexpr GemmDecode kDecode = GemmDecode::kMid;
  static constexpr bool kOutScale = false;
  static constexpr bool kPermK = true;
  struct Res {
    __amdgpu_buffer_rsrc_t wr, sr, mr;
    int Kc;
  };
  struct Stage {
    Dwords<DW> b[B_CH];
  };
  struct Dq {
    uint32_t e, o;
    f16x2 te, to;
    u32x4 outv;
    f16x2 sv[B_CH], mv[B_CH];
  };
  static __device__ __forceinline__ Res make(const GemmArgs& p, int e = 0) {
    Res r;
    r.Kc = p.K >> 5;
    r.wr = make_rsrc((const char*)p.w + (long long)e * p.g_w_stride, (uint32_t)p.N * ((uint32_t)p.K >> 1));
    r.sr = make_rsrc((const char*)p.scale + (long long)e * p.g_s_stride, (uint32_t)p.N * (uint32_t)r.Kc * 2u);
    r.mr = make_rsrc((const char*)p.zp + (long long)e * p.g_z_stride, (uint32_t)p.N * (uint32_t)r.Kc * 2u);
    return r;
  }
  static __device__ __forceinline__ uint32_t chunk_addr(Res&, int, int n, int kc, int K) {
    return (uint32_t)n * ((uint32_t)K >> 1) + (uint32_t)(kc * DW * 4);
  }
  static __device__ __forceinline__ void load1(const Res& r, Stage& st, const uint32_t (&boff)[B_CH], int kt, uint32_t dead, int i) {
    load_dwords<DW>(st.b[i], r.wr, boff[i] | dead, (uint32_t)kt * (kBK / 2));
  }
  static __device__ __forceinline__ void side_load(const Res& r, Side& d, int n, int pair, uint32_t dead) {
    const uint32_t off = (uint32_t)n * (uint32_t)r.Kc * 2u | dead;
    d.s = __builtin_amdgcn_raw_buffer_load_b64(r.sr, off, (uint32_t)pair * 8u, 0);
    d.m = __builtin_amdgcn_raw_buffer_load_b64(r.mr, off, (uint32_t)pair * 8u, 0);
  }
  static __device__ __forceinline__ void side_store(const Side& d, unsigned char* at) { *reinterpret_cast<u32x4*>(at) = scale_min_pairs(d.s, d.m); }
  static __device__ __forceinline__ void begin(const Res&, const uint32_t (&v)[B_CH], Dq& q) {
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      q.sv[i] = both_bits(v[i]);
      q.mv[i] = both_bits(v[i] >> 16);
    }
  }
  static __device__ __forceinline__ void piece(const Stage& st, Dq& q, int I, unsigned char* const (&dst)[B_CH]) {
#pragma clang fp contract(off)
    const int dword = I / PPD, part = I % PPD;
    const int i = dword / DW, dw = dword % DW;
    if (part == 0) {
      const uint32_t w = st.b[i][dw];
      q.e = w & 0x0F0F0F0Fu;
      q.o = (w >> 4) & 0x0F0F0F0Fu;
    } else if (part == 1 || part == 4) {
      q.te = nibbles_f16(q.e, part == 4);
      q.to = nibbles_f16(q.o, part == 4);
    } else if (part == 2 || part == 5) q.outv[part == 5 ? 2 : 0] = bits(q.te * q.sv[i] - q.mv[i]);
    else if (part == 3 || part == 6) q.outv[part == 6 ? 3 : 1] = bits(q.to * q.sv[i] - q.mv[i]);
    else *reinterpret_cast<u32x4*>(dst[i] + dw * 16) = q.outv;
  }
  static __device__ __forceinline__ float out_scale(const Res&, const GemmArgs&, int) { return 1.0f; }
};

// ------------------------------------------------------------------ GGUF Q4_0 / Q8_0 / Q5_K / Q6_K (repacked)
// fp16 activations only, packed fp16 arithmetic (an MFMA hides two vector instructions, so their number sets the
// time).  Q4_0 is the int4 layout with one scale per 32 k and zero-point 8.  The others bring a byte u per weight
// into place and plant it in 1024 + u:
//   Q8_0: u = code + 128 (sign bit flipped); w = fp16((1024 + u - 1152) s);
//   Q6_K: u = nibble | 2 high bits << 4;     w = fp16((1024 + u - 1056) s); two scales per chunk of 32 k;
//   Q5_K: u = nibble | high bit << 4;        w = fp16(fp16(u s) - min), two roundings, as Q4_K;
// each with the rounding(s) of the dense dequantization.  The high bits are tile-shuffled: inside
// 512 k, byte t holds element p * 128 + t in its 2-bit field p (Q6_K), element p * 64 + t in bit p
// (Q5_K), so the 32 weights of a chunk take one field of 32 consecutive bytes, the same field for
// the whole 64-wide step; the bytes come through L1 again for the other fields.
// GT_Q5P / GT_Q6P: the high bits in element order (the MoE down stacks): a dword's 8 weights take one / two
// consecutive bytes, spread to one field per byte with shifts and masks.
enum { GT_Q40 = 3, GT_Q80 = 4, GT_Q5K = 5, GT_Q6K = 6, GT_Q5P = 7, GT_Q6P = 8 };    // the format numbers of gemv_rows.hpp, skinny_kernel.hpp
template <class Act, int BN, int FMT>
struct WGguf {
  static constexpr int F = FMT == GT_Q5P ? GT_Q5K : FMT == GT_Q6P ? GT_Q6K : FMT;
  static constexpr bool kPlainH = FMT == GT_Q5P || FMT == GT_Q6P;
  static_assert(Act::dt == DT_F16, "GGUF formats run in fp16");
  static constexpr bool kHigh = F == GT_Q5K || F == GT_Q6K;
  static constexpr int CPR = F == GT_Q80 || BN <= 64 ? 4 : 2;
  static constexpr int DW = F == GT_Q80 ? 4 : 8 / CPR;   // dwords per chunk (nibbles: 8 bytes on narrow tiles, as INT4)
  static_assert(!kPlainH || DW == 4, "high bits in element order: whole chunks of 32");
  static constexpr double kWeightBytesPerK = F == GT_Q80 ? 1.0 : F == GT_Q6K ? 0.75 : F == GT_Q5K ? 0.625 : 0.5;
  static constexpr int B_CH = (BN * CPR + 255) / 256;
  static constexpr int kEntry = 16;
  static constexpr bool kHalfEntry = F == GT_Q6K && DW == 2;            // a chunk of 16 k: one of its entry's two scales
  static constexpr int LPC = 1 + (!kHigh ? 0 : kPlainH ? 1 : DW / 2);
  static constexpr int PPD = F == GT_Q5K ? 13 : F == GT_Q6K ? 9 : F == GT_Q40 ? 8 : 3;   // pieces per dword (8 nibbles / 4 bytes)
  static constexpr int kPieces = B_CH * DW * PPD;
  static constexpr GemmDecode kDecode = kHigh ? GemmDecode::kDear : GemmDecode::kMid;
  static constexpr bool kOutScale = false;
  static constexpr bool kPermK = F != GT_Q80;            // pairs (0 2)(1 3)(4 6)(5 7); Q8_0 in order
  struct Res {
    __amdgpu_buffer_rsrc_t wr, sr, mr, hr;
    int Ks;                                           // bytes of scales per row
    uint32_t hoff[kHigh ? B_CH : 1];
  };
  struct Stage {
    Dwords<DW> b[B_CH];
    u32x4 h[kHigh && !kPlainH ? B_CH : 1][DW / 2];
    u32x2 hp[kPlainH ? B_CH : 1];
    uint32_t sh;                                      // shift of this step's field of the high-bit bytes (uniform)
  };
  struct Dq {
    uint32_t e, o, h0, h1;
    f16x2 te, to;
    u32x4 outv;
    f16x2 sv[B_CH][F == GT_Q6K ? DW / 2 : 1], mv[F == GT_Q5K ? B_CH : 1];
  };
  static __device__ __forceinline__ Res make(const GemmArgs& p, int e = 0) {
    Res r;
    const uint32_t nk = (uint32_t)p.N * (uint32_t)p.K;      // < 2^31 (checked by the host)
    r.Ks = (F == GT_Q6K ? p.K >> 4 : p.K >> 5) * 2;
    r.wr = make_rsrc((const char*)p.w + (long long)e * p.g_w_stride, F == GT_Q80 ? nk : nk / 2);
    r.sr = make_rsrc((const char*)p.scale + (long long)e * p.g_s_stride, (uint32_t)p.N * (uint32_t)r.Ks);
    r.mr = make_rsrc((const char*)p.zp + (long long)e * p.g_z_stride, F == GT_Q5K ? (uint32_t)p.N * (uint32_t)r.Ks : 0u);
    r.hr = make_rsrc((const char*)p.qh + (long long)e * p.g_h_stride, F == GT_Q6K ? nk / 4 : F == GT_Q5K ? nk / 8 : 0u);
    return r;
  }
  static __device__ __forceinline__ uint32_t chunk_addr(Res& r, int i, int n, int kc, int K) {
    if constexpr (kHigh) r.hoff[i] = (uint32_t)n * (F == GT_Q6K ? (uint32_t)K >> 2 : (uint32_t)K >> 3) +
                                     (uint32_t)(kc * (!kPlainH ? DW * 8 : F == GT_Q6K ? 8 : 4));
    return (uint32_t)n * (F == GT_Q80 ? (uint32_t)K : (uint32_t)K >> 1) + (uint32_t)(kc * DW * 4);
  }
  static __device__ __forceinline__ void load1(const Res& r, Stage& st, const uint32_t (&boff)[B_CH], int kt, uint32_t dead, int idx) {
    const uint32_t k0 = (uint32_t)kt * kBK;
    const int i = idx / LPC, kind = idx % LPC;
    if (kind == 0) load_dwords<DW>(st.b[i], r.wr, boff[i] | dead, F == GT_Q80 ? k0 : k0 >> 1);
    else if constexpr (kPlainH) {
      if constexpr (F == GT_Q6K) st.hp[i] = __builtin_amdgcn_raw_buffer_load_b64(r.hr, r.hoff[i] | dead, k0 >> 2, 0);
      else st.hp[i][0] = __builtin_amdgcn_raw_buffer_load_b32(r.hr, r.hoff[i] | dead, k0 >> 3, 0);
    } else if constexpr (kHigh) {
      const uint32_t tile = F == GT_Q6K ? (k0 >> 9) * 128u + (k0 & 127u) : (k0 >> 9) * 64u;
      st.h[i][kind - 1] = __builtin_amdgcn_raw_buffer_load_b128(r.hr, r.hoff[i] | dead, tile + (uint32_t)(kind - 1) * 16u, 0);
      st.sh = F == GT_Q6K ? (k0 >> 7 & 3u) * 2u : k0 >> 6 & 7u;
    }
  }
  struct Side { u32x4 s; u32x2 m; };                  // a row's scales (Q6_K 8, others 4) and mins of 128 k
  static __device__ __forceinline__ void side_load(const Res& r, Side& d, int n, int pair, uint32_t dead) {
    const uint32_t off = (uint32_t)n * (uint32_t)r.Ks | dead;
    if constexpr (F == GT_Q6K) d.s = __builtin_amdgcn_raw_buffer_load_b128(r.sr, off, (uint32_t)pair * 16u, 0);
    else {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r.sr, off, (uint32_t)pair * 8u, 0);
      d.s = u32x4{v[0], v[1], 0u, 0u};
      if constexpr (F == GT_Q5K) d.m = __builtin_amdgcn_raw_buffer_load_b64(r.mr, off, (uint32_t)pair * 8u, 0);
    }
  }
  static __device__ __forceinline__ void side_store(const Side& d, unsigned char* at) {
    if constexpr (F == GT_Q6K) *reinterpret_cast<u32x4*>(at) = d.s;       // the two scales of every 32 k
    else *reinterpret_cast<u32x4*>(at) = scale_min_pairs(u32x2{d.s[0], d.s[1]}, F == GT_Q5K ? d.m : u32x2{0u, 0u});
  }
  static __device__ __forceinline__ void begin(const Res&, const uint32_t (&v)[B_CH], Dq& q) {
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      q.sv[i][0] = both_bits(v[i]);
      if constexpr (F == GT_Q6K && DW == 4) q.sv[i][1] = both_bits(v[i] >> 16);
      if constexpr (F == GT_Q5K) q.mv[i] = both_bits(v[i] >> 16);
    }
  }
  static __device__ __forceinline__ void piece(const Stage& st, Dq& q, int I, unsigned char* const (&dst)[B_CH]) {
#pragma clang fp contract(off)
    const int dword = I / PPD, part = I % PPD;
    const int i = dword / DW, dw = dword % DW;
    const uint32_t w = st.b[i][dw];
    if constexpr (F == GT_Q40) {
      const f16x2 s = q.sv[i][0], m8 = both(-8.0f);
      if (part == 0) {
        q.e = w & 0x0F0F0F0Fu;
        q.o = (w >> 4) & 0x0F0F0F0Fu;
      } else if (part == 1 || part == 4) {
        q.te = nibbles_f16(q.e, part == 4);
        q.to = nibbles_f16(q.o, part == 4);
      } else if (part == 7) *reinterpret_cast<u32x4*>(dst[i] + dw * 16) = q.outv;
      else if (part == 2 || part == 5) q.outv[part == 5 ? 2 : 0] = bits((q.te + m8) * s);
      else q.outv[part == 6 ? 3 : 1] = bits((q.to + m8) * s);
    } else if constexpr (F == GT_Q80) {
      // one dword = 4 weights = half of a 16-byte LDS write
      if (part == 0) q.e = w ^ 0x80808080u;
      else {
        q.outv[(dw & 1) * 2 + part - 1] = bits((planted_f16(q.e, part == 2) + both(-1152.0f)) * q.sv[i][0]);
        if (part == 2 && (dw & 1)) *reinterpret_cast<u32x4*>(dst[i] + (dw >> 1) * 16) = q.outv;
      }
    } else {
      constexpr uint32_t kField = F == GT_Q6K ? 0x03030303u : 0x01010101u;
      if (part == 0) {
        q.e = w & 0x0F0F0F0Fu;
        q.o = (w >> 4) & 0x0F0F0F0Fu;
      } else if (kPlainH && part == 1) {
        if constexpr (kPlainH && F == GT_Q6K) {
          const uint32_t v = st.hp[i][dw >> 1] >> (16 * (dw & 1)) & 0xffffu;    // field t: element t
          q.h0 = (v | v << 8) & 0x00FF00FFu;
        } else if constexpr (kPlainH) {
          const uint32_t v = st.hp[i][0] >> (8 * dw) & 0xffu;                   // bit t: element t
          q.h0 = (v | v << 12) & 0x000F000Fu;
        }
      } else if (kPlainH && part == 2) {
        q.h0 = F == GT_Q6K ? (q.h0 | q.h0 << 4) & 0x0F0F0F0Fu : (q.h0 | q.h0 << 6) & 0x03030303u;   // byte m: elements 2 m, 2 m + 1
        q.h1 = F == GT_Q6K ? (q.h0 & 0x0C0C0C0Cu) << 2 : (q.h0 & 0x02020202u) << 3;
      } else if (kPlainH && part == 3) {
        q.e |= (q.h0 & kField) << 4;
        q.o |= q.h1;
      } else if (!kPlainH && part == 1) {
        if constexpr (!kPlainH) {
          q.h0 = st.h[i][dw >> 1][(dw & 1) * 2] >> st.sh & kField;         // elements 0 1 2 3 of the dword's 8
          q.h1 = st.h[i][dw >> 1][(dw & 1) * 2 + 1] >> st.sh & kField;     // elements 4 5 6 7
        }
      } else if (part == 2) {
        const uint32_t he = __builtin_amdgcn_perm(q.h1, q.h0, 0x06040200u);
        q.h1 = __builtin_amdgcn_perm(q.h1, q.h0, 0x07050301u);
        q.h0 = he;
      } else if (part == 3) {
        q.e |= q.h0 << 4;
        q.o |= q.h1 << 4;
      } else if (part == PPD - 1) *reinterpret_cast<u32x4*>(dst[i] + dw * 16) = q.outv;
      else {
        const int pr = F == GT_Q6K ? part - 4 : (part - 4) >> 1;       // outv[pr]: pairs of e, o, e, o
        const bool first = F == GT_Q6K || (part & 1) == 0;
        if (first) q.te = planted_f16(pr & 1 ? q.o : q.e, pr >> 1) + both(F == GT_Q6K ? -1056.0f : -1024.0f);
        if constexpr (F == GT_Q6K) q.outv[pr] = bits(q.te * q.sv[i][dw >> 1]);   // dw >> 1: 16-wide group of the chunk
        else if (!first) q.outv[pr] = bits(q.te * q.sv[i][0] - q.mv[i]);
      }
    }
  }
  static __device__ __forceinline__ float out_scale(const Res&, const GemmArgs&, int) { return 1.0f; }
};

// ------------------------------------------------------------------ FP8 E4M3
// 16 codes per 16-byte chunk, four chunks per row and step.  BLOCK = false: the decode is exact
// (every E4M3 value is a 16-bit float) and the per-channel or per-tensor scale multiplies the
// finished sum.  BLOCK = true: one fp32 scale per 128 x 128 block, folded into the weight
// (decode to fp32, multiply, one rounding to the activation type) because the accumulators
// cannot be rescaled per K block.
template <class Act, int BN, bool BLOCK>
struct WFp8 {
  static constexpr int CPR = 4;
  static constexpr double kWeightBytesPerK = 1.0;
  static constexpr int B_CH = (BN * CPR + 255) / 256;
  static constexpr int LPC = 1, kEntry = BLOCK ? 4 : 0;
  static constexpr bool kHalfEntry = false;
  static constexpr int kPPC = BLOCK ? 10 : 4;         // pieces per chunk
  static constexpr int kPieces = B_CH * kPPC;
  static constexpr GemmDecode kDecode = BLOCK ? GemmDecode::kMid : GemmDecode::kCheap;
  static constexpr bool kOutScale = !BLOCK;
  static constexpr bool kPermK = false;
  struct Res {
    __amdgpu_buffer_rsrc_t wr, sr;
    const void* se;                                   // this expert's scales
    int Kb;
  };
  struct Stage {
    u32x4 b[B_CH];
  };
  struct Side { uint32_t s; };                        // block scale, fp32 bits
  struct Dq {
    u32x4 outv;
    float s[BLOCK ? B_CH : 1];
  };
  // e: expert of a grouped launch (its matrices start e * stride bytes in)
  static __device__ __forceinline__ Res make(const GemmArgs& p, int e = 0) {
    Res r;
    r.Kb = (p.K + 127) >> 7;
    r.wr = make_rsrc((const char*)p.w + (long long)e * p.g_w_stride, (uint32_t)p.N * (uint32_t)p.K);
    r.sr = make_rsrc((const char*)p.scale + (long long)e * p.g_s_stride,
                     BLOCK ? (uint32_t)((p.N + 127) >> 7) * (uint32_t)r.Kb * 4u : 0u);
    r.se = (const char*)p.scale + (long long)e * p.g_s_stride;
    return r;
  }
  static __device__ __forceinline__ uint32_t chunk_addr(Res&, int, int n, int kc, int K) { return (uint32_t)n * (uint32_t)K + (uint32_t)(kc * 16); }
  static __device__ __forceinline__ void load1(const Res& r, Stage& st, const uint32_t (&boff)[B_CH], int kt, uint32_t dead, int i) {
    st.b[i] = __builtin_amdgcn_raw_buffer_load_b128(r.wr, boff[i] | dead, (uint32_t)kt * kBK, 0);
  }
  static __device__ __forceinline__ void side_load(const Res& r, Side& d, int n, int pair, uint32_t dead) {
    d.s = __builtin_amdgcn_raw_buffer_load_b32(r.sr, (uint32_t)(n >> 7) * (uint32_t)r.Kb * 4u | dead, (uint32_t)pair * 4u, 0);
  }
  static __device__ __forceinline__ void side_store(const Side& d, unsigned char* at) { *reinterpret_cast<uint32_t*>(at) = d.s; }
  static __device__ __forceinline__ void begin(const Res&, const uint32_t (&v)[B_CH], Dq& q) {
#pragma unroll
    for (int i = 0; i < (BLOCK ? B_CH : 0); ++i) q.s[i] = __builtin_bit_cast(float, v[i]);
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (Act::dt == DT_F16) {
      const f16x2 r = {(_Float16)a, (_Float16)b};
      return __builtin_bit_cast(uint32_t, r);
    } else {
      const bf16x2 r = {(__bf16)a, (__bf16)b};
      return __builtin_bit_cast(uint32_t, r);
    }
  }
  static __device__ __forceinline__ void piece(const Stage& st, Dq& q, int I, unsigned char* const (&dst)[B_CH]) {
    const int i = I / kPPC, part = I % kPPC;
    if constexpr (!BLOCK) {
      // piece = one dword of four codes -> two packed pairs; a 16-byte write after every second
      const uint32_t w = st.b[i][part];
      uint32_t p0, p1;
      if constexpr (Act::dt == DT_F16) {
        p0 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false));
        p1 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true));
      } else {
        p0 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false));
        p1 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true));
      }
      q.outv[(part & 1) * 2] = p0;
      q.outv[(part & 1) * 2 + 1] = p1;
      if (part & 1) *reinterpret_cast<u32x4*>(dst[i] + (part >> 1) * 16) = q.outv;
    } else {
      // pieces 0-3 and 5-8: half a dword (two codes) -> fp32, scale, one rounding; 4 and 9: write
      const int half = part / 5, sub = part % 5;
      if (sub == 4) {
        *reinterpret_cast<u32x4*>(dst[i] + half * 16) = q.outv;
      } else {
        const uint32_t w = st.b[i][half * 2 + (sub >> 1)];
        const f32x2 f = (sub & 1) ? __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true)
                                  : __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
        q.outv[sub] = pack2(f[0] * q.s[i], f[1] * q.s[i]);
      }
    }
  }
  static __device__ __forceinline__ float out_scale(const Res& r, const GemmArgs& p, int n) {
    if (p.scale_mode == 1) return ((const float*)r.se)[0];
    if (p.scale_mode == 3) return ((const float*)r.se)[n >= p.n_half ? 1 : 0];
    return p.scale_f16 ? (float)((const _Float16*)r.se)[n] : ((const float*)r.se)[n];
  }
};

// LDS of a tile: two weight tiles of 64 k, and behind them two tables of scales (128 k, one entry per row).
template <class Fmt> struct TileLds {
  static constexpr int kTileBytes = Fmt::B_CH * 256 / Fmt::CPR * kPitch * 2;
  static constexpr int kBytes = 2 * kTileBytes + 2 * 256 * Fmt::kEntry;
};

template <int... I, class F>
__device__ __forceinline__ void fold_pieces(std::integer_sequence<int, I...>, F f) {
  (f(I), ...);
}

// ------------------------------------------------------------------ kernel
// GROUPED: the M-tiles come from a device-built table of (expert, rows) instead of a regular grid
// (MoE: rows sorted by expert, one weight matrix per expert).  FUSE: the tile's weight rows
// alternate, 16 at a time, between a gate block and the up block n_half rows further on, and the
// epilogue writes act(gate) * up (N / 2 output columns).
// OCC: workgroups per CU that the registers have to leave room for.  WR: rows of the grid of wavefronts.
// SPLIT: blockIdx.y takes one slice of K and the fp32 sums go to a workspace in accumulator order (1 KiB
// per store); split_reduce_kernel adds the slices and writes the output.
template <class Act, class Fmt, int BM, int BN, bool GROUPED = false, bool FUSE = false, bool SPLIT = false, int OCC = 1, int WR = 2>
__global__ __launch_bounds__(256, OCC) void gemm_tiled_kernel(const GemmArgs p) {
  using Elem = typename Act::elem;
  constexpr int WC = 4 / WR;                          // the wavefronts form a WR x WC grid
  constexpr int WM = BM / WR, WN = BN / WC;           // wave sub-tile
  constexpr int TM = WM / 16, TN = WN / 16;
  constexpr int B_CH = Fmt::B_CH;                     // weight chunks of the tile per thread
  constexpr int CPR = Fmt::CPR;
  constexpr int BNP = B_CH * 256 / CPR;               // LDS rows of the weight tile (>= BN)
  constexpr int kLoads = Fmt::LPC * B_CH;             // load instructions per stage and thread
  static_assert(WM % 16 == 0 && WN % 16 == 0 && BNP >= BN, "tile shape");

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];        // [2][BNP][kPitch], tables of scales
  using Lds = TileLds<Fmt>;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int wn0 = wave % WC * WN;

  // Tile order.  The 8 XCDs take workgroups round-robin and each has its own L2, so the tile of a
  // workgroup is derived from (XCD = id % 8, slot on that XCD = id / 8):
  //   dense: the XCDs form an xcd_m x (8 / xcd_m) grid over the tile matrix and each walks its
  //     block of it M-tile first, so that the workgroups resident on an XCD share a few weight
  //     tiles and a few slabs of x and every operand byte is fetched by as few L2s as possible
  //     (xcd_m = 0: plain order, consecutive workgroups share the weight tile);
  //   grouped: XCD x owns one M-tile of every 8 and walks the N-tiles of one M-tile
  //     back to back, so an M-tile's activations are fetched into one L2 once (its N-tiles read
  //     different weight rows: there is nothing else to share).
  int tm, tn;
  if constexpr (GROUPED) {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int round = slot / p.tiles_n;               // rotate, so that no XCD gets all the experts' short last tiles
    tm = round * 8 + ((xcd + round) & 7);
    tn = slot - round * p.tiles_n;
  } else if (p.xcd_m) {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int per_m = p.tiles_m / p.xcd_m, per_n = p.tiles_n / (8 / p.xcd_m);
    tm = (xcd % p.xcd_m) * per_m + slot % per_m;
    tn = (xcd / p.xcd_m) * per_n + slot / per_m;
  } else {
    tn = blockIdx.x / p.tiles_m;
    tm = blockIdx.x - tn * p.tiles_m;
  }
  int m0 = tm * BM;
  const int n0 = FUSE ? tn * (BN / 2) : (GROUPED && p.w1 && tn >= p.tiles_n >> 1 ? tn - (p.tiles_n >> 1) : tn) * BN;   // FUSE: first gate row
  int M = p.M;
  const int N = p.N, K = p.K;
  const int Q = K / 32;                               // 32-wide MFMA steps
  int kt0 = 0, KT = K / kBK;                          // 64-wide steps of this workgroup (even: K % 128 == 0)
  if constexpr (SPLIT) {
    kt0 = blockIdx.y * p.split_steps;
    KT = kt0 + p.split_steps < KT ? kt0 + p.split_steps : KT;
  }
  const int Qe = 2 * KT;
  int expert = 0, row0 = 0, xblk0 = 0;
  if constexpr (GROUPED) {
    if (tm >= p.g_count[0]) return;                   // the grid is an upper bound of the tile count
    expert = p.g_tile[4 * tm];
    row0 = p.g_tile[4 * tm + 1];
    M = p.g_tile[4 * tm + 2];                         // rows of this tile
    xblk0 = p.g_tile[4 * tm + 3];
    m0 = 0;
  }

  const int Mp = (p.M + 15) & ~15;
  const uint32_t xtiles = GROUPED ? (uint32_t)p.x_blocks : (uint32_t)(Mp >> 4);
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(p.x, xtiles * 16u * (uint32_t)K * 2u);
  int col0 = 0;                                       // first output column of this workgroup's matrix
  const void *mw = p.w, *ms = p.scale, *mz = p.zp;
  if constexpr (GROUPED && !FUSE) {
    if (p.w1 && tn >= p.tiles_n >> 1) {
      mw = p.w1; ms = p.scale1; mz = p.zp1;
      col0 = N;
    }
  }
  GemmArgs mat = p;
  mat.w = mw; mat.scale = ms; mat.zp = mz;
  typename Fmt::Res res = Fmt::make(mat, expert);
  // 16-row activation tile b of this wavefront inside the BM-row tile.  GROUPED: the wavefronts stacked along M
  // take the tiles in turn and a wavefront multiplies only the first 4, 3, 2 or 1 of its tiles, as many as have rows of the
  // expert in them (the K loop exists in these lengths; a branch per MFMA costs more than it saves), so an expert's
  // short last tile costs a fraction of the matrix-core time.
  const int wr = wave / WC;
  auto mtile = [&](int b) { return GROUPED ? WR * b + wr : wr * TM + b; };
  int live = TM;
  if constexpr (GROUPED) live = __builtin_amdgcn_readfirstlane((((M + 15) >> 4) - wr + WR - 1) / WR);
  // weight row of row r of the LDS tile
  auto tile_row = [&](int r) { return FUSE ? n0 + (r >> 5) * 16 + (r & 15) + ((r >> 4) & 1) * p.n_half : n0 + r; };

  f32x4 acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- activations: register ring.  Block (16-row tile t, 32-wide step q) of the
  // re-tiled x sits at (t * Q + q) * 1024; tile and step enter as a scalar offset.
  const uint32_t xlane = (uint32_t)lane * 16u;
  const uint32_t xtile0 = (uint32_t)xblk0 + (uint32_t)(m0 >> 4);
  u32x4 xring[4][TM];
  uint32_t xtoff[TM];                                 // scalar: byte offset of tile b's block row
#pragma unroll
  for (int b = 0; b < TM; ++b) {
    const uint32_t t = xtile0 + mtile(b) < xtiles ? xtile0 + mtile(b) : xtiles - 1;   // tiles past M: any valid block
    xtoff[b] = __builtin_amdgcn_readfirstlane(t * (uint32_t)Q * 1024u);
  }
  auto load_x1 = [&](int slot, int b, int q) {        // a step beyond the last re-reads the last (never used)
    const uint32_t qc = (uint32_t)(q < Qe ? q : Qe - 1);
    xring[slot][b] = __builtin_amdgcn_raw_buffer_load_b128(xr, xlane, xtoff[b] + qc * 1024u, 0);
  };
  auto load_x = [&](int slot, int q) {
#pragma unroll
    for (int b = 0; b < TM; ++b) load_x1(slot, b, q);
  };

  // ---- weights: per-thread chunk addresses at k = 0
  auto row_live = [&](int row) { return row < BN && (FUSE ? n0 + (row >> 5) * 16 + (row & 15) < p.n_half : n0 + row < N); };
  uint32_t boff[B_CH];
  unsigned char* blds[B_CH];
#pragma unroll
  for (int i = 0; i < B_CH; ++i) {
    const int row = (tid + i * 256) / CPR, kc = (tid + i * 256) % CPR;
    const uint32_t dead = (uint32_t)!row_live(row) << 31;
    boff[i] = Fmt::chunk_addr(res, i, tile_row(row), kc, K) | dead;
    blds[i] = smem + (row * kPitch + kc * (kBK / CPR)) * 2;
  }
  using StageB = typename Fmt::Stage;                 // weight chunks of one 64-wide step, in registers
  // One of the loads of a stage, so that the main loop can issue them one at a time between
  // MFMAs: a wavefront that issues vector-memory instructions back to back stalls ~35 cycles
  // on each.
  auto load_b1 = [&](StageB& st, int kt, int idx) {
    const uint32_t dead = kt < KT ? 0u : 0x80000000u;
    Fmt::load1(res, st, boff, kt, dead, idx);
  };
  auto load_b = [&](StageB& st, int kt) {
#pragma unroll
    for (int idx = 0; idx < kLoads; ++idx) load_b1(st, kt, idx);
  };

  // Scales and mins through LDS.  Loaded by the threads that dequantize a chunk they are 2 to 4 bytes of a line per row,
  // array and step, and the lines do not stay in L1 until the next step.  Thread t loads 128 k of tile row t at once, one table
  // entry, every second step.  In step kt (even) table kt / 2 + 1 is written; the steps that read it are kt + 1 and kt + 2, and
  // its place was read last in step kt - 2.  With loads per chunk / with the table, us, M x K x N: Q4_K 2048 x 5120 x 5120 112 / 109,
  // Q5_K 1000 x 4096 x 12288 118 / 113, Q6_K 110 / 106, Q8_0 96.5 / 94, INT4 2048 x 4096 x 14336 201 / 199, Q4_K 500 x 5120 x 10240 75 / 71;
  // block-scaled FP8 (one load per chunk that a wavefront shares) the same within 1 %.
  constexpr int kEntry = Fmt::kEntry;
  unsigned char* const side = smem + 2 * Lds::kTileBytes;
  auto side_at = [&](int pair) { return side + (pair & 1) * (256 * kEntry); };
  auto load_side = [&](auto& d, int pair) __attribute__((always_inline)) {
    if constexpr (kEntry != 0) Fmt::side_load(res, d, tile_row(tid), pair, (uint32_t)(!row_live(tid) || 2 * pair >= KT) << 31);
  };
  auto begin_stage = [&](int kt, auto& q) __attribute__((always_inline)) {
    uint32_t v[B_CH];
    if constexpr (kEntry != 0) {
      const int kc = tid % CPR;
      const unsigned char* at = side_at(kt >> 1) + tid / CPR * kEntry + (kEntry == 16 ? (kt & 1) * 8 + kc * 2 / CPR * 4 : 0);
#pragma unroll
      for (int i = 0; i < B_CH; ++i) {
        if constexpr (Fmt::kHalfEntry) v[i] = *reinterpret_cast<const uint16_t*>(at + i * (256 / CPR * kEntry) + (kc & 1) * 2);
        else v[i] = *reinterpret_cast<const uint32_t*>(at + i * (256 / CPR * kEntry));
      }
    }
    Fmt::begin(res, v, q);
  };

  constexpr int kPieces = Fmt::kPieces;
  using DqState = typename Fmt::Dq;
  auto dq_piece = [&](const StageB& st, int buf, int I, DqState& q) {
    unsigned char* dst[B_CH];
#pragma unroll
    for (int i = 0; i < B_CH; ++i) dst[i] = blds[i] + buf * Lds::kTileBytes;
    Fmt::piece(st, q, I, dst);
  };

  typename Fmt::Side sd;
  // One 64-wide K step: multiply out of LDS buffer `buf` (two 32-wide MFMA steps,
  // ring slots slot0 and slot0 + 1) while the next step's weights (`cur`, loaded one
  // step earlier) are dequantized into the other buffer and the weights two steps
  // ahead are fetched into `nxt`.
  // pieces are spread evenly over the MFMAs of the step: piece I goes behind the
  // first MFMA slot with (slot + 1) * kPieces / kMfmas > I
  auto step64 = [&](auto live_c, int kt, int buf, int slot0, StageB& cur, StageB& nxt) __attribute__((always_inline)) {
    constexpr int L = decltype(live_c)::value;        // activation tiles multiplied (<= TM)
    constexpr int U = 2 * TN, kMfmas = U * L;         // weight operands of the step
    constexpr int R = L > 6 ? 2 : U < 8 ? 3 : 4;      // operands in registers: read from LDS R - 1 rows of MFMAs ahead
    constexpr int kLead = L;                          // MFMAs ahead of the first piece, while the scales are read
    DqState q;
    begin_stage(kt + 1, q);
    if constexpr (kEntry != 0) {
      if (buf == 0) {
        Fmt::side_store(sd, side_at((kt >> 1) + 1) + tid * kEntry);
        load_side(sd, (kt >> 1) + 2);
      }
    }
    const unsigned char* const wread = smem + buf * Lds::kTileBytes + ((wn0 + j) * kPitch + g * 8) * 2;
    auto rd_w = [&](int u) { return *reinterpret_cast<const u32x4*>(wread + (u % TN * 16 * kPitch + u / TN * 32) * 2); };
    u32x4 wring[R];
#pragma unroll
    for (int u = 0; u + 1 < R; ++u) wring[u] = rd_w(u);
    constexpr int kHalf = TN * L;                     // MFMAs per 32-wide step
    constexpr int kBEvery = kHalf / kLoads > 0 ? kHalf / kLoads : 1;
    // a fold, not a loop: the body exceeds what "#pragma unroll" expands, and a rolled loop would keep the rings on the stack
    fold_pieces(std::make_integer_sequence<int, U>{}, [&](int u) __attribute__((always_inline)) {
      const int s = u / TN, a = u % TN;
      if (u + R - 1 < U) wring[(u + R - 1) % R] = rd_w(u + R - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < L; ++b) {
        mfma_agpr<Act>(acc[a][b], wring[u % R], xring[slot0 + s][b]);
        const int m = a * L + b, slot = u * L + b;    // MFMA inside this 32-wide step, and inside the step
        const int p0 = slot < kLead ? 0 : (slot - kLead) * kPieces / (kMfmas - kLead);
        const int p1 = slot < kLead ? 0 : (slot + 1 - kLead) * kPieces / (kMfmas - kLead);
#pragma unroll
        for (int I = p0; I < p1; ++I) dq_piece(cur, buf ^ 1, I, q);
        // global loads, one at a time: the ring slot multiplied in the previous
        // 32-wide step is refilled 3 steps ahead, and in the first half the weight
        // chunks two 64-wide steps ahead are fetched
        if (m % TN == TN / 2 && m / TN < L) load_x1((slot0 + s + 3) & 3, m / TN, 2 * kt + s + 3);
        if (s == 0 && m % kBEvery == 0 && m / kBEvery < kLoads) load_b1(nxt, kt + 2, m / kBEvery);
        // keep MFMAs, vector-ALU pieces and memory accesses in this order
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    // 8 wait states from the last MFMA until its result may be touched (as the compiler keeps them behind the same instruction as a
    // builtin): exits of the loop begin with copies of accumulators, also ahead of a wait that stands behind the loop.  Here
    // they run in the shadow of the LDS writes (Q6_K 500 x 5120 x 5120 47.0 us with and without; 16 of them cost 0.5 %).
    if (buf == 1) asm volatile("s_nop 7" ::: "memory");
    __syncthreads();
  };

  StageB s0, s1;
  {
    // everything that the loop waits for is requested ahead of the ring's loads: the loop's waits are those of its first turn
    typename Fmt::Side sd0;
    load_side(sd0, kt0 >> 1);
    load_side(sd, (kt0 >> 1) + 1);
    load_b(s0, kt0);
    __builtin_amdgcn_sched_barrier(0);
    load_b(s1, kt0 + 1);
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      __builtin_amdgcn_sched_barrier(0);             // keep the ring's loads in issue order
      load_x(r, 2 * kt0 + r);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kEntry != 0) {
      Fmt::side_store(sd0, side_at(kt0 >> 1) + tid * kEntry);
      __syncthreads();
    }
    DqState q;
    begin_stage(kt0, q);
    // a fold, not a loop: the pieces of the longer formats exceed what "#pragma unroll" expands, and a rolled
    // loop would keep the stage on the stack
    fold_pieces(std::make_integer_sequence<int, kPieces>{}, [&](int I) __attribute__((always_inline)) { dq_piece(s0, 0, I, q); });
  }
  __syncthreads();
  auto k_loop = [&](auto live_c) __attribute__((always_inline)) {
    for (int kt = kt0; kt < KT; kt += 2) {
      step64(live_c, kt, 0, 0, s1, s0);
      step64(live_c, kt + 1, 1, 2, s0, s1);
    }
  };
  if constexpr (!GROUPED) {
    k_loop(std::integral_constant<int, TM>{});
  } else {
    static_assert(TM == 4, "loop lengths");
    if (live > 3) k_loop(std::integral_constant<int, 4>{});
    else if (live > 2) k_loop(std::integral_constant<int, 3>{});
    else if (live > 1) k_loop(std::integral_constant<int, 2>{});
    else k_loop(std::integral_constant<int, 1>{});
  }

  // D = W-tile (rows n) x X-tile^T: lane holds n = 4 g + v (v = 0..3), m = j
  if constexpr (SPLIT) {
    f32x4* dst = reinterpret_cast<f32x4*>(p.partial) +
                 (((size_t)blockIdx.y * (size_t)(p.tiles_m * p.tiles_n) + (size_t)(tn * p.tiles_m + tm)) * 4 + wave) * (TN * TM * 64) + lane;
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
      for (int b = 0; b < TM; ++b)
        if (m0 + mtile(b) * 16 < M) dst[(a * TM + b) * 64] = acc[a][b];       // uniform: row tiles with rows of x in them
    return;
  }
  Elem* out = (Elem*)p.out;
  const int n_out = FUSE ? p.n_half : N;              // output columns
  const int ld = GROUPED && p.out_ld ? p.out_ld : n_out;
  // output row of this lane's row of activation tile b, or -1
  int orow[TM];
  float rw[TM];
#pragma unroll
  for (int b = 0; b < TM; ++b) {
    const int m = m0 + mtile(b) * 16 + j;
    orow[b] = m < M ? m : -1;
    rw[b] = 1.0f;
    if constexpr (GROUPED) {
      if (m < M) {
        const int pos = row0 + m;
        const int dst = p.out_map ? p.out_map[pos] : pos;
        orow[b] = (unsigned)dst < (unsigned)p.out_rows ? dst : -1;   // a mapped row outside the output is dropped
        if (p.row_weight && orow[b] >= 0) rw[b] = Act::to_f32(((const Elem*)p.row_weight)[dst]);
      }
    }
  }
  constexpr int TNO = FUSE ? TN / 2 : TN;             // output column tiles of this wavefront
  // first of this lane's 4 output columns in column tile ao; FUSE: gate tile 2 ao pairs with up tile 2 ao + 1
  auto col_of = [&](int ao) { return FUSE ? n0 + (wn0 >> 1) + ao * 16 + g * 4 : n0 + wn0 + ao * 16 + g * 4; };
  [[maybe_unused]] float os_all[Fmt::kOutScale ? TNO : 1][4];
  [[maybe_unused]] float os_up = 1.0f;
  if constexpr (Fmt::kOutScale) {
    if constexpr (FUSE) os_up = Fmt::out_scale(res, p, p.n_half);
#pragma unroll
    for (int ao = 0; ao < TNO; ++ao)
#pragma unroll
      for (int v = 0; v < 4; ++v) os_all[ao][v] = Fmt::out_scale(res, p, col_of(ao) + v < N ? col_of(ao) + v : N - 1);
  }
  const bool two_scales = p.scale_mode == 3;
  // the lane's 4 results of (row tile b, column tile ao), before the rounding
  auto result4 = [&](auto gelu_c, int b, int ao, float (&r)[4]) __attribute__((always_inline)) {
    const int a = FUSE ? 2 * ao : ao;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float osv = Fmt::kOutScale ? os_all[Fmt::kOutScale ? ao : 0][v] : 1.0f;
      if constexpr (FUSE) {
        // one factor per tensor / expert, or one for the gate rows and one for the up rows
        const float gate = acc[a][b][v] * osv, up = acc[a + 1][b][v] * (two_scales ? os_up : osv);
        if constexpr (decltype(gelu_c)::value) {
          float two_z = 2.0f * (0.7978845608f * (gate + 0.044715f * (gate * gate * gate)));
          two_z = fminf(fmaxf(two_z, -30.0f), 30.0f);
          const float ex = __expf(two_z);
          r[v] = 0.5f * gate * (1.0f + (ex - 1.0f) / (ex + 1.0f)) * up;
        } else {
          r[v] = gate * __builtin_amdgcn_rcpf(1.0f + __expf(-gate)) * up;   // reciprocal to 1 ulp, before a 16-bit rounding
        }
      } else {
        r[v] = Fmt::kOutScale ? acc[a][b][v] * osv : acc[a][b][v];
      }
      if constexpr (GROUPED) r[v] *= rw[b];
    }
  };
  const size_t out_bytes = (size_t)(GROUPED ? p.out_rows : p.M) * (size_t)ld * 2u;
  constexpr int WNO = FUSE ? WN / 2 : WN;             // output columns of this wavefront
  constexpr int LPR = WNO / 8;                        // lanes, 16 bytes each, per output row of the wave tile
  constexpr int RPP = 64 / LPR;                       // rows per store instruction
  constexpr int PASSES = (16 + RPP - 1) / RPP;
  constexpr int OPITCH = WNO * 2 + 16;                // a row of the wave tile + a slot for the row's offset
  static_assert(WNO % 8 == 0 && 4 * 16 * OPITCH <= 2 * Lds::kTileBytes, "output staging tile");
  if (((n_out | ld) & 7) == 0 && out_bytes < (1ull << 31) && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0) {
    // Each 16-row tile of results is rounded, turned through a tile in LDS that belongs to this
    // wavefront alone (the weight tiles are free after the K loop's last barrier; the LDS queue of a
    // wavefront runs in order, so no barrier) and leaves as 16 bytes per lane, a row's columns in
    // adjacent lanes: a store instruction writes RPP rows of WNO * 2 contiguous bytes instead of 32
    // bytes in each of 16 rows — the workgroup's path to L2 takes a request per row piece, whatever
    // its size.  Rows and column groups outside the output get an offset past the buffer and are dropped.
    const __amdgpu_buffer_rsrc_t orsrc = make_rsrc(p.out, (uint32_t)out_bytes);
    unsigned char* otile = smem + wave * (16 * OPITCH);
    unsigned char* wr_at = otile + j * OPITCH + g * 8;
    const int rr = lane / LPR, cc = lane - rr * LPR;
    const int colr = (FUSE ? n0 + (wn0 >> 1) : n0 + wn0) + cc * 8;     // this lane's 8 columns when it stores
    const bool lane_ok = rr < RPP && colr < n_out;
    auto emit = [&](auto gelu_c) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < TM; ++b) {
        if (GROUPED && b >= live) break;              // uniform: the tiles past the expert's rows
        *reinterpret_cast<uint32_t*>(otile + j * OPITCH + WNO * 2) =
            orow[b] >= 0 ? (uint32_t)orow[b] * (uint32_t)ld * 2u : kOOB;
#pragma unroll
        for (int ao = 0; ao < TNO; ++ao) {
          float r[4];
          result4(gelu_c, b, ao, r);
          u32x2 d;
          if constexpr (Act::dt == DT_F16) {
            d[0] = __builtin_bit_cast(uint32_t, f16x2{(_Float16)r[0], (_Float16)r[1]});
            d[1] = __builtin_bit_cast(uint32_t, f16x2{(_Float16)r[2], (_Float16)r[3]});
          } else {
            d[0] = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)r[0], (__bf16)r[1]});
            d[1] = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)r[2], (__bf16)r[3]});
          }
          *reinterpret_cast<u32x2*>(wr_at + ao * 32) = d;
        }
        if constexpr (GROUPED && WNO % 32 == 0) {
          if (p.out_packed) {
            // block (activation tile, 32-wide step) = 1 KiB in operand order: lane 16 g + j holds row j,
            // columns 8 g .. 8 g + 7 of the step; rows past the expert's last are zeros here (their
            // activations were) as the re-tiling pass would write them
            const uint32_t tile = (uint32_t)xblk0 + (uint32_t)mtile(b);
            const int cb = FUSE ? n0 + (wn0 >> 1) : n0 + wn0;
#pragma unroll
            for (int qq = 0; qq < WNO / 32; ++qq) {
              const u32x4 v = *reinterpret_cast<const u32x4*>(otile + j * OPITCH + (qq * 32 + g * 8) * 2);
              const uint32_t q = (uint32_t)(cb >> 5) + qq;
              __builtin_amdgcn_raw_buffer_store_b128(
                  v, orsrc, cb + qq * 32 < n_out ? (tile * (uint32_t)(n_out >> 5) + q) * 1024u + (uint32_t)lane * 16u : kOOB, 0, 0);
            }
            continue;
          }
        }
#pragma unroll
        for (int ps = 0; ps < PASSES; ++ps) {
          const int row = ps * RPP + rr;
          const unsigned char* src = otile + (row < 16 ? row : 15) * OPITCH;
          const u32x4 v = *reinterpret_cast<const u32x4*>(src + cc * 16);
          const uint32_t ro = *reinterpret_cast<const uint32_t*>(src + WNO * 2);
          const bool ok = lane_ok && row < 16;
          __builtin_amdgcn_raw_buffer_store_b128(v, orsrc, ok ? ro + (uint32_t)(colr + col0) * 2u : kOOB, 0, 0);
        }
      }
    };
    if (FUSE && p.gelu) emit(std::true_type{});
    else emit(std::false_type{});
  } else {
    auto emit = [&](auto gelu_c) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < TM; ++b) {
        if (orow[b] < 0) continue;
#pragma unroll
        for (int ao = 0; ao < TNO; ++ao) {
          const int n = col_of(ao);
          float r[4];
          result4(gelu_c, b, ao, r);
          Elem* dst = out + (size_t)orow[b] * ld + col0 + n;
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (n + v < n_out) dst[v] = Act::from_f32(r[v]);
        }
      }
    };
    if (FUSE && p.gelu) emit(std::true_type{});
    else emit(std::false_type{});
  }
}

// Re-tile x [M, K] (16-bit, row-major) into MFMA operand order: block (t, q) holds
// rows 16 t .. 16 t + 15, k = 32 q .. 32 q + 31; lane l = 16 g + j of the block
// (16 bytes at l * 16) holds row 16 t + j, k = 32 q + 8 g .. + 7.  Rows past M are
// zero.  One workgroup writes four blocks, contiguously.  (Reading the rows contiguously and
// turning them through an LDS tile, as the grouped variant does, was measured slower here:
// 9.1 against 7.3 us for 2048 x 4096.)
// perm_k: the 8 elements of a lane leave in the order 0 2 1 3 4 6 5 7 (weight formats whose
// dequantization produces that order).
constexpr int kPackQ = 16;                            // grouped variant: 32-wide steps per workgroup
constexpr int kPackPitch = kPackQ * 64 + 16;          // and its LDS row pitch (operand reads hit distinct banks)
// dwords (x0 x1)(x2 x3)(x4 x5)(x6 x7) -> (x0 x2)(x1 x3)(x4 x6)(x5 x7)
__device__ __forceinline__ u32x4 perm_k8(u32x4 v) {
  return u32x4{__builtin_amdgcn_perm(v[1], v[0], 0x05040100u), __builtin_amdgcn_perm(v[1], v[0], 0x07060302u),
               __builtin_amdgcn_perm(v[3], v[2], 0x05040100u), __builtin_amdgcn_perm(v[3], v[2], 0x07060302u)};
}
static __global__ __launch_bounds__(256) void pack_x_kernel(const uint16_t* __restrict__ x, u32x4* __restrict__ xp,
                                                            int M, int K, int Q, int perm_k) {
  const int l = threadIdx.x & 63;
  const int nq4 = (Q + 3) >> 2;                       // flat grid: 4 steps of one row tile per workgroup
  const int t = blockIdx.x / nq4;
  const int q = (blockIdx.x - t * nq4) * 4 + (threadIdx.x >> 6);
  if (q >= Q) return;
  const int m = t * 16 + (l & 15);
  u32x4 v = {0u, 0u, 0u, 0u};
  if (m < M) v = *reinterpret_cast<const u32x4*>(x + (size_t)m * K + q * 32 + (l >> 4) * 8);
  if (perm_k) v = perm_k8(v);
  xp[((size_t)t * Q + q) * 64 + l] = v;
}

// Gather + re-tile: block b of the table -> MFMA operand order (see pack_x_kernel); rows past the
// block's count are zero.  One workgroup re-tiles 16 consecutive 32-wide steps of one block: each
// wavefront reads 1 KiB of each of four (gathered) rows, the rows meet in an LDS tile and leave
// as 16 contiguous blocks.
template <bool PERM = false>
__global__ __launch_bounds__(256) void pack_x_grouped_kernel(const uint16_t* __restrict__ x,
                                                             const int32_t* __restrict__ row_map,
                                                             const int32_t* __restrict__ blk,
                                                             const int32_t* __restrict__ counts,
                                                             u32x4* __restrict__ xp, int a_rows, int K, int Q,
                                                             int row_div) {
  __shared__ __attribute__((aligned(16))) unsigned char tile[16 * kPackPitch];
  const int nq = (Q + kPackQ - 1) / kPackQ;           // flat grid: kPackQ steps of one block per workgroup
  const int b = blockIdx.x / nq;
  if (b >= counts[1]) return;
  const int l = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q0 = (blockIdx.x - b * nq) * kPackQ;
  const int live = blk[2 * b + 1], first = blk[2 * b];
  // Unconditional loads with indices held in range, the surplus zeroed afterwards: a branch around
  // each (map entry, row piece) pair would make the four pairs eight dependent round trips.
  u32x4 v[4];
  unsigned row[4];
  const int k = q0 * 32 + l * 8;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = wave * 4 + i;
    const int pos = first + (r < live ? r : 0);
    row[i] = row_map ? (unsigned)row_map[pos] : (unsigned)pos;
  }
  if (row_map && row_div != 1) {                      // after all four entries have been requested
#pragma unroll
    for (int i = 0; i < 4; ++i) row[i] /= (unsigned)row_div;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool ok = wave * 4 + i < live && k < K && row[i] < (unsigned)a_rows;
    v[i] = *reinterpret_cast<const u32x4*>(x + (ok ? (size_t)row[i] * K + k : (size_t)0));
    if (!ok) v[i] = u32x4{0u, 0u, 0u, 0u};
    if constexpr (PERM) v[i] = perm_k8(v[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(tile + (wave * 4 + i) * kPackPitch + l * 16) = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = q0 + wave * 4 + i;
    if (q < Q)
      xp[((size_t)b * Q + q) * 64 + l] =
          *reinterpret_cast<const u32x4*>(tile + (l & 15) * kPackPitch + (wave * 4 + i) * 64 + (l >> 4) * 16);
  }
}

// Adds the K slices of a SPLIT launch (in slice order), scales, rounds and writes the output.  A wavefront
// takes one 16 x 16 accumulator tile: lane 16 g + j holds row j, columns 4 g .. 4 g + 3.  grid (tiles, 4 TN TM / 4).
template <class Act, class Fmt, int BM, int BN, int WR>
__global__ __launch_bounds__(256) void split_reduce_kernel(const GemmArgs p) {
  using Elem = typename Act::elem;
  constexpr int WC = 4 / WR, TM = BM / WR / 16, TN = BN / WC / 16;
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  const int tile = blockIdx.x;
  const int at = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + (threadIdx.x >> 6));   // [wave][column tile][row tile]
  const int wave = at / (TN * TM), a = at / TM % TN, b = at % TM;
  const int tn = tile / p.tiles_m, tm = tile - tn * p.tiles_m;
  const int m = tm * BM + wave / WC * (BM / WR) + b * 16, n = tn * BN + wave % WC * (BN / WC) + a * 16 + g * 4;
  if (m >= p.M) return;                               // uniform
  const size_t slice = (size_t)p.tiles_m * p.tiles_n * (BM * BN / 4);                   // in f32x4
  const f32x4* src = reinterpret_cast<const f32x4*>(p.partial) + (size_t)tile * (BM * BN / 4) + (size_t)at * 64 + lane;
  f32x4 sum = src[0];
#pragma unroll 4
  for (int i = 1; i < p.splits; ++i) sum += src[(size_t)i * slice];
  if (m + j >= p.M) return;
  if constexpr (Fmt::kOutScale) {
    const typename Fmt::Res res = Fmt::make(p);
#pragma unroll
    for (int v = 0; v < 4; ++v) sum[v] *= Fmt::out_scale(res, p, n + v < p.N ? n + v : p.N - 1);
  }
  Elem* out = (Elem*)p.out + (size_t)(m + j) * p.N + n;
  if (n + 3 < p.N && (p.N & 3) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 7) == 0) {
    Elem r[4] = {Act::from_f32(sum[0]), Act::from_f32(sum[1]), Act::from_f32(sum[2]), Act::from_f32(sum[3])};
    *reinterpret_cast<u32x2*>(out) = __builtin_bit_cast(u32x2, r);
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (n + v < p.N) out[v] = Act::from_f32(sum[v]);
  }
}

template <class Act, class Fmt, int BM, int BN, bool SPLIT = false, int WR = 2>
static int launch_gemm_tiled(GemmArgs p, hipStream_t st) {
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  // XCD grid: among the splits that divide both tile counts, the one with the least operand
  // traffic (a weight tile is fetched by xcd_m L2s, a slab of x by 8 / xcd_m)
  p.xcd_m = 0;
  {
    const double wbytes = (double)p.N * p.K * Fmt::kWeightBytesPerK, xbytes = (double)p.M * p.K * 2.0;
    double best = 0.0;
    for (int a = 1; a <= 8; a *= 2) {
      if (p.tiles_m % a || p.tiles_n % (8 / a)) continue;
      const double cost = a * wbytes + (8 / a) * xbytes;
      if (!p.xcd_m || cost < best) { best = cost; p.xcd_m = a; }
    }
  }
  constexpr size_t lds = TileLds<Fmt>::kBytes;
  auto kern = gemm_tiled_kernel<Act, Fmt, BM, BN, false, false, SPLIT, 1, WR>;
  if (lds > 64 * 1024) {
    static bool raised = false;                       // opt in to > 64 KiB of dynamic LDS once
    if (!raised) {
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds) != hipSuccess)
        return MI_ERR_LAUNCH;
      raised = true;
    }
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_m * p.tiles_n), (unsigned)(SPLIT ? p.splits : 1)), dim3(256), lds, st, p);
  if constexpr (SPLIT)
    hipLaunchKernelGGL((split_reduce_kernel<Act, Fmt, BM, BN, WR>), dim3((unsigned)(p.tiles_m * p.tiles_n), BM * BN / 1024), dim3(256), 0, st, p);
  return launch_status();
}

// Per K step a workgroup pays for its tile's columns (MFMAs) plus a part that does not shrink with
// the tile (activation loads, barrier, pipeline fill): measured on 5120 x 5120 and 14336 x 4096
// weights, 160- and 192-column tiles cost about (BN + 48) / (256 + 48) of a 256-column tile.
constexpr long kTileFixedCols = 48;

static inline long device_cu_count_gemm() {
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      cus = prop.multiProcessorCount;
    if (cus <= 0) cus = 256;
  }
  return cus;
}

static inline bool gemm_big_tiles(long M, long N) {
  return M > 128 && ((M + 255) / 256) * ((N + 255) / 256) * 2 > device_cu_count_gemm();
}

// K slices of a problem, counted on 128 x 128 tiles.  A tile is a chain of K / 64 steps of about 0.65 us whether its
// neighbours' CUs are busy or not, so a problem with few tiles leaves the chip idle: slices up to one workgroup
// per CU (two per CU share the path from L2 to the CU and gain nothing: Q8_0 1000 x 4096 x 4096, 256 tiles:
// 50 us in one piece, 55 in two).  Every slice writes and reads fp32 sums of the whole output, 8 bytes per
// element at about 5 TB/s, which sets the best number where tiles are few.  The alternative is one piece on a smaller
// tile (gemm_small_tile); slices have to make up for the second launch and the start of their chains.  The line (0.48 us a step in one
// piece, 0.55 in slices) was drawn on 128 x 96 and 128 x 128, and both sides have become faster since.  One piece / slices as they are now in us, M x N x
// K: FP8 block-scaled 320 x 2760 x 1024 11.2 / 15.8 and INT4 256 x 5688 x 1536 14.9 / 21.1 (one piece); INT4 128 x 4096 x 4096 29.4 / 20.5, Q4_K 100 x
// 5120 x 5120 35.0 / 23.7, Q6_K 129 x 5120 x 5120 38.1 / 27.1, INT4 1024 x 2048 x 6144 48.9 / 43.1, FP8 70 x 1024 x 1024 11.1 / 9.6 (slices).
// Of 696 problems in slices (nine formats, M 65 .. 1024, N 128 .. 14336, K 384 .. 8448) 56 would be faster in one piece by more than 3 %, at
// most 1.27 times (Q4_0 81 x 13864 x 2560 19.8 / 25.1); of 81 in one piece none in 2 to 4 slices.
static inline int gemm_splits(long M, long N, long K) {
  if (M <= 64 || N <= 0 || gemm_big_tiles(M, N)) return 1;
  const long tiles = ((M + 127) / 128) * ((N + 127) / 128);
  const long most = std::min(device_cu_count_gemm() / tiles, K / 128);
  const double chain = 0.65 * (double)(K / 64), sums = (double)((M + 15) / 16 * 16) * (double)N * 8.0 / 5e6;   // us
  int best = 1;
  for (long s = 2; s <= most; ++s)
    if (chain / s + sums * s < chain / best + (best > 1 ? sums * best : -2.0)) best = (int)s;     // the second launch: 2 us
  const long steps = (K / 128 + best - 1) / best * 2;                                             // of the longest slice
  return 2.0 + 0.55 * (double)steps + sums * best < 0.48 * (double)(K / 64) ? best : 1;
}

// Tile of the K slices: 128 x 128, or as many tiles of 256 x 64 where these pad no more rows.  256 x 64 decodes a weight
// for twice the rows, but every workgroup reads 256 rows of x instead of 128.  It is ahead where x is small beside the weights (one or
// two row tiles, or no more rows than columns; half of that where the decoding is cheap), where 128 columns would be padding, and where
// a slice is long enough for the decoding to count.  128 x 128 / 256 x 64 in us, M x N x K: Q5_K 145 x 7384 x 2560 30.2 / 23.7, INT4 387 x
// 1720 x 5120 27.1 / 24.6, FP8 block-scaled 978 x 1720 x 6144 45.0 / 38.9; Q4_0 1002 x 224 x 2048 13.2 / 16.4, FP8 per-channel 1189 x 528
// x 8192 33.6 / 41.1, Q4_0 5352 x 280 x 6144 62.4 / 73.8.  Over 1780 problems whose rows pad alike (M 129 .. 6144, N 64 .. 8192) the time
// over that of the better tile is 1.049 on 128 x 128, 1.019 on 256 x 64 and 1.008 by this line (geometric means); 73 are slower than on
// 128 x 128 by more than 3 %, at most 1.16 (on 256 x 64 throughout 355, at most 1.35), 94 slower than on 256 x 64, at most 1.23.
static inline bool gemm_slices_tall(long M, long N, long steps, GemmDecode decode) {
  if ((M + 255) / 256 * 2 != (M + 127) / 128) return false;
  const bool cheap = decode == GemmDecode::kCheap, dear = decode == GemmDecode::kDear;
  if (M <= (cheap ? 256 : 512) || N >= (cheap ? 2 * M : M)) return true;
  if (N <= 64 || (M > 1280 && N > 128 && N <= 192)) return true;
  return dear ? steps >= 8 : !cheap && M <= 1024 && steps >= 10;
}

// Tile of a problem that 256 x 256 tiles would leave half of the chip idle on, K in one piece.  What a
// step costs there is not the matrix pipe but the issue of the dequantization (Q6_K 500 x 5120 x 5120 on 128 x 96: 64 us,
// without the dequantization 34, without the MFMAs 60), and a tile dequantizes its columns whatever its rows.  So tall and
// narrow: the four wavefronts stack up along M, every one takes all columns of the tile, and x is read once per workgroup
// instead of once per wavefront column.  Time of a step relative to 256 x 64 with whole rounds of one workgroup per CU (110
// problems of nine formats, M 66 .. 1024): 256 x 48 0.93, 192 x 64 0.92, 128 x 64 0.89 (four reads of the weight tile from LDS
// for 128 rows, but the shortest chain), on two wavefront columns 128 x 96 1.15, 128 x 128 1.25; where the decode is one
// conversion (unscaled FP8), these are 0.90 and 1.10.  M x K x N, the better of 128 x 96 and 128 x 128 against the choice, us: Q6_K 500 x 5120 x
// 5120 61.0 -> 46.8 (192 x 64), Q5_K 947 x 5120 x 5176 117 -> 95 (192 x 64; 256 x 48 88), Q4_K 352 x 4096 x 13056 75 -> 60 (192 x 64), FP8
// block-scaled 201 x 2048 x 12288 23.5 -> 20.6 (256 x 48), FP8 per-channel 207 x 5120 x 14168 46.5 -> 41.9 (256 x 64), Q4_K 85 x 1536 x
// 14080 17.7 -> 14.2 (128 x 64).  Of 204 problems 13 are more than 3 % off the best of the six, at most 1.13 (unscaled FP8 on 128 x 96).
struct GemmTile { int rows, columns; };
static inline GemmTile gemm_small_tile(long M, long N, GemmDecode decode) {
  const long cus = device_cu_count_gemm();
  const bool cheap = decode == GemmDecode::kCheap;
  const struct { GemmTile tile; long cost; } shapes[] = {{{128, 64}, 89},  {{192, 64}, 92},  {{256, 48}, 93},
                                                         {{256, 64}, 100}, {{128, 96}, cheap ? 90 : 115}, {{128, 128}, cheap ? 110 : 125}};
  GemmTile best{};
  long least = 0;
  for (const auto& s : shapes) {
    const long tiles = ((M + s.tile.rows - 1) / s.tile.rows) * ((N + s.tile.columns - 1) / s.tile.columns);
    const long cost = (tiles + cus - 1) / cus * s.cost;
    if (!least || cost < least) { least = cost; best = s.tile; }
  }
  return best;
}

// 256 rows x 256 / 224 / 192 / 160 columns, whichever needs the least time over its rounds of resident workgroups: rounds x
// (columns of a tile + a fixed part per K step).  A 5120-column weight is 32 tiles of 160: with 8 row tiles exactly one
// round of 256 workgroups, where 256-column tiles fill 160 of the 256 CUs.
static inline GemmTile gemm_big_tile(long M, long N) {
  const long cus = device_cu_count_gemm(), tiles_m = (M + 255) / 256;
  auto cost = [&](long bn) { return ((tiles_m * ((N + bn - 1) / bn) + cus - 1) / cus) * (bn + kTileFixedCols); };
  int best = 256;
  for (int bn : {224, 192, 160})
    if (cost(bn) < cost(best)) best = bn;
  return {256, best};
}

// bytes of the re-tiled activations and, behind them, of the slices' sums
static inline long long gemm_workspace(long M, long N, long K, int splits) {
  const long long packed = ((M + 15) & ~15LL) * K * 2;
  return splits < 2 ? packed : packed + (long long)splits * ((M + 127) / 128) * ((N + 127) / 128) * (128 * 128 * 4);
}

// The launch of a problem: its tile, and the slices of K with their length in 64-wide steps.  K slices or a small tile while
// 256 x 256 tiles would leave more than half of the chip idle, else tiles of 256 rows and 160 and more columns.
struct GemmPlan { GemmTile tile; int splits, split_steps; };
static inline GemmPlan gemm_plan(long M, long N, long K, GemmDecode decode, long long workspace_bytes) {
  if (gemm_big_tiles(M, N)) return {gemm_big_tile(M, N), 1, (int)(K / kBK)};
  const int most = gemm_splits(M, N, K);
  if (most < 2 || workspace_bytes < gemm_workspace(M, N, K, most)) return {gemm_small_tile(M, N, decode), 1, (int)(K / kBK)};
  const int steps = (int)((K / 128 + most - 1) / most) * 2, splits = (int)((K / kBK + steps - 1) / steps);
  return {gemm_slices_tall(M, N, steps, decode) ? GemmTile{256, 64} : GemmTile{128, 128}, splits, steps};
}

// Re-tiles x into `workspace` and runs the launch that gemm_plan picks.  FMT is a template taking (Act, BN).
template <class Act, template <class, int> class FMT>
static int run_gemm_tiled(GemmArgs p, const void* x, void* workspace, long long workspace_bytes, hipStream_t st) {
  const int Mp = (p.M + 15) & ~15;
  const int Q = p.K / 32;
  hipLaunchKernelGGL(pack_x_kernel, dim3((unsigned)(((Q + 3) / 4) * (Mp / 16))), dim3(256), 0, st, (const uint16_t*)x,
                     (u32x4*)workspace, p.M, p.K, Q, FMT<Act, 128>::kPermK ? 1 : 0);
  p.x = workspace;
  const GemmPlan plan = gemm_plan(p.M, p.N, p.K, FMT<Act, 128>::kDecode, workspace_bytes);
  if (plan.splits > 1) {
    p.splits = plan.splits;
    p.split_steps = plan.split_steps;
    p.partial = (float*)((char*)workspace + gemm_workspace(p.M, p.N, p.K, 1));
    if (plan.tile.rows == 256) return launch_gemm_tiled<Act, FMT<Act, 64>, 256, 64, true, 4>(p, st);
    return launch_gemm_tiled<Act, FMT<Act, 128>, 128, 128, true>(p, st);
  }
  switch (plan.tile.rows << 16 | plan.tile.columns) {
    case 128 << 16 | 64: return launch_gemm_tiled<Act, FMT<Act, 64>, 128, 64, false, 4>(p, st);
    case 192 << 16 | 64: return launch_gemm_tiled<Act, FMT<Act, 64>, 192, 64, false, 4>(p, st);
    case 256 << 16 | 48: return launch_gemm_tiled<Act, FMT<Act, 48>, 256, 48, false, 4>(p, st);
    case 256 << 16 | 64: return launch_gemm_tiled<Act, FMT<Act, 64>, 256, 64, false, 4>(p, st);
    case 128 << 16 | 96: return launch_gemm_tiled<Act, FMT<Act, 96>, 128, 96>(p, st);
    case 128 << 16 | 128: return launch_gemm_tiled<Act, FMT<Act, 128>, 128, 128>(p, st);
    case 256 << 16 | 160: return launch_gemm_tiled<Act, FMT<Act, 160>, 256, 160>(p, st);
    case 256 << 16 | 192: return launch_gemm_tiled<Act, FMT<Act, 192>, 256, 192>(p, st);
    case 256 << 16 | 224: return launch_gemm_tiled<Act, FMT<Act, 224>, 256, 224>(p, st);
    default: return launch_gemm_tiled<Act, FMT<Act, 256>, 256, 256>(p, st);
  }
}

}  // namespace qlin
