// What the grouped GEMM kernels share: their parameters and the fp8 matrix instruction.
#pragma once
#include "common.hpp"

namespace aamd {

constexpr int kBK = 128;  // contraction bytes per step == scale block
constexpr int kLargeTile = 256;  // rows of an L and R tile of gemm_rows.hip

enum GemmMode { kRaggedRows = 0, kRaggedK = 1 };

typedef float v16f __attribute__((ext_vector_type(16)));

struct GemmParams {
  const uint8_t* L;
  const uint8_t* R;
  const float* Ls;
  const float* Rs;
  void* C;
  const void* bias;
  const int64_t* goff;      // [E+1] rows per group prefix (device); nullptr: one group [0, Lrows)
  int64_t ldl, ldr;                          // row strides of L and R (bytes)
  int64_t l_kb_stride, r_kb_stride;          // bytes between consecutive 128-wide contraction blocks of a row
  int64_t r_group_stride;                    // bytes between the R matrices of consecutive groups
  int64_t ls_row_stride, ls_blk_stride;      // L scale (row, block) strides, floats
  int64_t rs_row_stride, rs_blk_stride, rs_group_stride;
  int64_t ldc, c_group_stride;               // elements
  int64_t bias_group_stride;
  int64_t Lrows;   // kRaggedRows: total token rows; kRaggedK: rows of L (= N of dW)
  int64_t Rrows;   // rows of R per group
  int nkb;         // kRaggedRows: K / 128
  int E;
  int nRt;         // R tiles
  int nLt;         // kRaggedK: L tiles
  int max_kb;      // kRaggedK: contraction blocks the operand buffers hold (ld_t / 128)
  int accumulate;
  int group_r;     // the tile order groups R tiles (inside each group of rows / expert) instead of L tiles
  int bias_dtype;
  int gl;          // L tiles that share an R panel in the tile order
  int run;         // kRaggedK: tiles of short groups that a workgroup takes one after the other (0: none)
  int short_kb;    // kRaggedK: the most contraction blocks of a short group
  int zeroers;     // kRaggedK with runs: the most workgroups that write the gradients of groups without rows, ahead of the tiles' (0: none)
  int max_split;   // row_tiles_kernel: the most parts of a tile's contraction; more than one: ws holds kRowPartsBytes
  float* ws;
  int higher;      // row_tiles_kernel: tiles of up to 288 rows (1), of 256 (-1), or as the groups' rows have it (0)
  int slices;      // row_tiles_kernel with these: every XCD takes an eighth of every group
  int stream_out;  // row_tiles_kernel: the output is stored past the caches
  int ls_batch;    // kRaggedRows: L scales are fetched eight contraction blocks at a time
};

__device__ __forceinline__ v16f mfma_fp8_32x32x64(const v8i& a, const v8i& b, const v16f& c) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// Eight bytes of an 8 (rows) x 16 (bytes) block in the LDS, transposed: see grouped_gemm_kernel.
__device__ __forceinline__ v2i lds_read_transposed(uint32_t addr) {
  return __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)(uintptr_t)addr);
}

// A 64-bit offset the compiler can keep in scalar registers (it is the same in every lane).
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): a loop whose index is a constant
// expression inside the body.
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Row-ragged GEMM with block-scaled R for groups of few rows (gemm_few.hip); reads L, R, their scales and strides, C,
// bias, goff, E, Lrows, Rrows and nkb of the parameters.  r_rows: R is stored [contraction, Rrows] (R_ROWS of gemm.hip).
int launch_few_rows(const GemmParams& p, int c_dtype, int64_t M, int waves, bool r_rows, hipStream_t st);
// The same from bf16 rows, see aamd_quant_grouped_gemm_fp8_nt.
int launch_few_rows_quantising(const GemmParams& p, int what, const void* rows, int64_t ld, const int64_t* sorted_idx, int topk, int64_t T,
                               int64_t M, int waves, hipStream_t st);
// The same of permuted rows from the router's choices, see aamd_route_quant_grouped_gemm_fp8_nt: p.Lrows of them, at most 64.
int launch_few_rows_routing(const GemmParams& p, const void* ids, int ids_are_i64, const void* rows, int64_t ld, int topk, int64_t T,
                            int64_t* sorted_idx, int32_t* row_map, int64_t* goff, int waves, hipStream_t st);
// The second GEMM of a decoding step with the weighted combine in it, see aamd_quant_grouped_gemm_combine_fp8_nt: T tokens of topk slots.
int launch_few_rows_combine(GemmParams p, int what, const void* rows, int64_t ld, const void* ids, int ids_are_i64, const int32_t* row_map,
                            const void* probs, int probs_dtype, int topk, int64_t T, void* out, hipStream_t st);

// Are tiles of more rows worth it?  They save the tiles of remainders, which fetch their weights once more whatever few rows they have
// (us, 28672 outputs x 4096, 8 groups of 512 rows 430, 513 to 576 548 to 560, 640 595, 768 640), and cost every step something, more
// where addresses are made in the step.  In 256ths of a tile: 270 for one of theirs and 60 for 32 rows more in it, 176 and 185 for a
// remainder's own.  With few rounds a launch is as long as the workgroup whose tiles are all full, or all higher; and a round counts
// whole, but for a last one of few tiles, which is shared out.  Counts are of an R tile; n1: the tiles that the XCDs would have if all had
// as many as the one with the most.  All in whole numbers: the kernels of a launch have to come to the same.
// Fitted to 3000 launches of 1 to 64 groups of 240 to 1790 rows on average, 4096 to 32768 outputs and a contraction of 1024 to 14336.  Of 1800
// others it takes these for 446, 0.894 of the time, 19 of them 1 % slower or more, the worst 1.09 (4210 rows in 4, 10240 x 1024 65 -> 71);
// the lines that this replaces, without rounds past the third, for 506, 0.909, 59 and 1.18.  Of 300 without groups for 27, 0.863, the slowest
// 0.99.  Plain tiles -> these: 28672 x 4096 in 8 groups of about 512 523 -> 502, of 264 373 -> 302, of 520 558 -> 489; 4096 x 14336 in 8 of
// about 512 273 -> 251.  No longer taken: 2339 rows in 8, 16128 x 11392 555 -> 625; 2546 in 2, 9344 x 7680 185 -> 225; 6599 in 8, 4096 x
// 7424 200 -> 237.
__host__ __device__ inline uint32_t higher_tile_rounds(uint32_t n, uint32_t shared_out, bool parts) {  // in tiles
  const uint32_t left = n & 255u;
  return n - left + (left == 0 ? 0 : left > shared_out ? 256 : parts ? 92 + (164 * left >> 8) : 143 + (113 * left >> 8));
}
__host__ __device__ inline bool higher_tiles_pay(uint32_t full, uint32_t own0, uint32_t own1, uint32_t shared, uint32_t nRt, uint32_t n1, bool parts) {
  const uint32_t t0 = full + own0, t1 = full + own1, n0 = t0 * nRt;
  const uint32_t w0 = 256 * full + 176 * own0, w1 = 270 * full + 185 * own1 + 60 * shared;  // of an R tile, if all workgroups had the same
  const uint32_t d0 = 256 * t0 - w0, d1 = (shared > 0 ? 330 : 270) * t1 - w1;               // and what the longest has beyond
  const uint32_t l0 = w0 + (n0 <= 210 ? d0 : 210 * d0 / n0), l1 = w1 + (n1 <= 210 ? d1 : 210 * d1 / n1);
  const uint32_t r0 = higher_tile_rounds(n0, 128, parts), r1 = higher_tile_rounds(n1, parts ? 112 : 128, parts);
  return 32 * (uint64_t)r1 * l1 * t0 < 31 * (uint64_t)r0 * l0 * t1;
}

constexpr int64_t kRowPartsBytes = (int64_t)256 * kLargeTile * kLargeTile * 4;  // a tile of fp32 for each of 256 workgroups
// Row-ragged GEMM with block-scaled R on 256 x 256 tiles (gemm_rows.hip): at least eight contraction blocks, p.ls_batch 1 where
// rows of scales are 16-byte aligned; `tiles`: no fewer than there are.
int launch_row_tiles(GemmParams p, int c_dtype, int64_t tiles, bool r_rows, hipStream_t st);
// Weight gradient on 256 x 256 tiles (gemm_wgrad.hip): at most 64 groups, written and not added to.
int launch_wgrad_tiles(const GemmParams& p, int c_dtype, hipStream_t st);

}  // namespace aamd
