// Ragged grouped block-scaled FP8 GEMM for gfx950 (forward, dgrad, wgrad and the dense case).
//
// One kernel template covers the three GEMM families.  Both operands are "K-major" byte
// matrices (rows of fp8 codes along the contraction), called L and R here:
//
//   L = the operand whose row index ends up on the MFMA column / lane axis
//       (forward+dgrad: the token rows; wgrad: the rows of dY^T),
//   R = the operand whose row index ends up on the MFMA row / register axis
//       (forward+dgrad: the weight rows of the group's expert; wgrad: the rows of X^T).
//
// Output is C[l, r] with r contiguous, so the four consecutive MFMA rows a lane owns are four
// consecutive output elements.  The contraction advances in steps of 128 bytes = one scale
// block.  Per step and 32x32 sub-tile two chained v_mfma_f32_32x32x64_f8f6f4 give the raw
// 128-deep dot products, which are folded into the fp32 accumulator with the step's scales:
//   acc += p * (l_scale[l, kb] * r_scale)      r_scale per 128x128 block (one scalar) or per row.
// The per-lane l_scale sits in one VGPR because the L row is the lane axis.
//
// Why this shape of MFMA: measured on MI355X, VALU instructions co-execute with the 16-pass
// 32x32x64 MFMA (8 FMAs per MFMA cost ~4 %), but not with the 8-pass 16x16x128 one (there every
// FMA adds its full 4 cycles).  The fold needs 8 FMAs per MFMA, so only the former keeps the
// matrix pipe busy.
//
// Data path: global -> LDS directly (global_load_lds, 16 bytes per lane, no register stop),
// two stages, one workgroup barrier per step (two in the 256 x 256 configuration, whose L tile is
// requested two steps ahead; it serves row-ragged launches of one round of tiles, longer ones and weight
// gradients have kernels of their own, gemm_rows.hip and gemm_wgrad.hip).  Rows are 128 bytes; the 16-byte chunks of a row
// are XOR-swizzled so that the linear 1 KB writes of the direct loads and the 32-row MFMA
// operand reads are both bank-conflict free on the 64-bank LDS (measured: ~235 of 256 B/clk).
#include <algorithm>
#include <cmath>

#include "gemm.hpp"
#ifdef AAMD_TUNING
#include "../../include/atorch_amd_probes.h"
#endif

namespace aamd {

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// XOR swizzle of the 16-byte chunk index inside a 128-byte LDS row (depends on row % 16 only).
__device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

template <typename OUT>
__device__ __forceinline__ void store4(OUT* dst, v4f o, bool accumulate) {
  if constexpr (sizeof(OUT) == 4) {
    if (accumulate) o += *reinterpret_cast<const v4f*>(dst);
    *reinterpret_cast<v4f*>(dst) = o;
  } else {
    if (accumulate) {
      const v2i old = *reinterpret_cast<const v2i*>(dst);
      o[0] += bf16_bits_to_f32((uint32_t)old[0] & 0xffffu);
      o[1] += bf16_bits_to_f32((uint32_t)old[0] >> 16);
      o[2] += bf16_bits_to_f32((uint32_t)old[1] & 0xffffu);
      o[3] += bf16_bits_to_f32((uint32_t)old[1] >> 16);
    }
    v2i w;
    w[0] = (int)pack_bf16x2(o[0], o[1]);
    w[1] = (int)pack_bf16x2(o[2], o[3]);
    *reinterpret_cast<v2i*>(dst) = w;
  }
}

// Tile configuration: WR x WL waves, each computing (WTR*32) R rows x (WTL*32) L rows.
template <int WR_, int WL_, int WTR_, int WTL_, int PRB_ = 2, bool LAHEAD_ = false>
struct Cfg {
  static constexpr bool LAHEAD = LAHEAD_;  // load the L tile two steps ahead (extra barrier per step)
  static constexpr int WR = WR_, WL = WL_, WTR = WTR_, WTL = WTL_;
  static constexpr int PRB = PRB_;  // raw-product buffers: 2 folds a sub-tile under the next one's MFMAs
  static constexpr int NT = 64 * WR * WL;   // threads
  static constexpr int BM = WL * WTL * 32;  // L rows per workgroup tile
  static constexpr int BN = WR * WTR * 32;  // R rows per workgroup tile
  static constexpr int LCH = BM * 8 / NT;   // 16-byte chunks per thread and step (L)
  static constexpr int RCH = BN * 8 / NT;
  static_assert(NT >= BM + BN, "one thread per scale value");
  static_assert(BM % 64 == 0 && BN % 128 == 0, "whole waves per scale side; R tiles cover whole scale blocks");
  static_assert((WTR * 32) % 128 == 0 || BN == 128, "a wave's R rows stay inside one 128-row scale block");
  static_assert(LCH * NT == BM * 8 && RCH * NT == BN * 8, "tile rows divide evenly over the threads");
  static_assert((NT / 8) % 16 == 0, "the swizzle of a slab depends on the wave only");
};
typedef Cfg<2, 2, 2, 2, 3> CfgSmall;  // 256 threads, 128 (L) x 128 (R), two workgroups per CU
typedef Cfg<2, 4, 4, 2, 1, true> CfgLarge;  // 512 threads, 256 (L) x 256 (R); one product buffer: 256 registers per lane
typedef Cfg<2, 4, 2, 2> CfgWgrad;  // 512 threads, 256 (L) x 128 (R): room for the per-row R scales

// ---- weight gradient of short groups -----------------------------------------------------------
// A tile of a group of few rows is over after one or two 128-deep steps, and what it costs in grouped_gemm_kernel is the
// workgroup's turnover: launch, group lookup, first loads and the stores follow each other, with two workgroups per CU to
// hide one behind the other.  Here a workgroup takes `run` consecutive 128 x 128 tiles of the groups in `mask` (a row of
// tiles of the output after the other) and the loads of the next step, which may be the next tile's, are in flight under
// the step and the stores before it.  The arithmetic and its order are those of grouped_gemm_kernel: the same bits.
// What bounds it is the stream of gradients written (and read, where they accumulate).
//
// LDS: two stages of 32 KB, [L rows | R rows], and their scales; the output of a tile is staged in the stage it was
// computed from, 8 KB per wave, rows of 128 bytes with their 16-byte chunks XORed with three bits of the row.
struct ShortTiles {
  unsigned long long mask;  // groups
  int total;                // their tiles
  GroupRanges gr;           // lane e: the contraction blocks of group e
};

template <typename OUT, bool ACC>
__device__ __forceinline__ void wgrad_short_tiles(const GemmParams& p, uint8_t* lds, float* Sc, const ShortTiles& st, int unit) {
  constexpr int kStage = 2 * kTile * kBK;
  constexpr int WT = 2;  // 2 x 2 waves of 2 x 2 sub-tiles
  typedef typename std::conditional<ACC, float, OUT>::type ST;  // staging: float where the old output is added
  constexpr int CW = 128 / (int)sizeof(ST), SUBS = CW / 32, VL = 16 / (int)sizeof(ST);
  // vector memory instructions of a thread's stores of a tile, at least: what may stay in flight when the loads issued
  // before them have to have landed
  constexpr int kStores = 8 * (WT / SUBS);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hg = lane >> 5;
  const int wr = wave >> 1, wl = wave & 1;
  const int per_g = p.nLt * p.nRt;
  int left = st.total - unit * p.run;  // tiles from the first of this unit to the end of the list
  if (left <= 0) return;
  if (left > p.run) left = p.run;

  // ---- the tile under way: group, tile row and column, contraction blocks
  struct Tile {
    int g, lt, rt, kb, n;
    bool nan;
    unsigned long long rest;  // groups of the list behind g
  };
  auto enter = [&](Tile& t) {
    t.kb = __builtin_amdgcn_readlane(st.gr.t_lo, t.g);
    const int hi = __builtin_amdgcn_readlane(st.gr.t_hi, t.g);
    t.nan = hi > p.max_kb;  // operand buffers too short: never read past them, and make the failure visible
    t.n = t.nan ? 0 : hi - t.kb;
  };
  auto next_group = [&](Tile& t) {
    t.g = __builtin_ctzll(t.rest);
    t.rest &= t.rest - 1;
    enter(t);
  };
  Tile cur;
  {
    int turn = unit * p.run / per_g;
    const int pos = unit * p.run - turn * per_g;
    cur.rest = st.mask;
    for (; turn > 0; turn--) cur.rest &= cur.rest - 1;
    next_group(cur);
    cur.lt = pos / p.nRt;
    cur.rt = pos - cur.lt * p.nRt;
  }
  auto advance = [&](Tile& t) {
    if (++t.rt < p.nRt) return;
    t.rt = 0;
    if (++t.lt < p.nLt) return;
    t.lt = 0;
    next_group(t);
  };

  // ---- loads: the slabs and swizzle of grouped_gemm_kernel (rows and columns of the output are whole tiles here)
  auto lds_addr = [](const void* q) { return (uint32_t)(uintptr_t)(lds_ptr_t)q; };
  const int r8 = lane >> 3;
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ r8 ^ (wave & 1)) << 4);
  const uint32_t voffL = (uint32_t)r8 * (uint32_t)p.ldl + chunk, voffR = (uint32_t)r8 * (uint32_t)p.ldr + chunk;
  const uint32_t soff = (uint32_t)(tid & (kTile - 1)) * 4u;
  auto load = [&](const Tile& t, int k, int s) {
    const int64_t kb = t.kb + k;
    const uint8_t* L = p.L + uniform_i64((int64_t)t.lt * kTile * p.ldl + kb * p.l_kb_stride);
    const uint8_t* R = p.R + uniform_i64((int64_t)t.rt * kTile * p.ldr + kb * p.r_kb_stride);
#pragma unroll
    for (int n = 0; n < 4; n++) {
      const int row = wave * 8 + 32 * n;
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voffL),
                   "s"(L + (uint32_t)row * (uint32_t)p.ldl), "s"(lds_addr(lds) + (uint32_t)(s * kStage + row * kBK))
                   : "memory");
    }
#pragma unroll
    for (int n = 0; n < 4; n++) {
      const int row = wave * 8 + 32 * n;
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voffR),
                   "s"(R + (uint32_t)row * (uint32_t)p.ldr), "s"(lds_addr(lds) + (uint32_t)(s * kStage + (kTile + row) * kBK))
                   : "memory");
    }
    // waves 0 and 1: the scales of the L rows, 2 and 3: of the R rows
    const float* sb = wave < 2 ? p.Ls + (kb * p.ls_blk_stride + t.lt * kTile) : p.Rs + (kb * p.rs_blk_stride + t.rt * kTile);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(soff), "s"(sb),
                 "s"(lds_addr(Sc) + (uint32_t)(s * 1024 + wave * 256))
                 : "memory");
  };

  v16f acc[WT][WT], zero;
#pragma unroll
  for (int r = 0; r < 16; r++) zero[r] = 0.f;
  auto clear = [&](const Tile& t) {
    const float v = t.nan ? __builtin_nanf("") : 0.f;
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
      for (int j = 0; j < WT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = v;
  };
  const int sw = swz(l32);
  auto compute = [&](int s) {
    const uint8_t* const Lt = lds + s * kStage + (wl * 64 + l32) * kBK;
    const uint8_t* const Rt = lds + s * kStage + (kTile + wr * 64 + l32) * kBK;
    const float* const S = Sc + s * 256;
    auto frag = [&](const uint8_t* row, int h) {
      const v4i lo = *reinterpret_cast<const v4i*>(row + (((4 * h + 2 * hg) ^ sw) << 4));
      const v4i hi = *reinterpret_cast<const v4i*>(row + (((4 * h + 2 * hg + 1) ^ sw) << 4));
      return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    v8i lf[WT][2], rf[WT][2];
    float cs[WT];
#pragma unroll
    for (int j = 0; j < WT; j++) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        lf[j][h] = frag(Lt + j * 32 * kBK, h);
        rf[j][h] = frag(Rt + j * 32 * kBK, h);
      }
      cs[j] = S[wl * 64 + j * 32 + l32];
    }
#pragma unroll
    for (int i = 0; i < WT; i++) {
      v4f rs[4];
#pragma unroll
      for (int q = 0; q < 4; q++) rs[q] = *reinterpret_cast<const v4f*>(&S[kTile + wr * 64 + i * 32 + 8 * q + 4 * hg]);
#pragma unroll
      for (int j = 0; j < WT; j++) {
        v16f pr = mfma_fp8_32x32x64(rf[i][0], lf[j][0], zero);
        pr = mfma_fp8_32x32x64(rf[i][1], lf[j][1], pr);
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = __builtin_fmaf(pr[r], cs[j] * rs[r / 4][r % 4], acc[i][j][r]);
      }
    }
  };
  auto store = [&](const Tile& t, int s) {
    uint8_t* const stg = lds + s * kStage + wave * (64 * 128);
    OUT* const Cg = reinterpret_cast<OUT*>(p.C) + (int64_t)t.g * p.c_group_stride;
#pragma unroll
    for (int ci = 0; ci < WT / SUBS; ci++) {
#pragma unroll
      for (int si = 0; si < SUBS; si++)
#pragma unroll
        for (int j = 0; j < WT; j++)
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const v16f& a = acc[ci * SUBS + si][j];
            const v4f o = v4f{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
            const int row = j * 32 + l32, byte = (si * 32 + 8 * q + 4 * hg) * (int)sizeof(ST);
            uint8_t* const dst = stg + row * 128 + (((byte >> 4) ^ ((row >> 1) & 7)) << 4) + (byte & 15);
            if constexpr (sizeof(ST) == 4) *reinterpret_cast<v4f*>(dst) = o;
            else *reinterpret_cast<v2i*>(dst) = v2i{(int)pack_bf16x2(o[0], o[1]), (int)pack_bf16x2(o[2], o[3])};
          }
      __builtin_amdgcn_wave_barrier();  // same wave, in-order LDS: the reads below see the writes above
      OUT* const out0 = Cg + ((int64_t)t.lt * kTile + wl * 64 + r8) * p.ldc + (t.rt * kTile + wr * 64 + ci * CW + (lane & 7) * VL);
      v4i raws[8];
#pragma unroll
      for (int ps = 0; ps < 8; ps++) {
        const int row = ps * 8 + r8;
        raws[ps] = *reinterpret_cast<const v4i*>(stg + row * 128 + (((lane & 7) ^ ((row >> 1) & 7)) << 4));
      }
      if constexpr (ACC && sizeof(OUT) == 4) {
#pragma unroll
        for (int half = 0; half < 8; half += 4) {
          v4f olds[4];
#pragma unroll
          for (int ps = 0; ps < 4; ps++) olds[ps] = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(out0 + (half + ps) * 8 * p.ldc));
#pragma unroll
          for (int ps = 0; ps < 4; ps++) {
            const v4f o = __builtin_bit_cast(v4f, raws[half + ps]) + olds[ps];
            __builtin_nontemporal_store(o, reinterpret_cast<v4f*>(out0 + (half + ps) * 8 * p.ldc));
          }
        }
      } else {
#pragma unroll
        for (int ps = 0; ps < 8; ps++) {
          if constexpr (sizeof(ST) == sizeof(OUT)) __builtin_nontemporal_store(raws[ps], reinterpret_cast<v4i*>(out0 + ps * 8 * p.ldc));
          else store4<OUT>(out0 + ps * 8 * p.ldc, __builtin_bit_cast(v4f, raws[ps]), true);
        }
      }
      __builtin_amdgcn_wave_barrier();  // the next chunk overwrites the region
    }
  };

  if (cur.n > 0) load(cur, 0, 0);
  clear(cur);
  bool stored = false;
  for (int k = 0, s = 0;; s ^= 1) {
    const bool last = k + 1 >= cur.n;  // (a tile without a contraction is one empty step)
    const bool more = !last || left > 1;
    Tile nxt = cur;
    int kn = k + 1;
    if (last) {
      kn = 0;
      if (left > 1) advance(nxt);
    }
    // this step's loads have landed and every wave is done with the other stage (loads and stores are counted in order,
    // and the stores of the tile before were issued behind these loads)
    if (stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kStores) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (more && nxt.n > 0) load(nxt, kn, s ^ 1);
    if (cur.n > 0) compute(s);
    stored = last;
    if (last) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave has read the stage
      store(cur, s);
      if (--left == 0) return;
      clear(nxt);
    }
    cur = nxt;
    k = kn;
  }
}

// Gradients of groups without rows that are written and not added to are zeros, a stream of stores that leaves the matrix cores alone.
// As tiles like the others they come at the end, at 3.7 TB/s; here the launch's first workgroups write them beside the tiles of the
// others, at up to 5.  How many, 0 where it does not pay: each takes half a CU from the tiles, and what one workgroup computes, a long
// contraction or a run of short ones, takes longer beside one.  So most groups have to be without rows, and their zeros a stream that
// outlasts that (7 MB a block); more of them where there is much to compute besides.  us, as tiles -> by 48 / 64 / 96 / 128 workgroups:
//   60 groups, 16001 rows (108 blocks and less), 2816 x 2048 fp32     325 -> 301 / 257 / 275 / 261    zeros 1223 MB
//   64 groups, 8192 rows (56 blocks and less), 2048 x 7168 bf16       457 -> 399 / 377 / 361 / 359    1644 MB
//   64 groups, 189 rows (2 blocks), 2816 x 2432 fp32                  337 -> 468 (32) / 256 / 300 / 305    1698 MB
//   60 groups, 467 rows (4 blocks), 2688 x 1024 bf16                  86 -> 86 (32) / 49 / 56 / 58    314 MB
//   not: 32 groups, 12000 rows (81 blocks), 3072 x 1024 fp32          84 -> 104 / 99 / 104 / 109    315 MB
//   60 groups, 39191 rows (173 blocks), 640 x 3840 fp32               189 -> 193 (32) / 224 / 240 / 216    187 MB
// Of 683 drawn launches with two thirds of the groups without rows (4 to 64 of 512 x 512 to 7168 x 7168, 64 to 46000 rows) the rule takes
// 443: 0.83 of the time as tiles, two of them 3 and 4 % slower.  With 96 workgroups always, launches were up to 30 % slower.
constexpr int kZeroers = 96, kZeroersOfShort = 64;  // (multiples of 8)
template <typename OUT>
__device__ __forceinline__ int zeroers_of(const GemmParams& p, unsigned long long empty, int n, int steps) {
  const int groups = __popcll(empty);
  const int64_t bytes = (int64_t)groups * p.Lrows * p.ldc * (int64_t)sizeof(OUT);
  const int chain = n <= p.short_kb ? n * p.run : n;
  if (3 * groups < 2 * p.E || __ballot((int64_t)chain * 7000000 > bytes) != 0) return 0;
  return bytes >= 400000000 && steps >= 30 * 512 ? kZeroers : kZeroersOfShort;
}
// Workgroup `part` of `parts` writes its share.
template <typename OUT>
__device__ __forceinline__ void zero_groups(const GemmParams& p, unsigned long long mask, int part, int parts) {
  const int64_t bytes = p.Lrows * p.ldc * (int64_t)sizeof(OUT);
  for (; mask != 0; mask &= mask - 1) {
    uint8_t* const out = reinterpret_cast<uint8_t*>(reinterpret_cast<OUT*>(p.C) + (int64_t)__builtin_ctzll(mask) * p.c_group_stride);
    for (int64_t at = ((int64_t)part * blockDim.x + threadIdx.x) * 16; at < bytes; at += (int64_t)parts * blockDim.x * 16)
      __builtin_nontemporal_store(v4i{0, 0, 0, 0}, reinterpret_cast<v4i*>(out + at));
  }
}

// R_ROWS: the R operand as it is stored where its contraction runs down the rows, [contraction, Rrows] (the codes of a
// weight read for the product with its transpose: one scale per 128x128 block, so that the codes are the same bytes in
// either orientation).  A step's R tile is then 128 rows of BN bytes, and the fragments are read with
// ds_read_b64_tr_b8: of every 16 lanes, lanes 2r and 2r + 1 name the halves of 16 bytes of row r, and lane l receives
// byte l of the eight rows.  The 16-byte chunks of a row are XORed with twice the low bits of its place among the rows
// that share the 64 banks, so that the 32 lanes of a read phase (two chunks of eight rows) meet no bank twice (measured: 2.0
// clocks per instruction and CU with eight waves, as ds_read_b64 of consecutive bytes; 12 without the XOR).
template <int MODE, bool R_PER_ROW, typename OUT, typename C, bool R_ROWS>
__global__ __launch_bounds__(C::NT, C::NT == 256 ? 2 : 1) void grouped_gemm_kernel(const GemmParams p) {
  constexpr int BM = C::BM, BN = C::BN, NT = C::NT;
  // LDS: two stages of an L tile and an R tile of 128-byte rows, then the two stages' scales
  // ([L rows | R rows or R blocks | unused], NT floats each).  After the contraction loop the same
  // memory stages the output tile for the row-contiguous stores of the epilogue.
  constexpr int kStage = (BM + BN) * kBK;
  constexpr int kStgBytes = 64 * 144;  // per-wave epilogue staging: 64 rows x (128 + 16) bytes
  static_assert(2 * kStage >= (NT / 64) * kStgBytes, "the epilogue staging fits in the stage buffers");
  // kRaggedRows keeps two batches of L scales besides: [BM rows][8 contraction blocks] floats each.
  constexpr int kLsBatch = MODE == kRaggedRows ? BM * 8 * 4 : 0;
  static_assert(NT == 2 * BM, "two threads fetch the 32 bytes of a row's scale batch");
  static_assert(!R_ROWS || (MODE == kRaggedRows && !R_PER_ROW), "one scale per row along the contraction has one orientation");
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * kStage + 2 * NT * 4 + 2 * kLsBatch];
  // both L stages first, then both R stages: every fragment of a side is within 64 KB of one base
  // address, so the stage and the sub-tile row go into the immediate offset of the LDS reads
  uint8_t* const Lbuf0 = lds;
  uint8_t* const Lbuf1 = lds + BM * kBK;
  uint8_t* const Rbuf0 = lds + 2 * BM * kBK;
  uint8_t* const Rbuf1 = lds + 2 * BM * kBK + BN * kBK;
  static_assert(2 * BM * kBK <= 65536 && 2 * BN * kBK <= 65536, "immediate LDS offsets are 16 bits");
  float* const Sc0 = reinterpret_cast<float*>(lds + 2 * kStage);
  float* const Sc1 = Sc0 + NT;
  float* const LsB0 = Sc1 + NT;  // scale batches (kRaggedRows)

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, lives in an SGPR
  const int lane = tid & 63;

  // ---- which tile -------------------------------------------------------------------------
  // One tile per workgroup (a loop over tiles inside the kernel costs registers and the
  // hardware's own dispatch balances ragged tiles better).  Workgroup ids go round-robin over
  // the 8 XCDs; every XCD gets one contiguous range of tile ids so that tiles sharing operand
  // panels meet in the same L2.
  // Row-ragged launches look their group up in the device-side offsets.  Every wave does it on its
  // own, without LDS or barriers: lane e computes the tile range of group e (group_ranges), the lane whose group
  // holds the tile is found with a ballot and its values are broadcast with readlane.
  int total_lt;
  GroupRanges gr = {};
  if (MODE == kRaggedRows && p.goff != nullptr) {
    gr = group_ranges<BM>(p.goff, p.E, 0, 0);
    total_lt = gr.total;
    for (int base = 64; base < p.E; base += 64) total_lt = group_ranges<BM>(p.goff, p.E, base, total_lt).total;
  } else {
    total_lt = (int)((p.Lrows + BM - 1) / BM);  // kRaggedRows without groups
  }
  const int64_t bid = blockIdx.x;
  const int64_t xcd = bid % 8, idx = bid / 8;
  const int GL = p.gl;
  int g, lt, rt;
  int kb_lo = 0, kb_hi = 0;  // kRaggedK: the contraction blocks of group g
  int64_t pid = 0;
  bool by_group = false;
  if constexpr (MODE == kRaggedK) {
    // The length of the contraction, and with it the time of a tile, differs from group to group, so every XCD takes
    // an eighth of the tiles of every group (one range of tiles over all groups left the XCD that owned the busiest
    // groups working alone: 16001 rows Zipf-distributed over 60 groups, 2816 x 2048 fp32 outputs, 800 us against 295 us), and
    // the groups that are longer than average go first, so that the launch ends on short tiles.
    const int per_g = p.nLt * p.nRt;  // tiles of a group
    const int per_x = (per_g + 7) >> 3;
    int turn = __builtin_amdgcn_readfirstlane((int)((uint32_t)idx / (uint32_t)per_x));
    int pos = (int)idx - turn * per_x;
    g = turn;
    if (turn >= p.E && p.run == 0) return;
    if (p.goff == nullptr) {  // one group over the whole contraction
      kb_hi = p.max_kb;
    } else if (p.E <= 64) {
      gr = group_ranges<kBK>(p.goff, p.E, 0, 0);
      const int n = gr.t_hi - gr.t_lo;
      bool live = lane < p.E;
      if constexpr (NT == 256) if (p.run > 0) {
        // the groups of few blocks leave the list of this loop: behind the long groups' tiles a workgroup takes a run of
        // theirs (and of the groups that the operand buffers do not hold, which are written as NaN)
        const bool empty = live && n == 0 && gr.t_hi <= p.max_kb;
        const int zeroers = p.zeroers > 0 ? zeroers_of<OUT>(p, __ballot(empty), live ? n : 0, gr.total * per_g) : 0;
        int from = (int)idx;  // this workgroup's place among those that have tiles
        if (zeroers > 0) {
          if (bid < zeroers) {
            zero_groups<OUT>(p, __ballot(empty), (int)bid, zeroers);
            return;
          }
          from -= zeroers / 8;
          turn = __builtin_amdgcn_readfirstlane((int)((uint32_t)from / (uint32_t)per_x));
          pos = from - turn * per_x;
        }
        const bool none = empty && (p.accumulate || zeroers > 0);  // nothing to add, or zeros that are being written
        const bool few = live && !none && (gr.t_hi > p.max_kb || n <= p.short_kb);
        live = live && !few && !none;
        const int nlong = __popcll(__ballot(live));
        if (turn >= nlong) {
          ShortTiles st;
          st.mask = __ballot(few);
          st.total = __popcll(st.mask) * per_g;
          st.gr = gr;
          const int unit = (from - nlong * per_x) * 8 + (int)xcd;
          if (p.accumulate) wgrad_short_tiles<OUT, true>(p, lds, Sc0, st, unit);
          else wgrad_short_tiles<OUT, false>(p, lds, Sc0, st, unit);
          return;
        }
      }
      const unsigned long long big = __ballot(live && (int64_t)n * p.E > 2 * (int64_t)gr.total);
      const unsigned long long mid = __ballot(live && (int64_t)n * p.E > (int64_t)gr.total) & ~big;
      const unsigned long long low = __ballot(live) & ~(big | mid);
      // this lane's group is the r-th of the order: all of `big`, then all of `mid`, then the rest
      const unsigned long long below = (1ull << lane) - 1ull;
      const int nbig = __popcll(big), nmid = __popcll(mid);
      const int r = (big >> lane) & 1 ? __popcll(big & below)
                    : (mid >> lane) & 1 ? nbig + __popcll(mid & below) : nbig + nmid + __popcll(low & below);
      g = __builtin_ctzll(__ballot(live && r == turn));
      kb_lo = __builtin_amdgcn_readlane(gr.t_lo, g);
      kb_hi = __builtin_amdgcn_readlane(gr.t_hi, g);
    } else {
      for (int base = 0, carry = 0; base < p.E; base += 64) {
        gr = group_ranges<kBK>(p.goff, p.E, base, carry);
        if (g - base < 64) {
          kb_lo = __builtin_amdgcn_readlane(gr.t_lo, g - base);
          kb_hi = __builtin_amdgcn_readlane(gr.t_hi, g - base);
          break;
        }
        carry = gr.total;
      }
    }
    // this XCD's eighth; which one rotates with the group, so that remainders spread over the XCDs
    const int part = (int)(xcd + turn) & 7, size = per_g >> 3, rem = per_g & 7;
    if (pos >= size + (part < rem ? 1 : 0)) return;
    const int pe = part * size + (part < rem ? part : rem) + pos;
    // groups of GL tiles of the longer side of the gradient, all tiles of the shorter one inside
    if (p.group_r) {
      const int width = GL * p.nLt, first = pe / width * GL, in_grp = pe % width;
      const int gsz = p.nRt - first < GL ? p.nRt - first : GL;
      rt = first + in_grp % gsz;
      lt = in_grp / gsz;
    } else {
      const int width = GL * p.nRt, first = pe / width * GL, in_grp = pe % width;
      const int gsz = p.nLt - first < GL ? p.nLt - first : GL;
      lt = first + in_grp % gsz;
      rt = in_grp / gsz;
    }
  } else {
    const int64_t ntot = (int64_t)total_lt * p.nRt;
    if (bid >= ntot) return;
    const int64_t per = ntot / 8, rem = ntot % 8;
    pid = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
    by_group = p.goff != nullptr && p.group_r;  // tile order per group, below
    // inside the range: groups of GL L tiles, R tile index outer, L tile inner
    const int64_t width = (int64_t)GL * p.nRt;
    const int first = (int)(pid / width) * GL;
    const int gsz = total_lt - first < GL ? total_lt - first : GL;
    const int in_grp = (int)(pid % width);
    lt = first + in_grp % gsz;
    rt = in_grp / gsz;
  }

  int64_t l0;     // first L row of the tile
  int lvalid;     // valid L rows in the tile
  int kb0, nkb;   // contraction blocks [kb0, kb0 + nkb)
  bool short_operands = false;
  if constexpr (MODE == kRaggedRows) {
    if (p.goff) {
      // exactly one group holds tile lt (empty groups hold none)
      // With group_r the tile ids of a group are contiguous and ordered in batches of GL R tiles,
      // all L tiles of the group inside a batch, R index fastest: the weights of the group, the
      // large operand, are then fetched once, and the group's few L panels are what gets re-read.
      g = p.E;
      l0 = 0;
      lvalid = 0;
      for (int base = 0; base < p.E; base += 64) {
        if (base > 0) gr = group_ranges<BM>(p.goff, p.E, base, gr.total);  // more than 64 groups: the next 64
        const int t_lo = gr.t_lo, t_hi = gr.t_hi;
        int my_lt = lt, my_rt = 0;
        bool mine = lt >= t_lo && lt < t_hi;  // empty groups (and lanes past E) hold no tile
        if (by_group) {
          const int64_t p_lo = (int64_t)t_lo * p.nRt, p_hi = (int64_t)t_hi * p.nRt;
          mine = pid >= p_lo && pid < p_hi;
          const int nl = mine ? t_hi - t_lo : 1;
          const int64_t pe = pid - p_lo, width = (int64_t)GL * nl;
          const int first_r = (int)(pe / width) * GL;
          const int gsz = p.nRt - first_r < GL ? p.nRt - first_r : GL;
          const int in_grp = (int)(pe % width);
          my_rt = first_r + in_grp % (gsz > 0 ? gsz : 1);
          my_lt = t_lo + in_grp / (gsz > 0 ? gsz : 1);
        }
        const unsigned long long hit = __ballot(mine);
        if (hit != 0) {  // exactly one group holds the tile
          const int src = __builtin_ctzll(hit);
          const int64_t first = gr.r_lo + (int64_t)(my_lt - t_lo) * BM, left = gr.r_hi - first;
          const int lv = left < BM ? (int)left : BM;
          g = base + src;
          l0 = readlane_i64(first, src);
          lvalid = __builtin_amdgcn_readlane(lv, src);
          if (by_group) rt = __builtin_amdgcn_readlane(my_rt, src);
          break;
        }
      }
      if (g >= p.E) return;
    } else {
      g = 0;
      l0 = (int64_t)lt * BM;
      const int64_t left = p.Lrows - l0;
      lvalid = left < BM ? (int)left : BM;
    }
    kb0 = 0;
    nkb = p.nkb;
  } else {
    l0 = (int64_t)__builtin_amdgcn_readfirstlane(lt) * BM;
    const int64_t left = p.Lrows - l0;
    lvalid = left < BM ? (int)left : BM;
    kb0 = kb_lo;
    nkb = kb_hi - kb_lo;
    kb0 = __builtin_amdgcn_readfirstlane(kb0);
    // Operand buffers too short for the padded token count (ld_t below the device-side total): never
    // read past them, and make the failure visible: the group's gradient tile is written as NaN.
    if (kb0 + nkb > p.max_kb) {
      nkb = 0;
      short_operands = true;
    }
    nkb = __builtin_amdgcn_readfirstlane(nkb);
  }
  g = __builtin_amdgcn_readfirstlane(g);
  rt = __builtin_amdgcn_readfirstlane(rt);
  const int64_t r0 = (int64_t)rt * BN;
  const int64_t rleft = p.Rrows - r0;
  const int rvalid = rleft < BN ? (int)rleft : BN;  // a multiple of 128

  // uniform tile bases + per-thread 32-bit offsets
  const uint8_t* Lbase = p.L + uniform_i64(l0 * p.ldl + (int64_t)kb0 * p.l_kb_stride);
  const uint8_t* Rbase = p.R + uniform_i64((int64_t)g * p.r_group_stride + (R_ROWS ? r0 : r0 * p.ldr) + (int64_t)kb0 * p.r_kb_stride);
  const float* Lsg = p.Ls + (int64_t)kb0 * p.ls_blk_stride;
  const float* Rsg = p.Rs + (int64_t)g * p.rs_group_stride + (int64_t)kb0 * p.rs_blk_stride;

  // ---- global -> LDS without a register stop ---------------------------------------------------
  // One wave instruction of the direct load writes 1 KB of LDS, lane l at base + 16 l: eight
  // tile rows of 128 bytes.  Lane l owns LDS position (row l/8, chunk l%8) and fetches the
  // global chunk the swizzle assigns to that position.
  // A wave instruction n covers the 8-row slab starting at tile row wave*8 + (NT/8)*n.  The lane
  // part of the address (row inside the slab, swizzled chunk) is the same for every slab of a
  // wave: (row & 7) is lane/8 and ((row >> 3) & 1) is wave & 1 because NT/8 is a multiple of 16.
  // The slab part is wave-uniform and lives in scalar registers.  Rows past the valid part of a
  // tile are never stored, so they may read whatever follows them in the operand; only the end
  // of the operand itself must not be crossed: slabs beyond the last readable row are moved onto
  // the last slab that holds one, and that slab clamps its rows per lane.
  const int r8 = lane >> 3;
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ r8 ^ (wave & 1)) << 4);
  const int64_t l_rows_left = p.Lrows - l0;
  const int availL = l_rows_left < BM ? (int)l_rows_left : BM;  // >= 1
  const int bmaxL = ((availL - 1) >> 3) << 3, tailL = availL - bmaxL;
  const uint32_t voffL = (uint32_t)r8 * (uint32_t)p.ldl + chunk;
  const uint32_t voffLt = (uint32_t)(r8 < tailL ? r8 : tailL - 1) * (uint32_t)p.ldl + chunk;
  // rvalid is a multiple of 128: whole slabs
  uint32_t voffR = (uint32_t)r8 * (uint32_t)p.ldr + chunk;
  if constexpr (R_ROWS) {
    // 1 KB = 1024 / BN rows of the tile; columns past the valid ones re-read valid ones of the same row
    constexpr int kChunks = BN / 16;
    const int row = ((wave * 1024) / BN + lane / kChunks) & 7;
    const int ch = ((lane % kChunks) ^ (2 * (row / (256 / BN)))) & (rvalid / 16 - 1);
    static_assert((BN == 256 || BN == 128) && (NT * 16 / BN) % 8 == 0, "the swizzle of a slab depends on the wave only");
    voffR = (uint32_t)(lane / kChunks) * (uint32_t)p.ldr + (uint32_t)ch * 16u;
  }
  uint32_t lslab[C::LCH], rslab[C::RCH];  // scalar byte offsets of the slabs
  bool ltail[C::LCH];
#pragma unroll
  for (int n = 0; n < C::LCH; n++) {
    const int b = wave * 8 + (NT / 8) * n;
    ltail[n] = b >= bmaxL;
    lslab[n] = __builtin_amdgcn_readfirstlane((uint32_t)(ltail[n] ? bmaxL : b) * (uint32_t)p.ldl);
  }
#pragma unroll
  for (int n = 0; n < C::RCH; n++) {
    const int b = wave * 8 + (NT / 8) * n;
    rslab[n] = __builtin_amdgcn_readfirstlane((uint32_t)(R_ROWS ? b * kBK / BN : b < rvalid ? b : rvalid - 8) * (uint32_t)p.ldr);
  }
  // scales: thread t < BM fetches the L scale of row t; thread BM + t the R scale of row t
  // (per-row scales) or of 128-row block t (block scales); the rest re-read a valid value.
  // Whole waves are on one side (BM is a multiple of 64), so base and step are wave-uniform.
  const bool l_side = wave < BM / 64;
  const float* sbase = l_side ? Lsg + l0 * p.ls_row_stride : Rsg + (R_PER_ROW ? r0 : r0 / kTile) * p.rs_row_stride;
  const int64_t s_step = l_side ? p.ls_blk_stride : p.rs_blk_stride;
  uint32_t soff;  // element offset of this thread's scale from sbase
  if (l_side) {
    const int lrow = tid < lvalid ? tid : lvalid - 1;
    soff = (uint32_t)lrow * (uint32_t)p.ls_row_stride;
  } else {
    const int t = tid - BM;
    const int nvalid = R_PER_ROW ? rvalid : rvalid / kTile;
    const int rr = t < nvalid ? t : nvalid - 1;
    soff = (uint32_t)rr * (uint32_t)p.rs_row_stride;
  }

  // All loads of the contraction loop are issued from inline assembly, with the wait counts kept
  // by hand: the compiler's own bookkeeping of direct-to-LDS loads is conservative (it tracks
  // eight of them individually and otherwise waits for every outstanding load).  Per step and
  // thread: LCH + RCH 16-byte tile loads and the scale loads; all of them write LDS only,
  // so no VGPR is ever written behind the compiler's back.
  auto lds_addr = [](const void* q) { return (uint32_t)(uintptr_t)(lds_ptr_t)q; };
  const uint32_t soff_b = soff * 4u;
  // L scales of a row-major [rows, K/128] operand: one 4-byte value per row and step would touch
  // as many cache lines as the tile itself.  Instead 32 bytes per row (eight contraction blocks)
  // are fetched every eighth step, 16 bytes per thread, into [row][8] floats.  The last batch is
  // shifted back so that it ends at the last block.
  const bool batch = MODE == kRaggedRows && p.ls_batch != 0;  // uniform; implies nkb >= 8
  // this wave loads a scale every step (never in the configuration that takes all its scales in batches)
  const bool step_scale = !C::LAHEAD && !(batch && l_side);
  const int brow = (tid >> 1) < lvalid ? (tid >> 1) : lvalid - 1;
  const uint32_t boff = ((uint32_t)brow * (uint32_t)p.ls_row_stride + (uint32_t)(tid & 1) * 4u) * 4u;
  auto batch_start = [&](int b) { return 8 * b + 8 <= nkb ? 8 * b : nkb - 8; };
  auto dma_scale_batch = [&](int b) {
    if constexpr (MODE == kRaggedRows) {
      const uint8_t* sb = reinterpret_cast<const uint8_t*>(Lsg + uniform_i64(l0 * p.ls_row_stride + batch_start(b)));
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   ::"v"(boff), "s"(sb), "s"(lds_addr(LsB0 + (b & 1) * (BM * 8)) + (uint32_t)(wave * 1024))
                   : "memory");
    }
  };
  auto dma_scale = [&](int kb, float* Sd) {
    const uint8_t* sb = reinterpret_cast<const uint8_t*>(sbase + (int64_t)kb * s_step);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                   ::"v"(soff_b), "s"(sb), "s"(lds_addr(Sd) + (uint32_t)(wave * 256))
                   : "memory");
  };
  // One wave instruction of the L (R) tile of a step; the last one of a half also carries that
  // half's scale loads.  L half: the L tile and, from the waves that own them, the L scales.
  auto dmaL_tile = [&](int n, int kb, uint8_t* Ld) {
    const uint8_t* lb = Lbase + (int64_t)kb * p.l_kb_stride;
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 ::"v"(ltail[n] ? voffLt : voffL), "s"(lb + lslab[n]),
                   "s"(lds_addr(Ld) + (uint32_t)((wave * 8 + (NT / 8) * n) * kBK))
                 : "memory");
  };
  auto dmaL_scales = [&](int kb, float* Sd) {
    if (l_side && step_scale) dma_scale(kb, Sd);
  };
  auto dmaR_tile = [&](int n, int kb, uint8_t* Rd) {
    const uint8_t* rb = Rbase + (int64_t)kb * p.r_kb_stride;
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 ::"v"(voffR), "s"(rb + rslab[n]),
                   "s"(lds_addr(Rd) + (uint32_t)((wave * 8 + (NT / 8) * n) * kBK))
                 : "memory");
  };
  auto dmaR_scales = [&](int kb, float* Sd) {
    if constexpr (!C::LAHEAD) {
      if (!l_side) dma_scale(kb, Sd);
      if (batch && (kb & 7) == 0) dma_scale_batch(kb >> 3);  // lands a step before its first use
    }
  };
  auto dmaL_one = [&](int n, int kb, uint8_t* Ld, float* Sd) {
    dmaL_tile(n, kb, Ld);
    if (n == C::LCH - 1) dmaL_scales(kb, Sd);
  };
  auto dmaR_one = [&](int n, int kb, uint8_t* Rd, float* Sd) {
    dmaR_tile(n, kb, Rd);
    if (n == C::RCH - 1) dmaR_scales(kb, Sd);
  };
  auto dmaL = [&](int kb, uint8_t* Ld, float* Sd) {
#pragma unroll
    for (int n = 0; n < C::LCH; n++) dmaL_one(n, kb, Ld, Sd);
  };
  auto dmaR = [&](int kb, uint8_t* Rd, float* Sd) {
#pragma unroll
    for (int n = 0; n < C::RCH; n++) dmaR_one(n, kb, Rd, Sd);
  };
  auto dma = [&](int kb, uint8_t* Ld, uint8_t* Rd, float* Sd) {
    dmaL(kb, Ld, Sd);
    dmaR(kb, Rd, Sd);
  };
  // End of a step: this thread's loads have landed, then the workgroup barrier.
  auto dma_wait_and_sync = [&]() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  // ---- MFMA tiling ------------------------------------------------------------------------
  // v_mfma_f32_32x32x64_f8f6f4: lane l supplies operand row l%32 and 32 contraction bytes chosen
  // by l/32; with two MFMAs per 128-byte step a lane reads, per row and K half h, the logical
  // chunks 4h + 2(l/32) and 4h + 2(l/32) + 1.  Any assignment works as long as L and R use the
  // same one.  D: lane l holds column l%32, rows 8(r/4) + 4(l/32) + r%4 for r = 0..15.
  // Wave w runs on SIMD w % 4.  With eight waves the two on a SIMD share their R half and take L
  // row blocks half a tile apart, so that in a tile whose valid rows end in the first half every
  // SIMD keeps one wave with work and one that only loads: such a tile finishes in about two
  // thirds of the time instead of leaving two SIMDs idle and two fully loaded (measured +2 % on a
  // Zipf-ragged 64-group launch; pairs that differ in both halves measured 1 % slower overall).
  constexpr bool kRemap = NT == 512 && C::WR == 2 && C::WL == 4;
  const int wr = kRemap ? wave & 1 : wave / C::WL;
  const int wl = kRemap ? ((wave & 3) >> 1) + 2 * (wave >> 2) : wave % C::WL;
  const int l32 = lane & 31, hg = lane >> 5;
  const int sw = swz(l32);
  int chk[2][2];  // byte offset of the two chunks of K half h inside this lane's row
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int c = 0; c < 2; c++) chk[h][c] = ((4 * h + 2 * hg + c) ^ sw) << 4;
  const int wrow0 = wr * C::WTR * 32;            // first R row of this wave inside the tile
  const int wlrow0 = wl * C::WTL * 32;           // first L row of this wave inside the tile
  // LDS byte addresses of this lane's four chunks in its row of the wave's first sub-tile, stage 0.
  // Kept opaque: every fragment read is one of these plus a compile-time offset.
  uint32_t la[2][2], ra[2][2];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int c = 0; c < 2; c++) {
      la[h][c] = (uint32_t)(uintptr_t)(lds_ptr_t)Lbuf0 + (uint32_t)((wlrow0 + l32) * kBK + chk[h][c]);
      if constexpr (R_ROWS) {
        // sub-tile row i = 2 h + c: the half chunk of contraction row 32 hg + tr that this lane names; the other rows of its
        // fragment are 8 and 64 rows on
        const int i = (2 * h + c) % C::WTR, tr = (lane & 15) >> 1;
        const int ch = (wrow0 / 16 + 2 * i + ((lane >> 4) & 1)) ^ (2 * (tr / (256 / BN)));
        ra[h][c] = (uint32_t)(uintptr_t)(lds_ptr_t)Rbuf0 + (uint32_t)((32 * hg + tr) * BN + ch * 16 + (lane & 1) * 8);
      } else {
        ra[h][c] = (uint32_t)(uintptr_t)(lds_ptr_t)Rbuf0 + (uint32_t)((wrow0 + l32) * kBK + chk[h][c]);
      }
      asm volatile("" : "+v"(la[h][c]));
      asm volatile("" : "+v"(ra[h][c]));
    }
  static_assert(!R_ROWS || C::WTR <= 4, "an address per sub-tile row");
  // fragment of sub-tile row `sub` (32 rows each) of one side in stage s, K half h
  typedef const __attribute__((address_space(3))) v4i* lds_v4i_t;
  auto frag = [&](const uint32_t (&base)[2][2], int s, int rows_per_stage, int sub, int h) __attribute__((always_inline)) {
    const uint32_t delta = (uint32_t)((s * rows_per_stage + sub * 32) * kBK);
    const v4i lo = *(lds_v4i_t)(uintptr_t)(base[h][0] + delta);
    const v4i hi = *(lds_v4i_t)(uintptr_t)(base[h][1] + delta);
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto fragR = [&](int s, int sub, int h) __attribute__((always_inline)) {
    if constexpr (R_ROWS) {
      v8i f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const v2i o = lds_read_transposed(ra[sub / 2][sub % 2] + (uint32_t)(s * BN * kBK + (64 * h + 8 * j) * BN));
        f[2 * j] = o[0];
        f[2 * j + 1] = o[1];
      }
      return f;
    } else {
      return frag(ra, s, BN, sub, h);
    }
  };
  const bool wave_active = wrow0 < rvalid;        // whole wave in or out: rvalid % 128 == 0
  // a wave none of whose L rows or R rows is valid takes part in loads and barriers only
  const bool has_work = __builtin_amdgcn_readfirstlane((int)(wave_active && wlrow0 < lvalid)) != 0;

  v16f acc[C::WTR][C::WTL];
#pragma unroll
  for (int i = 0; i < C::WTR; i++)
#pragma unroll
    for (int j = 0; j < C::WTL; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = short_operands ? __builtin_nanf("") : 0.f;

  // One 128-deep step on the stage (Lt, Rt, Sct).  Per 32x32 sub-tile t: two chained MFMAs, then
  // the 16 scale-and-accumulate FMAs of sub-tile t-1 run in their shadow.  The wanted issue
  // order is described to the scheduler with group barriers and fenced with scheduling
  // barriers; the accumulators are tied to the end of the step so the FMAs cannot drift past
  // the workgroup barrier.  Branch free: waves outside a partial R tile compute on clamped
  // rows and skip only the final store.
  constexpr int NTILES = C::WTR * C::WTL;
  auto compute = [&](int kb, int stage, const float* Sct, auto&& after_l_reads, auto&& per_tile) {
    __builtin_amdgcn_sched_barrier(0);
    // L scale of tile row r: Lsc[r * lsc_stride]
    const int bsel = kb >> 3;
    const float* Lsc = batch ? LsB0 + (bsel & 1) * (BM * 8) + (kb - batch_start(bsel)) : Sct;
    const int lsc_stride = batch ? 8 : 1;
    const float* Rsc = Sct + BM;
    v8i lf[C::WTL][2];
    float cs[C::WTL];
    const float rblk = R_PER_ROW ? 1.f : Rsc[wrow0 / kTile];
    v8i rf[2][2];
    // LDS reads in the order of first use: the first MFMA waits for two fragments only, the rest
    // arrive in its shadow
    lf[0][0] = frag(la, stage, BM, 0, 0);
    rf[0][0] = fragR(stage, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    lf[0][1] = frag(la, stage, BM, 0, 1);
    rf[0][1] = fragR(stage, 0, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < C::WTL; j++) {
      const int row = wlrow0 + j * 32 + l32;
      if (j > 0) {
        lf[j][0] = frag(la, stage, BM, j, 0);
        lf[j][1] = frag(la, stage, BM, j, 1);
      }
      cs[j] = Lsc[row * lsc_stride] * rblk;
    }
    v4f rs[2][4];  // R_PER_ROW: scales of the 16 R rows this lane holds in a sub-tile
    auto load_r = [&](int i) {
      if (i > 0) {
        rf[i & 1][0] = fragR(stage, i, 0);
        rf[i & 1][1] = fragR(stage, i, 1);
      }
      if constexpr (R_PER_ROW) {
#pragma unroll
        for (int q = 0; q < 4; q++)
          rs[i & 1][q] = *reinterpret_cast<const v4f*>(&Rsc[wrow0 + i * 32 + 8 * q + 4 * hg]);
      }
    };
    // raw-product buffers: sub-tile t's fold runs D = PRB - 1 sub-tiles later (0: right after it).
    // Per-row R scales live in a two-slot ring that allows at most D = 1.
    constexpr int PRB = R_PER_ROW && C::PRB > 2 ? 2 : C::PRB;
    constexpr int D = PRB - 1;
    v16f pr[PRB];
    load_r(0);
    // acc of sub-tile t += raw product * scales, registers [8*half, 8*half + 8) of the sub-tile
    auto fold_half = [&](int t, int half) {
      const int i = t / C::WTL, j = t % C::WTL;
#pragma unroll
      for (int r = 8 * half; r < 8 * half + 8; r++) {
        const float sc = R_PER_ROW ? cs[j] * rs[i & 1][r / 4][r % 4] : cs[j];
        acc[i][j][r] = __builtin_fmaf(pr[t % PRB][r], sc, acc[i][j][r]);
      }
    };
    v16f zero;
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.f;
    // Issue order per sub-tile, kept by full scheduling barriers: first MFMA, half of the previous
    // sub-tile's fold, second MFMA, the other half, then the LDS reads of the next R row.  Each MFMA
    // (16 passes) covers its own issue plus eight FMAs of another sub-tile.
    static_for<NTILES>([&](auto T) {
      constexpr int t = decltype(T)::value;
      constexpr int i = t / C::WTL, j = t % C::WTL;
      __builtin_amdgcn_sched_barrier(0);
      pr[t % PRB] = mfma_fp8_32x32x64(rf[i & 1][0], lf[j][0], zero);
      __builtin_amdgcn_sched_barrier(0);
      if (D >= 1 && t >= D) fold_half(t - D, 0);
      __builtin_amdgcn_sched_barrier(0);
      pr[t % PRB] = mfma_fp8_32x32x64(rf[i & 1][1], lf[j][1], pr[t % PRB]);
      __builtin_amdgcn_sched_barrier(0);
      if (D >= 1 && t >= D) fold_half(t - D, 1);
      if (D == 0) {
        fold_half(t, 0);
        fold_half(t, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      // the next R row overwrites the fragment and scale slot of row i - 1, whose last fold is done
      if (j == 0 && i + 1 < C::WTR) load_r(i + 1);
      __builtin_amdgcn_sched_barrier(0);
      // every L fragment has been an MFMA operand by now, so it has left the LDS: the hook (a
      // barrier and the next L loads) costs no extra wait here
      per_tile(T);
      if (t == C::WTL - 1) after_l_reads();
    });
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = NTILES - D; t < NTILES; t++) {
      fold_half(t, 0);
      fold_half(t, 1);
    }
    // tie the accumulators to this point: the FMAs above may not drift past the barrier below
#pragma unroll
    for (int i = 0; i < C::WTR; i++)
#pragma unroll
      for (int j = 0; j < C::WTL; j++) asm volatile("" : "+v"(acc[i][j]));
    __builtin_amdgcn_sched_barrier(0);
  };

  auto nothing = [] {};
  auto no_feed = [](auto) {};
  // Two workgroups per CU: the loads of a step go out in one burst after the barrier (issued a few
  // at a time behind the sub-tiles they measured 6 % slower here: they have less time to arrive,
  // and the other workgroup already fills the issue gap).
  if constexpr (!C::LAHEAD) {
    if (nkb > 0) dma(0, Lbuf0, Rbuf0, Sc0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // a wave without valid rows runs its own copy of the loop, loads and barriers only
    auto loop = [&](auto W) {
      constexpr bool kWork = decltype(W)::value;
      int kb = 0;
      for (; kb + 1 < nkb; kb += 2) {  // two steps per trip: the stage addresses are compile-time constants
        dma(kb + 1, Lbuf1, Rbuf1, Sc1);
        if constexpr (kWork) compute(kb, 0, Sc0, nothing, no_feed);
        dma_wait_and_sync();
        dma(kb + 2 < nkb ? kb + 2 : kb + 1, Lbuf0, Rbuf0, Sc0);  // the last prefetch re-reads a valid block
        if constexpr (kWork) compute(kb + 1, 1, Sc1, nothing, no_feed);
        dma_wait_and_sync();
      }
      if constexpr (kWork)
        if (kb < nkb) compute(kb, 0, Sc0, nothing, no_feed);  // odd number of steps
    };
    if (has_work) loop(std::true_type{});
    else loop(std::false_type{});
  } else {
    // One workgroup per CU, eight waves, two per SIMD.  The matrix pipe of a SIMD idles whenever both
    // of its waves are away from their MFMAs at the same time, which is what a workgroup barrier
    // followed by LDS reads produces.  So the two barriers of a step stand where register-resident
    // MFMA work follows them:
    //   Q (start of step k): every wave holds the L fragments of step k, so the L half of stage k is
    //     free and the L tile of step k+2 is requested behind the first sub-tiles;
    //   P (before the last R row of sub-tiles): every wave has read the last fragments of stage k
    //     and the tiles of step k+1 have landed; behind it the R tile of step k+2 is requested and
    //     the first fragments of step k+1 are read from the LDS while the last R row, whose operands
    //     are already in registers, runs on the matrix pipe.  The fragment registers of step k are
    //     reused as they die, so the prefetch costs no registers.
    // The fold of the sub-tile in front of a barrier is issued behind it: the wave that arrives last
    // has just issued its MFMAs, and the one that waited folds while those still run.
    // Loads complete in issue order, so "all but the newest L group" is one wait count.  Past the
    // end the loads re-read the last block to keep the counts uniform.
    static_assert(!R_PER_ROW && MODE == kRaggedRows, "the two-barrier pipeline is written for block-scaled R operands");
    static_assert(C::PRB == 1 && C::WTR % 2 == 0 && C::RCH % C::WTL == 0 && C::LCH <= NTILES, "pipeline shape");
    constexpr int PT = (C::WTR - 1) * C::WTL - 1;  // the sub-tile in front of barrier P
    constexpr int RPER = C::RCH / C::WTL;
    auto kclamp = [&](int k) { return k < nkb ? k : nkb - 1; };
    // Scales of this pipeline come in batches of eight contraction blocks only (the launcher takes the other
    // configuration when K has fewer than eight blocks), so a
    // step issues no scale load and takes no branch: batch b (blocks 8 b .. 8 b + 7, the last one shifted
    // back to end at the last block) is requested behind barrier P of step 8 (b - 1), eight steps before
    // its first use.  L scales: every wave fetches 32 rows x 32 bytes into LsB[b & 1][row][8]; R block
    // scales: wave 0 fetches the tile's two 128-row blocks x 32 bytes into RsB[b & 1][block][8] (lanes past
    // the fourth repeat those addresses: the direct-to-LDS load always writes 1 KB).
    // Scale rows that are not 16-byte aligned (a number of contraction blocks that is not a multiple of four, an
    // unaligned base) take 4-byte loads instead: four per wave and batch for the L scales (lane l of load q fetches
    // float 64 q + l of the wave's 32 rows x 8 floats), one for the R scales.
    float* const RsB0 = Sc0;  // [2][NT] floats, the first 16 of each in use
    const bool x4 = p.ls_batch == 1;
    const int rblocks = rvalid / kTile;
    const int rlane_blk = ((lane >> 1) & 1) < rblocks ? (lane >> 1) & 1 : rblocks - 1;
    const uint32_t roff = ((uint32_t)rlane_blk * (uint32_t)p.rs_row_stride + (uint32_t)(lane & 1) * 4u) * 4u;
    const int rlane_blk1 = ((lane >> 3) & 1) < rblocks ? (lane >> 3) & 1 : rblocks - 1;
    const uint32_t roff1 = ((uint32_t)rlane_blk1 * (uint32_t)p.rs_row_stride + (uint32_t)(lane & 7) * (uint32_t)p.rs_blk_stride) * 4u;
    uint32_t boff1[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int row = wave * 32 + q * 8 + (lane >> 3);
      boff1[q] = ((uint32_t)(row < lvalid ? row : lvalid - 1) * (uint32_t)p.ls_row_stride + (uint32_t)(lane & 7)) * 4u;
    }
    auto dma_batches = [&](int b) {
      const uint8_t* lsb = reinterpret_cast<const uint8_t*>(Lsg + uniform_i64(l0 * p.ls_row_stride + batch_start(b)));
      const uint8_t* rsb = reinterpret_cast<const uint8_t*>(Rsg + uniform_i64((r0 / kTile) * p.rs_row_stride + batch_start(b) * p.rs_blk_stride));
      const uint32_t ldst = lds_addr(LsB0 + (b & 1) * (BM * 8)) + (uint32_t)(wave * 1024);
      const uint32_t rdst = lds_addr(RsB0 + (b & 1) * NT);
      if (x4) {
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(boff), "s"(lsb), "s"(ldst) : "memory");
        if (!R_ROWS && wave == 0)
          asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(roff), "s"(rsb), "s"(rdst) : "memory");
      } else {
#pragma unroll
        for (int q = 0; q < 4; q++)
          asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(boff1[q]), "s"(lsb), "s"(ldst + (uint32_t)(q * 256)) : "memory");
        if (!R_ROWS && wave == 0)
          asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(roff1), "s"(rsb), "s"(rdst) : "memory");
      }
      if (R_ROWS && wave == 0)  // a row of scales per contraction block: never 16 bytes of one block
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(roff1), "s"(rsb), "s"(rdst) : "memory");
    };
    if (nkb > 0) {
      dmaL(0, Lbuf0, Sc0);  // (the per-step scale hooks of these helpers are off: see step_scale)
      dmaR(0, Rbuf0, Sc0);
      dma_batches(0);
      dmaL(kclamp(1), Lbuf1, Sc1);
      dmaR(kclamp(1), Rbuf1, Sc1);
      // the tiles of step 0 and the first scale batch have landed; those of step 1 may still be on their way
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::LCH + C::RCH) : "memory");
      auto barrier_q = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
      // all but this step's L tile loads have landed (loads complete in issue order)
      auto barrier_p = [&]() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::LCH) : "memory"); };
      if (has_work) {
        v8i lf[C::WTL][2], rf[2][2];
        float cs[C::WTL], csn[C::WTL], rblkn;
        float cs_last = 0.f;  // scale of the sub-tile whose fold is still owed (the last one of the step before)
        v16f pr, zero;
#pragma unroll
        for (int r = 0; r < 16; r++) zero[r] = pr[r] = 0.f;
        // scales of step kb: the lane's L row scales and the R block scale of the wave; their product is
        // formed where it is first needed, not where the reads are issued
        auto read_scales = [&](int kb, float (&dst)[C::WTL], float& rblk) {
          const int b = kb >> 3, in_batch = kb - batch_start(b);
          const float* Lsc = LsB0 + (b & 1) * (BM * 8) + in_batch;
          rblk = RsB0[(b & 1) * NT + (wrow0 / kTile) * 8 + in_batch];
#pragma unroll
          for (int j = 0; j < C::WTL; j++) dst[j] = Lsc[(wlrow0 + j * 32 + l32) * 8];
        };
        // (the empty volatile statements pin MFMAs and folds between the memory instructions around
        // them: plain arithmetic is otherwise free to drift past inline assembly)
        auto fold = [&](int i, int j, float sc) {
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][j][r] = __builtin_fmaf(pr[r], sc, acc[i][j][r]);
          asm volatile("" : "+v"(acc[i][j]));
        };
        // fragments and scales of step 0
#pragma unroll
        for (int h = 0; h < 2; h++) {
          lf[0][h] = frag(la, 0, BM, 0, h);
          rf[0][h] = fragR(0, 0, h);
        }
#pragma unroll
        for (int j = 1; j < C::WTL; j++)
#pragma unroll
          for (int h = 0; h < 2; h++) lf[j][h] = frag(la, 0, BM, j, h);
        read_scales(0, cs, rblkn);
#pragma unroll
        for (int j = 0; j < C::WTL; j++) cs[j] *= rblkn;
        // FIRST: the first step of a run of eight, which requests the next scale batch behind barrier P
        auto step = [&](int kb, auto S, auto FIRST) {
          constexpr int s = decltype(S)::value;
          constexpr bool kFirst = decltype(FIRST)::value;
          uint8_t* const Lc = s ? Lbuf1 : Lbuf0;
          uint8_t* const Rc = s ? Rbuf1 : Rbuf0;
          const int k2 = kclamp(kb + 2);
          __builtin_amdgcn_sched_barrier(0);
          barrier_q();
          __builtin_amdgcn_sched_barrier(0);
          fold(C::WTR - 1, C::WTL - 1, cs_last);  // owed by the step before (adds zero in the first step)
          static_for<NTILES>([&](auto T) {
            constexpr int t = decltype(T)::value;
            constexpr int i = t / C::WTL, j = t % C::WTL;
            __builtin_amdgcn_sched_barrier(0);
            pr = mfma_fp8_32x32x64(rf[i & 1][0], lf[j][0], zero);
            pr = mfma_fp8_32x32x64(rf[i & 1][1], lf[j][1], pr);
            asm volatile("" : "+v"(pr));
            __builtin_amdgcn_sched_barrier(0);
            // memory instructions go out while the MFMAs run, ahead of the fold that waits for them
            if constexpr (t < C::LCH) dmaL_tile(t, k2, Lc);
            if constexpr (j == 0 && i + 1 < C::WTR) {
#pragma unroll
              for (int h = 0; h < 2; h++) rf[(i + 1) & 1][h] = fragR(s, i + 1, h);
            }
            if constexpr (t == PT) {
              __builtin_amdgcn_sched_barrier(0);
              barrier_p();
              __builtin_amdgcn_sched_barrier(0);
              if constexpr (kFirst) {
                if (kb + 8 < nkb) dma_batches((kb >> 3) + 1);
              }
              // row C::WTR - 2 has been consumed: its registers take the first R row of the next step
#pragma unroll
              for (int h = 0; h < 2; h++) rf[0][h] = fragR(s ^ 1, 0, h);
              read_scales(kclamp(kb + 1), csn, rblkn);
            }
            if constexpr (t > PT) {
              constexpr int jn = t - PT - 1;  // == j: this sub-tile was the last user of lf[j]
              static_for<RPER>([&](auto N) { dmaR_tile(jn * RPER + decltype(N)::value, k2, Rc); });
#pragma unroll
              for (int h = 0; h < 2; h++) lf[jn][h] = frag(la, s ^ 1, BM, jn, h);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (t + 1 < NTILES) fold(i, j, cs[j]);
          });
          cs_last = cs[C::WTL - 1];
#pragma unroll
          for (int j = 0; j < C::WTL; j++) cs[j] = csn[j] * rblkn;
        };
        // runs of eight steps (the contraction has at least eight blocks; the last run may be shorter), two
        // steps per trip so that the stage addresses are compile-time constants
        constexpr std::integral_constant<int, 0> S0{};
        constexpr std::integral_constant<int, 1> S1{};
        for (int kb = 0; kb < nkb; kb += 8) {
          const int n = nkb - kb < 8 ? nkb - kb : 8;
          step(kb, S0, std::true_type{});
          if (n > 1) step(kb + 1, S1, std::false_type{});
          int kk = 2;
          for (; kk + 1 < n; kk += 2) {
            step(kb + kk, S0, std::false_type{});
            step(kb + kk + 1, S1, std::false_type{});
          }
          if (kk < n) step(kb + kk, S0, std::false_type{});  // odd number of steps
        }
        __builtin_amdgcn_sched_barrier(0);
        fold(C::WTR - 1, C::WTL - 1, cs_last);
      } else {
        // a wave without valid rows: loads and barriers only, in the order of the working waves
        auto step = [&](int kb, uint8_t* Lc, uint8_t* Rc, bool first) {
          const int k2 = kclamp(kb + 2);
          barrier_q();
#pragma unroll
          for (int n = 0; n < C::LCH; n++) dmaL_tile(n, k2, Lc);
          barrier_p();
          if (first && kb + 8 < nkb) dma_batches((kb >> 3) + 1);
#pragma unroll
          for (int n = 0; n < C::RCH; n++) dmaR_tile(n, k2, Rc);
        };
        int kb = 0;
        for (; kb + 1 < nkb; kb += 2) {
          step(kb, Lbuf0, Rbuf0, (kb & 7) == 0);
          step(kb + 1, Lbuf1, Rbuf1, false);
        }
        if (kb < nkb) step(kb, Lbuf0, Rbuf0, (kb & 7) == 0);
      }
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the trailing loads must not land in the epilogue's staging
    }
  }

  // ---- epilogue ------------------------------------------------------------------------------
  // A lane holds, for one output row, groups of four consecutive columns; stored directly that
  // would be 8-byte pieces in 32 different rows per instruction.  Each wave instead transposes its
  // tile through its own LDS region and writes 128-byte row segments: 8 lanes x 16 bytes per row.
  if (MODE == kRaggedK && nkb == 0 && p.accumulate && !short_operands) return;  // empty group: leave dW untouched
  __syncthreads();  // every wave is done with the stage buffers
  if (!has_work) return;
  OUT* Cg = reinterpret_cast<OUT*>(p.C) + (int64_t)g * p.c_group_stride;
  uint8_t* const stg = lds + wave * kStgBytes;
  constexpr int WROWS = C::WTL * 32;
  static_assert(WROWS <= 64 && WROWS % 8 == 0, "the staging region holds 64 rows");
  // (the bias is a compile-time case: without one the staging is two conversions and a write per
  // four values instead of a uniform branch, four adds and the moves that feed them)
  // (inlined by order: called, it would hold everything it captures in memory)
  auto flush = [&](auto tag, auto with_bias) __attribute__((always_inline)) {
    using ST = decltype(tag);  // staging type: OUT, or float when the old output is added in fp32
    constexpr bool kBias = decltype(with_bias)::value;
    constexpr int CW = 128 / (int)sizeof(ST);  // columns per chunk
    constexpr int SUBS = CW / 32;              // 32-column sub-tiles per chunk
    constexpr int PITCH = 128 + (sizeof(ST) == 2 ? 8 : 16);
    constexpr int VL = 16 / (int)sizeof(ST);   // columns per lane in the store phase
    static_assert(C::WTR % SUBS == 0, "chunks cover whole sub-tiles");
#pragma unroll
    for (int ci = 0; ci < C::WTR / SUBS; ci++) {
#pragma unroll
      for (int si = 0; si < SUBS; si++) {
        const int i = ci * SUBS + si;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int64_t rcol = r0 + wrow0 + i * 32 + 8 * q + 4 * hg;
          v4f b4 = {0.f, 0.f, 0.f, 0.f};
          if constexpr (kBias) {
            if (p.bias_dtype == AAMD_F32) {
              b4 = *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(p.bias) + g * p.bias_group_stride + rcol);
            } else {
              const v2i raw = *reinterpret_cast<const v2i*>(reinterpret_cast<const u16*>(p.bias) + g * p.bias_group_stride + rcol);
              b4[0] = bf16_bits_to_f32((uint32_t)raw[0] & 0xffffu);
              b4[1] = bf16_bits_to_f32((uint32_t)raw[0] >> 16);
              b4[2] = bf16_bits_to_f32((uint32_t)raw[1] & 0xffffu);
              b4[3] = bf16_bits_to_f32((uint32_t)raw[1] >> 16);
            }
          }
#pragma unroll
          for (int j = 0; j < C::WTL; j++) {
            v4f o = v4f{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            if constexpr (kBias) o += b4;
            uint8_t* dst = stg + (j * 32 + l32) * PITCH + (si * 32 + 8 * q + 4 * hg) * (int)sizeof(ST);
            if constexpr (sizeof(ST) == 4) {
              *reinterpret_cast<v4f*>(dst) = o;
            } else {
              v2i w;
              w[0] = (int)pack_bf16x2(o[0], o[1]);
              w[1] = (int)pack_bf16x2(o[2], o[3]);
              *reinterpret_cast<v2i*>(dst) = w;
            }
          }
        }
      }
      __builtin_amdgcn_wave_barrier();  // same wave, in-order LDS: the reads below see the writes above
      const int64_t col = r0 + wrow0 + ci * CW + (lane & 7) * VL;
      // all rows of the chunk leave the LDS before the first store: inside the row-valid branches
      // each read would be followed by its own wait.  One 64-bit row address per chunk, then steps
      // of eight rows.
      v4i raws[WROWS / 8];
#pragma unroll
      for (int ps = 0; ps < WROWS / 8; ps++)
        raws[ps] = *reinterpret_cast<const v4i*>(stg + (ps * 8 + (lane >> 3)) * PITCH + (lane & 7) * 16);
#pragma unroll
      for (int ps = 0; ps < WROWS / 8; ps++) asm volatile("" : "+v"(raws[ps]));
      OUT* const out_row0 = Cg + (l0 + wlrow0 + (lane >> 3)) * p.ldc + col;
      const int64_t row_step = 8 * p.ldc;
      // accumulation into an fp32 output: the old values of all rows are requested before the
      // first is used (one trip to memory per chunk instead of one per row)
      // (only the weight gradient accumulates; in the row-ragged kernels the old values cost registers and spills)
      constexpr bool kAddF32 = MODE == kRaggedK && sizeof(ST) == sizeof(OUT) && sizeof(OUT) == 4;
      v4f olds[kAddF32 ? WROWS / 8 : 1];
      if constexpr (kAddF32) {
        if (p.accumulate) {
          OUT* o_row = out_row0;
#pragma unroll
          for (int ps = 0; ps < WROWS / 8; ps++) {
            olds[ps] = v4f{0.f, 0.f, 0.f, 0.f};
            if (wlrow0 + ps * 8 + (lane >> 3) < lvalid) olds[ps] = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(o_row));
            o_row += row_step;
          }
#pragma unroll
          for (int ps = 0; ps < WROWS / 8; ps++) asm volatile("" : "+v"(olds[ps]));
          // (added here, not at the stores: held next to the new values until then they do not fit, and ten registers of
          // every thread went through memory, an eighth of what the launch writes.  Us with and
          // without: 8 groups of 4096 rows, 28672 x 4096 outputs written over 4800, 4660, added 5480, 4975; 60 groups of 1092
          // rows, 2816 x 2048, 756, 670 and 990, 806)
#pragma unroll
          for (int ps = 0; ps < WROWS / 8; ps++) raws[ps] = __builtin_bit_cast(v4i, __builtin_bit_cast(v4f, raws[ps]) + olds[ps]);
        }
      }
      OUT* out_row = out_row0;
#pragma unroll
      for (int ps = 0; ps < WROWS / 8; ps++) {
        const int lrow = wlrow0 + ps * 8 + (lane >> 3);
        const v4i raw = raws[ps];
        OUT* out = out_row;
        out_row += row_step;
        if (lrow < lvalid) {
          if constexpr (sizeof(ST) == sizeof(OUT)) {
            // the output is not read again by this launch: streaming stores keep it from
            // evicting operand panels from L2 (measured +1-2 % where the output is large)
            __builtin_nontemporal_store(raw, reinterpret_cast<v4i*>(out));
          } else {  // fp32 staging, bf16 output with accumulation
            store4<OUT>(out, __builtin_bit_cast(v4f, raw), true);
          }
        }
      }
      __builtin_amdgcn_wave_barrier();  // the next chunk overwrites the region
    }
  };
  const bool with_bias = MODE == kRaggedRows && p.bias != nullptr;
  auto flush_as = [&](auto tag) __attribute__((always_inline)) {
    if constexpr (MODE == kRaggedRows) {
      if (with_bias) flush(tag, std::true_type{});
      else flush(tag, std::false_type{});
    } else {
      flush(tag, std::false_type{});
    }
  };
  if constexpr (sizeof(OUT) == 4) {
    flush_as(float{});
  } else {
    if (MODE == kRaggedK && p.accumulate) flush_as(float{});
    else flush_as(u16{});
  }
}

// Launch choices a caller of the measurement build may pin per call (-1 = the library chooses, which is
// all the product entry points ever pass).
struct GemmOptions {
  int tile = -1;      // 0: 128x128 tiles, 1: 256x256 tiles, 2 / 3: the kernel for few rows, 3 in its split form, 7 / 8 with two waves and one, 4: a workgroup per 256x256 tile, 6: 256x256 tiles of up to 288 rows
  int group_r = -1;   // tile order groups R tiles (1) or L tiles (0)
  int gl = -1;        // tiles that share a panel in the tile order
  int ls_batch = -1;  // 0: L scales fetched one contraction block at a time
};

// Tiles that share panels: the order of the tiles (rows: L rows of a tile).
template <int MODE>
static void tile_order(GemmParams& p, int rows, const GemmOptions& g_opt) {
  // L tiles per group of the tile order: 8 for the row-ragged launches; 4 for wgrad, whose operand
  // panels run over all tokens of an expert and are several times larger (measured: 5 % faster
  // at 4096 tokens per expert and 28672 x 4096 outputs, within 3 % either way elsewhere)
  p.gl = MODE == kRaggedK ? 4 : 8;
  // group along the side with more tiles per expert.  256 x 256 tiles, persistent, us, L tiles in groups of 4 / 8 and R tiles in
  // batches of 2 / 4 / 8 / 16: 32768 rows in 8 groups, 28672 x 4096 3638 / 3592 and 3567 / 3505 / 3512 / 3622, 4096 x 14336 1805 /
  // 1823 and 1867 / 1793 / 1807 / 1873; along the weights' rows, 4096 x 28672 3670 / 3681 and 3811 / 3666 / 3689 / 3900, 14336 x
  // 4096 1870 / 1827 and 1835 / 1804 / 1818 / 1843; 65536 uneven rows in 64, 4096 x 7168 1947 / 1993 and 1918 / 1864 / 1877 / 1951;
  // 131072 in 60, 2816 x 2048 and 2048 x 1408: within 4 %, the noise of the run.
  if (MODE == kRaggedK) p.group_r = p.nRt > p.nLt;
  else p.group_r = p.goff != nullptr && (int64_t)p.nRt * rows * p.E > p.Lrows;
  if (MODE == kRaggedRows && p.group_r) p.gl = 4;
  // per-call overrides (measurement build only)
  if (g_opt.group_r >= 0) p.group_r = g_opt.group_r != 0 && (MODE == kRaggedK || p.goff != nullptr);
  if (g_opt.gl > 0) p.gl = g_opt.gl;
}

template <int MODE, bool R_PER_ROW, typename C, bool R_ROWS = false>
static int launch_gemm(GemmParams p, int c_dtype, int64_t blocks, hipStream_t st, const GemmOptions& g_opt) {
  if (blocks <= 0) return AAMD_OK;
  tile_order<MODE>(p, C::BM, g_opt);
  AAMD_REQUIRE(blocks < 0x7fffffffLL, "grouped_gemm: grid too large");
  dim3 grid((unsigned)blocks), block(C::NT);
  if (c_dtype == AAMD_BF16)
    grouped_gemm_kernel<MODE, R_PER_ROW, u16, C, R_ROWS><<<grid, block, 0, st>>>(p);
  else
    grouped_gemm_kernel<MODE, R_PER_ROW, float, C, R_ROWS><<<grid, block, 0, st>>>(p);
  AAMD_LAUNCH_CHECK("grouped_gemm");
  return AAMD_OK;
}

// The 256 x 256 tiles' last round may share out its contraction (row_tiles_kernel) from this many blocks on; shorter ones share rows (row_shares).
// us, rows shared and contraction shared, 2048 outputs, one round of 256 tiles and a last one of 1 / 4 / 8 / 12 / 16 tiles per XCD (in 8 / 8 /
// 4 / 2 / 2 parts): 40 blocks 113 / 113 / 115 / 125 / 130 and 103 / 107 / 119 / 125 / 134, 48 133 / 133 / 136 / 148 / 152 and 118 / 124 / 133 /
// 142 / 153, 64 173 / 174 / 178 / 192 / 197 and 148 / 156 / 164 / 178 / 190, 112 295 / 296 / 301 / 317 / 325 and 234 / 250 / 267 / 293 / 312.
// Where nothing is shared the second launch costs 2 to 6 us of at least 100 (choose_nt).
constexpr int kSplitBlocks = 48;
// The most parts of a contraction: eight blocks at least in each, see row_part.
static int row_max_split(int64_t nkb) { return (int)std::min<int64_t>(8, nkb / 8); }

// Which kernel a row-ragged launch with block-scaled R takes: the one whose estimated time is least.  The estimates (us) were
// fitted to 3280 timings on MI355X of launches of 1 to 40000 rows in 1 to 64 groups, even and uneven (Zipf) ones, 512 to 18000
// outputs and a contraction of 512 to 14336, weights along either side and in a cache or in none, each with all of the kernels
// (n: 128-deep steps):
//   - 128 x 128 tiles, two of them per CU: up to a tile per CU 5.4 and 0.76 per step; else 2.9, and 3.3 and 1.045 per step for
//     every round of 512 tiles; the last of few rounds up to 0.08 per step less where not every CU has two, 0.85 where none has;
//   - 256 x 256 tiles 6.5, and 6.3 and 0.78 to 1.08 per step for every round of 256, by how full the tiles and the round are;
//     with a last round in parts 20 and 10 times what it fills, for writing and adding them, and its steps by the number of
//     parts; 4 more where a workspace is at hand and the last round turns out not to be shared;
//   - a 64 x 64 block of the kernel for few rows 2.7 ns and 1.1 ns per step, spread over the chip, with two waves 1.1 and 1.135, with
//     one 0.26 and 1.135; a 32 x 32 block of its split form 3.6 and 0.47; and no less than a wave's own chain of every fourth (second,
//     single, eighth) step;
//   - and none can beat the weights' stream from memory.
// The groups' sizes are known on the device only.  Groups with rows are expected to be E (1 - exp(-0.6 M / E)), token tiles one
// per such group with few rows and 0.56 of a tile per group more than the rows fill with many; what depends on rounds is the mean
// over that many tiles and up to 16 % more and less, by what the groups' own tiles are of them.  The kernel taken is 1.2 % slower
// than the best of them (geometric mean; more than 5 % slower in 7 %) over those timings, and 1.3 % over 4400 others; the lines these
// replace, which priced the large tiles as they were with a workgroup per tile and took whole rounds of expected tiles, came to
// 3.2 and 3.2 % (15 %).  Where the kernel changed it takes 0.90 of the time on average.  us: 83 rows in 64 groups, 768 x 768 9.6 ->
// 3.9; 2965 in 60 (Zipf), 2048 x 11008 200 -> 97; 726 in 8, 6528 x 6656 141 -> 85; 1394 in 16, 5888 x 9216 186 -> 116.  Of the
// others 2.9 % take 3 % or more longer than before, 11 % that much less; the worst are uneven groups, whose empty ones the host
// does not know of (1776 in 60, 25856 x 512 63 -> 110; 3532 in 16, 1664 x 6144 53 -> 67).
enum NtKernel { kSmallTiles = 0, kLargeTiles = 1, kFewRows = 2, kFewRowsSplit = 3, kLargeOnce = 4, kLargeShared = 5, kLargeMore = 6, kFewRowsTwo = 7, kFewRowsOne = 8 };
static bool is_few_rows(NtKernel k) { return k == kFewRows || k == kFewRowsSplit || k == kFewRowsTwo || k == kFewRowsOne; }
static int few_rows_waves(NtKernel k) { return k == kFewRowsSplit ? 8 : k == kFewRowsTwo ? 2 : k == kFewRowsOne ? 1 : 4; }
// b_rows: weights read along their rows, which the split form and those of one and two waves cannot.  share_last: with a workspace for
// parts of the last round of 256 x 256 tiles.
//
// How many waves share the contraction of a 64 x 64 block: a CU holds two blocks of four waves, four of two or eight of one, with as
// many loads in flight.  With fewer waves there is less to add up at the end, and 513 to 1024 (2048) blocks are no second round: 544
// blocks of 4 steps 8.9 us with four, 7.3 with two, 512 blocks 6.5 and 6.9; 1440 blocks of few rows, of 1 / 2 / 4 / 8 / 16 steps,
// four waves 11.1 / 11.6 / 15.2 / 20.5 / 31.8, one 5.6 / 6.4 / 11.2 / 17.5 / 30.0.  The blocks of a
// launch without groups are known, and 512 (1024) are a round of four (two) waves yet: 512 blocks of 4 / 8 / 16 steps 6.2 / 7.5 / 10.6 with
// four, 6.6 / 8.4 / 11.9 with two; 516 8.4 / 10.5 / 14.3 and 6.8 / 8.9 / 12.4; 1024 8.2 / 12.2 / 18.8 with two, 8.6 / 13.8 / 19.8 with one.
// Of groups the lines lie where the mean of 12400 drawn launches
// (1 to 64 groups, 8 to 6000 rows, 512 to 5120 outputs and a contraction of 256 to 5120, replayed in a graph) turns; past 20 steps, or
// 14 with weights beyond the last-level cache, the weights' stream bounds such launches (64 groups of 6 rows, 7168 x 2048: 164 with four,
// 168 with one).  Of 14351 others, even and Zipf, 4000 take these forms, 0.819 of the time, 83 of them 3 % slower or more (2414 rows in 61,
// 512 x 896 7.0 -> 8.3; 1742 in 23, 2560 x 1024 19.7 -> 23.3); with two thirds of the groups empty, which the host does not know, 0.853 and a
// fifth of them (86 rows in 7 of 32, 2560 x 2048 9.4 -> 13.7).  One wave not where the rows
// of a group, which every 64 outputs read again, fill much of an XCD's L2, nor where the output and the weights pass the last-level cache, unless
// most of that are weights: 128 x 128 tiles and one wave, us, 30000 rows, 4096 x 256 88 and 117; 8195 rows in 2, 21760 x 256 137 and 163; 9600
// in 32, fp32 8192 x 256 78 and 118.  Of 2500 launches of 1 to 8 steps and 700 blocks or more these lines take it for 848, 0.815 of the time, 32
// of them 3 % slower or more; without them for 1162, 0.910 and 314.  A wave's chain of sums is as much longer, one wave's the tiles' own; against
// 64-bit sums all are off by the same, 1.42e-5 in fp32 (19 steps).  The forms that quantise their rows take the same, and give the same bits:
// eight tokens to 8 of 128 experts, 2048 x 768, layer 59 -> 53, 256, 1024 x 512 36 -> 33.
static NtKernel choose_nt(int64_t M, int64_t N, int64_t nkb, int64_t E, bool grouped, bool b_rows, bool share_last, int c_dtype, const GemmOptions& g_opt) {
  if (g_opt.tile >= 0) return (g_opt.tile == 1 || g_opt.tile == 4 || g_opt.tile == 6) && nkb < 8 ? kSmallTiles : (NtKernel)g_opt.tile;
  const bool one = !grouped || E == 1;
  const double n = (double)nkb, rows = (double)M;
  const double groups = one ? 1.0 : std::min({rows, (double)E, (double)E * (1.0 - std::exp(-0.6 * rows / (double)E))});
  auto token_tiles = [&](int64_t size) {
    return one ? (double)((M + size - 1) / size) : std::max(rows / (double)size + 0.56 * groups, groups);
  };
  // the time of a launch of about tiles x per rounds
  auto mean = [&](double tiles, double per, auto&& time) {
    const double x = tiles * per, d = std::min(0.16, 0.45 * groups / tiles);
    return one ? time(x) : (time((1.0 - d) * x) + time(x) + time((1.0 + d) * x)) / 3.0;
  };
  const double weights = groups * (double)N * n * (double)kBK * 1e-6;  // MB

  // (with many rounds the tiles' times spread and part of a round is lost at the end)
  auto small_time = [&](double x) {
    if (x <= 1.0) return 5.4 + 0.76 * n;
    const double round = 3.3 + 1.045 * n;
    if (x >= 6.0) return 2.9 + (0.5 * x + 0.6) * round;
    const double whole = std::ceil(0.5 * x) - 1.0, left = x - 2.0 * whole;
    return 2.9 + whole * round + (left <= 1.0 && whole > 0.0 ? 3.5 + 0.85 * n : round - 0.08 * (2.0 - left) * n);
  };
  const double small = std::max(mean(token_tiles(128), (double)(N / 128) / 256.0, small_time), weights / 5.1);

  // (the 256 x 256 tiles take their scales in batches of eight contraction blocks)
  const double tiles_l = token_tiles(256), fill = std::min(1.0, rows / (256.0 * tiles_l)), per_l = (double)((N + 255) / 256) / 256.0;
  auto round_l = [&](double x) { return 6.3 + (0.78 + 0.16 * fill + 0.14 * std::min(x, 1.0)) * n; };
  auto large_time = [&](double x) { return 6.5 + (x <= 1.0 ? 1.0 : x < 3.0 ? std::ceil(x) : x + 0.66) * round_l(x); };
  auto shared_time = [&](double x) {
    const double whole = std::floor(x), left = x - whole;
    if (left > 0.5) return 4.0 + large_time(x);
    if (whole >= 1.0 && left <= 1.0 / 32.0) return 4.0 + 6.5 + whole * round_l(x);
    const double parts = std::min((double)row_max_split(nkb), std::floor(1.0 / left));
    return 20.0 + 10.0 * left + 6.5 + whole * round_l(x) + (0.92 + 0.16 * fill) * n / parts;
  };
  const double large = nkb < 8 ? 1e30 : std::max(mean(tiles_l, per_l, large_time), weights / 6.7);
  const double shared = nkb < 8 || !share_last ? 1e30 : std::max(mean(tiles_l, per_l, shared_time), weights / 6.7);

  const double blocks_f = token_tiles(64) * (double)(N / 64), blocks_s = token_tiles(32) * (double)(N / 32);
  const bool fewer_waves = !b_rows && nkb < (weights <= 256.0 ? 20 : 14);
  const bool many = blocks_f >= (nkb < 4 ? 724.0 : one ? 1025.0 : 1024.0);
  const double written = rows * (double)N * (c_dtype == AAMD_BF16 ? 2e-6 : 4e-6), read_again = rows / groups * n * (double)kBK * 1e-6;
  const bool one_wave = fewer_waves && many && read_again <= 1.5 && (0.8 * weights + written <= 240.0 || 3.0 * written <= 2.0 * weights);
  const bool two_waves = fewer_waves && !many && blocks_f >= (one ? 513.0 : 500.0);
  const double few = one_wave    ? std::max({5.8 + 1e-3 * blocks_f * (1.135 * n + 0.26), 4.4 + 0.64 * n, weights / 6.8})
                     : two_waves ? std::max({5.3 + 1e-3 * blocks_f * (1.135 * n + 1.1), 4.5 + 0.65 * std::ceil(n / 2.0), weights / 6.8})
                                 : std::max({4.5 + 1e-3 * blocks_f * (1.1 * n + 2.7) * (b_rows ? 1.015 : 1.0), 3.2 + 1.12 * std::ceil(n / 4.0), weights / 6.8});
  const double split = b_rows ? 1e30 : std::max({2.6 + 1e-3 * blocks_s * (0.47 * n + 3.6), 3.8 + 0.52 * std::ceil(n / 8.0), weights / 6.8});

  const double tiles = std::min({small, large, shared});
  if (std::min(few, split) <= tiles) return split < few ? kFewRowsSplit : one_wave ? kFewRowsOne : two_waves ? kFewRowsTwo : kFewRows;
  if (small <= tiles) return kSmallTiles;
  if (shared <= tiles) return kLargeShared;
  // A workgroup per tile where none would have a second one: the step of grouped_gemm_kernel has no bookkeeping of a stream of
  // tiles (next tile, next scales; with an odd number of steps also the addresses of the stages) and is 1 to 3 % shorter, which
  // counts while power does not bound the launch.  Persistent over this form, 486 launches of at most a round, mean ratio: up to 0.25
  // rounds 1.01, 0.5 1.02, 0.75 1.04 (the most 1.11), 1 1.02; 1 to 1.5 0.99, 2 0.97, more 0.94 to 0.97.
  return tiles_l * per_l <= 1.0 ? kLargeOnce : kLargeTiles;
}
static bool takes_slices(const GemmParams& p) { return p.group_r && p.E <= 64 && p.nRt >= 32; }
// Tiles of up to 288 rows: the kernel decides by the groups' rows (0), where there can be enough remainders (a group's own tile costs two
// thirds of one, and its full tiles a twentieth of one each: not with more than seven of them; nor with much less than one) and the 0.2 to 0.5
// us that deciding takes are little.
static int choose_higher(const GemmParams& p, bool parts) {
  if (p.goff != nullptr)
    return p.E > 64 || p.Lrows >= (int64_t)7 * kLargeTile * p.E || p.Lrows < (int64_t)kLargeTile * 15 / 16 * p.E || p.nRt < 16 || p.nRt > 1024 ? -1 : 0;
  const uint32_t full = (uint32_t)std::min<int64_t>(p.Lrows / kLargeTile, 8), over = (uint32_t)(p.Lrows % kLargeTile), more = (over + 31) / 32;
  return over > 0 && more <= full && full < 8 && p.nRt <= 1024 && higher_tiles_pay(full, 1, 0, more, (uint32_t)p.nRt, full * (uint32_t)p.nRt, parts) ? 1 : -1;
}
// Tile-scaled R (per-row scales, the dense weight gradient): 256 x 128 tiles when there are enough of them.
static bool use_large_tiles(int64_t tiles_256, const GemmOptions& g_opt) {
  return g_opt.tile >= 0 ? g_opt.tile == 1 : tiles_256 >= 512;
}

// Weight gradient: the tiles of groups of at most kShortBlocks contraction blocks (1024 rows) are taken in runs
// (wgrad_short_tiles) where the groups have kShortAverage blocks or fewer on average; longer ones cover a tile's turnover by
// themselves.  Runs of four tiles (two for an fp32 output that is written only, whose stores alone keep the memory busy),
// and fewer where the launch would have less than kShortUnits workgroups.  Measured on MI355X, us, one tile per workgroup
// -> runs of 1 / 2 / 4 / 8 tiles with the line at 8 blocks, the line at 4 and runs of 4, and the stream of the outputs:
//   64 groups, 8192 rows (Zipf), 2048 x 7168 bf16          531 -> 480 / 447 / 454 / 461, 478    342
//   60 groups, 16001 rows (Zipf), 2816 x 2048 fp32, added  224 -> 178 / 169 / 151 / 164, 163
//   60 groups, 32764 rows (uneven), 2816 x 2048 bf16       365 -> 362 / 333 / 321 / 340, 330    126
//   60 groups, 4096 rows, 2816 x 2048 bf16                 201 -> 181 / 147 / 128 / 132, 139    126
//   8 groups, 1000 rows, 4096 x 1024 bf16                   23 -> 23 / 19 / 19 / 19, 19          12
//   60 groups, 400 rows, 1408 x 2048 fp32                  119 -> 115 / 118 / 139 / 162, 140    126
//   8 groups, 8192 rows, 4096 x 4096 bf16                  221 -> 238 / 227 / 226 / 250, 210     49
// (the last is where the average rule ends it: from there on both forms are within the noise of each other)
constexpr int kShortBlocks = 8, kShortAverage = 8, kShortUnits = 1024;
static bool use_short_runs(const GemmParams& p) {
  return p.goff != nullptr && p.E <= 64 && p.max_kb <= (int64_t)kShortAverage * p.E &&
         (int64_t)p.E * p.nLt * p.nRt < (1 << 27);
}

// Weight gradient on 256 x 256 tiles (wgrad_tiles_kernel)?  Its workgroups take their tiles in a fixed order, a round of 256 after the
// other, so a group's tiles have to fill their rounds nearly (the length of a round is its group's, known on the device only),
// and so have all of them.  Measured on MI355X, bf16, us, 128 x 128 tiles -> these:
//   32768 rows in 8 groups (33 blocks each), 28672 x 4096 4495 -> 4119, Zipf 4540 -> 4183; 4096 x 14336 2244 -> 2095, Zipf 2236 -> 2169
//   16384 rows in 16 groups (8), 4096 x 4096 436 -> 374, Zipf 426 -> 397; 12288 (6) 399 -> 319, Zipf 316 -> 331
//   8192 rows in 8 groups (8), 28672 x 4096 1624 -> 1301; 3584 x 8192 397 -> 334; 4096 x 14336, Zipf 739 -> 673
//   4096 rows in 8 groups (4), 28672 x 4096 970 -> 840, Zipf 871 -> 878; 4096 x 4096 148 -> 120, Zipf 133 -> 128; 2048 (2) 589 -> 631
//   rounds that are not filled: 131072 rows in 60 groups (Zipf), 2816 x 2048 (88 tiles a group) 1037 -> 1425; one group of 16384,
//   14336 x 4096 (3.5 rounds) 996 -> 1113
// fp32, whose stores are twice as long and come at once: 32768 rows in 8 groups, 28672 x 4096 4569 -> 4397, 16384, 14336 x 4096
// 1355 -> 1296, 32768, 4096 x 4096 658 -> 645, 16384 in 16 groups 447 -> 464.
static bool use_large_wgrad(const GemmParams& p, int c_dtype, const GemmOptions& g_opt) {
  const bool can = p.E <= 64 && !p.accumulate && p.Lrows < (1 << 23) && p.Rrows < (1 << 23);
  if (g_opt.tile >= 0) return can && g_opt.tile == 1;
  if (!can) return false;
  const int64_t blocks = p.goff != nullptr ? p.max_kb - p.E : p.max_kb;  // (the operands are padded to whole blocks per group)
  const int64_t tiles = ((p.Lrows + kLargeTile - 1) / kLargeTile) * ((p.Rrows + kLargeTile - 1) / kLargeTile), per_x = (tiles + 7) / 8;
  const int64_t group_rounds = (per_x + 31) / 32, rounds = (p.E * per_x + 31) / 32;
  const double full = (double)p.Lrows * (double)p.Rrows / (256.0 * kLargeTile * kLargeTile);  // rounds a group would fill
  if ((double)group_rounds > 1.15 * full || (double)rounds > 1.05 * p.E * full) return false;
  if (c_dtype == AAMD_F32) return blocks >= 16LL * p.E && rounds >= 24;
  return blocks >= 8LL * p.E || (p.E <= 8 && blocks >= 4LL * p.E);
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace aamd

using namespace aamd;

// b_rows: b is [E, K, N], b_s [E, K/128, N/128] (see R_ROWS); block scales only.
static int gemm_nt_impl(const uint8_t* a, int64_t lda, const float* a_s, const uint8_t* b, const float* b_s,
                        int b_tile_scaled, bool b_rows, const int64_t* group_offsets, int E, int64_t M, int64_t N, int64_t K, void* c,
                        int c_dtype, int64_t ldc, const void* bias, int bias_dtype, void* stream,
                        const GemmOptions& g_opt = GemmOptions(), float* ws = nullptr) {
  AAMD_REQUIRE(c_dtype == AAMD_BF16 || c_dtype == AAMD_F32, "grouped_gemm_nt: unsupported output dtype %d", c_dtype);
  AAMD_REQUIRE(M >= 0 && N >= 0 && K >= 0, "grouped_gemm_nt: negative size");
  AAMD_REQUIRE(K % kBK == 0 && N % kTile == 0, "grouped_gemm_nt: K=%lld and N=%lld must be multiples of 128",
               (long long)K, (long long)N);
  AAMD_REQUIRE(E >= 1, "grouped_gemm_nt: E must be >= 1");
  AAMD_REQUIRE(group_offsets != nullptr || E == 1, "grouped_gemm_nt: group_offsets required when E > 1");
  AAMD_REQUIRE(bias == nullptr || bias_dtype == AAMD_BF16 || bias_dtype == AAMD_F32, "grouped_gemm_nt: bad bias dtype");
  if (M == 0 || N == 0) return AAMD_OK;
  AAMD_REQUIRE(a && a_s && b && b_s && c, "grouped_gemm_nt: null pointer");
  AAMD_REQUIRE(lda >= K && lda % 16 == 0 && aligned16(a) && aligned16(b), "grouped_gemm_nt: operands must be 16-byte aligned");
  AAMD_REQUIRE(ldc >= N && (ldc * (c_dtype == AAMD_BF16 ? 2 : 4)) % 16 == 0 && aligned16(c),
               "grouped_gemm_nt: output rows must be 16-byte aligned");
  AAMD_REQUIRE(K > 0, "grouped_gemm_nt: K must be positive");
  AAMD_REQUIRE(lda < (1LL << 23) && K < (1LL << 23) && (!b_rows || N < (1LL << 23)), "grouped_gemm_nt: row stride too large");
  hipStream_t st = (hipStream_t)stream;
  // scale batches of eight contraction blocks; their 16-byte loads need aligned rows and whole groups of four blocks
  const bool batches = (K / kBK) >= 8 && g_opt.ls_batch != 0;
  const bool batches16 = batches && (K / kBK) % 4 == 0 && aligned16(a_s);
  const NtKernel kernel = b_tile_scaled ? (use_large_tiles(((M + 255) / 256 + (group_offsets ? E : 0)) * ((N + 255) / 256), g_opt) ? kLargeTiles : kSmallTiles)
                                        : choose_nt(M, N, K / kBK, E, group_offsets != nullptr, b_rows, ws != nullptr, c_dtype, g_opt);
  // (output rows of 8 M elements are out of reach of the large tiles' 32-bit offsets)
  const bool once = kernel == kLargeOnce && !b_tile_scaled;
  const bool large = once || ((kernel == kLargeTiles || kernel == kLargeShared || kernel == kLargeMore) && (b_tile_scaled || ldc < (1LL << 23)));
  const int BM = large ? kLargeTile : CfgSmall::BM;
  const int BN = large ? (b_tile_scaled ? CfgWgrad::BN : kLargeTile) : CfgSmall::BN;
  static_assert(CfgWgrad::BM == kLargeTile, "L rows of a large tile");
  GemmParams p = {};
  p.L = a; p.ldl = lda; p.Ls = a_s; p.ls_row_stride = K / kBK; p.ls_blk_stride = 1;
  p.l_kb_stride = p.r_kb_stride = kBK;
  // 1: batches by 16-byte loads; 2 (256x256 tiles only): by 4-byte loads
  p.ls_batch = large && !b_tile_scaled ? (batches16 && aligned16(b_s) ? 1 : 2) : (batches16 ? 1 : 0);
  p.R = b; p.ldr = K; p.r_group_stride = N * K;
  p.Rs = b_s;
  p.rs_row_stride = K / kBK; p.rs_blk_stride = 1;
  p.rs_group_stride = b_tile_scaled ? N * (K / kBK) : (N / kTile) * (K / kBK);
  if (b_rows) {
    p.ldr = N; p.r_kb_stride = N * kBK;
    p.rs_row_stride = 1; p.rs_blk_stride = N / kTile;
  }
  p.C = c; p.ldc = ldc; p.c_group_stride = 0;
  p.bias = bias; p.bias_dtype = bias_dtype; p.bias_group_stride = N;
  p.goff = group_offsets;
  p.Lrows = M; p.Rrows = N; p.nkb = (int)(K / kBK); p.E = E; p.nRt = (int)((N + BN - 1) / BN); p.nLt = 0;
  p.accumulate = 0;
  if (is_few_rows(kernel)) return launch_few_rows(p, c_dtype, M, few_rows_waves(kernel), b_rows, st);
  const int64_t max_lt = group_offsets ? M / BM + E : (M + BM - 1) / BM;
  const int64_t blocks = max_lt * p.nRt;
  if (once)
    return b_rows ? launch_gemm<kRaggedRows, false, CfgLarge, true>(p, c_dtype, blocks, st, g_opt)
                  : launch_gemm<kRaggedRows, false, CfgLarge>(p, c_dtype, blocks, st, g_opt);
  if (large && !b_tile_scaled) {
    tile_order<kRaggedRows>(p, kLargeTile, g_opt);
    p.slices = takes_slices(p);
    p.higher = g_opt.tile >= 0 ? (kernel == kLargeMore ? 1 : -1) : choose_higher(p, ws != nullptr);
    p.ws = ws;
    p.max_split = ws != nullptr ? row_max_split(p.nkb) : 1;
    return launch_row_tiles(p, c_dtype, blocks, b_rows, st);
  }
  if (b_rows) return launch_gemm<kRaggedRows, false, CfgSmall, true>(p, c_dtype, blocks, st, g_opt);
  if (large) return launch_gemm<kRaggedRows, true, CfgWgrad>(p, c_dtype, blocks, st, g_opt);
  return b_tile_scaled ? launch_gemm<kRaggedRows, true, CfgSmall>(p, c_dtype, blocks, st, g_opt)
                       : launch_gemm<kRaggedRows, false, CfgSmall>(p, c_dtype, blocks, st, g_opt);
}

#ifndef AAMD_TUNING
extern "C" int aamd_grouped_gemm_fp8_nt(const uint8_t* a, int64_t lda, const float* a_s, const uint8_t* b,
                                        const float* b_s, int b_tile_scaled, const int64_t* group_offsets, int E,
                                        int32_t* /*tile_ws*/, int64_t M, int64_t N, int64_t K, void* c, int c_dtype,
                                        int64_t ldc, const void* bias, int bias_dtype, void* stream) {
  return gemm_nt_impl(a, lda, a_s, b, b_s, b_tile_scaled, false, group_offsets, E, M, N, K, c, c_dtype, ldc, bias, bias_dtype,
                      stream);
}

// The same GEMM without a workspace argument.  (Neither form uses one: the kernels find their group in the offsets
// themselves.  The limit on the groups is the entry point's contract.)
extern "C" int aamd_grouped_gemm_fp8_nt_static(const uint8_t* a, int64_t lda, const float* a_s, const uint8_t* b,
                                               const float* b_s, int b_tile_scaled, const int64_t* group_offsets,
                                               int E, int64_t M, int64_t N, int64_t K, void* c, int c_dtype,
                                               int64_t ldc, const void* bias, int bias_dtype, void* stream) {
  AAMD_REQUIRE(E >= 1 && E <= AAMD_STATIC_MAX_GROUPS, "grouped_gemm_nt_static: E=%d exceeds the limit of %d groups (no static scratch is behind it; it is the entry point's contract)",
               E, AAMD_STATIC_MAX_GROUPS);
  return gemm_nt_impl(a, lda, a_s, b, b_s, b_tile_scaled, false, group_offsets, E, M, N, K, c, c_dtype, ldc, bias, bias_dtype,
                      stream);
}

extern "C" int aamd_grouped_gemm_fp8_nn(const uint8_t* a, int64_t lda, const float* a_s, const uint8_t* b, const float* b_s,
                                        const int64_t* group_offsets, int E, int64_t M, int64_t N, int64_t K, void* c,
                                        int c_dtype, int64_t ldc, const void* bias, int bias_dtype, void* stream) {
  return gemm_nt_impl(a, lda, a_s, b, b_s, 0, true, group_offsets, E, M, N, K, c, c_dtype, ldc, bias, bias_dtype, stream);
}

constexpr int64_t kQuantisingRows = 64;
static NtKernel quantising_kernel(int64_t M, int64_t N, int64_t K, int E) {
  if (M < 1 || M > kQuantisingRows || N < kTile || K < kBK || N % kTile != 0 || K % kBK != 0 || E < 1 || K >= (1LL << 23)) return kSmallTiles;
  return choose_nt(M, N, K / kBK, E, true, false, false, AAMD_BF16, GemmOptions());
}
// Workgroups of `rows` weight rows over the places of 512, where every row may have its own group.
static double few_rows_rounds(int64_t M, int64_t N, int E, int rows) {
  return std::max(1.0, (double)((M < E ? M : E) * (N / rows)) / 512.0);
}
// Worth it?  It saves a launch of 3 to 4 us and puts a tenth of a microsecond into every step of every round of workgroups, four
// rows of a group at a time; from the ninth row on the rows of a step are fetched when their turn comes.  A block of experts,
// SwiGLU, us, with both of its quantisers as launches -> in the GEMMs (E, H, F, k; T tokens): 60, 2048, 1408, 4: T 1 30.1 -> 22.3,
// 2 31.0 -> 24.9, 4 39.5 -> 34.0, 8 50.7 -> 47.8; 64, 7168, 2048, 8: T 1 85.4 -> 79.7, 4 230 -> 226; 8, 4096, 14336, 2 (long
// streams: 40 and more steps): T 1 75.8 -> 72.0, 4 219 -> 225, 8 242 -> 251, 16 247 -> 316; one group of 32 rows, 1024 x 4096
// 28.7 -> 49.2.
extern "C" int aamd_quant_grouped_gemm_fits(int64_t M, int64_t N, int64_t K, int E, int64_t most) {
  const NtKernel kernel = quantising_kernel(M, N, K, E);
  if (!is_few_rows(kernel)) return 0;
  const int64_t nkb = K / kBK;
  const int waves = kernel == kFewRowsSplit ? 8 : 4, rows = kernel == kFewRowsSplit ? 32 : 64;  // (fewer waves: as many more places)
  return most <= 8 && few_rows_rounds(M, N, E, rows) * (double)((nkb + waves - 1) / waves) <= 24.0;
}
static GemmParams quantising_params(const uint8_t* b, const float* b_s, const int64_t* group_offsets, int E, int64_t M, int64_t N,
                                    int64_t K, void* c, int64_t ldc, const void* bias, int bias_dtype) {
  GemmParams p = {};
  p.r_kb_stride = kBK;
  p.R = b; p.ldr = K; p.r_group_stride = N * K;
  p.Rs = b_s; p.rs_row_stride = K / kBK; p.rs_blk_stride = 1; p.rs_group_stride = (N / kTile) * (K / kBK);
  p.C = c; p.ldc = ldc;
  p.bias = bias; p.bias_dtype = bias_dtype; p.bias_group_stride = N;
  p.goff = group_offsets;
  p.Lrows = M; p.Rrows = N; p.nkb = (int)(K / kBK); p.E = E;
  return p;
}
extern "C" int aamd_quant_grouped_gemm_fp8_nt(int what, const void* rows, int64_t ld, const int64_t* sorted_idx, int topk, int64_t T,
                                              const uint8_t* b, const float* b_s, const int64_t* group_offsets, int E, int64_t M,
                                              int64_t N, int64_t K, void* c, int64_t ldc, const void* bias, int bias_dtype,
                                              void* stream) {
  AAMD_REQUIRE(what >= AAMD_ROWS_PERMUTED && what <= AAMD_ROWS_GELU, "quant_grouped_gemm_nt: unknown source %d", what);
  const NtKernel kernel = quantising_kernel(M, N, K, E);
  AAMD_REQUIRE(is_few_rows(kernel), "quant_grouped_gemm_nt: not for M=%lld, N=%lld, K=%lld in %d groups", (long long)M,
               (long long)N, (long long)K, E);
  AAMD_REQUIRE(bias == nullptr || bias_dtype == AAMD_BF16 || bias_dtype == AAMD_F32, "quant_grouped_gemm_nt: bad bias dtype");
  AAMD_REQUIRE(rows && b && b_s && c && group_offsets && (what != AAMD_ROWS_PERMUTED || (sorted_idx && topk >= 1 && T >= 1 && T < (1LL << 31))),
               "quant_grouped_gemm_nt: null pointer or bad routing");
  AAMD_REQUIRE(ld >= (what == AAMD_ROWS_SWIGLU ? 2 * K : K) && ld % 8 == 0 && aligned16(rows) && aligned16(b), "quant_grouped_gemm_nt: operands must be 16-byte aligned");
  AAMD_REQUIRE(ldc >= N && ldc % 8 == 0 && aligned16(c), "quant_grouped_gemm_nt: output rows must be 16-byte aligned");
  const GemmParams p = quantising_params(b, b_s, group_offsets, E, M, N, K, c, ldc, bias, bias_dtype);
  return launch_few_rows_quantising(p, what, rows, ld, sorted_idx, topk, T, M, few_rows_waves(kernel), (hipStream_t)stream);
}
// From the router's choices.  It saves the routing's launch, 3 us and its gap, and puts 0.3 us into every round of workgroups, which look
// among the choices for their pairs before they know their weights.  Routing and GEMM, replayed in a graph, us, two launches -> one
// (E, N, K, topk; T tokens): 60, 2816, 2048, 4: T 1 9.1 -> 6.7, 8 29.2 -> 27.8; 512, 1024, 2048, 8: T 8 41.6 -> 24.7; 1024, 512, 1024,
// 8: T 8 29.0 -> 9.9; 60, 16384, 512, 6: T 2 (6 rounds) 27.8 -> 27.3; 16, 28672, 1024, 4: T 2 (7) 39.7 -> 40.3; 32, 28672, 512, 4: T 3
// (10.5) 42.8 -> 44.2; 32, 16384, 512, 6: T 8 (16) 51.3 -> 54.3.  Other weights and choices in every launch (from memory): of 78 draws of
// two to five rounds none slower by 0.3 us and half of them faster by 2; 64, 6144, 1536, 8: T 4 (6) 51.6 -> 52.8; 64, 28672, 1024, 2: T 4
// (7) 49.0 -> 50.4.  (With a sort of the pairs in every wave, a loop over them for every 64 experts, 64 pairs took up to four times as
// long as with the launch: the block of 1024 experts 54 -> 228.)
constexpr double kRouteRounds = 5.0;  // (of 64 weight rows to a workgroup, also where the form of 32 is taken)
extern "C" int aamd_route_quant_grouped_gemm_fits(int64_t T, int topk, int64_t N, int64_t K, int E) {
  if (T < 1 || topk < 1 || T > kQuantisingRows || topk > kQuantisingRows || T * topk > kQuantisingRows || E > 1024) return 0;
  const int64_t M = T * topk;
  return aamd_quant_grouped_gemm_fits(M, N, K, E, T) &&  // (a token goes to an expert once)
         few_rows_rounds(M, N, E, 64) <= kRouteRounds;
}
extern "C" int aamd_route_quant_grouped_gemm_fp8_nt(const void* ids, int ids_are_i64, int topk, int64_t T, const void* rows, int64_t ld,
                                                    const uint8_t* b, const float* b_s, int E, int64_t N, int64_t K, void* c, int64_t ldc,
                                                    const void* bias, int bias_dtype, int64_t* sorted_idx, int32_t* row_map,
                                                    int64_t* group_offsets, void* stream) {
  AAMD_REQUIRE(topk >= 1 && T >= 1 && T <= kQuantisingRows && topk <= kQuantisingRows && E <= 1024, "route_quant_grouped_gemm_nt: bad routing");
  const int64_t M = T * topk;
  const NtKernel kernel = quantising_kernel(M, N, K, E);
  AAMD_REQUIRE(is_few_rows(kernel), "route_quant_grouped_gemm_nt: not for M=%lld, N=%lld, K=%lld in %d groups", (long long)M,
               (long long)N, (long long)K, E);
  AAMD_REQUIRE(bias == nullptr || bias_dtype == AAMD_BF16 || bias_dtype == AAMD_F32, "route_quant_grouped_gemm_nt: bad bias dtype");
  AAMD_REQUIRE(ids && rows && b && b_s && c && sorted_idx && row_map && group_offsets, "route_quant_grouped_gemm_nt: null pointer");
  AAMD_REQUIRE(ld >= K && ld % 8 == 0 && aligned16(rows) && aligned16(b), "route_quant_grouped_gemm_nt: operands must be 16-byte aligned");
  AAMD_REQUIRE(ldc >= N && ldc % 8 == 0 && aligned16(c), "route_quant_grouped_gemm_nt: output rows must be 16-byte aligned");
  const GemmParams p = quantising_params(b, b_s, nullptr, E, M, N, K, c, ldc, bias, bias_dtype);
  return launch_few_rows_routing(p, ids, ids_are_i64, rows, ld, topk, T, sorted_idx, row_map, group_offsets, few_rows_waves(kernel),
                                 (hipStream_t)stream);
}

// With the combine (few_rows_combine_kernel)?  It saves a launch and its gap, 2.5 us of a step that is queued launch by launch, and has a
// workgroup per token and 32 outputs, one per CU, where the GEMM alone has one per row and two per CU: what it loses is long chains of
// steps on few CUs, further rounds, and weights that several tokens share, which are read for each.  A chain of a few steps in one round
// is always taken: with two slots a wave has as many steps as in the GEMM alone, and else such a launch is hardly longer than its
// latencies (at most 0.7 us lost in a graph, the saved launch won where it bounds).  The others by estimates of both, us, fitted to 890
// launches of 4 to 256 experts, 512 x 256 to 7168 x 14336, that read their weights from the caches (11 and 9 % off), a microsecond apart.
// What the rule takes of these is faster by 2.7 us on average, 14 of 710 are slower by 0.2 to 1.8; with other weights in every launch, from
// memory, 2.8 of 223 and none is slower (up to sixteen steps were taken before: 58 of 329 slower there, 8, 4096, 14336, 2: T 1 28.3 ->
// 32.9).  SwiGLU, replayed in a graph, two launches -> one (E, N, K, topk; T tokens): 60, 2048, 1408, 4: T 1 7.1 -> 6.8, 8 21.0 -> 18.2;
// 8, 1024, 4096, 2: T 8 10.6 -> 8.4; 256, 512, 4096, 2: T 8 11.0 -> 8.0; 16, 512, 512, 8: T 1 7.0 -> 7.3; 4, 2048, 8192, 2: T 2 15.0 ->
// 16.8; not taken: 16, 512, 4096, 8: T 4 (16 steps) 11.3 -> 19.6; 8, 7168, 768, 2: T 4 (4 rounds) 12.9 -> 16.0.  The block of 60
// experts, one token, queued: 19.6 -> 16.5.
extern "C" int aamd_quant_grouped_gemm_combine_fits(int64_t T, int topk, int64_t N, int64_t K, int E) {
  if (T < 1 || T > kQuantisingRows || topk < 1 || topk > 8 || T * topk > kQuantisingRows) return 0;
  if (quantising_kernel(T * topk, N, K, E) != kFewRowsSplit) return 0;
  const int64_t per = topk <= 2 ? 8 : topk <= 4 ? 4 : 2;  // waves per slot: launch_combine
  const int64_t nkb = K / kBK, wgs = T * (N / 32), rounds = (wgs + 255) / 256, steps = (nkb + per - 1) / per;
  if (rounds == 1 && (steps <= 5 || (topk <= 2 && steps * wgs < 1024))) return 1;
  if (rounds > 2 || rounds * steps > 8) return 0;
  const double groups = E * (1.0 - std::pow(1.0 - std::min(1.0, (double)topk / E), (double)T));  // that a random routing reaches
  const double MB = (double)N * K * 1e-6, alone = groups * (N / 32) / 512.0, alone_rounds = std::ceil(alone), alone_steps = (double)((nkb + 7) / 8);
  const double one = 1.9 + rounds * (1.6 + 0.83 * steps * (per * topk) / 16.0) + 0.061 * T * topk * MB;
  const double two = 4.5 + alone_rounds * (0.95 + 0.55 * alone_steps) + 0.28 * alone * alone_steps + 0.096 * groups * MB + 20e-6 * T * topk * N;
  return one + 1.0 < two;
}
extern "C" int aamd_quant_grouped_gemm_combine_fp8_nt(int what, const void* rows, int64_t ld, const void* ids, int ids_are_i64,
                                                      const int32_t* row_map, const void* probs, int probs_dtype, int topk, int64_t T,
                                                      const uint8_t* b, const float* b_s, int E, int64_t N, int64_t K, void* out,
                                                      const void* bias, int bias_dtype, void* stream) {
  AAMD_REQUIRE(what == AAMD_ROWS_SWIGLU || what == AAMD_ROWS_GELU, "quant_grouped_gemm_combine: unknown source %d", what);
  AAMD_REQUIRE(T >= 1 && T <= kQuantisingRows && topk >= 1 && topk <= 8 && T * topk <= kQuantisingRows, "quant_grouped_gemm_combine: bad routing");
  AAMD_REQUIRE(E >= 1 && N >= kTile && N % kTile == 0 && K >= kBK && K % kBK == 0 && K < (1LL << 23), "quant_grouped_gemm_combine: bad sizes");
  AAMD_REQUIRE(probs_dtype == AAMD_BF16 || probs_dtype == AAMD_F32, "quant_grouped_gemm_combine: bad type of the router weights");
  AAMD_REQUIRE(bias == nullptr || bias_dtype == AAMD_BF16 || bias_dtype == AAMD_F32, "quant_grouped_gemm_combine: bad bias dtype");
  AAMD_REQUIRE(rows && ids && row_map && probs && b && b_s && out, "quant_grouped_gemm_combine: null pointer");
  AAMD_REQUIRE(ld >= (what == AAMD_ROWS_SWIGLU ? 2 * K : K) && ld % 8 == 0 && aligned16(rows) && aligned16(b), "quant_grouped_gemm_combine: operands must be 16-byte aligned");
  const GemmParams p = quantising_params(b, b_s, nullptr, E, T * topk, N, K, out, N, bias, bias_dtype);
  return launch_few_rows_combine(p, what, rows, ld, ids, ids_are_i64, row_map, probs, probs_dtype, topk, T, out, (hipStream_t)stream);
}

extern "C" int64_t aamd_grouped_gemm_fp8_ws_bytes(int64_t M, int64_t N, int64_t K, int E, int grouped, int b_rows) {
  const int64_t nkb = K / kBK;
  if (M <= 0 || N <= 0 || E < 1 || nkb < kSplitBlocks) return 0;
  // (the tiles of groups are counted on the device)
  const int64_t tiles = (M + kLargeTile - 1) / kLargeTile * ((N + kLargeTile - 1) / kLargeTile), left = (tiles + 7) / 8 % 32;
  if (!grouped && (left == 0 || left > 16)) return 0;
  return choose_nt(M, N, nkb, E, grouped != 0, b_rows != 0, true, AAMD_BF16, GemmOptions()) == kLargeShared ? kRowPartsBytes : 0;
}
extern "C" int aamd_grouped_gemm_fp8_ws(const uint8_t* a, int64_t lda, const float* a_s, const uint8_t* b, const float* b_s,
                                        int b_rows, const int64_t* group_offsets, int E, int64_t M, int64_t N, int64_t K, void* c,
                                        int c_dtype, int64_t ldc, const void* bias, int bias_dtype, float* ws, int64_t ws_bytes,
                                        void* stream) {
  AAMD_REQUIRE(ws == nullptr || (ws_bytes >= kRowPartsBytes && aligned16(ws)), "grouped_gemm_ws: the workspace needs %lld bytes, 16-byte aligned", (long long)kRowPartsBytes);
  return gemm_nt_impl(a, lda, a_s, b, b_s, 0, b_rows != 0, group_offsets, E, M, N, K, c, c_dtype, ldc, bias, bias_dtype, stream,
                      GemmOptions(), ws);
}
#endif  // !AAMD_TUNING

static int wgrad_impl(const uint8_t* dyt, const float* sdyt, const uint8_t* xt, const float* sxt, int64_t ld_t,
                      int q_t_layout, const int64_t* group_offsets, int E, int64_t N, int64_t K, void* dw,
                      int dw_dtype, int64_t expert_stride, int accumulate, void* stream,
                      const GemmOptions& g_opt = GemmOptions()) {
  AAMD_REQUIRE(dw_dtype == AAMD_BF16 || dw_dtype == AAMD_F32, "grouped_gemm_wgrad: unsupported output dtype %d", dw_dtype);
  AAMD_REQUIRE(N >= 0 && K >= 0 && N % kTile == 0 && K % kTile == 0,
               "grouped_gemm_wgrad: N=%lld and K=%lld must be multiples of 128", (long long)N, (long long)K);
  AAMD_REQUIRE(E >= 1 && (group_offsets || E == 1), "grouped_gemm_wgrad: group_offsets required when E > 1");
  AAMD_REQUIRE(ld_t >= 0 && ld_t % kBK == 0, "grouped_gemm_wgrad: ld_t=%lld must be a multiple of 128", (long long)ld_t);
  AAMD_REQUIRE(ld_t < (1LL << 23), "grouped_gemm_wgrad: ld_t too large");
  AAMD_REQUIRE(q_t_layout == AAMD_QT_ROWS || q_t_layout == AAMD_QT_BLOCKED, "grouped_gemm_wgrad: unknown operand layout %d", q_t_layout);
  if (N == 0 || K == 0) return AAMD_OK;
  AAMD_REQUIRE(dw && (ld_t == 0 || (dyt && sdyt && xt && sxt)), "grouped_gemm_wgrad: null pointer");
  AAMD_REQUIRE(aligned16(dyt) && aligned16(xt) && aligned16(dw), "grouped_gemm_wgrad: pointers must be 16-byte aligned");
  AAMD_REQUIRE(expert_stride >= N * K && expert_stride % 4 == 0, "grouped_gemm_wgrad: bad expert stride");
  hipStream_t st = (hipStream_t)stream;
  GemmParams p = {};
  p.L = dyt; p.Ls = sdyt; p.ls_row_stride = 1; p.ls_blk_stride = N;
  p.R = xt; p.r_group_stride = 0;
  if (q_t_layout == AAMD_QT_BLOCKED) {  // [ld_t / 128, rows, 128]: a contraction block of all rows is one slab
    p.ldl = p.ldr = kBK;
    p.l_kb_stride = N * kBK; p.r_kb_stride = K * kBK;
  } else {
    p.ldl = p.ldr = ld_t;
    p.l_kb_stride = p.r_kb_stride = kBK;
  }
  p.Rs = sxt; p.rs_row_stride = 1; p.rs_blk_stride = K; p.rs_group_stride = 0;
  p.C = dw; p.ldc = K; p.c_group_stride = expert_stride;
  p.bias = nullptr; p.bias_dtype = AAMD_NONE; p.bias_group_stride = 0;
  p.goff = group_offsets;
  p.Lrows = N; p.Rrows = K; p.nkb = 0; p.E = E;
  p.max_kb = (int)(ld_t / kBK);
  p.accumulate = accumulate;
  if (use_large_wgrad(p, dw_dtype, g_opt)) {
    p.nLt = (int)((N + kLargeTile - 1) / kLargeTile); p.nRt = (int)((K + kLargeTile - 1) / kLargeTile);
    tile_order<kRaggedK>(p, kLargeTile, g_opt);
    return launch_wgrad_tiles(p, dw_dtype, st);
  }
  p.nLt = (int)(N / kTile); p.nRt = (int)(K / kTile);
  const int64_t per_g = (int64_t)p.nLt * p.nRt, per_x = (per_g + 7) / 8;  // every XCD takes an eighth of a group
  int64_t blocks = (int64_t)E * per_x * 8;
  if (g_opt.tile < 0 && use_short_runs(p)) {
    p.short_kb = kShortBlocks;
    p.zeroers = accumulate ? 0 : kZeroers;
    p.run = (int)std::min<int64_t>(dw_dtype == AAMD_F32 && !accumulate ? 2 : 4, std::max<int64_t>(1, E * per_g / kShortUnits));
    // long groups have more than short_kb blocks each, so that the operand buffers bound their number
    const int64_t longs = std::min<int64_t>(E, p.max_kb / (p.short_kb + 1));
    blocks = (longs * per_x + (E * per_g + 8 * p.run - 1) / (8 * p.run)) * 8 + p.zeroers;
  }
  return launch_gemm<kRaggedK, true, CfgSmall>(p, dw_dtype, blocks, st, g_opt);
}

#ifndef AAMD_TUNING
extern "C" int aamd_grouped_gemm_fp8_wgrad(const uint8_t* dyt, const float* sdyt, const uint8_t* xt,
                                           const float* sxt, int64_t ld_t, int q_t_layout,
                                           const int64_t* group_offsets, int E, int32_t* /*tile_ws*/, int64_t N,
                                           int64_t K, void* dw, int dw_dtype, int64_t expert_stride, int accumulate,
                                           void* stream) {
  return wgrad_impl(dyt, sdyt, xt, sxt, ld_t, q_t_layout, group_offsets, E, N, K, dw, dw_dtype, expert_stride, accumulate,
                    stream);
}
#else
// Measurement build (libatorch_amd_probes.so): the same two GEMMs with the launch choices pinned per call.
// opts = {tile, group_r, gl, ls_batch}, -1 = the library's own choice.
extern "C" int aamd_tuning_grouped_gemm_fp8_nt(const uint8_t* a, int64_t lda, const float* a_s, const uint8_t* b,
                                               const float* b_s, int b_tile_scaled, const int64_t* group_offsets,
                                               int E, int32_t* /*tile_ws*/, int64_t M, int64_t N, int64_t K, void* c,
                                               int c_dtype, int64_t ldc, const void* bias, int bias_dtype,
                                               const int* opts, void* stream) {
  AAMD_REQUIRE(opts != nullptr, "tuning_grouped_gemm_nt: null options");
  GemmOptions o;
  o.tile = opts[0]; o.group_r = opts[1]; o.gl = opts[2]; o.ls_batch = opts[3];
  return gemm_nt_impl(a, lda, a_s, b, b_s, b_tile_scaled, false, group_offsets, E, M, N, K, c, c_dtype, ldc, bias, bias_dtype,
                      stream, o);
}
extern "C" int aamd_tuning_grouped_gemm_choice(int64_t M, int64_t N, int64_t K, int E, int grouped, int b_rows, int workspace,
                                               int c_dtype, const int64_t* host_offsets) {
  if (M < 1 || N < kTile || K < kBK || N % kTile != 0 || K % kBK != 0 || E < 1 || (E > 1 && !grouped)) return -1;
  const NtKernel kernel = choose_nt(M, N, K / kBK, E, grouped != 0, b_rows != 0, workspace != 0, c_dtype, GemmOptions());
  if (kernel != kLargeTiles && kernel != kLargeShared) return kernel;
  GemmParams p = {};
  const int64_t none = 0;
  p.goff = grouped ? (host_offsets ? host_offsets : &none) : nullptr;
  p.Lrows = M; p.E = E; p.nRt = (int)((N + kLargeTile - 1) / kLargeTile);
  tile_order<kRaggedRows>(p, kLargeTile, GemmOptions());
  int higher = choose_higher(p, workspace != 0);
  if (higher == 0 && host_offsets != nullptr) {  // what higher_tiles of gemm_rows.hip counts
    uint32_t full = 0, own0 = 0, own1 = 0, shared = 0, longest = 0, of_xcd[8] = {};
    for (int e = 0; e < E; e++) {
      const uint32_t rows = (uint32_t)(host_offsets[e + 1] - host_offsets[e]), f = rows / kLargeTile, more = (rows % kLargeTile + 31) / 32;
      full += f;
      own0 += more > 0;
      own1 += more > f;
      shared += more > f ? 0 : more;
      const uint32_t tiles = (more > f ? f + 1 : f) * (uint32_t)p.nRt;
      for (int x = 0; x < 8; x++) of_xcd[x] += tiles / 8 + (uint32_t)((x + e) % 8 < (int)(tiles % 8));
    }
    for (uint32_t n : of_xcd) longest = std::max(longest, n);
    const uint32_t n1 = takes_slices(p) ? 8 * longest : (full + own1) * (uint32_t)p.nRt;
    higher = own0 != own1 && higher_tiles_pay(full, own0, own1, shared, (uint32_t)p.nRt, n1, workspace != 0 && row_max_split(K / kBK) > 1);
  }
  return higher > 0 ? kLargeMore : kernel;
}
extern "C" int aamd_tuning_grouped_gemm_fp8_nn(const uint8_t* a, int64_t lda, const float* a_s, const uint8_t* b,
                                               const float* b_s, const int64_t* group_offsets, int E, int64_t M, int64_t N,
                                               int64_t K, void* c, int c_dtype, int64_t ldc, const void* bias, int bias_dtype,
                                               const int* opts, void* stream) {
  AAMD_REQUIRE(opts != nullptr, "tuning_grouped_gemm_nn: null options");
  GemmOptions o;
  o.tile = opts[0]; o.group_r = opts[1]; o.gl = opts[2]; o.ls_batch = opts[3];
  return gemm_nt_impl(a, lda, a_s, b, b_s, 0, true, group_offsets, E, M, N, K, c, c_dtype, ldc, bias, bias_dtype, stream, o);
}
extern "C" int aamd_tuning_grouped_gemm_fp8_wgrad(const uint8_t* dyt, const float* sdyt, const uint8_t* xt,
                                                  const float* sxt, int64_t ld_t, int q_t_layout,
                                                  const int64_t* group_offsets, int E, int32_t* /*tile_ws*/, int64_t N,
                                                  int64_t K, void* dw, int dw_dtype, int64_t expert_stride,
                                                  int accumulate, const int* opts, void* stream) {
  AAMD_REQUIRE(opts != nullptr, "tuning_grouped_gemm_wgrad: null options");
  GemmOptions o;
  o.tile = opts[0]; o.group_r = opts[1]; o.gl = opts[2]; o.ls_batch = opts[3];
  return wgrad_impl(dyt, sdyt, xt, sxt, ld_t, q_t_layout, group_offsets, E, N, K, dw, dw_dtype, expert_stride,
                    accumulate, stream, o);
}
#endif
