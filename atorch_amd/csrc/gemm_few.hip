// Row-ragged block-scaled FP8 GEMM for groups of few rows (decoding, small batches, many experts).
//
// With at most a few dozen rows per group every weight byte is used once or twice, so the launch is bound by how fast
// the weights stream from HBM, and the tiles of gemm.hip are the wrong shape for that: they stage 128 or 256 token
// rows that are mostly not there, have one or two workgroups per CU with two steps of loads in flight, and a workgroup
// walks the whole contraction alone, which leaves most of the chip idle when few groups have rows or the output is
// small.  Here a wave takes 32 WTR weight rows x 32 WTL token rows, the waves of a workgroup split the contraction
// (wave w takes the 128-deep blocks w, w + W, ...) and add up through the LDS at the end.
// The arithmetic is that of gemm.hip: two chained v_mfma_f32_32x32x64_f8f6f4 per 128-deep block, the raw product folded
// into fp32 accumulators with the block's scales; only the order of the sum over blocks differs.
//
// Measured (us, the 128 x 128 tiles of gemm.hip -> here; weights beyond the last-level cache):
//   64 groups of 6 rows, 4096 x 7168 weights (1.88 GB)      358 -> 305  (6.2 TB/s; a stream that only reads: 7.1)
//   64 groups of 6 rows, 7168 x 2048 weights (0.94 GB)      183 -> 157
//   60 groups of 16 / 48 rows, 1408 x 2048 (0.17 GB)         49 -> 37 / 43
//   8 groups of 16 / 48 rows, 4096 x 14336 (0.47 GB)        119 -> 81 / 113
//   one group of 1 / 144 rows, 896 x 6016                    41 -> 9  (split form)
// From about 64 rows per group the operand reuse of the larger tiles wins.
#include "gemm.hpp"
#include "quant.hpp"

namespace aamd {

// Token rows that come as bf16 and are quantised by the waves that multiply them: read through a routing (BF16: row j is row
// sorted_idx[j] / topk of `rows`), or the activation of the rows as they are (GLU, GELU).
struct FewSource {
  const u16* rows;
  int64_t ld, gate_off;        // elements
  const int64_t* sorted_idx;
  uint32_t topk, T;
  // Choices: the router's choices of T tokens, at most 64 in all, and where the routing made of them is left
  const void* ids;
  int ids_are_i64;
  int64_t *sorted_out, *goff_out;
  int32_t* map_out;
};
constexpr int kCombineWaves = 16, kCombineSlots = 8;  // of few_rows_combine_kernel: the most waves of a workgroup, and slots of a token
struct Codes {};    // the token rows are codes
struct Choices {};  // BF16 rows whose routing is made here

// The tables of the router preprocess from the experts of the pairs, one to a lane (-1: none), and their places inside an expert.
template <int W>
__device__ __forceinline__ void leave_routing(const GemmParams& p, const FewSource& src, int choice, int place, int wave, int lane) {
  auto below = [&](uint32_t e) __attribute__((always_inline)) {  // pairs of experts below e
    int n = 0;
    for (int k = 0; k < (int)p.Lrows; k += 8)
#pragma unroll
      for (int u = 0; u < 8; u++) n += (uint32_t)__builtin_amdgcn_readlane(choice, k + u) < e ? 1 : 0;  // (no expert: above all)
    return n;
  };
  if (wave == W - 1) {
    const int row = below((uint32_t)choice) + place;
    if (lane < (int)p.Lrows) src.map_out[lane] = choice >= 0 ? row : -1;
    if (choice >= 0) src.sorted_out[row] = lane;
  }
  for (int first = wave * 64; first <= p.E; first += 64 * W) {
    const int n = below((uint32_t)(first + lane));
    if (first + lane <= p.E) src.goff_out[first + lane] = n;
  }
}

// W waves, tiles of 32 WTR weight rows x 32 WTL token rows.  R_ROWS: the weights are stored [contraction, Rrows] and read
// transposed from the LDS, as in gemm.hip; a block of them is 128 rows of BR bytes there.  That form takes whole cache lines
// of a row, 128 weight rows x 32 token rows (us, 64 and 32 weight rows x 64 and 32 token rows, 128 x 32 with three waves, with
// four, and the other orientation: 64 groups of 6 rows, 7168 x 2048 197, 260, 166, 167, 159; 4096 x 7168 350, 474, 324, 326,
// 307; 64 uneven groups of 128, 2048 x 7168 324, 817, 254, 253, 284), its scales in registers so that two workgroups of
// 80 KB fit a CU.
//
// IN: what the token rows are.  A launch of a few rows is as long as its latencies, and quantising the rows ahead of it is another
// one; here every wave quantises the 128-wide blocks of its own steps, four rows at a time, into its stage while its weights are on
// their way (one token, four of 60 experts, 2048 wide: quantiser 3.4 + GEMM 7.0 us, activation 2.6 + GEMM 6.0).  The arithmetic is
// that of quant_1x128_kernel: the same codes.
//
// Choices: with at most 64 (token, expert) pairs a lane holds one, and a workgroup needs no sort to find its tile: a few ballots name
// the pairs of every lane's expert, the first of which stands for the group, and count the rows before the group's.  They cost the same
// for any number of pairs and a few instructions more for twice the experts, in every wave of every workgroup, in place of a launch
// (route_small_kernel 3.1 us) and of a look at its tables.  The first workgroup leaves the tables for the launches that follow.
template <typename OUT, int W, int WTR, int WTL, bool R_ROWS, typename IN = Codes>
__global__ __launch_bounds__(64 * W) void few_rows_kernel(const GemmParams p, const FewSource src) {
  constexpr bool kQuantise = !std::is_same<IN, Codes>::value;
  constexpr bool kChoices = std::is_same<IN, Choices>::value, kPermuted = kChoices || std::is_same<IN, BF16>::value;
  constexpr int BL = 32 * WTL, BR = 32 * WTR;
  constexpr int kPitch = BR + 4;  // floats per row of a wave's partial result in the LDS
  constexpr int kStage = (BR + BL) * kBK + (WTL == 1 && !kQuantise ? 0 : BL * 4 + 256);  // weight rows, token rows, scales
  constexpr int PL = WTR > 2 ? 32 : BL;  // token rows whose partial results are in the LDS at a time
  constexpr int kLds = W * (kStage > PL * kPitch * 4 ? kStage : PL * kPitch * 4);
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  float (*const part)[PL][kPitch] = reinterpret_cast<float (*)[PL][kPitch]>(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hg = lane >> 5;

  // ---- which tile: groups in order, inside a group the token tiles of one weight tile follow each other (they share
  // the weights), every XCD a contiguous range
  GroupRanges gr = {};
  int total = (int)((p.Lrows + BL - 1) / BL);
  int choice = -1, place = 0;  // (kChoices) lane i: the expert of pair i, -1 if there is none, and its place among the expert's pairs
  if constexpr (kChoices) {
    if (lane < (int)p.Lrows) {
      const int64_t e = src.ids_are_i64 ? ((const int64_t*)src.ids)[lane] : (int64_t)((const int32_t*)src.ids)[lane];
      choice = e >= 0 && e < p.E ? (int)e : -1;
    }
    unsigned long long same = __ballot(choice >= 0);  // the pairs of this lane's expert
    for (int b = 0; (p.E - 1) >> b != 0; b++) {
      const bool on = (choice >> b) & 1;
      const unsigned long long with = __ballot(on);
      same &= on ? with : ~with;
    }
    place = __popcll(same & ((1ull << lane) - 1ull));
    if (blockIdx.x == 0) {
      leave_routing<W>(p, src, choice, place, wave, lane);
      return;
    }
    const int n = choice >= 0 && place == 0 ? (__popcll(same) + BL - 1) / BL : 0;
    gr.t_hi = wave_inclusive_sum(n);
    gr.t_lo = gr.t_hi - n;
    total = __builtin_amdgcn_readlane(gr.t_hi, 63);
  } else if (p.goff != nullptr) {
    gr = group_ranges<BL>(p.goff, p.E, 0, 0);
    total = gr.total;
    for (int base = 64; base < p.E; base += 64) total = group_ranges<BL>(p.goff, p.E, base, total).total;
  }
  const int64_t ntot = (int64_t)total * p.nRt, bid = (int64_t)blockIdx.x - (kChoices ? 1 : 0);
  if (bid >= ntot) return;
  const int64_t per = ntot / 8, rem = ntot % 8, xcd = bid % 8, idx = bid / 8;
  const int64_t pid = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
  int g = 0, rt, lvalid, order = 0, order_at = 0;  // (kChoices) lane i: the i-th pair of the group; that of the tile's first row
  int64_t l0;
  if (kChoices || p.goff != nullptr) {
    g = p.E;
    l0 = 0;
    rt = lvalid = 0;
    for (int base = 0; base < p.E; base += 64) {
      if constexpr (!kChoices) if (base > 0) gr = group_ranges<BL>(p.goff, p.E, base, gr.total);
      const unsigned long long hit = __ballot(pid >= (int64_t)gr.t_lo * p.nRt && pid < (int64_t)gr.t_hi * p.nRt);
      if (hit != 0) {
        const int at = __builtin_ctzll(hit);
        const int t_lo = __builtin_amdgcn_readlane(gr.t_lo, at), nl = __builtin_amdgcn_readlane(gr.t_hi, at) - t_lo;
        int64_t r_lo, r_hi;
        if constexpr (kChoices) {
          g = __builtin_amdgcn_readlane(choice, at);
          r_lo = __popcll(__ballot(choice >= 0 && choice < g));
          r_hi = r_lo + __popcll(__ballot(choice == g));
          // (every lane takes part: one that is switched off would receive nothing.  Where lanes are not of the group, pair 63 is none.)
          order = __builtin_amdgcn_ds_permute((choice == g ? place : 63) * 4, lane);
        } else {
          g = base + at;
          r_lo = readlane_i64(gr.r_lo, at);
          r_hi = readlane_i64(gr.r_hi, at);
        }
        const uint32_t pe = (uint32_t)(pid - (int64_t)t_lo * p.nRt);
        rt = (int)(pe / (uint32_t)nl);
        order_at = (int)(pe - (uint32_t)rt * (uint32_t)nl) * BL;
        l0 = r_lo + order_at;
        lvalid = r_hi - l0 < BL ? (int)(r_hi - l0) : BL;
        break;
      }
      if constexpr (kChoices) break;
    }
    if (g >= p.E) return;
  } else {
    rt = (int)(pid / total);
    l0 = (pid - (int64_t)rt * total) * BL;
    lvalid = p.Lrows - l0 < BL ? (int)(p.Lrows - l0) : BL;
  }
  g = __builtin_amdgcn_readfirstlane(g);
  rt = __builtin_amdgcn_readfirstlane(rt);
  lvalid = __builtin_amdgcn_readfirstlane(lvalid);
  l0 = uniform_i64(l0);
  const int r0 = rt * BR;

  // ---- operands: every wave stages its own blocks in its own part of the LDS, without barriers.
  // One direct-to-LDS instruction moves 8 rows x 128 bytes, whole cache lines; the 16-byte chunks of a row are
  // XOR-swizzled as in gemm.hip, so that fragment reads meet no bank twice.  (Loads straight into the matrix
  // instruction's registers touch 32 lines each, four times over: with enough of them in flight to cover the latency
  // the lines leave the 32 KB L1 in between and are fetched again.)  Token rows past the group's end are not
  // loaded beyond the last slab of eight that holds one, re-read the last row inside it, and are not stored.
  // One block in flight per wave, and two workgroups per CU, of 69.6 KB of LDS (8 waves) or, in the split form, 67.6 KB (16
  // waves): two or three blocks per wave measured no faster where the weights' stream is the bound (1.9 GB).
  const int nkb = p.nkb;
  uint8_t* const mine = lds + wave * kStage;
  const uint8_t* const Lb = p.L + uniform_i64(l0 * p.ldl);
  const uint8_t* const Rb = p.R + uniform_i64((int64_t)g * p.r_group_stride + (R_ROWS ? (int64_t)r0 : (int64_t)r0 * p.ldr));
  const int r8 = lane >> 3;
  const uint32_t chunk[2] = {(uint32_t)(((lane & 7) ^ r8) << 4), (uint32_t)(((lane & 7) ^ r8 ^ 1) << 4)};
  const uint32_t roff[2] = {(uint32_t)r8 * (uint32_t)p.ldr + chunk[0], (uint32_t)r8 * (uint32_t)p.ldr + chunk[1]};
  // (R_ROWS) the chunks of row k are XORed with twice its place among the eight rows that are read together, counted in
  // rows of 256 bytes
  constexpr int kChunks = BR / 16, kRowsPer1K = 1024 / BR, kRowsPer256 = 256 / BR;
  const uint32_t roff_t = (uint32_t)(lane / kChunks) * (uint32_t)p.ldr +
                          (uint32_t)((lane % kChunks) ^ (2 * (((lane / kChunks) & 7) / kRowsPer256))) * 16u;
  const int tr = (lane & 15) >> 1;
  uint32_t loff[4 * WTL];
#pragma unroll
  for (int n = 0; n < 4 * WTL; n++) {
    const int row = n * 8 + r8 < lvalid ? n * 8 + r8 : lvalid - 1;
    loff[n] = (uint32_t)row * (uint32_t)p.ldl + chunk[n & 1];
  }
  const int nl = (lvalid + 7) >> 3;  // slabs of token rows, >= 1
  // scales of a block: with 32 token rows in registers, requested ahead of the block, else [BL token rows][the weights' block]
  // in the stage
  const float* const rs = p.Rs + (int64_t)g * p.rs_group_stride + (int64_t)(r0 / kTile) * p.rs_row_stride;
  const float* sbase[(WTL + 1) / 2];
#pragma unroll
  for (int n = 0; n < (WTL + 1) / 2; n++) {
    const int row = WTL == 1 ? l32 : n * 64 + lane;
    sbase[n] = p.Ls + (l0 + (row < lvalid ? row : lvalid - 1)) * p.ls_row_stride;
  }
  float ls_next = 0.f, rs_next = 0.f;  // (WTL == 1)
  // (kQuantise) the first eight rows are requested with the weights; 16 lanes per row
  constexpr int kAhead = 2;
  typedef typename std::conditional<kQuantise && !kPermuted, IN, BF16>::type Elem;
  Raw8<Elem> raw[kAhead];
  const int q4 = lane >> 4, q16 = lane & 15;
  auto raw_row = [&](int r) __attribute__((always_inline)) {  // clamped to the rows there are
    const int in_tile = r < lvalid ? r : lvalid - 1;
    const int64_t row = l0 + in_tile;
    if constexpr (kPermuted) {
      uint32_t pair;
      if constexpr (kChoices) pair = (uint32_t)__builtin_amdgcn_ds_bpermute((order_at + in_tile) * 4, order);
      else pair = (uint32_t)src.sorted_idx[row];
      const uint32_t token = pair / src.topk;
      return src.rows + (int64_t)(token < src.T ? token : src.T - 1) * src.ld;
    } else {
      return src.rows + row * src.ld;
    }
  };
  auto request = [&](Raw8<Elem>& to, const u16* row, int k) __attribute__((always_inline)) {
    const u16* const from = row + k * kTile + q16 * 8;
    to.a = *reinterpret_cast<const v4i*>(from);
    if constexpr (std::is_same<IN, GLU>::value) to.b = *reinterpret_cast<const v4i*>(from + src.gate_off);
  };
  const u16* raw_at[kAhead] = {};
  if constexpr (kQuantise) {
#pragma unroll
    for (int u = 0; u < kAhead; u++) raw_at[u] = raw_row(4 * u + q4);
  }
  constexpr int kScales = (BR + BL) * kBK;  // offset in the stage
  const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)mine;
  auto load = [&](int k) __attribute__((always_inline)) {
    const uint8_t* const R = Rb + k * p.r_kb_stride;
    const uint8_t* const L = Lb + (int64_t)k * kBK;
    if constexpr (kQuantise) {
#pragma unroll
      for (int u = 0; u < kAhead; u++)
        if (u == 0 || 4 * u < lvalid) request(raw[u], raw_at[u], k);
      rs_next = rs[k * p.rs_blk_stride];
    } else if constexpr (WTL == 1) {
      ls_next = sbase[0][k];
      rs_next = rs[k * p.rs_blk_stride];
    }
#pragma unroll
    for (int n = 0; n < BR / 8; n++)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(R_ROWS ? roff_t : roff[n & 1]), "s"(R + (int64_t)(n * (R_ROWS ? kRowsPer1K : 8)) * p.ldr), "s"(base + n * 1024) : "memory");
#pragma unroll
    for (int n = 0; n < (kQuantise ? 0 : 4 * WTL); n++)
      if (n < nl)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(loff[n]), "s"(L), "s"(base + BR * kBK + n * 1024) : "memory");
    if constexpr (WTL > 1 && !kQuantise) {
#pragma unroll
      for (int n = 0; n < (WTL + 1) / 2; n++)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(sbase[n] + k), "s"(base + kScales + n * 256) : "memory");
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(rs + k * p.rs_blk_stride), "s"(base + kScales + BL * 4) : "memory");
    }
  };
  v16f acc[WTR][WTL], zero;
#pragma unroll
  for (int r = 0; r < 16; r++) zero[r] = 0.f;
#pragma unroll
  for (int i = 0; i < WTR; i++)
#pragma unroll
    for (int j = 0; j < WTL; j++) acc[i][j] = zero;
  const int sw = (l32 & 7) ^ ((l32 >> 3) & 1);
  if (wave < nkb) load(wave);
  for (int kb = wave; kb < nkb; kb += W) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the block has landed
    const float rs_now = rs_next;
    if constexpr (kQuantise) {
      auto quantise = [&](const Raw8<Elem>& from, int row) __attribute__((always_inline)) {
        float v[8];
        from.get(v);
        const Divider d = make_scale(row16_max(amax8(v)), 0.f, false);
        const v2i codes = quant8<false>(v, d);
        if (row < lvalid) {
          uint8_t* const to = mine + (BR + row) * kBK + (((q16 >> 1) ^ ((row & 7) ^ ((row >> 3) & 1))) << 4) + (q16 & 1) * 8;
          *reinterpret_cast<v2i*>(to) = codes;
          if (q16 == 0) *reinterpret_cast<float*>(mine + kScales + row * 4) = d.s;
        }
      };
#pragma unroll
      for (int u = 0; u < kAhead; u++)
        if (u == 0 || 4 * u < lvalid) quantise(raw[u], 4 * u + q4);
      for (int r = 4 * kAhead; r < lvalid; r += 4) {
        Raw8<Elem> more;
        request(more, raw_row(r + q4), kb);
        quantise(more, r + q4);
      }
      __builtin_amdgcn_wave_barrier();  // same wave, in-order LDS: the reads below see the writes above
    }
    v8i rf[WTR][2], lf[WTL][2];
    float sc[WTL];
    auto frag = [&](const uint8_t* row, int h) {
      const v4i lo = *reinterpret_cast<const v4i*>(row + (((4 * h + 2 * hg) ^ sw) << 4));
      const v4i hi = *reinterpret_cast<const v4i*>(row + (((4 * h + 2 * hg + 1) ^ sw) << 4));
      return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    const float* const S = reinterpret_cast<const float*>(mine + kScales);
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int j = 0; j < WTL; j++) lf[j][h] = frag(mine + (BR + j * 32 + l32) * kBK, h);
#pragma unroll
      for (int i = 0; i < WTR; i++) {
        if constexpr (R_ROWS) {
          const uint32_t at = base + (uint32_t)((64 * h + 32 * hg + tr) * BR + (((2 * i + ((lane >> 4) & 1)) ^ (2 * (tr / kRowsPer256))) << 4) + (lane & 1) * 8);
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const v2i o = lds_read_transposed(at + (uint32_t)(8 * j * BR));
            rf[i][h][2 * j] = o[0];
            rf[i][h][2 * j + 1] = o[1];
          }
        } else {
          rf[i][h] = frag(mine + (i * 32 + l32) * kBK, h);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < WTL; j++) sc[j] = kQuantise ? S[j * 32 + l32] * rs_now : WTL == 1 ? ls_next * rs_next : S[j * 32 + l32] * S[BL];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and has been read: its place may be filled again
    if (kb + W < nkb) load(kb + W);
#pragma unroll
    for (int i = 0; i < WTR; i++)
#pragma unroll
      for (int j = 0; j < WTL; j++) {
        v16f pr = mfma_fp8_32x32x64(rf[i][0], lf[j][0], zero);
        pr = mfma_fp8_32x32x64(rf[i][1], lf[j][1], pr);
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = __builtin_fmaf(pr[r], sc[j], acc[i][j][r]);
      }
  }
  __syncthreads();  // every wave is done with its stages: the memory holds the partial results now

  // ---- sum over the waves, through the LDS; a lane holds column l32 and rows 8q + 4hg .. + 3 of every 32 x 32 sub-tile
  // (with 128 weight rows 32 token rows at a time, which fit the stages' memory)
  static_for<BL / PL>([&](auto J0) {
    constexpr int j0 = decltype(J0)::value * (PL / 32);
    if (j0 > 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < WTR; i++)
#pragma unroll
      for (int j = 0; j < PL / 32; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const v16f& a = acc[i][j0 + j];
          *reinterpret_cast<v4f*>(&part[wave][j * 32 + l32][i * 32 + 8 * q + 4 * hg]) = v4f{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
        }
    __syncthreads();
    for (int c = tid; c < PL * (BR / 4); c += 64 * W) {
      const int prow = c / (BR / 4), row = j0 * 32 + prow, col = (c % (BR / 4)) * 4;
      if (row >= lvalid) break;  // (rows only grow with c)
      v4f o = *reinterpret_cast<const v4f*>(&part[0][prow][col]);
#pragma unroll
      for (int w = 1; w < W; w++) o += *reinterpret_cast<const v4f*>(&part[w][prow][col]);
      if (p.bias != nullptr) {
        const int64_t at = (int64_t)g * p.bias_group_stride + r0 + col;
        if (p.bias_dtype == AAMD_F32) {
          o += *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(p.bias) + at);
        } else {
          const v2i raw = *reinterpret_cast<const v2i*>(reinterpret_cast<const u16*>(p.bias) + at);
          o += v4f{bf16_bits_to_f32((uint32_t)raw[0] & 0xffffu), bf16_bits_to_f32((uint32_t)raw[0] >> 16),
                   bf16_bits_to_f32((uint32_t)raw[1] & 0xffffu), bf16_bits_to_f32((uint32_t)raw[1] >> 16)};
        }
      }
      OUT* const dst = reinterpret_cast<OUT*>(p.C) + (l0 + row) * p.ldc + r0 + col;
      if constexpr (sizeof(OUT) == 4) {
        *reinterpret_cast<v4f*>(dst) = o;
      } else {
        *reinterpret_cast<v2i*>(dst) = v2i{(int)pack_bf16x2(o[0], o[1]), (int)pack_bf16x2(o[2], o[3])};
      }
    }
  });
}

// Upper bound of the token tiles of M rows in E groups (the groups' sizes are known on the device only).
static int64_t few_rows_tiles(int64_t M, int E, int rows) {
  const int64_t groups = M < E ? M : E;
  return M / rows + groups < M ? M / rows + groups : M;
}

template <typename OUT, int W, int WTR, int WTL, bool R_ROWS, typename IN = Codes>
static int launch_few(GemmParams p, int64_t M, hipStream_t st, const FewSource& src = FewSource()) {
  p.nRt = (int)(p.Rrows / (32 * WTR));
  const int64_t lt = p.goff || src.ids ? few_rows_tiles(M, p.E, 32 * WTL) : (M + 32 * WTL - 1) / (32 * WTL);
  const int64_t blocks = lt * p.nRt + (std::is_same<IN, Choices>::value ? 1 : 0);
  AAMD_REQUIRE(blocks < 0x7fffffffLL, "grouped_gemm: grid too large");
  few_rows_kernel<OUT, W, WTR, WTL, R_ROWS, IN><<<dim3((unsigned)blocks), dim3(64 * W), 0, st>>>(p, src);
  AAMD_LAUNCH_CHECK("grouped_gemm (few rows)");
  return AAMD_OK;
}

// `waves`: eight in the split form for launches of few workgroups, which takes half the weight rows and token rows per workgroup; four;
// two or one for many workgroups of a short contraction (see choose_nt).
template <typename OUT, typename IN>
static int launch_few_as(const GemmParams& p, int64_t M, int waves, hipStream_t st, const FewSource& src = FewSource()) {
  switch (waves) {
    case 8: return launch_few<OUT, 8, 1, 1, false, IN>(p, M, st, src);
    case 2: return launch_few<OUT, 2, 2, 2, false, IN>(p, M, st, src);
    case 1: return launch_few<OUT, 1, 2, 2, false, IN>(p, M, st, src);
    default: return launch_few<OUT, 4, 2, 2, false, IN>(p, M, st, src);
  }
}
int launch_few_rows(const GemmParams& p, int c_dtype, int64_t M, int waves, bool r_rows, hipStream_t st) {
  if (r_rows) return c_dtype == AAMD_BF16 ? launch_few<u16, 4, 4, 1, true>(p, M, st) : launch_few<float, 4, 4, 1, true>(p, M, st);
  return c_dtype == AAMD_BF16 ? launch_few_as<u16, Codes>(p, M, waves, st) : launch_few_as<float, Codes>(p, M, waves, st);
}

int launch_few_rows_quantising(const GemmParams& p, int what, const void* rows, int64_t ld, const int64_t* sorted_idx, int topk, int64_t T,
                               int64_t M, int waves, hipStream_t st) {
  FewSource src = {};
  src.rows = (const u16*)rows; src.ld = ld; src.gate_off = (int64_t)p.nkb * kTile;
  src.sorted_idx = sorted_idx; src.topk = (uint32_t)topk; src.T = (uint32_t)T;
  if (what == AAMD_ROWS_PERMUTED) return launch_few_as<u16, BF16>(p, M, waves, st, src);
  return what == AAMD_ROWS_SWIGLU ? launch_few_as<u16, GLU>(p, M, waves, st, src) : launch_few_as<u16, GELU>(p, M, waves, st, src);
}
int launch_few_rows_routing(const GemmParams& p, const void* ids, int ids_are_i64, const void* rows, int64_t ld, int topk, int64_t T,
                            int64_t* sorted_idx, int32_t* row_map, int64_t* goff, int waves, hipStream_t st) {
  FewSource src = {};
  src.rows = (const u16*)rows; src.ld = ld; src.topk = (uint32_t)topk; src.T = (uint32_t)T;
  src.ids = ids; src.ids_are_i64 = ids_are_i64; src.sorted_out = sorted_idx; src.map_out = row_map; src.goff_out = goff;
  return launch_few_as<u16, Choices>(p, p.Lrows, waves, st, src);
}

// The second GEMM of a decoding step with the weighted combine in it: out[t] = sum over the slots j of probs[t, j] (b[e_j] act(row_j)),
// e_j the expert of slot j and row_j its row of `rows`.  A step of one token is a chain of launches of a few microseconds each, and
// the combine, a gather of topk rows, was the last of them.  A workgroup takes 32 outputs of one token, eight, four or two waves
// (`per`) for a slot; the blocks of the contraction are dealt to eight sums like those of the eight waves of few_rows_kernel's split
// form, a wave makes some of these one after the other, two blocks in flight, and they are added in its order, the slots in that of
// unpermute_combine_kernel: the same bits as of the two launches.  Bound by latency: a wave's steps behind each other, and the fetch of
// the routing ahead.
// A wave quantises four of its blocks at a time, 16 lanes each.  With one at a time, in all lanes alike, the vector unit bound it (us,
// one token: four of 60 experts, 2048 x 1408 9.5 -> 8.0; two of 8, 1024 x 4096 9.6 -> 7.2), and 8 or 16 outputs per workgroup, which
// quantise the same rows more often, took longer still.
// IN: GLU or GELU.  PD: type of the router weights, and of the output.
template <typename IN, int PD>
__global__ __launch_bounds__(1024) void few_rows_combine_kernel(const GemmParams p, const FewSource src, const int32_t* __restrict__ row_map,
                                                                const void* __restrict__ probs, void* __restrict__ out, int per) {
#pragma clang fp contract(off)
  constexpr int BR = 32, kSums = 8, kStages = 2, kBatch = 4;
  constexpr int kCodes = kStages * BR * kBK, kWave = kCodes + kBatch * kBK + 256;  // stages of weight rows, codes and scales of the token row
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kCombineWaves * kWave];
  __shared__ __attribute__((aligned(16))) float part[kCombineSlots][kSums][BR];
  __shared__ float weight[kCombineSlots];
  __shared__ int expert[kCombineSlots];  // -1: a dropped copy, which adds zeros
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hg = lane >> 5, r8 = lane >> 3, q4 = lane >> 4, q16 = lane & 15;
  const int topk = (int)src.topk, slot = wave / per, first = wave - slot * per;
  const uint32_t t = blockIdx.x / (uint32_t)p.nRt;
  const int r0 = (int)(blockIdx.x - t * (uint32_t)p.nRt) * BR;
  const int64_t pair = (int64_t)t * topk + slot, id = src.ids_are_i64 ? ((const int64_t*)src.ids)[pair] : (int64_t)((const int32_t*)src.ids)[pair];
  const int to = row_map[pair];
  const float pv = PD == AAMD_BF16 ? bf16_bits_to_f32(reinterpret_cast<const u16*>(probs)[pair]) : reinterpret_cast<const float*>(probs)[pair];
  const int row = __builtin_amdgcn_readfirstlane(to >= 0 && to < p.Lrows && id >= 0 && id < p.E ? to : -1);
  const int e = __builtin_amdgcn_readfirstlane(row >= 0 ? (int)id : 0);

  v16f zero;
#pragma unroll
  for (int r = 0; r < 16; r++) zero[r] = 0.f;
  // a lane holds rows 8 q + 4 hg .. + 3 of 32, the same in every column
  auto keep = [&](int i, const v16f& a) __attribute__((always_inline)) {
    if (l32 != 0) return;
#pragma unroll
    for (int q = 0; q < BR / 8; q++)
      *reinterpret_cast<v4f*>(&part[slot][i][8 * q + 4 * hg]) = v4f{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
  };
  if (row >= 0) {
    uint8_t* const mine = lds + wave * kWave;
    uint8_t* const codes = mine + kCodes;
    float* const scales = reinterpret_cast<float*>(codes + kBatch * kBK);
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)mine;
    const uint8_t* const Rb = p.R + uniform_i64((int64_t)e * p.r_group_stride + (int64_t)r0 * p.ldr);
    const float* const rs = p.Rs + (int64_t)e * p.rs_group_stride + (int64_t)(r0 / kTile) * p.rs_row_stride;
    const u16* const from = src.rows + (int64_t)row * src.ld + q16 * 8;
    // (16-byte chunks XOR-swizzled as in few_rows_kernel)
    const uint32_t roff[2] = {(uint32_t)r8 * (uint32_t)p.ldr + (uint32_t)(((lane & 7) ^ r8) << 4),
                              (uint32_t)r8 * (uint32_t)p.ldr + (uint32_t)(((lane & 7) ^ r8 ^ 1) << 4)};
    const int sw = (l32 & 7) ^ ((l32 >> 3) & 1);
    const int nkb = p.nkb;
    float rs_now = 0.f, rs_next = 0.f;
    uint32_t stage = 0;  // of the block under way
    constexpr uint32_t kStage = BR * kBK, kRing = kStages * kStage - 1;
    auto request = [&](int k, uint32_t at) __attribute__((always_inline)) {
      rs_next = rs[k];
      const uint8_t* const R = Rb + (int64_t)k * kBK;
#pragma unroll
      for (int n = 0; n < BR / 8; n++)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(roff[n & 1]), "s"(R + (int64_t)(n * 8) * p.ldr), "s"(base + at + n * 1024) : "memory");
    };
    // the blocks of this wave: those of one sum after the other
    auto after = [&](int k) __attribute__((always_inline)) {
      const int next = k + kSums;
      return k >= nkb ? nkb : next < nkb ? next : (k & (kSums - 1)) + per < kSums && (k & (kSums - 1)) + per < nkb ? (k & (kSums - 1)) + per : nkb;
    };
    // the token row's codes of four blocks, 16 lanes each
    auto quantise = [&](int k) __attribute__((always_inline)) {
      const int k1 = after(k), k2 = after(k1), k3 = after(k2), theirs = q4 == 0 ? k : q4 == 1 ? k1 : q4 == 2 ? k2 : k3;
      const u16* const at = from + (theirs < nkb ? theirs : k) * kTile;
      Raw8<IN> raw;
      raw.a = *reinterpret_cast<const v4i*>(at);
      if constexpr (std::is_same<IN, GLU>::value) raw.b = *reinterpret_cast<const v4i*>(at + src.gate_off);
      float v[8];
      raw.get(v);
      const Divider d = make_scale(row16_max(amax8(v)), 0.f, false);
      const v2i c8 = quant8<false>(v, d);
      *reinterpret_cast<v2i*>(codes + q4 * kBK + q16 * 8) = c8;
      if (q16 == 0) scales[q4] = d.s;
      __builtin_amdgcn_wave_barrier();  // same wave, in-order LDS: later reads see the writes
    };
    int in_batch = 0;
    auto step = [&](int k, v16f& sum) __attribute__((always_inline)) {
      rs_now = rs_next;
      const int next = after(k);
      if (next < nkb) request(next, (stage + kStage) & kRing);
      if (in_batch == 0) quantise(k);
      // (what was requested behind this block may be on its way)
      if (next < nkb) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(BR / 8) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      auto frag = [&](const uint8_t* at, int h, int x) __attribute__((always_inline)) {
        const v4i lo = *reinterpret_cast<const v4i*>(at + (((4 * h + 2 * hg) ^ x) << 4));
        const v4i hi = *reinterpret_cast<const v4i*>(at + (((4 * h + 2 * hg + 1) ^ x) << 4));
        return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      };
      v8i rf[2], lf[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        lf[h] = frag(codes + in_batch * kBK, h, 0);  // (the token row in all 32 columns)
        rf[h] = frag(mine + stage + l32 * kBK, h, sw);
      }
      const float sc = scales[in_batch] * rs_now;
      in_batch = (in_batch + 1) & (kBatch - 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage has been read and may be filled again
      v16f pr = mfma_fp8_32x32x64(rf[0], lf[0], zero);
      pr = mfma_fp8_32x32x64(rf[1], lf[1], pr);
#pragma unroll
      for (int r = 0; r < 16; r++) sum[r] = __builtin_fmaf(pr[r], sc, sum[r]);
      stage = (stage + kStage) & kRing;
    };
    if (first < nkb) request(first, 0);
    for (int i = first; i < kSums; i += per) {
      v16f sum = zero;
      for (int k = i; k < nkb; k += kSums) step(k, sum);
      keep(i, sum);
    }
  }
  if (first == 0 && lane == 0) {
    expert[slot] = row >= 0 ? e : -1;
    weight[slot] = pv;
  }
  __syncthreads();
  if (tid >= BR) return;
  float tot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < kCombineSlots; j++) {
    if (j >= topk) break;
    float o = 0.f;
    if (expert[j] >= 0) {
      o = part[j][0][tid];
#pragma unroll
      for (int w = 1; w < kSums; w++) o += part[j][w][tid];
      if (p.bias != nullptr) {
        const int64_t at = (int64_t)expert[j] * p.bias_group_stride + r0 + tid;
        o += p.bias_dtype == AAMD_F32 ? reinterpret_cast<const float*>(p.bias)[at] : bf16_bits_to_f32(reinterpret_cast<const u16*>(p.bias)[at]);
      }
      o = __uint_as_float(pack_bf16x2(o, 0.f) << 16);
    }
    float prod = o * weight[j];
    if constexpr (PD == AAMD_BF16) prod = __uint_as_float(pack_bf16x2(prod, 0.f) << 16);
    tot[j & 3] = tot[j & 3] + prod;
  }
  const float sum = ((tot[0] + tot[1]) + tot[2]) + tot[3];
  const int64_t at = (int64_t)t * p.ldc + r0 + tid;
  if constexpr (PD == AAMD_BF16) reinterpret_cast<u16*>(out)[at] = (u16)(pack_bf16x2(sum, 0.f) & 0xffffu);
  else reinterpret_cast<float*>(out)[at] = sum;
}
template <typename IN, int PD>
static void launch_combine(const GemmParams& p, const FewSource& src, const int32_t* row_map, const void* probs, void* out, hipStream_t st) {
  const unsigned topk = src.topk, per = topk <= 2 ? 8 : topk <= 4 ? 4 : 2;
  few_rows_combine_kernel<IN, PD><<<src.T * (unsigned)p.nRt, 64 * per * topk, 0, st>>>(p, src, row_map, probs, out, (int)per);
}
int launch_few_rows_combine(GemmParams p, int what, const void* rows, int64_t ld, const void* ids, int ids_are_i64, const int32_t* row_map,
                            const void* probs, int probs_dtype, int topk, int64_t T, void* out, hipStream_t st) {
  FewSource src = {};
  src.rows = (const u16*)rows; src.ld = ld; src.gate_off = (int64_t)p.nkb * kTile;
  src.topk = (uint32_t)topk; src.T = (uint32_t)T; src.ids = ids; src.ids_are_i64 = ids_are_i64;
  p.nRt = (int)(p.Rrows / 32);
  AAMD_REQUIRE(T * p.nRt < 0x7fffffffLL, "quant_grouped_gemm_combine: grid too large");
  if (what == AAMD_ROWS_SWIGLU) {
    if (probs_dtype == AAMD_BF16) launch_combine<GLU, AAMD_BF16>(p, src, row_map, probs, out, st);
    else launch_combine<GLU, AAMD_F32>(p, src, row_map, probs, out, st);
  } else {
    if (probs_dtype == AAMD_BF16) launch_combine<GELU, AAMD_BF16>(p, src, row_map, probs, out, st);
    else launch_combine<GELU, AAMD_F32>(p, src, row_map, probs, out, st);
  }
  AAMD_LAUNCH_CHECK("grouped_gemm (few rows, combined)");
  return AAMD_OK;
}

}  // namespace aamd
