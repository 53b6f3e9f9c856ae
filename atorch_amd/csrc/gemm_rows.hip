// Row-ragged block-scaled FP8 GEMM on 256 x 256 tiles, one persistent workgroup per CU (forward, dgrad, dense).  (Launches of
// at most one round of tiles take the form with a workgroup per tile, see choose_nt in gemm.hip.)
//
// What a step does and why is the same as in gemm.hip: 128-deep blocks, two chained v_mfma_f32_32x32x64_f8f6f4 per 32 x 32
// sub-tile, the raw product folded into fp32 accumulators with the block's scales, operands moved global -> LDS without a
// register stop, 16-byte chunks XOR-swizzled.  Eight waves of 128 (R) x 64 (L), two per SIMD.
//
// The matrix pipe of a SIMD idles whenever both of its waves are away from their MFMAs at the same time, which is what a
// workgroup barrier followed by LDS reads produces.  So the two barriers of a step stand where register-resident MFMA work
// follows them:
//   Q (start of step k): every wave holds the L fragments of step k, so the L half of its stage is free and the L tile of
//     step k + 2 is requested behind the first sub-tiles;
//   P (before the last R row of sub-tiles): every wave has read the last fragments of the stage and the tiles of step k + 1
//     have landed; behind it the R tile of step k + 2 is requested and the first fragments of step k + 1 are read while the
//     last R row, whose operands are already in registers, runs on the matrix pipe.
// The fold of the sub-tile in front of a barrier is issued behind it.
//
// One workgroup per tile costs 9 to 10 us beside the steps of 1.45 us (stamps taken inside the kernel, 32768 rows x 28672
// outputs x 4096 in 8 groups): 2.0 from the end of one workgroup to the start of the next on a CU, 1.7 to find its group, 2.0
// until its first operands are there, 4.1 to turn the tile round through the LDS and store it.  So a workgroup stays and takes
// one tile after the other, and the steps of its tiles are one stream: the last two steps of a tile request the first two
// blocks of the next one, its last step reads the next one's first fragments, and the finished tile goes from the registers
// to memory (lanes swap what they hold, so that eight of them have 128 consecutive bytes of a row) while those loads are in flight, as
// the stage buffers hold them.  What a tile needs besides are scalars: rows past its end and columns past the weights' end
// are left to the range check of buffer instructions, which neither reads nor writes them.
//
// The last round of tiles seldom fills the card.  Where at most half the workgroups of an XCD have a tile in it and the
// contraction is long, two to eight of them share the contraction of a tile: each leaves its fp32 sums in a workspace, and a
// second kernel adds them in the order of the contraction, so that the result does not depend on which comes first.
#include <algorithm>

#include "gemm_tiles.hpp"

namespace aamd {

namespace rows {
constexpr int BM = 256, BN = 256, NT = 512, WTR = 4, WTL = 2, NTILES = WTR * WTL;
constexpr int kSide = 256 * kBK;        // bytes of an L (R) tile of a step
constexpr int kScaleBatch = BM * 8 + 256;  // floats: the scales of eight contraction blocks, [L row][8] and [R block][8]
constexpr int kLds = 4 * kSide + 2 * kScaleBatch * 4 + 64 * (int)sizeof(int64_t) * 3;
constexpr int kWorkgroups = 256;        // one per CU
}  // namespace rows

// A tile of the output, or a part of its contraction.
struct RowTile {
  int64_t l0;                 // first L row
  int g, lvalid, r0, rvalid;  // group, valid L rows, first R row and valid R rows (a multiple of 128)
  int kb0, steps;             // contraction blocks
};
// Tile `pid` of the launch (its whole contraction).  table: rows and tiles of up to 64 groups in the LDS, or null.
template <typename ARGS>
__device__ __forceinline__ RowTile row_tile(ARGS a, const int64_t* table, uint32_t pid, uint32_t nRt, int total_lt) {
  using namespace rows;
  const uint32_t GL = (uint32_t)a->gl;
  RowTile t;
  uint32_t lt, rt;
  // groups of GL L tiles, R tile index outer, L tile inner
  {
    const uint32_t width = GL * nRt, grp = pid / width, in = pid - grp * width, first = grp * GL;
    const uint32_t gsz = (uint32_t)total_lt - first < GL ? (uint32_t)total_lt - first : GL;
    rt = in / gsz;
    lt = first + (in - rt * gsz);
  }
  t.g = 0;
  int64_t r_lo = 0, r_hi = a->Lrows;
  uint32_t t_lo = 0;
  if (opaque(a->goff != nullptr)) {
    // exactly one group holds the tile; with group_r the tile ids of a group are contiguous, in batches of GL R tiles, all L
    // tiles of the group inside a batch, R index fastest: the weights, the large operand, are then fetched once
    const int by_group = opaque(a->group_r), in_table = opaque(table != nullptr);
    GroupRanges r;
    if (in_table) {
      const int64_t* const e = table + lane_here() * 3;
      r.r_lo = e[0];
      r.r_hi = e[1];
      const int64_t tt = e[2];
      r.t_lo = (int)(uint32_t)(uint64_t)tt;
      r.t_hi = (int)(uint32_t)((uint64_t)tt >> 32);
    }
    for (int base = 0, carry = 0; base < a->E; base += 64) {
      if (!in_table) {
        r = group_ranges<BM>(a->goff, a->E, base, carry);
        carry = r.total;
      }
      const bool mine = by_group ? pid >= (uint32_t)r.t_lo * nRt && pid < (uint32_t)r.t_hi * nRt
                                  : lt >= (uint32_t)r.t_lo && lt < (uint32_t)r.t_hi;  // (empty groups hold no tile)
      const unsigned long long hit = __ballot(mine);
      if (hit != 0) {
        const int src = __builtin_ctzll(hit);
        t.g = base + src;
        t_lo = (uint32_t)__builtin_amdgcn_readlane(r.t_lo, src);
        r_lo = readlane_i64(r.r_lo, src);
        r_hi = readlane_i64(r.r_hi, src);
        if (by_group) {
          const uint32_t nl = (uint32_t)__builtin_amdgcn_readlane(r.t_hi, src) - t_lo;
          const uint32_t pe = pid - t_lo * nRt, width = GL * nl, batch = pe / width, in = pe - batch * width, first = batch * GL;
          const uint32_t gsz = nRt - first < GL ? nRt - first : GL;
          const uint32_t l = in / gsz;
          rt = first + (in - l * gsz);
          lt = t_lo + l;
        }
        break;
      }
    }
  }
  t.l0 = uniform_i64(r_lo + (int64_t)(lt - t_lo) * BM);
  const int64_t left = (r_hi < a->Lrows ? r_hi : a->Lrows) - t.l0;
  t.lvalid = __builtin_amdgcn_readfirstlane(left < BM ? (int)left : BM);
  t.g = __builtin_amdgcn_readfirstlane(t.g);
  t.r0 = __builtin_amdgcn_readfirstlane((int)(rt * BN));
  t.rvalid = (int)(a->Rrows - t.r0 < BN ? a->Rrows - t.r0 : BN);
  t.kb0 = 0;
  t.steps = a->nkb;
  return t;
}

// The tiles of an XCD, a contiguous range, and how its workgroups share what is left in the last round: with few tiles left
// several of them take parts of the contraction of one.
struct RowTiles {
  uint32_t first, end;
  __device__ RowTiles(uint32_t ntot, uint32_t xcd) {
    const uint32_t per = ntot >> 3, rem = ntot & 7u;
    first = xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per;
    end = first + per + (xcd < rem ? 1u : 0u);
  }
};
// Workgroups per tile when `left` tiles are left for nwg of them: 1, or up to max_split.
__device__ __forceinline__ uint32_t row_split(uint32_t left, uint32_t nwg, uint32_t max_split) {
  const uint32_t s = left > 0 ? nwg / left : 1;
  return s < 1 ? 1 : s < max_split ? s : max_split;
}
// First contraction block of a part: whole groups of four (16 bytes of scales) but for the end of the last part.  With
// nkb >= 8 split every part has eight blocks or more.
__device__ __forceinline__ uint32_t row_part(uint32_t nkb, uint32_t split, uint32_t part) {
  return part == split ? nkb : 4u * ((nkb >> 2) * part / split);
}

// R_ROWS: the R operand is stored [contraction, Rrows] and its fragments are read transposed, see grouped_gemm_kernel.
// PAIRS: an even number of steps per tile, so that a step's number says which stage it works on and the stage goes into the
// immediate offset of its LDS reads; else the addresses change with every step (eight instructions more, 2 % of it).
template <typename OUT, bool R_ROWS, bool PAIRS>
__global__ __launch_bounds__(rows::NT, 1) void row_tiles_kernel(const GemmParams p) {
  // (the arguments of what is done once per tile are fetched there: scalar registers are short in the loop; in front of it
  // they come all at once)
  auto args = [&]() __attribute__((always_inline)) { return (const __attribute__((address_space(4))) GemmParams*)(uintptr_t)args_here(); };
  using namespace rows;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds];
  // [L stage 0 | L stage 1 | R stage 0 | R stage 1 | two batches of scales | rows and tiles of the groups]
  float* const scales = reinterpret_cast<float*>(lds + 4 * kSide);
  int64_t* const table = reinterpret_cast<int64_t*>(scales + 2 * kScaleBatch);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hg = lane >> 5;

  // ---- the tiles of this workgroup ------------------------------------------------------------
  // Workgroup ids go round-robin over the 8 XCDs; every XCD gets one contiguous range of tile ids, in which tiles that share
  // operand panels are neighbours, and its workgroups take them side by side.
  GroupRanges gr = {};
  int total_lt = (int)((p.Lrows + BM - 1) / BM);
  if (p.goff != nullptr) {
    gr = group_ranges<BM>(p.goff, p.E, 0, 0);
    total_lt = gr.total;
    for (int base = 64; base < p.E; base += 64) total_lt = group_ranges<BM>(p.goff, p.E, base, total_lt).total;
    if (p.E <= 64) {  // the group of every later tile is found from here
      table[lane * 3] = gr.r_lo;
      table[lane * 3 + 1] = gr.r_hi;
      table[lane * 3 + 2] = (int64_t)(((uint64_t)(uint32_t)gr.t_hi << 32) | (uint32_t)gr.t_lo);
    }  // (every wave writes the same values, and reads what it wrote)
  }
  const uint32_t nRt = (uint32_t)p.nRt, ntot = (uint32_t)total_lt * nRt;
  const uint32_t xcd = blockIdx.x & 7u, nwg = gridDim.x >> 3;
  const RowTiles mine(ntot, xcd);

  // Workgroups that share a panel should stay the same ones: then the first of them to reach a block waits for memory and the
  // others catch up.  With short contractions, whose panels the L2 holds whole, a workgroup moves five places on with every round
  // instead, so that none gets the short last tile of every group.  (Places moved by 5 and by none, us: 32768 rows in 8 groups, 28672
  // x 4096 3425 and 3403, fetched beyond the L2 9.7 and 7.9 GB; 64 groups, 7168 x 2048 218 and 213; 4096 rows, 28672 x 4096 562 and
  // 554; 60 uneven groups, 2048 x 2816 228 and 229, 1408 x 2048 130 and 132, 2048 x 1408 (11 blocks) 134 and 138.)
  const uint32_t places = p.nkb >= 16 ? 0u : nwg > 5u ? 5u : 1u;
  uint32_t round_first = mine.first, turn = blockIdx.x >> 3;
  // the next tile of this workgroup, false if there is none; part and parts: of the contraction it takes, slot: where a part goes
  uint32_t part = 0, parts = 1;
  int n_slot = -1;
  auto take = [&](uint32_t& pid) __attribute__((always_inline)) {
    const uint32_t left = mine.end > round_first ? mine.end - round_first : 0u;
    uint32_t at = turn;
    if (left < nwg && p.max_split > 1) {
      parts = row_split(left, nwg, (uint32_t)p.max_split);
      if (parts > 1) {
        n_slot = turn < left * parts ? (int)(xcd * nwg + turn) : -1;
        part = turn / left;
        at = n_slot >= 0 ? turn - part * left : left;
      }
    }
    pid = round_first + at;
    round_first += nwg;
    turn += places;
    turn = turn >= nwg ? turn - nwg : turn;
    return at < left;
  };
  uint32_t pid;
  if (!take(pid)) return;  // (rounds before the last are whole, so a workgroup that has no tile in one has none later)
  // (plain variables: as structures the two would live in memory)
  int64_t c_l0, n_l0;
  int c_g, c_lvalid, c_r0, c_rvalid, c_kb0, c_steps, c_slot, n_g, n_lvalid, n_r0, n_rvalid, n_kb0, n_steps;
  auto take_tile = [&](uint32_t id, auto a) __attribute__((always_inline)) {
    const RowTile t = row_tile(a, opaque(a->goff != nullptr && a->E <= 64) ? table : nullptr, id, nRt, total_lt);
    n_l0 = t.l0, n_g = t.g, n_lvalid = t.lvalid, n_r0 = t.r0, n_rvalid = t.rvalid, n_kb0 = 0, n_steps = t.steps;
    if (n_slot >= 0) {
      n_kb0 = (int)row_part((uint32_t)t.steps, parts, part);
      n_steps = (int)row_part((uint32_t)t.steps, parts, part + 1) - n_kb0;
    }
  };
  auto next_is_current = [&]() __attribute__((always_inline)) {
    c_l0 = n_l0, c_g = n_g, c_lvalid = n_lvalid, c_r0 = n_r0, c_rvalid = n_rvalid, c_kb0 = n_kb0, c_steps = n_steps, c_slot = n_slot;
  };
  auto current = [&]() __attribute__((always_inline)) { return RowTile{c_l0, c_g, c_lvalid, c_r0, c_rvalid, c_kb0, c_steps}; };
  take_tile(pid, &p);
  next_is_current();

  // ---- loads -------------------------------------------------------------------------------------
  // A wave instruction of a tile load fills 1 KB of the LDS, lane l at base + 16 l; lane l fetches the chunk the swizzle puts
  // there.  n-th instruction of wave w: rows 8 w + 64 n .. + 7 of the tile (R_ROWS: contraction rows 4 w + 32 n .. + 3).
  const int r8 = lane >> 3;
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ r8 ^ (wave & 1)) << 4);
  uint32_t voffL[4], voffR[4];
  const int rrow = R_ROWS ? wave * 4 + (lane >> 4) : wave * 8 + r8;
#pragma unroll
  for (int n = 0; n < 4; n++) {
    voffL[n] = (uint32_t)(wave * 8 + 64 * n + r8) * (uint32_t)p.ldl + chunk;
    voffR[n] = (uint32_t)(rrow + (R_ROWS ? 32 : 64) * n) * (uint32_t)p.ldr + (R_ROWS ? (uint32_t)(((lane & 15) ^ (2 * (rrow & 7))) << 4) : chunk);
  }
  // Where the next block to be requested lies: it runs through the blocks of a tile and on into the next tile; behind the
  // last one it stays on the last block, to keep the wait counts uniform.
  v4i lbuf, rbuf;
  int to_load;         // blocks left in the tile
  int next_block = 0;  // of the next tile: 0, or the last one where that is still the tile under way
  auto enter_next = [&](auto a) __attribute__((always_inline)) {
    const int block = n_kb0 + next_block;
    const int64_t l_at = n_l0 * a->ldl + block * kBK;
    const int64_t r_at = (int64_t)n_g * a->r_group_stride + (R_ROWS ? (int64_t)n_r0 : n_r0 * a->ldr) + block * a->r_kb_stride;
    lbuf = buffer_at(a->L + uniform_i64(l_at), (uint32_t)__builtin_amdgcn_readfirstlane((n_lvalid - 1) * (int)a->ldl + kBK));
    rbuf = buffer_at(a->R + uniform_i64(r_at), (uint32_t)__builtin_amdgcn_readfirstlane(
                                                   R_ROWS ? 127 * (int)a->ldr + n_rvalid : (n_rvalid - 1) * (int)a->ldr + kBK));
    to_load = n_steps - next_block;
  };
  enter_next(&p);
  auto advance = [&]() __attribute__((always_inline)) {
    advance_buffer(lbuf, kBK);
    advance_buffer(rbuf, p.r_kb_stride);
    if (--to_load == 0) enter_next(args());
  };
  // where this wave's loads go, in the stage of the step under way (PAIRS: in stage 0)
  uint32_t to_lds = lds_offset(lds) + (uint32_t)(wave * 1024);
  auto load_l = [&](auto S, auto N) __attribute__((always_inline)) {
    load_lds_x4<(PAIRS ? decltype(S)::value * kSide : 0) + decltype(N)::value * 8192>(voffL[decltype(N)::value], lbuf, to_lds);
  };
  auto load_r = [&](auto S, auto N) __attribute__((always_inline)) {
    load_lds_x4<2 * kSide + (PAIRS ? decltype(S)::value * kSide : 0) + decltype(N)::value * 8192>(voffR[decltype(N)::value], rbuf, to_lds);
  };
  auto load_tile = [&](auto S) __attribute__((always_inline)) {
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_l(S, N); });
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_r(S, N); });
  };
  auto other_stage = [&]() __attribute__((always_inline)) {
    if constexpr (!PAIRS) to_lds ^= kSide;
  };

  // Scales come in batches of eight contraction blocks (the last batch of a tile is shifted back to end at its last block): a
  // row of 32 bytes per L row and per 128 R rows.  Batch b of a tile is
  // requested in step 8 b - 3, batch 0 of the next tile in one of the last three steps (see `ask_next`), when the batch before
  // the one in use has been read for the last time.  Rows of scales that are not 16-byte aligned take 4-byte loads.
  const int x4 = p.ls_batch == 1;
  const uint32_t lsr = (uint32_t)p.ls_row_stride, rsr = (uint32_t)p.rs_row_stride, rsb = (uint32_t)p.rs_blk_stride;
  auto ask_scales = [&](const RowTile t, int b, int parity, auto a) __attribute__((always_inline)) {
    const int at = t.kb0 + (8 * b + 8 <= t.steps ? 8 * b : t.steps - 8), ln = lane_here();
    const v4i lb = buffer_at(a->Ls + uniform_i64(t.l0 * lsr + at), (uint32_t)__builtin_amdgcn_readfirstlane(((t.lvalid - 1) * (int)lsr + 8) * 4));
    const uint32_t ld = lds_offset(scales + parity * kScaleBatch) + (uint32_t)(wave * 1024);
    const int wide = opaque(x4);
    if (wide) {
      load_lds_x4<0>(((uint32_t)(wave * 32 + (ln >> 1)) * lsr + (uint32_t)(ln & 1) * 4u) * 4u, lb, ld);
    } else {
#pragma unroll
      for (int q = 0; q < 4; q++)
        load_lds_x1(((uint32_t)(wave * 32 + q * 8 + (ln >> 3)) * lsr + (uint32_t)(ln & 7)) * 4u, lb, ld + (uint32_t)(q * 256));
    }
    if (wave == 0) {
      const int blocks = t.rvalid / kTile;
      const v4i rb = buffer_at(a->Rs + uniform_i64((int64_t)t.g * a->rs_group_stride + (int64_t)(t.r0 / kTile) * rsr + (int64_t)at * rsb),
                               (uint32_t)__builtin_amdgcn_readfirstlane((R_ROWS ? 7 * (int)rsb + blocks : (blocks - 1) * (int)rsr + 8) * 4));
      const uint32_t rd = lds_offset(scales + parity * kScaleBatch + BM * 8);
      if (wide && !R_ROWS) load_lds_x4<0>(((uint32_t)((ln >> 1) & 1) * rsr + (uint32_t)(ln & 1) * 4u) * 4u, rb, rd);
      else load_lds_x1(((uint32_t)((ln >> 3) & 1) * rsr + (uint32_t)(ln & 7) * rsb) * 4u, rb, rd);
    }
  };

  // ---- matrix tiling: as in grouped_gemm_kernel.  The two waves of a SIMD (w and w + 4) share their R half and take L row
  // blocks half a tile apart, so that a tile whose valid rows end in its first half keeps a working wave on every SIMD.
  const int wr = wave & 1, wl = ((wave & 3) >> 1) + 2 * (wave >> 2);
  const int wrow0 = wr * WTR * 32, wlrow0 = wl * WTL * 32;
  const int sw = (l32 & 7) ^ ((l32 >> 3) & 1);
  uint32_t la[2][2], ra[2][2];  // LDS addresses of this lane's chunks, stage 0
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const uint32_t chk = (uint32_t)(((4 * h + 2 * hg + c) ^ sw) << 4);
      la[h][c] = lds_offset(lds) + (uint32_t)((wlrow0 + l32) * kBK) + chk;
      if constexpr (R_ROWS) {
        const int tr = (lane & 15) >> 1;
        const int ch = (wrow0 / 16 + 2 * (2 * h + c) + ((lane >> 4) & 1)) ^ (2 * tr);
        ra[h][c] = lds_offset(lds) + 2 * kSide + (uint32_t)((32 * hg + tr) * BN + ch * 16 + (lane & 1) * 8);
      } else {
        ra[h][c] = lds_offset(lds) + 2 * kSide + (uint32_t)((wrow0 + l32) * kBK) + chk;
      }
    }
  // (without PAIRS: during a step `la` names the stage of the next one, and `ra` too from the middle of the step on)
  auto other_l = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int c = 0; c < 2; c++) la[h][c] ^= kSide;
  };
  auto other_r = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int c = 0; c < 2; c++) ra[h][c] ^= kSide;
  };
  typedef const __attribute__((address_space(3))) v4i* lds_v4i_t;
  auto frag = [&](const uint32_t (&base)[2][2], int s, int sub, int h) __attribute__((always_inline)) {
    const uint32_t at = (uint32_t)((PAIRS ? s * kSide : 0) + sub * 32 * kBK);
    const v4i lo = *(lds_v4i_t)(uintptr_t)(base[h][0] + at);
    const v4i hi = *(lds_v4i_t)(uintptr_t)(base[h][1] + at);
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto fragR = [&](int s, int sub, int h) __attribute__((always_inline)) {
    if constexpr (R_ROWS) {
      v8i f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const v2i o = lds_read_transposed(ra[sub / 2][sub % 2] + (uint32_t)((PAIRS ? s * kSide : 0) + (64 * h + 8 * j) * BN));
        f[2 * j] = o[0];
        f[2 * j + 1] = o[1];
      }
      return f;
    } else {
      return frag(ra, s, sub, h);
    }
  };
  auto barrier_q = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  v16f acc[WTR][WTL], pr;
  v8i lf[WTL][2], rf[2][2];
  float cs[WTL], csn[WTL], rblkn, cs_last = 0.f;

  // Scales of a block: the lane's L row scales and the wave's R block scale; sc_at: where the next block's are, sc_left: blocks
  // from there to the end of the batch, sc_more: batches of the tile behind it.
  int last_batch = 0, in_last = 0;  // of the tile under way: its last batch, and the blocks of it that are new
  int sc_parity = 0;  // of the tile's batch 0
  uint32_t sc_at = 0;
  int sc_left = 0, sc_more = 0;
  const uint32_t sc_l = lds_offset(scales) + (uint32_t)((wlrow0 + l32) * 32), sc_r = lds_offset(scales) + (uint32_t)(BM * 32 + (wrow0 / kTile) * 32);
  auto read_scales = [&]() __attribute__((always_inline)) {
    typedef const __attribute__((address_space(3))) float* lds_float_t;
    const lds_float_t l = (lds_float_t)(uintptr_t)(sc_l + sc_at);
    rblkn = *(lds_float_t)(uintptr_t)(sc_r + sc_at);
#pragma unroll
    for (int j = 0; j < WTL; j++) csn[j] = l[j * 32 * 8];
    sc_at += 4;
    if (--sc_left == 0) {
      // (the first word of the other batch; past the tile's last block nobody uses what is read)
      sc_at = sc_at > kScaleBatch * 4u ? 0u : kScaleBatch * 4u;
      sc_left = 8;
      if (--sc_more == 0) {  // the last batch ends at the last block
        sc_left = in_last;
        sc_at += (uint32_t)(8 - in_last) * 4u;
      }
    }
  };
  auto first_scales = [&]() __attribute__((always_inline)) {
    sc_at = (uint32_t)(sc_parity * kScaleBatch * 4);
    sc_left = 8;
    sc_more = last_batch;
    read_scales();
  };
  // The step that requests batch 0 of the next tile: from step 8 last_batch - 1 on the batch in front of the last is free, and
  // the last step comes too late for what the next tile begins with.
  int ask_at = 0, ask_batch = 0, ask_next = 0;
  auto first_ask = [&]() __attribute__((always_inline)) {
    ask_next = c_steps - 4 > 8 * last_batch - 1 ? c_steps - 4 : 8 * last_batch - 1;
    ask_batch = 1;
    ask_at = last_batch > 0 ? 5 : ask_next;
  };

  // (the empty volatile statements pin MFMAs and folds between the memory instructions around them)
  auto fold = [&](int i, int j, float sc) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][j][r] = __builtin_fmaf(pr[r], sc, acc[i][j][r]);
    asm volatile("" : "+v"(acc[i][j]));
  };
  auto first_fragments = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      rf[0][h] = fragR(0, 0, h);
#pragma unroll
      for (int j = 0; j < WTL; j++) lf[j][h] = frag(la, 0, j, h);
    }
  };

  auto ask_in_step = [&](int kb) __attribute__((always_inline)) {
    if (kb != ask_at) return;
    const bool of_next = ask_batch > last_batch;
    ask_scales(RowTile{of_next ? +n_l0 : +c_l0, of_next ? +n_g : +c_g, of_next ? +n_lvalid : +c_lvalid, of_next ? +n_r0 : +c_r0,
                       of_next ? +n_rvalid : +c_rvalid, of_next ? +n_kb0 : +c_kb0, of_next ? +n_steps : +c_steps},
               of_next ? 0 : ask_batch, (sc_parity + ask_batch) & 1, args());
    ask_batch++;
    ask_at = ask_batch <= last_batch ? kb + 8 : ask_batch == last_batch + 1 ? ask_next : -1;
  };

  constexpr int PT = (WTR - 1) * WTL - 1;  // the sub-tile in front of barrier P
  constexpr int kStores = NTILES * (sizeof(OUT) == 4 ? 4 : 2);  // of a wave and tile
  bool stored = false;
  // S: the stage (0 without PAIRS)
  auto step = [&](int kb, auto S) __attribute__((always_inline)) {
    constexpr int s = decltype(S)::value;
    __builtin_amdgcn_sched_barrier(0);
    barrier_q();
    __builtin_amdgcn_sched_barrier(0);
    fold(WTR - 1, WTL - 1, cs_last);  // owed by the step before (adds zero in the first one)
    if (!PAIRS) other_l();
    static_for<NTILES>([&](auto T) __attribute__((always_inline)) {
      constexpr int t = decltype(T)::value;
      constexpr int i = t / WTL, j = t % WTL;
      __builtin_amdgcn_sched_barrier(0);
      pr = mfma_fp8_32x32x64(rf[i & 1][0], lf[j][0], v16f{});
      pr = mfma_fp8_32x32x64(rf[i & 1][1], lf[j][1], pr);
      asm volatile("" : "+v"(pr));
      __builtin_amdgcn_sched_barrier(0);
      // memory instructions go out while the MFMAs run, ahead of the fold that waits for them
      if constexpr (t < 4) load_l(S, T);
      if constexpr (j == 0 && i + 1 < WTR) {
#pragma unroll
        for (int h = 0; h < 2; h++) rf[(i + 1) & 1][h] = fragR(s, i + 1, h);
      }
      if constexpr (t == PT) {
        __builtin_amdgcn_sched_barrier(0);
        // all but this step's L tile loads have landed (loads and stores are counted in issue order; the stores of the tile
        // before were issued behind the loads this step waits for)
        if (kb == 0 && stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(4 + kStores) : "memory");
        else asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        ask_in_step(kb);
        if (!PAIRS) other_r();
        // row WTR - 2 has been consumed: its registers take the first R row of the next step
#pragma unroll
        for (int h = 0; h < 2; h++) rf[0][h] = fragR(s ^ 1, 0, h);
        read_scales();
      }
      if constexpr (t > PT) {
        constexpr int jn = t - PT - 1;  // == j: this sub-tile was the last user of lf[j]
        load_r(S, std::integral_constant<int, 2 * jn>{});
        load_r(S, std::integral_constant<int, 2 * jn + 1>{});
#pragma unroll
        for (int h = 0; h < 2; h++) lf[jn][h] = frag(la, s ^ 1, jn, h);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (t + 1 < NTILES) fold(i, j, cs[j]);
    });
    cs_last = cs[WTL - 1];
#pragma unroll
    for (int j = 0; j < WTL; j++) cs[j] = csn[j] * rblkn;
    advance();
    other_stage();
  };
  // a wave without valid rows: loads and barriers only, in the order of the working waves
  auto idle_step = [&](int kb, auto S) __attribute__((always_inline)) {
    barrier_q();
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_l(S, N); });
    if (kb == 0 && stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(4 + kStores) : "memory");
    else asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    ask_in_step(kb);
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_r(S, N); });
    advance();
    other_stage();
  };

  // ---- a finished tile: registers -> memory
  auto store_tile = [&](const RowTile t) __attribute__((always_inline)) {
    const auto a = args();
    constexpr uint32_t kEl = sizeof(OUT);
    const int left = t.lvalid - wlrow0, rows = left < 64 ? left : 64;
    if (opaque(c_slot >= 0)) {  // a part: as it is, into the workspace
      const v4i out = buffer_at(a->ws + ((int64_t)c_slot * (BM * BN) + wlrow0 * BN + wrow0), ((uint32_t)(rows - 1) * BN + 128u) * 4u);
      const uint32_t at = store_offset<float>(lane_here(), BN);
      static_for<NTILES / 2>([&](auto T) __attribute__((always_inline)) {
        constexpr int i = 2 * (decltype(T)::value % (WTR / 2)), j = decltype(T)::value / (WTR / 2);
        store_sub_tiles<float, i * 32, false>(acc[i][j], acc[i + 1][j], at + (uint32_t)(j * 32 * BN * 4), BN, out);
      });
      return;
    }
    const v4i out = buffer_at(reinterpret_cast<OUT*>(a->C) + ((t.l0 + wlrow0) * a->ldc + t.r0 + wrow0),
                              ((uint32_t)(rows - 1) * (uint32_t)a->ldc + 128u) * kEl);
    const int ln = lane_here(), h5 = ln >> 5;
    const uint32_t at = store_offset<OUT>(ln, (uint32_t)a->ldc);
    if (opaque(a->bias != nullptr)) {
#pragma unroll
      for (int i = 0; i < WTR; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int64_t col = (int64_t)t.g * a->bias_group_stride + t.r0 + wrow0 + i * 32 + 8 * q + 4 * h5;
          v4f b;
          if (opaque(a->bias_dtype == AAMD_F32)) {
            b = *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(a->bias) + col);
          } else {
            const v2i raw = *reinterpret_cast<const v2i*>(reinterpret_cast<const u16*>(a->bias) + col);
            b = v4f{bf16_bits_to_f32((uint32_t)raw[0] & 0xffffu), bf16_bits_to_f32((uint32_t)raw[0] >> 16),
                    bf16_bits_to_f32((uint32_t)raw[1] & 0xffffu), bf16_bits_to_f32((uint32_t)raw[1] >> 16)};
          }
#pragma unroll
          for (int j = 0; j < WTL; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][4 * q + r] += b[r];
        }
    }
    auto store_as = [&](auto nt) __attribute__((always_inline)) {
      static_for<NTILES / 2>([&](auto T) __attribute__((always_inline)) {
        constexpr int i = 2 * (decltype(T)::value % (WTR / 2)), j = decltype(T)::value / (WTR / 2);
        store_sub_tiles<OUT, i * 32, decltype(nt)::value>(acc[i][j], acc[i + 1][j], at + (uint32_t)(j * 32) * (uint32_t)a->ldc * kEl,
                                                          (uint32_t)a->ldc, out);
      });
    };
    if (opaque(a->stream_out)) store_as(std::true_type{});
    else store_as(std::false_type{});
  };

  // ---- the first tile's blocks 0 and 1
  constexpr std::integral_constant<int, 0> S0{};
  constexpr std::integral_constant<int, 1> S1{};
  load_tile(S0);
  ask_scales(current(), 0, 0, &p);
  advance_buffer(lbuf, kBK);
  advance_buffer(rbuf, p.r_kb_stride);
  other_stage();
  load_tile(S1);
  advance_buffer(lbuf, kBK);
  advance_buffer(rbuf, p.r_kb_stride);
  other_stage();
  to_load -= 2;

  bool first = true;
  for (;;) {
    const bool more = take(pid);
    if (more) take_tile(pid, args());
    next_block = more ? 0 : n_steps - 1;
    last_batch = (c_steps - 1) >> 3;
    in_last = c_steps - 8 * last_batch;
    first_ask();
    if (first) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the first tile's block 0 and scales
    first = false;
    const bool work = wrow0 < c_rvalid && wlrow0 < c_lvalid;
    if (work) {
      first_fragments();
      first_scales();
#pragma unroll
      for (int j = 0; j < WTL; j++) cs[j] = csn[j] * rblkn;
#pragma unroll
      for (int i = 0; i < WTR; i++)
#pragma unroll
        for (int j = 0; j < WTL; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++) pr[r] = 0.f;
      cs_last = 0.f;
      for (int kb = 0; kb < c_steps; kb++) {
        step(kb, S0);
        if constexpr (PAIRS) step(++kb, S1);
      }
      __builtin_amdgcn_sched_barrier(0);
      fold(WTR - 1, WTL - 1, cs_last);
      store_tile(current());
    } else {
      for (int kb = 0; kb < c_steps; kb++) {
        idle_step(kb, S0);
        if constexpr (PAIRS) idle_step(++kb, S1);
      }
      if (!PAIRS && (c_steps & 1)) {
        other_l();
        other_r();
      }
    }
    stored = work;
    if (!more) break;
    sc_parity = (sc_parity + last_batch + 1) & 1;
    next_is_current();
  }
  // No load may land in an LDS that is no longer this workgroup's; the stores behind the last loads need nobody to wait.
  if (stored) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kStores) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// The sums of the parts of the tiles that row_tiles_kernel has split, in the order of the contraction, with the bias: eight XCDs x
// tiles left in the last round x eight slices of 32 rows.  Bound by memory, of which some is still in the caches: 12 tiles per XCD
// in two parts, 50 MB, 17 us; slices of 32 rows make 768 workgroups of them, and one load of 16 bytes per lane and part is
// in flight for each of eight rows.
template <typename OUT>
__global__ __launch_bounds__(256) void row_parts_kernel(const GemmParams p) {
  using namespace rows;
  constexpr int kSlices = 8, kRows = BM / kSlices;
  constexpr uint32_t nwg = kWorkgroups / 8;
  const uint32_t xcd = blockIdx.x & 7u, j = (blockIdx.x >> 3) / kSlices, slice = (blockIdx.x >> 3) % kSlices;
  int total_lt = (int)((p.Lrows + BM - 1) / BM);
  if (p.goff != nullptr) {
    total_lt = group_ranges<BM>(p.goff, p.E, 0, 0).total;
    for (int base = 64; base < p.E; base += 64) total_lt = group_ranges<BM>(p.goff, p.E, base, total_lt).total;
  }
  const RowTiles mine((uint32_t)total_lt * (uint32_t)p.nRt, xcd);
  const uint32_t left = (mine.end - mine.first) % nwg, parts = row_split(left, nwg, (uint32_t)p.max_split);
  if (parts < 2 || j >= left) return;
  const RowTile t = row_tile(&p, nullptr, mine.end - left + j, (uint32_t)p.nRt, total_lt);
  const int col = (int)(threadIdx.x & 63) * 4, row0 = (int)(slice * kRows + (threadIdx.x >> 6));
  if (col >= t.rvalid) return;
  v4f b = {0.f, 0.f, 0.f, 0.f};
  if (p.bias != nullptr) {
    const int64_t at = (int64_t)t.g * p.bias_group_stride + t.r0 + col;
    if (p.bias_dtype == AAMD_F32) {
      b = *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(p.bias) + at);
    } else {
      const v2i raw = *reinterpret_cast<const v2i*>(reinterpret_cast<const u16*>(p.bias) + at);
      b = v4f{bf16_bits_to_f32((uint32_t)raw[0] & 0xffffu), bf16_bits_to_f32((uint32_t)raw[0] >> 16),
              bf16_bits_to_f32((uint32_t)raw[1] & 0xffffu), bf16_bits_to_f32((uint32_t)raw[1] >> 16)};
    }
  }
  const float* const from = p.ws + ((int64_t)(xcd * nwg + j) * (BM * BN) + col);
#pragma unroll
  for (int r = 0; r < kRows; r += 4) {
    const int row = row0 + r;
    if (row >= t.lvalid) return;
    v4f sum = *reinterpret_cast<const v4f*>(from + row * BN);
    for (uint32_t i = 1; i < parts; i++) sum += *reinterpret_cast<const v4f*>(from + (int64_t)(i * left) * (BM * BN) + row * BN);
    sum += b;
    OUT* const out = reinterpret_cast<OUT*>(p.C) + (t.l0 + row) * p.ldc + t.r0 + col;
    if constexpr (sizeof(OUT) == 4) *reinterpret_cast<v4f*>(out) = sum;
    else *reinterpret_cast<v2i*>(out) = v2i{(int)pack_bf16x2(sum[0], sum[1]), (int)pack_bf16x2(sum[2], sum[3])};
  }
}

template <typename OUT, bool R_ROWS>
static void launch_row_tiles_as(const GemmParams& p, unsigned blocks, hipStream_t st) {
  if (p.nkb % 2 == 0) row_tiles_kernel<OUT, R_ROWS, true><<<blocks, rows::NT, 0, st>>>(p);
  else row_tiles_kernel<OUT, R_ROWS, false><<<blocks, rows::NT, 0, st>>>(p);
}
int launch_row_tiles(GemmParams p, int c_dtype, int64_t tiles, bool r_rows, hipStream_t st) {
  AAMD_REQUIRE(tiles < 0x7fffffffLL, "grouped_gemm: grid too large");
  unsigned blocks = (unsigned)std::min<int64_t>((tiles + 7) / 8 * 8, rows::kWorkgroups);
  // Streaming stores keep a large output from evicting the operands from the last-level cache, and cost a launch that is short
  // of steps to hide them (us, plain and streaming: 4096 x 32768 outputs (268 MB), contraction 4096 492 -> 464, 2048 267 -> 272,
  // 1024 160 -> 175; 32768 x 28672 (1.9 GB), 4096 3449 -> 3414; 4096 x 14336 (117 MB), 4096 222 both).
  p.stream_out = p.nkb >= 32 && p.Lrows * p.Rrows * (c_dtype == AAMD_BF16 ? 2 : 4) >= (int64_t)1 << 28;
  if (p.max_split > 1) blocks = rows::kWorkgroups;
  if (c_dtype == AAMD_BF16) {
    if (r_rows) launch_row_tiles_as<u16, true>(p, blocks, st);
    else launch_row_tiles_as<u16, false>(p, blocks, st);
  } else {
    if (r_rows) launch_row_tiles_as<float, true>(p, blocks, st);
    else launch_row_tiles_as<float, false>(p, blocks, st);
  }
  AAMD_LAUNCH_CHECK("grouped_gemm (256 x 256 tiles)");
  if (p.max_split > 1) {
    const unsigned sums = 8 * (rows::kWorkgroups / 8 / 2) * 8;  // (a tile is split where at most half the workgroups have one)
    if (c_dtype == AAMD_BF16) row_parts_kernel<u16><<<sums, 256, 0, st>>>(p);
    else row_parts_kernel<float><<<sums, 256, 0, st>>>(p);
    AAMD_LAUNCH_CHECK("grouped_gemm (parts)");
  }
  return AAMD_OK;
}

}  // namespace aamd
