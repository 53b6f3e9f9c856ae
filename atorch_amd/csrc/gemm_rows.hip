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
//
// A group's rows seldom are a multiple of 256, and the tile of the few that are left costs half a full one or more: it fetches all
// the weights once more, 1.1 us a step where those of full tiles take 1.9 (28672 outputs x 4096, 8 groups, us: 512 rows each 430,
// 520 550, 640 595, 768 640).  So there is a second form of the loop for tiles of up to 288 rows, which hand what is left out to the full
// tiles of the group: a ninth load instruction of a wave and step, one sub-tile more for each of the eight waves (the 32 rows by 256
// columns of all of them).  The registers for it come from addresses, which are made in the step, and from what a tile is, which lies in
// the LDS; that costs 4 to 10 % of a step, so the kernel that holds both forms takes it where the rows of the groups save more (see
// higher_tiles_pay, and for what it gives).  By the counters, the same launch: 512 rows each 8.9 % more cycles of the CUs, 8 % more
// vector instructions, the matrix pipes busy for 54.5 % of the time instead of 59, 1.20 GB fetched instead of 1.07 (every XCD takes an eighth of
// all groups); 485 to 542 rows 8.9 % fewer cycles, 3.6 % fewer products, 1.54 GB instead of 1.44.
#include <algorithm>

#include "gemm_tiles.hpp"

namespace aamd {

namespace rows {
constexpr int BM = 256, BN = 256, NT = 512, WTR = 4, WTL = 2, NTILES = WTR * WTL;
constexpr int kSide = 256 * kBK;        // bytes of an L (R) tile of a step
constexpr int kMore = 32, kMoreSide = kMore * kBK;  // rows that a tile may have beyond BM, and their bytes in a step
constexpr int kTileWords = 12;          // of a RowTile and where a part goes
// workgroups of an XCD that may share out the contraction of its last tiles, as the workspace has room for
constexpr uint32_t part_places(bool more) { return more ? 28 : 32; }
constexpr int high_tile(bool more) { return more ? BM + kMore : BM; }
// floats: the scales of eight contraction blocks, [L row][8] and [R block][8]
constexpr int scale_batch(bool more) { return high_tile(more) * 8 + 256; }
constexpr int table_at(bool either) { return 4 * kSide + (either ? 2 * kMoreSide : 0) + 2 * scale_batch(either) * 4; }  // rows and tiles of the groups
constexpr int lds_bytes(bool either) { return table_at(either) + 64 * (int)sizeof(int64_t) * 3 + (either ? 8 * 2 * kTileWords * 4 : 0); }
constexpr int kWorkgroups = 256;        // one per CU
static_assert(8 * part_places(true) * high_tile(true) * BN * 4 <= kRowPartsBytes && 8 * part_places(false) * BM * BN * 4 <= kRowPartsBytes, "the parts fit the workspace");
}  // namespace rows

// A tile of the output, or a part of its contraction.
struct RowTile {
  int64_t l0;                 // first L row
  int g, lvalid, r0, rvalid;  // group, valid L rows, first R row and valid R rows (a multiple of 128)
  int kb0, steps;             // contraction blocks
};
// With MORE the rows of a group beyond its full tiles go to these, 32 to each, where there are enough of them; else, and without, to a
// tile of their own.
template <bool MORE>
__device__ __forceinline__ int row_tiles_of(int64_t rows) {
  using namespace rows;
  if constexpr (MORE) return (int)(rows / BM) + ((int)(rows % BM) > kMore * (int)(rows / BM) ? 1 : 0);
  else return (int)((rows + BM - 1) / BM);
}
// First and last row of group base + lane (none past E), and group_ranges of these tiles.
struct GroupRows {
  int64_t lo, hi;
};
__device__ __forceinline__ GroupRows group_rows(const int64_t* __restrict__ goff, int E, int base) {
  const int e = base + ((int)threadIdx.x & 63);
  GroupRows r = {0, 0};
  if (e < E) {
    r.lo = goff[e];
    r.hi = goff[e + 1];
  }
  return r;
}
template <bool MORE>
__device__ __forceinline__ GroupRanges row_ranges(const GroupRows& rows, int carry) {
  GroupRanges r;
  r.r_lo = rows.lo;
  r.r_hi = rows.hi;
  const int n = row_tiles_of<MORE>(rows.hi - rows.lo);
  r.t_hi = carry + wave_inclusive_sum(n);
  r.t_lo = r.t_hi - n;
  r.total = __builtin_amdgcn_readlane(r.t_hi, 63);
  return r;
}
template <bool MORE>
__device__ __forceinline__ GroupRanges row_ranges(const int64_t* __restrict__ goff, int E, int base, int carry) {
  return row_ranges<MORE>(group_rows(goff, E, base), carry);
}
// At most 64 groups of less than 1792 rows on average: the launcher sees to that, and to the rest itself where there are no groups.  (What
// a workgroup executes in front of its first tile is fetched from beyond the instruction cache: 250 instructions took 0.7 us.)
template <typename ARGS>
__device__ __forceinline__ bool higher_tiles(ARGS p, const GroupRows& of_lane) {
  using namespace rows;
  if (p->higher != 0) return p->higher > 0;
  const uint32_t rows = (uint32_t)(of_lane.hi - of_lane.lo), f = rows / BM, over = rows % BM, more = (over + kMore - 1) / kMore;
  // full tiles, remainders with a tile of their own without and with MORE, 32 rows more
  const uint32_t own0 = (uint32_t)__popcll(__ballot(over > 0)), own1 = (uint32_t)__popcll(__ballot(more > f));
  if (own0 == own1) return false;
  const uint32_t sums = (uint32_t)__builtin_amdgcn_readlane(wave_inclusive_sum((int)(f << 16 | (more > f ? 0u : more))), 63);
  const uint32_t full = sums >> 16, tiles = (more > f ? f + 1 : f) * (uint32_t)p->nRt;
  uint32_t n1 = (full + own1) * (uint32_t)p->nRt;
  if (p->slices && p->nRt % 8 != 0) {  // the longest of the XCDs' slices
    uint32_t most = 0;
#pragma unroll 1
    for (uint32_t xcd = 0; xcd < 8; xcd++) {
      const uint32_t n = (uint32_t)__popcll(__ballot(((xcd + threadIdx.x) & 7u) < (tiles & 7u)));
      most = n > most ? n : most;
    }
    n1 = 8 * ((uint32_t)__builtin_amdgcn_readlane(wave_inclusive_sum((int)(tiles >> 3)), 63) + most);
  }
  return higher_tiles_pay(full, own0, own1, sums & 0xffffu, (uint32_t)p->nRt, n1, p->max_split > 1);
}
// With MORE every XCD may take an eighth of every group's tiles, R tile by R tile with all L tiles of it: tiles of more rows are then
// spread over all of them (with one range of tiles for each XCD the one whose groups had the most of them took longest: 8 groups,
// one of 560 rows, 28672 x 4096 601 -> 483).  From 32 R tiles a group on: 0.96 of the time of ranges, 0.98 from 16, 1.01 below.
struct Slice {
  uint32_t first, count;
};
__device__ __forceinline__ Slice slice_of(uint32_t tiles, uint32_t g, uint32_t xcd) {
  const uint32_t part = (xcd + g) & 7u, size = tiles >> 3, rem = tiles & 7u;  // (remainders rotate over the XCDs)
  return {part * size + (part < rem ? part : rem), size + (part < rem ? 1u : 0u)};
}
// A lane's group in this order: its tiles of this XCD.
template <bool MORE>
__device__ __forceinline__ GroupRanges row_slices(const GroupRows& rows, uint32_t nRt, uint32_t xcd) {
  GroupRanges r;
  r.r_lo = rows.lo;
  r.r_hi = rows.hi;
  const int n = (int)slice_of((uint32_t)row_tiles_of<MORE>(rows.hi - rows.lo) * nRt, threadIdx.x & 63, xcd).count;
  r.t_hi = wave_inclusive_sum(n);
  r.t_lo = r.t_hi - n;
  r.total = __builtin_amdgcn_readlane(r.t_hi, 63);
  return r;
}
// Tile `pid` of the launch, with slices of the XCD (its whole contraction).  table: rows and tiles of up to 64 groups in the LDS, or null.
template <bool MORE, typename ARGS>
__device__ __forceinline__ RowTile row_tile(ARGS a, const int64_t* table, uint32_t pid, uint32_t nRt, int total_lt, uint32_t xcd) {
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
  uint32_t t_lo = 0, t_n = (uint32_t)total_lt, turn = 0;
  if (opaque(a->goff != nullptr)) {
    // exactly one group holds the tile; with group_r the tile ids of a group are contiguous, in batches of GL R tiles, all L
    // tiles of the group inside a batch, R index fastest: the weights, the large operand, are then fetched once
    const int by_group = opaque(a->group_r), in_table = opaque(table != nullptr), slices = MORE ? opaque(a->slices) : 0;
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
        r = row_ranges<MORE>(a->goff, a->E, base, carry);
        carry = r.total;
      }
      const uint32_t each = slices ? 1u : nRt;
      const bool mine = by_group ? pid >= (uint32_t)r.t_lo * each && pid < (uint32_t)r.t_hi * each
                                  : lt >= (uint32_t)r.t_lo && lt < (uint32_t)r.t_hi;  // (empty groups hold no tile)
      const unsigned long long hit = __ballot(mine);
      if (hit != 0) {
        const int src = __builtin_ctzll(hit);
        t.g = base + src;
        t_lo = (uint32_t)__builtin_amdgcn_readlane(r.t_lo, src);
        t_n = (uint32_t)__builtin_amdgcn_readlane(r.t_hi, src) - t_lo;
        r_lo = readlane_i64(r.r_lo, src);
        r_hi = readlane_i64(r.r_hi, src);
        if (MORE && slices) {
          t_n = (uint32_t)row_tiles_of<MORE>(r_hi - r_lo);
          const uint32_t pe = slice_of(t_n * nRt, (uint32_t)t.g, xcd).first + pid - t_lo;
          rt = pe / t_n;
          lt = t_lo + (pe - rt * t_n);
          turn = (rt >> 2) + (rt >> 3) + (rt >> 4);
        } else if (by_group) {
          const uint32_t nl = t_n;
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
  uint32_t i = lt - t_lo;
  int64_t at = r_lo;
  int high = BM;
  if (MORE && (int64_t)t_n * BM <= r_hi - r_lo) {
    // The tiles with rows beyond BM are others from round to round: none of the workgroups gets them all.
    const uint32_t over = (uint32_t)(r_hi - r_lo) - t_n * BM;
    if (over > 0) i = (i + turn) % t_n;
    const uint32_t more = i * kMore;  // rows that the tiles in front may have taken
    high = more < over ? (over - more < kMore ? BM + (int)(over - more) : BM + kMore) : BM;
    at += more < over ? more : over;
  }
  t.l0 = uniform_i64(at + (int64_t)i * BM);
  const int64_t left = (r_hi < a->Lrows ? r_hi : a->Lrows) - t.l0;
  t.lvalid = __builtin_amdgcn_readfirstlane(left < high ? (int)left : high);
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
// Where the contraction is not shared and at most half the workgroups have a tile in the last round, two or four of them share the rows
// of one, in pieces of 64.  The step of such a piece waits for its loads, which are asked for one step ahead: with 256 rows and half of the
// chip idle 1.3 us, with 128 1.25, with 64 1.0 (a step of a whole round: 1.8).  us, 4096 rows, last round of 1 to 8 tiles per XCD:
// 8704 x 1024 60 -> 57, x 4096 164 -> 157; 12800 x 2048 126 -> 121; 16640 x 4096 279 -> 271; of 16 tiles 14336 x 4096 229 -> 228; 16001 uneven
// rows in 60 groups, 2048 x 2816 120 -> 114.  Parts of long contractions give more (1 tile per XCD, 56 blocks 150 -> 126, these 139), and
// pieces of 128 rows x 128 columns no more than these.
__device__ __forceinline__ uint32_t row_shares(uint32_t left, uint32_t nwg) { return left == 0 || 2 * left > nwg ? 1 : 4 * left > nwg ? 2 : 4; }
// The last row that is loaded (a share may have none, and then loads one).
__host__ __device__ constexpr int last_row(int valid) { return valid > 0 ? valid - 1 : 0; }
// Bytes to the end of its block: 288 rows that are 8 MB apart are more than an int holds.
__host__ __device__ constexpr uint32_t rows_end(int valid, int64_t ld) { return (uint32_t)last_row(valid) * (uint32_t)ld + kBK; }
static_assert(rows_end(rows::high_tile(true), (1 << 23) - 1) == (int64_t)(rows::high_tile(true) - 1) * ((1 << 23) - 1) + kBK, "the rows of a tile are in reach of 32 bits");
// First contraction block of a part: whole groups of four (16 bytes of scales) but for the end of the last part.  With
// nkb >= 8 split every part has eight blocks or more.
__device__ __forceinline__ uint32_t row_part(uint32_t nkb, uint32_t split, uint32_t part) {
  return part == split ? nkb : 4u * ((nkb >> 2) * part / split);
}

// R_ROWS: the R operand is stored [contraction, Rrows] and its fragments are read transposed, see grouped_gemm_kernel.
// PAIRS: an even number of steps per tile, so that a step's number says which stage it works on and the stage goes into the
// immediate offset of its LDS reads; else the addresses change with every step (eight instructions more, 2 % of it).
// MORE: tiles of up to 32 rows more, see row_tiles_of.  EITHER: of a kernel that holds both forms, with the rows of the groups in the LDS.
template <typename OUT, bool R_ROWS, bool PAIRS, bool MORE, bool EITHER, typename ARGS>
__device__ __forceinline__ void row_tiles(ARGS& p, uint8_t* const lds) {
  // (the arguments of what is done once per tile are fetched there: scalar registers are short in the loop; in front of it
  // they come all at once)
  auto args = [&]() __attribute__((always_inline)) { return (const __attribute__((address_space(4))) GemmParams*)(uintptr_t)args_here(); };
  using namespace rows;
  constexpr int kScaleBatch = scale_batch(MORE);
  // [L stage 0 | L stage 1 | R stage 0 | R stage 1 | two stages of L rows beyond BM | two batches of scales | rows and tiles of the groups]
  float* const scales = reinterpret_cast<float*>(lds + 4 * kSide + (MORE ? 2 * kMoreSide : 0));
  int64_t* const table = reinterpret_cast<int64_t*>(lds + table_at(EITHER));

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hg = lane >> 5;

  // ---- the tiles of this workgroup ------------------------------------------------------------
  // Workgroup ids go round-robin over the 8 XCDs; every XCD gets one contiguous range of tile ids, in which tiles that share
  // operand panels are neighbours, and its workgroups take them side by side.
  GroupRanges gr = {};
  int total_lt = row_tiles_of<MORE>(p.Lrows), slices = -1;
  if (p.goff != nullptr) {
    gr = row_ranges<MORE>(EITHER ? GroupRows{table[lane * 3], table[lane * 3 + 1]} : group_rows(p.goff, p.E, 0), 0);
    total_lt = gr.total;
    for (int base = 64; base < p.E; base += 64) total_lt = row_ranges<MORE>(p.goff, p.E, base, total_lt).total;
    if (MORE && p.slices) {
      gr = row_slices<MORE>(GroupRows{table[lane * 3], table[lane * 3 + 1]}, (uint32_t)p.nRt, blockIdx.x & 7u);
      slices = gr.total;
    }
    if (p.E <= 64) {  // the group of every later tile is found from here
      if (!EITHER) {
        table[lane * 3] = gr.r_lo;
        table[lane * 3 + 1] = gr.r_hi;
      }
      table[lane * 3 + 2] = (int64_t)(((uint64_t)(uint32_t)gr.t_hi << 32) | (uint32_t)gr.t_lo);
    }  // (every wave writes the same values, and reads what it wrote)
  }
  const uint32_t nRt = (uint32_t)p.nRt, ntot = (uint32_t)total_lt * nRt;
  const uint32_t xcd = blockIdx.x & 7u, nwg = gridDim.x >> 3;
  RowTiles mine(ntot, xcd);
  if (slices >= 0) mine.first = 0, mine.end = (uint32_t)slices;

  // Workgroups that share a panel should stay the same ones: then the first of them to reach a block waits for memory and the
  // others catch up.  With short contractions, whose panels the L2 holds whole, a workgroup moves five places on with every round
  // instead, so that none gets the short last tile of every group.  (Places moved by 5 and by none, us: 32768 rows in 8 groups, 28672
  // x 4096 3425 and 3403, fetched beyond the L2 9.7 and 7.9 GB; 64 groups, 7168 x 2048 218 and 213; 4096 rows, 28672 x 4096 562 and
  // 554; 60 uneven groups, 2048 x 2816 228 and 229, 1408 x 2048 130 and 132, 2048 x 1408 (11 blocks) 134 and 138.)
  const uint32_t places = p.nkb >= 16 ? 0u : nwg > 5u ? 5u : 1u;
  uint32_t round_first = mine.first, turn = blockIdx.x >> 3;
  // the next tile of this workgroup, false if there is none; part and parts: of the contraction it takes, slot: where a part goes
  // (-1: of the tile's rows, see row_shares)
  uint32_t part = 0, parts = 1;
  int n_slot = -1;
  auto take = [&](uint32_t& pid) __attribute__((always_inline)) {
    const uint32_t left = mine.end > round_first ? mine.end - round_first : 0u;
    uint32_t at = turn;
    if (left < nwg && p.max_split > 1) {
      parts = row_split(left, part_places(MORE), (uint32_t)p.max_split);
      if (parts > 1) {
        n_slot = turn < left * parts ? (int)(xcd * part_places(MORE) + turn) : -1;
        part = turn / left;
        at = n_slot >= 0 ? turn - part * left : left;
      }
    }
    if (left < nwg && parts == 1) {
      parts = row_shares(left, nwg);
      if (parts > 1) {
        part = turn / left;
        at = turn < left * parts ? turn - part * left : left;
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
  // The tile under way and the next one are plain variables (as structures they would live in memory).  With MORE, where scalar
  // registers are shorter still, they lie in the LDS, a copy for each wave, and are read where they are used: 2 % of a tile of 32 steps.
  const uint32_t tile_words = lds_offset(lds) + (uint32_t)(table_at(true) + 64 * 3 * 8) + (uint32_t)(wave * 2 * kTileWords * 4);
  constexpr uint32_t kNext = kTileWords * 4;
  int64_t c_l0, n_l0;
  int c_g, c_lvalid, c_r0, c_rvalid, c_kb0, c_steps, c_slot, n_g, n_lvalid, n_r0, n_rvalid, n_kb0, n_steps;
  auto take_tile = [&](uint32_t id, auto a) __attribute__((always_inline)) {
    const RowTile t = row_tile<MORE>(a, opaque(a->goff != nullptr && a->E <= 64) ? table : nullptr, id, nRt, total_lt, xcd);
    int kb0 = 0, steps = t.steps, lvalid = t.lvalid;
    int64_t l0 = t.l0;
    if (n_slot >= 0) {
      kb0 = (int)row_part((uint32_t)t.steps, parts, part);
      steps = (int)row_part((uint32_t)t.steps, parts, part + 1) - kb0;
    } else if (parts > 1) {
      // (without rows, where the tile has few: a workgroup that stores nothing)
      const int size = (lvalid + 64 * (int)parts - 1) / (64 * (int)parts) * 64, from = (int)part * size, rest = lvalid - from;
      l0 += rest > 0 ? from : 0;
      lvalid = rest < 0 ? 0 : rest < size ? rest : size;
    }
    if constexpr (MORE) {
      put_words(tile_words + kNext, v4i{(int)(uint32_t)(uint64_t)l0, (int)((uint64_t)l0 >> 32), t.g, lvalid});
      put_words(tile_words + kNext + 16, v4i{t.r0, t.rvalid, kb0, steps});
      put_words(tile_words + kNext + 32, v4i{n_slot, 0, 0, 0});
    } else {
      n_l0 = l0, n_g = t.g, n_lvalid = lvalid, n_r0 = t.r0, n_rvalid = t.rvalid, n_kb0 = kb0, n_steps = steps;
    }
  };
  auto no_more_tiles = [&]() __attribute__((always_inline)) {
    if constexpr (MORE) put_words(tile_words + kNext + 32, v4i{0, 1, 0, 0});
  };
  auto next_is_current = [&]() __attribute__((always_inline)) {
    if constexpr (MORE) {
#pragma unroll
      for (uint32_t i = 0; i < kTileWords * 4; i += 16) copy_words(tile_words + i, tile_words + kNext + i);
      c_steps = word_here(tile_words + 28);
    } else {
      c_l0 = n_l0, c_g = n_g, c_lvalid = n_lvalid, c_r0 = n_r0, c_rvalid = n_rvalid, c_kb0 = n_kb0, c_steps = n_steps, c_slot = n_slot;
    }
  };
  auto tile_at = [&](uint32_t at) __attribute__((always_inline)) {
    const v4i u = words_here(at), v = words_here(at + 16);
    return RowTile{(int64_t)(((uint64_t)(uint32_t)u[1] << 32) | (uint32_t)u[0]), u[2], u[3], v[0], v[1], v[2], v[3]};
  };
  auto current = [&]() __attribute__((always_inline)) {
    if constexpr (MORE) return tile_at(tile_words);
    else return RowTile{c_l0, c_g, c_lvalid, c_r0, c_rvalid, c_kb0, c_steps};
  };
  auto slot_of_current = [&]() __attribute__((always_inline)) {
    if constexpr (MORE) return word_here(tile_words + 32);
    else return c_slot;
  };
  take_tile(pid, &p);
  next_is_current();

  // ---- loads -------------------------------------------------------------------------------------
  // A wave instruction of a tile load fills 1 KB of the LDS, lane l at base + 16 l; lane l fetches the chunk the swizzle puts
  // there.  n-th instruction of wave w: rows 8 w + 64 n .. + 7 of the tile (R_ROWS: contraction rows 4 w + 32 n .. + 3).
  const int r8 = lane >> 3;
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ r8 ^ (wave & 1)) << 4);
  const int rrow = R_ROWS ? wave * 4 + (lane >> 4) : wave * 8 + r8;
  // (where registers do not reach, the later ones are made where they are used: 3 % where all are)
  constexpr int kHeldL = !MORE ? 4 : R_ROWS || !PAIRS ? 1 : 2, kHeldR = kHeldL;
  uint32_t voffL[kHeldL], voffR[kHeldR];
  const uint32_t lstep = 64u * (uint32_t)p.ldl, rstep = (R_ROWS ? 32u : 64u) * (uint32_t)p.ldr;
#pragma unroll
  for (int n = 0; n < kHeldL; n++) voffL[n] = (uint32_t)(wave * 8 + 64 * n + r8) * (uint32_t)p.ldl + chunk;
#pragma unroll
  for (int n = 0; n < kHeldR; n++)
    voffR[n] = (uint32_t)(rrow + (R_ROWS ? 32 : 64) * n) * (uint32_t)p.ldr + (R_ROWS ? (uint32_t)(((lane & 15) ^ (2 * (rrow & 7))) << 4) : chunk);
  auto voff = [&](auto& of, auto HELD, uint32_t step, auto N) __attribute__((always_inline)) {
    constexpr int n = decltype(N)::value;
    if constexpr (n < decltype(HELD)::value) return +of[n];
    else return add_here(of[0], (uint32_t)n * step);
  };
  // Where the next block to be requested lies: it runs through the blocks of a tile and on into the next tile; behind the
  // last one it stays on the last block, to keep the wait counts uniform.
  v4i lbuf, rbuf;
  int to_load;         // blocks left in the tile
  int next_block = 0;  // of the next tile: 0, or the last one where that is still the tile under way
  int more_lanes = 0;  // that request rows beyond BM: all or none
  auto enter_next = [&](auto a) __attribute__((always_inline)) {
    RowTile t;
    int last;  // (no next tile: its last block once more)
    if constexpr (MORE) {
      t = tile_at(tile_words + kNext);
      last = word_here(tile_words + kNext + 36) != 0 ? t.steps - 1 : 0;
    } else {
      t = RowTile{n_l0, n_g, n_lvalid, n_r0, n_rvalid, n_kb0, n_steps};
      last = next_block;
    }
    const int block = t.kb0 + last;
    const int64_t l_at = t.l0 * a->ldl + block * kBK;
    const int64_t r_at = (int64_t)t.g * a->r_group_stride + (R_ROWS ? (int64_t)t.r0 : t.r0 * a->ldr) + block * a->r_kb_stride;
    lbuf = buffer_at(a->L + uniform_i64(l_at), (uint32_t)__builtin_amdgcn_readfirstlane((int)rows_end(t.lvalid, a->ldl)));
    rbuf = buffer_at(a->R + uniform_i64(r_at), (uint32_t)__builtin_amdgcn_readfirstlane(
                                                   R_ROWS ? 127 * (int)a->ldr + t.rvalid : (t.rvalid - 1) * (int)a->ldr + kBK));
    to_load = t.steps - last;
    if constexpr (MORE) more_lanes = __builtin_amdgcn_readfirstlane(t.lvalid > BM && wave < 4 ? -1 : 0);
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
    load_lds_x4<(PAIRS ? decltype(S)::value * kSide : 0) + decltype(N)::value * 8192>(voff(voffL, std::integral_constant<int, kHeldL>{}, lstep, N), lbuf, to_lds);
  };
  auto load_r = [&](auto S, auto N) __attribute__((always_inline)) {
    load_lds_x4<2 * kSide + (PAIRS ? decltype(S)::value * kSide : 0) + decltype(N)::value * 8192>(voff(voffR, std::integral_constant<int, kHeldR>{}, rstep, N), rbuf, to_lds);
  };
  // The rows beyond BM of the tile that is being requested, eight by each of waves 0 to 3; otherwise the instruction is there for no
  // lane, to keep the wait counts uniform (for lanes out of range it costs as much as a load: the loads take 9 % longer).
  const uint32_t more_rows = (uint32_t)BM * (uint32_t)p.ldl;
  uint32_t to_more = lds_offset(lds) + (uint32_t)(4 * kSide + (wave & 3) * 1024);
  auto load_more = [&](auto S) __attribute__((always_inline)) {
    load_lds_x4_for<(PAIRS ? decltype(S)::value * kMoreSide : 0)>(more_lanes, add_here(voffL[0], more_rows), lbuf, to_more);
  };
  auto load_tile = [&](auto S) __attribute__((always_inline)) {
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_l(S, N); });
    if constexpr (MORE) load_more(S);
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_r(S, N); });
  };
  auto other_stage = [&](auto TURN) __attribute__((always_inline)) {
    if constexpr (decltype(TURN)::value) {
      to_lds ^= kSide;
      if constexpr (MORE) to_more ^= kMoreSide;
    }
  };

  // Scales come in batches of eight contraction blocks (the last batch of a tile is shifted back to end at its last block): a
  // row of 32 bytes per L row and per 128 R rows.  Batch b of a tile is
  // requested in step 8 b - 3, batch 0 of the next tile in one of the last three steps (see `ask_next`), when the batch before
  // the one in use has been read for the last time.  Rows of scales that are not 16-byte aligned take 4-byte loads.
  const int x4 = p.ls_batch == 1;
  const uint32_t lsr = (uint32_t)p.ls_row_stride, rsr = (uint32_t)p.rs_row_stride, rsb = (uint32_t)p.rs_blk_stride;
  auto ask_scales = [&](const RowTile t, int b, int parity, auto a) __attribute__((always_inline)) {
    const int at = t.kb0 + (8 * b + 8 <= t.steps ? 8 * b : t.steps - 8), ln = lane_here();
    const v4i lb = buffer_at(a->Ls + uniform_i64(t.l0 * lsr + at), (uint32_t)__builtin_amdgcn_readfirstlane((last_row(t.lvalid) * (int)lsr + 8) * 4));
    const uint32_t ld = lds_offset(scales + parity * kScaleBatch) + (uint32_t)(wave * 1024);
    const int wide = opaque(x4);
    if (wide) {
      load_lds_x4<0>(((uint32_t)(wave * 32 + (ln >> 1)) * lsr + (uint32_t)(ln & 1) * 4u) * 4u, lb, ld);
    } else {
#pragma unroll
      for (int q = 0; q < 4; q++)
        load_lds_x1(((uint32_t)(wave * 32 + q * 8 + (ln >> 3)) * lsr + (uint32_t)(ln & 7)) * 4u, lb, ld + (uint32_t)(q * 256));
    }
    if (MORE && wave == 1 && t.lvalid > BM) {
      const uint32_t md = lds_offset(scales + parity * kScaleBatch) + BM * 32;
      if (wide) {
        load_lds_x4<0>(((uint32_t)(BM + (ln >> 1)) * lsr + (uint32_t)(ln & 1) * 4u) * 4u, lb, md);
      } else {
#pragma unroll
        for (int q = 0; q < 4; q++)
          load_lds_x1(((uint32_t)(BM + q * 8 + (ln >> 3)) * lsr + (uint32_t)(ln & 7)) * 4u, lb, md + (uint32_t)(q * 256));
      }
    }
    if (wave == 0) {
      const int blocks = t.rvalid / kTile;
      const v4i rb = buffer_at(a->Rs + uniform_i64((int64_t)t.g * a->rs_group_stride + (int64_t)(t.r0 / kTile) * rsr + (int64_t)at * rsb),
                               (uint32_t)__builtin_amdgcn_readfirstlane((R_ROWS ? 7 * (int)rsb + blocks : (blocks - 1) * (int)rsr + 8) * 4));
      const uint32_t rd = lds_offset(scales + parity * kScaleBatch + high_tile(MORE) * 8);
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
  int turned = 0;  // `wl`, where it is used
  // HIGH: in a tile with rows beyond BM a wave also makes one 32 x 32 sub-tile of these, from R sub-tile `wl`, which therefore is its
  // first: sub-tile i is the (i ^ wl)-th of its R half.
  auto fragR = [&](int s, int sub, int h, auto HIGH) __attribute__((always_inline)) {
    constexpr bool high = decltype(HIGH)::value;
    if constexpr (R_ROWS) {
      v8i f;
      uint32_t at = ra[sub / 2][sub % 2];
      if constexpr (high) at = xor_here(at, (uint32_t)(turned << 5));
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const v2i o = lds_read_transposed(at + (uint32_t)((PAIRS ? s * kSide : 0) + (64 * h + 8 * j) * BN));
        f[2 * j] = o[0];
        f[2 * j + 1] = o[1];
      }
      return f;
    } else if constexpr (high) {
      const uint32_t to = (uint32_t)((sub ^ turned) << 12);
      const v4i lo = *(lds_v4i_t)(uintptr_t)(xor_here(ra[h][0], to) + (uint32_t)(PAIRS ? s * kSide : 0));
      const v4i hi = *(lds_v4i_t)(uintptr_t)(xor_here(ra[h][1], to) + (uint32_t)(PAIRS ? s * kSide : 0));
      return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    } else {
      return frag(ra, s, sub, h);
    }
  };
  // of the rows beyond BM; from: what lies between a stage's first row of this wave and them
  auto frag_more = [&](int s, int h, uint32_t from) __attribute__((always_inline)) {
    const v4i lo = *(lds_v4i_t)(uintptr_t)(add_here(la[h][0], from) + (uint32_t)(PAIRS ? s * kMoreSide : 0));
    const v4i hi = *(lds_v4i_t)(uintptr_t)(add_here(la[h][1], from) + (uint32_t)(PAIRS ? s * kMoreSide : 0));
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  const uint32_t to_more_rows = (uint32_t)(4 * kSide - wlrow0 * kBK);  // (without PAIRS: from stage 0)
  auto barrier_q = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  v16f acc[WTR][WTL], pr;
  v8i lf[WTL][2], rf[2][2];
  float cs[WTL], csn[WTL], rblkn, cs_last = 0.f;
  // rows beyond BM: their fragments lie in rf[1] until the second R row comes
  v16f acc_more;
  float cm = 0.f, cmn = 0.f;
  uint32_t more_at = to_more_rows;

  // Scales of a block: the lane's L row scales and the wave's R block scale; sc_at: where the next block's are, sc_left: blocks
  // from there to the end of the batch, sc_more: batches of the tile behind it.
  int last_batch = 0, in_last = 0;  // of the tile under way: its last batch, and the blocks of it that are new
  int sc_parity = 0;  // of the tile's batch 0
  uint32_t sc_at = 0;
  int sc_left = 0, sc_more = 0;
  const uint32_t sc_l = lds_offset(scales) + (uint32_t)((wlrow0 + l32) * 32), sc_r = lds_offset(scales) + (uint32_t)(high_tile(MORE) * 32 + (wrow0 / kTile) * 32);
  auto read_scales = [&](auto HIGH) __attribute__((always_inline)) {
    typedef const __attribute__((address_space(3))) float* lds_float_t;
    const lds_float_t l = (lds_float_t)(uintptr_t)(sc_l + sc_at);
    rblkn = *(lds_float_t)(uintptr_t)(sc_r + sc_at);
#pragma unroll
    for (int j = 0; j < WTL; j++) csn[j] = l[j * 32 * 8];
    if constexpr (decltype(HIGH)::value) cmn = *(lds_float_t)(uintptr_t)add_here(sc_l, sc_at + (uint32_t)((BM - wlrow0) * 32));
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
  auto first_scales = [&](auto HIGH) __attribute__((always_inline)) {
    sc_at = (uint32_t)(sc_parity * kScaleBatch * 4);
    sc_left = 8;
    sc_more = last_batch;
    read_scales(HIGH);
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
  auto first_fragments = [&](auto HIGH) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      rf[0][h] = fragR(0, 0, h, HIGH);
      if constexpr (decltype(HIGH)::value) rf[1][h] = frag_more(0, h, more_at);
#pragma unroll
      for (int j = 0; j < WTL; j++) lf[j][h] = frag(la, 0, j, h);
    }
  };

  auto ask_in_step = [&](int kb) __attribute__((always_inline)) {
    if (kb != ask_at) return;
    const bool of_next = ask_batch > last_batch;
    if constexpr (MORE) {
      ask_scales(tile_at(tile_words + (of_next ? kNext : 0u)), of_next ? 0 : ask_batch, (sc_parity + ask_batch) & 1, args());
    } else {
      ask_scales(RowTile{of_next ? +n_l0 : +c_l0, of_next ? +n_g : +c_g, of_next ? +n_lvalid : +c_lvalid, of_next ? +n_r0 : +c_r0,
                         of_next ? +n_rvalid : +c_rvalid, of_next ? +n_kb0 : +c_kb0, of_next ? +n_steps : +c_steps},
                 of_next ? 0 : ask_batch, (sc_parity + ask_batch) & 1, args());
    }
    ask_batch++;
    ask_at = ask_batch <= last_batch ? kb + 8 : ask_batch == last_batch + 1 ? ask_next : -1;
  };

  constexpr int PT = (WTR - 1) * WTL - 1;  // the sub-tile in front of barrier P
  constexpr int kStores = NTILES * (sizeof(OUT) == 4 ? 4 : 2);  // of a wave and tile
  constexpr int kAhead = MORE ? 5 : 4;                          // loads of the L side of a step
  bool stored = false;
  // S: the stage (0 without PAIRS)
  auto step = [&](int kb, auto S, auto HIGH) __attribute__((always_inline)) {
    // (with rows beyond BM the stage changes in the addresses, as without PAIRS: S is 0 then)
    constexpr bool high = decltype(HIGH)::value, turn = !PAIRS || high;
    constexpr int s = decltype(S)::value, other = turn ? s : s ^ 1;
    __builtin_amdgcn_sched_barrier(0);
    barrier_q();
    __builtin_amdgcn_sched_barrier(0);
    fold(WTR - 1, WTL - 1, cs_last);  // owed by the step before (adds zero in the first one)
    if (turn) {
      other_l();
      if constexpr (high) more_at = 2 * to_more_rows + kMoreSide - kSide - more_at;
    }
    if constexpr (high) {
      __builtin_amdgcn_sched_barrier(0);
      pr = mfma_fp8_32x32x64(rf[0][0], rf[1][0], v16f{});
      pr = mfma_fp8_32x32x64(rf[0][1], rf[1][1], pr);
      asm volatile("" : "+v"(pr));
      __builtin_amdgcn_sched_barrier(0);
      load_more(S);
#pragma unroll
      for (int h = 0; h < 2; h++) rf[1][h] = fragR(s, 1, h, HIGH);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 16; r++) acc_more[r] = __builtin_fmaf(pr[r], cm, acc_more[r]);
      asm volatile("" : "+v"(acc_more));
    }
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
      if constexpr (MORE && t == 4 && !high) load_more(S);
      if constexpr (j == 0 && i + 1 < WTR && !(high && i == 0)) {
#pragma unroll
        for (int h = 0; h < 2; h++) rf[(i + 1) & 1][h] = fragR(s, i + 1, h, HIGH);
      }
      if constexpr (t == PT) {
        __builtin_amdgcn_sched_barrier(0);
        // all but this step's L tile loads have landed (loads and stores are counted in issue order; the stores of the tile
        // before were issued behind the loads this step waits for)
        if (kb == 0 && stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kAhead + kStores) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kAhead) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        ask_in_step(kb);
        if (turn) other_r();
        // row WTR - 2 has been consumed: its registers take the first R row of the next step
#pragma unroll
        for (int h = 0; h < 2; h++) rf[0][h] = fragR(other, 0, h, HIGH);
        read_scales(HIGH);
      }
      if constexpr (t > PT) {
        constexpr int jn = t - PT - 1;  // == j: this sub-tile was the last user of lf[j]
        load_r(S, std::integral_constant<int, 2 * jn>{});
        load_r(S, std::integral_constant<int, 2 * jn + 1>{});
#pragma unroll
        for (int h = 0; h < 2; h++) lf[jn][h] = frag(la, other, jn, h);
      }
      if constexpr (high && t + 1 == NTILES) {
#pragma unroll
        for (int h = 0; h < 2; h++) rf[1][h] = frag_more(other, h, more_at);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (t + 1 < NTILES) fold(i, j, cs[j]);
    });
    cs_last = cs[WTL - 1];
#pragma unroll
    for (int j = 0; j < WTL; j++) cs[j] = csn[j] * rblkn;
    if constexpr (high) cm = cmn * rblkn;
    advance();
    other_stage(std::integral_constant<bool, turn>{});
  };
  // a wave without valid rows: loads and barriers only, in the order of the working waves
  auto idle_step = [&](int kb, auto S) __attribute__((always_inline)) {
    barrier_q();
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_l(S, N); });
    if constexpr (MORE) load_more(S);
    if (kb == 0 && stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kAhead + kStores) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kAhead) : "memory");
    ask_in_step(kb);
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_r(S, N); });
    advance();
    other_stage(std::integral_constant<bool, !PAIRS>{});
  };

  // ---- a finished tile: registers -> memory
  // four columns of the bias
  auto bias_of = [&](auto a, int64_t at) __attribute__((always_inline)) {
    if (opaque(a->bias_dtype == AAMD_F32)) return *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(a->bias) + at);
    const v2i raw = *reinterpret_cast<const v2i*>(reinterpret_cast<const u16*>(a->bias) + at);
    return v4f{bf16_bits_to_f32((uint32_t)raw[0] & 0xffffu), bf16_bits_to_f32((uint32_t)raw[0] >> 16),
               bf16_bits_to_f32((uint32_t)raw[1] & 0xffffu), bf16_bits_to_f32((uint32_t)raw[1] >> 16)};
  };
  // The sub-tile of the rows beyond BM; then the wave's sub-tiles i and i + 1 change places where `wl` is odd, so that they are
  // side by side again.
  auto store_more = [&](const RowTile t) __attribute__((always_inline)) {
    const auto a = args();
    const int w_r = opaque_s(wrow0), wl = opaque_s(wlrow0 / (WTL * 32)), rows = t.lvalid - BM, slot = slot_of_current();
    if (opaque(slot >= 0)) {
      const v4i out = buffer_at(a->ws + ((int64_t)slot * (high_tile(MORE) * BN) + BM * BN + w_r + wl * 32), ((uint32_t)(rows - 1) * BN + 32u) * 4u);
      store_sub_tile<float>(acc_more, lane_here(), BN, out);
    } else {
      if (opaque(a->bias != nullptr)) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const v4f b = bias_of(a, (int64_t)t.g * a->bias_group_stride + t.r0 + w_r + wl * 32 + 8 * q + 4 * (lane_here() >> 5));
#pragma unroll
          for (int r = 0; r < 4; r++) acc_more[4 * q + r] += b[r];
        }
      }
      const v4i out = buffer_at(reinterpret_cast<OUT*>(a->C) + ((t.l0 + BM) * a->ldc + t.r0 + w_r + wl * 32),
                                ((uint32_t)(rows - 1) * (uint32_t)a->ldc + 32u) * (uint32_t)sizeof(OUT));
      store_sub_tile<OUT>(acc_more, lane_here(), (uint32_t)a->ldc, out);
    }
    if (wl & 1) {
#pragma unroll
      for (int i = 0; i < WTR; i += 2)
#pragma unroll
        for (int j = 0; j < WTL; j++) {
          const v16f u = acc[i][j];
          acc[i][j] = acc[i + 1][j];
          acc[i + 1][j] = u;
        }
    }
  };
  // swap: 2 where the wave's second pair of sub-tiles comes first
  auto store_tile = [&](const RowTile t, int swap) __attribute__((always_inline)) {
    const auto a = args();
    constexpr uint32_t kEl = sizeof(OUT);
    const int w_r = MORE ? opaque_s(wrow0) : wrow0, w_l = MORE ? opaque_s(wlrow0) : wlrow0, left = t.lvalid - w_l, rows = left < 64 ? left : 64, slot = slot_of_current();
    if (opaque(slot >= 0)) {  // a part: as it is, into the workspace
      const v4i out = buffer_at(a->ws + ((int64_t)slot * (high_tile(MORE) * BN) + w_l * BN + w_r), ((uint32_t)(rows - 1) * BN + 128u) * 4u);
      const uint32_t at = store_offset<float>(lane_here(), BN);
      static_for<NTILES / 2>([&](auto T) __attribute__((always_inline)) {
        constexpr int i = 2 * (decltype(T)::value % (WTR / 2)), j = decltype(T)::value / (WTR / 2);
        constexpr int kCol = MORE ? 0 : i * 32;  // (in the instruction, where it is known)
        store_sub_tiles<float, kCol, false>(acc[i][j], acc[i + 1][j], at + (uint32_t)((j * 32 * BN + (i ^ swap) * 32 - kCol) * 4), BN, out);
      });
      return;
    }
    const v4i out = buffer_at(reinterpret_cast<OUT*>(a->C) + ((t.l0 + w_l) * a->ldc + t.r0 + w_r),
                              ((uint32_t)(rows - 1) * (uint32_t)a->ldc + 128u) * kEl);
    const int ln = lane_here(), h5 = ln >> 5;
    const uint32_t at = store_offset<OUT>(ln, (uint32_t)a->ldc);
    if (opaque(a->bias != nullptr)) {
#pragma unroll
      for (int i = 0; i < WTR; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const v4f b = bias_of(a, (int64_t)t.g * a->bias_group_stride + t.r0 + w_r + (i ^ swap) * 32 + 8 * q + 4 * h5);
#pragma unroll
          for (int j = 0; j < WTL; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][4 * q + r] += b[r];
        }
    }
    auto store_as = [&](auto nt) __attribute__((always_inline)) {
      static_for<NTILES / 2>([&](auto T) __attribute__((always_inline)) {
        constexpr int i = 2 * (decltype(T)::value % (WTR / 2)), j = decltype(T)::value / (WTR / 2);
        constexpr int kCol = MORE ? 0 : i * 32;
        store_sub_tiles<OUT, kCol, decltype(nt)::value>(acc[i][j], acc[i + 1][j], at + ((uint32_t)(j * 32) * (uint32_t)a->ldc + (uint32_t)((i ^ swap) * 32 - kCol)) * kEl,
                                                        (uint32_t)a->ldc, out);
      });
    };
    if (opaque(a->stream_out)) store_as(std::true_type{});
    else store_as(std::false_type{});
  };

  // ---- the first tile's blocks 0 and 1
  constexpr std::integral_constant<int, 0> S0{};
  constexpr std::integral_constant<int, 1> S1{};
  constexpr std::integral_constant<bool, !PAIRS> kTurn{};
  load_tile(S0);
  ask_scales(current(), 0, 0, &p);
  advance_buffer(lbuf, kBK);
  advance_buffer(rbuf, p.r_kb_stride);
  other_stage(kTurn);
  load_tile(S1);
  advance_buffer(lbuf, kBK);
  advance_buffer(rbuf, p.r_kb_stride);
  other_stage(kTurn);
  to_load -= 2;

  bool first = true;
  for (;;) {
    const bool more = take(pid);
    if (more) take_tile(pid, args());
    else no_more_tiles();
    if constexpr (!MORE) next_block = more ? 0 : n_steps - 1;
    last_batch = (c_steps - 1) >> 3;
    in_last = c_steps - 8 * last_batch;
    first_ask();
    if (first) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kAhead + 4) : "memory");  // the first tile's block 0 and scales
    first = false;
    const int high = MORE ? word_here(tile_words + 12) : +c_lvalid;
    const bool work = wrow0 < (MORE ? word_here(tile_words + 20) : +c_rvalid) && wlrow0 < high;
    if (work) {
#pragma unroll
      for (int i = 0; i < WTR; i++)
#pragma unroll
        for (int j = 0; j < WTL; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++) pr[r] = 0.f;
      cs_last = 0.f;
      auto all_steps = [&](auto HIGH) __attribute__((always_inline)) {
        first_fragments(HIGH);
        first_scales(HIGH);
#pragma unroll
        for (int j = 0; j < WTL; j++) cs[j] = csn[j] * rblkn;
        if constexpr (decltype(HIGH)::value) cm = cmn * rblkn;
        for (int kb = 0; kb < c_steps; kb++) {
          step(kb, S0, HIGH);
          if constexpr (PAIRS && !decltype(HIGH)::value) step(++kb, S1, HIGH);
        }
        __builtin_amdgcn_sched_barrier(0);
        fold(WTR - 1, WTL - 1, cs_last);
      };
      int swap = 0;
      if (MORE && opaque_s(high) > BM) {
        turned = opaque_s(wl);
        more_at = to_more_rows;
        if (!PAIRS)
          more_at = to_more_rows - ((((uint32_t)__builtin_amdgcn_readfirstlane((int)la[0][0]) - lds_offset(lds)) / kSide) & 1u) * (uint32_t)(kSide - kMoreSide);
#pragma unroll
        for (int r = 0; r < 16; r++) acc_more[r] = 0.f;
        all_steps(std::true_type{});
        store_more(current());
        swap = turned & 2;
      } else {
        all_steps(std::false_type{});
      }
      store_tile(current(), MORE ? swap : 0);
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

// EITHER: with tiles of up to 32 rows more where the groups' rows make them worth it.  (A kernel of its own: holding both forms and
// deciding take 0.2 to 0.5 us.)
template <typename OUT, bool R_ROWS, bool PAIRS, bool EITHER>
__global__ __launch_bounds__(rows::NT, 1) void row_tiles_kernel(const GemmParams p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[rows::lds_bytes(EITHER)];
  if constexpr (EITHER) {
    typedef const __attribute__((address_space(4))) GemmParams* args_t;
    // the rows of the first 64 groups: fetched once, into the place where the groups of later tiles are looked up
    GroupRows of_lane = {0, 0};
    if (p.goff != nullptr) {
      of_lane = group_rows(p.goff, p.E, 0);
      int64_t* const table = reinterpret_cast<int64_t*>(lds + rows::table_at(true)) + (threadIdx.x & 63) * 3;
      table[0] = of_lane.lo;
      table[1] = of_lane.hi;
    }  // (every wave writes the same values, and reads what it wrote)
    // (the form of more rows fetches its arguments itself: what both used would be fetched in front, and held.  The other takes them as they
    // come, all at once: a launch that decides against more rows, 4096 rows in 8 groups, 4736 x 1024 31.9 us without the choice, 32.1 with
    // it, 32.7 where this form too fetched them one by one)
    if (higher_tiles(&p, of_lane)) row_tiles<OUT, R_ROWS, PAIRS, true, true>(*(args_t)(uintptr_t)args_here(), lds);
    else row_tiles<OUT, R_ROWS, PAIRS, false, true>(p, lds);
  } else {
    row_tiles<OUT, R_ROWS, PAIRS, false, false>(p, lds);
  }
}

// The sums of the parts of the tiles that row_tiles_kernel has split, in the order of the contraction, with the bias: eight XCDs x
// tiles left in the last round x eight slices of 32 rows.  Bound by memory, of which some is still in the caches: 12 tiles per XCD
// in two parts, 50 MB, 17 us; slices of 32 rows make 768 workgroups of them, and one load of 16 bytes per lane and part is
// in flight for each of eight rows.
template <typename OUT, bool MORE, bool EITHER>
__device__ __forceinline__ void row_parts(const GemmParams& p, const GroupRows& of_lane, int64_t* table) {
  using namespace rows;
  constexpr int kSlices = high_tile(EITHER) / 32, kRows = 32;
  constexpr uint32_t nwg = kWorkgroups / 8;
  const uint32_t xcd = blockIdx.x & 7u, j = (blockIdx.x >> 3) / kSlices, slice = (blockIdx.x >> 3) % kSlices;
  int total_lt = row_tiles_of<MORE>(p.Lrows);
  GroupRanges gr = {};
  if (p.goff != nullptr) {
    gr = row_ranges<MORE>(of_lane, 0);
    total_lt = gr.total;
    for (int base = 64; base < p.E; base += 64) total_lt = row_ranges<MORE>(p.goff, p.E, base, total_lt).total;
  }
  RowTiles mine((uint32_t)total_lt * (uint32_t)p.nRt, xcd);
  const bool in_table = p.goff != nullptr && p.E <= 64;
  if (in_table) {
    if (MORE && p.slices) {
      gr = row_slices<MORE>(of_lane, (uint32_t)p.nRt, xcd);
      mine.first = 0;
      mine.end = (uint32_t)gr.total;
    }
    int64_t* const of = table + (threadIdx.x & 63) * 3;
    of[0] = gr.r_lo;
    of[1] = gr.r_hi;
    of[2] = (int64_t)(((uint64_t)(uint32_t)gr.t_hi << 32) | (uint32_t)gr.t_lo);
  }  // (every wave writes the same values, and reads what it wrote)
  const uint32_t left = (mine.end - mine.first) % nwg, parts = row_split(left, part_places(MORE), (uint32_t)p.max_split);
  if (parts < 2 || j >= left) return;
  const RowTile t = row_tile<MORE>(&p, in_table ? table : nullptr, mine.end - left + j, (uint32_t)p.nRt, total_lt, xcd);
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
  const float* const from = p.ws + ((int64_t)(xcd * part_places(MORE) + j) * (high_tile(MORE) * BN) + col);
#pragma unroll
  for (int r = 0; r < kRows; r += 4) {
    const int row = row0 + r;
    if (row >= t.lvalid) return;
    v4f sum = *reinterpret_cast<const v4f*>(from + row * BN);
    for (uint32_t i = 1; i < parts; i++) sum += *reinterpret_cast<const v4f*>(from + (int64_t)(i * left) * (high_tile(MORE) * BN) + row * BN);
    sum += b;
    OUT* const out = reinterpret_cast<OUT*>(p.C) + (t.l0 + row) * p.ldc + t.r0 + col;
    if constexpr (sizeof(OUT) == 4) *reinterpret_cast<v4f*>(out) = sum;
    else *reinterpret_cast<v2i*>(out) = v2i{(int)pack_bf16x2(sum[0], sum[1]), (int)pack_bf16x2(sum[2], sum[3])};
  }
}

template <typename OUT, bool EITHER>
__global__ __launch_bounds__(256) void row_parts_kernel(const GemmParams p) {
  __shared__ int64_t table[64 * 3];
  const GroupRows of_lane = p.goff != nullptr ? group_rows(p.goff, p.E, 0) : GroupRows{0, 0};
  if constexpr (EITHER) {
    if (higher_tiles(&p, of_lane)) return row_parts<OUT, true, true>(p, of_lane, table);
  }
  row_parts<OUT, false, EITHER>(p, of_lane, table);
}

template <typename OUT, bool R_ROWS, bool EITHER>
static void launch_row_tiles_as(const GemmParams& p, unsigned blocks, hipStream_t st) {
  if (p.nkb % 2 == 0) row_tiles_kernel<OUT, R_ROWS, true, EITHER><<<blocks, rows::NT, 0, st>>>(p);
  else row_tiles_kernel<OUT, R_ROWS, false, EITHER><<<blocks, rows::NT, 0, st>>>(p);
  if (p.max_split > 1) {
    // (a tile is split where at most half the workgroups have one)
    const unsigned sums = 8 * (rows::kWorkgroups / 8 / 2) * (rows::high_tile(EITHER) / 32);
    row_parts_kernel<OUT, EITHER><<<sums, 256, 0, st>>>(p);
  }
}
template <bool EITHER>
static void launch_row_tiles_of(const GemmParams& p, int c_dtype, unsigned blocks, bool r_rows, hipStream_t st) {
  if (c_dtype == AAMD_BF16) r_rows ? launch_row_tiles_as<u16, true, EITHER>(p, blocks, st) : launch_row_tiles_as<u16, false, EITHER>(p, blocks, st);
  else r_rows ? launch_row_tiles_as<float, true, EITHER>(p, blocks, st) : launch_row_tiles_as<float, false, EITHER>(p, blocks, st);
}
// Both halves of the launches, one in each unit that is made of this file (gemm_rows_higher.hip).
void launch_row_tiles_higher(const GemmParams& p, int c_dtype, unsigned blocks, bool r_rows, hipStream_t st);
#ifdef AAMD_ROW_TILES_HIGHER
void launch_row_tiles_higher(const GemmParams& p, int c_dtype, unsigned blocks, bool r_rows, hipStream_t st) {
  launch_row_tiles_of<true>(p, c_dtype, blocks, r_rows, st);
}
#else
int launch_row_tiles(GemmParams p, int c_dtype, int64_t tiles, bool r_rows, hipStream_t st) {
  AAMD_REQUIRE(tiles < 0x7fffffffLL, "grouped_gemm: grid too large");
  unsigned blocks = (unsigned)std::min<int64_t>((tiles + 7) / 8 * 8, rows::kWorkgroups);
  // Streaming stores keep a large output from evicting the operands from the last-level cache, and cost a launch that is short
  // of steps to hide them (us, plain and streaming: 4096 x 32768 outputs (268 MB), contraction 4096 492 -> 464, 2048 267 -> 272,
  // 1024 160 -> 175; 32768 x 28672 (1.9 GB), 4096 3449 -> 3414; 4096 x 14336 (117 MB), 4096 222 both).
  p.stream_out = p.nkb >= 32 && p.Lrows * p.Rrows * (c_dtype == AAMD_BF16 ? 2 : 4) >= (int64_t)1 << 28;
  if (p.max_split > 1) blocks = rows::kWorkgroups;
  if (p.higher >= 0) launch_row_tiles_higher(p, c_dtype, blocks, r_rows, st);
  else launch_row_tiles_of<false>(p, c_dtype, blocks, r_rows, st);
  AAMD_LAUNCH_CHECK("grouped_gemm (256 x 256 tiles)");
  return AAMD_OK;
}
#endif

}  // namespace aamd
