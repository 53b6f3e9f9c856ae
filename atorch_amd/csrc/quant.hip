// Memory-bound quantisation kernels for gfx950: 1x128 tile quant (optionally with the token
// permute fused in as a scatter), row-wise + transposed quant of ragged groups in one pass,
// 128x128 block quant with the transposed copy, and dequant.
//
// All of them stream HBM with 128-bit accesses; amax reductions over a 128-element tile run
// inside one 16-lane DPP row.  Scales and codes are part of a bit-exact contract, so every
// quotient gives the code of the correctly rounded one (the IEEE division or its checked two-instruction form).
#include <atomic>
#include <mutex>

#include "quant.hpp"

namespace aamd {

static __device__ __attribute__((aligned(16))) u16 g_gelu_lut[2 * kLutN];
static __device__ __attribute__((aligned(16))) float g_gelub_lut[2 * kLutN];
__global__ __launch_bounds__(256) void gelu_lut_kernel() {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= 2 * kLutN) return;
  const uint32_t sign = i >= kLutN ? 1u : 0u;
  const float x = __uint_as_float(((sign << 15) | (kLutLo + i - sign * kLutN)) << 16);
  g_gelu_lut[i] = (u16)f32_to_bf16_bits(x * gelu_phi(x));
  g_gelub_lut[i] = gelu_grad_factor(x);
}
// ---------------------------------------------------------------------------------------
// 1x128 quant, 16 lanes per tile, U tiles per lane group.  SCATTER: write each quantised
// row to its topk destinations (row_map), reading it once.
// ---------------------------------------------------------------------------------------
// floor(n / d) for n < 2^31 as one widening multiply and a shift: magic = floor(2^sh / d) + 1, sh = 31 + ceil(log2 d)
struct FastDiv {
  uint32_t magic;
  int sh;
  __device__ __forceinline__ uint32_t div(uint32_t n) const { return (uint32_t)(((uint64_t)n * magic) >> sh); }
};
static FastDiv make_fastdiv(uint32_t d) {
  int l = 0;
  while (((uint64_t)1 << l) < d) l++;
  FastDiv f;
  f.sh = 31 + l;
  f.magic = (uint32_t)((((uint64_t)1 << f.sh) / (uint64_t)d) + 1);
  return f;
}

// tiles per 16-lane group and pass: two keep enough loads in flight (one and four measured slower)
constexpr int kQuantU = 2;
constexpr int64_t kMaxRowLd = (int64_t)1 << 24;  // row strides (elements) of the row-wise quantisers' inputs
// A workgroup takes 16 U consecutive tiles of the row-major tile order.  These kernels run close to the rate at
// which the vector ALUs issue, so nothing that is the same in every lane is computed in the lanes: the position
// of the block's first tile comes from the scalar unit, a lane adds its small tile number to it, and every
// access is a scalar base plus a 32-bit lane offset.  The outputs are dense, so tile t of the order lies at
// byte 128 t of q; the input needs (row, column tile) only where its rows are strided.
// (the launchers keep ldx below 2^24: 16 U rows of it stay within the 32-bit offset)
template <typename IN, bool SCATTER, int U>
__device__ __forceinline__ void quant_1x128_tiles(const typename IN::elem* __restrict__ x, int64_t ldx,
                                                  int nt, FastDiv nt_div, int64_t total_tiles,
                                                  const int32_t* __restrict__ row_map, int topk,
                                                  int64_t M_out, uint8_t* __restrict__ q,
                                                  float* __restrict__ s, float eps, int64_t gate_off,
                                                  u16* __restrict__ h_out) {
  // the short division is checked for bf16 values over scales of bf16 maxima only
  const bool plain_div = !kBf16Values<IN> || eps != 0.f;
  const int grp = threadIdx.x >> 4, l = threadIdx.x & 15;
  constexpr uint32_t kEl = sizeof(typename IN::elem);
  const int64_t base = (int64_t)blockIdx.x * (16 * U);  // first tile of the block: the same in every lane
  const int64_t tiles_left = total_tiles - base;
  const uint32_t left = tiles_left < 16 * U ? (uint32_t)tiles_left : 16u * U;  // >= 1
  const int64_t cols = (int64_t)nt * kTile;
  const bool dense = !SCATTER && ldx == cols;
  int64_t row0 = 0;
  uint32_t tc0 = 0;
  if (!dense) {
    row0 = total_tiles < ((int64_t)1 << 31) ? (int64_t)nt_div.div((uint32_t)base) : base / nt;
    tc0 = (uint32_t)(base - row0 * nt);
  }
  const typename IN::elem* const xb = dense ? x + base * kTile : x + row0 * ldx;

  Raw8<IN> raw[U];
  uint32_t jt[U], wrow[U], tc[U];
  bool valid[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    uint32_t j = (uint32_t)(u * 16 + grp);
    valid[u] = j < left;
    if (!valid[u]) j = left - 1;
    jt[u] = j;
    uint32_t xoff;  // elements from xb
    if (dense) {
      xoff = j * kTile;
      wrow[u] = tc[u] = 0;
    } else {
      const uint32_t t = tc0 + j;  // below nt + 16 U
      wrow[u] = nt >= 16 * U ? (t >= (uint32_t)nt ? 1u : 0u) : nt_div.div(t);
      tc[u] = t - wrow[u] * (uint32_t)nt;
      xoff = wrow[u] * (uint32_t)ldx + tc[u] * kTile;
    }
    raw[u].load(xb, (xoff + (uint32_t)l * 8) * kEl, gate_off);
  }
  u16* const hb = h_out ? h_out + base * kTile : nullptr;
  uint8_t* const qb = q + base * kTile;
  float* const sb = s + base;
#pragma unroll
  for (int u = 0; u < U; u++) {
    float v[8];
    raw[u].get(v);
    const Divider dv = make_scale(row16_max(amax8(v)), eps, plain_div);
    const float sc = dv.s;
    const v2i codes = quant8(v, dv);
    if (!valid[u]) continue;
    const uint32_t off = jt[u] * kTile + (uint32_t)l * 8;  // element of the dense outputs, from the block's first tile
    if (h_out != nullptr) st_nt(hb, off * 2, pack8_bf16(v));  // the activation itself, for callers that keep it
    // the codes are not read again by this kernel: streaming stores keep them out of the way
    if constexpr (!SCATTER) {
      st_nt(qb, off, codes);
      if (l == 0) sb[jt[u]] = sc;
    } else {
      const int64_t row = row0 + wrow[u];
      for (int j = 0; j < topk; j++) {
        const int64_t dst = row_map[row * topk + j];
        if (dst < 0 || dst >= M_out) continue;
        __builtin_nontemporal_store(codes, reinterpret_cast<v2i*>(q + dst * cols + (int64_t)tc[u] * kTile + l * 8));
        if (l == 0) s[dst * nt + tc[u]] = sc;
      }
    }
  }
}

template <typename IN, bool SCATTER, int U>
__global__ __launch_bounds__(256) void quant_1x128_kernel(const typename IN::elem* __restrict__ x, int64_t ldx,
                                                          int nt, FastDiv nt_div, int64_t total_tiles,
                                                          const int32_t* __restrict__ row_map, int topk,
                                                          int64_t M_out, uint8_t* __restrict__ q,
                                                          float* __restrict__ s, float eps, int64_t gate_off,
                                                          u16* __restrict__ h_out) {
  quant_1x128_tiles<IN, SCATTER, U>(x, ldx, nt, nt_div, total_tiles, row_map, topk, M_out, q, s, eps, gate_off, h_out);
}
// The rows of a grouped product whose groups' sizes are a host list: one workgroup more stores the offsets, which come as an
// argument, for the launches behind this one (2048 rows in 4 groups, 512 x 1024: a launch of 1.4 us and its gap less).
constexpr int kOffsetsHere = 64;
struct OffsetsHere {
  int32_t v[kOffsetsHere + 1];
  int n;
};
template <typename IN, int U>
__global__ __launch_bounds__(256) void quant_1x128_offsets_kernel(const typename IN::elem* __restrict__ x, int64_t ldx, int nt,
                                                                  FastDiv nt_div, int64_t total_tiles, uint8_t* __restrict__ q,
                                                                  float* __restrict__ s, float eps, int64_t rows,
                                                                  const OffsetsHere off, int64_t* __restrict__ goff) {
  if (blockIdx.x == gridDim.x - 1) {
    if ((int)threadIdx.x < off.n) goff[threadIdx.x] = off.v[threadIdx.x];
    return;
  }
  quant_1x128_tiles<IN, false, U>(x, ldx, nt, nt_div, total_tiles, nullptr, 1, rows, q, s, eps, 0, nullptr);
}

// ---------------------------------------------------------------------------------------
// 128x128 register tile shared by the dual (row + transposed) quant and the block quant:
// 256 threads, thread (gr = tid/16, c = tid%16) holds rows gr*8 .. gr*8+7, columns c*8 .. c*8+7.
// ---------------------------------------------------------------------------------------
constexpr int kTLd = kTile + 16;  // LDS row stride (bytes) of the transposed code tile
// 128 rows of a tile are addressed with 32-bit byte offsets: row strides (elements, at most 4 bytes each) stay below this
constexpr int64_t kMaxTileLd = (int64_t)1 << 22;

// A row past the group's end: zeros, or, where the activation comes from a table, values that are in it: zeros are not,
// and took a tile of few rows through the out-of-line arithmetic, a call per pair (60 groups of 68 rows, 1408 columns,
// GELU and its backward 27 -> 14 and 30 -> 15 us, SwiGLU backward 31 -> 23; 8 groups of 125 rows, 4096 columns, GELU 21 ->
// 11; 32764 rows in 60 uneven groups 61 -> 49 and 70 -> 58).  The GELU's own result is cleared by its reader.
constexpr v4i kOnes = {0x3f803f80, 0x3f803f80, 0x3f803f80, 0x3f803f80};  // bf16
template <typename IN>
__device__ __forceinline__ void absent_row(Raw8<IN>& raw) {
  raw.zero();
  if constexpr (std::is_same<IN, GELU>::value || std::is_same<IN, GELUB>::value) raw.a = kOnes;
}
// `x` is the tile's origin, the same in every lane; FULL: all 128 rows are valid
template <typename IN, bool FULL>
__device__ __forceinline__ void issue_tile_loads(const typename IN::elem* __restrict__ x, uint32_t ldx, int rows_valid,
                                                 Raw8<IN> (&raw)[8], int64_t gate_off = 0) {
  const int gr = (int)threadIdx.x >> 4, c = (int)threadIdx.x & 15;
  constexpr uint32_t kEl = sizeof(typename IN::elem);
  const uint32_t off0 = ((uint32_t)(gr * 8) * ldx + (uint32_t)c * 8) * kEl;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    if (FULL || gr * 8 + i < rows_valid)
      raw[i].load(x, off0 + (uint32_t)i * ldx * kEl, gate_off);
    else
      absent_row(raw[i]);
  }
}
template <typename IN, bool FULL>
__device__ __forceinline__ void load_tile(const typename IN::elem* __restrict__ x, uint32_t ldx, int rows_valid,
                                          float (&v)[8][8], int64_t gate_off = 0) {
  Raw8<IN> raw[8];
  issue_tile_loads<IN, FULL>(x, ldx, rows_valid, raw, gate_off);
#pragma unroll
  for (int i = 0; i < 8; i++) raw[i].get(v[i]);
}

// Byte `b` of row `r` of the staged code tile.  A thread writes the few codes it holds of a row, and the lanes
// c = 0..15 of a wave do so in rows eight apart: 8 * 144 bytes is a multiple of 128, so without more ado sixteen
// lanes would meet in one or two LDS banks.  The 16-byte chunk index inside the row is therefore XORed with three
// bits of the row: the 64 lanes of a write then spread evenly over all banks, and a row is still read back as
// eight whole 16-byte chunks, in permuted order.
__device__ __forceinline__ int staged_off(int r, int b) { return r * kTLd + (b ^ (((r >> 4) & 7) << 4)); }

// the staged 128 x 128 code tile written as rows of 128 bytes, one 16-byte store per lane
// (`out`: the tile's origin, the same in every lane; 128 ld_out < 2^32)
__device__ __forceinline__ void store_staged_tile(const uint8_t* tile_t, uint8_t* __restrict__ out, uint32_t ld_out) {
  __syncthreads();
#pragma unroll
  for (int n = 0; n < 4; n++) {
    const int idx = (int)threadIdx.x + 256 * n;
    const int r = idx >> 3, ch = idx & 7;
    st_nt(out, (uint32_t)r * ld_out + (uint32_t)ch * 16, *reinterpret_cast<const v4i*>(tile_t + staged_off(r, ch * 16)));
  }
}

// Where tile (token tile pt, column tile kc) of the transposed codes goes, and the stride of its 128 rows.
// Layout 0: q_t is [cols, ld_t], a row per column of x; layout 1 (AAMD_QT_BLOCKED): q_t is [ld_t / 128, cols, 128],
// token-block-major, so that a tile is 16 KB of consecutive bytes and the tiles of a token block follow each other:
// the kernel then writes the transposed codes as one sequential sweep instead of 128-byte pieces ld_t apart.
__device__ __forceinline__ uint8_t* qt_tile(uint8_t* q_t, int blocked, int64_t cols, uint32_t ld_t, int pt, int kc, uint32_t* ld) {
  *ld = blocked == AAMD_QT_BLOCKED ? (uint32_t)kTile : ld_t;
  return blocked == AAMD_QT_BLOCKED ? q_t + ((int64_t)pt * cols + (int64_t)kc * kTile) * kTile
                 : q_t + (int64_t)kc * kTile * ld_t + (int64_t)pt * kTile;
}

// One 128 x 128 tile of the dual quantiser: token tile pt of group g, column tile kc.  Everything that
// locates the tile is the same in every lane, so each access is a scalar base plus a 32-bit lane offset
// (the launchers bound the row strides so that 128 rows stay below 2^32 bytes).
// GATHER: row r of the tile is source row src_row[r] of x (the token permute fused in: x is in token order,
// the outputs in expert-contiguous order); src_row lives in LDS and holds every valid row of the tile.
// SUMS: the tile's column sums (a bias gradient's share of these 128 tokens) go to tile_sums[pt, column].
// WEIGHTED (with GATHER): row r is multiplied by row_w[r], which lives in LDS too, and rounded to bf16.
template <typename IN, bool FULL, bool GATHER = false, bool SUMS = false, bool WEIGHTED = false>
__device__ __forceinline__ void dual_tile(const typename IN::elem* __restrict__ x, uint32_t ldx, int nt, int64_t m0,
                                          int mvalid, int pt, int kc, uint8_t* __restrict__ q, float* __restrict__ s,
                                          uint8_t* __restrict__ q_t, float* __restrict__ s_t, uint32_t ld_t, int blocked,
                                          float eps, int64_t gate_off, u16* __restrict__ h_out, uint8_t* tile_t,
                                          Divider* cdiv, const uint32_t* src_row = nullptr, const void* lut = nullptr,
                                          float* __restrict__ tile_sums = nullptr, const float* row_w = nullptr) {
  const bool plain_div = !(kBf16Values<IN> || WEIGHTED) || eps != 0.f;  // see make_scale
  float (*part)[kTile] = reinterpret_cast<float (*)[kTile]>(tile_t);
  const int64_t cols = (int64_t)nt * kTile;
  const int gr = (int)threadIdx.x >> 4, c = (int)threadIdx.x & 15;

  // The GELU kernels hold their results, which are bf16 numbers, packed two to a register until the column pass
  // (the erf evaluation needs the registers: unpacked, two workgroups fit on a CU instead of four).  For the other
  // inputs the 64 values of a thread stay in fp32: the packed form compiles to more registers there, not fewer.
  constexpr bool kPacked = std::is_same<IN, GELU>::value || std::is_same<IN, GELUB>::value;
  Raw8<IN> raw[8];
  if constexpr (GATHER) {
    // a row's 256-byte segment (16 lanes x 16 bytes) stays one coalesced access; only its base is looked up
    constexpr uint32_t kEl = sizeof(typename IN::elem);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (FULL || gr * 8 + i < mvalid)
        raw[i].load(x + (int64_t)src_row[gr * 8 + i] * ldx + (int64_t)kc * kTile, (uint32_t)c * 8 * kEl, gate_off);
      else
        absent_row(raw[i]);
    }
  } else {
    issue_tile_loads<IN, FULL>(x + m0 * ldx + (int64_t)kc * kTile, ldx, mvalid, raw, gate_off);
  }
  float v[kPacked ? 1 : 8][8];
  uint32_t vp[kPacked ? 8 : 1][4];

  // row-wise 1x128 codes and scales (a tile row lives in one 16-lane DPP row)
  u16* const hb = h_out ? h_out + m0 * cols + (int64_t)kc * kTile : nullptr;
  uint8_t* const qb = q ? q + m0 * cols + (int64_t)kc * kTile : nullptr;
  float* const sb = q ? s + m0 * nt + kc : nullptr;
  const uint32_t ucols = (uint32_t)cols;
  float cm[8];
#pragma unroll
  for (int j = 0; j < 8; j++) cm[j] = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const uint32_t r = (uint32_t)(gr * 8 + i);
    const bool live = FULL || (int)r < mvalid;
    float (&vi)[8] = v[kPacked ? 0 : i];
    // (a row is unpacked where its turn comes: hoisted to the top, the rows of the whole tile would be live unpacked)
    if constexpr (kPacked) {
      raw[i].pin();
      raw[i].get(vi, lut);  // the activation from its table in LDS
      if constexpr (!FULL && std::is_same<IN, GELU>::value) {
#pragma unroll
        for (int j = 0; j < 8; j++) vi[j] = live ? vi[j] : 0.f;
      }
    } else {
      raw[i].get(vi);
      if constexpr (WEIGHTED) {
        const float w = FULL || live ? row_w[r] : 0.f;
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          const uint32_t pk = pack_bf16x2(vi[j] * w, vi[j + 1] * w);
          vi[j] = __uint_as_float(pk << 16);
          vi[j + 1] = __uint_as_float(pk & 0xffff0000u);
        }
      }
    }
    if constexpr (kPacked) {
      const v4i pk = pack8_bf16(vi);
#pragma unroll
      for (int k = 0; k < 4; k++) vp[i][k] = (uint32_t)pk[k];
#pragma unroll
      for (int j = 0; j < 8; j++) cm[j] = fmaxf(cm[j], fabsf(vi[j]));
    }
    if (hb != nullptr && live) st_nt(hb, (r * ucols + (uint32_t)c * 8) * 2, pack8_bf16(vi));
    if (qb != nullptr) {
      // (a row past the group's end has no codes; a maximum of zero would send it through the plain division)
      const float amax = row16_max(amax8(vi));
      const Divider dv = make_scale(live ? amax : 1.f, eps, plain_div);
      const v2i codes = quant8(vi, dv);
      if (live) {
        st_nt(qb, r * ucols + (uint32_t)c * 8, codes);
        if (c == 0) *reinterpret_cast<float*>(reinterpret_cast<char*>(sb) + r * (uint32_t)nt * 4) = dv.s;
      }
    }
    if constexpr (kPacked) {
#pragma unroll
      for (int k = 0; k < 4; k++) asm volatile("" : "+v"(vp[i][k]));  // the row is finished before the next one is unpacked
    }
  }
  // column amax over the 128 tokens of the tile (two rows per three-operand maximum)
#pragma unroll
  for (int j = 0; j < 8; j++) {
    if constexpr (!kPacked) {
#pragma unroll
      for (int i = 0; i < 8; i += 2) cm[j] = fmaxf(fmaxf(cm[j], fabsf(v[i][j])), fabsf(v[i + 1][j]));
    }
    part[gr][c * 8 + j] = cm[j];
  }
  __syncthreads();
  if ((int)threadIdx.x < kTile) {
    float m = part[0][(int)threadIdx.x];
#pragma unroll
    for (int i = 1; i < 16; i++) m = fmaxf(m, part[i][(int)threadIdx.x]);
    const Divider dv = make_scale(m, eps, plain_div);
    cdiv[((int)threadIdx.x & 7) * 16 + ((int)threadIdx.x >> 3)] = dv;  // [column % 8][column / 8]: lanes of a row read 16 neighbours
    if (blocked == AAMD_QT_ROWS_SCALES) s_t[((int64_t)kc * kTile + (int)threadIdx.x) * (int64_t)(ld_t / kTile) + pt] = dv.s;
    else (s_t + (int64_t)pt * cols + (int64_t)kc * kTile)[(int)threadIdx.x] = dv.s;
  }
  __syncthreads();
  if constexpr (SUMS) {  // in the region of the maxima, which have been read
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if constexpr (kPacked) sum += __uint_as_float(j & 1 ? vp[i][j / 2] & 0xffff0000u : vp[i][j / 2] << 16);
        else sum += v[i][j];
      }
      part[gr][c * 8 + j] = sum;
    }
    __syncthreads();
    if ((int)threadIdx.x < kTile) {
      float sum = part[0][(int)threadIdx.x];
#pragma unroll
      for (int i = 1; i < 16; i++) sum += part[i][(int)threadIdx.x];
      tile_sums[(int64_t)pt * cols + (int64_t)kc * kTile + (int)threadIdx.x] = sum;
    }
    __syncthreads();
  }
  // codes of the 8x8 register block, transposed through LDS, written as rows of 128 bytes
#pragma unroll
  for (int j = 0; j < 8; j++) {
    float col[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if constexpr (kPacked) col[i] = __uint_as_float(j & 1 ? vp[i][j / 2] & 0xffff0000u : vp[i][j / 2] << 16);
      else col[i] = v[i][j];
    }
    *reinterpret_cast<v2i*>(tile_t + staged_off(c * 8 + j, gr * 8)) = quant8(col, cdiv[j * 16 + c]);
  }
  uint32_t ld_out;
  uint8_t* const out_t = qt_tile(q_t, blocked, cols, ld_t, pt, kc, &ld_out);
  store_staged_tile(tile_t, out_t, ld_out);
}

template <typename IN, bool SUMS = false>
__global__ __launch_bounds__(256) void quant_dual_grouped_kernel(
    const typename IN::elem* __restrict__ x, int64_t ldx, int nt, const int64_t* __restrict__ goff,
    int E, int64_t M, uint8_t* __restrict__ q, float* __restrict__ s,
    uint8_t* __restrict__ q_t, float* __restrict__ s_t, int64_t ld_t, int blocked, float eps, int64_t gate_off,
    u16* __restrict__ h_out, float* __restrict__ tile_sums = nullptr) {
  // the per-row-group column maxima are dead before the transposed codes are staged: one region
  __shared__ __attribute__((aligned(16))) uint8_t tile_t[kTile * kTLd];
  static_assert(sizeof(float) * 16 * kTile <= sizeof(tile_t), "the column maxima fit in the staging region");
  __shared__ Divider cdiv[kTile];  // scale and divider of every column of the tile
  // the activation's table (GELU forms only), copied from the library's array
  __shared__ __attribute__((aligned(16))) uint8_t lut_s[kLutBytes<IN> ? kLutBytes<IN> : 16];
  if constexpr (kLutBytes<IN> != 0) {
    const v4i* const src = reinterpret_cast<const v4i*>(std::is_same<IN, GELU>::value ? (const void*)g_gelu_lut : (const void*)g_gelub_lut);
    for (uint32_t i = threadIdx.x; i < kLutBytes<IN> / 16; i += 256) reinterpret_cast<v4i*>(lut_s)[i] = src[i];
  }

  // Workgroups go to the eight XCDs in turn, and the row-wise scales of a tile are 128 single floats, one
  // per row: with tile = workgroup index, the eight floats of a 32-byte sector would come from eight
  // different L2 caches and reach memory as eight partial writes.  The index is therefore re-dealt so
  // that eight consecutive workgroups of one XCD take eight consecutive column tiles of one token tile.
  uint32_t bx = blockIdx.x, by = blockIdx.y;
  {
    const uint32_t ntx = gridDim.x, per_row = ntx >> 3;
    const uint32_t lin = by * ntx + bx, chunks = gridDim.y * per_row;
    if ((ntx & 7) == 0 && lin < (chunks & ~7u) * 8) {
      const uint32_t j = lin >> 3, chunk = (j & ~7u) + (lin & 7);
      by = chunk / per_row;
      bx = (chunk - by * per_row) * 8 + (j & 7);
    }
  }
  const int pt = (int)by, kc = (int)bx;
  const GroupOfTile at = find_group<kTile>(goff, E, pt, M);
  if (at.g >= E) return;
  const int64_t m0 = at.r_lo + (int64_t)(pt - at.t_lo) * kTile;
  const int64_t left = at.r_hi - m0;
  const int mvalid = left < kTile ? (int)left : kTile;
  if constexpr (kLutBytes<IN> != 0) __syncthreads();  // the copy of the table
  if (mvalid == kTile)
    dual_tile<IN, true, false, SUMS>(x, (uint32_t)ldx, nt, m0, mvalid, pt, kc, q, s, q_t, s_t, (uint32_t)ld_t, blocked, eps, gate_off, h_out, tile_t, cdiv, nullptr, lut_s, tile_sums);
  else
    dual_tile<IN, false, false, SUMS>(x, (uint32_t)ldx, nt, m0, mvalid, pt, kc, q, s, q_t, s_t, (uint32_t)ld_t, blocked, eps, gate_off, h_out, tile_t, cdiv, nullptr, lut_s, tile_sums);
}

// The dual quantiser with the token permute fused in: x holds the tokens in their original order, and permuted
// row j (the rows of every output) is a copy of token sorted_idx[j] / topk, the stable order of the router
// preprocess.  A workgroup looks up the source rows of its 128 permuted rows once (flat index / topk by a
// multiply and a shift: magic = floor(2^sh / topk) + 1 with 2^(sh - 31) >= topk, exact for indices below 2^31)
// and then runs the tile of the grouped kernel on gathered rows.  Source rows are clamped to the token count,
// so a corrupt index reads a wrong row, never beyond x.
// WEIGHTED: the row is bf16(token * probs[flat index]), the combine's gradient with respect to it.  Written by a kernel of its own and
// read here those rows were a third of the two kernels' traffic (8191 tokens to 4 of 60 experts, 2048 wide, with the gradient of the
// weights 107 us, this and a kernel for the weights' gradient alone 86; gathers_gradient in host.cpp says where it is taken).
template <typename IN, bool WEIGHTED = false, bool SUMS = false>
__global__ __launch_bounds__(256) void quant_dual_gather_kernel(
    const typename IN::elem* __restrict__ x, int64_t ldx, int nt, const int64_t* __restrict__ sorted_idx,
    uint32_t magic, int sh, uint32_t T, const int64_t* __restrict__ goff, int E, int64_t M,
    uint8_t* __restrict__ q, float* __restrict__ s, uint8_t* __restrict__ q_t, float* __restrict__ s_t, int64_t ld_t,
    int blocked, float eps, const void* __restrict__ probs = nullptr, int probs_f32 = 0, uint32_t n_flat = 0,
    float* __restrict__ tile_sums = nullptr) {
  __shared__ __attribute__((aligned(16))) uint8_t tile_t[kTile * kTLd];
  __shared__ Divider cdiv[kTile];
  __shared__ uint32_t src_row[kTile];
  __shared__ float row_w[WEIGHTED ? kTile : 1];
  uint32_t bx = blockIdx.x, by = blockIdx.y;  // eight column tiles of a token tile on one XCD: see quant_dual_grouped_kernel
  {
    const uint32_t ntx = gridDim.x, per_row = ntx >> 3;
    const uint32_t lin = by * ntx + bx, chunks = gridDim.y * per_row;
    if ((ntx & 7) == 0 && lin < (chunks & ~7u) * 8) {
      const uint32_t j = lin >> 3, chunk = (j & ~7u) + (lin & 7);
      by = chunk / per_row;
      bx = (chunk - by * per_row) * 8 + (j & 7);
    }
  }
  const int pt = (int)by, kc = (int)bx;
  const GroupOfTile at = find_group<kTile>(goff, E, pt, M);
  if (at.g >= E) return;
  const int64_t m0 = at.r_lo + (int64_t)(pt - at.t_lo) * kTile;
  const int64_t left = at.r_hi - m0;
  const int mvalid = left < kTile ? (int)left : kTile;
  if ((int)threadIdx.x < mvalid) {
    const uint32_t flat = (uint32_t)sorted_idx[m0 + (int)threadIdx.x];
    const uint32_t tok = (uint32_t)(((uint64_t)flat * magic) >> sh);
    src_row[threadIdx.x] = tok < T ? tok : T - 1;
    if constexpr (WEIGHTED) {
      const uint32_t at = flat < n_flat ? flat : n_flat - 1;
      row_w[threadIdx.x] = probs_f32 ? reinterpret_cast<const float*>(probs)[at] : bf16_bits_to_f32(reinterpret_cast<const u16*>(probs)[at]);
    }
  }
  __syncthreads();
  if (mvalid == kTile)
    dual_tile<IN, true, true, SUMS, WEIGHTED>(x, (uint32_t)ldx, nt, m0, mvalid, pt, kc, q, s, q_t, s_t, (uint32_t)ld_t, blocked, eps, 0, nullptr, tile_t, cdiv, src_row, nullptr, tile_sums, row_w);
  else
    dual_tile<IN, false, true, SUMS, WEIGHTED>(x, (uint32_t)ldx, nt, m0, mvalid, pt, kc, q, s, q_t, s_t, (uint32_t)ld_t, blocked, eps, 0, nullptr, tile_t, cdiv, src_row, nullptr, tile_sums, row_w);
}

// ---------------------------------------------------------------------------------------
// SwiGLU backward with both quantisations: rows [a | b] plus the gradient dh of h give the [da | db] row,
//   da = bf16(bf16(dh*b) * sig(a) * (1 + a*(1 - sig(a)))),  db = bf16(dh * bf16(silu(a))),
// what autograd makes of the two torch ops on bf16 tensors (grouped_gemm_moe.py:331-334).  One workgroup of 512
// threads per 128 tokens x 128 features makes the da tile and the db tile of those features from one read of a, b
// and dh and one sigmoid per position.
// Thread (gr = tid / 16, c = tid % 16) holds rows gr*4 .. gr*4+3, columns c*8 .. c*8+7 of both tiles.
// ---------------------------------------------------------------------------------------
// sigmoid(a) in fp32 per bf16 value a, for |a| in [2^-14, 2^4), read from LDS like the GELU tables (filled
// by the kernel's own sigmoid; inside the table range a sigmoid(a) equals the scaled form's silu bit
// for bit: neither product leaves the normal range there)
constexpr uint32_t kSigLo = (uint32_t)(127 - 14) << 7;
constexpr uint32_t kSigN = (uint32_t)(14 + 4) << 7;
static __device__ __attribute__((aligned(16))) float g_sigmoid_lut[2 * kSigN];
__global__ __launch_bounds__(256) void sigmoid_lut_kernel() {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= 2 * kSigN) return;
  const uint32_t sign = i >= kSigN ? 1u : 0u;
  const float x = __uint_as_float(((sign << 15) | (kSigLo + i - sign * kSigN)) << 16);
  g_sigmoid_lut[i] = sigmoid_scaled(x) * 0x1p-16f;
}

// 4 values / one scale -> 4 codes in one dword
__device__ __forceinline__ int quant4(const float* v, const Divider& d) {
  float t[4];
  if (__builtin_expect(d.plain, 0)) {
#pragma unroll
    for (int i = 0; i < 4; i++) t[i] = v[i] / d.s;
    return pack2_fp8<true>(t[2], t[3], pack2_fp8<false>(t[0], t[1], 0));
  }
#pragma unroll
  for (int i = 0; i < 4; i++) t[i] = __builtin_fmaf(v[i], d.yh, v[i] * d.yl);
  return pack2_fp8<true>(t[2], t[3], pack2_fp8<false>(t[0], t[1], 0));
}

template <bool FULL, bool SUMS>
__device__ __forceinline__ void swiglu_bwd_dual_tile(const u16* __restrict__ xa /* a at the tile's origin */, uint32_t ld,
                                                     int64_t gate_off, const u16* __restrict__ xd, uint32_t ld_dh, int nt,
                                                     int64_t m0, int mvalid, int pt, int f, uint8_t* __restrict__ q,
                                                     float* __restrict__ s, uint8_t* __restrict__ q_t,
                                                     float* __restrict__ s_t, uint32_t ld_t, int blocked,
                                                     u16* __restrict__ g_out, uint8_t (*tile_t)[kTile * kTLd],
                                                     Divider (*cdiv)[kTile], const float* sig_lut, float* __restrict__ tile_sums) {
  const int tid = threadIdx.x, gr = tid >> 4, c = tid & 15;
  const int half = nt / 2;
  const int64_t cols = (int64_t)nt * kTile;
  const uint32_t ucols = (uint32_t)cols;
  // ---- loads, then da and db of the thread's 4 x 8 positions
  v4i ra[4], rb[4], rd[4];
  {
    const uint32_t off0 = ((uint32_t)(gr * 4) * ld + (uint32_t)c * 8) * 2, off0d = ((uint32_t)(gr * 4) * ld_dh + (uint32_t)c * 8) * 2;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (FULL || gr * 4 + i < mvalid) {
        ra[i] = ld16_nt(xa, off0 + (uint32_t)i * ld * 2);
        rb[i] = ld16_nt(xa + gate_off, off0 + (uint32_t)i * ld * 2);
        rd[i] = ld16_nt(xd, off0d + (uint32_t)i * ld_dh * 2);
      } else {
        ra[i] = kOnes;  // (absent: inside the table, and the gradient is zero with rd)
        rb[i] = rd[i] = v4i{0, 0, 0, 0};
      }
    }
  }
  uint32_t vp[2][4][4];  // [da | db][row][column pair]: the results are bf16 numbers and wait for the column pass packed
  float (*part)[32][kTile] = reinterpret_cast<float (*)[32][kTile]>(&tile_t[0][0]);  // [2][32][128] floats: dead before the staging
  static_assert(sizeof(float) * 2 * 32 * kTile <= 2 * sizeof(tile_t[0]), "the column maxima fit in the staging regions");
  float cm[2][8];
#pragma unroll
  for (int w = 0; w < 2; w++)
#pragma unroll
    for (int j = 0; j < 8; j++) cm[w][j] = 0.f;
  // one row at a time, from the packed inputs to the stored codes of both tiles
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t r = (uint32_t)(gr * 4 + i);
    const bool live = FULL || (int)r < mvalid;
    float fa[8], fb[8], fd[8], v[2][8];
    unpack8(ra[i], fa);
    unpack8(rb[i], fb);
    unpack8(rd[i], fd);
    // sigmoid(a) of the row's eight values from the table, all reads issued together; silu = a sigmoid(a)
    float sg[8], sil[8];
    {
      uint32_t t[8];
      bool ok = true;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint32_t w = (uint32_t)ra[i][k];
        const uint32_t m0 = (w & 0x7fffu) - kSigLo, m1 = ((w >> 16) & 0x7fffu) - kSigLo;
        ok = ok && m0 < kSigN && m1 < kSigN;
        t[2 * k] = m0 < kSigN ? m0 + ((w >> 15) & 1u) * kSigN : 0u;
        t[2 * k + 1] = m1 < kSigN ? m1 + (w >> 31) * kSigN : 0u;
      }
#pragma unroll
      for (int k = 0; k < 8; k++) sg[k] = sig_lut[t[k]];
#pragma unroll
      for (int k = 0; k < 8; k++) sil[k] = fa[k] * sg[k];
      if (__builtin_expect(!ok, 0)) {  // values outside the table (zeros, outliers): the arithmetic
#pragma unroll
        for (int k = 0; k < 8; k++) {
          if ((__float_as_uint(fa[k]) >> 16 & 0x7fffu) - kSigLo >= kSigN) {
            const float rs = sigmoid_scaled(fa[k]);
            sg[k] = rs * 0x1p-16f;
            sil[k] = silu_from(fa[k], rs);
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
      // db = bf16(dh * bf16(silu(a)))
      const uint32_t sl = pack_bf16x2(sil[k], sil[k + 1]);
      const uint32_t ob = pack_bf16x2(fd[k] * __uint_as_float(sl << 16), fd[k + 1] * __uint_as_float(sl & 0xffff0000u));
      vp[1][i][k / 2] = ob;
      v[1][k] = __uint_as_float(ob << 16);
      v[1][k + 1] = __uint_as_float(ob & 0xffff0000u);
      // da = bf16(bf16(dh * b) * sig(a) * (1 + a * (1 - sig(a))))
      const float sg0 = sg[k], sg1 = sg[k + 1];
      const uint32_t gb = pack_bf16x2(fd[k] * fb[k], fd[k + 1] * fb[k + 1]);
      const uint32_t oa = pack_bf16x2((__uint_as_float(gb << 16) * sg0) * (1.0f + fa[k] * (1.0f - sg0)),
                                      (__uint_as_float(gb & 0xffff0000u) * sg1) * (1.0f + fa[k + 1] * (1.0f - sg1)));
      vp[0][i][k / 2] = oa;
      v[0][k] = __uint_as_float(oa << 16);
      v[0][k + 1] = __uint_as_float(oa & 0xffff0000u);
    }
#pragma unroll
    for (int w = 0; w < 2; w++) {
      const int kc = w == 0 ? f : half + f;
#pragma unroll
      for (int j = 0; j < 8; j++) cm[w][j] = fmaxf(cm[w][j], fabsf(v[w][j]));
      if (g_out != nullptr && live)
        st_nt(g_out + m0 * cols + (int64_t)kc * kTile, (r * ucols + (uint32_t)c * 8) * 2,
              v4i{(int)vp[w][i][0], (int)vp[w][i][1], (int)vp[w][i][2], (int)vp[w][i][3]});
      if (q != nullptr) {
        const float amax = row16_max(amax8(v[w]));
        const Divider dv = make_scale(live ? amax : 1.f, 0.f, false);
        const v2i codes = quant8<false>(v[w], dv);
        if (live) {
          st_nt(q + m0 * cols + (int64_t)kc * kTile, r * ucols + (uint32_t)c * 8, codes);
          if (c == 0) *reinterpret_cast<float*>(reinterpret_cast<char*>(s + m0 * nt + kc) + r * (uint32_t)nt * 4) = dv.s;
        }
      }
    }
#pragma unroll
    for (int w = 0; w < 2; w++)
#pragma unroll
      for (int j = 0; j < 4; j++) asm volatile("" : "+v"(vp[w][i][j]));  // the row is finished before the next one starts
  }
#pragma unroll
  for (int w = 0; w < 2; w++)
#pragma unroll
    for (int j = 0; j < 8; j++) part[w][gr][c * 8 + j] = cm[w][j];
  __syncthreads();
  if (tid < 2 * kTile) {
    const int w = tid >> 7, col = tid & (kTile - 1);
    float m = part[w][0][col];
#pragma unroll
    for (int i = 1; i < 32; i++) m = fmaxf(m, part[w][i][col]);
    const Divider dv = make_scale(m, 0.f, false);
    cdiv[w][(col & 7) * 16 + (col >> 3)] = dv;  // [column % 8][column / 8]: lanes of a row read 16 neighbours
    (s_t + (int64_t)pt * cols + (int64_t)(w == 0 ? f : half + f) * kTile)[col] = dv.s;
  }
  __syncthreads();
  if constexpr (SUMS) {  // column sums of both tiles, in the region of the maxima, which have been read
#pragma unroll
    for (int w = 0; w < 2; w++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) sum += __uint_as_float(j & 1 ? vp[w][i][j / 2] & 0xffff0000u : vp[w][i][j / 2] << 16);
        part[w][gr][c * 8 + j] = sum;
      }
    __syncthreads();
    if (tid < 2 * kTile) {
      const int w = tid >> 7, col = tid & (kTile - 1);
      float sum = part[w][0][col];
#pragma unroll
      for (int i = 1; i < 32; i++) sum += part[w][i][col];
      tile_sums[(int64_t)pt * cols + (int64_t)(w == 0 ? f : half + f) * kTile + col] = sum;
    }
    __syncthreads();
  }
  // ---- transposed codes through the LDS
#pragma unroll
  for (int w = 0; w < 2; w++)
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float col[4];
#pragma unroll
      for (int i = 0; i < 4; i++) col[i] = __uint_as_float(j & 1 ? vp[w][i][j / 2] & 0xffff0000u : vp[w][i][j / 2] << 16);
      *reinterpret_cast<int*>(&tile_t[w][staged_off(c * 8 + j, gr * 4)]) = quant4(col, cdiv[w][j * 16 + c]);
      if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // a few dividers at a time: sixteen of them are 64 registers
    }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 2; w++) {
    uint32_t ld_out;
    uint8_t* const out = qt_tile(q_t, blocked, cols, ld_t, pt, w == 0 ? f : half + f, &ld_out);
#pragma unroll
    for (int n = 0; n < 2; n++) {
      const int idx = tid + 512 * n;
      const int r = idx >> 3, ch = idx & 7;
      st_nt(out, (uint32_t)r * ld_out + (uint32_t)ch * 16, *reinterpret_cast<const v4i*>(&tile_t[w][staged_off(r, ch * 16)]));
    }
  }
}

template <bool SUMS>
__global__ __launch_bounds__(512, 4) void swiglu_bwd_dual_kernel(const u16* __restrict__ fc1, int64_t ld, int64_t gate_off,
                                                              const u16* __restrict__ dh, int64_t ld_dh, int nt,
                                                              const int64_t* __restrict__ goff,
                                                              int E, int64_t M,
                                                              uint8_t* __restrict__ q, float* __restrict__ s,
                                                              uint8_t* __restrict__ q_t, float* __restrict__ s_t,
                                                              int64_t ld_t, int blocked, u16* __restrict__ g_out,
                                                              float* __restrict__ tile_sums) {
  __shared__ __attribute__((aligned(16))) uint8_t tile_ts[2][kTile * kTLd];
  __shared__ Divider cdivs[2][kTile];
  __shared__ __attribute__((aligned(16))) float sig_s[2 * kSigN];
  for (uint32_t i = threadIdx.x; i < 2 * kSigN / 4; i += 512)
    reinterpret_cast<v4i*>(sig_s)[i] = reinterpret_cast<const v4i*>(g_sigmoid_lut)[i];
  // consecutive workgroups of one XCD take the eight consecutive feature tiles of a scale sector
  // (see quant_dual_grouped_kernel)
  uint32_t bx = blockIdx.x, by = blockIdx.y;
  {
    const uint32_t ntx = gridDim.x, per_row = ntx >> 3;
    const uint32_t lin = by * ntx + bx, chunks = gridDim.y * per_row;
    if ((ntx & 7) == 0 && lin < (chunks & ~7u) * 8) {
      const uint32_t j = lin >> 3, chunk = (j & ~7u) + (lin & 7);
      by = chunk / per_row;
      bx = (chunk - by * per_row) * 8 + (j & 7);
    }
  }
  const int pt = (int)by, f = (int)bx;
  const GroupOfTile at = find_group<kTile>(goff, E, pt, M);
  if (at.g >= E) return;
  const int64_t m0 = at.r_lo + (int64_t)(pt - at.t_lo) * kTile;
  const int64_t left = at.r_hi - m0;
  const int mvalid = left < kTile ? (int)left : kTile;
  const u16* const xa = fc1 + m0 * ld + (int64_t)f * kTile;
  const u16* const xd = dh + m0 * ld_dh + (int64_t)f * kTile;
  __syncthreads();  // the copy of the table
  if (mvalid == kTile)
    swiglu_bwd_dual_tile<true, SUMS>(xa, (uint32_t)ld, gate_off, xd, (uint32_t)ld_dh, nt, m0, mvalid, pt, f, q, s, q_t, s_t,
                               (uint32_t)ld_t, blocked, g_out, tile_ts, cdivs, sig_s, tile_sums);
  else
    swiglu_bwd_dual_tile<false, SUMS>(xa, (uint32_t)ld, gate_off, xd, (uint32_t)ld_dh, nt, m0, mvalid, pt, f, q, s, q_t, s_t,
                                (uint32_t)ld_t, blocked, g_out, tile_ts, cdivs, sig_s, tile_sums);
}

// The 8x8 byte matrix held as eight rows of two dwords, transposed with byte permutes: cols[j]
// holds byte j of rows 0..7.  (v_perm_b32 selects bytes 0-3 from its second source, 4-7 from the first.)
__device__ __forceinline__ void transpose8x8_bytes(const v2i (&rows)[8], v2i (&cols)[8]) {
#pragma unroll
  for (int jb = 0; jb < 2; jb++)
#pragma unroll
    for (int ib = 0; ib < 2; ib++) {
      const uint32_t a = (uint32_t)rows[4 * ib][jb], b = (uint32_t)rows[4 * ib + 1][jb];
      const uint32_t c = (uint32_t)rows[4 * ib + 2][jb], d = (uint32_t)rows[4 * ib + 3][jb];
      const uint32_t x0 = __builtin_amdgcn_perm(b, a, 0x05010400u);  // a0 b0 a1 b1
      const uint32_t x1 = __builtin_amdgcn_perm(b, a, 0x07030602u);  // a2 b2 a3 b3
      const uint32_t y0 = __builtin_amdgcn_perm(d, c, 0x05010400u);
      const uint32_t y1 = __builtin_amdgcn_perm(d, c, 0x07030602u);
      cols[4 * jb + 0][ib] = (int)__builtin_amdgcn_perm(y0, x0, 0x05040100u);  // a0 b0 c0 d0
      cols[4 * jb + 1][ib] = (int)__builtin_amdgcn_perm(y0, x0, 0x07060302u);
      cols[4 * jb + 2][ib] = (int)__builtin_amdgcn_perm(y1, x1, 0x05040100u);
      cols[4 * jb + 3][ib] = (int)__builtin_amdgcn_perm(y1, x1, 0x07060302u);
    }
}

constexpr int64_t kBlockOrderElements = (int64_t)1 << 27;
template <typename IN>
__global__ __launch_bounds__(256) void quant_128x128_kernel(const typename IN::elem* __restrict__ w,
                                                            int64_t expert_stride, int64_t N, int64_t K,
                                                            uint8_t* __restrict__ q, float* __restrict__ s,
                                                            uint8_t* __restrict__ q_t, float* __restrict__ s_t,
                                                            float eps, int rows_per_xcd, const int64_t* __restrict__ goff) {
  const bool plain_div = !kBf16Values<IN> || eps != 0.f;  // see make_scale
  __shared__ float part[16];
  __shared__ __attribute__((aligned(16))) uint8_t tile_t[kTile * kTLd];
  const int nkb = (int)(K / kTile), nnb = (int)(N / kTile), e = blockIdx.z;
  // An expert without rows, whose codes no product of this call reads (64 x 2048 x 7168 with 8192 rows, Zipf-distributed: 5 to 10 of the
  // 64 have rows, 446 -> 64 us).
  if (goff != nullptr && goff[e + 1] <= goff[e]) return;
  // Workgroups go to the eight XCDs in turn.  With rows_per_xcd, of every 64 consecutive ones those of one XCD take eight
  // consecutive blocks of a row of blocks, so that an XCD reads and writes kilobytes of a matrix row, not 128 bytes here
  // and there (us, one block after the other -> this, with the transposed copy and without: 64 x 2048 x 7168 702 -> 642,
  // 489 -> 444; 8 x 28672 x 4096 697 -> 657, 483 -> 434; 60 x 2816 x 2048 247 -> 231, 177 -> 161; 8 x 4096 x 14336 369 ->
  // 356, 238 -> 221; one contiguous eighth per XCD: 665, 659, 230, 339 with the copy, 457, 453, 162, 245 without).
  int kb = blockIdx.x, nb = blockIdx.y;
  if (rows_per_xcd) {
    const uint32_t lin = blockIdx.y * gridDim.x + blockIdx.x;
    if (lin < (((uint32_t)nkb * (uint32_t)nnb) & ~63u)) {
      const uint32_t id = (lin & ~63u) + (lin & 7u) * 8 + ((lin >> 3) & 7u);
      nb = (int)(id / (uint32_t)nkb);
      kb = (int)(id - (uint32_t)nb * (uint32_t)nkb);
    }
  }
  const int gr = threadIdx.x >> 4, c = threadIdx.x & 15;

  float v[8][8];
  load_tile<IN, true>(w + e * expert_stride + (int64_t)nb * kTile * K + (int64_t)kb * kTile, (uint32_t)K, kTile, v);
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) m = fmaxf(m, amax8(v[i]));
  m = row16_max(m);
  if (c == 0) part[gr] = m;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; i++) m = fmaxf(m, part[i]);
  const Divider dv = make_scale(m, eps, plain_div);
  const float sc = dv.s;
  if (threadIdx.x == 0) {
    if (s != nullptr) s[((int64_t)e * nnb + nb) * nkb + kb] = sc;
    if (s_t != nullptr) s_t[((int64_t)e * nkb + kb) * nnb + nb] = sc;
  }
  v2i codes[8];
#pragma unroll
  for (int i = 0; i < 8; i++) codes[i] = quant8(v[i], dv);
  if (q != nullptr) {
    uint8_t* qe = q + (int64_t)e * N * K + (int64_t)nb * kTile * K + (int64_t)kb * kTile;
#pragma unroll
    for (int i = 0; i < 8; i++) st_nt(qe, (uint32_t)(gr * 8 + i) * (uint32_t)K + (uint32_t)c * 8, codes[i]);
  }
  if (q_t != nullptr) {
    // one scale for the whole block: the transposed copy holds the same codes, so the 8x8 block of
    // this thread is transposed bytewise instead of being quantised a second time
    v2i cols[8];
    transpose8x8_bytes(codes, cols);
#pragma unroll
    for (int j = 0; j < 8; j++) *reinterpret_cast<v2i*>(tile_t + staged_off(c * 8 + j, gr * 8)) = cols[j];
    store_staged_tile(tile_t, q_t + (int64_t)e * N * K + (int64_t)kb * kTile * N + (int64_t)nb * kTile, (uint32_t)N);
  }
}

// out[g, c] = the sum of tile_sums[t, c] over the token tiles t of group g: what is left of a bias gradient after the
// quantisers have summed their tiles.  A thread per column, its loads independent of each other.
template <typename OUT>
__global__ __launch_bounds__(256) void group_sums_kernel(const float* __restrict__ tile_sums, int64_t cols,
                                                         const int64_t* __restrict__ goff, int E, OUT* __restrict__ out) {
  const int g = (int)blockIdx.y;
  int t_lo = 0, t_hi = 0, carry = 0;
  for (int base = 0; base <= g; base += 64) {
    const GroupRanges r = group_ranges<kTile>(goff, E, base, carry);
    if (g - base < 64) {
      t_lo = __builtin_amdgcn_readlane(r.t_lo, g - base);
      t_hi = __builtin_amdgcn_readlane(r.t_hi, g - base);
    }
    carry = r.total;
  }
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= cols) return;
  float sum = 0.f;
#pragma unroll 8
  for (int t = t_lo; t < t_hi; t++) sum += tile_sums[(int64_t)t * cols + c];
  if constexpr (sizeof(OUT) == 4) out[(int64_t)g * cols + c] = sum;
  else out[(int64_t)g * cols + c] = (OUT)f32_to_bf16_bits(sum);
}

// [rows, blocks] scales to [blocks, rows], through 32 x 32 tiles in the LDS; two matrices one behind the other (a launch of its own
// for either is 5.5 us of latency)
struct ScaleMatrix {
  const float* s;
  float* s_t;
  int rows;
};
__global__ __launch_bounds__(256) void transpose_scales_kernel(const ScaleMatrix a, const ScaleMatrix b, int blocks) {
  __shared__ float tile[32][33];
  const int c = (int)threadIdx.x & 31, r = (int)threadIdx.x >> 5;
  const int tiles_a = (a.rows + 31) / 32, first = (int)blockIdx.x < tiles_a;
  const float* __restrict__ s = first ? a.s : b.s;
  float* __restrict__ s_t = first ? a.s_t : b.s_t;
  const int rows = first ? a.rows : b.rows;
  const int row0 = ((int)blockIdx.x - (first ? 0 : tiles_a)) * 32, blk0 = (int)blockIdx.y * 32;
#pragma unroll
  for (int i = 0; i < 32; i += 8)
    if (row0 + r + i < rows && blk0 + c < blocks) tile[r + i][c] = s[(int64_t)(row0 + r + i) * blocks + blk0 + c];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 32; i += 8)
    if (row0 + c < rows && blk0 + r + i < blocks) s_t[(int64_t)(blk0 + r + i) * rows + row0 + c] = tile[c][r + i];
}

template <typename OUT>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ q, const float* __restrict__ s,
                                                      int64_t M, int64_t N, int tile_scale,
                                                      OUT* __restrict__ y) {
  // one lane: 16 consecutive codes of one row
  const int64_t chunks_per_row = N / 16;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * chunks_per_row) return;
  const int64_t r = idx / chunks_per_row, ch = idx - r * chunks_per_row;
  const int64_t nt = N / kTile;
  const float sc = tile_scale ? s[r * nt + ch / 8] : s[(r / kTile) * nt + ch / 8];
  const v4i raw = *reinterpret_cast<const v4i*>(q + r * N + ch * 16);
  float o[16];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(raw[i], false);
    auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(raw[i], true);
    o[4 * i] = lo[0] * sc;
    o[4 * i + 1] = lo[1] * sc;
    o[4 * i + 2] = hi[0] * sc;
    o[4 * i + 3] = hi[1] * sc;
  }
  OUT* dst = y + r * N + ch * 16;
  if constexpr (sizeof(OUT) == 4) {
#pragma unroll
    for (int i = 0; i < 4; i++)
      reinterpret_cast<v4f*>(dst)[i] = v4f{o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]};
  } else {
    v4i w0, w1;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      w0[i] = (int)pack_bf16x2(o[2 * i], o[2 * i + 1]);
      w1[i] = (int)pack_bf16x2(o[8 + 2 * i], o[8 + 2 * i + 1]);
    }
    reinterpret_cast<v4i*>(dst)[0] = w0;
    reinterpret_cast<v4i*>(dst)[1] = w1;
  }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Makes sure that a table of constants on the current device is filled before what follows on the stream.  Until the
// host sees the flag that a kernel behind a completed fill has set, every call fills the table again on its own stream,
// so no call waits for another; after that a call launches nothing (a fill took 4.5 us of the stream's time ahead of
// every launch).  A call under graph capture that finds no flag records the fill and leaves the flag alone: what is
// captured has not run.
__global__ void set_flag_kernel(int32_t* flag) { __hip_atomic_store(flag, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM); }
struct TableState {
  std::atomic<int32_t*> flag[64];  // per device, in pinned host memory, kept until the process ends
  std::mutex lock;
};
static int fill_table(TableState& state, void (*kernel)(), unsigned entries, hipStream_t st) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  const bool tracked = dev >= 0 && dev < 64;
  int32_t* flag = tracked ? state.flag[dev].load(std::memory_order_acquire) : nullptr;
  if (flag != nullptr && __atomic_load_n(flag, __ATOMIC_ACQUIRE) != 0) return AAMD_OK;
  kernel<<<dim3((entries + 255) / 256), dim3(256), 0, st>>>();
  AAMD_LAUNCH_CHECK("table of constants");
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (!tracked || hipStreamIsCapturing(st, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) return AAMD_OK;
  if (flag == nullptr) {
    std::lock_guard<std::mutex> guard(state.lock);
    flag = state.flag[dev].load(std::memory_order_acquire);
    if (flag == nullptr) {
      // (an allocation may not break a capture that another thread has under way)
      hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
      const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
      const hipError_t got = hipHostMalloc(reinterpret_cast<void**>(&flag), sizeof(int32_t), hipHostMallocDefault);
      if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
      if (got != hipSuccess) {
        (void)hipGetLastError();  // (no pinned memory: the next call fills again)
        return AAMD_OK;
      }
      *flag = 0;
      state.flag[dev].store(flag, std::memory_order_release);
    }
  }
  set_flag_kernel<<<1, 1, 0, st>>>(flag);
  AAMD_LAUNCH_CHECK("table of constants (flag)");
  return AAMD_OK;
}
static TableState g_gelu_tables, g_sigmoid_table;

}  // namespace aamd

using namespace aamd;

extern "C" int aamd_quant_1x128(const void* x, int x_dtype, int64_t rows, int64_t cols, int64_t ldx, uint8_t* q,
                                float* s, float eps, void* stream) {
  return aamd_permute_quant_1x128(x, x_dtype, rows, cols, ldx, nullptr, 1, rows, q, s, eps, stream);
}

extern "C" int aamd_quant_1x128_with_offsets(const void* x, int x_dtype, int64_t rows, int64_t cols, int64_t ldx, const int64_t* counts,
                                             int E, int64_t* group_offsets, uint8_t* q, float* s, float eps, void* stream) {
  AAMD_REQUIRE(x_dtype == AAMD_BF16 || x_dtype == AAMD_F32 || x_dtype == AAMD_F16, "quant_1x128: unsupported dtype %d", x_dtype);
  AAMD_REQUIRE(rows >= 0 && cols >= 0 && cols % kTile == 0 && ldx >= cols && ldx % 8 == 0 && ldx < kMaxRowLd, "quant_1x128: bad sizes");
  AAMD_REQUIRE(E >= 1 && counts && group_offsets, "quant_1x128_with_offsets: null pointer or no groups");
  OffsetsHere off;
  int64_t run = 0;
  for (int e = 0; e <= E && e <= kOffsetsHere; e++) {
    off.v[e] = (int32_t)run;
    if (e < E) run += counts[e];
    if (run < 0 || run >= 0x7fffffffLL) e = E;  // (left to the general form)
  }
  const int64_t total = rows * (cols / kTile), blocks = (total + 16 * kQuantU - 1) / (16 * kQuantU);
  if (E > kOffsetsHere || total == 0 || total >= ((int64_t)1 << 31) || run < 0 || run >= 0x7fffffffLL) {
    const int rc = aamd_group_offsets(counts, 1, E, group_offsets, stream);
    return rc ? rc : aamd_quant_1x128(x, x_dtype, rows, cols, ldx, q, s, eps, stream);
  }
  AAMD_REQUIRE(x && q && s && aligned16(x) && aligned16(q), "quant_1x128: null or unaligned pointer");
  off.n = E + 1;
  hipStream_t st = (hipStream_t)stream;
  const int nt = (int)(cols / kTile);
  const FastDiv nd = make_fastdiv((uint32_t)nt);
  const unsigned grid = (unsigned)blocks + 1;
  if (x_dtype == AAMD_BF16)
    quant_1x128_offsets_kernel<BF16, kQuantU><<<grid, 256, 0, st>>>((const u16*)x, ldx, nt, nd, total, q, s, eps, rows, off, group_offsets);
  else if (x_dtype == AAMD_F16)
    quant_1x128_offsets_kernel<F16, kQuantU><<<grid, 256, 0, st>>>((const u16*)x, ldx, nt, nd, total, q, s, eps, rows, off, group_offsets);
  else
    quant_1x128_offsets_kernel<F32, kQuantU><<<grid, 256, 0, st>>>((const float*)x, ldx, nt, nd, total, q, s, eps, rows, off, group_offsets);
  AAMD_LAUNCH_CHECK("quant_1x128_with_offsets");
  return AAMD_OK;
}

extern "C" int aamd_permute_quant_1x128(const void* x, int x_dtype, int64_t T, int64_t cols, int64_t ldx,
                                        const int32_t* row_map, int topk, int64_t M_out, uint8_t* q, float* s,
                                        float eps, void* stream) {
  AAMD_REQUIRE(x_dtype == AAMD_BF16 || x_dtype == AAMD_F32 || x_dtype == AAMD_F16, "quant_1x128: unsupported dtype %d", x_dtype);
  AAMD_REQUIRE(T >= 0 && cols >= 0 && cols % kTile == 0, "quant_1x128: cols=%lld must be a multiple of 128",
               (long long)cols);
  AAMD_REQUIRE(ldx >= cols && ldx % 8 == 0 && ldx < kMaxRowLd, "quant_1x128: ldx=%lld must be >= cols, a multiple of 8 and below 2^24",
               (long long)ldx);
  AAMD_REQUIRE(topk >= 1 && M_out >= 0, "quant_1x128: bad topk/M_out");
  if (T == 0 || cols == 0) return AAMD_OK;
  AAMD_REQUIRE(x && q && s, "quant_1x128: null pointer");
  AAMD_REQUIRE(aligned16(x) && aligned16(q), "quant_1x128: x and q must be 16-byte aligned");
  const int nt = (int)(cols / kTile);
  const int64_t total = T * nt;
  AAMD_REQUIRE(total < (int64_t)1 << 40, "quant_1x128: too many tiles");
  hipStream_t st = (hipStream_t)stream;
  constexpr int U = kQuantU;
  const int64_t blocks = (total + 16 * U - 1) / (16 * U);
  AAMD_REQUIRE(blocks < 0x7fffffffLL, "quant_1x128: grid too large");
  dim3 grid((unsigned)blocks), block(256);
  const FastDiv nd = make_fastdiv((uint32_t)nt);
  if (row_map == nullptr) {
    if (x_dtype == AAMD_BF16)
      quant_1x128_kernel<BF16, false, U><<<grid, block, 0, st>>>((const u16*)x, ldx, nt, nd, total, nullptr, 1, M_out, q, s, eps, 0, nullptr);
    else if (x_dtype == AAMD_F16)
      quant_1x128_kernel<F16, false, U><<<grid, block, 0, st>>>((const u16*)x, ldx, nt, nd, total, nullptr, 1, M_out, q, s, eps, 0, nullptr);
    else
      quant_1x128_kernel<F32, false, U><<<grid, block, 0, st>>>((const float*)x, ldx, nt, nd, total, nullptr, 1, M_out, q, s, eps, 0, nullptr);
  } else {
    if (x_dtype == AAMD_BF16)
      quant_1x128_kernel<BF16, true, U><<<grid, block, 0, st>>>((const u16*)x, ldx, nt, nd, total, row_map, topk, M_out, q, s, eps, 0, nullptr);
    else if (x_dtype == AAMD_F16)
      quant_1x128_kernel<F16, true, U><<<grid, block, 0, st>>>((const u16*)x, ldx, nt, nd, total, row_map, topk, M_out, q, s, eps, 0, nullptr);
    else
      quant_1x128_kernel<F32, true, U><<<grid, block, 0, st>>>((const float*)x, ldx, nt, nd, total, row_map, topk, M_out, q, s, eps, 0, nullptr);
  }
  AAMD_LAUNCH_CHECK("quant_1x128");
  return AAMD_OK;
}

static int quant_dual(const void* x, int x_dtype, int64_t M, int64_t cols, int64_t ldx, const int64_t* group_offsets, int E,
                      uint8_t* q, float* s, uint8_t* q_t, float* s_t, int64_t ld_t, int q_t_layout, float eps,
                      float* tile_sums, void* stream) {
  AAMD_REQUIRE(x_dtype == AAMD_BF16 || x_dtype == AAMD_F32 || x_dtype == AAMD_F16, "quant_dual: unsupported dtype %d", x_dtype);
  AAMD_REQUIRE(q_t_layout == AAMD_QT_ROWS || q_t_layout == AAMD_QT_BLOCKED || q_t_layout == AAMD_QT_ROWS_SCALES, "quant_dual: unknown q_t layout %d", q_t_layout);
  AAMD_REQUIRE(M >= 0 && cols >= 0 && cols % kTile == 0, "quant_dual: cols=%lld must be a multiple of 128",
               (long long)cols);
  AAMD_REQUIRE(ldx >= cols && ldx % 8 == 0 && ldx < kMaxTileLd, "quant_dual: bad ldx=%lld", (long long)ldx);
  AAMD_REQUIRE(ld_t < kMaxTileLd, "quant_dual: ld_t=%lld too large", (long long)ld_t);
  AAMD_REQUIRE(E >= 1 && (group_offsets || E == 1), "quant_dual: group_offsets required when E > 1");
  AAMD_REQUIRE(ld_t % kTile == 0 && ld_t >= 0, "quant_dual: ld_t=%lld must be a multiple of 128", (long long)ld_t);
  AAMD_REQUIRE((q == nullptr) == (s == nullptr), "quant_dual: q and s go together");
  AAMD_REQUIRE(q_t && s_t, "quant_dual: q_t / s_t required");
  if (cols == 0) return AAMD_OK;
  // The padded tile count sum_g ceil(M_g/128) is known only on the device; floor(M/128) + E bounds
  // it.  The grid covers min(bound, ld_t/128) tiles, so no tile can land beyond column ld_t of the
  // transposed outputs; tiles past the real total find no group and exit.
  const int64_t max_tiles = M / kTile + E;
  const int64_t grid_tiles = ld_t / kTile < max_tiles ? ld_t / kTile : max_tiles;
  if (grid_tiles == 0) return AAMD_OK;
  AAMD_REQUIRE(aligned16(x) && aligned16(q_t) && (!q || aligned16(q)), "quant_dual: pointers must be 16-byte aligned");
  AAMD_REQUIRE(grid_tiles <= 65535, "quant_dual: more than 65535 token tiles");
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)(cols / kTile), (unsigned)grid_tiles), block(256);
  const int nt = (int)(cols / kTile);
  if (tile_sums)
    quant_dual_grouped_kernel<BF16, true><<<grid, block, 0, st>>>((const u16*)x, ldx, nt, group_offsets, E, M, q, s, q_t, s_t, ld_t, q_t_layout, eps, 0, nullptr, tile_sums);
  else if (x_dtype == AAMD_BF16)
    quant_dual_grouped_kernel<BF16><<<grid, block, 0, st>>>((const u16*)x, ldx, nt, group_offsets, E, M, q, s, q_t, s_t, ld_t, q_t_layout, eps, 0, nullptr);
  else if (x_dtype == AAMD_F16)
    quant_dual_grouped_kernel<F16><<<grid, block, 0, st>>>((const u16*)x, ldx, nt, group_offsets, E, M, q, s, q_t, s_t, ld_t, q_t_layout, eps, 0, nullptr);
  else
    quant_dual_grouped_kernel<F32><<<grid, block, 0, st>>>((const float*)x, ldx, nt, group_offsets, E, M, q, s, q_t, s_t, ld_t, q_t_layout, eps, 0, nullptr);
  AAMD_LAUNCH_CHECK("quant_dual_grouped");
  return AAMD_OK;
}

// probs: the rows are weighted
static int permute_dual(const void* x, int x_dtype, int64_t T, int64_t cols, int64_t ldx, const int64_t* sorted_idx, int topk, int64_t M,
                        const int64_t* group_offsets, int E, const void* probs, int probs_f32, uint8_t* q, float* s, uint8_t* q_t,
                        float* s_t, int64_t ld_t, int q_t_layout, float eps, float* tile_sums, void* stream) {
  AAMD_REQUIRE(x_dtype == AAMD_BF16 || x_dtype == AAMD_F32 || x_dtype == AAMD_F16, "permute_quant_dual: unsupported dtype %d", x_dtype);
  AAMD_REQUIRE(q_t_layout == AAMD_QT_ROWS || q_t_layout == AAMD_QT_BLOCKED, "permute_quant_dual: unknown q_t layout %d", q_t_layout);
  AAMD_REQUIRE(T >= 0 && M >= 0 && cols >= 0 && cols % kTile == 0, "permute_quant_dual: cols=%lld must be a multiple of 128",
               (long long)cols);
  AAMD_REQUIRE(ldx >= cols && ldx % 8 == 0, "permute_quant_dual: bad ldx=%lld", (long long)ldx);
  AAMD_REQUIRE(topk >= 1 && topk <= 32768, "permute_quant_dual: topk=%d out of range", topk);
  AAMD_REQUIRE(T * topk < ((int64_t)1 << 31) && M <= T * topk, "permute_quant_dual: T * topk must stay below 2^31 and M within it");
  AAMD_REQUIRE(ld_t < kMaxTileLd && cols < kMaxTileLd, "permute_quant_dual: ld_t=%lld too large", (long long)ld_t);
  AAMD_REQUIRE(E >= 1 && (group_offsets || E == 1), "permute_quant_dual: group_offsets required when E > 1");
  AAMD_REQUIRE(ld_t % kTile == 0 && ld_t >= 0, "permute_quant_dual: ld_t=%lld must be a multiple of 128", (long long)ld_t);
  AAMD_REQUIRE((q == nullptr) == (s == nullptr), "permute_quant_dual: q and s go together");
  AAMD_REQUIRE(q_t && s_t, "permute_quant_dual: q_t / s_t required");
  if (cols == 0 || M == 0) return AAMD_OK;
  AAMD_REQUIRE(T > 0 && x && sorted_idx, "permute_quant_dual: null input");
  const int64_t max_tiles = M / kTile + E;
  const int64_t grid_tiles = ld_t / kTile < max_tiles ? ld_t / kTile : max_tiles;
  if (grid_tiles == 0) return AAMD_OK;
  AAMD_REQUIRE(aligned16(x) && aligned16(q_t) && (!q || aligned16(q)), "permute_quant_dual: pointers must be 16-byte aligned");
  AAMD_REQUIRE(grid_tiles <= 65535, "permute_quant_dual: more than 65535 token tiles");
  // flat / topk == (flat * magic) >> sh for flat < 2^31: magic = floor(2^sh / topk) + 1, sh = 31 + ceil(log2 topk)
  int l = 0;
  while ((1 << l) < topk) l++;
  const int sh = 31 + l;
  const uint32_t magic = (uint32_t)((((uint64_t)1 << sh) / (uint64_t)topk) + 1);
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)(cols / kTile), (unsigned)grid_tiles), block(256);
  const int nt = (int)(cols / kTile);
  auto launch = [&](auto kernel, auto* in) {
    kernel<<<grid, block, 0, st>>>(in, ldx, nt, sorted_idx, magic, sh, (uint32_t)T, group_offsets, E, M, q, s, q_t, s_t, ld_t, q_t_layout, eps,
                                   probs, probs_f32, (uint32_t)(T * topk), tile_sums);
  };
  if (probs && tile_sums) {
    if (x_dtype == AAMD_BF16) launch(quant_dual_gather_kernel<BF16, true, true>, (const u16*)x);
    else launch(quant_dual_gather_kernel<F32, true, true>, (const float*)x);
  } else if (probs) {
    if (x_dtype == AAMD_BF16) launch(quant_dual_gather_kernel<BF16, true>, (const u16*)x);
    else launch(quant_dual_gather_kernel<F32, true>, (const float*)x);
  } else if (x_dtype == AAMD_BF16) {
    launch(quant_dual_gather_kernel<BF16>, (const u16*)x);
  } else if (x_dtype == AAMD_F16) {
    launch(quant_dual_gather_kernel<F16>, (const u16*)x);
  } else {
    launch(quant_dual_gather_kernel<F32>, (const float*)x);
  }
  AAMD_LAUNCH_CHECK("permute_quant_dual_grouped");
  return AAMD_OK;
}
extern "C" int aamd_permute_quant_1x128_dual_grouped(const void* x, int x_dtype, int64_t T, int64_t cols, int64_t ldx,
                                                     const int64_t* sorted_idx, int topk, int64_t M,
                                                     const int64_t* group_offsets, int E, int32_t* /*tile_ws*/, uint8_t* q,
                                                     float* s, uint8_t* q_t, float* s_t, int64_t ld_t, int q_t_layout,
                                                     float eps, void* stream) {
  return permute_dual(x, x_dtype, T, cols, ldx, sorted_idx, topk, M, group_offsets, E, nullptr, 0, q, s, q_t, s_t, ld_t, q_t_layout, eps,
                      nullptr, stream);
}
extern "C" int aamd_combine_grad_quant_1x128_dual_grouped(const void* dout, int dtype, int64_t T, int64_t cols, const int64_t* sorted_idx,
                                                          int topk, int64_t M, const void* probs, int probs_dtype,
                                                          const int64_t* group_offsets, int E, uint8_t* q, float* s, uint8_t* q_t,
                                                          float* s_t, int64_t ld_t, int q_t_layout, float* tile_sums, void* stream) {
  AAMD_REQUIRE(dtype == AAMD_BF16 || dtype == AAMD_F32, "combine_grad_quant_dual: unsupported dtype %d", dtype);
  AAMD_REQUIRE(probs_dtype == AAMD_BF16 || probs_dtype == AAMD_F32, "combine_grad_quant_dual: unsupported dtype %d of the weights", probs_dtype);
  AAMD_REQUIRE(probs || T <= 0, "combine_grad_quant_dual: null weights");
  return permute_dual(dout, dtype, T, cols, cols, sorted_idx, topk, M, group_offsets, E, probs, probs_dtype == AAMD_F32, q, s, q_t, s_t, ld_t,
                      q_t_layout, 0.f, tile_sums, stream);
}

// ---------------------------------------------------------------------------------------
// SwiGLU fused into the quantisation of the intermediate activations
// ---------------------------------------------------------------------------------------
extern "C" int aamd_swiglu_quant_1x128(const void* fc1, int64_t rows, int64_t F, int64_t ld, void* h_out, uint8_t* q,
                                       float* s, void* stream) {
  AAMD_REQUIRE(rows >= 0 && F >= 0 && F % kTile == 0, "swiglu_quant: F=%lld must be a multiple of 128", (long long)F);
  AAMD_REQUIRE(ld >= 2 * F && ld % 8 == 0 && ld < kMaxRowLd, "swiglu_quant: ld=%lld must be >= 2F, a multiple of 8 and below 2^24", (long long)ld);
  if (rows == 0 || F == 0) return AAMD_OK;
  AAMD_REQUIRE(fc1 && q && s, "swiglu_quant: null pointer");
  AAMD_REQUIRE(aligned16(fc1) && aligned16(q) && aligned16(h_out), "swiglu_quant: pointers must be 16-byte aligned");
  const int nt = (int)(F / kTile);
  const int64_t total = rows * nt;
  AAMD_REQUIRE(total < (int64_t)1 << 40, "swiglu_quant: too many tiles");
  constexpr int U = kQuantU;
  const int64_t blocks = (total + 16 * U - 1) / (16 * U);
  AAMD_REQUIRE(blocks < 0x7fffffffLL, "swiglu_quant: grid too large");
  quant_1x128_kernel<GLU, false, U><<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
      (const u16*)fc1, ld, nt, make_fastdiv((uint32_t)nt), total, nullptr, 1, rows, q, s, 0.f, F, (u16*)h_out);
  AAMD_LAUNCH_CHECK("swiglu_quant_1x128");
  return AAMD_OK;
}

extern "C" int aamd_swiglu_quant_1x128_dual_grouped(const void* fc1, int64_t M, int64_t F, int64_t ld,
                                                    const int64_t* group_offsets, int E, int32_t* /*tile_ws*/,
                                                    void* h_out, uint8_t* q, float* s, uint8_t* q_t, float* s_t,
                                                    int64_t ld_t, int q_t_layout, void* stream) {
  AAMD_REQUIRE(q_t_layout == AAMD_QT_ROWS || q_t_layout == AAMD_QT_BLOCKED, "swiglu_quant_dual: unknown q_t layout %d", q_t_layout);
  AAMD_REQUIRE(M >= 0 && F >= 0 && F % kTile == 0, "swiglu_quant_dual: F=%lld must be a multiple of 128", (long long)F);
  AAMD_REQUIRE(ld >= 2 * F && ld % 8 == 0 && ld < kMaxTileLd && ld_t < kMaxTileLd, "swiglu_quant_dual: bad ld=%lld", (long long)ld);
  AAMD_REQUIRE(E >= 1 && (group_offsets || E == 1), "swiglu_quant_dual: group_offsets required when E > 1");
  AAMD_REQUIRE(ld_t % kTile == 0 && ld_t >= 0, "swiglu_quant_dual: ld_t=%lld must be a multiple of 128", (long long)ld_t);
  AAMD_REQUIRE((q == nullptr) == (s == nullptr), "swiglu_quant_dual: q and s go together");
  AAMD_REQUIRE(q_t && s_t, "swiglu_quant_dual: q_t / s_t required");
  if (F == 0) return AAMD_OK;
  const int64_t max_tiles = M / kTile + E;
  const int64_t grid_tiles = ld_t / kTile < max_tiles ? ld_t / kTile : max_tiles;
  if (grid_tiles == 0) return AAMD_OK;
  AAMD_REQUIRE(aligned16(fc1) && aligned16(q_t) && (!q || aligned16(q)) && aligned16(h_out),
               "swiglu_quant_dual: pointers must be 16-byte aligned");
  AAMD_REQUIRE(grid_tiles <= 65535, "swiglu_quant_dual: more than 65535 token tiles");
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)(F / kTile), (unsigned)grid_tiles), block(256);
  quant_dual_grouped_kernel<GLU><<<grid, block, 0, st>>>((const u16*)fc1, ld, (int)(F / kTile), group_offsets, E, M,
                                                         q, s, q_t, s_t, ld_t, q_t_layout, 0.f, F, (u16*)h_out);
  AAMD_LAUNCH_CHECK("swiglu_quant_dual_grouped");
  return AAMD_OK;
}

// GELU fused into the quantisers: same launches with the GELU / GELU-backward loaders
extern "C" int aamd_gelu_quant_1x128(const void* x, int64_t rows, int64_t F, int64_t ld, void* h_out, uint8_t* q, float* s,
                                     void* stream) {
  AAMD_REQUIRE(rows >= 0 && F >= 0 && F % kTile == 0, "gelu_quant: F=%lld must be a multiple of 128", (long long)F);
  AAMD_REQUIRE(ld >= F && ld % 8 == 0 && ld < kMaxRowLd, "gelu_quant: ld=%lld must be >= F, a multiple of 8 and below 2^24", (long long)ld);
  if (rows == 0 || F == 0) return AAMD_OK;
  AAMD_REQUIRE(x && q && s, "gelu_quant: null pointer");
  AAMD_REQUIRE(aligned16(x) && aligned16(q) && aligned16(h_out), "gelu_quant: pointers must be 16-byte aligned");
  const int nt = (int)(F / kTile);
  const int64_t total = rows * nt;
  AAMD_REQUIRE(total < (int64_t)1 << 40, "gelu_quant: too many tiles");
  constexpr int U = kQuantU;
  const int64_t blocks = (total + 16 * U - 1) / (16 * U);
  AAMD_REQUIRE(blocks < 0x7fffffffLL, "gelu_quant: grid too large");
  quant_1x128_kernel<GELU, false, U><<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
      (const u16*)x, ld, nt, make_fastdiv((uint32_t)nt), total, nullptr, 1, rows, q, s, 0.f, 0, (u16*)h_out);
  AAMD_LAUNCH_CHECK("gelu_quant_1x128");
  return AAMD_OK;
}

// dh == nullptr: forward (h = gelu(x)); else backward (g = dh * gelu'(x)), dh dense with the row stride of x
static int gelu_dual(const void* x, const void* dh, int64_t M, int64_t F, int64_t ld, const int64_t* group_offsets, int E,
                     void* h_out, uint8_t* q, float* s, uint8_t* q_t, float* s_t, int64_t ld_t, int q_t_layout,
                     float* tile_sums, void* stream) {
  AAMD_REQUIRE(q_t_layout == AAMD_QT_ROWS || q_t_layout == AAMD_QT_BLOCKED, "gelu_quant_dual: unknown q_t layout %d", q_t_layout);
  AAMD_REQUIRE(M >= 0 && F >= 0 && F % kTile == 0, "gelu_quant_dual: F=%lld must be a multiple of 128", (long long)F);
  AAMD_REQUIRE(ld >= F && ld % 8 == 0 && ld < kMaxTileLd && ld_t < kMaxTileLd, "gelu_quant_dual: bad ld=%lld", (long long)ld);
  AAMD_REQUIRE(E >= 1 && (group_offsets || E == 1), "gelu_quant_dual: group_offsets required when E > 1");
  AAMD_REQUIRE(ld_t % kTile == 0 && ld_t >= 0, "gelu_quant_dual: ld_t=%lld must be a multiple of 128", (long long)ld_t);
  AAMD_REQUIRE((q == nullptr) == (s == nullptr), "gelu_quant_dual: q and s go together");
  AAMD_REQUIRE(q_t && s_t, "gelu_quant_dual: q_t / s_t required");
  if (F == 0) return AAMD_OK;
  const int64_t max_tiles = M / kTile + E;
  const int64_t grid_tiles = ld_t / kTile < max_tiles ? ld_t / kTile : max_tiles;
  if (grid_tiles == 0) return AAMD_OK;
  AAMD_REQUIRE(x != nullptr, "gelu_quant_dual: null input");
  AAMD_REQUIRE(aligned16(x) && aligned16(dh) && aligned16(q_t) && (!q || aligned16(q)) && aligned16(h_out),
               "gelu_quant_dual: pointers must be 16-byte aligned");
  AAMD_REQUIRE(grid_tiles <= 65535, "gelu_quant_dual: more than 65535 token tiles");
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)(F / kTile), (unsigned)grid_tiles), block(256);
  const int rc = fill_table(g_gelu_tables, gelu_lut_kernel, 2 * kLutN, st);
  if (rc) return rc;
  if (dh == nullptr) {
    quant_dual_grouped_kernel<GELU><<<grid, block, 0, st>>>((const u16*)x, ld, (int)(F / kTile), group_offsets, E, M, q, s,
                                                            q_t, s_t, ld_t, q_t_layout, 0.f, 0, (u16*)h_out);
  } else {
    const int64_t dh_off = (const u16*)dh - (const u16*)x;  // elements; the loader reads dh at x + dh_off
    if (tile_sums)
      quant_dual_grouped_kernel<GELUB, true><<<grid, block, 0, st>>>((const u16*)x, ld, (int)(F / kTile), group_offsets, E, M, q, s,
                                                                     q_t, s_t, ld_t, q_t_layout, 0.f, dh_off, (u16*)h_out, tile_sums);
    else
      quant_dual_grouped_kernel<GELUB><<<grid, block, 0, st>>>((const u16*)x, ld, (int)(F / kTile), group_offsets, E, M, q, s,
                                                               q_t, s_t, ld_t, q_t_layout, 0.f, dh_off, (u16*)h_out);
  }
  AAMD_LAUNCH_CHECK("gelu_quant_dual_grouped");
  return AAMD_OK;
}

static int swiglu_bwd_dual(const void* dh, int64_t ld_dh, const void* fc1, int64_t ld, int64_t M, int64_t F,
                           const int64_t* group_offsets, int E, void* g_out, uint8_t* q, float* s, uint8_t* q_t, float* s_t,
                           int64_t ld_t, int q_t_layout, float* tile_sums, void* stream) {
  AAMD_REQUIRE(q_t_layout == AAMD_QT_ROWS || q_t_layout == AAMD_QT_BLOCKED, "swiglu_bwd_quant_dual: unknown q_t layout %d", q_t_layout);
  AAMD_REQUIRE(M >= 0 && F >= 0 && F % kTile == 0, "swiglu_bwd_quant_dual: F=%lld must be a multiple of 128", (long long)F);
  AAMD_REQUIRE(ld >= 2 * F && ld % 8 == 0 && ld_dh >= F && ld_dh % 8 == 0 && ld < kMaxTileLd && ld_dh < kMaxTileLd && ld_t < kMaxTileLd,
               "swiglu_bwd_quant_dual: bad ld=%lld / ld_dh=%lld",
               (long long)ld, (long long)ld_dh);
  AAMD_REQUIRE(E >= 1 && (group_offsets || E == 1), "swiglu_bwd_quant_dual: group_offsets required when E > 1");
  AAMD_REQUIRE(ld_t % kTile == 0 && ld_t >= 0, "swiglu_bwd_quant_dual: ld_t=%lld must be a multiple of 128", (long long)ld_t);
  AAMD_REQUIRE((q == nullptr) == (s == nullptr), "swiglu_bwd_quant_dual: q and s go together");
  AAMD_REQUIRE(q_t && s_t, "swiglu_bwd_quant_dual: q_t / s_t required");
  if (F == 0) return AAMD_OK;
  const int64_t max_tiles = M / kTile + E;
  const int64_t grid_tiles = ld_t / kTile < max_tiles ? ld_t / kTile : max_tiles;
  if (grid_tiles == 0) return AAMD_OK;
  AAMD_REQUIRE(dh && fc1, "swiglu_bwd_quant_dual: null input");
  AAMD_REQUIRE(aligned16(fc1) && aligned16(dh) && aligned16(q_t) && (!q || aligned16(q)) && aligned16(g_out),
               "swiglu_bwd_quant_dual: pointers must be 16-byte aligned");
  AAMD_REQUIRE(grid_tiles <= 65535, "swiglu_bwd_quant_dual: more than 65535 token tiles");
  hipStream_t st = (hipStream_t)stream;
  const int nt = (int)(2 * F / kTile);
  dim3 grid((unsigned)(nt / 2), (unsigned)grid_tiles), block(512);  // two teams: the da and the db tile of a feature tile
  const int rc = fill_table(g_sigmoid_table, sigmoid_lut_kernel, 2 * kSigN, st);
  if (rc) return rc;
  if (tile_sums)
    swiglu_bwd_dual_kernel<true><<<grid, block, 0, st>>>((const u16*)fc1, ld, F, (const u16*)dh, ld_dh, nt, group_offsets, E, M,
                                                         q, s, q_t, s_t, ld_t, q_t_layout, (u16*)g_out, tile_sums);
  else
    swiglu_bwd_dual_kernel<false><<<grid, block, 0, st>>>((const u16*)fc1, ld, F, (const u16*)dh, ld_dh, nt, group_offsets, E, M,
                                                          q, s, q_t, s_t, ld_t, q_t_layout, (u16*)g_out, nullptr);
  AAMD_LAUNCH_CHECK("swiglu_bwd_quant_dual_grouped");
  return AAMD_OK;
}

// ---- the entry points of the three: without and with the column sums of the tiles
extern "C" int aamd_quant_1x128_dual_grouped(const void* x, int x_dtype, int64_t M, int64_t cols, int64_t ldx,
                                             const int64_t* group_offsets, int E, int32_t* /*tile_ws*/, uint8_t* q,
                                             float* s, uint8_t* q_t, float* s_t, int64_t ld_t, int q_t_layout,
                                             float eps, void* stream) {
  return quant_dual(x, x_dtype, M, cols, ldx, group_offsets, E, q, s, q_t, s_t, ld_t, q_t_layout, eps, nullptr, stream);
}
extern "C" int aamd_gelu_quant_1x128_dual_grouped(const void* x, const void* dh, int64_t M, int64_t F, int64_t ld,
                                                  const int64_t* group_offsets, int E, int32_t* /*tile_ws*/, void* h_out,
                                                  uint8_t* q, float* s, uint8_t* q_t, float* s_t, int64_t ld_t,
                                                  int q_t_layout, void* stream) {
  return gelu_dual(x, dh, M, F, ld, group_offsets, E, h_out, q, s, q_t, s_t, ld_t, q_t_layout, nullptr, stream);
}
extern "C" int aamd_swiglu_bwd_quant_1x128_dual_grouped(const void* dh, int64_t ld_dh, const void* fc1, int64_t ld,
                                                        int64_t M, int64_t F, const int64_t* group_offsets, int E,
                                                        int32_t* /*tile_ws*/, void* g_out, uint8_t* q, float* s,
                                                        uint8_t* q_t, float* s_t, int64_t ld_t, int q_t_layout,
                                                        void* stream) {
  return swiglu_bwd_dual(dh, ld_dh, fc1, ld, M, F, group_offsets, E, g_out, q, s, q_t, s_t, ld_t, q_t_layout, nullptr, stream);
}
extern "C" int aamd_dual_grouped_with_sums(int what, const void* x, const void* dh, int64_t M, int64_t width,
                                           const int64_t* group_offsets, int E, uint8_t* q, float* s, uint8_t* q_t,
                                           float* s_t, int64_t ld_t, int q_t_layout, float eps, float* tile_sums,
                                           void* stream) {
  AAMD_REQUIRE(tile_sums != nullptr, "dual_grouped_with_sums: null sums");
  AAMD_REQUIRE(what == AAMD_SUMS_PLAIN || dh != nullptr, "dual_grouped_with_sums: null gradient");
  if (what == AAMD_SUMS_PLAIN)
    return quant_dual(x, AAMD_BF16, M, width, width, group_offsets, E, q, s, q_t, s_t, ld_t, q_t_layout, eps, tile_sums, stream);
  AAMD_REQUIRE(eps == 0.f, "dual_grouped_with_sums: eps must be 0 here");
  if (what == AAMD_SUMS_GELU_BWD)
    return gelu_dual(x, dh, M, width, width, group_offsets, E, nullptr, q, s, q_t, s_t, ld_t, q_t_layout, tile_sums, stream);
  AAMD_REQUIRE(what == AAMD_SUMS_SWIGLU_BWD && width % 2 == 0, "dual_grouped_with_sums: unknown form %d", what);
  return swiglu_bwd_dual(dh, width / 2, x, width, M, width / 2, group_offsets, E, nullptr, q, s, q_t, s_t, ld_t, q_t_layout,
                         tile_sums, stream);
}
extern "C" int aamd_group_sums(const float* tile_sums, int64_t cols, const int64_t* group_offsets, int E, void* out,
                               int out_dtype, void* stream) {
  AAMD_REQUIRE(out_dtype == AAMD_BF16 || out_dtype == AAMD_F32, "group_sums: unsupported dtype %d", out_dtype);
  AAMD_REQUIRE(cols >= 0 && E >= 1 && E <= 65535 && group_offsets, "group_sums: bad sizes");
  if (cols == 0) return AAMD_OK;
  AAMD_REQUIRE(tile_sums && out, "group_sums: null pointer");
  dim3 grid((unsigned)((cols + 255) / 256), (unsigned)E);
  if (out_dtype == AAMD_F32)
    group_sums_kernel<float><<<grid, 256, 0, (hipStream_t)stream>>>(tile_sums, cols, group_offsets, E, (float*)out);
  else
    group_sums_kernel<u16><<<grid, 256, 0, (hipStream_t)stream>>>(tile_sums, cols, group_offsets, E, (u16*)out);
  AAMD_LAUNCH_CHECK("group_sums");
  return AAMD_OK;
}

// q and s, or q_t and s_t, may be null
static int block_quant_impl(const void* w, int w_dtype, int64_t E, int64_t N, int64_t K, int64_t expert_stride, uint8_t* q,
                            float* s, uint8_t* q_t, float* s_t, float eps, void* stream, const int64_t* goff = nullptr) {
  AAMD_REQUIRE(w_dtype == AAMD_BF16 || w_dtype == AAMD_F32 || w_dtype == AAMD_F16, "quant_128x128: unsupported dtype %d", w_dtype);
  AAMD_REQUIRE(E >= 0 && N >= 0 && K >= 0 && N % kTile == 0 && K % kTile == 0,
               "quant_128x128: N=%lld and K=%lld must be multiples of 128", (long long)N, (long long)K);
  AAMD_REQUIRE(N < kMaxTileLd && K < kMaxTileLd, "quant_128x128: N=%lld or K=%lld too large", (long long)N, (long long)K);
  if (E == 0 || N == 0 || K == 0) return AAMD_OK;
  AAMD_REQUIRE(w && ((q && s) || (q_t && s_t)), "quant_128x128: null pointer");
  AAMD_REQUIRE(expert_stride >= N * K && expert_stride % 8 == 0, "quant_128x128: bad expert stride");
  AAMD_REQUIRE(aligned16(w) && (!q || aligned16(q)) && (!q_t || aligned16(q_t)), "quant_128x128: pointers must be 16-byte aligned");
  AAMD_REQUIRE(N / kTile <= 65535 && E <= 65535, "quant_128x128: grid too large");
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)(K / kTile), (unsigned)(N / kTile), (unsigned)E), block(256);
  // Below 2^27 elements (256 MB of bf16, what the last-level cache holds) plain order is as fast or faster: 1 x 14336 x 4096
  // 42 us, 43 with rows per XCD; 8 x 4096 x 1024 23 both ways.  A little above it the two differ little (60 x 2048 x 1408,
  // 1.3 times the line, 110 both ways; 16 x 3072 x 5120, 1.9 times, 176 and 172), far above it by 4 to 9 % (see the kernel).
  const int rows_per_xcd = E * N * K >= kBlockOrderElements;
  if (w_dtype == AAMD_BF16)
    quant_128x128_kernel<BF16><<<grid, block, 0, st>>>((const u16*)w, expert_stride, N, K, q, s, q_t, s_t, eps, rows_per_xcd, goff);
  else if (w_dtype == AAMD_F16)
    quant_128x128_kernel<F16><<<grid, block, 0, st>>>((const u16*)w, expert_stride, N, K, q, s, q_t, s_t, eps, rows_per_xcd, goff);
  else
    quant_128x128_kernel<F32><<<grid, block, 0, st>>>((const float*)w, expert_stride, N, K, q, s, q_t, s_t, eps, rows_per_xcd, goff);
  AAMD_LAUNCH_CHECK("quant_128x128");
  return AAMD_OK;
}

extern "C" int aamd_quant_128x128(const void* w, int w_dtype, int64_t E, int64_t N, int64_t K,
                                  int64_t expert_stride, uint8_t* q, float* s, uint8_t* q_t, float* s_t, float eps,
                                  void* stream) {
  AAMD_REQUIRE((q_t == nullptr) == (s_t == nullptr), "quant_128x128: q_t and s_t go together");
  AAMD_REQUIRE((q && s) || E <= 0 || N <= 0 || K <= 0, "quant_128x128: null pointer");
  return block_quant_impl(w, w_dtype, E, N, K, expert_stride, q, s, q_t, s_t, eps, stream);
}

extern "C" int aamd_quant_128x128_t(const void* w, int w_dtype, int64_t E, int64_t N, int64_t K, int64_t expert_stride,
                                    uint8_t* q_t, float* s_t, float eps, void* stream) {
  return block_quant_impl(w, w_dtype, E, N, K, expert_stride, nullptr, nullptr, q_t, s_t, eps, stream);
}

extern "C" int aamd_quant_128x128_grouped(const void* w, int w_dtype, int64_t E, int64_t N, int64_t K, int64_t expert_stride,
                                          const int64_t* group_offsets, uint8_t* q, float* s, uint8_t* q_t, float* s_t, float eps,
                                          void* stream) {
  AAMD_REQUIRE(group_offsets || E <= 0, "quant_128x128_grouped: null pointer");
  AAMD_REQUIRE((q == nullptr) == (s == nullptr) && (q_t == nullptr) == (s_t == nullptr), "quant_128x128_grouped: codes and scales go together");
  return block_quant_impl(w, w_dtype, E, N, K, expert_stride, q, s, q_t, s_t, eps, stream, group_offsets);
}

extern "C" int aamd_transpose_scales(const float* s, int64_t rows, int64_t blocks, float* s_t, void* stream) {
  AAMD_REQUIRE(rows >= 0 && blocks >= 0 && rows < 0x7fffffffLL && (blocks + 31) / 32 <= 65535, "transpose_scales: bad sizes");
  if (rows == 0 || blocks == 0) return AAMD_OK;
  AAMD_REQUIRE(s && s_t, "transpose_scales: null pointer");
  transpose_scales_kernel<<<dim3((unsigned)((rows + 31) / 32), (unsigned)((blocks + 31) / 32)), 256, 0, (hipStream_t)stream>>>(
      ScaleMatrix{s, s_t, (int)rows}, ScaleMatrix{}, (int)blocks);
  AAMD_LAUNCH_CHECK("transpose_scales");
  return AAMD_OK;
}
extern "C" int aamd_transpose_scales_pair(const float* a, int64_t rows_a, float* a_t, const float* b, int64_t rows_b, float* b_t,
                                          int64_t blocks, void* stream) {
  AAMD_REQUIRE(rows_a >= 1 && rows_b >= 1 && blocks >= 1 && rows_a < 0x3fffffffLL && rows_b < 0x3fffffffLL && (blocks + 31) / 32 <= 65535,
               "transpose_scales_pair: bad sizes");
  AAMD_REQUIRE(a && a_t && b && b_t, "transpose_scales_pair: null pointer");
  transpose_scales_kernel<<<dim3((unsigned)((rows_a + 31) / 32 + (rows_b + 31) / 32), (unsigned)((blocks + 31) / 32)), 256, 0,
                            (hipStream_t)stream>>>(ScaleMatrix{a, a_t, (int)rows_a}, ScaleMatrix{b, b_t, (int)rows_b}, (int)blocks);
  AAMD_LAUNCH_CHECK("transpose_scales_pair");
  return AAMD_OK;
}

extern "C" int aamd_dequant(const uint8_t* q, const float* s, int64_t M, int64_t N, int tile_scale, void* y,
                            int y_dtype, void* stream) {
  AAMD_REQUIRE(y_dtype == AAMD_BF16 || y_dtype == AAMD_F32, "dequant: unsupported dtype %d", y_dtype);
  AAMD_REQUIRE(M >= 0 && N >= 0 && N % kTile == 0, "dequant: N=%lld must be a multiple of 128", (long long)N);
  AAMD_REQUIRE(tile_scale || M % kTile == 0, "dequant: block scales need M %% 128 == 0");
  if (M == 0 || N == 0) return AAMD_OK;
  AAMD_REQUIRE(q && s && y && aligned16(q) && aligned16(y), "dequant: null or unaligned pointer");
  const int64_t n = M * (N / 16);
  const int64_t blocks = (n + 255) / 256;
  AAMD_REQUIRE(blocks < 0x7fffffffLL, "dequant: grid too large");
  hipStream_t st = (hipStream_t)stream;
  if (y_dtype == AAMD_F32)
    dequant_kernel<float><<<(unsigned)blocks, 256, 0, st>>>(q, s, M, N, tile_scale, (float*)y);
  else
    dequant_kernel<u16><<<(unsigned)blocks, 256, 0, st>>>(q, s, M, N, tile_scale, (u16*)y);
  AAMD_LAUNCH_CHECK("dequant");
  return AAMD_OK;
}
