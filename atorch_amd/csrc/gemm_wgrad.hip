// Weight gradient dW_g[n, k] = sum over the tokens m of group g of dY[m, n] X[m, k] on 256 x 256 tiles, one persistent workgroup
// per CU, for groups of many tokens; both operands transposed, 1x128-scaled along the tokens.
//
// The step is row_tiles_kernel's (gemm_rows.hip: barriers P and Q, eight waves of 128 x 64, blocks requested two steps ahead, the
// steps of a workgroup's tiles one stream, a finished tile from the registers to memory under the next one's loads), with a
// scale per row on both sides: the raw product is folded with acc += product * (l_scale * r_scale), sixteen multiplications more
// per sub-tile, and a step's 2 KB of scales, 256 L rows and 256 R rows of the block, come with its operands into one of four
// slots.  The products and their order are those of the 128 x 128 tiles: the same bits.
//
// What bounds it: 32 vector instructions to fold what two matrix instructions give, and the power both draw (a loop of these
// alone, operands in registers, 2.8 PFLOP/s where the fold of one scale reaches 3.4).  256 tiles of 256 blocks take 2.17 us a
// step, the 128 x 128 tiles 2.20; what is gained lies in half the bytes from the L2 and in the turnover of a tile, 5 us in
// bf16, of which two small ones per CU took more: 32768 rows in 8 groups, 28672 x 4096, 4495 -> 4119 us (1.72 -> 1.88
// PFLOP/s), 8192 rows 1624 -> 1301.  The stores go through the caches (past them 4096 x 4096 of 8 groups 609 us, else 591).
#include <algorithm>

#include "gemm_tiles.hpp"

namespace aamd {

namespace wgrad {
constexpr int BM = 256, BN = 256, NT = 512, WTR = 4, WTL = 2, NTILES = WTR * WTL;
constexpr int kSide = 256 * kBK;      // bytes of an L (R) tile of a step
constexpr int kSlot = (BM + BN) * 4;  // bytes of a step's scales
constexpr int kLds = 4 * kSide + 4 * kSlot + 64 * 16;
constexpr int kWorkgroups = 256;      // one per CU
}  // namespace wgrad

template <typename OUT>
__global__ __launch_bounds__(wgrad::NT, 1) void wgrad_tiles_kernel(const GemmParams p) {
  using namespace wgrad;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds];
  // [L stage 0 | L stage 1 | R stage 0 | R stage 1 | four slots of scales | groups by rank: group, first block, blocks]
  int* const table = reinterpret_cast<int*>(lds + 4 * kSide + 4 * kSlot);
  auto args = [&]() __attribute__((always_inline)) { return (const __attribute__((address_space(4))) GemmParams*)(uintptr_t)args_here(); };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hg = lane >> 5;

  // ---- the tiles of this workgroup: groups longest first, every XCD an eighth of each, its workgroups side by side
  int ranks = 0;
  {
    GroupRanges gr = {};
    int n = 0;
    if (p.goff != nullptr) {
      gr = group_ranges<kBK>(p.goff, p.E, 0, 0);
      n = gr.t_hi - gr.t_lo;
    } else {
      gr.t_hi = n = lane == 0 ? p.max_kb : 0;
    }
    // operand buffers too short: never read past them, and make the failure visible
    const bool nan = lane < p.E && gr.t_hi > p.max_kb;
    const bool live = lane < p.E && !nan && n > 0;
    n = live ? n : 0;
    const unsigned long long nans = __ballot(nan), empty = __ballot(lane < p.E && !live && !nan);
    ranks = __popcll(__ballot(live));
    int rank = 0;
    for (int e = 0; e < p.E; e++) {
      const int m = __builtin_amdgcn_readlane(n, e);
      rank += m > n || (m == n && e < lane) ? 1 : 0;
    }
    if (live) *reinterpret_cast<v4i*>(table + rank * 4) = v4i{lane, gr.t_lo, n, 0};
    // (every wave writes the same values, and reads what it wrote)
    for (unsigned long long left = nans | empty; left != 0; left &= left - 1) {  // groups without a contraction
      const int g = __builtin_ctzll(left);
      const float v = (nans >> g) & 1 ? __builtin_nanf("") : 0.f;
      const int w = sizeof(OUT) == 4 ? __builtin_bit_cast(int, v) : (int)pack_bf16x2(v, v);
      uint8_t* const out = reinterpret_cast<uint8_t*>(reinterpret_cast<OUT*>(p.C) + (int64_t)g * p.c_group_stride);
      const int64_t bytes = p.Lrows * p.ldc * (int64_t)sizeof(OUT);
      for (int64_t at = ((int64_t)blockIdx.x * NT + tid) * 16; at < bytes; at += (int64_t)gridDim.x * NT * 16)
        *reinterpret_cast<v4i*>(out + at) = v4i{w, w, w, w};
    }
  }
  const uint32_t nLt = (uint32_t)p.nLt, nRt = (uint32_t)p.nRt, per_g = nLt * nRt, per_x = (per_g + 7) >> 3;
  const uint32_t xcd = blockIdx.x & 7u, nwg = gridDim.x >> 3, slots = per_x * (uint32_t)ranks;
  uint32_t next_slot = blockIdx.x >> 3;
  int64_t c_at, n_at;  // first output element of the tile
  int c_lvalid, c_rvalid, c_n, n_l0, n_r0, n_lvalid, n_rvalid, n_kb, n_n;
  auto take = [&](auto a) __attribute__((always_inline)) {  // the next tile of this workgroup, false if there is none
    for (; next_slot < slots; next_slot += nwg) {
      const uint32_t turn = next_slot / per_x, pos = next_slot - turn * per_x;
      // this XCD's eighth; which one rotates with the group, so that remainders spread over the XCDs
      const uint32_t part = (xcd + turn) & 7u, size = per_g >> 3, rem = per_g & 7u;
      if (pos >= size + (part < rem ? 1u : 0u)) continue;
      const uint32_t pe = part * size + (part < rem ? part : rem) + pos;
      // groups of gl tiles of the longer side of the gradient, all tiles of the shorter one inside
      const int by_r = opaque(a->group_r);
      const uint32_t along = by_r ? nRt : nLt, across = by_r ? nLt : nRt, gl = (uint32_t)a->gl;
      const uint32_t width = gl * across, batch = pe / width, first = batch * gl, in = pe - batch * width;
      const uint32_t gsz = along - first < gl ? along - first : gl;
      const uint32_t outer = in / gsz, inner = first + (in - outer * gsz);
      n_l0 = __builtin_amdgcn_readfirstlane((int)((by_r ? outer : inner) * BM));
      n_r0 = __builtin_amdgcn_readfirstlane((int)((by_r ? inner : outer) * BN));
      const v4i e = *reinterpret_cast<const v4i*>(table + turn * 4);
      n_kb = __builtin_amdgcn_readfirstlane(e[1]);
      n_n = __builtin_amdgcn_readfirstlane(e[2]);
      n_lvalid = (int)(a->Lrows - n_l0 < BM ? a->Lrows - n_l0 : BM);
      n_rvalid = (int)(a->Rrows - n_r0 < BN ? a->Rrows - n_r0 : BN);
      n_at = (int64_t)__builtin_amdgcn_readfirstlane(e[0]) * a->c_group_stride + n_l0 * a->ldc + n_r0;
      next_slot += nwg;
      return true;
    }
    return false;
  };
  auto next_is_current = [&]() __attribute__((always_inline)) { c_at = n_at, c_lvalid = n_lvalid, c_rvalid = n_rvalid, c_n = n_n; };
  if (!take(&p)) return;
  next_is_current();

  // ---- loads: n-th instruction of wave w for a side: rows 8 w + 64 n .. + 7, the 16-byte chunks of a row XOR-swizzled; waves 0
  // to 3 bring the scales of the L rows, the others those of the R rows.
  const int r8 = lane >> 3;
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ r8 ^ (wave & 1)) << 4);
  // (both sides have one row stride; the offsets of the later instructions are made where they are used, for want of registers)
  const uint32_t voff0 = (uint32_t)(wave * 8 + r8) * (uint32_t)p.ldl + chunk, rows64 = 64u * (uint32_t)p.ldl;
  auto voff = [&](auto N) __attribute__((always_inline)) {
    constexpr uint32_t n = (uint32_t)decltype(N)::value;
    if constexpr (n == 0) return voff0;
    uint32_t v;
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(v) : "s"(n * rows64), "v"(voff0));
    return v;
  };
  const int l_scales = wave < 4;
  // Where the next block to be requested lies: it runs through the blocks of a tile and on into the next tile; behind the last
  // one it stays on the last block, to keep the wait counts uniform.  A tile takes two steps at least, as blocks are requested
  // two steps ahead: that of one block takes it twice, the second time with scales of zero.
  v4i lbuf, rbuf, sbuf;
  int l_step, r_step, s_step;
  int to_load;
  auto enter_next = [&](bool more, auto a) __attribute__((always_inline)) {
    if (more) {
      const int64_t kb = n_kb;
      lbuf = buffer_at(a->L + uniform_i64(n_l0 * a->ldl + kb * a->l_kb_stride), (uint32_t)__builtin_amdgcn_readfirstlane((n_lvalid - 1) * (int)a->ldl + kBK));
      rbuf = buffer_at(a->R + uniform_i64(n_r0 * a->ldr + kb * a->r_kb_stride), (uint32_t)__builtin_amdgcn_readfirstlane((n_rvalid - 1) * (int)a->ldr + kBK));
      const float* const s = l_scales ? a->Ls + (kb * a->ls_blk_stride + n_l0) : a->Rs + (kb * a->rs_blk_stride + n_r0);
      sbuf = buffer_at((const float*)uniform_i64((int64_t)(uintptr_t)s), (uint32_t)__builtin_amdgcn_readfirstlane((l_scales ? n_lvalid : n_rvalid) * 4));
      const int move = n_n > 1;
      l_step = __builtin_amdgcn_readfirstlane(move ? (int)a->l_kb_stride : 0);
      r_step = __builtin_amdgcn_readfirstlane(move ? (int)a->r_kb_stride : 0);
      s_step = __builtin_amdgcn_readfirstlane(move ? (int)(l_scales ? a->ls_blk_stride : a->rs_blk_stride) * 4 : 0);
      to_load = __builtin_amdgcn_readfirstlane(n_n > 1 ? n_n : 2);
    } else {
      // (the buffers have moved on behind the last block)
      advance_buffer(lbuf, -(int64_t)l_step);
      advance_buffer(rbuf, -(int64_t)r_step);
      advance_buffer(sbuf, -(int64_t)s_step);
      l_step = r_step = s_step = 0;
      to_load = 0x7fffffff;
    }
  };
  auto advance = [&]() __attribute__((always_inline)) {
    advance_buffer(lbuf, l_step);
    advance_buffer(rbuf, r_step);
    advance_buffer(sbuf, s_step);
    to_load--;
  };
  uint32_t to_lds = lds_offset(lds) + (uint32_t)(wave * 1024), to_slot = 0;
  auto load_l = [&](auto N) __attribute__((always_inline)) { load_lds_x4<decltype(N)::value * 8192>(voff(N), lbuf, to_lds); };
  auto load_r = [&](auto N) __attribute__((always_inline)) { load_lds_x4<2 * kSide + decltype(N)::value * 8192>(voff(N), rbuf, to_lds); };
  auto load_s = [&]() __attribute__((always_inline)) {
    load_lds_x1((uint32_t)((wave & 3) * 64 + lane_here()) * 4u, sbuf, lds_offset(lds) + 4 * kSide + (uint32_t)(wave * 256) + to_slot);
    to_slot = (to_slot + kSlot) & (4 * kSlot - 1);
  };

  // ---- matrix tiling: as in row_tiles_kernel
  const int wr = wave & 1, wl = ((wave & 3) >> 1) + 2 * (wave >> 2);
  const int wrow0 = wr * WTR * 32, wlrow0 = wl * WTL * 32;
  const int sw = (l32 & 7) ^ ((l32 >> 3) & 1);
  uint32_t la[2][2], ra[2][2];  // LDS addresses of this lane's chunks (`la` names the stage of the next step during a step, and
                                // `ra` too from the middle on)
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const uint32_t chk = (uint32_t)(((4 * h + 2 * hg + c) ^ sw) << 4);
      la[h][c] = lds_offset(lds) + (uint32_t)((wlrow0 + l32) * kBK) + chk;
      ra[h][c] = lds_offset(lds) + 2 * kSide + (uint32_t)((wrow0 + l32) * kBK) + chk;
    }
  auto other = [&](uint32_t (&x)[2][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int c = 0; c < 2; c++) x[h][c] ^= kSide;
  };
  typedef const __attribute__((address_space(3))) v4i* lds_v4i_t;
  typedef const __attribute__((address_space(3))) v4f* lds_v4f_t;
  typedef const __attribute__((address_space(3))) float* lds_float_t;
  auto frag = [&](const uint32_t (&base)[2][2], int sub, int h) __attribute__((always_inline)) {
    const v4i lo = *(lds_v4i_t)(uintptr_t)(base[h][0] + (uint32_t)(sub * 32 * kBK));
    const v4i hi = *(lds_v4i_t)(uintptr_t)(base[h][1] + (uint32_t)(sub * 32 * kBK));
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  v16f acc[WTR][WTL], pr;
  v8i lf[WTL][2], rf[2][2];
  float cs[WTL], csn[WTL], cs_last = 0.f;
  v4f rs[4];
  const uint32_t rs_at = lds_offset(lds) + 4 * kSide + (uint32_t)((BM + wrow0 + 4 * hg) * 4);
  uint32_t slot = 0;  // of the step under way
  auto read_cs = [&](uint32_t s) __attribute__((always_inline)) {
    const uint32_t cs_at = lds_offset(lds) + 4 * kSide + (uint32_t)((wlrow0 + (lane_here() & 31)) * 4);
#pragma unroll
    for (int j = 0; j < WTL; j++) csn[j] = *(lds_float_t)(uintptr_t)(cs_at + s + (uint32_t)(j * 128));
  };
  auto read_rs = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; q++) rs[q] = *(lds_v4f_t)(uintptr_t)(rs_at + slot + (uint32_t)(i * 128 + q * 32));
  };
  auto fold = [&](int i, int j, float sc) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][j][r] = __builtin_fmaf(pr[r], sc * rs[r / 4][r % 4], acc[i][j][r]);
    asm volatile("" : "+v"(acc[i][j]));
  };
  auto barrier_q = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  constexpr int PT = (WTR - 1) * WTL - 1;                     // the sub-tile in front of barrier P
  constexpr int kStores = NTILES * (sizeof(OUT) == 4 ? 4 : 2);  // of a wave and tile
  bool stored = false;
  auto barrier_p = [&](int kb) __attribute__((always_inline)) {
    // all but this step's L tile loads have landed (loads and stores are counted in issue order; the stores of the tile before
    // were issued behind the loads this step waits for)
    if (kb == 0 && stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(4 + kStores) : "memory");
    else asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  bool more = false;
  auto step = [&](int kb) __attribute__((always_inline)) {
    if (to_load == 0) enter_next(more, args());
    const uint32_t next = (slot + kSlot) & (4 * kSlot - 1);
    __builtin_amdgcn_sched_barrier(0);
    barrier_q();
    __builtin_amdgcn_sched_barrier(0);
    fold(WTR - 1, WTL - 1, cs_last);  // owed by the step before (adds zero in the first one)
    other(la);
    static_for<NTILES>([&](auto T) __attribute__((always_inline)) {
      constexpr int t = decltype(T)::value;
      constexpr int i = t / WTL, j = t % WTL;
      __builtin_amdgcn_sched_barrier(0);
      pr = mfma_fp8_32x32x64(rf[i & 1][0], lf[j][0], v16f{});
      pr = mfma_fp8_32x32x64(rf[i & 1][1], lf[j][1], pr);
      asm volatile("" : "+v"(pr));
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (j == 0) read_rs(i);
      if constexpr (t < 4) load_l(T);
      if constexpr (j == 0 && i + 1 < WTR) {
#pragma unroll
        for (int h = 0; h < 2; h++) rf[(i + 1) & 1][h] = frag(ra, i + 1, h);
      }
      if constexpr (t == PT) {
        __builtin_amdgcn_sched_barrier(0);
        barrier_p(kb);
        __builtin_amdgcn_sched_barrier(0);
        other(ra);
#pragma unroll
        for (int h = 0; h < 2; h++) rf[0][h] = frag(ra, 0, h);
        read_cs(next);
      }
      if constexpr (t > PT) {
        constexpr int jn = t - PT - 1;
        load_r(std::integral_constant<int, 2 * jn>{});
        load_r(std::integral_constant<int, 2 * jn + 1>{});
        if constexpr (jn == 1) load_s();
#pragma unroll
        for (int h = 0; h < 2; h++) lf[jn][h] = frag(la, jn, h);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (t + 1 < NTILES) fold(i, j, cs[j]);
    });
    cs_last = cs[WTL - 1];
    const int there = kb + 1 < c_n ? -1 : 0;  // (what is read behind the last step is not used)
#pragma unroll
    for (int j = 0; j < WTL; j++) cs[j] = __builtin_bit_cast(float, __builtin_bit_cast(int, csn[j]) & there);
    slot = next;
    advance();
    to_lds ^= kSide;
  };
  // a wave without valid rows: loads and barriers only, in the order of the working waves
  auto idle_step = [&](int kb) __attribute__((always_inline)) {
    if (to_load == 0) enter_next(more, args());
    barrier_q();
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_l(N); });
    barrier_p(kb);
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_r(N); });
    load_s();
    slot = (slot + kSlot) & (4 * kSlot - 1);
    advance();
    to_lds ^= kSide;
  };

  // ---- a finished tile: registers -> memory
  auto store_tile = [&]() __attribute__((always_inline)) {
    const auto a = args();
    const int left = c_lvalid - wlrow0, rows = left < 64 ? left : 64;
    const v4i out = buffer_at(reinterpret_cast<OUT*>(a->C) + (c_at + wlrow0 * a->ldc + wrow0),
                              ((uint32_t)(rows - 1) * (uint32_t)a->ldc + 128u) * (uint32_t)sizeof(OUT));
    const uint32_t at = store_offset<OUT>(lane_here(), (uint32_t)a->ldc);
    static_for<NTILES / 2>([&](auto T) __attribute__((always_inline)) {
      constexpr int i = 2 * (decltype(T)::value % (WTR / 2)), j = decltype(T)::value / (WTR / 2);
      store_sub_tiles<OUT, i * 32, false>(acc[i][j], acc[i + 1][j], at + (uint32_t)(j * 32) * (uint32_t)a->ldc * (uint32_t)sizeof(OUT),
                                         (uint32_t)a->ldc, out);
    });
  };

  // ---- the first tile's blocks 0 and 1
  enter_next(true, &p);
#pragma unroll
  for (int s = 0; s < 2; s++) {
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_l(N); });
    static_for<4>([&](auto N) __attribute__((always_inline)) { load_r(N); });
    load_s();
    advance();
    to_lds ^= kSide;
  }
  bool first = true;
  for (;;) {
    more = take(args());
    const int steps = c_n > 1 ? c_n : 2;
    if (first) asm volatile("s_waitcnt vmcnt(9) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the first tile's block 0 and scales
    first = false;
    const bool work = wrow0 < c_rvalid && wlrow0 < c_lvalid;
    if (work) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        rf[0][h] = frag(ra, 0, h);
#pragma unroll
        for (int j = 0; j < WTL; j++) lf[j][h] = frag(la, j, h);
      }
      read_cs(slot);
#pragma unroll
      for (int j = 0; j < WTL; j++) cs[j] = csn[j];
#pragma unroll
      for (int i = 0; i < WTR; i++)
#pragma unroll
        for (int j = 0; j < WTL; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        pr[r] = 0.f;
        rs[r / 4][r % 4] = 0.f;
      }
      cs_last = 0.f;
      for (int kb = 0; kb < steps; kb++) step(kb);
      __builtin_amdgcn_sched_barrier(0);
      fold(WTR - 1, WTL - 1, cs_last);
      store_tile();
    } else {
      for (int kb = 0; kb < steps; kb++) idle_step(kb);
      if (steps & 1) {
        other(la);
        other(ra);
      }
    }
    stored = work;
    if (!more) break;
    next_is_current();
  }
  // No load may land in an LDS that is no longer this workgroup's; the stores behind the last loads need nobody to wait.
  if (stored) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kStores) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

int launch_wgrad_tiles(const GemmParams& p, int c_dtype, hipStream_t st) {
  const int64_t per_x = ((int64_t)p.nLt * p.nRt + 7) / 8;
  const unsigned blocks = (unsigned)std::min<int64_t>(per_x * p.E * 8, wgrad::kWorkgroups);
  if (c_dtype == AAMD_BF16) wgrad_tiles_kernel<u16><<<blocks, wgrad::NT, 0, st>>>(p);
  else wgrad_tiles_kernel<float><<<blocks, wgrad::NT, 0, st>>>(p);
  AAMD_LAUNCH_CHECK("grouped_gemm (weight gradient, 256 x 256 tiles)");
  return AAMD_OK;
}

}  // namespace aamd
