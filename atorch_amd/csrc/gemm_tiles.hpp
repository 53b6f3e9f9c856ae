// Buffer instructions past the compiler's bookkeeping, and the way of a finished tile from the registers to memory.
#pragma once
#include "gemm.hpp"

namespace aamd {

__device__ __forceinline__ uint32_t lds_offset(const void* q) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)q; }

// A raw buffer of `bytes` bytes at `base`: reads past it give 0, writes past it are dropped.
__device__ __forceinline__ v4i buffer_at(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  return v4i{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), (int)bytes, 0x00020000};  // (addresses have 47 bits)
}
template <int OFFSET>
__device__ __forceinline__ void load_lds_x4(uint32_t off, const v4i& buf, uint32_t lds) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(buf), "s"(lds), "i"(OFFSET) : "memory", "scc");
}
// The same for all lanes or none (-1 or 0); counted like a load either way.
template <int OFFSET>
__device__ __forceinline__ void load_lds_x4_for(int lanes, uint32_t off, const v4i& buf, uint32_t lds) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_mov_b32 exec_lo, %4\n\ts_mov_b32 exec_hi, %4\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(buf), "s"(lds), "i"(OFFSET), "s"(lanes) : "memory", "scc");
}
__device__ __forceinline__ void advance_buffer(v4i& b, int64_t by) {
  const uint64_t a = (((uint64_t)(uint32_t)b[1] << 32) | (uint32_t)b[0]) + (uint64_t)by;
  b[0] = (int)(uint32_t)a;
  b[1] = (int)(uint32_t)(a >> 32);
}
__device__ __forceinline__ void load_lds_x1(uint32_t off, const v4i& buf, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tbuffer_load_dword %0, %1, 0 offen lds" ::"v"(off), "s"(buf), "s"(lds) : "memory");
}

// A uniform value the compiler knows nothing about: a branch on it inside the tile loop stays there (a loop per case would be a
// copy of the whole kernel each).
__device__ __forceinline__ int opaque(int v) {
  v = __builtin_amdgcn_readfirstlane(v);
  asm volatile("" : "+s"(v));
  return __builtin_amdgcn_readfirstlane(v);
}
// The same of what lies in a scalar register (no copy of it in a vector register, which would be made in front of the loop).
__device__ __forceinline__ int opaque_s(int v) {
  asm volatile("" : "+s"(v));
  return __builtin_amdgcn_readfirstlane(v);
}
// The lane, counted anew: what is computed from it lives where it is used, not in registers across the tile loop.
__device__ __forceinline__ int lane_here() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}
// v + s and v ^ s, made where they are used: what the compiler can move in front of the loop costs a register for the whole of it.
__device__ __forceinline__ uint32_t add_here(uint32_t v, uint32_t s) {
  uint32_t r;
  asm volatile("v_add_u32 %0, %1, %2" : "=v"(r) : "s"(s), "v"(v));
  return r;
}
__device__ __forceinline__ uint32_t xor_here(uint32_t v, uint32_t s) {
  uint32_t r;
  asm volatile("v_xor_b32 %0, %1, %2" : "=v"(r) : "s"(s), "v"(v));
  return r;
}
// A word of the LDS that is the same for every lane, by one vector register and with its wait (five wait states behind it, for memory
// instructions that take it as an operand), and 16 bytes of them.
__device__ __forceinline__ int word_here(uint32_t at) {
  int r, v;
  asm volatile("v_mov_b32 %1, %2\n\tds_read_b32 %1, %1\n\ts_waitcnt lgkmcnt(0)\n\tv_readfirstlane_b32 %0, %1\n\ts_nop 4" : "=s"(r), "=&v"(v) : "s"(at) : "memory");
  return __builtin_amdgcn_readfirstlane(r);
}
__device__ __forceinline__ v4i words_here(uint32_t at) {
  asm volatile("" : "+s"(at));
  const v4i v = *(const __attribute__((address_space(3))) v4i*)(uintptr_t)at;
  return v4i{__builtin_amdgcn_readfirstlane(v[0]), __builtin_amdgcn_readfirstlane(v[1]), __builtin_amdgcn_readfirstlane(v[2]), __builtin_amdgcn_readfirstlane(v[3])};
}
__device__ __forceinline__ void put_words(uint32_t at, const v4i& w) { *(__attribute__((address_space(3))) v4i*)(uintptr_t)at = w; }
__device__ __forceinline__ void copy_words(uint32_t to, uint32_t from) {
  const v4i w = *(const __attribute__((address_space(3))) v4i*)(uintptr_t)from;
  put_words(to, w);
}
// The kernel's arguments, fetched anew where they are used.
__device__ __forceinline__ uint64_t args_here() {
  uint64_t a = (uint64_t)(uintptr_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return (uint64_t)uniform_i64((int64_t)a);
}
// (the compiler does not see what is inside: five wait states in front, for scalar registers that the vector unit has just
// written, and two behind, before the data registers are written again)
template <int OFFSET, bool NT>
__device__ __forceinline__ void store_x4(const v4i& v, uint32_t off, const v4i& buf) {
  if constexpr (NT)
    asm volatile("s_nop 4\n\tbuffer_store_dwordx4 %0, %1, %2, 0 offen offset:%3 nt\n\ts_nop 1" ::"v"(v), "v"(off), "s"(buf), "n"(OFFSET) : "memory");
  else
    asm volatile("s_nop 4\n\tbuffer_store_dwordx4 %0, %1, %2, 0 offen offset:%3\n\ts_nop 1" ::"v"(v), "v"(off), "s"(buf), "n"(OFFSET) : "memory");
}

// a.upper half of the lanes <-> b.lower half; odd rows of 16 lanes of a <-> even rows of b
__device__ __forceinline__ void swap32(int& a, int& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = (int)r[0];
  b = (int)r[1];
}
__device__ __forceinline__ void swap16(int& a, int& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = (int)r[0];
  b = (int)r[1];
}


// lanes 8 .. 15 of every 16 of a <-> lanes 0 .. 7 of b
__device__ __forceinline__ void swap8(int& a, int& b) {
  const int ra = __builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false);  // row_ror:8, upper half written
  b = __builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false);
  a = ra;
}

// A finished 32 x 32 sub-tile: lane l holds, for output row l % 32, columns 8 q + 4 (l / 32) .. + 3 (q = 0 .. 3, four registers
// each).  Lanes exchange what they hold until each has 16 bytes and eight of them the 128 bytes of a whole cache line of one
// row, eight rows to an instruction: two sub-tiles side by side in bf16, one in fp32.  (With 64 bytes of a row, one exchange
// less, 4096 x 4096 outputs of a contraction of 1024 take 24.2 us, with it 23.4; x 32768 outputs 163 and 160.)  store_offset: bytes from the tile's first row to what this lane stores first.
template <typename OUT>
__device__ __forceinline__ uint32_t store_offset(int lane, uint32_t ldc) {
  const uint32_t b3 = (uint32_t)(lane >> 3) & 1u, b4 = (uint32_t)(lane >> 4) & 1u, h5 = (uint32_t)lane >> 5;
  return ((uint32_t)(lane & 7) * ldc + (sizeof(OUT) == 4 ? 16 * b3 + 8 * b4 + 4 * h5 : 32 * b3 + 8 * (2 * b4 + h5))) * (uint32_t)sizeof(OUT);
}
// rows 0 .. 7 of x, then 8 .. 15 of y
template <int COL, bool NT>
__device__ __forceinline__ void store_lines(v4i x, v4i y, uint32_t row, uint32_t rows8, const v4i& out) {
#pragma unroll
  for (int r = 0; r < 4; r++) {
    int u = x[r], v = y[r];
    swap8(u, v);
    x[r] = u;
    y[r] = v;
  }
  store_x4<COL, NT>(x, row, out);
  store_x4<COL, NT>(y, row + rows8, out);
}
// the 16 bytes of bf16 columns 8 q .. + 7 a lane then holds: x of row l % 16, y of row 16 + l % 16, q = 2 (l / 16 % 2) + l / 32
__device__ __forceinline__ void gather_bf16(const v16f& o, v4i& x, v4i& y) {
  int w[2][4];  // [pair of q][the 16 bytes of q = 2 pair + lane / 32]
#pragma unroll
  for (int qp = 0; qp < 2; qp++)
#pragma unroll
    for (int r = 0; r < 2; r++) {
      int u = (int)pack_bf16x2(o[8 * qp + 2 * r], o[8 * qp + 2 * r + 1]), v = (int)pack_bf16x2(o[8 * qp + 4 + 2 * r], o[8 * qp + 5 + 2 * r]);
      swap32(u, v);
      w[qp][r] = u;
      w[qp][2 + r] = v;
    }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    swap16(w[0][r], w[1][r]);
    x[r] = w[0][r];
    y[r] = w[1][r];
  }
}
// Two sub-tiles side by side, the first at column COL (elements) of `row` (bytes).
template <typename OUT, int COL, bool NT>
__device__ __forceinline__ void store_sub_tiles(const v16f& a, const v16f& b, uint32_t row, uint32_t ldc, const v4i& out) {
  const uint32_t rows8 = 8u * ldc * (uint32_t)sizeof(OUT);
  if constexpr (sizeof(OUT) == 4) {
    static_for<2>([&](auto T) __attribute__((always_inline)) {
      const v16f& o = decltype(T)::value ? b : a;
      v4i x[2], y[2];  // [pair of q]: four columns of rows l % 16 and 16 + l % 16
#pragma unroll
      for (int qp = 0; qp < 2; qp++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float f = o[8 * qp + r], h = o[8 * qp + 4 + r];  // (a bit cast of a vector's element takes element 0)
          int u = __builtin_bit_cast(int, f), v = __builtin_bit_cast(int, h);
          swap16(u, v);
          x[qp][r] = u;
          y[qp][r] = v;
        }
      store_lines<(COL + decltype(T)::value * 32) * 4, NT>(x[0], x[1], row, rows8, out);
      store_lines<(COL + decltype(T)::value * 32) * 4, NT>(y[0], y[1], row + 2 * rows8, rows8, out);
    });
  } else {
    v4i xa, ya, xb, yb;
    gather_bf16(a, xa, ya);
    gather_bf16(b, xb, yb);
    store_lines<COL * 2, NT>(xa, xb, row, rows8, out);
    store_lines<COL * 2, NT>(ya, yb, row + 2 * rows8, rows8, out);
  }
}

// One sub-tile alone, from the first byte of `out` on: 64 (bf16) or 128 bytes of a row.
template <typename OUT>
__device__ __forceinline__ void store_sub_tile(const v16f& o, int lane, uint32_t ldc, const v4i& out) {
  if constexpr (sizeof(OUT) == 4) {
    const uint32_t row = store_offset<float>(lane, ldc), rows8 = 8u * ldc * 4u;
    v4i x[2], y[2];
#pragma unroll
    for (int qp = 0; qp < 2; qp++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float f = o[8 * qp + r], h = o[8 * qp + 4 + r];
        int u = __builtin_bit_cast(int, f), v = __builtin_bit_cast(int, h);
        swap16(u, v);
        x[qp][r] = u;
        y[qp][r] = v;
      }
    store_lines<0, false>(x[0], x[1], row, rows8, out);
    store_lines<0, false>(y[0], y[1], row + 2 * rows8, rows8, out);
  } else {
    v4i x, y;
    gather_bf16(o, x, y);
    const uint32_t at = ((uint32_t)(lane & 15) * ldc + 8u * (2u * ((uint32_t)(lane >> 4) & 1u) + ((uint32_t)lane >> 5))) * 2u;
    store_x4<0, false>(x, at, out);
    store_x4<0, false>(y, at + 16u * ldc * 2u, out);
  }
}

}  // namespace aamd
