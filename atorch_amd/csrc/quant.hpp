// What the quantising kernels share: loaders of eight elements with the activations that are applied on the way, the scale of a tile
// and its codes.
#pragma once
#include "common.hpp"

namespace aamd {

// ---------------------------------------------------------------------------------------
// tile loaders: 8 consecutive elements per lane
// ---------------------------------------------------------------------------------------
// 16 bytes at a byte offset from a base pointer.  With a base that is the same in every lane the
// address is a scalar register pair plus a 32-bit lane offset: no 64-bit arithmetic per access.
template <typename T>
__device__ __forceinline__ v4i ld16(const T* base, uint32_t boff) {
  return *reinterpret_cast<const v4i*>(reinterpret_cast<const char*>(base) + boff);
}
template <typename T>
__device__ __forceinline__ v4i ld16_nt(const T* base, uint32_t boff) {
  return __builtin_nontemporal_load(reinterpret_cast<const v4i*>(reinterpret_cast<const char*>(base) + boff));
}
template <typename V, typename T>
__device__ __forceinline__ void st_nt(T* base, uint32_t boff, V val) {
  __builtin_nontemporal_store(val, reinterpret_cast<V*>(reinterpret_cast<char*>(base) + boff));
}

template <typename IN>
struct Raw8;
template <>
struct Raw8<BF16> {
  v4i a;
  __device__ __forceinline__ void load(const u16* p, uint32_t boff, int64_t) { a = ld16_nt(p, boff); }
  __device__ __forceinline__ void zero() { a = v4i{0, 0, 0, 0}; }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a)); }
  __device__ __forceinline__ void get(float* v) const { unpack8(a, v); }
};
template <>
struct Raw8<F32> {
  v4i a, b;
  __device__ __forceinline__ void load(const float* p, uint32_t boff, int64_t) {
    a = ld16_nt(p, boff);
    b = ld16_nt(p + 4, boff);
  }
  __device__ __forceinline__ void zero() { a = b = v4i{0, 0, 0, 0}; }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a), "+v"(b)); }
  __device__ __forceinline__ void get(float* v) const {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      v[i] = __int_as_float(a[i]);
      v[4 + i] = __int_as_float(b[i]);
    }
  }
};

template <>
struct Raw8<F16> {
  v4i a;
  __device__ __forceinline__ void load(const u16* p, uint32_t boff, int64_t) { a = ld16_nt(p, boff); }
  __device__ __forceinline__ void zero() { a = v4i{0, 0, 0, 0}; }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a)); }
  __device__ __forceinline__ void get(float* v) const {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t w = (uint32_t)a[i];
      v[2 * i] = (float)__builtin_bit_cast(_Float16, (unsigned short)(w & 0xffffu));
      v[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (unsigned short)(w >> 16));
    }
  }
};

// sigmoid on the hardware transcendental units, one v_exp_f32 and one v_rcp_f32 per value.  Both
// flush results below the normal range, and 1 / (1 + e^-x) gets there for x below about -87 while
// x times it is still a normal number, so the reciprocal is taken of the sum scaled by 2^-16
// (x r' stays finite for |x| < 2^112):
//   e = e^-x (inf where it overflows, 0 where it leaves the normal range), r' = 1 / (2^-16 + 2^-16 e)
//   = 2^16 sigmoid(x).
// silu(x) = (x r') 2^-16, sigmoid(x) = r' 2^-16.  A few fp32 ulps of error (more for |x| in the tens,
// where x log2(e) itself is rounded), far below the bf16 rounding that follows; e^-x = inf gives
// r' = 0 and silu = -0 as in fp32 arithmetic.
__device__ __forceinline__ float sigmoid_scaled(float x) {
  const float e = __builtin_amdgcn_exp2f(x * -1.4426950408889634f);
  return __builtin_amdgcn_rcpf(__builtin_fmaf(e, 0x1p-16f, 0x1p-16f));
}
__device__ __forceinline__ float silu_from(float x, float r_scaled) { return (x * r_scaled) * 0x1p-16f; }

// SwiGLU on load: a and b halves of a row, h = silu(a) * b with both roundings to bf16 that the
// reference's two torch ops make (F.silu on a bf16 tensor, then the product; fp32 inside).
template <>
struct Raw8<GLU> {
  v4i a, b;
  __device__ __forceinline__ void load(const u16* p, uint32_t boff, int64_t gate_off) {
    a = ld16_nt(p, boff);
    b = ld16_nt(p + gate_off, boff);
  }
  __device__ __forceinline__ void zero() { a = b = v4i{0, 0, 0, 0}; }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a), "+v"(b)); }
  __device__ __forceinline__ void get(float* v) const {
    float fa[8], fb[8];
    unpack8(a, fa);
    unpack8(b, fb);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const float s0 = silu_from(fa[i], sigmoid_scaled(fa[i]));
      const float s1 = silu_from(fa[i + 1], sigmoid_scaled(fa[i + 1]));
      const uint32_t sl = pack_bf16x2(s0, s1);
      const uint32_t h = pack_bf16x2(__uint_as_float(sl << 16) * fb[i], __uint_as_float(sl & 0xffff0000u) * fb[i + 1]);
      v[i] = __uint_as_float(h << 16);
      v[i + 1] = __uint_as_float(h & 0xffff0000u);
    }
  }
};

// GELU on load, h = bf16(x Phi(x)), and its backward dh (Phi(x) + x pdf(x)), pdf = exp(-x^2 / 2) / sqrt(2 pi).
// The reference evaluates Phi as (1 + erf(x / sqrt 2)) / 2 in fp32 (torch.nn.functional.gelu on a bf16 tensor).
// Here Phi comes from the complementary function, without branches and without the cancellation of 1 + erf
// for negative x:
//   erfc(t) / 2 = exp(-t^2) q(u),  u = 1 / (1 + t / 2),  t = |x| / sqrt 2,
// q a polynomial of degree 7 (a least-squares fit of erfcx(t) / 2 at Chebyshev nodes of u over 0 <= t <= 4.3,
// relative error 6e-8; beyond 4.3, where erfc / 2 is below 1e-9, q stays at its value there), Phi(x) = erfc(t) / 2
// for x < 0 and 1 - erfc(t) / 2 otherwise.  With s = |x| sqrt(log2(e) / 2) the exponential is exp2(-s^2) and
// t / 2 = 0.41628 s: one v_rcp_f32, one v_exp_f32 and a dozen multiply-adds against the three divergent ranges of
// the library's erff.  In fp32 arithmetic x Phi(x) comes out within 2.3e-6 of its value for |x| <= 6: rounded to
// bf16 it equals the correctly rounded product for every normal bf16 x >= -4, and below that it keeps digits
// where 1 + erf(x / sqrt 2) has lost them.  Infinities and NaNs give what the reference's formula gives.
__device__ __forceinline__ float gelu_phi(float x, float* exp_neg_half_sq = nullptr) {
  const float s = fabsf(x) * 0.8493217825889587f;  // sqrt(log2(e) / 2) |x|
  const float u = __builtin_amdgcn_rcpf(__builtin_fmaf(fminf(s, 5.164826393127441f), 0.41627731919288635f, 1.0f));
  float q = 0.042140234261751175f;
  q = __builtin_fmaf(q, u, -0.16624070703983307f);
  q = __builtin_fmaf(q, u, 0.1660318523645401f);
  q = __builtin_fmaf(q, u, 0.05331931263208389f);
  q = __builtin_fmaf(q, u, 0.11762023717164993f);
  q = __builtin_fmaf(q, u, 0.14757198095321655f);
  q = __builtin_fmaf(q, u, 0.13941511511802673f);
  q = __builtin_fmaf(q, u, 0.00014206925698090345f);
  const float e = __builtin_amdgcn_exp2f(-(s * s));  // exp(-x^2 / 2) = exp(-t^2)
  if (exp_neg_half_sq) *exp_neg_half_sq = e;
  const float h = q * e;  // erfc(t) / 2
  return x < 0.f ? h : 1.0f - h;
}
// Both GELU forms are functions of one bf16 value, x Phi(x) rounded to bf16 and Phi(x) + x pdf(x) in fp32, and cost
// two dozen vector instructions per value, which is what bounds the fused kernels.  The dual kernels therefore read
// them from tables in LDS indexed by the bits of x, for |x| in [2^-14, 2^3) (17 binades x 128 x 2 signs); values
// outside (exact zeros, outliers) take the arithmetic.  The tables are filled by the same functions, by a small
// kernel ahead of the launch, into arrays of the library on the device, until the host has seen that a fill has
// completed (fill_table): every call writes the same values, so calls that overlap do not disturb each other.
constexpr uint32_t kLutLo = (uint32_t)(127 - 14) << 7;        // first magnitude (bits without the sign) of the tables
constexpr uint32_t kLutN = (uint32_t)(14 + 3) << 7;           // magnitudes per sign
__device__ __forceinline__ float gelu_grad_factor(float x) {
  float e;  // exp(-x^2 / 2)
  const float cdf = gelu_phi(x, &e);
  const float pdf = 0.39894228040143267794f * e;
  return cdf + x * pdf;
}
// a pair of values outside the tables: out of line, these are rare
static __device__ __attribute__((noinline)) uint32_t gelu_pair_plain(uint32_t w) {
  const float x0 = __uint_as_float(w << 16), x1 = __uint_as_float(w & 0xffff0000u);
  return pack_bf16x2(x0 * gelu_phi(x0), x1 * gelu_phi(x1));
}
static __device__ __attribute__((noinline)) uint32_t gelu_grad_pair_plain(uint32_t w, uint32_t gw) {
  const float x0 = __uint_as_float(w << 16), x1 = __uint_as_float(w & 0xffff0000u);
  const float g0 = __uint_as_float(gw << 16), g1 = __uint_as_float(gw & 0xffff0000u);
  return pack_bf16x2(g0 * gelu_grad_factor(x0), g1 * gelu_grad_factor(x1));
}
// Table position of the bf16 value whose magnitude bits are `mag` and whose sign is `sign` (0 / 1); `ok` is cleared
// when the value lies outside the tables (position 0 is returned then, so the read that follows stays inside).
__device__ __forceinline__ uint32_t lut_index(uint32_t mag, uint32_t sign, bool& ok) {
  const uint32_t m = mag - kLutLo;
  const bool in = m < kLutN;
  ok = ok && in;
  return in ? m + sign * kLutN : 0u;
}
template <typename IN>
inline constexpr uint32_t kLutBytes = 0;
template <>
inline constexpr uint32_t kLutBytes<GELU> = 2 * kLutN * sizeof(u16);
template <>
inline constexpr uint32_t kLutBytes<GELUB> = 2 * kLutN * sizeof(float);

template <>
struct Raw8<GELU> {
  v4i a;
  __device__ __forceinline__ void load(const u16* p, uint32_t boff, int64_t) { a = ld16_nt(p, boff); }
  __device__ __forceinline__ void zero() { a = v4i{0, 0, 0, 0}; }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a)); }
  __device__ __forceinline__ void get(float* v) const {
    float x[8];
    unpack8(a, x);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const float g0 = x[i] * gelu_phi(x[i]);
      const float g1 = x[i + 1] * gelu_phi(x[i + 1]);
      const uint32_t h = pack_bf16x2(g0, g1);
      v[i] = __uint_as_float(h << 16);
      v[i + 1] = __uint_as_float(h & 0xffff0000u);
    }
  }
  // the same values from the table (a copy of g_gelu_lut in LDS): all eight reads are issued together, and a
  // value outside the table, which is rare, sends its pair through the arithmetic afterwards
  __device__ __forceinline__ void get(float* v, const void* lut) const {
    const u16* const T = static_cast<const u16*>(lut);
    uint32_t t[8], h[4];
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t w = (uint32_t)a[i];
      t[2 * i] = lut_index(w & 0x7fffu, (w >> 15) & 1u, ok);
      t[2 * i + 1] = lut_index((w >> 16) & 0x7fffu, w >> 31, ok);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) h[i] = (uint32_t)T[t[2 * i]] | ((uint32_t)T[t[2 * i + 1]] << 16);
    if (__builtin_expect(!ok, 0)) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t w = (uint32_t)a[i];
        if ((w & 0x7fffu) - kLutLo >= kLutN || ((w >> 16) & 0x7fffu) - kLutLo >= kLutN) h[i] = gelu_pair_plain(w);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      v[2 * i] = __uint_as_float(h[i] << 16);
      v[2 * i + 1] = __uint_as_float(h[i] & 0xffff0000u);
    }
  }
};
template <>
struct Raw8<GELUB> {
  v4i a, d;
  __device__ __forceinline__ void load(const u16* p, uint32_t boff, int64_t dh_off) {
    a = ld16_nt(p, boff);
    d = ld16_nt(p + dh_off, boff);
  }
  __device__ __forceinline__ void zero() { a = d = v4i{0, 0, 0, 0}; }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a), "+v"(d)); }
  __device__ __forceinline__ void get(float* v) const {
    float x[8], g[8];
    unpack8(a, x);
    unpack8(d, g);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const uint32_t h = pack_bf16x2(g[i] * gelu_grad_factor(x[i]), g[i + 1] * gelu_grad_factor(x[i + 1]));
      v[i] = __uint_as_float(h << 16);
      v[i + 1] = __uint_as_float(h & 0xffff0000u);
    }
  }
  // the same values with the factor from the table (a copy of g_gelub_lut in LDS), read like the forward's
  __device__ __forceinline__ void get(float* v, const void* lut) const {
    const float* const T = static_cast<const float*>(lut);
    uint32_t t[8], h[4];
    float f[8];
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t w = (uint32_t)a[i];
      t[2 * i] = lut_index(w & 0x7fffu, (w >> 15) & 1u, ok);
      t[2 * i + 1] = lut_index((w >> 16) & 0x7fffu, w >> 31, ok);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) f[i] = T[t[i]];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t gw = (uint32_t)d[i];
      h[i] = pack_bf16x2(__uint_as_float(gw << 16) * f[2 * i], __uint_as_float(gw & 0xffff0000u) * f[2 * i + 1]);
    }
    if (__builtin_expect(!ok, 0)) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t w = (uint32_t)a[i];
        if ((w & 0x7fffu) - kLutLo >= kLutN || ((w >> 16) & 0x7fffu) - kLutLo >= kLutN)
          h[i] = gelu_grad_pair_plain(w, (uint32_t)d[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      v[2 * i] = __uint_as_float(h[i] << 16);
      v[2 * i + 1] = __uint_as_float(h[i] & 0xffff0000u);
    }
  }
};

// 8 values that are bf16-representable -> 16 bytes
__device__ __forceinline__ v4i pack8_bf16(const float* v) {
  v4i w;
#pragma unroll
  for (int i = 0; i < 4; i++) w[i] = (int)pack_bf16x2(v[2 * i], v[2 * i + 1]);
  return w;
}

}  // namespace aamd
