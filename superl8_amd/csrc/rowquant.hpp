// Device code of the per-row int8 quantisers: storage types, lane-group reductions, the code
// forms and the Hadamard rotation of a row held in registers.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace sl8 {
namespace {

// Reduction over aligned groups of LPR lanes (a power of two <= 64) with no
// LDS round trip: DPP inside a 16-lane row (quad_perm [1,0,3,2], quad_perm
// [2,3,0,1], row_half_mirror, row_mirror: after each step a lane holds the
// reduction over 2, 4, 8, 16 lanes), then v_permlane16_swap across the row
// pair and v_permlane32_swap across the wave halves. Every lane of the group
// ends with the result; op must be associative and commutative (max, integer
// add: exact in any order).
template <int LPR, typename F>
__device__ __forceinline__ uint32_t lane_group_reduce(uint32_t v, F op) {
  static_assert(LPR >= 1 && LPR <= 64 && (LPR & (LPR - 1)) == 0, "LPR: a power of two <= 64");
  auto dpp = [](uint32_t x, auto ctrl) __attribute__((always_inline)) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xF, 0xF, false);
  };
  if constexpr (LPR >= 2) v = op(v, dpp(v, std::integral_constant<int, 0xB1>{}));
  if constexpr (LPR >= 4) v = op(v, dpp(v, std::integral_constant<int, 0x4E>{}));
  if constexpr (LPR >= 8) v = op(v, dpp(v, std::integral_constant<int, 0x141>{}));
  if constexpr (LPR >= 16) v = op(v, dpp(v, std::integral_constant<int, 0x140>{}));
  if constexpr (LPR >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = op(r[0], r[1]);
  }
  if constexpr (LPR >= 64) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = op(r[0], r[1]);
  }
  return v;
}
// v >= 0 and not NaN (an amax started at 0 and grown by fmaxf, which drops
// NaN): the unsigned order of the bit patterns is the float order, and 0 is
// the identity of the unsigned max the DPP moves fold into
template <int LPR>
__device__ __forceinline__ float lane_group_max(float v) {
  return __uint_as_float(lane_group_reduce<LPR>(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return a > b ? a : b;
  }));
}
template <int LPR>
__device__ __forceinline__ int lane_group_sum(int v) {
  return (int)lane_group_reduce<LPR>((uint32_t)v, [](uint32_t a, uint32_t b) { return a + b; });
}

template <int DT> struct Elem;
template <> struct Elem<SL8_DTYPE_F16> {
  using T = uint16_t;
  __device__ static float ld(const T* p, int64_t i) { return h2f(p[i]); }
  __device__ static float round(float v) { return h2f(f2h_bits(v)); }
};
template <> struct Elem<SL8_DTYPE_BF16> {
  using T = uint16_t;
  __device__ static float ld(const T* p, int64_t i) { return bf2f(p[i]); }
  __device__ static float round(float v) { return bf2f(f2bf_bits(v)); }
};
template <> struct Elem<SL8_DTYPE_F32> {
  using T = float;
  __device__ static float ld(const T* p, int64_t i) { return p[i]; }
  __device__ static float round(float v) { return v; }
};

__device__ __forceinline__ int8_t code_of(float v, float safe) {
  float r = rintf(__fdiv_rn(v, safe));
  r = fminf(fmaxf(r, -127.f), 127.f);
  return static_cast<int8_t>(r);
}

template <int DT> struct VecIO;
template <> struct VecIO<SL8_DTYPE_F16> {
  static constexpr int EPV = 8;
  __device__ static void unpack(uint4 v, float* f) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) { f[2 * i] = h2f(w[i] & 0xFFFF); f[2 * i + 1] = h2f(w[i] >> 16); }
  }
};
template <> struct VecIO<SL8_DTYPE_BF16> {
  static constexpr int EPV = 8;
  __device__ static void unpack(uint4 v, float* f) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) { f[2 * i] = bf2f(w[i] & 0xFFFF); f[2 * i + 1] = bf2f(w[i] >> 16); }
  }
};
template <> struct VecIO<SL8_DTYPE_F32> {
  static constexpr int EPV = 4;
  __device__ static void unpack(uint4 v, float* f) {
    f[0] = __uint_as_float(v.x); f[1] = __uint_as_float(v.y);
    f[2] = __uint_as_float(v.z); f[3] = __uint_as_float(v.w);
  }
};

// Eight codes clamp(rint(fl(x / safe))) without a division per element.
// |x| <= amax, so |x / safe| <= 127 * (1 + 2^-23) and, with inv = v_rcp_f32(safe)
// (at most 1 ulp from 1 / safe; safe is normal and above 2^-120: fp16 rows always
// are, 2^-24 / 127 at least, bf16 callers check), the exact product x * inv is within
// 128 * 2^-23 = 2^-16 of x / safe, and fl(x / safe) within 2^-17 of that. One fma
// against 1.5 * 2^23 rounds the product to the nearest integer n (ties to even) and
// leaves n's two's complement in the low bits; a second one gives its distance from
// n. Unless that exceeds 0.5 - 2^-14, fl(x / safe) rounds to n too. Lanes holding a
// farther element (about 1e-4 of them) or a NaN take the IEEE division, under a
// wave-uniform branch so the common path never executes it: 4.3 VALU instructions an
// element, where a product, its rounding, a comparison, the clamp and the conversion took 8.5.
// safe, inv: per element (codes8: one scale for all); fast: every scale is in that range, else
// every element is divided.
__device__ __forceinline__ uint2 codes8_each(const float* f, const float* safe, const float* inv,
                                             bool fast) {
  constexpr float MAGIC = 12582912.f;  // 1.5 * 2^23
  float t[8], far = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    t[e] = fmaf(f[e], inv[e], MAGIC);
    // (maximum: NaN stays)
    far = __builtin_elementwise_maximum(far, fabsf(fmaf(f[e], inv[e], MAGIC - t[e])));
  }
  const bool amb = !fast || !(far <= 0.5f - 0x1p-14f);
  if (__builtin_expect(__ballot(amb) != 0, 0)) {
    if (amb) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float n = rintf(__fdiv_rn(f[e], safe[e]));
        // NaN: the clamp of fmaxf / fminf gives -127
        t[e] = (n != n ? -127.f : fminf(fmaxf(n, -127.f), 127.f)) + MAGIC;
      }
    }
  }
  uint32_t w[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    // the low bytes of four words -> one dword (v_perm_b32: selectors 0-3 pick the
    // second operand's bytes, 4-7 the first's, 0x0c a zero byte)
    const uint32_t lo = __builtin_amdgcn_perm(__float_as_uint(t[4 * i + 1]), __float_as_uint(t[4 * i]),
                                              0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm(__float_as_uint(t[4 * i + 3]),
                                              __float_as_uint(t[4 * i + 2]), 0x04000c0cu);
    w[i] = lo | hi;
  }
  return make_uint2(w[0], w[1]);
}
__device__ __forceinline__ uint2 codes8(const float* f, float safe) {
  const float s[8] = {safe, safe, safe, safe, safe, safe, safe, safe};
  const float r = __builtin_amdgcn_rcpf(safe);
  const float inv[8] = {r, r, r, r, r, r, r, r};
  return codes8_each(f, s, inv, true);
}

// The same codes by IEEE division (any safe).
__device__ __forceinline__ uint2 codes8_exact(const float* f, float safe) {
  uint32_t w[2] = {0, 0};
#pragma unroll
  for (int e = 0; e < 8; ++e) w[e / 4] |= (uint32_t)(uint8_t)code_of(f[e], safe) << (8 * (e % 4));
  return make_uint2(w[0], w[1]);
}

// Eight codes of a 16-bit row (see codes8; bf16 rows may have scales below its range).
template <int DT>
__device__ __forceinline__ uint2 row_codes8(const float* f, float safe) {
  return DT == SL8_DTYPE_F16 || safe >= 0x1p-120f ? codes8(f, safe) : codes8_exact(f, safe);
}

// Lanes per row (8 elements, 16 bytes each); the first D / 8 of them hold elements.
constexpr int row_lanes(int D) { return D <= 32 ? 4 : D <= 64 ? 8 : D <= 128 ? 16 : 32; }

// Normalised Sylvester-Hadamard transform of a row of D values (a power of two, 32..256) held
// 8 per lane by row_lanes(D) consecutive lanes (element 8 * lane + e): the same orthogonal
// rotation as x @ M, M[i][j] = (-1)^popcount(i & j) / sqrt(D), in D log2(D) adds instead of D^2
// multiply-adds. 32-bit sums over log2(D) levels: a rounding error of at most log2(D) * 2^-24 of
// the row's 2-norm per element, where a running sum of D products has up to D * 2^-24 of it.
// Lane partners by DPP (xor 1, 2; xor 4 and 8 as two mirrors / a rotation inside the 16-lane
// row), xor 16 by v_permlane16_swap.
// WIDE (bf16 rows, whose sums can pass the largest float where the result does not): a power of two
// of the factor goes first, which changes no rounding.
template <int D, bool WIDE>
__device__ __forceinline__ void hadamard_row(float* f, int lane) {
  static_assert(D >= 32 && D <= 256 && (D & (D - 1)) == 0, "power-of-two head dim");
  constexpr int LPR = row_lanes(D);
  constexpr float PRE = D >= 128 ? 0x1p-4f : 0x1p-3f;
  static_assert(PRE * PRE * D <= 1.f && PRE * PRE * D >= 0.5f, "the power of two below 1 / sqrt(D)");
  if constexpr (WIDE) {
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] *= PRE;
  }
#pragma unroll
  for (int s = 1; s < 8; s <<= 1)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (!(e & s)) {
        const float a = f[e], b = f[e | s];
        f[e] = a + b;
        f[e | s] = a - b;
      }
  auto dpp = [](float x, auto ctrl) __attribute__((always_inline)) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value,
                                                      0xF, 0xF, false));
  };
  auto stage = [&](int bit, auto partner) __attribute__((always_inline)) {
    const float sgn = (lane & bit) ? -1.f : 1.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = fmaf(f[e], sgn, partner(f[e]));
  };
  using std::integral_constant;
  stage(1, [&](float x) { return dpp(x, integral_constant<int, 0xB1>{}); });  // quad_perm 1,0,3,2
  stage(2, [&](float x) { return dpp(x, integral_constant<int, 0x4E>{}); });  // quad_perm 2,3,0,1
  if constexpr (LPR >= 8)  // xor 7 (row_half_mirror), then xor 3 (quad_perm 3,2,1,0)
    stage(4, [&](float x) {
      return dpp(dpp(x, integral_constant<int, 0x141>{}), integral_constant<int, 0x1B>{});
    });
  if constexpr (LPR >= 16)  // row_ror:8
    stage(8, [&](float x) { return dpp(x, integral_constant<int, 0x128>{}); });
  if constexpr (LPR >= 32)
    stage(16, [&](float x) {
      const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
      return __uint_as_float((lane & 16) ? r[0] : r[1]);
    });
  const float rs = (float)(1.0 / __builtin_sqrt((double)D)) * (WIDE ? 1.f / PRE : 1.f);
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] *= rs;
}

// The rotation of a row as its own pass would store it: rounded to its storage type.
template <int DT, int D>
__device__ __forceinline__ void rotate_row(float* f, int lane) {
  hadamard_row<D, DT != SL8_DTYPE_F16>(f, lane);
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = Elem<DT>::round(f[e]);
}

}  // namespace
}  // namespace sl8
