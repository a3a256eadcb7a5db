// Tiled Q4_K / Q5_K GEMM for M > 16 (prefill; reference csrc/include/gemm_q4k_dp4a.cuh:60-350,
// csrc/kernel/gemm_dp4a.cu:146-193), gfx950.
//
//   y[m,n] = x_scale[m] * sum_j ( d*sc_j*<x_j, q_j> - dmin*m_j*sum(x_j) )
//
// The products run on v_mfma_f32_32x32x16_f16 with integer operands that fp16 holds exactly: the
// int8 activation codes, and q * sc <= 31 * 63 = 1953 < 2048. A super-block's sum is an integer of at
// most 256 * 127 * 1953 = 6.3e7 in magnitude (Q4_K: half of it), held in the fp32 accumulator: exact
// while every running sum stays below 2^24 = 1.7e7, as those of usual activations do (at most 2.5e6
// over 1e7 sums of N(0, 1) rows and random Q5_K blocks); beyond, each of the 16 steps rounds at 2^-24
// of the running sum, where an int32 sum would be rounded once. Relative error against 64 bits of fp32
// outputs, M x N x K: 17 x 4096 x 4096 0.8e-7, 512 x 17408 x 5120 1.2e-7 (the int8 kernels, which sum
// the super-blocks in one run, 1.1e-7 and 1.2e-7).
// One fp16 MFMA per 16 elements costs what the two int8 MFMAs (Q4_K: the 6-bit scale in 3-bit
// halves; Q5_K: three) per 32 elements did, but it leaves one accumulator instead of two: a wave
// owns 32 columns x 128 rows at two waves per SIMD, so a weight operand is built once per 128 rows,
// and a super-block's sum enters the result with one fma instead of a shift-add, a conversion and
// an fma. What bounds it: MFMA and VALU issue of the same SIMD add up (a 32x32 MFMA takes 15.5 ns,
// each VALU instruction about 1 ns beyond the first few); per super-block a wave issues 64 MFMAs
// and 310 VALU instructions (operands 160, sums 128).
//
// Workgroup: 4 waves, wave w over output columns 32 w .. 32 w + 31 of its 128 and all its RB * 32
// rows; two workgroups a CU, so that one's operand building, sums and barriers run under the
// other's MFMAs. N = 17408, K = 5120, M = 512 / 2000 with the activations' preparation: Q4_K
// 107 / 400 us (830 / 890 useful TFLOP/s; a large bf16 library product reaches 1350 on the card,
// whose clock drops under either), Q5_K 114 / 425; the int8 kernels before it 135 and 159 us at
// M = 512. Small calls gain by the K split: M = 20, N = K = 4096 36 -> 11 us.
//   * weights: raw super-blocks, global -> LDS by DMA one super-block ahead;
//   * activations: the codes as fp16 in the order below and their 16-element sums, made once per
//     call by kq_prep_* and copied global -> LDS by DMA one phase (1 / PH of a super-block) ahead.
//     XI8: no scratch for those was given; int8 codes go through registers instead (64-row tiles
//     where they are faster than gemm_kq_tile_i8.hip's: plan_q45_whole);
//   * operand order: lane half h of the MFMA holds the elements of sub-blocks 4 h .. 4 h + 3, so a
//     lane's weight bytes are contiguous (64 of a super-block's 128) and its scales are one dword.
//     MFMA step t of a super-block: 8 elements 8 p .. of sub-block 4 h + 2 hs + hi, with t =
//     8 hs + 2 p + hi (hi: the high nibbles of the bytes whose low ones step t - 1 took). 8 elements are kept in
//     the order 0 2 1 3 4 6 5 7 in both operands: the order a dword of nibbles yields with one
//     shift (bytes 0 and 2, then 1 and 3);
//   * q * sc: a masked nibble as an fp16 subnormal times the scale, one packed multiply;
//   * min term: U = sum_j m_j xsum_j by one MFMA per row block and super-block on the 16-element
//     sums (|s| <= 2032) and the 6-bit mins.
//
// Tiles that do not fill a round of the chip are split over K (fp32 partials, summed in order by a
// second kernel): see plan_tiles.

#include <algorithm>

#include "kquant.hpp"
#include "rowquant.hpp"

namespace sl8 {
namespace {

typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ v2h as_v2h(uint32_t x) { return __builtin_bit_cast(v2h, x); }

// Barrier that orders LDS only: DMA and register loads of later stages stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 8 codes (two dwords of bytes) as fp16 in operand order: bytes 0, 2, 1, 3 of each dword
__device__ __forceinline__ uint4 codes_to_h8(uint32_t a, uint32_t b) {
  const v2h bias = {(_Float16)-1152.f, (_Float16)-1152.f};
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t u = (k ? b : a) ^ 0x80808080u;
    // (u0, 0x64, u2, 0x64) and (u1, 0x64, u3, 0x64): 1024 + x + 128
    const uint32_t e = __builtin_amdgcn_perm(0x64646464u, u, 0x04020400u);
    const uint32_t d = __builtin_amdgcn_perm(0x64646464u, u, 0x04030401u);
    o[2 * k] = __builtin_bit_cast(uint32_t, as_v2h(e) + bias);
    o[2 * k + 1] = __builtin_bit_cast(uint32_t, as_v2h(d) + bias);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}
__device__ __forceinline__ int sum4(uint32_t x, int acc) {
  return __builtin_amdgcn_sdot4((int)x, 0x01010101, acc, false);
}

// A tile call's activations: fp16 codes [M][K] and 16-element sums [M][K / 16], or (XI8) the codes.
struct TileX {
  const int8_t* x8;
  const uint16_t *xh, *xsum;
  const float* scale;
};

template <int FMT, int OUT_DT, int RB, int PH, bool XI8>
__global__ void __launch_bounds__(256, 2)
gemm_kq_tile_kernel(const TileX tx, const uint8_t* __restrict__ w, void* __restrict__ out, int M,
                    int N, int K, const TileWork tw) {
  constexpr int NT = 256, BM = 32 * RB, BN = 128;
  constexpr int BB = FMT == 4 ? 144 : 176;  // bytes per super-block
  constexpr int CH = BB / 16;
  constexpr int QS = FMT == 4 ? 16 : 48;    // offset of the nibbles
  constexpr int SPP = 16 / PH;              // MFMA steps per phase
  constexpr int CPR = 2 * SPP;              // 16-byte activation chunks per row and phase
  constexpr int XL = XI8 ? BM * 8 / NT : BM * CPR / NT;  // activation copies per thread and phase
  static_assert(!XI8 || PH == 2, "the register path stages half super-blocks");
  static_assert(BM * CPR % NT == 0 && BN * CH * 2 % NT == 0, "whole copies");
  // one LDS object per stage: a copy into one never aliases reads of another
  __shared__ uint4 xs0[BM * CPR], xs1[BM * CPR];  // fp16 [row][h * SPP + step], swizzled by row
  __shared__ uint4 ws0[BN * CH], ws1[BN * CH];
  __shared__ uint4 su_l[BM * 2];                  // the super-block's sums, fp16 [row][piece]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int nsb = K >> 8;
  const TileRange tr = tile_range(tw, nsb);
  const int sb0 = tr.sb0, sb1 = tr.sb1, n0 = tr.ct * BN, m0 = tr.rt * BM;
  const int64_t row_bytes = (int64_t)nsb * BB;
  // LDS rows of 8 chunks are half a bank line, of 16 a whole one
  auto swz = [](int row) { return CPR == 8 ? (row >> 1) & 7 : row & 15; };

  // The operands through buffer resources: per-lane offsets fixed for the kernel, the super-block
  // in the scalar offset (no address arithmetic in the loop); rows past M or N read as zeros.
  const int mrows = min(BM, M - m0);
  const brsrc_t r_w = make_rsrc(w + (int64_t)n0 * row_bytes, (uint32_t)(min(BN, N - n0) * row_bytes));
  const brsrc_t r_x = XI8 ? make_rsrc(tx.x8 + (int64_t)m0 * K, (uint32_t)(mrows * K))
                          : make_rsrc(tx.xh + (int64_t)m0 * K, (uint32_t)(mrows * K * 2));
  const brsrc_t r_s = make_rsrc(XI8 ? nullptr : tx.xsum + (int64_t)m0 * (K / 16),
                                XI8 ? 0u : (uint32_t)(mrows * (K / 8)));
  constexpr int WCH = BN * CH, WL = (WCH + NT - 1) / NT;  // weight chunks of a super-block, copies
  uint32_t wo[WL], xo[XL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int P = i * NT + tid, row = P / CH;
    wo[i] = (uint32_t)(row * row_bytes) + 16u * (P - CH * row);
  }
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int P = i * NT + tid;
    if constexpr (XI8) {  // 16-element piece q of row P / 8: lane half q / 4, piece q % 4
      const int q = P & 7;
      xo[i] = (uint32_t)((P >> 3) * K + 128 * (q >> 2) + 16 * (q & 3));
    } else {  // LDS chunk P holds chunk c of its row: lane half c / SPP, step s of the phase
      const int row = P / CPR, c = (P % CPR) ^ swz(row), s = c % SPP;
      xo[i] = 2u * (uint32_t)(row * K + 128 * (c / SPP) + 64 * (s >> 3) + 32 * (s & 1) + 8 * ((s >> 1) & 3));
    }
  }
  const uint32_t so = (uint32_t)((tid >> 1) * (K / 8) + 16 * (tid & 1));
  // weight super-block sb -> wd; chunk P of the tile lands at wd[P]
  auto load_w = [&](int sb, uint4* wd) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WL; ++i)
      if (i * NT + wave * 64 < WCH)  // wave-uniform: the last copy may be a part
        buf16_to_lds(r_w, wd + i * NT + wave * 64, wo[i], (uint32_t)sb * BB);
  };
  uint4 xr[XI8 ? XL : 1];
  // activations of phase ph of super-block sb
  auto load_x = [&](int sb, int ph, uint4* xd) __attribute__((always_inline)) {
    if constexpr (XI8) {
#pragma unroll
      for (int i = 0; i < XL; ++i)
        xr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                              r_x, xo[i], (uint32_t)(sb * 256 + 64 * ph), 0));
    } else {
      const int t0 = ph * SPP;  // first step: 64 elements per 8 steps, 8 per 2
      const uint32_t off = 2u * (uint32_t)(sb * 256 + 64 * (t0 >> 3) + 8 * ((t0 >> 1) & 3));
#pragma unroll
      for (int i = 0; i < XL; ++i) buf16_to_lds(r_x, xd + i * NT + wave * 64, xo[i], off);
    }
  };
  auto load_sums = [&](int sb) __attribute__((always_inline)) {
    if constexpr (!XI8) {
      if (wave * 64 < BM * 2) buf16_to_lds(r_s, su_l + wave * 64, so, (uint32_t)sb * 32);
    }
  };
  auto store_x = [&](uint4* xd, int ph) __attribute__((always_inline)) {
    if constexpr (XI8) {
#pragma unroll
      for (int i = 0; i < XL; ++i) {
        const int P = i * NT + tid, row = P >> 3, q = P & 7;
        const uint4 v = xr[i];
        // elements 16 (q % 4) .. of the phase's 64: sub-block (q % 4) / 2 (hi), step pairs p, p + 1
        const int c = SPP * (q >> 2) + 4 * (q & 1) + ((q >> 1) & 1);
        xd[row * CPR + (c ^ swz(row))] = codes_to_h8(v.x, v.y);
        xd[row * CPR + ((c + 2) ^ swz(row))] = codes_to_h8(v.z, v.w);
        const int sum = sum4(v.w, sum4(v.z, sum4(v.y, sum4(v.x, 0))));
        reinterpret_cast<_Float16*>(su_l)[row * 16 + 8 * (q >> 2) + 4 * ph + (q & 3)] = (_Float16)(float)sum;
      }
    }
  };

  float f[RB][16];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int e = 0; e < 16; ++e) f[rb][e] = 0.f;
  v16f T[RB];
  float d = 0.f, dmin = 0.f;
  uint32_t scw = 0, mnw = 0;  // scales and mins of sub-blocks 4 h .. 4 h + 3

  // the SPP steps of phase ph
  auto compute = [&](const uint4* xt, const uint4* wt, auto ph_tag) __attribute__((always_inline)) {
    constexpr int ph = decltype(ph_tag)::value, t0 = ph * SPP;
    const uint8_t* wr = reinterpret_cast<const uint8_t*>(wt) + (32 * wave + l32) * BB;
    if constexpr (ph == 0) {
      const uint4 hd = *reinterpret_cast<const uint4*>(wr);
      d = 16384.f * h2f(hd.x & 0xFFFFu);  // 2^14: see the operand scale below
      dmin = h2f(hd.x >> 16);
      const ScMin sm = unpack_scmin(hd.y, hd.z, hd.w);
      scw = h ? sm.sc_hi : sm.sc_lo;
      mnw = h ? sm.mn_hi : sm.mn_lo;
    }
    // the phase's weight dwords (two per step pair) and, Q5_K, their 5th bits
    constexpr int NP = SPP / 2;
    uint32_t qw[2 * NP], qh[FMT == 5 ? 2 * NP : 1];
    v2h mul[NP >= 4 ? NP / 4 : 1][2];
#pragma unroll
    for (int k = 0; k < NP / 2; ++k) {  // 16 bytes: step pairs p0, p0 + 1
      const int tp = t0 + 4 * k, hs = tp >> 3, p0 = (tp >> 1) & 3;
      const uint4 a = *reinterpret_cast<const uint4*>(wr + QS + 64 * h + 32 * hs + 8 * p0);
      qw[4 * k] = a.x; qw[4 * k + 1] = a.y; qw[4 * k + 2] = a.z; qw[4 * k + 3] = a.w;
      if constexpr (FMT == 5) {
        // bit 2 (2 h + hs) (+ 1) of byte l is the 5th bit of element l
        const uint4 b = *reinterpret_cast<const uint4*>(wr + 16 + 8 * p0);
        const int sh = 4 * h + 2 * hs;
        qh[4 * k] = b.x >> sh; qh[4 * k + 1] = b.y >> sh; qh[4 * k + 2] = b.z >> sh; qh[4 * k + 3] = b.w >> sh;
      }
    }
    // A code q in the low bits of a 16-bit half is the fp16 subnormal q * 2^-24 (16 q * 2^-24 for
    // a high nibble in place): times sc * 2^10 (sc * 2^6), all exact, it is q * sc * 2^-14, an fp16
    // normal or zero; the 2^14 goes into d.
#pragma unroll
    for (int k = 0; k < (NP >= 4 ? NP / 4 : 1); ++k) {
      const int hs = (t0 + 8 * k) >> 3;
      const _Float16 m0h = (_Float16)(1024.f * (float)((scw >> (16 * hs)) & 0xFF));
      const _Float16 m1h = (_Float16)((FMT == 4 ? 64.f : 1024.f) * (float)((scw >> (16 * hs + 8)) & 0xFF));
      mul[k][0] = v2h{m0h, m0h};
      mul[k][1] = v2h{m1h, m1h};
    }
    v8h A[2][RB], B[2];
    auto read_a = [&](int s, int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int row = 32 * rb + l32;
        A[buf][rb] = __builtin_bit_cast(v8h, xt[row * CPR + ((SPP * h + s) ^ swz(row))]);
      }
    };
    // step s of the phase: 8 low (s even) or high (s odd) nibbles of dwords 2 (s / 2) and the next
    auto build = [&](int s, int buf) __attribute__((always_inline)) {
      const int hi = s & 1;
      const v2h mv = mul[s >> 3][hi];
      uint32_t r[4];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int i = 2 * (s >> 1) + k;
        uint32_t e, o;
        if constexpr (FMT == 4) {
          const uint32_t msk = hi ? 0x00F000F0u : 0x000F000Fu;
          e = qw[i] & msk;
          o = (qw[i] >> 8) & msk;
        } else {
          const uint32_t q = ((hi ? qw[i] >> 4 : qw[i]) & 0x0F0F0F0Fu) |
                             ((hi ? qh[i] << 3 : qh[i] << 4) & 0x10101010u);
          e = q & 0x00FF00FFu;
          o = (q >> 8) & 0x00FF00FFu;
        }
        r[2 * k] = __builtin_bit_cast(uint32_t, as_v2h(e) * mv);
        r[2 * k + 1] = __builtin_bit_cast(uint32_t, as_v2h(o) * mv);
      }
      B[buf] = __builtin_bit_cast(v8h, make_uint4(r[0], r[1], r[2], r[3]));
    };
    read_a(0, 0);
    build(0, 0);
#pragma unroll
    for (int s = 0; s < SPP; ++s) {
      const int c = s & 1;
      __builtin_amdgcn_sched_barrier(0);
      if (s < SPP - 1) read_a(s + 1, c ^ 1);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
        T[rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[c][rb], B[c], t0 + s == 0 ? v16f{} : T[rb],
                                                       0, 0, 0);
      if (s < SPP - 1) build(s + 1, c ^ 1);
      __builtin_amdgcn_sched_group_barrier(0x100, RB, 0);  // the LDS reads first
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, (FMT == 4 ? 10 : 20) / RB, 0);  // VALU
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // f += d * T - dmin * U of the super-block
  auto flush = [&]() __attribute__((always_inline)) {
    v8h ub;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const _Float16 mv = (_Float16)(float)((mnw >> (8 * j)) & 0xFF);
      ub[2 * j] = mv;
      ub[2 * j + 1] = mv;
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const v8h a = __builtin_bit_cast(v8h, su_l[(32 * rb + l32) * 2 + h]);
      const v16f u = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ub, v16f{}, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 16; ++e) f[rb][e] = fmaf(d, T[rb][e], f[rb][e]);
#pragma unroll
      for (int e = 0; e < 16; ++e) f[rb][e] = fmaf(-dmin, u[e], f[rb][e]);
    }
  };

  // One super-block: phase ph computes from one activation stage while the other fills. The
  // activations' copies are issued first, so waiting for them leaves the later ones in flight.
  auto superblock = [&](int sb, const uint4* wc, uint4* wn) __attribute__((always_inline)) {
    const bool more = sb + 1 < sb1;
    auto phase = [&](auto ph_tag) __attribute__((always_inline)) {
      constexpr int ph = decltype(ph_tag)::value;
      uint4* xc = (ph & 1) ? xs1 : xs0;
      uint4* xn = (ph & 1) ? xs0 : xs1;
      const bool next = ph + 1 < PH || more;
      if (next) load_x(ph + 1 < PH ? sb : sb + 1, (ph + 1) % PH, xn);
      if constexpr (ph == 0) {
        // (in this order: the wait below counts on it)
        __builtin_amdgcn_sched_barrier(0);
        load_sums(sb);
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_w(sb + 1, wn);
        __builtin_amdgcn_sched_barrier(0);
      }
      compute(xc, wc, ph_tag);
      if constexpr (ph == PH - 1) flush();
      if constexpr (XI8) {
        if (ph == PH - 1) lds_barrier();  // the sums are rewritten
        if (next) store_x(xn, (ph + 1) % PH);
      }
      // phase 0: the next weights' copies (at least WCH / NT of a wave's) may stay in flight
      constexpr unsigned LATER = XI8 || PH == 1 || ph != 0 ? 0 : WCH / NT;
      if (LATER && more) __builtin_amdgcn_s_waitcnt(0x0F70 | LATER);
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      lds_barrier();
    };
    phase(std::integral_constant<int, 0>{});
    if constexpr (PH >= 2) phase(std::integral_constant<int, 1>{});
    if constexpr (PH >= 4) {
      phase(std::integral_constant<int, 2>{});
      phase(std::integral_constant<int, 3>{});
    }
  };
  static_assert(PH == 2 || PH == 4, "an even number of phases: a super-block starts in stage 0");

  load_x(sb0, 0, xs0);
  load_w(sb0, ws0);
  store_x(xs0, 0);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  lds_barrier();
  for (int sb = sb0; sb < sb1; sb += 2) {
    superblock(sb, ws0, ws1);
    if (sb + 1 < sb1) superblock(sb + 1, ws1, ws0);
  }

  const int cl = 32 * wave + l32, n = n0 + cl;
  if (tr.part) {
    float* pt = tr.part + (int64_t)BM * BN * tr.sp;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int e = 0; e < 16; ++e) pt[(32 * rb + 8 * (e >> 2) + 4 * h + (e & 3)) * BN + cl] = f[rb][e];
    return;
  }
  // the row scales first, unconditionally (clamped rows): one wait, not one per element
  float xsv[RB][16];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int e = 0; e < 16; ++e)
      xsv[rb][e] = tx.scale[min(m0 + 32 * rb + 8 * (e >> 2) + 4 * h + (e & 3), M - 1)];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int m = m0 + 32 * rb + 8 * (e >> 2) + 4 * h + (e & 3);
      if (m < M && n < N) st_out<OUT_DT>(out, (int64_t)m * N + n, f[rb][e] * xsv[rb][e]);
    }
}

// The activations of a call, one workgroup per row: int8 codes and scale as sl8_quantize_i8_rowwise
// (16-bit x), stored as fp16 in operand order, and their 16-element sums.
template <int DT, int BT, int NV>
__global__ void __launch_bounds__(BT)
kq_prep_rows_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ xh,
                    uint16_t* __restrict__ xsum, float* __restrict__ scale, int K) {
  const int64_t row = blockIdx.x;
  const uint4* xr = reinterpret_cast<const uint4*>(x + row * K);
  const int nvec = K / 8;  // a multiple of 32: no wave holds a part of a 16-element pair
  uint4 raw[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = v * BT + threadIdx.x;
    raw[v] = i < nvec ? xr[i] : make_uint4(0, 0, 0, 0);
  }
  float f[NV][8], amax = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    VecIO<DT>::unpack(raw[v], f[v]);
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(f[v][e]));
  }
  __shared__ float red[BT / 64];
  amax = lane_group_max<64>(amax);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < BT / 64; ++i) amax = fmaxf(amax, red[i]);
  const float s = amax * (1.0f / 127.0f);
  const float safe = (s == 0.f) ? 1.f : s;
  if (threadIdx.x == 0) scale[row] = safe;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = v * BT + threadIdx.x;
    if (i < nvec) {
      const uint2 c = row_codes8<DT>(f[v], safe);
      reinterpret_cast<uint4*>(xh + row * K)[i] = codes_to_h8(c.x, c.y);
      const int sum = lane_group_sum<2>(sum4(c.y, sum4(c.x, 0)));
      if (!(i & 1)) xsum[row * (K / 16) + (i >> 1)] = f2h_bits((float)sum);
    }
  }
}

// The same from int8 codes: a thread per 16 elements.
__global__ void __launch_bounds__(256)
kq_prep_codes_kernel(const int8_t* __restrict__ x, uint16_t* __restrict__ xh,
                     uint16_t* __restrict__ xsum, int64_t pieces) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  const uint4 v = reinterpret_cast<const uint4*>(x)[i];
  reinterpret_cast<uint4*>(xh)[2 * i] = codes_to_h8(v.x, v.y);
  reinterpret_cast<uint4*>(xh)[2 * i + 1] = codes_to_h8(v.z, v.w);
  xsum[i] = f2h_bits((float)sum4(v.w, sum4(v.z, sum4(v.y, sum4(v.x, 0)))));
}

// Sums the S partials of each split tile in order, scales the rows and stores them: one thread per
// 4 columns of a row.
template <int OUT_DT>
__global__ void __launch_bounds__(256)
gemm_kq_reduce_kernel(const float* __restrict__ x_scale, void* __restrict__ out, int M, int N, int BM,
                      int BN, const TileWork tw) {
  const int per_tile = BM * BN / 4 / 256;  // blocks per tile
  const int i = blockIdx.x / per_tile;
  const int id = (blockIdx.x % per_tile) * 256 + threadIdx.x;
  const int row = id / (BN / 4), col = 4 * (id % (BN / 4));
  int ct, rt;
  kq_tile_coords(tw.nfull + i, tw.nt_x, tw.xcd_m, ct, rt);
  const int m = rt * BM + row, n = ct * BN + col;
  if (m >= M || n >= N) return;
  const float* p = tw.part + (int64_t)i * tw.S * BM * BN + (int64_t)row * BN + col;
  float4 a = *reinterpret_cast<const float4*>(p);
#pragma unroll 4
  for (int s = 1; s < tw.S; ++s) {
    const float4 b = *reinterpret_cast<const float4*>(p + (int64_t)s * BM * BN);
    a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
  }
  const float xs = x_scale[m];
  const float v[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) st_out<OUT_DT>(out, (int64_t)m * N + n + e, v[e] * xs);
}

}  // namespace

// The tile shape and the K split of a call, by a model of its time: rounds of whole tiles over the
// chip, then the remaining tiles, each split over K into S parts (of at least two super-blocks) if
// that is faster with the partials' traffic. A round that leaves workgroup slots of a CU empty is
// faster per workgroup, but not in proportion.
// us of nsb super-blocks of n workgroups of a shape, in rounds over P CUs
static double rounds_us(int64_t n, int P, int nsb, const TileShape& s) {
  const int64_t slots = (int64_t)P * s.wgs_per_cu, rem = n % slots;
  double t = (double)(n / slots) * nsb * s.us_per_sb;
  if (rem) {
    const int64_t k = (rem + P - 1) / P;  // workgroups per CU
    t += (double)nsb * s.us_per_sb * (0.3 + 0.7 * (double)k / s.wgs_per_cu);
  }
  return t;
}

TilePlan plan_tiles(int M, int N, int K, const TileShape* shapes, int count, bool may_split) {
  const int P = cu_count(), nsb = K >> 8;
  TilePlan best{};
  best.us = 1e30;
  for (int i = 0; i < count; ++i) {
    const TileShape& s = shapes[i];
    const int nt_x = (N + s.bn - 1) / s.bn;
    const int64_t T = (int64_t)nt_x * ((M + s.bm - 1) / s.bm);
    const int64_t slots = (int64_t)P * s.wgs_per_cu, full = T / slots, rem = T % slots;
    const int smax = may_split && rem ? (int)std::max<int64_t>(1, std::min<int64_t>({slots / rem, nsb / 2, 16})) : 1;
    for (int S = 1; S <= smax; ++S) {
      double t = rounds_us(full * slots, P, nsb, s) + rounds_us(rem * S, P, (nsb + S - 1) / S, s);
      if (S > 1) t += 3.0 + (double)rem * S * s.bm * s.bn * 8 / 5e6;
      if (t < best.us) best = TilePlan{i, nt_x, S, S > 1 ? T - rem : T, S > 1 ? rem : 0, 0, t};
    }
  }
  best.part_bytes = (size_t)best.nsplit * best.S * shapes[best.shape].bm * shapes[best.shape].bn * 4;
  return best;
}

TailPlan plan_tail(int M, int N, int K, const TileShape& tile, const TileShape& quarter) {
  const int P = cu_count(), nsb = K >> 8, nt_x = (N + tile.bn - 1) / tile.bn;
  const int64_t T = (int64_t)nt_x * ((M + tile.bm - 1) / tile.bm), rem = T % P;
  const int64_t cut = T >= P && rem <= P / 2 ? rem : 0;
  TailPlan p{nt_x, T - cut, cut, rounds_us(T - cut, P, nsb, tile)};
  if (cut) p.us += 3.0 + rounds_us(4 * cut, P, nsb, quarter);
  return p;
}

namespace {

// us_per_sb: one super-block of one workgroup with every slot of its CU taken (measured)
constexpr TileShape SHAPES4[] = {{128, 128, 2, 4.7}, {64, 128, 2, 2.7}, {32, 128, 3, 2.5}};
constexpr TileShape SHAPES5[] = {{128, 128, 2, 5.0}, {64, 128, 2, 3.1}, {32, 128, 2, 2.1}};

// Without scratch: the int8 kernel's 128-row tiles (gemm_kq_tile_i8.hip) and row quarters, or this
// one's 64-row tiles from int8 codes, whichever the model has faster. The latter win where the CUs
// are not filled or a last round of the former would be long, the former at even rounds and short
// last ones. M x N x K, us as 128-row / 64-row tiles: Q4_K 512 x 17408 x 5120 125 / 135, 512 x 5120
// x 17408 145 / 163, 300 x 17408 x 5120 94 / 84, 32 x 4096 x 4096 35 / 27; Q5_K 512 x 5120 x 17408
// 185 / 196, 1500 x 4096 x 4096 105 / 84.
constexpr TileShape I8_TILE[] = {{128, 128, 1, 2.45}, {128, 128, 1, 3.15}};    // Q4_K, Q5_K
constexpr TileShape I8_QUARTER[] = {{32, 128, 1, 1.2}, {32, 128, 1, 1.47}};
constexpr TileShape XI8_TILE[] = {{64, 128, 2, 2.6}, {64, 128, 2, 3.2}};

template <int FMT>
void launch_tiles(const TilePlan& p, const TileX& tx, const uint8_t* w, void* out, int odt, int M,
                  int N, int K, float* part, hipStream_t st) {
  const TileShape& s = (FMT == 4 ? SHAPES4 : SHAPES5)[p.shape];
  const TileWork tw = tile_work(p, s, M, part);
  const unsigned grid = (unsigned)(p.nfull + p.nsplit * p.S);
  auto go = [&](auto dt) {
    constexpr int DT = decltype(dt)::value;
    if (tx.x8) gemm_kq_tile_kernel<FMT, DT, 2, 2, true><<<grid, 256, 0, st>>>(tx, w, out, M, N, K, tw);
    else if (p.shape == 0) gemm_kq_tile_kernel<FMT, DT, 4, 4, false><<<grid, 256, 0, st>>>(tx, w, out, M, N, K, tw);
    else if (p.shape == 1) gemm_kq_tile_kernel<FMT, DT, 2, 2, false><<<grid, 256, 0, st>>>(tx, w, out, M, N, K, tw);
    else gemm_kq_tile_kernel<FMT, DT, 1, 2, false><<<grid, 256, 0, st>>>(tx, w, out, M, N, K, tw);
  };
  if (odt == SL8_DTYPE_F16) go(std::integral_constant<int, SL8_DTYPE_F16>{});
  else if (odt == SL8_DTYPE_BF16) go(std::integral_constant<int, SL8_DTYPE_BF16>{});
  else go(std::integral_constant<int, SL8_DTYPE_F32>{});
  if (p.nsplit) launch_kq_reduce(p, s, tw, tx.scale, out, odt, M, N, st);
}

}  // namespace

void launch_kq_reduce(const TilePlan& p, const TileShape& s, const TileWork& tw, const float* xs,
                      void* out, int odt, int M, int N, hipStream_t st) {
  const unsigned grid = (unsigned)(p.nsplit * (s.bm * s.bn / 1024));
  if (odt == SL8_DTYPE_F16) gemm_kq_reduce_kernel<SL8_DTYPE_F16><<<grid, 256, 0, st>>>(xs, out, M, N, s.bm, s.bn, tw);
  else if (odt == SL8_DTYPE_BF16) gemm_kq_reduce_kernel<SL8_DTYPE_BF16><<<grid, 256, 0, st>>>(xs, out, M, N, s.bm, s.bn, tw);
  else gemm_kq_reduce_kernel<SL8_DTYPE_F32><<<grid, 256, 0, st>>>(xs, out, M, N, s.bm, s.bn, tw);
}

namespace {

// Scratch of a Q4_K / Q5_K call: fp16 codes, sums, scales, then the split tiles' partials.
struct TileScratch {
  TilePlan plan;
  size_t sums, scales, part, bytes;
};
TileScratch tile_scratch(int fmt, int M, int N, int K) {
  TileScratch s{};
  s.plan = plan_tiles(M, N, K, fmt == 4 ? SHAPES4 : SHAPES5, 3, true);
  auto at = [&](size_t n) { const size_t o = s.bytes; s.bytes += (n + 255) / 256 * 256; return o; };
  at((size_t)M * K * 2);
  s.sums = at((size_t)M * K / 8);
  s.scales = at((size_t)M * 4);
  s.part = at(s.plan.part_bytes);
  return s;
}

}  // namespace

size_t q45_tile_workspace(int fmt, int M, int N, int K) { return tile_scratch(fmt, M, N, K).bytes; }
TilePlan plan_q45_tile(int fmt, int M, int N, int K) { return tile_scratch(fmt, M, N, K).plan; }

TailPlan plan_q45_whole(int fmt, int M, int N, int K, TilePlan& tiles) {
  const int i = fmt - 4;
  TailPlan p = plan_tail(M, N, K, I8_TILE[i], I8_QUARTER[i]);
  tiles = plan_tiles(M, N, K, XI8_TILE + i, 1, false);
  tiles.shape = 1;
  if (tiles.us <= p.us) p.whole = 0;
  return p;
}

void launch_q45_tile(int fmt, const void* x, int x_dtype, const float* xs, const uint8_t* w, void* out,
                     int odt, int M, int N, int K, void* workspace, hipStream_t st) {
  if (!workspace) {
    TilePlan p;
    const int8_t* x8 = static_cast<const int8_t*>(x);
    const TailPlan tail = plan_q45_whole(fmt, M, N, K, p);
    if (tail.whole) return launch_q45_tile_i8(fmt, tail, x8, xs, w, out, odt, M, N, K, st);
    const TileX tx{x8, nullptr, nullptr, xs};
    if (fmt == 4) launch_tiles<4>(p, tx, w, out, odt, M, N, K, nullptr, st);
    else launch_tiles<5>(p, tx, w, out, odt, M, N, K, nullptr, st);
    return;
  }
  const TileScratch s = tile_scratch(fmt, M, N, K);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  uint16_t* xh = reinterpret_cast<uint16_t*>(ws);
  uint16_t* sums = reinterpret_cast<uint16_t*>(ws + s.sums);
  float* scales = reinterpret_cast<float*>(ws + s.scales);
  if (x_dtype == SL8_KQ_I8) {
    const int64_t pieces = (int64_t)M * K / 16;
    kq_prep_codes_kernel<<<(unsigned)((pieces + 255) / 256), 256, 0, st>>>(
        static_cast<const int8_t*>(x), xh, sums, pieces);
  } else {
    const uint16_t* x16 = static_cast<const uint16_t*>(x);
    auto rows = [&](auto dt, auto bt, auto nv) {
      kq_prep_rows_kernel<decltype(dt)::value, decltype(bt)::value, decltype(nv)::value>
          <<<(unsigned)M, decltype(bt)::value, 0, st>>>(x16, xh, sums, scales, K);
    };
    auto by_k = [&](auto dt) {
      using B = std::integral_constant<int, 256>;
      using L = std::integral_constant<int, 1024>;
      if (K <= 2048) rows(dt, B{}, std::integral_constant<int, 1>{});
      else if (K <= 4096) rows(dt, B{}, std::integral_constant<int, 2>{});
      else if (K <= 8192) rows(dt, B{}, std::integral_constant<int, 4>{});
      else if (K <= 16384) rows(dt, L{}, std::integral_constant<int, 2>{});
      else if (K <= 32768) rows(dt, L{}, std::integral_constant<int, 4>{});
      else rows(dt, L{}, std::integral_constant<int, 8>{});
    };
    if (x_dtype == SL8_DTYPE_F16) by_k(std::integral_constant<int, SL8_DTYPE_F16>{});
    else by_k(std::integral_constant<int, SL8_DTYPE_BF16>{});
  }
  const TileX tx{nullptr, xh, sums, x_dtype == SL8_KQ_I8 ? xs : scales};
  float* part = reinterpret_cast<float*>(ws + s.part);
  if (fmt == 4) launch_tiles<4>(s.plan, tx, w, out, odt, M, N, K, part, st);
  else launch_tiles<5>(s.plan, tx, w, out, odt, M, N, K, part, st);
}

}  // namespace sl8
