// Tiled Q4_K / Q5_K GEMM for M > 16 without scratch (the entries that take no workspace; reference
// csrc/include/gemm_q4k_dp4a.cuh:60-350, csrc/kernel/gemm_dp4a.cu:146-193), gfx950: 128 x 128
// output tiles on the int8 codes. gemm_kq_tile.hip's kernel takes the calls that have scratch, and
// of the others those that its 64-row tiles serve faster (launch_q45_tile).
//
// A workgroup of 8 waves, two per SIMD, each owning 32 output columns x 64 rows (2 blocks of 32 x
// 32; each B operand is built by the two waves of its columns). Per super-block the x tile (128 x
// 256 int8) and the 128 weight super-blocks are copied global -> LDS one super-block ahead
// (double-buffered). The products are exact integers on v_mfma_i32_32x32x32_i8, one K = 32 step per
// sub-block j (lane half h holds its elements 16 h .. 16 h + 15), the 6-bit sc_j split in 3-bit
// halves so that each B operand fits int8:
//   Q4_K  q * sc_j = q (sc_j & 7) + 8 (q (sc_j >> 3)), operands <= 105;
//   Q5_K  with q = n + 16 b (n the low nibble, b the 5th bit): n (sc_j & 7) + 8 (n (sc_j >> 3) +
//         2 b sc_j), operands <= 126;
// two (three) MFMAs into T_lo, T_hi (, T_hi), and once per super-block f += d * (T_lo + 8 T_hi).
// The min term U = sum_j m_j * sum(x_j) is one v_mfma_f32_32x32x16_f16 per row block and super-block
// on the x half-sums and the mins (both exact in fp16; |U| <= 8 * 4064 * 63 < 2^24 an exact fp32
// integer), applied as f -= dmin * U one super-block later: the half-sums of the tile's rows are
// formed once, spread over the waves, and shared through LDS.
// x chunks are XOR-swizzled in LDS by row (rows are 256 B = one bank line); weight rows are 144 or
// 176 B apart, which already spreads 16 rows over all banks.
//
// A last round of tiles that would hold at most half the CUs runs as 4 row quarters each (a second
// launch of 4 waves over 32 rows, the same per-element arithmetic). M = 512, N = 17408, K = 5120:
// Q4_K 125 us (135 as 64-row tiles, whose last round is as long as any), Q5_K 158.

#include <type_traits>

#include "kquant.hpp"

namespace sl8 {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i_t __attribute__((ext_vector_type(16)));
typedef float v16f_t __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int TBM = 128, TBN = 128;  // output tile

// QTR: the quarter blockIdx.x & 3 (32 rows) of tile tile0 + blockIdx.x / 4; else tile0 + blockIdx.x
template <int FMT, int OUT_DT, bool QTR>
__global__ void __launch_bounds__(QTR ? 256 : 512, 1)
gemm_kq_tile_i8_kernel(const int8_t* __restrict__ x, const float* __restrict__ x_scale,
                       const uint8_t* __restrict__ w, void* __restrict__ out, int M, int N, int K,
                       int nt_x, int xcd_m, int tile0) {
  constexpr int RB = QTR ? 1 : 2;           // 32-row blocks per wave
  constexpr int NT = QTR ? 256 : 512;
  constexpr int BB = FMT == 4 ? 144 : 176;  // bytes per super-block
  constexpr int CH = BB / 16;
  constexpr int QS = FMT == 4 ? 16 : 48;    // offset of the nibbles
  constexpr int WCH = (TBN * CH + NT - 1) / NT * NT;  // weight-tile 16-byte chunks, whole copies
  __shared__ __attribute__((aligned(16))) int8_t xs0[TBM * 256];
  __shared__ __attribute__((aligned(16))) int8_t xs1[TBM * 256];
  __shared__ __attribute__((aligned(16))) uint8_t ws0[WCH * 16];
  __shared__ __attribute__((aligned(16))) uint8_t ws1[WCH * 16];
  // full tiles: the min-term MFMA's A operands (x half-sums) of one super-block, [slot][row
  // block][lane], formed by the waves together and read after the next workgroup barrier
  __shared__ __attribute__((aligned(16))) uint4 xh_l[QTR ? 1 : 2][QTR ? 1 : 4][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int tile = tile0 + (QTR ? (int)(blockIdx.x >> 2) : (int)blockIdx.x);
  int ct, rt;
  kq_tile_coords(tile, nt_x, xcd_m, ct, rt);
  const int n0 = ct * TBN, m0 = rt * TBM;
  const int rb0 = QTR ? (int)(blockIdx.x & 3) : 0;
  const int cg = wave & 3;                            // the wave's 32 output columns
  const int rbw = QTR ? rb0 : (wave >> 2) * RB;       // its first row block
  const int nsb = K >> 8;
  const int64_t row_bytes = (int64_t)nsb * BB;

  // copies of super-block sb into (xd, wd); chunk P of the tile lands at P * 16 (a quarter copies
  // only its 32 rows)
  auto load = [&](int sb, int8_t* xd, uint8_t* wd) __attribute__((always_inline)) {
    constexpr int XCH = QTR ? 512 : TBM * 16;
#pragma unroll
    for (int i = 0; i < XCH / NT; ++i) {
      const int P0 = rb0 * 512 + i * NT;
      const int P = P0 + tid, row = P >> 4;
      const int c = (P & 15) ^ (row & 15);
      const int8_t* src = x + (int64_t)min(m0 + row, M - 1) * K + (int64_t)sb * 256 + 16 * c;
      __builtin_amdgcn_global_load_lds((kq_gptr_t)src, (kq_lptr_t)(xd + (P0 + wave * 64) * 16), 16, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < WCH / NT; ++i) {
      const int P = min(i * NT + tid, TBN * CH - 1), row = P / CH, c = P - CH * row;
      const uint8_t* src = w + (int64_t)min(n0 + row, N - 1) * row_bytes + (int64_t)sb * BB + 16 * c;
      __builtin_amdgcn_global_load_lds((kq_gptr_t)src, (kq_lptr_t)(wd + (i * NT + wave * 64) * 16), 16, 0, 0);
    }
  };

  float f[RB][16];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int e = 0; e < 16; ++e) f[rb][e] = 0.f;

  // The min term, one super-block late. Quarter waves share their rows and form the half-sum operand
  // themselves, and apply U just as late, so their per-element arithmetic is that of the full tiles.
  float u_dmin = 0.f;      // dmin of the super-block whose U is pending
  v8h u_b = {}, u_a = {};  // its m_j operand and (quarters) its half-sum operand
  auto u_step = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const v8h a = QTR ? u_a : __builtin_bit_cast(v8h, xh_l[slot][rbw + rb][lane]);
      const v16f_t u = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, u_b, v16f_t{}, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 16; ++e) f[rb][e] -= u_dmin * u[e];
    }
  };
  // the half-sums this wave forms: row block urb, sub-blocks ju0 .. ju0 + JN - 1
  constexpr int JN = QTR ? 8 : 4;
  const int urb = QTR ? rb0 : (wave & 3);
  const int ju0 = QTR ? 0 : 4 * (wave >> 2);
  const int urow = 32 * urb + l32;

  // Step j + 1's A reads and B operands are formed while step j's MFMAs run (one scheduling region
  // per step). slot: the LDS slot this super-block's half-sums go to (full tiles); -2 for the first
  // super-block (no U pending yet, slot 0).
  auto compute = [&](const int8_t* xt, const uint8_t* wt, int slot) __attribute__((always_inline)) {
    const uint8_t* wr = wt + (32 * cg + l32) * BB;
    const uint4 hd = *reinterpret_cast<const uint4*>(wr);
    const float d = h2f(hd.x & 0xFFFFu), dmin = h2f(hd.x >> 16);
    const ScMin sm = unpack_scmin(hd.y, hd.z, hd.w);
    uint32_t qh[4] = {0, 0, 0, 0};
    if constexpr (FMT == 5) {  // the 5th bits of elements 16 h .. 16 h + 15
      const uint4 qhv = *reinterpret_cast<const uint4*>(wr + 16 + 16 * h);
      qh[0] = qhv.x; qh[1] = qhv.y; qh[2] = qhv.z; qh[3] = qhv.w;
    }
    uint32_t qw[4][4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint4 qv = *reinterpret_cast<const uint4*>(wr + QS + 32 * g + 16 * h);
      qw[g][0] = qv.x; qw[g][1] = qv.y; qw[g][2] = qv.z; qw[g][3] = qv.w;
    }
    float hsum[8];
    v4i A[2][RB], bl[2], bh[2], bb[2];
    auto read_a = [&](int j, int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int row = 32 * (rbw + rb) + l32;
        A[buf][rb] = *reinterpret_cast<const v4i*>(xt + row * 256 + 16 * ((2 * j + h) ^ (row & 15)));
      }
    };
    // half-sum of sub-block ju0 + jj (jj < JN) of this lane's row urow, half h
    auto xsum_half = [&](int jj) __attribute__((always_inline)) {
      const int j = ju0 + jj;
      const v4i xv = QTR ? A[jj & 1][0]
                         : *reinterpret_cast<const v4i*>(xt + urow * 256 + 16 * ((2 * j + h) ^ (urow & 15)));
      int sacc = __builtin_amdgcn_sdot4(xv[0], 0x01010101, 0, false);
      sacc = __builtin_amdgcn_sdot4(xv[1], 0x01010101, sacc, false);
      sacc = __builtin_amdgcn_sdot4(xv[2], 0x01010101, sacc, false);
      sacc = __builtin_amdgcn_sdot4(xv[3], 0x01010101, sacc, false);
      hsum[jj] = (float)sacc;
    };
    auto build = [&](int j, int buf) __attribute__((always_inline)) {
      const uint32_t scw = j < 4 ? sm.sc_lo : sm.sc_hi;
      const uint32_t sc = (scw >> (8 * (j & 3))) & 0xFF;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t nib = (qw[j >> 1][e] >> (4 * (j & 1))) & 0x0F0F0F0Fu;
        bl[buf][e] = (int)mul_bytes(nib, sc & 7);  // <= 15 * 7 per byte
        bh[buf][e] = (int)mul_bytes(nib, sc >> 3);
        if constexpr (FMT == 5) bb[buf][e] = (int)mul_bytes((qh[e] >> j) & 0x01010101u, 2 * sc);  // <= 126
      }
    };
    v16i_t tl[RB], th[RB];
    read_a(0, 0);
    build(0, 0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = j & 1;
      __builtin_amdgcn_sched_barrier(0);
      if (j < 7) read_a(j + 1, c ^ 1);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        tl[rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[c][rb], bl[c], j == 0 ? v16i_t{} : tl[rb], 0, 0, 0);
        th[rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[c][rb], bh[c], j == 0 ? v16i_t{} : th[rb], 0, 0, 0);
        if constexpr (FMT == 5)
          th[rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[c][rb], bb[c], th[rb], 0, 0, 0);
      }
      // a quarter wave sums step j's own A operand; a full tile's sub-blocks are spread over the steps
      if constexpr (JN == 8) xsum_half(j);
      else if (j & 1) xsum_half(j >> 1);
      if (j < 7) build(j + 1, c ^ 1);
      __builtin_amdgcn_sched_group_barrier(0x100, RB + (QTR ? 0 : 1), 0);  // the LDS reads first
#pragma unroll
      for (int k = 0; k < (FMT == 4 ? 2 : 3) * RB; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);  // VALU
      }
    }
    v8h ub;
#pragma unroll
    for (int jj = 0; jj < 8; ++jj)
      ub[jj] = (_Float16)(float)(((jj < 4 ? sm.mn_lo : sm.mn_hi) >> (8 * (jj & 3))) & 0xFF);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int e = 0; e < 16; ++e) f[rb][e] += d * (float)(tl[rb][e] + 8 * th[rb][e]);
    // the previous super-block's U (in a full tile its operands were published before the barrier
    // this compute follows), then this one's goes pending
    if (slot >= 0) u_step(slot ^ 1);
    if constexpr (QTR) {
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) u_a[jj] = (_Float16)hsum[jj];
    } else {
      v4h ua;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) ua[jj] = (_Float16)hsum[jj];
      reinterpret_cast<uint2*>(&xh_l[slot & 1][urb][lane])[ju0 >> 2] = __builtin_bit_cast(uint2, ua);
    }
    u_dmin = dmin;
    u_b = ub;
  };

  load(0, xs0, ws0);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  int sb = 0;
  for (; sb + 1 < nsb; sb += 2) {
    load(sb + 1, xs1, ws1);
    compute(xs0, ws0, sb == 0 ? -2 : 0);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    if (sb + 2 < nsb) load(sb + 2, xs0, ws0);
    compute(xs1, ws1, 1);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
  }
  if (sb < nsb) {
    compute(xs0, ws0, sb == 0 ? -2 : 0);
    if constexpr (!QTR) __syncthreads();
  }
  u_step((nsb - 1) & 1);  // the last super-block's U

  const int n = n0 + 32 * cg + l32;
  // the row scales first, unconditionally (clamped rows): one wait, not one per element
  float xsv[RB][16];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int e = 0; e < 16; ++e)
      xsv[rb][e] = x_scale[min(m0 + 32 * (rbw + rb) + 8 * (e >> 2) + 4 * h + (e & 3), M - 1)];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int m = m0 + 32 * (rbw + rb) + 8 * (e >> 2) + 4 * h + (e & 3);
      if (m < M && n < N) st_out<OUT_DT>(out, (int64_t)m * N + n, f[rb][e] * xsv[rb][e]);
    }
}

}  // namespace

void launch_q45_tile_i8(int fmt, const TailPlan& p, const int8_t* x, const float* xs, const uint8_t* w,
                        void* out, int odt, int M, int N, int K, hipStream_t st) {
  const int xm = xcd_rows(p.nt_x, M, TBM);
  auto go = [&](auto f, auto dt) {
    constexpr int F = decltype(f)::value, DT = decltype(dt)::value;
    gemm_kq_tile_i8_kernel<F, DT, false><<<(unsigned)p.whole, 512, 0, st>>>(x, xs, w, out, M, N, K, p.nt_x, xm, 0);
    if (p.cut)
      gemm_kq_tile_i8_kernel<F, DT, true><<<(unsigned)(4 * p.cut), 256, 0, st>>>(x, xs, w, out, M, N, K, p.nt_x,
                                                                                xm, (int)p.whole);
  };
  auto by_dt = [&](auto f) {
    if (odt == SL8_DTYPE_F16) go(f, std::integral_constant<int, SL8_DTYPE_F16>{});
    else if (odt == SL8_DTYPE_BF16) go(f, std::integral_constant<int, SL8_DTYPE_BF16>{});
    else go(f, std::integral_constant<int, SL8_DTYPE_F32>{});
  };
  if (fmt == 4) by_dt(std::integral_constant<int, 4>{});
  else by_dt(std::integral_constant<int, 5>{});
}

}  // namespace sl8
