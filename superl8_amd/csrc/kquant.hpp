// Shared pieces of the GGUF k-quant kernels (Q4_K, Q5_K, Q6_K).
#pragma once

#include <type_traits>

#include "common.hpp"

#ifndef SL8_KQ_XCD
#define SL8_KQ_XCD 1
#endif

namespace sl8 {

// Packed 6-bit sub-scales / mins of a Q4_K / Q5_K super-block (4 per dword,
// byte j % 4), unpacked from the 12-byte get_scale_min_k4 layout.
struct ScMin {
  uint32_t sc_lo, sc_hi, mn_lo, mn_hi;
};
__device__ __forceinline__ ScMin unpack_scmin(uint32_t s0, uint32_t s1, uint32_t s2) {
  ScMin r;
  r.sc_lo = s0 & 0x3F3F3F3Fu;
  r.mn_lo = s1 & 0x3F3F3F3Fu;
  r.sc_hi = (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
  r.mn_hi = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
  return r;
}
// Tile order o -> (column tile ct, row tile rt) of the k-quant tile GEMMs.
// xcd_m > 0 (the number of row tiles; used when the column-tile count is a
// multiple of 8): workgroup o runs on XCD o % 8, and the xcd_m row tiles of
// one weight column tile are consecutive workgroups of the same XCD, so the
// column's weights come from HBM into that XCD's L2 once and are re-read
// from there by the other row tiles running beside it. xcd_m = 0: row-major.
__device__ __forceinline__ void kq_tile_coords(int o, int nt_x, int xcd_m, int& ct, int& rt) {
  if (xcd_m > 0) {
    const int k = o >> 3;
    ct = (o & 7) + 8 * (k / xcd_m);
    rt = k % xcd_m;
  } else {
    ct = o % nt_x;
    rt = o / nt_x;
  }
}
__device__ __forceinline__ int byte_of(uint32_t w, int i) { return (w >> (8 * i)) & 0xFF; }

// Four byte lanes times one small factor, for products that stay below 256
// per byte (no carries between bytes): one packed 16-bit multiply
// (v_pk_mul_lo_u16, full rate) instead of a 32-bit integer multiply (quarter
// rate); each 16-bit half holds two bytes and its product stays below 2^16.
__device__ __forceinline__ uint32_t mul_bytes(uint32_t bytes, uint32_t f) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  const u16x2 a = __builtin_bit_cast(u16x2, bytes);
  const u16x2 b = {(unsigned short)f, (unsigned short)f};
  return __builtin_bit_cast(uint32_t, a * b);
}

// Q5_K decode GEMV for M <= 2 on the Q4_K M <= 2 kernel (gemm_q4k.hip)
void launch_gemv_q5k_small(const int8_t* x, const float* xs, const uint8_t* w, void* out, int odt,
                           int M, int N, int K, hipStream_t st);
// Q5_K decode GEMV for 3 <= M <= 16 on the int8 MFMA (gemm_q4k.hip)
void launch_gemv_q5k_mfma(const int8_t* x, const float* xs, const uint8_t* w, void* out, int odt,
                          int M, int N, int K, hipStream_t st);

// XCD-aware tile order (see kq_tile_coords) when the column tiles split evenly over the 8 XCDs
inline int xcd_rows(int nt_x, int M, int bm) { return SL8_KQ_XCD && nt_x % 8 == 0 ? (M + bm - 1) / bm : 0; }

// Tiled GEMMs (M > 16): a tile shape with the workgroups of it a CU holds and the time one
// super-block of one takes then, and the plan of a call: tiles [0, nfull) whole, nsplit more
// tiles split S ways over K into part_bytes of fp32 partials.
struct TileShape {
  int bm, bn, wgs_per_cu;
  double us_per_sb;
};
struct TilePlan {
  int shape, nt_x, S;
  int64_t nfull, nsplit;
  size_t part_bytes;
  double us;  // the model's time
};
TilePlan plan_tiles(int M, int N, int K, const TileShape* shapes, int count, bool may_split);

// Without scratch, 128 x 128 tiles whose last round, where it would hold at most half the CUs, runs
// as 4 row quarters each in a second launch: tiles [0, whole), then `cut` more.
struct TailPlan {
  int nt_x;
  int64_t whole, cut;
  double us;
};
TailPlan plan_tail(int M, int N, int K, const TileShape& tile, const TileShape& quarter);

// Which part of the problem a workgroup computes: workgroups below nfull a whole tile, the others
// a K range of tiles nfull .., S per tile, into part[tile - nfull][split][BM][BN]. quarter0 >= 0:
// workgroup o computes row quarter o & 3 (the kernel's BM rows) of tile quarter0 + o / 4.
struct TileWork {
  int nt_x, xcd_m, nfull, S, tile_elems;
  float* part;
  int quarter0;
};
inline TileWork tile_work(const TilePlan& p, const TileShape& s, int M, float* part) {
  return TileWork{p.nt_x, xcd_rows(p.nt_x, M, s.bm), (int)p.nfull, p.S, s.bm * s.bn, part, -1};
}
struct TileRange {
  int ct, rt, sb0, sb1, sp;
  float* part;  // the tile's S partials, null for a whole tile
};
__device__ __forceinline__ TileRange tile_range(const TileWork& tw, int nsb) {
  TileRange r{0, 0, 0, nsb, 0, nullptr};
  int tile = blockIdx.x;
  if (tw.quarter0 >= 0) {
    kq_tile_coords(tw.quarter0 + (tile >> 2), tw.nt_x, tw.xcd_m, r.ct, r.rt);
    r.rt = 4 * r.rt + (tile & 3);
    return r;
  }
  if (tile >= tw.nfull) {
    const int i = tile - tw.nfull, t = i / tw.S;
    tile = tw.nfull + t;
    r.sp = i % tw.S;
    r.sb0 = r.sp * nsb / tw.S;
    r.sb1 = (r.sp + 1) * nsb / tw.S;
    r.part = tw.part + (int64_t)t * tw.S * tw.tile_elems;
  }
  kq_tile_coords(tile, tw.nt_x, tw.xcd_m, r.ct, r.rt);
  return r;
}
void launch_kq_reduce(const TilePlan& p, const TileShape& s, const TileWork& tw, const float* xs,
                      void* out, int odt, int M, int N, hipStream_t st);
// Q6_K (gemm_kq56.hip). part: the partials of a split plan; null: a plan without (plan_q6_whole)
TilePlan plan_q6_tile(int M, int N, int K);
void launch_q6_tile(const int8_t* x, const float* xs, const uint8_t* w, void* out, int odt, int M,
                    int N, int K, float* part, hipStream_t st);
// the plan without scratch: 128-row tiles with a cut last round (whole > 0), or one tile shape
TailPlan plan_q6_whole(int M, int N, int K, TilePlan& tiles);
// Q4_K / Q5_K (gemm_kq_tile.hip): x int8 codes with their row scales xs (x_dtype SL8_KQ_I8), or
// fp16 / bf16 rows that are quantised in the call (with a workspace only; 16-byte aligned).
// workspace: q45_tile_workspace() bytes, or null.
constexpr int SL8_KQ_I8 = 3;
size_t q45_tile_workspace(int fmt, int M, int N, int K);
TilePlan plan_q45_tile(int fmt, int M, int N, int K);
TailPlan plan_q45_whole(int fmt, int M, int N, int K, TilePlan& tiles);  // as plan_q6_whole
void launch_q45_tile(int fmt, const void* x, int x_dtype, const float* xs, const uint8_t* w, void* out,
                     int odt, int M, int N, int K, void* workspace, hipStream_t st);
// gemm_kq_tile_i8.hip: 128-row tiles on the int8 codes
void launch_q45_tile_i8(int fmt, const TailPlan& p, const int8_t* x, const float* xs, const uint8_t* w,
                        void* out, int odt, int M, int N, int K, hipStream_t st);

typedef __attribute__((address_space(1))) const void* kq_gptr_t;
typedef __attribute__((address_space(3))) void* kq_lptr_t;

}  // namespace sl8
