// Per-row symmetric int8 quantisation and K-smoothing for gfx950.
//
// Numerics contract (reference csrc/include/quant_rowwise.cuh:33-91 and
// superl8/quant/core.py:47-62,70-95):
//   scale = amax|row| * fp32(1/127)   (reciprocal multiply, not division)
//   safe  = scale == 0 ? 1 : scale
//   q     = clamp(rint(x / safe), -127, 127)   with IEEE round-to-nearest
//           division and round-half-to-even.
// K-smoothing subtracts the fp32 per-channel key mean and rounds back to the
// storage dtype before quantising, exactly as torch.sub(k, mean, out=k_s).
//
// Layout: one row is handled by LPR lanes of a wave64 (LPR in {16,32,64});
// 256-thread blocks hold 256/LPR rows. Rows are read twice (amax pass, code
// pass); the second read is served by L2 for the row sizes used here.

#include "common.hpp"
#include "rowquant.hpp"

#include <cmath>
#include <type_traits>
#include <string>

namespace sl8 {

static thread_local std::string g_last_error;

void set_error(const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
}
void clear_error() { g_last_error.clear(); }

namespace {

constexpr int QTHREADS = 256;

// Value of element d of a row after the optional mean shift.
template <int DT, bool MEAN>
__device__ __forceinline__ float row_val(const typename Elem<DT>::T* xr, const float* mr, int d) {
  float v = Elem<DT>::ld(xr, d);
  if constexpr (MEAN) v = Elem<DT>::round(v - mr[d]);
  return v;
}

// rows = G*N; row r uses mean row r / rows_per_mean.
template <int DT, int LPR, bool MEAN>
__global__ void __launch_bounds__(QTHREADS)
quant_rows_kernel(const typename Elem<DT>::T* __restrict__ x, const float* __restrict__ mean,
                  int8_t* __restrict__ q, float* __restrict__ scale, int64_t rows,
                  int64_t rows_per_mean, int K, float scale_mul) {
  using T = typename Elem<DT>::T;
  const int lane = threadIdx.x % LPR;
  const int64_t row = (int64_t)blockIdx.x * (QTHREADS / LPR) + threadIdx.x / LPR;
  const bool live = row < rows;
  const int64_t r = live ? row : 0;
  const T* xr = x + r * K;
  const float* mr = MEAN ? mean + (r / rows_per_mean) * K : nullptr;

  float amax = 0.f;
  if (live) {
    for (int d = lane; d < K; d += LPR) amax = fmaxf(amax, fabsf(row_val<DT, MEAN>(xr, mr, d)));
  }
  amax = lane_group_max<LPR>(amax);
  if (!live) return;

  const float s = amax * (1.0f / 127.0f);
  const float safe = (s == 0.f) ? 1.f : s;
  if (lane == 0) scale[row] = safe * scale_mul;

  int8_t* qr = q + r * K;
  if ((K & 3) == 0) {
    // 4 codes per 32-bit store.
    for (int d = lane * 4; d < K; d += LPR * 4) {
      uint32_t packed = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        packed |= (uint32_t)(uint8_t)code_of(row_val<DT, MEAN>(xr, mr, d + e), safe) << (8 * e);
      *reinterpret_cast<uint32_t*>(qr + d) = packed;
    }
  } else {
    for (int d = lane; d < K; d += LPR) qr[d] = code_of(row_val<DT, MEAN>(xr, mr, d), safe);
  }
}


// Vectorised variant: LPR lanes per row (LPR = BT: one workgroup per row),
// each lane holding NV 16-byte vectors of the row in registers for both the
// amax and the code pass (one HBM read per element). Needs K a multiple of
// the elements per 16 bytes (EPV) and a 16-byte aligned base.
template <int DT, int BT, int LPR, int NV, bool MEAN>
__global__ void __launch_bounds__(BT)
quant_rows_vec_kernel(const typename Elem<DT>::T* __restrict__ x, const float* __restrict__ mean,
                      int8_t* __restrict__ q, float* __restrict__ scale, int64_t rows,
                      int64_t rows_per_mean, int K, float scale_mul) {
  using T = typename Elem<DT>::T;
  constexpr int EPV = VecIO<DT>::EPV;
  static_assert(LPR <= 64 || LPR == BT, "a row is a lane group or the whole workgroup");
  const int lane = threadIdx.x % LPR;
  const int64_t row = (int64_t)blockIdx.x * (BT / LPR) + threadIdx.x / LPR;
  const bool live = row < rows;
  const int64_t r = live ? row : 0;
  const T* xr = x + r * K;
  const float* mr = MEAN ? mean + (r / rows_per_mean) * K : nullptr;
  const int nvec = K / EPV;

  uint4 raw[NV];  // every load of the thread's row part is in flight before any is used
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int vi = v * LPR + lane;
    raw[v] = make_uint4(0, 0, 0, 0);
    if (live && vi < nvec) raw[v] = reinterpret_cast<const uint4*>(xr)[vi];
  }
  float f[NV][EPV];
  float amax = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    VecIO<DT>::unpack(raw[v], f[v]);
    if constexpr (MEAN) {
      const int vi = v * LPR + lane;
      const bool ok = live && vi < nvec;
#pragma unroll
      for (int e = 0; e < EPV; ++e)
        f[v][e] = ok ? Elem<DT>::round(f[v][e] - mr[vi * EPV + e]) : 0.f;
    }
#pragma unroll
    for (int e = 0; e < EPV; ++e) amax = fmaxf(amax, fabsf(f[v][e]));
  }
  if constexpr (LPR <= 64) {
    amax = lane_group_max<LPR>(amax);
  } else {
    __shared__ float red[BT / 64];
    amax = lane_group_max<64>(amax);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < BT / 64; ++w) amax = fmaxf(amax, red[w]);
  }
  if (!live) return;
  const float s = amax * (1.0f / 127.0f);
  const float safe = (s == 0.f) ? 1.f : s;
  if (lane == 0) scale[row] = safe * scale_mul;
  int8_t* qr = q + r * K;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int vi = v * LPR + lane;
    if (vi < nvec) {
      if constexpr (EPV == 8) {
        *reinterpret_cast<uint2*>(qr + vi * EPV) = row_codes8<DT>(f[v], safe);
      } else {
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) w |= (uint32_t)(uint8_t)code_of(f[v][e], safe) << (8 * e);
        *reinterpret_cast<uint32_t*>(qr + vi * EPV) = w;
      }
    }
  }
}

template <int DT, bool MEAN>
int launch_quant(const void* x, const float* mean, int8_t* q, float* scale, int64_t rows,
                 int64_t rows_per_mean, int64_t K, float scale_mul, hipStream_t st) {
  using T = typename Elem<DT>::T;
  const T* xp = static_cast<const T*>(x);
  auto go = [&](auto lpr_tag) {
    constexpr int LPR = decltype(lpr_tag)::value;
    const int64_t rpb = QTHREADS / LPR;
    const dim3 grid((unsigned)((rows + rpb - 1) / rpb));
    quant_rows_kernel<DT, LPR, MEAN><<<grid, QTHREADS, 0, st>>>(xp, mean, q, scale, rows,
                                                                rows_per_mean, (int)K, scale_mul);
  };
  constexpr int EPV = VecIO<DT>::EPV;
  constexpr int LT = 1024;  // threads of a long row's workgroup
  if (K % EPV == 0 && aligned(x, 16) && aligned(q, EPV) && K / EPV <= 8 * LT) {
    const int64_t nvec = K / EPV;
    auto gv = [&](auto bt_tag, auto lpr_tag, auto nv_tag) {
      constexpr int BT = decltype(bt_tag)::value, LPR = decltype(lpr_tag)::value,
                    NV = decltype(nv_tag)::value;
      const int64_t rpb = BT / LPR;
      const dim3 grid((unsigned)((rows + rpb - 1) / rpb));
      quant_rows_vec_kernel<DT, BT, LPR, NV, MEAN><<<grid, BT, 0, st>>>(
          xp, mean, q, scale, rows, rows_per_mean, (int)K, scale_mul);
    };
    using B = std::integral_constant<int, QTHREADS>;
    using L = std::integral_constant<int, LT>;
    using N1 = std::integral_constant<int, 1>;
    using N2 = std::integral_constant<int, 2>;
    using N4 = std::integral_constant<int, 4>;
    using N5 = std::integral_constant<int, 5>;
    using N8 = std::integral_constant<int, 8>;
    if (nvec <= 16) gv(B{}, std::integral_constant<int, 16>{}, N1{});
    else if (nvec <= 32) gv(B{}, std::integral_constant<int, 32>{}, N1{});
    else if (nvec <= 64) gv(B{}, std::integral_constant<int, 64>{}, N1{});
    else if (nvec <= 128) gv(B{}, std::integral_constant<int, 64>{}, N2{});
    else if (nvec <= 256) gv(B{}, B{}, N1{});
    else if (nvec <= 512) gv(B{}, B{}, N2{});
    // longer rows: 1024 threads, so the few rows of a decode batch (one CU each) have 16 waves
    // of loads in flight. 8 bf16 rows of 17408 (past the 16384 that 256 threads of 8 vectors
    // held): 92.0 us in the element-wise kernel below, about 4 us here. Rows that two workgroups a
    // CU do not hold at once and that would leave many of 1024 threads idle take 256 threads of 4
    // or 5 vectors: 8192 rows of 5120, fp16 22 us against 44, bf16 22 / 40 (2048 rows: 8 / 13)
    else if (nvec <= 1024 && rows > 2 * (int64_t)cu_count()) gv(B{}, B{}, N4{});
    else if (nvec <= 1280 && rows > 2 * (int64_t)cu_count()) gv(B{}, B{}, N5{});
    else if (nvec <= 1024) gv(L{}, L{}, N1{});
    else if (nvec <= 2048) gv(L{}, L{}, N2{});
    else if (nvec <= 4096) gv(L{}, L{}, N4{});
    else gv(L{}, L{}, N8{});
  } else if (K <= 128) {
    go(std::integral_constant<int, 16>{});
  } else if (K <= 512) {
    go(std::integral_constant<int, 32>{});
  } else {
    go(std::integral_constant<int, 64>{});
  }
  SL8_CHECK_LAUNCH("quantize_i8_rowwise");
  return SL8_OK;
}

int dispatch_quant(const void* x, int dt, const float* mean, int8_t* q, float* scale,
                   int64_t rows, int64_t rows_per_mean, int64_t K, float scale_mul,
                   hipStream_t st) {
  if (mean) {
    switch (dt) {
      case SL8_DTYPE_F16: return launch_quant<SL8_DTYPE_F16, true>(x, mean, q, scale, rows, rows_per_mean, K, scale_mul, st);
      case SL8_DTYPE_BF16: return launch_quant<SL8_DTYPE_BF16, true>(x, mean, q, scale, rows, rows_per_mean, K, scale_mul, st);
      default: return launch_quant<SL8_DTYPE_F32, true>(x, mean, q, scale, rows, rows_per_mean, K, scale_mul, st);
    }
  }
  switch (dt) {
    case SL8_DTYPE_F16: return launch_quant<SL8_DTYPE_F16, false>(x, nullptr, q, scale, rows, 1, K, scale_mul, st);
    case SL8_DTYPE_BF16: return launch_quant<SL8_DTYPE_BF16, false>(x, nullptr, q, scale, rows, 1, K, scale_mul, st);
    default: return launch_quant<SL8_DTYPE_F32, false>(x, nullptr, q, scale, rows, 1, K, scale_mul, st);
  }
}

// ---- K mean -------------------------------------------------------------
// fp16: every value is an integer multiple of 2^-24 below 2^16 in magnitude,
// so sum(x * 2^24) is an exact int64 for N < 2^23 rows: the mean does not
// depend on summation order. Blocks take (64 columns, a chunk of rows); a
// block's exact partial sum is added to the int64 workspace with an integer
// atomic (exact, so still order free), and a last pass scales it.
constexpr int MEAN_COLS = 64;
constexpr int MEAN_PHASES = 16;
constexpr int MEAN_CHUNK = 256;  // rows per block

__global__ void __launch_bounds__(256) i64_zero_kernel(unsigned long long* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

__global__ void __launch_bounds__(MEAN_COLS * MEAN_PHASES)
k_mean_f16_kernel(const uint16_t* __restrict__ k, unsigned long long* __restrict__ acc, int64_t N,
                  int D) {
  __shared__ long long part[MEAN_PHASES][MEAN_COLS];
  const int col = threadIdx.x % MEAN_COLS;
  const int ph = threadIdx.x / MEAN_COLS;
  const int64_t g = blockIdx.y;
  const int d = blockIdx.x * MEAN_COLS + col;
  const int64_t n0 = (int64_t)blockIdx.z * MEAN_CHUNK;
  const int64_t n1 = min(N, n0 + MEAN_CHUNK);
  long long a = 0;
  if (d < D) {
    const uint16_t* kg = k + g * N * D + d;
#pragma unroll 4
    for (int64_t n = n0 + ph; n < n1; n += MEAN_PHASES)
      a += (long long)ldexpf(h2f(kg[n * D]), 24);  // exact: |v| * 2^24 < 2^40, integral
  }
  part[ph][col] = a;
  __syncthreads();
  if (ph == 0 && d < D) {
    long long t = 0;
#pragma unroll
    for (int p = 0; p < MEAN_PHASES; ++p) t += part[p][col];
    atomicAdd(acc + g * D + d, (unsigned long long)t);  // two's complement: exact mod 2^64
  }
}

__global__ void __launch_bounds__(256)
k_mean_finish_kernel(const unsigned long long* __restrict__ acc, float* __restrict__ mean,
                     int64_t n, int64_t N) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) mean[i] = (float)(((double)(long long)acc[i] * 0x1p-24) / (double)N);
}

// bf16 / f32: fp64 sums in a fixed order (the rows of a phase, then the phases). One block per
// (group, COLS columns) with PHASES row phases: one thread per column over all N rows in turn took
// 1439 us for 8 groups of 6121 bf16 rows of 128.
template <int DT, int COLS, int PHASES>
__global__ void __launch_bounds__(COLS * PHASES)
k_mean_seq_kernel(const typename Elem<DT>::T* __restrict__ k, float* __restrict__ mean,
                  int64_t N, int D) {
  __shared__ double part[PHASES][COLS];
  const int64_t g = blockIdx.y;
  const int col = threadIdx.x % COLS, ph = threadIdx.x / COLS;
  const int d = blockIdx.x * COLS + col;
  double s = 0.0;
  if (d < D) {
    const typename Elem<DT>::T* kg = k + g * N * D + d;
#pragma unroll 8
    for (int64_t n = ph; n < N; n += PHASES) s += (double)Elem<DT>::ld(kg, n * D);
  }
  part[ph][col] = s;
  __syncthreads();
  if (ph == 0 && d < D) {
    double t = 0.0;
#pragma unroll 8
    for (int p = 0; p < PHASES; ++p) t += part[p][col];
    mean[g * D + d] = (float)(t / (double)N);
  }
}
// 64 phases of 16 columns where the groups are few, 4 of 64 where they fill the chip (or the rows
// would not fill the phases): 4096 groups of 16 rows of 64, bf16 40 us against 11
template <int DT>
void launch_k_mean_seq(const void* k, float* mean, int64_t G, int64_t N, int64_t D, hipStream_t st) {
  auto go = [&](auto cols, auto phases) {
    constexpr int C = decltype(cols)::value, P = decltype(phases)::value;
    k_mean_seq_kernel<DT, C, P><<<dim3((unsigned)((D + C - 1) / C), (unsigned)G), C * P, 0, st>>>(
        static_cast<const typename Elem<DT>::T*>(k), mean, N, (int)D);
  };
  using std::integral_constant;
  if (N <= 64 || G * ((D + 63) / 64) >= 2 * (int64_t)cu_count())
    go(integral_constant<int, 64>{}, integral_constant<int, 4>{});
  else
    go(integral_constant<int, 16>{}, integral_constant<int, 64>{});
}

// ---- per-channel (column) quantisation over the key axis ----------------
// scale[g,d] = amax_n |x[g,n,d]| * fp32(1/127) (1 if 0); max is order-free.
// Blocks take (64 columns, a chunk of rows) and fold their max into the
// scale buffer with an integer atomic max on the (non-negative) float bits;
// a last pass turns the maxima into scales.
template <int DT>
__global__ void __launch_bounds__(MEAN_COLS * MEAN_PHASES)
col_amax_kernel(const typename Elem<DT>::T* __restrict__ x, unsigned int* __restrict__ amax_bits,
                int64_t N, int D) {
  __shared__ float part[MEAN_PHASES][MEAN_COLS];
  const int col = threadIdx.x % MEAN_COLS, ph = threadIdx.x / MEAN_COLS;
  const int64_t g = blockIdx.y;
  const int d = blockIdx.x * MEAN_COLS + col;
  const int64_t n0 = (int64_t)blockIdx.z * MEAN_CHUNK;
  const int64_t n1 = min(N, n0 + MEAN_CHUNK);
  float m = 0.f;
  if (d < D) {
    const typename Elem<DT>::T* xg = x + g * N * D + d;
#pragma unroll 4
    for (int64_t n = n0 + ph; n < n1; n += MEAN_PHASES) m = fmaxf(m, fabsf(Elem<DT>::ld(xg, n * D)));
  }
  part[ph][col] = m;
  __syncthreads();
  if (ph == 0 && d < D) {
#pragma unroll
    for (int p = 1; p < MEAN_PHASES; ++p) m = fmaxf(m, part[p][col]);
    atomicMax(amax_bits + g * D + d, __float_as_uint(m));
  }
}

__global__ void __launch_bounds__(256) col_scale_kernel(float* __restrict__ scale, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float s = scale[i] * (1.0f / 127.0f);  // scale holds the column max here
  scale[i] = (s == 0.f) ? 1.f : s;
}

__global__ void __launch_bounds__(256) u32_zero_kernel(unsigned int* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

template <int DT>
__global__ void __launch_bounds__(256)
col_quant_kernel(const typename Elem<DT>::T* __restrict__ x, const float* __restrict__ scale,
                 int8_t* __restrict__ q, int64_t N, int D, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int d = (int)(i % D);
  const int64_t g = i / ((int64_t)N * D);
  q[i] = code_of(Elem<DT>::ld(x, i), scale[g * D + d]);
}

}  // namespace
}  // namespace sl8

using namespace sl8;

extern "C" int sl8_quantize_i8_cols(const void* x, int dtype, int64_t G, int64_t N, int64_t D,
                                    int8_t* q, float* scale, void* stream) {
  clear_error();
  SL8_CHECK_ARG(dtype == SL8_DTYPE_F16 || dtype == SL8_DTYPE_BF16 || dtype == SL8_DTYPE_F32,
                "quantize_v_perchannel: input must be float16/bfloat16/float32");
  SL8_CHECK_ARG(G >= 0 && N >= 0 && D >= 0 && D < (1LL << 31), "quantize_v_perchannel: bad shape");
  if (G == 0 || D == 0) return SL8_OK;
  SL8_CHECK_ARG(x && q && scale, "quantize_v_perchannel: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t nsc = G * D;
  const dim3 grid((unsigned)((D + MEAN_COLS - 1) / MEAN_COLS), (unsigned)G,
                  (unsigned)((N + MEAN_CHUNK - 1) / MEAN_CHUNK));
  const int64_t total = G * N * D;
  const unsigned qgrid = (unsigned)((total + 255) / 256);
  const unsigned sgrid = (unsigned)((nsc + 255) / 256);
  unsigned int* bits = reinterpret_cast<unsigned int*>(scale);
  u32_zero_kernel<<<sgrid, 256, 0, st>>>(bits, nsc);
  switch (dtype) {
    case SL8_DTYPE_F16:
      if (N) col_amax_kernel<SL8_DTYPE_F16><<<grid, MEAN_COLS * MEAN_PHASES, 0, st>>>(
          static_cast<const uint16_t*>(x), bits, N, (int)D);
      col_scale_kernel<<<sgrid, 256, 0, st>>>(scale, nsc);
      if (total) col_quant_kernel<SL8_DTYPE_F16><<<qgrid, 256, 0, st>>>(
          static_cast<const uint16_t*>(x), scale, q, N, (int)D, total);
      break;
    case SL8_DTYPE_BF16:
      if (N) col_amax_kernel<SL8_DTYPE_BF16><<<grid, MEAN_COLS * MEAN_PHASES, 0, st>>>(
          static_cast<const uint16_t*>(x), bits, N, (int)D);
      col_scale_kernel<<<sgrid, 256, 0, st>>>(scale, nsc);
      if (total) col_quant_kernel<SL8_DTYPE_BF16><<<qgrid, 256, 0, st>>>(
          static_cast<const uint16_t*>(x), scale, q, N, (int)D, total);
      break;
    default:
      if (N) col_amax_kernel<SL8_DTYPE_F32><<<grid, MEAN_COLS * MEAN_PHASES, 0, st>>>(
          static_cast<const float*>(x), bits, N, (int)D);
      col_scale_kernel<<<sgrid, 256, 0, st>>>(scale, nsc);
      if (total) col_quant_kernel<SL8_DTYPE_F32><<<qgrid, 256, 0, st>>>(
          static_cast<const float*>(x), scale, q, N, (int)D, total);
      break;
  }
  SL8_CHECK_LAUNCH("quantize_v_perchannel");
  return SL8_OK;
}

extern "C" const char* sl8_last_error(void) { return g_last_error.c_str(); }
extern "C" const char* sl8_version(void) { return "superl8-hip 0.1 gfx950"; }

extern "C" int sl8_quantize_i8_rowwise(const void* x, int x_dtype, int64_t M, int64_t K,
                                       int8_t* q, float* scale, void* stream) {
  clear_error();
  SL8_CHECK_ARG(x_dtype == SL8_DTYPE_F16 || x_dtype == SL8_DTYPE_BF16 || x_dtype == SL8_DTYPE_F32,
                "quantize_i8_rowwise input must be float16/bfloat16/float32");
  SL8_CHECK_ARG(M >= 0 && K >= 0 && K < (1LL << 31), "quantize_i8_rowwise: bad shape [%lld,%lld]",
                (long long)M, (long long)K);
  if (M == 0 || K == 0) return SL8_OK;
  SL8_CHECK_ARG(x && q && scale, "quantize_i8_rowwise: null pointer");
  SL8_CHECK_ARG((K & 3) != 0 || aligned(q, 4), "quantize_i8_rowwise: q must be 4-byte aligned");
  return dispatch_quant(x, x_dtype, nullptr, q, scale, M, 1, K, 1.0f,
                        static_cast<hipStream_t>(stream));
}

namespace sl8 {
namespace {

// ---------------------------------------------------------------------------
// Row-group quantisation (one scale per R consecutive rows of a [G][N][K]
// tensor, groups restarting at every G slice): the per-wavefront Q / per-tile
// K scheme. One workgroup per group: pass 1 takes the
// amax of the (optionally mean-shifted, dtype-rounded) values over the R x K
// block, pass 2 writes the codes (the block is re-read from L2). The scale,
// safe value and code follow the row-wise contract above with the group's
// amax in place of the row's; every row of the group stores the group scale.
// ---------------------------------------------------------------------------
template <int DT, bool MEAN>
__global__ void __launch_bounds__(QTHREADS)
quant_row_groups_kernel(const typename Elem<DT>::T* __restrict__ x, const float* __restrict__ mean,
                        int8_t* __restrict__ q, float* __restrict__ scale, int64_t N, int K, int R,
                        float scale_mul) {
  using T = typename Elem<DT>::T;
  __shared__ float red[QTHREADS / 64];
  const int64_t g = blockIdx.y;                  // slice
  const int64_t r0 = (int64_t)blockIdx.x * R;    // first row of the group in the slice
  const int nr = (int)min((int64_t)R, N - r0);
  const T* xb = x + (g * N + r0) * K;
  const float* mr = MEAN ? mean + g * K : nullptr;
  const int total = nr * K;
  float amax = 0.f;
  for (int i = threadIdx.x; i < total; i += QTHREADS)
    amax = fmaxf(amax, fabsf(row_val<DT, MEAN>(xb + (i / K) * K, mr, i % K)));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = amax * (1.0f / 127.0f);
  const float safe = (s == 0.f) ? 1.f : s;
  for (int i = threadIdx.x; i < nr; i += QTHREADS) scale[g * N + r0 + i] = safe * scale_mul;
  int8_t* qb = q + (g * N + r0) * K;
  for (int i = threadIdx.x; i < total; i += QTHREADS)
    qb[i] = code_of(row_val<DT, MEAN>(xb + (i / K) * K, mr, i % K), safe);
}

}  // namespace
}  // namespace sl8

extern "C" int sl8_quantize_i8_row_groups(const void* x, int x_dtype, int64_t G, int64_t N,
                                          int64_t D, int64_t rows_per_group, const float* mean,
                                          float scale_mul, int8_t* q, float* scale, void* stream) {
  clear_error();
  SL8_CHECK_ARG(x_dtype == SL8_DTYPE_F16 || x_dtype == SL8_DTYPE_BF16 || x_dtype == SL8_DTYPE_F32,
                "quantize: input must be float16/bfloat16/float32");
  SL8_CHECK_ARG(G >= 0 && N >= 0 && D >= 0 && D < (1 << 20) && rows_per_group >= 1 &&
                    rows_per_group * D < (1LL << 30) && G < 65536,
                "quantize_row_groups: bad shape");
  if (G == 0 || N == 0 || D == 0) return SL8_OK;
  SL8_CHECK_ARG(x && q && scale, "quantize: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)((N + rows_per_group - 1) / rows_per_group), (unsigned)G);
#define SL8_RG(DT, MN)                                                                          \
  quant_row_groups_kernel<DT, MN><<<grid, QTHREADS, 0, st>>>(                                   \
      static_cast<const typename Elem<DT>::T*>(x), mean, q, scale, N, (int)D, (int)rows_per_group, \
      scale_mul)
  if (mean) {
    if (x_dtype == SL8_DTYPE_F16) SL8_RG(SL8_DTYPE_F16, true);
    else if (x_dtype == SL8_DTYPE_BF16) SL8_RG(SL8_DTYPE_BF16, true);
    else SL8_RG(SL8_DTYPE_F32, true);
  } else {
    if (x_dtype == SL8_DTYPE_F16) SL8_RG(SL8_DTYPE_F16, false);
    else if (x_dtype == SL8_DTYPE_BF16) SL8_RG(SL8_DTYPE_BF16, false);
    else SL8_RG(SL8_DTYPE_F32, false);
  }
#undef SL8_RG
  SL8_CHECK_LAUNCH("quantize_row_groups");
  return SL8_OK;
}

extern "C" int sl8_quantize_i8_rows_centered(const void* x, int x_dtype, int64_t G, int64_t N,
                                             int64_t D, const float* mean, float scale_mul,
                                             int8_t* q, float* scale, void* stream) {
  clear_error();
  SL8_CHECK_ARG(x_dtype == SL8_DTYPE_F16 || x_dtype == SL8_DTYPE_BF16 || x_dtype == SL8_DTYPE_F32,
                "quantize: input must be float16/bfloat16/float32");
  SL8_CHECK_ARG(G >= 0 && N >= 0 && D >= 0 && D < (1LL << 31), "quantize: bad shape");
  if (G == 0 || N == 0 || D == 0) return SL8_OK;
  SL8_CHECK_ARG(x && q && scale, "quantize: null pointer");
  SL8_CHECK_ARG((D & 3) != 0 || aligned(q, 4), "quantize: q must be 4-byte aligned");
  return dispatch_quant(x, x_dtype, mean, q, scale, G * N, N, D, scale_mul,
                        static_cast<hipStream_t>(stream));
}

extern "C" size_t sl8_k_mean_workspace(int64_t G, int64_t D) {
  if (G <= 0 || D <= 0) return 0;
  return (size_t)(G * D) * sizeof(long long);
}

extern "C" int sl8_k_mean(const void* k, int dtype, int64_t G, int64_t N, int64_t D,
                          float* mean, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  SL8_CHECK_ARG(dtype == SL8_DTYPE_F16 || dtype == SL8_DTYPE_BF16 || dtype == SL8_DTYPE_F32,
                "k_mean: input must be float16/bfloat16/float32");
  SL8_CHECK_ARG(G >= 0 && N >= 0 && D >= 0 && D < (1LL << 31), "k_mean: bad shape");
  SL8_CHECK_ARG(N < (1LL << 23), "k_mean: N must be < 2^23 keys, got %lld", (long long)N);
  if (G == 0 || D == 0) return SL8_OK;
  SL8_CHECK_ARG(N > 0, "k_mean: mean over zero keys");
  SL8_CHECK_ARG(k && mean, "k_mean: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == SL8_DTYPE_F16) {
    const size_t need = sl8_k_mean_workspace(G, D);
    SL8_CHECK_ARG(workspace && workspace_bytes >= need && aligned(workspace, 8),
                  "k_mean: workspace needs %zu bytes", need);
    unsigned long long* acc = static_cast<unsigned long long*>(workspace);
    const int64_t n = G * D;
    const unsigned ng = (unsigned)((n + 255) / 256);
    i64_zero_kernel<<<ng, 256, 0, st>>>(acc, n);
    const dim3 grid((unsigned)((D + MEAN_COLS - 1) / MEAN_COLS), (unsigned)G,
                    (unsigned)((N + MEAN_CHUNK - 1) / MEAN_CHUNK));
    k_mean_f16_kernel<<<grid, MEAN_COLS * MEAN_PHASES, 0, st>>>(static_cast<const uint16_t*>(k),
                                                                 acc, N, (int)D);
    k_mean_finish_kernel<<<ng, 256, 0, st>>>(acc, mean, n, N);
  } else {
    if (dtype == SL8_DTYPE_BF16) launch_k_mean_seq<SL8_DTYPE_BF16>(k, mean, G, N, D, st);
    else launch_k_mean_seq<SL8_DTYPE_F32>(k, mean, G, N, D, st);
  }
  SL8_CHECK_LAUNCH("k_mean");
  return SL8_OK;
}

// ---------------------------------------------------------------------------
// Outlier gate (reference superl8/quant/core.py:113-145): any row of Q with
// max|q| / (median|q| + 1e-10) > ratio (fp32) routes the call to full
// precision. One wave per row of D <= 64 E elements (lanes past D hold no
// element: they never count as "below" and add 0 to the max). The median is torch's
// lower median, the ((D-1)/2)-th smallest |q|, found exactly by a radix
// select on the fp32 bit patterns (non-negative floats order like their bits):
// 31 rounds of "how many elements lie below this prefix" (ballot + popcount).
// A row holding a NaN reports NaN for both and never fires, as in torch.
// ---------------------------------------------------------------------------
namespace sl8 {
namespace {

template <int DT, int E>
__global__ void __launch_bounds__(256)
q_gate_kernel(const void* __restrict__ q, int64_t rows, int D, float ratio,
              int32_t* __restrict__ flag, float* __restrict__ stats) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // wave-uniform
  uint32_t bits[E];
  float mx = 0.f;
  bool nan = false;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int c = e * 64 + lane;
    const int64_t i = row * D + (c < D ? c : 0);
    float x;
    if constexpr (DT == SL8_DTYPE_F32) x = static_cast<const float*>(q)[i];
    else x = u16_to_f<DT>(static_cast<const uint16_t*>(q)[i]);
    x = c < D ? fabsf(x) : 0.f;
    nan |= x != x;
    bits[e] = c < D ? __float_as_uint(x) : 0xFFFFFFFFu;
    mx = fmaxf(mx, x);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  const int K = (D - 1) / 2;
  uint32_t ans = 0;
  for (int b = 30; b >= 0; --b) {
    const uint32_t t = ans | (1u << b);
    int cnt = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) cnt += __popcll(__ballot(bits[e] < t));
    if (cnt <= K) ans = t;
  }
  float med = __uint_as_float(ans);
  if (__ballot(nan)) {  // torch's amax and median both propagate NaN: the row never fires
    mx = __uint_as_float(0x7fc00000u);
    med = mx;
  }
  if (lane == 0) {
    if (stats) {
      stats[2 * row] = mx;
      stats[2 * row + 1] = med;
    }
    if (__fdiv_rn(mx, med + 1e-10f) > ratio) atomicOr(flag, 1);
  }
}

}  // namespace
}  // namespace sl8

extern "C" int sl8_q_outlier_gate(const void* q, int dtype, int64_t rows, int64_t D, float ratio,
                                  int32_t* flag, float* stats, void* stream) {
  clear_error();
  SL8_CHECK_ARG(rows >= 0 && D >= 1 && D <= 256,
                "fni8 outlier gate: head dim must be 1..256, got %lld", (long long)D);
  SL8_CHECK_ARG(dtype == SL8_DTYPE_F16 || dtype == SL8_DTYPE_BF16 || dtype == SL8_DTYPE_F32,
                "fni8 outlier gate: q must be float16, bfloat16 or float32");
  if (rows == 0) return SL8_OK;
  SL8_CHECK_ARG(q && flag, "fni8 outlier gate: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)((rows + 3) / 4));
#define SL8_GATE(DT, E) q_gate_kernel<DT, E><<<grid, 256, 0, st>>>(q, rows, (int)D, ratio, flag, stats)
#define SL8_GATE_D(DT) \
  if (D <= 64) SL8_GATE(DT, 1); else if (D <= 128) SL8_GATE(DT, 2); else SL8_GATE(DT, 4);
  if (dtype == SL8_DTYPE_F16) { SL8_GATE_D(SL8_DTYPE_F16) }
  else if (dtype == SL8_DTYPE_BF16) { SL8_GATE_D(SL8_DTYPE_BF16) }
  else { SL8_GATE_D(SL8_DTYPE_F32) }
#undef SL8_GATE_D
#undef SL8_GATE
  SL8_CHECK_LAUNCH("outlier gate");
  return SL8_OK;
}

// ---------------------------------------------------------------------------
// Fused attention prologue for fp16 / bf16 Q/K (reference superl8/quant/core.py
// quantize_qk + smooth_k, and the outlier gate of superl8/ops.py:115-147):
// two launches instead of six, Q read once, K read twice, no zeroing pass.
//
// Launch A: K-mean partials. Block (g, c) sums the key rows of chunk c of
//   group g with 16-byte loads, a pass of a thread's rows in flight at once,
//   and stores its D partial sums: fp16 exactly in int64 fixed point (value *
//   2^24, decoded from the fp16 bits), hence independent of the summation
//   order; bf16 in fp64, whose 53 bits hold sums of 8-bit significands exactly
//   unless one column spans more than about 2^30 in magnitude (then the order
//   is fixed: rows of a thread, threads, chunks). Block 0 clears the gate flag.
// Launch B, two roles chosen per block:
//   * K: issues its key rows' loads, forms the group's mean from the C
//     partials meanwhile (as sl8_k_mean; the first block of each group also
//     stores it), subtracts it from each row with the rounding of torch.sub
//     and quantises the row;
//   * Q: per-row int8 quantisation (scale * q_scale_mul) and, with a gate
//     ratio, the outlier decision for every row. f(x) = fl(max / fl(x + 1e-10))
//     is non-increasing in x >= 0, so f(median) > ratio iff more than (D-1)/2
//     of the row's |x| have f(|x|) > ratio: the row is decided exactly with
//     no median search (the division is needed only for elements within
//     2^-18 of max / ratio). A row holding a NaN never fires (torch's amax and
//     median are NaN there). A block with a firing row ORs 1 into the flag
//     (atomicOr), so the flag is set iff some row fires. The caller's host copy of the flag, if
//     any, is stored to by the same thread: a copy behind the launch cost 4 us on the device and
//     3.5 us on the host (a prefill of 8 heads x 512, D = 64: 52.0 us, 46.5 here).
// sl8_quantize_qkv adds V's per-channel codes (column maxima in A, codes in B) and the rotation of
// Q and the smoothed K; without Q it builds a K/V cache. Bound by HBM: K and V are read twice
// (the second time from the MALL where they fit). 16384 keys of 8 heads, D = 128: 93 us as nine
// launches (a byte store per element in the column kernel, the smoothed K written and read back), 37 us here.
// Head dims 72 and 80 take the 16 lanes per row of 128 with 9 and 10 of them
// holding elements.
// ---------------------------------------------------------------------------
namespace sl8 {
namespace {

constexpr int PRO_CHUNK = 128;      // key rows per mean partial, up to PRO_CHUNKS_MAX partials;
// beyond, the chunks grow: every K block of B reads all its group's partials, which at 128 rows
// a partial would be more bytes than its own rows from N = 2048 on (16-bit D = 128: 1 KB a
// partial, 16 KB of rows) and grow with N * N
constexpr int PRO_CHUNKS_MAX = 48;
constexpr int PRO_KROWS = 64;       // key rows per quantise block (each K block also forms its group's mean: 32 measured 1 us slower at config 2, 128 0.3 us)
constexpr int PRO_QBLOCKS_MAX = 16384;
constexpr int PRO_QP = 1;           // Q rows per thread per pass (1: measured fastest; more rows per thread cost occupancy)

int64_t pro_chunk_rows(int64_t N) {
  const int64_t per = (N + PRO_CHUNKS_MAX - 1) / PRO_CHUNKS_MAX;
  return std::max<int64_t>(PRO_CHUNK, (per + PRO_CHUNK - 1) / PRO_CHUNK * PRO_CHUNK);
}

// fp16 bits -> value * 2^24 as an exact integer (finite inputs: |result| < 2^40)
__device__ __forceinline__ long long f16_fixed24(uint32_t h) {
  const uint32_t e = (h >> 10) & 31u, m = h & 1023u;
  const long long v = e ? (long long)(1024u + m) << (e - 1) : (long long)m;
  return (h & 0x8000u) ? -v : v;
}

// The K-mean partial sums of a storage type.
template <int DT> struct MeanSum;
template <> struct MeanSum<SL8_DTYPE_F16> {
  using T = long long;
  __device__ static T of(uint32_t bits) { return f16_fixed24(bits); }
  __device__ static float mean(T sum, int64_t N) {
    return (float)(((double)sum * 0x1p-24) / (double)N);
  }
};
template <> struct MeanSum<SL8_DTYPE_BF16> {
  using T = double;
  __device__ static T of(uint32_t bits) { return (double)bf2f((uint16_t)bits); }
  __device__ static float mean(T sum, int64_t N) { return (float)(sum / (double)N); }
};

// Partial sums over rows [n0, n1) of k[., D] by a 256-thread block -> part[0, D).
template <int DT, int D>
__device__ __forceinline__ void mean_chunk(const uint16_t* __restrict__ kg, int64_t n0, int64_t n1,
                                           typename MeanSum<DT>::T* __restrict__ part) {
  using S = MeanSum<DT>;
  constexpr int LPR = row_lanes(D), NL = D / 8;
  constexpr int RPP = 256 / LPR;                     // rows per pass
  constexpr int NIT = PRO_CHUNK / RPP < 8 ? PRO_CHUNK / RPP : 8;  // passes in flight
  const int lane = threadIdx.x % LPR, sub = threadIdx.x / LPR;
  const bool on = lane < NL;
  __shared__ typename S::T red[RPP][D];
  typename S::T acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0;
  for (int64_t b = n0; b < n1; b += NIT * RPP) {
    uint4 raw[NIT];
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
      const int64_t n = b + sub + i * RPP;
      raw[i] = on && n < n1 ? reinterpret_cast<const uint4*>(kg + n * D)[lane] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const uint32_t w[4] = {raw[it].x, raw[it].y, raw[it].z, raw[it].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] += S::of(w[i] & 0xFFFFu);
        acc[2 * i + 1] += S::of(w[i] >> 16);
      }
    }
  }
  if (on) {
#pragma unroll
    for (int e = 0; e < 8; ++e) red[sub][lane * 8 + e] = acc[e];
  }
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += 256) {
    typename S::T t = 0;
#pragma unroll 8
    for (int p = 0; p < RPP; ++p) t += red[p][d];
    part[d] = t;
  }
}

// Smooth (+ rotate) + quantise `rows` key rows from n0 on, by a 256-thread block: the first rows'
// loads are issued first, the group's mean is formed from its C partials under them.
template <int DT, int D, bool ROT>
__device__ __forceinline__ void smooth_rows(const uint16_t* __restrict__ kg, int64_t n0, int rows, int64_t N,
                                            const typename MeanSum<DT>::T* __restrict__ part, int C,
                                            float* __restrict__ mean_out,
                                            int8_t* __restrict__ kq, float* __restrict__ kscale) {
  using S = MeanSum<DT>;
  constexpr int LPR = row_lanes(D), NL = D / 8, RPP = 256 / LPR, NP = PRO_KROWS / RPP;
  const int lane = threadIdx.x % LPR, sub = threadIdx.x / LPR;
  const bool on = lane < NL;
  uint4 raw[NP];
  const int64_t n_end = min(N, n0 + rows);
  auto load = [&](int64_t b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int64_t n = b + i * RPP + sub;
      raw[i] = on && n < n_end ? reinterpret_cast<const uint4*>(kg + n * D)[lane] : make_uint4(0, 0, 0, 0);
    }
  };
  load(n0);
  // column d summed by PS threads over every PS-th partial, then in LDS
  constexpr int PS = 256 / D;
  __shared__ typename S::T mred[PS][D];
  __shared__ float mean_s[D];
  if (threadIdx.x < PS * D) {
    const int d = threadIdx.x % D, ps = threadIdx.x / D;
    typename S::T t = 0;
#pragma unroll 8
    for (int c = ps; c < C; c += PS) t += part[(int64_t)c * D + d];
    mred[ps][d] = t;
  }
  __syncthreads();
  if (threadIdx.x < D) {
    typename S::T t = 0;
#pragma unroll
    for (int p = 0; p < PS; ++p) t += mred[p][threadIdx.x];
    const float m = S::mean(t, N);
    mean_s[threadIdx.x] = m;
    if (mean_out) mean_out[threadIdx.x] = m;
  }
  __syncthreads();
  float mv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) mv[e] = on ? mean_s[lane * 8 + e] : 0.f;
  auto rows_of = [&](const uint4 (&r)[NP], int64_t b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int64_t n = b + i * RPP + sub;
      float f[8];
      VecIO<DT>::unpack(r[i], f);
      float mx = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = Elem<DT>::round(f[e] - mv[e]);
      if constexpr (ROT) rotate_row<DT, D>(f, lane);
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(f[e]));
      mx = lane_group_max<LPR>(mx);
      const float s = mx * (1.0f / 127.0f);
      const float safe = (s == 0.f) ? 1.f : s;
      if (on && n < n_end) {
        if (lane == 0) kscale[n] = safe;
        reinterpret_cast<uint2*>(kq + n * D)[lane] = row_codes8<DT>(f, safe);
      }
    }
  };
  for (int64_t b = n0; b < n_end; b += PRO_KROWS) {
    uint4 cur[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) cur[i] = raw[i];
    if (b + PRO_KROWS < n_end) load(b + PRO_KROWS);  // in flight under this pass
    rows_of(cur, b);
  }
}

// Column maxima of |v| over rows [n0, n1) by a 256-thread block -> part[0, D) (NaN elements are
// skipped, as by fmaxf).
template <int DT, int D>
__device__ __forceinline__ void amax_chunk(const uint16_t* __restrict__ vg, int64_t n0, int64_t n1,
                                           float* __restrict__ part) {
  constexpr int LPR = row_lanes(D), NL = D / 8, RPP = 256 / LPR;
  constexpr int NIT = PRO_CHUNK / RPP < 8 ? PRO_CHUNK / RPP : 8;
  const int lane = threadIdx.x % LPR, sub = threadIdx.x / LPR;
  const bool on = lane < NL;
  __shared__ float red[RPP][D];
  float mx[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) mx[e] = 0.f;
  for (int64_t b = n0; b < n1; b += NIT * RPP) {
    uint4 raw[NIT];
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
      const int64_t n = b + sub + i * RPP;
      raw[i] = on && n < n1 ? reinterpret_cast<const uint4*>(vg + n * D)[lane] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
      float f[8];
      VecIO<DT>::unpack(raw[i], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) mx[e] = fmaxf(mx[e], fabsf(f[e]));
    }
  }
  if (on) {
#pragma unroll
    for (int e = 0; e < 8; ++e) red[sub][lane * 8 + e] = mx[e];
  }
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += 256) {
    float m = 0.f;
#pragma unroll 8
    for (int p = 0; p < RPP; ++p) m = fmaxf(m, red[p][d]);
    part[d] = m;
  }
}

// Per-channel codes of `rows` rows from n0 on, the group's scales formed from its C partial
// maxima (codes8 with a scale per element).
template <int DT, int D>
__device__ __forceinline__ void channel_rows(const uint16_t* __restrict__ vg, int64_t n0, int rows,
                                             int64_t N, const float* __restrict__ part, int C,
                                             float* __restrict__ scale_out, int8_t* __restrict__ vq) {
  constexpr int LPR = row_lanes(D), NL = D / 8, RPP = 256 / LPR, NP = PRO_KROWS / RPP;
  const int lane = threadIdx.x % LPR, sub = threadIdx.x / LPR;
  const bool on = lane < NL;
  uint4 raw[NP];
  const int64_t n_end = min(N, n0 + rows);
  auto load = [&](int64_t b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int64_t n = b + i * RPP + sub;
      raw[i] = on && n < n_end ? reinterpret_cast<const uint4*>(vg + n * D)[lane] : make_uint4(0, 0, 0, 0);
    }
  };
  load(n0);
  constexpr int PS = 256 / D;
  __shared__ float mred[PS][D], scale_s[D];
  if (threadIdx.x < PS * D) {
    const int d = threadIdx.x % D, ps = threadIdx.x / D;
    float m = 0.f;
#pragma unroll 8
    for (int c = ps; c < C; c += PS) m = fmaxf(m, part[(int64_t)c * D + d]);
    mred[ps][d] = m;
  }
  __syncthreads();
  if (threadIdx.x < D) {
    float m = 0.f;
#pragma unroll
    for (int p = 0; p < PS; ++p) m = fmaxf(m, mred[p][threadIdx.x]);
    const float s = m * (1.0f / 127.0f);
    const float safe = (s == 0.f) ? 1.f : s;
    scale_s[threadIdx.x] = safe;
    if (scale_out) scale_out[threadIdx.x] = safe;
  }
  __syncthreads();
  float safe[8], inv[8];
  bool fast = true;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    safe[e] = on ? scale_s[lane * 8 + e] : 1.f;
    inv[e] = __builtin_amdgcn_rcpf(safe[e]);
    fast &= DT == SL8_DTYPE_F16 || safe[e] >= 0x1p-120f;
  }
  for (int64_t b = n0; b < n_end; b += PRO_KROWS) {
    uint4 cur[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) cur[i] = raw[i];
    if (b + PRO_KROWS < n_end) load(b + PRO_KROWS);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int64_t n = b + i * RPP + sub;
      float f[8];
      VecIO<DT>::unpack(cur[i], f);
      if (on && n < n_end)
        reinterpret_cast<uint2*>(vq + n * D)[lane] = codes8_each(f, safe, inv, fast);
    }
  }
}

// A: K-mean partials of `chunk`-row chunks, one block per (group, chunk), then the column maxima
// of V's chunks.
template <int DT, int D, bool HASV>
__global__ void __launch_bounds__(256)
prologue_a_kernel(const uint16_t* __restrict__ k, int64_t N, int C, int64_t chunk,
                  typename MeanSum<DT>::T* __restrict__ part, int32_t* __restrict__ flag,
                  int nka, const uint16_t* __restrict__ v, float* __restrict__ vpart) {
  if (flag && blockIdx.x == 0 && threadIdx.x == 0) *flag = 0;
  const bool is_v = HASV && (int)blockIdx.x >= nka;
  const int64_t i = blockIdx.x - (is_v ? nka : 0), g = i / C, c = i % C;
  const int64_t n0 = c * chunk, n1 = min(N, n0 + chunk);
  if constexpr (HASV) {
    if (is_v) return amax_chunk<DT, D>(v + g * N * D, n0, n1, vpart + i * D);
  }
  mean_chunk<DT, D>(k + g * N * D, n0, n1, part + i * D);
}

// B: the smoothed K rows (blocks [0, nkb): krows rows of group
// blockIdx / kbg each), V's rows (nvb blocks, likewise) and the Q rows with the outlier gate (the
// rest). The Q work does not depend on the mean, but sharing this launch keeps it off the
// critical path A -> mean -> B of the K side.
template <int DT, int D, bool GATE, bool ROT, bool HASV>
__global__ void __launch_bounds__(256)
prologue_b_kernel(const uint16_t* __restrict__ k, int64_t N,
                  const typename MeanSum<DT>::T* __restrict__ part,
                  int C, float* __restrict__ k_mean,
                  int8_t* __restrict__ k_i8, float* __restrict__ k_scale, int krows, int kbg, int nkb,
                  const uint16_t* __restrict__ q, int64_t qrows, float qmul, float ratio,
                  int8_t* __restrict__ q_i8, float* __restrict__ q_scale,
                  int32_t* __restrict__ flag, int32_t* flag_host, int nvb,
                  const uint16_t* __restrict__ v, const float* __restrict__ vpart, int8_t* __restrict__ v_i8,
                  float* __restrict__ v_scale) {
  constexpr int LPR = row_lanes(D), NL = D / 8, RPP = 256 / LPR;
  const int lane = threadIdx.x % LPR, sub = threadIdx.x / LPR;
  if ((int)blockIdx.x < nkb) {
    const int64_t g = blockIdx.x / kbg;
    const int b = blockIdx.x % kbg;
    smooth_rows<DT, D, ROT>(k + g * N * D, (int64_t)b * krows, krows, N, part + g * C * D, C,
                            b == 0 && k_mean ? k_mean + g * D : nullptr, k_i8 + g * N * D,
                            k_scale + g * N);
    return;
  }
  if constexpr (HASV) {
    if ((int)blockIdx.x < nkb + nvb) {
      const int64_t g = (blockIdx.x - nkb) / kbg;
      const int b = (blockIdx.x - nkb) % kbg;
      return channel_rows<DT, D>(v + g * N * D, (int64_t)b * krows, krows, N, vpart + g * C * D, C,
                                 b == 0 ? v_scale + g * D : nullptr, v_i8 + g * N * D);
    }
  }
  const bool on = lane < NL;
  const int qb = blockIdx.x - nkb - nvb, nqb = gridDim.x - nkb - nvb;
  int fired = 0;
  const float rinv = 1.f / ratio;
  for (int64_t base = (int64_t)qb * RPP * PRO_QP; base < qrows;
       base += (int64_t)nqb * RPP * PRO_QP) {
    uint4 raw[PRO_QP];  // all of this thread's rows are fetched before any is processed
#pragma unroll
    for (int p = 0; p < PRO_QP; ++p) {
      const int64_t r = base + p * RPP + sub;
      raw[p] = on && r < qrows ? reinterpret_cast<const uint4*>(q + r * D)[lane]
                               : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int p = 0; p < PRO_QP; ++p) {
      const int64_t r = base + p * RPP + sub;
      const bool live = r < qrows;
      float f[8];
      VecIO<DT>::unpack(raw[p], f);
      if constexpr (ROT) rotate_row<DT, D>(f, lane);
      float mx = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(f[e]));
      mx = lane_group_max<LPR>(mx);
      const float s = mx * (1.0f / 127.0f);
      const float safe = (s == 0.f) ? 1.f : s;
      if (live && on) {
        if (lane == 0) q_scale[r] = safe * qmul;
        reinterpret_cast<uint2*>(q_i8 + r * D)[lane] = row_codes8<DT>(f, safe);
      }
      if constexpr (GATE) {
        // y = fl(|x| + 1e-10) against t = max / ratio: far from t the exact test
        // fl(max / y) > ratio is decided by y < t; within 2^-18 of t (relative)
        // the IEEE division decides.
        // (t below 2^-100: every element takes the division.)
        const float t = mx * rinv;
        const bool tiny = t < 0x1p-100f;
        const float thi = tiny ? INFINITY : t * (1.f + 0x1p-18f);
        // first an upper bound of the count, |x| <= thi: rows that could fire are rare, and only a
        // wave that holds one counts exactly
        int cnt = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) cnt += fabsf(f[e]) <= thi;
        if (!on) cnt = 0;  // a lane without elements
        cnt = lane_group_sum<LPR>(cnt);
        const bool maybe = live && cnt > (D - 1) / 2;
        if (__builtin_expect(__ballot(maybe) == 0, 1)) continue;
        const float tlo = tiny ? 0.f : t * (1.f - 0x1p-18f);
        int nan = 0;
        cnt = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float a = fabsf(f[e]);
          nan |= a != a;
          const float y = a + 1e-10f;
          cnt += y < tlo || (y <= thi && __fdiv_rn(mx, y) > ratio);
        }
        if (!on) cnt = 0;
        cnt = lane_group_sum<LPR>(cnt + (nan << 16));  // NaN count in the high half
        if (live && (cnt >> 16) == 0 && (cnt & 0xFFFF) > (D - 1) / 2) fired = 1;
      }
    }
  }
  if constexpr (GATE) {
    fired = __syncthreads_or(fired);
    if (fired && threadIdx.x == 0) {
      atomicOr(flag, 1);  // cleared by A, earlier on the stream
      if (flag_host)
        __hip_atomic_store(flag_host, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

int prologue_nqb(int64_t qrows, int D) {
  const int64_t rpp = 256 / row_lanes(D) * PRO_QP;
  return (int)std::min<int64_t>(PRO_QBLOCKS_MAX, (qrows + rpp - 1) / rpp);
}

// The sizes of one prologue call and its launches for a storage type and head dim.
struct Prologue {
  const uint16_t *q, *k, *v;  // null: no queries (qrows 0), keys, values
  int64_t qrows, G, N;
  float q_scale_mul, gate_ratio;
  int8_t *q_i8, *k_i8, *v_i8;
  float *q_scale, *k_scale, *v_scale, *k_mean;
  int32_t *flag, *flag_host;
  bool rotate;
  void* part;
  hipStream_t st;
  int64_t chunk;
  int C, krows, kbg;

  // A (K-mean partials) -> B (the mean, K and Q rows, gate): the Q rows, the
  // bulk of the bytes, run beside the K rows in B instead of ahead of the mean
  template <int DT, int D>
  void go() const {
    using S = typename MeanSum<DT>::T;
    const int nka = k ? (int)(G * C) : 0, nkb = k ? (int)(G * kbg) : 0;
    const int nva = v ? (int)(G * C) : 0, nvb = v ? (int)(G * kbg) : 0;
    const int nqb = qrows ? prologue_nqb(qrows, D) : 0;
    S* pt = static_cast<S*>(part);
    float* vpt = reinterpret_cast<float*>(pt + (int64_t)nka * D);
    using T = std::true_type;
    using F = std::false_type;
    auto run = [&](auto gate, auto rot, auto hasv) {
      constexpr bool HV = decltype(hasv)::value;
      prologue_a_kernel<DT, D, HV><<<nka + nva, 256, 0, st>>>(k, N, C, chunk, pt, flag, nka, v, vpt);
      prologue_b_kernel<DT, D, decltype(gate)::value, decltype(rot)::value, HV>
          <<<nkb + nvb + nqb, 256, 0, st>>>(k, N, pt, C, k_mean, k_i8, k_scale, krows, kbg, nkb, q,
                                            qrows, q_scale_mul, gate_ratio, q_i8, q_scale, flag,
                                            flag_host, nvb, v, vpt, v_i8, v_scale);
    };
    if constexpr ((D & (D - 1)) == 0) {
      if (rotate) return v ? run(F{}, T{}, T{}) : run(F{}, T{}, F{});
    }
    if (flag) run(T{}, F{}, F{});
    else if (v) run(F{}, F{}, T{});
    else run(F{}, F{}, F{});
  }
  template <int DT>
  void go(int64_t D) const {
    switch (D) {
      case 32: return go<DT, 32>();
      case 64: return go<DT, 64>();
      case 72: return go<DT, 72>();
      case 80: return go<DT, 80>();
      case 128: return go<DT, 128>();
      default: return go<DT, 256>();
    }
  }
};

// Checks and launches shared by the entries (q_i8 .. as in Prologue).
int prologue(Prologue p, int dtype, int64_t D, void* workspace, size_t workspace_bytes,
             size_t need, void* stream) {
  SL8_CHECK_ARG(dtype == SL8_DTYPE_F16 || dtype == SL8_DTYPE_BF16,
                "fused prologue: q and k must be float16 or bfloat16");
  SL8_CHECK_ARG(D == 32 || D == 64 || D == 72 || D == 80 || D == 128 || D == 256,
                "fused prologue: head dim must be 32/64/72/80/128/256, got %lld", (long long)D);
  SL8_CHECK_ARG(!p.rotate || (D & (D - 1)) == 0,
                "fused prologue: Hadamard needs a power-of-two dim, got %lld", (long long)D);
  SL8_CHECK_ARG(p.G > 0 && p.N > 0 && p.N < (1LL << 23),
                "fused prologue: bad shape (rows %lld, groups %lld, keys %lld)", (long long)p.qrows,
                (long long)p.G, (long long)p.N);
  SL8_CHECK_ARG((p.k || p.v) && (!p.k || (p.k_i8 && p.k_scale)) && (!p.qrows || (p.q && p.q_i8 && p.q_scale)) &&
                    (!p.v || (p.v_i8 && p.v_scale)),
                "fused prologue: null pointer");
  SL8_CHECK_ARG(aligned(p.q, 16) && aligned(p.k, 16) && aligned(p.v, 16) && aligned(p.q_i8, 8) &&
                    aligned(p.k_i8, 8) && aligned(p.v_i8, 8),
                "fused prologue: q/k/v must be 16-byte and codes 8-byte aligned");
  SL8_CHECK_ARG(workspace && workspace_bytes >= need && aligned(workspace, 8),
                "fused prologue: workspace needs %zu bytes", need);
  // rows per quantise block: up to 256 while two blocks per CU remain (K's alone), since every
  // block reads all its group's partials: 16384 keys of 8 heads, D = 128, K and V: 64 rows a block
  // 30.0 us, 128 rows 21.9, 256 rows 20.7 (101 MB at 4.9 TB/s)
  int64_t krows = PRO_KROWS;
  while (krows < 4 * PRO_KROWS && p.G * (p.N / (2 * krows)) >= 512) krows *= 2;
  const int64_t kbg = (p.N + krows - 1) / krows;  // quantise blocks per group
  p.chunk = pro_chunk_rows(p.N);
  p.C = (int)((p.N + p.chunk - 1) / p.chunk);
  p.krows = (int)krows;
  p.kbg = (int)kbg;
  SL8_CHECK_ARG(p.G * kbg < (1LL << 29) && p.G < 65536, "fused prologue: too many key groups");
  p.part = workspace;
  p.st = static_cast<hipStream_t>(stream);
  if (dtype == SL8_DTYPE_F16) p.go<SL8_DTYPE_F16>(D);
  else p.go<SL8_DTYPE_BF16>(D);
  SL8_CHECK_LAUNCH("fused prologue");
  return SL8_OK;
}

}  // namespace
}  // namespace sl8

extern "C" size_t sl8_quantize_qk_workspace(int64_t BHq_M, int64_t G, int64_t N, int64_t D) {
  if (G <= 0 || N <= 0 || D <= 0) return 0;
  const int64_t chunk = pro_chunk_rows(N), C = (N + chunk - 1) / chunk;
  (void)BHq_M;  // the Q rows need no workspace (the gate sets the flag directly)
  return (size_t)(G * C * D) * sizeof(long long);  // the K-mean partials
}

extern "C" int sl8_quantize_qk_hostflag(const void* q, const void* k, int dtype, int64_t qrows,
                                        int64_t G, int64_t N, int64_t D, float q_scale_mul,
                                        float gate_ratio, int8_t* q_i8, float* q_scale,
                                        int8_t* k_i8, float* k_scale, float* k_mean,
                                        int32_t* gate_flag, int32_t* gate_flag_host,
                                        void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  const bool gate = gate_ratio > 0.f;
  SL8_CHECK_ARG(!gate || gate_flag, "fused prologue: gate_flag required with a gate ratio");
  SL8_CHECK_ARG(qrows > 0, "fused prologue: bad shape (rows %lld)", (long long)qrows);
  SL8_CHECK_ARG(k && k_mean, "fused prologue: null pointer");
  const Prologue p{static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k), nullptr, qrows,
                   G, N, q_scale_mul, gate_ratio, q_i8, k_i8, nullptr, q_scale, k_scale, nullptr,
                   k_mean, gate ? gate_flag : nullptr, gate ? gate_flag_host : nullptr, false, nullptr,
                   nullptr, 0, 0, 0, 0};
  return prologue(p, dtype, D, workspace, workspace_bytes,
                  sl8_quantize_qk_workspace(qrows, G, N, D), stream);
}

extern "C" int sl8_quantize_qk(const void* q, const void* k, int dtype, int64_t qrows, int64_t G,
                               int64_t N, int64_t D, float q_scale_mul, float gate_ratio,
                               int8_t* q_i8, float* q_scale, int8_t* k_i8, float* k_scale,
                               float* k_mean, int32_t* gate_flag, void* workspace,
                               size_t workspace_bytes, void* stream) {
  return sl8_quantize_qk_hostflag(q, k, dtype, qrows, G, N, D, q_scale_mul, gate_ratio, q_i8, q_scale,
                                  k_i8, k_scale, k_mean, gate_flag, nullptr, workspace,
                                  workspace_bytes, stream);
}

extern "C" size_t sl8_quantize_qkv_workspace(int64_t G, int64_t N, int64_t D) {
  return sl8_quantize_qk_workspace(0, G, N, D) / sizeof(long long) * (sizeof(long long) + sizeof(float));
}

extern "C" int sl8_quantize_qkv(const void* q, const void* k, const void* v, int dtype,
                                int64_t qrows, int64_t G, int64_t N, int64_t D, int rotate,
                                float q_scale_mul, int8_t* q_i8, float* q_scale, int8_t* k_i8,
                                float* k_scale, float* k_mean, int8_t* v_i8, float* v_scale,
                                void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  SL8_CHECK_ARG(qrows >= 0 && (q || qrows == 0), "fused prologue: bad shape (rows %lld)",
                (long long)qrows);
  const Prologue p{static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k),
                   static_cast<const uint16_t*>(v), qrows, G, N, q_scale_mul, 0.f, q_i8, k_i8, v_i8,
                   q_scale, k_scale, v_scale, k_mean, nullptr, nullptr, rotate != 0, nullptr, nullptr, 0, 0, 0, 0};
  return prologue(p, dtype, D, workspace, workspace_bytes, sl8_quantize_qkv_workspace(G, N, D),
                  stream);
}
