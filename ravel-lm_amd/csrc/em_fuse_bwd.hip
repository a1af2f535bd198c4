// Weight gradient of the lookup fused with the linear map (gfx950 MFMA).
//
// Replaces the grad_weight of ravel_lm/triton_memory.py:428-475:
//   gw[m, q] = sum_n grad[n, m] * A[n, q],   n = b*T + t, q = c*P + p,
// with A the looked-up rows (payload[src[n*C + c]], zeros where src < 0),
// which are gathered straight from the payload and never stored.
//
// The sum runs over all B*T rows while the result is small (M x C*P), so the
// rows are split: a block owns BM x 256 results over one range of rows, and
// writes fp32 partial sums that a second kernel adds in a fixed order (no
// atomics: the result does not depend on timing) and rounds once.
//
// Both operands arrive row-major in n, but an MFMA operand wants 8 consecutive
// n of one column per lane.  A thread therefore loads one 16-byte unit (8
// columns) of 8 consecutive rows, transposes the 8 x 8 values in registers (32
// byte-permutes) and writes 8 units of 8 n each to LDS at [n / 8][column], from
// where a wave reads its operands 16 bytes a lane without bank conflicts: unit
// j of column group u sits at slot j ^ (u % 8), which spreads both the 128-byte
// strides of the stores and the reads over the banks.  A step covers 64 rows;
// while it multiplies out of one LDS buffer, the rows of the next are in flight
// into registers and the sources of the one after that are loaded.
//
// Bound by the matrix cores and the LDS reads of their operands (10 units of
// 1 KiB per 24 MFMAs a wave at BM = 192).  At 131072 rows, M = 192, C*P = 1024
// bf16: 96.5 us (0.53 PFLOP/s) and 8.6 us for the sum of 64 partial results,
// where the gather of the looked-up rows and the library product took 591 us
// (its grid had no split of the long sum).

#include <type_traits>

#include "em_common.h"

namespace rem {

namespace {

constexpr int kGwThreads = 512;
constexpr int kGwStep = 64;   // rows a step
constexpr int kGwCols = 256;  // result columns of a block
constexpr int kGwTarget = 256;  // blocks wanted: one per CU (LDS and registers hold one)

typedef __bf16 gw_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 gw_f16x8 __attribute__((ext_vector_type(8)));
typedef float gw_f32x4 __attribute__((ext_vector_type(4)));

__device__ u32x4 kGwZero = {0u, 0u, 0u, 0u};  // never written: what a missing unit reads

template <bool F16>
__device__ __forceinline__ gw_f32x4 gw_mfma(u32x4 a, u32x4 b, gw_f32x4 c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gw_f16x8, a),
                                                  __builtin_bit_cast(gw_f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gw_bf16x8, a),
                                                   __builtin_bit_cast(gw_bf16x8, b), c, 0, 0, 0);
}

// Slot of the unit of column q (within 16-byte units of 8 n) in its LDS row.
__device__ __forceinline__ int gw_slot(int q) { return (q & ~7) | ((q ^ (q >> 3)) & 7); }

// MT: 16-row result tiles per wave; the block covers BM = 32 * MT rows of gw
// (2 wave rows) and 256 columns (4 wave columns of 64).
template <bool F16, int MT>
__global__ __launch_bounds__(kGwThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void weight_grad_kernel(
    const unsigned char* __restrict__ payload, const int32_t* __restrict__ src,
    const unsigned char* __restrict__ grad, int64_t NR, int C, int P, FastDiv byP, int M,
    int64_t nsrc, int nkt, int nmt, int64_t nlogical, int64_t steps, int nsplit,
    float* __restrict__ part) {
  constexpr int BM = 32 * MT;
  constexpr int NG = kGwStep / 8;               // groups of 8 n
  constexpr int ROWU = kGwCols + BM;            // units of one n group: A columns, then grad's
  constexpr int BUF = NG * ROWU;                // units of a step
  __shared__ __align__(16) u32x4 lds[2 * BUF];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int64_t logical = xcd_block(blockIdx.x, gridDim.x);  // tiles of one row range share an XCD
  if (logical >= nlogical) return;  // padding block of the XCD-rounded grid (uniform)
  const int ntile = nkt * nmt;
  const int split = (int)(logical / ntile);
  const int tile = (int)(logical - (int64_t)split * ntile);
  const int k0 = (tile % nkt) * kGwCols, m0 = (tile / nkt) * BM;
  const int K = C * P;
  const int64_t s0 = steps * split / nsplit, s1 = steps * (split + 1) / nsplit;
  // Loading roles (wave-uniform): threads 0..255 the looked-up rows (32 column
  // groups x 8 n groups), the next BM threads grad's (BM / 8 column groups).
  constexpr int AT = (kGwCols / 8) * NG, GT = (BM / 8) * NG;
  const bool isA = tid < AT, isG = !isA && tid < AT + GT;
  const int li = isA ? tid : tid - AT;
  const int lu = isA ? (li & 31) : li % (BM / 8);  // column group
  const int lg = isA ? (li >> 5) : li / (BM / 8);  // n group
  const int q = k0 + lu * 8;
  const int c = isA && q < K ? (int)fdiv((uint32_t)q, byP) : 0;
  const int pq = q - c * P;  // column inside the head
  const int mcol = m0 + lu * 8;
  const bool incol = isA ? q < K : (isG && mcol < M);
  const u32x4* zero = &kGwZero;
  auto load_src = [&](int64_t st, int32_t (&sv)[8]) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int64_t n = st * kGwStep + lg * 8 + r;
      sv[r] = -1;
      if (isA && incol && st < s1 && n < NR) sv[r] = src[n * C + c];
    }
  };
  auto load_rows = [&](int64_t st, const int32_t (&sv)[8], u32x4 (&x)[8]) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int64_t n = st * kGwStep + lg * 8 + r;
      const u32x4* p = zero;
      if (isA) {
        if (sv[r] >= 0 && sv[r] < nsrc) p = (const u32x4*)(payload + ((int64_t)sv[r] * P + pq) * 2);
      } else if (incol && st < s1 && n < NR) {
        p = (const u32x4*)(grad + (n * M + mcol) * 2);
      }
      x[r] = *p;
    }
  };
  auto store_rows = [&](int buf, const u32x4 (&x)[8]) {
    if (!isA && !isG) return;  // wave-uniform
    u32x4* row = lds + buf * BUF + lg * ROWU + (isA ? 0 : kGwCols);
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // column j of the 8 x 8 block: its 8 n
      const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
      u32x4 t;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        t[e] = __builtin_amdgcn_perm(x[2 * e + 1][j >> 1], x[2 * e][j >> 1], sel);
      row[gw_slot(lu * 8 + j)] = t;
    }
  };
  gw_f32x4 acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = gw_f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = wave & 1, wk = wave >> 1;
  auto multiply = [&](int buf) {
    const u32x4* base = lds + buf * BUF;
#pragma unroll
    for (int h = 0; h < kGwStep / 32; ++h) {  // one 16x16x32 k-step: n groups 4h .. 4h + 3
      const u32x4* row = base + (4 * h + (lane >> 4)) * ROWU;
      u32x4 b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = row[gw_slot(wk * 64 + j * 16 + (lane & 15))];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const u32x4 a = row[kGwCols + gw_slot(wm * 16 * MT + i * 16 + (lane & 15))];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = gw_mfma<F16>(a, b[j], acc[i][j]);
      }
    }
  };
  if (s0 < s1) {
    int32_t sv[8];
    u32x4 x[8];
    load_src(s0, sv);
    load_rows(s0, sv, x);
    load_src(s0 + 1, sv);
    store_rows(0, x);
    __syncthreads();
    for (int64_t st = s0; st < s1; ++st) {
      const int buf = (int)(st - s0) & 1;
      load_rows(st + 1, sv, x);  // zeros past the range
      load_src(st + 2, sv);
      multiply(buf);
      __builtin_amdgcn_sched_barrier(0);  // the MFMAs issue before the stores wait
      store_rows(buf ^ 1, x);
      __syncthreads();
    }
  }
  // partial sums [split][M][K]
  float* out = part + (int64_t)split * M * K;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm * 16 * MT + i * 16 + (lane >> 4) * 4 + e;
        const int col = k0 + wk * 64 + j * 16 + (lane & 15);
        if (m < M && col < K) out[(int64_t)m * K + col] = acc[i][j][e];
      }
}

// gw = the partial sums added in split order, rounded once.  n4: groups of 4
// results (K is a multiple of 8).
template <bool F16>
__global__ __launch_bounds__(256) void weight_reduce_kernel(const gw_f32x4* __restrict__ part,
                                                           int64_t n4, int nsplit,
                                                           u32x2* __restrict__ gw) {
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i >= n4) return;
  gw_f32x4 s = {0.f, 0.f, 0.f, 0.f};
  constexpr int B = 8;
  int k = 0;
  for (; k + B <= nsplit; k += B) {
    gw_f32x4 v[B];
#pragma unroll
    for (int j = 0; j < B; ++j) v[j] = part[(int64_t)(k + j) * n4 + i];
#pragma unroll
    for (int j = 0; j < B; ++j) s += v[j];
  }
  for (; k < nsplit; ++k) s += part[(int64_t)k * n4 + i];
  typedef __bf16 b4 __attribute__((ext_vector_type(4)));
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  if constexpr (F16)
    gw[i] = __builtin_bit_cast(u32x2, __builtin_convertvector(s, h4));
  else
    gw[i] = __builtin_bit_cast(u32x2, __builtin_convertvector(s, b4));
}

struct GwPlan {
  int mt, nkt, nmt, nsplit;
  int64_t steps;
};

GwPlan gw_plan(int64_t NR, int64_t K, int64_t M) {
  GwPlan p;
  p.mt = M >= 256 ? 8 : (int)((M + 63) / 64) * 2;
  p.nkt = (int)((K + kGwCols - 1) / kGwCols);
  p.nmt = (int)((M + 32 * p.mt - 1) / (32 * p.mt));
  p.steps = (NR + kGwStep - 1) / kGwStep;
  // One block per CU; a row range of at least 4 steps, so that the partial
  // sums (written and read once per range) stay a small part of the rows read.
  int64_t sp = kGwTarget / ((int64_t)p.nkt * p.nmt);
  if (sp > p.steps / 4) sp = p.steps / 4;
  p.nsplit = sp < 1 ? 1 : (int)sp;
  return p;
}

}  // namespace

bool weight_grad_apply(int dtype, int64_t NR, int64_t C, int64_t P, int64_t M, const void* payload,
                       const void* grad, const void* gw) {
  return (dtype == kBF16 || dtype == kF16) && P >= 8 && P % 8 == 0 && M >= 8 && M % 8 == 0 &&
         C >= 1 && C * P < ((int64_t)1 << 24) && M < ((int64_t)1 << 24) && NR >= 1 &&
         (((uintptr_t)payload | (uintptr_t)grad) & 15) == 0 && ((uintptr_t)gw & 7) == 0;
}

size_t weight_grad_floats(int64_t NR, int64_t C, int64_t P, int64_t M) {
  return (size_t)gw_plan(NR, C * P, M).nsplit * (size_t)(M * C * P);
}

hipError_t weight_grad(const void* payload, const int32_t* src, const void* grad, int dtype,
                       int64_t NR, int64_t C, int64_t P, int64_t M, float* part, void* gw,
                       hipStream_t s) {
  if (!weight_grad_apply(dtype, NR, C, P, M, payload, grad, gw)) return hipErrorInvalidValue;
  const int64_t K = C * P;
  const GwPlan p = gw_plan(NR, K, M);
  const int64_t nlogical = (int64_t)p.nkt * p.nmt * p.nsplit;
  if (nlogical > INT32_MAX / 2) return hipErrorInvalidValue;
  const unsigned grid = xcd_grid(nlogical, 1, (int64_t)1 << 31);
  const FastDiv byP = make_fastdiv((uint32_t)P);
  auto go = [&](auto f16) {
    constexpr bool F16 = decltype(f16)::value;
#define REM_GW(MT)                                                                            \
  weight_grad_kernel<F16, MT><<<grid, kGwThreads, 0, s>>>(                                    \
      (const unsigned char*)payload, src, (const unsigned char*)grad, NR, (int)C, (int)P, byP, \
      (int)M, NR * C, p.nkt, p.nmt, nlogical, p.steps, p.nsplit, part)
    switch (p.mt) {
      case 2: REM_GW(2); break;
      case 4: REM_GW(4); break;
      case 6: REM_GW(6); break;
      default: REM_GW(8); break;
    }
#undef REM_GW
    const int64_t n4 = M * K / 4;
    weight_reduce_kernel<F16><<<(unsigned)((n4 + 255) / 256), 256, 0, s>>>(
        (const gw_f32x4*)part, n4, p.nsplit, (u32x2*)gw);
  };
  if (dtype == kF16)
    go(std::true_type{});
  else
    go(std::false_type{});
  return hipGetLastError();
}

}  // namespace rem
