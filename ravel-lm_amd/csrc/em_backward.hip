// Backward of the latest-k gather (gfx950).
//
// The reference has no custom backward on its generic path: autograd turns the
// index_select of ravel_lm/ravel_memory.py:173-174 into an index_add_ into the
// payload gradient; its GPU arms use float atomics (triton_latest1.py:71-83,
// :132-142).  Here:
//   chain   read == write without write_mask.  Record s is read by exactly its
//           successors in its stream: the reader whose slot 0 is s, that
//           reader's slot-0 successor, and so on.  next[src[r,0]] = r builds the
//           chain without collisions, and each gradient row is summed in slot
//           order j = 0..k-1: deterministic, no atomics.
//   sorted  separate reads or masked writes: the slots' source ids are sorted
//           and each source's slots summed in slot order by the segmented-sum
//           kernels (em_api.hip, latest_k_bwd_sorted): deterministic too.

#include <type_traits>

#include "em_common.h"
#include "em_elem.h"

namespace rem {

namespace {

__global__ __launch_bounds__(256) void fill_i32_kernel(int32_t* __restrict__ p, int64_t n,
                                                      int32_t v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ __launch_bounds__(256) void next_chain_kernel(const int32_t* __restrict__ src,
                                                        int64_t N, int k,
                                                        int32_t* __restrict__ next) {
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < N;
       r += (int64_t)gridDim.x * blockDim.x) {
    const int32_t s0 = src[r * k];
    if (s0 >= 0 && s0 < N) next[s0] = (int32_t)r;
  }
}

// One thread per (record, unit of 4..16 bytes of its row), ILP records a thread:
// it first follows the record's chain (KU steps, the same words for all lanes
// of a row), then has all of its gradient rows in flight before the first sum.
// Bound by the rows: each is read once, at random, and every sum written once.
// At N = 2.1M records of 128 bytes, k = 1 (37 % of them read) the launch takes
// 62 us (5.9 TB/s), where the form with one thread per element took 282; at
// 262k rows of 64 bytes, k = 4, 13.3 us against 27.9.  Longer chains than KU
// run in rounds.
template <int DT, typename V, int KU, int ILP>
__global__ __launch_bounds__(256) void chain_grad_kernel(const int32_t* __restrict__ next,
                                                        const V* __restrict__ gv, int64_t N,
                                                        int upr, int rpb, int k,
                                                        V* __restrict__ gp) {
  using E = Elem<DT>;
  using S = typename E::store_t;
  using Acc = typename E::acc_t;
  constexpr int EPU = (int)(sizeof(V) / sizeof(S));  // elements of a unit
  const int r0 = threadIdx.x / upr;
  if (r0 >= rpb) return;  // 256 / upr whole rows a block
  const int64_t s0 = (int64_t)blockIdx.x * rpb * ILP + r0;
  for (int v = threadIdx.x - r0 * upr; v < upr; v += 256) {  // one turn unless upr > 256
    int32_t p[ILP];
    Acc acc[ILP][EPU];
#pragma unroll
    for (int i = 0; i < ILP; ++i) {
      const int64_t s = s0 + (int64_t)i * rpb;
      p[i] = s < N ? next[s] : -1;
#pragma unroll
      for (int e = 0; e < EPU; ++e) acc[i][e] = Acc(0);
    }
    for (int j0 = 0; j0 < k; j0 += KU) {
      int32_t q[KU][ILP];
#pragma unroll
      for (int j = 0; j < KU; ++j) {
#pragma unroll
        for (int i = 0; i < ILP; ++i) {
          const bool on = j0 + j < k && p[i] >= 0 && p[i] < N;
          q[j][i] = on ? p[i] : -1;
          if (KU > 1 || k > 1) p[i] = on ? next[p[i]] : -1;
        }
      }
      V x[KU][ILP];
#pragma unroll
      for (int j = 0; j < KU; ++j) {
#pragma unroll
        for (int i = 0; i < ILP; ++i) {
          x[j][i] = V{};
          if (q[j][i] >= 0)
            x[j][i] = __builtin_nontemporal_load(&gv[((int64_t)q[j][i] * k + j0 + j) * upr + v]);
        }
      }
#pragma unroll
      for (int j = 0; j < KU; ++j) {
#pragma unroll
        for (int i = 0; i < ILP; ++i) {
          union { V u; S e[EPU]; } c;
          c.u = x[j][i];
#pragma unroll
          for (int e = 0; e < EPU; ++e) acc[i][e] += E::load(c.e[e]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < ILP; ++i) {
      const int64_t s = s0 + (int64_t)i * rpb;
      union { V u; S e[EPU]; } c;
#pragma unroll
      for (int e = 0; e < EPU; ++e) c.e[e] = E::store(acc[i][e]);
      if (s < N) __builtin_nontemporal_store(c.u, &gp[s * upr + v]);
    }
  }
}

template <int DT, typename V>
hipError_t chain_rows(const int32_t* next, const void* gv, int64_t N, int64_t upr, int k, void* gp,
                      hipStream_t s) {
  if (upr > INT32_MAX) return hipErrorInvalidValue;
  const int rpb = upr < 256 ? (int)(256 / upr) : 1;
#define REM_CH(KU, ILP)                                                                       \
  do {                                                                                       \
    const int64_t blocks = (N + (int64_t)rpb * ILP - 1) / ((int64_t)rpb * ILP);              \
    chain_grad_kernel<DT, V, KU, ILP><<<(unsigned)blocks, 256, 0, s>>>(                      \
        next, (const V*)gv, N, (int)upr, rpb, k, (V*)gp);                                    \
  } while (0)
  if (k == 1)
    REM_CH(1, 4);
  else if (k == 2)
    REM_CH(2, 2);
  else
    REM_CH(4, 2);
#undef REM_CH
  return hipGetLastError();
}

template <int DT>
hipError_t chain_t(const int32_t* src, const void* gv, int64_t N, int64_t D, int k, int32_t* next,
                   void* gp, hipStream_t s) {
  using S = typename Elem<DT>::store_t;
  fill_i32_kernel<<<grid_for(N, 256), 256, 0, s>>>(next, N, -1);
  next_chain_kernel<<<grid_for(N, 256), 256, 0, s>>>(src, N, k, next);
  // the widest unit that the row size and both base addresses allow
  const int64_t row = D * (int64_t)sizeof(S);
  const uintptr_t align = (uintptr_t)gv | (uintptr_t)gp | (uintptr_t)row;
  if ((align & 15) == 0) return chain_rows<DT, u32x4>(next, gv, N, row / 16, k, gp, s);
  if ((align & 7) == 0) return chain_rows<DT, u32x2>(next, gv, N, row / 8, k, gp, s);
  if (sizeof(S) <= 4 && (align & 3) == 0)
    return chain_rows<DT, typename std::conditional<sizeof(S) <= 4, uint32_t, S>::type>(
        next, gv, N, row / 4, k, gp, s);
  return chain_rows<DT, S>(next, gv, N, D, k, gp, s);
}

}  // namespace

hipError_t latest_k_bwd_chain(const int32_t* src, const void* grad_values, int dtype, int64_t N,
                              int64_t D, int k, int32_t* next, void* grad_payload, hipStream_t s) {
  switch (dtype) {
    case kF32: return chain_t<kF32>(src, grad_values, N, D, k, next, grad_payload, s);
    case kF64: return chain_t<kF64>(src, grad_values, N, D, k, next, grad_payload, s);
    case kBF16: return chain_t<kBF16>(src, grad_values, N, D, k, next, grad_payload, s);
    case kF16: return chain_t<kF16>(src, grad_values, N, D, k, next, grad_payload, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace rem
