// The segmented walk of a sorted tape, any row width, in either direction
// (gfx950): one kernel template behind
//   the backward of the segmented sum and of the latest-k lookup, one or both
//   in one pass (REV: sorted positions in descending order), and
//   the forward segmented sum (FWD).
//
// Replaces, of the reference, the autograd of ravel_lm/ravel_memory.py:173-175
// and :216-241 (index_add_ of the slots' gradients; the cumsum's backward), and
// its cumsum-minus-prefix forward.
//
// A sorted tape lists every (b, c, a) stream's items in time order.  With reads
// at the write addresses and no mask, item p is a record, read and write of one
// time (a consumer, then a loader, in the terms below).  Otherwise a segment has 2T items a << tbits | 2t + kind, kind 0 the read
// and 1 the write of time t, so a read sorts after the writes before its time
// and before the write of its own.
//
// REV.  Walking a run backwards, keep S = sum of grad_sum over the reads passed
// and P[j] = sum of grad_values[r, j'] over the reads r passed whose slot j' is
// now the j-th latest write ahead.  A read adds its rows (S += gs, P[j] +=
// gv[j]); a write takes S + P[0] as its gradient and shifts P down by one.
// FWD.  A write adds its payload row to S, a read takes S.
// So in both directions a "loader" item adds rows, a "consumer" item takes the
// sum, and every row is read, and every result written, once.  A loader that no
// later consumer of its run needs is not loaded, and of a read's k rows only
// those of the writes that exist (the count is taken on the sorted keys).
//
// Work: a block takes a part of up to 1024 items of one segment (smaller parts
// where the tape is too short to fill the chip), a walker of G lanes (one unit of
// UB bytes each) a contiguous range of them.
//   1. code words: one 32-bit word per item (time, run start, counts, flags);
//   2. every walker sums from the last run start of its range to its end (the
//      state that leaves the range);
//   3. the states are composed over the walkers of a wave (shuffles), the waves
//      (LDS) and, where a run crosses parts, the earlier parts (published words,
//      read newest first in a fixed order): (f1, m1, S1, P1) then (f2, m2, S2,
//      P2) = f2 ? second : (f1, m1 + m2, S1 + S2, P2[j] + P1[j + m2]), f "holds a
//      run start", m consumers passed;
//   4. every walker walks its range again with the state that enters it.
// Sums are formed in an order that does not depend on timing; they accumulate in
// fp32 for 16-bit rows and fp64 otherwise and are rounded once.
//
// Measured (launch alone): joint backward of 2.1M records, separate reads, k = 4,
// bf16 D = 64: 300 us, where the sort of N k source ids as one segment, its run
// totals, the reads' atomics, the walk and the addition took 5.5 ms; of 262k
// records, reads = writes, k = 8, fp32 D = 32: 75 us (4.5 TB/s) against 140; the
// sum's backward of 4.2M records, bf16 D = 64: 161 us (5.0 TB/s of random rows)
// against 221 for the walker that branches.
//
// Loads and stores go through buffer descriptors of the segment's rows: a set
// bit 31 of the offset lies past every range, which turns a skipped load into
// zeros and a skipped store into nothing, so the walk has no branches.
#pragma once

#include <type_traits>

#include "em_common.h"
#include "em_elem.h"
#include "em_pub.h"

namespace rem {

// One launch, filled by tape_walk() (em_walk.hip).
struct WalkArgs {
  const void* keys;      // sorted keys [nseg][L], 32 or 64 bits
  int wide;              // 64-bit keys
  int same;              // items are records, else reads and writes
  int tbits;             // bits of the item index in a key
  int64_t nseg, T, L, C;
  int part;              // items per part (256, 512 or 1024)
  int64_t nparts;
  int G, gtot, ncb;      // lanes per walker, units per row, column blocks
  const void* sum_in;    // rows [B,T,C,D] or null
  const void* val_in;    // rows [B,T,C,k,D] or null
  int k;
  void* out;             // rows [B,T,C,D]
  uint8_t* omask;        // FWD: [B,T,C] "some earlier write"
  uint64_t* words;       // published states, zero on entry (nparts > 1)
  uint64_t* tickets;     // [ncb][nseg], zero on entry (nparts > 1)
  uint32_t* err;
};

constexpr int kTwThreads = 256;
constexpr int kTwWaves = kTwThreads / kWave;
constexpr int kTwMaxPart = 1024;
constexpr int kTwAhead = 9;        // items past the part that a block keeps
constexpr int kTwColBytes = 512;   // accumulators of one state component of a block

// Code words: the time in bits 0..23 (the 24-bit multiplies ignore the rest), the
// rows to load of a read in bits 24..27.
constexpr uint32_t kTwTime = (1u << 24) - 1u;
constexpr int kTwCount = 24;
constexpr uint32_t kTwStart = 1u << 28, kTwLoader = 1u << 29, kTwNoStore = 1u << 30,
                   kTwNoLoad = 1u << 31;
constexpr uint32_t kTwPad = kTwNoStore | kTwNoLoad;
constexpr int kTwRsrc3 = 0x00020000;  // gfx9 buffer descriptor word 3 (raw access)
constexpr int kTwStream = 2;          // nontemporal bit of buffer loads and stores

template <int UB>
struct BufUnit;
template <>
struct BufUnit<16> {
  using T = u32x4;
  template <int AUX>
  static __device__ __forceinline__ T load(__amdgpu_buffer_rsrc_t r, uint32_t o) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, AUX);
  }
  static __device__ __forceinline__ void store(T v, __amdgpu_buffer_rsrc_t r, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b128(v, r, o, 0, kTwStream);
  }
};
template <>
struct BufUnit<8> {
  using T = u32x2;
  template <int AUX>
  static __device__ __forceinline__ T load(__amdgpu_buffer_rsrc_t r, uint32_t o) {
    return __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, AUX);
  }
  static __device__ __forceinline__ void store(T v, __amdgpu_buffer_rsrc_t r, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b64(v, r, o, 0, kTwStream);
  }
};
template <>
struct BufUnit<4> {
  using T = uint32_t;
  template <int AUX>
  static __device__ __forceinline__ T load(__amdgpu_buffer_rsrc_t r, uint32_t o) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, AUX);
  }
  static __device__ __forceinline__ void store(T v, __amdgpu_buffer_rsrc_t r, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b32(v, r, o, 0, 0);
  }
};
template <>
struct BufUnit<2> {
  using T = uint16_t;
  template <int AUX>
  static __device__ __forceinline__ T load(__amdgpu_buffer_rsrc_t r, uint32_t o) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, o, 0, AUX);
  }
  static __device__ __forceinline__ void store(T v, __amdgpu_buffer_rsrc_t r, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b16(v, r, o, 0, 0);
  }
};

// CPU accumulators, rounded once, as one unit (16-bit values convert in pairs).
template <int DT, typename V, int CPU>
__device__ __forceinline__ V walk_pack(const typename Elem<DT>::acc_t* t) {
  using X = typename Elem<DT>::store_t;
  if constexpr (sizeof(X) == 2 && CPU > 1) {
    union { V u; uint32_t w[CPU / 2]; } o;
#pragma unroll
    for (int e = 0; e < CPU / 2; ++e) o.w[e] = Elem<DT>::store2(t[2 * e], t[2 * e + 1]);
    return o.u;
  } else {
    union { V u; X e[CPU]; } o;
#pragma unroll
    for (int e = 0; e < CPU; ++e) o.e[e] = Elem<DT>::store(t[e]);
    return o.u;
  }
}

template <int DT, int UB, int KS, bool FWD>
__global__ __launch_bounds__(kTwThreads) void tape_walk_kernel(const WalkArgs a) {
  using E = Elem<DT>;
  using X = typename E::store_t;
  using Acc = typename E::acc_t;
  using BU = BufUnit<UB>;
  using V = typename BU::T;
  constexpr int CPU = UB / (int)sizeof(X);  // columns per lane
  constexpr int MAXC = kTwColBytes / (int)sizeof(Acc);
  constexpr int NC = KS + 1;                // state components: S, P[0..KS-1]
  constexpr int KR = KS > 0 ? KS : 1;
  // items in flight: every loader has up to 1 + KS rows
  constexpr int RB = KS == 0 ? 16 : KS == 1 ? 8 : KS <= 4 ? 4 : 2;
  static_assert(!FWD || KS == 0, "the forward walk sums only");
  static_assert((KS & (KS - 1)) == 0 && KS <= 8, "shifts by powers of two");
  __shared__ uint64_t kk[kTwMaxPart + 1 + kTwAhead];  // kk[i + 1]: key of walk item i
  __shared__ __align__(16) uint32_t cw[kTwMaxPart + 16];
  __shared__ uint64_t sbits[kTwMaxPart / 64 + 1];      // run starts
  __shared__ Acc agg[(kTwWaves + 1) * NC * MAXC];     // [wave, then carry][component][column]
  __shared__ int wf[kTwWaves], wm[kTwWaves], wc[kTwWaves], wb[kTwWaves];
  __shared__ uint8_t hm[FWD ? kTwMaxPart : 4];
  __shared__ uint32_t s_part;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int64_t seg = blockIdx.x / a.nparts;
  const int cb = blockIdx.y;
  int64_t q = 0;
  if (a.nparts > 1) {  // parts start in ticket order: a part waits on running blocks only
    if (tid == 0)
      s_part = (uint32_t)atomicAdd((unsigned long long*)&a.tickets[cb * a.nseg + seg], 1ull);
    __syncthreads();
    q = s_part;
    if (q >= a.nparts) return;  // uniform
  }
  const int64_t b = seg / a.C, c = seg - b * a.C;
  const int64_t p0 = q * a.part;
  const int n = (int)((a.L - p0) < a.part ? (a.L - p0) : a.part);
  const int tb = a.tbits;
  const uint64_t imask = (((uint64_t)1) << tb) - 1;
  auto key_at = [&](int64_t wi) -> uint64_t {  // walk item wi of the segment
    const int64_t p = seg * a.L + (FWD ? wi : a.L - 1 - wi);
    return a.wide ? ((const uint64_t*)a.keys)[p] : (uint64_t)((const uint32_t*)a.keys)[p];
  };
  for (int i = tid; i < n + 1 + kTwAhead; i += kTwThreads) {
    const int64_t wi = p0 - 1 + i;
    kk[i] = wi >= 0 && wi < a.L ? key_at(wi) : 0;
  }
  __syncthreads();
  // whether a run ends after walk item p0 + i (i = -1: before the part)
  auto ends = [&](int i) -> bool {
    const int64_t wi = p0 + i;
    return wi < 0 || wi + 1 >= a.L || (kk[i + 1] >> tb) != (kk[i + 2] >> tb);
  };
  const bool same = a.same != 0;
  auto consumes = [&](uint64_t key) -> bool { return same || ((key & 1) != 0) != FWD; };
  const bool open = !ends(n - 1);  // the last run goes on in the next part
  // Consumers of that run past the part, up to kc (what a count can use).
  const int kc = KS > 0 ? a.k : 1;
  int ext = 0;
  if (open) {  // uniform
    bool done = false;
    for (int i = n; i < n + kTwAhead && !done; ++i) {
      ext += consumes(kk[i + 1]) ? 1 : 0;
      done = ext >= kc || p0 + i + 1 >= a.L ||
             (i + 1 < n + kTwAhead && (kk[i + 1] >> tb) != (kk[i + 2] >> tb));
    }
    // a long stretch without a consumer: 1024 items a round
    const uint64_t ra = kk[n] >> tb;
    for (int64_t w0 = p0 + n + kTwAhead; !done && w0 < a.L; w0 += 4 * kTwThreads) {
      bool other = false;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t wi = w0 + j * kTwThreads + tid;
        const uint64_t key = wi < a.L ? key_at(wi) : 0;
        const bool in = wi < a.L && (key >> tb) == ra;
        other = other || !in;
        ext += __syncthreads_count(in && consumes(key));
      }
      done = ext >= kc || __syncthreads_or(other);
    }
    ext = ext < kc ? ext : kc;
  }
  // 1. code words: thread tid has items [tid ipt, (tid + 1) ipt); a segmented
  // suffix scan over the threads counts the consumers after each item in its run
  {
    const int ipt = a.part / kTwThreads;
    int cn[4], op[4];
    int cs = 0, bs = 0;
#pragma unroll
    for (int j = 3; j >= 0; --j) {
      const int i = tid * ipt + j;
      cn[j] = op[j] = 0;
      if (j < ipt && i < n) {
        if (ends(i)) cs = 0, bs = 1;
        cn[j] = cs;
        op[j] = !bs;
        cs += consumes(kk[i + 1]) ? 1 : 0;
      }
    }
    int ic = cs, ib = bs;  // inclusive over the lanes from this one up
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int oc = __shfl_down(ic, o, kWave), ob = __shfl_down(ib, o, kWave);
      if (lane + o < kWave && !ib) ic += oc, ib = ob;
    }
    if (lane == 0) wc[wave] = ic, wb[wave] = ib;
    int xc = __shfl_down(ic, 1, kWave), xb = __shfl_down(ib, 1, kWave);
    if (lane == kWave - 1) xc = xb = 0;
    __syncthreads();
    if (!xb) {
      int w2 = wave + 1;
      for (; w2 < kTwWaves; ++w2) {
        xc += wc[w2];
        if (wb[w2]) break;
      }
      if (w2 == kTwWaves) xc += ext;
    }
    for (int j = 0; j < ipt; ++j) {
      const int i = tid * ipt + j;
      uint32_t code = kTwPad;
      if (i < n) {
        const uint64_t key = kk[i + 1];
        const uint32_t idx = (uint32_t)(key & imask);
        int cnt = cn[j] + (op[j] ? xc : 0);
        cnt = cnt < kc ? cnt : kc;
        const bool cons = consumes(key), load = same || !cons;
        if (!load) cnt = 0;
        code = (same ? idx : idx >> 1) | ((uint32_t)cnt << kTwCount) |
               (ends(i - 1) ? kTwStart : 0u) | (load ? kTwLoader : 0u) |
               (cons ? 0u : kTwNoStore) | (cnt > 0 ? 0u : kTwNoLoad);
      }
      cw[i] = code;
    }
    if (tid < 16) cw[a.part + tid] = kTwPad;
  }
  __syncthreads();
  for (int i = wave; i * 64 < a.part; i += kTwWaves) {
    const uint64_t m = __ballot((cw[i * 64 + lane] & kTwStart) != 0);
    if (lane == 0) sbits[i] = m;
  }
  __syncthreads();
  const int nr = (n + RB - 1) & ~(RB - 1);
  const int G = a.G;
  const int wpw = kWave / G;  // walkers per wave
  const int wi = lane / G, v = lane - (lane / G) * G;
  const int NW = wpw * kTwWaves;
  const int w = wave * wpw + wi;
  const int len = (((nr + NW - 1) / NW) + RB - 1) & ~(RB - 1);
  const bool on = wi < wpw;
  const int rs = on && w * len < nr ? w * len : nr;
  const int re = (rs + len) < nr ? (rs + len) : nr;
  const int vcol = cb * G + v;
  const uint32_t vo = (uint32_t)vcol * UB;
  const uint32_t vbad = on && vcol < a.gtot ? 0u : 0x80000000u;
  const uint32_t row = (uint32_t)a.gtot * UB;
  const uint32_t tstride = (uint32_t)a.C * row, vstride = tstride * (uint32_t)a.k;
  const int64_t rec0 = b * a.T * a.C + c;
  const uint32_t ext_row = (uint32_t)((a.T - 1) * tstride + row);
  const __amdgpu_buffer_rsrc_t srs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const unsigned char*)a.sum_in + (a.sum_in ? rec0 * row : 0)), 0,
      a.sum_in ? (int)ext_row : 0, kTwRsrc3);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const unsigned char*)a.val_in + (a.val_in ? rec0 * a.k * (int64_t)row : 0)), 0,
      KS > 0 && a.val_in ? (int)((a.T - 1) * vstride + row * (uint32_t)a.k) : 0, kTwRsrc3);
  const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((unsigned char*)a.out + rec0 * row), 0, (int)ext_row, kTwRsrc3);
  Acc S[CPU], P[KR][CPU];
  int mc = 0;  // REV: consumers passed in the run; FWD: loaders passed
  auto walk = [&](int from, int to, auto store_tag) {
    constexpr bool STORE = decltype(store_tag)::value;
    constexpr int AUX = STORE ? kTwStream : 0;
    for (int i0 = from & ~(RB - 1); i0 < to; i0 += RB) {
      uint32_t k4[RB];
      if constexpr (RB >= 4) {
#pragma unroll
        for (int m = 0; m < RB / 4; ++m) {
          const u32x4 x = *(const u32x4*)&cw[i0 + 4 * m];
          k4[4 * m] = x.x, k4[4 * m + 1] = x.y, k4[4 * m + 2] = x.z, k4[4 * m + 3] = x.w;
        }
      } else {
        const u32x2 x = *(const u32x2*)&cw[i0];
        k4[0] = x.x, k4[1] = x.y;
      }
#pragma unroll
      for (int m = 0; m < RB; ++m)
        if (i0 + m < from || i0 + m >= to) k4[m] = kTwPad;
      V xs[RB], xv[RB][KR];
#pragma unroll
      for (int m = 0; m < RB; ++m) {
        xs[m] = BU::template load<AUX>(
            srs, (__umul24(k4[m], tstride) + vo) | (k4[m] & kTwNoLoad) | vbad);
        if constexpr (KS > 0) {
          const uint32_t cnt = (k4[m] >> kTwCount) & 15u;
          const uint32_t o = __umul24(k4[m], vstride) + vo;
#pragma unroll
          for (int j = 0; j < KS; ++j)
            xv[m][j] = BU::template load<AUX>(
                vrs, (o + (uint32_t)j * row) | ((uint32_t)j < cnt ? vbad : 0x80000000u));
        }
      }
#pragma unroll
      for (int m = 0; m < RB; ++m) {
        const uint32_t k = k4[m];
        const bool st = k & kTwStart, cons = !(k & kTwNoStore);
#pragma unroll
        for (int e = 0; e < CPU; ++e) S[e] = st ? Acc(0) : S[e];
        mc = st ? 0 : mc;
        if constexpr (KS > 0) {
#pragma unroll
          for (int j = 0; j < KS; ++j)
#pragma unroll
            for (int e = 0; e < CPU; ++e) P[j][e] = st ? Acc(0) : P[j][e];
        }
        if (STORE) {
          Acc t[CPU];
#pragma unroll
          for (int e = 0; e < CPU; ++e) {
            t[e] = S[e];
            if constexpr (KS > 0) t[e] += P[0][e];
          }
          BU::store(walk_pack<DT, V, CPU>(t), ors, (__umul24(k, tstride) + vo) | ((k & kTwNoStore) << 1) | vbad);
          if (FWD && v == 0 && cons) hm[i0 + m] = mc > 0 ? 1 : 0;
        }
        if constexpr (KS > 0) {
#pragma unroll
          for (int j = 0; j < KS; ++j)
#pragma unroll
            for (int e = 0; e < CPU; ++e) {
              const Acc up = j + 1 < KS ? P[j + 1 < KS ? j + 1 : 0][e] : Acc(0);
              P[j][e] = cons ? up : P[j][e];
            }
        }
        mc += FWD ? ((k & kTwLoader) ? 1 : 0) : (cons ? 1 : 0);
        union { V u; X e[CPU]; } x;
        x.u = xs[m];
#pragma unroll
        for (int e = 0; e < CPU; ++e) S[e] += E::load(x.e[e]);
        if constexpr (KS > 0) {
#pragma unroll
          for (int j = 0; j < KS; ++j) {
            x.u = xv[m][j];
#pragma unroll
            for (int e = 0; e < CPU; ++e) P[j][e] += E::load(x.e[e]);
          }
        }
      }
    }
  };
  // 2. the state leaving the walker's range
  int last = -1;  // its last run start
  if (rs < re) {
    for (int word = (re - 1) >> 6; word >= rs >> 6 && last < 0; --word) {
      uint64_t m = sbits[word];
      const int lo = word << 6;
      if (re - lo < 64) m &= (1ull << (re - lo)) - 1ull;
      if (rs > lo) m &= ~0ull << (rs - lo);
      if (m) last = lo + 63 - __builtin_clzll(m);
    }
  }
#pragma unroll
  for (int e = 0; e < CPU; ++e) S[e] = Acc(0);
#pragma unroll
  for (int j = 0; j < KR; ++j)
#pragma unroll
    for (int e = 0; e < CPU; ++e) P[j][e] = Acc(0);
  walk(last >= 0 ? last : rs, re, std::false_type{});
  int f = last >= 0 ? 1 : 0;
  mc = mc < 15 ? mc : 15;
  // 3. inclusive composition over the wave's walkers
  for (int d = 1; d < wpw; d <<= 1) {
    const int from = lane - d * G;
    const bool take = from >= 0 && wi >= d && !f;
    const int src = from >= 0 ? from : lane;
    const int pf = __shfl(f, src, kWave), pm = __shfl(mc, src, kWave);
#pragma unroll
    for (int e = 0; e < CPU; ++e) {
      const Acc t = __shfl(S[e], src, kWave);
      S[e] = take ? S[e] + t : S[e];
    }
    if constexpr (KS > 0) {
#pragma unroll
      for (int e = 0; e < CPU; ++e) {
        Acc t[KR];
#pragma unroll
        for (int j = 0; j < KS; ++j) t[j] = __shfl(P[j][e], src, kWave);
#pragma unroll
        for (int s2 = 1; s2 < KS; s2 <<= 1)
#pragma unroll
          for (int j = 0; j < KS; ++j) {
            const Acc up = j + s2 < KS ? t[j + s2 < KS ? j + s2 : 0] : Acc(0);
            t[j] = (mc & s2) ? up : t[j];
          }
#pragma unroll
        for (int j = 0; j < KS; ++j)
          P[j][e] = take && mc < KS ? P[j][e] + t[j] : P[j][e];
      }
    }
    if (take) {
      mc = mc + pm < 15 ? mc + pm : 15;
      f = pf;
    }
  }
  const int cols = G * CPU;
  if (on && wi == wpw - 1) {
#pragma unroll
    for (int e = 0; e < CPU; ++e) {
      agg[(wave * NC) * MAXC + v * CPU + e] = S[e];
      if constexpr (KS > 0) {
#pragma unroll
        for (int j = 0; j < KS; ++j) agg[(wave * NC + 1 + j) * MAXC + v * CPU + e] = P[j][e];
      }
    }
    if (v == 0) wf[wave] = f, wm[wave] = mc;
  }
  // exclusive: the state of the wave's walkers before this one
  {
    const int src = lane >= G ? lane - G : lane;
    const bool any = wi > 0;
#pragma unroll
    for (int e = 0; e < CPU; ++e) {
      const Acc t = __shfl(S[e], src, kWave);
      S[e] = any ? t : Acc(0);
    }
    if constexpr (KS > 0) {
#pragma unroll
      for (int j = 0; j < KS; ++j)
#pragma unroll
        for (int e = 0; e < CPU; ++e) {
          const Acc t = __shfl(P[j][e], src, kWave);
          P[j][e] = any ? t : Acc(0);
        }
    }
    const int pf = __shfl(f, src, kWave), pm = __shfl(mc, src, kWave);
    f = any ? pf : 0;
    mc = any ? pm : 0;
  }
  __syncthreads();
  // the block's state, published where the next part's first run needs it; then
  // the state of the earlier parts, where this part's first run needs it
  constexpr int PW = Pub<Acc>::W;
  const int64_t pstride = (int64_t)NC * cols * PW;
  uint64_t* mine = a.words + ((seg * a.nparts + q) * a.ncb + cb) * pstride;
  const bool joined = q > 0 && !(cw[0] & kTwStart);  // uniform
  if (tid < cols) {
    if (open) {
      Acc bs = Acc(0), bp[KR];
      int bm = 0, bf = 0;
#pragma unroll
      for (int j = 0; j < KR; ++j) bp[j] = Acc(0);
      for (int w2 = kTwWaves - 1; w2 >= 0 && !bf; --w2) {
        bs += agg[(w2 * NC) * MAXC + tid];
        if constexpr (KS > 0) {
#pragma unroll
          for (int j = 0; j < KS; ++j)
            if (j + bm < KS) bp[j] += agg[(w2 * NC + 1 + j + bm) * MAXC + tid];
        }
        bm = bm + wm[w2] < 15 ? bm + wm[w2] : 15;
        bf = wf[w2];
      }
      const uint32_t flag = 1u | ((uint32_t)bf << 1) | ((uint32_t)bm << 4);
      Pub<Acc>::put(mine + (int64_t)tid * PW, bs, flag);
      if constexpr (KS > 0) {
#pragma unroll
        for (int j = 0; j < KS; ++j)
          Pub<Acc>::put(mine + ((int64_t)(1 + j) * cols + tid) * PW, bp[j], flag);
      }
    }
    Acc ls = Acc(0), lp[KR];
#pragma unroll
    for (int j = 0; j < KR; ++j) lp[j] = Acc(0);
    if (joined) {
      auto at = [&](int64_t part, int comp) {
        return a.words + ((seg * a.nparts + part) * a.ncb + cb) * pstride +
               ((int64_t)comp * cols + tid) * PW;
      };
      int64_t j0 = q - 1;
      int lm = 0;
      bool done = false;
      uint32_t fl = 0;
      if constexpr (KS > 0) {
        while (!done && j0 >= 0 && lm < KS) {  // parts whose P can still reach this one
          Acc val;
          if (!Pub<Acc>::get(at(j0, 0), &val, &fl)) {
            atomicOr(a.err, kStatusSumWait);
            done = true;
            break;
          }
          ls = val + ls;
          const uint32_t f0 = fl;
#pragma unroll
          for (int j = 0; j < KS; ++j) {
            if (j + lm < KS) {
              if (!Pub<Acc>::get(at(j0, 1 + j + lm), &val, &fl)) {
                atomicOr(a.err, kStatusSumWait);
                done = true;
              } else {
                lp[j] += val;
              }
            }
          }
          lm += (int)(f0 >> 4);
          done = done || (f0 & 2u);
          --j0;
        }
        if (!a.sum_in) done = true;  // only the slots' sums are wanted
      }
      constexpr int LB = 8;  // earlier parts read at once
      for (; j0 >= 0 && !done; j0 -= LB) {
        uint64_t wv[LB][PW];
#pragma unroll
        for (int i = 0; i < LB; ++i)
          if (j0 - i >= 0) Pub<Acc>::peek(at(j0 - i, 0), wv[i]);
#pragma unroll
        for (int i = 0; i < LB; ++i) {
          if (done || j0 - i < 0) break;
          Acc val;
          if (!Pub<Acc>::decode(wv[i], &val, &fl) && !Pub<Acc>::get(at(j0 - i, 0), &val, &fl)) {
            atomicOr(a.err, kStatusSumWait);
            done = true;
            break;
          }
          ls = val + ls;
          lm += (int)(fl >> 4);
          if (fl & 2u) done = true;
        }
      }
      if (FWD && tid == 0) wc[0] = lm;  // FWD: loaders before the part
    } else if (FWD && tid == 0) {
      wc[0] = 0;
    }
    agg[(kTwWaves * NC) * MAXC + tid] = ls;
    if constexpr (KS > 0) {
#pragma unroll
      for (int j = 0; j < KS; ++j) agg[(kTwWaves * NC + 1 + j) * MAXC + tid] = lp[j];
    }
  }
  __syncthreads();
  // the state entering this walker's range
  for (int w2 = wave - 1; w2 >= -1 && !f; --w2) {
    const int g = w2 >= 0 ? w2 : kTwWaves;  // the carry last
#pragma unroll
    for (int e = 0; e < CPU; ++e) {
      const int col = v * CPU + e;
      S[e] += agg[(g * NC) * MAXC + col];
      if constexpr (KS > 0) {
#pragma unroll
        for (int j = 0; j < KS; ++j)
          if (j + mc < KS) P[j][e] += agg[(g * NC + 1 + j + mc) * MAXC + col];
      }
    }
    if (w2 >= 0) {
      mc = mc + wm[w2] < 15 ? mc + wm[w2] : 15;
      f = wf[w2];
    } else if (FWD) {
      mc += wc[0];
    }
  }
  // 4. the walk
  walk(rs, re, std::true_type{});
  if constexpr (FWD) {
    __syncthreads();
    if (cb == 0) {
      const __amdgpu_buffer_rsrc_t mrs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(a.omask + rec0), 0, (int)((a.T - 1) * a.C + 1), kTwRsrc3);
      for (int i = tid; i < n; i += kTwThreads) {
        const uint32_t k = cw[i];
        if (!(k & kTwNoStore))
          __builtin_amdgcn_raw_buffer_store_b8(hm[i], mrs, (k & kTwTime) * (uint32_t)a.C, 0, 0);
      }
    }
  }
}

// The launches of one row type (em_walk_<type>.hip); ub 16, 8, 4 or 2.
hipError_t tape_walk_f32(const WalkArgs& a, int ub, int ks, bool fwd, hipStream_t s);
hipError_t tape_walk_f64(const WalkArgs& a, int ub, int ks, bool fwd, hipStream_t s);
hipError_t tape_walk_bf16(const WalkArgs& a, int ub, int ks, bool fwd, hipStream_t s);
hipError_t tape_walk_f16(const WalkArgs& a, int ub, int ks, bool fwd, hipStream_t s);

template <int DT, int UB>
hipError_t tape_walk_unit(const WalkArgs& a, int ks, bool fwd, hipStream_t s) {
  const dim3 grid((unsigned)(a.nseg * a.nparts), (unsigned)a.ncb);
#define REM_TW(K, F) tape_walk_kernel<DT, UB, K, F><<<grid, kTwThreads, 0, s>>>(a)
  if (fwd) {
    REM_TW(0, true);
  } else {
    switch (ks) {
      case 0: REM_TW(0, false); break;
      case 1: REM_TW(1, false); break;
      case 2: REM_TW(2, false); break;
      case 4: REM_TW(4, false); break;
      case 8: REM_TW(8, false); break;
      default: return hipErrorInvalidValue;
    }
  }
#undef REM_TW
  return hipGetLastError();
}

}  // namespace rem
