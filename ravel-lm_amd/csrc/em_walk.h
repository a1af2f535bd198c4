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
// FWD.  A write adds its payload row to S, a read takes S; with values, a write
// also enters the ring of its run's last k rows, which a read stores.
// So in both directions a "loader" item adds rows, a "consumer" item takes the
// sum, and every row is read, and every result written, once.  A loader that no
// later consumer of its run needs is dropped from the walk, and of a read's k
// gradient rows only those of the writes that exist are read (the counts are
// taken on the sorted keys).
//
// Work: a block takes a part of up to 928 items of one segment (smaller parts
// where the tape is too short to fill the chip), a walker of G lanes (one unit of
// UB bytes each) a contiguous range of them.  Where every run is short, walkers
// take whole runs and steps 2 and 3 fall away; else
//   1. code words: one 32-bit word per kept item (time, counts, flags);
//   2. every walker sums from the last run start of its range to its end (the
//      state that leaves the range);
//   3. the states are composed over the walkers of a wave (shuffles), the waves
//      (LDS) and, where a run crosses parts, the earlier parts (published words,
//      read newest first in a fixed order): (f1, m1, S1, P1) then (f2, m2, S2,
//      P2) = f2 ? second : (f1, m1 + m2, S1 + S2, P2[j] + P1[j + m2]), f "a run
//      starts or ends in it", m consumers passed (FWD: m writes passed, and the ring of
//      their times, m2 of the second before those of the first);
//   4. every walker walks its range again with the state that enters it.
// Sums are formed in an order that does not depend on timing; they accumulate in
// fp32 for 16-bit rows and fp64 otherwise and are rounded once.
//
// Measured (launch alone): joint backward of 2.1M records, separate reads, k = 4,
// bf16 D = 64: 162 us, where the sort of N k source ids as one segment, its run
// totals, the reads' atomics, the walk and the addition took 5.5 ms (300 us with
// every slot of every item walked); of 262k records, reads = writes, k = 8, fp32
// D = 32: 58 us (5.8 TB/s) against 140; the sum's backward of 4.2M records, bf16
// D = 64: 160 us (5.0 TB/s of random rows) against 221 for a walker that
// branches; its forward 172 us, as the walker of power-of-two rows before it; the
// joint forward of 6 x 6007 x 6 masked records with separate reads, rows of 96
// bytes, k = 2: 44 us, where the searches, gathers and chunked sums took 118.
//
// Loads and stores go through buffer descriptors of the segment's rows: a set
// bit 31 of the offset lies past every range, which turns a skipped load into
// zeros and a skipped store into nothing, so the walk has no branches within a
// batch.  The reverse walk is bound by its vector instructions (each slot costs
// some 32 an item and lane), so a batch runs the form for the deepest slot that
// any of the wave's walkers has in use: most reads of a spread-out tape have one
// earlier write or none.
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
  int part;              // items per part (at most 928)
  int64_t nparts;
  int G, gtot, ncb;      // lanes per walker, units per row, column blocks
  const void* sum_in;    // rows [B,T,C,D] or null
  const void* val_in;    // rows [B,T,C,k,D] or null
  int k;
  void* out;             // rows [B,T,C,D]
  uint8_t* omask;        // FWD: [B,T,C] "some earlier write"
  void* val_out;         // FWD: rows [B,T,C,k,D] of the last k writes, or null
  uint8_t* vmask;        // FWD: [B,T,C,k], with val_out and k > 1 (else omask's bytes)
  uint64_t* words;       // published states, zero on entry (nparts > 1)
  uint64_t* tickets;     // [ncb][nseg], zero on entry (nparts > 1)
  uint32_t* err;
};

constexpr int kTwThreads = 256;
constexpr int kTwWaves = kTwThreads / kWave;
constexpr int kTwMaxPart = 928;     // items of a part: see walk_part()
constexpr int kTwCross = 64;       // a run's items past a part that stay with the part
constexpr int kTwMaxItems = kTwMaxPart + kTwCross;
constexpr int kTwColBytes = 512;   // accumulators of one state component of a block

// Code words: the time in bits 0..23 (the 24-bit multiplies ignore the rest), the
// rows to load of a read in bits 24..27.
constexpr uint32_t kTwTime = (1u << 24) - 1u;
constexpr int kTwCount = 24;
constexpr uint32_t kTwLast = 1u << 29, kTwNoStore = 1u << 30, kTwNoLoad = 1u << 31;
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

// c ? x : y by value (a conditional on two array elements would select their
// addresses and keep the arrays in memory)
template <typename V>
__device__ __forceinline__ V pick(bool c, V x, V y) {
  return c ? x : y;
}

// Waves per SIMD that the registers are held to, and the items in flight of a
// reverse batch whose deepest slot is kd: a few values of scratch at four waves
// measured 2 % faster than none at three (joint backward, k = 4, bf16).
constexpr int walk_waves(int ks, bool fwd) { return fwd || ks <= 4 ? 4 : 2; }
constexpr int walk_batch(int kd) { return kd <= 1 ? 4 : kd == 2 ? 2 : 1; }

template <int DT, int UB, int KS, bool FWD>
__global__ __launch_bounds__(kTwThreads)
__attribute__((amdgpu_waves_per_eu(walk_waves(KS, FWD), 8))) void tape_walk_kernel(const WalkArgs a) {
  using E = Elem<DT>;
  using X = typename E::store_t;
  using Acc = typename E::acc_t;
  using BU = BufUnit<UB>;
  using V = typename BU::T;
  constexpr int CPU = UB / (int)sizeof(X);  // columns per lane
  constexpr int MAXC = kTwColBytes / (int)sizeof(Acc);
  constexpr int KP = FWD ? 0 : KS;          // slot sums
  constexpr int KF = FWD ? KS : 0;          // ring of rows
  constexpr int NC = KP + 1;                // state components: S, P[0..KP-1]
  constexpr int KR = KP > 0 ? KP : 1, KG = KF > 0 ? KF : 1;
    constexpr int RB = KS == 0 || (FWD && KS == 1) ? 16 : FWD ? 8 : 4;  // items of a batch
  static_assert((KS & (KS - 1)) == 0 && KS <= 8, "shifts by powers of two");
  __shared__ uint64_t kk[kTwMaxItems + 2];         // kk[i + 1]: key of walk item i
  __shared__ uint32_t cw[kTwMaxItems + 64];
  __shared__ uint64_t sbits[kTwMaxItems / 64 + 1];  // run starts
  __shared__ int astart[kTwThreads];               // per walker: its first run start
  __shared__ Acc agg[(kTwWaves + 1) * NC * MAXC];     // [wave, then carry][component][column]
  __shared__ uint32_t ring_s[kTwWaves + 1][KG];       // [wave, then carry]
  __shared__ int wf[kTwWaves], wm[kTwWaves + 1], wc[kTwWaves], wb[kTwWaves];
  __shared__ uint8_t hm[FWD ? kTwMaxItems : 4];
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
  for (int i = tid; i < n + 2 + kTwCross; i += kTwThreads) {
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
  // A run that crosses into a part and ends within kTwCross items of it stays
  // whole, with the part before; both sides see the same end.  Only longer runs
  // pass their state on.
  bool open = !ends(n - 1);  // the last run goes on in the next part
  bool joined = !ends(-1);   // the first run comes from the part before
  int i0 = 0, i1 = n;        // the part's items
  if (open) {
    const uint64_t m = __ballot(p0 + n + lane < a.L && ends(n + lane));
    if (m) i1 = n + __builtin_ctzll(m) + 1, open = false;
  }
  if (joined) {
    const uint64_t m = __ballot(p0 + lane < a.L && ends(lane));
    if (m) i0 = __builtin_ctzll(m) + 1, joined = false;
  }
  // Records: the ring that enters the part is the keys before it.
  if (KF > 0 && same && joined && wave == 0) {
    const int64_t wi = p0 - 1 - lane;
    uint64_t key = kk[0];
    if (KF > 1 && lane > 0 && lane < KF && wi >= 0) key = key_at(wi);
    const bool in = lane < KF && wi >= 0 && (key >> tb) == (kk[1] >> tb);
    if (in) ring_s[kTwWaves][lane] = (uint32_t)(key & imask);
    const int held = __popcll(__ballot(in));
    if (lane == 0) wm[kTwWaves] = held;
  }
  // Consumers of the last run past the part, up to kc (what a count can use).
  const int kc = KP > 0 ? a.k : 1;
  int ext = 0;
  if (open && !same) {  // uniform: at least kTwCross items of the run follow
    const uint64_t ra = kk[n] >> tb;
    ext = __popcll(__ballot(consumes(kk[n + 1 + lane])));
    bool done = ext >= kc;
    // a long stretch without a consumer: 1024 items a round
    for (int64_t w0 = p0 + n + kTwCross; !done && w0 < a.L; w0 += 4 * kTwThreads) {
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
  // 1. code words.  Records need no scan: their consumers are the records after
  // them, none is dropped.  Otherwise thread tid has items [i0 + tid ipt, + ipt);
  // a segmented suffix scan over the threads counts the consumers after each item in its run.
  // A loader with none ends the part of its run that matters: it and what follows
  // of the run are dropped (a dropped item starts a run only if all of the run
  // is), and the kept items close ranks.
  int nk;  // kept items
  if (same) {
    nk = i1 - i0;
    for (int i = i0 + tid; i < i1 + 64; i += kTwThreads) {
      uint32_t code = kTwPad;
      if (i < i1) {
        int cnt = 0;
        while (cnt < kc && !ends(i + cnt)) ++cnt;
        code = (uint32_t)(kk[i + 1] & imask) | ((uint32_t)cnt << kTwCount) |
               (cnt > 0 ? 0u : kTwLast | kTwNoLoad);
      }
      cw[i - i0] = code;
    }
  } else {
    constexpr int IPT = (kTwMaxItems + kTwThreads - 1) / kTwThreads;
    const int ipt = (i1 - i0 + kTwThreads - 1) / kTwThreads;
    int cn[IPT], op[IPT];
    int cs = 0, bs = 0;
#pragma unroll
    for (int j = IPT - 1; j >= 0; --j) {
      const int i = i0 + tid * ipt + j;
      cn[j] = op[j] = 0;
      if (j < ipt && i < i1) {
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
    uint32_t code[IPT];
    uint32_t kept = 0;
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const int i = i0 + tid * ipt + j;
      code[j] = 0;
      if (j < ipt && i < i1) {
        const uint64_t key = kk[i + 1];
        const uint32_t idx = (uint32_t)(key & imask);
        int cnt = cn[j] + (op[j] ? xc : 0);
        cnt = cnt < kc ? cnt : kc;
        const bool cons = consumes(key);
        const uint32_t last = cons && cnt == 0 ? kTwLast : 0u;
        if (cons) cnt = 0;
        if (cons || cnt > 0) {
          code[j] = (idx >> 1) | ((uint32_t)cnt << kTwCount) | last |
                    (cons ? 0u : kTwNoStore) | (cnt > 0 ? 0u : kTwNoLoad);
          kept |= 1u << j;
        }
      }
    }
    const uint32_t mine = (uint32_t)__popc(kept);
    const uint32_t incl = wave_incl_scan(mine);
    __syncthreads();  // wc, wb are read
    if (lane == kWave - 1) wc[wave] = (int)incl;
    __syncthreads();
    uint32_t at = incl - mine;
    nk = 0;
    for (int w2 = 0; w2 < kTwWaves; ++w2) {
      if (w2 < wave) at += (uint32_t)wc[w2];
      nk += wc[w2];
    }
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      if (kept & (1u << j)) cw[at++] = code[j];
    if (tid < 64) cw[nk + tid] = kTwPad;  // whole batches and ballots
  }
  __syncthreads();
  // Starts: the first item where no state enters the part, and every item after a
  // run's last consumer (the kept items of a run end with it), so that one past
  // the kept items can be one too.
  for (int i = wave; i * 64 <= nk; i += kTwWaves) {
    const int at = i * 64 + lane;
    const uint64_t m = __ballot(at == 0 ? !joined : at <= nk && (cw[at - 1] & kTwLast) != 0);
    if (lane == 0) sbits[i] = m;
  }
  __syncthreads();
  const int G = a.G;
  const int wpw = kWave / G;  // walkers per wave
  const int wi = lane / G, v = lane - (lane / G) * G;
  const int NW = wpw * kTwWaves;
  const int w = wave * wpw + wi;
  const int len = (nk + NW - 1) / NW;
  const bool on = wi < wpw;
  const int rs = on && w * len < nk ? w * len : nk;
  const int re = (rs + len) < nk ? (rs + len) : nk;
  const int vcol = cb * G + v;
  const uint32_t vo = (uint32_t)vcol * UB;
  const uint32_t vbad = on && vcol < a.gtot ? 0u : 0x80000000u;
  const uint32_t row = (uint32_t)a.gtot * UB;
  const uint32_t tstride = (uint32_t)a.C * row, vstride = tstride * (uint32_t)a.k;
  const int64_t rec0 = b * a.T * a.C + c;
  const uint32_t ext_row = (uint32_t)((a.T - 1) * tstride + row);
  const uint32_t ext_val = (uint32_t)((a.T - 1) * vstride + row * (uint32_t)a.k);
  const __amdgpu_buffer_rsrc_t srs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const unsigned char*)a.sum_in + (a.sum_in ? rec0 * row : 0)), 0,
      a.sum_in ? (int)ext_row : 0, kTwRsrc3);
  // the slots' rows: gradients read (REV) or values written (FWD)
  const unsigned char* vbase = FWD ? (const unsigned char*)a.val_out : (const unsigned char*)a.val_in;
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(vbase + (vbase ? rec0 * a.k * (int64_t)row : 0)), 0,
      KS > 0 && vbase ? (int)ext_val : 0, kTwRsrc3);
  const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((unsigned char*)a.out + rec0 * row), 0, (int)ext_row, kTwRsrc3);
  Acc S[CPU], P[KR][CPU];
  int mc = 0;  // REV: consumers passed in the run; FWD: loaders passed
  int pd = 0;  // REV: slot sums from pd on are zero
  uint32_t rt[KG];  // FWD: times of the run's last writes, newest first
  V vr[KG];         // and, in the final walk, their rows
  // NB items from i0 on; slots below KD are in use (held: their rows are in hx).
  V hx[KP == 0 ? RB : 1];
  auto batch = [&](int i0, int to, auto nb_tag, auto kd_tag, auto store_tag, auto held_tag) {
    constexpr int NB = decltype(nb_tag)::value, KD = decltype(kd_tag)::value;
    constexpr bool STORE = decltype(store_tag)::value;
    // the last use of a row streams, except beside several value stores a read
    // (cached measured 10 % faster there: 6 x 6007 x 6 reads, k = 2)
    constexpr int AUX = STORE && KF <= 1 ? kTwStream : 0;
    uint32_t k4[NB];
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      k4[m] = cw[i0 + m];
      if (i0 + m >= to) k4[m] = kTwPad;
    }
    V xs[NB], xv[NB][KD > 0 ? KD : 1];
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      if constexpr (decltype(held_tag)::value)
        xs[m] = hx[m];
      else
        xs[m] = BU::template load<AUX>(
            srs, (__umul24(k4[m], tstride) + vo) | (k4[m] & kTwNoLoad) | vbad);
      if constexpr (KD > 0) {
        const uint32_t cnt = (k4[m] >> kTwCount) & 15u;
        const uint32_t o = __umul24(k4[m], vstride) + vo;
#pragma unroll
        for (int j = 0; j < KD; ++j)
          xv[m][j] = BU::template load<AUX>(
              vrs, (o + (uint32_t)j * row) | ((uint32_t)j < cnt ? vbad : 0x80000000u));
      }
    }
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      const uint32_t k = k4[m];
      // The last consumer of a run leaves a zero state behind: its S is dropped,
      // and no slot sum reaches past the run's writes.
      const bool end = k & kTwLast, cons = !(k & kTwNoStore);
      const uint32_t ns = ((k & kTwNoStore) << 1) | vbad;
      if (STORE) {
        Acc t[CPU];
#pragma unroll
        for (int e = 0; e < CPU; ++e) {
          t[e] = S[e];
          if constexpr (KD > 0) t[e] += P[0][e];
        }
        BU::store(walk_pack<DT, V, CPU>(t), ors, (__umul24(k, tstride) + vo) | ns);
        if constexpr (KF > 0) {
          const uint32_t o = __umul24(k, vstride) + vo;
#pragma unroll
          for (int j = 0; j < KF; ++j)
            BU::store(pick(j < mc, vr[j], V{}), vrs,
                      (o + (uint32_t)j * row) | (j < a.k ? ns : 0x80000000u));
        }
        if (FWD && v == 0 && cons) hm[i0 + m] = (uint8_t)(mc < 15 ? mc : 15);
      }
      if constexpr (KD > 0) {
#pragma unroll
        for (int j = 0; j < KD; ++j)
#pragma unroll
          for (int e = 0; e < CPU; ++e) {
            const Acc up = j + 1 < KD ? P[j + 1 < KD ? j + 1 : 0][e] : Acc(0);
            P[j][e] = cons ? up : P[j][e];
          }
      }
      if constexpr (KP > 0) {
        const int cnt = (int)((k >> kTwCount) & 15u);
        pd = end ? 0 : cons && pd > 0 ? pd - 1 : pd;
        pd = cnt > pd ? cnt : pd;
      }
#pragma unroll
      for (int e = 0; e < CPU; ++e) S[e] = end ? Acc(0) : S[e];
      const bool ld = !(k & kTwNoLoad);
      mc = (end ? 0 : mc) + (FWD ? (ld ? 1 : 0) : (cons ? 1 : 0));
      if constexpr (KF > 0) {
#pragma unroll
        for (int j = KF - 1; j > 0; --j) rt[j] = ld ? rt[j - 1] : rt[j];
        rt[0] = ld ? (k & kTwTime) : rt[0];
        if (STORE) {
#pragma unroll
          for (int j = KF - 1; j > 0; --j) vr[j] = pick(ld, vr[j - 1], vr[j]);
          vr[0] = pick(ld, xs[m], vr[0]);
        }
      }
      union { V u; X e[CPU]; } x;
      x.u = xs[m];
#pragma unroll
      for (int e = 0; e < CPU; ++e) S[e] += E::load(x.e[e]);
      if constexpr (KD > 0) {
#pragma unroll
        for (int j = 0; j < KD; ++j) {
          x.u = xv[m][j];
#pragma unroll
          for (int e = 0; e < CPU; ++e) P[j][e] += E::load(x.e[e]);
        }
      }
    }
  };
  auto walk = [&](int from, int to, auto store_tag) {
    for (int i0 = from; i0 < to; i0 += RB) {
      if constexpr (KP == 0) {
        batch(i0, to, std::integral_constant<int, RB>{}, std::integral_constant<int, 0>{},
              store_tag, std::false_type{});
      } else {
        // the deepest slot in use by the wave's active walkers; deep forms run in
        // sub-batches, whose rows the registers hold
        uint32_t most = (uint32_t)pd;
#pragma unroll
        for (int m = 0; m < RB; ++m) {
          const uint32_t cnt = (cw[i0 + m] >> kTwCount) & 15u;
          most = cnt > most && i0 + m < to ? cnt : most;
        }
        auto parts = [&](auto kd_tag) {
          constexpr int NB = walk_batch(decltype(kd_tag)::value);
#pragma unroll 1
          for (int h = 0; h < RB; h += NB)
            batch(i0 + h, to, std::integral_constant<int, NB>{}, kd_tag, store_tag,
                  std::false_type{});
        };
        if (!__any(most > 0)) {
          parts(std::integral_constant<int, 0>{});
        } else if (KP == 1 || !__any(most > 1)) {
          parts(std::integral_constant<int, 1>{});
        } else if (KP == 2 || !__any(most > 2)) {
          if constexpr (KP >= 2) parts(std::integral_constant<int, 2>{});
        } else if (KP == 4 || !__any(most > 4)) {
          if constexpr (KP >= 4) parts(std::integral_constant<int, 4>{});
        } else {
          if constexpr (KP >= 8) parts(std::integral_constant<int, 8>{});
        }
      }
    }
  };
  // KP == 0: the state of items [tail, to) of one run, in the range from `from`
  // on: the sum of their rows, and the newest loaders.  The range's first batch
  // comes last and stays in hx for the final walk: inside a long run, where every
  // row is read twice, that is half of the second reads (4.2M records, 90 % of
  // each segment's in one run, bf16 D = 64: the sum 333 -> 317 us).
  auto tail_sums = [&](int from, int tail, int to) {
    for (int i0 = from + (to - from - 1) / RB * RB; i0 > from && i0 + RB > tail; i0 -= RB) {
      V xs[RB];
#pragma unroll
      for (int m = 0; m < RB; ++m) {
        const int i = i0 + m;
        const uint32_t k = i >= tail && i < to ? cw[i] : kTwPad;
        xs[m] = BU::template load<0>(srs, (__umul24(k, tstride) + vo) | (k & kTwNoLoad) | vbad);
      }
#pragma unroll
      for (int m = 0; m < RB; ++m) {
        union { V u; X e[CPU]; } x;
        x.u = xs[m];
#pragma unroll
        for (int e = 0; e < CPU; ++e) S[e] += E::load(x.e[e]);
      }
    }
#pragma unroll
    for (int m = 0; m < RB; ++m) {
      const uint32_t k = from + m < to ? cw[from + m] : kTwPad;
      hx[KP == 0 ? m : 0] =
          BU::template load<0>(srs, (__umul24(k, tstride) + vo) | (k & kTwNoLoad) | vbad);
    }
#pragma unroll
    for (int m = 0; m < RB; ++m) {
      union { V u; X e[CPU]; } x;
      x.u = pick(from + m >= tail, hx[KP == 0 ? m : 0], V{});
#pragma unroll
      for (int e = 0; e < CPU; ++e) S[e] += E::load(x.e[e]);
    }
    if constexpr (FWD) {
      for (int i = to - 1; i >= tail && mc < KG; --i) {
        const uint32_t k = cw[i];
        if (k & kTwNoLoad) continue;
#pragma unroll
        for (int j = 0; j < KG; ++j) rt[j] = j == mc ? k & kTwTime : rt[j];
        ++mc;
      }
    }
  };
  // The first start in the walker's range, and the last in it or right after it.
  int first = nk, last = -1;
  if (rs < re) {
    for (int word = rs >> 6; word <= re >> 6; ++word) {
      uint64_t m = sbits[word];
      const int lo = word << 6;
      if (re - lo < 63) m &= (2ull << (re - lo)) - 1ull;
      if (rs > lo) m &= ~0ull << (rs - lo);
      if (m) {
        if (first == nk) first = lo + __builtin_ctzll(m);
        last = lo + 63 - __builtin_clzll(m);
      }
    }
    first = first < re ? first : nk;
  }
  // Whole runs: where no state enters or leaves the part, a walker takes the runs
  // that start in its range, up to the first start of the next walker that has
  // one, from a zero state; where that would make some walker's share more than
  // twice the even one (long runs), the block takes even ranges and composes.
  int from = rs, to = re;
  bool even = open || joined;
  if (!even) {  // uniform
    if (on && v == 0) astart[w] = first < nk ? first : (rs < re ? -1 : nk);
    __syncthreads();
    bool over = false;
    if (first < nk) {
      const int a1 = w + 1 < NW ? astart[w + 1] : nk;
      const int a2 = w + 2 < NW ? astart[w + 2] : nk;
      from = first;
      to = a1 >= 0 ? a1 : a2;
      over = to < 0 || to - from > 2 * len;
    }
    even = __syncthreads_or(over);
  }
#pragma unroll
  for (int e = 0; e < CPU; ++e) S[e] = Acc(0);
#pragma unroll
  for (int j = 0; j < KR; ++j)
#pragma unroll
    for (int e = 0; e < CPU; ++e) P[j][e] = Acc(0);
#pragma unroll
  for (int j = 0; j < KG; ++j) rt[j] = 0u, vr[j] = V{};
  if (even) {
  from = rs, to = re;
  // 2. the state leaving the walker's range
  if constexpr (KP > 0)
    walk(last >= 0 ? last : rs, re, std::false_type{});
  else
    tail_sums(rs, last >= 0 ? last : rs, re);
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
    if constexpr (KP > 0) {
      const int ppd = __shfl(pd, src, kWave);
      if (__any(take && ppd > mc)) {  // some slot sum of an earlier walker reaches past
#pragma unroll
        for (int e = 0; e < CPU; ++e) {
          Acc t[KR];
#pragma unroll
          for (int j = 0; j < KP; ++j) t[j] = __shfl(P[j][e], src, kWave);
#pragma unroll
          for (int s2 = 1; s2 < KP; s2 <<= 1)
#pragma unroll
            for (int j = 0; j < KP; ++j) {
              const Acc up = j + s2 < KP ? t[j + s2 < KP ? j + s2 : 0] : Acc(0);
              t[j] = (mc & s2) ? up : t[j];
            }
#pragma unroll
          for (int j = 0; j < KP; ++j) P[j][e] = take && mc < KP ? P[j][e] + t[j] : P[j][e];
        }
      }
      if (take) pd = ppd - mc > pd ? ppd - mc : pd;
    }
    if constexpr (KF > 0) {
      uint32_t t[KG];
#pragma unroll
      for (int j = 0; j < KF; ++j) t[j] = (uint32_t)__shfl((int)rt[j], src, kWave);
#pragma unroll
      for (int s2 = 1; s2 < KF; s2 <<= 1)
#pragma unroll
        for (int j = KF - 1; j >= 0; --j)
          t[j] = (mc & s2) && j >= s2 ? t[j >= s2 ? j - s2 : 0] : t[j];
#pragma unroll
      for (int j = 0; j < KF; ++j) rt[j] = take && j >= mc ? t[j] : rt[j];
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
      if constexpr (KP > 0) {
#pragma unroll
        for (int j = 0; j < KP; ++j) agg[(wave * NC + 1 + j) * MAXC + v * CPU + e] = P[j][e];
      }
    }
    if (v == 0) {
      wf[wave] = f;
      wm[wave] = mc;
      if constexpr (KF > 0) {
#pragma unroll
        for (int j = 0; j < KF; ++j) ring_s[wave][j] = rt[j];
      }
    }
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
    if constexpr (KP > 0) {
      const int ppd = __shfl(pd, src, kWave);
      const bool deep = __any(pd > 0);
#pragma unroll
      for (int j = 0; j < KP; ++j)
#pragma unroll
        for (int e = 0; e < CPU; ++e) {
          const Acc t = deep ? __shfl(P[j][e], src, kWave) : Acc(0);
          P[j][e] = any ? t : Acc(0);
        }
      pd = any ? ppd : 0;
    }
    if constexpr (KF > 0) {
#pragma unroll
      for (int j = 0; j < KF; ++j) rt[j] = (uint32_t)__shfl((int)rt[j], src, kWave);
    }
    const int pf = __shfl(f, src, kWave), pm = __shfl(mc, src, kWave);
    f = any ? pf : 0;
    mc = any ? pm : 0;
  }
  __syncthreads();
  // the block's state, published where the next part's first run needs it; then
  // the state of the earlier parts, where this part's first run needs it
  constexpr int PW = Pub<Acc>::W;
  const int64_t pstride = (int64_t)NC * cols * PW + KF;
  auto part_at = [&](int64_t part) -> uint64_t* {
    return a.words + ((seg * a.nparts + part) * a.ncb + cb) * pstride;
  };
  if (tid < cols) {
    if (open) {
      Acc bs = Acc(0), bp[KR];
      int bm = 0, bf = 0;
      uint64_t* mine = part_at(q);
#pragma unroll
      for (int j = 0; j < KR; ++j) bp[j] = Acc(0);
      for (int w2 = kTwWaves - 1; w2 >= 0 && !bf; --w2) {
        bs += agg[(w2 * NC) * MAXC + tid];
        if constexpr (KP > 0) {
#pragma unroll
          for (int j = 0; j < KP; ++j)
            if (j + bm < KP) bp[j] += agg[(w2 * NC + 1 + j + bm) * MAXC + tid];
        }
        if (KF > 0 && !same && tid == 0) {  // ring words that this wave fills
          for (int j = 0; j < wm[w2] && j + bm < KF; ++j)
            Pub<float>::put(mine + (int64_t)NC * cols * PW + bm + j,
                            __uint_as_float(ring_s[w2][j]), 1u);
        }
        bm = bm + wm[w2] < 15 ? bm + wm[w2] : 15;
        bf = wf[w2];
      }
      if (!joined) bf = 1;
      const uint32_t flag = 1u | ((uint32_t)bf << 1) | ((uint32_t)bm << 4);
      Pub<Acc>::put(mine + (int64_t)tid * PW, bs, flag);
      if constexpr (KP > 0) {
#pragma unroll
        for (int j = 0; j < KP; ++j)
          Pub<Acc>::put(mine + ((int64_t)(1 + j) * cols + tid) * PW, bp[j], flag);
      }
    }
    Acc ls = Acc(0), lp[KR];
    int lm = 0;
#pragma unroll
    for (int j = 0; j < KR; ++j) lp[j] = Acc(0);
    if (joined) {
      auto at = [&](int64_t part, int comp) {
        return part_at(part) + ((int64_t)comp * cols + tid) * PW;
      };
      int64_t j0 = q - 1;
      bool done = false;
      uint32_t fl = 0;
      if (KS > 0 && !(KF > 0 && same)) {
        while (!done && j0 >= 0 && lm < KS) {  // parts whose slots can still reach this one
          Acc val;
          if (!Pub<Acc>::get(at(j0, 0), &val, &fl)) {
            atomicOr(a.err, kStatusSumWait);
            done = true;
            break;
          }
          ls = val + ls;
          const uint32_t f0 = fl;
          const int pm = (int)(f0 >> 4);
          if constexpr (KP > 0) {
#pragma unroll
            for (int j = 0; j < KP; ++j) {
              if (j + lm < KP) {
                if (!Pub<Acc>::get(at(j0, 1 + j + lm), &val, &fl)) {
                  atomicOr(a.err, kStatusSumWait);
                  done = true;
                } else {
                  lp[j] += val;
                }
              }
            }
          }
          if (KF > 0 && tid == 0) {
            for (int j = 0; j < pm && j + lm < KF; ++j) {
              float t = 0.f;
              if (!Pub<float>::get(part_at(j0) + (int64_t)NC * cols * PW + j, &t, &fl))
                atomicOr(a.err, kStatusSumWait);
              ring_s[kTwWaves][lm + j] = __float_as_uint(t);
            }
          }
          lm += pm;
          done = done || (f0 & 2u);
          --j0;
        }
        if (!FWD && !a.sum_in) done = true;  // only the slots' sums are wanted
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
    }
    if (tid == 0 && !(KF > 0 && same && joined)) wm[kTwWaves] = lm < 15 ? lm : 15;
    agg[(kTwWaves * NC) * MAXC + tid] = ls;
    if constexpr (KP > 0) {
#pragma unroll
      for (int j = 0; j < KP; ++j) agg[(kTwWaves * NC + 1 + j) * MAXC + tid] = lp[j];
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
      if constexpr (KP > 0) {
#pragma unroll
        for (int j = 0; j < KP; ++j)
          if (j + mc < KP) P[j][e] += agg[(g * NC + 1 + j + mc) * MAXC + col];
      }
    }
    if constexpr (KP > 0) pd = KP;  // unknown: any slot may be in use
    if constexpr (KF > 0) {
#pragma unroll
      for (int j = 0; j < KF; ++j)
        if (j >= mc && j - mc < wm[g]) rt[j] = ring_s[g][j - mc];
    }
    mc = mc + wm[g] < 15 ? mc + wm[g] : 15;
    if (w2 >= 0) f = wf[w2];
  }
  if constexpr (KF > 0) {  // the rows of the writes before the range
    if (rs < re) {
#pragma unroll
      for (int j = 0; j < KF; ++j)
        vr[j] = BU::template load<0>(
            srs, (__umul24(rt[j], tstride) + vo) | (j < mc ? vbad : 0x80000000u));
    }
  }
  if constexpr (KP == 0) {  // the range's first batch
    if (rs < re)
      batch(rs, re, std::integral_constant<int, RB>{}, std::integral_constant<int, 0>{},
            std::true_type{}, std::true_type{});
    from += RB;
  }
  } else if (first == nk) {
    from = to = nk;
  }
  // 4. the walk
  walk(from, to, std::true_type{});
  if constexpr (FWD) {
    __syncthreads();
    if (cb == 0) {
      const __amdgpu_buffer_rsrc_t mrs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(a.omask + rec0), 0, (int)((a.T - 1) * a.C + 1), kTwRsrc3);
      const __amdgpu_buffer_rsrc_t lrs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(a.vmask + (KF > 1 ? rec0 * a.k : 0)), 0,
          KF > 1 ? (int)(((a.T - 1) * a.C + 1) * a.k) : 0, kTwRsrc3);
      for (int i = tid; i < nk; i += kTwThreads) {
        const uint32_t k = cw[i];
        if (k & kTwNoStore) continue;
        const int cnt = hm[i];
        const uint32_t mo = (k & kTwTime) * (uint32_t)a.C;
        __builtin_amdgcn_raw_buffer_store_b8(cnt > 0 ? 1 : 0, mrs, mo, 0, 0);
        if constexpr (KF > 1) {
          if (a.k == 4) {
            const uint32_t m4 = cnt >= 4 ? 0x01010101u : 0x01010101u & ((1u << (8 * cnt)) - 1u);
            __builtin_amdgcn_raw_buffer_store_b32(m4, lrs, mo * 4u, 0, 0);
          } else {
            for (int j = 0; j < a.k; ++j)
              __builtin_amdgcn_raw_buffer_store_b8(j < cnt ? 1 : 0, lrs,
                                                   mo * (uint32_t)a.k + (uint32_t)j, 0, 0);
          }
        }
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
    switch (ks) {
      case 0: REM_TW(0, true); break;
      case 1: REM_TW(1, true); break;
      case 2:
      case 4: REM_TW(4, true); break;
      case 8: REM_TW(8, true); break;
      default: return hipErrorInvalidValue;
    }
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
