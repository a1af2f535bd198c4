// Host side of the segmented walks (em_walk.h) and the merged address tape of
// calls whose reads have addresses or a write mask of their own.

#include "em_walk.h"

#include "em_addr.h"

namespace rem {

namespace {

// Reads and writes of a [B,T,C] tape as one address tensor [B,2T,C]: time 2t is
// the read of t, 2t + 1 its write (a masked write: the sentinel A).  The sort
// of that tensor as a tape of 2T steps then orders a stream's reads and writes
// together.  Bound by its streams: 16 bytes in and 2 or 4 times 2 bytes out a
// record for int64 addresses.
template <typename AS, typename O>
__global__ __launch_bounds__(256) void merge_addresses_kernel(
    const AS wa, const AS ra, const uint8_t* __restrict__ wmask, int64_t N, int64_t T, uint32_t C,
    FastDiv by_c, int64_t A, int trunc32, O* __restrict__ out) {
  constexpr int ILP = 4;
  const int64_t base = (int64_t)blockIdx.x * 256 * ILP + threadIdx.x;
  int64_t w[ILP], r[ILP];
  uint32_t bt[ILP], m[ILP];
#pragma unroll
  for (int i = 0; i < ILP; ++i) {
    const int64_t g = base + i * 256;
    const bool in = g < N;
    w[i] = in ? (int64_t)wa.p[g] : 0;
    r[i] = in ? (int64_t)ra.p[g] : 0;
    bt[i] = in ? fdiv((uint32_t)g, by_c) : 0u;
    m[i] = in && wmask ? wmask[bt[i]] : 1u;
  }
#pragma unroll
  for (int i = 0; i < ILP; ++i) {
    const int64_t g = base + i * 256;
    if (g >= N) continue;
    const int64_t o = g + (int64_t)bt[i] * C;  // 2 C per step: (2 bt) C + c
    out[o] = (O)reduce_addr(r[i], A, kWrap, trunc32 != 0);
    out[o + C] = m[i] ? (O)reduce_addr(w[i], A, kWrap, trunc32 != 0) : (O)A;
  }
}

int next_pow2(int x) {
  int p = 1;
  while (p < x) p <<= 1;
  return p;
}

int unit_bytes(int dtype, int64_t row, uintptr_t align) {
  const uintptr_t m = align | (uintptr_t)row;
  switch (dtype) {
    case kF64: return (m & 7) == 0 ? 8 : 0;
    case kF32: return (m & 15) == 0 ? 16 : (m & 3) == 0 ? 4 : 0;
    default: return (m & 15) == 0 ? 16 : (m & 3) == 0 ? 4 : (m & 1) == 0 ? 2 : 0;
  }
}

// Lanes per walker, column blocks and published words of one unit size.
void walk_columns(int dtype, int64_t row, int ub, int* gtot, int* G, int* ncb) {
  const int per = ub / dtype_size(dtype);                       // columns per lane
  const int maxc = kTwColBytes / (int)acc_bytes(dtype);
  int lim = maxc / per;
  if (lim > kWave) lim = kWave;
  *gtot = (int)(row / ub);
  *ncb = (*gtot + lim - 1) / lim;
  *G = (*gtot + *ncb - 1) / *ncb;
}

// Items per part: 928, fewer while the tape would not give every CU two blocks.
// A walker of 8 lanes (128-byte rows) then has 29 items, so that whole runs from
// its first start on still fit two batches of 16 in nearly every walker: 1024
// items (32 each) took a third batch for the one or two that hang over (sum of
// 4.2M records, bf16 D = 64: 239 us against 232; 896 the same).  The parts of a
// segment are of one size: a last part of 96 items beside one of 928 made the
// training step of 32 x 1024 x 8 records, k = 8 fp32, 167 us instead of 133.
int walk_part(int64_t nseg, int64_t L) {
  int64_t part = kTwMaxPart;
  for (int h = 0; h < 2 && nseg * ((L + part - 1) / part) < 512; ++h) part /= 2;
  const int64_t nparts = (L + part - 1) / part;
  return (int)((L + nparts - 1) / nparts);
}

int64_t state_words(int64_t nseg, int64_t L, int64_t D, int dtype, int ks, int ub) {
  int gtot, G, ncb;
  walk_columns(dtype, D * dtype_size(dtype), ub, &gtot, &G, &ncb);
  const int64_t nparts = (L + walk_part(nseg, L) - 1) / walk_part(nseg, L);
  const int64_t cols = (int64_t)G * (ub / dtype_size(dtype));
  return nseg * nparts * ncb * ((ks + 1) * cols * (int64_t)(acc_bytes(dtype) / 4) + 8) + nseg * ncb;
}

}  // namespace

// State components of k slots (0: the sum alone): a power of two.
int walk_slots(int64_t k) { return k <= 0 ? 0 : next_pow2((int)k); }

bool walk_applies(const Tape& tp, int64_t D, int dtype, int64_t k) {
  const int64_t row = D * dtype_size(dtype);
  const int64_t kk = k > 0 ? k : 1;
  // 24-bit times and strides, a segment's rows below 2^31 bytes of its base
  return k <= 8 && tp.T >= 1 && tp.T <= ((int64_t)1 << 24) && row < ((int64_t)1 << 24) &&
         tp.C * kk < ((int64_t)1 << 24) && tp.C * row * kk < ((int64_t)1 << 24) &&
         tp.T * tp.C * row * kk < ((int64_t)1 << 31) &&
         tp.nseg() * (2 * tp.T / (kTwMaxPart / 4) + 1) <= INT32_MAX;
}

size_t walk_words(int64_t nseg, int64_t L, int64_t D, int dtype, int64_t k) {
  const int ks = walk_slots(k);
  int64_t most = 0;  // the unit size depends on the pointers: room for any of them
  for (int ub = dtype_size(dtype); ub <= 16; ub *= 2) {
    if ((D * dtype_size(dtype)) % ub) break;
    const int64_t n = state_words(nseg, L, D, dtype, ks, ub);
    if (n > most) most = n;
  }
  return (size_t)most;
}

hipError_t tape_walk(const void* keys, bool wide, int tbits, bool same, bool fwd, const Tape& tp,
                     int64_t D, int dtype, const void* sum_in, const void* val_in, int64_t k,
                     void* out, uint8_t* omask, void* val_out, uint8_t* vmask, uint64_t* words,
                     hipStream_t s) {
  const int64_t row = D * dtype_size(dtype);
  if (!walk_applies(tp, D, dtype, k) || !tp.status) return hipErrorInvalidValue;
  const int ub = unit_bytes(dtype, row, (uintptr_t)sum_in | (uintptr_t)val_in | (uintptr_t)out |
                                            (uintptr_t)val_out);
  if (!ub) return hipErrorInvalidValue;
  WalkArgs a;
  a.keys = keys;
  a.wide = wide ? 1 : 0;
  a.same = same ? 1 : 0;
  a.tbits = tbits;
  a.nseg = tp.nseg();
  a.T = tp.T;
  a.L = same ? tp.T : 2 * tp.T;
  a.C = tp.C;
  a.part = walk_part(a.nseg, a.L);
  a.nparts = (a.L + a.part - 1) / a.part;
  walk_columns(dtype, row, ub, &a.gtot, &a.G, &a.ncb);
  if (a.ncb > 65535 || a.nseg * a.nparts > INT32_MAX) return hipErrorInvalidValue;
  a.sum_in = sum_in;
  a.val_in = val_in;
  a.k = k > 0 ? (int)k : 1;
  a.out = out;
  a.omask = omask;
  a.val_out = val_out;
  a.vmask = vmask;
  a.tickets = words;
  a.words = words + a.nseg * a.ncb;
  a.err = tp.status;
  const int ks = val_in || val_out ? walk_slots(k) : 0;
  hipError_t e = hipErrorInvalidValue;
  switch (dtype) {
    case kF32: e = tape_walk_f32(a, ub, ks, fwd, s); break;
    case kF64: e = tape_walk_f64(a, ub, ks, fwd, s); break;
    case kBF16: e = tape_walk_bf16(a, ub, ks, fwd, s); break;
    case kF16: e = tape_walk_f16(a, ub, ks, fwd, s); break;
    default: break;
  }
  // latest-1: both masks are the same bytes, and a copy in order costs less than
  // a second byte at every random record (5 us against 13 at 4.2M records)
  if (e == hipSuccess && val_out && k == 1) e = copy_bytes(vmask, omask, (size_t)tp.n(), s);
  return e;
}

Tape merged_tape(const Tape& tp) {
  Tape m = make_tape(tp.B, 2 * tp.T, tp.C, tp.A, true, kNegLast);
  m.status = tp.status;
  return m;
}

// The smallest kind that holds [0, A]: 2, 4 or 8 bytes.
int merged_kind(int64_t A) { return A < 65536 ? kU16 : A < ((int64_t)1 << 32) ? kU32 : kI64; }

size_t merged_bytes(const Tape& tp) {
  const int kind = merged_kind(tp.A);
  return (size_t)(2 * tp.n()) * (kind == kU16 ? 2 : kind == kU32 ? 4 : 8);
}

hipError_t merge_addresses(const AddrIn& wa, const AddrIn& ra, const uint8_t* wmask, const Tape& tp,
                           void* buf, AddrIn* out, hipStream_t s) {
  const int64_t N = tp.n();
  if (N == 0 || N > INT32_MAX || wa.kind != ra.kind) return hipErrorInvalidValue;
  out->kind = merged_kind(tp.A);
  out->dense = buf;
  const FastDiv by_c = make_fastdiv((uint32_t)tp.C);
  const unsigned grid = (unsigned)((N + 1023) / 1024);
  return with_addr(wa, tp, [&](auto w) {
    auto r = w;
    r.p = (decltype(w.p))ra.dense;
    auto go = [&](auto* o) {
      merge_addresses_kernel<<<grid, 256, 0, s>>>(w, r, wmask, N, tp.T, (uint32_t)tp.C, by_c, tp.A,
                                                  tp.trunc32 ? 1 : 0, o);
      return hipGetLastError();
    };
    switch (out->kind) {
      case kU16: return go((uint16_t*)buf);
      case kU32: return go((uint32_t*)buf);
      default: return go((int64_t*)buf);
    }
  });
}

}  // namespace rem
