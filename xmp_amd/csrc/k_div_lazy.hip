// k_div_lazy.hip -- long division without carry chains.
//
// Reference: src/div.cu:35-517, digitmp/div.h:108-423 (schoolbook digits with
// estimate, multiply-subtract and add-back).  Here the quotient digits are
// signed and the remainder is never carried:
//
//  * operands are radix-2^D digits (D = 28, or 27 and 26 for longer divisors),
//    the divisor V shifted up to ND = L*K digits with its top bit set, the
//    remainder ND signed 64-bit lazy sums.
//    A step takes the next dividend digit in, R' = 2^D R + u, and subtracts
//    q V with q the nearest integer to R' / V: one v_mad_i64_i32 per digit,
//    where 32-bit limbs with borrows cost a multiply-add and two
//    subtractions, in one serial chain from digit to digit;
//  * q comes from the top three sums in double precision: what they leave
//    out, and the rounding, move R'/V by less than 2^-14, so |R| stays below
//    (1/2 + 2^-14) V, no digit is ever corrected, and adding 1.5 * 2^52 in
//    the last multiply-add leaves -q in the low word;
//  * a sum gains little more than 2^(2D-1) a step and leaves the window after
//    ND steps: below 2^63 for 160 digits at D = 28, 304 at 27 and 1,280 at 26.
//    The top sum, folded into the one below it, is small because R is;
//  * a division spans L lanes of K digits, the top digits on the group's
//    first lane, whose q the others take by the same DPP moves as the
//    Montgomery quotient; one 64-bit sum moves a lane up a step;
//  * the dividend's digits wait in LDS, each replaced by its quotient digit;
//    at the end R is carried once (V added and the quotient lowered by one
//    if it is negative) and the signed quotient digits once.
//
// Division by zero writes q = 0 and r = a.
#include <algorithm>

#include "devmp.hpp"
#include "kernels.hpp"
#include "lanes.hpp"
#include "powm.hpp"

namespace xmp {

namespace {

// digits whose bits are whole limbs (a lane fetches 14, 13 or 27 limbs at a time)
template <int D>
constexpr int kRun = D == 27 ? 32 : 16;
// digits and limbs of an aligned piece of a result
template <int D>
constexpr int kPieceDigits = D == 28 ? 8 : D == 27 ? 32 : 16;
template <int D>
constexpr int kPieceLimbs = kPieceDigits<D> * D / 32;

// Dividends and divisors.  load<N>: limbs k0 .. k0 + N - 1, 0 outside
// [0, len), all loads unconditional, at limbs that exist, and masked (a select
// lets the compiler put a load under a branch, and then every load waits for
// the one before).  Where every lane's limbs exist the row's address is
// scalar and a lane's offset one register for all of them.
struct ArrayDividend {
  const uint32_t *data;
  uint32_t stride, len, inst;
  template <int N>
  __device__ __forceinline__ void load(uint32_t (&x)[N], int32_t k0) const {
    const bool inside = k0 >= 0 && k0 + N <= (int32_t)len && (uint64_t)len * stride < (1ull << 30);
    if (__builtin_amdgcn_ballot_w64(!inside) == 0) {
      const uint32_t off = ((uint32_t)k0 * stride + inst) * 4u;
#pragma unroll
      for (int k = 0; k < N; k++)
        x[k] = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(data + (size_t)k * stride) + off);
    } else {
#pragma unroll
      for (int k = 0; k < N; k++) {
        const int32_t kc = min(max(k0 + k, 0), (int32_t)len - 1);
        const uint32_t v = data[(size_t)(uint32_t)kc * stride + inst], m = kc == k0 + k ? ~0u : 0u;
        x[k] = v & m;
      }
    }
  }
  __device__ __forceinline__ uint32_t limb(int32_t k) const {
    uint32_t x[1];
    load<1>(x, k);
    return x[0];
  }
};
struct PowerDividend {   // 2^e
  uint32_t e, len;
  __device__ __forceinline__ uint32_t limb(int32_t k) const {
    return k >= 0 && (uint32_t)k == (e >> 5) ? 1u << (e & 31) : 0u;
  }
  template <int N>
  __device__ __forceinline__ void load(uint32_t (&x)[N], int32_t k0) const {
#pragma unroll
    for (int k = 0; k < N; k++) x[k] = limb(k0 + k);
  }
};

// N digits from bit `off` (0 .. 31) of limb w up (they may lie below 0 or past the top)
template <int D, int N, class Dividend>
__device__ __forceinline__ void digits_at(uint32_t (&d)[N], const Dividend &a, int32_t w, uint32_t off) {
  constexpr int NW = (D * N + 31) / 32;
  uint32_t x[NW + 1];
  a.template load<NW + 1>(x, w);
#pragma unroll
  for (int j = 0; j < NW; j++) x[j] = funnel(x[j + 1], x[j], off);
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int j = (D * k) >> 5, s = (D * k) & 31;
    d[k] = (s + D <= 32 ? x[j] >> s : funnel(x[j + 1 < NW ? j + 1 : j], x[j], s)) & ((1u << D) - 1);
  }
}

// piece m's limbs of an integer whose radix-2^D digits 0 .. n-1 are at d, taken
// from digit `skip` and bit s (0 .. D-1) of it up
template <int D>
__device__ __forceinline__ void piece_limbs(uint32_t (&w)[kPieceLimbs<D>], const uint32_t *d, int32_t n, int32_t m,
                                            int32_t skip, uint32_t s) {
  constexpr int P = kPieceDigits<D>;
  uint32_t x[P + 1];
#pragma unroll
  for (int k = 0; k <= P; k++) {
    const int32_t at = P * m + skip + k;
    const uint32_t v = d[min(at, n - 1)], keep = at < n ? ~0u : 0u;
    x[k] = v & keep;
  }
#pragma unroll
  for (int k = 0; k < P; k++) x[k] = (x[k] >> s) | ((x[k + 1] << (D - s)) & ((1u << D) - 1));
#pragma unroll
  for (int j = 0; j < kPieceLimbs<D>; j++) {
    const int k = 32 * j / D, b = 32 * j - D * k;
    w[j] = (x[k] >> b) | (x[k + 1] << (D - b));
    if (2 * D - b < 32) w[j] |= x[k + 2 < P ? k + 2 : k] << (2 * D - b);
  }
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int L, int K, int D>
struct Lazy {
  static constexpr int ND = L * K;
  static constexpr uint32_t MASK = (1u << D) - 1;
  static_assert(K >= 3 && (double)(ND + 1) * (double)(1ull << (2 * D - 1)) < 9.2e18,
                "the estimate's digits on one lane; sums below 2^63");
  const Group<L> g;
  __device__ __forceinline__ explicit Lazy(int lane) : g(lane) {}

  // the next lane's (lower digits') value, 0 on the group's last lane
  __device__ __forceinline__ int64_t from_below(int64_t x) const {
    if constexpr (L == 1) return 0;
    const uint32_t lo = g.from_next((uint32_t)x), hi = g.from_next((uint32_t)(x >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
  }
  // every lane's copy of the group's first lane's value
  __device__ __forceinline__ uint32_t top(uint32_t x) const { return g.bcast0(x); }

  // r = the sums' digits; returns the signed carry out of the top digit (0 or -1 for |R| < V)
  __device__ __forceinline__ int32_t carry(uint32_t (&r)[K], const int64_t (&t)[K]) const {
    int64_t c = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int64_t x = t[k] + c;
      r[k] = (uint32_t)x & MASK;
      c = x >> D;
    }
    int32_t out = (int32_t)c;
    if constexpr (L > 1) {
      for (int round = 1; round < L; round++) {
        c = from_below(c);
        if (__builtin_amdgcn_ballot_w64(c != 0) == 0) break;
#pragma unroll
        for (int k = 0; k < K; k++) {
          const int64_t x = (int64_t)r[k] + c;
          r[k] = (uint32_t)x & MASK;
          c = x >> D;
        }
        out += (int32_t)c;
      }
    }
    return (int32_t)top((uint32_t)out);
  }
};

struct LazyOut {
  uint32_t *q, *r;   // nullable, at the instance's column
  uint32_t q_len, q_stride, r_len, r_stride;
};

// digits an instance's LDS row holds: the dividend's below the first window
// (at most all of them, and one), or the remainder's
__host__ __device__ inline uint32_t lazy_row(uint32_t a_len, uint32_t nd, uint32_t d) {
  const uint32_t n = (32u * a_len + d - 1) / d + 2;
  return (n > nd ? n : nd) | 1u;   // odd: the groups' rows start in different banks
}

template <int L, int K, int D, class Dividend>
__device__ __forceinline__ void divide_lazy(const Dividend &A, const ArrayDividend &B, const LazyOut &o, uint32_t *row,
                                            bool active) {
  using Z = Lazy<L, K, D>;
  constexpr int ND = Z::ND;
  constexpr uint32_t MASK = Z::MASK;
  const Z z(threadIdx.x & 63);
  const int l = z.g.l;
  const int32_t base = (L - 1 - l) * K;   // this lane's lowest digit

  // the divisor's length in bits, from the top
  int32_t bits = 0;
  for (int32_t k = (int32_t)B.len - 1;; k -= L) {
    const uint32_t x = B.limb(k - l);
    if (x) bits = max(bits, 32 * (k - l) + 32 - __builtin_clz(x));
    if constexpr (L > 1) {
#pragma unroll
      for (int d = 1; d < L; d <<= 1) bits = max(bits, __shfl_xor(bits, d, L));
    }
    if (k < L || __builtin_amdgcn_ballot_w64(bits == 0) == 0) break;
  }
  const bool zero = bits == 0;
  // dividends of fewer limbs: q = 0 and r = a where the divisor is the longer
  if (A.len < B.len && __builtin_amdgcn_ballot_w64(!zero && bits <= (int32_t)(32 * A.len)) == 0) {
    if (active && o.q)
      for (uint32_t k = (uint32_t)l; k < o.q_len; k += L) o.q[(size_t)k * o.q_stride] = 0u;
    if (o.r)
      for (uint32_t k0 = 8 * (uint32_t)l; k0 < o.r_len; k0 += 8 * L) {
        uint32_t x[8];
        A.template load<8>(x, (int32_t)k0);
        if (active) {
#pragma unroll
          for (uint32_t k = 0; k < 8; k++)
            if (k0 + k < o.r_len) o.r[(size_t)(k0 + k) * o.r_stride] = x[k];
        }
      }
    return;
  }
  const int32_t sh = D * ND - bits;
  int32_t v[K];
  {
    uint32_t x[K];
    const int32_t at = D * base - sh;
    digits_at<D, K>(x, B, at >> 5, (uint32_t)at & 31u);
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = (int32_t)x[k];
  }
  // -1 / (the top digits), on the group's first lane
  const double vt = (double)v[K - 1] + (double)v[K - 2] * (1.0 / (double)(1u << D));
  const double ninv = zero ? 0.0 : -1.0 / vt;

  // quotient digits: those of the wave's shortest divisor, the same count for all
  int32_t nq = (int32_t)(32 * A.len) - bits;
  nq = nq < 0 ? 1 : (nq + D - 1) / D + 1;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) nq = max(nq, __shfl_xor(nq, d, 64));
  nq = __builtin_amdgcn_readfirstlane(nq);
  const int32_t most = (int32_t)((32 * A.len + D - 1) / D) + 1;
  nq = nq < most ? nq : most;

  // the dividend's digits below the window, a run of them a lane at a time
  // (whole limbs, so every run starts at the same bit of one)
  constexpr int RUN = kRun<D>;
  for (int32_t j = l; RUN * j < nq; j += L) {
    uint32_t x[RUN];
    digits_at<D, RUN>(x, A, D * RUN / 32 * j + (-sh >> 5), (uint32_t)-sh & 31u);
#pragma unroll
    for (int k = 0; k < RUN; k++)
      if (RUN * j + k < nq) row[RUN * j + k] = x[k];
  }
  // the window starts as the ND - 1 digits above digit nq - 1 of a 2^sh
  int64_t t[K];
  {
    uint32_t x[K];
    const int32_t at = D * (nq + base) - sh;
    digits_at<D, K>(x, A, at >> 5, (uint32_t)at & 31u);
#pragma unroll
    for (int k = 0; k < K; k++) t[k] = base + k < ND - 1 ? (int64_t)(uint64_t)x[k] : 0;
  }
  wave_sync();

  uint32_t u = row[nq - 1];
  for (int32_t j = nq - 1; j >= 0; j--) {
    const uint32_t un = row[j > 0 ? j - 1 : 0];
    // R' at the top digit's weight; the top two sums exactly, the third's high word
    const int64_t y = (int64_t)((uint64_t)t[K - 1] << D) + t[K - 2];
    const double f = __builtin_fma((double)(int32_t)(y >> 32), 0x1p32, (double)(uint32_t)y);
    const double e = __builtin_fma((double)(int32_t)(t[K - 3] >> 32), (double)(1u << (32 - D)), f);
    const double m = __builtin_fma(e, ninv, 0x1.8p52);
    const int32_t q = (int32_t)z.top((uint32_t)__builtin_bit_cast(uint64_t, m));   // -q
    const int64_t below = z.from_below(t[K - 1]);
    const bool first = L == 1 || l == 0, last = L == 1 || l == L - 1;
    t[K - 1] = (first ? y : t[K - 2]) + (int64_t)q * v[K - 1];
#pragma unroll
    for (int k = K - 2; k > 0; k--) t[k] = t[k - 1] + (int64_t)q * v[k];
    t[0] = (last ? (int64_t)(uint64_t)u : below) + (int64_t)q * v[0];
    row[j] = (uint32_t)-q;
    u = un;
  }
  // carry R; negative: one V more and one less in the quotient
  uint32_t r[K];
  const int32_t sign = z.carry(r, t);
  if (__builtin_amdgcn_ballot_w64(sign < 0) != 0) {
#pragma unroll
    for (int k = 0; k < K; k++) t[k] = (int64_t)r[k] + (sign < 0 ? v[k] : 0);
    (void)z.carry(r, t);
  }
  wave_sync();
  constexpr uint32_t W = kPieceLimbs<D>;
  if (o.q) {
    // carry the quotient's digits: each lane a run of them, then its borrow
    // up the runs while there is one
    const int32_t run = (nq + L - 1) / L;
    const int32_t lo = min(l * run, nq), hi = min(lo + run, nq);
    int32_t c = l == 0 && sign < 0 ? -1 : 0;
    for (int32_t k = lo; k < hi; k += 8) {
      int32_t x[8];
#pragma unroll
      for (int i = 0; i < 8; i++) x[i] = (int32_t)row[min(k + i, hi - 1)];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int32_t y = x[i] + c;
        if (k + i < hi) {
          row[k + i] = (uint32_t)y & MASK;
          c = y >> D;
        }
      }
    }
    if constexpr (L > 1) {
      for (int round = 1; round < L; round++) {
        c = (int32_t)__shfl_up(c, 1, L);
        if (l == 0) c = 0;
        if (__builtin_amdgcn_ballot_w64(c != 0) == 0) break;
        for (int32_t k = lo; k < hi && c != 0; k++) {
          const int32_t x = (int32_t)row[k] + c;
          row[k] = (uint32_t)x & MASK;
          c = x >> D;
        }
      }
    }
    wave_sync();
    for (uint32_t m = (uint32_t)l; W * m < o.q_len; m += L) {
      uint32_t w[W];
      piece_limbs<D>(w, row, nq, (int32_t)m, 0, 0);
      if (active) {
#pragma unroll
        for (uint32_t j = 0; j < W; j++)
          if (W * m + j < o.q_len) o.q[(size_t)(W * m + j) * o.q_stride] = zero ? 0u : w[j];
      }
    }
  }
  if (o.r) {
    wave_sync();
#pragma unroll
    for (int k = 0; k < K; k++) row[base + k] = r[k];
    wave_sync();
    const int32_t skip = sh / D;
    for (uint32_t m = (uint32_t)l; W * m < o.r_len; m += L) {
      uint32_t w[W];
      piece_limbs<D>(w, row, ND, (int32_t)m, skip, (uint32_t)(sh - D * skip));
      if (active) {
#pragma unroll
        for (uint32_t j = 0; j < W; j++) {
          const uint32_t k = W * m + j;
          if (k < o.r_len) o.r[(size_t)k * o.r_stride] = zero ? A.limb((int32_t)k) : w[j];
        }
      }
    }
  }
}

// one wave a workgroup, 64 / L divisions
template <int L, int K, int D>
__global__ void __launch_bounds__(64) divmod_lazy_kernel(OutOperand q, OutOperand r, Operand a, Operand b,
                                                         uint32_t count) {
  extern __shared__ uint32_t div_rows[];
  const uint32_t grp = threadIdx.x / L;
  const uint32_t t = blockIdx.x * (64 / L) + grp;
  const bool active = t < count;
  const uint32_t i = active ? t : count - 1;   // groups past the end divide the last pair and store nothing
  LazyOut o{};
  if (q.data) {
    o.q = q.data + out_index(q, i);
    o.q_len = q.len;
    o.q_stride = q.stride;
  }
  if (r.data) {
    o.r = r.data + out_index(r, i);
    o.r_len = r.len;
    o.r_stride = r.stride;
  }
  const ArrayDividend A{a.data, a.stride, a.len, in_index(a, i)}, B{b.data, b.stride, b.len, in_index(b, i)};
  divide_lazy<L, K, D>(A, B, o, div_rows + grp * lazy_row(a.len, L * K, D), active);
}

// 2^e mod m
template <int L, int K, int D>
__global__ void __launch_bounds__(64) pow2_mod_lazy_kernel(uint32_t *out, uint32_t out_len, uint32_t out_stride,
                                                           const uint32_t *m, uint32_t m_len, uint32_t m_stride,
                                                           uint32_t count, uint32_t e) {
  extern __shared__ uint32_t div_rows[];
  const uint32_t grp = threadIdx.x / L;
  const uint32_t t = blockIdx.x * (64 / L) + grp;
  const bool active = t < count;
  const uint32_t i = active ? t : count - 1;
  LazyOut o{};
  o.r = out + i;
  o.r_len = out_len;
  o.r_stride = out_stride;
  const PowerDividend A{e, (e >> 5) + 1};
  const ArrayDividend B{m, m_stride, m_len, i};
  divide_lazy<L, K, D>(A, B, o, div_rows + grp * lazy_row(A.len, L * K, D), active);
}

struct LazyEntry {
  uint32_t lanes, digits, radix;
  void (*div)(OutOperand, OutOperand, Operand, Operand, uint32_t);
  void (*pow2)(uint32_t *, uint32_t, uint32_t, const uint32_t *, uint32_t, uint32_t, uint32_t, uint32_t);
};
#define XMP_LAZY(L, K, D) {L, K, D, divmod_lazy_kernel<L, K, D>, pow2_mod_lazy_kernel<L, K, D>}
const LazyEntry kLazy[] = {
    XMP_LAZY(4, 5, 28),   XMP_LAZY(8, 5, 28),   XMP_LAZY(16, 5, 28),  XMP_LAZY(4, 10, 28), XMP_LAZY(8, 10, 28),
    XMP_LAZY(16, 10, 28), XMP_LAZY(1, 28, 28),  XMP_LAZY(2, 28, 28),  XMP_LAZY(4, 28, 28), XMP_LAZY(1, 37, 28),
    XMP_LAZY(2, 37, 28),  XMP_LAZY(4, 37, 28),  XMP_LAZY(2, 19, 28),  XMP_LAZY(4, 19, 28), XMP_LAZY(8, 19, 28),
    XMP_LAZY(16, 15, 27), XMP_LAZY(8, 29, 27),  XMP_LAZY(32, 10, 27), XMP_LAZY(16, 19, 27), XMP_LAZY(8, 38, 27),
    XMP_LAZY(64, 10, 26), XMP_LAZY(16, 40, 26), XMP_LAZY(64, 20, 26),
};
#undef XMP_LAZY

// The lanes a division takes: few for a full batch, whose steps are bound by
// issue (K multiply-adds and about 20 other instructions a lane), many for a
// small one, whose steps are bound by the estimate's latency.  For a divisor
// that `digits` hold, batches up to `count` take the entry.  Measured on one
// MI355X, us: 2048/1024 bits x 300 (8,5) 10.6, (4,10) 12.0, (1,37) 18.8; x
// 16,384 18.4, 13.9, 19.6; x 65,536 41, 29, 24; 4096/2048 x 300 (16,5) 14.1,
// (8,10) 16.4, (4,19) 20, (2,37) 26; x 16,384 38, 30, 27, 29; x 65,536 121,
// 78, 56, 48; 8192/4096 x 300 (16,10) 23, (8,19) 29, (4,37) 39; x 16,384 75,
// 55, 49.  Against the 32-bit kernels, one and two lanes a division with
// borrow chains: 4096/2048 x 300 51 us, x 65,536 71, x 131,072 109 (here 86);
// 8192/4096 x 32,768 144 (here 72); 1024/512 x 300 12.2 (here (4,5) 9.0), x
// 65,536 14.0 (here 14.1 and more: up to 512-bit divisors only small batches
// come here, and none up to 256 bits).
//   Longer divisors, against one wave a division with 32-bit limbs in LDS:
// 12288/6144 x 100 (16,15) 37, 199, x 16,384 (8,29) 98, 752; 16384/8192 x 100
// (32,10) 43, 291, x 4,096 (16,19) 68, 402, x 16,384 (8,38) 146, 1084;
// 24576/16384 x 100 (64,10) 43, 415, x 4,096 (16,40) 102, 578; 49152/32000 x
// 1,024 (64,20) 129, 1822.
struct LazyRule {
  uint32_t limbs, count, lanes, digits, radix;
};
constexpr uint32_t kAny = 0xFFFFFFFFu;
const LazyRule kRules[] = {
    {16, 16384, 4, 5, 28},
    {24, 4096, 8, 5, 28},    {24, 32768, 4, 10, 28},  {24, kAny, 1, 28, 28},
    {32, 4096, 8, 5, 28},    {32, 32768, 4, 10, 28},  {32, kAny, 1, 37, 28},
    {33, 4096, 8, 5, 28},    {33, 32768, 4, 10, 28},  {33, kAny, 2, 19, 28},
    {35, 4096, 8, 5, 28},    {35, 32768, 4, 10, 28},  {35, kAny, 2, 28, 28},
    {49, 2048, 16, 5, 28},   {49, 8192, 8, 10, 28},   {49, 16384, 4, 19, 28},  {49, kAny, 2, 28, 28},
    {64, 2048, 16, 5, 28},   {64, 8192, 8, 10, 28},   {64, 24576, 4, 19, 28},  {64, kAny, 2, 37, 28},
    {66, 2048, 16, 5, 28},   {66, 8192, 8, 10, 28},   {66, kAny, 4, 19, 28},
    {98, 2048, 16, 10, 28},  {98, 8192, 8, 19, 28},   {98, kAny, 4, 28, 28},
    {129, 2048, 16, 10, 28}, {129, 8192, 8, 19, 28},  {129, kAny, 4, 37, 28},
    {195, 8192, 16, 15, 27}, {195, kAny, 8, 29, 27},
    {256, 512, 32, 10, 27},  {256, 8192, 16, 19, 27}, {256, kAny, 8, 38, 27},
    {520, 2048, 64, 10, 26}, {520, kAny, 16, 40, 26},
    {1040, kAny, 64, 20, 26},
};
constexpr size_t kLazyLds = 64 * 1024, kCuLds = 160 * 1024;
constexpr uint32_t kCuInstances = 256 * 64;   // instances of one lane that are a wave a CU

size_t lazy_lds(const LazyRule &r, uint32_t a_len) {
  return 4 * (size_t)(64 / r.lanes) * lazy_row(a_len, r.lanes * r.digits, r.radix);
}

// The rule for a division, or null for the 32-bit kernels.  Long dividends'
// rows in LDS leave a CU few waves: where those are fewer than the batch has
// for it (four are enough), a rule of more lanes, whose rows are fewer, is as
// fast or faster for the quotient's sake, and with no quotient stored where
// rows leave two.  Measured, with the quotient, against the batch's own rule:
// 5120/1024 bits x 65,536 76 and 105 us, 4480/640 72 and 86.  A dividend too long
// for its rows takes the first of the divisor's rules that holds it.
const LazyRule *lazy_rule(uint32_t a_len, uint32_t b_len, uint32_t count, bool quotient) {
  const LazyRule *first = nullptr, *own = nullptr, *end = kRules;
  for (const LazyRule &r : kRules) {
    if (b_len > r.limbs || (first && r.limbs != first->limbs)) continue;
    if (!first) first = &r;
    if (!own && count <= r.count) own = &r;
    end = &r + 1;
  }
  if (b_len <= 8 || !own) return nullptr;
  const size_t residents = kCuLds / lazy_lds(*own, a_len);
  if (count > 32768 && b_len <= 64 && (quotient || (b_len > 24 && residents <= 2))) {
    auto crowded = [&](const LazyRule &r) {
      const uint64_t waves = ((uint64_t)count * r.lanes + kCuInstances - 1) / kCuInstances;
      return kCuLds / lazy_lds(r, a_len) < std::min<uint64_t>(4, waves);
    };
    while (own != first && crowded(*own)) own--;
  }
  if (lazy_lds(*own, a_len) > kLazyLds)
    for (own = first; own != end && lazy_lds(*own, a_len) > kLazyLds;) own++;
  if (own == end || (count + 63ull) * own->lanes >> 32) return nullptr;   // (a grid has fewer than 2^32 threads)
  return own;
}

const LazyEntry *lazy_entry(uint32_t a_len, uint32_t b_len, uint32_t count, bool quotient) {
  if (const LazyRule *r = lazy_rule(a_len, b_len, count, quotient))
    for (const LazyEntry &e : kLazy)
      if (e.lanes == r->lanes && e.digits == r->digits && e.radix == r->radix) return &e;
  return nullptr;
}

// Divisions that the 32-bit kernels (registers up to 128 limbs, a wave each up
// to 1,040) do as fast or faster though the digits above hold them.
//
// Short quotients: a signed-digit division first finds the divisor's length and
// stages the dividend, and carries both results at its end, which takes as long
// as a few of the 32-bit kernels' limbs.  Up to so many limbs of quotient
// (dividend's limbs less divisor's) without and with the quotient stored; the
// ranges are where those kernels' registers are just filled, or where a batch
// just opens another round of this one's waves.  Measured, signed digits and
// 32-bit kernels, us: 512/512 bits x 1,000 6.0 and 4.5, 1024/1024 x 8,192 7.1
// and 6.4, x 65,536 10.9 and 9.2, 3072/3072 x 65,536 22.1 and 18.9, 6144/6144 x
// 16 12.5 and 5.2, x 1,000 13.3 and 8.3; 980/980 limbs x 30,000 1096 and 895.
struct ShortRule {
  uint32_t from, to;           // divisor's limbs
  uint32_t count_from, count_to;
  int32_t quotient, stored;    // limbs
};
const ShortRule kShort[] = {
    {9, 15, 1, 16384, 0, 2},         {16, 16, 1, 16384, 4, 5},
    {30, 32, 4097, 16384, 1, 2},     {17, 24, 16385, 32768, 1, 3},   {25, 29, 16385, 32768, 2, 4},
    {30, 32, 16385, 32768, 4, 7},    {25, 32, 32769, 98304, 2, 4},   {32, 32, 131073, 280000, 4, 10},
    {60, 64, 16385, 24576, -1, 6},   {56, 64, 65537, 98304, 4, 8},
    {72, 87, 57344, 65536, 3, 3},    {88, 96, 49152, 65536, 3, 5},   {96, 96, 131072, 135168, 4, 4},
    {96, 96, 262144, kAny, 7, 12},   {129, 129, 1, 600, 3, 4},       {130, 195, 1, 600, 8, 9},
    {130, 195, 601, 2000, 4, 5},     {130, 195, 2001, 4000, 2, 4},   {196, 256, 1, 512, 4, 6},
    {196, 256, 513, 1500, 1, 1},     {257, 384, 1, 600, 0, 1},       {750, 849, 8192, kAny, 4, 9},
    {850, 960, 8192, kAny, 6, 9},    {896, 1016, 4096, 8191, 1, 1},   {961, 1016, 8192, kAny, 2, 3},
    {1017, 1040, 3000, 11999, 5, 5}, {1017, 1040, 12000, kAny, 6, 9},
};
// Long dividends of batches that fill the lane pairs once or a few times: from
// so many limbs of dividend on, without and with the quotient stored, and for
// dividends that an index array gathers.  The 32-bit kernels read a limb of
// every instance at a time, which the caches then hold for the rows'
// neighbours; here a wave reads whole dividends, and a gather fetches most
// lines once for each instance.  Measured, us: 576/24 limbs x 58,000 379 and
// 307, 480/40 x 65,536 with the quotient 419 and 346; gathered in random order
// 384/24 x 65,536 503 and 249, 144/24 153 and 119, 288/96 454 and 351, 96/48 x
// 131,072 310 and 164.
struct LongRule {
  uint32_t from, to;           // divisor's limbs
  uint32_t count_from, count_to;
  uint32_t dividend, stored, gathered;
};
const LongRule kLong[] = {
    {17, 24, 24576, 33000, kAny, 576, 272},    {17, 24, 33001, 50000, kAny, kAny, 192},
    {17, 24, 50001, 66000, 240, 320, 144},     {17, 24, 66001, 131071, 240, 288, 144},
    {25, 32, 24576, 33000, 768, 600, 256},     {25, 32, 33001, 50000, 672, 672, 192},
    {25, 32, 50001, 66000, 448, 336, 150},     {25, 32, 66001, 131071, 384, 256, 150},
    {33, 48, 24576, 33000, 1152, 960, 288},    {33, 48, 33001, 50000, 960, 960, 320},
    {33, 48, 50001, 66000, 576, 480, 192},     {33, 48, 66001, 131071, kAny, 576, 240},
    {49, 64, 24576, 33000, 1176, 896, 294},    {49, 64, 33001, 50000, 1176, 896, 336},
    {49, 64, 50001, 66000, 448, 384, 168},     {49, 64, 66001, 131071, 448, 384, 192},
    {65, 96, 24576, 33000, 1280, 1152, 384},   {65, 96, 33001, 50000, kAny, 768, 480},
    {65, 96, 50001, 66000, 576, 576, 192},     {65, 96, 66001, 131071, kAny, kAny, 288},
    {97, 128, 24576, 33000, kAny, kAny, 448},  {97, 128, 50001, 66000, kAny, kAny, 768},
    // (above, one lane a division; those whose registers are just filled again)
    {17, 31, 131072, kAny, kAny, kAny, 72},    {32, 32, 131072, kAny, kAny, kAny, 48},
    {33, 47, 131072, 300000, kAny, kAny, 49},  {48, 48, 131072, kAny, kAny, kAny, 72},
    {49, 63, 131072, 300000, kAny, kAny, 73},  {64, 64, 131072, kAny, kAny, kAny, 96},
    {65, 79, 131072, 140000, kAny, kAny, 97},  {80, 95, 131072, 300000, kAny, kAny, 120},
    {96, 96, 131072, kAny, kAny, kAny, 144},   {97, 127, 131072, 140000, kAny, kAny, 145},
    {128, 128, 131072, kAny, kAny, kAny, 192},
};
// Long quotients of full batches: rows that leave a CU so few waves that the
// 32-bit kernels, which keep nothing in LDS, are ahead.  Measured, us: 5120/1024
// bits x 262,144 208 and 158 (with the quotient stored 313 and 182), 10752/1536
// x 131,072 349 and 258, 3072/1024 x 262,144 with the quotient 122 and 95.
bool register_division_pays(uint32_t a_len, uint32_t b_len, uint32_t count, bool quotient, bool gathered) {
  const int32_t more = a_len > b_len ? (int32_t)(a_len - b_len) : 0;
  for (const ShortRule &r : kShort)
    if (b_len >= r.from && b_len <= r.to && count >= r.count_from && count <= r.count_to &&
        more <= (quotient ? r.stored : r.quotient))
      return true;
  for (const LongRule &r : kLong)
    if (b_len >= r.from && b_len <= r.to && count >= r.count_from && count <= r.count_to &&
        a_len >= std::min(quotient ? r.stored : r.dividend, gathered ? r.gathered : kAny))
      return true;
  if (count < 131072 || b_len <= 16 || b_len > 64) return false;
  const LazyRule *r = kRules;
  while (b_len > r->limbs || count > r->count) r++;   // the batch's own rule
  const size_t residents = kCuLds / lazy_lds(*r, a_len);
  const bool loose = b_len <= 24 || (b_len > 48 && b_len <= 56);   // registers of the 32-bit kernels half filled
  return residents <= (!quotient ? (loose ? 2u : 3u) : loose ? 3u : b_len <= 32 ? 5u : 4u);
}

}  // namespace

bool divmod_lazy_takes(uint32_t a_len, uint32_t b_len, uint32_t count) {
  return lazy_entry(a_len, b_len, count, true) != nullptr;
}

bool launch_divmod_lazy(OutOperand q, OutOperand r, Operand a, Operand b, uint32_t count, hipStream_t stream,
                        hipError_t *st) {
  const LazyEntry *e = lazy_entry(a.len, b.len, count, q.data != nullptr);
  if (!e || register_division_pays(a.len, b.len, count, q.data != nullptr, a.idx != nullptr))
    return false;
  const uint32_t per = 64 / e->lanes;
  hipLaunchKernelGGL(e->div, dim3(div_round_up(count, per)), dim3(64), 4 * per * lazy_row(a.len, e->lanes * e->digits, e->radix),
                     stream, q, r, a, b, count);
  *st = hipGetLastError();
  return true;
}

bool launch_pow2_mod_lazy(uint32_t *out, uint32_t out_len, uint32_t out_stride, const uint32_t *m, uint32_t m_len,
                          uint32_t m_stride, uint32_t count, uint32_t exponent, hipStream_t stream, hipError_t *st) {
  const uint32_t a_len = (exponent >> 5) + 1;
  const LazyEntry *e = lazy_entry(a_len, m_len, count, false);
  if (!e) return false;
  const uint32_t per = 64 / e->lanes;
  hipLaunchKernelGGL(e->pow2, dim3(div_round_up(count, per)), dim3(64), 4 * per * lazy_row(a_len, e->lanes * e->digits, e->radix),
                     stream, out, out_len, out_stride, m, m_len, m_stride, count, exponent);
  *st = hipGetLastError();
  return true;
}

}  // namespace xmp
