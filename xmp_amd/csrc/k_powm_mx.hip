// k_powm_mx.hip -- modular exponentiation on the matrix cores.
//
// One wave holds one instance.  A Montgomery product is three N-byte products
// (x y, then q = low(x y) m' mod R, then q m; R = 256^N), each a contraction
// that v_mfma_i32_16x16x64_i8 sums exactly.
//
// Digits are balanced bytes (-128 .. 127).  With N = 16 S, digit 16 u + v of a
// product is
//   P[16u + v] = sum_{s,t} Y[16 s + v - t] X[16 (u - s) + t],   t = 0 .. 15,
// a 16 x 16 tile (rows v, columns u) of a matrix product over k = (s, t): the
// rows' operand is 16-byte windows of Y at byte offsets (T fragments), the
// columns' operand whole 16-byte blocks of X (C fragments).  Lane (g, i) of
// the wave, g = lane / 16, i = lane % 16, supplies row or column i at
// s = 4 kb + g, so a C fragment depends on u0 - 4 kb alone and is shared by
// the tiles; within a fragment both operands run t downwards, so windows of Y
// are read as stored and X is stored with the bytes of each block reversed.
// An accumulator tile leaves four consecutive digits in a lane, which are one
// 32-bit limb: limb 4 (16 r + i) + g of tile r.
//
// Carries: a tile's accumulators start at 128 per digit, so a lane's
// sum s = d0 + 2^8 d1 + 2^16 d2 + 2^24 d3 is the limb's balanced bytes plus
// 0x80808080, its low word taken as is.  Its high word (a few bits, signed)
// moves one limb up by one cross-lane move; what that addition carries is
// almost always nothing (a chance of 2^-15 a limb), and then resolved by
// rounds of the same move.  No digit is ever unpacked.
//
// Values stay balanced, |x| <= 0.502 R, for any m < R: q is balanced, so
// (x y + q m) / R is at most 0.252 R + 0.502 m, and the top limb's high word
// k, seen before any carry, says whether m is to be subtracted or added once
// (k m is subtracted whatever k is: no branch on the values but for the rare
// carries' rounds).
// The low half of x y + q m is zero mod R; what it carries into the high half
// is its top limb's total, rounded, of which a few digits are enough
// (low_carry).  m' = -1/m mod R comes from Newton's iteration on the same
// products.
#include <type_traits>

#include "devmp.hpp"
#include "powm.hpp"

namespace xmp {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr uint32_t kBias = 0x80808080u;

__device__ __forceinline__ void mx_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// -m0^-1 mod 2^32 for odd m0
__device__ __forceinline__ uint32_t neg_inverse32(uint32_t m0) {
  uint32_t inv = m0;
#pragma unroll
  for (int it = 0; it < 4; it++) inv = inv * (2u - m0 * inv);
  return 0u - inv;
}

// s + k m for a small signed k, with no branch on it
__device__ __forceinline__ int64_t add_multiple(int64_t s, int32_t k, uint32_t m) {
  const uint64_t x = (uint64_t)s + (uint64_t)(uint32_t)k * m;
  return (int64_t)(x - ((uint64_t)(m & (uint32_t)(k >> 31)) << 32));
}

// MP_LDS keeps m' in LDS, as fragments, instead of S registers: from 48 blocks
// on a second wave then fits the SIMD.
template <int S, bool MP_LDS>
struct Mx {
  static_assert(S % 4 == 0 && S >= 4, "whole k-blocks");
  static constexpr int N = 16 * S;            // bytes of R
  static constexpr int LIMBS = 4 * S;
  static constexpr int T = (S + 15) / 16;     // tiles of a half product
  static constexpr int KB = S / 4;            // k-blocks of s = 0 .. S-1; k-block KB holds s = S
  static constexpr int NF = (S + 12) / 4 + 1; // C fragments, u0 - 4 kb = -12 .. S
  static constexpr int NQ = 4 * (T - 1) + 4;  // those of a low half product, -12 .. 16 (T-1)
  static constexpr int DOTS = T == 1 ? 2 : 3; // digits of q m's top low limb that are summed,
  static constexpr int UNIT = T == 1 ? 16 : 18;   // in units of 2^UNIT: at most 2^31 - 2^22 in all
  static constexpr int TOP = (S - 1) % 16;    // column of the top limb in the last tile
  static constexpr bool PART = S % 16 != 0;   // the last tile's columns past TOP hold nothing
  static constexpr int C_BYTES = 16 * (S + 31);   // blocks -15 .. S+15
  static constexpr int T_BYTES = 16 * (S + 6);    // bytes -16 .. 16 (S+5) - 1
  static constexpr int LDS_BYTES = C_BYTES + T_BYTES + (MP_LDS ? 1024 * KB : 0);

  uint8_t *cb, *tb;     // LDS: X by reversed blocks, Y plain
  const uint8_t *cread; // this lane's C fragments (offset 16 (u0 - 4 kb + 12))
  const uint8_t *tread; // this lane's T fragments (offset 64 kb)
  int lane, i, g, rot;
  uint32_t tshift;
  int32_t k8, k16, k24;      // 2^8, 2^16, 2^24 in registers, for v_mad_i64_i32
  v4i bias4;
  v4i mp[MP_LDS ? 1 : KB];   // T fragments of m' and m
  v4i mt[KB + 1];
  uint32_t mw[T];            // this lane's limbs of m
  int wm[T][DOTS];           // the digits of m that meet this lane's digits in a low half's top digits

  __device__ __forceinline__ Mx(uint8_t *lds) {
    lane = threadIdx.x;
    i = lane & 15;
    g = lane >> 4;
    cb = lds;
    tb = lds + C_BYTES;
    cread = cb + 16 * (3 + i - g);
    tread = tb + 16 * g + ((1 + i) & ~3);
    tshift = (uint32_t)(1 + i) & 3u;
    rot = 4 * (g ? lane - 16 : (i ? 47 + i : 63));
    asm volatile("s_mov_b32 %0, 0x100" : "=s"(k8));
    asm volatile("s_mov_b32 %0, 0x10000" : "=s"(k16));
    asm volatile("s_mov_b32 %0, 0x1000000" : "=s"(k24));
    asm volatile("v_mov_b32 %0, 0x80" : "=v"(bias4.x));
    bias4 = v4i{bias4.x, bias4.x, bias4.x, bias4.x};
    for (int b = lane; b < (C_BYTES + T_BYTES) / 16; b += 64) *reinterpret_cast<v4i *>(lds + 16 * b) = v4i{0, 0, 0, 0};
    mx_fence();
  }

  __device__ __forceinline__ bool live(int r) const { return !PART || r < T - 1 || i <= TOP; }
  __device__ __forceinline__ uint32_t limb(int r) const { return (uint32_t)(4 * (16 * r + i) + g); }
  __device__ __forceinline__ static int top_lane(int r) { return r < T - 1 ? 63 : 48 + TOP; }

  // the digits of e, as bytes: plain for T fragments, reversed blocks for C
  __device__ __forceinline__ void put_c(const uint32_t (&e)[T]) const {
#pragma unroll
    for (int r = 0; r < T; r++)
      *reinterpret_cast<uint32_t *>(cb + 16 * (15 + 16 * r + i) + 4 * (3 - g)) = __builtin_bswap32(e[r] ^ kBias);
  }
  __device__ __forceinline__ void put_t(const uint32_t (&e)[T]) const {
#pragma unroll
    for (int r = 0; r < T; r++)
      if (live(r)) *reinterpret_cast<uint32_t *>(tb + 16 + 16 * (16 * r + i) + 4 * g) = e[r] ^ kBias;
  }
  __device__ __forceinline__ v4i cfrag(int f) const { return *reinterpret_cast<const v4i *>(cread + 64 * f); }
  // 16 bytes at this lane's byte offset, from the five words that hold them
  // (a byte-aligned 16-byte LDS read takes seven times an aligned one)
  __device__ __forceinline__ v4i tfrag(int kb) const {
    const uint32_t *w = reinterpret_cast<const uint32_t *>(tread + 64 * kb);
    v4i x;
    x.x = (int)__builtin_amdgcn_alignbyte(w[1], w[0], tshift);
    x.y = (int)__builtin_amdgcn_alignbyte(w[2], w[1], tshift);
    x.z = (int)__builtin_amdgcn_alignbyte(w[3], w[2], tshift);
    x.w = (int)__builtin_amdgcn_alignbyte(w[4], w[3], tshift);
    return x;
  }

  // 128 a digit: with one tile its two chains start at 64 each (an inline
  // constant of the instruction), with more the tiles share a register
  __device__ __forceinline__ v4i bias() const { return T == 1 ? v4i{64, 64, 64, 64} : bias4; }
  __device__ __forceinline__ static v4i bias2() { return v4i{64, 64, 64, 64}; }
  __device__ __forceinline__ v4i *mp_lds() const { return reinterpret_cast<v4i *>(tb + T_BYTES) + lane; }
  __device__ __forceinline__ v4i mpfrag(int kb) const { return MP_LDS ? mp_lds()[64 * kb] : mp[kb]; }
  static __device__ __forceinline__ v4i mfma(v4i t, v4i c, v4i acc) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(t, c, acc, 0, 0, 0);
  }

  __device__ __forceinline__ int64_t sum(v4i a) const {
    return (int64_t)a.w * k24 + ((int64_t)a.z * k16 + ((int64_t)a.y * k8 + a.x));
  }

  // the limb above takes c[r]; tile 0's first limb takes cin.  Returns what
  // leaves the top limb.
  __device__ __forceinline__ int32_t move_up(int32_t (&c)[T], int32_t cin) const {
#pragma unroll
    for (int r = 0; r < T; r++) {
      const int32_t top = __builtin_amdgcn_readlane(c[r], top_lane(r));
      const int32_t up = __builtin_amdgcn_ds_bpermute(rot, c[r]);
      c[r] = lane == 0 ? cin : (live(r) ? up : 0);
      cin = top;
    }
    return cin;
  }

  // e = lo + c moved up, resolved; returns the carry out of the top limb
  __device__ __forceinline__ int32_t resolve(uint32_t (&e)[T], const uint32_t (&lo)[T], int32_t (&c)[T],
                                             int32_t cin) const {
    int32_t out = move_up(c, cin);
    bool any = false;
#pragma unroll
    for (int r = 0; r < T; r++) {
      const int64_t x = (int64_t)(uint64_t)lo[r] + c[r];
      e[r] = (uint32_t)x;
      c[r] = (int32_t)(x >> 32);
      any |= c[r] != 0;
    }
    while (__builtin_amdgcn_ballot_w64(any) != 0) {
      out += move_up(c, 0);
      any = false;
#pragma unroll
      for (int r = 0; r < T; r++) {
        const int64_t x = (int64_t)(uint64_t)e[r] + c[r];
        e[r] = (uint32_t)x;
        c[r] = (int32_t)(x >> 32);
        any |= c[r] != 0;
      }
    }
    return out;
  }

  // biased digits of a half product's tiles; returns the carry out
  __device__ __forceinline__ int32_t digits(uint32_t (&e)[T], const v4i (&a)[T], int32_t cin) const {
    uint32_t lo[T];
    int32_t c[T];
#pragma unroll
    for (int r = 0; r < T; r++) {
      const int64_t s = sum(a[r]);
      lo[r] = live(r) ? (uint32_t)s : kBias;
      c[r] = live(r) ? (int32_t)(s >> 32) : 0;
    }
    return resolve(e, lo, c, cin);
  }

  // the same for limb sums s of a value to be kept within 0.502 R by adding
  // or subtracting m
  __device__ __forceinline__ void digits_mod(uint32_t (&e)[T], int64_t (&s)[T], int32_t cin) const {
    for (int it = 0; it < 4; it++) {
      const int32_t k = -__builtin_amdgcn_readlane((int32_t)(s[T - 1] >> 32), top_lane(T - 1));
#pragma unroll
      for (int r = 0; r < T; r++) s[r] = add_multiple(s[r], k, mw[r]);
      uint32_t lo[T];
      int32_t c[T];
#pragma unroll
      for (int r = 0; r < T; r++) {
        lo[r] = live(r) ? (uint32_t)s[r] : kBias;
        c[r] = live(r) ? (int32_t)(s[r] >> 32) : 0;
      }
      const int32_t out = resolve(e, lo, c, cin);
      if (out == 0) break;
      // the top limb's own carry was not seen above (rare): once more
      cin = 0;
#pragma unroll
      for (int r = 0; r < T; r++)
        s[r] = (int64_t)(uint64_t)e[r] + (r == T - 1 && lane == top_lane(r) ? (int64_t)out << 32 : 0);
    }
  }

  // low half of (T fragments from tf) * (X in LDS), and its carry out
  template <class F>
  __device__ __forceinline__ int32_t low_product(uint32_t (&e)[T], const F &tf, int32_t cin) const {
    v4i cf[NQ], a[T], b = bias2();
#pragma unroll
    for (int f = 0; f < NQ; f++) cf[f] = cfrag(f);
    if (T == 1) __builtin_amdgcn_sched_barrier(0);   // all reads in flight before the first use
#pragma unroll
    for (int r = 0; r < T; r++) a[r] = bias();
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      const v4i t = tf(kb);
#pragma unroll
      for (int r = 0; r < T; r++)
        if (kb < 4 * r + 4) {
          if (T == 1 && kb % 2 == 1) b = mfma(t, cf[4 * r - kb + 3], b);
          else a[r] = mfma(t, cf[4 * r - kb + 3], a[r]);
        }
    }
    if (T == 1) a[0] += b;
    return digits(e, a, cin);
  }

  // What the low half of x y + q m carries out, for the biased digits q and x
  // y's top low limb.  The half's total is a whole number of R, so its top
  // limb's, rounded, is enough: the limbs below it move it by less than
  // 2^-15.  Of q m's part of it the top two digits are summed (the third
  // adds less than 2^30 = 2^22 2^8 with one tile), or the top three.  A few
  // multiply-adds a lane and a sum over the wave; as one more tile of the
  // matrix product it took S/4 instructions, as many LDS reads and a limb sum
  // (2048 bits x 12,288 12.1 ms, now 10.1; 1536 x 12,288 7.8, now 6.6).
  __device__ __forceinline__ int32_t low_carry(const uint32_t (&q)[T], uint32_t low_top) const {
    int32_t x = 0;
#pragma unroll
    for (int d = 0; d < DOTS; d++) {
      int32_t t = 0;
#pragma unroll
      for (int r = 0; r < T; r++) t = __builtin_amdgcn_sdot4((int)(q[r] ^ kBias), wm[r][d], t, false);
      x += 24 - 8 * d >= UNIT ? t << ((24 - 8 * d - UNIT) & 31) : t >> ((UNIT - 24 + 8 * d) & 31);
    }
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr 1, 2, 4, 8
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, true);   // row_bcast 15, 31
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, true);
    const int32_t top = (int32_t)((uint32_t)__builtin_amdgcn_readlane((int)low_top, top_lane(T - 1)) >> UNIT);
    return (__builtin_amdgcn_readlane(x, 63) + top - (int32_t)(kBias >> UNIT) + (1 << (31 - UNIT))) >> (32 - UNIT);
  }

  // e = x y / R mod m for X in LDS (which this overwrites) and Y's T
  // fragments.  XTOP: X has a digit of its own in block S, cleared once read.
  template <bool XTOP = false, class F>
  __device__ __forceinline__ void mont(uint32_t (&e)[T], const F &tf) const {
    v4i hi[T], h2 = bias2();
    uint32_t q[T];
    int32_t carry;
    {
      v4i cf[NF], lo[T], l2 = bias2();
#pragma unroll
      for (int f = 0; f < NF; f++) cf[f] = cfrag(f);
      if (T == 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < T; r++) lo[r] = hi[r] = bias();
#pragma unroll
      for (int kb = 0; kb <= KB; kb++) {
        const v4i t = tf(kb);
#pragma unroll
        for (int r = 0; r < T; r++) {
          if (kb < KB && kb < 4 * r + 4) {
            if (T == 1 && kb % 2 == 1) l2 = mfma(t, cf[4 * r - kb + 3], l2);
            else lo[r] = mfma(t, cf[4 * r - kb + 3], lo[r]);
          }
          if (kb >= 4 * r) {
            if (T == 1 && kb % 2 == 1) h2 = mfma(t, cf[KB + 4 * r - kb + 3], h2);
            else hi[r] = mfma(t, cf[KB + 4 * r - kb + 3], hi[r]);
          }
        }
      }
      if (T == 1) lo[0] += l2;
      carry = digits(q, lo, 0);
    }
    const uint32_t low_top = q[T - 1];
    mx_fence();
    if (XTOP && lane == 0) cb[16 * (15 + S) + 15] = 0;
    put_c(q);
    mx_fence();
    (void)low_product(q, [&](int kb) { return mpfrag(kb); }, 0);
    mx_fence();
    put_c(q);
    mx_fence();
    carry += low_carry(q, low_top);
    v4i cf[NF];
#pragma unroll
    for (int f = 3; f < NF; f++) cf[f] = cfrag(f);
    if (T == 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kb = 0; kb <= KB; kb++) {
#pragma unroll
      for (int r = 0; r < T; r++)
        if (kb >= 4 * r) {
          if (T == 1 && kb % 2 == 1) h2 = mfma(mt[kb], cf[KB + 4 * r - kb + 3], h2);
          else hi[r] = mfma(mt[kb], cf[KB + 4 * r - kb + 3], hi[r]);
        }
    }
    if (T == 1) hi[0] += h2;
    int64_t s[T];
#pragma unroll
    for (int r = 0; r < T; r++) s[r] = sum(hi[r]);
    digits_mod(e, s, carry);
  }

  // m and m' into their fragments; returns whether m is odd and not 1
  __device__ __forceinline__ bool load_modulus(const Operand &mod, uint32_t mi) {
    uint32_t lo[T], e[T], z[T];
    int32_t c[T];
    bool other = false;
#pragma unroll
    for (int r = 0; r < T; r++) {
      mw[r] = live(r) ? ld_limb(mod, mi, limb(r)) : 0u;
      other |= mw[r] != (limb(r) == 0 ? 1u : 0u);
      const uint64_t x = (uint64_t)mw[r] + kBias;
      lo[r] = (uint32_t)x;
      c[r] = (int32_t)(x >> 32);
    }
    const bool not_one = __builtin_amdgcn_ballot_w64(other) != 0;
    const uint32_t m0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)mw[0]);
    // the digits past the top limb's: 0 or 1
    const int32_t top = resolve(e, lo, c, 0);
    put_t(e);
    if (lane == 0) tb[16 + N] = (uint8_t)top;
    mx_fence();
#pragma unroll
    for (int kb = 0; kb <= KB; kb++) mt[kb] = tfrag(kb);
#pragma unroll
    for (int r = 0; r < T; r++) {
      // digits N-1-d-4l down to N-4-d-4l, the highest first
      const uint32_t *w = reinterpret_cast<const uint32_t *>(tb + 16 + N - 8 - (live(r) ? 4 * (int)limb(r) : 0));
#pragma unroll
      for (int d = 0; d < DOTS; d++)
        wm[r][d] = live(r) ? (int)__builtin_bswap32(d ? __builtin_amdgcn_alignbyte(w[1], w[0], 4 - d) : w[1]) : 0;
    }
    mx_fence();
    if (lane == 0) tb[16 + N] = 0;
    // z = -1/m mod 2^32, then z (2 + m z) doubles the correct bits
#pragma unroll
    for (int r = 0; r < T; r++) {
      const uint64_t x = (uint64_t)(limb(r) == 0 ? neg_inverse32(m0) : 0u) + kBias;
      lo[r] = (uint32_t)x;
      c[r] = (int32_t)(x >> 32);
    }
    (void)resolve(z, lo, c, 0);
#pragma unroll 1
    for (int bits = 32; bits < 8 * N; bits *= 2) {
      put_c(z);
      put_t(z);
      mx_fence();
      (void)low_product(e, [&](int kb) { return mt[kb]; }, 2);
      mx_fence();
      put_c(e);
      mx_fence();
      (void)low_product(z, [&](int kb) { return tfrag(kb); }, 0);
      mx_fence();
    }
    put_t(z);
    mx_fence();
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      if (MP_LDS) mp_lds()[64 * kb] = tfrag(kb);
      else mp[kb] = tfrag(kb);
    }
    mx_fence();
    return not_one && (m0 & 1u) != 0;
  }
};

// Moduli of up to eight blocks: the whole product is one tile of 2 S columns,
// its low half in columns 0 .. S-1 and its high half, where the values live,
// in S .. 2S-1.  The tile of x y is the accumulator of q m, so the top low
// limb's total already holds everything that the low half carries: its
// rounded high word moves to the first high limb with the other high words,
// and what x y's low digits carry out is not needed for anything else.  Eight
// matrix instructions and three limb sums a product at S = 8, where the two
// tiles of the longer moduli would take twelve and four: a wave's serial chain
// and the matrix cores both shorten.  Measured at 1024 bits x 4,096 1.27 ms
// (two tiles: 1.42), x 64 0.71 (0.82); 512 bits x 2,048 0.38 (0.44).
template <int S>
struct MxHalf {
  static_assert(S == 4 || S == 8, "one tile");
  static constexpr int N = 16 * S, LIMBS = 4 * S, T = 1, KB = S / 4;
  static constexpr int C_BYTES = 16 * 31, T_BYTES = 16 * (S + 6), LDS_BYTES = C_BYTES + T_BYTES;
  static constexpr int TOP_LOW = 47 + S, TOP = 47 + 2 * S;   // lanes of the halves' top limbs

  uint8_t *cb, *tb;
  const uint8_t *cread, *tread;
  int lane, i, g, rot;
  uint32_t tshift;
  bool low, high;
  uint8_t *clow, *chigh, *twrite;
  int32_t k8, k16, k24;
  v4i mp[KB], mt[KB + 1];
  uint32_t mw[1];   // the high lane's limb of m

  __device__ __forceinline__ MxHalf(uint8_t *lds) {
    lane = threadIdx.x;
    i = lane & 15;
    g = lane >> 4;
    low = i < S;
    high = i >= S && i < 2 * S;
    cb = lds;
    tb = lds + C_BYTES;
    cread = cb + 16 * (15 + i - g);
    tread = tb + 16 * g + ((1 + i) & ~3);
    tshift = (uint32_t)(1 + i) & 3u;
    rot = 4 * (g ? lane - 16 : (i ? 47 + i : 63));
    clow = cb + 16 * (15 + i) + 4 * (3 - g);
    chigh = cb + 16 * (15 + ((i - S) & 15)) + 4 * (3 - g);
    twrite = tb + 16 + 16 * (i - S) + 4 * g;
    asm volatile("s_mov_b32 %0, 0x100" : "=s"(k8));
    asm volatile("s_mov_b32 %0, 0x10000" : "=s"(k16));
    asm volatile("s_mov_b32 %0, 0x1000000" : "=s"(k24));
    for (int b = lane; b < (C_BYTES + T_BYTES) / 16; b += 64) *reinterpret_cast<v4i *>(lds + 16 * b) = v4i{0, 0, 0, 0};
    mx_fence();
  }

  __device__ __forceinline__ bool live(int) const { return high; }
  __device__ __forceinline__ uint32_t limb(int) const { return (uint32_t)(4 * (i - S) + g); }

  // (lanes outside a value's half hold zero digits)
  __device__ __forceinline__ void put_c(const uint32_t (&e)[1]) const {
    *reinterpret_cast<uint32_t *>(chigh) = __builtin_bswap32(e[0] ^ kBias);
  }
  __device__ __forceinline__ void put_c_low(uint32_t e) const {
    *reinterpret_cast<uint32_t *>(clow) = __builtin_bswap32(e ^ kBias);
  }
  __device__ __forceinline__ void put_t(const uint32_t (&e)[1]) const {
    if (high) *reinterpret_cast<uint32_t *>(twrite) = e[0] ^ kBias;
  }
  __device__ __forceinline__ v4i cfrag(int kb) const { return *reinterpret_cast<const v4i *>(cread - 64 * kb); }
  __device__ __forceinline__ v4i tfrag(int kb) const {
    const uint32_t *w = reinterpret_cast<const uint32_t *>(tread + 64 * kb);
    v4i x;
    x.x = (int)__builtin_amdgcn_alignbyte(w[1], w[0], tshift);
    x.y = (int)__builtin_amdgcn_alignbyte(w[2], w[1], tshift);
    x.z = (int)__builtin_amdgcn_alignbyte(w[3], w[2], tshift);
    x.w = (int)__builtin_amdgcn_alignbyte(w[4], w[3], tshift);
    return x;
  }
  static __device__ __forceinline__ v4i mfma(v4i t, v4i c, v4i acc) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(t, c, acc, 0, 0, 0);
  }
  __device__ __forceinline__ int64_t sum(v4i a) const {
    return (int64_t)a.w * k24 + ((int64_t)a.z * k16 + ((int64_t)a.y * k8 + a.x));
  }

  // e = lo + the high words c, moved up a limb within one half (`mine`), until
  // nothing carries.  Lanes outside it give only what a caller leaves in the
  // lane below its first limb.  Returns what leaves the half's top limb
  // (lane `top`).
  template <bool OUT>
  __device__ __forceinline__ int32_t resolve(uint32_t &e, uint32_t lo, int32_t c, bool mine, int top) const {
    int32_t out = 0;
    e = lo;
    do {
      if (OUT) out += __builtin_amdgcn_readlane(c, top);
      const int32_t up = __builtin_amdgcn_ds_bpermute(rot, c);
      const int64_t x = (int64_t)(uint64_t)e + (mine ? up : 0);
      e = (uint32_t)x;
      c = (int32_t)(x >> 32);
    } while (__builtin_amdgcn_ballot_w64(c != 0) != 0);
    return out;
  }
  __device__ __forceinline__ int32_t resolve(uint32_t (&e)[1], const uint32_t (&lo)[1], int32_t (&c)[1], int32_t) const {
    return resolve<true>(e[0], lo[0], c[0], high, TOP);
  }
  // the low half's balanced digits, what they carry out dropped
  __device__ __forceinline__ void low_digits(uint32_t &e, v4i a) const {
    const int64_t s = sum(a);
    resolve<false>(e, low ? (uint32_t)s : kBias, low ? (int32_t)(s >> 32) : 0, low, TOP_LOW);
  }

  // the high half's digits of limb sums s, within 0.502 R; from_low joins the
  // first high limb (lane TOP_LOW's value)
  __device__ __forceinline__ void digits_mod(uint32_t (&e)[1], int64_t (&s)[1], int32_t from_low) const {
    for (int it = 0; it < 4; it++) {
      s[0] = add_multiple(s[0], -__builtin_amdgcn_readlane((int32_t)(s[0] >> 32), TOP), mw[0]);
      const int32_t c = high ? (int32_t)(s[0] >> 32) : (lane == TOP_LOW ? from_low : 0);
      const int32_t out = resolve<true>(e[0], high ? (uint32_t)s[0] : kBias, c, high, TOP);
      if (out == 0) break;
      from_low = 0;
      s[0] = (int64_t)(uint64_t)e[0] + (lane == TOP ? (int64_t)out << 32 : 0);
    }
  }

  // the low half of (T fragments from tf) * (X in LDS)
  template <class F>
  __device__ __forceinline__ void low_product(uint32_t &e, const F &tf, int32_t plus) const {
    const v4i half = v4i{64, 64, 64, 64};
    v4i a = mfma(tf(0), cfrag(0), half), b = half;
    if (KB == 2) b = mfma(tf(KB - 1), cfrag(KB - 1), half);
    a += b;
    if (lane == 0) a.x += plus;
    low_digits(e, a);
  }

  template <bool XTOP = false, class F>
  __device__ __forceinline__ void mont(uint32_t (&e)[1], const F &tf) const {
    const v4i half = v4i{64, 64, 64, 64}, zero = v4i{0, 0, 0, 0};
    uint32_t q;
    v4i p;
    {
      v4i c[KB + 1], t[KB + 1];
#pragma unroll
      for (int kb = 0; kb <= KB; kb++) {
        c[kb] = cfrag(kb);
        t[kb] = tf(kb);
      }
      p = mfma(t[0], c[0], half);
      const v4i b = mfma(t[1], c[1], half);
      if (KB == 2) p = mfma(t[KB], c[KB], p);
      p += b;
    }
    low_digits(q, p);
    mx_fence();
    if (XTOP && lane == 0) cb[16 * (15 + S) + 15] = 0;
    put_c_low(q);
    mx_fence();
    low_product(q, [&](int kb) { return mp[kb]; }, 0);
    mx_fence();
    put_c_low(q);
    mx_fence();
    v4i c[KB + 1];
#pragma unroll
    for (int kb = 0; kb <= KB; kb++) c[kb] = cfrag(kb);
    p = mfma(mt[0], c[0], p);
    const v4i b = mfma(mt[1], c[1], zero);
    if (KB == 2) p = mfma(mt[KB], c[KB], p);
    p += b;
    int64_t s[1] = {sum(p)};
    // (lane TOP_LOW: the low half's total is a whole number of R)
    digits_mod(e, s, (int32_t)((s[0] + (0x80000000ll - (int64_t)kBias)) >> 32));
  }

  __device__ __forceinline__ bool load_modulus(const Operand &mod, uint32_t mi) {
    mw[0] = high ? ld_limb(mod, mi, limb(0)) : 0u;
    const bool not_one = __builtin_amdgcn_ballot_w64(mw[0] != (lane == S ? 1u : 0u)) != 0;
    const uint32_t m0 = (uint32_t)__builtin_amdgcn_readlane((int)mw[0], S);
    uint32_t e[1], z;
    const uint64_t x = (uint64_t)mw[0] + kBias;
    const int32_t top = resolve<true>(e[0], (uint32_t)x, (int32_t)(x >> 32), high, TOP);
    put_t(e);
    if (lane == 0) tb[16 + N] = (uint8_t)top;
    mx_fence();
#pragma unroll
    for (int kb = 0; kb <= KB; kb++) mt[kb] = tfrag(kb);
    mx_fence();
    if (lane == 0) tb[16 + N] = 0;
    // z = -1/m mod 2^32 on the low lanes, then z (2 + m z) doubles the correct bits
    const uint64_t y = (uint64_t)(lane == 0 ? neg_inverse32(m0) : 0u) + kBias;
    resolve<false>(z, (uint32_t)y, (int32_t)(y >> 32), low, TOP_LOW);
    uint8_t *tlow = tb + 16 + 16 * i + 4 * g;
#pragma unroll 1
    for (int bits = 32; bits < 8 * N; bits *= 2) {
      put_c_low(z);
      if (low) *reinterpret_cast<uint32_t *>(tlow) = z ^ kBias;
      mx_fence();
      low_product(e[0], [&](int kb) { return mt[kb]; }, 2);
      mx_fence();
      put_c_low(e[0]);
      mx_fence();
      low_product(z, [&](int kb) { return tfrag(kb); }, 0);
      mx_fence();
    }
    if (low) *reinterpret_cast<uint32_t *>(tlow) = z ^ kBias;
    mx_fence();
#pragma unroll
    for (int kb = 0; kb < KB; kb++) mp[kb] = tfrag(kb);
    mx_fence();
    return not_one && (m0 & 1u) != 0;
  }
};

// R^2 mod m is 2^(5/4 8N) mod m, from a division, squared twice.  Each squaring
// less costs the division as many quotient bits again as it had: with nine to
// thirteen of them (a division of a few bits) 2048 bits x 12,288 took 0.33 ms
// with 32-bit exponents and 8192 x 2,048 0.49, with two 0.295 and 0.43, with
// none 0.297 and 0.436.
constexpr uint32_t kR2Squarings = 2;

// One wave an instance.  r2 holds 2^(5/4 8N) mod m.
template <int S, int WAVES, bool MP_LDS = false>
__global__ void __launch_bounds__(64, WAVES) powm_mx_kernel(PowmArgs args) {
  using M = std::conditional_t<(S <= 8), MxHalf<S <= 8 ? S : 8>, Mx<S, MP_LDS>>;
  constexpr int T = M::T;
  __shared__ __attribute__((aligned(16))) uint8_t lds[M::LDS_BYTES];
  const uint32_t local = blockIdx.x;
  const uint32_t gi = args.start + local;
  const uint32_t bi = in_index(args.base, gi), ei = in_index(args.exp, gi), mi = in_index(args.mod, gi);
  M mx(lds);
  const bool valid = mx.load_modulus(args.mod, mi);
  const uint32_t wbits = args.window_bits;
  uint32_t *table = args.table + ((size_t)local << wbits) * M::LIMBS;
  auto store_entry = [&](uint32_t x, const uint32_t (&e)[T]) {
#pragma unroll
    for (int r = 0; r < T; r++)
      if (mx.live(r)) table[(size_t)x * M::LIMBS + mx.limb(r)] = e[r];
  };
  auto load_entry = [&](uint32_t (&e)[T], uint32_t x) {
#pragma unroll
    for (int r = 0; r < T; r++) e[r] = mx.live(r) ? table[(size_t)x * M::LIMBS + mx.limb(r)] : kBias;
  };
  auto from_lds = [&](int kb) { return mx.tfrag(kb); };

  uint32_t e[T];
  int64_t s[T];
  // R^2 mod m
#pragma unroll
  for (int r = 0; r < T; r++) {
    const uint32_t w = mx.limb(r);
    s[r] = (int64_t)kBias + (mx.live(r) && w < args.mod.len ? args.r2[(size_t)w * args.r2_stride + mi] : 0u);
  }
  mx.digits_mod(e, s, 0);
  for (uint32_t j = 0; j < kR2Squarings; j++) {
    mx.put_c(e);
    mx.put_t(e);
    mx_fence();
    mx.mont(e, from_lds);
    mx_fence();
  }
  mx.put_t(e);
  // slot 0 = R mod m = 1 * R^2 / R
#pragma unroll
  for (int r = 0; r < T; r++) e[r] = mx.limb(r) == 0 ? kBias + 1u : kBias;
  mx.put_c(e);
  mx_fence();
  mx.mont(e, from_lds);
  mx_fence();
  store_entry(0, e);
  // slot 1 = base R mod m; a base at or above R/2 has one more digit, 1
  {
    uint32_t lo[T];
    int32_t c[T];
#pragma unroll
    for (int r = 0; r < T; r++) {
      const uint64_t x = (uint64_t)(mx.live(r) ? ld_limb(args.base, bi, mx.limb(r)) : 0u) + kBias;
      lo[r] = (uint32_t)x;
      c[r] = (int32_t)(x >> 32);
    }
    const int32_t top = mx.resolve(e, lo, c, 0);
    mx.put_c(e);
    mx_fence();
    if (mx.lane == 0) mx.cb[16 * (15 + S) + 15] = (uint8_t)top;
    mx_fence();
    mx.template mont<true>(e, from_lds);
    mx_fence();
  }
  store_entry(1, e);
  mx.put_c(e);
  mx.put_t(e);
  mx_fence();
  for (uint32_t x = 2; x < (1u << wbits); x++) {
    mx.mont(e, from_lds);
    mx_fence();
    store_entry(x, e);
    mx.put_c(e);
    mx_fence();
  }
  // every lane's table stores before any lane's loads
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");

  // exponent scan, top window first
  auto window = [&](uint32_t pos, uint32_t len) {
    const uint32_t w = pos >> 5;
    return funnel(ld_limb(args.exp, ei, w + 1), ld_limb(args.exp, ei, w), pos & 31) & ((1u << len) - 1);
  };
  const uint32_t bits = args.exp.len * 32;
  uint32_t pos = bits - ((bits % wbits) ? (bits % wbits) : wbits);
  load_entry(e, window(pos, bits - pos));
  while (pos > 0) {
    pos -= wbits;
    uint32_t f[T];   // the window's entry, on its way during the squarings
    load_entry(f, window(pos, wbits));
    for (uint32_t k = 0; k <= wbits; k++) {
      mx.put_c(e);
      if (k < wbits)
        mx.put_t(e);
      else
        mx.put_t(f);
      mx_fence();
      mx.mont(e, from_lds);
      mx_fence();
    }
  }
  // out of Montgomery form: x * 1 / R, at most 0.502 (m + 1) either way
  mx.put_c(e);
#pragma unroll
  for (int r = 0; r < T; r++) e[r] = mx.limb(r) == 0 ? kBias + 1u : kBias;
  mx.put_t(e);
  mx_fence();
  mx.mont(e, from_lds);
  uint32_t lo[T];
  int32_t c[T];
#pragma unroll
  for (int r = 0; r < T; r++) {
    const int64_t x = mx.live(r) ? (int64_t)(uint64_t)e[r] - (int64_t)kBias : 0;
    lo[r] = (uint32_t)x;
    c[r] = (int32_t)(x >> 32);
  }
  if (mx.resolve(e, lo, c, 0) < 0) {
#pragma unroll
    for (int r = 0; r < T; r++) {
      const uint64_t x = (uint64_t)e[r] + mx.mw[r];
      lo[r] = (uint32_t)x;
      c[r] = (int32_t)(x >> 32);
    }
    (void)mx.resolve(e, lo, c, 0);
  }
  uint32_t *out = args.out.data + out_index(args.out, gi);
#pragma unroll
  for (int r = 0; r < T; r++) {
    const uint32_t w = mx.limb(r);
    // an even modulus is outside Montgomery's domain: defined result 0
    if (mx.live(r) && w < args.out.len) out[(size_t)w * args.out.stride] = valid ? e[r] : 0u;
  }
}

// `crowded`: two waves a SIMD instead of one, for more instances than the GPU
// has SIMDs.  8192 bits x 8,192 with 256-bit exponents 8.15 -> 6.05 ms, x 2,048
// 2.14 -> 1.73; up to 1,024 instances the wave alone is faster (1.10 against
// 1.23; 6144 bits 0.73, 0.78).  Below 48 blocks the registers hold two waves
// as they are, and a third or fourth gains less than m' in LDS costs (3072 and
// 4096 bits within 5 % either way).
constexpr uint32_t kSimds = 1024;
struct MxEntry {
  uint32_t blocks;
  void (*kernel)(PowmArgs), (*crowded)(PowmArgs);
};
const MxEntry kMx[] = {
    {4, powm_mx_kernel<4, 4>, powm_mx_kernel<4, 4>},    {8, powm_mx_kernel<8, 4>, powm_mx_kernel<8, 4>},
    {12, powm_mx_kernel<12, 4>, powm_mx_kernel<12, 4>}, {16, powm_mx_kernel<16, 4>, powm_mx_kernel<16, 4>},
    {20, powm_mx_kernel<20, 3>, powm_mx_kernel<20, 3>}, {24, powm_mx_kernel<24, 3>, powm_mx_kernel<24, 3>},
    {28, powm_mx_kernel<28, 2>, powm_mx_kernel<28, 2>}, {32, powm_mx_kernel<32, 2>, powm_mx_kernel<32, 2>},
    {40, powm_mx_kernel<40, 2>, powm_mx_kernel<40, 2>}, {48, powm_mx_kernel<48, 1>, powm_mx_kernel<48, 2, true>},
    {56, powm_mx_kernel<56, 1>, powm_mx_kernel<56, 2, true>}, {64, powm_mx_kernel<64, 1>, powm_mx_kernel<64, 2, true>},
};

}  // namespace

uint32_t powm_mx_blocks(uint32_t precision) {
  for (const MxEntry &e : kMx)
    if (128u * e.blocks >= precision) return e.blocks;
  return 0;
}

// Where the matrix cores are faster than the lane layouts: up to a batch size
// that depends on the modulus.  A wave finishes one instance in a quarter to
// a tenth of a lane group's time, but a full GPU multiplies 64-bit digits of
// short moduli faster; and the lane layouts take the same time for any part
// of the 16,384 or 32,768 instances that fill the GPU, so that past a whole
// number of those the matrix cores are ahead again.  Measured on one MI355X,
// this kernel against the lane layouts, in ms:
//   exponents as long as the moduli: 160 bits x 512 0.127, 0.133; 256 x 256
//   0.179, 0.199, x 1,024 0.191, 0.199 (2,048: 0.207, 0.199); 288 x 3,072 0.256,
//   0.285; 384 x 3,072 0.32, 0.78 (4,096: 0.38, 0.35); 512 x 8,192 0.85, 1.04; 544 x 3,072
//   0.54, 1.12 (4,096: 0.64, 0.63); 768 x 6,144 1.20, 1.61; 1024 x 7,168 1.86,
//   2.14 (8,192: 2.22, 2.13); 1056 x 4,096 1.83, 1.91 (6,144: 2.63, 2.58);
//   1536 x 12,288 6.9, 8.4 (16,384: 9.0, 8.5; 20,480: 10.9, 15.6); 2048 x
//   1,024 1.9, 6.7, x 16,384 13.4, 14.3 (32,768: 26.0, 24.8; 65,536: 51, 47);
//   256-bit exponents: 672 x 6,144 0.49, 0.51 (7,168: 0.54, 0.52); 1280 x
//   6,144 0.69, 0.85 (12,288: 1.32, 1.21); 1568 x 24,576 2.9, 3.1 (28,672:
//   3.3, 3.1); 1664 x 28,672 3.4, 3.9; 2048 x 28,672 3.5, 3.7, x 57,344 6.7,
//   7.0; 2176 x 6,144 1.26, 1.70 (16,384: 3.2, 2.7); 2304 x 16,384 3.2, 3.4
//   (32,768: 6.1, 5.9); 2368 x 65,536 12.1, 14.5; 3072 x 65,536 14.4, 15.4;
//   32-bit exponents, where the set-up weighs more: 1312 x 12,288 0.245, 0.208;
//   1536 x 14,336 0.254, 0.269; 2048 x 16,384 0.331, 0.338, x 24,576 0.50,
//   0.59; 3072 x 65,536 2.42, 2.52; 4096 x 65,536 3.3, 4.2.
bool powm_mx_pays(uint32_t precision, uint32_t exp_bits, uint32_t count) {
  if (precision <= 128 || count >> 26) return false;   // (a wave an instance: a grid has fewer than 2^32 threads)
  if (precision <= 256) return count <= 1024;
  if (precision <= 480) return count <= 3072;
  if (precision <= 512) return count <= 8192;
  if (precision <= 640) return count <= 3072;
  if (precision <= 704) return count <= 6144;
  if (precision <= 1024) return count <= 7168;
  if (precision <= 1152) return count <= 4096;
  if (precision <= 1312) return count <= 6144;
  if (precision <= 1600) return count <= 14336 || (count > 16384 && count <= 24576 && exp_bits > 64);
  if (precision <= 2048) return count <= (exp_bits <= 64 ? 24576ull : 28672ull) * (((uint64_t)count + 32767) / 32768);
  if (precision <= 2208) return count <= 6144;
  if (precision <= 2304) return count <= 16384;
  return true;
}

size_t powm_mx_table_words(uint32_t blocks, uint32_t count, uint32_t window_bits) {
  return ((size_t)count << window_bits) * 4 * blocks;
}

hipError_t launch_mx_r2(uint32_t blocks, uint32_t *r2, uint32_t r2_stride, const uint32_t *m, uint32_t m_len,
                        uint32_t m_stride, uint32_t count, hipStream_t stream) {
  const uint32_t rbits = 128u * blocks;
  return launch_pow2_mod(r2, m_len, r2_stride, m, m_len, m_stride, count, rbits + (rbits >> kR2Squarings), nullptr,
                         stream);
}

hipError_t launch_powm_mx(uint32_t blocks, const PowmArgs &args, hipStream_t stream) {
  for (const MxEntry &e : kMx)
    if (e.blocks == blocks && args.count != 0) {
      hipLaunchKernelGGL(args.count > kSimds ? e.crowded : e.kernel, dim3(args.count), dim3(64), 0, stream, args);
      return hipGetLastError();
    }
  return hipErrorInvalidValue;
}

}  // namespace xmp
