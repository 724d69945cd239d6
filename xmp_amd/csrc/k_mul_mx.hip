// k_mul_mx.hip -- long products on the matrix cores.
//
// Reference: src/mul.cu:140-303 (any size, truncated to the output).  The
// operands become balanced bytes (-128 .. 127) in LDS and the product's
// digits the 16 x 16 tiles of an i8 contraction, as in k_powm_mx.hip: digit
// 16 u + v is the sum over k = (s, t) of Y[16 s + v - t] X[16 (u - s) + t], rows
// v from 16-byte windows of Y at byte offsets, columns u from whole blocks
// of X.  A lane's four accumulators of a tile are one 32-bit limb with a
// signed high word, which joins the limb above.
//
//  * A workgroup holds G products, W waves each.  A wave takes R consecutive
//    tiles at a time (R v4i accumulators); for k-blocks four apart, tile r + 1
//    needs the block fragment that tile r needed one step before, so each
//    step loads one fragment of X and one of Y for R matrix instructions.
//  * LDS holds X with its blocks' bytes reversed (fragments run t downwards)
//    and Y plain; a window at a byte offset is shifted out of five words (a
//    byte-aligned 16-byte LDS read takes seven times an aligned one).
//  * G neighbouring products load and store G-word rows of the interleaved
//    layout.
//  * A balanced digit's carry into limb j is decided by limb j - 1 alone
//    (0x7F7F7F80 or more) unless that limb is 0x7F7F7F7F, when the limb
//    below decides: no carry chain.
#include <algorithm>

#include "devmp.hpp"
#include "kernels.hpp"

namespace xmp {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
constexpr uint32_t kBias = 0x80808080u;
constexpr int kLoads = 4;  // operand rows that a thread has on their way at once
constexpr uint32_t kMaxThreads = 512, kMaxLds = 64 * 1024;
constexpr int kSpan = 8;   // limbs a thread resolves of each of its workgroup's products

// One product's LDS image: X in blocks with zero blocks either side (a step's
// fragments reach 16 R + 1 blocks below and 16 R + 2 above the operand's, and
// 16 more below where the next step's are fetched ahead), Y with zeros either
// side; then, in their place, the product's limbs, the carries into them (a
// byte each) and those into a group's first limb.
template <int R>
struct MulImage {
  static constexpr uint32_t PAD = 16 * R + 20;
  uint32_t x_bytes, tiles, limbs, bytes;
  __host__ __device__ MulImage(uint32_t a_len, uint32_t b_len, uint32_t out_len) {
    x_bytes = 16 * (a_len / 4 + 1 + 2 * PAD);
    const uint32_t y_bytes = 16 * (b_len / 4 + 24);
    const uint32_t len = a_len + b_len < out_len ? a_len + b_len : out_len;
    tiles = (len + 63) / 64;
    limbs = 64 * (tiles + R);
    const uint32_t in = x_bytes + y_bytes, out = 5 * limbs + 4 + 4 * (tiles / R + 3);
    bytes = ((in > out ? in : out) + 15) / 16 * 16;
  }
};

// limb j of an operand with its balanced digits' carry added: the digits are
// the bytes of the result, exclusive-or kBias
__device__ __forceinline__ uint32_t biased_limb(const uint32_t *d, uint32_t stride, uint32_t j, uint32_t x,
                                                uint32_t below) {
  uint32_t k = j;
  while (k > 0 && below == 0x7F7F7F7Fu) {
    k--;
    below = k > 0 ? d[(size_t)(k - 1) * stride] : 0u;
  }
  return x + kBias + (k > 0 && below >= 0x7F7F7F80u ? 1u : 0u);
}

template <int G>
struct Row {
  uint32_t v[G];
};

template <int G>
__device__ __forceinline__ Row<G> load_row(const Operand &o, const uint32_t (&at)[G], bool packed, uint32_t j) {
  Row<G> r;
  const uint32_t *row = o.data + (size_t)j * o.stride;
  if (packed) {
    typedef uint32_t vec __attribute__((ext_vector_type(G > 1 ? G : 2)));
    if constexpr (G > 1) {
      const vec x = *reinterpret_cast<const vec *>(row + at[0]);
#pragma unroll
      for (int g = 0; g < G; g++) r.v[g] = x[g];
    } else {
      r.v[0] = row[at[0]];
    }
  } else {
#pragma unroll
    for (int g = 0; g < G; g++) r.v[g] = row[at[g]];
  }
  return r;
}

template <int G, int R>
__global__ void __launch_bounds__(kMaxThreads, 2) mul_mx_kernel(OutOperand p, Operand a, Operand b, uint32_t count, bool square) {
  using Image = MulImage<R>;
  extern __shared__ __attribute__((aligned(16))) uint8_t mul_lds[];
  const Image im(a.len, b.len, p.len);
  const uint32_t tid = threadIdx.x, nt = blockDim.x;
  // workgroups are dealt to the eight XCDs in turn: each XCD takes one
  // contiguous range of products, whose rows then share lines in its L2
  uint32_t wg = blockIdx.x;
  {
    const uint32_t nb = gridDim.x, x = wg & 7u, per = nb >> 3, rem = nb & 7u;
    wg = (x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + (wg >> 3);
  }
  const uint32_t i0 = wg * G;
  uint32_t ai[G], bi[G];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const uint32_t i = i0 + g < count ? i0 + g : count - 1;
    ai[g] = in_index(a, i);
    bi[g] = in_index(b, i);
  }
  const bool whole = i0 + G <= count;
  const bool apack = whole && !a.idx && a.count >= count, bpack = whole && !b.idx && b.count >= count;
  for (uint32_t k = 16 * tid; k < G * im.bytes; k += 16 * nt) *reinterpret_cast<v4i *>(mul_lds + k) = v4i{0, 0, 0, 0};
  __syncthreads();

  // operands to balanced bytes; position len holds the top carry's digit.
  // (waves walk whole spans of 64 limbs, so that a limb finds the one below
  // in the lane below)
  const int lane = tid & 63, li = lane & 15, lg = lane >> 4;
  auto digits = [&](const Operand &o, const uint32_t (&at)[G], bool packed, uint32_t j0, auto &&put) {
    // kLoads spans' rows on their way at once: a row is a memory latency
    Row<G> x[kLoads], first[kLoads];
#pragma unroll
    for (int q = 0; q < kLoads; q++) {
      const uint32_t j = j0 + q * nt + lane;
      x[q] = first[q] = Row<G>{};
      if (j < o.len) x[q] = load_row<G>(o, at, packed, j);
      if (lane == 0 && j > 0 && j <= o.len) first[q] = load_row<G>(o, at, packed, j - 1);
    }
#pragma unroll
    for (int q = 0; q < kLoads; q++) {
      const uint32_t j = j0 + q * nt + lane;
#pragma unroll
      for (int g = 0; g < G; g++) {
        const uint32_t up = (uint32_t)__shfl_up((int)x[q].v[g], 1, 64);
        const uint32_t below = lane == 0 ? first[q].v[g] : up;
        if (j <= o.len) put(g, j, biased_limb(o.data + at[g], o.stride, j, x[q].v[g], below) ^ kBias);
      }
    }
  };
  for (uint32_t j0 = tid - lane; j0 <= a.len; j0 += kLoads * nt)
    digits(a, ai, apack, j0, [&](int g, uint32_t j, uint32_t d) {
      uint8_t *img = mul_lds + g * im.bytes;
      *reinterpret_cast<uint32_t *>(img + 16 * (Image::PAD + j / 4) + 4 * (3 - (j & 3))) = __builtin_bswap32(d);
      if (square) *reinterpret_cast<uint32_t *>(img + im.x_bytes + 16 + 4 * j) = d;
    });
  if (!square)
    for (uint32_t j0 = tid - lane; j0 <= b.len; j0 += kLoads * nt)
      digits(b, bi, bpack, j0, [&](int g, uint32_t j, uint32_t d) {
        *reinterpret_cast<uint32_t *>(mul_lds + g * im.bytes + im.x_bytes + 16 + 4 * j) = d;
      });
  __syncthreads();

  const uint32_t waves = nt / (64 * G);                                    // per product
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t g = wave / waves, w = wave - g * waves;
  uint8_t *img = mul_lds + g * im.bytes;
  // the lane's fragments: X's block u - s at 16 (PAD + u - s), Y's window at
  // byte 16 s + v - 15 of the operand
  const uint32_t shift = (uint32_t)(1 + li) & 3u;
  const uint8_t *xr = img + 16 * ((int)Image::PAD + li - lg);
  const uint8_t *yr = img + im.x_bytes + 16 * lg + ((1 + li) & ~3);
  auto window = [&](const uint8_t *at) {
    const uint32_t *q = reinterpret_cast<const uint32_t *>(at);
    return v4i{(int)__builtin_amdgcn_alignbyte(q[1], q[0], shift), (int)__builtin_amdgcn_alignbyte(q[2], q[1], shift),
               (int)__builtin_amdgcn_alignbyte(q[3], q[2], shift), (int)__builtin_amdgcn_alignbyte(q[4], q[3], shift)};
  };
  const int sa = (int)(a.len / 4), kb_top = (int)((b.len / 4 + 1) / 4);
  const uint32_t ngroups = (im.tiles + R - 1) / R;
  constexpr int NHOLD = 2;   // groups whose accumulators a wave holds until all waves have read
  v4i acc[NHOLD][R];
#pragma unroll
  for (int h = 0; h < NHOLD; h++) {
#pragma unroll
    for (int r = 0; r < R; r++) acc[h][r] = v4i{0, 0, 0, 0};
    // long and short groups in turn: w from one end, then from the other
    const uint32_t grp = h == 0 ? w : ngroups - 1 - w;
    const bool mine = h == 0 ? w < (ngroups + 1) / 2 : (w < ngroups / 2);
    if (mine) {
      const int r0 = (int)grp * R;
      const int lo = 16 * r0 - sa, kmin = lo > 0 ? lo >> 2 : 0;
      const int kmax = min(kb_top, 4 * (r0 + R) - 1);
      for (int ph = 0; ph < 4; ph++) {
        const int j0 = (kmin - ph + 3) >> 2, j1 = (kmax - ph) >> 2;   // k-blocks 4 j + ph
        if (j0 > j1) continue;
        const uint8_t *xp = xr + 16 * (16 * (r0 - j0) - 4 * ph);
        const uint8_t *yp = yr + 64 * (4 * j0 + ph);
        v4i cf[R];
#pragma unroll
        for (int r = 1; r < R; r++) cf[r] = *reinterpret_cast<const v4i *>(xp + 256 * r);
        v4i xn = *reinterpret_cast<const v4i *>(xp), yn = window(yp);
        auto next = [&]() {
          xp -= 256;
          yp += 256;
          xn = *reinterpret_cast<const v4i *>(xp);
          yn = window(yp);
        };
        int n = j1 - j0 + 1;
        for (; n >= R; n -= R) {
#pragma unroll
          for (int jj = 0; jj < R; jj++) {
            const v4i t = yn;
            cf[(R - jj) % R] = xn;
            next();
#pragma unroll
            for (int r = 0; r < R; r++)
              acc[h][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(t, cf[(r - jj + R) % R], acc[h][r], 0, 0, 0);
          }
        }
        // fewer than R steps: the fragments move up a tile in registers
        for (; n > 0; n--) {
          const v4i t = yn;
          cf[0] = xn;
          next();
#pragma unroll
          for (int r = 0; r < R; r++) acc[h][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(t, cf[r], acc[h][r], 0, 0, 0);
#pragma unroll
          for (int r = R - 1; r > 0; r--) cf[r] = cf[r - 1];
        }
      }
    }
  }
  __syncthreads();
  // the limbs into the image's place: a lane's high word joins the limb above,
  // and what that carries is left for the rounds below
  uint32_t *low = reinterpret_cast<uint32_t *>(img);
  int8_t *cin = reinterpret_cast<int8_t *>(low + im.limbs);
  int32_t *gin = reinterpret_cast<int32_t *>(low + im.limbs + im.limbs / 4 + 1);
  int32_t k8, k16, k24;   // in registers, for v_mad_i64_i32
  asm volatile("s_mov_b32 %0, 0x100" : "=s"(k8));
  asm volatile("s_mov_b32 %0, 0x10000" : "=s"(k16));
  asm volatile("s_mov_b32 %0, 0x1000000" : "=s"(k24));
  const int rot = 4 * (lg ? lane - 16 : (li ? 47 + li : 63));
  if (w == 0 && lane == 0) {
    cin[0] = 0;
    gin[0] = 0;
  }
#pragma unroll
  for (int h = 0; h < NHOLD; h++) {
    const uint32_t grp = h == 0 ? w : ngroups - 1 - w;
    const bool mine = h == 0 ? w < (ngroups + 1) / 2 : (w < ngroups / 2);
    if (mine) {
      int32_t below = 0;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const uint32_t limb = 4 * (16 * (grp * R + r) + (uint32_t)li) + (uint32_t)lg;
        const v4i x = acc[h][r];
        const int64_t s = (int64_t)x.w * k24 + ((int64_t)x.z * k16 + ((int64_t)x.y * k8 + x.x));
        const int32_t hi = (int32_t)(s >> 32);
        const int32_t up = __builtin_amdgcn_ds_bpermute(rot, hi);
        const int64_t y = (int64_t)(uint64_t)(uint32_t)s + (lane == 0 ? below : up);
        below = __builtin_amdgcn_readlane(hi, 63);
        low[limb] = (uint32_t)y;
        cin[limb + 1] = (int8_t)(y >> 32);
      }
      if (lane == 0) gin[grp + 1] = below;
    }
  }
  __syncthreads();
  // carries go up a limb a round until there are none (one round but for one
  // product in some)
  const uint32_t len = min(a.len + b.len, p.len);
  bool any = true, first = true;
  while (__syncthreads_or(any)) {
    any = false;
    int32_t c[kSpan][G];
#pragma unroll
    for (int q = 0; q < kSpan; q++) {
      const uint32_t limb = q * nt + tid;
#pragma unroll
      for (int gg = 0; gg < G; gg++) {
        c[q][gg] = 0;
        if (limb < len) {
          uint32_t *lw = reinterpret_cast<uint32_t *>(mul_lds + gg * im.bytes);
          int32_t in = reinterpret_cast<const int8_t *>(lw + im.limbs)[limb];
          if (first && limb % (64 * R) == 0) in += (int32_t)lw[im.limbs + im.limbs / 4 + 1 + limb / (64 * R)];
          const int64_t x = (int64_t)(uint64_t)lw[limb] + in;
          lw[limb] = (uint32_t)x;
          c[q][gg] = (int32_t)(x >> 32);
          any |= c[q][gg] != 0;
        }
      }
    }
    first = false;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kSpan; q++) {
      const uint32_t limb = q * nt + tid;
#pragma unroll
      for (int gg = 0; gg < G; gg++)
        if (limb < len)
          reinterpret_cast<int8_t *>(reinterpret_cast<uint32_t *>(mul_lds + gg * im.bytes) + im.limbs)[limb + 1] =
              (int8_t)c[q][gg];
    }
  }
  const bool ppack = whole && !p.idx;
  for (uint32_t limb = tid; limb < p.len; limb += nt) {
    uint32_t v[G];
#pragma unroll
    for (int gg = 0; gg < G; gg++)
      v[gg] = limb < len ? reinterpret_cast<const uint32_t *>(mul_lds + gg * im.bytes)[limb] : 0u;
    uint32_t *row = p.data + (size_t)limb * p.stride;
    if (ppack) {
      if constexpr (G > 1) {
        typedef uint32_t vec __attribute__((ext_vector_type(G > 1 ? G : 2)));
        vec x;
#pragma unroll
        for (int gg = 0; gg < G; gg++) x[gg] = v[gg];
        *reinterpret_cast<vec *>(row + i0) = x;
      } else {
        row[i0] = v[0];
      }
    } else {
#pragma unroll
      for (int gg = 0; gg < G; gg++)
        if (i0 + gg < count) row[out_index(p, i0 + gg)] = v[gg];
    }
  }
}

template <int G, int R>
hipError_t launch(const OutOperand &p, const Operand &a, const Operand &b, uint32_t count, bool square,
                  hipStream_t stream) {
  const MulImage<R> im(a.len, b.len, p.len);
  // two groups of R tiles a wave at most, and kSpan limbs a thread
  const uint32_t groups = div_round_up(im.tiles, R), threads = div_round_up(64 * im.tiles, kSpan);
  const uint32_t waves = std::max((groups + 1) / 2, div_round_up(threads, 64 * G));
  if (64 * G * waves > kMaxThreads || G * im.bytes > kMaxLds) return hipErrorInvalidValue;
  hipLaunchKernelGGL((mul_mx_kernel<G, R>), dim3(div_round_up(count, G)), dim3(64 * G * waves), G * im.bytes, stream,
                     p, a, b, count, square);
  return hipGetLastError();
}

}  // namespace

// a_len >= b_len: what a workgroup's threads and LDS hold (65,536 by 65,536
// bits), and no more products than a grid, which has fewer than 2^32 threads
bool mul_mx_holds(uint32_t a_len, uint32_t b_len, uint32_t count) {
  const MulImage<4> im(a_len, b_len, a_len + b_len);
  return im.tiles <= 64 && im.bytes <= kMaxLds && (count + 1ull) * 64 * div_round_up(im.tiles, 8) >> 32 == 0;
}

// Where the matrix cores are faster than the lane kernels.  A product's wave
// or waves finish early, so batches that leave lane groups' SIMDs idle gain
// at any size; full batches gain above 4096 bits.  Measured on one MI355X,
// this kernel against the lane kernels (and Karatsuba above 16384 bits):
// 1024 bits x 1,024 6.0 against 9.1 us (squares 6.9; x 4,096 8.2, 6.9); 2048
// x 4,096 9.9, 21.6 (squares 14.6; x 8,192 16.7, 14.9); 4096 x 8,192 23, 30
// (x 16,384 38, 34); 6144 x 32,768 106, 135; 8192 x 32,768 130, 189; 16384 x
// 4,096 46, 126; 32768 x 4,096 113, 467; 65536 x 64 32, 834, x 1,024 104, 970.
// A multiplier shorter than half leaves the lane kernels little to do: 8192 x
// 1024 bits x 16,384 40, 29.  Above 16384 bits they split first, and this is
// faster by any multiplier: 552 x 1 limbs x 8,220 40, 58; 614 x 7 x 14,013 57,
// 98; 1816 x 1 x 9,238 154, 236; 3461 x 5 x 4,847 154, 363.
//   The lane kernels stop at the product's last limb that is asked for, which
// this one gains little by: 640-bit products x 1,000 of 640 bits 5.2, 4.5, of 800
// 5.2, 5.1, of 960 5.2, 5.7; 896-bit squares x 1,000 of 896 4.9, 4.0, of 1120 4.9,
// 4.6, of 1344 5.0, 5.1; 544-bit squares whole 4.7, 4.5.
bool mul_mx_pays(uint32_t a_len, uint32_t b_len, uint32_t p_len, bool square, uint32_t count) {
  if (!mul_mx_holds(a_len, b_len, count)) return false;
  if (a_len > 512) return true;
  if (2 * b_len < a_len || a_len <= 16) return false;
  if (a_len <= 32) {
    if (b_len > 16 && std::min(a_len + b_len, p_len) <= (square ? 36 : 25)) return false;
    return count <= 2048;
  }
  if (a_len <= 64) return count <= 4096;
  return a_len > 128 || count <= 8192;
}

// Two neighbouring products a workgroup (8-byte rows) unless that leaves CUs
// without one or a product fills a workgroup; eight tiles at a time where a
// product has 16 or more and the batch is full.  Measured: 4096 bits x 4,096
// 13.3 us (two products, four tiles) against 14.6 (one) and 19.7 (two, eight);
// 16384 x 64 13.0 (one) and 13.0 (two), x 1,024 22.8 and 18.4; 32768 x 4,096
// 113 (two, eight), 130 (one, four) and 132 (two, four); 65536 x 1,024 104
// (one, four), 118 (two, eight).  Four products a workgroup were never faster.
hipError_t launch_mul_mx(OutOperand p, Operand a, Operand b, uint32_t count, bool square, hipStream_t stream) {
  if (count == 0) return hipSuccess;
  if (a.len < b.len) std::swap(a, b);
  if (a.len <= 64 || a.len > 1024 || count < 512) return launch<1, 4>(p, a, b, count, square, stream);
  if (a.len <= 512) return launch<2, 4>(p, a, b, count, square, stream);
  return launch<2, 8>(p, a, b, count, square, stream);
}

}  // namespace xmp
