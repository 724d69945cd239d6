// k_xfer.hip -- import / export / set kernels.
//
// The reference repacks words with xmpTransform (src/xmp.cu:461-489) into a
// compact buffer and transposes lazily to its strided layout with
// xmpC2S/xmpS2C (src/xmp.cu:817-843).  Here the repack and the transpose are
// one kernel: compact host-format words go straight to the interleaved
// device layout and back.  Formats that are whole 32-bit words in either
// order, with their bytes in either order (little- and big-endian integers of
// any word size among them), with no nails and no indices, move as 4 x 4
// blocks of words through a lane's registers: 16-byte accesses on both sides
// and no LDS; a limb count that is not a multiple of four (or a host buffer
// that is not 16-byte aligned) takes an LDS-tiled transpose, and the remaining
// formats one thread a word.
#include <type_traits>

#include "kernels.hpp"

namespace xmp {

namespace {

constexpr uint32_t kTileI = 64;  // instances per LDS tile

// byte k (little-endian significance) of a compact integer row held as
// `words` words of `size` bytes with the given order/endian/nails.
__device__ __forceinline__ uint32_t import_byte(const uint8_t *row, uint32_t k, uint32_t words, int32_t order,
                                                int32_t endian, uint32_t nails, uint32_t size) {
  uint32_t w = k / size;
  uint32_t kb = k - w * size;
  if (w >= words) return 0;
  uint32_t pos = (order == -1) ? w : words - 1 - w;
  uint32_t mem = (endian == -1) ? kb : size - 1 - kb;
  uint32_t v = row[(size_t)pos * size + mem];
  // mask word(-1) >> nails applied to the word value (reference xmp.cu:481-483)
  uint64_t wmask = (size == 8 ? ~0ull : ((1ull << (8 * size)) - 1)) >> nails;
  return v & (uint32_t)((wmask >> (8 * kb)) & 0xFF);
}

// Tiles of kTileI instances by 1 << LJ limbs, the fewest columns that hold a
// short row (for_tiles), so that it is not walked as 32 words.  One loop length
// a kernel: known at compile time, all of a lane's loads are in flight, and the
// code is short, which a small call waits for.  PLAIN: the words run from the
// least significant and keep their bytes.  Imports and exports of 1,115,080
// integers of nine limbs 0.020 and 0.018 ms, with 32 columns 0.035 and 0.028; of
// 2^23 of one limb 0.034, 0.19 and 0.17.
template <int LJ, bool PLAIN>
__global__ void __launch_bounds__(256) import_tile_kernel(uint32_t *__restrict__ dst, uint32_t stride, uint32_t nlimbs,
                                                          const uint32_t *__restrict__ src, uint32_t count, bool rev,
                                                          bool swap) {
  __shared__ uint32_t tile[kTileI][(1 << LJ) + 1];
  const uint32_t i0 = blockIdx.x * kTileI, j0 = blockIdx.y << LJ;
#pragma unroll
  for (uint32_t r = threadIdx.x; r < kTileI << LJ; r += 256) {
    uint32_t ii = r >> LJ, jj = r & ((1u << LJ) - 1);
    uint32_t i = i0 + ii, j = j0 + jj;
    const uint32_t at = !PLAIN && rev ? nlimbs - 1 - j : j;
    const uint32_t v = (i < count && j < nlimbs) ? src[(size_t)i * nlimbs + at] : 0u;
    tile[ii][jj] = !PLAIN && swap ? __builtin_bswap32(v) : v;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = threadIdx.x; r < kTileI << LJ; r += 256) {
    uint32_t jj = r / kTileI, ii = r % kTileI;
    uint32_t i = i0 + ii, j = j0 + jj;
    if (i < count && j < nlimbs) dst[(size_t)j * stride + i] = tile[ii][jj];
  }
}

template <int LJ, bool PLAIN>
__global__ void __launch_bounds__(256) export_tile_kernel(uint32_t *__restrict__ dst, const uint32_t *__restrict__ src,
                                                          uint32_t stride, uint32_t nlimbs, uint32_t count, bool rev,
                                                          bool swap) {
  __shared__ uint32_t tile[kTileI][(1 << LJ) + 1];
  const uint32_t i0 = blockIdx.x * kTileI, j0 = blockIdx.y << LJ;
#pragma unroll
  for (uint32_t r = threadIdx.x; r < kTileI << LJ; r += 256) {
    uint32_t jj = r / kTileI, ii = r % kTileI;
    uint32_t i = i0 + ii, j = j0 + jj;
    tile[ii][jj] = (i < count && j < nlimbs) ? src[(size_t)j * stride + i] : 0u;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = threadIdx.x; r < kTileI << LJ; r += 256) {
    uint32_t ii = r >> LJ, jj = r & ((1u << LJ) - 1);
    uint32_t i = i0 + ii, j = j0 + jj;
    const uint32_t v = tile[ii][jj], at = !PLAIN && rev ? nlimbs - 1 - j : j;
    if (i < count && j < nlimbs) dst[(size_t)i * nlimbs + at] = !PLAIN && swap ? __builtin_bswap32(v) : v;
  }
}

// the tile's columns and the grid
template <class F>
void for_tiles(uint32_t nlimbs, uint32_t count, F &&launch) {
  const uint32_t ni = div_round_up(count, kTileI);
  // (a small call waits for one tile, a large one wants whole lines of rows:
  // 300 of 33 limbs with the division before them 10.7 us, with 32 columns
  // 12.2; 655,360 0.048 ms, with 32 columns 0.037 to 0.043)
  if (nlimbs > 16 && count > 4096) launch(std::integral_constant<int, 5>(), dim3(ni, div_round_up(nlimbs, 32)));
  else if (nlimbs > 8) launch(std::integral_constant<int, 4>(), dim3(ni, div_round_up(nlimbs, 16)));
  else if (nlimbs > 4) launch(std::integral_constant<int, 3>(), dim3(ni));
  else if (nlimbs > 1) launch(std::integral_constant<int, 2>(), dim3(ni));
  else launch(std::integral_constant<int, 0>(), dim3(ni));
}

// 4 x 4 blocks: a lane moves limbs 4 jq .. 4 jq + 3 of instances 4 iq .. 4 iq + 3,
// four 16-byte loads and four 16-byte stores.  A wave's lanes are 64 >> LJ
// instance quads by 1 << LJ limb quads: 8 by 8 makes whole 128-byte lines on
// both sides; short integers take fewer limb quads.  `rev`: the compact words
// run from the most significant; `swap`: their bytes too.  Bound by memory:
// 2^20 exports of 2048 bits, 537 MB, 0.093 ms (5.8 TB/s), imports 0.093; with the
// LDS tiles' 4-byte accesses 0.146 and 0.130, and as big-endian bytes, one
// thread a word, 3.3 and 1.5.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u32x4 to_words(u32x4 v, bool rev, bool swap) {
  if (swap) v = u32x4{__builtin_bswap32(v.x), __builtin_bswap32(v.y), __builtin_bswap32(v.z), __builtin_bswap32(v.w)};
  return rev ? u32x4{v.w, v.z, v.y, v.x} : v;
}

template <bool NT>
__device__ __forceinline__ u32x4 ld_quad(const uint32_t *p) {
  if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
  else return *reinterpret_cast<const u32x4 *>(p);
}
template <bool NT>
__device__ __forceinline__ void st_quad(uint32_t *p, u32x4 v) {
  if constexpr (NT) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(p));
  else *reinterpret_cast<u32x4 *>(p) = v;
}

template <int LJ>
__device__ __forceinline__ bool quad_at(uint32_t nq, uint32_t count, uint32_t *iq, uint32_t *jq) {
  // a workgroup's four waves: two by two tiles of 8 x 8, else four along the instances
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  constexpr uint32_t NJ = 1 << LJ, NI = 64 >> LJ;
  constexpr uint32_t WJ = LJ == 3 ? 2 : 1, WI = 4 / WJ;
  *iq = (blockIdx.x * WI + w / WJ) * NI + (lane & (NI - 1));
  *jq = (blockIdx.y * WJ + w % WJ) * NJ + lane / NI;
  return *jq < nq && 4 * *iq < count;
}

template <int LJ, bool NT, bool LINES>
__global__ void __launch_bounds__(256) import_quads_kernel(uint32_t *__restrict__ dst, uint32_t stride, uint32_t nlimbs,
                                                           const uint32_t *__restrict__ src, uint32_t count, bool rev,
                                                           bool swap) {
  uint32_t iq, jq;
  const uint32_t nq = nlimbs / 4;
  if (!quad_at<LJ>(nq, count, &iq, &jq)) return;
  const uint32_t i = 4 * iq, n = min(4u, count - i);
  const uint32_t *row = src + (size_t)i * nlimbs + 4 * (rev ? nq - 1 - jq : jq);
  u32x4 v[4];
#pragma unroll
  for (uint32_t e = 0; e < 4; e++)   // (the last row again in the place of those past the end)
    v[e] = to_words(ld_quad<LINES>(row + (size_t)min(e, n - 1) * nlimbs), rev, swap);
  uint32_t *out = dst + (size_t)(4 * jq) * stride + i;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    if (n == 4) {
      st_quad<NT>(out + (size_t)k * stride, u32x4{v[0][k], v[1][k], v[2][k], v[3][k]});
    } else {
      for (uint32_t e = 0; e < n; e++) out[(size_t)k * stride + e] = e == 0 ? v[0][k] : e == 1 ? v[1][k] : v[2][k];
    }
  }
}

template <int LJ, bool LINES>
__global__ void __launch_bounds__(256) export_quads_kernel(uint32_t *__restrict__ dst, const uint32_t *__restrict__ src,
                                                           uint32_t stride, uint32_t nlimbs, uint32_t count, bool rev,
                                                           bool swap) {
  uint32_t iq, jq;
  const uint32_t nq = nlimbs / 4;
  if (!quad_at<LJ>(nq, count, &iq, &jq)) return;
  const uint32_t i = 4 * iq;
  const uint32_t *in = src + (size_t)(4 * jq) * stride + i;   // (rows are padded to 64 instances)
  u32x4 r[4];
#pragma unroll
  for (int k = 0; k < 4; k++)
    r[k] = ld_quad<true>(in + (size_t)k * stride);
  uint32_t *row = dst + (size_t)i * nlimbs + 4 * (rev ? nq - 1 - jq : jq);
#pragma unroll
  for (int e = 0; e < 4; e++)
    if (i + (uint32_t)e < count)
      st_quad<LINES>(row + (size_t)e * nlimbs, to_words(u32x4{r[0][e], r[1][e], r[2][e], r[3][e]}, rev, swap));
}

// whether a format is 32-bit words in either order with their bytes in either
// order, over whole limbs, and what it does with them
bool as_words(uint32_t words, int32_t order, int32_t endian, uint32_t nails, uint32_t size, uint32_t nlimbs, bool *rev,
              bool *swap) {
  if (nails != 0 || (uint64_t)words * size != 4ull * nlimbs) return false;
  const bool big = order == 1;
  *rev = big;
  *swap = size == 1 ? big : endian == 1;
  return size == 4 || *swap == big;   // one-, two- and eight-byte words: all little- or all big-endian
}

// the limb quads of a wave's lanes, and the grid
template <class F>
void for_quads(uint32_t nlimbs, uint32_t count, F &&launch) {
  const uint32_t nq = nlimbs / 4, ni = div_round_up(count, 4);
  if (nq > 4) launch(std::integral_constant<int, 3>(), dim3(div_round_up(ni, 16), div_round_up(nq, 16)));
  else if (nq > 2) launch(std::integral_constant<int, 2>(), dim3(div_round_up(ni, 64)));
  else if (nq > 1) launch(std::integral_constant<int, 1>(), dim3(div_round_up(ni, 128)));
  else launch(std::integral_constant<int, 0>(), dim3(div_round_up(ni, 256)));
}

// Which sides bypass the caches.  An export's limbs are read once, and its rows
// are written past the caches where they are whole lines (a partial line must wait in
// the L2 for its other part): an operation and its export, with rows by this rule
// and by its opposite, 64 limbs x 300,000 products 133 and 148 us, 128-limb
// quotients and 64-limb remainders x 65,536 62 and 66, 164 limbs x 82,196 96 and
// 110, 8 limbs x 10^6 sums 34 and 43.  An import's limbs are about to be used, so
// it stays in the caches that hold it (64 limbs x 300,000 24 and 31 us, 4 x
// 4,000,000 20 and 29), and passes them by beyond (128 x 2^20 191, 208).
constexpr size_t kCached = 192u << 20;   // compact bytes; as many again on the other side

// whole words to or from pinned host memory, over the bus: 4 MiB of writes 86 us, 51 GB/s
__global__ void __launch_bounds__(256) copy_kernel(uint32_t *__restrict__ dst, const uint32_t *__restrict__ src,
                                                   uint32_t words) {
  const uint32_t i = 4 * (blockIdx.x * 256 + threadIdx.x);
  if (i + 4 <= words)
    *reinterpret_cast<u32x4 *>(dst + i) = *reinterpret_cast<const u32x4 *>(src + i);
  else
    for (uint32_t k = i; k < words; k++) dst[k] = src[k];
}

__global__ void import_general_kernel(uint32_t *__restrict__ dst, uint32_t stride, uint32_t nlimbs,
                                      const uint8_t *__restrict__ src, uint32_t count, uint32_t words,
                                      int32_t order, int32_t endian, uint32_t nails, uint32_t size,
                                      const uint32_t *__restrict__ in_idx, uint32_t in_idx_count) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t j = blockIdx.y;
  if (i >= count || j >= nlimbs) return;
  uint32_t row = in_idx ? in_idx[i % in_idx_count] : i;
  const uint8_t *r = src + (size_t)row * words * size;
  uint32_t v = 0;
#pragma unroll
  for (uint32_t b = 0; b < 4; b++) v |= import_byte(r, 4 * j + b, words, order, endian, nails, size) << (8 * b);
  dst[(size_t)j * stride + i] = v;
}

// one thread per output word (size bytes) of the compact output
__global__ void export_general_kernel(uint8_t *__restrict__ dst, const uint32_t *__restrict__ src, uint32_t stride,
                                      uint32_t nlimbs, uint32_t count, uint32_t words, int32_t order,
                                      int32_t endian, uint32_t nails, uint32_t size,
                                      const uint32_t *__restrict__ out_idx, uint32_t out_idx_count) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t j = blockIdx.y;
  if (i >= count || j >= words) return;
  uint32_t orow = out_idx ? out_idx[i % out_idx_count] : i;
  uint32_t pos = (order == -1) ? j : words - 1 - j;
  uint64_t wmask = (size == 8 ? ~0ull : ((1ull << (8 * size)) - 1)) >> nails;
  uint8_t *o = dst + ((size_t)orow * words + j) * size;
  for (uint32_t p = 0; p < size; p++) {
    uint32_t sig = (endian == -1) ? p : size - 1 - p;   // significance of memory byte p after swap
    uint32_t k = pos * size + sig;                       // byte of the integer
    uint32_t limb = k >> 2;
    uint32_t v = limb < nlimbs ? src[(size_t)limb * stride + i] : 0u;
    uint32_t byte = (v >> (8 * (k & 3))) & 0xFF;
    o[p] = (uint8_t)(byte & (uint32_t)((wmask >> (8 * p)) & 0xFF));
  }
}

__global__ void set_kernel(uint32_t *__restrict__ out, uint32_t out_stride, uint32_t out_limbs,
                           const uint32_t *__restrict__ in, uint32_t in_stride, uint32_t in_limbs, uint32_t in_count,
                           uint32_t count, const uint32_t *__restrict__ out_idx, uint32_t out_idx_count,
                           const uint32_t *__restrict__ in_idx, uint32_t in_idx_count) {
  uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t j = blockIdx.y;
  if (k >= count || j >= out_limbs) return;
  uint32_t i = in_idx ? in_idx[k % in_idx_count] % in_count : k;
  uint32_t o = out_idx ? out_idx[k % out_idx_count] : k;
  out[(size_t)j * out_stride + o] = j < in_limbs ? in[(size_t)j * in_stride + i] : 0u;
}

}  // namespace

bool transfer_in_words(uint32_t words, int32_t order, int32_t endian, uint32_t nails, uint32_t size, uint32_t nlimbs) {
  bool rev, swap;
  return as_words(words, order, endian, nails, size, nlimbs, &rev, &swap);
}

hipError_t launch_copy(void *dst, const void *src, size_t bytes, hipStream_t stream) {
  const uint32_t words = (uint32_t)(bytes / 4);
  hipLaunchKernelGGL(copy_kernel, dim3(div_round_up(words, 1024)), dim3(256), 0, stream,
                     static_cast<uint32_t *>(dst), static_cast<const uint32_t *>(src), words);
  return hipGetLastError();
}

hipError_t launch_import(uint32_t *dst, uint32_t dst_stride, uint32_t nlimbs, const uint8_t *src, uint32_t count,
                         uint32_t words, int32_t order, int32_t endian, uint32_t nails, uint32_t size,
                         const uint32_t *in_idx, uint32_t in_idx_count, hipStream_t stream) {
  bool rev = false, swap = false;
  const bool plain = in_idx == nullptr && (uintptr_t)src % 4 == 0 &&
                     as_words(words, order, endian, nails, size, nlimbs, &rev, &swap);
  if (plain && nlimbs % 4 == 0 && (uintptr_t)src % 16 == 0) {
    const bool cached = (size_t)4 * nlimbs * count <= kCached;
    for_quads(nlimbs, count, [&](auto lj, dim3 grid) {
      auto kernel = cached             ? import_quads_kernel<lj(), false, false>
                    : nlimbs % 32 == 0 ? import_quads_kernel<lj(), true, true>
                                       : import_quads_kernel<lj(), true, false>;
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, dst, dst_stride, nlimbs,
                         reinterpret_cast<const uint32_t *>(src), count, rev, swap);
    });
  } else if (plain) {
    for_tiles(nlimbs, count, [&](auto lj, dim3 grid) {
      hipLaunchKernelGGL((rev || swap ? import_tile_kernel<lj(), false> : import_tile_kernel<lj(), true>), grid,
                         dim3(256), 0, stream, dst, dst_stride, nlimbs, reinterpret_cast<const uint32_t *>(src), count,
                         rev, swap);
    });
  } else {
    dim3 grid(div_round_up(count, 256), nlimbs);
    hipLaunchKernelGGL(import_general_kernel, grid, dim3(256), 0, stream, dst, dst_stride, nlimbs, src, count,
                       words, order, endian, nails, size, in_idx, in_idx_count);
  }
  return hipGetLastError();
}

hipError_t launch_export(uint8_t *dst, const uint32_t *src, uint32_t src_stride, uint32_t nlimbs, uint32_t count,
                         uint32_t words, int32_t order, int32_t endian, uint32_t nails, uint32_t size,
                         const uint32_t *out_idx, uint32_t out_idx_count, hipStream_t stream) {
  bool rev = false, swap = false;
  const bool plain = out_idx == nullptr && (uintptr_t)dst % 4 == 0 &&
                     as_words(words, order, endian, nails, size, nlimbs, &rev, &swap);
  if (plain && nlimbs % 4 == 0 && (uintptr_t)dst % 16 == 0) {
    for_quads(nlimbs, count, [&](auto lj, dim3 grid) {
      hipLaunchKernelGGL((nlimbs % 32 == 0 ? export_quads_kernel<lj(), true> : export_quads_kernel<lj(), false>), grid,
                         dim3(256), 0, stream, reinterpret_cast<uint32_t *>(dst), src, src_stride, nlimbs, count, rev,
                         swap);
    });
  } else if (plain) {
    for_tiles(nlimbs, count, [&](auto lj, dim3 grid) {
      hipLaunchKernelGGL((rev || swap ? export_tile_kernel<lj(), false> : export_tile_kernel<lj(), true>), grid,
                         dim3(256), 0, stream, reinterpret_cast<uint32_t *>(dst), src, src_stride, nlimbs, count, rev,
                         swap);
    });
  } else {
    dim3 grid(div_round_up(count, 256), words);
    hipLaunchKernelGGL(export_general_kernel, grid, dim3(256), 0, stream, dst, src, src_stride, nlimbs, count,
                       words, order, endian, nails, size, out_idx, out_idx_count);
  }
  return hipGetLastError();
}

hipError_t launch_set(uint32_t *out, uint32_t out_stride, uint32_t out_limbs, const uint32_t *in, uint32_t in_stride,
                      uint32_t in_limbs, uint32_t in_count, uint32_t count, const uint32_t *out_idx,
                      uint32_t out_idx_count, const uint32_t *in_idx, uint32_t in_idx_count, hipStream_t stream) {
  dim3 grid(div_round_up(count, 256), out_limbs);
  hipLaunchKernelGGL(set_kernel, grid, dim3(256), 0, stream, out, out_stride, out_limbs, in, in_stride, in_limbs,
                     in_count, count, out_idx, out_idx_count, in_idx, in_idx_count);
  return hipGetLastError();
}

hipError_t launch_copy_words(uint32_t *dst, const uint32_t *src, size_t words, hipStream_t stream) {
  return hipMemcpyAsync(dst, src, words * sizeof(uint32_t), hipMemcpyDeviceToDevice, stream);
}

}  // namespace xmp
