// The reference's precise kernel, ReferenceKernel<f32> (src/kernel/mod.rs:
// 691-821 with the box filter of src/kernel/ref.rs), on the GPU: the
// "forensic" mode whose hashes follow the officially endorsed PDQ resampler
// (two passes of a 3-wide box filter along rows and columns, then nearest
// sampling at floor((2i + 1) 512 / 254)) instead of the optimised tent.
//
// The running sums are sequential along a line, so a line is a lane.  The four
// box passes (rows, columns, rows, columns) and the rest run as a chain of
// launches, each with eight waves of 64 lines per image, so that one image
// already spreads over several CUs:
//   rows      (f32 planes only) the first pass, through LDS tiles that turn
//             coalesced rows into one row per lane;
//   columns   the second pass; for u8 planes with the first one fused, whose
//             sums are whole numbers and so need no running sum;
//   sampled   the third pass, which stores only the 127 of 512 columns that
//             the sampling at floor((2i + 1) 512 / 254) reads;
//   finish    one block per image: the fourth pass over those 127 columns, the
//             samples in LDS, the reference's sequential DCT (mul then add, k
//             ascending, one accumulator per output), and on waves of their
//             own the gradient sum and quality, Torben's median (exact
//             tie-breaking) and the bits.
// A division by 3 is a product and a remainder step, correctly rounded for
// every |x| in [2^-124, 2^127] (checked exhaustively on the CPU).  Sums lie in
// it when every input is zero or in [2^-25, 2^100]: a sum or a third of
// multiples of 2^-k is zero or at least 2^-(k + 2) and a multiple of
// 2^-(k + 25).  u8 planes always do.  The first pass of an f32 plane looks for
// another value (NaN and Inf too): its 64 rows are then walked again with
// divisions, and the image's later passes divide as well.  Until its hash is
// written, byte r of an image's hash tells them whether run r found one.
// Bounds and times (us, u8 from HBM; one block per image with IEEE divisions
// and 64-byte row accesses before): one image 223 -> 49, 100 images 283 -> 91,
// 1024 images 2206 -> 733; f32 248 -> 63, 344 -> 126, 2469 -> 1263.  At 100
// images the column pass (35 us) writes 105 MB and reads 26 MB, 3.7 TB/s, the
// sampled rows (21 us) read them back, and the finish (28 us; 20 alone) is
// 512 dependent steps, 127 LDS steps and the median's chain.  With divisions one
// image takes 95, 100 images 149 (as one block per image behind the other
// passes, which they were before, 277 and 453).
// Every rounding happens where the reference's scalar code rounds, so the
// results are its bits.  Only the NORMAL orientation is computed.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "pdq_hash_common.h"

namespace ypdq {

namespace {

constexpr int kRefThreads = 512;

struct RefLds {
  union {
    float c[127 * 128];  // samples, row stride 128
    struct {
      float t[16 * kTS];  // DCT stage-1 rows
      float p[256];       // PDQF
    } d;
  } u;
  float dct_t[127 * 16];  // D transposed: dct_t[k * 16 + i] = D[i][k]
};

// x / 3, by a division or as the top of the file says.  The passes are the box
// filter of src/kernel/ref.rs:49-124 with window 3: half window 2, one leading
// accumulation, two short-window writes, full-window writes, one trailing
// short-window write (a short window holds two inputs, and a half is exact).
template <bool kDivide>
__device__ __forceinline__ float third(float x) {
  if constexpr (kDivide) return x / 3.0f;
  constexpr float r = 1.0f / 3.0f;
  const float q = x * r;
  return __builtin_fmaf(__builtin_fmaf(-q, 3.0f, x), r, q);
}

// Block -> (image, one of its eight runs of 64 lines).  Consecutive blocks go
// to the eight XCDs in turn, so an image's blocks are numbered eight apart:
// they share an L2, whose lines of neighbouring runs leave together.
__device__ __forceinline__ bool line_block(uint32_t n_images, uint32_t& img, int& run) {
  const uint32_t slot = blockIdx.x >> 3;
  img = (blockIdx.x & 7) + 8 * (slot >> 3);
  run = (int)(slot & 7);
  return img < n_images;
}

// The lanes of a wave walk 64 rows in tiles of 32 columns.  A tile is loaded
// and stored with eight lanes per row (whole 128-byte lines) and passes
// through LDS, where lane l reads its row l in 16-byte steps; a stride of 36
// floats keeps both sides free of bank conflicts.
constexpr int kTileCols = 32;
constexpr int kTileStride = 36;
constexpr int kTiles = 512 / kTileCols;
struct RowTiles {
  float v[2][64 * kTileStride];
};

__device__ __forceinline__ void tile_fetch(const float* __restrict__ src, int lane, int tile, f32x4 (&pf)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i++)
    pf[i] = *reinterpret_cast<const f32x4*>(src + (8 * i + (lane >> 3)) * 512 + kTileCols * tile + 4 * (lane & 7));
}
__device__ __forceinline__ void tile_put(float* __restrict__ buf, int lane, const f32x4 (&pf)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i++)
    *reinterpret_cast<f32x4*>(buf + (8 * i + (lane >> 3)) * kTileStride + 4 * (lane & 7)) = pf[i];
}
__device__ __forceinline__ void tile_row(const float* __restrict__ buf, int lane, float (&x)[kTileCols]) {
#pragma unroll
  for (int q = 0; q < kTileCols / 4; q++) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(buf + lane * kTileStride + 4 * q);
    x[4 * q] = v.x;
    x[4 * q + 1] = v.y;
    x[4 * q + 2] = v.z;
    x[4 * q + 3] = v.w;
  }
}

// Whether an f32 input keeps third() exact: zero or in [2^-25, 2^100], as the
// minimum of 2 |bits| - 1 (zero wraps to the largest) and the maximum of
// |x|; NaN shows in the running sum.
struct Range {
  uint32_t least = 0xffffffffu;
  float most = 0.0f;
  __device__ __forceinline__ void take(float x) {
    least = min(least, (__float_as_uint(x) << 1) - 1u);
    most = fmaxf(most, __builtin_fabsf(x));
  }
  __device__ __forceinline__ bool plain(float sum) const {
    return least >= ((102u << 24) - 1u) && most <= 0x1p100f && __builtin_isfinite(sum);
  }
};

// Whether a pass of the image divides: a byte per run, in the image's hash.
__device__ __forceinline__ bool divides(const uint8_t* __restrict__ hashes, uint32_t img) {
  uint64_t runs;
  __builtin_memcpy(&runs, hashes + (size_t)img * 32, 8);
  return runs != 0;
}

// First pass of f32 planes: out[j] = box of row j, all 512 columns, of 64 rows.
// Output j of a row is complete with input j + 1, so a tile also takes the first
// input of the next one.  Returns whether this lane's row keeps third() exact.
template <bool kDivide>
__device__ __forceinline__ bool rows_pass(const float* __restrict__ src, float* __restrict__ dst, RowTiles& L,
                                          int lane) {
  f32x4 pf[8];
  tile_fetch(src, lane, 0, pf);
  tile_put(L.v[0], lane, pf);
  tile_fetch(src, lane, 1, pf);
  float sum = 0.0f, h[3] = {0.0f, 0.0f, 0.0f};  // the last three inputs, oldest first
  Range range;
#pragma unroll 1
  for (int tile = 0; tile < kTiles; tile++) {
    float* buf = L.v[tile & 1];
    float* nbuf = L.v[(tile + 1) & 1];
    if (tile + 1 < kTiles) tile_put(nbuf, lane, pf);
    tile_fetch(src, lane, min(tile + 2, kTiles - 1), pf);
    wave_lds_sync();
    float x[kTileCols + 1], o[kTileCols];
    {
      float r[kTileCols];
      tile_row(buf, lane, r);
#pragma unroll
      for (int e = 0; e < kTileCols; e++) x[e] = r[e];
    }
    x[kTileCols] = nbuf[lane * kTileStride];  // past the last tile: not an input
#pragma unroll
    for (int e = 0; e < kTileCols; e++) range.take(x[e]);
    auto step = [&](float in, float old) {
      sum += in;
      sum -= old;
    };
    if (tile == 0) step(x[0], 0.0f);
#pragma unroll
    for (int e = 1; e <= kTileCols; e++) {
      const float old = e < 3 ? h[e] : x[e - 3];
      if (e < kTileCols || tile + 1 < kTiles) {
        step(x[e], old);
        o[e - 1] = third<kDivide>(sum);
      } else {
        sum -= old;  // the last output: the oldest input leaves the window
        o[e - 1] = sum * 0.5f;
      }
      if (e == 1 && tile == 0) o[0] = sum * 0.5f;
    }
    h[0] = 0.0f;  // (unused: input 0 of a tile was taken by the one before)
    h[1] = x[kTileCols - 2];
    h[2] = x[kTileCols - 1];
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < kTileCols / 4; q++)
      *reinterpret_cast<f32x4*>(buf + lane * kTileStride + 4 * q) =
          f32x4{o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]};
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < 8; i++)
      *reinterpret_cast<f32x4*>(dst + (8 * i + (lane >> 3)) * 512 + kTileCols * tile + 4 * (lane & 7)) =
          *reinterpret_cast<const f32x4*>(buf + (8 * i + (lane >> 3)) * kTileStride + 4 * (lane & 7));
    wave_lds_sync();
  }
  return range.plain(sum);
}

__global__ void __launch_bounds__(64) pdq_ref_rows_kernel(const float* __restrict__ planes, uint64_t plane_stride,
                                                          uint32_t n_images, float* __restrict__ work,
                                                          uint8_t* __restrict__ hashes) {
  __shared__ RowTiles L;
  uint32_t img;
  int run;
  if (!line_block(n_images, img, run)) return;
  const int row0 = 64 * run;
  const int lane = threadIdx.x;
  const float* src = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(planes) +
                                                    (size_t)img * plane_stride) + row0 * 512;
  float* dst = work + (size_t)img * 2 * 512 * 512 + row0 * 512;
  const bool divide = wave_any(!rows_pass<false>(src, dst, L, lane));
  if (divide) (void)rows_pass<true>(src, dst, L, lane);
  if (lane == 0) hashes[(size_t)img * 32 + run] = divide ? 1 : 0;
}

// One input row of the second pass at this lane's column: an f32 value of A,
// or four u8 pixels whose weighted sum is the first pass's window.
template <typename T>
struct ColumnSource;
template <>
struct ColumnSource<float> {
  const float* p;  // uniform; the lane's offset is added to each row's address
  uint32_t at;
  using Raw = float;
  __device__ __forceinline__ ColumnSource(const float* a, int c) : p(a), at((uint32_t)c) {}
  __device__ __forceinline__ Raw load(int r) const { return (p + r * 512)[at]; }
  __device__ __forceinline__ float value(Raw x) const { return x; }
};
template <>
struct ColumnSource<uint8_t> {
  const uint8_t* p;
  uint32_t at, weights;
  float div, rcp;
  using Raw = uint32_t;
  // columns c - 1 .. c + 1 of the row, in a (mostly unaligned) word that
  // stays inside the row; two columns at the row's ends
  __device__ __forceinline__ ColumnSource(const uint8_t* plane, int c) {
    const int first = min(max(c - 1, 0), 508);
    const uint32_t three = 0x010101u << (8 * (c - 1 - first) & 31);
    p = plane;
    at = (uint32_t)first;
    weights = c == 0 ? 0x0101u : three;
    div = c == 0 || c == 511 ? 2.0f : 3.0f;
    rcp = c == 0 || c == 511 ? 0.5f : 1.0f / 3.0f;
  }
  __device__ __forceinline__ Raw load(int r) const {
    uint32_t x;
    __builtin_memcpy(&x, p + r * 512 + at, 4);
    return x;
  }
  __device__ __forceinline__ float value(Raw x) const {
    const float s = (float)__builtin_amdgcn_udot4(x, weights, 0u, false);
    const float q = s * rcp;
    return __builtin_fmaf(__builtin_fmaf(-q, div, s), rcp, q);
  }
};

// Second pass (columns), a lane per column, into B; the next 32 rows load
// while these are summed.  A u8 wave reads 64 bytes of a row, too little in
// flight for HBM: one load of 64 rows (a row per lane) brings their lines into
// the cache two iterations ahead of the loads that use them.
template <typename T, bool kDivide>
__device__ __forceinline__ void cols_pass(const T* __restrict__ planes, uint64_t plane_stride, uint32_t img, int run,
                                          float* __restrict__ work) {
  constexpr int R = 32;
  const uint32_t c = 64 * run + threadIdx.x;
  const float* A = work + (size_t)img * 2 * 512 * 512;
  float* out = work + (size_t)img * 2 * 512 * 512 + 512 * 512;
  const T* in;
  if constexpr (std::is_same<T, float>::value) in = A;
  else in = reinterpret_cast<const T*>(reinterpret_cast<const uint8_t*>(planes) + (size_t)img * plane_stride);
  const ColumnSource<T> src(in, (int)c);
  constexpr bool kAhead = std::is_same<T, uint8_t>::value;
  auto ahead = [&](int r0) -> uint32_t {
    if constexpr (!kAhead) return 0u;
    else return in[min(r0 + (int)threadIdx.x, 511) * 512 + 64 * run];
  };
  uint32_t near = ahead(0), far = ahead(64);
  typename ColumnSource<T>::Raw cur[R], nxt[R];
#pragma unroll
  for (int e = 0; e < R; e++) cur[e] = src.load(e);
  float sum = 0.0f, h0 = 0.0f, h1 = 0.0f, h2 = 0.0f;
  auto chunk = [&](int r0, const typename ColumnSource<T>::Raw(&raw)[R]) {
#pragma unroll
    for (int e = 0; e < R; e++) {
      const float x = src.value(raw[e]);
      sum += x;
      sum -= h0;
      h0 = h1;
      h1 = h2;
      h2 = x;
      if (e == 0) {
        if (r0 > 0) (out + (r0 - 1) * 512)[c] = third<kDivide>(sum);
      } else if (e == 1) {
        (out + r0 * 512)[c] = r0 == 0 ? sum * 0.5f : third<kDivide>(sum);
      } else {
        (out + (r0 + e - 1) * 512)[c] = third<kDivide>(sum);
      }
    }
  };
#pragma unroll 1
  for (int r0 = 0; r0 < 512; r0 += 2 * R) {
#pragma unroll
    for (int e = 0; e < R; e++) nxt[e] = src.load(r0 + R + e);
    __builtin_amdgcn_sched_barrier(0);  // all loads before the sums
    chunk(r0, cur);
#pragma unroll
    for (int e = 0; e < R; e++) cur[e] = src.load(min(r0 + 2 * R, 512 - R) + e);
    asm volatile("" ::"v"(near));  // (arrived long ago)
    near = far;
    far = ahead(r0 + 4 * R);
    __builtin_amdgcn_sched_barrier(0);
    chunk(r0 + R, nxt);
  }
  sum -= h0;
  (out + 511 * 512)[c] = sum * 0.5f;
}

template <typename T>
__global__ void __launch_bounds__(64) pdq_ref_cols_kernel(const T* __restrict__ planes, uint64_t plane_stride,
                                                          uint32_t n_images, float* __restrict__ work,
                                                          const uint8_t* __restrict__ hashes) {
  uint32_t img;
  int run;
  if (!line_block(n_images, img, run)) return;
  if constexpr (std::is_same<T, float>::value)
    if (divides(hashes, img)) return cols_pass<T, true>(planes, plane_stride, img, run, work);
  cols_pass<T, false>(planes, plane_stride, img, run, work);
}

// Sample k of a line is output floor((2k + 1) 512 / 254), complete with input
//   k <= 31: 4k + 3    k = 32 .. 62: 4k + 4    k = 63 .. 94: 4k + 5
//   k >= 95: 4k + 6
// so, by groups of four inputs: group g < 32 completes sample g with its last
// input, group 32 none, and group g > 32 sample g - 1 with its first (g < 64),
// second (g < 96) or third input.
__device__ __forceinline__ constexpr int sample_input(int g) { return g < 32 ? 3 : g < 64 ? 0 : g < 96 ? 1 : 2; }

// Third pass (rows) from B; the samples go to A as 512 rows of 128, by the
// group that completes them (place 32 holds no sample).  A lane's samples
// gather in LDS and are stored a quarter of a row at a time, whole 128-byte
// lines.
template <int kQuarter, bool kDivide>
__device__ __forceinline__ void sampled_tile(const float (&x)[kTileCols], int first_group, float& sum, float (&h)[3],
                                             float* __restrict__ out) {
#pragma unroll
  for (int u = 0; u < kTileCols / 4; u++) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int i = 4 * u + e;
      sum += x[i];
      sum -= i < 3 ? h[i] : x[i - 3];
      if (e == sample_input(32 * kQuarter)) out[(first_group + u) & 31] = third<kDivide>(sum);
    }
  }
  h[0] = x[kTileCols - 3];
  h[1] = x[kTileCols - 2];
  h[2] = x[kTileCols - 1];
}

template <bool kDivide>
__device__ __forceinline__ void sampled_pass(RowTiles& L, uint32_t img, int run, float* __restrict__ work) {
  const int row0 = 64 * run;
  const int lane = threadIdx.x;
  float* A = work + (size_t)img * 2 * 512 * 512;
  const float* src = A + 512 * 512 + row0 * 512;
  float* dst = A + row0 * 128;
  float* out = L.v[1] + lane * kTileStride;
  f32x4 pa[8], pb[8];
  tile_fetch(src, lane, 0, pa);
  tile_fetch(src, lane, 1, pb);
  float sum = 0.0f, h[3] = {0.0f, 0.0f, 0.0f};
  // samples 32 q .. 32 q + 31 of the wave's rows
  auto flush = [&](int q) {
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < 8; i++)
      *reinterpret_cast<f32x4*>(dst + (8 * i + (lane >> 3)) * 128 + 32 * q + 4 * (lane & 7)) =
          *reinterpret_cast<const f32x4*>(L.v[1] + (8 * i + (lane >> 3)) * kTileStride + 4 * (lane & 7));
    wave_lds_sync();
  };
  auto step = [&](auto q, int tile, f32x4(&pf)[8]) {
    constexpr int kQuarter = decltype(q)::value;
    wave_lds_sync();
    tile_put(L.v[0], lane, pf);
    tile_fetch(src, lane, min(tile + 2, kTiles - 1), pf);
    wave_lds_sync();
    float x[kTileCols];
    tile_row(L.v[0], lane, x);
    sampled_tile<kQuarter, kDivide>(x, 8 * tile, sum, h, out);
  };
  auto quarter = [&](auto q) {
    constexpr int t0 = kTiles / 4 * decltype(q)::value;
#pragma unroll 1
    for (int k = 0; k < kTiles / 4; k += 2) {
      step(q, t0 + k, pa);
      step(q, t0 + k + 1, pb);
    }
    flush(decltype(q)::value);
  };
  quarter(std::integral_constant<int, 0>());
  quarter(std::integral_constant<int, 1>());
  quarter(std::integral_constant<int, 2>());
  quarter(std::integral_constant<int, 3>());
}

// kMayDivide: f32 planes.
template <bool kMayDivide>
__global__ void __launch_bounds__(64) pdq_ref_sampled_kernel(uint32_t n_images, float* __restrict__ work,
                                                             const uint8_t* __restrict__ hashes) {
  __shared__ RowTiles L;  // the tile, the samples
  uint32_t img;
  int run;
  if (!line_block(n_images, img, run)) return;
  if constexpr (kMayDivide)
    if (divides(hashes, img)) return sampled_pass<true>(L, img, run, work);
  sampled_pass<false>(L, img, run, work);
}

// Fourth pass (columns of the samples): lane k walks column k of the 512 x 128
// samples in A and keeps every sampled row's value in c.  Sixteen rows at a
// time, from LDS.
template <int kQuarter, bool kDivide>
__device__ __forceinline__ void finish_rows(const float* __restrict__ x0, int first_group, float& sum, float (&h)[3],
                                            float* __restrict__ c) {
  float x[16];
#pragma unroll
  for (int e = 0; e < 16; e++) x[e] = x0[e * 128];
#pragma unroll
  for (int u = 0; u < 4; u++) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int i = 4 * u + e;
      sum += x[i];
      sum -= i < 3 ? h[i] : x[i - 3];
      if (e == sample_input(32 * kQuarter)) {
        const int k = first_group + u - (kQuarter == 0 ? 0 : 1);
        if (kQuarter != 1 || k > 31) c[k * 128] = third<kDivide>(sum);
      }
    }
  }
  h[0] = x[13];
  h[1] = x[14];
  h[2] = x[15];
}

// Two waves walk while the whole block fetches: 64 rows at a time, two chunks
// in registers ahead of the two in LDS.
struct ColumnChunks {
  float v[2][64 * 128];
};

template <bool kDivide>
__device__ __forceinline__ void finish_columns(const float* __restrict__ src, ColumnChunks& S, float* __restrict__ c) {
  const int t = threadIdx.x;
  // the sample of place t; place 32's walk goes to the unused column 127
  const int column = t < 32 ? t : t == 32 ? 127 : t - 1;
  f32x4 ra[4], rb[4];
  auto fetch = [&](f32x4(&r)[4], int chunk) {
#pragma unroll
    for (int q = 0; q < 4; q++)
      r[q] = reinterpret_cast<const f32x4*>(src)[min(chunk, 7) * 2048 + q * kRefThreads + t];
  };
  float sum = 0.0f, h[3] = {0.0f, 0.0f, 0.0f};
  auto chunk = [&](auto q, int m, f32x4(&r)[4]) {
    constexpr int kQuarter = decltype(q)::value;
    float* buf = S.v[m & 1];
#pragma unroll
    for (int k = 0; k < 4; k++) reinterpret_cast<f32x4*>(buf)[k * kRefThreads + t] = r[k];
    fetch(r, m + 2);
    __syncthreads();
    if (t < 128) {
#pragma unroll
      for (int k = 0; k < 4; k++) finish_rows<kQuarter, kDivide>(buf + k * 16 * 128 + t, 16 * m + 4 * k, sum, h, c + column);
    }
  };
  auto quarter = [&](auto q) {
    chunk(q, 2 * decltype(q)::value, ra);
    chunk(q, 2 * decltype(q)::value + 1, rb);
  };
  fetch(ra, 0);
  fetch(rb, 1);
  quarter(std::integral_constant<int, 0>());
  quarter(std::integral_constant<int, 1>());
  quarter(std::integral_constant<int, 2>());
  quarter(std::integral_constant<int, 3>());
}

// Maximum and minimum over the wave, in every lane (no NaN among the values
// that matter: the callers select them by a comparison).
constexpr int kDppMirror = 0x140;  // row_mirror
__device__ __forceinline__ float wave_max(float x, int lane) {
  x = fmaxf(x, dpp_f<kDppXor1>(x));
  x = fmaxf(x, dpp_f<kDppXor2>(x));
  x = fmaxf(x, dpp_f<kDppHalfMirror>(x));
  x = fmaxf(x, dpp_f<kDppMirror>(x));
  x = fmaxf(x, row_swapf(x, lane));
  return fmaxf(x, half_swapf(x, lane));
}
__device__ __forceinline__ float wave_min(float x, int lane) { return -wave_max(-x, lane); }

// The first element, in flat order, of the extreme value `best` among lane
// l's elements 4l .. 4l+3 that `pick` selects: its bits (zeros of either sign
// compare equal), or `none` where no element is equal to best.
template <typename Pick>
__device__ __forceinline__ float first_equal(const float (&v)[4], float best, float none, Pick pick) {
  int e0 = -1;
#pragma unroll
  for (int e = 3; e >= 0; e--) e0 = pick(v[e]) && v[e] == best ? e : e0;
  const uint64_t found = __ballot(e0 >= 0);
  if (!found) return none;
  const float x = e0 == 0 ? v[0] : e0 == 1 ? v[1] : e0 == 2 ? v[2] : v[3];
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), __builtin_ctzll(found)));
}

// Torben's median (src/kernel/mod.rs:212-253) over P by one wave: lane l
// holds elements 4l .. 4l+3, so lane order is the reference's flat order.
// Counts are order-free ballots; maxltguess / mingtguess keep the reference's
// strict-comparison updates: the first element (in flat order) of the
// extreme value among those strictly beyond the initial bound, else the
// bound itself.
__device__ __forceinline__ float torben_median_wave(const float* __restrict__ P, int lane) {
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; e++) v[e] = P[4 * lane + e];
  float mn = v[0], mx = v[0];
#pragma unroll
  for (int e = 1; e < 4; e++) {
    mn = fminf(mn, v[e]);
    mx = fmaxf(mx, v[e]);
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    mn = fminf(mn, __shfl_xor(mn, m, 64));
    mx = fmaxf(mx, __shfl_xor(mx, m, 64));
  }
  const int half = (16 * 16 + 1) / 2;
  // Every iteration either returns or moves min or max to an element
  // strictly inside [min, max], so 257 iterations always suffice.
  float result = 0.0f;
#pragma unroll 1
  for (int iter = 0; iter < 300; iter++) {
    const float guess = (mn + mx) / 2.0f;
    uint32_t less = 0, greater = 0;
    float lt = mn, gt = mx;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const bool below = v[e] < guess, above = v[e] > guess;
      less += (uint32_t)__builtin_popcountll(__ballot(below));
      greater += (uint32_t)__builtin_popcountll(__ballot(above));
      lt = below && v[e] > lt ? v[e] : lt;
      gt = above && v[e] < gt ? v[e] : gt;
    }
    const uint32_t equal = 256 - less - greater;
    // an extreme equal to its bound is the bound (strict comparisons)
    const float lt_best = wave_max(lt, lane), gt_best = wave_min(gt, lane);
    float maxltguess = mn, mingtguess = mx;
    if (lt_best > mn) maxltguess = first_equal(v, lt_best, mn, [&](float x) { return x < guess; });
    if (gt_best < mx) mingtguess = first_equal(v, gt_best, mx, [&](float x) { return x > guess; });
    if (less <= (uint32_t)half && greater <= (uint32_t)half) {
      result = less >= (uint32_t)half ? maxltguess : (less + equal >= (uint32_t)half ? guess : mingtguess);
      break;
    } else if (less > greater) {
      mx = maxltguess;
    } else {
      mn = mingtguess;
    }
  }
  return result;
}

// One block per image: the fourth pass, dct2d, quality, median and bits.
template <typename T>
__global__ void __launch_bounds__(kRefThreads) pdq_ref_finish_kernel(float* __restrict__ work,
                                                                     uint8_t* __restrict__ hashes,
                                                                     float* __restrict__ quality,
                                                                     float* __restrict__ threshold,
                                                                     float* __restrict__ pdqf) {
  __shared__ RefLds L;
  const uint32_t img = blockIdx.x;
  const int t = threadIdx.x;
  float* A = work + (size_t)img * 2 * 512 * 512;
  float* c = L.u.c;
  __shared__ ColumnChunks S;
  for (int e = t; e < 127 * 16; e += kRefThreads) L.dct_t[e] = kDctT.v[e];
  if (std::is_same<T, float>::value && divides(hashes, img))  // the same for the whole block
    finish_columns<true>(A, S, c);
  else
    finish_columns<false>(A, S, c);
  __syncthreads();

  // dct2d (mod.rs:711-735): tmp[i][j] = sum_k D[i][k] * c[k][j], then
  // out[i][j] = sum_k tmp[i][k] * D[j][k]; each sum from 0.0, k ascending, a
  // product then an addition per term
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const int j = t & 127, i0 = 4 * (t >> 7);
#pragma unroll 8
  for (int k = 0; k < 127; k++) {
    const float cv = c[k * 128 + j];
    const f32x4 d = *reinterpret_cast<const f32x4*>(&L.dct_t[k * 16 + i0]);
    s[0] += d.x * cv;
    s[1] += d.y * cv;
    s[2] += d.z * cv;
    s[3] += d.w * cv;
  }
  __syncthreads();  // the samples are read: t overwrites them
#pragma unroll
  for (int q = 0; q < 4; q++) L.u.d.t[(i0 + q) * kTS + j] = s[q];
  __syncthreads();
  if (t < 256) {
    const int i = t >> 4, jj = t & 15;
    float v = 0.0f;
#pragma unroll 8
    for (int k = 0; k < 127; k++) v += L.u.d.t[i * kTS + k] * L.dct_t[k * 16 + jj];
    L.u.d.p[t] = v;
    if (pdqf) pdqf[(size_t)img * 256 + t] = v;
  }
  __syncthreads();

  // sum_of_gradients (mod.rs:737-761, the order of sum_of_gradients16) and
  // adjust_quality on one wave, quantize (mod.rs:764-788) on another
  const float* P = L.u.d.p;
  if (t == 64) quality[img] = adjust_quality(sum_of_gradients16(P));
  if (t >= 64) return;
  const float med = torben_median_wave(P, t);
  if (t == 0) threshold[img] = med;
  if (t < 32) {
    // byte 31 - t holds elements 8t .. 8t+7, bit j = element 8t + j > median
    uint32_t byte = 0;
#pragma unroll
    for (int b = 0; b < 8; b++) byte |= (P[8 * t + b] > med ? 1u : 0u) << b;
    hashes[(size_t)img * 32 + (31 - t)] = (uint8_t)byte;
  }
}

template <typename T>
void launch_ref_kind(const void* planes, uint64_t plane_stride, uint32_t n_images, float* work, uint8_t* hashes,
                     float* quality, float* threshold, float* pdqf, hipStream_t stream) {
  const T* p = static_cast<const T*>(planes);
  const dim3 lines(64 * ((n_images + 7) / 8)), wave(64);
  constexpr bool kF32 = std::is_same<T, float>::value;
  if constexpr (kF32)
    hipLaunchKernelGGL(pdq_ref_rows_kernel, lines, wave, 0, stream, p, plane_stride, n_images, work, hashes);
  hipLaunchKernelGGL(pdq_ref_cols_kernel<T>, lines, wave, 0, stream, p, plane_stride, n_images, work, hashes);
  hipLaunchKernelGGL(pdq_ref_sampled_kernel<kF32>, lines, wave, 0, stream, n_images, work, hashes);
  hipLaunchKernelGGL(pdq_ref_finish_kernel<T>, dim3(n_images), dim3(kRefThreads), 0, stream, work, hashes, quality,
                     threshold, pdqf);
}

}  // namespace

uint64_t hash_ref_workspace_bytes(uint32_t n_images) { return (uint64_t)n_images * 2 * 512 * 512 * sizeof(float); }

hipError_t launch_hash_ref(const void* planes, int input_kind, uint64_t plane_stride, uint32_t n_images, void* work,
                           uint8_t* hashes, float* quality, float* threshold, float* pdqf, hipStream_t stream) {
  if (n_images == 0) return hipSuccess;
  if (input_kind == kInputF32)
    launch_ref_kind<float>(planes, plane_stride, n_images, static_cast<float*>(work), hashes, quality, threshold, pdqf,
                           stream);
  else if (input_kind == kInputU8)
    launch_ref_kind<uint8_t>(planes, plane_stride, n_images, static_cast<float*>(work), hashes, quality, threshold,
                             pdqf, stream);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ypdq
