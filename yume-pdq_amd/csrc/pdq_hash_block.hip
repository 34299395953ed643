// Block-per-image form of the fused hash kernel for gfx950 (CDNA4): the
// wavefronts of one block share one 512x512 plane, so a launch of a few
// hundred images fills the chip and one image takes a fraction of the
// wave-per-image form's latency.
//
// Per image (kWaves wavefronts, 64 lanes each):
//   A. wave w compresses its band of rows of the 127x127 plane with the same
//      tent FMA chains as the wave-per-image form (x86.rs:626-682 order,
//      lane t owns output columns 2t and 2t+1) and stores them in LDS as a
//      128x128 f32 plane whose row and column 127 are zero.
//   B. DCT stage 1, T = D C (16 x 128).
//        exact:        v_mfma_f32_16x16x4_f32 runs the reference's two
//                      alternating FMA chains over k2 = 0..126
//                      (x86.rs:161-225) -- the chains, operands and order of
//                      the wave form, so the values are the same bits;
//        matrix cores: v_mfma_f32_16x16x32_{bf16,f16}, operands rounded to
//                      bf16 or f16 (round to nearest even) with f32
//                      accumulation, or the three products hi*hi + hi*lo +
//                      lo*hi of split operands x = hi + lo.
//   C. stage 2 (exact: x86.rs:227-272, two AVX lanes per wave on four waves;
//      rounded: four 16x16x32 products on wave 0), then the dihedrals on every
//      wave, and the thresholds and bits beside the qualities.
// Planes holding NaN/Inf take the literal 56-tap compression and the exact
// stage 1 in every form.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "pdq_hash_common.h"
#include "pdq_hash_tail.h"

namespace ypdq {

namespace {

typedef float f32x4v __attribute__((ext_vector_type(4)));

struct ImageTail {
  WaveLds w;
  float part[4][256];           // stage 2: the four pairs of AVX lanes
  float grad[8 * kGradStride];  // absolute differences of the eight orientations
};

struct ImageLds {
  union {
    float c[128 * 128];  // compressed plane, row-major, stride 128
    ImageTail tail;      // after stage 1
  } u;
  float dct_t[128 * 16];  // exact stages: D transposed, dct_t[k2 * 16 + k] = D[k][k2], row 127 zero
};

// Rows in flight per wave in the band loop: D compressed-row steps of four
// input rows each.
template <typename T>
struct BandPrefetch {
  static constexpr int D = 2;
};
template <>
struct BandPrefetch<uint8_t> {
  static constexpr int D = 4;
};

// ---------------------------------------------------------------------------
// A. compression of one band of rows into LDS
// ---------------------------------------------------------------------------
template <int S, int D, bool kScalar, typename T, typename Raw>
__device__ __forceinline__ void band_step(const T* __restrict__ plane, int lane, int i, int i_end, Chains& cur,
                                          Chains& nxt, Raw (&pre)[D][4], float* __restrict__ c, const Luma& lc,
                                          float& z) {
  // The rows D steps ahead are loaded unconditionally, clamped into the
  // plane (past the band's end they are not used): a load under a branch
  // makes the compiler copy the ring's registers and wait for every load in
  // flight.
  const int r0 = 4 * (i + D) + 3;
  auto row = [&](int d) { return min(r0 + d, 511); };
  (void)i_end;
  if constexpr (std::is_same<T, float>::value) {
    // f32 rows feed from their ring slots, which reload after their last use
    // (a copy out of the slot would cost eight moves per row)
    chains_feed<2>(cur, pre[S][0]);
    check_edges(z, pre[S][0]);
    load_raw<kScalar>(plane, row(0), lane, pre[S][0]);
    chains_feed<3>(cur, pre[S][1]);
    check_edges(z, pre[S][1]);
    load_raw<kScalar>(plane, row(1), lane, pre[S][1]);
    chains_feed<4>(cur, pre[S][2]);
    check_edges(z, pre[S][2]);
    chains_feed<5>(cur, pre[S][3]);
    check_edges(z, pre[S][3]);
    chains_start(nxt, pre[S][2], pre[S][3]);
    load_raw<kScalar>(plane, row(2), lane, pre[S][2]);
    load_raw<kScalar>(plane, row(3), lane, pre[S][3]);
  } else {
    // converted rows free their slots at once
    Row8 x, x2, x3;
    to_f32(pre[S][0], x, lc);
    load_raw<kScalar>(plane, row(0), lane, pre[S][0]);
    chains_feed<2>(cur, x);
    to_f32(pre[S][1], x, lc);
    load_raw<kScalar>(plane, row(1), lane, pre[S][1]);
    chains_feed<3>(cur, x);
    to_f32(pre[S][2], x2, lc);
    load_raw<kScalar>(plane, row(2), lane, pre[S][2]);
    chains_feed<4>(cur, x2);
    to_f32(pre[S][3], x3, lc);
    load_raw<kScalar>(plane, row(3), lane, pre[S][3]);
    chains_feed<5>(cur, x3);
    chains_start(nxt, x2, x3);
  }
  float c0, c1;
  chains_finish(cur, c0, c1);
  if (lane == 63) c1 = 0.0f;  // column 127 is the zero pad
  if constexpr (std::is_same<T, float>::value) z = __builtin_fmaf(c0, c1, z);
  *reinterpret_cast<float2*>(&c[i * 128 + 2 * lane]) = make_float2(c0, c1);
}

// D steps; the two chain sets trade roles from step to step (the next row's
// chains are the current ones of the step after), so no step copies them.
// kAll: every step runs (no test, so the ring's registers stay fixed);
// otherwise the steps up to the band's end.
template <int S, int D, bool kAll, bool kScalar, typename T, typename Raw>
__device__ __forceinline__ void band_steps(const T* __restrict__ plane, int lane, int i, int i_end, Chains& a,
                                           Chains& b, Raw (&pre)[D][4], float* __restrict__ c, const Luma& lc,
                                           float& z) {
  static_assert(D % 2 == 0, "an even number of steps returns the chain sets to their roles");
  if (kAll || i + S < i_end) {
    if constexpr (S % 2 == 0)
      band_step<S, D, kScalar>(plane, lane, i + S, i_end, a, b, pre, c, lc, z);
    else
      band_step<S, D, kScalar>(plane, lane, i + S, i_end, b, a, pre, c, lc, z);
  }
  if constexpr (S + 1 < D) band_steps<S + 1, D, kAll, kScalar>(plane, lane, i, i_end, a, b, pre, c, lc, z);
}

// Compressed rows [i0, i1) into c; true if an input value that the reference
// reads for them is NaN or Inf (f32 planes).
template <bool kScalar, typename T>
__device__ __forceinline__ bool compress_band(const T* __restrict__ plane, int lane, int i0, int i1,
                                              float* __restrict__ c, const Luma& lc) {
  using Raw = typename RawRow<T>::type;
  constexpr int D = BandPrefetch<T>::D;
  Chains cur, nxt;
  Raw pre[D][4];
  float z = 0.0f;
  {
    Raw r1, r2;
    load_raw<kScalar>(plane, 4 * i0 + 1, lane, r1);
    load_raw<kScalar>(plane, 4 * i0 + 2, lane, r2);
#pragma unroll
    for (int s = 0; s < D; s++)
#pragma unroll
      for (int d = 0; d < 4; d++) load_raw<kScalar>(plane, min(4 * (i0 + s) + 3 + d, 511), lane, pre[s][d]);
    Row8 x1, x2;
    to_f32(r1, x1, lc);
    to_f32(r2, x2, lc);
    chains_start(cur, x1, x2);
    if constexpr (std::is_same<T, float>::value) {
      // rows 1 and 511 whole; the other bands' first two rows are the last
      // two of the band before
      if (i0 == 0) {
        check_row(z, x1);
        check_edges(z, x2);
      }
      if (i1 == 127) {
        Row8 last;
        load_row<kScalar>(plane, 511, lane, last);
        check_row(z, last);
      }
    }
  }
  int i = i0;
#pragma unroll 1
  for (; i + D <= i1; i += D) band_steps<0, D, true, kScalar>(plane, lane, i, i1, cur, nxt, pre, c, lc, z);
  if (i < i1) band_steps<0, D, false, kScalar>(plane, lane, i, i1, cur, nxt, pre, c, lc, z);
  return nonfinite(z);
}

// ---------------------------------------------------------------------------
// B. stage 1 and 2, exact, on matrix cores.
//
// v_mfma_f32_16x16x4_f32 is four fused multiply-adds in order of k, each
// rounded to nearest even, subnormals, infinities and NaN included (checked
// against fmaf chains), so the reference's FMA chains run on it as they are,
// four terms an instruction: lane l supplies A[l%16][l/16] and B[l/16][l%16]
// and receives D[4 (l/16) + r][l%16], r = 0..3.  On the vector ALU stage 1 was
// bound by issue and LDS, 508 FMAs a wave on eight waves (of one u8 image's
// 40000 cycles stage 1 with its barriers took 8400 and takes 4600, stage 2 1800
// and 1600).  One u8 plane 16.9 -> 14.9 us in all, 1000 planes 70.1 -> 63.6.
// ---------------------------------------------------------------------------
// The term of chain p (alt()) that lane group g supplies to its step s: chain
// 1 takes terms 0, 3, 4, 7, 8, .., chain 0 terms 1, 2, 5, 6, 9, ...
__device__ __forceinline__ int chain_term(int p, int s, int g) {
  const int even = g & 2;  // the first or second pair of four terms
  return 8 * s + 2 * even + (p == 1 ? (g & 1) * 3 : 1 + (g & 1));
}

// T[:, 16 jt .. 16 jt + 15] = D C: the two chains over k2 = 0..126
// (x86.rs:161-225; term 127 is zero on both sides), then their sum, a chain's
// NaN as zero, column 127 zero.  c: the plane, dt: the transposed DCT.
__device__ __forceinline__ f32x4v stage1_exact(const float* __restrict__ c, const float* __restrict__ dt, int lane,
                                               int jt) {
  const int m = lane & 15, g = lane >> 4;
  f32x4v acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
  for (int s = 0; s < 16; s++) {
#pragma unroll
    for (int p = 1; p >= 0; p--) {
      const int k = chain_term(p, s, g);
      acc[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(dt[k * 16 + m], c[k * 128 + 16 * jt + m], acc[p], 0, 0, 0);
    }
  }
  f32x4v t;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const float a0 = __builtin_isnan(acc[0][r]) ? 0.0f : acc[0][r];
    const float a1 = __builtin_isnan(acc[1][r]) ? 0.0f : acc[1][r];
    t[r] = 16 * jt + m == 127 ? 0.0f : a0 + a1;
  }
  return t;
}

// Stage 2 (x86.rs:227-272) for AVX lanes 2 w and 2 w + 1: the two chains of
// each over its 16 terms, 8 c + l for chunk c, and (lane 2 w) + (lane 2 w + 1)
// of their sums, the first level of the reference's horizontal tree, into
// part[k * 16 + j].
__device__ __forceinline__ void stage2_exact(const WaveLds& W, const float* __restrict__ dt, int lane, int w,
                                             float* __restrict__ part) {
  const int m = lane & 15, g = lane >> 4;
  f32x4v v[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int l = 2 * w + i;
    f32x4v acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const int k = 8 * chain_term(p, s, g) + l;
        // term 127 holds the reference's over-read D_flat[127 j + 127], which
        // is D[j + 1][0] (0 after row 15)
        const float d = dt[k < 127 ? k * 16 + m : m < 15 ? m + 1 : 0];
        acc[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.t[m * kTS + k], k == 127 && m == 15 ? 0.0f : d, acc[p], 0, 0,
                                                      0);
      }
    v[i] = acc[0] + acc[1];
  }
#pragma unroll
  for (int r = 0; r < 4; r++) part[(4 * g + r) * 16 + m] = v[0][r] + v[1][r];
}

// ---------------------------------------------------------------------------
// B'. stage 1 and 2 on matrix cores.
//
// v_mfma_f32_16x16x32_{bf16,f16}: lane l supplies row l%16 of A and column
// l%16 of B, eight consecutive k each (group g = l/16 holds k = 8g .. 8g+7 of
// the 32); it receives D[4g + r][l%16], r = 0..3.  A and B use the same k
// assignment, so the contraction is right whatever order the unit sums in.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// bf16 bits of a finite float, rounded to nearest even.
__device__ __forceinline__ uint32_t bf16_rne(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// Eight floats as an operand pair: hi = round(x), lo = round(x - hi).
template <int kPrec>
struct Operand;

template <>
struct Operand<kDctBf16> {
  bf16x8 hi, lo;
  __device__ __forceinline__ void set(const float (&x)[8], bool split) {
    u32x4 h, l;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const uint32_t a = bf16_rne(x[2 * e]), b = bf16_rne(x[2 * e + 1]);
      h[e] = a | (b << 16);
      if (split) {
        const uint32_t al = bf16_rne(x[2 * e] - __uint_as_float(a << 16));
        const uint32_t bl = bf16_rne(x[2 * e + 1] - __uint_as_float(b << 16));
        l[e] = al | (bl << 16);
      } else {
        l[e] = 0;
      }
    }
    hi = __builtin_bit_cast(bf16x8, h);
    lo = __builtin_bit_cast(bf16x8, l);
  }
  static __device__ __forceinline__ f32x4v mma(const bf16x8& a, const bf16x8& b, const f32x4v& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

template <>
struct Operand<kDctF16> {
  f16x8 hi, lo;
  __device__ __forceinline__ void set(const float (&x)[8], bool split) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const _Float16 h = (_Float16)x[e];
      hi[e] = h;
      lo[e] = split ? (_Float16)(x[e] - (float)h) : (_Float16)0.0f;
    }
  }
  static __device__ __forceinline__ f32x4v mma(const f16x8& a, const f16x8& b, const f32x4v& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// Operand type and split flag of each matrix-core precision.
template <int kPrec>
struct Precision {
  static constexpr int kBase = (kPrec == kDctBf16 || kPrec == kDctBf16x3) ? kDctBf16 : kDctF16;
  static constexpr bool kSplit = kPrec == kDctBf16x3 || kPrec == kDctF16x3;
  using Op = Operand<kBase>;
};

// acc += a * b (hi + lo split: the two cross terms first, then hi * hi).
template <int kPrec>
__device__ __forceinline__ f32x4v mma_acc(const typename Precision<kPrec>::Op& a,
                                          const typename Precision<kPrec>::Op& b, f32x4v acc) {
  using Op = typename Precision<kPrec>::Op;
  if constexpr (Precision<kPrec>::kSplit) {
    acc = Op::mma(a.lo, b.hi, acc);
    acc = Op::mma(a.hi, b.lo, acc);
  }
  return Op::mma(a.hi, b.hi, acc);
}

// Row l%16 of the DCT matrix, k = 32s + 8g .. +7 (column 127 is zero).
template <int kPrec>
__device__ __forceinline__ void dct_operands(int lane, typename Precision<kPrec>::Op (&d)[4]) {
  const int m = lane & 15, g = lane >> 4;
#pragma unroll
  for (int s = 0; s < 4; s++) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int k = 32 * s + 8 * g + e;
      x[e] = k < 127 ? kDct[m * 127 + k] : 0.0f;
    }
    d[s].set(x, Precision<kPrec>::kSplit);
  }
}

// T[:, 16 jt .. 16 jt + 15] = D C on matrix cores.
template <int kPrec>
__device__ __forceinline__ f32x4v stage1_mfma(const float* __restrict__ c, int lane, int jt,
                                              const typename Precision<kPrec>::Op (&d)[4]) {
  const int n = lane & 15, g = lane >> 4;
  f32x4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < 4; s++) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = c[(32 * s + 8 * g + e) * 128 + 16 * jt + n];
    typename Precision<kPrec>::Op b;
    b.set(x, Precision<kPrec>::kSplit);
    acc = mma_acc<kPrec>(d[s], b, acc);
  }
  return acc;
}

// PDQF = T D^T on matrix cores (one wave): A = T rows, B = the DCT operands.
template <int kPrec>
__device__ __forceinline__ void stage2_mfma(WaveLds& W, int lane, const typename Precision<kPrec>::Op (&d)[4]) {
  const int m = lane & 15, g = lane >> 4;
  f32x4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const f32x4* tp = reinterpret_cast<const f32x4*>(&W.t[m * kTS + 32 * s + 8 * g]);
    const f32x4 ta = tp[0], tb = tp[1];
    const float x[8] = {ta.x, ta.y, ta.z, ta.w, tb.x, tb.y, tb.z, tb.w};
    typename Precision<kPrec>::Op a;
    a.set(x, Precision<kPrec>::kSplit);
    acc = mma_acc<kPrec>(a, d[s], acc);
  }
#pragma unroll
  for (int r = 0; r < 4; r++) W.p[(4 * g + r) * 16 + m] = acc[r];
  wave_lds_sync();
}

// ---------------------------------------------------------------------------
// The kernel: one block of kWaves wavefronts per image.
// ---------------------------------------------------------------------------
template <typename T, int kPrec, int kWaves>
__global__ void __launch_bounds__(64 * kWaves) pdq_hash_block_kernel(const T* __restrict__ planes,
                                                                     uint64_t plane_stride, uint32_t n_images,
                                                                     const uint32_t* __restrict__ d_n, uint32_t mode,
                                                                     HashOutputs out, Luma lc) {
  static_assert(kWaves == 4 || kWaves == 8 || kWaves == 16, "four, eight or sixteen waves per image");
  static_assert(kWaves <= 8 || kPrec == kDctExact, "sixteen waves: exact arithmetic only");
  constexpr int kBand = (127 + kWaves - 1) / kWaves;  // compressed rows per wave
  if (out.clear && blockIdx.x == 0 && threadIdx.x == 0) *out.clear = 0;
  const uint32_t n = d_n ? min(*d_n, n_images) : n_images;
  const uint32_t img = blockIdx.x;
  if (img >= n) return;
  __shared__ ImageLds L;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const T* plane = reinterpret_cast<const T*>(reinterpret_cast<const uint8_t*>(planes) + (size_t)img * plane_stride);
  float* c = L.u.c;

  // A. compression; the DCT table for stage 1 is copied into LDS after it,
  // so the first plane rows are requested at the kernel's start
  const int i0 = wv * kBand, i1 = min(i0 + kBand, 127);
  constexpr bool kScalar = kWaves == 16 || !std::is_same<T, uint8_t>::value;  // row addresses (row_words)
  const bool bad = compress_band<kScalar>(plane, lane, i0, i1, c, lc);
  if (wv == kWaves - 1) *reinterpret_cast<float2*>(&c[127 * 128 + 2 * lane]) = make_float2(0.0f, 0.0f);
  if (kPrec == kDctExact || std::is_same<T, float>::value)
    for (int e = t; e < 128 * 16; e += 64 * kWaves) L.dct_t[e] = e < 127 * 16 ? kDctT.v[e] : 0.0f;
  const bool literal = __syncthreads_or(bad ? 1 : 0) != 0;
  if constexpr (std::is_same<T, float>::value) {
    if (literal) {
      // 56 literal taps per output (NaN/Inf propagate through zero weights
      // as in the reference)
#pragma unroll 1
      for (int i = i0; i < i1; i++) {
        const float a = compress_one_literal(plane, i, 2 * lane, lc);
        const float b = lane == 63 ? 0.0f : compress_one_literal(plane, i, 2 * lane + 1, lc);
        *reinterpret_cast<float2*>(&c[i * 128 + 2 * lane]) = make_float2(a, b);
      }
      __syncthreads();
    }
  }
  if (out.buf1) {
    float* b1 = out.buf1 + (size_t)img * 128 * 128;
    for (int e = t; e < 128 * 128; e += 64 * kWaves) b1[e] = c[e];
  }

  WaveLds& W = L.u.tail.w;
  if (kPrec == kDctExact || literal) {
    // B. exact stage 1: wave w computes column tiles w, w + kWaves, ...
    constexpr int kTiles = kWaves < 8 ? 8 / kWaves : 1;
    f32x4v tile[kTiles];
    if (wv < 8) {
#pragma unroll
      for (int q = 0; q < kTiles; q++) tile[q] = stage1_exact(c, L.dct_t, lane, wv + kWaves * q);
    }
    __syncthreads();  // every read of the plane is done: T overwrites it
    if (wv < 8) {
      const int nn = lane & 15, g = lane >> 4;
#pragma unroll
      for (int q = 0; q < kTiles; q++)
#pragma unroll
        for (int r = 0; r < 4; r++) W.t[(4 * g + r) * kTS + 16 * (wv + kWaves * q) + nn] = tile[q][r];
    }
  } else if constexpr (kPrec != kDctExact) {
    // B'. stage 1 on matrix cores: wave w computes column tiles w, w + kWaves
    typename Precision<kPrec>::Op d[4];
    dct_operands<kPrec>(lane, d);
    constexpr int kTiles = 8 / kWaves;
    f32x4v acc[kTiles];
#pragma unroll
    for (int q = 0; q < kTiles; q++) acc[q] = stage1_mfma<kPrec>(c, lane, wv + kWaves * q, d);
    __syncthreads();
    const int nn = lane & 15, g = lane >> 4;
#pragma unroll
    for (int q = 0; q < kTiles; q++)
#pragma unroll
      for (int r = 0; r < 4; r++) W.t[(4 * g + r) * kTS + 16 * (wv + kWaves * q) + nn] = acc[q][r];
  }
  __syncthreads();

  // C. stage 2 and the tail
  if (kPrec == kDctExact || literal) {
    if (wv < 4) stage2_exact(W, L.dct_t, lane, wv, L.u.tail.part[wv]);
    __syncthreads();
    if (t < 256) {
      const float(&s)[4][256] = L.u.tail.part;
      W.p[t] = (s[0][t] + s[1][t]) + (s[2][t] + s[3][t]);
    }
  } else if (wv == 0) {
    typename Precision<kPrec>::Op d[4];
    dct_operands<kPrec>(lane, d);
    stage2_mfma<kPrec>(W, lane, d);
  }
  if (wv == kWaves - 1) write_tmp(W, lane, out, img);
  __syncthreads();
  // the eight orientations' PDQFs, written by every wave (two orientations
  // per element and thread with sixteen waves)
  {
    constexpr int kPer = 8 / (kWaves / 4);  // orientations per thread
    const int idx = t & 255, d0 = (t >> 8) * kPer;
    dihedral_pdqf_element(W, idx, d0, kPer, mode, kWaves >= 8 ? L.u.tail.grad : nullptr);
  }
  __syncthreads();
  if constexpr (kWaves >= 8) {
    // waves 0..3 search the four thresholds and write the hashes, wave 4 the
    // qualities, the others the optional PDQF outputs
    if (wv < 4) {
      tail_rows_thresholds_bits(W, lane, wv, out, img, nullptr);
    } else if (wv == 4) {
      tail_quality_sums(L.u.tail.grad, W, lane, out, img);
    } else {
      tail_copy_pdqfs(W, t - 5 * 64, 64 * (kWaves - 5), out, img);
    }
  } else {
    // the quality on wave 1 while wave 0 searches the thresholds
    if (wv == 1) tail_quality(W, lane, out, img, true);
    if (wv == 0) tail_thresholds_bits(W, lane, out, img, nullptr);
  }
}

template <typename T, int kPrec, int kWaves>
void launch_block_kind(const void* planes, uint64_t plane_stride, uint32_t n_max, const uint32_t* d_n, uint32_t mode,
                       const HashOutputs& out, const Luma& lc, hipStream_t stream) {
  hipLaunchKernelGGL((pdq_hash_block_kernel<T, kPrec, kWaves>), dim3(n_max), dim3(64 * kWaves), 0, stream,
                     static_cast<const T*>(planes), plane_stride, n_max, d_n, mode, out, lc);
}

template <typename T, int kWaves>
hipError_t launch_block_dct(int dct, const void* planes, uint64_t plane_stride, uint32_t n_max, const uint32_t* d_n,
                            uint32_t mode, const HashOutputs& out, const Luma& lc, hipStream_t stream) {
  switch (dct) {
    case kDctExact: launch_block_kind<T, kDctExact, kWaves>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    case kDctBf16: launch_block_kind<T, kDctBf16, kWaves>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    case kDctF16: launch_block_kind<T, kDctF16, kWaves>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    case kDctBf16x3: launch_block_kind<T, kDctBf16x3, kWaves>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    case kDctF16x3: launch_block_kind<T, kDctF16x3, kWaves>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int kWaves>
hipError_t launch_block_waves(const void* planes, int input_kind, uint64_t plane_stride, uint32_t n_max,
                              const uint32_t* d_n, uint32_t mode, int dct, const HashOutputs& out, const Luma& lc,
                              hipStream_t stream) {
  switch (input_kind) {
    case kInputF32: return launch_block_dct<float, kWaves>(dct, planes, plane_stride, n_max, d_n, mode, out, lc, stream);
    case kInputU8: return launch_block_dct<uint8_t, kWaves>(dct, planes, plane_stride, n_max, d_n, mode, out, lc, stream);
    case kInputRgb8: return launch_block_dct<Rgb8, kWaves>(dct, planes, plane_stride, n_max, d_n, mode, out, lc, stream);
    case kInputRgba8: return launch_block_dct<Rgba8, kWaves>(dct, planes, plane_stride, n_max, d_n, mode, out, lc, stream);
    default: return hipErrorInvalidValue;
  }
}

// Sixteen waves per image: exact arithmetic only.
hipError_t launch_block_waves16(const void* planes, int input_kind, uint64_t plane_stride, uint32_t n_max,
                                const uint32_t* d_n, uint32_t mode, int dct, const HashOutputs& out, const Luma& lc,
                                hipStream_t stream) {
  if (dct != kDctExact) return hipErrorInvalidValue;
  switch (input_kind) {
    case kInputF32: launch_block_kind<float, kDctExact, 16>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    case kInputU8: launch_block_kind<uint8_t, kDctExact, 16>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    case kInputRgb8: launch_block_kind<Rgb8, kDctExact, 16>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    case kInputRgba8: launch_block_kind<Rgba8, kDctExact, 16>(planes, plane_stride, n_max, d_n, mode, out, lc, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
                                              hipSuccess)
    return 0;
  return cus;
}

}  // namespace

int hash_layout_for(uint32_t n_images, int input_kind, int dct) {
  // Exact arithmetic: blocks of sixteen waves while a handful of images leaves
  // most CUs to themselves and the rows' conversion is what their waves do,
  // then eight, until the batch is large enough that a wave per image fills the
  // GPU with less LDS per image.  Sixteen / eight waves, in us:
  //   images          1           32           64          128          256
  //   u8       14.9 / 15.0  17.6 / 16.9  18.2 / 17.2  19.0 / 17.6  23.6 / 21.1
  //   f32      17.7 / 16.9  19.1 / 18.4  23.4 / 22.1  30.5 / 28.7  55.0 / 51.6
  //   RGB8     21.1 / 22.0  22.0 / 22.9  22.6 / 23.5  27.0 / 24.3  44.9 / 38.9
  //   RGBA8    19.5 / 20.2  20.5 / 21.2  24.5 / 22.1  32.2 / 28.6  57.1 / 50.7
  // (u8 crosses between 8 and 16 images, RGB8 at 96, RGBA8 between 32 and 48.)
  // The upper lines cross at 5.5 images per CU (u8 and RGB8 a little above,
  // f32 and RGBA8 there); eight waves / a wave per image:
  //   images      1100        1365        1536        2048
  //   u8        75 / 91     88 / 92     93 / 95   120 / 108
  //   RGB8     167 / 202   201 / 226   215 / 230   282 / 292
  //   f32      231 / 273   278 / 285   293 / 291   385 / 367
  //   RGBA8    230 / 267   276 / 284   301 / 294   397 / 376
  // Matrix-core arithmetic exists only in the block forms of 4 and 8 waves.
  if (dct != kDctExact) return 8;
  const uint32_t cus = (uint32_t)std::max(0, device_cus());
  if (cus == 0) return n_images > 1024 ? 1 : 8;
  const uint32_t sixteen = input_kind == kInputU8      ? cus / 32
                           : input_kind == kInputRgb8  ? cus / 8 * 3
                           : input_kind == kInputRgba8 ? cus / 8
                                                       : 0;
  return n_images <= sixteen ? 16 : n_images <= cus * 11 / 2 ? 8 : 1;
}

hipError_t launch_hash(const void* planes, int input_kind, uint64_t plane_stride, uint32_t n_images, uint32_t mode,
                       const HashOutputs& out, hipStream_t stream, const float* luma) {
  const int layout = hash_layout_for(n_images, input_kind, kDctExact);
  if (layout == 1)
    return launch_hash_wave(planes, input_kind, plane_stride, n_images, nullptr, mode, out, luma, stream);
  return launch_hash_block(planes, input_kind, plane_stride, n_images, nullptr, mode, kDctExact, layout, out, luma,
                           stream);
}

hipError_t launch_hash_device_count(const void* planes, int input_kind, uint64_t plane_stride, uint32_t n_max,
                                    const uint32_t* d_n, uint32_t mode, const HashOutputs& out, hipStream_t stream) {
  const int layout = hash_layout_for(n_max, input_kind, kDctExact);
  if (layout == 1)
    return launch_hash_wave(planes, input_kind, plane_stride, n_max, d_n, mode, out, nullptr, stream);
  return launch_hash_block(planes, input_kind, plane_stride, n_max, d_n, mode, kDctExact, layout, out, nullptr,
                           stream);
}

hipError_t launch_hash_block(const void* planes, int input_kind, uint64_t plane_stride, uint32_t n_max,
                             const uint32_t* d_n, uint32_t mode, int dct, int waves, const HashOutputs& out,
                             const float* luma, hipStream_t stream) {
  if (n_max == 0) return hipSuccess;
  Luma lc{0.299f, 0.587f, 0.114f};
  if (luma) lc = Luma{luma[0], luma[1], luma[2]};
  if (waves == 16) return launch_block_waves16(planes, input_kind, plane_stride, n_max, d_n, mode, dct, out, lc, stream);
  if (waves == 8) return launch_block_waves<8>(planes, input_kind, plane_stride, n_max, d_n, mode, dct, out, lc, stream);
  if (waves == 4) return launch_block_waves<4>(planes, input_kind, plane_stride, n_max, d_n, mode, dct, out, lc, stream);
  return hipErrorInvalidValue;
}

}  // namespace ypdq
