// Matrix-core Hamming matcher for large query batches (gfx950, fp4 MFMA).
//
// The reference's predicate is popcount(q ^ r) <= threshold over 256 bits
// (src/matching/mod.rs:232-257, 336-362).  Writing each bit as +1/-1, the
// dot product of two such vectors over the first 128 bits is
//     dot128 = 128 - 2 * d128,     d128 = popcount of the first 128 XOR bits,
// and d128 <= d256 always, so d256 <= t  implies  dot128 >= 128 - 2t.
// +-1 are exact fp4 (e2m1) values and |dot128| <= 128 is exact in the fp32
// accumulator, so one v_mfma_scale_f32_16x16x128_f8f6f4 computes d128 for a
// 16-query x 16-row tile exactly.  Tiles whose maximum clears the bound
// (for random rows with t = 31: about 1e-9 of pairs, plus the true hits) are
// re-checked pair by pair with the full 256-bit integer distance, so the
// result is the exact set the reference defines -- the matrix pass is only a
// filter that can never drop a pair.  Used for t < 64 (above that the prefix
// bound passes everything) and batches of 32 queries, 12 at threshold <= 40.
//
// Operand layout (measured on gfx950): lane l holds row/column (l & 15) and
// K quarter (l >> 4), i.e. 32 fp4 values = one 32-bit word of the 128-bit
// prefix; the output element C[m][n] is in lane (n + 16*(m >> 2)), register
// (m & 3).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <thread>
#include <tuple>
#include <utility>

#include "pdq_device.h"

namespace ypdq {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kMfmaWaves = 4;
constexpr int kMfmaTilesPerWave = 64;  // 16-row tiles streamed per wave per block

// Operand codes, fp4 e2m1: 0x2 = +1.0 (bit clear), 0xA = -1.0 (bit set), 0x0
// = 0.  A bit is its code's sign, so a word expands by masks alone: register k
// takes the bits at positions 3 - k, 7 - k, .. 31 - k as its eight signs.
// Queries and rows go through the same function, so every bit meets its
// counterpart, and the order of a dot product's terms is free (its partial
// sums are exact whole numbers).  Seven vector instructions per word, as many
// as the addresses of a byte table in LDS took, without its reads, its set-up
// at each block's start or its barrier (same times at full occupancy).
struct Expanded {
  uint32_t d[4];
};

__device__ __forceinline__ void expand_word(uint32_t w, Expanded& e) {
#pragma unroll
  for (int k = 0; k < 4; k++) e.d[k] = ((w << k) & 0x88888888u) | 0x22222222u;
}

__device__ __forceinline__ v4f mfma_prefix(const Expanded& a, const Expanded& b) {
  v8i av = {(int)a.d[0], (int)a.d[1], (int)a.d[2], (int)a.d[3], 0, 0, 0, 0};
  v8i bv = {(int)b.d[0], (int)b.d[1], (int)b.d[2], (int)b.d[3], 0, 0, 0, 0};
  v4f c = {0.0f, 0.0f, 0.0f, 0.0f};
  // cbsz = blgp = 4: both operands fp4 e2m1; no scales
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 4, 4, 0, 0, 0, 0);
}

__device__ __forceinline__ uint32_t full_distance(const uint32_t* __restrict__ a, const uint32_t* __restrict__ b) {
  uint32_t d = 0;
#pragma unroll
  for (int w = 0; w < 8; w++) d += (uint32_t)__builtin_popcount(a[w] ^ b[w]);
  return d;
}

// A block's hits gather in LDS and take their places in the hit buffer with
// one atomic: thousands of appends to the one global counter from a short
// kernel serialise on it (measured in the recheck kernel: 49 of 68
// microseconds for 4938 hits).  Hits past the list append directly.
template <uint32_t kList>
struct HitList {
  MatchHit stage[kList];
  uint32_t n;
  unsigned long long base;
};
constexpr uint32_t kStageHits = 4096;  // recheck kernel: two blocks per CU, about two million per launch
// Even layout: four blocks per CU, two million per launch too (32 KiB each).
// With 512 a block, 10^6 rows that each match one of 512 queries took 5.8 ms,
// nearly all of it half a million appends of their own, and take 0.27.
constexpr uint32_t kEvenStage = 2040;
constexpr uint32_t kHeldStage = 512;  // held layout: what two blocks' query codes leave in LDS

template <uint32_t kList>
__device__ __forceinline__ void hits_init(HitList<kList>& L) {
  if (threadIdx.x == 0) L.n = 0;
  __syncthreads();
}

// The gathered hits into the buffer: one run of places.  Every thread of the
// block calls it.
template <uint32_t kList>
__device__ __forceinline__ void hits_flush(HitList<kList>& L, MatchHit* __restrict__ hits, uint64_t capacity,
                                           unsigned long long* __restrict__ counter) {
  __syncthreads();
  const uint32_t n = min(L.n, kList);
  if (n == 0) return;  // the same for the whole block
  if (threadIdx.x == 0) L.base = atomicAdd(counter, (unsigned long long)n);
  __syncthreads();
  const unsigned long long base = L.base;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
    if (base + i < capacity) hits[base + i] = L.stage[i];
}

// Exact check of query tile t's candidates in this lane's four outputs.
template <uint32_t kList>
__device__ __forceinline__ void stage_candidates(v4f cv, int t, uint64_t tbase, uint32_t qbase, int rn, int kq,
                                                float bound, const uint32_t* __restrict__ queries,
                                                const uint32_t* __restrict__ db, uint32_t n_queries, uint64_t n_rows,
                                                uint32_t threshold, HitList<kList>& L,
                                                MatchHit* __restrict__ hits, uint64_t capacity,
                                                unsigned long long* __restrict__ counter, uint64_t index_base) {
  const uint64_t row = tbase + rn;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const float v = r == 0 ? cv.x : r == 1 ? cv.y : r == 2 ? cv.z : cv.w;
    if (v >= bound) {
      const uint32_t qi = qbase + 16 * t + 4 * kq + r;
      if (qi < n_queries && row < n_rows) {
        const uint32_t d = full_distance(queries + (size_t)qi * 8, db + row * 8);
        if (d <= threshold) {
          MatchHit h;
          h.query = qi;
          h.distance = d;
          h.index = index_base + row;
          const uint32_t s = atomicAdd(&L.n, 1u);
          if (s < kList) {
            L.stage[s] = h;
          } else {
            const unsigned long long slot = atomicAdd(counter, 1ull);
            if (slot < capacity) hits[slot] = h;
          }
        }
      }
    }
  }
}

// Packed candidate flags: the filter of the streaming loops.  The products
// of one row tile with two query tiles share one accumulator.  The first
// MFMA adds dot_a to C0 = 2^23 + K + 512 K, the second adds 512 dot_b (its
// query operand scaled by 2^9 through the MFMA's block scale), so each
// result is
//     2^23 + f_a + 512 f_b,   f = dot + K,   K = 256 - bound,
// an integer in [2^23, 2^24) -- as is every partial sum, in any order of
// accumulation -- so it is exact, and its low 23 bits are the two fields.
// dot is in [-128, 128], so f is in [128 - bound, 384 - bound], below 512
// (no carry between fields; bound = 128 - 2t is in [2, 128] for t < 64), and
// f >= 256 exactly when dot >= bound: bit 8 flags pair a, bit 17 pair b.
// One OR of the four results' bits then tests 8 pairs, where a maximum
// needs one instruction per 2 values.
constexpr uint32_t kFlagMask = (1u << 8) | (1u << 17);
constexpr int kFlagChains = 4;
constexpr int kScale1 = 127;      // 2^0
constexpr int kScale512 = 127 + 9;  // 2^9

__device__ __forceinline__ v4f flags_c0(float bound) {
  const float k = 256.0f - bound;
  const float c = 8388608.0f + k + 512.0f * k;  // exact: an integer below 2^24
  return v4f{c, c, c, c};
}

// A scale of one is left out: zero for both scale operands is the product
// without them, whose issue costs one vector instruction less (16x16x128
// products beside two vector instructions each: 19.8 against 23.4 cycles; 10^7
// rows against 1000 queries 347 us with it, 336 without, 200 queries 90.1 and
// 87.8).
template <int kScaleA>
__device__ __forceinline__ v4f mfma_acc(const Expanded& a, const Expanded& b, const v4f& c) {
  v8i av = {(int)a.d[0], (int)a.d[1], (int)a.d[2], (int)a.d[3], 0, 0, 0, 0};
  v8i bv = {(int)b.d[0], (int)b.d[1], (int)b.d[2], (int)b.d[3], 0, 0, 0, 0};
  if constexpr (kScaleA == kScale1)
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 4, 4, 0, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 4, 4, 0, kScaleA, 0, kScale1);
}

// The empty asm pins m here: without it the compiler gathers every fold of a
// group into one OR tree at the group's end, which keeps all the group's
// results live at once.
__device__ __forceinline__ void fold_flags(const v4f& v, uint32_t& m) {
  m = m | __float_as_uint(v.x) | __float_as_uint(v.y);
  m = m | __float_as_uint(v.z) | __float_as_uint(v.w);
  asm volatile("" : "+v"(m));
}

// Query tiles per wave of the shared-rows layout.
constexpr int kSharedQt = 16;
constexpr int kSharedPairs = kSharedQt / 2;  // per row tile

// The query pair of pair P of a row tile.  Pair P's products go to result
// register P % 4 and are folded into flag chain P % 4; the pairs are ordered so
// that chains 0 and 1 hold query tiles 0-7 and chains 2 and 3 tiles 8-15, so one
// vote per half tells which half of the query tiles has candidates.
__device__ constexpr int query_pair(int p) {
  constexpr int order[kSharedPairs] = {0, 1, 4, 5, 2, 3, 6, 7};
  return order[p % kSharedPairs];
}

// Pair P (row tile P / 8, query tiles 2 query_pair(P) and +1): its first
// product issues at step P into result register P % 4, its second at step
// P + 1 (one product after, so the accumulation does not wait), and its bits
// are folded at step P + 4, before the register takes pair P + 4.  The four
// result registers are named, not an array, so the compiler keeps each in
// place.
template <int kTiles, int S>
__device__ __forceinline__ void group_flags_step(const Expanded (&qa)[kSharedQt], const Expanded (&rb)[kTiles],
                                                 const v4f& c0, uint32_t (&acc)[kFlagChains], v4f& r0, v4f& r1,
                                                 v4f& r2, v4f& r3) {
  constexpr int kN = kSharedPairs * kTiles;  // pairs
  v4f& cur = (S % 4 == 0) ? r0 : (S % 4 == 1) ? r1 : (S % 4 == 2) ? r2 : r3;
  v4f& prev = (S % 4 == 1) ? r0 : (S % 4 == 2) ? r1 : (S % 4 == 3) ? r2 : r3;
  if constexpr (S >= 4) fold_flags(cur, acc[(S - 4) % kFlagChains]);
  if constexpr (S < kN) cur = mfma_acc<kScale1>(qa[2 * query_pair(S)], rb[S / kSharedPairs], c0);
  if constexpr (S >= 1 && S - 1 < kN)
    prev = mfma_acc<kScale512>(qa[2 * query_pair(S - 1) + 1], rb[(S - 1) / kSharedPairs], prev);
  // keep this order: hoisting the products runs out of registers
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (S + 1 < kN + 4) group_flags_step<kTiles, S + 1>(qa, rb, c0, acc, r0, r1, r2, r3);
}

template <int kTiles>
__device__ __forceinline__ void group_flags(const Expanded (&qa)[kSharedQt], const Expanded (&rb)[kTiles],
                                            const v4f& c0, uint32_t (&acc)[kFlagChains]) {
  v4f r0, r1, r2, r3;
  group_flags_step<kTiles, 0>(qa, rb, c0, acc, r0, r1, r2, r3);
}

// Three products per accumulator (sixteen query tiles, thresholds 28..63).
// The products of one row tile with query tiles a, b, c add dot_a (scale
// 2^0), 2^7 dot_b and 2^15 dot_c to
//     C0 = 2^23 + K_a + 2^8 K_b + 2^16 K_c,
//     K_a = 128 - bound,  K_b = 129 - bound/2,  K_c = 64 - bound/2,
// so, dot being even, the result is 2^23 + f_a + 2^8 f_b + 2^16 f_c with
// f_a = dot_a + K_a, f_b = dot_b/2 + K_b, f_c = dot_c/2 + K_c.  Every
// partial sum, in any order, is an integer in (2^22, 2^24): exact.
//   bit 7:  f_a >= 128, i.e. dot_a >= bound (f_a <= 254: no carry);
//   bit 15: f_b >= 128, i.e. dot_b >= bound - 2 (f_b in [1, 192]);
//   bit 22: f_c >= 64, i.e. dot_c >= bound (f_c <= 127).
// f_a or f_c below zero (dot < bound - 128: a prefix distance above 64 + t,
// about 6e-9 of random pairs at t = 31) borrows: a borrow from f_a shows
// in bit 7 (f_a + 256 >= 128) and lowers f_b by one, which the slack of
// K_b (a flag from dot_b >= bound - 2) absorbs; a borrow from f_c takes the
// result below 2^23, which changes the exponent's lowest bit, bit 23.  So a
// pair at the bound always sets one of the four bits, and the other causes
// are rare false candidates that the recheck discards.  tests/test_flag_fields.py
// checks this over every (dot_a, dot_b, dot_c) and threshold.
// Per row tile the sixteen query tiles form accumulators of (0,1,2),
// (3,4,5), (6,7), (8,9,10), (11,12,13), (14,15): twelve folds instead of
// sixteen; accumulators 0-2 hold the first half of the query tiles.
constexpr uint32_t kFlagMaskTri = (1u << 7) | (1u << 15) | (1u << 22) | (1u << 23);
constexpr uint32_t kTriMinThreshold = 28;  // below it, distant pairs borrow too often
constexpr int kScale128 = 127 + 7;         // 2^7
constexpr int kScale32k = 127 + 15;        // 2^15

__device__ __forceinline__ v4f flags_c0_tri(float bound) {
  const int b = (int)bound;
  const int c = 8388608 + (128 - b) + 256 * (129 - b / 2) + 65536 * (64 - b / 2);  // below 2^24: exact
  const float f = (float)c;
  return v4f{f, f, f, f};
}

// Accumulator m (0..5) of a row tile: its first query tile and its size.
__device__ constexpr int tri_first(int m) { return m < 3 ? 3 * m : 8 + 3 * (m - 3); }
__device__ constexpr int tri_size(int m) { return (m == 2 || m == 5) ? 2 : 3; }
// Flag chain of accumulator P: two per half of the query tiles.
__device__ constexpr int tri_chain(int p) { return 2 * ((p % 6) >= 3 ? 1 : 0) + (p & 1); }

// Accumulator P (row tile P / 6, accumulator P % 6): its first product issues
// at step P into result register P % 4, its second at step P + 1 and its
// third at step P + 2, and its bits are folded at step P + 4, before the
// register takes accumulator P + 4.
template <int kTiles, int S>
__device__ __forceinline__ void group_flags_tri_step(const Expanded (&qa)[kSharedQt], const Expanded (&rb)[kTiles],
                                                     const v4f& c0, uint32_t (&acc)[kFlagChains], v4f& r0, v4f& r1,
                                                     v4f& r2, v4f& r3) {
  constexpr int kN = 6 * kTiles;  // accumulators
  v4f& cur = (S % 4 == 0) ? r0 : (S % 4 == 1) ? r1 : (S % 4 == 2) ? r2 : r3;
  v4f& p1 = (S % 4 == 1) ? r0 : (S % 4 == 2) ? r1 : (S % 4 == 3) ? r2 : r3;
  v4f& p2 = (S % 4 == 2) ? r0 : (S % 4 == 3) ? r1 : (S % 4 == 0) ? r2 : r3;
  if constexpr (S >= 4) fold_flags(cur, acc[tri_chain(S - 4)]);
  if constexpr (S < kN) cur = mfma_acc<kScale1>(qa[tri_first(S % 6)], rb[S / 6], c0);
  if constexpr (S >= 1 && S - 1 < kN)
    p1 = mfma_acc<kScale128>(qa[tri_first((S - 1) % 6) + 1], rb[(S - 1) / 6], p1);
  if constexpr (S >= 2 && S - 2 < kN) {
    if constexpr (tri_size((S - 2) % 6) == 3)
      p2 = mfma_acc<kScale32k>(qa[tri_first((S - 2) % 6) + 2], rb[(S - 2) / 6], p2);
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (S + 1 < kN + 4) group_flags_tri_step<kTiles, S + 1>(qa, rb, c0, acc, r0, r1, r2, r3);
}

template <int kTiles>
__device__ __forceinline__ void group_flags_tri(const Expanded (&qa)[kSharedQt], const Expanded (&rb)[kTiles], const v4f& c0,
                                                uint32_t (&acc)[kFlagChains]) {
  v4f r0, r1, r2, r3;
  group_flags_tri_step<kTiles, 0>(qa, rb, c0, acc, r0, r1, r2, r3);
}

// Where a wave's row words come from.  Lane (rn, kq) needs word kq of row
// 16 * tile + rn.  Raw rows: db[r * 8 + kq] -- 16 of every 32 bytes,
// scattered over 4 cache lines per tile.  Prefix plane (the first 16 bytes of
// every row, packed): plane[r * 4 + kq], so a tile is 256 contiguous bytes and
// a launch reads half the bytes.
template <bool kPlane>
struct RowSource {
  const uint32_t* __restrict__ p;
  __device__ __forceinline__ RowSource(const uint32_t* db, const uint32_t* plane, uint64_t row0, int lane)
      : p(kPlane ? plane + (row0 + (lane & 15)) * 4 + (lane >> 4) : db + (row0 + (lane & 15)) * 8 + (lane >> 4)) {}
  __device__ __forceinline__ uint32_t operator()(uint32_t tile) const {
    return p[(size_t)tile * (kPlane ? 64 : 128)];
  }
};

// Shared-rows work item, for batches of kMfmaWaves or more query groups: the
// block's waves stream the same kSharedTiles 16-row tiles (rows
// sub * kSharedRows ...), wave w against query group kMfmaWaves * sgroup + w.
// For every group of kGroupTiles tiles, wave w loads and expands tiles
// kGroupTiles * g + kMfmaWaves * s + w (s < kStagePerWave) once, into LDS
// (double-buffered, one barrier per group), and every wave reads the group's
// expanded tiles with one 16-byte LDS read each.  Each wave would otherwise
// load and expand every tile itself; shared, a product costs a quarter of the
// loads and expansions, which is what more query tiles per wave would buy
// without their registers.  A wave whose group lies past the last query still
// loads and expands its tiles for the others.  Candidates become records, one
// per wave and item, for the recheck kernel.
constexpr int kSharedTiles = 64;
constexpr uint64_t kSharedRows = (uint64_t)kSharedTiles * 16;
constexpr int kStagePerWave = 1;                          // tiles a wave stages per group
constexpr int kGroupTiles = kMfmaWaves * kStagePerWave;  // tiles per barrier and per vote
static_assert(kSharedTiles % kGroupTiles == 0 && kSharedTiles / kGroupTiles <= 32,
              "one bit of a 32-bit record mask per group of tiles");
// A record's mask holds query tiles 0-7's groups in its low bits and tiles
// 8-15's from bit kHalfShift.
constexpr int kHalfShift = 16;
static_assert(kSharedTiles / kGroupTiles <= kHalfShift, "two halves in a record mask");
static_assert((uint64_t)kMfmaWaves * kMfmaTilesPerWave * 16 % kSharedRows == 0, "sub-chunks of a chunk");
constexpr uint64_t kSubsPerChunk = (uint64_t)kMfmaWaves * kMfmaTilesPerWave * 16 / kSharedRows;

struct SharedRowsLds {
  u32x4 ex[2][kGroupTiles][64];  // two groups of expanded tiles, lane-major
};

// The shared-rows stream of one sub-chunk.  kFull (all kSharedTiles tiles
// exist, every sub-chunk but a database's last) has a loop with fixed bounds
// and no branch: a branch in the loop makes the compiler wait for every load
// in flight at each group.
template <bool kFull, bool kPlane, bool kTri>
__device__ __forceinline__ void stream_shared(const Expanded (&qa)[kSharedQt], SharedRowsLds& S, const RowSource<kPlane>& src,
                                              const uint32_t* __restrict__ db, uint64_t row0, uint64_t n_rows,
                                              uint32_t qbase, int wave, int lane, float bound,
                                              uint4* __restrict__ recs, uint32_t* __restrict__ rec_count,
                                              uint32_t rec_cap, uint64_t rec_sub_base) {
  const int rn = lane & 15, kq = lane >> 4;
  const uint64_t left = n_rows - row0;
  const uint32_t tiles = kFull ? (uint32_t)kSharedTiles : (uint32_t)((left + 15) / 16);
  const uint32_t ngroups =
      kFull ? (uint32_t)(kSharedTiles / kGroupTiles) : (tiles + kGroupTiles - 1) / kGroupTiles;
  // This wave's word of its s-th tile of group g, loaded unconditionally: the
  // tile is clamped into the sub-chunk (the plane is padded to whole tiles)
  // and a raw row past the end is clamped to the last row; stage() zeroes
  // both.
  auto word = [&](uint32_t g, int s) -> uint32_t {
    const uint32_t tt = min(kGroupTiles * g + kMfmaWaves * s + (uint32_t)wave, tiles - 1);
    if (kPlane || kFull) return src(tt);
    const uint64_t r = min((uint64_t)tt * 16 + rn, left - 1);
    return db[(row0 + r) * 8 + kq];
  };
  // staging in two halves: the expansion, then the store, with the group's
  // products between them
  auto store = [&](uint32_t g, int s, const Expanded& e, int buf) {
    const uint32_t tt = kGroupTiles * g + kMfmaWaves * s + (uint32_t)wave;
    // zero operands (not the expansion of a zero word, whose every code is +1),
    // selected without a branch
    const bool have = kFull ? tt < tiles : (tt < tiles && (uint64_t)tt * 16 + rn < left);
    const uint32_t keep = have ? 0xffffffffu : 0u;
    u32x4 v;
    v.x = e.d[0] & keep;
    v.y = e.d[1] & keep;
    v.z = e.d[2] & keep;
    v.w = e.d[3] & keep;
    S.ex[buf][kMfmaWaves * s + wave][lane] = v;
  };
  auto stage = [&](uint32_t g, int s, uint32_t w, int buf) {
    Expanded e;
    expand_word(w, e);
    store(g, s, e, buf);
  };
  // ring[a] holds this wave's words of group g0 + a + 1, loaded kRing groups
  // ahead; with the inner loop unrolled the slots are fixed registers
  constexpr int kRing = 4;
  static_assert((kSharedTiles / kGroupTiles) % kRing == 0, "whole rounds of the ring");
  uint32_t ring[kRing][kStagePerWave];
#pragma unroll
  for (int a = 0; a < kRing; a++)
#pragma unroll
    for (int st = 0; st < kStagePerWave; st++) ring[a][st] = word(a + 1 < (int)ngroups ? a + 1 : ngroups - 1, st);
#pragma unroll
  for (int st = 0; st < kStagePerWave; st++) stage(0, st, word(0, st), 0);
  __syncthreads();
  uint32_t acc[kFlagChains];
#pragma unroll
  for (int m = 0; m < kFlagChains; m++) acc[m] = 0u;
  const v4f c0 = kTri ? flags_c0_tri(bound) : flags_c0(bound);
  uint64_t pending = 0;  // groups of tiles whose products reached the bound
#pragma unroll 1
  for (uint32_t g0 = 0; g0 < ngroups; g0 += kRing) {
#pragma unroll
    for (int a = 0; a < kRing; a++) {
      const uint32_t g = g0 + a;
      if (!kFull && g >= ngroups) break;  // the same for the whole block
      // The group's expanded tiles, read together so their latencies
      // overlap, and before the staging below: LDS operations complete in
      // order, so the products then wait for these reads only, not for the
      // write of the next group.
      u32x4 vt[kGroupTiles];
#pragma unroll
      for (int j = 0; j < kGroupTiles; j++) vt[j] = S.ex[g & 1][j][lane];
      __builtin_amdgcn_sched_barrier(0);
      // The next group is expanded now and its store follows the products, so
      // neither waits for the other.  The buffer written
      // here was last read before the previous barrier; after the last group
      // this stages rows nobody reads.
      Expanded next[kStagePerWave];
#pragma unroll
      for (int st = 0; st < kStagePerWave; st++) expand_word(ring[a][st], next[st]);
      __builtin_amdgcn_sched_barrier(0);
      Expanded rb[kGroupTiles];
#pragma unroll
      for (int j = 0; j < kGroupTiles; j++) {
        rb[j].d[0] = vt[j].x;
        rb[j].d[1] = vt[j].y;
        rb[j].d[2] = vt[j].z;
        rb[j].d[3] = vt[j].w;
      }
      if constexpr (kTri)
        group_flags_tri<kGroupTiles>(qa, rb, c0, acc);
      else
        group_flags<kGroupTiles>(qa, rb, c0, acc);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int st = 0; st < kStagePerWave; st++) {
        if (kFull || g + 1 < ngroups) store(g + 1, st, next[st], (g + 1) & 1);
        ring[a][st] = word(g + 1 + kRing < ngroups ? g + 1 + kRing : ngroups - 1, st);
      }
      // the vote is a wave-uniform mask, so the pending bits stay in scalar
      // registers; one vote per half of the query tiles, the second half's bits
      // kHalfShift above the first's
      constexpr uint32_t kMask = kTri ? kFlagMaskTri : kFlagMask;
      const uint64_t lo = __ballot(((acc[0] | acc[1]) & kMask) != 0);
      const uint64_t hi = __ballot(((acc[2] | acc[3]) & kMask) != 0);
      pending |= (uint64_t)(lo != 0) << g | (uint64_t)(hi != 0) << (g + kHalfShift);
#pragma unroll
      for (int m = 0; m < kFlagChains; m++) acc[m] = 0u;
      __syncthreads();
    }
  }
  // The rare path is a record for the resolve kernel (sub-chunk number, plus
  // rec_sub_base for a shard of a set; this wave's first query; the pending
  // groups): checking pairs here, even in code that never runs, slows the
  // loop by a tenth.
  if (pending && lane == 0) {
    const uint32_t slot = atomicAdd(rec_count, 1u);
    const uint64_t sub = rec_sub_base + row0 / kSharedRows;
    if (slot < rec_cap) recs[slot] = make_uint4((uint32_t)sub, (uint32_t)(sub >> 32), qbase, (uint32_t)pending);
  }
}

template <bool kPlane, bool kTri>
__device__ __forceinline__ void mfma_item_shared(SharedRowsLds& S,
                                                 const uint32_t* __restrict__ db, const uint32_t* __restrict__ plane,
                                                 uint64_t n_rows, uint64_t sub, uint32_t sgroup,
                                                 const uint32_t* __restrict__ queries, uint32_t n_queries,
                                                 uint32_t threshold, uint4* __restrict__ recs,
                                                 uint32_t* __restrict__ rec_count, uint32_t rec_cap,
                                                 uint64_t rec_sub_base) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: the tests on it are scalar
  const int rn = lane & 15, kq = lane >> 4;
  const float bound = (float)(128 - 2 * (int)threshold);
  const uint64_t row0 = sub * kSharedRows;
  if (row0 >= n_rows) return;  // the same for every wave of the block

  // query operands; a wave whose group lies past the last query gets zero
  // operands (its products never reach the bound) and still stages its tiles
  const uint32_t qbase = (sgroup * kMfmaWaves + wave) * (uint32_t)(kSharedQt * 16);
  uint32_t qw[kSharedQt];
#pragma unroll
  for (int t = 0; t < kSharedQt; t++) {
    const uint32_t qi = qbase + 16 * t + rn;
    qw[t] = queries[(size_t)(qi < n_queries ? qi : n_queries - 1) * 8 + kq];
  }
  Expanded qa[kSharedQt];
#pragma unroll
  for (int t = 0; t < kSharedQt; t++) {
    expand_word(qw[t], qa[t]);
    if (qbase + 16 * t + rn >= n_queries) qa[t].d[0] = qa[t].d[1] = qa[t].d[2] = qa[t].d[3] = 0;
  }

  const RowSource<kPlane> src(db, plane, row0, lane);
  if (row0 + kSharedRows <= n_rows)
    stream_shared<true, kPlane, kTri>(qa, S, src, db, row0, n_rows, qbase, wave, lane, bound, recs,
                                          rec_count, rec_cap, rec_sub_base);
  else
    stream_shared<false, kPlane, kTri>(qa, S, src, db, row0, n_rows, qbase, wave, lane, bound, recs,
                                           rec_count, rec_cap, rec_sub_base);
}

// Work item -> (row chunk, query group).  Consecutive workgroups are dealt
// round-robin to the 8 XCDs, each with its own L2; items are numbered so that
// all query groups of a row chunk run on the same XCD (row chunk = xcd +
// 8 * (slot / groups)) and read its rows from that XCD's L2 after the first
// one brought them in from HBM.
__device__ __forceinline__ void item_coords(uint64_t item, uint32_t groups, uint64_t& chunk, uint32_t& group) {
  const uint64_t xcd = item & 7, slot = item >> 3;
  chunk = xcd + 8 * (slot / groups);
  group = (uint32_t)(slot % groups);
}

// The shared-rows layout over one database, one block per work item:
// 1024-row sub-chunks x groups of kMfmaWaves query groups of sixteen tiles,
// whose candidates become records for pdq_match_resolve_kernel.  Block 0 first
// stores zero to clear_rec and clear_hits where they are given: the record
// count of the stream's next call, and this call's hit counter (this kernel
// appends no hits).
template <bool kPlane, bool kTri>
__global__ void __launch_bounds__(64 * kMfmaWaves) __attribute__((amdgpu_waves_per_eu(3))) pdq_match_mfma_kernel(
    const uint32_t* __restrict__ db, const uint32_t* __restrict__ plane, uint64_t n_rows,
    const uint32_t* __restrict__ queries, uint32_t n_queries, uint32_t threshold, uint32_t sgroups,
    uint4* __restrict__ recs, uint32_t* __restrict__ rec_count, uint32_t rec_cap, uint32_t* __restrict__ clear_rec,
    unsigned long long* __restrict__ clear_hits) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (clear_rec) *clear_rec = 0u;
    if (clear_hits) *clear_hits = 0ull;
  }
  uint64_t sub;
  uint32_t sgroup;
  item_coords(blockIdx.x, sgroups, sub, sgroup);
  __shared__ SharedRowsLds S;
  mfma_item_shared<kPlane, kTri>(S, db, plane, n_rows, sub, sgroup, queries, n_queries, threshold, recs,
                                            rec_count, rec_cap, 0);
}

// ---------------------------------------------------------------------------
// The even layout: every wave streams an even share of the rows against its
// own query group, and checks its candidates itself.
//
// Bounded by the matrix cores (16 cycles a product) and, below eight query
// tiles, by the vector instructions around them (some 45 per 64 rows and wave
// besides the folds) and the rows' bytes.  All waves are resident at once with
// equal parts, so no last round of blocks runs nearly empty, each wave loads
// its queries once, and a small database still spreads over the chip; four
// tiles of rows come with one 16-byte load per lane and are transposed in
// registers.  Fixed parts of 1024 rows per wave, a word per lane and tile,
// took (us, over the plane, before and after): 10^7 rows x 32 / 128 / 200 / 384
// queries 49 / 66 / 114 / 164 -> 32 / 61 / 90 / 145; 10^6 x 48 / 200 15 / 25 ->
// 10 / 20; 10^5 x 200 / 1000 29 / 29 -> 10 / 18; raw rows 10^7 x 32 / 200
// 89 / 183 -> 53 / 99.
// ---------------------------------------------------------------------------
constexpr int kEvenRows = 64;        // rows per group: four 16-row tiles, one load per lane
constexpr uint32_t kEvenGroups = 64;  // most groups per wave: one pending bit each
// Groups a wave loads ahead.  A group's products take 64 QT matrix-core
// cycles per wave, so two cover the latency where QT leaves no registers for
// more.
constexpr int even_ahead(int qt) { return qt >= 14 ? 2 : 4; }
constexpr uint32_t kEvenRound = 4;  // part sizes in groups: whole rounds of either depth

// Lane l holds the four prefix words of row l of the group; afterwards
// register j of lane (rn, kq) is word kq of row 16 j + rn, tile j's operand: a
// transpose of a 4 x 4 matrix of 16-lane rows in two steps of swaps.
__device__ __forceinline__ void transpose_rows(uint32_t (&w)[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  w[0] = c[0];
  w[1] = c[1];
  w[2] = d[0];
  w[3] = d[1];
}

// Accumulators of at most three (kTri) or two products over QT query tiles.
template <int QT, bool kTri>
struct EvenShape {
  static constexpr int kPer = kTri ? 3 : 2;
  static constexpr int kAccs = (QT + kPer - 1) / kPer;
};

// Step S issues the first product of accumulator S of the group (tile S /
// kAccs), the second of S - 1 and the third of S - 2, and folds S - 4, before
// its register takes accumulator S.
template <int QT, bool kTri, int S>
__device__ __forceinline__ void even_step(const Expanded (&qa)[QT], const Expanded (&rb)[4], const v4f& c0,
                                          uint32_t (&acc)[2], v4f& r0, v4f& r1, v4f& r2, v4f& r3) {
  using E = EvenShape<QT, kTri>;
  constexpr int kN = 4 * E::kAccs;
  v4f& cur = (S % 4 == 0) ? r0 : (S % 4 == 1) ? r1 : (S % 4 == 2) ? r2 : r3;
  v4f& p1 = (S % 4 == 1) ? r0 : (S % 4 == 2) ? r1 : (S % 4 == 3) ? r2 : r3;
  v4f& p2 = (S % 4 == 2) ? r0 : (S % 4 == 3) ? r1 : (S % 4 == 0) ? r2 : r3;
  if constexpr (S >= 4) fold_flags(cur, acc[S % 2]);
  if constexpr (S < kN) cur = mfma_acc<kScale1>(qa[E::kPer * (S % E::kAccs)], rb[S / E::kAccs], c0);
  if constexpr (S >= 1 && S - 1 < kN) {
    constexpr int t = E::kPer * ((S - 1) % E::kAccs) + 1;
    if constexpr (t < QT) p1 = mfma_acc<kTri ? kScale128 : kScale512>(qa[t], rb[(S - 1) / E::kAccs], p1);
  }
  if constexpr (kTri && S >= 2 && S - 2 < kN) {
    constexpr int t = E::kPer * ((S - 2) % E::kAccs) + 2;
    if constexpr (t < QT) p2 = mfma_acc<kScale32k>(qa[t], rb[(S - 2) / E::kAccs], p2);
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (S + 1 < kN + 4) even_step<QT, kTri, S + 1>(qa, rb, c0, acc, r0, r1, r2, r3);
}

// A 64-row group of a database.
struct RowGroup {
  const uint4 *db, *plane;
  uint64_t n_rows, index_base;
  uint64_t row;  // its first
};

// Rows `row`, row + step, ... of a database, the prefix plane's 16 bytes or the
// raw row's first: lane's row of the group k steps on.  Rows past the end repeat
// the last one; their pairs are never reported.
template <bool kPlane>
struct GroupRows {
  const uint4* base;  // uniform, as the rest
  uint32_t step, left;
  __device__ __forceinline__ GroupRows(const RowGroup& g, uint32_t stride)
      : base(kPlane ? g.plane + g.row : g.db + 2 * g.row),
        step(stride * kEvenRows),
        left((uint32_t)min(g.n_rows - g.row, (uint64_t)0x7fffffffu)) {}
  __device__ __forceinline__ uint4 load(uint32_t k, int lane) const {
    const uint32_t r = min(k * step + (uint32_t)lane, left - 1);
    return base[kPlane ? r : 2 * r];
  }
};

// Row groups of one database: group k is `first` + k `stride`.
struct DbGroups {
  const uint4 *db, *plane;
  uint64_t n_rows, index_base;
  uint32_t first, stride;
  __device__ __forceinline__ RowGroup at(uint32_t k) const {
    return RowGroup{db, plane, n_rows, index_base, (uint64_t)(first + k * stride) * kEvenRows};
  }
};

// Exact check of the pairs of one 64-row group that reach the bound.
template <int QT, bool kPlane, uint32_t kList>
__device__ __forceinline__ void even_check(HitList<kList>& H, const Expanded (&qa)[QT], const RowGroup& group,
                                           uint32_t qbase, const uint32_t* __restrict__ queries, uint32_t n_queries,
                                           uint32_t threshold, MatchHit* __restrict__ hits, uint64_t capacity,
                                           unsigned long long* __restrict__ counter) {
  const int lane = threadIdx.x & 63;
  const int rn = lane & 15, kq = lane >> 4;
  const float bound = (float)(128 - 2 * (int)threshold);
  const int ibound = __float_as_int(bound);
  const uint4 v = GroupRows<kPlane>(group, 0).load(0, lane);
  uint32_t w[4] = {v.x, v.y, v.z, v.w};
  transpose_rows(w);
#pragma unroll 1
  for (int j = 0; j < 4; j++) {
    Expanded e;
    expand_word(w[0], e);
    w[0] = w[1];  // (a rolled loop cannot index registers)
    w[1] = w[2];
    w[2] = w[3];
    uint32_t tmask = 0;
#pragma unroll
    for (int t = 0; t < QT; t++) {
      const v4f c = mfma_prefix(qa[t], e);
      const int m = max(max(__float_as_int(c.x), __float_as_int(c.y)), max(__float_as_int(c.z), __float_as_int(c.w)));
      tmask |= (wave_any(m >= ibound) ? 1u : 0u) << t;
    }
    while (tmask) {
      const int t = __builtin_ctz(tmask);
      tmask &= tmask - 1;
      Expanded a = qa[0];  // qa[t], selected
#pragma unroll
      for (int k = 1; k < QT; k++)
        if (t == k) a = qa[k];
      stage_candidates(mfma_prefix(a, e), t, group.row + 16 * j, qbase, rn, kq, bound, queries,
                       reinterpret_cast<const uint32_t*>(group.db), n_queries, group.n_rows, threshold, H, hits,
                       capacity, counter, group.index_base);
    }
  }
}

// How the rows' groups are cut: the waves of one XCD, all resident at once,
// hold as many parts as they have room for per query group; more rows take
// several equal rounds.  Parts are whole rounds of loads.
//
// 40 neighbouring parts take the groups of their stretch in turn: where many
// rows in a row match (a film's frames), their checks, some 4 us a group, spread
// over as many waves.  With consecutive groups in each part one wave did up to
// 64 of them after the others had ended (10^7 rows over the plane with eight
// runs of 5000 near rows, consecutive / in turn, us: 12 queries 188 / 33, 64
// 209 / 40, 512 384 / 182; without runs 31 / 30, 43 / 40, 184 / 180).  Turns of
// 64 make most stretches a power of two long, and all waves then read the same
// channels (8.4x10^6 rows x 16 queries 28 -> 39 us; 24, 40 and 56 28); turns
// over all parts spread a wave's rows over as many pages (10^6 raw rows x 200
// queries 14.6 -> 17.9).
constexpr uint32_t kEvenTurn = 40;
struct EvenParts {
  uint32_t groups;   // row groups per part, at most
  uint32_t per_xcd;  // parts per XCD
};
__host__ __device__ inline EvenParts even_parts(uint32_t row_groups, uint32_t query_groups, uint32_t waves_per_xcd) {
  const uint32_t at_once = waves_per_xcd / query_groups;
  const uint64_t round = 8ull * (at_once ? at_once : 1);  // parts resident at once
  const uint64_t rounds = ((uint64_t)row_groups + round * kEvenGroups - 1) / (round * kEvenGroups);
  const uint64_t all = round * (rounds ? rounds : 1);
  uint32_t n = (uint32_t)(((uint64_t)row_groups + all - 1) / all);
  n = (n + kEvenRound - 1) / kEvenRound * kEvenRound;
  n = n == 0 ? kEvenRound : n > kEvenGroups ? kEvenGroups : n;
  return EvenParts{n, (uint32_t)((((uint64_t)row_groups + n - 1) / n + 7) / 8)};
}
// The groups of one part: count of them, first, first + stride, ...
struct PartGroups {
  uint32_t first, stride, count;
};
__device__ __forceinline__ PartGroups part_row_groups(uint32_t part, const EvenParts& parts, uint32_t row_groups) {
  const uint32_t turn = part / kEvenTurn * kEvenTurn;  // the stretch's first part
  const uint32_t stride = min(kEvenTurn, parts.per_xcd * 8 - turn);
  const uint64_t begin = (uint64_t)turn * parts.groups;
  const uint64_t first = begin + (part - turn), end = min(begin + (uint64_t)stride * parts.groups, (uint64_t)row_groups);
  return PartGroups{(uint32_t)first, stride, first < end ? (uint32_t)((end - first + stride - 1) / stride) : 0u};
}

// `ngroups` (1 .. kEvenGroups) row groups against query group qbase.
template <int QT, bool kPlane, bool kTri, uint32_t kList>
__device__ __forceinline__ void even_part(HitList<kList>& H, const DbGroups& groups, uint32_t ngroups,
                                          const uint32_t* __restrict__ queries, uint32_t n_queries, uint32_t qbase,
                                          uint32_t threshold, MatchHit* __restrict__ hits, uint64_t capacity,
                                          unsigned long long* __restrict__ counter) {
  constexpr int kAhead = even_ahead(QT);
  const int lane = threadIdx.x & 63;
  const int rn = lane & 15, kq = lane >> 4;
  const GroupRows<kPlane> rows(groups.at(0), groups.stride);
  auto load = [&](uint32_t k) { return rows.load(min(k, ngroups - 1), lane); };
  uint4 ring[kAhead];
#pragma unroll
  for (int a = 0; a < kAhead; a++) ring[a] = load(a);

  uint32_t qw[QT];
#pragma unroll
  for (int t = 0; t < QT; t++) {
    const uint32_t qi = qbase + 16 * t + rn;
    qw[t] = queries[(size_t)(qi < n_queries ? qi : n_queries - 1) * 8 + kq];
  }
  Expanded qa[QT];
#pragma unroll
  for (int t = 0; t < QT; t++) {
    expand_word(qw[t], qa[t]);
    if (qbase + 16 * t + rn >= n_queries)
      qa[t].d[0] = qa[t].d[1] = qa[t].d[2] = qa[t].d[3] = 0;  // zero rows never reach the bound
  }
  const float bound = (float)(128 - 2 * (int)threshold);
  const v4f c0 = kTri ? flags_c0_tri(bound) : flags_c0(bound);
  uint64_t pending = 0;
#pragma unroll 1
  for (uint32_t g0 = 0; g0 < ngroups; g0 += kAhead) {
#pragma unroll
    for (int a = 0; a < kAhead; a++) {
      uint32_t w[4] = {ring[a].x, ring[a].y, ring[a].z, ring[a].w};
      transpose_rows(w);
      Expanded rb[4];
#pragma unroll
      for (int j = 0; j < 4; j++) expand_word(w[j], rb[j]);
      ring[a] = load(g0 + a + kAhead);
      uint32_t acc[2] = {0u, 0u};
      v4f r0, r1, r2, r3;
      even_step<QT, kTri, 0>(qa, rb, c0, acc, r0, r1, r2, r3);
      const uint64_t vote = __ballot(((acc[0] | acc[1]) & (kTri ? kFlagMaskTri : kFlagMask)) != 0);
      pending |= (uint64_t)(vote != 0) << (g0 + a);
    }
  }
  if (ngroups < 64) pending &= (1ull << ngroups) - 1;  // the last round's groups past the part
  while (pending) {
    const uint32_t k = (uint32_t)__builtin_ctzll(pending);
    pending &= pending - 1;
    even_check<QT, kPlane>(H, qa, groups.at(k), qbase, queries, n_queries, threshold, hits, capacity, counter);
  }
}

// One part per wave.  Part part_x * 8 + xcd: the waves that match one part
// against the query groups are neighbours on one XCD and share its rows in the
// caches.
template <int QT, bool kPlane, bool kTri>
__global__ void __launch_bounds__(64 * kMfmaWaves) __attribute__((amdgpu_waves_per_eu(4))) pdq_match_even_kernel(
    const uint4* __restrict__ db, const uint4* __restrict__ plane, uint64_t n_rows, uint32_t row_groups,
    const uint32_t* __restrict__ queries, uint32_t n_queries, uint32_t threshold, MatchHit* __restrict__ hits,
    uint64_t capacity, unsigned long long* __restrict__ counter, uint64_t index_base, uint32_t groups,
    EvenParts parts) {
  __shared__ HitList<kEvenStage> H;
  hits_init(H);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t id = (blockIdx.x >> 3) * kMfmaWaves + wave;
  const uint32_t part_x = id / groups;
  if (part_x < parts.per_xcd) {
    const PartGroups rows = part_row_groups(part_x * 8 + (blockIdx.x & 7), parts, row_groups);
    if (rows.count)
      even_part<QT, kPlane, kTri>(H, DbGroups{db, plane, n_rows, index_base, rows.first, rows.stride}, rows.count,
                                  queries, n_queries, (id - part_x * groups) * (uint32_t)(QT * 16), threshold, hits,
                                  capacity, counter);
  }
  hits_flush(H, hits, capacity, counter);
}

// ---------------------------------------------------------------------------
// The held-rows layout: few rows against many queries.
//
// The even layout holds query tiles in registers and streams rows past them;
// with few rows a part is a handful of loads, and a wave's time the latency of
// loading and expanding its 256 queries first.  Here a block expands up to 64
// query tiles into LDS once, together, and each of its waves holds 192 rows (or
// 128, two products per accumulator) and runs all the tiles past them: 12 products for one LDS read, no expansion in the loop.
// The prefix products, their flags and the exact check are the even layout's.
// The matrix cores bound a wave's loop (24 products beside about 20 vector
// instructions per pair of tiles); the launch, 9.3 us as measured, bounds the
// calls with the fewest rows.
//
// Kernel times with the reset, even layout / here, us:
//   rows       256         512        1000        2048 queries
//   10^4    19.1 /  8.7  20.7 /  8.7  23.9 /  9.6  29.0 / 13.4
//   10^5    11.4 /  9.2  12.5 / 10.8  17.6 / 13.1  26.3 / 19.9
//   3x10^5  14.9 / 12.0  17.8 / 15.6  24.0 / 22.3  43.5 / 37.1
//   7x10^5  17.4 / 15.7  24.0 / 22.4  38.1 / 35.4  69.4 / 63.3
// ---------------------------------------------------------------------------
constexpr int kHeldWaves = 8;          // waves per block, sharing the block's query codes
constexpr uint32_t kHeldTiles = 64;    // most query tiles per block (64 KiB of codes)

// Rows per wave and group: four accumulators of kPer products, a 16-row tile
// each.
template <int kPer>
struct Held {
  static constexpr int kTiles = 4 * kPer;
  static constexpr int kLoads = kTiles / 4;  // 16 bytes per lane: 64 rows each
  static constexpr uint32_t kRows = 16 * kTiles;
};

__device__ __forceinline__ Expanded codes_from(const u32x4& v) {
  Expanded e;
  e.d[0] = v.x;
  e.d[1] = v.y;
  e.d[2] = v.z;
  e.d[3] = v.w;
  return e;
}

template <int kPer>
constexpr int held_scale(int p) {
  return p == 0 ? kScale1 : kPer == 2 ? kScale512 : p == 1 ? kScale128 : kScale32k;
}

// Query tile q against the held rows: accumulator k takes its first product
// while k - 1 takes its second and k - 2 its third (of this query tile or, for
// the last ones, of the one before), so no product waits for the one before
// it; the result of the tile before is folded just before.  Once the tile
// before has issued its last product, `refill` loads the next tile's codes
// into its place.
template <int kPer, int K = 0, class Refill>
__device__ __forceinline__ void held_tile(const Expanded& q, Expanded& before, Refill&& refill,
                                          const Expanded (&rows)[4 * kPer], const v4f& c0, uint32_t (&acc)[2],
                                          v4f (&r)[4]) {
  fold_flags(r[K], acc[K % 2]);
  r[K] = mfma_acc<held_scale<kPer>(0)>(q, rows[kPer * K], c0);
  if constexpr (kPer >= 2) {
    constexpr int k = (K + 3) % 4;
    r[k] = mfma_acc<held_scale<kPer>(1)>(K >= 1 ? q : before, rows[kPer * k + 1], r[k]);
  }
  if constexpr (kPer >= 3) {
    constexpr int k = (K + 2) % 4;
    r[k] = mfma_acc<held_scale<kPer>(2)>(K >= 2 ? q : before, rows[kPer * k + 2], r[k]);
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (K == 1) refill(before);
  if constexpr (K + 1 < 4) held_tile<kPer, K + 1>(q, before, static_cast<Refill&&>(refill), rows, c0, acc, r);
}

// What is left after the last query tile.
template <int kPer>
__device__ __forceinline__ void held_last(const Expanded (&rows)[4 * kPer], const Expanded& q, uint32_t (&acc)[2],
                                          v4f (&r)[4]) {
  if constexpr (kPer >= 2) r[3] = mfma_acc<held_scale<kPer>(1)>(q, rows[kPer * 3 + 1], r[3]);
  if constexpr (kPer >= 3) {
    r[2] = mfma_acc<held_scale<kPer>(2)>(q, rows[kPer * 2 + 2], r[2]);
    r[3] = mfma_acc<held_scale<kPer>(2)>(q, rows[kPer * 3 + 2], r[3]);
  }
#pragma unroll
  for (int k = 0; k < 4; k++) fold_flags(r[k], acc[k % 2]);
}

// The block's query codes, a lane's 16 bytes of each tile side by side.
struct HeldLds {
  u32x4 q[kHeldTiles][64];
  HitList<kHeldStage> hits;
};

// Codes of query tiles t0 .. t0 + n - 1 into S.q; padding queries get zero
// codes, whose products never reach the bound.
__device__ __forceinline__ void held_queries(HeldLds& S, const uint32_t* __restrict__ queries, uint32_t n_queries,
                                             uint32_t t0, uint32_t n) {
  for (uint32_t i = threadIdx.x; i < n * 64; i += 64 * kHeldWaves) {
    const uint32_t lane = i & 63, qi = 16 * (t0 + (i >> 6)) + (lane & 15);
    Expanded e;
    expand_word(queries[(size_t)min(qi, n_queries - 1) * 8 + (lane >> 4)], e);
    const uint32_t keep = qi < n_queries ? 0xffffffffu : 0u;
    S.q[i >> 6][lane] = u32x4{e.d[0] & keep, e.d[1] & keep, e.d[2] & keep, e.d[3] & keep};
  }
}

// Query tiles per vote.
constexpr uint32_t kHeldVote = 8;

// Rows row0 .. row0 + left - 1 against the block's n query tiles (t0 the first
// of them among all).
template <int kPer, bool kPlane>
__device__ __forceinline__ void held_rows(HeldLds& S, const uint4* __restrict__ db, const uint4* __restrict__ plane,
                                          uint64_t n_rows, uint64_t row0, uint32_t left,
                                          const uint32_t* __restrict__ queries, uint32_t n_queries, uint32_t t0,
                                          uint32_t n, uint32_t threshold, MatchHit* __restrict__ hits,
                                          uint64_t capacity, unsigned long long* __restrict__ counter,
                                          uint64_t index_base) {
  using H = Held<kPer>;
  const int lane = threadIdx.x & 63;
  const int rn = lane & 15, kq = lane >> 4;
  const uint4* base = kPlane ? plane + row0 : db + 2 * row0;  // uniform
  // rows past the end repeat the last one; their pairs are never reported
  auto load = [&](uint32_t r) -> uint4 {
    r = min(r + (uint32_t)lane, left - 1);
    return base[kPlane ? r : 2 * r];
  };
  uint4 raw[H::kLoads];
#pragma unroll
  for (int l = 0; l < H::kLoads; l++) raw[l] = load(64 * l);
  const float bound = (float)(128 - 2 * (int)threshold);
  const int ibound = __float_as_int(bound);
  const v4f c0 = kPer == 3 ? flags_c0_tri(bound) : flags_c0(bound);
  constexpr uint32_t kMask = kPer == 3 ? kFlagMaskTri : kFlagMask;
  const Expanded zero = {{0u, 0u, 0u, 0u}};
  auto code = [&](uint32_t t) { return codes_from(S.q[t][lane]); };
#pragma unroll 1
  for (uint32_t g = 0; g < left; g += H::kRows) {
    Expanded rows[H::kTiles];
#pragma unroll
    for (int l = 0; l < H::kLoads; l++) {
      uint32_t w[4] = {raw[l].x, raw[l].y, raw[l].z, raw[l].w};
      transpose_rows(w);
#pragma unroll
      for (int j = 0; j < 4; j++) expand_word(w[j], rows[4 * l + j]);
      raw[l] = load(g + H::kRows + 64 * l);
    }
    uint32_t acc[2] = {0u, 0u};
    v4f r[4];
#pragma unroll
    for (int k = 0; k < 4; k++) r[k] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    Expanded x = code(0), y = zero;
    // bit i: a flag among query tiles 8 i - 1 .. 8 i + 6 (a tile's results are
    // folded with the next one); the last bit, what remains
    uint32_t pending = 0, bit = 0;
    auto vote = [&] {
      const uint64_t v = __ballot(((acc[0] | acc[1]) & kMask) != 0);
      pending |= (uint32_t)(v != 0) << bit;
      bit++;
      acc[0] = acc[1] = 0u;
    };
    uint32_t t = 0;
#pragma unroll 1
    for (; t + kHeldVote <= n; t += kHeldVote) {
#pragma unroll 1
      for (uint32_t k = 0; k < kHeldVote; k += 2) {
        held_tile<kPer>(x, y, [&](Expanded& e) { e = code(t + k + 1); }, rows, c0, acc, r);
        held_tile<kPer>(y, x, [&](Expanded& e) { e = code(min(t + k + 2, n - 1)); }, rows, c0, acc, r);
      }
      vote();
    }
#pragma unroll 1
    for (; t + 2 <= n; t += 2) {
      held_tile<kPer>(x, y, [&](Expanded& e) { e = code(t + 1); }, rows, c0, acc, r);
      held_tile<kPer>(y, x, [&](Expanded& e) { e = code(min(t + 2, n - 1)); }, rows, c0, acc, r);
    }
    if (t < n) {
      held_tile<kPer>(x, y, [&](Expanded& e) { e = x; }, rows, c0, acc, r);
      // y holds the last tile's codes, as after a pair
    }
    held_last<kPer>(rows, y, acc, r);
    vote();
    if (pending) {
#pragma unroll 1
      for (uint32_t q = 0; q < n; q++) {
        // the bits that cover tile q: its vote's, or the last one
        const uint32_t b = min((q + 1) / kHeldVote, bit - 1);
        if (!(pending >> b & 1u)) continue;
        const Expanded qe = code(q);
        uint32_t tmask = 0;
#pragma unroll
        for (int j = 0; j < H::kTiles; j++) {
          const v4f c = mfma_prefix(qe, rows[j]);
          const int m = max(max(__float_as_int(c.x), __float_as_int(c.y)),
                            max(__float_as_int(c.z), __float_as_int(c.w)));
          tmask |= (wave_any(m >= ibound) ? 1u : 0u) << j;
        }
        while (tmask) {
          const int j = __builtin_ctz(tmask);
          tmask &= tmask - 1;
          Expanded e = rows[0];  // rows[j], selected (registers cannot be indexed)
#pragma unroll
          for (int k = 1; k < H::kTiles; k++)
            if (j == k) e = rows[k];
          stage_candidates(mfma_prefix(qe, e), (int)q, row0 + g + 16 * j, 16 * t0, rn, kq, bound, queries,
                           reinterpret_cast<const uint32_t*>(db), n_queries, n_rows, threshold, S.hits, hits,
                           capacity, counter, index_base);
        }
      }
    }
  }
}

// How a call is cut: `chunks` groups of at most `tiles` query tiles, each
// block holding one of them; a wave's rows are `groups` row groups.
struct HeldPlan {
  uint32_t chunks, tiles, groups, blocks_per_xcd;  // blocks per XCD and chunk
  uint64_t cost;
};
// The cut that costs least, in cycles of a wave: its products (12 or 8 of 18.1
// cycles and their share of the rest per tile and row group), about two tiles'
// time for loading and expanding the rows of a group, times the blocks that
// share a CU, and the queries' expansion.  kPer = 2 is rated a little higher
// than it measures alone: at equal costs it lost 5 % (7x10^5 rows x 2048 queries
// 63.8 / 67.8 us).  cus: of one XCD; two blocks are resident on each (72 KiB of
// LDS).
template <int kPer>
HeldPlan held_plan(uint64_t n_rows, uint32_t tiles, uint32_t cus) {
  constexpr uint64_t kTile = kPer == 3 ? 224 : 166, kGroup = kPer == 3 ? 464 : 330;
  const uint64_t row_groups = (n_rows + Held<kPer>::kRows - 1) / Held<kPer>::kRows;
  const uint32_t blocks_per_xcd = 2 * cus;
  HeldPlan best{1, 1, 1, 1, ~0ull};
  const uint32_t first = (tiles + kHeldTiles - 1) / kHeldTiles;
  for (uint32_t c = first; c < 2 * first + 16 && c <= tiles; c++) {
    const uint32_t t = (tiles + c - 1) / c;
    const uint32_t at_once = blocks_per_xcd / c ? blocks_per_xcd / c : 1;
    const uint64_t waves = 8ull * kHeldWaves * at_once;  // per chunk
    const uint64_t g = (row_groups + waves - 1) / waves;
    const uint64_t need = (row_groups + g * 8 * kHeldWaves - 1) / (g * 8 * kHeldWaves);  // blocks per XCD
    const uint64_t per_cu = (need * c + cus - 1) / cus;
    const uint64_t cost = g * (t * kTile + kGroup) * per_cu + t * 64;
    if (cost < best.cost) best = HeldPlan{c, t, (uint32_t)g, (uint32_t)need, cost};
  }
  return best;
}

template <int kPer, bool kPlane>
__global__ void __launch_bounds__(64 * kHeldWaves) __attribute__((amdgpu_waves_per_eu(4))) pdq_match_held_kernel(
    const uint4* __restrict__ db, const uint4* __restrict__ plane, uint64_t n_rows,
    const uint32_t* __restrict__ queries, uint32_t n_queries, uint32_t threshold, MatchHit* __restrict__ hits,
    uint64_t capacity, unsigned long long* __restrict__ counter, uint64_t index_base, HeldPlan plan) {
  __shared__ HeldLds S;
  const uint32_t slot = blockIdx.x >> 3;
  const uint32_t chunk = slot % plan.chunks;
  const uint32_t t0 = chunk * plan.tiles, all = (n_queries + 15) / 16;
  if (t0 >= all) return;  // the same for the whole block
  const uint32_t n = min(plan.tiles, all - t0);
  held_queries(S, queries, n_queries, t0, n);
  hits_init(S.hits);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t part = ((uint64_t)(slot / plan.chunks) * kHeldWaves + wave) * 8 + (blockIdx.x & 7);
  const uint64_t rows = (uint64_t)plan.groups * Held<kPer>::kRows;
  const uint64_t row0 = part * rows;
  if (row0 < n_rows)
    held_rows<kPer, kPlane>(S, db, plane, n_rows, row0, (uint32_t)min(n_rows - row0, rows), queries, n_queries, t0, n,
                            threshold, hits, capacity, counter, index_base);
  hits_flush(S.hits, hits, capacity, counter);
}

// The second kernel of the shared-rows layout, in blocks of kResolveWaves
// waves.  Each wave takes records in turn: for every pending group of the
// record's sub-chunk it recomputes the group's products, and for each query
// tile with a pair at the bound checks every such pair with the exact
// 256-bit distance.  The block's hits gather in LDS and take their slots in
// the hit buffer with one atomic.  If the records overflowed their area (more
// than rec_cap: dense hits), all rows are matched again in the even layout
// instead, a part per wave, which checks its own candidates (the first kernel
// appended no hits), so the set stays exact.
constexpr int kResolveWaves = 8;
// Two blocks per CU (16 waves; the kernel fits 128 VGPRs at its at most 8
// query tiles per wave): a
// record's check is a chain of dependent loads, so waves in flight set its
// rate.  Measured against one block per CU: 19 against 22.5 us at the
// bench's sparse hits, 578 against 871 us at 271k hits per batch.
constexpr int kResolveBlocksPerCu = 2;

uint32_t match_resolve_blocks(int cus) { return (uint32_t)std::max(1, cus) * kResolveBlocksPerCu; }

using ResolveLds = HitList<kStageHits>;

// The rerun after an overflow: parts of kEvenGroups groups of rows against
// groups of six query tiles, a wave each (eight leave one block per CU).
constexpr int kRerunQt = 6;
constexpr uint64_t kRerunRows = (uint64_t)kEvenGroups * kEvenRows;
// Row groups of its part `part`.
__device__ __forceinline__ uint32_t rerun_groups(uint64_t n_rows, uint64_t part) {
  return (uint32_t)((min(n_rows - part * kRerunRows, kRerunRows) + kEvenRows - 1) / kEvenRows);
}

// The loads of one record part that do not depend on its products: the
// query words of its tiles and the tile words of its first pending group.  A
// wave issues them for its next part before it checks the current one, so a
// part's check waits only on its own exact-distance loads.
template <int QT>
struct PartLoads {
  uint32_t qw[QT];
  uint32_t w[kGroupTiles];
};

// Tiles of the sub-chunk at row0 (16 rows each; the last sub-chunk's may be
// partial).
__device__ __forceinline__ uint32_t sub_tiles(uint64_t n_rows, uint64_t row0) {
  const uint64_t left = n_rows - row0;
  return left >= kSharedRows ? (uint32_t)kSharedTiles : (uint32_t)((left + 15) / 16);
}

// Group g's tile words (lane rn, word kq of each tile), clamped into the
// sub-chunk's tiles (and, for raw rows, its rows).
template <bool kPlane>
__device__ __forceinline__ void load_group(uint32_t (&w)[kGroupTiles], const uint32_t* __restrict__ db,
                                           const uint32_t* __restrict__ plane, uint64_t n_rows, uint64_t row0,
                                           uint32_t g) {
  const int lane = threadIdx.x & 63;
  const int rn = lane & 15, kq = lane >> 4;
  const uint64_t left = n_rows - row0;
  const uint32_t tiles = sub_tiles(n_rows, row0);
  const RowSource<kPlane> src(db, plane, row0, lane);
#pragma unroll
  for (int j = 0; j < kGroupTiles; j++) {
    const uint32_t tt = min(kGroupTiles * g + (uint32_t)j, tiles - 1);
    if (kPlane) {
      w[j] = src(tt);
    } else {
      const uint64_t rr = min((uint64_t)tt * 16 + rn, left - 1);
      w[j] = db[(row0 + rr) * 8 + kq];
    }
  }
}

template <int QT, bool kPlane>
__device__ __forceinline__ void part_load(PartLoads<QT>& P, const uint32_t* __restrict__ db,
                                          const uint32_t* __restrict__ plane, uint64_t n_rows, uint64_t row0,
                                          uint32_t qbase, uint32_t pending, const uint32_t* __restrict__ queries,
                                          uint32_t n_queries) {
  if (pending == 0) return;  // nothing to check (the same for the whole wave)
  const int lane = threadIdx.x & 63;
  const int rn = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int t = 0; t < QT; t++) {
    const uint32_t qi = qbase + 16 * t + rn;
    P.qw[t] = queries[(size_t)(qi < n_queries ? qi : n_queries - 1) * 8 + kq];
  }
  load_group<kPlane>(P.w, db, plane, n_rows, row0, (uint32_t)__builtin_ctz(pending));
}

// One pending group g of a record part: its tiles' products with the part's
// query tiles qa, and the pairs of the query tiles that reach the bound
// checked exactly.  w holds the group's tile words.
template <int QT>
__device__ __forceinline__ void check_group(ResolveLds& L, const Expanded (&qa)[QT], uint32_t g,
                                            const uint32_t (&words)[kGroupTiles], uint32_t tiles, uint64_t left,
                                            uint64_t row0, uint32_t qbase, float bound,
                                            const uint32_t* __restrict__ queries, const uint32_t* __restrict__ db,
                                            uint32_t n_queries, uint64_t n_rows, uint32_t threshold,
                                            MatchHit* __restrict__ hits, uint64_t capacity,
                                            unsigned long long* __restrict__ counter, uint64_t index_base) {
  const int lane = threadIdx.x & 63;
  const int rn = lane & 15, kq = lane >> 4;
  const int ibound = __float_as_int(bound);
  // tile j's word is w[0] in iteration j (the words move down one place per
  // tile: a rolled loop cannot index registers, and a select by j becomes an
  // indexed copy in scratch memory)
  uint32_t w[kGroupTiles];
#pragma unroll
  for (int k = 0; k < kGroupTiles; k++) w[k] = words[k];
#pragma unroll 1
  for (int j = 0; j < kGroupTiles; j++) {
    const uint32_t tt = kGroupTiles * g + (uint32_t)j;
    if (tt >= tiles) break;  // the same for the whole wave
    const uint32_t wj = w[0];
#pragma unroll
    for (int k = 0; k + 1 < kGroupTiles; k++) w[k] = w[k + 1];
    Expanded eg;
    expand_word(wj, eg);
    if ((uint64_t)tt * 16 + rn >= left) eg.d[0] = eg.d[1] = eg.d[2] = eg.d[3] = 0;
    // which query tiles have a pair at the bound (a wave-uniform mask); the
    // products go in pairs, so that one product's reads overlap the next's
    // matrix-core latency instead of each waiting on the last
    uint32_t tmask = 0;
#pragma unroll
    for (int t = 0; t < QT; t += 2) {
      const v4f c0 = mfma_prefix(qa[t], eg);
      const v4f c1 = t + 1 < QT ? mfma_prefix(qa[t + 1 < QT ? t + 1 : t], eg) : c0;
      const int m0 = max(max(__float_as_int(c0.x), __float_as_int(c0.y)), max(__float_as_int(c0.z), __float_as_int(c0.w)));
      const int m1 = max(max(__float_as_int(c1.x), __float_as_int(c1.y)), max(__float_as_int(c1.z), __float_as_int(c1.w)));
      tmask |= (wave_any(m0 >= ibound) ? 1u : 0u) << t;
      if (t + 1 < QT) tmask |= (wave_any(m1 >= ibound) ? 1u : 0u) << (t + 1);
    }
    // only those tiles' products are recomputed and checked, by one inlined
    // check in a loop over the mask: QT inlined copies keep several hundred
    // registers live, and an out-of-line check saves and restores registers
    // through scratch memory at every call
    while (tmask) {
      const int t = __builtin_ctz(tmask);
      tmask &= tmask - 1;
      Expanded a = qa[0];  // qa[t], selected (registers cannot be indexed)
#pragma unroll
      for (int k = 1; k < QT; k++)
        if (t == k) a = qa[k];
      stage_candidates(mfma_prefix(a, eg), t, row0 + (uint64_t)tt * 16, qbase, rn, kq, bound, queries, db, n_queries,
                       n_rows, threshold, L, hits, capacity, counter, index_base);
    }
  }
}

// One record part, checked by one wave: sub-chunk rows row0 ... of a
// database of n_rows rows (global index index_base + row), queries qbase ...
// (QT x 16), pending groups of kGroupTiles tiles, with P holding its
// part_load.  Groups after the first load their tile words here.  `next` is
// called once P's words are taken (it issues the wave's next loads): a wait
// for P then never covers those newer loads.
template <int QT, bool kPlane, class Next>
__device__ __forceinline__ void resolve_record(ResolveLds& L, const PartLoads<QT>& P,
                                               const uint32_t* __restrict__ db,
                                               const uint32_t* __restrict__ plane, uint64_t n_rows, uint64_t row0,
                                               uint32_t qbase, uint32_t pending, const uint32_t* __restrict__ queries,
                                               uint32_t n_queries, uint32_t threshold, MatchHit* __restrict__ hits,
                                               uint64_t capacity, unsigned long long* __restrict__ counter,
                                               uint64_t index_base, Next&& next) {
  if (pending == 0) {  // a half of a record with no candidates
    next();
    return;
  }
  const int rn = threadIdx.x & 15;
  const float bound = (float)(128 - 2 * (int)threshold);
  const uint64_t left = n_rows - row0;
  const uint32_t tiles = sub_tiles(n_rows, row0);
  Expanded qa[QT];
#pragma unroll
  for (int t = 0; t < QT; t++) {
    expand_word(P.qw[t], qa[t]);
    if (qbase + 16 * t + rn >= n_queries) qa[t].d[0] = qa[t].d[1] = qa[t].d[2] = qa[t].d[3] = 0;
  }
  // The first group's words come with P, outside the loop over the other
  // groups: where the two meet, a wait for the loop's own loads would also
  // wait for the loads `next` has issued.
  uint32_t w0[kGroupTiles];
#pragma unroll
  for (int j = 0; j < kGroupTiles; j++) w0[j] = P.w[j];
  next();
  check_group<QT>(L, qa, (uint32_t)__builtin_ctz(pending), w0, tiles, left, row0, qbase, bound, queries, db,
                  n_queries, n_rows, threshold, hits, capacity, counter, index_base);
  pending &= pending - 1;
  while (pending) {  // rare: a part with candidates in more than one group
    const uint32_t g = (uint32_t)__builtin_ctz(pending);
    pending &= pending - 1;
    uint32_t w[kGroupTiles];
    load_group<kPlane>(w, db, plane, n_rows, row0, g);
    check_group<QT>(L, qa, g, w, tiles, left, row0, qbase, bound, queries, db, n_queries, n_rows, threshold, hits,
                    capacity, counter, index_base);
  }
}

// Query tiles per wave in the recheck.  A record is checked as two halves (query
// tiles 0-7 and 8-15, each with its own pending groups), one after the other by
// the wave that holds the record: sixteen tiles' operands need more registers
// than two blocks per CU leave, and a half without candidates costs nothing.
constexpr int kResolveQt = kSharedQt / 2;
constexpr uint32_t kParts = 2;

// The pending groups of half `part` of a record.
__device__ __forceinline__ uint32_t part_groups(uint32_t mask, uint32_t part) {
  return (mask >> (kHalfShift * part)) & ((1u << kHalfShift) - 1);
}

template <bool kPlane>
__global__ void __launch_bounds__(64 * kResolveWaves) pdq_match_resolve_kernel(
    const uint32_t* __restrict__ db, const uint32_t* __restrict__ plane, uint64_t n_rows,
    const uint32_t* __restrict__ queries, uint32_t n_queries, uint32_t threshold, MatchHit* __restrict__ hits,
    uint64_t capacity, unsigned long long* __restrict__ counter, uint64_t index_base,
    const uint4* __restrict__ recs, const uint32_t* __restrict__ rec_count, uint32_t rec_cap) {
  __shared__ ResolveLds L;
  hits_init(L);
  const int wave = (int)(threadIdx.x >> 6);
  const uint32_t n_recs = *rec_count;
  if (n_recs > rec_cap) {
    const uint32_t groups = (n_queries + kRerunQt * 16 - 1) / (kRerunQt * 16);
    const uint64_t items = (n_rows + kRerunRows - 1) / kRerunRows * groups;
    for (uint64_t item = (uint64_t)blockIdx.x * kResolveWaves + wave; item < items;
         item += (uint64_t)gridDim.x * kResolveWaves) {
      even_part<kRerunQt, kPlane, false>(
          L, DbGroups{reinterpret_cast<const uint4*>(db), reinterpret_cast<const uint4*>(plane), n_rows, index_base,
                      (uint32_t)(item / groups) * kEvenGroups, 1},
          rerun_groups(n_rows, item / groups), queries, n_queries, (uint32_t)(item % groups) * (kRerunQt * 16),
          threshold, hits, capacity, counter);
    }
    hits_flush(L, hits, capacity, counter);
    return;
  }
  // The wave's records are w, w + S, w + 2S, ... (w its number in the
  // grid, S the grid's waves); its item j is part j % kParts of the
  // (j / kParts)-th of them.  Whole records per wave, rather than parts
  // dealt out one by one, bound the parts with candidates that one wave
  // checks (a record's candidates are usually in one part).  The record of
  // the item after next is fetched, and the next item's loads are issued,
  // while this one is checked.
  const uint32_t w0 = blockIdx.x * kResolveWaves + wave;
  const uint32_t S = gridDim.x * kResolveWaves;
  auto rec_of = [&](uint32_t j) { return w0 + (j / kParts) * S; };
  auto fetch = [&](uint32_t j) {
    const uint32_t i = rec_of(j);
    return i < n_recs ? recs[i] : make_uint4(0, 0, 0, 0);
  };
  auto row0_of = [](const uint4& x) { return ((uint64_t)x.y << 32 | x.x) * kSharedRows; };
  // the pending groups of item j (none past the last record)
  auto pending_of = [&](const uint4& x, uint32_t j) {
    return rec_of(j) < n_recs ? part_groups(x.w, j % kParts) : 0u;
  };
  auto qbase_of = [](const uint4& x, uint32_t j) { return x.z + (j % kParts) * (kResolveQt * 16); };
  uint32_t j = 0;
  uint4 rec = fetch(0);
  uint4 rec_next = fetch(1);
  PartLoads<kResolveQt> P;
  part_load<kResolveQt, kPlane>(P, db, plane, n_rows, row0_of(rec), qbase_of(rec, 0), pending_of(rec, 0), queries,
                         n_queries);
  // The first part's words arrive here (vmcnt 0; expcnt and lgkmcnt left
  // alone), as every later part's do at the end of the previous iteration:
  // the compiler then sees them complete on every path into the loop and
  // does not make the loop's waits for them cover the next part's loads.
  __builtin_amdgcn_s_waitcnt(0x0F70);
  for (; rec_of(j) < n_recs; j++) {
    uint4 rec_after;
    PartLoads<kResolveQt> Pn;
    resolve_record<kResolveQt, kPlane>(L, P, db, plane, n_rows, row0_of(rec), qbase_of(rec, j), pending_of(rec, j),
                                queries, n_queries, threshold, hits, capacity, counter, index_base, [&] {
                                  rec_after = fetch(j + 2);
                                  part_load<kResolveQt, kPlane>(Pn, db, plane, n_rows, row0_of(rec_next),
                                                         qbase_of(rec_next, j + 1), pending_of(rec_next, j + 1),
                                                         queries, n_queries);
                                });
    rec = rec_next;
    rec_next = rec_after;
    P = Pn;
  }
  hits_flush(L, hits, capacity, counter);
}

// The shard holding MFMA row chunk `chunk` (views in chunk order).
__device__ __forceinline__ uint32_t shard_of_chunk(const ShardView* __restrict__ shards, uint32_t n_shards,
                                                   uint64_t chunk) {
  uint32_t sh = 0;
  while (sh + 1 < n_shards && shards[sh + 1].chunk_begin <= chunk) sh++;
  return sh;
}

// The shared-rows layout over a set of shards, persistent: a fixed grid (a
// multiple of 8 blocks) walks (global sub-chunk, group of kMfmaWaves query
// groups) items, the sub-chunks of shard s numbered from its first chunk x
// kSubsPerChunk.  The query count is read from device memory (`d_nq`, capped
// at nq_cap), so one captured launch serves batches of any size.  Records
// carry the global sub-chunk number.
template <bool kTri>
__global__ void __launch_bounds__(64 * kMfmaWaves) __attribute__((amdgpu_waves_per_eu(4))) pdq_match_mfma_shards_shared_kernel(
    const ShardView* __restrict__ shards, uint32_t n_shards, uint64_t total_chunks,
    const uint32_t* __restrict__ queries, const uint32_t* __restrict__ d_nq, uint32_t nq_cap, uint32_t threshold,
    uint4* __restrict__ recs, uint32_t* __restrict__ rec_count, uint32_t rec_cap) {
  const uint32_t nq = d_nq ? min(*d_nq, nq_cap) : nq_cap;
  if (nq == 0) return;
  __shared__ SharedRowsLds S;
  const uint32_t groups = (nq + kSharedQt * 16 - 1) / (kSharedQt * 16);
  const uint32_t sgroups = (groups + kMfmaWaves - 1) / kMfmaWaves;
  const uint64_t items = total_chunks * kSubsPerChunk * sgroups;
  for (uint64_t item = blockIdx.x; item < items; item += gridDim.x) {
    uint64_t gsub;
    uint32_t sgroup;
    item_coords(item, sgroups, gsub, sgroup);
    const ShardView& v = shards[shard_of_chunk(shards, n_shards, gsub / kSubsPerChunk)];
    const uint64_t sub_base = v.chunk_begin * kSubsPerChunk;
    mfma_item_shared<true, kTri>(S, reinterpret_cast<const uint32_t*>(v.rows),
                                       reinterpret_cast<const uint32_t*>(v.plane), v.n_rows, gsub - sub_base, sgroup,
                                       queries, nq, threshold, recs, rec_count, rec_cap, sub_base);
  }
}

// Its recheck kernel: as pdq_match_resolve_kernel, with each record's shard
// found from its global sub-chunk, and the rerun after an overflow walking
// the parts of every shard.
__global__ void __launch_bounds__(64 * kResolveWaves) pdq_match_resolve_shards_kernel(
    const ShardView* __restrict__ shards, uint32_t n_shards,
    const uint32_t* __restrict__ queries, const uint32_t* __restrict__ d_nq, uint32_t nq_cap, uint32_t threshold,
    MatchHit* __restrict__ hits, uint64_t capacity, unsigned long long* __restrict__ counter,
    const uint4* __restrict__ recs, const uint32_t* __restrict__ rec_count, uint32_t rec_cap) {
  const uint32_t nq = d_nq ? min(*d_nq, nq_cap) : nq_cap;
  if (nq == 0) return;
  __shared__ ResolveLds L;
  hits_init(L);
  const int wave = (int)(threadIdx.x >> 6);
  const uint32_t n_recs = *rec_count;
  if (n_recs > rec_cap) {
    const uint32_t groups = (nq + kRerunQt * 16 - 1) / (kRerunQt * 16);
    for (uint32_t sh = 0; sh < n_shards; sh++) {
      const ShardView& v = shards[sh];
      const uint64_t items = (v.n_rows + kRerunRows - 1) / kRerunRows * groups;
      for (uint64_t item = (uint64_t)blockIdx.x * kResolveWaves + wave; item < items;
           item += (uint64_t)gridDim.x * kResolveWaves) {
        even_part<kRerunQt, true, false>(
            L, DbGroups{v.rows, v.plane, v.n_rows, v.index_base, (uint32_t)(item / groups) * kEvenGroups, 1},
            rerun_groups(v.n_rows, item / groups), queries, nq, (uint32_t)(item % groups) * (kRerunQt * 16), threshold,
            hits, capacity, counter);
      }
    }
    hits_flush(L, hits, capacity, counter);
    return;
  }
  // whole records per wave, as in pdq_match_resolve_kernel
  const uint32_t stride = gridDim.x * kResolveWaves;
  uint32_t i = blockIdx.x * kResolveWaves + wave;
  uint4 rec = i < n_recs ? recs[i] : make_uint4(0, 0, 0, 0);
  for (; i < n_recs; i += stride) {
    const uint4 next = i + stride < n_recs ? recs[i + stride] : make_uint4(0, 0, 0, 0);
    const uint64_t gsub = (uint64_t)rec.y << 32 | rec.x;
    const ShardView& v = shards[shard_of_chunk(shards, n_shards, gsub / kSubsPerChunk)];
    const uint64_t row0 = (gsub - v.chunk_begin * kSubsPerChunk) * kSharedRows;
    const uint32_t* rows = reinterpret_cast<const uint32_t*>(v.rows);
    const uint32_t* vplane = reinterpret_cast<const uint32_t*>(v.plane);
#pragma unroll 1
    for (uint32_t part = 0; part < kParts; part++) {
      const uint32_t qbase = rec.z + part * (kResolveQt * 16);
      const uint32_t pending = part_groups(rec.w, part);
      PartLoads<kResolveQt> P;
      part_load<kResolveQt, true>(P, rows, vplane, v.n_rows, row0, qbase, pending, queries, nq);
      resolve_record<kResolveQt, true>(L, P, rows, vplane, v.n_rows, row0, qbase, pending, queries, nq, threshold, hits,
                                  capacity, counter, v.index_base, [] {});
    }
    rec = next;
  }
  hits_flush(L, hits, capacity, counter);
}

// The even layout over a set of shards.  The shards' row groups, one shard
// after the other, are cut into parts as for one database; a part that reaches
// over a shard's end is matched piece by piece.  The query count is read from device
// memory (`d_nq`, capped at nq_cap), so one captured launch of resident waves
// serves batches of any size: every wave works out the parts from it.  The
// matrix cores bound it as they do one database.  Before, a wave took 512-row
// items of its own query group one after the other, with up to a group's
// width of padding and a last round in which most waves had nothing left:
// five shards, 26.1M rows together, with batches of 37 images (296 queries) took
// 516 us and take 455, 100 images (800) 1136 and 908.
template <int QT, bool kTri>
__global__ void __launch_bounds__(64 * kMfmaWaves) __attribute__((amdgpu_waves_per_eu(4))) pdq_match_even_shards_kernel(
    const ShardView* __restrict__ shards, uint32_t n_shards, uint32_t row_groups,
    const uint32_t* __restrict__ queries, const uint32_t* __restrict__ d_nq, uint32_t nq_cap, uint32_t threshold,
    MatchHit* __restrict__ hits, uint64_t capacity, unsigned long long* __restrict__ counter) {
  const uint32_t nq = d_nq ? min(*d_nq, nq_cap) : nq_cap;
  if (nq == 0) return;
  __shared__ HitList<kEvenStage> H;
  hits_init(H);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t groups = (nq + QT * 16 - 1) / (QT * 16);
  const uint32_t waves_per_xcd = gridDim.x / 8 * kMfmaWaves;
  const EvenParts parts = even_parts(row_groups, groups, waves_per_xcd);
  for (uint32_t id = (blockIdx.x >> 3) * kMfmaWaves + wave;; id += waves_per_xcd) {
    const uint32_t part_x = id / groups;
    if (part_x >= parts.per_xcd) break;
    PartGroups rows = part_row_groups(part_x * 8 + (blockIdx.x & 7), parts, row_groups);
    uint32_t sh = 0;
    while (rows.count) {
      while (sh + 1 < n_shards && shards[sh + 1].group_begin <= rows.first) sh++;
      const ShardView& v = shards[sh];
      uint32_t n = rows.count;  // of them in this shard
      if (sh + 1 < n_shards)
        n = min(n, ((uint32_t)shards[sh + 1].group_begin - rows.first - 1) / rows.stride + 1);
      even_part<QT, true, kTri>(H, DbGroups{v.rows, v.plane, v.n_rows, v.index_base,
                                            rows.first - (uint32_t)v.group_begin, rows.stride},
                                n, queries, nq, (id - part_x * groups) * (uint32_t)(QT * 16), threshold, hits,
                                capacity, counter);
      rows.first += n * rows.stride;
      rows.count -= n;
    }
  }
  hits_flush(H, hits, capacity, counter);
}

// Record areas of the shared-rows layout: one per (device, stream), made on
// the stream's first such launch and kept for the life of the process, with
// a mutex so that the count reset, the filter and the resolve kernel of one
// call are enqueued together even when threads share a stream.  At most
// kMaxStreamAreas streams of a device get an area; calls on further streams,
// and on a stream being captured into a graph (which cannot allocate), run
// the even layout, which needs none.
constexpr uint32_t kRecordCap = 1u << 20;  // 16 MiB; more records (dense hits) rerun every item per wave
constexpr size_t kMaxStreamAreas = 16;     // per device

// The record cap passed to the kernels: kRecordCap, or less when set by
// set_match_record_cap (tests reach the overflow path at small sizes with
// it); the environment's YUME_PDQ_AMD_MATCH_RECORD_CAP (1 .. kRecordCap) is
// its initial value, read once.
static uint32_t env_record_cap() {
  const char* v = getenv("YUME_PDQ_AMD_MATCH_RECORD_CAP");
  if (!v || !*v) return kRecordCap;
  char* end = nullptr;
  const unsigned long long c = strtoull(v, &end, 10);
  return (end && *end == 0 && c >= 1 && c <= kRecordCap) ? (uint32_t)c : kRecordCap;
}
static std::atomic<uint32_t> g_record_cap{env_record_cap()};
static uint32_t record_cap() { return g_record_cap.load(std::memory_order_relaxed); }

bool set_match_record_cap(uint32_t cap) {
  if (cap > kRecordCap) return false;
  g_record_cap.store(cap == 0 ? kRecordCap : cap, std::memory_order_relaxed);
  return true;
}

// A stream's record area: the records, then two record-count slots
// (kCountSlotStride words apart).  Calls on the stream take the slots in
// turn, and each call's first kernel clears the slot of the next call, so a
// call needs no launch of its own to clear its count while the previous
// call's kernels were all enqueued.  slot and slot_clear are host state.
constexpr uint32_t kCountSlotStride = 32;
static_assert(2 * kCountSlotStride * sizeof(uint32_t) <= 256, "both count slots in the area's 256-byte tail");
struct RecordArea {
  uint4* recs = nullptr;
  uint32_t* count = nullptr;
  int cus = 0;  // compute units of the area's device
  uint32_t slot = 0;        // the count slot of the stream's next call
  bool slot_clear = false;  // that slot holds zero once the enqueued work has run
};

static std::mutex g_record_mu;

static hipError_t record_area(hipStream_t stream, RecordArea** out, bool* usable) {
  *usable = false;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  hipError_t e = hipStreamIsCapturing(stream, &cs);
  if (e != hipSuccess) return e;
  if (cs != hipStreamCaptureStatusNone) return hipSuccess;
  int dev = 0;
  if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
  // keyed by device and stream; hipStreamPerThread names a different
  // stream in each host thread, so its areas are also keyed by the thread
  using Key = std::tuple<int, hipStream_t, std::thread::id>;
  static std::map<Key, RecordArea> areas;  // guarded by g_record_mu
  static std::map<int, size_t> per_device;  // areas made per device
  const Key key{dev, stream, stream == hipStreamPerThread ? std::this_thread::get_id() : std::thread::id()};
  auto it = areas.find(key);
  if (it == areas.end()) {
    if (per_device[dev] >= kMaxStreamAreas) return hipSuccess;  // not usable: the even layout
    void* p = nullptr;
    if ((e = hipMalloc(&p, (size_t)kRecordCap * sizeof(uint4) + 256)) != hipSuccess) return e;
    RecordArea ra;
    if ((e = hipDeviceGetAttribute(&ra.cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) {
      (void)hipFree(p);
      return e;
    }
    ra.recs = static_cast<uint4*>(p);
    ra.count = reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(p) + (size_t)kRecordCap * sizeof(uint4));
    it = areas.emplace(key, ra).first;
    per_device[dev]++;
  }
  *out = &it->second;
  *usable = true;
  return hipSuccess;
}

// The record area of the no-allocation entry point: kScratchRecords records,
// then the count, in the code object's own device memory.  Each GPU the
// library runs on holds one copy (16 MiB + 256 B) until the process ends.
// Host code never names the array in a launch: its device address, per
// device, comes from hipGetSymbolAddress (scratch_area below).
constexpr uint32_t kScratchRecords = 1u << 20;
static __device__ __align__(256) uint4 scratch[kScratchRecords + 16];

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxScratchDevices];  // guarded by g_scratch_mu
static int g_scratch_cus[kMaxScratchDevices];

uint32_t match_scratch_records() { return kScratchRecords; }

// The current device's scratch area, its address looked up on the device's
// first call (with that device current) and kept.
static hipError_t scratch_area(RecordArea* out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxScratchDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if ((e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch))) != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    int cus = 0;
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    g_scratch_cus[dev] = cus;
    g_scratch_ptr[dev] = p;
  }
  out->recs = static_cast<uint4*>(g_scratch_ptr[dev]);
  out->count = reinterpret_cast<uint32_t*>(out->recs + kScratchRecords);
  out->cus = g_scratch_cus[dev];
  return hipSuccess;
}

// Clears the candidate-record count and, when asked, the hit counter.
__global__ void reset_counts_kernel(uint32_t* rec_count, unsigned long long* counter) {
  if (rec_count) *rec_count = 0u;
  if (counter) *counter = 0ull;
}

// The shared-rows layout's launches; *done is false where the call cannot use
// it (no record area for the stream).  fixed: the caller's area (the
// no-allocation entry point's scratch, sized for this call's worst case), else
// this stream's own.
static hipError_t launch_shared(const void* db, const void* plane, uint64_t n_rows, const void* queries,
                                uint32_t n_queries, uint32_t threshold, MatchHit* hits, uint64_t capacity,
                                unsigned long long* counter, uint64_t index_base, hipStream_t stream, bool reset,
                                const RecordArea* fixed, bool* done) {
  *done = false;
  const uint32_t groups = (n_queries + kSharedQt * 16 - 1) / (kSharedQt * 16);
  const uint32_t sgroups = (groups + kMfmaWaves - 1) / kMfmaWaves;
  const uint64_t blocks = ((n_rows + kSharedRows - 1) / kSharedRows + 7) / 8 * 8 * sgroups;  // whole XCD rounds
  if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
  std::lock_guard<std::mutex> g(g_record_mu);
  RecordArea ra;
  RecordArea* area = nullptr;  // the stream's own area, whose count slots alternate
  if (fixed) {
    ra = *fixed;
  } else {
    bool usable = false;
    const hipError_t e = record_area(stream, &area, &usable);
    if (e != hipSuccess || !usable) return e;
    ra = *area;
  }
  *done = true;
  const uint32_t* d = static_cast<const uint32_t*>(db);
  const uint32_t* p = static_cast<const uint32_t*>(plane);
  const uint32_t* q = static_cast<const uint32_t*>(queries);
  const uint32_t cap = fixed ? kScratchRecords : record_cap();
  // this call's count slot; the stream's area has the streaming kernel clear
  // the next call's slot, and the hit counter when this slot is already clear
  uint32_t* rc = ra.count;
  uint32_t* rc_next = nullptr;
  unsigned long long* hits_clear = nullptr;
  if (area) {
    rc = area->count + kCountSlotStride * area->slot;
    rc_next = area->count + kCountSlotStride * (area->slot ^ 1u);
  }
  if (area && area->slot_clear)
    hits_clear = reset ? counter : nullptr;
  else
    hipLaunchKernelGGL(reset_counts_kernel, dim3(1), dim3(1), 0, stream, rc, reset ? counter : nullptr);
  // the recheck kernel's resident blocks; the rerun after an overflow walks
  // all items with them
  const dim3 grid((unsigned)blocks), block(64 * kMfmaWaves);
  const dim3 rgrid(match_resolve_blocks(ra.cus)), rblock(64 * kResolveWaves);
  auto launch = [&](auto pl, auto tr) {
    constexpr bool kPlane = decltype(pl)::value, kTri = decltype(tr)::value;
    hipLaunchKernelGGL((pdq_match_mfma_kernel<kPlane, kTri>), grid, block, 0, stream, d, p, n_rows, q, n_queries,
                       threshold, sgroups, ra.recs, rc, cap, rc_next, hits_clear);
    hipLaunchKernelGGL((pdq_match_resolve_kernel<kPlane>), rgrid, rblock, 0, stream, d, p, n_rows, q,
                       n_queries, threshold, hits, capacity, counter, index_base, ra.recs, rc, cap);
  };
  using T = std::integral_constant<bool, true>;
  using F = std::integral_constant<bool, false>;
  // three products per accumulator where they apply
  const bool tri = threshold >= kTriMinThreshold;
  if (plane && tri) launch(T(), T());
  else if (plane) launch(T(), F());
  else if (tri) launch(F(), T());
  else launch(F(), F());
  const hipError_t e = hipGetLastError();
  if (area) {
    // the next call's slot is clear only if this call's kernels were all
    // enqueued; otherwise the next call clears it with a launch
    if (e == hipSuccess) area->slot ^= 1u;
    area->slot_clear = e == hipSuccess;
  }
  return e;
}

// f(integral_constant<int, qt>()) for the widths the even layout is built for:
// every one, since with the even ones only half of all batches compute a tile of
// padding per group (10^7 rows, even widths only / all, us: 48 queries 43.6 /
// 38.0, 112 64.9 / 61.0, 144 75.5 / 69.6, 264 131 / 122, 400 168 / 160).
template <class F>
static hipError_t with_query_tiles(int qt, F&& f) {
  switch (qt) {
    case 2: return f(std::integral_constant<int, 2>());
    case 3: return f(std::integral_constant<int, 3>());
    case 4: return f(std::integral_constant<int, 4>());
    case 5: return f(std::integral_constant<int, 5>());
    case 6: return f(std::integral_constant<int, 6>());
    case 7: return f(std::integral_constant<int, 7>());
    case 8: return f(std::integral_constant<int, 8>());
    case 9: return f(std::integral_constant<int, 9>());
    case 10: return f(std::integral_constant<int, 10>());
    case 11: return f(std::integral_constant<int, 11>());
    case 12: return f(std::integral_constant<int, 12>());
    case 13: return f(std::integral_constant<int, 13>());
    case 14: return f(std::integral_constant<int, 14>());
    case 15: return f(std::integral_constant<int, 15>());
    case 16: return f(std::integral_constant<int, 16>());
    default: return hipErrorInvalidValue;
  }
}

// The even layout's waves that are resident at once: four per SIMD.
static uint32_t even_waves_per_xcd(int cus) { return (uint32_t)std::max(1, cus) * 16 / 8; }

// The held-rows layout's launch.
template <int kPer>
static hipError_t launch_held_plan(const HeldPlan& plan, const void* db, const void* plane, uint64_t n_rows,
                                   const void* queries, uint32_t n_queries, uint32_t threshold, MatchHit* hits,
                                   uint64_t capacity, unsigned long long* counter, uint64_t index_base,
                                   hipStream_t stream, bool reset) {
  const dim3 grid((unsigned)(8 * plan.blocks_per_xcd * plan.chunks)), block(64 * kHeldWaves);
  const uint4* rows = static_cast<const uint4*>(db);
  const uint4* prefix = static_cast<const uint4*>(plane);
  const uint32_t* q = static_cast<const uint32_t*>(queries);
  if (reset) hipLaunchKernelGGL(reset_counts_kernel, dim3(1), dim3(1), 0, stream, nullptr, counter);
  if (plane)
    hipLaunchKernelGGL((pdq_match_held_kernel<kPer, true>), grid, block, 0, stream, rows, prefix, n_rows, q, n_queries,
                       threshold, hits, capacity, counter, index_base, plan);
  else
    hipLaunchKernelGGL((pdq_match_held_kernel<kPer, false>), grid, block, 0, stream, rows, prefix, n_rows, q,
                       n_queries, threshold, hits, capacity, counter, index_base, plan);
  return hipGetLastError();
}

static hipError_t launch_held(const void* db, const void* plane, uint64_t n_rows, const void* queries,
                              uint32_t n_queries, uint32_t threshold, MatchHit* hits, uint64_t capacity,
                              unsigned long long* counter, uint64_t index_base, hipStream_t stream, bool reset) {
  int dev = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
  const uint32_t per_xcd = (uint32_t)std::max(8, cus) / 8, tiles = (n_queries + 15) / 16;
  const HeldPlan two = held_plan<2>(n_rows, tiles, per_xcd), three = held_plan<3>(n_rows, tiles, per_xcd);
  // two products per accumulator serve every threshold; three take fewer
  // instructions a product, but hold 192 rows a wave, which leaves small
  // databases with fewer waves (10^4 rows x 2048 queries, three / two: 17.4 /
  // 13.4 us, 3x10^4 x 2048 16.1 / 11.7, 4x10^5 x 256 14.5 / 12.5)
  if (threshold >= kTriMinThreshold && three.cost <= two.cost)
    return launch_held_plan<3>(three, db, plane, n_rows, queries, n_queries, threshold, hits, capacity, counter,
                               index_base, stream, reset);
  return launch_held_plan<2>(two, db, plane, n_rows, queries, n_queries, threshold, hits, capacity, counter,
                             index_base, stream, reset);
}

template <int QT>
static hipError_t launch_even(const void* db, const void* plane, uint64_t n_rows, const void* queries,
                              uint32_t n_queries, uint32_t threshold, MatchHit* hits, uint64_t capacity,
                              unsigned long long* counter, uint64_t index_base, hipStream_t stream, bool reset) {
  int dev = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
  const uint32_t groups = (n_queries + QT * 16 - 1) / (QT * 16);
  const uint64_t row_groups = (n_rows + kEvenRows - 1) / kEvenRows;
  if (row_groups > 0xffffffffull) return hipErrorInvalidValue;
  const EvenParts parts = even_parts((uint32_t)row_groups, groups, even_waves_per_xcd(cus));
  const uint64_t waves = (uint64_t)parts.per_xcd * groups;  // per XCD
  const uint64_t blocks = 8 * ((waves + kMfmaWaves - 1) / kMfmaWaves);
  if (blocks > 0x7fffffffull || waves > 0xffffffffull) return hipErrorInvalidValue;
  if (reset) hipLaunchKernelGGL(reset_counts_kernel, dim3(1), dim3(1), 0, stream, nullptr, counter);
  const bool tri = QT > 2 && threshold >= kTriMinThreshold;
  auto launch = [&](auto pl, auto tr) {
    hipLaunchKernelGGL((pdq_match_even_kernel<QT, decltype(pl)::value, decltype(tr)::value>), dim3((unsigned)blocks),
                       dim3(64 * kMfmaWaves), 0, stream, static_cast<const uint4*>(db),
                       static_cast<const uint4*>(plane), n_rows, (uint32_t)row_groups,
                       static_cast<const uint32_t*>(queries), n_queries, threshold, hits, capacity, counter,
                       index_base, groups, parts);
  };
  using T = std::integral_constant<bool, true>;
  using F = std::integral_constant<bool, false>;
  if (plane && tri) launch(T(), T());
  else if (plane) launch(T(), F());
  else if (tri) launch(F(), T());
  else launch(F(), F());
  return hipGetLastError();
}

// Prefix plane: plane[r * 4 + k] = word k of row r (the row's first 16
// bytes), zero for the padding rows up to a whole 16-row tile.
__global__ void build_prefix_plane_kernel(const uint4* __restrict__ db, uint64_t n_rows, uint4* __restrict__ plane,
                                          uint64_t n_padded) {
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_padded) return;
  plane[r] = r < n_rows ? db[2 * r] : make_uint4(0, 0, 0, 0);
}

uint64_t prefix_plane_bytes(uint64_t n_rows) { return (n_rows + 15) / 16 * 256; }

hipError_t launch_build_prefix_plane(const void* db, uint64_t n_rows, void* plane, hipStream_t stream) {
  const uint64_t n_padded = (n_rows + 15) / 16 * 16;
  if (n_padded == 0) return hipSuccess;
  const uint64_t blocks = (n_padded + 255) / 256;
  if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
  hipLaunchKernelGGL(build_prefix_plane_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                     static_cast<const uint4*>(db), n_rows, static_cast<uint4*>(plane), n_padded);
  return hipGetLastError();
}

uint64_t mfma_chunks(uint64_t n_rows) {
  const uint64_t rows_per_block = (uint64_t)kMfmaWaves * kMfmaTilesPerWave * 16;
  return ((n_rows + rows_per_block - 1) / rows_per_block + 7) / 8 * 8;
}

template <int QT>
static hipError_t launch_even_shards(const ShardView* shards, uint32_t n_shards, uint64_t row_groups,
                                     const void* queries, const uint32_t* d_nq, uint32_t nq_cap, uint32_t threshold,
                                     MatchHit* hits, uint64_t capacity, unsigned long long* counter, int cus,
                                     hipStream_t stream) {
  // resident blocks, fewer where the largest batch has fewer parts
  const uint32_t groups = (nq_cap + QT * 16 - 1) / (QT * 16);
  const EvenParts parts = even_parts((uint32_t)row_groups, groups ? groups : 1, even_waves_per_xcd(cus));
  const uint64_t most = ((uint64_t)parts.per_xcd * groups + kMfmaWaves - 1) / kMfmaWaves;
  const uint64_t per_xcd = std::max<uint64_t>(1, std::min<uint64_t>(even_waves_per_xcd(cus) / kMfmaWaves, most));
  const dim3 grid((unsigned)(8 * per_xcd)), block(64 * kMfmaWaves);
  const uint32_t* q = static_cast<const uint32_t*>(queries);
  if (QT > 2 && threshold >= kTriMinThreshold)
    hipLaunchKernelGGL((pdq_match_even_shards_kernel<QT, true>), grid, block, 0, stream, shards, n_shards,
                       (uint32_t)row_groups, q, d_nq, nq_cap, threshold, hits, capacity, counter);
  else
    hipLaunchKernelGGL((pdq_match_even_shards_kernel<QT, false>), grid, block, 0, stream, shards, n_shards,
                       (uint32_t)row_groups, q, d_nq, nq_cap, threshold, hits, capacity, counter);
  return hipGetLastError();
}

hipError_t launch_match_even_shards(int qt, const ShardView* shards, uint32_t n_shards, uint64_t row_groups,
                                    const void* queries, const uint32_t* d_nq, uint32_t nq_cap, uint32_t threshold,
                                    MatchHit* hits, uint64_t capacity, unsigned long long* counter, int cus,
                                    hipStream_t stream) {
  if (threshold >= 64 || row_groups > 0xffffffffull) return hipErrorInvalidValue;
  return with_query_tiles(qt, [&](auto q) {
    return launch_even_shards<decltype(q)::value>(shards, n_shards, row_groups, queries, d_nq, nq_cap, threshold,
                                                  hits, capacity, counter, cus, stream);
  });
}

uint64_t match_row_groups(uint64_t n_rows) { return (n_rows + kEvenRows - 1) / kEvenRows; }

uint64_t match_record_area_bytes() { return (uint64_t)kRecordCap * sizeof(uint4) + 256; }

hipError_t launch_match_shared_shards(const ShardView* shards, uint32_t n_shards, uint64_t total_chunks,
                                      const void* queries, const uint32_t* d_nq, uint32_t nq_cap, uint32_t threshold,
                                      MatchHit* hits, uint64_t capacity, unsigned long long* counter,
                                      void* record_area, uint32_t grid, uint32_t rgrid, hipStream_t stream) {
  if (threshold >= 64 || grid == 0 || grid % 8 || rgrid == 0 || !record_area) return hipErrorInvalidValue;
  uint4* recs = static_cast<uint4*>(record_area);
  uint32_t* count =
      reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(record_area) + (size_t)kRecordCap * sizeof(uint4));
  const uint32_t* q = static_cast<const uint32_t*>(queries);
  const dim3 block(64 * kMfmaWaves), rblock(64 * kResolveWaves);
  const uint32_t cap = record_cap();
  hipLaunchKernelGGL(reset_counts_kernel, dim3(1), dim3(1), 0, stream, count, nullptr);
  if (threshold >= kTriMinThreshold)  // three products per accumulator
    hipLaunchKernelGGL((pdq_match_mfma_shards_shared_kernel<true>), dim3(grid), block, 0, stream, shards, n_shards,
                       total_chunks, q, d_nq, nq_cap, threshold, recs, count, cap);
  else
    hipLaunchKernelGGL((pdq_match_mfma_shards_shared_kernel<false>), dim3(grid), block, 0, stream, shards, n_shards,
                       total_chunks, q, d_nq, nq_cap, threshold, recs, count, cap);
  hipLaunchKernelGGL(pdq_match_resolve_shards_kernel, dim3(rgrid), rblock, 0, stream, shards, n_shards, q, d_nq,
                     nq_cap, threshold, hits, capacity, counter, recs, count, cap);
  return hipGetLastError();
}

// From 12 queries the one group of two query tiles, mostly padding, costs less
// than the vector-ALU scan, which pays per query, as long as candidates are
// rare.  10^7 rows over the plane, vector ALU / matrix cores in us: 8 queries
// 27 / 31, 12 36 / 31, 16 46 / 31, 24 65 / 32, 31 82 / 31 at threshold 31; 16
// queries 46 / 35 at 40, 48 / 57 at 44 and 65 / 144 at 48 (raw rows cross at 16
// queries, 53 / 51; below 10^6 rows both are one launch).
bool match_mfma_applicable(uint32_t n_queries, uint32_t threshold) {
  return n_queries >= 32 ? threshold < 64 : n_queries >= 12 && threshold <= 40;
}

// Which layout a call runs, and its query tiles per wave.  Costs, in tenths of
// a query tile's products over all rows (0.45 us per 10^7 rows), fitted to
// 10^7 rows over the plane (us at 2 / 4 / 8 / 12 / 14 / 16 tiles in one group:
// 32 / 42 / 60 / 77 / 87 / 97; 16 tiles in two and four groups: 186 and 348):
// a query group costs its tiles and 2.7 more (the rows' loads and expansions,
// the votes), so few wide groups, as long as they are full.  The shared-rows
// layout always computes whole groups of 64 tiles, at 73 per 64, and its
// recheck kernel takes some 8 us: it wins where the tiles nearly fill
// its groups and the rows are many (64 tiles: 338 against 348 us at 10^7 rows,
// 48 against 48 at 10^6, 35 against 17 at 10^5; 128 tiles: 83 against 88 us at
// 10^6, 46 against 28 at 10^5).
constexpr int kEvenCost = 27;
constexpr int kSharedCost = 733;
constexpr uint64_t kSharedGain = 30000000;  // rows x cost units that pay for the recheck

MatchPlan match_plan(uint64_t n_rows, uint32_t n_queries, int most_qt) {
  const uint64_t tiles = ((uint64_t)n_queries + 15) / 16;
  MatchPlan plan{false, 2};
  uint64_t best = ~0ull;
  for (int qt = 2; qt <= most_qt; qt++) {
    const uint64_t cost = (tiles + qt - 1) / qt * (uint64_t)(kEvenCost + 10 * qt);
    if (cost < best) {
      best = cost;
      plan.qt = qt;
    }
  }
  const uint64_t shared = (tiles + 63) / 64 * kSharedCost;
  plan.shared = shared < best && n_rows >= kSharedGain / (best - shared);
  return plan;
}

// The held-rows layout takes databases up to 7x10^5 rows from 193 queries, and
// up to 5x10^4 from 65: at its lines (even layout / held, us) 7x10^5 rows x 200
// queries 15.8 / 14.0 and x 2048 69.4 / 63.3, but 10^6 rows x 256 19.9 / 22.4;
// 5x10^5 rows x 160 queries 11.1 / 12.7, x 200 13.5 / 13.5; 10^4 rows x 97
// queries 9.5 / 9.2, 10^3 rows x 65 13.5 / 9.1.  Raw rows and thresholds with
// two products per accumulator lie the same or a little further in its favour.
static bool held_pays(uint64_t n_rows, uint32_t n_queries) {
  return n_rows <= 700000 && n_queries > (n_rows <= 50000 ? 64u : 192u);
}

static hipError_t launch_match_mfma_any(const void* db, const void* plane, uint64_t n_rows, const void* queries,
                                        uint32_t n_queries, uint32_t threshold, MatchHit* hits, uint64_t capacity,
                                        unsigned long long* counter, uint64_t index_base, hipStream_t stream,
                                        bool reset_counter, const RecordArea* fixed) {
  if (threshold >= 64) return hipErrorInvalidValue;
  if (n_rows == 0 || n_queries == 0) {
    if (!reset_counter) return hipSuccess;
    hipLaunchKernelGGL(reset_counts_kernel, dim3(1), dim3(1), 0, stream, nullptr, counter);
    return hipGetLastError();
  }
  if (held_pays(n_rows, n_queries))
    return launch_held(db, plane, n_rows, queries, n_queries, threshold, hits, capacity, counter, index_base, stream,
                       reset_counter);
  const MatchPlan plan = match_plan(n_rows, n_queries);
  if (plan.shared) {
    bool done = false;
    const hipError_t e = launch_shared(db, plane, n_rows, queries, n_queries, threshold, hits, capacity, counter,
                                       index_base, stream, reset_counter, fixed, &done);
    if (e != hipSuccess || done) return e;
  }
  return with_query_tiles(plan.qt, [&](auto qt) {
    return launch_even<decltype(qt)::value>(db, plane, n_rows, queries, n_queries, threshold, hits, capacity, counter,
                                            index_base, stream, reset_counter);
  });
}

hipError_t launch_match_mfma(const void* db, const void* plane, uint64_t n_rows, const void* queries,
                             uint32_t n_queries, uint32_t threshold, MatchHit* hits, uint64_t capacity,
                             unsigned long long* counter, uint64_t index_base, hipStream_t stream,
                             bool reset_counter) {
  return launch_match_mfma_any(db, plane, n_rows, queries, n_queries, threshold, hits, capacity, counter, index_base,
                               stream, reset_counter, nullptr);
}

// The no-allocation entry point's limit: the records of a layout with eight
// query tiles per wave up to 1008 queries and sixteen above, which is what it
// has always accepted.  No call of the shared-rows layout writes more.
uint64_t match_mfma_scratch_records(uint64_t n_rows, uint32_t n_queries) {
  const uint32_t tiles = (n_queries + 15) / 16;
  const uint32_t qt = tiles <= 2 ? 2 : tiles <= 4 ? 4 : tiles < 64 ? 8 : 16;
  const uint32_t groups = (n_queries + qt * 16 - 1) / (qt * 16);
  if (n_rows == 0 || groups < (uint32_t)kMfmaWaves) return 0;
  const uint64_t subs8 = ((n_rows + kSharedRows - 1) / kSharedRows + 7) / 8 * 8;
  const uint64_t sgroups = (groups + kMfmaWaves - 1) / kMfmaWaves;
  return subs8 * sgroups * kMfmaWaves;  // at most one record per wave of each block
}

hipError_t launch_match_mfma_noalloc(const void* db, const void* plane, uint64_t n_rows, const void* queries,
                                     uint32_t n_queries, uint32_t threshold, MatchHit* hits, uint64_t capacity,
                                     unsigned long long* counter, uint64_t index_base, hipStream_t stream,
                                     bool reset_counter) {
  if (match_mfma_scratch_records(n_rows, n_queries) > kScratchRecords) return hipErrorInvalidValue;
  RecordArea ra;
  hipError_t e = scratch_area(&ra);
  if (e != hipSuccess) return e;
  return launch_match_mfma_any(db, plane, n_rows, queries, n_queries, threshold, hits, capacity, counter, index_base,
                               stream, reset_counter, &ra);
}

}  // namespace ypdq
