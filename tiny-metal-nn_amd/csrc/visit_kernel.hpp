// visit_kernel.hpp -- the lazy-Adam visit flags of a batch, from its positions
// alone, and the hash-grid backward that then only has to add what does not
// truncate to 0.
//
// A point visits every corner of its cell at every level whatever its
// gradient is (mask semantics: emit_active_hash_tracking,
// mlp_kernel_emitter.cpp:48-71). Stored by the backward itself those flags are
// one byte store per point, level and pair of corners at a random table
// entry, each a memory request of its own: at 4D, 16 levels of 2^22 entries
// and 2^20 points they are the whole 1395 us of hash_scatter_level_kernel
// once training converges (every contribution truncates to 0). Here a block
// collects one level's flags (or one 2^20-entry range of them) of its share
// of the points as bits in LDS, where a corner costs one LDS atomic, and writes
// the bits out; visit_expand_kernel then stores the flag bytes, once for all
// shares (byte stores by every share took a third of the pass).
#pragma once

#include "scatter_kernel.hpp"

namespace tmnn_hip {

// 1024-thread blocks; a block's bits cover at most 2^20 entries (128 KB LDS).
constexpr int kVisitThreads = 1024;
constexpr uint32_t kVisitLog2Range = 20;

struct VisitArgs {
  int32_t n;                // points
  int32_t share;            // points per block (blockIdx.x-th share)
  uint32_t log2T;
  uint32_t log2W;           // 2^log2W LDS words of 32 entries: min(T, 2^20) entries
  float res[kMaxLevels];
  const float *pos;         // [n][D], any order
  uint32_t *bits;           // [shares][rows][W] (rows: gridDim.y)
};

// blockIdx.y = level * ranges + range (RANGED: more than one range a level).
// Entry e of the range is bit e / W of word e % W: a run of cells along x
// falls into different words and banks, and lanes that walk the bits of
// consecutive words reach consecutive entries. The hash's terms are kept
// times 4, so that an entry's masked bits are its word's byte address.
typedef __attribute__((address_space(3))) uint32_t visit_word;

__device__ __forceinline__ visit_word *visit_word_at(uint32_t byte) {
  // the bits are the kernel's only LDS: they start at address 0 (checked when
  // a trainer is created; through the array's own address the kernels take 5%
  // more instructions)
  return reinterpret_cast<visit_word *>(byte);
}

__device__ __forceinline__ void visit_or(uint32_t byte, uint32_t bit) {
  __hip_atomic_fetch_or(visit_word_at(byte), bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The corners of one point. DENSE: the bit is read first, so that points
// sharing a cell (a sorted or scanned batch on a coarse level) do not
// serialise on one word's atomic.
template <int D, bool RANGED, bool DENSE>
__device__ __forceinline__ void visit_point(const VisitArgs &a, int i, float rl, uint32_t tmask,
                                            uint32_t rbase, uint32_t amask, uint32_t ashift) {
  constexpr uint32_t kPrimes[4] = {1u, kPrimeY, kPrimeZ, kPrimeW};
  float p[D];
#pragma unroll
  for (int k = 0; k < D; ++k) p[k] = a.pos[static_cast<size_t>(i) * D + k];
  const Cell<D> c = cell_of<D>(p, rl);
  uint32_t term[D][2];  // hash_corner's terms times 4, from this range's base
#pragma unroll
  for (int k = 0; k < D; ++k)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint32_t t = (static_cast<uint32_t>(c.bc[k] + s) * kPrimes[k]) & tmask;
      term[k][s] = (RANGED && k == D - 1 ? t ^ rbase : t) << 2;
    }
  uint32_t row[1 << (D - 1)];  // the corners' terms but x's
#pragma unroll
  for (int m = 0; m < (1 << (D - 1)); ++m) {
    row[m] = term[1][m & 1];
#pragma unroll
    for (int k = 2; k < D; ++k) row[m] ^= term[k][(m >> (k - 1)) & 1];
  }
  if constexpr (DENSE) {
    uint32_t seen[1 << D];
#pragma unroll
    for (int m = 0; m < (1 << D); ++m)
      seen[m] = *visit_word_at((row[m >> 1] ^ term[0][m & 1]) & amask);
#pragma unroll
    for (int m = 0; m < (1 << D); ++m) {
      const uint32_t e4 = row[m >> 1] ^ term[0][m & 1];
      const uint32_t b = e4 >> ashift;  // 32 and above: another range's entry
      const uint32_t bit = 1u << (b & 31u);
      if ((!RANGED || b < 32u) && !(seen[m] & bit)) visit_or(e4 & amask, bit);
    }
  } else if (RANGED && __any((term[0][0] ^ term[0][1]) >> (ashift + 5u))) {
    // a cell whose x and x + 1 corners lie in different ranges (x ends in 20
    // one bits): each corner by itself
#pragma unroll
    for (int m = 0; m < (1 << D); ++m) {
      const uint32_t e4 = row[m >> 1] ^ term[0][m & 1];
      const uint32_t b = e4 >> ashift;
      if (b < 32u) visit_or(e4 & amask, 1u << (b & 31u));
    }
  } else {
#pragma unroll
    for (int m = 0; m < (1 << (D - 1)); ++m) {
      const uint32_t e0 = row[m] ^ term[0][0], e1 = row[m] ^ term[0][1];
      if (!RANGED || (e0 >> ashift) < 32u) {
        visit_or(e0 & amask, 1u << ((e0 >> ashift) & 31u));
        visit_or(e1 & amask, 1u << ((e1 >> ashift) & 31u));
      }
    }
  }
}

template <int D, bool RANGED>
__global__ void __launch_bounds__(kVisitThreads) visit_kernel(VisitArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint32_t visit_bits[];
  const uint32_t log2S = RANGED ? a.log2T - (a.log2W + 5u) : 0u;
  const int l = static_cast<int>(blockIdx.y >> log2S);
  const uint32_t range = blockIdx.y & ((1u << log2S) - 1u);
  const uint32_t W = 1u << a.log2W;
  for (uint32_t w = threadIdx.x; w < W; w += kVisitThreads) visit_bits[w] = 0u;
  __syncthreads();
  const uint32_t tmask = (1u << a.log2T) - 1u;
  const uint32_t rbase = range << (a.log2W + 5u);
  const uint32_t amask = (W - 1u) << 2, ashift = a.log2W + 2u;
  const float rl = a.res[l];
  const int begin = static_cast<int>(blockIdx.x) * a.share;
  const int end = min(a.n, begin + a.share);
  // a level whose grid has few cells is hit many times per entry
  float cells = 1.0f;
#pragma unroll
  for (int k = 0; k < D; ++k) cells *= rl + 1.0f;
  const bool dense = static_cast<float>(end - begin) * (1 << D) >=
                     4.0f * fminf(cells, static_cast<float>(1u << a.log2T));
  if (dense) {
    for (int i = begin + static_cast<int>(threadIdx.x); i < end; i += kVisitThreads)
      visit_point<D, RANGED, true>(a, i, rl, tmask, rbase, amask, ashift);
  } else {
    for (int i = begin + static_cast<int>(threadIdx.x); i < end; i += kVisitThreads)
      visit_point<D, RANGED, false>(a, i, rl, tmask, rbase, amask, ashift);
  }
  __syncthreads();
  uint4 *out = reinterpret_cast<uint4 *>(
      a.bits + ((static_cast<size_t>(blockIdx.x) * gridDim.y + blockIdx.y) << a.log2W));
  for (uint32_t w = threadIdx.x; w < W / 4u; w += kVisitThreads)
    out[w] = reinterpret_cast<const uint4 *>(visit_bits)[w];
}

// One thread per word of a row (level and range): the flags of the entries
// that any share visited. mask: [L][T]; the rows' entries are contiguous.
constexpr int kVisitExpandThreads = 256;

struct VisitExpandArgs {
  const uint32_t *bits;  // [shares][total words]
  uint32_t total;        // words of one share: L * T / 32
  uint32_t log2W;
  int32_t shares;
  uint8_t *mask;
};

__global__ void __launch_bounds__(kVisitExpandThreads) visit_expand_kernel(VisitExpandArgs a) {
  const uint32_t i = blockIdx.x * kVisitExpandThreads + threadIdx.x;
  if (i >= a.total) return;
  uint32_t bits = 0u;
#pragma unroll 8
  for (int s = 0; s < a.shares; ++s) bits |= a.bits[static_cast<size_t>(s) * a.total + i];
  uint8_t *flags = a.mask + (static_cast<size_t>(i >> a.log2W) << (a.log2W + 5u)) +
                   (i & ((1u << a.log2W) - 1u));
#pragma unroll 8
  for (uint32_t b = 0; b < 32u; ++b)
    if ((bits >> b) & 1u) flags[b << a.log2W] = 1;
}

// The hash-grid backward of a batch that stores no visit flags (a.mask is null:
// visit_kernel has them). A block takes 64 consecutive points: it reads their
// dx rows once, coalesced, and notes per level whether any contribution can be
// nonzero (grads_vanish, the test of scatter_point_level); its waves then run
// the levels that have one, lanes on consecutive points as in
// hash_scatter_kernel. A batch whose contributions all truncate to 0 costs
// one pass over dx (4D, T = 2^22, 2^20 points: step 4904 -> 3600 us). Tables
// above 8 MB a level run it too although their flag-storing backward goes
// level by level: with 5 to 63% of the entries reached by nonzero contributions
// 2031 -> 1668 us and 7624 -> 7709 (3D 16x4, T = 2^21, 2^19 points), 6530 ->
// 4167 and 14177 -> 13921 (that 4D shape).
constexpr int kNonzeroPoints = 64;

template <int D, int F>
__global__ void __launch_bounds__(kScatterThreads) hash_scatter_nonzero_kernel(ScatterArgs a) {
  __shared__ uint32_t live;  // bit per level
  const int first = static_cast<int>(blockIdx.x) * kNonzeroPoints;
  const int count = min(kNonzeroPoints, a.n - first);
  if (threadIdx.x == 0) live = 0u;
  __syncthreads();
  const float *rows = a.dx + static_cast<size_t>(first) * a.IN;
  const int total = count * a.IN;
  uint32_t mine = 0u;
  if ((a.IN & 3) == 0) {
    // IN divides the row walk evenly: quad q of the block's rows
#pragma unroll 4
    for (int e = static_cast<int>(threadIdx.x) * 4; e < total; e += kScatterThreads * 4) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>(rows + e);
      const int c = e % a.IN;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float d[1] = {v[r]};
        if (!grads_vanish<1>(d)) mine |= 1u << ((c + r) / F);
      }
    }
  } else {
    for (int e = static_cast<int>(threadIdx.x); e < total; e += kScatterThreads) {
      const float d[1] = {rows[e]};
      if (!grads_vanish<1>(d)) mine |= 1u << ((e % a.IN) / F);
    }
  }
  if (mine) atomicOr(&live, mine);
  __syncthreads();
  uint32_t todo = live;
  if (todo == 0u) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool valid = lane < count;
  const int i = first + (valid ? lane : 0);
  float p[D];
#pragma unroll
  for (int k = 0; k < D; ++k) p[k] = a.pos[static_cast<size_t>(i) * D + k];
  for (int turn = 0; todo != 0u; ++turn) {
    const int l = __ffs(static_cast<int>(todo)) - 1;
    todo &= todo - 1u;
    if ((turn & (kScatterThreads / 64 - 1)) != wave) continue;
    float d[F];
#pragma unroll
    for (int f = 0; f < F; ++f) d[f] = a.dx[static_cast<size_t>(i) * a.IN + l * F + f];
    scatter_point_level<D, F>(a, l, p, d, valid, lane);
  }
}

}  // namespace tmnn_hip
