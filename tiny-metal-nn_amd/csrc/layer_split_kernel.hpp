// layer_split_kernel.hpp -- the layer-wise path's wide products (layer_kernels.hpp)
// on the bf16 matrix cores with fp32 operands split in three.
//
// v_mfma_f32_16x16x4_f32 runs at a sixteenth of the bf16 rate. An fp32 value
// is exactly the sum of three bf16 values (h = bf16(x), m = bf16(x - h), l =
// x - h - m: 8 significand bits each, round to nearest, so each part's sign is
// free), products of bf16 values are exact in fp32, and of the nine partial
// products the three dropped ones (m l, l m, l l) sum to at most 2^-24 of the
// product (|m| <= 2^-8 |x|, |l| <= 2^-17 |x|: twice 2^-25): six
// v_mfma_f32_16x16x32_bf16 per 32 K replace eight fp32 MFMAs at 6/16 of their
// time. The running accumulator takes a step's leading product and the sum of
// the five smaller ones: two roundings per 32 K where the fp32 MFMAs round
// eight times, and results closer to 64 bits than theirs (256 wide: outputs
// 2.5e-7 against 4.3e-7, weight gradients of 66001 points 3.5e-7 against
// 9.8e-7; with all six products on the running accumulator they ended 5 to 50%
// further off). Parts below bf16's smallest value (2^-133) are lost: operands
// under 1e-34 keep fewer than 24 bits (1e-36: 1.6e-5, where the fp32 MFMAs hold
// 1.7e-7 down to 1e-37).
// An infinity or a value above bf16's largest (3.39e38) has no such parts: its
// products are NaN. An output whose sum is not finite is computed again in
// fp32 before its epilogue (ls_exact), whose ReLU would otherwise turn that
// NaN into 0.
//
// Tile: 64 x TC outputs (TC 64 or 128) per 256-thread block, each of its four
// waves a quarter, K in steps of 32 whose split planes sit in LDS. The split's
// VALU work and the LDS traffic each take about as long as the MFMAs, so more
// resident blocks beat larger tiles: 128 x 128 (two blocks per CU) was as fast
// as 64 x 128 at 65536 x 256 x 256 and slower everywhere below. The
// weights' side is the MFMA's row operand, so that a lane ends up with four
// consecutive columns of one output row: 16-byte epilogue accesses without a
// pass through LDS. 65536 x 256 x 256: forward 101 -> 69 us, delta 104 -> 64,
// weight gradient 131 -> 76 (the fp32 MFMA tiles ran at 82 to 85 TFLOP/s), the
// h256_3d step 534 -> 405 us (423 with its batch sorted).
#pragma once

#include "layer_kernels.hpp"

namespace tmnn_hip {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kLsK = 32;     // K per step
constexpr int kLsRows = 64;  // output rows per tile

// The three bf16 parts of two floats, packed.
struct LsSplit {
  uint32_t h, m, l;
};

__device__ __forceinline__ uint32_t ls_pack(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float ls_low(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float ls_high(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }

__device__ __forceinline__ LsSplit ls_split(float a, float b) {
  LsSplit s;
  s.h = ls_pack(a, b);
  a -= ls_low(s.h);
  b -= ls_high(s.h);
  s.m = ls_pack(a, b);
  a -= ls_low(s.m);
  b -= ls_high(s.m);
  s.l = ls_pack(a, b);
  return s;
}

// An operand of T rows in LDS: plane h, m, l, each [T][32] bf16 with the four
// 16-byte slots of a row permuted by an XOR with (-(row / 4)) % 4, so that
// every 16-lane cycle of the operand read (lane p + 16 q: slot q of row p)
// covers the 64 banks once (the bank model of layer_kernels.hpp).
template <int T>
__device__ __forceinline__ int ls_slot(int row, int q) {
  return row * 64 + 16 * (q ^ (-(row >> 2) & 3));
}

// Global side of an operand tile: T rows by 32 K from (r0, k0), NQ quads of
// four floats per thread. KFAST: K contiguous in memory (quad: four K of one
// row; eight lanes read a row's 128 bytes). Else rows contiguous (quad: four
// rows at one K; neighbouring lanes take neighbouring K, so that a 16-lane
// store covers whole rows of the LDS planes; lanes along the rows met four to a
// bank: the 257 x 256 weight gradient of 65536 points 84 us against 76).
template <int T, bool KFAST>
struct LsOperand {
  static constexpr int NQ = T / 32;  // quads per thread
  static constexpr int kRowQuads = T / 4;
  static constexpr int kGroups = 256 / kRowQuads;   // row-fast: K groups
  static_assert(kLsK / kGroups == NQ, "row-fast threads take NQ consecutive K");
  f32x4 v[NQ];

  __device__ __forceinline__ void load(const float *src, int ld, int r0, int rows, int k0, int ke) {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int r = r0 + (KFAST ? t / 8 + 32 * i : 4 * (t / kGroups));
      const int k = k0 + (KFAST ? 4 * (t % 8) : (t % kGroups) * NQ + i);
      // the host checked that rows (row-fast) or K (K-fast) is a multiple of 4
      const bool in = r < rows && k < ke;
      const size_t at = KFAST ? static_cast<size_t>(in ? r : 0) * ld + (in ? k : 0)
                              : static_cast<size_t>(in ? k : 0) * ld + (in ? r : 0);
      const f32x4 x = *reinterpret_cast<const f32x4 *>(src + at);
      v[i] = in ? x : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }

  __device__ __forceinline__ void stage(unsigned char *S) const {
    const int t = threadIdx.x;
    constexpr int plane = T * 64;
    if constexpr (KFAST) {
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int row = t / 8 + 32 * i, kq = t % 8;
        const LsSplit a = ls_split(v[i][0], v[i][1]), b = ls_split(v[i][2], v[i][3]);
        unsigned char *d = S + ls_slot<T>(row, kq >> 1) + 8 * (kq & 1);
        *reinterpret_cast<uint2 *>(d) = make_uint2(a.h, b.h);
        *reinterpret_cast<uint2 *>(d + plane) = make_uint2(a.m, b.m);
        *reinterpret_cast<uint2 *>(d + 2 * plane) = make_uint2(a.l, b.l);
      }
    } else {
      const int row0 = 4 * (t / kGroups), k = (t % kGroups) * NQ;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        unsigned char *d = S + ls_slot<T>(row0 + e, k >> 3) + 2 * (k & 7);
        const LsSplit a = ls_split(v[0][e], v[1][e]);
        if constexpr (NQ == 4) {
          const LsSplit b = ls_split(v[2][e], v[3][e]);
          *reinterpret_cast<uint2 *>(d) = make_uint2(a.h, b.h);
          *reinterpret_cast<uint2 *>(d + plane) = make_uint2(a.m, b.m);
          *reinterpret_cast<uint2 *>(d + 2 * plane) = make_uint2(a.l, b.l);
        } else {
          *reinterpret_cast<uint32_t *>(d) = a.h;
          *reinterpret_cast<uint32_t *>(d + plane) = a.m;
          *reinterpret_cast<uint32_t *>(d + 2 * plane) = a.l;
        }
      }
    }
  }
};

__device__ __forceinline__ bool ls_finite(float v) {
  return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u;
}

// Outputs (r, c .. c + 3) over K in [kb, ke): where the split sum in o is not
// finite, the sum of the fp32 products instead. Finite sums had finite parts
// and stay. Rare, so its loop is small rather than fast.
template <int AM, int BT>
__device__ __forceinline__ f32x4 ls_exact(const LwGemmArgs &g, int r, int c, int kb, int ke,
                                          f32x4 o) {
  bool keep[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) keep[e] = ls_finite(o[e]);
  if (keep[0] && keep[1] && keep[2] && keep[3]) return o;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int k = kb; k < ke; ++k) {
    const float a = lw_a<AM>(g, r, k);
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = __builtin_fmaf(a, lw_b<BT>(g, k, c + e), s[e]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = keep[e] ? o[e] : s[e];
  return s;
}

template <int TC, int AM, int BT, int EPI>
__global__ void __launch_bounds__(256, 4) lw_split_kernel(LwGemmArgs g) {
  constexpr int TR = kLsRows;
  constexpr bool kAKFast = AM == kLwARow;
  constexpr int kAPlane = TR * 64, kBPlane = TC * 64;
  constexpr int MR = TR / 32, MC = TC / 32;  // 16 x 16 tiles of a wave's quarter
  __shared__ __align__(16) unsigned char smem[3 * (kAPlane + kBPlane)];
  unsigned char *As = smem, *Bs = smem + 3 * kAPlane;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int p = lane & 15, q = lane >> 4;
  const int wr = (wave & 1) * (TR / 2), wc = (wave >> 1) * (TC / 2);
  const int r0 = blockIdx.x * TR, c0 = blockIdx.y * TC;
  const int rows = g.R - (g.ones_row ? 1 : 0);
  const int kb = blockIdx.z * g.k_chunk;
  const int ke = min(g.K, kb + g.k_chunk);
  f32x4 acc[MR][MC];
#pragma unroll
  for (int i = 0; i < MR; ++i)
#pragma unroll
    for (int j = 0; j < MC; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  LsOperand<TR, kAKFast> a;
  LsOperand<TC, BT != 0> b;
  // bias gradients (ones_row): the column sums of B, by the first row of blocks
  const bool sums = EPI == kLwEpiPartial && g.ones_row && blockIdx.x == 0;
  f32x4 colsum = {0.f, 0.f, 0.f, 0.f};
  auto load = [&](int k0) {
    a.load(g.A, g.lda, r0, rows, k0, ke);
    b.load(g.B, g.ldb, c0, g.C, k0, ke);
  };
  auto stage = [&]() {
    a.stage(As);
    b.stage(Bs);
    if constexpr (EPI == kLwEpiPartial) {
      if (sums)
#pragma unroll
        for (int i = 0; i < TC / 32; ++i) colsum += b.v[i];
    }
  };
  if (kb < ke) {
    load(kb);
    stage();
  }
  __syncthreads();
  for (int k0 = kb; k0 < ke; k0 += kLsK) {
    const bool more = k0 + kLsK < ke;  // uniform over the block
    if (more) load(k0 + kLsK);
    bf16x8 af[MR][3];
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
      for (int s = 0; s < 3; ++s)
        af[i][s] = *reinterpret_cast<const bf16x8 *>(As + s * kAPlane + ls_slot<TR>(wr + 16 * i + p, q));
#pragma unroll
    for (int j = 0; j < MC; ++j) {
      bf16x8 bf[3];
#pragma unroll
      for (int s = 0; s < 3; ++s)
        bf[s] = *reinterpret_cast<const bf16x8 *>(Bs + s * kBPlane + ls_slot<TC>(wc + 16 * j + p, q));
      // a step's five smaller products from zero, smallest first
      constexpr int kSmall[5][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}};
      f32x4 low[MR];
#pragma unroll
      for (int t = 0; t < 5; ++t)
#pragma unroll
        for (int i = 0; i < MR; ++i)
          low[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              bf[kSmall[t][0]], af[i][kSmall[t][1]], t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : low[i], 0,
              0, 0);
#pragma unroll
      for (int i = 0; i < MR; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[0], af[i][0], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MR; ++i) acc[i][j] += low[i];
    }
    __syncthreads();
    if (more) {
      stage();
      __syncthreads();
    }
  }
  // D layout with B as the row operand: lane p + 16 q holds columns 4 q ..
  // 4 q + 3 of row p of each 16 x 16 tile (C is a multiple of 4)
#pragma unroll
  for (int i = 0; i < MR; ++i) {
    const int r = r0 + wr + 16 * i + p;
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < MC; ++j) {
      const int c = c0 + wc + 16 * j + 4 * q;
      if (c >= g.C) continue;
      f32x4 o = ls_exact<AM, BT>(g, r, c, kb, ke, acc[i][j]);
      if constexpr (EPI == kLwEpiHidden) {
        const f32x4 bias = *reinterpret_cast<const f32x4 *>(g.bias + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = fmaxf(o[e] + bias[e], 0.0f);
        *reinterpret_cast<f32x4 *>(g.out + static_cast<size_t>(r) * g.ldo + c) = o;
      } else if constexpr (EPI == kLwEpiMask) {
        const f32x4 m = *reinterpret_cast<const f32x4 *>(g.mask + static_cast<size_t>(r) * g.ldm + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = m[e] > 0.0f ? o[e] : 0.0f;
        *reinterpret_cast<f32x4 *>(g.out + static_cast<size_t>(r) * g.ldo + c) = o;
      } else if constexpr (EPI == kLwEpiScale) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] *= g.scale;
        *reinterpret_cast<f32x4 *>(g.out + static_cast<size_t>(r) * g.ldo + c) = o;
      } else {
        // partial rows start at any float (the layout's odd bias counts)
        float *dst = g.dst + blockIdx.z * g.dst_stride + g.dst_off + static_cast<int64_t>(r) * g.C + c;
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = o[e];
      }
    }
  }
  if constexpr (EPI == kLwEpiPartial) {
    if (!sums) return;  // uniform over the block
    // threads t / kGroups share four columns; K groups in ascending order
    constexpr int kQuads = TC / 4, kGroups = 256 / kQuads;
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);
    __syncthreads();
    red[tid] = colsum;
    __syncthreads();
    if (tid < kQuads && c0 + 4 * tid < g.C) {
      f32x4 t = red[tid * kGroups];
#pragma unroll
      for (int k = 1; k < kGroups; ++k) t += red[tid * kGroups + k];
      float *dst = g.dst + blockIdx.z * g.dst_stride + g.dst_off +
                   static_cast<int64_t>(rows) * g.C + c0 + 4 * tid;
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[e] = t[e];
    }
  }
}

// Whether g runs on lw_split_kernel: operands in rows with 16-byte accesses
// everywhere (the host sets a_vec, b_vec, o_vec) and quads that never straddle
// an edge; the input features' products (X tiles, at most 128 of them) stay on
// lw_gemm_kernel: they are bound by memory (forward) or have too few rows (dW_0
// 32.9 us against 39.6 at 65536 x 16 x 256).
inline bool lw_split_ok(const LwGemmArgs &g) {
  const int rows = g.R - (g.ones_row ? 1 : 0);
  if (g.a_mode != kLwARow && g.a_mode != kLwACol) return false;
  if (!g.a_vec || !g.b_vec || g.C % 4 != 0) return false;
  if ((g.a_mode == kLwARow ? g.K : rows) % 4 != 0 || (g.b_trans != 0 && g.K % 4 != 0)) return false;
  if (g.epi == kLwEpiOutput || (g.epi != kLwEpiPartial && !g.o_vec)) return false;
  return g.C > 16 && g.K >= 96 && rows >= 16;
}

template <int TC>
inline LwGemmFn lw_split_fn_of(const LwGemmArgs &g) {
  if (g.b_trans == 0 && g.a_mode == kLwARow && g.epi == kLwEpiHidden)
    return lw_split_kernel<TC, kLwARow, 0, kLwEpiHidden>;
  if (g.b_trans == 0 && g.a_mode == kLwACol && g.epi == kLwEpiPartial)
    return lw_split_kernel<TC, kLwACol, 0, kLwEpiPartial>;
  if (g.b_trans != 0 && g.a_mode == kLwARow && g.epi == kLwEpiMask)
    return lw_split_kernel<TC, kLwARow, 1, kLwEpiMask>;
  if (g.b_trans != 0 && g.a_mode == kLwARow && g.epi == kLwEpiScale)
    return lw_split_kernel<TC, kLwARow, 1, kLwEpiScale>;
  return nullptr;
}

// The instance and its columns per tile: 128 where that still leaves four
// blocks per CU (steps with 64 / 128 columns, us: 65536 points 256 wide
// 397 / 373, 128 wide 440 / 444; 20000 points 256 wide 198 / 209; fp32 MFMA
// tiles 502, 563, 238).
inline LwGemmFn lw_split_fn(const LwGemmArgs &g, int chunks, int cu_count, int *tc) {
  const int rows = g.R - (g.ones_row ? 1 : 0);
  const int64_t blocks = static_cast<int64_t>((rows + kLsRows - 1) / kLsRows) *
                         ((g.C + 127) / 128) * chunks;
  *tc = blocks >= 4 * cu_count ? 128 : 64;
  return *tc == 128 ? lw_split_fn_of<128>(g) : lw_split_fn_of<64>(g);
}

}  // namespace tmnn_hip
