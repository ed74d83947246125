// grad_kernel.hpp -- position gradient of the field (FieldEvaluator::
// evaluate_with_gradient): given dx = d out_m / d(features) of every point
// (the fused kernel in kModeInputGrad), accumulate
//   d out_m / d pos_a += (dx[l][f] * r_l) * d feat_{l,f} / d frac_a
// over levels l (outer) and features f, with the reference's derivative forms
// (neural_sdf_analytical_eval_gradient_points, mlp_kernel_emitter.cpp:
// 1865-2090): the lerp form of trilinear_feature_grad (:1677-1704) in 3D and
// for the lifted 2D points (fz = 0: the z = 1 terms vanish exactly), the
// product loops (:2034-2056) in 4D.
#pragma once

#include "aux_kernels.hpp"
#include "device_common.hpp"

namespace tmnn_hip {

struct PosGradArgs {
  int32_t n, L, F, M, m;      // points, levels, features/level, outputs, this output
  uint32_t log2T;
  float res[kMaxLevels];
  const float *pos;           // [n][D]
  const float *table;         // [L][T][F]
  const float *dx;            // [n][L*F]
  float *grads;               // [n][M][D]
};

// d feat / d frac of one feature from its corner values cv[corner]
// (corner_of's order: bit a of the index is axis a's upper corner).
template <int D>
__device__ __forceinline__ void frac_grad(const float (&fr)[D], const float (&cv)[1 << D],
                                          float (&g)[D]) {
  const float fx = fr[0], fy = fr[1];
  if constexpr (D == 2) {
    g[0] = (1.0f - fy) * (cv[1] - cv[0]) + fy * (cv[3] - cv[2]);
    g[1] = (1.0f - fx) * (cv[2] - cv[0]) + fx * (cv[3] - cv[1]);
  } else if constexpr (D == 3) {
    const float fz = fr[2];
    g[0] = (1.0f - fz) * ((1.0f - fy) * (cv[1] - cv[0]) + fy * (cv[3] - cv[2])) +
           fz * ((1.0f - fy) * (cv[5] - cv[4]) + fy * (cv[7] - cv[6]));
    g[1] = (1.0f - fz) * ((1.0f - fx) * (cv[2] - cv[0]) + fx * (cv[3] - cv[1])) +
           fz * ((1.0f - fx) * (cv[6] - cv[4]) + fx * (cv[7] - cv[5]));
    g[2] = (1.0f - fy) * ((1.0f - fx) * (cv[4] - cv[0]) + fx * (cv[5] - cv[1])) +
           fy * ((1.0f - fx) * (cv[6] - cv[2]) + fx * (cv[7] - cv[3]));
  } else {
    // per axis, over the eight corners of the others (w outermost)
    auto w = [&](int d, int axis) { return d == 0 ? (1.0f - fr[axis]) : fr[axis]; };
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      g[a] = 0.0f;
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        float wt = 1.0f;
        int lo = 0, bit = 0;
        bool first = true;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (k == a) continue;
          const int d = (m >> bit) & 1;
          ++bit;
          lo |= d << k;
          wt = first ? w(d, k) : wt * w(d, k);
          first = false;
        }
        g[a] += wt * (cv[lo | (1 << a)] - cv[lo]);
      }
    }
  }
}

// One thread per point and level (the levels of a point on neighbouring
// lanes), whose terms meet in LDS and are added in the reference's order,
// level then feature, by one thread per point and axis. One thread per point
// walked its levels' dependent gathers in turn, 16 blocks at 4096 points:
// 48.4 us there (3D, 16x2, T = 2^19), all of it latency; the whole
// evaluate_with_gradient call went 113.8 -> 72.7 us.
constexpr int kPosGradThreads = 256;

template <int D, int F>
__global__ void __launch_bounds__(kPosGradThreads) pos_grad_kernel(PosGradArgs a, int log2L) {
  __shared__ float terms[D][F][kPosGradThreads];
  const int Lp = 1 << log2L;  // levels rounded up to a power of two
  const int points = kPosGradThreads >> log2L;
  const int first = static_cast<int>(blockIdx.x) * points;
  const int l = static_cast<int>(threadIdx.x) & (Lp - 1);
  const int i = first + (static_cast<int>(threadIdx.x) >> log2L);
  if (i < a.n && l < a.L) {
    float p[D];
#pragma unroll
    for (int k = 0; k < D; ++k) p[k] = a.pos[static_cast<size_t>(i) * D + k];
    const float r = a.res[l];
    const Cell<D> c = cell_of<D>(p, r);
    const float *level = a.table + (static_cast<size_t>(l) << a.log2T) * F;
    float cv[1 << D][F];
#pragma unroll
    for (int k = 0; k < (1 << D); ++k) {
      int co[D];
#pragma unroll
      for (int x = 0; x < D; ++x) co[x] = c.bc[x] + ((k >> x) & 1);
      load_vec<F>(level + static_cast<size_t>(hash_corner<D>(co, (1u << a.log2T) - 1u)) * F, cv[k]);
    }
    float d[F];
    load_vec<F>(a.dx + (static_cast<size_t>(i) * a.L + l) * F, d);
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const float s = d[f] * r;
      float v[1 << D], g[D];
#pragma unroll
      for (int k = 0; k < (1 << D); ++k) v[k] = cv[k][f];
      frac_grad<D>(c.fr, v, g);
#pragma unroll
      for (int k = 0; k < D; ++k) terms[k][f][threadIdx.x] = s * g[k];
    }
  }
  __syncthreads();
  for (int t = static_cast<int>(threadIdx.x); t < points * D; t += kPosGradThreads) {
    const int pt = t / D, k = t % D;
    if (first + pt >= a.n) break;
    float gp = 0.0f;
    for (int lv = 0; lv < a.L; ++lv)
#pragma unroll
      for (int f = 0; f < F; ++f) gp = gp + terms[k][f][(pt << log2L) + lv];
    a.grads[(static_cast<size_t>(first + pt) * a.M + a.m) * D + k] = gp;
  }
}

}  // namespace tmnn_hip
