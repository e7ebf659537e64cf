// Device helpers shared by the interpolative-decomposition kernels
// (rs_kernels.hip, rs_rid_big.hip): ID rows, Householder scalars, MFMA tiles.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rs_device.hpp"

namespace iegpu {

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Visits the ID row DOFs of box b in reference order (source boxes in
// order, each list in order, filtered by the proxy circle at level >= 3).
// Called by one full wave; `emit(pos, dof)` receives the compacted index.
template <typename F>
__device__ inline int for_each_row_dof(const DevGeom& g, const DevTree& t,
                                const DevState& s, int b, bool filter,
                                F emit) {
  const int lane = threadIdx.x & 63;
  const double cx = t.cx[b], cy = t.cy[b], side = t.side[b];
  int cnt = 0;
  const int so = t.src_off[b], sc = t.src_cnt[b];
  for (int u = 0; u < sc; u++) {
    const DofList L = source_dofs(t, s, t.src[so + u]);
    for (int base = 0; base < L.n; base += 64) {
      const int i = base + lane;
      int dof = -1;
      bool keep = false;
      if (i < L.n) {
        dof = L.p[i];
        keep = !filter || in_proxy_circle(g, dof, cx, cy, side);
      }
      const uint64_t mask = __ballot(keep);
      const uint64_t below = (lane == 0) ? 0ull : (mask & ((~0ull) >> (64 - lane)));
      if (keep) emit(cnt + __popcll(below), dof);
      cnt += __popcll(mask);
    }
  }
  return cnt;
}

__device__ inline int proxy_rows(const DevGeom& g, int level) {
  if (level < 3) return 0;
  return (g.pde == kPdeStokes) ? 4 * kNumProxy : 2 * kNumProxy;
}

// Row DOFs and proxy points of box b into LDS (all threads; the caller
// synchronises).  Returns the number of row DOFs (cnt).
__device__ inline int id_setup(const DevGeom& g, const DevTree& t, const DevState& s,
                               int b, int level, int m, int* rows,
                               double (*pxy)[kNumProxy]) {
  const int tid = threadIdx.x;
  if (tid < 64)
    for_each_row_dof(g, t, s, b, level >= 3, [&](int pos, int dof) { rows[pos] = dof; });
  if (level >= 3 && tid < kNumProxy) {
    double px, py, n1, n2;
    proxy_point(t.cx[b], t.cy[b], t.side[b] * kRadiusRatio, tid, &px, &py, &n1, &n2);
    pxy[0][tid] = px;
    pxy[1][tid] = py;
    pxy[2][tid] = n1;
    pxy[3][tid] = n2;
  }
  return (m - proxy_rows(g, level)) / 2;
}

__device__ inline double proxy_weight(const DevTree& t, int b) {
  return 2.0 * M_PI * (t.side[b] * kRadiusRatio) / kNumProxy;
}

// LAPACK dlarfg on (alpha, x) with ||x||^2 = xn2: beta = -sign(alpha)
// ||(alpha, x)||, tau = (beta - alpha) / beta, scale 1 / (alpha - beta).
// (The ID matrices hold moderate entries, so ||(alpha, x)|| is formed
// directly rather than through dlapy2's scaling, and the two quotients use
// independent reciprocals.)
template <typename R>
__device__ inline R recip_any(R d) {
  if constexpr (sizeof(R) == 8) return recip(d);
  else return R(1) / d;
}
template <typename R>
__device__ inline void householder_scalars(R alpha, R xn2, R* beta, R* tau, R* sc) {
  if (xn2 == 0) {
    *tau = 0;
    *beta = alpha;
    *sc = 0;
  } else {
    *beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
    *tau = (*beta - alpha) * recip_any(*beta);
    *sc = recip_any(alpha - *beta);
  }
}

// Output layout of the 16x16x4 MFMAs: lane l, element v holds D(i, l % 16)
// with i = l / 16 + 4 v (f64) or 4 (l / 16) + v (f32).
template <typename R>
struct Mfma16 {
  typedef R V4 __attribute__((ext_vector_type(4)));
  __device__ static int row(int q, int v) { return sizeof(R) == 8 ? q + 4 * v : 4 * q + v; }
};
__device__ inline Mfma16<double>::V4 mfma16x16x4(double a, double b, Mfma16<double>::V4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline Mfma16<float>::V4 mfma16x16x4(float a, float b, Mfma16<float>::V4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

}  // namespace iegpu
