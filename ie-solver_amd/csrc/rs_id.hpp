// Device helpers shared by the interpolative-decomposition kernels
// (rs_kernels.hip, rs_qrcp.hip, rs_rid.hip, rs_rid_big.hip, rs_gram.hip): ID
// rows, Householder scalars, MFMA tiles, sketches.
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

// |R_jj| of a sketch of l rows at step j as the rank cut takes it (against
// tol |R_00|).  The sketch keeps l - j dimensions, which shrinks |R_jj| by
// about sqrt((l - j) / l) against |R_00|, and the factor 2 is a margin.
// FULL: T from a sketch near its last rows carries the first column left
// out enlarged by about sqrt(l / (l - j)) (Halko, Martinsson & Tropp 2011,
// sec. 10), so that factor once more.  The 64- and 128-row sketches reach
// ranks of 58 and 122 with six rows to spare: without it Stokes stars of
// 1,000 to 16,385 points came out 3 to 25 % further off than with the full
// QR for those boxes (means of 16 seeds), with it 34 to 41 % closer, for 1 %
// more ranks in the same time.
template <bool FULL, typename R>
__device__ inline R sketch_diag(R beta, int l, int j) {
  const R q = static_cast<R>(l) / static_cast<R>(l - j);
  return 2 * fabs(beta) * (FULL ? q : sqrt(q));
}

// A point as pair_entries takes it: for Laplace the normal scaled by w / (2
// pi), so that an entry is one product.
template <int PDE>
__device__ inline DofGeo pair_geo(DofGeo d) {
  if constexpr (PDE == kPdeLaplace) {
    const double s = d.w * (1.0 / (2 * M_PI));
    d.n1 *= s;
    d.n2 *= s;
  }
  return d;
}

// Entries of row point q and column c in both directions, et = K(q, c) and
// es = K(c, q) (the kernels of rs_device.hpp): they share r, |r|^2 and its
// reciprocal, which are most of an entry's arithmetic.  NEAR: boundary DOFs,
// which may coincide.
template <int PDE, bool NEAR>
__device__ __forceinline__ void pair_entries(const DofGeo& q, const DofGeo& c, double& et,
                                             double& es) {
  const double r0 = q.x - c.x, r1 = q.y - c.y;
  const double inv = recip(fma(r0, r0, r1 * r1));
  const double rc = fma(r0, c.n1, r1 * c.n2), rq = fma(r0, q.n1, r1 * q.n2);
  if constexpr (PDE == kPdeStokes) {
    const double tn = q.c ? q.n2 : q.n1, cn = c.c ? c.n2 : c.n1;
    const double rr = (q.c ? r1 : r0) * (c.c ? r1 : r0) * (inv * inv) * (1.0 / M_PI);
    et = c.w * fma(rc, rr, tn * cn);
    es = q.w * fma(-rq, rr, tn * cn);
  } else if constexpr (PDE == kPdeLaplaceNeumann) {
    const double s = inv * (1.0 / (2 * M_PI));
    et = c.w * fma(rq, s, 1.0);
    es = q.w * fma(-rc, s, 1.0);
  } else {
    et = -rc * inv;
    es = rq * inv;
  }
  if (NEAR && r0 == 0 && r1 == 0) {  // the source's diagonal value
    if constexpr (PDE == kPdeLaplace) {
      const double h = 0.25 / M_PI;
      et = fma(h * c.k, c.w, 0.5);
      es = fma(h * q.k, q.w, 0.5);
    } else {
      et = kernel_entry(PDE, q, c, true);
      es = kernel_entry(PDE, c, q, true);
    }
  }
}

// Sketch of one part of a box's ID matrix: row points 0 .. items - 1 (NEAR:
// near DOFs; else proxy rows), whose entries with the box as source are ID
// rows trow + i and as target srow + i, times Omega (ld LD) into NQ 16-row
// tiles.  The lane's column is cg; row geometry (pair_geo) comes from the LDS
// table at idx0 + i (>> 1 for the proxy rows of Stokes).  Blocks of 4 U
// points part, part + parts, ...; the next block's Omega operands are loaded
// before this block's entries when AHEAD.  Points past the end carry zero
// Omega; the tiles of columns past the box's are never read.
// An entry pair's arithmetic is 40% less than two entries'; the MFMAs (64
// cycles for a 16 x 16 x 4 product in FP64) then bound the large levels.
// Learned widths, 262,144 points: k_rid 1430 us per factorization with one
// direction at a time, 1264 with both; Stokes, 16,385 points: k_rid_wide
// 2.1 and 1.9 ms.
template <typename R, int PDE, bool NEAR, int NQ, int LD, int U, bool AHEAD, int TR>
__device__ __forceinline__ void sketch_pairs(const double (*tab)[TR], const int* rowdofs,
                                             const double* omega, int items, int trow, int srow,
                                             int idx0, int part, int parts, const DofGeo& cg,
                                             typename Mfma16<R>::V4 (&acc)[NQ]) {
  constexpr bool stokes = PDE == kPdeStokes;
  const int lane = threadIdx.x & 63, cl = lane & 15, kq = lane >> 4;
  const int step = 4 * U * parts;
  if (4 * U * part >= items) return;
  auto load_omega = [&](int i0, R (&w)[U][2][NQ]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + 4 * u + kq, ic = min(i, items - 1);
      const double* ot = omega + (int64_t)(trow + ic) * LD + cl;
      const double* os = omega + (int64_t)(srow + ic) * LD + cl;
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        w[u][0][q] = i < items ? static_cast<R>(ot[16 * q]) : R(0);
        w[u][1][q] = i < items ? static_cast<R>(os[16 * q]) : R(0);
      }
    }
  };
  R nw[U][2][NQ];
  if (AHEAD) load_omega(4 * U * part, nw);
  for (int i0 = 4 * U * part; i0 < items; i0 += step) {
    R w[U][2][NQ];
    if (AHEAD) {
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int q = 0; q < NQ; q++) {
          w[u][0][q] = nw[u][0][q];
          w[u][1][q] = nw[u][1][q];
        }
      if (i0 + step < items) load_omega(i0 + step, nw);
    } else {
      load_omega(i0, w);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = min(i0 + 4 * u + kq, items - 1);
      const int idx = idx0 + ((stokes && !NEAR) ? i >> 1 : i);
      DofGeo rg;
      rg.x = tab[0][idx];
      rg.y = tab[1][idx];
      rg.n1 = tab[2][idx];
      rg.n2 = tab[3][idx];
      rg.w = tab[4][idx];
      rg.k = tab[5][idx];
      rg.c = stokes ? (NEAR ? rowdofs[i] & 1 : i & 1) : 0;
      double et, es;
      pair_entries<PDE, NEAR>(rg, cg, et, es);
      const R a = static_cast<R>(et), b = static_cast<R>(es);
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        acc[q] = mfma16x16x4(w[u][0][q], a, acc[q]);
        acc[q] = mfma16x16x4(w[u][1][q], b, acc[q]);
      }
    }
  }
}

}  // namespace iegpu
