// Randomized interpolative decomposition with a 128-row sketch: the large
// boxes of the top tree levels (up to kRidBigCols columns, ranks up to
// kRidRowsB - kRidOver), which the 16- to 64-row sketches of rs_rid.hip
// cannot take.  Same sketch and outputs as there.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rs_device.hpp"
#include "rs_id.hpp"
#include "rs_kernels.hpp"

namespace iegpu {

namespace {

// ---------------------------------------------------------------------------
// Few boxes of a level are these (4 on level 1, a few on the next), each
// with the most rows and columns of the tree, and every level above waits
// for them: a box's sketch is spread over a workgroup per 64 columns and
// row part (kRidBigParts), its QR takes one workgroup.
//
// k_rid_big_sketch: the part's row points (every kRidBigParts-th block of
// four) times Omega into eight 16-row MFMA tiles per wave, the partial
// sketch to the box's scratch.
//
// k_rid_big_qr: column-pivoted Householder QR of the summed sketch in
// registers.  Thread (q, c) of 4 x 128 holds rows 4 i + q of columns c and
// c + 128, shifted so that the quarter's next row is register 0; row j of R
// leaves quarter j % 4 at step j.  (One column per thread on 1024 threads
// read the pivot column from LDS twice per step in 16 waves, 4.9 us a step;
// here eight waves read it once and keep it.)  Three barriers per step: column norms (every
// wave then finds the pivot itself), the pivot column, partial dots.  T =
// R11^{-1} R12 by back substitution, four lanes per column.
//
// Bound by the latency of the QR's steps (2.9 us each with three barriers).
// Stokes, 16,385 points, levels 1 and 2 (boxes of 107 to 152 DOFs, about 900
// and 2,000 ID rows, ranks up to 99): 38 + 356 us a level, against 7,263 and
// 6,175 us for the full pivoted QR of their matrices in k_qrcp.
// ---------------------------------------------------------------------------

template <typename R, int PDE>
__global__ __launch_bounds__(256, 2) void k_rid_big_sketch(DevGeom g, DevTree t, DevState s,
                                                           int start, int level) {
  using V4 = typename Mfma16<R>::V4;
  constexpr int TR = kRidMaxNearW + kNumProxy;
  __shared__ double tab[6][TR];
  __shared__ int rowdofs[kRidMaxNearW];
  if (!pools_ok(s)) return;
  const int nl = list_count(s, level, kLstRidBig);
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  const int part = blockIdx.z;
  for (int li = blockIdx.x; li < nl; li += gridDim.x) {
    const int b = list_at(s, start, kLstRidBig, li);
    const int n = s.act_cnt[b], m = s.m_rows[b];
    if (64 * (int)blockIdx.y >= n) continue;
    const int n16 = (n + 15) / 16 * 16;
    const int P = proxy_rows(g, level) / 2;  // rows per proxy block
    const int cnt = (m - 2 * P) / 2;
    __syncthreads();  // the previous box's table
    if (wv == 0)
      for_each_row_dof(g, t, s, b, level >= 3, [&](int pos, int dof) { rowdofs[pos] = dof; });
    if (level >= 3 && tid < kNumProxy) {
      double px, py, n1, n2;
      proxy_point(t.cx[b], t.cy[b], t.side[b] * kRadiusRatio, tid, &px, &py, &n1, &n2);
      const double pw = proxy_weight(t, b);
      const DofGeo d = pair_geo<PDE>(DofGeo{px, py, n1, n2, pw, 0, 0});
      tab[0][cnt + tid] = px;
      tab[1][cnt + tid] = py;
      tab[2][cnt + tid] = d.n1;
      tab[3][cnt + tid] = d.n2;
      tab[4][cnt + tid] = pw;
      tab[5][cnt + tid] = 0;
    }
    __syncthreads();
    for (int i = tid; i < cnt; i += 256) {
      const DofGeo d = pair_geo<PDE>(dof_geo(g, rowdofs[i]));
      tab[0][i] = d.x;
      tab[1][i] = d.y;
      tab[2][i] = d.n1;
      tab[3][i] = d.n2;
      tab[4][i] = d.w;
      tab[5][i] = d.k;
    }
    __syncthreads();
    const int kq = lane >> 4;
    const int c = 64 * blockIdx.y + 16 * wv + (lane & 15);
    if (c - (lane & 15) >= n16) continue;
    const int* act = s.act_list + (int64_t)b * s.ncap;
    const DofGeo cg = pair_geo<PDE>(dof_geo(g, act[min(c, n - 1)]));
    V4 acc[8];
#pragma unroll
    for (int q = 0; q < 8; q++) acc[q] = V4{0, 0, 0, 0};
    sketch_pairs<R, PDE, true, 8, kRidRowsB, 1, false>(tab, rowdofs, s.omega_b, cnt, 0, cnt, 0,
                                                       part, kRidBigParts, cg, acc);
    sketch_pairs<R, PDE, false, 8, kRidRowsB, 1, false>(tab, rowdofs, s.omega_b, P, 2 * cnt,
                                                        2 * cnt + P, cnt, part, kRidBigParts, cg,
                                                        acc);
    R* Y = reinterpret_cast<R*>(s.id_pool) + s.big_off[b] + (int64_t)part * kRidRowsB * n16;
#pragma unroll
    for (int q = 0; q < 8; q++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        Y[(int64_t)(16 * q + Mfma16<R>::row(kq, v)) * n16 + c] = acc[q][v];
  }
}

constexpr int kBigNT = 512;
constexpr int kBigKmax = kRidRowsB - kRidOver;
constexpr int kBigLd = kBigKmax + 2;  // columns of R11 in LDS

template <typename R>
struct RidBigLds {
  alignas(16) R vb[4][kRidRowsB / 4];  // the pivot column, by quarter
  R pn[4][kRidBigCols];                // partial norms (-1: taken)
  R pd[4][kRidBigCols];                // partial dots
  int spiv[kRidRowsB];                 // pivot column of each step
  int rcol[kRidBigCols];               // redundant columns in order
  int wcnt[4];
  R rdiag[kBigKmax];
  R r11[kBigKmax * kBigLd + 8];        // R11, zero below the diagonal
};

// QR of a box's sketch with NC columns per thread; the rank, -1 when no
// cut shows.  All threads; avail[h] says whether column c0 + 128 h is left.
template <typename R, int NC>
__device__ __forceinline__ int big_qr(RidBigLds<R>& sh, const R* Y, R* rr, int n, R tol,
                                      bool (&avail)[2]) {
  constexpr int L = kRidRowsB, NR = L / 4;
  const int n16 = (n + 15) / 16 * 16;
  const int tid = threadIdx.x, lane = tid & 63, q = wave_id() >> 1, c0 = tid & 127;
  R y[NC][NR], nq[NC];
  auto norm = [&](int h) {
    R a[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NR; i++) a[i & 3] += y[h][i] * y[h][i];
    nq[h] = (a[0] + a[1]) + (a[2] + a[3]);
  };
#pragma unroll
  for (int h = 0; h < NC; h++) {
    const int c = c0 + 128 * h;
#pragma unroll
    for (int i = 0; i < NR; i++) y[h][i] = R(0);
#pragma unroll 1
    for (int p = 0; p < kRidBigParts; p++) {
      const R* yp = Y + (int64_t)(p * L + q) * n16 + min(c, n - 1);
#pragma unroll
      for (int i = 0; i < NR; i++) y[h][i] += c < n ? yp[(int64_t)4 * i * n16] : R(0);
    }
    norm(h);
  }
  R thresh = 0;
  const int jlim = min(n, kBigKmax);
  for (int j = 0; j < jlim; j++) {
#pragma unroll
    for (int h = 0; h < NC; h++) sh.pn[q][c0 + 128 * h] = avail[h] ? nq[h] : R(-1);
    __syncthreads();
    double key = -1.0;
#pragma unroll
    for (int h = 0; h < 2 * NC; h++) {
      const int cc = lane + 64 * h;
      const R v0 = sh.pn[0][cc];
      const R v = (v0 + sh.pn[1][cc]) + (sh.pn[2][cc] + sh.pn[3][cc]);
      key = fmax(key, v0 >= R(0) ? pivot_key<R, 8>(v, cc) : -1.0);
    }
    const double best = wave_max(key);
    if (!(best >= 0)) return -1;  // no usable column left (norms not finite)
    const int p = pivot_key_pos<8>(best);
    const int jq = j & 3;
#pragma unroll
    for (int h = 0; h < NC; h++)
      if (c0 + 128 * h == p) {
#pragma unroll
        for (int i = 0; i < NR; i++) sh.vb[q][i] = y[h][i];
      }
    __syncthreads();
    const R* v = &sh.vb[0][0];
    const R alpha = sh.vb[jq][0];
    const R a0 = lane == NR * jq ? R(0) : v[lane];
    const R a1 = lane + 64 == NR * jq ? R(0) : v[lane + 64];
    R beta, tau, sc;
    householder_scalars(alpha, wave_total(a0 * a0 + a1 * a1), &beta, &tau, &sc);
    if (j == 0) thresh = fabs(tol * beta);
    else if (sketch_diag<true>(beta, L, j) < thresh) return j;
    if (tid == 0) sh.spiv[j] = p;
    // the pivot column's rows of the quarter, eight at a time (all 32 do not
    // fit the registers beside two columns)
    const R* vq = sh.vb[q];
    R d[NC][2];
#pragma unroll
    for (int h = 0; h < NC; h++) d[h][0] = d[h][1] = R(0);
#pragma unroll
    for (int i0 = 0; i0 < NR; i0 += 8) {
      R w[8];
#pragma unroll
      for (int i = 0; i < 8; i++) w[i] = vq[i0 + i];
      if (i0 == 0) w[0] = q == jq ? R(0) : w[0];  // row j: its own term below
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int h = 0; h < NC; h++) d[h][i & 1] += w[i] * y[h][i0 + i];
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int h = 0; h < NC; h++) {
      if (c0 + 128 * h == p) avail[h] = false;
      sh.pd[q][c0 + 128 * h] = (q == jq ? y[h][0] : R(0)) + sc * (d[h][0] + d[h][1]);
    }
    __syncthreads();
    R ws[NC];
#pragma unroll
    for (int h = 0; h < NC; h++) {
      const int c = c0 + 128 * h;
      const R w = tau * ((sh.pd[0][c] + sh.pd[1][c]) + (sh.pd[2][c] + sh.pd[3][c]));
      ws[h] = w * sc;
      if (q == jq && c < n) rr[(int64_t)j * n16 + c] = c == p ? beta : y[h][0] - w;
      d[h][0] = d[h][1] = R(0);
    }
    const bool up = q == jq;  // row j left this quarter: its rows shift up
#pragma unroll
    for (int i0 = 0; i0 < NR; i0 += 8) {
      R w[9];
#pragma unroll
      for (int i = 0; i < 9; i++) w[i] = i0 + i < NR ? vq[i0 + i] : R(0);
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int h = 0; h < NC; h++) {
          const R nxt = i0 + i + 1 < NR ? y[h][i0 + i + 1] : R(0);
          const R v = up ? nxt - ws[h] * w[i + 1] : y[h][i0 + i] - ws[h] * w[i];
          y[h][i0 + i] = v;
          d[h][i & 1] += v * v;
        }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int h = 0; h < NC; h++) nq[h] = d[h][0] + d[h][1];
  }
  return jlim == n ? n : -1;  // every column taken: nothing redundant
}

template <typename R>
__global__ __launch_bounds__(kBigNT) void k_rid_big_qr(DevState s, int start, int level,
                                                       double tol_d) {
  constexpr int L = kRidRowsB, NR = L / 4;
  static_assert(NR == 32 && kRidBigCols == 256 && kBigNT == 512, "4 x 128 threads");
  typedef R V16 __attribute__((ext_vector_type(16)));
  __shared__ RidBigLds<R> sh;
  if (!pools_ok(s)) return;
  const int nl = list_count(s, level, kLstRidBig);
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  for (int li = blockIdx.x; li < nl; li += gridDim.x) {
    const int b = list_at(s, start, kLstRidBig, li);
    const int n = s.act_cnt[b];
    const int n16 = (n + 15) / 16 * 16;
    const R* Y = reinterpret_cast<const R*>(s.id_pool) + s.big_off[b];
    R* rr = reinterpret_cast<R*>(s.id_pool) + s.big_off[b] + (int64_t)kRidBigParts * L * n16;
    bool avail[2] = {(tid & 127) < n, (tid & 127) + 128 < n};
    const int k = n > 128 ? big_qr<R, 2>(sh, Y, rr, n, static_cast<R>(tol_d), avail)
                          : big_qr<R, 1>(sh, Y, rr, n, static_cast<R>(tol_d), avail);
    __syncthreads();
    if (k < 0) {  // no cut within the sketch: the full QRCP takes the box
      if ((s.qkind[b] == kQrcpReg || s.qkind[b] == kQrcpStack) && tid == 0) {
        const int pos = atomicAdd(list_slot(s, level, kLstFallback), 1);
        s.lists[(int64_t)kLstFallback * s.nbox + start + pos] = b;
      }
      continue;
    }
    // redundant columns in order: waves 0 and 1 hold 64 columns of either half
    uint64_t mask[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      mask[h] = __ballot(avail[h]);
      if (wv < 2 && lane == 0) sh.wcnt[2 * h + wv] = __popcll(mask[h]);
    }
    for (int e = tid; e < k * kBigLd; e += kBigNT) {
      const int i = e % kBigLd, p = e / kBigLd;
      sh.r11[e] = i <= p ? rr[(int64_t)i * n16 + sh.spiv[p]] : R(0);
    }
    __syncthreads();
    if (tid < k) sh.rdiag[tid] = recip_any(sh.r11[tid + kBigLd * tid]);
    if (wv < 2)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        int cp = __popcll(mask[h] & ((1ull << lane) - 1));
        for (int w = 0; w < 2 * h + wv; w++) cp += sh.wcnt[w];
        if (avail[h]) sh.rcol[cp] = (tid & 127) + 128 * h;
      }
    __syncthreads();
    // T = R11^{-1} R12: four lanes per column, lane sub holding rows 4 i +
    // sub; every step subtracts its whole column of R11 (zeros below the
    // diagonal; rows past k are never used).
    const int r = n - k, sub = tid & 3;
    const int* act = s.act_list + (int64_t)b * s.ncap;
    R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
    for (int w0 = 16 * wv; w0 < r; w0 += 16 * (kBigNT / 64)) {
      const int col = w0 + (lane >> 2);
      V16 x[2];
      const int cc = sh.rcol[min(col, r - 1)];
#pragma unroll
      for (int i = 0; i < NR; i++)
        x[i >> 4][i & 15] = 4 * i + sub < k ? rr[(int64_t)(4 * i + sub) * n16 + cc] : R(0);
#pragma unroll
      for (int hi = 1; hi >= 0; hi--) {
        for (int st = min(k, 64 * hi + 64) - 1; st >= 64 * hi; st--) {
          const int i0 = (st >> 2) & 15;
          const R xv = x[hi][i0];
          const R tq = __shfl(xv, (lane & ~3) | (st & 3), 64) * sh.rdiag[st];
          const R* cl = sh.r11 + kBigLd * st + sub;
#pragma unroll
          for (int i = 0; i < NR; i++) {
            if (i >= 16 && hi == 0) break;
            x[i >> 4][i & 15] -= cl[4 * i] * tq;
          }
          x[hi][i0] = sub == (st & 3) ? tq : x[hi][i0];
        }
      }
      if (col < r)
#pragma unroll
        for (int i = 0; i < NR; i++)
          if (4 * i + sub < k) F[4 * i + sub + (int64_t)k * col] = x[i >> 4][i & 15];
    }
    int* out = s.out_list + (int64_t)b * s.ncap;
    int* rl = s.red_list + (int64_t)b * s.ncap;
    int* pm = s.perm + (int64_t)b * s.ncap;
    for (int i = tid; i < n; i += kBigNT) {
      const int cc = i < k ? sh.spiv[i] : sh.rcol[i - k];
      pm[i] = cc;
      if (i < k) out[i] = act[cc];
      else rl[i - k] = act[cc];
    }
    if (tid == 0) {
      s.rank[b] = k;
      s.out_cnt[b] = k;
      s.rid_done[b] = 1;
    }
    __syncthreads();  // the next box reuses the LDS
  }
}

constexpr int kBigGrid = 256;  // boxes of the list in flight

}  // namespace

template <typename R>
void launch_rid_big(const DevGeom& g, const DevTree& t, const DevState& s, int start, int level,
                    int listed, double tol, hipStream_t st) {
  const int nb = listed < kBigGrid ? listed : kBigGrid;
  const dim3 grid(nb, kRidBigCols / 64, kRidBigParts);
  if (g.pde == kPdeStokes)
    k_rid_big_sketch<R, kPdeStokes><<<grid, 256, 0, st>>>(g, t, s, start, level);
  else if (g.pde == kPdeLaplaceNeumann)
    k_rid_big_sketch<R, kPdeLaplaceNeumann><<<grid, 256, 0, st>>>(g, t, s, start, level);
  else
    k_rid_big_sketch<R, kPdeLaplace><<<grid, 256, 0, st>>>(g, t, s, start, level);
  k_rid_big_qr<R><<<nb, kBigNT, 0, st>>>(s, start, level, tol);
}

template void launch_rid_big<double>(const DevGeom&, const DevTree&, const DevState&, int, int,
                                     int, double, hipStream_t);
template void launch_rid_big<float>(const DevGeom&, const DevTree&, const DevState&, int, int,
                                    int, double, hipStream_t);

}  // namespace iegpu
