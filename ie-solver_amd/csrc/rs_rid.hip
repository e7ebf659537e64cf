// Randomized interpolative decomposition with 16- to 64-row Gaussian
// sketches on the matrix cores (stands in for ie_mat.cpp:548-588 when
// selected), and the sketches' Gaussian tables.

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "rs_device.hpp"
#include "rs_id.hpp"
#include "rs_kernels.hpp"

namespace iegpu {

namespace {

// ---------------------------------------------------------------------------
// Randomized interpolative decomposition.  The sketch Y = Omega A (l x n,
// l = sk_w[b] in {16, 32}) is formed on the matrix cores: A's entries are
// evaluated straight into the B operand of v_mfma_{f64,f32}_16x16x4 (lane:
// row k0 + lane / 16, column lane % 16 of a 16-column tile) and Omega, a
// fixed Gaussian table indexed by the ID row, is the A operand.  Y moves
// through LDS to one column per lane and is factored by column-pivoted
// Householder QR with the reference's rank rule (ie_mat.cpp:561-568)
// applied to the sketch, |R_jj| corrected for the dimensions the sketch
// has left; T = R11^{-1} R12 of the sketch is the ID of A (Halko,
// Martinsson & Tropp 2011, sec. 5.2).  A box whose sketch shows no cut
// within l - kRidOver pivots leaves rid_done = 0 and the full QRCP kernels
// take it.
// ---------------------------------------------------------------------------

// One workgroup (4 waves) per box.  The box's row geometry (near DOFs,
// then the proxy circle) is staged in LDS; wave w sketches the 16-column
// tile w (n <= 64) over the near DOFs, then the proxy circle, both directions
// of an entry at once (sketch_pairs).  The tiles of Y go to LDS, and
// wave 0 alone runs the pivoted QR of Y, the other waves ending there.
// QR layout: lane c holds column c's active rows, shifted so that the
// step's row is always register 0; row j of R leaves the registers for
// LDS (rr[j][c]) at step j, where the T solve finds R11 and R12.  The
// pivot column reaches every lane through readlane (uniform registers),
// not LDS: 93 registers, five workgroups per CU.
template <typename R, int PDE>
__global__ __launch_bounds__(256, 5) void k_rid(DevGeom g, DevTree t, DevState s, int start,
                                             int level, double tol_d) {
  constexpr int LM = kRidRows, YLD = 65, TR = kRidMaxNear + kNumProxy;
  using V4 = typename Mfma16<R>::V4;
  // Row geometry x, y, n1, n2, w, k during the sketch; Y (row-major, ld
  // YLD), then the rows of R, afterwards.
  __shared__ double tab[6][TR];
  __shared__ int rowdofs[kRidMaxNear];
  __shared__ int spiv[64];  // pivot column (lane) of each step
  static_assert(LM * YLD * sizeof(R) <= sizeof(tab), "Y fits the row table");
  R* ybuf = reinterpret_cast<R*>(&tab[0][0]);
  if (!pools_ok(s)) return;
  if ((int)blockIdx.x >= list_count(s, level, kLstRid)) return;
  const int b = list_at(s, start, kLstRid, blockIdx.x);
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  const int n = s.act_cnt[b], m = s.m_rows[b], l = s.sk_w[b];
  const int P = proxy_rows(g, level) / 2;  // rows per proxy block
  const int cnt = (m - 2 * P) / 2;
  const int* act = s.act_list + (int64_t)b * s.ncap;
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

  // Sketch: wave wv takes columns 16 wv .. 16 wv + 15.
  const int kq = lane >> 4;
  const int c = 16 * wv + (lane & 15);
  V4 acc[2] = {V4{0, 0, 0, 0}, V4{0, 0, 0, 0}};
  if (16 * wv < n) {
    const DofGeo cg = pair_geo<PDE>(dof_geo(g, act[min(c, n - 1)]));
    if (l > 16) {
      sketch_pairs<R, PDE, true, 2, LM, 2, true>(tab, rowdofs, s.omega, cnt, 0, cnt, 0, 0, 1, cg,
                                                 acc);
      sketch_pairs<R, PDE, false, 2, LM, 2, true>(tab, rowdofs, s.omega, P, 2 * cnt, 2 * cnt + P,
                                                  cnt, 0, 1, cg, acc);
    } else {
      V4 one[1] = {acc[0]};
      sketch_pairs<R, PDE, true, 1, LM, 2, true>(tab, rowdofs, s.omega, cnt, 0, cnt, 0, 0, 1, cg,
                                                 one);
      sketch_pairs<R, PDE, false, 1, LM, 2, true>(tab, rowdofs, s.omega, P, 2 * cnt, 2 * cnt + P,
                                                  cnt, 0, 1, cg, one);
      acc[0] = one[0];
    }
  }
  __syncthreads();  // the row table becomes Y
  // acc[q][v] = Y[16 q + row(kq, v)][c]; rows past l are 0, columns past n
  // unused.
#pragma unroll
  for (int v = 0; v < 4; v++) {
    ybuf[Mfma16<R>::row(kq, v) * YLD + c] = acc[0][v];
    ybuf[(16 + Mfma16<R>::row(kq, v)) * YLD + c] = acc[1][v];
  }
  __syncthreads();
  if (wv != 0) return;

  // Pivoted QR of the sketch (wave 0).
  R y[LM];
#pragma unroll
  for (int r = 0; r < LM; r++) y[r] = ybuf[r * YLD + lane];
  R* rr = ybuf;  // rows of R, rr[j * YLD + c]
  const R tol = static_cast<R>(tol_d);
  bool avail = lane < n;
  int k = -1;
  R thresh = 0;
  R tl = 0;  // squared norm of the active rows past the first
  {
    R p4[4] = {0, 0, 0, 0};
#pragma unroll
    for (int r = 1; r < LM; r++) p4[r & 3] += y[r] * y[r];
    tl = (p4[0] + p4[1]) + (p4[2] + p4[3]);
  }
  const int jlim = min(n, l - kRidOver);
  int j = 0;
  for (; j < jlim; j++) {
    const double key = avail ? pivot_key<R, 6>(y[0] * y[0] + tl, lane) : -1.0;
    const double best = wave_max(key);
    const int p = __ffsll((unsigned long long)__ballot(key == best)) - 1;
    const R alpha = lane_value(y[0], p), xt = lane_value(tl, p);
    R beta, tau, sc;
    householder_scalars(alpha, xt, &beta, &tau, &sc);
    if (j == 0) {
      thresh = fabs(tol * beta);
    } else if (sketch_diag<false>(beta, l, j) < thresh) {
      k = j;
      break;
    }
    if (lane == p) {
      spiv[j] = p;
      avail = false;
    }
    // The pivot column's entries below row j, uniform across the wave:
    // the Householder vector is (1, sc yp[1], ..., sc yp[LM-1]).
    R yp[LM];
#pragma unroll
    for (int r = 1; r < LM; r++) yp[r] = lane_value(y[r], p);
    R d4[4] = {0, 0, 0, 0};
#pragma unroll
    for (int r = 1; r < LM; r++) d4[r & 3] += yp[r] * y[r];
    const R w = tau * (y[0] + sc * ((d4[0] + d4[1]) + (d4[2] + d4[3])));
    const R ws = w * sc;
    // Row j of R leaves; the rest shift up one register.
    rr[j * YLD + lane] = (lane == p) ? beta : y[0] - w;
    R t4[4] = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < LM - 1; r++) {
      y[r] = y[r + 1] - ws * yp[r + 1];
      if (r > 0) t4[r & 3] += y[r] * y[r];
    }
    y[LM - 1] = 0;
    tl = (t4[0] + t4[1]) + (t4[2] + t4[3]);
  }
  wave_sync();
  if (k < 0) {
    if (j < n) {  // the sketch ran out before a cut: the full QRCP takes it
      if (lane == 0) {
        const int pos = atomicAdd(list_slot(s, level, kLstFallback), 1);
        s.lists[(int64_t)kLstFallback * s.nbox + start + pos] = b;
      }
      return;
    }
    k = n;  // every column taken: nothing redundant
  }

  // T = R11^{-1} R12 by a column sweep in registers: lane c holds column c
  // of R (rows 0..k-1), R11(i, q) = rr[i][spiv[q]] is read from LDS; the
  // redundant lanes' columns become T.
  constexpr int KMAX = LM - kRidOver;
  const bool red = avail;
  R x[KMAX];
#pragma unroll
  for (int i = 0; i < KMAX; i++) x[i] = i < k ? rr[i * YLD + lane] : R(0);
#pragma unroll
  for (int q = KMAX - 1; q >= 0; q--) {
    if (q < k) {
      const int pq = spiv[q];
      const R tq = x[q] * recip_any(rr[q * YLD + pq]);
      x[q] = tq;
#pragma unroll
      for (int i = 0; i < q; i++) x[i] -= rr[i * YLD + pq] * tq;
    }
  }
  const uint64_t redmask = __ballot(red);
  const int cp = __popcll(redmask & ((1ull << lane) - 1));  // redundant index
  R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
  if (red) {
#pragma unroll
    for (int i = 0; i < KMAX; i++)
      if (i < k) F[i + (int64_t)k * cp] = x[i];
  }
  int* out = s.out_list + (int64_t)b * s.ncap;
  int* rl = s.red_list + (int64_t)b * s.ncap;
  int* pm = s.perm + (int64_t)b * s.ncap;
  if (lane < k) {
    const int cc = spiv[lane];
    pm[lane] = cc;
    out[lane] = act[cc];
  }
  if (red) {
    pm[k + cp] = lane;
    rl[cp] = act[lane];
  }
  if (lane == 0) {
    s.rank[b] = k;
    s.out_cnt[b] = k;
    s.rid_done[b] = 1;
  }
}

// Wide randomized ID: the boxes too large for k_rid, by columns or by near
// DOFs, and on the top levels those whose predicted rank passes its widest
// sketch (up to kRidMaxNearW near DOFs and kRidWideCols columns, ranks up to
// kRidRowsW - kRidOver).  With the rank model on every level: k_qrcp took 2.0
// to 3.4 ms for a level of 70 to 100 boxes of 65 to 87 Stokes DOFs, whose
// stacked triangles do not fit the register QRCP, this form 230 us.  Same
// sketch and outputs as k_rid with kRidRowsW rows from its own table, on 8
// waves: wave w sketches the 16-column tile w % (4 QW) over every (8 / 4
// QW)-th 16-row block, the row parts added in a fixed order.  QW waves then
// run the pivoted QR, wave q holding columns 64 q + lane: QW = 1 for n <= 64
// (one wave, no barrier), QW = 2 for n <= 128 (each wave publishes its best
// column's Householder vector and key, both read the winner's; one barrier
// per step).  A box whose sketch shows no cut goes on to the 128-row sketch
// on the top levels; below them a register-QRCP box joins the fallback list
// and any other is still on its full-QRCP list (whose kernels skip the boxes
// a sketch took).
constexpr int kRidWideWaves = 8;

// LDS of the wide sketch: the row table, then Y, then the rows of R (a
// raw buffer sized for two QR waves), and the QR's small arrays.
template <typename R>
struct RidWideLds {
  static constexpr int TR = kRidMaxNearW + kNumProxy;
  static constexpr int YMAX = kRidRowsW * (2 * 64 + 1);  // two QR waves' Y
  static constexpr int kBuf = (YMAX * (int)sizeof(R) + 7) / 8 > 6 * TR
                                  ? (YMAX * (int)sizeof(R) + 7) / 8
                                  : 6 * TR;
  double buf[kBuf];
  int rowdofs[kRidMaxNearW];
  R vbuf[4][kRidRowsW];  // two QR waves: each wave's candidate Householder
                         // vector, by step parity
  int spiv[64];
  double kbest[4];  // two QR waves: each wave's pivot key, by step parity
  R hs[4][2];       // two QR waves: each candidate's beta and tau
  int nred0;        // two QR waves: redundant columns of wave 0
};

// Fixed widths, which keep this sketch to the top levels' boxes, cut as the
// narrow sketches do.
template <typename R>
__device__ inline R wide_diag(const DevState& s, R beta, int l, int j) {
  return s.rid_mode == 2 ? sketch_diag<true>(beta, l, j) : sketch_diag<false>(beta, l, j);
}

template <typename R, int PDE, int QW, bool LOOP>
__device__ __forceinline__ void rid_wide_box(const DevGeom& g, const DevTree& t,
                                             const DevState& s, int start, int level,
                                             double tol_d, int b, RidWideLds<R>& sh) {
  constexpr int kTiles = 4 * QW, kParts = kRidWideWaves / kTiles;
  constexpr int NT = 64 * kRidWideWaves;
  constexpr int LM = kRidRowsW, YLD = 64 * QW + 1, TR = RidWideLds<R>::TR;
  using V4 = typename Mfma16<R>::V4;
  double (*tab)[TR] = reinterpret_cast<double (*)[TR]>(sh.buf);
  R* ybuf = reinterpret_cast<R*>(sh.buf);
  int* rowdofs = sh.rowdofs;
  int* spiv = sh.spiv;
  double* kbest = sh.kbest;
  const int n = s.act_cnt[b], m = s.m_rows[b], l = s.sk_w[b];
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  const int P = proxy_rows(g, level) / 2;
  const int cnt = (m - 2 * P) / 2;
  const int* act = s.act_list + (int64_t)b * s.ncap;
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
  for (int i = tid; i < cnt; i += NT) {
    const DofGeo d = pair_geo<PDE>(dof_geo(g, rowdofs[i]));
    tab[0][i] = d.x;
    tab[1][i] = d.y;
    tab[2][i] = d.n1;
    tab[3][i] = d.n2;
    tab[4][i] = d.w;
    tab[5][i] = d.k;
  }
  __syncthreads();

  // Sketch: wave wv takes tile wv % kTiles, row part wv / kTiles.
  const int kq = lane >> 4;
  const int tile = wv % kTiles, part = wv / kTiles;
  V4 acc[4];
#pragma unroll
  for (int q = 0; q < 4; q++) acc[q] = V4{0, 0, 0, 0};
  const int c = 16 * tile + (lane & 15);
  if (16 * tile < n) {
    const DofGeo cg = pair_geo<PDE>(dof_geo(g, act[min(c, n - 1)]));
    sketch_pairs<R, PDE, true, 4, LM, 2, true>(tab, rowdofs, s.omega_w, cnt, 0, cnt, 0, part,
                                               kParts, cg, acc);
    sketch_pairs<R, PDE, false, 4, LM, 2, true>(tab, rowdofs, s.omega_w, P, 2 * cnt, 2 * cnt + P,
                                                cnt, part, kParts, cg, acc);
  }
  __syncthreads();  // the row table becomes Y
  for (int p = 0; p < kParts; p++) {  // the row parts added in order
    if (part == p) {
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          R* y = &ybuf[(16 * q + Mfma16<R>::row(kq, v)) * YLD + c];
          *y = p == 0 ? acc[q][v] : *y + acc[q][v];
        }
    }
    __syncthreads();
  }
  const int jlim = min(n, l - kRidOver);
  if (wv >= QW) {
    // With one box per workgroup the other waves end here; where the
    // workgroup takes more boxes they keep step with the two QR waves'
    // barriers, from the same published pivots.
    if (LOOP && QW == 2) {
      int j = 0;
      R thresh = 0;
      bool cut = false;
      for (; j < jlim && !cut; j++) {
        __syncthreads();
        const int par = j & 1;
        const double best = fmax(kbest[2 * par], kbest[2 * par + 1]);
        const R beta = sh.hs[2 * par + (pivot_key_pos<7>(best) >> 6)][0];
        if (j == 0) thresh = fabs(static_cast<R>(tol_d) * beta);
        else cut = wide_diag(s, beta, l, j) < thresh;
      }
      if (cut || j >= n) __syncthreads();  // the redundant counts
    }
    return;
  }

  // Pivoted QR of the sketch: wave wv holds column col = 64 wv + lane.
  const int col = 64 * wv + lane;
  R y[LM];
#pragma unroll
  for (int r = 0; r < LM; r++) y[r] = ybuf[r * YLD + col];
  R* rr = ybuf;  // rows of R, rr[j * YLD + c]
  const R tol = static_cast<R>(tol_d);
  bool av = col < n;
  R tl;
  {
    R p4[4] = {0, 0, 0, 0};
#pragma unroll
    for (int r = 1; r < LM; r++) p4[r & 3] += y[r] * y[r];
    tl = (p4[0] + p4[1]) + (p4[2] + p4[3]);
  }
  int k = -1;
  R thresh = 0;
  int j = 0;
  for (; j < jlim; j++) {
    double best = wave_max(av ? pivot_key<R, 7>(y[0] * y[0] + tl, col) : -1.0);
    int p, pw, pl;
    R beta = 0, tau = 0, sc = 0;
    const R* vb = nullptr;
    if (QW == 2) {
      // Each wave publishes its own best column's Householder vector before
      // the step's one barrier; after it both read the winner's (by step
      // parity: a wave a step ahead writes the other slot).
      const int par = j & 1;
      if (best >= 0) {
        const int ql = pivot_key_pos<7>(best) & 63;
        const R alpha = lane_value(y[0], ql), xt = lane_value(tl, ql);
        R b0, t0, s0;
        householder_scalars(alpha, xt, &b0, &t0, &s0);
        if (lane == ql) {
          R* w = sh.vbuf[2 * par + wv];
          w[0] = R(1);
#pragma unroll
          for (int r = 1; r < LM; r++) w[r] = y[r] * s0;
          sh.hs[2 * par + wv][0] = b0;
          sh.hs[2 * par + wv][1] = t0;
        }
      }
      if (lane == 0) kbest[2 * par + wv] = best;
      __syncthreads();
      best = fmax(kbest[2 * par], kbest[2 * par + 1]);
      p = pivot_key_pos<7>(best);  // column index
      pw = p >> 6;
      pl = p & 63;
      beta = sh.hs[2 * par + pw][0];
      tau = sh.hs[2 * par + pw][1];
      vb = sh.vbuf[2 * par + pw];
      if (wv == 0 && lane == 0) spiv[j] = p;
    } else {
      p = pivot_key_pos<7>(best);  // column index
      pw = p >> 6;
      pl = p & 63;
      const R alpha = lane_value(y[0], pl), xt = lane_value(tl, pl);
      householder_scalars(alpha, xt, &beta, &tau, &sc);
    }
    if (j == 0) {
      thresh = fabs(tol * beta);
    } else if (wide_diag(s, beta, l, j) < thresh) {
      k = j;
      break;
    }
    if (col == p) av = false;
    R t4[4] = {0, 0, 0, 0};
    if (QW == 1) {
      // One wave: the pivot column reaches every lane through readlane
      // (twice: kept between the dot and the update it would not fit the
      // registers beside y); the Householder vector is (1, sc yp[1..]).
      if (lane == pl) spiv[j] = p;
      R d4[4] = {0, 0, 0, 0};
#pragma unroll
      for (int r = 1; r < LM; r++) d4[r & 3] += lane_value(y[r], pl) * y[r];
      const R w = tau * (y[0] + sc * ((d4[0] + d4[1]) + (d4[2] + d4[3])));
      const R ws = w * sc;
      rr[j * YLD + col] = (col == p) ? beta : y[0] - w;
      int pl2 = pl;
      __asm__ volatile("" : "+s"(pl2));
#pragma unroll
      for (int r = 0; r < LM - 1; r++) {
        y[r] = y[r + 1] - ws * lane_value(y[r + 1], pl2);
        if (r > 0) t4[r & 3] += y[r] * y[r];
      }
    } else {
      R d4[4] = {0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < LM; r++) d4[r & 3] += vb[r] * y[r];
      const R w = tau * ((d4[0] + d4[1]) + (d4[2] + d4[3]));
      rr[j * YLD + col] = (col == p) ? beta : y[0] - w;
      // the vector is read again below rather than kept in registers beside y
      __asm__ volatile("" ::: "memory");
#pragma unroll
      for (int r = 0; r < LM - 1; r++) {
        y[r] = y[r + 1] - w * vb[r + 1];
        if (r > 0) t4[r & 3] += y[r] * y[r];
      }
    }
    y[LM - 1] = 0;
    tl = (t4[0] + t4[1]) + (t4[2] + t4[3]);
    if (QW == 1) wave_sync();
  }
  const bool regq = s.qkind[b] == kQrcpReg || s.qkind[b] == kQrcpStack;
  if (k < 0) {
    if (j < n) {  // no cut within the sketch: a wider one or the full QRCP takes the box
      if (level <= kRidBigTop && tid == 0) {
        // Its slot comes from what the level's scan left of the ID pool: few
        // 64-row sketches fail, and a slot for each of them is 330 KB at 64
        // columns.
        const int64_t need = rid_big_scratch(n);
        const int64_t off = (int64_t)atomicAdd(
            reinterpret_cast<unsigned long long*>(s.id_top + level), (unsigned long long)need);
        s.big_off[b] = (level & 1) * s.id_cap + off;
        if (off + need > s.id_cap) {  // k_rid_big_* stop; the host repeats with more
          atomicOr(s.err, kErrIdPool);
          atomicMax(s.err + 2, (int)((off + need + 1023) >> 10));
        }
        const int pos = atomicAdd(list_slot(s, level, kLstRidBig), 1);
        s.lists[(int64_t)kLstRidBig * s.nbox + start + pos] = b;
        s.sk_w[b] = kRidRowsB;
      } else if (regq && tid == 0) {
        const int pos = atomicAdd(list_slot(s, level, kLstFallback), 1);
        s.lists[(int64_t)kLstFallback * s.nbox + start + pos] = b;
      }
      return;
    }
    k = n;
  }
  // Every wave's rows of R are in LDS; wave 0's redundant count for wave 1.
  const uint64_t mk = __ballot(av);
  if (QW == 2) {
    if (wv == 0 && lane == 0) sh.nred0 = __popcll(mk);
    __syncthreads();
  }

  // T = R11^{-1} R12 by a column sweep in registers, R11 read from LDS.
  constexpr int KMAX = LM - kRidOver;
  R x[KMAX];
#pragma unroll
  for (int i = 0; i < KMAX; i++) x[i] = i < k ? rr[i * YLD + col] : R(0);
#pragma unroll
  for (int q = KMAX - 1; q >= 0; q--) {
    if (q < k) {
      const int pq = spiv[q];
      const R tq = x[q] * recip_any(rr[q * YLD + pq]);
      x[q] = tq;
#pragma unroll
      for (int i = 0; i < q; i++) x[i] -= rr[i * YLD + pq] * tq;
    }
  }
  const int cp = (wv == 1 ? sh.nred0 : 0) + __popcll(mk & ((1ull << lane) - 1));  // redundant index
  R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
  int* out = s.out_list + (int64_t)b * s.ncap;
  int* rl = s.red_list + (int64_t)b * s.ncap;
  int* pm = s.perm + (int64_t)b * s.ncap;
  if (av) {
#pragma unroll
    for (int i = 0; i < KMAX; i++)
      if (i < k) F[i + (int64_t)k * cp] = x[i];
    pm[k + cp] = col;
    rl[cp] = act[col];
  }
  if (wv == 0 && lane < k) {
    const int cc = spiv[lane];
    pm[lane] = cc;
    out[lane] = act[cc];
  }
  if (tid == 0) {
    s.rank[b] = k;
    s.out_cnt[b] = k;
    s.rid_done[b] = 1;
  }
}

// One launch for both forms: boxes with n <= 64 run the one-wave QR,
// the others the two-wave QR.  LOOP: the workgroups walk the level's list
// (levels with more boxes than kRidWideGrid, most of which are on other
// lists: a workgroup of 512 threads and 67 KB of LDS per box of the level
// would be launched for nothing).
constexpr int kRidWideGrid = 512;

template <typename R, int PDE, bool LOOP>
__global__ __launch_bounds__(64 * kRidWideWaves, 1) void k_rid_wide(
    DevGeom g, DevTree t, DevState s, int start, int level, double tol_d) {
  __shared__ RidWideLds<R> sh;
  if (s.halt[level]) return;  // not err, which this kernel's own boxes write
  const int nl = list_count(s, level, kLstRidWide);
  for (int li = blockIdx.x; li < nl; li += LOOP ? (int)gridDim.x : nl) {
    const int b = list_at(s, start, kLstRidWide, li);
    if (s.act_cnt[b] > 64) rid_wide_box<R, PDE, 2, LOOP>(g, t, s, start, level, tol_d, b, sh);
    else rid_wide_box<R, PDE, 1, LOOP>(g, t, s, start, level, tol_d, b, sh);
    if (LOOP) __syncthreads();
  }
}

// Gaussian table for the sketches: z = sqrt(-2 ln u1) cos(2 pi u2) (Box and
// Muller 1958) from two 53-bit uniforms of a SplitMix64 hash of the index.
__device__ inline uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
__global__ __launch_bounds__(256) void k_gaussian(double* out, int64_t n, uint64_t seed) {
  for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const uint64_t h1 = splitmix64(seed ^ (2 * (uint64_t)i));
    const uint64_t h2 = splitmix64(seed ^ (2 * (uint64_t)i + 1));
    const double u1 = ((h1 >> 11) + 1) * (1.0 / 9007199254740992.0);  // (0, 1]
    const double u2 = (h2 >> 11) * (1.0 / 9007199254740992.0);        // [0, 1)
    out[i] = sqrt(-2.0 * log(u1)) * cos(2.0 * M_PI * u2);
  }
}

}  // namespace

void launch_gaussian(double* out, int64_t n, uint64_t seed, hipStream_t st) {
  k_gaussian<<<256, 256, 0, st>>>(out, n, seed);
}

template <typename R, int PDE>
void launch_rid_wide(const DevGeom& g, const DevTree& t, const DevState& s, int start,
                     int level, int listed, double tol, hipStream_t st) {
  if (listed <= kRidWideGrid)
    k_rid_wide<R, PDE, false><<<listed, 64 * kRidWideWaves, 0, st>>>(g, t, s, start, level, tol);
  else
    k_rid_wide<R, PDE, true>
        <<<kRidWideGrid, 64 * kRidWideWaves, 0, st>>>(g, t, s, start, level, tol);
}

template <typename R>
void launch_rid(const DevGeom& g, const DevTree& t, const DevState& s, int level, int start,
                int listed, double tol, hipStream_t st, int skip) {
  if (skip & kSkipRid) {
    // no 16- or 32-row sketch on this level (launch plan)
  } else if (g.pde == kPdeStokes) {
    k_rid<R, kPdeStokes><<<listed, 256, 0, st>>>(g, t, s, start, level, tol);
  } else if (g.pde == kPdeLaplaceNeumann) {
    k_rid<R, kPdeLaplaceNeumann><<<listed, 256, 0, st>>>(g, t, s, start, level, tol);
  } else {
    k_rid<R, kPdeLaplace><<<listed, 256, 0, st>>>(g, t, s, start, level, tol);
  }
  if (!(skip & kSkipRidWide)) {
    if (g.pde == kPdeStokes)
      launch_rid_wide<R, kPdeStokes>(g, t, s, start, level, listed, tol, st);
    else if (g.pde == kPdeLaplaceNeumann)
      launch_rid_wide<R, kPdeLaplaceNeumann>(g, t, s, start, level, listed, tol, st);
    else
      launch_rid_wide<R, kPdeLaplace>(g, t, s, start, level, listed, tol, st);
  }
  // after the 64-row sketches, whose failures it takes
  if (level <= kRidBigTop && !(skip & kSkipRidBig))
    launch_rid_big<R>(g, t, s, start, level, listed, tol, st);
}

template void launch_rid<double>(const DevGeom&, const DevTree&, const DevState&, int, int, int,
                                 double, hipStream_t, int);
template void launch_rid<float>(const DevGeom&, const DevTree&, const DevState&, int, int, int,
                                double, hipStream_t, int);

}  // namespace iegpu
