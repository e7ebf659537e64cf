// Interpolative decomposition of the FP32 factorization's boxes from the
// Gram matrix of their ID matrices, formed and factored in FP64
// (ie_mat.cpp:548-588, the pivoted QR it stands in for).

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "rs_device.hpp"
#include "rs_id.hpp"
#include "rs_kernels.hpp"

namespace iegpu {

namespace {

// ---------------------------------------------------------------------------
// With G = A^T A, pivoted Cholesky of G takes the columns that column-pivoted
// QR of A takes and gives the same R (up to signs): the pivot is the largest
// remaining column norm, |R_jj| its square root.  G's rounding, 2^-53 |A|^2,
// limits |R_jj| to about 1e-8 |A|, finer than the 2^-24 |A| at which QR in
// FP32 stops, while A's rows are summed on the matrix cores as they are
// evaluated: no m x n matrix is stored, no step runs over the rows.  FP64
// factorizations keep the QR (their tolerances lie below G's limit), and so
// does an FP32 one at a tolerance under kGramTol.
//
// k_gram_id: boxes of up to NMAX = 32 or 64 columns, one workgroup each.
// A wave evaluates blocks of four row points against every column tile, both
// directions at once (K(row, box) and K(box, row) share |r|^2 and its
// reciprocal), and accumulates the tile pairs of G; the four waves' sums are
// added in order and wave 0 factors G, a lane per column.
// k_gram_blocks / k_gram_chol: 65 to 256 columns, a workgroup per 32 x 32
// block of G, then one per box.
// Entry evaluation and its MFMAs bound k_gram_id, the latency of the steps
// k_gram_chol.  Stokes with 8 holes, 131,072 points, plain FP32 at 1e-6: 4.3
// ms per factorization (k_gram_id 2.5, k_gram_blocks 0.14, k_gram_chol 1.6)
// against 25.1 for row compression, register and general QR and assembly.
// ---------------------------------------------------------------------------

constexpr int kItems = 256;      // row points staged at a time
// A column's squared norm is enlarged by kGramRound^2 of itself, about what
// FP32's rounding of the entries and of the steps (2^-24 each) added to it in
// the QR: without it T's rows at diagonals near that level grow, and the FP32
// blocks formed with T lose more (Stokes, tolerance 1e-6: backward error of
// the unrefined solve 5 to 8 % larger than with the QR, whatever the cut
// between 0.5 and 1).  The cut is |R_jj| < kGramCut tol |R_00|, the factor
// offsetting what the enlargement adds to |R_jj|.  Backward error against the
// FP32 QR's, means over 320 stars, wavy boundaries and circles with holes of
// 900 and 3,000 points in three kernels per tolerance: 0.70 at 5e-7, 0.94 at
// 1e-6, 0.98 at 1e-5, 0.91 at 1e-4; ranks 1 % larger (3 % at 5e-7).
constexpr double kGramRound = 2e-7;
constexpr double kGramCut = 0.9;
__device__ inline double rounded_norm2(double g) { return fma(g, kGramRound * kGramRound, g); }

struct RowItems {
  double x[kItems], y[kItems], n1[kItems], n2[kItems], w[kItems], k[kItems];
  int c[kItems];
};

__device__ inline void stage_item(RowItems& it, int i, const DofGeo& d) {
  it.x[i] = d.x;
  it.y[i] = d.y;
  it.n1[i] = d.n1;
  it.n2[i] = d.n2;
  it.w[i] = d.w;
  it.k[i] = d.k;
  it.c[i] = d.c;
}
__device__ inline DofGeo load_item(const RowItems& it, int i) {
  DofGeo d;
  d.x = it.x[i];
  d.y = it.y[i];
  d.n1 = it.n1[i];
  d.n2 = it.n2[i];
  d.w = it.w[i];
  d.k = it.k[i];
  d.c = it.c[i];
  return d;
}

typedef Mfma16<double>::V4 D4;

// Every row of box b's ID matrix, in blocks of four row points per wave:
// f(NEAR, item) is called with the lane's row point (lane / 16 of the block)
// and whether it is one.  256 threads; rowdofs is filled here.
template <int PDE, typename F>
__device__ __forceinline__ void for_row_blocks(const DevGeom& g, const DevTree& t,
                                               const DevState& s, int b, int level, int cnt,
                                               int* rowdofs, RowItems& items, F&& f) {
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id(), kq = lane >> 4;
  if (wv == 0)
    for_each_row_dof(g, t, s, b, level >= 3, [&](int pos, int dof) { rowdofs[pos] = dof; });
  __syncthreads();
  for (int base = 0; base < cnt; base += kItems) {
    const int ni = min(kItems, cnt - base);
    if (tid < ni) stage_item(items, tid, pair_geo<PDE>(dof_geo(g, rowdofs[base + tid])));
    __syncthreads();
    for (int i0 = 4 * wv; i0 < ni; i0 += 16) {
      const int i = min(i0 + kq, ni - 1);
      f(std::true_type{}, load_item(items, i), i0 + kq < ni);
    }
    __syncthreads();
  }
  if (level >= 3) {
    constexpr bool stokes = PDE == kPdeStokes;
    constexpr int ni = stokes ? 2 * kNumProxy : kNumProxy;
    static_assert(ni <= kItems, "one block of proxy rows");
    if (tid < ni) {
      DofGeo d;
      proxy_point(t.cx[b], t.cy[b], t.side[b] * kRadiusRatio, stokes ? tid >> 1 : tid, &d.x, &d.y,
                  &d.n1, &d.n2);
      d.w = proxy_weight(t, b);
      d.k = 0;
      d.c = stokes ? tid & 1 : 0;
      stage_item(items, tid, pair_geo<PDE>(d));
    }
    __syncthreads();
    for (int i0 = 4 * wv; i0 < ni; i0 += 16)
      f(std::false_type{}, load_item(items, i0 + kq), true);
    __syncthreads();
  }
}

// Box li of this level's Gram boxes of up to 64 columns, -1 past the last.
__device__ inline int gram_box(const DevState& s, int start, int level, int li, bool half) {
  if (s.rid_mode != 0) {  // only the boxes without a successful sketch
    if (li >= list_count(s, level, kLstFallback)) return -1;
    const int b = list_at(s, start, kLstFallback, li);
    return half == (s.act_cnt[b] <= kHalfCols) ? b : -1;
  }
  const int L = half ? kLstRegHalf : kLstReg;
  return li < list_count(s, level, L) ? list_at(s, start, L, li) : -1;
}

template <typename R, int PDE, int NMAX>
__global__ __launch_bounds__(256, NMAX == 32 ? 4 : 2) void k_gram_id(DevGeom g, DevTree t, DevState s, int start,
                                                 int level, double tol) {
  constexpr int NT = NMAX / 16, LD = NMAX + 1;
  __shared__ union {
    struct {
      RowItems items;
      int rowdofs[kGramNear];
    } rows;
    struct {
      double G[NMAX * LD], rr[NMAX * LD];
    } m;
  } sh;
  __shared__ int spiv[NMAX];
  if (!pools_ok(s)) return;
  const int b = gram_box(s, start, level, blockIdx.x, NMAX == kHalfCols);
  if (b < 0) return;
  const int n = s.act_cnt[b], m = s.m_rows[b], nt = (n + 15) / 16;
  const int cnt = (m - proxy_rows(g, level)) / 2;
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id(), kq = lane >> 4, cl = lane & 15;
  const int* act = s.act_list + (int64_t)b * s.ncap;
  DofGeo cg[NT];
#pragma unroll
  for (int q = 0; q < NT; q++) cg[q] = pair_geo<PDE>(dof_geo(g, act[min(16 * q + cl, n - 1)]));
  D4 acc[NT * (NT + 1) / 2];
#pragma unroll
  for (int q = 0; q < NT * (NT + 1) / 2; q++) acc[q] = D4{0, 0, 0, 0};
  for_row_blocks<PDE>(
      g, t, s, b, level, cnt, sh.rows.rowdofs, sh.rows.items,
      [&](auto near, const DofGeo& row, bool live) {
        double et[NT], es[NT];
#pragma unroll
        for (int q = 0; q < NT; q++) {
          et[q] = es[q] = 0;
          if (q < nt) {
            pair_entries<PDE, decltype(near)::value>(row, cg[q], et[q], es[q]);
            const bool on = live && 16 * q + cl < n;
            et[q] = on ? et[q] : 0.0;
            es[q] = on ? es[q] : 0.0;
          }
        }
#pragma unroll
        for (int J = 0; J < NT; J++)
          if (J < nt)
#pragma unroll
            for (int I = 0; I <= J; I++) {
              D4& a = acc[J * (J + 1) / 2 + I];
              a = mfma16x16x4(et[I], et[J], a);
              a = mfma16x16x4(es[I], es[J], a);
            }
      });
  for (int w = 0; w < 4; w++) {  // the waves' parts added in order
    if (wv == w)
#pragma unroll
      for (int J = 0; J < NT; J++)
        if (J < nt)
#pragma unroll
          for (int I = 0; I <= J; I++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
              double* e = &sh.m.G[(16 * I + Mfma16<double>::row(kq, v)) * LD + 16 * J + cl];
              const double a = acc[J * (J + 1) / 2 + I][v];
              *e = w == 0 ? a : *e + a;
            }
    __syncthreads();
  }
  if (wv != 0) return;

  // Pivoted Cholesky, lane = column: rows of R to LDS as they are formed.
  double* G = sh.m.G;
  double* Rm = sh.m.rr;
  bool avail = lane < n;
  double d = avail ? rounded_norm2(G[lane * LD + lane]) : 0.0;
  int k = 0;
  double thresh = 0;
  const int kmax = min(m, n);
  for (; k < kmax; k++) {
    const double best = wave_max(avail ? pivot_key<double, 6>(fmax(d, 0.0), lane) : -1.0);
    if (!(best >= 0)) break;
    const int p = pivot_key_pos<6>(best);
    const double dp = lane_value(d, p), rjj = sqrt(dp);
    if (!(dp > 0) || (k > 0 && rjj < thresh)) break;
    if (k == 0) thresh = kGramCut * tol * rjj;
    // G is stored by tile pairs I <= J: the lower ones mirrored
    double a0 = (p >> 4) <= (lane >> 4) ? G[p * LD + min(lane, NMAX - 1)] : G[lane * LD + p];
    double a1 = 0;
    int i = 0;
    for (; i + 2 <= k; i += 2) {
      a0 -= Rm[i * LD + p] * Rm[i * LD + min(lane, NMAX - 1)];
      a1 -= Rm[(i + 1) * LD + p] * Rm[(i + 1) * LD + min(lane, NMAX - 1)];
    }
    if (i < k) a0 -= Rm[i * LD + p] * Rm[i * LD + min(lane, NMAX - 1)];
    const double v = avail ? (a0 + a1) * (1.0 / rjj) : 0.0;
    if (lane < NMAX) Rm[k * LD + lane] = lane == p ? rjj : v;
    if (lane == p) {
      spiv[k] = p;
      avail = false;
    }
    d -= v * v;
    wave_sync();
  }
  int* out = s.out_list + (int64_t)b * s.ncap;
  if (k == 0) {  // an empty or non-finite block stays uncompressed
    for (int i = lane; i < n; i += 64) out[i] = act[i];
    if (lane == 0) {
      s.rank[b] = 0;
      s.out_cnt[b] = n;
      s.rid_done[b] = kIdGram;
    }
    return;
  }
  const uint64_t mask = __ballot(avail);
  const int cp = __popcll(mask & ((1ull << lane) - 1));
  R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
  if (avail) {  // T = R11^{-1} R12 by back substitution, over the column of R
    for (int i = k - 1; i >= 0; i--) {
      double a0 = Rm[i * LD + lane], a1 = 0;
      int l = i + 1;
      for (; l + 2 <= k; l += 2) {
        a0 -= Rm[i * LD + spiv[l]] * Rm[l * LD + lane];
        a1 -= Rm[i * LD + spiv[l + 1]] * Rm[(l + 1) * LD + lane];
      }
      if (l < k) a0 -= Rm[i * LD + spiv[l]] * Rm[l * LD + lane];
      const double tv = (a0 + a1) * (1.0 / Rm[i * LD + spiv[i]]);
      Rm[i * LD + lane] = tv;
      F[i + (int64_t)k * cp] = static_cast<R>(tv);
    }
  }
  int* rl = s.red_list + (int64_t)b * s.ncap;
  int* pm = s.perm + (int64_t)b * s.ncap;
  if (lane < k) {
    const int cc = spiv[lane];
    pm[lane] = cc;
    out[lane] = act[cc];
  }
  if (avail) {
    pm[k + cp] = lane;
    rl[cp] = act[lane];
  }
  if (lane == 0) {
    s.rank[b] = k;
    s.out_cnt[b] = k;
    s.rid_done[b] = kIdGram;
  }
}

// Box li of this level's Gram boxes of 65 to kGramCols columns, -1 for one
// another kernel takes.
__device__ inline int gram_big_box(const DevGeom& g, const DevState& s, int start, int level,
                                   int li, int n8) {
  const int b = li < n8 ? list_at(s, start, kLstReg8, li) : list_at(s, start, kLstLds, li - n8);
  const int n = s.act_cnt[b];
  if (s.rid_done[b] == 1 || n <= 64 || n > kGramCols ||
      (s.m_rows[b] - proxy_rows(g, level)) / 2 > kGramNear)
    return -1;
  return b;
}

// Block (bi, bj), bi <= bj, of 32 x 32 entries of G into the box's scratch
// (n16 x n16 doubles, both triangles).
template <typename R, int PDE>
__global__ __launch_bounds__(256) void k_gram_blocks(DevGeom g, DevTree t, DevState s, int start,
                                                     int level) {
  __shared__ RowItems items;
  __shared__ int rowdofs[kGramNear];
  __shared__ double part[4][32][33];
  if (!pools_ok(s)) return;
  const int n8 = list_count(s, level, kLstReg8), nl = n8 + list_count(s, level, kLstLds);
  const int lane = threadIdx.x & 63, wv = wave_id(), kq = lane >> 4, cl = lane & 15;
  for (int li = blockIdx.x; li < nl; li += gridDim.x) {
    const int b = gram_big_box(g, s, start, level, li, n8);
    if (b < 0) continue;
    const int n = s.act_cnt[b], nb = (n + 31) / 32, n16 = (n + 15) / 16 * 16;
    int bi = blockIdx.y, bj = 0;  // pair blockIdx.y of the upper triangle
    while (bi > bj) bi -= ++bj;
    if (bj >= nb) continue;
    const int cnt = (s.m_rows[b] - proxy_rows(g, level)) / 2;
    const int* act = s.act_list + (int64_t)b * s.ncap;
    DofGeo ci[2], cj[2];
    bool oi[2], oj[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int a = 32 * bi + 16 * q + cl, c = 32 * bj + 16 * q + cl;
      oi[q] = a < n;
      oj[q] = c < n;
      ci[q] = pair_geo<PDE>(dof_geo(g, act[min(a, n - 1)]));
      cj[q] = pair_geo<PDE>(dof_geo(g, act[min(c, n - 1)]));
    }
    D4 acc[2][2];
#pragma unroll
    for (int q = 0; q < 4; q++) acc[q >> 1][q & 1] = D4{0, 0, 0, 0};
    for_row_blocks<PDE>(g, t, s, b, level, cnt, rowdofs, items,
                        [&](auto near, const DofGeo& row, bool live) {
                          double ti[2], si[2], tj[2], sj[2];
#pragma unroll
                          for (int q = 0; q < 2; q++) {
                            pair_entries<PDE, decltype(near)::value>(row, ci[q], ti[q], si[q]);
                            pair_entries<PDE, decltype(near)::value>(row, cj[q], tj[q], sj[q]);
                            ti[q] = live && oi[q] ? ti[q] : 0.0;
                            si[q] = live && oi[q] ? si[q] : 0.0;
                            tj[q] = live && oj[q] ? tj[q] : 0.0;
                            sj[q] = live && oj[q] ? sj[q] : 0.0;
                          }
#pragma unroll
                          for (int I = 0; I < 2; I++)
#pragma unroll
                            for (int J = 0; J < 2; J++) {
                              acc[I][J] = mfma16x16x4(ti[I], tj[J], acc[I][J]);
                              acc[I][J] = mfma16x16x4(si[I], sj[J], acc[I][J]);
                            }
                        });
#pragma unroll
    for (int I = 0; I < 2; I++)
#pragma unroll
      for (int J = 0; J < 2; J++)
#pragma unroll
        for (int v = 0; v < 4; v++)
          part[wv][16 * I + Mfma16<double>::row(kq, v)][16 * J + cl] = acc[I][J][v];
    __syncthreads();
    double* G = reinterpret_cast<double*>(reinterpret_cast<R*>(s.id_pool) + s.id_off[b]);
    for (int e = threadIdx.x; e < 1024; e += 256) {
      const int i = e >> 5, j = e & 31;
      const double v = (part[0][i][j] + part[1][i][j]) + (part[2][i][j] + part[3][i][j]);
      const int gi = 32 * bi + i, gj = 32 * bj + j;
      if (gi < n && gj < n) {
        G[(int64_t)gi * n16 + gj] = v;
        if (bi != bj) G[(int64_t)gj * n16 + gi] = v;
      }
    }
    __syncthreads();  // the next box reuses the LDS
  }
}

// Pivoted Cholesky of a box's G and T, thread = column.  The first rows of
// R (as many as fit kCholLds) stay in LDS, the others in the scratch.
constexpr int kCholLds = 16384;

template <typename R>
__global__ __launch_bounds__(256) void k_gram_chol(DevGeom g, DevState s, int start, int level,
                                                   double tol) {
  __shared__ double Rl[kCholLds];
  __shared__ double wk[2][4];
  __shared__ double wd[2][4];
  __shared__ int spiv[kGramCols];
  __shared__ double rinv[kGramCols];
  __shared__ int rcnt[4];
  if (!pools_ok(s)) return;
  const int n8 = list_count(s, level, kLstReg8), nl = n8 + list_count(s, level, kLstLds);
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  for (int li = blockIdx.x; li < nl; li += gridDim.x) {
    const int b = gram_big_box(g, s, start, level, li, n8);
    if (b < 0) continue;
    const int n = s.act_cnt[b], n16 = (n + 15) / 16 * 16;
    const double* G = reinterpret_cast<const double*>(reinterpret_cast<R*>(s.id_pool) + s.id_off[b]);
    double* Rg = const_cast<double*>(G) + (int64_t)n16 * n16;
    const int jl = kCholLds / n16;  // rows of R in LDS
    bool avail = tid < n;
    const int c = min(tid, n - 1);
    double d = avail ? rounded_norm2(G[(int64_t)c * n16 + c]) : 0.0;
    double thresh = 0;
    int k = 0;
    const int kmax = min(s.m_rows[b], n);
    // sum_{i in [i0, i1)} R(i, p) R(i, c) over LDS or scratch rows
    auto dots = [&](const double* M, int i0, int i1, int p) {
      double a[4] = {0, 0, 0, 0};
      int i = i0;
      for (; i + 4 <= i1; i += 4)
#pragma unroll
        for (int u = 0; u < 4; u++) a[u] += M[(i + u) * n16 + p] * M[(i + u) * n16 + c];
      for (; i < i1; i++) a[0] += M[i * n16 + p] * M[i * n16 + c];
      return (a[0] + a[1]) + (a[2] + a[3]);
    };
    for (; k < kmax; k++) {
      const double best = wave_max(avail ? pivot_key<double, 8>(fmax(d, 0.0), tid) : -1.0);
      const int par = k & 1;
      if (avail && best >= 0 && pivot_key_pos<8>(best) == tid) wd[par][wv] = d;
      if (lane == 0) wk[par][wv] = best;
      __syncthreads();
      double top = wk[par][0];
      int tw = 0;
#pragma unroll
      for (int q = 1; q < 4; q++)
        if (wk[par][q] > top) {
          top = wk[par][q];
          tw = q;
        }
      if (!(top >= 0)) break;
      const int p = pivot_key_pos<8>(top);
      const double dp = wd[par][tw], rjj = sqrt(dp);
      if (!(dp > 0) || (k > 0 && rjj < thresh)) break;
      if (k == 0) thresh = kGramCut * tol * rjj;
      double v = G[(int64_t)p * n16 + c] - dots(Rl, 0, min(k, jl), p);
      if (k > jl) v -= dots(Rg, jl, k, p);
      const double ir = 1.0 / rjj;
      v = avail ? v * ir : 0.0;
      double* row = k < jl ? Rl + k * n16 : Rg + (int64_t)k * n16;
      if (tid < n) row[tid] = tid == p ? rjj : v;
      if (tid == p) {
        spiv[k] = p;
        rinv[k] = ir;
        avail = false;
      }
      d -= v * v;
      __syncthreads();
    }
    __syncthreads();
    const int* act = s.act_list + (int64_t)b * s.ncap;
    int* out = s.out_list + (int64_t)b * s.ncap;
    if (k == 0) {
      for (int i = tid; i < n; i += 256) out[i] = act[i];
      if (tid == 0) {
        s.rank[b] = 0;
        s.out_cnt[b] = n;
        s.rid_done[b] = kIdGram;
      }
      __syncthreads();
      continue;
    }
    const uint64_t mask = __ballot(avail);
    if (lane == 0) rcnt[wv] = __popcll(mask);
    __syncthreads();
    int cp = __popcll(mask & ((1ull << lane) - 1));
    for (int w = 0; w < wv; w++) cp += rcnt[w];
    R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
    if (avail) {
      for (int i = k - 1; i >= 0; i--) {
        const double* ri = i < jl ? Rl + i * n16 : Rg + (int64_t)i * n16;
        double a[2] = {ri[tid], 0};
        for (int l = i + 1; l < k; l++) {
          const double* rl = l < jl ? Rl + l * n16 : Rg + (int64_t)l * n16;
          a[l & 1] -= ri[spiv[l]] * rl[tid];
        }
        const double tv = (a[0] + a[1]) * rinv[i];
        double* w = i < jl ? Rl + i * n16 : Rg + (int64_t)i * n16;
        w[tid] = tv;
        F[i + (int64_t)k * cp] = static_cast<R>(tv);
      }
    }
    int* rl = s.red_list + (int64_t)b * s.ncap;
    int* pm = s.perm + (int64_t)b * s.ncap;
    if (tid < k) {
      const int cc = spiv[tid];
      pm[tid] = cc;
      out[tid] = act[cc];
    }
    if (avail) {
      pm[k + cp] = tid;
      rl[cp] = act[tid];
    }
    if (tid == 0) {
      s.rank[b] = k;
      s.out_cnt[b] = k;
      s.rid_done[b] = kIdGram;
    }
    __syncthreads();  // the next box reuses the LDS
  }
}

template <typename R, int PDE>
void launch_gram_pde(const DevGeom& g, const DevTree& t, const DevState& s, int level, int start,
                     int listed, double tol, hipStream_t st, int skip) {
  if (!(skip & kSkipRegQrcp)) {
    k_gram_id<R, PDE, 32><<<listed, 256, 0, st>>>(g, t, s, start, level, tol);
    k_gram_id<R, PDE, 64><<<listed, 256, 0, st>>>(g, t, s, start, level, tol);
  }
  if (!(skip & kSkipReg8Qrcp) || !(skip & kSkipAssemble)) {
    const int nb = listed < 256 ? listed : 256, blocks = kGramCols / 32;
    k_gram_blocks<R, PDE>
        <<<dim3(nb, blocks * (blocks + 1) / 2), 256, 0, st>>>(g, t, s, start, level);
    k_gram_chol<R><<<nb, 256, 0, st>>>(g, s, start, level, tol);
  }
}

}  // namespace

template <typename R>
void launch_gram(const DevGeom& g, const DevTree& t, const DevState& s, int level, int start,
                 int listed, double tol, hipStream_t st, int skip) {
  if (g.pde == kPdeStokes)
    launch_gram_pde<R, kPdeStokes>(g, t, s, level, start, listed, tol, st, skip);
  else if (g.pde == kPdeLaplaceNeumann)
    launch_gram_pde<R, kPdeLaplaceNeumann>(g, t, s, level, start, listed, tol, st, skip);
  else
    launch_gram_pde<R, kPdeLaplace>(g, t, s, level, start, listed, tol, st, skip);
}

template void launch_gram<float>(const DevGeom&, const DevTree&, const DevState&, int, int, int,
                                 double, hipStream_t, int);

}  // namespace iegpu
