// Column-pivoted QR interpolative decompositions (ie_mat.cpp:548-588):
// register-resident shapes with row compression of tall matrices, and the
// general form in LDS or global memory.

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "rs_device.hpp"
#include "rs_id.hpp"
#include "rs_kernels.hpp"

namespace iegpu {

namespace {

template <typename R>
struct Eps;
template <>
struct Eps<double> {
  // LAPACK dlamch('Epsilon') = 2^-53; dlaqp2 recomputes a column norm when
  // the downdated estimate falls below sqrt of it.
  static constexpr double tol3z = 1.0536712127723509e-08;
};
template <>
struct Eps<float> {
  static constexpr float tol3z = 2.44140625e-04f;
};

// ---------------------------------------------------------------------------
// Register-resident QR kernels (1024 threads, 16 waves).  Wave w holds
// columns CPW w .. CPW w + CPW - 1 of an m x n matrix (m <= 64 RPL,
// n <= 16 CPW) in the column interleave of rs_device.hpp: row i on lane
// i % 64, register i / 64, column CPW w + (sl ^ slot_class(lane)) in slot
// sl.  Two shapes: 4 columns x 8 row registers (n <= 64, m <= 512) and
// 8 columns x 4 row registers (n <= 128, m <= 256).  A Householder step:
// the wave owning the pivot column publishes the reflector through LDS;
// every wave then updates its columns in registers with one interleaved
// column reduction.  Waves past the last column only take part in the
// barriers.
// ---------------------------------------------------------------------------

constexpr int kXThreads = 1024;

template <int CPW>
struct RegShape {
  static constexpr int RPL = CPW == 4 ? 8 : 4;  // row registers per lane
  static constexpr int MAXM = 64 * RPL;
  static constexpr int MAXN = 16 * CPW;
};

// Entries of the column in slot psl (per lane) of the interleave.
template <typename R, int RPL, int CPW>
__device__ inline void pick_slot(const R (&a)[CPW][RPL], int psl, R (&x)[RPL]) {
#pragma unroll
  for (int r = 0; r < RPL; r++) x[r] = a[0][r];
#pragma unroll
  for (int sl = 1; sl < CPW; sl++) {
    const bool me = psl == sl;
#pragma unroll
    for (int r = 0; r < RPL; r++) x[r] = me ? a[sl][r] : x[r];
  }
}

// Row i (wave-uniform) of a column held as x[RPL], in every lane.  Each
// register is read out before the select: selecting first turns into a
// dynamically indexed extract, which the compiler lowers through scratch.
template <typename R, int RPL>
__device__ inline R row_value(const R (&x)[RPL], int i) {
  const int ri = i >> 6, li = i & 63;
  R v = lane_value(x[0], li);
#pragma unroll
  for (int r = 1; r < RPL; r++) {
    const R t = lane_value(x[r], li);
    v = (r == ri) ? t : v;
  }
  return v;
}

// Reflector v of column x at step j: v(0:j-1) = 0, v_j = 1,
// v(j+1:) = x(j+1:) sc; all 64 RPL rows (rows past the matrix hold zeros).
template <typename R, int RPL>
__device__ inline void write_reflector(const R (&x)[RPL], int j, R sc, R* vb) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < RPL; r++) {
    const int i = lane + 64 * r;
    vb[i] = i > j ? x[r] * sc : (i == j ? R(1) : R(0));
  }
}

// a <- (I - tau v v^T) a on this wave's columns; `live` says whether the
// class slot_class(lane) is still to be updated (pivoted columns keep
// their R entries).
template <typename R, int RPL, int CPW>
__device__ inline void apply_reflector(R (&a)[CPW][RPL], const R* vb, R tau, bool live) {
  const int lane = threadIdx.x & 63;
  R vr[RPL];
#pragma unroll
  for (int r = 0; r < RPL; r++) vr[r] = vb[lane + 64 * r];
  R p[CPW];
#pragma unroll
  for (int sl = 0; sl < CPW; sl++) {
    R p0 = 0, p1 = 0;  // two chains halve the dependent FMA latency
#pragma unroll
    for (int r = 0; r < RPL; r += 2) {
      p0 += vr[r] * a[sl][r];
      if (r + 1 < RPL) p1 += vr[r + 1] * a[sl][r + 1];
    }
    p[sl] = p0 + p1;
  }
  R t = wave_total_cols<R, CPW>(p);
  t = live ? tau * t : R(0);
  R tw[CPW];
  spread_cols<R, CPW>(t, tw);
#pragma unroll
  for (int sl = 0; sl < CPW; sl++)
#pragma unroll
    for (int r = 0; r < RPL; r++) a[sl][r] -= tw[sl] * vr[r];
}

// Sum of squares of rows > i of each of this wave's columns (i = -1: all
// rows); lanes 0..CPW-1 return column CPW w + lane.
template <typename R, int RPL, int CPW, int MAXN>
__device__ inline R tail_sq(const R (&a)[CPW][RPL], int i) {
  const int lane = threadIdx.x & 63;
  R p[CPW];
#pragma unroll
  for (int sl = 0; sl < CPW; sl++) {
    p[sl] = 0;
#pragma unroll
    for (int r = 0; r < RPL; r++) {
      // With at most 64 columns, i < 64: registers past the first are
      // below row i.
      if (MAXN <= 64 && r > 0) p[sl] += a[sl][r] * a[sl][r];
      else p[sl] += (lane + 64 * r > i) ? a[sl][r] * a[sl][r] : R(0);
    }
  }
  return class_by_lane_cols<R, CPW>(wave_total_cols<R, CPW>(p));
}

// Row i of this wave's columns into dst[column].  With at most 64 columns
// row i < 64 sits in register 0 of lane i; the wide shape
// reads the row out of every register that can hold it (rows < 128) and
// selects, so that no register is indexed at run time (that would move the
// whole matrix to scratch memory).
template <typename R, int RPL, int CPW, int MAXN>
__device__ inline void publish_row(const R (&a)[CPW][RPL], int i, R* dst) {
  const int lane = threadIdx.x & 63, c0 = CPW * wave_id();
  if constexpr (MAXN <= 64) {
    const int cls = slot_class<CPW>(i);  // lane i's class: uniform addresses
    if (lane == i) {
#pragma unroll
      for (int sl = 0; sl < CPW; sl++) dst[c0 + (sl ^ cls)] = a[sl][0];
    }
  } else {
    constexpr int NR = (MAXN + 63) / 64 < RPL ? (MAXN + 63) / 64 : RPL;
    const int li = i & 63, ri = i >> 6;
    const int cls = slot_class<CPW>(li);
#pragma unroll
    for (int sl = 0; sl < CPW; sl++) {
      R v = lane_value(a[sl][0], li);
#pragma unroll
      for (int r = 1; r < NR; r++) {
        const R t = lane_value(a[sl][r], li);
        v = (r == ri) ? t : v;
      }
      if (lane == 0) dst[c0 + (sl ^ cls)] = v;
    }
  }
}

template <typename R, int RPL, int CPW>
__device__ inline void load_columns(const R* A, int64_t ld, int row0, int rows, int n,
                                    R (&a)[CPW][RPL]) {
  const int lane = threadIdx.x & 63, c0 = CPW * wave_id();
  const int cls = slot_class<CPW>(lane);
#pragma unroll
  for (int sl = 0; sl < CPW; sl++) {
    const int c = c0 + (sl ^ cls);
#pragma unroll
    for (int r = 0; r < RPL; r++) {
      const int i = lane + 64 * r;
      a[sl][r] = (c < n && i < rows) ? A[row0 + i + ld * c] : R(0);
    }
  }
}

// Entries of rows [row0, row0 + rows) of a box's ID matrix, evaluated into
// the interleave (range row i on lane i % 64, register i / 64).  The wave's
// columns are read once as wave-uniform values (scalar loads); each row's
// entries are formed in natural column order and then placed in the
// interleaved slots.
template <typename R, int RPL, int CPW>
__device__ inline void eval_columns(const DevGeom& g, const int* act, const int* rowdofs,
                                    int cnt, const double (*pxy)[kNumProxy], double pw,
                                    int row0, int rows, int n, R (&a)[CPW][RPL]) {
  const int lane = threadIdx.x & 63, c0 = CPW * wave_id();
  const int cls = slot_class<CPW>(lane);
  DofGeo cg[CPW];
#pragma unroll
  for (int q = 0; q < CPW; q++) cg[q] = dof_geo(g, act[min(c0 + q, n - 1)]);
#pragma unroll
  for (int r = 0; r < RPL; r++) {
    const int i = lane + 64 * r;
    R nat[CPW];
#pragma unroll
    for (int q = 0; q < CPW; q++) nat[q] = R(0);
    if (i < rows) {
      const IdRow rw = id_row(g, rowdofs, cnt, pxy, pw, row0 + i);
#pragma unroll
      for (int q = 0; q < CPW; q++)
        if (c0 + q < n) nat[q] = static_cast<R>(id_entry(g.pde, rw, cg[q]));
    }
#pragma unroll
    for (int sl = 0; sl < CPW; sl++) {
      const int want = sl ^ cls;
      R v = nat[0];
#pragma unroll
      for (int q = 1; q < CPW; q++) v = (want == q) ? nat[q] : v;
      a[sl][r] = v;
    }
  }
}

// Row compression of a tall ID matrix: chunk q of box b (rows
// [q ch, q ch + rows), ch = ceil(m / chunks)) is reduced by unpivoted
// Householder QR to its n x n triangle R_q, written to rows [q n, q n + n)
// of the box's stack (ld chunks * n, in its scratch slot).  The stack is
// Q^T A for an orthogonal Q, so its pivoted QR has the same R and column
// order as that of A.  Grid-strided over the level's jobs of this shape;
// one barrier per step (double-buffered reflector).
template <typename R, int CPW>
__global__ __launch_bounds__(kXThreads) void k_rowcomp(DevGeom g, DevTree t, DevState s,
                                                       int start, int level) {
  constexpr int RPL = RegShape<CPW>::RPL, MAXM = RegShape<CPW>::MAXM;
  constexpr int MAXN = RegShape<CPW>::MAXN;
  constexpr int kind = CPW == 4 ? kQrcpStack : kQrcpStack8;
  __shared__ R vbuf[2][MAXM];
  __shared__ R sh_tau[2];
  __shared__ int rowdofs[kMaxChunks * kRegMaxRows / 2];
  __shared__ double pxy[4][kNumProxy];
  __shared__ R rdiag[MAXN];  // R_jj of step j (the register keeps alpha)
  if (!pools_ok(s)) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  const int cls = slot_class<CPW>(lane);
  const int c0 = CPW * wv;
  const int* jobs = s.jobs + (int64_t)2 * kMaxChunks * start;
  // With the randomized ID only its fallbacks need row compression: their
  // (box, chunk) pairs come from the fallback list.
  const bool fb = kind == kQrcpStack && s.rid_mode != 0;
  const int total = fb ? list_count(s, level, kLstFallback) * kMaxChunks : s.njobs[level];
  for (int job = blockIdx.x; job < total; job += gridDim.x) {
    int b, q;
    if (fb) {
      b = list_at(s, start, kLstFallback, job / kMaxChunks);
      q = job % kMaxChunks;
      if (s.qkind[b] != kind || q >= id_chunks(s.m_rows[b], MAXM)) continue;
    } else {
      b = jobs[2 * job];
      q = jobs[2 * job + 1];
      if (s.qkind[b] != kind || s.rid_done[b]) continue;  // rid_done: sketched
    }
    const int n = s.act_cnt[b], m = s.m_rows[b];
    const int nch = id_chunks(m, MAXM);
    const int ch = (m + nch - 1) / nch;
    const int r0 = q * ch, rows = min(ch, m - r0);
    R* S = reinterpret_cast<R*>(s.id_pool) + s.id_off[b];
    const int64_t lds = (int64_t)nch * n;
    const bool active = c0 < n;
    const int* act = s.act_list + (int64_t)b * s.ncap;
    const int cnt = id_setup(g, t, s, b, level, m, rowdofs, pxy);
    __syncthreads();
    R a[CPW][RPL];
    eval_columns<R, RPL, CPW>(g, act, rowdofs, cnt, pxy, proxy_weight(t, b), r0, rows, n, a);
    const int steps = min(rows, n);
    int dmask = 0;
    for (int j = 0; j < steps; j++) {
      if (wv == j / CPW) {
        const int pcls = j % CPW, psl = pcls ^ cls;
        R x[RPL];
        pick_slot<R, RPL, CPW>(a, psl, x);
        const R alpha = row_value<R, RPL>(x, j);
        R ss = 0;
#pragma unroll
        for (int r = 0; r < RPL; r++) ss += (lane + 64 * r > j) ? x[r] * x[r] : R(0);
        R beta, tau, sc;
        householder_scalars(alpha, wave_total(ss), &beta, &tau, &sc);
        write_reflector<R, RPL>(x, j, sc, vbuf[j & 1]);
        dmask |= 1 << pcls;
        if (lane == 0) {
          sh_tau[j & 1] = tau;
          rdiag[j] = beta;
        }
        __builtin_amdgcn_s_setprio(0);
      }
      __syncthreads();
      // Waves whose columns are all reduced are done with the updates; the
      // next pivot column's wave goes first, its reflector being what the
      // next barrier waits for.  Stokes, 16,385 points, learned widths: 3.9
      // ms per factorization with all waves updating in any order, 2.9 so.
      if (active && dmask != (1 << CPW) - 1) {
        if (wv == (j + 1) / CPW) __builtin_amdgcn_s_setprio(3);
        apply_reflector<R, RPL, CPW>(a, vbuf[j & 1], sh_tau[j & 1], ((dmask >> cls) & 1) == 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    // Column c was reduced at step c: rows below its diagonal are zero.
    if (active) {
#pragma unroll
      for (int sl = 0; sl < CPW; sl++) {
        const int c = c0 + (sl ^ cls);
#pragma unroll
        for (int r = 0; r < RPL; r++) {
          const int i = lane + 64 * r;
          if (c < n && i < n)
            S[(int64_t)q * n + i + lds * c] =
                i > c ? R(0) : (i == c && c < steps ? rdiag[c] : a[sl][r]);
        }
      }
    }
    __syncthreads();
  }
}

// Interpolative decomposition by column-pivoted Householder QR, stopped at
// the first |R_jj| < tol |R_00| (ie_mat.cpp:548-588).  The pivot rule,
// Householder form and column-norm downdating follow LAPACK dgeqp3/dlaqp2.
// Lanes 0..CPW-1 of each wave keep the downdated norms, logical position
// and pivot key of the wave's columns; the pivot is the largest key
// (pivot_key), found by one wave maximum; the wave owning the pivot column
// forms the reflector and the stop decision.
template <typename R, int CPW, int RPL, int NW>
__device__ __forceinline__ void qrcp_id_box(const DevGeom& g, const DevTree& t, const DevState& s,
                            int start, int level, int b, double tol_d) {
  constexpr int MAXM = 64 * RPL;
  constexpr int NT = 64 * NW, MAXN = CPW * NW, KH = (MAXN + 63) / 64;
  __shared__ R vbuf[MAXM];
  __shared__ R rowj[MAXN];    // row j after step j (downdating)
  __shared__ R rdiag[MAXN];   // R_jj of step j (the register keeps alpha)
  __shared__ R sh_tau, sh_thresh;
  __shared__ int sh_stop;
  __shared__ double keys[MAXN];
  __shared__ R rbuf[MAXN * MAXN];
  __shared__ int colmap[MAXN];
  __shared__ int rowdofs[MAXM / 2];
  __shared__ double pxy[4][kNumProxy];
  if (s.rid_done[b]) return;  // the wide sketch took it

  const int kind = s.qkind[b];
  const int n = s.act_cnt[b];
  int m = s.m_rows[b];
  const R tol = static_cast<R>(tol_d);
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  const int cls = slot_class<CPW>(lane);
  const int c0 = CPW * wv;
  const bool active = c0 < n;
  const int* act = s.act_list + (int64_t)b * s.ncap;

  R a[CPW][RPL];
  if (kind == kQrcpReg || kind == kQrcpReg8) {
    const int cnt = id_setup(g, t, s, b, level, m, rowdofs, pxy);
    __syncthreads();
    eval_columns<R, RPL, CPW>(g, act, rowdofs, cnt, pxy, proxy_weight(t, b), 0, m, n, a);
  } else {
    // The stacked triangles of the row compression.
    m = id_chunks(m, MAXM) * n;
    load_columns<R, RPL, CPW>(reinterpret_cast<const R*>(s.id_pool) + s.id_off[b], m, 0, m,
                              n, a);
  }
  // Lanes 0..CPW-1: column c0 + lane.
  const int myc = c0 + (lane % CPW);
  R vn1 = 0, vn2 = 0;
  int pos = myc;
  bool avail = lane < CPW && myc < n;
  if (active) {
    vn1 = sqrt(tail_sq<R, RPL, CPW, MAXN>(a, -1));
    vn2 = vn1;
  }
  if (lane < CPW) keys[myc] = avail ? pivot_key(vn1, pos) : -1.0;
  __syncthreads();

  const int kmax = min(m, n);
  int k = kmax;
  R thresh = 0;
  int dmask = 0;  // classes of this wave already pivoted
  for (int j = 0; j < kmax; j++) {
    double kv[KH];
    double best = -1.0;
#pragma unroll
    for (int h = 0; h < KH; h++) {
      kv[h] = (lane + 64 * h < MAXN) ? keys[lane + 64 * h] : -1.0;
      best = fmax(best, kv[h]);
    }
    best = wave_max(best);
    if (!(best >= 0)) {  // every wave sees the same keys
      k = j;
      break;
    }
    int p = -1;
#pragma unroll
    for (int h = KH - 1; h >= 0; h--) {
      const uint64_t hit = __ballot(kv[h] == best);
      if (hit) p = 64 * h + __ffsll((unsigned long long)hit) - 1;
    }
    const int q = pivot_key_pos(best);
    if (lane < CPW) {
      if (myc == p) {
        pos = j;
        avail = false;
      } else if (pos == j) {
        pos = q;
      }
    }
    if (wv == p / CPW) {
      const int psl = (p % CPW) ^ cls;
      R x[RPL];
      pick_slot<R, RPL, CPW>(a, psl, x);
      // With four columns per wave j < 64: row j sits in register 0.
      const R alpha = MAXN <= 64 ? lane_value(x[0], j) : row_value<R, RPL>(x, j);
      R ss = 0;
#pragma unroll
      for (int r = 0; r < RPL; r++) {
        if (MAXN <= 64 && r > 0) ss += x[r] * x[r];
        else ss += (lane + 64 * r > j) ? x[r] * x[r] : R(0);
      }
      R beta, tau, sc;
      householder_scalars(alpha, wave_total(ss), &beta, &tau, &sc);
      write_reflector<R, RPL>(x, j, sc, vbuf);
      const R th = (j == 0) ? fabs(tol * beta) : thresh;
      const int stop = (j >= 1 && fabs(beta) < th) ? 1 : 0;
      if (!stop) dmask |= 1 << (p % CPW);
      if (lane == 0) {
        sh_tau = tau;
        sh_stop = stop;
        rdiag[j] = beta;
        if (j == 0) sh_thresh = th;
      }
    }
    __syncthreads();
    if (sh_stop) {
      k = j;
      break;
    }
    if (j == 0) thresh = sh_thresh;
    if (active) {
      apply_reflector<R, RPL, CPW>(a, vbuf, sh_tau, ((dmask >> cls) & 1) == 0);
      publish_row<R, RPL, CPW, MAXN>(a, j, rowj);
      wave_sync();
      bool need = false;
      if (avail && vn1 != 0) {
        R temp = fabs(rowj[myc]) * recip_any(vn1);
        temp = 1 - temp * temp;
        temp = temp > 0 ? temp : R(0);
        const R rat = vn1 * recip_any(vn2);
        if (temp * rat * rat <= Eps<R>::tol3z) need = true;
        else vn1 = vn1 * sqrt(temp);
      }
      if (__ballot(need)) {  // dlaqp2 recomputes the norm of rows j+1..
        const R t2 = tail_sq<R, RPL, CPW, MAXN>(a, j);
        if (need) {
          const R nv = (j < m - 1) ? sqrt(t2) : R(0);
          vn1 = nv;
          vn2 = nv;
        }
      }
      if (lane < CPW) keys[myc] = avail ? pivot_key(vn1, pos) : -1.0;
    }
    __syncthreads();
  }

  // Logical order and rows 0..k-1 of R (physical column order, ld k).
  if (lane < CPW && myc < n) colmap[pos] = myc;
  if (active) {
#pragma unroll
    for (int sl = 0; sl < CPW; sl++) {
      const int c = c0 + (sl ^ cls);
#pragma unroll
      for (int r = 0; r < RPL; r++) {
        const int i = lane + 64 * r;
        if (c < n && i < k) rbuf[i + k * c] = a[sl][r];
      }
    }
  }
  __syncthreads();
  if (tid < k) {
    rbuf[tid + k * colmap[tid]] = rdiag[tid];
    rdiag[tid] = R(1) / rdiag[tid];  // reciprocal diagonal for the solve below
  }
  __syncthreads();

  int* out = s.out_list + (int64_t)b * s.ncap;
  if (k == 0) {
    for (int i = tid; i < n; i += NT) out[i] = act[i];
    if (tid == 0) {
      s.rank[b] = 0;
      s.out_cnt[b] = n;
    }
    return;
  }
  // T = R11^{-1} R12: one wave per column, lane l holds rows l, l + 64, ...
  const int r = n - k;
  R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
  for (int cp = wv; cp < r; cp += NW) {
    const int pcol = colmap[k + cp];
    R tv[KH];
#pragma unroll
    for (int h = 0; h < KH; h++) {
      const int i = lane + 64 * h;
      tv[h] = (i < k) ? rbuf[i + k * pcol] : R(0);
    }
    for (int i = k - 1; i >= 0; i--) {
      const int ci = colmap[i];
      const R ti = row_value<R, KH>(tv, i) * rdiag[i];
#pragma unroll
      for (int h = 0; h < KH; h++) {
        const int row = lane + 64 * h;
        if (row == i) tv[h] = ti;
        if (row < i) tv[h] -= rbuf[row + k * ci] * ti;
      }
    }
#pragma unroll
    for (int h = 0; h < KH; h++) {
      const int row = lane + 64 * h;
      if (row < k) F[row + (int64_t)k * cp] = tv[h];
    }
  }
  int* red = s.red_list + (int64_t)b * s.ncap;
  int* pm = s.perm + (int64_t)b * s.ncap;
  for (int i = tid; i < n; i += NT) {
    const int c = colmap[i];
    pm[i] = c;
    if (i < k) out[i] = act[c];
    else red[i - k] = act[c];
  }
  if (tid == 0) {
    s.rank[b] = k;
    s.out_cnt[b] = k;
  }
}

// Register shapes (columns per wave x row registers per lane x waves):
// 4 x 8 x 8 for n <= 32 (two boxes share a CU), 4 x 8 x 16 for n <= 64,
// 8 x 4 x 16 for n <= 128 with m <= 256.  Four waves per SIMD are needed to
// hide the FP64 latency of the step loop: an 8 x 8 x 8 shape (256
// registers, two waves per SIMD) measured 22% slower than 4 x 8 x 16.
template <int CPW, int RPL, int NW>
struct QrcpShape {
  static constexpr int kMaxN = CPW * NW;
  static constexpr int kList = kMaxN > 64 ? kLstReg8 : (kMaxN <= 32 ? kLstRegHalf : kLstReg);
  static constexpr int kWavesPerSimd = CPW * RPL > 32 ? 2 : 4;  // register budget
};

// One workgroup per list entry for the n <= 64 shapes (a loop over boxes
// would keep more values live across the step loop than the registers
// hold); the few n <= 128 boxes share a small strided grid, and so do the
// randomized ID's few fallbacks (STRIDE: the loop's spills stay there).
template <typename R, int CPW, int RPL, int NW, bool STRIDE, bool LOOP = true>
__global__ __launch_bounds__(64 * NW, (QrcpShape<CPW, RPL, NW>::kWavesPerSimd)) void k_qrcp_id(
    DevGeom g, DevTree t, DevState s, int start, int level, double tol_d) {
  constexpr int L = QrcpShape<CPW, RPL, NW>::kList;
  if (!pools_ok(s)) return;
  const int nl = list_count(s, level, L);
  if constexpr (!STRIDE) {
    if ((int)blockIdx.x < nl)
      qrcp_id_box<R, CPW, RPL, NW>(g, t, s, start, level, list_at(s, start, L, blockIdx.x), tol_d);
  } else {
    // With the randomized ID the n <= 64 shapes take only its fallbacks.
    const bool fb = L != kLstReg8 && s.rid_mode != 0;
    const int LL = fb ? kLstFallback : L;
    const int cnt = list_count(s, level, LL);
    if constexpr (LOOP) {
      for (int li = blockIdx.x; li < cnt; li += gridDim.x) {
        const int b = list_at(s, start, LL, li);
        if (fb && (L == kLstRegHalf) != (s.act_cnt[b] <= kHalfCols)) continue;
        qrcp_id_box<R, CPW, RPL, NW>(g, t, s, start, level, b, tol_d);
        __syncthreads();
      }
    } else {  // the grid covers the list: one box per workgroup
      if ((int)blockIdx.x >= cnt) return;
      const int b = list_at(s, start, LL, blockIdx.x);
      if (fb && (L == kLstRegHalf) != (s.act_cnt[b] <= kHalfCols)) return;
      qrcp_id_box<R, CPW, RPL, NW>(g, t, s, start, level, b, tol_d);
    }
  }
}

// Both n <= 64 shapes in one launch, for levels of at most kQrcpPairBoxes
// boxes (one workgroup per box, all of them resident): a box of n <= 32
// keeps eight of the sixteen waves.  Each shape's launch lasts as long as
// its slowest box's chain of steps, one behind the other.
// Circle of 4096 points: 50 + 43 us per level, 52 in one launch; star of
// 65,536, levels of up to 256 boxes: 58 + 53 and 76.  With more boxes the
// separate launches pack two n <= 32 boxes into a CU.
constexpr int kQrcpPairBoxes = 256;

template <typename R>
__global__ __launch_bounds__(kXThreads, 4) void k_qrcp_pair(DevGeom g, DevTree t, DevState s,
                                                            int start, int level, double tol_d) {
  if (!pools_ok(s)) return;
  int b;
  if (s.rid_mode != 0) {  // the boxes without a successful sketch
    if ((int)blockIdx.x >= list_count(s, level, kLstFallback)) return;
    b = list_at(s, start, kLstFallback, blockIdx.x);
  } else {
    const int nb = list_count(s, level, kLstReg), i = (int)blockIdx.x - nb;
    if (i >= list_count(s, level, kLstRegHalf)) return;
    b = i < 0 ? list_at(s, start, kLstReg, blockIdx.x) : list_at(s, start, kLstRegHalf, i);
  }
  if (s.act_cnt[b] > kHalfCols) {
    qrcp_id_box<R, 4, 8, 16>(g, t, s, start, level, b, tol_d);
  } else {
    if (wave_id() >= 8) return;
    qrcp_id_box<R, 4, 8, 8>(g, t, s, start, level, b, tol_d);
  }
}

// General form (any box the register form does not take): the matrix lives
// in LDS when it fits, else in the box's scratch slot; each wave owns a
// strided set of columns.
template <typename R, int NT>
__device__ __forceinline__ void qrcp_general_box(const DevState& s, int start, int level, int b, double tol_d) {
  constexpr int NW = NT / 64;
  constexpr int kLdsElems = 131072 / sizeof(R);
  __shared__ R smat[kLdsElems];
  __shared__ R vn1[kMaxBoxDofs];
  __shared__ R vn2[kMaxBoxDofs];
  __shared__ int col[kMaxBoxDofs];
  __shared__ R sh_tau;
  __shared__ int sh_stop;

  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int n = s.act_cnt[b], m = s.m_rows[b];
  const int* act = s.act_list + (int64_t)b * s.ncap;
  int* out = s.out_list + (int64_t)b * s.ncap;
  const R tol = static_cast<R>(tol_d);
  R* A = reinterpret_cast<R*>(s.id_pool) + s.id_off[b];
  const int64_t mn = (int64_t)m * n;
  if (mn <= kLdsElems) {
    for (int64_t i = tid; i < mn; i += NT) smat[i] = A[i];
    A = smat;
  }
  for (int c = tid; c < n; c += NT) col[c] = c;
  __syncthreads();
  for (int c = wv; c < n; c += NW) {
    const R* a = A + (int64_t)m * c;
    R ss = 0;
    for (int i = lane; i < m; i += 64) ss += a[i] * a[i];
    ss = wave_sum(ss);
    if (lane == 0) {
      vn1[c] = sqrt(ss);
      vn2[c] = vn1[c];
    }
  }
  __syncthreads();

  const int kmax = min(m, n);
  int k = 0;
  R thresh = 0;
  for (int j = 0; j < kmax; j++) {
    if (wv == 0) {
      R best = -1;
      int bi = n;
      for (int q = j + lane; q < n; q += 64) {
        const R v = vn1[q];
        if (v > best) {
          best = v;
          bi = q;
        }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const R ob = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if (bi >= n) bi = j;  // all-NaN column norms: keep the current column
      const int cj = col[j], cb = col[bi];
      const R v1 = vn1[j], v2 = vn2[j];
      wave_sync();
      if (lane == 0 && bi != j) {
        col[j] = cb;
        col[bi] = cj;
        vn1[bi] = v1;
        vn2[bi] = v2;
      }
      const int pc = (bi != j) ? cb : cj;
      R* v = A + (int64_t)m * pc;
      const R alpha = v[j];
      R ss = 0;
      for (int i = j + 1 + lane; i < m; i += 64) ss += v[i] * v[i];
      ss = wave_sum(ss);
      const R xnorm = sqrt(ss);
      R beta, tau;
      if (xnorm == 0) {
        tau = 0;
        beta = alpha;
      } else {
        beta = -copysign(hypot(alpha, xnorm), alpha);
        tau = (beta - alpha) / beta;
        const R sc = 1 / (alpha - beta);
        for (int i = j + 1 + lane; i < m; i += 64) v[i] *= sc;
      }
      if (j == 0) thresh = fabs(tol * beta);
      const int stop = (j >= 1 && fabs(beta) < thresh) ? 1 : 0;
      if (lane == 0) {
        if (!stop) v[j] = beta;
        sh_tau = tau;
        sh_stop = stop;
      }
    }
    __syncthreads();
    if (sh_stop) {
      k = j;
      break;
    }
    const R tau = sh_tau;
    const R* v = A + (int64_t)m * col[j];
    for (int q = j + 1 + wv; q < n; q += NW) {
      R* cq = A + (int64_t)m * col[q];
      R part = 0;
      for (int i = j + 1 + lane; i < m; i += 64) part += v[i] * cq[i];
      part = wave_sum(part);
      const R w = cq[j] + part;
      const R tw = tau * w;
      for (int i = j + 1 + lane; i < m; i += 64) cq[i] -= tw * v[i];
      const R rjc = cq[j] - tw;
      wave_sync();
      if (lane == 0) cq[j] = rjc;
      const R v1 = vn1[q];
      if (v1 != 0) {
        R temp = fabs(rjc) / v1;
        temp = 1 - temp * temp;
        temp = temp > 0 ? temp : R(0);
        const R rat = v1 / vn2[q];
        const R temp2 = temp * rat * rat;
        if (temp2 <= Eps<R>::tol3z) {
          R ss2 = 0;
          for (int i = j + 1 + lane; i < m; i += 64) ss2 += cq[i] * cq[i];
          ss2 = wave_sum(ss2);
          const R nv = (j < m - 1) ? sqrt(ss2) : R(0);
          if (lane == 0) {
            vn1[q] = nv;
            vn2[q] = nv;
          }
        } else if (lane == 0) {
          vn1[q] = v1 * sqrt(temp);
        }
      }
    }
    __syncthreads();
  }
  if (k == 0) {
    for (int i = tid; i < n; i += NT) out[i] = act[i];
    if (tid == 0) {
      s.rank[b] = 0;
      s.out_cnt[b] = n;
    }
    return;
  }
  // T = R11^{-1} R12 (k x r), one thread per column, back substitution.
  const int r = n - k;
  R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
  for (int c = tid; c < r; c += NT) {
    const R* y = A + (int64_t)m * col[k + c];
    R* tc = F + (int64_t)k * c;
    for (int i = k - 1; i >= 0; i--) {
      R acc = y[i];
      for (int l = i + 1; l < k; l++) acc -= A[i + (int64_t)m * col[l]] * tc[l];
      tc[i] = acc / A[i + (int64_t)m * col[i]];
    }
  }
  int* red = s.red_list + (int64_t)b * s.ncap;
  int* pm = s.perm + (int64_t)b * s.ncap;
  for (int i = tid; i < n; i += NT) {
    const int c = col[i];
    pm[i] = c;
    if (i < k) out[i] = act[c];
    else red[i - k] = act[c];
  }
  if (tid == 0) {
    s.rank[b] = k;
    s.out_cnt[b] = k;
  }
}

template <typename R, int NT>
__global__ __launch_bounds__(NT) void k_qrcp(DevState s, int start, int level, double tol_d) {
  if (!pools_ok(s)) return;
  const int nl = list_count(s, level, kLstLds);
  for (int li = blockIdx.x; li < nl; li += gridDim.x) {
    const int b = list_at(s, start, kLstLds, li);
    if (s.rid_done[b]) continue;  // the wide sketch took it
    qrcp_general_box<R, NT>(s, start, level, b, tol_d);
    __syncthreads();
  }
}

}  // namespace

template <typename R>
void launch_qrcp(const DevGeom& g, const DevTree& t, const DevState& s, int level, int start,
                 int listed, double tol, const LaunchCaps& caps, hipStream_t st, int skip) {
  // A register-QRCP kernel whose grid covers its whole list (known from
  // the level's box listed) runs one box per workgroup, without the
  // grid-stride loop and the registers it keeps live (no spills).
  const int jobs_max = listed * kMaxChunks;
  if (skip & kSkipRegQrcp) {
    // no register-QRCP box on this level (launch plan)
  } else if (s.rid_mode != 0) {
    // Only the boxes without a successful sketch reach the full QRCP.
    k_rowcomp<R, 4><<<min(jobs_max, caps.rowcomp4), kXThreads, 0, st>>>(g, t, s, start,
                                                                        level);
    if (listed <= min(kQrcpPairBoxes, caps.qrcp_id)) {
      k_qrcp_pair<R><<<listed, kXThreads, 0, st>>>(g, t, s, start, level, tol);
    } else if (listed <= caps.qrcp_id) {
      k_qrcp_id<R, 4, 8, 8, true, false><<<listed, 512, 0, st>>>(g, t, s, start, level, tol);
      k_qrcp_id<R, 4, 8, 16, true, false><<<listed, kXThreads, 0, st>>>(g, t, s, start,
                                                                       level, tol);
    } else {
      const int grid = caps.qrcp_id;
      k_qrcp_id<R, 4, 8, 8, true><<<grid, 512, 0, st>>>(g, t, s, start, level, tol);
      k_qrcp_id<R, 4, 8, 16, true><<<grid, kXThreads, 0, st>>>(g, t, s, start, level, tol);
    }
  } else {
    k_rowcomp<R, 4><<<min(2 * listed, caps.rowcomp4), kXThreads, 0, st>>>(g, t, s, start,
                                                                        level);
    if (listed <= kQrcpPairBoxes) {
      k_qrcp_pair<R><<<listed, kXThreads, 0, st>>>(g, t, s, start, level, tol);
    } else {
      k_qrcp_id<R, 4, 8, 8, false><<<listed, 512, 0, st>>>(g, t, s, start, level, tol);
      k_qrcp_id<R, 4, 8, 16, false><<<listed, kXThreads, 0, st>>>(g, t, s, start, level, tol);
    }
  }
  if (!(skip & kSkipReg8Qrcp)) {
    k_rowcomp<R, 8><<<min(2 * listed, caps.rowcomp8), kXThreads, 0, st>>>(g, t, s, start,
                                                                        level);
    if (listed <= caps.qrcp_id8)
      k_qrcp_id<R, 8, 4, 16, true, false><<<listed, kXThreads, 0, st>>>(g, t, s, start,
                                                                       level, tol);
    else
      k_qrcp_id<R, 8, 4, 16, true><<<caps.qrcp_id8, kXThreads, 0, st>>>(g, t, s, start,
                                                                        level, tol);
  }
  if (!(skip & kSkipAssemble))
    k_qrcp<R, 512><<<min(listed, caps.qrcp), 512, 0, st>>>(s, start, level, tol);
}

template void launch_qrcp<double>(const DevGeom&, const DevTree&, const DevState&, int, int, int,
                                  double, const LaunchCaps&, hipStream_t, int);
template void launch_qrcp<float>(const DevGeom&, const DevTree&, const DevState&, int, int, int,
                                 double, const LaunchCaps&, hipStream_t, int);

}  // namespace iegpu
