// Decouple of the boxes with four or more waves each
// (skel_factorization.cpp:77-128, 323-381) and the root blocks
// (:172-186): assembly, and the one-workgroup inverse of a batch's roots.

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "rs_device.hpp"
#include "rs_id.hpp"
#include "rs_inv.hpp"
#include "rs_kernels.hpp"

namespace iegpu {

namespace {

// ---------------------------------------------------------------------------
// Gauss-Jordan inversion with partial pivoting.  Step j pivots on the row
// with the largest |entry| of column j among rows not yet pivoted (first
// index on ties, LAPACK dgetrf's choice) without moving rows: with pivot
// row prow[j] at step j the result M satisfies
//   X^{-1}(j, prow[jj]) = M(prow[j], jj).
// Steps alternate between two n x n buffers (ld n) starting in `a`, so M
// lands in `a` for even n and in `b` for odd n.  All NT threads take part;
// every wave picks the pivot itself, so a step needs one barrier.
// Returns 0, or j + 1 for the first zero pivot.  n <= 2048.
// ---------------------------------------------------------------------------

template <typename R, int NT>
__device__ int gj_invert(R* a, R* b, int n, int* prow) {
  const int tid = threadIdx.x, lane = tid & 63;
  uint32_t used = 0;  // bit u: row lane + 64 u already pivoted
  int info = 0;
  R* cur = a;
  R* nxt = b;
  const int i0 = tid % n, c0 = tid / n, di = NT % n, dc = NT / n;
  for (int j = 0; j < n; j++) {
    R best = -1;
    int bi = 0x7fffffff;
    for (int u = 0; lane + 64 * u < n; u++) {
      if ((used >> u) & 1) continue;
      const int i = lane + 64 * u;
      const R v = fabs(cur[i + (int64_t)n * j]);
      const R key = (v == v) ? v : R(-0.5);  // NaN rows after all others
      if (key > best) {
        best = key;
        bi = i;
      }
    }
    const int p = wave_argmax<R>(best, bi);
    if ((p & 63) == lane) used |= 1u << (p >> 6);
    if (tid == 0) prow[j] = p;
    const R piv = cur[p + (int64_t)n * j];
    if (piv == R(0) && info == 0) info = j + 1;
    const R inv = R(1) / piv;
    int i = i0, c = c0;
    while (c < n) {
      const int64_t idx = i + (int64_t)n * c;
      const R rp = ((c == j) ? R(1) : cur[p + (int64_t)n * c]) * inv;
      nxt[idx] = (i == p) ? rp : ((c == j) ? R(0) : cur[idx]) - cur[i + (int64_t)n * j] * rp;
      i += di;
      c += dc;
      if (i >= n) {
        i -= n;
        c++;
      }
    }
    __syncthreads();
    R* t = cur;
    cur = nxt;
    nxt = t;
  }
  return info;
}

// Gauss-Jordan inverse of X (r x r, r <= 16 U, in LDS or global memory,
// ld r) with the matrix in the registers of 256 threads on a 16 x 16 grid,
// thread (tr, tc) holding rows tr + 16 u and columns tc + 16 v (U x U
// entries).  Per step:
//   * every thread reads its rows of the pivot column (kept in LDS by its
//     owners) and the pivot row is the largest packed key (same rule as
//     gj_invert) over the 16 lanes of its DPP row, which together hold all
//     16 U rows, so every lane finds it without a block barrier;
//   * the pivot and the pivot row's entries that a thread needs (columns
//     tc + 16 v) are held by lane tr = p % 16 of the same 16-lane group,
//     read with a lane permute (no LDS store, no barrier);
//   * each entry takes one FMA; column j restarts from zero and the pivot
//     row becomes the scaled pivot row;
//   * the owners of column j + 1 publish it, then one block barrier.
// M (as gj_invert) is written back to X.  colbuf holds 2 x 16 U entries.
// Returns 0, or j + 1 for the first zero pivot.
template <typename R, int U = 4>
__device__ __forceinline__ int gj_invert_regs(R* X, int r, int* prow, R* colbuf) {
  constexpr int RM = 16 * U;
  const int tid = threadIdx.x;
  const int tr = tid & 15, tc = tid >> 4;
  R a[U][U];
#pragma unroll
  for (int u = 0; u < U; u++)
#pragma unroll
    for (int v = 0; v < U; v++) {
      const int i = tr + 16 * u, c = tc + 16 * v;
      a[u][v] = (i < r && c < r) ? X[i + r * c] : R(0);
    }
  if (tc == 0) {
#pragma unroll
    for (int u = 0; u < U; u++)
      if (tr + 16 * u < r) colbuf[tr + 16 * u] = a[u][0];
  }
  __syncthreads();
  unsigned used = 0;  // bit u: row tr + 16 u already pivoted
  int info = 0;
  for (int j = 0; j < r; j++) {
    const R* col = colbuf + RM * (j & 1);
    R* coln = colbuf + RM * ((j + 1) & 1);
    R cv[U];
    double key = -1.0;
    unsigned cand = 0;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int row = tr + 16 * u;
      cv[u] = row < r ? col[row] : R(0);
      const bool c = row < r && !((used >> u) & 1);
      cand |= c ? (1u << u) : 0u;
      const R mag = fabs(cv[u]);
      key = fmax(key, (c && mag == mag) ? pivot_key(mag, row) : -1.0);
    }
    key = fmax(key, dpp_f64<dpp::kQuadSwap1, 0xF>(key));
    key = fmax(key, dpp_f64<dpp::kQuadSwap2, 0xF>(key));
    key = fmax(key, dpp_f64<dpp::kRowHalfMirror, 0xF>(key));
    key = fmax(key, dpp_f64<dpp::kRowMirror, 0xF>(key));
    int p;
    if (key >= 0) {
      p = pivot_key_pos(key);
    } else {  // NaN column: the first row not yet pivoted
      int f = cand ? tr + 16 * (__ffs(cand) - 1) : 0x7fffffff;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) f = min(f, __shfl_xor(f, o, 16));
      p = f;
    }
    p = __builtin_amdgcn_readfirstlane(p);  // the same in every lane
    const int up = p >> 4, pr = p & 15;
    if (tr == pr) used |= 1u << up;
    if (tid == 0) prow[j] = p;
    // Lane pr of this 16-lane row holds row p's entries of the row's
    // columns, and cv[up] = the pivot.
    R pc = cv[0];
#pragma unroll
    for (int u = 1; u < U; u++) pc = (u == up) ? cv[u] : pc;
    const int src = (threadIdx.x & 48) | pr;
    const R piv = __shfl(pc, src, 64);
    if (piv == R(0) && info == 0) info = j + 1;
    const R inv = R(1) / piv;
    R rv[U];
#pragma unroll
    for (int v = 0; v < U; v++) {
      const int c = tc + 16 * v;
      R pv = a[0][v];
#pragma unroll
      for (int u = 1; u < U; u++) pv = (u == up) ? a[u][v] : pv;
      pv = __shfl(pv, src, 64);
      rv[v] = c < r ? ((c == j) ? R(1) : pv) * inv : R(0);
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int v = 0; v < U; v++) {
        const bool colj = tc + 16 * v == j, rowp = tr + 16 * u == p;
        const R base = colj ? R(0) : a[u][v];
        const R val = base - cv[u] * rv[v];
        a[u][v] = rowp ? rv[v] : val;
      }
    if (j + 1 < r && tc == ((j + 1) & 15)) {
      const int vn = (j + 1) >> 4;
#pragma unroll
      for (int u = 0; u < U; u++) {
        R x = a[u][0];
#pragma unroll
        for (int v = 1; v < U; v++) x = (v == vn) ? a[u][v] : x;
        if (tr + 16 * u < r) coln[tr + 16 * u] = x;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < U; u++)
#pragma unroll
    for (int v = 0; v < U; v++) {
      const int i = tr + 16 * u, c = tc + 16 * v;
      if (i < r && c < r) X[i + r * c] = a[u][v];
    }
  __syncthreads();
  return info;
}

// Inverts X (r x r) in place through the scratch buffer W (>= r^2): the
// steps start in W when r is odd, so M ends in X.
template <typename R, int NT>
__device__ int gj_invert_into(R* X, R* W, int r, int* prow) {
  if (r & 1) {
    for (int idx = threadIdx.x; idx < r * r; idx += NT) W[idx] = X[idx];
    __syncthreads();
    return gj_invert<R, NT>(W, X, r, prow);
  }
  return gj_invert<R, NT>(X, W, r, prow);
}

// Carried Schur block of child q at (local i, local j); 0 outside the
// child's diagonal block.
template <typename R>
struct ChildUpdates {
  // The four child blocks and sizes stay in LDS (indexing a private copy
  // by the runtime child id would place it in scratch memory).
  const R* const* S;
  const int* N;
  const signed char* pch;
  const short* ploc;
  __device__ R operator()(int i, int j) const {
    const int q = pch[i];
    if (q < 0 || q != pch[j] || S[q] == nullptr) return R(0);
    return S[q][ploc[i] + (int64_t)N[q] * ploc[j]];
  }
};



// Children's carried blocks and the position map of a box's active list.
template <typename R>
__device__ void load_child_blocks(const DevTree& t, const DevState& s, int b,
                                  int n, const R** chS, int* chN,
                                  signed char* pch, short* ploc, int NT) {
  const int tid = threadIdx.x;
  const bool leaf = t.leaf[b] != 0;
  if (tid < 4) {
    const int c = leaf ? -1 : t.child[4 * b + tid];
    chS[tid] = (c >= 0) ? carried_block<R>(s, c) : nullptr;
    chN[tid] = (c >= 0) ? s.out_cnt[c] : 0;
  }
  __syncthreads();
  for (int i = tid; i < n; i += NT) {
    int q = -1, loc = 0;
    if (!leaf) {
      for (int u = 0; u < 4; u++) {
        const int p0 = s.chpos[4 * b + u];
        if (i >= p0 && i < p0 + chN[u]) {
          q = u;
          loc = i - p0;
        }
      }
    }
    pch[i] = (signed char)q;
    ploc[i] = (short)loc;
  }
}

// ---------------------------------------------------------------------------
// Decouple one box (skel_factorization.cpp:77-128): with s/r the skeleton
// and redundant positions and K_BN = K(act, act) - (children's carried
// Schur blocks),
//   K_rs = K(r,s) - T^T K(s,s)
//   K_sr = K(s,r) - K(s,s) T
//   X_rr = K(r,r) - T^T K(s,r) - K_rs T
//   L = K_sr X_rr^{-1},  U = X_rr^{-1} K_rs,  schur = K_sr X_rr^{-1} K_rs
// and the box's carried block = (children's update on s,s) + schur.  X_rr
// is inverted by Gauss-Jordan (the reference LU-factors it and solves): the
// factor slot keeps X_rr^{-1}, so L, U, the carried block and the solve's
// diagonal step are plain products.  Uncompressed boxes carry their
// children's blocks unchanged.
// ---------------------------------------------------------------------------

// P (n x n, skeleton positions first) -> K_rs, K_sr, X_rr.
// sum_l a[sa l] b[sb l], l < len, in four partial sums (a dependent FP64
// FMA chain costs its latency per term; global operands add a load
// latency per term besides).
template <typename R>
__device__ inline R dot2(const R* a, int64_t sa, const R* b, int64_t sb, int len) {
  R s0 = 0, s1 = 0, s2 = 0, s3 = 0;
  int l = 0;
  for (; l + 4 <= len; l += 4) {
    s0 += a[sa * l] * b[sb * l];
    s1 += a[sa * (l + 1)] * b[sb * (l + 1)];
    s2 += a[sa * (l + 2)] * b[sb * (l + 2)];
    s3 += a[sa * (l + 3)] * b[sb * (l + 3)];
  }
  for (; l < len; l++) s0 += a[sa * l] * b[sb * l];
  return (s0 + s1) + (s2 + s3);
}

template <typename R, int NT>
__device__ void decouple_blocks(const R* P, const R* T, int n, int k, R* Krs, R* Ksr, R* X) {
  const int tid = threadIdx.x, r = n - k;
  for (int idx = tid; idx < r * k; idx += NT) {
    const int i = idx % r, a = idx / r;
    Krs[idx] = P[(k + i) + (int64_t)n * a] - dot2(T + k * i, 1, P + (int64_t)n * a, 1, k);
  }
  for (int idx = tid; idx < k * r; idx += NT) {
    const int a = idx % k, j = idx / k;
    Ksr[idx] = P[a + (int64_t)n * (k + j)] - dot2(P + a, n, T + k * j, 1, k);
  }
  __syncthreads();
  for (int idx = tid; idx < r * r; idx += NT) {
    const int i = idx % r, j = idx / r;
    X[idx] = P[(k + i) + (int64_t)n * (k + j)] - dot2(T + k * i, 1, P + (int64_t)n * (k + j), 1, k) -
             dot2(Krs + i, r, T + k * j, 1, k);
  }
  __syncthreads();
}

// From M / prow of gj_invert on X_rr: U, L, X_rr^{-1} and the carried block
// into the factor slot.  W has room for r k entries; uss, when given, holds
// the children's updates on the skeleton block (k x k), else upd forms them.
template <typename R, int NT, typename Upd>
__device__ void decouple_tail(const R* M, const int* prow, const R* Krs, const R* Ksr,
                              R* W, int r, int k, R* F, const FacLayout& fl,
                              const Upd& upd, const short* sperm, const R* uss = nullptr) {
  const int tid = threadIdx.x;
  for (int idx = tid; idx < r * k; idx += NT) {  // U = X^{-1} K_rs
    const int j = idx % r, a = idx / r;
    const R* mrow = M + prow[j];
    const R* kc = Krs + (int64_t)r * a;
    R s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    int jj = 0;
    for (; jj + 4 <= r; jj += 4) {
      s0 += mrow[(int64_t)r * jj] * kc[prow[jj]];
      s1 += mrow[(int64_t)r * (jj + 1)] * kc[prow[jj + 1]];
      s2 += mrow[(int64_t)r * (jj + 2)] * kc[prow[jj + 2]];
      s3 += mrow[(int64_t)r * (jj + 3)] * kc[prow[jj + 3]];
    }
    for (; jj < r; jj++) s0 += mrow[(int64_t)r * jj] * kc[prow[jj]];
    const R acc = (s0 + s1) + (s2 + s3);
    W[idx] = acc;
    F[fl.U + idx] = acc;
  }
  for (int idx = tid; idx < k * r; idx += NT) {  // L = K_sr X^{-1}
    const int a = idx % k, jj = idx / k;
    const R* mcol = M + (int64_t)r * jj;
    R s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    int j = 0;
    for (; j + 4 <= r; j += 4) {
      s0 += Ksr[a + (int64_t)k * j] * mcol[prow[j]];
      s1 += Ksr[a + (int64_t)k * (j + 1)] * mcol[prow[j + 1]];
      s2 += Ksr[a + (int64_t)k * (j + 2)] * mcol[prow[j + 2]];
      s3 += Ksr[a + (int64_t)k * (j + 3)] * mcol[prow[j + 3]];
    }
    for (; j < r; j++) s0 += Ksr[a + (int64_t)k * j] * mcol[prow[j]];
    F[fl.L + a + (int64_t)k * prow[jj]] = (s0 + s1) + (s2 + s3);
  }
  for (int idx = tid; idx < r * r; idx += NT) {
    const int j = idx % r, jj = idx / r;
    F[fl.X + j + (int64_t)r * prow[jj]] = M[prow[j] + (int64_t)r * jj];
  }
  __syncthreads();
  for (int idx = tid; idx < k * k; idx += NT) {  // carried block
    const int a = idx % k, c = idx / k;
    const R u = uss ? uss[idx] : upd(sperm[a], sperm[c]);
    F[fl.S + idx] = u + dot2(Ksr + a, k, W + (int64_t)r * c, 1, r);
  }
}

// Compressed boxes with NMIN < |active| <= NMAX (<= 64), every operand in
// LDS.  Only the skeleton rows of K_BN are stored (K(s,s), K(s,r)); the
// redundant rows are evaluated where K_rs and X_rr need them, which keeps
// the buffer at n^2 + 2 k r <= 1.5 NMAX^2 entries: three boxes per CU for
// NMAX = 64, five for NMAX = 44.
template <typename R, int NMIN, int NMAX>
__global__ __launch_bounds__(256) void k_decouple_small(DevGeom g, DevTree t,
                                                        DevState s, int start, int level) {
  constexpr int NT = 256;
  // >= n^2 + 2 k r (k r <= n^2 / 4); the two size classes let the boxes
  // with n <= kSmallBox1 run at a higher occupancy
  constexpr int kBuf = NMAX * NMAX + NMAX * NMAX / 2;
  static_assert(NMAX * sizeof(DofGeo) >= 2 * 64 * sizeof(R), "pivot columns fit in geo");
  __shared__ R buf[kBuf];
  __shared__ DofGeo geo[NMAX];
  __shared__ signed char pch[NMAX];
  __shared__ short ploc[NMAX];
  __shared__ short sperm[NMAX];
  __shared__ int prow[NMAX];
  __shared__ const R* chS[4];
  __shared__ int chN[4];

  const int b = start + blockIdx.x;
  const int tid = threadIdx.x;
  if (s.halt[level] || box_clean(s, b)) return;
  const int n = s.act_cnt[b], k = s.rank[b];
  if (n > NMAX || (n <= NMIN && (NMIN > 0 || n > 0))) return;  // another kernel's box
  if (k == 0) {
    pass_children<R>(t, s, b, n, NT);
    return;
  }
  load_child_blocks<R>(t, s, b, n, chS, chN, pch, ploc, NT);
  const int* act = s.act_list + (int64_t)b * s.ncap;
  for (int i = tid; i < n; i += NT) {
    const int q = s.perm[(int64_t)b * s.ncap + i];
    sperm[i] = (short)q;
    geo[i] = dof_geo(g, act[q]);
  }
  __syncthreads();
  ChildUpdates<R> upd;
  upd.S = chS;
  upd.N = chN;
  upd.pch = pch;
  upd.ploc = ploc;
  const int r = n - k;
  const FacLayout fl = FacLayout::make(k, r);
  R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
  // K_BN entry at permuted positions (skeleton first).
  auto kbn = [&](int i, int c) -> R {
    return static_cast<R>(kernel_entry(g.pde, geo[i], geo[c])) - upd(sperm[i], sperm[c]);
  };
  R* Pss = buf;          // k x k
  R* Psr = Pss + k * k;  // k x r
  R* T = Psr + k * r;    // k x r
  R* X = T + k * r;      // r x r
  R* Krs = X + r * r;    // r x k
  R* Ksr = Krs + r * k;  // k x r
  for (int idx = tid; idx < k * r; idx += NT) T[idx] = F[fl.T + idx];
  for (int idx = tid; idx < k * n; idx += NT) {
    const int a = idx % k, c = idx / k;  // Pss and Psr are contiguous (ld k)
    Pss[idx] = kbn(a, c);
  }
  __syncthreads();
  for (int idx = tid; idx < r * k; idx += NT) {  // K_rs = K(r,s) - T^T K(s,s)
    const int i = idx % r, a = idx / r;
    Krs[idx] = kbn(k + i, a) - dot2(T + k * i, 1, Pss + k * a, 1, k);
  }
  for (int idx = tid; idx < k * r; idx += NT) {  // K_sr = K(s,r) - K(s,s) T
    const int a = idx % k, j = idx / k;
    Ksr[idx] = Psr[idx] - dot2(Pss + a, k, T + k * j, 1, k);
  }
  __syncthreads();
  for (int idx = tid; idx < r * r; idx += NT) {  // X_rr = K(r,r) - T^T K(s,r) - K_rs T
    const int i = idx % r, j = idx / r;
    X[idx] = kbn(k + i, k + j) - dot2(T + k * i, 1, Psr + k * j, 1, k) -
             dot2(Krs + i, r, T + k * j, 1, k);
  }
  __syncthreads();
  if (s.fwd_pool) {
    R* Xf = reinterpret_cast<R*>(s.fwd_pool) + s.fac_off[b];
    for (int idx = tid; idx < r * r; idx += NT) Xf[idx] = X[idx];
  }
  // The DOF geometry is dead: its space holds the pivot columns.
  R* colbuf = reinterpret_cast<R*>(geo);
  const int info = gj_invert_regs<R>(X, r, prow, colbuf);
  if (info != 0 && tid == 0) atomicOr(s.err, kErrSingular);
  decouple_tail<R, NT>(X, prow, Krs, Ksr, buf, r, k, F, fl, upd, sperm);
  if (tid == 0) s.upd_kind[b] = 1;
}

// The boxes above kSmallBox DOFs, walked by a small grid from their list
// (few boxes of a level are these; walking the whole level for them took
// 167 us per factorization at N = 262,144 against 26, and 7.8 ms against 2.3
// for a batch of 256 problems): compressed ones keep P and X_rr in LDS when they fit and in the
// box's scratch slot otherwise, uncompressed ones pass their children's
// blocks on.
constexpr int kDecGeoMax = 96;

template <typename R, int NT>
__global__ __launch_bounds__(NT) void k_decouple(DevGeom g, DevTree t,
                                                 DevState s, int start, int level) {
  // 128 KB: P, X_rr, K_rs and K_sr of a box up to 90 DOFs (FP64) stay in
  // LDS; the Schur products are then LDS-bound, not bound by L2 latency.
  constexpr int kLdsElems = 131072 / sizeof(R);
  __shared__ R sbuf[kLdsElems];
  __shared__ R gjcol[2 * 16 * 8];  // the register Gauss-Jordan's column buffers
  __shared__ DofGeo geo[kDecGeoMax];  // the box's DOFs, permuted, when n fits
  __shared__ signed char pch[kMaxBoxDofs];
  __shared__ short ploc[kMaxBoxDofs];
  __shared__ short sperm[kMaxBoxDofs];
  __shared__ int prow[kMaxBoxDofs];
  __shared__ const R* chS[4];
  __shared__ int chN[4];

  const int tid = threadIdx.x;
  if (s.halt[level]) return;
  const int nl = list_count(s, level, kLstBig);
  for (int bi = blockIdx.x; bi < nl; bi += gridDim.x) {
  const int b = list_at(s, start, kLstBig, bi);
  const int n = s.act_cnt[b];
  if (s.rank[b] == 0) {
    pass_children<R>(t, s, b, n, NT);
    continue;
  }
  __syncthreads();  // the previous box's LDS
  load_child_blocks<R>(t, s, b, n, chS, chN, pch, ploc, NT);
  __syncthreads();
  ChildUpdates<R> upd;
  upd.S = chS;
  upd.N = chN;
  upd.pch = pch;
  upd.ploc = ploc;
  const int k = s.rank[b];
  R* F = reinterpret_cast<R*>(s.fac_pool) + s.fac_off[b];
  const int r = n - k;
  const FacLayout fl = FacLayout::make(k, r);
  const int* act = s.act_list + (int64_t)b * s.ncap;
  const bool lgeo = n <= kDecGeoMax;
  for (int i = tid; i < n; i += NT) {
    const int q = s.perm[(int64_t)b * s.ncap + i];
    sperm[i] = (short)q;
    if (lgeo) geo[i] = dof_geo(g, act[q]);
  }
  __syncthreads();
  // n^2 + r^2 + 2 r k <= 2 n^2 entries.
  R* P = (2 * (int64_t)n * n <= kLdsElems)
             ? sbuf
             : reinterpret_cast<R*>(s.dec_pool) + s.dec_off[b];
  R* X = P + (int64_t)n * n;
  R* Krs = X + (int64_t)r * r;
  R* Ksr = Krs + (int64_t)r * k;
  // T (k x r) and the children's updates on the skeleton block (k x k)
  // join them in LDS when they fit: the Schur products then read no
  // global memory.
  const bool stage = P == sbuf && (int64_t)n * n + (int64_t)r * r + 3 * (int64_t)r * k +
                                          (int64_t)k * k <= kLdsElems;
  R* Tl = Ksr + (int64_t)r * k;
  R* Uss = stage ? Tl + (int64_t)r * k : nullptr;
  if (stage)
    for (int idx = tid; idx < r * k; idx += NT) Tl[idx] = F[fl.T + idx];
  for (int64_t idx = tid; idx < (int64_t)n * n; idx += NT) {
    const int i = (int)(idx % n), c = (int)(idx / n);
    const int ia = sperm[i], ic = sperm[c];
    const R u = upd(ia, ic);
    const double kv = lgeo ? kernel_entry(g.pde, geo[i], geo[c]) : kernel_entry(g, act[ia], act[ic]);
    P[idx] = static_cast<R>(kv) - u;
    if (Uss && i < k && c < k) Uss[i + k * c] = u;
  }
  __syncthreads();
  decouple_blocks<R, NT>(P, stage ? Tl : F + fl.T, n, k, Krs, Ksr, X);
  if (s.fwd_pool) {
    R* Xf = reinterpret_cast<R*>(s.fwd_pool) + s.fac_off[b];
    for (int64_t idx = tid; idx < (int64_t)r * r; idx += NT) Xf[idx] = X[idx];
    __syncthreads();
  }
  // X_rr^{-1}: in registers for r <= 128, else step by step.
  int info;
  if (NT == 256 && r <= 64) info = gj_invert_regs<R, 4>(X, r, prow, gjcol);
  else if (NT == 256 && r <= 128) info = gj_invert_regs<R, 8>(X, r, prow, gjcol);
  else info = gj_invert_into<R, NT>(X, P, r, prow);
  if (info != 0 && tid == 0) atomicOr(s.err, kErrSingular);
  decouple_tail<R, NT>(X, prow, Krs, Ksr, P, r, k, F, fl, upd, sperm, Uss);
  if (tid == 0) s.upd_kind[b] = 1;
  }
}

// ---------------------------------------------------------------------------
// Root: K(allskel, allskel) - carried blocks of the level-1 boxes, inverted.
// ---------------------------------------------------------------------------

// Assembly of root block blockIdx.x: gridDim.y workgroups share its n^2
// entries (one workgroup was latency-bound on the kernel's gathers).
constexpr int kRootSplit = 64;

template <typename R, int NT>
__global__ __launch_bounds__(NT) void k_root(DevGeom g, DevTree t, DevState s) {
  __shared__ signed char pch[kMaxBoxDofs];
  __shared__ short ploc[kMaxBoxDofs];
  __shared__ const R* chS[4];
  __shared__ int chN[4];
  const int b = blockIdx.x;  // root of problem b
  const int tid = threadIdx.x;
  const bool lead = blockIdx.y == 0 && tid == 0;
  if (lead) {  // the root is never compressed
    s.rank[b] = 0;
    s.m_rows[b] = 0;
    s.out_cnt[b] = s.act_cnt[b];
  }
  if (blockIdx.y == 0)  // the block inverse's panel flags
    for (int i = tid; i < kInvFlags; i += NT) root_pivots(s, b)[s.ncap + i] = 0;
  if (b == 0 && lead && s.plan_skip != nullptr) {
    // The launch plan skipped kernels whose lists it expected empty: any
    // that is not makes the host run the factorization again in full.
    for (int lv = 1; lv < t.n_levels; lv++)
      if (s.plan_skip[lv] & ~plan_skippable(s, lv)) {
        atomicOr(s.err, kErrPlan);
        break;
      }
  }
  if (!pools_ok(s)) return;
  const int n = s.act_cnt[b];
  const bool leaf = t.leaf[b] != 0;
  if (tid < 4) {
    const int c = leaf ? -1 : t.child[4 * b + tid];
    chS[tid] = (c >= 0) ? carried_block<R>(s, c) : nullptr;
    chN[tid] = (c >= 0) ? s.out_cnt[c] : 0;
  }
  __syncthreads();
  for (int i = tid; i < n; i += NT) {
    int q = -1, loc = 0;
    if (!leaf) {
      for (int u = 0; u < 4; u++) {
        const int p0 = s.chpos[4 * b + u];
        if (i >= p0 && i < p0 + chN[u]) {
          q = u;
          loc = i - p0;
        }
      }
    }
    pch[i] = (signed char)q;
    ploc[i] = (short)loc;
  }
  __syncthreads();
  ChildUpdates<R> upd;
  upd.S = chS;
  upd.N = chN;
  upd.pch = pch;
  upd.ploc = ploc;
  const int* act = s.act_list + (int64_t)b * s.ncap;
  R* A = root_block<R>(s, b);
  R* Af = s.root_fwd ? reinterpret_cast<R*>(s.root_fwd) + (int64_t)s.ncap * s.ncap * b : nullptr;
  const int64_t nn = (int64_t)n * n, per = (nn + gridDim.y - 1) / gridDim.y;
  const int64_t e0 = per * blockIdx.y, e1 = min(nn, e0 + per);
  for (int64_t idx = e0 + tid; idx < e1; idx += NT) {
    const int i = (int)(idx % n), j = (int)(idx / n);
    const R v = static_cast<R>(kernel_entry(g, act[i], act[j])) - upd(i, j);
    A[idx] = v;
    if (Af) Af[idx] = v;
  }
}

// Gauss-Jordan inverse of the root block with the matrix in registers,
// blocked over panels of kRootPB columns: 1024 threads on a 32 x 32 grid,
// thread (tr, tc) holding rows tr + 32 u and columns tc + 32 v (n <= 192;
// 6 x 6 entries each), so that one wave holds every row of its 12 columns.
// The block is bordered by the identity up to n8, a multiple of kRootPB
// (its pivots stay in the block: border rows hold zeros in its columns and
// lose every tie to a block row), and rows and columns past n8 are zero, so
// no step or entry needs a bound.
//
// Wave 0 runs each panel's pivot steps on the panel's columns alone (they
// depend on nothing else): pivot search as in gj_invert, scaling,
// elimination; it records each step's pivot row p_k, 1 / pivot and the
// column as it was before the step (C[m][i]).  Applying panel P:
//  a. in every wave, the owners of its pivot rows copy them to LDS and one
//     lane per column forms the scaled pivot rows the steps would have
//     made, R_k = (row p_k - sum_{m<k} C[m][p_k] R_m) / pivot_k;
//  b. every thread applies the steps to its entries in step order,
//     a -= C[m][i] R_m, a pivot row restarting from R_k at its own step;
//     panel entries take wave 0's result.
// With one step of lookahead: after (a), the owners of panel P+1's columns
// apply P to a copy of those columns and publish it; after a barrier wave 0
// eliminates panel P+1 from that copy while every wave (wave 0 after it)
// applies P to all its entries; a barrier ends the panel.  Per entry these are the
// operations of the unblocked elimination in its order, so the inverse is
// the same.  The inverse, unpermuted, goes after the assembled matrix.
constexpr int kRootTR = 32, kRootTC = 32, kRootRU = 6, kRootCV = 6;
constexpr int kRootPB = 8;

template <typename R>
__global__ __launch_bounds__(kRootTR * kRootTC) void k_root_inv(DevState s) {
  constexpr int NMAX = kRootRegMax, PB = kRootPB, NS = NMAX / 64;
  static_assert(kRootTC % PB == 0 && NMAX == kRootTR * kRootRU && NMAX == kRootTC * kRootCV &&
                NMAX % 64 == 0 && NMAX % PB == 0 && NMAX <= 256 && PB * PB <= 64,
                "root tiling");
  __shared__ R pan[2][PB][NMAX];   // panel columns, in and out of the elimination
  __shared__ R cpre[2][PB][NMAX];  // column m before step m (zero where row i
                                   // is pivot at a step >= m); by panel parity
  __shared__ R cpiv[2][PB][PB];    // C[m][p_k], m < k
  __shared__ R pinv[2][PB];
  __shared__ R rowk[PB][NMAX];     // pivot rows, then R_k (each wave its columns)
  __shared__ int pstep[NMAX];      // elimination step that pivots on row i
  __shared__ int prow[NMAX];
  __shared__ int invrow[NMAX];
  __shared__ R park[kRootRU * kRootCV][64];
  if (!pools_ok(s)) return;
  const int n = s.act_cnt[blockIdx.x];
  if (n == 0 || n > NMAX) return;
  const int n8 = (n + PB - 1) / PB * PB;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tr = tid % kRootTR, tc = tid / kRootTR;
  R* A = root_block<R>(s, blockIdx.x);
  R a[kRootRU][kRootCV];
#pragma unroll
  for (int u = 0; u < kRootRU; u++)
#pragma unroll
    for (int v = 0; v < kRootCV; v++) {
      const int i = tr + kRootTR * u, c = tc + kRootTC * v;
      a[u][v] = (i < n && c < n) ? A[i + (int64_t)n * c] : (i == c && i < n8) ? R(1) : R(0);
    }
  if (tid < NMAX) pstep[tid] = NMAX;
  // wave 0: bit q set once row lane + 64 q is a pivot row (rows past n8
  // never are)
  uint32_t used = 0;
#pragma unroll
  for (int q = 0; q < NS; q++)
    if (lane + 64 * q >= n8) used |= 1u << q;
  int info = 0;

  // The thread owns panel j0's column in its entries a[.][vj] when
  // tc in [tc0, tc0 + PB) (the same for both halves of a wave).
  auto owns = [&](int j0) { return tc >= j0 % kRootTC && tc < j0 % kRootTC + PB; };
  auto publish = [&](int j0, int pb) {
    const int vj = j0 / kRootTC;
#pragma unroll
    for (int v = 0; v < kRootCV; v++) {
      if (v != vj) continue;
#pragma unroll
      for (int u = 0; u < kRootRU; u++) pan[pb][tc - j0 % kRootTC][tr + kRootTR * u] = a[u][v];
    }
  };
  // wave 0, its own entries parked in LDS meanwhile (the panel and the
  // matrix do not fit its registers)
  auto eliminate = [&](int j0, int pb) {
#pragma unroll
    for (int u = 0; u < kRootRU; u++)
#pragma unroll
      for (int v = 0; v < kRootCV; v++) park[u * kRootCV + v][lane] = a[u][v];
    R x[NS][PB];
#pragma unroll
    for (int q = 0; q < NS; q++)
#pragma unroll
      for (int k = 0; k < PB; k++) x[q][k] = pan[pb][k][lane + 64 * q];
    // pivot keys of column k over the rows not yet pivots (the next
    // column's are formed at the end of each step, beside its updates)
    uint32_t cand = 0;
    auto column_best = [&](int k) {
      // the lane index is formed here each time: kept across the steps,
      // the rows' key bits were spilled
      int l = lane;
      __asm__ volatile("" : "+v"(l));
      double key = -1.0;
      cand = 0;
#pragma unroll
      for (int q = 0; q < NS; q++) {
        const bool ok = !((used >> q) & 1);
        cand |= (ok ? 1u : 0u) << q;
        const R v = fabs(x[q][k]);
        const double kq = pivot_key<R, 8>(v, l + 64 * q);
        key = fmax(key, (ok && v == v) ? kq : -1.0);
      }
      return wave_max(key);
    };
    double best = column_best(0);
#pragma unroll
    for (int k = 0; k < PB; k++) {
      int p;
      if (best >= 0) {
        p = pivot_key_pos<8>(best);
      } else {  // NaN column: the first row not yet pivoted
        p = 0x7fffffff;
#pragma unroll
        for (int q = 0; q < NS; q++) {
          const uint64_t m = __ballot((cand >> q) & 1);
          if (m && p == 0x7fffffff) p = 64 * q + __ffsll((unsigned long long)m) - 1;
        }
      }
      const int pq = p >> 6, pl = p & 63;
      // the pivot row's panel entries, in every lane
      R xp[PB];
#pragma unroll
      for (int k2 = 0; k2 < PB; k2++) {
        R v = x[0][k2];
#pragma unroll
        for (int q = 1; q < NS; q++)
          if (pq == q) v = x[q][k2];
        xp[k2] = lane_value(v, pl);
      }
      const R piv = xp[k];
      if (piv == R(0) && info == 0) info = j0 + k + 1;
      const R inv = R(1) / piv;
      if (lane == 0) {
        pinv[pb][k] = inv;
        prow[j0 + k] = p;
        pstep[p] = j0 + k;
      }
#pragma unroll
      for (int q = 0; q < NS; q++) cpre[pb][k][lane + 64 * q] = x[q][k];
      R rv[PB];
#pragma unroll
      for (int k2 = 0; k2 < PB; k2++) rv[k2] = (k2 == k ? R(1) : xp[k2]) * inv;
#pragma unroll
      for (int q = 0; q < NS; q++) {
        const R c = x[q][k];
        x[q][k] = R(0);
#pragma unroll
        for (int k2 = 0; k2 < PB; k2++) x[q][k2] -= c * rv[k2];
      }
      if (lane == pl) {
        used |= 1u << pq;
#pragma unroll
        for (int q = 0; q < NS; q++)
          if (q == pq) {
#pragma unroll
            for (int k2 = 0; k2 < PB; k2++) x[q][k2] = rv[k2];
          }
      }
      if (k + 1 < PB) best = column_best(k + 1);
      __builtin_amdgcn_sched_barrier(0);  // one step's registers at a time
    }
#pragma unroll
    for (int q = 0; q < NS; q++)
#pragma unroll
      for (int k = 0; k < PB; k++) pan[pb][k][lane + 64 * q] = x[q][k];
    // C at the pivot rows, one (step k, step m <= k) pair per lane: the
    // steps before a row's own step go to cpiv (they form R_k), cpre
    // keeps only the steps after it
    if (lane < PB * PB) {
      const int k = lane / PB, m = lane % PB;
      if (m <= k) {
        const int pk = prow[j0 + k];
        if (m < k) cpiv[pb][k][m] = cpre[pb][m][pk];
        cpre[pb][m][pk] = R(0);
      }
    }
#pragma unroll
    for (int u = 0; u < kRootRU; u++)
#pragma unroll
      for (int v = 0; v < kRootCV; v++) a[u][v] = park[u * kRootCV + v][lane];
  };

  // prologue: panel 0 eliminated
  if (owns(0)) publish(0, 0);
  __syncthreads();
  if (wave == 0) eliminate(0, 0);
  __syncthreads();
  for (int j0 = 0, pb = 0; j0 < n8; j0 += PB, pb ^= 1) {
    const int j1 = j0 + PB, pn = pb ^ 1;
    const bool nxt = j1 < n8;
    // a. the wave's pivot rows of panel j0, then R_k for the wave's columns
    int kk[kRootRU];
#pragma unroll
    for (int u = 0; u < kRootRU; u++) {
      const int q = pstep[tr + kRootTR * u] - j0;
      kk[u] = (q >= 0 && q < PB) ? q : -1;
      if (kk[u] >= 0) {
#pragma unroll
        for (int v = 0; v < kRootCV; v++) rowk[kk[u]][tc + kRootTC * v] = a[u][v];
      }
    }
    wave_sync();
    if (lane < 2 * kRootCV) {
      const int c = (tc & ~1) + (lane & 1) + kRootTC * (lane >> 1);
      R r[PB];
#pragma unroll
      for (int k = 0; k < PB; k++) {
        R t = rowk[k][c];
#pragma unroll
        for (int m = 0; m < k; m++) t -= cpiv[pb][k][m] * r[m];
        r[k] = t * pinv[pb][k];
        rowk[k][c] = r[k];
      }
    }
    wave_sync();
    // lookahead: panel j1's columns take panel j0's steps (as in b, which
    // repeats them on the thread's entries) and are published
    if (nxt && owns(j1)) {
      const int v1 = j1 / kRootTC;
#pragma unroll
      for (int v = 0; v < kRootCV; v++) {
        if (v != v1) continue;
        const int c = tc + kRootTC * v;
        R col[kRootRU];
#pragma unroll
        for (int u = 0; u < kRootRU; u++) col[u] = kk[u] >= 0 ? rowk[kk[u]][c] : a[u][v];
#pragma unroll
        for (int m = 0; m < PB; m++) {
          const R rv = rowk[m][c];
#pragma unroll
          for (int u = 0; u < kRootRU; u++) col[u] -= cpre[pb][m][tr + kRootTR * u] * rv;
        }
#pragma unroll
        for (int u = 0; u < kRootRU; u++) pan[pn][tc - j1 % kRootTC][tr + kRootTR * u] = col[u];
      }
    }
    __syncthreads();
    if (wave == 0 && nxt) eliminate(j1, pn);
    // b. panel j0's steps on the thread's entries (the pivot steps of panel
    // j1 are after j0's in pstep: kk formed again, not kept across)
#pragma unroll
    for (int u = 0; u < kRootRU; u++) {
      const int q = pstep[tr + kRootTR * u] - j0;
      kk[u] = (q >= 0 && q < PB) ? q : -1;
    }
#pragma unroll
    for (int u = 0; u < kRootRU; u++) {
      if (kk[u] < 0) continue;
#pragma unroll
      for (int v = 0; v < kRootCV; v++) a[u][v] = rowk[kk[u]][tc + kRootTC * v];
    }
#pragma unroll
    for (int m = 0; m < PB; m++) {
      R cv[kRootRU], rv[kRootCV];
#pragma unroll
      for (int u = 0; u < kRootRU; u++) cv[u] = cpre[pb][m][tr + kRootTR * u];
#pragma unroll
      for (int v = 0; v < kRootCV; v++) rv[v] = rowk[m][tc + kRootTC * v];
#pragma unroll
      for (int u = 0; u < kRootRU; u++)
#pragma unroll
        for (int v = 0; v < kRootCV; v++) a[u][v] -= cv[u] * rv[v];
    }
    if (owns(j0)) {
      const int vj = j0 / kRootTC;
#pragma unroll
      for (int v = 0; v < kRootCV; v++) {
        if (v != vj) continue;
#pragma unroll
        for (int u = 0; u < kRootRU; u++) a[u][v] = pan[pb][tc - j0 % kRootTC][tr + kRootTR * u];
      }
    }
    __syncthreads();
  }
  if (tid < n8) invrow[prow[tid]] = tid;
  __syncthreads();
  R* B = A + (int64_t)n * n;
#pragma unroll
  for (int u = 0; u < kRootRU; u++)
#pragma unroll
    for (int v = 0; v < kRootCV; v++) {
      const int i = tr + kRootTR * u, c = tc + kRootTC * v;
      if (i < n && c < n) B[invrow[i] + (int64_t)n * prow[c]] = a[u][v];
    }
  if (info != 0 && tid == 0) atomicOr(s.err, kErrSingular);
}

}  // namespace

template <typename R>
void launch_decouple(const DevGeom& g, const DevTree& t, const DevState& s, int level, int start,
                     int count, int listed, const LaunchCaps& caps, hipStream_t st, int skip,
                     hipStream_t st_big) {
  if (count >= caps.dsweep) {  // one wave per box with |active| <= 64
    launch_decouple_sweep<R>(g, t, s, level, start, count, st);
  } else if (count >= caps.dsplit) {
    k_decouple_small<R, 0, kSmallBox1><<<count, 256, 0, st>>>(g, t, s, start, level);
    k_decouple_small<R, kSmallBox1, kSmallBox><<<count, 256, 0, st>>>(g, t, s, start, level);
  } else {
    k_decouple_small<R, 0, kSmallBox><<<count, 256, 0, st>>>(g, t, s, start, level);
  }
  // the boxes above the small-box bound on st_big when given (their
  // own stream: the two kernels touch different boxes), there with
  // 1024 threads (level 1's two 84-DOF boxes: the P fill 47k -> 16k
  // cycles, 12 % less in all)
  if (skip & kSkipDecBig) {
    // no such box on this level (launch plan)
  } else if (st_big) {
    k_decouple<R, 1024><<<min(listed, 512), 1024, 0, st_big>>>(g, t, s, start, level);
  } else {
    k_decouple<R, 256><<<min(listed, 512), 256, 0, st>>>(g, t, s, start, level);
  }
}

template <typename R>
void launch_root(const DevGeom& g, const DevTree& t, const DevState& s,
                 int n_roots, bool factor_lu, hipStream_t st) {
  launch_active(t, s, 0, n_roots, st);
  k_root<R, 256><<<dim3(n_roots, kRootSplit), 256, 0, st>>>(g, t, s);
  if (!factor_lu) return;  // with holes the bordered system holds the root block
  // A batch inverts the blocks that fit one workgroup's registers there (one
  // workgroup per root fills the chip: 256 roots of about 130 DOFs take 253
  // us, 1,721 us over many workgroups each); a few roots leave it idle and
  // take the panels of k_inv_panel at every size (150 DOFs: 195 against 210
  // us, 12 DOFs: 19 against 28 us).
  const int one_wg = n_roots >= kRootBatch ? kRootRegMax : 0;
  if (one_wg) k_root_inv<R><<<n_roots, kRootTR * kRootTC, 0, st>>>(s);
  InvBlocks<R> blk;
  blk.a = reinterpret_cast<R*>(s.root_mat);
  blk.out = nullptr;
  blk.stride = 2 * (int64_t)s.ncap * s.ncap;
  blk.piv = s.root_piv;
  blk.piv_stride = s.ncap + kRootPiv;
  blk.extra = 0;
  launch_block_inverse<R>(s, blk, n_roots, one_wg, s.ncap, st);
}

#define IEGPU_INSTANTIATE_DEC(R)                                                            \
  template void launch_decouple<R>(const DevGeom&, const DevTree&, const DevState&, int, int, \
                                   int, int, const LaunchCaps&, hipStream_t, int, hipStream_t);  \
  template void launch_root<R>(const DevGeom&, const DevTree&, const DevState&, int, bool,  \
                               hipStream_t);

IEGPU_INSTANTIATE_DEC(double)
IEGPU_INSTANTIATE_DEC(float)

}  // namespace iegpu
