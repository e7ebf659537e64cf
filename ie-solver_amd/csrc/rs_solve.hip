// Solve-phase kernels of the RS factorization: the upward and downward
// sweeps, the block-diagonal and root solves (skel_factorization.cpp:388-426,
// 507-592), and the compressed forward apply (:429-504).

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rs_device.hpp"
#include "rs_kernels.hpp"

namespace iegpu {

namespace {

// ---------------------------------------------------------------------------
// Sweeps.  One wave per box (boxes of one level touch disjoint DOFs): the
// box's entries are gathered to LDS, updated and scattered back.
//
// A box is a chain of dependent memory accesses (index list, entries,
// factors), so its factors (T, L or U, X_rr^{-1}: 1 to 8 KB for a typical
// box) are read into LDS by coalesced loads issued beside the gather; the
// products then read LDS only.  Boxes whose factors do not fit read them
// in place.  C columns of a multi-column right-hand side go through the box
// together: lane l works on column l % C and rows l / C, l / C + 64 / C, ...,
// so a factor entry is read once for C columns and few rows still fill the
// wave.  Every row sum is formed by dot_ld in one order whatever C is, so a
// column's result does not depend on the columns beside it.
// Laplace, 262,144 unknowns, 12 levels: up 140, down 107 us for one column
// (187 and 120 with factors read in place); 614 and 303 us for 16 columns
// (1,460 and 869 column by column).
// ---------------------------------------------------------------------------

// sum_j p[stride j] v[vs j], j < len: eight loads in flight, four partial
// sums (a per-lane loop is otherwise one load latency per term).
template <typename R>
__device__ inline double dot_ld(const R* p, int64_t stride, const double* v, int vs, int len) {
  double a0 = 0, a1 = 0, a2 = 0, a3 = 0;
  int j = 0;
  for (; j + 8 <= len; j += 8) {
    R q[8];
#pragma unroll
    for (int u = 0; u < 8; u++) q[u] = p[stride * (j + u)];
    a0 = fma((double)q[0], v[vs * j], a0);
    a1 = fma((double)q[1], v[vs * (j + 1)], a1);
    a2 = fma((double)q[2], v[vs * (j + 2)], a2);
    a3 = fma((double)q[3], v[vs * (j + 3)], a3);
    a0 = fma((double)q[4], v[vs * (j + 4)], a0);
    a1 = fma((double)q[5], v[vs * (j + 5)], a1);
    a2 = fma((double)q[6], v[vs * (j + 6)], a2);
    a3 = fma((double)q[7], v[vs * (j + 7)], a3);
  }
  for (; j < len; j++) a0 = fma((double)p[stride * j], v[vs * j], a0);
  return (a0 + a1) + (a2 + a3);
}

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// LDS of one box in doubles: its entries (n x C), then the staged factors.
// C = 1: the entries of the largest box, or a box of about 32 DOFs with its
// factors; C = 16: 128 DOFs, or about 32 with their factors.
template <int C>
struct SweepBuf {
  static constexpr int kLen = C == 1 ? 1024 : 2048;
};

// The box's entries of columns c0 .. c0 + C - 1 (zeros past the last) into
// x[position * C + column]; positions: skeleton, then redundant.
template <int C>
__device__ inline void gather_box(const SolveVec& v, const int* sk, const int* rd, int k, int n,
                                  int c0, double* x) {
  const int lane = threadIdx.x & 63, rg = lane / C, col = lane % C;
  const bool live = c0 + col < v.nrhs;
  for (int p = rg; p < n; p += 64 / C) {
    const int64_t dof = p < k ? sk[p] : rd[p - k];
    x[p * C + col] = live ? v.x[v.si * dof + v.sc * (c0 + col)] : 0.0;
  }
}

template <typename R>
__device__ inline void stage_factor(R* dst, const R* src, int len) {
  for (int i = threadIdx.x & 63; i < len; i += 64) dst[i] = src[i];
}

// Upward step of one box: x_r -= T^T x_s; x_s -= L x_r (U^T x_r when
// use_Ut); x_r = X_rr^{-1} x_r when diag (to dx where it is given).
template <typename R, int C>
__device__ void box_up(const SolveVec& v, const R* F, int k, int r, const int* sk, const int* rd,
                       int c0, bool use_Ut, bool diag, double* dx, double* buf, int len) {
  constexpr int RG = 64 / C;
  const int lane = threadIdx.x & 63, rg = lane / C, col = lane % C;
  const int n = k + r, kr = k * r;
  const bool live = c0 + col < v.nrhs;
  const FacLayout fl = FacLayout::make(k, r);
  double* xs = buf + col;
  double* xr = buf + k * C + col;
  R* f = reinterpret_cast<R*>(buf + n * C);
  auto run = [&](const R* T, const R* L, const R* X) {
    for (int i = rg; i < r; i += RG) xr[i * C] -= dot_ld(T + (int64_t)k * i, 1, xs, C, k);
    wave_sync();
    for (int a = rg; a < k; a += RG)
      xs[a * C] -= use_Ut ? dot_ld(L + (int64_t)r * a, 1, xr, C, r) : dot_ld(L + a, k, xr, C, r);
    for (int i = rg; i < r; i += RG) {
      const double y = diag ? dot_ld(X + i, r, xr, C, r) : xr[i * C];
      if (!live) continue;
      const int64_t at = v.si * rd[i] + v.sc * (c0 + col);
      if (dx) dx[at] = y;
      v.x[at] = dx ? xr[i * C] : y;
    }
    for (int a = rg; a < k; a += RG)
      if (live) v.x[v.si * sk[a] + v.sc * (c0 + col)] = xs[a * C];
  };
  const int nf = 2 * kr + (diag ? r * r : 0);
  if (n * C + (nf * (int)sizeof(R) + 7) / 8 <= len) {
    stage_factor(f, F + fl.T, kr);
    stage_factor(f + kr, F + (use_Ut ? fl.U : fl.L), kr);
    if (diag) stage_factor(f + 2 * kr, F + fl.X, r * r);
    gather_box<C>(v, sk, rd, k, n, c0, buf);
    wave_sync();
    run(f, f + kr, f + 2 * kr);
  } else {
    gather_box<C>(v, sk, rd, k, n, c0, buf);
    wave_sync();
    run(F + fl.T, F + (use_Ut ? fl.U : fl.L), F + fl.X);
  }
  wave_sync();  // the next columns reuse the buffer
}

// Downward step of one box: x_r -= U x_s; x_s -= T x_r.
template <typename R, int C>
__device__ void box_down(const SolveVec& v, const R* F, int k, int r, const int* sk,
                         const int* rd, int c0, double* buf, int len) {
  constexpr int RG = 64 / C;
  const int lane = threadIdx.x & 63, rg = lane / C, col = lane % C;
  const int n = k + r, kr = k * r;
  const bool live = c0 + col < v.nrhs;
  const FacLayout fl = FacLayout::make(k, r);
  double* xs = buf + col;
  double* xr = buf + k * C + col;
  R* f = reinterpret_cast<R*>(buf + n * C);
  auto run = [&](const R* T, const R* U) {
    for (int i = rg; i < r; i += RG) {
      const double y = xr[i * C] - dot_ld(U + i, r, xs, C, k);
      xr[i * C] = y;
      if (live) v.x[v.si * rd[i] + v.sc * (c0 + col)] = y;
    }
    wave_sync();
    for (int a = rg; a < k; a += RG) {
      const double y = xs[a * C] - dot_ld(T + a, k, xr, C, r);
      if (live) v.x[v.si * sk[a] + v.sc * (c0 + col)] = y;
    }
  };
  if (n * C + (2 * kr * (int)sizeof(R) + 7) / 8 <= len) {
    stage_factor(f, F + fl.T, kr);
    stage_factor(f + kr, F + fl.U, kr);
    gather_box<C>(v, sk, rd, k, n, c0, buf);
    wave_sync();
    run(f, f + kr);
  } else {
    gather_box<C>(v, sk, rd, k, n, c0, buf);
    wave_sync();
    run(F + fl.T, F + fl.U);
  }
  wave_sync();
}

template <typename R, int C>
__global__ __launch_bounds__(64) void k_sweep_up(DevState s, int start, SolveVec v, int use_Ut,
                                                 int diag, double* dx) {
  __shared__ double buf[SweepBuf<C>::kLen];
  static_assert(SweepBuf<C>::kLen >= kMaxBoxDofs, "one column of the largest box");
  const int b = start + blockIdx.x;
  const int k = s.rank[b];
  if (k == 0) return;
  const int r = s.act_cnt[b] - k;
  const R* F = reinterpret_cast<const R*>(s.fac_pool) + s.fac_off[b];
  const int* sk = s.out_list + (int64_t)b * s.ncap;
  const int* rd = s.red_list + (int64_t)b * s.ncap;
  if ((k + r) * C <= SweepBuf<C>::kLen) {
    for (int c = 0; c < v.nrhs; c += C)
      box_up<R, C>(v, F, k, r, sk, rd, c, use_Ut, diag, dx, buf, SweepBuf<C>::kLen);
  } else if (C > 1) {  // a box too large for C columns: one at a time
    for (int c = 0; c < v.nrhs; c++) {
      SolveVec one = v;
      one.x = v.x + v.sc * c;
      one.nrhs = 1;
      box_up<R, 1>(one, F, k, r, sk, rd, 0, use_Ut, diag, dx ? dx + v.sc * c : nullptr, buf,
                   SweepBuf<C>::kLen);
    }
  }
}

template <typename R, int C>
__global__ __launch_bounds__(64) void k_sweep_down(DevState s, int start, SolveVec v) {
  __shared__ double buf[SweepBuf<C>::kLen];
  const int b = start + blockIdx.x;
  const int k = s.rank[b];
  if (k == 0) return;
  const int r = s.act_cnt[b] - k;
  const R* F = reinterpret_cast<const R*>(s.fac_pool) + s.fac_off[b];
  const int* sk = s.out_list + (int64_t)b * s.ncap;
  const int* rd = s.red_list + (int64_t)b * s.ncap;
  if ((k + r) * C <= SweepBuf<C>::kLen) {
    for (int c = 0; c < v.nrhs; c += C)
      box_down<R, C>(v, F, k, r, sk, rd, c, buf, SweepBuf<C>::kLen);
  } else if (C > 1) {
    for (int c = 0; c < v.nrhs; c++) {
      SolveVec one = v;
      one.x = v.x + v.sc * c;
      one.nrhs = 1;
      box_down<R, 1>(one, F, k, r, sk, rd, 0, buf, SweepBuf<C>::kLen);
    }
  }
}

// x_root <- (root inverse) x_root, one workgroup per root.  A row's sum is
// four quarter sums added in order: with one column the quarters go to four
// threads, with several a thread forms them one after another for its
// column (16 at once while the entries fit LDS).
constexpr int kRootSolveBuf = 8192;

template <typename R>
__global__ __launch_bounds__(1024) void k_root_solve(DevState s, SolveVec v) {
  __shared__ double xa[kRootSolveBuf];
  __shared__ double red[4][256];
  const int tid = threadIdx.x;
  const int n = s.act_cnt[blockIdx.x];
  const int* act = s.act_list + (int64_t)blockIdx.x * s.ncap;
  const R* Ai = reinterpret_cast<const R*>(s.root_mat) +
                2 * (int64_t)s.ncap * s.ncap * blockIdx.x + (int64_t)n * n;
  const int q4 = (n + 3) / 4;
  auto quarter = [&](int i, int q, const double* x, int vs) {
    const int lo = min(q * q4, n), hi = min(lo + q4, n);
    return dot_ld(Ai + i + (int64_t)n * lo, n, x + (int64_t)vs * lo, vs, hi - lo);
  };
  const int C = v.nrhs > 1 && n * 16 <= kRootSolveBuf ? 16 : 1;
  for (int c0 = 0; c0 < v.nrhs; c0 += C) {
    for (int idx = tid; idx < n * C; idx += 1024) {
      const int col = c0 + idx % C;
      xa[idx] = col < v.nrhs ? v.x[v.si * act[idx / C] + v.sc * col] : 0.0;
    }
    __syncthreads();
    if (C == 1) {
      for (int i0 = 0; i0 < n; i0 += 256) {
        const int i = i0 + (tid & 255), q = tid >> 8;
        red[q][tid & 255] = i < n ? quarter(i, q, xa, 1) : 0.0;
        __syncthreads();
        if (q == 0 && i < n)
          v.x[v.si * act[i] + v.sc * c0] =
              (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
        __syncthreads();
      }
    } else {
      const int col = tid & 15;
      for (int i = tid >> 4; i < n; i += 64) {
        const double q0 = quarter(i, 0, xa + col, 16), q1 = quarter(i, 1, xa + col, 16);
        const double q2 = quarter(i, 2, xa + col, 16), q3 = quarter(i, 3, xa + col, 16);
        if (c0 + col < v.nrhs) v.x[v.si * act[i] + v.sc * (c0 + col)] = (q0 + q1) + (q2 + q3);
      }
      __syncthreads();
    }
  }
}

// dst (row-major n x h) <- src (column-major), or back, through LDS: both
// sides read and write whole lines.
__global__ __launch_bounds__(256) void k_transpose(double* dst, const double* src, int64_t n,
                                                   int h, int to_rows) {
  __shared__ double t[16][65];
  const int64_t r0 = (int64_t)blockIdx.x * 64;
  const int c0 = blockIdx.y * 16;
  for (int e = threadIdx.x; e < 1024; e += 256) {
    const int r = to_rows ? e % 64 : e / 16, c = to_rows ? e / 64 : e % 16;
    if (r0 + r < n && c0 + c < h)
      t[c][r] = src[to_rows ? r0 + r + n * (c0 + c) : (r0 + r) * h + c0 + c];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 1024; e += 256) {
    const int r = to_rows ? e / 16 : e % 64, c = to_rows ? e % 16 : e / 64;
    if (r0 + r < n && c0 + c < h)
      dst[to_rows ? (r0 + r) * h + c0 + c : r0 + r + n * (c0 + c)] = t[c][r];
  }
}

// ---------------------------------------------------------------------------
// Compressed forward apply b = A x (SkelFactorization::sparse_matvec,
// skel_factorization.cpp:429-504): the solve's steps undone in reverse
// order.  Per compressed box, levels leaves first:
//   b_s += T b_r;  b_r += U b_s;  b_r = X_rr b_r
// (X_rr may follow each box at once: no later box touches its redundant
// entries); then every root b = A_root b; then, root side first,
//   b_s += L b_r;  b_r += T^T b_s.
// One wave per box.
// ---------------------------------------------------------------------------

template <typename R>
__global__ __launch_bounds__(64) void k_fwd_up(DevState s, int start, double* x) {
  __shared__ double xs[kMaxBoxDofs];
  __shared__ double xr[kMaxBoxDofs];
  const int b = start + blockIdx.x;
  const int k = s.rank[b];
  if (k == 0) return;
  const int lane = threadIdx.x;
  const int r = s.act_cnt[b] - k;
  const FacLayout fl = FacLayout::make(k, r);
  const R* F = reinterpret_cast<const R*>(s.fac_pool) + s.fac_off[b];
  const R* Xf = reinterpret_cast<const R*>(s.fwd_pool) + s.fac_off[b];
  const int* sk = s.out_list + (int64_t)b * s.ncap;
  const int* rd = s.red_list + (int64_t)b * s.ncap;
  for (int a = lane; a < k; a += 64) xs[a] = x[sk[a]];
  for (int i = lane; i < r; i += 64) xr[i] = x[rd[i]];
  wave_sync();
  for (int a = lane; a < k; a += 64) xs[a] += dot_ld(F + fl.T + a, k, xr, 1, r);
  wave_sync();
  for (int i = lane; i < r; i += 64) xr[i] += dot_ld(F + fl.U + i, r, xs, 1, k);
  wave_sync();
  double y[kMaxBoxDofs / 64];
#pragma unroll
  for (int q = 0; q < kMaxBoxDofs / 64; q++) {
    const int i = lane + 64 * q;
    y[q] = i < r ? dot_ld(Xf + i, r, xr, 1, r) : 0.0;
  }
  for (int a = lane; a < k; a += 64) x[sk[a]] = xs[a];
#pragma unroll
  for (int q = 0; q < kMaxBoxDofs / 64; q++) {
    const int i = lane + 64 * q;
    if (i < r) x[rd[i]] = y[q];
  }
}

template <typename R>
__global__ __launch_bounds__(256) void k_fwd_root(DevState s, double* x) {
  __shared__ double xa[kMaxBoxDofs];
  const int tid = threadIdx.x;
  const int n = s.act_cnt[blockIdx.x];
  const int* act = s.act_list + (int64_t)blockIdx.x * s.ncap;
  const R* A = reinterpret_cast<const R*>(s.root_fwd) + (int64_t)s.ncap * s.ncap * blockIdx.x;
  for (int i = tid; i < n; i += 256) xa[i] = x[act[i]];
  __syncthreads();
  double y[kMaxBoxDofs / 256];
#pragma unroll
  for (int q = 0; q < kMaxBoxDofs / 256; q++) {
    const int i = tid + 256 * q;
    y[q] = i < n ? dot_ld(A + i, n, xa, 1, n) : 0.0;
  }
#pragma unroll
  for (int q = 0; q < kMaxBoxDofs / 256; q++) {
    const int i = tid + 256 * q;
    if (i < n) x[act[i]] = y[q];
  }
}

template <typename R>
__global__ __launch_bounds__(64) void k_fwd_down(DevState s, int start, double* x) {
  __shared__ double xs[kMaxBoxDofs];
  __shared__ double xr[kMaxBoxDofs];
  const int b = start + blockIdx.x;
  const int k = s.rank[b];
  if (k == 0) return;
  const int lane = threadIdx.x;
  const int r = s.act_cnt[b] - k;
  const FacLayout fl = FacLayout::make(k, r);
  const R* F = reinterpret_cast<const R*>(s.fac_pool) + s.fac_off[b];
  const int* sk = s.out_list + (int64_t)b * s.ncap;
  const int* rd = s.red_list + (int64_t)b * s.ncap;
  for (int a = lane; a < k; a += 64) xs[a] = x[sk[a]];
  for (int i = lane; i < r; i += 64) xr[i] = x[rd[i]];
  wave_sync();
  for (int a = lane; a < k; a += 64) xs[a] += dot_ld(F + fl.L + a, k, xr, 1, r);
  wave_sync();
  for (int i = lane; i < r; i += 64) xr[i] += dot_ld(F + fl.T + (int64_t)k * i, 1, xs, 1, k);
  wave_sync();
  for (int a = lane; a < k; a += 64) x[sk[a]] = xs[a];
  for (int i = lane; i < r; i += 64) x[rd[i]] = xr[i];
}

}  // namespace

// One column, or 16 at a time: a box's factors are read once per 16
// columns, and two or three columns in the 16-column form still cost less
// than a pass over the factors each.
template <typename R>
void launch_sweep_up(const DevState& s, int start, int count, SolveVec v, bool use_Ut, bool diag,
                     hipStream_t st, double* dx) {
  if (count <= 0) return;
  if (v.nrhs == 1)
    k_sweep_up<R, 1><<<count, 64, 0, st>>>(s, start, v, use_Ut ? 1 : 0, diag ? 1 : 0, dx);
  else
    k_sweep_up<R, 16><<<count, 64, 0, st>>>(s, start, v, use_Ut ? 1 : 0, diag ? 1 : 0, dx);
}

template <typename R>
void launch_sweep_down(const DevState& s, int start, int count, SolveVec v, hipStream_t st) {
  if (count <= 0) return;
  if (v.nrhs == 1) k_sweep_down<R, 1><<<count, 64, 0, st>>>(s, start, v);
  else k_sweep_down<R, 16><<<count, 64, 0, st>>>(s, start, v);
}

template <typename R>
void launch_root_solve(const DevState& s, int n_roots, SolveVec v, hipStream_t st) {
  k_root_solve<R><<<n_roots, 1024, 0, st>>>(s, v);
}

void launch_transpose(double* dst, const double* src, int64_t n, int h, bool to_rows,
                      hipStream_t st) {
  const dim3 grid((unsigned)((n + 63) / 64), (h + 15) / 16);
  k_transpose<<<grid, 256, 0, st>>>(dst, src, n, h, to_rows ? 1 : 0);
}

template <typename R>
void launch_fwd_up(const DevState& s, int start, int count, double* x, hipStream_t st) {
  if (count > 0) k_fwd_up<R><<<count, 64, 0, st>>>(s, start, x);
}
template <typename R>
void launch_fwd_root(const DevState& s, int n_roots, double* x, hipStream_t st) {
  k_fwd_root<R><<<n_roots, 256, 0, st>>>(s, x);
}
template <typename R>
void launch_fwd_down(const DevState& s, int start, int count, double* x, hipStream_t st) {
  if (count > 0) k_fwd_down<R><<<count, 64, 0, st>>>(s, start, x);
}

#define IEGPU_INSTANTIATE_SOLVE(R)                                                     \
  template void launch_sweep_up<R>(const DevState&, int, int, SolveVec, bool, bool,    \
                                   hipStream_t, double*);                              \
  template void launch_sweep_down<R>(const DevState&, int, int, SolveVec, hipStream_t); \
  template void launch_root_solve<R>(const DevState&, int, SolveVec, hipStream_t);     \
  template void launch_fwd_up<R>(const DevState&, int, int, double*, hipStream_t);     \
  template void launch_fwd_root<R>(const DevState&, int, double*, hipStream_t);        \
  template void launch_fwd_down<R>(const DevState&, int, int, double*, hipStream_t);

IEGPU_INSTANTIATE_SOLVE(double)
IEGPU_INSTANTIATE_SOLVE(float)

}  // namespace iegpu
