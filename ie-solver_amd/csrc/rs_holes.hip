// Bordered system for multiply connected domains
// (skel_factorization.cpp:188-305 factor side, :596-777 solve side).
//
// With the upward-swept border matrices mU (ndof x h) and mPsi^T
// (ndof x h) and D the block diagonal of the boxes' X_rr:
//   S = [ A_ss            mU(skel,:)                          ]
//       [ mPsi^T(skel,:)^T  -I - mPsi^T(red,:)^T D^{-1} mU(red,:) ]
// "skel" is the root's active list and "red" every other DOF.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "rs_device.hpp"
#include "rs_holes.hpp"
#include "rs_inv.hpp"

namespace iegpu {

namespace {

__global__ void k_fill_int(int* p, int64_t n, int v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_mark_skel(const DevState s, int* mask) {
  const int n = s.act_cnt[0];
  for (int i = threadIdx.x; i < n; i += blockDim.x) mask[s.act_list[i]] = 1;
}

__global__ void k_copy(double* dst, const double* src, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// The border blocks are row-major (ndof x h): the h entries of a row are
// one or two cache lines, read by neighbouring lanes.

// partial[blk][a + h*c] = sum over redundant rows i of chunk blk of
// P[i,a] * C[i,c].  Rows are staged gram_rows(h) at a time in LDS, a thread
// owning four of the h^2 sums per pass over the chunk (one pass up to
// h = 32).  LDS reads bound it: 139 us at 262,144 DOFs and h = 24 (1,982 us
// with the blocks column-major, each row's 2 h entries on 2 h lines).
constexpr int kGramLds = 4096;  // doubles for each block's rows
__device__ inline int gram_rows(int h) { return min(64, kGramLds / h); }

__global__ __launch_bounds__(256) void k_gram_partial(const double* P, const double* C,
                                                      const int* mask, int64_t ndof, int h,
                                                      int64_t chunk, double* partial) {
  __shared__ double sp[kGramLds], sc[kGramLds];
  const int64_t lo = blockIdx.x * chunk;
  const int64_t hi = lo + chunk < ndof ? lo + chunk : ndof;
  const int tr = gram_rows(h);
  for (int e0 = 0; e0 < h * h; e0 += 1024) {
    double acc[4] = {0, 0, 0, 0};
    int ea[4], ec[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int e = min(e0 + (int)threadIdx.x + 256 * u, h * h - 1);
      ea[u] = e % h;
      ec[u] = e / h;
    }
    for (int64_t r0 = lo; r0 < hi; r0 += tr) {
      const int rows = (int)min((int64_t)tr, hi - r0);
      __syncthreads();
      for (int i = threadIdx.x; i < rows * h; i += 256) {
        const bool skel = mask[r0 + i / h] != 0;  // C is not defined there
        sp[i] = skel ? 0.0 : P[r0 * h + i];
        sc[i] = skel ? 0.0 : C[r0 * h + i];
      }
      __syncthreads();
      for (int i = 0; i < rows; i++)
#pragma unroll
        for (int u = 0; u < 4; u++) acc[u] = fma(sp[i * h + ea[u]], sc[i * h + ec[u]], acc[u]);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int e = e0 + threadIdx.x + 256 * u;
      if (e < h * h) partial[blockIdx.x * (int64_t)h * h + e] = acc[u];
    }
  }
}

// partial[blk][a] = sum over the rows i of chunk blk (mask given: the
// redundant ones) of P[i,a] * x[i]: 256 / h rows at a time, then the row
// lanes added in order.  Reads 50 MB at 262,144 DOFs and h = 24: 22 us (656
// us with 64 one-wave workgroups on column-major blocks).
__global__ __launch_bounds__(256) void k_gemv_partial(const double* P, const double* x,
                                                      const int* mask, int64_t ndof, int h,
                                                      int64_t chunk, double* partial) {
  __shared__ double red[256];
  const int rl = 256 / h, a = threadIdx.x % h, rr = threadIdx.x / h;
  const int64_t lo = blockIdx.x * chunk;
  const int64_t hi = lo + chunk < ndof ? lo + chunk : ndof;
  double acc = 0;
  if (rr < rl)
    for (int64_t i = lo + rr; i < hi; i += rl)
      acc += (mask && mask[i]) ? 0.0 : P[i * h + a] * x[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  if (threadIdx.x < h) {
    for (int q = 1; q < rl; q++) acc += red[a + h * q];
    partial[blockIdx.x * (int64_t)h + a] = acc;
  }
}

// Sum over blocks of partial[blk][j], in every thread of a workgroup of 256
// (fixed order: deterministic).
__device__ inline double sum_partials(const double* partial, int nblk, int64_t len, int j,
                                      double* red) {
  double acc = 0;
  for (int b = threadIdx.x; b < nblk; b += 256) acc += partial[b * len + j];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  return red[0];
}

// out[j] = sum_blk partial[blk][j] - sub[j] (sub may be null), j = workgroup.
__global__ __launch_bounds__(256) void k_reduce_partials(const double* partial, int nblk, int len,
                                                         double* out, const double* sub) {
  __shared__ double red[256];
  const int j = blockIdx.x;
  const double v = sum_partials(partial, nblk, len, j, red);
  if (threadIdx.x == 0) out[j] = v - (sub ? sub[j] : 0.0);
}

// S (ns + h square, column-major), and its inverse's panel flags cleared.
template <typename R>
__global__ __launch_bounds__(256) void k_border_assemble(DevState s, const double* mU,
                                                         const double* mPsiT, const double* gram,
                                                         int h, double* Smat, int* flags) {
  const int ns = s.act_cnt[0];
  const int N = ns + h;
  const int* act = s.act_list;
  const R* A = reinterpret_cast<const R*>(s.root_mat);
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < kInvFlags; i += 256) flags[i] = 0;
  for (int64_t idx = blockIdx.x * 256 + threadIdx.x; idx < (int64_t)N * N;
       idx += gridDim.x * 256) {
    const int i = (int)(idx % N), j = (int)(idx / N);
    double v;
    if (i < ns && j < ns) v = (double)A[i + (int64_t)ns * j];
    else if (i >= ns && j < ns) v = mPsiT[(int64_t)act[j] * h + (i - ns)];
    else if (i < ns) v = mU[(int64_t)act[i] * h + (j - ns)];
    else v = (i == j ? -1.0 : 0.0) - gram[(i - ns) + h * (j - ns)];
    Smat[idx] = v;
  }
}

// rhs = [x(skel); g - the sum of the partial products mPsi^T(red,:) x]  (g:
// the right-hand side of the border rows; null: zero, as in the reference's
// [f; 0]).  Workgroups 0 .. h-1 form one border entry each, the others copy.
__global__ __launch_bounds__(256) void k_border_rhs(DevState s, const double* x,
                                                    const double* partial, int nblk, int h,
                                                    const double* g, double* rhs) {
  __shared__ double red[256];
  const int ns = s.act_cnt[0], a = blockIdx.x;
  if (a < h) {
    const double v = sum_partials(partial, nblk, h, a, red);
    if (threadIdx.x == 0) rhs[ns + a] = (g ? g[a] : 0.0) - v;
    return;
  }
  const int i = (a - h) * 256 + threadIdx.x;
  if (i < ns) rhs[i] = x[s.act_list[i]];
}

// y = S^{-1} rhs; x(skel) = y_head, alpha = y_tail: 16 rows per workgroup,
// a row's sum in 16 strided parts added in order (a 354-DOF S: 982 us by
// triangular solves in one wave, 12 us).
__global__ __launch_bounds__(256) void k_border_solve(DevState s, const double* Sinv, int h,
                                                      const double* rhs, double* x,
                                                      double* alpha) {
  __shared__ double red[16][17];
  const int ns = s.act_cnt[0], N = ns + h;
  const int row = threadIdx.x & 15, part = threadIdx.x >> 4;
  const int i = blockIdx.x * 16 + row;
  double acc = 0;
  if (i < N)
    for (int j = part; j < N; j += 16) acc = fma(Sinv[i + (int64_t)N * j], rhs[j], acc);
  red[part][row] = acc;
  __syncthreads();
  if (part == 0 && i < N) {
    double y = 0;
#pragma unroll
    for (int q = 0; q < 16; q++) y += red[q][row];
    if (i < ns) x[s.act_list[i]] = y;
    else alpha[i - ns] = y;
  }
}

// x(red) -= C(red,:) alpha.
__global__ void k_red_update(double* x, const double* C, const int* mask, const double* alpha,
                             int64_t ndof, int h) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < ndof;
       i += (int64_t)gridDim.x * blockDim.x) {
    if (mask[i]) continue;
    double acc = x[i];
    for (int c = 0; c < h; c++) acc -= C[i * h + c] * alpha[c];
    x[i] = acc;
  }
}

// y[i] += sum_c U[i,c] a[c].
__global__ void k_border_apply_u(double* y, const double* U, const double* a, int64_t ndof,
                                 int h) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < ndof;
       i += (int64_t)gridDim.x * blockDim.x) {
    double acc = y[i];
    for (int c = 0; c < h; c++) acc += U[i * h + c] * a[c];
    y[i] = acc;
  }
}

// Rows of a partial sum: 1,024 workgroups of a product at 262,144 DOFs (256
// rows; 64 of 4,096 rows left the chip idle), the Gram matrix's h^2 sums in
// fewer.
constexpr int64_t kChunk = 256;
inline int64_t gram_chunk(int h) { return h <= 48 ? 1024 : 4096; }
inline int blocks_of(int64_t n, int64_t chunk) { return (int)((n + chunk - 1) / chunk); }

}  // namespace

void launch_mark_skel(const DevState& s, int* mask, int64_t ndof,
                      hipStream_t st) {
  k_fill_int<<<256, 256, 0, st>>>(mask, ndof, 0);
  k_mark_skel<<<1, 1024, 0, st>>>(s, mask);
}

void launch_copy(double* dst, const double* src, int64_t n, hipStream_t st) {
  k_copy<<<512, 256, 0, st>>>(dst, src, n);
}

// dst row r = src row map[r] (rows of row_words 32-bit words); rows with
// map[r] < 0 are zeroed.
__global__ void k_gather_rows(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src,
                              const int* __restrict__ map, int n_rows, int row_words) {
  const int64_t total = (int64_t)n_rows * row_words;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(i / row_words);
    const int o = map[r];
    dst[i] = o >= 0 ? src[(int64_t)o * row_words + (i - (int64_t)r * row_words)] : 0u;
  }
}

void launch_gather_rows(void* dst, const void* src, const int* map, int n_rows, int row_words,
                        hipStream_t st) {
  if (n_rows <= 0 || row_words <= 0) return;
  const int64_t total = (int64_t)n_rows * row_words;
  const int blocks = (int)std::min<int64_t>((total + 255) / 256, 8192);
  k_gather_rows<<<blocks, 256, 0, st>>>(static_cast<uint32_t*>(dst),
                                        static_cast<const uint32_t*>(src), map, n_rows,
                                        row_words);
}

int64_t border_partials(int64_t ndof, int h) {
  return std::max((int64_t)blocks_of(ndof, kChunk) * h,
                  (int64_t)blocks_of(ndof, gram_chunk(h)) * h * h);
}

void launch_border_gram(const double* P, const double* C, const int* mask,
                        int64_t ndof, int h, double* partial, double* out,
                        hipStream_t st) {
  const int nb = blocks_of(ndof, gram_chunk(h));
  k_gram_partial<<<nb, 256, 0, st>>>(P, C, mask, ndof, h, gram_chunk(h), partial);
  k_reduce_partials<<<h * h, 256, 0, st>>>(partial, nb, h * h, out, nullptr);
}

template <typename R>
void launch_border_factor(const DevState& s, const double* mU, const double* mPsiT,
                          const double* gram, int h, double* Smat, double* Sinv, int* Spiv,
                          hipStream_t st) {
  const int piv_stride = s.ncap + h + kInvFlags;
  k_border_assemble<R><<<128, 256, 0, st>>>(s, mU, mPsiT, gram, h, Smat,
                                            Spiv + piv_stride - kInvFlags);
  InvBlocks<double> blk;
  blk.a = Smat;
  blk.out = Sinv;
  blk.stride = 0;
  blk.piv = Spiv;
  blk.piv_stride = piv_stride;
  blk.extra = h;
  launch_block_inverse<double>(s, blk, 1, 0, s.ncap + h, st);
}

void launch_border_solve(const DevState& s, const double* mPsiT, const double* Sinv,
                         const int* mask, int64_t ndof, int h, double* x, const double* g,
                         double* alpha, double* partial, double* rhs, hipStream_t st) {
  const int nb = blocks_of(ndof, kChunk), nmax = s.ncap + h;
  k_gemv_partial<<<nb, 256, 0, st>>>(mPsiT, x, mask, ndof, h, kChunk, partial);
  k_border_rhs<<<h + (s.ncap + 255) / 256, 256, 0, st>>>(s, x, partial, nb, h, g, rhs);
  k_border_solve<<<(nmax + 15) / 16, 256, 0, st>>>(s, Sinv, h, rhs, x, alpha);
}

void launch_red_update(double* x, const double* C, const int* mask,
                       const double* alpha, int64_t ndof, int h,
                       hipStream_t st) {
  k_red_update<<<1024, 256, 0, st>>>(x, C, mask, alpha, ndof, h);
}

void launch_border_apply(const double* U, const double* PsiT, const double* x,
                         const double* alpha, int64_t ndof, int h, double* partial, double* y,
                         double* z, hipStream_t st) {
  const int nb = blocks_of(ndof, kChunk);
  k_border_apply_u<<<1024, 256, 0, st>>>(y, U, alpha, ndof, h);
  k_gemv_partial<<<nb, 256, 0, st>>>(PsiT, x, nullptr, ndof, h, kChunk, partial);
  k_reduce_partials<<<h, 256, 0, st>>>(partial, nb, h, z, alpha);
}

template void launch_border_factor<double>(const DevState&, const double*, const double*,
                                           const double*, int, double*, double*, int*,
                                           hipStream_t);
template void launch_border_factor<float>(const DevState&, const double*, const double*,
                                          const double*, int, double*, double*, int*,
                                          hipStream_t);

}  // namespace iegpu
