// Inverse of a dense block over many workgroups: the root blocks above
// kRootRegMax DOFs (skel_factorization.cpp:172-186) and the bordered system
// of multiply connected domains (:188-305), which the reference LU-factors.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rs_device.hpp"
#include "rs_inv.hpp"

namespace iegpu {

namespace {

// ---------------------------------------------------------------------------
// Blocked Gauss-Jordan with partial pivoting, rows not moved.  One
// workgroup owns the kInvB = 16 columns of panel j, thread t the rows
// t, t + 512, ...: a panel's 16 elimination steps run on registers
// (pivot row: largest |entry| among the rows not yet pivoted, one barrier
// per step), and the other columns take them at once: with W the final slab
// of panel q and P its pivot rows' old values, the steps turn a column x
// into x + sum_k W_k x_{p_k}, a pivot row's own value being replaced rather
// than added to.
//
// k_inv_panel: workgroup j applies panels 0 .. j-1 to its columns as they
// are published, eliminates its own and publishes it (the slab over its own
// columns of the block, the pivot rows, then the panel's flag).  A
// workgroup draws its panel when it starts (a counter per block), so the
// panels it waits for belong to workgroups that run already: the wait ends
// whatever order the workgroups start in and whatever other launches (a
// second context's inverses) hold the rest of the chip.
// k_inv_finish: the columns of panel j take the panels j+1, ... (all
// published), four columns per workgroup, and the unpermuted inverse is
// written.
//
// Bound by the chain of panels (wait, one update, 16 pivot steps, publish):
// about 17 us per panel in FP64, mostly the steps' instructions.  A block of
// 212 DOFs takes 235 us and one of 393 504 us, k_inv_finish 21 and 42 (with
// the panels handed over through agent-scope fences, every wave in every
// step and the pivot rows stored step by step both kernels took 258 and 507
// us where they took 228 and 463 without).  One workgroup streaming the block from L2 took 986 us for 212 DOFs and 2,984 for 393, an LU in one
// workgroup 7,570 us for the 354-DOF bordered system of Stokes with 8 holes.
// ---------------------------------------------------------------------------

constexpr int kInvB = 16;       // columns of a panel
constexpr int kInvNT = 512;     // threads: rows per pass
constexpr int kInvCF = 4;       // columns of a k_inv_finish workgroup
constexpr int kInvNW = kInvNT / 64;
static_assert(kInvMax <= 3 * kInvNT, "rows per thread");
static_assert(kInvNW == 8, "the waves' candidates fill half a DPP row");

__device__ inline unsigned wave_max_u32(unsigned v) {
  v = max(v, (unsigned)dpp_i32<dpp::kQuadSwap1, 0xF>((int)v));
  v = max(v, (unsigned)dpp_i32<dpp::kQuadSwap2, 0xF>((int)v));
  v = max(v, (unsigned)dpp_i32<dpp::kRowHalfMirror, 0xF>((int)v));
  v = max(v, (unsigned)dpp_i32<dpp::kRowMirror, 0xF>((int)v));
  v = max(v, (unsigned)dpp_i32<dpp::kRowBcast15, 0xA>((int)v));
  v = max(v, (unsigned)dpp_i32<dpp::kRowBcast31, 0xC>((int)v));
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// A pivot candidate's magnitude in two words that order as it does, the
// first one up so that 0 is left for a row that is no candidate.  A
// non-finite entry counts as zero: every unpivoted row stays a candidate.
__device__ inline void pivot_words(double v, bool used, unsigned& hi, unsigned& lo) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned h = (unsigned)(b >> 32) & 0x7fffffffu;
  const bool fin = h < 0x7ff00000u;
  hi = used ? 0u : (fin ? h + 1 : 1u);
  lo = fin ? (unsigned)b : 0u;
}
__device__ inline void pivot_words(float v, bool used, unsigned& hi, unsigned& lo) {
  const unsigned h = __float_as_uint(v) & 0x7fffffffu;
  hi = used ? 0u : (h < 0x7f800000u ? h + 1 : 1u);
  lo = 0u;
}

// The first of the lanes in `lanes` with the largest (hi, lo); best: the
// largest hi.  Lanes that share it are rare, so the low words are mostly not
// looked at.
template <typename R>
__device__ inline int top_lane(unsigned hi, unsigned lo, unsigned best, uint64_t lanes) {
  uint64_t m = __ballot(hi == best) & lanes;
  if (sizeof(R) == 8 && (m & (m - 1)) != 0) {
    const unsigned bl = wave_max_u32(hi == best ? lo : 0u);
    m = __ballot(hi == best && lo == bl) & lanes;
  }
  return __ffsll((unsigned long long)m) - 1;
}

// Wait of a workgroup for panel flag *f: bounded (about two seconds), false
// if it never came.
__device__ inline bool wait_flag(const int* f) {
  for (int spin = 0; spin < (1 << 22); spin++) {
    if (__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return true;
    __builtin_amdgcn_s_sleep(1);
  }
  return false;
}

// What workgroups of one launch hand each other (slabs, pivot rows) goes
// through agent-scope accesses, which pass the XCDs' L2s: a publisher waits
// for its stores' acknowledgements before the flag, and neither side writes
// back or invalidates a whole L2 (fences took a third of a panel).
template <typename T>
__device__ inline void publish(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool SHARED, typename T>
__device__ inline T fetch(const T* p) {
  return SHARED ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *p;
}

// x (columns CB of the thread's RT rows) takes panel q: W from the block's
// columns, the pivot rows' old values through LDS.  pstep[row] is the step
// that pivots on a row (kInvMax: none yet) and is extended by the panel's.
// SHARED: the panel was published in this launch.  All threads of the
// workgroup.
template <typename R, int RT, int CB, bool SHARED>
__device__ inline void apply_panel(const R* A, const int* prow, int n, int q, R (&x)[RT][CB],
                                   short* pstep, R (*P)[CB]) {
  const int tid = threadIdx.x, q0 = q * kInvB, bw = min(kInvB, n - q0);
  R w[RT][kInvB];
#pragma unroll
  for (int u = 0; u < RT; u++) {
    const int i = tid + kInvNT * u;
#pragma unroll
    for (int k = 0; k < kInvB; k++) {  // all loads in flight at once
      const R v = fetch<SHARED>(A + min(i, n - 1) + (int64_t)n * (q0 + min(k, bw - 1)));
      w[u][k] = (i < n && k < bw) ? v : R(0);
    }
  }
  if (tid < bw) pstep[fetch<SHARED>(prow + q0 + tid)] = (short)(q0 + tid);
  if (bw < kInvB && tid < kInvB * CB) P[tid / CB][tid % CB] = R(0);  // steps past the last
  __syncthreads();
#pragma unroll
  for (int u = 0; u < RT; u++) {
    const int i = tid + kInvNT * u;
    const int st = i < n ? pstep[i] - q0 : -1;
    if (st >= 0 && st < bw) {
#pragma unroll
      for (int c = 0; c < CB; c++) {
        P[st][c] = x[u][c];
        x[u][c] = R(0);
      }
    }
  }
  __syncthreads();
  if (64 * wave_id() >= n) return;
#pragma unroll
  for (int k = 0; k < kInvB; k++)
#pragma unroll
    for (int c = 0; c < CB; c++) {
      const R p = P[k][c];
#pragma unroll
      for (int u = 0; u < RT; u++) x[u][c] = fma(w[u][k], p, x[u][c]);
    }
}

template <typename R, int RT>
__global__ __launch_bounds__(kInvNT) void k_inv_panel(DevState s, InvBlocks<R> blk, int nmin,
                                                      int nmax) {
  __shared__ R P[kInvB][kInvB];
  __shared__ R cand[2][kInvNW][kInvB];  // each wave's candidate row, by step parity
  __shared__ unsigned keyh[2][kInvNW], keyl[2][kInvNW];  // its magnitude
  __shared__ int crow[2][kInvNW];                        // its row
  __shared__ short pstep[kInvMax];
  __shared__ int ok, panel, sprow[kInvB];
  if (!pools_ok(s)) return;
  const int root = blockIdx.x;
  const int n = s.act_cnt[root] + blk.extra;
  if (n <= nmin || n > nmax || kInvB * (int)blockIdx.y >= n) return;
  R* A = blk.a + blk.stride * root;
  int* prow = blk.piv + (int64_t)blk.piv_stride * root;
  int* flags = prow + blk.piv_stride - kInvFlags;
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  if (tid == 0) panel = atomicAdd(flags + kInvFlags - 1, 1);
  __syncthreads();
  const int j = __builtin_amdgcn_readfirstlane(panel), j0 = j * kInvB;
  const int bw = min(kInvB, n - j0);
  R x[RT][kInvB];
#pragma unroll
  for (int u = 0; u < RT; u++) {
    const int i = tid + kInvNT * u;
#pragma unroll
    for (int k = 0; k < kInvB; k++) {
      const R v = A[min(i, n - 1) + (int64_t)n * (j0 + min(k, bw - 1))];
      x[u][k] = (i < n && k < bw) ? v : R(0);
    }
  }
  for (int i = tid; i < n; i += kInvNT) pstep[i] = (short)kInvMax;
  for (int q = 0; q < j; q++) {
    if (tid == 0) ok = wait_flag(flags + q) ? 1 : 0;
    __syncthreads();
    if (!ok) {
      if (tid == 0) atomicOr(s.err, kErrWait);
      return;
    }
    apply_panel<R, RT, kInvB, true>(A, prow, n, q, x, pstep, P);
    __syncthreads();
  }
  // the panel's own steps
  bool used[RT];
#pragma unroll
  for (int u = 0; u < RT; u++) {
    const int i = tid + kInvNT * u;
    used[u] = i >= n || pstep[i] != kInvMax;
  }
  int info = 0;
  // Waves past the block's rows only keep the barriers.
  const bool live = 64 * wv < n;
  if (!live && lane == 0) keyh[0][wv] = keyh[1][wv] = keyl[0][wv] = keyl[1][wv] = 0;
#pragma unroll
  for (int k = 0; k < kInvB; k++) {
    if (k < bw && !live) {
      __syncthreads();
    } else if (k < bw) {
      // The wave's candidate: the largest |entry| of the step's column among
      // its rows not yet pivoted.
      const int par = k & 1;
      unsigned hi, lo;
      int best_u = 0;
      pivot_words(x[0][k], used[0], hi, lo);
#pragma unroll
      for (int u = 1; u < RT; u++) {
        unsigned h, l;
        pivot_words(x[u][k], used[u], h, l);
        const bool up = h > hi || (h == hi && l > lo);
        hi = up ? h : hi;
        lo = up ? l : lo;
        best_u = up ? u : best_u;
      }
      const unsigned best = wave_max_u32(hi);
      if (best == 0) {
        if (lane == 0) keyh[par][wv] = keyl[par][wv] = 0;
      } else if (lane == top_lane<R>(hi, lo, best, ~0ull)) {
        keyh[par][wv] = hi;
        keyl[par][wv] = lo;
        crow[par][wv] = tid + kInvNT * best_u;
#pragma unroll
        for (int u = 0; u < RT; u++)
          if (u == best_u) {
#pragma unroll
            for (int c = 0; c < kInvB; c++) cand[par][wv][c] = x[u][c];
          }
      }
      __syncthreads();
      // the waves' candidates, eight lanes each
      const unsigned wh = keyh[par][lane & 7], wl = keyl[par][lane & 7];
      unsigned top = wh;
      top = max(top, (unsigned)dpp_i32<dpp::kQuadSwap1, 0xF>((int)top));
      top = max(top, (unsigned)dpp_i32<dpp::kQuadSwap2, 0xF>((int)top));
      top = max(top, (unsigned)dpp_i32<dpp::kRowHalfMirror, 0xF>((int)top));
      const int tw = top_lane<R>(wh, wl, top, 0xffull);
      const int p = crow[par][tw];
      R rv[kInvB];
#pragma unroll
      for (int c = 0; c < kInvB; c++) rv[c] = cand[par][tw][c];
      const R piv = rv[k];
      if (piv == R(0) && info == 0) info = j0 + k + 1;
      const R inv = R(1) / piv;
#pragma unroll
      for (int c = 0; c < kInvB; c++) rv[c] = c == k ? inv : rv[c] * inv;
#pragma unroll
      for (int u = 0; u < RT; u++) {
        const R m = x[u][k];
        const bool me = tid + kInvNT * u == p;
        x[u][k] = R(0);
#pragma unroll
        for (int c = 0; c < kInvB; c++) x[u][c] = me ? rv[c] : fma(-m, rv[c], x[u][c]);
        used[u] = used[u] || me;
      }
      if (tid == 0) sprow[k] = p;  // a global store here is waited for at the next step
    }
  }
#pragma unroll
  for (int u = 0; u < RT; u++) {
    const int i = tid + kInvNT * u;
    if (i >= n) continue;
    if (bw == kInvB) {  // no branch, and so no wait, between the stores
#pragma unroll
      for (int k = 0; k < kInvB; k++) publish(A + i + (int64_t)n * (j0 + k), x[u][k]);
    } else {
#pragma unroll
      for (int k = 0; k < kInvB; k++)
        if (k < bw) publish(A + i + (int64_t)n * (j0 + k), x[u][k]);
    }
  }
  if (info != 0 && tid == 0) atomicOr(s.err, kErrSingular);
  if (tid < bw) publish(prow + j0 + tid, sprow[tid]);
  __builtin_amdgcn_s_waitcnt(0);  // this wave's part of the slab has arrived
  __syncthreads();
  if (tid == 0) publish(flags + j, 1);
}

template <typename R, int RT>
__global__ __launch_bounds__(kInvNT) void k_inv_finish(DevState s, InvBlocks<R> blk, int nmin,
                                                       int nmax) {
  __shared__ R P[2][kInvB][kInvCF];
  __shared__ short pstep[kInvMax];
  if (!pools_ok(s) || (s.err[0] & kErrWait)) return;
  const int root = blockIdx.x, c0 = blockIdx.y * kInvCF;
  const int n = s.act_cnt[root] + blk.extra;
  if (n <= nmin || n > nmax || c0 >= n) return;
  const R* A = blk.a + blk.stride * root;
  R* B = blk.out ? blk.out + blk.stride * root : blk.a + blk.stride * root + (int64_t)n * n;
  const int* prow = blk.piv + (int64_t)blk.piv_stride * root;
  const int tid = threadIdx.x;
  R x[RT][kInvCF];
#pragma unroll
  for (int u = 0; u < RT; u++) {
    const int i = tid + kInvNT * u;
#pragma unroll
    for (int c = 0; c < kInvCF; c++)
      x[u][c] = (i < n && c0 + c < n) ? A[i + (int64_t)n * (c0 + c)] : R(0);
  }
  for (int st = tid; st < n; st += kInvNT) pstep[prow[st]] = (short)st;
  const int np = (n + kInvB - 1) / kInvB;
  for (int q = c0 / kInvB + 1; q < np; q++)
    apply_panel<R, RT, kInvCF, false>(A, prow, n, q, x, pstep, P[q & 1]);
  __syncthreads();
  // entry (row i, column c): inverse row = the step that pivoted on i,
  // column = the row step c pivoted on
#pragma unroll
  for (int u = 0; u < RT; u++) {
    const int i = tid + kInvNT * u;
    if (i >= n) continue;
    const int row = pstep[i];
#pragma unroll
    for (int c = 0; c < kInvCF; c++)
      if (c0 + c < n) B[row + (int64_t)n * prow[c0 + c]] = x[u][c];
  }
}

}  // namespace

template <typename R>
void launch_block_inverse(const DevState& s, const InvBlocks<R>& blk, int n_blocks, int nmin,
                          int nmax, hipStream_t st) {
  // one row per thread, or three
  const int m1 = nmax < kInvNT ? nmax : kInvNT;
  auto grid = [&](int n, int cols) { return dim3(n_blocks, (n + cols - 1) / cols); };
  if (nmin < kInvNT) {
    k_inv_panel<R, 1><<<grid(m1, kInvB), kInvNT, 0, st>>>(s, blk, nmin, m1);
    k_inv_finish<R, 1><<<grid(m1, kInvCF), kInvNT, 0, st>>>(s, blk, nmin, m1);
  }
  if (nmax > kInvNT) {
    const int lo = nmin > kInvNT ? nmin : kInvNT;
    k_inv_panel<R, 3><<<grid(nmax, kInvB), kInvNT, 0, st>>>(s, blk, lo, nmax);
    k_inv_finish<R, 3><<<grid(nmax, kInvCF), kInvNT, 0, st>>>(s, blk, lo, nmax);
  }
}

template void launch_block_inverse<double>(const DevState&, const InvBlocks<double>&, int, int,
                                           int, hipStream_t);
template void launch_block_inverse<float>(const DevState&, const InvBlocks<float>&, int, int,
                                          int, hipStream_t);

}  // namespace iegpu
