// Interior evaluation u = K_domain mu + U_forward alpha, matrix-free
// (ie_solver/initialization.cpp:11-135, linear_solve.cpp:140-154,188-266).
//
// Laplace: u(x) = sum_j -(w_j / 2 pi) ((x - y_j) . n_j) / |x - y_j|^2 mu_j.
// Stokes:  u_a(x) = sum_j (w_j / pi) ((x - y_j) . n_j) / |x - y_j|^4
//                   r_a (r_0 mu_2j + r_1 mu_2j+1)   (no n n^T term off the
//                   boundary, kernel.cpp:29-63 with tgt.is_boundary = false).
// Targets outside the domain give 0 (initialization.cpp:43-49).
//
// Grid: (blocks of kTargets targets) x (source chunks); k_eval_partial
// forms the sums of one chunk, k_eval_finish adds the chunks in a fixed
// order with the hole terms.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>

#include "rs_device.hpp"
#include "rs_eval.hpp"

namespace iegpu {

// Partial sums of the allocation-free evaluation (iegpu_evaluate_noalloc):
// one copy per GPU, held until the process ends.  Host code uses the
// address hipGetSymbolAddress returns for the current device, never this
// name (which is a host-side stand-in, not a device address).
static __device__ __align__(256) double scratch[kEvalScratchElems];

namespace {

// k_eval_partial: 8 waves share kTargets = 128 targets, two per lane; wave
// w takes sources 64 w .. 64 w + 63 of every staged tile of kTile, and the
// eight waves' sums are added in wave order.  FP64 issue bounds it: a
// Laplace pair costs eight FP64 instructions and a reciprocal of five (a
// division alone costs as much as both), and two targets per lane share each
// source's LDS reads, which one per lane would make the bound (two b128
// broadcasts per pair and wave).  10,000 targets x 65,536 Laplace sources:
// 954 us with one target per thread, divisions and 320 workgroups of four
// waves; 367 us (353 with one Newton step, which is not as accurate).
constexpr int kTargets = 128, kTile = 512;
// Points past this magnitude (and NaN) take the division: |r|^2 would
// overflow, and the Newton steps turn the reciprocal's 0 into NaN.
constexpr double kFar = 1e150;
__device__ inline bool is_far(double2 p) { return !(fabs(p.x) < kFar && fabs(p.y) < kFar); }

// 1 / d from v_rcp_f64 (2e8 eps off) and two Newton steps: within half an
// eps, as the division; one step is up to 9.6 eps off (a million values).
__device__ inline double recip_full(double d) {
  double y = __builtin_amdgcn_rcp(d);
  y = fma(y, fma(-d, y, 1.0), y);
  return fma(y, fma(-d, y, 1.0), y);
}

// One source's contribution at the target p, added to a: xy the point; ab
// -w mu n / (2 pi) (Laplace), (w mu / (4 pi), 0) (Neumann) or w n / pi
// (Stokes); m the Stokes density.  FAST: recip_full, else the division.
template <int PDE, bool FAST>
__device__ inline void eval_pair(double2 p, double2 xy, double2 ab, double2 m, double2& a) {
  const double r0 = p.x - xy.x, r1 = p.y - xy.y;
  const double d2 = fma(r0, r0, r1 * r1);
  if constexpr (PDE == kPdeLaplaceNeumann) {
    a.x = fma(ab.x, log(d2), a.x);  // single layer w (1/2 pi) log|r| (kernel.cpp:95-102)
  } else {
    const double inv = FAST ? recip_full(d2) : 1.0 / d2;
    const double rn = fma(r0, ab.x, r1 * ab.y);
    if constexpr (PDE == kPdeStokes) {
      const double pot = rn * inv * inv * fma(r0, m.x, r1 * m.y);
      a.x = fma(pot, r0, a.x);
      a.y = fma(pot, r1, a.y);
    } else {
      a.x = fma(rn, inv, a.x);
    }
  }
}

template <int PDE>
__global__ __launch_bounds__(kTile) void k_eval_partial(DevGeom g, int nt, const double* tg,
                                                        const double* mu, int64_t chunk,
                                                        double* partial) {
  constexpr bool stokes = PDE == kPdeStokes;
  constexpr int NW = kTile / 64, SD = stokes ? 2 : 1;
  __shared__ double2 sxy[kTile], sab[kTile], sm[stokes ? kTile : 1];
  __shared__ double red[NW][kTargets][SD];
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
  const int t0 = blockIdx.x * kTargets + lane;
  const int64_t lo = blockIdx.y * chunk;
  const int64_t hi = lo + chunk < g.n_points ? lo + chunk : g.n_points;
  double2 p[2], acc[2];
  bool far = false;
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int t = min(t0 + 64 * u, nt - 1);
    p[u] = make_double2(tg[2 * (int64_t)t], tg[2 * (int64_t)t + 1]);
    acc[u] = make_double2(0, 0);
    far = far || is_far(p[u]);
  }
  for (int64_t base = lo; base < hi; base += kTile) {
    const int64_t j = base + tid;
    bool slow = far;
    if (j < hi) {
      sxy[tid] = make_double2(g.pts[2 * j], g.pts[2 * j + 1]);
      slow = slow || is_far(sxy[tid]);
      const double n0 = g.nrm[2 * j], n1 = g.nrm[2 * j + 1], w = g.wts[j];
      if constexpr (stokes) {
        sab[tid] = make_double2(w * (1.0 / M_PI) * n0, w * (1.0 / M_PI) * n1);
        sm[tid] = make_double2(mu[2 * j], mu[2 * j + 1]);
      } else if constexpr (PDE == kPdeLaplaceNeumann) {
        sab[tid] = make_double2(w * (0.25 / M_PI) * mu[j], 0);
      } else {
        const double c = -w * (0.5 / M_PI) * mu[j];
        sab[tid] = make_double2(c * n0, c * n1);
      }
    }
    __syncthreads();
    const int q0 = 64 * wv, q1 = min((int64_t)q0 + 64, hi - base);
    // a wave's targets, and its own 64 sources of the tile
    if (!__any(slow)) {
#pragma unroll 4
      for (int q = q0; q < q1; q++)
#pragma unroll
        for (int u = 0; u < 2; u++)
          eval_pair<PDE, true>(p[u], sxy[q], sab[q], sm[stokes ? q : 0], acc[u]);
    } else {
      for (int q = q0; q < q1; q++)
#pragma unroll
        for (int u = 0; u < 2; u++)
          eval_pair<PDE, false>(p[u], sxy[q], sab[q], sm[stokes ? q : 0], acc[u]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 2; u++) {
    red[wv][lane + 64 * u][0] = acc[u].x;
    if constexpr (stokes) red[wv][lane + 64 * u][SD - 1] = acc[u].y;
  }
  __syncthreads();
  for (int i = tid; i < kTargets * SD; i += kTile) {
    const int t = blockIdx.x * kTargets + i / SD;
    if (t >= nt) continue;
    double v = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) v += red[w][i / SD][i % SD];
    partial[((int64_t)blockIdx.y * nt + t) * SD + i % SD] = v;
  }
}

// Sum chunks in order, add U_forward alpha (linear_solve.cpp:20-67 on the
// targets), zero targets outside the domain.
__global__ void k_eval_finish(DevGeom g, int nt, const double* tg,
                              const int* in_domain, const double* partial,
                              int nchunks, int n_holes, const double* hc,
                              const double* alpha, double* out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nt) return;
  const int sd = g.sol_dim;
  double a0 = 0, a1 = 0;
  for (int c = 0; c < nchunks; c++) {
    a0 += partial[(int64_t)c * sd * nt + (int64_t)sd * t];
    if (sd == 2) a1 += partial[(int64_t)c * sd * nt + (int64_t)sd * t + 1];
  }
  const double x0 = tg[2 * t], x1 = tg[2 * t + 1];
  for (int k = 0; k < n_holes && alpha; k++) {
    const double r0 = x0 - hc[2 * k], r1 = x1 - hc[2 * k + 1];
    const double rn = sqrt(r0 * r0 + r1 * r1);
    if (g.pde == kPdeStokes) {
      const double s = 1.0 / (4 * M_PI), rn2 = rn * rn;
      const double* al = alpha + 3 * k;
      a0 += s * (log(1 / rn) + r0 * r0 / rn2) * al[0] + s * (r0 * r1 / rn2) * al[1] +
            r1 * (s / rn2) * al[2];
      a1 += s * (r1 * r0 / rn2) * al[0] + s * (log(1 / rn) + r1 * r1 / rn2) * al[1] -
            r0 * (s / rn2) * al[2];
    } else {
      a0 += log(rn) * alpha[k];
    }
  }
  const bool inside = in_domain ? in_domain[t] != 0 : true;
  out[(int64_t)sd * t] = inside ? a0 : 0.0;
  if (sd == 2) out[(int64_t)sd * t + 1] = inside ? a1 : 0.0;
}

}  // namespace

int eval_scratch_address(int device, double** ptr) {
  static std::mutex mu;
  static double* addr[kEvalMaxDevices] = {};
  if (device < 0 || device >= kEvalMaxDevices || !ptr) return (int)hipErrorInvalidValue;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[device]) {
    // the device must be current: each GPU holds its own copy
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return (int)e;
    if (cur != device) return (int)hipErrorInvalidDevice;
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    addr[device] = static_cast<double*>(p);
  }
  *ptr = addr[device];
  return 0;
}

int64_t eval_scratch_need(int64_t n_points, int sol_dim, int64_t n_targets) {
  return (int64_t)eval_chunks(n_points, sol_dim, n_targets) * sol_dim * n_targets;
}

// At least one chunk per 8192 sources (64 at most), and more where the
// target blocks alone leave the chip idle: enough for 1024 workgroups (four
// per CU; a host call with 65,536 sources takes 98 us at 100 targets and 126
// at 1,000, against 203 and 205 with 8 chunks, 432 against 440 at 10,000),
// while a chunk keeps a tile of sources and the partial sums stay
// within the static scratch of the allocation-free call.
int eval_chunks(int64_t n_points, int sol_dim, int64_t n_targets) {
  const int64_t c = std::min<int64_t>(std::max<int64_t>((n_points + 8191) / 8192, 1), 64);
  const int64_t blocks = std::max<int64_t>((n_targets + kTargets - 1) / kTargets, 1);
  const int64_t fill = std::min((1024 + blocks - 1) / blocks, (n_points + kTile - 1) / kTile);
  const int64_t room = kEvalScratchElems / (sol_dim * std::max<int64_t>(n_targets, 1));
  return (int)std::max(c, std::min(fill, room));
}

void launch_eval(const DevGeom& g, int nt, const double* tg, const int* in_domain,
                 const double* mu, int n_holes, const double* hole_centers,
                 const double* alpha, double* partial, double* out,
                 hipStream_t st) {
  if (nt <= 0) return;
  const int nc = eval_chunks(g.n_points, g.sol_dim, nt);
  const int64_t chunk = (g.n_points + nc - 1) / nc;
  const dim3 grid((nt + kTargets - 1) / kTargets, nc);
  if (g.pde == kPdeStokes)
    k_eval_partial<kPdeStokes><<<grid, kTile, 0, st>>>(g, nt, tg, mu, chunk, partial);
  else if (g.pde == kPdeLaplaceNeumann)
    k_eval_partial<kPdeLaplaceNeumann><<<grid, kTile, 0, st>>>(g, nt, tg, mu, chunk, partial);
  else
    k_eval_partial<kPdeLaplace><<<grid, kTile, 0, st>>>(g, nt, tg, mu, chunk, partial);
  k_eval_finish<<<(nt + 255) / 256, 256, 0, st>>>(g, nt, tg, in_domain, partial, nc,
                                                  n_holes, hole_centers, alpha, out);
}

}  // namespace iegpu
