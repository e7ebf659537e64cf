// RS factorization and solve kernels for gfx950 (CDNA4, wave64).
//
// One workgroup per box of a tree level; levels run bottom-up (factor,
// upward sweep) or top-down (downward sweep) as stream-ordered launches,
// so the whole factorization is a fixed launch sequence with no host
// synchronisation (capturable in a HIP graph).
//
// Reference stages (paths relative to the reference root):
//   k_active    quadtree.cpp:1028-1074 (active = children's skeletons)
//   k_rows      kernel.cpp:293-423     (ID row count: near field + proxy)
//   k_assemble  kernel.cpp:123-591     (ID matrix assembly)
//   k_qrcp      ie_mat.cpp:548-588     (dgeqp3 rank cut + dtrtrs)
//   k_decouple  skel_factorization.cpp:77-128, 323-381
//   k_root_*    skel_factorization.cpp:172-186
//   k_sweep_*   skel_factorization.cpp:388-426, 507-592

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
// Level bookkeeping
// ---------------------------------------------------------------------------

__global__ void k_reset(DevState s) {
  if (threadIdx.x == 0) {
    s.err[0] = 0;
    s.err[1] = 0;
    s.err[2] = 0;
    s.err[3] = 0;
    // an incremental run appends new factor slots past the kept ones
    if (!s.dirty) *s.fac_top = 0;
  }
  if (threadIdx.x < kMaxLevels) s.njobs[threadIdx.x] = 0;
  for (int i = threadIdx.x; i < kMaxLevels * kNumLists; i += blockDim.x) s.lcnt[i] = 0;
}

// active(box) = concatenation of the children's outgoing lists (skeleton if
// compressed, active otherwise) in child order bl, tl, tr, br; a leaf's
// active list is its original DOF list.
__global__ __launch_bounds__(64) void k_active(DevTree t, DevState s,
                                               int start) {
  const int b = start + blockIdx.x;
  if (box_clean(s, b)) return;
  const int lane = threadIdx.x;
  int* dst = s.act_list + (int64_t)b * s.ncap;
  int n = 0;
  if (t.leaf[b]) {
    n = t.orig_cnt[b];
    if (n > s.ncap) {
      if (lane == 0) atomicOr(s.err, kErrBoxCap);
      n = 0;
    }
    const int* src = t.orig_dofs + t.orig_off[b];
    for (int i = lane; i < n; i += 64) dst[i] = src[i];
  } else {
    int pos = 0;
    for (int q = 0; q < 4; q++) {
      const int c = t.child[4 * b + q];
      const int cnt = min(max(s.out_cnt[c], 0), s.ncap);
      if (lane == 0) s.chpos[4 * b + q] = pos;
      if (pos + cnt <= s.ncap) {
        const int* src = s.out_list + (int64_t)c * s.ncap;
        for (int i = lane; i < cnt; i += 64) dst[pos + i] = src[i];
      }
      pos += cnt;
    }
    n = pos;
    if (n > s.ncap) {
      if (lane == 0) atomicOr(s.err, kErrBoxCap);
      n = 0;
    }
  }
  if (lane == 0) s.act_cnt[b] = n;
}

// Rank-model features of box b (every lane returns them): log2 |active|,
// log2 ID rows, level, log2(near rows + 1), side x mean and max |curvature|
// of the active DOFs, 1 - |mean normal| (how far the curve turns inside
// the box), -log10 tol, Stokes flag.
__device__ inline void box_features(const DevGeom& g, const DevTree& t, const DevState& s, int b,
                                    int level, int n, int m, int cnt, double tol, float* f) {
  const int lane = threadIdx.x & 63;
  const int* act = s.act_list + (int64_t)b * s.ncap;
  double ks = 0, km = 0, nx = 0, ny = 0;
  for (int i = lane; i < n; i += 64) {
    const DofGeo d = dof_geo(g, act[i]);
    const double k = fabs(d.k);
    ks += k;
    km = fmax(km, k);
    nx += d.n1;
    ny += d.n2;
  }
  ks = wave_total(ks);
  km = wave_max(km);
  nx = wave_total(nx);
  ny = wave_total(ny);
  const double side = t.side[b], nn = n > 0 ? n : 1;
  f[0] = (float)log2((double)nn);
  f[1] = (float)log2((double)(m > 0 ? m : 1));
  f[2] = (float)level;
  f[3] = (float)log2((double)cnt + 1.0);
  f[4] = (float)(side * ks / nn);
  f[5] = (float)(side * km);
  f[6] = (float)(1.0 - sqrt(nx * nx + ny * ny) / nn);
  f[7] = (float)(-log10(tol));
  f[8] = g.pde == kPdeStokes ? 1.0f : 0.0f;
}

// Rank predicted by the model for features f (lanes 0..kHid-1 own the
// hidden units; every lane returns the prediction).
__device__ inline float mlp_rank(const float* M, const float* f, float* hb) {
  const int lane = threadIdx.x & 63;
  const int j = lane & (kHid - 1);
  float z = M[kMlpB1 + j];
#pragma unroll
  for (int q = 0; q < kFeat; q++)
    z += M[kMlpW1 + q * kHid + j] * ((f[q] - M[kMlpMu + q]) / M[kMlpSd + q]);
  if (lane < kHid) hb[j] = tanhf(z);
  __syncthreads();
  float z2 = M[kMlpB2 + j];
  for (int i = 0; i < kHid; i++) z2 += M[kMlpW2 + i * kHid + j] * hb[i];
  double o = lane < kHid ? (double)(M[kMlpW3 + j] * tanhf(z2)) : 0.0;
  o = wave_total(o) + M[kMlpB3];
  return (float)o * M[kMlpYSd] + M[kMlpYMu];
}

__global__ __launch_bounds__(64) void k_rows(DevGeom g, DevTree t, DevState s,
                                             int start, int level, double tol) {
  __shared__ float hb[kHid];
  const int b = start + blockIdx.x;
  if (box_clean(s, b)) return;
  const int n = s.act_cnt[b];
  int m = 0;
  if (n >= kMinCompress) {
    const int cnt =
        for_each_row_dof(g, t, s, b, level >= 3, [](int, int) {});
    m = 2 * cnt + proxy_rows(g, level);
  }
  int kind = kQrcpNone;
  if (m > 0) {
    const int nch4 = id_chunks(m, kRegMaxRows), nch8 = id_chunks(m, kRegMaxRows8);
    if (n <= kRegMaxCols && m <= kRegMaxRows) kind = kQrcpReg;
    else if (n <= kRegMaxCols && nch4 <= kMaxChunks && nch4 * n <= kRegMaxRows)
      kind = kQrcpStack;
    else if (n <= kRegMaxCols8 && m <= kRegMaxRows8) kind = kQrcpReg8;
    else if (n <= kRegMaxCols8 && nch8 <= kMaxChunks && nch8 * n <= kRegMaxRows8)
      kind = kQrcpStack8;
    else kind = kQrcpLds;
  }
  if (threadIdx.x == 0) {
    s.m_rows[b] = m;
    s.qkind[b] = kind;
    // Scratch: the assembled matrix (and the general decouple's operands)
    // for the general QRCP, the stacked triangles for row compression;
    // register-QRCP boxes evaluate their entries in place.
    const int64_t ld = m > 2 * n ? m : 2 * n;
    int64_t scratch = kind == kQrcpLds ? ld * n : 0;
    if (kind == kQrcpStack || kind == kQrcpStack8)
      scratch = (int64_t)id_chunks(m, kind == kQrcpStack ? kRegMaxRows : kRegMaxRows8) * n * n;
    // A box that the Gram form takes needs its G and R instead, above 64 DOFs.
    if (s.gram && n > kRegMaxCols) {
      if (m > 0 && n <= kGramCols && m - proxy_rows(g, level) <= 2 * kGramNear)
        scratch = gram_scratch(n);
    } else if (s.gram && kind == kQrcpStack) {
      scratch = 0;
    }
    s.id_sz[b] = scratch;
    // k_decouple keeps the operands of a box with more than kSmallBox
    // active DOFs (n^2 + r^2 + 2 r k <= 2 n^2 entries) in the decouple pool
    // when they do not fit its LDS buffer.
    s.dec_sz[b] = n > kSmallBox ? 2 * (int64_t)n * n : 0;
    s.row_sz[b] = kind == kQrcpLds ? (m - proxy_rows(g, level)) / 2 : 0;
    // fac_sz holds a box's slot size; in an incremental run a re-factored
    // box whose kept slot fits its new factors reuses it (marked by the
    // negated size, which k_scan restores) instead of taking a new one.
    const int64_t need = (n > 0) ? fac_slot_size(n) : 0;
    const int64_t old = s.fac_sz[b];
    const bool reuse = s.dirty != nullptr && need <= old && s.fac_off[b] + old <= s.kept_top;
    s.fac_sz[b] = reuse ? -old : need;
  }
  // Sketch width: fixed, or from the rank model (0: straight to the full
  // QRCP when the predicted rank does not fit the widest sketch).  Boxes
  // too large for the narrow sketch on the top levels take the wide one.
  const int near = (m - proxy_rows(g, level)) / 2;
  const bool elig = s.rid_mode != 0 && (kind == kQrcpReg || kind == kQrcpStack) &&
                    near <= kRidMaxNear;
  const bool eligb = s.rid_mode != 0 && m > 0 && level <= kRidBigTop && n <= kRidBigCols &&
                     near <= kRidMaxNearW;
  // fixed widths keep the 64-row sketch to the top levels
  const bool eligw = s.rid_mode != 0 && m > 0 && n <= kRidWideCols && near <= kRidMaxNearW &&
                     (level <= kRidBigTop || s.rid_mode == 2);
  int w = elig ? s.rid_width : (eligw ? kRidRowsW : (eligb ? kRidRowsB : 0));
  if (m > 0 && (s.feat != nullptr || ((elig || eligw || eligb) && s.rid_mode == 2))) {
    float f[kFeat];
    box_features(g, t, s, b, level, n, m, near, tol, f);
    if (s.feat != nullptr && threadIdx.x == 0)
      for (int q = 0; q < kFeat; q++) s.feat[(int64_t)b * kFeat + q] = f[q];
    if ((elig || eligw || eligb) && s.rid_mode == 2) {
      // The narrowest sketch the predicted rank fits; a narrow sketch's box
      // past 26 below the top levels, where boxes are many and the register
      // QRCP takes them, and a box none is eligible for go straight to the
      // full QRCP.  The 64-row sketch is tried without the margin: a box it
      // fails goes on to the 128-row one, which costs more than as much
      // again.  For Laplace, whose ranks of 48 to 54 on level 1 the model
      // puts at 57 to 62, it is tried up to 14 past its limit (262,144 points:
      // 2.79 ms per factorization with those boxes sent straight to the
      // 128-row sketch, 2.62 so; an incremental one 2.36 and 2.14).
      const float kw = kRidRowsW - kRidOver + (g.pde == kPdeLaplace ? 14 : 0);
      const float kp = mlp_rank(s.rank_model, f, hb) + (float)s.rid_margin;
      w = (elig && kp <= 16 - kRidOver) ? 16
          : (elig && kp <= kRidRows - kRidOver) ? kRidRows
          : (elig && level > kRidBigTop) ? 0
          : (eligw && (kp - s.rid_margin <= kw || !eligb)) ? kRidRowsW
          : eligb ? kRidRowsB
                  : 0;
    }
  }
  if (threadIdx.x == 0) {
    s.sk_w[b] = w;
    s.rid_done[b] = 0;
    // The 128-row sketch's partial sums and rows of R (a box that a failed
    // 64-row sketch passes on to it takes its slot then).
    if (w == kRidRowsB) s.id_sz[b] = max(s.id_sz[b], rid_big_scratch(n));
    s.id_sz[b] = (s.id_sz[b] + 3) & ~int64_t(3);  // slots hold doubles
  }
  // Until its ID succeeds a box passes its active DOFs on uncompressed:
  // boxes a failed (retried) attempt never reaches still hold a consistent
  // outgoing list for the next level's k_active.
  const int* act = s.act_list + (int64_t)b * s.ncap;
  int* out = s.out_list + (int64_t)b * s.ncap;
  for (int i = threadIdx.x; i < n; i += 64) out[i] = act[i];
  if (threadIdx.x == 0) {
    s.rank[b] = 0;
    s.out_cnt[b] = n;
  }
}

// Scanned per box: ID scratch, row-list and factor sizes, register-QRCP
// and general-QRCP list entries, row-compression jobs, sketches, decouple
// operands, boxes above kSmallBox DOFs.
constexpr int kScanQ = 14;
constexpr int kScanLd = 16;      // words per block in scan_blk
constexpr int kScanMulti = 2048; // levels of at least this many boxes: three kernels

// What the scan reads of a box, loaded before any store (a load behind a
// store that may alias it waits for it).
struct ScanBox {
  int64_t id, row, fac, dec;
  int kind, n, w, jobs;
  bool on;
};

__device__ inline ScanBox scan_load(const DevState& s, int b) {
  ScanBox v;
  v.kind = s.qkind[b];
  v.n = s.act_cnt[b];
  v.w = s.sk_w[b];
  v.id = s.id_sz[b];
  v.row = s.row_sz[b];
  v.fac = s.fac_sz[b];
  v.dec = s.dec_sz[b];
  v.jobs = row_jobs(s, b);
  v.on = !box_clean(s, b);
  return v;
}

__device__ inline bool reg_kind(const ScanBox& v) {
  return v.kind == kQrcpReg || v.kind == kQrcpStack;
}

__device__ inline void scan_counts(const DevState& s, const ScanBox& v, int64_t (&own)[kScanQ]) {
  if (!v.on) return;
  own[0] += v.id;
  own[1] += v.row;
  own[2] += max(v.fac, int64_t(0));
  own[3] += (reg_kind(v) && v.n > kHalfCols) ? 1 : 0;
  own[7] += (reg_kind(v) && v.n <= kHalfCols) ? 1 : 0;
  own[4] += (v.kind == kQrcpLds) ? 1 : 0;
  own[5] += v.jobs;
  own[6] += (v.kind == kQrcpReg8 || v.kind == kQrcpStack8) ? 1 : 0;
  own[8] += (v.w > 0 && v.w <= kRidRows) ? 1 : 0;
  own[9] += (s.rid_mode != 0 && reg_kind(v) && v.w == 0) ? 1 : 0;
  own[10] += v.dec;
  own[11] += (v.w == kRidRowsW) ? 1 : 0;
  own[12] += (v.n > kSmallBox) ? 1 : 0;
  own[13] += (v.w == kRidRowsB) ? 1 : 0;
}

// Box b's slots and list entries from the exclusive offsets off (advanced
// past the box).
__device__ inline void scan_place(const DevState& s, const ScanBox& v, int b, int start,
                                  int level, int64_t fbase, int64_t (&off)[kScanQ]) {
  if (!v.on) return;
  auto list = [&](int L) { return s.lists + (int64_t)L * s.nbox + start; };
  int* jobs = s.jobs + (int64_t)2 * kMaxChunks * start;
  // Scratch of odd and even levels in separate halves: a level's ID runs
  // while the level below it is still being decoupled.
  s.id_off[b] = (level & 1) * s.id_cap + off[0];
  s.big_off[b] = s.id_off[b];
  s.row_off[b] = off[1];
  if (v.fac < 0) {  // keeps its slot
    s.fac_sz[b] = -v.fac;
  } else {
    s.fac_off[b] = fbase + off[2];
    off[2] += v.fac;
  }
  s.dec_off[b] = off[10];
  off[10] += v.dec;
  off[0] += v.id;
  off[1] += v.row;
  if (reg_kind(v)) {
    if (v.n > kHalfCols) list(kLstReg)[off[3]++] = b;
    else list(kLstRegHalf)[off[7]++] = b;
  }
  if (v.kind == kQrcpLds) list(kLstLds)[off[4]++] = b;
  if (v.kind == kQrcpReg8 || v.kind == kQrcpStack8) list(kLstReg8)[off[6]++] = b;
  if (v.w > 0 && v.w <= kRidRows) list(kLstRid)[off[8]++] = b;
  if (v.w == kRidRowsW) list(kLstRidWide)[off[11]++] = b;
  if (v.w == kRidRowsB) list(kLstRidBig)[off[13]++] = b;
  // A register-QRCP box the randomized ID does not sketch goes to the full
  // QRCP list.
  if (s.rid_mode != 0 && reg_kind(v) && v.w == 0) list(kLstFallback)[off[9]++] = b;
  if (v.n > kSmallBox) list(kLstBig)[off[12]++] = b;
  for (int q = 0; q < v.jobs; q++) {
    jobs[2 * off[5]] = b;
    jobs[2 * off[5] + 1] = q;
    off[5]++;
  }
}

// The level's list lengths, pool checks and the factor-pool top.  ok:
// pools_ok before this level.
__device__ inline void scan_finish(const DevState& s, int level, const int64_t* tot,
                                   int64_t fbase, bool ok) {
  const int64_t ta = tot[0], tb = tot[1], tc = tot[2];
  list_slot(s, level, kLstReg)[0] = (int)tot[3];
  list_slot(s, level, kLstLds)[0] = (int)tot[4];
  list_slot(s, level, kLstReg8)[0] = (int)tot[6];
  list_slot(s, level, kLstRegHalf)[0] = (int)tot[7];
  list_slot(s, level, kLstRid)[0] = (int)tot[8];
  list_slot(s, level, kLstRidWide)[0] = (int)tot[11];
  list_slot(s, level, kLstRidBig)[0] = (int)tot[13];  // k_rid_wide appends
  list_slot(s, level, kLstFallback)[0] = (int)tot[9];  // k_rid appends
  list_slot(s, level, kLstBig)[0] = (int)tot[12];
  s.njobs[level] = (int)tot[5];
  s.id_top[level] = ta;
  int e = 0;
  if (ta > s.id_cap) {
    e |= kErrIdPool;
    atomicMax(s.err + 2, (int)((ta + 1023) >> 10));  // size needed, in 1024 elements
  }
  if (tb > s.row_cap) {
    e |= kErrRowPool;
    atomicMax(s.err + 3, (int)((tb + 1023) >> 10));
  }
  if (fbase + tc > s.fac_cap) e |= kErrFacPool;
  if (tot[10] > s.dec_cap) {
    e |= kErrDecPool;
    atomicMax(s.err + 1, (int)((tot[10] + 1023) >> 10));
  }
  if (e) atomicOr(s.err, e);
  s.halt[level] = (e != 0 || !ok) ? 1 : 0;
  *s.fac_top = fbase + tc;
}

// Exclusive scan of the kScanQ values of the block's threads (NT a
// multiple of 64): off = sum over lower threads; tot (LDS, kScanQ) = the
// block's totals.  wtot: kScanQ x NT/64 LDS words.
template <int NT>
__device__ inline void block_scan(const int64_t (&own)[kScanQ], int64_t (&off)[kScanQ],
                                  int64_t (*wtot)[NT / 64], int64_t* tot) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int64_t inc[kScanQ];
#pragma unroll
  for (int q = 0; q < kScanQ; q++) {
    const int64_t v = wave_scan(own[q]);
    inc[q] = v;
    if (lane == 63) wtot[q][wv] = v;
  }
  __syncthreads();
  if (tid < kScanQ) {
    int64_t run = 0;
    for (int w = 0; w < NT / 64; w++) {
      const int64_t t = wtot[tid][w];
      wtot[tid][w] = run;
      run += t;
    }
    tot[tid] = run;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kScanQ; q++) off[q] = wtot[q][wv] + inc[q] - own[q];
}

// Exclusive scans of the per-box sizes of one level (single workgroup of
// one wave, four or sixteen by the level's boxes; each thread a contiguous
// chunk of boxes).  Latency: sixteen waves at every level, scanning through
// ds_bpermute with every load behind a store, took 11 to 14 us; 4.6, 5.6 and
// 12 us with DPP scans, the loads first and the waves the level needs.  ID scratch and row lists are
// level-local; factor slots append to the running pool offset.
// With the randomized ID, a register-QRCP box that gets no sketch (not
// eligible, or sent straight to the full QRCP by the rank model) starts the
// level's full-QRCP list; k_rid appends the boxes whose sketch fails.
template <int NT>
__global__ __launch_bounds__(NT) void k_scan(DevState s, int start, int count, int level) {
  __shared__ int64_t wtot[kScanQ][NT / 64];
  __shared__ int64_t tot[kScanQ];
  const int tid = threadIdx.x;
  const int chunk = (count + NT - 1) / NT;
  const int lo = min(count, tid * chunk), hi = min(count, lo + chunk);
  int64_t own[kScanQ] = {};
  for (int i = lo; i < hi; i++) scan_counts(s, scan_load(s, start + i), own);
  int64_t off[kScanQ];
  block_scan<NT>(own, off, wtot, tot);
  const int64_t fbase = *s.fac_top;
  const bool pools = pools_ok(s);
  for (int i = lo; i < hi; i++)
    scan_place(s, scan_load(s, start + i), start + i, start, level, fbase, off);
  __syncthreads();
  if (tid == 0) scan_finish(s, level, tot, fbase, pools);
}

// The same for levels of kScanMulti boxes or more over many workgroups of
// 256 boxes (one workgroup walked them at one chunk of boxes per thread
// at 15-70 us per level): each block's totals (k_scan_blocks), their
// exclusive scan and the level's totals (k_scan_totals; the factor-pool
// base goes after the block offsets), then each box's offsets
// (k_scan_place).  Same offsets and list order as k_scan.
__global__ __launch_bounds__(256) void k_scan_blocks(DevState s, int start, int count) {
  __shared__ int64_t wtot[kScanQ][4];
  __shared__ int64_t tot[kScanQ];
  const int i = blockIdx.x * 256 + threadIdx.x;
  int64_t own[kScanQ] = {};
  if (i < count) scan_counts(s, scan_load(s, start + i), own);
  int64_t off[kScanQ];
  block_scan<256>(own, off, wtot, tot);
  if (threadIdx.x < kScanQ) s.scan_blk[(int64_t)blockIdx.x * kScanLd + threadIdx.x] = tot[threadIdx.x];
}

__global__ __launch_bounds__(1024) void k_scan_totals(DevState s, int nblk, int level) {
  __shared__ int64_t wtot[kScanQ][16];
  __shared__ int64_t tot[kScanQ];
  const int tid = threadIdx.x;
  const int chunk = (nblk + 1023) / 1024;
  const int lo = min(nblk, tid * chunk), hi = min(nblk, lo + chunk);
  int64_t own[kScanQ] = {};
  for (int j = lo; j < hi; j++)
#pragma unroll
    for (int q = 0; q < kScanQ; q++) own[q] += s.scan_blk[(int64_t)j * kScanLd + q];
  int64_t off[kScanQ];
  block_scan<1024>(own, off, wtot, tot);
  for (int j = lo; j < hi; j++)
#pragma unroll
    for (int q = 0; q < kScanQ; q++) {
      int64_t* w = s.scan_blk + (int64_t)j * kScanLd + q;
      const int64_t t = *w;
      *w = off[q];
      off[q] += t;
    }
  __syncthreads();
  if (tid == 0) {
    const int64_t fbase = *s.fac_top;
    s.scan_blk[(int64_t)nblk * kScanLd] = fbase;
    scan_finish(s, level, tot, fbase, pools_ok(s));
  }
}

__global__ __launch_bounds__(256) void k_scan_place(DevState s, int start, int count,
                                                    int level, int nblk) {
  __shared__ int64_t wtot[kScanQ][4];
  __shared__ int64_t tot[kScanQ];
  const int i = blockIdx.x * 256 + threadIdx.x;
  int64_t own[kScanQ] = {};
  ScanBox v = {};
  if (i < count) {
    v = scan_load(s, start + i);
    scan_counts(s, v, own);
  }
  int64_t off[kScanQ];
  block_scan<256>(own, off, wtot, tot);
  if (i >= count) return;
  const int64_t* base = s.scan_blk + (int64_t)blockIdx.x * kScanLd;
#pragma unroll
  for (int q = 0; q < kScanQ; q++) off[q] += base[q];
  scan_place(s, v, start + i, start, level, s.scan_blk[(int64_t)nblk * kScanLd], off);
}


// ---------------------------------------------------------------------------
// ID matrix assembly: [K(ic, box); K(box, ic)^T; proxy] (m x n,
// column-major, ld m), kernel.cpp:293-423.  The register QR kernels
// evaluate their boxes' entries in place; this kernel writes the matrix of
// the boxes the general QRCP takes.
// ---------------------------------------------------------------------------

template <typename R>
__global__ __launch_bounds__(256) void k_assemble(DevGeom g, DevTree t,
                                                  DevState s, int start,
                                                  int level) {
  __shared__ double pxy[4][kNumProxy];
  if (!pools_ok(s)) return;
  const int nl = list_count(s, level, kLstLds);
  for (int li = blockIdx.x; li < nl; li += gridDim.x) {
    const int b = list_at(s, start, kLstLds, li);
    if (s.rid_done[b]) continue;  // a sketch took it
    const int m = s.m_rows[b];
    const int n = s.act_cnt[b];
    const int tid = threadIdx.x;
    const int* act = s.act_list + (int64_t)b * s.ncap;
    int* rows = s.row_pool + s.row_off[b];
    R* A = reinterpret_cast<R*>(s.id_pool) + s.id_off[b];
    const int cnt = id_setup(g, t, s, b, level, m, rows, pxy);
    __syncthreads();
    const double pw = proxy_weight(t, b);
    for (int i = tid; i < m; i += 256) {
      const IdRow rw = id_row(g, rows, cnt, pxy, pw, i);
      for (int j = 0; j < n; j++)
        A[i + (int64_t)m * j] = static_cast<R>(id_entry(g.pde, rw, dof_geo(g, act[j])));
    }
    __syncthreads();
  }
}

}  // namespace

void launch_active(const DevTree& t, const DevState& s, int start, int count, hipStream_t st) {
  k_active<<<count, 64, 0, st>>>(t, s, start);
}

void launch_reset(const DevState& s, hipStream_t st) {
  k_reset<<<1, 64, 0, st>>>(s);
}

template <typename R>
void launch_factor_stage(int stage, const DevGeom& g, const DevTree& t,
                         const DevState& s, int level, int start, int count,
                         int listed, double tol, const LaunchCaps& caps, hipStream_t st, int skip,
                         hipStream_t st_big) {
  if (count <= 0 || listed <= 0) return;
  switch (stage) {
    case kStageActive:
      k_active<<<count, 64, 0, st>>>(t, s, start);
      break;
    case kStageRows:
      k_rows<<<count, 64, 0, st>>>(g, t, s, start, level, tol);
      break;
    case kStageScan:
      if (count >= kScanMulti) {
        const int nblk = (count + 255) / 256;
        k_scan_blocks<<<nblk, 256, 0, st>>>(s, start, count);
        k_scan_totals<<<1, 1024, 0, st>>>(s, nblk, level);
        k_scan_place<<<nblk, 256, 0, st>>>(s, start, count, level, nblk);
      } else if (count > 256) {
        k_scan<1024><<<1, 1024, 0, st>>>(s, start, count, level);
      } else if (count > 64) {
        k_scan<256><<<1, 256, 0, st>>>(s, start, count, level);
      } else {
        k_scan<64><<<1, 64, 0, st>>>(s, start, count, level);
      }
      break;
    case kStageAssemble:
      if (!(skip & kSkipAssemble) && !s.gram)
        k_assemble<R><<<min(listed, caps.assemble), 256, 0, st>>>(g, t, s, start, level);
      break;
    case kStageRid:
      if (s.rid_mode != 0) launch_rid<R>(g, t, s, level, start, listed, tol, st, skip);
      break;
    case kStageQrcp:
      if constexpr (sizeof(R) == 4) {
        if (s.gram) {
          launch_gram<R>(g, t, s, level, start, listed, tol, st, skip);
          if (skip & kSkipAssemble) break;
          // the boxes too large for it
          k_assemble<R><<<min(listed, caps.assemble), 256, 0, st>>>(g, t, s, start, level);
          skip |= kSkipRegQrcp | kSkipReg8Qrcp;
        }
      }
      launch_qrcp<R>(g, t, s, level, start, listed, tol, caps, st, skip);
      break;
    case kStageDecouple:
      launch_decouple<R>(g, t, s, level, start, count, listed, caps, st, skip, st_big);
      break;
    default:
      break;
  }
}

#define IEGPU_INSTANTIATE(R)                                                   \
  template void launch_factor_stage<R>(int, const DevGeom&, const DevTree&,   \
                                       const DevState&, int, int, int, int,    \
                                       double, const LaunchCaps&, hipStream_t, int, \
                                       hipStream_t);

IEGPU_INSTANTIATE(double)
IEGPU_INSTANTIATE(float)

}  // namespace iegpu
