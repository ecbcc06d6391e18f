// Supernodal forward/backward solves over the level schedule, multi-RHS.
//
// Reference (one rhs, recursive): src/taucs_sn_llt.c:2597-2720 (forward:
// gather, trsm, gemm, scatter) and :2723-2841 (backward: gather, gemm^T,
// trsm^T, scatter).  Here each front owns an m x nrhs workspace block W_f
// (column-major, at W + offW * nrhs):
//   forward:  W_f[0:s] starts as b[cols], W_f[s:m] as 0; children add their
//             update parts at the relative rows (fixed order, no atomics);
//             then, 64 columns at a time, y_blk = inv(L_kk) w_blk (the block
//             inverses come from the factorization) and every row below the
//             block is updated by many workgroups: W_f[r] -= L[r, blk] y_blk.
//             y is kept in Y, indexed by global column.
//   backward: top-down.  W_f[s:m] receives x of the update rows from the
//             ancestors; z = y - L21^T x2 is formed one wave per column
//             (k_bwd_cols); then blocks from the last to the first:
//             x_blk = inv(L_kk)^T z_blk and the update of every earlier
//             column by the block's rows (k_bwd_step).
// Right-hand sides are processed 16 at a time (nrhs <= 16 per call).
#include "kernels.h"

namespace tamd {

#define SMAXR 16

// W_f <- [b(cols, :); 0].  One wave per task (a front's rows r0 .. r0+nr-1,
// nr <= 64), four tasks per workgroup.
template <typename T>
__global__ __launch_bounds__(256) void k_solve_init(const FrontDesc* __restrict__ fr,
                                                    const PanelTask* __restrict__ tasks, int count,
                                                    const int* __restrict__ rows,
                                                    const double* __restrict__ b, int ldb,
                                                    T* __restrict__ W, int nrhs)
{
  const int ti = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (ti >= count) return;
  const PanelTask t = tasks[ti];
  const FrontDesc d = fr[t.front];
  const int i = t.r0 + lane;
  if (lane >= t.nr) return;
  T* w = W + d.offW * nrhs + i;
  const int col = i < d.s ? rows[d.rows + i] : 0;
  for (int r = 0; r < nrhs; r++)
    w[(long long)r * d.m] = i < d.s ? (T)b[col + (long long)r * ldb] : (T)0;
}

// ---- LDS-tiled pieces ---------------------------------------------------------
// All block operations work on 64 x 64 tiles of L staged in LDS (Lt[i + j*65],
// loaded column by column so global reads are coalesced) against small
// 64 x nrhs blocks of right-hand-side values (V[i + r*64]).  A 256-thread
// workgroup assigns thread t to tile row/column t % 64 and right-hand sides
// 4*(t/64) .. 4*(t/64)+3.

template <typename T>
__device__ __forceinline__ void load_tile(T* Lt, const T* src, long long ld, int nr, int nc)
{
  // src(i, j) = src[i + j*ld], i < nr rows, j < nc columns; zero padded
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    int i = e & 63, j = e >> 6;
    Lt[i + j * 65] = (i < nr && j < nc) ? src[i + (long long)j * ld] : (T)0;
  }
}

template <typename T>
__device__ __forceinline__ void load_inv(T* It, const T* iv)
{
  // row-major 64 x 64 inverse block -> It[i + q*65] = inv(i, q)
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    int q = e & 63, i = e >> 6;
    It[i + q * 65] = iv[i * 64 + q];
  }
}

// The same two loads issued together: all 32 global loads of a thread are in
// flight before the first LDS store (the step kernels are latency-bound).
template <typename T>
__device__ __forceinline__ void load_inv_and_tile(T* It, const T* iv, T* Lt, const T* src,
                                                  long long ld, int nr, int nc)
{
  T a[16], b[16];
#pragma unroll
  for (int u = 0; u < 16; u++) {
    const int e = threadIdx.x + 256 * u;
    a[u] = iv[e];
    const int i = e & 63, j = e >> 6;
    b[u] = (i < nr && j < nc) ? src[i + (long long)j * ld] : (T)0;
  }
#pragma unroll
  for (int u = 0; u < 16; u++) {
    const int e = threadIdx.x + 256 * u;
    It[(e >> 6) + (e & 63) * 65] = a[u];
    Lt[(e & 63) + (e >> 6) * 65] = b[u];
  }
}

// One 64-column block step of the forward solve.  Every task forms
// y_blk = inv(L_kk) w_blk from the block's rows of W_f (read-only in this
// step) and updates its 64 rows of the diagonal block's column range below
// the block: W_f[r] -= L[r, blk] y_blk (rows inside L11 only; the L21 rows
// get one pass with all columns in k_fwd_rect).  The task whose rows start
// right below the block also stores y_blk into Y (by global column).
template <typename T>
__global__ __launch_bounds__(256) void k_fwd_step(const FrontDesc* __restrict__ fr,
                                                  const PanelTask* __restrict__ tasks,
                                                  const int* __restrict__ rows,
                                                  const T* __restrict__ L,
                                                  const T* __restrict__ Inv, T* __restrict__ W,
                                                  T* __restrict__ Y, int ldy, int nrhs)
{
  __shared__ T It[64 * 65];
  __shared__ T Lt[64 * 65];
  __shared__ T Wb[64 * SMAXR];
  __shared__ T Yb[64 * SMAXR];
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc d = fr[t.front];
  const int m = d.m, kb = t.kb, tid = threadIdx.x;
  T* w = W + d.offW * nrhs;
  load_inv_and_tile(It, Inv + d.offI + (long long)(t.k0 / 64) * 4096, Lt,
                    L + d.offL + t.r0 + (long long)t.k0 * m, m, t.nr, kb);
  for (int e = tid; e < 64 * nrhs; e += 256) {
    int i = e & 63, r = e >> 6;
    Wb[i + r * 64] = i < kb ? w[t.k0 + i + r * m] : (T)0;
  }
  __syncthreads();
  for (int e = tid; e < 64 * nrhs; e += 256) {
    int i = e & 63, r = e >> 6;
    T acc = (T)0;
    for (int q = 0; q <= i; q++) acc += It[i + q * 65] * Wb[q + r * 64];
    Yb[i + r * 64] = acc;
  }
  __syncthreads();
  if (t.r0 == t.k0 + kb) {
    const int* rw = rows + d.rows + t.k0;
    for (int e = tid; e < kb * nrhs; e += 256) {
      int i = e % kb, r = e / kb;
      Y[rw[i] + (long long)r * ldy] = Yb[i + r * 64];
    }
  }
  if (t.nr <= 0) return;
  const int i = tid & 63, g = tid >> 6;
  if (i < t.nr) {
    for (int q = 0; q < 4; q++) {
      int r = 4 * g + q;
      if (r >= nrhs) break;
      T acc = (T)0;
      for (int j = 0; j < kb; j++) acc += Lt[i + j * 65] * Yb[j + r * 64];
      w[t.r0 + i + r * m] -= acc;
    }
  }
}

// L21 rows of the forward solve, split over column chunks: the task's rows
// r0..r0+nr-1 (>= s) times y of columns [c0, c0+nc) (k0 = c0, kb = nc) into
// the partial block Part[slot] (64 x nrhs); k_fwd_rect_reduce subtracts the
// partial blocks from W_f in slot order, so the sum is deterministic.
template <typename T>
__global__ __launch_bounds__(256) void k_fwd_rect(const FrontDesc* __restrict__ fr,
                                                  const PanelTask* __restrict__ tasks,
                                                  const int* __restrict__ rows,
                                                  const T* __restrict__ L,
                                                  const T* __restrict__ Y, int ldy,
                                                  T* __restrict__ Part, int nrhs)
{
  __shared__ T Lt[64 * 65];
  __shared__ T Yc[64 * SMAXR];
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc d = fr[t.front];
  const int m = d.m, tid = threadIdx.x, i = tid & 63, g = tid >> 6;
  const int* rw = rows + d.rows;
  T acc[4] = {(T)0, (T)0, (T)0, (T)0};
  for (int c0 = t.k0; c0 < t.k0 + t.kb; c0 += 64) {
    const int nc = t.k0 + t.kb - c0 < 64 ? t.k0 + t.kb - c0 : 64;
    __syncthreads();
    load_tile(Lt, L + d.offL + t.r0 + (long long)c0 * m, m, t.nr, nc);
    for (int e = tid; e < 64 * nrhs; e += 256) {
      int j = e & 63, r = e >> 6;
      Yc[j + r * 64] = j < nc ? Y[rw[c0 + j] + (long long)r * ldy] : (T)0;
    }
    __syncthreads();
    for (int q = 0; q < 4; q++) {
      int r = 4 * g + q;
      if (r >= nrhs) break;
      T a = (T)0;
      for (int j = 0; j < nc; j++) a += Lt[i + j * 65] * Yc[j + r * 64];
      acc[q] += a;
    }
  }
  T* part = Part + (long long)blockIdx.x * (64LL * nrhs);
  for (int q = 0; q < 4; q++) {
    int r = 4 * g + q;
    if (r >= nrhs) break;
    part[i + r * 64] = acc[q];
  }
}

// W_f[r0 + i] -= sum over slots k0 .. k0+kb-1 of Part[slot][i]
template <typename T>
__global__ void k_fwd_rect_reduce(const FrontDesc* __restrict__ fr,
                                  const PanelTask* __restrict__ tasks,
                                  const T* __restrict__ Part, T* __restrict__ W, int nrhs)
{
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc d = fr[t.front];
  T* w = W + d.offW * nrhs;
  for (int e = threadIdx.x; e < 64 * nrhs; e += blockDim.x) {
    int i = e & 63, r = e >> 6;
    if (i >= t.nr) continue;
    T sum = (T)0;
    for (int q = 0; q < t.kb; q++) sum += Part[(long long)(t.k0 + q) * (64LL * nrhs) + i + r * 64];
    w[t.r0 + i + r * d.m] -= sum;
  }
}

// dst[k * ldd] += src[k * lds] for the right-hand sides k < nrhs, eight at a
// time with all loads before the stores (child and parent rows are distinct
// memory, which the compiler cannot know: both lie in the workspace).
template <typename T>
__device__ __forceinline__ void ext_row(T* dst, int ldd, const T* src, int lds, int nrhs)
{
  for (int k0 = 0; k0 < nrhs; k0 += 8) {
    T a[8], b[8];
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (k0 + k < nrhs) {
        a[k] = src[(long long)(k0 + k) * lds];
        b[k] = dst[(long long)(k0 + k) * ldd];
      }
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (k0 + k < nrhs) dst[(long long)(k0 + k) * ldd] = b[k] + a[k];
  }
}

// Child update rows added into the parent's workspace (rows r0..r0+nr-1 of
// the child's update part).
template <typename T>
__global__ void k_solve_ext(const FrontDesc* __restrict__ fr, const PanelTask* __restrict__ tasks,
                            const int* __restrict__ rel, T* __restrict__ W, int nrhs)
{
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc c = fr[t.front];
  const FrontDesc p = fr[c.parent];
  const int* r = rel + c.rel;
  T* wp = W + p.offW * nrhs;
  const T* wc = W + c.offW * nrhs + c.s;
  const int i = t.r0 + threadIdx.x;
  if (threadIdx.x >= t.nr) return;
  ext_row(wp + r[i], p.m, wc + i, c.m, nrhs);
}

// The children's updates of a level in one launch: one workgroup per parent, or
// per piece of a wide parent's rows, heads[b] = {front: first task, k0: count}, a
// task the rows r0 .. r0+nr-1 of a child's update part, added in sibling-rank
// order, so each parent row receives its children's values in that order.
// By a workgroup, or (WAVE) by one wave, whose memory operations are performed in
// order: no barrier between children.
template <typename T, bool WAVE>
__device__ __forceinline__ void ext_head(const FrontDesc* __restrict__ fr, const PanelTask h,
                                         const PanelTask* __restrict__ tasks, const int* __restrict__ rel,
                                         T* W, int nrhs)
{
  PanelTask t = tasks[h.front];
  FrontDesc c = fr[t.front];
  const FrontDesc p = fr[c.parent];
  T* wp = W + p.offW * nrhs;
  for (int q = 0; q < h.k0; q++) {
    if (!WAVE && q > 0) __syncthreads();
    const int* r = rel + c.rel + t.r0;
    const T* wc = W + c.offW * nrhs + c.s + t.r0;
    const int m = c.m, nr = t.nr;
    if (q + 1 < h.k0) {
      t = tasks[h.front + q + 1];
      c = fr[t.front];
    }
    for (int i = WAVE ? threadIdx.x & 63 : threadIdx.x; i < nr; i += WAVE ? 64 : 256)
      ext_row(wp + r[i], p.m, wc + i, m, nrhs);
    if (WAVE) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_solve_ext_seq(const FrontDesc* __restrict__ fr,
                                                       const PanelTask* __restrict__ heads,
                                                       const PanelTask* __restrict__ tasks,
                                                       const int* __restrict__ rel, T* W, int nrhs)
{
  ext_head<T, false>(fr, heads[blockIdx.x], tasks, rel, W, nrhs);
}

// The same with one parent per wave, four to a workgroup, for launches of so many
// parents that they fill the chip: children of a few rows leave most of a
// workgroup's threads idle, and a child's descriptors, places and values are a
// chain of loads, so that what bounds a launch is the parents in flight.
// 512 grids of 16 to 128 points a side, 75 thousand parents in a launch, one
// right-hand side: 291 -> 113 us.  The first `wide` parents, which would keep a wave
// long, have a workgroup each.
template <typename T>
__global__ __launch_bounds__(256) void k_solve_ext_wave(const FrontDesc* __restrict__ fr,
                                                        const PanelTask* __restrict__ heads, int wide,
                                                        int nheads, const PanelTask* __restrict__ tasks,
                                                        const int* __restrict__ rel, T* W, int nrhs)
{
  const int b = blockIdx.x;
  if (b < wide) {
    ext_head<T, false>(fr, heads[b], tasks, rel, W, nrhs);
    return;
  }
  const int hd = wide + 4 * (b - wide) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (hd < nheads) ext_head<T, true>(fr, heads[hd], tasks, rel, W, nrhs);
}

// Backward: W_f[s + i] <- x(update row i) for rows r0..r0+nr-1 of the update part.
template <typename T>
__global__ void k_bwd_gather(const FrontDesc* __restrict__ fr, const PanelTask* __restrict__ tasks,
                             const int* __restrict__ rows, const double* __restrict__ x, int ldx,
                             T* __restrict__ W, int nrhs)
{
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc d = fr[t.front];
  const int i = t.r0 + threadIdx.x;
  if (threadIdx.x >= t.nr) return;
  const int gi = rows[d.rows + d.s + i];
  T* w = W + d.offW * nrhs + d.s;
  for (int r = 0; r < nrhs; r++) w[i + r * d.m] = (T)x[gi + (long long)r * ldx];
}

// z = y - L21^T x2, split over row chunks: columns [r0, r0+nr) of a front
// times the update rows [k0, k0+kb) (>= s) into Part[slot];
// k_bwd_cols_reduce subtracts the partials from Y in slot order.
template <typename T>
__global__ __launch_bounds__(256) void k_bwd_cols(const FrontDesc* __restrict__ fr,
                                                  const PanelTask* __restrict__ tasks,
                                                  const T* __restrict__ L,
                                                  const T* __restrict__ W,
                                                  T* __restrict__ Part, int nrhs)
{
  __shared__ T Lt[64 * 65];
  __shared__ T Xc[64 * SMAXR];
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc d = fr[t.front];
  const int m = d.m, tid = threadIdx.x, j = tid & 63, g = tid >> 6;
  const T* w = W + d.offW * nrhs;
  T acc[4] = {(T)0, (T)0, (T)0, (T)0};
  for (int i0 = t.k0; i0 < t.k0 + t.kb; i0 += 64) {
    const int ni = t.k0 + t.kb - i0 < 64 ? t.k0 + t.kb - i0 : 64;
    __syncthreads();
    load_tile(Lt, L + d.offL + i0 + (long long)t.r0 * m, m, ni, t.nr);
    for (int e = tid; e < 64 * nrhs; e += 256) {
      int ii = e & 63, r = e >> 6;
      Xc[ii + r * 64] = ii < ni ? w[i0 + ii + r * m] : (T)0;
    }
    __syncthreads();
    for (int q = 0; q < 4; q++) {
      int r = 4 * g + q;
      if (r >= nrhs) break;
      T a = (T)0;
      for (int ii = 0; ii < ni; ii++) a += Lt[ii + j * 65] * Xc[ii + r * 64];
      acc[q] += a;
    }
  }
  T* part = Part + (long long)blockIdx.x * (64LL * nrhs);
  for (int q = 0; q < 4; q++) {
    int r = 4 * g + q;
    if (r >= nrhs) break;
    part[j + r * 64] = acc[q];
  }
}

// Y[col(r0 + j)] -= sum over slots k0 .. k0+kb-1 of Part[slot][j]
template <typename T>
__global__ void k_bwd_cols_reduce(const FrontDesc* __restrict__ fr,
                                  const PanelTask* __restrict__ tasks,
                                  const int* __restrict__ rows, const T* __restrict__ Part,
                                  T* __restrict__ Y, int ldy, int nrhs)
{
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc d = fr[t.front];
  for (int e = threadIdx.x; e < 64 * nrhs; e += blockDim.x) {
    int j = e & 63, r = e >> 6;
    if (j >= t.nr) continue;
    T sum = (T)0;
    for (int q = 0; q < t.kb; q++) sum += Part[(long long)(t.k0 + q) * (64LL * nrhs) + j + r * 64];
    Y[rows[d.rows + t.r0 + j] + (long long)r * ldy] -= sum;
  }
}

// One 64-column block step of the backward solve (blocks from the last to
// the first).  Every task forms x_blk = inv(L_kk)^T z_blk from the block's
// entries of Y (read-only in this step) and updates its 64 columns
// j in [r0, r0+nr) < k0: z_j -= sum_{i in blk} L[i][j] x_i.  The task with
// r0 == 0 also stores x_blk into the solution.
template <typename T>
__global__ __launch_bounds__(256) void k_bwd_step(const FrontDesc* __restrict__ fr,
                                                  const PanelTask* __restrict__ tasks,
                                                  const int* __restrict__ rows,
                                                  const T* __restrict__ L,
                                                  const T* __restrict__ Inv, T* __restrict__ Y,
                                                  int ldy, double* __restrict__ x, int ldx,
                                                  int nrhs)
{
  __shared__ T It[64 * 65];
  __shared__ T Lt[64 * 65];
  __shared__ T Zb[64 * SMAXR];
  __shared__ T Xb[64 * SMAXR];
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc d = fr[t.front];
  const int m = d.m, kb = t.kb, tid = threadIdx.x;
  const int* rw = rows + d.rows;
  load_inv_and_tile(It, Inv + d.offI + (long long)(t.k0 / 64) * 4096, Lt,
                    L + d.offL + t.k0 + (long long)t.r0 * m, m, kb, t.nr);
  for (int e = tid; e < 64 * nrhs; e += 256) {
    int i = e & 63, r = e >> 6;
    Zb[i + r * 64] = i < kb ? Y[rw[t.k0 + i] + (long long)r * ldy] : (T)0;
  }
  __syncthreads();
  for (int e = tid; e < 64 * nrhs; e += 256) {
    int i = e & 63, r = e >> 6;
    T acc = (T)0;
    for (int q = i; q < kb; q++) acc += It[q + i * 65] * Zb[q + r * 64];
    Xb[i + r * 64] = acc;
  }
  __syncthreads();
  if (t.r0 == 0) {
    for (int e = tid; e < kb * nrhs; e += 256) {
      int i = e % kb, r = e / kb;
      x[rw[t.k0 + i] + (long long)r * ldx] = (double)Xb[i + r * 64];
    }
  }
  if (t.nr <= 0) return;
  const int j = tid & 63, g = tid >> 6;
  if (j < t.nr) {
    const int gj = rw[t.r0 + j];
    for (int q = 0; q < 4; q++) {
      int r = 4 * g + q;
      if (r >= nrhs) break;
      T acc = (T)0;
      for (int i = 0; i < kb; i++) acc += Lt[i + j * 65] * Xb[i + r * 64];
      Y[gj + (long long)r * ldy] -= acc;
    }
  }
}

// ---- chained sweeps: one launch per level --------------------------------------
// The block steps of a front's triangular solve form a chain (block i needs
// the solution of blocks 0..i-1 forward, i+1..nb-1 backward).  Instead of one
// launch per block step, one launch per level runs a task per 64-row tile of
// every front, and a task reads the blocks it needs as soon as they exist.
//
// Readiness travels with the data: before a sweep, the forward solution Y
// and the solution x are filled with a signaling-NaN bit pattern (no
// arithmetic result is a signaling NaN), every value a task publishes is one
// relaxed device-scope atomic store, and a reader polls each value it needs
// with relaxed device-scope atomic loads until the pattern is gone.  Each
// value is its own flag, so no fence (and no L2 write-back or invalidation)
// is needed on either side.
//
// Forward progress does not depend on how many workgroups are resident: a
// task takes its index from a ticket counter, tasks are listed so that every
// task waits only for tasks of smaller index, and a task that holds a ticket
// is running, so the smallest unfinished ticket can always proceed.  Every
// wait is still bounded: after SPIN_LIMIT polls the value is taken as it is,
// the error word is marked and the task finishes (the solve reports failure);
// every other wait of the launch gives up within its next 32 polls, when it looks at
// the error word.
// Launches whose tasks wait for nothing run with ticket == nullptr (task =
// blockIdx).


// (Sentinel<T>, publish: the readiness protocol, in kernels.h)

// One wave's 16 rows of a product with a 64 x 16 right-hand-side block in LDS,
// in NSET sets of four right-hand sides (1, 2 or 4), on the MFMAs made of 4 x 4
// blocks: FP64 4 x 4 x 4, four blocks = 16 rows, 16 cycles a set; FP32 4 x 4 x 1,
// sixteen blocks = 16 rows at four k, 8 cycles a set.  Four sets cost what the
// 16 x 16 x 4 MFMA costs (64 and 32 cycles), so a chain step of few right-hand
// sides spends a quarter (half) of that in its two products; four FP64 sets are
// that MFMA, which reads one value of the block where they read four.  The order of
// summation does not depend on NSET, so a column's bits do not depend on how many
// columns there are: FP64 sums along k one after the other (as the 16 x 16 x 4
// MFMA does), FP32 the four residues of k mod 4 apart, which sum() adds in pairs.
// The A operand: lane l holds row l % 16, column l / 16.  Result e of a lane is
// row(lane, e) of the wave's rows, right-hand side col(lane, e).  A row of the block
// has LD values, right-hand side r at pos(r), so that a lane's sets are one load.
// Measured against the 16 x 16 x 4 MFMA: FP64 solve of mesh3d 40^3 with one
// right-hand side 1305 -> 1101 us, of mesh3d 60^3 with 8 3569 -> 3167; FP32, with
// the copies to and from the host, of mesh3d 40^3 with 1, 8 and 16 1206 -> 1082,
// 1806 -> 1625 and 2652 -> 2526.  (With a row's right-hand sides in order, four
// loads a step, 12 and 16 were slower than on the 16 x 16 x 4: 2332 and 2696.)
template <typename T, int NSET> struct RhsTile {
  typedef typename std::conditional<sizeof(T) == 8, double, f4_t>::type set_t;
  typedef T sets_t __attribute__((ext_vector_type(NSET)));
  struct acc_t { set_t v[NSET]; };
  static constexpr int LD = sizeof(T) == 8 ? 18 : 20;  // 16-byte rows, padded against bank conflicts
  static __device__ int pos(int r) { return 4 * (r & 3) + (r >> 2); }
  static __device__ int row(int lane, int) { return 4 * ((lane >> 2) & 3) + (lane >> 4); }
  static __device__ int col(int lane, int e) { return 4 * e + (lane & 3); }
  static __device__ void zero(acc_t& c)
  {
#pragma unroll
    for (int e = 0; e < NSET; e++) c.v[e] = set_t{};
  }
  // c += A(:, 4 st .. 4 st + 3) x the block's rows 4 st ..; b: row 4 st + lane / 16
  static __device__ void step(T a, const T* b, int lane, acc_t& c)
  {
    const sets_t bs = *reinterpret_cast<const sets_t*>(b + 4 * (lane & 3));
#pragma unroll
    for (int e = 0; e < NSET; e++)
      if constexpr (sizeof(T) == 8)
        c.v[e] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, bs[e], c.v[e], 0, 0, 0);
      else
        c.v[e] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, bs[e], c.v[e], 0, 0, 0);
  }
  // out[e] = the lane's element of c + d, set e
  static __device__ void sum(const acc_t& c, const acc_t& d, T* out)
  {
#pragma unroll
    for (int e = 0; e < NSET; e++)
      if constexpr (sizeof(T) == 8) {
        out[e] = c.v[e] + d.v[e];
      } else {
        // register i of a lane: row 4 * (lane / 4 % 4) + i, the k = lane / 16 mod 4;
        // two exchanges add the four k and leave row i with the lanes 16 i ..
        const f4_t v = c.v[e] + d.v[e];
        const float lo = swap_add<32>(v[0], v[2]), hi = swap_add<32>(v[1], v[3]);
        out[e] = swap_add<16>(lo, hi);
      }
  }
  // lanes with bit N of the lane number clear: x + x of the lane N further;
  // the others: y + y of the lane N before
  template <int N> static __device__ float swap_add(float x, float y)
  {
    const auto r = N == 32
        ? __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false)
        : __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
};

template <> struct RhsTile<double, 4> {
  struct acc_t { d4_t v; };
  static constexpr int LD = 17;
  static __device__ int pos(int r) { return r; }
  static __device__ int row(int lane, int e) { return Mfma<double>::drow(lane, e); }
  static __device__ int col(int lane, int) { return lane & 15; }
  static __device__ void zero(acc_t& c) { c.v = d4_t{}; }
  static __device__ void step(double a, const double* b, int lane, acc_t& c)
  {
    c.v = Mfma<double>::step(a, b[lane & 15], c.v);
  }
  static __device__ void sum(const acc_t& c, const acc_t& d, double* out)
  {
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = c.v[e] + d.v[e];
  }
};

// Vl[i*R::LD + R::pos(r)] <- V[col + r*ldv] for i < nv, r < nrhs (0 elsewhere in the
// 64 x 16 block), awaiting each value.  Thread t handles row i = t & 63
// (right-hand sides t/64 + 4k), whose global column `col` the caller has loaded
// ahead.  A poll is one round trip to memory (about 1 us, past the L2s of the
// other XCDs): all of a thread's values are polled together, and the error word
// only every 32nd time, so that a wait ends one round trip after its last value
// is there.  (One value after the other, each with a look at the error word, a
// chain step of the mesh3d 60^3 root took 3.2 us with 8 right-hand sides;
// together 3.0.)
template <typename R, typename T, typename V>
__device__ __forceinline__ void await_rows(T* Vl, const V* Vg, int ldv, int col, int nv, int nrhs,
                                           int* err)
{
  typedef typename Sentinel<V>::U U;
  const int i = threadIdx.x & 63, r0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  U* const a = reinterpret_cast<U*>(const_cast<V*>(Vg + col + (long long)r0 * ldv));
  U bits[4];
  // true once every value of this thread is there
  auto poll = [&]() {
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (r0 + 4 * k < nrhs)
        bits[k] = __hip_atomic_load(a + 4LL * k * ldv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool there = true;
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (r0 + 4 * k < nrhs) there = there && bits[k] != Sentinel<V>::bits;
    return there;
  };
  if (r0 < nrhs && i < nv) {
    int it = 0;
    while (!poll()) {
      if (++it > SPIN_LIMIT) {
        atomicOr(err, 1);
        break;
      }
      if ((it & 31) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
      __builtin_amdgcn_s_sleep(1);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; k++)
    Vl[i * R::LD + R::pos(r0 + 4 * k)] =
        r0 + 4 * k < nrhs && i < nv ? (T)__builtin_bit_cast(V, bits[k]) : (T)0;
}

// Y (n x nrhs, ld n) and x (rows < n of n x nrhs, ld ldx) <- the pattern;
// tickets <- 0.  The first op of every chained solve.
template <typename T>
__global__ void k_sweep_clear(T* __restrict__ Y, double* __restrict__ x, int n, int ldx, int nrhs,
                              int* __restrict__ tickets, int nt)
{
  const long long tot = (long long)n * nrhs;
  const T ys = __builtin_bit_cast(T, Sentinel<T>::bits);
  const double xs = __builtin_bit_cast(double, Sentinel<double>::bits);
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < tot;
       e += (long long)gridDim.x * blockDim.x) {
    const long long r = e / n, i = e - r * n;
    Y[e] = ys;
    x[i + r * ldx] = xs;
  }
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nt; e += gridDim.x * blockDim.x)
    tickets[e] = 0;
}

// Values loaded ahead stay in registers from here on (the compiler may otherwise
// move their loads behind the waits, to their first use).  The chains hold the
// block inverse's operands this way: staged in LDS they were read on the chain's
// critical path.  Resident workgroups did not grow with it: the 33 KiB of LDS (FP64)
// had left three a CU; the registers now leave three for up to eight right-hand sides
// (149 to 156) and two for nine to sixteen (175 and 169), and three instead of four
// to FP32's forward chain of those.  Solves, us, one, eight, nine and sixteen
// right-hand sides: FP64 mesh3d 40^3 1083 -> 992, 1414 -> 1292, 1703 -> 1555, 2036 ->
// 1864; 60^3 with eight, nine and sixteen 3045 -> 2888, 3675 -> 3461, 4600 -> 4329; FP32
// with sixteen 40^3 1670 -> 1500, 60^3 3789 -> 3415.
template <typename T> __device__ __forceinline__ void pin(T (&v)[16])
{
#pragma unroll
  for (int k = 0; k < 16; k++) asm volatile("" : "+v"(v[k]));
}

// Forward sweep of one level (fronts with m > 64).  Task (front, tile t):
// rows [64t, 64t+64) of the front's workspace W_f (m x nrhs, the right-hand
// side plus the children's updates).  Tile t < nb (nb = ceil(s/64)) owns
// diagonal block t: it subtracts L[rows, blk j] y_j for j < t as the y_j
// appear, forms y_t = inv(L_tt) w_t, publishes it in Y (by global column),
// and (last block only) updates the sub-diagonal rows that share its tile.
// Tiles t >= nb hold sub-diagonal rows only: they subtract all nb blocks and
// store the result in W_f for the parent's extend-add.
// The products run on the MFMA (RhsTile): wave w owns rows 16w..16w+15 of the
// tile and all right-hand sides (those beyond nrhs are zero), A = L rows
// (loaded one dependency ahead), B = the awaited y_j block in LDS; the sum
// over dependencies stays in the accumulators.
template <typename T, int NSET>
__global__ __launch_bounds__(256) void k_fwd_chain(const FrontDesc* __restrict__ fr,
                                                   const PanelTask* __restrict__ tasks,
                                                   const int* __restrict__ rows,
                                                   const T* __restrict__ L,
                                                   const T* __restrict__ Inv, T* __restrict__ W,
                                                   T* Y, int ldy, int* ticket, int* err, int nrhs)
{
  typedef RhsTile<T, NSET> R;
  typedef typename R::acc_t acc_t;
  __shared__ alignas(16) T Yl[2][64 * R::LD];
  __shared__ int sh_task;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c16 = lane & 15, kq = lane >> 4;
  if (tid == 0) sh_task = ticket ? atomicAdd(ticket, 1) : (int)blockIdx.x;
  __syncthreads();
  const PanelTask t = tasks[sh_task];
  const FrontDesc d = fr[t.front];
  const int m = d.m, s = d.s, nb = (s + 63) >> 6, tile = t.k0, r0 = tile * 64;
  const int nr = min(64, m - r0);
  const bool isblk = tile < nb;
  const int kb = isblk ? min(64, s - r0) : 0;
  const int ndep = isblk ? tile : nb;
  T* w = W + d.offW * nrhs;
  const T* Lf = L + d.offL;
  const int* rw = rows + d.rows;  // global column of each of the front's first s rows
  const int arow = 16 * wv + c16;
  T w0[NSET];
#pragma unroll
  for (int k = 0; k < NSET; k++) {
    const int i = 16 * wv + R::row(lane, k);
    const int c = R::col(lane, k);
    w0[k] = (c < nrhs && i < nr) ? w[r0 + i + (long long)c * m] : (T)0;
  }
  // global columns loaded ahead: the rows this lane publishes, and the row
  // (tid & 63) of each dependency block this thread awaits
  int pcol[NSET];
#pragma unroll
  for (int k = 0; k < NSET; k++) {
    const int i = 16 * wv + R::row(lane, k);
    pcol[k] = (isblk && i < kb) ? rw[r0 + i] : 0;
  }
  // the inverse's A operands, in registers before the first wait
  T ia[16];
  const T* iv = Inv + d.offI + (isblk ? (long long)tile * 4096 + arow * 64 + kq : 0);
#pragma unroll
  for (int st = 0; st < 16; st++) ia[st] = iv[4 * st];
  acc_t D0, D1;  // even and odd k steps: two independent MFMA chains
  R::zero(D0);
  R::zero(D1);
  T lv[16];
  int dcol = 0;
  auto fetch = [&](int j) {
    const int c0 = j * 64, kbj = min(64, s - c0);
#pragma unroll
    for (int st = 0; st < 16; st++) {
      const int k = 4 * st + kq;
      lv[st] = (arow < nr && k < kbj) ? Lf[r0 + arow + (long long)(c0 + k) * m] : (T)0;
    }
    dcol = (tid & 63) < kbj ? rw[c0 + (tid & 63)] : 0;
  };
  if (ndep > 0) fetch(0);
  pin(ia);
  for (int j = 0; j < ndep; j++) {
    T* yb = Yl[j & 1];
    await_rows<R>(yb, Y, ldy, dcol, min(64, s - 64 * j), nrhs, err);
    __syncthreads();
    T cur[16];
#pragma unroll
    for (int st = 0; st < 16; st++) cur[st] = lv[st];
    if (j + 1 < ndep) fetch(j + 1);
#pragma unroll
    for (int st = 0; st < 16; st += 2) {
      R::step(cur[st], yb + (4 * st + kq) * R::LD, lane, D0);
      R::step(cur[st + 1], yb + (4 * st + 4 + kq) * R::LD, lane, D1);
    }
  }
  T acc[NSET];
  R::sum(D0, D1, acc);
#pragma unroll
  for (int k = 0; k < NSET; k++) acc[k] = w0[k] - acc[k];
  if (!isblk) {
#pragma unroll
    for (int k = 0; k < NSET; k++) {
      const int i = 16 * wv + R::row(lane, k);
      const int c = R::col(lane, k);
      if (c < nrhs && i < nr) w[r0 + i + (long long)c * m] = acc[k];
    }
    return;
  }
  // y = inv(L_tt) acc: A = inverse rows (zero beyond kb), B = acc (64 x 16)
  T* Ac = Yl[ndep & 1];  // not read since the last dependency's barrier
#pragma unroll
  for (int k = 0; k < NSET; k++)
    Ac[(16 * wv + R::row(lane, k)) * R::LD + R::pos(R::col(lane, k))] = acc[k];
  __syncthreads();
  acc_t Ya, Yb;
  R::zero(Ya);
  R::zero(Yb);
#pragma unroll
  for (int st = 0; st < 16; st += 2) {
    R::step(ia[st], Ac + (4 * st + kq) * R::LD, lane, Ya);
    R::step(ia[st + 1], Ac + (4 * st + 4 + kq) * R::LD, lane, Yb);
  }
  T Yd[NSET];
  R::sum(Ya, Yb, Yd);
#pragma unroll
  for (int k = 0; k < NSET; k++) {
    const int i = 16 * wv + R::row(lane, k);
    const int c = R::col(lane, k);
    if (i < kb && c < nrhs) publish(Y + pcol[k] + (long long)c * ldy, Yd[k]);
  }
  if (nr > kb) {  // sub-diagonal rows in the last block's tile: acc -= L[rows, blk t] y_t
    T* Yv = Yl[(ndep + 1) & 1];  // free since the barrier above
#pragma unroll
    for (int k = 0; k < NSET; k++)
      Yv[(16 * wv + R::row(lane, k)) * R::LD + R::pos(R::col(lane, k))] = Yd[k];
    __syncthreads();
    acc_t D2, zero;
    R::zero(D2);
    R::zero(zero);
#pragma unroll
    for (int st = 0; st < 16; st++) {
      const int k = 4 * st + kq;
      const T a = (arow < nr && k < kb) ? Lf[r0 + arow + (long long)(r0 + k) * m] : (T)0;
      R::step(a, Yv + k * R::LD, lane, D2);
    }
    T d2[NSET];
    R::sum(D2, zero, d2);
#pragma unroll
    for (int k = 0; k < NSET; k++) {
      const int i = 16 * wv + R::row(lane, k);
      const int c = R::col(lane, k);
      if (i >= kb && i < nr && c < nrhs) w[r0 + i + (long long)c * m] = acc[k] - d2[k];
    }
  }
}

// Backward sweep of one level (fronts with m > 64).  Task (front, block b,
// kb = first Part slot, nr = slot count): the update rows' part L21^T x2 of
// the block's columns comes from k_bwd_upd as nr partial blocks, summed in
// slot order; z = y_b - that - sum_{j > b} L[blk j, blk b]^T x_j with the x_j
// of the same front awaited as they are published; then x_b = inv(L_bb)^T z
// is published in x.  MFMA products as in k_fwd_chain with wave w owning the
// block's columns 16w..16w+15: A = L^T (read down the block's columns, one
// dependency ahead), B = the awaited x_j block in LDS.
template <typename T, int NSET>
__global__ __launch_bounds__(256) void k_bwd_chain(const FrontDesc* __restrict__ fr,
                                                   const PanelTask* __restrict__ tasks,
                                                   const int* __restrict__ rows,
                                                   const T* __restrict__ L,
                                                   const T* __restrict__ Inv,
                                                   const T* __restrict__ Y, int ldy,
                                                   const T* __restrict__ Part, double* x,
                                                   int ldx, int* ticket, int* err, int nrhs)
{
  typedef RhsTile<T, NSET> R;
  typedef typename R::acc_t acc_t;
  __shared__ alignas(16) T Xl[2][64 * R::LD];
  __shared__ int sh_task;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c16 = lane & 15, kq = lane >> 4;
  if (tid == 0) sh_task = ticket ? atomicAdd(ticket, 1) : (int)blockIdx.x;
  __syncthreads();
  const PanelTask t = tasks[sh_task];
  const FrontDesc d = fr[t.front];
  const int m = d.m, s = d.s, nb = (s + 63) >> 6, blk = t.k0, c0 = blk * 64;
  const int kb = min(64, s - c0);
  const T* Lf = L + d.offL;
  const int* rw = rows + d.rows;
  const int acol = 16 * wv + c16;  // A-operand row = block column of this lane
  T y0[NSET];
#pragma unroll
  for (int k = 0; k < NSET; k++) {
    const int q = 16 * wv + R::row(lane, k), c = R::col(lane, k);
    // slot stride 64 x nrhs: only the columns c < nrhs exist
    const long long pst = 64LL * nrhs;
    const T* ps = Part + (long long)t.kb * pst + q + c * 64;
    T s0 = (T)0, s1 = (T)0, s2 = (T)0, s3 = (T)0;  // slots in four interleaved sums
    if (c < nrhs) {
      int u = 0;
      for (; u + 3 < t.nr; u += 4) {
        s0 += ps[(long long)u * pst];
        s1 += ps[(long long)(u + 1) * pst];
        s2 += ps[(long long)(u + 2) * pst];
        s3 += ps[(long long)(u + 3) * pst];
      }
      for (; u < t.nr; u++) s0 += ps[(long long)u * pst];
    }
    const T sum = (s0 + s1) + (s2 + s3);
    y0[k] = (c < nrhs && q < kb) ? Y[rw[c0 + q] + (long long)c * ldy] - sum : (T)0;
  }
  // the inverse's A operands, in registers before the first wait
  T ia[16];
  const T* iv = Inv + d.offI + (long long)blk * 4096 + acol + kq * 64;
#pragma unroll
  for (int st = 0; st < 16; st++) ia[st] = iv[256 * st];
  const int ndep = nb - 1 - blk;  // blocks nb-1 down to blk+1
  int pcol[NSET];  // the columns this lane publishes, loaded ahead
#pragma unroll
  for (int k = 0; k < NSET; k++) {
    const int q = 16 * wv + R::row(lane, k);
    pcol[k] = q < kb ? rw[c0 + q] : 0;
  }
  acc_t D0, D1;  // even and odd k steps: two independent MFMA chains
  R::zero(D0);
  R::zero(D1);
  T lv[16];
  int dcol = 0;
  auto fetch = [&](int u) {
    const int rr0 = 64 * (nb - 1 - u), nrr = min(64, s - rr0);
#pragma unroll
    for (int st = 0; st < 16; st++) {
      const int i = 4 * st + kq;
      lv[st] = (acol < kb && i < nrr) ? Lf[rr0 + i + (long long)(c0 + acol) * m] : (T)0;
    }
    dcol = (tid & 63) < nrr ? rw[rr0 + (tid & 63)] : 0;
  };
  if (ndep > 0) fetch(0);
  pin(ia);
  for (int u = 0; u < ndep; u++) {
    const int rr0 = 64 * (nb - 1 - u);
    T* xb = Xl[u & 1];
    await_rows<R>(xb, x, ldx, dcol, min(64, s - rr0), nrhs, err);
    __syncthreads();
    T cur[16];
#pragma unroll
    for (int st = 0; st < 16; st++) cur[st] = lv[st];
    if (u + 1 < ndep) fetch(u + 1);
#pragma unroll
    for (int st = 0; st < 16; st += 2) {
      R::step(cur[st], xb + (4 * st + kq) * R::LD, lane, D0);
      R::step(cur[st + 1], xb + (4 * st + 4 + kq) * R::LD, lane, D1);
    }
  }
  T* Z = Xl[ndep & 1];  // not read since the last dependency's barrier
  T dk[NSET];
  R::sum(D0, D1, dk);
#pragma unroll
  for (int k = 0; k < NSET; k++)
    Z[(16 * wv + R::row(lane, k)) * R::LD + R::pos(R::col(lane, k))] = y0[k] - dk[k];
  __syncthreads();
  // x = inv(L_bb)^T z: A[q][p] = inv(p, q)
  acc_t Xa, Xb;
  R::zero(Xa);
  R::zero(Xb);
#pragma unroll
  for (int st = 0; st < 16; st += 2) {
    R::step(ia[st], Z + (4 * st + kq) * R::LD, lane, Xa);
    R::step(ia[st + 1], Z + (4 * st + 4 + kq) * R::LD, lane, Xb);
  }
  T xk[NSET];
  R::sum(Xa, Xb, xk);
#pragma unroll
  for (int k = 0; k < NSET; k++) {
    const int q = 16 * wv + R::row(lane, k);
    const int c = R::col(lane, k);
    if (q < kb && c < nrhs) publish(x + pcol[k] + (long long)c * ldx, (double)xk[k]);
  }
}

// Backward sweep, update rows of the fronts with m > 64, split over row
// chunks (before the chained launch): Part[slot] (64 columns x 16 rhs) =
// L[rows i0 .. i0+cnt-1, columns c0 .. c0+nc-1]^T x(rows), task (front, k0 =
// i0, kb = cnt <= BU_ROWS, r0 = c0, nr = nc); k_bwd_cols_reduce subtracts the
// slots from Y in order.  x of the update rows is final (the ancestors'
// levels wrote it) and is read through the front's row list.  MFMA as in
// k_bwd_chain: wave w owns columns 16w..16w+15, A = L^T, B = x rows in LDS.
// (One chain of 32 MFMAs: at 16 instead of 64 cycles each, solve of mesh3d 40^3
// with one right-hand side 956 -> 945 us.)
#define BU_ROWS 128
template <typename T, int NSET>
__global__ __launch_bounds__(256) void k_bwd_upd(const FrontDesc* __restrict__ fr,
                                                 const PanelTask* __restrict__ tasks,
                                                 const int* __restrict__ rows,
                                                 const T* __restrict__ L,
                                                 const double* __restrict__ x, int ldx,
                                                 T* __restrict__ Part, int nrhs)
{
  typedef RhsTile<T, NSET> R;
  __shared__ alignas(16) T Xl[BU_ROWS * R::LD];
  const PanelTask t = tasks[blockIdx.x];
  const FrontDesc d = fr[t.front];
  const int m = d.m, i0 = t.k0, cnt = t.kb, c0 = t.r0, nc = t.nr;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c16 = lane & 15, kq = lane >> 4;
  const int* rw = rows + d.rows;
  const int acol = 16 * wv + c16;
  const T* Lc = L + d.offL + i0 + (long long)(c0 + acol) * m;  // column c0+acol from row i0
  T a[BU_ROWS / 4];
#pragma unroll
  for (int st = 0; st < BU_ROWS / 4; st++) {
    const int i = 4 * st + kq;
    a[st] = (acol < nc && i < cnt) ? Lc[i] : (T)0;
  }
#pragma unroll
  for (int k = 0; k < BU_ROWS * 16 / 256; k++) {
    const int e = tid + 256 * k, i = e & (BU_ROWS - 1), r = e / BU_ROWS;
    Xl[i * R::LD + R::pos(r)] = (i < cnt && r < nrhs) ? (T)x[rw[i0 + i] + (long long)r * ldx] : (T)0;
  }
  __syncthreads();
  typename R::acc_t D0, zero;
  R::zero(D0);
  R::zero(zero);
  const int nst = (cnt + 3) >> 2;
#pragma unroll
  for (int st = 0; st < BU_ROWS / 4; st++)
    if (st < nst) R::step(a[st], Xl + (4 * st + kq) * R::LD, lane, D0);
  T D[NSET];
  R::sum(D0, zero, D);
  // slot stride 64 x nrhs: the columns c >= nrhs are not stored
  T* part = Part + (long long)blockIdx.x * (64LL * nrhs);
#pragma unroll
  for (int k = 0; k < NSET; k++) {
    const int c = R::col(lane, k);
    if (c < nrhs) part[16 * wv + R::row(lane, k) + c * 64] = D[k];
  }
}

// Fronts with m <= 64, one wave each (four per workgroup), no waits: the
// whole front's right-hand side fits one wave's rows.
//   forward:  y = inv(L11) w[0:s] into Y; w[s:m] -= L21 y for the parent.
//   backward: z = y - L21^T x(update rows); x = inv(L11)^T z.
// Per-wave LDS holds the m x nrhs values that every lane needs.
__device__ __forceinline__ void wave_sync_lds()
{
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
}

// A lane's column of a small front or of its inverse: the values at p = lo .. hi-1,
// `stride` apart, N in flight and the next N loading behind their use (8, of 16
// right-hand sides, whose sums fill the registers, 4).
// (One at a time, a front waited for s + m round trips to memory, each for as
// little as one fused multiply-add a lane: the backward launch of 42 thousand fronts
// of an 80 x 72 x 64 grid, four right-hand sides, took 91 us, this way 60; of 54
// thousand fronts of 512 planes, one right-hand side, 124 and 87.  The largest
// forward launch, the 512 planes' 210 thousand leaves, is bound by its loads and lost,
// 284 and 305 us, for the masked entries that are now read too; the backward launch of
// the same leaves went from 348 to 299, the whole solve from 3.07 to 2.85 ms.)
template <typename T, int N> struct SmallRows {
  const T* a;
  int stride, lo, hi;
  __device__ SmallRows(const T* a_, int stride_, int lo_, int hi_) : a(a_), stride(stride_), lo(lo_), hi(hi_) {}
  // v <- the values at p .. p + N - 1 (past the end the last one: read, dropped)
  __device__ __forceinline__ void fetch(T (&v)[N], int p) const
  {
#pragma unroll
    for (int q = 0; q < N; q++) v[q] = a[(long long)min(p + q, hi - 1) * stride];
  }
  // use(p, value) in order; v: the first N, fetched ahead
  template <typename F> __device__ __forceinline__ void each(T (&v)[N], F use) const
  {
    for (int p = lo; p < hi; p += N) {
      T c[N];
#pragma unroll
      for (int q = 0; q < N; q++) c[q] = v[q];
      if (p + N < hi) fetch(v, p + N);
#pragma unroll
      for (int q = 0; q < N; q++)
        if (p + q < hi) use(p + q, c[q]);
    }
  }
};

// NR: right-hand sides per pass rounded up to 1, 4, 8 or 16 (compile-time, so
// the loops over them carry no guards); columns beyond nrhs hold zeros.
template <typename T, int NR>
__global__ __launch_bounds__(256) void k_fwd_small(const FrontDesc* __restrict__ fr,
                                                   const PanelTask* __restrict__ tasks, int count,
                                                   const int* __restrict__ rows,
                                                   const T* __restrict__ L,
                                                   const T* __restrict__ Inv, T* __restrict__ W,
                                                   T* __restrict__ Y, int ldy, int nrhs)
{
  constexpr int NB = NR <= 8 ? 8 : 4;
  typedef SmallRows<T, NB> Rows;
  __shared__ T Ws[4][64 * NR];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ti = blockIdx.x * 4 + wv;
  if (ti >= count) return;
  const FrontDesc d = fr[tasks[ti].front];
  const int m = d.m, s = d.s;
  const Rows iv(Inv + d.offI + min(lane, s - 1) * 64, 1, 0, s);
  const Rows lf(L + d.offL + min(lane, m - 1), m, 0, s);
  T ia[NB], la[NB];
  iv.fetch(ia, 0);
  lf.fetch(la, 0);
  T* w = W + d.offW * nrhs;
  T* ws = Ws[wv];
  const int* rw = rows + d.rows;
  T v[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) {
    v[r] = (r < nrhs && lane < m) ? w[lane + r * m] : (T)0;
    ws[lane + r * 64] = v[r];
  }
  wave_sync_lds();
  T y[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) y[r] = (T)0;
  iv.each(ia, [&](int p, T a) {
    a = (lane < s && p <= lane) ? a : (T)0;
#pragma unroll
    for (int r = 0; r < NR; r++) y[r] += a * ws[p + r * 64];
  });
  wave_sync_lds();
  if (lane < s) {
#pragma unroll
    for (int r = 0; r < NR; r++) {
      ws[lane + r * 64] = y[r];
      if (r < nrhs) Y[rw[lane] + (long long)r * ldy] = y[r];
    }
  }
  wave_sync_lds();
  if (m == s) return;
  lf.each(la, [&](int p, T a) {
    a = (lane >= s && lane < m) ? a : (T)0;
#pragma unroll
    for (int r = 0; r < NR; r++) v[r] -= a * ws[p + r * 64];
  });
  if (lane >= s && lane < m) {
#pragma unroll
    for (int r = 0; r < NR; r++)
      if (r < nrhs) w[lane + r * m] = v[r];
  }
}

template <typename T, int NR>
__global__ __launch_bounds__(256) void k_bwd_small(const FrontDesc* __restrict__ fr,
                                                   const PanelTask* __restrict__ tasks, int count,
                                                   const int* __restrict__ rows,
                                                   const T* __restrict__ L,
                                                   const T* __restrict__ Inv,
                                                   const T* __restrict__ Y, int ldy,
                                                   double* __restrict__ x, int ldx, int nrhs)
{
  constexpr int NB = NR <= 8 ? 8 : 4;
  typedef SmallRows<T, NB> Rows;
  __shared__ T Ws[4][64 * NR];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ti = blockIdx.x * 4 + wv;
  if (ti >= count) return;
  const FrontDesc d = fr[tasks[ti].front];
  const int m = d.m, s = d.s;
  // column `lane` of the panel's update rows and of the inverse
  const Rows lf(L + d.offL + (long long)min(lane, s - 1) * m, 1, s, m);
  const Rows iv(Inv + d.offI + min(lane, s - 1), 64, 0, s);
  T la[NB], ia[NB];
  lf.fetch(la, s);
  iv.fetch(ia, 0);
  const int* rw = rows + d.rows;
  T* ws = Ws[wv];
  T z[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) {
    z[r] = (r < nrhs && lane < s) ? Y[rw[lane] + (long long)r * ldy] : (T)0;
    ws[lane + r * 64] =
        (r < nrhs && lane >= s && lane < m) ? (T)x[rw[lane] + (long long)r * ldx] : (T)0;
  }
  wave_sync_lds();
  lf.each(la, [&](int i, T a) {
    a = lane < s ? a : (T)0;
#pragma unroll
    for (int r = 0; r < NR; r++) z[r] -= a * ws[i + r * 64];
  });
  if (lane < s) {
#pragma unroll
    for (int r = 0; r < NR; r++) ws[lane + r * 64] = z[r];
  }
  wave_sync_lds();
  T xv[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) xv[r] = (T)0;
  iv.each(ia, [&](int p, T a) {
    a = (lane < s && p >= lane) ? a : (T)0;
#pragma unroll
    for (int r = 0; r < NR; r++) xv[r] += a * ws[p + r * 64];
  });
  if (lane < s) {
#pragma unroll
    for (int r = 0; r < NR; r++)
      if (r < nrhs) x[rw[lane] + (long long)r * ldx] = (double)xv[r];
  }
}

#define SMALL_INST(T, NR)                                                                       \
  template __global__ void k_fwd_small<T, NR>(const FrontDesc*, const PanelTask*, int, const int*, \
                                              const T*, const T*, T*, T*, int, int);            \
  template __global__ void k_bwd_small<T, NR>(const FrontDesc*, const PanelTask*, int, const int*, \
                                              const T*, const T*, const T*, int, double*, int, int);
#define CHAIN_INST(T, NSET)                                                                     \
  template __global__ void k_fwd_chain<T, NSET>(const FrontDesc*, const PanelTask*, const int*, \
                                                const T*, const T*, T*, T*, int, int*, int*, int); \
  template __global__ void k_bwd_chain<T, NSET>(const FrontDesc*, const PanelTask*, const int*, \
                                                const T*, const T*, const T*, int, const T*,    \
                                                double*, int, int*, int*, int);                          \
  template __global__ void k_bwd_upd<T, NSET>(const FrontDesc*, const PanelTask*, const int*,   \
                                              const T*, const double*, int, T*, int);
#define TAMD_SINST(T)                                                                           \
  template __global__ void k_solve_init<T>(const FrontDesc*, const PanelTask*, int, const int*,  \
                                           const double*, int, T*, int);                        \
  template __global__ void k_fwd_step<T>(const FrontDesc*, const PanelTask*, const int*,         \
                                         const T*, const T*, T*, T*, int, int);                 \
  template __global__ void k_fwd_rect<T>(const FrontDesc*, const PanelTask*, const int*,         \
                                         const T*, const T*, int, T*, int);                     \
  template __global__ void k_fwd_rect_reduce<T>(const FrontDesc*, const PanelTask*, const T*, T*, int); \
  template __global__ void k_bwd_cols_reduce<T>(const FrontDesc*, const PanelTask*, const int*,  \
                                                const T*, T*, int, int);                        \
  template __global__ void k_solve_ext<T>(const FrontDesc*, const PanelTask*, const int*, T*, int); \
  template __global__ void k_solve_ext_seq<T>(const FrontDesc*, const PanelTask*, const PanelTask*, \
                                              const int*, T*, int);                             \
  template __global__ void k_solve_ext_wave<T>(const FrontDesc*, const PanelTask*, int, int,     \
                                               const PanelTask*, const int*, T*, int);          \
  template __global__ void k_bwd_gather<T>(const FrontDesc*, const PanelTask*, const int*,        \
                                           const double*, int, T*, int);                        \
  template __global__ void k_bwd_cols<T>(const FrontDesc*, const PanelTask*, const T*, const T*, \
                                         T*, int);                                              \
  template __global__ void k_bwd_step<T>(const FrontDesc*, const PanelTask*, const int*,         \
                                         const T*, const T*, T*, int, double*, int, int);       \
  template __global__ void k_sweep_clear<T>(T*, double*, int, int, int, int*, int);           \
  CHAIN_INST(T, 1) CHAIN_INST(T, 2) CHAIN_INST(T, 4)                                            \
  SMALL_INST(T, 1) SMALL_INST(T, 4) SMALL_INST(T, 8) SMALL_INST(T, 16)
TAMD_SINST(double)
TAMD_SINST(float)

}  // namespace tamd
