// Blocked Cholesky on one MI355X: diagonal-block factor, panel TRSM and the
// MFMA trailing update, scheduled with one panel of look-ahead on two streams.
//
// Reference algorithm: FLA_Chol_l_blk_var3
//   (src/lapack/dec/chol/l/flamec/FLA_Chol_l_blk_var3.c:13-66):
//     A11 := chol(A11); A21 := A21 * inv(tril(A11))'; A22 := A22 - A21*A21'
// and its leaf FLA_Chol_l_opd_var2 (src/lapack/dec/chol/l/flamec/FLA_Chol_l_opt_var2.c:136-193),
// whose failure rule (pivot <= 0 or NaN, bl1_dsqrte in
// src/base/flamec/include/blis_macro_defs.h:134-136) and 0-based failing
// column index (FLA_Chol_l_blk_var3.c:42-43) are kept.  The upper case
// (FLA_Chol_u_blk_var3.c:38-54) is the lower algorithm on A' (the triangles
// are exchanged in place before and after).
#include "fla_hip_frag.h"
#include "fla_hip_internal.h"

#include <utility>

namespace {

using namespace fla_frag;

constexpr int PB = FB;  // panel sub-block width (diagonal block order)


// Single-workgroup Cholesky of the nb x nb lower block at A (nb <= 128, padded
// with the identity) over 16-column blocks with the whole block in registers:
// wave w owns block row w (blocks (w, 0..w) in fragment order).  Step b, after
// one barrier: every wave below applies the previous step's update to its
// block (w, b), solves it against the factored diagonal block b, applies it
// to its own diagonal block, and publishes it through LDS; wave b + 1 then
// factors its diagonal block (factor16) while the others apply the previous
// step's update to their remaining blocks.  An update sums its sixteen terms
// from zero: subtracted from the block one by one they left the factor of
// B B'/n + I, n = 128, 2.1e-16 off (1.0e-16 from zero in a model of both).
// Bound: the serial chain of 128 pivots (broadcast, root, reciprocal, scale,
// update: about 200 cycles each) plus a block substitution and its updates
// (about 3000 cycles) per 16 columns.  128 columns take 27 us alone, 73
// with the block in LDS, lane reads for the multipliers and three barriers
// per 32 columns.  Its registers are a whole CU's: beside an update without a
// CU mask it waits for a CU to drain (n = 32768: 399 us on average, 15 ms at
// most, hidden while the update is the longer chain).
// W receives the blocks of L for the panel solve (see frag_q0).  A failed
// block leaves its columns from the failing one on unwritten.
__global__ __launch_bounds__(512) void potrf_blk_kernel(int nb, double* __restrict__ A, long lda,
                                                        int col_offset, int* __restrict__ info,
                                                        d2* __restrict__ W) {
  if (*info >= 0) return;
  __shared__ d2 Xf[2][NT16][2][64];  // the solved blocks (negated) of a block column, by parity
  __shared__ __attribute__((aligned(16))) double Z[2][17 * ZLD];
  // the failing column found in block b's factor, or -1, by b's parity: read
  // only after the barrier that follows the write
  __shared__ int fail[2];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 15, lk = lane >> 4;
  // c[i]: block (w, b + i) at step b (i < w - b); dg: block (w, w)
  d4 c[NT16 - 1], dg;
  const int row = 16 * w + li;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int col = 16 * w + lk + 4 * r;
    const int i = row > col ? row : col, j = row > col ? col : row;  // the lower triangle's copy
    dg[r] = i < nb ? A[(long)i + (long)j * lda] : (row == col ? 1.0 : 0.0);
  }
#pragma unroll
  for (int k = 0; k < NT16 - 1; ++k) {
    if (k >= w) break;  // uniform
#pragma unroll
    for (int r = 0; r < 4; ++r)
      c[k][r] = row < nb ? A[(long)row + (long)(16 * k + lk + 4 * r) * lda] : 0.0;
  }
  if (w == 0) {
    const int f = factor16(dg, Z[0], lane);
    if (lane == 0) fail[0] = f;
  }
  int flim = -1;
  d4 xr = {0.0, 0.0, 0.0, 0.0};  // this row's block of the previous block column
  for (int b = 0; b < NT16; ++b) {
    lds_barrier();
    const int par = b & 1;
    const double* const z = Z[par];
    flim = fail[par];
    if (w > b && flim < 0) {
      __builtin_amdgcn_s_setprio(2);
      d4 l, cf[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int cc = lk + 4 * s;
        l[s] = -z[li * ZLD + cc];  // above the diagonal never used
        cf[s][0] = z[16 * ZLD + cc];
#pragma unroll
        for (int q = 0; q < 3; ++q) cf[s][1 + q] = -z[cc * ZLD + 4 * s + q];
      }
      d4 cur = c[0];
      if (b > 0) cur += mfma_block(Xf[par ^ 1][b][0][lane], Xf[par ^ 1][b][1][lane], xr, d4{});
      const d4 xn = solve_block(l, cf, cur, lk);
      const d2 n0 = d2{-xn[0], -xn[1]}, n1 = d2{-xn[2], -xn[3]};
      Xf[par][w][0][lane] = n0;
      Xf[par][w][1][lane] = n1;
      dg += mfma_block(n0, n1, xn, d4{});
      if (w == b + 1) {
        __builtin_amdgcn_s_setprio(3);
        const int f = factor16(dg, Z[par ^ 1], lane);
        if (lane == 0) fail[par ^ 1] = f < 0 ? -1 : 16 * w + f;
      }
      __builtin_amdgcn_s_setprio(0);
      // the previous step's update of the blocks right of b, moved one place
#pragma unroll
      for (int i = 1; i < NT16 - 1; ++i) {
        if (i >= w - b) break;  // uniform
        c[i - 1] = c[i];
        if (b > 0)
          c[i - 1] += mfma_block(Xf[par ^ 1][b + i][0][lane], Xf[par ^ 1][b + i][1][lane], xr, d4{});
      }
      xr = xn;
      d2* const Wq = W + (frag_q0(w) + b) * 128;
      Wq[lane] = n0;
      Wq[64 + lane] = n1;
      if (row < nb) {
#pragma unroll
        for (int r = 0; r < 4; ++r) A[(long)row + (long)(16 * b + lk + 4 * r) * lda] = xn[r];
      }
    } else if (w == b) {
      // the diagonal block: L to A (up to a failing column), -L and cf to W
      const int jend = flim < 0 ? 16 : flim - 16 * b;
      d2* const Wq = W + (frag_q0(b) + b) * 128;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int k0 = lk + 8 * p, k1 = k0 + 4;
        const double v0 = z[li * ZLD + k0], v1 = z[li * ZLD + k1];
        if (k0 <= li && row < nb && k0 < jend) A[(long)row + (long)(16 * b + k0) * lda] = v0;
        if (k1 <= li && row < nb && k1 < jend) A[(long)row + (long)(16 * b + k1) * lda] = v1;
        Wq[64 * p + lane] = d2{k0 <= li ? -v0 : 0.0, k1 <= li ? -v1 : 0.0};
      }
      const int cc = lk + (lane & 12), q = (lane & 3) - 1;  // cf[lk][(lane / 4) % 4][lane % 4]
      const double v = q < 0 ? z[16 * ZLD + cc] : -z[cc * ZLD + (lane & 12) + (q < 0 ? 0 : q)];
      reinterpret_cast<double*>(Wq + 128)[lane] = lk > q ? v : 0.0;
    }
    if (flim >= 0) break;
  }
  if (t == 0 && flim >= 0) *info = col_offset + flim;
}

// Exchanges A(i,j) and A(j,i) for all i > j, 32x32 tile pairs through LDS.
__global__ __launch_bounds__(256) void transpose_swap_kernel(int n, double* __restrict__ A, long lda) {
  __shared__ double P[32][33];
  __shared__ double Q[32][33];
  // Lower tile (I, J), I >= J, enumerated row by row.
  const int b = blockIdx.x;
  int I = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
  while ((long)I * (I + 1) / 2 > b) --I;
  while ((long)(I + 1) * (I + 2) / 2 <= b) ++I;
  const int J = b - I * (I + 1) / 2;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // ty 0..7
  const int ri = I * 32, cj = J * 32;
  for (int y = ty; y < 32; y += 8) {
    const int i = ri + tx, j = cj + y;  // lower tile element (i, j)
    P[y][tx] = (i < n && j < n) ? A[(long)i + (long)j * lda] : 0.0;
    const int i2 = cj + tx, j2 = ri + y;  // upper tile element (i2, j2)
    Q[y][tx] = (i2 < n && j2 < n) ? A[(long)i2 + (long)j2 * lda] : 0.0;
  }
  __syncthreads();
  for (int y = ty; y < 32; y += 8) {
    // new lower (ri+tx, cj+y) := old upper (cj+y, ri+tx) = Q[tx][y]
    const int i = ri + tx, j = cj + y;
    if (i < n && j < n && i > j) A[(long)i + (long)j * lda] = Q[tx][y];
    const int i2 = cj + tx, j2 = ri + y;
    if (i2 < n && j2 < n && i2 < j2) A[(long)i2 + (long)j2 * lda] = P[tx][y];
  }
}

__global__ void set_int_kernel(int* p, int v) { *p = v; }

}  // namespace

// A21 := A21 inv(L11)' for an m x 128 strip, L11 given by the blocks that
// potrf_blk_kernel left in W.  Each wave owns 16 rows, all 128 columns in
// registers in fragment order; per 16-column block the contributions of the
// solved blocks, then the diagonal block.  No LDS, so the workgroups fit
// beside the update kernel's.  (32 rows per wave, with half the reads of L, spilled registers.)
// Bound: one wave's chain (112 matrix steps and eight block substitutions)
// while the rows fit the chip once.  n = 5003: about 12 us a launch on average against 87 for one
// thread per row.
__global__ __launch_bounds__(256, 2) void trsm_rlt_kernel(int m, const d2* __restrict__ W,
                                                          double* __restrict__ X, long ldx,
                                                          const int* __restrict__ abort) {
  if (abort && *abort >= 0) return;
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int row0 = ((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6)) * 16;
  if (row0 >= m) return;
  const bool in = row0 + li < m;
  double* const xp = X + (in ? row0 + li : m - 1) + (long)lk * ldx;
  d4 c[NT16];
#pragma unroll
  for (int k = 0; k < NT16; ++k)
#pragma unroll
    for (int r = 0; r < 4; ++r) c[k][r] = xp[(long)(16 * k + 4 * r) * ldx];
  solve_rows<ByReciprocal>(W, c, lane, [&](int jb) {
    if (in) {
#pragma unroll
      for (int r = 0; r < 4; ++r) xp[(long)(16 * jb + 4 * r) * ldx] = c[jb][r];
    }
  });
}

// Single-workgroup Cholesky of an nb x nb lower diagonal block (nb <= 128);
// the blocks of L for launch_trsm_rlt go to W.
static int launch_potrf_diag(hipStream_t s, int nb, double* A, long lda, int col_offset, int* info,
                             double* W) {
  if (nb <= 0) return FLA_HIP_OK;
  if (nb > PB) return FLA_HIP_EARG;
  hipLaunchKernelGGL(potrf_blk_kernel, dim3(1), dim3(512), 0, s, nb, A, lda, col_offset, info,
                     reinterpret_cast<d2*>(W));
  FLA_HIP_CHECK(hipGetLastError());
  return FLA_HIP_OK;
}

static int launch_trsm_rlt(hipStream_t s, int m, const double* W, double* A21, long lda,
                           const int* abort_flag) {
  if (m <= 0) return FLA_HIP_OK;
  hipLaunchKernelGGL(trsm_rlt_kernel, dim3((unsigned)((m + 63) / 64)), dim3(256), 0, s, m,
                     reinterpret_cast<const d2*>(W), A21, lda, abort_flag);
  FLA_HIP_CHECK(hipGetLastError());
  return FLA_HIP_OK;
}

int launch_transpose_swap(hipStream_t s, int n, double* A, long lda) {
  if (n <= 1) return FLA_HIP_OK;
  const int T = (n + 31) / 32;
  const long nblk = (long)T * (T + 1) / 2;
  hipLaunchKernelGGL(transpose_swap_kernel, dim3((unsigned)nblk), dim3(256), 0, s, n, A, lda);
  FLA_HIP_CHECK(hipGetLastError());
  return FLA_HIP_OK;
}

// Factors columns [k, k+kb) of the lower matrix (rows k..n-1): per 128-column
// sub-block, the diagonal factor, the panel solve of everything below it
// (only a matrix's last sub-block is narrower than 128, and nothing is below
// it), and the update of the panel's remaining columns.  All on stream s.
int chol_panel_f64(hipStream_t s, int n, double* A, long lda, int k, int kb, int* info) {
  double* W = fla_ctx().dlinv;
  for (int kk = k; kk < k + kb; kk += PB) {
    const int ib = (k + kb - kk) < PB ? (k + kb - kk) : PB;
    double* Akk = A + (long)kk + (long)kk * lda;
    FLA_TRY(launch_potrf_diag(s, ib, Akk, lda, kk, info, W));
    const int mb = n - kk - ib;
    if (mb <= 0) continue;
    if (ib != PB) return FLA_HIP_EARG;
    FLA_TRY(launch_trsm_rlt(s, mb, W, Akk + ib, lda, info));
    const int w = k + kb - kk - ib;  // remaining columns of this panel
    if (w > 0) {
      const double* P = Akk + ib;  // mb x ib
      FLA_TRY(launch_dgemm_mfma(s, false, true, 1, mb, w, ib, -1.0, P, lda, P, lda, 1.0,
                                A + (long)(kk + ib) + (long)(kk + ib) * lda, lda, info));
    }
  }
  return FLA_HIP_OK;
}

// Trailing order from which the updates move to the stream that leaves CUs to
// the panels.  A CU mask costs the update an eighth of its rate even if it
// takes 8 of 256 CUs (the XCDs' shader engines get equal shares of the
// workgroups and the one with fewer CUs is last: 58.5 against 66.9 TFLOP/s),
// but a panel kernel then never waits for CUs.  FLA_Chol with 0, 6000, 9000,
// 13000, 20000: n = 32768 199.1, 199.5, 199.0, 198.4, 199.1 ms; n = 16384
// 32.7, 32.3, 32.0, 31.6, 32.0 ms; n = 8192 7.07, 6.73, 6.63, 6.62, 6.62 ms
// (all updates on a stream that leaves 8 CUs: 212.0, 32.5 and 6.9 ms).
constexpr int kMaskedOrder = 13000;

// Lower blocked Cholesky with look-ahead: the panel of step k+1 runs on
// s_panel while the bulk of step k's trailing update runs on s_update.
static int chol_lower(int n, double* A, long lda, int* dinfo) {
  FlaHipCtx& c = fla_ctx();
  const int nb = fla_chol_nb(n);
  hipStream_t sp = c.s_panel, su = c.s_update;
  int evi = 0;
  auto next_event = [&]() { hipEvent_t e = c.ev[evi]; evi = (evi + 1) % FlaHipCtx::kEvents; return e; };

  // Both streams start after whatever the caller queued on s_update.
  hipEvent_t start = next_event();
  FLA_HIP_CHECK(hipEventRecord(start, su));
  FLA_HIP_CHECK(hipStreamWaitEvent(sp, start, 0));

  // Panel 0.
  int kb0 = n < nb ? n : nb;
  FLA_TRY(chol_panel_f64(sp, n, A, lda, 0, kb0, dinfo));
  for (int k = 0; k < n;) {
    const int kb = (n - k) < nb ? (n - k) : nb;
    hipEvent_t panel_done = next_event();
    FLA_HIP_CHECK(hipEventRecord(panel_done, sp));
    FLA_HIP_CHECK(hipStreamWaitEvent(su, panel_done, 0));
    const int k2 = k + kb;      // first column of the trailing matrix
    const int m2 = n - k2;      // its order
    if (m2 <= 0) break;
    if (su == c.s_update && m2 <= kMaskedOrder && fla_chol_tail_on_lp()) {
      // from here on the panel chain outlasts the update: it gets CUs of its own
      hipEvent_t sw = next_event();
      FLA_HIP_CHECK(hipEventRecord(sw, su));
      su = c.s_update_lp;
      FLA_HIP_CHECK(hipStreamWaitEvent(su, sw, 0));
    }
    const double* P = A + (long)k2 + (long)k * lda;  // m2 x kb, the factored panel
    const int kb2 = m2 < nb ? m2 : nb;             // width of the next panel
    // (a) next panel's columns: rows k2.., columns [k2, k2+kb2) (lower part)
    void* tok = fla_stats_begin(su);
    FLA_TRY(launch_dgemm_mfma(su, false, true, 1, m2, kb2, kb, -1.0, P, lda, P, lda, 1.0,
                              A + (long)k2 + (long)k2 * lda, lda, dinfo));
    fla_stats_end(su, tok, 0, lower_update_flops(m2, kb2, kb));
    hipEvent_t next_ready = next_event();
    FLA_HIP_CHECK(hipEventRecord(next_ready, su));
    // (b) the rest of the trailing matrix
    const int m3 = m2 - kb2;
    if (m3 > 0) {
      const double* P3 = P + kb2;
      tok = fla_stats_begin(su);
      FLA_TRY(launch_dgemm_mfma(su, false, true, 1, m3, m3, kb, -1.0, P3, lda, P3, lda, 1.0,
                                A + (long)(k2 + kb2) + (long)(k2 + kb2) * lda, lda, dinfo));
      fla_stats_end(su, tok, 0, lower_update_flops(m3, m3, kb));
    }
    // Next panel on the panel stream, concurrent with (b).
    FLA_HIP_CHECK(hipStreamWaitEvent(sp, next_ready, 0));
    FLA_TRY(chol_panel_f64(sp, n, A, lda, k2, kb2, dinfo));
    k = k2;
  }
  // Join: s_update waits for the last panel.
  hipEvent_t fin = next_event();
  FLA_HIP_CHECK(hipEventRecord(fin, sp));
  FLA_HIP_CHECK(hipStreamWaitEvent(c.s_update, fin, 0));
  if (su != c.s_update) {
    hipEvent_t last = next_event();
    FLA_HIP_CHECK(hipEventRecord(last, su));
    FLA_HIP_CHECK(hipStreamWaitEvent(c.s_update, last, 0));
  }
  return FLA_HIP_OK;
}

extern "C" int fla_hip_dpotrf(int uplo, int n, double* A, int lda, int* info) {
  FLA_USER_STREAM_SCOPE;
  FLA_TRY(fla_ensure_ready());
  if (uplo != kLower && uplo != kUpper) return FLA_HIP_EARG;
  if (n < 0 || lda < (n > 1 ? n : 1)) return FLA_HIP_EARG;
  *info = kSuccess;
  if (n == 0) return FLA_HIP_OK;
  FlaHipCtx& c = fla_ctx();
  int* dinfo = c.dscratch;
  hipLaunchKernelGGL(set_int_kernel, dim3(1), dim3(1), 0, c.s_update, dinfo, kSuccess);
  FLA_HIP_CHECK(hipGetLastError());
  if (uplo == kUpper) FLA_TRY(launch_transpose_swap(c.s_update, n, A, lda));
  FLA_TRY(chol_lower(n, A, lda, dinfo));
  if (uplo == kUpper) FLA_TRY(launch_transpose_swap(c.s_update, n, A, lda));
  int h = kSuccess;
  FLA_HIP_CHECK(hipMemcpyAsync(&h, dinfo, sizeof(int), hipMemcpyDeviceToHost, c.s_update));
  FLA_HIP_CHECK(hipStreamSynchronize(c.s_update));
  fla_stats_harvest();
  *info = h;
  return FLA_HIP_OK;
}
