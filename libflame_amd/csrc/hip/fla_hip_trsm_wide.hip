// Triangular solves with many right-hand sides (FLA_Trsm's general path,
// src/base/flamec/wrappers/blas/3/hip/FLA_Trsm_external_hip.c:19): blocked
// substitution, 128 rows or columns of the triangle at a time, with the
// updates as matrix products.
//
// Every case is one solve of row vectors with a lower-triangular block L on
// the right, x L' = b, ascending: a solve from the left is its transpose
// (the right-hand sides are the rows), and a descending one has its indices
// reversed.  One launch per kWideBlocks diagonal blocks writes them in that
// form and in the order the solve reads them; one wave then solves 16 right-hand sides
// by substitution (dtrsm_'s update order; its division by the diagonal from the
// left, its multiplication by the reciprocal from the right).
#include "fla_hip_frag.h"
#include "fla_hip_internal.h"

#include <type_traits>

namespace {

using namespace fla_frag;

constexpr long kBlockStride = (long)FB * FB;  // doubles of workspace per diagonal block
// Blocks per group: the product with everything outside a group contracts
// over 512, so that the right-hand sides are read and written n / 512 times.
constexpr int kGroup = 4;

static_assert(kWideBlocks % kGroup == 0, "a group's blocks are written together");

// Diagonal block k0 + blockIdx.x of the triangle A: L(i, j) = U(j, i) for
// ascending solves x U = b (U upper), reversed otherwise; U(k, c) =
// swap ? A(c, k) : A(k, c).  Identity beyond the block's order.  recip: the
// diagonal's reciprocals among the coefficients, else the diagonal.
__global__ __launch_bounds__(512) void pack_blocks_kernel(int n, int k0,
                                                          const double* __restrict__ A, long lda,
                                                          int swap, int rev, int unit, int recip,
                                                          double* __restrict__ W) {
  __shared__ double S[FB * (FB + 1)];  // A's block: (i, j) at S[j * (FB + 1) + i]
  const int r0 = (k0 + blockIdx.x) * FB, nb = min(FB, n - r0);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int li = lane & 15, lk = lane >> 4;
  for (int q0 = 0; q0 < FB * FB / 512; q0 += 8) {
    double v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = t + (q0 + q) * 512, i = e % FB, j = e / FB;
      v[q] = (i < nb && j < nb) ? A[(long)(r0 + i) + (long)(r0 + j) * lda] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = t + (q0 + q) * 512;
      S[(e / FB) * (FB + 1) + e % FB] = v[q];
    }
  }
  __syncthreads();
  auto at = [&](int i, int j) {  // L(i, j), i >= j
    if (i >= nb) return i == j ? 1.0 : 0.0;
    if (i == j && unit) return 1.0;
    const int k = rev ? nb - 1 - j : j, c = rev ? nb - 1 - i : i;  // U(k, c)
    return swap ? S[k * (FB + 1) + c] : S[c * (FB + 1) + k];
  };
  double* const Wk = W + blockIdx.x * kBlockStride;
  // wave w writes block row w
  for (int k = 0; k <= w; ++k) {
    d2* const o = reinterpret_cast<d2*>(Wk) + (frag_q0(w) + k) * 128;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int i = 16 * w + li, j0 = 16 * k + lk + 8 * p, j1 = j0 + 4;
      o[64 * p + lane] = d2{j0 <= i ? -at(i, j0) : 0.0, j1 <= i ? -at(i, j1) : 0.0};
    }
  }
  const int r = lane & 12, q = (lane & 3) - 1, c = 16 * w + lk + r;
  double v = 0.0;
  if (q < 0)
    v = recip ? 1.0 / at(c, c) : at(c, c);
  else if (lk > q)
    v = -at(c, 16 * w + r + q);
  Wk[(long)(frag_q0(w) + w + 1) * 256 + lane] = v;
}

// Solves nrhs right-hand sides with one diagonal block in place.  LEFT: they
// are the columns of the nb x nrhs B, else the rows of the nrhs x nb B.
template <bool LEFT>
__global__ __launch_bounds__(256, 2) void solve_block_kernel(int nrhs, int nb, int rev,
                                                             const d2* __restrict__ W,
                                                             double* __restrict__ B, long ldb) {
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int row0 = ((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6)) * 16;
  if (row0 >= nrhs) return;
  const bool in = row0 + li < nrhs;
  const long row = in ? row0 + li : nrhs - 1;
  const long rs = LEFT ? ldb : 1, cs = LEFT ? 1 : ldb;
  double* const bp = B + row * rs;
  auto col = [&](int k, int r) {  // the block's column 16 k + lk + 4 r in memory, or -1
    const int c = 16 * k + lk + 4 * r;
    return c < nb ? (rev ? nb - 1 - c : c) : -1;
  };
  d4 c[NT16];
#pragma unroll
  for (int k = 0; k < NT16; ++k)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = col(k, r);
      const double v = bp[(j < 0 ? 0 : j) * cs];
      c[k][r] = j < 0 ? 0.0 : v;
    }
  // dtrsm_ divides from the left and multiplies by the reciprocal from the right
  solve_rows<std::conditional_t<LEFT, ByDivision, ByReciprocal>>(W, c, lane, [&](int jb) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = col(jb, r);
      if (in && j >= 0) bp[j * cs] = c[jb][r];
    }
  });
}

}  // namespace

int trsm_wide(hipStream_t s, bool left, bool upper, bool tr, bool unit, int m, int n,
              const double* A, long lda, double* B, long ldb, double* W) {
  const int na = left ? m : n, nrhs = left ? n : m;
  const int nblk = (na + FB - 1) / FB;
  const bool op_lower = upper == tr;
  const bool fwd = left ? op_lower : !op_lower;
  const int swap = left ? !tr : tr;
  // B[lo:hi) -= its product with the solved part [c0, c0 + k) of the triangle
  auto update = [&](int lo, int hi, int c0, int k) -> int {
    if (hi <= lo) return FLA_HIP_OK;
    if (left) {
      const double* Ap = tr ? A + (long)c0 + (long)lo * lda : A + (long)lo + (long)c0 * lda;
      return launch_dgemm_mfma(s, tr, false, 0, hi - lo, n, k, -1.0, Ap, lda, B + c0, ldb, 1.0,
                               B + lo, ldb, nullptr);
    }
    const double* Ap = tr ? A + (long)lo + (long)c0 * lda : A + (long)c0 + (long)lo * lda;
    return launch_dgemm_mfma(s, false, tr, 0, m, hi - lo, k, -1.0, B + (long)c0 * ldb, ldb, Ap, lda,
                             1.0, B + (long)lo * ldb, ldb, nullptr);
  };
  const dim3 grid((unsigned)((nrhs + 63) / 64));
  int k0 = 0;  // the first diagonal block in W
  for (int q0 = 0; q0 < nblk; q0 += kGroup) {
    if (q0 % kWideBlocks == 0) {
      const int nw = nblk - q0 < kWideBlocks ? nblk - q0 : kWideBlocks;
      k0 = fwd ? q0 : nblk - q0 - nw;
      hipLaunchKernelGGL(pack_blocks_kernel, dim3((unsigned)nw), dim3(512), 0, s, na, k0, A, lda,
                         swap, fwd ? 0 : 1, unit ? 1 : 0, left ? 0 : 1, W);
      FLA_HIP_CHECK(hipGetLastError());
    }
    const int q1 = q0 + kGroup < nblk ? q0 + kGroup : nblk;
    // the group's rows (columns) of the triangle
    const int g0 = (fwd ? q0 : nblk - q1) * FB;
    const int g1 = fwd ? (q1 * FB < na ? q1 * FB : na) : ((nblk - q0) * FB < na ? (nblk - q0) * FB : na);
    for (int q = q0; q < q1; ++q) {
      const int kb = fwd ? q : nblk - 1 - q;
      const int c0 = kb * FB, nb = na - c0 < FB ? na - c0 : FB;
      const d2* w = reinterpret_cast<const d2*>(W + (kb - k0) * kBlockStride);
      if (left)
        hipLaunchKernelGGL(solve_block_kernel<true>, grid, dim3(256), 0, s, nrhs, nb, fwd ? 0 : 1,
                           w, B + c0, ldb);
      else
        hipLaunchKernelGGL(solve_block_kernel<false>, grid, dim3(256), 0, s, nrhs, nb, fwd ? 0 : 1,
                           w, B + (long)c0 * ldb, ldb);
      FLA_HIP_CHECK(hipGetLastError());
      if (fwd)
        FLA_TRY(update(c0 + nb, g1, c0, nb));
      else
        FLA_TRY(update(g0, c0, c0, nb));
    }
    if (fwd)
      FLA_TRY(update(g1, na, g0, g1 - g0));
    else
      FLA_TRY(update(0, g0, g0, g1 - g0));
  }
  return FLA_HIP_OK;
}
