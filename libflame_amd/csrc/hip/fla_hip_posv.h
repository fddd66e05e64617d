// Cholesky factorization and solve of one small SPD matrix (n <= 512) by one
// workgroup, for the batched calls.
//
// The matrix is taken in 16 x 16 blocks in matrix-step fragment order
// (fla_hip_frag.h), left-looking: block column b of the factor is the matrix's
// block column minus the products of the finished block rows, summed in
// registers, so that every element is written once (the right-looking form
// reads and writes the whole trailing triangle per 16 columns).  Wave w owns
// the block rows i with i % 8 == w.  The right-hand sides are block rows below
// the matrix: their rows of the factor are the forward-substituted solution.
// Per block column: every wave sums its blocks, the owner of the diagonal
// block factors it (one wave, registers) meanwhile, a barrier, every wave
// solves its blocks by substitution in registers and stores them, a barrier.
// The backward substitution keeps the right-hand sides' block columns in the
// waves' registers (wave w: blocks j % 8 == w) and walks the diagonal blocks
// from the last, one barrier each.
#pragma once

#include "fla_hip_frag.h"

#include <type_traits>

namespace fla_posv {

using fla_frag::lds_barrier;

constexpr int NW = 8;           // waves
constexpr int MAXB = 512 / 16;  // block rows of the largest matrix
constexpr int ZLD = fla_frag::ZLD;

// Register r of a lane (li, lk) holds column col(lk, r) of row li of a block,
// and is the lane's operand of step r of a product over those columns.
template <typename T>
struct Frag;
template <>
struct Frag<double> {
  typedef double V __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ int col(int lk, int r) { return lk + 4 * r; }
  static __device__ __forceinline__ V step(double c, double r, V a) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(c, r, a, 0, 0, 0);
  }
};
template <>
struct Frag<float> {
  typedef float V __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ int col(int lk, int r) { return 4 * lk + r; }
  static __device__ __forceinline__ V step(float c, float r, V a) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(c, r, a, 0, 0, 0);
  }
};
// The steps' result with the wait states (10) that the vector unit needs before
// it reads it: where only branches follow, the compiler can leave them out.
__device__ __forceinline__ Frag<float>::V settled(Frag<float>::V a) {
  asm("s_nop 9" : "+v"(a));
  return a;
}
// acc + R C'
template <typename T>
__device__ __forceinline__ typename Frag<T>::V product(typename Frag<T>::V c, typename Frag<T>::V r,
                                                       typename Frag<T>::V acc) {
#pragma unroll
  for (int s = 0; s < 4; ++s) acc = Frag<T>::step(c[s], r[s], acc);
  return acc;
}

// What a substitution with a lower-triangular block L needs: l = -L in
// fragment order; cf[r]: of the lane's column c = col(lk, r) the reciprocal of
// the diagonal and the negated entries of row c in the lane's group of four
// columns before c (FP64: columns 4r..4r+2, which sit in the other rows of 16
// lanes; FP32: columns 4 lk..4 lk + 2, which sit in the lane's own registers).
template <typename T>
struct Tri {
  typename Frag<T>::V l, cf[4];
};
// at(i, j): L(i, j) for j < i, any value for j >= i (never used); inv(i):
// 1 / L(i, i).
template <typename T, typename At, typename Inv>
__device__ __forceinline__ void load_tri(Tri<T>& t, int li, int lk, At at, Inv inv) {
  constexpr bool D = sizeof(T) == 8;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = Frag<T>::col(lk, r);
    t.l[r] = -at(li, c);
    t.cf[r][0] = inv(c);
#pragma unroll
    for (int q = 0; q < 3; ++q) t.cf[r][1 + q] = -at(c, (D ? 4 * r : 4 * lk) + q);
  }
}
// Right-hand sides are divided by the diagonal (dtrsm_ from the left), rows of
// the matrix multiplied by its reciprocal (dpotf2_).  The diagonal is a root,
// so that it and its reciprocal are in the normal range.
template <typename T>
__device__ __forceinline__ typename Frag<T>::V load_diag(const T* z, int lk) {
  typename Frag<T>::V d;
#pragma unroll
  for (int r = 0; r < 4; ++r) d[r] = z[Frag<T>::col(lk, r) * (ZLD + 1)];
  return d;
}

// X := X inv(L)' by substitution (x_j *= 1/l_jj, or with DIV x_j /= l_jj, d
// holding the diagonal; then x_c -= x_j l_cj).
template <bool DIV>
__device__ __forceinline__ Frag<double>::V solve(const Tri<double>& t, Frag<double>::V x, int lk,
                                                 Frag<double>::V d) {
  using S = std::conditional_t<DIV, fla_frag::ByQuotient, fla_frag::ByReciprocal>;
  return fla_frag::solve_block<S>(t.l, t.cf, x, lk, d);
}
template <bool DIV>
__device__ __forceinline__ Frag<float>::V solve(const Tri<float>& t, Frag<float>::V x, int lk,
                                                Frag<float>::V d) {
  // columns 4q..4q+3 sit in the registers of the lanes with lk == q: solved
  // there, then four matrix steps with that k slot (the others zero on both
  // sides) update the later columns; the solved ones are kept as they are
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const bool me = lk == q;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float y = x[r];
#pragma unroll
      for (int p = 0; p < r; ++p) y = fmaf(t.cf[r][1 + p], x[p], y);
      y = DIV ? fla_frag::quotient(y, t.cf[r][0], d[r]) : y * t.cf[r][0];
      x[r] = me ? y : x[r];
    }
    if (q < 3) {
      Frag<float>::V y = x;
#pragma unroll
      for (int s = 0; s < 4; ++s)
        y = Frag<float>::step(me ? t.l[s] : 0.0f, me ? x[s] : 0.0f, y);
      y = settled(y);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = lk > q ? y[r] : x[r];
    }
  }
  return x;
}

// Factors the block dg (both triangles) into z: rows 0..15 L, row 16 the
// reciprocals of its diagonal; returns the first failing column or -1.
__device__ __forceinline__ int factor(Frag<double>::V dg, double* z, int lane) {
  return fla_frag::factor16(dg, z, lane);
}
template <int C>
__device__ __forceinline__ void fmac_bcast_f(float& x, float xs, float nx) {
  asm volatile("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(x)
               : "v"(xs), "v"(nx), "i"(C));
}
template <int J, int... C>
__device__ __forceinline__ void sweep_column_f(float (&x)[16], int li, float& pinv, int& f,
                                               std::integer_sequence<int, C...>) {
  const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x[J]), J));
  if (f < 0 && !(a > 0.0f)) f = J;
  const float d = sqrtf(a), inv = 1.0f / d;
  float xs = x[J] * inv;
  const float nx = -xs;
  asm volatile("s_nop 1" : "+v"(xs));  // a VALU result is a DPP source two wait states later
  (fmac_bcast_f<J + 1 + C>(x[J + 1 + C], xs, nx), ...);
  x[J] = li == J ? d : xs;
  pinv = li == J ? inv : pinv;
}
template <int... J>
__device__ __forceinline__ void sweep_f(float (&x)[16], int li, float& pinv, int& f,
                                        std::integer_sequence<int, J...>) {
  (sweep_column_f<J>(x, li, pinv, f, std::make_integer_sequence<int, 15 - J>{}), ...);
}
__device__ __forceinline__ int factor(Frag<float>::V dg, float* z, int lane) {
  // LDS addresses formed here: kept from one block column to the next they
  // are spilled, and the reload waits for memory inside the chain
  asm volatile("" : "+v"(lane));
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) z[li * ZLD + Frag<float>::col(lk, r)] = dg[r];
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  float x[16], pinv = 0.0f;
#pragma unroll
  for (int c = 0; c < 16; ++c) x[c] = z[li * ZLD + c];
  int f = -1;
  sweep_f(x, li, pinv, f, std::make_integer_sequence<int, 16>{});
  if (lane < 16) {
#pragma unroll
    for (int c = 0; c < 16; ++c) z[lane * ZLD + c] = x[c];
    z[16 * ZLD + lane] = pinv;
  }
  return f;
}

template <typename T>
struct Shared {
  alignas(16) T z[2][17 * ZLD];  // factored diagonal blocks (by parity, backward)
  typename Frag<T>::V x[2][64];  // a solved block of the backward substitution, by parity
  int fail;
};

// Element (li, 16 k + col(lk, r)) of a block row is base[(16 k + CS r) cs +
// lane]: everything but `lane` is uniform over the wave.
template <typename T>
struct Row {
  T* base;
  long lane, cs;
  bool in;  // the lane's row exists (else lane names an existing one)
  static constexpr int CS = sizeof(T) == 8 ? 4 : 1;
  __device__ __forceinline__ T* at(int k, int r) const { return base + (long)(16 * k + CS * r) * cs + lane; }
};

// Factor (lower) of the n x n A and, with nrhs > 0, B := inv(A) B.  Returns
// the first failing column or -1; the columns before it are the factor's.
// n >= 1, or n = 0 and nrhs = 0 (the staging of the items sees to it).
template <typename T>
__device__ int posv_one(T* A, long lda, int n, T* B, long ldb, int nrhs, Shared<T>& S, int t) {
  typedef typename Frag<T>::V V;
  constexpr int TMAX = (MAXB + 256 / 16) / NW;  // block rows of a wave
  constexpr int CS = Row<T>::CS;
  const int lane = t & 63, li = lane & 15, lk = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int c0 = Frag<T>::col(lk, 0);
  const int nb = (n + 15) / 16, nr = (nrhs + 15) / 16;
  if (t == 0) S.fail = -1;
  auto block_row = [&](int i) {  // matrix rows, then right-hand sides
    Row<T> o;
    if (i < nb) {
      o.base = A + 16 * i;
      o.in = 16 * i + li < n;
      o.cs = lda;
      o.lane = (o.in ? li : n - 1 - 16 * i) + (long)c0 * lda;
    } else {
      const int j = 16 * (i - nb);
      o.base = B + (long)j * ldb;
      o.in = j + li < nrhs;
      o.cs = 1;
      o.lane = (long)(o.in ? li : nrhs - 1 - j) * ldb + c0;
    }
    return o;
  };
  for (int b = 0; b < nb; ++b) {
    // ---- sums: block (i, b) minus the products of the finished columns, 16
    // columns' terms at a time (summed into the block one by one, the FP32
    // solutions came out twice as far off: 1.5e-6 against 6.3e-7, relative) ----
    V acc[TMAX];
    const Row<T> pb = block_row(b);
    const bool ragb = 16 * b + 16 > n;
    // the wave's block rows from b on: i0 + NW u
    const int i0 = b + ((w - b) & (NW - 1));
#pragma unroll
    for (int u = 0; u < TMAX; ++u) {
      const int i = i0 + NW * u;
      if (i >= nb + nr) break;  // uniform
      const Row<T> p = block_row(i);
      V a;
      if (i == b) {  // the lower triangle's copy, the identity past the end
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = 16 * b + c0 + CS * r, row = 16 * b + li;
          const int x = row > c ? row : c, y = row > c ? c : row;
          a[r] = x < n ? A[(long)x + (long)y * lda] : (row == c ? (T)1 : (T)0);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          a[r] = (!ragb || 16 * b + c0 + CS * r < n) ? *p.at(b, r) : (T)0;
      }
      V ra[3], rb[3];
      auto load = [&](V& x, V& y, int k) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x[r] = *p.at(k, r);
          y[r] = *pb.at(k, r);
        }
        if (ragb && !pb.in) {
          y = V{0, 0, 0, 0};
          if (i == b) x = y;
        }
      };
      if (b > 0) {
        const int last = b - 1;
        load(ra[0], rb[0], 0);
        load(ra[1], rb[1], last < 1 ? last : 1);
        for (int k = 0; k < b; k += 3) {
          load(ra[2], rb[2], k + 2 < b ? k + 2 : last);
          a -= product<T>(rb[0], ra[0], V{0, 0, 0, 0});
          if (k + 1 >= b) break;
          load(ra[0], rb[0], k + 3 < b ? k + 3 : last);
          a -= product<T>(rb[1], ra[1], V{0, 0, 0, 0});
          if (k + 2 >= b) break;
          load(ra[1], rb[1], k + 4 < b ? k + 4 : last);
          a -= product<T>(rb[2], ra[2], V{0, 0, 0, 0});
        }
      }
      acc[u] = a;
      if (i == b) {
        const int f = factor(a, S.z[0], lane);
        if (lane == 0 && f >= 0) S.fail = 16 * b + f;
      }
    }
    lds_barrier();
    const int fail = S.fail;
    const int jend = fail < 0 ? 16 : fail - 16 * b;
    if (i0 == b) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = c0 + CS * r;
        if (c <= li && pb.in && c < jend) *pb.at(b, r) = S.z[0][li * ZLD + c];
      }
    }
    // (from a failing column on it holds anything, which no earlier one reads)
    Tri<T> tri;
    load_tri<T>(
        tri, li, lk, [&](int i, int j) { return S.z[0][i * ZLD + j]; },
        [&](int i) { return S.z[0][16 * ZLD + i]; });
#pragma unroll
    for (int u = 0; u < TMAX; ++u) {
      const int i = i0 + NW * u;
      if (i >= nb) break;  // uniform
      if (i == b) continue;
      const Row<T> p = block_row(i);
      const V x = solve<false>(tri, acc[u], lk, V{});
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (p.in && c0 + CS * r < jend) *p.at(b, r) = x[r];
    }
    if (fail >= 0) return fail;
    // the right-hand sides (usually one block row, of one wave)
    const V dg = load_diag(S.z[0], lk);
    for (int i = nb + ((w - nb) & (NW - 1)); i < nb + nr; i += NW) {
      V x = acc[0];
#pragma unroll
      for (int u = 1; u < TMAX; ++u)
        if (i0 + NW * u == i) x = acc[u];
      x = solve<true>(tri, x, lk, dg);
      const Row<T> p = block_row(i);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (p.in && (!ragb || 16 * b + c0 + CS * r < n)) *p.at(b, r) = x[r];
    }
    __syncthreads();  // the stored rows of L are visible to the workgroup
  }
  // ---- X := X inv(L) for the rows X of the right-hand sides, 16 at a time;
  // columns in reversed order inside a block (c' = 15 - c) ----
  for (int rt = 0; rt < nr; ++rt) {
    const bool in = 16 * rt + li < nrhs;
    T* const p = B + (long)(in ? 16 * rt + li : nrhs - 1) * ldb + (15 - c0);
    V y[MAXB / NW];
#pragma unroll
    for (int u = 0; u < MAXB / NW; ++u) {
      const int j = w + NW * u;
      if (j >= nb) break;
      const bool rag = 16 * j + 16 > n;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        y[u][r] = (!rag || 16 * j + 15 - c0 - CS * r < n) ? p[16 * j - CS * r] : (T)0;
    }
    // the diagonal block of step b, reversed (L(15 - j, 15 - i) at (i, j)),
    // to LDS one step ahead
    auto stage_diag = [&](int b) {
      const T* const D = A + (long)(16 * b) * (lda + 1);
      const int m = n - 16 * b;  // rows of the block inside the matrix
      T* const z = S.z[b & 1];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = c0 + CS * r;
        const T v = j <= li && 15 - j < m ? D[(15 - j) + (long)(15 - li) * lda] : (T)0;
        z[li * ZLD + j] = v;
        if (j == li) z[16 * ZLD + li] = 15 - li < m ? (T)1 / v : (T)1;
      }
    };
    if (w == ((nb - 1) & (NW - 1))) stage_diag(nb - 1);
    lds_barrier();
    const T* const Al = A + (15 - c0) + (long)(15 - li) * lda;
    for (int b = nb - 1; b >= 0; --b) {
      const int par = b & 1;
      const bool rag = 16 * b + 16 > n;
      if (w == (b & (NW - 1))) {
        V x = y[0];
#pragma unroll
        for (int u = 1; u < MAXB / NW; ++u)
          if (u == b / NW) x = y[u];
        Tri<T> tri;
        load_tri<T>(
            tri, li, lk, [&](int i, int j) { return S.z[par][i * ZLD + j]; },
            [&](int i) { return S.z[par][16 * ZLD + i]; });
        x = solve<true>(tri, x, lk, load_diag(S.z[par], lk));
        S.x[par][lane] = x;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (in && (!rag || 16 * b + 15 - c0 - CS * r < n)) p[16 * b - CS * r] = x[r];
      }
      // this step's blocks L(b, j) of the wave, before the wait
      V lb[MAXB / NW];
#pragma unroll
      for (int u = 0; u < MAXB / NW; ++u) {
        const int j = w + NW * u;
        if (j >= b) break;  // uniform
        const T* const q = Al + 16 * b + (long)(16 * j) * lda;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          lb[u][r] = (!rag || 16 * b + 15 - c0 - CS * r < n) ? q[-CS * r] : (T)0;
      }
      if (b > 0 && w == ((b - 1) & (NW - 1))) stage_diag(b - 1);
      lds_barrier();
      const V x = S.x[par][lane];
#pragma unroll
      for (int u = 0; u < MAXB / NW; ++u) {
        const int j = w + NW * u;
        if (j >= b) break;
        // accumulated by the matrix steps themselves: as y -= L x the
        // subtraction opens the block behind the next pass's branch, where the
        // compiler left out the wait for the steps' last register (a test
        // searches the built code for such reads)
        y[u] = product<T>(-lb[u], x, y[u]);
      }
    }
    lds_barrier();
  }
  return -1;
}

}  // namespace fla_posv
