// 16 x 16 FP64 blocks in matrix-step fragment order and solves with a
// lower-triangular 128 x 128 block, shared by the Cholesky panel and the
// triangular solves with many right-hand sides.
#pragma once

#include <hip/hip_runtime.h>

namespace fla_frag {

constexpr int FB = 128;        // order of a triangular block
constexpr int NT16 = FB / 16;  // its 16-blocks per side

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

// 16 x 16 blocks in fragment order.  v_mfma_f64_16x16x4f64 leaves D(x, y) in
// lane 16*(x%4) + y, register x/4; with x the column and y the row of a
// block X, lane (li = lane%16, lk = lane/16) holds X(li, lk + 4 s) in
// register s.  That register is at the same time the lane's operand of step
// s of a product over X's columns, as the row operand (X Z') and as the
// column operand (Z X'), so blocks move between products without any
// shuffle.  In memory a block is 128 d2: entry [p][lane] = steps 2p, 2p+1.
__device__ __forceinline__ d4 mfma_step(double colf, double rowf, d4 acc) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(colf, rowf, acc, 0, 0, 0);
}
// acc + R C' for blocks R (row operand) and C (column operand: c0, c1).
__device__ __forceinline__ d4 mfma_block(d2 c0, d2 c1, d4 r, d4 acc) {
  acc = mfma_step(c0.x, r[0], acc);
  acc = mfma_step(c0.y, r[1], acc);
  acc = mfma_step(c1.x, r[2], acc);
  return mfma_step(c1.y, r[3], acc);
}
// Lanes of row Q of 16 lanes, copied to all four rows (two swaps a word).
template <int Q>
__device__ __forceinline__ unsigned row_to_all(unsigned x) {
  const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);  // {0,0,2,2}, {1,1,3,3}
  const unsigned p = a[Q & 1];
  const auto b = __builtin_amdgcn_permlane32_swap(p, p, false, false);  // {0,1,0,1}, {2,3,2,3}
  return b[Q >> 1];
}
template <int Q>
__device__ __forceinline__ double row_to_all(double x) {
  return __hiloint2double((int)row_to_all<Q>((unsigned)__double2hiint(x)),
                          (int)row_to_all<Q>((unsigned)__double2loint(x)));
}

// X := T inv(L)' for a block T by substitution, dtrsm_'s operations in its
// order (x_j *= 1/l_jj, then t_c -= x_j l_cj).  The four columns 4r..4r+3 sit
// in register r of the four rows of 16 lanes: within them the solved column
// is copied across the rows, then one matrix step updates the later columns.
// l: -L; cf[r]: of the lane's column c = lk + 4r the reciprocal 1/l_cc and
// -l_cj for j = 4r..4r+2 (0 where c <= j).  About 1100 cycles; a matrix step
// per column, whose result has to come back through the vector unit each
// time, took 3200.
__device__ __forceinline__ d4 solve_block(d4 l, const d4 (&cf)[4], d4 t, int li, int lk) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    double x = t[r];
    x *= lk == 0 ? cf[r][0] : 1.0;
    x = fma(cf[r][1], row_to_all<0>(x), x);
    x *= lk == 1 ? cf[r][0] : 1.0;
    x = fma(cf[r][2], row_to_all<1>(x), x);
    x *= lk == 2 ? cf[r][0] : 1.0;
    x = fma(cf[r][3], row_to_all<2>(x), x);
    x *= lk == 3 ? cf[r][0] : 1.0;
    t[r] = x;
    if (r < 3) t = mfma_step(li >= 4 * (r + 1) ? l[r] : 0.0, x, t);
  }
  return t;
}

// The blocks of a lower-triangular 128 x 128 block L as a solve with L' on the
// right reads them: for 16-column block jb the negated blocks left of the diagonal
// -L(jb, 0..jb-1), then -L(jb, jb), then the coefficients cf[lk][r][4] of
// solve_block (64 doubles).
constexpr int frag_q0(int jb) { return jb * (jb - 1) / 2 + 2 * jb; }
constexpr int NFRAG = frag_q0(NT16);
static_assert(NFRAG * 256 <= FB * FB, "the fragments fit the 128 x 128 scratch block");

// The order in which a solve reads L's blocks: row jb's, left to right (the
// coefficients after each diagonal block are read separately).
constexpr int NQ = NT16 * (NT16 + 1) / 2;
struct Stream {
  int block[NQ];
};
constexpr Stream make_stream() {
  Stream s{};
  for (int jb = 0, q = 0; jb < NT16; ++jb)
    for (int k = 0; k <= jb; ++k, ++q) s.block[q] = frag_q0(jb) + k;
  return s;
}

// The solve itself, one wave: c[k] (fragment order, k = 0..7) holds 16 rows of
// the 128 columns and is overwritten by c inv(L)'; W: L's blocks.  They are
// read PF blocks ahead of their use (88 KB, shared by every wave through the
// caches); done(jb) is called when column block jb is final.
template <typename F>
__device__ __forceinline__ void solve_rows(const d2* __restrict__ W, d4 (&c)[NT16], int lane,
                                           F done) {
  constexpr int PF = 6;
  constexpr Stream kStream = make_stream();
  const int li = lane & 15, lk = lane >> 4;
  d2 ring[PF][2];
  d4 cf[4];
  const d2* const Wl = W + lane;
  auto coefs = [&](int jb) {
    const d2* const p = W + (frag_q0(jb) + jb + 1) * 128 + lk * 8;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const d2 u = p[2 * r], v = p[2 * r + 1];
      cf[r] = d4{u.x, u.y, v.x, v.y};
    }
  };
#pragma unroll
  for (int q = 0; q < PF; ++q) {
    ring[q][0] = Wl[kStream.block[q] * 128];
    ring[q][1] = Wl[kStream.block[q] * 128 + 64];
  }
  coefs(0);
#pragma unroll
  for (int jb = 0; jb < NT16; ++jb) {
#pragma unroll
    for (int k = 0; k < NT16; ++k) {
      if (k > jb) break;
      const int q = jb * (jb + 1) / 2 + k;
      const d2 l0 = ring[q % PF][0], l1 = ring[q % PF][1];
      if (k < jb)
        c[jb] = mfma_block(l0, l1, c[k], c[jb]);
      else
        c[jb] = solve_block(d4{l0.x, l0.y, l1.x, l1.y}, cf, c[jb], li, lk);
      if (q + PF < NQ) {
        ring[q % PF][0] = Wl[kStream.block[q + PF] * 128];
        ring[q % PF][1] = Wl[kStream.block[q + PF] * 128 + 64];
      }
      if (k == jb && jb + 1 < NT16) coefs(jb + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    done(jb);
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace fla_frag
