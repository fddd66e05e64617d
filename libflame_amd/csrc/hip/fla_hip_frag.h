// 16 x 16 FP64 blocks in matrix-step fragment order and solves with a
// lower-triangular 128 x 128 block, shared by the Cholesky panel and the
// triangular solves with many right-hand sides.
#pragma once

#include <hip/hip_runtime.h>

#include <utility>

namespace fla_frag {

constexpr int FB = 128;        // order of a triangular block
constexpr int NT16 = FB / 16;  // its 16-blocks per side

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double readlane_d(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Barrier that orders LDS accesses only: __syncthreads would also wait for
// the global stores in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

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

// What a substitution does with the diagonal entry of the lane's column when
// that column's turn comes (me); the other columns keep their value.  c and d:
// the column's coefficients.
// Multiplies by the reciprocal c (dtrsm_ from the right, dpotrf_).
struct ByReciprocal {
  static __device__ __forceinline__ double apply(double x, double c, double, bool me) {
    return x * (me ? c : 1.0);
  }
};
// Divides by the diagonal entry c (dtrsm_ from the left).
struct ByDivision {
  static __device__ __forceinline__ double apply(double x, double c, double, bool me) {
    return x / (me ? c : 1.0);
  }
};
// The quotient x / d from c = 1 / d rounded, where neither is subnormal: the
// product corrected by its residual, which rounds correctly (Markstein).  Of an
// infinite or NaN product the residual is NaN or infinite; held finite, it
// leaves the product as it is.
__device__ __forceinline__ double quotient(double x, double c, double d) {
  const double q = x * c, y = fma(fma(-d, q, x), c, q);
  return fabs(q) < __builtin_inf() ? y : q;
}
__device__ __forceinline__ float quotient(float x, float c, float d) {
  const float q = x * c;
  return fmaf(__builtin_amdgcn_fmed3f(fmaf(-d, q, x), -0x1p126f, 0x1p126f), c, q);
}
struct ByQuotient {
  static __device__ __forceinline__ double apply(double x, double c, double d, bool me) {
    const double q = quotient(x, c, d);
    return me ? q : x;
  }
};

// X := T inv(L)' for a block T by substitution, dtrsm_'s operations in its
// order (x_j *= 1/l_jj or x_j /= l_jj, then t_c -= x_j l_cj).  The four
// columns 4r..4r+3 sit in register r of the four rows of 16 lanes: within them
// the solved column is copied across the rows, then one matrix step updates
// the later columns.  Columns already solved are kept by selects and by taking
// only the matrix step's later registers, not by zero multipliers: x_j may be
// infinite.  l: -L (any value on and above the diagonal); cf[r]: of the lane's
// column c = lk + 4r what SCALE takes and -l_cj for j = 4r..4r+2 (any value
// where c <= j); d[r]: SCALE's second coefficient.  About 1100 cycles with
// reciprocals; a matrix step per column,
// whose result has to come back through the vector unit each time, took 3200.
template <typename SCALE = ByReciprocal>
__device__ __forceinline__ d4 solve_block(d4 l, const d4 (&cf)[4], d4 t, int lk,
                                          d4 d = d4{}) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    double x = t[r], y;
    x = SCALE::apply(x, cf[r][0], d[r], lk == 0);
    y = fma(cf[r][1], row_to_all<0>(x), x);
    x = lk > 0 ? y : x;
    x = SCALE::apply(x, cf[r][0], d[r], lk == 1);
    y = fma(cf[r][2], row_to_all<1>(x), x);
    x = lk > 1 ? y : x;
    x = SCALE::apply(x, cf[r][0], d[r], lk == 2);
    y = fma(cf[r][3], row_to_all<2>(x), x);
    x = lk > 2 ? y : x;
    x = SCALE::apply(x, cf[r][0], d[r], lk == 3);
    t[r] = x;
    if (r < 3) {
      const d4 u = mfma_step(l[r], x, t);
#pragma unroll
      for (int q = r + 1; q < 4; ++q) t[q] = u[q];
    }
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
template <typename SCALE, typename F>
__device__ __forceinline__ void solve_rows(const d2* __restrict__ W, d4 (&c)[NT16], int lane,
                                           F done) {
  constexpr int PF = 6;
  constexpr Stream kStream = make_stream();
  const int lk = lane >> 4;
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
        c[jb] = solve_block<SCALE>(d4{l0.x, l0.y, l1.x, l1.y}, cf, c[jb], lk);
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

// One wave factors a 16 x 16 symmetric block.  Lane li of each row of 16 lanes
// holds row li (x[c] = a(li, c)).  Column j: d = sqrt(a_jj), x_j *= 1/d, then
// x_c -= x_j l_cj, with l_cj broadcast from lane c by the update instruction
// itself (DPP row_newbcast).  (Through lane reads the pivot alone took 80
// cycles from its update to its first use, and every multiplier two reads.)
// A VALU result is a DPP source only two wait states later: the statements
// below keep other instructions in between, or carry the s_nop.
template <int C>
__device__ __forceinline__ void sweep_update(double& x, double xs, double nx) {
  asm volatile("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(x)
               : "v"(xs), "v"(nx), "i"(C));
}
// Updates of the columns C0 <= C < C1 (none past 15).
template <int C0, int C1>
__device__ __forceinline__ void sweep_updates(double (&x)[16], double xs, double nx) {
  if constexpr (C0 < C1 && C0 < 16) {
    sweep_update<C0>(x[C0], xs, nx);
    sweep_updates<C0 + 1, C1>(x, xs, nx);
  }
}
template <int J>
__device__ __forceinline__ double bcast16(double x) {
  double a;
  asm volatile("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
               : "=v"(a)
               : "v"(x), "i"(J));
  return a;
}

// Column J with the pivot a already broadcast.  The root by Goldschmidt's
// iteration from v_rsq_f64 (g -> sqrt(a), h -> 1/(2 sqrt(a))) and a residual
// correction, the reciprocal by a Newton step against the rounded root
// (Markstein): exact roots and reciprocals come out exact, as the reference's
// sqrt and division give them.  The updates of column J - 1 right of column J
// (xsp, nxp) fill the chain's latencies; column J + 1 is updated first, so
// that the next pivot is on its way at the end.  piv, pinv: lane J's root and
// reciprocal.
template <int J>
__device__ __forceinline__ void sweep_column(double (&x)[16], int li, double& piv, double& pinv,
                                             double& a, double& xsp, double& nxp) {
  constexpr int N = J > 0 ? 15 - J : 0, C1 = J + 1 + (N + 2) / 3, C2 = J + 1 + (2 * N + 2) / 3;
  const double y = __builtin_amdgcn_rsq(a);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (J > 0) sweep_updates<J + 1, C1>(x, xsp, nxp);
  __builtin_amdgcn_sched_barrier(0);
  double g = a * y, h = 0.5 * y;
  double e = fma(-h, g, 0.5);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (J > 0) sweep_updates<C1, C2>(x, xsp, nxp);
  __builtin_amdgcn_sched_barrier(0);
  h = fma(h, e, h);
  g = fma(g, e, g);
  e = fma(-g, g, a);
  const double h2 = h + h;
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (J > 0) sweep_updates<C2, 16>(x, xsp, nxp);
  __builtin_amdgcn_sched_barrier(0);
  const double d = fma(e, h, g);
  const double inv = fma(fma(-d, h2, 1.0), h2, h2);
  xsp = x[J] * inv;
  nxp = -xsp;
  asm volatile("s_nop 1" : "+v"(xsp));
  if constexpr (J < 15) {
    sweep_update<J + 1>(x[J + 1], xsp, nxp);
    a = bcast16<J + 1>(x[J + 1]);
  }
  x[J] = li == J ? d : xsp;
  piv = li == J ? d : piv;
  pinv = li == J ? inv : pinv;
}
template <int... J>
__device__ __forceinline__ void sweep16(double (&x)[16], int li, double& piv, double& pinv,
                                        std::integer_sequence<int, J...>) {
  double a = bcast16<0>(x[0]), xsp = 0.0, nxp = 0.0;
  (sweep_column<J>(x, li, piv, pinv, a, xsp, nxp), ...);
}

// A factored 16 x 16 diagonal block in LDS: rows 0..15 hold L (below and on
// the diagonal), row 16 the reciprocals of its diagonal.  The row length keeps
// 16-byte accesses aligned and spreads the rows over the banks.
constexpr int ZLD = 18;

// The sweep with the library's root and division, any pivot range, in place
// in LDS (rare: it takes no registers from the fast one); returns the first
// column whose pivot is <= 0 or NaN (bl1_dsqrte's rule), else -1.
__device__ __forceinline__ int sweep16_any(double* z, int lane) {
  const int li = lane & 15;
  int f = -1;
#pragma unroll 1
  for (int j = 0; j < 16; ++j) {
    const double a = z[j * ZLD + j];
    if (f < 0 && !(a > 0.0)) f = j;
    const double d = sqrt(a), inv = 1.0 / d;
    const double xs = z[li * ZLD + j] * inv;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (lane < 16) {
      if (li > j) z[li * ZLD + j] = xs;
      if (li == j) {
        z[j * ZLD + j] = d;
        z[16 * ZLD + j] = inv;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll 1
    for (int c = j + 1; c < 16; ++c)
      if (lane < 16 && li >= c) z[li * ZLD + c] = fma(-xs, z[c * ZLD + j], z[li * ZLD + c]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  return __builtin_amdgcn_readfirstlane(f);
}

// Factors the symmetric block dg (fragment order) into z, one wave.  Returns
// the first failing column or -1.  Pivots outside [2^-700, 2^1000] (products
// of the fast sweep could under- or overflow) and failing ones take the
// general sweep.
__device__ __forceinline__ int factor16(d4 dg, double* z, int lane) {
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) z[li * ZLD + lk + 4 * r] = dg[r];
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  double x[16], piv = 0.0, pinv = 0.0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const d2 v = *reinterpret_cast<const d2*>(z + li * ZLD + 2 * q);
    x[2 * q] = v.x;
    x[2 * q + 1] = v.y;
  }
  sweep16(x, li, piv, pinv, std::make_integer_sequence<int, 16>{});
  if (!__all(piv >= 0x1p-350 && piv <= 0x1p500)) return sweep16_any(z, lane);
  if (lane < 16) {
#pragma unroll
    for (int q = 0; q < 8; ++q)
      *reinterpret_cast<d2*>(z + lane * ZLD + 2 * q) = d2{x[2 * q], x[2 * q + 1]};
    z[16 * ZLD + lane] = pinv;
  }
  return -1;
}

}  // namespace fla_frag
