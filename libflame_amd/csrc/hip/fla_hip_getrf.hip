// Blocked LU with partial pivoting on one MI355X.
//
// Reference algorithm: FLA_LU_piv_blk_var5
//   (src/lapack/dec/lu/piv/vars/flamec/FLA_LU_piv_blk_var5.c:13-114):
//     [A11;A21], p1 := LU_piv([A11;A21]);  apply p1 to [A10;A20] and [A12;A22];
//     A12 := inv(trilu(A11)) * A12;         A22 := A22 - A21 * A12
// with the leaf's pivot rule (bl1_damax -> idamax_, first maximal |x|;
// src/flablas/f2c/idamax.c:40-46), FLAME-native relative pivots
// (src/lapack/util/app/piv/ln/flamec/FLA_Apply_pivots_ln_opt_var1.c:323), and
// the null-pivot rule of FLA_LU_piv_opd_var4 (FLA_LU_piv_opt_var4.c:277-283,
// 325-332): the first null pivot's index is returned, its interchange and
// scaling are skipped, the update uses the unchanged row j, and the sweep
// continues.
//
// Panel: 128 columns as sub-panels of 32.  A sub-panel is one kernel that
// keeps its rows in VGPRs (a thread owns whole rows), 1024 rows a workgroup;
// up to 1024 rows there is nothing to exchange.  With more rows each column
// costs one all-to-all exchange: every workgroup publishes its pivot
// candidate together with the candidate's row, reads all of them, and picks
// the same pivot.  The exchange words live in uncached device memory (no L2
// write-back or invalidate across the XCDs) and carry their own tags, so no
// store needs to be acknowledged before another one and no separate flag is
// polled: each 8-byte word holds a 32-bit payload and the 32-bit tag of the
// (launch, column) it belongs to, and a reader takes a word only once its
// tag is current.  Every wait is bounded.  Between sub-panels one kernel
// applies the interchanges to the panel's other columns and solves for U12,
// and a product updates the columns to the right.
#include <hip/hip_runtime.h>

#include <utility>

#include "fla_hip_internal.h"

namespace {

constexpr int PW = 128;  // maximum panel width
constexpr int SW = 32;   // sub-panel width
constexpr int NT = 512;  // threads of a sub-panel workgroup
constexpr int RQ = 2;    // rows per thread
constexpr int ROWS_PER_WG = NT * RQ;
constexpr unsigned long long kSpinTicks = 200000000ULL;  // 2 s of the 100 MHz wall clock
constexpr int MAX_P = 64;  // sub-panel workgroups
constexpr int SLOT = 40;   // exchange entries of a slot: 32 values, 3 header entries, padding

typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) u64x2 g_u64x2;
typedef __attribute__((address_space(1))) unsigned long long g_u64;

// Exchange area (tagged 16-byte entries, two parities: column j uses j & 1):
// slots [2][P + 1][SLOT], slot w < P from workgroup w, slot P (the diagonal
// row j) from workgroup 0.  Entries 0..31: the row's values; 32: {candidate
// |v|}; 33: {its row, its original row}; 34: {the workgroup's last NaN row or
// -1}.  The candidate is the first maximum after the last NaN, or the last
// NaN itself with |v| = -1 when nothing follows it.  A slot is five whole
// 128-byte lines, stored by one instruction: a partial-line write to uncached
// memory is a read-modify-write.
struct PanelComm {
  u64x2* slots;
  int* err;       // wait-limit flag
  int* orig[2];   // original row (in the panel) of every row, before / after a sub-panel
  int* submoved;  // the current sub-panel's row moves
};

// Stores need no ordering among themselves (each word carries its tag): a
// plain 16-byte store.  Loads are relaxed atomics of the two 8-byte words, so
// a polling loop re-reads memory without waiting after every load.
__device__ __forceinline__ void put(u64x2* p, unsigned lo, unsigned hi, unsigned tag) {
  u64x2 w;
  w.x = (unsigned long long)lo | ((unsigned long long)tag << 32);
  w.y = (unsigned long long)hi | ((unsigned long long)tag << 32);
  *(g_u64x2*)p = w;
}
__device__ __forceinline__ u64x2 get(const u64x2* p) {
  g_u64* q = (g_u64*)p;
  u64x2 w;
  w.x = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  w.y = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return w;
}
__device__ __forceinline__ bool tagged(u64x2 w, unsigned tag) {
  return (unsigned)(w.x >> 32) == tag && (unsigned)(w.y >> 32) == tag;
}
__device__ __forceinline__ double as_d(u64x2 w) {
  return __longlong_as_double((long long)((w.x & 0xffffffffull) | (w.y << 32)));
}
__device__ __forceinline__ int lo_i(u64x2 w) { return (int)(unsigned)w.x; }
__device__ __forceinline__ int hi_i(u64x2 w) { return (int)(unsigned)w.y; }

// Wave reductions with DPP: prefix within each row of 16 lanes (row_shr 1,
// 2, 4, 8), then across rows (row_bcast 15, 31); lane 63 ends with the
// result.  Lanes whose source is out of range keep their own value.
template <int CTRL, int ROWM>
__device__ __forceinline__ int dpp_i(int x) {
  return __builtin_amdgcn_update_dpp(x, x, CTRL, ROWM, 0xf, false);
}
template <int CTRL, int ROWM>
__device__ __forceinline__ double dpp_d(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = dpp_i<CTRL, ROWM>((int)b), hi = dpp_i<CTRL, ROWM>((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double readlane_d(double x, int l) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_max_d(double x) {
  x = fmax(x, dpp_d<0x111, 0xf>(x));
  x = fmax(x, dpp_d<0x112, 0xf>(x));
  x = fmax(x, dpp_d<0x114, 0xf>(x));
  x = fmax(x, dpp_d<0x118, 0xf>(x));
  x = fmax(x, dpp_d<0x142, 0xa>(x));
  x = fmax(x, dpp_d<0x143, 0xc>(x));
  return readlane_d(x, 63);
}
__device__ __forceinline__ int wave_max_i(int x) {
  x = max(x, dpp_i<0x111, 0xf>(x));
  x = max(x, dpp_i<0x112, 0xf>(x));
  x = max(x, dpp_i<0x114, 0xf>(x));
  x = max(x, dpp_i<0x118, 0xf>(x));
  x = max(x, dpp_i<0x142, 0xa>(x));
  x = max(x, dpp_i<0x143, 0xc>(x));
  return __builtin_amdgcn_readlane(x, 63);
}
__device__ __forceinline__ int wave_min_i(int x) {
  x = min(x, dpp_i<0x111, 0xf>(x));
  x = min(x, dpp_i<0x112, 0xf>(x));
  x = min(x, dpp_i<0x114, 0xf>(x));
  x = min(x, dpp_i<0x118, 0xf>(x));
  x = min(x, dpp_i<0x142, 0xa>(x));
  x = min(x, dpp_i<0x143, 0xc>(x));
  return __builtin_amdgcn_readlane(x, 63);
}

// Barrier that orders LDS accesses only (the exchange stores stay in flight).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// a += lane (C & 15) of u (in each row of 16 lanes) times b: one instruction
// per element of the rank-1 update, with the pivot row spread over the lanes.
template <int C>
__device__ __forceinline__ void fmac_bcast(double& a, double u, double b) {
  asm volatile("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(a)
               : "v"(u), "v"(b), "i"(C & 15));
}
// The thread rows are held as four chunks of eight columns, rotated so that
// the current column is position I of chunk 0; finished chunks are at the end.
// Position I becomes the multiplier l, the positions right of it (in the
// nlive unfinished chunks) take the rank-1 update, x the next position's value.
template <int I, int... C>
__device__ __forceinline__ void update_tail(double (&v)[SW], double u0, double nl,
                                            std::integer_sequence<int, C...>) {
  (fmac_bcast<I + 1 + C>(v[I + 1 + C], u0, nl), ...);
}
template <int I>
__device__ __forceinline__ void update_first(double (&v)[SW], double u0, double l, double nl,
                                             double& x) {
  v[I] = l;
  update_tail<I>(v, u0, nl, std::make_integer_sequence<int, 7 - I>{});
  if constexpr (I < 7) x = v[I + 1];
}
template <int CH, int... I>
__device__ __forceinline__ void update_chunk(double (&v)[SW], double u, double nl,
                                             std::integer_sequence<int, I...>) {
  (fmac_bcast<8 * CH + I>(v[8 * CH + I], u, nl), ...);
}

// Copies the row of lane cl (register row cq, uniform) to dst in LDS.
__device__ __forceinline__ void stage_row(double* dst, const double (&v)[RQ][SW], int cq, int lane,
                                          int cl) {
  if (lane != cl) return;
  if (cq == 0) {
#pragma unroll
    for (int c = 0; c < SW; ++c) dst[c] = v[0][c];
  } else {
#pragma unroll
    for (int c = 0; c < SW; ++c) dst[c] = v[1][c];
  }
}

__device__ __forceinline__ unsigned wave_max_u(unsigned x) {
  x = max(x, (unsigned)dpp_i<0x111, 0xf>((int)x));
  x = max(x, (unsigned)dpp_i<0x112, 0xf>((int)x));
  x = max(x, (unsigned)dpp_i<0x114, 0xf>((int)x));
  x = max(x, (unsigned)dpp_i<0x118, 0xf>((int)x));
  x = max(x, (unsigned)dpp_i<0x142, 0xa>((int)x));
  x = max(x, (unsigned)dpp_i<0x143, 0xc>((int)x));
  return (unsigned)__builtin_amdgcn_readlane((int)x, 63);
}
// Maximum over lanes 0..7.
__device__ __forceinline__ double max8_d(double x) {
  x = fmax(x, dpp_d<0x111, 0xf>(x));
  x = fmax(x, dpp_d<0x112, 0xf>(x));
  x = fmax(x, dpp_d<0x114, 0xf>(x));
  return readlane_d(x, 7);
}

// The wave's first maximum of the keys (>= 0, or -1 for none) in row order
// (register row, then lane).  The high words (plus one; 0: none) decide it
// unless two of the largest agree in them.
__device__ __forceinline__ void wave_first_max(const double (&key)[RQ], int& cq, int& cl) {
  unsigned h[RQ];
#pragma unroll
  for (int q = 0; q < RQ; ++q)
    h[q] = key[q] >= 0.0 ? (unsigned)__double2hiint(key[q]) + 1u : 0u;
  const unsigned m = wave_max_u(max(h[0], h[1]));
  unsigned long long b0 = __ballot(h[0] == m), b1 = __ballot(h[1] == m);
  if (__builtin_popcountll(b0) + __builtin_popcountll(b1) > 1) {
    const double d = wave_max_d(fmax(key[0], key[1]));
    b0 = __ballot(key[0] == d);
    b1 = __ballot(key[1] == d);
  }
  cq = b0 ? 0 : 1;
  cl = __builtin_ctzll(b0 ? b0 : b1);
}

struct SubHead {
  double val;  // the wave's largest |a|, -1: none
  int row;     // its row in the sub-panel
  int nan;     // the wave's last NaN row, -1: none
};

// LU with partial pivoting of the M x W sub-panel at A (W <= 32), column k of
// the matrix first.  piv: its pivots; cm.submoved: its row moves; cm.orig:
// the panel's row origins before (first == 0: the identity) and after;
// pmoved, when given: the whole panel's row moves.  `first`: the sub-panel's
// first row in the panel.
// Per column: every wave's candidate to LDS, a barrier, every wave picks the
// workgroup's; the candidate's owner copies its row to LDS and (one
// workgroup) a barrier makes it visible, or (more) publishes it, all waves
// poll the workgroups' slots into LDS, a barrier, and every wave picks the
// pivot.  Only the winner's row is copied: a single lane's 16-byte LDS writes
// cost as much as a full wave's, and all eight waves doing so took 1500
// cycles.  The column loop is not unrolled (450 KB of code, every column
// fetched from L2 once, 2-5 us a column); only the update's first chunk
// depends on the column's position at compile time.
// Bound: the chain of LDS, cross-lane and scalar steps of the search per
// column, and with more workgroups the exchange's memory round trip.  32
// columns take 79 us with one workgroup and 130-155 with 2-16 (n = 16384: 141
// on average); a 128-column panel as one kernel with a second round trip for
// the pivot row took 620 us at any height.
__global__ __launch_bounds__(NT, 2) void lu_sub_kernel(int M, int W, double* __restrict__ A,
                                                       long lda, int k, int* __restrict__ piv,
                                                       int* __restrict__ info, PanelComm cm,
                                                       int flip, int first,
                                                       int* __restrict__ pmoved,
                                                       unsigned tagbase) {
  // A wait that expired in an earlier launch of this factorization aborts all
  // later ones; their move lists are empty (an older, taller panel's would
  // move rows past this one's last).
  if (__hip_atomic_load(cm.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      __hip_atomic_store(&cm.submoved[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (pmoved) __hip_atomic_store(&pmoved[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return;
  }
  constexpr int NW = NT / 64;
  __shared__ __attribute__((aligned(16))) double crow[2][SW];  // the candidate's row, by parity
  __shared__ __attribute__((aligned(16))) double jrow[2][SW];  // row j before the interchange
  __shared__ __attribute__((aligned(16))) double gx[MAX_P + 1][SW];  // the exchanged rows
  __shared__ SubHead head[2][NW];
  __shared__ double gval[MAX_P + 1];
  __shared__ int corg[2], jorg[2];
  __shared__ int grow[MAX_P + 1], gorg[MAX_P + 1], gnan[MAX_P + 1], dead, pivs[SW], first_null;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int base = blockIdx.x * ROWS_PER_WG, P = gridDim.x;
  if (t == 0) {
    dead = 0;
    first_null = -1;
    if (base == 0) {
      // The move lists are appended to only after every workgroup has read
      // this workgroup's first slot, which is stored after this reset
      // completes.
      __hip_atomic_store(&cm.submoved[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (pmoved) __hip_atomic_store(&pmoved[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_s_waitcnt(0);
    }
  }
  double v[RQ][SW], x[RQ];  // x: the current column
  int og[RQ];               // original row
#pragma unroll
  for (int q = 0; q < RQ; ++q) {
    const int r = base + q * NT + t;
    og[q] = r;
    const double* const a = A + (r < M ? r : M - 1);
    if (W == SW) {
#pragma unroll
      for (int c = 0; c < SW; ++c) v[q][c] = a[(long)c * lda];
    } else {
#pragma unroll
      for (int c = 0; c < SW; ++c) {
        const double y = a[(long)(c < W ? c : 0) * lda];
        v[q][c] = c < W ? y : 0.0;
      }
    }
    x[q] = v[q][0];
  }
  __syncthreads();

#pragma unroll 1
  for (int j = 0; j < SW; ++j) {
    const int pos = j & 7, nlive = 4 - (j >> 3);
    if (j < W) {
      const int par = j & 1;
      // ---- this wave's candidate ----
      double key[RQ];
      int nanrow = -1;
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        const int r = base + q * NT + t;
        const bool act = r >= j && r < M;
        key[q] = (act && x[q] == x[q]) ? fabs(x[q]) : -1.0;
        const unsigned long long nb = __ballot(act && x[q] != x[q]);
        if (nb) nanrow = base + q * NT + 64 * wave + 63 - __builtin_clzll(nb);
      }
      int cq, cl;
      wave_first_max(key, cq, cl);
      if (lane == cl)
        head[par][wave] = SubHead{cq ? key[1] : key[0], base + cq * NT + t, nanrow};
      lds_barrier();
      // ---- the workgroup's candidate lrow, |a| = lval ----
      SubHead hd = head[par][lane & (NW - 1)];
      int lnan = -1;
      if (__ballot(hd.nan >= 0)) {  // a NaN: the search restarts after the last one (rare)
        lnan = wave_max_i(hd.nan);
        lds_barrier();
#pragma unroll
        for (int q = 0; q < RQ; ++q)
          if (base + q * NT + t <= lnan) key[q] = -1.0;
        wave_first_max(key, cq, cl);
        if (lane == cl)
          head[par][wave] = SubHead{cq ? key[1] : key[0], base + cq * NT + t, nanrow};
        lds_barrier();
        hd = head[par][lane & (NW - 1)];
      }
      const double lval = max8_d(hd.val);
      int lrow;
      {
        const unsigned long long b = __ballot(hd.val == lval && lane < NW);
        if (!(lval >= 0.0))
          lrow = lnan;  // nothing but the NaN
        else if ((b & (b - 1)) == 0)
          lrow = __builtin_amdgcn_readlane(hd.row, __builtin_ctzll(b));
        else  // equal maxima: the smallest row
          lrow = wave_min_i((b >> lane) & 1ull ? hd.row : 0x7fffffff);
      }
      // ---- its row (and row j) to LDS ----
      const int lt = (lrow - base) & (NT - 1);
      const bool own = wave == (lt >> 6), ownj = base == 0 && wave == 0;
      if (own) {
        const int q = (lrow - base) / NT;
        stage_row(crow[par], v, q, lane, lt & 63);
        if (lane == (lt & 63)) corg[par] = q ? og[1] : og[0];
      }
      if (ownj) {
        stage_row(jrow[par], v, 0, lane, j);
        if (lane == j) jorg[par] = og[0];
      }
      const double* prow = crow[par];
      const double* jr = jrow[par];
      const int *orgs = corg + par, *orgj = jorg + par;
      int r = lrow;
      if (P == 1) {
        lds_barrier();
      } else {
        // ---- all-to-all exchange ----
        const unsigned tag = tagbase | (unsigned)(j + 1);
        u64x2* const area = cm.slots + (long)par * (MAX_P + 1) * SLOT;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        auto publish = [&](const double* row, int slot, int gr, int go) {
          unsigned lo = 0, hi = 0;
          if (lane <= SW) {
            const double d = lane < SW ? row[lane & (SW - 1)] : lval;
            const unsigned long long b = (unsigned long long)__double_as_longlong(d);
            lo = (unsigned)b;
            hi = (unsigned)(b >> 32);
          } else if (lane == SW + 1) {
            lo = (unsigned)gr;
            hi = (unsigned)go;
          } else if (lane == SW + 2) {
            lo = (unsigned)lnan;
          }
          if (lane < SLOT) put(area + (long)slot * SLOT + lane, lo, hi, tag);
        };
        if (own) publish(prow, base / ROWS_PER_WG, lrow, corg[par]);
        if (ownj) publish(jr, P, j, jorg[par]);
        constexpr int U = 3;  // slots polled together
        for (int s0 = wave; s0 <= P; s0 += U * NW) {
          u64x2 e[U];
          unsigned long long t0 = 0;
          for (unsigned spin = 1;; ++spin) {
            bool done = true;
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (s0 + u * NW <= P && lane < SW + 3)
                e[u] = get(area + (long)(s0 + u * NW) * SLOT + lane);
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (s0 + u * NW <= P && lane < SW + 3) done = done && tagged(e[u], tag);
            if (__all(done)) break;
            // the flag and the clock cost as much as a poll: every 64th
            if (spin & 63) continue;
            if (t0 == 0) t0 = wall_clock64();
            if (__hip_atomic_load(cm.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
                wall_clock64() - t0 > kSpinTicks) {
              if (lane == 0) {
                __hip_atomic_store(cm.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                dead = 1;
              }
              break;
            }
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int s = s0 + u * NW;
            if (s > P) continue;
            if (lane < SW) gx[s][lane] = as_d(e[u]);
            if (lane == SW) gval[s] = as_d(e[u]);
            if (lane == SW + 1) {
              grow[s] = lo_i(e[u]);
              gorg[s] = hi_i(e[u]);
            }
            if (lane == SW + 2) gnan[s] = lo_i(e[u]);
          }
        }
        lds_barrier();
        if (dead) return;
        const int sl = lane < P ? lane : 0;
        const double gv = lane < P ? gval[sl] : -1.0;
        const int gr = grow[sl], gn = gnan[sl];
        const unsigned long long nb = __ballot(lane < P && gn >= 0);
        const int lo = nb ? 63 - __builtin_clzll(nb) : 0;  // the slab of the last NaN
        // the first of the largest, by the high word unless two agree in it
        const double kk = lane >= lo ? gv : -1.0;
        const unsigned h = kk >= 0.0 ? (unsigned)__double2hiint(kk) + 1u : 0u;
        const unsigned mh = wave_max_u(h);
        unsigned long long b = __ballot(h == mh);
        if (b & (b - 1)) b = __ballot(kk == wave_max_d(kk));
        const int gw = mh ? __builtin_ctzll(b) : lo;
        prow = gx[gw];
        jr = gx[P];
        r = __builtin_amdgcn_readlane(gr, gw);
        orgs = gorg + gw;
        orgj = gorg + P;
      }
      const double piv_val = prow[pos];
      const bool null_pivot = piv_val == 0.0;
      const bool swap = !null_pivot && r != j;
      if (base == 0 && t == 0) {
        pivs[j] = r - j;
        if (null_pivot && first_null < 0) first_null = j;
      }
      // the pivot row (row j when nothing moves) spread over each row of 16 lanes
      const double* const u = swap ? prow : jr;
      double u0 = u[lane & 15], u1 = u[16 + (lane & 15)];
      // ---- interchange rows j and r (skipped for a null pivot) ----
      if (swap) {
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
          const int rr = base + q * NT + t;
          if (!__any(rr == j || rr == r)) continue;
          const double* const w = rr == j ? prow : jr;
          if (rr == j || rr == r) {
#pragma unroll
            for (int c = 0; c < SW; ++c) v[q][c] = w[c];
            og[q] = rr == j ? *orgs : *orgj;
            x[q] = w[pos];
          }
        }
      }
      // ---- multipliers (scaled by the reciprocal, skipped for a null pivot
      // or a pivot of 1, as bl1_dinvscalv) and the rank-1 update ----
      const bool scale = !null_pivot && piv_val != 1.0;
      const double inv = scale ? 1.0 / piv_val : 1.0;
      double l[RQ], nl[RQ];
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        l[q] = scale ? x[q] * inv : x[q];
        nl[q] = -l[q];
      }
      // The finished rows 0..j are lanes of the first wave's first register
      // row: they keep their values by a zero multiplier or, should the pivot
      // row hold an infinity or NaN, by selects.
      bool select = false;
      if (ownj) {
        select = !__all(fabs(u0) < __builtin_inf() && fabs(u1) < __builtin_inf());
        nl[0] = lane > j ? nl[0] : 0.0;
        l[0] = lane > j ? l[0] : x[0];
      }
      if (select) {
        // the whole update of this wave's rows; what follows then adds zeros
#pragma unroll
        for (int c = 0; c < SW; ++c) {
          const bool live = c > pos && c < 8 * nlive;
          const double y0 = fma(nl[0], u[c], v[0][c]), y1 = fma(nl[1], u[c], v[1][c]);
          if (live && lane > j) v[0][c] = y0;
          if (live) v[1][c] = y1;
        }
        nl[0] = nl[1] = 0.0;
        u0 = fabs(u0) < __builtin_inf() ? u0 : 0.0;
        u1 = fabs(u1) < __builtin_inf() ? u1 : 0.0;
      }
      // (rows past M take garbage here and are never stored or searched)
      // a VALU result is a DPP source only two wait states later
      asm volatile("s_nop 1" : "+v"(u0), "+v"(u1));
#define FLA_LU_POS(I)                                 \
  case I:                                             \
    update_first<I>(v[0], u0, l[0], nl[0], x[0]);     \
    update_first<I>(v[1], u0, l[1], nl[1], x[1]);     \
    break;
      switch (pos) {
        FLA_LU_POS(0)
        FLA_LU_POS(1)
        FLA_LU_POS(2)
        FLA_LU_POS(3)
        FLA_LU_POS(4)
        FLA_LU_POS(5)
        FLA_LU_POS(6)
        FLA_LU_POS(7)
      }
#undef FLA_LU_POS
      constexpr auto seq = std::make_integer_sequence<int, 8>{};
      if (nlive > 1) {
        update_chunk<1>(v[0], u0, nl[0], seq);
        update_chunk<1>(v[1], u0, nl[1], seq);
      }
      if (nlive > 2) {
        update_chunk<2>(v[0], u1, nl[0], seq);
        update_chunk<2>(v[1], u1, nl[1], seq);
      }
      if (nlive > 3) {
        update_chunk<3>(v[0], u1, nl[0], seq);
        update_chunk<3>(v[1], u1, nl[1], seq);
      }
    }
    if (pos == 7) {  // the finished chunk goes to the end
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const double f = v[q][c];
          v[q][c] = v[q][c + 8];
          v[q][c + 8] = v[q][c + 16];
          v[q][c + 16] = v[q][c + 24];
          v[q][c + 24] = f;
        }
        x[q] = v[q][0];
      }
    }
  }
  __syncthreads();
  if (base == 0) {
    for (int j = t; j < W; j += NT) piv[k + j] = pivs[j];
    if (t == 0 && first_null >= 0) atomicCAS(info, -1, k + first_null);
  }
  asm volatile("" : "+s"(lda));  // the column offsets are not kept through the loop
  const int* const before = cm.orig[flip];
  int* const after = cm.orig[flip ^ 1];
  auto note = [](int* list, int dst, int src) {
    const int slot = atomicAdd(&list[0], 1);
    list[1 + 2 * slot] = dst;
    list[2 + 2 * slot] = src;
  };
  if (pmoved && base == 0 && t < first) {
    // rows finished by an earlier sub-panel keep the origin that it wrote
    const int po = cm.orig[((t / SW) & 1) ^ 1][t];
    if (po != t) note(pmoved, t, po);
  }
#pragma unroll
  for (int q = 0; q < RQ; ++q) {
    const int r = base + q * NT + t;
    if (r >= M) continue;
    double* const a = A + r;
    if (W == SW) {
#pragma unroll
      for (int c = 0; c < SW; ++c) a[(long)c * lda] = v[q][c];
    } else {
#pragma unroll
      for (int c = 0; c < SW; ++c)
        if (c < W) a[(long)c * lda] = v[q][c];
    }
    if (og[q] != r) note(cm.submoved, r, og[q]);
    const int pr = first + r, po = first == 0 ? og[q] : before[first + og[q]];
    after[pr] = po;
    if (pmoved && po != pr) note(pmoved, pr, po);
  }
}

// After a sub-panel of w columns at row and column c0 of the panel: its row
// moves (at most 64, one per lane) on the panel's columns [0, c0) and
// [c0 + w, c0 + w + nright), and on the latter U12 := inv(L11) A12 (unit
// lower), also written transposed to Ut.  One wave per column; lane i holds
// row i of the solve.
__global__ __launch_bounds__(256) void lu_sub_apply_kernel(int c0, int w, int nright,
                                                           double* __restrict__ A, long lda,
                                                           const int* __restrict__ moved,
                                                           double* __restrict__ Ut, long ldu) {
  __shared__ double top[4][SW];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ci = blockIdx.x * 4 + wave;
  if (ci >= c0 + nright) return;
  const bool right = ci >= c0;
  double* const rows = A + c0;  // row c0 of the panel
  double* const col = rows + (long)(right ? ci + w : ci) * lda;
  const int i = lane & (SW - 1);
  double l[SW], a = 0.0;
  if (right) {
    a = i < w ? col[i] : 0.0;
#pragma unroll
    for (int k = 0; k < SW - 1; ++k) l[k] = (k < i && i < w) ? rows[i + (long)(c0 + k) * lda] : 0.0;
    top[wave][i] = a;
  }
  const int cnt = moved[0];
  const bool mv = lane < cnt;
  const int dst = mv ? moved[1 + 2 * lane] : 0, src = mv ? moved[2 + 2 * lane] : 0;
  const double x = mv ? col[src] : 0.0;
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // every lane has read its row
  if (mv && (!right || dst >= w)) col[dst] = x;
  if (!right) return;
  if (mv && dst < w) top[wave][dst] = x;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  a = top[wave][i];
#pragma unroll
  for (int k = 0; k < SW - 1; ++k) {
    const double y = fma(-l[k], readlane_d(a, k), a);
    a = i > k ? y : a;
  }
  if (lane < w) {
    col[lane] = a;
    Ut[(ci - c0) + (long)lane * ldu] = a;
  }
}

// Applies the panel's row moves to columns [0, ncols) of the (M-row) block
// at A: new row q := old row orig, through registers (all reads of a
// workgroup's columns precede its writes).
constexpr int GC = 16;  // columns per workgroup
template <typename T>
__global__ __launch_bounds__(256) void lu_row_gather_kernel(int ncols, T* __restrict__ A, long lda,
                                                            const int* __restrict__ moved) {
  const int cnt = moved[0];
  const int c0 = blockIdx.x * GC;
  T val[GC];
  const int t = threadIdx.x;
  // cnt <= 2 * PW = 256: one pair per thread.
  int dst = -1, src = -1;
  if (t < cnt) {
    dst = moved[1 + 2 * t];
    src = moved[2 + 2 * t];
  }
  if (src >= 0) {
#pragma unroll
    for (int c = 0; c < GC; ++c)
      val[c] = (c0 + c < ncols) ? A[(long)src + (long)(c0 + c) * lda] : T(0);
  }
  __syncthreads();
  if (dst >= 0) {
#pragma unroll
    for (int c = 0; c < GC; ++c)
      if (c0 + c < ncols) A[(long)dst + (long)(c0 + c) * lda] = val[c];
  }
}

// dst(j, l) := src(l, j) for an r x c block (32 x 32 tiles through LDS).
__global__ __launch_bounds__(256) void transpose_kernel(int r, int c, const double* __restrict__ src,
                                                        long lds, double* __restrict__ dst,
                                                        long ldd) {
  __shared__ double tile[32][33];
  const int l0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int q = ty; q < 32; q += 8) {
    const int l = l0 + tx, j = j0 + q;
    tile[q][tx] = (l < r && j < c) ? src[(long)l + (long)j * lds] : 0.0;
  }
  __syncthreads();
  for (int q = ty; q < 32; q += 8) {
    const int j = j0 + tx, l = l0 + q;
    if (l < r && j < c) dst[(long)j + (long)l * ldd] = tile[tx][q];
  }
}

__global__ void set_int_kernel(int* p, int v) { *p = v; }

}  // namespace

// Exchange area of the panel kernel (one, shared by every launch: the tags
// keep launches apart) and four move lists: a panel must not reset a list
// that row gathers still queued on the update stream read (two per 256-column
// block, alternated between blocks; the 128-column path alternates two).
struct LuBufs {
  PanelComm cm;
  int* moved;
};

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

constexpr int MAX_ROWS = MAX_P * ROWS_PER_WG;
constexpr size_t kSlotBytes = sizeof(u64x2) * 2 * (MAX_P + 1) * SLOT;
constexpr size_t kOrigBytes = sizeof(int) * MAX_ROWS;
constexpr size_t kMovedBytes = sizeof(int) * (1 + 4 * PW);
static_assert(kSlotBytes + 2 * kOrigBytes + 16 * 256 + 5 * kMovedBytes < kUcLuBytes,
              "LU exchange area");

static void lu_carve(char* p, LuBufs (&b)[4]) {
  PanelComm cm;
  cm.slots = reinterpret_cast<u64x2*>(p);
  p += align256(kSlotBytes);
  for (int s = 0; s < 2; ++s) {
    cm.orig[s] = reinterpret_cast<int*>(p);
    p += align256(kOrigBytes);
  }
  cm.submoved = reinterpret_cast<int*>(p);
  p += align256(kMovedBytes);
  cm.err = nullptr;  // set by the caller
  for (int s = 0; s < 4; ++s) {
    b[s].cm = cm;
    b[s].moved = reinterpret_cast<int*>(p);
    p += align256(kMovedBytes);
  }
}

static __global__ void zero_kernel(unsigned long long* p, long n) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    p[i] = 0;
}

// Launch counter: its low 24 bits tag every exchange word of a launch.  When
// it wraps, the exchange area is cleared, so no word written 2^24 launches
// earlier can carry a current tag.
static unsigned g_lu_epoch = 0;

static int lu_panel(hipStream_t s, int M, int W, double* Ap, long lda, int k, int* piv,
                    int* dinfo, const LuBufs& b) {
  double* const Ut = fla_ctx().dlinv;  // transposed U12 of a sub-panel, at most 96 x 32
  void* tok = fla_stats_begin(s);
  for (int c0 = 0, sub = 0; c0 < W; c0 += SW, ++sub) {
    const int w = (W - c0) < SW ? (W - c0) : SW;
    const int m = M - c0, nright = W - c0 - w;
    double* As = Ap + (long)c0 + (long)c0 * lda;
    g_lu_epoch = (g_lu_epoch + 1) & 0xffffffu;
    if (g_lu_epoch == 0) {
      hipLaunchKernelGGL(zero_kernel, dim3(256), dim3(256), 0, s,
                         reinterpret_cast<unsigned long long*>(b.cm.slots),
                         (long)(kSlotBytes / 8));
      FLA_HIP_CHECK(hipGetLastError());
      g_lu_epoch = 1;
    }
    hipLaunchKernelGGL(lu_sub_kernel, dim3((m + ROWS_PER_WG - 1) / ROWS_PER_WG), dim3(NT), 0, s, m,
                       w, As, lda, k + c0, piv, dinfo, b.cm, sub & 1, c0,
                       nright == 0 ? b.moved : nullptr, g_lu_epoch << 8);
    FLA_HIP_CHECK(hipGetLastError());
    if (c0 + nright > 0) {
      hipLaunchKernelGGL(lu_sub_apply_kernel, dim3((c0 + nright + 3) / 4), dim3(256), 0, s, c0, w,
                         nright, Ap, lda, b.cm.submoved, Ut, (long)PW);
      FLA_HIP_CHECK(hipGetLastError());
    }
    if (nright > 0 && m > w)
      FLA_TRY(launch_dgemm_mfma(s, false, true, 0, m - w, nright, w, -1.0, As + w, lda, Ut, PW, 1.0,
                                As + (long)w + (long)w * lda, lda, nullptr));
  }
  double fl = 0.0;
  for (int j = 0; j < W; ++j) fl += (double)(M - j - 1) * (1.0 + 2.0 * (W - j - 1));
  fla_stats_end(s, tok, 2, fl);
  return FLA_HIP_OK;
}

static int lu_gather(hipStream_t s, int ncols, double* A, long lda, const int* moved) {
  if (ncols <= 0) return FLA_HIP_OK;
  // measurement kind 6: time of the interchange kernels (the moved bytes
  // depend on the pivots and are counted by the caller from them)
  void* tok = fla_stats_begin(s);
  hipLaunchKernelGGL(lu_row_gather_kernel<double>, dim3((ncols + GC - 1) / GC), dim3(256), 0, s,
                     ncols, A, lda, moved);
  fla_stats_end(s, tok, 6, 0.0);
  FLA_HIP_CHECK(hipGetLastError());
  return FLA_HIP_OK;
}

// Row interchanges, A12 solve and A22 update for columns [c0, c0+nc) after
// the panel at (k, kb).  U12 is copied transposed into Ut (ld ldu) so that
// the update's right operand is read with j contiguous, as in the Cholesky
// update (16-deep K chunks, coalesced loads).
static int lu_update_cols(hipStream_t s, int m, double* A, long lda, int k, int kb, int c0,
                          int nc, const int* moved, double* Ut, long ldu) {
  if (nc <= 0) return FLA_HIP_OK;
  double* Ak = A + (long)k;  // row k
  FLA_TRY(lu_gather(s, nc, Ak + (long)c0 * lda, lda, moved));
  double* A11 = A + (long)k + (long)k * lda;
  double* A12 = A + (long)k + (long)c0 * lda;
  FLA_TRY(launch_trsm_llnu(s, nc, kb, A11, lda, A12, lda));
  const int mr = m - k - kb;
  if (mr > 0) {
    hipLaunchKernelGGL(transpose_kernel, dim3((kb + 31) / 32, (nc + 31) / 32), dim3(256), 0, s, kb,
                       nc, A12, lda, Ut, ldu);
    FLA_HIP_CHECK(hipGetLastError());
    void* tok = fla_stats_begin(s);
    FLA_TRY(launch_dgemm_mfma(s, false, true, 0, mr, nc, kb, -1.0, A11 + kb, lda, Ut, ldu, 1.0,
                              A + (long)(k + kb) + (long)c0 * lda, lda, nullptr));
    fla_stats_end(s, tok, 1, 2.0 * mr * (double)nc * kb);
  }
  return FLA_HIP_OK;
}

// Blocks of one panel of width nb <= 128 (look-ahead over panels): the
// next panel's columns first, then the remaining columns.
static int lu_blocked1(FlaHipCtx& c, int m, int n, double* A, long lda, int* p, int* dinfo,
                       LuBufs (&bufs)[4], double* Ut, long ldu) {
  const int mn = m < n ? m : n;
  const int nb = c.lu_nb <= PW ? c.lu_nb : PW;
  hipStream_t su = c.s_update, sq = c.s_panel;
  int evi = 0;
  auto next_event = [&]() {
    hipEvent_t e = c.ev[evi];
    evi = (evi + 1) % FlaHipCtx::kEvents;
    return e;
  };
  hipEvent_t start = next_event();
  FLA_HIP_CHECK(hipEventRecord(start, su));
  FLA_HIP_CHECK(hipStreamWaitEvent(sq, start, 0));

  int step = 0;
  int kb = mn < nb ? mn : nb;
  FLA_TRY(lu_panel(sq, m, kb, A, lda, 0, p, dinfo, bufs[0]));
  for (int k = 0; k < mn; ++step) {
    const LuBufs& b = bufs[step & 1];
    hipEvent_t pd = next_event();
    FLA_HIP_CHECK(hipEventRecord(pd, sq));
    FLA_HIP_CHECK(hipStreamWaitEvent(su, pd, 0));
    const int k2 = k + kb;
    const int kb2 = (mn - k2) < nb ? (mn - k2) : nb;  // next panel width (0 at the end)
    // (a) the next panel's columns, so that panel can start
    FLA_TRY(lu_update_cols(su, m, A, lda, k, kb, k2, kb2 > 0 ? kb2 : 0, b.moved, Ut, ldu));
    hipEvent_t ready = next_event();
    FLA_HIP_CHECK(hipEventRecord(ready, su));
    // Interchanges on the columns left of the panel (off the next panel's path).
    FLA_TRY(lu_gather(su, k, A + (long)k, lda, b.moved));
    // (b) the remaining columns
    FLA_TRY(lu_update_cols(su, m, A, lda, k, kb, k2 + kb2, n - k2 - kb2, b.moved, Ut + kb2, ldu));
    if (kb2 <= 0) break;
    FLA_HIP_CHECK(hipStreamWaitEvent(sq, ready, 0));
    FLA_TRY(lu_panel(sq, m - k2, kb2, A + (long)k2 + (long)k2 * lda, lda, k2, p, dinfo,
                     bufs[(step + 1) & 1]));
    k = k2;
    kb = kb2;
  }
  hipEvent_t fin = next_event();
  FLA_HIP_CHECK(hipEventRecord(fin, sq));
  FLA_HIP_CHECK(hipStreamWaitEvent(su, fin, 0));
  return FLA_HIP_OK;
}

// The same for a 256-column block factored as two panels, a at (k, k) of
// width kba and b at (k + kba, k + kba) of width kbb: both panels'
// interchanges, U12 := inv(L11) A12 with L11 = [La 0; Lba Lb] (two 128
// solves around Bb -= Lba Xa), and one update with K = kba + kbb.
static int lu_update_cols2(hipStream_t s, int m, double* A, long lda, int k, int kba, int kbb,
                           int c0, int nc, const int* moved_a, const int* moved_b, double* Ut,
                           long ldu) {
  if (nc <= 0) return FLA_HIP_OK;
  if (kbb <= 0) return lu_update_cols(s, m, A, lda, k, kba, c0, nc, moved_a, Ut, ldu);
  const int kb = kba + kbb, kb1 = k + kba;
  FLA_TRY(lu_gather(s, nc, A + (long)k + (long)c0 * lda, lda, moved_a));
  FLA_TRY(lu_gather(s, nc, A + (long)kb1 + (long)c0 * lda, lda, moved_b));
  double* Xa = A + (long)k + (long)c0 * lda;
  double* Xb = A + (long)kb1 + (long)c0 * lda;
  FLA_TRY(launch_trsm_llnu(s, nc, kba, A + (long)k + (long)k * lda, lda, Xa, lda));
  FLA_TRY(launch_dgemm_mfma(s, false, false, 0, kbb, nc, kba, -1.0, A + (long)kb1 + (long)k * lda,
                            lda, Xa, lda, 1.0, Xb, lda, nullptr));
  FLA_TRY(launch_trsm_llnu(s, nc, kbb, A + (long)kb1 + (long)kb1 * lda, lda, Xb, lda));
  const int mr = m - k - kb;
  if (mr > 0) {
    hipLaunchKernelGGL(transpose_kernel, dim3((kb + 31) / 32, (nc + 31) / 32), dim3(256), 0, s, kb,
                       nc, Xa, lda, Ut, ldu);
    FLA_HIP_CHECK(hipGetLastError());
    void* tok = fla_stats_begin(s);
    FLA_TRY(launch_dgemm_mfma(s, false, true, 0, mr, nc, kb, -1.0, A + (long)(k + kb) + (long)k * lda,
                              lda, Ut, ldu, 1.0, A + (long)(k + kb) + (long)c0 * lda, lda, nullptr));
    fla_stats_end(s, tok, 1, 2.0 * mr * (double)nc * kb);
  }
  return FLA_HIP_OK;
}

// 256-column blocks ("pairs") of two 128-column panels A and B.  The update
// stream carries the chain: panel A; B's columns updated with A; panel B; B's
// interchanges on A's columns; the next pair's 256 columns updated with the
// pair (K = 256), after which the next panel A starts.  The bulk stream
// (s_update_lp: its CU mask leaves 32 CUs to the panel kernel) updates every
// column beyond the next pair (K = 256) and applies the pair's
// interchanges left of it, concurrently with the next pair's two panels; the
// chain waits for it only before the following pair's columns.  Ut holds the
// transposed U12 of the bulk update in rows [0, n) and of the chain's updates
// in rows [n, n + 256) (ld ldu >= n + 256).
static int lu_blocked2(FlaHipCtx& c, int m, int n, double* A, long lda, int* p, int* dinfo,
                       LuBufs (&bufs)[4], double* Ut, long ldu) {
  const int mn = m < n ? m : n;
  hipStream_t su = c.s_update, sb = c.s_update_lp, sq = c.s_panel;
  double* Utn = Ut + n;
  int evi = 0;
  auto next_event = [&]() {
    hipEvent_t e = c.ev[evi];
    evi = (evi + 1) % FlaHipCtx::kEvents;
    return e;
  };
  hipEvent_t start = next_event();
  FLA_HIP_CHECK(hipEventRecord(start, su));
  FLA_HIP_CHECK(hipStreamWaitEvent(sq, start, 0));
  FLA_HIP_CHECK(hipStreamWaitEvent(sb, start, 0));
  int blk = 0;
  int kba = mn < PW ? mn : PW;
  hipEvent_t bulk_done = nullptr;
  FLA_TRY(lu_panel(sq, m, kba, A, lda, 0, p, dinfo, bufs[0]));
  for (int k = 0;; ++blk) {
    const LuBufs& ba = bufs[2 * (blk & 1)];
    const LuBufs& bb = bufs[2 * (blk & 1) + 1];
    hipEvent_t pa = next_event();
    FLA_HIP_CHECK(hipEventRecord(pa, sq));
    FLA_HIP_CHECK(hipStreamWaitEvent(su, pa, 0));
    const int kb1 = k + kba;
    const int kbb = (mn - kb1) < PW ? (mn - kb1) : PW;
    if (kbb > 0) {
      FLA_TRY(lu_update_cols(su, m, A, lda, k, kba, kb1, kbb, ba.moved, Utn, ldu));
      hipEvent_t rb = next_event();
      FLA_HIP_CHECK(hipEventRecord(rb, su));
      FLA_HIP_CHECK(hipStreamWaitEvent(sq, rb, 0));
      FLA_TRY(lu_panel(sq, m - kb1, kbb, A + (long)kb1 + (long)kb1 * lda, lda, kb1, p, dinfo, bb));
      hipEvent_t pb = next_event();
      FLA_HIP_CHECK(hipEventRecord(pb, sq));
      FLA_HIP_CHECK(hipStreamWaitEvent(su, pb, 0));
      FLA_TRY(lu_gather(su, kba, A + (long)kb1 + (long)k * lda, lda, bb.moved));
    }
    const int k2 = kb1 + (kbb > 0 ? kbb : 0);  // the next pair
    const int nw = (mn - k2) < 2 * PW ? (mn - k2) : 2 * PW;
    if (bulk_done) FLA_HIP_CHECK(hipStreamWaitEvent(su, bulk_done, 0));
    FLA_TRY(lu_update_cols2(su, m, A, lda, k, kba, kbb, k2, nw > 0 ? nw : 0, ba.moved, bb.moved,
                            Utn, ldu));
    hipEvent_t ready = next_event();
    FLA_HIP_CHECK(hipEventRecord(ready, su));
    const int c0 = k2 + (nw > 0 ? nw : 0);
    FLA_HIP_CHECK(hipStreamWaitEvent(sb, ready, 0));
    FLA_TRY(lu_update_cols2(sb, m, A, lda, k, kba, kbb, c0, n - c0, ba.moved, bb.moved, Ut, ldu));
    FLA_TRY(lu_gather(sb, k, A + (long)k, lda, ba.moved));
    if (kbb > 0) FLA_TRY(lu_gather(sb, k, A + (long)kb1, lda, bb.moved));
    bulk_done = next_event();
    FLA_HIP_CHECK(hipEventRecord(bulk_done, sb));
    if (nw <= 0) break;
    const int kbn = nw < PW ? nw : PW;
    FLA_HIP_CHECK(hipStreamWaitEvent(sq, ready, 0));
    FLA_TRY(lu_panel(sq, m - k2, kbn, A + (long)k2 + (long)k2 * lda, lda, k2, p, dinfo,
                     bufs[2 * ((blk + 1) & 1)]));
    k = k2;
    kba = kbn;
  }
  hipEvent_t fin = next_event();
  FLA_HIP_CHECK(hipEventRecord(fin, sq));
  FLA_HIP_CHECK(hipStreamWaitEvent(su, fin, 0));
  FLA_HIP_CHECK(hipStreamWaitEvent(su, bulk_done, 0));
  return FLA_HIP_OK;
}

extern "C" int fla_hip_dgetrf(int m, int n, double* A, int lda, int* p, int* info) {
  FLA_USER_STREAM_SCOPE;
  FLA_TRY(fla_ensure_ready());
  if (m < 0 || n < 0 || lda < (m > 1 ? m : 1)) return FLA_HIP_EARG;
  *info = kSuccess;
  const int mn = m < n ? m : n;
  if (mn == 0) return FLA_HIP_OK;
  FlaHipCtx& c = fla_ctx();
  const int Pmax = (m + ROWS_PER_WG - 1) / ROWS_PER_WG;
  // Every panel workgroup must be resident at once (one per CU at most).
  if (Pmax > c.num_cus || Pmax > MAX_P) {
    std::fprintf(stderr, "libflame_amd: dgetrf supports m <= %d on this device\n", MAX_ROWS);
    return FLA_HIP_EARG;
  }
  // exchange area in the uncached region, laid out for MAX_P workgroups
  LuBufs bufs[4];
  lu_carve(c.uc, bufs);
  // transposed U12 of a step: (n + 2 PW) x 2 PW, ld n + 2 PW
  void* wut = nullptr;
  const long ldu = (long)n + 2 * PW;
  FLA_TRY(fla_workspace((size_t)ldu * 2 * PW * sizeof(double), &wut));
  double* Ut = static_cast<double*>(wut);
  int* dinfo = c.dscratch;
  int* derr = c.dscratch + 4;  // one wait-failure flag for the whole factorization
  for (auto& b : bufs) b.cm.err = derr;
  hipStream_t su = c.s_update, sq = c.s_panel;
  hipLaunchKernelGGL(set_int_kernel, dim3(1), dim3(1), 0, su, dinfo, kSuccess);
  hipLaunchKernelGGL(set_int_kernel, dim3(1), dim3(1), 0, su, derr, 0);
  if (c.lu_nb > PW) {
    FLA_TRY(lu_blocked2(c, m, n, A, lda, p, dinfo, bufs, Ut, ldu));
  } else {
    FLA_TRY(lu_blocked1(c, m, n, A, lda, p, dinfo, bufs, Ut, ldu));
  }
  int h[2] = {kSuccess, 0};
  FLA_HIP_CHECK(hipMemcpyAsync(&h[0], dinfo, sizeof(int), hipMemcpyDeviceToHost, su));
  FLA_HIP_CHECK(hipMemcpyAsync(&h[1], derr, sizeof(int), hipMemcpyDeviceToHost, su));
  FLA_HIP_CHECK(hipStreamSynchronize(su));
  fla_stats_harvest();
  if (h[1] != 0) return FLA_HIP_ESPIN;
  *info = h[0];
  return FLA_HIP_OK;
}

// ---- building blocks of the reduced-precision LU (fla_hip_mixed.hip) ----------

static LuBufs g_mp_bufs[4];

int fla_lu_panel_setup(int m, int* derr) {
  FlaHipCtx& c = fla_ctx();
  const int Pmax = (m + ROWS_PER_WG - 1) / ROWS_PER_WG;
  if (Pmax > c.num_cus || Pmax > MAX_P) {
    std::fprintf(stderr, "libflame_amd: the LU panel supports m <= %d on this device\n",
                 MAX_ROWS);
    return FLA_HIP_EARG;
  }
  lu_carve(c.uc, g_mp_bufs);
  for (auto& b : g_mp_bufs) b.cm.err = derr;
  return FLA_HIP_OK;
}

int fla_lu_panel_run(hipStream_t s, int set, int M, int W, double* Ap, long lda, int k, int* piv,
                     int* dinfo) {
  if (W > PW) return FLA_HIP_EARG;
  return lu_panel(s, M, W, Ap, lda, k, piv, dinfo, g_mp_bufs[set & 1]);
}

int fla_lu_gather_rows(hipStream_t s, int set, int ncols, double* A, long lda) {
  return lu_gather(s, ncols, A, lda, g_mp_bufs[set & 1].moved);
}

int fla_lu_gather_rows_f(hipStream_t s, int set, int ncols, float* A, long lda) {
  if (ncols <= 0) return FLA_HIP_OK;
  hipLaunchKernelGGL(lu_row_gather_kernel<float>, dim3((ncols + GC - 1) / GC), dim3(256), 0, s,
                     ncols, A, lda, g_mp_bufs[set & 1].moved);
  FLA_HIP_CHECK(hipGetLastError());
  return FLA_HIP_OK;
}
