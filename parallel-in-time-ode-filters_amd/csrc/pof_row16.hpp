// Scan combines with one matrix row per lane and sixteen lanes per worker (CDNA3/4, D <= 16).
//
// A worker is one DPP row: the 16 lanes l & ~15 .. l | 15 of a wavefront, four workers to a
// wavefront.  Lane r < D holds row r of every matrix of the element in registers.  What one lane
// needs of another's row arrives as the broadcast operand of the multiply-add that uses it
// (v_fmac_f64_dpp with row_newbcast: the one DPP control that 64-bit operations take, at the
// rate of a plain v_fma_f64: 3.97 and 4.18 ns per operation of one wave, 2.3 ns and 2.3 ns at four
// waves per SIMD), so nothing passes through LDS and no worker waits for another.  The scalar part
// of a Householder pivot (square root, reciprocal, selects) is issued once for the wavefront's four
// combines.
//
// Against rows split over two lanes of a whole-wavefront worker, with each pivot row passed through
// LDS and every lane repeating the pivot's scalar part: about 5,300 instructions per combine became
// about 4,300 per four (5,100 with a wait in front of every group and groups of at most eight), and at
// D = 12 a level of 32,768 combines went from 364 to 91 us (up) and from 205 to 61 us (down), the latency
// of one combine from 19 to 13 us and from 13 to 9.5 us.  A narrow level is bound by the instructions of one combine
// in order (a wave issues an FP64 operation every 8.5 to 9 cycles).  A wide one has two waves per SIMD (221 registers) and
// takes 2.5 ns per instruction, against the 1.67 ns of the FP64 peak: the counters show the vector ALUs 46 to 50 % busy
// and 12 of 16 lanes hold a row at D = 12; what holds the two waves back from there is not known.
//
// Lanes r >= D of a row repeat row 0; only lanes r < D are ever the source of a broadcast or store.
// A whole row is active or not (a worker past the end returns as a whole), so a broadcast never
// reads an inactive lane.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "pof_core.hpp"
#include "pof_engine.hpp"

#pragma clang fp contract(off)

namespace pof {
namespace r16 {

constexpr int kRow = 16;            // lanes per worker
constexpr int kBlock = 64;          // threads per block of the element kernels: one wavefront
constexpr int kPerBlock = kBlock / kRow;
constexpr int kStageBlock = kStageWorkers * kRow;  // threads per block of the scan stages: four wavefronts

// ------------------------------------------------------------- broadcasts
__device__ double update_dpp_f64(double, double, int, int, int, bool) __asm("llvm.amdgcn.update.dpp.f64");

// Lane L's value in every lane of its row.
template <int L>
__device__ __forceinline__ double bcast(double v) {
  return update_dpp_f64(v, v, 0x150 + L, 0xf, 0xf, true);
}

// y += (lane l's p) * x.  A DPP operand must not have been written by the two instructions before
// (the hardware does not wait for it and the compiler does not look into an asm statement): each group
// begins with two instructions that write none of its DPP operands, or with s_nop 1, which costs a wavefront
// as much as a multiply-add.  Within a group no source is a result.  Results are early clobbers: an input
// that holds the same value as a result's initial one (two zeros) must not share its register.
#define POF_FMAC(y, p, x, l) \
  "v_fmac_f64_dpp %[" #y "], %[" #p "], " x " row_newbcast:%[" #l "] row_mask:0xf bank_mask:0xf\n"

// M(0) M(1) ... and M(0), M(1), ... of the group sizes
#define POF_SEQ1(M) M(0)
#define POF_SEQ2(M) POF_SEQ1(M) M(1)
#define POF_SEQ3(M) POF_SEQ2(M) M(2)
#define POF_SEQ4(M) POF_SEQ3(M) M(3)
#define POF_SEQ5(M) POF_SEQ4(M) M(4)
#define POF_SEQ6(M) POF_SEQ5(M) M(5)
#define POF_SEQ7(M) POF_SEQ6(M) M(6)
#define POF_SEQ8(M) POF_SEQ7(M) M(7)
#define POF_SEQ9(M) POF_SEQ8(M) M(8)
#define POF_SEQ10(M) POF_SEQ9(M) M(9)
#define POF_SEQ11(M) POF_SEQ10(M) M(10)
#define POF_SEQ12(M) POF_SEQ11(M) M(11)
#define POF_SEQ13(M) POF_SEQ12(M) M(12)
#define POF_SEQ14(M) POF_SEQ13(M) M(13)
#define POF_SEQ15(M) POF_SEQ14(M) M(14)
#define POF_SEQ16(M) POF_SEQ15(M) M(15)
#define POF_CSV1(M) M(0)
#define POF_CSV2(M) POF_CSV1(M), M(1)
#define POF_CSV3(M) POF_CSV2(M), M(2)
#define POF_CSV4(M) POF_CSV3(M), M(3)
#define POF_CSV5(M) POF_CSV4(M), M(4)
#define POF_CSV6(M) POF_CSV5(M), M(5)
#define POF_CSV7(M) POF_CSV6(M), M(6)
#define POF_CSV8(M) POF_CSV7(M), M(7)
#define POF_CSV9(M) POF_CSV8(M), M(8)
#define POF_CSV10(M) POF_CSV9(M), M(9)
#define POF_CSV11(M) POF_CSV10(M), M(10)
#define POF_CSV12(M) POF_CSV11(M), M(11)
#define POF_CSV13(M) POF_CSV12(M), M(12)
#define POF_CSV14(M) POF_CSV13(M), M(13)
#define POF_CSV15(M) POF_CSV14(M), M(14)
#define POF_CSV16(M) POF_CSV15(M), M(15)
// CASE(n) for the group sizes
#define POF_CASES(CASE)                                                                                            \
  CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) \
      CASE(15) CASE(16)
// the parity of a group's index
#define POF_PAR0 "0"
#define POF_PAR1 "1"
#define POF_PAR2 "0"
#define POF_PAR3 "1"
#define POF_PAR4 "0"
#define POF_PAR5 "1"
#define POF_PAR6 "0"
#define POF_PAR7 "1"
#define POF_PAR8 "0"
#define POF_PAR9 "1"
#define POF_PAR10 "0"
#define POF_PAR11 "1"
#define POF_PAR12 "0"
#define POF_PAR13 "1"
#define POF_PAR14 "0"
#define POF_PAR15 "1"
#define POF_PAR(i) POF_PAR##i
constexpr int kGroup = 16;  // largest group
#define POF_Y(i) [y##i] "+&v"(y[i])
#define POF_P(i) [p##i] "v"(p[i])
#define POF_Q(i) [q##i] "v"(q[i])
#define POF_L(i) [l##i] "n"(L + i)

// y[c] += bcast_L(p[c]) x, c < N
template <int L, int N>
__device__ __forceinline__ void fma_rows(double* y, const double* p, double x) {
  if constexpr (N > kGroup) {
    fma_rows<L, kGroup>(y, p, x);
    fma_rows<L, N - kGroup>(y + kGroup, p + kGroup, x);
  }
#define POF_OP(i) POF_FMAC(y##i, p##i, "%[x]", l)
#define POF_CASE(n)      \
  if constexpr (N == n)  \
    asm volatile("s_nop 1\n" POF_SEQ##n(POF_OP) : POF_CSV##n(POF_Y) : POF_CSV##n(POF_P), [x] "v"(x), [l] "n"(L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
}

// y[c] += bcast_{L + c}(p) x, c < N
template <int L, int N>
__device__ __forceinline__ void fma_lanes(double* y, double p, double x) {
#define POF_OP(i) POF_FMAC(y##i, p, "%[x]", l##i)
#define POF_CASE(n)      \
  if constexpr (N == n)  \
    asm volatile("s_nop 1\n" POF_SEQ##n(POF_OP) : POF_CSV##n(POF_Y) : [p] "v"(p), [x] "v"(x), POF_CSV##n(POF_L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
}

// x *= d, then y[c] -= bcast_{L + c}(p) x, c < N
template <int L, int N>
__device__ __forceinline__ void scale_fma_lanes(double& x, double d, double* y, double p) {
  if constexpr (N == 0) x *= d;
#define POF_OP(i) POF_FMAC(y##i, p, "-%[x]", l##i)
#define POF_CASE(n)                                                             \
  if constexpr (N == n)                                                         \
    asm volatile("v_mul_f64 %[x], %[x], %[d]\ns_nop 0\n" POF_SEQ##n(POF_OP)     \
                 : [x] "+&v"(x), POF_CSV##n(POF_Y)                              \
                 : [p] "v"(p), [d] "v"(d), POF_CSV##n(POF_L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
}

// sum_c bcast_L(p[c]) p[c], c < N: even and odd c in a sum each (the second sum's zero stands where a wait would)
template <int L, int N>
__device__ __forceinline__ double dot_self(const double* p) {
  double s = 0.0, o;
#define POF_OP(i)                                                                                       \
  "v_fmac_f64_dpp %[s" POF_PAR(i) "], %[p" #i "], %[p" #i "] row_newbcast:%[l] row_mask:0xf bank_mask:0xf\n"
#define POF_CASE(n)                                                                                            \
  if constexpr (N == n)                                                                                        \
    asm volatile("v_mov_b64 %[s0], 0\nv_mov_b64 %[s1], 0\n" POF_SEQ##n(POF_OP) "v_add_f64 %[s0], %[s0], %[s1]\n" \
                 : [s0] "=&v"(s), [s1] "=&v"(o)                                                                \
                 : POF_CSV##n(POF_P), [l] "n"(L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
  if constexpr (N > kGroup) {
    s = dot_self<L, kGroup>(p);
    s += dot_self<L, N - kGroup>(p + kGroup);
  }
  return s;
}

// s = sum_c bcast_L(p[c]) p[c], t = sum_c bcast_L(p[c]) q[c], c < N
template <int L, int N>
__device__ __forceinline__ void dot_pair(double& s, double& t, const double* p, const double* q) {
  if constexpr (N == 0) s = t = 0.0;
#define POF_OP(i) POF_FMAC(s, p##i, "%[p" #i "]", l) POF_FMAC(t, p##i, "%[q" #i "]", l)
#define POF_CASE(n)                                                             \
  if constexpr (N == n)                                                         \
    asm volatile("v_mov_b64 %[s], 0\nv_mov_b64 %[t], 0\n" POF_SEQ##n(POF_OP)    \
                 : [s] "=&v"(s), [t] "=&v"(t)                                   \
                 : POF_CSV##n(POF_P), POF_CSV##n(POF_Q), [l] "n"(L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
  if constexpr (N > kGroup) {
    double s2, t2;
    dot_pair<L, kGroup>(s, t, p, q);
    dot_pair<L, N - kGroup>(s2, t2, p + kGroup, q + kGroup);
    s += s2;
    t += t2;
  }
}

// sum_c bcast_L(p[c]) q[c], c < N
template <int L, int N>
__device__ __forceinline__ double dot_rows(const double* p, const double* q) {
  double s;
#define POF_OP(i) POF_FMAC(s, p##i, "%[q" #i "]", l)
#define POF_CASE(n)                                                \
  if constexpr (N == n)                                            \
    asm volatile("v_mov_b64 %[s], 0\ns_nop 0\n" POF_SEQ##n(POF_OP) \
                 : [s] "=&v"(s)                                    \
                 : POF_CSV##n(POF_P), POF_CSV##n(POF_Q), [l] "n"(L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
  return s;
}

// t = rb (a + sc dot), y[c] -= bcast_L(p[c]) t, c < N: a reflector applied to the tail of other rows
// (see Pivot).  Returns t.
template <int L, int N>
__device__ __forceinline__ double reflect_rows(double* y, const double* p, double rb, double sc, double dot, double a) {
  double t;
  if constexpr (N == 0 || N > kGroup) t = rb * fma(sc, dot, a);
#define POF_OP(i) POF_FMAC(y##i, p##i, "-%[t]", l)
#define POF_CASE(n)                                                                                           \
  if constexpr (N == n)                                                                                       \
    asm volatile("v_fma_f64 %[t], %[sc], %[dot], %[a]\nv_mul_f64 %[t], %[rb], %[t]\n" POF_SEQ##n(POF_OP)      \
                 : [t] "=&v"(t), POF_CSV##n(POF_Y)                                                            \
                 : POF_CSV##n(POF_P), [sc] "v"(sc), [dot] "v"(dot), [a] "v"(a), [rb] "v"(rb), [l] "n"(L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
  if constexpr (N > kGroup) fma_rows<L, N>(y, p, -t);
  return t;
}

// The same to the tails of the rows of lane L's own set (its values feed the products before they change)
template <int L, int N>
__device__ __forceinline__ double reflect_self(double* y, double rb, double sc, double dot, double a) {
  double t;
  if constexpr (N == 0) t = rb * fma(sc, dot, a);
#define POF_OP(i) POF_FMAC(y##i, y##i, "-%[t]", l)
#define POF_CASE(n)                                                                                           \
  if constexpr (N == n)                                                                                       \
    asm volatile("v_fma_f64 %[t], %[sc], %[dot], %[a]\nv_mul_f64 %[t], %[rb], %[t]\n" POF_SEQ##n(POF_OP)      \
                 : [t] "=&v"(t), POF_CSV##n(POF_Y)                                                            \
                 : [sc] "v"(sc), [dot] "v"(dot), [a] "v"(a), [rb] "v"(rb), [l] "n"(L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
  if constexpr (N > kGroup) {
    t = reflect_self<L, kGroup>(y, rb, sc, dot, a);
    const double t2 = reflect_self<L, N - kGroup>(y + kGroup, rb, sc, dot, a);
    (void)t2;  // the same value
  }
  return t;
}

// y[c] -= bcast_L(y[c]) t, c < N (lane L's own values feed the products before they change)
template <int L, int N>
__device__ __forceinline__ void fnma_self(double* y, double t) {
#define POF_OP(i) POF_FMAC(y##i, y##i, "-%[t]", l)
#define POF_CASE(n)     \
  if constexpr (N == n) \
    asm volatile("s_nop 1\n" POF_SEQ##n(POF_OP) : POF_CSV##n(POF_Y) : [t] "v"(t), [l] "n"(L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
  if constexpr (N > kGroup) {
    fnma_self<L, kGroup>(y, t);
    fnma_self<L, N - kGroup>(y + kGroup, t);
  }
}

// init + sum_{k < N} bcast_k(v) x[k]: a row (or, of a transposed matrix, a column) times a vector whose
// entry k sits in lane k
template <int N>
__device__ __forceinline__ double dot_lanes(const double* x, double v, double init = 0.0) {
  constexpr int L = 0;
  const double* q = x;
  double s = init;
#define POF_OP(i) POF_FMAC(s, v, "%[q" #i "]", l##i)
#define POF_CASE(n)      \
  if constexpr (N == n)  \
    asm volatile("s_nop 1\n" POF_SEQ##n(POF_OP) : [s] "+&v"(s) : [v] "v"(v), POF_CSV##n(POF_Q), POF_CSV##n(POF_L));
  POF_CASES(POF_CASE)
#undef POF_CASE
#undef POF_OP
  return s;
}

// ------------------------------------------------------------- compile-time loops
template <int I, int N, class F>
__device__ __forceinline__ void unroll(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unroll<I + 1, N>(f);
  }
}
template <int I, int N, class F>  // I, I - 1, ..., N
__device__ __forceinline__ void unroll_down(F&& f) {
  if constexpr (I >= N) {
    f(std::integral_constant<int, I>{});
    unroll_down<I - 1, N>(f);
  }
}

// x is formed here (not recomputed from its operands where it is used, which would hold all of them)
__device__ __forceinline__ void keep(double& x) { asm volatile("" : "+v"(x)); }

// ------------------------------------------------------------- products
// y[c] += sum_k x[k] (row k of B)[c] over the columns c < min(N, k + LOW) of row k (LOW = 1: B lower
// triangular; LOW >= N: full)
template <int K, int N, int LOW>
__device__ __forceinline__ void mul_rows(double* y, const double* x, const double* B) {
  unroll<0, K>([&](auto k) {
    constexpr int kk = decltype(k)::value;
    fma_rows<kk, (kk + LOW < N) ? kk + LOW : N>(y, B, x[kk]);
  });
}

// ------------------------------------------------------------- Householder pivot
// The scalar part of a pivot with entry alpha and squared tail sig, as LAPACK dlarfg:
// beta = -sign(alpha) sqrt(alpha^2 + sig), v = [1, tail / (alpha - beta)], tau = (beta - alpha) / beta.
// Applied to another row with entry a at the pivot and product `dot` with the tail:
//   w = a + dot / (alpha - beta),  entry -= tau w,  tail -= tau w / (alpha - beta) tail,
// and tau / (alpha - beta) = -1 / beta, so one reciprocal serves.
// rb = -1 / beta = sign(alpha) / norm, den = alpha - beta, sc = 1 / den.
struct Pivot {
  double beta, rb, den, sc;
};

// norm and 1 / norm of x > 0: the hardware's estimate y (about 2^-24) and one third-order step,
// e = 1 - x y^2, (1 - e)^(-1/2) = 1 + e / 2 + 3 e^2 / 8 + O(e^3): 2^-72 before rounding.  Rounded, over 4 million x from
// 1e-290 to 1e290: the norm within 0.75 ulp (mean 0.27), its reciprocal within 0.99 (0.28).  sqrt_rsqrt, which the D > 16
// kernels use, has 0.50 (0.25) and 1.61 (0.31): one step more for the norm, one less for the reciprocal.
__device__ __forceinline__ void norm_rnorm(double x, double& n, double& rn) {
  const double y = __builtin_amdgcn_rsq(x);
  const double g = x * y;
  const double e = fma(-g, y, 1.0);
  const double q = e * fma(e, 0.375, 0.5);
  n = fma(g, q, g);
  rn = fma(y, q, y);
}

// 1 / x for normal x: the estimate and one third-order step (1 + e + e^2); within 0.50 ulp over the same x
__device__ __forceinline__ double rcp3(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// A pivot whose tail cannot vanish.
__device__ __forceinline__ Pivot pivot_nz(double alpha, double sig) {
  Pivot p;
  double n, rn;
  norm_rnorm(fma(alpha, alpha, sig), n, rn);
  p.beta = -copysign(n, alpha);  // Fortran SIGN: honours the sign of -0.0
  p.den = alpha - p.beta;
  p.sc = rcp3(p.den);
  p.rb = copysign(rn, alpha);
  return p;
}

// Any pivot: a zero tail leaves the rows as they are (rb = 0; beta = alpha).
__device__ __forceinline__ Pivot pivot(double alpha, double sig, bool& nz) {
  nz = sig != 0.0;
  const double x = fma(alpha, alpha, sig);
  Pivot p;
  double n, rn;
  norm_rnorm(nz ? x : 1.0, n, rn);
  p.beta = -copysign(n, alpha);
  p.den = alpha - p.beta;
  p.sc = rcp3(p.den);
  p.rb = nz ? copysign(rn, alpha) : 0.0;
  return p;
}

// ------------------------------------------------------------- LQ, one row set
// Pivots 0 .. K - 1 of the LQ of a matrix of N columns a (rows in lanes 0 .. K - 1): on return a holds the
// lower triangle of the factor in its columns <= row (entries above are left over and not cleared).  The columns
// from B1 on are a second block, whose row r is zero beyond its column max(r, W2) (W2 = N: a full block, or none);
// so is the reflector of pivot r, and those columns are left out.
template <int K, int N, int B1 = N, int W2 = N>
__device__ __forceinline__ void lq1(double* a, int r) {
  unroll<0, K>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    constexpr int band = B1 + (i > W2 ? i : W2) + 1;
    constexpr int n = (band < N ? band : N) - 1 - i;
    if constexpr (n > 0) {  // a length-1 tail: H = I
      const double dot = dot_self<i, n>(a + i + 1);
      bool nz;
      const Pivot p = pivot(bcast<i>(a[i]), bcast<i>(dot), nz);
      const double t = reflect_self<i, n>(a + i + 1, p.rb, p.sc, dot, a[i]);
      a[i] = (r == i && nz) ? p.beta : fma(-p.den, t, a[i]);
    }
  });
}

// ------------------------------------------------------------- memory
// Row of N contiguous doubles (16-byte accesses where every row of an N-column matrix is aligned)
template <int N>
__device__ __forceinline__ void load_row16(double (&x)[N], const double* p) {
  if constexpr (N % 2 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 2) {
      const double2 v = *reinterpret_cast<const double2*>(p + i);
      x[i] = v.x;
      x[i + 1] = v.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = p[i];
  }
}
template <int N>
__device__ __forceinline__ void store_row16(double* p, const double* x) {
  if constexpr (N % 2 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 2) *reinterpret_cast<double2*>(p + i) = make_double2(x[i], x[i + 1]);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = x[i];
  }
}
// column r of an N x N matrix: the lanes of a row read one matrix row together
template <int N>
__device__ __forceinline__ void load_col16(double (&x)[N], const double* M, int r) {
#pragma unroll
  for (int k = 0; k < N; ++k) x[k] = M[k * N + r];
}
// the lower triangle of a factor, its strict upper part cleared
template <int N>
__device__ __forceinline__ void store_lower16(double* p, double* x, int r) {
#pragma unroll
  for (int c = 1; c < N; ++c) x[c] = (c > r) ? 0.0 : x[c];
  store_row16<N>(p, x);
}

// ------------------------------------------------------------- filter combine
// pof/parallel_filtsmooth/filter.py:117-142, as filter_combine() of pof_core.hpp: e = e1 o e2, e1
// earlier.  SO (state only): e1 is a prefix state (s1.m, s1.L) and (so.m, so.L) receives the result.
//
// DZ: columns of the elements' Z: d at a leaf level ([Zr | 0] stored as Zr), D above it (lower
// triangular).  Columns of zeros are left out of every sum and update (they add exact zeros); at a
// leaf level this leaves pivot i of the Xi factorisation max(d - 1 - i, 0) + i tail columns instead
// of D - 1 in each of its four passes.
//
// Xi = [[U1^T Z2, I], [Z2, 0]], rows 0 .. D - 1 (a) and D .. 2D - 1 (b) of a lane's two row sets.
// Column i of the second block is still the identity's when pivot i comes: it adds 1 to the pivot
// row's squared tail (so no tail vanishes) and its update is -tau w v_i without a product.
//
// PARTS: the results that this worker forms: U, (b, A), (eta, Z).  A second worker can form the rest at the same time
// from the same Xi, which both factor; the instructions of a result are the same either way.
constexpr int kPartU = 1, kPartA = 2, kPartZ = 4;
template <int D, int DZ, bool SO, int PARTS>
__device__ __forceinline__ void filter_combine(int r, const FiltArrays& x1, const StateArrays& s1, size_t i1,
                                               const FiltArrays& x2, size_t i2, const FiltArrays& y,
                                               const StateArrays& so, size_t o) {
  constexpr size_t DD = (size_t)D * D;
  constexpr bool kLeaf = DZ < D;
  constexpr bool pU = PARTS & kPartU, pA = PARTS & kPartA, pZ = !SO && (PARTS & kPartZ), pM = pU || pA;
  constexpr int kLow = kLeaf ? D : 1;  // Z2's row k holds columns < min(DZ, k + kLow)
  const bool act = r < D;
  const int rr = act ? r : 0;
  const double* U1 = (SO ? s1.L : x1.U) + i1 * DD;
  const double* A1 = SO ? nullptr : x1.A + i1 * DD;
  const double* Z1 = SO ? nullptr : x1.Z + i1 * DD;
  const double* A2 = x2.A + i2 * DD;
  const double* U2 = x2.U + i2 * DD;
  const double* Z2 = x2.Z + i2 * DD;

  // Reads are issued ahead of the phases that use them (the asm groups keep them in place), as far as the
  // registers hold them: all of them here (D <= 8), or those of the first two phases here and the rest half
  // way (D <= 12); beyond, each phase's at its head (more would spill).  A combine alone on its SIMD waits for
  // memory at each such point, five times in the last form: at D = 12 reading ahead took the 10 iterations over
  // 65,536 steps from 10.8 to 10.2 ms (with the shorter tail of an iteration), at D = 4 from 3.29 to 2.95 ms.
  constexpr bool kAll = D <= 8, kTwo = D <= 12;
  double u1t[D], z2[DZ], z2t[SO ? 1 : D], w[D], u1[D], u2[D], ar[SO ? 1 : D], a1t[SO ? 1 : D], z1[SO ? 1 : DZ];
  auto load_z = [&](double (&z)[DZ], const double* Z) {
    if constexpr (kLeaf) {
#pragma unroll
      for (int c = 0; c < DZ; ++c) z[c] = Z[rr * DZ + c];
    } else {
      load_row16<DZ>(z, Z + rr * D);
    }
  };
  auto load_rest1 = [&] {
    if constexpr (pU) load_row16<D>(u2, U2 + rr * D);
    if constexpr (pA && !SO) load_row16<D>(ar, A1 + rr * D);
  };
  auto load_rest2 = [&] {
    if constexpr (pZ) {
      load_col16<D>(a1t, A1, rr);
      load_z(z1, Z1);
    }
  };
  const double b1r = (SO ? s1.m : x1.b)[i1 * D + rr];
  const double eta2r = x2.eta[i2 * D + rr];
  load_col16<D>(u1t, U1, rr);
  load_z(z2, Z2);
  if constexpr (pZ) {
    if constexpr (kLeaf) {
      const int rz = (r < DZ) ? r : 0;  // lanes past the last column hold no entry of Z2^T b1
#pragma unroll
      for (int k = 0; k < D; ++k) z2t[k] = Z2[k * DZ + rz];
    } else {
      load_col16<D>(z2t, Z2, rr);
    }
  }
  if constexpr (kTwo && pM) {
    load_row16<D>(w, A2 + rr * D);
    load_row16<D>(u1, U1 + rr * D);
  }
  const double b2r = pA ? x2.b[i2 * D + rr] : 0.0;
  const double eta1r = pZ ? x1.eta[i1 * D + rr] : 0.0;
  if constexpr (kAll) {
    load_rest1();
    load_rest2();
  }

  double s2 = 0.0, uu = 0.0;
  double x11[D], x21[D], b[DZ + D], rd = 0.0;  // Xi11, Xi21; rd: 1 / Xi11[r][r] in lane r
  if constexpr (pZ) {
    // s2 = eta2 - Z2 (Z2^T b1), uu = U1^T s2
    const double t = dot_lanes<D>(z2t, b1r);
    s2 = eta2r - dot_lanes<DZ>(z2, t);
    uu = dot_lanes<D>(u1t, s2);
  }
  const double u = pA ? dot_lanes<D>(u1t, eta2r) : 0.0;
  {
    double a[DZ + D];
    zero(a);
    mul_rows<D, DZ, kLow>(a, u1t, z2);
#pragma unroll
    for (int c = 0; c < DZ; ++c) b[c] = z2[c];
    unroll<0, D>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      // the tail: columns i + 1 .. DZ - 1 of the first block, 0 .. i - 1 of the second
      constexpr int c0 = (i < DZ) ? i + 1 : DZ, n = DZ + i - c0;
      double da, db;
      dot_pair<i, n>(da, db, a + c0, b + c0);
      const double sig = bcast<i>(da) + 1.0;
      double ta, tb, rp;
      if constexpr (i < DZ) {
        const Pivot p = pivot_nz(bcast<i>(a[i]), sig);
        tb = reflect_rows<i, n>(b + c0, a + c0, p.rb, p.sc, db, b[i]);
        ta = reflect_self<i, n>(a + c0, p.rb, p.sc, da, a[i]);
        x11[i] = fma(-p.den, ta, a[i]);
        x21[i] = fma(-p.den, tb, b[i]);
        rp = -p.rb;
      } else {
        // column i of the first block is zero: alpha = 0, den = norm, beta = -norm
        double nr, rn;
        norm_rnorm(sig, nr, rn);
        tb = reflect_rows<i, n>(b + c0, a + c0, rn, rn, db, 0.0);
        ta = reflect_self<i, n>(a + c0, rn, rn, da, 0.0);
        x11[i] = -rn * da;
        x21[i] = -rn * db;
        rp = -rn;
      }
      rd = (r == i) ? rp : rd;
      keep(rd);
      keep(x11[i]);
      keep(x21[i]);
      a[DZ + i] = -ta;
      b[DZ + i] = -tb;
    });
  }
  double* x22 = b + DZ;
  if constexpr (!kTwo && pM) {
    load_row16<D>(w, A2 + rr * D);
    load_row16<D>(u1, U1 + rr * D);
  } else if constexpr (kTwo && !kAll) {
    load_rest1();
  }

  // MT = A2 U1 Xi11^-T, W = A2 - MT Xi21^T, b = W (b1 + U1 u) + b2
  double mt[2 * D], bo = 0.0;
  if constexpr (pM) {
    zero(mt);
    mul_rows<D, D, 1>(mt, w, u1);
    double sv = 0.0;
    if constexpr (pA) sv = dot_lanes<D>(u1, u, b1r);
    unroll<0, D>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      scale_fma_lanes<j + 1, D - 1 - j>(mt[j], bcast<j>(rd), mt + j + 1, x11[j]);
    });
    if constexpr (pA) {
      unroll<0, D>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        fma_lanes<0, D>(w, x21[j], -mt[j]);
      });
      bo = dot_lanes<D>(w, sv, b2r);
    }
  }

  double s3 = 0.0;
  if constexpr (pZ) {
    // eta = A1^T (s2 - Xi21 Xi11^-1 U1^T s2) + eta1
    double w2 = 0.0;
    {
      double x = uu;
      unroll<0, D>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const double wj = bcast<j>(x * rd);
        w2 = (r == j) ? wj : w2;
        x = fma(-x11[j], wj, x);
      });
    }
    s3 = s2 - dot_lanes<D>(x21, w2);
  }
  if constexpr (kTwo && !kAll) load_rest2();
  if constexpr (pA && !SO) {
    if constexpr (!kTwo) load_row16<D>(ar, A1 + rr * D);
    // A = W A1
    double a[D];
    zero(a);
    mul_rows<D, D, D>(a, w, ar);
    if (act) store_row16<D>(y.A + (o * D + r) * D, a);
  }
  if constexpr (pZ) {
    // Xi22 triangular, then Z = tria([A1^T Xi22 | Z1])
    lq1<D, D>(x22, r);
    if constexpr (!kTwo) load_rest2();
    double z[D + DZ];
    const double eo = dot_lanes<D>(a1t, s3, eta1r);
    if (act) y.eta[o * D + r] = eo;
    zero(z);
    mul_rows<D, D, 1>(z, a1t, x22);
#pragma unroll
    for (int c = 0; c < DZ; ++c) z[D + c] = z1[c];
    lq1<D, D + DZ, D, kLeaf ? DZ - 1 : 0>(z, r);
    if (act) store_lower16<D>(y.Z + (o * D + r) * D, z, r);
  }
  if constexpr (pA) {
    if (act) (SO ? so.m : y.b)[o * D + r] = bo;
  }
  // U = tria([MT | U2])
  if constexpr (pU) {
    if constexpr (!kTwo) load_row16<D>(u2, U2 + rr * D);
#pragma unroll
    for (int c = 0; c < D; ++c) mt[D + c] = u2[c];
    lq1<D, 2 * D, D, 0>(mt, r);
    if (act) store_lower16<D>((SO ? so.L : y.U) + (o * D + r) * D, mt, r);
  }
}

// ------------------------------------------------------------- smoother combine
// pof/parallel_filtsmooth/smoother.py:53-63 under reverse=True, as smoother_combine() of pof_core.hpp:
// e1 is the aggregate later in time, (g, E, D) = (E2 g1 + g2, E2 E1, tria([E2 D1 | D2])); SO: (m, L) =
// (E2 m1 + g2, tria([E2 L1 | D2])).  wc = false: no factors (means-only iterations).
template <int D, bool SO>
__device__ __forceinline__ void smoother_combine(int r, const SmoArrays& x1, const StateArrays& s1, size_t i1,
                                                 const SmoArrays& x2, size_t i2, const SmoArrays& y,
                                                 const StateArrays& so, size_t o, bool wc) {
  constexpr size_t DD = (size_t)D * D;
  const bool act = r < D;
  const int rr = act ? r : 0;
  double e2[D], e1[SO ? 1 : D];
  load_row16<D>(e2, x2.E + i2 * DD + rr * D);
  if constexpr (!SO) load_row16<D>(e1, x1.E + i1 * DD + rr * D);
  const double g1 = (SO ? s1.m : x1.g)[i1 * D + rr];
  const double g = x2.g[i2 * D + rr] + dot_lanes<D>(e2, g1);
  if (act) (SO ? so.m : y.g)[o * D + r] = g;
  if constexpr (!SO) {
    double e[D];
    zero(e);
    mul_rows<D, D, D>(e, e2, e1);
    if (act) store_row16<D>(y.E + o * DD + r * D, e);
  }
  if (wc) {
    double d1[D], d2[D], t[2 * D];
    load_row16<D>(d1, (SO ? s1.L : x1.Dm) + i1 * DD + rr * D);
    load_row16<D>(d2, x2.Dm + i2 * DD + rr * D);
    zero(t);
    mul_rows<D, D, D>(t, e2, d1);  // the first aggregate's D may be a caller's factor, not triangular
#pragma unroll
    for (int c = 0; c < D; ++c) t[D + c] = d2[c];
    lq1<D, 2 * D, D, 0>(t, r);
    if (act) store_lower16<D>((SO ? so.L : y.Dm) + o * DD + r * D, t, r);
  }
}

// ------------------------------------------------------------- observation model
// Affine observation y = H x + c of one element, noise factor R (zero for EK1).  EK1 (Obs of
// pof_core.hpp): row i of H is hc[i][l] at the columns l q1 and hd[i] at column i q1 + 1, the same
// in every lane.  Otherwise lane i < d holds row i of the caller's H and R.
template <int D, int d, bool EK1>
struct ObsRow;

template <int D, int d>
struct ObsRow<D, d, true> {
  static constexpr int q1 = D / d;
  static constexpr int NR = 0;  // noise columns
  Obs<D, d, true> o;
  double c[d];
  // (the parameters are read where they are.  The dual numbers of the field are an array that its cases index at run time: with
  // three equations it takes 152 B of scratch per lane, with four 232 B, in every kernel that linearises.)
  __device__ __forceinline__ void load(const GroupArgs& g, int j, long long base, int k, int) {
    const double* lin = (g.cur[j] ? g.means1 : g.means0) + (size_t)base * D;
    o.load_at(g.kind[j], g.params + (size_t)j * kMaxParams, g.Pd + (size_t)j * D, lin + (size_t)(k + 1) * D);
#pragma unroll
    for (int i = 0; i < d; ++i) c[i] = o.c[i];
  }
  // at the mean's entries i q1
  __device__ __forceinline__ void load_entries(int kind, const double* params, const double* Pd, const double (&mi)[d]) {
    o.load_entries(kind, params, Pd, mi);
#pragma unroll
    for (int i = 0; i < d; ++i) c[i] = o.c[i];
  }
  __device__ __forceinline__ double r_at(int) const { return 0.0; }
  // out[c] += (H M)[r][c] for r < d, M's row j (columns < j + LOW) in lane j
  template <int LOW>
  __device__ __forceinline__ void times_rows(int r, const double (&M)[D], double (&out)[D]) const {
    unroll<0, d>([&](auto lc) {
      constexpr int l = decltype(lc)::value;
      double h = o.hc[0][l];
#pragma unroll
      for (int i = 1; i < d; ++i) h = (r == i) ? o.hc[i][l] : h;
      constexpr int n = (l * q1 + LOW < D) ? l * q1 + LOW : D;
      fma_rows<l * q1, n>(out, M, h);
    });
    unroll<0, d>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      constexpr int n = (i * q1 + 1 + LOW < D) ? i * q1 + 1 + LOW : D;
      fma_rows<i * q1 + 1, n>(out, M, (r == i) ? o.hd[i] : 0.0);
    });
  }
  // y[i] = c_i + (H v)_i, v's entry j in lane j
  __device__ __forceinline__ void predict(double v, double (&y)[d]) const {
    double p[d], n[d];
    unroll<0, d>([&](auto lc) {
      constexpr int l = decltype(lc)::value;
      p[l] = bcast<l * q1>(v);
      n[l] = bcast<l * q1 + 1>(v);
    });
#pragma unroll
    for (int i = 0; i < d; ++i) {
      double h = o.hc[i][0] * p[0];
#pragma unroll
      for (int l = 1; l < d; ++l) h = fma(o.hc[i][l], p[l], h);
      y[i] = c[i] + fma(o.hd[i], n[i], h);
    }
  }
  // y[i] = (H F)[i][r]
  __device__ __forceinline__ void times_col(const double* F, int r, double (&y)[d]) const {
    double p[d];
#pragma unroll
    for (int l = 0; l < d; ++l) p[l] = F[(l * q1) * D + r];
#pragma unroll
    for (int i = 0; i < d; ++i) {
      double h = o.hc[i][0] * p[0];
#pragma unroll
      for (int l = 1; l < d; ++l) h = fma(o.hc[i][l], p[l], h);
      y[i] = fma(o.hd[i], F[(i * q1 + 1) * D + r], h);
    }
  }
  // x[c] -= (K H M)[c] for the lane's row K of a gain
  __device__ __forceinline__ void sub_gain(const double (&K)[d], const double (&M)[D], double (&x)[D]) const {
    unroll<0, d>([&](auto lc) {
      constexpr int l = decltype(lc)::value;
      double h = 0.0;
#pragma unroll
      for (int i = 0; i < d; ++i) h = fma(K[i], o.hc[i][l], h);
      fma_rows<l * q1, D>(x, M, -h);
    });
    unroll<0, d>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      fma_rows<i * q1 + 1, D>(x, M, -(K[i] * o.hd[i]));
    });
  }
};

template <int D, int d>
struct ObsRow<D, d, false> {
  static constexpr int NR = d;
  double h[D], R[d], c[d];
  __device__ __forceinline__ void load(const GroupArgs& g, int, long long, int k, int r) {
    const int i = (r < d) ? r : 0;
    const double* H = g.Hx + ((size_t)k * d + i) * D;
#pragma unroll
    for (int j = 0; j < D; ++j) h[j] = (r < d) ? H[j] : 0.0;
#pragma unroll
    for (int j = 0; j < d; ++j) R[j] = (g.Rx && r < d) ? g.Rx[((size_t)k * d + i) * d + j] : 0.0;
#pragma unroll
    for (int j = 0; j < d; ++j) c[j] = g.cx[(size_t)k * d + j];
  }
  __device__ __forceinline__ double r_at(int j) const { return R[j]; }
  template <int LOW>
  __device__ __forceinline__ void times_rows(int, const double (&M)[D], double (&out)[D]) const {
    mul_rows<D, D, LOW>(out, h, M);
  }
  __device__ __forceinline__ void predict(double v, double (&y)[d]) const {
    const double s = dot_lanes<D>(h, v);
    unroll<0, d>([&](auto ic) { y[decltype(ic)::value] = c[decltype(ic)::value] + bcast<decltype(ic)::value>(s); });
  }
  __device__ __forceinline__ void times_col(const double* F, int r, double (&y)[d]) const {
    double f[D];
    load_col16<D>(f, F, r);
    unroll<0, d>([&](auto ic) { y[decltype(ic)::value] = dot_rows<decltype(ic)::value, D>(h, f); });
  }
  __device__ __forceinline__ void sub_gain(const double (&K)[d], const double (&M)[D], double (&x)[D]) const {
    double kh[D];
    zero(kh);
    unroll<0, d>([&](auto ic) { fma_rows<decltype(ic)::value, D>(kh, h, -K[decltype(ic)::value]); });
    mul_rows<D, D, D>(x, kh, M);
  }
};

// A d x d lower triangular factor held by lanes 0 .. d - 1 (row i in lane i), the same in every lane
// of the row: entries and reciprocal diagonal.
template <int d>
struct Small {
  double l[d][d], rd[d];
  template <int N>
  __device__ __forceinline__ void load(const double (&rows)[N]) {
    unroll<0, d>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      unroll<0, i + 1>([&](auto jc) { l[i][decltype(jc)::value] = bcast<i>(rows[decltype(jc)::value]); });
      rd[i] = 1.0 / l[i][i];
    });
  }
  // x = L^-1 x
  __device__ __forceinline__ void solve(double (&x)[d]) const {
#pragma unroll
    for (int j = 0; j < d; ++j) {
#pragma unroll
      for (int i = 0; i < j; ++i) x[j] = fma(-x[i], l[j][i], x[j]);
      x[j] *= rd[j];
    }
  }
  // x = L^-T x (the row vector x L^-1)
  __device__ __forceinline__ void solve_t(double (&x)[d]) const {
#pragma unroll
    for (int j = d - 1; j >= 0; --j) {
#pragma unroll
      for (int i = j + 1; i < d; ++i) x[j] = fma(-x[i], l[i][j], x[j]);
      x[j] *= rd[j];
    }
  }
};

// The first d pivots of the LQ of [[t], [n]]: d rows t (lanes 0 .. d - 1) and D rows n of NC columns each.  Leaves the
// factor of the first block row in t and its columns of the second in n[0 .. d - 1].
template <int d, int NC>
__device__ __forceinline__ void lq_obs(double (&t)[NC], double (&n)[NC], int r) {
  unroll<0, d>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    constexpr int nt = NC - 1 - i;
    double dt, dn;
    dot_pair<i, nt>(dt, dn, t + i + 1, n + i + 1);
    bool nz;
    const Pivot p = pivot(bcast<i>(t[i]), bcast<i>(dt), nz);
    const double tn = reflect_rows<i, nt>(n + i + 1, t + i + 1, p.rb, p.sc, dn, n[i]);
    const double tt = reflect_self<i, nt>(t + i + 1, p.rb, p.sc, dt, t[i]);
    t[i] = (r == i && nz) ? p.beta : fma(-p.den, tt, t[i]);
    n[i] = fma(-p.den, tn, n[i]);
  });
}

// ------------------------------------------------------------- filter element
// _get_element (pof/parallel_filtsmooth/filter.py:50-81) for element k, as filter_element() of
// pof_core.hpp; element 0 carries the prior (x0m, x0L), the others a zero one.  The element's
// Z = [Zr | 0] is stored as its d columns alone, rows packed ([D, d] at the element's place).
//
// Psi = tria([[H N1, R], [N1, 0]]): the d rows of the first block row in t, the D rows of the second
// in n.  The first d pivots leave Psi11 (t) and Psi21 (n's first d columns), the rest U = Psi22.
// Without noise the last d columns are zero throughout and are left out.
template <int D, int d, bool EK1>
__device__ __forceinline__ void filter_element(int r, const GroupArgs& g, int j, long long base, int k,
                                               const FiltArrays& out) {
  using O = ObsRow<D, d, EK1>;
  constexpr int NR = O::NR, NC = D + NR;
  constexpr size_t DD = (size_t)D * D;
  const bool act = r < D;
  const int rr = act ? r : 0;
  O ob;
  ob.load(g, j, base, k, r);
  double f[D];
  load_row16<D>(f, g.F + rr * D);
  double n[NC];
  double m1 = 0.0;
  {
    double n1[D];
    load_row16<D>(n1, g.N1z + rr * D);
    if (k == 0) {
      m1 = dot_lanes<D>(f, g.x0m[(size_t)j * D + rr]);
      double l0[D];
      load_row16<D>(l0, g.x0L + (size_t)j * DD + rr * D);
      bool nz = false;
#pragma unroll
      for (int c = 0; c < D; ++c) nz = nz || l0[c] != 0.0;
      // N1 = tria([F L0 | LQ]); of a zero L0 it is N1z
      if ((__ballot(nz) >> ((threadIdx.x & 63) & ~(kRow - 1))) & 0xffffull) {
        double lq[D], m[2 * D];
        load_row16<D>(lq, g.LQ + rr * D);
        zero(m);
        mul_rows<D, D, D>(m, f, l0);
#pragma unroll
        for (int c = 0; c < D; ++c) m[D + c] = lq[c];
        lq1<D, 2 * D>(m, r);
#pragma unroll
        for (int c = 0; c < D; ++c) n1[c] = (c > r) ? 0.0 : m[c];
      }
    }
#pragma unroll
    for (int c = 0; c < D; ++c) n[c] = n1[c];
  }
#pragma unroll
  for (int c = D; c < NC; ++c) n[c] = 0.0;
  double t[NC];
  {
    double hn[D];
    zero(hn);
    double n1[D];
#pragma unroll
    for (int c = 0; c < D; ++c) n1[c] = n[c];
    ob.template times_rows<1>(r, n1, hn);
#pragma unroll
    for (int c = 0; c < D; ++c) t[c] = hn[c];
  }
#pragma unroll
  for (int c = D; c < NC; ++c) t[c] = ob.r_at(c - D);
  lq_obs<d, NC>(t, n, r);
  Small<d> p11;
  p11.load(t);
  // gain K = Psi21 Psi11^-1; A = F - K H F, b = m1 - K (H m1 + c)
  double K[d];
#pragma unroll
  for (int i = 0; i < d; ++i) K[i] = n[i];
  p11.solve_t(K);
  const size_t o = (size_t)k * D + rr;
  {
    double A[D];
#pragma unroll
    for (int c = 0; c < D; ++c) A[c] = f[c];
    ob.sub_gain(K, f, A);
    if (act) store_row16<D>(out.A + o * D, A);
  }
  {
    double y[d];
    ob.predict(m1, y);  // m1 = 0 without a prior
    double b = m1;
#pragma unroll
    for (int i = 0; i < d; ++i) b = fma(-K[i], y[i], b);
    // Z row = (Psi11^-1 (H F)[:, r])^T, eta = -Z Psi11^-1 c
    double z[d], w[d];
    ob.times_col(g.F, rr, z);
    p11.solve(z);
#pragma unroll
    for (int i = 0; i < d; ++i) w[i] = ob.c[i];
    p11.solve(w);
    double e = 0.0;
#pragma unroll
    for (int i = 0; i < d; ++i) e = fma(-z[i], w[i], e);
    if (act) {
      out.b[o] = b;
      out.eta[o] = e;
#pragma unroll
      for (int i = 0; i < d; ++i) out.Z[(size_t)k * DD + r * d + i] = z[i];
    }
  }
  // U = Psi22: the remaining pivots, rows of n in the columns from d on (NR < d: the last columns zero)
  {
    double u[D];
#pragma unroll
    for (int c = 0; c < D; ++c) u[c] = (d + c < NC) ? n[(d + c < NC) ? d + c : 0] : 0.0;
    lq1<NC - d, NC - d>(u, r);  // the last pivot has no tail
    if (act) store_lower16<D>(out.U + o * D, u, r);
  }
}

// ------------------------------------------------------------- smoother element, statistics
// Smoother element of filtered state (m, L) (pof/parallel_filtsmooth/smoother.py:37-50) and, with
// OBS, the predicted observation's statistics (filter.py:84-114): see k_filter_post.
//   Phi = tria([[F L, LQ], [L, 0]]), E = Phi21 Phi11^-1, g = m - E F m, D = Phi22,
//   S = tria([H Phi11 | R]), yhat = H F m + c.
// EK1: L and LQ are lower triangular with LQ's diagonal nonzero (GroupArgs::own_factors).
template <int D, int d, bool EK1>
__device__ __forceinline__ void filter_post(int r, const GroupArgs& g, int j, long long base, int s, const double* mp,
                                            const double* Lp, bool obs, bool dm_only, bool wc, const SmoArrays& sel, size_t ro,
                                            double* t_ssq, double* t_nll) {
  using O = ObsRow<D, d, EK1>;
  constexpr int NR = O::NR;
  const bool act = r < D;
  const int rr = act ? r : 0;
  O ob;
  // early, so that the reads are over when they are needed; beyond D = 8 its values cost more as registers held through the
  // factorisation (D = 12, 65,536 points: 107 us early, 97 us late; at 1,000 points no difference)
  if (D <= 8 && obs) ob.load(g, j, base, s, r);
  double x11[D], b[2 * D], fm, mr, rd = 0.0;
  {
    double a[2 * D], f[D], l0[D], lq[D];
    mr = mp[rr];
    load_row16<D>(l0, Lp + rr * D);
    load_row16<D>(f, g.F + rr * D);
    load_row16<D>(lq, g.LQ + rr * D);
    fm = dot_lanes<D>(f, mr);
    zero(a);
    mul_rows<D, D, EK1 ? 1 : D>(a, f, l0);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      a[D + c] = lq[c];
      b[c] = l0[c];
      b[D + c] = 0.0;
    }
    unroll<0, D>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      constexpr int n = EK1 ? D : 2 * D - 1 - i;  // LQ lower triangular: second-block columns 0 .. i
      double da, db;
      dot_pair<i, n>(da, db, a + i + 1, b + i + 1);
      const double alpha = bcast<i>(a[i]), sig = bcast<i>(da);
      bool nz = true;
      const Pivot p = EK1 ? pivot_nz(alpha, sig) : pivot(alpha, sig, nz);
      const double tb = reflect_rows<i, n>(b + i + 1, a + i + 1, p.rb, p.sc, db, b[i]);
      const double ta = reflect_self<i, n>(a + i + 1, p.rb, p.sc, da, a[i]);
      const double beta = nz ? p.beta : alpha;
      x11[i] = (r == i) ? beta : fma(-p.den, ta, a[i]);
      b[i] = fma(-p.den, tb, b[i]);
      const double rp = EK1 ? -p.rb : 1.0 / beta;
      rd = (r == i) ? rp : rd;
      keep(rd);
      keep(x11[i]);
      keep(b[i]);
    });
  }
  if (wc) {
    lq1<D, D>(b + D, r);
    if (act) store_lower16<D>(sel.Dm + (ro * D + r) * D, b + D, r);
  }
  if (dm_only) return;
  // E = Phi21 Phi11^-1
  unroll_down<D - 1, 0>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    b[j] = b[j] * bcast<j>(rd);
    fma_rows<j, j>(b, x11, -b[j]);
  });
  const double gr = mr - dot_lanes<D>(b, fm);
  if (act) {
    store_row16<D>(sel.E + (ro * D + r) * D, b);
    sel.g[ro * D + r] = gr;
  }
  if (!obs) {
    if (r == 0 && t_ssq) {
      t_ssq[s] = 0.0;
      t_nll[s] = 0.0;
    }
    return;
  }
  if (D > 8) ob.load(g, j, base, s, r);
  double sr[D + NR];
  {
    double h[D];
    zero(h);
    ob.template times_rows<1>(r, x11, h);
#pragma unroll
    for (int c = 0; c < D; ++c) sr[c] = h[c];
#pragma unroll
    for (int c = D; c < D + NR; ++c) sr[c] = ob.r_at(c - D);
  }
  lq1<d, D + NR>(sr, r);
  Small<d> S;
  S.load(sr);
  double yh[d], w[d];
  ob.predict(fm, yh);
#pragma unroll
  for (int i = 0; i < d; ++i) w[i] = yh[i];
  S.solve_t(w);   // S^T w = yhat
  S.solve(yh);    // S y = yhat
  // lane i < d takes the logarithm of its own diagonal entry
  double di = S.l[0][0];
#pragma unroll
  for (int i = 1; i < d; ++i) di = (r == i) ? S.l[i][i] : di;
  const double lg = log(fabs(di));
  double ss = 0.0, nn = 0.0, ld = 0.0;
  unroll<0, d>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    ss = fma(w[i], w[i], ss);
    nn = fma(yh[i], yh[i], nn);
    ld += bcast<i>(lg);
  });
  if (r == 0) {
    t_ssq[s] = ss;
    // -loglik = 0.5 |S^-1 y|^2 + sum log|S_ii| + d log(2 pi) / 2
    t_nll[s] = 0.5 * nn + (ld + d * log(2.0 * M_PI) / 2.0);
  }
}

// ------------------------------------------------------------- sequential filter and smoother
// k_seq_filter of one IVP (pof/sequential_filtsmooth/filter.py:9-92), state and model in the registers of one row.
// A step is a serial chain of about 2 D + d pivots and its one wavefront issues an FP64 instruction every 8.5
// cycles, so it is the instructions of a step that count: the predicted factor never leaves the registers, the
// model's values are read a step ahead, and the step's logarithms wait for sixteen steps, a step per lane.
// Against a whole wavefront per IVP with its tiles in LDS, filter and smoother of 513 points: 8.6 -> 2.1 ms at
// D = 8, 16.1 -> 3.6 ms at D = 12, 22.4 -> 5.4 ms at D = 15 (17.4, 31 and 44 us per step before).
// LOW: LQ and the prior's factor are lower triangular (GroupArgs::own_factors): a caller's need not be.
template <int D, int d, bool EK1, bool AT_PRED, bool LOW>
__device__ __forceinline__ void seq_filter(int r, const GroupArgs& g, int j, long long base, int Ns,
                                           const StateArrays& fp, double* shared) {
  using O = ObsRow<D, d, EK1>;
  constexpr int NR = O::NR, NC = D + NR, q1 = D / d;
  const bool act = r < D;
  const int rr = act ? r : 0;
  double* t_ssq = g.t_ssq + base;
  double* t_nll = g.t_nll + base;
  const double* lin = (g.cur[j] ? g.means1 : g.means0) + (size_t)base * D;
  const int kind = EK1 ? g.kind[j] : 0;
  double* Pd = shared;  // [D], then the field's parameters
  double* params = shared + D;
  if constexpr (EK1) {
    if (act) Pd[r] = g.Pd[(size_t)j * D + r];
    if (r < kMaxParams) params[r] = g.params[(size_t)j * kMaxParams + r];
    wsync();
  }
  double f[D], lq[D], l[D];
  load_row16<D>(f, g.F + rr * D);
  load_row16<D>(lq, g.LQ + rr * D);
  load_row16<D>(l, g.x0L + (size_t)j * D * D + rr * D);
  double m = g.x0m[(size_t)j * D + rr];
  O ob, next;      // (affine) the model of this step and of the next
  double y1[d];    // (EK1 at given means) the next step's
  auto fetch = [&](int k) {
    if constexpr (!EK1) {
      next.load(g, j, base, k, r);
    } else if constexpr (!AT_PRED) {
#pragma unroll
      for (int i = 0; i < d; ++i) y1[i] = lin[(size_t)(k + 1) * D + i * q1];
    }
  };
  if (Ns > 0) fetch(0);
  double dg[d], nn = 0.0, ss = 0.0;  // lane k % 16: step k's diagonal of I, |I^-1 y|^2, |I^-T y|^2
#pragma unroll
  for (int i = 0; i < d; ++i) dg[i] = 1.0;
  for (int k = 0; k < Ns; ++k) {
    if constexpr (!EK1) {
      ob = next;
    } else if constexpr (!AT_PRED) {
      ob.load_entries(kind, params, Pd, y1);
    }
    if (k + 1 < Ns) fetch(k + 1);
    // predict: mp = F m, N1 = tria([F L | LQ])
    const double mp = dot_lanes<D>(f, m);
    double n[NC];
    {
      double a[2 * D];
      zero(a);
      mul_rows<D, D, LOW ? 1 : D>(a, f, l);
#pragma unroll
      for (int c = 0; c < D; ++c) a[D + c] = lq[c];
      lq1<D, 2 * D, D, LOW ? 0 : D>(a, r);
#pragma unroll
      for (int c = 0; c < D; ++c) n[c] = (c > r) ? 0.0 : a[c];
#pragma unroll
      for (int c = D; c < NC; ++c) n[c] = 0.0;
    }
    if constexpr (EK1 && AT_PRED) {
      double mi[d];
      unroll<0, d>([&](auto ic) { mi[decltype(ic)::value] = bcast<decltype(ic)::value * q1>(mp); });
      ob.load_entries(kind, params, Pd, mi);
    }
    // update: tria([[H N1, R], [N1, 0]]) = [[I, 0], [G, L]]
    double t[NC];
    {
      double hn[D], n1[D];
      zero(hn);
#pragma unroll
      for (int c = 0; c < D; ++c) n1[c] = n[c];
      ob.template times_rows<1>(r, n1, hn);
#pragma unroll
      for (int c = 0; c < D; ++c) t[c] = hn[c];
#pragma unroll
      for (int c = D; c < NC; ++c) t[c] = ob.r_at(c - D);
    }
    lq_obs<d, NC>(t, n, r);
    Small<d> S;
    S.load(t);
    double z[d], w[d];
    ob.predict(mp, z);
#pragma unroll
    for (int i = 0; i < d; ++i) w[i] = z[i] = -z[i];
    S.solve(z);    // I z = y
    S.solve_t(w);  // I^T w = y (whiten)
    m = mp;
#pragma unroll
    for (int i = 0; i < d; ++i) m = fma(n[i], z[i], m);
#pragma unroll
    for (int c = 0; c < D; ++c) l[c] = (d + c < NC) ? n[(d + c < NC) ? d + c : 0] : 0.0;
    lq1<NC - d, NC - d>(l, r);  // the last pivot has no tail
#pragma unroll
    for (int c = 1; c < D; ++c) l[c] = (c > r) ? 0.0 : l[c];
    if (act) {
      fp.m[(size_t)k * D + r] = m;
      store_row16<D>(fp.L + ((size_t)k * D + r) * D, l);
    }
    double sn = 0.0, sw = 0.0;
#pragma unroll
    for (int i = 0; i < d; ++i) {
      sn = fma(z[i], z[i], sn);
      sw = fma(w[i], w[i], sw);
    }
    const int e = k % kRow;
    const bool mine = r == e;
    nn = mine ? sn : nn;
    ss = mine ? sw : ss;
#pragma unroll
    for (int i = 0; i < d; ++i) dg[i] = mine ? S.l[i][i] : dg[i];
    if (e == kRow - 1 || k + 1 == Ns) {
      double ld = 0.0;
#pragma unroll
      for (int i = 0; i < d; ++i) ld += log(fabs(dg[i]));
      if (r <= e) {
        t_ssq[k - e + r] = ss;
        // mvn_loglikelihood (utils.py:22-30): -|I^-1 y|^2 / 2 - sum log|I_ii| - d log(2 pi) / 2
        t_nll[k - e + r] = -0.5 * nn - (ld + d * log(2.0 * M_PI) / 2.0);
      }
    }
  }
}

// The RTS recursion (pof/sequential_filtsmooth/smoother.py:8-48) over gains E and factors Phi22 = D formed beforehand
// for all steps at once (filter_post; its other half is what a step would otherwise spend most of its time on):
//   mean = mf + E (mean - F mf), L = tria([D | E L]),
// state Ns - s of the smoother arrays as k_seq_smooth.  A step's reads are issued a step ahead.
template <int D>
__device__ __forceinline__ void seq_smooth(int r, const GroupArgs& g, int j, int Ns, const StateArrays& fp,
                                           const StateArrays& sp, const SmoArrays& sel) {
  const bool act = r < D;
  const int rr = act ? r : 0;
  const bool wc = g.wchol[j] != 0;
  const double* x0m = g.x0m + (size_t)j * D;
  double f[D], l[D];
  load_row16<D>(f, g.F + rr * D);
  load_row16<D>(l, (Ns == 0 ? g.x0L + (size_t)j * D * D : fp.L + (size_t)(Ns - 1) * D * D) + rr * D);
  double m = (Ns == 0 ? x0m : fp.m + (size_t)(Ns - 1) * D)[rr];
  if (act) {
    sp.m[r] = m;
    if (wc) store_row16<D>(sp.L + r * D, l);
  }
  double e1[D], d1[D], mf1 = 0.0;  // the next step's
  zero(d1);
  auto fetch = [&](int s) {  // s = Ns - k
    const int k = Ns - s;
    mf1 = ((k == 0) ? x0m : fp.m + (size_t)(k - 1) * D)[rr];
    load_row16<D>(e1, sel.E + ((size_t)s * D + rr) * D);
    if (wc) load_row16<D>(d1, sel.Dm + ((size_t)s * D + rr) * D);
  };
  if (Ns > 0) fetch(1);
  for (int s = 1; s <= Ns; ++s) {
    double e[D], a[D];
    const double mf = mf1;
#pragma unroll
    for (int c = 0; c < D; ++c) {
      e[c] = e1[c];
      a[c] = d1[c];
    }
    if (s < Ns) fetch(s + 1);
    m = dot_lanes<D>(e, m - dot_lanes<D>(f, mf), mf);
    if (act) sp.m[(size_t)s * D + r] = m;
    if (wc) {
      double t[D];
      zero(t);
      mul_rows<D, D, D>(t, e, l);  // the last state's factor may be a caller's, not triangular
      // D's row i ends at column i, and so does what the reflectors before pivot i leave of it
      unroll<0, D>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const double dot = dot_self<i, D>(t);
        bool nz;
        const Pivot p = pivot(bcast<i>(a[i]), bcast<i>(dot), nz);
        const double x = reflect_self<i, D>(t, p.rb, p.sc, dot, a[i]);
        a[i] = (r == i && nz) ? p.beta : fma(-p.den, x, a[i]);
      });
#pragma unroll
      for (int c = 0; c < D; ++c) l[c] = (c > r) ? 0.0 : a[c];
      if (act) store_row16<D>(sp.L + ((size_t)s * D + r) * D, l);
    }
  }
}

}  // namespace r16
}  // namespace pof

#pragma clang fp contract(fast)
