// sfgs_math.hpp -- device-side 3x3 algebra, cone operations and the local
// Signorini-Coulomb solvers of one contact row, templated on the arithmetic
// type (double for the FP64 path, float for the mixed-precision sweeps).
//
// Semantics follow the reference:
//   scf_project<T>        scf.c:136-174  (SCF_Project)
//   scf_residual<T>       scf.c:28-133   (SCF_Linearize, C and optionally X, Y)
//   solve3<T>             dgesv on 3x3 as called at dbs.c:282, 317
//   projected_gradient<T> dbs.c:35-94
//   de_saxce_feng<T>      dbs.c:96-140
//   semismooth_newton<T>  dbs.c:142-303
//   projected_newton<T>   dbs.c:305-326
// Matrices are column-major (M[r + 3c]), frames [t1 t2 n].  Everything lives in
// registers; there is no memory traffic here.
#pragma once
#include <hip/hip_runtime.h>
#include <cfloat>
#include <climits>

namespace sfgs {

template <typename T> struct V3 { T x, y, z; };

template <typename T> __device__ __forceinline__ T tmax(T a, T b) { return a > b ? a : b; }
template <typename T> __device__ __forceinline__ T tmin(T a, T b) { return a < b ? a : b; }

// Division and square root of the local solvers: IEEE in FP64; in the FP32
// sweeps of the mixed mode the hardware reciprocal and square root (1 ulp),
// whose error stays below the FP32 local tolerance (the FP64 refinement sweeps
// settle the final state)
template <typename T> __device__ __forceinline__ T fdiv(T a, T b) { return a / b; }
template <> __device__ __forceinline__ float fdiv<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
template <typename T> __device__ __forceinline__ T fsqrt(T x) { return sqrt(x); }
template <> __device__ __forceinline__ float fsqrt<float>(float x) { return __builtin_amdgcn_sqrtf(x); }

// 1/x and 1/sqrt(x) in FP64 for normal x (rsqrt64: positive), to about one ulp:
// the hardware estimates are good to 2^-22 or better, so two steps of Newton's
// iteration (rcp64) or of Goldschmidt's coupled one (rsqrt64) reach 2^-53.  An
// infinite or NaN argument gives NaN; the caller excludes zero and subnormal ones.
__device__ __forceinline__ double rcp64(double x)
{
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  return fma(r, fma(-x, r, 1.0), r);
}
__device__ __forceinline__ double rsqrt64(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  double h = 0.5*y, g = x*y, e = fma(-h, g, 0.5);
  h = fma(h, e, h); g = fma(g, e, g);
  e = fma(-h, g, 0.5);
  h = fma(h, e, h);
  return h + h;
}

// y = c + M v
template <typename T>
__device__ __forceinline__ void mv_add(const T *c, const T *M, const T *v, T *y)
{
  T y0 = c[0] + (M[0]*v[0] + M[3]*v[1] + M[6]*v[2]);
  T y1 = c[1] + (M[1]*v[0] + M[4]*v[1] + M[7]*v[2]);
  T y2 = c[2] + (M[2]*v[0] + M[5]*v[1] + M[8]*v[2]);
  y[0] = y0; y[1] = y1; y[2] = y2;
}

template <typename T>
__device__ __forceinline__ T rel_change(const T *R, const T *R0)
{
  T d0 = R[0] - R0[0], d1 = R[1] - R0[1], d2 = R[2] - R0[2];
  T rr = R[0]*R[0] + R[1]*R[1] + R[2]*R[2];
  return fsqrt(fdiv(d0*d0 + d1*d1 + d2*d2, tmax(rr, T(1))));
}

// LU with partial pivoting on a 3x3 (column-major), b overwritten with x.
// Returns nonzero on an exactly zero pivot (dgesv info > 0).
template <typename T>
__device__ __forceinline__ int solve3(T *a, T *b)
{
#pragma unroll
  for (int k = 0; k < 3; k ++)
  {
    int p = k;
    T amax = fabs(a[k + 3*k]);
#pragma unroll
    for (int i = k + 1; i < 3; i ++)
    {
      T v = fabs(a[i + 3*k]);
      if (v > amax) { amax = v; p = i; }
    }
    if (amax == T(0)) return k + 1;
    if (p != k)
    {
#pragma unroll
      for (int c = 0; c < 3; c ++)
      {
        // select-based swap keeps the arrays in registers
        T ak = a[k + 3*c], ap = a[p + 3*c];
        a[k + 3*c] = ap;
#pragma unroll
        for (int i = k + 1; i < 3; i ++) if (i == p) a[i + 3*c] = ak;
      }
      T bk = b[k], bp = b[p];
      b[k] = bp;
#pragma unroll
      for (int i = k + 1; i < 3; i ++) if (i == p) b[i] = bk;
    }
    T inv = fdiv(T(1), a[k + 3*k]);
    a[k + 3*k] = inv;   // kept for the back substitution
#pragma unroll
    for (int i = k + 1; i < 3; i ++)
    {
      T l = a[i + 3*k] * inv;
#pragma unroll
      for (int c = k + 1; c < 3; c ++) a[i + 3*c] -= l * a[k + 3*c];
      b[i] -= l * b[k];
    }
  }
#pragma unroll
  for (int k = 2; k >= 0; k --)
  {
    b[k] *= a[k + 3*k];
#pragma unroll
    for (int i = 0; i < k; i ++) b[i] -= b[k] * a[i + 3*k];
  }
  return 0;
}

// 3x3 inverse by LU with partial pivoting (dgetrf/dgetri as MX_Inverse calls
// them); 0 on success
template <typename T>
__device__ __forceinline__ int inverse3(const T *W, T *A)
{
#pragma unroll
  for (int c = 0; c < 3; c ++)
  {
    T M[9], x[3] = {c == 0 ? T(1) : T(0), c == 1 ? T(1) : T(0), c == 2 ? T(1) : T(0)};
#pragma unroll
    for (int k = 0; k < 9; k ++) M[k] = W[k];
    if (solve3(M, x)) return -1;
    A[3*c] = x[0]; A[3*c + 1] = x[1]; A[3*c + 2] = x[2];
  }
  return 0;
}

// spectral factorisation of S with respect to the cone (orientation of scf.c)
template <typename T>
__device__ __forceinline__ void spectral(T fri, const T *S, T &l1, T &l2, T *u1, T *u2, T &slen)
{
  T onefri2 = T(1) + fri*fri;
  slen = fsqrt(S[0]*S[0] + S[1]*S[1]);
  l1 = fdiv(-(S[2] + fri*slen), onefri2);
  l2 = fdiv(slen - fri*S[2], onefri2);
  if (slen != T(0)) { u2[0] = S[0]/slen; u2[1] = S[1]/slen; }
  else { u2[0] = T(1); u2[1] = T(0); }
  u2[2] = -fri;
  u1[0] = -fri*u2[0]; u1[1] = -fri*u2[1]; u1[2] = T(-1);
}

// R = projection of S onto the friction cone shifted by the cohesion
template <typename T>
__device__ __forceinline__ void scf_project(T fri, T coh, const T *S, T *R)
{
  T Sc[3] = {S[0], S[1], S[2] + coh}, l1, l2, u1[3], u2[3], sl;
  spectral(fri, Sc, l1, l2, u1, u2, sl);
  T g1 = tmax(l1, T(0)), g2 = tmax(l2, T(0));
  T m0 = g1*u1[0] + g2*u2[0], m1 = g1*u1[1] + g2*u2[1], m2 = g1*u1[2] + g2*u2[2];
  T s0 = S[0], s1 = S[1], s2 = S[2];
  R[0] = s0 - m0; R[1] = s1 - m1; R[2] = s2 - m2;
}

// C(U,R) with UT = -1 and zero smoothing (the merit form, mrf.c:82) and, when
// X != nullptr, the Jacobians X = dC/dU, Y = dC/dR (scf.c:92-132).
// 'shift' is the dashed-normal offset: dynamic e*min(V_N,0), static max(gap,0)/h.
template <typename T>
__device__ __forceinline__ void scf_residual(T fri, T coh, T shift, const T *U, const T *R, T *C, T *X, T *Y)
{
  T fri2 = fri*fri, onefri2 = T(1) + fri2;
  T udash = U[2] + shift;
  T ulen = sqrt(U[0]*U[0] + U[1]*U[1]);
  T F[3] = {U[0], U[1], udash + fri*ulen};
  T S[3] = {R[0] - F[0], R[1] - F[1], R[2] - F[2] + coh};
  T l1, l2, u1[3], u2[3], slen;
  spectral(fri, S, l1, l2, u1, u2, slen);
  T sq1 = fabs(l1), sq2 = fabs(l2);
  T g1 = T(0.5)*(sq1 + l1), g2 = T(0.5)*(sq2 + l2);
  C[0] = F[0] + (g1*u1[0] + g2*u2[0]);
  C[1] = F[1] + (g1*u1[1] + g2*u2[1]);
  C[2] = F[2] + (g1*u1[2] + g2*u2[2]);
  if (X)
  {
    T dF[9] = {T(1), T(0), fri*U[0]/ulen, T(0), T(1), fri*U[1]/ulen, T(0), T(0), T(1)};
    T dg1 = T(0.5)*(T(1) + l1/sq1), sdot = S[0]*S[0] + S[1]*S[1];
    if (slen != T(0))
    {
      T dg2 = T(0.5)*(T(1) + l2/sq2);
      T a = T(0.5)*(T(1) + (l2 + fri*l1)/(sq2 + fri*sq1));
      T b = (fri2*dg1 + dg2)/onefri2;
      T c = (fri*(dg1 - dg2))/onefri2;
      T d = (dg1 + fri2*dg2)/onefri2;
      Y[0] = a + (b - a)*S[0]*S[0]/sdot;
      Y[1] = (b - a)*S[1]*S[0]/sdot;
      Y[2] = c*S[0]/slen;
      Y[3] = Y[1];
      Y[4] = a + (b - a)*S[1]*S[1]/sdot;
      Y[5] = c*S[1]/slen;
      Y[6] = Y[2];
      Y[7] = Y[5];
      Y[8] = d;
    }
    else
    {
      Y[1] = Y[2] = Y[3] = Y[5] = Y[6] = Y[7] = T(0);
      Y[0] = Y[4] = Y[8] = dg1;
    }
#pragma unroll
    for (int c = 0; c < 3; c ++)
#pragma unroll
      for (int r = 0; r < 3; r ++)
        X[r + 3*c] = dF[r + 3*c] - (Y[r]*dF[3*c] + Y[r + 3]*dF[3*c + 1] + Y[r + 6]*dF[3*c + 2]);
  }
}

// C(U,R) of the merit in FP64: scf_residual without the Jacobians, with the
// quotients shared (1/(1 + mu^2) once, |U_T| and 1/|S_T| from one reciprocal root
// each) instead of three roots and five divisions, which took 920 of a slice's
// clocks.  A tangential part whose square is subnormal counts as none: u2 = (1, 0)
// as in spectral.  What is not finite stays so, as there: 0.5 (|l| + l), the half
// taken into the shared quotient, carries a NaN and makes one of -inf where a maximum
// would give 0, and a tangential part that is NaN or whose square overflows is NaN and
// not none.  Only the merit sums depend on it.
__device__ __forceinline__ void merit_residual(double fri, double coh, double shift, const double *U, const double *R,
                                               double *C)
{
  const double ho = 0.5*rcp64(1.0 + fri*fri);
  const double uu = U[0]*U[0] + U[1]*U[1];
  const double ulen = uu < DBL_MIN ? 0.0 : uu*rsqrt64(uu);
  const double F2 = U[2] + shift + fri*ulen;
  const double S0 = R[0] - U[0], S1 = R[1] - U[1], S2 = R[2] - F2 + coh;
  const double ss = S0*S0 + S1*S1;
  const bool none = ss < DBL_MIN;
  const double is = none ? 0.0 : rsqrt64(ss), sl = ss*is;
  const double l1 = -(S2 + fri*sl)*ho, l2 = (sl - fri*S2)*ho;   // half of each
  const double g1 = fabs(l1) + l1, g2 = fabs(l2) + l2;
  const double gt = g2 - fri*g1;
  C[0] = U[0] + gt*(none ? 1.0 : S0*is);
  C[1] = U[1] + gt*(S1*is);
  C[2] = F2 - (g1 + fri*g2);
}

// per-row constants of the local problem
template <typename T>
struct RowLaw {
  T fri, coh, shift, rho;
  bool separated;   // dynamic && gap > 0: R = 0, U = B
};

template <typename T>
__device__ __forceinline__ int projected_gradient(const RowLaw<T> &L, T eps, int maxiter, const T *W, const T *B, T *U, T *R)
{
  if (L.separated) { R[0] = R[1] = R[2] = T(0); U[0] = B[0]; U[1] = B[1]; U[2] = B[2]; return 0; }
  int iter = 0;
  T err;
  do
  {
    T R0[3] = {R[0], R[1], R[2]};
    mv_add(B, W, R, U);
    T UN = U[2] + L.shift;
    R[0] -= L.rho*U[0];
    R[1] -= L.rho*U[1];
    R[2] -= L.rho*UN - L.coh;
    R[2] = tmax(T(0), R[2]);
    T t = sqrt(R[0]*R[0] + R[1]*R[1]);
    if (t >= L.fri*R[2])
    {
      if (t > T(0)) t = L.fri*R[2]/t;
      R[0] *= t; R[1] *= t;
    }
    R[2] -= L.coh;
    err = rel_change(R, R0);
  }
  while (++ iter < maxiter && err > eps);
  return iter;
}

template <typename T>
__device__ __forceinline__ int de_saxce_feng(const RowLaw<T> &L, T eps, int maxiter, const T *W, const T *B, T *U, T *R)
{
  if (L.separated) { R[0] = R[1] = R[2] = T(0); U[0] = B[0]; U[1] = B[1]; U[2] = B[2]; return 0; }
  int iter = 0;
  T err;
  do
  {
    T R0[3] = {R[0], R[1], R[2]}, tau[3];
    mv_add(B, W, R, U);
    T UN = U[2] + L.shift;
    tau[0] = R[0] - L.rho*U[0];
    tau[1] = R[1] - L.rho*U[1];
    tau[2] = R[2] - L.rho*(UN + L.fri*sqrt(U[0]*U[0] + U[1]*U[1]));
    scf_project(L.fri, L.coh, tau, R);
    err = rel_change(R, R0);
  }
  while (++ iter < maxiter && err > eps);
  return iter;
}

// The local solve of a sweep launch is its longest chain: a wavefront issues one
// instruction at a time, about five clocks each, so the loop costs its number of
// instructions.  It is written for few of them (600 -> about 300 per FP64
// iteration with sliding and sticking rows in one wavefront; 8.5-9.2k -> 6.5-7.0k
// clocks for three iterations in FP64, 5.6k -> 4.7k in FP32; with selects for the
// sliding entries instead of a branch 7.1k and 5.0k):
//  * one system for all states, completed in a branch for sliding,
//    instead of four branches whose nine entries meet in moves; one division
//    serves sliding (1/|d_T|) and sticking (1/d_N);
//  * the pivot exchanges only where a lane of the wavefront has one;
//  * alfa, delta and beta only where a lane has R.d < 0 (alfa < 0 elsewhere
//    leaves beta = 1);
//  * the error bound by squares, |dR|^2 against eps^2 max(|R|^2, 1), with the
//    quotient and the root only within their rounding of equality.
// Every operation that reaches U, R or a decision is the one it was, with the
// same rounding (the fused multiply-adds are explicit and contraction is off):
// whether a row at rest counts as open hangs on the last bit of U_N.
template <typename T> struct ErrBound {
  T lo, hi;   // |dR|^2 / max(|R|^2, 1) surely at most eps^2, surely above it
  __device__ __forceinline__ explicit ErrBound(T eps)
  {
    // the quotient and the root are within a few ulp: 1e-13 (FP64), 4e-6 (FP32).
    // A tolerance whose square is no normal number, and a negative one, which no
    // change is within, leave every decision to the quotient and the root.
    const T e2 = eps*eps, m = sizeof(T) == 8 ? T(1e-13) : T(4e-6);
    const bool ok = eps > T(0) && e2 > (sizeof(T) == 8 ? T(1e-290) : T(1e-30));
    lo = ok ? e2*(T(1) - m) : T(-1);
    hi = ok ? e2*(T(1) + m) : T(INFINITY);
  }
};

// a 3x3 solve as solve3 (the same pivots and operations), in registers without
// branches but the exchanges; singular is set instead of a return
template <typename T>
__device__ __forceinline__ void lu3(T a0, T a1, T a2, T a3, T a4, T a5, T a6, T a7, T a8, T b0, T b1, T b2, T &x0, T &x1,
                                    T &x2, bool &singular)
{
#pragma clang fp contract(off)
  T m = fabs(a0);
  const bool p1 = fabs(a1) > m;
  m = p1 ? fabs(a1) : m;
  const bool p2 = fabs(a2) > m;
  if (__any(p1 || p2))
  {
    // row 0 with row 2 where p2, else with row 1 where p1
    const bool q1 = p1 && !p2;
    T t;
    t = a0; a0 = p2 ? a2 : q1 ? a1 : a0; a1 = q1 ? t : a1; a2 = p2 ? t : a2;
    t = a3; a3 = p2 ? a5 : q1 ? a4 : a3; a4 = q1 ? t : a4; a5 = p2 ? t : a5;
    t = a6; a6 = p2 ? a8 : q1 ? a7 : a6; a7 = q1 ? t : a7; a8 = p2 ? t : a8;
    t = b0; b0 = p2 ? b2 : q1 ? b1 : b0; b1 = q1 ? t : b1; b2 = p2 ? t : b2;
  }
  const T i0 = fdiv(T(1), a0);
  singular = a0 == T(0);
  const T l1 = a1*i0, l2 = a2*i0;
  a4 = fma(-l1, a3, a4); a7 = fma(-l1, a6, a7); b1 = fma(-l1, b0, b1);
  a5 = fma(-l2, a3, a5); a8 = fma(-l2, a6, a8); b2 = fma(-l2, b0, b2);
  const bool p = fabs(a5) > fabs(a4);
  if (__any(p))
  {
    T t;
    t = a4; a4 = p ? a5 : a4; a5 = p ? t : a5;
    t = a7; a7 = p ? a8 : a7; a8 = p ? t : a8;
    t = b1; b1 = p ? b2 : b1; b2 = p ? t : b2;
  }
  const T i1 = fdiv(T(1), a4);
  singular = singular || a4 == T(0);
  const T l = a5*i1;
  a8 = fma(-l, a7, a8); b2 = fma(-l, b1, b2);
  singular = singular || a8 == T(0);
  x2 = b2*fdiv(T(1), a8);
  x1 = fma(-x2, a7, b1)*i1;
  x0 = fma(-x1, a3, fma(-x2, a6, b0))*i0;
}

template <typename T>
__device__ __forceinline__ int semismooth_newton(const RowLaw<T> &L, T eps, int maxiter, const T *W, const T *B, T *U, T *R)
{
#pragma clang fp contract(off)
  if (L.separated) { R[0] = R[1] = R[2] = T(0); U[0] = B[0]; U[1] = B[1]; U[2] = B[2]; return 0; }
  const T fri = L.fri, coh = L.coh;
  const ErrBound<T> bound(eps);
  T rho = L.rho;
  const int divi = maxiter / 10;
  int iter = 0, left = divi > 0 ? divi : INT_MAX;
  bool more;
  do
  {
    const T UN = U[2] + L.shift, RN = R[2] + coh;
    const T d0 = fma(-rho, U[0], R[0]), d1 = fma(-rho, U[1], R[1]), d2 = fma(-rho, UN, RN);
    const T s0 = (B[0] + fma(W[6], R[2], fma(W[3], R[1], W[0]*R[0]))) - U[0];
    const T s1 = (B[1] + fma(W[7], R[2], fma(W[4], R[1], W[1]*R[0]))) - U[1];
    const T s2 = (B[2] + fma(W[8], R[2], fma(W[5], R[1], W[2]*R[0]))) - U[2];
    T x0 = -R[0], x1 = -R[1], x2 = -R[2];   // open: R = 0
    if (d2 >= T(0))
    {
      const T norm = fsqrt(fma(d0, d0, d1*d1)), lim = fri*d2;
      const bool out = norm >= lim, slide = out && lim > T(0);
      const T inv = fdiv(T(1), slide ? norm : d2);
      const T s = fma(rho*U[2], inv, T(1));
      T a0 = W[0], a1 = W[1], a3 = W[3], a4 = W[4], a6 = fma(U[0], inv, W[6]), a7 = fma(U[1], inv, W[7]);
      T b0 = fma(-s, U[0], -s0), b1 = fma(-s, U[1], -s1);
      const T b2 = -UN - s2;
      if (out)
      {
        if (slide)
        {
          const T len = fsqrt(fma(R[1], R[1], R[0]*R[0])), r0 = R[0]*d0, r1 = R[1]*d1, num = r0 + r1;
          const T iden = fdiv(T(1), tmax(lim, len)*norm), e = lim*inv;
          T beta = T(1);
          if (num < T(0) && len != T(0))
          {
            const T alfa = fdiv(num, len*norm), delta = tmin(fdiv(len, lim), T(1));
            beta = alfa < T(0) ? fdiv(T(1), fma(-alfa, delta, T(1))) : T(1);
          }
          const T M0 = e*fma(-r0, iden, T(1)), M1 = -e*((R[1]*d0)*iden);
          const T M2 = -e*((R[0]*d1)*iden), M3 = e*fma(-r1, iden, T(1));
          const T f0 = fri*(d0*inv), f1 = fri*(d1*inv);
          a0 = fma(rho, fma(W[1], M2, W[0]*M0), fma(-beta, M0, T(1)));
          a1 = fma(rho, fma(W[0], M1, W[1]*M3), -(beta*M1));
          a3 = fma(rho, fma(W[4], M2, W[3]*M0), -(beta*M2));
          a4 = fma(rho, fma(W[3], M1, W[4]*M3), fma(-beta, M3, T(1)));
          a6 = fma(rho, fma(W[7], M2, W[6]*M0), -f0);
          a7 = fma(rho, fma(W[6], M1, W[7]*M3), -f1);
          b0 = fma(-rho, fma(s1, M2, s0*M0), fma(RN, f0, -R[0]));
          b1 = fma(-rho, fma(s0, M1, s1*M3), fma(RN, f1, -R[1]));
        }
        else
        {
          a0 = a4 = T(1);
          a1 = a3 = a6 = a7 = T(0);
          b0 = -R[0] - s0;
          b1 = -R[1] - s1;
        }
      }
      bool singular;
      lu3(a0, a1, W[2], a3, a4, W[5], a6, a7, W[8], b0, b1, b2, x0, x1, x2, singular);
      if (singular) return -1;
    }
    if (!isfinite(x0 + x1 + x2)) return -1;

    U[0] += s0 + fma(W[6], x2, fma(W[3], x1, W[0]*x0));
    U[1] += s1 + fma(W[7], x2, fma(W[4], x1, W[1]*x0));
    U[2] += s2 + fma(W[8], x2, fma(W[5], x1, W[2]*x0));
    const T p0 = R[0] + x0, p1 = R[1] + x1, p2 = R[2] + x2;
    const T e0 = p0 - R[0], e1 = p1 - R[1], e2 = p2 - R[2];
    R[0] = p0; R[1] = p1; R[2] = p2;
    const T dd = fma(e2, e2, fma(e1, e1, e0*e0));
    const T mx = tmax(fma(p2, p2, fma(p1, p1, p0*p0)), T(1));
    more = dd > bound.hi*mx;
    if (!more && !(dd < bound.lo*mx)) more = fsqrt(fdiv(dd, mx)) > eps;
    iter ++;
    if (-- left == 0)
    {
      left = divi;
      rho *= T(10);
      if (isinf(rho)) return -1;
    }
  }
  while (iter < maxiter && more);
  return iter;
}

template <typename T>
__device__ __forceinline__ int projected_newton(const RowLaw<T> &L, T eps, int maxiter, const T *W, const T *B, T *U, T *R)
{
  T X[9], Y[9], C[3], Tm[9], merit;
  int iter = 0;
  mv_add(B, W, R, U);
  scf_residual(L.fri, L.coh, L.shift, U, R, C, X, Y);
  do
  {
#pragma unroll
    for (int c = 0; c < 3; c ++)
#pragma unroll
      for (int r = 0; r < 3; r ++)
        Tm[r + 3*c] = (X[r]*W[3*c] + X[r + 3]*W[3*c + 1] + X[r + 6]*W[3*c + 2]) + Y[r + 3*c];
    if (solve3(Tm, C)) return -1;
    R[0] -= C[0]; R[1] -= C[1]; R[2] -= C[2];
    scf_project(L.fri, L.coh, R, R);
    mv_add(B, W, R, U);
    scf_residual(L.fri, L.coh, L.shift, U, R, C, X, Y);
    merit = sqrt(C[0]*C[0] + C[1]*C[1] + C[2]*C[2]);
  }
  while (merit > eps && ++ iter < maxiter);
  return iter;
}

template <typename T>
__device__ __forceinline__ int local_solve(int solver, const RowLaw<T> &L, T eps, int maxiter, const T *W, const T *B, T *U, T *R)
{
  switch (solver)
  {
  case 0: return projected_gradient(L, eps, maxiter, W, B, U, R);
  case 1: return de_saxce_feng(L, eps, maxiter, W, B, U, R);
  case 3: return projected_newton(L, eps, maxiter, W, B, U, R);
  default: return semismooth_newton(L, eps, maxiter, W, B, U, R);
  }
}

// SCF_Linearize (scf.c:28-133) with UT < 0 and smoothing omega = eps > 0, as
// the Newton solver calls it (nts.c:1075): C(U, R), X = dC/dU, Y = dC/dR with
// |U_T| -> sqrt(|U_T|^2 + eps^2) and |l| -> sqrt(l^2 + 4 eps^2 (mu^2)).
__device__ __forceinline__ void scf_linearize_smooth(double fri, double coh, double shift, double eps, const double *U,
                                                     const double *R, double *C, double *X, double *Y)
{
  const double eps2 = eps*eps, fri2 = fri*fri, onefri2 = 1.0 + fri2;
  const double udash = U[2] + shift;
  const double ulen = sqrt(U[0]*U[0] + U[1]*U[1] + eps2);
  const double F[3] = {U[0], U[1], udash + fri*(ulen - eps)};
  double S[3] = {R[0] - F[0], R[1] - F[1], R[2] - F[2] + coh};
  const double sdot = S[0]*S[0] + S[1]*S[1], slen = sqrt(sdot);
  const double l1 = -(S[2] + fri*slen)/onefri2, l2 = (slen - fri*S[2])/onefri2;
  double u1[3], u2[3];
  if (slen != 0.0) { u2[0] = S[0]/slen; u2[1] = S[1]/slen; }
  else { u2[0] = 1.0; u2[1] = 0.0; }
  u2[2] = -fri;
  u1[0] = -fri*u2[0]; u1[1] = -fri*u2[1]; u1[2] = -1.0;
  const double sq1 = sqrt(l1*l1 + 4.0*eps2), sq2 = sqrt(l2*l2 + 4.0*eps2*fri2);
  const double g1 = 0.5*(sq1 + l1), g2 = 0.5*(sq2 + l2);
  C[0] = F[0] + (g1*u1[0] + g2*u2[0]);
  C[1] = F[1] + (g1*u1[1] + g2*u2[1]);
  C[2] = F[2] + (g1*u1[2] + g2*u2[2]);
  const double dF[9] = {1.0, 0.0, fri*U[0]/ulen, 0.0, 1.0, fri*U[1]/ulen, 0.0, 0.0, 1.0};
  const double dg1 = 0.5*(1.0 + l1/sq1);
  if (slen != 0.0)
  {
    const double dg2 = 0.5*(1.0 + l2/sq2);
    const double a = 0.5*(1.0 + (l2 + fri*l1)/(sq2 + fri*sq1));
    const double b = (fri2*dg1 + dg2)/onefri2, c = (fri*(dg1 - dg2))/onefri2, d = (dg1 + fri2*dg2)/onefri2;
    Y[0] = a + (b - a)*S[0]*S[0]/sdot;
    Y[1] = (b - a)*S[1]*S[0]/sdot;
    Y[2] = c*S[0]/slen;
    Y[3] = Y[1];
    Y[4] = a + (b - a)*S[1]*S[1]/sdot;
    Y[5] = c*S[1]/slen;
    Y[6] = Y[2];
    Y[7] = Y[5];
    Y[8] = d;
  }
  else
  {
    Y[1] = Y[2] = Y[3] = Y[5] = Y[6] = Y[7] = 0.0;
    Y[0] = Y[4] = Y[8] = dg1;
  }
  // X = dF - Y dF  ([I - dm/dS] dF/dU)
#pragma unroll
  for (int r = 0; r < 3; r ++)
#pragma unroll
    for (int c = 0; c < 3; c ++)
      X[r + 3*c] = dF[r + 3*c] - (Y[r]*dF[3*c] + Y[r + 3]*dF[3*c + 1] + Y[r + 6]*dF[3*c + 2]);
}

} // namespace sfgs
