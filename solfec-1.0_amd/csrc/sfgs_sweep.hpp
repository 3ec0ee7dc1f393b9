// sfgs_sweep.hpp -- device code of the colour-major Gauss-Seidel sweep and of
// the merit pass, shared by the per-colour kernels (sfgs_kernels.hip) and the
// persistent batched kernel (sfgs_batch.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "sfgs_ctx.hpp"
#include "sfgs_math.hpp"

namespace sfgs {

static const int TPB = 256;          // threads per block (4 wavefronts)
static const int SLICE = 64;         // rows per slice (one wavefront)

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// =====================================================================
// Gauss-Seidel sweep of one colour (bgs.c:950-1019) with the merit of the
// previous iteration fused in (mrf.c:35-184)
//
// R lives in two buffers.  Sweep k reads P (R at the end of sweep k-1, all
// rows) and writes Q.  Row i gathers Q_j for neighbours already updated in
// this sweep (permuted index in [upd_lo, upd_hi)) and P_j otherwise, which is
// the serial colour-major Gauss-Seidel order.  When the merit is on, sweep
// k >= 1 also forms U_i = B_i + W_ii P_i + sum_j W_ij P_j, i.e. the merit
// update of U after iteration k-1 (mrf.c:61-76), accumulates C'AC for it, keeps
// that U in Um and starts the local solve from it, exactly as the reference's
// next sweep does after MERIT_Function.  The termination test of iteration k-1
// therefore completes after sweep k; when it stops, P and Um are the state.
// G lanes cooperate on one row (blocks k = g, g+G, ...), reduce B' across the
// group with cross-lane adds, and run the local solve redundantly; lane g = 0
// writes.
// =====================================================================

template <typename T>
struct SweepArgs {
  const int *row0, *nrows, *rowlen;   // row0, nrows, slen: as in tab
  const int *rowoff;    // first block of each row in its slice
  const int *slen;
  const SliceTab *tab;
  const T *W;
  const int *wcol;
  const T *Wd, *B, *rho, *fri, *coh, *shift;
  const double *A;      // merit weights (FP64 sweeps)
  const float4 *rec;    // FP32 sweeps: the row records (B, law, W_ii, A; k_rec32); the merit arithmetic stays FP64
  const unsigned char *sep;
  const T *P;
  T *Q, *U, *Um;
  const T *Uin;         // local-solver start U (U itself except in the dataflow schedule)
  int n;
  T diageps;
  int diagmaxiter, diagsolver, failure;
  int store_U;          // write the local solver's U; a merit sweep's U is not the final state unless
                        // the solve can abort inside it (FAILURE_EXIT), then U is that state
  int store_Um;         // write the merit pass's U (Um); a caller that forms the final U = B + W R
                        // afterwards (k_merit with update_U) leaves it off
  double *partials;     // 3 per block: errup, errlo, merit numerator
  unsigned long long *failkey;
  int *failcount;
  Ctrl *ctrl;
};

template <int G, typename T>
__device__ __forceinline__ T gsum(T v)
{
  if (G >= 2) v += __shfl_xor(v, 1, 64);
  if (G >= 4) v += __shfl_xor(v, 2, 64);
  if (G >= 8) v += __shfl_xor(v, 4, 64);
  if (G >= 16) v += __shfl_xor(v, 8, 64);
  return v;
}

// deterministic block sum of three values over a block of NT threads; thread 0
// returns them (the shared slots may be reused after the next barrier)
template <int NT = TPB>
__device__ __forceinline__ void block_sum3(double &a, double &b, double &c)
{
  __shared__ double sa[NT/64], sb[NT/64], sc[NT/64];
  a = wave_sum(a); b = wave_sum(b); c = wave_sum(c);
  int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sa[w] = a; sb[w] = b; sc[w] = c; }
  __syncthreads();
  if (threadIdx.x == 0)
  {
    a = sa[0]; b = sb[0]; c = sc[0];
    for (int k = 1; k < NT/64; k ++) { a += sa[k]; b += sb[k]; c += sc[k]; }
  }
}

// Reactions shared between wavefronts of one persistent launch (the dataflow
// schedule) are read and written with device-scope relaxed atomics: those bypass
// the per-XCD L2's stale lines without the cache-wide write-back / invalidate
// that a device-scope fence costs.  Ordinary accesses otherwise.
template <bool COH, typename T>
__device__ __forceinline__ T r_ld(const T *p)
{
  if (COH) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return *p;
}

template <bool COH, typename T>
__device__ __forceinline__ void r_st(T *p, T v)
{
  if (COH) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}

// ---- the gather of a slice: sum_j W_ij x_j of its rows ----
//
// The blocks of a slice are stored row after row without gaps, block q in lane
// q mod 64 of slot q / 64, so a wavefront reads them one per lane whatever the
// rows' lengths: no padding but in the last slot (the slices of a 200k packing
// were one third padding with a fixed number of slots per row), every load full,
// and few load instructions, which is what this phase is bound by: a slice of 32
// rows with 7.4 blocks each takes 4 slots of 9 + 1 coalesced loads and a gather of
// 16-byte reactions.  Each lane forms its block's product and leaves it in LDS;
// then the G lanes of a row add the row's products, lane g those of blocks g,
// g + G, ..., in that order, so that the sums do not depend on the layout.
// CS slots are in flight together, the indices ahead of the blocks and nothing
// else waited for (straight-line code per number of slots: branches around single
// slots, or zeros merged into a lane without a row, cost a wait each and made this
// slower than the padded layout).  A slice with more slots goes round again; six
// (FP32) and four (FP64) hold most slices in one round within the registers of
// three and two wavefronts per SIMD.  1000 mixed sweeps of a 200k-sphere packing
// (417k rows): the whole step 158.5 -> 135.4 ms, 500 FP64 ones 138.7 -> 126.6 ms,
// 64 scenes of 628k rows, 300 mixed sweeps, 84.6 -> 72.6 ms; clock cycles of this
// phase in a large colour 14-16k -> 9-11k (FP32), 22-37k -> 13k (FP64).
template <typename T> struct Gather {
  static const int CS = sizeof(T) == 8 ? 4 : 6;   // slots in flight
  static const int CB = CS*SLICE;
  static const int LDS2 = 6*CB, LDS1 = 3*CB;      // LDS values per wavefront: two products of a block, or one
};

// reaction (or other 3-vector) j at x + S j: 16-byte loads where the stride keeps them aligned
template <bool COH, int S, typename T>
__device__ __forceinline__ void load3(const T *x, int j, T (&v)[3])
{
  const T *p = x + (size_t)S*j;
  if constexpr (!COH && S == 4 && sizeof(T) == 4)
  {
    const float4 q = *reinterpret_cast<const float4 *>(p);
    v[0] = q.x; v[1] = q.y; v[2] = q.z;
  }
  else if constexpr (!COH && S == 4)
  {
    const double2 q = *reinterpret_cast<const double2 *>(p);
    v[0] = q.x; v[1] = q.y; v[2] = p[2];
  }
  else { v[0] = r_ld<COH>(p); v[1] = r_ld<COH>(p + 1); v[2] = r_ld<COH>(p + 2); }
}

__device__ __forceinline__ void wave_lds_fence()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// N slots: each lane's block times its reaction(s), into d[c CB + 64 q] (slot q)
template <typename T, int N, bool TWO, bool COH, int S>
__device__ __forceinline__ void gather_slots(const T *W, const int *cb, const T *P, const T *Q, int upd_lo, int upd_hi,
                                             T *d)
{
  constexpr int CB = Gather<T>::CB;
  int jj[N];
  T wv[N][9], rv[N][3], pv[N][3];
#pragma unroll
  for (int q = 0; q < N; q ++) jj[q] = cb[q*SLICE];
#pragma unroll
  for (int q = 0; q < N; q ++)
#pragma unroll
    for (int e = 0; e < 9; e ++) wv[q][e] = W[(9*q + e)*SLICE];
  // the block loads ahead of the first wait for the indices
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < N; q ++)
  {
    const int j = jj[q];
    load3<COH, S>(j >= upd_lo && j < upd_hi ? Q : P, j, rv[q]);
    if (TWO) load3<COH, S>(P, j, pv[q]);
  }
#pragma unroll
  for (int q = 0; q < N; q ++)
#pragma unroll
    for (int c = 0; c < 3; c ++)
    {
      // explicit fused multiply-adds: the same rounding wherever this is inlined
      d[c*CB + q*SLICE] = fma(wv[q][6 + c], rv[q][2], fma(wv[q][3 + c], rv[q][1], wv[q][c]*rv[q][0]));
      if (TWO) d[(3 + c)*CB + q*SLICE] = fma(wv[q][6 + c], pv[q][2], fma(wv[q][3 + c], pv[q][1], wv[q][c]*pv[q][0]));
    }
}

// sums b of W_ij (upd ? Q : P)_j over the row's blocks and, when TWO, u of
// W_ij P_j.  off and total (wave-uniform): the slice's first block slot and its
// number of blocks; rs, len: the row's first block and their number and
// whether the lane has a row.  The sums over the G lanes are complete on return.
template <typename T, int G, bool TWO, bool COH, int S>
__device__ __forceinline__ void gather_rows(const T *W, const int *wcol, long long off, int total, int rs, int len,
                                            bool act, const T *P, const T *Q, int upd_lo, int upd_hi, T *lds,
                                            T (&b)[3], T (&u)[3])
{
  constexpr int CS = Gather<T>::CS, CB = Gather<T>::CB;
  const int l = threadIdx.x & 63, g = l % G, ns = (total + SLICE - 1) / SLICE;
  const T *Wb = W + 9*off + l;
  const int *cb = wcol + off + l;
#pragma unroll
  for (int c = 0; c < 3; c ++) b[c] = u[c] = T(0);
  int k = g;
  for (int m0 = 0; m0 < ns; m0 += CS)
  {
    const T *Wm = Wb + 9*m0*SLICE;
    const int *cm = cb + m0*SLICE;
    // straight-line code per number of slots: all loads of a round in flight
    switch (min(ns - m0, CS))
    {
    case 1: gather_slots<T, 1, TWO, COH, S>(Wm, cm, P, Q, upd_lo, upd_hi, lds + l); break;
    case 2: gather_slots<T, 2, TWO, COH, S>(Wm, cm, P, Q, upd_lo, upd_hi, lds + l); break;
    case 3: gather_slots<T, 3, TWO, COH, S>(Wm, cm, P, Q, upd_lo, upd_hi, lds + l); break;
    case 4: gather_slots<T, 4, TWO, COH, S>(Wm, cm, P, Q, upd_lo, upd_hi, lds + l); break;
    case 5: if constexpr (CS >= 5) gather_slots<T, 5, TWO, COH, S>(Wm, cm, P, Q, upd_lo, upd_hi, lds + l); break;
    default: if constexpr (CS >= 6) gather_slots<T, 6, TWO, COH, S>(Wm, cm, P, Q, upd_lo, upd_hi, lds + l); break;
    }
    wave_lds_fence();
    // rs and len may still be in flight: not used, nor hoisted, before here
    int rr = rs, ln = len;
    asm volatile("" : "+v"(rr), "+v"(ln));
    const int end = act ? min(ln, m0*SLICE + CB - rr) : 0, base = rr - m0*SLICE;
    for (; k < end; k += 4*G)
    {
      T t[4][6];
#pragma unroll
      for (int q = 0; q < 4; q ++)
      {
        const T *d = lds + base + min(k + q*G, end - 1);
#pragma unroll
        for (int c = 0; c < (TWO ? 6 : 3); c ++) t[q][c] = d[c*CB];
      }
#pragma unroll
      for (int q = 0; q < 4; q ++)
        if (k + q*G < end)
        {
#pragma unroll
          for (int c = 0; c < 3; c ++) { b[c] += t[q][c]; if (TWO) u[c] += t[q][3 + c]; }
        }
    }
    // the last round may have stepped past the chunk: back to the lane's first block beyond it
    if (k > end) k = end > g ? g + (end - g + G - 1)/G*G : g;
    wave_lds_fence();
  }
#pragma unroll
  for (int c = 0; c < 3; c ++) { b[c] = gsum<G>(b[c]); if (TWO) u[c] = gsum<G>(u[c]); }
}

// One slice (up to 64/G rows of one colour, one wavefront) of a sweep; false when *stop
// (a solve that has stopped; null: none) left it untouched.  eu, el and
// up receive this lane's contributions to the error sums and to the merit
// numerator.  A failed local solve is recorded in failkey / failcount, keyed by
// the sweep number *sweepno, and raises *abortflag under FAILURE_EXIT.  The flag
// is read together with the slice table, so both cost one memory round trip.
// COH: P and Q are shared with other wavefronts of the same launch (r_ld / r_st).
// tabs: a.tab, apart from a so that a kernel may have it among its first arguments.
// lds: this wavefront's Gather<T>::LDS2 (merit) or LDS1 values.  s and valid are
// the same in all lanes of the wavefront.
template <typename T, int G, bool MERIT, bool COH = false>
__device__ __forceinline__ bool sweep_slice(const SweepArgs<T> &a, const SliceTab *tabs, int s, bool valid, int upd_lo, int upd_hi,
                                            int backward, const int *sweepno, unsigned long long *failkey,
                                            int *failcount, int *abortflag, double &eu, double &el, double &up,
                                            T *lds, const int *stop = nullptr)
{
  const int l = threadIdx.x & 63, r = l / G, g = l % G;
  const int n = a.n;
  if (!__builtin_amdgcn_readfirstlane(valid)) return !(stop && *stop);
  s = __builtin_amdgcn_readfirstlane(s);
  const SliceTab tab = tabs[s];
  const int stopped = __builtin_amdgcn_readfirstlane(stop ? *stop : 0);
  const int nr = __builtin_amdgcn_readfirstlane(tab.nrows), r0 = __builtin_amdgcn_readfirstlane(tab.row0);
  const int total = __builtin_amdgcn_readfirstlane(tab.blocks);
  const long long off = (long long)__builtin_amdgcn_readfirstlane((int)(tab.off >> 32)) << 32 |
                        (unsigned)__builtin_amdgcn_readfirstlane((int)tab.off);
  // all of them loaded here, none behind the branch
  asm volatile("" :: "s"(nr), "s"(r0), "s"(total), "s"(off), "s"(stopped));
  if (stopped) return false;
  const bool act = r < nr;
  // The row's own data first, so that its loads are in flight with the gather's.
  // Nothing is computed from them before the gather (a use waits for them), and
  // lanes without a row load the last one's (so would a merge of two paths).
  const int p = r0 + min(r, nr - 1), rs = a.rowoff[p], len = a.rowlen[p];
  T Bi[3], Wi[9], R[3], U[3], A64[9];
  float4 rec[5];
  RowLaw<T> L;
  unsigned char sep = 0;
  if constexpr (sizeof(T) == 4)
  {
    // the row record: five 16-byte loads (k_rec32)
#pragma unroll
    for (int k = 0; k < 5; k ++) rec[k] = a.rec[5*(size_t)p + k];
  }
  else
  {
    Bi[0] = a.B[p]; Bi[1] = a.B[(size_t)n + p]; Bi[2] = a.B[2*(size_t)n + p];
#pragma unroll
    for (int e = 0; e < 9; e ++) Wi[e] = a.Wd[(size_t)e*n + p];
    if (MERIT)
    {
#pragma unroll
      for (int e = 0; e < 9; e ++) A64[e] = a.A[(size_t)e*n + p];
    }
    L = RowLaw<T>{a.fri[p], a.coh[p], a.shift[p], a.rho[p], false};
    sep = a.sep[p];
  }
  load3<COH, 4>(a.P, p, R);
  if (!MERIT)
  {
#pragma unroll
    for (int k = 0; k < 3; k ++) U[k] = a.Uin[(size_t)k*n + p];
  }
  T b[3], u[3];
  gather_rows<T, G, MERIT, COH, 4>(a.W, a.wcol, off, total, rs, len, act, a.P, a.Q, upd_lo, upd_hi, lds, b, u);

  if (act)
  {
    double Ai[9];
    if constexpr (sizeof(T) == 4)
    {
      Bi[0] = rec[0].x; Bi[1] = rec[0].y; Bi[2] = rec[0].z;
      const int ls = __float_as_int(rec[1].w);
      L = RowLaw<T>{rec[1].x, rec[1].y, rec[1].z, rec[0].w, (ls & 1) != 0};
      Wi[0] = rec[2].x; Wi[1] = Wi[3] = rec[2].y; Wi[2] = Wi[6] = rec[2].z; Wi[4] = rec[2].w;
      Wi[5] = Wi[7] = rec[3].x; Wi[8] = rec[3].y;
      if (MERIT)
      {
        Ai[0] = rec[3].z; Ai[1] = Ai[3] = rec[3].w; Ai[2] = Ai[6] = rec[4].x;
        Ai[4] = rec[4].y; Ai[5] = Ai[7] = rec[4].z; Ai[8] = rec[4].w;
      }
    }
    else
    {
      L.separated = sep != 0;
      if (MERIT)
      {
#pragma unroll
        for (int e = 0; e < 9; e ++) Ai[e] = A64[e];
      }
    }
    T Bp[3] = {Bi[0] + b[0], Bi[1] + b[1], Bi[2] + b[2]};
    const T R0[3] = {R[0], R[1], R[2]};
    if (MERIT)
    {
      // merit of the previous iteration at this row (mrf.c:63-84)
      mv_add(Bi, Wi, R, U);
      U[0] += u[0]; U[1] += u[1]; U[2] += u[2];
      // the merit is evaluated in FP64 whatever the sweep type
      double C[3], Ud[3] = {U[0], U[1], U[2]}, Rd[3] = {R[0], R[1], R[2]};
      merit_residual(L.fri, L.coh, L.shift, Ud, Rd, C);
      const double q0 = Ai[0]*C[0] + Ai[3]*C[1] + Ai[6]*C[2];
      const double q1 = Ai[1]*C[0] + Ai[4]*C[1] + Ai[7]*C[2];
      const double q2 = Ai[2]*C[0] + Ai[5]*C[1] + Ai[8]*C[2];
      if (g == 0)
      {
        up += q0*C[0] + q1*C[1] + q2*C[2];
        if (a.store_Um)
        {
#pragma unroll
          for (int k = 0; k < 3; k ++) a.Um[(size_t)k*n + p] = U[k];
        }
      }
    }

    int d = local_solve(a.diagsolver, L, a.diageps, a.diagmaxiter, Wi, Bp, U, R);
    if (d >= a.diagmaxiter || d < 0)
    {
      if (g == 0)
      {
        unsigned code = d < 0 ? SFGS_GS_DIAGONAL_FAILED : SFGS_GS_DIAGONAL_DIVERGED;
        unsigned long long pos = backward ? (unsigned long long)(n - 1 - p) : (unsigned long long)p;
        atomicMax(failkey, ((unsigned long long)(r_ld<COH>(sweepno) + 1) << 40) | (pos << 2) | code);
        atomicAdd(failcount, 1);
        if (a.failure == SFGS_FAILURE_EXIT) atomicExch(abortflag, 1);
      }
      if (a.failure == SFGS_FAILURE_CONTINUE)
      {
        const int chain[4] = {SFGS_DS_SEMISMOOTH_NEWTON, SFGS_DS_PROJECTED_GRADIENT,
                              SFGS_DS_DE_SAXCE_FENG, SFGS_DS_PROJECTED_NEWTON};
        for (int c = 0; c < 4; c ++)
        {
          if (chain[c] == a.diagsolver) continue;
          R[0] = R0[0]; R[1] = R0[1]; R[2] = R0[2];
          d = local_solve(chain[c], L, a.diageps, a.diagmaxiter, Wi, Bp, U, R);
          if (d < a.diagmaxiter && d >= 0) break;
        }
        if (d >= a.diagmaxiter || d < 0) { R[0] = R0[0]; R[1] = R0[1]; R[2] = R0[2]; }
      }
    }
    if (g == 0)
    {
      if constexpr (sizeof(T) == 4 && !COH)
        *reinterpret_cast<float4 *>(a.Q + 4*(size_t)p) = make_float4(R[0], R[1], R[2], 0.0f);
      else
      {
#pragma unroll
        for (int k = 0; k < 3; k ++) r_st<COH>(a.Q + 4*(size_t)p + k, R[k]);
        r_st<COH>(a.Q + 4*(size_t)p + 3, T(0));
      }
      if (!MERIT || a.store_U)
      {
#pragma unroll
        for (int k = 0; k < 3; k ++) a.U[(size_t)k*n + p] = U[k];
      }
      const double d0 = (double)R[0] - R0[0], d1 = (double)R[1] - R0[1], d2 = (double)R[2] - R0[2];
      eu += d0*d0 + d1*d1 + d2*d2;
      el += (double)R[0]*R[0] + (double)R[1]*R[1] + (double)R[2]*R[2];
    }
  }
  return true;
}

// standalone merit (MERIT_Function with update_U, mrf.c:35-184) on the
// canonical R buffer; one launch over all slices
struct MeritArgs {
  const SliceTab *tab;
  const int *rowlen, *rowoff;
  const double *W;
  const int *wcol;
  const double *Wd, *A, *B, *fri, *coh, *shift;
  const double *R;
  double *U;
  int n, update_U;
  double *mpartials;
  double *conmerit;   // may be null: per-row C'AC (colour-major)
  const int *stop;    // may be null: nonzero leaves everything as it is
};

// merit terms C'AC of the rows of one slice, added to up (lane g = 0 of each
// row); lds: this wavefront's Gather<double>::LDS1 values.  A wavefront's time is
// its chain of loads, so the slice comes as one table entry and the row's data but
// for A go out ahead of the gather: 26.6 us at 133k rows (108 MB, 21 us at 5.2 TB/s).
template <int G>
__device__ __forceinline__ void merit_slice(const MeritArgs &a, int s, bool valid, double &up, double *lds)
{
  const int l = threadIdx.x & 63, r = l / G, g = l % G;
  const int n = a.n;
  if (!__builtin_amdgcn_readfirstlane(valid)) return;
  s = __builtin_amdgcn_readfirstlane(s);
  const SliceTab tab = a.tab[s];
  const int stopped = a.stop ? *a.stop : 0;
  const int nr = __builtin_amdgcn_readfirstlane(tab.nrows), r0 = __builtin_amdgcn_readfirstlane(tab.row0);
  const int total = __builtin_amdgcn_readfirstlane(tab.blocks);
  const long long off = (long long)__builtin_amdgcn_readfirstlane((int)(tab.off >> 32)) << 32 |
                        (unsigned)__builtin_amdgcn_readfirstlane((int)tab.off);
  if (__builtin_amdgcn_readfirstlane(stopped)) return;
  const bool act = r < nr;
  const int p = r0 + min(r, nr - 1), rs = a.rowoff[p], len = a.rowlen[p];
  double R[3], Wi[9], Bv[3], U[3], fri = a.fri[p], coh = a.coh[p], shift = a.shift[p];
  load3<false, 4>(a.R, p, R);
  if (a.update_U)
  {
#pragma unroll
    for (int k = 0; k < 3; k ++) Bv[k] = a.B[(size_t)k*n + p];
#pragma unroll
    for (int e = 0; e < 9; e ++) Wi[e] = a.Wd[(size_t)e*n + p];
    // the sweep's multiply-adds (sweep_slice), so that U equals the fused merit pass's
    double u[3], none[3];
    gather_rows<double, G, false, false, 4>(a.W, a.wcol, off, total, rs, len, act, a.R, a.R, 0, 0, lds, u, none);
    mv_add(Bv, Wi, R, U);
    U[0] += u[0]; U[1] += u[1]; U[2] += u[2];
    if (act && g == 0)
#pragma unroll
      for (int k = 0; k < 3; k ++) a.U[(size_t)k*n + p] = U[k];
  }
  else
  {
#pragma unroll
    for (int k = 0; k < 3; k ++) U[k] = a.U[(size_t)k*n + p];
  }
  if (!act) return;
  double C[3], Ai[9];
#pragma unroll
  for (int e = 0; e < 9; e ++) Ai[e] = a.A[(size_t)e*n + p];
  merit_residual(fri, coh, shift, U, R, C);
  const double q0 = Ai[0]*C[0] + Ai[3]*C[1] + Ai[6]*C[2];
  const double q1 = Ai[1]*C[0] + Ai[4]*C[1] + Ai[7]*C[2];
  const double q2 = Ai[2]*C[0] + Ai[5]*C[1] + Ai[8]*C[2];
  if (g == 0)
  {
    const double t = q0*C[0] + q1*C[1] + q2*C[2];
    up += t;
    if (a.conmerit) a.conmerit[p] = t;
  }
}

} // namespace sfgs
