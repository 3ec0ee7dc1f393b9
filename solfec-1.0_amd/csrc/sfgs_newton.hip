// sfgs_newton.hip -- the NEWTON_SOLVER (nts.c) on the assembled local dynamics
// of a context: a projected semismooth Newton method over all contacts at once,
// each step a linear solve by flexible GMRES (or a per-row "diagonalised"
// step), then the Gauss-Seidel solve as the fallback of an unconverged run.
//
// Vectors of the Newton step are 3 doubles per row in the colour-major row
// order of the store, so the W products reuse the slices the sweeps
// stream.  The kernels:
//   k_nt_lin     per row: C(U, R), X = dC/dU, Y = dC/dR of the smoothed cone
//                residual (scf.c:28-133), b = -C, T = X W_ii + Y
//                (nts.c:1072-1081); GMRES: P = (T + delta I)^-1
//                (nts.c:1095-1103); DIAG: T d = b, dr = (1 - theta) dr +
//                theta d, R = proj(R + dr) (nts.c:1084-1093)
//   k_nt_matvec  y = beta y + alpha (X (W x) + Y x) + alpha delta x: the
//                operator of the linear step (Matvec, nts.c:584-652), W x
//                by the gather of the sweeps (gather_rows)
//   k_nt_dot     deterministic per-block partial sums of x'y, into host memory
//                (the host adds them in block order)
//   k_nt_mgs     one step of modified Gram-Schmidt, with the dot product of
//                the next; k_nt_arnoldi the end of an Arnoldi step (norm,
//                scaling, Givens update); k_nt_start and k_nt_cycle the start
//                and the end of a cycle (ext/krylov/flexgmres.c)
//   k_nt_axpy, k_nt_precond, k_nt_update  the other vector work of flexible
//                GMRES and R = proj(R + dr)
// The diagonal solve runs its loop on the device (NtCtl); the GMRES driver runs on the
// host, with the Arnoldi steps and the Hessenberg system (at most 21 x 20) on the
// device and one wait per step for the residual estimate.  All of this is HBM-bound
// vector work (a W product streams the same bytes as a sweep); the sweeps remain the
// solver of the hot path.
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstring>
#include <cfloat>
#include <vector>
#include <algorithm>
#include "sfgs_ctx.hpp"
#include "sfgs_math.hpp"
#include "sfgs_host.hpp"

using namespace sfgs;

namespace {

#define NT_DISPATCH_G(G, CALL) \
  switch (G) { \
  case 1: { constexpr int GG = 1; CALL; } break; \
  case 2: { constexpr int GG = 2; CALL; } break; \
  case 8: { constexpr int GG = 8; CALL; } break; \
  default: { constexpr int GG = 4; CALL; } break; }

constexpr int NT_KDIM = 20;        // hypre_FlexGMRESCreate default k_dim (flexgmres.c:91)
constexpr int NT_DOT_BLOCKS = 256; // most partials of one dot product
static_assert(NT_DOT_BLOCKS <= TPB, "nt_dot_sum: one partial per thread");

struct NtRows {
  int n;
  const double *R;      // 4 per row
  const double *U;      // SoA planes
  const double *Wd;     // SoA planes
  const double *fri, *coh, *shift;
  double *X, *Y, *P;    // SoA planes, 9 per row
  double *b, *dr;       // 3 per row
  int *singular;
};

// The control block of a diagonal Newton solve, whose loop is tested on the device:
// the host enqueues iterations ahead and reads this once per batch of them.  With a
// read-back of the merit's partial sums an iteration each took 70 us at 133k rows,
// 43 us of them on the device; now
// 200 iterations take 9.6 ms on the device, the whole solve 12.0 ms in place of 15.4.
struct NtCtl {
  // RING merits are kept; the host reads them once per batch of at most BATCH iterations
  static constexpr int RING = 64, BATCH = 32;
  static_assert(BATCH <= RING, "a batch's merits are read before they are overwritten");
  int done, iters, nan;
  double merit;
  double hist[RING];     // merit of iteration k at k % RING
};

struct NtTest {
  NtCtl *ctl;            // null: no test
  int k;                 // iterations before this launch
  const double *part;    // the merit's partial sums after them
  int np, maxiter;
  double lo, meritval;
};

// the test of the loop after iteration k (nts.c:1199-1223), taken by every
// workgroup alike from the same sums; workgroup 0 keeps the record.  True when the
// loop has ended.
__device__ __forceinline__ bool nt_test(const NtTest &t)
{
  __shared__ int ended;
  double s = 0.0, z1 = 0.0, z2 = 0.0;
  for (int k = threadIdx.x; k < t.np; k += TPB) s += t.part[k];
  block_sum3(s, z1, z2);
  if (threadIdx.x == 0)
  {
    // the loop's end in an earlier launch; one that workgroup 0 of this launch has
    // written already is what this workgroup finds as well
    int done = __hip_atomic_load(&t.ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!done && t.k > 0)
    {
      const double merit = 0.5*s/t.lo;
      const int nan = merit != merit;
      done = nan || t.k >= t.maxiter || !(merit > t.meritval);
      if (blockIdx.x == 0)
      {
        t.ctl->merit = merit;
        t.ctl->nan = nan;
        if (!nan) { t.ctl->iters = t.k; t.ctl->hist[(t.k - 1) % NtCtl::RING] = merit; }
        if (done) __hip_atomic_store(&t.ctl->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    ended = done;
  }
  __syncthreads();
  return ended != 0;
}

__global__ __launch_bounds__(TPB) void k_nt_lin(NtRows a, int diag, double omega, double delta, double theta,
                                                 double *Rw, NtTest test)
{
  if (test.ctl && nt_test(test)) return;
  const int p = blockIdx.x*blockDim.x + threadIdx.x;
  if (p >= a.n) return;
  const int n = a.n;
  double R[3], U[3], W[9], C[3], X[9], Y[9], T[9];
#pragma unroll
  for (int k = 0; k < 3; k ++) { R[k] = a.R[4*(size_t)p + k]; U[k] = a.U[(size_t)k*n + p]; }
#pragma unroll
  for (int e = 0; e < 9; e ++) W[e] = a.Wd[(size_t)e*n + p];
  const double fri = a.fri[p], coh = a.coh[p];
  scf_linearize_smooth(fri, coh, a.shift[p], omega, U, R, C, X, Y);
  double b[3] = {-C[0], -C[1], -C[2]};
#pragma unroll
  for (int r = 0; r < 3; r ++)
#pragma unroll
    for (int c = 0; c < 3; c ++)
      T[r + 3*c] = (X[r]*W[3*c] + X[r + 3]*W[3*c + 1] + X[r + 6]*W[3*c + 2]) + Y[r + 3*c];
  if (diag)
  {
    if (solve3(T, b)) { atomicAdd(a.singular, 1); b[0] = b[1] = b[2] = 0.0; }
    const double gamma = 1.0 - theta;
    double d[3];
#pragma unroll
    for (int k = 0; k < 3; k ++)
    {
      d[k] = gamma*a.dr[3*(size_t)p + k] + theta*b[k];
      a.dr[3*(size_t)p + k] = d[k];
      R[k] += d[k];
    }
    double Rp[3];
    scf_project(fri, coh, R, Rp);
#pragma unroll
    for (int k = 0; k < 3; k ++) Rw[4*(size_t)p + k] = Rp[k];
    return;
  }
  T[0] += delta; T[4] += delta; T[8] += delta;
  double Pm[9];
  if (inverse3(T, Pm)) atomicAdd(a.singular, 1);
#pragma unroll
  for (int e = 0; e < 9; e ++)
  {
    a.X[(size_t)e*n + p] = X[e];
    a.Y[(size_t)e*n + p] = Y[e];
    a.P[(size_t)e*n + p] = Pm[e];
  }
#pragma unroll
  for (int k = 0; k < 3; k ++) a.b[3*(size_t)p + k] = b[k];
}

struct NtMat {
  const int *row0, *nrows, *rowlen, *rowoff, *slen;
  const long long *off;
  const double *W;
  const int *wcol;
  const double *Wd, *X, *Y;
  int n;
  double delta;
};

template <int G>
__global__ __launch_bounds__(TPB) void k_nt_matvec(NtMat a, int nslices, double alpha, const double *x, double beta,
                                                    double *y)
{
  const int sl = blockIdx.x*(TPB/SLICE) + (threadIdx.x >> 6);
  if (sl >= nslices) return;   // uniform over the wavefront
  const int l = threadIdx.x & 63, r = l / G, g = l % G, n = a.n;
  const int s = __builtin_amdgcn_readfirstlane(sl);
  const bool act = r < a.nrows[s];
  const int p = a.row0[s] + (act ? r : 0), len = a.rowlen[p], rs = a.rowoff[p];
  __shared__ double lds[TPB/SLICE][Gather<double>::LDS1];
  double zz[3], none[3];
  gather_rows<double, G, false, false, 3>(a.W, a.wcol, a.off[s], a.slen[s], rs, len, act, x, x, 0, 0, lds[threadIdx.x >> 6],
                                          zz, none);
  if (!act || g != 0) return;
  const double xp[3] = {x[3*(size_t)p], x[3*(size_t)p + 1], x[3*(size_t)p + 2]};
  double Wi[9], X[9], Y[9];
#pragma unroll
  for (int e = 0; e < 9; e ++)
  {
    Wi[e] = a.Wd[(size_t)e*n + p];
    X[e] = a.X[(size_t)e*n + p];
    Y[e] = a.Y[(size_t)e*n + p];
  }
  const double z[3] = {Wi[0]*xp[0] + Wi[3]*xp[1] + Wi[6]*xp[2] + zz[0],
                       Wi[1]*xp[0] + Wi[4]*xp[1] + Wi[7]*xp[2] + zz[1],
                       Wi[2]*xp[0] + Wi[5]*xp[1] + Wi[8]*xp[2] + zz[2]};
  const double ad = alpha*a.delta;
#pragma unroll
  for (int k = 0; k < 3; k ++)
  {
    const double u = (X[k]*z[0] + X[k + 3]*z[1] + X[k + 6]*z[2]) + (Y[k]*xp[0] + Y[k + 3]*xp[1] + Y[k + 6]*xp[2]);
    double q = beta*y[3*(size_t)p + k];
    q = q + alpha*u;
    y[3*(size_t)p + k] = q + ad*xp[k];
  }
}

__global__ __launch_bounds__(TPB) void k_nt_dot(long long N, const double *a, const double *b, double *part)
{
  double s = 0.0, z1 = 0.0, z2 = 0.0;
  for (long long i = (long long)blockIdx.x*TPB + threadIdx.x; i < N; i += (long long)gridDim.x*TPB) s += a[i]*b[i];
  block_sum3(s, z1, z2);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_nt_axpy(long long N, double alpha, const double *x, double *y)
{
  const long long i = (long long)blockIdx.x*blockDim.x + threadIdx.x;
  if (i < N) y[i] += alpha*x[i];
}

__global__ void k_nt_precond(int n, const double *P, const double *b, double *x)
{
  const int p = blockIdx.x*blockDim.x + threadIdx.x;
  if (p >= n) return;
  const double q[3] = {b[3*(size_t)p], b[3*(size_t)p + 1], b[3*(size_t)p + 2]};
#pragma unroll
  for (int r = 0; r < 3; r ++)
    x[3*(size_t)p + r] = P[(size_t)r*n + p]*q[0] + P[(size_t)(r + 3)*n + p]*q[1] + P[(size_t)(r + 6)*n + p]*q[2];
}

// R = proj(R + dr) (nts.c:1139-1154)
__global__ void k_nt_update(int n, double *R, const double *dr, const double *fri, const double *coh)
{
  const int p = blockIdx.x*blockDim.x + threadIdx.x;
  if (p >= n) return;
  double S[3], Rp[3];
#pragma unroll
  for (int k = 0; k < 3; k ++) S[k] = R[4*(size_t)p + k] + dr[3*(size_t)p + k];
  scf_project(fri[p], coh[p], S, Rp);
#pragma unroll
  for (int k = 0; k < 3; k ++) R[4*(size_t)p + k] = Rp[k];
}

// the Arnoldi scalars of one GMRES cycle live on the device: the Hessenberg
// matrix hh (row-major, (k_dim + 1) x k_dim), the right-hand side rs and the
// Givens rotations c, s, and the last residual estimate
struct NtScal {
  double hh[(NT_KDIM + 1)*NT_KDIM];
  double rs[NT_KDIM + 1], c[NT_KDIM], s[NT_KDIM];
  double rnorm;
};

// the sum of a dot product's block partials, in a fixed order, in all threads
__device__ __forceinline__ double nt_dot_sum(const double *part, int np)
{
  __shared__ double sum;
  double v = threadIdx.x < np ? part[threadIdx.x] : 0.0, z1 = 0.0, z2 = 0.0;
  block_sum3(v, z1, z2);
  if (threadIdx.x == 0) sum = v;
  __syncthreads();
  v = sum;
  __syncthreads();   // before the slots' next use
  return v;
}

// One modified Gram-Schmidt step: y -= h x0 with h the dot product whose partial
// sums the launch before left in p0 (kept in *out; x0 null: no update), then the
// partial sums of x1 . y (x1 null: of y . y) into p1.  A step is bound by its
// launches (3-4 us each for 124k values), so the update, the sum of the partials and the
// next product are one launch instead of three, the step's end one
// instead of five, and what the host needs is written to its memory: 12 linearisations of
// 41k contacts in body space with 62 steps took 10.6 ms and take 6.8.
__global__ __launch_bounds__(TPB) void k_nt_mgs(long long N, const double *x0, const double *p0, double *out,
                                                 const double *x1, double *y, double *p1)
{
  const double h = x0 ? nt_dot_sum(p0, gridDim.x) : 0.0, mh = -1.0*h;
  if (x0 && blockIdx.x == 0 && threadIdx.x == 0) *out = h;
  double s = 0.0, z1 = 0.0, z2 = 0.0;
  for (long long i = (long long)blockIdx.x*TPB + threadIdx.x; i < N; i += (long long)gridDim.x*TPB)
  {
    double v = y[i];
    if (x0) { v += mh*x0[i]; y[i] = v; }
    s += (x1 ? x1[i] : v)*v;
  }
  block_sum3(s, z1, z2);
  if (threadIdx.x == 0) p1[blockIdx.x] = s;
}

// x *= t, and *rs = r: the start of a cycle
__global__ void k_nt_start(long long N, double t, double *x, double *rs, double r)
{
  const long long i = (long long)blockIdx.x*blockDim.x + threadIdx.x;
  if (i == 0) *rs = r;
  if (i < N) x[i] *= t;
}

// column i - 1 of the Arnoldi step: the previous rotations, a new one, the
// updated right-hand side and the residual estimate |rs[i]| (flexgmres.c:531-557)
__device__ void nt_givens(NtScal *sc, int i)
{
#pragma clang fp contract(off)
  double *hh = sc->hh, *c = sc->c, *s = sc->s, *rs = sc->rs, t;
#define HH(a, b) hh[(a)*NT_KDIM + (b)]
  for (int j = 1; j < i; j ++)
  {
    t = HH(j - 1, i - 1);
    HH(j - 1, i - 1) = s[j - 1]*HH(j, i - 1) + c[j - 1]*t;
    HH(j, i - 1) = -s[j - 1]*t + c[j - 1]*HH(j, i - 1);
  }
  t = HH(i, i - 1)*HH(i, i - 1);
  t += HH(i - 1, i - 1)*HH(i - 1, i - 1);
  double gamma = sqrt(t);
  if (gamma == 0.0) gamma = 1.e-16;
  c[i - 1] = HH(i - 1, i - 1)/gamma;
  s[i - 1] = HH(i, i - 1)/gamma;
  rs[i] = -HH(i, i - 1)*rs[i - 1];
  rs[i] /= gamma;
  rs[i - 1] = c[i - 1]*rs[i - 1];
  HH(i - 1, i - 1) = s[i - 1]*HH(i, i - 1) + c[i - 1]*HH(i - 1, i - 1);
  sc->rnorm = fabs(rs[i]);
#undef HH
}

// the end of Arnoldi step i: its norm from the partial sums of the launch before, y
// scaled by it (unless it is 0), and in workgroup 0 the Givens update; the residual
// estimate goes to the host's memory
__global__ __launch_bounds__(TPB) void k_nt_arnoldi(long long N, const double *part, int np, double *y, NtScal *sc, int i,
                                                     double *rnorm)
{
  const double t = sqrt(nt_dot_sum(part, np));
  if (t != 0.0)
    for (long long k = (long long)blockIdx.x*TPB + threadIdx.x; k < N; k += (long long)gridDim.x*TPB) y[k] *= 1.0/t;
  if (blockIdx.x == 0 && threadIdx.x == 0)
  {
    sc->hh[i*NT_KDIM + i - 1] = t;
    nt_givens(sc, i);
    *rnorm = sc->rnorm;
  }
}

// the end of a cycle of m steps: back-substitution in the Hessenberg system (every
// workgroup for itself; hh and rs stay as they are) and x += sum_j rs_j pre_j
__global__ __launch_bounds__(TPB) void k_nt_cycle(long long N, const NtScal *sc, int m, const double *pre, double *x)
{
  __shared__ double hh[(NT_KDIM + 1)*NT_KDIM], rs[NT_KDIM + 1];
  for (int k = threadIdx.x; k < m*NT_KDIM; k += TPB) hh[k] = sc->hh[k];
  if (threadIdx.x < m) rs[threadIdx.x] = sc->rs[threadIdx.x];
  __syncthreads();
  if (threadIdx.x == 0)
  {
#pragma clang fp contract(off)
    rs[m - 1] = rs[m - 1]/hh[(m - 1)*NT_KDIM + m - 1];
    for (int k = m - 2; k >= 0; k --)
    {
      double t = 0.0;
      for (int j = k + 1; j < m; j ++) t -= hh[k*NT_KDIM + j]*rs[j];
      t += rs[k];
      rs[k] = t/hh[k*NT_KDIM + k];
    }
  }
  __syncthreads();
  for (long long i = (long long)blockIdx.x*TPB + threadIdx.x; i < N; i += (long long)gridDim.x*TPB)
  {
    // explicit multiply-adds: the sums of one vector update after the other
#pragma clang fp contract(off)
    double w = pre[(size_t)(m - 1)*N + i]*rs[m - 1];
    for (int j = m - 2; j >= 0; j --) w = fma(rs[j], pre[(size_t)j*N + i], w);
    x[i] += w;
  }
}

// the device vectors of one Newton solve
struct NtWork {
  sfgs_ctx *ctx;
  int n;
  long long N;
  double *X, *Y, *P, *b, *dr, *R0, *kry, *pre, *r, *part;
  NtScal *sc;
  NtMat mat;
  int bodyspace = 0;
  int matvecs = 0;
  double *hpart;             // in host memory that kernels write: partials of a dot product, a residual estimate

  double *kv(int k) const { return kry + (size_t)k*N; }
  double *pv(int k) const { return pre + (size_t)k*N; }

  int matvec(double alpha, const double *x, double beta, double *y)
  {
    if (bodyspace)
    {
      CHK(bodyspace_product(ctx, x, 3, 0, X, Y, alpha, beta, mat.delta, y));
      matvecs ++;
      return 0;
    }
    const int ns = ctx->nslices, grid = (ns + TPB/SLICE - 1) / (TPB/SLICE);
    if (grid > 0)
      NT_DISPATCH_G(ctx->G_built, auto kern = k_nt_matvec<GG>; hipLaunchKernelGGL(kern, dim3(grid), dim3(TPB), 0,
                       ctx->stream, mat, ns, alpha, x, beta, y));
    matvecs ++;
    HIPCHK(hipGetLastError());
    return 0;
  }

  int dot_grid() const { return std::max(1, std::min(NT_DOT_BLOCKS, nblk(N))); }

  // the partial sums straight into host memory: one wait, no copy
  int dot(const double *a, const double *b2, double &out)
  {
    const int grid = dot_grid();
    hipLaunchKernelGGL(k_nt_dot, dim3(grid), dim3(TPB), 0, ctx->stream, N, a, b2, hpart);
    HIPCHK(hipStreamSynchronize(ctx->stream));
    double s = 0.0;
    for (int k = 0; k < grid; k ++) s += hpart[k];
    out = s;
    return 0;
  }

  // modified Gram-Schmidt of kv(i) against kv(0) .. kv(i - 1), column i - 1 of the
  // Hessenberg matrix, and the Givens update
  void arnoldi(int i)
  {
    const int grid = dot_grid();
    double *p[2] = {part, part + NT_DOT_BLOCKS}, *y = kv(i);
    for (int j = 0; j <= i; j ++)
      hipLaunchKernelGGL(k_nt_mgs, dim3(grid), dim3(TPB), 0, ctx->stream, N, j > 0 ? kv(j - 1) : (const double *)nullptr,
                         (const double *)p[(j + 1) & 1], sc->hh + (j > 0 ? j - 1 : 0)*NT_KDIM + i - 1,
                         j < i ? kv(j) : (const double *)nullptr, y, p[j & 1]);
    hipLaunchKernelGGL(k_nt_arnoldi, dim3(grid), dim3(TPB), 0, ctx->stream, N, (const double *)p[i & 1], grid, y, sc, i,
                       hpart + NT_DOT_BLOCKS);
  }

  void axpy(double alpha, const double *x, double *y)
  {
    if (N > 0) hipLaunchKernelGGL(k_nt_axpy, dim3(nblk(N)), dim3(TPB), 0, ctx->stream, N, alpha, x, y);
  }

  int copy(const double *x, double *y)
  {
    if (N > 0) HIPCHK(hipMemcpyAsync(y, x, sizeof(double)*(size_t)N, hipMemcpyDeviceToDevice, ctx->stream));
    return 0;
  }

  void precond(const double *bb, double *x)
  {
    if (n > 0) hipLaunchKernelGGL(k_nt_precond, dim3(nblk(n)), dim3(TPB), 0, ctx->stream, n, P, bb, x);
  }

  // hypre_FlexGMRESSolve (flexgmres.c:260-700) with rel_change off, cf_tol 0,
  // r_tol 0, k_dim 20: x updated in place.  The Arnoldi steps and the solve of the
  // Hessenberg system run on the device (dot products reduced there, the Givens
  // update in one thread); the host reads the residual estimate once per step, the
  // norms at a cycle's start, and the Hessenberg system only where a cycle restarts.
  // bnorm2: bb . bb
  int gmres(const double *bb, double bnorm2, double *x, int max_iter, int min_iter, double a_tol)
  {
    const int k_dim = NT_KDIM;
    NtScal h;
    double r_norm, b_norm, t;
    int iter = 0, i = 0;
#define HHH(a, b) h.hh[(a)*NT_KDIM + (b)]
    CHK(copy(bb, kv(0)));
    CHK(matvec(-1.0, x, 1.0, kv(0)));
    b_norm = std::sqrt(bnorm2);
    if (b_norm != 0.0 && !std::isfinite(b_norm)) return 0;   // non-finite input: x untouched
    CHK(dot(kv(0), kv(0), t)); r_norm = std::sqrt(t);
    if (r_norm != 0.0 && !std::isfinite(r_norm)) return 0;
    const double epsilon = a_tol;
    while (iter < max_iter)
    {
      if (r_norm == 0.0) break;
      if (r_norm <= epsilon && iter >= min_iter)
      {
        CHK(copy(bb, r));
        CHK(matvec(-1.0, x, 1.0, r));
        CHK(dot(r, r, t)); r_norm = std::sqrt(t);
        if (r_norm <= epsilon) break;
      }
      hipLaunchKernelGGL(k_nt_start, dim3(nblk(std::max(N, 1LL))), dim3(TPB), 0, ctx->stream, N, 1.0/r_norm, kv(0), sc->rs,
                         r_norm);
      i = 0;
      while (i < k_dim && iter < max_iter)
      {
        i ++;
        iter ++;
        precond(kv(i - 1), pv(i - 1));
        CHK(matvec(1.0, pv(i - 1), 0.0, kv(i)));
        arnoldi(i);
        HIPCHK(hipStreamSynchronize(ctx->stream));
        r_norm = hpart[NT_DOT_BLOCKS];
        if (r_norm <= epsilon && iter >= min_iter) break;
      }
      const int m = i;
      hipLaunchKernelGGL(k_nt_cycle, dim3(dot_grid()), dim3(TPB), 0, ctx->stream, N, (const NtScal *)sc, m,
                         (const double *)pre, x);
      HIPCHK(hipGetLastError());
      if (r_norm <= epsilon && iter >= min_iter)
      {
        CHK(copy(bb, r));
        CHK(matvec(-1.0, x, 1.0, r));
        CHK(dot(r, r, t)); r_norm = std::sqrt(t);
        if (r_norm <= epsilon) break;
        CHK(copy(r, kv(0)));   // false convergence
        i = 0;
      }
      if (iter >= max_iter) break;
      // a restart: the residual from the Krylov vectors
      HIPCHK(hipMemcpyAsync(&h, sc, sizeof(NtScal), hipMemcpyDeviceToHost, ctx->stream));
      HIPCHK(hipStreamSynchronize(ctx->stream));
      h.rs[m - 1] = h.rs[m - 1]/HHH(m - 1, m - 1);
      for (int k = m - 2; k >= 0; k --)
      {
        t = 0.0;
        for (int j = k + 1; j < m; j ++) t -= HHH(k, j)*h.rs[j];
        t += h.rs[k];
        h.rs[k] = t/HHH(k, k);
      }
      for (int j = i; j > 0; j --)
      {
        h.rs[j - 1] = -h.s[j - 1]*h.rs[j];
        h.rs[j] = h.c[j - 1]*h.rs[j];
      }
      if (i) axpy(h.rs[i] - 1.0, kv(i), kv(i));
      for (int j = i - 1; j > 0; j --) axpy(h.rs[j], kv(j), kv(i));
      if (i)
      {
        axpy(h.rs[0] - 1.0, kv(0), kv(0));
        axpy(1.0, kv(i), kv(0));
      }
    }
#undef HHH
    HIPCHK(hipGetLastError());
    return 0;
  }
};

} // namespace

void sfgs_newton_release(sfgs_ctx *ctx)
{
  release(ctx->nt_mem);
  release(ctx->nt_ctl);
  if (ctx->nt_host) (void)hipHostFree(ctx->nt_host);
  ctx->nt_host = nullptr;
}

extern "C" {

// NEWTON_Solve (nts.c:1333-1379) with LOCDYN_ON
int SFGS_Newton_Solve(sfgs_ctx *ctx, const SFGS_NEWTON_PARAM *par, double *merhist, int *mvhist,
                      SFGS_NEWTON_REPORT *rep)
{
  if (!ctx || !par) return SFGS_E_ARG;
  if (!(par->meritval > 0.0) || par->maxiter <= 0 || par->linmaxiter <= 0 || par->maxmatvec <= 0 ||
      !(par->epsilon > 0.0) || !(par->delta >= 0.0) || !(par->theta > 0.0 && par->theta <= 1.0) ||
      !(par->omega > 0.0) || (par->linver != SFGS_NT_GMRES && par->linver != SFGS_NT_DIAG) ||
      par->reldelta < 0 || par->reldelta > 3 || (par->bodyspace != 0 && par->bodyspace != 1)) return SFGS_E_ARG;
  if (!ctx->assembled) { ctx->err = "solve before LOCDYN assembly"; return SFGS_E_STATE; }
  if (ctx->diag_only) { ctx->err = "the store holds a penalty solve, not an assembled system"; return SFGS_E_STATE; }
  if (ctx->nscenes > 1) { ctx->err = "the system holds independent scenes"; return SFGS_E_STATE; }
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int n = ctx->nc;
  const long long N = 3LL*n;
  const size_t N1 = (size_t)std::max(N, 1LL), n1 = (size_t)std::max(n, 1);

  // one allocation: X, Y, P (9 per row), b, dr, r (3 per row), R0 (4 per
  // row), the Krylov and the preconditioned vectors, dot partials
  const size_t scal_words = (sizeof(NtScal) + 7)/8;
  const size_t words = 27*n1 + 3*N1 + 4*n1 + (size_t)(2*NT_KDIM + 1)*N1 + 2*NT_DOT_BLOCKS + scal_words;
  CHK(ensure(ctx, ctx->nt_mem, words));
  NtWork wk;
  double *m0 = ctx->nt_mem.p;
  wk.ctx = ctx; wk.n = n; wk.N = N;
  wk.X = m0; wk.Y = wk.X + 9*n1; wk.P = wk.Y + 9*n1; wk.b = wk.P + 9*n1; wk.dr = wk.b + N1; wk.r = wk.dr + N1;
  wk.R0 = wk.r + N1; wk.kry = wk.R0 + 4*n1; wk.pre = wk.kry + (size_t)(NT_KDIM + 1)*N1;
  wk.part = wk.pre + (size_t)NT_KDIM*N1;
  wk.sc = (NtScal*)(wk.part + 2*NT_DOT_BLOCKS);
  if (!ctx->nt_host) HIPCHK(hipHostMalloc((void**)&ctx->nt_host, sizeof(double)*(NT_DOT_BLOCKS + 1), hipHostMallocDefault));
  wk.hpart = ctx->nt_host;
  HIPCHK(hipMemsetAsync(m0, 0, sizeof(double)*words, st));
  if (n > 0) HIPCHK(hipMemcpyAsync(wk.R0, ctx->R.p, sizeof(double)*4*(size_t)n, hipMemcpyDeviceToDevice, st));
  CHK(ensure(ctx, ctx->failcount, 4));
  HIPCHK(hipMemsetAsync(ctx->failcount.p, 0, sizeof(int)*4, st));

  // W norm of the relative delta (LOCDYN_avgWii / minWii / maxWii, ldy.c:1146-1193)
  double W_norm = 1.0;
  if (par->reldelta != 0 && n > 0)
  {
    std::vector<double> d(3*(size_t)n);
    for (int e = 0; e < 3; e ++)
      HIPCHK(hipMemcpyAsync(d.data() + (size_t)e*n, ctx->Wd.p + (size_t)(4*e)*n, sizeof(double)*(size_t)n,
                            hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (par->reldelta == 1)
    {
      double sum = 0.0, div = 0.0;
      for (int p = 0; p < n; p ++) { sum += d[p] + d[(size_t)n + p] + d[2*(size_t)n + p]; div += 3.0; }
      W_norm = sum/div;
    }
    else if (par->reldelta == 2) W_norm = *std::min_element(d.begin(), d.end());
    else W_norm = std::max(0.0, *std::max_element(d.begin(), d.end()));
  }
  else if (par->reldelta == 2) W_norm = DBL_MAX;
  else if (par->reldelta == 3) W_norm = 0.0;
  const double delta = par->delta*W_norm;

  wk.mat = NtMat{ctx->slice_row0.p, ctx->slice_nrows.p, ctx->rowlen.p, ctx->rowoff.p, ctx->slice_len.p,
                 ctx->slice_off.p, ctx->W.p, ctx->wcol.p, ctx->Wd.p, wk.X, wk.Y, n, delta};
  NtRows rows{n, ctx->R.p, ctx->U.p, ctx->Wd.p, ctx->pfri.p, ctx->pcoh.p, ctx->shift.p, wk.X, wk.Y, wk.P, wk.b, wk.dr,
              ctx->failcount.p};

  wk.bodyspace = par->bodyspace;
  if (par->bodyspace && !ctx->from_bodies)
  {
    ctx->err = "locdyn OFF needs a system assembled from bodies";
    return SFGS_E_STATE;
  }
  if (!par->bodyspace && ctx->upmin)
  {
    ctx->err = "locdyn ON needs the off-diagonal blocks (SFGS_Locdyn_Update_Begin)";
    return SFGS_E_STATE;
  }
  // U = W R + B (U_WR_B, nts.c:255-431), then the merit (nts.c:929, 1199); in
  // body space W R is formed through the bodies
  auto merit_of = [&](double &m) -> int {
    if (!par->bodyspace) return SFGS_Merit(ctx, 1, &m, nullptr);
    CHK(bodyspace_product(ctx, ctx->R.p, 4, 1, nullptr, nullptr, 0.0, 0.0, 0.0, nullptr));
    return SFGS_Merit(ctx, 0, &m, nullptr);
  };
  double merit = 0.0;
  CHK(merit_of(merit));
  int iters = 0, nan = 0;
  const bool diag = par->linver == SFGS_NT_DIAG;
  if (diag && iters < par->maxiter && merit > par->meritval && n > 0)
  {
    // batches of iterations without a read-back: 4, 8, 16, 32, 32, ...; every launch
    // past the loop's end, the body products too, sees ctl->done and returns at once
    // (29 iterations of 1.4 ms products that end one into a batch: 83 ms without the
    // products' test of it, 43 with)
    CHK(ensure(ctx, ctx->nt_ctl, sizeof(NtCtl)));
    NtCtl *ctl = (NtCtl*)ctx->nt_ctl.p, h;
    std::memset(&h, 0, sizeof(h));
    HIPCHK(hipMemcpyAsync(ctl, &h, sizeof(h), hipMemcpyHostToDevice, st));
    const double lo = ctx->energy < DBL_EPSILON ? 1.0 : ctx->energy;
    NtTest test{ctl, 0, ctx->mpartials.p, 0, par->maxiter, lo, par->meritval};
    for (int batch = 4; !h.done; batch = std::min(2*batch, NtCtl::BATCH))
    {
      const int last = (int)std::min((long long)test.k + batch, (long long)par->maxiter + 1);
      for (; test.k < last; test.k ++)
      {
        hipLaunchKernelGGL(k_nt_lin, dim3(nblk(n)), dim3(TPB), 0, st, rows, 1, par->omega, delta, par->theta, ctx->R.p,
                           test);
        HIPCHK(hipGetLastError());
        if (test.k == par->maxiter) continue;   // the last launch only tests
        if (par->bodyspace)
          CHK(bodyspace_product(ctx, ctx->R.p, 4, 1, nullptr, nullptr, 0.0, 0.0, 0.0, nullptr, &ctl->done));
        CHK(launch_merit(ctx, par->bodyspace ? 0 : 1, nullptr, &ctl->done, &test.np));
      }
      HIPCHK(hipMemcpyAsync(&h, ctl, sizeof(h), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      for (; iters < h.iters; iters ++)
      {
        if (merhist) merhist[iters] = h.hist[iters % NtCtl::RING];
        if (mvhist) mvhist[iters] = 0;
      }
    }
    merit = h.merit;
    nan = h.nan;
  }
  while (!diag && iters < par->maxiter && wk.matvecs < par->maxmatvec && merit > par->meritval)
  {
    if (n > 0)
      hipLaunchKernelGGL(k_nt_lin, dim3(nblk(n)), dim3(TPB), 0, st, rows, 0, par->omega, delta, par->theta, ctx->R.p,
                         NtTest{});
    HIPCHK(hipGetLastError());
    double bb = 0.0;
    CHK(wk.dot(wk.b, wk.b, bb));
    CHK(wk.gmres(wk.b, bb, wk.dr, par->linmaxiter, 1, par->epsilon*std::sqrt(bb)));
    if (n > 0)
      hipLaunchKernelGGL(k_nt_update, dim3(nblk(n)), dim3(TPB), 0, st, n, ctx->R.p, wk.dr, ctx->pfri.p, ctx->pcoh.p);
    HIPCHK(hipGetLastError());
    CHK(merit_of(merit));
    if (std::isnan(merit)) { nan = 1; break; }
    if (merhist) merhist[iters] = merit;
    if (mvhist) mvhist[iters] = wk.matvecs;
    iters ++;
  }
  int singular = 0;
  HIPCHK(hipMemcpyAsync(&singular, ctx->failcount.p, sizeof(int), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  SFGS_NEWTON_REPORT r;
  std::memset(&r, 0, sizeof(r));
  r.iters = iters;
  r.matvecs = wk.matvecs;
  r.converged = !nan && merit <= par->meritval;
  r.singular = singular;
  r.merit = merit;
  r.W_norm = W_norm;
  if (!r.converged && par->gsflag && par->bodyspace)
  {
    // the reference aborts here (nts.c:1370-1374: no Gauss-Seidel without the
    // assembled blocks); this library reports the failure instead
    if (rep) *rep = r;
    ctx->err = "NEWTON_SOLVER failed in body space mode";
    return SFGS_E_STATE;
  }
  if (!r.converged && par->gsflag)
  {
    // R back to its initial value; GAUSS_SEIDEL_Create (1.0, maxiter, meritval,
    // GS_FAILURE_CONTINUE, 1E-9, 100, DS_SEMISMOOTH_NEWTON) (nts.c:1363)
    if (n > 0) HIPCHK(hipMemcpyAsync(ctx->R.p, wk.R0, sizeof(double)*4*(size_t)n, hipMemcpyDeviceToDevice, st));
    SFGS_PARAM gp;
    std::memset(&gp, 0, sizeof(gp));
    gp.epsilon = 1.0; gp.maxiter = par->maxiter; gp.meritval = par->meritval; gp.failure = SFGS_FAILURE_CONTINUE;
    gp.diagepsilon = 1e-9; gp.diagmaxiter = 100; gp.diagsolver = SFGS_DS_SEMISMOOTH_NEWTON;
    gp.precision = SFGS_PREC_FP64;
    SFGS_REPORT gr;
    CHK(SFGS_Solve(ctx, &gp, nullptr, nullptr, &gr));
    r.gs_fallback = 1;
    r.gs_iters = gr.iters;
    r.merit = gr.merit;
  }
  if (rep) *rep = r;
  return 0;
}

} // extern "C"
