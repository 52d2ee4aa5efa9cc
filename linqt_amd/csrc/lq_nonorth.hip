// Non-orthogonal basis: overlap solves and the non-orthogonal spectral moments.
//
// linalg::orthogonalize (src/mkl_linear_algebra.cpp:100-131) solves S x = b
// with Eigen's BiCGSTAB (diagonal preconditioner, zero initial guess, stop
// when |r|^2 <= tol^2 |b|^2 or after maxit iterations; tol 1e-4 and 2000 in
// the reference), where S is the overlap CSR mapped as a general matrix.
// Moments1D_nonOrth (src/chebyshev_moments.cpp:63-153) and
// SpectralMoments_nonOrth (src/chebyshev_solver.cpp:203-229) run the
// Chebyshev recursion with such a solve after every Hamiltonian product:
//   T0 = [OP] S^-1 phi,  T1 = S^-1 H T0,  T_{m+1} = 2 S^-1 H T_m - T_{m-1},
//   mu_m += (2/R)(1/2 if m = 0) <phi|T_m>.
//
// Here every BiCGSTAB vector and scalar lives in HBM.  An iteration is five
// launches: p/y, v = S y with <r0|v>, s/z, t = S z with <t|t> and <t|s>, x/r with
// |r|^2 and <r0|r>.  The kernels that need a dot product's value sum the partials
// of the blocks before them, every block for itself, in one fixed order; the
// stopping test is theirs too, and an iteration queued past it leaves the vectors
// alone.  So the host queues as many iterations as the solve before took, at most
// 16, and only then looks (one small copy), where a copy and a wait for each of three dot
// products had taken most of an iteration's 100 us (N = 16380, 147 iterations in
// 49 solves: 15.1 -> 5.5 ms; what is left is launches of 4 to 5 us).
#include <algorithm>
#include <cmath>
#include <vector>

#include "lq_internal.h"

namespace lq {
namespace {

constexpr int kNbThreads = 256;
constexpr int kNbBlocks = 512;
// Most iterations queued before the host looks.  A look costs half an iteration's
// launches; an iteration queued past the end costs all of them and its two products,
// which test no state (a load before their first one took 4 % of a solve).
constexpr int kNbQueue = 16;

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// conj(a) * b
__device__ __forceinline__ double2 cdot1(double2 a, double2 b) {
  return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// Block sum of two complex values; thread 0 writes partial[blockIdx.x * 2 + j].
__device__ void block_store2(double2 a, double2 b, double2 *__restrict__ partial) {
  __shared__ double2 sh[2][kNbThreads];
  const int t = threadIdx.x;
  sh[0][t] = a;
  sh[1][t] = b;
  __syncthreads();
  for (int w = kNbThreads / 2; w > 0; w >>= 1) {
    if (t < w) {
      sh[0][t] = cadd(sh[0][t], sh[0][t + w]);
      sh[1][t] = cadd(sh[1][t], sh[1][t + w]);
    }
    __syncthreads();
  }
  if (t == 0) {
    partial[2 * blockIdx.x] = sh[0][0];
    partial[2 * blockIdx.x + 1] = sh[1][0];
  }
}

// partial <- per-block sums of conj(x1) y1 and conj(x2) y2 (x2 == nullptr: 0).
__global__ __launch_bounds__(kNbThreads) void k_nb_dot2(int n, const double2 *__restrict__ x1,
                                                         const double2 *__restrict__ y1,
                                                         const double2 *__restrict__ x2,
                                                         const double2 *__restrict__ y2, double2 *__restrict__ partial) {
  double2 a = make_double2(0.0, 0.0), b = make_double2(0.0, 0.0);
  for (int i = blockIdx.x * kNbThreads + threadIdx.x; i < n; i += gridDim.x * kNbThreads) {
    a = cadd(a, cdot1(x1[i], y1[i]));
    if (x2) b = cadd(b, cdot1(x2[i], y2[i]));
  }
  block_store2(a, b, partial);
}

// out[j] = sum over blocks of partial[b*2 + j]; with acc != nullptr also
// acc[0] += scal * out[0] (a moment).
__global__ __launch_bounds__(kNbThreads) void k_nb_final(const double2 *__restrict__ partial, int nblk,
                                                          double2 *__restrict__ out, double scal,
                                                          double2 *__restrict__ acc) {
  __shared__ double2 sh[2][kNbThreads];
  const int t = threadIdx.x;
  double2 a = make_double2(0.0, 0.0), b = make_double2(0.0, 0.0);
  for (int q = t; q < nblk; q += kNbThreads) {
    a = cadd(a, partial[2 * q]);
    b = cadd(b, partial[2 * q + 1]);
  }
  sh[0][t] = a;
  sh[1][t] = b;
  __syncthreads();
  for (int w = kNbThreads / 2; w > 0; w >>= 1) {
    if (t < w) {
      sh[0][t] = cadd(sh[0][t], sh[0][t + w]);
      sh[1][t] = cadd(sh[1][t], sh[1][t + w]);
    }
    __syncthreads();
  }
  if (t == 0) {
    out[0] = sh[0][0];
    out[1] = sh[1][0];
    if (acc) acc[0] = make_double2(acc[0].x + scal * sh[0][0].x, acc[0].y + scal * sh[0][0].y);
  }
}

// r = r0 = b, x = p = v = 0; partials of |b|^2.
__global__ __launch_bounds__(kNbThreads) void k_nb_init(int n, const double2 *__restrict__ b, double2 *__restrict__ r,
                                                         double2 *__restrict__ r0, double2 *__restrict__ x,
                                                         double2 *__restrict__ p, double2 *__restrict__ v,
                                                         double2 *__restrict__ partial) {
  double2 a = make_double2(0.0, 0.0);
  const double2 z = make_double2(0.0, 0.0);
  for (int i = blockIdx.x * kNbThreads + threadIdx.x; i < n; i += gridDim.x * kNbThreads) {
    const double2 bi = b[i];
    r[i] = bi;
    r0[i] = bi;
    x[i] = z;
    p[i] = z;
    v[i] = z;
    a = cadd(a, cdot1(bi, bi));
  }
  block_store2(a, z, partial);
}

// Scalars of a solve.  A kernel's block 0 writes the ones it computes; every
// block of a kernel computes them for itself, and reads only what kernels before
// it wrote (rho by parity of the iteration).
enum NbState { kNbRunning = 0, kNbDone = 1, kNbRestart = 2 };
struct NbScal {
  double2 rho[2], alpha, w;
  double rhs_sq, r0_sq, r_sq;
  int state, it, i;
};

// Power of two of a's larger component (0 for zero, infinities and NaN).
__device__ __forceinline__ int scale_of(double2 a) {
  const double m = fmax(fabs(a.x), fabs(a.y));
  return m > 0.0 && m < HUGE_VAL ? ilogb(m) : 0;
}
__device__ __forceinline__ double2 scaled(double2 a, int e) { return make_double2(ldexp(a.x, e), ldexp(a.y, e)); }

// a / b with both brought to the size of 1 by powers of two: the solver's scalars
// grow with |b|^2 of the system, so the square of a divisor would leave the
// exponent's range for right-hand sides beyond 1e-77 .. 1e77.
__device__ __forceinline__ double2 cdiv(double2 a, double2 b) {
  const int ea = scale_of(a), eb = scale_of(b);
  a = scaled(a, -ea);
  b = scaled(b, -eb);
  const double m = b.x * b.x + b.y * b.y;
  return scaled(make_double2((a.x * b.x + a.y * b.y) / m, (a.y * b.x - a.x * b.y) / m), ea - eb);
}

// Every thread: (sum, sum) of nblk pairs (NV = 2) or single values of partials, in
// one fixed order.
template <int NV>
__device__ __forceinline__ void sum_partials(const double2 *__restrict__ partial, int nblk, double2 &a, double2 &b) {
  __shared__ double2 sh[2][kNbThreads];
  const int t = threadIdx.x;
  double2 u = make_double2(0.0, 0.0), v = u;
  for (int q = t; q < nblk; q += kNbThreads) {
    u = cadd(u, partial[NV * q]);
    if (NV == 2) v = cadd(v, partial[NV * q + 1]);
  }
  sh[0][t] = u;
  if (NV == 2) sh[1][t] = v;
  __syncthreads();
  for (int w = kNbThreads / 2; w > 0; w >>= 1) {
    if (t < w) {
      sh[0][t] = cadd(sh[0][t], sh[0][t + w]);
      if (NV == 2) sh[1][t] = cadd(sh[1][t], sh[1][t + w]);
    }
    __syncthreads();
  }
  a = sh[0][0];
  if (NV == 2) b = sh[1][0];
}

// Iteration i (the count-th that maxit bounds): the stopping test, rho and beta;
// then p = r + beta (p - w v), y = dinv p.  partial: of |r|^2 and <r0|r> (first: of
// |b|^2).  resumed: after a restart, rho and the test are settled.
__global__ __launch_bounds__(kNbThreads) void k_nb_p(int n, int i, int count, int first, int resumed, double tol,
                                                      int maxit, const double2 *__restrict__ partial, int nblk,
                                                      NbScal *sc,
                                                      const double2 *__restrict__ r, double2 *__restrict__ p,
                                                      const double2 *__restrict__ v, const double2 *__restrict__ dinv,
                                                      double2 *__restrict__ y) {
  if (!first && !resumed && sc->state != kNbRunning) return;
  const double2 one = make_double2(1.0, 0.0);
  double2 rho, rho_old = first ? one : sc->rho[i & 1], alpha = first ? one : sc->alpha, w = first ? one : sc->w;
  if (resumed) {
    rho = sc->rho[(i + 1) & 1];
  } else {
    double2 rr, r0r;
    sum_partials<2>(partial, nblk, rr, r0r);
    if (first) r0r = make_double2(rr.x, 0.0);
    const double rhs_sq = first ? rr.x : sc->rhs_sq, r0_sq = first ? rr.x : sc->r0_sq;
    rho = r0r;
    int state = kNbRunning;
    if ((first && rhs_sq == 0.0) || !(rr.x > tol * tol * rhs_sq) || count >= maxit)
      state = kNbDone;
    else if (hypot(rho.x, rho.y) < 4.930380657631324e-32 * r0_sq)  // r too orthogonal to r0
      state = kNbRestart;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      sc->state = state;
      sc->r_sq = rr.x;
      if (first) {
        sc->rhs_sq = sc->r0_sq = rr.x;
        sc->rho[i & 1] = sc->alpha = sc->w = one;
      }
      sc->it = count;
      sc->i = i;
      if (state == kNbRunning) sc->rho[(i + 1) & 1] = rho;
    }
    if (state != kNbRunning) return;
  }
  const double2 beta = cmul(cdiv(rho, rho_old), cdiv(alpha, w));
  for (int e = blockIdx.x * kNbThreads + threadIdx.x; e < n; e += gridDim.x * kNbThreads) {
    const double2 pi = cadd(r[e], cmul(beta, csub(p[e], cmul(w, v[e]))));
    p[e] = pi;
    y[e] = cmul(dinv[e], pi);
  }
}

// alpha = rho / <r0|v> (partial); s = r - alpha v; z = dinv s
__global__ __launch_bounds__(kNbThreads) void k_nb_s(int n, int i, const double2 *__restrict__ partial, int nblk,
                                                      NbScal *sc, const double2 *__restrict__ r,
                                                      const double2 *__restrict__ v, const double2 *__restrict__ dinv,
                                                      double2 *__restrict__ s, double2 *__restrict__ z) {
  if (sc->state != kNbRunning) return;
  double2 r0v, none;
  sum_partials<1>(partial, nblk, r0v, none);
  const double2 alpha = cdiv(sc->rho[(i + 1) & 1], r0v);
  if (blockIdx.x == 0 && threadIdx.x == 0) sc->alpha = alpha;
  for (int e = blockIdx.x * kNbThreads + threadIdx.x; e < n; e += gridDim.x * kNbThreads) {
    const double2 si = csub(r[e], cmul(alpha, v[e]));
    s[e] = si;
    z[e] = cmul(dinv[e], si);
  }
}

// w = <t|s> / <t|t> (pin); x += alpha y + w z; r = s - w t; partials of |r|^2
// and <r0|r>.
__global__ __launch_bounds__(kNbThreads) void k_nb_xr(int n, const double2 *__restrict__ pin, int nblk, NbScal *sc,
                                                       double2 *__restrict__ x, const double2 *__restrict__ y,
                                                       const double2 *__restrict__ z, const double2 *__restrict__ s,
                                                       const double2 *__restrict__ t, double2 *__restrict__ r,
                                                       const double2 *__restrict__ r0, double2 *__restrict__ partial) {
  if (sc->state != kNbRunning) return;
  double2 tt, ts;
  sum_partials<2>(pin, nblk, tt, ts);
  const double2 alpha = sc->alpha;
  const double2 w = tt.x > 0.0 ? make_double2(ts.x / tt.x, ts.y / tt.x) : make_double2(0.0, 0.0);
  if (blockIdx.x == 0 && threadIdx.x == 0) sc->w = w;
  double2 a = make_double2(0.0, 0.0), b = make_double2(0.0, 0.0);
  for (int e = blockIdx.x * kNbThreads + threadIdx.x; e < n; e += gridDim.x * kNbThreads) {
    x[e] = cadd(x[e], cadd(cmul(alpha, y[e]), cmul(w, z[e])));
    const double2 ri = csub(s[e], cmul(w, t[e]));
    r[e] = ri;
    a = cadd(a, cdot1(ri, ri));
    b = cadd(b, cdot1(r0[e], ri));
  }
  block_store2(a, b, partial);
}

// After k_nb_restart of iteration i: r0_sq = rho = |r|^2 (partial), running again.
__global__ __launch_bounds__(kNbThreads) void k_nb_resume(const double2 *__restrict__ partial, int nblk, int i,
                                                           NbScal *sc) {
  double2 rr, none;
  sum_partials<2>(partial, nblk, rr, none);
  if (threadIdx.x == 0) {
    sc->r0_sq = rr.x;
    sc->rho[(i + 1) & 1] = make_double2(rr.x, 0.0);
    sc->state = kNbRunning;
  }
}

// DiagonalPreconditioner from the sliced-ELL form: 1 / (the row's first diagonal
// entry) when that is nonzero, else 1 (padding: own column, value 0).
__global__ __launch_bounds__(kNbThreads) void k_nb_dinv(int n, const int *__restrict__ sptr,
                                                         const int *__restrict__ col, const double2 *__restrict__ val,
                                                         double2 *__restrict__ dinv) {
  const int i = blockIdx.x * kNbThreads + threadIdx.x;
  if (i >= n) return;
  const int base = sptr[i / kSlice], w = (sptr[i / kSlice + 1] - base) / kSlice;
  double2 d = make_double2(1.0, 0.0);
  for (int j = 0; j < w; ++j) {
    const size_t q = (size_t)base + (size_t)j * kSlice + i % kSlice;
    if (col[q] != i) continue;
    const double2 e = val[q];
    if (e.x != 0.0 || e.y != 0.0) d = cdiv(make_double2(1.0, 0.0), e);
    break;
  }
  dinv[i] = d;
}

// restart: r = r0 = b - t; partials of |r|^2
__global__ __launch_bounds__(kNbThreads) void k_nb_restart(int n, const double2 *__restrict__ b,
                                                            const double2 *__restrict__ t, double2 *__restrict__ r,
                                                            double2 *__restrict__ r0, double2 *__restrict__ partial) {
  double2 a = make_double2(0.0, 0.0);
  for (int i = blockIdx.x * kNbThreads + threadIdx.x; i < n; i += gridDim.x * kNbThreads) {
    const double2 ri = csub(b[i], t[i]);
    r[i] = ri;
    r0[i] = ri;
    a = cadd(a, cdot1(ri, ri));
  }
  block_store2(a, make_double2(0.0, 0.0), partial);
}

// c0 = 2 u - c0
__global__ __launch_bounds__(kNbThreads) void k_nb_cheb(int n, const double2 *__restrict__ u, double2 *__restrict__ c0) {
  for (int i = blockIdx.x * kNbThreads + threadIdx.x; i < n; i += gridDim.x * kNbThreads) {
    const double2 ui = u[i], ci = c0[i];
    c0[i] = make_double2(2.0 * ui.x - ci.x, 2.0 * ui.y - ci.y);
  }
}

int nb_grid(int n) { return std::max(1, std::min(kNbBlocks, (n + kNbThreads - 1) / kNbThreads)); }

// BiCGSTAB state on the device for systems with S (n rows), in buffers of the
// context that outlive the call (freed by lq_ctx_release).
struct Bicg {
  lq_ctx ctx = nullptr;
  lq_csr S = nullptr;
  int n = 0, grid = 1, dots = 1;  // blocks of the vector kernels and of a product with dots
  double2 *r = nullptr, *r0 = nullptr, *p = nullptr, *v = nullptr, *y = nullptr, *z = nullptr, *s = nullptr,
          *t = nullptr, *dinv = nullptr, *partial = nullptr, *dpart = nullptr, *res = nullptr;
  NbScal *sc = nullptr, *host = nullptr;  // host: pinned
  long long iterations = 0;
  int expect = 1;  // iterations the last solve took

  int init(lq_ctx c, lq_csr S_) {
    ctx = c;
    S = S_;
    n = S->n;
    grid = nb_grid(n);
    dots = spmm_dot_grid(n, 1);
    const size_t row = ((size_t)n + 15) / 16 * 16;
    double2 *vec;
    LQ_TRY(ctx_buf(ctx, "nb_vec", sizeof(double2) * 9 * row, (void **)&vec));
    double2 **const all[9] = {&r, &r0, &p, &v, &y, &z, &s, &t, &dinv};
    for (int q = 0; q < 9; ++q) *all[q] = vec + q * row;
    LQ_TRY(ctx_buf(ctx, "nb_part", sizeof(double2) * (2 * (size_t)kNbBlocks + 2 * (size_t)dots + 2), (void **)&partial));
    dpart = partial + 2 * (size_t)kNbBlocks;
    res = dpart + 2 * (size_t)dots;
    LQ_TRY(ctx_buf(ctx, "nb_scal", sizeof(NbScal), (void **)&sc));
    LQ_TRY(ctx_pinned(ctx, sizeof(NbScal), (void **)&host));
    hipLaunchKernelGGL(k_nb_dinv, dim3((n + kNbThreads - 1) / kNbThreads), dim3(kNbThreads), 0, ctx->stream, n,
                       S->dev.sptr, S->dev.col, S->dev.val, dinv);
    LQ_HIP_CHECK(hipGetLastError());
    return LQ_OK;
  }

  int apply_S(const double2 *in, double2 *out, int dot_mode, const double2 *phi) {
    VecSet set{in, nullptr, out, 1};
    hipEvent_t ev;
    LQ_TRY(time_begin(ctx, kCatSpmv, &ev));
    LQ_TRY(launch_spmm(ctx->stream, S->dev, make_double2(1.0, 0.0), make_double2(0.0, 0.0), &set, 1, dot_mode, phi,
                       dot_mode == kDotNone ? nullptr : dpart, nullptr));
    return time_end(ctx, kCatSpmv, ev, 20.0 * (double)S->col.size() + 4.0 * (n + 1) + 32.0 * n);
  }

  // x = S^-1 b (Eigen's BiCGSTAB); b and x are distinct device vectors of n.
  int solve(const double2 *b, double2 *x, double tol, int maxit, int *iters, double *error) {
    const dim3 g(grid), blk(kNbThreads);
    const hipStream_t st = ctx->stream;
    hipLaunchKernelGGL(k_nb_init, g, blk, 0, st, n, b, r, r0, x, p, v, partial);
    LQ_HIP_CHECK(hipGetLastError());
    // i numbers the iterations queued (rho is stored by its parity); the count that
    // maxit bounds starts anew at the first restart, as the sources' does
    int i = 0, base = 0, restarts = 0, queue = 1 + std::min(kNbQueue, expect);
    bool first = true, resumed = false;
    auto rest = [&]() -> int {  // iteration i after its k_nb_p
      LQ_TRY(apply_S(y, v, kDotPhi, r0));
      hipLaunchKernelGGL(k_nb_s, g, blk, 0, st, n, i, dpart, dots, sc, r, v, dinv, s, z);
      LQ_TRY(apply_S(z, t, kDotSelf, s));
      hipLaunchKernelGGL(k_nb_xr, g, blk, 0, st, n, dpart, dots, sc, x, y, z, s, t, r, r0, partial);
      LQ_HIP_CHECK(hipGetLastError());
      return LQ_OK;
    };
    for (;;) {
      // `queue` stopping tests with the iterations between them, then a look
      for (int q = 0;; ++q) {
        hipLaunchKernelGGL(k_nb_p, g, blk, 0, st, n, i, i - base, first ? 1 : 0, resumed ? 1 : 0, tol, maxit, partial,
                           grid, sc, r, p, v, dinv, y);
        LQ_HIP_CHECK(hipGetLastError());
        first = resumed = false;
        if (q + 1 >= queue) break;
        LQ_TRY(rest());
        ++i;
      }
      LQ_HIP_CHECK(hipMemcpyAsync(host, sc, sizeof(NbScal), hipMemcpyDeviceToHost, st));
      LQ_HIP_CHECK(hipStreamSynchronize(st));
      if (host->state == kNbDone) break;
      if (host->state == kNbRestart) {  // from the current x, within iteration host->i
        LQ_TRY(apply_S(x, t, kDotNone, nullptr));
        i = host->i;
        if (restarts++ == 0) base = i;
        hipLaunchKernelGGL(k_nb_restart, g, blk, 0, st, n, b, t, r, r0, partial);
        hipLaunchKernelGGL(k_nb_resume, dim3(1), blk, 0, st, partial, grid, i, sc);
        LQ_HIP_CHECK(hipGetLastError());
        resumed = true;
        queue = 2;
      } else {  // the last test went on
        LQ_TRY(rest());
        ++i;
        queue = 1 + std::min(kNbQueue, (i - base) / 4);
      }
    }
    iterations += host->it;
    expect = host->it;
    if (iters) *iters = host->it;
    if (error) *error = host->rhs_sq == 0.0 ? 0.0 : std::sqrt(host->r_sq / host->rhs_sq);
    return LQ_OK;
  }
};

int check_square(lq_csr A, int n, const char *what) {
  if (A && A->n != n) {
    set_error("%s: operator sizes differ (%d vs %d)", what, A->n, n);
    return LQ_ERR_ARG;
  }
  return LQ_OK;
}

}  // namespace
}  // namespace lq

using namespace lq;

extern "C" int lq_overlap_solve(lq_csr S, const double *b, double *x, double tol, int maxit, int *iterations,
                                double *error) try {
  if (!S || !S->ctx || !b || !x || b == x) {
    set_error("lq_overlap_solve: need an operator and distinct device vectors b, x");
    return LQ_ERR_ARG;
  }
  lq_ctx ctx = S->ctx;
  DeviceGuard g(ctx->device);
  Bicg bc;
  LQ_TRY(bc.init(ctx, S));
  return bc.solve((const double2 *)b, (double2 *)x, tol > 0 ? tol : 1e-4, maxit > 0 ? maxit : 2000, iterations,
                  error);
} LQ_ABI_CATCH

extern "C" int lq_spectral_moments_nonorth(lq_csr H, lq_csr OP, lq_csr S, const double *phi, int R, int M,
                                           double tol, int maxit, double *mu, long long *iterations) try {
  if (!H || !S || !phi || !mu || R <= 0 || M <= 0) {
    set_error("lq_spectral_moments_nonorth: invalid arguments");
    return LQ_ERR_ARG;
  }
  const int n = H->n;
  LQ_TRY(check_square(S, n, "lq_spectral_moments_nonorth"));
  LQ_TRY(check_square(OP, n, "lq_spectral_moments_nonorth"));
  if (S->ctx != H->ctx || (OP && OP->ctx != H->ctx)) {
    set_error("lq_spectral_moments_nonorth: operators belong to different contexts");
    return LQ_ERR_ARG;
  }
  tol = tol > 0 ? tol : 1e-4;
  maxit = maxit > 0 ? maxit : 2000;
  lq_ctx ctx = H->ctx;
  DeviceGuard g(ctx->device);
  Bicg bc;
  LQ_TRY(bc.init(ctx, S));
  const size_t row = ((size_t)n + 15) / 16 * 16;
  double2 *vec, *dmu;
  LQ_TRY(ctx_buf(ctx, "nb_cheb", sizeof(double2) * 5 * row, (void **)&vec));
  LQ_TRY(ctx_buf(ctx, "nb_mu", sizeof(double2) * (size_t)M, (void **)&dmu));
  double2 *c0 = vec, *c1 = vec + row, *tmp = vec + 2 * row, *tmp2 = vec + 3 * row, *ph = vec + 4 * row;
  LQ_HIP_CHECK(hipMemcpyAsync(dmu, mu, sizeof(double2) * (size_t)M, hipMemcpyHostToDevice, ctx->stream));
  const dim3 gr(bc.grid), blk(kNbThreads);
  for (int r = 0; r < R; ++r) {
    LQ_TRY(upload_states(ctx, phi, n, r, 1, ph));
    // SetInitVectors_nonOrthogonal: T0 = [OP] S^-1 phi, T1 = S^-1 H T0
    if (!OP) {
      LQ_TRY(bc.solve(ph, c0, tol, maxit, nullptr, nullptr));
    } else {
      LQ_TRY(bc.solve(ph, tmp, tol, maxit, nullptr, nullptr));
      LQ_TRY(lq_spmv(OP, 1.0, 0.0, (const double *)tmp, 0.0, 0.0, (double *)c0, 1));
    }
    LQ_TRY(lq_spmv(H, 1.0, 0.0, (const double *)c0, 0.0, 0.0, (double *)tmp, 1));
    LQ_TRY(bc.solve(tmp, c1, tol, maxit, nullptr, nullptr));
    for (int m = 0; m < M; ++m) {
      double scal = 2.0 / R;
      if (m == 0) scal *= 0.5;
      hipLaunchKernelGGL(k_nb_dot2, gr, blk, 0, ctx->stream, n, ph, c0, nullptr, nullptr, bc.partial);
      LQ_HIP_CHECK(hipGetLastError());
      hipLaunchKernelGGL(k_nb_final, dim3(1), blk, 0, ctx->stream, bc.partial, bc.grid, bc.res, scal, dmu + m);
      LQ_HIP_CHECK(hipGetLastError());
      if (m + 1 == M) break;  // the reference's last Iterate leaves mu unchanged
      // Iterate_nonOrthogonal: T0 <- 2 S^-1 H T1 - T0, swap
      LQ_TRY(lq_spmv(H, 1.0, 0.0, (const double *)c1, 0.0, 0.0, (double *)tmp, 1));
      LQ_TRY(bc.solve(tmp, tmp2, tol, maxit, nullptr, nullptr));
      hipLaunchKernelGGL(k_nb_cheb, gr, blk, 0, ctx->stream, n, tmp2, c0);
      LQ_HIP_CHECK(hipGetLastError());
      std::swap(c0, c1);
    }
  }
  LQ_HIP_CHECK(hipMemcpyAsync(mu, dmu, sizeof(double2) * (size_t)M, hipMemcpyDeviceToHost, ctx->stream));
  LQ_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  if (iterations) *iterations = bc.iterations;
  return LQ_OK;
} LQ_ABI_CATCH
