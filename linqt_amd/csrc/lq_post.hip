// lq_post.hip -- moment epilogues, Jackson damping and energy-grid sums.
//
// All FP64.  The single-thread sequential scans (cumulative integrals) keep
// the reference's left-to-right summation order.
#include <algorithm>

#include "lq_internal.h"

namespace lq {

namespace {

constexpr double kPi = 3.14159265358979323846;

// Order of the Chebyshev vector the reference stores at padded index p when
// BATCH_SIZE = B: every IterateAll call after the first restarts at the last
// stored order (src/chebyshev_vectors.cpp:4-21), so block q covers orders
// q*(B-1) .. q*(B-1)+B-1.
__device__ __forceinline__ int batch_order(int p, int B) { return (p / B) * (B - 1) + (p % B); }

// Scaling + Hermitian symmetrisation of CorrelationExpansionMoments
// (src/chebyshev_solver.cpp:149-162) on the padded table, restricted to the
// M0 x M1 block that survives the final truncation (:165-169).  raw holds
// true-order moments summed over states; init (nullable) the caller's table.
__global__ void k_corr_epilogue(const double2 *__restrict__ raw, int ldr, const double2 *__restrict__ init, int M0,
                                int M1, int B, int R, double2 *__restrict__ out) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)M0 * M1) return;
  const int p = (int)(t / M1), q = (int)(t % M1);
  const int op = batch_order(p, B), oq = batch_order(q, B);
  double2 apq = raw[(size_t)op * ldr + oq];
  double2 aqp = raw[(size_t)oq * ldr + op];
  if (init) {
    const double2 i1 = init[(size_t)p * M1 + q];
    apq.x += i1.x;
    apq.y += i1.y;
    if (q < M0 && p < M1) {
      const double2 i2 = init[(size_t)q * M1 + p];
      aqp.x += i2.x;
      aqp.y += i2.y;
    }
  }
  // the reference visits each unordered pair once with mL <= mR
  const int lo = p <= q ? p : q, hi = p <= q ? q : p;
  const double2 first = p <= q ? apq : aqp;   // mu(lo, hi)
  const double2 second = p <= q ? aqp : apq;  // mu(hi, lo)
  double scal = 4.0 / R;
  if (lo == 0) scal *= 0.5;
  if (hi == 0) scal *= 0.5;
  const double tx = scal * (first.x + second.x) / 2.0;
  const double ty = scal * (first.y - second.y) / 2.0;
  out[t] = p <= q ? make_double2(tx, ty) : make_double2(tx, -ty);
}

// ---- sums along a table's diagonals -------------------------------------------
// The energy-grid formulas weigh mu(m0, m1) by products of one factor in m0 and
// one in m1 that are cosines, sines or e^{-i m theta}, some times m.  Such a
// product depends on m0 + m1 and m1 - m0 only, so a formula at any number of
// energies needs no more than the table's sums along its antidiagonals and
// diagonals, O(M) terms per energy in place of O(M^2).  At M = 512 the 15360
// energies of the linear-grid Bastin tool took 2.28 ms as a matrix-vector
// product per energy (bound by re-reading the table from L2: 64 GB) and take
// 0.05 ms for the sums and 0.07 ms for the energies; the 2048 energies of a
// Kubo table 0.32 ms and now 0.06, 8e-16 from exact angles instead of 1e-14.
//
// part[chunk][4][Q], Q = M0 + M1 - 1, of the rows m0 of the chunk, index t:
//   0: sum over m0 + m1 = t of v, 1: of w v, 2: over m1 - m0 = t - (M0 - 1) of v,
//   3: of w v;  v = c[m0] c[m1] mu(m0, m1) (c null: 1), w = m0 or m1.
// Thread t reads one element of each row, consecutive threads consecutive ones.
__global__ __launch_bounds__(64) void k_diag_sums(const double2 *__restrict__ mu, int ld, int M0, int M1, int rows,
                                                  const double *__restrict__ c, int weight_m1,
                                                  double2 *__restrict__ part) {
  const int Q = M0 + M1 - 1;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int r0 = blockIdx.y * rows, r1 = min(M0, r0 + rows);
  if (t >= Q) return;
  double2 a = make_double2(0.0, 0.0), a1 = a, b = a, b1 = a;
  auto add = [&](double2 &s, double2 &s1, int m0, int m1) {
    if (m1 < 0 || m1 >= M1) return;
    double2 v = mu[(size_t)m0 * ld + m1];
    if (c) {
      const double f = c[m0] * c[m1];
      v.x *= f;
      v.y *= f;
    }
    const double w = weight_m1 ? m1 : m0;
    s.x += v.x;
    s.y += v.y;
    s1.x = fma(w, v.x, s1.x);
    s1.y = fma(w, v.y, s1.y);
  };
#pragma unroll 4
  for (int m0 = r0; m0 < r1; ++m0) {
    add(a, a1, m0, t - m0);
    add(b, b1, m0, t - (M0 - 1) + m0);
  }
  double2 *o = part + (size_t)blockIdx.y * 4 * Q + t;
  o[0] = a;
  o[Q] = a1;
  o[2 * (size_t)Q] = b;
  o[3 * (size_t)Q] = b1;
}

__device__ __forceinline__ double2 diag_sum(const double2 *__restrict__ part, int nchunk, int Q, int which, int t) {
  double2 v = make_double2(0.0, 0.0);
  for (int c = 0; c < nchunk; ++c) {
    const double2 p = part[((size_t)c * 4 + which) * Q + t];
    v.x += p.x;
    v.y += p.y;
  }
  return v;
}

// Sequences of a Kubo table for launch_kubo_energies, scaled: A at 0, B at F
// (B_q at index q mod F) and, with deriv, A' at 2 F.
__global__ __launch_bounds__(64) void k_diag_kubo(const double2 *__restrict__ part, int nchunk, int M, int F, int deriv,
                                                  double scale, double2 *__restrict__ seq) {
  const int Q = 2 * M - 1, t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= Q) return;
  const double2 a = diag_sum(part, nchunk, Q, 0, t), b = diag_sum(part, nchunk, Q, 2, t);
  const int q = t - (M - 1);
  seq[t] = make_double2(scale * a.x, scale * a.y);
  seq[F + (q < 0 ? q + F : q)] = make_double2(scale * b.x, scale * b.y);
  if (deriv) {
    const double2 d = diag_sum(part, nchunk, Q, 1, t);
    seq[2 * F + t] = make_double2(scale * d.x, scale * d.y);
  }
}

// U_q for q >= 0, interleaved [Q][4], of the grid tools (weight m1):
//   0: Re, even in q:  (A_q + B_q + B_-q) / 2,     1: Im, odd:  (A_q + B_q - B_-q) / 2,
//   2: Im, even, of the weighted sums,             3: Re, odd, of the weighted sums.
__global__ __launch_bounds__(64) void k_diag_grid(const double2 *__restrict__ part, int nchunk, int M0, int M1,
                                                  double *__restrict__ seq) {
  const int Q = M0 + M1 - 1, q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= Q) return;
  const double2 z = make_double2(0.0, 0.0);
  const double2 a = diag_sum(part, nchunk, Q, 0, q), a1 = diag_sum(part, nchunk, Q, 1, q);
  const bool p = q <= M1 - 1, m = q > 0 && q <= M0 - 1;
  const double2 bp = p ? diag_sum(part, nchunk, Q, 2, M0 - 1 + q) : z, bp1 = p ? diag_sum(part, nchunk, Q, 3, M0 - 1 + q) : z;
  const double2 bm = m ? diag_sum(part, nchunk, Q, 2, M0 - 1 - q) : z, bm1 = m ? diag_sum(part, nchunk, Q, 3, M0 - 1 - q) : z;
  seq[4 * q] = 0.5 * (a.x + bp.x + bm.x);
  seq[4 * q + 1] = 0.5 * (a.y + bp.y - bm.y);
  seq[4 * q + 2] = 0.5 * (a1.y + bp1.y + bm1.y);
  seq[4 * q + 3] = 0.5 * (a1.x + bp1.x - bm1.x);
}

// rearrange_crescent_order (src/Kubo_solver_FFT_postProcess.cpp:98-116) as an
// index map: position j of the rearranged array holds original index src(j).
__device__ __forceinline__ int crescent_src(int j, int nump) {
  // second pass reverses the first nump/2 pairs: j <-> nump-1-j for j < nump/2
  int i = j;
  if (j < nump / 2)
    i = nump - 1 - j;
  else if (j >= nump - nump / 2)
    i = nump - 1 - j;
  // first pass: even 2k <- k, odd 2k+1 <- nump-1-k (k < nump/2); others unchanged
  if (i < 2 * (nump / 2)) return (i % 2 == 0) ? i / 2 : nump - 1 - i / 2;
  return i;
}

// out(i) = sum of term(j), j <= i, for i < n, by one block of 256 threads in the
// reference's order, left to right: the terms of a chunk are formed by all
// threads, added up by thread 0, and stored by all.  15360 terms read, added and
// stored by one thread took 3.65 ms (a memory round trip each); 0.19 ms here,
// where the chain of dependent additions is what is left.
constexpr int kScan = 2048;
template <class Term, class Store>
__device__ void ordered_sums(int n, Term term, Store store) {
  __shared__ double sh[kScan];
  const int tid = threadIdx.x;
  double acc = 0.0;
  for (int base = 0; base < n; base += kScan) {
    const int len = min(kScan, n - base);
    for (int i = tid; i < kScan; i += 256) sh[i] = i < len ? term(base + i) : 0.0;
    __syncthreads();
    if (tid == 0) {
      for (int i = 0; i < len; i += 16) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = sh[i + u];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = acc += v[u];
#pragma unroll
        for (int u = 0; u < 16; ++u) sh[i + u] = v[u];
      }
    }
    __syncthreads();
    for (int i = tid; i < len; i += 256) store(base + i, sh[i]);
    __syncthreads();
  }
}

// Kubo_solver_FFT_postProcess (src/Kubo_solver_FFT_postProcess.cpp:8-16, 36-47,
// 120-273, 279-397): the columns of each energy; Bastin's cumulative sum in
// k_kubo_post_sums.
__device__ __forceinline__ double kubo_energy(int j, int nump) {
  return cos(kPi * (2 * crescent_src(j, nump) + 0.5) / nump);
}

__global__ __launch_bounds__(64) void k_kubo_post(int formula, const double2 *__restrict__ fd, int nump, int n, double W,
                                                  double Ec, double *__restrict__ Eo, double *__restrict__ so,
                                                  double *__restrict__ integ) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nump) return;
  const double a = W / 2.0, b = Ec;
  const double omega = n / (a * a);
  const int k = crescent_src(j, nump);
  const double e = kubo_energy(j, nump);
  Eo[j] = a * e - b;
  if (formula == LQ_KUBO_BASTIN) {
    double v = e * fd[k].x - (sqrt(1.0 - e * e) * fd[k + nump].y);
    v *= 1.0 / pow((1.0 - e * e), 2.0);
    v *= omega / (kPi);
    integ[j] = v;
  } else {
    so[j] = 2.0 * omega * fd[k].x / (1.0 - e * e) / (2 * kPi);
    if (integ) integ[j] = 0.0;
  }
}

// ascending energies, left-Riemann cumulative sum
__global__ __launch_bounds__(256) void k_kubo_post_sums(int nump, const double *__restrict__ integ,
                                                        double *__restrict__ so) {
  ordered_sums(
      nump - 1, [&](int i) { return integ[i] * (kubo_energy(i + 1, nump) - kubo_energy(i, nump)); },
      [&](int i, double v) { so[i] = v; });
  if (threadIdx.x == 0) so[nump - 1] = 0.0;
}

// Moments1D::ApplyJacksonKernel (src/chebyshev_moments1D.cpp:79-86).
__global__ void k_jackson_1d(double2 *__restrict__ mu, int maxMom) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= maxMom) return;
  const double phi_J = kPi / (double)(maxMom + 1.0);
  const double g = ((double)(maxMom - m + 1) * cos(phi_J * m) + sin(phi_J * m) * cos(phi_J) / sin(phi_J)) * phi_J /
                   kPi;
  mu[m].x *= g;
  mu[m].y *= g;
}

// Moments2D::MomentNumber + ApplyJacksonKernel (src/chebyshev_moments2D.cpp:87-117).
__global__ void k_jackson_2d(const double2 *__restrict__ in, int M1_in, double2 *__restrict__ out, int mm0, int mm1) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)mm0 * mm1) return;
  const int m0 = (int)(t / mm1), m1 = (int)(t % mm1);
  const double phi0 = kPi / (double)(mm0 + 1.0), phi1 = kPi / (double)(mm1 + 1.0);
  const double g0 = ((mm0 - m0 + 1) * cos(phi0 * m0) + sin(phi0 * m0) * cos(phi0) / sin(phi0)) * phi0 / kPi;
  const double g1 = ((mm1 - m1 + 1) * cos(phi1 * m1) + sin(phi1 * m1) * cos(phi1) / sin(phi1)) * phi1 / kPi;
  const double g = g0 * g1;
  const double2 v = in[(size_t)m0 * M1_in + m1];
  out[t] = make_double2(v.x * g, v.y * g);
}

// include/chebyshev_coefficients.hpp:8-32; pow(complex, m) as libstdc++ does
// it: polar(exp(m log|z|), m arg z).
__device__ __forceinline__ double delta_chebF(double x, double m) {
  const double f0 = sqrt(1.0 - x * x);
  return cos(m * acos(x)) / f0 / kPi;
}

__device__ __forceinline__ double2 zpow(double zr, double zi, double m) {
  const double lr = log(hypot(zr, zi)), li = atan2(zi, zr);
  const double rho = exp(m * lr);
  double sn, cs;
  sincos(m * li, &sn, &cs);
  return make_double2(rho * cs, rho * sn);
}

__device__ __forceinline__ double2 greenR_chebF(double x, double m) {
  const double f0 = sqrt(1.0 - x * x);
  const double2 fm = zpow(x, -f0, m);
  // -I * fm / f0
  return make_double2(fm.y / f0, -fm.x / f0);
}

__device__ __forceinline__ double2 DgreenR_chebF(double x, double m) {
  const double f0 = sqrt(1.0 - x * x);
  const double2 p = zpow(x, -f0, m);
  const double2 fm = make_double2(p.x * x - p.y * (m * f0), p.x * (m * f0) + p.y * x);
  // -I * fm / f0 / f0 / f0
  return make_double2(fm.y / f0 / f0 / f0, -fm.x / f0 / f0 / f0);
}

// spectralFunctionFromChebmom_FFTgrid.cpp:60-73.
// One wavefront per energy: lane l sums the moments m = l, l + 64, ..., then
// the 64 lane sums are added in a fixed tree (deterministic).
__global__ __launch_bounds__(64) void k_dos_fftgrid(const double2 *__restrict__ mu, int M, int n, double W, double Ec,
                                                    int num_div, double *__restrict__ E, double *__restrict__ rho) {
  __shared__ double sh[64];
  const int i = blockIdx.x;
  const int l = threadIdx.x;
  const double a = W / 2.0;
  const double energ = cos(kPi * (i + 0.5) / num_div);
  double part = 0;
  for (int m0 = l; m0 < M; m0 += 64) part += delta_chebF(energ, m0) * mu[m0].x;
  sh[l] = part;
  __syncthreads();
  for (int h = 32; h > 0; h >>= 1) {
    if (l < h) sh[l] += sh[l + h];
    __syncthreads();
  }
  if (l == 0) {
    E[i] = energ * a + Ec;
    rho[i] = fabs(sh[0] * (n / a));
  }
}

// kuboGreenwoodFromChebmom_FFTgrid.cpp:57-66 and kuboBastinFromChebmom_FFTgrid.cpp:77-86:
// one block per energy; thread j owns columns m1 = j, j+256, ...:
//   kernel = sum_m1 Im( G(E, m1) * sum_m0 delta(E, m0) mu(m0, m1) ).
// Not through the table's diagonal sums: these grids go up to the band edges,
// where the sum over m0 cancels and 1/f^4 magnifies what is left of it; from
// the diagonal sums the Bastin curve at M = 512 was 1.3e-10 off instead of 9e-12
// (0.13 ms against 0.09).
template <int DERIV>
__global__ __launch_bounds__(256) void k_grid2d(const double2 *__restrict__ mu, int M0, int M1, const double *__restrict__ energies,
                                                double *__restrict__ kern) {
  extern __shared__ double dl[];  // delta(E, m0)
  const int i = blockIdx.x;
  const double energ = energies[i];
  for (int m0 = threadIdx.x; m0 < M0; m0 += blockDim.x) dl[m0] = delta_chebF(energ, m0);
  __syncthreads();
  double acc = 0;
  for (int m1 = threadIdx.x; m1 < M1; m1 += blockDim.x) {
    double zr = 0, zi = 0;
    for (int m0 = 0; m0 < M0; ++m0) {
      const double2 v = mu[(size_t)m0 * M1 + m1];
      zr = fma(dl[m0], v.x, zr);
      zi = fma(dl[m0], v.y, zi);
    }
    const double2 g = DERIV ? DgreenR_chebF(energ, m1) : greenR_chebF(energ, m1);
    acc += g.x * zi + g.y * zr;  // Im(g * z)
  }
  __shared__ double red[256];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) kern[i] = red[0];
}

// Linear-grid tools (src/*FromChebmom.cpp), kinds as LQ_LIN_*.  Every tool's
// double sum is sum_m1 proj( b_m1(x) * sum_m0 a_m0(x) mu(m0, m1) ) with
// (a, b, proj) = (delta, gR, Im) Greenwood/BastinI, (delta, DgR, Im) Bastin,
// (delta, delta, Re) Surf, (Im gR, Re DgR, 4 Im) Sea; BastinII uses the two left
// vectors gR and DgR: -Re(DgR_m1 z_gR - gR_m1 z_DgR).
__device__ __forceinline__ double lin_xgrid(int kind, int i, int num_div) {
  const double xb = kind == 2 ? 0.99 : 1.0;
  return -xb + i * (2 * xb) / (num_div - 1);
}

// Blocks of kLinE energies, the sums as written above: every energy of the tools
// Spectral, BastinII, Sea and of small tables (ends = num_div), else the first and
// last `ends` energies, see k_grid_energies.  x = +-1 makes every coefficient
// infinite, and the printed NaN or infinity is the one the sources' order of
// operations gives.  What bounds them is the wait for the table's rows, 4 MB a block
// at M = 512: the energies of a block share a reading, eight rows are on their way
// at a time (the compiler waits for each row where the batch may end early), and
// all blocks are resident.  620 energies at M = 512, Bastin: 51 us; two energies
// 73; two and one row at a time 133, with 256 threads 250.
template <int KIND>
constexpr int kLinE = KIND == 0 || KIND == 4 ? 1 : 4;
constexpr int kLinRows = 8;
template <int KIND>
constexpr int kLinT = KIND == 0 || KIND == 4 ? 256 : 512;

template <int KIND>
__global__ __launch_bounds__(kLinT<KIND>) void k_linear_kernel(const double2 *__restrict__ mu, int M0, int M1,
                                                               int num_div, int ends, int count, double scale,
                                                               double *__restrict__ kern) {
  extern __shared__ double2 lv[];  // left vectors: [M0][kE] doubles (BastinII: [2][M0] complex)
  constexpr int kE = kLinE<KIND>;
  double *lx = (double *)lv;
  int i[kE];
  double x[kE];
#pragma unroll
  for (int e = 0; e < kE; ++e) {
    const int t = min((int)blockIdx.x * kE + e, count - 1);
    i[e] = t < ends ? t : num_div - count + t;
    x[e] = lin_xgrid(KIND, i[e], num_div);
  }
  for (int m0 = threadIdx.x; m0 < M0; m0 += blockDim.x) {
    if (KIND == 4) {
      lv[m0] = greenR_chebF(x[0], m0);
      lv[M0 + m0] = DgreenR_chebF(x[0], m0);
    } else {
#pragma unroll
      for (int e = 0; e < kE; ++e) lx[m0 * kE + e] = KIND == 5 ? greenR_chebF(x[e], m0).y : delta_chebF(x[e], m0);
    }
  }
  __syncthreads();
  double acc[kE] = {};
  if (KIND == 0) {
    for (int m0 = threadIdx.x; m0 < M0; m0 += blockDim.x) acc[0] += lx[m0] * mu[m0].x;
  } else {
    for (int m1 = threadIdx.x; m1 < M1; m1 += blockDim.x) {
      double zr[kE] = {}, zi[kE] = {}, wr = 0, wi = 0;
      auto add = [&](int m0, double2 v) {
        if (KIND == 4) {
          const double2 l = lv[m0], dl = lv[M0 + m0];
          zr[0] += l.x * v.x - l.y * v.y;
          zi[0] += l.x * v.y + l.y * v.x;
          wr += dl.x * v.x - dl.y * v.y;
          wi += dl.x * v.y + dl.y * v.x;
        } else {
#pragma unroll
          for (int e = 0; e < kE; ++e) {
            const double l = lx[m0 * kE + e];
            zr[e] = fma(l, v.x, zr[e]);
            zi[e] = fma(l, v.y, zi[e]);
          }
        }
      };
      int m0 = 0;
      for (; m0 + kLinRows <= M0; m0 += kLinRows) {
        double2 row[kLinRows];
#pragma unroll
        for (int u = 0; u < kLinRows; ++u) row[u] = mu[(size_t)(m0 + u) * M1 + m1];
        __builtin_amdgcn_sched_barrier(0);  // all on their way before the first is used
#pragma unroll
        for (int u = 0; u < kLinRows; ++u) add(m0 + u, row[u]);
      }
      for (; m0 < M0; ++m0) add(m0, mu[(size_t)m0 * M1 + m1]);
#pragma unroll
      for (int e = 0; e < kE; ++e) {
        if (KIND == 1 || KIND == 3) {
          const double2 g = greenR_chebF(x[e], m1);
          acc[e] += g.x * zi[e] + g.y * zr[e];  // Im(g z)
        } else if (KIND == 2) {
          const double2 g = DgreenR_chebF(x[e], m1);
          acc[e] += g.x * zi[e] + g.y * zr[e];
        } else if (KIND == 6) {
          acc[e] += delta_chebF(x[e], m1) * zr[e];
        } else if (KIND == 5) {
          acc[e] += 4.0 * DgreenR_chebF(x[e], m1).x * zi[e];
        } else {  // 4: -Re(DgR z_gR - gR z_DgR)
          const double2 d = DgreenR_chebF(x[e], m1), g = greenR_chebF(x[e], m1);
          acc[e] += -((d.x * zr[e] - d.y * zi[e]) - (g.x * wr - g.y * wi));
        }
      }
    }
  }
  __shared__ double red[kE][kLinT<KIND>];
#pragma unroll
  for (int e = 0; e < kE; ++e) red[e][threadIdx.x] = acc[e];
  __syncthreads();
  for (int s = kLinT<KIND> / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
#pragma unroll
      for (int e = 0; e < kE; ++e) red[e][threadIdx.x] += red[e][threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
#pragma unroll
    for (int e = 0; e < kE; ++e) kern[i[e]] = red[e][0] * scale;
  }
}

// The same sums through the table's diagonal sums U (k_diag_grid): with
// theta = acos x, f = sin theta,
//   C1 = sum cos m0 cos m1 Re mu = sum_q U0 cos q theta,  S1 = sum cos m0 sin m1 Im mu = sum U1 sin,
//   C2 = sum m1 cos m0 cos m1 Im mu = sum U2 cos,         S2 = sum m1 cos m0 sin m1 Re mu = sum U3 sin,
//   Greenwood, BastinI  -(C1 + S1) / (pi f^2);   Surf  C1 / (pi f)^2;
//   Bastin  [f (C2 - S2) - x (C1 + S1)] / (pi f^4).
// One wavefront for kEw energies (the U of a lane's q are loaded once for all), i
// from `ends` to num_div - ends: towards the band ends the sums over one index
// nearly cancel and 1/f^4 magnifies what is left of U's rounding, so there the
// double sums are formed as written (k_linear_kernel).  The phase q theta' is
// reduced with its rounding (theta' = acos |x|, with the parity of q for x < 0).
constexpr int kEw = 4;
template <int KIND>
__global__ __launch_bounds__(64) void k_grid_energies(const double *__restrict__ seq, int Q, int num_div, int ends,
                                                      double scale, double *__restrict__ kern) {
  const int l = threadIdx.x, i0 = ends + blockIdx.x * kEw;
  double x[kEw], th[kEw], u[kEw], v[kEw];
#pragma unroll
  for (int e = 0; e < kEw; ++e) {
    const int i = min(i0 + e, num_div - 1);
    x[e] = lin_xgrid(KIND, i, num_div);
    th[e] = acos(fabs(x[e]));
    u[e] = v[e] = 0.0;
  }
  for (int q = l; q < Q; q += 64) {
    const double4 w = *(const double4 *)(seq + 4 * (size_t)q);
#pragma unroll
    for (int e = 0; e < kEw; ++e) {
      const double ph = q * th[e], lo = fma((double)q, th[e], -ph);
      double s0, c0;
      sincos(ph, &s0, &c0);
      double sn = fma(c0, lo, s0), cs = fma(-s0, lo, c0);
      if (x[e] < 0.0) {  // q theta = q pi - q theta'
        if (q & 1)
          cs = -cs;
        else
          sn = -sn;
      }
      // u: the sum without the weight m1, v: the weighted one
      if (KIND == 6) {
        u[e] = fma(w.x, cs, u[e]);
      } else {
        u[e] = fma(w.x, cs, fma(w.y, sn, u[e]));
        if (KIND == 2) v[e] = fma(w.z, cs, fma(-w.w, sn, v[e]));
      }
    }
  }
#pragma unroll
  for (int e = 0; e < kEw; ++e) {
    for (int d = 32; d > 0; d >>= 1) {
      u[e] += __shfl_down(u[e], d);
      v[e] += __shfl_down(v[e], d);
    }
    const int i = i0 + e;
    if (l == 0 && i < num_div - ends) {
      const double f2 = 1.0 - x[e] * x[e], f = sqrt(f2);
      double r;
      if (KIND == 6)
        r = u[e] / f2 / (kPi * kPi);
      else if (KIND == 2)
        r = (f * v[e] - x[e] * u[e]) / f2 / f2 / kPi;
      else
        r = -u[e] / f2 / kPi;
      kern[i] = r * scale;
    }
  }
}

// The printed columns: E and the values that need no running sum.
__global__ __launch_bounds__(64) void k_linear_columns(int kind, int num_div, double a, double Ec,
                                                       const double *__restrict__ kern, double *__restrict__ E,
                                                       double *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (kind == 0 ? num_div : num_div - 1)) return;
  E[i] = lin_xgrid(kind, i, num_div) * a + Ec;
  switch (kind) {
    case 0: case 1: out[i] = kern[i]; break;
    case 3: out[i] = 0.5 * (kern[i] + kern[i + 1]); break;
    case 6: out[i] = (kern[i + 1] + kern[i]) / 2.0; break;
    default: break;  // k_linear_sums
  }
}

__global__ __launch_bounds__(256) void k_linear_sums(int kind, int num_div, const double *__restrict__ kern,
                                                     double *__restrict__ out) {
  ordered_sums(
      num_div - 1,
      [&](int i) {
        const double dx = lin_xgrid(kind, i + 1, num_div) - lin_xgrid(kind, i, num_div);
        return kind == 2 ? kern[i] * dx : kind == 4 ? (kern[i] + kern[i + 1]) * dx : 0.5 * (kern[i] + kern[i + 1]) * dx;
      },
      [&](int i, double v) { out[i] = v; });
}

// y (=|+=) c x over count complex elements (Bessel-Chebyshev time evolution).
__global__ void k_caxpy(double2 c, const double2 *__restrict__ x, double2 *__restrict__ y, size_t count,
                        int overwrite) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const double2 v = x[i];
  double2 r = make_double2(c.x * v.x - c.y * v.y, c.x * v.y + c.y * v.x);
  if (!overwrite) {
    const double2 o = y[i];
    r.x += o.x;
    r.y += o.y;
  }
  y[i] = r;
}

// MomentsTD::ApplyJacksonKernel (src/chebyshev_momentsTD.cpp:135-154): row m of
// the M x nT table (rows kept: maxMom) times g_m.
__global__ void k_jackson_td(double2 *__restrict__ mu, int maxMom, int nT) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)maxMom * nT) return;
  const int m = (int)(t / nT);
  const double phi_J = kPi / (double)(maxMom + 1.0);
  const double g = ((maxMom - m + 1) * cos(phi_J * m) + sin(phi_J * m) * cos(phi_J) / sin(phi_J)) * phi_J / kPi;
  mu[t].x *= g;
  mu[t].y *= g;
}

// timeCorrelationsFromChebmom.cpp:60-70: one thread per time step.
__global__ void k_timecorr_post(const double2 *__restrict__ mu, int M, int nT, int n, double a, double x, double dt,
                                double *__restrict__ tout, double *__restrict__ out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nT) return;
  double o = 0.0;
  for (int m = 0; m < M; ++m) o += delta_chebF(x, m) * mu[(size_t)m * nT + t].x;
  tout[t] = t * dt;
  out[t] = o * (n / a);
}

__global__ void k_greenwood_energies(int num_div, double *__restrict__ e) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < num_div) e[i] = cos(kPi * (2 * i + 0.5) / num_div);
}

__global__ void k_bastin_energies(int num_div, double *__restrict__ e) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < num_div) e[j] = cos(kPi * (2 * crescent_src(j, num_div) + 0.5) / num_div);
}

__global__ void k_greenwood_finish(int num_div, int n, double W, double Ec, const double *__restrict__ energies,
                                   const double *__restrict__ kern, double *__restrict__ E, double *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num_div - 1) return;
  const double a = W / 2.0;
  E[i] = energies[i] * a + Ec;
  out[i] = -1.0 * kern[i] * (n / a / a);
}

__global__ __launch_bounds__(256) void k_bastin_finish(int num_div, int n, double W, double Ec,
                                                       const double *__restrict__ energies,
                                                       const double *__restrict__ kern, double *__restrict__ E,
                                                       double *__restrict__ out) {
  const double a = W / 2.0;
  for (int i = threadIdx.x; i < num_div - 1; i += 256) E[i] = energies[i] * a + Ec;
  ordered_sums(
      num_div - 1, [&](int i) { return kern[i] * (-2.0 * n / a / a) * (energies[i + 1] - energies[i]); },
      [&](int i, double v) { out[i] = v; });
}

// Rows of a table summed by one block of k_diag_sums: enough blocks for the
// chip at M = 512 (16 x 16), at most 64 partial sums of a diagonal.
int diag_rows(int M0) { return std::max(32, (M0 + 63) / 64); }
int diag_chunks(int M0) { return (M0 + diag_rows(M0) - 1) / diag_rows(M0); }

int launch_diag_sums(hipStream_t st, const double2 *mu, int ld, int M0, int M1, const double *c, int weight_m1,
                     double2 *part) {
  const int Q = M0 + M1 - 1, rows = diag_rows(M0);
  hipLaunchKernelGGL(k_diag_sums, dim3((Q + 63) / 64, diag_chunks(M0)), dim3(64), 0, st, mu, ld, M0, M1, rows, c,
                     weight_m1, part);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

// kern[i], ends <= i < num_div - ends, of a grid tool (kinds as k_grid_energies)
// from the table's diagonal sums.
int launch_grid_kernel(hipStream_t st, int kind, const double2 *mu, int M0, int M1, int num_div, int ends, double scale,
                       double2 *diag, double *kern) {
  const int Q = M0 + M1 - 1;
  LQ_TRY(launch_diag_sums(st, mu, M1, M0, M1, nullptr, 1, diag));
  double *seq = (double *)(diag + (size_t)4 * Q * diag_chunks(M0));
  hipLaunchKernelGGL(k_diag_grid, dim3((Q + 63) / 64), dim3(64), 0, st, diag, diag_chunks(M0), M0, M1, seq);
  const dim3 grid((num_div - 2 * ends + kEw - 1) / kEw);
  switch (kind) {
#define LQ_GE(K) \
  hipLaunchKernelGGL((k_grid_energies<K>), grid, dim3(64), 0, st, seq, Q, num_div, ends, scale, kern)
    case 1: case 3: LQ_GE(1); break;
    case 2: LQ_GE(2); break;
    case 6: LQ_GE(6); break;
#undef LQ_GE
  }
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

}  // namespace

size_t diag_bytes(int M0, int M1) {
  return sizeof(double2) * (size_t)4 * (M0 + M1 - 1) * diag_chunks(M0) + 4 * sizeof(double) * (size_t)(M0 + M1 - 1);
}

int launch_diag_kubo(hipStream_t st, const double2 *raw, int M, const double *coef, int formula, double scale, int F,
                     double2 *diag, double2 *seq) {
  const int Q = 2 * M - 1;
  LQ_TRY(launch_diag_sums(st, raw, M, M, M, coef, 0, diag));
  hipLaunchKernelGGL(k_diag_kubo, dim3((Q + 63) / 64), dim3(64), 0, st, diag, diag_chunks(M), M, F,
                     formula == LQ_KUBO_BASTIN ? 1 : 0, scale, seq);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_linear_grid(hipStream_t st, int kind, const double2 *mu, int M0, int M1, int n, double W, double Ec,
                       int num_div, double2 *diag, double *kern, double *E, double *out) {
  const double a = W / 2.0;
  double scale;
  switch (kind) {
    case 0: scale = n / a; break;
    case 1: case 3: scale = -1.0 * (n / a / a); break;
    case 2: scale = -2.0 * n / a / a; break;
    case 4: case 5: scale = n / a / a / 2 / kPi; break;
    case 6: scale = kPi * n / a / a; break;
    default:
      set_error("launch_linear_grid: unknown kind %d", kind);
      return LQ_ERR_ARG;
  }
  const int most_orders = kind == 4 ? 2048 : 4096;
  if (M0 > most_orders) {
    set_error("launch_linear_grid: %d moments exceed the LDS table (max %d)", M0, most_orders);
    return LQ_ERR_UNSUPPORTED;
  }
  // Through the diagonal sums from 64 x 64 moments on; below, the double sums take a
  // few microseconds.  Energies with |x| > 0.95 are left to the double sums.  Damped
  // tables of 64 to 512 orders with levels inside (-0.93, 0.93), largest error against
  // 80-bit sums over the curve's largest value, double / diagonal sums: |x| < 0.95
  // 2e-15 .. 6e-13 / 3e-16 .. 3e-14 (never the larger one), but 0.97 < |x| < 0.99
  // (Bastin) 8e-16 .. 2e-14 / 4e-15 .. 2e-13 and beyond 0.998 (Greenwood, Surf)
  // 1e-15 .. 1e-13 / 4e-15 .. 3e-13.
  // Sea stays with the double sums throughout: its running sum begins with the NaN of
  // x = -1, so no printed value could show an error of another form.
  const bool diagonal = (kind == 1 || kind == 2 || kind == 3 || kind == 6) && (long long)M0 * M1 >= 4096;
  const double xb = kind == 2 ? 0.99 : 1.0;
  const int most = (num_div + 1) / 2;
  const int ends = diagonal ? std::max(1, std::min(most, (int)((xb - 0.95) / (2 * xb) * (num_div - 1)) + 1)) : num_div;
  const int count = std::min(num_div, 2 * ends);
  auto direct = [&](auto kernel, int per, int threads) -> int {
    const size_t lds = kind == 4 ? sizeof(double2) * 2 * (size_t)M0 : sizeof(double) * per * (size_t)M0;
    LQ_HIP_CHECK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kernel, dim3((count + per - 1) / per), dim3(threads), lds, st, mu, M0, M1, num_div, ends, count,
                       scale, kern);
    return LQ_OK;
  };
  if (diagonal && count < num_div) LQ_TRY(launch_grid_kernel(st, kind, mu, M0, M1, num_div, ends, scale, diag, kern));
  switch (kind) {
#define LQ_LIN(K) LQ_TRY(direct(k_linear_kernel<K>, kLinE<K>, kLinT<K>))
    case 0: LQ_LIN(0); break;
    case 1: case 3: LQ_LIN(1); break;
    case 2: LQ_LIN(2); break;
    case 4: LQ_LIN(4); break;
    case 5: LQ_LIN(5); break;
    case 6: LQ_LIN(6); break;
#undef LQ_LIN
  }
  hipLaunchKernelGGL(k_linear_columns, dim3((num_div + 63) / 64), dim3(64), 0, st, kind, num_div, a, Ec, kern, E, out);
  if (kind == 2 || kind == 4 || kind == 5)
    hipLaunchKernelGGL(k_linear_sums, dim3(1), dim3(256), 0, st, kind, num_div, kern, out);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_caxpy(hipStream_t st, double2 c, const double2 *x, double2 *y, size_t count, int overwrite) {
  hipLaunchKernelGGL(k_caxpy, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, c, x, y, count, overwrite);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_jackson_td(hipStream_t st, double2 *mu, int maxMom, int nT) {
  const long long total = (long long)maxMom * nT;
  if (total <= 0) return LQ_OK;
  hipLaunchKernelGGL(k_jackson_td, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, mu, maxMom, nT);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_timecorr_post(hipStream_t st, const double2 *mu, int M, int nT, int n, double W, double Ec, double dt,
                         double EF, double *t, double *out) {
  const double a = W / 2.0;
  hipLaunchKernelGGL(k_timecorr_post, dim3((nT + 127) / 128), dim3(128), 0, st, mu, M, nT, n, a, (EF - Ec) / a, dt, t,
                     out);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_corr_epilogue(hipStream_t st, const double2 *raw, int ldr, const double2 *init, int M0, int M1, int B,
                         int R, double2 *out) {
  const long long total = (long long)M0 * M1;
  hipLaunchKernelGGL(k_corr_epilogue, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, raw, ldr, init, M0,
                     M1, B, R, out);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_kubo_post(hipStream_t st, int formula, const double2 *final_data, int nump, int n, double W, double Ec,
                     double *E, double *sigma, double *integrand) {
  if ((size_t)nump * sizeof(double) > 64 * 1024) {
    set_error("kubo_post: nump = %d exceeds 8192", nump);
    return LQ_ERR_ARG;
  }
  hipLaunchKernelGGL(k_kubo_post, dim3((nump + 63) / 64), dim3(64), 0, st, formula, final_data, nump, n, W, Ec, E, sigma,
                     integrand);
  if (formula == LQ_KUBO_BASTIN)
    hipLaunchKernelGGL(k_kubo_post_sums, dim3(1), dim3(256), 0, st, nump, integrand, sigma);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_jackson_1d(hipStream_t st, double2 *mu, int maxMom) {
  hipLaunchKernelGGL(k_jackson_1d, dim3((maxMom + 255) / 256), dim3(256), 0, st, mu, maxMom);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_jackson_2d(hipStream_t st, const double2 *mu_in, int M1_in, double2 *mu_out, int mm0, int mm1) {
  const long long total = (long long)mm0 * mm1;
  hipLaunchKernelGGL(k_jackson_2d, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, mu_in, M1_in, mu_out, mm0,
                     mm1);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_dos_fftgrid(hipStream_t st, const double2 *mu, int M, int n, double W, double Ec, int num_div, double *E,
                       double *rho) {
  hipLaunchKernelGGL(k_dos_fftgrid, dim3(num_div), dim3(64), 0, st, mu, M, n, W, Ec, num_div, E, rho);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_greenwood_fftgrid(hipStream_t st, const double2 *mu, int M0, int M1, int n, double W, double Ec,
                             int num_div, double *scratch, double *E, double *out) {
  double *energies = scratch, *kern = scratch + num_div;
  const size_t lds = sizeof(double) * (size_t)M0;
  if (lds > 64 * 1024) {
    set_error("greenwood_fftgrid: M0 = %d exceeds 8192", M0);
    return LQ_ERR_ARG;
  }
  hipLaunchKernelGGL(k_greenwood_energies, dim3((num_div + 255) / 256), dim3(256), 0, st, num_div, energies);
  hipLaunchKernelGGL((k_grid2d<0>), dim3(num_div), dim3(256), lds, st, mu, M0, M1, energies, kern);
  hipLaunchKernelGGL(k_greenwood_finish, dim3((num_div + 255) / 256), dim3(256), 0, st, num_div, n, W, Ec, energies,
                     kern, E, out);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_bastin_fftgrid(hipStream_t st, const double2 *mu, int M0, int M1, int n, double W, double Ec, int num_div,
                          double *scratch, double *E, double *out) {
  double *energies = scratch, *kern = scratch + num_div;
  const size_t lds = sizeof(double) * (size_t)M0;
  if (lds > 64 * 1024) {
    set_error("bastin_fftgrid: M0 = %d exceeds 8192", M0);
    return LQ_ERR_ARG;
  }
  hipLaunchKernelGGL(k_bastin_energies, dim3((num_div + 255) / 256), dim3(256), 0, st, num_div, energies);
  hipLaunchKernelGGL((k_grid2d<1>), dim3(num_div), dim3(256), lds, st, mu, M0, M1, energies, kern);
  hipLaunchKernelGGL(k_bastin_finish, dim3(1), dim3(256), 0, st, num_div, n, W, Ec, energies, kern, E, out);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

}  // namespace lq
