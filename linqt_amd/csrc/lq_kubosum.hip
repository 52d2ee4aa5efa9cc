// lq_kubosum.hip -- Kubo energy sums straight from the stored vectors.
//
// Kubo_solver_FFT (src/Kubo_solver_FFT.cpp:12-136, src/Greenwood_FFTs.cpp,
// src/Bastin_FFTs.cpp) forms, per energy, sums over the orders (m, n) of
// mu_mn = <L_m|R_n> times cos(m theta), exp(i n theta) and their derivatives.
// A product of two such factors depends on m + n or n - m alone, so the whole
// M x M table is not needed, only its weighted sums along the antidiagonals
// and diagonals (c_m the damping coefficients):
//   A_q  = sum_{m+n=q} c_m c_n mu_mn,   A'_q = sum_{m+n=q} m c_m c_n mu_mn,
//   B_q  = sum_{n-m=q} c_m c_n mu_mn,
//   Greenwood  r = Re (1/2) [ sum_q A_q cos q theta + sum_q B_q cos q theta ]
//   Bastin     p = sum_q A_q cos q phi + sum_q B_q e^{i q phi}        (phi = +-theta)
//              w = sum_q A'_q cos q phi - (1/2) sum_q q (A_q + B_q) e^{i q phi}.
// mu_mn is itself a sum over the N R stored elements of one site and state, and
// for one of them A and B are a convolution and a correlation of its two
// sequences of M orders.  Those are products of discrete Fourier transforms of
// length F >= 2M - 1, which are summed over the sites at each frequency; one
// inverse transform at the end gives A, A' and B.  Per site and state that is
// 2 + nopr transforms of length F instead of nopr M^2 complex multiply-adds:
// at M = 512 and two operators 0.25 Mflop instead of 3.1.
#include <algorithm>
#include <cmath>

#include "lq_internal.h"

namespace lq {

namespace {

constexpr int kP = 512;   // transform length of one frequency set
constexpr int kS = 4;     // sites a block transforms together
constexpr int kT = 512;   // threads of a block
constexpr int kTw = 64;   // twiddle table: first powers, the others are multiplied up

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 mul_mi(double2 a) { return make_double2(a.y, -a.x); }  // -i a
__device__ __forceinline__ void cfma(double2 &acc, double2 a, double2 b) {
  acc.x = fma(a.x, b.x, acc.x);
  acc.x = fma(-a.y, b.y, acc.x);
  acc.y = fma(a.x, b.y, acc.y);
  acc.y = fma(a.y, b.x, acc.y);
}

// y_k = sum_j x_j e^{-2 pi i j k / 8}, in place, natural order.
__device__ __forceinline__ void radix8(double2 (&x)[8]) {
  const double h = 0.70710678118654752440;
  double2 a0 = cadd(x[0], x[4]), a4 = csub(x[0], x[4]);
  double2 a2 = cadd(x[2], x[6]), a6 = mul_mi(csub(x[2], x[6]));
  double2 a1 = cadd(x[1], x[5]), a5 = csub(x[1], x[5]);
  double2 a3 = cadd(x[3], x[7]), a7 = mul_mi(csub(x[3], x[7]));
  const double2 b0 = cadd(a0, a2), b2 = csub(a0, a2);
  const double2 b1 = cadd(a1, a3), b3 = mul_mi(csub(a1, a3));
  const double2 c0 = cadd(a4, a6), c2 = csub(a4, a6);
  double2 c1 = cadd(a5, a7), c3 = csub(a5, a7);
  c1 = make_double2(h * (c1.x + c1.y), h * (c1.y - c1.x));   // e^{-i pi/4} c1
  c3 = make_double2(h * (c3.y - c3.x), -h * (c3.x + c3.y));  // e^{-3 i pi/4} c3
  x[0] = cadd(b0, b1);
  x[4] = csub(b0, b1);
  x[2] = cadd(b2, b3);
  x[6] = csub(b2, b3);
  x[1] = cadd(c0, c1);
  x[5] = csub(c0, c1);
  x[3] = cadd(c2, c3);
  x[7] = csub(c2, c3);
}

// t[i] = w^i, i = 1..7 (at most three products deep)
__device__ __forceinline__ void powers(double2 w, double2 (&t)[8]) {
  t[1] = w;
  t[2] = cmul(w, w);
  t[3] = cmul(t[2], w);
  t[4] = cmul(t[2], t[2]);
  t[5] = cmul(t[4], w);
  t[6] = cmul(t[4], t[2]);
  t[7] = cmul(t[4], t[3]);
}

// Barrier for LDS data alone: __syncthreads would also wait for the next tile's
// points, which are still on their way from memory.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct SumArgs {
  const double2 *L;      // [M][ld]
  const double2 *R[2];   // [M][ld] each
  long long K, ld;       // elements (sites x states) of one order, and between orders
  int M, H, fold;        // orders, frequency sets (F = 512 H), fold = ceil(M / 512)
  const double2 *wt;     // [H][512 fold]: c_m e^{-2 pi i h m / F}, 0 for m >= M
  const double2 *tw;     // [64]: e^{-2 pi i k / 512}
  double2 *partial;      // [blocks][arrays][F]
};

// The remaining two radix-8 passes of a 512-point transform by one wavefront, in
// the LDS region z.  Before: slot (64 k1 + j) ^ sw holds the first pass's output
// k1 of the points j, j + 64, ..., twiddled.  After: slot g holds frequency g.
// t: powers of e^{-2 pi i j1 / 64}, j1 = lane % 8.  A wavefront's LDS accesses
// complete in order, so no barrier is needed between the passes; the slots
// between them are swizzled against bank conflicts.
__device__ __forceinline__ void finish_fft(double2 *z, int sw, const double2 (&t)[8], int lane) {
  const int lo = lane & 7, hi = lane >> 3;
  double2 x[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = z[64 * hi + 8 * i + (lo ^ sw)];  // k1 = hi, j1 = lo, j2 = i
  radix8(x);
#pragma unroll
  for (int i = 1; i < 8; ++i) x[i] = cmul(x[i], t[i]);
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i) z[64 * hi + 8 * i + (lo ^ i ^ hi)] = x[i];  // [k1][k2][j1], swizzled
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = z[64 * lo + 8 * hi + (i ^ hi ^ lo)];  // k1 = lo, k2 = hi, j1 = i
  radix8(x);
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i) z[lane + 64 * i] = x[i];  // g = k1 + 8 k2 + 64 k3
}

// One block: frequency sets set0 .. set0 + NSET - 1 (set h: frequencies
// f = H g + h, g < 512) of the site tiles it walks over.  A tile's kS sites are
// consecutive, 64 bytes of each order.  Per tile and set:
//   1. thread (site s, j < 64) of a vector weighs its points j + 64 k, does the
//      first radix-8 pass over k and stores the eight results in LDS;
//   2. each wavefront finishes whole transforms (finish_fft);
//   3. thread g adds the products of the tile's spectra at its frequency.
// Jobs (spectra): 0 conj(L), 1 m conj(L) (DERIV), then R_0, R_1, and last L
// itself when the set does not contain its own negative frequencies.
// FOLD: M > 512, the points m, m + 512, ... are folded into one while loading
// (one set per block, no points held over from the tile before).
//
// What bounds it (M = 512, two operators, 2^21 elements, 51.5 GB, Bastin): with
// the loads taken out the same work takes 20.4 ms (vector units busy 65 % of
// the cycles, LDS 50 %), the loads alone 11.9 ms; together 24.8 ms = 2.1 TB/s,
// where the two 512 x 512 contractions of the table took 93.2 ms at 90 % of
// the FP64 matrix peak.  Choices on the way, same size: barriers that wait for
// the loads in flight (__syncthreads) and spilled registers 37.9 ms; bare LDS
// barriers, no spills, tables in LDS 39.6 with orders 2^21 elements apart and
// 27.9 with 9 cache lines more (see store_ld); the first vector loaded a whole
// tile ahead 24.8.  1024 threads with 128 registers 27.5; two blocks per CU of
// half the sites (32-byte reads) 60.
template <int NOPR, bool DERIV, int NSET, bool FOLD>
__global__ __launch_bounds__(kT) void k_site_sums(SumArgs a, int ntiles) {
  extern __shared__ double2 lds[];
  constexpr int kA = DERIV ? 2 : 1;  // jobs of the left vector
  constexpr int kArr = kA + 1;       // accumulators per operator: A, B, (A')
  const int tid0 = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6);
  // phase 1: 256 threads per vector, thread (site s, point j)
  const bool lefts = wave < 4;
  const int set0 = NSET == 1 ? blockIdx.y : 0;
  const int nblk = gridDim.x;
  // consecutive tiles go to blocks of one XCD (blocks are dealt round-robin),
  // so two tiles of one 128-byte line are read through the same L2
  const int b0 = blockIdx.x, q8 = nblk / 8;
  const int first = nblk % 8 == 0 ? (b0 & 7) * q8 + (b0 >> 3) : b0;

  double2 acc[NSET][NOPR][kArr];
#pragma unroll
  for (int h = 0; h < NSET; ++h)
#pragma unroll
    for (int o = 0; o < NOPR; ++o)
#pragma unroll
      for (int r = 0; r < kArr; ++r) acc[h][o][r] = make_double2(0.0, 0.0);

  // this thread's points of the tile: 8 of L (left threads) or 8 of every R;
  // points past M have weight 0 and sites past K are left out of the products
  double2 xv[NOPR][8];
  auto load1 = [&](double2(&x)[8], const double2 *v, int tile, int r) {
    int t = tid0;
    asm volatile("" : "+v"(t));
    const int j = (t >> 2) & 63;
    const double2 *p = v + min((long long)tile * kS + (t & 3), a.K - 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = p[(size_t)min(j + 64 * k + kP * r, a.M - 1) * a.ld];
  };
  // The next tile's first vector is loaded into nx behind the first set, a
  // second one into its own place once the last set has taken its points.
  double2 nx[8];
  auto load_first = [&](int tile) { load1(nx, lefts ? a.L : a.R[0], tile, 0); };
  auto load_second = [&](int tile) {
    if (NOPR == 2 && !lefts) load1(xv[NOPR - 1], a.R[NOPR - 1], tile, 0);
  };
  // The tables of the block's sets stay in LDS beside the spectra (FOLD: read
  // from global memory, five jobs leave no room).  From global memory their
  // loads would wait for the next tile's points, which are loaded before them.
  double2 *lt = lds + (kA + NOPR) * kS * kP, *lw = lt + kTw;
  if (!FOLD) {
    for (int i = tid0; i < kTw; i += kT) lt[i] = a.tw[i];
    for (int i = tid0; i < NSET * kP; i += kT) lw[i] = a.wt[i];
    load_first(first);
    load_second(first);
    __syncthreads();
  }
  for (int tile = first; tile < ntiles; tile += nblk) {
    if (!FOLD) {
#pragma unroll
      for (int k = 0; k < 8; ++k) xv[0][k] = nx[k];
    }
#pragma unroll
    for (int hh = 0; hh < NSET; ++hh) {
      const int h = set0 + hh;
      const bool self = NSET == 2 || h == 0 || 2 * h == a.H;
      const int njobs = kA + NOPR + (self ? 0 : 1);
      // indices are recomputed for every tile: kept in registers they would not
      // fit beside the points, so the compiler is not to take them out of the loop
      int tid = tid0;
      asm volatile("" : "+v"(tid));
      const int s = tid & 3;
      int j = (tid >> 2) & 63;
      const double2 *wt = FOLD ? a.wt + (size_t)h * kP * a.fold : lw + hh * kP;
      const double2 *tw = FOLD ? a.tw : lt;
      // ---- 1. weights and the first pass
      double2 t[8];
      powers(tw[j], t);
      auto put = [&](double2(&v)[8], int job) {
        __builtin_amdgcn_sched_barrier(0);
        radix8(v);
        double2 *z = lds + (job * kS + s) * kP + (j ^ (2 * s));
        z[0] = v[0];
#pragma unroll
        for (int k = 1; k < 8; ++k) z[64 * k] = cmul(v[k], t[k]);
        __builtin_amdgcn_sched_barrier(0);
      };
      // y (+)= weighted points x of fold r; kind 0: x, 1: conj x, 2: m conj x
      auto weigh = [&](double2(&y)[8], const double2(&x)[8], int r, int kind) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int m = j + 64 * k + kP * r;
          double2 c = cmul(kind == 0 ? x[k] : make_double2(x[k].x, -x[k].y), wt[m]);
          if (kind == 2) c = make_double2(m * c.x, m * c.y);
          y[k] = FOLD ? cadd(y[k], c) : c;
        }
      };
      auto job = [&](const double2(&x)[8], int index, int kind) {
        asm volatile("" : "+v"(j));
        double2 y[8];
        weigh(y, x, 0, kind);
        put(y, index);
      };
      if (FOLD) {
        // one load of a point serves conj L and m conj L
        auto fold = [&](double2(&y0)[8], double2(&y1)[8], const double2 *v0, int kind0, const double2 *v1, int kind1) {
          for (int r = 0; r < a.fold; ++r) {
            double2 x[8];
            load1(x, v0, tile, r);
            weigh(y0, x, r, kind0);
            if (!v1) continue;
            if (v1 != v0) load1(x, v1, tile, r);
            weigh(y1, x, r, kind1);
          }
        };
        double2 y0[8], y1[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) y0[k] = y1[k] = make_double2(0.0, 0.0);
        if (lefts) {
          fold(y0, y1, a.L, 1, DERIV ? a.L : nullptr, 2);
          put(y0, 0);
          if (DERIV) put(y1, 1);
          if (!self) {
#pragma unroll
            for (int k = 0; k < 8; ++k) y0[k] = make_double2(0.0, 0.0);
            fold(y0, y1, a.L, 0, nullptr, 0);
            put(y0, kA + NOPR);
          }
        } else {
          fold(y0, y1, a.R[0], 0, NOPR == 2 ? a.R[NOPR - 1] : nullptr, 0);
          put(y0, kA);
          if (NOPR == 2) put(y1, kA + 1);
        }
      } else if (lefts) {
        job(xv[0], 0, 1);
        if (DERIV) job(xv[0], 1, 2);
      } else {
#pragma unroll
        for (int o = 0; o < NOPR; ++o) job(xv[o], kA + o, 0);
      }
      if (!FOLD && tile + nblk < ntiles) {
        if (hh == 0) load_first(tile + nblk);
        if (hh == NSET - 1) load_second(tile + nblk);
      }
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();
      // ---- 2. the other two passes: job (q, site) = wave, wave + 8, ...
      const int total = njobs * kS;
      double2 t64[8];
      powers(tw[8 * (tid & 7)], t64);  // e^{-2 pi i j1 k2 / 64}
      for (int q = wave; q < total; q += 8) finish_fft(lds + q * kP, 2 * (q & 3), t64, tid & 63);
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();
      // ---- 3. products at frequency g = tid
      const int g = tid;
      const int mirror = h == 0 ? (kP - g) & (kP - 1) : kP - 1 - g;
#pragma unroll
      for (int st = 0; st < kS; ++st) {
        if ((long long)tile * kS + st >= a.K) break;
        const double2 al = lds[st * kP + g];
        double2 bl;  // conj of L's transform
        if (self) {
          bl = lds[st * kP + mirror];
        } else {
          bl = lds[((kA + NOPR) * kS + st) * kP + g];
          bl.y = -bl.y;
        }
        double2 dl;
        if (DERIV) dl = lds[(kS + st) * kP + g];
#pragma unroll
        for (int o = 0; o < NOPR; ++o) {
          const double2 b = lds[((kA + o) * kS + st) * kP + g];
          cfma(acc[hh][o][0], al, b);
          cfma(acc[hh][o][1], bl, b);
          if (DERIV) cfma(acc[hh][o][kArr - 1], dl, b);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      lds_barrier();
    }
  }
#pragma unroll
  for (int hh = 0; hh < NSET; ++hh)
#pragma unroll
    for (int o = 0; o < NOPR; ++o)
#pragma unroll
      for (int r = 0; r < kArr; ++r)
        a.partial[((size_t)blockIdx.x * (NOPR * kArr) + o * kArr + r) * ((size_t)kP * a.H) +
                  (size_t)a.H * tid0 + set0 + hh] = acc[hh][o][r];
}

// wt[h][m] = c_m e^{-2 pi i h m / F} (0 past M), tw[k] = e^{-2 pi i k / 512}
// (k < 64), tf[k] = e^{2 pi i k / F}.
__global__ void k_sum_tables(const double *__restrict__ coef, int M, int H, int fold, double2 *__restrict__ wt,
                             double2 *__restrict__ tw, double2 *__restrict__ tf) {
  const int F = kP * H, per = kP * fold;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < H * per; t += gridDim.x * blockDim.x) {
    const int h = t / per, m = t % per;
    double sn, cs;
    sincospi(-2.0 * ((h * m) % F) / F, &sn, &cs);
    wt[t] = m < M ? make_double2(coef[m] * cs, coef[m] * sn) : make_double2(0.0, 0.0);
  }
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < F; t += gridDim.x * blockDim.x) {
    double sn, cs;
    sincospi(2.0 * t / F, &sn, &cs);
    tf[t] = make_double2(cs, sn);
    if (t < kTw) {
      sincospi(-2.0 * t / kP, &sn, &cs);
      tw[t] = make_double2(cs, sn);
    }
  }
}

// spec[i] (+)= sum over blocks of partial[block][i], i < count, in a fixed
// order: 8 strided sums per element, then those in order.
__global__ __launch_bounds__(256) void k_sum_partials(const double2 *__restrict__ partial, int nblk, int count,
                                                      double2 *__restrict__ spec, int accumulate) {
  __shared__ double2 sh[8][32];
  const int e = threadIdx.x & 31, p = threadIdx.x >> 5;
  const int i = blockIdx.x * 32 + e;
  double2 v = make_double2(0.0, 0.0);
  if (i < count)
    for (int b = p; b < nblk; b += 8) v = cadd(v, partial[(size_t)b * count + i]);
  sh[p][e] = v;
  __syncthreads();
  if (p == 0 && i < count) {
    for (int u = 1; u < 8; ++u) v = cadd(v, sh[u][e]);
    spec[i] = accumulate ? cadd(spec[i], v) : v;
  }
}

// One wavefront per (array, q): seq[arr][q] = scale sum_f spec[arr][f] e^{2 pi i f q / F}.
__global__ __launch_bounds__(64) void k_sum_inverse(const double2 *__restrict__ spec, int F,
                                                    const double2 *__restrict__ tf, double scale,
                                                    double2 *__restrict__ seq) {
  const int q = blockIdx.x, l = threadIdx.x;
  const double2 *sp = spec + (size_t)blockIdx.y * F;
  double2 v = make_double2(0.0, 0.0);
  for (int f = l; f < F; f += 64) cfma(v, sp[f], tf[(int)(((long long)f * q) % F)]);
  for (int d = 32; d > 0; d >>= 1) {
    v.x += __shfl_down(v.x, d);
    v.y += __shfl_down(v.y, d);
  }
  if (l == 0) seq[(size_t)blockIdx.y * F + q] = make_double2(scale * v.x, scale * v.y);
}

// The energy sums from the sequences (per operator A, B and, for Bastin, A';
// B_q at index q mod F), one wavefront per energy: angles q theta_k =
// 2 pi (4k + 1) q / (4 nump), reduced exactly in integers.
template <bool BASTIN>
__global__ __launch_bounds__(64) void k_sum_energies(const double2 *__restrict__ seq, int F, int M, int nump,
                                                     double2 *__restrict__ out) {
  const int k = blockIdx.x, l = threadIdx.x, o = blockIdx.y;
  constexpr int kArr = BASTIN ? 3 : 2;
  const double2 *A = seq + (size_t)o * kArr * F, *B = A + F, *D = A + 2 * F;
  out += (size_t)o * 2 * nump;
  const int Q = 4 * nump;
  const double sgn = k < nump / 2 ? 1.0 : -1.0;
  double2 p = make_double2(0.0, 0.0), w = make_double2(0.0, 0.0);
  for (int q = l; q < 2 * M - 1; q += 64) {
    double sn, cs;
    const long long x = ((4LL * k + 1) * q) % Q;
    sincospi(2.0 * (double)x / Q, &sn, &cs);
    sn *= sgn;
    const double2 aq = A[q];
    double2 bp = make_double2(0.0, 0.0), bm = bp;  // B_q, B_-q
    if (q < M) bp = B[q];
    if (q > 0 && q < M) bm = B[F - q];
    p.x = fma(aq.x + bp.x + bm.x, cs, p.x);
    p.y = fma(aq.y + bp.y + bm.y, cs, p.y);
    if (BASTIN) {
      const double2 df = csub(bp, bm);  // (B_q - B_-q) i sin
      p.x = fma(-df.y, sn, p.x);
      p.y = fma(df.x, sn, p.y);
      const double2 d = D[q];
      w.x = fma(d.x, cs, w.x);
      w.y = fma(d.y, cs, w.y);
      // -(q/2) [A_q e^{iq phi} + B_q e^{iq phi} - B_-q e^{-iq phi}]
      const double hq = -0.5 * q;
      const double2 c = cadd(aq, df), si = cadd(aq, cadd(bp, bm));
      w.x = fma(hq, c.x * cs - si.y * sn, w.x);
      w.y = fma(hq, c.y * cs + si.x * sn, w.y);
    }
  }
  for (int d = 32; d > 0; d >>= 1) {
    p.x += __shfl_down(p.x, d);
    p.y += __shfl_down(p.y, d);
    w.x += __shfl_down(w.x, d);
    w.y += __shfl_down(w.y, d);
  }
  if (l == 0) {
    if (BASTIN) {
      out[k] = p;
      out[k + nump] = w;
    } else {
      out[k] = make_double2(0.5 * p.x, 0.0);
      out[k + nump] = make_double2(0.0, 0.0);
    }
  }
}

int sum_sets(int M) { return (2 * M - 1 + kP - 1) / kP; }
int sum_fold(int M) { return (M + kP - 1) / kP; }
int sum_arrays(int formula) { return formula == LQ_KUBO_BASTIN ? 3 : 2; }
// blocks along the sites: one per CU (a block holds most of a CU's LDS) when a
// block does every frequency set, fewer when the sets have blocks of their own
int sum_blocks(int H) { return H <= 2 ? 256 : std::max(8, 512 / H / 8 * 8); }

}  // namespace

bool kubosum_supported(int M) { return M >= 1 && M <= 4096; }

size_t kubosum_table_bytes(int M) {
  const size_t H = sum_sets(M);
  return sizeof(double2) * (H * kP * sum_fold(M) + kTw + kP * H);
}

size_t kubosum_spec_count(int M, int formula, int nopr) { return (size_t)sum_arrays(formula) * nopr * kP * sum_sets(M); }

size_t kubosum_partial_bytes(int M, int formula) {
  return sizeof(double2) * (size_t)sum_blocks(sum_sets(M)) * 2 * sum_arrays(formula) * kP * sum_sets(M);
}

double kubosum_flops(int M, int formula, int nopr, long long K) {
  const double F = (double)kP * sum_sets(M);
  const int left = formula == LQ_KUBO_BASTIN ? 2 : 1;
  return (double)K * ((left + nopr) * 5.0 * F * log2(F) + sum_arrays(formula) * nopr * 8.0 * F);
}

int launch_kubosum_tables(hipStream_t st, const double *coef, int M, double2 *tables) {
  const int H = sum_sets(M), fold = sum_fold(M);
  double2 *wt = tables, *tw = wt + (size_t)H * kP * fold, *tf = tw + kTw;
  hipLaunchKernelGGL(k_sum_tables, dim3(64), dim3(256), 0, st, coef, M, H, fold, wt, tw, tf);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

template <int NOPR, bool DERIV>
static int launch_site_sums(hipStream_t st, const SumArgs &a, int nblk, int ntiles) {
  constexpr int jobs = NOPR + (DERIV ? 2 : 1);
  const size_t lds =
      sizeof(double2) * (a.H > 2 ? (size_t)(jobs + 1) * kS * kP : (size_t)jobs * kS * kP + kTw + (size_t)a.H * kP);
  auto go = [&](auto kernel, int sets) -> int {
    LQ_HIP_CHECK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kernel, dim3(nblk, sets), dim3(kT), lds, st, a, ntiles);
    return LQ_OK;
  };
  if (a.H == 1)
    LQ_TRY(go(k_site_sums<NOPR, DERIV, 1, false>, 1));
  else if (a.H == 2)
    LQ_TRY(go(k_site_sums<NOPR, DERIV, 2, false>, 1));
  else
    LQ_TRY(go(k_site_sums<NOPR, DERIV, 1, true>, a.H));
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_kubosum(hipStream_t st, int formula, const double2 *L, const double2 *R, long long ld, long long K, int M,
                   int nopr, const double2 *tables, double2 *partial, double2 *spec, int accumulate) {
  if (!kubosum_supported(M) || K <= 0 || nopr <= 0) {
    set_error("launch_kubosum: bad sizes M=%d K=%lld nopr=%d", M, K, nopr);
    return LQ_ERR_ARG;
  }
  const int H = sum_sets(M), fold = sum_fold(M), arr = sum_arrays(formula);
  const long long tiles = (K + kS - 1) / kS;
  if (tiles > 0x7fffffffLL - 1024) {
    set_error("launch_kubosum: too many elements");
    return LQ_ERR_ARG;
  }
  const int nblk = (int)std::min<long long>(tiles, sum_blocks(H));
  SumArgs a{};
  a.L = L;
  a.K = K;
  a.ld = ld;
  a.M = M;
  a.H = H;
  a.fold = fold;
  a.wt = tables;
  a.tw = tables + (size_t)H * kP * fold;
  a.partial = partial;
  for (int o = 0; o < nopr; o += 2) {
    const int no = std::min(2, nopr - o);
    a.R[0] = R + (size_t)o * M * ld;
    a.R[1] = no == 2 ? R + (size_t)(o + 1) * M * ld : a.R[0];
    int rc;
    if (formula == LQ_KUBO_BASTIN)
      rc = no == 2 ? launch_site_sums<2, true>(st, a, nblk, (int)tiles) : launch_site_sums<1, true>(st, a, nblk, (int)tiles);
    else
      rc = no == 2 ? launch_site_sums<2, false>(st, a, nblk, (int)tiles)
                   : launch_site_sums<1, false>(st, a, nblk, (int)tiles);
    LQ_TRY(rc);
    const int count = no * arr * kP * H;
    hipLaunchKernelGGL(k_sum_partials, dim3((count + 31) / 32), dim3(256), 0, st, partial, nblk, count,
                       spec + (size_t)o * arr * kP * H, accumulate);
    LQ_HIP_CHECK(hipGetLastError());
  }
  return LQ_OK;
}

int kubosum_length(int M) { return kP * sum_sets(M); }

int launch_kubosum_sequences(hipStream_t st, int formula, const double2 *spec, const double2 *tables, int M, int nopr,
                             double scale, double2 *seq) {
  const int H = sum_sets(M), F = kP * H;
  const double2 *tf = tables + (size_t)H * kP * sum_fold(M) + kTw;
  hipLaunchKernelGGL(k_sum_inverse, dim3(F, sum_arrays(formula) * nopr), dim3(64), 0, st, spec, F, tf, scale / F, seq);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

int launch_kubo_energies(hipStream_t st, int formula, const double2 *seq, int M, int nopr, int nump, double2 *out) {
  const int F = kubosum_length(M);
  if (formula == LQ_KUBO_BASTIN)
    hipLaunchKernelGGL((k_sum_energies<true>), dim3(nump, nopr), dim3(64), 0, st, seq, F, M, nump, out);
  else
    hipLaunchKernelGGL((k_sum_energies<false>), dim3(nump, nopr), dim3(64), 0, st, seq, F, M, nump, out);
  LQ_HIP_CHECK(hipGetLastError());
  return LQ_OK;
}

}  // namespace lq
