// Parameter-space stochastic reconfiguration by MINRES, resident on the
// device: (S + shift I) dp = g with
//   S x = O^T (O x) / Ns - (Obar . x) Obar,   Obar = mean_s O,
//   g   = (1/Ns) sum_s (E_s - E_mean) O_s,
// S never formed.  The Lanczos / Givens recurrence of Paige and Saunders
// (the form of scipy.sparse.linalg.minres: convergence when
// |phibar| < rtol ||A|| ||x|| with the running estimate of ||A||) keeps all
// of its scalars in device memory; one-thread kernels update them, and a
// device flag set on convergence turns every later launch of the loop into
// an immediate return, so the host never waits inside the solve.
//
// The update is not determined by its inputs alone at the usual settings (heavy-tailed O,
// shift 1e-2): the Lanczos vectors lose their orthogonality, and another order of the sums
// gives an update that differs by per cents.  So every sum has one order, whatever the
// form: products and vector sums by one fma chain per thread of the blocks of
// mr_dot_partial / mr_gemv_rows, then trees; column sums over kRowChunks row chunks.
//
// Per iteration, up to kNarrowNp parameters, four launches:
//   mr_rows        inner = O v (256 threads a row), and, in workgroups of their own,
//                  Obar . v and the previous iteration's x update and convergence test;
//   mr_colsum_rows the row-chunk sums of O^T inner;
//   mr_form_y_narrow    the chunk sums added up, and y;
//   mr_finish      alfa, the orthogonalised y, ||y||, the Givens rotation (one workgroup).
// A launch costs 2 - 3 us whatever it does, so the count of launches bounds small and
// medium problems: a solve of 2900 samples and 2160 parameters, 100 iterations launched and
// a third of them made, takes 1.7 ms, of 516 and 480 1.4 ms (15 launches: 4.6 to 6.2 and 6.0;
// the same bits); an iteration that is made 30 us (rows 10.7, column sums 10.1, y 4.9, finish
// 4.5).  Above kNarrowNp the length-Np work takes the whole chip, in 15
// launches: one workgroup would walk 53 MB an iteration at 2.2 M parameters.
#include <hip/hip_runtime.h>

#include <cmath>

#include "kernels.h"

namespace vmcx {

namespace {

struct Neu2 {
  double s = 0.0, c = 0.0;
  __device__ __forceinline__ void add(double x) {
    const double t = s + x;
    c += (fabs(s) >= fabs(x)) ? (s - t) + x : (x - t) + s;
    s = t;
  }
};

constexpr int kRowChunks = 64;     // row chunks of the O^T w column sums
constexpr int kDotBlocks = 1024;   // first-stage blocks of a length-Np dot (one per 2048)
constexpr int kNarrowBlocks = 4;   // first-stage blocks that one workgroup of 1024 stands for
constexpr int64_t kNarrowNp = 2048 * kNarrowBlocks;

// scalar slots
enum {
  S_BETA = 0, S_OLDB, S_ALFA, S_CS, S_SN, S_DBAR, S_EPSLN, S_PHIBAR, S_ANORM2, S_OLDEPS,
  S_DELTA, S_GAMMA, S_PHI, S_DONE, S_ITN, S_MV, S_YNORM2, S_BETA2, S_BNORM2, S_INFO,
  S_EMEAN, S_EVAR, S_STOP, S_ZERO = 31, S_COUNT = 32
};

// row-chunk sums of O and of O^T w
__global__ void __launch_bounds__(256)
    mr_colsum_partial(int64_t Ns, int64_t Np, const void *O, int o_dtype, int64_t ldo,
                      int64_t rows, const double *__restrict__ w, double *partial,
                      double *partial2) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= Np) return;
  const int64_t r0 = (int64_t)blockIdx.y * rows;
  const int64_t r1 = (r0 + rows < Ns) ? r0 + rows : Ns;
  Neu2 a, b;
  for (int64_t s = r0; s < r1; ++s) {
    const double v = o_dtype == 0 ? ((const double *)O)[s * ldo + p]
                                  : (double)((const float *)O)[s * ldo + p];
    a.add(v);
    b.add(v * w[s]);
  }
  partial[(int64_t)blockIdx.y * Np + p] = a.s + a.c;
  partial2[(int64_t)blockIdx.y * Np + p] = b.s + b.c;
}

// a += the products of K rows of O with w, in order; the K loads in flight together
template <int K, typename T>
__device__ __forceinline__ void mr_add_rows(const T *O, int64_t ldo, const double *w, Neu2 &a) {
  T v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = O[k * ldo];
#pragma unroll
  for (int k = 0; k < K; ++k) {
#pragma clang fp contract(off)
    const double x = (double)v[k] * w[k];   // rounded: not fused with the sum
    a.add(x);
  }
}

// The row-chunk sums of O^T w of an iteration, over the same chunks in row order.  Bound by the
// latency of a thread's chain of Ns / kRowChunks loads: 2900 samples, 2160 parameters 22 us with
// one row at a time, 10 us with eight.
template <typename T>
__global__ void __launch_bounds__(256)
    mr_colsum_rows(int64_t Ns, int64_t Np, const T *__restrict__ O, int64_t ldo, int64_t rows,
                   const double *__restrict__ w, double *__restrict__ partial,
                   const double *skip) {
  if (skip[0] != 0.0) return;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= Np) return;
  int64_t s = (int64_t)blockIdx.y * rows;
  const int64_t r1 = (s + rows < Ns) ? s + rows : Ns;
  Neu2 a;
  for (; s + 8 <= r1; s += 8) mr_add_rows<8>(O + s * ldo + p, ldo, w + s, a);
  if (s + 4 <= r1) {
    mr_add_rows<4>(O + s * ldo + p, ldo, w + s, a);
    s += 4;
  }
  for (; s < r1; ++s) mr_add_rows<1>(O + s * ldo + p, ldo, w + s, a);
  partial[(int64_t)blockIdx.y * Np + p] = a.s + a.c;
}

__global__ void __launch_bounds__(256)
    mr_colsum_final(int64_t Np, const double *partial, double scale, double *out,
                    const double *skip) {
  if (skip[0] != 0.0) return;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= Np) return;
  Neu2 a;
  for (int r = 0; r < kRowChunks; ++r) a.add(partial[(int64_t)r * Np + p]);
  out[p] = (a.s + a.c) * scale;
}

// two-stage dot product a . b -> sc[slot]
__global__ void __launch_bounds__(256)
    mr_dot_partial(int64_t n, const double *a, const double *b, double *part,
                   const double *skip) {
  if (skip[0] != 0.0) return;
  __shared__ double sh[4];
  double acc = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    acc += a[i] * b[i];
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ void __launch_bounds__(1024)
    mr_dot_final(int nb, const double *part, const double *skip, double *sc, int slot) {
  if (skip[0] != 0.0) return;
  __shared__ double sh[16];
  double acc = 0.0;
  for (int i = threadIdx.x; i < nb; i += blockDim.x) acc += part[i];
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    Neu2 a;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k) a.add(sh[k]);
    sc[slot] = a.s + a.c;
  }
}

// E statistics and w = E - E_mean (one block)
__global__ void __launch_bounds__(1024)
    mr_energy(int64_t Ns, const double *E, double given_mean, int use_given, double *w,
              double *sc) {
  __shared__ double sh[2][16];
  __shared__ double mean_sh;
  Neu2 a, b;
  for (int64_t s = threadIdx.x; s < Ns; s += blockDim.x) {
    a.add(E[s]);
    b.add(E[s] * E[s]);
  }
  double v0 = a.s + a.c, v1 = b.s + b.c;
  for (int o = 32; o > 0; o >>= 1) {
    v0 += __shfl_down(v0, o, 64);
    v1 += __shfl_down(v1, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    sh[0][threadIdx.x >> 6] = v0;
    sh[1][threadIdx.x >> 6] = v1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    Neu2 x, y;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k) {
      x.add(sh[0][k]);
      y.add(sh[1][k]);
    }
    const double m = (x.s + x.c) / (double)Ns;
    sc[S_EMEAN] = m;
    sc[S_EVAR] = (y.s + y.c) / (double)Ns - m * m;
    mean_sh = use_given ? given_mean : m;
  }
  __syncthreads();
  const double em = mean_sh;
  for (int64_t s = threadIdx.x; s < Ns; s += blockDim.x) w[s] = E[s] - em;
}

__global__ void mr_zero(int64_t n, double *x) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

__global__ void mr_copy(int64_t n, const double *a, double *b) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

// beta1 = ||g||; trivial right-hand side ends the solve with x = 0
__global__ void mr_init(double *sc, int maxiter) {
  for (int k = 0; k < S_COUNT; ++k)
    if (k != S_EMEAN && k != S_EVAR && k != S_BNORM2) sc[k] = 0.0;
  const double bn = sqrt(sc[S_BNORM2]);
  sc[S_BETA] = bn;
  sc[S_CS] = -1.0;
  sc[S_PHIBAR] = bn;
  sc[S_INFO] = (double)maxiter;
  if (bn == 0.0) {
    sc[S_STOP] = 1.0;
    sc[S_DONE] = 1.0;
    sc[S_INFO] = 0.0;
  }
}

// the Givens rotation of the new Lanczos column, beta = ||y|| (one thread)
__device__ void mr_rotate_step(double alfa, double oldb, double beta, double *sc) {
  const double cs = sc[S_CS], sn = sc[S_SN], dbar = sc[S_DBAR], phibar = sc[S_PHIBAR];
  sc[S_OLDB] = oldb;
  sc[S_BETA] = beta;
  sc[S_OLDEPS] = sc[S_EPSLN];
  sc[S_DELTA] = fma(alfa, sn, cs * dbar);
  const double gbar = fma(sn, dbar, -(cs * alfa));
  sc[S_EPSLN] = sn * beta;
  sc[S_DBAR] = -cs * beta;
  double gamma = sqrt(fma(beta, beta, gbar * gbar));
  gamma = gamma > 1e-300 ? gamma : 1e-300;
  sc[S_GAMMA] = gamma;
  const double ncs = gbar / gamma, nsn = beta / gamma;
  sc[S_CS] = ncs;
  sc[S_SN] = nsn;
  sc[S_PHI] = ncs * phibar;
  sc[S_PHIBAR] = nsn * phibar;
  sc[S_ANORM2] += fma(beta, beta, fma(alfa, alfa, oldb * oldb));
}

// the convergence test after an update of x (one thread)
__device__ void mr_test(double rtol, double ynorm2, int flag, double *sc) {
  sc[S_ITN] += 1.0;
  const double rnorm = fabs(sc[S_PHIBAR]);
  if (rnorm < rtol * sqrt(sc[S_ANORM2]) * sqrt(ynorm2) || sc[S_BETA] == 0.0) {
    sc[flag] = 1.0;
    sc[S_INFO] = 0.0;
  }
}

// ------------------------------------------------------------ Np > kNarrowNp
// v[s] = sum_p O[s][p] x[p]
__global__ void __launch_bounds__(256)
    mr_gemv_rows(int64_t Np, const void *O, int o_dtype, int64_t ldo, const double *x,
                 double *v, const double *sc) {
  if (sc[S_DONE] != 0.0) return;
  __shared__ double sh[4];
  const int64_t s = blockIdx.x;
  double acc = 0.0;
  if (o_dtype == 0) {
    const double *row = (const double *)O + s * ldo;
    for (int64_t p = threadIdx.x; p < Np; p += blockDim.x) acc = fma(row[p], x[p], acc);
  } else {
    const float *row = (const float *)O + s * ldo;
    for (int64_t p = threadIdx.x; p < Np; p += blockDim.x) acc = fma((double)row[p], x[p], acc);
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) v[s] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// v = r2 / beta
__global__ void mr_scale_v(int64_t n, const double *r2, double *v, const double *sc) {
  if (sc[S_DONE] != 0.0) return;
  const double s = 1.0 / sc[S_BETA];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = s * r2[i];
}

// y = Sx - (Obar . v) Obar + shift v - (beta / oldb) r1   (last term after
// the first iteration)
__device__ __forceinline__ double mr_y(double sx, double m, double v, double r1, double shift,
                                       double mv, double c) {
  const double t = fma(shift, v, fma(-mv, m, sx));
  return c != 0.0 ? fma(-c, r1, t) : t;
}
__global__ void mr_form_y(int64_t n, const double *Sx, const double *m, const double *v,
                          const double *r1, double shift, double *y, const double *sc) {
  if (sc[S_DONE] != 0.0) return;
  const double c = sc[S_ITN] >= 1.0 ? sc[S_BETA] / sc[S_OLDB] : 0.0;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = mr_y(Sx[i], m[i], v[i], r1[i], shift, sc[S_MV], c);
}

// y -= (alfa / beta) r2
__global__ void mr_orth_y(int64_t n, const double *r2, double *y, const double *sc) {
  if (sc[S_DONE] != 0.0) return;
  const double c = sc[S_ALFA] / sc[S_BETA];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = fma(-c, r2[i], y[i]);
}

__global__ void mr_rotate(double *sc) {
  if (sc[S_DONE] != 0.0) return;
  mr_rotate_step(sc[S_ALFA], sc[S_BETA], sqrt(sc[S_BETA2]), sc);
}

// w = (v - oldeps w1 - delta w2) / gamma, x += phi w
struct MrStep {
  double oe, de, ig, ph;
};
__device__ __forceinline__ MrStep mr_step(const double *sc) {
  return {sc[S_OLDEPS], sc[S_DELTA], 1.0 / sc[S_GAMMA], sc[S_PHI]};
}
__device__ __forceinline__ double mr_w(const MrStep &c, double v, double w1, double w2) {
  return fma(-c.de, w2, fma(-c.oe, w1, v)) * c.ig;
}
__global__ void mr_update_x(int64_t n, const double *v, const double *w1, const double *w2,
                            double *w, double *x, const double *sc) {
  if (sc[S_DONE] != 0.0) return;
  const MrStep c = mr_step(sc);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const double wi = mr_w(c, v[i], w1[i], w2[i]);
    w[i] = wi;
    x[i] = fma(c.ph, wi, x[i]);
  }
}

__global__ void mr_check(double rtol, double *sc) {
  if (sc[S_DONE] != 0.0) return;
  mr_test(rtol, sc[S_YNORM2], S_DONE, sc);
}

// ------------------------------------------------------------ Np <= kNarrowNp
// The sum of a length-n dot's per-thread parts in a workgroup of 1024, which stands for the
// nb blocks of mr_dot_partial (thread t: thread t % 256 of block t / 256, elements from
// 256 (t / 256) + t % 256 = t in steps of 256 nb) and for mr_dot_final.  The same in every
// thread.
__device__ __forceinline__ double mr_total(double acc, int nb, double *sh) {
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  double p[kNarrowBlocks];
#pragma unroll
  for (int b = 0; b < kNarrowBlocks; ++b)
    p[b] = b < nb ? (sh[4 * b] + sh[4 * b + 1]) + (sh[4 * b + 2] + sh[4 * b + 3]) : 0.0;
  Neu2 a;
  a.add((p[0] + p[2]) + (p[1] + p[3]));
  return a.s + a.c;
}

struct MrVecs {
  const double *r1, *r2, *m;   // r2: beta v of this iteration, r1: oldb v of the last
  const double *w1, *w2;       // the last iteration's update: w <- (v, w1, w2), x += phi w
  double *w, *x;
  int first;                   // no last iteration
};

// the x update of an iteration, with v = r1 / oldb, and its convergence test into sc[flag]
__device__ void mr_narrow_update(int n, int nb, const MrVecs &q, double rtol, int flag,
                                 double *sc, double *sh) {
  const MrStep c = mr_step(sc);
  const double s = 1.0 / sc[S_OLDB];
  double a = 0.0;
  if ((int)threadIdx.x < 256 * nb)
    for (int i = threadIdx.x; i < n; i += 256 * nb) {
      const double wi = mr_w(c, s * q.r1[i], q.w1[i], q.w2[i]);
      q.w[i] = wi;
      const double xi = fma(c.ph, wi, q.x[i]);
      q.x[i] = xi;
      a = fma(xi, xi, a);
    }
  a = mr_total(a, nb, sh);
  if (threadIdx.x == 0) mr_test(rtol, a, flag, sc);
}

// inner = O v, four rows a workgroup; the first two workgroups: Obar . v and the last x
// update.  That update's test sets S_STOP, which this launch does not read: S_DONE, which it
// does, follows in mr_finish (waves of a workgroup that read a flag while it is set would
// disagree on the way to their barrier).
__global__ void __launch_bounds__(1024)
    mr_rows(int64_t Ns, int n, int nb, const void *O, int o_dtype, int64_t ldo, MrVecs q,
            double rtol, double *inner, double *sc) {
  if (sc[S_DONE] != 0.0) return;
  __shared__ double sh[16];
  const int tid = threadIdx.x;
  const double is = 1.0 / sc[S_BETA];
  if (blockIdx.x == 1) {
    if (!q.first) mr_narrow_update(n, nb, q, rtol, S_STOP, sc, sh);
    return;
  }
  double acc = 0.0;
  if (blockIdx.x == 0) {
    if (tid < 256 * nb)
      for (int i = tid; i < n; i += 256 * nb) acc = fma(q.m[i], is * q.r2[i], acc);
    acc = mr_total(acc, nb, sh);
    if (tid == 0) sc[S_MV] = acc;
    return;
  }
  const int64_t s = 4 * ((int64_t)blockIdx.x - 2) + (tid >> 8);
  if (s < Ns) {
    if (o_dtype == 0) {
      const double *row = (const double *)O + s * ldo;
#pragma unroll 4
      for (int p = tid & 255; p < n; p += 256) acc = fma(row[p], is * q.r2[p], acc);
    } else {
      const float *row = (const float *)O + s * ldo;
#pragma unroll 4
      for (int p = tid & 255; p < n; p += 256) acc = fma((double)row[p], is * q.r2[p], acc);
    }
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if ((tid & 63) == 0) sh[tid >> 6] = acc;
  __syncthreads();
  const int b = tid >> 6;
  if ((tid & 255) == 0 && s < Ns) inner[s] = (sh[b] + sh[b + 1]) + (sh[b + 2] + sh[b + 3]);
}

// mr_colsum_final and mr_form_y
__global__ void __launch_bounds__(64)
    mr_form_y_narrow(int n, const double *__restrict__ partial, double scale,
                     const double *__restrict__ m, const double *__restrict__ r1,
                     const double *__restrict__ r2, double shift, double *y, const double *sc) {
  if (sc[S_STOP] != 0.0) return;
  const int p = blockIdx.x * 64 + threadIdx.x;
  if (p >= n) return;
  Neu2 a;
#pragma unroll 16
  for (int r = 0; r < kRowChunks; ++r) a.add(partial[(int64_t)r * n + p]);
  const double c = sc[S_ITN] >= 1.0 ? sc[S_BETA] / sc[S_OLDB] : 0.0;
  y[p] = mr_y((a.s + a.c) * scale, m[p], r2[p] * (1.0 / sc[S_BETA]), r1[p], shift, sc[S_MV], c);
}

// alfa = v . y, y -= (alfa / beta) r2, ||y|| and the Givens rotation (one workgroup: a vector
// of this length is a few us for one CU, as is another launch)
__global__ void __launch_bounds__(1024)
    mr_finish(int n, int nb, const double *__restrict__ r2, double *y, double *sc) {
  if (sc[S_STOP] != 0.0) {
    if (threadIdx.x == 0) sc[S_DONE] = 1.0;
    return;
  }
  __shared__ double sh[2][16];
  const int tid = threadIdx.x, step = 256 * nb;
  const bool on = tid < step;
  const double beta = sc[S_BETA], is = 1.0 / beta;
  double a = 0.0;
  if (on)
    for (int i = tid; i < n; i += step) a = fma(is * r2[i], y[i], a);
  const double alfa = mr_total(a, nb, sh[0]), c = alfa / beta;
  a = 0.0;
  if (on)
    for (int i = tid; i < n; i += step) {
      const double yi = fma(-c, r2[i], y[i]);
      y[i] = yi;
      a = fma(yi, yi, a);
    }
  a = mr_total(a, nb, sh[1]);
  if (tid != 0) return;
  sc[S_ALFA] = alfa;
  mr_rotate_step(alfa, beta, sqrt(a), sc);
}

// the x update of the last iteration
__global__ void __launch_bounds__(1024)
    mr_last_update(int n, int nb, MrVecs q, double rtol, double *sc) {
  if (sc[S_DONE] != 0.0) return;
  __shared__ double sh[16];
  mr_narrow_update(n, nb, q, rtol, S_STOP, sc, sh);
}

// stats <- [mean E, var E, |phibar| (residual estimate), ||g||, iterations]
__global__ void mr_stats(const double *sc, double *stats, int32_t *info) {
  if (stats) {
    stats[0] = sc[S_EMEAN];
    stats[1] = sc[S_EVAR];
    stats[2] = fabs(sc[S_PHIBAR]);
    stats[3] = sqrt(sc[S_BNORM2]);
    stats[4] = sc[S_ITN];
  }
  if (info) info[0] = (int32_t)sc[S_INFO];
}

inline size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

struct MrLayout {
  size_t vec[6], m, g, w, inner, partial, dotp, sc, total;
};

MrLayout mr_layout(int64_t Ns, int64_t Np) {
  MrLayout L{};
  size_t off = 0;
  auto take = [&](size_t b) {
    const size_t o = off;
    off += al256(b);
    return o;
  };
  for (auto &v : L.vec) v = take((size_t)Np * 8);
  L.m = take((size_t)Np * 8);
  L.g = take((size_t)Np * 8);
  L.w = take((size_t)Ns * 8);
  L.inner = take((size_t)Ns * 8);
  L.partial = take((size_t)2 * kRowChunks * Np * 8);
  L.dotp = take((size_t)kDotBlocks * 8);
  L.sc = take((size_t)S_COUNT * 8);
  L.total = off;
  return L;
}

}  // namespace

int64_t sr_minres_workspace_bytes(int64_t Ns, int64_t Np) {
  if (Ns <= 0 || Np <= 0) return -1;
  return (int64_t)mr_layout(Ns, Np).total;
}

int sr_minres(int64_t Ns, int64_t Np, const void *O, int o_dtype, int64_t ldo, const double *E,
              double energy_mean, double diag_shift, double rtol, int maxiter, void *ws,
              int64_t ws_bytes, double *dp, double *stats, int32_t *info, hipStream_t st) {
  VMCX_CHECK_ARG(Ns >= 1 && Np >= 1, "Ns and Np must be positive");
  VMCX_CHECK_ARG(ldo >= Np, "ldo < Np");
  VMCX_CHECK_ARG(o_dtype == 0 || o_dtype == 1, "o_dtype must be 0 (f64) or 1 (f32)");
  VMCX_CHECK_ARG(maxiter >= 0, "maxiter must be >= 0");
  VMCX_CHECK_ARG(rtol >= 0.0, "rtol must be >= 0");
  VMCX_CHECK_ARG(O && E && dp && ws, "null pointer argument");
  const MrLayout L = mr_layout(Ns, Np);
  VMCX_CHECK_ARG(ws_bytes >= (int64_t)L.total, "workspace too small");
  char *w = (char *)ws;
  double *vecs[6];
  for (int k = 0; k < 6; ++k) vecs[k] = (double *)(w + L.vec[k]);
  double *m = (double *)(w + L.m), *g = (double *)(w + L.g), *wE = (double *)(w + L.w);
  double *inner = (double *)(w + L.inner), *partial = (double *)(w + L.partial);
  double *partial2 = partial + (int64_t)kRowChunks * Np;
  double *dotp = (double *)(w + L.dotp), *sc = (double *)(w + L.sc);
  double *x = dp;
  const unsigned gn = (unsigned)((Np + 255) / 256);
  const int64_t rows = (Ns + kRowChunks - 1) / kRowChunks;
  const int nb = (int)((Np + 2047) / 2048 < kDotBlocks ? (Np + 2047) / 2048 : kDotBlocks);
  const int nbd = nb > 0 ? nb : 1;
  // launches outside the loop take the flag that stays zero, those inside the
  // convergence flag
  const double *always = sc + S_ZERO, *done = sc + S_DONE;
  auto dot = [&](const double *a, const double *b, int slot, const double *skip) {
    hipLaunchKernelGGL(mr_dot_partial, dim3(nbd), dim3(256), 0, st, Np, a, b, dotp, skip);
    hipLaunchKernelGGL(mr_dot_final, dim3(1), dim3(1024), 0, st, nbd, dotp, skip, sc, slot);
  };
  hipLaunchKernelGGL(mr_zero, dim3(1), dim3(S_COUNT), 0, st, (int64_t)S_COUNT, sc);
  VMCX_LAUNCHED();
  // E statistics, w = E - E_mean; Obar and g from one read of O
  const int use_given = std::isfinite(energy_mean) ? 1 : 0;
  hipLaunchKernelGGL(mr_energy, dim3(1), dim3(1024), 0, st, Ns, E, energy_mean, use_given, wE,
                     sc);
  hipLaunchKernelGGL(mr_colsum_partial, dim3(gn, kRowChunks), dim3(256), 0, st, Ns, Np, O,
                     o_dtype, ldo, rows, (const double *)wE, partial, partial2);
  hipLaunchKernelGGL(mr_colsum_final, dim3(gn), dim3(256), 0, st, Np, partial,
                     1.0 / (double)Ns, m, always);
  hipLaunchKernelGGL(mr_colsum_final, dim3(gn), dim3(256), 0, st, Np, partial2,
                     1.0 / (double)Ns, g, always);
  VMCX_LAUNCHED();
  dot(g, g, S_BNORM2, always);
  if (maxiter == 0)  // the energy gradient only
    hipLaunchKernelGGL(mr_copy, dim3(gn), dim3(256), 0, st, Np, g, x);
  else
    hipLaunchKernelGGL(mr_zero, dim3(gn), dim3(256), 0, st, Np, x);
  hipLaunchKernelGGL(mr_init, dim3(1), dim3(1), 0, st, sc, maxiter);
  // Lanczos vectors: r1, r2, y rotate through vecs[0..2]; w1, w2, w through vecs[3..5]
  double *r1 = vecs[0], *r2 = vecs[1], *y = vecs[2];
  double *w1 = vecs[3], *w2 = vecs[4], *wn = vecs[5];
  hipLaunchKernelGGL(mr_copy, dim3(gn), dim3(256), 0, st, Np, g, r1);
  hipLaunchKernelGGL(mr_copy, dim3(gn), dim3(256), 0, st, Np, g, r2);
  hipLaunchKernelGGL(mr_zero, dim3(gn), dim3(256), 0, st, Np, w1);
  hipLaunchKernelGGL(mr_zero, dim3(gn), dim3(256), 0, st, Np, w2);
  hipLaunchKernelGGL(mr_zero, dim3(gn), dim3(256), 0, st, Np, wn);
  VMCX_LAUNCHED();
  // partial <- row-chunk sums of O^T inner
  auto colsum = [&](const double *skip) {
    const dim3 grid(gn, kRowChunks), block(256);
    if (o_dtype == 0)
      hipLaunchKernelGGL(mr_colsum_rows<double>, grid, block, 0, st, Ns, Np, (const double *)O,
                         ldo, rows, inner, partial, skip);
    else
      hipLaunchKernelGGL(mr_colsum_rows<float>, grid, block, 0, st, Ns, Np, (const float *)O, ldo,
                         rows, inner, partial, skip);
  };
  if (Np <= kNarrowNp) {
    const int n = (int)Np;
    MrVecs q{};
    q.m = m;
    q.x = x;
    for (int it = 0; it < maxiter; ++it) {
      q.r1 = r1;
      q.r2 = r2;
      q.first = it == 0;
      hipLaunchKernelGGL(mr_rows, dim3((unsigned)((Ns + 3) / 4 + 2)), dim3(1024), 0, st, Ns, n,
                         nbd, O, o_dtype, ldo, q, rtol, inner, sc);
      colsum(sc + S_STOP);
      hipLaunchKernelGGL(mr_form_y_narrow, dim3((unsigned)((Np + 63) / 64)), dim3(64), 0, st, n,
                         partial, 1.0 / (double)Ns, m, r1, r2, diag_shift, y, sc);
      hipLaunchKernelGGL(mr_finish, dim3(1), dim3(1024), 0, st, n, nbd, r2, y, sc);
      VMCX_LAUNCHED();
      // r1 <- r2 <- y; the x update of this iteration (with its v = r2 / beta, then r1 /
      // oldb) runs in the next one's first launch: w1 <- w2 <- w (buffers rotate on the
      // host; once the device flag is set nothing reads them again)
      double *t = r1;
      r1 = r2;
      r2 = y;
      y = t;
      q.w1 = w1;
      q.w2 = w2;
      q.w = wn;
      t = w1;
      w1 = w2;
      w2 = wn;
      wn = t;
    }
    if (maxiter > 0) {
      q.r1 = r1;
      q.r2 = r2;
      hipLaunchKernelGGL(mr_last_update, dim3(1), dim3(1024), 0, st, n, nbd, q, rtol, sc);
    }
  } else {
    // v and S v: the second set of chunk sums is free after Obar and g
    double *v = partial2, *Sx = partial2 + Np;
    for (int it = 0; it < maxiter; ++it) {
      hipLaunchKernelGGL(mr_scale_v, dim3(gn), dim3(256), 0, st, Np, r2, v, sc);
      // S v without S: O v, then O^T (O v) / Ns
      hipLaunchKernelGGL(mr_gemv_rows, dim3((unsigned)Ns), dim3(256), 0, st, Np, O, o_dtype, ldo,
                         v, inner, sc);
      colsum(done);
      hipLaunchKernelGGL(mr_colsum_final, dim3(gn), dim3(256), 0, st, Np, partial,
                         1.0 / (double)Ns, Sx, done);
      dot(m, v, S_MV, done);
      hipLaunchKernelGGL(mr_form_y, dim3(gn), dim3(256), 0, st, Np, Sx, m, v, r1, diag_shift, y,
                         sc);
      dot(v, y, S_ALFA, done);
      hipLaunchKernelGGL(mr_orth_y, dim3(gn), dim3(256), 0, st, Np, r2, y, sc);
      dot(y, y, S_BETA2, done);
      hipLaunchKernelGGL(mr_rotate, dim3(1), dim3(1), 0, st, sc);
      hipLaunchKernelGGL(mr_update_x, dim3(gn), dim3(256), 0, st, Np, v, w1, w2, wn, x, sc);
      dot(x, x, S_YNORM2, done);
      hipLaunchKernelGGL(mr_check, dim3(1), dim3(1), 0, st, rtol, sc);
      VMCX_LAUNCHED();
      // r1 <- r2 <- y ; w1 <- w2 <- w (buffers rotate on the host; once the
      // device flag is set nothing reads them again)
      double *t = r1;
      r1 = r2;
      r2 = y;
      y = t;
      t = w1;
      w1 = w2;
      w2 = wn;
      wn = t;
    }
  }
  hipLaunchKernelGGL(mr_stats, dim3(1), dim3(1), 0, st, sc, stats, info);
  VMCX_LAUNCHED();
  return 0;
}

}  // namespace vmcx
