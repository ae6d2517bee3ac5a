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
// Per iteration three launches (four when Np > 8192):
//   mr_apply      inner = O v and the row-chunk sums of O^T inner from ONE read of O
//                 (a workgroup keeps its rows and its sums in registers; Np > 8192:
//                 mr_gemv_rows, then mr_colsum_partial, two reads), and, in workgroups
//                 of their own, Obar . v and the previous iteration's x update and
//                 convergence test;
//   mr_form_y     the chunk sums added up, y, and v . y per block;
//   mr_finish     alfa, the orthogonalised y, ||y||, the Givens rotation.
// A launch of this size costs 2 - 3 us whatever it does, so the count of launches bounds
// small and medium problems: at Ns = 2900, Np = 2160 an iteration takes 17 us (measured);
// 15 launches and two reads of O took 45 to 67.
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
constexpr int kApplyChunks = 2 * kRowChunks;  // row chunks of mr_apply (one workgroup each):
                                              // as many sums as the two kept before
constexpr int64_t kApplyNp = 8192; // widest row of mr_apply (8 columns a thread)
constexpr int kDotBlocks = 1024;   // first-stage blocks of a length-Np dot

// scalar slots
enum {
  S_BETA = 0, S_OLDB, S_ALFA, S_CS, S_SN, S_DBAR, S_EPSLN, S_PHIBAR, S_ANORM2, S_OLDEPS,
  S_DELTA, S_GAMMA, S_PHI, S_DONE, S_ITN, S_MV, S_YNORM2, S_BETA2, S_BNORM2, S_INFO,
  S_EMEAN, S_EVAR, S_ZERO = 31, S_COUNT = 32
};

__global__ void __launch_bounds__(256)
    mr_colsum_partial(int64_t Ns, int64_t Np, const void *O, int o_dtype, int64_t ldo,
                      int64_t rows, const double *__restrict__ w, const double *__restrict__ w2,
                      double *partial, double *partial2, const double *skip) {
  if (skip[0] != 0.0) return;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= Np) return;
  const int64_t r0 = (int64_t)blockIdx.y * rows;
  const int64_t r1 = (r0 + rows < Ns) ? r0 + rows : Ns;
  Neu2 a, b;
  for (int64_t s = r0; s < r1; ++s) {
    const double v = o_dtype == 0 ? ((const double *)O)[s * ldo + p]
                                  : (double)((const float *)O)[s * ldo + p];
    a.add(w ? v * w[s] : v);
    if (w2) b.add(v * w2[s]);
  }
  partial[(int64_t)blockIdx.y * Np + p] = a.s + a.c;
  if (w2) partial2[(int64_t)blockIdx.y * Np + p] = b.s + b.c;
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
    sc[S_DONE] = 1.0;
    sc[S_INFO] = 0.0;
  }
}

// block-wide sums of NV values (512 or 1024 threads), the same in every thread
template <int NT, int NV>
__device__ __forceinline__ void block_sums(double (&v)[NV], double (*sh)[NT / 64]) {
#pragma unroll
  for (int i = 0; i < NV; ++i)
    for (int o = 32; o > 0; o >>= 1) v[i] += __shfl_xor(v[i], o, 64);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < NV; ++i) sh[i][threadIdx.x >> 6] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < NT / 64; ++k) t += sh[i][k];
    v[i] = t;
  }
}

struct MrVecs {
  const double *r1, *r2, *m;   // r2: beta v of this iteration, r1: oldb v of the last
  const double *w1, *w2;       // the last iteration's update: w <- (v, w1, w2), x += phi w
  double *w, *x;
  int first;                   // no last iteration
};

// Obar . v (one workgroup)
template <int NT>
__device__ void mr_mean_dot(int64_t n, const MrVecs &q, double *sc, double (*sh)[NT / 64]) {
  const double s = 1.0 / sc[S_BETA];
  double a[1] = {0.0};
  for (int64_t i = threadIdx.x; i < n; i += NT) a[0] += q.m[i] * (s * q.r2[i]);
  block_sums<NT, 1>(a, sh);
  if (threadIdx.x == 0) sc[S_MV] = a[0];
}

// w = (v - oldeps w1 - delta w2) / gamma, x += phi w with the last iteration's v, and its
// convergence test (one workgroup)
template <int NT>
__device__ void mr_update_x(int64_t n, const MrVecs &q, double rtol, double *sc,
                            double (*sh)[NT / 64]) {
  const double oe = sc[S_OLDEPS], de = sc[S_DELTA], ig = 1.0 / sc[S_GAMMA], ph = sc[S_PHI];
  const double s = 1.0 / sc[S_OLDB];
  double a[1] = {0.0};
  for (int64_t i = threadIdx.x; i < n; i += NT) {
    const double wi = (s * q.r1[i] - oe * q.w1[i] - de * q.w2[i]) * ig;
    q.w[i] = wi;
    const double xi = q.x[i] + ph * wi;
    q.x[i] = xi;
    a[0] += xi * xi;
  }
  block_sums<NT, 1>(a, sh);
  if (threadIdx.x == 0) {
    sc[S_YNORM2] = a[0];
    sc[S_ITN] += 1.0;
    const double rnorm = fabs(sc[S_PHIBAR]);
    if (rnorm < rtol * sqrt(sc[S_ANORM2]) * sqrt(a[0]) || sc[S_BETA] == 0.0) {
      sc[S_DONE] = 1.0;
      sc[S_INFO] = 0.0;
    }
  }
}

// inner = O v and the sums of O^T inner over this workgroup's rows from one read of O:
// thread t holds the columns t, t + 1024, ... (E of them) of RB rows, of v and of the
// compensated sums in registers; the next RB rows are loaded while the products of these
// are summed over the workgroup (RB = 2 while that fits 128 registers: half the barriers).
// Workgroups beyond the row chunks: Obar . v and the last x update (a flag that the latter
// sets while the others run is seen by the next launch, which then ignores what they
// wrote).
template <int E, int RB, typename T>
__global__ void __launch_bounds__(1024)
    mr_apply(int64_t Ns, int64_t Np, const T *__restrict__ O, int64_t ldo, int64_t rows,
             int chunks, MrVecs q, double rtol, double *__restrict__ partial, double *sc) {
  if (sc[S_DONE] != 0.0) return;
  __shared__ double sh[2][RB][16];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x >= chunks) {
    if ((int)blockIdx.x == chunks)
      mr_mean_dot<1024>(Np, q, sc, sh[0]);
    else if (!q.first)
      mr_update_x<1024>(Np, q, rtol, sc, sh[0]);
    return;
  }
  const int64_t r0 = blockIdx.x * rows, r1 = (r0 + rows < Ns) ? r0 + rows : Ns;
  const double s = 1.0 / sc[S_BETA];
  double v[E];
  Neu2 acc[E];
  T cur[RB][E], nxt[RB][E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int64_t p = tid + 1024 * (int64_t)e;
    v[e] = p < Np ? s * q.r2[p] : 0.0;
  }
  auto load = [&](int64_t r, T (&d)[RB][E]) {
#pragma unroll
    for (int k = 0; k < RB; ++k)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int64_t p = tid + 1024 * (int64_t)e;
        d[k][e] = (r + k < r1 && p < Np) ? O[(r + k) * ldo + p] : (T)0;
      }
  };
  load(r0, cur);
  int buf = 0;
  for (int64_t r = r0; r < r1; r += RB, buf ^= 1) {
    load(r + RB, nxt);
    double d[RB];
#pragma unroll
    for (int k = 0; k < RB; ++k) {
      d[k] = 0.0;
#pragma unroll
      for (int e = 0; e < E; ++e) d[k] += (double)cur[k][e] * v[e];
    }
    block_sums<1024, RB>(d, sh[buf]);
#pragma unroll
    for (int k = 0; k < RB; ++k)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        acc[e].add((double)cur[k][e] * d[k]);
        cur[k][e] = nxt[k][e];
      }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int64_t p = tid + 1024 * (int64_t)e;
    if (p < Np) partial[(int64_t)blockIdx.x * Np + p] = acc[e].s + acc[e].c;
  }
}

// O v by rows when a row does not fit a workgroup's registers; the last two workgroups as
// in mr_apply
__global__ void __launch_bounds__(512)
    mr_gemv_rows(int64_t Ns, int64_t Np, const void *O, int o_dtype, int64_t ldo, MrVecs q,
                 double rtol, double *inner, double *sc) {
  if (sc[S_DONE] != 0.0) return;
  __shared__ double sh[1][8];
  const int64_t s = blockIdx.x;
  if (s >= Ns) {
    if (s == Ns)
      mr_mean_dot<512>(Np, q, sc, sh);
    else if (!q.first)
      mr_update_x<512>(Np, q, rtol, sc, sh);
    return;
  }
  const double is = 1.0 / sc[S_BETA];
  double acc[1] = {0.0};
  if (o_dtype == 0) {
    const double *row = (const double *)O + s * ldo;
    for (int64_t p = threadIdx.x; p < Np; p += 512) acc[0] += row[p] * (is * q.r2[p]);
  } else {
    const float *row = (const float *)O + s * ldo;
    for (int64_t p = threadIdx.x; p < Np; p += 512) acc[0] += (double)row[p] * (is * q.r2[p]);
  }
  block_sums<512, 1>(acc, sh);
  if (threadIdx.x == 0) inner[s] = acc[0];
}

// y = S v - (Obar . v) Obar + shift v - (beta / oldb) r1 (last term after the first
// iteration) from the chunk sums of O^T (O v), and the block's part of v . y: 16 columns
// per block, 64 threads over the chunks of each
__global__ void __launch_bounds__(1024)
    mr_form_y(int64_t n, int chunks, const double *__restrict__ partial, double scale,
              const double *__restrict__ m, const double *__restrict__ r1,
              const double *__restrict__ r2, double shift, double *y, double *part,
              const double *sc) {
  if (sc[S_DONE] != 0.0) return;
  __shared__ double sh[64][17];
  const int col = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int64_t p = (int64_t)blockIdx.x * 16 + col;
  Neu2 a;
  if (p < n)
    for (int c = g; c < chunks; c += 64) a.add(partial[(int64_t)c * n + p]);
  sh[g][col] = a.s + a.c;
  __syncthreads();
  if (g < 4) {
    Neu2 b;
    for (int k = 0; k < 16; ++k) b.add(sh[g * 16 + k][col]);
    // the four partial sums of a column sit in lanes 16 apart of the first wave
    Neu2 t;
    const double own = b.s + b.c;
    for (int k = 0; k < 4; ++k) t.add(__shfl(own, k * 16 + col, 64));
    double vy = 0.0;
    if (g == 0 && p < n) {
      const double v = r2[p] * (1.0 / sc[S_BETA]);
      const double c = sc[S_ITN] >= 1.0 ? sc[S_BETA] / sc[S_OLDB] : 0.0;
      double yi = (t.s + t.c) * scale - sc[S_MV] * m[p] + shift * v;
      if (c != 0.0) yi -= c * r1[p];
      y[p] = yi;
      vy = v * yi;
    }
    for (int o = 8; o > 0; o >>= 1) vy += __shfl_xor(vy, o, 64);
    if (threadIdx.x == 0) part[blockIdx.x] = vy;
  }
}

// alfa = v . y, y -= (alfa / beta) r2, and the Givens rotation of the new Lanczos column
// (one workgroup: a length-Np vector is a few us for one CU, as is another launch)
__global__ void __launch_bounds__(1024)
    mr_finish(int64_t n, int64_t nb, const double *__restrict__ part,
              const double *__restrict__ r2, double *y, double *sc) {
  if (sc[S_DONE] != 0.0) return;
  __shared__ double sh[2][1][16];
  double a[1] = {0.0};
  for (int64_t i = threadIdx.x; i < nb; i += 1024) a[0] += part[i];
  block_sums<1024, 1>(a, sh[0]);
  const double alfa = a[0], oldb = sc[S_BETA], c = alfa / oldb;
  a[0] = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    const double yi = y[i] - c * r2[i];
    y[i] = yi;
    a[0] += yi * yi;
  }
  block_sums<1024, 1>(a, sh[1]);
  if (threadIdx.x != 0) return;
  const double beta = sqrt(a[0]);
  const double cs = sc[S_CS], sn = sc[S_SN], dbar = sc[S_DBAR];
  sc[S_ALFA] = alfa;
  sc[S_OLDB] = oldb;
  sc[S_BETA] = beta;
  sc[S_OLDEPS] = sc[S_EPSLN];
  sc[S_DELTA] = cs * dbar + sn * alfa;
  const double gbar = sn * dbar - cs * alfa;
  sc[S_EPSLN] = sn * beta;
  sc[S_DBAR] = -cs * beta;
  double gamma = sqrt(gbar * gbar + beta * beta);
  gamma = gamma > 1e-300 ? gamma : 1e-300;
  sc[S_GAMMA] = gamma;
  const double ncs = gbar / gamma, nsn = beta / gamma;
  sc[S_CS] = ncs;
  sc[S_SN] = nsn;
  sc[S_PHI] = ncs * sc[S_PHIBAR];
  sc[S_PHIBAR] = nsn * sc[S_PHIBAR];
  sc[S_ANORM2] += alfa * alfa + oldb * oldb + beta * beta;
}

// the x update of the last iteration
__global__ void __launch_bounds__(512) mr_last_update(int64_t n, MrVecs q, double rtol,
                                                      double *sc) {
  if (sc[S_DONE] != 0.0) return;
  __shared__ double sh[1][8];
  mr_update_x<512>(n, q, rtol, sc, sh);
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
  const size_t yblocks = (size_t)(Np + 15) / 16;
  L.dotp = take((yblocks > kDotBlocks ? yblocks : kDotBlocks) * 8);
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
                     o_dtype, ldo, rows, (const double *)nullptr, (const double *)wE, partial,
                     partial2, always);
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
  // rows of a chunk: even (taken in pairs), all chunks in use
  const int64_t arows = ((Ns + kApplyChunks - 1) / kApplyChunks + 1) & ~(int64_t)1;
  const bool fused = Np <= kApplyNp;
  const int chunks = fused ? (int)((Ns + arows - 1) / arows) : kRowChunks;
  const unsigned yb = (unsigned)((Np + 15) / 16);
  auto apply = [&](const MrVecs &q) {
    const dim3 grid((unsigned)chunks + 2), block(1024);
#define MR_APPLY(E, RB)                                                                         \
  do {                                                                                          \
    if (o_dtype == 0)                                                                           \
      hipLaunchKernelGGL((mr_apply<E, RB, double>), grid, block, 0, st, Ns, Np,                 \
                         (const double *)O, ldo, arows, chunks, q, rtol, partial, sc);          \
    else                                                                                        \
      hipLaunchKernelGGL((mr_apply<E, RB, float>), grid, block, 0, st, Ns, Np,                  \
                         (const float *)O, ldo, arows, chunks, q, rtol, partial, sc);           \
  } while (0)
    const int64_t e = (Np + 1023) / 1024;
    if (e <= 1)
      MR_APPLY(1, 2);
    else if (e <= 2)
      MR_APPLY(2, 2);
    else if (e <= 3)
      MR_APPLY(3, 2);
    else if (e <= 4)
      MR_APPLY(4, 2);
    else if (e <= 6)
      MR_APPLY(6, 1);
    else
      MR_APPLY(8, 1);
#undef MR_APPLY
  };
  MrVecs q{};
  q.m = m;
  q.x = x;
  for (int it = 0; it < maxiter; ++it) {
    q.r1 = r1;
    q.r2 = r2;
    q.first = it == 0;
    if (fused) {
      apply(q);
    } else {
      hipLaunchKernelGGL(mr_gemv_rows, dim3((unsigned)(Ns + 2)), dim3(512), 0, st, Ns, Np, O,
                         o_dtype, ldo, q, rtol, inner, sc);
      hipLaunchKernelGGL(mr_colsum_partial, dim3(gn, kRowChunks), dim3(256), 0, st, Ns, Np, O,
                         o_dtype, ldo, rows, (const double *)inner, (const double *)nullptr,
                         partial, partial2, done);
    }
    hipLaunchKernelGGL(mr_form_y, dim3(yb), dim3(1024), 0, st, Np, chunks, partial,
                       1.0 / (double)Ns, m, r1, r2, diag_shift, y, dotp, sc);
    hipLaunchKernelGGL(mr_finish, dim3(1), dim3(1024), 0, st, Np, (int64_t)yb, dotp, r2, y, sc);
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
    hipLaunchKernelGGL(mr_last_update, dim3(1), dim3(512), 0, st, Np, q, rtol, sc);
  }
  hipLaunchKernelGGL(mr_stats, dim3(1), dim3(1), 0, st, sc, stats, info);
  VMCX_LAUNCHED();
  return 0;
}

}  // namespace vmcx
