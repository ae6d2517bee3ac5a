// Chi-truncated boundary-MPS contraction of fPEPS / NN-fTNS amplitudes on
// gfx950: the reference's fPEPS_Model_GPU.amplitude with max_bond = chi
// (GPU/models/pureTNS.py:81-146: quimb contract_boundary_from_xmin over rows
// 0 .. Lx/2-1 and from_xmax over rows Lx-1 .. Lx/2, mode "mps", cutoff 0,
// canonize, then the two boundaries contracted exactly).
//
// Signed slices S_s[l,u,d,r] as in fpeps.hip (the sign convention of that
// file).  Each side is a boundary MPS B_y[a][v][b] along the row (a, b:
// boundary bonds, v: the open vertical leg).  Absorbing a row multiplies
// the bonds by the PEPS bond D:
//   A_y[(a,l)][v][(b,r)] = sum_u B_y[a][u][b] S_y[l][u][v][r]
// (u: the slice's leg facing the boundary, v: its open leg).  When a bond
// then exceeds chi, the MPS is truncated left to right onto the chi
// leading Schmidt vectors of each cut (the result of canonizing from the
// right and truncating by SVD from the left) by the density-matrix form:
//   right Grams  R_y = sum_v A_v R_{y+1} A_v^T   (y = Ly-1 .. 1, R_Ly = 1),
//   then for y = 0 .. Ly-2, with P the projection carried from the left:
//     C[(k,v)][(b,r)] = sum_{(a,l)} P[k][(a,l)] A_y[(a,l)][v][(b,r)],
//     rho = C R_{y+1} C^T, its chi leading eigenvectors U,
//     B'_y[k][v][j] = U[(k,v)][j],  P <- U^T C;
//   and B'_{Ly-1} = C.
// The tensors are Z2-graded, so rho is block diagonal in the parity of
// (k, v) (par(k) from the sector each kept eigenvector came from); each
// block is diagonalised by one-sided Jacobi on its pivoted Cholesky factor,
// in the registers of one wave (bm_jacobi_wave; blocks above 32: two-sided
// Jacobi in LDS, bm_jacobi).  Norms are carried as FP64 log scales.
//
// One workgroup of 256 threads per (configuration, side); the Grams and the
// boundary tensors live in a per-slot workspace in HBM, the 64 x 64 working
// matrices in LDS.  A second kernel joins the two boundaries (one wave per
// configuration).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "kernels.h"

namespace vmcx {

namespace {

constexpr int BT = 256;         // threads per (configuration, side)
constexpr int BN = 64;          // largest absorbed bond (chi * D)
constexpr int BLD = 65;         // LDS row stride of the BN x BN buffers
constexpr int BMAX_NS = 64;     // sites
constexpr int BMAX_LY = 16;
constexpr int BMAX_TS = 2048;   // largest stored tensor cb * D * cb
constexpr int BMAX_CHI = 32;
constexpr int BMAX_SWEEPS = 30;
// rho is scaled to a largest diagonal entry of 1; off-diagonal entries below
// this floor are not rotated away (singular values below ~1e-9 of the
// largest, which move an amplitude by about that much relative)
constexpr double BM_ROT_FLOOR = 1e-18;
// A pivot of the Cholesky factor must exceed BM_PIVOT_FLOOR (of the block's largest diagonal
// entry) and BM_PIVOT_NOISE of its own row's diagonal entry at the start.
// The second: a remainder d below the rounding of its row's entries (a few ulp of the
// diagonal) is noise, and noise^2 / d, which may be of any size where d happens to be small,
// would enter the factor.  With d above one ulp LL^T stays within 1e-13 of the block, in units
// of sqrt(A_ii A_jj) (NumPy, 2e5 16 x 16 blocks of rank 8: worst 3e-10 without, 1e-13 with
// half an ulp, 3e-14 with two), and no noise column is larger than a direction of
// eigenvalue 256 ulp, which it could push out of the chi kept ones: a D = 2 state written with
// D = 4, 6x6 chi = 8, 32768 amplitudes: 99.9 % within 3e-10, worst 8e-8; without 2e-9 and 1e-5
// (two-sided Jacobi 1e-9 and 1e-5).
// Neither may be larger: graded states (bond entries that fall off by 10 per index) need the
// small singular values, which the factor and one-sided Jacobi keep to relative accuracy, and
// their rows are graded likewise.  Against the QR / SVD truncation, median relative error of
// an amplitude, 6x6 D = 4 chi = 8 and 6x6 D = 2 chi = 6: 7e-11 and 2.6e-12 (two-sided Jacobi
// 8e-10 and 6e-12; BM_PIVOT_NOISE of 16 ulp 8e-11 and 9e-12; a floor of 4.4e-16 3e-8).
constexpr double BM_PIVOT_FLOOR = 1e-30;
constexpr double BM_PIVOT_NOISE = 2.220446049250313e-16;
// int64 header words per boundary buffer: [0] log scale (double bits),
// [1 .. Ly+1] bond dimensions, [Ly+2 .. 2Ly+2] bond parity masks
constexpr int BHDR = 40;

struct BmGeo {
  int Lx, Ly, D, N, chi, cb;    // cb = max(chi, D): bound of a stored bond
  int nbuf;                     // boundaries kept per side: 1 (amplitude), Lx - 1 (every
                                // row's environments) or max(h, Lx - h) (half, the cache)
  int half;                     // buffered sides stop at the middle (the sweep cache)
  const int32_t *dmap;
  const double *theta;
  int64_t theta_stride;
  int64_t slot;                 // doubles per (configuration, side)
  int64_t ts;                   // doubles per stored tensor, cb * D * cb
};

__device__ __forceinline__ int bqpar(int k, int d) { return d == 1 ? 0 : (k >= (d >> 1)); }
__device__ __forceinline__ int hdim(const BmGeo &g, int y) {
  return (y == 0 || y == g.Ly) ? 1 : g.D;
}

struct BmCfg {
  int p[BMAX_NS], pr[BMAX_NS], doff[BMAX_NS];
};

__device__ void bm_load_cfg(const BmGeo &g, const int64_t *c, BmCfg &cs) {
  const int tid = threadIdx.x;
  if (tid < g.N) cs.p[tid] = (int)c[tid];
  __syncthreads();
  if (tid < g.N) {
    const int x = tid / g.Ly, y = tid - x * g.Ly;
    int pr = 0;
    for (int yy = y + 1; yy < g.Ly; ++yy) {
      const int v = cs.p[x * g.Ly + yy];
      pr += (v == 1 || v == 2);
    }
    cs.pr[tid] = pr & 1;
  }
  if (tid == 0) {
    int off = 0;
    for (int s = 0; s < g.N; ++s) {
      const int x = s / g.Ly, y = s - x * g.Ly;
      const int dl = y == 0 ? 1 : g.D, du = x == 0 ? 1 : g.D;
      const int dd = x == g.Lx - 1 ? 1 : g.D, dr = y == g.Ly - 1 ? 1 : g.D;
      cs.doff[s] = off;
      off += 4 * dl * du * dd * dr;
    }
  }
  __syncthreads();
}

// signed slice of site (x, y) as dst[l][f][o][r]: f the leg facing the
// boundary (up from the top side, down from the bottom), o the open leg
__device__ void bm_slice(const BmGeo &g, const BmCfg &cs, const double *__restrict__ th, int x,
                         int y, bool down, double *dst) {
  const int dl = y == 0 ? 1 : g.D, du = x == 0 ? 1 : g.D;
  const int dd = x == g.Lx - 1 ? 1 : g.D, dr = y == g.Ly - 1 ? 1 : g.D;
  const int s = x * g.Ly + y;
  const int n = dl * du * dd * dr;
  const int base = cs.doff[s] + cs.p[s] * n;
  const int pr = cs.pr[s];
  for (int idx = threadIdx.x; idx < n; idx += BT) {
    const int r = idx % dr, d = (idx / dr) % dd, u = (idx / (dr * dd)) % du;
    const int l = idx / (dr * dd * du);
    const int k = g.dmap[base + idx];
    double v = k >= 0 ? th[k] : 0.0;
    if ((bqpar(d, dd) * (bqpar(r, dr) + pr)) & 1) v = -v;
    if (down)
      dst[((l * du + u) * dd + d) * dr + r] = v;
    else
      dst[((l * dd + d) * du + u) * dr + r] = v;
  }
}

__device__ double bm_max(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double m = red[0];
  for (int i = 1; i < BT / 64; ++i) m = fmax(m, red[i]);
  __syncthreads();
  return m;
}

template <int NB>
struct BmShT {
  static constexpr int LD = NB + 1;   // LDS row stride of the NB x NB buffers
  double R[NB * LD];        // right Gram; then rho
  double A[NB * LD];        // A_v; then C
  double T[NB * LD];        // A_v R; then W, G, V
  // the boundary tensor of the current site (na x D x nb) and the projection
  // carried from the left (kept-bond rows): bonds never exceed NB / 2 here
  // (NB = 32 holds cb * D <= 32, so bonds <= 16 for D >= 2 and stay 1 for
  // D = 1; NB = 64 holds chi <= 32)
  double Bt[NB * (NB / 2)];
  double Sl[256];           // its slice [l][f][o][r]
  double P[(NB / 2) * NB];
  double2 jcs[NB / 2 + 1];  // rotation (c, s) of each pair slot: one 16-byte load
  double jt[NB / 2 + 1];
  int jpq[NB / 2 + 1];      // its rows p | q << 8
  int perm[NB], pos[NB], sel[NB];
  int kpar[NB];             // parity of the current left bond's indices
  int bd[BMAX_LY + 1], nbd[BMAX_LY + 1];
  uint64_t bpm[BMAX_LY + 1], npm[BMAX_LY + 1];   // bond parity masks
  double red[BT / 64];
  double lam[NB];           // eigenvalues by column of T
  int sec[4];               // m0, m1, n0, n1
  int rot;
};

// B_y (dims na x D x nb, stride cb) from the slot into Bt
__device__ void bm_load_tensor(const BmGeo &g, const double *slot, int y, int na, int nb,
                               double *Bt) {
  const double *src = slot + (int64_t)y * g.ts;
  const int n = na * g.D * nb;
  for (int idx = threadIdx.x; idx < n; idx += BT) {
    const int b = idx % nb, av = idx / nb;
    Bt[idx] = src[av * g.cb + b];
  }
}

// Bt-shaped (na x D x nb, dense) LDS tensor scaled by 1 / max into the slot;
// returns ln max (-inf for a zero tensor)
__device__ double bm_store_scaled(const BmGeo &g, double *slot, int y, int na, int nb,
                                  const double *src, double *red) {
  const int n = na * g.D * nb;
  double m = 0.0;
  for (int idx = threadIdx.x; idx < n; idx += BT) m = fmax(m, fabs(src[idx]));
  m = bm_max(m, red);
  if (!(m > 0.0) || !std::isfinite(m)) return -INFINITY;
  const double inv = 1.0 / m;
  double *dst = slot + (int64_t)y * g.ts;
  for (int idx = threadIdx.x; idx < n; idx += BT) {
    const int b = idx % nb, av = idx / nb;
    dst[av * g.cb + b] = src[idx] * inv;
  }
  return log(m);
}

// out (n x m, stride LD) = X (n x K, stride LD) * Y (K x m, stride LD); TS x TS
// tiles on a 16 x 16 thread grid (TS = 2 covers 32 x 32, TS = 4 covers 64 x 64)
template <int LD, int TS>
__device__ void bm_mm(int n, int m, int K, const double *X, const double *Y, double *out) {
  const int ti = threadIdx.x >> 4, tj = threadIdx.x & 15;
  const int i0 = TS * ti, j0 = TS * tj;
  if (i0 >= n || j0 >= m) return;
  double acc[TS][TS] = {};
  for (int k = 0; k < K; ++k) {
    double xa[TS], yb[TS];
#pragma unroll
    for (int q = 0; q < TS; ++q) {
      xa[q] = (i0 + q < n) ? X[(i0 + q) * LD + k] : 0.0;
      yb[q] = (j0 + q < m) ? Y[k * LD + j0 + q] : 0.0;
    }
#pragma unroll
    for (int a = 0; a < TS; ++a)
#pragma unroll
      for (int b = 0; b < TS; ++b) acc[a][b] = fma(xa[a], yb[b], acc[a][b]);
  }
#pragma unroll
  for (int a = 0; a < TS; ++a)
#pragma unroll
    for (int b = 0; b < TS; ++b)
      if (i0 + a < n && j0 + b < m) out[(i0 + a) * LD + j0 + b] = acc[a][b];
}

// -------------------------------------------------- one-sided Jacobi in registers
// x of lane (l ^ M) within a 16-lane row, by data-parallel primitives (no LDS):
// quad permutes for 1 and 2, half-mirror (^7) after a quad mirror (^3) for 4,
// a rotation by 8 for 8.
template <int M>
__device__ __forceinline__ int bm_xor32(int v) {
  if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);
  if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);
  if constexpr (M == 4)
    return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(v, 0x1B, 0xF, 0xF, true), 0x141, 0xF,
                                    0xF, true);
  return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);
}
template <int M>
__device__ __forceinline__ double bm_xor(double x) {
  return __hiloint2double(bm_xor32<M>(__double2hiint(x)), bm_xor32<M>(__double2loint(x)));
}
// sum of x over lanes l and l ^ 16 (M = 16) or l ^ 32 (M = 32): the row and half
// swaps of gfx950; both lanes get the same bits
template <int M>
__device__ __forceinline__ double bm_swap_sum(double x) {
  const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
  if constexpr (M == 16) {
    const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
  } else {
    const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
  }
}

// 1 / sqrt(x): hardware estimate and one cubically convergent step
__device__ __forceinline__ double bm_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// Eigenvectors of a symmetric positive semidefinite m x m block (rows and columns
// off .. off + m of the upper triangle in R, scaled to a largest diagonal entry of 1,
// m <= 4 RPL): pivoted Cholesky L L^T = block, then one-sided Jacobi on the columns of
// L (Veselic and Hari, Numer. Math. 56, 1989): they are rotated in pairs until they are
// orthogonal; their squared norms are then the eigenvalues and the normalised columns
// the eigenvectors (no matrix of rotations is kept).  The pivoted factor is close to
// orthogonal columns already: 5.5 sweeps on average for the 16 x 16 blocks of a 6x6
// D = 4 chi = 8 boundary, against 13 for the columns of the block itself (half of them
// rounding noise of a rank-deficient block) and 9 for two-sided Jacobi.
// One wave holds the block in registers: lane (row group, j) has RPL rows of the two
// columns t and b of pair j, JB bits of j, four row groups; with JB = 3 a wave works
// on two blocks at once (lanes 32 .. 63: off, m of the second).  A sweep meets every
// pair of columns once: with groups of G lanes, the columns b visit the group's lanes
// in Gray-code order (G rounds, one cross-lane exchange by a single bit per round),
// then the t columns of a group pair up among themselves in one half of its lanes and
// the b columns in the other, and G halves.
//
// What bounds it: instruction issue of the one wave (about 80 per round, all vector
// ALU; the rotations are found redundantly in every row group, so nothing waits on
// LDS or a barrier).  The angle is found in FP32 from the FP64 sums (an angle off by
// 1e-7 leaves 1e-7 of the pair's product for the next sweep); its cosine and sine are
// orthonormal to FP64.  Measured on 6x6 D = 4 chi = 8, per 32 x 32 eigensolve with four
// workgroups on a CU: 80 k cycles; 198 k on the columns of the block itself, and 1754 us
// per launch of 2048 workgroups with two-sided Jacobi in LDS against 1020 us with this.
// Columns are orthogonal to 4e-15 of their own norms; what the
// factorisation leaves out (BM_PIVOT_FLOOR, BM_PIVOT_NOISE) comes out as zero vectors.
// row: LDS scratch of 4 RPL doubles per block.
// Output, compacted: columns off .. off + m of T (rows off .. off + m) and lam; the
// caller has zeroed both, or (CLEAR, JB = 3, off = 0, 16 x ld each) they are zeroed here
// once R, which T may then be, is in registers.
template <int JB, int RPL, bool CLEAR = false>
__device__ __forceinline__ void bm_jacobi_wave(const double *R, int ld, int off, int m, int mmax, double *row,
                               double *T, double *lam) {
  constexpr int NJ = 1 << JB;   // columns j and j + NJ
  const int lane = threadIdx.x & 63;
  const int j = lane & (NJ - 1), rg = (lane >> JB) & 3;
  double t[RPL] = {}, b[RPL] = {};
  int rank = 0;
  {
    // pivoted Cholesky, the remaining block at and ab, its diagonal at the two columns
    // in dt, db of every row group; the pivot row goes through LDS (same wave: in order)
    double at[RPL], ab[RPL];
    const int c0 = j, c1 = j + NJ;
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int r = rg * RPL + k;
      at[k] = (r < m && c0 < m) ? R[(off + (r < c0 ? r : c0)) * ld + off + (r < c0 ? c0 : r)]
                                : 0.0;
      ab[k] = (r < m && c1 < m) ? R[(off + (r < c1 ? r : c1)) * ld + off + (r < c1 ? c1 : r)]
                                : 0.0;
    }
    double dt = c0 < m ? R[(off + c0) * (ld + 1)] : 0.0;
    double db = c1 < m ? R[(off + c1) * (ld + 1)] : 0.0;
    const double ft = fmax(BM_PIVOT_FLOOR, BM_PIVOT_NOISE * dt);
    const double fb = fmax(BM_PIVOT_FLOOR, BM_PIVOT_NOISE * db);
    constexpr unsigned IM = 2 * NJ - 1;
    for (int step = 0; step < mmax; ++step) {
      // largest remaining diagonal entry (to FP32 precision, the column in the low bits)
      const unsigned kt = dt > ft ? (__float_as_uint((float)dt) & ~IM) | c0 : 0u;
      const unsigned kb = db > fb ? (__float_as_uint((float)db) & ~IM) | c1 : 0u;
      unsigned key = kt > kb ? kt : kb;
      key = max(key, (unsigned)bm_xor32<1>((int)key));
      key = max(key, (unsigned)bm_xor32<2>((int)key));
      key = max(key, (unsigned)bm_xor32<4>((int)key));
      if constexpr (JB == 4) key = max(key, (unsigned)bm_xor32<8>((int)key));
      if (!__any(key != 0u)) break;
      rank = step + 1;
      const int q = (int)(key & IM);
      if (rg == q / RPL) {
        double vt = at[0], vb = ab[0];
#pragma unroll
        for (int k = 1; k < RPL; ++k) {
          vt = (q % RPL) == k ? at[k] : vt;
          vb = (q % RPL) == k ? ab[k] : vb;
        }
        row[c0] = vt;
        row[c1] = vb;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const double rs = key != 0u ? bm_rsqrt(row[q]) : 0.0;
      const double lt = row[c0] * rs, lb = row[c1] * rs;
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const double lr = row[rg * RPL + k] * rs;
        at[k] = fma(-lr, lt, at[k]);
        ab[k] = fma(-lr, lb, ab[k]);
        t[k] = step == c0 ? lr : t[k];
        b[k] = step == c1 ? lr : b[k];
      }
      dt = c0 == q ? 0.0 : fma(-lt, lt, dt);
      db = c1 == q ? 0.0 : fma(-lb, lb, db);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  if constexpr (CLEAR) {
    for (int i = lane & 31; i < 16 * ld; i += 32) T[i] = 0.0;
    if ((lane & 31) < 16) lam[lane & 31] = 0.0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  // columns 0 .. rank - 1 are set: pairs over the first G0 lanes
  int G0 = 1;
  while (2 * G0 < rank) G0 <<= 1;
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    // column j + G0 of L: in t of lane j + G0 when G0 < NJ, in b of lane j otherwise
    double v = b[k];
    if (G0 == 1) v = bm_xor<1>(t[k]);
    if (G0 == 2) v = bm_xor<2>(t[k]);
    if (G0 == 4 && NJ > 4) v = bm_xor<4>(t[k]);
    if (G0 == 8 && NJ > 8) v = bm_xor<8>(t[k]);
    b[k] = j < G0 ? v : 0.0;
    t[k] = j < G0 ? t[k] : 0.0;
  }
  auto total = [](double x) {
    if constexpr (JB == 3) {
      x += bm_xor<8>(x);
      return bm_swap_sum<16>(x);
    } else {
      return bm_swap_sum<32>(bm_swap_sum<16>(x));
    }
  };
  for (int sweep = 0; sweep < BMAX_SWEEPS; ++sweep) {
    bool any = false;
    for (int G = G0; G >= 1; G >>= 1) {
      for (int r = 1; r <= G; ++r) {
        double pp = 0.0, qq = 0.0, pq = 0.0;
#pragma unroll
        for (int k = 0; k < RPL; ++k) {
          pp = fma(t[k], t[k], pp);
          qq = fma(b[k], b[k], qq);
          pq = fma(t[k], b[k], pq);
        }
        pp = total(pp);
        qq = total(qq);
        pq = total(pq);
        const bool big = pq * pq > 1.6e-29 * (pp * qq);
        if (__any(big)) {
          any = true;
          // t' = c t - s b, b' = s t + c b with tan = sgn(th) / (|th| + sqrt(th^2 + 1))
          const double th = (qq - pp) * __builtin_amdgcn_rcp(2.0 * pq);
          const float a = fabsf((float)th);
          const float d = a < 1e9f ? a + __builtin_amdgcn_sqrtf(fmaf(a, a, 1.0f)) : 2.0f * a;
          const float tf = big ? copysignf(__builtin_amdgcn_rcpf(d), (float)th) : 0.0f;
          const double tn = (double)tf;
          const double c = bm_rsqrt(fma(tn, tn, 1.0));
          const double s = tn * c;
#pragma unroll
          for (int k = 0; k < RPL; ++k) {
            const double tk = t[k], bk = b[k];
            t[k] = fma(-s, bk, c * tk);
            b[k] = fma(s, tk, c * bk);
          }
        }
        if (r < G) {
          // next lane of the Gray code: the lowest set bit of r
          if (r & 1) {
#pragma unroll
            for (int k = 0; k < RPL; ++k) b[k] = bm_xor<1>(b[k]);
          } else if (r & 2) {
#pragma unroll
            for (int k = 0; k < RPL; ++k) b[k] = bm_xor<2>(b[k]);
          } else if (r & 4) {
#pragma unroll
            for (int k = 0; k < RPL; ++k) b[k] = bm_xor<4>(b[k]);
          } else {
#pragma unroll
            for (int k = 0; k < RPL; ++k) b[k] = bm_xor<8>(b[k]);
          }
        }
      }
      if (G > 1) {
        // lanes of the lower half of a group take two t columns, the others two b
        const int bit = G >> 1;
        const bool up = j & bit;
#pragma unroll
        for (int k = 0; k < RPL; ++k) {
          const double out = up ? t[k] : b[k];
          const double in = bit == 1   ? bm_xor<1>(out)
                            : bit == 2 ? bm_xor<2>(out)
                            : bit == 4 ? bm_xor<4>(out)
                                       : bm_xor<8>(out);
          if (up)
            t[k] = in;
          else
            b[k] = in;
        }
      }
    }
    if (!any) break;
  }
  double pp = 0.0, qq = 0.0;
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    pp = fma(t[k], t[k], pp);
    qq = fma(b[k], b[k], qq);
  }
  pp = total(pp);
  qq = total(qq);
  const bool ot = pp > 1e-60, ob = qq > 1e-60;
  const int base = JB == 3 ? (lane & 32) : 0;   // row group 0 of this lane's block
  const uint64_t low = (1ull << (1 << JB)) - 1;
  const uint64_t mt = (__ballot(ot) >> base) & low, mb = (__ballot(ob) >> base) & low;
  const uint64_t below = (1ull << j) - 1;
  const int ct = off + __popcll(mt & below);
  const int cb = off + __popcll(mt) + __popcll(mb & below);
  const double it = bm_rsqrt(pp), ib = bm_rsqrt(qq);
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = rg * RPL + k;
    if (r < m && ot) T[(off + r) * ld + ct] = t[k] * it;
    if (r < m && ob) T[(off + r) * ld + cb] = b[k] * ib;
  }
  if (rg == 0) {
    if (ot) lam[ct] = pp;
    if (ob) lam[cb] = qq;
  }
}

// cyclic Jacobi on the two diagonal blocks [0, m0) and [m0, m0 + m1) of the
// symmetric S.R, kept as its upper triangle (entry (a, b) at
// [min(a,b)][max(a,b)], so that rounding cannot make it asymmetric: a skew
// residue would survive every rotation and keep the relative stopping test
// from being met); block sizes even, padding rows / columns zero;
// eigenvectors into S.T
template <int NB>
__device__ void bm_jacobi(BmShT<NB> &S, int m0, int m1) {
  constexpr int LD = BmShT<NB>::LD;
  const int tid = threadIdx.x;
  const int np0 = m0 >> 1, np1 = m1 >> 1, npr = np0 + np1;
  const int mt = m0 + m1;
  for (int idx = tid; idx < mt * mt; idx += BT) {
    const int i = idx / mt, j = idx - i * mt;
    S.T[i * LD + j] = i == j ? 1.0 : 0.0;
  }
  const int rounds = (m0 > m1 ? m0 : m1) - 1;
  if (rounds <= 0) {
    __syncthreads();
    return;
  }
  // the work of every thread is the same in every round (only the pairing
  // changes), so its items are decoded once here, not per round:
  // phase 1: the pair this thread rotates (block b, index i, size mb)
  const int pb = tid >= np0, pi_ = pb ? tid - np0 : tid;
  const int pmb = pb ? m1 : m0, poff = pb ? m0 : 0;
  // phase 2a: pair blocks (i1 <= i2) of the upper triangle, compacted
  constexpr int NBK = ((NB / 2) * (NB / 2 + 1) / 2 + BT - 1) / BT;
  const int nt0 = np0 * (np0 + 1) / 2, nt1 = np1 * (np1 + 1) / 2;
  int bk1[NBK], bk2[NBK];
#pragma unroll
  for (int k = 0; k < NBK; ++k) {
    int wi = tid + k * BT;
    bk1[k] = -1;
    bk2[k] = -1;
    if (wi < nt0 + nt1) {
      const int b = wi >= nt0;
      const int np = b ? np1 : np0, base = b ? np0 : 0;
      if (b) wi -= nt0;
      int i1 = 0;
      while (wi >= np - i1) {   // row i1 of the triangle holds np - i1 items
        wi -= np - i1;
        ++i1;
      }
      bk1[k] = base + i1;
      bk2[k] = base + i1 + wi;
    }
  }
  // phase 2b: rows of V and the pair whose columns they rotate
  constexpr int NV = (NB * NB / 2 + BT - 1) / BT;
  const int nv0 = m0 * np0, nv1 = m1 * np1;
  int vrow[NV], vpi[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int wi = tid + k * BT;
    vrow[k] = -1;
    vpi[k] = 0;
    if (wi < nv0) {
      vrow[k] = wi / np0;
      vpi[k] = wi - vrow[k] * np0;
    } else if (wi < nv0 + nv1) {
      const int w2 = wi - nv0;
      vrow[k] = m0 + w2 / np1;
      vpi[k] = np0 + w2 % np1;
    }
  }
  for (int sweep = 0; sweep < BMAX_SWEEPS; ++sweep) {
    if (tid == 0) S.rot = 0;
    __syncthreads();
    int rr = 0;   // the round within a block of size pmb: r mod (pmb - 1)
    for (int r = 0; r < rounds; ++r) {
      if (tid < npr) {
        int p = 0, q = 0;
        double c = 1.0, s = 0.0, t = 0.0;
        if (pmb >= 2) {
          if (pi_ == 0) {
            p = pmb - 1;
            q = rr;
          } else {
            p = rr + pi_;
            if (p >= pmb - 1) p -= pmb - 1;
            q = rr - pi_;
            if (q < 0) q += pmb - 1;
          }
          p += poff;
          q += poff;
          const double app = S.R[p * LD + p], aqq = S.R[q * LD + q];
          const double apq = S.R[(p < q ? p : q) * LD + (p < q ? q : p)];
          // |a_pq| > max(1e-15 sqrt|a_pp a_qq|, floor), compared in squares (no square root)
          if (apq * apq > fmax(1e-30 * fabs(app * aqq), BM_ROT_FLOOR * BM_ROT_FLOOR)) {
            // t = sgn(theta) / (|theta| + sqrt(theta^2 + 1)), theta = tau / zeta, written
            // with one square root and one division (|t| <= 1); c = 1 / sqrt(1 + t^2)
            // by the hardware estimate and three Newton steps (the estimate's 2^-22
            // relative error squared three times is below the FP64 rounding)
            const double tau = aqq - app, zeta = 2.0 * apq;
            t = copysign(1.0, tau) * zeta / (fabs(tau) + sqrt(tau * tau + zeta * zeta));
            const double x = 1.0 + t * t;
            double y = __builtin_amdgcn_rsq(x);
#pragma unroll
            for (int it = 0; it < 3; ++it) y = y * fma(-0.5 * x * y, y, 1.5);
            c = y;
            s = t * c;
            S.rot = 1;
          }
          if (++rr == pmb - 1) rr = 0;
        }
        S.jpq[tid] = p | (q << 8);
        S.jcs[tid] = make_double2(c, s);
        S.jt[tid] = t;
      }
      __syncthreads();
      // rho <- J^T rho J on the upper triangle of pair blocks
#pragma unroll
      for (int k = 0; k < NBK; ++k) {
        const int i1 = bk1[k], i2 = bk2[k];
        if (i1 < 0) continue;
        const double2 cs1 = S.jcs[i1], cs2 = S.jcs[i2];
        const double s1 = cs1.y, s2 = cs2.y;
        if (s1 == 0.0 && s2 == 0.0) continue;
        const int pq1 = S.jpq[i1];
        const int p1 = pq1 & 255, q1 = pq1 >> 8;
        if (i1 == i2) {
          // the rotated pair itself: its off-diagonal entry becomes zero
          const double t = S.jt[i1];
          const int lo = p1 < q1 ? p1 : q1, hi = p1 < q1 ? q1 : p1;
          const double apq = S.R[lo * LD + hi];
          S.R[p1 * LD + p1] -= t * apq;
          S.R[q1 * LD + q1] += t * apq;
          S.R[lo * LD + hi] = 0.0;
          continue;
        }
        const int pq2 = S.jpq[i2];
        const int p2 = pq2 & 255, q2 = pq2 >> 8;
        const double c1 = cs1.x, c2 = cs2.x;
        // entries of distinct pairs: never on the diagonal
        const int e0 = p1 < p2 ? p1 * LD + p2 : p2 * LD + p1;
        const int e1 = p1 < q2 ? p1 * LD + q2 : q2 * LD + p1;
        const int e2 = q1 < p2 ? q1 * LD + p2 : p2 * LD + q1;
        const int e3 = q1 < q2 ? q1 * LD + q2 : q2 * LD + q1;
        const double xpp = S.R[e0], xpq = S.R[e1], xqp = S.R[e2], xqq = S.R[e3];
        const double ypp = c1 * xpp - s1 * xqp, ypq = c1 * xpq - s1 * xqq;
        const double yqp = s1 * xpp + c1 * xqp, yqq = s1 * xpq + c1 * xqq;
        S.R[e0] = ypp * c2 - ypq * s2;
        S.R[e1] = ypp * s2 + ypq * c2;
        S.R[e2] = yqp * c2 - yqq * s2;
        S.R[e3] = yqp * s2 + yqq * c2;
      }
      // V <- V J over the rows of each block (loads issued before the stores)
      {
        int ip[NV], iq[NV];
        double vp[NV], vq[NV], cc[NV], ss[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          const bool on = vrow[k] >= 0;
          const double2 cs = on ? S.jcs[vpi[k]] : make_double2(1.0, 0.0);
          const int pq = on ? S.jpq[vpi[k]] : 0;
          ss[k] = cs.y;
          cc[k] = cs.x;
          ip[k] = on ? vrow[k] * LD + (pq & 255) : 0;
          iq[k] = on ? vrow[k] * LD + (pq >> 8) : 0;
        }
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          vp[k] = S.T[ip[k]];
          vq[k] = S.T[iq[k]];
        }
#pragma unroll
        for (int k = 0; k < NV; ++k)
          if (ss[k] != 0.0) {
            S.T[ip[k]] = cc[k] * vp[k] - ss[k] * vq[k];
            S.T[iq[k]] = ss[k] * vp[k] + cc[k] * vq[k];
          }
      }
      __syncthreads();
    }
    const int any = S.rot;
    __syncthreads();
    if (!any) break;
  }
}

// eigenvalues (S.lam) and eigenvectors (columns of S.T) of the two blocks
// [0, m0) and [m0, m0 + m1) of S.R, columns of a block at its positions.  Blocks of
// up to 32 go to one-sided Jacobi in the registers of one wave (both blocks, up to 16)
// or two (S.P, free until the new projection, as scratch); larger ones (D = 3 with
// chi > 16) to the workgroup's two-sided Jacobi in LDS.
template <int NB>
__device__ void bm_eigen(BmShT<NB> &S, int m0, int m1) {
  constexpr int LD = BmShT<NB>::LD;
  const int tid = threadIdx.x, wave = tid >> 6;
  const int mt = m0 + m1, mmax = m0 > m1 ? m0 : m1;
  if (NB > 32 && mmax > 32) {
    bm_jacobi<NB>(S, m0, m1);
    for (int i = tid; i < mt; i += BT) {
      const double l = S.R[i * LD + i];
      S.lam[i] = l == l ? l : 0.0;   // NaN: any order, but every rank taken once
    }
    __syncthreads();
    return;
  }
  for (int idx = tid; idx < mt * mt; idx += BT) {
    const int i = idx / mt, j = idx - i * mt;
    S.T[i * LD + j] = 0.0;
  }
  if (tid < mt) S.lam[tid] = 0.0;
  __syncthreads();
  // the working wave moves with the workgroup, so that workgroups that share a CU
  // use different SIMDs
  const int w0 = (blockIdx.x + 2 * blockIdx.y) & 3;
  if (mmax <= 16) {
    if (wave == w0) {
      const bool hi = tid & 32;
      bm_jacobi_wave<3, 4>(S.R, LD, hi ? m0 : 0, hi ? m1 : m0, mmax, S.P + (hi ? 16 : 0), S.T,
                           S.lam);
    }
  } else {
    const int blk = (wave - w0) & 3;
    if (blk < 2)
      // NB = 32: chi D <= 32, blocks of more than 16 only with D = 3: at most 2 chi <= 20
      bm_jacobi_wave<4, NB == 32 ? 5 : 8>(S.R, LD, blk ? m0 : 0, blk ? m1 : m0, blk ? m1 : m0, S.P + 32 * blk,
                           S.T, S.lam);
  }
  __syncthreads();
}

}  // namespace

// the side steps a move between sites sa and sb (spin offset N allowed)
// changes: st >= the side's row count means unchanged
__device__ __forceinline__ void bm_move_starts(const BmGeo &g, uint32_t mv, int &st_top,
                                               int &st_bot) {
  int sa = mv & 0xFF, sb = (mv >> 8) & 0xFF;
  if (sa >= g.N) sa -= g.N;
  if (sb >= g.N) sb -= g.N;
  const int ra = sa / g.Ly, rb = sb / g.Ly, h = g.Lx / 2;
  const int rmin = ra < rb ? ra : rb, rmax = ra < rb ? rb : ra;
  st_top = rmin <= h - 1 ? rmin : h;
  st_bot = rmax >= h ? g.Lx - 1 - rmax : g.Lx - h;
}

// ------------------------------------------------------------ one side
// grid (rows, 2): blockIdx.y = 0 the top side (rows 0 .. Lx/2-1, open down
// legs), 1 the bottom side (rows Lx-1 .. Lx/2, open up legs).  With
// g.nbuf = Lx - 1 every side runs over Lx - 1 rows and keeps the boundary
// after each (buffer i: rows 0 .. i from the top, Lx-1 .. Lx-1-i from the
// bottom): the environments of every row (quimb's compute_x_environments);
// with g.nbuf = 1 it stops at the middle and works in place.
template <int NB>
__global__ void __launch_bounds__(BT, NB == 32 ? 4 : 1)
    peps_bmps_side_kernel(BmGeo g, int64_t rows, const int64_t *__restrict__ cfg,
                          const int32_t *__restrict__ flag, double *ws, int64_t *hdr,
                          int st_top, int st_bot, const double *__restrict__ cache,
                          const int64_t *__restrict__ chdr, const int32_t *__restrict__ parent,
                          const uint32_t *__restrict__ cmove) {
  constexpr int LD = BmShT<NB>::LD;
  constexpr int TS = NB / 16;   // register tile of the dense products (16 x 16 threads)
  const int64_t w = blockIdx.x;
  if (w >= rows) return;
  if (flag && !(flag[w] & 1)) return;
  const int side = blockIdx.y;
  const bool down = side == 0;
  const int tid = threadIdx.x;
  // rows 0 .. start-1 of this side are those of the cached walker (parent[w],
  // or w): resume from its boundary after them (start >= nrows: the side is
  // unchanged); per configuration from its move when cmove is given
  if (cache && cmove) bm_move_starts(g, cmove[w], st_top, st_bot);
  const int start = cache ? (down ? st_top : st_bot) : 0;
  const int64_t pw = parent ? (int64_t)parent[w] : w;
  __shared__ BmCfg cs;
  __shared__ BmShT<NB> S;
  bm_load_cfg(g, cfg + w * g.N, cs);
  const double *th = g.theta + w * g.theta_stride;
  double *slot = ws + (w * 2 + side) * g.slot;
  const int64_t bstride = (int64_t)g.Ly * g.ts;
  double *Rg = slot + g.nbuf * bstride;
  int64_t *hd = hdr + (w * 2 + side) * g.nbuf * BHDR;
  const int Ly = g.Ly, D = g.D, h = g.Lx / 2;
  const int nrows = (g.nbuf > 1 && !g.half) ? g.Lx - 1 : (down ? h : g.Lx - h);
  if (start >= nrows) return;
  const int bufd = g.nbuf > 1 ? 1 : 0;   // buffer index step per row
  const double *cslot = cache ? cache + (pw * 2 + side) * g.slot : nullptr;
  const int64_t *chd = chdr ? chdr + (pw * 2 + side) * g.nbuf * BHDR : nullptr;
  const uint64_t dmask = D == 1 ? 0ull : (((1ull << D) - 1) & ~((1ull << (D >> 1)) - 1));
  double lg = 0.0;
  bool dead = false;
  if (start > 0) {
    const int64_t *c = chd + (start - 1) * bufd * BHDR;
    if (tid <= Ly) {
      S.bd[tid] = (int)c[1 + tid];
      S.bpm[tid] = (uint64_t)c[Ly + 2 + tid];
    }
    lg = __longlong_as_double(c[0]);
    dead = std::isinf(lg);
  } else if (tid <= Ly) {
    S.bd[tid] = hdim(g, tid);
    S.bpm[tid] = hdim(g, tid) == 1 ? 0ull : dmask;
  }
  __syncthreads();
  // first row: B_y[l][v][r] = S[l][0][v][r]
  if (start == 0) {
    const int x = down ? 0 : g.Lx - 1;
    for (int y = 0; y < Ly && !dead; ++y) {
      bm_slice(g, cs, th, x, y, down, S.Sl);
      __syncthreads();
      const int dl = hdim(g, y), dr = hdim(g, y + 1);
      const double l2 = bm_store_scaled(g, slot, y, dl, dr, S.Sl, S.red);
      __syncthreads();
      if (std::isinf(l2)) dead = true;
      lg += l2;
    }
    if (tid <= Ly) {
      hd[1 + tid] = S.bd[tid];
      hd[Ly + 2 + tid] = (int64_t)S.bpm[tid];
    }
    if (tid == 0) hd[0] = __double_as_longlong(dead ? -INFINITY : lg);
  }
  for (int ri = start > 1 ? start : 1; ri < nrows && !dead; ++ri) {
    const int x = down ? ri : g.Lx - 1 - ri;
    // boundary after row ri - 1 (the cache's for the first resumed row) ->
    // after row ri (the same buffer when nbuf = 1)
    const double *src = (start > 0 && ri == start) ? cslot + (ri - 1) * bstride
                                                   : slot + (ri - 1) * bufd * bstride;
    double *dst = slot + ri * bufd * bstride;
    if (tid <= Ly) {
      const int hd = hdim(g, tid), b = S.bd[tid];
      S.nbd[tid] = b * hd;
      uint64_t m = 0;
      for (int a = 0; a < b; ++a)
        for (int l = 0; l < hd; ++l)
          if ((((S.bpm[tid] >> a) & 1) ^ bqpar(l, hd))) m |= 1ull << (a * hd + l);
      S.npm[tid] = m;
    }
    __syncthreads();
    int mxb = 0;
    for (int y = 0; y <= Ly; ++y) mxb = S.nbd[y] > mxb ? S.nbd[y] : mxb;
    if (mxb <= g.chi) {
      // absorb without truncation
      for (int y = 0; y < Ly && !dead; ++y) {
        const int na = S.bd[y], nb = S.bd[y + 1], dl = hdim(g, y), dr = hdim(g, y + 1);
        bm_load_tensor(g, src, y, na, nb, S.Bt);
        bm_slice(g, cs, th, x, y, down, S.Sl);
        __syncthreads();
        const int ni = na * dl, nj = nb * dr, n = ni * D * nj;
        for (int idx = tid; idx < n; idx += BT) {
          const int j = idx % nj, v = (idx / nj) % D, i = idx / (nj * D);
          const int a = i / dl, l = i - a * dl, b = j / dr, r = j - b * dr;
          double s = 0.0;
          for (int u = 0; u < D; ++u)
            s = fma(S.Bt[(a * D + u) * nb + b], S.Sl[((l * D + u) * D + v) * dr + r], s);
          S.A[idx] = s;
        }
        __syncthreads();
        const double l2 = bm_store_scaled(g, dst, y, ni, nj, S.A, S.red);
        __syncthreads();
        if (std::isinf(l2)) dead = true;
        lg += l2;
      }
      if (tid <= Ly) {
        S.bd[tid] = S.nbd[tid];
        S.bpm[tid] = S.npm[tid];
      }
      __syncthreads();
      if (tid <= Ly) {
        hd[ri * bufd * BHDR + 1 + tid] = S.bd[tid];
        hd[ri * bufd * BHDR + Ly + 2 + tid] = (int64_t)S.bpm[tid];
      }
      if (tid == 0) hd[ri * bufd * BHDR] = __double_as_longlong(dead ? -INFINITY : lg);
      continue;
    }
    // ---- backward: right Grams R_y, y = Ly-1 .. 1 (R_Ly = 1)
    if (tid == 0) S.R[0] = 1.0;
    for (int y = Ly - 1; y >= 1; --y) {
      const int na = S.bd[y], nb = S.bd[y + 1], dl = hdim(g, y), dr = hdim(g, y + 1);
      const int n = na * dl, m = nb * dr;
      bm_load_tensor(g, src, y, na, nb, S.Bt);
      bm_slice(g, cs, th, x, y, down, S.Sl);
      __syncthreads();
      const int ti = tid >> 4, tj = tid & 15, i0 = TS * ti, j0 = TS * tj;
      double acc[TS][TS] = {};
      for (int v = 0; v < D; ++v) {
        for (int idx = tid; idx < n * m; idx += BT) {
          const int i = idx / m, j = idx - i * m;
          const int a = i / dl, l = i - a * dl, b = j / dr, r = j - b * dr;
          double s = 0.0;
          for (int u = 0; u < D; ++u)
            s = fma(S.Bt[(a * D + u) * nb + b], S.Sl[((l * D + u) * D + v) * dr + r], s);
          S.A[i * LD + j] = s;
        }
        __syncthreads();
        bm_mm<LD, TS>(n, m, m, S.A, S.R, S.T);
        __syncthreads();
        if (i0 < n && j0 < n) {
          for (int k = 0; k < m; ++k) {
            double xa[TS], yb[TS];
#pragma unroll
            for (int q = 0; q < TS; ++q) {
              xa[q] = (i0 + q < n) ? S.T[(i0 + q) * LD + k] : 0.0;
              yb[q] = (j0 + q < n) ? S.A[(j0 + q) * LD + k] : 0.0;
            }
#pragma unroll
            for (int a = 0; a < TS; ++a)
#pragma unroll
              for (int b = 0; b < TS; ++b) acc[a][b] = fma(xa[a], yb[b], acc[a][b]);
          }
        }
        __syncthreads();
      }
      double mx = 0.0;
#pragma unroll
      for (int a = 0; a < TS; ++a)
#pragma unroll
        for (int b = 0; b < TS; ++b) mx = fmax(mx, fabs(acc[a][b]));
      mx = bm_max(mx, S.red);
      const double inv = mx > 0.0 ? 1.0 / mx : 0.0;
      double *Rd = Rg + (int64_t)y * BN * BN;
#pragma unroll
      for (int a = 0; a < TS; ++a)
#pragma unroll
        for (int b = 0; b < TS; ++b)
          if (i0 + a < n && j0 + b < n) {
            const double v = acc[a][b] * inv;
            S.R[(i0 + a) * LD + j0 + b] = v;
            Rd[(i0 + a) * BN + j0 + b] = v;
          }
      __syncthreads();
    }
    // ---- forward: truncation left to right
    if (tid == 0) {
      S.P[0] = 1.0;
      S.kpar[0] = 0;
      S.nbd[0] = 1;
      S.npm[0] = 0;
    }
    __syncthreads();
    int k = 1;
    for (int y = 0; y < Ly && !dead; ++y) {
      const int na = S.bd[y], nb = S.bd[y + 1], dl = hdim(g, y), dr = hdim(g, y + 1);
      const int m = nb * dr, nC = k * D;
      bm_load_tensor(g, src, y, na, nb, S.Bt);
      bm_slice(g, cs, th, x, y, down, S.Sl);
      __syncthreads();
      // W[kk][l][u][b] = sum_a P[kk][(a,l)] B[a][u][b]  (into T)
      const int nw = k * dl * D * nb;
      for (int idx = tid; idx < nw; idx += BT) {
        const int b = idx % nb, u = (idx / nb) % D, l = (idx / (nb * D)) % dl;
        const int kk = idx / (nb * D * dl);
        double s = 0.0;
        for (int a = 0; a < na; ++a)
          s = fma(S.P[kk * NB + a * dl + l], S.Bt[(a * D + u) * nb + b], s);
        S.T[idx] = s;
      }
      __syncthreads();
      // C[(kk,v)][(b,r)] = sum_{l,u} W[kk][l][u][b] S[l][u][v][r]  (into A)
      for (int idx = tid; idx < nC * m; idx += BT) {
        const int j = idx % m, i = idx / m;
        const int kk = i / D, v = i - kk * D, b = j / dr, r = j - b * dr;
        double s = 0.0;
        for (int l = 0; l < dl; ++l)
          for (int u = 0; u < D; ++u)
            s = fma(S.T[((kk * dl + l) * D + u) * nb + b], S.Sl[((l * D + u) * D + v) * dr + r],
                    s);
        S.A[i * LD + j] = s;
      }
      __syncthreads();
      if (y == Ly - 1) {
        // last site: B'[kk][v][0] = C[(kk,v)][0]
        for (int idx = tid; idx < nC; idx += BT) S.T[idx] = S.A[idx * LD];
        __syncthreads();
        const double l2 = bm_store_scaled(g, dst, y, k, 1, S.T, S.red);
        __syncthreads();
        if (std::isinf(l2)) dead = true;
        lg += l2;
        if (tid == 0) {
          S.nbd[Ly] = 1;
          S.npm[Ly] = 0;
        }
        break;
      }
      double *dsty = dst + (int64_t)y * g.ts;
      int kn;
      if (nC <= g.chi) {
        // no truncation at this bond: the identity basis, P = C
        kn = nC;
        for (int idx = tid; idx < k * D * kn; idx += BT) {
          const int j = idx % kn, kv = idx / kn;
          dsty[kv * g.cb + j] = j == kv ? 1.0 : 0.0;
        }
        for (int idx = tid; idx < kn * m; idx += BT) {
          const int j = idx % m, i = idx / m;
          S.P[i * NB + j] = S.A[i * LD + j];
        }
        __syncthreads();
        if (tid < kn) S.sel[tid] = S.kpar[tid / D] ^ bqpar(tid % D, D);
        __syncthreads();
        if (tid < kn) S.kpar[tid] = S.sel[tid];
      } else {
        kn = g.chi;
        // R_{y+1} from the slot
        const double *Rs = Rg + (int64_t)(y + 1) * BN * BN;
        for (int idx = tid; idx < m * m; idx += BT) {
          const int i = idx / m, j = idx - i * m;
          S.R[i * LD + j] = Rs[i * BN + j];
        }
        if (tid == 0) {
          int n0 = 0;
          for (int i = 0; i < nC; ++i) n0 += !(S.kpar[i / D] ^ bqpar(i % D, D));
          const int n1 = nC - n0, m0 = n0 + (n0 & 1), m1 = n1 + (n1 & 1);
          int c0 = 0, c1 = m0;
          for (int i = 0; i < nC; ++i) {
            const int sct = S.kpar[i / D] ^ bqpar(i % D, D);
            const int pi = sct ? c1++ : c0++;
            S.perm[pi] = i;
            S.pos[i] = pi;
          }
          if (n0 & 1) S.perm[m0 - 1] = -1;
          if (n1 & 1) S.perm[m0 + m1 - 1] = -1;
          S.sec[0] = m0;
          S.sec[1] = m1;
        }
        __syncthreads();
        const int m0 = S.sec[0], m1 = S.sec[1], mt = m0 + m1;
        // G = C R (into T)
        bm_mm<LD, TS>(nC, m, m, S.A, S.R, S.T);
        __syncthreads();
        // rho (permuted, block diagonal) = G C^T (into R)
        for (int idx = tid; idx < mt * mt; idx += BT) {
          const int p1 = idx / mt, p2 = idx - p1 * mt;
          const int i1 = S.perm[p1], i2 = S.perm[p2];
          double s = 0.0;
          if (p1 <= p2 && i1 >= 0 && i2 >= 0 && ((p1 < m0) == (p2 < m0)))
            for (int j = 0; j < m; ++j) s = fma(S.T[i1 * LD + j], S.A[i2 * LD + j], s);
          S.R[p1 * LD + p2] = s;     // upper triangle only (the rest unused)
        }
        __syncthreads();
        double dmx = 0.0;
        for (int i = tid; i < mt; i += BT) dmx = fmax(dmx, fabs(S.R[i * LD + i]));
        dmx = bm_max(dmx, S.red);
        if (!(dmx > 0.0)) {
          dead = true;
          break;
        }
        const double dinv = 1.0 / dmx;
        for (int idx = tid; idx < mt * mt; idx += BT) {
          const int p1 = idx / mt, p2 = idx - p1 * mt;
          S.R[p1 * LD + p2] *= dinv;
        }
        __syncthreads();
        bm_eigen<NB>(S, m0, m1);
        // the chi leading eigenvalues (ties by position), padding excluded
        if (tid < mt && S.perm[tid] >= 0) {
          const double lam = S.lam[tid];
          int rank = 0;
          for (int q = 0; q < mt; ++q) {
            if (S.perm[q] < 0) continue;
            const double lq = S.lam[q];
            rank += (lq > lam) || (lq == lam && q < tid);
          }
          if (rank < kn) S.sel[rank] = tid;
        }
        __syncthreads();
        // B'[kk][v][j] = V[pos(kk,v)][sel j]
        for (int idx = tid; idx < nC * kn; idx += BT) {
          const int j = idx % kn, kv = idx / kn;
          dsty[kv * g.cb + j] = S.T[S.pos[kv] * LD + S.sel[j]];
        }
        // P'[j][(b,r)] = sum_pi V[pi][sel j] C[perm pi][(b,r)]
        for (int idx = tid; idx < kn * m; idx += BT) {
          const int jj = idx % m, j = idx / m;
          const int sj = S.sel[j];
          const int lo = sj < m0 ? 0 : m0, hi = sj < m0 ? m0 : mt;
          double s = 0.0;
          for (int pi = lo; pi < hi; ++pi) {
            const int i = S.perm[pi];
            if (i >= 0) s = fma(S.T[pi * LD + sj], S.A[i * LD + jj], s);
          }
          S.P[j * NB + jj] = s;
        }
        __syncthreads();
        if (tid < kn) S.kpar[tid] = S.sel[tid] >= m0;
      }
      __syncthreads();
      // renormalise P
      double pm = 0.0;
      for (int idx = tid; idx < kn * m; idx += BT) {
        const int j = idx % m, i = idx / m;
        pm = fmax(pm, fabs(S.P[i * NB + j]));
      }
      pm = bm_max(pm, S.red);
      if (!(pm > 0.0) || !std::isfinite(pm)) {
        dead = true;
        break;
      }
      const double pinv = 1.0 / pm;
      for (int idx = tid; idx < kn * m; idx += BT) {
        const int j = idx % m, i = idx / m;
        S.P[i * NB + j] *= pinv;
      }
      lg += log(pm);
      if (tid == 0) {
        S.nbd[y + 1] = kn;
        uint64_t msk = 0;
        for (int j = 0; j < kn; ++j) msk |= (uint64_t)S.kpar[j] << j;
        S.npm[y + 1] = msk;
      }
      __syncthreads();
      k = kn;
    }
    __syncthreads();
    if (tid <= Ly) {
      S.bd[tid] = S.nbd[tid];
      S.bpm[tid] = S.npm[tid];
    }
    __syncthreads();
    if (tid <= Ly) {
      hd[ri * bufd * BHDR + 1 + tid] = S.bd[tid];
      hd[ri * bufd * BHDR + Ly + 2 + tid] = (int64_t)S.bpm[tid];
    }
    if (tid == 0) hd[ri * bufd * BHDR] = __double_as_longlong(dead ? -INFINITY : lg);
  }
  // buffers never reached (a vanishing boundary): mark them zero
  if (dead && tid == 0)
    for (int i = start; i < nrows; ++i) hd[i * bufd * BHDR] = __double_as_longlong(-INFINITY);
}

// ------------------------------------------------------------ one side, one wave
// The same side in one wave with the dense products on v_mfma_f64_16x16x4f64, for bonds
// whose Z2 sectors hold at most 16 absorbed indices (bm_wave_fits).  Lane l, register r of
// a result holds D[4 r + l / 16][l % 16]; k-step r of an operand holds A[l % 16][4 r + l / 16]
// and B[4 r + l / 16][l % 16], so a result read as the A operand is its transpose.
//
// Absorbed bond indices (a, l) are numbered within their sector.  The block (s, c) of
// A_v[(a,l)][(b,r)] is nonzero for v of one parity, so number t of the even and of the odd
// v make one operand F (p64-style pairs: two at D = 4, one at D = 2), whose fragments each
// lane forms from B and the slice (two of the u are nonzero).  Then, per block (s, c):
//   T^T = R_c F^T  (R_c symmetric: a result serves as the A operand),
//   R'_s += T F^T  (T^T as a result is T as the A operand; F^T as before),
// so the Grams stay in registers from the last column to the first; each is also stored
// for the way back.  There C = sum P F, rho_s = C R C^T by the same two steps, its
// eigenvectors (bm_jacobi_wave, both sectors), P' = U^T C.
//
// Bound by the latency of one wave's chain; the workgroup-per-side kernel kept three of
// four waves idle in the eigensolver, read two LDS operands per multiply-add in the
// products and did four times as many (the zero blocks).  LDS 12 KB: up to 13 waves on a
// CU instead of 4 sides.  6x6 D = 4 chi = 8, 1024 walkers: sampling phase 133.8 ->
// 47.2 ms (with the join below; some 8 and 24 % more when held to 168 and 128 registers).
constexpr int BWL = 17;   // LDS row stride of the 16 x 16 blocks

bool bm_wave_fits(int D, int cb) {
  const int sector = D == 3 ? 2 * cb : D * cb / 2;
  return D >= 2 && sector <= 16;
}

// number t of the even (odd = 0) or odd values of a leg of dimension D; -1: none
template <int D>
__device__ __forceinline__ int bm_leg(int odd, int t) {
  constexpr int ne = D >> 1;
  const int v = odd ? ne + t : t;
  return (odd ? v < D : t < ne) ? v : -1;
}

struct BmWaveSh {
  double Sl[256];            // slice [l][f][o][r]
  double U[2][16 * BWL];     // rho, then its eigenvectors; P [16][33] until the next C
  double C[2][16 * BWL];     // by sector of (k, v)
  double lam[32], row[32];
  int perm[2][32];           // left / right bond: sector 16 + number -> a | l << 8 | par(a) << 16
  int kv[32];                // (k, v) -> sector << 8 | number
  int sel[32];
};

__device__ __forceinline__ void bm_wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
__device__ __forceinline__ double bm_wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

typedef double bmd4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bmd4 bm_mfma4(const double (&a)[4], const double (&b)[4], bmd4 acc) {
#pragma unroll
  for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], b[r], acc, 0, 0, 0);
  return acc;
}

template <int D>
__global__ void __launch_bounds__(64, 2)
    peps_bmps_wave_kernel(BmGeo g, int64_t rows, const int64_t *__restrict__ cfg,
                          const int32_t *__restrict__ flag, double *ws, int64_t *hdr, int st_top,
                          int st_bot, const double *__restrict__ cache,
                          const int64_t *__restrict__ chdr, const int32_t *__restrict__ parent,
                          const uint32_t *__restrict__ cmove) {
  constexpr int NPAIR = D > 2 ? 2 : 1;      // pairs of an even and an odd leg value
  const int64_t w = blockIdx.x;
  if (w >= rows) return;
  if (flag && !(flag[w] & 1)) return;
  const int side = blockIdx.y;
  const bool down = side == 0;
  const int lane = threadIdx.x, li = lane & 15, lk = lane >> 4;
  if (cache && cmove) bm_move_starts(g, cmove[w], st_top, st_bot);
  const int start = cache ? (down ? st_top : st_bot) : 0;
  const int64_t pw = parent ? (int64_t)parent[w] : w;
  const int Ly = g.Ly, h = g.Lx / 2, cb = g.cb;
  const int nrows = (g.nbuf > 1 && !g.half) ? g.Lx - 1 : (down ? h : g.Lx - h);
  if (start >= nrows) return;
  __shared__ BmWaveSh S;
  const double *th = g.theta + w * g.theta_stride;
  double *slot = ws + (w * 2 + side) * g.slot;
  const int64_t bstride = (int64_t)Ly * g.ts;
  double *Rg = slot + g.nbuf * bstride;       // [y][sector][register][lane]
  int64_t *hd = hdr + (w * 2 + side) * g.nbuf * BHDR;
  const int bufd = g.nbuf > 1 ? 1 : 0;
  const double *cslot = cache ? cache + (pw * 2 + side) * g.slot : nullptr;
  const int64_t *chd = chdr ? chdr + (pw * 2 + side) * g.nbuf * BHDR : nullptr;

  // the configuration as bit masks; lane s: dense offset of site s
  const int code = lane < g.N ? (int)cfg[w * g.N + lane] : 0;
  const uint64_t dn = __ballot(code & 1), up = __ballot(code & 2), sing = dn ^ up;
  int doff;
  {
    const int x = lane / Ly, y = lane - x * Ly;
    const int n = lane < g.N ? 4 * (y == 0 ? 1 : D) * (x == 0 ? 1 : D) *
                                   (x == g.Lx - 1 ? 1 : D) * (y == Ly - 1 ? 1 : D)
                             : 0;
    int sum = n;
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(sum, o);
      if (lane >= o) sum += t;
    }
    doff = sum - n;
  }
  auto site_par = [&](int x, int y) { return (int)((sing >> (x * Ly + y)) & 1); };
  auto leg = [&](int y) { return (y == 0 || y == Ly) ? 1 : D; };   // horizontal bond y
  // signed slice of site (x, y): entries lane, lane + 64, ... in registers
  auto fetch = [&](int x, int y, double (&sv)[4]) {
    const int s = x * Ly + y;
    const int dl = leg(y), dr = leg(y + 1), du = x == 0 ? 1 : D, dd = x == g.Lx - 1 ? 1 : D;
    const int n = dl * du * dd * dr;
    const int p = (int)((dn >> s) & 1) | ((int)((up >> s) & 1) << 1);
    const uint64_t right = s + 1 < 64 ? (sing >> (s + 1)) & ((1ull << (Ly - 1 - y)) - 1) : 0;
    const int pr = __popcll(right) & 1;
    const int base = __builtin_amdgcn_readlane(doff, s) + p * n;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int idx = lane + 64 * q;
      const int r = dr == 1 ? 0 : idx % D, i1 = dr == 1 ? idx : idx / D;
      const int d = dd == 1 ? 0 : i1 % D;
      const int k = idx < n ? g.dmap[base + idx] : -1;
      double v = k >= 0 ? th[k] : 0.0;
      if ((bqpar(d, dd) * (bqpar(r, dr) + pr)) & 1) v = -v;
      sv[q] = v;
    }
  };
  // ... into LDS as [l][f][o][r] (f: the leg facing the boundary)
  auto stash = [&](int x, int y, const double (&sv)[4]) {
    const int dl = leg(y), dr = leg(y + 1), du = x == 0 ? 1 : D, dd = x == g.Lx - 1 ? 1 : D;
    const int n = dl * du * dd * dr;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int idx = lane + 64 * q;
      if (idx >= n) continue;
      int to = idx;
      if (!down) {
        const int r = dr == 1 ? 0 : idx % D, i1 = dr == 1 ? idx : idx / D;
        const int d = dd == 1 ? 0 : i1 % D, i2 = dd == 1 ? i1 : i1 / D;
        const int u = du == 1 ? 0 : i2 % D, l = du == 1 ? i2 : i2 / D;
        to = ((l * dd + d) * du + u) * dr + r;
      }
      S.Sl[to] = sv[q];
    }
  };

  double lg = 0.0;
  bool dead = false;
  // lane y: dimension and parity mask of bond y; cm: bit y = parity of the nonzero
  // entries of B_y
  int bd = 1, bpm = 0, cm = 0;
  constexpr int dmask = ((1 << D) - 1) & ~((1 << (D >> 1)) - 1);
  if (start > 0) {
    const int64_t *c = chd + (start - 1) * bufd * BHDR;
    if (lane <= Ly) {
      bd = (int)c[1 + lane];
      bpm = (int)c[Ly + 2 + lane];
    }
    cm = __builtin_amdgcn_readfirstlane((int)c[2 * Ly + 3]);
    lg = __longlong_as_double(c[0]);
    dead = std::isinf(lg);
  } else if (lane <= Ly) {
    bd = leg(lane);
    bpm = bd == 1 ? 0 : dmask;
  }
  auto write_header = [&](int64_t *to) {
    if (lane <= Ly) {
      to[1 + lane] = bd;
      to[Ly + 2 + lane] = (int64_t)bpm;
    }
    if (lane == 0) {
      to[0] = __double_as_longlong(dead ? -INFINITY : lg);
      to[2 * Ly + 3] = cm;
    }
  };
  // tensor entries v[q] at offsets to[q] (-1: none) scaled by 1 / max; false: a zero tensor
  auto store_scaled = [&](double *dst, const double (&v)[8], const int (&to)[8]) {
    double m = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q) m = fmax(m, to[q] >= 0 ? fabs(v[q]) : 0.0);
    m = bm_wave_max(m);
    if (!(m > 0.0) || !std::isfinite(m)) return false;
    const double inv = 1.0 / m;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (to[q] >= 0) dst[to[q]] = v[q] * inv;
    lg += log(m);
    return true;
  };
  // first row: B_y[l][v][r] = S[l][0][v][r]
  if (start == 0) {
    const int x = down ? 0 : g.Lx - 1;
    for (int y = 0; y < Ly && !dead; ++y) {
      double sv[4];
      fetch(x, y, sv);
      const int dl = leg(y), dr = leg(y + 1), n = dl * D * dr;
      // the facing leg has dimension 1: [l][v][r] whichever side
      double v[8] = {sv[0], 0, 0, 0, 0, 0, 0, 0};
      int to[8] = {lane < n ? (dr == 1 ? lane : lane / D) * cb + (dr == 1 ? 0 : lane % D) : -1,
                   -1, -1, -1, -1, -1, -1, -1};
      if (!store_scaled(slot + (int64_t)y * g.ts, v, to)) dead = true;
      cm |= site_par(x, y) << y;
    }
    write_header(hd);
  }
  for (int ri = start > 1 ? start : 1; ri < nrows && !dead; ++ri) {
    const int x = down ? ri : g.Lx - 1 - ri;
    const double *src = (start > 0 && ri == start) ? cslot + (ri - 1) * bstride
                                                   : slot + (ri - 1) * bufd * bstride;
    double *dst = slot + ri * bufd * bstride;
    bm_wave_fence();   // the last row's tensors are this row's
    double sv[4], svn[4];
    if (__ballot(lane <= Ly && bd * leg(lane) > g.chi) == 0) {
      // absorb without truncation
      for (int y = 0; y < Ly && !dead; ++y) {
        fetch(x, y, sv);
        stash(x, y, sv);
        bm_wave_fence();
        const int na = __builtin_amdgcn_readlane(bd, y), nb = __builtin_amdgcn_readlane(bd, y + 1);
        const int dl = leg(y), dr = leg(y + 1), nj = nb * dr, n = na * dl * D * nj;
        const double *B = src + (int64_t)y * g.ts;
        double v[8];
        int to[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int idx = lane + 64 * q;
          v[q] = 0.0;
          to[q] = -1;
          if (idx < n) {
            const int j = idx % nj, iv = idx / nj, vv = iv % D, i = iv / D;
            const int a = dl == 1 ? i : i / D, l = dl == 1 ? 0 : i % D;
            const int b = dr == 1 ? j : j / D, r = dr == 1 ? 0 : j % D;
            double t = 0.0;
#pragma unroll
            for (int u = 0; u < D; ++u)
              t = fma(B[(a * D + u) * cb + b], S.Sl[((l * D + u) * D + vv) * dr + r], t);
            v[q] = t;
            to[q] = iv * cb + j;
          }
        }
        if (!store_scaled(dst + (int64_t)y * g.ts, v, to)) dead = true;
        bm_wave_fence();
        cm ^= site_par(x, y) << y;
      }
      const int hdy = lane <= Ly ? leg(lane) : 1;
      int m = 0;
      for (int a = 0; a < bd; ++a)
        for (int l = 0; l < hdy; ++l)
          if (((bpm >> a) & 1) ^ bqpar(l, hdy)) m |= 1 << (a * hdy + l);
      bd *= hdy;
      bpm = m;
      write_header(hd + ri * bufd * BHDR);
      continue;
    }
    // sector numbering of absorbed bond y into perm[o]
    auto number_bond = [&](int y, int o) {
      const int nb = __builtin_amdgcn_readlane(bd, y), mk = __builtin_amdgcn_readlane(bpm, y);
      const int hdy = leg(y), n = nb * hdy;
      const int a = hdy == 1 ? lane : lane / D, l = hdy == 1 ? 0 : lane % D;
      const int pa = (mk >> (a & 31)) & 1, par = pa ^ bqpar(l, hdy);
      const uint64_t odd = __ballot(lane < n && par), even = __ballot(lane < n && !par);
      const int num = __popcll((par ? odd : even) & ((1ull << lane) - 1));
      if (lane < 32) S.perm[o][lane] = -1;
      bm_wave_fence();
      if (lane < n) S.perm[o][par * 16 + num] = a | (l << 8) | (pa << 16);
      bm_wave_fence();
    };
    // B[a][u][b] of the two nonzero u of an entry (left code, right code), and the entry of
    // A_v from them
    auto b_entry = [&](const double *B, int cy, int lc, int rc, double (&bv)[2]) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int u = bm_leg<D>(cy ^ ((lc >> 16) & 1) ^ ((rc >> 16) & 1), q);
        bv[q] = (q < NPAIR && (lc | rc) >= 0 && u >= 0)
                    ? B[((lc & 255) * D + u) * cb + (rc & 255)]
                    : 0.0;
      }
    };
    auto a_entry = [&](int cy, int lc, int rc, const double (&bv)[2], int v, int dr) {
      double t = 0.0;
      if (v >= 0 && (lc | rc) >= 0)
#pragma unroll
        for (int q = 0; q < NPAIR; ++q) {
          const int u = bm_leg<D>(cy ^ ((lc >> 16) & 1) ^ ((rc >> 16) & 1), q);
          if (u >= 0)
            t = fma(bv[q], S.Sl[((((lc >> 8) & 255) * D + u) * D + v) * dr + ((rc >> 8) & 255)], t);
        }
      return t;
    };
    // ---- right Grams, y = Ly-1 .. 1 (R_Ly = 1 at the even index 0)
    double R[2][4] = {{lane == 0 ? 1.0 : 0.0, 0, 0, 0}, {0, 0, 0, 0}};
    fetch(x, Ly - 1, sv);
    number_bond(Ly, 1);
    for (int y = Ly - 1; y >= 1; --y) {
      const int lo = (Ly - 1 - y) & 1, ro = lo ^ 1;   // perm buffers of the left and right bond
      number_bond(y, lo);
      stash(x, y, sv);
      bm_wave_fence();
      fetch(x, y > 1 ? y - 1 : 0, svn);
      const int cy = (cm >> y) & 1, ey = cy ^ site_par(x, y), dr = leg(y + 1);
      const double *B = src + (int64_t)y * g.ts;
      bmd4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int lc = S.perm[lo][s * 16 + li];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          double bv[4][2];
          int rc[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            rc[r] = S.perm[ro][c * 16 + 4 * r + lk];
            b_entry(B, cy, lc, rc[r], bv[r]);
          }
#pragma unroll
          for (int t = 0; t < NPAIR; ++t) {
            const int v = bm_leg<D>(ey ^ s ^ c, t);
            if (v < 0) continue;
            double F[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) F[r] = a_entry(cy, lc, rc[r], bv[r], v, dr);
            const bmd4 z = {0, 0, 0, 0};
            const bmd4 tt = bm_mfma4(R[c], F, z);
            const double T[4] = {tt[0], tt[1], tt[2], tt[3]};
            acc[s] = bm_mfma4(T, F, acc[s]);
          }
        }
      }
      double mx = 0.0;
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmax(mx, fmax(fabs(acc[0][r]), fabs(acc[1][r])));
      mx = bm_wave_max(mx);
      const double inv = mx > 0.0 ? 1.0 / mx : 0.0;
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          R[s][r] = acc[s][r] * inv;
          Rg[(((int64_t)y * 2 + s) * 4 + r) * 64 + lane] = R[s][r];
        }
#pragma unroll
      for (int q = 0; q < 4; ++q) sv[q] = svn[q];
      bm_wave_fence();
    }
    // ---- forward: truncation left to right
    double *P = &S.U[0][0];
    constexpr int PLD = 33;
    for (int i = lane; i < 16 * PLD; i += 64) P[i] = 0.0;
    int k = 1, kp = 0, E = 0;        // kept bond: dimension, parity mask; parity so far
    int nbd = lane == 0 ? 1 : 0, npm = 0;
    bm_wave_fence();
    if (lane == 0) P[0] = 1.0;
    fetch(x, 0, sv);
    number_bond(0, 0);
    for (int y = 0; y < Ly && !dead; ++y) {
      const int lo = y & 1, ro = lo ^ 1;
      number_bond(y + 1, ro);
      stash(x, y, sv);
      const int nC = k * D;
      int nkv[2];
      {
        const int kk = lane / D, v = lane % D;
        const int par = ((kp >> (kk & 31)) & 1) ^ bqpar(v, D);
        const uint64_t odd = __ballot(lane < nC && par), even = __ballot(lane < nC && !par);
        nkv[0] = __popcll(even);
        nkv[1] = __popcll(odd);
        if (lane < nC) S.kv[lane] = (par << 8) | __popcll((par ? odd : even) & ((1ull << lane) - 1));
      }
      for (int i = lane; i < 2 * 16 * BWL; i += 64) (&S.C[0][0])[i] = 0.0;
      bm_wave_fence();
      fetch(x, y + 1 < Ly ? y + 1 : y, svn);
      const int cy = (cm >> y) & 1, ey = cy ^ site_par(x, y), dr = leg(y + 1);
      const int E2 = E ^ ey;
      const double *B = src + (int64_t)y * g.ts;
      // C[(k,v)][(b,r)] = sum_{(a,l)} P[k][(a,l)] A_v[(a,l)][(b,r)]: the row k of the
      // product has its (a,l) in sector par(k) ^ E, hence one v per pair
      double Pf[2][4];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) Pf[s][r] = P[li * PLD + s * 16 + 4 * r + lk];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        bmd4 acc[NPAIR];
#pragma unroll
        for (int t = 0; t < NPAIR; ++t) acc[t] = (bmd4){0, 0, 0, 0};
        const int rc = S.perm[ro][c * 16 + li];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          double bv[4][2];
          int lc[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            lc[r] = S.perm[lo][s * 16 + 4 * r + lk];
            b_entry(B, cy, lc[r], rc, bv[r]);
          }
#pragma unroll
          for (int t = 0; t < NPAIR; ++t) {
            const int v = bm_leg<D>(ey ^ s ^ c, t);
            if (v < 0) continue;
            double F[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) F[r] = a_entry(cy, lc[r], rc, bv[r], v, dr);
            acc[t] = bm_mfma4(Pf[s], F, acc[t]);
          }
        }
        // rows (k, v) of the sector that belongs to column sector c
#pragma unroll
        for (int t = 0; t < NPAIR; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int kk = 4 * r + lk;
            const int v = bm_leg<D>(E2 ^ c ^ ((kp >> kk) & 1), t);
            if (kk < k && v >= 0) {
              const int at = S.kv[kk * D + v];
              S.C[at >> 8][(at & 255) * BWL + li] = acc[t][r];
            }
          }
      }
      bm_wave_fence();
      if (y == Ly - 1) {
        // last site: B'[k][v][0] = C[(k,v)][0]
        double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        int to[8] = {-1, -1, -1, -1, -1, -1, -1, -1};
        if (lane < nC) {
          const int at = S.kv[lane];
          v[0] = S.C[at >> 8][(at & 255) * BWL];
          // the other sector's only nonzero column is not this one
          if ((at >> 8) != E2) v[0] = 0.0;
          to[0] = lane * cb;
        }
        if (!store_scaled(dst + (int64_t)y * g.ts, v, to)) dead = true;
        if (lane == Ly) {
          nbd = 1;
          npm = 0;
        }
        cm = E2 << (Ly - 1);
        break;
      }
      double *dsty = dst + (int64_t)y * g.ts;
      int kn, kpn;
      double pm = 0.0;
      if (nC <= g.chi) {
        // no truncation at this bond: the identity basis, P = C
        kn = nC;
        const int at0 = lane < nC ? S.kv[lane] : 0;
        kpn = (int)__ballot(lane < nC && (at0 >> 8));
        for (int idx = lane; idx < nC * kn; idx += 64) {
          const int j = idx % kn, kv = idx / kn;
          dsty[kv * cb + j] = j == kv ? 1.0 : 0.0;
        }
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          // entry (row kv, position) of P: kv = (lane + 64 q) / 32
          const int idx = lane + 64 * q, kv = idx >> 5, pos = idx & 31;
          v[q] = 0.0;
          if (kv < nC) {
            const int at = S.kv[kv];
            if (((at >> 8) ^ E2) == (pos >> 4)) v[q] = S.C[at >> 8][(at & 255) * BWL + (pos & 15)];
          }
          pm = fmax(pm, fabs(v[q]));
        }
        pm = bm_wave_max(pm);
        const double pinv = 1.0 / pm;
        if (pm > 0.0)
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int idx = lane + 64 * q;
            P[(idx >> 5) * PLD + (idx & 31)] = v[q] * pinv;
          }
      } else {
        kn = g.chi;
        // rho_s = C_s R C_s^T
        bmd4 rho[2];
        double dmx = 0.0;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          double Rf[4], Cf[4];
          const double *Rs = Rg + ((int64_t)(y + 1) * 2 + (s ^ E2)) * 256;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            Rf[r] = Rs[r * 64 + lane];
            Cf[r] = S.C[s][li * BWL + 4 * r + lk];
          }
          const bmd4 z = {0, 0, 0, 0};
          const bmd4 tt = bm_mfma4(Rf, Cf, z);
          const double T[4] = {tt[0], tt[1], tt[2], tt[3]};
          rho[s] = bm_mfma4(T, Cf, z);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (4 * r + lk == li) dmx = fmax(dmx, fabs(rho[s][r]));
        }
        dmx = bm_wave_max(dmx);
        if (!(dmx > 0.0)) {
          dead = true;
          break;
        }
        const double dinv = 1.0 / dmx;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int r = 0; r < 4; ++r) S.U[s][(4 * r + lk) * BWL + li] = rho[s][r] * dinv;
        bm_wave_fence();
        const int hs = lane >> 5;
        bm_jacobi_wave<3, 4, true>(S.U[hs], BWL, 0, hs ? nkv[1] : nkv[0], nkv[0] > nkv[1] ? nkv[0] : nkv[1],
                                   S.row + 16 * hs, S.U[hs], S.lam + 16 * hs);
        bm_wave_fence();
        // the chi leading eigenvalues: column (sector, number) = lane
        const double lam = (lane < 32 && li < (lk ? nkv[1] : nkv[0])) ? S.lam[lane] : -1.0;
        int rank = 0;
#pragma unroll
        for (int q = 0; q < 32; ++q) {
          const double lq = __shfl(lam, q);
          rank += (lq > lam) || (lq == lam && q < lane);
        }
        const int rk = (lane < 32 && lam >= 0.0 && rank < kn) ? rank : -1;
        if (rk >= 0) S.sel[rk] = lane;
        bm_wave_fence();
        kpn = (int)__ballot(lane < kn && (S.sel[lane & 31] >> 4));
        for (int idx = lane; idx < nC * kn; idx += 64) {
          const int j = idx % kn, kv = idx / kn, at = S.kv[kv], sj = S.sel[j];
          dsty[kv * cb + j] = (at >> 8) == (sj >> 4) ? S.U[at >> 8][(at & 255) * BWL + (sj & 15)] : 0.0;
        }
        // P' = U^T C: all columns of a sector at once, the chosen ones kept
        bmd4 pn[2];
        int to[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          double Uf[4], Cf[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            Uf[r] = S.U[s][(4 * r + lk) * BWL + li];
            Cf[r] = S.C[s][(4 * r + lk) * BWL + li];
          }
          const bmd4 z = {0, 0, 0, 0};
          pn[s] = bm_mfma4(Uf, Cf, z);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            to[s][r] = __shfl(rk, s * 16 + 4 * r + lk);
            if (to[s][r] >= 0) pm = fmax(pm, fabs(pn[s][r]));
          }
        }
        pm = bm_wave_max(pm);
        bm_wave_fence();
        for (int i = lane; i < 16 * PLD; i += 64) P[i] = 0.0;
        bm_wave_fence();
        const double pinv = 1.0 / pm;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (to[s][r] >= 0) P[to[s][r] * PLD + (s ^ E2) * 16 + li] = pn[s][r] * pinv;
      }
      if (!(pm > 0.0) || !std::isfinite(pm)) {
        dead = true;
        break;
      }
      lg += log(pm);
      if (lane == y + 1) {
        nbd = kn;
        npm = kpn;
      }
      k = kn;
      kp = kpn;
      E = E2;
#pragma unroll
      for (int q = 0; q < 4; ++q) sv[q] = svn[q];
      bm_wave_fence();
    }
    bd = nbd;
    bpm = npm;
    write_header(hd + ri * bufd * BHDR);
  }
  // buffers never reached (a vanishing boundary): mark them zero
  if (dead && lane == 0)
    for (int i = start; i < nrows; ++i) hd[i * bufd * BHDR] = __double_as_longlong(-INFINITY);
}

// ------------------------------------------------------------ join
// the amplitude from the top boundary in buffer bt and the bottom one in bb
__global__ void __launch_bounds__(64)
    peps_bmps_join_kernel(BmGeo g, int64_t rows, const int64_t *__restrict__ cfg,
                          const int32_t *__restrict__ flag, const double *__restrict__ ws,
                          const int64_t *__restrict__ hdr, int bt, int bb, double *sign,
                          double *logabs, int ct, int cb_, const double *__restrict__ cache,
                          const int64_t *__restrict__ chdr, const int32_t *__restrict__ parent,
                          const uint32_t *__restrict__ cmove) {
  const int64_t w = blockIdx.x;
  if (w >= rows) return;
  if (flag && !(flag[w] & 1)) return;
  const int tid = threadIdx.x;
  __shared__ double E[BMAX_CHI * BMAX_CHI], X[BMAX_TS];
  // a side taken from the cache (ct / cb_ set: unchanged since the walker
  // parent[w], or w; per configuration from its move when cmove is given)
  if (cache && cmove) {
    int s0, s1;
    bm_move_starts(g, cmove[w], s0, s1);
    ct = s0 >= g.Lx / 2;
    cb_ = s1 >= g.Lx - g.Lx / 2;
  }
  const int64_t pw = parent ? (int64_t)parent[w] : w;
  const int64_t *ht = ct ? chdr + ((pw * 2) * g.nbuf + bt) * BHDR
                         : hdr + ((w * 2) * g.nbuf + bt) * BHDR;
  const int64_t *hb = cb_ ? chdr + ((pw * 2 + 1) * g.nbuf + bb) * BHDR
                          : hdr + ((w * 2 + 1) * g.nbuf + bb) * BHDR;
  const double lt = __longlong_as_double(ht[0]), lb = __longlong_as_double(hb[0]);
  const double lo = log(1e-45);
  int P = 0;
  for (int s = 0; s < g.N; ++s) {
    const int v = (int)cfg[w * g.N + s];
    P += (v == 1 || v == 2);
  }
  if (std::isinf(lt) || std::isinf(lb)) {
    if (tid == 0) {
      sign[w] = 0.0;
      logabs[w] = lo;
    }
    return;
  }
  const int64_t bstride = (int64_t)g.Ly * g.ts;
  const double *Tt = ct ? cache + (pw * 2) * g.slot + bt * bstride
                        : ws + (w * 2) * g.slot + bt * bstride;
  const double *Tb = cb_ ? cache + (pw * 2 + 1) * g.slot + bb * bstride
                         : ws + (w * 2 + 1) * g.slot + bb * bstride;
  const int D = g.D, cb = g.cb;
  if (tid == 0) E[0] = 1.0;
  __syncthreads();
  double lsc = 0.0;
  for (int y = 0; y < g.Ly; ++y) {
    const int ta = (int)ht[1 + y], tb = (int)ht[2 + y], ba = (int)hb[1 + y], bb = (int)hb[2 + y];
    const double *T = Tt + (int64_t)y * g.ts, *Bo = Tb + (int64_t)y * g.ts;
    // X[a'][v][b] = sum_a E[a][a'] T[a][v][b]
    for (int idx = tid; idx < ba * D * tb; idx += 64) {
      const int b = idx % tb, v = (idx / tb) % D, ap = idx / (tb * D);
      double s = 0.0;
      for (int a = 0; a < ta; ++a) s = fma(E[a * BMAX_CHI + ap], T[(a * D + v) * cb + b], s);
      X[idx] = s;
    }
    __syncthreads();
    // E'[b][b'] = sum_{a',v} X[a'][v][b] Bo[a'][v][b']
    double mx = 0.0;
    for (int idx = tid; idx < tb * bb; idx += 64) {
      const int bp = idx % bb, b = idx / bb;
      double s = 0.0;
      for (int ap = 0; ap < ba; ++ap)
        for (int v = 0; v < D; ++v) s = fma(X[(ap * D + v) * tb + b], Bo[(ap * D + v) * cb + bp], s);
      E[b * BMAX_CHI + bp] = s;
      mx = fmax(mx, fabs(s));
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
    __syncthreads();
    if (!(mx > 0.0) || !std::isfinite(mx)) {
      if (tid == 0) {
        sign[w] = 0.0;
        logabs[w] = lo;
      }
      return;
    }
    const double inv = 1.0 / mx;
    for (int idx = tid; idx < tb * bb; idx += 64) {
      const int bp = idx % bb, b = idx / bb;
      E[b * BMAX_CHI + bp] *= inv;
    }
    lsc += log(mx);
    __syncthreads();
  }
  if (tid == 0) {
    const double v = E[0] * (((P * (P - 1) / 2) & 1) ? -1.0 : 1.0);
    if (v == 0.0 || !std::isfinite(v)) {
      sign[w] = 0.0;
      logabs[w] = lo;
    } else {
      sign[w] = v > 0.0 ? 1.0 : -1.0;
      logabs[w] = fmax(log(fabs(v)) + lsc + lt + lb, lo);
    }
  }
}

// The same join for bonds of at most 16, on v_mfma_f64_16x16x4f64 with everything in
// registers (layouts as in peps_bmps_wave_kernel): X_v = E^T T_v and E' += X_v^T Bo_v, each
// result being the next product's A operand; the next site's tensors are loaded during the
// products.  Bound by the latency of a wave's chain of Ly sites: 18 us for 1024
// configurations of 6x6 D = 4 chi = 8; over the calls of a sampling phase 31 us on average
// against 103 us with E and X in LDS.
template <int D>
__global__ void __launch_bounds__(64)
    peps_bmps_join_wave_kernel(BmGeo g, int64_t rows, const int64_t *__restrict__ cfg,
                               const int32_t *__restrict__ flag, const double *__restrict__ ws,
                               const int64_t *__restrict__ hdr, int bt, int bb, double *sign,
                               double *logabs, int ct, int cb_, const double *__restrict__ cache,
                               const int64_t *__restrict__ chdr,
                               const int32_t *__restrict__ parent,
                               const uint32_t *__restrict__ cmove) {
  const int64_t w = blockIdx.x;
  if (w >= rows) return;
  if (flag && !(flag[w] & 1)) return;
  const int lane = threadIdx.x, li = lane & 15, lk = lane >> 4;
  if (cache && cmove) {
    int s0, s1;
    bm_move_starts(g, cmove[w], s0, s1);
    ct = s0 >= g.Lx / 2;
    cb_ = s1 >= g.Lx - g.Lx / 2;
  }
  const int64_t pw = parent ? (int64_t)parent[w] : w;
  const int64_t *ht = ct ? chdr + ((pw * 2) * g.nbuf + bt) * BHDR
                         : hdr + ((w * 2) * g.nbuf + bt) * BHDR;
  const int64_t *hb = cb_ ? chdr + ((pw * 2 + 1) * g.nbuf + bb) * BHDR
                          : hdr + ((w * 2 + 1) * g.nbuf + bb) * BHDR;
  const double lt = __longlong_as_double(ht[0]), lb = __longlong_as_double(hb[0]);
  const double lo = log(1e-45);
  const int code = lane < g.N ? (int)cfg[w * g.N + lane] : 0;
  const int P = __popcll(__ballot(code == 1 || code == 2));
  const int64_t bstride = (int64_t)g.Ly * g.ts;
  const double *Tt = ct ? cache + (pw * 2) * g.slot + bt * bstride
                        : ws + (w * 2) * g.slot + bt * bstride;
  const double *Tb = cb_ ? cache + (pw * 2 + 1) * g.slot + bb * bstride
                         : ws + (w * 2 + 1) * g.slot + bb * bstride;
  const int cb = g.cb, Ly = g.Ly;
  bool zero = std::isinf(lt) || std::isinf(lb);
  double e0 = 0.0, lsc = 0.0;
  if (!zero) {
    const int dt = lane <= Ly ? (int)ht[1 + lane] : 0, db = lane <= Ly ? (int)hb[1 + lane] : 0;
    struct Ops {
      double t[D][4], b[D][4];
    };
    auto load = [&](int y, Ops &o) {
      const int ta = __builtin_amdgcn_readlane(dt, y), tb = __builtin_amdgcn_readlane(dt, y + 1);
      const int ba = __builtin_amdgcn_readlane(db, y), bb2 = __builtin_amdgcn_readlane(db, y + 1);
      const double *T = Tt + (int64_t)y * g.ts, *Bo = Tb + (int64_t)y * g.ts;
#pragma unroll
      for (int v = 0; v < D; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int a = 4 * r + lk;
          o.t[v][r] = (a < ta && li < tb) ? T[(a * D + v) * cb + li] : 0.0;
          o.b[v][r] = (a < ba && li < bb2) ? Bo[(a * D + v) * cb + li] : 0.0;
        }
    };
    bmd4 E = {lane == 0 ? 1.0 : 0.0, 0.0, 0.0, 0.0};
    Ops cur, nxt;
    load(0, cur);
    for (int y = 0; y < Ly; ++y) {
      const int ta = __builtin_amdgcn_readlane(dt, y), ba = __builtin_amdgcn_readlane(db, y);
      load(y + 1 < Ly ? y + 1 : y, nxt);
      bmd4 X[D], out[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
      for (int v = 0; v < D; ++v) X[v] = (bmd4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * r < ta)
#pragma unroll
          for (int v = 0; v < D; ++v)
            X[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(E[r], cur.t[v][r], X[v], 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * r < ba)
#pragma unroll
          for (int v = 0; v < D; ++v)
            out[v & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(X[v][r], cur.b[v][r], out[v & 1], 0,
                                                              0, 0);
      double mx = 0.0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        E[r] = out[0][r] + out[1][r];
        mx = fmax(mx, fabs(E[r]));
      }
      mx = bm_wave_max(mx);
      if (!(mx > 0.0) || !std::isfinite(mx)) {
        zero = true;
        break;
      }
      const double inv = 1.0 / mx;
#pragma unroll
      for (int r = 0; r < 4; ++r) E[r] *= inv;
      lsc += log(mx);
      cur = nxt;
    }
    e0 = E[0];
  }
  if (lane == 0) {
    const double v = zero ? 0.0 : e0 * (((P * (P - 1) / 2) & 1) ? -1.0 : 1.0);
    if (v == 0.0 || !std::isfinite(v)) {
      sign[w] = 0.0;
      logabs[w] = lo;
    } else {
      sign[w] = v > 0.0 ? 1.0 : -1.0;
      logabs[w] = fmax(log(fabs(v)) + lsc + lt + lb, lo);
    }
  }
}

// ------------------------------------------------------------ cheap gradient
// d ln|psi| / d theta of the sites of row r with the boundary environments of
// the row held fixed (the reference's cheap gradient, pureTNS.py:2230-2334):
// Z_r = <top_r| row r |bot_r>, top_r the boundary of rows < r (buffer r-1 of
// the top side), bot_r of rows > r (buffer Lx-2-r of the bottom side); the
// right strip environments R_y[b][r][b'] first (kept in renv), then a left
// sweep with L_y[a][l][a'] that forms
//   dZ/dS_y[l][u][d][r] = sum L_y[a][l][a'] T_y[a][u][b] Bo_y[a'][d][b'] R_{y+1}[b][r][b'],
// divided by psi (sign, logabs of the join) and scattered to theta's entries
// of the configuration's local states (G rows zeroed beforehand).
struct GrSh {
  double T[BMAX_TS], Bo[BMAX_TS], L[BMAX_TS], R[BMAX_TS];
  double X[BN * BN], Y[BN * BN];
  double Sl[256], dS[256];
  double red[BT / 64];
  int bt[BMAX_LY + 1], bb[BMAX_LY + 1];
};

__global__ void __launch_bounds__(BT)
    peps_bmps_grad_kernel(BmGeo g, int64_t rows, const int64_t *__restrict__ cfg,
                          const int32_t *__restrict__ flag, const double *__restrict__ ws,
                          const int64_t *__restrict__ hdr, const double *__restrict__ sign,
                          const double *__restrict__ logabs, double *renv, double *G,
                          int64_t ldg) {
  const int64_t w = blockIdx.x;
  const int r = blockIdx.y;
  if (w >= rows) return;
  if (flag && !(flag[w] & 1)) return;
  if (sign[w] == 0.0) return;
  const int tid = threadIdx.x;
  __shared__ BmCfg cs;
  __shared__ GrSh S;
  bm_load_cfg(g, cfg + w * g.N, cs);
  const double *th = g.theta + w * g.theta_stride;
  const int Lx = g.Lx, Ly = g.Ly, D = g.D;
  const int64_t bstride = (int64_t)Ly * g.ts;
  const bool ttriv = r == 0, btriv = r == Lx - 1;
  const double *tsrc = ws + (w * 2) * g.slot + (ttriv ? 0 : (r - 1) * bstride);
  const double *bsrc = ws + (w * 2 + 1) * g.slot + (btriv ? 0 : (Lx - 2 - r) * bstride);
  const int64_t *th_ = hdr + ((w * 2) * g.nbuf + (ttriv ? 0 : r - 1)) * BHDR;
  const int64_t *hb_ = hdr + ((w * 2 + 1) * g.nbuf + (btriv ? 0 : Lx - 2 - r)) * BHDR;
  const double lt = ttriv ? 0.0 : __longlong_as_double(th_[0]);
  const double lb = btriv ? 0.0 : __longlong_as_double(hb_[0]);
  if (std::isinf(lt) || std::isinf(lb)) return;
  if (tid <= Ly) {
    S.bt[tid] = ttriv ? 1 : (int)th_[1 + tid];
    S.bb[tid] = btriv ? 1 : (int)hb_[1 + tid];
  }
  int P = 0;
  for (int q = 0; q < g.N; ++q) P += (cs.p[q] == 1 || cs.p[q] == 2);
  const double gsign = ((P * (P - 1) / 2) & 1) ? -1.0 : 1.0;
  const int du = r == 0 ? 1 : D, dd = r == Lx - 1 ? 1 : D;
  double *rs = renv + (w * Lx + r) * ((int64_t)(Ly + 1) * g.ts + Ly + 1);
  double *rlog = rs + (int64_t)(Ly + 1) * g.ts;
  __syncthreads();
  // load T_y (ta x du x tb) and Bo_y (ba x dd x bb) densely
  auto load_env = [&](int y) {
    const int ta = S.bt[y], tb = S.bt[y + 1], ba = S.bb[y], bb = S.bb[y + 1];
    for (int idx = tid; idx < ta * du * tb; idx += BT) {
      const int b = idx % tb, au = idx / tb;
      S.T[idx] = ttriv ? 1.0 : tsrc[(int64_t)y * g.ts + au * g.cb + b];
    }
    for (int idx = tid; idx < ba * dd * bb; idx += BT) {
      const int b = idx % bb, ad = idx / bb;
      S.Bo[idx] = btriv ? 1.0 : bsrc[(int64_t)y * g.ts + ad * g.cb + b];
    }
  };
  // ---- right strip environments R_y, y = Ly-1 .. 1 (R_Ly = 1)
  if (tid == 0) {
    S.R[0] = 1.0;
    rlog[Ly] = 0.0;
  }
  double lr = 0.0;
  for (int y = Ly - 1; y >= 1; --y) {
    const int ta = S.bt[y], tb = S.bt[y + 1], ba = S.bb[y], bb = S.bb[y + 1];
    const int dl = hdim(g, y), dr = hdim(g, y + 1);
    load_env(y);
    bm_slice(g, cs, th, r, y, true, S.Sl);
    __syncthreads();
    // Z1[a][u][rr][b'] = sum_b T[a][u][b] R[b][rr][b']
    for (int idx = tid; idx < ta * du * dr * bb; idx += BT) {
      const int bp = idx % bb, rr = (idx / bb) % dr, au = idx / (bb * dr);
      double v = 0.0;
      for (int b = 0; b < tb; ++b) v = fma(S.T[au * tb + b], S.R[(b * dr + rr) * bb + bp], v);
      S.X[idx] = v;
    }
    __syncthreads();
    // Z2[a][l][d][b'] = sum_{u,rr} Z1[a][u][rr][b'] S[l][u][d][rr]
    for (int idx = tid; idx < ta * dl * dd * bb; idx += BT) {
      const int bp = idx % bb, d = (idx / bb) % dd, l = (idx / (bb * dd)) % dl;
      const int a = idx / (bb * dd * dl);
      double v = 0.0;
      for (int u = 0; u < du; ++u)
        for (int rr = 0; rr < dr; ++rr)
          v = fma(S.X[((a * du + u) * dr + rr) * bb + bp], S.Sl[((l * du + u) * dd + d) * dr + rr],
                  v);
      S.Y[idx] = v;
    }
    __syncthreads();
    // R_y[a][l][a'] = sum_{d,b'} Z2[a][l][d][b'] Bo[a'][d][b']
    double mx = 0.0;
    const int nr = ta * dl * ba;
    for (int idx = tid; idx < nr; idx += BT) {
      const int ap = idx % ba, al = idx / ba;
      double v = 0.0;
      for (int d = 0; d < dd; ++d)
        for (int bp = 0; bp < bb; ++bp)
          v = fma(S.Y[(al * dd + d) * bb + bp], S.Bo[(ap * dd + d) * bb + bp], v);
      S.L[idx] = v;
      mx = fmax(mx, fabs(v));
    }
    mx = bm_max(mx, S.red);
    if (!(mx > 0.0) || !std::isfinite(mx)) return;   // uniform: a vanishing strip
    const double inv = 1.0 / mx;
    lr += log(mx);
    for (int idx = tid; idx < nr; idx += BT) {
      const double v = S.L[idx] * inv;
      S.R[idx] = v;
      rs[(int64_t)y * g.ts + idx] = v;
    }
    if (tid == 0) rlog[y] = lr;
    __syncthreads();
  }
  // ---- left sweep with the derivative of every site
  if (tid == 0) S.L[0] = 1.0;
  double ll = 0.0;
  const double base = lt + lb - logabs[w];
  const double sg = sign[w] * gsign;
  for (int y = 0; y < Ly; ++y) {
    const int ta = S.bt[y], tb = S.bt[y + 1], ba = S.bb[y], bb = S.bb[y + 1];
    const int dl = hdim(g, y), dr = hdim(g, y + 1);
    load_env(y);
    bm_slice(g, cs, th, r, y, true, S.Sl);
    const double lry = y == Ly - 1 ? 0.0 : rlog[y + 1];
    if (y == Ly - 1) {
      if (tid == 0) S.R[0] = 1.0;
    } else {
      for (int idx = tid; idx < tb * dr * bb; idx += BT)
        S.R[idx] = rs[(int64_t)(y + 1) * g.ts + idx];
    }
    __syncthreads();
    // X1[l][a'][u][b] = sum_a L[a][l][a'] T[a][u][b]
    for (int idx = tid; idx < dl * ba * du * tb; idx += BT) {
      const int b = idx % tb, u = (idx / tb) % du, ap = (idx / (tb * du)) % ba;
      const int l = idx / (tb * du * ba);
      double v = 0.0;
      for (int a = 0; a < ta; ++a) v = fma(S.L[(a * dl + l) * ba + ap], S.T[(a * du + u) * tb + b], v);
      S.X[idx] = v;
    }
    // Y2[a'][d][b][rr] = sum_b' Bo[a'][d][b'] R[b][rr][b']
    for (int idx = tid; idx < ba * dd * tb * dr; idx += BT) {
      const int rr = idx % dr, b = (idx / dr) % tb, ad = idx / (dr * tb);
      double v = 0.0;
      for (int bp = 0; bp < bb; ++bp) v = fma(S.Bo[ad * bb + bp], S.R[(b * dr + rr) * bb + bp], v);
      S.Y[idx] = v;
    }
    __syncthreads();
    // dS[l][u][d][rr] = sum_{a',b} X1[l][a'][u][b] Y2[a'][d][b][rr] -> G
    {
      const int n = dl * du * dd * dr;
      const int s_ = r * Ly + y;
      const int gbase = cs.doff[s_] + cs.p[s_] * n;
      const int pr = cs.pr[s_];
      const double coef = sg * exp(ll + lry + base);
      for (int idx = tid; idx < n; idx += BT) {
        const int rr = idx % dr, d = (idx / dr) % dd, u = (idx / (dr * dd)) % du;
        const int l = idx / (dr * dd * du);
        const int k = g.dmap[gbase + idx];
        if (k < 0) continue;
        double v = 0.0;
        for (int ap = 0; ap < ba; ++ap)
          for (int b = 0; b < tb; ++b)
            v = fma(S.X[((l * ba + ap) * du + u) * tb + b], S.Y[((ap * dd + d) * tb + b) * dr + rr],
                    v);
        if ((bqpar(d, dd) * (bqpar(rr, dr) + pr)) & 1) v = -v;
        G[w * ldg + k] = coef * v;
      }
    }
    if (y == Ly - 1) break;
    __syncthreads();
    // X2[a'][b][d][rr] = sum_{l,u} X1[l][a'][u][b] S[l][u][d][rr]  (into Y)
    for (int idx = tid; idx < ba * tb * dd * dr; idx += BT) {
      const int rr = idx % dr, d = (idx / dr) % dd, b = (idx / (dr * dd)) % tb;
      const int ap = idx / (dr * dd * tb);
      double v = 0.0;
      for (int l = 0; l < dl; ++l)
        for (int u = 0; u < du; ++u)
          v = fma(S.X[((l * ba + ap) * du + u) * tb + b], S.Sl[((l * du + u) * dd + d) * dr + rr],
                  v);
      S.Y[idx] = v;
    }
    __syncthreads();
    // L_{y+1}[b][rr][b'] = sum_{a',d} X2[a'][b][d][rr] Bo[a'][d][b']
    double mx = 0.0;
    const int nl = tb * dr * bb;
    for (int idx = tid; idx < nl; idx += BT) {
      const int bp = idx % bb, rr = (idx / bb) % dr, b = idx / (bb * dr);
      double v = 0.0;
      for (int ap = 0; ap < ba; ++ap)
        for (int d = 0; d < dd; ++d)
          v = fma(S.Y[((ap * tb + b) * dd + d) * dr + rr], S.Bo[(ap * dd + d) * bb + bp], v);
      S.X[idx] = v;
      mx = fmax(mx, fabs(v));
    }
    mx = bm_max(mx, S.red);
    if (!(mx > 0.0) || !std::isfinite(mx)) return;
    const double inv = 1.0 / mx;
    ll += log(mx);
    for (int idx = tid; idx < nl; idx += BT) S.L[idx] = S.X[idx] * inv;
    __syncthreads();
  }
}

// the boundaries an accepted proposal recomputed (buffers start .. nrows-1
// of each side, and their headers) into its walker's cache
__global__ void __launch_bounds__(256)
    bm_commit_kernel(BmGeo g, int64_t rows, const int32_t *__restrict__ acc, int st_top,
                     int st_bot, const double *__restrict__ ws, const int64_t *__restrict__ hdr,
                     double *cache, int64_t *chdr) {
  const int64_t w = blockIdx.x;
  if (w >= rows || !acc[w]) return;
  const int side = blockIdx.y;
  const bool down = side == 0;
  const int h = g.Lx / 2, nrows = down ? h : g.Lx - h;
  const int start = down ? st_top : st_bot;
  if (start >= nrows) return;
  const int bufd = g.nbuf > 1 ? 1 : 0;
  const int64_t bstride = (int64_t)g.Ly * g.ts;
  const double *src = ws + (w * 2 + side) * g.slot;
  double *dst = cache + (w * 2 + side) * g.slot;
  const int64_t *hs = hdr + (w * 2 + side) * g.nbuf * BHDR;
  int64_t *hc = chdr + (w * 2 + side) * g.nbuf * BHDR;
  for (int b = start; b < nrows; ++b) {
    const int64_t o = b * bufd * bstride;
    for (int64_t i = threadIdx.x; i < bstride; i += 256) dst[o + i] = src[o + i];
    for (int i = threadIdx.x; i < BHDR; i += 256) hc[b * bufd * BHDR + i] = hs[b * bufd * BHDR + i];
  }
}

__global__ void bm_zero_rows_kernel(int64_t rows, int64_t P, double *G, int64_t ldg) {
  const int64_t n = rows * P;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t w = i / P, k = i - w * P;
    G[w * ldg + k] = 0.0;
  }
}

// ------------------------------------------------------------ host side
namespace {
BmGeo bm_geo(int Lx, int Ly, int D, int chi, int nbuf, int half = 0) {
  BmGeo g{};
  g.half = half;
  g.Lx = Lx;
  g.Ly = Ly;
  g.D = D;
  g.N = Lx * Ly;
  g.chi = chi;
  g.cb = chi > D ? chi : D;
  g.nbuf = nbuf;
  g.ts = (int64_t)g.cb * D * g.cb;
  g.slot = (int64_t)nbuf * Ly * g.ts + (int64_t)Ly * (bm_wave_fits(D, g.cb) ? 512 : BN * BN);
  return g;
}
// a wave per side when the sectors fit 16 x 16 blocks; else the workgroup kernel, with
// 32 x 32 working matrices when chi * D allows (38 KB of LDS, several workgroups per CU)
// or 64 x 64 (one per CU)
void launch_side(const BmGeo &g, int64_t n, const int64_t *c, const int32_t *f, double *slots,
                 int64_t *hdr, hipStream_t st, int st_top = 0, int st_bot = 0,
                 const double *cache = nullptr, const int64_t *chdr = nullptr,
                 const int32_t *parent = nullptr, const uint32_t *cmove = nullptr) {
  if (bm_wave_fits(g.D, g.cb)) {
    const auto kern = g.D == 2   ? peps_bmps_wave_kernel<2>
                      : g.D == 3 ? peps_bmps_wave_kernel<3>
                                 : peps_bmps_wave_kernel<4>;
    hipLaunchKernelGGL(kern, dim3((unsigned)n, 2), dim3(64), 0, st, g, n, c, f, slots, hdr,
                       st_top, st_bot, cache, chdr, parent, cmove);
  } else if (g.cb * g.D <= 32)
    hipLaunchKernelGGL(peps_bmps_side_kernel<32>, dim3((unsigned)n, 2), dim3(BT), 0, st, g, n,
                       c, f, slots, hdr, st_top, st_bot, cache, chdr, parent, cmove);
  else
    hipLaunchKernelGGL(peps_bmps_side_kernel<64>, dim3((unsigned)n, 2), dim3(BT), 0, st, g, n,
                       c, f, slots, hdr, st_top, st_bot, cache, chdr, parent, cmove);
}

// (sign, ln|psi|) of n configurations from the boundaries in buffers bt and bb; one wave
// each, on the matrix cores while the bonds fit one 16 x 16 tile
void launch_join(const BmGeo &g, int64_t n, const int64_t *c, const int32_t *f,
                 const double *slots, const int64_t *hdr, int bt, int bb, double *sign,
                 double *logabs, hipStream_t st, int ct = 0, int cb = 0,
                 const double *cache = nullptr, const int64_t *chdr = nullptr,
                 const int32_t *parent = nullptr, const uint32_t *cmove = nullptr) {
  const auto kern = g.cb > 16  ? peps_bmps_join_kernel
                    : g.D == 1 ? peps_bmps_join_wave_kernel<1>
                    : g.D == 2 ? peps_bmps_join_wave_kernel<2>
                    : g.D == 3 ? peps_bmps_join_wave_kernel<3>
                               : peps_bmps_join_wave_kernel<4>;
  hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3(64), 0, st, g, n, c, f, slots, hdr, bt, bb,
                     sign, logabs, ct, cb, cache, chdr, parent, cmove);
}
}  // namespace

const char *bmps_check(int Lx, int Ly, int D, int chi) {
  if (chi < 1 || chi > BMAX_CHI) return "max_bond (chi) must be 1..32";
  if (Lx < 2 || Lx > 16 || Ly < 1 || Ly > BMAX_LY || Lx * Ly > BMAX_NS)
    return "boundary MPS needs 2 <= Lx <= 16, 1 <= Ly <= 16, Lx * Ly <= 64";
  if (D < 1 || D > 4) return "D must be 1..4";
  const int cb = chi > D ? chi : D;
  if (cb * D > BN || cb * D * cb > BMAX_TS) return "max(chi, D) * D must be <= 64";
  return nullptr;
}

int64_t bmps_workspace_bytes(int Lx, int Ly, int D, int chi, int64_t rows) {
  const BmGeo g = bm_geo(Lx, Ly, D, chi, 1);
  return rows * 2 * (g.slot * 8 + BHDR * 8);
}

int64_t bmps_logderiv_workspace_bytes(int Lx, int Ly, int D, int chi, int64_t rows) {
  const BmGeo g = bm_geo(Lx, Ly, D, chi, Lx - 1);
  return rows * 2 * (g.slot * 8 + g.nbuf * BHDR * 8) +
         rows * Lx * ((int64_t)(Ly + 1) * g.ts + Ly + 1) * 8;
}

int bmps_amplitudes(int Lx, int Ly, int D, int chi, const int32_t *dmap, const double *theta,
                    int64_t theta_stride, int64_t rows, const int64_t *cfg, const int32_t *flag,
                    double *sign, double *logabs, void *ws, int64_t rows_per_pass,
                    hipStream_t st) {
  BmGeo g = bm_geo(Lx, Ly, D, chi, 1);
  g.dmap = dmap;
  double *slots = (double *)ws;
  int64_t *hdr = (int64_t *)(slots + rows_per_pass * 2 * g.slot);
  for (int64_t r0 = 0; r0 < rows; r0 += rows_per_pass) {
    const int64_t n = rows - r0 < rows_per_pass ? rows - r0 : rows_per_pass;
    g.theta = theta + r0 * theta_stride;
    g.theta_stride = theta_stride;
    const int64_t *c = cfg + r0 * g.N;
    const int32_t *f = flag ? flag + r0 : nullptr;
    launch_side(g, n, c, f, slots, hdr, st);
    VMCX_LAUNCHED();
    launch_join(g, n, c, f, slots, hdr, 0, 0, sign + r0, logabs + r0, st);
    VMCX_LAUNCHED();
  }
  return 0;
}

// ---- the sweep's boundary cache (plain fPEPS: the site tensors do not
// depend on the configuration).  Every walker keeps the boundary of each
// side after each of its rows (top: rows 0 .. h-1, bottom: Lx-1 .. h); a
// proposal on an edge between rows rmin <= rmax recomputes a side only
// from its first changed row on, starting from the walker's boundary before
// it, and takes an unchanged side from the cache as it is.  The arithmetic
// of a recomputed row is that of the full contraction on the same inputs, so
// the amplitudes equal the full recomputation's bit for bit.
namespace {
BmGeo bm_cache_geo(int Lx, int Ly, int D, int chi) {
  const int h = Lx / 2;
  return bm_geo(Lx, Ly, D, chi, h > Lx - h ? h : Lx - h, 1);
}
struct BmCacheWs {
  double *cache, *prop;
  int64_t *chdr, *phdr;
  int32_t *acc;
};
// slots for proposals and connected configurations: a launch of one wave per side needs
// some 8192 configurations to fill the chip (a walker has about as many connected
// configurations as edges), and its slots are small
int64_t bm_prop_rows(const BmGeo &g, int64_t B) {
  if (!bm_wave_fits(g.D, g.cb)) return B;
  const int64_t p = 8 * B < 8192 ? 8 * B : 8192;
  return p > B ? p : B;
}
BmCacheWs bm_cache_ws(const BmGeo &g, int64_t B, void *ws) {
  BmCacheWs c;
  const int64_t P = bm_prop_rows(g, B);
  c.cache = (double *)ws;
  c.prop = c.cache + B * 2 * g.slot;
  c.chdr = (int64_t *)(c.prop + P * 2 * g.slot);
  c.phdr = c.chdr + B * 2 * g.nbuf * BHDR;
  c.acc = (int32_t *)(c.phdr + P * 2 * g.nbuf * BHDR);
  return c;
}
}  // namespace

int64_t bmps_sweep_cache_bytes(int Lx, int Ly, int D, int chi, int64_t B) {
  const BmGeo g = bm_cache_geo(Lx, Ly, D, chi);
  return (B + bm_prop_rows(g, B)) * 2 * (g.slot + g.nbuf * BHDR) * 8 + B * 4;
}

int32_t *bmps_sweep_accept_flags(int Lx, int Ly, int D, int chi, int64_t B, void *ws) {
  return bm_cache_ws(bm_cache_geo(Lx, Ly, D, chi), B, ws).acc;
}

int bmps_sweep_init(int Lx, int Ly, int D, int chi, const int32_t *dmap, const double *theta,
                    int64_t B, const int64_t *cfg, void *ws, hipStream_t st) {
  BmGeo g = bm_cache_geo(Lx, Ly, D, chi);
  g.dmap = dmap;
  g.theta = theta;
  g.theta_stride = 0;
  const BmCacheWs c = bm_cache_ws(g, B, ws);
  launch_side(g, B, cfg, nullptr, c.cache, c.chdr, st);
  VMCX_LAUNCHED();
  return 0;
}

// the side steps an edge between rows r0 and r1 changes
static void bm_edge_starts(int Lx, int r0, int r1, int &st_top, int &st_bot) {
  const int h = Lx / 2;
  const int rmin = r0 < r1 ? r0 : r1, rmax = r0 < r1 ? r1 : r0;
  st_top = rmin <= h - 1 ? rmin : h;
  st_bot = rmax >= h ? Lx - 1 - rmax : Lx - h;
}

int bmps_sweep_amplitudes(int Lx, int Ly, int D, int chi, const int32_t *dmap,
                          const double *theta, int64_t B, const int64_t *pcfg,
                          const int32_t *flag, int r0, int r1, void *ws, double *sign,
                          double *logabs, hipStream_t st) {
  BmGeo g = bm_cache_geo(Lx, Ly, D, chi);
  g.dmap = dmap;
  g.theta = theta;
  g.theta_stride = 0;
  const BmCacheWs c = bm_cache_ws(g, B, ws);
  int st_top, st_bot;
  bm_edge_starts(Lx, r0, r1, st_top, st_bot);
  const int h = Lx / 2;
  launch_side(g, B, pcfg, flag, c.prop, c.phdr, st, st_top, st_bot, c.cache, c.chdr);
  VMCX_LAUNCHED();
  launch_join(g, B, pcfg, flag, c.prop, c.phdr, h - 1, Lx - h - 1, sign, logabs, st,
              st_top >= h ? 1 : 0, st_bot >= Lx - h ? 1 : 0, c.cache, c.chdr);
  VMCX_LAUNCHED();
  return 0;
}

// amplitudes of T connected configurations, each one move (cmove) away from
// its walker cparent, from the walkers' cached boundaries (bmps_sweep_init
// of the walkers first), in passes through the proposal slots
int bmps_conn_amplitudes(int Lx, int Ly, int D, int chi, const int32_t *dmap,
                         const double *theta, int64_t B, int64_t T, const int64_t *etas,
                         const int32_t *cparent, const uint32_t *cmove, void *ws, double *sign,
                         double *logabs, hipStream_t st) {
  BmGeo g = bm_cache_geo(Lx, Ly, D, chi);
  g.dmap = dmap;
  g.theta = theta;
  g.theta_stride = 0;
  const BmCacheWs c = bm_cache_ws(g, B, ws);
  const int h = Lx / 2;
  const int64_t P = bm_prop_rows(g, B);
  for (int64_t r0 = 0; r0 < T; r0 += P) {
    const int64_t n = T - r0 < P ? T - r0 : P;
    const int64_t *e = etas + r0 * g.N;
    launch_side(g, n, e, nullptr, c.prop, c.phdr, st, 0, 0, c.cache, c.chdr, cparent + r0,
                cmove + r0);
    VMCX_LAUNCHED();
    launch_join(g, n, e, nullptr, c.prop, c.phdr, h - 1, Lx - h - 1, sign + r0, logabs + r0, st,
                0, 0, c.cache, c.chdr, cparent + r0, cmove + r0);
    VMCX_LAUNCHED();
  }
  return 0;
}

int bmps_sweep_commit(int Lx, int Ly, int D, int chi, int64_t B, int r0, int r1, void *ws,
                      hipStream_t st) {
  const BmGeo g = bm_cache_geo(Lx, Ly, D, chi);
  const BmCacheWs c = bm_cache_ws(g, B, ws);
  int st_top, st_bot;
  bm_edge_starts(Lx, r0, r1, st_top, st_bot);
  hipLaunchKernelGGL(bm_commit_kernel, dim3((unsigned)B, 2), dim3(256), 0, st, g, B, c.acc,
                     st_top, st_bot, c.prop, c.phdr, c.cache, c.chdr);
  VMCX_LAUNCHED();
  return 0;
}

int bmps_logderiv(int Lx, int Ly, int D, int chi, const int32_t *dmap, const double *theta,
                  int64_t theta_stride, int64_t n_params, int64_t rows, const int64_t *cfg,
                  double *G, int64_t ldg, double *sign, double *logabs, void *ws,
                  int64_t rows_per_pass, hipStream_t st) {
  BmGeo g = bm_geo(Lx, Ly, D, chi, Lx - 1);
  g.dmap = dmap;
  double *slots = (double *)ws;
  int64_t *hdr = (int64_t *)(slots + rows_per_pass * 2 * g.slot);
  double *renv = (double *)(hdr + rows_per_pass * 2 * g.nbuf * BHDR);
  const int h = Lx / 2;
  for (int64_t r0 = 0; r0 < rows; r0 += rows_per_pass) {
    const int64_t n = rows - r0 < rows_per_pass ? rows - r0 : rows_per_pass;
    g.theta = theta + r0 * theta_stride;
    g.theta_stride = theta_stride;
    const int64_t *c = cfg + r0 * g.N;
    double *Gr = G + r0 * ldg;
    launch_side(g, n, c, nullptr, slots, hdr, st);
    VMCX_LAUNCHED();
    launch_join(g, n, c, nullptr, slots, hdr, h - 1, Lx - h - 1, sign + r0, logabs + r0, st);
    VMCX_LAUNCHED();
    const int64_t nz = n * n_params;
    const unsigned gz = (unsigned)((nz + 255) / 256 < 16384 ? (nz + 255) / 256 : 16384);
    hipLaunchKernelGGL(bm_zero_rows_kernel, dim3(gz), dim3(256), 0, st, n, n_params, Gr, ldg);
    VMCX_LAUNCHED();
    hipLaunchKernelGGL(peps_bmps_grad_kernel, dim3((unsigned)n, (unsigned)Lx), dim3(BT), 0, st,
                       g, n, c, nullptr, slots, hdr, sign + r0, logabs + r0, renv, Gr, ldg);
    VMCX_LAUNCHED();
  }
  return 0;
}

}  // namespace vmcx
