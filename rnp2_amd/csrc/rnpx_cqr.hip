// rnpx_cqr.hip -- panel factorization by CholeskyQR2 with Householder
// reconstruction, for real panels of 64 columns.
//
// The column-by-column panel (rnpx_panel.hip) needs one grid-wide reduction
// per column.  This kernel needs two grid-wide reductions per panel:
//
//   1. Q1 R1 = A     (CholeskyQR: Gram A^T A over the grid, Cholesky, A R1^-1)
//   2. Q  R2 = Q1    (the second pass restores orthogonality to working
//                     precision when the first pass was accurate enough)
//   3. Householder reconstruction: Q - [D; 0] = Y U (LU without pivoting,
//      D = diag(+-1) chosen column by column), so that
//        Y = the Householder vectors V (unit lower trapezoidal),
//        tau_j = -U_jj D_j,  T = -U D Y1^-T,  R_householder = D R2 R1.
//
// In exact arithmetic this is the factorization the column-by-column
// reflectors produce (RNP/LA/QR.hpp:78-102 with Reflector::Generate,
// RNP/LA/Reflector.hpp:117-158): with the panel's Householder form
// H = I - Y T Y^T, H [I; 0] = Q D, hence Q D - [I; 0] = -Y T Y1^T, an LU
// factorization with a unit lower factor.  The sign D_j = -sign of the
// running pivot makes |U_jj| = tau_j in [1, 2] and matches Generate's
// choice beta_j = -sign(alpha_j) |.|; a zero pivot takes D_j = +1, the
// reference's beta > 0 when real(alpha) == 0 (Reflector.hpp:131).
//
// The second pass's Gram G2 = Q1^T Q1 = I + E is within 2^-27 of I or the
// panel is rejected.  When |E| <= 2^-40 its Cholesky factor is taken to
// first order, R2 = I + E_U with E_U = triu(E) - diag(E)/2, and
// R2^-1 = I - E_U (both exact to O(|E|^2) <= 2^-68); otherwise it is
// factored.
//
// The panel is refactored column by column instead (by workgroup 0, inside
// the same launch; the fail flag records it) when the first Cholesky meets a
// pivot below 2^-40 of its diagonal entry, a column whose squared norm is
// outside [2^-600, 2^600] (so the Gram entries cannot under/overflow), a
// non-finite value, or the second pass's test above fails.  Every workgroup
// takes the same decision from the same reduced Gram.
//
// Layout: G workgroups of 256 threads; workgroup g stages rows
// [g*RW, (g+1)*RW) of the panel in LDS (row-major, padded), so the panel is
// read from HBM once and written once.  Gram partials use FP64 MFMA over the
// 10 upper 16x16 tiles; they are summed in groups of 16 workgroups by the
// last workgroup of each group to arrive, then across groups by the last
// group, always in workgroup order (deterministic); everybody else waits on
// a done flag.  The 64x64 Cholesky, triangular inverses and the LU run in
// 16x16 diagonal blocks (one wave each step, v_readlane broadcasts) with the
// off-diagonal blocks as MFMA block products over the four waves
// (rnpx_small64.hpp); workgroup 0 does the LU and publishes U^-1, workgroup 1
// forms R, one more workgroup forms T.
#include "rnpx_kernels.hpp"
#include "rnpx_small64.hpp"
#include "rnpx_team.hpp"

#include <algorithm>
#include <cstdlib>

namespace rnpx {

namespace {

constexpr int NB = 64;
constexpr int LDA_S = NB + 1;  // padded LDS row stride (doubles)
constexpr int kTiles = 10;     // upper 16x16 tiles of a 64x64 symmetric matrix
constexpr int kGramElems = kTiles * 256;
constexpr int kGroup = 16;     // workgroups per first-level reduction group
constexpr double kFirstOrder = 0x1p-40;
constexpr double kSecondPass = 0x1p-27;
// sync words: [pass*32 + grp] group arrivals, [pass*32 + 16] group-leader
// arrivals, [pass*32 + 17] done flag; [64] U^-1 published.
constexpr int kSyncTop = 16, kSyncDone = 17, kSyncPub = 64;

__device__ __forceinline__ void tile_of(int t, int& ti, int& tj) {
  // (0,0) (0,1) (0,2) (0,3) (1,1) (1,2) (1,3) (2,2) (2,3) (3,3)
  ti = (t >= 4) + (t >= 7) + (t >= 9);
  const int first = (ti == 0) ? 0 : (ti == 1) ? 4 : (ti == 2) ? 7 : 9;
  tj = ti + (t - first);
}

// Partial Gram P = Ab^T Ab of this workgroup's RW rows; tile t of the 10 is
// written row-major (16x16) to out[t*256 ...].
template <int RW>
__device__ __forceinline__ void gram_partial(const double (*Ab)[LDA_S], double* out, int lane, int wave) {
  const int t0 = (wave == 0) ? 0 : (wave == 1) ? 3 : (wave == 2) ? 6 : 8;  // 3, 3, 2, 2 tiles
  const int nt = (wave < 2) ? 3 : 2;
  for (int q = 0; q < nt; ++q) {
    int ti, tj;
    tile_of(t0 + q, ti, tj);
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int k0 = 0; k0 < RW; k0 += 4) {
      const double x = Ab[k0 + (lane >> 4)][16 * ti + (lane & 15)];
      const double y = Ab[k0 + (lane >> 4)][16 * tj + (lane & 15)];
      acc = mfma16(x, y, acc);
    }
    // item r = P[16 ti + lane/16 + 4r][16 tj + lane%16]
#pragma unroll
    for (int r = 0; r < 4; ++r) out[(t0 + q) * 256 + ((lane >> 4) + 4 * r) * 16 + (lane & 15)] = acc[r];
  }
}

// Sum of partials src[w * kGramElems + e], w = 0..n-1 (n <= 16), in order.
// Thread tid owns the entry pairs 2 tid + 512 q; eight partials' loads are
// in flight at once.
template <int ELEMS = kGramElems, int STRIDE = ELEMS>
__device__ __forceinline__ void sum_partials(const double* src, int n, double* dst, int tid) {
  constexpr int Q = ELEMS / 512;  // pairs per thread
  constexpr int W = 8;                 // partials per batch
  double2 acc[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) acc[q] = make_double2(0.0, 0.0);
  for (int w0 = 0; w0 < n; w0 += W) {
    double2 v[W][Q];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const double2* p = reinterpret_cast<const double2*>(src + (size_t)(w0 + w) * STRIDE) + tid;
#pragma unroll
      for (int q = 0; q < Q; ++q) v[w][q] = (w0 + w < n) ? p[256 * q] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int w = 0; w < W; ++w)
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (w0 + w < n) {
          acc[q].x += v[w][q].x;
          acc[q].y += v[w][q].y;
        }
  }
  double2* d = reinterpret_cast<double2*>(dst) + tid;
#pragma unroll
  for (int q = 0; q < Q; ++q) d[256 * q] = acc[q];
}

// After this workgroup's partial is in part[g]: the reduced Gram of the
// pass lands in gs for every workgroup.
__device__ __forceinline__ void gram_allreduce(const CqrArgs& a, int pass, int G, int g, int tid, unsigned* slot) {
  unsigned* sw = a.sync + pass * 32;
  double* gs = a.gsum + pass * kGramElems;
  const int grp = g / kGroup, ngroups = (G + kGroup - 1) / kGroup;
  const int gbeg = grp * kGroup, gsize = min(kGroup, G - gbeg);
  if (arrive(&sw[grp], slot) == (unsigned)(gsize - 1)) {
    // last of its group
    if (ngroups == 1) {
      sum_partials(a.part, gsize, gs, tid);
      publish(&sw[kSyncDone]);
    } else {
      sum_partials(a.part + (size_t)gbeg * kGramElems, gsize, a.gpart + (size_t)grp * kGramElems, tid);
      if (arrive(&sw[kSyncTop], slot) == (unsigned)(ngroups - 1)) {
        sum_partials(a.gpart, ngroups, gs, tid);
        publish(&sw[kSyncDone]);
      }
    }
  }
  wait_flag(&sw[kSyncDone], a.abortf);
}

// Load the reduced symmetric Gram into M (full 64x64).  Here and in the
// other global-to-LDS copies every load is issued before the first LDS
// store, so that the loads' round trips overlap.
__device__ __forceinline__ void load_gram(const double* gs, double (*M)[LDA_S], int tid) {
  constexpr int Q = kGramElems / 256;
  double v[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) v[q] = gs[tid + 256 * q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int e = tid + 256 * q;
    const int t = e >> 8, r = (e >> 4) & 15, c = e & 15;
    int ti, tj;
    tile_of(t, ti, tj);
    if (ti == tj && r > c) continue;  // one writer per entry of a diagonal tile
    M[16 * ti + r][16 * tj + c] = v[q];
    M[16 * tj + c][16 * ti + r] = v[q];
  }
}

// M := the row-major 64x64 block at src (global memory).
__device__ __forceinline__ void load64(const double* src, double (*M)[LDA_S], int tid) {
  constexpr int Q = NB * NB / 256;
  double v[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) v[q] = src[tid + 256 * q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int e = tid + 256 * q;
    M[e / NB][e % NB] = v[q];
  }
}

// Rows [0, RW) of Ab := Ab * X for an upper triangular X (64x64) on MFMA;
// Ab is overwritten after every wave has read its operands.
template <int RW>
__device__ __forceinline__ void times_upper(double (*Ab)[LDA_S], const double (*X)[LDA_S], int lane, int wave) {
  constexpr int RT = RW / 64;  // row tiles per wave
  f64x4 acc[RT][4];
#pragma unroll
  for (int q = 0; q < RT; ++q) {
    const int t = wave + 4 * q;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[q][c] = f64x4{0.0, 0.0, 0.0, 0.0};
    // the reduction outside, a step's four columns' MFMAs independent of one
    // another
#pragma unroll
    for (int k0 = 0; k0 < 64; k0 += 4) {
      const double x = Ab[16 * t + (lane & 15)][k0 + (lane >> 4)];
#pragma unroll
      for (int c = k0 / 16; c < 4; ++c)  // X[k][16c..] = 0 for k >= 16(c+1)
        acc[q][c] = mfma16(x, X[k0 + (lane >> 4)][16 * c + (lane & 15)], acc[q][c]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < RT; ++q) {
    const int t = wave + 4 * q;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) Ab[16 * t + (lane >> 4) + 4 * r][16 * c + (lane & 15)] = acc[q][c][r];
  }
  __syncthreads();
}

// Wave w's tile row of C = A B for 64x64 upper triangular A, B (row-major in
// LDS; entries of A below its diagonal are treated as zero when mask_a, and
// column k of A is scaled by dcol[k] when dcol is given):
// acc[tj] item r = C[16 w + lane/16 + 4r][16 tj + lane%16].
template <bool TB = false>  // TB: B is given transposed (B[k][j] read as B[j][k])
__device__ __forceinline__ void upper_product_row(const double (*A)[LDA_S], const double (*B)[LDA_S], bool mask_a, const double* dcol,
                                  f64x4 (&acc)[4], int lane, int wave) {
  const int ti = wave;
#pragma unroll
  for (int tj = 0; tj < 4; ++tj) acc[tj] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    // (A's blocks left of its diagonal count as zero)
#pragma unroll
    for (int k0 = 16 * kb; k0 < 16 * kb + 16; k0 += 4) {
      const int i = 16 * ti + (lane & 15), k = k0 + (lane >> 4);
      double x = A[i][k];
      if (kb < ti || (mask_a && k < i)) x = 0.0;
      if (dcol) x *= dcol[k];
#pragma unroll
      for (int tj = kb; tj < 4; ++tj)
        acc[tj] = mfma16(x, TB ? B[16 * tj + (lane & 15)][k] : B[k][16 * tj + (lane & 15)], acc[tj]);
    }
  }
}

// Largest |M - I| over the workgroup (a NaN entry makes the result NaN).
__device__ __forceinline__ double dev_from_identity(const double (*M)[LDA_S], double* red4, int tid) {
  double d = 0.0;
  for (int e = tid; e < NB * NB; e += 256) {
    const int i = e / NB, j = e % NB;
    const double x = fabs(M[i][j] - (i == j ? 1.0 : 0.0));
    d = (x > d || x != x) ? x : d;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const double o = __shfl_xor(d, off, 64);
    d = (o > d || o != o) ? o : d;
  }
  if ((tid & 63) == 0) red4[tid >> 6] = d;
  __syncthreads();
  double r = red4[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) r = (red4[w] > r || red4[w] != red4[w]) ? red4[w] : r;
  __syncthreads();
  return r;
}

// The column-by-column refactorization of a rejected panel, by one
// workgroup after every other has left the kernel: team_factor
// (Reflector::Generate's rules, RNP/LA/Reflector.hpp:117-158, and the
// Householder application of QR::Factor_unblocked, QR.hpp:78-102) in place,
// the clean V, then T from V's Gram (GenerateBlockTr("F","C"),
// Reflector.hpp:580-626): T(c,c) = tau_c, T(0:c,c) = -tau_c T(0:c,0:c)
// V(:,0:c)^T v_c.  Column-serial, so slow, but rejections are rare.  No
// workgroup reads A after staging its rows, so rewriting A here is safe.
__device__ void refactor_columnwise(const CqrArgs& a, double (*Gs)[LDA_S], double (*Ts)[LDA_S], double* sh, int tid) {
  if (tid == 0) *a.fail = 1u;
  const int mp = a.mp;
  team_factor<double, 256, true>(mp, NB, a.A, (int)a.lda, a.tau, sh);
  __syncthreads();
  for (long e = tid; e < (long)mp * NB; e += 256) {
    const int r = (int)(e % mp), c = (int)(e / mp);
    a.V[(size_t)r + (size_t)c * a.ldv] = (r > c) ? a.A[(size_t)r + (size_t)c * a.lda] : (r == c ? 1.0 : 0.0);
  }
  __syncthreads();
  for (int e = tid; e < NB * NB; e += 256) {
    const int l = e / NB, c = e % NB;
    double gv = 0.0;
    if (l < c)
      for (int r = c; r < mp; ++r) gv = fma(a.V[(size_t)r + (size_t)l * a.ldv], a.V[(size_t)r + (size_t)c * a.ldv], gv);
    Gs[l][c] = gv;
    Ts[l][c] = 0.0;
  }
  __syncthreads();
  for (int c = 0; c < NB; ++c) {
    const double tc = a.tau[c];
    if (tid < c) {
      double sacc = 0.0;
      for (int l = tid; l < c; ++l) sacc = fma(Ts[tid][l], Gs[l][c], sacc);
      Ts[tid][c] = -tc * sacc;
    }
    if (tid == c) Ts[c][c] = tc;
    __syncthreads();
  }
  for (int e = tid; e < NB * NB; e += 256) {
    const int i = e % NB, j = e / NB;
    a.T[(size_t)i + (size_t)j * a.ldt] = Ts[i][j];
  }
}

}  // namespace

template <int RW>
__global__ __launch_bounds__(256) void cqr_panel_kernel(CqrArgs a) {
  __shared__ double Ab[RW][LDA_S];
  __shared__ double M1[NB][LDA_S];
  __shared__ double M2[NB][LDA_S];
  __shared__ double rowbuf[NB];
  __shared__ double red4[4];
  __shared__ double gdiag[NB];
  __shared__ double tmpb[small64::kTmpDoubles];
  __shared__ unsigned slot;
  __shared__ int okf;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = blockIdx.x, G = gridDim.x;
  const int r0 = g * RW;
  const int mp = a.mp;
  double* rsave = a.scratch;          // R1 (saved and used by workgroup 1)
  double* uinv = a.scratch + 4096;    // U^-1
  double* ulp = a.scratch + 8192;     // U and L packed
  double* dpub = a.scratch + 12288;   // D
  const int tgrp = (G > 2) ? 2 : 1;   // the workgroup that forms T

  // Stage this workgroup's rows (coalesced down each column), zero padding.
  {
    constexpr int PER = RW * NB / 256;
    double v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = tid + 256 * q, r = e % RW, c = e / RW;
      v[q] = (r0 + r < mp) ? a.A[(size_t)(r0 + r) + (size_t)c * a.lda] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = tid + 256 * q;
      Ab[e % RW][e / RW] = v[q];
    }
  }
  __syncthreads();

  // Pass 1: Q1 = A R1^-1.
  gram_partial<RW>(Ab, a.part + (size_t)g * kGramElems, lane, wave);
  gram_allreduce(a, 0, G, g, tid, &slot);
  load_gram(a.gsum, M1, tid);
  __syncthreads();
  if (tid < NB) gdiag[tid] = M1[tid][tid];
  const bool ok1 = small64::chol64<LDA_S>(&M1[0][0], &M2[0][0], tmpb, gdiag, &okf, tid);  // M1 = R1, M2 = R1^-1
  if (!ok1) {
    // Every workgroup factored the same Gram and takes this branch; nothing
    // of the panel has been written.
    if (g == 0) refactor_columnwise(a, M1, M2, rowbuf, tid);
    return;
  }
  if (g == 1)
    for (int e = tid; e < NB * NB; e += 256) rsave[e] = M1[e / NB][e % NB];
  times_upper<RW>(Ab, M2, lane, wave);

  // Pass 2: Q = Q1 R2^-1.
  gram_partial<RW>(Ab, a.part + (size_t)g * kGramElems, lane, wave);
  gram_allreduce(a, 1, G, g, tid, &slot);
  load_gram(a.gsum + kGramElems, M1, tid);
  __syncthreads();
  const double dev = dev_from_identity(M1, red4, tid);
  if (!(dev <= kSecondPass)) {
    if (g == 0) refactor_columnwise(a, M1, M2, rowbuf, tid);
    return;
  }
  if (dev <= kFirstOrder) {
    for (int e = tid; e < NB * NB; e += 256) {
      const int i = e / NB, j = e % NB;
      const double E = M1[i][j] - (i == j ? 1.0 : 0.0);
      const double eu = (i < j) ? E : ((i == j) ? 0.5 * E : 0.0);
      M1[i][j] = (i == j ? 1.0 : 0.0) + eu;  // R2
      M2[i][j] = (i == j ? 1.0 : 0.0) - eu;  // R2^-1
    }
    __syncthreads();
  } else {
    if (tid < NB) gdiag[tid] = M1[tid][tid];
    small64::chol64<LDA_S>(&M1[0][0], &M2[0][0], tmpb, gdiag, &okf, tid);
  }
  times_upper<RW>(Ab, M2, lane, wave);
  // Ab = Q (this workgroup's rows), M1 = R2.

  if (g == 0) {
    // LU of Q_top - D, published with U^-1.
    for (int e = tid; e < NB * NB; e += 256) M1[e / NB][e % NB] = Ab[e / NB][e % NB];
    __syncthreads();
    small64::lu64<LDA_S>(&M1[0][0], rowbuf, &M2[0][0], tmpb, &okf, tid);  // M1 = U and L, M2 = U^-1
    for (int e = tid; e < NB * NB; e += 256) {
      ulp[e] = M1[e / NB][e % NB];
      uinv[e] = M2[e / NB][e % NB];
    }
    if (tid < NB) dpub[tid] = rowbuf[tid];
    publish(&a.sync[kSyncPub]);
    // Rows 64..RW-1 of this workgroup: Y = Q U^-1.
    if constexpr (RW > NB) {
      __syncthreads();
      times_upper<RW>(Ab, M2, lane, wave);
      for (int e = tid; e < (RW - NB) * NB; e += 256) {
        const int r = NB + e % (RW - NB), c = e / (RW - NB);
        const int gr = r0 + r;
        if (gr < mp) {
          const double v = Ab[r][c];
          a.A[(size_t)gr + (size_t)c * a.lda] = v;
          a.V[(size_t)gr + (size_t)c * a.ldv] = v;
        }
      }
    }
    // Top block: L below the diagonal (R above is written by workgroup 1),
    // V's unit lower block, tau.
    for (int e = tid; e < NB * NB; e += 256) {
      const int i = e % NB, j = e / NB;
      const double l = M1[i][j];
      if (i > j) a.A[(size_t)i + (size_t)j * a.lda] = l;
      a.V[(size_t)i + (size_t)j * a.ldv] = (i == j) ? 1.0 : ((i > j) ? l : 0.0);
    }
    if (tid < NB) a.tau[tid] = -M1[tid][tid] * rowbuf[tid];
    return;
  }

  f64x4 racc[4];
  if (g == 1) {
    // R = R2 R1 while workgroup 0 reconstructs.
    for (int e = tid; e < NB * NB; e += 256) M2[e / NB][e % NB] = rsave[e];
    __syncthreads();
    upper_product_row(M1, M2, false, nullptr, racc, lane, wave);
  }
  wait_flag(&a.sync[kSyncPub], a.abortf);
  if (g == 1) {
    // R_householder = D R, the upper triangle of the top block.
#pragma unroll
    for (int tj = 0; tj < 4; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * wave + (lane >> 4) + 4 * r, j = 16 * tj + (lane & 15);
        if (i <= j) a.A[(size_t)i + (size_t)j * a.lda] = dpub[i] * racc[tj][r];
      }
  }
  // Y = Q U^-1 for this workgroup's rows.
  __syncthreads();
  for (int e = tid; e < NB * NB; e += 256) M2[e / NB][e % NB] = uinv[e];
  __syncthreads();
  times_upper<RW>(Ab, M2, lane, wave);
  for (int e = tid; e < RW * NB; e += 256) {
    const int r = e % RW, c = e / RW;
    const int gr = r0 + r;
    if (gr < mp) {
      const double v = Ab[r][c];
      a.A[(size_t)gr + (size_t)c * a.lda] = v;
      a.V[(size_t)gr + (size_t)c * a.ldv] = v;
    }
  }
  if (g == tgrp) {
    // T = -U D Z^T with Z = L^-1.
    for (int e = tid; e < NB * NB; e += 256) M1[e / NB][e % NB] = ulp[e];
    if (tid < NB) rowbuf[tid] = dpub[tid];
    __syncthreads();
    small64::inv_unit_lower64<LDA_S>(&M1[0][0], &M2[0][0], tmpb, tid);  // M2 = L^-1 (lower blocks)
    // Z^T is upper: stage it transposed in Ab's top rows.
    for (int e = tid; e < NB * NB; e += 256) Ab[e % NB][e / NB] = M2[e / NB][e % NB];
    __syncthreads();
    f64x4 tacc[4];
    upper_product_row(M1, Ab, true, rowbuf, tacc, lane, wave);
#pragma unroll
    for (int tj = 0; tj < 4; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * wave + (lane >> 4) + 4 * r, j = 16 * tj + (lane & 15);
        a.T[(size_t)i + (size_t)j * a.ldt] = (i <= j) ? -tacc[tj][r] : 0.0;
      }
  }
}

// ---------------------------------------------------------------------------
// One outer block of up to 128 columns in one launch, by CholeskyQR2 of all
// its columns at once and Householder reconstruction in two 64-column halves
// (one when w <= 64).  Workgroup g holds rows [64 g, 64 g + 64) of both halves
// in LDS; columns beyond w and rows beyond mp are zero (their Gram diagonal is
// taken as one), so any width and height of a factorization's end runs here.
//   1. The Gram of the block [A1 A2] by one grid reduction; every workgroup
//      factors it itself: R11 = chol(G11), R12 = R11^-T G12,
//      R22 = chol(G22 - R12^T R12); Q1 = A1 R11^-1, Q2 = (A2 - Q1 R12) R22^-1.
//   2. The Gram I + E of [Q1 Q2] by a second reduction.  |E| <= 2^-40: first
//      order, R = I + triu(E) - diag(E)/2 (exact to |E|^2).  |E| <= 2^-27:
//      factored as in 1, which leaves Q orthonormal to working precision.
//      |E| <= 2^-3: factored, and the Gram taken again (a block of condition
//      up to about 1e7; CholeskyQR iterated).  Otherwise the block is
//      rejected, as it is when a pivot falls below 2^-40 of its column's
//      squared norm, a squared norm is outside [2^-600, 2^600] or a value is
//      not finite.  A pivot of the second half may fall that low because its
//      columns lie near the first half's span (collinear regressors), which
//      says nothing about their part outside it: A2 - Q1 R12 then goes into the
//      next pass as it is (R22 = I), up to twice (what is left along Q1 after one
//      projection, the first half's loss of orthogonality, can still be the
//      larger part), and is held against its own norms there.  Every workgroup takes the same decision from the same
//      reduced Gram, and A is untouched until the block is accepted; a rejected
//      block is refactored column by column (blk_columnwise).
//   3. Reconstruction [Q1 Q2] - [D; 0] = L U without another reduction:
//      workgroup 0 factors Q1's top block (L11, U11, D1) and forms
//      U12 = L11^-1 Q2(0:64), everybody V1 = Q1 U11^-1 and Q2 - V1 U12,
//      workgroup 1 factors that one's rows 64..127 (L22, U22, D2), everybody
//      V2 = (Q2 - V1 U12) U22^-1.  tau_j = -U_jj D_j,
//      T = -U D L^-T: T11 = -U11 D1 L11^-T, T22 = -U22 D2 L22^-T and
//      T12 = -(T11 L21^T + U12 D2) L22^-T with L21 = V1(64:128).
//      R = D times the product of the passes' factors, by workgroup 2 beside
//      the two LUs.
// In a square last block (mp == w) the last column has no entries below it and
// so no reflector (tau = 0, Reflector.hpp:122-125): there D takes the running
// pivot's own sign and T's column is zero.  Any other column whose entries
// below the diagonal are exactly zero has no reflector either, which the
// reconstruction cannot tell from tiny entries (both give tau = 2 to rounding):
// in the halves named by zero_tails such a running pivot (within 2^-40 of one)
// rejects the block.
// Bound by the chain of two grid reductions, two Cholesky and two LU
// factorizations of 64 x 64: 168 us per block at 1931 rows and below, 275 at
// 16384; 1931 x 1207 factors in 2.18 ms, 8192^2 in 26.4, 100 x 100 in 0.24.  Two
// 64-column panels joined inside the launch (six reductions, the second panel's
// Gram after the first one's reconstruction; 370 KB of unrolled code where this is
// 96 KB, most of it cold in the instruction cache) and ragged ends column by
// column take 201 us, 2.70, 29.4 and 0.55 ms.
// ---------------------------------------------------------------------------
namespace {

constexpr int kBlkMarkWords = 64;                  // a byte per workgroup (grid_step)
constexpr int kBlkPub1 = 192;                      // LU of the first half published
static_assert(4 * kBlkMarkWords == 16 * kGroup && kBlkMarkWords <= kBlkPub1, "block marks");
constexpr int kBlkPubU12 = kBlkPub1 + 1;           // U12 published
constexpr int kBlkPubT1 = kBlkPub1 + 2;            // T11 published
constexpr int kBlkPub2 = kBlkPub1 + 3;             // LU of the second half published
constexpr int kBlkResident = kBlkPub1 + 4;         // workgroups started (for the gate below)
static_assert(kBlkResident < kCqrBlockSyncWords, "block sync words");
constexpr int kCross = 16 * 256;                   // a 64x64 product in 16 tiles
constexpr int kBlkElems = kCqrBlockPart;           // upper tiles of a 128x128 Gram: G11, G12, G22
static_assert(2 * kGramElems + kCross == kBlkElems, "Gram layout: tiles 0..9, 10..25, 26..35");
constexpr int kBlkPasses = blk::kPasses;
// a second half may be projected without being normalized in the passes before
// this one (two passes are left to normalize it and to see that it is)
constexpr int kBlkProject = kBlkPasses - 2;
constexpr double kThirdPass = 0x1p-3;
constexpr unsigned kRejected = 2u;                 // flag value: the block goes column by column
constexpr int kBR = blk::kR, kBU1i = blk::kU1i, kBU12 = blk::kU12, kBT1 = blk::kT1, kBU2i = blk::kU2i,
              kBD1 = blk::kD1, kBD2 = blk::kD2, kBG = blk::kGram, kBTF = blk::kTFactor,
              kBRow = blk::kRow;

// wait_flag, and the flag's value in every thread.
__device__ __forceinline__ unsigned wait_verdict(unsigned* flag, unsigned* abortf, unsigned* slot) {
  wait_flag(flag, abortf);
  if (threadIdx.x == 0) *slot = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const unsigned v = *slot;
  __syncthreads();
  return v;
}

// A double on its way to other workgroups: written through, so no cache
// write-back is needed before the mark that says it is there.
__device__ __forceinline__ void store_through(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Grid-wide step `step` (1, 2, ...): workgroup g marks its byte once all its
// store_through()s have arrived, then waits until every workgroup's byte says
// `step`.  A byte each, not a counter: 256 additions to one word take 13 us and
// more, one after the other, and the write-back of a release as long again.
__device__ __forceinline__ void grid_step(const CqrBlockArgs& a, int step, int g, int G, int tid) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  if (tid < 64) {
    unsigned char* marks = reinterpret_cast<unsigned char*>(a.sync);
    if (tid == 0) __hip_atomic_store(marks + g, (unsigned char)step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t t0 = wall_clock64();
    for (;;) {
      const unsigned v = __hip_atomic_load(a.sync + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      bool there = true;
#pragma unroll
      for (int b = 0; b < 4; ++b) there = there && (4 * tid + b >= G || ((v >> (8 * b)) & 255u) >= (unsigned)step);
      if (__ballot(!there) == 0) break;
      if (__hip_atomic_load(a.abortf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) break;
      if (wall_clock64() - t0 > kBarrierTimeoutTicks) {
        __hip_atomic_store(a.abortf, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
}

// Reduction of G partials (elems doubles each, kBlkElems apart from a.part)
// into gs, by reduce-scatter.  Once every workgroup has stored its partial, each
// sums its slice of the entries over the partials in a fixed order (so the result
// does not depend on timing) and stores it; the sum is complete at the second
// grid-wide step.  red: 512 doubles of LDS scratch.  With counters and agent-scope
// releases a reduction takes 10 us at 64 workgroups, 21 at 128 and 38 at 256; with
// marks and stores written through the 256-workgroup block (16384 rows) is 28 us
// faster in all (least squares 16384 x 2048: 8.46 ms against 8.92).
__device__ __forceinline__ void blk_allreduce(const CqrBlockArgs& a, int elems, int pass, int g, int G, double* gs,
                                              double* red, int tid) {
  grid_step(a, 2 * pass + 1, g, G, tid);
  // the slice in pairs; P threads per pair, each over every P-th partial, 16
  // partials' loads in flight; then the P sums
  const int S = (elems / 2 + G - 1) / G, e0 = g * S, len = max(0, min(S, elems / 2 - e0));
  const int P = max(1, 256 / S), j = min(tid / S, P);
  for (int x0 = 0; x0 < len; x0 += 256) {
    const int x = x0 + (P > 1 ? tid - j * S : tid);
    double2 sum = {0.0, 0.0};
    if (x < len && (P == 1 || j < P)) {
      const double2* src = reinterpret_cast<const double2*>(a.part) + e0 + x;
      for (int q0 = (P > 1 ? j : 0); q0 < G; q0 += 16 * P) {
        double2 v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = src[(size_t)min(q0 + u * P, G - 1) * (kBlkElems / 2)];
#pragma unroll
        for (int u = 0; u < 16; ++u)
          if (q0 + u * P < G) {
            sum.x += v[u].x;
            sum.y += v[u].y;
          }
      }
    }
    double2* out = reinterpret_cast<double2*>(gs) + e0;
    if (P == 1) {
      if (x < len) {
        store_through(&out[x].x, sum.x);
        store_through(&out[x].y, sum.y);
      }
    } else {
      red[2 * tid] = sum.x;
      red[2 * tid + 1] = sum.y;
      __syncthreads();
      if (tid < len) {
        for (int q = 1; q < P; ++q) {
          sum.x += red[2 * (q * S + tid)];
          sum.y += red[2 * (q * S + tid) + 1];
        }
        store_through(&out[tid].x, sum.x);
        store_through(&out[tid].y, sum.y);
      }
    }
  }
  grid_step(a, 2 * pass + 2, g, G, tid);
}

// This workgroup's partial Gram over its 64 rows: the 10 upper tiles of
// X^T X, and for two halves the 16 of X^T Y and the 10 upper of Y^T Y.
__device__ __forceinline__ void blk_gram(const double (*X)[LDA_S], const double (*Y)[LDA_S], bool two, double* out,
                                         int lane, int wave) {
  // Three tiles at a time per wave (their MFMAs independent of one another),
  // every fourth tile from `wave` on; past the end, the last tile again.
  const int nt = two ? 36 : 10;
#pragma unroll 1
  for (int t0 = wave; t0 < nt; t0 += 12) {
    const double *xp[3], *yp[3];
    f64x4 acc[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int t = min(t0 + 4 * q, nt - 1);
      int ti, tj;
      tile_of(t < 10 ? t : t - 26, ti, tj);
      const bool cross = t >= 10 && t < 26;
      const int k = lane >> 4, c = lane & 15;
      xp[q] = &(t < 26 ? X : Y)[k][16 * (cross ? (t - 10) >> 2 : ti) + c];
      yp[q] = &(t < 10 ? X : Y)[k][16 * (cross ? (t - 10) & 3 : tj) + c];
      acc[q] = f64x4{0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll 4
    for (int k0 = 0; k0 < 64; k0 += 4)
#pragma unroll
      for (int q = 0; q < 3; ++q) acc[q] = mfma16(xp[q][k0 * LDA_S], yp[q][k0 * LDA_S], acc[q]);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      if (t0 + 4 * q >= nt) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        store_through(&out[(t0 + 4 * q) * 256 + ((lane >> 4) + 4 * r) * 16 + (lane & 15)], acc[q][r]);
    }
  }
}

// The reduced Gram in registers: entry (tid / 16, tid % 16) of each tile.
struct BlkGram {
  double v[36];
};
__device__ __forceinline__ void read_gram(const double* gs, bool two, BlkGram& b, int tid) {
#pragma unroll
  for (int t = 0; t < 36; ++t) b.v[t] = (t < 10 || two) ? gs[t * 256 + tid] : 0.0;
}

// Largest |G - I| of it (NaN if any entry is); w columns.
__device__ __forceinline__ double blk_dev(const BlkGram& b, int w, double* red4, int tid) {
  const bool two = w > NB;
  const int r = tid >> 4, c = tid & 15;
  double d = 0.0;
#pragma unroll
  for (int t = 0; t < 36; ++t) {
    if (t >= 10 && !two) break;
    double want = 0.0;
    if (t < 10 || t >= 26) {
      int ti, tj;
      tile_of(t < 10 ? t : t - 26, ti, tj);
      if (ti == tj && r == c && 16 * ti + r + (t < 10 ? 0 : NB) < w) want = 1.0;
    }
    const double x = fabs(b.v[t] - want);
    d = (x > d || x != x) ? x : d;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const double o = __shfl_xor(d, off, 64);
    d = (o > d || o != o) ? o : d;
  }
  if ((tid & 63) == 0) red4[tid >> 6] = d;
  __syncthreads();
  double m = red4[0];
#pragma unroll
  for (int q = 1; q < 4; ++q) m = (red4[q] > m || red4[q] != red4[q]) ? red4[q] : m;
  __syncthreads();
  return m;
}

// M := the symmetric 64x64 block of the 10 tiles from T0 on, ones on the
// diagonal beyond w columns.  Barrier after.
template <int T0>
__device__ __forceinline__ void put_gram(const BlkGram& b, double (*M)[LDA_S], int w, int tid) {
  const int r = tid >> 4, c = tid & 15;
#pragma unroll
  for (int t = 0; t < 10; ++t) {
    int ti, tj;
    tile_of(t, ti, tj);
    if (ti == tj && r > c) continue;  // one writer per entry of a diagonal tile
    const double v = (ti == tj && r == c && 16 * ti + r >= w) ? 1.0 : b.v[T0 + t];
    M[16 * ti + r][16 * tj + c] = v;
    M[16 * tj + c][16 * ti + r] = v;
  }
  __syncthreads();
}
// M := G12.  Barrier after.
__device__ __forceinline__ void put_cross(const BlkGram& b, double (*M)[LDA_S], int tid) {
#pragma unroll
  for (int t = 0; t < 16; ++t) M[16 * (t >> 2) + (tid >> 4)][16 * (t & 3) + (tid & 15)] = b.v[10 + t];
  __syncthreads();
}

// acc[tj] = row block `wave` of op(A) op(B) over k in [0, klim), 64x64 operands in
// LDS, op(X) = X^T with the flag; item r = C[16 wave + lane/16 + 4 r][16 tj + lane%16].
// KB: op(B) is upper triangular, k < 16 (tj + 1).
template <bool TA, bool TB = false, bool KB = false>
__device__ __forceinline__ void prod64(const double (*A)[LDA_S], const double (*B)[LDA_S], int klim, f64x4 (&acc)[4],
                                       int lane, int wave) {
#pragma unroll
  for (int tj = 0; tj < 4; ++tj) acc[tj] = f64x4{0.0, 0.0, 0.0, 0.0};
  if constexpr (KB) {
#pragma unroll
    for (int k0 = 0; k0 < 64; k0 += 4) {
      const int i = 16 * wave + (lane & 15), k = k0 + (lane >> 4);
      const double x = TA ? A[k][i] : A[i][k];
#pragma unroll
      for (int tj = k0 / 16; tj < 4; ++tj) {
        const int j = 16 * tj + (lane & 15);
        acc[tj] = mfma16(x, TB ? B[j][k] : B[k][j], acc[tj]);
      }
    }
    return;
  }
#pragma unroll 1
  for (int kb = 0; kb < klim; kb += 16) {
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4) {
      const int i = 16 * wave + (lane & 15), k = kb + k0 + (lane >> 4);
      const double x = TA ? A[k][i] : A[i][k];
#pragma unroll
      for (int tj = 0; tj < 4; ++tj) {
        const int j = 16 * tj + (lane & 15);
        acc[tj] = mfma16(x, TB ? B[j][k] : B[k][j], acc[tj]);
      }
    }
  }
}

__device__ __forceinline__ void store_acc(const f64x4 (&acc)[4], double (*C)[LDA_S], double scale, int lane, int wave) {
#pragma unroll
  for (int tj = 0; tj < 4; ++tj)
#pragma unroll
    for (int r = 0; r < 4; ++r) C[16 * wave + (lane >> 4) + 4 * r][16 * tj + (lane & 15)] = scale * acc[tj][r];
}
__device__ __forceinline__ void add_acc(const f64x4 (&acc)[4], double (*C)[LDA_S], double scale, int lane, int wave) {
#pragma unroll
  for (int tj = 0; tj < 4; ++tj)
#pragma unroll
    for (int r = 0; r < 4; ++r) C[16 * wave + (lane >> 4) + 4 * r][16 * tj + (lane & 15)] += scale * acc[tj][r];
}
__device__ __forceinline__ void save_acc(const f64x4 (&acc)[4], double* dst, int lane, int wave) {
#pragma unroll
  for (int tj = 0; tj < 4; ++tj)
#pragma unroll
    for (int r = 0; r < 4; ++r) dst[(16 * wave + (lane >> 4) + 4 * r) * NB + 16 * tj + (lane & 15)] = acc[tj][r];
}
__device__ __forceinline__ void save64(const double (*M)[LDA_S], double* dst, int tid) {
  for (int e = tid; e < NB * NB; e += 256) dst[e] = M[e / NB][e % NB];
}

// A uniform condition that the compiler must not pull out of a loop (loop
// unswitching would give the loop's body, thousands of instructions, two copies).
__device__ __forceinline__ bool one_copy(bool b) {
  int v = __builtin_amdgcn_readfirstlane((int)b);
  asm volatile("" : "+s"(v));
  return v != 0;
}

// Rejected block with norms that need scaling: its w columns column by column in
// place (team_factor), the clean V, and T from V's Gram by the recursion of
// GenerateBlockTr("F","C") (Reflector.hpp:580-626), the Gram and T held in
// scratch.  One workgroup; no other reads or writes the block any more.
__device__ __noinline__ void blk_refactor(CqrBlockArgs a, double* sh, int tid) {
  const int K = a.w, mp = a.mp;
  double* Gm = a.scratch + kBG;
  double* Tm = a.scratch + kBTF;
  team_factor<double, 256, true>(mp, K, a.A, (int)a.lda, a.tau, sh);
  __syncthreads();
  for (long e = tid; e < (long)mp * K; e += 256) {
    const int r = (int)(e % mp), c = (int)(e / mp);
    a.V[(size_t)r + (size_t)c * a.ldv] = (r > c) ? a.A[(size_t)r + (size_t)c * a.lda] : (r == c ? 1.0 : 0.0);
  }
  __syncthreads();
  for (int e = tid; e < K * K; e += 256) {
    const int l = e / K, c = e % K;
    double gv = 0.0;
    if (l < c)
      for (int r = c; r < mp; ++r) gv = fma(a.V[(size_t)r + (size_t)l * a.ldv], a.V[(size_t)r + (size_t)c * a.ldv], gv);
    Gm[e] = gv;
    Tm[e] = 0.0;
  }
  __syncthreads();
  for (int c = 0; c < K; ++c) {
    const double tc = a.tau[c];
    if (tid < c) {
      double sacc = 0.0;
      for (int l = tid; l < c; ++l) sacc = fma(Tm[tid * K + l], Gm[l * K + c], sacc);
      Tm[tid * K + c] = -tc * sacc;
    }
    if (tid == c) Tm[c * K + c] = tc;
    __syncthreads();
  }
  for (int e = tid; e < K * K; e += 256) {
    const int i = e % K, j = e / K;
    a.T[(size_t)i + (size_t)j * a.ldt] = Tm[i * K + j];
  }
}

typedef __attribute__((address_space(3))) double LdsD;

// Rejected block: column by column by every workgroup, its 64 rows in registers
// (a thread 32 rows of one column), with Reflector::Generate's rules
// (Reflector.hpp:117-158).  One grid-wide step per column c: every workgroup
// hands out its part of x^T a_j for all columns j, x the entries of column c below
// the diagonal -- the norm (j = c), the reflector's application (j > c) and V's
// Gram (j < c), since V = x / (alpha - beta) -- and the owner of row c that row.
// Then T by workgroup 0, a thread per row of the recursion of
// GenerateBlockTr("F","C") (Reflector.hpp:580-626).  False, with A untouched,
// when a column's squared norm is outside [2^-600, 2^600] but not zero.
// Bound by a grid-wide step per column, 6 us with three workgroups and 14 with
// 160: 10000 x 100 takes 1.7 ms in all, 180 x 128 1.0, 779 x 55 0.46.  (One
// workgroup alone, on the block in memory: 72, 2.0 and 1.2 ms; a column-wise
// launch for 64 columns and less, without the attempt before it: 0.5 ms at
// 90 x 90, where the attempt and this take 0.7.)
// step: the first unused number of the grid-wide steps.  X, Y, M1, M2: scratch,
// 64 x LDA_S each.
__device__ __noinline__ bool blk_columnwise(CqrBlockArgs a, int step, LdsD* X, LdsD* Y, LdsD* M1, LdsD* M2) {
  RNPX_CQR_GLOBAL(a);
  const int tid = threadIdx.x, g = blockIdx.x, G = gridDim.x;
  const int K = a.w, mp = a.mp;
  const int j = tid & 127, half = tid >> 7, h0 = 32 * half, r0 = 64 * g + h0;  // this thread's column, its first row
  double* Gm = a.scratch + kBG;
  double y[32];
#pragma unroll
  for (int r = 0; r < 32; ++r)
    y[r] = (r0 + r < mp && j < K) ? a.A[(size_t)(r0 + r) + (size_t)j * a.lda] : 0.0;
  for (int c = -1; c < K; ++c) {  // c = -1: the columns' norms, which must be in range
    double* slot = a.part + 256 * (c & 1);
    double* rowc = a.scratch + kBRow + 128 * (c & 1);
    LdsD* const xs = X + h0;
    double d = 0.0, mx = 0.0;
    if (c >= 0) {
      double yc = 0.0;
#pragma unroll
      for (int r = 0; r < 32; ++r) {
        if (j == c) xs[r] = r0 + r > c ? y[r] : 0.0;
        if (r0 + r == c) yc = y[r];
      }
      if (c >= r0 && c < r0 + 32) store_through(rowc + j, yc);
      __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 32; ++r) {
      const double x = c < 0 ? y[r] : xs[r];
      d = fma(x, y[r], d);
      mx = fmax(mx, fabs(x));
    }
    M1[tid] = d;
    M1[256 + tid] = mx;
    __syncthreads();
    if (tid < 128) {
      double* my = slot + (size_t)g * kBlkElems;
      store_through(my + tid, M1[tid] + M1[128 + tid]);
      if (c < 0 || tid == 0) store_through(my + 128 + tid, fmax(M1[256 + tid], M1[384 + tid]));
    }
    grid_step(a, step++, g, G, tid);
    // the sum of a column's products (at c = -1 the largest entry beside it): two
    // threads, every other workgroup's each, 16 loads in flight
    d = mx = 0.0;
    for (int q0 = half; q0 < G; q0 += 32) {
      double v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = slot[(size_t)min(q0 + 2 * u, G - 1) * kBlkElems + j];
#pragma unroll
      for (int u = 0; u < 16; ++u)
        if (q0 + 2 * u < G) d += v[u];
    }
    if (c < 0)
      for (int q = half; q < G; q += 2) mx = fmax(mx, slot[(size_t)q * kBlkElems + 128 + j]);
    else if (tid < G)
      mx = slot[(size_t)tid * kBlkElems + 128];
    const double rj = c >= 0 ? rowc[j] : 0.0;  // row c, column j
    if (c >= 0) mx = wave_max(mx);
    M1[tid] = d;
    M1[256 + tid] = mx;
    if (tid < 128) M1[512 + tid] = rj;
    __syncthreads();
    d = M1[j] + M1[128 + j];
    if (c < 0) {
      const double m = fmax(M1[256 + j], M1[384 + j]);
      if (__syncthreads_or(!(d >= 0x1p-600 && d <= 0x1p600) && !(d == 0.0 && m == 0.0))) return false;
      continue;
    }
    const double ss = M1[c] + M1[128 + c], alpha = M1[512 + c];
    const double xmax = fmax(fmax(M1[256], M1[320]), fmax(M1[384], M1[448]));
    double tau = 0.0, inv = 0.0;
    if (ss >= 0x1p-600 && ss <= 0x1p600) {
      double beta = hypot3(alpha, 0.0, sqrt(ss));
      if (alpha > 0.0) beta = -beta;
      tau = (beta - alpha) / beta;
      inv = recip_t(alpha - beta);
      const double cw = tau * fma(inv, d, rj);
      const double diag = j == c ? beta : rj - cw;
#pragma unroll
      for (int r = 0; r < 32; ++r) {
        const double v = xs[r] * inv;
        if (j > c) y[r] -= v * cw;  // (xs is zero from row c up)
        if (j == c && r0 + r > c) y[r] = v;
        if (j >= c && r0 + r == c) y[r] = diag;
      }
    } else if (!(ss == 0.0 && xmax == 0.0)) {
      return false;
    }
    if (g == 0) {
      if (tid < c) Gm[tid * K + c] = fma(inv, d, rj);
      if (tid == 0) a.tau[c] = tau;
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 32; ++r) {
    const int gr = r0 + r;
    if (gr < mp && j < K) {
      a.A[(size_t)gr + (size_t)j * a.lda] = y[r];
      a.V[(size_t)gr + (size_t)j * a.ldv] = (gr > j) ? y[r] : (gr == j ? 1.0 : 0.0);
    }
  }
  if (g != 0) return true;
  __syncthreads();
  // T's row i by thread i: columns 0..63 in M1 (i < 64) or nowhere, 64..127 in M2 or X
  LdsD* const lo = M1 + tid * LDA_S;
  LdsD* const hi = (tid < NB ? M2 + tid * LDA_S : X + (tid & (NB - 1)) * LDA_S) - NB;
  // (zeros left of the diagonal, so that every row's sum starts at column 0)
  for (int e = tid; e < 64 * LDA_S; e += 256) M1[e] = M2[e] = X[e] = 0.0;
  for (int c0 = 0; c0 < K; c0 += 32) {  // 32 columns of the Gram, then of T
    __syncthreads();
    for (int e = tid; e < 32 * 128; e += 256) {
      const int c = c0 + e / 128, l = e % 128;
      if (c < K) Y[e] = l < c ? Gm[l * K + c] : (l == c ? a.tau[c] : 0.0);
    }
    __syncthreads();
    if (tid < 128)
      for (int c = max(c0, tid); c < min(c0 + 32, K); ++c) {
        LdsD* const gc = Y + (c - c0) * 128;
        double s = 0.0, s2 = 0.0;
        if (tid < NB)
#pragma unroll 8
          for (int l = 0; l < min(c, NB); ++l) s = fma(lo[l], gc[l], s);
        if (c > NB)
#pragma unroll 8
          for (int l = NB; l < c; ++l) s2 = fma(hi[l], gc[l], s2);
        (c < NB ? lo : hi)[c] = (tid == c) ? gc[c] : -gc[c] * (s + s2);
      }
  }
  __syncthreads();
  if (tid < K)
    for (int c = 0; c < K; ++c)
      a.T[(size_t)tid + (size_t)c * a.ldt] = (tid > c) ? 0.0 : (c < NB ? lo : hi)[c];
  return true;
}

// What every workgroup does with a rejected block.
__device__ __noinline__ void blk_rejected(CqrBlockArgs a, int step, LdsD* X, LdsD* Y, LdsD* M1, LdsD* M2, double* sh) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.fail = 1u;
  if (!blk_columnwise(a, step, X, Y, M1, M2) && blockIdx.x == 0) blk_refactor(a, sh, threadIdx.x);
}

// T = -U D Z^T (upper) from U in M1 (on and above the diagonal), D in dcol and
// Z = L^-1 in M2 (lower blocks); column `last` (no reflector) zero.
__device__ __forceinline__ void blk_t_factor(const double (*M1)[LDA_S], const double (*M2)[LDA_S], const double* dcol,
                                             int last, f64x4 (&acc)[4], int lane, int wave) {
  upper_product_row<true>(M1, M2, true, dcol, acc, lane, wave);
#pragma unroll
  for (int tj = 0; tj < 4; ++tj)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * wave + (lane >> 4) + 4 * r, j = 16 * tj + (lane & 15);
      acc[tj][r] = (i <= j && j != last) ? -acc[tj][r] : 0.0;
    }
}

}  // namespace

__global__ __launch_bounds__(256) void cqr_block_kernel(CqrBlockArgs a) {
  RNPX_CQR_GLOBAL(a);
  if (threadIdx.x == 0) __hip_atomic_fetch_add(&a.sync[kBlkResident], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __shared__ double Ab1[64][LDA_S];
  __shared__ double Ab2[64][LDA_S];
  __shared__ double M1[NB][LDA_S];
  __shared__ double M2[NB][LDA_S];
  __shared__ double rowbuf[NB];
  __shared__ double red4[4];
  __shared__ double gdiag[NB];
  __shared__ double tmpb[small64::kTmpDoubles];
  __shared__ unsigned slot;
  __shared__ int okf;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = blockIdx.x, G = gridDim.x;
  const int r0 = 64 * g;
  const int mp = a.mp, w = a.w, w2 = w - NB;  // w2: columns of the second half
  const bool two = w2 > 0;
  double* sc = a.scratch;
  double* part = a.part + (size_t)g * kBlkElems;
  // step: the first grid-wide step not taken yet, the same in every workgroup
  auto rejected = [&](int step) {
    __syncthreads();
    blk_rejected(a, step, (LdsD*)&Ab1[0][0], (LdsD*)&Ab2[0][0], (LdsD*)&M1[0][0], (LdsD*)&M2[0][0], rowbuf);
  };

  // Both halves' rows of this workgroup, zero outside the block.
  {
    constexpr int PER = 64 * NB / 256;
    double v[2][PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = tid + 256 * q, r = e % 64, c = e / 64;
      const bool in = r0 + r < mp;
      v[0][q] = (in && c < w) ? a.A[(size_t)(r0 + r) + (size_t)c * a.lda] : 0.0;
      v[1][q] = (in && c < w2) ? a.A[(size_t)(r0 + r) + (size_t)(c + NB) * a.lda] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = tid + 256 * q;
      Ab1[e % 64][e / 64] = v[0][q];
      Ab2[e % 64][e / 64] = v[1][q];
    }
  }
  __syncthreads();

  // ---- 1 and 2: passes; workgroup 2 keeps their factors for R ----
  int np = 0;  // passes done (factors at sc + kBR + 3 * 4096 * pass)
  bool later = false;  // the second half is projected only so far (R22 = I)
#pragma unroll 1
  for (int pass = 0;; ++pass) {
    blk_gram(Ab1, Ab2, two, part, lane, wave);
    double* gs = a.gsum + (size_t)pass * kBlkElems;
    blk_allreduce(a, two ? kBlkElems : kGramElems, pass, g, G, gs, tmpb, tid);
    BlkGram gm;
    read_gram(gs, two, gm, tid);
    double dev = 1.0;
    if (pass > 0) dev = blk_dev(gm, later ? NB : w, red4, tid);
    double* rp = sc + kBR + (size_t)3 * 4096 * pass;
    const bool is_first = pass > 0 && dev <= kFirstOrder;
    const bool was_later = later;
    bool ok = pass == 0 || (dev <= kThirdPass && ((is_first && !later) || pass < kBlkPasses));
    // A zero tail in the first column (triangular, diagonal input) would reject
    // the block in the reconstruction, some 170 us later.
    if (pass == 0 && (a.zero_tails & 1)) {
      const double d0 = gs[0], a0 = a.A[0];
      ok = !(d0 - a0 * a0 <= 0x1p-42 * d0);
    }
#pragma unroll 1
    for (int half = 0; half < (two ? 2 : 1) && ok; ++half) {
      const bool first = one_copy(is_first && !(half != 0 && was_later)), second_half = one_copy(half != 0), keep = one_copy(g == 2);
      double(*X)[LDA_S] = second_half ? M2 : M1;   // the Gram, then R
      double(*Xi)[LDA_S] = second_half ? M1 : M2;  // R^-1
      f64x4 acc[4];
      if (!second_half) {
        put_gram<0>(gm, M1, w, tid);
        if (tid < NB) gdiag[tid] = M1[tid][tid];
      } else {
        put_cross(gm, M1, tid);
        if (!first) {
          prod64<true>(M2, M1, 16 * (wave + 1), acc, lane, wave);  // R12 = R11^-T G12 (first order: E12)
          __syncthreads();
          store_acc(acc, M1, 1.0, lane, wave);
        }
        put_gram<26>(gm, M2, w2, tid);  // its barrier: M1 is complete too
        if (keep) save64(M1, rp + 4096, tid);
        prod64<false>(Ab1, M1, 64, acc, lane, wave);
        add_acc(acc, Ab2, -1.0, lane, wave);  // A2 - Q1 R12
        if (!first) {
          if (tid < NB) gdiag[tid] = M2[tid][tid];  // the columns' own norms
          prod64<true>(M1, M1, 64, acc, lane, wave);
          __syncthreads();
          add_acc(acc, M2, -1.0, lane, wave);  // G22 - R12^T R12
        }
        __syncthreads();
      }
      double* rs = rp + (second_half ? 8192 : 0);
      if (first) {
        // R = I + S, R^-1 = I - S with S = triu(E) - diag(E)/2
        for (int e = tid; e < NB * NB; e += 256) {
          const int i = e / NB, c = e % NB;
          const double one = (i == c) ? 1.0 : 0.0, E = X[i][c] - one, S = (i < c) ? E : 0.5 * one * E;
          Xi[i][c] = one - S;
          if (keep) rs[e] = one + S;
        }
        __syncthreads();
      } else {
        ok = small64::chol64<LDA_S>(&X[0][0], &Xi[0][0], tmpb, gdiag, &okf, tid);
        if (second_half) {
          later = !ok && pass < kBlkProject;
          if (later) {
            ok = true;
            if (keep)
              for (int e = tid; e < NB * NB; e += 256) rs[e] = (e / NB == e % NB) ? 1.0 : 0.0;
            continue;
          }
        }
        if (ok && keep)
          for (int e = tid; e < NB * NB; e += 256) rs[e] = (e / NB <= e % NB) ? X[e / NB][e % NB] : 0.0;
      }
      if (ok) times_upper<64>(second_half ? Ab2 : Ab1, Xi, lane, wave);
    }
    if (!ok) {
      rejected(2 * pass + 3);
      return;
    }
    np = pass + 1;
    if (pass > 0 && dev <= kSecondPass && !was_later && !later) break;  // orthonormal to working precision now
  }

  // ---- 3: reconstruction ----
  const int last = (mp == w) ? w - 1 : -1;  // the column without a reflector
  f64x4 racc[3][4];
  if (g == 2) {
    // R's product of the passes' factors, in place of the first one's
    double* c0 = sc + kBR;
    for (int p = 1; p < np; ++p) {
      const double* rp = sc + kBR + (size_t)3 * 4096 * p;
      __syncthreads();
      load64(rp, M1, tid);
      load64(c0, M2, tid);
      __syncthreads();
      upper_product_row(M1, M2, false, nullptr, racc[0], lane, wave);
      if (two) {
        __syncthreads();
        load64(c0 + 4096, M2, tid);
        __syncthreads();
        prod64<false>(M1, M2, 64, racc[1], lane, wave);
        __syncthreads();
        load64(rp + 4096, M1, tid);
        load64(c0 + 8192, M2, tid);
        __syncthreads();
        f64x4 x[4];
        prod64<false, false, true>(M1, M2, 64, x, lane, wave);
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) racc[1][tj] += x[tj];
        __syncthreads();
        load64(rp + 8192, M1, tid);
        __syncthreads();
        upper_product_row(M1, M2, false, nullptr, racc[2], lane, wave);
      }
      if (p + 1 < np) {
        __syncthreads();
        save_acc(racc[0], c0, lane, wave);
        if (two) {
          save_acc(racc[1], c0 + 4096, lane, wave);
          save_acc(racc[2], c0 + 8192, lane, wave);
        }
      }
    }
    __syncthreads();
  }
#pragma unroll 1
  for (int half = 0; half < (two ? 2 : 1); ++half) {
    const bool sh = one_copy(half != 0), mine = one_copy(g == half), fh = one_copy(two && half == 0);
    double(*Ab)[LDA_S] = sh ? Ab2 : Ab1;
    unsigned* pub = &a.sync[sh ? kBlkPub2 : kBlkPub1];
    double* ui = sc + (sh ? kBU2i : kBU1i);
    double* dd = sc + (sh ? kBD2 : kBD1);
    const int o = sh ? NB : 0, wh = min(w - o, NB);                 // this half's first column, its width
    const int lasth = (last >= o && last < o + NB) ? last - o : -1;  // its column without a reflector
    f64x4 acc[4];
    if (mine) {
      for (int e = tid; e < NB * NB; e += 256) M1[e / NB][e % NB] = Ab[e / NB][e % NB];
      __syncthreads();
      // M1 = U and L, M2 = U^-1
      const bool fits = small64::lu64<LDA_S>(&M1[0][0], rowbuf, &M2[0][0], tmpb, &okf, tid, lasth,
                                                  ((a.zero_tails >> half) & 1) ? 1.0 - 0x1p-40 : 2.0);
      save64(M2, ui, tid);
      if (tid < NB) dd[tid] = rowbuf[tid];
      publish(pub, fits ? 1u : kRejected);
      if (!fits) {
        rejected(2 * np + 1);
        return;
      }
      for (int e = tid; e < NB * NB; e += 256) {
        const int i = e / NB, j = e % NB;
        const double v = (i > j) ? M1[i][j] : (i == j ? 1.0 : 0.0);
        if (!sh) Ab1[i][j] = v;  // V1's top block: L11
        else M1[i][j] = (i > j) ? v : M1[i][j];
      }
      if (tid < wh) a.tau[o + tid] = (tid == lasth) ? 0.0 : -M1[tid][tid] * rowbuf[tid];
      __syncthreads();
      small64::inv_unit_lower64<LDA_S>(&M1[0][0], &M2[0][0], tmpb, tid);  // M2 = L^-1 (lower blocks)
      if (fh) {
        prod64<false>(M2, Ab2, 16 * (wave + 1), acc, lane, wave);  // U12 = L11^-1 Q2(0:64)
        save_acc(acc, sc + kBU12, lane, wave);
        publish(&a.sync[kBlkPubU12]);
      }
      blk_t_factor(M1, M2, rowbuf, lasth, acc, lane, wave);
      if (fh) {
        save_acc(acc, sc + kBT1, lane, wave);
        publish(&a.sync[kBlkPubT1]);
      }
#pragma unroll
      for (int tj = 0; tj < 4; ++tj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * wave + (lane >> 4) + 4 * r, j = 16 * tj + (lane & 15);
          a.T[(size_t)(o + i) + (size_t)(o + j) * a.ldt] = acc[tj][r];
        }
      // A only once the second half is accepted too
      if (fh && wait_verdict(&a.sync[kBlkPub2], a.abortf, &slot) == kRejected) {
        rejected(2 * np + 1);
        return;
      }
      for (int e = tid; e < NB * NB; e += 256) {
        const int i = e % NB, j = e / NB;
        const double l = M1[i][j];
        if (o + i < mp && j < wh) {
          if (i > j) a.A[(size_t)(o + i) + (size_t)(o + j) * a.lda] = l;
          a.V[(size_t)(o + i) + (size_t)(o + j) * a.ldv] = (i > j) ? l : (i == j ? 1.0 : 0.0);
        }
        if (!sh) {
          if (j < w2) a.V[(size_t)i + (size_t)(j + NB) * a.ldv] = 0.0;
          if (fh) a.T[(size_t)(i + NB) + (size_t)j * a.ldt] = 0.0;
        } else if (NB + i < mp) {
          const double v = Ab1[i][j];
          a.A[(size_t)(NB + i) + (size_t)j * a.lda] = v;
          a.V[(size_t)(NB + i) + (size_t)j * a.ldv] = v;
        }
      }
      if (!sh) return;
      // T12 = -(T11 L21^T + U12 D2) L22^-T
      wait_flag(&a.sync[kBlkPubT1], a.abortf);  // its barrier: M1 is free
      load64(sc + kBT1, M1, tid);
      __syncthreads();
      prod64<false, true>(M1, Ab1, 64, acc, lane, wave);
      __syncthreads();
#pragma unroll
      for (int tj = 0; tj < 4; ++tj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * wave + (lane >> 4) + 4 * r, j = 16 * tj + (lane & 15);
          M1[i][j] = acc[tj][r] + sc[kBU12 + i * NB + j] * rowbuf[j];
        }
      __syncthreads();
      prod64<false, true, true>(M1, M2, 64, acc, lane, wave);
#pragma unroll
      for (int tj = 0; tj < 4; ++tj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * wave + (lane >> 4) + 4 * r, j = 16 * tj + (lane & 15);
          a.T[(size_t)i + (size_t)(NB + j) * a.ldt] = (j == lasth) ? 0.0 : -acc[tj][r];
        }
      return;
    }
    if (g < half) return;  // (workgroup 0 left above)
    if (wait_verdict(pub, a.abortf, &slot) == kRejected) {
      rejected(2 * np + 1);
      return;
    }
    load64(ui, M2, tid);
    __syncthreads();
    times_upper<64>(Ab, M2, lane, wave);  // V rows of this half
    if (fh) {
      wait_flag(&a.sync[kBlkPubU12], a.abortf);
      load64(sc + kBU12, M1, tid);
      __syncthreads();
      prod64<false>(Ab1, M1, 64, acc, lane, wave);
      add_acc(acc, Ab2, -1.0, lane, wave);  // Q2 - V1 U12
      __syncthreads();
    }
  }
  for (int e = tid; e < 64 * NB; e += 256) {
    const int r = e % 64, c = e / 64, gr = r0 + r;
    if (gr < mp && c < w) {
      const double v = Ab1[r][c];
      a.A[(size_t)gr + (size_t)c * a.lda] = v;
      a.V[(size_t)gr + (size_t)c * a.ldv] = v;
    }
    if (gr < mp && c < w2) {
      const double v = Ab2[r][c];
      a.A[(size_t)gr + (size_t)(c + NB) * a.lda] = v;
      a.V[(size_t)gr + (size_t)(c + NB) * a.ldv] = v;
    }
  }
  if (g == 2) {
#pragma unroll
    for (int tj = 0; tj < 4; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * wave + (lane >> 4) + 4 * r, j = 16 * tj + (lane & 15);
        if (i <= j && j < w) a.A[(size_t)i + (size_t)j * a.lda] = sc[kBD1 + i] * racc[0][tj][r];
        if (j < w2) {
          a.A[(size_t)i + (size_t)(NB + j) * a.lda] = sc[kBD1 + i] * racc[1][tj][r];
          if (i <= j) a.A[(size_t)(NB + i) + (size_t)(NB + j) * a.lda] = sc[kBD2 + i] * racc[2][tj][r];
        }
      }
  }
}

int cqr_block_groups(int mp, int w, int max_groups) {
  // Fewer than 16 columns, in the first half or beyond it, are left to the
  // column-wise panel: the launch costs 108 us for one half and 230 for two at
  // any width up to 1000 rows, that panel 5 to 7 us a column (16 columns: 108 us
  // at 250 rows, 134 at 1000, 147 at 8000 against 138 here).
  if (w < 16 || (w > NB && w < NB + 16) || w > 2 * NB || mp < w) return 0;
  const int G = std::max(3, (mp + 63) / 64);  // the roles of three workgroups
  return (G <= max_groups && G <= 16 * kGroup) ? G : 0;
}

hipError_t launch_cqr_block(const CqrBlockArgs& a, int G, hipStream_t st) {
  if (a.w < 1 || a.w > 2 * NB || a.mp < a.w || G < 3 || (long)G * 64 < a.mp || (G > 3 && (long)(G - 1) * 64 >= a.mp) ||
      a.lda < a.mp || a.ldv < a.mp || a.ldt < 2 * NB || !a.fail || !a.sync || !a.abortf)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(cqr_block_kernel, dim3(G), dim3(256), 0, st, a);
  return hipGetLastError();
}

// Scheduling gate for the look-ahead: one thread waits until all G
// workgroups of the block kernel whose sync words start at block_sync have
// started, so that a GEMM queued behind the gate on another stream cannot
// take the CUs those workgroups need first.  Only the order of dispatch
// depends on it (the GEMM reads nothing the block kernel writes), so the
// wait gives up after 2 ms.  A wait that gives up sets *off, which turns every
// later gate of the handle into a no-op: the runtime can map the two
// streams onto one hardware queue (more streams in the process than
// queues), and then the block kernel sits behind the gate and every wait
// would run to its limit.
__global__ void cqr_gate_kernel(const unsigned* block_sync, unsigned G, unsigned* off) {
  if (threadIdx.x != 0) return;
  if (__hip_atomic_load(off, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return;
  const unsigned* c = block_sync + kBlkResident;
  const uint64_t t0 = wall_clock64();
  while (__hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < G) {
    if (wall_clock64() - t0 > 200000ull) {
      __hip_atomic_store(off, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
}

hipError_t launch_cqr_gate(const unsigned* block_sync, int G, unsigned* off, hipStream_t st) {
  if (!block_sync || !off || G < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(cqr_gate_kernel, dim3(1), dim3(64), 0, st, block_sync, (unsigned)G, off);
  return hipGetLastError();
}

int cqr_panel_groups(int mp, int max_groups, int* rw) {
  if (mp < 2 * NB) return 0;
  if (max_groups > kCqrMaxGroups) max_groups = kCqrMaxGroups;
  static const int first_rw = [] {
    const char* e = getenv("RNPX_CQR_RW");  // 128: fewer, larger workgroups
    return (e && atoi(e) == 128) ? 128 : 64;
  }();
  for (int r : {first_rw, 64, 128}) {
    const int G = (mp + r - 1) / r;
    if (G >= 2 && G <= max_groups) {
      *rw = r;
      return G;
    }
  }
  return 0;
}

hipError_t launch_cqr_panel(const CqrArgs& a, int G, int rw, hipStream_t st) {
  if (a.mp < 2 * NB || G < 2 || G > kCqrMaxGroups || (long)G * rw < a.mp || (long)(G - 1) * rw >= a.mp ||
      a.lda < a.mp || a.ldv < a.mp || a.ldt < NB)
    return hipErrorInvalidValue;
  if (rw == 64)
    hipLaunchKernelGGL((cqr_panel_kernel<64>), dim3(G), dim3(256), 0, st, a);
  else if (rw == 128)
    hipLaunchKernelGGL((cqr_panel_kernel<128>), dim3(G), dim3(256), 0, st, a);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace rnpx
