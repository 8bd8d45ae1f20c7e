// rnpx_trsm.hip -- triangular solves with the QR factor R for the least-squares
// driver and its refinement, in place on B (n x nrhs):
//
//   trans 'N':  R X = B     (back substitution; SolveTrM "L","U","N","N",
//                            RNP/BLAS/BLAS_mix.hpp:2096)
//   trans 'C':  R^H X = B   (forward substitution; the semi-normal
//                            equations' first solve)
//
// R is upper triangular (n x n, leading dimension ldr) -- the upper triangle
// of the factored A.  The same kernel, templated on the triangle, the
// operation (N, T, C) and a unit diagonal, does LU::Solve's four solves
// (SolveTrM "L","L"/"U", LU.hpp:117-144).
//
// Blocked and sync-free: one workgroup per (64-row block p, four right-hand
// sides).  Workgroup w solves block p = nblk-1-w ('N') or p = w ('C'), so it
// depends only on lower-numbered workgroups of the same right-hand sides,
// which the dispatcher started before it: every wait ends.  A workgroup
// stages its diagonal block in LDS while it waits, adds the off-diagonal
// products R_pq x_q in a fixed order as the blocks q it needs are published
// (flags per block and right-hand side holding the call's epoch), then wave v
// solves the diagonal block for right-hand side v by substitution (lane = row,
// the pivot broadcast by v_readlane) and publishes x_p.  Quotients are
// y * (1/r) with one correction step, y/r to within an ulp.
//
// What bounds it is the chain from one block's x to the next: the flag's and
// x's trips through memory, the last off-diagonal product, 64 dependent
// quotients.  Nothing else is on it: R_pq is loaded before the flag is polled,
// x goes without fences, and with four right-hand sides to a workgroup every
// workgroup of n = 8192, 16 right-hand sides is resident at once and R is read a
// quarter as often.  That solve takes 920 us (7.2 us a block), with one right-hand
// side to a workgroup, R loaded after the flag and an agent-scope fence on each
// side 2650.
#include "rnpx_kernels.hpp"

namespace rnpx {

namespace {

constexpr int TB = 64;  // block rows per workgroup

constexpr int RHS = 4;  // right-hand sides per workgroup, one per wave in the substitution

// x passes between workgroups in agent-scope relaxed stores and loads, which
// don't go through a cache that another workgroup's stores leave stale: no fence,
// whose cache write-back and invalidation would sit on the chain.
__device__ __forceinline__ void store_x(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_x(zd* p, zd v) {
  store_x(&p->x, v.x);
  store_x(&p->y, v.y);
}
__device__ __forceinline__ double load_x(double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ zd load_x(zd* p) {
  zd v = S<zd>::zero();
  v.x = load_x(&p->x);
  v.y = load_x(&p->y);
  return v;
}

// op(M) X = B with M the upper (UPPER) or lower triangle of R, op = N, T
// (transpose, OP = 1) or C (conjugate transpose, OP = 2), unit diagonal
// when UNIT.  E = op(M) is upper when UPPER == (OP == 0): backward
// substitution, blocks from the last; forward otherwise.
template <typename T, bool UPPER, int OP, bool UNIT>
__global__ __launch_bounds__(256) void trsm_tri_kernel(int n, int nrhs, const T* __restrict__ R, long ldr, T* B,
                                                       long ldb, unsigned* flags, unsigned epoch, unsigned* abortf) {
  constexpr bool EUP = (UPPER == (OP == 0));
  constexpr int CW = TB / 4;  // columns of an off-diagonal block per wave
  __shared__ T Rs[TB][TB + 1];  // E's diagonal block, row-major
  __shared__ T rinv[TB];
  __shared__ T xs[2][RHS][TB];
  __shared__ T red[4][RHS][TB];
  __shared__ int bad;
  const int nblk = (n + TB - 1) / TB;
  const int w = blockIdx.x, c0 = blockIdx.y * RHS, nr = min(RHS, nrhs - c0);
  const int p = EUP ? nblk - 1 - w : w;
  const int i0 = p * TB, bs = min(TB, n - i0);
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const T zero = S<T>::zero(), one = S<T>::one();
  // this wave's right-hand side (the last one again beyond nr: never published)
  T* b = B + (size_t)(c0 + min(wave, nr - 1)) * ldb;
  unsigned* fl = flags + (size_t)(c0 + min(wave, nr - 1)) * nblk;
  if (t == 0) bad = 0;
  // Diagonal block E(i0 + r, i0 + q), identity beyond bs (read down R's columns).
  for (int e = t; e < TB * TB; e += 256) {
    const int r = e % TB, q = e / TB;  // R(i0 + r, i0 + q)
    T v = (r == q) ? one : zero;
    const bool in_tri = UPPER ? (r <= q) : (r >= q);
    if (r < bs && q < bs && in_tri && !(UNIT && r == q)) v = R[(size_t)(i0 + r) + (size_t)(i0 + q) * ldr];
    if (OP == 0)
      Rs[r][q] = v;
    else
      Rs[q][r] = (OP == 2) ? S<T>::conj(v) : v;
  }
  T y = (lane < bs) ? b[i0 + lane] : zero;
  __syncthreads();
  if (t < TB) rinv[t] = UNIT ? one : recip_t(Rs[t][t]);

  // Off-diagonal blocks, in the order they are finished.
  T acc[RHS];
#pragma unroll
  for (int v = 0; v < RHS; ++v) acc[v] = zero;
  for (int d = 0; d < w; ++d) {
    const int q = EUP ? nblk - 1 - d : d;
    const int j0 = q * TB, bq = min(TB, n - j0), jw = wave * CW;
    // R_pq needs no x: on its way while the flag is polled
    T rij[CW];
#pragma unroll
    for (int jj = 0; jj < CW; ++jj) {
      const int j = jw + jj;
      rij[jj] = zero;
      if (lane < bs && j < bq)
        rij[jj] = (OP == 0) ? R[(size_t)(i0 + lane) + (size_t)(j0 + j) * ldr]
                            : R[(size_t)(j0 + j) + (size_t)(i0 + lane) * ldr];
    }
    const uint64_t t0 = wall_clock64();
    while (__hip_atomic_load(&fl[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != epoch) {
      if (__hip_atomic_load(abortf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
        bad = 1;
        break;
      }
      if (wall_clock64() - t0 > kBarrierTimeoutTicks) {
        __hip_atomic_store(abortf, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bad = 1;
        break;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // x's loads stay behind the flag's
    // two buffers: a wave that runs ahead writes the one nobody reads any more
    xs[d & 1][wave][lane] = (lane < bq) ? load_x(&b[j0 + lane]) : zero;
    __syncthreads();
    if (bad) return;
#pragma unroll
    for (int jj = 0; jj < CW; ++jj) {
      const T r = (OP == 2) ? S<T>::conj(rij[jj]) : rij[jj];
#pragma unroll
      for (int v = 0; v < RHS; ++v)
        if (v < nr) acc[v] = acc[v] + r * xs[d & 1][v][jw + jj];
    }
  }
#pragma unroll
  for (int v = 0; v < RHS; ++v) red[wave][v][lane] = acc[v];
  __syncthreads();
  if (wave >= nr) return;
  if (lane < bs)
    y = y - ((red[0][wave][lane] + red[1][wave][lane]) + (red[2][wave][lane] + red[3][wave][lane]));
#pragma unroll 8
  for (int k = 0; k < TB; ++k) {
    const int i = EUP ? TB - 1 - k : k;
    const T ri = Rs[lane][i];
    const T yi = readlane_t(y, i);
    T xi = yi * rinv[i];
    if (!UNIT) xi = xi + (yi - xi * Rs[i][i]) * rinv[i];
    if (lane == i) y = xi;
    else if (EUP ? lane < i : lane > i) y = y - ri * xi;
  }
  if (lane < bs) store_x(&b[i0 + lane], y);
  // x has reached memory before the flag leaves
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (lane == 0) __hip_atomic_store(&fl[p], epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

int trsm_flag_words(int n, int nrhs) { return ((n + TB - 1) / TB) * nrhs; }

template <typename T, bool UPPER, int OP, bool UNIT>
static void launch_tri(const dim3& grid, hipStream_t st, int n, int nrhs, const T* R, long ldr, T* B, long ldb,
                       unsigned* flags, unsigned epoch, unsigned* abortf) {
  hipLaunchKernelGGL((trsm_tri_kernel<T, UPPER, OP, UNIT>), grid, dim3(256), 0, st, n, nrhs, R, ldr, B, ldb, flags,
                     epoch, abortf);
}

template <typename T>
hipError_t launch_trsm_tri(char uplo, char op, char diag, int n, int nrhs, const T* R, long ldr, T* B, long ldb,
                           unsigned* flags, unsigned epoch, unsigned* abortf, hipStream_t st) {
  if (n < 0 || nrhs < 0 || ldr < std::max(1, n) || ldb < std::max(1, n) || epoch == 0u || !flags || !abortf)
    return hipErrorInvalidValue;
  if ((uplo != 'U' && uplo != 'L') || (op != 'N' && op != 'T' && op != 'C') || (diag != 'N' && diag != 'U'))
    return hipErrorInvalidValue;
  if (n == 0 || nrhs == 0) return hipSuccess;
  if (nrhs > 65535) return hipErrorInvalidValue;
  const dim3 grid((n + TB - 1) / TB, (nrhs + RHS - 1) / RHS);
  const bool up = (uplo == 'U'), unit = (diag == 'U');
  const int o = (op == 'N') ? 0 : (op == 'T' ? 1 : 2);
#define RNPX_TRI(U, O, D) \
  if (up == U && o == O && unit == D) { launch_tri<T, U, O, D>(grid, st, n, nrhs, R, ldr, B, ldb, flags, epoch, abortf); return hipGetLastError(); }
  RNPX_TRI(true, 0, false) RNPX_TRI(true, 1, false) RNPX_TRI(true, 2, false)
  RNPX_TRI(true, 0, true) RNPX_TRI(true, 1, true) RNPX_TRI(true, 2, true)
  RNPX_TRI(false, 0, false) RNPX_TRI(false, 1, false) RNPX_TRI(false, 2, false)
  RNPX_TRI(false, 0, true) RNPX_TRI(false, 1, true) RNPX_TRI(false, 2, true)
#undef RNPX_TRI
  return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_trsm_blocked(char trans, int n, int nrhs, const T* R, long ldr, T* B, long ldb, unsigned* flags,
                               unsigned epoch, unsigned* abortf, hipStream_t st) {
  if (trans != 'N' && trans != 'C') return hipErrorInvalidValue;
  return launch_trsm_tri<T>('U', trans, 'N', n, nrhs, R, ldr, B, ldb, flags, epoch, abortf, st);
}

// The inverses of the 64 x 64 diagonal blocks of an upper-triangular R
// (the last one may be smaller), written over the same blocks of X (the
// rest of X untouched).  One wave per block, the block staged in LDS; lane j
// back-substitutes column j of the inverse: x_j = 1 / r_jj, then for
// i = j-1 .. 0, x_i = -(sum_{k=i+1..j} r_ik x_k) / r_ii.
__global__ __launch_bounds__(64) void trtri_diag_kernel(int n, const double* __restrict__ R, long ldr,
                                                       double* __restrict__ X, long ldx) {
  __shared__ double Rs[64][65];
  __shared__ double Xs[64][65];
  const int lane = threadIdx.x;
  const int b0 = blockIdx.x * 64, nb = min(64, n - b0);
  for (int j = 0; j < nb; ++j) {
    Rs[lane][j] = lane < nb ? R[(size_t)(b0 + lane) + (size_t)(b0 + j) * ldr] : 0.0;
    Xs[lane][j] = 0.0;
  }
  __syncthreads();
  if (lane < nb) {
    const int j = lane;
    Xs[j][j] = 1.0 / Rs[j][j];
    for (int i = j - 1; i >= 0; --i) {
      double sacc = 0.0;
      for (int k = i + 1; k <= j; ++k) sacc += Rs[i][k] * Xs[k][j];
      Xs[i][j] = -sacc / Rs[i][i];
    }
  }
  __syncthreads();
  for (int j = 0; j < nb; ++j)
    if (lane < nb) X[(size_t)(b0 + lane) + (size_t)(b0 + j) * ldx] = Xs[lane][j];
}

hipError_t launch_trtri_diag(int n, const double* R, long ldr, double* X, long ldx, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(trtri_diag_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, n, R, ldr, X, ldx);
  return hipGetLastError();
}

template hipError_t launch_trsm_blocked<double>(char, int, int, const double*, long, double*, long, unsigned*, unsigned,
                                                unsigned*, hipStream_t);
template hipError_t launch_trsm_blocked<zd>(char, int, int, const zd*, long, zd*, long, unsigned*, unsigned, unsigned*,
                                            hipStream_t);
template hipError_t launch_trsm_tri<double>(char, char, char, int, int, const double*, long, double*, long, unsigned*,
                                            unsigned, unsigned*, hipStream_t);
template hipError_t launch_trsm_tri<zd>(char, char, char, int, int, const zd*, long, zd*, long, unsigned*, unsigned,
                                        unsigned*, hipStream_t);

}  // namespace rnpx
