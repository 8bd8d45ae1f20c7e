// rnpx_tfactor.hip -- the T-factor kernel (the larft analogue,
// Reflector::GenerateBlockTr "F","C", RNP/LA/Reflector.hpp:573-626) and the
// Grams that feed it when V comes from a stored factorization (QR::MultQ /
// QR::GenerateQ recompute T per block, QR.hpp:395, 557; here every block's T
// is formed before the first is applied, since all of V is there).
//
// RNP builds T column by column: T(0:c,c) = -tau_c T(0:c,0:c) V^H v_c.
// Row j of that recurrence only touches row j of T, so here it runs as:
//   1. leaf blocks of 16 on the diagonal, one thread per row, each thread
//      walking its own row of the leaf with the recurrence above;
//   2. recursive doubling: for adjacent blocks, T12 = -T11 (V1^H V2) T22,
//      which is the same product H1 H2 written block-wise.
// Both use the Gram matrix G = V^H V (strict upper part) and tau, all in LDS.
// A tau_c == 0 column comes out zero, as at Reflector.hpp:584-587.
#include "rnpx_kernels.hpp"

#include <algorithm>

namespace rnpx {

// One workgroup per NB-column leaf of a set of w-column blocks (w a multiple of
// NB; w = NB for a single T): leaf l belongs to block l NB / w, reads the
// diagonal NB x NB part of that block's Gram (leading dimension ldg, blocks
// gstride apart) and writes its w x NB strip of the block's T (zero outside the
// diagonal part: the products that join two leaves fill in the part above).
// kcols columns in all (a leaf beyond them: zeros).  Latency-bound (23 us, one leaf or fifty), so every
// leaf of a stored factorization goes in one launch.
template <typename T, int NB>
__global__ __launch_bounds__(256) void tfactor_kernel(const T* __restrict__ gram, int ldg, size_t gstride, int w,
                                                       int kcols, T* __restrict__ Tout, int ldt, size_t tstride,
                                                       const unsigned* run_if) {
  if (run_if && *run_if == 0u) return;
  const int leaf0 = blockIdx.x * NB, blk = leaf0 / w, off = leaf0 - blk * w;
  const int k = min(NB, kcols - leaf0);
  gram += blk * gstride + (size_t)off * ldg + off;
  Tout += blk * tstride + (size_t)off * ldt;
  constexpr int LEAF = 16;
  __shared__ T Gs[NB][NB + 1];  // Gs[l][c] = G(l,c), l < c; diagonal = tau
  __shared__ T Ts[NB][NB + 1];
  __shared__ T Xs[NB / 2][NB / 2 + 1];
  const int tid = threadIdx.x;
  for (int e = tid; e < NB * NB; e += 256) {
    const int l = e % NB, c = e / NB;
    Gs[l][c] = (l <= c && c < k) ? gram[(size_t)l + (size_t)c * ldg] : S<T>::zero();
    Ts[l][c] = S<T>::zero();
  }
  __syncthreads();
  // 1. leaves
  if (tid < k) {
    const int j = tid;
    const int b1 = min((j / LEAF + 1) * LEAF, k);
    Ts[j][j] = Gs[j][j];
    for (int c = j + 1; c < b1; ++c) {
      T s = S<T>::zero();
      for (int l = j; l < c; ++l) s = s + Ts[j][l] * Gs[l][c];
      Ts[j][c] = (S<T>::zero() - Gs[c][c]) * s;
    }
  }
  __syncthreads();
  // 2. doubling: blocks of h -> 2h
  for (int h = LEAF; h < k; h *= 2) {
    const int npairs = (k + 2 * h - 1) / (2 * h);
    // X = G12 * T22 for every pair: X(r, c) = sum_{l in blk2, l <= c} G(i1+r, l) T(l, c)
    for (int e = tid; e < npairs * h * h; e += 256) {
      const int pr = e / (h * h), rc = e % (h * h);
      const int r = rc % h, cc = rc / h;
      const int i1 = pr * 2 * h, i2 = i1 + h;
      const int c = i2 + cc;
      T s = S<T>::zero();
      if (i2 < k && c < k) {
        for (int l = i2; l <= c; ++l) s = s + Gs[i1 + r][l] * Ts[l][c];
      }
      // Xs is (NB/2) x (NB/2); pairs are packed along the rows
      if (pr * h + r < NB / 2 && cc < NB / 2) Xs[pr * h + r][cc] = s;
    }
    __syncthreads();
    // T12 = -T11 * X
    for (int e = tid; e < npairs * h * h; e += 256) {
      const int pr = e / (h * h), rc = e % (h * h);
      const int r = rc % h, cc = rc / h;
      const int i1 = pr * 2 * h, i2 = i1 + h;
      const int c = i2 + cc;
      if (i2 < k && c < k) {
        T s = S<T>::zero();
        for (int l = r; l < h; ++l) s = s + Ts[i1 + r][i1 + l] * Xs[pr * h + l][cc];
        Ts[i1 + r][c] = S<T>::zero() - s;
      }
    }
    __syncthreads();
  }
  for (int e = tid; e < w * NB; e += 256) {
    const int l = e % w, c = e / w, d = l - off;
    Tout[(size_t)l + (size_t)c * ldt] = (d >= 0 && d < NB) ? Ts[d][c] : S<T>::zero();
  }
}

template <typename T>
hipError_t launch_tfactor(const T* gram, int ldg, int k, int nb, T* Tout, int ldt, hipStream_t st,
                          const unsigned* run_if) {
  if (k < 0 || k > nb || ldg < nb || ldt < nb) return hipErrorInvalidValue;
  if (nb == 16)
    hipLaunchKernelGGL((tfactor_kernel<T, 16>), dim3(1), dim3(256), 0, st, gram, ldg, (size_t)0, nb, k, Tout, ldt,
                       (size_t)0, run_if);
  else if (nb == 32)
    hipLaunchKernelGGL((tfactor_kernel<T, 32>), dim3(1), dim3(256), 0, st, gram, ldg, (size_t)0, nb, k, Tout, ldt,
                       (size_t)0, run_if);
  else if (nb == 64)
    hipLaunchKernelGGL((tfactor_kernel<T, 64>), dim3(1), dim3(256), 0, st, gram, ldg, (size_t)0, nb, k, Tout, ldt,
                       (size_t)0, run_if);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

template <typename T>
hipError_t launch_tfactor_blocks(const T* gram, int w, int k, T* Tout, hipStream_t st) {
  if (k < 1) return hipErrorInvalidValue;
  const size_t ws = (size_t)w * w;
  if (w == 32)
    hipLaunchKernelGGL((tfactor_kernel<T, 32>), dim3((k + 31) / 32), dim3(256), 0, st, gram, w, ws, w, k, Tout, w, ws,
                       (const unsigned*)nullptr);
  else if (w == 64 || w == 128)
    hipLaunchKernelGGL((tfactor_kernel<T, 64>), dim3((k + w - 1) / w * (w / 64)), dim3(256), 0, st, gram, w, ws, w, k, Tout, w, ws,
                       (const unsigned*)nullptr);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

// gram[b](j, c), j < c, of every block from its ns row slices (added in slice
// order), tau on the diagonal, zero below it and beyond the k columns.
template <typename T>
__global__ void gram_sum_blocks_kernel(int k, int w, int ns, const T* __restrict__ part, const T* __restrict__ tau,
                                       T* __restrict__ gram) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
  if (e >= w * w) return;
  const size_t ws = (size_t)w * w;
  const int j = e % w, c = e / w, col = b * w + c;
  T s = S<T>::zero();
  if (col < k && j < c)
    s = sum_strided(part + (size_t)b * ns * ws + e, ns, ws);
  else if (col < k && j == c)
    s = tau[col];
  gram[b * ws + e] = s;
}

int gram_blocks_slices(int n, int k, int w, int most, int* kslice) {
  const int nblk = (k + w - 1) / w, tiles = (w <= 64 ? 1 : 4) * nblk;
  // about three workgroups per CU in all, slices of at least 32 rows (16 rows
  // of a slice take about a microsecond, whatever else is idle) and at most
  // `most` of them (their sum takes about half a microsecond for eight)
  int ns = std::max(1, std::min({most, n / 32, 768 / tiles}));
  *kslice = ((n + ns - 1) / ns + 15) / 16 * 16;
  return (n + *kslice - 1) / *kslice;
}

template <typename T>
hipError_t launch_gram_blocks(int n, int k, int w, int most, const T* V, long ldv, const T* tau, T* gram, T* part,
                              hipStream_t st) {
  if (k < 1 || n < k || ldv < n) return hipErrorInvalidValue;
  int kslice = 0;
  const int ns = gram_blocks_slices(n, k, w, most, &kslice), full = k / w, rest = k - full * w;
  const size_t ws = (size_t)w * w;
  const int nblk = full + (rest > 0), wlast = rest > 0 ? rest : w;
  if constexpr (S<T>::cplx)
    RNPX_LAUNCH_CHECK(zgemm_gram_batched(n, w, wlast, V, ldv, kslice, ns, part, nblk, st));
  else
    RNPX_LAUNCH_CHECK(dgemm_gram_batched(n, w, wlast, V, ldv, kslice, ns, part, nblk, st));
  hipLaunchKernelGGL((gram_sum_blocks_kernel<T>), dim3((unsigned)((ws + 255) / 256), nblk), dim3(256), 0,
                     st, k, w, ns, part, tau, gram);
  return hipGetLastError();
}

#define RNPX_TF_INST(T)                                                                                       \
  template hipError_t launch_tfactor<T>(const T*, int, int, int, T*, int, hipStream_t, const unsigned*);      \
  template hipError_t launch_tfactor_blocks<T>(const T*, int, int, T*, hipStream_t);                          \
  template hipError_t launch_gram_blocks<T>(int, int, int, int, const T*, long, const T*, T*, T*, hipStream_t);
RNPX_TF_INST(double)
RNPX_TF_INST(zd)
#undef RNPX_TF_INST

}  // namespace rnpx
