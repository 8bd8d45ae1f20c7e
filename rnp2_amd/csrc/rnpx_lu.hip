// rnpx_lu.hip -- LU with partial pivoting (RNP/LA/LU.hpp) on gfx950.
//
// LU::Factor (LU.hpp:77-115) works in panels of 64 columns, each factored by
// one launch whose workgroups keep the panel resident and meet once per column
// c (Factor_unblocked, LU.hpp:52-75): every workgroup offers its candidate
// pivot (BLAS::MaximumIndex, BLAS_mix.hpp:798-810: the first row of largest
// |re|+|im|) with that row, every workgroup reduces the offers itself (ties to
// the lower row, so the result is the sequential scan's), scales its part of
// column c by 1/pivot and applies the rank-1 update to its rows.  Waits are
// bounded (2 s, abort flag).
//  * real panels (lu_row_panel_kernel): a thread keeps a row in registers,
//    rows move only when the panel is written back, and the hand-off needs no
//    fence (words that carry their column's tag);
//  * complex panels (lu_panel_kernel): a workgroup keeps 128 rows in LDS (a
//    complex row does not fit a thread's registers), rows are swapped there,
//    the hand-off is a counter with release and acquire.
// Both leave the list of the rows that moved; the interchanges are then
// applied to the columns outside the panel (lu_laswp_kernel: the rows of the
// list gathered through LDS), U12 = L11^-1 A12 by substitution
// (lu_trsm_kernel, L11 in LDS, a column per wave), and the trailing update
// A22 -= L21 U12 is a GEMM.
#include "rnpx_kernels.hpp"

#include <algorithm>
#include <cstdlib>

namespace rnpx {

namespace {

constexpr int kLuNB = 64;  // panel width (LU::Tuning::factor_block_size)

__device__ __forceinline__ double norm1_of(double x) { return fabs(x); }
__device__ __forceinline__ double norm1_of(zd x) { return fabs(x.x) + fabs(x.y); }

// (value, row) candidate order: the larger value, on ties the lower row.
// NaN values never win (the sequential scan's "cv > mv" never takes one).
__device__ __forceinline__ bool better(double va, int ia, double vb, int ib) {
  return (va > vb) || (va == vb && ia < ib);
}

// A complex entry in the panel's scratch.
__device__ __forceinline__ zd ld_part(const double* p) { return mkz(p[0], p[1]); }
__device__ __forceinline__ void st_part(double* p, zd v) {
  p[0] = v.x;
  p[1] = v.y;
}

}  // namespace

// A panel's interchanges (row c with pivs[c], in order) as the list of rows
// that end up elsewhere: moves[0] = count, then (from, to) pairs.  One
// workgroup of at least 64 threads.
__device__ __forceinline__ void compose_moves(const int* pivs, int jb, int* __restrict__ moves, int tid) {
  constexpr int NB = kLuNB, MAXT = kLuMaxMoves;
  __shared__ int rows[MAXT], src[MAXT], tp[NB], fq[NB];
  // Touched rows: the panel's first jb (slots 0..jb-1), then each pivot row
  // below them at its first appearance (slots jb.., in that order).
  if (tid < jb) {
    const int p = pivs[tid];
    int f = tid;
    if (p >= jb)
      for (int q = 0; q < tid; ++q)
        if (pivs[q] == p) {
          f = q;
          break;
        }
    fq[tid] = f;
  }
  __syncthreads();
  if (tid < jb) {  // its slot
    const int p = pivs[tid];
    int t = p;
    if (p >= jb) {
      int cnt = 0;
      for (int q = 0; q < fq[tid]; ++q) cnt += (pivs[q] >= jb && fq[q] == q) ? 1 : 0;
      t = jb + cnt;
      if (fq[tid] == tid) rows[t] = p;
    }
    tp[tid] = t;
    rows[tid] = tid;
  }
  __syncthreads();
  if (tid == 0) {
    int n = jb;
    for (int i = 0; i < jb; ++i) n = max(n, tp[i] + 1);
    for (int t = 0; t < n; ++t) src[t] = rows[t];
    for (int i = 0; i < jb; ++i) {  // the swaps in order, on the slot contents
      const int t2 = tp[i];
      const int x = src[i];
      src[i] = src[t2];
      src[t2] = x;
    }
    int cnt = 0;
    for (int t = 0; t < n; ++t)
      if (src[t] != rows[t]) {
        moves[1 + 2 * cnt] = src[t];
        moves[2 + 2 * cnt] = rows[t];
        ++cnt;
      }
    moves[0] = cnt;
  }
}

// ---------------------------------------------------------------------------
// Real panel: rows in registers.
// ---------------------------------------------------------------------------

// Largest of v across the wave (DPP within rows, then row broadcasts; the
// result of lane 63 broadcast).  No NaN among v.
__device__ __forceinline__ double wave_max_dpp(double v) {
#define RNPX_MAX_STEP(CTRL)                                                                       \
  v = fmax(v, mkd(__builtin_amdgcn_update_dpp(lo32(v), lo32(v), CTRL, 0xF, 0xF, false),            \
                  __builtin_amdgcn_update_dpp(hi32(v), hi32(v), CTRL, 0xF, 0xF, false)))
  RNPX_MAX_STEP(0x111);  // row_shr 1, 2, 4, 8
  RNPX_MAX_STEP(0x112);
  RNPX_MAX_STEP(0x114);
  RNPX_MAX_STEP(0x118);
  RNPX_MAX_STEP(0x142);  // row_bcast 15, 31
  RNPX_MAX_STEP(0x143);
#undef RNPX_MAX_STEP
  return readlane_t(v, 63);
}

// The lowest pos among the lanes whose v is mx (one, unless values tie).
__device__ __forceinline__ int lowest_of(double v, double mx, int pos, int* lane_out) {
  unsigned long long mk = __ballot(v == mx);
  int bl = (int)__ffsll(mk) - 1, bp = __builtin_amdgcn_readlane(pos, bl);
  mk &= mk - 1;
  while (mk) {
    const int l = (int)__ffsll(mk) - 1, q = __builtin_amdgcn_readlane(pos, l);
    if (q < bp) {
      bp = q;
      bl = l;
    }
    mk &= mk - 1;
  }
  *lane_out = bl;
  return bp;
}

// Hand-off words: 32 bits of payload under the column's 32-bit tag, stored and
// loaded as one 8-byte agent-scope access, so a word is either of this column
// or visibly not: no fence, no counter, one trip each way.
typedef unsigned long long Word;
__device__ __forceinline__ void put_word(Word* p, unsigned payload, unsigned tag) {
  __hip_atomic_store(p, ((Word)tag << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ Word get_word(const Word* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Thread t of workgroup g keeps row 512 g + t in registers and its current
// position among the panel's rows; nothing is swapped until the rows are
// written to their final positions.  The loop over columns runs in eights with
// the registers rotated by eight columns after each, so that every index is a
// constant; column 8b + s is register s, columns to its right are s + 1 ..
// 63 - 8b.  Per column: the largest entry of a wave by DPP, of the workgroup
// through LDS; its row to the slot of this column's parity (read by all before
// any workgroup can reach the column after next, which reuses it); each wave
// reads every workgroup's offer, then the winner's row.
// Bound by that hand-off's latency: 3.5 us per column at 8192 rows on 16
// workgroups, against 7.2 us for rows in LDS on 64 workgroups with row swaps, a
// counter, and a release and acquire per column.  With the list of moved rows
// below, 8192^2 and the solve of 16 right-hand sides take 37 ms.
__global__ __launch_bounds__(kLuRowThreads) void lu_row_panel_kernel(LuPanelArgs a) {
  constexpr int NB = kLuNB, NW = kLuRowThreads / 64;
  __shared__ double wv[NW], urow[NB], uw[NW][NB];
  __shared__ int wp[NW], wt[NW];
  RNPX_LU_GLOBAL(a);
  double* A = reinterpret_cast<double*>(a.A);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = blockIdx.x, G = gridDim.x, mp = a.mp, jb = a.jb;
  const int row = g * kLuRowThreads + tid;
  double r[NB];
  {
    const double* src = A + min(row, mp - 1);
#pragma unroll
    for (int c = 0; c < NB; ++c) r[c] = src[(size_t)min(c, jb - 1) * a.lda];
  }
  bool live = row < mp;  // not yet a pivot row
  int pos = live ? row : 0x7fffffff;
  int zero_last = -1;
  bool lost = false;  // a wait ran out: results are reported invalid
  for (int b = 0; b < 8; ++b) {
    const int ng = 8 - b;  // groups of eight columns still in play
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int c = 8 * b + s;
      if (c >= jb) break;
      const unsigned tag = a.tag0 + (unsigned)c;
      // this workgroup's offer; a NaN is never preferred, except that the scan
      // starts from row c and keeps a NaN there (offered as position -1)
      double v = live ? fabs(r[s]) : -2.0;
      int ps = pos;
      if (v != v) {
        const bool here = pos == c;
        v = here ? __builtin_inf() : -1.0;
        ps = here ? -1 : pos;
      }
      double mx = wave_max_dpp(v);
      int bl = 0, bp = 0x7fffffff;
      if (mx > -2.0) bp = lowest_of(v, mx, ps, &bl);
      if (lane == 0) {
        wv[wave] = mx;
        wp[wave] = bp;
        wt[wave] = wave * 64 + bl;
      }
      __syncthreads();
      int bt = wt[0];
      mx = wv[0];
      bp = wp[0];
#pragma unroll
      for (int w = 1; w < NW; ++w)
        if (better(wv[w], wp[w], mx, bp)) {
          mx = wv[w];
          bp = wp[w];
          bt = wt[w];
        }
      if (tid == bt) {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (q < ng) {
#pragma unroll
            for (int i = 0; i < 8; ++i) urow[8 * q + i] = r[8 * q + i];
          }
      }
      __syncthreads();
      const double* u = urow;
      if (G > 1) {
        Word* slots = a.ll + (size_t)(c & 1) * G * kLuSlotWords;
        Word* my = slots + (size_t)g * kLuSlotWords;
        if (wave == 0) {
          const double x = urow[lane];
          put_word(my + 2 * lane, lo32(x), tag);
          put_word(my + 2 * lane + 1, hi32(x), tag);
        } else if (wave == 1 && lane < 3) {
          put_word(my + 2 * NB + lane, lane == 0 ? lo32(mx) : lane == 1 ? hi32(mx) : (unsigned)bp, tag);
        }
        // every workgroup's offer, a lane per workgroup (two: up to 128)
        const uint64_t t0 = wall_clock64();
        double gv[2];
        int gp[2];
        while (true) {
          bool ok = true;
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            gv[k] = -3.0;
            gp[k] = 0x7fffffff;
            const int q = lane + 64 * k;
            if (q < G) {
              const Word* o = slots + (size_t)q * kLuSlotWords + 2 * NB;
              const Word w0 = get_word(o), w1 = get_word(o + 1), w2 = get_word(o + 2);
              ok = ok && (unsigned)(w0 >> 32) == tag && (unsigned)(w1 >> 32) == tag && (unsigned)(w2 >> 32) == tag;
              gv[k] = mkd((unsigned)w0, (unsigned)w1);
              gp[k] = (int)(unsigned)w2;
            }
          }
          if (__all(ok)) break;
          if (lost || __hip_atomic_load(a.abortf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u ||
              wall_clock64() - t0 > kBarrierTimeoutTicks) {
            __hip_atomic_store(a.abortf, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            lost = true;
            break;
          }
        }
        const bool second = better(gv[1], gp[1], gv[0], gp[0]);
        const double lv = second ? gv[1] : gv[0];
        const int lp = second ? gp[1] : gp[0];
        int wl = 0;
        bp = lowest_of(lv, wave_max_dpp(lv), lp, &wl);
        const int win = wl + 64 * __builtin_amdgcn_readlane((int)second, wl);
        const Word* o = slots + (size_t)min(win, G - 1) * kLuSlotWords + 2 * lane;
        Word x0, x1;
        while (true) {
          x0 = get_word(o);
          x1 = get_word(o + 1);
          if (__all((unsigned)(x0 >> 32) == tag && (unsigned)(x1 >> 32) == tag)) break;
          if (lost || wall_clock64() - t0 > 2 * kBarrierTimeoutTicks) {
            __hip_atomic_store(a.abortf, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            lost = true;
            break;
          }
        }
        uw[wave][lane] = mkd((unsigned)x0, (unsigned)x1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        u = uw[wave];
      }
      const int p = bp < 0 ? c : bp;
      const double piv = u[s];
      const bool nz = piv != 0.0;
      if (!nz) zero_last = c;
      if (g == 0 && tid == 0) a.piv[c] = p;
      if (live) {
        if (pos == p) {
          live = false;
          pos = c;
        } else {
          if (pos == c) pos = p;
          const double l = nz ? r[s] * recip_t(piv) : r[s];
          r[s] = l;
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (q < ng) {
#pragma unroll
              for (int i = 0; i < 8; ++i)
                if (8 * q + i > s) r[8 * q + i] = r[8 * q + i] + l * (0.0 - u[8 * q + i]);
            }
        }
      }
    }
    double t8[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) t8[i] = r[i];
#pragma unroll
    for (int i = 0; i < NB - 8; ++i) r[i] = r[i + 8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r[NB - 8 + i] = t8[i];
  }
  // Every workgroup's rows were in its registers before the last column's
  // offers, so the positions may be overwritten.
  if (row < mp && pos >= 0 && pos < mp) {
    double* dst = A + pos;
#pragma unroll
    for (int c = 0; c < NB; ++c)
      if (c < jb) dst[(size_t)c * a.lda] = r[c];
    if (pos != row) {
      const int e = (int)__hip_atomic_fetch_add((unsigned*)a.moves, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (e < kLuMaxMoves) {
        a.moves[1 + 2 * e] = row;
        a.moves[2 + 2 * e] = pos;
      }
    }
  }
  if (g == 0 && tid == 0) *a.zero_last = zero_last;
}

// Scratch layout (doubles): part[2][G][kLuSlot] candidate slots (value,
// row, then the row's kLuNB entries), rowc[2][2*kLuNB] (row c).
constexpr int kLuSlot = 2 + 2 * kLuNB;

template <int RW>
__global__ __launch_bounds__(256) void lu_panel_kernel(LuPanelArgs a) {
  using T = zd;
  constexpr int NB = kLuNB, LDS_S = NB + 1;
  __shared__ T Sl[RW][LDS_S];
  __shared__ T ubuf[NB], ocbuf[NB];
  __shared__ double redv[4];
  __shared__ int redi[4], redw[4];
  __shared__ int pw[2];
  RNPX_LU_GLOBAL(a);
  T* A = reinterpret_cast<T*>(a.A);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = blockIdx.x, G = gridDim.x;
  const int gr0 = g * RW, mp = a.mp, jb = a.jb;
  const T zero = S<T>::zero();

  // Stage this workgroup's rows (zero padding beyond mp and jb).
  for (int e = tid; e < RW * NB; e += 256) {
    const int r = e % RW, c = e / RW;
    T v = zero;
    if (gr0 + r < mp && c < jb) v = A[(size_t)(gr0 + r) + (size_t)c * a.lda];
    Sl[r][c] = v;
  }
  __syncthreads();

  __shared__ int pivs[NB];
  int zero_last = -1;
  for (int c = 0; c < jb; ++c) {
    const int par = c & 1;
    double* part = a.part + (size_t)par * G * kLuSlot;
    double* rowc = a.rowc + (size_t)par * 2 * NB;
    // 1. local candidate
    double bv = -2.0;
    int bi = 0x7fffffff;
    for (int r = tid; r < RW; r += 256) {
      const int gr = gr0 + r;
      if (gr >= c && gr < mp) {
        double v = norm1_of(Sl[r][c]);
        if (v != v) v = -1.0;  // NaN: never preferred
        if (better(v, gr, bv, bi)) {
          bv = v;
          bi = gr;
        }
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const double ov = __shfl_xor(bv, off, 64);
      const int oi = __shfl_xor(bi, off, 64);
      if (better(ov, oi, bv, bi)) {
        bv = ov;
        bi = oi;
      }
    }
    if (lane == 0) {
      redv[wave] = bv;
      redi[wave] = bi;
    }
    __syncthreads();
    bv = redv[0];
    bi = redi[0];
    for (int w = 1; w < 4; ++w)
      if (better(redv[w], redi[w], bv, bi)) {
        bv = redv[w];
        bi = redi[w];
      }
    // 2. candidate slot (and row c from its owner), then arrive
    double* my = part + (size_t)g * kLuSlot;
    if (tid == 0) {
      my[0] = bv;
      my[1] = (double)bi;
    }
    if (bi != 0x7fffffff)
      for (int q = tid; q < NB; q += 256) st_part(my + 2 + 2 * q, Sl[bi - gr0][q]);
    if (c >= gr0 && c < gr0 + RW)
      for (int q = tid; q < NB; q += 256) st_part(rowc + 2 * q, Sl[c - gr0][q]);
    // every workgroup waits for all the candidates, then reduces them in
    // workgroup order itself (no second hand-off)
    unsigned* cnt = a.sync + 2 * c;
    wait_stores();
    __syncthreads();
    if (tid == 0) {
      release_agent();
      __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint64_t t0 = wall_clock64();
      while (__hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < (unsigned)G) {
        if (__hip_atomic_load(a.abortf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) break;
        if (wall_clock64() - t0 > kBarrierTimeoutTicks) {
          __hip_atomic_store(a.abortf, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    // Old row c does not depend on the pivot: its loads go out with the
    // candidates' (one round trip fewer per column).
    static_assert(NB <= 256, "a thread per entry of row c");
    T ocv = zero;
    if (tid < NB) ocv = ld_part(rowc + 2 * tid);
    {
      double v = -2.0;
      int i = 0x7fffffff, w = -1;
      for (int q = tid; q < G; q += 256) {
        const double* o = part + (size_t)q * kLuSlot;
        const double ov = o[0];
        const int oi = (int)o[1];
        if (better(ov, oi, v, i)) {
          v = ov;
          i = oi;
          w = q;
        }
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        const double ov = __shfl_xor(v, off, 64);
        const int oi = __shfl_xor(i, off, 64);
        const int ow = __shfl_xor(w, off, 64);
        if (better(ov, oi, v, i)) {
          v = ov;
          i = oi;
          w = ow;
        }
      }
      if (lane == 0) {
        redv[wave] = v;
        redi[wave] = i;
        redw[wave] = w;
      }
      if (tid < NB) ocbuf[tid] = ocv;
      __syncthreads();
      if (tid == 0) {
        double bv2 = redv[0];
        int bi2 = redi[0], bw2 = redw[0];
        for (int q = 1; q < 4; ++q)
          if (better(redv[q], redi[q], bv2, bi2)) {
            bv2 = redv[q];
            bi2 = redi[q];
            bw2 = redw[q];
          }
        // The sequential scan starts from row c: a NaN there is kept.
        const T xc = ocbuf[c];
        const double nc = norm1_of(xc);
        if (nc != nc || bi2 == 0x7fffffff) {
          bi2 = c;
          bw2 = -1;
        }
        pw[0] = bi2;
        pw[1] = bw2;
      }
      __syncthreads();
    }
    const int p = pw[0], w = pw[1];
    // 3. pivot row u: the winner's row, or row c itself (already in ocbuf)
    if (tid < NB) ubuf[tid] = (w >= 0) ? ld_part(part + (size_t)w * kLuSlot + 2 + 2 * tid) : ocbuf[tid];
    __syncthreads();
    if (c >= gr0 && c < gr0 + RW)
      for (int q = tid; q < NB; q += 256) Sl[c - gr0][q] = ubuf[q];
    if (p != c && p >= gr0 && p < gr0 + RW)
      for (int q = tid; q < NB; q += 256) Sl[p - gr0][q] = ocbuf[q];
    __syncthreads();
    const T piv = ubuf[c];
    const bool nz = !S<T>::is_zero(piv);
    if (!nz) zero_last = c;
    const T rinv = nz ? recip_t(piv) : S<T>::one();
    // scale column c of the rows below c, then the rank-1 update
    for (int r = tid; r < RW; r += 256) {
      const int gr = gr0 + r;
      if (gr > c && gr < mp && nz) Sl[r][c] = Sl[r][c] * rinv;
    }
    __syncthreads();
    const int ncols = jb - c - 1;
    for (int e = tid; e < RW * ncols; e += 256) {
      const int r = e % RW, cc = c + 1 + e / RW;
      const int gr = gr0 + r;
      if (gr > c && gr < mp) Sl[r][cc] = Sl[r][cc] + Sl[r][c] * (zero - ubuf[cc]);
    }
    if (tid == 0) pivs[c] = p;
    if (g == 0 && tid == 0) a.piv[c] = p;
    __syncthreads();
  }
  // Write the panel back.
  for (int e = tid; e < RW * NB; e += 256) {
    const int r = e % RW, c = e / RW;
    if (gr0 + r < mp && c < jb) A[(size_t)(gr0 + r) + (size_t)c * a.lda] = Sl[r][c];
  }
  if (g == 0) {
    if (tid == 0) *a.zero_last = zero_last;
    compose_moves(pivs, jb, a.moves, tid);
  }
}

// The interchanges of one panel (its list of moved rows, relative to row j)
// applied to ncols columns starting at column c0.  A workgroup takes CW
// columns: 32, or 8 where only the next panel's 64 columns are due and one
// workgroup would do them all.  Bound by the scattered entries (a cache line
// per row and column, twice).
template <typename T, int CW>
__global__ __launch_bounds__(256) void lu_laswp_kernel(int j, const int* __restrict__ moves, T* A, long lda, int c0,
                                                       int ncols) {
  constexpr int MAXT = kLuMaxMoves;
  __shared__ T buf[CW][MAXT + 1];
  const int tid = threadIdx.x, t = tid % MAXT;
  const int n = min(moves[0], MAXT);
  const int cb = c0 + blockIdx.x * CW, nc = min(CW, c0 + ncols - cb);
  const bool on = t < n;
  const int src = on ? j + moves[1 + 2 * t] : 0, dst = on ? j + moves[2 + 2 * t] : 0;
#pragma unroll
  for (int q0 = 0; q0 < CW; q0 += 256 / MAXT) {
    const int q = q0 + tid / MAXT;
    if (on && q < nc) buf[q][t] = A[(size_t)src + (size_t)(cb + q) * lda];
  }
  __syncthreads();
#pragma unroll
  for (int q0 = 0; q0 < CW; q0 += 256 / MAXT) {
    const int q = q0 + tid / MAXT;
    if (on && q < nc) A[(size_t)dst + (size_t)(cb + q) * lda] = buf[q][t];
  }
}

// U12 = L11^-1 A12 (L11 the jb x jb unit lower triangle at L, A12 jb x ncols
// at B): a wave per column, lane = row, forward substitution with x_k
// broadcast by v_readlane and L11 read from LDS (each lane its own row).
// A wave takes CPW columns: 4, or 1 where only the next panel's 64 columns are
// due (the substitution is a chain of 64 LDS reads per column).
template <typename T, int CPW>
__global__ __launch_bounds__(256) void lu_trsm_kernel(int jb, const T* __restrict__ L, long ldl, T* B, long ldb,
                                                      int ncols) {
  constexpr int NB = kLuNB;
  __shared__ T Ls[NB][NB + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < NB * NB; e += 256) {
    const int r = e % NB, c = e / NB;
    Ls[r][c] = (r < jb && c < jb && r > c) ? L[(size_t)r + (size_t)c * ldl] : S<T>::zero();
  }
  __syncthreads();
  const int cb = blockIdx.x * 4 * CPW;
  for (int q = wave; q < 4 * CPW; q += 4) {
    const int col = cb + q;
    if (col >= ncols) break;
    T* b = B + (size_t)col * ldb;
    T x = (lane < jb) ? b[lane] : S<T>::zero();
#pragma unroll 8
    for (int k = 0; k < jb - 1; ++k) {
      const T xk = readlane_t(x, k);
      if (lane > k) x = x - Ls[lane][k] * xk;
    }
    if (lane < jb) b[lane] = x;
  }
}

// Row gather b(i, :) = a(src[i], :) for an n x nrhs block (LU::Solve's
// interchanges composed into one permutation on the host).
template <typename T>
__global__ __launch_bounds__(256) void lu_gather_kernel(int n, int nrhs, const int* __restrict__ src,
                                                        const T* __restrict__ X, long ldx, T* __restrict__ Y,
                                                        long ldy) {
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long long)n * nrhs) return;
  const int i = (int)(e % n), c = (int)(e / n);
  Y[(size_t)i + (size_t)c * ldy] = X[(size_t)src[i] + (size_t)c * ldx];
}

// RefineSolution's denominators: rw_i = |b_i| + sum_k |A(i,k)| |x_k| for
// op "N" (a thread per row, coalesced down the columns) and
// rw_k = |b_k| + sum_i |A(i,k)| |x_i| for "T"/"C" (a wave per column);
// |.| is |re| + |im| (Traits<T>::norm1).
template <typename T>
__global__ __launch_bounds__(256) void lu_absmv_kernel(int n, int transposed, const T* __restrict__ A, long lda,
                                                       const T* __restrict__ x, const T* __restrict__ b,
                                                       double* __restrict__ rw) {
  if (!transposed) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int k = 0; k < n; ++k) s += norm1_of(A[(size_t)i + (size_t)k * lda]) * norm1_of(x[k]);
    rw[i] = norm1_of(b[i]) + s;
  } else {
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (k >= n) return;
    double s = 0.0;
    for (int i = lane; i < n; i += 64) s += norm1_of(A[(size_t)i + (size_t)k * lda]) * norm1_of(x[i]);
    s = wave_sum(s);
    if (lane == 0) rw[k] = norm1_of(b[k]) + s;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void lu_axpy_kernel(int n, const T* __restrict__ x, T* __restrict__ y) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) y[i] = y[i] + x[i];
}

template <typename T>
hipError_t launch_lu_absmv(int n, bool transposed, const T* A, long lda, const T* x, const T* b, double* rw,
                           hipStream_t st) {
  if (n < 0 || lda < std::max(1, n)) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  if (!transposed)
    hipLaunchKernelGGL((lu_absmv_kernel<T>), dim3((n + 255) / 256), dim3(256), 0, st, n, 0, A, lda, x, b, rw);
  else
    hipLaunchKernelGGL((lu_absmv_kernel<T>), dim3((n + 3) / 4), dim3(256), 0, st, n, 1, A, lda, x, b, rw);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_lu_axpy(int n, const T* x, T* y, hipStream_t st) {
  if (n < 0) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL((lu_axpy_kernel<T>), dim3((n + 255) / 256), dim3(256), 0, st, n, x, y);
  return hipGetLastError();
}

int lu_panel_rows(int mp, int max_groups, int cplx) {
  // Real: 512 rows per workgroup (at most 128 workgroups offer a candidate).
  if (!cplx) return mp <= 256 * max_groups && mp <= 128 * kLuRowThreads ? kLuRowThreads : 0;
  // Complex: 128-row blocks; RNPX_LU_PANEL_RW (64 or 128) overrides, for
  // complex panels only.
  static const int pref = [] {
    const char* e = getenv("RNPX_LU_PANEL_RW");
    return e ? atoi(e) : 0;
  }();
  if ((pref == 64 || pref == 128) && (mp + pref - 1) / pref <= max_groups) return pref;
  return (mp + 127) / 128 <= max_groups ? 128 : 0;
}

template <typename T>
hipError_t launch_lu_panel(const LuPanelArgs& a, int rw, hipStream_t st) {
  if (a.mp <= 0 || a.jb <= 0 || a.jb > kLuNB || a.jb > a.mp || a.lda < a.mp || !a.abortf || !a.piv || !a.zero_last ||
      !a.moves || rw <= 0)
    return hipErrorInvalidValue;
  const int G = (a.mp + rw - 1) / rw;
  if (G < 1 || G > 256) return hipErrorInvalidValue;
  if constexpr (!S<T>::cplx) {
    if (rw != kLuRowThreads || G > 128 || !a.ll) return hipErrorInvalidValue;
    hipLaunchKernelGGL(lu_row_panel_kernel, dim3(G), dim3(kLuRowThreads), 0, st, a);
  } else {
    if (!a.sync || !a.part || !a.rowc) return hipErrorInvalidValue;
    if (rw == 64) hipLaunchKernelGGL((lu_panel_kernel<64>), dim3(G), dim3(256), 0, st, a);
    else if (rw == 128) hipLaunchKernelGGL((lu_panel_kernel<128>), dim3(G), dim3(256), 0, st, a);
    else return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_lu_laswp(int j, const int* moves, T* A, long lda, int c0, int ncols, hipStream_t st) {
  if (j < 0 || c0 < 0 || ncols < 0 || !moves) return hipErrorInvalidValue;
  if (ncols == 0) return hipSuccess;
  if (ncols <= kLuNB)
    hipLaunchKernelGGL((lu_laswp_kernel<T, 8>), dim3((ncols + 7) / 8), dim3(256), 0, st, j, moves, A, lda, c0, ncols);
  else
    hipLaunchKernelGGL((lu_laswp_kernel<T, 32>), dim3((ncols + 31) / 32), dim3(256), 0, st, j, moves, A, lda, c0,
                       ncols);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_lu_trsm(int jb, const T* L, long ldl, T* B, long ldb, int ncols, hipStream_t st) {
  if (jb <= 0 || jb > kLuNB || ncols < 0 || ldl < jb || ldb < jb) return hipErrorInvalidValue;
  if (ncols == 0) return hipSuccess;
  if (ncols <= kLuNB)
    hipLaunchKernelGGL((lu_trsm_kernel<T, 1>), dim3((ncols + 3) / 4), dim3(256), 0, st, jb, L, ldl, B, ldb, ncols);
  else
    hipLaunchKernelGGL((lu_trsm_kernel<T, 4>), dim3((ncols + 15) / 16), dim3(256), 0, st, jb, L, ldl, B, ldb, ncols);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_lu_gather(int n, int nrhs, const int* src, const T* X, long ldx, T* Y, long ldy, hipStream_t st) {
  if (n < 0 || nrhs < 0 || ldx < std::max(1, n) || ldy < std::max(1, n)) return hipErrorInvalidValue;
  const long long total = (long long)n * nrhs;
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL((lu_gather_kernel<T>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, n, nrhs, src, X,
                     ldx, Y, ldy);
  return hipGetLastError();
}

#define RNPX_INST(T)                                                                                    \
  template hipError_t launch_lu_panel<T>(const LuPanelArgs&, int, hipStream_t);                         \
  template hipError_t launch_lu_laswp<T>(int, const int*, T*, long, int, int, hipStream_t);             \
  template hipError_t launch_lu_trsm<T>(int, const T*, long, T*, long, int, hipStream_t);               \
  template hipError_t launch_lu_gather<T>(int, int, const int*, const T*, long, T*, long, hipStream_t);      \
  template hipError_t launch_lu_absmv<T>(int, bool, const T*, long, const T*, const T*, double*, hipStream_t); \
  template hipError_t launch_lu_axpy<T>(int, const T*, T*, hipStream_t);
RNPX_INST(double)
RNPX_INST(zd)
#undef RNPX_INST

}  // namespace rnpx
