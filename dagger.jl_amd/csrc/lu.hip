// LU with partial pivoting (RowMaximum) and without (NoPivot) on a tiled
// matrix: the panel and row-swap tile operations of Dagger's lu!
// (src/array/lu.jl:5-55 NoPivot, :221-371 RowMaximum); the TRSM and GEMM
// tile operations of the same loop nests run on the existing kernels.
//
// Panel (block column k, tiles k..mt-1, a tall Mp x W matrix): as the
// reference's CPU path does (factor_panel_lapack!, :160-204), the panel's
// tiles are gathered into one contiguous column-major buffer, factored by
// LAPACK's getrf semantics (partial pivoting by maximum magnitude, the
// first maximum on ties, a zero pivot sets info and skips the scaling) and
// scattered back.  The factorization is LAPACK getrf2's recursion:
//   left half (recursively); its row swaps applied to the right half;
//   A12 := L11^-1 A12 (unit lower TRSM); A22 -= A21 A12 (GEMM);
//   right half (recursively); its row swaps applied to the left half,
// with leaves of 32 columns factored in one workgroup, from registers where
// the rows fit.  Row swaps of the other block columns (swaprows_trail!,
// :239-262) apply the permutation that the panel's pivots amount to.
#include <algorithm>
#include <limits>
#include <type_traits>
#include "dm_internal.h"

namespace dm {

constexpr int LU_LEAF = 32;       // columns of a leaf panel
constexpr int LU_THREADS = 1024;  // the one workgroup of a leaf in memory
constexpr int LR_THREADS = 512;   // and of a leaf in registers

// Global row r of a tiled block column starting at tile row 0 of `base`
// (tiles of mb rows, all `cols` wide, each with ld = its row count).
template <typename T>
__device__ __forceinline__ T* tiled_at(T* base, int64_t rows_total, int mb, int cols, int64_t r,
                                       int c) {
  const int64_t t = r / mb;
  const int64_t lr = r - t * mb;
  const int64_t ld = std::min<int64_t>(mb, rows_total - t * mb);
  return base + t * (int64_t)mb * cols + (int64_t)c * ld + lr;
}

// Tiled block-column region <-> contiguous Mp x W buffer (ld = Mp).
template <typename T>
__global__ void panel_pack_kernel(T* __restrict__ dst, T* __restrict__ tiles, int64_t Mp, int W,
                                  int mb, int unpack) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= Mp * W) return;
  const int c = (int)(i / Mp);
  const int64_t r = i - (int64_t)c * Mp;
  T* t = tiled_at(tiles, Mp, mb, W, r, c);
  if (unpack) *t = dst[i];
  else dst[i] = *t;
}

// A leaf with more rows than registers hold: factor columns [c0, c0 + nc) of
// the contiguous panel P (Mp x W, ld = Mp), rows [c0, Mp), in memory (32
// columns of 32000 rows: 5.95 ms in FP64, bound by the passes over the leaf).
// For each column j, pick the pivot (maximum |P[r, j]|, r >= j, first on ties)
// when `pivot`, swap rows j and p within the leaf's columns, scale the column
// below the diagonal by the pivot's reciprocal (skipped for a zero pivot, which
// sets *info to j + 1 if unset) and update the rest of the leaf.  piv[j]
// receives p (0-based, panel rows).
template <typename T>
__global__ __launch_bounds__(LU_THREADS) void getf2_leaf_kernel(T* __restrict__ P, int64_t Mp,
                                                                int c0, int nc,
                                                                int* __restrict__ piv,
                                                                int* __restrict__ info,
                                                                const int* __restrict__ abort,
                                                                int pivot) {
  __shared__ T bval[LU_THREADS / 64];
  __shared__ int64_t bidx[LU_THREADS / 64];
  __shared__ int64_t pv;
  if (abort && *abort) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t ld = Mp;
  for (int j = c0; j < c0 + nc && j < Mp; ++j) {
    T* colj = P + (int64_t)j * ld;
    if (pivot) {
      // per-thread maximum over rows j + tid, j + tid + 1024, ... (first on ties)
      T best = T(-1);
      int64_t bi = Mp;
      for (int64_t r = j + tid; r < Mp; r += LU_THREADS) {
        const T v = fabs(colj[r]);
        if (v > best) { best = v; bi = r; }
      }
      // wave then workgroup reduction: larger value, then smaller row
      for (int off = 32; off > 0; off >>= 1) {
        const T ov = __shfl_down(best, off, 64);
        const int64_t oi = __shfl_down(bi, off, 64);
        if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
      }
      if (lane == 0) { bval[wave] = best; bidx[wave] = bi; }
      __syncthreads();
      if (tid == 0) {
        T b = bval[0];
        int64_t x = bidx[0];
        for (int w = 1; w < LU_THREADS / 64; ++w)
          if (bval[w] > b || (bval[w] == b && bidx[w] < x)) { b = bval[w]; x = bidx[w]; }
        if (x >= Mp) x = j;  // an all-NaN column keeps its row
        pv = x;
        piv[j] = (int)x;
      }
      __syncthreads();
      const int64_t p = pv;
      if (p != j)
        for (int c = c0 + tid; c < c0 + nc; c += LU_THREADS) {
          T* a = P + (int64_t)c * ld;
          const T t = a[j];
          a[j] = a[p];
          a[p] = t;
        }
    } else if (tid == 0) {
      piv[j] = j;
    }
    __syncthreads();
    const T d = colj[j];
    if (d == T(0)) {
      if (tid == 0 && info && *info == 0) *info = j + 1;
    } else if (fabs(d) >= std::numeric_limits<T>::min()) {
      const T inv = T(1) / d;  // LAPACK getf2: scale by the reciprocal
      for (int64_t r = j + 1 + tid; r < Mp; r += LU_THREADS) colj[r] *= inv;
    } else {                   // ... or divide when it would overflow
      for (int64_t r = j + 1 + tid; r < Mp; r += LU_THREADS) colj[r] /= d;
    }
    __syncthreads();
    // rank-1 update of the leaf's remaining columns
    const int rest = c0 + nc - (j + 1);
    if (rest > 0) {
      for (int64_t r = j + 1 + tid; r < Mp; r += LU_THREADS) {
        const T l = colj[r];
        for (int c = j + 1; c < c0 + nc; ++c) {
          T* a = P + (int64_t)c * ld;
          a[r] -= l * a[j];
        }
      }
    }
    __syncthreads();
  }
}

// Value of lane l (uniform) in every lane.
template <typename T> __device__ __forceinline__ T wave_bcast(T v, int l) {
  if (sizeof(T) == 8) {
    const long long b = __builtin_bit_cast(long long, (double)v);
    const int lo = __builtin_amdgcn_readlane((int)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return (T)__builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
  }
  return (T)__builtin_bit_cast(float,
                               __builtin_amdgcn_readlane(__builtin_bit_cast(int, (float)v), l));
}

// Largest of the 64 lanes' values, in every lane (emulated lane by lane on the host).
template <typename T> __device__ __forceinline__ T wave_max(T v) {
#ifdef __HIP_DEVICE_COMPILE__
  auto step = [&](auto ctrl) {
    T o;
    if (sizeof(T) == 8) {
      const long long b = __builtin_bit_cast(long long, (double)v);
      const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, ctrl.value, 0xf, 0xf, false);
      const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), ctrl.value, 0xf,
                                                 0xf, false);
      o = (T)__builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
    } else {
      const int b = __builtin_bit_cast(int, (float)v);
      o = (T)__builtin_bit_cast(
          float, __builtin_amdgcn_update_dpp(b, b, ctrl.value, 0xf, 0xf, false));
    }
    v = fmax(v, o);
  };
  step(std::integral_constant<int, 0x111>{});  // row_shr 1, 2, 4, 8: lane 15 of each row of 16
  step(std::integral_constant<int, 0x112>{});
  step(std::integral_constant<int, 0x114>{});
  step(std::integral_constant<int, 0x118>{});
  step(std::integral_constant<int, 0x142>{});  // row_bcast 15, 31: lane 63
  step(std::integral_constant<int, 0x143>{});
  return wave_bcast(v, 63);
#else
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl(v, (threadIdx.x & 63) ^ off, 64));
  return v;
#endif
}

// Smallest key of the wave, in every lane; lanes without one hold INT_MAX.
__device__ __forceinline__ int wave_first(int key) {
#ifdef __HIP_DEVICE_COMPILE__
  unsigned long long m = __builtin_amdgcn_ballot_w64(key != std::numeric_limits<int>::max());
  int best = std::numeric_limits<int>::max();
  while (m) {  // one lane but for ties
    best = std::min(best, __builtin_amdgcn_readlane(key, __builtin_ctzll(m)));
    m &= m - 1;
  }
  return best;
#else
  for (int off = 32; off > 0; off >>= 1)
    key = std::min(key, __shfl(key, (threadIdx.x & 63) ^ off, 64));
  return key;
#endif
}

// f(i) for the uniform i in [I, I + N) that equals `at`, by halves.  (The asm
// keeps the compiler from merging the cases into one that indexes an array of
// registers by a variable, which would put the array into memory.)
template <int I, int N, typename F> __device__ __forceinline__ void at_index(int at, F&& f) {
  if constexpr (N == 1) {
    f(std::integral_constant<int, I>{});
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("; %0" ::"n"(I));
#endif
  } else if (at < I + N / 2) {
    at_index<I, N / 2>(at, f);
  } else {
    at_index<I + N / 2, N - N / 2>(at, f);
  }
}

// The same leaf, rows [c0, c0 + 512 R): C columns at a time live in the
// registers of the one workgroup, thread t holding rows t, t + 512, ... .
// Every element sees the operations of the kernel above in the same order, so
// the results are the same bits; the leaf's earlier columns reach a chunk as
// products (their rows of U first, by wave 0), and the chunk's swaps reach the
// leaf's other columns at its end, all at once.  A column costs one barrier:
// each wave offers its largest element with that row of the chunk, the owner
// of row j offers row j, and then every thread finds the winner by itself.
//
// Bound by the chain of a column (maximum, exchange, reciprocal: about 2 us on
// few rows) and by the products on one CU.  32 columns of 512, 1024, 2048, 4096,
// 8192 and 16384 rows, FP64: 72, 72, 87, 125, 335 and 1070 us, against 203, 308,
// 502, 893, 1669 and 3225 for the kernel above (a pass over the leaf in memory
// per column and three barriers with a single thread between them); FP32: 64,
// 64, 72, 92, 143 and 296 against 171, 180, 263, 423, 743 and 1412.
template <typename T, int R, int C>
__global__ __launch_bounds__(LR_THREADS) void getf2_reg_kernel(T* __restrict__ P, int64_t Mp,
                                                               int c0, int nc,
                                                               int* __restrict__ piv,
                                                               int* __restrict__ info,
                                                               const int* __restrict__ abort,
                                                               int pivot) {
  constexpr int NW = LR_THREADS / 64;
  __shared__ T candv[2][NW], cand[2][NW][C], rowj[2][C], U[LU_LEAF][C];
  __shared__ T L11[LU_LEAF][LU_LEAF];
  __shared__ int candr[2][NW], q[C], tgt[2 * C], src[2 * C];
  if (abort && *abort) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readlane(tid >> 6, 0);
  const int64_t ld = Mp;
  T* const base = P + (int64_t)c0 * ld + c0;  // row 0, column 0 of the leaf
  const int M = (int)(Mp - c0);
  T a[R][C];
  // this thread's rows; those past the end are zeros that no comparison picks
  // (their products may turn them to NaN) and that are never stored
  unsigned ro[R];
#pragma unroll
  for (int i = 0; i < R; ++i) ro[i] = std::min(tid + LR_THREADS * i, M - 1);
#pragma unroll 1
  for (int k0 = 0; k0 < nc; k0 += C) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const T* const col = base + (int64_t)std::min(k0 + c, nc - 1) * ld;
#pragma unroll
      for (int i = 0; i < R; ++i) a[i][c] = col[ro[i]];
    }
    if (k0 > 0) {
      for (int e = tid; e < k0 * LU_LEAF; e += LR_THREADS) {
        const int k = e / LU_LEAF, r = e % LU_LEAF;
        if (r < k0) L11[k][r] = base[(int64_t)k * ld + r];
      }
      T l[2][R];
      auto load_l = [&](int k, T (&x)[R]) {
        const T* const col = base + (int64_t)std::min(k, k0 - 1) * ld;
#pragma unroll
        for (int i = 0; i < R; ++i) x[i] = col[ro[i]];
      };
      if (R <= 4) load_l(0, l[0]);
      __syncthreads();
      if (wave == 0) {
        T lk = L11[0][lane & (LU_LEAF - 1)];
        for (int k = 0; k < k0; ++k) {
          const T lv = lk;
          lk = L11[std::min(k + 1, k0 - 1)][lane & (LU_LEAF - 1)];
          T u[C];
#pragma unroll
          for (int c = 0; c < C; ++c) u[c] = wave_bcast(a[0][c], k);
          if (lane > k && lane < k0)
#pragma unroll
            for (int c = 0; c < C; ++c) a[0][c] -= lv * u[c];
        }
        if (lane < k0)
#pragma unroll
          for (int c = 0; c < C; ++c) U[lane][c] = a[0][c];
      }
      __syncthreads();
      auto update = [&](int k, const T (&x)[R]) {
        T u[C];
#pragma unroll
        for (int c = 0; c < C; ++c) u[c] = U[k][c];
        if (tid >= k0)
#pragma unroll
          for (int c = 0; c < C; ++c) a[0][c] -= x[0] * u[c];
#pragma unroll
        for (int i = 1; i < R; ++i)
#pragma unroll
          for (int c = 0; c < C; ++c) a[i][c] -= x[i] * u[c];
      };
      static_assert(C % 2 == 0, "the earlier columns are taken in pairs");
      if (R <= 4) {  // registers for a column ahead
        for (int k = 0; k < k0; k += 2) {
          load_l(k + 1, l[1]);
          update(k, l[0]);
          load_l(k + 2, l[0]);
          update(k + 1, l[1]);
        }
      } else {
#pragma unroll 1
        for (int k = 0; k < k0; ++k) {
          load_l(k, l[0]);
          update(k, l[0]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (tid + LR_THREADS * i >= M)
#pragma unroll
        for (int c = 0; c < C; ++c) a[i][c] = T(0);
#pragma unroll
    for (int jj = 0; jj < C; ++jj) {
      const int j = k0 + jj, par = jj & 1;
      if (j >= nc) break;
      if (pivot) {
        // the wave's maximum over rows >= j (NaN never wins), then its first row
        T best = tid >= j ? fmax(T(-1), fabs(a[0][jj])) : T(-1);
#pragma unroll
        for (int i = 1; i < R; ++i) best = fmax(best, fabs(a[i][jj]));
        best = wave_max(best);
        int br = std::numeric_limits<int>::max();
#pragma unroll
        for (int i = R - 1; i > 0; --i)
          if (fabs(a[i][jj]) == best) br = tid + LR_THREADS * i;
        if (tid >= j && fabs(a[0][jj]) == best) br = tid;
        br = wave_first(br);
        const int bi = __builtin_amdgcn_readlane(br / LR_THREADS, 0);
        if (tid == (br & (LR_THREADS - 1)))
          at_index<0, R>(bi, [&](auto i) {
#pragma unroll
            for (int c = 0; c < C; ++c) cand[par][wave][c] = a[i.value][c];
          });
        if (lane == 0) { candv[par][wave] = best; candr[par][wave] = br; }
      }
      if (tid == j)
#pragma unroll
        for (int c = 0; c < C; ++c) rowj[par][c] = a[0][c];
      __syncthreads();
      int p = j;
      const T* pr = rowj[par];
      if (pivot) {
        T b = candv[par][0];
        int x = candr[par][0], w = 0;
#pragma unroll
        for (int o = 1; o < NW; ++o) {
          const T v = candv[par][o];
          const int r = candr[par][o];
          if (v > b || (v == b && r < x)) { b = v; x = r; w = o; }
        }
        if (x < M && x != j) {  // (an all-NaN column keeps its row)
          p = x;
          pr = cand[par][w];
        }
      }
      T u[C];
#pragma unroll
      for (int c = 0; c < C; ++c) u[c] = pr[c];
      if (p != j) {
        const int pi = __builtin_amdgcn_readlane(p / LR_THREADS, 0);
        if (tid == (p & (LR_THREADS - 1)))
          at_index<0, R>(pi, [&](auto i) {
#pragma unroll
            for (int c = 0; c < C; ++c) a[i.value][c] = rowj[par][c];
          });
        if (tid == j)
#pragma unroll
          for (int c = 0; c < C; ++c) a[0][c] = u[c];
      }
      const T d = u[jj];
      if (tid == 0) {
        piv[c0 + j] = c0 + p;
        q[jj] = p;
        if (d == T(0) && info && *info == 0) *info = c0 + j + 1;
      }
      if (fabs(d) >= std::numeric_limits<T>::min()) {
        const T inv = T(1) / d;  // LAPACK getf2: scale by the reciprocal
        if (tid > j) a[0][jj] *= inv;
#pragma unroll
        for (int i = 1; i < R; ++i) a[i][jj] *= inv;
      } else if (d != T(0)) {    // ... or divide when it would overflow
        if (tid > j) a[0][jj] /= d;
#pragma unroll
        for (int i = 1; i < R; ++i) a[i][jj] /= d;
      }
      if (tid > j)
#pragma unroll
        for (int c = jj + 1; c < C; ++c) a[0][c] -= a[0][jj] * u[c];
#pragma unroll
      for (int i = 1; i < R; ++i)
#pragma unroll
        for (int c = jj + 1; c < C; ++c) a[i][c] -= a[i][jj] * u[c];
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (k0 + c >= nc) break;
      T* const col = base + (int64_t)(k0 + c) * ld;
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (tid + LR_THREADS * i < M) col[ro[i]] = a[i][c];
    }
    const int cc = std::min(C, nc - k0);
    if (pivot && nc > cc) {
      // the chunk's swaps on the leaf's other columns: row tgt[] takes what
      // row src[] held (rows that stay where they are: -1)
      __syncthreads();
      if (tid < C) {
        int row[2] = {-1, -1}, from[2] = {-1, -1};
        if (tid < cc) {
          bool last = q[tid] >= k0 + cc;
          for (int t = tid + 1; t < cc; ++t) last = last && q[t] != q[tid];
          row[0] = k0 + tid;
          from[0] = q[tid];
          if (last) { row[1] = q[tid]; from[1] = k0 + tid; }
          // what row `from` held before step tid: trace it back
#pragma unroll
          for (int e = 0; e < 2; ++e)
            for (int t = tid - 1; t >= 0; --t)
              if (q[t] == from[e]) from[e] = k0 + t;
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          tgt[2 * tid + e] = row[e] != from[e] ? row[e] : -1;
          src[2 * tid + e] = from[e];
        }
      }
      __syncthreads();
      const int e = tid % (2 * C);
      int c = tid / (2 * C);
      if (c >= k0) c += cc;
      const bool moves = c < nc && tgt[e] >= 0;
      T v = T(0);
      if (moves) v = base[(int64_t)c * ld + src[e]];
      __syncthreads();
      if (moves) base[(int64_t)c * ld + tgt[e]] = v;
    }
    __syncthreads();
  }
}

// Panel-relative 0-based pivots -> the reference's ipiv (global 1-based
// rows); the panel's first zero pivot (local, 1-based) -> the global info.
__global__ void lu_ipiv_kernel(const int* __restrict__ piv, int npiv, int64_t row0,
                               int* __restrict__ ipiv, const int* __restrict__ local_info,
                               int* __restrict__ info, int* __restrict__ abort) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < npiv) ipiv[i] = (int)(row0 + piv[i] + 1);
  if (i == 0 && *local_info != 0) {
    if (info && *info == 0) *info = (int)(row0 + *local_info);
    (void)abort;
  }
}

// Row swaps of a tiled block-column region (a contiguous panel is one with
// mb = Mr): for p = p0..p1-1 in order, swap rows p and piv[p - p0] - off (an
// index out of range swaps nothing).
//
// The pivots of up to 512 steps are turned into the permutation they amount to
// and every element moves once: thread t takes the new row p0 + t and, if its
// step is the last to name a row below the steps' own, that row.  A step
// names its own row or a later one, so what comes to rest at row p is what
// row piv[p] held before step p, and before step b a row holds what the last
// earlier step that names it had as its own row then (a chain of such steps
// back to a row that none names).  A list with a step that names an earlier
// row is applied one swap at a time.
//
// Bound by the latency of three phases (the lists, the loads, the stores);
// four columns a workgroup spread the elements over the chip.  512 steps on
// 512 columns of 4096 rows, FP64: 33 us, against 215 us with one thread a
// column that made the swaps one after the other; the swaps within a panel
// 6 against 23 us.  Fewer steps than threads (2^lg or fewer) take as many times
// the columns: 8 steps on 1000000 columns 30 us, 726 with four a workgroup.
constexpr int LS_THREADS = 512, LS_COLS = 4;
template <typename T>
__global__ __launch_bounds__(LS_THREADS) void laswp_kernel(T* __restrict__ base, int64_t Mr, int W,
                                                           int mb, int c0, int c1, int p0, int p1,
                                                           int lg, const int* __restrict__ piv,
                                                           int64_t off,
                                                           const int* __restrict__ abort) {
  __shared__ int q[LS_THREADS], home[LS_THREADS];
  __shared__ int backward;
  if (abort && *abort) return;
  // thread t of a set of 2^lg: step t of columns c0, c0 + sets, ...
  const int t = threadIdx.x & ((1 << lg) - 1), set = threadIdx.x >> lg, sets = LS_THREADS >> lg;
  c0 += blockIdx.x * (sets * LS_COLS);
  for (int b0 = p0; b0 < p1; b0 += LS_THREADS) {
    const int n = std::min(LS_THREADS, p1 - b0), p = b0 + t;
    int mine = -1;
    if (t < n) {
      const int64_t to = (int64_t)piv[p - p0] - off;
      mine = to >= 0 && to < Mr ? (int)to : p;
    }
    if (threadIdx.x == 0) backward = 0;
    if (set == 0) q[t] = mine;
    __syncthreads();
    if (t < n && mine < p) backward = 1;
    // the last earlier step that names this step's row, the last earlier one
    // that names the same row, whether a later one does
    int own = -1, same = -1;
    bool later = false;
#pragma unroll 8
    for (int i = 0; i < n; ++i) {
      const int x = q[i];
      if (i < t && x == p) own = i;
      if (i < t && x == mine) same = i;
      if (i > t && x == mine) later = true;
    }
    if (set == 0) home[t] = own;
    __syncthreads();
    if (backward) {
      const int64_t end = std::min<int64_t>((int64_t)c0 + sets * LS_COLS, c1);
      for (int64_t c = (int64_t)c0 + threadIdx.x; c < end; c += LS_THREADS)
        for (int i = 0; i < n; ++i)
          if (q[i] != b0 + i) {
            T* a = tiled_at(base, Mr, mb, W, b0 + i, c);
            T* b = tiled_at(base, Mr, mb, W, q[i], c);
            const T v = *a;
            *a = *b;
            *b = v;
          }
      __syncthreads();
      continue;
    }
    int to[2] = {-1, -1}, from[2] = {-1, -1};
    if (t < n) {
      to[0] = p;
      from[0] = mine;
      for (int i = same; i >= 0; i = home[i]) from[0] = b0 + i;
      if (mine >= b0 + n && !later) {
        to[1] = mine;
        from[1] = p;
        for (int i = own; i >= 0; i = home[i]) from[1] = b0 + i;
      }
    }
    T v[2][LS_COLS];
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (to[e] != from[e]) {
        const int64_t k = from[e] / mb, l = std::min<int64_t>(mb, Mr - k * mb);
        const T* a = base + k * (int64_t)mb * W + (from[e] - k * mb);
#pragma unroll
        for (int c = 0; c < LS_COLS; ++c) {
          const int64_t col = (int64_t)c0 + set + sets * c;
          if (col < c1) v[e][c] = a[col * l];
        }
      }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (to[e] != from[e]) {
        const int64_t k = to[e] / mb, l = std::min<int64_t>(mb, Mr - k * mb);
        T* a = base + k * (int64_t)mb * W + (to[e] - k * mb);
#pragma unroll
        for (int c = 0; c < LS_COLS; ++c) {
          const int64_t col = (int64_t)c0 + set + sets * c;
          if (col < c1) a[col * l] = v[e][c];
        }
      }
    __syncthreads();
  }
}

namespace {
unsigned blocks_of(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

// Columns [c0, c1) of a tiled region or contiguous panel (mb = Mr).
template <typename T>
int laswp_launch(T* base, int64_t Mr, int W, int mb, int c0, int c1, int p0, int p1,
                 const int* piv, int64_t off, const int* abort, hipStream_t s) {
  // sets of threads no larger than the steps need, as long as every CU has columns
  int lg = 0;
  while ((1 << lg) < std::min(p1 - p0, LS_THREADS) ||
         ((1 << lg) < LS_THREADS && blocks_of(c1 - c0, (LS_THREADS >> lg) * LS_COLS) < 256))
    ++lg;
  hipLaunchKernelGGL((laswp_kernel<T>), dim3(blocks_of(c1 - c0, (LS_THREADS >> lg) * LS_COLS)),
                     dim3(LS_THREADS), 0, s, base, Mr, W, mb, c0, c1, p0, p1, lg, piv, off, abort);
  DM_LAUNCH_CHECK("laswp_kernel");
  return 0;
}

// A leaf: C columns of all its rows in a thread's registers, R x C elements of
// them, fewer columns for more rows (8 while they fit: each chunk passes over the
// leaf's earlier columns again).  The FP64 leaves of 8, 16 and 32 rows a thread use
// all 256 registers and spill 20, 82 and 177 more, the FP32 leaf of 32 rows 22.
// Beyond 16384 rows, where a chunk would be one column, a leaf is factored in
// memory.
template <typename T, int R, int C>
int getf2_reg_launch(T* P, int64_t Mp, int c0, int nc, int* piv, int* linfo, int* abort,
                     bool pivot, hipStream_t s) {
  hipLaunchKernelGGL((getf2_reg_kernel<T, R, C>), dim3(1), dim3(LR_THREADS), 0, s, P, Mp, c0, nc,
                     piv, linfo, abort, pivot ? 1 : 0);
  DM_LAUNCH_CHECK("getf2_reg_kernel");
  return 0;
}
template <typename T>
int getf2_leaf(T* P, int64_t Mp, int c0, int nc, int* piv, int* linfo, int* abort, bool pivot,
               hipStream_t s) {
  const int64_t r = (Mp - c0 + LR_THREADS - 1) / LR_THREADS;
  if (r <= 2) return getf2_reg_launch<T, 2, 8>(P, Mp, c0, nc, piv, linfo, abort, pivot, s);
  if (r <= 4) return getf2_reg_launch<T, 4, 8>(P, Mp, c0, nc, piv, linfo, abort, pivot, s);
  if (r <= 8) return getf2_reg_launch<T, 8, 8>(P, Mp, c0, nc, piv, linfo, abort, pivot, s);
  if (r <= 16) return getf2_reg_launch<T, 16, 4>(P, Mp, c0, nc, piv, linfo, abort, pivot, s);
  // (1 to 3 FP64 columns of 12000 rows: 80, 89 and 112 us from registers, which
  // spill here, 64, 81 and 97 in memory)
  if (r <= 32 && (sizeof(T) == 4 || nc > 3))
    return getf2_reg_launch<T, 32, 2>(P, Mp, c0, nc, piv, linfo, abort, pivot, s);
  hipLaunchKernelGGL((getf2_leaf_kernel<T>), dim3(1), dim3(LU_THREADS), 0, s, P, Mp, c0, nc, piv,
                     linfo, abort, pivot ? 1 : 0);
  DM_LAUNCH_CHECK("getf2_leaf_kernel");
  return 0;
}

// getrf2's recursion on columns [c0, c0 + nc) of the contiguous panel.
template <typename T>
int getrf_rec(T* P, int64_t Mp, int c0, int nc, int* piv, int* linfo, int* abort,
              bool pivot, hipStream_t s) {
  if (nc <= LU_LEAF) return getf2_leaf<T>(P, Mp, c0, nc, piv, linfo, abort, pivot, s);
  const int n1 = ((nc / 2 + LU_LEAF - 1) / LU_LEAF) * LU_LEAF, n2 = nc - n1;
  int rc = getrf_rec<T>(P, Mp, c0, n1, piv, linfo, abort, pivot, s);
  if (rc) return rc;
  const int64_t ld = Mp;
  if (pivot) {  // left half's swaps on the right half
    rc = laswp_launch<T>(P, Mp, 0, (int)Mp, c0 + n1, c0 + nc, c0, c0 + n1, piv + c0, 0, abort, s);
    if (rc) return rc;
  }
  T* A11 = P + (int64_t)c0 * ld + c0;
  T* A12 = P + (int64_t)(c0 + n1) * ld + c0;
  T* A21 = P + (int64_t)c0 * ld + c0 + n1;
  T* A22 = P + (int64_t)(c0 + n1) * ld + c0 + n1;
  rc = trsm_full<T>('L', 'L', 'N', 'U', n1, n2, T(1), A11, (int)ld, A12, (int)ld, abort, s);
  if (rc) return rc;
  if (Mp > c0 + n1) {
    rc = gemm_single<T>(false, false, (int)(Mp - c0 - n1), n2, n1, T(-1), A21, (int)ld, A12,
                        (int)ld, T(1), A22, (int)ld, 0, abort, s);
    if (rc) return rc;
  }
  if (Mp > c0 + n1) {
    rc = getrf_rec<T>(P, Mp, c0 + n1, n2, piv, linfo, abort, pivot, s);
    if (rc) return rc;
    if (pivot) {  // right half's swaps on the left half
      rc = laswp_launch<T>(P, Mp, 0, (int)Mp, c0, c0 + n1, c0 + n1,
                           (int)std::min<int64_t>(c0 + nc, Mp), piv + c0 + n1, 0, abort, s);
      if (rc) return rc;
    }
  }
  return 0;
}
}  // namespace

// Workspace bytes of a panel factorization: the contiguous panel, then W + 1
// ints (pivots, local info).
template <typename T>
size_t getrf_panel_ws_bytes(int64_t Mp, int W) {
  const size_t panel = sizeof(T) * (size_t)Mp * W;
  return ((panel + 255) / 256) * 256 + 4 * ((size_t)W + 64);
}

// LU of a tiled panel: the tiles (k..mt-1, k) starting at `tiles` (Mp rows
// in tiles of mb, W columns), pivots to ipiv (global 1-based, row0 = the
// panel's first global row), info to *info (global, first zero pivot).
template <typename T>
int getrf_panel(T* tiles, int64_t Mp, int W, int mb, int64_t row0, int* ipiv, int* info,
                int* abort, bool pivot, void* wsp, hipStream_t s) {
  if (Mp <= 0 || W <= 0) return 0;
  char* w = (char*)wsp;
  T* P = (T*)w;
  const size_t panel = ((sizeof(T) * (size_t)Mp * W + 255) / 256) * 256;
  int* piv = (int*)(w + panel);
  int* linfo = piv + W;
  const int npiv = (int)std::min<int64_t>(Mp, W);
  int rc = fill_i32_launch(linfo, 0, 1, s);
  if (rc) return rc;
  hipLaunchKernelGGL((panel_pack_kernel<T>), dim3(blocks_of(Mp * W, 256)), dim3(256), 0, s, P,
                     tiles, Mp, W, mb, 0);
  DM_LAUNCH_CHECK("panel_pack_kernel");
  rc = getrf_rec<T>(P, Mp, 0, npiv, piv, linfo, abort, pivot, s);
  if (rc) return rc;
  if (W > npiv) {  // a panel wider than tall: the rest gets the swaps and L11^-1
    if (pivot) {
      rc = laswp_launch<T>(P, Mp, 0, (int)Mp, npiv, W, 0, npiv, piv, 0, abort, s);
      if (rc) return rc;
    }
    rc = trsm_full<T>('L', 'L', 'N', 'U', npiv, W - npiv, T(1), P, (int)Mp,
                      P + (int64_t)npiv * Mp, (int)Mp, abort, s);
    if (rc) return rc;
  }
  hipLaunchKernelGGL((panel_pack_kernel<T>), dim3(blocks_of(Mp * W, 256)), dim3(256), 0, s, P,
                     tiles, Mp, W, mb, 1);
  DM_LAUNCH_CHECK("panel_pack_kernel");
  hipLaunchKernelGGL(lu_ipiv_kernel, dim3(blocks_of(std::max(npiv, 1), 256)), dim3(256), 0, s,
                     piv, npiv, row0, ipiv, linfo, info, abort);
  DM_LAUNCH_CHECK("lu_ipiv_kernel");
  return 0;
}

template <typename T>
int laswp_tiled(T* base, int64_t Mr, int W, int mb, const int* ipiv, int npiv, int64_t row0,
                const int* abort, hipStream_t s) {
  if (Mr <= 0 || W <= 0 || npiv <= 0) return 0;
  return laswp_launch<T>(base, Mr, W, mb, 0, W, 0, npiv, ipiv, row0 + 1, abort, s);
}

template size_t getrf_panel_ws_bytes<double>(int64_t, int);
template size_t getrf_panel_ws_bytes<float>(int64_t, int);
template int getrf_panel<double>(double*, int64_t, int, int, int64_t, int*, int*, int*, bool, void*,
                                 hipStream_t);
template int getrf_panel<float>(float*, int64_t, int, int, int64_t, int*, int*, int*, bool, void*,
                                hipStream_t);
template int laswp_tiled<double>(double*, int64_t, int, int, const int*, int, int64_t, const int*,
                                 hipStream_t);
template int laswp_tiled<float>(float*, int64_t, int, int, const int*, int, int64_t, const int*,
                                hipStream_t);

}  // namespace dm
