// Cholesky factorization of a diagonal tile (LAPACK potrf) on CDNA4.
//
// Replaces LAPACK.potrf! as called by potrf_checked! (src/array/cholesky.jl:
// 2-18, spawned at :39/:84).  info follows LAPACK: 0, or k > 0 when the
// leading minor of order k is not positive definite (pivot <= 0 or NaN).
//
// Structure: blocked right-looking factorization with 64-wide panels, one
// launch per panel (potrf_step_kernel) after the first diagonal block
// (potrf_diag_kernel).  A launch takes the factored diagonal block U_kk, and
// each of its workgroups owns one 64 x 64 tile (i, j) of the trailing
// triangle: it solves the two panel-row blocks it needs, U_ki = U_kk^-T A_ki
// and U_kj, in LDS for itself and updates its tile.  Solving them in every
// workgroup costs 2 x 64^3 flops on a chip that is mostly idle and saves the
// launch (and the trip through memory) that a separate panel-row step needs.
// Workgroup 0 owns the next diagonal block, keeps it in LDS and factors it.
// The panel row in memory stays unsolved meanwhile (other workgroups still
// read it); the next launch's extra workgroups finish it, beside that
// launch's tiles, which only touch later rows.  The last launch has a single
// tile and finishes its own row.
//
// Tiles of several thousand columns take separate launches for their first
// panels (potrf_fused_blocks).
//
// Bound by the chain of launches and pivots, not by flops.  Measured per 64
// columns of a 512 tile (FP64): one launch of 20 us, 8 of them pb_factor; the
// panel row and the update as two launches, with the block factored by one lane
// per column from LDS rows, took 23 + 40 us.
//
// After a failed pivot the remaining launches do nothing but finish the rows
// before it (the factor of the leading minor is whole, as LAPACK leaves it).  A
// workgroup decides that once, for all its waves (potrf_stop), by the order of
// the diagonal block it starts from: its own launch's workgroup 0 may report the
// next one's failure while others have yet to start.
#include <type_traits>
#include "dm_internal.h"
#include "gemm_tiles.h"
#include "potrf_diag.h"

namespace dm {

// Factor the block in M (columns from kb on the identity's), store it at j0,
// report a failed pivot.
template <typename T, bool UPPER>
__device__ __forceinline__ void potrf_block(T* M, int* fail, T* __restrict__ A, int lda, int j0,
                                            int kb, int* __restrict__ info,
                                            int* __restrict__ abort, int global_base) {
  const int bad = pb_factor<T>(M, kb, fail);
  pb_store_diag<T, UPPER>(A, lda, j0, kb, bad ? bad - 1 : kb, M);
  if (bad && threadIdx.x == 0) {
    if (info) *info = j0 + bad;
    if (abort) *abort = global_base + j0 + bad;
  }
}

// Whether a pivot of order at most `upto` in this tile has failed, by the
// report of potrf_block; with `abort`, also whether one of an earlier tile or an
// earlier task has (orders up to 0).  For one thread of a workgroup: the words
// may change while it runs.
__device__ __forceinline__ bool potrf_stop(const int* info, const int* abort, int global_base,
                                           int upto) {
  const int* const p = abort ? abort : info;
  const int order = p ? *p : 0;
  return order != 0 && order - (abort ? global_base : 0) <= upto;
}

template <typename T, bool UPPER>
__global__ __launch_bounds__(256) void potrf_diag_kernel(T* __restrict__ A, int n, int lda, int j0,
                                                         int* __restrict__ info,
                                                         int* __restrict__ abort,
                                                         int global_base) {
  __shared__ T M[PBE];
  __shared__ int fail, stop;
  raise_wave_priority();  // always on the critical path of a factorization
  const int kb = min(PB, n - j0);
  T v[16];
  pb_load_diag<T, UPPER>(A, lda, j0, kb, v);
  if (threadIdx.x == 0) {
    stop = (abort && *abort) || (info && *info);
    // an info word that was set before this call stops its other launches too
    if (stop && abort && !*abort) *abort = global_base + 1;
  }
  pb_put<T, UPPER>(M, v);
  __syncthreads();
  if (stop) return;
  potrf_block<T, UPPER>(M, &fail, A, lda, j0, kb, info, abort, global_base);
}

// The launch of panel j0 (see above): workgroups [0, ntile) own the tiles of
// the trailing triangle, the others finish the row of panel j0 - 64.
template <typename T, bool UPPER>
__global__ __launch_bounds__(256) void potrf_step_kernel(T* __restrict__ A, int n, int lda, int j0,
                                                         int ntile, int* __restrict__ info,
                                                         int* __restrict__ abort,
                                                         int global_base) {
  typedef typename PMfma<T>::v4 v4;
  __shared__ T M[PBE];
  __shared__ T X[2 * PBE];  // column blocks j and i
  __shared__ T nrec[PB];
  __shared__ int fail, stop;
  raise_wave_priority();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int t = blockIdx.x;
  const bool finish = t >= ntile;
  const int jp = finish ? j0 - PB : j0;
  int ti, tj;
  if (finish) ti = tj = t - ntile;
  else upper_tri_decode(t, ti, tj);
  const int ci = jp + PB + PB * ti, cj = jp + PB + PB * tj;
  const bool two = ti != tj;
  // every load of the launch is issued before the first wait
  T v[16], xi[16], xj[16];
  pb_load_diag<T, UPPER>(A, lda, jp, PB, v);
  pb_load<T, UPPER>(A, lda, jp, cj, n - cj, xj);
  if (two) pb_load<T, UPPER>(A, lda, jp, ci, n - ci, xi);
  // this wave's 32 x 32 quadrant of the tile: element (m, n) of block (p, q)
  // in item r, the matrix's contiguous axis along the lanes
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  const bool work = !finish && (two || wm <= wn);
  auto row_of = [&](int p, int r) { return wm + 16 * p + (UPPER ? lr : PMfma<T>::row(lk, r)); };
  auto col_of = [&](int q, int r) { return wn + 16 * q + (UPPER ? PMfma<T>::row(lk, r) : lr); };
  auto inside = [&](int m, int c) { return ci + m < n && cj + c < n && (two || m <= c); };
  T old[2][2][4];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = row_of(p, r), c = col_of(q, r);
        old[p][q][r] =
            *gptr(pb_at<T, UPPER>(A, lda, min(ci + m, n - 1), min(cj + c, n - 1)));
      }
  if (threadIdx.x == 0) stop = potrf_stop(info, abort, global_base, jp + PB);
  pb_put<T, UPPER>(M, v);
  __syncthreads();
  if (stop) return;
  pb_recip<T>(M, nrec);
  const T* const Xj = X;
  const T* const Xi = two ? X + PBE : X;
  pb_put<T, UPPER>(X, xj);
  if (two) pb_put<T, UPPER>(X + PBE, xi);
  __syncthreads();
  pb_solve<T>(M, nrec, X, wave * 16);
  if (two) pb_solve<T>(M, nrec, X + PBE, wave * 16);
  __syncthreads();
  if (finish) {
    pb_store<T, UPPER>(A, lda, jp, cj, n - cj, Xj);
    return;
  }
  if (ntile == 1) pb_store<T, UPPER>(A, lda, j0, cj, n - cj, Xj);  // the only reader of this row
  if (work) {
    // the 64 products are summed by themselves and subtracted once: rounding
    // at the tile's own magnitude happens once, not at every k-step
    v4 acc[2][2];
    acc[0][0] = acc[0][1] = acc[1][0] = acc[1][1] = v4{0, 0, 0, 0};
#pragma unroll 4
    for (int s = 0; s < PB / 4; ++s) {
      const int k = (4 * s + lk) * PBS;
      T a[2], b[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) a[p] = Xi[k + wm + 16 * p + lr];
#pragma unroll
      for (int q = 0; q < 2; ++q) b[q] = Xj[k + wn + 16 * q + lr];
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          acc[p][q] = UPPER ? PMfma<T>::mac(b[q], a[p], acc[p][q])
                            : PMfma<T>::mac(a[p], b[q], acc[p][q]);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = row_of(p, r), c = col_of(q, r);
          const T v = old[p][q][r] - acc[p][q][r];
          if (t == 0) M[m * PBS + c] = inside(m, c) ? v : (m == c ? T(1) : T(0));
          else if (inside(m, c)) *gptr(pb_at<T, UPPER>(A, lda, ci + m, cj + c)) = v;
        }
  }
  if (t != 0) return;
  __syncthreads();
  potrf_block<T, UPPER>(M, &fail, A, lda, j0 + PB, min(PB, n - j0 - PB), info, abort, global_base);
}

namespace {
// Column blocks right of a panel up to which its row, the trailing update and
// the next diagonal block are one launch.  Beyond them the launch has several
// rounds of workgroups (in FP64 a CU holds one), each solving its two row blocks
// again, and a launch each for the row, the update (a product with K = 64 on the
// GEMM's tiles) and the diagonal block is faster.  U, FP64, lines at 23, 31 and 47
// blocks and none: n = 2048 774, 755, 753 and 755 us, 3072 1497, 1478, 1632 and
// 1634, 4096 2765, 2755, 2914 and 3133, 8192 13.8, 13.8, 14.0 and 20.2 ms; FP32
// 2048 577, 504, 504 and 504 us, 3072 1055, 980, 949 and 949, 4096 1630, 1558, 1541
// and 1658, 8192 5.9, 5.8, 5.7 and 8.5 ms.
template <typename T> constexpr int potrf_fused_blocks = sizeof(T) == 8 ? 31 : 47;

template <typename T, bool UPPER>
int potrf_panels(int n, T* A, int lda, int* info, int* abort, int global_offset, hipStream_t s) {
  // Launches after a failed pivot are no-ops: they watch the plan-level
  // abort flag when there is one, else info.
  if (n <= 0) return 0;
  auto diag = [&](int j0) {
    hipLaunchKernelGGL((potrf_diag_kernel<T, UPPER>), dim3(1), dim3(256), 0, s, A, n, lda, j0, info,
                       abort, global_offset);
    DM_LAUNCH_CHECK("potrf_diag_kernel");
    return 0;
  };
  auto step = [&](int j0, int ntile, int nfin) {
    hipLaunchKernelGGL((potrf_step_kernel<T, UPPER>), dim3((unsigned)(ntile + nfin)), dim3(256), 0, s,
                       A, n, lda, j0, ntile, info, abort, global_offset);
    DM_LAUNCH_CHECK("potrf_step_kernel");
    return 0;
  };
  int rc = diag(0);
  bool finish = false;  // the row of the panel before is not yet solved
  for (int j0 = 0; !rc && n - j0 > PB; j0 += PB) {
    const int nt = (n - j0 - 1) / PB;  // 64-column blocks right of the panel
    if (nt <= potrf_fused_blocks<T>) {
      rc = step(j0, nt * (nt + 1) / 2, finish ? nt + 1 : 0);
      finish = true;
      continue;
    }
    const int j1 = j0 + PB, rest = n - j1;
    const T* const row = A + (UPPER ? (size_t)j1 * lda + j0 : (size_t)j0 * lda + j1);
    rc = step(j1, 0, nt);
    if (!rc)
      rc = gemm_single<T>(UPPER, !UPPER, rest, rest, PB, T(-1), row, lda, row, lda, T(1),
                          A + (size_t)j1 * lda + j1, lda, UPPER ? 1 : 2, abort ? abort : info, s);
    if (!rc) rc = diag(j1);
  }
  return rc;
}
}  // namespace

template <typename T>
int potrf_full(bool upper, int n, T* A, int lda, int* info, int* abort, int global_offset, T* ws,
               hipStream_t s) {
  (void)ws;
  return upper ? potrf_panels<T, true>(n, A, lda, info, abort, global_offset, s)
               : potrf_panels<T, false>(n, A, lda, info, abort, global_offset, s);
}

template int potrf_full<double>(bool, int, double*, int, int*, int*, int, double*, hipStream_t);
template int potrf_full<float>(bool, int, float*, int, int*, int*, int, float*, hipStream_t);

// ------------------------------------------------------------ gemv
// y := alpha op(A) x + beta y.  'N': a workgroup owns GN_ROWS rows, its groups of
// as many lanes split the columns (coalesced along rows, eight columns a group in
// flight) and reduce through LDS.  Bound by the latency of its few loads per thread
// and by how many CUs a tile reaches: 512 x 512 FP64 as 32 groups on 32 rows 6 us,
// against 39 us for 64 rows on four waves, one load at a time.  Other shapes where
// 32 groups would have no column each or the rows alone fill the chip
// (gemv_launch): 1000000 rows of 1, 4, 16 and 64 columns took 57, 81, 92 and 193 us
// as 32 groups on 32 rows.
// 'T': one wave per output element (column dot product, coalesced).
// An empty inner dimension (n = 0 for 'N', m = 0 for 'T') leaves
// y := beta y, as BLAS does (beta == 0 writes zeros without reading y).
template <typename T, int GN_ROWS, int GN_GROUPS>
__global__ __launch_bounds__(GN_ROWS * GN_GROUPS) void gemv_n_kernel(
    int m, int n, T alpha, const T* __restrict__ A, int lda, const T* __restrict__ x, int incx,
    T beta, T* __restrict__ y, int incy, const int* __restrict__ abort) {
  __shared__ T part[GN_GROUPS][GN_ROWS];
  if (abort && *abort) return;
  const int r = threadIdx.x % GN_ROWS, g = threadIdx.x / GN_ROWS;
  const int i = blockIdx.x * GN_ROWS + r;
  T acc = T(0);
  if (i < m) {
    int j = g;
    for (; j + 7 * GN_GROUPS < n; j += 8 * GN_GROUPS) {
      T a[8], b[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        a[u] = A[(size_t)(j + u * GN_GROUPS) * lda + i];
        b[u] = x[(size_t)(j + u * GN_GROUPS) * incx];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += a[u] * b[u];
    }
    for (; j < n; j += GN_GROUPS) acc += A[(size_t)j * lda + i] * x[(size_t)j * incx];
  }
  part[g][r] = acc;
  __syncthreads();
  if (g == 0 && i < m) {
    T v = T(0);
#pragma unroll
    for (int u = 0; u < GN_GROUPS; ++u) v += part[u][r];
    v *= alpha;
    T* py = y + (size_t)i * incy;
    *py = (beta == T(0)) ? v : v + beta * *py;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void gemv_t_kernel(int m, int n, T alpha,
                                                     const T* __restrict__ A, int lda,
                                                     const T* __restrict__ x, int incx,
                                                     T beta, T* __restrict__ y,
                                                     int incy, const int* __restrict__ abort) {
  if (abort && *abort) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = blockIdx.x * 4 + wave;
  if (j >= n) return;
  T acc = T(0);
  for (int i = lane; i < m; i += 64) acc += A[(size_t)j * lda + i] * x[(size_t)i * incx];
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if (lane == 0) {
    const T v = alpha * acc;
    T* py = y + (size_t)j * incy;
    *py = (beta == T(0)) ? v : v + beta * *py;
  }
}

template <typename T>
int gemv_launch(bool trans, int m, int n, T alpha, const T* A, int lda, const T* x, int incx,
                T beta, T* y, int incy, const int* abort, hipStream_t s) {
  const int ly = trans ? n : m;  // output length
  if (ly <= 0) return 0;
  // an empty inner dimension still scales y (both kernels then skip the
  // products: the 'N' kernel's column loop and the 'T' kernel's row loop
  // run zero times)
  if (!trans) {
    // about eight columns a group; from 65536 rows on (1024 workgroups of 64) few
    // groups on more rows, whose columns are longer contiguous pieces
#define DM_GEMV_N(R, G)                                                                           \
  hipLaunchKernelGGL((gemv_n_kernel<T, R, G>), dim3((unsigned)(((long)m + R - 1) / R)), dim3(R * G), \
                     0, s, m, n, alpha, A, lda, x, incx, beta, y, incy, abort)
    if (m >= 65536) {
      if (n <= 8) DM_GEMV_N(256, 1);
      else DM_GEMV_N(64, 4);
    } else if (n <= 16) {
      DM_GEMV_N(32, 2);
    } else if (n <= 128) {
      DM_GEMV_N(32, 8);
    } else {
      DM_GEMV_N(32, 32);
    }
#undef DM_GEMV_N
  } else {
    hipLaunchKernelGGL(gemv_t_kernel<T>, dim3((n + 3) / 4), dim3(256), 0, s, m, n, alpha, A, lda,
                       x, incx, beta, y, incy, abort);
  }
  DM_LAUNCH_CHECK("gemv_kernel");
  return 0;
}

template int gemv_launch<double>(bool, int, int, double, const double*, int, const double*, int,
                                 double, double*, int, const int*, hipStream_t);
template int gemv_launch<float>(bool, int, int, float, const float*, int, const float*, int,
                                float, float*, int, const int*, hipStream_t);

// ------------------------------------------------------------ fill
__global__ void fill_i32_kernel(int* __restrict__ dst, int value, size_t count) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) dst[i] = value;
}

int fill_i32_launch(int* dst, int value, size_t count, hipStream_t s) {
  if (count == 0) return 0;
  hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, dst,
                     value, count);
  DM_LAUNCH_CHECK("fill_i32_kernel");
  return 0;
}

__global__ void copy_i32_kernel(int* __restrict__ dst, const int* __restrict__ src, size_t count) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) dst[i] = src[i];
}

int copy_i32_launch(int* dst, const int* src, size_t count, hipStream_t s) {
  if (count == 0) return 0;
  hipLaunchKernelGGL(copy_i32_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, dst,
                     src, count);
  DM_LAUNCH_CHECK("copy_i32_kernel");
  return 0;
}

// ------------------------------------------------------------ generator
// Philox4x32-10 (Salmon et al., "Parallel random numbers: as easy as 1, 2,
// 3", SC'11), counter = (i lo, i hi, 0, 0), key = (seed lo, seed hi).
// Two 53-bit uniforms in (0,1) from the four words, then Box-Muller.
__device__ __forceinline__ void philox_round(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
  const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
  const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
  const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
  const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
  const uint32_t n0 = hi1 ^ c[1] ^ k0;
  const uint32_t n2 = hi0 ^ c[3] ^ k1;
  c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
}

__global__ void randn_kernel(double* __restrict__ x, size_t count, uint64_t seed,
                             uint64_t offset) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const uint64_t idx = offset + i;
  uint32_t c[4] = {(uint32_t)idx, (uint32_t)(idx >> 32), 0u, 0u};
  uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    philox_round(c, k0, k1);
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  const double two53 = 9007199254740992.0;
  const double u = ((double)(c[0] >> 5) * 67108864.0 + (double)(c[1] >> 6) + 0.5) / two53;
  const double v = ((double)(c[2] >> 5) * 67108864.0 + (double)(c[3] >> 6) + 0.5) / two53;
  x[i] = sqrt(-2.0 * log(u)) * cos(6.283185307179586 * v);
}

int randn_launch(double* x, size_t count, uint64_t seed, uint64_t offset, hipStream_t s) {
  if (count == 0) return 0;
  hipLaunchKernelGGL(randn_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, x,
                     count, seed, offset);
  DM_LAUNCH_CHECK("randn_kernel");
  return 0;
}

}  // namespace dm
