// Triangular solves with many right-hand sides (BLAS trsm) on CDNA4.
//
// Replaces BLAS.trsm! tile calls at src/array/cholesky.jl:41,86 and
// src/array/trsm.jl:95-183.
//
// Every trsm is reduced to one "effective" left solve  Tm X = alpha V:
//   * Tm is op(A) (side L) or op(A)^T (side R), read from A directly or
//     transposed, lower or upper triangular;
//   * the right-hand-side vectors are the columns (side L) or rows (side R)
//     of B, solved in place.
// Solves longer than TRSM_LEAF are split on the host: solve the first part,
// update the second part with one (batched) GEMM on the MFMA GEMM kernel,
// solve the second part -- so most of the flops of a long solve run at GEMM
// speed.  A leaf is one launch of trsm_kernel; it needs no workspace.
#include <algorithm>
#include "dm_internal.h"
#include "trsm_plan.h"

namespace dm {

template <typename T> struct MfmaT;
// Output layouts (lane l, accumulator item r; 16x16 block D[i][j], j = l%16):
//   f64 16x16x4: i = 4*r + l/16        f32 16x16x4: i = 4*(l/16) + r
// (the f64 layout was measured on gfx950 with a one-hot lane probe).
template <> struct MfmaT<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * r + lk; }
  static __device__ __forceinline__ v4 mac(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <> struct MfmaT<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
  static __device__ __forceinline__ v4 mac(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// Two elements at an address aligned to one.
template <typename T> struct Pair;
template <> struct Pair<double> { typedef double t __attribute__((ext_vector_type(2), aligned(8))); };
template <> struct Pair<float> { typedef float t __attribute__((ext_vector_type(2), aligned(4))); };

constexpr int TB = 16;                 // block row
constexpr int TW = 16;                 // waves of a workgroup
constexpr int trsm_rows_per_wave(bool is_short) { return is_short ? 1 : TRSM_LEAF / (TB * TW); }
// Steps of the triangle in flight, as many as the 128 registers of 16 waves hold
// (FP64 with two vector blocks, above 256 rows, spills two).
template <typename T, int NB> constexpr int trsm_depth() {
  return sizeof(T) == 4 ? 4 : NB == 1 ? 2 : 1;
}
constexpr int TIS = TB + 1;            // LDS row stride of an inverted diagonal block

// A wave-uniform element offset, kept out of the optimizer's sight: it would
// otherwise turn every (step, row, column) of the unrolled loop into a vector
// pointer of its own and spill.  In 32-bit halves: as one 64-bit asm operand
// the compiler puts a negative constant such as -32 into an s_mov_b64 with a
// 32-bit literal, which the hardware extends with zeros.
__device__ __forceinline__ ptrdiff_t uniform_offset(ptrdiff_t o) {
#ifdef __HIP_DEVICE_COMPILE__
  int lo = (int)o, hi = (int)(o >> 32);
  asm volatile("" : "+s"(lo), "+s"(hi));
  o = (ptrdiff_t)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
#endif
  return o;
}

// Orders this wave's LDS writes before its later LDS reads.
__device__ __forceinline__ void trsm_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One leaf solve.  A workgroup owns 16 NB vectors and the whole triangle; an
// upper triangle is solved as the lower one that reversing both axes gives,
// so everything below is forward substitution over 16-row blocks.  Wave w
// owns block rows w, w + 16, ...: their right-hand sides, their sums
// sum_k T_pk X_k in matrix-core accumulators, and W_p, the inverse of their
// diagonal blocks (16 x 16, formed first, in LDS):
//   X_p = W_p (alpha V_p - sum_{k<p} T_pk X_k).
// The chain from X_J to X_{J+1} is two block products, a trip through LDS and
// a barrier; the other waves' products (T_pJ X_J, p > J + 1) run beside it.
// (W_p T_{p,p-1} formed ahead would halve the chain, but it measured no faster
// and loses accuracy where a diagonal block is badly conditioned.)  T comes
// straight from global memory as matrix-core operands, loaded a few steps
// ahead.
//
// Bound by three things in turn: 512 rows and 16 vectors in FP64 are 13 us of
// matrix-core work for one CU, and the 32 steps cost about 0.2 us each for the
// barrier and 0.4 us each for the chain.  Measured with the launch, 512 rows
// (left side, A^T; A; right side): 16 vectors FP64 51, 45 and 41 us, FP32 44,
// 32 and 29; 16384 vectors FP64 158, 150 and 139 us, FP32 127, 104 and 95.  The
// launches this replaces took about 210 us for 16 vectors (four solves of 128
// rows at 31 us that kept a whole 32-row chain in one wave, the products
// between them and the inversion of the diagonal blocks).  Loads made
// unconditional or a deeper prefetch measured slower or the same.
//
// SHORT: triangles of up to 256 rows, with a wave per block row and no more, their
// diagonal blocks in as much LDS, and many vectors by a loop in each workgroup:
// 16 waves and the whole LDS for a few block rows left most of a CU idle, and
// every 32 vectors paid for the inverses again.  FP64, from the left: 8 rows,
// 2000000 vectors 63 us, 1126 without; 64 rows, 100000 vectors 43 and 120; 256
// rows, 100000 vectors 351 and 411; 64 rows, 64 vectors 8.5 and 10.2.
template <typename T, bool LOWER, bool TTRANS, bool SIDE_L, int NB, bool SHORT>
__global__ __launch_bounds__(64 * TW) void trsm_kernel(const TrsmJob<T>* __restrict__ jobs,
                                                       int njobs, TrsmJob<T> single, int unit,
                                                       int prio, int nb,
                                                       const int* __restrict__ abort) {
  typedef typename MfmaT<T>::v4 v4;
  constexpr int TD = trsm_depth<T, NB>(), TQ = trsm_rows_per_wave(SHORT);
  __shared__ T Wd[SHORT ? 1 : TRSM_LEAF / TB][TB * TIS];
  // diagonal blocks, then their inverses
  auto Wb = [&](int p) -> T* {
    if constexpr (SHORT) {
      DM_DYNAMIC_LDS(trsm_lds);
      return (T*)trsm_lds + p * TB * TIS;
    } else {
      return Wd[p];
    }
  };
  __shared__ T Xs[2][TB * TB * NB];            // X_J: [k][vector]
  if (abort && *abort) return;
  if (prio) raise_wave_priority();
  TrsmJob<T> job;
  int local = blockIdx.x;
  if (njobs == 0) {
    job = single;
  } else {
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (jobs[mid].wg_begin <= local) lo = mid; else hi = mid - 1;
    }
    job = jobs[lo];
    local -= job.wg_begin;
  }
  const int L = job.L, NV = job.NV, nblk = (L + TB - 1) / TB;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  const auto A = gptr(job.A);
  const auto B = gptr(job.B);
  const size_t lda = job.lda, ldb = job.ldb;
  // element (i, k) of the lower triangle, element i of vector j
  auto a_off = [&](int i, int k) -> size_t {
    if (!LOWER) {
      i = L - 1 - i;
      k = L - 1 - k;
    }
    return TTRANS ? (size_t)i * lda + k : (size_t)k * lda + i;
  };
  // this lane's element of block row 0 and the steps along rows and vectors
  const ptrdiff_t bstep = (LOWER ? 1 : -1) * (SIDE_L ? 1 : (ptrdiff_t)ldb);
  const ptrdiff_t vstep = SIDE_L ? (ptrdiff_t)ldb : 1;
  unsigned j0 = (unsigned)local * TB * (SHORT ? nb : NB);
  auto brow = B + (LOWER ? 0 : (L - 1) * (SIDE_L ? 1 : (ptrdiff_t)ldb)) +
              MfmaT<T>::row(lk, 0) * bstep + (ptrdiff_t)(j0 + lr) * vstep;
  constexpr int RS = sizeof(T) == 8 ? 4 : 1;  // row(lk, r) = row(lk, 0) + RS r
  auto b_at = [&](int p, int r, int n) {
    return brow + uniform_offset((TB * p + RS * r) * bstep + TB * n * vstep);
  };
  // T_pJ as the operand of four k-steps: row 16 p + lr, columns 16 J + tk(lk, s)
  // (rows past the triangle repeat its last one; their results are dropped).
  // tk makes the lanes of a row read whole 64-byte pieces of it.
  auto tk = [](int k, int s) { return 2 * k + (s & 1) + 8 * (s >> 1); };
  // trow[q]: this lane's row of the wave's block row q at column tk(lk, 0)
  decltype(gptr(job.A)) trow[TQ];
#pragma unroll
  for (int q = 0; q < TQ; ++q)
    trow[q] = A + a_off(min(TB * (wave + TW * q) + lr, L - 1),
                        2 * lk + (TTRANS && !LOWER ? 1 : 0));
  const ptrdiff_t kstep = (LOWER ? 1 : -1) * (TTRANS ? 1 : (ptrdiff_t)lda);
  auto load_t = [&](int q, int J, T (&t)[4]) {
    const int p = wave + TW * q;
    if (J >= p || p >= nblk) return;
    const auto src = trow[q] + uniform_offset((ptrdiff_t)(TB * J) * kstep);
    if (TTRANS) {
      typedef typename Pair<T>::t V2;
      const V2 u = *(const DM_GLOBAL_AS V2*)src, v = *(const DM_GLOBAL_AS V2*)(src + 8 * kstep);
      t[0] = LOWER ? u[0] : u[1];
      t[1] = LOWER ? u[1] : u[0];
      t[2] = LOWER ? v[0] : v[1];
      t[3] = LOWER ? v[1] : v[0];
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) t[s] = src[tk(0, s) * kstep];
    }
  };

  // ---- inverses of the diagonal blocks, the wave's all at once: lane group g
  // of 16 inverts block wave + 16 g (its two 8 x 8 diagonal blocks by
  // substitution, one column per lane, then the coupling block -V1 (L21 V0))
#pragma unroll
  for (int q = 0; q < TQ; ++q) {
    const int p = wave + TW * q;
    if (p >= nblk) continue;
    T d[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int x = lr, y = 4 * e + lk;  // x along the contiguous axis
      const int r = TTRANS ? y : x, c = TTRANS ? x : y;
      const bool in = TB * p + r < L && TB * p + c < L && r >= c;
      d[e] = A[in ? a_off(TB * p + r, TB * p + c) : 0];
      if (!in || (unit && r == c)) d[e] = r == c ? T(1) : T(0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int x = lr, y = 4 * e + lk;
      Wb(p)[(TTRANS ? y : x) * TIS + (TTRANS ? x : y)] = d[e];
    }
  }
  trsm_wave_sync();
  static_assert(TQ <= 4, "one lane group of 16 per diagonal block");
  {
    const int p = wave + TW * lk;
    const bool on = lk < TQ && p < nblk;
    T* W = Wb(on ? p : wave % nblk);
    const int o = lr & 8, c = lr & 7;
    T x[8], z[4];
    const T dinv = T(1) / W[lr * TIS + lr];
    // the block's two 8 x 8 triangles, columns by lane
#pragma unroll
    for (int r = 0; r < 8; ++r) x[r] = r == c ? T(1) : T(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const T d = __shfl(dinv, (lane & 56) + r, 64);
      x[r] = r < c ? T(0) : x[r] * d;  // zero above the diagonal, also for d infinite
#pragma unroll
      for (int i = r + 1; i < 8; ++i) x[i] -= W[(o + i) * TIS + o + r] * x[r];
    }
    trsm_wave_sync();
    if (on)
#pragma unroll
      for (int r = 0; r < 8; ++r) W[(o + r) * TIS + o + c] = x[r];
    trsm_wave_sync();
    // Z = L21 V0 (rows 4 (lr / 8) + y, column c), through the upper block
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      z[y] = T(0);
#pragma unroll
      for (int k = 0; k < 8; ++k) z[y] += W[(8 + (o >> 1) + y) * TIS + k] * W[k * TIS + c];
    }
    trsm_wave_sync();
    if (on)
#pragma unroll
      for (int y = 0; y < 4; ++y) W[((o >> 1) + y) * TIS + 8 + c] = z[y];
    trsm_wave_sync();
    T w21[4];
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      w21[y] = T(0);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        w21[y] -= W[(8 + (o >> 1) + y) * TIS + 8 + k] * W[k * TIS + 8 + c];
    }
    trsm_wave_sync();
    if (on)
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        W[(8 + (o >> 1) + y) * TIS + c] = w21[y];
        W[((o >> 1) + y) * TIS + 8 + c] = T(0);
      }
    trsm_wave_sync();
  }

  // (no load is moved above this point: the registers are needed above)
  asm volatile("" ::: "memory");
  // ---- NB vector blocks
  int left = std::min(nb, (int)(NV - j0 - 1) / TB + 1);
  for (;;) {
    // this wave's right-hand sides (accumulator layout)
    T vals[TQ][NB][4];
#pragma unroll
    for (int q = 0; q < TQ; ++q) {
      const int p = wave + TW * q;
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = TB * p + MfmaT<T>::row(lk, r);
          const bool in = i < L && j0 + TB * n + lr < (unsigned)NV;
          vals[q][n][r] = *(in ? b_at(p, r, n) : B);
          if (!in) vals[q][n][r] = T(0);
        }
    }
    // the triangle's first TD steps
    T t[TD][TQ][4];
#pragma unroll
    for (int u = 0; u < TD; ++u)
#pragma unroll
      for (int q = 0; q < TQ; ++q) {
        if (nblk > 1) load_t(q, u, t[u][q]);
      }
    // ---- forward substitution
    v4 acc[TQ][NB];
#pragma unroll
    for (int q = 0; q < TQ; ++q)
#pragma unroll
      for (int n = 0; n < NB; ++n) acc[q][n] = v4{0, 0, 0, 0};
    const T alpha = job.alpha;
    // X_p of block row p = wave + 16 q: to B, and to LDS for the later rows
    auto finish = [&](int p, const v4 (&x)[NB]) {
#pragma unroll
      for (int n = 0; n < NB; ++n) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          Xs[p & 1][(MfmaT<T>::row(lk, r) * NB + n) * TB + lr] = x[n][r];
      }
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = TB * p + MfmaT<T>::row(lk, r);
          if (i < L && j0 + TB * n + lr < (unsigned)NV) *b_at(p, r, n) = x[n][r];
        }
    };
    // X_p = W_p (alpha V_p - sum)
    auto solve = [&](int p, const T (&v)[NB][4], const v4 (&sum)[NB]) {
      T w[4];
      v4 x[NB];
#pragma unroll
      for (int s = 0; s < 4; ++s) w[s] = Wb(p)[lr * TIS + MfmaT<T>::row(lk, s)];
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        x[n] = v4{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          // the accumulator's item s is the operand of k-step s (same lane)
          const T rhs =
              TB * p + MfmaT<T>::row(lk, s) < L ? alpha * v[n][s] - sum[n][s] : T(0);
          x[n] = MfmaT<T>::mac(w[s], rhs, x[n]);
        }
      }
      finish(p, x);
    };
    if (wave == 0) solve(0, vals[0], acc[0]);
    __syncthreads();
    auto step = [&](int J, T (&tj)[TQ][4]) {
      T x[NB][4];
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int s = 0; s < 4; ++s) x[n][s] = Xs[J & 1][(tk(lk, s) * NB + n) * TB + lr];
      auto update = [&](int q) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int n = 0; n < NB; ++n) acc[q][n] = MfmaT<T>::mac(tj[q][s], x[n][s], acc[q][n]);
      };
      // the next block row first, ahead of the other waves
#pragma unroll
      for (int q = 0; q < TQ; ++q)
        if (wave + TW * q == J + 1 && J + 1 < nblk) {
          __builtin_amdgcn_s_setprio(3);
          update(q);
          solve(J + 1, vals[q], acc[q]);
          if (!prio) __builtin_amdgcn_s_setprio(0);  // back to the launch's own
        }
#pragma unroll
      for (int q = 0; q < TQ; ++q) {
        const int p = wave + TW * q;
        if (p > J + 1 && p < nblk) update(q);
      }
#pragma unroll
      for (int q = 0; q < TQ; ++q) load_t(q, J + TD, tj[q]);
      __syncthreads();
    };
    // steps past the last block row only load (again) and pass the barrier
#pragma unroll 1
    for (int J = 0; J + 1 < nblk; J += TD) {
#pragma unroll
      for (int u = 0; u < TD; ++u) step(J + u, t[u]);
    }
    if (!SHORT || (left -= NB) <= 0) break;
    j0 += TB * NB;
    brow += TB * NB * vstep;
  }
}

// ------------------------------------------------------------ host side
template <typename T>
int trsm_launch(const TrsmShape& sh, const TrsmJob<T>* jobs_dev, int njobs,
                const TrsmJob<T>& single, int L, long total_wg, const int* abort, hipStream_t s,
                int nb) {
  if (total_wg <= 0) return 0;
  if (total_wg > 0x7fffffffL) return arg_fail(0, "trsm: too many workgroups");
  const int nblk = (L + TB - 1) / TB, waves = std::min(nblk, TW);
  const size_t lds = nblk <= TW ? sizeof(T) * nblk * TB * TIS : 0;
#define DM_TRSM_NB(LO, TT, SL, N, SH)                                                              \
  hipLaunchKernelGGL((trsm_kernel<T, LO, TT, SL, N, SH>), dim3((unsigned)total_wg),                \
                     dim3(64 * waves), lds, s, jobs_dev, njobs, single, sh.unit ? 1 : 0,           \
                     single.prio, nb, abort)
#define DM_TRSM_GO(LO, TT, SL)                                                \
  do {                                                                        \
    if (nblk <= TW) {                                                         \
      if (nb > 1) DM_TRSM_NB(LO, TT, SL, 2, true);                            \
      else DM_TRSM_NB(LO, TT, SL, 1, true);                                   \
    } else {                                                                  \
      if (nb > 1) DM_TRSM_NB(LO, TT, SL, 2, false);                           \
      else DM_TRSM_NB(LO, TT, SL, 1, false);                                  \
    }                                                                         \
  } while (0)
  if (sh.lower) {
    if (sh.ttrans) { if (sh.side_l) DM_TRSM_GO(true, true, true); else DM_TRSM_GO(true, true, false); }
    else { if (sh.side_l) DM_TRSM_GO(true, false, true); else DM_TRSM_GO(true, false, false); }
  } else {
    if (sh.ttrans) { if (sh.side_l) DM_TRSM_GO(false, true, true); else DM_TRSM_GO(false, true, false); }
    else { if (sh.side_l) DM_TRSM_GO(false, false, true); else DM_TRSM_GO(false, false, false); }
  }
#undef DM_TRSM_GO
#undef DM_TRSM_NB
  DM_LAUNCH_CHECK("trsm_kernel");
  return 0;
}

// Unbatched solve, recursive above one leaf.
template <typename T>
static int trsm_eff(const TrsmShape& sh, int L, int NV, T alpha, const T* A, int lda, T* B,
                    int ldb, const int* abort, hipStream_t s) {
  if (L <= 0 || NV <= 0) return 0;
  if (L <= TRSM_LEAF) {
    TrsmJob<T> j{};
    j.A = A; j.B = B; j.L = L; j.NV = NV; j.lda = lda; j.ldb = ldb; j.alpha = alpha;
    const int nb = trsm_vec_blocks(L, NV);
    return trsm_launch<T>(sh, nullptr, 0, j, L, trsm_wgs(NV, nb), abort, s, nb);
  }
  const TrsmSplit sp = trsm_split(sh, L);
  int rc = trsm_eff<T>(sh, sp.first_n, NV, alpha, tm_sub(sh, A, lda, sp.first_r, sp.first_r), lda,
                       vsub(sh, B, ldb, sp.first_r), ldb, abort, s);
  if (rc) return rc;
  bool ta, tb;
  const GemmJob<T> g = trsm_update_job<T>(sh, sp, NV, alpha, A, lda, B, ldb, ta, tb);
  rc = gemm_single<T>(ta, tb, g.M, g.N, g.K, g.alpha, g.A, g.lda, g.B, g.ldb, g.beta, g.C, g.ldc, 0,
                      abort, s);
  if (rc) return rc;
  return trsm_eff<T>(sh, sp.second_n, NV, T(1), tm_sub(sh, A, lda, sp.second_r, sp.second_r), lda,
                     vsub(sh, B, ldb, sp.second_r), ldb, abort, s);
}

template <typename T>
int trsm_full(char side, char uplo, char transa, char diag, int m, int n, T alpha, const T* A,
              int lda, T* B, int ldb, const int* abort, hipStream_t s) {
  const TrsmShape sh = trsm_shape(side, uplo, transa, diag);
  const int L = sh.side_l ? m : n;
  const int NV = sh.side_l ? n : m;
  if (m <= 0 || n <= 0) return 0;
  if (alpha == T(0)) {
    // B := 0 (BLAS: A not referenced)
    return gemm_single<T>(false, false, m, n, 0, T(0), B, ldb, B, ldb, T(0), B, ldb, 0, abort, s);
  }
  return trsm_eff<T>(sh, L, NV, alpha, A, lda, B, ldb, abort, s);
}

template int trsm_launch<double>(const TrsmShape&, const TrsmJob<double>*, int,
                                 const TrsmJob<double>&, int, long, const int*, hipStream_t, int);
template int trsm_launch<float>(const TrsmShape&, const TrsmJob<float>*, int,
                                const TrsmJob<float>&, int, long, const int*, hipStream_t, int);
template int trsm_full<double>(char, char, char, char, int, int, double, const double*, int,
                               double*, int, const int*, hipStream_t);
template int trsm_full<float>(char, char, char, char, int, int, float, const float*, int, float*,
                              int, const int*, hipStream_t);

}  // namespace dm
