// Complex (ComplexF64 / ComplexF32) tile operations of the tiled Cholesky
// and its solves: LAPACK.potrf!, BLAS.trsm!, BLAS.herk! and BLAS.gemm! with
// conjugate transposes, as _chol! calls them for T <: Complex
// (src/array/cholesky.jl:27-28,44-45,48-50,89-95) and trsm! passes 'C'
// through to its GEMM tasks (src/array/trsm.jl:103-111,157-163).
//
// Elements are (re, im) pairs of R (Julia's layout).  Design:
//  * GEMM/HERK: tiles of C of 64 x 64 or 32 x 32, 4 waves, on the real matrix
//    cores (v_mfma_f64_16x16x4f64 / v_mfma_f32_16x16x4f32): each complex
//    product takes four real ones, re += ar*br - ai*bi, im += ar*bi + ai*br.
//    op(A) and op(B) are staged into LDS as separate re/im planes with the
//    conjugation of 'C' applied while staging.  HERK is the same kernel
//    restricted to one triangle of C with the imaginary part of C's diagonal
//    set to zero (BLAS herk semantics).
//  * POTRF: the recursion n -> (n1, n2) of LAPACK's potrf2 (factor A11;
//    A12 := A11^-H A12 / A21 := A21 A11^-H; A22 -= herk; factor A22) down to
//    64 x 64 leaves factored in the registers of one workgroup.
//  * TRSM: the same recursion on the triangle (solve, GEMM update, solve)
//    down to 256 x 256 leaves, where a workgroup solves 16 right-hand-side
//    vectors by block rows of 16: substitution within a block row, products on
//    the matrix cores between them.
// Every kernel returns at once when the abort word is set (a failed pivot),
// so the rest of a failed factorization becomes a no-op.
#include <algorithm>
#include "dm_internal.h"
#include "complex_ops.h"
#include "potrf_diag.h"

namespace dm {

namespace {

template <typename R> using Mf = PMfma<R>;

constexpr int ZLEAF = 64;         // POTRF leaf
constexpr int ZTB = 16;           // TRSM block row
constexpr int ZTRSM_LEAF = 256;   // TRSM leaf: one block row per wave of a workgroup

// C = alpha op(A) op(B) + beta C on one ZT x ZT tile per workgroup, k by ZBK
// steps.  A step's elements are loaded into registers a step ahead and written
// to LDS as separate re/im planes (the other buffer) after the products.
//
// Bound by the matrix cores on tiles of 64 (2048 x 2048 x 256 FP64: 191 us, 262
// before the loads were taken a step ahead); a launch with too few of those to
// fill the chip takes tiles of 32 (zgemm_launch; 256 x 256 x 256: 20 us, 74 in
// tiles of 64 without the prefetch).
template <typename R, int ZT, int ZBK>
__global__ __launch_bounds__(256) void zgemm_kernel(ZGemmArgs<R> g, const int* __restrict__ abort) {
  typedef typename Mf<R>::v4 v4;
  typedef R v2 __attribute__((ext_vector_type(2)));
  constexpr int ZS = ZT + 4;        // LDS row stride of the [k][mn] planes
  constexpr int W = ZT / 2, MI = W / 16, NQ = ZT * ZBK / 256;
  __shared__ R As[2][2][ZBK * ZS];  // [buffer][re/im][k * ZS + m]
  __shared__ R Bs[2][2][ZBK * ZS];  // [buffer][re/im][k * ZS + n]
  if (abort && *abort) return;
  const int tiles_m = (g.M + ZT - 1) / ZT;
  const int m0 = (blockIdx.x % tiles_m) * ZT, n0 = (blockIdx.x / tiles_m) * ZT;
  if (g.tri == 1 && m0 > n0 + ZT - 1) return;  // tile below the upper triangle
  if (g.tri == 2 && n0 > m0 + ZT - 1) return;  // tile above the lower triangle
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int wm0 = (wave & 1) * W, wn0 = (wave >> 1) * W;
  v4 cre[MI][MI], cim[MI][MI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j) cre[i][j] = cim[i][j] = v4{0, 0, 0, 0};

  // this thread's NQ elements of each operand per step: op(A)[m, k] reads
  // X[k, m] for 'T' and 'C' (k contiguous in memory: lanes walk k first), X[m, k]
  // else; op(B)[k, n] the other way round.  Rows and columns past the end read
  // the last ones (their results are dropped), k past the end gives zero.
  const bool kfa = g.opa == 1 || g.opa == 2, kfb = g.opb == 0 || g.opb == 3;
  const R sa = g.opa >= 2 ? R(-1) : R(1), sb = g.opb >= 2 ? R(-1) : R(1);
  int ak[NQ], bk[NQ], as[NQ], bs[NQ];
  const v2* ap[NQ];
  const v2* bp[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int e = tid + 256 * q;
    const int am = kfa ? e / ZBK : e % ZT, bn = kfb ? e / ZBK : e % ZT;
    ak[q] = kfa ? e % ZBK : e / ZT;
    bk[q] = kfb ? e % ZBK : e / ZT;
    as[q] = ak[q] * ZS + am;
    bs[q] = bk[q] * ZS + bn;
    const int m = min(m0 + am, g.M - 1), n = min(n0 + bn, g.N - 1);
    ap[q] = (const v2*)g.A + (kfa ? (int64_t)m * g.lda : m);
    bp[q] = (const v2*)g.B + (kfb ? (int64_t)n * g.ldb : n);
  }
  const int64_t astep = kfa ? 1 : g.lda, bstep = kfb ? 1 : g.ldb;
  v2 av[NQ], bv[NQ];
  auto load = [&](int k0) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      av[q] = *gptr(ap[q] + min(k0 + ak[q], g.K - 1) * astep);
      bv[q] = *gptr(bp[q] + min(k0 + bk[q], g.K - 1) * bstep);
    }
  };
  auto store = [&](int buf, int k0) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const bool a = k0 + ak[q] < g.K, b = k0 + bk[q] < g.K;
      As[buf][0][as[q]] = a ? av[q].x : R(0);
      As[buf][1][as[q]] = a ? sa * av[q].y : R(0);
      Bs[buf][0][bs[q]] = b ? bv[q].x : R(0);
      Bs[buf][1][bs[q]] = b ? sb * bv[q].y : R(0);
    }
  };
  const int nk = (g.K + ZBK - 1) / ZBK;
  if (nk > 0) {
    load(0);
    store(0, 0);
  }
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < nk;
    if (more) load((kt + 1) * ZBK);
#pragma unroll
    for (int kk = 0; kk < ZBK / 4; ++kk) {
      const int k = kk * 4 + lk;
      R ar[MI], ai[MI], br[MI], bi[MI], nbi[MI];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        ar[i] = As[cur][0][k * ZS + wm0 + i * 16 + lr];
        ai[i] = As[cur][1][k * ZS + wm0 + i * 16 + lr];
      }
#pragma unroll
      for (int j = 0; j < MI; ++j) {
        br[j] = Bs[cur][0][k * ZS + wn0 + j * 16 + lr];
        bi[j] = Bs[cur][1][k * ZS + wn0 + j * 16 + lr];
        nbi[j] = -bi[j];
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j) {
          cre[i][j] = Mf<R>::mac(br[j], ar[i], cre[i][j]);
          cim[i][j] = Mf<R>::mac(bi[j], ar[i], cim[i][j]);
          cre[i][j] = Mf<R>::mac(nbi[j], ai[i], cre[i][j]);
          cim[i][j] = Mf<R>::mac(br[j], ai[i], cim[i][j]);
        }
    }
    if (more) store(cur ^ 1, (kt + 1) * ZBK);  // read in step kt-1, ended by its barrier
    __syncthreads();
  }
  // lane holds C[m][n], m = m0 + wm0 + 16i + lr, n = n0 + wn0 + 16j + row(lk, r)
  const bool bz = g.beta_re == R(0) && g.beta_im == R(0);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm0 + i * 16 + lr, n = n0 + wn0 + j * 16 + Mf<R>::row(lk, r);
        bool ok = m < g.M && n < g.N;
        if (g.tri == 1) ok = ok && m <= n;
        else if (g.tri == 2) ok = ok && m >= n;
        if (!ok) continue;
        const R pr = cre[i][j][r], pi = cim[i][j][r];
        R vr = g.alpha_re * pr - g.alpha_im * pi;
        R vi = g.alpha_re * pi + g.alpha_im * pr;
        auto c = gptr((v2*)(g.C + 2 * ((int64_t)n * g.ldc + m)));
        if (!bz) {
          const v2 o = *c;
          vr += g.beta_re * o.x - g.beta_im * o.y;
          vi += g.beta_re * o.y + g.beta_im * o.x;
        }
        if (g.herk && m == n) vi = R(0);
        *c = v2{vr, vi};
      }
}

// Cholesky of an n x n (n <= 64) Hermitian block in place, one workgroup:
// the 'U' factor in the upper triangle (A = U^H U) or the 'L' factor in the
// lower one (A = L L^H); the other strict triangle is left alone.  The
// diagonal's imaginary part is ignored and set to zero (LAPACK potrf2).  A
// non-positive or NaN pivot at column j sets *info = info_off + j + 1 (when
// *info is 0) and the abort word to global_base + info_off + j + 1 (the
// global column, as the real kernels report it), and leaves the block
// partly factored.
//
// Thread (tx, ty) of 16 x 16 holds the elements (ty + 16 i, tx + 16 k) of the
// upper view (A, or A^T for 'L': both factor as M[x][y] -= conj(M[j][x]) M[j][y])
// in registers.  A column is one barrier: the owners of row j put it into LDS
// unscaled, and every thread scales it by the pivot's reciprocal root itself.
// Bound by that chain.  64 columns: 34 us FP64, against 101 us with the block in
// LDS (three barriers a column, an integer division per element).
template <typename R, bool UPPER>
__global__ __launch_bounds__(256) void zpotrf_leaf_kernel(R* __restrict__ A, int n, int lda,
                                                          int* __restrict__ info, int info_off,
                                                          int* __restrict__ abort,
                                                          int global_base) {
  typedef R v2 __attribute__((ext_vector_type(2)));
  constexpr int NB = ZLEAF / 16;
  __shared__ v2 row[2][ZLEAF];
  if (abort && *abort) return;
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  v2 m[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int x = ty + 16 * i, y = tx + 16 * k;
      const int r = UPPER ? x : y, c = UPPER ? y : x;
      m[i][k] = v2{x == y ? R(1) : R(0), R(0)};
      if (x <= y && y < n) m[i][k] = *gptr((const v2*)A + (int64_t)c * lda + r);
    }
  bool failed = false;
#pragma unroll
  for (int jb = 0; jb < NB; ++jb)
#pragma unroll 1
    for (int jj = 0; jj < 16; ++jj) {
      const int j = 16 * jb + jj;
      if (failed || j >= n) break;
      v2* const s = row[j & 1];
      if (ty == jj)
#pragma unroll
        for (int k = jb; k < NB; ++k) s[tx + 16 * k] = m[jb][k];
      __syncthreads();
      const R d = s[j].x;
      if (!(d > R(0))) {
        if (tid == 0) {
          if (info && *info == 0) *info = info_off + j + 1;
          if (abort) *abort = global_base + info_off + j + 1;
        }
        failed = true;
        break;
      }
      const bool fast = PivotBits<R>::of(d) <= PivotBits<R>::span;
      const R inv = fast ? inv_sqrt(d) : R(1) / R(sqrt(d));
      v2 u[NB], v[NB];
#pragma unroll
      for (int k = jb; k < NB; ++k) {
        u[k] = s[ty + 16 * k] * inv;
        v[k] = s[tx + 16 * k] * inv;
      }
      if (ty == jj) {
#pragma unroll
        for (int k = jb; k < NB; ++k) m[jb][k] = v[k];
        if (tx == jj) m[jb][jb] = v2{fast ? sqrt_of(d) : R(sqrt(d)), R(0)};
      }
#pragma unroll
      for (int i = jb; i < NB; ++i)
        if (i > jb || ty > jj)
#pragma unroll
          for (int k = i; k < NB; ++k) {
            m[i][k].x -= u[i].x * v[k].x + u[i].y * v[k].y;
            m[i][k].y -= u[i].x * v[k].y - u[i].y * v[k].x;
          }
    }
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int x = ty + 16 * i, y = tx + 16 * k;
      const int r = UPPER ? x : y, c = UPPER ? y : x;
      if (x <= y && y < n) *gptr((v2*)A + (int64_t)c * lda + r) = m[i][k];
    }
}

// -1 / d, scaled by the larger part: no square over- or underflows.
template <typename V> __device__ __forceinline__ V neg_recip(V d) {
  if (fabs(d.x) >= fabs(d.y)) {
    const auto r = d.y / d.x, n = -1 / (d.x + d.y * r);
    return V{n, -r * n};
  }
  const auto r = d.x / d.y, n = -1 / (d.x * r + d.y);
  return V{r * n, -n};
}

// Solves op(T) x = alpha b for the vectors of B, T an L x L (L <= 256)
// triangle.  Vector v's element i is B[v * vstride + i * estride].  op: 0 T,
// 1 T^T, 2 T^H, 3 conj(T).  A workgroup owns 16 vectors and the whole triangle,
// its wave p block row p of 16; an upper op(T) is solved as the lower triangle
// that reversing both axes gives.  As in the real kernel, right-hand sides stay
// in registers and sums in accumulators:
//   T_pp X_p = alpha V_p - sum_{k<p} T_pk X_k,
// each complex product four real ones, T straight from global memory, the
// diagonal block from LDS by substitution (see pb_solve: the product with its
// inverse loses accuracy where it is badly conditioned).
//
// Bound by the matrix cores (256 rows are 13 us of products on one CU) and the
// chain from block to block (two block products and a barrier, about 1 us
// each).  256 rows FP64: 16 vectors 45-46 us, 2048 48-49 us, 20000 225-232 us,
// against 670-700, 680-700 and 1350 us for the launches this replaces (four leaves
// of 64 rows at 145 us, one thread a vector walking the triangle in LDS, and the
// products between them).  One step of T in flight in FP64: with two the
// registers of 16 waves do not hold the substitution's operands (16 vectors 51 us).
//
// SHORT: up to 32 rows, with a loop over the vectors in each workgroup and the
// diagonal blocks in as much LDS as they need (the LDS of 256 rows lets a CU hold
// one workgroup of one or two waves): 1 row, 2000000 vectors FP64 72 us, 671
// without, 16 rows, 1000000 vectors 100 and 435; from 64 rows on the loop's
// registers cost more than it gives (100000 vectors 184 and 142 us).
template <typename R, bool SHORT>
__global__ __launch_bounds__(SHORT ? 512 : 1024) void ztrsm_leaf_kernel(const R* __restrict__ T, int L, int ldt,
                                                          bool lower, int op, bool unit,
                                                          R alpha_re, R alpha_im,
                                                          R* __restrict__ B, int64_t estride,
                                                          int64_t vstride, int nvec, int nb,
                                                          const int* __restrict__ abort) {
  typedef typename Mf<R>::v4 v4;
  typedef R v2 __attribute__((ext_vector_type(2)));
  constexpr int S = ZTB + 1, D = sizeof(R) == 4 ? 2 : 1;  // LDS row stride; steps of T in flight
  __shared__ v2 Xs[2][ZTB * ZTB];  // X_J: [row][vector]
  if (abort && *abort) return;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int p = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  const int nblk = (L + ZTB - 1) / ZTB;
  const bool tt = op == 1 || op == 2, lo = tt ? !lower : lower;
  const R sg = op >= 2 ? R(-1) : R(1);  // conjugation
  // element (i, k) of the lower triangle: t0[i * rs + k * cs]
  int64_t rs = tt ? ldt : 1, cs = tt ? 1 : ldt, es = estride;
  const v2* t0 = (const v2*)T;
  v2* b0 = (v2*)B;
  if (!lo) {
    t0 += (L - 1) * (rs + cs);
    b0 += (L - 1) * es;
    rs = -rs;
    cs = -cs;
    es = -es;
  }
  // T_pJ as the operand of four k-steps: row 16 p + lr, columns 16 J + 2 lk + tk(s)
  auto tk = [](int s) { return (s & 1) + 8 * (s >> 1); };
  const v2* const trow = t0 + min(ZTB * p + lr, L - 1) * rs + 2 * lk * cs;
  auto load_t = [&](int J, v2 (&t)[4]) {
    if (J >= p) return;
#pragma unroll
    for (int s = 0; s < 4; ++s) t[s] = *gptr(trow + (ZTB * J + tk(s)) * cs);
  };
  // ---- the diagonal block, the identity's past the end, and -1 / T_rr
  constexpr int TE = ZTB * S + ZTB;  // LDS elements of both
  v2* W;
  if constexpr (SHORT) {
    DM_DYNAMIC_LDS(ztrsm_lds);
    W = (v2*)ztrsm_lds + p * TE;
  } else {
    __shared__ v2 Td[ZTRSM_LEAF / ZTB][TE];
    W = Td[p];
  }
  v2* const Rd = W + ZTB * S;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int x = lr, y = 4 * e + lk;  // x along the contiguous axis
    const int r = tt ? y : x, c = tt ? x : y;
    const bool in = ZTB * p + r < L && ZTB * p + c < L && r >= c;
    v2 d = v2{r == c ? R(1) : R(0), R(0)};
    if (in && !(unit && r == c)) {
      d = *gptr(t0 + (ZTB * p + r) * rs + (ZTB * p + c) * cs);
      d.y *= sg;
    }
    W[r * S + c] = d;
    if (r == c) Rd[r] = neg_recip(d);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  unsigned j0 = blockIdx.x * (unsigned)(ZTB * (SHORT ? nb : 1));
  int left = std::min(nb, (int)(nvec - j0 - 1) / ZTB + 1);
  for (;;) {
    asm volatile("" ::: "memory");  // (no operand is kept from one pass to the next)
    v2 t[D][4];
#pragma unroll
    for (int u = 0; u < D; ++u) load_t(u, t[u]);
    // the right-hand side in the accumulator layout
    v2 v[4];
    v2* const bvec = b0 + (int64_t)(j0 + lr) * vstride;
    const bool mine = j0 + lr < (unsigned)nvec;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = ZTB * p + Mf<R>::row(lk, r);
      v[r] = v2{0, 0};
      if (mine && i < L) v[r] = *gptr((const v2*)bvec + i * es);
    }
    // ---- forward substitution
    v4 ar = v4{0, 0, 0, 0}, ai = v4{0, 0, 0, 0};
    // X_p from the sums: four rows at a time by substitution, a product of depth 4
    // for the rows below, in sums of the opposite sign (as pb_solve).  The operands
    // of a step are read while the matrix cores are at the one before.
    v2 u[4][4], q[4];
    auto read = [&](int s) {
      const int o = 4 * s;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int k = 0; k < i; ++k) u[i][k] = W[(o + i) * S + o + k];
        q[i] = Rd[o + i];
      }
    };
    auto solve = [&] {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bool in = ZTB * p + Mf<R>::row(lk, s) < L;
        ar[s] = in ? ar[s] - (alpha_re * v[s].x - alpha_im * v[s].y) : R(0);
        ai[s] = in ? ai[s] - (alpha_re * v[s].y + alpha_im * v[s].x) : R(0);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int o = 4 * s;
        if (SHORT && ZTB * p + o >= L) break;
        R xr[4], xi[4];
        four_rows(ar, s, xr);
        four_rows(ai, s, xi);
        const v2 a = W[lr * S + o + lk];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int k = 0; k < i; ++k) {
            const v2 d = u[i][k];
            xr[i] += d.x * xr[k];
            xi[i] += d.x * xi[k];
            xr[i] -= d.y * xi[k];
            xi[i] += d.y * xr[k];
          }
          const v2 d = q[i];
          const R w = xr[i];
          xr[i] = w * d.x - xi[i] * d.y;
          xi[i] = w * d.y + xi[i] * d.x;
        }
        const v2 x = v2{row_by_group(xr, s), row_by_group(xi, s)};
        if (s < 3) {
          ar = Mf<R>::mac(a.x, x.x, ar);
          ai = Mf<R>::mac(a.x, x.y, ai);
          ar = Mf<R>::mac(-a.y, x.y, ar);
          __builtin_amdgcn_sched_barrier(0);
          read(s + 1);
          __builtin_amdgcn_sched_barrier(0);
          ai = Mf<R>::mac(a.y, x.x, ai);
        }
        const int i = ZTB * p + o + lk;
        Xs[p & 1][(o + lk) * ZTB + lr] = x;
        if (mine && i < L) *gptr(bvec + i * es) = x;
      }
    };
    if (p == 0) {
      read(0);
      solve();
    }
    __syncthreads();
    auto step = [&](int J, v2 (&tj)[4]) {
      if (J < p && J + 1 < nblk) {
        if (p == J + 1) {
          __builtin_amdgcn_s_setprio(3);
          read(0);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const v2 x = Xs[J & 1][(2 * lk + tk(s)) * ZTB + lr];
          const R tr = tj[s].x, ti = sg * tj[s].y;
          ar = Mf<R>::mac(tr, x.x, ar);
          ai = Mf<R>::mac(tr, x.y, ai);
          ar = Mf<R>::mac(-ti, x.y, ar);
          ai = Mf<R>::mac(ti, x.x, ai);
        }
        if (p == J + 1) {
          solve();
          __builtin_amdgcn_s_setprio(0);
        }
        load_t(J + D, tj);
      }
      __syncthreads();
    };
#pragma unroll 1
    for (int J = 0; J + 1 < nblk; J += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) step(J + u, t[u]);
    }
    if (!SHORT || --left <= 0) break;
    j0 += ZTB;
  }
}

int op_code(char t) { return is_notrans(t) ? 0 : (t == 'T' || t == 't') ? 1 : 2; }

int split_point(int n) { return ((n / 2 + 31) / 32) * 32; }

}  // namespace

template <typename R>
int zgemm_launch(const ZGemmArgs<R>& g, const int* abort, hipStream_t s) {
  if (g.M <= 0 || g.N <= 0) return 0;
  // tiles of 64 once they fill the 256 CUs, else four times as many of 32
  auto tiles = [&](long t) { return ((g.M + t - 1) / t) * ((g.N + t - 1) / t); };
  const bool big = tiles(64) >= 256;
  const long n = tiles(big ? 64 : 32);
  if (n > 0x7fffffffL) return arg_fail(0, "zgemm: too many tiles");
  if (big)
    hipLaunchKernelGGL((zgemm_kernel<R, 64, 8>), dim3((unsigned)n), dim3(256), 0, s, g, abort);
  else
    hipLaunchKernelGGL((zgemm_kernel<R, 32, 16>), dim3((unsigned)n), dim3(256), 0, s, g, abort);
  DM_LAUNCH_CHECK("zgemm_kernel");
  return 0;
}

template <typename R>
int zgemm_call(char ta, char tb, int m, int n, int k, R ar, R ai, const R* A, int lda, const R* B,
               int ldb, R br, R bi, R* C, int ldc, int tri, int herk, const int* abort,
               hipStream_t s) {
  ZGemmArgs<R> g{};
  g.A = A; g.B = B; g.C = C;
  g.M = m; g.N = n; g.K = (ar == R(0) && ai == R(0)) ? 0 : k;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.alpha_re = ar; g.alpha_im = ai; g.beta_re = br; g.beta_im = bi;
  g.opa = op_code(ta); g.opb = op_code(tb);
  g.tri = tri; g.herk = herk;
  return zgemm_launch<R>(g, abort, s);
}

// trsm(side, uplo, trans, diag, alpha, T, B) by recursion on the triangle
template <typename R>
int ztrsm_rec(bool left, bool lower, int op, bool unit, int L, R ar, R ai, const R* T, int ldt,
              R* B, int ldb, int nv, const int* abort, hipStream_t s) {
  if (L <= 0 || nv <= 0) return 0;
  if (L <= ZTRSM_LEAF) {
    // left: vectors are B's columns; right: x op(T) = b as op(T)^T x^T = b^T
    // on B's rows (op N<->T, H<->conj)
    const int lop = left ? op : (op == 0 ? 1 : op == 1 ? 0 : op == 2 ? 3 : 2);
    const int64_t es = left ? 1 : ldb, vs = left ? ldb : 1;
    const int nblk = (L + ZTB - 1) / ZTB;
    const long blocks = ((long)nv + ZTB - 1) / ZTB;
    if (nblk <= 2) {
      // from two rounds of 12 waves a CU on, one round takes all vectors
      const long round = 256 * 12 / nblk;
      const int nb = blocks < 2 * round ? 1 : (int)((blocks + round - 1) / round);
      const size_t lds = 2 * sizeof(R) * nblk * (ZTB * (ZTB + 1) + ZTB);
      hipLaunchKernelGGL((ztrsm_leaf_kernel<R, true>), dim3((unsigned)((blocks + nb - 1) / nb)),
                         dim3(64 * nblk), lds, s, T, L, ldt, lower, lop, unit, ar, ai, B, es, vs, nv,
                         nb, abort);
    } else {
      hipLaunchKernelGGL((ztrsm_leaf_kernel<R, false>), dim3((unsigned)blocks), dim3(64 * nblk), 0, s,
                         T, L, ldt, lower, lop, unit, ar, ai, B, es, vs, nv, 1, abort);
    }
    DM_LAUNCH_CHECK("ztrsm_leaf_kernel");
    return 0;
  }
  const int P = split_point(L), Q = L - P;
  const R* T11 = T;
  const R* T22 = T + 2 * ((int64_t)P * ldt + P);
  const R* T21 = T + 2 * (int64_t)P;               // rows P.., cols 0..P-1
  const R* T12 = T + 2 * ((int64_t)P * ldt);       // rows 0..P-1, cols P..
  const bool lo = (op == 0) ? lower : !lower;      // op(T) lower
  const char opc = op == 0 ? 'N' : op == 1 ? 'T' : 'C';
  // op(T)21 = op(T21) for N, op(T12) for T/H; op(T)12 the mirror
  const R* O21 = op == 0 ? T21 : T12;
  const R* O12 = op == 0 ? T12 : T21;
  int rc;
  if (left) {
    R* B1 = B;
    R* B2 = B + 2 * (int64_t)P;  // rows P..
    if (lo) {
      if ((rc = ztrsm_rec<R>(true, lower, op, unit, P, ar, ai, T11, ldt, B1, ldb, nv, abort, s))) return rc;
      if ((rc = zgemm_call<R>(opc, 'N', Q, nv, P, R(-1), R(0), O21, ldt, B1, ldb, ar, ai, B2, ldb, 0, 0, abort, s))) return rc;
      return ztrsm_rec<R>(true, lower, op, unit, Q, R(1), R(0), T22, ldt, B2, ldb, nv, abort, s);
    }
    if ((rc = ztrsm_rec<R>(true, lower, op, unit, Q, ar, ai, T22, ldt, B2, ldb, nv, abort, s))) return rc;
    if ((rc = zgemm_call<R>(opc, 'N', P, nv, Q, R(-1), R(0), O12, ldt, B2, ldb, ar, ai, B1, ldb, 0, 0, abort, s))) return rc;
    return ztrsm_rec<R>(true, lower, op, unit, P, R(1), R(0), T11, ldt, B1, ldb, nv, abort, s);
  }
  // right: X op(T) = alpha B, B = [B1 B2] by columns, nv = rows of B
  R* B1 = B;
  R* B2 = B + 2 * ((int64_t)P * ldb);
  if (!lo) {  // op(T) upper: X1 first, then X2 op(T)22 = alpha B2 - X1 op(T)12
    if ((rc = ztrsm_rec<R>(false, lower, op, unit, P, ar, ai, T11, ldt, B1, ldb, nv, abort, s))) return rc;
    if ((rc = zgemm_call<R>('N', opc, nv, Q, P, R(-1), R(0), B1, ldb, O12, ldt, ar, ai, B2, ldb, 0, 0, abort, s))) return rc;
    return ztrsm_rec<R>(false, lower, op, unit, Q, R(1), R(0), T22, ldt, B2, ldb, nv, abort, s);
  }
  if ((rc = ztrsm_rec<R>(false, lower, op, unit, Q, ar, ai, T22, ldt, B2, ldb, nv, abort, s))) return rc;
  if ((rc = zgemm_call<R>('N', opc, nv, P, Q, R(-1), R(0), B2, ldb, O21, ldt, ar, ai, B1, ldb, 0, 0, abort, s))) return rc;
  return ztrsm_rec<R>(false, lower, op, unit, P, R(1), R(0), T11, ldt, B1, ldb, nv, abort, s);
}

template <typename R>
int ztrsm_call(char side, char uplo, char trans, char diag, int m, int n, R ar, R ai, const R* A,
               int lda, R* B, int ldb, const int* abort, hipStream_t s) {
  const bool left = is_left(side);
  return ztrsm_rec<R>(left, is_lower(uplo), op_code(trans), is_unit(diag), left ? m : n, ar, ai,
                      A, lda, B, ldb, left ? n : m, abort, s);
}

// potrf(uplo, A) by potrf2's recursion; info gets the global 1-based column
// of the first failed pivot (offset info_off), abort is set with it.
template <typename R>
int zpotrf_rec(bool upper, int n, R* A, int lda, int* info, int info_off, int* abort,
               int global_base, hipStream_t s) {
  if (n <= 0) return 0;
  if (n <= ZLEAF) {
    if (upper)
      hipLaunchKernelGGL((zpotrf_leaf_kernel<R, true>), dim3(1), dim3(256), 0, s, A, n, lda, info,
                         info_off, abort, global_base);
    else
      hipLaunchKernelGGL((zpotrf_leaf_kernel<R, false>), dim3(1), dim3(256), 0, s, A, n, lda, info,
                         info_off, abort, global_base);
    DM_LAUNCH_CHECK("zpotrf_leaf_kernel");
    return 0;
  }
  const int P = split_point(n), Q = n - P;
  R* A11 = A;
  R* A22 = A + 2 * ((int64_t)P * lda + P);
  int rc = zpotrf_rec<R>(upper, P, A11, lda, info, info_off, abort, global_base, s);
  if (rc) return rc;
  if (upper) {
    R* A12 = A + 2 * ((int64_t)P * lda);
    if ((rc = ztrsm_call<R>('L', 'U', 'C', 'N', P, Q, R(1), R(0), A11, lda, A12, lda, abort, s))) return rc;
    if ((rc = zgemm_call<R>('C', 'N', Q, Q, P, R(-1), R(0), A12, lda, A12, lda, R(1), R(0), A22, lda, 1, 1, abort, s))) return rc;
  } else {
    R* A21 = A + 2 * (int64_t)P;
    if ((rc = ztrsm_call<R>('R', 'L', 'C', 'N', Q, P, R(1), R(0), A11, lda, A21, lda, abort, s))) return rc;
    if ((rc = zgemm_call<R>('N', 'C', Q, Q, P, R(-1), R(0), A21, lda, A21, lda, R(1), R(0), A22, lda, 2, 1, abort, s))) return rc;
  }
  return zpotrf_rec<R>(upper, Q, A22, lda, info, info_off + P, abort, global_base, s);
}

template int zgemm_call<double>(char, char, int, int, int, double, double, const double*, int,
                                const double*, int, double, double, double*, int, int, int,
                                const int*, hipStream_t);
template int zgemm_call<float>(char, char, int, int, int, float, float, const float*, int,
                               const float*, int, float, float, float*, int, int, int, const int*,
                               hipStream_t);
template int ztrsm_call<double>(char, char, char, char, int, int, double, double, const double*,
                                int, double*, int, const int*, hipStream_t);
template int ztrsm_call<float>(char, char, char, char, int, int, float, float, const float*, int,
                               float*, int, const int*, hipStream_t);
template int zpotrf_rec<double>(bool, int, double*, int, int*, int, int*, int, hipStream_t);
template int zpotrf_rec<float>(bool, int, float*, int, int*, int, int*, int, hipStream_t);

}  // namespace dm

// ------------------------------------------------------------ C ABI
using namespace dm;

namespace {

template <typename R>
int zpotrf_api(char uplo, int n, void* A, int lda, int* info_dev, dm_stream_t s) {
  if (!is_upper(uplo) && !is_lower(uplo)) return arg_fail(1, "uplo must be 'U' or 'L'");
  if (n < 0) return arg_fail(2, "n < 0");
  if (lda < (n > 1 ? n : 1)) return arg_fail(4, "lda < max(1,n)");
  if (!info_dev) return arg_fail(5, "info is NULL");
  int rc = ensure_init();
  if (rc) return rc;
  hipStream_t st = stream_of(s);
  // the abort word of this call: a failed pivot makes the rest of the
  // recursion a no-op (per-stream scratch; calls on one stream are ordered)
  int* abort = (int*)stream_workspace(st, 256);
  if (!abort) return arg_fail(0, "potrf: workspace allocation failed");
  if ((rc = fill_i32_launch(info_dev, 0, 1, st))) return rc;
  if ((rc = fill_i32_launch(abort, 0, 1, st))) return rc;
  return zpotrf_rec<R>(is_upper(uplo), n, (R*)A, lda, info_dev, 0, abort, 0, st);
}

template <typename R>
int ztrsm_api(char side, char uplo, char transa, char diag, int m, int n, const R* alpha,
              const void* A, int lda, void* B, int ldb, dm_stream_t s) {
  if (!is_left(side) && !is_right(side)) return arg_fail(1, "side must be 'L' or 'R'");
  if (!is_upper(uplo) && !is_lower(uplo)) return arg_fail(2, "uplo must be 'U' or 'L'");
  if (!is_trans(transa) && !is_notrans(transa)) return arg_fail(3, "transa must be 'N','T','C'");
  if (!is_unit(diag) && !is_nonunit(diag)) return arg_fail(4, "diag must be 'N' or 'U'");
  if (m < 0) return arg_fail(5, "m < 0");
  if (n < 0) return arg_fail(6, "n < 0");
  if (!alpha) return arg_fail(7, "alpha is NULL");
  const int ka = is_left(side) ? m : n;
  if (lda < (ka > 1 ? ka : 1)) return arg_fail(9, "lda too small");
  if (ldb < (m > 1 ? m : 1)) return arg_fail(11, "ldb < max(1,m)");
  int rc = ensure_init();
  if (rc) return rc;
  return ztrsm_call<R>(side, uplo, transa, diag, m, n, alpha[0], alpha[1], (const R*)A, lda,
                       (R*)B, ldb, nullptr, stream_of(s));
}

template <typename R>
int zherk_api(char uplo, char trans, int n, int k, R alpha, const void* A, int lda, R beta,
              void* C, int ldc, dm_stream_t s) {
  if (!is_upper(uplo) && !is_lower(uplo)) return arg_fail(1, "uplo must be 'U' or 'L'");
  if (!is_notrans(trans) && trans != 'C' && trans != 'c') return arg_fail(2, "trans must be 'N' or 'C'");
  if (n < 0) return arg_fail(3, "n < 0");
  if (k < 0) return arg_fail(4, "k < 0");
  const int rows = is_notrans(trans) ? n : k;
  if (lda < (rows > 1 ? rows : 1)) return arg_fail(7, "lda too small");
  if (ldc < (n > 1 ? n : 1)) return arg_fail(10, "ldc < max(1,n)");
  int rc = ensure_init();
  if (rc) return rc;
  if (n == 0 || ((alpha == R(0) || k == 0) && beta == R(1))) return 0;  // BLAS quick return
  const bool tr = !is_notrans(trans);
  // 'C': C = alpha A^H A + beta C;  'N': C = alpha A A^H + beta C
  return zgemm_call<R>(tr ? 'C' : 'N', tr ? 'N' : 'C', n, n, k, alpha, R(0), (const R*)A, lda,
                       (const R*)A, lda, beta, R(0), (R*)C, ldc, is_upper(uplo) ? 1 : 2, 1,
                       nullptr, stream_of(s));
}

template <typename R>
int zgemm_api(char transa, char transb, int m, int n, int k, const R* alpha, const void* A,
              int lda, const void* B, int ldb, const R* beta, void* C, int ldc, dm_stream_t s) {
  if (!is_trans(transa) && !is_notrans(transa)) return arg_fail(1, "transa must be 'N','T','C'");
  if (!is_trans(transb) && !is_notrans(transb)) return arg_fail(2, "transb must be 'N','T','C'");
  if (m < 0) return arg_fail(3, "m < 0");
  if (n < 0) return arg_fail(4, "n < 0");
  if (k < 0) return arg_fail(5, "k < 0");
  if (!alpha) return arg_fail(6, "alpha is NULL");
  if (!beta) return arg_fail(11, "beta is NULL");
  const int ra = is_notrans(transa) ? m : k, rb = is_notrans(transb) ? k : n;
  if (lda < (ra > 1 ? ra : 1)) return arg_fail(8, "lda too small");
  if (ldb < (rb > 1 ? rb : 1)) return arg_fail(10, "ldb too small");
  if (ldc < (m > 1 ? m : 1)) return arg_fail(13, "ldc < max(1,m)");
  int rc = ensure_init();
  if (rc) return rc;
  return zgemm_call<R>(transa, transb, m, n, k, alpha[0], alpha[1], (const R*)A, lda,
                       (const R*)B, ldb, beta[0], beta[1], (R*)C, ldc, 0, 0, nullptr,
                       stream_of(s));
}

}  // namespace

extern "C" {
int dm_zpotrf(char uplo, int n, void* A, int lda, int* info_dev, dm_stream_t s) {
  return zpotrf_api<double>(uplo, n, A, lda, info_dev, s);
}
int dm_cpotrf(char uplo, int n, void* A, int lda, int* info_dev, dm_stream_t s) {
  return zpotrf_api<float>(uplo, n, A, lda, info_dev, s);
}
int dm_ztrsm(char side, char uplo, char transa, char diag, int m, int n, const double* alpha,
             const void* A, int lda, void* B, int ldb, dm_stream_t s) {
  return ztrsm_api<double>(side, uplo, transa, diag, m, n, alpha, A, lda, B, ldb, s);
}
int dm_ctrsm(char side, char uplo, char transa, char diag, int m, int n, const float* alpha,
             const void* A, int lda, void* B, int ldb, dm_stream_t s) {
  return ztrsm_api<float>(side, uplo, transa, diag, m, n, alpha, A, lda, B, ldb, s);
}
int dm_zherk(char uplo, char trans, int n, int k, double alpha, const void* A, int lda,
             double beta, void* C, int ldc, dm_stream_t s) {
  return zherk_api<double>(uplo, trans, n, k, alpha, A, lda, beta, C, ldc, s);
}
int dm_cherk(char uplo, char trans, int n, int k, float alpha, const void* A, int lda,
             float beta, void* C, int ldc, dm_stream_t s) {
  return zherk_api<float>(uplo, trans, n, k, alpha, A, lda, beta, C, ldc, s);
}
int dm_zgemm(char transa, char transb, int m, int n, int k, const double* alpha, const void* A,
             int lda, const void* B, int ldb, const double* beta, void* C, int ldc,
             dm_stream_t s) {
  return zgemm_api<double>(transa, transb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
}
int dm_cgemm(char transa, char transb, int m, int n, int k, const float* alpha, const void* A,
             int lda, const void* B, int ldb, const float* beta, void* C, int ldc,
             dm_stream_t s) {
  return zgemm_api<float>(transa, transb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
}
}  // extern "C"
