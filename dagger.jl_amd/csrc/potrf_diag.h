// The 64-wide panel of the tile POTRF as steps of a 256-thread workgroup on
// LDS-resident blocks, shared by the tile kernels (potrf.hip) and the batched
// level-synchronous factorization (batched.hip):
//   pb_load / pb_store   a 64 x 64 block of the matrix <-> LDS
//   pb_factor            Cholesky of a block in LDS
//   pb_recip             reciprocals of its diagonal, negated
//   pb_solve             U^-T X for 16 columns of X per wave
//
// Blocks are kept as the matrix's upper view: element (r, c) is A[r, c] for
// 'U' and A[c, r] for 'L' (so the factor is always U with U^T U = view).
// An LDS block is row-major with an odd stride of 65 elements: reads along a
// row and along a column of 8-byte elements both touch distinct banks.
#pragma once
#include "dm_internal.h"

namespace dm {

constexpr int PB = 64;        // panel width
constexpr int PBS = PB + 1;   // LDS row stride of a block
constexpr int PBE = PB * PBS; // LDS elements of a block

template <typename T> struct PMfma;
// Output layouts (lane l, accumulator item r; 16x16 block D[i][j], j = l%16):
//   f64 16x16x4: i = 4*r + l/16        f32 16x16x4: i = 4*(l/16) + r
template <> struct PMfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * r + lk; }
  static __device__ __forceinline__ v4 mac(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <> struct PMfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
  static __device__ __forceinline__ v4 mac(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// Lane l's value in every lane (l uniform): a scalar register, no LDS trip.
__device__ __forceinline__ float lane_bcast(float v, int l) {
  int i;
  __builtin_memcpy(&i, &v, 4);
  i = __builtin_amdgcn_readlane(i, l);
  __builtin_memcpy(&v, &i, 4);
  return v;
}
__device__ __forceinline__ double lane_bcast(double v, int l) {
  int i[2];
  __builtin_memcpy(i, &v, 8);
  i[0] = __builtin_amdgcn_readlane(i[0], l);
  i[1] = __builtin_amdgcn_readlane(i[1], l);
  __builtin_memcpy(&v, i, 8);
  return v;
}

// 1/sqrt(d) for a pivot d in the normal range (PivotBits): the hardware
// estimate y (relative error at most 2^-22) gets one third-order step,
// y + y e (1/2 + 3/8 e) with e = 1 - d y^2, whose error of order e^3 is below
// the rounding (FP32: one Newton step).  Straight-line and four dependent
// operations long, against a correctly rounded sqrt and a division of several
// tens each: it sits on the serial chain of every column.
__device__ __forceinline__ double inv_sqrt(double d) {
  const double y = __builtin_amdgcn_rsq(d);
  const double e = __builtin_fma(-d * y, y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ float inv_sqrt(float d) {
  const float y = __builtin_amdgcn_rsqf(d);
  const float e = __builtin_fmaf(-d * y, y, 1.0f);
  return __builtin_fmaf(0.5f * y, e, y);
}
// sqrt(d): d / sqrt(d) corrected once by its residual.
template <typename T>
__device__ __forceinline__ T sqrt_of(T d) {
  const T y = inv_sqrt(d), s = d * y;
  return s + T(0.5) * y * (d - s * s);
}
// The normal range of a pivot by its exponent bits as an unsigned number
// counted from lo: at most span exactly for 2^-960 <= d < 2^960 (FP32: 2^-96
// and 2^96); zero, negative, infinite and NaN pivots lie outside too.
template <typename T> struct PivotBits;
template <> struct PivotBits<double> {
  static constexpr unsigned lo = (1023u - 960u) << 20, span = (1920u << 20) - 1;
  static __device__ __forceinline__ unsigned of(double d) {
    unsigned long long b;
    __builtin_memcpy(&b, &d, 8);
    return (unsigned)(b >> 32) - lo;
  }
};
template <> struct PivotBits<float> {
  static constexpr unsigned lo = (127u - 96u) << 23, span = (192u << 23) - 1;
  static __device__ __forceinline__ unsigned of(float d) {
    unsigned b;
    __builtin_memcpy(&b, &d, 4);
    return b - lo;
  }
};

// This thread's wave, as a scalar the compiler knows to be uniform (branches
// on it are scalar branches instead of execution masks).
__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
}

// Address of element (r, c) of the upper view.
template <typename T, bool UPPER>
__device__ __forceinline__ T* pb_at(T* A, int lda, int r, int c) {
  return UPPER ? A + (size_t)c * lda + r : A + (size_t)r * lda + c;
}

// This thread's 16 elements of a 64 x 64 block: element q is (r, c) with the
// contiguous axis of the matrix along the lanes.
template <bool UPPER>
__device__ __forceinline__ void pb_coord(int q, int& r, int& c) {
  const int a = threadIdx.x & 63, b = (threadIdx.x >> 6) + 4 * q;
  r = UPPER ? a : b;
  c = UPPER ? b : a;
}

// v = rows r0.. and columns c0.. of the view, zero from column ncol >= 1 on.
// The loads carry no condition (past the end they repeat the last column):
// with a branch around each the compiler waits between them, and the step of
// the 1024-row FP32 tile took 21.4 us instead of 20.2.
template <typename T, bool UPPER>
__device__ __forceinline__ void pb_load(const T* A, int lda, int r0, int c0, int ncol, T (&v)[16]) {
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    int r, c;
    pb_coord<UPPER>(q, r, c);
    v[q] = *gptr(pb_at<T, UPPER>(const_cast<T*>(A), lda, r0 + r, c0 + min(c, ncol - 1)));
  }
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    int r, c;
    pb_coord<UPPER>(q, r, c);
    if (c >= ncol) v[q] = T(0);
  }
}
// The upper triangle of the kb x kb diagonal block at j0; the rest of the
// 64 x 64 block is the identity's (so a narrow block factors like a full one).
// Loaded whole, for the same reason.
template <typename T, bool UPPER>
__device__ __forceinline__ void pb_load_diag(const T* A, int lda, int j0, int kb, T (&v)[16]) {
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    int r, c;
    pb_coord<UPPER>(q, r, c);
    v[q] = *gptr(pb_at<T, UPPER>(const_cast<T*>(A), lda, j0 + min(r, kb - 1), j0 + min(c, kb - 1)));
  }
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    int r, c;
    pb_coord<UPPER>(q, r, c);
    if (r > c || c >= kb) v[q] = r == c ? T(1) : T(0);
  }
}
template <typename T, bool UPPER>
__device__ __forceinline__ void pb_put(T* M, const T (&v)[16]) {
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    int r, c;
    pb_coord<UPPER>(q, r, c);
    M[r * PBS + c] = v[q];
  }
}
template <typename T, bool UPPER>
__device__ __forceinline__ void pb_store(T* A, int lda, int r0, int c0, int ncol, const T* M) {
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    int r, c;
    pb_coord<UPPER>(q, r, c);
    if (c < ncol) *gptr(pb_at<T, UPPER>(A, lda, r0 + r, c0 + c)) = M[r * PBS + c];
  }
}
// Upper triangle of the first nrow rows of a factored kb x kb block.
template <typename T, bool UPPER>
__device__ __forceinline__ void pb_store_diag(T* A, int lda, int j0, int kb, int nrow, const T* M) {
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    int r, c;
    pb_coord<UPPER>(q, r, c);
    if (r <= c && c < kb && r < nrow)
      *gptr(pb_at<T, UPPER>(A, lda, j0 + r, j0 + c)) = M[r * PBS + c];
  }
}

// Cholesky of the 64 x 64 block in M (upper triangle; columns from kb on are
// the identity's), in place.  Returns 0, or the failed column + 1 (its row
// and the later ones are then not final).  fail: one LDS int.
//
// Bound by the serial chain of 64 pivots.  Eight rows at a time (pb_chain):
// wave 0 holds them with one column per lane, so a step is a readlane of the
// pivot, the reciprocal square root, a scaling and at most seven rank-1
// updates whose multipliers are readlanes too -- no LDS trip and no branch
// inside the chain (pivots outside the normal range are noticed at the end of
// the eight rows, which are then done again in the exact form).  The rows
// below get the eight rows' update on the matrix cores: wave w keeps the
// blocks of the 16 columns from 16 w on in its accumulators all the way down
// (acc[q]: block row blk + q) and hands the next eight rows to wave 0 through
// M; the blocks below those are updated while wave 0 is already at its next
// eight rows.
// Measured per block (cycles): the chain 1280 of 2500 per eight rows, the
// hand-over the rest; one column per lane and all 64 steps from LDS rows, as
// this step was done before, took 75000 for the block, this 19000.
template <typename T>
__device__ __forceinline__ int pb_chain(T* M, int base, T& diag) {
  const int lane = threadIdx.x & 63;
  T v[8];
  T* rows = M + base * PBS + lane;
#pragma unroll
  for (int r = 0; r < 8; ++r) v[r] = rows[r * PBS];
  unsigned far = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const T d = lane_bcast(v[j], base + j);
    const unsigned e = PivotBits<T>::of(d);
    far = e > far ? e : far;
    if (lane == base + j) diag = d;
    const T u = v[j] = v[j] * inv_sqrt(d);
#pragma unroll
    for (int i = j + 1; i < 8; ++i) v[i] -= lane_bcast(u, base + i) * u;
  }
  if (__builtin_expect(far <= PivotBits<T>::span, 1)) {  // uniform
#pragma unroll
    for (int r = 0; r < 8; ++r) rows[r * PBS] = v[r];
    return 0;
  }
#pragma unroll 1
  for (int j = 0; j < 8; ++j) {
    const T w = rows[j * PBS], d = lane_bcast(w, base + j);
    if (!(d > T(0))) return base + j + 1;
    // tiny, huge or infinite: the exact forms
    const T sd = sqrt(d), u = w * (T(1) / sd);
    rows[j * PBS] = lane == base + j ? sd : u;
    if (lane == base + j) diag = T(0);  // already final
#pragma unroll 1
    for (int i = j + 1; i < 8; ++i) rows[i * PBS] -= lane_bcast(u, base + i) * u;
  }
  return 0;
}

template <typename T>
__device__ __forceinline__ int pb_factor(T* M, int kb, int* fail) {
  typedef typename PMfma<T>::v4 v4;
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int lr = lane & 15, lk = lane >> 4;
  v4 acc[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      acc[q][r] = M[(16 * q + PMfma<T>::row(lk, r)) * PBS + 16 * wave + lr];
  T diag = T(0);  // lane c: pivot c
  int bad = 0;
#pragma unroll 1
  for (int blk = 0; 16 * blk < kb; ++blk) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int base = 16 * blk + 8 * half;
      if (wave == 0) {
        const int f = pb_chain<T>(M, base, diag);
        if (lane == 0) *fail = f;
      }
      __syncthreads();
      const int q0 = half;  // block row of the next eight rows
      const T* row = M + (base + lk) * PBS + lr;
      auto update = [&](int q) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
          acc[q] = PMfma<T>::mac(-row[4 * s * PBS + 16 * (blk + q)], row[4 * s * PBS + 16 * wave],
                                 acc[q]);
      };
      if (wave >= blk + q0) {
        update(q0);
        T* out = M + (base + 8) * PBS + 16 * wave + lr;
        // half 0: rows 8 .. 15 of the block, half 1: rows 0 .. 7 of the next
        if (sizeof(T) == 8) {
          out[lk * PBS] = acc[q0][half ? 0 : 2];
          out[(4 + lk) * PBS] = acc[q0][half ? 1 : 3];
        } else if ((lk >> 1) == 1 - half) {
#pragma unroll
          for (int r = 0; r < 4; ++r) out[(4 * (lk & 1) + r) * PBS] = acc[q0][r];
        }
      }
      bad = *fail;
      __syncthreads();
      if (bad || base + 8 >= kb) break;
#pragma unroll
      for (int q = q0 + 1; q < 4; ++q)
        if (wave >= blk + q) update(q);
    }
    if (bad) break;
#pragma unroll
    for (int q = 0; q < 3; ++q) acc[q] = acc[q + 1];
  }
  if (wave == 0 && diag > T(0)) M[lane * PBS + lane] = sqrt_of(diag);
  __syncthreads();
  return bad;
}

// Swaps of 16-lane groups between two registers (emulated lane by lane on the
// host): the odd groups of a with the even ones of b; groups 2 and 3 of a with
// groups 0 and 1 of b.
__device__ __forceinline__ void swap_odd_groups(float& a, float& b) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a),
                                                  __builtin_bit_cast(unsigned, b), false, false);
  const unsigned ra = r[0], rb = r[1];
  a = __builtin_bit_cast(float, ra);
  b = __builtin_bit_cast(float, rb);
#else
  const int l = threadIdx.x & 63;
  const bool odd = l & 16;
  const float x = __shfl(a, l ^ 16, 64), y = __shfl(b, l ^ 16, 64);
  if (odd) a = y;
  else b = x;
#endif
}
__device__ __forceinline__ void swap_halves(float& a, float& b) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a),
                                                  __builtin_bit_cast(unsigned, b), false, false);
  const unsigned ra = r[0], rb = r[1];
  a = __builtin_bit_cast(float, ra);
  b = __builtin_bit_cast(float, rb);
#else
  const int l = threadIdx.x & 63;
  const bool upper = l & 32;
  const float x = __shfl(a, l ^ 32, 64), y = __shfl(b, l ^ 32, 64);
  if (upper) a = y;
  else b = x;
#endif
}
template <void (*SWAP)(float&, float&)>
__device__ __forceinline__ void swap_words(double& a, double& b) {
  float x[2], y[2];
  __builtin_memcpy(x, &a, 8);
  __builtin_memcpy(y, &b, 8);
  SWAP(x[0], y[0]);
  SWAP(x[1], y[1]);
  __builtin_memcpy(&a, x, 8);
  __builtin_memcpy(&b, y, 8);
}

// Four consecutive rows of a block in the accumulator layout, block row s of
// four: into v, row by row, where a lane can compute with them, and from v to
// the layout of a product's operand, row k in lane group k.  FP64: the rows are
// item s of the four groups, so every lane gets all of them and keeps one.
// FP32: they are the four items of group s; the other groups compute with rows of
// their own to no end, and a transposition hands out group s's.
__device__ __forceinline__ void four_rows(const PMfma<double>::v4& x, int s, double (&v)[4]) {
  v[0] = v[2] = x[s];
  swap_words<swap_halves>(v[0], v[2]);
  v[1] = v[0];
  v[3] = v[2];
  swap_words<swap_odd_groups>(v[0], v[1]);
  swap_words<swap_odd_groups>(v[2], v[3]);
}
__device__ __forceinline__ void four_rows(const PMfma<float>::v4& x, int, float (&v)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = x[q];
}
__device__ __forceinline__ double row_by_group(const double (&v)[4], int) {
  const int k = (threadIdx.x >> 4) & 3;
  const double a = k & 1 ? v[1] : v[0], b = k & 1 ? v[3] : v[2];
  return k & 2 ? b : a;
}
__device__ __forceinline__ float row_by_group(const float (&v)[4], int s) {
  float a = v[0], b = v[1], c = v[2], d = v[3];
  swap_odd_groups(a, b);
  swap_odd_groups(c, d);
  if (s & 1) {
    swap_halves(b, d);
    return s & 2 ? d : b;
  }
  swap_halves(a, c);
  return s & 2 ? c : a;
}

// The negative reciprocals of the diagonal of the factored block in M, for
// pb_solve (a barrier follows).
template <typename T>
__device__ __forceinline__ void pb_recip(const T* M, T* nrec) {
  if (threadIdx.x < PB) nrec[threadIdx.x] = T(-1) / M[threadIdx.x * PBS + threadIdx.x];
}

// Columns c0 .. c0+15 of X := U^-T X for the factored block M (with pb_recip's
// nrec), by one wave: substitution by four rows at a time on the vector unit and
// products of depth 4 on the matrix cores for the rows below, in sums of the
// opposite sign (U^T X - B).
//
// Substitution rather than products with inverted diagonal blocks, whose error
// grows with those blocks' condition: neighbouring rows of a covariance matrix
// (256 of them) made the factor's error 2e-15 |A| at a nugget of 1e-12 and a pivot
// negative at 1e-13, where substitution keeps to 2e-16 and succeeds.  It costs
// 1.0 us (FP32: 0.5) of the tile POTRF's 20 us step.
//
// Bound by the chain of the 16 steps (one product, seven operations, the trips
// between the layouts).  The order below is the one that the wave issues in:
// operands a step ahead, and the products that the next step does not need in
// the gaps of the chain, where they would otherwise hold it up.
template <typename T>
__device__ __forceinline__ void pb_solve(const T* M, const T* nrec, T* X, int c0) {
  typedef typename PMfma<T>::v4 v4;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  v4 x[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) x[b][r] = -X[(16 * b + PMfma<T>::row(lk, r)) * PBS + c0 + lr];
  // of step t: U_oo of its four rows, their reciprocals, the products' other
  // operand
  T u[2][4][4], d[2][4], a[3][4], y = T(0);
  auto read = [&](int t) {
    const int o = 4 * t;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
#pragma unroll
      for (int q = p + 1; q < 4; ++q) u[t & 1][p][q] = M[(o + p) * PBS + o + q];
      d[t & 1][p] = nrec[o + p];
      if (16 * p + 15 >= o) a[t % 3][p] = M[(o + lk) * PBS + 16 * p + lr];
    }
  };
  read(0);
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int b = t / 4, s = t % 4, o = 4 * t, e = t & 1;
    // the previous rows' product with block i
    auto product = [&](int i) {
      if (t > 0 && i < 4) x[i] = PMfma<T>::mac(a[(t + 2) % 3][i], y, x[i]);
    };
    product(b);
    T v[4];
    four_rows(x[b], s, v);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      __builtin_amdgcn_sched_barrier(0);
      product(b + 1 + q);
      if (q == 0 && t < 15) read(t + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < q; ++p) v[q] += u[e][p][q] * v[p];
      v[q] *= d[e][q];
    }
    y = row_by_group(v, s);
    X[(o + lk) * PBS + c0 + lr] = y;
  }
}

}  // namespace dm
