// The 64-wide panel of the tile POTRF as steps of a 256-thread workgroup on
// LDS-resident blocks, shared by the tile kernels (potrf.hip) and the batched
// level-synchronous factorization (batched.hip):
//   pb_load / pb_store   a 64 x 64 block of the matrix <-> LDS
//   pb_factor            Cholesky of a block in LDS
//   pb_inv16             inverses of its four 16 x 16 diagonal blocks
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
constexpr int PIS = 17;       // LDS row stride of an inverted 16 x 16 block
constexpr int PIE = 4 * 16 * PIS + 64;  // LDS elements of pb_inv16's result

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

// W_g = (U_gg)^-T (lower triangular, 16 x 16) of the four diagonal blocks of
// the factored block in M: W_g(r, c) at Wi[g * 16 * PIS + r * PIS + c].  Wave
// g inverts block g: its two 8 x 8 diagonal blocks by substitution (one
// column per lane), then W21 = -V1 (L21 V0).  The caller's barrier follows.
template <typename T>
__device__ __forceinline__ void pb_inv16(const T* M, T* Wi) {
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const T* Mg = M + (g * 16) * PBS + g * 16;  // U_gg(p, r) = Mg[p * PBS + r] = L(r, p)
  T* W = Wi + g * 16 * PIS;
  T* dinv = Wi + 4 * 16 * PIS + g * 16;
  if (lane < 16) dinv[lane] = T(1) / Mg[lane * PBS + lane];
  for (int e = lane; e < 256; e += 64) W[(e >> 4) * PIS + (e & 15)] = T(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int o = (lane >> 3) * 8, c = lane & 7;
  if (lane < 16) {
    T x[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) x[r] = r == c ? T(1) : T(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      x[r] *= dinv[o + r];
#pragma unroll
      for (int i = r + 1; i < 8; ++i) x[i] -= Mg[(o + r) * PBS + o + i] * x[r];
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) W[(o + r) * PIS + o + c] = x[r];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  // Z = L21 V0 in W's (otherwise zero) upper right block
  const int r8 = lane >> 3;
  T z = T(0);
#pragma unroll
  for (int p = 0; p < 8; ++p) z += Mg[p * PBS + 8 + r8] * W[p * PIS + c];
  W[r8 * PIS + 8 + c] = z;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  T y = T(0);
#pragma unroll
  for (int p = 0; p < 8; ++p) y -= W[(8 + r8) * PIS + 8 + p] * W[p * PIS + 8 + c];
  __builtin_amdgcn_wave_barrier();  // every lane has read the block
  W[(8 + r8) * PIS + c] = y;
  W[r8 * PIS + 8 + c] = T(0);
}

// Columns c0 .. c0+15 of X := U^-T X for the factored block M (with pb_inv16's
// Wi), by one wave on matrix cores: block row b needs sum_{i<b} U_ib^T X_i and
// then a product with W_b.  An accumulator of the matrix core holds rows
// row(lk, r) of a column in item r, and the next product's operand of k-step
// s is rows row(lk, s): the same lane and item, so the chain of 40 products
// stays in registers.
template <typename T>
__device__ __forceinline__ void pb_solve(const T* M, const T* Wi, T* X, int c0) {
  typedef typename PMfma<T>::v4 v4;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  v4 x[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) x[b][r] = X[(16 * b + PMfma<T>::row(lk, r)) * PBS + c0 + lr];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
#pragma unroll
    for (int i = 0; i < b; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        x[b] = PMfma<T>::mac(-M[(16 * i + PMfma<T>::row(lk, s)) * PBS + 16 * b + lr], x[i][s], x[b]);
    v4 y = v4{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s)
      y = PMfma<T>::mac(Wi[b * 16 * PIS + lr * PIS + PMfma<T>::row(lk, s)], x[b][s], y);
    x[b] = y;
#pragma unroll
    for (int r = 0; r < 4; ++r) X[(16 * b + PMfma<T>::row(lk, r)) * PBS + c0 + lr] = y[r];
  }
}

}  // namespace dm
