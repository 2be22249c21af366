// LU without pivoting of the dense diagonal blocks of the Newton matrix, and
// the CSR product used to refine its solves.
//
// The Newton driver factors its block-banded matrix block by block (block
// Gaussian elimination in j- or i-line blocks); the diagonal block of each
// step is dense (B = 5 im or 5 jm unknowns, ~1000-2000) and factored here in
// place, A = L U with L unit lower, row-major with leading dimension ld:
//
//   for each 32-column panel k:
//     k_lu_panel_np   the 32 x 32 diagonal tile factored in LDS, then the
//                     row panel to its right (L^-1 A, a column per thread)
//                     and the column panel below it (A U^-1, a row per
//                     thread);
//     k_gemm_f64_sub  the trailing matrix minus the product of the two
//                     panels, 64 x 64 output tiles on the FP64 matrix cores
//                     (v_mfma_f64_16x16x4f64), panels staged in LDS.
//
// No pivoting: downwards, as the flow runs, the relaxed (or pure) Newton
// Jacobians of these flows factor stably without it (element growth below 5 on
// the oracle's Jacobians, solves as accurate as the pivoted ones).  The
// two-ended elimination's upward half runs against the flow and loses some
// digits on a weakly relaxed boundary layer.  A pivot below tiny * its tile's
// largest entry is reported, which does not show growth across the blocks: the
// Newton driver's solves are corrected once with the CSR residual, and where
// the residual then says that entries grew, the driver factors again downwards
// only, then with pivoting.
#pragma once
#include <hip/hip_runtime.h>

#include "scheme.h"

namespace bca {

constexpr int LU_NB = 32;

typedef double f64x4 __attribute__((ext_vector_type(4)));

// One panel step at the diagonal tile A (ld), nb = min(LU_NB, rows left),
// m rows/columns past the tile; one wave per workgroup, so the barriers of
// the tile's 32 elimination steps cost next to nothing.  Every workgroup
// factors the tile in LDS (nb^3/3 flops, cheaper than a launch); workgroup 0
// reports a pivot below tiny times the tile's largest |entry| in *bad and
// stores the factored tile; workgroups 1..nrb solve row-panel columns c
// (A(0:nb, nb + c) = L^-1 A(0:nb, nb + c), unit L), the next nrb
// column-panel rows r (A(nb + r, 0:nb) = A(nb + r, 0:nb) U^-1), one per
// thread.
constexpr int LU_THREADS = 64;
__global__ void __launch_bounds__(LU_THREADS) k_lu_panel_np(double* __restrict__ A, long ld, int nb, int m, int nrb,
                                                            double tiny, int* __restrict__ bad,
                                                            double* __restrict__ work) {
  __shared__ double T[LU_NB][LU_NB + 1];
  __shared__ double X[LU_THREADS][LU_NB + 1];
  const int tid = threadIdx.x;
  double amax = 0.0;
  for (int x = tid; x < LU_NB * LU_NB; x += LU_THREADS) {
    const int r = x / LU_NB, c = x % LU_NB;
    const double v = (r < nb && c < nb) ? A[r * ld + c] : (r == c ? 1.0 : 0.0);
    T[r][c] = v;
    amax = fmax(amax, (r < nb && c < nb) ? fabs(v) : 0.0);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) amax = fmax(amax, __shfl_xor(amax, off));
  const double thr = tiny * amax;
  __syncthreads();
  for (int j = 0; j < nb; ++j) {
    const double p = T[j][j];
    if (blockIdx.x == 0 && tid == 0 && !(fabs(p) > thr)) *bad = 1;
    const double pinv = 1.0 / p;
    if (tid > j && tid < nb) T[tid][j] *= pinv;
    __syncthreads();
    const int q = nb - j - 1;
    for (int x = tid; x < q * q; x += LU_THREADS) {
      const int r = j + 1 + x / q, c = j + 1 + x % q;
      T[r][c] -= T[r][j] * T[j][c];
    }
    __syncthreads();
  }
  if (blockIdx.x == 0) {
    // the other workgroups may still be loading the tile from A: unless it
    // is alone (no panels) workgroup 0 leaves the factored tile in `work`,
    // and the trailing update's first workgroup puts it in place
    double* dst = m == 0 ? A : work;
    const long ldd = m == 0 ? ld : LU_NB;
    for (int x = tid; x < nb * nb; x += LU_THREADS) dst[(x / nb) * ldd + x % nb] = T[x / nb][x % nb];
    return;
  }
  // each thread solves one column (row panel) or row (column panel) of
  // length nb, kept in LDS
  double* x = X[tid];
  if ((int)blockIdx.x <= nrb) {
    const int c = (blockIdx.x - 1) * LU_THREADS + tid;
    if (c >= m) return;
    double* col = A + nb + c;
    for (int r = 0; r < nb; ++r) x[r] = col[r * ld];
    for (int r = 1; r < nb; ++r) {
      double sum = x[r];
      for (int i = 0; i < r; ++i) sum -= T[r][i] * x[i];
      x[r] = sum;
    }
    for (int r = 0; r < nb; ++r) col[r * ld] = x[r];
  } else {
    const int r = (blockIdx.x - 1 - nrb) * LU_THREADS + tid;
    if (r >= m) return;
    double* row = A + (long)(nb + r) * ld;
    for (int c = 0; c < nb; ++c) x[c] = row[c];
    for (int c = 0; c < nb; ++c) {
      double sum = x[c];
      for (int i = 0; i < c; ++i) sum -= x[i] * T[i][c];
      x[c] = sum / T[c][c];
    }
    for (int c = 0; c < nb; ++c) row[c] = x[c];
  }
}

// C (M x N, ldc) -= A (M x K, lda) B (K x N, ldb), row-major, K <= LU_NB.
// Workgroup of 4 waves per 64 x 64 tile of C, each wave a 32 x 32 quarter
// as 2 x 2 MFMA tiles.  v_mfma_f64_16x16x4f64: lane l holds A(l % 16, l / 16)
// and B(l / 16, l % 16) of the 16 x 4 / 4 x 16 operands and receives
// D(l / 16 + 4 t, l % 16) in its t-th result, t = 0..3 (checked against
// torch's FP64 product by the GPU tests).  Operands past M, N, K read as 0.
// With tile != nullptr, workgroup (0, 0) also copies the factored nb x nb
// tile from `work` (ld LU_NB) to `tile` (ldt): the panel step's write-back.
__global__ void __launch_bounds__(256) k_gemm_f64_sub(int M, int N, int K, const double* __restrict__ A, long lda,
                                                      const double* __restrict__ B, long ldb,
                                                      double* __restrict__ C, long ldc,
                                                      double* __restrict__ tile = nullptr, long ldt = 0,
                                                      const double* __restrict__ work = nullptr, int nb = 0) {
  __shared__ double As[64][LU_NB + 1];
  __shared__ double Bs[LU_NB][64 + 1];
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  if (tile && blockIdx.x == 0 && blockIdx.y == 0)
    for (int x = tid; x < nb * nb; x += 256) tile[(x / nb) * ldt + x % nb] = work[(x / nb) * LU_NB + x % nb];
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  for (int x = tid; x < 64 * LU_NB; x += 256) {
    const int r = x / LU_NB, k = x % LU_NB;
    As[r][k] = (m0 + r < M && k < K) ? A[(long)(m0 + r) * lda + k] : 0.0;
    const int kb = x / 64, c = x % 64;
    Bs[kb][c] = (kb < K && n0 + c < N) ? B[(long)kb * ldb + n0 + c] : 0.0;
  }
  __syncthreads();
  const int wm = (wave / 2) * 32, wn = (wave % 2) * 32;
  const int lr = lane % 16, lk = lane / 16;
  f64x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
  const int kend = (K + 3) / 4 * 4;
  for (int k0 = 0; k0 < kend; k0 += 4) {
    double av[2], bv[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) av[a] = As[wm + 16 * a + lr][k0 + lk];
#pragma unroll
    for (int b = 0; b < 2; ++b) bv[b] = Bs[k0 + lk][wn + 16 * b + lr];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a], bv[b], acc[a][b], 0, 0, 0);
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = m0 + wm + 16 * a + lk + 4 * t, c = n0 + wn + 16 * b + lr;
        if (r < M && c < N) C[(long)r * ldc + c] -= acc[a][b][t];
      }
}

// ------------------------------------------------------------------ inverse
// Inverse without pivoting of a dense n x n block by Gauss-Jordan steps on
// GJ_NB-column panels, each step one launch from Ain to Aout (every entry
// written, so the caller alternates two buffers).  For the panel kk =
// k0..k0+nb-1 with pivot tile P = A(kk, kk):
//
//   Aout(kk, kk) = P^-1                      Aout(kk, j) = P^-1 A(kk, j)
//   Aout(i, kk)  = -A(i, kk) P^-1            Aout(i, j)  = A(i, j) - A(i, kk) P^-1 A(kk, j)
//
// for i, j outside kk.  Every entry is one product out = A' - T U of a
// GJ_T x GJ_T output tile, with T = A(i, kk) P^-1 (rows of kk: T = -P^-1)
// and U = A(kk, j) (columns of kk: U = the identity), A' = A off the panel
// rows and columns and 0 on them.  Panels are processed in turn, so the steps
// are a serial chain and what bounds a block of 500-1000 unknowns is the
// latency of one step, first of all the inversion of P.  That inversion is
// therefore taken out of the step: nothing but the next step needs the next
// pivot tile, so one extra workgroup of each launch forms that tile's update
// from the same inputs, inverts it and stores the inverse in the tile's
// place, beside the workgroups of the update; the step after it finds P^-1
// where P would be (the first panel's comes from a launch of its own).  A step
// on 640 unknowns takes 11 us against 37 with P inverted in every workgroup of
// the step, column by column through lane shuffles, and 128 x 128 tiles; the
// inverse 0.22 against 0.73 ms (480: 0.18 / 0.57, 1920: 1.33 / 2.29 ms).
constexpr int GJ_NB = 32;
constexpr int GJ_T = 64;
constexpr int GJ_RANGE = 300;  // binary exponents up to which a tile is inverted as it is

// Doubles of a row-major tile through a buffer descriptor of its rows: an
// index of NOWHERE is out of the descriptor's range, so such a load gives 0
// and such a store is dropped, without a branch around either (a branch per
// guarded load serialises the loads of a tile).
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
constexpr unsigned NOWHERE = ~0u;
template <bool WIDE = false>
struct TileBuf {
  __amdgpu_buffer_rsrc_t r;
  // rows rows of pitch ld from p, n columns (at least one row)
  __device__ TileBuf(const double* p, int rows, long ld, int n)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), 0, (int)(unsigned)(((rows - 1) * ld + n) * 8L),
                                            0x00027000)) {}
  __device__ double load(unsigned off) const {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  }
  __device__ void store(unsigned off, double v) const {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 0);
  }
  __device__ double load(bool in, int row, long ld, int col) const {
    return load(in ? (unsigned)(row * (int)ld + col) * 8u : NOWHERE);
  }
  __device__ void store(bool in, int row, long ld, int col, double v) const {
    store(in ? (unsigned)(row * (int)ld + col) * 8u : NOWHERE, v);
  }
};

// The same by 64-bit addresses, for rows too far apart for the 32-bit offsets of a
// descriptor.
template <>
struct TileBuf<true> {
  double* p;
  __device__ TileBuf(const double* q, int, long, int) : p(const_cast<double*>(q)) {}
  __device__ double load(bool in, int row, long ld, int col) const { return in ? p[row * ld + col] : 0.0; }
  __device__ void store(bool in, int row, long ld, int col, double v) const {
    if (in) p[row * ld + col] = v;
  }
};

__device__ inline double rcp64(double x) {
  // v_rcp_f64 and two Newton steps: the reciprocal to within an ulp
  double r = __builtin_amdgcn_rcp(x);
  r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}
__device__ inline double readlane_f64(double x, int l) {
  const long long b = __double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Inverse of a 2 x 2 block; amin / rmax: its two pivots |a| and |det / a| go
// into the smallest |a| and the largest 1 / |det / a| seen.
__device__ inline void inv2(double (&m)[2][2], double& amin, double& rmax) {
  const double a = m[0][0], b = m[0][1], c = m[1][0], d = m[1][1];
  const double r = rcp64(__builtin_fma(a, d, -(b * c)));
  amin = fmin(amin, fabs(a));
  rmax = fmax(rmax, fabs(a * r));
  m[0][0] = d * r;
  m[0][1] = -b * r;
  m[1][0] = -c * r;
  m[1][1] = a * r;
}
__device__ inline void mul2(const double (&x)[2][2], const double (&y)[2][2], double (&z)[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) z[i][j] = __builtin_fma(x[i][1], y[1][j], x[i][0] * y[0][j]);
}

// In-place inverse of a 32 x 32 tile held by one wave in the accumulator
// layout of v_mfma_f64_16x16x4f64 -- X[a][b][t] of lane l is S(16 a + l / 16 +
// 4 t, 16 b + l % 16) -- by Gauss-Jordan steps on 4 pivots at a time.  In that
// layout the register X[a][b][t] holds the rows 16 a + 4 t .. + 3, one per 16
// lanes, which is the layout of a B operand (4 x 16), and the same register of
// the transpose is the A operand (16 x 4) of the columns: with Y = S^T kept
// beside X the rank-4 update is S -= C W with C from Y and W = Q R (R the
// four pivot rows, Q the inverse of the 4 x 4 pivot block, by its 2 x 2
// blocks), and Y -= W^T C^T swaps the operands; no value crosses lanes but the
// 16 entries of the pivot block.  A chain of 8 such steps, against 32 of a
// column-by-column elimination whose pivot rows go through lane shuffles.
// Returns the smallest |pivot|, 0 where the inverse is not finite.
__device__ inline double gj_inv32(f64x4 (&X)[2][2], f64x4 (&Y)[2][2]) {
  const int lane = threadIdx.x % 64, lk = lane / 16;
  const bool dg = lane % 4 == lk;
  double amin = 1.7976931348623157e308, rmax = 0.0;
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    constexpr f64x4 zero4 = {0.0, 0.0, 0.0, 0.0};
    const int ga = g / 4, gt = g % 4;
    // the pivot block in 2 x 2 blocks (uniform over the wave)
    double q[2][2][2][2];
    const double piv = X[ga][ga][gt];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) q[i / 2][j / 2][i % 2][j % 2] = readlane_f64(piv, 16 * i + 4 * gt + j);
    // this lane's column lies in the pivot columns of block column ga
    const bool pc = lane % 16 / 4 == gt;
    double br[2], ac[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      br[b] = X[ga][b][gt];
      ac[b] = -Y[ga][b][gt];
    }
    // pivot columns of R: the identity; pivot rows of -C: the identity; both
    // panels of the old tile: zero
    br[ga] = pc ? (dg ? 1.0 : 0.0) : br[ga];
    ac[ga] = pc ? (dg ? 1.0 : 0.0) : ac[ga];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      X[ga][a][gt] = 0.0;
      Y[ga][a][gt] = 0.0;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (a == ga && t == gt) continue;
        X[a][ga][t] = pc ? 0.0 : X[a][ga][t];
        Y[a][ga][t] = pc ? 0.0 : Y[a][ga][t];
      }
    }
    // Q = inverse of [A B; C D]: A^-1, S = D - C A^-1 B, S^-1, then the blocks
    double ab[2][2], ca[2][2], cab[2][2], z[2][2];
    inv2(q[0][0], amin, rmax);
    mul2(q[0][0], q[0][1], ab);
    mul2(q[1][0], q[0][0], ca);
    mul2(q[1][0], ab, cab);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) q[1][1][i][j] -= cab[i][j];
    inv2(q[1][1], amin, rmax);
    mul2(ab, q[1][1], q[0][1]);
    mul2(q[1][1], ca, q[1][0]);
    mul2(q[0][1], ca, z);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        q[0][0][i][j] += z[i][j];
        q[0][1][i][j] = -q[0][1][i][j];
        q[1][0][i][j] = -q[1][0][i][j];
      }
    // Q as an A operand: row l % 16 (rows past 3 zero), k = l / 16
    double qr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double lo = lk % 2 ? q[i / 2][0][i % 2][1] : q[i / 2][0][i % 2][0];
      const double hi = lk % 2 ? q[i / 2][1][i % 2][1] : q[i / 2][1][i % 2][0];
      qr[i] = lk / 2 ? hi : lo;
    }
    const double q01 = lane % 2 ? qr[1] : qr[0], q23 = lane % 2 ? qr[3] : qr[2];
    const double qa = lane % 16 < 4 ? (lane % 4 / 2 ? q23 : q01) : 0.0;
    double w[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) w[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(qa, br[b], zero4, 0, 0, 0)[0];
    // the next pivot block's tile first
    const int na = (g + 1) / 4 % 2;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int a = (s / 2 + na) % 2, b = (s % 2 + na) % 2;
      X[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(ac[a], w[b], X[a][b], 0, 0, 0);
      Y[b][a] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[b], ac[a], Y[b][a], 0, 0, 0);
    }
  }
  double nan = 0.0;
#pragma unroll
  for (int x = 0; x < 16; ++x) nan = __builtin_fma(X[x / 8][x / 4 % 2][x % 4], 0.0, nan);
  return __ballot(nan != nan) ? 0.0 : fmin(amin, 1.0 / rmax);
}

// LDS of one workgroup: P^-1, A(i, kk) (then T) and U.  The pitches keep the
// 32 lanes of a b64 access on 32 different bank pairs: an A operand reads
// (row l % 16, k l / 16), so its pitch is 2 mod 32 doubles, a B operand (k,
// column), pitch 16 mod 32.
struct GjSmem {
  double P[GJ_NB][GJ_NB + 16];
  double AT[GJ_T][GJ_NB + 2];
  double U[GJ_NB][GJ_T + 16];
};

// The inverse of the nb x nb tile S(r, c) = get(in, r, c) (a diagonal where in is
// false), read by one wave in both layouts, stored through put(in, r, c, value); a pivot
// below tiny times the tile's largest |entry| sets *bad.
template <class Get, class Put>
__device__ inline void gj_invert_tile(int nb, double tiny, int* bad, const Get& get, const Put& put) {
  const int lane = threadIdx.x % 64, lr = lane % 16, lk = lane / 16;
  f64x4 X[2][2], Y[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 16 * a + lk + 4 * t, c = 16 * b + lr;
        const bool in = r < nb && c < nb;
        X[a][b][t] = get(in, r, c);
        Y[a][b][t] = get(in, c, r);
      }
  // the diagonal past nb: the power of two above the first pivot, |S(0, 0)|, so
  // that the padded pivots are never the smallest and no rounding depends on them
  int e = __builtin_amdgcn_readfirstlane(__builtin_amdgcn_frexp_exp(readlane_f64(X[0][0][0], 0)));
  // the 2 x 2 determinants are of the order of its square: a tile where that
  // would leave the range of a double is inverted scaled (exactly) by it
  const int shift = e > GJ_RANGE || e < -GJ_RANGE ? e : 0;
  if (__builtin_expect(shift != 0, 0)) {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      X[x / 8][x / 4 % 2][x % 4] = ldexp(X[x / 8][x / 4 % 2][x % 4], -shift);
      Y[x / 8][x / 4 % 2][x % 4] = ldexp(Y[x / 8][x / 4 % 2][x % 4], -shift);
    }
    e = 0;
  }
  const double pad = ldexp(1.0, e);
  double amax = 0.0;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 16 * a + lk + 4 * t, c = 16 * b + lr;
        const bool in = r < nb && c < nb;
        amax = fmax(amax, in ? fabs(X[a][b][t]) : 0.0);
        X[a][b][t] = in ? X[a][b][t] : (r == c ? pad : 0.0);
        Y[a][b][t] = in ? Y[a][b][t] : (r == c ? pad : 0.0);
      }
  const double pmin = gj_inv32(X, Y);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) amax = fmax(amax, __shfl_xor(amax, off));
  if (lane == 0 && !(pmin > tiny * amax)) *bad = 1;
  if (__builtin_expect(shift != 0, 0))
#pragma unroll
    for (int x = 0; x < 16; ++x) X[x / 8][x / 4 % 2][x % 4] = ldexp(X[x / 8][x / 4 % 2][x % 4], -shift);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 16 * a + lk + 4 * t, c = 16 * b + lr;
        put(r < nb && c < nb, r, c, X[a][b][t]);
      }
}

// The blocks of one launch (blockIdx.y): the two ends of a band go through
// their steps together.
constexpr int GJ_BATCH = 2;
struct GjPair {
  double* in[GJ_BATCH];
  double* out[GJ_BATCH];
};

// The first panel's pivot tile, inverted in place (one wave).
template <bool WIDE>
__global__ void __launch_bounds__(64) k_gj_first(GjPair m, long lda, int nb, double tiny, int* __restrict__ bad) {
  __builtin_amdgcn_s_setprio(3);
  double* A = m.in[blockIdx.y];
  const TileBuf<WIDE> t(A, nb, lda, nb);
  gj_invert_tile(nb, tiny, bad, [&](bool in, int r, int c) { return t.load(in, r, lda, c); },
                 [&](bool in, int r, int c, double v) { t.store(in, r, lda, c, v); });
}

// One step, panel k0 .. k0 + nb - 1 (its pivot tile in Ain already inverted);
// nb2 columns in the panel after it (0: none), whose pivot tile the last
// workgroup updates and inverts.
template <bool WIDE>
__global__ void __launch_bounds__(256) k_gj_step(GjPair m, long lda, long ldo, int n, int k0, int nb, int nb2,
                                                 double tiny, int* __restrict__ bad) {
  __shared__ GjSmem sm;
  const double* Ain = m.in[blockIdx.y];
  double* Aout = m.out[blockIdx.y];
  __builtin_amdgcn_s_setprio(3);  // the chain goes before the bulk products on its CU
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int lr = lane % 16, lk = lane / 16;
  const int nt = (n + GJ_T - 1) / GJ_T;
  const bool ahead = (int)blockIdx.x == nt * nt;  // the look-ahead workgroup
  const int kn = k0 + nb;                         // next panel
  const int i0 = ahead ? kn : (int)blockIdx.x / nt * GJ_T, j0 = ahead ? kn : (int)blockIdx.x % nt * GJ_T;
  const int ni = ahead ? nb2 : n - i0, nj = ahead ? nb2 : n - j0;  // rows and columns present
  auto in_panel = [&](int g) { return g >= k0 && g < kn; };
  // the tile's rows and the panel's rows
  const TileBuf<WIDE> rows(Ain + (long)i0 * lda, ni < GJ_T ? ni : GJ_T, lda, n), kk(Ain + (long)k0 * lda, nb, lda, n);
#pragma unroll
  for (int x = 0; x < GJ_T * GJ_NB / 256; ++x) {
    const int r = x * 8 + tid / GJ_NB, c = tid % GJ_NB;
    sm.AT[r][c] = rows.load(r < ni && c < nb, r, lda, k0 + c);
    const int q = x * 4 + tid / GJ_T, cc = tid % GJ_T;
    const double u = kk.load(cc < nj && q < nb, q, lda, j0 + cc);
    sm.U[q][cc] = in_panel(j0 + cc) ? (q == j0 + cc - k0 ? 1.0 : 0.0) : u;
  }
#pragma unroll
  for (int x = 0; x < GJ_NB * GJ_NB / 256; ++x) {
    const int r = x * 8 + tid / GJ_NB, c = tid % GJ_NB;
    sm.P[r][c] = kk.load(r < nb && c < nb, r, lda, k0 + c);
  }
  // A' of this thread's outputs: D(lk + 4 t, lr) of the wave's 2 x 2 MFMA
  // tiles (the look-ahead tile: one 16 x 16 quadrant per wave)
  const int wm = ahead ? wave / 2 * 16 : wave / 2 * 32, wn = ahead ? wave % 2 * 16 : wave % 2 * 32;
  f64x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = wm + 16 * a + lk + 4 * t, c = wn + 16 * b + lr;
        const bool in = r < ni && c < nj && !in_panel(i0 + r) && !in_panel(j0 + c);
        acc[a][b][t] = rows.load(in, r, lda, j0 + c);
      }
  __syncthreads();
  // -T = -A(i, kk) P^-1 in place of A(i, kk): wave w its rows 16 w .. 16 w + 15
  // (the look-ahead tile's 32 rows: waves 0 and 1); rows of kk: P^-1
  if (!ahead || wave < 2) {
    f64x4 t2[2] = {f64x4{0.0, 0.0, 0.0, 0.0}, f64x4{0.0, 0.0, 0.0, 0.0}};
    double av[GJ_NB / 4], pv[GJ_NB / 4][2];
#pragma unroll
    for (int k = 0; k < GJ_NB / 4; ++k) {
      av[k] = sm.AT[16 * wave + lr][4 * k + lk];
#pragma unroll
      for (int b = 0; b < 2; ++b) pv[k][b] = sm.P[4 * k + lk][16 * b + lr];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < GJ_NB / 4; ++k)
#pragma unroll
      for (int b = 0; b < 2; ++b) t2[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[k], pv[k][b], t2[b], 0, 0, 0);
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 16 * wave + lk + 4 * t, c = 16 * b + lr;
        sm.AT[r][c] = in_panel(i0 + r) ? sm.P[i0 + r - k0][c] : -t2[b][t];
      }
  }
  __syncthreads();
  const TileBuf<WIDE> out(Aout + (long)i0 * ldo, ni < GJ_T ? ni : GJ_T, ldo, n);
  if (ahead) {
    // S = A(next, next) - T U, through LDS to wave 0, which inverts it
    double av[GJ_NB / 4], bv[GJ_NB / 4];
#pragma unroll
    for (int k = 0; k < GJ_NB / 4; ++k) {
      av[k] = sm.AT[wm + lr][4 * k + lk];
      bv[k] = sm.U[4 * k + lk][wn + lr];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < GJ_NB / 4; ++k)
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[k], bv[k], acc[0][0], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < 4; ++t) sm.P[wm + lk + 4 * t][wn + lr] = acc[0][0][t];
    __syncthreads();
    if (wave == 0)
      gj_invert_tile(nb2, tiny, bad, [&](bool, int r, int c) { return sm.P[r][c]; },
                     [&](bool in, int r, int c, double v) { out.store(in, r, ldo, kn + c, v); });
    return;
  }
  double av[GJ_NB / 4][2], bv[GJ_NB / 4][2];
#pragma unroll
  for (int k = 0; k < GJ_NB / 4; ++k)
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      av[k][a] = sm.AT[wm + 16 * a + lr][4 * k + lk];
      bv[k][a] = sm.U[4 * k + lk][wn + 16 * a + lr];
    }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < GJ_NB / 4; ++k)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[k][a], bv[k][b], acc[a][b], 0, 0, 0);
  auto next_tile = [&](int g) { return g >= kn && g < kn + nb2; };
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = wm + 16 * a + lk + 4 * t, c = wn + 16 * b + lr;
        out.store(r < ni && c < nj && !(next_tile(i0 + r) && next_tile(j0 + c)), r, ldo, j0 + c, acc[a][b][t]);
      }
}

// ------------------------------------------------------------------ block products
// C (=, or -=) A B for a list of B x B blocks in one launch, row-major with
// their own pitches: the products of one block step are independent, and one
// launch over all their tiles fills the chip where a launch per product leaves
// a partly filled last round each.  A workgroup of 2 x 2 waves forms a
// (32 MT) x (32 NT) tile of one product, each wave MT x NT MFMA tiles
// (v_mfma_f64_16x16x4f64, 64 cycles each), K in slices of KS through two LDS
// buffers, the next slice loaded into registers under the current one's
// products.  Offsets within a slice are fixed per thread and only the
// descriptors move: with the offsets formed anew for each slice a lone
// workgroup on a CU spent as long on them as on its products.  64 x 64 tiles,
// slices of 16 (four workgroups a CU): 8 products of 640^3 in 92 us (46
// TFLOP/s: 800 tiles are 3.1 a CU), of 1920^3 in 1.71 ms (66; the card's
// matrix cores sustain 69).  The elimination's chain has one product at a
// time: 32 x 32 tiles and slices of 32 put 640^3 on every CU, 22 us against 41
// with 64 x 64.
// The bulk products ask for BG_RESERVE bytes of LDS they do not use: with two
// of them on a CU instead of four there is room for a workgroup of the
// elimination's chain, which would otherwise wait for one of them to end.
constexpr int BG_MAX = 16;
constexpr int BG_RESERVE = 16 * 1024;
struct BlockProduct {
  const double* A;
  const double* B;
  double* C;
  int lda, ldb, ldc;
};
struct BlockProducts {
  BlockProduct p[BG_MAX];
};

template <int MT, int NT, int KS, bool SUB>
__global__ void __launch_bounds__(256) k_block_products(BlockProducts list, int n) {
  constexpr int TM = 32 * MT, TN = 32 * NT;
  // pitches: an A operand reads (row l % 16, k l / 16), a B operand (k l / 16,
  // column l % 16); 2 mod 4 and 16 mod 32 doubles spread 32 lanes over all banks
  __shared__ double As[2][TM][KS + 2];
  __shared__ double Bs[2][KS][TN + 16];
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int lr = lane % 16, lk = lane / 16;
  const int ntn = (n + TN - 1) / TN;
  int bx, by;
  xcd_block(bx, by);
  const BlockProduct q = list.p[by];
  if constexpr (MT == 1) __builtin_amdgcn_s_setprio(3);
  const int m0 = bx / ntn * TM, n0 = bx % ntn * TN;
  const int mr = min(TM, n - m0);
  const int wm = wave / 2 * 16 * MT, wn = wave % 2 * 16 * NT;
  constexpr int NA = TM * KS / 256, NB = TN * KS / 256;
  static_assert(256 % KS == 0 && 256 % TN == 0, "staging shape");
  // this thread's elements of a slice: fixed offsets from its first one, which
  // moves by a scalar amount from slice to slice
  unsigned oa[NA], ob[NB];
#pragma unroll
  for (int x = 0; x < NA; ++x) {
    const int r = x * (256 / KS) + tid / KS;
    oa[x] = r < mr ? (unsigned)(r * q.lda + tid % KS) * 8u : NOWHERE;
  }
#pragma unroll
  for (int x = 0; x < NB; ++x) {
    const int r = x * (256 / TN) + tid / TN;
    ob[x] = n0 + tid % TN < n ? (unsigned)(r * q.ldb + n0 + tid % TN) * 8u : NOWHERE;
  }
  double ra[NA], rb[NB];
  auto fetch = [&](int k0) {
    const int kr = min(KS, n - k0);
    const TileBuf<> ta(q.A + (long)m0 * q.lda + k0, mr, q.lda, kr), tb(q.B + (long)k0 * q.ldb, kr, q.ldb, n);
    if (kr == KS) {
#pragma unroll
      for (int x = 0; x < NA; ++x) ra[x] = ta.load(oa[x]);
#pragma unroll
      for (int x = 0; x < NB; ++x) rb[x] = tb.load(ob[x]);
    } else {
      // the last, shorter slice: zeros past it
#pragma unroll
      for (int x = 0; x < NA; ++x) ra[x] = ta.load(tid % KS < kr ? oa[x] : NOWHERE);
#pragma unroll
      for (int x = 0; x < NB; ++x) rb[x] = tb.load(x * (256 / TN) + tid / TN < kr ? ob[x] : NOWHERE);
    }
  };
  auto stage = [&](int s) {
#pragma unroll
    for (int x = 0; x < NA; ++x) As[s][x * (256 / KS) + tid / KS][tid % KS] = ra[x];
#pragma unroll
    for (int x = 0; x < NB; ++x) Bs[s][x * (256 / TN) + tid / TN][tid % TN] = rb[x];
  };
  const TileBuf<> tc(q.C + (long)m0 * q.ldc, mr, q.ldc, n);
  f64x4 acc[MT][NT], cv[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
  auto slice = [&](int k0, int s) {
    const bool more = k0 + KS < n;
    if (more) fetch(k0 + KS);
#pragma unroll
    for (int k = 0; k < KS; k += 4) {
      double av[MT], bv[NT];
#pragma unroll
      for (int a = 0; a < MT; ++a) av[a] = As[s][wm + 16 * a + lr][k + lk];
#pragma unroll
      for (int b = 0; b < NT; ++b) bv[b] = Bs[s][k + lk][wn + 16 * b + lr];
#pragma unroll
      for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a], bv[b], acc[a][b], 0, 0, 0);
    }
    if (more) stage(s ^ 1);
    __syncthreads();
  };
  fetch(0);
  stage(0);
  __syncthreads();
  for (int k0 = 0; k0 < n; k0 += 2 * KS) {
    slice(k0, 0);
    if (k0 + KS < n) slice(k0 + KS, 1);
  }
  // all of C in flight together
  auto coff = [&](int a, int b, int t) {
    const int r = wm + 16 * a + lk + 4 * t, c = n0 + wn + 16 * b + lr;
    return r < mr && c < n ? (unsigned)(r * q.ldc + c) * 8u : NOWHERE;
  };
  if constexpr (SUB)
#pragma unroll
    for (int x = 0; x < MT * NT * 4; ++x) cv[x / 4 / NT][x / 4 % NT][x % 4] = tc.load(coff(x / 4 / NT, x / 4 % NT, x % 4));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int x = 0; x < MT * NT * 4; ++x) {
    const int a = x / 4 / NT, b = x / 4 % NT, t = x % 4;
    tc.store(coff(a, b, t), SUB ? cv[a][b][t] - acc[a][b][t] : acc[a][b][t]);
  }
}

// Scratch blocks into place: dst(r, c) = src(r, c) for n x n blocks, a row per
// workgroup.
struct CopyRow {
  const double* src;
  double* dst;
  int lds, ldd;
};
struct CopyRows {
  CopyRow c[BG_MAX];
};
__global__ void __launch_bounds__(256) k_copy_rows(CopyRows list, int n) {
  const CopyRow q = list.c[blockIdx.y];
  const double* s = q.src + (long)blockIdx.x * q.lds;
  double* d = q.dst + (long)blockIdx.x * q.ldd;
  for (int c = threadIdx.x; c < n; c += 256) d[c] = s[c];
}

// ------------------------------------------------------------------ band solve
// Matrix-vector products of one step of the band solve, one wave per row: for
// every job, y(r) (=, or -=) sum_c A(r, c) x(c), r < rows, c < n.  A step's
// jobs are independent (both ends of the band, all block rows a step reaches),
// so they share a launch; what bounds the solve is the chain of launches, two
// a block row forward and one back.
constexpr int BV_MAX = 8;
struct BandVec {
  const double* A;
  const double* x;
  double* y;
  long lda;
  int n, sub;
};
struct BandVecs {
  BandVec j[BV_MAX];
};
__global__ void __launch_bounds__(256) k_band_vec(BandVecs list, int rows) {
  const BandVec q = list.j[blockIdx.y];
  const int r = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x % 64;
  if (r >= rows) return;
  const double* a = q.A + r * q.lda;
  double s0 = 0.0, s1 = 0.0;
  int c = lane;
  for (; c + 64 < q.n; c += 128) {
    s0 += a[c] * q.x[c];
    s1 += a[c + 64] * q.x[c + 64];
  }
  if (c < q.n) s0 += a[c] * q.x[c];
  s0 += s1;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s0 += __shfl_xor(s0, off);
  if (lane == 0) q.y[r] = q.sub ? q.y[r] - s0 : s0;
}

// y = A x for a CSR matrix, or b - A x where b is given: one wave per row, so
// that a row's ~145 entries are consecutive loads (with one row per thread
// each lane walked its own row: 390 us for 164k rows of the 256 x 128 boundary
// layer).
__global__ void __launch_bounds__(256) k_csr_spmv(long n, const int* __restrict__ indptr,
                                                  const int* __restrict__ indices, const double* __restrict__ data,
                                                  const double* __restrict__ x, const double* __restrict__ b,
                                                  double* __restrict__ y) {
  const long r = (long)blockIdx.x * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (r >= n) return;
  double s = 0.0;
  const int end = indptr[r + 1];
  for (int p = indptr[r] + lane; p < end; p += 64) s += data[p] * x[indices[p]];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (lane == 0) y[r] = b ? b[r] - s : s;
}

}  // namespace bca
