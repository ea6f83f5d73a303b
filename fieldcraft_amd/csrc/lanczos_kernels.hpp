// Tall-skinny kernels of the shift-invert block Lanczos on the device (gfx950, wave64): the
// basis Q and its M products MQ are n x m column-major in HBM; a block W is n x b (b <= 8).
// Both kernels stream the basis once per call: HBM-bound on large problems, a few microseconds of
// launch and reduction on small ones. Six modes of a tet10 block of 5 x 7 x 9 cells (some 9 000
// unknowns) took 26.6 ms with one copy and one synchronization for each set of coefficients and
// chunks of 4 096 rows, now 14.1.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fc {

constexpr int TS_ROWS = 4096;   // most rows of one partial sum of ts_dots (and of the argmax chunks)
constexpr int TS_COLS = 8;      // basis columns one ts_dots workgroup takes
constexpr int TS_MAXB = 8;      // block columns

// Rows of a partial sum for n rows: TS_ROWS, or fewer (whole sweeps of a workgroup) so that a small
// block is spread over up to 128 chunks (at 9 000 rows, chunks of 4 096 were three workgroups a tile
// of the basis and 30 us a launch; chunks of 256 take 6 us).
inline int64_t ts_rows(int64_t n) {
  const int64_t r = (n + 127) / 128, s = (r + 255) / 256 * 256;
  return s < TS_ROWS ? s : TS_ROWS;
}

// partial[(chunk * m + i) * b + j] = sum over the chunk's rows r of A[r, i] B[r, j], for the
// TS_COLS columns i of this workgroup's tile: each thread walks rows r = chunk start + tid +
// 256 k with the b entries of B's row in registers, then the workgroup reduces its TS_COLS x
// TS_MAXB sums in a fixed order, so every partial is the same bits on every run: within a wave by
// halving exchanges (a lane keeps half of its values each time and adds its partner's: 63 exchanges,
// lane l ending with sum l, instead of six for every sum), then the four waves in order.
__global__ __launch_bounds__(256) void k_ts_dots(int64_t n, int64_t rows, const double* __restrict__ A, int64_t lda, int m,
                                                 const double* __restrict__ B, int64_t ldb, int b,
                                                 double* __restrict__ partial) {
  const int tile = blockIdx.y, chunk = blockIdx.x;
  const int i0 = tile * TS_COLS;
  const int cols = min(TS_COLS, m - i0);
  const int64_t r0 = (int64_t)chunk * rows, r1 = min<int64_t>(n, r0 + rows);
  double acc[TS_COLS * TS_MAXB];
#pragma unroll
  for (int q = 0; q < TS_COLS * TS_MAXB; ++q) acc[q] = 0.0;
  for (int64_t r = r0 + threadIdx.x; r < r1; r += 256) {
    double bv[TS_MAXB], av[TS_COLS];
#pragma unroll
    for (int j = 0; j < TS_MAXB; ++j) bv[j] = j < b ? B[(int64_t)j * ldb + r] : 0.0;
#pragma unroll
    for (int i = 0; i < TS_COLS; ++i) av[i] = i < cols ? A[(int64_t)(i0 + i) * lda + r] : 0.0;
#pragma unroll
    for (int i = 0; i < TS_COLS; ++i)
#pragma unroll
      for (int j = 0; j < TS_MAXB; ++j) acc[i * TS_MAXB + j] += av[i] * bv[j];
  }
  __shared__ double red[4][TS_COLS * TS_MAXB];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) {  // values [0, 2 h) of a lane: keep the half its bit h names
    const bool up = lane & h;
#pragma unroll
    for (int q = 0; q < h; ++q) {
      const double give = up ? acc[q] : acc[q + h], keep = up ? acc[q + h] : acc[q];
      acc[q] = keep + __shfl_xor(give, h, 64);
    }
  }
  red[wave][lane] = acc[0];
  __syncthreads();
  for (int q = threadIdx.x; q < cols * b; q += 256) {
    const int i = q / b, j = q % b, e = i * TS_MAXB + j;
    partial[((int64_t)chunk * m + i0 + i) * b + j] = red[0][e] + red[1][e] + red[2][e] + red[3][e];
  }
}

// C[i * b + j] = sum over chunks, in chunk order, of the partials (eight loads in flight). out, if not
// null, is pinned host memory that gets the same values: a copy of its own for each of the small
// results a block step reads cost 3 us and its call.
__global__ void k_ts_dots_sum(const double* __restrict__ partial, int chunks, int m, int b, double* __restrict__ C,
                              double* __restrict__ out) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= m * b) return;
  double v = 0.0;
  int c = 0;
  for (; c + 8 <= chunks; c += 8) {
    double p[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) p[t] = partial[(int64_t)(c + t) * m * b + q];
#pragma unroll
    for (int t = 0; t < 8; ++t) v += p[t];
  }
  for (; c < chunks; ++c) v += partial[(int64_t)c * m * b + q];
  C[q] = v;
  if (out) out[q] = v;
}

// B[r, j] = beta B[r, j] + alpha sum_i A[r, i] C[i * ldc + j] for j < b: one thread per row,
// the coefficients in LDS (m x b <= TS_MAXC entries), each row's sums in column order.
constexpr int TS_MAXC = 4096;
__global__ __launch_bounds__(256) void k_ts_update(int64_t n, const double* __restrict__ A, int64_t lda, int m,
                                                   const double* __restrict__ C, int ldc, double* __restrict__ B,
                                                   int64_t ldb, int b, double alpha, double beta) {
  __shared__ double c[TS_MAXC];
  for (int q = threadIdx.x; q < m * b; q += 256) c[q] = C[(q / b) * ldc + q % b];
  __syncthreads();
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= n) return;
  double acc[TS_MAXB];
#pragma unroll
  for (int j = 0; j < TS_MAXB; ++j) acc[j] = 0.0;
  int i = 0;
  for (; i + 8 <= m; i += 8) {  // eight basis columns in flight
    double a[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) a[t] = A[(int64_t)(i + t) * lda + r];
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int j = 0; j < TS_MAXB; ++j)
        if (j < b) acc[j] += a[t] * c[(i + t) * b + j];
  }
  for (; i < m; ++i) {
    const double a = A[(int64_t)i * lda + r];
#pragma unroll
    for (int j = 0; j < TS_MAXB; ++j)
      if (j < b) acc[j] += a * c[i * b + j];
  }
#pragma unroll
  for (int j = 0; j < TS_MAXB; ++j)
    if (j < b) {
      double* p = B + (int64_t)j * ldb + r;
      *p = (beta == 0.0 ? 0.0 : beta * *p) + alpha * acc[j];  // beta = 0: B is not read
    }
}

// x[r] *= s (one column)
__global__ void k_scale(int64_t n, double* __restrict__ x, double s) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r < n) x[r] *= s;
}

// q[r] = s v[r] and mv[r] *= s: a finished vector's place in the basis and its M product
__global__ void k_normalize(int64_t n, const double* __restrict__ v, double* __restrict__ q, double* __restrict__ mv, double s) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= n) return;
  q[r] = v[r] * s;
  mv[r] *= s;
}

// per chunk of TS_ROWS rows: the first index of the largest |x| (ties: the lower index)
__global__ void k_argmax_abs(int64_t n, const double* __restrict__ x, int64_t* __restrict__ at) {
  __shared__ double bv[256];
  __shared__ int64_t bi[256];
  const int64_t r0 = (int64_t)blockIdx.x * TS_ROWS, r1 = min<int64_t>(n, r0 + TS_ROWS);
  double best = -1.0;
  int64_t bidx = r0;
  for (int64_t r = r0 + threadIdx.x; r < r1; r += 256) {
    const double v = fabs(x[r]);
    if (v > best) {
      best = v;
      bidx = r;
    }
  }
  bv[threadIdx.x] = best;
  bi[threadIdx.x] = bidx;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      const double o = bv[threadIdx.x + s];
      const int64_t oi = bi[threadIdx.x + s];
      if (o > bv[threadIdx.x] || (o == bv[threadIdx.x] && oi < bi[threadIdx.x])) {
        bv[threadIdx.x] = o;
        bi[threadIdx.x] = oi;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) at[blockIdx.x] = bi[0];
}

}  // namespace fc
