// Small fronts in one launch per level (gfx950).
//
// The tree's leaf and near-leaf fronts are many and tiny (at hex8 80^3, 14 755 fronts of median
// width 18 and 180 rows at the bottom level): too small for the tiled kernels' 128 x 128 tiles
// and 128-column diagonal blocks, where each of a level's dense steps is a launch of its own.
// The small fronts of a level (no wider than SMALL_W columns, their update matrices at most
// SMALL_SYRK multiply-adds) take one launch between the level's two extend-add launches, in
// which each workgroup does one front's dense steps, all sums in FP64 whatever the storage:
//   1. its diagonal block, factored and inverted in LDS (diag_potrf_inv), L11 and the inverse
//      written out;
//   2. the rows below by block substitution on the matrix cores, sixteen rows a wave
//      (substitute_block; the FP64 factor refines each block once, as the tiled path does);
//   3. its update matrix U = -L21 L21^T (lower triangle), 32 x 32 tiles a wave on the matrix cores.
// The values end where the tiled path puts them (L, Inv, U); the FP32-storage forms write no
// BF16 copies for them, since no product of the tiled path reads a small front.
//
// Bound: a workgroup's own chain (diagonal block, rows, products), since a level has few fronts of
// equal weight. Rows as one thread each and products on the vector units took 266 us in the
// largest launch of the 40 x 8 x 8 cantilever's FP64 factor and 192 us of the 40^3 cube's mixed one (the
// FP64 row code spilled); on the matrix cores 74 and 104 us, with the levels counted from the root and
// so more fronts in them (41 and 66 on average).
#pragma once

#include "panel_kernels.hpp"

namespace fc {

constexpr int SMALL_W = 64;            // widest small front
constexpr int SMALL_MU = 768;          // most rows below a small front's columns
constexpr double SMALL_SYRK = 2.0e6;   // most multiply-adds of a small front's update matrix

// Workgroup b takes the front items[b].f (the launch's items are costliest first, so the
// hardware's dispatch in order balances the CUs).
template <typename T>
__global__ __launch_bounds__(256, 2) void k_small_fronts(const Item* __restrict__ items,
                                                         const FrontDev* __restrict__ fronts, T* __restrict__ L,
                                                         T* __restrict__ U, const double* __restrict__ diag,
                                                         unsigned long long* __restrict__ fail, T* __restrict__ Inv) {
  __shared__ double S[SMALL_W][SMALL_W + 1];
  __shared__ DiagX<SMALL_W> X;
  constexpr uint32_t OUT = 0x80000000u;  // a lane offset past a buffer resource: reads 0, stores nothing
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const FrontDev F = fronts[items[blockIdx.x].f];
  const int w = F.w, mu = F.m - F.w, nb = (w + DB - 1) / DB;
  T* base = L + F.lpos;
  const auto rs = raw_rsrc(base);
  const uint32_t ldb = (uint32_t)F.ld * sizeof(T);
  // 1. the diagonal block (thread t: row t % 64, columns t / 64 + 4 q; the loads issued before any
  // is used, those outside the triangle reading 0 through the buffer unit's range check)
  {
    const int i = tid & (SMALL_W - 1), j0 = tid >> 6;
    T v[SMALL_W / 4];
#pragma unroll
    for (int q = 0; q < SMALL_W / 4; ++q) {
      const int j = j0 + 4 * q;
      v[q] = buf_load<T>(rs, (i < w && j <= i) ? (uint32_t)(i * sizeof(T)) : OUT, j * ldb);
    }
#pragma unroll
    for (int q = 0; q < SMALL_W / 4; ++q) {
      const int j = j0 + 4 * q;
      S[i][j] = (i == j && i >= w) ? 1.0 : (double)v[q];
    }
  }
  __syncthreads();
  diag_potrf_inv<SMALL_W, sizeof(T) == 8>(S, X, w, tid, diag + F.col0, F.col0, fail);
  // L11 out, and the inverse (column-major, ld = w, zeros above the diagonal)
  for (int e = tid; e < w * w; e += blockDim.x) {
    const int i = e % w, j = e / w;
    if (j <= i) base[(int64_t)j * F.ld + i] = (T)S[i][j];
    Inv[F.inv0 + (int64_t)j * w + i] = i >= j ? (T)diag_inv<SMALL_W>(S, X, i, j) : T(0);
  }
  // 2. the rows below, sixteen a wave: entry v of x[k] is row i, column 16 k + lane / 16 + 4 v
  const int r = lane & 15, g = lane >> 4;
  constexpr int NBK = SMALL_W / DB;
  for (int i0 = 16 * wave; i0 < mu; i0 += 64) {
    const uint32_t lo = i0 + r < mu ? (uint32_t)(w + i0 + r) * sizeof(T) + g * ldb : OUT;
    v4d x[NBK];
    T b[NBK][4];
#pragma unroll
    for (int k = 0; k < NBK; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) b[k][v] = buf_load<T>(rs, 16 * k + 4 * v + g < w ? lo : OUT, (16 * k + 4 * v) * ldb);
#pragma unroll
    for (int k = 0; k < NBK; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) x[k][v] = (double)b[k][v];
#pragma unroll
    for (int k = 0; k < NBK; ++k) {
      if (k >= nb) break;
      substitute_block<double, sizeof(T) == 8, false>(
          x, k, [&](int j, int s) { return S[16 * k + r][16 * j + 4 * s + g]; },
          [&](int s) { return X[k][4 * s + g][r]; },
          [&](int s) {
            const int c = 4 * s + g;
            const double v = S[16 * k + r][16 * k + c];
            return c <= r ? v : 0.0;
          });
    }
#pragma unroll
    for (int k = 0; k < NBK; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) buf_store<T>(rs, (T)x[k][v], 16 * k + 4 * v + g < w ? lo : OUT, (16 * k + 4 * v) * ldb);
  }
  __syncthreads();  // every row below final before the products read them
  // 3. U = -L21 L21^T by lower 32 x 32 tiles, a wave each (2 x 2 blocks of the MFMA): operand rows
  // read from L (the workgroup's own stores), KS steps of four columns in flight at once, rows
  // past mu and columns past w as 0
  constexpr int KS = 4;
  const int nt = (mu + 31) / 32, tiles = nt * (nt + 1) / 2;
  for (int t = wave; t < tiles; t += 4) {
    int tj = 0, q = t;
    while (q >= nt - tj) q -= nt - tj, ++tj;
    const int j0 = 32 * tj, i0 = j0 + 32 * q;
    uint32_t oi[2], oj[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      oi[a] = i0 + 16 * a + r < mu ? (uint32_t)(w + i0 + 16 * a + r) * sizeof(T) + g * ldb : OUT;
      oj[a] = j0 + 16 * a + r < mu ? (uint32_t)(w + j0 + 16 * a + r) * sizeof(T) + g * ldb : OUT;
    }
    v4d acc[2][2] = {};
    for (int k0 = 0; k0 < w; k0 += 4 * KS) {
      T fi[KS][2], fj[KS][2];
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const int k = k0 + 4 * s;
          fi[s][a] = buf_load<T>(rs, k + g < w ? oi[a] : OUT, k * ldb);
          fj[s][a] = buf_load<T>(rs, k + g < w ? oj[a] : OUT, k * ldb);
        }
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[a][c] = Mma<double>::step((double)fj[s][c], (double)fi[s][a], acc[a][c]);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = i0 + 16 * a + r, j = j0 + 16 * c + g + 4 * v;
          if (i < mu && j <= i) U[F.upos + (int64_t)j * mu + i] = (T)(-acc[a][c][v]);
        }
  }
}

}  // namespace fc
