// A panel's diagonal block and the rows below it on the matrix cores (gfx950).
//
// diag_potrf_inv factors and inverts a diagonal block of up to 128 columns in LDS by one
// workgroup (k_potrf_blk: a panel's; k_small_fronts: a small front's); substitute_block solves
// sixteen rows a wave against a factored block without leaving the wave's registers.
#pragma once

#include "gemm_kernels.hpp"

namespace fc {

constexpr int DB = 16;  // columns of a diagonal-block step: one MFMA tile
constexpr double PIVOT_TOL = 1e-10;  // cholesky.rs:48

// A double from one lane (uniform index) to the whole wave, by scalar reads of its halves.
__device__ __forceinline__ double readlane_d(double v, int l) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// d = sqrt(p), correctly rounded on all of 4 000 values over 2^-600 .. 2^600, and rd = 1 / d to a
// rounding: the hardware's estimate, one coupled Newton step on (sqrt p, 1 / (2 sqrt p)), then each
// corrected by its own residual.
__device__ __forceinline__ void root_pair(double p, double& d, double& rd) {
  const double y = __builtin_amdgcn_rsq(p);
  double s = p * y, h = 0.5 * y;
  const double e = fma(-h, s, 0.5);
  s = fma(s, e, s);
  h = fma(h, e, h);
  d = fma(fma(-s, s, p), h, s);
  const double r = h + h;
  rd = fma(fma(-d, r, 1.0), r, r);
}

// The h x h block (h <= NMAX, whole steps of DB columns) at S[0.., 0..], factored with the
// reference's pivot test (cholesky.rs:1161) and inverted, in FP64 (EXACT: the quotients by the
// pivot's root rounded as divisions, for FP64 storage). On entry S holds A in its lower
// triangle over the 16 nb x 16 nb square (nb = ceil(h / 16)), zeros above it, and an identity in
// the rows and columns past h; on return S[i][j] = L(i, j) for i >= j, the inverse's diagonal
// blocks are X[b] (transposed: X[b][c][r] = Linv(16 b + r, 16 b + c), zeros for r < c) and its other
// blocks lie transposed above the diagonal blocks of S, S[k][i] = Linv(i, k) (diag_inv reads an
// entry). The entries of S above the diagonal inside a diagonal block are left undefined. One wave
// per 16 rows of NMAX calls it together; it ends on a barrier.
//
// A block of 128 columns is a chain of 128 dependent pivots, so what sets its time is the
// latency of a step. Each step of 16 columns is taken by every wave on its own copy of the 16 x 16
// pivot block (lanes 0..15, a row a lane) with 48 other rows in the wave's other lanes: the
// rows below, and, since the rows of an identity appended below the block become the columns of
// the inverse, the identity's rows too. One instruction stream then gives L, the rows below it by
// true substitution and the inverse, with the pivot column broadcast by scalar reads (no
// LDS round trip and no barrier inside a step). Row c of the identity is nonzero from column c
// on, so its entries live in the upper triangle of S and each step has 16 nb rows to take. The
// trailing update S(r, j) -= P(r) L(j)^T (rows below, and identity rows already started) goes
// through the 16x16x4 MFMA, row block r by wave r. Measured, a 128-column block: 90 us with a wave's
// 8 x 8 lane grid passing columns through LDS shuffles on 32-column quarters, and products between
// the quarters (FP32 arithmetic: 60 us); 37 us in this form, the pivots' chain some 12 us of it, the tiles 9.
template <int NMAX>
using DiagX = double[NMAX / DB][DB][DB + 1];

template <int NMAX, bool EXACT>
__device__ inline void diag_potrf_inv(double (*S)[NMAX + 1], DiagX<NMAX>& X, int h, int tid,
                                      const double* __restrict__ dg, int64_t col,
                                      unsigned long long* __restrict__ fail) {
  constexpr int ROWS = 64 - DB;  // rows a wave takes beside the pivot block
  static_assert(NMAX / DB * ROWS >= NMAX, "a step's rows fit the workgroup's waves");
  const int lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
  const int nb = (h + DB - 1) / DB;
  for (int kb = 0; kb < nb; ++kb) {
    const int c0 = DB * kb;
    // slot 0..15: the identity's rows c0 ..; then the block's other rows in order
    const int slot = wave * ROWS + lane - DB;
    const bool piv = lane < DB, ident = !piv && slot < DB, act = !piv && slot < DB * nb;
    const int row = (piv || ident || !act) ? c0 + (piv ? lane : 0) : (slot - DB < c0 ? slot - DB : slot);
    const bool work = wave * ROWS < DB * nb;  // uniform
    double a[DB];
    if (work) {
#pragma unroll
      for (int t = 0; t < DB; ++t) a[t] = S[row][c0 + t];
      if (ident)
#pragma unroll
        for (int t = 0; t < DB; ++t) a[t] = t == slot ? 1.0 : 0.0;
    }
    const double dl = (lane < DB && c0 + lane < h) ? fabs(dg[c0 + lane]) : 0.0;
    __syncthreads();  // every copy of the pivot block read before it is overwritten
    if (work) {
      double pv = 0.0;  // lane j: pivot j
      double p = readlane_d(a[0], 0), d, rd;
      root_pair(p, d, rd);
#pragma unroll
      for (int j = 0; j < DB; ++j) {
        pv = lane == j ? p : pv;
        double l = a[j] * rd;
        if constexpr (EXACT) l = fma(fma(-l, d, a[j]), rd, l);  // a[j] / d to a rounding
        a[j] = l;
        // the next pivot first: its reciprocal root is the step's dependent chain, the other
        // columns' updates fill it (one scheduling region a step: the broadcasts of several steps
        // together do not fit the scalar registers)
        if (j + 1 < DB) {
          a[j + 1] = fma(-l, readlane_d(l, j + 1), a[j + 1]);
          p = readlane_d(a[j + 1], j + 1);
          root_pair(p, d, rd);
        }
#pragma unroll
        for (int k = j + 2; k < DB; ++k) a[k] = fma(-l, readlane_d(l, k), a[k]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (wave == 0 && lane < DB && c0 + lane < h && (!(pv > PIVOT_TOL * dl) || !isfinite(pv)))
        atomicMin(fail, (unsigned long long)(col + c0 + lane));
      if (act || (piv && wave == 0)) {
        double dv, rv;  // L(t, t): the root itself (the quotient p / d is a rounding further off)
        root_pair(pv, dv, rv);
        double* dst = ident ? X[kb][slot] : &S[row][c0];
#pragma unroll
        for (int t = 0; t < DB; ++t) dst[t] = lane == t ? dv : a[t];
      }
    }
    __syncthreads();
    // row block `wave`: every column block after kb up to its own (below), or all (the identity's)
    const int hi = wave > kb ? min(wave, nb - 1) : nb - 1;
    if (wave < nb) {
      const double* src = wave == kb ? X[kb][r] : &S[DB * wave + r][c0];
      double fi[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) fi[s] = src[4 * s + g];
      for (int jb = kb + 1; jb <= hi; ++jb) {
        double* out = &S[DB * wave + r][DB * jb + g];
        double fj[4], old[4];
        v4d acc = {0, 0, 0, 0};  // the products by themselves: one rounding of the entry, not sixteen
#pragma unroll
        for (int s = 0; s < 4; ++s) fj[s] = S[DB * jb + r][c0 + 4 * s + g];
#pragma unroll
        for (int v = 0; v < 4; ++v) old[v] = out[4 * v];
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = Mma<double>::step(fj[s], fi[s], acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) out[4 * v] = old[v] - acc[v];
      }
    }
    __syncthreads();
  }
}

// Linv(i, j), i >= j, of a block diag_potrf_inv has left.
template <int NMAX>
__device__ __forceinline__ double diag_inv(const double (*S)[NMAX + 1], const DiagX<NMAX>& X, int i, int j) {
  return i / DB == j / DB ? X[i / DB][j % DB][i % DB] : S[j][i];
}

// The diagonal block of a panel (any width up to NB; item: f, a = c0): factored with the
// reference's pivot test (cholesky.rs:1146-1171: a pivot not above 1e-10 |A_jj|, or not finite,
// fails the column) and inverted, in FP64 arithmetic whatever the storage. L11 goes over the
// block's lower triangle in L, Linv (pw x pw, column-major, zeros above the diagonal) to the
// panel's slot of Inv (F.inv0 + (c0 / NB) NB^2). One workgroup a block: the chain of pivots bounds
// it (diag_potrf_inv), so the loads and stores around it are made in one batch each.
constexpr int POTRF_THREADS = 512;
template <typename T>
__global__ __launch_bounds__(POTRF_THREADS, 1) void k_potrf_blk(const Item* __restrict__ items,
                                                                const FrontDev* __restrict__ fronts, T* __restrict__ L,
                                                                const double* __restrict__ diag,
                                                                unsigned long long* __restrict__ fail, T* __restrict__ Inv,
                                                                __bf16* __restrict__ Lh, __bf16* __restrict__ Ll,
                                                                const int32_t* __restrict__ fexp) {
  static_assert(POTRF_THREADS == 64 * (NB / DB), "a wave a row block");
  __shared__ double S[NB][NB + 1];
  __shared__ DiagX<NB> X;
  constexpr int CQ = POTRF_THREADS / NB, Q = NB / CQ;  // thread: one row, every CQ-th column
  const Item it = items[blockIdx.x];
  const FrontDev F = fronts[it.f];
  const int c0 = it.a, pw = min(NB, F.w - c0);
  T* base = L + F.lpos + (int64_t)c0 * F.ld + c0;
  const int tid = threadIdx.x, rr = tid & (NB - 1), jp = tid / NB;
  {
    // the lower triangle through a buffer resource (the block spans far below 2 GiB of L): an entry
    // outside it takes the lane offset 2^31, past the resource's 2^31 - 1 bytes, and reads 0 from
    // the buffer unit's range check, with no branch around the load
    const auto rs = raw_rsrc(base);
    const uint32_t ldb = (uint32_t)F.ld * sizeof(T);
    T v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int j = jp + CQ * q;
      v[q] = buf_load<T>(rs, (rr < pw && j <= rr) ? (uint32_t)(rr * sizeof(T)) : 0x80000000u, j * ldb);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int j = jp + CQ * q;
      S[rr][j] = (rr == j && rr >= pw) ? 1.0 : (double)v[q];
    }
  }
  __syncthreads();
  diag_potrf_inv<NB, sizeof(T) == 8>(S, X, pw, tid, diag + F.col0 + c0, (int64_t)F.col0 + c0, fail);
  {
    T* inv = Inv + F.inv0 + (int64_t)(c0 / NB) * NB * NB;
    T v[Q], x[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int j = jp + CQ * q;
      v[q] = (T)S[rr][j];
      x[q] = (rr >= j && rr < pw) ? (T)diag_inv<NB>(S, X, rr, j) : T(0);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int j = jp + CQ * q;
      if (rr < pw && j <= rr) base[(int64_t)j * F.ld + rr] = v[q];
      if (rr < pw && j < pw) inv[(int64_t)j * pw + rr] = x[q];
    }
  }
  // Mixed form (Lh given): the block's scaled BF16 copies, from the same FP32 values as L (zero
  // above the diagonal and past the block up to the next multiple of 32 columns), 8 columns of a
  // row per 16-byte store.
  if (Lh) {
    const float sc = ldexpf(1.0f, -fexp[it.f]);
    const int ncp = (c0 + pw + 31) / 32 * 32 - c0;
    for (int e = tid; e < pw * (ncp / 8); e += POTRF_THREADS) {
      const int r = e % pw, g = e / pw;
      v8bf h, l;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int j = 8 * g + q;
        const float x = (j <= r ? (float)(T)S[r][min(j, NB - 1)] : 0.0f) * sc;
        h[q] = (__bf16)x;
        l[q] = (__bf16)(x - (float)h[q]);
      }
      const int col = c0 + 8 * g;
      const int64_t o = F.bpos + ((int64_t)(col / 32) * F.ld + c0 + r) * 32 + col % 32;
      *(v8bf*)(Lh + o) = h;
      *(v8bf*)(Ll + o) = l;
    }
  }
}

// X L11^T = B for sixteen rows a wave, by blocks of 16 columns in the wave's registers:
//   X_k = (B_k - sum_{j < k} X_j L_kj^T) L_kk^-T
// x[k] holds B_k on entry and X_k on return, in the MFMA's output layout (entry v of a lane: row
// lane % 16, column 16 k + row(lane, v)). That layout is also the layout of the next product's
// row operand when the products sum their 16 columns in the order row(lane, s), so no value moves
// between lanes. Lop(j, s), Xop(s) and Dop(s) return the lane's column operand: entry
// (lane % 16, row(lane, s)) of L_kj, L_kk^-1 and L_kk (k a constant of the unrolled caller).
// REFINE corrects each X_k once against L_kk (a product with an explicit inverse alone is not
// backward stable). DIAG (unrefined, 32-bit products): Xop leaves the inverse's diagonal out and
// Dop(s) is its entry of column row(lane, s), whose term, the largest, is then added last.
//
// Rounding: each earlier block's product is summed from zero and the sums leave B_k at once, and the
// residual is B_k less one sum that ends with X_k L_kk^T, so that a value takes three roundings of its own
// size. Residuals of rows below a well-conditioned 128-column block, rms over |x| |L11|, in units of
// u / sqrt(128): FP64 0.51, FP32 0.85; with the products carried on the running value 3.4 and 3.3;
// products with the whole block's inverse 0.57 (refined) and 1.4. Below 64 columns of a small front,
// FP64: 0.49, against 2.4 both ways before.
template <typename M, bool REFINE, bool DIAG, int NBK, class FL, class FX, class FD>
__device__ __forceinline__ void substitute_block(typename Mma<M>::acc_t (&x)[NBK], int k, FL Lop, FX Xop, FD Dop) {
  typedef typename Mma<M>::acc_t acc_t;
  acc_t sum = {0, 0, 0, 0}, y = {0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < NBK; ++j)
    if (j < k) {
      acc_t t = {0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < 4; ++s) t = Mma<M>::step(Lop(j, s), x[j][s], t);
      sum = j == 0 ? t : sum + t;
    }
  const acc_t b = k > 0 ? x[k] - sum : x[k];
#pragma unroll
  for (int s = 0; s < 4; ++s) y = Mma<M>::step(Xop(s), b[s], y);
  if constexpr (DIAG)
#pragma unroll
    for (int s = 0; s < 4; ++s) y[s] = fma(Dop(s), b[s], y[s]);
  if constexpr (REFINE) {
#pragma unroll
    for (int s = 0; s < 4; ++s) sum = Mma<M>::step(Dop(s), y[s], sum);
    const acc_t res = x[k] - sum;
    acc_t d = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) d = Mma<M>::step(Xop(s), res[s], d);
    y += d;
  }
  x[k] = y;
}

// The rows below a panel's diagonal block, X L11^T = B in place (item: f, a = c0, b = first row):
// each wave takes sixteen rows through the panel's blocks of sixteen columns in its registers, as
// substitute_block does, with the factored block's operands read from L and the inverse's diagonal
// blocks from Inv (both in L2: every wave of the launch reads the same 72 KB) one block row ahead
// of their use. No LDS, no barrier, and a launch has as many waves as rows / 16, so that the few
// rows of a small level still spread over the chip: the product with the whole inverse on 128-row
// tiles gave a level of 2 000 rows 16 workgroups, and the FP64 factor four launches (copy,
// product, residual, correction) of three times this one's products.
// SPLIT (mixed form): the rows' scaled BF16 copies too (see k_gemm_b16): a lane's four values of a
// block are consecutive columns of one row, one 8-byte store a copy; columns from the panel's
// width up to the next multiple of 32 are zeros (their operands read 0).
constexpr int TRSM_WAVES = 4;  // waves of a workgroup in launches of many rows (else 1)
template <typename T, bool SPLIT>
__global__ __launch_bounds__(64 * TRSM_WAVES) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_trsm(const Item* __restrict__ items,
                                                          const FrontDev* __restrict__ fronts, T* L,
                                                          const T* __restrict__ Inv, __bf16* __restrict__ Lh,
                                                          __bf16* __restrict__ Ll, const int32_t* __restrict__ fexp) {
  typedef typename Mma<T>::acc_t acc_t;
  constexpr bool REFINE = sizeof(T) == 8;
  constexpr int NBK = NB / DB;
  constexpr uint32_t OUT = 0x80000000u;
  const Item it = items[blockIdx.x];
  const FrontDev F = fronts[it.f];
  const int lane = threadIdx.x & 63, r = lane & 15;
  const int c0 = it.a, pw = min(NB, F.w - c0), i = it.b + 16 * (int)(threadIdx.x >> 6) + r;
  const int q0 = Mma<T>::row(lane, 0), dq = Mma<T>::row(lane, 1) - q0;  // a lane's columns of a block: q0 + dq v
  const bool in = i < F.m;
  const auto rs = raw_rsrc(L + F.lpos + (int64_t)c0 * F.ld);
  const auto ri = raw_rsrc(Inv + F.inv0 + (int64_t)(c0 / NB) * NB * NB);
  const uint32_t ldb = (uint32_t)F.ld * sizeof(T), pwb = (uint32_t)pw * sizeof(T);
  const uint32_t li = (uint32_t)i * sizeof(T) + q0 * ldb;
  acc_t x[NBK];
#pragma unroll
  for (int k = 0; k < NBK; ++k)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      x[k][v] = buf_load<T>(rs, in && 16 * k + q0 + dq * v < pw ? li : OUT, (16 * k + dq * v) * ldb);
  // block row k's operands: L_kj (j < k), L_kk^-1 and, to refine, L_kk
  auto fetch = [&](int k, T (&lo)[NBK][4], T (&xo)[4], T (&dd)[4]) {
    const bool rin = 16 * k + r < pw;
    const uint32_t lr = (uint32_t)(c0 + 16 * k + r) * sizeof(T) + q0 * ldb;
    const uint32_t lx = (uint32_t)(16 * k + r) * sizeof(T) + (16 * k + q0) * pwb;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bool cin = rin && q0 + dq * s <= r;  // the lower triangle of the diagonal blocks
      xo[s] = buf_load<T>(ri, cin ? lx : OUT, dq * s * pwb);
      if (REFINE) dd[s] = buf_load<T>(rs, cin ? lr : OUT, (16 * k + dq * s) * ldb);
    }
#pragma unroll
    for (int j = 0; j < NBK; ++j)
      if (j < k)
#pragma unroll
        for (int s = 0; s < 4; ++s) lo[j][s] = buf_load<T>(rs, rin ? lr : OUT, (16 * j + dq * s) * ldb);
  };
  T lo[2][NBK][4], xo[2][4], dd[2][4];
  fetch(0, lo[0], xo[0], dd[0]);
#pragma unroll
  for (int k = 0; k < NBK; ++k) {
    const int cur = k & 1;
    if (k + 1 < NBK) fetch(k + 1, lo[cur ^ 1], xo[cur ^ 1], dd[cur ^ 1]);
    __builtin_amdgcn_sched_barrier(0);  // the next row's loads are issued before this one's products
    substitute_block<T, REFINE, !REFINE>(
        x, k, [&](int j, int s) { return lo[cur][j][s]; },
        [&](int s) { return REFINE || q0 + dq * s != r ? xo[cur][s] : T(0); },
        [&](int s) { return REFINE ? dd[cur][s] : __shfl(xo[cur][s], (lane & 48) + q0 + dq * s); });
  }
#pragma unroll
  for (int k = 0; k < NBK; ++k)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      buf_store<T>(rs, (T)x[k][v], in && 16 * k + q0 + dq * v < pw ? li : OUT, (16 * k + dq * v) * ldb);
  if constexpr (SPLIT) {
    static_assert(sizeof(T) == 4, "copies of an FP32 result");
    const float sc = ldexpf(1.0f, -fexp[it.f]);
    const int ncp = (pw + 31) / 32 * 32;  // c0 is a multiple of 32
#pragma unroll
    for (int k = 0; k < NBK; ++k) {
      const int j = 16 * k + q0;
      if (in && j < ncp) {
        __bf16 h[4], l[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float y = (float)x[k][v] * sc;
          h[v] = (__bf16)y;
          l[v] = (__bf16)(y - (float)h[v]);
        }
        const int col = c0 + j;
        const int64_t o = F.bpos + ((int64_t)(col / 32) * F.ld + i) * 32 + col % 32;
        *(uint2*)(Lh + o) = *(const uint2*)h;
        *(uint2*)(Ll + o) = *(const uint2*)l;
      }
    }
  }
}

}  // namespace fc
