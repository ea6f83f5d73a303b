// Supernodal triangular solves over the fronts (the reference's solve_group,
// cholesky.rs:904-1037, reorganised for levels of the front tree) and the FP64 vector steps of
// refinement.
//
// Forward, leaves first: a front adds up its children's contributions (each child hands up the
// products of its rows below, u_c = v_c,below - L21_c y_c), solves L11 y = v_own and hands up
// u = v_below - L21 y. Backward, root first: x_own = L11^-T (y - L21^T x_below), the rows below
// read from the solution. Contributions travel up the tree instead of being scattered into
// ancestors, so no two workgroups write one entry and no atomics are used.
//
// A front is solved by blocks of SNB = 128 columns, its factorization's panels, whose diagonal
// blocks' inverses the factorization keeps (column-major, ld = the block's width, zeros above
// the diagonal). A level is one launch forward and two backward (the products with the rows below
// first), or one more each way where it has many one-block fronts beside wider ones: a front's
// workgroups each take 128 of its rows (forward) or columns (backward) through its blocks in order,
// and the one that finishes the rows or columns of a block forms that block's solution. A block's
// solution formed elsewhere is waited for value by value: the values to come are marked PENDING, a
// signalling NaN that no arithmetic produces, before the launch; the forming workgroup writes each
// with a device-coherent atomic store and a waiting thread polls its own values until they are not
// PENDING (no fence: each value is its own signal). A workgroup waits only on workgroups of its own
// front placed earlier in the launch, so the waits resolve in dispatch order; every wait is bounded,
// and one that runs past `limit` polls sets *err and gives up (the host reports the solve as
// failed), so every wave exits.
//
// The products run on the FP64 matrix cores (16x16x4): 16 rows of L by 16 right-hand sides, the
// right-hand sides of an equation side by side in memory (entry k of side r at k nr + r), so that
// every entry of L is read once for all of them. One right-hand side uses one column of sixteen:
// 64 entries of L cost an MFMA either way, some 2.4e12 entries a second, above the 1.2e12 (FP32) that
// memory delivers, and each side's sums run in the same order however many are solved together: the
// same bits.
//
// Bound: the top levels' chains of blocks, each a wait, two 128 x 128 products and a publication: 5 us
// a block backward, 6 us forward (FP64, the 36^3 cube's root of 49 blocks), and below them the
// levels' launches. Measured against a launch a block on the vector units, with a launch of one workgroup
// a front to gather and one to start each level: 8 right-hand sides of the 20 x 23 x 17 hex8 block
// 2.78 -> 0.61 ms; a refined solve of 16 vectors on the mixed factor of the 13^3 tet10 block 25.0 ->
// 5.1 ms; one right-hand side of the 36^3 cube (one launch a level before, too) 3.60 -> 2.12 ms. One-block
// fronts with up to 512 rows below took their products in k_bwd itself at first, a launch less for
// many levels: 0.70, 5.5 and 2.23 ms (one workgroup a front is too few waves for its rows).
#pragma once

#include <type_traits>

#include "gemm_kernels.hpp"

namespace fc {

constexpr int SNB = 128;       // columns of a solve block (the factorization's panel width)
constexpr int SRHS = 16;       // right-hand sides of one product
constexpr int MAX_RHS = 64;    // right-hand sides one solve pass handles (the host splits larger blocks)
constexpr int STHREADS = 512;  // threads of a solve workgroup: eight waves of 16 rows or columns
// A block solution not yet formed: a signalling NaN, which no arithmetic result is.
constexpr uint64_t PENDING = 0x7FF0DEAD0000BEEFull;

__device__ __forceinline__ void publish(double* p, double v) {
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t peek(const double* p) {
  return __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The right-hand sides of a workgroup: `n` of them from `n0`, of `nr` side by side in memory (more than
// 16 NG of them run as groups side by side in the launch, group after group: their accumulators and
// the operands in flight would not fit the registers together).
struct Sides {
  int nr, n0, n;
};
template <int NG>
__device__ __forceinline__ Sides sides(int nr, int grp) {
  const int n0 = SRHS * NG * grp;
  return Sides{nr, n0, min(nr - n0, SRHS * NG)};
}

// The sides' values of pw equations from p on into rows 0 .. pw - 1 of V, zeros below them, once every
// one is published; all of a thread's loads in flight, then the missing ones again. Bounded
// (limit < 0: give up at once, a test's way in). Starts and ends on a barrier.
template <int NG>
__device__ __forceinline__ void await_block(double (*V)[SRHS * NG], const double* p, int pw, const Sides& sd,
                                            int64_t limit, int32_t* err) {
  constexpr int RS = STHREADS / SRHS, Q = SNB / RS * NG;  // thread: side tid % 16 (+ 16), every RS-th row
  const int c = threadIdx.x & (SRHS - 1), k0 = threadIdx.x / SRHS;
  p += sd.n0;
  __syncthreads();  // every read of the previous block done
  uint64_t b[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k = k0 + RS * (q / NG), n = c + SRHS * (q % NG);
    b[q] = k < pw && n < sd.n ? peek(p + (int64_t)k * sd.nr + n) : 0;
  }
  if (limit < 0) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int64_t tries = 0; limit >= 0; ++tries) {  // every missing value again, together
    bool miss = false;
#pragma unroll
    for (int q = 0; q < Q; ++q) miss = miss || b[q] == PENDING;
    if (!miss) break;
    if (tries >= limit ||
        ((tries & 255) == 255 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
      __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int k = k0 + RS * (q / NG), n = c + SRHS * (q % NG);
      if (b[q] == PENDING) b[q] = peek(p + (int64_t)k * sd.nr + n);
    }
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) V[k0 + RS * (q / NG)][c + SRHS * (q % NG)] = __builtin_bit_cast(double, b[q]);
  __syncthreads();
}

// A wave's 16 rows of values (output layout: entry v of a lane is row lane / 16 + 4 v of them, side
// 16 g + lane % 16) into rows row0 .. of V, rows from pw on as zeros.
template <int NG>
__device__ __forceinline__ void to_lds(double (*V)[SRHS * NG], const v4d (&val)[NG], int row0, int pw, int lane) {
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = row0 + (lane >> 4) + 4 * v;
      V[row][16 * g + (lane & 15)] = row < pw ? val[g][v] : 0.0;
    }
}

// Four consecutive entries of T at byte offset lane + off of a resource: two (FP64) or one 16-byte
// loads, or where `part` is set one load an entry, those from `valid` on reading 0. As they lie in
// memory, or converted to V.
template <typename T, typename V>
__device__ __forceinline__ void load4(V (&a)[4], __amdgpu_buffer_rsrc_t rs, uint32_t lane, uint32_t off, bool part,
                                      int valid) {
  typedef unsigned int u32x4 __attribute__((__vector_size__(16)));
  if (part) {
#pragma unroll
    for (int s = 0; s < 4; ++s) a[s] = (V)buf_load<T>(rs, s < valid ? lane + s * (uint32_t)sizeof(T) : 0x80000000u, off);
  } else if constexpr (sizeof(T) == 8) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(rs, lane + 16 * h, off, 0);
      a[2 * h] = __builtin_bit_cast(double, (uint64_t)w[0] | (uint64_t)w[1] << 32);
      a[2 * h + 1] = __builtin_bit_cast(double, (uint64_t)w[2] | (uint64_t)w[3] << 32);
    }
  } else {
    const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(rs, lane, off, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const unsigned e = w[s];  // (a bit cast of the vector's element itself reads element 0)
      a[s] = (V)__builtin_bit_cast(float, e);
    }
  }
}

// Rows p0 .. p0 + 15 of front F before its own solution: their entry of v (the front's own, in xp; marked
// PENDING afterwards where `mark` is set) and the children's contributions, in the output layout.
// Entries gptr[p] .. gptr[p + 1] of gsrc list the rows of u that land on front row p, child after child.
template <int NG>
__device__ __forceinline__ void gather_rows(v4d (&val)[NG], const FrontDev& F, int p0, const uint32_t* __restrict__ gptr,
                                            const uint32_t* __restrict__ gsrc, double* xp, const double* u,
                                            const Sides& sd, int lane, bool mark) {
  const int r = lane & 15, q = lane >> 4;
  const uint32_t* gp = gptr + F.rows_off;
  uint32_t a[4], e[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int p = p0 + q + 4 * v;
    a[v] = p < F.m ? gp[p] : 0;
    e[v] = p < F.m ? gp[p + 1] : 0;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const bool in = p < F.w && 16 * g + r < sd.n;
      double* x = xp + (int64_t)(F.col0 + p) * sd.nr + sd.n0 + 16 * g + r;
      val[g][v] = in ? *x : 0.0;
      if (mark && in) *reinterpret_cast<uint64_t*>(x) = PENDING;
    }
  }
  for (;;) {
    bool more = false;
    uint32_t s[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      more = more || a[v] < e[v];
      s[v] = a[v] < e[v] ? gsrc[a[v]] : 0;
    }
    if (!__any(more)) break;
    double add[NG][4];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int g = 0; g < NG; ++g)
        add[g][v] = (a[v] < e[v] && 16 * g + r < sd.n) ? u[(int64_t)s[v] * sd.nr + sd.n0 + 16 * g + r] : 0.0;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (a[v] < e[v]) {
#pragma unroll
        for (int g = 0; g < NG; ++g) val[g][v] += add[g][v];
        ++a[v];
      }
  }
}

// Forward, item (f, a = t): rows 128 t .. of front f. Rows start from gather_rows (the sums pull their
// terms, so that a front's rows are gathered by as many workgroups as it has row tiles) and lose L(rows, block) y_b for every
// block before them; tile t of block t then forms y_t = Inv_t v_t. In a front of one block every
// tile forms y_0 for itself from the block's rows: nothing is waited for. Rows below the front's
// columns end as its contribution u. A front of several blocks marks its own entries of xp PENDING
// (only their tile reads them) for the backward chain.
template <typename T, int NG>
__global__ __launch_bounds__(STHREADS) void k_fwd(const Item* __restrict__ items, const FrontDev* __restrict__ fronts,
                                                  const uint32_t* __restrict__ gptr, const uint32_t* __restrict__ gsrc,
                                                  const T* __restrict__ L, const T* __restrict__ Inv, double* xp,
                                                  double* y, double* u, const int64_t* __restrict__ uoff, int nr,
                                                  int nitems, int32_t* err, int64_t limit) {
  constexpr int KS = SNB / 4;
  constexpr uint32_t OUT = 0x80000000u;
  __shared__ double Ys[SNB][SRHS * NG];
  const int grp = blockIdx.x / nitems;
  const Item it = items[blockIdx.x - grp * nitems];
  const Sides sd = sides<NG>(nr, grp);
  const FrontDev F = fronts[it.f];
  const int t = it.a, w = F.w, m = F.m, nb = (w + SNB - 1) / SNB, r0 = t * SNB;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int last = min(t, nb);               // blocks whose y another workgroup forms (nb > 1)
  const bool single = nb == 1, own = t < nb;
  const int bf = own ? t : 0;                // the block this workgroup forms (own or single)
  const int cf = bf * SNB, pf = min(SNB, w - cf);
  const uint32_t ldb = (uint32_t)F.ld * sizeof(T);
  // the wave's rows i0 .. of block b, those before row `from` left out
  const int i0 = r0 + 16 * wave, i = i0 + r;
  auto fetch = [&](int b, int from, T (&lf)[KS]) {
    const int c0 = b * SNB, pw = min(SNB, w - c0);
    const auto rs = raw_rsrc(L + F.lpos + (int64_t)c0 * F.ld);
    const uint32_t lo = (i < m && i >= from) ? (uint32_t)i * sizeof(T) + q * ldb : OUT;
#pragma unroll
    for (int s = 0; s < KS; ++s) lf[s] = buf_load<T>(rs, 4 * s + q < pw ? lo : OUT, 4 * s * ldb);
  };
  auto fetch_inv = [&](T (&lf)[KS]) {
    const auto rs = raw_rsrc(Inv + F.inv0 + (int64_t)bf * SNB * SNB);
    const uint32_t pb = (uint32_t)pf * sizeof(T), lo = 16 * wave + r < pf ? (uint32_t)(16 * wave + r) * sizeof(T) + q * pb : OUT;
#pragma unroll
    for (int s = 0; s < KS; ++s) lf[s] = buf_load<T>(rs, 4 * s + q < pf ? lo : OUT, 4 * s * pb);
  };
  // p = lf Ys over the first kn columns (summed by itself: a block's products then leave the row's value
  // one rounding, not 128): a whole block with no test between the products (a test would make each
  // wait for its own LDS read), or by sixteen columns
  auto mul = [&](const T (&lf)[KS], v4d (&p)[NG], int kn) {
#pragma unroll
    for (int g = 0; g < NG; ++g) p[g] = v4d{0, 0, 0, 0};
    auto step = [&](int s) {
#pragma unroll
      for (int g = 0; g < NG; ++g) p[g] = Mma<double>::step((double)lf[s], Ys[4 * s + q][16 * g + r], p[g]);
    };
    if (kn == SNB) {
#pragma unroll
      for (int s = 0; s < KS; ++s) step(s);
    } else {
#pragma unroll
      for (int s0 = 0; s0 < KS; s0 += 4)
        if (4 * s0 < kn)
#pragma unroll
          for (int s = 0; s < 4; ++s) step(s0 + s);
    }
  };
  // the inverse before any wait; L's values of a block just before the wait for its y (further ahead,
  // the polls' answers would queue behind them: a wave's loads return in order)
  T inv[KS], cur[KS];
  if (own || single) fetch_inv(inv);
  v4d val[NG];
  gather_rows<NG>(val, F, i0, gptr, gsrc, xp, u, sd, lane, own && !single);
  if (!single)
    for (int b = 0; b < last; ++b) {
      fetch(b, 0, cur);
      const int pw = min(SNB, w - b * SNB);
      await_block<NG>(Ys, y + (int64_t)(F.col0 + b * SNB) * nr, pw, sd, limit, err);
      v4d p[NG];
      mul(cur, p, pw);
#pragma unroll
      for (int g = 0; g < NG; ++g) val[g] -= p[g];
    }
  if (own || single) {
    const bool rest = r0 + SNB > cf + pf && m > cf + pf;  // rows below the formed block (uniform)
    if (rest) fetch(bf, cf + pf, cur);
    v4d vb[NG];
    if (own) {
#pragma unroll
      for (int g = 0; g < NG; ++g) vb[g] = val[g];
    } else {
      gather_rows<NG>(vb, F, 16 * wave, gptr, gsrc, xp, u, sd, lane, false);
    }
    __syncthreads();  // the last block's reads of Ys done
    to_lds<NG>(Ys, vb, 16 * wave, pf, lane);
    __syncthreads();
    mul(inv, vb, min(16 * wave + 16, pf));  // Inv is zero above its diagonal
    if (own)
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * wave + q + 4 * v;
          if (row < pf && 16 * g + r < sd.n) publish(y + (int64_t)(F.col0 + cf + row) * nr + sd.n0 + 16 * g + r, vb[g][v]);
        }
    if (rest) {
      __syncthreads();  // every wave's reads of v done
      to_lds<NG>(Ys, vb, 16 * wave, pf, lane);
      __syncthreads();
      v4d p[NG];
      mul(cur, p, pf);
#pragma unroll
      for (int g = 0; g < NG; ++g) val[g] -= p[g];
    }
  }
  double* uf = u + uoff[it.f] * nr;
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int p = i0 + q + 4 * v;
      if (p >= w && p < m && 16 * g + r < sd.n) uf[(int64_t)(p - w) * nr + sd.n0 + 16 * g + r] = val[g][v];
    }
}

// acc[cb] += L21(:, j0 + 16 cb ..)^T x_below over the rows 16 it .. 16 it + 15, it = it0, it0 + step, ..
// of the front's rows below (x_below read from the solution by their columns' numbers). Lane
// (r, q) loads four consecutive rows of column r, so a wave's loads cover 16 consecutive rows of 16
// columns.
template <typename T, int NG, int CB, int BT>
__device__ __forceinline__ void below_products(v4d (&acc)[CB][NG], const FrontDev& F, const T* __restrict__ L,
                                               const int32_t* __restrict__ rows, const double* xp, const Sides& sd, int j0,
                                               int it0, int step, int lane) {
  const int r = lane & 15, q = lane >> 4, mu = F.m - F.w;
  const auto rs = raw_rsrc(L + F.lpos + (int64_t)j0 * F.ld + F.w);
  const int32_t* below = rows + F.rows_off + F.w;
  uint32_t lo[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
    lo[cb] = (uint32_t)(min(j0 + 16 * cb + r, F.w - 1) - j0) * F.ld * sizeof(T) + 4 * q * (uint32_t)sizeof(T);
  // BT steps of 16 rows at a time, every load of theirs in flight together; the next ones' column
  // numbers are read with them. In FP32 a lane's four by one load: an entry costs half the bytes there, so the
  // instructions beside it count (a load each in FP64: by one load its 8-side solve took 2 % longer).
  const auto ri = raw_rsrc(below);
  auto index = [&](int it, int (&ix)[BT][4]) {
#pragma unroll
    for (int t = 0; t < BT; ++t) {
      const int b = 16 * (it + t * step);
      if constexpr (sizeof(T) == 4) {
        float e[4];
        load4<float>(e, ri, 16 * q, (uint32_t)b * 4, b + 16 > mu, mu - b - 4 * q);
#pragma unroll
        for (int s = 0; s < 4; ++s) ix[t][s] = __builtin_bit_cast(int, e[s]);
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) ix[t][s] = below[min(b + 4 * q + s, mu - 1)];
      }
    }
  };
  if (16 * it0 >= mu) return;
  int ix[BT][4];
  index(it0, ix);
  for (int it = it0; 16 * it < mu; it += BT * step) {
    T a[BT][CB][4];
    double x[BT][NG][4];
#pragma unroll
    for (int t = 0; t < BT; ++t) {
      const int b = 16 * (it + t * step);
      if (b < mu) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int g = 0; g < NG; ++g)
            x[t][g][s] = (b + 4 * q + s < mu && 16 * g + r < sd.n) ? xp[(int64_t)ix[t][s] * sd.nr + sd.n0 + 16 * g + r] : 0.0;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) load4<T>(a[t][cb], rs, lo[cb], (uint32_t)b * sizeof(T), b + 16 > mu, mu - b - 4 * q);
      }
    }
    index(it + BT * step, ix);
#pragma unroll
    for (int t = 0; t < BT; ++t)
      if (16 * (it + t * step) < mu)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int g = 0; g < NG; ++g) acc[cb][g] = Mma<double>::step((double)a[t][cb][s], x[t][g][s], acc[cb][g]);
  }
}

// Backward, item (f, a = j0): z_j = y_j - L21(:, j)^T x_below for the columns j0 .. j0 + 16 CB - 1, in
// place in y. The eight waves share the rows; their sums are added in order. Bound: memory, through as
// many loads in flight as registers allow. FP32 holds its operands unconverted, and where a step loads two
// column blocks takes two steps at a time, not four: 86 registers leave a CU two workgroups. With
// four steps, converted operands (160 registers, one workgroup) and a load for each column number the
// launches of one side on the 80^3 hex8 factor took 5.4 ms, now 4.2; FP64 keeps four steps (two: 2 % slower
// with 8 sides).
template <typename T, int NG, int CB>
__global__ __launch_bounds__(STHREADS) void k_bwd_below(const Item* __restrict__ items,
                                                        const FrontDev* __restrict__ fronts, const T* __restrict__ L,
                                                        const int32_t* __restrict__ rows, const double* __restrict__ xp,
                                                        double* __restrict__ z, int nr, int nitems) {
  __shared__ double part[8][16 * CB][SRHS + 1];
  const int grp = blockIdx.x / nitems;
  const Item it = items[blockIdx.x - grp * nitems];
  const Sides sd = sides<NG>(nr, grp);
  const FrontDev F = fronts[it.f];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  v4d acc[CB][NG];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int g = 0; g < NG; ++g) acc[cb][g] = v4d{0, 0, 0, 0};
  below_products<T, NG, CB, (NG * CB > 2 || (sizeof(T) == 4 && CB > 1) ? 2 : 4)>(acc, F, L, rows, xp, sd, it.a, wave, 8, lane);
#pragma unroll
  for (int g = 0; g < NG; ++g) {
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int v = 0; v < 4; ++v) part[wave][16 * cb + q + 4 * v][r] = acc[cb][g][v];
    __syncthreads();
    for (int e = threadIdx.x; e < 256 * CB; e += STHREADS) {
      const int j = e / 16, n = e % 16;
      if (it.a + j < F.w && 16 * g + n < sd.n) {
        double s = part[0][j][n];
#pragma unroll
        for (int k = 1; k < 8; ++k) s += part[k][j][n];
        z[(int64_t)(F.col0 + it.a + j) * nr + sd.n0 + 16 * g + n] -= s;
      }
    }
    __syncthreads();
  }
}

// Backward, item (f, a = jb): the columns of block jb lose L(b, jb)^T x_b for every later block b, last
// first, then x_jb = Inv_jb^T z_jb. A front's items are in decreasing jb, so the workgroup forming a block's
// x precedes every one waiting for it.
template <typename T, int NG>
__global__ __launch_bounds__(STHREADS) void k_bwd(const Item* __restrict__ items, const FrontDev* __restrict__ fronts,
                                                  const T* __restrict__ L, const T* __restrict__ Inv,
                                                  const double* __restrict__ z, double* xp, int nr, int nitems,
                                                  int32_t* err, int64_t limit) {
  constexpr int KI = SNB / 16;  // steps of 16 rows
  __shared__ double Xs[SNB][SRHS * NG];
  const int grp = blockIdx.x / nitems;
  const Item it = items[blockIdx.x - grp * nitems];
  const Sides sd = sides<NG>(nr, grp);
  const FrontDev F = fronts[it.f];
  const int jb = it.a, j0 = jb * SNB, nb = (F.w + SNB - 1) / SNB, pw = min(SNB, F.w - j0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int jl = min(16 * wave + r, pw - 1);  // the lane's column as an operand (those past the block are not stored)
  double inv[KI][4];  // the block's inverse, loaded before any wait: nothing but x_jb's own products follows the last
  {
    const auto rs = raw_rsrc(Inv + F.inv0 + (int64_t)jb * SNB * SNB);
    const uint32_t lo = (uint32_t)(jl * pw + 4 * q) * sizeof(T);
#pragma unroll
    for (int k = 0; k < KI; ++k) load4<T>(inv[k], rs, lo, 16 * k * (uint32_t)sizeof(T), pw < SNB, pw - 16 * k - 4 * q);
  }
  v4d zv[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = 16 * wave + q + 4 * v;
      zv[g][v] = (j < pw && 16 * g + r < sd.n) ? z[(int64_t)(F.col0 + j0 + j) * nr + sd.n0 + 16 * g + r] : 0.0;
    }
  // four rows of KI steps of a column: block b of L, or the block's inverse
  auto fetch = [&](int b, double (&a)[KI][4]) {
    const int c0 = b * SNB, pb = min(SNB, F.w - c0);
    const auto rs = raw_rsrc(L + F.lpos + (int64_t)j0 * F.ld + c0);
    const uint32_t lo = ((uint32_t)jl * F.ld + 4 * q) * sizeof(T);
#pragma unroll
    for (int k = 0; k < KI; ++k) load4<T>(a[k], rs, lo, 16 * k * (uint32_t)sizeof(T), pb < SNB, pb - 16 * k - 4 * q);
  };
  auto mul = [&](const double (&a)[KI][4], v4d (&p)[NG], int k0, int kn) {  // p = a Xs (as k_fwd's)
#pragma unroll
    for (int g = 0; g < NG; ++g) p[g] = v4d{0, 0, 0, 0};
    auto step = [&](int k) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int g = 0; g < NG; ++g) p[g] = Mma<double>::step(a[k][s], Xs[16 * k + 4 * q + s][16 * g + r], p[g]);
    };
    if (k0 == 0 && kn == SNB) {  // no test between the products (as in k_fwd)
#pragma unroll
      for (int k = 0; k < KI; ++k) step(k);
    } else {
#pragma unroll
      for (int k = 0; k < KI; ++k)
        if (k >= k0 && 16 * k < kn) step(k);
    }
  };
  for (int b = nb - 1; b > jb; --b) {
    double a[KI][4];
    fetch(b, a);
    const int pb = min(SNB, F.w - b * SNB);
    await_block<NG>(Xs, xp + (int64_t)(F.col0 + b * SNB) * nr, pb, sd, limit, err);
    v4d p[NG];
    mul(a, p, 0, pb);
#pragma unroll
    for (int g = 0; g < NG; ++g) zv[g] -= p[g];
  }
  __syncthreads();  // the last block's reads of Xs done
  to_lds<NG>(Xs, zv, 16 * wave, pw, lane);
  __syncthreads();
  mul(inv, zv, wave, pw);  // Inv is zero above its diagonal
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = 16 * wave + q + 4 * v;
      if (j < pw && 16 * g + r < sd.n) publish(xp + (int64_t)(F.col0 + j0 + j) * nr + sd.n0 + 16 * g + r, zv[g][v]);
    }
}

// The same for fronts of one block, in levels of many of them: workgroups of four waves and few
// registers, so that a CU holds several (a level of 1 400 such fronts is bound by how many are in
// flight, not by one's products). KB steps of four columns in flight at a time.
constexpr int ONE_THREADS = 256;
constexpr int ONE_ROWS = 256;  // rows of a forward workgroup

// p = A V over kn columns: A's entry (the lane's row, column c) at lane offset lo + c cb of rs
// (lo past the resource: zeros).
template <typename T, int NG>
__device__ __forceinline__ void mul_stream(v4d (&p)[NG], __amdgpu_buffer_rsrc_t rs, uint32_t lo, uint32_t cb,
                                           const double (*V)[SRHS * NG], int kn, int lane) {
  constexpr int KB = 8;
  const int r = lane & 15, q = lane >> 4;
#pragma unroll
  for (int g = 0; g < NG; ++g) p[g] = v4d{0, 0, 0, 0};
  for (int k0 = 0; k0 < kn; k0 += 4 * KB) {
    T a[KB];
#pragma unroll
    for (int s = 0; s < KB; ++s) a[s] = buf_load<T>(rs, k0 + 4 * s + q < kn ? lo + q * cb : 0x80000000u, (k0 + 4 * s) * cb);
#pragma unroll
    for (int s = 0; s < KB; ++s)
      if (k0 + 4 * s < kn)
#pragma unroll
        for (int g = 0; g < NG; ++g)
          p[g] = Mma<double>::step((double)a[s], V[k0 + 4 * s + q][16 * g + r], p[g]);
  }
}

// Forward, item (f, a = first row, b = end): y_0 from the block's rows (every workgroup of the front forms
// it; the one of row 0 writes it), then the rows a .. b - 1 below the block.
template <typename T, int NG>
__global__ __launch_bounds__(ONE_THREADS) void k_fwd_one(const Item* __restrict__ items, const FrontDev* __restrict__ fronts,
                                                         const uint32_t* __restrict__ gptr,
                                                         const uint32_t* __restrict__ gsrc, const T* __restrict__ L,
                                                         const T* __restrict__ Inv, double* xp, double* __restrict__ y,
                                                         double* u, const int64_t* __restrict__ uoff, int nr, int nitems) {
  constexpr uint32_t OUT = 0x80000000u;
  __shared__ double Ys[SNB][SRHS * NG];
  const int grp = blockIdx.x / nitems;
  const Item it = items[blockIdx.x - grp * nitems];
  const Sides sd = sides<NG>(nr, grp);
  const FrontDev F = fronts[it.f];
  const int w = F.w, m = F.m;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const auto rs = raw_rsrc(L + F.lpos);
  double* uf = u + uoff[it.f] * nr;
  // the first rows below too, so that their gather's round trips overlap the block's
  const int p1 = max(it.a, w) + 16 * wave;
  v4d first[NG];
  for (int h = 16 * wave; h < w; h += 64) {
    v4d v[NG];
    gather_rows<NG>(v, F, h, gptr, gsrc, xp, u, sd, lane, false);
    to_lds<NG>(Ys, v, h, w, lane);
  }
  if (p1 < it.b) gather_rows<NG>(first, F, p1, gptr, gsrc, xp, u, sd, lane, false);
  __syncthreads();
  v4d yv[2][NG];
  {
    const auto rs = raw_rsrc(Inv + F.inv0);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int h = 16 * wave + 64 * c;
      if (h < w)
        mul_stream<T, NG>(yv[c], rs, h + r < w ? (uint32_t)(h + r) * sizeof(T) : OUT, (uint32_t)w * sizeof(T), Ys,
                                 min(h + 16, w), lane);
    }
  }
  __syncthreads();  // every read of v done
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int h = 16 * wave + 64 * c;
    if (h < w) {
      to_lds<NG>(Ys, yv[c], h, w, lane);
      if (it.a == 0)
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int row = h + q + 4 * v;
            if (row < w && 16 * g + r < sd.n) y[(int64_t)(F.col0 + row) * nr + sd.n0 + 16 * g + r] = yv[c][g][v];
          }
    }
  }
  __syncthreads();
  for (int p0 = p1; p0 < it.b; p0 += 64) {
    v4d val[NG];
    if (p0 == p1) {
#pragma unroll
      for (int g = 0; g < NG; ++g) val[g] = first[g];
    } else {
      gather_rows<NG>(val, F, p0, gptr, gsrc, xp, u, sd, lane, false);
    }
    v4d p[NG];
    mul_stream<T, NG>(p, rs, p0 + r < m ? (uint32_t)(p0 + r) * sizeof(T) : OUT, (uint32_t)F.ld * sizeof(T), Ys, w, lane);
#pragma unroll
    for (int g = 0; g < NG; ++g) val[g] -= p[g];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = p0 + q + 4 * v;
        if (i < it.b && 16 * g + r < sd.n) uf[(int64_t)(i - w) * nr + sd.n0 + 16 * g + r] = val[g][v];
      }
  }
}

// Backward, item (f): x = Inv^T z.
template <typename T, int NG>
__global__ __launch_bounds__(STHREADS, NG == 1 ? 4 : 2) void k_bwd_one(const Item* __restrict__ items,
                                                                       const FrontDev* __restrict__ fronts,
                                                                       const T* __restrict__ Inv,
                                                                       const double* __restrict__ z, double* xp, int nr,
                                                                       int nitems) {
  constexpr int KI = SNB / 16;
  __shared__ double Xs[SNB][SRHS * NG];
  const int grp = blockIdx.x / nitems;
  const Item it = items[blockIdx.x - grp * nitems];
  const Sides sd = sides<NG>(nr, grp);
  const FrontDev F = fronts[it.f];
  const int w = F.w, nc = (w + 15) / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int h = 16 * wave;
  v4d zv[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = h + q + 4 * v;
      zv[g][v] = (j < w && 16 * g + r < sd.n) ? z[(int64_t)(F.col0 + j) * nr + sd.n0 + 16 * g + r] : 0.0;
    }
  // the inverse's columns (zero above its diagonal: rows h on), in flight over the barrier
  T inv[KI][4];
  {
    const auto rs = raw_rsrc(Inv + F.inv0);
    const uint32_t lo = (uint32_t)(min(h + r, w - 1) * w + 4 * q) * sizeof(T);
#pragma unroll
    for (int k = 0; k < KI; ++k)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        inv[k][s] = buf_load<T>(rs, (16 * k >= h && 16 * k + 4 * q + s < w) ? lo + s * (uint32_t)sizeof(T) : 0x80000000u,
                                16 * k * (uint32_t)sizeof(T));
  }
  if (wave < nc) to_lds<NG>(Xs, zv, h, w, lane);
  __syncthreads();
  if (wave >= nc) return;
#pragma unroll
  for (int g = 0; g < NG; ++g) zv[g] = v4d{0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < KI; ++k)
    if (16 * k >= h && 16 * k < w)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int g = 0; g < NG; ++g)
          zv[g] = Mma<double>::step((double)inv[k][s], Xs[16 * k + 4 * q + s][16 * g + r], zv[g]);
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = h + q + 4 * v;
      if (j < w && 16 * g + r < sd.n) xp[(int64_t)(F.col0 + j) * nr + sd.n0 + 16 * g + r] = zv[g][v];
    }
}

// x[k nr + c] = b[c ldb + perm[k]] and y marked PENDING.
__global__ void k_solve_in(const double* __restrict__ b, double* __restrict__ x, double* __restrict__ y,
                           const int64_t* __restrict__ perm, int64_t n, int nr, int64_t ldb) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * nr; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = e / nr;
    x[e] = b[(e - k * nr) * ldb + perm[k]];
    reinterpret_cast<uint64_t*>(y)[e] = PENDING;
  }
}

// b[c ldb + perm[k]] = x[k nr + c].
__global__ void k_solve_out(const double* __restrict__ x, double* __restrict__ b, const int64_t* __restrict__ perm,
                            int64_t n, int nr, int64_t ldb) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * nr; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = e / nr;
    b[(e - k * nr) * ldb + perm[k]] = x[e];
  }
}

// ------------------------------------------------------------------------------------------
// Vector steps of refinement, FP64, on blocks of k <= MAX_RHS columns (column c at c * ld).
// Reductions are two-stage: each workgroup of a launch reduces one row block of one column
// (row blocks never straddle a segment of independent equations), and the host combines the
// partials in a fixed order, so results are the same on every run.

// Y = A X by rows (Csr::mul, sparse.rs:42-50): eight lanes per row, partial sums combined in a
// fixed order; columns in chunks of eight so a row's entries are read once per chunk.
__global__ __launch_bounds__(256) void k_spmm(int64_t n, const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                                              const double* __restrict__ val, const double* __restrict__ x,
                                              double* __restrict__ y, int k, int64_t ld) {
  const int sub = threadIdx.x & 7;
  for (int64_t r = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 3; r < n; r += ((int64_t)gridDim.x * blockDim.x) >> 3) {
    const int64_t t0 = ptr[r], t1 = ptr[r + 1];
    for (int c0 = 0; c0 < k; c0 += 8) {
      double s[8] = {};
      // The lane's entries t, t + 8, t + 16, t + 24 at a time: their values and columns, then
      // their x in every column of the chunk, all in flight together rather than each entry's
      // loads waited on in turn. Entries past the row read its last entry and add nothing; the
      // sums keep entry order. The chunk's column count is a constant of the sweep, so no
      // column takes a test of its own.
      auto sweep = [&](auto nc) {
        for (int64_t t = t0 + sub; t < t1; t += 32) {
          double v[4];
          int64_t j[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int64_t tt = min(t + 8 * u, t1 - 1);
            v[u] = val[tt];
            j[u] = idx[tt];
          }
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (q < decltype(nc)::value) {
              double xv[4];
#pragma unroll
              for (int u = 0; u < 4; ++u) xv[u] = x[(int64_t)(c0 + q) * ld + j[u]];
#pragma unroll
              for (int u = 0; u < 4; ++u) s[q] = t + 8 * u < t1 ? s[q] + v[u] * xv[u] : s[q];
            }
        }
      };
      switch (min(k - c0, 8)) {
        case 1: sweep(std::integral_constant<int, 1>{}); break;
        case 2: sweep(std::integral_constant<int, 2>{}); break;
        case 3: sweep(std::integral_constant<int, 3>{}); break;
        case 4: sweep(std::integral_constant<int, 4>{}); break;
        case 5: sweep(std::integral_constant<int, 5>{}); break;
        case 6: sweep(std::integral_constant<int, 6>{}); break;
        case 7: sweep(std::integral_constant<int, 7>{}); break;
        default: sweep(std::integral_constant<int, 8>{}); break;
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        s[q] += __shfl_xor(s[q], 1);
        s[q] += __shfl_xor(s[q], 2);
        s[q] += __shfl_xor(s[q], 4);
      }
      if (sub == 0)
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (c0 + q < k) y[(int64_t)(c0 + q) * ld + r] = s[q];
    }
  }
}

struct Coefs {
  double v[MAX_RHS];
};

// r = b - ax over n entries
__global__ void k_residual(int64_t n, const double* __restrict__ b, const double* __restrict__ ax,
                           double* __restrict__ r) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    r[i] = b[i] - ax[i];
}

// Y[:, c] += a_c X[:, c]
__global__ void k_axpy_cols(int64_t n, int k, int64_t ld, Coefs a, const double* __restrict__ x, double* __restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n * k; i += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(i / n);
    const int64_t e = (int64_t)c * ld + i % n;
    y[e] += a.v[c] * x[e];
  }
}

// Y[:, c] = X[:, c] + b_c Y[:, c]
__global__ void k_xpby_cols(int64_t n, int k, int64_t ld, const double* __restrict__ x, Coefs b, double* __restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n * k; i += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(i / n);
    const int64_t e = (int64_t)c * ld + i % n;
    y[e] = x[e] + b.v[c] * y[e];
  }
}

// partial[c * nblk + blk] = sum a*b (mode 0) or max |a| (mode 1) over rows [rb[blk], rb[blk + 1])
// of column c; grid (nblk, k)
__global__ __launch_bounds__(256) void k_reduce(const int64_t* __restrict__ rb, int nblk, const double* __restrict__ a,
                                                const double* __restrict__ b, int64_t ld, int mode,
                                                double* __restrict__ partial) {
  __shared__ double red[4];
  const int blk = blockIdx.x, c = blockIdx.y;
  const double* ac = a + (int64_t)c * ld;
  const double* bc = b + (int64_t)c * ld;
  double s = 0.0;
  for (int64_t i = rb[blk] + threadIdx.x; i < rb[blk + 1]; i += blockDim.x)
    s = mode == 0 ? s + ac[i] * bc[i] : fmax(s, fabs(ac[i]));
  for (int o = 32; o > 0; o >>= 1) {
    const double t = __shfl_xor(s, o);
    s = mode == 0 ? s + t : fmax(s, t);
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = red[0];
    for (int w = 1; w < 4; ++w) t = mode == 0 ? t + red[w] : fmax(t, red[w]);
    partial[(int64_t)c * nblk + blk] = t;
  }
}

}  // namespace fc
