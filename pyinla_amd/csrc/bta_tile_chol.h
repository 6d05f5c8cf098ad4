// In-workgroup Cholesky factorisation and inverse of one 64x64 FP64 tile.
//
// The tile is 4 x 4 blocks of 16; A (-> L) and E (-> L^-1) live in LDS.  For
// each block column j:
//   phase 1: wave 0 applies the update of block column j-1 to the diagonal
//            block, A_jj -= L_j,j-1 L_j,j-1^T (the one trailing update on the
//            critical path), then factors and inverts A_jj in registers
//            (chol16_inv16 below); meanwhile waves 1..3 apply the remaining
//            trailing updates of block column j-1, A_ik -= L_i,j-1 L_k,j-1^T
//            (j <= k <= i, (i, k) != (j, j)), and form
//            T_jk = sum_{m=k}^{j-1} L_jm E_mk for the inverse row j (k < j);
//   phase 2: the blocks below the diagonal, L_ij = A_ij E_jj^T (i > j; wave 0
//            takes i = j+1, whose update it applies at the start of the next
//            phase 1), and the inverse blocks E_jk = -E_jj T_jk (k < j):
//            always three 16x16 products.
// Two barriers per block column; every off-diagonal product is a 16x16x16
// FP64 MFMA product (4 v_mfma_f64_16x16x4f64) on LDS operands.  For a full
// tile the strict upper blocks of A and E are cleared by waves 1..3 during
// the first factorization (nothing else touches them); a partial tile (valid
// block mv < 64) is set to the identity outside the valid block first.
// What bounds it is the chain of 64 pivots.  Measured on MI355X, cycles of one
// tile (s_memtime): 8-wide panels 48 k; this blocking with v_readlane broadcasts
// in the 16x16 factorization and three barriers per block column 32 k; two
// barriers and the 16x16 block by column (one row broadcast and two FMAs per row
// and pivot) 24 k.  With the 16x16 block in four panels of 4, each lane repeating
// the 4x4 pivot block and one MFMA per panel for the rows below (chol16_panel), a
// kernel that factors one tile takes 14.6 us instead of 19.1.  A partial tile
// factors only the block columns it has: a block's panel at b = 92 37.3 -> 33.8
// us, at b = 400 105 -> 99.
#pragma once
#include "bta_device.h"

// 1/sqrt(x): the hardware estimate y (relative error below 2^-22) and one step
// of third order, y (1 + e/2 + 3 e^2 / 8) with e = 1 - x y^2 (the next term is
// below 2^-66).  A non-positive pivot propagates as NaN and is reported by the
// caller.
__device__ __forceinline__ double rsq_f64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

struct TileCholResult {
  double logsum;  // sum of log(pivot) over the valid part (thread 0 only)
  int fail;       // first non-positive / NaN pivot in the valid part, or -1 (thread 0 only)
};

__device__ __forceinline__ f64x4 load16(const double* __restrict__ C, int r0, int c0) {
  const int lane = threadIdx.x & 63;
  f64x4 v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = C[(r0 + 4 * r + (lane >> 4)) * BTA_LDS_LD + c0 + (lane & 15)];
  return v;
}

__device__ __forceinline__ void store16(double* __restrict__ C, int r0, int c0, f64x4 v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < 4; ++r) C[(r0 + 4 * r + (lane >> 4)) * BTA_LDS_LD + c0 + (lane & 15)] = v[r];
}

// Store the lower triangle (i >= j) of a 16x16 tile (all of it off the diagonal).
__device__ __forceinline__ void store16_lower(double* __restrict__ C, int r0, int c0, f64x4 v) {
  const int lane = threadIdx.x & 63;
  const int j = c0 + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = r0 + 4 * r + (lane >> 4);
    if (j <= i) C[i * BTA_LDS_LD + j] = v[r];
  }
}

// acc +/-= op(X) * op(Y), K = 16, LDS stride BTA_LDS_LD.  X rows rx.., K cols
// kx.. (TX == 0) or its transpose, rows kx.. (K), cols rx.. (TX == 1); Y in NT
// form (TY == 0: rows ry.., K cols ky..) or NN form (TY == 1: rows ky.. (K),
// cols ry..).
template <bool NEG, int TY, int TX = 0>
__device__ __forceinline__ f64x4 mma16x16(const double* __restrict__ X, int rx, int kx, const double* __restrict__ Y,
                                          int ry, int ky, f64x4 acc) {
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  double a[4], b[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    a[k] = TX == 0 ? X[(rx + li) * BTA_LDS_LD + kx + 4 * k + lk] : X[(kx + 4 * k + lk) * BTA_LDS_LD + rx + li];
    b[k] = TY == 0 ? Y[(ry + li) * BTA_LDS_LD + ky + 4 * k + lk] : Y[(ky + 4 * k + lk) * BTA_LDS_LD + ry + li];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) acc = NEG ? mfma_f64_nega(a[k], b[k], acc) : mfma_f64(a[k], b[k], acc);
  return acc;
}

// v moved from lane P of its 16-lane row to every lane of that row (DPP
// row_newbcast, a single 64-bit move on gfx950).
template <int P>
__device__ __forceinline__ double bcast_row16(double v) {
  return __longlong_as_double(__builtin_amdgcn_mov_dpp(__double_as_longlong(v), 0x150 + P, 0xf, 0xf, true));
}

// x[r] = v of the lane with the same lane % 16 in 16-lane row r: swapping the
// odd rows of one register with the even rows of another (v_permlane16_swap),
// then the halves (v_permlane32_swap), spreads each row over all four.
__device__ __forceinline__ void gather_rows(double v, double (&x)[4]) {
  const long long b = __double_as_longlong(v);
  const unsigned w[2] = {(unsigned)b, (unsigned)(b >> 32)};
  unsigned g[4][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const auto t = __builtin_amdgcn_permlane16_swap(w[h], w[h], false, false);  // rows 0 0 2 2 | 1 1 3 3
    const auto e = __builtin_amdgcn_permlane32_swap(t[0], t[0], false, false);
    const auto o = __builtin_amdgcn_permlane32_swap(t[1], t[1], false, false);
    g[0][h] = e[0];
    g[1][h] = o[0];
    g[2][h] = e[1];
    g[3][h] = o[1];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) x[r] = __longlong_as_double(((long long)g[r][1] << 32) | g[r][0]);
}

// Rows 4P .. 4P+3 of a 16x16 Cholesky with inverse, and recursively the ones
// after them.  a and e are in the MFMA accumulator layout (element q of lane
// j + 16 r is row 4q + r, column j); a holds the symmetric trailing matrix, e
// starts as the identity.  Every lane factors the 4x4 pivot block S = C C^T
// (its entries come by row broadcasts) and solves C v = A[4P.., j] and
// C u = E[4P.., j] for its column: v is column block P of L (v_r of lane j is
// L[j][4P+r]), u is rows 4P.. of L^-1.  One MFMA each then applies
// A -= L_P L_P^T and E -= L_P u to the rows below (the rows up to 4P+3, which
// it also touches, keep their old registers).  Finished columns compute
// values that nothing reads.
template <int P>
__device__ __forceinline__ void chol16_panel(f64x4& a, f64x4& e) {
  const int r = (threadIdx.x & 63) >> 4;
  double x[4], u[4];
  gather_rows(a[P], x);
  const double s00 = bcast_row16<4 * P>(x[0]), s10 = bcast_row16<4 * P>(x[1]), s20 = bcast_row16<4 * P>(x[2]),
               s30 = bcast_row16<4 * P>(x[3]), s11 = bcast_row16<4 * P + 1>(x[1]),
               s21 = bcast_row16<4 * P + 1>(x[2]), s31 = bcast_row16<4 * P + 1>(x[3]),
               s22 = bcast_row16<4 * P + 2>(x[2]), s32 = bcast_row16<4 * P + 2>(x[3]),
               s33 = bcast_row16<4 * P + 3>(x[3]);
  gather_rows(e[P], u);
  const double r0 = rsq_f64(s00);
  const double l10 = s10 * r0, l20 = s20 * r0, l30 = s30 * r0;
  const double r1 = rsq_f64(fma(-l10, l10, s11));
  const double l21 = fma(-l20, l10, s21) * r1, l31 = fma(-l30, l10, s31) * r1;
  const double r2 = rsq_f64(fma(-l21, l21, fma(-l20, l20, s22)));
  const double l32 = fma(-l31, l21, fma(-l30, l20, s32)) * r2;
  const double r3 = rsq_f64(fma(-l32, l32, fma(-l31, l31, fma(-l30, l30, s33))));
  auto solve = [&](double (&y)[4]) {
    y[0] *= r0;
    y[1] = fma(-l10, y[0], y[1]) * r1;
    y[2] = fma(-l21, y[1], fma(-l20, y[0], y[2])) * r2;
    y[3] = fma(-l32, y[2], fma(-l31, y[1], fma(-l30, y[0], y[3]))) * r3;
  };
  solve(x);
  solve(u);
  const double v = r < 2 ? (r == 0 ? x[0] : x[1]) : (r == 2 ? x[2] : x[3]);
  const double y = r < 2 ? (r == 0 ? u[0] : u[1]) : (r == 2 ? u[2] : u[3]);
  if constexpr (P < 3) {
    f64x4 a2 = mfma_f64_nega(v, v, a);
    f64x4 e2 = mfma_f64_nega(v, y, e);
#pragma unroll
    for (int q = P + 1; q < 4; ++q) {
      a[q] = a2[q];
      e[q] = e2[q];
    }
  }
  a[P] = v;
  e[P] = y;
  if constexpr (P < 3) chol16_panel<P + 1>(a, e);
}

// 16x16 Cholesky and inverse by one wave: a (symmetric, accumulator layout)
// becomes L^T's rows and e the inverse's, as store_chol16 expects them.  A
// non-positive pivot leaves NaN on the diagonal of L from there on.
__device__ __forceinline__ void chol16_inv16(f64x4& a, f64x4& e) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < 4; ++q) e[q] = (4 * q + (lane >> 4) == (lane & 15)) ? 1.0 : 0.0;
  chol16_panel<0>(a, e);
}

// L (zero strict upper) to s and L^-1 to w, at block (r0, r0).
__device__ __forceinline__ void store_chol16(f64x4 a, f64x4 e, double* __restrict__ s, double* __restrict__ w, int r0) {
  const int lane = threadIdx.x & 63;
  const int j = lane & 15, r = lane >> 4;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    s[(r0 + j) * BTA_LDS_LD + r0 + 4 * q + r] = (j >= 4 * q + r) ? a[q] : 0.0;
    w[(r0 + 4 * q + r) * BTA_LDS_LD + r0 + j] = e[q];
  }
}

// The lower triangle of the 16x16 block at (r0, r0), mirrored.
__device__ __forceinline__ f64x4 load16_sym(const double* __restrict__ C, int r0) {
  const int lane = threadIdx.x & 63;
  const int j = lane & 15;
  f64x4 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = 4 * q + (lane >> 4);
    v[q] = C[(r0 + max(i, j)) * BTA_LDS_LD + r0 + min(i, j)];
  }
  return v;
}

// Zeros of the strict upper 16x16 blocks of a full tile's s and w, by threads
// t of nt.
__device__ __forceinline__ void clear_upper_blocks(double* __restrict__ s, double* __restrict__ w, int t, int nt) {
  for (int e = t; e < 6 * 256; e += nt) {  // (0,1) (0,2) (0,3) (1,2) (1,3) (2,3)
    const int blk = e >> 8, q = e & 255;
    const int bi = blk < 3 ? 0 : (blk < 5 ? 1 : 2);
    const int bk = blk < 3 ? blk + 1 : (blk < 5 ? blk - 1 : 3);
    const int idx = (16 * bi + (q >> 4)) * BTA_LDS_LD + 16 * bk + (q & 15);
    s[idx] = 0.0;
    w[idx] = 0.0;
  }
}

// The block columns of a tile in LDS; with FIRST the first one's diagonal block
// is already factored (L_00 in s, E_00 in w, a full tile's upper blocks clear).
// `spare` is run by wave 3 beside the last 16x16 factorization.  nblk: block
// columns to factor (a padded tile's last ones are the identity already).
template <bool FIRST, class F>
__device__ __forceinline__ void tile_chol_blocks(double* __restrict__ s, double* __restrict__ w, int mv, F&& spare,
                                                 int nblk = 4) {
  const int tid = threadIdx.x;
  const int wv = tid >> 6;
#pragma unroll 1
  for (int jb = 0; jb < nblk; ++jb) {
    const int r0 = 16 * jb;
    if (!FIRST || jb > 0) {
      // ---- phase 1
      if (wv == 0) {
        f64x4 acc = load16_sym(s, r0), e;
        if (jb > 0) acc = mma16x16<true, 0>(s, r0, r0 - 16, s, r0, r0 - 16, acc);
        chol16_inv16(acc, e);
        store_chol16(acc, e, s, w, r0);
      } else if (jb == 0) {
        if (mv == 64) clear_upper_blocks(s, w, tid - 64, BTA_THREADS - 64);
      } else {
        // trailing tiles of block column jb-1 other than (jb, jb), then the T_jk
        const int nr = nblk - jb, nl = nr * (nr + 1) / 2 - 1;
        for (int t = wv - 1; t < nl + jb; t += 3) {
          if (t < nl) {
            int rr = 0, cc = t + 1;  // lower-triangle tile t+1 of the trailing block, row-major
            while (cc > rr) {
              cc -= rr + 1;
              ++rr;
            }
            const int ib = jb + rr, kb = jb + cc;
            f64x4 acc = load16(s, 16 * ib, 16 * kb);
            acc = mma16x16<true, 0>(s, 16 * ib, r0 - 16, s, 16 * kb, r0 - 16, acc);
            if (ib == kb) store16_lower(s, 16 * ib, 16 * kb, acc);
            else store16(s, 16 * ib, 16 * kb, acc);
          } else {
            const int k = t - nl;
            f64x4 acc = f64x4{0.0, 0.0, 0.0, 0.0};
            for (int m = k; m < jb; ++m) acc = mma16x16<false, 1>(s, r0, 16 * m, w, 16 * k, 16 * m, acc);
            store16(w, r0, 16 * k, acc);
          }
        }
        if (jb == nblk - 1 && wv == 3) spare();
      }
      lds_barrier();
    }
    // ---- phase 2: product q < nd is L_(jb+1+q),jb, the others E_jb,(q - nd)
    {
      const int nd = nblk - 1 - jb, q = nd > 0 ? wv : wv - 1;
      if (q >= 0 && q < nblk - 1) {
        f64x4 acc = f64x4{0.0, 0.0, 0.0, 0.0};
        if (q < nd) {
          const int ib = jb + 1 + q;
          acc = mma16x16<false, 0>(s, 16 * ib, r0, w, r0, r0, acc);  // A_ib,jb E_jj^T
          store16(s, 16 * ib, r0, acc);
        } else {
          const int k = q - nd;
          acc = mma16x16<true, 1>(w, r0, r0, w, 16 * k, r0, acc);    // -E_jj T_jk
          store16(w, r0, 16 * k, acc);
        }
      }
    }
    lds_barrier();
  }
}

// Identity outside the valid block, in s and E alike, zero strict upper
// triangle, E = 0 inside.
__device__ __forceinline__ void tile_chol_pad(double* __restrict__ s, double* __restrict__ w, int mv) {
  for (int e = threadIdx.x; e < 64 * 64; e += BTA_THREADS) {
    const int i = e >> 6, j = e & 63;
    if (i >= mv || j >= mv || j > i) s[i * BTA_LDS_LD + j] = (i == j) ? 1.0 : 0.0;
    w[i * BTA_LDS_LD + j] = (i == j && i >= mv) ? 1.0 : 0.0;
  }
}

// By one wave, lane i holding l_ii: the sum of log pivots (log d_i = 2 log l_ii)
// by a fixed butterfly (deterministic order), and the first non-positive pivot.
__device__ __forceinline__ TileCholResult tile_log_pivots(double lii, int mv) {
  const int lane = threadIdx.x & 63;
  TileCholResult res;
  const unsigned long long bad = __ballot(lane < mv && !(lii > 0.0));
  res.fail = bad ? __ffsll((long long)bad) - 1 : -1;
  double v = (lane < mv) ? 2.0 * log(lii) : 0.0;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  res.logsum = v;
  return res;
}

// The same for the factored tile in s, by wave 0 (thread 0 gets the result).
__device__ __forceinline__ TileCholResult tile_chol_result(const double* __restrict__ s, int mv) {
  const int lane = threadIdx.x & 63;
  if ((threadIdx.x >> 6) == 0) return tile_log_pivots(s[lane * BTA_LDS_LD + lane], mv);
  return TileCholResult{0.0, -1};
}

// s: 64x64 LDS tile (stride BTA_LDS_LD) holding the SPD matrix in its lower
// triangle (upper triangle ignored); rows / cols >= mv are treated as
// identity.  On exit s holds L (zero strict upper) and w holds L^-1 (zero
// strict upper), both with stride BTA_LDS_LD.  (tile_chol_result reads the log
// pivots off s: apart, so that whoever waits for the inverse does not wait for
// the logarithms.)
__device__ __forceinline__ void tile_chol_inv(double* __restrict__ s, double* __restrict__ w, int mv) {
  if (mv < 64) {
    tile_chol_pad(s, w, mv);
    __syncthreads();
  }
  tile_chol_blocks<false>(s, w, mv, [] {}, (mv + 15) / 16);
}
