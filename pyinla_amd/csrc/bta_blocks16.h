// 16x16 blocks of a 64x64 tile dealt over the waves of a workgroup, for the
// kernels that hold a whole block (b <= 64) in LDS.
#pragma once
#include "bta_tile_chol.h"

namespace bta {

// A 16x16 block of a row-major global matrix (accumulator layout); elements
// outside rows x cols are zero / not stored.
__device__ __forceinline__ f64x4 gload16(const double* g, int ld, int r0, int c0, int rows, int cols) {
  const int lane = threadIdx.x & 63, c = c0 + (lane & 15);
  f64x4 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = r0 + 4 * q + (lane >> 4);
    v[q] = (r < rows && c < cols) ? gview(g)[(int64_t)r * ld + c] : 0.0;
  }
  return v;
}
// The first 16x16 block, its upper triangle from the lower one.
__device__ __forceinline__ f64x4 gload16_sym(const double* g, int ld, int rows) {
  const int lane = threadIdx.x & 63, j = lane & 15;
  f64x4 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = 4 * q + (lane >> 4), r = max(i, j), c = min(i, j);
    v[q] = r < rows ? gview(g)[(int64_t)r * ld + c] : 0.0;
  }
  return v;
}
__device__ __forceinline__ void gstore16(double* g, int ld, int r0, int c0, int rows, int cols, f64x4 v) {
  const int lane = threadIdx.x & 63, c = c0 + (lane & 15);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = r0 + 4 * q + (lane >> 4);
    if (r < rows && c < cols) gview(g)[(int64_t)r * ld + c] = v[q];
  }
}

// Up to U 16x16 blocks of one of W waves: block u is (row[u], col[u]); n of them.
template <int U, int W = 4>
struct Blocks {
  f64x4 v[U];
  int row[U], col[U], n;
  // the wave's share of a lower triangle of m block rows, or of m x c blocks,
  // dealt one by one over the last `waves` waves, starting `first` after the
  // first of them, block number `skip` the first to go
  __device__ __forceinline__ void deal(int m, int c, bool lower, int first, int waves = W, int skip = 0) {
    const int me = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) - (W - waves);
    const int at = me - first < 0 ? me - first + waves : me - first, total = lower ? m * (m + 1) / 2 : m * c;
    n = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = skip + at + waves * u;
      int r = 0, k = e;
      while (k >= (lower ? r + 1 : max(c, 1))) {
        k -= lower ? r + 1 : c;
        if (++r >= 4) break;
      }
      row[u] = 16 * r;
      col[u] = 16 * k;
      n += me >= 0 && e < total;
    }
  }
  __device__ __forceinline__ void load(const double* g, int ld, int rows, int cols) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < n) v[u] = gload16(g, ld, row[u], col[u], rows, cols);
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = f64x4{0.0, 0.0, 0.0, 0.0};
  }
  // one 16-wide K block of v -= or += op(X) op(Y) (forms as of mma16x16); TRI:
  // Y is lower triangular
  template <bool NEG, int TY, int TX, bool TRI = false>
  __device__ __forceinline__ void product(const double* X, const double* Y, int k) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < n && (!TRI || k <= col[u])) v[u] = mma16x16<NEG, TY, TX>(X, row[u], k, Y, col[u], k, v[u]);
  }
  __device__ __forceinline__ void to_lds(double* s) const {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < n) store16(s, row[u], col[u], v[u]);
  }
  // blocks of a lower triangle and their mirror images, the matrix exactly
  // symmetric: element (r, c), r >= c, goes to both places
  __device__ __forceinline__ void store_sym(double* s, double* g, int ld, int rows) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < n)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = row[u] + 4 * q + (lane >> 4), c = col[u] + (lane & 15);
          if (r < c) continue;
          s[r * BTA_LDS_LD + c] = v[u][q];
          s[c * BTA_LDS_LD + r] = v[u][q];
          if (r < rows && c < rows) {
            gview(g)[(int64_t)r * ld + c] = v[u][q];
            gview(g)[(int64_t)c * ld + r] = v[u][q];
          }
        }
  }
  __device__ __forceinline__ void store(double* g, int ld, int rows, int cols) const {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < n) gstore16(g, ld, row[u], col[u], rows, cols, v[u]);
  }
};

}  // namespace bta
