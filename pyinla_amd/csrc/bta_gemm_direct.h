// Grouped FP64 GEMM without LDS staging: every wave loads its MFMA operands
// straight from global memory into registers, S steps of K = 8 ahead, and
// waits for nobody else.  Included by bta_gemm.hip (job search, tile order and
// the rule that chooses between the kernels are there).
//
// What bounds it: full launches the matrix cores (64 x 64 tiles, one wave per
// tile: NN 2000^3 293 -> 262 us, 54 -> 61 TFLOP/s, against k_gemm_grouped,
// whose waves stage K chunks through LDS between two barriers); launches that
// leave CUs idle the latency of one tile, so that these take 32 x 32 tiles and
// four waves that share K (417^3 31 -> 12 us, 92^3 10.7 -> 7.3 us, 800^3 54 ->
// 35 us).  The operands a CU's waves read take 16 (64 x 64) or 32 bytes per
// clock at the matrix cores' rate.  32 x 32 tiles with both operands K-contiguous are the exception:
// a step takes half of each line, and the other half is gone before its turn.
#pragma once
#include "bta_gemm.h"

namespace bta {

// 16 bytes at 8-byte alignment (odd leading dimensions)
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));
typedef __attribute__((address_space(1))) f64x2u gf64x2u;
typedef __attribute__((address_space(1))) char gchar;

// One operand of a wave: 32 * NX rows (op(A) rows or op(B) columns) times the
// 8 K of a step, as NX * 2 pair loads per lane (lane = li + 16 g):
//   form 0, K contiguous in memory (A untransposed, B transposed):
//     pair q of group X is row 32 X + 2 li + q, K 2 g and 2 g + 1
//   form 1, rows contiguous:
//     pair q of group X is K 2 g + q, rows 32 X + 2 li and 2 li + 1
// Either way element (x, p) -- row 32 X + 2 li + x, K 2 g + p -- feeds the
// MFMA of row half x and K half p, so the two forms differ by one swap and
// segments of different forms add into the same accumulator.
template <int NX>
struct DirectOp {
  const char* base;     // tile origin at K = 0, less PAIR bytes
  uint32_t off[NX][2];  // byte offsets of the pairs of the step at K = 0, from base
  uint32_t kstep;       // bytes per K
  int form, K;
  bool narrow;  // a single row (form 1) or K (form 0): elements are loaded one by one
  static constexpr int PAIR = 16;
  // rows: valid rows of the operand in the tile.  Rows past the end repeat the
  // last ones (they feed outputs that are not stored).
  __device__ __forceinline__ void init(const double* g0, int ld, int form_, int rows, int K_) {
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    base = reinterpret_cast<const char*>(g0) - PAIR;
    form = form_;
    K = K_;
    kstep = form ? (uint32_t)ld * 8u : 8u;
    narrow = (form ? rows : K) < 2;
#pragma unroll
    for (int X = 0; X < NX; ++X)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int r = 32 * X + 2 * li;
        off[X][q] = PAIR + (form ? ((uint32_t)(2 * g + q) * (uint32_t)ld + (uint32_t)max(min(r, rows - 2), 0)) * 8u
                                 : ((uint32_t)min(r + q, rows - 1) * (uint32_t)ld + (narrow ? 0u : 2u * (uint32_t)g)) * 8u);
      }
  }
  // The step at k, inside K: scalar base plus the lanes' offsets.
  __device__ __forceinline__ void load(f64x2 (&v)[NX][2], int k) const {
    const gchar* bk = (const gchar*)(base + (int64_t)k * kstep);
#pragma unroll
    for (int X = 0; X < NX; ++X)
#pragma unroll
      for (int q = 0; q < 2; ++q) v[X][q] = *(const gf64x2u*)(bk + off[X][q]);
  }
  // Any step with k < K: pairs past the end of K are moved back to its last
  // ones (no load leaves the operand); fix undoes the move.
  __device__ __forceinline__ void load_edge(f64x2 (&v)[NX][2], int k) const {
    const gchar* bk = (const gchar*)(base + (int64_t)k * kstep);
    uint32_t dq[2] = {0, 0};
    if (k + 8 > K) {
      const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int kk = form ? k + 2 * g + q : k + 2 * g;
        if (form || !narrow) dq[q] = (uint32_t)(min(kk, form ? K - 1 : K - 2) - kk) * kstep;
      }
    }
    if (narrow) {
#pragma unroll
      for (int X = 0; X < NX; ++X)
#pragma unroll
        for (int q = 0; q < 2; ++q) v[X][q] = f64x2{*(const gdouble*)(bk + (off[X][q] + dq[q])), 0.0};
    } else {
#pragma unroll
      for (int X = 0; X < NX; ++X)
#pragma unroll
        for (int q = 0; q < 2; ++q) v[X][q] = *(const gf64x2u*)(bk + (off[X][q] + dq[q]));
    }
  }
  // element (x, p) of group X
  __device__ __forceinline__ static void frag(const f64x2 (&v)[NX][2], double (&e)[NX][2][2], int form) {
#pragma unroll
    for (int X = 0; X < NX; ++X) {
      e[X][0][0] = v[X][0].x;
      e[X][1][1] = v[X][1].y;
      e[X][0][1] = form ? v[X][1].x : v[X][0].y;
      e[X][1][0] = form ? v[X][0].y : v[X][1].x;
    }
  }
  // In place, the corrections of a step at an edge, each under a uniform test:
  // pairs that init or load_edge moved back, K past ke, masked elements (i0:
  // index of the tile's first row in the operand).
  __device__ __forceinline__ static void fix(f64x2 (&v)[NX][2], int form, int rows, int k, int K, int ke, int mask,
                                             int i0, bool odd) {
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int kl = k + 2 * g;  // K of p = 0
    if (odd || (!form && k + 8 > K && K > 1)) {
#pragma unroll
      for (int X = 0; X < NX; ++X) {
        const bool moved = form ? 32 * X + 2 * li > rows - 2 : kl > K - 2;
#pragma unroll
        for (int q = 0; q < 2; ++q) v[X][q].x = moved ? v[X][q].y : v[X][q].x;
      }
    }
    if (k + 8 > ke) {
#pragma unroll
      for (int X = 0; X < NX; ++X)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          if (kl + (form ? q : 0) >= ke) v[X][q].x = 0.0;
          if (kl + (form ? q : 1) >= ke) v[X][q].y = 0.0;
        }
    }
    mask = chunk_mask(mask, i0, 32 * NX, k, 8);
    if (mask != MASK_NONE) {
      const int s = mask == MASK_K_LT_I ? 1 : -1;  // kept: s (K - row) >= 0
#pragma unroll
      for (int X = 0; X < NX; ++X) {
        const int d = s * (kl - (i0 + 32 * X + 2 * li));
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int dq = form ? d + s * q : d - s * q;  // element .x, and .y one row (form 1) or K (form 0) on
          const int dy = form ? dq - s : dq + s;
          if (dq < 0) v[X][q].x = 0.0;
          if (dy < 0) v[X][q].y = 0.0;
        }
      }
    }
  }
};

// by value: a conditional between the members themselves would select their
// addresses and put the descriptors into scratch memory
template <class T>
__device__ __forceinline__ T pick3(int q, T a, T b, T c) {
  return q == 0 ? a : (q == 1 ? b : c);
}

// Output tiles of 32 NX x 32 NX, K in WK parts, one wave each; S steps of K = 8
// in registers, OCC waves per SIMD the register budget is cut for.
template <int NX, int WK, int S, int OCC>
__global__ void __launch_bounds__(64 * WK, OCC)
    k_gemm_direct(const GemmJob* __restrict__ jobs, const int* __restrict__ prefix, int njobs) {
  constexpr int TS = 32 * NX;
  const int jid = find_job(prefix, njobs, blockIdx.x);
  const GemmJob& g = jobs[jid];
  // the whole descriptor at once: read piece by piece, each piece would add a
  // memory latency ahead of the first operand load
  const GemmSeg s0 = g.seg[0], s1 = g.seg[1], s2 = g.seg[2];
  const int nseg = g.nseg, lower = g.lower, mirror = g.mirror, m = g.m, n = g.n, ldc = g.ldc;
  const double beta = g.beta;
  gdouble* C = gview(g.C);
#define BTA_SEG(f, sid) pick3(sid, s0.f, s1.f, s2.f)
  const int local = blockIdx.x - prefix[jid];
  int tr, tc;
  const int tm = (m + TS - 1) / TS, tn = (n + TS - 1) / TS;
  if (lower) decode_lower(s0.tri ? local : xcd_share(local, tm * (tm + 1) / 2), tr, tc);
  else xcd_tile(local, tm, tn, s0.tri, tr, tc);
  const int r0 = (tr * TS + TS > m && m >= TS) ? m - TS : tr * TS;
  const int c0 = (tc * TS + TS > n && n >= TS) ? n - TS : tc * TS;
  const int wrows = min(TS, m - r0), wcols = min(TS, n - c0);
  const int wk = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);  // this wave's part of K
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;

  const double alpha = nseg > 0 ? s0.alpha : 1.0;
  const bool unit = alpha == 1.0 || alpha == -1.0;
  const bool pre = beta != 0.0 && unit && wk == 0;  // C is loaded ahead of the products
  f64x4 acc[NX][2][NX][2];
#pragma unroll
  for (int X = 0; X < NX; ++X)
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int Y = 0; Y < NX; ++Y)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[X][x][Y][y] = f64x4{0.0, 0.0, 0.0, 0.0};
  if (pre) {
    const double s = alpha * beta;
#pragma unroll
    for (int X = 0; X < NX; ++X)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = min(32 * X + 2 * (4 * r + lg) + x, wrows - 1);
#pragma unroll
          for (int Y = 0; Y < NX; ++Y)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
              const int j = min(32 * Y + 2 * li + y, wcols - 1);
              acc[X][x][Y][y][r] = s * C[(int64_t)(r0 + i) * ldc + c0 + j];
            }
        }
  }

  auto range = [&](int sid, int& kb, int& ke) {
    const int tri = BTA_SEG(tri, sid);
    kb = 0;
    ke = BTA_SEG(k, sid);
    if (tri & TRI_A_LOWER) ke = min(ke, (tr + 1) * TS);
    if (tri & TRI_A_UPPER) kb = max(kb, tr * TS);
    if (tri & TRI_B_LOWER) kb = max(kb, tc * TS);
    if (tri & TRI_B_UPPER) ke = min(ke, (tc + 1) * TS);
  };
  int total = 0;
  for (int sid = 0; sid < nseg; ++sid) {
    int kb, ke;
    range(sid, kb, ke);
    if (ke > kb) total += (ke - kb + 7) >> 3;
  }
  const int t0 = WK == 1 ? 0 : total * wk / WK;
  const int t1 = WK == 1 ? total : total * (wk + 1) / WK;
  const int nt = t1 - t0;

  // position of one side of the pipeline (loads or products)
  struct Pos {
    int seg, k, kb, ke, K;
  };
  auto enter = [&](Pos& p, int sid) {
    p.seg = sid;
    range(sid, p.kb, p.ke);
    p.k = p.kb;
    p.K = BTA_SEG(k, sid);
  };
  DirectOp<NX> oa;
  DirectOp<NX> ob;
  auto bind = [&](int sid) {
    const double *A = BTA_SEG(A, sid), *B = BTA_SEG(B, sid);
    const int lda = BTA_SEG(lda, sid), ldb = BTA_SEG(ldb, sid), ta = BTA_SEG(ta, sid), tb = BTA_SEG(tb, sid);
    const int K = BTA_SEG(k, sid);
    oa.init(A + (ta ? (int64_t)r0 : (int64_t)r0 * lda), lda, ta, wrows, K);
    ob.init(B + (tb ? (int64_t)c0 * ldb : (int64_t)c0), ldb, 1 - tb, wcols, K);
  };
  if (nt > 0) {
    Pos L, P;
    enter(L, 0);
    {
      int skip = t0;
      while (true) {
        const int ns = L.ke > L.kb ? (L.ke - L.kb + 7) >> 3 : 0;
        if (skip < ns) break;
        skip -= ns;
        enter(L, L.seg + 1);
      }
      L.k += 8 * skip;
    }
    P = L;
    bind(L.seg);
    int fa = oa.form, fb = ob.form;  // forms and mask of the segment being multiplied
    int ma = 0, mb = 0;
    auto masks = [&](int sid) {
      const int tri = BTA_SEG(tri, sid);
      ma = (tri & TRI_A_LOWER) ? MASK_K_GT_I : ((tri & TRI_A_UPPER) ? MASK_K_LT_I : MASK_NONE);
      mb = (tri & TRI_B_LOWER) ? MASK_K_LT_I : ((tri & TRI_B_UPPER) ? MASK_K_GT_I : MASK_NONE);
    };
    masks(P.seg);
    // a narrow operand of odd width stored along its rows: its last pair was
    // moved back (outputs past the width are not stored)
    bool odda = fa && wrows < TS && (wrows & 1) && wrows > 1, oddb = fb && wcols < TS && (wcols & 1) && wcols > 1;
    f64x2 va[S][NX][2], vb[S][NX][2];
    int left = nt;  // steps not yet loaded
    auto issue = [&](int st) {
      if (L.k + 8 <= L.K && !oa.narrow && !ob.narrow) {
        oa.load(va[st], L.k);
        ob.load(vb[st], L.k);
      } else {
        oa.load_edge(va[st], L.k);
        ob.load_edge(vb[st], L.k);
      }
      if (--left > 0) {  // past the last step: that step again, never used
        L.k += 8;
        if (L.k >= L.ke) {
          int sid = L.seg;
          do enter(L, ++sid);
          while (L.ke <= L.kb);
          bind(L.seg);
        }
      }
    };
    auto products = [&](const double (&ea)[NX][2][2], const double (&eb)[NX][2][2]) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int X = 0; X < NX; ++X)
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int Y = 0; Y < NX; ++Y)
#pragma unroll
              for (int y = 0; y < 2; ++y)
                acc[X][x][Y][y] = mfma_f64(ea[X][x][p], eb[Y][y][p], acc[X][x][Y][y]);
    };
    auto multiply = [&](int st) {
      double ea[NX][2][2], eb[NX][2][2];
      if (odda || P.k + 8 > P.ke || chunk_mask(ma, r0, TS, P.k, 8))
        DirectOp<NX>::fix(va[st], fa, wrows, P.k, P.K, P.ke, ma, r0, odda);
      if (oddb || P.k + 8 > P.ke || chunk_mask(mb, c0, TS, P.k, 8))
        DirectOp<NX>::fix(vb[st], fb, wcols, P.k, P.K, P.ke, mb, c0, oddb);
      DirectOp<NX>::frag(va[st], ea, fa);
      DirectOp<NX>::frag(vb[st], eb, fb);
      products(ea, eb);
      P.k += 8;
    };
    auto next_seg = [&]() {
      if (P.k >= P.ke) {
        int sid = P.seg;
        do enter(P, ++sid);
        while (P.ke <= P.kb);
        masks(P.seg);
        fa = BTA_SEG(ta, P.seg);
        fb = 1 - BTA_SEG(tb, P.seg);
        odda = fa && wrows < TS && (wrows & 1) && wrows > 1;
        oddb = fb && wcols < TS && (wcols & 1) && wcols > 1;
      }
    };
#pragma unroll
    for (int u = 0; u < S - 1; ++u) issue(u);
    int t = 0;
    while (t < nt) {
      // S interior steps of one segment on both sides: no tests in between
      if (!odda && !oddb && !oa.narrow && !ob.narrow && L.seg == P.seg && left > S && L.k + 8 * S < L.ke &&
          !chunk_mask(ma, r0, TS, P.k, 8 * S) && !chunk_mask(mb, c0, TS, P.k, 8 * S)) {
        do {
#pragma unroll
          for (int u = 0; u < S; ++u) {
            oa.load(va[(u + S - 1) % S], L.k);
            ob.load(vb[(u + S - 1) % S], L.k);
            L.k += 8;
            double ea[NX][2][2], eb[NX][2][2];
            DirectOp<NX>::frag(va[u], ea, fa);
            DirectOp<NX>::frag(vb[u], eb, fb);
            products(ea, eb);
#pragma unroll
            for (int z = 0; z < 4 * NX; ++z) {
              __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
              __builtin_amdgcn_sched_group_barrier(0x008, 2 * NX, 0);
            }
          }
          P.k += 8 * S;
          left -= S;
          t += S;
        } while (left > S && L.k + 8 * S < L.ke && !chunk_mask(ma, r0, TS, P.k, 8 * S) &&
                 !chunk_mask(mb, c0, TS, P.k, 8 * S));
        continue;
      }
#pragma unroll
      for (int u = 0; u < S; ++u) {
        issue((u + S - 1) % S);
        if (t + u < nt) {
          next_seg();
          multiply(u);
        }
      }
      t += S;
    }
  }

  if (WK > 1) {  // partial sums of the K parts, added in the order of the parts
    __shared__ double red[WK > 1 ? (WK - 1) * NX * NX * 16 * 64 : 1];
    if (wk > 0) {
#pragma unroll
      for (int X = 0; X < NX; ++X)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int Y = 0; Y < NX; ++Y)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                red[(((((wk - 1) * NX + X) * 2 + x) * NX + Y) * 2 + y) * 256 + r * 64 + lane] = acc[X][x][Y][y][r];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int q = 1; q < WK; ++q)
#pragma unroll
      for (int X = 0; X < NX; ++X)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int Y = 0; Y < NX; ++Y)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                acc[X][x][Y][y][r] += red[(((((q - 1) * NX + X) * 2 + x) * NX + Y) * 2 + y) * 256 + r * 64 + lane];
  }

  // epilogue: pairs of columns (and of rows for the mirrored half)
#pragma unroll
  for (int X = 0; X < NX; ++X)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int Y = 0; Y < NX; ++Y) {
        const int gi = r0 + 32 * X + 2 * (4 * r + lg), gj = c0 + 32 * Y + 2 * li;
        double v[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) v[x][y] = alpha * acc[X][x][Y][y][r];
        bool keep[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y)
            keep[x][y] = gi + x >= tr * TS && gj + y >= tc * TS && gi + x < m && gj + y < n && (!lower || gi + x >= gj + y);
        if (beta != 0.0 && !unit) {
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
              if (keep[x][y]) v[x][y] += beta * C[(int64_t)(gi + x) * ldc + gj + y];
        }
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          gdouble* p = C + (int64_t)(gi + x) * ldc + gj;
          if (keep[x][0] && keep[x][1]) *(gf64x2u*)p = f64x2u{v[x][0], v[x][1]};
          else if (keep[x][0]) p[0] = v[x][0];
          else if (keep[x][1]) p[1] = v[x][1];
        }
        if (lower && mirror) {
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            gdouble* p = C + (int64_t)(gj + y) * ldc + gi;
            const bool k0 = keep[0][y] && gi > gj + y, k1 = keep[1][y] && gi + 1 > gj + y;
            if (k0 && k1) *(gf64x2u*)p = f64x2u{v[0][y], v[1][y]};
            else if (k0) p[0] = v[0][y];
            else if (k1) p[1] = v[1][y];
          }
        }
      }
}

#undef BTA_SEG

}  // namespace bta
