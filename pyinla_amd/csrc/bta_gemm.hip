// Grouped FP64 GEMM kernels + device job-table plans.
#include <algorithm>
#include <stdexcept>

#include "bta_gemm.h"
#include "bta_internal.h"

namespace bta {

// K chunk of the 64x64-tile kernel: 32 keeps the LDS footprint at 34 KB, so
// four workgroups share a CU (latency hiding, and 1024 resident tiles)
#ifndef BTA_GEMM_KC
#define BTA_GEMM_KC 32
#endif
#define BTA_GEMM_LD (BTA_GEMM_KC + 1)  // odd stride: conflict-free 16-row fragment reads
#ifndef BTA_GEMM_PAIRS
#define BTA_GEMM_PAIRS 1  // 16-byte loads of interior chunks where aligned
#endif
#ifndef BTA_GEMM_MINB
#define BTA_GEMM_MINB 4  // resident workgroups per CU the register budget is cut for
#endif

// acc += sA(64 x K) * sB(64 x K)^T over k in [0, kend) (LDS stride LD; any
// alpha was applied to sA when it was stored).
template <int LD>
__device__ __forceinline__ void mma_nt_ld(TileAcc& t, const double* __restrict__ sA,
                                          const double* __restrict__ sB, int kend) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
  const double* a0p = sA + (wm + li) * LD + lk;
  const double* a1p = sA + (wm + 16 + li) * LD + lk;
  const double* b0p = sB + (wn + li) * LD + lk;
  const double* b1p = sB + (wn + 16 + li) * LD + lk;
#pragma unroll 4
  for (int k = 0; k < kend; k += 4) {
    const double a0 = a0p[k], a1 = a1p[k], b0 = b0p[k], b1 = b1p[k];
    t.c[0][0] = mfma_f64(a0, b0, t.c[0][0]);
    t.c[0][1] = mfma_f64(a0, b1, t.c[0][1]);
    t.c[1][0] = mfma_f64(a1, b0, t.c[1][0]);
    t.c[1][1] = mfma_f64(a1, b1, t.c[1][1]);
  }
}

__device__ __forceinline__ int find_job(const int* __restrict__ prefix, int njobs, int bid) {
  int lo = 0, hi = njobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= bid) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Output tile of workgroup `local` of a tm x tn job.  Workgroups are
// dispatched to the 8 XCDs round-robin (blockIdx % 8), so the tiles are put in
// an order and XCD x takes the x-th eighth of it: a compact region whose A and
// B panels its L2 shares.  The order is bands of 8 tile rows, column by column,
// where all tiles have the same K; where K depends on the tile column or row
// (triangular operand) every XCD takes whole rows or columns of tiles, or the
// XCDs' shares differ by up to 3:1 (L W at b = 2000, 12 blocks in a launch:
// 210 us per block in bands, 160 by rows).
__device__ __forceinline__ int xcd_share(int local, int T) {
  const int x = local & 7, r = T & 7;
  return x * (T >> 3) + min(x, r) + (local >> 3);
}
__device__ __forceinline__ void xcd_tile(int local, int tm, int tn, int tri, int& tr, int& tc) {
  const int t = xcd_share(local, tm * tn);
  const bool ka = tri & (TRI_A_LOWER | TRI_A_UPPER), kb = tri & (TRI_B_LOWER | TRI_B_UPPER);
  if (kb && !ka) {
    tr = t / tn;
    tc = t % tn;
  } else if (ka && !kb) {
    tc = t / tm;
    tr = t % tm;
    if (tri & TRI_A_LOWER) tr = tm - 1 - tr;  // longest K first
  } else {
    const int band = t / (8 * tn), idx = t - band * 8 * tn, h = min(8, tm - 8 * band);
    tr = 8 * band + idx % h;
    tc = idx / h;
  }
}

__device__ __forceinline__ void decode_lower(int idx, int& tr, int& tc) {
  int r = (int)((sqrt(8.0 * idx + 1.0) - 1.0) * 0.5);
  while ((r + 1) * (r + 2) / 2 <= idx) ++r;
  while (r * (r + 1) / 2 > idx) --r;
  tr = r;
  tc = idx - r * (r + 1) / 2;
}

// A 64 x BTA_GEMM_KC operand chunk staged global -> registers -> LDS (same
// conventions as TilePrefetch: LDS layout s[i][k] of op(X)).  Thread t holds
// pairs of contiguous elements: with H = KC / 2 threads per chunk row,
// r[2q + u] is (i, k) = (t / H + (256 / H) q, 2 (t % H) + u) of a row-major
// chunk (trans 0) or (k, i) = (t / 32 + 8q, 2 (t % 32) + u) of a transposed
// one (trans 1), so an interior chunk with an even leading dimension and a
// 16-byte aligned origin is fetched with 16-byte loads.
struct ChunkPrefetch {
  static_assert(BTA_THREADS == 256 && BTA_GEMM_KC % 8 == 0 && BTA_GEMM_KC <= 64, "pair mapping");
  static constexpr int N = 64 * BTA_GEMM_KC / BTA_THREADS;
  static constexpr int H = BTA_GEMM_KC / 2;     // threads per row of a row-major chunk
  static constexpr int RQ = BTA_THREADS / H;    // its rows per pair step
  double r[N];
  __device__ __forceinline__ void load(const double* __restrict__ g0, int64_t ld, int trans, int rows, int kw,
                                       int mask, int i0, int k0) {
    const gdouble* g = gview(g0);
    mask = chunk_mask(mask, i0, rows, k0, kw);
    const int64_t step = trans == 0 ? RQ * ld : 8 * ld;
    const gdouble* t = trans == 0 ? g + (int64_t)(threadIdx.x / H) * ld + 2 * (threadIdx.x % H)
                                  : g + (int64_t)(threadIdx.x >> 5) * ld + 2 * (threadIdx.x & 31);
    if (mask == MASK_NONE && rows >= 64 && kw >= BTA_GEMM_KC) {  // interior chunk: no tests
      if (BTA_GEMM_PAIRS && (ld & 1) == 0 && (reinterpret_cast<uintptr_t>(g0) & 15) == 0) {
#pragma unroll
        for (int q = 0; q < N / 2; ++q) {
          const f64x2 x = *(const gf64x2*)(t + q * step);
          r[2 * q] = x.x;
          r[2 * q + 1] = x.y;
        }
      } else {
#pragma unroll
        for (int q = 0; q < N / 2; ++q) {
          r[2 * q] = t[q * step];
          r[2 * q + 1] = t[q * step + 1];
        }
      }
      return;
    }
#pragma unroll
    for (int q = 0; q < N / 2; ++q)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        int i, k;
        if (trans == 0) {
          i = threadIdx.x / H + RQ * q;
          k = 2 * (threadIdx.x % H) + u;
        } else {
          k = (threadIdx.x >> 5) + 8 * q;
          i = 2 * (threadIdx.x & 31) + u;
        }
        r[2 * q + u] = (i < rows && k < kw && !masked_out(mask, i0 + i, k0 + k)) ? t[q * step + u] : 0.0;
      }
  }
  __device__ __forceinline__ void store(double* __restrict__ s, int trans, double alpha = 1.0) const {
#pragma unroll
    for (int q = 0; q < N / 2; ++q) {
      if (trans == 0) {
        const int i = threadIdx.x / H + RQ * q, k = 2 * (threadIdx.x % H);
        s[i * BTA_GEMM_LD + k] = alpha * r[2 * q];
        s[i * BTA_GEMM_LD + k + 1] = alpha * r[2 * q + 1];
      } else {
        const int k = (threadIdx.x >> 5) + 8 * q, i = 2 * (threadIdx.x & 31);
        s[i * BTA_GEMM_LD + k] = alpha * r[2 * q];
        s[(i + 1) * BTA_GEMM_LD + k] = alpha * r[2 * q + 1];
      }
    }
  }
};

__global__ void __launch_bounds__(BTA_THREADS, BTA_GEMM_MINB) k_gemm_grouped(const GemmJob* __restrict__ jobs,
                                                             const int* __restrict__ prefix, int njobs) {
  __shared__ double sA[64 * BTA_GEMM_LD];
  __shared__ double sB[64 * BTA_GEMM_LD];
  const int jid = find_job(prefix, njobs, blockIdx.x);
  const GemmJob& g = jobs[jid];
  const int local = blockIdx.x - prefix[jid];
  int tr, tc;
  if (g.lower) decode_lower(local, tr, tc);
  else {
    const int tm = (g.m + 63) / 64, tn = (g.n + 63) / 64;
    xcd_tile(local, tm, tn, g.seg[0].tri, tr, tc);
  }
  const int rows = min(64, g.m - tr * 64), cols = min(64, g.n - tc * 64);
  // A tile at a ragged edge of a job at least 64 wide works on the 64-wide
  // window that ends at the edge (origin r0 / c0, overlapping the previous
  // tile) and writes only its own rows / columns: every chunk of it then
  // takes the same unguarded loads as an interior tile (measured: guarded
  // edge tiles held a 2000 x 2000 product at 397 us against 339 us for
  // 1984 x 1984).  Overlap rows and columns may miss K terms outside the
  // tile's own triangular range; they are never stored.
  const int r0 = (rows < 64 && g.m >= 64) ? g.m - 64 : tr * 64;
  const int c0 = (cols < 64 && g.n >= 64) ? g.n - 64 : tc * 64;
  const int wrows = min(64, g.m - r0), wcols = min(64, g.n - c0);
  double* ct = g.C + (int64_t)r0 * g.ldc + c0;
  TileAcc acc;
  if (g.beta != 0.0) {
    acc_load(acc, ct, g.ldc, wrows, wcols);
    if (g.beta != 1.0) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc.c[x][y] *= g.beta;
    }
  } else {
    acc_zero(acc);
  }
  // K chunks of all segments form one pipeline: chunk q+1 is fetched into
  // registers while chunk q is multiplied out of LDS.
  int seg_id = 0, k0 = 0, kmax = 0;
  auto seg_range = [&](int sid, int& kb, int& ke) {
    const GemmSeg& sg = g.seg[sid];
    kb = 0;
    ke = sg.k;
    if (sg.tri & TRI_A_LOWER) ke = min(ke, (tr + 1) * 64);
    if (sg.tri & TRI_A_UPPER) kb = max(kb, tr * 64);
    if (sg.tri & TRI_B_LOWER) kb = max(kb, tc * 64);
    if (sg.tri & TRI_B_UPPER) ke = min(ke, (tc + 1) * 64);
  };
  // advance (seg_id, k0) to the next non-empty chunk; returns false at the end
  auto next_chunk = [&](bool first) -> bool {
    if (!first) k0 += BTA_GEMM_KC;
    while (seg_id < g.nseg) {
      if (first || k0 >= kmax) {
        if (!first) ++seg_id;
        if (seg_id >= g.nseg) return false;
        int kb;
        seg_range(seg_id, kb, kmax);
        k0 = kb;
        first = false;
        if (k0 < kmax) return true;
        continue;
      }
      return true;
    }
    return false;
  };
  ChunkPrefetch pa, pb;
  auto fetch = [&]() {
    const GemmSeg& sg = g.seg[seg_id];
    const int kw = min(BTA_GEMM_KC, kmax - k0);
    const int ma = (sg.tri & TRI_A_LOWER) ? MASK_K_GT_I : ((sg.tri & TRI_A_UPPER) ? MASK_K_LT_I : MASK_NONE);
    const int mb = (sg.tri & TRI_B_LOWER) ? MASK_K_LT_I : ((sg.tri & TRI_B_UPPER) ? MASK_K_GT_I : MASK_NONE);
    if (sg.ta == 0) pa.load(sg.A + (int64_t)r0 * sg.lda + k0, sg.lda, 0, wrows, kw, ma, r0, k0);
    else pa.load(sg.A + (int64_t)k0 * sg.lda + r0, sg.lda, 1, wrows, kw, ma, r0, k0);
    if (sg.tb == 1) pb.load(sg.B + (int64_t)c0 * sg.ldb + k0, sg.ldb, 0, wcols, kw, mb, c0, k0);
    else pb.load(sg.B + (int64_t)k0 * sg.ldb + c0, sg.ldb, 1, wcols, kw, mb, c0, k0);
  };
  bool have = (g.nseg > 0) && next_chunk(true);
  if (have) fetch();
  while (have) {
    const GemmSeg& sg = g.seg[seg_id];
    const int kw = min(BTA_GEMM_KC, kmax - k0);
    pa.store(sA, sg.ta, sg.alpha);
    pb.store(sB, sg.tb == 1 ? 0 : 1);
    __syncthreads();
    have = next_chunk(false);
    if (have) fetch();
    mma_nt_ld<BTA_GEMM_LD>(acc, sA, sB, (kw + 3) & ~3);
    lds_barrier();  // not a wait for the next chunk's loads: its stores wait for them
  }
  // epilogue
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = acc_row(x, r), j = acc_col(y);
        const int gi = r0 + i, gj = c0 + j;  // global row / column
        if (i >= wrows || j >= wcols || gi < tr * 64 || gj < tc * 64) continue;
        const double v = acc.c[x][y][r];
        gdouble* cg = gview(g.C);
        if (g.lower && tr == tc) {
          if (gi >= gj) {
            cg[(int64_t)gi * g.ldc + gj] = v;
            if (g.mirror && gi > gj) cg[(int64_t)gj * g.ldc + gi] = v;
          }
        } else {
          cg[(int64_t)gi * g.ldc + gj] = v;
          if (g.lower && g.mirror) cg[(int64_t)gj * g.ldc + gi] = v;
        }
      }
}

}  // namespace bta

#include "bta_gemm_direct.h"

namespace bta {

// ------------------------------------------- 64x64 tiles, pipelined K loop
//
// Variant of the grouped GEMM (BTA_OPT_GEMM_KERNEL 1; measured slower on
// MI355X than the kernels above, NN 2000^3 354 us against 293 for k_gemm_grouped
// and 262 for k_gemm_direct, and kept for comparison).  K advances in chunks of 16; the
// A chunk (64 rows of op(A) x 16) is kept in LDS as sA[i][k] (odd stride 17)
// and the B chunk (16 x 64 columns of op(B)) as sB[k][j] (stride 68), so the
// MFMA operand reads of a wave (16 rows x 4 k) hit distinct banks.  Two LDS
// buffers and two register sets: while chunk t is multiplied out of one
// buffer, chunk t+1 (loaded two chunks earlier) is stored to the other and
// the loads of chunk t+3 are issued -- each global load has two chunks of
// MFMA work to arrive.
//
// Every chunk is loaded the same way, as pairs of doubles from addresses
// clamped into the operand (rows past the edge of the matrix, K past the end
// of the segment's range), and everything else -- zero fill at ragged edges
// and partial chunks, triangular masks, alpha -- is applied when the chunk is
// stored to LDS.  The load sequence is then the same straight-line code for
// every chunk, so the compiler can count the loads in flight and wait for one
// register set only.  Past the last chunk the loop re-loads the first one
// into the idle set (never stored).  Needs even leading dimensions and
// 16-byte aligned operands (DevPlan::launch falls back to the single-buffered
// kernel otherwise): a clamped pair then never leaves its matrix row.

#define G2_KC 16
#define G2_LDA (G2_KC + 1)
#define G2_LDB (64 + 4)


// Four elements of one 64 x 16 operand chunk per thread.  form 0 ("K
// contiguous"): element (r, k) at g[r * ld + k], the thread owns rows t/8 and
// t/8 + 32, columns 2 (t%8) and 2 (t%8) + 1; form 1 ("rows contiguous"):
// element (r, k) at g[k * ld + r], the thread owns k = t/32 and t/32 + 8, rows
// 2 (t%32) and 2 (t%32) + 1.  rows / kw: valid rows / K columns of the chunk.
struct G2Op {
  double r[4];
  // (row, k) inside the chunk of element u of pair q, and the memory offset
  // (in elements, from the chunk origin) of pair q before clamping
  __device__ __forceinline__ static void coord(int form, int q, int u, int& i, int& k) {
    const int t = threadIdx.x;
    const int i0 = (t >> 3) + 32 * q, k0 = 2 * (t & 7) + u;  // form 0
    const int i1 = 2 * (t & 31) + u, k1 = (t >> 5) + 8 * q;  // form 1
    i = form ? i1 : i0;
    k = form ? k1 : k0;
  }
  // The same two paired loads for either form: only the addresses differ.
  __device__ __forceinline__ void load(const double* __restrict__ g0, int64_t ld, int form, int rows, int kw) {
    const int t = threadIdx.x;
    const gdouble* g = gview(g0);
    const int kc = min(2 * (t & 7), (kw - 1) & ~1);
    const int rc = min(2 * (t & 31), (rows - 1) & ~1);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int rr = min((t >> 3) + 32 * q, rows - 1);
      const int kq = min((t >> 5) + 8 * q, kw - 1);
      const int64_t off = form ? (int64_t)kq * ld + rc : (int64_t)rr * ld + kc;
      const f64x2 v = *(const gf64x2*)(g + off);
      r[2 * q] = v.x;
      r[2 * q + 1] = v.y;
    }
  }
  // value of element (q, u) after the zero fill and the triangular mask,
  // evaluated without branches (bitwise, not short-circuit)
  __device__ __forceinline__ double val(int form, int q, int u, int rows, int kw, int mask, int i0, int k0) const {
    int i, k;
    coord(form, q, u, i, k);
    const int ig = i0 + i, kg = k0 + k;
    const bool out = (mask == MASK_K_GT_I) & (kg > ig) | (mask == MASK_K_LT_I) & (kg < ig);
    const bool keep = (i < rows) & (k < kw) & !out;
    return keep ? r[2 * q + u] : 0.0;
  }
  // A operand: sA[i][k] scaled by alpha
  __device__ __forceinline__ void store_a(double* __restrict__ sA, int form, double alpha, int rows, int kw, int mask,
                                          int i0, int k0) const {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        int i, k;
        coord(form, q, u, i, k);
        sA[i * G2_LDA + k] = alpha * val(form, q, u, rows, kw, mask, i0, k0);
      }
  }
  // B operand: sB[k][j]
  __device__ __forceinline__ void store_b(double* __restrict__ sB, int form, int cols, int kw, int mask, int j0,
                                          int k0) const {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        int i, k;
        coord(form, q, u, i, k);
        sB[k * G2_LDB + i] = val(form, q, u, cols, kw, mask, j0, k0);
      }
  }
};

// One staged chunk: both operands and the chunk they hold.
struct G2Stage {
  G2Op a, b;
  int seg, k0, kw;
};

__global__ void __launch_bounds__(BTA_THREADS, 4) k_gemm_grouped_db(const GemmJob* __restrict__ jobs,
                                                                   const int* __restrict__ prefix, int njobs) {
  __shared__ double sA[2][64 * G2_LDA];
  __shared__ double sB[2][G2_KC * G2_LDB];
  const int jid = find_job(prefix, njobs, blockIdx.x);
  const GemmJob& g = jobs[jid];
  const int local = blockIdx.x - prefix[jid];
  int tr, tc;
  if (g.lower) decode_lower(local, tr, tc);
  else {
    const int tm = (g.m + 63) / 64, tn = (g.n + 63) / 64;
    xcd_tile(local, tm, tn, g.seg[0].tri, tr, tc);
  }
  const int rows = min(64, g.m - tr * 64), cols = min(64, g.n - tc * 64);
  double* ct = g.C + (int64_t)(tr * 64) * g.ldc + tc * 64;
  TileAcc acc;
  if (g.beta != 0.0) {
    acc_load(acc, ct, g.ldc, rows, cols);
    if (g.beta != 1.0) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc.c[x][y] *= g.beta;
    }
  } else {
    acc_zero(acc);
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
  auto mma = [&](int buf) {
    const double* a0p = &sA[buf][(wm + li) * G2_LDA + lk];
    const double* a1p = a0p + 16 * G2_LDA;
    const double* b0p = &sB[buf][lk * G2_LDB + wn + li];
    const double* b1p = b0p + 16;
#pragma unroll
    for (int k = 0; k < G2_KC; k += 4) {
      const double a0 = a0p[k], a1 = a1p[k], b0 = b0p[k * G2_LDB], b1 = b1p[k * G2_LDB];
      acc.c[0][0] = mfma_f64(a0, b0, acc.c[0][0]);
      acc.c[0][1] = mfma_f64(a0, b1, acc.c[0][1]);
      acc.c[1][0] = mfma_f64(a1, b0, acc.c[1][0]);
      acc.c[1][1] = mfma_f64(a1, b1, acc.c[1][1]);
    }
  };
  // One pipeline per segment, its fields read once: the K loop then touches
  // no memory but the operands (segments are few, so refilling the pipeline
  // at a segment boundary costs little).
  for (int sid = 0; sid < g.nseg; ++sid) {
    const GemmSeg sg = g.seg[sid];
    int kb = 0, ke = sg.k;  // K range of this tile (triangular operands skip zero chunks)
    if (sg.tri & TRI_A_LOWER) ke = min(ke, (tr + 1) * 64);
    if (sg.tri & TRI_A_UPPER) kb = max(kb, tr * 64);
    if (sg.tri & TRI_B_LOWER) kb = max(kb, tc * 64);
    if (sg.tri & TRI_B_UPPER) ke = min(ke, (tc + 1) * 64);
    if (ke <= kb) continue;
    const int nch = (ke - kb + G2_KC - 1) / G2_KC;
    const int ma = (sg.tri & TRI_A_LOWER) ? MASK_K_GT_I : ((sg.tri & TRI_A_UPPER) ? MASK_K_LT_I : MASK_NONE);
    const int mb = (sg.tri & TRI_B_LOWER) ? MASK_K_LT_I : ((sg.tri & TRI_B_UPPER) ? MASK_K_GT_I : MASK_NONE);
    // chunk q (past the last one: the last one again, loaded and never used)
    auto fetch = [&](int q, G2Stage& st) {
      const int c0 = kb + G2_KC * min(q, nch - 1);
      const int kw = min(G2_KC, ke - c0);
      const int64_t oa = sg.ta ? (int64_t)c0 * sg.lda + tr * 64 : (int64_t)(tr * 64) * sg.lda + c0;
      const int64_t ob = sg.tb ? (int64_t)(tc * 64) * sg.ldb + c0 : (int64_t)c0 * sg.ldb + tc * 64;
      st.a.load(sg.A + oa, sg.lda, sg.ta, rows, kw);
      st.b.load(sg.B + ob, sg.ldb, 1 - sg.tb, cols, kw);
      st.k0 = c0;
      st.kw = kw;
    };
    auto stage = [&](const G2Stage& st, int buf) {
      st.a.store_a(sA[buf], sg.ta, sg.alpha, rows, st.kw, ma, tr * 64, st.k0);
      st.b.store_b(sB[buf], 1 - sg.tb, cols, st.kw, mb, tc * 64, st.k0);
    };
    // Chunk t sits in LDS buffer t % 2 when it is multiplied; every pass
    // issues the same loads and stores, only the MFMAs of a missing odd
    // chunk are skipped.
    G2Stage s0, s1;
    fetch(0, s0);
    fetch(1, s1);
    stage(s0, 0);
    fetch(2, s0);
    __syncthreads();
    for (int t = 0; t < nch; t += 2) {
      mma(0);           // chunk t
      stage(s1, 1);     // chunk t + 1
      fetch(t + 3, s1);
      lds_barrier();
      if (t + 1 < nch) mma(1);
      stage(s0, 0);     // chunk t + 2
      fetch(t + 4, s0);
      lds_barrier();
    }
  }
  // epilogue
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = acc_row(x, r), j = acc_col(y);
        if (i >= rows || j >= cols) continue;
        const double v = acc.c[x][y][r];
        gdouble* cg = gview(ct);
        if (g.lower && tr == tc) {
          if (i >= j) {
            cg[(int64_t)i * g.ldc + j] = v;
            if (g.mirror && i > j) cg[(int64_t)j * g.ldc + i] = v;
          }
        } else {
          cg[(int64_t)i * g.ldc + j] = v;
          if (g.lower && g.mirror) gview(g.C)[(int64_t)(tc * 64 + j) * g.ldc + tr * 64 + i] = v;
        }
      }
}

// ------------------------------------------------- 128x128 output tiles
//
// Same job semantics as k_gemm_grouped with 128x128 output tiles: wave w owns
// the 64x64 quadrant (64*(w/2), 64*(w%2)) as 4x4 MFMA 16x16 accumulators, K
// advances in chunks of 16 staged through LDS, the next chunk is fetched into
// registers while the current one is multiplied.

#define BIG_TS 128
#ifndef BIG_KC
#define BIG_KC 16
#endif
// odd row stride in doubles: the 16 rows of an MFMA operand fetch start on
// 16 distinct even dword banks, so the 64-bit reads are conflict-free
#define BIG_LD (BIG_KC + 1)

struct BigOp {
  static constexpr int N = BIG_TS * BIG_KC / BTA_THREADS;
  double r[N];
  // trans == 0: X row-major rows x K -> element (i, k) = X[i][k]
  // trans == 1: X row-major K x rows -> element (i, k) = X[k][i]
  __device__ __forceinline__ void load(const double* __restrict__ g0, int64_t ld, int trans, int rows, int kw,
                                       int mask, int i0, int k0) {
    const gdouble* g = gview(g0);
    mask = chunk_mask(mask, i0, rows, k0, kw);
    if (mask == MASK_NONE && rows >= BIG_TS && kw >= BIG_KC) {  // interior chunk: no tests
      if (trans == 0) {
        const gdouble* t = g + (int64_t)(threadIdx.x / BIG_KC) * ld + threadIdx.x % BIG_KC;
#pragma unroll
        for (int p = 0; p < N; ++p) r[p] = t[(int64_t)p * (BTA_THREADS / BIG_KC) * ld];
      } else {
        const gdouble* t = g + (int64_t)(threadIdx.x >> 7) * ld + (threadIdx.x & 127);
#pragma unroll
        for (int p = 0; p < N; ++p) r[p] = t[(int64_t)p * (BTA_THREADS / BIG_TS) * ld];
      }
      return;
    }
#pragma unroll
    for (int p = 0; p < N; ++p) {
      const int e = threadIdx.x + BTA_THREADS * p;
      if (trans == 0) {
        const int i = e / BIG_KC, k = e % BIG_KC;
        r[p] = (i < rows && k < kw && !masked_out(mask, i0 + i, k0 + k)) ? g[(int64_t)i * ld + k] : 0.0;
      } else {
        const int k = e >> 7, i = e & 127;
        r[p] = (i < rows && k < kw && !masked_out(mask, i0 + i, k0 + k)) ? g[(int64_t)k * ld + i] : 0.0;
      }
    }
  }
  __device__ __forceinline__ void store(double* __restrict__ s, int trans) const {
#pragma unroll
    for (int p = 0; p < N; ++p) {
      const int e = threadIdx.x + BTA_THREADS * p;
      if (trans == 0) s[(e / BIG_KC) * BIG_LD + (e % BIG_KC)] = r[p];
      else s[(e & 127) * BIG_LD + (e >> 7)] = r[p];
    }
  }
};

__global__ void __launch_bounds__(BTA_THREADS, 1) k_gemm_grouped_big(const GemmJob* __restrict__ jobs,
                                                                    const int* __restrict__ prefix, int njobs) {
  // two LDS buffers per operand: chunk q is multiplied out of one while chunk
  // q+1, fetched into registers before the multiply, is stored to the other
  __shared__ double sA[2][BIG_TS * BIG_LD];
  __shared__ double sB[2][BIG_TS * BIG_LD];
  const int jid = find_job(prefix, njobs, blockIdx.x);
  const GemmJob& g = jobs[jid];
  const int local = blockIdx.x - prefix[jid];
  int tr, tc;
  if (g.lower) decode_lower(local, tr, tc);
  else {
    const int tn = (g.n + BIG_TS - 1) / BIG_TS;
    tr = local / tn;
    tc = local % tn;
  }
  const int rows = min(BIG_TS, g.m - tr * BIG_TS), cols = min(BIG_TS, g.n - tc * BIG_TS);
  double* ct = g.C + (int64_t)(tr * BIG_TS) * g.ldc + tc * BIG_TS;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = (w >> 1) * 64, wn = (w & 1) * 64;
  const int li = lane & 15, lk = lane >> 4;
  f64x4 acc[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      if (g.beta != 0.0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = wm + 16 * x + 4 * r + lk, j = wn + 16 * y + li;
          acc[x][y][r] = (i < rows && j < cols) ? g.beta * gview(ct)[(int64_t)i * g.ldc + j] : 0.0;
        }
      } else {
        acc[x][y] = f64x4{0.0, 0.0, 0.0, 0.0};
      }
    }
  int seg_id = 0, k0 = 0, kmax = 0;
  auto seg_range = [&](int sid, int& kb, int& ke) {
    const GemmSeg& sg = g.seg[sid];
    kb = 0;
    ke = sg.k;
    if (sg.tri & TRI_A_LOWER) ke = min(ke, (tr + 1) * BIG_TS);
    if (sg.tri & TRI_A_UPPER) kb = max(kb, tr * BIG_TS);
    if (sg.tri & TRI_B_LOWER) kb = max(kb, tc * BIG_TS);
    if (sg.tri & TRI_B_UPPER) ke = min(ke, (tc + 1) * BIG_TS);
  };
  auto next_chunk = [&](bool first) -> bool {
    if (!first) k0 += BIG_KC;
    while (seg_id < g.nseg) {
      if (first || k0 >= kmax) {
        if (!first) ++seg_id;
        if (seg_id >= g.nseg) return false;
        int kb;
        seg_range(seg_id, kb, kmax);
        k0 = kb;
        first = false;
        if (k0 < kmax) return true;
        continue;
      }
      return true;
    }
    return false;
  };
  BigOp pa, pb;
  auto fetch = [&]() {
    const GemmSeg& sg = g.seg[seg_id];
    const int kw = min(BIG_KC, kmax - k0);
    const int ma = (sg.tri & TRI_A_LOWER) ? MASK_K_GT_I : ((sg.tri & TRI_A_UPPER) ? MASK_K_LT_I : MASK_NONE);
    const int mb = (sg.tri & TRI_B_LOWER) ? MASK_K_LT_I : ((sg.tri & TRI_B_UPPER) ? MASK_K_GT_I : MASK_NONE);
    if (sg.ta == 0) pa.load(sg.A + (int64_t)(tr * BIG_TS) * sg.lda + k0, sg.lda, 0, rows, kw, ma, tr * BIG_TS, k0);
    else pa.load(sg.A + (int64_t)k0 * sg.lda + tr * BIG_TS, sg.lda, 1, rows, kw, ma, tr * BIG_TS, k0);
    if (sg.tb == 1) pb.load(sg.B + (int64_t)(tc * BIG_TS) * sg.ldb + k0, sg.ldb, 0, cols, kw, mb, tc * BIG_TS, k0);
    else pb.load(sg.B + (int64_t)k0 * sg.ldb + tc * BIG_TS, sg.ldb, 1, cols, kw, mb, tc * BIG_TS, k0);
  };
  bool have = (g.nseg > 0) && next_chunk(true);
  int buf = 0;
  if (have) {
    fetch();
    const GemmSeg& sg = g.seg[seg_id];
    pa.store(sA[0], sg.ta);
    pb.store(sB[0], (sg.tb == 1) ? 0 : 1);
    __syncthreads();
  }
  while (have) {
    const int kw = min(BIG_KC, kmax - k0);
    const double alpha = g.seg[seg_id].alpha;
    const bool more = next_chunk(false);
    if (more) fetch();
    const double* cA = sA[buf];
    const double* cB = sB[buf];
#pragma unroll
    for (int k = 0; k < BIG_KC; k += 4) {
      if (k < kw) {
        double av[4], bv[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) av[x] = alpha * cA[(wm + 16 * x + li) * BIG_LD + k + lk];
#pragma unroll
        for (int y = 0; y < 4; ++y) bv[y] = cB[(wn + 16 * y + li) * BIG_LD + k + lk];
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int y = 0; y < 4; ++y) acc[x][y] = mfma_f64(av[x], bv[y], acc[x][y]);
      }
    }
    if (more) {
      const GemmSeg& sg = g.seg[seg_id];
      pa.store(sA[buf ^ 1], sg.ta);
      pb.store(sB[buf ^ 1], (sg.tb == 1) ? 0 : 1);
    }
    // one barrier per chunk: the buffer stored above was last read before
    // the previous barrier, the one read next was stored before this one
    __syncthreads();
    buf ^= 1;
    have = more;
  }
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = wm + 16 * x + 4 * r + lk, j = wn + 16 * y + li;
        if (i >= rows || j >= cols) continue;
        const double v = acc[x][y][r];
        gdouble* cg = gview(ct);
        if (g.lower && tr == tc) {
          if (i >= j) {
            cg[(int64_t)i * g.ldc + j] = v;
            if (g.mirror && i > j) cg[(int64_t)j * g.ldc + i] = v;
          }
        } else {
          cg[(int64_t)i * g.ldc + j] = v;
          if (g.lower && g.mirror) gview(g.C)[(int64_t)(tc * BIG_TS + j) * g.ldc + tr * BIG_TS + i] = v;
        }
      }
}

// ------------------------------------------------------------------- plans

DevPlan::~DevPlan() { release(); }

void DevPlan::release() {
  if (d_jobs) hipFree(d_jobs);
  if (d_prefix) hipFree(d_prefix);
  d_jobs = nullptr;
  d_prefix = nullptr;
  bytes = 0;
  launches.clear();
}

// Kernels of a launch of 64-wide tiles (BTA_OPT_GEMM_KERNEL 0).
enum GemmKernel : int {
  KER_LDS,   // k_gemm_grouped
  KER_D32,   // k_gemm_direct, 32 x 32 tiles, four waves each with a quarter of K
  KER_D32W,  // 32 x 32 tiles, one wave each
  KER_D64,   // 64 x 64 tiles, one wave each
  KER_D64K   // 64 x 64 tiles, two waves each with a half of K
};

// The kernel by the number of tiles; times in us of one b x b x b product
// (NN / lower triangle of TN with mirrored output) measured on MI355X:
//            b = 417      800        1200       1600        2000       4500
//   LDS      31 / 31      54 / 53    105 / 81   181 / 131   293 / 228  3070 / 1580
//   D32      12 / 13      34 / 23    87 / 48    162 / 90    331 / 165
//   D32W     23 / 25      36 / 37    90 / 60    172 / 117   299 / 154
//   D64      64 / 66      109 / 112  160 / 163  210 / 212   262 / 263  2845 / 1731
//   D64K     39 / 41      63 / 64    90 / 91    217 / 117   274 / 271  2895 / 1470
// One wave per SIMD runs a 64 x 64 tile (1024 at a time), two run 32 x 32 tiles
// (2048): D64 and D64K are the fastest where their last turn is 85 % full, else
// the smaller tiles are.  Triangular products have short and uneven K ranges
// and mask a good part of their chunks: LDS (block inverses, 20 blocks of b =
// 2000, 512-wide merge: LDS 145 us, D32W 177, D64 204; L W 160 us per block
// against 165 with D64).  Both operands K-contiguous (A B^T: the block updates
// of the factorization): LDS too.  32 x 32 tiles run into the half lines there
// (b = 1600: 244 us against 186), and K in parts changes what the updates
// round: D_{i+1} - L_i L_i^T cancels, and the coregional model's f moves by
// 1e-10 of its value.
static GemmKernel pick_kernel(const GemmLaunch& l) {
  bool nt = false, mixed = false;
  int64_t t32 = 0, t64 = 0, tri64 = 0;
  for (const GemmJob& j : l.jobs) {
    t32 += GemmLaunch::job_tiles(j, 32);
    t64 += GemmLaunch::job_tiles(j, 64);
    if (j.seg[0].tri) tri64 += GemmLaunch::job_tiles(j, 64);
    for (int q = 0; q < j.nseg; ++q) {
      const GemmSeg& sg = j.seg[q];
      nt = nt || (sg.ta == 0 && sg.tb == 1);
      mixed = mixed || sg.alpha != j.seg[0].alpha;
    }
  }
  // k_gemm_direct scales a job's sum once, with the alpha of its first segment
  if (mixed || nt || 2 * tri64 > t64) return KER_LDS;
  auto fill = [](int64_t t, int64_t slots) { return (double)t / (double)((t + slots - 1) / slots * slots); };
  const double u1 = fill(t64, 1024), u2 = 0.96 * fill(2 * t64, 1024);
  if (u1 >= 0.85 && u1 >= u2) return KER_D64;
  if (u2 >= 0.85) return KER_D64K;
  return t32 <= 700 || fill(t32, 2048) < 0.85 ? KER_D32 : KER_D32W;
}

int DevPlan::build(const std::vector<GemmLaunch>& ls) {
  release();
  std::vector<GemmJob> all;
  std::vector<int> pre;
  for (const auto& l : ls) {
    Entry e;
    e.job_off = (int)all.size();
    e.pre_off = (int)pre.size();
    e.njobs = (int)l.jobs.size();
    e.tiles = l.tiles();
    e.ts = l.ts;
    e.vec = 1;
    for (const GemmJob& j : l.jobs) {
      for (int q = 0; q < j.nseg; ++q) {
        const GemmSeg& sg = j.seg[q];
        if ((sg.lda & 1) || (sg.ldb & 1) || (reinterpret_cast<uintptr_t>(sg.A) & 15) ||
            (reinterpret_cast<uintptr_t>(sg.B) & 15))
          e.vec = 0;
      }
    }
    e.kernel = l.ts == 64 ? pick_kernel(l) : KER_LDS;
    e.kpre_off = e.pre_off;
    e.ktiles = e.tiles;
    pre.insert(pre.end(), l.prefix.begin(), l.prefix.end());
    if (e.kernel == KER_D32 || e.kernel == KER_D32W) {
      e.kpre_off = (int)pre.size();
      e.ktiles = 0;
      for (const GemmJob& j : l.jobs) {
        pre.push_back(e.ktiles);
        e.ktiles += GemmLaunch::job_tiles(j, 32);
      }
      pre.push_back(e.ktiles);
    }
    launches.push_back(e);
    all.insert(all.end(), l.jobs.begin(), l.jobs.end());
  }
  if (all.empty()) return 0;
  hipError_t e;
  if ((e = hipMalloc(&d_jobs, all.size() * sizeof(GemmJob))) != hipSuccess) return (int)e;
  if ((e = hipMalloc(&d_prefix, pre.size() * sizeof(int))) != hipSuccess) return (int)e;
  if ((e = hipMemcpy(d_jobs, all.data(), all.size() * sizeof(GemmJob), hipMemcpyHostToDevice)) != hipSuccess)
    return (int)e;
  if ((e = hipMemcpy(d_prefix, pre.data(), pre.size() * sizeof(int), hipMemcpyHostToDevice)) != hipSuccess)
    return (int)e;
  bytes = all.size() * sizeof(GemmJob) + pre.size() * sizeof(int);
  return 0;
}

void DevPlan::launch(int idx, hipStream_t st, int variant) const {
  const Entry& e = launches[idx];
  if (e.tiles <= 0) return;
  const GemmJob* jobs = d_jobs + e.job_off;
  auto run = [&](auto* kernel, int tiles, int threads, int pre_off) {
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(threads), 0, st, jobs, d_prefix + pre_off, e.njobs);
  };
  if (e.ts == BIG_TS) return run(k_gemm_grouped_big, e.tiles, BTA_THREADS, e.pre_off);
  if (variant == 1 && e.vec) return run(k_gemm_grouped_db, e.tiles, BTA_THREADS, e.pre_off);
  switch (e.kernel) {
    case KER_D32: return run(k_gemm_direct<1, 4, 4, 2>, e.ktiles, 256, e.kpre_off);
    case KER_D32W: return run(k_gemm_direct<1, 1, 4, 2>, e.ktiles, 64, e.kpre_off);
    case KER_D64: return run(k_gemm_direct<2, 1, 3, 1>, e.ktiles, 64, e.kpre_off);
    case KER_D64K: return run(k_gemm_direct<2, 2, 3, 1>, e.ktiles, 128, e.kpre_off);
    default: return run(k_gemm_grouped, e.ktiles, BTA_THREADS, e.kpre_off);
  }
}

}  // namespace bta
