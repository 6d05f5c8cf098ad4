// Grouped FP64 GEMM on 32x32 to 128x128 output tiles (FP64 MFMA), driven by a job table
// in device memory.  One launch covers any number of independent jobs of any
// shapes; a workgroup finds its job by binary search over the tile prefix
// sums.  Each job computes
//     C = beta * C + sum_s alpha_s * op(A_s) * op(B_s)
// over up to three segments (K-concatenation), optionally only on the tiles on
// or below the diagonal (symmetric output), optionally mirroring them so the
// full symmetric matrix is written.  Triangular operands restrict each tile's
// K range so structurally-zero products are skipped.
#pragma once
#include <vector>

#include "bta_device.h"

namespace bta {

enum : int {
  TRI_A_LOWER = 1,  // op(A)[i][k] == 0 for k > i   -> k < (tr+1)*64
  TRI_A_UPPER = 2,  // op(A)[i][k] == 0 for k < i   -> k >= tr*64
  TRI_B_LOWER = 4,  // op(B)[k][j] == 0 for k < j   -> k >= tc*64
  TRI_B_UPPER = 8,  // op(B)[k][j] == 0 for k > j   -> k < (tc+1)*64
};

struct GemmSeg {
  const double* A;
  const double* B;
  double alpha;
  int k;       // inner dimension
  int lda, ldb;
  int ta, tb;  // 0: op(X) = X, 1: op(X) = X^T
  int tri;     // TRI_* flags
};

struct GemmJob {
  double* C;
  double beta;   // 0: C is not read
  int m, n, ldc;
  int lower;     // 1: only tiles with tr >= tc
  int mirror;    // with lower: also write the transpose into the upper triangle
  int nseg;
  GemmSeg seg[3];
};

// Host-side helper: builds the job table and tile prefix for one launch.
struct GemmLaunch {
  std::vector<GemmJob> jobs;
  std::vector<int> prefix;  // njobs + 1
  int ts = 64;              // output tile edge: 64 or 128
  explicit GemmLaunch(int tile = 64) : ts(tile) {}
  int tiles() const { return prefix.empty() ? 0 : prefix.back(); }
  static int job_tiles(const GemmJob& j, int edge) {
    const int tm = (j.m + edge - 1) / edge, tn = (j.n + edge - 1) / edge;
    return j.lower ? tm * (tm + 1) / 2 : tm * tn;
  }
  void add(const GemmJob& j) {
    if (j.m <= 0 || j.n <= 0) return;
    if (prefix.empty()) prefix.push_back(0);
    jobs.push_back(j);
    prefix.push_back(prefix.back() + job_tiles(j, ts));
  }
};

// Default output tile edge: 64 (DevPlan::build takes 32 x 32 tiles where a
// launch has few of them).  Measured on MI355X at b = 2000 and 4500 64x64 tiles
// beat the 128x128 kernel for every product of the factorization and the
// selected inversion (1.44x on the selected inversion at b = 2000).  128 stays
// available to the autotuner.
inline int pick_tile(int m, int n) {
  (void)m;
  (void)n;
  return 64;
}

inline GemmSeg seg(const double* A, int lda, int ta, const double* B, int ldb, int tb, int k,
                   double alpha, int tri = 0) {
  GemmSeg s;
  s.A = A;
  s.B = B;
  s.alpha = alpha;
  s.k = k;
  s.lda = lda;
  s.ldb = ldb;
  s.ta = ta;
  s.tb = tb;
  s.tri = tri;
  return s;
}

inline GemmJob job(double* C, int m, int n, int ldc, double beta, int lower = 0, int mirror = 0) {
  GemmJob j = {};
  j.C = C;
  j.beta = beta;
  j.m = m;
  j.n = n;
  j.ldc = ldc;
  j.lower = lower;
  j.mirror = mirror;
  j.nseg = 0;
  return j;
}

inline GemmJob& add_seg(GemmJob& j, const GemmSeg& s) {
  if (s.k > 0) j.seg[j.nseg++] = s;
  return j;
}

// A set of grouped-GEMM launches whose job tables live in device memory.  Built
// once (hipMalloc + hipMemcpy, never during stream capture), then launched any
// number of times, including from inside a captured hipGraph.
struct DevPlan {
  // vec: every operand has an even leading dimension and a 16-byte aligned
  // base (the pipelined kernel's paired loads need both)
  // kernel: GemmKernel of the default variant, its tiles and their prefix sums
  struct Entry { int job_off, pre_off, njobs, tiles, ts, vec, kernel, kpre_off, ktiles; };
  GemmJob* d_jobs = nullptr;
  int* d_prefix = nullptr;
  size_t bytes = 0;  // device bytes of the job table and prefix sums
  std::vector<Entry> launches;
  DevPlan() = default;
  DevPlan(const DevPlan&) = delete;
  DevPlan& operator=(const DevPlan&) = delete;
  ~DevPlan();
  void release();
  int build(const std::vector<GemmLaunch>& ls);
  void launch(int idx, hipStream_t st, int variant = 0) const;
  bool empty() const { return launches.empty(); }
};

}  // namespace bta
