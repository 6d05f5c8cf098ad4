// Triangular sweeps with the BTA factor (pobtas / pobts) on gfx950.
//
// With the block inverses W_i = D_i^-1 (built once per factor), both sweeps
// are chains of matrix-vector products:
//   forward  ("N"):  y_i = W_i (r_i - L_{i-1} y_{i-1});  r_a -= sum_i B_i y_i;
//                    y_a = T^-1 r_a
//   backward ("C"):  x_a = T^-T y_a;
//                    x_i = W_i^T (y_i - L_i^T x_{i+1} - B_i^T x_a)
// The right-hand side is overwritten in place (N x nrhs, row-major, leading
// dimension ldrhs), as the reference's in-place pobtas does.
//
// One persistent launch runs a whole sweep.  What bounds it: the factor is
// read once per sweep (HBM), and the 2n products of the chain depend on each
// other, so between two of them every workgroup needs the whole vector the
// others just produced.  One launch per product (four per block) spends that
// hand-over as a kernel boundary plus cold loads; here a workgroup has the
// rows of its next product in registers before the vector arrives.
//
// Measured on MI355X, us per product (2n of them in a sweep), forward /
// backward, against one launch per product:
//   b = 48            0.63 / 0.89   (7.1 / 6.2)   one workgroup, vectors in LDS
//   b = 92            1.3 / 1.4     (7.2 / 7.4)
//   b = 400           1.3 / 1.5     (7.3 / 8.7)
//   b = 800           2.3 / 2.8     (8.6 / 11.1)
//   b = 1600          4.1 / 5.6     (11.3 / 13.7) its bytes at 5 TB/s: 3.1
//   b = 4500          25 / 34       (37 / 37)     its bytes at 5 TB/s: 24
//   b = 800, 8 right-hand sides     3.8 / 3.8; 16 6.4 on average (78 / 55)
#include <algorithm>

#include "bta_internal.h"
#include "bta_sweep_walk.h"

namespace bta {

namespace {

// 16-byte load that needs 8-byte alignment only (odd leading dimensions).
typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));
typedef __attribute__((address_space(1))) d2 gd2;

// Hand-over marker: a signalling NaN.  Every value handed over is the result
// of an FP64 operation, and those quiet NaNs, so no value can equal it.
constexpr unsigned long long kPending = 0x7FF4C0DEC0DE0001ull;
// Largest block swept by a single workgroup: one CU reads its matrices at 25 to
// 32 GB/s, at b = 92 (68 KB) 2.1 / 2.7 us per product against 1.3 / 1.4 with the
// hand-over.
constexpr int kSolo = 64;
constexpr int kSoloThreads = 512;   // kSolo x 8
constexpr int kSweepThreads = 512;  // the multiplying waves

struct SweepArgs {
  const double* L;
  const double* B;
  const double* W;
  double* X;                   // first column of the group
  double* vec;                 // (products + 1) vectors of b x R (backward: two partial vectors each)
  unsigned* claims;            // seats: nonzero once a workgroup has taken it
  int* fail;                   // a wait of this launch has given up
  int* err;                    // the same in host memory, set until the host has read it
  unsigned long long spin_ticks;
  int n, b, a, ldx, nr;        // nr <= R right-hand sides
  int parts;                   // work items per product
  int seats;                   // workgroups per group of R right-hand sides
  int64_t gstride;             // doubles from one group's scratch to the next's

  // Groups of R columns run side by side: the arguments of group g.
  __device__ __forceinline__ void enter_group(int R, int g) {
    X += (int64_t)g * R;
    vec += g * gstride;
    claims += g * gstride * (int64_t)(sizeof(double) / sizeof(unsigned));
    nr = min(R, nr - g * R);
  }
};

// Length of a hand-over vector: whole 128-byte lines.
__host__ __device__ inline int64_t vec_len(int b, int R) { return ((int64_t)b * R + 15) & ~15ll; }

__device__ __forceinline__ unsigned long long ld_bits(const double* p) {
  return __hip_atomic_load(reinterpret_cast<unsigned long long*>(const_cast<double*>(p)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

// 0 for the first workgroup that asks.
__device__ __forceinline__ unsigned claim_seat(unsigned* claim) {
  return __hip_atomic_exchange(claim, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Sums of lanes without LDS traffic.  row_sum<S>: over the lanes of a 16-lane
// row that agree modulo S (DPP row rotations); wave_sum<S>: over all four rows
// as well (v_permlane16/32_swap of a register with itself leaves the two
// halves' values side by side).  Every lane gets the total.
template <int CTRL>
__device__ __forceinline__ double add_dpp(double v) {
  const long long x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), CTRL, 0xf, 0xf, true);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int S>
__device__ __forceinline__ double row_sum(double v) {
  v = add_dpp<0x128>(v);  // row_ror:8
  if constexpr (S <= 4) v = add_dpp<0x124>(v);
  if constexpr (S <= 2) v = add_dpp<0x122>(v);
  if constexpr (S <= 1) v = add_dpp<0x121>(v);
  return v;
}
template <int S>
__device__ __forceinline__ double wave_sum(double v) {
  v = row_sum<S>(v);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const long long x = __double_as_longlong(v);
    const unsigned lo = (unsigned)x, hi = (unsigned)(x >> 32);
    const auto l = h == 0 ? __builtin_amdgcn_permlane16_swap(lo, lo, false, false)
                          : __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto u = h == 0 ? __builtin_amdgcn_permlane16_swap(hi, hi, false, false)
                          : __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    v = __longlong_as_double(((long long)u[0] << 32) | l[0]) + __longlong_as_double(((long long)u[1] << 32) | l[1]);
  }
  return v;
}
// Sum over each group of 8 consecutive lanes (quad permutes, then the other
// quad of the half row).
__device__ __forceinline__ double sum8(double v) {
  v = add_dpp<0xB1>(v);         // quad_perm [1,0,3,2]
  v = add_dpp<0x4E>(v);         // quad_perm [2,3,0,1]
  return add_dpp<0x141>(v);     // row_half_mirror
}

// -------------------------------------------------------- several workgroups
//
// The items of a sweep, who runs them and why the launch always ends:
// bta_sweep_walk.h.
//
// Hand-over: every stage has a vector of its own, filled with kPending before
// the launch; an item stores its outputs there with write-through stores (whole
// 64-byte sectors), and readers poll the elements themselves until none is
// kPending: one trip to memory.  (A flag per item behind the data, and the data
// then read through L2, cost 0.4 us more per stage at every size.)
//
// Work items.  Forward: 8 rows, one per wave, 16-byte loads along the row.
// Backward (columns of a row-major matrix): 16 columns, i.e. whole 128-byte
// lines, of one half of the rows -- two partial vectors, added by the readers
// and by k_sweep_finish; strips of 8 columns fetched every line twice (1.8
// times the bytes).  A wave has up to U loads of its item in flight before the
// vector arrives; larger blocks run in rounds.

// What the two kinds of waves of a workgroup share.
template <int R, int U, bool T>
struct SweepLds {
  static constexpr int RK = (T ? 64 : 128) * U;   // vector elements per round
  static constexpr int LV = R > 1 ? RK + 2 : RK;  // one vector per right-hand side
  static constexpr int NO = T ? 16 : 8;           // outputs of an item
  alignas(16) double v[LV * R];
  double red[T ? 8 * NO * R : NO * R];
  double xa[T ? 64 * R : 1];
  int seat[kSeats];  // the seats of this workgroup
  int victim;        // at the gate: distance from the own seat to a free one (kSeats: none)
  int got;           // the seat that was taken over (-1: another workgroup has it)
  int dead;          // the own seat was taken
};

constexpr unsigned kPatience = 1000000;  // s_memrealtime ticks (100 MHz): 10 ms

// The claims of the seats that a waiting thread looks after.
template <int NP>
struct SweepClaims {
  static constexpr int N = kSeats / (64 * NP);
  unsigned c[N];
  __device__ __forceinline__ void load(const SweepArgs& p, int t) {
#pragma unroll
    for (int j = 0; j < N; ++j)
      c[j] = __hip_atomic_load(p.claims + min(t + 64 * NP * j, p.seats - 1), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
  }
  // Distance from the own seat to a free one, kSeats if all are claimed: each
  // workgroup takes over another one first.
  __device__ __forceinline__ int free_seat(const SweepArgs& p, int t, int own) const {
    int d = kSeats;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int s = min(t + 64 * NP * j, p.seats - 1), e = s - own;
      if (c[j] == 0) d = min(d, e < 0 ? e + p.seats : e);
    }
    return d;
  }
};

// The gate, called by all threads: returns once every seat is claimed, or with
// the walk at the stage-0 items of a seat this workgroup has taken over.  `look`:
// what this thread finds (kSeats: no free seat), after some time of waiting.
template <class Lds, class Look>
__device__ __forceinline__ void sweep_gate(const SweepArgs& p, Lds& l, SweepWalk& walk, int own, bool chief,
                                           Look&& look) {
  for (bool first = walk.count == 1;; first = false) {
    const int d = look(first);
    if (d < kSeats) atomicMin(&l.victim, d);
    lds_barrier();
    const int v = __builtin_amdgcn_readfirstlane(l.victim);
    if (v >= kSeats) {
      walk.open = true;
      return;
    }
    lds_barrier();
    if (chief) {
      const int s = own + v < p.seats ? own + v : own + v - p.seats;
      l.victim = kSeats;
      l.got = claim_seat(p.claims + s) == 0 ? s : -1;
      if (l.got >= 0) l.seat[walk.count] = s;
    }
    lds_barrier();
    const int s = __builtin_amdgcn_readfirstlane(l.got);
    if (s >= 0) {
      walk.take_over(s);
      return;
    }
  }
}

// Brings elements [ks, ks + cnt / R) of the vector before stage g.stage into
// LDS, by threads t of nt; `waiting` says whether to go on waiting.
template <int R, int U, bool T, class Wait>
__device__ __forceinline__ void sweep_stage(const SweepArgs& p, SweepLds<R, U, T>& l, const SweepItem<T>& g, int ks,
                                            int cnt, int t, int nt, Wait&& waiting) {
  using Lds = SweepLds<R, U, T>;
  const int64_t half = vec_len(p.b, R);
  const double* sr = p.vec + g.stage * (T ? 2 * half : half) + (int64_t)ks * R;  // stage s writes vector s + 1
  // loads in flight per thread and vector: one batch brings a round's vector
  constexpr int Q = R > 1 ? (T ? 4 : 8) : U / 2;
  for (int e0 = t; e0 < cnt; e0 += Q * nt) {
    unsigned long long v[Q], h[T ? Q : 1];
    auto pending = [&]() {
      bool x = false;
#pragma unroll
      for (int q = 0; q < Q; ++q) x |= v[q] == kPending || (T && h[T ? q : 0] == kPending);
      return x;
    };
    do {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int e = min(e0 + q * nt, cnt - 1);
        v[q] = ld_bits(sr + e);
        if constexpr (T) h[q] = ld_bits(sr + half + e);
      }
    } while (pending() && waiting());
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (const int e = e0 + q * nt; e < cnt) {
        double x = __longlong_as_double((long long)v[q]);
        if constexpr (T) x += __longlong_as_double((long long)h[q]);
        l.v[e % R * Lds::LV + e / R] = x;
      }
  }
}

// Bound on a wait of a thread: it ends for good, with fail and err, after
// spin_ticks, or once another workgroup has raised fail (looked at after 10 ms:
// polled by everyone from the start, that one word would be a hot spot).  What is
// missing then stays kPending, a NaN, and spreads through what follows.
struct SweepWait {
  const SweepArgs& p;
  unsigned long long t0 = 0;
  __device__ __forceinline__ bool operator()() {
    __builtin_amdgcn_s_sleep(1);
    const unsigned long long now = __builtin_amdgcn_s_memrealtime();
    if (t0 == 0) t0 = now;
    if (now - t0 < p.spin_ticks)
      return now - t0 < kPatience || __hip_atomic_load(p.fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == 0;
    __hip_atomic_store(p.fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(p.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return false;
  }
};

// Waves that wait: they bring the vector into LDS while the others' loads are
// in flight (loads return in order: a wave with matrix loads outstanding would
// see the vector only after them).  With several right-hand sides, whose vectors
// are larger, all waves do.
template <int R, int U, bool T, int NP>
__device__ __forceinline__ void sweep_poller(const SweepArgs& p, SweepLds<R, U, T>& l, int stages, int own) {
  using Lds = SweepLds<R, U, T>;
  const int t = (int)threadIdx.x - kSweepThreads;
  SweepWalk walk(stages, p.parts, p.seats, own);
  // the claims, loaded in stage 0 beside the products and looked at from the gate on
  SweepClaims<NP> claims;
  auto look = [&](bool first) {
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    int d;
    while ((d = claims.free_seat(p, t, own)) < kSeats &&
           __builtin_amdgcn_s_memrealtime() - t0 < (first ? kPatience : kPatience / 100)) {
      __builtin_amdgcn_s_sleep(1);
      claims.load(p, t);
    }
    return d;
  };
  do {
    if (walk.at_gate()) sweep_gate(p, l, walk, own, t == 0, look);
    const SweepItem<T> g(p.n, p.b, p.a, walk.stage, walk.part);
    for (int ks = g.kbeg; ks < g.kend; ks += Lds::RK) {
      if (ks > g.kbeg) lds_barrier();  // the previous round's reads are done
      sweep_stage<R, U, T>(p, l, g, ks, min(Lds::RK, g.kend - ks) * R, R > 1 ? threadIdx.x : t,
                           R > 1 ? kSweepThreads + 64 * NP : 64 * NP, SweepWait{p});
      lds_barrier();
    }
    if (walk.stage == 0) claims.load(p, t);
    lds_barrier();  // [red]
    lds_barrier();  // [end]
  } while (walk.more(l.seat));
}

// Waves that multiply: 8 of them, each with up to U 16-byte loads of the
// item's matrix in flight while the others wait.
template <int R, int U, bool T, int NP>
__device__ __forceinline__ void sweep_worker(const SweepArgs& p, SweepLds<R, U, T>& l, int stages, int own) {
  using Lds = SweepLds<R, U, T>;
  constexpr int RK = Lds::RK, LV = Lds::LV, NO = Lds::NO, NA = T ? 2 * R : R;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = p.b, a = p.a;
  const int64_t half = vec_len(b, R), vlen = T ? 2 * half : half;
  SweepWalk walk(stages, p.parts, p.seats, own);
  do {
    if (walk.at_gate()) sweep_gate(p, l, walk, own, false, [](bool) { return kSeats; });
    const SweepItem<T> g(p.n, b, a, walk.stage, walk.part);
    const int i = g.i;
    const double* M = g.isw || !g.hasm ? p.W + (int64_t)i * b * b : p.L + (int64_t)(T ? i : i - 1) * b * b;
    const int row = T ? g.out0 : g.out0 + w;  // this wave's output row / the strip's first column
    const bool live = T || row < b;
    const int kend = T ? g.kend : (!live ? 0 : (g.isw ? row + 1 : b));
    const int j = row + 2 * (lane & 7), cl = min(j, b - 2);  // backward: this lane's column pair
    const int lim = min(max(kend - 1, 0) & ~1, b - 2);
    d2 m[U];
    // Straight-line loads, clamped into the operand (a whole wave past the end
    // reads one line): under tests the compiler waits for each load before it
    // issues the next.
    auto fetch = [&](int ks) {
      const gdouble* q = gview(M) + (T ? (int64_t)cl : (int64_t)(live ? row : 0) * b);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if constexpr (T) m[u] = *(const gd2*)(q + (int64_t)min(ks + 8 * (w + 8 * u) + (lane >> 3), b - 1) * b);
        else m[u] = *(const gd2*)(q + min(ks + 128 * u + 2 * lane, lim));
      }
    };
    fetch(g.kbeg);
    // the item's other operands: the vector it adds to, the arrow rows
    const int orow = g.out0 + tid / R, orc = tid % R;  // this thread's output
    const bool outp = tid < NO * R && orow < b;
    double base = 0.0;
    d2 mb = {0.0, 0.0};
    if (!g.isw && g.hf == 0 && outp && orc < p.nr) base = p.X[((int64_t)i * b + orow) * p.ldx + orc];
    const int qb = 8 * w + (lane >> 3);
    const bool arrow = T && !g.isw && g.hf == 0 && qb < a;
    if (arrow) mb = *(const gd2*)(gview(p.B) + ((int64_t)i * a + qb) * b + cl);
    double acc[NA];
#pragma unroll
    for (int q = 0; q < NA; ++q) acc[q] = 0.0;
    for (int ks = g.kbeg; ks < g.kend; ks += RK) {
      if (ks > g.kbeg) {
        lds_barrier();
        fetch(ks);
      }
      if constexpr (R > 1)
        sweep_stage<R, U, T>(p, l, g, ks, min(RK, g.kend - ks) * R, tid, kSweepThreads + 64 * NP, SweepWait{p});
      lds_barrier();
      const int ke = min(ks + RK, kend);
      // tests only every few steps: the LDS reads of a step overlap the products
      // of the one before
      constexpr int UG = R > 1 ? 1 : 4;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (u > 0 && u % UG == 0 && ks + (T ? 64 : 128) * u >= ke) break;
        if constexpr (T) {
          const int k = ks + 8 * (w + 8 * u) + (lane >> 3);
          // a pair moved left by the matrix edge holds column j in its second half
          const double x = j > cl ? m[u].y : m[u].x;
          const bool k0 = k < ke && (!g.isw || k >= j), k1 = k < ke && (!g.isw || k > j);
#pragma unroll
          for (int q = 0; q < R; ++q) {
            const double v = l.v[q * LV + k - ks];
            const double s0 = fma(x, v, acc[2 * q]), s1 = fma(m[u].y, v, acc[2 * q + 1]);
            acc[2 * q] = k0 ? s0 : acc[2 * q];
            acc[2 * q + 1] = k1 ? s1 : acc[2 * q + 1];
          }
        } else {
          const int k = ks + 128 * u + 2 * lane;
          const double x = k > lim ? m[u].y : m[u].x;
#pragma unroll
          for (int q = 0; q < R; ++q) {
            const f64x2 v = *(const f64x2*)&l.v[q * LV + k - ks];
            const double s0 = fma(x, v.x, acc[q]);
            acc[q] = k < ke ? s0 : acc[q];
            const double s1 = fma(m[u].y, v.y, acc[q]);
            acc[q] = k + 1 < ke ? s1 : acc[q];
          }
        }
      }
    }
    double out = 0.0;
    if constexpr (T) {
      if (arrow) {
        const double x = j > cl ? mb.y : mb.x;
#pragma unroll
        for (int q = 0; q < R; ++q) {
          acc[2 * q] = fma(x, l.xa[qb * R + q], acc[2 * q]);
          acc[2 * q + 1] = fma(mb.y, l.xa[qb * R + q], acc[2 * q + 1]);
        }
      }
#pragma unroll
      for (int q = 0; q < NA; ++q) acc[q] = wave_sum<8>(acc[q]);
      if (lane < 8) {
#pragma unroll
        for (int q = 0; q < R; ++q) {
          l.red[(w * NO + 2 * lane) * R + q] = acc[2 * q];
          l.red[(w * NO + 2 * lane + 1) * R + q] = acc[2 * q + 1];
        }
      }
      lds_barrier();  // [red]
      if (outp) {
#pragma unroll
        for (int q = 0; q < 8; ++q) out += l.red[q * NO * R + tid];
      }
    } else {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const double s = wave_sum<1>(acc[q]);
        if (lane == q) l.red[w * R + q] = s;
      }
      lds_barrier();  // [red]
      if (outp) out = l.red[tid];
    }
    if (outp) {
      const double v = g.isw ? out : base - out;
      st_sys(p.vec + (g.stage + 1) * vlen + g.hf * half + (int64_t)orow * R + orc, v);
      if (!T && g.isw && orc < p.nr) p.X[((int64_t)i * b + orow) * p.ldx + orc] = v;
    }
    lds_barrier();  // [end]: v and red are free for the next item
  } while (walk.more(l.seat));
}

template <int R, int U, bool T, int NP>
__global__ void __launch_bounds__(kSweepThreads + 64 * NP, 4) k_sweep(SweepArgs p) {
  __shared__ SweepLds<R, U, T> l;
  const int stages = sweep_stages(p.n, p.a, T);
  const int group = (int)blockIdx.x / p.seats, own = (int)blockIdx.x - group * p.seats;
  p.enter_group(R, group);
  if (threadIdx.x == 0) {
    l.dead = claim_seat(p.claims + own) != 0;
    l.seat[0] = own;
    l.victim = kSeats;
  }
  if constexpr (T)
    for (int e = threadIdx.x; e < p.a * R; e += blockDim.x)
      l.xa[e] = (e % R < p.nr) ? p.X[((int64_t)p.n * p.b + e / R) * p.ldx + e % R] : 0.0;
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(l.dead)) return;
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= kSweepThreads / 64) sweep_poller<R, U, T, NP>(p, l, stages, own);
  else sweep_worker<R, U, T, NP>(p, l, stages, own);
}

// Before a sweep: its fail word, the hand-over vectors (vector 0: the first block of the
// sweep, the others kPending) and the claims, and before a backward
// sweep x_a = T^-T y_a of all right-hand sides (`tip` > 0: their number), in
// place.
// (pieces: partial vectors per vector; the second one of vector 0 is zero)
__global__ void __launch_bounds__(BTA_THREADS) k_sweep_init(SweepArgs p, const double* x0, int R, int pieces,
                                                           int64_t vectors, int64_t nclaims, double* Xtip,
                                                           const double* tinv, int tip) {
  const int group = blockIdx.y;
  if (blockIdx.x == 0 && group == 0) {
    if (threadIdx.x == 0) *p.fail = 0;
    const int a = p.a, per = tip > 0 ? BTA_THREADS / a : 1;
    for (int c0 = 0; c0 < tip; c0 += per) {
      const int q = threadIdx.x / per, rc = c0 + threadIdx.x % per;
      const bool on = q < a && rc < tip;
      double s = 0.0;
      if (on)
        for (int r = q; r < a; ++r) s = fma(tinv[r * 64 + q], Xtip[(int64_t)r * p.ldx + rc], s);
      __syncthreads();
      if (on) Xtip[(int64_t)q * p.ldx + rc] = s;
      __syncthreads();
    }
  }
  p.enter_group(R, group);
  x0 += (int64_t)group * R;
  const int64_t len = (int64_t)p.b * R, pad = vec_len(p.b, R);
  const int64_t t0 = (int64_t)blockIdx.x * BTA_THREADS + threadIdx.x, stride = (int64_t)gridDim.x * BTA_THREADS;
  for (int64_t e = t0; e < vectors * pad; e += stride) {
    // + 0.0: a signalling NaN of the caller's becomes a quiet one
    if (e < len) p.vec[e] = (e % R < p.nr) ? x0[e / R * p.ldx + e % R] + 0.0 : 0.0;
    else if (e < pieces * pad) p.vec[e] = 0.0;
    else reinterpret_cast<unsigned long long*>(p.vec)[e] = kPending;
  }
  for (int64_t e = t0; e < nclaims; e += stride) p.claims[e] = 0;
}

// After a backward sweep: X_i = sum of the two partial vectors of W_i's stage.
__global__ void __launch_bounds__(BTA_THREADS) k_sweep_finish(SweepArgs p, int R) {
  p.enter_group(R, blockIdx.y);
  const int64_t len = (int64_t)p.b * R, pad = vec_len(p.b, R), tot = p.n * len;
  const int first = p.a > 0 ? 0 : 1;
  for (int64_t e = (int64_t)blockIdx.x * BTA_THREADS + threadIdx.x; e < tot; e += (int64_t)gridDim.x * BTA_THREADS) {
    const int64_t step = e / len, q = e % len;
    const double* v = p.vec + 2 * pad * (2 * step + 2 - first) + q;
    if (q % R < p.nr) p.X[((p.n - 1 - step) * p.b + q / R) * p.ldx + q % R] = v[0] + v[pad];
  }
}

// ---------------------------------------------------------- one workgroup
//
// Blocks up to kSolo: the vectors stay in the LDS of one workgroup (per group
// of R right-hand sides, one per grid entry), so a product costs two LDS
// barriers instead of a trip through memory.  The whole block row of L and of
// W sits in registers, each loaded while the other one's product runs.
//   forward:  8 threads per row, columns t % 8 + 8u
//   backward: 128 threads per column, rows t / 128 + 8u, summed through LDS
// All loads of a block are the same straight-line code whatever b is (the
// number of loads in flight stays known to the compiler): K >= b / 8 of them,
// those past the block clamped into it or, forward, cut off by the buffer
// descriptor's bounds check.
template <int R, int K, bool T>
__global__ void __launch_bounds__(kSoloThreads) k_sweep_solo(SweepArgs p, int nrhs) {
  __shared__ double sy[kSolo * R];  // result of the last W product
  __shared__ double sz[kSolo * R];  // operand of the next one
  __shared__ double sxa[T ? 64 * R : 1];
  __shared__ double red[T ? 8 * kSolo * R : 1];
  const int tid = threadIdx.x, n = p.n, b = p.b, a = p.a;
  double* X = p.X + (int64_t)blockIdx.x * R;
  const int nr = min(R, nrhs - (int)blockIdx.x * R);
  const int o = T ? tid & (kSolo - 1) : tid >> 3;  // output index of this thread
  const int pt = T ? __builtin_amdgcn_readfirstlane(tid / kSolo) : tid & 7;
  const int oc = min(o, b - 1);
  double ml[K], mw[K], mb[T ? 8 : 1], xv[R];
  // element (o, pt + 8u) of M (forward) / (pt + 8u, o) (backward)
  auto fetch = [&](double (&m)[K], const double* M) {
    if constexpr (T) {
#pragma unroll
      for (int u = 0; u < K; ++u) m[u] = (gview(M) + (int64_t)min(pt + 8 * u, b - 1) * b)[(unsigned)oc];
    } else {
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(M), 0, b * b * 8, 0x00020000);
#pragma unroll
      for (int u = 0; u < K; ++u) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, (oc * b + pt) * 8 + 64 * u, 0, 0);
        m[u] = __longlong_as_double(((long long)v[1] << 32) | (unsigned)v[0]);
      }
    }
  };
  auto fetch_x = [&](int i) {
#pragma unroll
    for (int q = 0; q < R; ++q) xv[q] = q < nr ? X[((int64_t)i * b + oc) * p.ldx + q] : 0.0;
    if constexpr (T) {
      const gdouble* g = gview(p.B) + (int64_t)i * a * b + oc;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (8 * u < a) mb[u] = g[(int64_t)min(pt + 8 * u, a - 1) * b];
    }
  };
  // sum over the matrix elements of this thread's output; lo / hi: valid k
  auto dot = [&](const double (&m)[K], const double* v, int lo, int hi, double (&acc)[R]) {
#pragma unroll
    for (int u = 0; u < K; ++u) {
      const int k = pt + 8 * u;
      const bool in = k >= lo && k < hi;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const double t = fma(m[u], v[k * R + q], acc[q]);
        acc[q] = in ? t : acc[q];
      }
    }
  };
  // combine the 8 threads of an output; returns whether this thread stores
  // element (so, sq), whose total is then in tot
  int so = o, sq = 0;
  auto combine = [&](double (&acc)[R], double& tot) -> bool {
    if constexpr (T) {
#pragma unroll
      for (int q = 0; q < R; ++q) red[(pt * kSolo + o) * R + q] = acc[q];
      lds_barrier();
      if (tid >= kSolo * R) return false;
      so = tid / R;
      sq = tid % R;
      tot = 0.0;
#pragma unroll
      for (int q = 0; q < 8; ++q) tot += red[q * kSolo * R + tid];
      return so < b;
    } else {
#pragma unroll
      for (int q = 0; q < R; ++q) acc[q] = sum8(acc[q]);
      tot = acc[0];
#pragma unroll
      for (int q = 1; q < R; ++q)
        if (pt == q) tot = acc[q];
      sq = pt;
      return pt < R && o < b;
    }
  };
  const int i0 = T ? n - 1 : 0, di = T ? -1 : 1;
  fetch(mw, p.W + (int64_t)i0 * b * b);
  if constexpr (T) {
    for (int e = tid; e < a * R; e += kSoloThreads)
      sxa[e] = (e % R < nr) ? X[((int64_t)n * b + e / R) * p.ldx + e % R] : 0.0;
    for (int e = tid; e < 64 * R; e += kSoloThreads)
      if (e >= a * R) sxa[e] = 0.0;
  }
  for (int e = tid; e < b * R; e += kSoloThreads) {
    const int64_t at = ((int64_t)i0 * b + e / R) * p.ldx + e % R;
    double v = (e % R < nr) ? X[at] : 0.0;
    if constexpr (T) {
      for (int q = 0; q < a; ++q)
        if (e % R < nr) v = fma(-p.B[((int64_t)i0 * a + q) * b + e / R], X[((int64_t)n * b + q) * p.ldx + e % R], v);
    }
    sz[e] = v;
  }
  if (n > 1) {
    fetch(ml, p.L + (int64_t)(T ? n - 2 : 0) * b * b);
    fetch_x(i0 + di);
  }
  lds_barrier();
  for (int s = 0, i = i0; s < n; ++s, i += di) {
    double acc[R], tot;
#pragma unroll
    for (int q = 0; q < R; ++q) acc[q] = 0.0;
    dot(mw, sz, T ? o : 0, T ? b : o + 1, acc);
    if (combine(acc, tot)) {
      sy[so * R + sq] = tot;
      if (sq < nr) X[((int64_t)i * b + so) * p.ldx + sq] = tot;
    }
    if (s == n - 1) break;
    fetch(mw, p.W + (int64_t)(i + di) * b * b);
    lds_barrier();
#pragma unroll
    for (int q = 0; q < R; ++q) acc[q] = 0.0;
    dot(ml, sy, 0, b, acc);
    if constexpr (T) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (8 * u < a && pt + 8 * u < a) {
#pragma unroll
          for (int q = 0; q < R; ++q) acc[q] = fma(mb[u], sxa[(pt + 8 * u) * R + q], acc[q]);
        }
    }
    // the vector the product is taken from, in the layout of the stores
    double xs = xv[0];
    if constexpr (!T) {
#pragma unroll
      for (int q = 1; q < R; ++q)
        if (pt == q) xs = xv[q];
    } else if constexpr (R > 1) {
      if (pt == 0) {
#pragma unroll
        for (int q = 0; q < R; ++q) sz[o * R + q] = xv[q];
      }
    }
    const bool st = combine(acc, tot);
    if (st) {
      if constexpr (T && R > 1) xs = sz[so * R + sq];
      sz[so * R + sq] = xs - tot;
    }
    if (s + 2 < n) {
      fetch(ml, p.L + (int64_t)(T ? i + 2 * di : i + 1) * b * b);
      fetch_x(i + 2 * di);
    }
    lds_barrier();
  }
}

// ----------------------------------------------------------------- the arrow
//
// y_a = T^-1 (r_a - sum_i B_i y_i), after the forward sweep has left every y_i
// in X: workgroup g sums a contiguous run of blocks into part[g][a][nr]; the
// last one to count itself adds the partial sums in order of g (the order of
// summation is fixed) and multiplies by T^-1, then resets the counter.
__global__ void __launch_bounds__(BTA_THREADS) k_sweep_arrow(SweepArgs p, const double* __restrict__ tinv,
                                                            double* part, int* cnt) {
  __shared__ double st[64 * 4];
  __shared__ int last_sh;
  const int n = p.n, b = p.b, a = p.a, nr = p.nr, G = gridDim.x, g = blockIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lo = (int)((int64_t)n * g / G), hi = (int)((int64_t)n * (g + 1) / G);
  for (int e = w; e < a * nr; e += 4) {
    const int q = e / nr, rc = e % nr;
    double acc = 0.0;
    for (int i = lo; i < hi; ++i) {
      const double* Bq = p.B + ((int64_t)i * a + q) * b;
      const double* x = p.X + (int64_t)i * b * p.ldx + rc;
#pragma unroll 4
      for (int c = lane; c < b; c += 64) acc = fma(Bq[c], x[(int64_t)c * p.ldx], acc);
    }
    acc = wave_sum<1>(acc);
    if (lane == 0) st_sys(part + (int64_t)g * a * nr + e, acc);
  }
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int before = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (before == G - 1) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    last_sh = before;
  }
  __syncthreads();
  if (last_sh != G - 1) return;
  double* xa = p.X + (int64_t)n * b * p.ldx;
  for (int c0 = 0; c0 < nr; c0 += 4) {
    const int q = threadIdx.x >> 2, rc = c0 + (threadIdx.x & 3);
    const bool on = q < a && rc < nr;
    if (on) {
      double s = 0.0;
      for (int h = 0; h < G; ++h) s += ld_sys(part + ((int64_t)h * a + q) * nr + rc);
      st[threadIdx.x] = xa[(int64_t)q * p.ldx + rc] - s;
    }
    __syncthreads();
    if (on) {
      double s = 0.0;
      for (int r = 0; r <= q; ++r) s = fma(tinv[q * 64 + r], st[4 * r + (threadIdx.x & 3)], s);
      xa[(int64_t)q * p.ldx + rc] = s;
    }
    __syncthreads();
  }
}

// Groups of R right-hand sides from column p.X on (p.nr in all), side by side
// as far as `groups` scratches and the CUs go.  Returns the columns done.
template <int R, int U, int NP>
int sweep_group(Workspace& ws, SweepArgs p, const double* x0, double* Xtip, int tip, int trans, int groups,
                hipStream_t st) {
  p.parts = sweep_parts(p.b, trans);
  // one workgroup per CU; two where a product has more items than that (their
  // rounds of loads then overlap: b = 4500 27 / 37 us per product forward /
  // backward against 35 / 48), which only the small R = 1, U = 8 form has the
  // registers for
  p.seats = std::min(p.parts, std::min(R == 1 && U == 8 && p.b > 2048 ? 2 * ws.cus : ws.cus, kSeats));
  const int64_t products = sweep_stages(p.n, p.a, trans), len = vec_len(p.b, R);
  const int64_t vectors = (products + 1) * (trans ? 2 : 1);
  p.gstride = vectors * len + kSeats / 2;
  groups = std::max(1, std::min({groups, (p.nr + R - 1) / R, ws.cus / p.seats}));
  p.nr = std::min(p.nr, groups * R);
  auto grid = [](int64_t e, int cap) {
    return dim3((unsigned)std::min<int64_t>((e + BTA_THREADS - 1) / BTA_THREADS, cap));
  };
  p.vec = ws.work;
  p.claims = reinterpret_cast<unsigned*>(ws.work + vectors * len);
  const int columns = p.nr;
  auto cover = [&](int64_t e) { return dim3(grid(e, 1024).x, groups); };
  hipLaunchKernelGGL(k_sweep_init, cover(vectors * len), dim3(BTA_THREADS), 0, st, p, x0, R, trans ? 2 : 1, vectors,
                     (int64_t)kSeats, Xtip, ws.tinv, tip);
  const dim3 wgs(p.seats * groups), th(kSweepThreads + 64 * NP);
  if (trans) {
    hipLaunchKernelGGL((k_sweep<R, U, true, NP>), wgs, th, 0, st, p);
    hipLaunchKernelGGL(k_sweep_finish, cover((int64_t)p.n * p.b * R), dim3(BTA_THREADS), 0, st, p, R);
  } else {
    hipLaunchKernelGGL((k_sweep<R, U, false, NP>), wgs, th, 0, st, p);
  }
  return columns;
}

template <int R, int K>
void sweep_solo(const SweepArgs& p, int nrhs, int trans, hipStream_t st) {
  const dim3 wgs((nrhs + R - 1) / R), th(kSoloThreads);
  if (trans) hipLaunchKernelGGL((k_sweep_solo<R, K, true>), wgs, th, 0, st, p, nrhs);
  else hipLaunchKernelGGL((k_sweep_solo<R, K, false>), wgs, th, 0, st, p, nrhs);
}

}  // namespace

static size_t group_doubles(int n, int b, int R) {
  return (2 * (size_t)n + 1) * 2 * (size_t)vec_len(b, R) + kSeats / 2;
}

// A scratch of 3 b^2 doubles, or 32 MB where that is more.
static size_t sweep_room(int b) { return std::max(3 * (size_t)b * b, (size_t)1 << 22); }

// Right-hand sides per group (8, 4 or 1): as many as fit the scratch.
static int group_size(int n, int b) {
  const size_t room = sweep_room(b);
  return group_doubles(n, b, 8) <= room ? 8 : (group_doubles(n, b, 4) <= room ? 4 : 1);
}

// Groups of that size that the scratch holds side by side: what fits as well, at
// most 4.
static int group_count(int n, int b) {
  return (int)std::max<size_t>(1, std::min<size_t>(4, sweep_room(b) / group_doubles(n, b, group_size(n, b))));
}

// Scratch of the sweeps in doubles (0: swept by single workgroups).
size_t sweep_doubles(int n, int b) {
  return b <= kSolo ? 0 : group_count(n, b) * group_doubles(n, b, group_size(n, b));
}

int potrs_enqueue(Workspace& ws, const double* L, const double* B, int n, int b, int a, double* rhs, int nrhs,
                  int ldrhs, int trans, hipStream_t st) {
  SweepArgs p;
  p.L = L;
  p.B = B;
  p.W = ws.wfull;
  p.X = rhs;
  p.vec = nullptr;
  p.claims = nullptr;
  p.fail = ws.sweep_fail;
  p.err = ws.solve_err;
  p.spin_ticks = ws.wait_ticks;
  p.n = n;
  p.b = b;
  p.a = a;
  p.ldx = ldrhs;
  p.nr = nrhs;
  p.parts = p.seats = 0;
  p.gstride = 0;
  double* Xtip = rhs + (int64_t)n * b * ldrhs;
  int tip = (trans && a > 0) ? nrhs : 0;
  TimedScope ts(ws, KC_GEMV, st);
  if (b <= kSolo) {
    if (tip)
      hipLaunchKernelGGL(k_sweep_init, dim3(1), dim3(BTA_THREADS), 0, st, p, nullptr, 1, 1, (int64_t)0,
                         (int64_t)0, Xtip, ws.tinv, tip);
    if (nrhs == 1) sweep_solo<1, 8>(p, nrhs, trans, st);
    else sweep_solo<4, 8>(p, nrhs, trans, st);
  } else {
    // Groups of 1, 4 or 8 right-hand sides share one pass over the factor, as
    // many groups side by side as the scratch and the CUs hold: the size whose
    // passes take the least (one of 1, 4 and 8 is as 1 : 1.6 : 2.5).  Measured on
    // MI355X, ms for 1, 4, 8, 16, 32 right-hand sides, in brackets with one
    // group of 4 or 8 after the other:
    //   n = 50, b = 92     0.31 0.32 0.32 0.35 0.68   (0.36 0.62 0.95 1.87 3.72)
    //   n = 40, b = 300    0.28 0.29 0.52 0.54 0.81   (0.32 0.60 0.91 1.80 3.57)
    //   n = 40, b = 800    0.45 0.68 0.67 1.02 2.08   (0.50 0.79 1.22 2.44 4.92)
    const double* x0 = rhs + (trans ? (int64_t)(n - 1) * b * ldrhs : 0);
    const int room = std::max(1, ws.cus / std::min((b + 7) / 8, ws.cus));
    auto slots = [&](int R) { return (int)std::min<size_t>(ws.work_doubles / group_doubles(n, b, R), room); };
    const int size[3] = {1, 4, 8}, cols[3] = {std::max(1, slots(1)), 4 * slots(4), 8 * slots(8)};
    const double pass[3] = {1.0, 1.6, 2.5};
    auto passes_of_one_size = [&](int left) {  // the least time for the rest
      double t = 0.0;
      for (int q = 0; q < 3; ++q)
        if (cols[q] > 0) {
          const double x = pass[q] * ((left + cols[q] - 1) / cols[q]);
          t = q == 0 ? x : std::min(t, x);
        }
      return t;
    };
    for (int c0 = 0; c0 < nrhs;) {
      int R = 1;
      double best = 0.0;
      for (int q = 0; q < 3; ++q) {
        if (cols[q] == 0) continue;
        const double t = pass[q] + passes_of_one_size(std::max(0, nrhs - c0 - cols[q]));
        if (q == 0 || t < best) {
          R = size[q];
          best = t;
        }
      }
      const int groups = slots(R);
      p.X = rhs + c0;
      p.nr = nrhs - c0;
      const double* x = x0 + c0;
      if (R == 1 && b <= 512) c0 += sweep_group<1, 4, 4>(ws, p, x, Xtip, tip, trans, groups, st);
      else if (R == 1 && (b <= 1024 || b > 2048)) c0 += sweep_group<1, 8, 4>(ws, p, x, Xtip, tip, trans, groups, st);
      else if (R == 1) c0 += sweep_group<1, 16, 4>(ws, p, x, Xtip, tip, trans, groups, st);
      else if (R == 4) c0 += sweep_group<4, 8, 4>(ws, p, x, Xtip, tip, trans, groups, st);
      else c0 += sweep_group<8, 8, 4>(ws, p, x, Xtip, tip, trans, groups, st);
      tip = 0;
    }
  }
  if (!trans && a > 0) {
    // partial sums in the scratch: column groups that fit it
    const int group = (int)std::max<size_t>(1, std::min<size_t>((size_t)nrhs, ws.work_doubles / a));
    for (int c0 = 0; c0 < nrhs; c0 += group) {
      p.X = rhs + c0;
      p.nr = std::min(group, nrhs - c0);
      const size_t fit = ws.work_doubles / ((size_t)a * p.nr);
      const int G = (int)std::max<size_t>(1, std::min<size_t>({fit, (size_t)n, (size_t)256}));
      hipLaunchKernelGGL(k_sweep_arrow, dim3(G), dim3(BTA_THREADS), 0, st, p, ws.tinv, ws.work, ws.sweep_count);
    }
  }
  return (int)hipGetLastError();
}

}  // namespace bta
