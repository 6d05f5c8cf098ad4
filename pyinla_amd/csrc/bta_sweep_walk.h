// Which work items of a triangular sweep a workgroup runs, and in what order:
// plain integer code, the same on the device (bta_potrs.hip) and in a host model
// that takes workgroups away.
//
// A sweep is a list of products ("stages"): per block the coupling with the
// block before it (L_{i-1} y_{i-1}, or L_i^T x_{i+1} + B_i^T x_a) and the
// product with W_i.  A stage is cut into work items; seat k of the launch owns
// items k, k + seats, ... of every stage.  (Items taken by ticket instead: two
// items of one stage often went to the same workgroup, which then ended 6 us
// after the others at b = 1600.)
//
// The launch must end whatever number of its workgroups the device keeps
// resident beside other kernels.  A workgroup therefore claims its seat when it
// starts, and before its first item of stage 1 it stands at a gate until every
// seat is claimed.  One that has waited there for 10 ms (another sweep of the
// same size would have made room by then) claims a seat that is still free, runs
// its items of stage 0, stands at the gate again, and from then on runs the items
// of all its seats in every stage; the workgroup the seat was meant for finds it
// taken and ends.  Nothing of stage 0 waits, and past the gate every seat belongs
// to a running workgroup, whose items of a stage wait for the stage before only:
// so by induction every stage completes.  (The gate looks at the claims and not
// at the outputs of stage 0: the items of a backward sweep's first triangular
// product read the rows from their own on, so that nobody reads what the first
// seats owe.)
#pragma once
#include <stdint.h>

namespace bta {

constexpr int kSeats = 512;  // at most

// Work items of a stage.  Forward: 8 rows, one per wave.  Backward: 16 columns
// of one half of the rows.
__host__ __device__ inline int sweep_parts(int b, bool trans) {
  return trans ? 2 * ((b + 15) / 16) : (b + 7) / 8;
}

// Stages: the first block has no coupling, but a backward sweep's has an arrow term.
__host__ __device__ inline int sweep_stages(int n, int a, bool trans) {
  return 2 * n - ((trans && a > 0) ? 0 : 1);
}

// Geometry of an item.
template <bool T>
struct SweepItem {
  int stage, part, i, out0, hf;
  bool isw, hasm;
  int kbeg, kend;  // vector range: what the item waits for of the stage before
  __host__ __device__ __forceinline__ SweepItem(int n, int b, int a, int stage_, int part_)
      : stage(stage_), part(part_) {
    constexpr int NO = T ? 16 : 8;
    // forward: W(0), L(0), W(1), ...; backward: the last block's arrow term
    // when there is an arrow, W(n-1), L(n-2), W(n-2), ...
    const int first = (T && a > 0) ? 0 : 1;
    isw = ((stage + first) & 1) != 0;  // product with W
    const int step = (stage + first) >> 1;
    i = T ? n - 1 - step : step;
    hasm = isw || !T || i < n - 1;  // the arrow term alone has no matrix
    hf = T ? part & 1 : 0;          // half of the rows
    out0 = NO * (T ? part >> 1 : part);
    kbeg = 0;
    kend = !hasm ? 0 : ((!T && isw) ? (out0 + NO < b ? out0 + NO : b) : b);
    if (T && hasm) {  // W is zero above its diagonal
      const int lo = isw ? out0 : 0, mid = (lo + b + 1) >> 1;
      kbeg = hf ? mid : lo;
      kend = hf ? b : mid;
    }
  }
};

// The items of a workgroup in order, the same in all its threads: its seats'
// items of a stage, then those of the next stage.
struct SweepWalk {
  int stages, parts, seats, count = 1, stage = 0, q = 0, part;
  bool open = false;  // past the gate
  __host__ __device__ __forceinline__ SweepWalk(int stages_, int parts_, int seats_, int seat)
      : stages(stages_), parts(parts_), seats(seats_), part(seat) {}
  __host__ __device__ __forceinline__ bool at_gate() const { return stage == 1 && !open; }
  // On to the next item; false past the last.  seat[0 .. count-1]: the workgroup's seats.
  __host__ __device__ __forceinline__ bool more(const int* seat) {
    part += seats;
    if (part < parts) return true;
    if (++q == count) {
      q = 0;
      ++stage;
    }
    part = __builtin_amdgcn_readfirstlane(seat[q]);
    return stage < stages;
  }
  // At the gate: the walk goes on with the stage-0 items of one more seat and
  // comes back to the gate after them.
  __host__ __device__ __forceinline__ void take_over(int seat) {
    stage = 0;
    q = count++;
    part = seat;
  }
};

}  // namespace bta
