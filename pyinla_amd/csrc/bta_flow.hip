// Persistent dataflow panel factorization (see bta_flow.h for the scheme).
//
// Replaces the nT launches per block of the column-by-column panel with one
// launch of 1 + P resident workgroups: the chain (workgroup 0) runs the
// diagonal Cholesky + inverse, TRSM of the sub-diagonal tile and the rank-64
// update of the next diagonal tile back to back, while P helpers work through
// their task lists.  Same algorithm and outputs as the per-column path
// (the published pobtaf block loop: POTRF of D_i, TRSM of L_i and B_i, then the
// updates of D_{i+1}, B_{i+1} and T; called by the reference at
// structured_solver.py:83-88): L_ii in D_i,
// L_{i+1,i} in L_i, L_{a,i} in B_i, inverse of every diagonal tile in winv and
// per-tile log-pivot sums in logpart.
#include <algorithm>
#include <queue>

#include "bta_internal.h"
#include "bta_flow.h"
#include "bta_tile_chol.h"

namespace bta {

// ---------------------------------------------------------------- schedule

// Ownership.  The tiles on the chain's path -- (c, c), (c+1, c) and (c+2, c)
// of D, whose updates and solves the chain waits for one or two columns later
// -- are dealt round-robin over a small pool of "near" helpers that own
// nothing else, so none of their tasks ever queues behind bulk work.  All
// other tiles are dealt round-robin in column-major order (column c: D rows
// c+3..nT-1, then the L and arrow rows) over the remaining helpers, so each of
// them owns tiles spread evenly over the columns and its share of every
// column's updates stays balanced; the next-block updates go to the same
// pool.  Cleared upper tiles of D go by row-major index.
// Pool size: helpers / near_div, but at least min(10, helpers / 8).  Measured
// on MI355X (factorization pair on two streams, 255 helpers each): 31 near
// helpers 1.42 ms per block pair at b = 2000 and 15.8 ms at b = 4500; 15-21
// helpers 1.34 / 15.3; 10 helpers 1.33 / 15.0; 7 helpers 1.65 (too few: the
// chain waits on them).  The floor keeps about 10 for the smaller helper
// counts of batched launches.
static int flow_near_pool(const FlowShape& s, int helpers) {
  const int div = s.near_div > 0 ? s.near_div : 16;
  if (helpers < 8) return 0;
  return std::min(3 * s.nT, std::max(helpers / div, std::min(10, helpers / 8)));
}

static bool flow_is_near(int nT, int rho, int c) { return rho < nT && rho >= c && rho - c <= 2; }

int flow_owner(const FlowShape& s, int rho, int c, int helpers) {
  const int nT = s.nT, below = s.nTL + s.nTa;
  if (rho < nT && rho < c) return (int)(((long long)rho * nT + c) % helpers);
  const int hn = flow_near_pool(s, helpers);
  if (hn > 0 && flow_is_near(nT, rho, c)) return (3 * c + (rho - c)) % hn;
  long long t = 0;  // column-major index among the other tiles
  for (int cc = 0; cc < c; ++cc) {
    const int nd = nT - cc;
    t += (hn > 0 ? nd - std::min(3, nd) : nd) + below;
  }
  if (rho < nT) t += hn > 0 ? rho - c - 3 : rho - c;
  else t += (hn > 0 ? std::max(0, nT - c - 3) : nT - c) + (rho - nT);
  return hn + (int)(t % (helpers - hn));
}

// Owner of a next-block update target (never a near helper).
static int flow_next_owner(const FlowShape& s, int rho, int c, int helpers) {
  const int hn = flow_near_pool(s, helpers);
  const long long t = (long long)rho * (s.nT + 1) + c;
  return hn + (int)(t % (helpers - hn));
}

// Level order (delta >= 1): each helper runs its tasks by dependency level;
// far tiles take their updates in groups of `delta` columns.
static void flow_build_levels(const FlowShape& s, int helpers, int delta, FlowSchedule& out) {
  struct Item {
    unsigned long long key;
    uint32_t word;
    int h;
  };
  std::vector<Item> v;
  const int nT = s.nT, R = s.rows();
  const int hn = flow_near_pool(s, helpers);  // near tiles are never grouped
  auto push = [&](int level, int prio, int op, int rho, int c, int k) {
    const unsigned long long key = ((unsigned long long)level << 42) | ((unsigned long long)prio << 31) |
                                   ((unsigned long long)c << 21) | ((unsigned long long)rho << 10) |
                                   (unsigned long long)k;
    v.push_back({key, flow_encode(op, rho, c, k), flow_owner(s, rho, c, helpers)});
  };
  // next-block updates: one task per target tile and span of S columns of
  // L_i / B_i, at the level of the span's last column, lowest priority
  auto push_next = [&](int rho, int c) {
    for (int k = 0; k < nT; k = flow_next_end(k, nT)) {
      const int klast = flow_next_end(k, nT) - 1;
      const unsigned long long key = ((unsigned long long)(3 * klast + 2) << 42) | (1023ull << 31) |
                                     ((unsigned long long)c << 21) | ((unsigned long long)rho << 10) |
                                     (unsigned long long)k;
      v.push_back({key, flow_encode(FLOW_NEXT, rho, c, k), flow_next_owner(s, rho, c, helpers)});
    }
  };
  if (s.fold && s.nTL > 0) {
    for (int r = 0; r < nT; ++r)
      for (int c = 0; c <= r; ++c) push_next(r, c);
    if (s.nTa > 0)
      for (int c = 0; c < nT; ++c) push_next(nT, c);
  }
  if (s.fold && s.nTa > 0) push_next(nT + 1, 0);
  for (int rho = 0; rho < R; ++rho) {
    for (int c = 0; c < nT; ++c) {
      if (rho < nT && rho < c) {  // strict upper tile of D: cleared
        push(0, 0, FLOW_ZERO, rho, c, 0);
        continue;
      }
      const bool diag = (rho == c);
      const bool hand = flow_is_handoff(nT, rho, c);
      const int cap = diag ? c - 2 : c - 1;
      for (int j = 0; j < c; ++j) {
        if (diag && j == c - 1) continue;  // applied by the chain
        // far tiles take their updates in groups of `delta` columns at the
        // group's last column: consecutive in the owner's list, so the
        // accumulator stays in registers across the group
        const int grp = (hn > 0 && flow_is_near(nT, rho, c)) ? 1 : std::max(delta, 1);
        const int round = hand ? j : std::min((j / grp + 1) * grp - 1, cap);
        const int prio = hand ? 0 : 1 + (c - round);
        push(3 * round + 2, prio, FLOW_UPD, rho, c, j);
      }
      if (!diag && !(rho < nT && rho == c + 1)) push(3 * c + 1, rho - c, FLOW_TRSM, rho, c, c);
    }
  }
  std::stable_sort(v.begin(), v.end(), [](const Item& x, const Item& y) {
    return x.h != y.h ? x.h < y.h : x.key < y.key;
  });
  out.helpers = helpers;
  out.tasks.resize(v.size());
  out.off.assign(helpers + 1, 0);
  for (size_t q = 0; q < v.size(); ++q) {
    out.tasks[q] = v[q].word;
    out.off[v[q].h + 1] += 1;
  }
  for (int h = 0; h < helpers; ++h) out.off[h + 1] += out.off[h];
}

// List order (delta == 0).  The launch is simulated on the host with the task
// costs below (core clock cycles, from s_memtime stamps on MI355X): whenever a
// helper is idle it starts the ready task of highest upward rank (its cost
// plus the longest path of costs and flag latencies from it to the end of the
// launch), so the solves and updates the chain is about to wait for come
// before bulk updates of tiles needed much later and the next-block updates
// fill the gaps.  Each helper's list is the order of its tasks in that
// simulation.  The costs and the group size were tuned together on MI355X: with
// the costs of a slower update (12 k, of which 3 k are saved by a carried
// accumulator, solve 14.5 k, groups of 2) a lone factorization takes 638 us per
// block at b = 2000 and a pair 1026; with these 550 and 883 (b = 1600: 379 and
// 372; b <= 800: the chain's time per column either way).  Solve costs of 12, 16,
// 20 k: 591, 573, 564 at groups of 8; groups of 4, 8, 12, 16: 609, 584, 567, 599;
// a margin of 0, 2, 3 instead of 1: 2-4 % slower.
// The simulated start times order all tasks, the chain's included, consistently
// with every dependency and with every list, so with all workgroups resident the
// earliest unfinished task in that order can always run, whatever the real
// durations: no interleaving can deadlock.
#ifndef FLOW_COST_CHOL
#define FLOW_COST_CHOL 21000  // chain: factor + inverse of a diagonal tile, stores, publish
#endif
#ifndef FLOW_COST_CTRSM
#define FLOW_COST_CTRSM 8000  // chain: solve of the sub-diagonal tile, stores
#endif
#ifndef FLOW_COST_CUPD
#define FLOW_COST_CUPD 4500  // chain: update of the next diagonal tile
#endif
#ifndef FLOW_COST_UPD
#define FLOW_COST_UPD 9000  // rank-64 update, accumulator loaded and stored
#endif
#ifndef FLOW_COST_CARRY
#define FLOW_COST_CARRY 5000  // saved when the previous task left the accumulator in registers
#endif
#ifndef FLOW_COST_TRSM
#define FLOW_COST_TRSM 24000  // tile solve (11 k), exchange copy, and what a helper behind in its list waits
#endif
#ifndef FLOW_COST_NEXTCOL
#define FLOW_COST_NEXTCOL 6000  // one column of a next-block task
#endif
#ifndef FLOW_COST_ZERO
#define FLOW_COST_ZERO 500
#endif
#ifndef FLOW_UPD_GROUP
#define FLOW_UPD_GROUP 10  // columns per held-back update group
#endif
#ifndef FLOW_UPD_MARGIN
#define FLOW_UPD_MARGIN 1  // the updates by the last columns before a tile's own are not held back
#endif
#ifndef FLOW_COST_LAT
#define FLOW_COST_LAT 1500  // flag store to flag seen by another workgroup
#endif

static bool flow_build_list(const FlowShape& s, int helpers, FlowSchedule& out) {
  const int nT = s.nT, R = s.rows();
  const int chain = helpers;  // agent id of the chain
  std::vector<uint32_t> word;
  std::vector<int> agent, cost, tile, op;
  auto add = [&](int a, int c, int o, uint32_t w, int t) {
    agent.push_back(a);
    cost.push_back(c);
    op.push_back(o);
    word.push_back(w);
    tile.push_back(t);
    return (int)agent.size() - 1;
  };
  std::vector<std::vector<int>> succ;
  std::vector<int> npred;
  auto edge = [&](int from, int to) {
    if (from < 0 || to < 0) return;
    if ((int)succ.size() < (int)agent.size()) succ.resize(agent.size());
    succ[from].push_back(to);
  };
  // chain: CF(k) factor, CT(k) solve of (k+1, k), CU(k) update of (k+1, k+1)
  std::vector<int> cf(nT, -1), ct(nT, -1), cu(nT, -1);
  for (int k = 0; k < nT; ++k) {
    cf[k] = add(chain, FLOW_COST_CHOL, -1, 0, -1);
    if (k + 1 < nT) {
      ct[k] = add(chain, FLOW_COST_CTRSM, -1, 0, -1);
      cu[k] = add(chain, FLOW_COST_CUPD, -1, 0, -1);
    }
  }
  // producer of X(rho, c); last helper update of each tile
  std::vector<int> xprod((size_t)R * nT, -1), last_upd((size_t)R * nT, -1);
  std::vector<std::pair<int, int>> upd_in;  // (task, j) for the X edges
  for (int k = 0; k + 1 < nT; ++k) xprod[(size_t)(k + 1) * nT + k] = ct[k];
  for (int rho = 0; rho < R; ++rho)
    for (int c = 0; c < nT; ++c) {
      const int owner = flow_owner(s, rho, c, helpers);
      const int tid = rho * nT + c;
      if (rho < nT && rho < c) {
        add(owner, FLOW_COST_ZERO, FLOW_ZERO, flow_encode(FLOW_ZERO, rho, c, 0), -1);
        continue;
      }
      const bool diag = (rho == c);
      const bool hand = flow_is_handoff(nT, rho, c);
      int prev = -1;
      for (int j = 0; j < c; ++j) {
        if (diag && j == c - 1) continue;  // applied by the chain
        const int t = add(owner, FLOW_COST_UPD, FLOW_UPD, flow_encode(FLOW_UPD, rho, c, j), hand ? -1 : tid);
        upd_in.push_back({t, j});
        edge(prev, t);  // one accumulator: updates of a tile in column order
        prev = t;
      }
      last_upd[tid] = prev;
      if (!diag && !(rho < nT && rho == c + 1)) {
        const int t = add(owner, FLOW_COST_TRSM, FLOW_TRSM, flow_encode(FLOW_TRSM, rho, c, c), tid);
        edge(prev, t);
        // inv(L_cc) is published right after the chain's factorization
        edge(cf[c], t);
        xprod[tid] = t;
      }
    }
  // next-block updates: one task per target and span of columns.  Each
  // target goes to the helper outside the near pool with the least work so
  // far.  (Given to the near pool as gap filler, they ran when the chain's
  // solves were already due -- the device takes longer than the simulated
  // costs -- and the chain waited on them: measured on MI355X at b = 2000,
  // keeping them off the near pool cut the chain's wait per column from
  // 19 k to 8 k cycles.)
  std::vector<double> load(helpers + 1, 0.0);
  for (size_t t = 0; t < agent.size(); ++t) load[agent[t]] += cost[t];
  const int hn_next = flow_near_pool(s, helpers);
  auto push_next = [&](int rho, int c) {
    const int ra = rho < nT ? nT + rho : nT + s.nTL;
    const int rb = rho < nT ? nT + c : (rho == nT ? nT + c : nT + s.nTL);
    int owner = hn_next;
    for (int h = owner + 1; h < helpers; ++h)
      if (load[h] < load[owner]) owner = h;
    load[owner] += (double)FLOW_COST_NEXTCOL * nT;
    int prev = -1;
    for (int k = 0; k < nT; k = flow_next_end(k, nT)) {
      const int kend = flow_next_end(k, nT);
      const int t = add(owner, FLOW_COST_NEXTCOL * (kend - k), FLOW_NEXT, flow_encode(FLOW_NEXT, rho, c, k), -1);
      edge(prev, t);
      prev = t;
      for (int kk = k; kk < kend; ++kk) {
        edge(xprod[(size_t)ra * nT + kk], t);
        if (rb != ra) edge(xprod[(size_t)rb * nT + kk], t);
      }
    }
  };
  succ.resize(agent.size());
  for (auto& u : upd_in) {
    int o, rho, c, j;
    flow_decode(word[u.first], o, rho, c, j);
    edge(xprod[(size_t)rho * nT + j], u.first);
    if (rho != c) edge(xprod[(size_t)c * nT + j], u.first);
    // Updates of a tile by columns far from its own are held back to the
    // last column of their group of FLOW_UPD_GROUP: the helper then applies
    // the group back to back with the accumulator kept in registers (one
    // load and one store of the tile per group instead of per column).  Only
    // the simulated order sees these edges; the device waits for the real
    // flags.
    const int g1 = std::min((j / FLOW_UPD_GROUP + 1) * FLOW_UPD_GROUP - 1, c - 1 - FLOW_UPD_MARGIN);
    if (g1 > j && !flow_is_handoff(nT, rho, c)) {
      edge(xprod[(size_t)rho * nT + g1], u.first);
      if (rho != c) edge(xprod[(size_t)c * nT + g1], u.first);
    }
  }
  if (s.fold && s.nTL > 0) {
    for (int r = 0; r < nT; ++r)
      for (int c = 0; c <= r; ++c) push_next(r, c);
    if (s.nTa > 0)
      for (int c = 0; c < nT; ++c) push_next(nT, c);
  }
  if (s.fold && s.nTa > 0) push_next(nT + 1, 0);
  succ.resize(agent.size());
  // chain order and its waits on the hand-off tiles
  for (int k = 0; k < nT; ++k) {
    if (k + 1 < nT) {
      edge(cf[k], ct[k]);
      edge(ct[k], cu[k]);
      edge(cu[k], cf[k + 1]);
      if (k >= 1) {  // the chain fetches both hand-off tiles before the solve
        edge(last_upd[(size_t)(k + 1) * nT + k], ct[k]);
        edge(last_upd[(size_t)(k + 1) * nT + k + 1], ct[k]);
      }
    }
  }
  const int N = (int)agent.size();
  npred.assign(N, 0);
  for (int t = 0; t < N; ++t)
    for (int v : succ[t]) ++npred[v];
  // topological order, then upward ranks
  std::vector<int> topo;
  topo.reserve(N);
  {
    std::vector<int> np = npred;
    for (int t = 0; t < N; ++t)
      if (np[t] == 0) topo.push_back(t);
    for (size_t q = 0; q < topo.size(); ++q)
      for (int v : succ[topo[q]])
        if (--np[v] == 0) topo.push_back(v);
  }
  if ((int)topo.size() != N) return false;  // dependency cycle
  std::vector<double> rank(N, 0.0);
  for (int q = N - 1; q >= 0; --q) {
    const int t = topo[q];
    double m = 0.0;
    for (int v : succ[t]) m = std::max(m, rank[v] + (agent[v] != agent[t] ? FLOW_COST_LAT : 0));
    rank[t] = cost[t] + m;
  }
  // list-scheduling simulation
  const int A = helpers + 1;
  using RQ = std::priority_queue<std::pair<double, int>>;                       // (rank, -task)
  using FQ = std::priority_queue<std::pair<double, int>, std::vector<std::pair<double, int>>,
                                 std::greater<std::pair<double, int>>>;         // (ready time, task)
  std::vector<RQ> ready(A);
  std::vector<FQ> future(A);
  std::vector<double> rtime(N, 0.0), busy(A, -1.0);
  std::vector<int> carried(A, -1), left = npred;
  std::vector<std::vector<int>> order(A);
  struct Ev {
    double t;
    int kind, x;  // kind 0: task x finishes, 1: agent x looks for work
    bool operator>(const Ev& o) const { return t != o.t ? t > o.t : kind > o.kind; }
  };
  std::priority_queue<Ev, std::vector<Ev>, std::greater<Ev>> ev;
  for (int t = 0; t < N; ++t)
    if (left[t] == 0) future[agent[t]].push({0.0, t});
  for (int a = 0; a < A; ++a) ev.push({0.0, 1, a});
  int done = 0;
  while (!ev.empty()) {
    const Ev e = ev.top();
    ev.pop();
    if (e.kind == 0) {
      const int t = e.x, a = agent[t];
      ++done;
      for (int v : succ[t]) {
        rtime[v] = std::max(rtime[v], e.t + (agent[v] != a ? FLOW_COST_LAT : 0));
        if (--left[v] == 0) {
          future[agent[v]].push({rtime[v], v});
          ev.push({rtime[v], 1, agent[v]});
        }
      }
      ev.push({e.t, 1, a});
      continue;
    }
    const int a = e.x;
    if (busy[a] > e.t) continue;  // still running a task; its finish re-posts
    while (!future[a].empty() && future[a].top().first <= e.t) {
      const int t = future[a].top().second;
      future[a].pop();
      ready[a].push({rank[t], -t});
    }
    if (ready[a].empty()) continue;  // woken again when a task becomes ready
    const int t = -ready[a].top().second;
    ready[a].pop();
    int c = cost[t];
    if (tile[t] >= 0 && tile[t] == carried[a]) c -= FLOW_COST_CARRY;
    carried[a] = (op[t] == FLOW_UPD && tile[t] >= 0) ? tile[t] : -1;
    busy[a] = e.t + c;
    order[a].push_back(t);
    ev.push({busy[a], 0, t});
  }
  if (done != N) return false;
  out.helpers = helpers;
  out.tasks.clear();
  out.off.assign(helpers + 1, 0);
  for (int h = 0; h < helpers; ++h) {
    for (int t : order[h]) out.tasks.push_back(word[t]);
    out.off[h + 1] = (int)out.tasks.size();
  }
  return true;
}

bool flow_build_schedule(const FlowShape& s, int helpers, int delta, FlowSchedule& out) {
  if (delta >= 1) {
    flow_build_levels(s, helpers, delta, out);
    return true;
  }
  return flow_build_list(s, helpers, out);
}

// ------------------------------------------------------------------ device

__device__ __forceinline__ double* flow_tile(const FlowArgs& p, int rho, int c, int& rows, int& cols) {
  cols = min(64, p.b - 64 * c);
  if (rho < p.nT) {
    rows = min(64, p.b - 64 * rho);
    return p.D + (int64_t)(64 * rho) * p.b + 64 * c;
  }
  rho -= p.nT;
  if (rho < p.nTL) {
    rows = min(64, p.b - 64 * rho);
    return p.L + (int64_t)(64 * rho) * p.b + 64 * c;
  }
  rho -= p.nTL;
  rows = min(64, p.a - 64 * rho);
  return p.B + (int64_t)(64 * rho) * p.b + 64 * c;
}

__device__ __forceinline__ int flow_rows(const FlowArgs& p) { return p.nT + p.nTL + p.nTa; }
__device__ __forceinline__ double* xtile(const FlowArgs& p, int rho, int c) {
  return p.xbuf + ((int64_t)rho * p.nT + c) * 4096;
}
__device__ __forceinline__ unsigned long long* xflag(const FlowArgs& p, int rho, int c) {
  return p.flags + (int64_t)rho * p.nT + c;
}
__device__ __forceinline__ unsigned long long* wflag(const FlowArgs& p, int k) {
  return p.flags + (int64_t)flow_rows(p) * p.nT + k;
}
__device__ __forceinline__ unsigned long long* hflag(const FlowArgs& p, int k, int s) {
  return p.flags + (int64_t)flow_rows(p) * p.nT + p.nT + 2 * k + s;
}
__device__ __forceinline__ double* hsub(const FlowArgs& p, int c) { return p.hacc + (int64_t)c * 4096; }
__device__ __forceinline__ double* hdiag(const FlowArgs& p, int c) {
  return p.hacc + ((int64_t)p.nT + c) * 4096;
}

// Bounded wait of the calling lane for *flag == tag (nullptr: nothing to wait
// for).  Gives up (returns 0 and raises err) after spin_ticks, or, after a 1024th
// of them, when another workgroup has raised err (polled by every wave from the
// start, that one word would be a hot spot), so that every workgroup still
// reaches the end of its list.
__device__ __forceinline__ int flow_poll(const FlowArgs& p, unsigned long long* flag, unsigned long long tag) {
  if (flag == nullptr) return 1;
  if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == tag) return 1;
  const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
  while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != tag) {
    const unsigned long long dt = __builtin_amdgcn_s_memrealtime() - t0;
    if (dt > p.spin_ticks >> 10 && __hip_atomic_load(p.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0) return 0;
    if (dt > p.spin_ticks) {
      atomicOr(p.err, 1);
      return 0;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  return 1;
}

// The workgroup waits until both flags are set (f2 may be nullptr).  The
// barriers order LDS only: the guarded data are read after the second one in
// program order, and a full barrier would also wait for every global load the
// workgroup has in flight (the prefetched accumulator of the step).
__device__ __forceinline__ bool flow_wait2(const FlowArgs& p, unsigned long long* f1, unsigned long long* f2,
                                           unsigned long long tag, int* ok_sh) {
  if (threadIdx.x < 64) {  // lanes 0 and 1 poll one flag each, side by side
    const int ok = threadIdx.x < 2 ? flow_poll(p, threadIdx.x == 0 ? f1 : f2, tag) : 1;
    const bool all = __ballot(ok == 0) == 0;
    if (threadIdx.x == 0) *ok_sh = all ? 1 : 0;
  }
  lds_barrier();
  const int ok = *ok_sh;
  lds_barrier();
  return ok != 0;
}

// Stores, after the caller's st_sys data stores, the flag once they completed.
__device__ __forceinline__ void flow_publish(unsigned long long* flag, unsigned long long tag) {
  flag_publish(flag, tag);
}

// X = C inv(L_kk)^T, rows 16w .. 16w+15 by wave w: C in sC, inv(L_kk) (lower) in
// sW.  Element q of x.c[cb / 2][cb % 2] is row 16w + 4q + lane / 16, column
// 16cb + lane % 16.  The
// triangular inverse leaves 10 of 16 block products: 40 MFMAs for every wave
// (split in 32 x 32 quadrants, two of the waves have 64).
__device__ __forceinline__ void tile_solve(TileAcc& x, const double* sC, const double* sW, int w, int lane) {
  const int li = lane & 15, lk = lane >> 4;
  double a[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) a[t] = sC[(16 * w + li) * BTA_LDS_LD + 4 * t + lk];
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) x.c[cb >> 1][cb & 1] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int m = 0; m < 4; ++m) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int cb = m; cb < 4; ++cb)
        x.c[cb >> 1][cb & 1] = mfma_f64(a[4 * m + t], sW[(16 * cb + li) * BTA_LDS_LD + 16 * m + 4 * t + lk],
                                        x.c[cb >> 1][cb & 1]);
    __builtin_amdgcn_sched_barrier(0);  // bounds the operands read ahead (registers)
  }
}

// Stores of tile_solve's result: factor tile (rows x cols of it, row stride ld)
// and exchange tile.
__device__ __forceinline__ void solve_store(const TileAcc& x, double* g, int64_t ld, int rows, int cols, int w,
                                            int lane) {
  const int i0 = 16 * w + (lane >> 4), j0 = lane & 15;
  gdouble* t = gview(g) + (int64_t)i0 * ld + j0;
  if (rows == 64 && cols == 64) {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int q = 0; q < 4; ++q) t[4 * q * ld + 16 * cb] = x.c[cb >> 1][cb & 1][q];
  } else {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (i0 + 4 * q < rows && j0 + 16 * cb < cols) t[4 * q * ld + 16 * cb] = x.c[cb >> 1][cb & 1][q];
  }
}
// Exchange tiles hold X in the order of MFMA operands: element (i, k) of a 64x64
// tile at x_index(i, k).  Row block i / 16, k steps 2u and 2u + 1 as a pair: one
// 16-byte load per lane, 1 KB per wave.  Within that KB the rows go in fours,
// so that a store of the accumulator layout writes two runs of 256 bytes (by row
// it would be 64-byte pieces, which took the chain 1 us longer per column to
// complete).
__device__ __forceinline__ int x_lane(int lane) { return ((lane >> 2) & 3) * 32 + (lane >> 4) * 8 + (lane & 3) * 2; }
__device__ __forceinline__ int x_index(int i, int k) {
  return (i >> 4) * 1024 + (k >> 3) * 128 + x_lane((i & 15) + 16 * (k & 3)) + ((k >> 2) & 1);
}
__device__ __forceinline__ void solve_store_x(const TileAcc& x, double* g, int w, int lane) {
  double* t = g + x_index(16 * w + (lane >> 4), lane & 15);
#pragma unroll
  for (int cb = 0; cb < 4; ++cb)
#pragma unroll
    for (int q = 0; q < 4; ++q) st_sys(t + 32 * q + 256 * cb, x.c[cb >> 1][cb & 1][q]);
}

// Chain: store the factored diagonal tile k held in sA (L_kk) / sB (inverse).
// The flag is published separately (chain_flag), so that the write-through
// stores drain while the chain already computes.
__device__ __forceinline__ void chain_store_inv(const FlowArgs& p, int k, const double* sB) {
  double* w = p.winv + (int64_t)k * 4096;
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
#pragma unroll
  for (int h = 0; h < 16; h += 8) {  // two halves of 8 rows: reads first, then stores
    double v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = sB[(r0 + 4 * (h + j)) * BTA_LDS_LD + c];
#pragma unroll
    for (int j = 0; j < 8; ++j) st_sys(&w[(r0 + 4 * (h + j)) * 64 + c], v[j]);
  }
}

// ... then, after the inverse's flag, L_kk to the factor (no helper reads it;
// the strict upper triangle as zeros, whatever sA holds there).
__device__ __forceinline__ void chain_store_l(const FlowArgs& p, int k, const double* sA) {
  int rows, cols;
  double* g = flow_tile(p, k, k, rows, cols);
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
  gdouble* t = gview(g) + (int64_t)r0 * p.b + c;
#pragma unroll
  for (int h = 0; h < 16; h += 8) {
    double v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = r0 + 4 * (h + j);
      const double x = sA[r * BTA_LDS_LD + c];
      v[j] = c <= r ? x : 0.0;
    }
    if (rows == 64) {
#pragma unroll
      for (int j = 0; j < 8; ++j) t[(int64_t)4 * (h + j) * p.b] = v[j];
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (r0 + 4 * (h + j) < rows && c < cols) t[(int64_t)4 * (h + j) * p.b] = v[j];
    }
  }
}

// The log pivots of tile k from its diagonal (lane i: l_ii), by one wave.
__device__ __forceinline__ void chain_log(const FlowArgs& p, int k, double lii) {
  const TileCholResult res = tile_log_pivots(lii, min(64, p.b - 64 * k));
  if ((threadIdx.x & 63) == 0) {
    p.logpart[k] = res.logsum;
    if (res.fail >= 0) atomicMin(p.info, (unsigned long long)(p.row0 + (long long)k * 64 + res.fail));
  }
}

// Current value of a flag (`tag` for an absent flag).
__device__ __forceinline__ unsigned long long flag_value(const unsigned long long* f, unsigned long long tag) {
  return f == nullptr ? tag
                      : __hip_atomic_load(const_cast<unsigned long long*>(f), __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_SYSTEM);
}

// 16x16 block (bi, bj), bi >= bj, of the lower triangle of a rows x rows
// row-major tile (0 outside it) in the accumulator layout; a diagonal block is
// mirrored.  (Clamped addresses and selects: loads under tests are waited for
// one by one.)
__device__ __forceinline__ f64x4 block_load(const double* __restrict__ g, int ld, int rows, int bi, int bj, int lane) {
  f64x4 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i0 = 16 * bi + 4 * q + (lane >> 4), j0 = 16 * bj + (lane & 15);
    const int i = max(i0, j0), j = min(i0, j0);
    const double x = gview(g)[(unsigned)(min(i, rows - 1) * ld + min(j, rows - 1))];
    v[q] = i < rows ? x : 0.0;
  }
  return v;
}

// Per column k the chain
//   1. waits for the hand-off tiles (k+1, k) and (k+1, k+1) (updated by their
//      helpers through column k-1), issues the loads of both and meanwhile
//      stores L_kk into the factor;
//   2. solves X = C(k+1, k) inv(L_kk)^T, 16 rows per wave, so that a wave's rows
//      of C and X are its own and nothing waits for another wave until X is
//      complete;
//   3. applies C(k+1, k+1) -= X X^T, lower 16x16 blocks only: wave 0 takes the
//      first block and factors it at once; the others take three blocks each,
//      store X and publish it (the helpers' updates of the next hand-off tile
//      wait for it);
//   4. factors the rest of C(k+1, k+1), stores its inverse and publishes it at
//      once (the helpers' solves of column k+1 wait for it).  The log pivots of
//      tile k are taken by wave 3 beside the last 16x16 factorization.
// Measured on MI355X at b = 417, us per column: 15.1, against 20.7 with both
// products as 32 x 32 quadrants one after the other, X published behind them, L
// stored and the logarithms taken before the next wait, and the 16x16 blocks
// factored by column.
__device__ __forceinline__ void flow_chain(const FlowArgs& p, unsigned long long tag, double* sA, double* sB,
                           int* ok_sh) {
  const int nT = p.nT;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  {
    int rows, cols;
    const double* g = flow_tile(p, 0, 0, rows, cols);
    TileAcc acc;
    acc_load(acc, g, p.b, rows, cols);
    acc_to_lds(acc, sA);
    __syncthreads();
    tile_chol_inv(sA, sB, rows);
    chain_store_inv(p, 0, sB);
    flow_publish(wflag(p, 0), tag);
  }
  // blocks of the diagonal tile that wave w updates (wave 0: only the first)
  const int bi0 = w, bj0 = 0;
  const int bi1 = max(w, 1), bj1 = 1;
  const int bi2 = w == 1 ? 3 : max(w, 2), bj2 = w == 1 ? 3 : 2;
  bool ready = true;  // the hand-off flags of this column were seen set
  for (int k = 0; k + 1 < nT; ++k) {
    const int mv = min(64, p.b - 64 * (k + 1));
    int rows, cols;
    double* gx = flow_tile(p, k + 1, k, rows, cols);
    const double* gc = gx;
    const double* gd = flow_tile(p, k + 1, k + 1, rows, cols);
    int ld = p.b;
    rows = mv;
    // opaque, so that the addresses below are formed here and not kept (spilled)
    // across the columns
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int li = ln & 15, lk = ln >> 4;
    if (k > 0) {
      if (!ready && !flow_wait2(p, hflag(p, k, 0), hflag(p, k, 1), tag, ok_sh) && threadIdx.x == 0) atomicOr(p.err, 2);
      // final values, read by nobody on this XCD before: ordinary loads
      gc = hsub(p, k);
      gd = hdiag(p, k + 1);
      ld = 64;
    }
    // C rows 16w .. 16w+15 as pairs: row 2q + ln / 32, columns 2 (ln % 32), +1
    double c[16];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const unsigned at = min(16 * w + 2 * q + (ln >> 5), rows - 1) * ld + 2 * (ln & 31);
      c[2 * q] = gview(gc)[at];
      c[2 * q + 1] = gview(gc)[at + 1];
    }
    f64x4 d0 = block_load(gd, ld, rows, bi0, bj0, ln);
    f64x4 d1 = block_load(gd, ld, rows, bi1, bj1, ln);
    f64x4 d2 = block_load(gd, ld, rows, bi2, bj2, ln);
    // while those loads are in flight: L_kk out of sA
    chain_store_l(p, k, sA);
    const double lii = sA[ln * BTA_LDS_LD + ln];
    if (threadIdx.x == 0) ok_sh[1] = 0;  // waves whose stores of X have completed
    lds_barrier();
    // the wave's rows of C through its own rows of sA into MFMA operands
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int r = 16 * w + 2 * q + (ln >> 5);
      const bool in = r < rows;
      *(f64x2*)&sA[r * BTA_LDS_LD + 2 * (ln & 31)] = f64x2{in ? c[2 * q] : 0.0, in ? c[2 * q + 1] : 0.0};
    }
    TileAcc x;
    tile_solve(x, sA, sB, w, ln);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int q = 0; q < 4; ++q) sA[(16 * w + 4 * q + lk) * BTA_LDS_LD + 16 * cb + li] = x.c[cb >> 1][cb & 1][q];
    lds_barrier();  // X is complete in sA
    f64x4 e0;
    if (w == 0) {
      f64x4 d0b = f64x4{0.0, 0.0, 0.0, 0.0};  // two chains of dependent MFMAs
#pragma unroll
      for (int t = 0; t < 16; t += 2) {
        const double u = sA[li * BTA_LDS_LD + 4 * t + lk], v = sA[li * BTA_LDS_LD + 4 * t + 4 + lk];
        d0 = mfma_f64_nega(u, u, d0);
        d0b = mfma_f64_nega(v, v, d0b);
      }
      d0 += d0b;
      if (mv == 64) chol16_inv16(d0, e0);
    } else {
      // X to the exchange tile: the wave's rows, and a third of wave 0's
      double* xt = xtile(p, k + 1, k);
      solve_store_x(x, xt, w, ln);
#pragma unroll
      for (int h = 0; h < 6; ++h) {  // 4 x 16 pieces, as above
        const int q = min(w - 1 + 3 * h, 15);
        const int r = 4 * (q & 3) + (ln >> 4), c16 = 16 * (q >> 2) + (ln & 15);
        st_sys(xt + x_index(r, c16), sA[r * BTA_LDS_LD + c16]);
      }
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const double a0 = sA[(16 * bi0 + li) * BTA_LDS_LD + 4 * t + lk];
        const double a2 = sA[(16 * bi2 + li) * BTA_LDS_LD + 4 * t + lk];
        const double b0 = sA[(16 * bj0 + li) * BTA_LDS_LD + 4 * t + lk];
        const double b1 = sA[(16 * bj1 + li) * BTA_LDS_LD + 4 * t + lk];
        const double b2 = sA[(16 * bj2 + li) * BTA_LDS_LD + 4 * t + lk];
        d0 = mfma_f64_nega(a0, b0, d0);
        d1 = mfma_f64_nega(a0, b1, d1);
        d2 = mfma_f64_nega(a2, b2, d2);
        if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
      // the last of the three waves whose stores have completed publishes X
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_s_waitcnt(0);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      if (ln == 0 && atomicAdd(&ok_sh[1], 1) == 2)
        __hip_atomic_store(xflag(p, k + 1, k), tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    solve_store(x, gx, p.b, rows, 64, w, ln);  // ... and to the factor
    lds_barrier();  // X in sA and inv(L_kk) in sB are no longer read
    if (w == 0) {
      if (mv == 64) store_chol16(d0, e0, sA, sB, 0);
      else store16(sA, 0, 0, d0);
    } else {
      store16(sA, 16 * bi0, 16 * bj0, d0);
      store16(sA, 16 * bi1, 16 * bj1, d1);
      store16(sA, 16 * bi2, 16 * bj2, d2);
    }
    lds_barrier();
    if (mv == 64) {
      tile_chol_blocks<true>(sA, sB, 64, [&] { chain_log(p, k, lii); });
    } else {
      tile_chol_inv(sA, sB, mv);
      if (w == 3) chain_log(p, k, lii);
    }
    chain_store_inv(p, k + 1, sB);
    // the hand-off flags of the next column, loaded while the stores drain
    unsigned long long hv = tag;
    if (k + 2 < nT && threadIdx.x < 2) hv = flag_value(hflag(p, k + 1, threadIdx.x), tag);
    if (threadIdx.x < 64) {
      const bool all = __ballot(hv != tag) == 0;
      if (threadIdx.x == 0) ok_sh[2] = all ? 1 : 0;
    }
    flow_publish(wflag(p, k + 1), tag);
    // a word of its own: flow_wait2 writes ok_sh[0] with no barrier after this read
    ready = ok_sh[2] != 0;
  }
  chain_store_l(p, nT - 1, sA);
  if (w == 0) chain_log(p, nT - 1, sA[lane * BTA_LDS_LD + lane]);
}

// One 64-column product of a helper: its operand tiles and the flags they wait
// for (f2: nullptr if one tile is both).
struct HStep {
  const double* a;
  const double* b;
  unsigned long long* f1;
  unsigned long long* f2;
};

__device__ __forceinline__ HStep step_of(const FlowArgs& p, int ra, int rb, int k) {
  return HStep{xtile(p, ra, k), xtile(p, rb, k), xflag(p, ra, k), ra != rb ? xflag(p, rb, k) : nullptr};
}

// A task: op, tile (rho, c), column k.
struct HTask {
  int op, rho, c, k;
};

// The task words are uniform and constant for the launch: scalar loads, so that
// everything decoded stays in scalar registers and reading ahead in the list
// waits for no vector load.
__device__ __forceinline__ HTask task_at(const FlowArgs& p, int t) {
  HTask h;
  flow_decode(((const __attribute__((address_space(4))) uint32_t*)p.tasks)[t], h.op, h.rho, h.c, h.k);
  return h;
}

// Half of a product's operands (K = 32) of one wave, as MFMA operands: its two
// row blocks of either tile, k steps 2u and 2u + 1 of the half in element u.
struct StepHalf {
  f64x2 a[2][4], b[2][4];
  // The exchange tiles are written once per launch (before their flag), so
  // ordinary cached loads after the flag see them; the L2 lines cannot be older
  // than the launch.
  __device__ __forceinline__ void load(const HStep& st, int w, int lane, int half) {
    const gdouble* pa = gview(st.a) + ((w >> 1) * 2048 + half * 512);
    const gdouble* pb = gview(st.b) + ((w & 1) * 2048 + half * 512);
    const unsigned at = x_lane(lane);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        a[x][u] = *(const gf64x2*)(pa + (x * 1024 + u * 128) + at);
        b[x][u] = *(const gf64x2*)(pb + (x * 1024 + u * 128) + at);
      }
  }
  // acc -= A B^T over the half
  __device__ __forceinline__ void mma(TileAcc& t) const {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        t.c[0][0] = mfma_f64_nega(a[0][u][e], b[0][u][e], t.c[0][0]);
        t.c[0][1] = mfma_f64_nega(a[0][u][e], b[1][u][e], t.c[0][1]);
        t.c[1][0] = mfma_f64_nega(a[1][u][e], b[0][u][e], t.c[1][0]);
        t.c[1][1] = mfma_f64_nega(a[1][u][e], b[1][u][e], t.c[1][1]);
      }
  }
};

// The wave waits for the flags of a product (lanes 0 and 1 poll one each).
__device__ __forceinline__ void step_wait(const FlowArgs& p, const HStep& st, int lane, unsigned long long tag) {
  const int ok = lane < 2 ? flow_poll(p, lane == 0 ? st.f1 : st.f2, tag) : 1;
  if (__ballot(ok == 0) != 0 && lane == 0) atomicOr(p.err, 4);
}
// The flags' values now (even lanes f1, odd lanes f2), to be looked at later.
__device__ __forceinline__ unsigned long long step_probe(const HStep& st, int lane) {
  return __hip_atomic_load((lane & 1) && st.f2 ? st.f2 : st.f1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A helper's target tile in memory, accumulator layout.  Full tiles (all but
// the last of a ragged size): loads back to back, not waited for here.
__device__ __forceinline__ void target_load(TileAcc& t, const double* __restrict__ g, int ld, int rows, int cols, int w,
                                            int lane) {
  const int r0 = (w >> 1) * 32 + (lane >> 4), c0 = (w & 1) * 32 + (lane & 15);
  if (rows == 64 && cols == 64) {
    const unsigned at = r0 * ld + c0;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int y = 0; y < 2; ++y) t.c[x][y][r] = (gview(g) + ((16 * x + 4 * r) * ld + 16 * y))[at];
  } else {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          const int i = r0 + 16 * x + 4 * r, j = c0 + 16 * y;
          const double v = gview(g)[(unsigned)(min(i, rows - 1) * ld + min(j, cols - 1))];
          t.c[x][y][r] = i < rows && j < cols ? v : 0.0;
        }
  }
}
__device__ __forceinline__ void target_store(const TileAcc& t, double* __restrict__ g, int ld, int rows, int cols,
                                             int w, int lane) {
  const int r0 = (w >> 1) * 32 + (lane >> 4), c0 = (w & 1) * 32 + (lane & 15);
  const unsigned at = r0 * ld + c0;
  if (rows == 64 && cols == 64) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int y = 0; y < 2; ++y) (gview(g) + ((16 * x + 4 * r) * ld + 16 * y))[at] = t.c[x][y][r];
  } else {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          if (r0 + 16 * x + 4 * r < rows && c0 + 16 * y < cols)
            (gview(g) + ((16 * x + 4 * r) * ld + 16 * y))[at] = t.c[x][y][r];
  }
}

// ... and a hand-off tile in its buffer (64 x 64), past the caches.
__device__ __forceinline__ void hand_load(TileAcc& t, const double* __restrict__ g, int w, int lane) {
  const double* at = g + ((w >> 1) * 32 + (lane >> 4)) * 64 + (w & 1) * 32 + (lane & 15);
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int y = 0; y < 2; ++y) t.c[x][y][r] = ld_sys(at + (16 * x + 4 * r) * 64 + 16 * y);
}
__device__ __forceinline__ void hand_store(const TileAcc& t, double* __restrict__ g, int w, int lane) {
  double* at = g + ((w >> 1) * 32 + (lane >> 4)) * 64 + (w & 1) * 32 + (lane & 15);
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int y = 0; y < 2; ++y) st_sys(at + (16 * x + 4 * r) * 64 + 16 * y, t.c[x][y][r]);
}

// Helper h runs its task list.  The operands of an update come from the exchange
// tiles in MFMA operand order straight into registers: no LDS, and no barrier
// between the four waves, each of which polls, loads and multiplies its 32 x 32
// quadrant on its own.  A run of updates of one tile (the columns of a
// next-block task, or consecutive updates and then the solve of a panel tile)
// keeps the tile in registers.
// Up to b = 1600 nothing waits for it but the chain; beyond, it is bound by the
// waits for tiles of other helpers (the matrix cores are busy 60 % of a launch at
// b = 2000).  Measured on MI355X, against operands staged through LDS with two
// barriers per product: b = 1600 445 -> 379 us per block (the chain's own time),
// b = 2000 770 -> 638, a pair of factorizations at b = 2000 1125 -> 1026; with the
// task costs above and the exchange order of fours 359, 542 and 872.
// Loading the next product's first half during the second, or the next task's
// target during the last product, is slower (655-690): the loads then queue
// ahead of those that a waiting helper needs first.
__device__ __forceinline__ void flow_helper(const FlowArgs& p, int h, unsigned long long tag, double* sA, double* sB) {
  const int nT = p.nT;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const auto* off = (const __attribute__((address_space(4))) int*)p.off;
  const int t1 = off[h + 1];
  int t = off[h];
  while (t < t1) {
    // opaque, so that the addresses below are formed here and not kept (spilled)
    // from run to run
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    HTask cur = task_at(p, t);
    int rows = 0, cols = 0, ld = p.b;
    double* g = nullptr;
    int ra = cur.rho, rb = cur.c;  // operand tile rows of an update
    if (cur.op == FLOW_NEXT) {
      if (cur.rho < nT) {
        g = p.Dn + (int64_t)(64 * cur.rho) * p.b + 64 * cur.c;
        rows = min(64, p.b - 64 * cur.rho);
        cols = min(64, p.b - 64 * cur.c);
        ra = nT + cur.rho;
        rb = nT + cur.c;
      } else if (cur.rho == nT) {
        g = p.Bn + 64 * cur.c;
        rows = p.a;
        cols = min(64, p.b - 64 * cur.c);
        ra = nT + p.nTL;
        rb = nT + cur.c;
      } else {
        g = p.T;
        rows = cols = ld = p.a;
        ra = rb = nT + p.nTL;
      }
    } else {
      g = flow_tile(p, cur.rho, cur.c, rows, cols);
      if (cur.op == FLOW_ZERO) {
        for (int r = w; r < rows; r += 4)
          if (lane < cols) g[(int64_t)r * p.b + lane] = 0.0;
        ++t;
        continue;
      }
    }
    TileAcc acc;
    const bool hand = cur.op == FLOW_UPD && flow_is_handoff(nT, cur.rho, cur.c);
    double* hb = cur.rho == cur.c ? hdiag(p, cur.c) : hsub(p, cur.c);
    if (cur.op == FLOW_TRSM) {
      target_load(acc, g, ld, rows, cols, w, lane);
    } else {
      int k = cur.k;
      const int kend = cur.op == FLOW_NEXT ? flow_next_end(cur.k, nT) : k + 1;
      HStep st = step_of(p, ra, rb, k);
      unsigned long long fv = step_probe(st, lane);
      // (a hand-off tile's buffer holds earlier writes of this workgroup only,
      // which went past the caches)
      if (hand && cur.k > 0) hand_load(acc, hb, w, lane);
      else target_load(acc, g, ld, rows, cols, w, lane);
      StepHalf h0, h1;
      if (__ballot(fv != tag) != 0) step_wait(p, st, lane, tag);
      for (;;) {
        h0.load(st, w, lane, 0);
        h1.load(st, w, lane, 1);
        // the next column of the run (hand-off tiles are never carried: every
        // update goes to the buffer)
        if (cur.op == FLOW_NEXT && k + 1 < kend) {
          ++k;
        } else {
          k = -1;
          ++t;
          if (cur.op == FLOW_UPD && !hand && t < t1) {
            const HTask nx = task_at(p, t);
            if (nx.op == FLOW_UPD && nx.rho == cur.rho && nx.c == cur.c) k = nx.k;
          }
          if (k < 0) break;
        }
        st = step_of(p, ra, rb, k);
        fv = step_probe(st, lane);
        h0.mma(acc);
        h1.mma(acc);
        if (__ballot(fv != tag) != 0) step_wait(p, st, lane, tag);
      }
      h0.mma(acc);
      h1.mma(acc);
      bool solve = false;  // the tile's solve follows
      if (cur.op == FLOW_UPD && !hand && t < t1) {
        const HTask nx = task_at(p, t);
        solve = nx.op == FLOW_TRSM && nx.rho == cur.rho && nx.c == cur.c;
      }
      if (!solve) {
        if (hand) {
          hand_store(acc, hb, w, lane);
          if (cur.rho == cur.c + 1 && cur.k == cur.c - 1) flow_publish(hflag(p, cur.c, 0), tag);
          else if (cur.rho == cur.c && cur.k == cur.c - 2) flow_publish(hflag(p, cur.c - 1, 1), tag);
        } else {
          target_store(acc, g, ld, rows, cols, w, lane);
        }
        continue;
      }
    }
    // the solve of tile (rho, c)
    ++t;
    const double* wi = p.winv + (int64_t)cur.c * 4096;
    step_wait(p, HStep{wi, nullptr, wflag(p, cur.c), nullptr}, lane, tag);
    f64x2 iv[8];  // rows 16w + lane / 32 + 2q, columns 2 (lane % 32), +1
    const unsigned ia = (16 * w + (lane >> 5)) * 64 + 2 * (lane & 31);
#pragma unroll
    for (int q = 0; q < 8; ++q) iv[q] = *(const gf64x2*)(gview(wi) + (128 * q) + ia);
    // (the barrier of the last solve's publication: sA and sB are free)
    double* sc = sA + ((w >> 1) * 32 + (lane >> 4)) * BTA_LDS_LD + (w & 1) * 32 + (lane & 15);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[(16 * x + 4 * r) * BTA_LDS_LD + 16 * y] = acc.c[x][y][r];
    double* si = sB + (16 * w + (lane >> 5)) * BTA_LDS_LD + 2 * (lane & 31);
#pragma unroll
    for (int q = 0; q < 8; ++q) *(f64x2*)(si + 2 * q * BTA_LDS_LD) = iv[q];
    lds_barrier();
    tile_solve(acc, sA, sB, w, lane);
    solve_store(acc, g, p.b, rows, cols, w, lane);
    solve_store_x(acc, xtile(p, cur.rho, cur.c), w, lane);
    flow_publish(xflag(p, cur.rho, cur.c), tag);
  }
}

__global__ void __launch_bounds__(BTA_THREADS, 2) k_panel_flow(FlowArgs p) {
  __shared__ double sA[64 * BTA_LDS_LD];
  __shared__ double sB[64 * BTA_LDS_LD];
  __shared__ int ok_sh[3];
  const unsigned long long tag = (p.epoch[0] << 20) | (unsigned long long)p.blk;
  if (blockIdx.x == 0) flow_chain(p, tag, sA, sB, ok_sh);
  else flow_helper(p, blockIdx.x - 1, tag, sA, sB);
}

// -------------------------------------------------------------------- host

int flow_capacity(int device);

FlowPlan::~FlowPlan() { release(); }

void FlowPlan::release() {
  for (auto& sc : scheds) {
    if (sc.d_tasks) hipFree(sc.d_tasks);
    if (sc.d_off) hipFree(sc.d_off);
  }
  scheds.clear();
  if (xbuf) hipFree(xbuf);
  if (flags) hipFree(flags);
  xbuf = nullptr;
  flags = nullptr;
  hacc = nullptr;
  nT = -1;
}

size_t FlowPlan::bytes_for(int nT, int nTa) {
  const size_t R = 2 * (size_t)nT + nTa;
  return ((R * nT + 2 * (size_t)nT) * 4096) * sizeof(double) + (R * nT + 3 * (size_t)nT) * 8;
}

int FlowPlan::build(int nT_, int nTa_) {
  release();
  nT = nT_;
  nTa = nTa_;
  const int R = 2 * nT + nTa;
  hipError_t e;
  const size_t xd = ((size_t)R * nT + 2 * (size_t)nT) * 4096;
  if ((e = hipMalloc(&xbuf, xd * sizeof(double))) != hipSuccess) return (int)e;
  hacc = xbuf + (size_t)R * nT * 4096;
  const size_t nf = (size_t)R * nT + 3 * (size_t)nT;
  if ((e = hipMalloc(&flags, nf * sizeof(unsigned long long))) != hipSuccess) return (int)e;
  if ((e = hipMemset(flags, 0, nf * sizeof(unsigned long long))) != hipSuccess) return (int)e;
  buf_bytes = bytes_for(nT, nTa);
  return 0;
}

int FlowPlan::sched(int nTa_s, int helpers, int delta, int near_div, int fold, const FlowSched** out) {
  if (nTa_s > nTa) return (int)hipErrorInvalidValue;
  for (const auto& sc : scheds)
    if (sc.helpers == helpers && sc.delta == delta && sc.nTa == nTa_s && sc.near_div == near_div &&
        sc.fold == fold) {
      *out = &sc;
      return 0;
    }
  FlowSched sc;
  sc.helpers = helpers;
  sc.delta = delta;
  sc.nTa = nTa_s;
  sc.near_div = near_div;
  sc.fold = fold;
  std::vector<uint32_t> all;
  std::vector<int> off;
  for (int v = 0; v < 2; ++v) {  // 0: block with L, 1: last block (no L)
    FlowShape s{nT, v == 0 ? nT : 0, nTa_s, near_div, fold};
    FlowSchedule h;
    if (!flow_build_schedule(s, helpers, delta, h)) return -1;
    const int base = (int)all.size();
    sc.off_base[v] = (int)off.size();
    for (int q = 0; q <= helpers; ++q) off.push_back(h.off[q] + base);
    all.insert(all.end(), h.tasks.begin(), h.tasks.end());
  }
  hipError_t e;
  if ((e = hipMalloc(&sc.d_tasks, std::max<size_t>(1, all.size()) * sizeof(uint32_t))) != hipSuccess) return (int)e;
  if ((e = hipMalloc(&sc.d_off, off.size() * sizeof(int))) != hipSuccess) return (int)e;
  if (!all.empty() && (e = hipMemcpy(sc.d_tasks, all.data(), all.size() * 4, hipMemcpyHostToDevice)) != hipSuccess)
    return (int)e;
  if ((e = hipMemcpy(sc.d_off, off.data(), off.size() * sizeof(int), hipMemcpyHostToDevice)) != hipSuccess)
    return (int)e;
  sc.bytes = std::max<size_t>(1, all.size()) * sizeof(uint32_t) + off.size() * sizeof(int);
  scheds.push_back(sc);
  *out = &scheds.back();
  return 0;
}

int flow_helpers_default(int device) {
  // room for two factorizations in flight (prior and conditional chains)
  const int cap = flow_capacity(device);
  return cap > 0 ? std::max(1, cap / 2 - 1) : 0;
}

unsigned long long flow_spin_ticks(int device, double seconds) {
  int khz = 0;
  if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) != hipSuccess || khz <= 0) khz = 100000;
  return (unsigned long long)(seconds * 1e3 * khz);
}

FlowArgs flow_args(const FlowPlan& fp, const FlowSched& sc, double* D, double* L, double* B, double* T, double* winv,
                   double* logpart, const unsigned long long* epoch, unsigned long long* info, int* err, int i,
                   int n, int b, int a) {
  FlowArgs p;
  const int nT = fp.nT;
  p.D = D + (int64_t)i * b * b;
  p.L = (i < n - 1) ? L + (int64_t)i * b * b : nullptr;
  p.B = (a > 0) ? B + (int64_t)i * a * b : nullptr;
  p.Dn = (i < n - 1) ? D + (int64_t)(i + 1) * b * b : nullptr;
  p.Bn = (a > 0 && i < n - 1) ? B + (int64_t)(i + 1) * a * b : nullptr;
  p.T = (a > 0) ? T : nullptr;
  p.winv = winv + (int64_t)i * nT * 4096;
  p.xbuf = fp.xbuf;
  p.hacc = fp.hacc;
  p.logpart = logpart + (int64_t)i * nT;
  p.flags = fp.flags;
  const int v = (i < n - 1) ? 0 : 1;
  p.tasks = sc.d_tasks;
  p.off = sc.d_off + sc.off_base[v];
  p.epoch = epoch;
  p.info = info;
  p.err = err;
  p.row0 = (long long)i * b;
  p.spin_ticks = fp.spin_ticks;
  p.b = b;
  p.a = a;
  p.nT = nT;
  p.nTL = (i < n - 1) ? nT : 0;
  p.nTa = sc.nTa;
  p.blk = i + 1;
  p.helpers = sc.helpers;
  return p;
}

void flow_launch_block(const Workspace& ws, const FlowPlan& fp, const FlowSched& sc, double* D, double* L,
                       double* B, double* T, int i, int n, int b, int a, hipStream_t st) {
  const FlowArgs p = flow_args(fp, sc, D, L, B, T, ws.winv, ws.logpart, ws.epoch, ws.info, ws.err, i, n, b, a);
  hipLaunchKernelGGL(k_panel_flow, dim3(1 + sc.helpers), dim3(BTA_THREADS), 0, st, p);
}

// Batched form: every entry's chain and helpers in one launch (layout in
// FlowBatch).  All entries' workgroups are resident together (their sum is
// within the device's capacity).
__global__ void __launch_bounds__(BTA_THREADS, 2) k_panel_flow_batched(FlowBatch fb) {
  __shared__ double sA[64 * BTA_LDS_LD];
  __shared__ double sB[64 * BTA_LDS_LD];
  __shared__ int ok_sh[3];
  const int wg = (int)blockIdx.x;
  int pos = wg;  // position in the entries' ranges of `begin`
  if (fb.iso) {
    if (wg >= fb.cus && wg < fb.cus + fb.nent) return;  // the CU partner of a chain
    if (wg < fb.nent) pos = -1;                         // chain of entry wg
    else pos = wg < fb.cus ? wg - fb.nent : wg - 2 * fb.nent;
  }
  if (pos >= fb.begin[fb.nent]) return;
  int lo = 0, local = 0;
  if (pos < 0) {
    lo = wg;
  } else {
    int hi = fb.nent - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (fb.begin[mid] <= pos) lo = mid;
      else hi = mid - 1;
    }
    local = pos - fb.begin[lo] + (fb.iso ? 1 : 0);
  }
  const FlowArgs p = fb.e[lo];
  const unsigned long long tag = (p.epoch[0] << 20) | (unsigned long long)p.blk;
  if (local == 0) flow_chain(p, tag, sA, sB, ok_sh);
  else flow_helper(p, local - 1, tag, sA, sB);
}

void flow_launch_batched(const FlowBatch& fb, int total, hipStream_t st) {
  hipLaunchKernelGGL(k_panel_flow_batched, dim3(total), dim3(BTA_THREADS), 0, st, fb);
}

int flow_capacity(int device) {
  int cus = 0, per = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0)
    return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_panel_flow, BTA_THREADS, 0) != hipSuccess || per <= 0)
    return 0;
  int per_b = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_b, k_panel_flow_batched, BTA_THREADS, 0) == hipSuccess &&
      per_b > 0)
    per = std::min(per, per_b);
  return cus * per;
}

}  // namespace bta
