// Host model of a sweep's workgroups (bta_sweep_walk.h) with some of them taken
// away.  Lines on stdin:  trans n b a cap watch late
//   cap    workgroups the sweep may have, watch 1: look at the claims (the gate),
//   0: look for the seats whose stage-0 outputs the own stage-1 item waits for;
//   late   the seats whose workgroups start only when the others have ended, comma-separated ("-": none)
// and for each "1 0" if every element of every stage was produced, else "0 <number
// of stages that are whole>".
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <iostream>
#include <set>
#include <sstream>
#include <string>
#include <vector>

#define __host__
#define __device__
#define __forceinline__ inline
static int first_lane(int x) { return x; }
#define __builtin_amdgcn_readfirstlane first_lane
#include "bta_sweep_walk.h"

using namespace bta;

struct Group {
  SweepWalk walk;
  std::vector<int> seat;
  bool done;
};

template <bool T>
static void simulate(int n, int b, int a, int cap, bool watch, const std::set<int>& late) {
  const int parts = sweep_parts(b, T), stages = sweep_stages(n, a, T), halves = T ? 2 : 1, no = T ? 16 : 8;
  const int seats = std::min(std::min(parts, cap), kSeats);
  // produced[stage][half][row]; the vector before stage 0 is there from the start
  std::vector<std::vector<std::vector<char>>> produced(stages, std::vector<std::vector<char>>(halves, std::vector<char>(b, 0)));
  std::vector<char> claimed(seats, 0);
  std::vector<Group> groups;
  for (int s = 0; s < seats; ++s)
    if (!late.count(s)) {
      claimed[s] = 1;
      groups.push_back(Group{SweepWalk(stages, parts, seats, s), {s}, false});
    }
  bool moved = true;
  while (moved) {
    moved = false;
    for (Group& g : groups) {  // a step each: an item, a seat taken over or the gate passed
      if (g.done) continue;
      const SweepItem<T> it(n, b, a, g.walk.stage, g.walk.part);
      std::set<int> missing;  // seats that the item waits for
      if (it.stage > 0)
        for (int e = it.kbeg; e < it.kend; ++e)
          for (int h = 0; h < halves; ++h)
            if (!produced[it.stage - 1][h][e]) missing.insert((T ? 2 * (e / no) + h : e / no) % seats);
      if (watch ? g.walk.at_gate() : it.stage == 1) {
        int victim = -1;
        for (int d = 0; d < seats && victim < 0; ++d) {
          const int s = watch ? (g.seat[0] + d) % seats : d;
          if (!claimed[s] && (watch || missing.count(s))) victim = s;
        }
        if (victim >= 0) {
          claimed[victim] = 1;
          g.seat.push_back(victim);
          g.walk.take_over(victim);
          moved = true;
          continue;
        }
        if (watch) {
          g.walk.open = true;
          moved = true;
          continue;
        }
      }
      if (!missing.empty()) continue;
      for (int e = it.out0; e < std::min(it.out0 + no, b); ++e) produced[it.stage][it.hf][e] = 1;
      moved = true;
      g.done = !g.walk.more(g.seat.data());
    }
    // with everyone gone there is room for the late workgroups
    if (!moved && std::all_of(groups.begin(), groups.end(), [](const Group& g) { return g.done; }))
      for (int s = 0; s < seats; ++s)
        if (!claimed[s]) {
          claimed[s] = 1;
          groups.push_back(Group{SweepWalk(stages, parts, seats, s), {s}, false});
          moved = true;
        }
  }
  int whole = 0;
  for (; whole < stages; ++whole)
    for (const auto& half : produced[whole])
      for (const char x : half)
        if (!x) {
          std::printf("0 %d\n", whole);
          return;
        }
  for (const Group& g : groups)
    if (!g.done) {
      std::printf("0 %d\n", stages);
      return;
    }
  std::printf("1 0\n");
}

int main() {
  int trans, n, b, a, cap, watch;
  std::string list;
  while (std::cin >> trans >> n >> b >> a >> cap >> watch >> list) {
    std::set<int> late;
    std::stringstream ss(list == "-" ? "" : list);
    for (std::string x; std::getline(ss, x, ',');) late.insert(std::atoi(x.c_str()));
    if (trans) simulate<true>(n, b, a, cap, watch != 0, late);
    else simulate<false>(n, b, a, cap, watch != 0, late);
  }
  return 0;
}
