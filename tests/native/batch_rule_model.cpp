// bta_batch_rule.h on the command line's terms: "t cus cap nT..." prints a step's
// estimate in us, "l most cus cap n:nT..." the problems per wave.
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>

#include "bta_batch_rule.h"

int main() {
  for (std::string line; std::getline(std::cin, line);) {
    std::stringstream ss(line);
    std::string what;
    int most = 0, cus, cap;
    ss >> what;
    if (what == "l") ss >> most;
    ss >> cus >> cap;
    if (what == "t") {
      std::vector<int> nT;
      for (int t; ss >> t;) nT.push_back(t);
      std::printf("%.6f\n", bta::step_time(nT, cus, cap));
    } else {
      std::vector<bta::BatchShape> ps;
      bta::BatchShape s;
      char colon;
      while (ss >> s.n >> colon >> s.nT) ps.push_back(s);
      std::printf("%d\n", bta::pick_lanes(ps, most, cus, cap));
    }
  }
  return 0;
}
