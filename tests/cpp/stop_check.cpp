// CPU model of the launches of a Krylov solve and of the words through which
// they learn of the stop (xyst_amd/csrc/xg_stop.hpp): stop_check SEED.
// Per iteration a launch that tests and one that updates; the waves of all
// workgroups ask and the first workgroup writes in any order.  The waves of a
// workgroup must agree, every workgroup must work up to the iteration of the
// stop and none after it.  Prints "ok" or what differs.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../xyst_amd/csrc/xg_stop.hpp"

int main(int argc, char** argv) {
  if (argc != 2) return 2;
  std::mt19937 g(atoi(argv[1]));
  const int groups = 5, waves = 4, iters = 6;
  for (int stop = 1; stop < iters; ++stop) {
    xg::CgState s{};
    xg::stop_clear(s);
    for (int j = 1; j <= iters; ++j)
      for (int launch = 0; launch < 2; ++launch) {
        const bool test = launch == 0;
        // what the first workgroup finds is known to it after its own waves
        // have asked; the others' waves may ask before or after its write
        std::vector<int> order(groups * waves);
        for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
        std::shuffle(order.begin(), order.end(), g);
        int seen[groups] = {}, asked0 = 0;
        for (int i : order) {
          const bool leaves = test ? xg::stop_past(s) : xg::stop_found(s);
          seen[i / waves] += leaves;
          if (i / waves == 0 && ++asked0 == waves) {
            if (seen[0] % waves) return printf("group 0 split in %d\n", j), 1;
            if (test && !seen[0] && j == stop) xg::stop_record(s, j - 1, 0.5, 1);
            if (!test && seen[0]) xg::stop_pass(s);
          }
        }
        for (int b = 0; b < groups; ++b) {
          if (seen[b] % waves) return printf("group %d split in %d\n", b, j), 1;
          const bool leaves = seen[b] != 0;
          if (leaves != (test ? j > stop : j >= stop))
            return printf("group %d, iteration %d of %d\n", b, j, stop), 1;
        }
      }
    if (s.it != stop - 1 || s.rr != 0.5 || s.converged != 1) return printf("state\n"), 1;
    xg::stop_clear(s);
    if (xg::stop_past(s) || xg::stop_found(s)) return printf("clear\n"), 1;
  }
  printf("ok\n");
  return 0;
}
