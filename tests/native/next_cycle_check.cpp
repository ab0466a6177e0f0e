// Host check of ResidWatch::expects_more (pyro_amd/csrc/solve_guard.hpp): may
// the next V-cycle be started before the residual of the iteration under way is
// known?  Residuals of solves (fires at 2, 4, 7 and 10 cm, a ragged grid) to
// every tolerance between 1e-2 and 1e-7, driven through the loops' control
// flow: a start that is not used (after the last iteration) in at most one
// solve of four, a start left out in at most one iteration of twelve.
#include <cmath>
#include <cstdio>
#include <vector>

#include "solve_guard.hpp"

static const std::vector<std::vector<double>> kSolves = {
    {5.3e-01, 3.2e-02, 6.3e-03, 3.8e-04, 3.1e-05, 4.5e-06, 3.4e-07, 4.3e-08, 5.9e-09},
    {2.7e-01, 8.3e-03, 1.8e-03, 8.9e-04, 3.5e-04, 2.3e-04, 7.1e-05, 2.9e-05, 1.3e-05, 3.1e-06, 1.9e-06, 1.2e-06, 3.6e-07, 2.1e-07, 6.3e-08, 1.9e-08, 1.0e-08, 3.8e-09},
    {9.5e-01, 2.4e-01, 7.7e-02, 3.9e-02, 2.5e-02, 1.8e-02, 1.3e-02, 9.2e-03, 6.8e-03, 5.0e-03, 3.7e-03, 2.8e-03, 2.1e-03, 1.6e-03, 1.2e-03, 8.9e-04, 6.7e-04, 5.1e-04, 3.9e-04, 2.9e-04},
    {1.0e+00, 6.8e-01, 2.9e-01, 1.1e-01, 4.1e-02, 1.6e-02, 6.1e-03, 2.3e-03, 1.2e-03, 4.9e-04, 2.0e-04, 7.9e-05, 3.2e-05, 1.3e-05, 6.6e-06, 2.3e-06, 8.4e-07, 3.8e-07, 1.8e-07, 8.0e-08},
    {5.7e-01, 1.9e-02, 1.9e-03, 2.5e-04, 5.3e-05, 1.1e-05, 2.3e-06, 4.9e-07, 1.1e-07, 2.4e-08, 5.2e-09},
};

int main() {
  int solves = 0, iterations = 0, unused = 0, left_out = 0, bad = 0;
  for (const auto &h : kSolves)
    for (double e = 2.0; e <= 7.0; e += 0.25) {
      const double tol = std::pow(10.0, -e);
      if (h.front() <= tol || h.back() > tol) continue;
      solves++;
      pyro::ResidWatch rw;
      rw.step(h[0], 0);
      for (size_t k = 1; k < h.size(); k++) {
        const bool head = rw.expects_more(tol), last = h[k] <= tol;
        iterations++;
        unused += head && last;
        left_out += !head && !last;
        if (last) break;
        rw.step(h[k], (int)k);
      }
    }
  std::printf("%d solves, %d iterations: %d starts unused, %d left out\n", solves, iterations, unused, left_out);
  if (solves < 50 || 4 * unused > solves || 12 * left_out > iterations) bad++;
  // a steady contraction is foreseen exactly; no tolerance is never reached
  pyro::ResidWatch rw;
  double rel = 1.0;
  rw.step(rel, 0);
  for (int k = 1; k < 12; k++) {
    rel *= 0.25;
    if (k > 1 && rw.expects_more(0.9 * rel) != true) bad++;
    if (k > 1 && rw.expects_more(1.1 * rel) != false) bad++;
    if (!rw.expects_more(0.0)) bad++;
    rw.step(rel, k);
  }
  std::printf("%d wrong\n", bad);
  return bad != 0;
}
