// solve_guard.hpp -- control flow of the pressure solves (poisson.hip) whose
// failures cannot be had on demand: the residual watch of the iterations, and
// what follows the solid flags.  Plain C++ without HIP so that the host tests
// tests/native/solve_guard_check.cpp and flags_check.cpp compile it with g++.
//
// Every relative residual a solve reads goes through ResidWatch::step:
//  - NaN or Inf stops the solve with an error (a NaN residual would pass
//    `rel > tol` as converged and never satisfy `rel <= tol`);
//  - a residual above kDivergeFactor times the best one so far stops it as
//    diverged (the reference V-cycle grows without bound on some hierarchies);
//  - from the last two residuals it says whether the one under way is expected
//    above the tolerance.
#ifndef PYRO_SOLVE_GUARD_HPP
#define PYRO_SOLVE_GUARD_HPP
#include <cmath>

namespace pyro {

constexpr double kDivergeFactor = 1e3;
constexpr double kFirstRate = 0.1;  // contraction of the first iteration, 0.01 to 0.5 on the solves in use

enum class Watch { Go = 0, NonFinite = 1, Diverged = 2 };

struct ResidWatch {
  double best = 0.0;
  double last = 0.0, rate = 0.0;  // the last residual, its contraction
  // k = number of iterations done (0 for the initial residual)
  Watch step(double rel, int k) {
    if (!std::isfinite(rel)) return Watch::NonFinite;
    if (k == 0 || rel < best) best = rel;
    rate = k > 0 && last > 0.0 ? rel / last : kFirstRate;
    last = rel;
    if (rel > kDivergeFactor * best) return Watch::Diverged;
    return Watch::Go;
  }
  // Is the residual of the iteration under way expected above tol?  The last
  // contraction is taken to hold; in 321 solves of fires and Gaussian sources
  // to 1e-2 .. 1e-7 (2333 iterations) that was wrong for 30 last iterations
  // and 59 others.
  bool expects_more(double tol) const { return last * rate > tol; }
};

// What a handle has formed from its solid flags (neighbour codes, fluid count,
// labels) follows new flags.  compare(changed) stores them and reports whether
// they differ, form() forms everything anew; both return 0 or an error.  The
// new flags are stored before the outcome is known, so nothing counts as formed
// until it is: after an error (or a throw) the next call forms everything.
template <class Compare, class Form>
int follow_flags(bool &formed, Compare compare, Form form) {
  const bool was = formed;
  formed = false;
  bool changed = true;
  int rc = compare(changed);
  if (!rc && (changed || !was)) rc = form();
  formed = rc == 0;
  return rc;
}

}  // namespace pyro
#endif
