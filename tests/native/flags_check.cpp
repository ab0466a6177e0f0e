// Host check of follow_flags (pyro_amd/csrc/solve_guard.hpp): a model handle
// whose compare stores the flags before it reports, as the device does, with an
// error at any step of any call.  After every call that returns 0 the formed
// data must be those of the flags given.
#include <cstdio>

#include "solve_guard.hpp"

struct Handle {
  int flags = 0, data = 0;  // data: the flags it was formed from
  bool formed = true;
  int forms = 0;
};

// fail: 0 nothing, 1 compare after it stored, 2 compare before, 3 form before, 4 form half way
static int set(Handle &h, int flags, int fail) {
  return pyro::follow_flags(
      h.formed,
      [&](bool &changed) {
        if (fail == 2) return 1;
        const bool differ = h.flags != flags;
        h.flags = flags;
        if (fail == 1) return 1;
        changed = differ;
        return 0;
      },
      [&] {
        if (fail == 3) return 1;
        h.data = fail == 4 ? -1 : flags;
        h.forms++;
        return fail == 4 ? 1 : 0;
      });
}

int main() {
  int bad = 0, calls = 0;
  // every sequence of four calls: flags 0..1, fail 0..4 each
  for (int seq = 0; seq < 10 * 10 * 10 * 10; seq++) {
    Handle h;
    for (int k = 0, s = seq; k < 4; k++, s /= 10) {
      const int flags = s % 2, fail = s / 2 % 5;
      calls++;
      if (set(h, flags, fail) == 0 && (h.data != flags || h.flags != flags)) bad++;
    }
  }
  // unchanged flags form nothing
  Handle h;
  for (int k = 0; k < 3; k++) bad += set(h, 0, 0) != 0;
  bad += h.forms != 0;
  bad += set(h, 1, 0) != 0 || h.forms != 1;
  bad += set(h, 1, 0) != 0 || h.forms != 1;
  std::printf("%d calls, %d wrong\n", calls, bad);
  return bad != 0;
}
