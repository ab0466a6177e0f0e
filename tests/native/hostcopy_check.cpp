// Host check of the pinned-slot copies (pyro_amd/csrc/hostcopy.hip, compiled
// here over fake_hip): every byte at sizes around the slots, streams of a
// device that is not current, an error in the middle, and nothing left when the
// last holder is gone.
#include <cstdio>
#include <vector>

#include "hostcopy.hip"

static int bad = 0;
static void expect(bool ok, const char *what) {
  std::printf("%-44s %s\n", what, ok ? "ok" : "WRONG");
  bad += !ok;
}

static std::vector<char> bytes(size_t n, unsigned seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; i++) v[i] = (char)((seed = seed * 1664525u + 1013904223u) >> 24);
  return v;
}

static bool round_trip(size_t n, hipStream_t s) {
  const std::vector<char> a = bytes(n, (unsigned)n);
  std::vector<char> dev(n), b(n);
  return pyro::copy_in(dev.data(), a.data(), n, s) == hipSuccess && dev == a &&
         pyro::copy_out(b.data(), dev.data(), n, s) == hipSuccess && b == a;
}

int main() {
  constexpr size_t MB = 1u << 20;
  FakeStream s0{0}, s1{1};
  {
    pyro::HostCopyUse use;
    bool ok = true;
    for (size_t n : {1 * MB, 8 * MB - 1, 8 * MB, 16 * MB + 1, 32 * MB, 33 * MB + 7, 72 * MB})
      ok = ok && round_trip(n, &s0) && round_trip(n, &s0);
    expect(ok, "every byte");
    expect(fake::live == 9, "one pool: the slots and eight events");
    fake::current = 0;
    ok = round_trip(33 * MB, &s1) && fake::current == 0;
    fake::current = 1;
    ok = ok && round_trip(33 * MB, &s1) && round_trip(33 * MB, &s0) && fake::current == 1;
    fake::current = 0;
    expect(ok, "a stream of another device than the current");
    const std::vector<char> a = bytes(40 * MB, 3);
    std::vector<char> b(a.size());
    fake::fail_at = fake::copies + 5;
    expect(pyro::copy_in(b.data(), a.data(), a.size(), &s0) == hipErrorInvalidValue, "a failed chunk is reported");
    fake::fail_at = fake::copies + 5;
    expect(pyro::copy_out(b.data(), a.data(), a.size(), &s0) == hipErrorInvalidValue, "the same on the way back");
    fake::fail_at = -1;
    expect(round_trip(33 * MB, &s0), "and the next copy is whole");
    pyro::HostCopyUse second;
    expect(round_trip(9 * MB, &s0), "a second holder");
  }
  expect(fake::live == 0, "all given back with the last holder");
  {
    pyro::HostCopyUse again;
    expect(round_trip(9 * MB, &s0) && fake::live > 0, "and made again");
  }
  expect(fake::live == 0, "and given back");
  std::printf("%d wrong\n", bad);
  return bad != 0;
}
