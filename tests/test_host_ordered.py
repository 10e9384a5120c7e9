"""The phases of k_learned_fallback (bl_ordered.h), compiled for the host: as
many groups as shares, of which only a few run at once and the rest start when
one of those has ended, as workgroups on a device that other launches fill.
Every phase is whole before the next begins, and every group ends.  With a
barrier over all groups in its place (waiting for a bounded time here)
no phase after the first is reached unless all groups run at once."""
import os
import subprocess

import pytest

from tests.conftest import ROOT

SOURCE = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#include "bl_ordered.h"

struct Counter {
  std::atomic<int>* p;
  int add(int n) const { return p->fetch_add(n); }
  int value() const { return p->load(); }
  void pause() const { std::this_thread::yield(); }
};
struct Group {
  bl::ShareCounters<Counter> counters;
  std::vector<int> held;
  int take() { return counters.taken.add(1); }
  int another(int shares) { return counters.another(shares); }
  void wait(int n, int all) { counters.wait(n, all); }
  void keep(int i, int v) { held.resize(i + 1); held[i] = v; }
  int kept(int i) { return held[i]; }
};

int main(int argc, char** argv) {
  const int shares = std::atoi(argv[1]), running = std::atoi(argv[2]), phases = std::atoi(argv[3]);
  const bool barrier = std::atoi(argv[4]);
  std::atomic<int> taken{0}, finished{0}, group{0}, ends{0}, early{0}, arrived{0}, stuck{0};
  std::vector<std::atomic<int>> count(phases * shares);
  for (auto& c : count) c = 0;
  auto work = [&](int phase, int share) {
    for (int k = 0; k < phase * shares; ++k) early += count[k] != 1;
    count[phase * shares + share]++;
  };
  const std::chrono::milliseconds limit(running < shares ? 200 : 20000);
  auto body = [&](int g) {
    if (barrier) {
      for (int phase = 0; phase < phases; ++phase) {
        work(phase, g);
        arrived++;
        const auto t0 = std::chrono::steady_clock::now();
        for (; arrived < (phase + 1) * shares; std::this_thread::yield())
          if (stuck || std::chrono::steady_clock::now() - t0 > limit) { stuck = 1; return; }
      }
    } else {
      Group group{{{&taken}, {&finished}, 3}, {}};
      bl::ordered_phases(group, shares, [&](int share) { work(0, share); },
                         [&] { return phases - 1; }, work);
    }
    ends++;
  };
  std::vector<std::thread> slots;
  for (int s = 0; s < running; ++s)
    slots.emplace_back([&] { for (int g; (g = group++) < shares;) body(g); });
  for (auto& t : slots) t.join();
  int once = 0;
  for (auto& c : count) once += c == 1;
  std::printf("%d %d %d %d\n", ends.load(), early.load(), once, stuck.load());
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("ordered")
    (d / "ordered.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I",
                    os.path.join(ROOT, "bookleaf_f90_amd", "csrc"), str(d / "ordered.cpp"),
                    "-o", str(d / "ordered")], check=True)

    def run(*args):
        r = subprocess.run([str(d / "ordered")] + [str(int(a)) for a in args],
                           capture_output=True, text=True, timeout=10, check=True)
        return tuple(int(v) for v in r.stdout.split())
    return run


@pytest.mark.parametrize("shares,running", [(1, 1), (2, 1), (7, 3), (16, 1), (16, 5), (16, 16),
                                            (3, 8)])
@pytest.mark.parametrize("phases", [1, 2, 9])
def test_every_phase_ends_whole(shares, running, phases, program):
    assert program(shares, running, phases, False) == (shares, 0, shares * phases, 0)


def test_a_barrier_needs_every_group(program):
    assert program(4, 4, 3, True)[2:] == (12, 0)
    ends, _, once, stuck = program(4, 3, 3, True)
    assert ends == 0 and once < 12 and stuck == 1
