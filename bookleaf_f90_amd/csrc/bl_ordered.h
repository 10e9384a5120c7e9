// Phases of work in one launch, each after the one before, without a
// workgroup ever waiting for one that may not have started.
#pragma once

#if defined(__HIPCC__)
#define BL_EITHER __host__ __device__ __forceinline__
#else
#define BL_EITHER inline
#endif

namespace bl {

// Every phase is the same number of shares.  A group (workgroup) takes a share
// when it starts and does it in every phase; at the end of a phase it waits
// until all shares are done.  A barrier over all groups would end only if all
// of them run at once, which no launch beside others (further handles, other
// processes) can count on.  Here a group at the end of the first phase that
// has waited a while and sees shares nobody took takes one of those too, for
// this and every later phase; a group that starts when none is left leaves at
// once.  So the first phase ends whatever number of groups runs (one alone
// takes every share in turn), all shares then being with groups that run, and
// a group's waits in later phases are for those only: every wait ends.
//
// The common counters (both start the launch at 0), used by one thread of
// each group.
template <typename Counter>
struct ShareCounters {
  Counter taken, finished;
  int patience;  // looks at the counter before a share that nobody took is taken
  // the share taken last is done in the first phase: another one, or -1 when
  // the phase has ended
  BL_EITHER int another(int shares) {
    finished.add(1);
    for (int k = 0; finished.value() < shares; ++k) {
      if (k >= patience && taken.value() < shares) {
        const int v = taken.add(1);
        if (v < shares) return v;
      }
      finished.pause();
    }
    return -1;
  }
  // n shares are done in a later phase; returns when `all` are, from the
  // launch's start on
  BL_EITHER void wait(int n, int all) {
    finished.add(n);
    while (finished.value() < all) finished.pause();
  }
};

// group.take(), group.another(shares), group.wait(n, all): the above, for
// every thread of the group and with what the group stored visible to the
// others; group.keep(i, v), group.kept(i): the shares it holds.  first(share):
// the first phase; phases(): how many follow it, asked when it has ended;
// later(phase, share): those, from 1 on.
template <typename Group, typename First, typename Phases, typename Later>
BL_EITHER void ordered_phases(Group& group, int shares, First first, Phases phases,
                              Later later) {
  int n = 0;
  for (int v = group.take(); v >= 0 && v < shares; v = group.another(shares)) {
    group.keep(n++, v);
    first(v);
  }
  if (n == 0) return;
  const int last = phases();
  for (int p = 1; p <= last; ++p) {
    for (int i = 0; i < n; ++i) later(p, group.kept(i));
    if (p < last) group.wait(n, (p + 1) * shares);
  }
}

}  // namespace bl
