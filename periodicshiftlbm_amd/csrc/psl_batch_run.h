// The groups of grids of a batch, the order of a call's launches and what it
// leaves in the host shifters (plain C++, no HIP types).
#pragma once

#include <cstddef>
#include <vector>

namespace psl {

// Groups of consecutive grids that are stepped together, as the positions past
// each: grids of `bytes` in turn, as many as fit `limit` together, the groups
// of a run of them about equal in size.  A grid above `limit` is a group of its
// own and ends the run, so that its size does not count in the shares of the
// others; neighbours above `lone` (at least `limit`) are one group.
inline std::vector<size_t> group_ends(const std::vector<size_t>& bytes, size_t limit, size_t lone) {
  std::vector<size_t> ends;
  for (size_t at = 0; at < bytes.size();) {
    if (bytes[at] > limit) {
      const bool together = bytes[at] > lone;
      do ++at;
      while (together && at < bytes.size() && bytes[at] > lone);
      ends.push_back(at);
      continue;
    }
    size_t end = at, total = 0;
    for (; end < bytes.size() && bytes[end] <= limit; ++end) total += bytes[end];
    const size_t want = total > limit ? (total + limit - 1) / limit : 1;
    const size_t share = (total + want - 1) / want;
    size_t in_group = 0, before = 0, groups = 1;
    for (; at < end; ++at) {
      if (in_group && (in_group + bytes[at] > limit || before + bytes[at] / 2 > share * groups)) {
        ends.push_back(at);
        in_group = 0;
        ++groups;
      }
      in_group += bytes[at];
      before += bytes[at];
    }
    ends.push_back(end);
  }
  return ends;
}

// `steps` steps of each of `groups` groups of grids, one group after the
// other.  enqueue(g, s) launches step s of group g and returns 0 or an error
// code; advance(g, n) moves the host shifters of group g's grids by n steps.
// At an error the call ends there, and every grid's shifter stands at the
// steps that were launched for it, as its populations do.
template <class Enqueue, class Advance>
int run_groups(size_t groups, int steps, Enqueue&& enqueue, Advance&& advance) {
  for (size_t g = 0; g < groups; ++g) {
    int done = 0, rc = 0;
    while (done < steps && (rc = enqueue(g, done)) == 0) ++done;
    advance(g, done);
    if (rc) return rc;
  }
  return 0;
}

// `steps` steps in launches of `many` consecutive steps (many > 1) while as
// many are left and of one step after them: launch(n) puts n steps on the
// stream, advance(n) moves the shifters by n.
template <class Launch, class Advance>
int run_graphs(int steps, int many, Launch&& launch, Advance&& advance) {
  int done = 0, rc = 0;
  while (done < steps && rc == 0) {
    const int n = many > 1 && steps - done >= many ? many : 1;
    rc = launch(n);
    if (rc == 0) done += n;
  }
  advance(done);
  return rc;
}

}  // namespace psl
