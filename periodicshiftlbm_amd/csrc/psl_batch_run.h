// Order of the launches of a batch call and what it leaves in the host
// shifters (plain C++, no HIP types).
#pragma once

#include <cstddef>

namespace psl {

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
