// Host build of the batch's groups and launch order (psl_batch_run.h), with a
// launch that fails where it is told to.  Test infrastructure only.
#include "../../periodicshiftlbm_amd/csrc/psl_batch_run.h"

extern "C" {
int br_ends(int n, const long long* bytes, long long limit, long long lone, int* ends) {
  const std::vector<size_t> e = psl::group_ends(std::vector<size_t>(bytes, bytes + n), (size_t)limit,
                                                    (size_t)lone);
  for (size_t i = 0; i < e.size(); ++i) ends[i] = (int)e[i];
  return (int)e.size();
}
// moved[g]: steps that group g's shifters moved; launched[g]: steps launched.
int br_groups(int groups, int steps, int fail_group, int fail_step, int* launched, int* moved) {
  return psl::run_groups(
      (size_t)groups, steps,
      [&](size_t g, int s) {
        if ((int)g == fail_group && s == fail_step) return 7;
        ++launched[g];
        return 0;
      },
      [&](size_t g, int n) { moved[g] += n; });
}
int br_graphs(int steps, int many, int fail_launch, int* launched, int* moved) {
  int at = 0;
  return psl::run_graphs(
      steps, many,
      [&](int n) {
        if (at++ == fail_launch) return 7;
        *launched += n;
        return 0;
      },
      [&](int n) { *moved += n; });
}
}
