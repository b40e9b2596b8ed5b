// What the planner of staged launches makes of one fill or chunk, for tests whose
// cases are to reach a given form:
//   share_cases fill BLOCKS:FRAGMENT:SEGMENTS:ELIGIBLE ...
//     -> "share BYTES staged UNITS launches N cut WHERE", WHERE being "none", "units"
//        (between two), or "unit K segment S" (inside)
//   share_cases pages COUNT PAGE_BYTES -> "pages N"
#include <cinttypes>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../pegaflow_amd/csrc/pf_runs.hpp"
#include "../../pegaflow_amd/csrc/pf_share.hpp"

int main(int argc, char** argv) {
  if (argc == 4 && std::strcmp(argv[1], "pages") == 0) {
    printf("pages %" PRIu64 "\n", pf::link_share_pages(strtoull(argv[2], nullptr, 10), strtoull(argv[3], nullptr, 10)));
    return 0;
  }
  if (argc < 3 || std::strcmp(argv[1], "fill") != 0) return 2;
  std::vector<pf::ShareUnit> units;
  uint64_t total = 0;
  for (int i = 2; i < argc; ++i) {
    pf::ShareUnit u = {};
    int eligible = 0;
    if (sscanf(argv[i], "%" SCNu64 ":%" SCNu64 ":%u:%d", &u.n_blocks, &u.frag_bytes, &u.n_seg, &eligible) != 4) return 2;
    u.eligible = eligible != 0;
    total += u.n_blocks * u.n_seg * u.frag_bytes;
    units.push_back(u);
  }
  const pf::ShareCut cut =
      pf::plan_link_share(units.size(), pf::link_share_bytes(total), [&](size_t k) { return units[k]; });
  const size_t staged = cut.bytes != 0 && cut.staged_frags != 0 ? cut.unit + 1 : cut.unit;
  const auto runs = pf::plan_launch_runs(staged, [&](size_t k) {
    return pf::LaunchUnit{units[k].n_blocks, units[k].n_seg, units[k].frag_bytes};
  });
  printf("share %" PRIu64 " staged %zu launches %zu cut ", cut.bytes, staged, runs.empty() ? 1 : runs.size());
  if (cut.bytes == 0) {
    printf("none\n");
  } else if (cut.staged_frags == 0) {
    printf("units\n");
  } else {
    printf("unit %zu segment %d\n", cut.unit, cut.staged_frags < units[cut.unit].n_blocks ? 0 : 1);
  }
  return 0;
}
