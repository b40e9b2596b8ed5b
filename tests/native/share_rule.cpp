// The share of a staging fill that crosses the link with its launch (pf_share.hpp):
// wherever the cut falls, it leaves whole fragments of the tail of the fill, of
// eligible units only, no more bytes than wanted and as many as fit, and never the
// whole fill.  Prints "all ok" and returns 0, or the first case that is wrong.
#include <cinttypes>
#include <cstdio>
#include <random>
#include <vector>

#include "../../pegaflow_amd/csrc/pf_share.hpp"

int main() {
  std::mt19937_64 rng(5);
  uint64_t cuts = 0, inside = 0, whole = 0;
  for (int round = 0; round < 200000; ++round) {
    std::vector<pf::ShareUnit> units(1 + rng() % 9);
    uint64_t total = 0;
    for (auto& u : units) {
      const uint64_t frags[] = {16, 1008, 4096, 16384, 32768, 73728, 1 << 20};
      u = {1 + rng() % (rng() % 2 ? 4 : 300), static_cast<uint32_t>(1 + rng() % 2), frags[rng() % 7], rng() % 8 != 0};
      total += u.n_blocks * u.n_seg * u.frag_bytes;
    }
    const uint64_t want = round % 2 ? pf::link_share_bytes(total) : rng() % (2 * total);
    const pf::ShareCut cut = pf::plan_link_share(units.size(), want, [&](size_t k) { return units[k]; });
    // The same fragment by fragment, from the end.
    uint64_t bytes = 0, left = 0;
    for (const auto& u : units) left += u.n_blocks * u.n_seg;
    size_t unit = units.size();
    uint64_t staged = 0;
    bool more = true;
    for (size_t k = units.size(); more && k-- > 0;) {
      uint64_t frags = units[k].n_blocks * units[k].n_seg;
      while (frags != 0 && (more = units[k].eligible && bytes + units[k].frag_bytes <= want && left > 1)) {
        bytes += units[k].frag_bytes;
        --frags;
        --left;
        unit = k;
        staged = frags;
      }
    }
    if (cut.bytes != bytes || cut.unit != unit || (bytes != 0 && cut.staged_frags != staged)) {
      printf("round %d: want %" PRIu64 ": unit %zu frags %" PRIu64 " bytes %" PRIu64 ", expected %zu %" PRIu64 " %" PRIu64 "\n",
             round, want, cut.unit, cut.staged_frags, cut.bytes, unit, staged, bytes);
      return 1;
    }
    cuts += bytes != 0;
    inside += bytes != 0 && staged != 0;
    whole += bytes != 0 && unit + 1 < units.size();
  }
  for (uint64_t frag = 1; frag < 100000; frag += 7) {
    for (const bool save : {false, true}) {
      const uint32_t w = pf::share_workgroups(frag, save);
      if (w < 16 || w > pf::kShareWorkgroupsMax) {
        printf("%u workgroups for fragments of %" PRIu64 "\n", w, frag);
        return 1;
      }
    }
  }
  if (cuts < 1000 || inside < 1000 || whole < 1000) {
    printf("only %" PRIu64 " cuts, %" PRIu64 " inside a unit, %" PRIu64 " of whole units\n", cuts, inside, whole);
    return 1;
  }
  printf("all ok\n");
  return 0;
}
