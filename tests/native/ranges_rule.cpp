// Ranges of the direct backend (pf_ranges.hpp): they hold every byte of the list in its
// order, merge by the reference's rule whatever the mapped addresses say, and name a
// mapped address only where every byte of the range lies behind it.  Prints "all ok" and
// returns 0, or the first case that is wrong.
#include <cinttypes>
#include <cstdio>
#include <random>
#include <vector>

#include "../../pegaflow_amd/csrc/pf_ranges.hpp"

int main() {
  std::mt19937_64 rng(11);
  uint64_t merged = 0, unmapped_tails = 0, other_mappings = 0;
  for (int round = 0; round < 100000; ++round) {
    // Where the next descriptor lies on each side if it continues the one before.
    std::vector<pf_copy_desc> list(1 + rng() % 12);
    uint64_t device = 1 << 20, host = 1 << 30, mapping = rng() % 2 ? 0 : uint64_t{1} << 40;
    uint64_t device_allocation = 0, host_allocation = 0;
    for (pf_copy_desc& c : list) {
      if (rng() % 6 == 0) device += 4096;
      if (rng() % 6 == 0) host += 4096;
      if (rng() % 6 == 0) ++device_allocation;
      if (rng() % 6 == 0) ++host_allocation;
      if (rng() % 4 == 0) mapping ^= uint64_t{1} << 41;
      const uint64_t sizes[] = {0, 16, 1000, 4096};
      const uint64_t size = sizes[rng() % 4];
      c = {device, reinterpret_cast<void*>(host), rng() % 4 ? mapping + host : 0, size, device_allocation, host_allocation};
      device += size;
      host += size;
    }
    const std::vector<pf::Range> ranges = pf::merge_ranges(list.data(), list.size());
    size_t i = 0;
    for (const pf::Range& r : ranges) {
      const size_t first = i;
      uint64_t size = 0;
      bool mapped = true;
      do {
        const pf_copy_desc& c = list[i];
        if (r.device + size != c.device || r.host + size != c.host || r.host_allocation != c.host_allocation ||
            list[first].device_allocation != c.device_allocation) {
          printf("round %d: descriptor %zu is not in the range of descriptor %zu\n", round, i, first);
          return 1;
        }
        mapped = mapped && c.host_device != 0 && c.host_device == list[first].host_device + size;
        unmapped_tails += i != first && list[first].host_device != 0 && c.host_device == 0;
        other_mappings += i != first && c.host_device != 0 && c.host_device != list[first].host_device + size;
        size += c.size;
        ++i;
      } while (i < list.size() && list[i].device_allocation == list[first].device_allocation &&
               list[i].host_allocation == list[first].host_allocation && r.device + size == list[i].device &&
               r.host + size == list[i].host);
      merged += i - first > 1;
      if (r.size != size || r.host_device != (mapped ? list[first].host_device : 0)) {
        printf("round %d: range of descriptors %zu to %zu: size %" PRIu64 " at %" PRIx64 ", expected %" PRIu64
               " %s mapped address\n", round, first, i - 1, r.size, r.host_device, size, mapped ? "with its" : "without a");
        return 1;
      }
    }
    if (i != list.size()) {
      printf("round %d: %zu of %zu descriptors\n", round, i, list.size());
      return 1;
    }
  }
  if (merged < 1000 || unmapped_tails < 1000 || other_mappings < 1000) {
    printf("only %" PRIu64 " merged ranges, %" PRIu64 " with an unmapped part, %" PRIu64 " with another mapping\n", merged,
           unmapped_tails, other_mappings);
    return 1;
  }
  printf("all ok\n");
  return 0;
}
