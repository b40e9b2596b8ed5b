// The ranges that the direct backend makes of a descriptor batch.  Arithmetic alone,
// for the backend and its test.
#pragma once

#include <cstdint>
#include <vector>

#include "../../include/pegahip.h"

namespace pf {

// A merged range that keeps what the staged forms need.
struct Range {
  uint64_t device;
  uint8_t* host;
  uint64_t host_device;  // 0: not all of it can be reached through one mapping
  uint64_t size;
  uint64_t host_allocation;
};

// The reference's merge rule (memcpy.rs:25-55), keeping the host allocation of the
// descriptor that opened a range, and its device-visible address for as long as the
// descriptors behind it continue that as they continue the host address.  Where one has
// no mapping or another one, the range is merged all the same and goes over the link by
// copies that take the host address.
inline std::vector<Range> merge_ranges(const pf_copy_desc* copies, uint64_t n) {
  std::vector<Range> out;
  out.reserve(n);
  uint64_t run_first = 0;
  for (uint64_t i = 0; i < n; ++i) {
    const pf_copy_desc& c = copies[i];
    if (!out.empty()) {
      Range& run = out.back();
      const pf_copy_desc& first = copies[run_first];
      if (first.device_allocation == c.device_allocation &&
          first.host_allocation == c.host_allocation && run.device + run.size == c.device &&
          run.host + run.size == static_cast<uint8_t*>(c.host)) {
        if (run.host_device + run.size != c.host_device) run.host_device = 0;
        run.size += c.size;
        continue;
      }
    }
    run_first = i;
    out.push_back({c.device, static_cast<uint8_t*>(c.host), c.host_device, c.size,
                   c.host_allocation});
  }
  return out;
}

}  // namespace pf
