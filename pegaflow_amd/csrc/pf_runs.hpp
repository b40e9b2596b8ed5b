// As how many launches a staging fill goes out.  Arithmetic alone, for the planner and
// its tests.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace pf {

constexpr uint32_t kRowsLaunchUnits = 8;  // units one launch_block_tiles_rows call takes
constexpr uint64_t kStagedTileBytes = 2048;  // bytes one workgroup of the staged kernels moves
constexpr uint64_t staged_tiles(uint64_t frag_bytes) {
  return (frag_bytes + kStagedTileBytes - 1) / kStagedTileBytes;
}

struct LaunchUnit {
  uint64_t n_blocks;
  uint64_t n_seg;
  uint64_t frag_bytes;
};
struct LaunchRun {
  size_t begin, end;  // units of one launch
};

// Units too unlike for one grid leave it full of workgroups that find no
// tile.  Those are cheap but not free (they start and end at ~6 000 per
// microsecond), and so is every further launch (~8 us of ramp, tail and
// hand-over): the fill is cut into runs of units that keep three quarters
// of their grids busy, and goes out as one rows launch per run when that
// saves more idle workgroups than the launches cost.  A task over cache
// groups of unlike size (8 full-attention layers of 625 blocks among 40
// sliding-window layers of 8: 82 % of the units-inner grid idle) does:
// gather 240 -> 136 us, scatter 241 -> 140 us.  Layers of 72 KiB and of
// 8 KiB blocks in turn (44 % idle) do not: one launch 170 us, a launch
// per layer 242 us.  Empty: one launch for all units.
template <typename UnitAt>
std::vector<LaunchRun> plan_launch_runs(size_t n_units, UnitAt unit_at) {
  // Workgroups the one-launch form would start: the rows form (up to
  // kRowsLaunchUnits units) starts every row with the tiles of the largest
  // fragment and the segments of the widest unit; the units-inner form also
  // gives every unit the rows of the longest.
  uint64_t max_blocks = 0, max_seg = 0, max_tiles = 0, total_rows = 0;
  for (size_t k = 0; k < n_units; ++k) {
    const LaunchUnit u = unit_at(k);
    max_blocks = std::max(max_blocks, u.n_blocks);
    max_seg = std::max(max_seg, u.n_seg);
    max_tiles = std::max(max_tiles, staged_tiles(u.frag_bytes));
    total_rows += u.n_blocks;
  }
  const uint64_t started =
      (n_units <= kRowsLaunchUnits ? total_rows : max_blocks * n_units) * max_tiles * max_seg;
  std::vector<LaunchRun> runs;
  uint64_t runs_started = 0;
  for (size_t k = 0; k < n_units;) {
    size_t e = k;
    uint64_t run_useful = 0, run_rows = 0, run_tiles = 0, run_seg = 0;
    while (e < n_units && e - k < kRowsLaunchUnits) {
      const LaunchUnit u = unit_at(e);
      const uint64_t tiles = staged_tiles(u.frag_bytes);
      const uint64_t nu = run_useful + u.n_blocks * tiles * u.n_seg;
      const uint64_t nr = run_rows + u.n_blocks;
      const uint64_t nt = std::max(run_tiles, tiles);
      const uint64_t ns = std::max(run_seg, u.n_seg);
      if (e > k && nu * 4 < nr * nt * ns * 3) break;
      run_useful = nu;
      run_rows = nr;
      run_tiles = nt;
      run_seg = ns;
      ++e;
    }
    runs.push_back({k, e});
    runs_started += run_rows * run_tiles * run_seg;
    k = e;
  }
  constexpr uint64_t kIdleWorkgroupsPerUs = 6000, kLaunchUs = 8;
  const bool in_runs = runs.size() > 1 && started > runs_started &&
                       (started - runs_started) / kIdleWorkgroupsPerUs > (runs.size() - 1) * kLaunchUs;
  return in_runs ? runs : std::vector<LaunchRun>();
}

}  // namespace pf
