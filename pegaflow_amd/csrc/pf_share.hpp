// Which part of a staging fill crosses the link with the gather / scatter launch
// itself.  Arithmetic alone, for the planner and its test.
#pragma once

#include <cstddef>
#include <cstdint>

namespace pf {

// A fill's link copy and its gather or scatter take turns on one stream, so the
// link has nothing to do while the launch moves the fill through HBM.  The launch
// therefore also moves a share of the fill straight between the cache and host
// memory, with a few workgroups of its own, and the link copy is shorter by it.  A
// launch of b bytes alone takes 4-6 us and b / 3.05 TB/s, in which the link moves b / 53
// and 250-350 KB; the share is about that much.  It does not ride along for nothing:
// with it the launch of a full slot of 512 MiB takes 186 us instead of 176 (16 KiB
// fragments: 193 instead of 178) for a link copy that is 10.4 MB = 181 us shorter.
// (A longer share gains nothing: the launch then waits for it instead of the link copy
// for the launch.)  Measured on MI355X, calls back to back,
// save / load in us without a share, with 64 KiB and b / 44, b / 52, b / 60: one layer
// of 20 MB 393.9 / 395.6, 390.5 / 389.4, 390.1 / 388.9, 389.9 / 389.0; 524 MB in twelve
// 9437 / 9409, 9247 / 9194, 9254 / 9228, 9277 / 9252; 1.3 GB in four 23 352 / 23 223,
// 23 106 / 23 001, 23 107 / 23 004, 23 135 / 23 053.  Link copies on a stream of their
// own run under the launches as it is: there a share only adds a third user of the
// link (a save and a load at once fell from 88 to 35 GB/s together in one repetition
// of nine).
constexpr uint64_t kShareBase = 64 << 10;
constexpr uint64_t kSharePart = 52;
constexpr uint64_t link_share_bytes(uint64_t launch_bytes) {
  return kShareBase + launch_bytes / kSharePart;
}

// A unit of a fill: n_blocks list positions of n_seg fragments, in the order
// (segment, position) both in the slot and in the host image.
struct ShareUnit {
  uint64_t n_blocks;
  uint32_t n_seg;
  uint64_t frag_bytes;
  bool eligible;  // its fragments can be moved over mapped host memory in 16-byte words
};

// The share is the tail of the fill, so that link copies which cross layers stay
// one copy: units [0, unit) and the first `staged_frags` fragments of unit `unit`
// go through the slot, everything behind them over the link.  bytes = 0: no share
// (unit = number of units).
struct ShareCut {
  size_t unit = 0;
  uint64_t staged_frags = 0;
  uint64_t bytes = 0;
};
// As many whole fragments as `want` holds, from the end of the fill up to the first
// unit that is not eligible; never the whole fill.
template <typename UnitAt>
ShareCut plan_link_share(size_t n_units, uint64_t want, UnitAt unit_at) {
  ShareCut cut;
  cut.unit = n_units;
  for (size_t k = n_units; k-- > 0;) {
    const ShareUnit u = unit_at(k);
    const uint64_t frags = u.n_blocks * u.n_seg;
    if (!u.eligible || u.frag_bytes == 0) break;
    uint64_t take = (want - cut.bytes) / u.frag_bytes;
    if (take > frags) take = frags;
    if (k == 0 && take == frags && take != 0) --take;
    if (take == 0) break;
    cut.unit = k;
    cut.staged_frags = frags - take;
    cut.bytes += take * u.frag_bytes;
    if (take != frags) break;
  }
  return cut;
}

// The same where pages are packed whole: pages at the end of a chunk of `count`.
constexpr uint64_t link_share_pages(uint64_t count, uint64_t page_bytes) {
  const uint64_t pages = link_share_bytes(count * page_bytes) / page_bytes;
  return pages < count ? pages : 0;
}

// A workgroup of a share moves a tile of one fragment at a time.  Full tiles keep
// the link busy with 16 workgroups on the way out, whose stores nobody waits for,
// and with 32 on the way in; more of them slow the rest of the launch (524 MB saved
// with 16 / 32 / 64 in 9267 / 9338 / 9342 us).  Smaller fragments take
// proportionally more (20 MB of 1 KiB fragments loaded with 16 / 64 / 256 in 444 /
// 409 / 411, without a share in 415).
constexpr uint64_t kShareTileBytes = 8192;
constexpr uint32_t kShareWorkgroupsMax = 256;
constexpr uint32_t share_workgroups(uint64_t min_frag, bool save) {
  const uint32_t full = save ? 16 : 32;
  if (min_frag == 0 || min_frag >= kShareTileBytes) return full;
  const uint64_t n = full * ((kShareTileBytes + min_frag - 1) / min_frag);
  return n < kShareWorkgroupsMax ? static_cast<uint32_t>(n) : kShareWorkgroupsMax;
}

}  // namespace pf
