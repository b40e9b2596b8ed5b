// The 16-byte chunks a fragment is cut into (kUnitChunks units and the tiles of
// unaligned copies).  Arithmetic alone, for the kernels and the planner alike.
#pragma once

#include <cstdint>

namespace pf {

// Chunk boundaries lie on 16-byte boundaries of one side, whose address is `mis`
// past one; the first and the last chunk overlap their neighbour and carry the
// same bytes, so nothing is moved byte by byte: chunk i starts at
// clamp(16 i - mis, 0, bytes - 16).  Needs 16 <= bytes <= kMaxChunkedBytes.
constexpr uint64_t kMaxChunkedBytes = 0xFFFFFFFFull - 30;  // bytes + mis + 15 stays in 32 bits
constexpr uint32_t chunk_count(uint32_t bytes, uint32_t mis) { return (bytes + mis + 15u) >> 4; }
constexpr uint32_t chunk_start(uint32_t i, uint32_t bytes, uint32_t mis) {
  const uint32_t raw = 16u * i;
  const uint32_t in = raw > mis ? raw - mis : 0u;
  const uint32_t last = bytes - 16u;
  return in < last ? in : last;
}

// 16-byte chunks of a fragment of a zero-copy unit that is to be cut into chunks
// (kUnitChunks), 0 when it keeps to tiles of one fragment.  `aligned`: every
// fragment of the unit starts on a 16-byte boundary on both sides; `far_starts`:
// the bitwise or of the numbers the host addresses of its fragments are sums of
// multiples of (segment bases and stride), 1 when they come from a table;
// `far_span`: bytes from the first to the end of the last fragment of a segment
// in host memory, 0 for a table.
//
// Chunks are the faster form for every fragment off the 16-byte grid and, on it,
// for fragments below 8 KiB, whose tiles leave lanes without work, except where
// one step of a tile takes the fragment whole and fills three quarters of its
// wavefronts (fills_one_step): there both reach the link's rate in a long call
// and the tile form, whose ids are scalar loads, is ahead in a short one.
// Measured on MI355X, two layers of K and V, 1 / 4 / 20 MB per call, loads in us,
// chunks against tiles: 2048 bytes 24.1 / 76.3 / 361 against 21.7 / 74.4 / 363,
// 3072 bytes 24.1 / 76.4 / 365 against 21.9 / 74.0 / 353, 4096 bytes 24.1 / 76.4 /
// 356 against 21.8 / 74.6 / 353, but 1040 bytes 24.4 / 77.9 / 375 against 28.0 /
// 101 / 507, 4112 bytes 23.3 / 77.7 / 359 against 22.7 / 80.5 / 380, 7680 bytes
// 22.2 / 75.8 / 354 against 21.9 / 76.2 / 366.  Saves gain from tiles later: 30
// layers, 20 MB, 2048 bytes 363 against 375, 2560 bytes 362 / 365, 3072 bytes 364 /
// 363.
constexpr bool fills_one_step(uint64_t frag, bool save) {
  return frag >= (save ? 3072 : 2048) && frag <= 4096 && frag * 4 >= 3 * ((frag + 1023) / 1024 * 1024);
}
constexpr uint32_t chunks_per_fragment(uint64_t frag, uint64_t n_blocks, bool aligned, bool save,
                                       uint64_t far_starts, uint64_t far_span) {
  // The kernel's chunk arithmetic is 32 bits wide and a segment's host image is
  // one buffer descriptor; the tile form counts in 64 bits.
  if (frag < 16 || frag > kMaxChunkedBytes || far_span > 0xFFFFFFF0ull) return 0;
  if (aligned && (frag >= 8192 || fills_one_step(frag, save))) return 0;
  // A fragment whose host side starts off a 16-byte boundary may have one chunk
  // more: the furthest off is what the alignment of all starts leaves open (1000
  // bytes at multiples of 8: 63 chunks either way).
  const uint64_t starts = aligned ? 16 : far_starts | 16;
  const uint64_t alignment = starts & (~starts + 1);
  const uint64_t chunks = (frag + (16 - alignment) + 15) / 16;
  if (chunks * n_blocks >= (1ull << 31)) return 0;
  return static_cast<uint32_t>(chunks);
}

// A segment whose host image is one gapless range is cut along the link's packets
// of 256 bytes instead (kUnitLines): chunk c is what lies of the range in the 16
// bytes from 16 c - lead on, `lead` being the range's start modulo 256; the chunks
// that stick out are shifted inwards.  A chunk may hold the end of one fragment and
// the head of the next, `tail` being the bytes of the first (16: all).  Needs
// frag >= 16 and a range of at most kMaxLinesRange (the starts of a whole last tile
// stay in 32 bits).
constexpr uint64_t kMaxLinesRange = 0xFFFFFFFFull - (64 << 10);
constexpr uint32_t kLinkPacket = 256;
constexpr uint32_t line_chunk_count(uint32_t range) { return (range + (kLinkPacket - 1) + 15u) >> 4; }
struct LineChunk {
  uint32_t start;  // in the range
  uint32_t pos;    // list position of its first byte
  uint32_t tail;
  bool any;        // something of the range lies in it
};
constexpr LineChunk line_chunk(uint32_t c, uint32_t lead, uint32_t range, uint32_t frag) {
  const uint32_t raw = 16u * c;
  const uint32_t in = raw > lead ? raw - lead : 0u;
  const uint32_t start = in < range - 16u ? in : range - 16u;
  const uint32_t pos = start / frag;
  const uint32_t left = (pos + 1) * frag - start;
  return {start, pos, left < 16u ? left : 16u, raw + 16u > lead && in < range};
}
// Workgroups that a unit of a zero-copy launch needs to keep the link full: of
// full tiles `full_tiles`, more of smaller ones, at most `most`.  Saves and units
// in chunks take a whole multiple for every started share of a tile; a load of
// whole fragments takes them in proportion, since reads beyond what the link holds
// slow it down: fragments of 12 288 bytes had 32 workgroups and 393 KB in flight
// and loaded (20 MB) in 367 us, with 22 in 352; 11 264 bytes 364 -> 352, 14 336
// bytes 364 -> 352, 15 360 bytes 362 -> 353.  (In proportion, saves of 24 layers of
// 13 312-byte fragments, 5 MB, took 86 us instead of 82, and loads in chunks, 30
// layers of 7680 bytes, 382 instead of 360: chunks wait for their ids first.)
constexpr uint32_t unit_workgroups(uint64_t frag, bool in_proportion, uint32_t tile, uint32_t full_tiles,
                                   uint32_t most) {
  if (frag == 0 || frag >= tile) return full_tiles;
  const uint64_t n = in_proportion ? (static_cast<uint64_t>(full_tiles) * tile + frag - 1) / frag
                                   : full_tiles * ((tile + frag - 1) / frag);
  return n < most ? static_cast<uint32_t>(n) : most;
}

}  // namespace pf
