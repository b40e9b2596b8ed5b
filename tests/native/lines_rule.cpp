// Chunks along the link's packets (line_chunk of pf_chunks.hpp): put together as the
// kernel does it, they write every byte of a range once or more with its own value
// and none outside; starts off the range's ends are 16-byte aligned.  Prints "all ok"
// and returns 0, or the first case that is wrong.
#include <cstdio>
#include <vector>

#include "../../pegaflow_amd/csrc/pf_chunks.hpp"

namespace {
bool check(uint32_t frag, uint32_t n, uint32_t lead, uint32_t tile_chunks) {
  const uint32_t range = frag * n, total = pf::line_chunk_count(range);
  const uint32_t launched = (total + tile_chunks - 1) / tile_chunks * tile_chunks;
  std::vector<int> image(range, -1);
  auto byte = [&](uint32_t pos, uint32_t at) { return static_cast<int>((pos * 31 + at * 7) & 255); };
  for (uint32_t i = 0; i < launched; ++i) {
    const pf::LineChunk c = pf::line_chunk(i, lead, range, frag);
    if (c.start + 16 > range || c.pos >= n || c.tail == 0 || c.tail > 16) return false;
    if (i >= total && c.any) return false;
    const uint32_t at = c.tail < 16 ? frag - 16 : c.start - c.pos * frag;
    if (at + 16 > frag || (c.tail < 16 && c.pos + 1 >= n)) return false;
    if (!c.any) continue;
    if (c.start != 0 && c.start != range - 16 && ((lead + c.start) & 15) != 0) return false;
    for (uint32_t b = 0; b < 16; ++b) {
      int value;
      if (c.tail == 16) {
        value = byte(c.pos, at + b);
      } else {
        value = b < c.tail ? byte(c.pos, at + 16 - c.tail + b) : byte(c.pos + 1, b - c.tail);
      }
      const uint32_t where = c.start + b;
      if (value != byte(where / frag, where % frag)) return false;
      image[where] = value;
    }
  }
  for (const int v : image) {
    if (v < 0) return false;
  }
  return true;
}
}  // namespace

int main() {
  for (uint32_t frag = 16; frag < 140; ++frag) {
    for (const uint32_t n : {1u, 2u, 3u, 17u}) {
      for (uint32_t lead = 0; lead < 256; ++lead) {
        if (!check(frag, n, lead, 256)) {
          printf("fragments of %u, %u of them, %u past a packet\n", frag, n, lead);
          return 1;
        }
      }
    }
  }
  for (const uint32_t frag : {1000u, 1023u, 4097u, 20004u}) {
    for (uint32_t lead = 0; lead < 256; ++lead) {
      if (!check(frag, 41, lead, 1024)) {
        printf("fragments of %u, %u past a packet\n", frag, lead);
        return 1;
      }
    }
  }
  // The last chunks of the longest range, without the bytes.
  const uint32_t range = static_cast<uint32_t>(pf::kMaxLinesRange), total = pf::line_chunk_count(range);
  for (uint32_t i = total - 10; i < total + 2048; ++i) {
    const pf::LineChunk c = pf::line_chunk(i, 255, range, range);
    const bool in = 16ull * i < 255ull + range;
    if (c.any != in || c.pos != 0 || c.tail != 16 || c.start > range - 16) {
      printf("chunk %u of the longest range\n", i);
      return 1;
    }
  }
  printf("all ok\n");
  return 0;
}
