// The chunk arithmetic of the copy kernels (pf_chunks.hpp) against 64-bit
// arithmetic: wherever the rule cuts a fragment into chunks, the 32-bit counts and
// starts the kernels compute are exact and the chunks cover the fragment.  Prints
// "all ok" and returns 0, or the first case that is wrong.
#include <cinttypes>
#include <cstdio>
#include <vector>

#include "../../pegaflow_amd/csrc/pf_chunks.hpp"

int main() {
  std::vector<uint64_t> frags;
  for (uint64_t f = 1; f <= 300; ++f) frags.push_back(f);
  for (uint64_t f : {1000ull, 1008ull, 4112ull, 8176ull, 8191ull, 8192ull, 8200ull, 100004ull}) frags.push_back(f);
  for (uint64_t at : {1ull << 31, 1ull << 32, (1ull << 32) + 4096, 1ull << 33, 1ull << 35}) {
    for (uint64_t f = at - 64; f <= at + 64; ++f) frags.push_back(f);
  }
  uint64_t cut = 0;
  for (const uint64_t frag : frags) {
    for (const bool aligned : {false, true}) {
      for (const uint64_t far_starts : {1ull, 2ull, 4ull, 8ull, 16ull, 1000ull, 0x7f0000000010ull}) {
        for (const uint64_t blocks : {1ull, 7ull, 4096ull, 1ull << 27}) {
          for (const bool table : {false, true}) {
            const uint64_t span = table ? 0 : (blocks - 1) * 512 + frag;
            const uint32_t n = pf::chunks_per_fragment(frag, blocks, aligned, blocks == 7, table ? 1 : far_starts, span);
            if (n == 0) continue;
            ++cut;
            bool ok = frag <= 0xFFFFFFFFull && static_cast<uint64_t>(n) * blocks < (1ull << 31) && span <= 0xFFFFFFF0ull;
            const uint64_t starts = aligned ? 0 : table ? 1 : far_starts;
            for (uint32_t mis = 0; ok && mis < 16; ++mis) {
              const uint64_t lowest = starts & (~starts + 1);  // starts are multiples of it
              if (starts == 0 ? mis != 0 : mis % (lowest < 16 ? lowest : 16) != 0) continue;
              const uint32_t bytes = static_cast<uint32_t>(frag);
              const uint64_t need = (frag + mis + 15) / 16;
              ok = pf::chunk_count(bytes, mis) == need && need <= n;
              uint64_t reached = 0;
              for (uint64_t i = 0; ok && i < n; ++i) {
                if (i == 20 && n > 60) {  // the middle of a long fragment follows the same line
                  i = n - 20;
                  reached = 16 * i - mis;
                }
                const uint64_t raw = 16 * i > mis ? 16 * i - mis : 0;
                const uint64_t want = raw < frag - 16 ? raw : frag - 16;
                ok = pf::chunk_start(static_cast<uint32_t>(i), bytes, mis) == want && want <= reached;
                reached = want + 16;
              }
              ok = ok && reached == frag;
              if (!ok) printf("mis %u: ", mis);
            }
            if (!ok) {
              printf("%" PRIu64 " bytes x %" PRIu64 " blocks, aligned %d, starts %" PRIx64 ", table %d: %u chunks\n", frag,
                     blocks, aligned, far_starts, table, n);
              return 1;
            }
          }
        }
      }
    }
  }
  // The form is used where it pays: aligned fragments that fill three quarters of
  // the wavefronts of one step (loads from 2 KiB, saves from 3 KiB, up to 4 KiB)
  // and those from 8 KiB on keep to tiles.
  auto aligned = [](uint64_t frag, bool save) { return pf::chunks_per_fragment(frag, 16, true, save, 16, 0) != 0; };
  for (uint64_t f : {16ull, 1024ull, 1536ull, 2032ull, 2064ull, 2288ull, 4112ull, 5120ull, 6144ull, 8176ull}) {
    if (!aligned(f, false) || !aligned(f, true)) return printf("%" PRIu64 " bytes in tiles\n", f), 1;
  }
  for (uint64_t f : {2048ull, 2304ull, 2560ull, 3072ull, 3088ull, 3584ull, 4080ull, 4096ull, 8192ull, 16384ull}) {
    if (aligned(f, false) || aligned(f, true) != (f < 3072)) return printf("%" PRIu64 " bytes in chunks\n", f), 1;
  }
  if (pf::chunks_per_fragment(1000, 777, false, true, 8, 777000) != 63 ||
      pf::chunks_per_fragment(4096, 16, false, false, 8, 1 << 20) != 257 || cut < 1000) {
    printf("rule\n");
    return 1;
  }
  // In proportion, fragments keep 256 KiB in flight, no more than a fragment over; never fewer
  // workgroups than full tiles need nor more than the cap.
  for (uint64_t f = 1; f <= 40000; ++f) {
    const uint64_t tiles = pf::unit_workgroups(f, true, 16384, 16, 64);
    const bool ok = f >= 16384 ? tiles == 16 : tiles == 64 ? f <= 4161 : tiles * f >= 262144 && (tiles - 1) * f < 262144;
    const uint64_t multiple = pf::unit_workgroups(f, false, 16384, 16, 64);
    if (!ok || multiple < tiles || multiple > 64 || multiple % 16 != 0) {
      return printf("%" PRIu64 " bytes: %" PRIu64 " / %" PRIu64 " workgroups\n", f, tiles, multiple), 1;
    }
  }
  printf("all ok\n");
  return 0;
}
