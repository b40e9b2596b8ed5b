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
            const uint32_t n = pf::chunks_per_fragment(frag, blocks, aligned, table ? 1 : far_starts, span);
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
  // The form is used where it pays.
  if (pf::chunks_per_fragment(1000, 777, false, 8, 777000) != 63 || pf::chunks_per_fragment(4096, 16, true, 16, 0) != 256 ||
      pf::chunks_per_fragment(8192, 16, true, 16, 0) != 0 || cut < 1000) {
    printf("rule\n");
    return 1;
  }
  printf("all ok\n");
  return 0;
}
