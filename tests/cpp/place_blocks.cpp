// Workgroups of a placement (cmi_place.hpp): within what a launch takes, and no
// workgroup in charge of many visits while others are free.
#include <stdio.h>

#include <initializer_list>

#include "../../parallelcmacionize_amd/csrc/cmi_place.hpp"

using namespace cmi;

int main() {
  for (uint64_t tiles : {1ull, 8ull, 512ull, 8192ull, 1ull << 21})
    for (uint64_t packets : {1ull, 64ull, 640ull, 100000ull, 1ull << 25, 0xfffffff0ull})
      for (uint32_t most : {256u, 512u}) {
        const uint32_t b = place_blocks(packets, tiles, most);
        const uint64_t visits = packets < tiles ? packets : tiles;
        if (b < 1 || b > most || (b < visits && b < most) || (b < packets / 1024 && b < most)) {
          printf("tiles %llu packets %llu: %u\n", (unsigned long long)tiles,
                 (unsigned long long)packets, b);
          return 1;
        }
      }
  printf("ok\n");
  return 0;
}
