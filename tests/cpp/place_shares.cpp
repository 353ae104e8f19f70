// Every piece of every visit is placed by exactly one workgroup, whatever the
// number of visits, workgroups and packets of a chunk (cmi_place.hpp), and the
// arithmetic stays within 32 bits.
#include <stdio.h>

#include <vector>

#include "../../parallelcmacionize_amd/csrc/cmi_place.hpp"

using namespace cmi;

static bool check(uint32_t visits, uint32_t blocks, uint32_t chunk) {
  const uint32_t pieces = (uint32_t)(((uint64_t)chunk + kPlacePiece - 1) / kPlacePiece);
  const uint32_t parts = place_share(0, blocks, chunk).parts;
  std::vector<unsigned char> seen((size_t)visits * parts, 0);
  uint64_t done = 0;
  for (uint32_t b = 0; b < blocks; ++b) {
    const PlaceShare s = place_share(b, blocks, chunk);
    if (s.parts != parts || s.part >= parts || s.visit_step == 0) return false;
    uint64_t next = s.visit;
    for (uint32_t v = s.visit; v < visits; v += s.visit_step) {
      if (v != next || seen[(size_t)v * parts + s.part]++) return false;
      next = (uint64_t)v + s.visit_step;
      ++done;
    }
  }
  if (done != (uint64_t)visits * parts) return false;
  // the parts' pieces are the visit's, each once; a full visit's last slot is reached
  std::vector<unsigned char> piece(pieces, 0);
  for (uint32_t p = 0; p < parts; ++p)
    for (uint64_t i0 = (uint64_t)p * kPlacePiece; i0 < chunk; i0 += (uint64_t)parts * kPlacePiece) {
      if (i0 + (uint64_t)parts * kPlacePiece > 0xffffffffull) return false;
      if (piece[i0 / kPlacePiece]++) return false;
    }
  for (unsigned char c : piece)
    if (c != 1) return false;
  return true;
}

int main() {
  for (uint32_t visits : {1u, 2u, 511u, 12207u, (1u << 18) - 1u, 1u << 18, 274625u, 1u << 21})
    for (uint32_t blocks : {1u, 2u, 7u, 256u, 512u})
      for (uint32_t chunk : {1u, 256u, 4095u, 4096u, 4097u, 8192u, 14336u, 32769u, 1u << 20,
                             1u << 23, 1u << 26})
        if (!check(visits, blocks, chunk)) {
          printf("visits %u blocks %u chunk %u\n", visits, blocks, chunk);
          return 1;
        }
  printf("ok\n");
  return 0;
}
