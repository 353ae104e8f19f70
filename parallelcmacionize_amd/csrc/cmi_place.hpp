// cmi_place.hpp -- how the workgroups of a placement share the survivors of a
// round's visits.  Plain arithmetic, on the host as on the device.
#pragma once

#include <stdint.h>

namespace cmi {

// Slots that a workgroup places at a time.
constexpr uint32_t kPlacePiece = 4096;

// A visit holds up to `chunk` survivors (the chunk that the round's plan cut,
// not the configured one: late rounds hold a few hundred packets a visit
// whatever is configured).  A visit of more than one piece is shared by up to
// kPlaceParts workgroups, its part p by pieces p, p + parts, ...; the visits
// go to the groups of `parts` workgroups in turn.  No number of all pieces is
// formed: 2^18 visits of 2^26-packet chunks have 2^32.  Eight parts: a round
// of chunks beyond 32768 packets has about a visit per resident workgroup
// (the plan's cut), enough for the launch.  256^3 cells, 2e7 packets, a
// transport at configured chunks of 8192, 2^16, 2^20 and 2^24: 5.5, 5.6, 5.6
// and 5.6 ms; with pieces counted from the configured chunk 5.5, 6.4, 20.8
// and 77.6.
constexpr uint32_t kPlaceParts = 8;

struct PlaceShare {
  uint32_t visit, visit_step;  // visits visit, visit + visit_step, ...
  uint32_t part, parts;        // pieces part, part + parts, ... of each
};

constexpr PlaceShare place_share(uint32_t block, uint32_t blocks, uint32_t chunk) {
  const uint32_t pieces = chunk / kPlacePiece + (chunk % kPlacePiece != 0 ? 1u : 0u);
  uint32_t parts = pieces < kPlaceParts ? pieces : kPlaceParts;
  if (parts > blocks) parts = blocks;
  if (parts == 0) parts = 1;
  const uint32_t step = blocks / parts;
  // workgroups beyond the last whole group have no share
  return PlaceShare{block < step * parts ? block / parts : 0xffffffffu, step, block % parts, parts};
}

// Workgroups of a placement: one per 1024 packets of the transport, and one
// per visit that a round of few packets can have (a visit costs its workgroup
// a chain of loads whatever it holds), up to `most`.  One workgroup for all of
// 512 visits make an iteration of 64 problems of 8 tiles, 10 packets each,
// take 0.53 ms instead of 0.28, of 1 packet each 0.38 instead of 0.28.
constexpr uint32_t place_blocks(uint64_t packets, uint64_t tiles, uint32_t most) {
  const uint64_t visits = packets < tiles ? packets : tiles;
  uint64_t blocks = packets / 1024 + 1;
  if (blocks < visits) blocks = visits;
  return blocks < most ? (uint32_t)blocks : most;
}

}  // namespace cmi
