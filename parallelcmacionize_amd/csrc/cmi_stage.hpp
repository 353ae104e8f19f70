// cmi_stage.hpp -- host <-> device transfers of a context's cell fields, whose
// order differs on the two sides (CellOrder).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "cmi_device.hpp"

namespace cmi {

// The reference's cell order (subgrid-major, ix*ny*nz + iy*nz + iz within a
// subgrid) and the device's (subgrid, tile, cell within the tile) of one grid.
struct CellOrder {
  int sc[3];      // cells per subgrid per axis
  int tshift[3];  // log2 of the tile size per axis
  int ntile[3];   // tiles per subgrid per axis
  int tile_cells;
  int cps;        // cells per subgrid
};

inline CellOrder cell_order(const GridDev &g) {
  CellOrder o;
  for (int a = 0; a < 3; ++a) {
    o.sc[a] = g.sc[a];
    o.tshift[a] = g.tshift[a];
    o.ntile[a] = g.ntile[a];
  }
  o.tile_cells = g.tile_cells;
  o.cps = g.cps;
  return o;
}

// One field of a transfer: the caller's array, the device's, and what every
// cell is multiplied by on the way.
struct CellField {
  double *host;
  double *dev;
  double scale;
};

// Pinned buffers that transfers go through, piece by piece.  Made at the first
// transfer, freed with the context.  One transfer at a time (a context's calls
// are serialised by its owner).
class Stage {
 public:
  ~Stage();
  // Fields of n cells between the caller's order and the device's, behind
  // what is queued on the stream.  A download is complete on return.  After an
  // upload the caller's arrays are free; it waits for the stream before the
  // next transfer.
  hipError_t upload_cells(int device, hipStream_t st, const CellOrder &o, size_t n,
                          const CellField *fields, int nfields);
  hipError_t download_cells(int device, hipStream_t st, const CellOrder &o, size_t n,
                            const CellField *fields, int nfields);

 private:
  static constexpr int kThreads = 4;            // host threads of a large transfer
  static constexpr int kSlots = 2 * kThreads;   // two per thread
  static constexpr size_t kPiece = 1u << 20;    // bytes of a slot
  static constexpr size_t kSmall = 1u << 17;    // bytes of a small download
  unsigned char *h_[kSlots] = {};
  hipEvent_t ev_[kSlots] = {};

  hipError_t ensure(int slots);
  template <class Piece>
  hipError_t run(int device, hipStream_t st, bool upload, size_t bytes, int arrays,
                 const Piece &piece);
};

}  // namespace cmi
