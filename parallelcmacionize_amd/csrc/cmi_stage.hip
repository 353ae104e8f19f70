// cmi_stage.hip -- transfers through pinned pieces, and the kernels that put
// cells into the other side's order on the way.
//
// A field of a 256^3 grid is 134 MB.  Reordering it on the host, cell by cell,
// and copying it from or to pageable memory made two fields take 55 ms in and
// 77 ms out.  Here the kernels below read or write the pinned pieces directly
// (PCIe-bound, 57 GB/s: the reordering costs nothing on top), and up to four
// host threads move pieces between the caller's array and the pinned buffers
// (one thread moves 25 GB/s, less into fresh pages): 6.4 and 8.5 ms.  Copies
// to a device buffer and kernels from there: 10 and 11.6.  Eight threads: 6.4
// and 7.0; pieces of half a MB: 8.2 and 8.2.  At 64^3 0.50 -> 0.18 and 1.19 ->
// 0.27 ms, at 32^3 0.22 -> 0.08 and 0.09 -> 0.045.
#include "cmi_stage.hpp"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <thread>

namespace cmi {

// Device cell of reference cell r (mirrors cell_addr()).
__device__ __forceinline__ size_t device_cell(const CellOrder &o, size_t r) {
  const size_t sub = r / (unsigned)o.cps;
  unsigned k = (unsigned)(r - sub * (unsigned)o.cps);
  const unsigned iz = k % (unsigned)o.sc[2];
  k /= (unsigned)o.sc[2];
  const unsigned iy = k % (unsigned)o.sc[1], ix = k / (unsigned)o.sc[1];
  const unsigned tx = ix >> o.tshift[0], ty = iy >> o.tshift[1], tz = iz >> o.tshift[2];
  const unsigned lx = ix - (tx << o.tshift[0]), ly = iy - (ty << o.tshift[1]),
                 lz = iz - (tz << o.tshift[2]);
  const unsigned t = (tx * o.ntile[1] + ty) * o.ntile[2] + tz;
  const unsigned l = (((lx << o.tshift[1]) + ly) << o.tshift[2]) + lz;
  return sub * (size_t)o.cps + (size_t)t * o.tile_cells + l;
}

// Bit for bit the value where there is nothing to scale.
__device__ __forceinline__ double scaled(double v, double scale) {
  return scale == 1. ? v : v * scale;
}

// n cells from reference cell r0 on: a piece in the reference's order into the
// device field, and back.
__global__ void __launch_bounds__(256) cells_in_kernel(CellOrder o, const double *__restrict__ piece,
                                                       size_t r0, unsigned n, double scale,
                                                       double *__restrict__ field) {
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    field[device_cell(o, r0 + i)] = scaled(piece[i], scale);
}
__global__ void __launch_bounds__(256) cells_out_kernel(CellOrder o, const double *__restrict__ field,
                                                        size_t r0, unsigned n, double scale,
                                                        double *__restrict__ piece) {
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    piece[i] = scaled(field[device_cell(o, r0 + i)], scale);
}

Stage::~Stage() {
  for (int s = 0; s < kSlots; ++s) {
    if (h_[s]) (void)hipHostFree(h_[s]);
    if (ev_[s]) (void)hipEventDestroy(ev_[s]);
  }
}

hipError_t Stage::ensure(int slots) {
  hipError_t e = hipSuccess;
  for (int s = 0; s < slots && e == hipSuccess; ++s) {
    if (!h_[s]) e = hipHostMalloc(reinterpret_cast<void **>(&h_[s]), kPiece);
    if (e == hipSuccess && !ev_[s])
      e = hipEventCreateWithFlags(&ev_[s], hipEventDisableTiming);
  }
  return e;
}

// Calls piece(slot, array, offset, bytes, begin) for every piece of `arrays`
// arrays of `bytes` each, twice: first with begin set (queue the work of the
// slot), and, before the slot is used again or at the end, without it (that
// work is done).  Pieces are dealt to the threads in turn; a thread works its
// two slots in turn.  Up to two pieces need no events: an upload is left to the
// caller's wait, a small download waits for the stream (two fields of 16^3 cells
// in and out 20 and 21 us, 24 and 24 with events; of 48^3 cells out 105 us, 93
// with events, whose copies to the caller overlap the other field's transfer).
template <class Piece>
hipError_t Stage::run(int device, hipStream_t st, bool upload, size_t bytes, int arrays,
                      const Piece &piece) {
  if (bytes == 0 || arrays == 0) return hipSuccess;
  const size_t each = (bytes + kPiece - 1) / kPiece, pieces = each * (size_t)arrays;
  // a thread is worth its start (tens of us) from four pieces on
  const int threads = (int)std::max<size_t>(1, std::min<size_t>(kThreads, pieces / 4));
  const hipError_t ee = ensure((int)std::min<size_t>(2 * threads, pieces));
  if (ee != hipSuccess) return ee;
  std::atomic<int> first_error{(int)hipSuccess};
  auto call = [&](int slot, size_t p, bool begin) {
    const size_t off = (p % each) * kPiece;
    return piece(slot, (int)(p / each), off, std::min(kPiece, bytes - off), begin);
  };
  if (pieces <= 2 && (upload || bytes * (size_t)arrays <= kSmall)) {
    hipError_t e = hipSetDevice(device);
    for (size_t p = 0; p < pieces && e == hipSuccess; ++p) e = call((int)p, p, true);
    if (upload && e == hipSuccess) return e;
    const hipError_t w = hipStreamSynchronize(st);
    if (e == hipSuccess) e = w;
    for (size_t p = 0; p < pieces && e == hipSuccess; ++p) e = call((int)p, p, false);
    return e;
  }
  auto work = [&](int t) {
    hipError_t e = hipSetDevice(device);
    size_t held[2];  // the slots' pieces
    bool busy[2] = {false, false};
    auto finish = [&](int k) {
      if (!busy[k]) return;
      busy[k] = false;
      const int s = 2 * t + k;
      const hipError_t w = hipEventSynchronize(ev_[s]);
      if (e == hipSuccess) e = w;
      if (e == hipSuccess) e = call(s, held[k], false);
    };
    int k = 0;
    for (size_t p = (size_t)t; p < pieces && e == hipSuccess; p += (size_t)threads, k ^= 1) {
      finish(k);
      if (e != hipSuccess) break;
      held[k] = p;
      e = call(2 * t + k, p, true);
      if (e == hipSuccess) e = hipEventRecord(ev_[2 * t + k], st);
      busy[k] = e == hipSuccess;
    }
    finish(k);
    finish(k ^ 1);
    if (e != hipSuccess) {
      (void)hipStreamSynchronize(st);  // nothing in flight uses the slots
      first_error = (int)e;
    }
  };
  std::thread extra[kThreads];
  int started = 1;
  for (; started < threads; ++started) {
    try {
      extra[started] = std::thread(work, started);
    } catch (const std::exception &) {
      break;  // no more threads: their pieces are done here
    }
  }
  work(0);
  for (int t = started; t < threads; ++t) work(t);
  for (int t = 1; t < started; ++t) extra[t].join();
  return (hipError_t)first_error.load();
}

hipError_t Stage::upload_cells(int device, hipStream_t st, const CellOrder &o, size_t n,
                               const CellField *fields, int nfields) {
  return run(device, st, true, n * sizeof(double), nfields,
             [&](int s, int a, size_t off, size_t len, bool begin) -> hipError_t {
               if (!begin) return hipSuccess;
               const CellField &f = fields[a];
               memcpy(h_[s], reinterpret_cast<const unsigned char *>(f.host) + off, len);
               const unsigned m = (unsigned)(len / sizeof(double));
               hipLaunchKernelGGL(cells_in_kernel, dim3((m + 255) / 256), dim3(256), 0, st, o,
                                  reinterpret_cast<const double *>(h_[s]), off / sizeof(double),
                                  m, f.scale, f.dev);
               return hipGetLastError();
             });
}

hipError_t Stage::download_cells(int device, hipStream_t st, const CellOrder &o, size_t n,
                                 const CellField *fields, int nfields) {
  return run(device, st, false, n * sizeof(double), nfields,
             [&](int s, int a, size_t off, size_t len, bool begin) -> hipError_t {
               const CellField &f = fields[a];
               if (!begin) {
                 memcpy(reinterpret_cast<unsigned char *>(f.host) + off, h_[s], len);
                 return hipSuccess;
               }
               const unsigned m = (unsigned)(len / sizeof(double));
               hipLaunchKernelGGL(cells_out_kernel, dim3((m + 255) / 256), dim3(256), 0, st, o,
                                  f.dev, off / sizeof(double), m, f.scale,
                                  reinterpret_cast<double *>(h_[s]));
               return hipGetLastError();
             });
}

}  // namespace cmi
