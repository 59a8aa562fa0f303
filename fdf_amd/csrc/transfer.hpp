// transfer.hpp -- host arrays to and from the device (transfer.hip).
#pragma once
#include "kernels.hpp"

namespace picgpu {

// what a host array of 64-bit values is on the device
enum class HostKind {
  Copy8,      // the same 8 bytes
  Real,       // double: `real` of the context's precision
  Int32,      // int64: int32
  Cell,       // int64[3]: packed cell, -1 outside the grid
  NodeCount,  // double per node slot: int32 per cell, 0 in the other slots (download)
  NodeReal,   // double per node slot: real per cell, 0 in the other slots (download)
  Volfrac,    // double per face: face volume fractions of direction dir from its counts (download)
};
struct HostSeg {
  HostKind kind;
  void *dev, *host;  // host is read only by an upload
  int64_t n;         // elements
  size_t stride;     // bytes of an element on the host: 24 for Cell, else 8
  int dir = 0;
};

// every context between its creation and its destruction: the pinned slots
// are kept while there is one
void rings_open();
void rings_close();

// Both wait until the arrays have been moved.
int host_download(picgpu_ctx *c, const HostSeg *segs, int nsegs);
int host_upload(picgpu_ctx *c, const HostSeg *segs, int nsegs);
// dev[0..n) = v in the context's precision, without waiting
int fill_real(picgpu_ctx *c, void *dev, int64_t n, double v);

}  // namespace picgpu
