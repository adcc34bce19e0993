// transfer.hpp -- per-node arrays between HBM and pageable host arrays
// (transfer.hip): populations, density and velocity in FP64 node order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "d3q19.hpp"

namespace hlbm {

// One per-node array: N values of the device's type in the node layout on the
// device, FP64 on the host.  q: the direction of a population plane in the
// domain's storage type (shifted storage adds or subtracts the rest state), or
// -1 for a plain FP64 array.
struct NodePlane {
  void* dev;
  double* host;  // first value of the host array (read only for planes_to_device)
  int q;
};

// The grid, its device layout and the host layout: node order (x fastest, N
// values per plane) or the reference's All box with two ghost layers, of which
// only the Real nodes are read or written.
struct TransferGrid {
  int n[3];
  NodeLayout lay;
  bool reference;
  int storage;
  RestShift shift;
};

// The pinned slots of a domain's transfers: had by its first large one (8 MiB, 16
// MiB from the first of 64 MiB and more), its own until it is destroyed.  Every
// destroyed domain calls return_ring, with its ring or nullptr: one ring per
// device waits there for the next domain.
struct TransferRing;
void return_ring(TransferRing* ring, int device);

enum TransferStatus { TRANSFER_DONE = 0, TRANSFER_DECLINED = 1, TRANSFER_FAILED = 2 };

// Copies all planes, in order, and returns when the host (device) arrays are
// complete.  Kernels run on `s`; *err holds the HIP error when FAILED.
// DECLINED: nothing was done (the arrays are too small for it to pay, or no
// pinned memory or thread could be had); the caller copies plane by plane.
int planes_to_host(TransferRing** ring, const TransferGrid& g, const NodePlane* planes, int count, hipStream_t s,
                   hipError_t* err);
int planes_to_device(TransferRing** ring, const TransferGrid& g, const NodePlane* planes, int count, hipStream_t s,
                     hipError_t* err);

}  // namespace hlbm
