// msm_copy.h -- copies between device memory and the caller's pageable host arrays through a small
// ring of pinned memory per GPU.
//
// The runtime's own copy of pageable memory ran at 3-6 GB/s here (it pins or bounces the caller's
// pages on one thread, and fresh pages fault one after another).  Here up to kCopySlots host threads
// take the transfer's chunks in turn: each copies a chunk over PCIe into its own pinned slot and from
// there to the caller's array, so the DMA of one chunk, the page faults and the memory copies of
// the others run together.  Transfers up to half a megabyte run on the calling thread alone.
// Measured, all per-atom arrays out: 136k atoms (14 MB) 4.4 -> 1.1 ms, 1.02M atoms (106 MB)
// 18 -> 3.7 ms (28 GB/s); one 54k-atom vector (1.3 MB) 0.11 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace msm {

constexpr int kCopySlots = 8;
constexpr size_t kCopySlotBytes = size_t(1) << 20;

// A GPU's contexts share its ring, one transfer at a time.  The first large copy pins it (0.13 ms), and
// it is given back with the last context; where it cannot be pinned, copies are plain ones.
void copy_ring_acquire(int device);
void copy_ring_release(int device);

// One piece of a device block and its place on the host.
struct CopyPart {
    size_t offset, bytes;
    void* host;
};

// base .. base + total (the parts in order of their offsets, without gaps) into the parts' host
// arrays, after everything queued on the stream; returns with the data there.
hipError_t copy_to_host(int device, const void* base, size_t total, const CopyPart* parts,
                        int nparts, hipStream_t stream);
// total bytes of host memory to dst; returns with the transfer done.
hipError_t copy_to_device(int device, void* dst, const void* host, size_t total,
                          hipStream_t stream);

}  // namespace msm
