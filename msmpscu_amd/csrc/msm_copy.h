// msm_copy.h -- copies from device memory to the caller's pageable host arrays, large ones and small
// ones in several parts through a small ring of pinned memory per GPU.
//
// The runtime's own copy into pageable memory runs on one thread, whose copying and page faults take
// longer than the DMA once a transfer is large.  There kCopySlots host threads take the transfer's
// chunks in turn: each copies a chunk over PCIe into its own pinned slot and from there to the
// caller's array, so that DMA, page faults and memory copies run together.  A small block in several
// parts goes through one slot on the calling thread, one copy instead of one a part.  Ring / plain
// copies of the same block, us, with everything else of the call:
//   five per-atom arrays   0.2 MB 51 / 86    0.4 MB 57 / 95    0.9 MB 109 / 104   3.1 MB 251 / 228
//                          5.4 MB 328 / 434  14 MB 563 / 979   102 MB 3,867 / 9,305
//   forces                 0.4 MB 52 / 41    1.3 MB 123 / 115  3.3 MB 247 / 255   10 MB 442 / 717
// To the device the plain copy is the faster one at every size (one vector of 0.4 MB 45 / 37, 1.3 MB
// 119 / 83, 3.3 MB 244 / 149, 25 MB 925 / 724).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace msm {

constexpr int kCopySlots = 8;
constexpr size_t kCopySlotBytes = size_t(1) << 20;
constexpr size_t kRingFrom = size_t(4) << 20;    // through the ring beyond this
constexpr size_t kOneSlot = size_t(512) << 10;  // several parts: through one slot up to this
static_assert(kOneSlot <= kCopySlotBytes, "one slot");

// A GPU's contexts share its ring, one transfer at a time.  The first copy that takes it pins it (0.13 ms), and
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

}  // namespace msm
