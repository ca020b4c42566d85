// Device results into the caller's host memory: a bounded, process-wide set of
// pinned staging slots and the loop that fills one while host threads empty
// the other.  The device side of a readback is a kernel that forms the values
// in the caller's layout and writes them straight into the pinned slot.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>

#include "eqd_device.h"

namespace eqd {

// One slot's size, slots per lease (one is filled while the other is
// emptied) and leases alive at once: at most 64 MiB of pinned memory in the
// process.  8 MiB keeps four 2 MiB host pages in flight per emptied slot;
// the first touch of a slot costs about 0.35 ms per MiB, once.
constexpr size_t kStageSlot = (size_t)8 << 20;
constexpr int kStageSlots = 2, kStageLeases = 4;

// Users of the staging slots (handles, start-up calls): the slots, and the
// threads that empty them, are given back when the last user goes.
void stage_retain();
void stage_release();

// `bytes` bytes to host memory at out in slot-sized pieces: fill(slot, first,
// count, stream) enqueues the work that leaves bytes [first, first + count) in
// the pinned slot.  Pieces start at multiples of `unit` bytes.  Returns when
// all of out is written.
typedef std::function<hipError_t(void *slot, size_t first, size_t count, hipStream_t s)> StageFill;
hipError_t stage_out(void *out, size_t bytes, size_t unit, hipStream_t s, const StageFill &fill);

// The same for values that already lie in device memory in the caller's layout.
hipError_t stage_copy(void *out, const void *dev, size_t bytes, hipStream_t s);

// Pack kernels: values of `count` nodes (pairs) from `first` on, in the
// reference's layout (velArr / dispArr: 3 per node; fric: 100 per pair).
hipError_t launch_pack_nodes(const NodeState &N, const FaultState &F, bool vel, int64_t first, int64_t count,
                             double *out, hipStream_t s);
hipError_t launch_pack_fric(const FaultState &F, int64_t first, int64_t count, double *out, hipStream_t s);

}  // namespace eqd
