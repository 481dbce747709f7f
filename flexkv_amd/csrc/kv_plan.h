// kv_plan.h - how a transfer's work is cut and how much of the device it
// takes: pure functions of sizes and counts, header-only and free of HIP, so a
// CPU-only test can hold them to what they promise.
#pragma once

#include <algorithm>

namespace fkv_detail {

// Workgroups that move a zero-copy transfer fastest where the host link bounds
// it (kv_zero_copy_kernel has the sweep behind them).
constexpr int kZeroCopyReaders = 14;    // host to device
constexpr int kZeroCopyWriters = 32;    // device to host

// Workgroups of a zero-copy transfer.  `transfer_cus`: compute units the
// caller lets it occupy, <= 0 for no bound; `occupancy`: workgroups of the
// kernel a compute unit holds.  A host cache in host memory takes the counts
// above.  One in device memory has no link to wait for: it takes every workgroup
// the compute units hold.
inline int zero_copy_workgroups(bool h2d, bool host_memory, int transfer_cus, int num_cus,
                                int occupancy) {
  const int cus = transfer_cus <= 0 ? num_cus : std::min(transfer_cus, num_cus);
  const int held = cus * occupancy;
  return host_memory ? std::min(h2d ? kZeroCopyReaders : kZeroCopyWriters, held) : held;
}

}  // namespace fkv_detail
