// kv_plan.h - how a transfer's work is cut and how much of the device it
// takes: pure functions of sizes and counts, header-only and free of HIP, so a
// CPU-only test can hold them to what they promise.
#pragma once

#include <algorithm>
#include <vector>

namespace fkv_detail {

// Workgroups that move a zero-copy transfer fastest where the host link bounds
// it (kv_zero_copy_kernel has the sweep behind them).
constexpr int kZeroCopyReaders = 14;    // host to device
constexpr int kZeroCopyWriters = 32;    // device to host

// Compute units up to which a caller's number bounds the grid over host
// memory; a larger one spreads it.  Eight (the workers' default) hold more
// than the fastest counts of either direction.  All the workgroups of more are
// a little slower, gentler to compute that runs already and harder on compute
// that starts after: 2 GiB on MI355X beside bf16 GEMMs started first, then
// queued after it, 14 / 256 readers slow those 1.44 / 1.10 and 1.39 / 2.05
// times at 57.4 / 54.9 GB/s, 32 / 256 writers 1.48 / 1.09 and 1.45 / 2.04
// times at 56.5 / 56.8 GB/s.
constexpr int kZeroCopySpreadCus = 8;

// Workgroups of a zero-copy transfer.  `transfer_cus`: compute units the
// caller lets it occupy, <= 0 for no bound; `occupancy`: workgroups of the
// kernel a compute unit holds.  A host cache in host memory takes the counts
// above, or all that more than kZeroCopySpreadCus compute units hold when the
// caller names them.  One in device memory has no link to wait for: it takes
// every workgroup the compute units hold.
inline int zero_copy_workgroups(bool h2d, bool host_memory, int transfer_cus, int num_cus,
                                int occupancy) {
  const int cus = transfer_cus <= 0 ? num_cus : std::min(transfer_cus, num_cus);
  const int held = cus * occupancy;
  return !host_memory || transfer_cus > kZeroCopySpreadCus
             ? held
             : std::min(h2d ? kZeroCopyReaders : kZeroCopyWriters, held);
}

// One past the last layer group that a legacy null stream's wait on `group`'s
// event also waits for: with `ordered` (the stream that records the events is
// one the null stream waits for by itself) every group queued so far, else only
// the groups after `group` that share its event.
template <class Event>
int null_wait_covers(const std::vector<Event>& done, int group, int queued, bool ordered) {
  if (ordered) return queued;
  int end = group + 1;
  while (end < static_cast<int>(done.size()) && done[end] == done[group]) ++end;
  return end;
}

}  // namespace fkv_detail
