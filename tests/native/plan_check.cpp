// CPU-only check of how transfers are cut and sized
// (flexkv_amd/csrc/kv_plan.h): no HIP, no device.  Prints one line per case
// and exits non-zero when one fails.
#include "kv_plan.h"

#include <cstdio>

using namespace fkv_detail;

namespace {

int failures = 0;

void check(bool ok, const char* what) {
  std::printf("%s: %s\n", ok ? "ok" : "FAIL", what);
  if (!ok) ++failures;
}

void device_memory_takes_the_chip() {
  bool all = true, bounded = true, host = true;
  for (int cus : {1, 32, 256})
    for (int occ : {1, 4, 8})
      for (bool h2d : {false, true}) {
        all = all && zero_copy_workgroups(h2d, false, -1, cus, occ) == cus * occ;
        all = all && zero_copy_workgroups(h2d, false, 0, cus, occ) == cus * occ;
        for (int bound : {1, 2, 8, 31, 256, 1000}) {
          const int n = zero_copy_workgroups(h2d, false, bound, cus, occ);
          bounded = bounded && n == (bound < cus ? bound : cus) * occ;
        }
        const int most = h2d ? 14 : 32;
        const int n = zero_copy_workgroups(h2d, true, -1, cus, occ);
        host = host && n == (most < cus * occ ? most : cus * occ);
      }
  check(all, "a host cache in device memory takes every workgroup the device holds");
  check(bounded, "and those of the caller's compute units when bounded");
  check(host, "one in host memory takes what fills the link");
}

void transfer_cus_bounds_and_spreads() {
  bool bounds = true, spreads = true;
  for (bool h2d : {false, true})
    for (int occ : {4, 8}) {
      const int most = h2d ? 14 : 32;
      for (int cus = 1; cus <= 8; ++cus) {
        const int n = zero_copy_workgroups(h2d, true, cus, 256, occ);
        bounds = bounds && n == (most < cus * occ ? most : cus * occ);
      }
      for (int cus : {9, 32, 64, 256, 4096})
        spreads = spreads && zero_copy_workgroups(h2d, true, cus, 256, occ) ==
                                 (cus < 256 ? cus : 256) * occ;
    }
  check(bounds, "up to 8 compute units bound a transfer over the link");
  check(spreads, "more of them are all filled");
}

void null_stream_waits_cover_what_they_wait_for() {
  const std::vector<int> done = {1, 1, 1, 2, 3, 3};   // groups of one launch share an event
  bool ordered = true, alone = true;
  const int shared_end[] = {3, 3, 3, 4, 6, 6};
  for (int g = 0; g < 6; ++g)
    for (int queued = g + 1; queued <= 6; ++queued) {
      ordered = ordered && null_wait_covers(done, g, queued, true) == queued;
      alone = alone && null_wait_covers(done, g, queued, false) == shared_end[g];
    }
  check(ordered, "a wait behind a blocking stream covers every group queued on it");
  check(alone, "one behind any other stream covers the groups of its own event");
}

}  // namespace

int main() {
  null_stream_waits_cover_what_they_wait_for();
  device_memory_takes_the_chip();
  transfer_cus_bounds_and_spreads();
  return failures ? 1 : 0;
}
