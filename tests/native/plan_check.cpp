// CPU-only check of how transfers are cut and sized
// (flexkv_amd/csrc/kv_plan.h): no HIP, no device.  Prints one line per case
// and exits non-zero when one fails.
#include "kv_plan.h"

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <vector>

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
        all = all && zero_copy_workgroups(h2d, false, -1, cus, occ, occ == 4) == cus * occ;
        all = all && zero_copy_workgroups(h2d, false, 0, cus, occ, occ == 4) == cus * occ;
        for (int bound : {1, 2, 8, 31, 256, 1000}) {
          const int n = zero_copy_workgroups(h2d, false, bound, cus, occ, occ == 4);
          bounded = bounded && n == (bound < cus ? bound : cus) * occ;
        }
        const int most = h2d ? 14 : 32;
        const int n = zero_copy_workgroups(h2d, true, -1, cus, occ, false);
        host = host && n == (most < cus * occ ? most : cus * occ);
      }
  check(all, "a host cache in device memory takes every workgroup the device holds");
  check(bounded, "and those of the caller's compute units when bounded");
  check(host, "one in host memory takes what fills the link");
}

// Every vector of every chunk is moved once, from the place the kernel computes
// for it to the place the staging layout gives it.
void staging_launches_cover_the_piece() {
  bool sizes = true, places = true, once = true, stops = true;
  int shapes[4] = {0, 0, 0, 0};   // one launch, whole blocks, items, parts of chunks
  for (int nb : {1, 2, 3, 7})
    for (int64_t items : {1, 2, 3, 6})
      for (int64_t cv : {1, 3, 64, 100})
        for (bool layer_major : {false, true})
          for (int64_t max_vec : {1, 2, 7, 64, 99, 100, 101, 250, 650, 5000}) {
            std::vector<int> seen(nb * items * cv);
            int calls = 0;
            auto launch = [&](const StagingPart& p) {
              ++calls;
              const int64_t n = p.nb * p.items * p.vec;
              sizes = sizes && n >= 1 && n <= max_vec;
              shapes[p.vec < cv ? 3 : p.items < items ? 2 : p.nb < nb ? 1 : 0]++;
              for (int64_t v = 0; v < n; ++v) {
                // kv_pack_kernel's walk
                const int64_t c = v / p.vec, inner = layer_major ? p.nb : p.items;
                const int64_t outer = c / inner, rest = c % inner;
                const int64_t b = p.b + (layer_major ? rest : outer);
                const int64_t item = p.item + (layer_major ? outer : rest);
                const int64_t at = p.off + v % p.vec;
                if (b >= nb || item >= items || at >= cv) {
                  places = false;
                  continue;
                }
                const int64_t want = (layer_major ? item * nb + b : b * items + item) * cv + at;
                places = places && p.packed + v == want;
                ++seen[want];
              }
              return 0;
            };
            const int rc = staging_launches(nb, items, cv, layer_major, max_vec, launch);
            once = once && rc == 0;
            for (int n : seen) once = once && n == 1;
            for (int fail_at : {1, calls}) {
              int k = 0;
              const int r = staging_launches(nb, items, cv, layer_major, max_vec,
                                             [&](const StagingPart&) { return ++k == fail_at ? 7 : 0; });
              stops = stops && r == 7 && k == fail_at;
            }
          }
  check(sizes, "staging launches stay within their limit");
  check(places, "each vector lies where the staging layout has it");
  check(once, "each vector of a piece moves once");
  check(stops, "the first staging launch that fails is the last");
  check(shapes[0] && shapes[1] && shapes[2] && shapes[3], "by one launch, blocks, items and parts");
}

void zero_copy_launches_cover_the_transfer() {
  bool sizes = true, once = true, runs = true, last = true, stops = true;
  int shapes[4] = {0, 0, 0, 0};   // one launch, runs of blocks, layers, parts of chunks
  for (int nb : {1, 2, 5, 40})
    for (int nl : {1, 3, 5})
      for (int kv : {1, 2})
        for (int64_t cv : {1, 5, 64, 100})
          for (int64_t max_vec : {64, 130, 1000, 100000})
            for (int64_t max_part : {16, 32, 1000})
              for (int64_t run_blocks : {3, 9, 1000})
                for (int layers : {2, 128})
                  for (int grid : {1, 4, 14}) {
                    const ZeroCopyLimits lim{max_vec, max_part, run_blocks, layers};
                    if (kv * std::min(cv, max_part) > max_vec) continue;
                    const int64_t group_vec = 8;
                    const int waves = 4;
                    std::vector<int> seen(nb * nl * kv * cv);
                    int calls = 0, ends = 0;
                    bool end_seen = false;
                    auto launch = [&](const ZeroCopyPart& p) {
                      ++calls;
                      shapes[p.vec < cv ? 3 : p.layers < nl ? 2 : p.nb < nb ? 1 : 0]++;
                      const int64_t row = static_cast<int64_t>(p.layers) * kv * p.vec;
                      sizes = sizes && p.nb >= 1 && p.num_vec == p.nb * row && p.num_vec <= max_vec &&
                              p.layers <= layers && p.vec <= max_part &&
                              p.workgroups() <= std::max(1, grid) &&
                              p.groups * group_vec >= p.num_vec;
                      runs = runs && (p.run_blocks <= run_blocks || p.nb == 1);
                      for (int64_t w = 0; w < p.workgroups(); ++w) {
                        // the blocks of the workgroup's run, as kv_zero_copy_kernel finds them
                        const int64_t g0 = w * p.groups_per_wg;
                        const int64_t g1 = std::min(g0 + p.groups_per_wg, p.groups);
                        const int64_t b0 = g0 * group_vec / row;
                        const int64_t b1 = (std::min(g1 * group_vec, p.num_vec) - 1) / row;
                        runs = runs && g0 < g1 && b1 - b0 + 1 <= p.run_blocks;
                      }
                      for (int64_t v = 0; v < p.num_vec; ++v) {
                        const int64_t c = v / p.vec, b = c / (p.layers * kv), item = c % (p.layers * kv);
                        const int64_t layer = p.layer + item / kv, k = item % kv;
                        ++seen[(((p.b + b) * nl + layer) * kv + k) * cv + p.off + v % p.vec];
                      }
                      last = last && !end_seen;
                      end_seen = p.last;
                      ends += p.last;
                      return 0;
                    };
                    const int rc = zero_copy_launches(nb, nl, kv, cv, group_vec, waves, grid, lim, launch);
                    last = last && ends == 1 && end_seen;
                    once = once && rc == 0;
                    for (int n : seen) once = once && n == 1;
                    int k = 0;
                    const int r = zero_copy_launches(nb, nl, kv, cv, group_vec, waves, grid, lim,
                                                     [&](const ZeroCopyPart&) { return ++k == calls ? 7 : 0; });
                    stops = stops && r == 7 && k == calls;
                  }
  check(sizes, "zero-copy launches stay within their limits");
  check(runs, "a workgroup's run holds the blocks its memory has room for");
  check(once, "each vector of a transfer moves once");
  check(last, "the last launch, and no other, is marked");
  check(stops, "a zero-copy launch that fails is the last");
  check(shapes[0] && shapes[1] && shapes[2] && shapes[3], "by one launch, blocks, layers and parts");
}

void transfer_cus_bounds_and_spreads() {
  bool bounds = true, spreads = true;
  for (bool h2d : {false, true})
    for (int occ : {4, 8}) {
      const int most = h2d ? 14 : 32;
      for (int cus = 1; cus <= 8; ++cus) {
        const int n = zero_copy_workgroups(h2d, true, cus, 256, occ, false);
        bounds = bounds && n == (most < cus * occ ? most : cus * occ);
      }
      for (int cus : {9, 32, 64, 256, 4096})
        spreads = spreads && zero_copy_workgroups(h2d, true, cus, 256, occ, false) ==
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

void readers_keep_pace_with_writers() {
  bool beside = true, writers = true;
  for (int occ : {1, 4, 8})
    for (int cus : {-1, 1, 2, 4, 8}) {
      const int held = (cus < 0 ? 256 : cus) * occ;
      beside = beside && zero_copy_workgroups(true, true, cus, 256, occ, true) == std::min(28, held);
      writers = writers && zero_copy_workgroups(false, true, cus, 256, occ, true) == std::min(32, held);
    }
  check(beside, "readers that start beside writers are 28, within the caller's compute units");
  check(writers, "writers are as many beside one another");
}

}  // namespace

int main() {
  readers_keep_pace_with_writers();
  null_stream_waits_cover_what_they_wait_for();
  device_memory_takes_the_chip();
  staging_launches_cover_the_piece();
  zero_copy_launches_cover_the_transfer();
  transfer_cus_bounds_and_spreads();
  return failures ? 1 : 0;
}
