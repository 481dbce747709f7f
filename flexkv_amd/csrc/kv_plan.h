// kv_plan.h - how a transfer's work is cut and how much of the device it
// takes: pure functions of sizes and counts, header-only and free of HIP, so a
// CPU-only test can hold them to what they promise.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace fkv_detail {

// Workgroups that move a zero-copy transfer fastest where the host link bounds
// it (kv_zero_copy_kernel has the sweep behind them).
constexpr int kZeroCopyReaders = 14;    // host to device
constexpr int kZeroCopyWriters = 32;    // device to host

// Readers of a call that starts while a zero-copy transfer writes to host memory
// on the same device.  Beside 32 writers 14 readers fall behind; 28, which alone
// are 5% slower than 14, keep pace.  MI355X, GB/s of both directions with 14 / 28
// readers (and in tiled kernels of 28 writers and 56 readers):
//   begun together, 1-2 GiB each        81-84 / 85-91  (88)
//   each direction call after call:
//     4 MiB     65 / 71  (59)       64 MiB    73 / 77  (65)
//     16 MiB    73 / 86  (64)       320 MiB   74 / 69  (67)
//     32 MiB    73 / 88  (71)       1 GiB     74 / 69  (67)
// Calls that began together run at 45 + 45 as long as they last; a long one that
// begins in the middle of the other way's gets 33 + 33, or 25 + 48 with 14
// readers.  48-56 writers and readers: 89-93 together, 69-71 from 320 MiB.
constexpr int kZeroCopyReadersBeside = 28;

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
// kernel a compute unit holds; `writing`: a zero-copy transfer to host memory is
// in flight on the device.  A host cache in host memory takes the counts above,
// or all that more than kZeroCopySpreadCus compute units hold when the caller
// names them.  One in device memory has no link to wait for: it takes every
// workgroup the compute units hold.
inline int zero_copy_workgroups(bool h2d, bool host_memory, int transfer_cus, int num_cus,
                                int occupancy, bool writing) {
  const int cus = transfer_cus <= 0 ? num_cus : std::min(transfer_cus, num_cus);
  const int held = cus * occupancy;
  if (!host_memory || transfer_cus > kZeroCopySpreadCus) return held;
  const int readers = writing ? kZeroCopyReadersBeside : kZeroCopyReaders;
  return std::min(h2d ? readers : kZeroCopyWriters, held);
}

// What one staging launch moves: blocks [b, b + nb) of the piece, items (layer,
// K|V) [item, item + items), and of each of their chunks the 16-byte vectors
// [off, off + vec).  `packed`: where in the staging buffer, in vectors.
struct StagingPart {
  int b, nb;
  int64_t item, items, off, vec, packed;
};

// Cuts a staging gather / scatter of `nb` blocks of `items` chunks of `chunk_vec`
// vectors into launches of at most `max_vec` vectors, each contiguous in the
// staging buffer (block -> item -> chunk or, `layer_major`, item -> block ->
// chunk): one, or whole blocks at a time, or one item at a time over as many
// blocks as are contiguous there, or parts of one chunk.  Ends at the first
// launch that returns an error, and returns it.
template <class Launch>
int staging_launches(int nb, int64_t items, int64_t chunk_vec, bool layer_major, int64_t max_vec,
                     Launch&& launch) {
  const int64_t block_vec = items * chunk_vec;
  int rc = 0;
  if (nb * block_vec <= max_vec) return launch(StagingPart{0, nb, 0, items, 0, chunk_vec, 0});
  if (!layer_major && block_vec <= max_vec) {
    const int step = static_cast<int>(max_vec / block_vec);
    for (int b = 0; b < nb && !rc; b += step)
      rc = launch(StagingPart{b, std::min(step, nb - b), 0, items, 0, chunk_vec, b * block_vec});
    return rc;
  }
  const int64_t part = std::min(chunk_vec, max_vec);
  const int step =
      layer_major && part == chunk_vec ? static_cast<int>(std::min<int64_t>(nb, max_vec / part)) : 1;
  for (int64_t i = 0; i < items && !rc; ++i)
    for (int b = 0; b < nb && !rc; b += step)
      for (int64_t off = 0; off < chunk_vec && !rc; off += part)
        rc = launch(StagingPart{b, std::min(step, nb - b), i, 1, off, std::min(part, chunk_vec - off),
                                (layer_major ? i * nb + b : b * items + i) * chunk_vec + off});
  return rc;
}

// What one zero-copy launch moves: blocks [b, b + nb) of the call, layers
// [layer, layer + layers) of the window, and of each of their chunks the vectors
// [off, off + vec).  Its num_vec vectors are cut into `groups`, groups_per_wg
// consecutive ones a workgroup, whose run touches at most run_blocks blocks.
struct ZeroCopyPart {
  int b, nb, layer, layers;
  int64_t off, vec, num_vec, groups, groups_per_wg, run_blocks;
  bool last;   // of the transfer's launches
  int64_t workgroups() const { return (groups + groups_per_wg - 1) / groups_per_wg; }
};

struct ZeroCopyLimits {
  int64_t max_vec;       // vectors of a launch
  int64_t max_part;      // vectors of a launch's chunk parts
  int64_t run_blocks;    // blocks of a workgroup's run
  int layers;            // layers of a launch
};

// Cuts a zero-copy transfer of `num_blocks` blocks and `nl` layers of `kv` chunks
// of `chunk_vec` vectors into launches of groups of `group_vec` vectors over at
// most `grid` workgroups of `waves` wavefronts: one launch, but for layers, parts
// of chunks and blocks beyond the limits.  Ends at the first launch that returns
// an error, and returns it.
template <class Launch>
int zero_copy_launches(int num_blocks, int nl, int kv, int64_t chunk_vec, int64_t group_vec,
                       int waves, int grid, const ZeroCopyLimits& lim, Launch&& launch) {
  const int64_t part_max = std::min(chunk_vec, lim.max_part);
  const int layers_max = static_cast<int>(std::min<int64_t>(
      {nl, lim.layers, std::max<int64_t>(1, lim.max_vec / (kv * part_max))}));
  for (int layer = 0; layer < nl; layer += layers_max)
    for (int64_t off = 0; off < chunk_vec; off += part_max) {
      ZeroCopyPart p;
      p.layer = layer;
      p.layers = std::min(layers_max, nl - layer);
      p.off = off;
      p.vec = std::min(part_max, chunk_vec - off);
      const int64_t block_vec = static_cast<int64_t>(p.layers) * kv * p.vec;
      for (p.b = 0; p.b < num_blocks; p.b += p.nb) {
        int64_t nb = std::min<int64_t>(num_blocks - p.b, lim.max_vec / block_vec);
        for (;; nb = (nb + 1) / 2) {
          p.groups = (nb * block_vec + group_vec - 1) / group_vec;
          const int64_t wgs = std::min<int64_t>(std::max(1, grid), (p.groups + waves - 1) / waves);
          p.groups_per_wg = (p.groups + wgs - 1) / wgs;
          p.run_blocks = std::min(nb, p.groups_per_wg * group_vec / block_vec + 2);
          if (p.run_blocks <= lim.run_blocks || nb == 1) break;
        }
        p.nb = static_cast<int>(nb);
        p.num_vec = nb * block_vec;
        p.last = p.b + p.nb == num_blocks && off + p.vec == chunk_vec && layer + p.layers == nl;
        const int rc = launch(static_cast<const ZeroCopyPart&>(p));
        if (rc) return rc;
      }
    }
  return 0;
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
