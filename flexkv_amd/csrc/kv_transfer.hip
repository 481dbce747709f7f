// kv_transfer.hip - GPU<->CPU KV-block transfer for MI355X (gfx950).
//
// The unit is the "chunk": a (layer, K|V, block) piece of the KV cache,
// `chunk_size` contiguous bytes on both sides (csrc/transfer.cu:39-53 gives
// the reference addressing).
//   * Zero-copy transfers: kv_zero_copy_kernel (kv_small_copy_kernel for the
//     smallest calls) moves chunks between the GPU cache and the pinned host
//     cache itself; its 16-byte loads or stores travel over PCIe.
//   * Copy-engine transfers and device gathers / scatters: a staging kernel
//     moves chunks between the GPU cache and a contiguous HBM buffer laid out
//     [block][layer][K|V][chunk]; for copy-engine transfers the SDMA engines
//     (queued through HSA) then move maximal contiguous host runs between
//     that buffer and the host cache.
//
// Staging work decomposition (kv_pack_kernel): the staging buffer's bytes are
// one contiguous sequence, cut into groups of kU rows (64 lanes x 16 B = 1 KiB)
// with a wavefront each, whatever the chunk size.
//
// This file holds the kernels, the transfer paths that launch them and the
// transfer entry points of the C ABI; kv_host.cpp holds validation, id staging
// and the host-only entry points, kv_sdma.cpp the copy engines.

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <optional>
#include <string>
#include <thread>
#include <vector>

#include "kv_internal.h"
#include "kv_plan.h"

using namespace fkv_detail;

namespace {

// Cache hints: loads are non-temporal everywhere, and so are stores into HBM
// (stores into host memory: store_system, kv_small_copy_kernel).
constexpr int kThreads = 256;               // 4 wavefronts of 64 lanes
constexpr int kWaves = kThreads / 64;
// Launches of at most this many blocks carry their (gpu_id, cpu_id) pairs in
// the kernel arguments, so no workgroup reads them over PCIe first (one host
// round trip less per launch).
constexpr int kInlineIdsZeroCopy = 96;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
// Every address the kernel touches is global memory (HBM or mapped pinned
// host memory); saying so lets the compiler emit global_* instead of flat_*.
typedef __attribute__((address_space(1))) u32x4 gvec;

// 16 bytes written through every cache (system scope).  The zero-copy kernel's
// stores into host memory go this way: left to the caches they arrive in the
// order of evictions, and a 16 MiB device-to-host call took 360 us instead of
// 317 (16 workgroups).  In assembly, as no builtin stores 16 bytes at system
// scope; the s_nop keeps the two wait states a wide store needs before its
// data registers are written again, which the compiler cannot see it needs.
__device__ inline void store_system(char* p, u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
}

// The same with the non-temporal hint, for HBM.
__device__ inline void store_through(char* p, u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
}

// n / d for n < 2^31 as a multiplication (Granlund and Montgomery, "Division
// by Invariant Integers using Multiplication", 1994): with 2^(l-1) < d <= 2^l,
// mul = ceil(2^(31+l) / d) < 2^32 and n / d = floor(n * mul / 2^(31+l)).
struct Divider {
  uint32_t d = 1, mul = 0, shift = 0;
  explicit Divider(uint32_t by = 1) : d(by) {
    int l = 0;
    while ((uint64_t(1) << l) < by) ++l;
    shift = static_cast<uint32_t>(31 + l);
    mul = static_cast<uint32_t>(((static_cast<unsigned __int128>(1) << shift) + by - 1) / by);
  }
  __device__ uint32_t div(uint32_t n) const {
    return static_cast<uint32_t>((static_cast<uint64_t>(n) * mul) >> shift);
  }
};

// The staging gather / scatter.  The packed (staging) side is contiguous: the
// launch's chunks in order, block -> layer -> K|V or layer -> K|V -> block.
// Its 16-byte vectors are cut into groups of kU rows of 64 and wavefront w of
// workgroup b moves group 4b + w (b in column order, launch_pack): no tile, no
// LDS, no barrier, and every wavefront moves a full group.  Lane j first
// resolves the address of the group's j-th chunk (a group touches at most 64,
// pack_fits), so ids and layer pointers cost one round of loads a group
// whatever the chunk size; each row then picks the chunk of each lane's vector
// out of those registers (ds_bpermute), so rows that cross chunks (sizes that
// are not whole KiB, or under one) leave no lane idle.  The scattered address
// is used in one of the two walks only, so nothing but the loaded data is held
// between them.
//
// HBM bounds the large launches and the launch the small ones.  Measured on
// MI355X, us a gather / scatter call, against a kernel per chunk shape (tiled
// groups, 2-5 bases a group, a row-by-row one) with the ids staged by a launch
// of their own: 2 GiB of 32 KiB chunks 727 / 808 -> 706 / 774, 1 GiB of 4 KiB
// 383 / 440 -> 379 / 407, 1 GiB of 2 KiB 462 / 462 -> 381 / 406, 47 MiB of 2
// KiB 57.2 / 57.0 -> 38.0 / 40.1, 64 MiB of 512 B 79.4 / 78.7 -> 47.2 / 46.3,
// 1 MiB of 32 KiB 18.8 / 20.6 -> 15.2 / 14.6.
constexpr int kPackInlineIds = 256;
// vectors of a launch: Divider takes numbers below 2^31, the last group's
// positions beyond the end included
constexpr int64_t kPackMaxVec = int64_t(1) << 30;

struct PackArgs {
  const int64_t* gids;       // device memory: gpu ids by launch block; null: inline_ids
  const uint64_t* ptrs;      // device memory: layer pointers; null: layer_ptr
  char* packed;              // staging address of the launch's first vector
  int64_t gpu_kv_stride;
  int64_t gpu_block_stride;
  Divider chunk;             // by the vectors of a chunk
  Divider inner;             // by the chunks of a block, or of a (layer, K|V) when layer_major
  uint32_t layer_major;
  uint32_t kv_dim;
  uint32_t num_vec;          // vectors of the launch
  uint32_t num_chunks;
  uint32_t num_groups;
  Divider columns;           // runs of column_wgs workgroups' groups, taken in turn
  uint32_t column_wgs;
  int32_t ptrs_per_layer;    // 1: layer_ptr[l] + k*gpu_kv_stride; kv: layer_ptr[l*kv + k]
  uint64_t layer_ptr[kMaxLayersPerLaunch];
  int64_t inline_ids[kPackInlineIds];
};

// Whether a group of `rows` rows touches at most 64 chunks of `chunk_vec`
// vectors, wherever it starts.
constexpr bool pack_fits(int rows, int64_t chunk_vec) {
  const int64_t vec = int64_t(rows) * 64;
  return (vec % chunk_vec == 0 ? vec / chunk_vec : (vec - 2) / chunk_vec + 2) <= 64;
}

// kRows: chunks are whole rows, so a row has one chunk and its address is
// wave-uniform (scalar registers).  With per-lane addresses a 1 GiB scatter of
// 72 KiB chunks took 404 us instead of 388.
// kThrough: stores bypass the caches, for scatters in column order.  Measured
// on MI355X, us against non-temporal stores: 2 GiB of 32 KiB chunks 795 -> 774,
// 1 GiB of 72 / 4 / 2 KiB 382 -> 368, 415 -> 407, 414 -> 406; a 2 GiB gather
// would take 896 instead of 707 and smaller scatters gain nothing.
template <bool kH2D, int kU, bool kRows, bool kThrough>
__global__ __launch_bounds__(kThreads) void kv_pack_kernel(PackArgs a) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t q = a.columns.div(blockIdx.x);
  const uint32_t wg = (blockIdx.x - q * a.columns.d) * a.column_wgs + q;
  const uint32_t g = wg * kWaves + wave;
  if (g >= a.num_groups) return;
  const uint32_t v0 = g * (kU * 64);
  const uint32_t c0 = a.chunk.div(v0);
  const uint32_t r0 = v0 - c0 * a.chunk.d;    // the group's start within chunk c0
  int64_t base;                               // lane j: the address chunk c0 + j gives position 0
  {
    const uint32_t c = min(c0 + lane, a.num_chunks - 1);
    const uint32_t outer = a.inner.div(c);
    const uint32_t rest = c - outer * a.inner.d;
    const uint32_t b = a.layer_major ? rest : outer;
    const uint32_t item = a.layer_major ? outer : rest;
    const uint32_t l = a.kv_dim == 1 ? item : item >> 1;
    const uint32_t k = item - l * a.kv_dim;
    const uint32_t pi = a.ptrs_per_layer == 1 ? l : item;
    const int64_t gid = a.gids ? a.gids[b] : a.inline_ids[b];
    const uint64_t ptr = a.ptrs ? a.ptrs[pi] : a.layer_ptr[pi];
    base = static_cast<int64_t>(ptr) + static_cast<int64_t>(k) * a.gpu_kv_stride +
           gid * a.gpu_block_stride +
           (static_cast<int64_t>(r0) - static_cast<int64_t>(lane) * a.chunk.d) * 16;
  }
  const int base_lo = static_cast<int>(base);
  const int base_hi = static_cast<int>(base >> 32);
  char* packed = a.packed + static_cast<int64_t>(v0) * 16;
  const uint32_t n = a.num_vec - v0;          // vectors from the group's start to the end
  u32x4 v[kU];
  if constexpr (kRows) {
    const uint32_t lane_off = lane * 16;
    // the scattered address of row u
    auto scattered = [&](uint32_t u) {
      const uint32_t j = a.chunk.div(r0 + u * 64);
      const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(base_lo, j));
      const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(base_hi, j));
      return reinterpret_cast<char*>(((static_cast<uint64_t>(hi) << 32) | lo) + u * 1024);
    };
#pragma unroll
    for (uint32_t u = 0; u < kU; ++u)
      if (u * 64 < n) {
        const char* src = kH2D ? packed + u * 1024 : scattered(u);
        v[u] = __builtin_nontemporal_load((const gvec*)(src + lane_off));
      }
#pragma unroll
    for (uint32_t u = 0; u < kU; ++u)
      if (u * 64 < n) {
        char* dst = (kH2D ? scattered(u) : packed + u * 1024) + lane_off;
        if (kThrough)
          store_through(dst, v[u]);
        else
          __builtin_nontemporal_store(v[u], (gvec*)dst);
      }
  } else {
    // the scattered address of the lane's vector at position i of the group
    auto scattered = [&](uint32_t i) {
      const int j = static_cast<int>(a.chunk.div(r0 + i)) * 4;
      const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(j, base_lo));
      const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(j, base_hi));
      return reinterpret_cast<char*>(((static_cast<uint64_t>(hi) << 32) | lo) +
                                     static_cast<uint64_t>(i) * 16);
    };
    // past the end a lane reloads the last vector and stores nothing
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint32_t i = min(u * 64 + lane, n - 1);
      const char* src = kH2D ? packed + i * 16 : scattered(i);
      v[u] = __builtin_nontemporal_load((const gvec*)src);
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint32_t i = u * 64 + lane;
      char* dst = kH2D ? scattered(min(i, n - 1)) : packed + i * 16;
      if (i < n) {
        if (kThrough)
          store_through(dst, v[u]);
        else
          __builtin_nontemporal_store(v[u], (gvec*)dst);
      }
    }
  }
}

// The zero-copy kernel: the launch's bytes as one sequence of 16-byte
// vectors, block -> layer -> K|V -> offset (host-address order for the
// block-wise host layout), cut into groups of kU rows of 64 vectors.  Each
// workgroup takes a run of consecutive groups, its wavefronts in turn, and
// each lane finds the two addresses of its vector by itself, so rows that
// cross chunks (sizes that are not whole KiB, or under one) leave no lane
// idle and every shape takes the same code.  Two divisions by multiplication
// and three LDS reads a row are nothing beside the link, which gives a
// wavefront a row every 2000 cycles.
//
// The link bounds it, and few loads or stores in flight fill the link.
// Measured on MI355X, us a call (host to device 32 MiB and 1 GiB, device to
// host 16 MiB and 320 MiB):
//   workgroups        8      12      14      16      20      24      32
//   H2D 32 MiB      603.9   603.6   603.1   603.5   616.6   636.1   641
//   H2D 1 GiB       18781   18755   18673   18721   19112   19778
//   D2H 16 MiB      315.6   311.1   312.6   317.3   315.0   312.7   310.1
//   D2H 320 MiB      6083    5921    5954            6079    5967    5910
// so 14 workgroups read (groups of 4 rows).  Writing (8 rows) 12 and 32 are as
// fast alone, but beside a transfer the other way 12 starve: 2 GiB each way at
// once moves 69 GB/s with 12 and 82-84 with 24-32, so 32 write; reading beside
// them takes 28 (kZeroCopyReadersBeside).  A tiled kernel of 28-56 workgroups
// took 326 us for the 16 MiB and 36.0 us for a 1 MiB host-to-device call of
// one layer (here 33.5).
//
// Groups of 8 rows find their addresses once for the loads and again for the
// stores, which leaves 46 registers and 8 wavefronts a SIMD.  Held through 8
// rows they take 80-110 registers and leave 6 or 4: within one compute unit
// 64 MiB device to host then take 1470 us instead of 1215.
//
// kHost: the host cache lies in host memory.  One in device memory (!kHost) has
// no link to wait for: loads in flight bound the launch, so it takes every
// compute unit (zero_copy_workgroups), and stores both ways with the
// non-temporal hint alone.  Measured on MI355X, us a device-to-host /
// host-to-device call, within the host cache's grid and stores -> now: 64 MiB of
// 32 KiB chunks 152 / 341 -> 38.3 / 38.5, 1 GiB 2208 / 5238 -> 433 / 435, 47 MiB
// of 2 KiB chunks 118 / 258 -> 33.5 / 33.8; within 8 compute units 64 MiB 73.3 /
// 72.2, 1 GiB 976 / 950.  12 and 16 rows: 1 GiB 440 / 445 and 440 / 440.
template <bool kH2D, bool kHost>
constexpr int zero_copy_rows() { return kHost && kH2D ? 4 : 8; }
constexpr int kMaxItems = 2 * kMaxLayersPerLaunch;   // (layer, K|V) pairs of a launch
// LDS for block offsets: with the item table, within the 64 KiB of a launch
constexpr int kZeroCopyMaxLds = 56 << 10;
// vectors of a launch: Divider divides numbers below 2^31
constexpr int64_t kZeroCopyMaxVec = (int64_t(1) << 31) - 1;
constexpr int64_t kZeroCopyMaxChunkVec = int64_t(1) << 29;

struct ZeroCopyArgs {
  const int64_t* ids;        // device-visible (gpu_id, cpu_id) pairs (inline_n == 0)
  char* cpu_base;            // host side of launch layer 0, block id 0
  int64_t gpu_kv_stride;
  int64_t gpu_block_stride;
  int64_t cpu_kv_stride;
  int64_t cpu_layer_stride;
  int64_t cpu_block_stride;
  Divider chunk;             // by the vectors of a chunk
  Divider items;             // by the chunks of a block, layers x K|V
  uint32_t kv_dim;
  uint32_t num_vec;          // vectors of the launch
  uint32_t num_groups;
  uint32_t groups_per_wg;
  int32_t ptrs_per_layer;    // 1: layer_ptr[l] + k*gpu_kv_stride; kv: layer_ptr[l*kv + k]
  int32_t inline_n;          // > 0: the launch's pairs are inline_ids, not ids
  int32_t ids_split;         // > 0: ids holds gpu ids, and cpu ids ids_split entries later
  uint64_t layer_ptr[kMaxLayersPerLaunch];
  int64_t inline_ids[2 * kInlineIdsZeroCopy];
};

template <bool kH2D, bool kHost>
__global__ __launch_bounds__(kThreads) void kv_zero_copy_kernel(ZeroCopyArgs a) {
  constexpr int kU = zero_copy_rows<kH2D, kHost>();
  constexpr uint32_t kGroupVec = kU * 64;
  extern __shared__ int64_t s_block[];      // byte offsets (gpu, cpu) of the run's blocks
  __shared__ int64_t s_item[2 * kMaxItems]; // address (gpu), byte offset (cpu) of (layer, K|V)
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t g0 = blockIdx.x * a.groups_per_wg;
  const uint32_t g1 = min(g0 + a.groups_per_wg, a.num_groups);
  // the blocks of the run
  const uint32_t b0 = a.items.div(a.chunk.div(g0 * kGroupVec));
  const uint32_t b1 = a.items.div(a.chunk.div(min(g1 * kGroupVec, a.num_vec) - 1));
  const uint32_t kv = a.kv_dim;
  const uint32_t ppl = static_cast<uint32_t>(a.ptrs_per_layer);
  for (uint32_t i = tid; i < a.items.d; i += kThreads) {
    const uint32_t l = kv == 1 ? i : i >> 1;
    const uint32_t k = i - l * kv;
    s_item[2 * i] = static_cast<int64_t>(a.layer_ptr[l * ppl + k * (ppl - 1)]) +
                    static_cast<int64_t>(k) * a.gpu_kv_stride;
    s_item[2 * i + 1] = static_cast<int64_t>(l) * a.cpu_layer_stride +
                        static_cast<int64_t>(k) * a.cpu_kv_stride;
  }
  for (uint32_t j = tid; j <= b1 - b0; j += kThreads) {
    const uint32_t b = b0 + j;
    int64_t gid, cid;
    if (a.inline_n) {
      gid = a.inline_ids[2 * b];
      cid = a.inline_ids[2 * b + 1];
    } else if (a.ids_split) {
      gid = a.ids[b];
      cid = a.ids[static_cast<uint32_t>(a.ids_split) + b];
    } else {
      gid = a.ids[2 * static_cast<int64_t>(b)];
      cid = a.ids[2 * static_cast<int64_t>(b) + 1];
    }
    s_block[2 * j] = gid * a.gpu_block_stride;
    s_block[2 * j + 1] = cid * a.cpu_block_stride;
  }
  __syncthreads();
  for (uint32_t g = g0 + wave; g < g1; g += kWaves) {
    uint32_t v0 = g * kGroupVec + lane;
    // the two addresses of the lane's vector in row u; past the end it reloads
    // the last vector and stores nothing
    auto locate = [&](int u, char** gpu, char** cpu) {
      const uint32_t v = min(v0 + u * 64, a.num_vec - 1);
      const uint32_t c = a.chunk.div(v);
      const uint32_t b = a.items.div(c);
      const uint32_t item = c - b * a.items.d;
      const int64_t off = static_cast<int64_t>(v - c * a.chunk.d) * 16;
      *gpu = reinterpret_cast<char*>(s_item[2 * item] + s_block[2 * (b - b0)] + off);
      *cpu = a.cpu_base + s_item[2 * item + 1] + s_block[2 * (b - b0) + 1] + off;
    };
    u32x4 v[kU];
    if constexpr (kHost && kH2D) {
      char *gpu[kU], *cpu[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) locate(u, &gpu[u], &cpu[u]);
#pragma unroll
      for (int u = 0; u < kU; ++u) v[u] = __builtin_nontemporal_load((const gvec*)cpu[u]);
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (v0 + u * 64 < a.num_vec) __builtin_nontemporal_store(v[u], (gvec*)gpu[u]);
    } else {
      char *gpu, *cpu;
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        locate(u, &gpu, &cpu);
        v[u] = __builtin_nontemporal_load((const gvec*)(kH2D ? cpu : gpu));
      }
      asm("" : "+v"(v0));   // nothing of the addresses is kept for the stores
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        locate(u, &gpu, &cpu);
        if (v0 + u * 64 < a.num_vec) {
          if (kHost)
            store_system(cpu, v[u]);
          else
            __builtin_nontemporal_store(v[u], (gvec*)(kH2D ? gpu : cpu));
        }
      }
    }
  }
}

// Copies n 64-bit values, `stride` apart in pinned memory, into a device table
// (ids, layer pointers) that every workgroup of a staging launch then reads.
__global__ __launch_bounds__(256) void stage_table_kernel(const int64_t* in, int stride,
                                                          int64_t* out, int n) {
  const int i = blockIdx.x * 256 + static_cast<int>(threadIdx.x);
  if (i < n) out[i] = in[static_cast<int64_t>(i) * stride];
}

// A system-scope acquire in every workgroup.  Launched with a workgroup per
// compute unit (so every XCD's L2 takes part) before a kernel reads memory
// the copy engines wrote outside any HIP stream: no stale line survives it.
__global__ __launch_bounds__(64) void acquire_system_kernel() {
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
}

// Small zero-copy transfers: the host cuts the call's chunks into pieces of
// at most small_piece_rows 1 KiB rows, resolves each piece's two addresses
// and passes them in the kernel arguments, indexed by workgroup.  A
// workgroup's first scalar loads fetch its piece, and its data loads follow
// at once.  The general kernel first walks its ids, layer table and tiling,
// four rounds of dependent loads from the argument segment before the first
// data load; in a kernel trace on MI355X it took 5.3 / 6.1 us (H2D / D2H) for
// one 64 KiB block row, against 3.0 us for a plain 64 KiB copy kernel.
constexpr int kSmallPieces = 128;
// 1 KiB rows per wavefront (a piece is 4 wavefronts' rows).  Measured on
// MI355X through the C-ABI, one block of 64 KiB / 16 blocks (1 MiB), one
// layer: device-to-host 2 / 4 / 8 rows 13.3 / 13.4 / 13.6 us and 34.3 / 30.7
// / 30.9 us; host-to-device 1 / 2 / 4 rows 14.4 / 14.2 / 14.4 us and (1 row:
// too many pieces, general kernel) 35.1 / 35.1 / 36.5 us.
#ifndef FKV_SMALL_U_D2H
#define FKV_SMALL_U_D2H 4
#endif
#ifndef FKV_SMALL_U_H2D
#define FKV_SMALL_U_H2D 2
#endif
// rows per wavefront and rows per piece, by direction
template <bool kH2D>
constexpr int small_rows_per_wave() { return kH2D ? FKV_SMALL_U_H2D : FKV_SMALL_U_D2H; }
template <bool kH2D>
constexpr int small_piece_rows() { return kWaves * small_rows_per_wave<kH2D>(); }
constexpr int64_t kSmallMaxBytes = int64_t(4) << 20;   // bytes moved per call

// Calls of at most this many pieces pass lists of that length: the host writes
// a launch's arguments over PCIe, 2.5 KiB of them for kSmallPieces.  Measured on
// MI355X through the C-ABI, one block of 64 KiB with the long / short list:
// 14.99 / 14.76 us device-to-host, 15.60 / 15.42 host-to-device.
constexpr int kFewPieces = 16;

template <int kPieces>
struct SmallArgs {
  uint64_t src[kPieces];
  uint64_t dst[kPieces];
  int32_t nvec[kPieces];   // 16-byte vectors of each piece
};

// One workgroup per piece (the host launches exactly as many as there are
// pieces, at most kPieces): wavefront `wave` of workgroup w takes rows
// wave + j * kWaves of piece w, j < small_rows_per_wave.  No branch sits
// between the argument loads and the data loads, so the piece's length and
// both addresses arrive in one round.  Device-to-host stores are plain: the
// kernel's end writes them back at once.  Written through (store_system), a call
// takes, plain -> through on MI355X, us: 4 KiB 13.69 -> 13.88, 64 KiB 15.04 ->
// 15.17, 256 KiB 18.57 -> 18.49, 1 MiB 32.62 -> 32.96.
template <bool kH2D, int kPieces>
__global__ __launch_bounds__(kThreads) void kv_small_copy_kernel(SmallArgs<kPieces> a) {
  constexpr int kU = small_rows_per_wave<kH2D>();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = blockIdx.x;
  const int n = a.nvec[w];
  const gvec* src = reinterpret_cast<const gvec*>(a.src[w]);
  gvec* dst = reinterpret_cast<gvec*>(a.dst[w]);
  // Every lane loads (past the piece's end it reloads the last vector, n >= 1),
  // so the loads carry no branch and all issue before the first wait.
  u32x4 v[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int vi = min((u * kWaves + wave) * 64 + lane, n - 1);
    v[u] = __builtin_nontemporal_load(src + vi);
  }
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int vi = (u * kWaves + wave) * 64 + lane;
    if (vi < n) {
      if (kH2D)
        __builtin_nontemporal_store(v[u], dst + vi);
      else
        dst[vi] = v[u];
    }
  }
}

std::mutex g_init_mu;

// ---------------------------------------------------------------------------
// Host-side policy of the transfer paths

// Compute units whose workgroups the small-transfer kernel may fill when the
// caller passes -1.
constexpr int kAutoSmallCus = 8;
// Copy-engine size policy: smallest transfer, and smallest bytes per engine
// copy, worth handing to the SDMA engines (ce_pays_off).  Measured on MI355X
// (block-wise host caches, random ids, GB/s zero-copy kernel / engines): the
// kernel is faster at every size (8 MiB of 2 MiB rows: D2H 46.1 / 45.9, H2D
// 50.0 / 45.8; 32 MiB: 55.3 / 53.5, 55.8 / 54.5; 64 MiB: 56.1 / 54.9, 56.7 /
// 55.2; 256 MiB: 56.8 / 55.9, 57.3 / 56.2), by 2-4% from 32 MiB, where the
// engines' leaving the compute units alone is worth more.  Below 32 MiB the
// kernel holds its workgroups for at most about 0.6 ms per transfer.
constexpr int64_t kCeMinBytesDefault = int64_t(32) << 20;
constexpr int64_t kCeMinRunBytes = int64_t(128) << 10;
// The copy-engine policy set through fkv_set_copy_engine_policy; -1: unset,
// so FLEXKV_CE_MIN_BYTES / FLEXKV_CE_RECT_COPIES, else the defaults, apply.
std::atomic<int64_t> g_ce_min_bytes{-1};
std::atomic<int> g_ce_rect_copies{-1};

int64_t ce_min_bytes() {
  const int64_t v = g_ce_min_bytes.load(std::memory_order_relaxed);
  if (v >= 0) return v;
  const char* e = getenv("FLEXKV_CE_MIN_BYTES");
  return e ? std::max<int64_t>(0, atoll(e)) : kCeMinBytesDefault;
}

// Whether a layer-wise host cache with scattered ids stays on the engines
// (rect copies) in copy-engine mode; default no (the zero-copy kernel).
bool ce_rect_copies() {
  const int v = g_ce_rect_copies.load(std::memory_order_relaxed);
  if (v >= 0) return v == 1;
  const char* r = getenv("FLEXKV_CE_RECT_COPIES");
  return r && atoi(r) == 1;
}
// The piece of a copy-engine transfer that runs without engine copies beside
// it (the first gather, the last scatter) is cut to 1 / kEdgePieceDiv of a
// staging half when it moves at least kEdgePieceMinBytes.
constexpr int kEdgePieceDiv = 8;
constexpr int64_t kEdgePieceMinBytes = int64_t(128) << 20;
// Default smallest engine copy per block of the copy-engine layer-wise
// pipeline (see layerwise_min_copy_bytes).  Measured on MI355X, Llama-3-8B
// one-layer groups (64 KiB per block), 1024 random blocks, engines 0-7:
// 37.6 / 47.2 / 50.5 / 51.1 / 51.1 GB/s with windows up to 64 KiB / 128 KiB /
// 256 KiB / 512 KiB / 1 MiB per block; per-layer GEMMs overlapped with it end
// within 0.0 / 0.5 / 0.6 / 8.3 / 8.3% of the transfer plus one layer's
// compute, and GEMMs beside it slow by the same few percent at every size.
constexpr int64_t kLayerwiseCeMinCopyBytes = int64_t(256) << 10;
// Average host run (bytes per (layer, K|V) run of consecutive blocks) from
// which a layer-wise host cache is staged layer-major and copied run by run
// instead of one rect copy per block.  Measured on MI355X at the Llama-3-8B
// shape, layer-major against rect copies (46.8 GB/s either way): runs of
// 128 KiB 41.2 / 32.4 GB/s (D2H / H2D), 256 KiB 51.1 / 42.0, 512 KiB
// 55.3 / 51.7.
constexpr int64_t kLayerRunBytes[2] = {int64_t(192) << 10, int64_t(384) << 10};   // [D2H, H2D]
// The average run from which layer-major staging is used;
// FLEXKV_CE_LAYER_RUN_BYTES overrides kLayerRunBytes.
int64_t layer_run_bytes(bool h2d) {
  const char* lr = getenv("FLEXKV_CE_LAYER_RUN_BYTES");
  return lr ? std::max<int64_t>(1, atoll(lr)) : kLayerRunBytes[h2d ? 1 : 0];
}
// transfer_staged's return when the copy engines cannot be set up (nothing
// was queued); not a hipError_t value
constexpr int kSdmaUnavailable = -1000;

int ensure_device_basics(int dev) {
  DeviceState& d = g_dev[dev];
  std::lock_guard<std::mutex> lk(g_init_mu);
  if (d.init) return 0;
  FKV_HIP(hipDeviceGetAttribute(&d.num_cus, hipDeviceAttributeMultiprocessorCount, dev));
  int o = 0;
  FKV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &o, reinterpret_cast<void*>(&kv_small_copy_kernel<false, kSmallPieces>), kThreads, 0));
  d.occ_small[0] = std::max(1, o);
  FKV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &o, reinterpret_cast<void*>(&kv_small_copy_kernel<true, kSmallPieces>), kThreads, 0));
  d.occ_small[1] = std::max(1, o);
  const void* zero_copy[2][2] = {   // [D2H, H2D][device memory, host memory]
      {reinterpret_cast<void*>(&kv_zero_copy_kernel<false, false>),
       reinterpret_cast<void*>(&kv_zero_copy_kernel<false, true>)},
      {reinterpret_cast<void*>(&kv_zero_copy_kernel<true, false>),
       reinterpret_cast<void*>(&kv_zero_copy_kernel<true, true>)}};
  for (int dir = 0; dir < 2; ++dir)
    for (int host = 0; host < 2; ++host) {
      FKV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&o, zero_copy[dir][host], kThreads, 0));
      d.occ_zero_copy[dir][host] = std::max(1, o);
    }
  d.init = true;
  return 0;
}

// Queue a copy of n values, `stride` apart in the pinned buffer `src`, into a
// device buffer held by `lease`, on `stream`.
int stage_table(const IdBuf& src, int stride, int n, int dev, hipStream_t stream,
                DevIdLease& lease) {
  lease.dev = dev;
  int rc = dev_ids_acquire(dev, static_cast<size_t>(n) * 8, &lease.buf);
  if (rc) return rc;
  (void)hipGetLastError();  // a stale error from elsewhere must not be blamed on this launch
  hipLaunchKernelGGL(stage_table_kernel, dim3((n + 255) / 256), dim3(256), 0, stream,
                     reinterpret_cast<const int64_t*>(src.dev), stride,
                     reinterpret_cast<int64_t*>(lease.buf.dev), n);
  FKV_HIP(hipGetLastError());
  return 0;
}

// The device tables of a transfer's staging launches: its gpu ids, and its
// layer pointers when a launch covers more than the kernel arguments hold.
struct StageTable {
  const int64_t* gids = nullptr;    // null: launches carry their ids inline
  const uint64_t* ptrs = nullptr;   // null: launches carry their layer pointers
};

// Queue the tables that launches of up to `nb` blocks and `nl` layers need.
int stage_tables(const Geometry& g, int nb, int nl, int dev, hipStream_t stream, IdLease& host,
                 DevIdLease& lease, StageTable* out) {
  const int n_ids = nb > kPackInlineIds ? g.num_blocks : 0;
  const int n_ptrs = nl > g.layers_per_launch() ? g.num_layers * g.ptrs_per_layer : 0;
  if (n_ids + n_ptrs == 0) return 0;
  int rc = ids_acquire(static_cast<size_t>(n_ids + n_ptrs) * 8, &host.buf);
  if (rc) return rc;
  memcpy(host.buf.host, g.gids, sizeof(int64_t) * n_ids);
  memcpy(host.buf.host + n_ids, g.layer_ptrs, sizeof(int64_t) * n_ptrs);
  if ((rc = stage_table(host.buf, 1, n_ids + n_ptrs, dev, stream, lease))) return rc;
  int64_t* dev_table = reinterpret_cast<int64_t*>(lease.buf.dev);
  if (n_ids) out->gids = dev_table;
  if (n_ptrs) out->ptrs = reinterpret_cast<uint64_t*>(dev_table + n_ids);
  return 0;
}

int64_t op_bytes(const Geometry& g) {
  return static_cast<int64_t>(g.num_blocks) * g.num_layers * g.kv * g.chunk;
}

// Workgroups of a zero-copy transfer of `g` on device `d`.
int zero_copy_grid(const Geometry& g, const DeviceState& d, int transfer_cus, bool h2d) {
  const bool host = !g.cpu_info.device;
  return zero_copy_workgroups(h2d, host, transfer_cus, d.num_cus, d.occ_zero_copy[h2d][host],
                              d.zero_copy_writes.load(std::memory_order_relaxed) > 0);
}

// Marks a synchronous zero-copy transfer of `g` that writes host memory as in
// flight for the lifetime of `mark`.  Layer-wise handles are not marked: a
// finished one may wait long for its release.
void mark_zero_copy(std::optional<BusyMark>& mark, const Geometry& g, DeviceState& d, bool h2d) {
  if (!h2d && !g.cpu_info.device) mark.emplace(d.zero_copy_writes);
}

// Shape of a staging launch, by its size.  Measured on MI355X, us a gather /
// scatter call (8 or 32 rows a wavefront; "columns": one workgroup per compute
// unit, held there by unused LDS, each walking its own run of the buffer):
//                                  8           32          32 columns
//   1 MiB, 32 KiB chunks       15.2 / 14.6  19.1 / 16.1
//   16 MiB, 32 KiB chunks      18.1 / 17.9  21.9 / 19.2
//   21 MiB, 72 KiB chunks      26.9 / 28.0  29.3 / 27.3
//   32 MiB, 32 KiB chunks      26.6 / 28.2  27.3 / 25.9
//   47 MiB, 2 KiB chunks       37.2 / 39.7  38.0 / 40.1   42.1 / 39.9
//   64 MiB, 4 KiB chunks       44.7 / 45.6  41.6 / 42.6   47.4 / 46.9
//   256 MiB, 18 KiB chunks      114 / 119    113 / 118     114 / 117
//   512 MiB, 32 KiB chunks      209 / 225    205 / 221     194 / 198
//   1 GiB, 72 KiB chunks        398 / 419    376 / 406     363 / 368
//   2 GiB, 32 KiB chunks        792 / 837    748 / 818     705 / 774
// So 8 rows until 32-row groups give every compute unit a workgroup, and
// columns from kPackColumnWgs workgroups a compute unit.
constexpr uint32_t kPackColumnWgs = 12;
constexpr unsigned kPackColumnLds = 84 << 10;

template <bool kH2D, int kU>
void launch_pack(PackArgs& pa, uint32_t num_cus, hipStream_t stream, hipEvent_t ea,
                 hipEvent_t eb) {
  pa.num_groups = (pa.num_vec + kU * 64 - 1) / (kU * 64);
  uint32_t grid = (pa.num_groups + kWaves - 1) / kWaves;
  const bool columns = kU == 32 && grid >= kPackColumnWgs * num_cus;
  pa.columns = Divider(columns ? num_cus : 1);
  pa.column_wgs = (grid + pa.columns.d - 1) / pa.columns.d;
  grid = pa.column_wgs * pa.columns.d;
  const unsigned lds = columns ? kPackColumnLds : 0;
  // chunks of whole rows always fit groups of 8 rows or more
  constexpr bool kWhole = kU > 1, kColumns = kH2D && kU == 32;
  const bool rows = pa.chunk.d % 64 == 0;
  auto kernel = rows ? kv_pack_kernel<kH2D, kU, kWhole, false> : kv_pack_kernel<kH2D, kU, false, false>;
  if (kH2D && columns)
    kernel = rows ? kv_pack_kernel<kH2D, kU, kWhole, kColumns>
                  : kv_pack_kernel<kH2D, kU, false, kColumns>;
  hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), lds, stream, ea, eb, 0, pa);
}

// Launch the staging gather / scatter over `nb` blocks of the call starting at
// block `b0` and GPU layers [l0, l0 + nl).  `packed` holds their chunks back to
// back, block -> layer -> K|V or, `layer_major`, layer -> K|V -> block.  More
// than kPackInlineIds blocks need table.gids, and layers beyond
// g.layers_per_launch() table.ptrs.
template <bool kH2D>
int launch_staging(const Geometry& g, const StageTable& table, char* packed, bool layer_major,
                   int b0, int nb, int l0, int nl, int dev, hipStream_t stream,
                   ProfRecorder& prof) {
  const int64_t items = static_cast<int64_t>(nl) * g.kv;
  PackArgs pa;
  return staging_launches(nb, items, g.chunk / 16, layer_major, kPackMaxVec,
                          [&](const StagingPart& p) -> int {
    const int b = b0 + p.b;
    const int64_t chunks = p.nb * p.items;
    // one item: its pointer with K|V applied
    const bool one = p.items == 1;
    const int64_t l = p.item / g.kv;
    const int lp = static_cast<int>(one ? 1 : p.items / g.kv);
    const bool wide = !one && lp > g.layers_per_launch();
    if ((p.nb > kPackInlineIds && !table.gids) || (wide && !table.ptrs))
      return fail(kInval, "internal: a staging launch of %d blocks and %d layers without its "
                  "tables", p.nb, lp);
    pa.gids = table.gids ? table.gids + b : nullptr;
    if (!pa.gids) memcpy(pa.inline_ids, g.gids + b, sizeof(int64_t) * p.nb);
    pa.ptrs = nullptr;
    if (one)
      pa.layer_ptr[0] = reinterpret_cast<uint64_t>(
          g.gpu_base(l0 + static_cast<int>(l), static_cast<int>(p.item % g.kv)) + p.off * 16);
    else if (wide)
      pa.ptrs = table.ptrs + (l0 + l) * g.ptrs_per_layer;
    else
      memcpy(pa.layer_ptr, g.layer_ptrs + (l0 + l) * g.ptrs_per_layer,
             sizeof(uint64_t) * lp * g.ptrs_per_layer);
    pa.packed = packed + p.packed * 16;
    pa.gpu_kv_stride = g.gks;
    pa.gpu_block_stride = g.gbs;
    pa.chunk = Divider(static_cast<uint32_t>(p.vec));
    pa.inner = Divider(static_cast<uint32_t>(layer_major ? p.nb : p.items));
    pa.layer_major = layer_major;
    pa.kv_dim = one ? 1 : static_cast<uint32_t>(g.kv);
    pa.ptrs_per_layer = one ? 1 : g.ptrs_per_layer;
    pa.num_chunks = static_cast<uint32_t>(chunks);
    pa.num_vec = static_cast<uint32_t>(chunks * p.vec);
    hipEvent_t ea = nullptr, eb = nullptr;
    int rc = prof.kernel_events(&ea, &eb);
    if (rc) return rc;
    prof.kernel_span(ea, eb, chunks * p.vec * 16);   // owns the events from here on
    (void)hipGetLastError();  // a stale error from elsewhere must not be blamed on this launch
    const uint32_t num_cus = static_cast<uint32_t>(g_dev[dev].num_cus);
    if (pack_fits(32, p.vec) && pa.num_vec >= int64_t(num_cus) * kWaves * 32 * 64)
      launch_pack<kH2D, 32>(pa, num_cus, stream, ea, eb);
    else if (pack_fits(8, p.vec))
      launch_pack<kH2D, 8>(pa, num_cus, stream, ea, eb);
    else
      launch_pack<kH2D, 1>(pa, num_cus, stream, ea, eb);
    FKV_HIP(hipGetLastError());
    return 0;
  });
}

// Launch kv_zero_copy_kernel over call layers [l0, l0 + nl) of every block of
// the call.  `cpu_base` is the host-side address of call layer 0 of block id
// 0; `ids` holds the packed pairs: `host` for the host's view, `dev` for the
// device's (the same pinned buffer), or with `split` > 0 `dev` holds the gpu
// ids and, `split` entries later, the cpu ids, and `host` is null; at most
// `grid_cap` workgroups a launch.  The limits are those of the layer pointers a
// launch carries, of Divider and of a workgroup's LDS.  `done` (null while
// profiling): an event the last launch completes, carried by its own packet
// instead of a marker behind it.
template <bool kH2D>
int launch_zero_copy(const Geometry& g, const IdBuf& ids, char* cpu_base, int l0, int nl,
                     int grid_cap, hipStream_t stream, ProfRecorder& prof, int32_t split = 0,
                     hipEvent_t done = nullptr) {
  const bool host = !g.cpu_info.device;
  const int64_t group_vec = (host ? zero_copy_rows<kH2D, true>() : zero_copy_rows<kH2D, false>()) * 64;
  const auto kernel = host ? kv_zero_copy_kernel<kH2D, true> : kv_zero_copy_kernel<kH2D, false>;
  const ZeroCopyLimits limits{kZeroCopyMaxVec, kZeroCopyMaxChunkVec, kZeroCopyMaxLds / 16,
                              g.layers_per_launch()};
  ZeroCopyArgs a;
  return zero_copy_launches(g.num_blocks, nl, g.kv, g.chunk / 16, group_vec, kWaves, grid_cap,
                            limits, [&](const ZeroCopyPart& p) -> int {
    const int lw = l0 + p.layer;
    a.ids = reinterpret_cast<const int64_t*>(ids.dev) + (split ? 1 : 2) * static_cast<int64_t>(p.b);
    a.ids_split = split;
    a.inline_n = 0;
    if (p.nb <= kInlineIdsZeroCopy && ids.host) {
      a.inline_n = p.nb;
      memcpy(a.inline_ids, ids.host + 2 * static_cast<int64_t>(p.b), sizeof(int64_t) * 2 * p.nb);
    }
    a.cpu_base = cpu_base + static_cast<int64_t>(lw) * g.cls + p.off * 16;
    a.gpu_kv_stride = g.gks;
    a.gpu_block_stride = g.gbs;
    a.cpu_kv_stride = g.cks;
    a.cpu_layer_stride = g.cls;
    a.cpu_block_stride = g.cbs;
    a.chunk = Divider(static_cast<uint32_t>(p.vec));
    a.items = Divider(static_cast<uint32_t>(p.layers * g.kv));
    a.kv_dim = static_cast<uint32_t>(g.kv);
    a.num_vec = static_cast<uint32_t>(p.num_vec);
    a.num_groups = static_cast<uint32_t>(p.groups);
    a.groups_per_wg = static_cast<uint32_t>(p.groups_per_wg);
    a.ptrs_per_layer = g.ptrs_per_layer;
    for (int i = 0; i < p.layers * g.ptrs_per_layer; ++i)
      a.layer_ptr[i] = reinterpret_cast<uint64_t>(g.layer_ptrs[lw * g.ptrs_per_layer + i]) +
                       static_cast<uint64_t>(p.off) * 16;
    hipEvent_t ea = nullptr, eb = nullptr;
    int rc = prof.kernel_events(&ea, &eb);
    if (rc) return rc;
    prof.kernel_span(ea, eb, p.num_vec * 16);
    if (!eb && p.last) eb = done;
    (void)hipGetLastError();  // a stale error from elsewhere must not be blamed on this launch
    hipExtLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(p.workgroups())), dim3(kThreads),
                          static_cast<uint32_t>(p.run_blocks * 16), stream, ea, eb, 0, a);
    FKV_HIP(hipGetLastError());
    return 0;
  });
}

// Pieces a call takes in kv_small_copy_kernel when it fits (at most
// kSmallPieces pieces, kSmallMaxBytes, and one workgroup per piece within
// the call's `grid_cap` workgroups), else 0.  FLEXKV_SMALL_KERNEL=0 sends
// every call to the general kernel.
int small_pieces(const Geometry& g, int grid_cap, bool h2d) {
  if (const char* e = getenv("FLEXKV_SMALL_KERNEL"))
    if (atoi(e) == 0) return 0;
  const int64_t chunks = static_cast<int64_t>(g.num_blocks) * g.num_layers * g.kv;
  if (chunks < 1 || chunks > kSmallPieces || chunks * g.chunk > kSmallMaxBytes) return 0;
  const int64_t piece_bytes =
      int64_t(h2d ? small_piece_rows<true>() : small_piece_rows<false>()) * 64 * 16;
  const int64_t n = chunks * ((g.chunk + piece_bytes - 1) / piece_bytes);
  return n > std::min(kSmallPieces, grid_cap) ? 0 : static_cast<int>(n);
}

// One launch of kv_small_copy_kernel over the whole call.  `cpu_dev` is the
// device-visible address of the host cache at call layer 0 (start layer and
// start offset applied).  Chunk sizes are multiples of 16 bytes here.
template <bool kH2D, int kPieces>
int launch_small(const Geometry& g, char* cpu_dev, int n_pieces, hipStream_t stream,
                   ProfRecorder& prof) {
  SmallArgs<kPieces> a;
  const int64_t piece_bytes = int64_t(small_piece_rows<kH2D>()) * 64 * 16;
  int p = 0;
  for (int l = 0; l < g.num_layers; ++l)
    for (int k = 0; k < g.kv; ++k)
      for (int i = 0; i < g.num_blocks; ++i) {
        char* gpu = g.gpu_base(l, k) + g.gids[i] * g.gbs;
        char* cpu = cpu_dev + static_cast<int64_t>(l) * g.cls + k * g.cks + g.cids[i] * g.cbs;
        for (int64_t off = 0; off < g.chunk; off += piece_bytes, ++p) {
          a.src[p] = reinterpret_cast<uint64_t>((kH2D ? cpu : gpu) + off);
          a.dst[p] = reinterpret_cast<uint64_t>((kH2D ? gpu : cpu) + off);
          a.nvec[p] = static_cast<int32_t>(std::min(piece_bytes, g.chunk - off) / 16);
        }
      }
  if (p != n_pieces) return fail(kInval, "internal: %d small-transfer pieces, expected %d", p,
                                 n_pieces);
  hipEvent_t ea = nullptr, eb = nullptr;
  int rc = prof.kernel_events(&ea, &eb);
  if (rc) return rc;
  prof.kernel_span(ea, eb, op_bytes(g));
  (void)hipGetLastError();  // a stale error from elsewhere must not be blamed on this launch
  hipExtLaunchKernelGGL((kv_small_copy_kernel<kH2D, kPieces>), dim3(n_pieces), dim3(kThreads), 0,
                        stream, ea, eb, 0, a);
  FKV_HIP(hipGetLastError());
  return 0;
}

template <bool kH2D>
int transfer_small(const Geometry& g, char* cpu_dev, int n_pieces, hipStream_t stream,
                   ProfRecorder& prof) {
  return n_pieces <= kFewPieces
             ? launch_small<kH2D, kFewPieces>(g, cpu_dev, n_pieces, stream, prof)
             : launch_small<kH2D, kSmallPieces>(g, cpu_dev, n_pieces, stream, prof);
}

int transfer_zero_copy(const Geometry& g, hipStream_t stream, int dev, int transfer_cus,
                       bool h2d) {
  DeviceState& d = g_dev[dev];
  const int small_cus = transfer_cus <= 0 ? std::min(kAutoSmallCus, d.num_cus)
                                          : std::min(transfer_cus, d.num_cus);
  if (const int n = small_pieces(g, small_cus * (h2d ? d.occ_small[1] : d.occ_small[0]), h2d)) {
    DrainOnError drain{stream};
    char* cpu_dev = g.cpu_info.dev_ptr + g.startoff +
                    static_cast<int64_t>(g.start_layer) * g.cls;
    ProfRecorder prof;
    const int rc = h2d ? transfer_small<true>(g, cpu_dev, n, stream, prof)
                       : transfer_small<false>(g, cpu_dev, n, stream, prof);
    if (rc) return rc;
    FKV_HIP(hipStreamSynchronize(stream));
    drain.armed = false;
    prof.flush();
    return 0;
  }
  IdLease ids;
  int rc = pack_ids(g, ids);
  if (rc) return rc;
  std::optional<BusyMark> writing;
  mark_zero_copy(writing, g, d, h2d);
  DrainOnError drain{stream};
  const int grid_cap = zero_copy_grid(g, d, transfer_cus, h2d);
  char* cpu_dev = g.cpu_info.dev_ptr + g.startoff +
                  static_cast<int64_t>(g.start_layer) * g.cls;
  ProfRecorder prof;
  rc = h2d ? launch_zero_copy<true>(g, ids.buf, cpu_dev, 0, g.num_layers, grid_cap, stream, prof)
           : launch_zero_copy<false>(g, ids.buf, cpu_dev, 0, g.num_layers, grid_cap, stream, prof);
  if (rc) return rc;
  FKV_HIP(hipStreamSynchronize(stream));
  drain.armed = false;
  prof.flush();
  return 0;
}

// ---------------------------------------------------------------------------
// The entry point that allocates nothing (fkv_transfer_kv_blocks_noalloc):
// the zero-copy transfer with its id lists staged in `scratch`, a fixed
// device array, instead of a pinned buffer the library allocates.  Each GPU
// holds its own copy of the array; host code reaches it only through the
// address hipGetSymbolAddress returns for the device (the array's name is a
// host-side stand-in, not a device address).  Every call on a device shares
// that device's array, so a call holds the device's scratch mutex from the
// copy of its ids into the array until its kernels have finished: calls
// from several threads on one device take turns instead of racing.

constexpr size_t kScratchBytes = size_t(1) << 20;
// gpu ids in the first half, cpu ids in the second
constexpr int kScratchMaxBlocks = static_cast<int>(kScratchBytes / (2 * sizeof(int64_t)));

static __device__ __align__(256) int64_t scratch[kScratchBytes / sizeof(int64_t)];

std::mutex g_scratch_mu;
int64_t* g_scratch_dev[kMaxDevices];   // scratch's address on each device, once resolved
// held by a call from its scratch copy until its stream is synchronised
std::mutex g_scratch_use_mu[kMaxDevices];

// scratch's device address on `dev` (resolved once per device, with the
// device current).
int scratch_address(int dev, int64_t** out) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    DeviceGuard guard;
    int rc = guard.set(dev);
    if (rc) return rc;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(static_cast<int>(e == hipSuccess ? hipErrorInvalidSymbol : e),
                  "hipGetSymbolAddress(scratch) on device %d failed: %s", dev,
                  hipGetErrorString(e));
    g_scratch_dev[dev] = static_cast<int64_t*>(p);
  }
  *out = g_scratch_dev[dev];
  return 0;
}

int transfer_zero_copy_noalloc(const Geometry& g, hipStream_t stream, int dev, int transfer_cus,
                               bool h2d) {
  DeviceState& d = g_dev[dev];
  if (g.num_blocks > kScratchMaxBlocks)
    return fail(kInval, "fkv_transfer_kv_blocks_noalloc moves at most %d blocks per call "
                "(its id scratch is %zu bytes), got %d", kScratchMaxBlocks, kScratchBytes,
                g.num_blocks);
  const int small_cus = transfer_cus <= 0 ? std::min(kAutoSmallCus, d.num_cus)
                                          : std::min(transfer_cus, d.num_cus);
  if (const int n = small_pieces(g, small_cus * (h2d ? d.occ_small[1] : d.occ_small[0]), h2d)) {
    DrainOnError drain{stream};
    char* cpu_dev = g.cpu_info.dev_ptr + g.startoff + static_cast<int64_t>(g.start_layer) * g.cls;
    ProfRecorder prof;
    prof.on = false;   // profiling events are allocations
    const int rc = h2d ? transfer_small<true>(g, cpu_dev, n, stream, prof)
                       : transfer_small<false>(g, cpu_dev, n, stream, prof);
    if (rc) return rc;
    FKV_HIP(hipStreamSynchronize(stream));
    drain.armed = false;
    return 0;
  }
  int64_t pairs[2 * kInlineIdsZeroCopy];
  IdBuf ids;
  int32_t split = 0;
  // Declared before the DrainOnError below, so an error path drains the
  // stream before the next call may overwrite the scratch.
  std::unique_lock<std::mutex> scratch_use(g_scratch_use_mu[dev], std::defer_lock);
  if (g.num_blocks <= kInlineIdsZeroCopy) {
    // the ids travel in the kernel arguments
    pack_ids_into(g, pairs);
    ids.host = pairs;
  } else {
    int64_t* sp = nullptr;
    int rc = scratch_address(dev, &sp);
    if (rc) return rc;
    scratch_use.lock();
    const size_t n = static_cast<size_t>(g.num_blocks) * sizeof(int64_t);
    DrainOnError copy_drain{stream};   // a failed second copy still waits for the first
    FKV_HIP(hipMemcpyAsync(sp, g.gids, n, hipMemcpyHostToDevice, stream));
    FKV_HIP(hipMemcpyAsync(sp + kScratchMaxBlocks, g.cids, n, hipMemcpyHostToDevice, stream));
    copy_drain.armed = false;
    ids.dev = reinterpret_cast<char*>(sp);
    split = kScratchMaxBlocks;
  }
  std::optional<BusyMark> writing;
  mark_zero_copy(writing, g, d, h2d);
  DrainOnError drain{stream};
  const int grid_cap = zero_copy_grid(g, d, transfer_cus, h2d);
  char* cpu_dev = g.cpu_info.dev_ptr + g.startoff + static_cast<int64_t>(g.start_layer) * g.cls;
  ProfRecorder prof;
  prof.on = false;   // profiling events are allocations
  const int rc = h2d ? launch_zero_copy<true>(g, ids, cpu_dev, 0, g.num_layers, grid_cap, stream,
                                              prof, split)
                     : launch_zero_copy<false>(g, ids, cpu_dev, 0, g.num_layers, grid_cap, stream,
                                               prof, split);
  if (rc) return rc;
  FKV_HIP(hipStreamSynchronize(stream));
  drain.armed = false;
  return 0;
}

// Copy-engine transfer: the SDMA engines move whole-block runs between the
// host cache and double-buffered HBM staging; a gather (D2H) or scatter
// (H2D) kernel on the caller's stream moves them between staging and the
// per-layer cache.  The host thread orders the two, so no compute unit
// takes part in the PCIe copies.
//  D2H, per piece: wait for the half's previous copies -> gather kernel ->
//  wait for it -> queue the half's copies.
//  H2D: queue the copies of the first two pieces; per piece: wait for its
//  copies -> system-scope acquire -> scatter kernel; once that has read the
//  half, queue the copies of the piece two ahead into it.
// fkv_prepare: polled completion signals it creates per staging half (one
// per block of a 1024-block layer-wise window; the pools grow on demand),
// and the pinned host buffer of its warm-up copies (4 KiB per engine).
constexpr size_t kPrepareSignalsPerHalf = 1024;
constexpr size_t kPrepareHostBytes = size_t(64) << 10;

// Staging for a copy-engine transfer (ensure_staging): 0; kSdmaUnavailable
// when the device has no memory left for it, so the transfer moves with the
// zero-copy kernel instead (warned once per device; later transfers try the
// allocation again); or another error.
int staging_or_fallback(DeviceState& d, int dev, CopyLane& ln, size_t need_half) {
  const int rc = ensure_staging(ln, need_half);
  if (rc != static_cast<int>(hipErrorOutOfMemory)) return rc;
  (void)hipGetLastError();
  if (!d.staging_oom_warned.exchange(true))
    fprintf(stderr, "flexkv: no device memory for copy-engine staging on device %d (%s); "
            "such transfers use the zero-copy kernel until the allocation succeeds\n", dev,
            last_error().c_str());
  last_error().clear();
  return kSdmaUnavailable;
}

// Edge pieces below kEdgePieceMinBytes: one of at least edge_small_min_bytes()
// (FLEXKV_CE_EDGE_MIN_BYTES, default 32 MiB) gives 1 / kEdgeSmallDiv of its
// blocks to a piece of its own.  Measured on MI355X, Llama-3-8B block rows
// (2 MiB), copy-engine transfers with / without the cut: 16 blocks 628.8 /
// 631.5 us D2H, 627.3 / 637.9 us H2D; 32 blocks 1216 / 1236 us D2H, 1214 /
// 1237 us H2D; 4 blocks (8 MiB) 181 / 183 us D2H but 198 / 183 us H2D, where
// the extra piece's host round trip is not hidden behind 2 MiB of copies.
constexpr int kEdgeSmallDiv = 4;
constexpr int64_t kEdgeSmallMinBytesDefault = int64_t(32) << 20;

int64_t edge_small_min_bytes() {
  const char* e = getenv("FLEXKV_CE_EDGE_MIN_BYTES");
  return e ? std::max<int64_t>(1, atoll(e)) : kEdgeSmallMinBytesDefault;
}

// Host-to-device engine copies shorter than this on average spread over the
// synchronous wide set (engines 0-5) instead of the direction's four (0-3).
// Measured on MI355X: 256 KiB copies 51.7 GB/s on 0-3, 56.1 on 0-5; 640 KiB
// copies (Llama-3-70B TP-8 shard) 57.0 on 0-3, 56.4 on 0-5.  While a D2H is
// in flight, host-to-device copies of any size take the duplex split
// instead (issue_sdma).
constexpr int64_t kWideCopyBytes = int64_t(384) << 10;
// Host-to-device copies on the wide set run beside the scatter of the
// previous piece, and every engine in flight slows that scatter (MI355X,
// Llama-3-70B TP-8 shard, 640 KiB copies: 512 MiB scatter pieces 4.26 /
// 4.65 / 4.90 TB/s beside 8 / 6 / 4 engines).  So the engines of the set
// beyond the first kHoldKeepEngines take their share of a piece only once
// that scatter is done (issue_sdma, SdmaHold).  held_fraction is the
// scatter's expected time, plus the host's wake-up, over the piece's time on
// the link; FLEXKV_SDMA_HOLD_SCALE scales it (0: no engine is held).
double held_fraction(int64_t prev_piece_bytes, int64_t piece_bytes) {
  const char* e = getenv("FLEXKV_SDMA_HOLD_SCALE");
  const double scale = e ? std::max(0.0, atof(e)) : 1.0;
  if (scale <= 0 || piece_bytes <= 0) return 0.0;
  constexpr double kScatterBytesPerS = 4.9e12;   // HBM bytes, read + write
  constexpr double kLinkBytesPerS = 56e9;
  constexpr double kWakeS = 20e-6;
  const double d = 2.0 * static_cast<double>(prev_piece_bytes) / kScatterBytesPerS + kWakeS;
  return scale * d / (static_cast<double>(piece_bytes) / kLinkBytesPerS);
}

int transfer_staged(const Geometry& g, hipStream_t stream, int dev, bool h2d) {
  DeviceState& d = g_dev[dev];
  CopyLane& ln = d.lane[h2d ? 1 : 0];
  // Staging order: block-major [block][layer][K|V][chunk] (contiguous block
  // rows, or one rect copy per block of a layer-wise cache), or layer-major
  // [layer][K|V][block][chunk] when a layer-wise cache's ids come in runs of
  // consecutive blocks long enough to copy each (layer, K|V) run linearly.
  const bool layer_major = layer_major_pays_off(g, layer_run_bytes(h2d));
  const bool row_contig = (g.kv == 1 || g.cks == g.chunk) &&
                          (g.num_layers == 1 || g.cls == g.kv * g.chunk);
  // A transfer of rect copies runs alone on the device: those go to the
  // engine the runtime picks, and the runtime must not see them beside copies
  // pinned to engines.  Other transfers hold their direction's lane only.
  const bool rect_copies = !row_contig && !layer_major;
  std::unique_lock<std::mutex> own(ln.mu, std::defer_lock);
  std::unique_lock<std::mutex> other(d.lane[h2d ? 0 : 1].mu, std::defer_lock);
  if (rect_copies)
    std::lock(own, other);
  else
    own.lock();
  BusyMark busy(d.busy[h2d ? 1 : 0]);
  DeviceGuard guard;
  int rc = guard.set(dev);
  if (rc) return rc;
  IdLease ids;
  DevIdLease dev_ids;   // released after the drain below
  StageTable table;

  // A piece is a run of whole blocks over a layer window; the window covers
  // all layers unless one block row would not fit a staging half.
  const size_t req = g_staging_request.load();
  const size_t half_default = (req ? req : kDefaultStagingBytes) / 2;
  int nl_piece = std::min(g.num_layers, g.layers_per_launch());
  while (nl_piece > 1 && static_cast<size_t>(nl_piece) * g.kv * g.chunk > half_default) nl_piece /= 2;
  const size_t row_bytes = static_cast<size_t>(nl_piece) * g.kv * g.chunk;
  rc = staging_or_fallback(d, dev, ln, row_bytes);
  if (rc) return rc;   // kSdmaUnavailable: the caller moves it with the zero-copy kernel
  if ((rc = ensure_sdma(d, dev, ln.staging))) {
    // nothing has been queued yet: the caller moves this transfer, and every
    // later one on the device, with the zero-copy kernel
    if (!d.sdma_failed.exchange(true))
      fprintf(stderr, "flexkv: copy engines unavailable on device %d (%s); copy-engine "
              "transfers use the zero-copy kernel\n", dev, last_error().c_str());
    last_error().clear();
    return kSdmaUnavailable;
  }
  const size_t half = ln.staging_bytes / 2;
  const int blocks_per_piece = static_cast<int>(std::max<size_t>(1, half / row_bytes));
  const hsa_agent_t host_agent = d.cpu_agent;   // device-resident caches never get here

  struct Piece {
    int l0, nl, b0, nb;
  };
  std::vector<Piece> pieces;
  for (int l0 = 0; l0 < g.num_layers; l0 += nl_piece)
    for (int b0 = 0; b0 < g.num_blocks; b0 += blocks_per_piece)
      pieces.push_back({l0, std::min(nl_piece, g.num_layers - l0), b0,
                        std::min(blocks_per_piece, g.num_blocks - b0)});
  // The first piece's gather (D2H) and the last piece's scatter (H2D) run
  // with no engine copies beside them.  When that piece is large, an eighth
  // of a half is cut off it, so the engines start, or the transfer ends,
  // after a short kernel.  A smaller edge piece of at least
  // edge_small_min_bytes() gives a quarter of its blocks instead; below that
  // it is not cut, since every piece costs a host round trip.
  if (!pieces.empty()) {
    const size_t edge = h2d ? pieces.size() - 1 : 0;
    const Piece p = pieces[edge];
    const int64_t bytes = static_cast<int64_t>(p.nb) * p.nl * g.kv * g.chunk;
    int cut = 0;
    if (bytes >= kEdgePieceMinBytes)
      cut = std::min(p.nb - 1, std::max(1, blocks_per_piece / kEdgePieceDiv));
    else if (bytes >= edge_small_min_bytes())
      cut = std::min(p.nb - 1, std::max(1, p.nb / kEdgeSmallDiv));
    if (cut >= 1) {
      Piece first = p, second = p;
      first.nb = h2d ? p.nb - cut : cut;
      second.b0 = p.b0 + first.nb;
      second.nb = p.nb - first.nb;
      pieces[edge] = first;
      pieces.insert(pieces.begin() + static_cast<std::ptrdiff_t>(edge) + 1, second);
    }
  }
  const int np = static_cast<int>(pieces.size());

  // Host-side waits order everything below against the caller's stream, so
  // work already queued on it comes first.
  FKV_HIP(hipStreamSynchronize(stream));
  // After the drain below (declared later, so it runs first), hand the host
  // blocks of device-to-host copies given up on to the calling thread
  // (fkv_last_unsafe_host_blocks).
  struct PublishUnsafeRows {
    CopyLane& ln;
    ~PublishUnsafeRows() {
      std::vector<int64_t> ids = ln.rows.take_unsafe();
      if (!ids.empty()) last_unsafe_host_blocks() = std::move(ids);
    }
  } publish{ln};
  DrainOnError drain{stream, &d, &ln};
  if ((rc = stage_tables(g, std::min(blocks_per_piece, g.num_blocks), nl_piece, dev, stream, ids,
                         dev_ids, &table)))
    return rc;
  ProfRecorder prof;
  std::vector<Run> runs;
  bool pending[2] = {false, false};
  int64_t dma_copies = 0, dma_bytes = 0, held_copies = 0;
  const auto t0 = std::chrono::steady_clock::now();
  // Host-to-device copies into one half run beside the scatter of the other
  // half's previous piece; the held engines' share of them waits for that
  // scatter (issue_sdma, SdmaHold) and is queued by release_held.
  SdmaHold hold[2];
  auto piece_bytes_of = [&](int pi) {
    const Piece& p = pieces[pi];
    return static_cast<int64_t>(p.nb) * p.nl * g.kv * g.chunk;
  };
  auto queue_copies = [&](int pi) -> int {
    const Piece& p = pieces[pi];
    const int h = pi & 1;
    build_runs(g, p.b0, p.nb, p.l0, p.nl, sdma_rect_available(), layer_major, runs);
    int64_t piece_bytes = 0;
    for (const Run& r : runs) piece_bytes += r.bytes * std::max<int64_t>(1, r.slices);
    dma_bytes += piece_bytes;
    dma_copies += static_cast<int64_t>(runs.size());
    pending[h] = true;
    if (!h2d) ln.rows.queued(h, g.cids + p.b0, static_cast<size_t>(p.nb));
    // Host-to-device copies shorter than kWideCopyBytes on average are bound
    // by the engines' per-copy cost and spread over the wide set
    const bool wide = h2d && !runs.empty() &&
                      piece_bytes < kWideCopyBytes * static_cast<int64_t>(runs.size());
    hold[h].held_fraction = wide && pi > 0 ? held_fraction(piece_bytes_of(pi - 1), piece_bytes)
                                           : 0.0;
    return issue_sdma(d, ln, runs, ln.staging + h * half, h2d, h, host_agent,
                      wide ? kEnginesWideSync : kEnginesOwn, &hold[h]);
  };
  auto release_held = [&](int pi) -> int {
    const int h = pi & 1;
    if (hold[h].deferred.empty()) return 0;
    held_copies += static_cast<int64_t>(hold[h].deferred.size());
    const int rc2 = issue_sdma(d, ln, hold[h].deferred, ln.staging + h * half, h2d, h,
                               host_agent, kEnginesWideSync, nullptr, /*held_part=*/true);
    hold[h].deferred.clear();
    return rc2;
  };
  auto launch = [&](int pi) -> int {
    const Piece& p = pieces[pi];
    char* stg = ln.staging + (pi & 1) * half;
    return h2d ? launch_staging<true>(g, table, stg, layer_major, p.b0, p.nb, p.l0, p.nl, dev,
                                      stream, prof)
               : launch_staging<false>(g, table, stg, layer_major, p.b0, p.nb, p.l0, p.nl, dev,
                                       stream, prof);
  };
  if (!h2d) {
    for (int pi = 0; pi < np; ++pi) {
      const int h = pi & 1;
      if (pending[h]) {
        pending[h] = false;
        if ((rc = sdma_wait(d, ln, h))) return rc;
      }
      if ((rc = launch(pi))) return rc;
      FKV_HIP(hipEventRecord(ln.ev_compute[h], stream));
      FKV_HIP(hipEventSynchronize(ln.ev_compute[h]));
      if ((rc = queue_copies(pi))) return rc;
    }
  } else {
    for (int pi = 0; pi < std::min(np, 2); ++pi)
      if ((rc = queue_copies(pi))) return rc;
    for (int pi = 0; pi < np; ++pi) {
      const int h = pi & 1;
      pending[h] = false;
      // the last piece has nothing behind it
      if ((rc = sdma_wait(d, ln, h, /*spin=*/pi + 1 == np))) return rc;
      hipLaunchKernelGGL(acquire_system_kernel, dim3(d.num_cus), dim3(64), 0, stream);
      FKV_HIP(hipGetLastError());
      if ((rc = launch(pi))) return rc;
      if (pi + 1 < np) {
        FKV_HIP(hipEventRecord(ln.ev_compute[h], stream));
        FKV_HIP(hipEventSynchronize(ln.ev_compute[h]));
        // the scatter of piece pi is done: the held engines take their share
        // of piece pi + 1, and piece pi + 2 goes into the half it read
        if ((rc = release_held(pi + 1))) return rc;
        if (pi + 2 < np && (rc = queue_copies(pi + 2))) return rc;
      }
    }
  }
  for (int h = 0; h < 2; ++h)
    if (pending[h]) {
      pending[h] = false;
      if ((rc = sdma_wait(d, ln, h, /*spin=*/true))) return rc;
    }
  FKV_HIP(hipStreamSynchronize(stream));
  drain.armed = false;
  if (prof.on) {
    const double ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    prof_add_dma(ms, dma_copies, dma_bytes, held_copies);
  }
  prof.flush();
  return 0;
}

// Gather (to_gpu = false) or scatter between the GPU cache and a contiguous
// buffer laid out [block][layer][K|V][chunk]; g.cpu_ptr is the buffer and
// g.cids is 0..n-1.  With the buffer in device memory the copy is HBM-bound
// and uses every compute unit.  A buffer in host memory is a host cache of its
// own: the link bounds the copy, and the staging kernel's many workgroups fill
// it worse than the zero-copy kernel's few.  Measured on MI355X, us a gather /
// scatter: 16 MiB of 32 KiB chunks 384 / 369 -> 309 / 308, of 528 B 386 / 377
// -> 313 / 312, 256 MiB of 32 KiB 5000 / 4841 -> 4722 / 4678.
int transfer_contiguous(const Geometry& g, hipStream_t stream, int dev, bool to_gpu) {
  if (!g.cpu_info.device) return transfer_zero_copy(g, stream, dev, -1, to_gpu);
  IdLease ids;
  DevIdLease dev_ids;
  StageTable table;
  DrainOnError drain{stream};
  int rc = stage_tables(g, g.num_blocks, g.num_layers, dev, stream, ids, dev_ids, &table);
  if (rc) return rc;
  ProfRecorder prof;
  char* buffer = g.cpu_info.dev_ptr;
  rc = to_gpu ? launch_staging<true>(g, table, buffer, false, 0, g.num_blocks, 0, g.num_layers,
                                     dev, stream, prof)
              : launch_staging<false>(g, table, buffer, false, 0, g.num_blocks, 0, g.num_layers,
                                      dev, stream, prof);
  if (rc) return rc;
  FKV_HIP(hipStreamSynchronize(stream));
  drain.armed = false;
  prof.flush();
  return 0;
}

int contiguous_entry(int num_blocks, int num_layers, const int64_t* gpu_block_ids,
                     void* const* gpu_layer_ptrs, int64_t gpu_kv_stride_bytes,
                     int64_t gpu_block_stride_bytes, int64_t chunk_size_bytes, void* buffer,
                     size_t buffer_bytes, fkv_stream_t stream, int is_mla, bool to_gpu) {
  try {
    last_error().clear();
    last_unsafe_host_blocks().clear();
    if (num_blocks == 0 || num_layers == 0) return 0;
    if (num_blocks < 0 || num_layers < 0)
      return fail(kInval, "negative count: num_blocks=%d num_layers=%d", num_blocks, num_layers);
    std::vector<int64_t> iota(static_cast<size_t>(num_blocks));
    for (int i = 0; i < num_blocks; ++i) iota[i] = i;
    Geometry g;
    g.num_blocks = num_blocks;
    g.start_layer = 0;
    g.num_layers = num_layers;
    g.kv = is_mla ? 1 : 2;
    g.gids = gpu_block_ids;
    g.cids = iota.data();
    g.layer_ptrs = gpu_layer_ptrs;
    g.gks = gpu_kv_stride_bytes;
    g.gbs = gpu_block_stride_bytes;
    g.chunk = chunk_size_bytes;
    g.cks = g.kv == 1 ? 0 : chunk_size_bytes;
    g.cls = static_cast<int64_t>(g.kv) * chunk_size_bytes;
    g.cbs = static_cast<int64_t>(num_layers) * g.cls;
    g.startoff = 0;
    g.cpu_ptr = static_cast<char*>(buffer);
    const __int128 need = static_cast<__int128>(num_blocks) * g.cbs;
    if (need > static_cast<__int128>(buffer_bytes))
      return fail(kInval, "buffer holds %zu bytes, the blocks need %lld", buffer_bytes,
                  static_cast<long long>(need));
    int rc = validate(g, FKV_XFER_KERNEL);
    if (rc) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    int dev = 0;
    if ((rc = stream_device(s, &dev))) return rc;
    if ((rc = ensure_device_basics(dev))) return rc;
    return transfer_contiguous(g, s, dev, to_gpu);
  } catch (const std::exception& e) {
    return fail(static_cast<int>(hipErrorUnknown), "exception: %s", e.what());
  } catch (...) {
    return fail(static_cast<int>(hipErrorUnknown), "unknown exception");
  }
}

// The reference copy-engine loop, csrc/transfer.cu:97-121: one async copy per
// (layer, K|V, block) chunk, issued layer-major then K|V then block.
int transfer_ce_per_chunk(const Geometry& g, hipStream_t stream, bool h2d) {
  DrainOnError drain{stream};
  ProfRecorder prof;
  hipEvent_t ev = nullptr;
  int rc = prof.begin(stream, &ev);
  if (rc) return rc;
  for (int l = 0; l < g.num_layers; ++l) {
    for (int k = 0; k < g.kv; ++k) {
      char* gk = g.gpu_base(l, k);
      for (int i = 0; i < g.num_blocks; ++i) {
        char* cpu = g.cpu_ptr + static_cast<int64_t>(l + g.start_layer) * g.cls + k * g.cks +
                    g.cids[i] * g.cbs + g.startoff;
        char* gpu = gk + g.gids[i] * g.gbs;
        if (h2d) {
          FKV_HIP(hipMemcpyAsync(gpu, cpu, g.chunk, hipMemcpyHostToDevice, stream));
        } else {
          FKV_HIP(hipMemcpyAsync(cpu, gpu, g.chunk, hipMemcpyDeviceToHost, stream));
        }
      }
    }
  }
  const int64_t copies = static_cast<int64_t>(g.num_layers) * g.kv * g.num_blocks;
  if ((rc = prof.end(stream, ev, copies * g.chunk, copies, true))) return rc;
  FKV_HIP(hipStreamSynchronize(stream));
  drain.armed = false;
  prof.flush();
  return 0;
}

// ---------------------------------------------------------------------------
// Asynchronous layer-grouped transfers.  A handle owns a pinned id buffer
// from the id pool (returned at release) and one event per group.  Live
// handles are registered, so a stale or released handle is refused and
// fkv_finalize can release the ones left.

}  // namespace

struct fkv_transfer_handle_s {
  int dev = 0;
  hipStream_t stream = nullptr;
  std::vector<hipEvent_t> done;   // per layer group, in order; groups of one launch share one
  std::vector<hipEvent_t> events; // the distinct events of `done`
  // the stream that records the groups' events is one the legacy null stream
  // waits for by itself (see fkv_handle_stream_wait)
  bool null_ordered = false;
  int null_upto = 0;              // groups the device's legacy null stream waits for (mu)
  IdBuf ids;
  DevIdLease dev_ids;             // copy-engine pipeline: the gpu ids of its scatters
  ProfRecorder prof;
  bool enqueued = false;          // every group was enqueued
  // Copy-engine pipeline: a driver thread queues each layer group's SDMA
  // copies into staging and, once they have landed, the group's scatter on
  // the lane's pipeline stream, then records done[g] there.  `recorded`
  // counts the events recorded so far; a caller that waits on a group (on
  // the host or through another stream) first waits for its event to exist.
  bool ce = false;
  std::thread driver;
  hipEvent_t start = nullptr;     // the caller's stream at the call
  std::mutex mu;
  std::condition_variable cv;
  int recorded = 0;
  int err = 0;
  std::string err_msg;
  int granularity = 1;
  Geometry geo;                   // points at the copies below
  std::vector<int64_t> gids, cids;
  std::vector<void*> ptrs;
};

namespace {

std::mutex g_handles_mu;
std::vector<fkv_transfer_handle_s*> g_handles;   // live handles

void handle_register(fkv_transfer_handle_s* h) {
  std::lock_guard<std::mutex> lk(g_handles_mu);
  g_handles.push_back(h);
}

// Removes h from the registry; false when it is not a live handle.
bool handle_unregister(fkv_transfer_handle_s* h) {
  std::lock_guard<std::mutex> lk(g_handles_mu);
  auto it = std::find(g_handles.begin(), g_handles.end(), h);
  if (it == g_handles.end()) return false;
  g_handles.erase(it);
  return true;
}

bool handle_live(fkv_transfer_handle_s* h) {
  std::lock_guard<std::mutex> lk(g_handles_mu);
  return std::find(g_handles.begin(), g_handles.end(), h) != g_handles.end();
}

// Whether `stream` is under HIP graph capture (or cannot tell).
bool stream_captured(hipStream_t stream) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (stream && hipStreamIsCapturing(stream, &cap) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return cap != hipStreamCaptureStatusNone;
}

// Whether the legacy null stream waits for work queued on `stream` by itself.
bool stream_blocks_null(hipStream_t stream) {
  unsigned flags = 0;
  if (stream && hipStreamGetFlags(stream, &flags) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return !(flags & hipStreamNonBlocking);
}

// Bytes a layer-wise launch of the zero-copy kernel aims for: groups smaller
// than this share launches, whose one event serves all of them.  Every launch
// costs about 8 us beyond its bytes' link time on the device (ramp, drain and
// the gap to the next) and 3-6 us on the host, so a 2 MiB handle of 32
// one-layer groups takes 349 us with a launch per group and 85 us in two.
// Launches grow from the minimum to the maximum and shrink towards the end
// (at most half of what is left), so the first groups arrive early and little
// compute is left when the last ones land.  Measured on MI355X, 80 MiB in 32
// groups of 2.5 MiB: 1877 us with a launch and a recorded event per group,
// 1771 us with the event on the kernel's packet, 1642 us with 4 MiB
// launches.
constexpr int64_t kLayerwiseMinLaunchBytes = int64_t(1) << 20;
constexpr int64_t kLayerwiseMaxLaunchBytes = int64_t(4) << 20;

int layerwise_enqueue(const Geometry& g, hipStream_t stream, int dev, int transfer_cus, bool h2d,
                      int granularity, fkv_transfer_handle_s* h) {
  DeviceState& d = g_dev[dev];
  int rc = ids_acquire(static_cast<size_t>(g.num_blocks) * 16, &h->ids);
  if (rc) return rc;
  pack_ids_into(g, h->ids.host);
  const int grid_cap = zero_copy_grid(g, d, transfer_cus, h2d);
  char* cpu_dev = g.cpu_info.dev_ptr + g.startoff + static_cast<int64_t>(g.start_layer) * g.cls;
  // Under capture the launches record plain events, as graph nodes.
  const bool captured = stream_captured(stream);
  // A launch's event rides on its kernel's packet, which costs 4% less than one
  // recorded behind it (80 MiB: 1579 / 1639 us).  The packet's end writes the
  // caches back before the event is seen: an SDMA engine, which does not look
  // into them, reads the group's bytes after a host wait, so a consumer on
  // another device or a network card may follow one as well.  Host-to-device
  // only: a device-to-host group's event has to release to the host.
  const bool on_kernel = h2d && !h->prof.on && !captured;
  h->null_ordered = !captured && stream_blocks_null(stream);
  const int ngroups = (g.num_layers + granularity - 1) / granularity;
  const int64_t group_bytes = static_cast<int64_t>(g.num_blocks) *
                              std::min(granularity, g.num_layers) * g.kv * g.chunk;
  const int64_t max_groups = std::max(1, g.layers_per_launch() / granularity);
  int64_t ramp = kLayerwiseMinLaunchBytes;
  for (int grp = 0; grp < ngroups;) {
    const int64_t left = static_cast<int64_t>(ngroups - grp) * group_bytes;
    const int64_t want = std::min({ramp, kLayerwiseMaxLaunchBytes,
                                   std::max(kLayerwiseMinLaunchBytes, left / 2)});
    ramp = std::min(2 * ramp, kLayerwiseMaxLaunchBytes);
    const int64_t take = std::min({std::max<int64_t>(1, (want + group_bytes / 2) / group_bytes),
                                   max_groups, static_cast<int64_t>(ngroups - grp)});
    const int gend = grp + static_cast<int>(take);
    const int lend = static_cast<int>(
        std::min<int64_t>(g.num_layers, static_cast<int64_t>(gend) * granularity));
    hipEvent_t ev = nullptr;
    FKV_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    h->events.push_back(ev);
    const int l0 = grp * granularity;
    hipEvent_t done = on_kernel ? ev : nullptr;
    rc = h2d ? launch_zero_copy<true>(g, h->ids, cpu_dev, l0, lend - l0, grid_cap, stream, h->prof,
                                      0, done)
             : launch_zero_copy<false>(g, h->ids, cpu_dev, l0, lend - l0, grid_cap, stream,
                                       h->prof);
    if (rc) return rc;
    if (!on_kernel) FKV_HIP(hipEventRecord(ev, stream));
    h->done.insert(h->done.end(), static_cast<size_t>(take), ev);
    grp = gend;
  }
  h->enqueued = true;
  return 0;
}

// Wait for everything the handle enqueued, then free it.  Safe on a handle
// whose enqueue failed part-way.
int handle_destroy(fkv_transfer_handle_s* h) {
  int rc = 0;
  if (h->driver.joinable()) h->driver.join();   // every event is recorded once it ends
  if (h->ce && h->err) rc = fail(h->err, "%s", h->err_msg.c_str());
  if (h->enqueued && !h->done.empty()) {
    hipError_t e = hipEventSynchronize(h->done.back());
    if (e != hipSuccess) rc = fail(static_cast<int>(e), "hipEventSynchronize: %s", hipGetErrorString(e));
  } else if (h->ids.host) {  // enqueue failed after taking ids: drain what was issued
    hipError_t e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) rc = fail(static_cast<int>(e), "hipStreamSynchronize: %s", hipGetErrorString(e));
  }
  h->prof.flush();
  for (hipEvent_t ev : h->events) (void)hipEventDestroy(ev);
  if (h->start) (void)hipEventDestroy(h->start);
  if (h->ids.host) ids_release(h->ids);
  delete h;
  return rc;
}

// Whether the copy-engine layer-wise pipeline takes this transfer: host to
// device from pinned host memory whose layer groups are contiguous per block
// (block-wise host rows), on a device whose engines work.  Anything else
// moves with the zero-copy kernel, as the synchronous path's policy would.
bool layerwise_ce_fits(const Geometry& g, int dev, bool h2d, int granularity) {
  if (!h2d || g.cpu_info.device || g_dev[dev].sdma_failed.load()) return false;
  const int nl = std::min(granularity, g.num_layers);
  return (g.kv == 1 || g.cks == g.chunk) && (nl == 1 || g.cls == g.kv * g.chunk);
}

// Smallest engine copy per block the copy-engine layer-wise pipeline aims for
// (bytes; FLEXKV_LAYERWISE_CE_MIN_COPY_BYTES), by carrying several layer
// groups in one window.  0 or 1: one group per window.
size_t layerwise_min_copy_bytes() {
  const char* e = getenv("FLEXKV_LAYERWISE_CE_MIN_COPY_BYTES");
  const long long v = e ? atoll(e) : static_cast<long long>(kLayerwiseCeMinCopyBytes);
  return v > 0 ? static_cast<size_t>(v) : 1;
}

// Smallest engine copy per block of a window, for handles of at least
// kLayerwiseShortMinBlocks blocks (with fewer, a window's copies take no longer
// than the host's round trip between windows).  A window takes one engine copy
// per block, about 0.75 us each over eight engines however short, so windows
// that grow from one layer group and shrink to one spend a layer-wise load of a
// tensor-parallel shard (8 KiB a block and layer) on copies of 8-64 KiB.
// Windows hold at least this much of a block, or as many groups as gpw allows
// (the last window: the groups left), and the groups before the first of them
// move with the zero-copy kernel, one event each.
//
// The last windows of short rows then hold many layers (16, 24, 16 and 9 of the
// shard's 80, against 2, 1 and 1), whose compute starts only after the load.
// That costs less than short copies do: measured on MI355X, us of the load
// alone and of a prefill that overlaps it, its compute about as long as the
// link's time (0.7-1.05 of it; 2.0 for 80 blocks), with windows from one group
// / 64 / 128 KiB a block, 128 KiB shrinking to one group at the end, and 128
// KiB with the last window's groups on the zero-copy kernel:
//   load alone (on the link)           one     64    128  shrink  kernel
//   Llama-3-8B, 256 blocks  (9419)   10750  10762  10463   10637   10299
//   70B TP-8, 3072 blocks  (35320)   63214  44635  40550   53349   38935
//     192 blocks            (2208)    4039   2982   2787    3597    2790
//     80 blocks              (920)    1746   1336   1312    1595    1326
//     8-bit, 1024 blocks    (5887)   17141   8598   7349   12924    6966
//   MLA, 477 blocks         (9409)   12670  10961  10386   11770   10383
//   Llama-3-8B, 4 tokens    (9198)   16811  12893  11577   14568   10586
//   overlapped prefill
//   Llama-3-8B, 256 blocks           12883  12941  12597   12563   12643
//   70B TP-8, 3072 blocks            63663  50644  49583   54765   51071
//     192 blocks                      4122   3251   3270    3672    3402
//     80 blocks                       2370   2179   2209    2213    2252
//     8-bit, 1024 blocks             17206   9359   9202   13017    9905
//   MLA, 477 blocks                  13644  12823  12502   12573   12529
//   Llama-3-8B, 4 tokens             17019  13179  12571   14954   12634
// With compute of 0.4 of the link's time 128 KiB is within 3% of the best.
constexpr size_t kLayerwiseShortCopyBytes = size_t(128) << 10;
constexpr int kLayerwiseShortMinBlocks = 64;

// Leading layer groups a copy-engine layer-wise handle moves with the
// zero-copy kernel before its engines start (FLEXKV_LAYERWISE_CE_KERNEL_GROUPS,
// default: the groups whose windows would be shorter than the shortest the
// engines get, `window` groups; at most all groups but one).  A one-group window
// is bound by the engines' per-copy cost (one copy per block of one group's
// rows), while a consumer waiting for the first group has nothing else to run, so
// the kernel's compute units cost it little then.
// Measured on MI355X at the Llama-3-8B shape with one layer per group, one
// kernel group brings the first group in after 1.3 ms instead of 2.1 ms and
// ends a prefill overlapped with 8 or 12 bf16 GEMMs per layer 1.1-1.7%
// sooner, but one with 4 GEMMs per layer, which the transfer outlasts,
// 0.5% later.
int layerwise_kernel_lead_groups(int ngroups, int window) {
  const char* e = getenv("FLEXKV_LAYERWISE_CE_KERNEL_GROUPS");
  const int v = e ? atoi(e) : window - 1;
  return std::max(0, std::min(v, ngroups - 1));
}

// The lane's pipeline stream: a stream with a full CU mask, so it has a
// hardware queue of its own and its scatters never wait behind compute
// kernels queued on a shared queue.
int pipeline_stream(CopyLane& ln, int dev, hipStream_t* out) {
  std::lock_guard<std::mutex> lk(ln.stream_mu);
  if (!ln.pipeline_stream) {
    DeviceGuard guard;
    int rc = guard.set(dev);
    if (rc) return rc;
    int ncu = 0;
    FKV_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    std::vector<uint32_t> mask(static_cast<size_t>((ncu + 31) / 32), 0u);
    for (int c = 0; c < ncu; ++c) mask[c / 32] |= 1u << (c % 32);
    FKV_HIP(hipExtStreamCreateWithCUMask(&ln.pipeline_stream, static_cast<uint32_t>(mask.size()),
                                         mask.data()));
  }
  *out = ln.pipeline_stream;
  return 0;
}

// Groups [first_group, end_group) of a copy-engine handle (all groups when
// end_group < 0) move host-to-device with the zero-copy kernel on the
// pipeline stream (the layer-wise kernel path's compute units), each group's
// event recorded after it: every group on a device whose engines cannot be
// set up, and the leading groups a handle moves before its engines start.
int layerwise_kernel_groups(fkv_transfer_handle_s* h, hipStream_t work, int first_group = 0,
                            int end_group = -1) {
  const Geometry& g = h->geo;
  DeviceState& d = g_dev[h->dev];
  const int grid_cap = zero_copy_grid(g, d, -1, true);
  char* cpu_dev = g.cpu_info.dev_ptr + g.startoff + static_cast<int64_t>(g.start_layer) * g.cls;
  const int end_layer = end_group < 0 ? g.num_layers
                                      : std::min(g.num_layers, end_group * h->granularity);
  int group = first_group;
  for (int g0 = first_group * h->granularity; g0 < end_layer; g0 += h->granularity, ++group) {
    const int gend = std::min(g.num_layers, g0 + h->granularity);
    int rc = launch_zero_copy<true>(g, h->ids, cpu_dev, g0, gend - g0, grid_cap, work, h->prof);
    if (rc) return rc;
    FKV_HIP(hipEventRecord(h->done[group], work));
    std::lock_guard<std::mutex> lk(h->mu);
    h->recorded = group + 1;
    h->cv.notify_all();
  }
  return 0;
}

// The driver's work: the leading group(s) with the zero-copy kernel (see
// layerwise_kernel_lead_groups), then the other layer groups in order, in
// windows cut into pieces of whole blocks that fit a staging half; SDMA copies
// (one per block: the window's rows are contiguous in block-wise host memory) on
// the wide engine set, double-buffered; each piece's scatter on the pipeline
// stream after a system-scope acquire; done[g] after the last piece of its
// window.  The host waits for a piece's scatter before reusing its half.
int layerwise_ce_run(fkv_transfer_handle_s* h, CopyLane& ln, hipStream_t work) {
  DeviceState& d = g_dev[h->dev];
  const Geometry& g = h->geo;
  DeviceGuard guard;
  int rc = guard.set(h->dev);
  if (rc) return rc;
  FKV_HIP(hipEventSynchronize(h->start));   // the caller's earlier work is done
  const int G = h->granularity;
  const size_t req = g_staging_request.load();
  const size_t half_default = (req ? req : kDefaultStagingBytes) / 2;
  const int nl_max = std::min({G, g.num_layers, g.layers_per_launch()});
  const size_t row_max = static_cast<size_t>(nl_max) * g.kv * g.chunk;
  // a half holds at least one block's row of one layer, so every window fits
  const size_t one_layer = static_cast<size_t>(g.kv) * g.chunk;
  rc = staging_or_fallback(d, h->dev, ln, std::max(std::min(row_max, half_default), one_layer));
  if (rc == kSdmaUnavailable) return layerwise_kernel_groups(h, work);
  if (rc) return rc;
  if ((rc = ensure_sdma(d, h->dev, ln.staging))) {
    // nothing has been queued yet: this handle, and every later copy-engine
    // transfer on the device, moves with the zero-copy kernel
    if (!d.sdma_failed.exchange(true))
      fprintf(stderr, "flexkv: copy engines unavailable on device %d (%s); copy-engine "
              "transfers use the zero-copy kernel\n", h->dev, last_error().c_str());
    last_error().clear();
    return layerwise_kernel_groups(h, work);
  }
  BusyMark busy(d.busy[1]);
  const size_t half = ln.staging_bytes / 2;
  struct Piece {
    int l0, nl, b0, nb, group;   // group: the last layer group the piece completes
    bool last;
  };
  // Consecutive groups share engine copies when a block's rows of several
  // layers are contiguous in host memory: a full window carries at least
  // layerwise_min_copy_bytes() per block, which the engines move faster than
  // one-group copies.  Every group's event is recorded when the window
  // holding it has landed.  Windows grow from the shortest (1, 2, 4, ... groups
  // where one group's rows are long enough), so the first group arrives early,
  // and near the end hold at most half of the groups left, but no fewer than the
  // shortest window: a consumer that keeps up has the last window's compute left
  // after the last transfer, which is one group's where the shortest window is
  // one group (see kLayerwiseShortCopyBytes for the others).
  const int lpl = g.layers_per_launch();
  const int ngroups = (g.num_layers + G - 1) / G;
  const size_t group_row = static_cast<size_t>(std::min(G, g.num_layers)) * g.kv * g.chunk;
  const size_t min_copy = layerwise_min_copy_bytes();
  int gpw = 1;   // groups per window
  if (G <= lpl && g.cls == static_cast<int64_t>(g.kv) * g.chunk) {
    gpw = static_cast<int>(std::max<size_t>(1, (min_copy + group_row - 1) / group_row));
    gpw = std::max(1, std::min(gpw, lpl / G));
    while (gpw > 1 && static_cast<size_t>(gpw) * group_row > half) --gpw;
  }
  // groups of the shortest window
  int window = 1;
  if (g.num_blocks >= kLayerwiseShortMinBlocks)
    window = static_cast<int>(std::min<size_t>(
        static_cast<size_t>(gpw), (kLayerwiseShortCopyBytes + group_row - 1) / group_row));
  // The leading groups move with the zero-copy kernel, alone on the link;
  // the engines start on the next group once they have landed.
  const int lead = layerwise_kernel_lead_groups(ngroups, window);
  std::vector<Piece> pieces;
  for (int grp = lead, ramp = window; grp < ngroups; ramp = std::min(2 * ramp, gpw)) {
    const int take = std::min({gpw, ramp, std::max(window, (ngroups - grp) / 2), ngroups - grp});
    const int l0 = grp * G;
    const int nl = std::min(take * G, g.num_layers - l0);
    grp += take;
    // a window moves in layer windows whose block rows fit a staging half
    // and whose layer pointers fit one launch's kernel arguments
    int win = std::min(nl, lpl);
    while (win > 1 && static_cast<size_t>(win) * g.kv * g.chunk > half) win = (win + 1) / 2;
    for (int w0 = l0; w0 < l0 + nl; w0 += win) {
      const int wn = std::min(win, l0 + nl - w0);
      const size_t row = static_cast<size_t>(wn) * g.kv * g.chunk;
      const int bpp = static_cast<int>(std::max<size_t>(1, half / row));
      for (int b0 = 0; b0 < g.num_blocks; b0 += bpp)
        pieces.push_back({w0, wn, b0, std::min(bpp, g.num_blocks - b0), grp - 1, false});
    }
    pieces.back().last = true;
  }
  const int np = static_cast<int>(pieces.size());
  std::vector<Run> runs;
  bool pending[2] = {false, false};
  int next_group = 0;   // the first group whose event is not yet recorded
  int64_t dma_copies = 0, dma_bytes = 0;
  const auto t0 = std::chrono::steady_clock::now();
  DrainOnError drain{work, &d, &ln};
  StageTable table;
  if (g.num_blocks > kPackInlineIds) {
    if ((rc = stage_table(h->ids, 2, g.num_blocks, h->dev, work, h->dev_ids))) return rc;
    table.gids = reinterpret_cast<int64_t*>(h->dev_ids.buf.dev);
  }
  auto queue_copies = [&](int pi) -> int {
    const Piece& p = pieces[pi];
    build_runs(g, p.b0, p.nb, p.l0, p.nl, false, false, runs);
    for (const Run& r : runs) dma_bytes += r.bytes;
    dma_copies += static_cast<int64_t>(runs.size());
    pending[pi & 1] = true;
    // Copies of one block's window are bound by the engines' per-copy cost,
    // so every window spreads over the wide engine set.
    return issue_sdma(d, ln, runs, ln.staging + (pi & 1) * half, true, pi & 1, d.cpu_agent,
                      kEnginesWide);
  };
  if (lead > 0) {
    if ((rc = layerwise_kernel_groups(h, work, 0, lead))) return rc;
    next_group = lead;
    // engine copies started beside the kernel share the link with it, and the
    // first group lands no earlier than with the engines alone
    FKV_HIP(hipEventSynchronize(h->done[lead - 1]));
  }
  for (int pi = 0; pi < std::min(np, 2); ++pi)
    if ((rc = queue_copies(pi))) return rc;
  for (int pi = 0; pi < np; ++pi) {
    const Piece& p = pieces[pi];
    const int hf = pi & 1;
    pending[hf] = false;
    // The host sleeps while the other half's copies keep the engines busy;
    // only the last wait, which nothing overlaps, spins (a wake from a sleep
    // costs 15-30 us).  Spinning throughout would hold a host core for the
    // whole transfer.
    if ((rc = sdma_wait(d, ln, hf, /*spin=*/pi + 1 == np))) return rc;
    hipLaunchKernelGGL(acquire_system_kernel, dim3(d.num_cus), dim3(64), 0, work);
    FKV_HIP(hipGetLastError());
    if ((rc = launch_staging<true>(g, table, ln.staging + hf * half, false, p.b0, p.nb, p.l0,
                                   p.nl, h->dev, work, h->prof)))
      return rc;
    if (p.last) {
      for (int gi = next_group; gi <= p.group; ++gi) FKV_HIP(hipEventRecord(h->done[gi], work));
      next_group = p.group + 1;
      std::lock_guard<std::mutex> lk(h->mu);
      h->recorded = next_group;
      h->cv.notify_all();
    }
    if (pi + 2 < np) {
      FKV_HIP(hipEventRecord(ln.ev_compute[hf], work));
      FKV_HIP(hipEventSynchronize(ln.ev_compute[hf]));
      if ((rc = queue_copies(pi + 2))) return rc;
    }
  }
  drain.armed = false;
  if (h->prof.on) {
    FKV_HIP(hipStreamSynchronize(work));
    prof_add_dma(std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0)
                     .count(),
                 dma_copies, dma_bytes);
  }
  return 0;
}

void layerwise_ce_drive(fkv_transfer_handle_s* h, hipStream_t work) {
  CopyLane& ln = g_dev[h->dev].lane[1];
  int rc = 0;
  std::string msg;
  {
    std::lock_guard<std::mutex> own(ln.mu);
    try {
      rc = layerwise_ce_run(h, ln, work);
    } catch (const std::exception& e) {
      rc = fail(static_cast<int>(hipErrorUnknown), "exception: %s", e.what());
    }
    if (rc) msg = last_error();
  }
  std::lock_guard<std::mutex> lk(h->mu);
  if (rc) {
    // every group's event is recorded even on failure, so no waiter blocks
    // for good; the handle reports the error
    h->err = rc;
    h->err_msg = msg;
    (void)hipSetDevice(h->dev);
    for (size_t gi = static_cast<size_t>(h->recorded); gi < h->done.size(); ++gi)
      (void)hipEventRecord(h->done[gi], work);
  }
  h->recorded = static_cast<int>(h->done.size());
  h->cv.notify_all();
}

// Set up the copy-engine pipeline of a handle and start its driver.  The
// caller's id lists and layer pointers are copied, since the driver reads
// them after the call returns.
int layerwise_ce_start(const Geometry& g, hipStream_t stream, int dev, int granularity,
                       fkv_transfer_handle_s* h) {
  h->ce = true;
  h->granularity = granularity;
  h->gids.assign(g.gids, g.gids + g.num_blocks);
  h->cids.assign(g.cids, g.cids + g.num_blocks);
  h->ptrs.assign(g.layer_ptrs, g.layer_ptrs + static_cast<int64_t>(g.num_layers) * g.ptrs_per_layer);
  h->geo = g;
  h->geo.gids = h->gids.data();
  h->geo.cids = h->cids.data();
  h->geo.layer_ptrs = h->ptrs.data();
  int rc = ids_acquire(static_cast<size_t>(g.num_blocks) * 16, &h->ids);
  if (rc) return rc;
  pack_ids_into(h->geo, h->ids.host);
  hipStream_t work = nullptr;
  if ((rc = pipeline_stream(g_dev[dev].lane[1], dev, &work))) return rc;
  h->null_ordered = stream_blocks_null(work);
  for (int g0 = 0; g0 < g.num_layers; g0 += granularity) {
    hipEvent_t ev = nullptr;
    FKV_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    h->done.push_back(ev);
    h->events.push_back(ev);
  }
  FKV_HIP(hipEventCreateWithFlags(&h->start, hipEventDisableTiming));
  FKV_HIP(hipEventRecord(h->start, stream));
  FKV_HIP(hipStreamWaitEvent(work, h->start, 0));
  h->driver = std::thread(layerwise_ce_drive, h, work);
  h->enqueued = true;
  return 0;
}

// A copy-engine handle's group g: wait until its event is recorded.  0, or
// the pipeline's error.
int ce_group_recorded(fkv_transfer_handle_s* h, int group) {
  std::unique_lock<std::mutex> lk(h->mu);
  h->cv.wait(lk, [&] { return h->recorded > group; });
  if (h->err) return fail(h->err, "%s", h->err_msg.c_str());
  return 0;
}

Geometry make_geometry(int num_blocks, int start_layer_id, int num_layers,
                       const int64_t* gpu_block_ids, void* const* gpu_layer_ptrs,
                       int64_t gpu_kv_stride_bytes, int64_t gpu_block_stride_bytes,
                       const int64_t* cpu_block_ids, void* cpu_ptr, int64_t cpu_kv_stride_bytes,
                       int64_t cpu_layer_stride_bytes, int64_t cpu_block_stride_bytes,
                       int64_t cpu_startoff_inside_chunks, int64_t chunk_size_bytes, int is_mla) {
  Geometry g;
  g.num_blocks = num_blocks;
  g.start_layer = start_layer_id;
  g.num_layers = num_layers;
  g.kv = is_mla ? 1 : 2;
  g.gids = gpu_block_ids;
  g.cids = cpu_block_ids;
  g.layer_ptrs = gpu_layer_ptrs;
  g.gks = gpu_kv_stride_bytes;
  g.gbs = gpu_block_stride_bytes;
  g.cks = cpu_kv_stride_bytes;
  g.cls = cpu_layer_stride_bytes;
  g.cbs = cpu_block_stride_bytes;
  g.startoff = cpu_startoff_inside_chunks;
  g.chunk = chunk_size_bytes;
  g.cpu_ptr = static_cast<char*>(cpu_ptr);
  return g;
}

// Copy-engine mode hands a transfer to the SDMA engines only when the
// engines pay off: the op moves at least ce_min_bytes() (default 32 MiB)
// and each engine copy moves at least 128 KiB: a contiguous host run, or one
// block's layer window as a rect copy when the host layout puts its chunks at
// one stride (layer-wise).  Each engine copy costs about 6 us and the
// host-side ordering about 40 us per call (MI355X: a 1 MiB op of 64 KiB runs
// takes 77 us on the engines, 39 us in the zero-copy kernel); smaller or
// finer-grained transfers, and caches in device memory, go to the zero-copy
// kernel, with identical results.
//
// A layer-wise host cache whose ids do not come in runs long enough for
// layer-major staging needs one rect copy per block, and the runtime runs
// every rect copy on a single engine per direction: 46.8 / 47.0 GB/s
// (D2H / H2D) at the Llama-3-8B shape, 82% of the link, against 56.5 /
// 57.2 GB/s for the zero-copy kernel.  Such transfers therefore move with
// the zero-copy kernel, which holds compute units for the whole transfer
// (bf16 GEMMs beside it take 1.4 times as long in either order, and 1.02 times
// beside the rect copies); fkv_set_copy_engine_policy (or
// FLEXKV_CE_RECT_COPIES=1) keeps them on the engines.
bool ce_pays_off(const Geometry& g, bool h2d) {
  // a "host" cache that is device memory has no PCIe copy to offload
  if (g.cpu_info.device) return false;
  const int64_t min_bytes = ce_min_bytes();
  const int64_t total = op_bytes(g);
  const bool row_contig = (g.kv == 1 || g.cks == g.chunk) &&
                          (g.num_layers == 1 || g.cls == g.kv * g.chunk);
  const int64_t row = static_cast<int64_t>(g.num_layers) * g.kv * g.chunk;
  const bool rect = !row_contig && host_slice_pitch(g, g.num_layers) > 0;
  if (rect && !layer_major_pays_off(g, layer_run_bytes(h2d)) && !ce_rect_copies()) return false;
  const int64_t run = (row_contig || rect) ? row : g.chunk;
  return total >= min_bytes && (min_bytes == 0 || run >= kCeMinRunBytes);
}

// Validate, then run one synchronous transfer in the requested mode.
// Copy-engine mode copies exact bytes for any geometry, as the reference's
// CE loop does (csrc/transfer.cu:97-121): a chunk size, stride, offset or
// pointer that is not a multiple of 16 bytes, which the kernels' 16-byte
// accesses cannot take, sends the transfer to the per-chunk engine loop.
int transfer_entry(Geometry& g, hipStream_t s, int transfer_cus, bool h2d, int mode) {
  if (mode == FKV_XFER_CE && !geometry_vec16(g)) mode = FKV_XFER_CE_PER_CHUNK;
  int rc = validate(g, mode);
  if (rc) return rc;
  int dev = 0;
  if ((rc = stream_device(s, &dev))) return rc;
  if ((rc = ensure_device_basics(dev))) return rc;
  switch (mode) {
    case FKV_XFER_KERNEL:
      return transfer_zero_copy(g, s, dev, transfer_cus, h2d);
    case FKV_XFER_CE:
      if (!ce_pays_off(g, h2d) || g_dev[dev].sdma_failed.load())
        return transfer_zero_copy(g, s, dev, transfer_cus, h2d);
      rc = transfer_staged(g, s, dev, h2d);
      return rc == kSdmaUnavailable ? transfer_zero_copy(g, s, dev, transfer_cus, h2d) : rc;
    default:
      return transfer_ce_per_chunk(g, s, h2d);
  }
}
}  // namespace

extern "C" {

int fkv_transfer_kv_blocks(int num_blocks, int start_layer_id, int num_layers,
                           const int64_t* gpu_block_ids, void* const* gpu_layer_ptrs,
                           int64_t gpu_kv_stride_bytes, int64_t gpu_block_stride_bytes,
                           const int64_t* cpu_block_ids, void* cpu_ptr,
                           int64_t cpu_kv_stride_bytes, int64_t cpu_layer_stride_bytes,
                           int64_t cpu_block_stride_bytes, int64_t cpu_startoff_inside_chunks,
                           int64_t chunk_size_bytes, fkv_stream_t stream, int transfer_cus,
                           int is_host_to_device, int use_ce_transfer, int is_mla) {
  try {
    last_error().clear();
    last_unsafe_host_blocks().clear();
    if (use_ce_transfer < FKV_XFER_KERNEL || use_ce_transfer > FKV_XFER_CE_PER_CHUNK)
      return fail(kInval, "use_ce_transfer must be 0 (kernel), 1 (CE) or 2 (CE per chunk), got %d",
                  use_ce_transfer);
    if (num_blocks == 0 || num_layers == 0) return 0;
    Geometry g = make_geometry(num_blocks, start_layer_id, num_layers, gpu_block_ids,
                               gpu_layer_ptrs, gpu_kv_stride_bytes, gpu_block_stride_bytes,
                               cpu_block_ids, cpu_ptr, cpu_kv_stride_bytes,
                               cpu_layer_stride_bytes, cpu_block_stride_bytes,
                               cpu_startoff_inside_chunks, chunk_size_bytes, is_mla);
    return transfer_entry(g, static_cast<hipStream_t>(stream), transfer_cus,
                          is_host_to_device != 0, use_ce_transfer);
  } catch (const std::exception& e) {
    return fail(static_cast<int>(hipErrorUnknown), "exception: %s", e.what());
  } catch (...) {
    return fail(static_cast<int>(hipErrorUnknown), "unknown exception");
  }
}

int fkv_transfer_kv_blocks_kv_ptrs(int num_blocks, int start_layer_id, int num_layers,
                                   const int64_t* gpu_block_ids, void* const* gpu_kv_ptrs,
                                   int64_t gpu_block_stride_bytes, const int64_t* cpu_block_ids,
                                   void* cpu_ptr, int64_t cpu_kv_stride_bytes,
                                   int64_t cpu_layer_stride_bytes, int64_t cpu_block_stride_bytes,
                                   int64_t cpu_startoff_inside_chunks, int64_t chunk_size_bytes,
                                   fkv_stream_t stream, int transfer_cus, int is_host_to_device,
                                   int use_ce_transfer, int is_mla) {
  try {
    last_error().clear();
    last_unsafe_host_blocks().clear();
    if (use_ce_transfer < FKV_XFER_KERNEL || use_ce_transfer > FKV_XFER_CE_PER_CHUNK)
      return fail(kInval, "use_ce_transfer must be 0 (kernel), 1 (CE) or 2 (CE per chunk), got %d",
                  use_ce_transfer);
    if (num_blocks == 0 || num_layers == 0) return 0;
    Geometry g = make_geometry(num_blocks, start_layer_id, num_layers, gpu_block_ids, gpu_kv_ptrs,
                               0, gpu_block_stride_bytes, cpu_block_ids, cpu_ptr,
                               cpu_kv_stride_bytes, cpu_layer_stride_bytes, cpu_block_stride_bytes,
                               cpu_startoff_inside_chunks, chunk_size_bytes, is_mla);
    g.ptrs_per_layer = g.kv;
    return transfer_entry(g, static_cast<hipStream_t>(stream), transfer_cus,
                          is_host_to_device != 0, use_ce_transfer);
  } catch (const std::exception& e) {
    return fail(static_cast<int>(hipErrorUnknown), "exception: %s", e.what());
  } catch (...) {
    return fail(static_cast<int>(hipErrorUnknown), "unknown exception");
  }
}

int fkv_transfer_kv_blocks_noalloc(int num_blocks, int start_layer_id, int num_layers,
                                   const int64_t* gpu_block_ids, void* const* gpu_layer_ptrs,
                                   int64_t gpu_kv_stride_bytes, int64_t gpu_block_stride_bytes,
                                   const int64_t* cpu_block_ids, void* cpu_ptr,
                                   int64_t cpu_kv_stride_bytes, int64_t cpu_layer_stride_bytes,
                                   int64_t cpu_block_stride_bytes,
                                   int64_t cpu_startoff_inside_chunks, int64_t chunk_size_bytes,
                                   fkv_stream_t stream, int transfer_cus, int is_host_to_device,
                                   int is_mla) {
  try {
    last_error().clear();
    last_unsafe_host_blocks().clear();
    if (num_blocks == 0 || num_layers == 0) return 0;
    Geometry g = make_geometry(num_blocks, start_layer_id, num_layers, gpu_block_ids,
                               gpu_layer_ptrs, gpu_kv_stride_bytes, gpu_block_stride_bytes,
                               cpu_block_ids, cpu_ptr, cpu_kv_stride_bytes,
                               cpu_layer_stride_bytes, cpu_block_stride_bytes,
                               cpu_startoff_inside_chunks, chunk_size_bytes, is_mla);
    hipStream_t s = static_cast<hipStream_t>(stream);
    // The call is synchronous and resolves its ids and addresses on the host
    // while it runs, so a captured call could not replay: refuse capture
    // before anything reaches the stream (the null stream is never captured).
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (s) FKV_HIP(hipStreamIsCapturing(s, &cap));
    if (cap != hipStreamCaptureStatusNone)
      return fail(static_cast<int>(hipErrorStreamCaptureUnsupported),
                  "fkv_transfer_kv_blocks_noalloc cannot run on a stream under HIP graph "
                  "capture (it synchronises the stream and stages ids from host memory)");
    int rc = validate(g, FKV_XFER_KERNEL);
    if (rc) return rc;
    int dev = 0;
    if ((rc = stream_device(s, &dev))) return rc;
    if ((rc = ensure_device_basics(dev))) return rc;
    return transfer_zero_copy_noalloc(g, s, dev, transfer_cus, is_host_to_device != 0);
  } catch (const std::exception& e) {
    return fail(static_cast<int>(hipErrorUnknown), "exception: %s", e.what());
  } catch (...) {
    return fail(static_cast<int>(hipErrorUnknown), "unknown exception");
  }
}

int fkv_gather_kv_blocks(int num_blocks, int num_layers, const int64_t* gpu_block_ids,
                         void* const* gpu_layer_ptrs, int64_t gpu_kv_stride_bytes,
                         int64_t gpu_block_stride_bytes, int64_t chunk_size_bytes, void* buffer,
                         size_t buffer_bytes, fkv_stream_t stream, int is_mla) {
  return contiguous_entry(num_blocks, num_layers, gpu_block_ids, gpu_layer_ptrs,
                          gpu_kv_stride_bytes, gpu_block_stride_bytes, chunk_size_bytes, buffer,
                          buffer_bytes, stream, is_mla, false);
}

int fkv_scatter_kv_blocks(int num_blocks, int num_layers, const int64_t* gpu_block_ids,
                          void* const* gpu_layer_ptrs, int64_t gpu_kv_stride_bytes,
                          int64_t gpu_block_stride_bytes, int64_t chunk_size_bytes,
                          const void* buffer, size_t buffer_bytes, fkv_stream_t stream,
                          int is_mla) {
  return contiguous_entry(num_blocks, num_layers, gpu_block_ids, gpu_layer_ptrs,
                          gpu_kv_stride_bytes, gpu_block_stride_bytes, chunk_size_bytes,
                          const_cast<void*>(buffer), buffer_bytes, stream, is_mla, true);
}

int fkv_transfer_kv_blocks_layerwise(
    int num_blocks, int start_layer_id, int num_layers, int layer_granularity,
    const int64_t* gpu_block_ids, void* const* gpu_layer_ptrs, int64_t gpu_kv_stride_bytes,
    int64_t gpu_block_stride_bytes, const int64_t* cpu_block_ids, void* cpu_ptr,
    int64_t cpu_kv_stride_bytes, int64_t cpu_layer_stride_bytes, int64_t cpu_block_stride_bytes,
    int64_t cpu_startoff_inside_chunks, int64_t chunk_size_bytes, fkv_stream_t stream,
    int transfer_cus, int is_host_to_device, int use_ce_transfer, int is_mla,
    fkv_transfer_handle* out) {
  try {
    last_error().clear();
    last_unsafe_host_blocks().clear();
    if (!out) return fail(kInval, "out handle pointer is null");
    if (use_ce_transfer != FKV_XFER_KERNEL && use_ce_transfer != FKV_XFER_CE)
      return fail(kInval, "use_ce_transfer must be 0 (kernel) or 1 (copy engines), got %d",
                  use_ce_transfer);
    *out = nullptr;
    if (layer_granularity < 1) return fail(kInval, "layer_granularity must be >= 1");
    if (num_blocks < 0 || num_layers < 0)
      return fail(kInval, "negative count: num_blocks=%d num_layers=%d", num_blocks, num_layers);
    Geometry g = make_geometry(num_blocks, start_layer_id, num_layers, gpu_block_ids,
                               gpu_layer_ptrs, gpu_kv_stride_bytes, gpu_block_stride_bytes,
                               cpu_block_ids, cpu_ptr, cpu_kv_stride_bytes,
                               cpu_layer_stride_bytes, cpu_block_stride_bytes,
                               cpu_startoff_inside_chunks, chunk_size_bytes, is_mla);
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto* h = new fkv_transfer_handle_s();
    h->stream = s;
    int rc = 0;
    if (num_blocks > 0 && num_layers > 0) {
      const bool h2d = is_host_to_device != 0;
      if ((rc = validate(g, FKV_XFER_KERNEL)) || (rc = stream_device(s, &h->dev)) ||
          (rc = ensure_device_basics(h->dev)) ||
          (rc = (use_ce_transfer == FKV_XFER_CE &&
                 layerwise_ce_fits(g, h->dev, h2d, layer_granularity))
                    ? layerwise_ce_start(g, s, h->dev, layer_granularity, h)
                    : layerwise_enqueue(g, s, h->dev, transfer_cus, h2d, layer_granularity, h))) {
        const std::string msg = last_error();
        (void)handle_destroy(h);
        last_error() = msg;
        return rc;
      }
    }
    handle_register(h);
    *out = h;
    return 0;
  } catch (const std::exception& e) {
    return fail(static_cast<int>(hipErrorUnknown), "exception: %s", e.what());
  } catch (...) {
    return fail(static_cast<int>(hipErrorUnknown), "unknown exception");
  }
}

int fkv_handle_num_groups(fkv_transfer_handle h) {
  last_error().clear();
  if (!h || !handle_live(h)) return fail(-1, "null, released or unknown handle");
  return static_cast<int>(h->done.size());
}

int fkv_handle_query(fkv_transfer_handle h, int group) {
  last_error().clear();
  if (!h || !handle_live(h) || group < 0 || group >= static_cast<int>(h->done.size()))
    return fail(-1, "bad handle or group %d", group);
  if (h->ce) {
    std::lock_guard<std::mutex> lk(h->mu);
    if (h->recorded <= group) return 0;
    if (h->err) return fail(-h->err, "%s", h->err_msg.c_str());
  }
  hipError_t e = hipEventQuery(h->done[group]);
  if (e == hipSuccess) return 1;
  (void)hipGetLastError();
  if (e == hipErrorNotReady) return 0;
  return fail(-static_cast<int>(e), "hipEventQuery: %s", hipGetErrorString(e));
}

int fkv_handle_wait(fkv_transfer_handle h, int group) {
  last_error().clear();
  if (!h || !handle_live(h) || group < 0 || group >= static_cast<int>(h->done.size()))
    return fail(kInval, "bad handle or group %d", group);
  if (h->ce) {
    const int rc = ce_group_recorded(h, group);
    if (rc) return rc;
  }
  FKV_HIP(hipEventSynchronize(h->done[group]));
  return 0;
}

int fkv_handle_stream_wait(fkv_transfer_handle h, int group, fkv_stream_t other) {
  last_error().clear();
  if (!h || !handle_live(h) || group < 0 || group >= static_cast<int>(h->done.size()))
    return fail(kInval, "bad handle or group %d", group);
  if (h->ce) {
    // the group's event exists once its copies have landed and its scatter
    // is queued; only then can another stream wait on it
    const int rc = ce_group_recorded(h, group);
    if (rc) return rc;
  }
  // The legacy null stream waits by itself for all work already queued on the
  // device's blocking streams, and every operation on it pays for that (about
  // 14 us of host time and 11 us of the stream's while a transfer runs).  So
  // one wait on it covers every group already queued on a blocking stream,
  // and later waits of the handle for those groups add nothing: 32 of them
  // beside an 80 MiB transfer made its pass 2.2 ms instead of 1.8 ms.
  hipStream_t st = static_cast<hipStream_t>(other);
  int cur = -1;
  if (!st) FKV_HIP(hipGetDevice(&cur));
  if (!st && cur == h->dev) {
    std::lock_guard<std::mutex> lk(h->mu);
    if (group < h->null_upto) return 0;
    const int queued = h->ce ? h->recorded : static_cast<int>(h->done.size());
    const int covers = null_wait_covers(h->done, group, queued, h->null_ordered);
    FKV_HIP(hipStreamWaitEvent(st, h->done[group], 0));
    h->null_upto = std::max(h->null_upto, covers);
    return 0;
  }
  FKV_HIP(hipStreamWaitEvent(st, h->done[group], 0));
  return 0;
}

int fkv_handle_release(fkv_transfer_handle h) {
  last_error().clear();
  if (!h) return 0;
  if (!handle_unregister(h)) return fail(kInval, "handle %p is released or unknown", (void*)h);
  return handle_destroy(h);
}

int fkv_set_copy_engine_policy(int64_t min_bytes, int rect_copies) {
  last_error().clear();
  if (min_bytes < -2)
    return fail(kInval, "min_bytes must be >= 0, -1 to unset or -2 to keep, got %lld",
                static_cast<long long>(min_bytes));
  if (rect_copies < -2 || rect_copies > 1)
    return fail(kInval, "rect_copies must be 0, 1, -1 to unset or -2 to keep, got %d",
                rect_copies);
  if (min_bytes != -2) g_ce_min_bytes.store(min_bytes);
  if (rect_copies != -2) g_ce_rect_copies.store(rect_copies);
  return 0;
}

int fkv_get_copy_engine_policy(int64_t* min_bytes, int* rect_copies) {
  last_error().clear();
  if (!min_bytes || !rect_copies) return fail(kInval, "null output pointer");
  *min_bytes = ce_min_bytes();
  *rect_copies = ce_rect_copies() ? 1 : 0;
  return 0;
}

int fkv_prepare(int device) {
  try {
    last_error().clear();
    int dev = device;
    if (dev < 0) FKV_HIP(hipGetDevice(&dev));
    int count = 0;
    FKV_HIP(hipGetDeviceCount(&count));
    if (dev >= count || dev >= kMaxDevices)
      return fail(kInval, "device %d out of range (%d devices)", dev, count);
    DeviceGuard guard;
    int rc = guard.set(dev);
    if (rc) return rc;
    if ((rc = ensure_device_basics(dev))) return rc;
    // the library's code object is loaded with its first kernel launch
    hipLaunchKernelGGL(acquire_system_kernel, dim3(1), dim3(64), 0, nullptr);
    FKV_HIP(hipGetLastError());
    FKV_HIP(hipStreamSynchronize(nullptr));
    DeviceState& d = g_dev[dev];
    if (d.sdma_failed.load()) return 0;   // copy-engine transfers use the zero-copy kernel
    IdLease host;
    if ((rc = ids_acquire(kPrepareHostBytes, &host.buf))) return rc;
    for (int dir = 0; dir < 2; ++dir) {
      CopyLane& ln = d.lane[dir];
      std::lock_guard<std::mutex> lk(ln.mu);
      rc = staging_or_fallback(d, dev, ln, 0);
      if (rc == kSdmaUnavailable) return 0;   // no memory for staging: the transfer falls back
      if (rc) return rc;
      if ((rc = ensure_sdma(d, dev, ln.staging))) {
        if (!d.sdma_failed.exchange(true))
          fprintf(stderr, "flexkv: copy engines unavailable on device %d (%s); copy-engine "
                  "transfers use the zero-copy kernel\n", dev, last_error().c_str());
        last_error().clear();
        return 0;
      }
      if ((rc = sdma_prepare_lane(d, ln, dir == 1, kPrepareSignalsPerHalf,
                                  reinterpret_cast<char*>(host.buf.host), kPrepareHostBytes)))
        return rc;
    }
    // the stream of the copy-engine layer-wise pipeline's scatters
    hipStream_t work = nullptr;
    return pipeline_stream(d.lane[1], dev, &work);
  } catch (const std::exception& e) {
    return fail(static_cast<int>(hipErrorUnknown), "exception: %s", e.what());
  } catch (...) {
    return fail(static_cast<int>(hipErrorUnknown), "unknown exception");
  }
}

int fkv_finalize(void) {
  try {
    last_error().clear();
    int rc = 0;
    auto keep = [&rc](int r) {
      if (r && !rc) rc = r;
    };
    // 1. layer-wise handles the caller never released: wait for their groups
    std::vector<fkv_transfer_handle_s*> handles;
    {
      std::lock_guard<std::mutex> lk(g_handles_mu);
      handles.swap(g_handles);
    }
    for (fkv_transfer_handle_s* h : handles) keep(handle_destroy(h));
    // TP groups: their rank threads and streams
    keep(tp_groups_destroy_all());
    // 2. streams made by fkv_stream_create (each is synchronised first)
    keep(streams_destroy_all());
    // 3. copy-engine lanes: queued copies, signals, events, staging
    for (int dev = 0; dev < kMaxDevices; ++dev) {
      DeviceState& d = g_dev[dev];
      for (CopyLane& ln : d.lane) {
        std::lock_guard<std::mutex> lk(ln.mu);
        const bool used = ln.staging || ln.ev_compute[0] || ln.ev_compute[1] ||
                          ln.pipeline_stream ||
                          !ln.polled_pool[0].empty() || !ln.irq_pool[0].empty() ||
                          !ln.polled_pool[1].empty() || !ln.irq_pool[1].empty();
        if (!used) continue;
        DeviceGuard guard;
        const int r = guard.set(dev);
        if (r) {
          keep(r);
          continue;
        }
        keep(lane_release(d, ln));
      }
    }
    // 4. pinned and device id buffers
    keep(ids_pool_free());
    keep(dev_ids_pool_free());
    return rc;
  } catch (const std::exception& e) {
    return fail(static_cast<int>(hipErrorUnknown), "exception: %s", e.what());
  } catch (...) {
    return fail(static_cast<int>(hipErrorUnknown), "unknown exception");
  }
}


}  // extern "C"
