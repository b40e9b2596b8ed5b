// gfx950 copy kernels of the KV block transfer path.
//
// All of them are pure byte movers bounded by HBM (device <-> device staging)
// or by the host link (device <-> mapped pinned host memory).  Shape:
//   * a workgroup is 256 lanes = 4 wavefronts of 64;
//   * a tile is 256 lanes x U x 16 bytes; every lane issues its U 16-byte
//     loads before the first store so U global_load_dwordx4 are in flight per
//     lane, and consecutive lanes touch consecutive 16-byte words, so each
//     wavefront's access is one 1 KiB contiguous burst;
//   * loads are non-temporal and stores "sc1 nt": the data is touched once (but see
//     copy_tile_in_hbm);
//   * all per-tile address arithmetic is wave-uniform (scalar registers), except
//     for units cut into chunks (block_chunks_unit).
#include "pf_kernels.hpp"

#include <hip/hip_ext.h>

#include <mutex>
#include <type_traits>

#include "pf_chunks.hpp"
#include "pf_common.hpp"

namespace pf {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
// Address-space-1 (global) views, so the compiler emits global_load/store
// instead of flat accesses for addresses that arrive as integers.
typedef __attribute__((address_space(1))) u32x4 g_u32x4;
typedef __attribute__((address_space(1))) unsigned char g_u8;
// 16 bytes at any address: the target allows unaligned global accesses, so
// these are one global_load_dwordx4 / global_store_dwordx4 all the same.
typedef u32x4 u32x4_any __attribute__((aligned(1)));
typedef __attribute__((address_space(1))) u32x4_any g_u32x4_any;
// Address-space-4 (constant) views for the read-only, wave-uniform id list
// and page table: uniform constant loads become scalar loads.
typedef __attribute__((address_space(4))) const uint32_t c_u32;
typedef __attribute__((address_space(4))) const uint64_t c_u64;
typedef __attribute__((address_space(4))) const BlockUnit c_unit;
typedef __attribute__((address_space(4))) const pf_copy_desc c_desc;

constexpr int kLanes = 256;
constexpr int kWave = 64;
constexpr uint32_t kMaxRowUnits = kRowsLaunchUnits;  // units of one block_tiles_rows_kernel launch

// 16-byte store with the cache policy "sc1 nt".  Measured on MI355X at the
// Llama shape (5000 x 2 x 32 KiB gathered or scattered per launch) over all 49
// load x store policy pairs: a destination written in ascending address order
// is written fastest with "sc1 nt" (gather 6.35 TB/s against 6.30 for plain
// nt; scatter in ascending-id row order 6.17 against 5.63 for "sc1" and 5.44
// for an ordinary store).  Stores into mapped host memory want the same: every
// policy with sc1 moves the Llama layer over the link at 56.3 GB/s (64
// workgroups; hipMemcpyAsync on the same box 56.1), plain and sc0 stores at
// 54.2, nt alone at 53.9; loads from host memory do not care (56.6 with any
// policy).
//
// The policy bits are not reachable from a plain C++ store, and the store must
// not be inline assembly: the compiler cannot see that an asm statement is a
// 16-byte store, so it neither keeps the data registers alive for the wait
// states such a store needs nor counts it for s_waitcnt.  (With the store
// written as asm, a four-store tile loop had the address of the fourth store
// computed into the data registers of the first two instructions after that
// one was issued, and the first store wrote address bits into lanes 12-15 of
// every 16-lane row.)  A raw buffer store carries the bits in its `aux`
// operand and is an ordinary instruction to the compiler.  The descriptor
// covers exactly the tile (wave-uniform base and byte count, no stride), so a
// store beyond the tile would be dropped by the hardware's range check.
constexpr int kAuxSc1Nt = (1 << 4) | (1 << 1);  // gfx940+: bit 4 = sc1, bit 1 = nt
constexpr int kRawBufferWord3 = 0x00020000;     // untyped 32-bit data, no swizzle, no tid

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_descriptor(uint64_t base, uint32_t bytes) {
  // The base is wave-uniform by construction; say so, or the compiler would
  // loop over the lanes to build one descriptor per distinct value.
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo), 0,
      static_cast<int>(__builtin_amdgcn_readfirstlane(bytes)), kRawBufferWord3);
}

__device__ __forceinline__ void store16_sc1_nt(__amdgpu_buffer_rsrc_t tile, uint32_t offset,
                                               u32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(v, tile, static_cast<int>(offset), 0, kAuxSc1Nt);
}

// Wait for the loads of a tile.  Where a store may be skipped, the compiler takes
// the load of its value to be open from then on, and starts the next tile (or
// unit) by waiting for everything in flight, the stores of this one included
// (a link trip per unit: 72 x 2 fragments of 12 096 bytes of two layers saved in
// 66.3 us instead of 64.5).  For saves: the stores of a load go to HBM, where
// letting the first of them out before the last load is back is worth more
// (fragments of 1000 bytes loaded at 55.1 GB/s, with this wait at 53.0).
__device__ __forceinline__ void wait_for_loads() {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt 0; expcnt and lgkmcnt as they are
}

// Run body(std::integral_constant<int, n>) for the wave-uniform n in 1..MAX,
// nothing for 0.  A tile that is not full is moved by the straight-line body of
// as many steps as the wavefront has work for.  A guard on every step instead
// (`if (i < n) v[k] = load`) costs the tile its overlap: the value of a guarded
// load is merged with what the register held before, and the compiler waits for
// each load at the merge.
template <int MAX, typename Body>
__device__ __forceinline__ void with_steps(uint32_t n, Body body) {
  if constexpr (MAX > 0) {
    if (n == MAX) {
      body(std::integral_constant<int, MAX>{});
    } else {
      with_steps<MAX - 1>(n, body);
    }
  }
}
// Steps of LANES items that the wavefront of `lane` has of n items.  All steps
// but the last are full.
template <int LANES>
__device__ __forceinline__ uint32_t wave_steps(uint32_t n, uint32_t lane) {
  const uint32_t first = __builtin_amdgcn_readfirstlane(lane);
  return first < n ? (n - first + LANES - 1) / LANES : 0u;
}

// Copy `bytes` <= U*LANES*16 from src to dst, both 16-byte aligned, by the LANES
// lanes (whole wavefronts) whose index is `lane`.
template <int U, int LANES>
__device__ __forceinline__ void copy_tile_vec(uint64_t dst, uint64_t src, uint32_t bytes,
                                              uint32_t lane) {
  constexpr uint32_t kTile = U * LANES * 16;
  const g_u32x4* __restrict__ s = reinterpret_cast<const g_u32x4*>(src);
  const __amdgpu_buffer_rsrc_t tile = tile_descriptor(dst, bytes & ~15u);
  if (bytes == kTile) {
    u32x4 v[U];
#pragma unroll
    for (int k = 0; k < U; ++k) v[k] = __builtin_nontemporal_load(s + lane + k * LANES);
#pragma unroll
    for (int k = 0; k < U; ++k) store16_sc1_nt(tile, (lane + k * LANES) * 16u, v[k]);
    return;
  }
  const uint32_t nvec = bytes >> 4;
  with_steps<U>(wave_steps<LANES>(nvec, lane), [&](auto steps) {
    constexpr int K = decltype(steps)::value;
    u32x4 v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const uint32_t idx = lane + k * LANES;
      v[k] = __builtin_nontemporal_load(s + (k + 1 < K || idx < nvec ? idx : nvec - 1));
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      // Lanes past the tile's end: dropped by the descriptor's range check.
      store16_sc1_nt(tile, (lane + k * LANES) * 16u, v[k]);
    }
  });
  // Fewer than 16 trailing bytes (fragment size not a multiple of 16).
  const uint32_t j = (nvec << 4) + lane;
  if (j < bytes) {
    reinterpret_cast<g_u8*>(dst)[j] = reinterpret_cast<const g_u8*>(src)[j];
  }
}

// Fragments that do not start on 16-byte boundaries are cut into 16-byte chunks
// whose starts are aligned on ONE side (the link side where there is one: `mis`
// is that side's address modulo 16) and unaligned on the other (chunk_start).
// Measured on MI355X against words or, off the 4-byte grid, single bytes (one
// load in flight per lane), descriptors over the link, 31 MB out and back:
// 4097-byte fragments 3248 -> 1220 us, 12345 bytes 5932 -> 1190, 100001 bytes
// 11717 -> 1230.
__device__ __forceinline__ u32x4 load16_any(uint64_t addr) {
  return __builtin_nontemporal_load(reinterpret_cast<const g_u32x4_any*>(addr));
}
__device__ __forceinline__ void store16_any(uint64_t addr, u32x4 v) {
  __builtin_nontemporal_store(v, reinterpret_cast<g_u32x4_any*>(addr));
}

// Copy `bytes` <= U*LANES*16 with no alignment assumption, by the LANES lanes
// whose index is `lane`; chunks are aligned on the destination or, with
// ALIGN_SRC, on the source.
template <int U, int LANES, bool ALIGN_SRC, bool IN_HBM = false>
__device__ __forceinline__ void copy_tile_any(uint64_t dst, uint64_t src, uint32_t bytes,
                                              uint32_t lane) {
  if (bytes < 16) {
    if (lane < bytes) reinterpret_cast<g_u8*>(dst)[lane] = reinterpret_cast<const g_u8*>(src)[lane];
    return;
  }
  const uint32_t mis = static_cast<uint32_t>(ALIGN_SRC ? src : dst) & 15u;
  const uint32_t n = chunk_count(bytes, mis);
  // A short row is one trip there and back, of which the choice of a body and of a
  // store policy below are a measurable part (48 rows of 24 bytes out and back
  // 25.8 us, this way 23.7; 1500 bytes 26.0 and 24.3).  From 188 chunks on the
  // body below is the faster one again (7000 rows of 3000 bytes 884 against 908).
  if (n <= LANES && n <= 2 * kWave) {
    if (lane < n) {
      const uint32_t at = chunk_start(lane, bytes, mis);
      if constexpr (IN_HBM) {
        *reinterpret_cast<g_u32x4_any*>(dst + at) = *reinterpret_cast<const g_u32x4_any*>(src + at);
      } else {
        store16_any(dst + at, load16_any(src + at));
      }
    }
    return;
  }
  const __amdgpu_buffer_rsrc_t tile = tile_descriptor(dst, bytes);
  // A full tile that starts off a boundary has one chunk more than U steps hold.
  with_steps<U + 1>(wave_steps<LANES>(n, lane), [&](auto steps) {
    constexpr int K = decltype(steps)::value;
    u32x4 v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      v[k] = load16_any(src + chunk_start(lane + k * LANES, bytes, mis));
    }
    if (!ALIGN_SRC) wait_for_loads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const uint32_t i = lane + k * LANES;
      const uint32_t at = chunk_start(i, bytes, mis);
      if (k + 1 == K && i >= n) continue;
      // Whole chunks of an aligned destination take the store policy of the link.
      if (!ALIGN_SRC && ((mis + at) & 15u) == 0) {
        store16_sc1_nt(tile, at, v[k]);
      } else {
        store16_any(dst + at, v[k]);
      }
    }
  });
}

// The same between two places in device memory, one chunk per lane and step, with
// ordinary loads and stores: a fragment off the 16-byte grid starts and ends
// inside a memory line that the next workgroup's fragment or tile shares, and the
// caches put the two halves together.  Streaming accesses send each half to
// memory by itself.  Measured on MI355X, 50 MB in two staged layers of K and V,
// save / load in us with streaming accesses, with words and single bytes, and
// with this: fragments of 516 bytes 1103 / 1045, 964 / 982, 961 / 966; 4100 bytes
// 972 / 970, 939 / 951, 934 / 938; 20 004 bytes 965 / 967, 934 / 948, 931 / 935;
// 1001 bytes 1023 / 1023, 970 / 999, 949 / 954; 20 bytes 2844 / 2753, 2466 / 2523,
// 2440 / 2496.
template <int LANES>
__device__ __forceinline__ void copy_tile_in_hbm(uint64_t dst, uint64_t src, uint32_t bytes,
                                                 uint32_t lane) {
  if (bytes < 16) {
    if (lane < bytes) reinterpret_cast<g_u8*>(dst)[lane] = reinterpret_cast<const g_u8*>(src)[lane];
    return;
  }
  const uint32_t mis = static_cast<uint32_t>(dst) & 15u;
  const uint32_t n = chunk_count(bytes, mis);
  for (uint32_t i = lane; i < n; i += LANES) {
    const uint32_t at = chunk_start(i, bytes, mis);
    *reinterpret_cast<g_u32x4_any*>(dst + at) = *reinterpret_cast<const g_u32x4_any*>(src + at);
  }
}

// A call's tables from mapped host memory to their place in device memory, 16 bytes
// per lane.  The launches behind it read them through the scalar cache of every XCD.
__global__ __launch_bounds__(kLanes) void table_upload_kernel(uint64_t dst, uint64_t src, uint32_t n) {
  for (uint32_t i = blockIdx.x * kLanes + threadIdx.x; i < n; i += gridDim.x * kLanes) {
    reinterpret_cast<g_u32x4*>(dst)[i] = reinterpret_cast<const g_u32x4*>(src)[i];
  }
}

// Rows of a descriptor table, wave-uniform.  Rows3: [dst, src, size] as the
// backends write it; Rows48: the caller's pf_copy_desc array as it is, so the
// host side repacks nothing.
template <bool IN_HBM>
struct Rows3 {
  static constexpr bool kInHbm = IN_HBM;  // both sides in device memory (packing)
  const uint64_t* table;
  __device__ __forceinline__ void get(uint32_t i, uint64_t* dst, uint64_t* src,
                                      uint64_t* size) const {
    c_u64* row = reinterpret_cast<c_u64*>(reinterpret_cast<uint64_t>(table)) + 3ull * i;
    *dst = row[0];
    *src = row[1];
    *size = row[2];
  }
};
template <bool HOST_IS_SRC>
struct Rows48 {
  static constexpr bool kInHbm = false;
  const pf_copy_desc* table;
  __device__ __forceinline__ void get(uint32_t i, uint64_t* dst, uint64_t* src,
                                      uint64_t* size) const {
    c_desc* row = reinterpret_cast<c_desc*>(reinterpret_cast<uint64_t>(table)) + i;
    *dst = HOST_IS_SRC ? row->device : row->host_device;
    *src = HOST_IS_SRC ? row->host_device : row->device;
    *size = row->size;
  }
};

// Rows first, first + step, ... of a table, tiles tile0, tile0 + tile_step, ...
// of each, by LANES lanes.  The next row is fetched before the current one is
// copied: the table may sit in mapped host memory (short batches skip the
// upload), where a row is a couple of microseconds away.
template <int U, int LANES, bool ALIGN_SRC, typename Rows>
__device__ __forceinline__ void copy_rows(const Rows rows, uint32_t n, uint32_t first, uint32_t step,
                                          uint32_t tile0, uint32_t tile_step, uint32_t lane) {
  constexpr uint64_t kTile = static_cast<uint64_t>(U) * LANES * 16;
  uint32_t i = first;
  if (i >= n) return;
  uint64_t dst, src, size;
  rows.get(i, &dst, &src, &size);
  for (;;) {
    const bool more = n - i > step;
    const uint32_t next = i + step;
    uint64_t next_dst = 0, next_src = 0, next_size = 0;
    if (more) rows.get(next, &next_dst, &next_src, &next_size);
    const uint64_t n_tiles = (size + kTile - 1) / kTile;
    const bool vec = ((dst | src) & 15ull) == 0;
    for (uint64_t t = tile0; t < n_tiles; t += tile_step) {
      const uint64_t off = t * kTile;
      const uint64_t left = size - off;
      const uint32_t bytes = left < kTile ? static_cast<uint32_t>(left) : static_cast<uint32_t>(kTile);
      if (vec) {
        copy_tile_vec<U, LANES>(dst + off, src + off, bytes, lane);
      } else {
        copy_tile_any<U, LANES, ALIGN_SRC, Rows::kInHbm>(dst + off, src + off, bytes, lane);
      }
    }
    if (!more) break;
    i = next;
    dst = next_dst;
    src = next_src;
    size = next_size;
  }
}

// Descriptor-table copy, a row per workgroup: blockIdx.x strides over
// descriptors, blockIdx.y over the tiles inside one, so a batch of few large
// copies still spreads over the whole chip.
template <int U, bool HOST_IS_SRC, typename Rows>
__global__ __launch_bounds__(kLanes) void desc_copy_kernel(Rows rows, uint32_t n) {
  copy_rows<U, kLanes, HOST_IS_SRC>(rows, n, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y,
                                    threadIdx.x);
}

// The same, a row per wavefront, for rows shorter than a workgroup's tile: four
// of them are in flight per workgroup instead of one.  Measured on MI355X over
// the link, 31 MB out and back: 600-byte rows 2844 -> 1360 us, 1 KiB 1460 ->
// 1190.
template <int U, bool HOST_IS_SRC, typename Rows>
__global__ __launch_bounds__(kLanes) void desc_copy_waves_kernel(Rows rows, uint32_t n) {
  constexpr uint32_t kWaves = kLanes / kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  copy_rows<U, kWave, HOST_IS_SRC>(rows, n, blockIdx.x * kWaves + wave, gridDim.x * kWaves, 0, 1,
                                   threadIdx.x % kWave);
}

// A packing launch: rows between the cache and staging, one per LANES lanes, and
// beside them, by the first `link_groups` workgroups, the rows of the run's share of
// the link (pf_share.hpp).
template <int U, bool HOST_IS_SRC, int LANES>
__global__ __launch_bounds__(kLanes) void desc_pack_kernel(Rows3<true> rows, uint32_t n,
                                                           Rows3<false> link, uint32_t n_link,
                                                           uint32_t link_groups) {
  constexpr uint32_t kRows = kLanes / LANES;  // of a workgroup at a time
  const uint32_t sub = __builtin_amdgcn_readfirstlane(threadIdx.x / LANES);
  const uint32_t lane = threadIdx.x % LANES;
  if (blockIdx.x < link_groups) {
    copy_rows<U, LANES, HOST_IS_SRC>(link, n_link, blockIdx.x * kRows + sub, link_groups * kRows,
                                     blockIdx.y, gridDim.y, lane);
  } else {
    copy_rows<U, LANES, HOST_IS_SRC>(rows, n, (blockIdx.x - link_groups) * kRows + sub,
                                     (gridDim.x - link_groups) * kRows, blockIdx.y, gridDim.y, lane);
  }
}

// The fields of a unit, wave-uniform: read once into scalar registers, all
// before the first branch on them, so that they cost one trip to memory.
struct UnitFields {
  uint64_t near_base, block_stride, kv_stride, frag_bytes, far_base0, far_base1, far_stride;
  c_u32* ids;
  c_u64* far_table;
  uint64_t far_table_off, seg1_bytes;
  uint32_t n_blocks, n_seg, tiles_per_frag, form, seg1_entries;
  bool paged, ids16;
};
template <typename UnitPtr>
__device__ __forceinline__ UnitFields unit_fields(UnitPtr up, uint64_t bias) {
  UnitFields f;
  f.near_base = up->near_base;
  f.block_stride = up->block_stride;
  f.kv_stride = up->kv_stride;
  f.frag_bytes = up->frag_bytes;
  f.far_base0 = up->far_base[0];
  f.far_base1 = up->far_base[1];
  f.far_stride = up->far_stride;
  f.ids = reinterpret_cast<c_u32*>(reinterpret_cast<uint64_t>(up->ids) + bias);
  f.paged = up->far_table != nullptr;
  f.far_table =
      reinterpret_cast<c_u64*>(reinterpret_cast<uint64_t>(up->far_table) + (f.paged ? bias : 0));
  f.far_table_off = up->far_table_off;
  // What segment 1 adds to a position's place in the table and to its base.
  f.seg1_entries = up->far_table_step;
  f.seg1_bytes = f.seg1_entries != 0 ? 0 : f.frag_bytes;
  f.n_blocks = up->n_blocks;
  f.n_seg = up->n_seg;
  f.tiles_per_frag = up->tiles_per_frag;
  f.form = up->form;
  f.ids16 = up->ids16 != 0;
  return f;
}

// Where the tiles of a unit begin in its row of workgroups: take() gives a
// workgroup's first tile of the next unit, the others follow grid_x apart.  The
// turn passes on to the workgroup behind the unit's last tile; beginning every
// unit at workgroup 0 gives the same workgroups the odd tiles of all units (24
// layers of 72 blocks of 3072 bytes, whole tiles, loaded in 126 us, in turn in 90;
// 30 layers of 136 blocks of 6144 bytes, 51 tiles of chunks each for 48
// workgroups, saved / loaded in 477 / 501, in turn in 450 / 451).  Units in chunks
// of which more than `most_odd` tiles are left after whole rounds stay at workgroup
// 0: 16 layers of 777 blocks of 1000 bytes (96 tiles, 64 workgroups) loaded in 458
// us, in turn in 464.  Units cut along the link's packets always pass it (the same
// saved in 452 us, with every unit beginning at workgroup 0 in 463).
struct RowTurn {
  uint32_t at = 0;  // workgroup whose turn it is
  __device__ __forceinline__ uint32_t take(uint32_t n_tiles, uint32_t wg, uint32_t grid_x,
                                           uint32_t most_odd) {
    const uint32_t first = wg >= at ? wg - at : wg + grid_x - at;
    const uint32_t odd = n_tiles < grid_x ? n_tiles : n_tiles % grid_x;
    if (odd <= most_odd) {
      at += odd;
      if (at >= grid_x) at -= grid_x;
    }
    return first;
  }
};

// A unit of the zero-copy form whose fragments are cut into 16-byte chunks (see
// chunk_start) that fill the lanes one after the other, whatever fragment they
// belong to: lane l of step k handles chunk 1024 t + 256 k + l of a segment.
// What bounds the tile form on fragments below its 16 KiB tile is the bytes in
// flight on the link (a workgroup holds one fragment at a time), and on
// fragments off the 16-byte grid the width of its accesses as well; here every
// tile is full.  The block id of a lane's chunk is a vector load; it costs a
// trip to the id list before the data loads can start, which the other
// workgroups cover.  Measured on MI355X, 25 MB in 16 layers of K and V, save /
// load in GB/s: fragments of 1000 bytes 47.9 / 41.4 -> 52.3 / 55.1, 1 KiB 54.8 /
// 39.1 -> 56.1 / 55.8, 4112 bytes 52.2 / 44.4 -> 56.1 / 55.9, 100 004 bytes
// (tile form with the chunks of copy_tile_any) 44.6 / 52.1 -> 52.8 / 54.8.
template <int U, bool TO_FAR>
__device__ __forceinline__ void block_chunks_unit(const UnitFields& f, uint32_t grid_x,
                                                  RowTurn& turn) {
  const uint32_t frag_bytes = static_cast<uint32_t>(f.frag_bytes);
  const uint32_t chunks_per_frag = f.tiles_per_frag;
  // The host keeps a unit's chunk count below 2^31.
  const uint32_t n_chunks = f.n_blocks * chunks_per_frag;
  const uint32_t tiles_per_seg = (n_chunks + U * kLanes - 1) / (U * kLanes);
  const uint32_t n_tiles = tiles_per_seg * f.n_seg;
  for (uint32_t t = turn.take(n_tiles, blockIdx.x, grid_x, grid_x / 4); t < n_tiles; t += grid_x) {
    const uint32_t seg = t >= tiles_per_seg ? 1u : 0u;
    const uint32_t first = (seg ? t - tiles_per_seg : t) * (U * kLanes) + threadIdx.x;
    const uint64_t near_seg = f.near_base + (seg ? f.kv_stride : 0);
    const uint64_t far_seg = seg ? f.far_base1 : f.far_base0;
    const uint32_t left = n_chunks - (first - threadIdx.x);  // > 0
    with_steps<U>(min(wave_steps<kLanes>(left, threadIdx.x), static_cast<uint32_t>(U)), [&](auto steps) {
      constexpr int K = decltype(steps)::value;
      uint64_t src[K], dst[K], far[K];
      uint32_t pos[K], id_word[K], chunk[K];
      bool ok[K];
      u32x4 v[K];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        ok[k] = k + 1 < K || first + k * kLanes < n_chunks;
        const uint32_t g = ok[k] ? first + k * kLanes : n_chunks - 1;
        pos[k] = g / chunks_per_frag;
        chunk[k] = g - pos[k] * chunks_per_frag;
        id_word[k] = f.ids[f.ids16 ? pos[k] >> 1 : pos[k]];
      }
      if (f.paged) {
#pragma unroll
        for (int k = 0; k < K; ++k) far[k] = f.far_table[pos[k] + (seg ? f.seg1_entries : 0)];
#pragma unroll
        for (int k = 0; k < K; ++k) far[k] += f.far_table_off + (seg ? f.seg1_bytes : 0);
      } else {
#pragma unroll
        for (int k = 0; k < K; ++k) far[k] = far_seg + pos[k] * f.far_stride;
      }
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const uint64_t id =
            f.ids16 ? ((pos[k] & 1u) ? id_word[k] >> 16 : id_word[k] & 0xFFFFu) : id_word[k];
        // chunks_per_frag is the largest count of any alignment that occurs.
        const uint32_t mis = static_cast<uint32_t>(far[k]) & 15u;
        ok[k] = ok[k] && chunk[k] < chunk_count(frag_bytes, mis);
        const uint32_t start = chunk_start(chunk[k], frag_bytes, mis);
        const uint64_t near_addr = near_seg + id * f.block_stride + start;
        src[k] = TO_FAR ? near_addr : far[k] + start;
        dst[k] = TO_FAR ? far[k] + start : near_addr;
      }
#pragma unroll
      for (int k = 0; k < K; ++k) v[k] = load16_any(src[k]);
      if (TO_FAR) wait_for_loads();
      if (TO_FAR && !f.paged) {
        // The far side of a segment is one range (below 4 GiB: the host checks),
        // so aligned chunks can take the store policy that the link wants.
        const uint64_t span = (f.n_blocks - 1) * f.far_stride + frag_bytes;
        const __amdgpu_buffer_rsrc_t range = tile_descriptor(far_seg, static_cast<uint32_t>(span));
#pragma unroll
        for (int k = 0; k < K; ++k) {
          if (!ok[k]) continue;
          if ((dst[k] & 15ull) == 0) {
            store16_sc1_nt(range, static_cast<uint32_t>(dst[k] - far_seg), v[k]);
          } else {
            store16_any(dst[k], v[k]);
          }
        }
      } else {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          if (ok[k]) store16_any(dst[k], v[k]);
        }
      }
    });
  }
}

// Saves of fragments off the 16-byte grid into a host image without gaps, cut along
// the link's packets (line_chunk): every wavefront writes whole ones, and a chunk that
// holds the end of one fragment and the head of the next is put together from both.
// With chunks of one fragment (block_chunks_unit) both ends of a fragment share a
// packet with a neighbour, and the link carries its parts one by one.  Measured on
// MI355X, GB/s queued, chunks of one fragment, along lines of 64 bytes, along packets
// of 256: 16 layers of 1000-byte fragments, 25 MB, 52.3 / 55.0 / 55.8, 600 bytes 50.5 /
// 53.9 / 54.7, 4100 bytes 53.7 / 55.2 / 55.9, 40 004 bytes (32 workgroups) 53.3 / 55.4 /
// 55.9; 2 MB of 516 bytes 43.2 / 51.7 / 52.1, of 20 bytes 17.4 / 40.2 / 40.4.  Loads gain
// nothing by it (25 MB of 1000 bytes 451 us either way, 1 MB 26.4 instead of 23.9): both
// parts of a shared packet are read anyway, and the chunks of two fragments have to be
// stored in pieces.
template <int U>
__device__ __forceinline__ void block_lines_unit(const UnitFields& f, uint32_t grid_x, RowTurn& turn) {
  typedef unsigned __int128 u128;
  const uint32_t frag = static_cast<uint32_t>(f.frag_bytes);
  const uint32_t range = f.n_blocks * frag;  // the host keeps it within kMaxLinesRange
  const uint32_t n_chunks = line_chunk_count(range);
  const uint32_t tiles_per_seg = (n_chunks + U * kLanes - 1) / (U * kLanes);
  const uint32_t n_tiles = tiles_per_seg * f.n_seg;
  for (uint32_t t = turn.take(n_tiles, blockIdx.x, grid_x, grid_x); t < n_tiles; t += grid_x) {
    const uint32_t seg = t >= tiles_per_seg ? 1u : 0u;
    const uint32_t first = (seg ? t - tiles_per_seg : t) * (U * kLanes) + threadIdx.x;
    const uint64_t near_seg = f.near_base + (seg ? f.kv_stride : 0);
    const uint64_t far_seg = seg ? f.far_base1 : f.far_base0;
    const uint32_t lead = static_cast<uint32_t>(far_seg) & (kLinkPacket - 1);
    const __amdgpu_buffer_rsrc_t image = tile_descriptor(far_seg, range);
    const uint32_t left = n_chunks - (first - threadIdx.x);  // > 0
    with_steps<U>(min(wave_steps<kLanes>(left, threadIdx.x), static_cast<uint32_t>(U)), [&](auto steps) {
      constexpr int K = decltype(steps)::value;
      LineChunk c[K];
      uint32_t word[K], next_word[K];
      u32x4 v[K], w[K];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        c[k] = line_chunk(first + k * kLanes, lead, range, frag);
        word[k] = f.ids[f.ids16 ? c[k].pos >> 1 : c[k].pos];
        next_word[k] = 0;
        if (c[k].tail < 16) next_word[k] = f.ids[f.ids16 ? (c[k].pos + 1) >> 1 : c[k].pos + 1];
      }
      auto near_of = [&](uint32_t pos, uint32_t id_word) {
        const uint64_t id = f.ids16 ? ((pos & 1u) ? id_word >> 16 : id_word & 0xFFFFu) : id_word;
        return near_seg + id * f.block_stride;
      };
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const uint32_t at = c[k].tail < 16 ? frag - 16u : c[k].start - c[k].pos * frag;
        v[k] = load16_any(near_of(c[k].pos, word[k]) + at);
        w[k] = v[k];
        if (c[k].tail < 16) w[k] = load16_any(near_of(c[k].pos + 1, next_word[k]));
      }
      wait_for_loads();
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (c[k].tail < 16) {
          v[k] = __builtin_bit_cast(u32x4, (__builtin_bit_cast(u128, v[k]) >> (8 * (16 - c[k].tail))) |
                                               (__builtin_bit_cast(u128, w[k]) << (8 * c[k].tail)));
        }
        if (!c[k].any) continue;
        if (((lead + c[k].start) & 15u) == 0) {
          store16_sc1_nt(image, c[k].start, v[k]);
        } else {
          store16_any(far_seg + c[k].start, v[k]);
        }
      }
    });
  }
}

// The tiles of a unit over mapped host memory, by workgroup `wg` of the `grid_x` of
// its row.  VEC_ONLY: the unit is known to be of the form kUnitVec, with one range
// of host memory per segment and 32-bit ids.
template <int U, int LANES, bool TO_FAR, bool VEC_ONLY>
__device__ __forceinline__ void unit_tiles(const UnitFields& f, RowTurn& turn, uint32_t wg,
                                           uint32_t grid_x) {
  constexpr uint64_t kTile = static_cast<uint64_t>(U) * LANES * 16;
  const bool vec_ok = VEC_ONLY || f.form == kUnitVec;
  const bool ids16 = !VEC_ONLY && f.ids16;
  // The host keeps a unit's tile count below 2^32, so 32-bit scalar division.
  const uint32_t tiles_per_seg = f.n_blocks * f.tiles_per_frag;
  const uint32_t n_tiles = tiles_per_seg * f.n_seg;
  for (uint32_t t = turn.take(n_tiles, wg, grid_x, grid_x); t < n_tiles; t += grid_x) {
    const uint32_t seg = t >= tiles_per_seg ? 1u : 0u;
    const uint32_t r = seg ? t - tiles_per_seg : t;
    // The quotient is wave-uniform; pin it to a scalar register so the id and
    // page-table reads below are scalar loads.
    const uint32_t pos = __builtin_amdgcn_readfirstlane(r / f.tiles_per_frag);
    const uint32_t c = r - pos * f.tiles_per_frag;
    const uint64_t off = static_cast<uint64_t>(c) * kTile;
    const uint64_t left = f.frag_bytes - off;
    const uint32_t bytes = left < kTile ? static_cast<uint32_t>(left) : static_cast<uint32_t>(kTile);
    // 16-bit ids sit two to a word (there is no scalar load of half a word).
    const uint32_t id_word = f.ids[ids16 ? pos >> 1 : pos];
    const uint64_t id = ids16 ? ((pos & 1u) ? id_word >> 16 : id_word & 0xFFFFu) : id_word;
    const uint64_t near_addr = f.near_base + id * f.block_stride + (seg ? f.kv_stride : 0) + off;
    uint64_t far_addr;
    if (!VEC_ONLY && f.paged) {
      far_addr = f.far_table[pos + (seg ? f.seg1_entries : 0)] + f.far_table_off +
                 (seg ? f.seg1_bytes : 0) + off;
    } else {
      far_addr = (seg ? f.far_base1 : f.far_base0) + static_cast<uint64_t>(pos) * f.far_stride + off;
    }
    const uint64_t dst = TO_FAR ? far_addr : near_addr;
    const uint64_t src = TO_FAR ? near_addr : far_addr;
    if (vec_ok) {
      copy_tile_vec<U, LANES>(dst, src, bytes, threadIdx.x);
    } else {
      copy_tile_any<U, LANES, !TO_FAR>(dst, src, bytes, threadIdx.x);
    }
  }
}

// Block-ID gather / scatter over mapped host memory (the zero-copy form).  The
// grid is a few rows of workgroups, as many workgroups in all as the launch
// may keep on the device.  Row y walks the units y, y + rows, ... one after the
// other and its workgroups stride over the tiles of each, so the workgroup
// count does not grow with the number of units.  With large units there is one
// row and the units complete in order; a call of many small units (a few
// blocks of every layer, the shape of a decode-time load) gets several rows,
// or most workgroups would find no tile in a unit of four tiles and the rest
// would walk all the units alone: 32 layers x 1 block loaded in 68 us with one
// row of 16 workgroups (4 of them busy, 32 tiles each one after the other,
// every tile a round trip over the link).  Tile order inside a unit is
// (segment, list position, tile in fragment), so at any moment the workgroups
// of a row touch neighbouring far-side addresses.
template <int U, bool TO_FAR, typename UnitPtr>
__device__ __forceinline__ void block_units_body(UnitPtr units, uint32_t n_units, uint32_t grid_x,
                                                 uint32_t grid_y, uint64_t bias) {
  RowTurn turn;
  for (uint32_t unit = blockIdx.y; unit < n_units; unit += grid_y) {
    const UnitFields f = unit_fields(units + unit, bias);
    if (f.form == kUnitChunks) {
      block_chunks_unit<U, TO_FAR>(f, grid_x, turn);
      continue;
    }
    if constexpr (TO_FAR) {
      if (f.form == kUnitLines) {
        block_lines_unit<U>(f, grid_x, turn);
        continue;
      }
    }
    unit_tiles<U, kLanes, TO_FAR, false>(f, turn, blockIdx.x, grid_x);
  }
}

template <int U, bool TO_FAR>
__global__ __launch_bounds__(kLanes) void block_units_kernel(const BlockUnit* __restrict__ units,
                                                             uint32_t n_units, uint32_t grid_x,
                                                             uint32_t grid_y) {
  block_units_body<U, TO_FAR, const BlockUnit*>(units, n_units, grid_x, grid_y, 0);
}

// The same kernel for short lists, with the units, id lists and page tables
// travelling in the kernel's arguments instead of a slab that has to be
// uploaded first: one command fewer on the stream (measured on MI355X, submit +
// synchronise of one small transfer: the upload costs 3.5 us of ~36 us at 1 MiB
// and of ~90 us at 4 MiB).  `slab` is the first argument, so it starts at
// offset 0 of the argument segment; a unit's `ids` / `far_table` hold byte
// offsets into it.
template <int U, bool TO_FAR>
__global__ __launch_bounds__(kLanes) void block_units_args_kernel(ArgSlab slab, uint32_t first_unit,
                                                                  uint32_t n_units, uint32_t grid_x,
                                                                  uint32_t grid_y) {
  (void)slab;
  const uint64_t base = reinterpret_cast<uint64_t>(__builtin_amdgcn_kernarg_segment_ptr());
  block_units_body<U, TO_FAR, c_unit*>(reinterpret_cast<c_unit*>(base) + first_unit, n_units, grid_x,
                                       grid_y, base);
}

// Block-ID gather / scatter, one small tile per workgroup (the HBM-bound form
// used between the KV cache and a device staging buffer).
//
// grid = (tiles per fragment, list positions, SEGS * units), SEGS being the
// largest segment count among the units of the launch; a workgroup of LT
// lanes moves LT*16 bytes with one 16-byte load per lane.  Measured on MI355X
// against the alternatives at the Llama shape (5000 x 2 x 32 KiB per launch):
// this form reaches ~6.3 TB/s (read+write), a 16 KiB-per-workgroup grid-stride
// loop ~5.6 TB/s, a persistent grid ~5.5 TB/s; the tiny register footprint
// keeps every SIMD full of waves, and the 3-D grid needs no division.
// Remapping workgroups so that each XCD owns whole fragments changed nothing
// (no data is reused, so there is no L2 locality to win).
// UNITS_INNER: grid.y walks the (unit, segment) pairs and grid.z the list
// positions, so workgroups that are dispatched together belong to one
// position; otherwise grid.y walks the positions of one (unit, segment).
// One tile of one fragment: row `row` of unit `up`, segment `seg`, tile blockIdx.x.
template <int LT, bool TO_FAR, typename UnitPtr>
__device__ __forceinline__ void block_tiles_copy(UnitPtr up, uint32_t row, uint32_t seg) {
  constexpr uint32_t kTile = LT * 16;
  if (row >= up->n_blocks) return;
  // Rows may visit the list positions in another order (see launch_block_tiles).
  uint32_t pos = row;
  if (up->order != nullptr) {
    c_u32* order = reinterpret_cast<c_u32*>(reinterpret_cast<uint64_t>(up->order));
    pos = order[row];
  }
  const uint64_t frag_bytes = up->frag_bytes;
  const uint64_t off = static_cast<uint64_t>(blockIdx.x) * kTile;
  // (Fragments of a segment that the unit does not have lie behind all it has.)
  if (pos >= up->n_blocks || seg * up->n_blocks + pos >= up->staged_frags || off >= frag_bytes) return;
  c_u32* ids = reinterpret_cast<c_u32*>(reinterpret_cast<uint64_t>(up->ids));
  const uint64_t id = ids[pos];
  const uint64_t near_addr =
      up->near_base + id * up->block_stride + (seg ? up->kv_stride : 0) + off;
  const uint64_t far_addr = (seg ? up->far_base[1] : up->far_base[0]) +
                            static_cast<uint64_t>(pos) * up->far_stride + off;
  const uint64_t dst = TO_FAR ? far_addr : near_addr;
  const uint64_t src = TO_FAR ? near_addr : far_addr;
  const uint64_t left = frag_bytes - off;
  const uint32_t bytes = left < kTile ? static_cast<uint32_t>(left) : kTile;
  const uint32_t lane = threadIdx.x;
  if (up->form == kUnitVec) {
    const g_u32x4* __restrict__ s = reinterpret_cast<const g_u32x4*>(src);
    const uint32_t nvec = bytes >> 4;
    const __amdgpu_buffer_rsrc_t tile = tile_descriptor(dst, nvec << 4);
    if (lane < nvec) {
      // Streaming load and store in both directions: nothing is read twice.
      // (Gather with an ordinary load of the scattered source: 5.90 TB/s at
      // the Llama shape, with the streaming load 6.14.)
      const u32x4 v = __builtin_nontemporal_load(s + lane);
      store16_sc1_nt(tile, lane * 16u, v);
    }
    const uint32_t j = (nvec << 4) + lane;
    if (j < bytes) reinterpret_cast<g_u8*>(dst)[j] = reinterpret_cast<const g_u8*>(src)[j];
  } else {
    copy_tile_in_hbm<LT>(dst, src, bytes, lane);
  }
}

// The launch's share of the link: the workgroups of the first `planes` planes of the
// grid (the first to be dispatched) move it while all others go through HBM.
// True for a workgroup of these planes.
template <int LT, bool TO_FAR>
__device__ __forceinline__ bool link_share(const LinkShare& share, uint32_t planes, bool planes_are_z) {
  if ((planes_are_z ? blockIdx.z : blockIdx.y) >= planes) return false;
  const uint32_t wg = blockIdx.x + gridDim.x * (planes_are_z ? blockIdx.y + gridDim.y * blockIdx.z
                                                             : blockIdx.y);
  if (wg >= share.workgroups || (!planes_are_z && blockIdx.z != 0)) return true;
  constexpr int kUnroll = kShareTileBytes / (LT * 16);
  RowTurn turn;
  for (uint32_t k = 0; k < share.n_units; ++k) {
    unit_tiles<kUnroll, LT, TO_FAR, true>(unit_fields(share.units + k, 0), turn, share.first + wg, share.all);
  }
  return true;
}

template <int LT, bool TO_FAR, int SEGS, bool UNITS_INNER, typename UnitPtr>
__device__ __forceinline__ void block_tiles_body(UnitPtr units, const LinkShare& share, uint32_t planes) {
  if (link_share<LT, TO_FAR>(share, planes, UNITS_INNER)) return;
  const uint32_t unit_seg = UNITS_INNER ? blockIdx.y : blockIdx.z;
  const uint32_t row = (UNITS_INNER ? blockIdx.z : blockIdx.y) - planes;
  UnitPtr up = units + (SEGS == 2 ? unit_seg >> 1 : unit_seg);
  const uint32_t seg = SEGS == 2 ? (unit_seg & 1u) : 0u;
  block_tiles_copy<LT, TO_FAR, UnitPtr>(up, row, seg);
}

template <int LT, bool TO_FAR, int SEGS, bool UNITS_INNER>
__global__ __launch_bounds__(LT) void block_tiles_kernel(const BlockUnit* __restrict__ units,
                                                         LinkShare share, uint32_t planes) {
  block_tiles_body<LT, TO_FAR, SEGS, UNITS_INNER, const BlockUnit*>(units, share, planes);
}

// A few units of different lengths in one launch (the fills of a staging slot:
// the tail of one layer, whole layers, the head of the next): grid.y runs over
// the rows of all units laid end to end, so that no workgroup is launched for a
// row a shorter unit does not have (with the grid of block_tiles_kernel, sized
// by the longest unit, up to 45 % of the workgroups of such a launch found
// nothing to do and it ran at 5.2 instead of 6.1 TB/s).  The running row counts
// arrive with the kernel's arguments, so finding the unit costs no memory access.
struct RowEnds {
  uint32_t end[kMaxRowUnits];  // end[k] = rows of units 0..k; UINT32_MAX past the last unit
};

template <int LT, bool TO_FAR, int SEGS>
__global__ __launch_bounds__(LT) void block_tiles_rows_kernel(const BlockUnit* __restrict__ units,
                                                              RowEnds ends, LinkShare share,
                                                              uint32_t planes) {
  if (link_share<LT, TO_FAR>(share, planes, false)) return;
  // More rows than one grid extent are folded over grid.z: z = chunk * SEGS + segment.
  const uint32_t chunk = SEGS == 2 ? blockIdx.z >> 1 : blockIdx.z;
  const uint32_t seg = SEGS == 2 ? blockIdx.z & 1u : 0u;
  const uint32_t row = chunk * (gridDim.y - planes) + blockIdx.y - planes;
  uint32_t unit = 0, first = 0;
#pragma unroll
  for (uint32_t k = 0; k + 1 < kMaxRowUnits; ++k) {
    if (row >= ends.end[k]) {
      unit = k + 1;
      first = ends.end[k];
    }
  }
  // (A row past the last unit's end, in the last chunk, finds no block there.)
  block_tiles_copy<LT, TO_FAR, const BlockUnit*>(units + unit, row - first, seg);
}

// One unit, passed by value: its fields arrive with the kernel's arguments
// instead of behind a pointer, one dependent scalar load fewer before the id of
// the workgroup's row is known (a workgroup lives for one load and one store, so
// every level of that chain is a measurable part of its life).  The unit is the
// first argument: offset 0 of the argument segment.
template <int LT, bool TO_FAR, int SEGS>
__global__ __launch_bounds__(LT) void block_tiles_one_kernel(BlockUnit unit, LinkShare share,
                                                             uint32_t planes) {
  (void)unit;
  block_tiles_body<LT, TO_FAR, SEGS, false, c_unit*>(
      reinterpret_cast<c_unit*>(reinterpret_cast<uint64_t>(__builtin_amdgcn_kernarg_segment_ptr())),
      share, planes);
}

// The two halves of streams_run_concurrently().  The wait is bounded by the
// constant-rate device clock (100 MHz), so the lane leaves whatever happens.
__global__ __launch_bounds__(64) void probe_wait_kernel(uint32_t* word, uint32_t* seen,
                                                        uint64_t max_ticks) {
  if (threadIdx.x != 0) return;
  const uint64_t begin = wall_clock64();
  uint32_t value = 0;
  for (;;) {
    value = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (value != 0 || wall_clock64() - begin > max_ticks) break;
    __builtin_amdgcn_s_sleep(16);
  }
  __hip_atomic_store(seen, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(64) void probe_post_kernel(uint32_t* word) {
  if (threadIdx.x == 0) __hip_atomic_store(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int U>
__global__ __launch_bounds__(kLanes) void plain_copy_kernel(uint64_t dst, uint64_t src,
                                                            uint64_t bytes) {
  constexpr uint64_t kTile = static_cast<uint64_t>(U) * kLanes * 16;
  const uint64_t n_tiles = (bytes + kTile - 1) / kTile;
  for (uint64_t t = blockIdx.x; t < n_tiles; t += gridDim.x) {
    const uint64_t off = t * kTile;
    const uint64_t left = bytes - off;
    copy_tile_vec<U, kLanes>(
        dst + off, src + off,
        left < kTile ? static_cast<uint32_t>(left) : static_cast<uint32_t>(kTile), threadIdx.x);
  }
}

// Plain copy in the one-tile-per-workgroup form of block_tiles_kernel.
template <int LT>
__global__ __launch_bounds__(LT) void plain_tiles_kernel(uint64_t dst, uint64_t src,
                                                         uint64_t bytes) {
  const uint64_t off = static_cast<uint64_t>(blockIdx.x) * (LT * 16ull) + threadIdx.x * 16ull;
  if (off < bytes) {
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const g_u32x4*>(src + off));
    __builtin_nontemporal_store(v, reinterpret_cast<g_u32x4*>(dst + off));
  }
}

constexpr int kTileLanes = 128;  // lanes of a block_tiles_kernel workgroup
static_assert(kTileLanes * 16 == kStagedTileBytes, "tile size the planner of launches assumes");
constexpr uint32_t kMaxGridX = 1u << 22;  // the kernels grid-stride past this
constexpr int kDescUnroll = 4;
constexpr uint32_t kMaxUploadWorkgroups = 64;

}  // namespace

bool unroll_supported(int unroll) { return unroll == 1 || unroll == 2 || unroll == 4 || unroll == 8; }

namespace {
// Grid of a zero-copy launch: `max_workgroups` (0 = no cap) in all; x strides
// over the tiles of a unit, y over the units.  Units as large as the cap or
// larger leave one row.
dim3 block_units_grid(uint32_t n_units, uint64_t max_tiles, uint32_t max_workgroups) {
  uint64_t gx = max_tiles < kMaxGridX ? max_tiles : kMaxGridX;
  if (max_workgroups != 0 && gx > max_workgroups) gx = max_workgroups;
  uint64_t gy = 1;
  if (max_workgroups != 0 && gx < max_workgroups) {
    gy = max_workgroups / gx;
    if (gy > n_units) gy = n_units;
    if (gy > 65535) gy = 65535;
    if (gy < 1) gy = 1;
  }
  return dim3(static_cast<uint32_t>(gx), static_cast<uint32_t>(gy), 1);
}
}  // namespace

namespace {
// A zero-copy launch; its dispatch completes `stop`, with no barrier behind it.
template <typename... Params>
hipError_t launch_units(void (*kernel)(Params...), dim3 grid, hipStream_t s, hipEvent_t stop,
                        Params... params) {
  const void* address = reinterpret_cast<const void*>(kernel);
  void* args[] = {&params...};
  const dim3 block(kLanes, 1, 1);
  return stop != nullptr ? hipExtLaunchKernel(address, grid, block, args, 0, s, nullptr, stop, 0)
                         : hipLaunchKernel(address, grid, block, args, 0, s);
}
}  // namespace

int launch_block_units(const BlockUnit* units, uint32_t n_units, uint64_t max_tiles, bool to_far,
                       int unroll, uint32_t max_workgroups_x, hipStream_t s, hipEvent_t stop) {
  if (n_units == 0 || max_tiles == 0) return PF_OK;
  if (max_tiles > 0x7FFFFFFFull) {
    return fail(PF_ERR_INVALID_ARGUMENT, "unit of %llu tiles exceeds the kernel limit",
                static_cast<unsigned long long>(max_tiles));
  }
  const dim3 grid = block_units_grid(n_units, max_tiles, max_workgroups_x);
  hipError_t e = hipSuccess;
#define PF_LAUNCH_UNITS(U_)                                                                    \
  case U_:                                                                                     \
    e = launch_units(to_far ? block_units_kernel<U_, true> : block_units_kernel<U_, false>,    \
                     grid, s, stop, units, n_units, grid.x, grid.y);                          \
    break;
  switch (unroll) {
    PF_LAUNCH_UNITS(1)
    PF_LAUNCH_UNITS(2)
    PF_LAUNCH_UNITS(4)
    PF_LAUNCH_UNITS(8)
    default:
      return fail(PF_ERR_INVALID_ARGUMENT, "unsupported tile unroll %d", unroll);
  }
#undef PF_LAUNCH_UNITS
  if (e != hipSuccess) return fail_hip(e, "block_units_kernel launch");
  return PF_OK;
}

int launch_block_units_args(const ArgSlab& slab, uint32_t first_unit, uint32_t n_units,
                            uint64_t max_tiles, bool to_far, int unroll, uint32_t max_workgroups_x,
                            hipStream_t s, hipEvent_t stop) {
  if (n_units == 0 || max_tiles == 0) return PF_OK;
  if (max_tiles > 0x7FFFFFFFull) {
    return fail(PF_ERR_INVALID_ARGUMENT, "unit of %llu tiles exceeds the kernel limit",
                static_cast<unsigned long long>(max_tiles));
  }
  const dim3 grid = block_units_grid(n_units, max_tiles, max_workgroups_x);
  hipError_t e = hipSuccess;
#define PF_LAUNCH_ARGS(U_)                                                                             \
  case U_:                                                                                             \
    e = launch_units(to_far ? block_units_args_kernel<U_, true> : block_units_args_kernel<U_, false>,  \
                     grid, s, stop, slab, first_unit, n_units, grid.x, grid.y);                       \
    break;
  switch (unroll) {
    PF_LAUNCH_ARGS(1)
    PF_LAUNCH_ARGS(2)
    PF_LAUNCH_ARGS(4)
    PF_LAUNCH_ARGS(8)
    default:
      return fail(PF_ERR_INVALID_ARGUMENT, "unsupported tile unroll %d", unroll);
  }
#undef PF_LAUNCH_ARGS
  if (e != hipSuccess) return fail_hip(e, "block_units_args_kernel launch");
  return PF_OK;
}

namespace {
// Planes of a grid, `per_plane` workgroups each, that hold a share's workgroups.
uint32_t share_planes(const LinkShare& share, uint64_t per_plane) {
  return static_cast<uint32_t>((share.workgroups + per_plane - 1) / per_plane);
}
}  // namespace

int launch_block_tiles_one(const BlockUnit& unit, bool to_far, hipStream_t s, const LinkShare& share) {
  if (unit.n_blocks == 0 || unit.frag_bytes == 0) return PF_OK;
  if (unit.n_seg != 1 && unit.n_seg != 2) {
    return fail(PF_ERR_INVALID_ARGUMENT, "tile launch: %u segments per block", unit.n_seg);
  }
  constexpr uint64_t kTile = kTileLanes * 16;
  const uint64_t gx = (unit.frag_bytes + kTile - 1) / kTile;
  const uint32_t planes = share_planes(share, gx);
  if (unit.n_blocks > kMaxTileBlocks - planes || gx > 0x7FFFFFFFull) {
    return fail(PF_ERR_INVALID_ARGUMENT, "tile launch out of range: %u blocks, %llu-byte fragments",
                unit.n_blocks, static_cast<unsigned long long>(unit.frag_bytes));
  }
  dim3 grid(static_cast<uint32_t>(gx), unit.n_blocks + planes, unit.n_seg);
  dim3 block(kTileLanes, 1, 1);
  if (unit.n_seg == 2) {
    if (to_far) {
      hipLaunchKernelGGL((block_tiles_one_kernel<kTileLanes, true, 2>), grid, block, 0, s, unit, share,
                         planes);
    } else {
      hipLaunchKernelGGL((block_tiles_one_kernel<kTileLanes, false, 2>), grid, block, 0, s, unit, share,
                         planes);
    }
  } else if (to_far) {
    hipLaunchKernelGGL((block_tiles_one_kernel<kTileLanes, true, 1>), grid, block, 0, s, unit, share,
                         planes);
  } else {
    hipLaunchKernelGGL((block_tiles_one_kernel<kTileLanes, false, 1>), grid, block, 0, s, unit, share,
                         planes);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail_hip(e, "block_tiles_one_kernel launch");
  return PF_OK;
}

int launch_block_tiles_rows(const BlockUnit* units, const BlockUnit* host_units, uint32_t n_units,
                            bool to_far, hipStream_t s, bool* launched, const LinkShare& share) {
  *launched = false;
  if (n_units == 0 || n_units > kMaxRowUnits) return PF_OK;
  RowEnds ends;
  uint64_t rows = 0, max_frag = 0;
  uint32_t max_seg = 0;
  for (uint32_t k = 0; k < kMaxRowUnits; ++k) {
    if (k < n_units) {
      const BlockUnit& u = host_units[k];
      if (u.n_seg != 1 && u.n_seg != 2) {
        return fail(PF_ERR_INVALID_ARGUMENT, "tile launch: %u segments per block", u.n_seg);
      }
      rows += u.n_blocks;
      max_frag = max_frag < u.frag_bytes ? u.frag_bytes : max_frag;
      max_seg = max_seg < u.n_seg ? u.n_seg : max_seg;
    }
    ends.end[k] = k + 1 < n_units ? static_cast<uint32_t>(rows) : UINT32_MAX;
  }
  constexpr uint64_t kTile = kTileLanes * 16;
  const uint64_t gx = (max_frag + kTile - 1) / kTile;
  if (rows == 0 || max_frag == 0) {
    *launched = true;
    return PF_OK;
  }
  // Rows beyond one grid extent go into further chunks of equal length along grid.z.
  const uint32_t planes = share_planes(share, gx);
  const uint64_t chunk_rows = kMaxTileBlocks - planes;
  const uint64_t chunks = (rows + chunk_rows - 1) / chunk_rows;
  const uint64_t gy = (rows + chunks - 1) / chunks + planes;
  if (chunks * max_seg > kMaxTileBlocks || rows >= 0xFFFFFFFFull || gx > 0x7FFFFFFFull) {
    return PF_OK;  // the caller takes another form
  }
  dim3 grid(static_cast<uint32_t>(gx), static_cast<uint32_t>(gy),
            static_cast<uint32_t>(chunks * max_seg));
  dim3 block(kTileLanes, 1, 1);
  if (max_seg == 2) {
    if (to_far) {
      hipLaunchKernelGGL((block_tiles_rows_kernel<kTileLanes, true, 2>), grid, block, 0, s, units, ends,
                         share, planes);
    } else {
      hipLaunchKernelGGL((block_tiles_rows_kernel<kTileLanes, false, 2>), grid, block, 0, s, units, ends,
                         share, planes);
    }
  } else if (to_far) {
    hipLaunchKernelGGL((block_tiles_rows_kernel<kTileLanes, true, 1>), grid, block, 0, s, units, ends,
                         share, planes);
  } else {
    hipLaunchKernelGGL((block_tiles_rows_kernel<kTileLanes, false, 1>), grid, block, 0, s, units, ends,
                         share, planes);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail_hip(e, "block_tiles_rows_kernel launch");
  *launched = true;
  return PF_OK;
}

int launch_block_tiles(const BlockUnit* units, uint32_t n_units, uint32_t max_blocks,
                       uint64_t max_frag_bytes, uint32_t max_seg, bool to_far, hipStream_t s,
                       const LinkShare& share) {
  if (n_units == 0 || max_blocks == 0 || max_frag_bytes == 0) return PF_OK;
  if (max_seg != 1 && max_seg != 2) {
    return fail(PF_ERR_INVALID_ARGUMENT, "tile launch: %u segments per block", max_seg);
  }
  constexpr uint64_t kTile = kTileLanes * 16;
  const uint64_t gx = (max_frag_bytes + kTile - 1) / kTile;
  if (n_units > kMaxTileUnits || max_blocks > kMaxTileBlocks || gx > 0x7FFFFFFFull) {
    return fail(PF_ERR_INVALID_ARGUMENT,
                "tile launch out of range: %u units, %u blocks, %llu-byte fragments", n_units,
                max_blocks, static_cast<unsigned long long>(max_frag_bytes));
  }
  // A launch over several units (the layers of page-first pages) makes the
  // units the inner grid dimension: the staging side is then walked page after
  // page and every cache in ascending position order.  Measured on the
  // DeepSeek-V3 page-first shape (61 units x 119 pages per launch): gather
  // 5.3 -> 5.9 TB/s, scatter 5.5 -> 6.2 TB/s against positions-inner.
  // A few units of equal length (page packing of a model with few layers) keep
  // the order of a single unit, one (unit, segment) after the other: with 2-4
  // units per launch that form measured 1-2 % faster than units-inner (Llama
  // shape, three layers per launch: 6.10 against 6.04 TB/s; fp8 shape, four:
  // 6.18 against 6.10).  Staging fills of up to eight units of unlike lengths
  // do not come here: launch_block_tiles_rows.
  constexpr uint32_t kUnitsInnerFrom = 9;
  const bool units_inner = n_units >= kUnitsInnerFrom;
  const uint32_t unit_segs = max_seg * n_units;
  const uint32_t planes = share_planes(share, units_inner ? gx * unit_segs : gx);
  if (max_blocks > kMaxTileBlocks - planes) {
    return fail(PF_ERR_INVALID_ARGUMENT, "tile launch out of range: %u blocks and a share of the link",
                max_blocks);
  }
  dim3 grid(static_cast<uint32_t>(gx), units_inner ? unit_segs : max_blocks + planes,
            units_inner ? max_blocks + planes : unit_segs);
  dim3 block(kTileLanes, 1, 1);
#define PF_LAUNCH_TILES(TO_FAR_, SEGS_, INNER_)                                                \
  hipLaunchKernelGGL((block_tiles_kernel<kTileLanes, TO_FAR_, SEGS_, INNER_>), grid, block, 0, s, \
                     units, share, planes)
  if (units_inner) {
    if (max_seg == 2) {
      if (to_far) {
        PF_LAUNCH_TILES(true, 2, true);
      } else {
        PF_LAUNCH_TILES(false, 2, true);
      }
    } else {
      if (to_far) {
        PF_LAUNCH_TILES(true, 1, true);
      } else {
        PF_LAUNCH_TILES(false, 1, true);
      }
    }
  } else if (max_seg == 2) {
    if (to_far) {
      PF_LAUNCH_TILES(true, 2, false);
    } else {
      PF_LAUNCH_TILES(false, 2, false);
    }
  } else {
    if (to_far) {
      PF_LAUNCH_TILES(true, 1, false);
    } else {
      PF_LAUNCH_TILES(false, 1, false);
    }
  }
#undef PF_LAUNCH_TILES
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail_hip(e, "block_tiles_kernel launch");
  return PF_OK;
}

}  // namespace pf

// The two words of the stream-concurrency probe ([0] the posted word, [1] what
// the waiter saw) live in the library's device image: a probe allocates and
// frees nothing, so it never waits for unrelated work on the device (hipFree
// synchronises the whole device).
static __device__ __align__(256) uint32_t probe_words[2];

namespace pf {

namespace {
constexpr int kProbeMaxDevices = 64;
std::mutex g_probe_mu;  // one probe at a time: they share the two words
uint32_t* g_probe_ptr[kProbeMaxDevices] = {};

int probe_words_on_current_device(uint32_t** out) {
  int device = -1;
  PF_HIP(hipGetDevice(&device));
  if (device < 0 || device >= kProbeMaxDevices) {
    return fail(PF_ERR_INVALID_ARGUMENT, "device %d is beyond the %d the probe supports", device,
                kProbeMaxDevices);
  }
  if (g_probe_ptr[device] == nullptr) {
    void* ptr = nullptr;
    PF_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(probe_words)));
    g_probe_ptr[device] = static_cast<uint32_t*>(ptr);
  }
  *out = g_probe_ptr[device];
  return PF_OK;
}
}  // namespace

int streams_run_concurrently(hipStream_t a, hipStream_t b, bool* out) {
  *out = false;
  std::lock_guard<std::mutex> lock(g_probe_mu);
  uint32_t* words = nullptr;
  int st = probe_words_on_current_device(&words);
  if (st != PF_OK) return st;
  uint32_t seen = 0;
  // Cleared on `a` and waited for there: no other stream of the device is touched.
  hipError_t e = hipMemsetAsync(words, 0, 2 * sizeof(uint32_t), a);
  if (e == hipSuccess) e = hipStreamSynchronize(a);
  if (e == hipSuccess) {
    constexpr uint64_t kMaxTicks = 200000;  // 2 ms of the 100 MHz clock
    hipLaunchKernelGGL(probe_wait_kernel, dim3(1), dim3(64), 0, a, words, words + 1, kMaxTicks);
    hipLaunchKernelGGL(probe_post_kernel, dim3(1), dim3(64), 0, b, words);
    e = hipGetLastError();
  }
  // Wait for both whatever was launched: the next probe reuses the words.
  const hipError_t ea = hipStreamSynchronize(a);
  const hipError_t eb = hipStreamSynchronize(b);
  if (e == hipSuccess) e = ea != hipSuccess ? ea : eb;
  if (e == hipSuccess) e = hipMemcpyAsync(&seen, words + 1, sizeof(seen), hipMemcpyDeviceToHost, a);
  if (e == hipSuccess) e = hipStreamSynchronize(a);
  if (e != hipSuccess) st = fail_hip(e, "stream concurrency probe");
  *out = seen != 0;
  return st;
}

int launch_plain_copy(void* dst, const void* src, uint64_t bytes, int unroll, hipStream_t s) {
  if (bytes == 0) return PF_OK;
  if ((bytes & 15ull) != 0 || (reinterpret_cast<uint64_t>(dst) & 15ull) != 0 ||
      (reinterpret_cast<uint64_t>(src) & 15ull) != 0) {
    return fail(PF_ERR_INVALID_ARGUMENT, "plain copy needs 16-byte aligned pointers and size");
  }
  if (unroll == 0) {
    constexpr uint64_t kTile = kTileLanes * 16;
    const uint64_t n = (bytes + kTile - 1) / kTile;
    // Exactly one workgroup per tile, like the gather / scatter grids: a
    // yardstick that launched idle workgroups (a 65 536-wide grid rounded up to
    // whole rows: 18 % of them for a 327 MB copy) read 4 % low.
    if (n > 0x7FFFFFFFull) return fail(PF_ERR_INVALID_ARGUMENT, "plain copy too large");
    hipLaunchKernelGGL(plain_tiles_kernel<kTileLanes>, dim3(static_cast<uint32_t>(n), 1, 1),
                       dim3(kTileLanes, 1, 1), 0, s, reinterpret_cast<uint64_t>(dst),
                       reinterpret_cast<uint64_t>(src), bytes);
    hipError_t e0 = hipGetLastError();
    if (e0 != hipSuccess) return fail_hip(e0, "plain_tiles_kernel launch");
    return PF_OK;
  }
  const uint64_t tile = tile_bytes(unroll);
  uint64_t tiles = (bytes + tile - 1) / tile;
  uint32_t gx = static_cast<uint32_t>(tiles < kMaxGridX ? tiles : kMaxGridX);
  dim3 grid(gx, 1, 1), block(kLanes, 1, 1);
  const uint64_t d = reinterpret_cast<uint64_t>(dst);
  const uint64_t c = reinterpret_cast<uint64_t>(src);
  switch (unroll) {
    case 1: hipLaunchKernelGGL(plain_copy_kernel<1>, grid, block, 0, s, d, c, bytes); break;
    case 2: hipLaunchKernelGGL(plain_copy_kernel<2>, grid, block, 0, s, d, c, bytes); break;
    case 4: hipLaunchKernelGGL(plain_copy_kernel<4>, grid, block, 0, s, d, c, bytes); break;
    case 8: hipLaunchKernelGGL(plain_copy_kernel<8>, grid, block, 0, s, d, c, bytes); break;
    default: return fail(PF_ERR_INVALID_ARGUMENT, "unsupported tile unroll %d", unroll);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail_hip(e, "plain_copy_kernel launch");
  return PF_OK;
}

int launch_table_upload(uint64_t dst, uint64_t src, uint64_t bytes, hipStream_t s) {
  const uint64_t n = bytes / 16;
  if (n == 0) return PF_OK;
  if ((bytes & 15ull) != 0 || ((dst | src) & 15ull) != 0 || n > 0xFFFFFFFFull - (kMaxUploadWorkgroups * kLanes)) {
    return fail(PF_ERR_INVALID_ARGUMENT, "table upload of %llu bytes", static_cast<unsigned long long>(bytes));
  }
  const uint64_t groups = (n + kLanes - 1) / kLanes;
  const dim3 grid(static_cast<uint32_t>(groups < kMaxUploadWorkgroups ? groups : kMaxUploadWorkgroups), 1, 1);
  hipLaunchKernelGGL(table_upload_kernel, grid, dim3(kLanes, 1, 1), 0, s, dst, src, static_cast<uint32_t>(n));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail_hip(e, "table_upload_kernel launch");
  return PF_OK;
}

namespace {
// Launch of a descriptor copy: a row per wavefront while the largest row is
// half a wavefront's tile and there are rows for more than kFewRows workgroups,
// otherwise a row per workgroup, x over descriptors and y over the tiles of the
// largest one.  From 4 KiB rows on both reach the link's rate in a long batch and
// a row per workgroup is ahead in a short one (437 rows of 4 KiB, there and back
// 78.6 against 79.5 us); few rows are a compute unit's work each (48 rows of 1500
// bytes 25.3 against 25.9).  The kernels stride over what the grid does not cover;
// `max_workgroups` (0 = no cap) bounds the whole launch.
constexpr uint64_t kWaveRowBytes = 2048;
constexpr uint64_t kFewRows = 64;

struct RowsGrid {
  uint32_t x, y;
  bool waves;  // a row per wavefront
};
RowsGrid rows_grid(uint64_t n, uint64_t max_size, uint32_t max_workgroups) {
  constexpr uint64_t kWaves = kLanes / kWave;
  if (max_size <= kWaveRowBytes && n > kFewRows) {
    uint64_t gx = (n + kWaves - 1) / kWaves;
    if (max_workgroups != 0 && gx > max_workgroups) gx = max_workgroups;
    if (gx > kMaxGridX) gx = kMaxGridX;
    return {static_cast<uint32_t>(gx), 1, true};
  }
  constexpr uint64_t kTile = tile_bytes(kDescUnroll);
  uint64_t gx = n < kMaxGridX ? n : kMaxGridX;
  uint64_t gy = (max_size + kTile - 1) / kTile;
  if (gy < 1) gy = 1;
  if (gy > 64) gy = 64;
  if (max_workgroups != 0) {
    while (gx * gy > max_workgroups && gy > 1) gy >>= 1;
    if (gx * gy > max_workgroups) gx = max_workgroups / gy ? max_workgroups / gy : 1;
  }
  // Keep the launch to a few million workgroups; a smaller grid only means
  // more iterations per workgroup.
  while (gx * gy > (1ull << 22) && gy > 1) gy >>= 1;
  return {static_cast<uint32_t>(gx), static_cast<uint32_t>(gy), false};
}

template <bool HOST_IS_SRC, typename Rows>
void launch_rows(const Rows rows, uint64_t n, uint64_t max_size, hipStream_t s,
                 uint32_t max_workgroups) {
  const RowsGrid g = rows_grid(n, max_size, max_workgroups);
  const dim3 grid(g.x, g.y, 1), block(kLanes, 1, 1);
  if (g.waves) {
    hipLaunchKernelGGL((desc_copy_waves_kernel<kDescUnroll, HOST_IS_SRC, Rows>), grid, block, 0, s,
                       rows, static_cast<uint32_t>(n));
  } else {
    hipLaunchKernelGGL((desc_copy_kernel<kDescUnroll, HOST_IS_SRC, Rows>), grid, block, 0, s, rows,
                       static_cast<uint32_t>(n));
  }
}

template <bool HOST_IS_SRC>
void launch_packing(const uint64_t* table, uint64_t n, uint64_t n_link, uint64_t max_size,
                    uint32_t link_workgroups, hipStream_t s, uint32_t max_workgroups) {
  const RowsGrid g = rows_grid(n, max_size, max_workgroups);
  // (Rows of the share are a tile at most: those of the grid's first layer move it.)
  const uint32_t link_groups = n_link == 0 ? 0 : link_workgroups;
  const dim3 grid(g.x + link_groups, g.y, 1), block(kLanes, 1, 1);
  const Rows3<true> rows{table};
  const Rows3<false> link{table + 3 * n};
  if (g.waves) {
    hipLaunchKernelGGL((desc_pack_kernel<kDescUnroll, HOST_IS_SRC, kWave>), grid, block, 0, s, rows,
                       static_cast<uint32_t>(n), link, static_cast<uint32_t>(n_link), link_groups);
  } else {
    hipLaunchKernelGGL((desc_pack_kernel<kDescUnroll, HOST_IS_SRC, kLanes>), grid, block, 0, s, rows,
                       static_cast<uint32_t>(n), link, static_cast<uint32_t>(n_link), link_groups);
  }
}
}  // namespace

int launch_desc_copy(const uint64_t* table, uint64_t n, uint64_t max_size, bool host_is_src,
                     hipStream_t s, uint32_t max_workgroups) {
  if (n == 0) return PF_OK;
  if (host_is_src) {
    launch_rows<true>(Rows3<false>{table}, n, max_size, s, max_workgroups);
  } else {
    launch_rows<false>(Rows3<false>{table}, n, max_size, s, max_workgroups);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail_hip(e, "desc_copy_kernel launch");
  return PF_OK;
}

int launch_desc_pack(const uint64_t* table, uint64_t n, uint64_t n_link, uint64_t max_size,
                     bool host_is_src, hipStream_t s, uint32_t max_workgroups,
                     uint32_t link_workgroups) {
  if (n == 0) return PF_OK;
  if (host_is_src) {
    launch_packing<true>(table, n, n_link, max_size, link_workgroups, s, max_workgroups);
  } else {
    launch_packing<false>(table, n, n_link, max_size, link_workgroups, s, max_workgroups);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail_hip(e, "desc_pack_kernel launch");
  return PF_OK;
}

}  // namespace pf

// ---------------------------------------------------------------------------
// Descriptor copy that allocates nothing
// ---------------------------------------------------------------------------
//
// The kernel backend keeps its descriptor table in device memory it allocates
// (and grows) on demand.  Callers that must not allocate get the same copy with
// the table in a fixed array that is part of the library's device image.  Every
// GPU the library runs on holds its own copy of the array, at its own address,
// until the process ends, and every call on a GPU shares it.  Nothing in it has
// to start at zero: a call overwrites rows [0, n) before its kernel reads
// exactly those rows.  Calls are ordered among themselves: the upload and the
// launch of a call are issued under one lock, and the upload waits (on the
// device) for an event recorded behind the previous call's kernel, whichever
// stream that ran on, so a call never overwrites rows a kernel is still
// reading.  Calls on different streams of one GPU therefore run one after the
// other; that is the price of the single table.

// Most descriptors one call takes: 32768 x 48 bytes = 1.5 MiB per GPU.
#define PF_NOALLOC_MAX_DESCS 32768u

static __device__ __align__(256) unsigned char scratch[PF_NOALLOC_MAX_DESCS * sizeof(pf_copy_desc)];

namespace {

constexpr int kNoAllocMaxDevices = 64;
// Same rule as the kernel backend: the host link wants few requesters, 16
// workgroups when the average fragment fills a 16 KiB tile, up to 64 below.
uint32_t noalloc_workgroups(uint64_t total_bytes, uint64_t n) {
  constexpr uint64_t kTile = 16384;
  const uint64_t avg = total_bytes / n ? total_bytes / n : 1;
  if (avg >= kTile) return 16;
  const uint64_t scaled = 16 * ((kTile + avg - 1) / avg);
  return static_cast<uint32_t>(scaled < 64 ? scaled : 64);
}

// Per device: the table's address, the event behind the last call's kernel, and
// whether there has been a call.  Set up on a device's first call (address and
// event are host-side objects: no device or pinned memory is allocated).
struct NoAllocDevice {
  void* table = nullptr;
  hipEvent_t last_done = nullptr;
  bool used = false;
};
std::mutex g_scratch_mu;
NoAllocDevice g_noalloc[kNoAllocMaxDevices];

// Device address of `scratch` on the current device.  The array's name is only
// a host-side handle for the symbol; the address comes from the runtime, once
// per device, and is what every later use takes.  g_scratch_mu held.
int noalloc_on_current_device(NoAllocDevice** out) {
  int device = -1;
  PF_HIP(hipGetDevice(&device));
  if (device < 0 || device >= kNoAllocMaxDevices) {
    return pf::fail(PF_ERR_INVALID_ARGUMENT, "device %d is beyond the %d this call supports",
                    device, kNoAllocMaxDevices);
  }
  NoAllocDevice& d = g_noalloc[device];
  if (d.table == nullptr) {
    void* ptr = nullptr;
    PF_HIP(hipGetSymbolAddress(reinterpret_cast<void**>(&ptr), HIP_SYMBOL(scratch)));
    if (ptr == nullptr) {
      return pf::fail(PF_ERR_DEVICE_INIT, "hipGetSymbolAddress(scratch) returned a null address");
    }
    hipEvent_t done = nullptr;
    PF_HIP(hipEventCreateWithFlags(&done, hipEventDisableTiming));
    d.last_done = done;
    d.table = ptr;
  }
  *out = &d;
  return PF_OK;
}

}  // namespace

extern "C" int pf_desc_copy_noalloc(const pf_copy_desc* copies, uint64_t n, int host_is_src,
                                    pf_stream_t s) {
  if (n == 0) return PF_OK;
  PF_REQUIRE_PTR(copies);
  if (n > PF_NOALLOC_MAX_DESCS) {
    return pf::fail(PF_ERR_INVALID_ARGUMENT,
                    "pf_desc_copy_noalloc takes at most %u descriptors per call, got %llu "
                    "(split the batch, or use pf_backend_h2d / pf_backend_d2h)",
                    PF_NOALLOC_MAX_DESCS, static_cast<unsigned long long>(n));
  }
  uint64_t max_size = 0, total_size = 0;
  for (uint64_t i = 0; i < n; ++i) {
    const pf_copy_desc& c = copies[i];
    total_size += c.size;
    if (c.size != 0 && (c.device == 0 || c.host_device == 0)) {
      // The kernel dereferences both addresses; a null one would fault the GPU.
      return pf::fail(PF_ERR_INVALID_ARGUMENT,
                      "descriptor %llu: the copy kernel needs a device address and a "
                      "device-visible host address",
                      static_cast<unsigned long long>(i));
    }
    if (c.size > max_size) max_size = c.size;
  }
  if (max_size == 0) return PF_OK;
  // Upload and launch under one lock: two threads cannot interleave their rows.
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  NoAllocDevice* dev = nullptr;
  int st = noalloc_on_current_device(&dev);
  if (st != PF_OK) return st;
  hipStream_t stream = pf::native(s);
  // The previous call's kernel may still be reading the table, on this stream
  // or another: this call's upload waits for it on the device.
  if (dev->used) PF_HIP(hipStreamWaitEvent(stream, dev->last_done, 0));
  // The caller's array is the table: one copy.  From pinned memory it is
  // asynchronous; from pageable memory the runtime stages it before returning.
  PF_HIP(hipMemcpyAsync(dev->table, copies, n * sizeof(pf_copy_desc), hipMemcpyHostToDevice, stream));
  const pf_copy_desc* rows = static_cast<const pf_copy_desc*>(dev->table);
  const uint32_t workgroups = noalloc_workgroups(total_size, n);
  if (host_is_src) {
    pf::launch_rows<true>(pf::Rows48<true>{rows}, n, max_size, stream, workgroups);
  } else {
    pf::launch_rows<false>(pf::Rows48<false>{rows}, n, max_size, stream, workgroups);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return pf::fail_hip(e, "desc_copy_kernel launch");
  PF_HIP(hipEventRecord(dev->last_done, stream));
  dev->used = true;
  return PF_OK;
}

extern "C" uint64_t pf_desc_copy_noalloc_max(void) { return PF_NOALLOC_MAX_DESCS; }
