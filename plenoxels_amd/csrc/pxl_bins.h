// pxl_bins.h -- trilinear gradients through tile bins instead of one memory atomic per corner.
//
// Measured (float32, 65537 rays x 192 samples through 160x128x145 cells, ~110 kept each): the
// backward kernel 1426 us with corner atomics; 341 us writing records, then 24 us sorting the
// runs and 127 us for the tile sums.  A 512^3 BF16 training step's 2^19 rays: 4671 us before;
// 1778 + 145 + 805 now.
// Float atomics run at the memory side at ~20-26 G requests/s device-wide (one request: a
// 64-byte segment touched by one wave instruction), and a trilinear sample's eight corners
// need four to five of them.  Here the kernels that produce gradients write one 32-byte record
// per sample (dL/dvalue and the sample's cell coordinates, plain coalesced stores) and one
// descriptor per run of consecutive samples in the same 8x8x8 tile of floor cells; the runs are
// then sorted by tile, and a workgroup per tile adds its records' corners in LDS and flushes
// the tile's 9x9x9 cells with at most ~3 requests per z row.  The clip-gradient mask belongs to
// the cell, so it is applied at that flush.
//
// The work buffer (BinLayout) is the caller's.  Record slots are fixed (ray * S + index), run
// slots per region (the rays of one wave): no allocation counters, nothing that can overflow.
#pragma once

#include <type_traits>

#include "pxl_device.h"

namespace pxl {

// A run of records of one floor-cell tile: `rank` among the tile's runs, records
// [start, start + len).
struct BinRun {
  uint32_t tile, rank, start, len;
};

struct BinItem {  // runs [begin, end) of the sorted list, all of `tile`
  uint32_t tile, begin, end, pad;
};

struct Bins {
  float4* rec;           // 2 per record: dL/dvalue; (nx, ny, nz, -)
  BinRun* runs;          // region r: [r * run_cap, ...) in the order the wave appended them
  uint32_t* n_runs;      // per region
  uint2* sorted;         // (start, len) grouped by tile
  uint32_t* ctr;         // [0] items, [1] sorted runs placed (one 64-bit sum); zeroed with tile_count
  uint32_t* tile_count;  // runs per tile
  uint32_t* tile_base;   // first sorted run of each tile
  BinItem* items;
  uint32_t n_tiles, run_cap, item_runs;
};

// Runs one ray can have: along a ray every coordinate is monotone in the sample index (each
// rounded step of its computation is), so the floor cell's tile changes at most once per tile
// boundary along each axis; a group of 64 kept samples starts a new run as well.
__host__ __device__ inline int64_t bin_ray_runs(int64_t X, int64_t Y, int64_t Z, int64_t S) {
  const int64_t cross = (X + 7) / 8 + (Y + 7) / 8 + (Z + 7) / 8;
  const int64_t most = cross + (S + 63) / 64;
  return S < most ? S : most;
}

// Where one wave's next group goes: records from `slot`, runs from region slot run0 + n.
struct BinCursor {
  uint32_t slot, run0, n;
  CellSums sums;  // nearest: the workgroup's cell sums (no slots: straight to the gradient)
};

// One group's kept samples as records slot + rank and runs.  Called by the whole wave.
// Samples that no cell takes a gradient from get no record: all of a trained grid's empty space, where
// alpha is below zero at every corner (open: not so; alpha's gradient is clipped, the colours' are zero).  256^3
// cells, 90% of them empty, no occupancy, a train step of 2^24 samples: 966 -> 558 us (664 with corner
// atomics, which skip zeros too); 64^3, 97% empty, 2^23 samples: 247 -> 80 (114).  Dense grids pay at
// most 1%.  Whether the colours are clipped is not looked at: that takes 16 to 21 more registers.
// A run goes on over dropped samples; the tiles of the kept ones are still monotone along a ray,
// so bin_ray_runs' bound holds.
__device__ __forceinline__ void emit_chunk(const KParams& P, const Bins& B, const Ray& R, int lane, int k, bool keep,
                                           bool open, const float4& gv, BinCursor& cur) {
  keep = keep && (gv.x != 0.f || gv.y != 0.f || gv.z != 0.f || (open && gv.w != 0.f));
  const uint64_t km = __ballot(keep);
  if (km == 0ull) return;
  float nx, ny, nz;
  sample_index(P, R, k, nx, ny, nz);
  uint32_t tile = 0xffffffffu;
  if (keep)
    tile = (((uint32_t)floorf(nx) >> 3) * P.occ_ty + ((uint32_t)floorf(ny) >> 3)) * P.occ_tz +
           ((uint32_t)floorf(nz) >> 3);
  const uint64_t below = km & ~(~0ull << lane);
  const uint32_t prev = (uint32_t)__shfl((int)tile, below ? 63 - __builtin_clzll(below) : lane);
  const bool head = keep && (below == 0ull || tile != prev);
  const uint64_t hm = __ballot(head);
  const uint32_t slot = cur.slot + (uint32_t)lane_rank(km);
  if (keep) {
    B.rec[2 * (size_t)slot] = gv;
    B.rec[2 * (size_t)slot + 1] = make_float4(nx, ny, nz, 0.f);
  }
  const uint32_t q = cur.n + (uint32_t)lane_rank(hm);
  if (head && q < B.run_cap) {  // bin_ray_runs bounds q; a region is never written past its end
    const uint64_t from = ~0ull << lane, later = hm & (from << 1);
    const uint64_t upto = later ? (1ull << __builtin_ctzll(later)) - 1ull : ~0ull;
    const uint32_t len = (uint32_t)__popcll(km & from & upto);
    const uint32_t rank = atomicAdd(B.tile_count + tile, 1u);
    B.runs[cur.run0 + q] = BinRun{tile, rank, slot, len};
  }
  cur.n = min(cur.n + (uint32_t)__popcll(hm), B.run_cap);
}

// Sorted-run ranges of the tiles (their order does not matter, so a workgroup takes a range
// for its tiles with one atomic) and the work items: at most item_runs runs of one tile each.
// Many runs per item save flushes (a 512^3 training step, 29 k tiles of ~130 runs: 512 runs per
// item 0.82 ms, 192 0.85, 96 1.11), few runs fill the chip when there are few tiles (48^3, 5%
// occupied, 2^20 samples: 96 runs 46 us for the whole backward, 192 58, 512 66).
constexpr int64_t kManyTiles = 4096;
__host__ __device__ constexpr int bin_item_runs(int64_t tiles) { return tiles >= kManyTiles ? 512 : 96; }

__device__ __forceinline__ uint32_t wave_prefix_add_u32(uint32_t x) {
  auto shr = [](uint32_t v, auto ctrl, auto mask) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, decltype(mask)::value, 0xf, false);
  };
  using full = std::integral_constant<int, 0xf>;
  x += shr(x, std::integral_constant<int, DPP_ROW_SHR1>{}, full{});
  x += shr(x, std::integral_constant<int, DPP_ROW_SHR2>{}, full{});
  x += shr(x, std::integral_constant<int, DPP_ROW_SHR4>{}, full{});
  x += shr(x, std::integral_constant<int, DPP_ROW_SHR8>{}, full{});
  x += shr(x, std::integral_constant<int, DPP_ROW_BCAST15>{}, std::integral_constant<int, 0xa>{});
  x += shr(x, std::integral_constant<int, DPP_ROW_BCAST31>{}, std::integral_constant<int, 0xc>{});
  return x;
}

constexpr int kTilesPerThread = 4;

__global__ __launch_bounds__(256) void k_bin_tiles(Bins B) {
  __shared__ uint64_t s_sum[4];
  __shared__ uint64_t s_base;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t t0 = (blockIdx.x * 256u + threadIdx.x) * kTilesPerThread;
  uint32_t c[kTilesPerThread], n_runs = 0u, n_items = 0u;
#pragma unroll
  for (int i = 0; i < kTilesPerThread; ++i) {
    c[i] = t0 + i < B.n_tiles ? B.tile_count[t0 + i] : 0u;
    n_runs += c[i];
    n_items += (c[i] + B.item_runs - 1u) / B.item_runs;
  }
  const uint32_t ci = wave_prefix_add_u32(n_runs), ii = wave_prefix_add_u32(n_items);
  if (lane == 63) s_sum[wave] = (uint64_t)ci << 32 | ii;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint64_t all = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
    s_base = all ? atomicAdd(reinterpret_cast<unsigned long long*>(B.ctr), (unsigned long long)all) : 0ull;
  }
  __syncthreads();
  if (n_runs == 0u) return;
  uint64_t base = s_base;
  for (int w = 0; w < wave; ++w) base += s_sum[w];
  uint32_t run = (uint32_t)(base >> 32) + ci - n_runs, item = (uint32_t)base + ii - n_items;
#pragma unroll
  for (int i = 0; i < kTilesPerThread; ++i) {
    if (c[i] == 0u) continue;
    B.tile_base[t0 + i] = run;
    for (uint32_t k = 0; k < c[i]; k += B.item_runs)
      B.items[item++] = BinItem{t0 + i, run + k, run + min(c[i], k + B.item_runs), 0u};
    run += c[i];
  }
}

// Every region's runs to their sorted places: 16 lanes per region.
__global__ __launch_bounds__(256) void k_bin_place(Bins B, uint32_t n_regions) {
  const uint32_t r = blockIdx.x * 16u + (threadIdx.x >> 4), l = threadIdx.x & 15u;
  if (r >= n_regions) return;
  const uint32_t n = B.n_runs[r];
  const BinRun* runs = B.runs + (size_t)r * B.run_cap;
  for (uint32_t i = l; i < n; i += 16u) {
    const BinRun q = runs[i];
    B.sorted[B.tile_base[q.tile] + q.rank] = make_uint2(q.start, q.len);
  }
}

// Tile sums: a workgroup per item adds the corners of its records to the tile's 9x9x9 cells in
// LDS, then the cells that were reached to grad, masked by the cell's own clip gradient, four
// lanes per cell in z order.
// The LDS sums are float64: ds_add_f32 costs ~195 clocks per wave instruction on gfx950 whatever
// the addresses, ds_add_f64 9 without and 26 with random bank conflicts, 41 when pairs of lanes
// share an address (measured; 7.2 M records took 1.40 ms with float32 sums).  A record's four
// channels sit in four lanes, so a wave instruction adds one corner of sixteen records as sixteen
// 32-byte cells, with few conflicts.
// Each of the four waves takes 64 runs at a time; their records are walked 64 at a time whatever
// the runs' lengths: a bit per record marks where a run starts, and a record's run is the number
// of marks up to it.
constexpr int kTileEdge = 9, kTileCells = kTileEdge * kTileEdge * kTileEdge;

template <int DT>
__device__ __forceinline__ float load_channel(const void* grid, size_t i) {
  if constexpr (DT == PXL_DTYPE_F32) return reinterpret_cast<const float*>(grid)[i];
  const uint32_t h = reinterpret_cast<const uint16_t*>(grid)[i];
  if constexpr (DT == PXL_DTYPE_BF16) return __uint_as_float(h << 16);
  return half_bits_to_float(h);
}

template <int DT>
__global__ __launch_bounds__(256) void k_bin_accumulate(Bins B, const void* __restrict__ grid, uint32_t X, uint32_t Y,
                                                        uint32_t Z, uint32_t TY, uint32_t TZ,
                                                        float* __restrict__ grad) {
  __shared__ double s_acc[kTileCells * 4];
  __shared__ uint64_t s_mark[4][kWave];
  __shared__ uint32_t s_start[4][kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, ch = lane & 3;
  const uint32_t n_items = B.ctr[0];
  const float* rec = reinterpret_cast<const float*>(B.rec);
  for (uint32_t it = blockIdx.x; it < n_items; it += gridDim.x) {
    const BinItem item = B.items[it];
    const uint32_t tz = item.tile % TZ, ty = (item.tile / TZ) % TY, tx = item.tile / (TZ * TY);
    const uint32_t x0 = tx * 8u, y0 = ty * 8u, z0 = tz * 8u;
    for (int i = threadIdx.x; i < kTileCells * 4; i += 256) s_acc[i] = 0.0;
    __syncthreads();
    // the waves share the runs evenly, each in batches of up to 64
    const uint32_t share = (item.end - item.begin + 3u) / 4u, first = item.begin + share * (uint32_t)wave;
    const uint32_t last = min(item.end, first + share);
    for (uint32_t b = first; b < last; b += kWave) {
      const uint2 d = b + lane < last ? B.sorted[b + lane] : make_uint2(0u, 0u);
      const uint32_t incl = wave_prefix_add_u32(d.y), excl = incl - d.y;
      const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);  // at most 64 * 64
      s_mark[wave][lane] = 0ull;
      s_start[wave][lane] = d.x - excl;
      wave_lds_sync();
      if (d.y) atomicOr(reinterpret_cast<unsigned long long*>(&s_mark[wave][excl >> 6]), 1ull << (excl & 63u));
      wave_lds_sync();
      uint32_t before = 0u;  // runs that start before this stretch of 64 records
      for (uint32_t j0 = 0; j0 < total; j0 += kWave) {
        const uint64_t marks = s_mark[wave][j0 >> 6];
        // the 64 records' loads are all issued first (lanes past the last record repeat it)
        float g[4];
        float4 n[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
          const uint32_t j = min(16u * q + ((uint32_t)lane >> 2), total - 1u - j0);
          const uint32_t r = before + (uint32_t)__popcll(marks & (~0ull >> (63u - j))) - 1u;
          const size_t slot = s_start[wave][r] + j0 + j;
          g[q] = rec[8 * slot + ch];
          n[q] = B.rec[2 * slot + 1];
        }
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
          if (j0 + 16u * q + ((uint32_t)lane >> 2) >= total) continue;
          const float bx = floorf(n[q].x), by = floorf(n[q].y), bz = floorf(n[q].z);
          const float fx = n[q].x - bx, fy = n[q].y - by, fz = n[q].z - bz;  // n >= 0: floor = trunc
          const uint32_t lx = (uint32_t)bx - x0, ly = (uint32_t)by - y0, lz = (uint32_t)bz - z0;
          // the ceil index is the floor index at an exact integer
          const uint32_t e = (lx * 81u + ly * 9u + lz) * 4u + (uint32_t)ch;
          const uint32_t ex = fx > 0.f ? 324u : 0u, ey = fy > 0.f ? 36u : 0u, ez = fz > 0.f ? 4u : 0u;
          const float gz[2] = {g[q] * fz, g[q] * (1.f - fz)}, wy[2] = {fy, 1.f - fy}, wx[2] = {fx, 1.f - fx};
#pragma unroll
          for (int c = 0; c < 8; ++c) {  // corner 4 ax + 2 ay + az, 0 = ceil
            const int ax = c >> 2, ay = (c >> 1) & 1, az = c & 1;
            unsafeAtomicAdd(&s_acc[e + (ax ? 0u : ex) + (ay ? 0u : ey) + (az ? 0u : ez)],
                            (double)((gz[az] * wy[ay]) * wx[ax]));
          }
        }
        before += (uint32_t)__popcll(marks);
      }
      wave_lds_sync();
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 4u * kTileCells; i += 256u) {
      const float v = (float)s_acc[i];
      if (v != 0.f) {
        const uint32_t cell = i >> 2;
        uint32_t x = x0 + cell / 81u, y = y0 + (cell / 9u) % 9u, z = z0 + cell % 9u;
        x = x >= X ? x - X : x;  // the ceil of the last index wraps to 0
        y = y >= Y ? y - Y : y;
        z = z >= Z ? z - Z : z;
        const size_t g = (((size_t)x * Y + y) * Z + z) * 4u + (i & 3u);
        const float raw = load_channel<DT>(grid, g);
        if (raw >= 0.f && raw <= 1.f) unsafeAtomicAdd(grad + g, v);
      }
    }
    __syncthreads();
  }
}

}  // namespace pxl
