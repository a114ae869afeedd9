// pxl_field.h -- one read of the grid for what a training step needs of the whole field: the
// alpha occupancy (which cells a sample can matter in) and the total-variation sum.
//
// Occupancy from the grid's own alpha: bit of cell (i, j, k) set when raw alpha >= 0 there
// (DILATE: at any of the corners (i+a, j+b, k+c), a,b,c in {0,1}, wrapped -- the cells a
// trilinear sample with floor cell (i, j, k) reads).  A sample whose cells all have raw alpha
// < 0 is exactly zero in the reference's chain: clamp gives alpha 0, so its colour weight and
// colour gradients vanish, and the clamp's gradient mask is 0 for every alpha it read.  NaN
// alpha counts as empty.
// TV: sum += the squared differences to the +y, +z and +x neighbours, in float64.
//
// Bound by the one read of the grid.  A workgroup covers four y rows (one wave each) x 64
// consecutive z (the lanes) and walks a slab of x planes with the loads of the plane after next
// in flight; the x neighbours are carried in registers, the z neighbour is the next lane's (DPP;
// only the wave's last lane loads one), the y neighbour the row the next wave loads as well.
// The ballots of eight planes are assembled into tile words through LDS with one barrier (one
// per plane before); the TV sum takes one atomic per workgroup (one per wave before: they all
// serialise on one address).  256^3 float32: TV 112 -> 74 us, nearest occupancy 86 -> part of one
// 97 us read with the TV sum; 512^3: TV 640 -> 416 us, dilated BF16 occupancy 379 -> 312 us.
#pragma once

#include <type_traits>

#include "pxl_device.h"

namespace pxl {

template <int DT>
__device__ __forceinline__ float load_alpha(const void* grid, size_t cell) {
  if constexpr (DT == PXL_DTYPE_F32) return reinterpret_cast<const float*>(grid)[cell * 4 + 3];
  const uint32_t h = reinterpret_cast<const uint16_t*>(grid)[cell * 4 + 3];
  if constexpr (DT == PXL_DTYPE_BF16) return __uint_as_float(h << 16);
  return half_bits_to_float(h);
}

__device__ __forceinline__ float alpha_of(float a) { return a; }
__device__ __forceinline__ float alpha_of(const float4& v) { return v.w; }

__device__ __forceinline__ double sq4(const float4& a, const float4& b) {
  const float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z, dw = a.w - b.w;
  return (double)(dx * dx) + (double)(dy * dy) + (double)(dz * dz) + (double)(dw * dw);
}

constexpr int kFieldThreads = 256;
// A workgroup per unit as long as there are units: at 512^3 the TV sum takes 416 us in 8192
// workgroups of one unit, 502 in 2048 of four.
constexpr unsigned kFieldWorkgroups = 32768;

template <int DT, bool DILATE, bool OCC, bool TV>
__global__ __launch_bounds__(kFieldThreads) void k_field(const void* __restrict__ grid, uint32_t X, uint32_t Y,
                                                         uint32_t Z, uint32_t slab, uint32_t* __restrict__ out,
                                                         double* __restrict__ sum) {
  static_assert(!TV || DT == PXL_DTYPE_F32, "the TV sum reads float32 cells");
  using Cell = typename std::conditional<TV, float4, float>::type;
  constexpr bool kNext = DILATE || TV;  // plane i needs plane i + 1
  struct Plane {
    Cell v, vy, e, ey;  // cell, its y + 1; of the last lane: z + 1, and that of y + 1
  };
  __shared__ uint64_t s_m[2][8][4];
  __shared__ double s_tv[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t TX = (X + 7u) >> 3, TY = (Y + 7u) >> 3, TZ = (Z + 7u) >> 3;
  const uint32_t planes = OCC ? TX * 8u : X;  // occupancy words cover the padded dims
  const uint32_t ZB = (TZ + 7u) >> 3, YQ = TY * 2u, XS = (planes + slab - 1u) / slab;
  const uint64_t n_units = (uint64_t)XS * YQ * ZB;
  double acc = 0.0;
  int buf = 0;
  for (uint64_t u = blockIdx.x; u < n_units; u += gridDim.x) {
    const uint32_t zb = (uint32_t)(u % ZB), yq = (uint32_t)((u / ZB) % YQ), xs = (uint32_t)(u / ((uint64_t)ZB * YQ));
    const uint32_t j = yq * 4u + (uint32_t)wave, k = zb * 64u + (uint32_t)lane;
    const bool row = j < Y, ok = row && k < Z;
    const uint32_t jc = min(j, Y - 1u), j1 = j + 1u >= Y ? 0u : j + 1u, kc = min(k, Z - 1u);
    const uint32_t end = min(zb * 64u + 64u, Z);  // one past the wave's last cell
    const bool tail = k + 1u == end;
    const uint32_t kn = end == Z ? 0u : end;
    auto load = [&](uint32_t i, uint32_t y, uint32_t z) -> Cell {
      const size_t cell = ((size_t)i * Y + y) * Z + z;
      if constexpr (TV) return load_cell<DT>(grid, (uint32_t)cell);
      else return load_alpha<DT>(grid, cell);
    };
    auto fetch = [&](uint32_t i) {
      const uint32_t ic = i < X ? i : (i == X ? 0u : X - 1u);
      Plane p{};
      p.v = load(ic, jc, kc);
      if constexpr (kNext) {
        p.vy = load(ic, j1, kc);
        if (tail) {
          p.e = load(ic, jc, kn);
          if constexpr (DILATE) p.ey = load(ic, j1, kn);
        }
      }
      return p;
    };
    // corners of plane i with alpha >= 0: the cell's own, or the four at (y + b, z + c)
    auto any_of = [&](const Plane& p) {
      uint64_t m = __ballot(ok && alpha_of(p.v) >= 0.f);
      if constexpr (DILATE) {
        const uint64_t me = __ballot(row && tail && alpha_of(p.e) >= 0.f);
        const uint64_t my = __ballot(ok && alpha_of(p.vy) >= 0.f);
        const uint64_t mey = __ballot(row && tail && alpha_of(p.ey) >= 0.f);
        m |= (m >> 1) | me | my | (my >> 1) | mey;
      }
      return m;
    };
    const uint32_t x0 = xs * slab, x1 = min(planes, x0 + slab);
    Plane cur = fetch(x0), nxt = fetch(x0 + 1u);
    uint64_t q = OCC ? any_of(cur) : 0ull;
    for (uint32_t i = x0; i < x1; ++i) {
      const Plane after = fetch(i + 2u);
      if constexpr (OCC) {
        const uint64_t qn = any_of(nxt);
        const uint64_t occ = i < X ? (DILATE ? q | qn : q) : 0ull;
        q = qn;
        if (lane == 0) s_m[buf][i & 7u][wave] = occ;
        if ((i & 7u) == 7u) {
          __syncthreads();
          if (threadIdx.x < 64u) {  // plane t >> 3 of the tile row, z tile 8 zb + (t & 7)
            const uint32_t t = threadIdx.x & 7u, p = threadIdx.x >> 3, tz = zb * 8u + t;
            if (tz < TZ) {
              uint32_t word = 0u;
#pragma unroll
              for (int w = 0; w < 4; ++w) word |= (uint32_t)((s_m[buf][p][w] >> (8u * t)) & 0xffu) << (8 * w);
              const uint32_t tile = ((i >> 3) * TY + (yq >> 1)) * TZ + tz;
              out[(size_t)tile * 16u + p * 2u + (yq & 1u)] = word;
            }
          }
          buf ^= 1;  // the next eight planes fill the other half; one barrier per eight planes
        }
      }
      if constexpr (TV) {
        float4 vz = make_float4(wave_shift_down(cur.v.x, 0.f), wave_shift_down(cur.v.y, 0.f),
                                wave_shift_down(cur.v.z, 0.f), wave_shift_down(cur.v.w, 0.f));
        if (tail) vz = cur.e;
        if (ok && i < X) {
          if (j + 1u < Y) acc += sq4(cur.v, cur.vy);
          if (k + 1u < Z) acc += sq4(cur.v, vz);
          if (i + 1u < X) acc += sq4(cur.v, nxt.v);
        }
      }
      cur = nxt;
      nxt = after;
    }
  }
  if constexpr (TV) {
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (lane == 0) s_tv[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) unsafeAtomicAdd(sum, (s_tv[0] + s_tv[1]) + (s_tv[2] + s_tv[3]));
  }
}

// Planes per slab (a multiple of 8): long ones re-read fewer planes between slabs, short ones
// give small grids enough workgroups (256^3 TV sum: 32 planes, 2048 workgroups 75 us; 16 planes
// 83; 8 planes 121).
inline uint32_t field_slab(int64_t X, int64_t Y, int64_t Z) {
  const int64_t columns = ((Y + 7) / 8 * 2) * ((Z + 63) / 64);
  uint32_t slab = 64;
  while (slab > 8 && (X + slab - 1) / slab * columns < 2048) slab /= 2;
  return slab;
}

}  // namespace pxl
