// Device side of one hash-grid evaluation: level table, cell and corner indices,
// weights, vectorised entry loads and row stores (the algorithm is described in
// hashgrid.hip).
#pragma once

#include "common.h"

namespace na {

struct LevelParams {
  float scale;
  uint32_t res;
  uint32_t off;
  uint32_t size;
  bool hashed;
};

__device__ inline LevelParams level_params(const na_grid_desc& d, int l) {
  LevelParams p;
  p.scale = d.scale[l];
  p.res = d.resolution[l];
  p.off = d.offset[l];
  p.size = d.offset[l + 1] - p.off;
  uint64_t r = p.res;
  p.hashed = r * r * r > (uint64_t)p.size;
  return p;
}

__device__ inline void pos_fract(float x, float scale, uint32_t& cell, float& t) {
  float pos = fmaf(scale, x, 0.5f);
  float fl = floorf(pos);
  cell = (uint32_t)(int)fl;
  t = pos - fl;
}

__device__ inline uint32_t corner_index(uint32_t x, uint32_t y, uint32_t z,
                                        const LevelParams& p) {
  if (p.hashed) {
    return (x ^ (y * 2654435761u) ^ (z * 805459861u)) & (p.size - 1u);
  }
  return (x + y * p.res + z * p.res * p.res) % p.size;
}

__device__ inline float corner_weight(int c, const float t[3]) {
  float w = (c & 1) ? t[0] : 1.0f - t[0];
  w *= (c & 2) ? t[1] : 1.0f - t[1];
  w *= (c & 4) ? t[2] : 1.0f - t[2];
  return w;
}

// The eight corner indices of one cell, as corner_index computes them.  The
// corners differ from corner 0 by fixed per-axis terms (uint32 arithmetic
// wraps the same way), so a hashed level costs two xors and a mask per corner
// and a dense level one add; both are formed and one is selected, since the
// lanes of a wave hold different levels.  The dense wrap (index % size) only
// changes corners past the grid's upper face or of points outside the unit
// cube, so it runs only when some corner of the cell needs it.
__device__ inline void cell_corners(const uint32_t (&cell)[3], const LevelParams& p,
                                    uint32_t (&id)[8]) {
  constexpr uint32_t kPy = 2654435761u, kPz = 805459861u;
  const uint32_t hx[2] = {cell[0], cell[0] + 1u};
  const uint32_t hy[2] = {cell[1] * kPy, cell[1] * kPy + kPy};
  const uint32_t hz[2] = {cell[2] * kPz, cell[2] * kPz + kPz};
  const uint32_t r1 = p.res, r2 = p.res * p.res;
  const uint32_t d0 = cell[0] + cell[1] * r1 + cell[2] * r2;
  const uint32_t dd[4] = {d0, d0 + r1, d0 + r2, d0 + r2 + r1};
  const uint32_t mask = p.size - 1u;
  bool wrap = false;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const uint32_t h = (hx[c & 1] ^ hy[(c >> 1) & 1] ^ hz[c >> 2]) & mask;
    const uint32_t d = dd[c >> 1] + (uint32_t)(c & 1);
    wrap = wrap || d >= p.size;
    id[c] = p.hashed ? h : d;
  }
  if (__builtin_expect(!p.hashed && wrap, 0)) {
#pragma unroll
    for (int c = 0; c < 8; ++c) id[c] = (dd[c >> 1] + (uint32_t)(c & 1)) % p.size;
  }
}

// Trilinear weights of the eight corners, multiplied in corner_weight's order.
__device__ inline void cell_weights(const float (&t)[3], float (&w)[8]) {
  const float wx[2] = {1.0f - t[0], t[0]}, wy[2] = {1.0f - t[1], t[1]};
  const float wz[2] = {1.0f - t[2], t[2]};
  float wxy[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) wxy[a] = wx[a & 1] * wy[a >> 1];
#pragma unroll
  for (int c = 0; c < 8; ++c) w[c] = wxy[c & 3] * wz[c >> 2];
}

// Load F table values of one entry as floats (vectorised).
template <int F, typename TT> struct EntryLoad;
template <int F> struct EntryLoad<F, float> {
  __device__ static inline void load(const float* __restrict__ p, float v[F]) {
    if constexpr (F == 8) {
      float4 a = *reinterpret_cast<const float4*>(p);
      float4 b = *reinterpret_cast<const float4*>(p + 4);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
      v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else if constexpr (F == 4) {
      float4 a = *reinterpret_cast<const float4*>(p);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    } else if constexpr (F == 2) {
      float2 a = *reinterpret_cast<const float2*>(p);
      v[0] = a.x; v[1] = a.y;
    } else {
      v[0] = p[0];
    }
  }
};
template <int F> struct EntryLoad<F, bf16_t> {
  __device__ static inline void load(const bf16_t* __restrict__ p, float v[F]) {
    if constexpr (F == 8) {
      uint4 a = *reinterpret_cast<const uint4*>(p);
      uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[2 * k] = bf16_to_f32((bf16_t)(w[k] & 0xffffu));
        v[2 * k + 1] = bf16_to_f32((bf16_t)(w[k] >> 16));
      }
    } else if constexpr (F == 4) {
      uint2 a = *reinterpret_cast<const uint2*>(p);
      v[0] = bf16_to_f32((bf16_t)(a.x & 0xffffu));
      v[1] = bf16_to_f32((bf16_t)(a.x >> 16));
      v[2] = bf16_to_f32((bf16_t)(a.y & 0xffffu));
      v[3] = bf16_to_f32((bf16_t)(a.y >> 16));
    } else if constexpr (F == 2) {
      uint32_t a = *reinterpret_cast<const uint32_t*>(p);
      v[0] = bf16_to_f32((bf16_t)(a & 0xffffu));
      v[1] = bf16_to_f32((bf16_t)(a >> 16));
    } else {
      v[0] = bf16_to_f32(p[0]);
    }
  }
};

template <int F, typename TO> struct RowStore;
template <int F> struct RowStore<F, float> {
  __device__ static inline void store(float* __restrict__ p, const float v[F]) {
    if constexpr (F == 8) {
      *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
    } else if constexpr (F == 4) {
      *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    } else if constexpr (F == 2) {
      *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
    } else {
      p[0] = v[0];
    }
  }
};
template <int F> struct RowStore<F, bf16_t> {
  __device__ static inline void store(bf16_t* __restrict__ p, const float v[F]) {
    uint32_t w[(F + 1) / 2];
#pragma unroll
    for (int k = 0; k < F / 2; ++k)
      w[k] = (uint32_t)f32_to_bf16(v[2 * k]) | ((uint32_t)f32_to_bf16(v[2 * k + 1]) << 16);
    if constexpr (F == 8) {
      *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
    } else if constexpr (F == 4) {
      *reinterpret_cast<uint2*>(p) = make_uint2(w[0], w[1]);
    } else if constexpr (F == 2) {
      *reinterpret_cast<uint32_t*>(p) = w[0];
    } else {
      p[0] = f32_to_bf16(v[0]);
    }
  }
};

// acc = sum over the eight corners of the cell of weight * entry (corner order
// 0..7, as the per-corner loops accumulate).
template <int F, typename TT>
__device__ inline void gather_cell(const TT* __restrict__ tab, const LevelParams& p,
                                   const uint32_t (&cell)[3], const float (&t)[3], float (&acc)[F]) {
  uint32_t id[8];
  float w[8];
  cell_corners(cell, p, id);
  cell_weights(t, w);
#pragma unroll
  for (int f = 0; f < F; ++f) acc[f] = 0.0f;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    float v[F];
    EntryLoad<F, TT>::load(tab + (size_t)id[c] * F, v);
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] = fmaf(w[c], v[f], acc[f]);
  }
}

// Input point -> unit-cube coordinate: u = (x - vmin) / vrange
// (projects/neuralangelo/utils/modules.py:82-83; vmin = 0, vrange = 1 is the
// tcnn convention of inputs already in [0,1]).
__device__ inline float normalize_coord(float x, float vmin, float vrange) {
  return (x - vmin) / vrange;
}

// The same coordinate for the gather kernels, where the division is a visible
// share of the work: a positive normal power-of-two range divides exactly by
// an exponent shift.
__device__ inline float normalize_coord_gather(float x, float vmin, float vrange) {
  const uint32_t b = __float_as_uint(vrange);
  if ((b & 0x807fffffu) == 0u && (b >> 23) != 0u) return ldexpf(x - vmin, 127 - (int)(b >> 23));
  return (x - vmin) / vrange;
}

}  // namespace na
