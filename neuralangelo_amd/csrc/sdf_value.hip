// SDF values of points without autograd state (the sampling passes of
// projects/neuralangelo/model.py:232-248 and the lattice of
// projects/neuralangelo/utils/mesh.py:98-118): hash-grid encoding, first layer,
// softplus and SDF head (mlp.py:55-69 with with_feat off) in one kernel.
//
// As separate launches each point's encoding (512 B in float32) and hidden layer (1 KB)
// went to memory and back, and the gather, which waits on memory, and the products, which
// wait on the matrix cores, ran one after the other.  Here a workgroup takes 64
// points: its threads gather (point, level) features into LDS as bf16 planes (one, or
// three that sum to the float32 value), each wave multiplies the 64 rows by its share of
// the hidden units and finishes softplus and head in registers; two or more workgroups
// per CU overlap their phases, and 4 B per point reach memory.  The weights come from L2
// as MFMA operands; a wave uses each once per tile.  The three point columns and the bias
// are added in float32, so a lattice's coordinates (whose low bits repeat from point to
// point) see no dropped products, and the head adds short chains, the last ones in double.
// float32 issue is mostly vector instructions (gather weights, the split of features and
// weights, softplus): eight waves with one 32-column block each, 16 waves per CU, hide
// more of the gather than four waves with two blocks in 244 registers (1925 us below).
// bf16 runs four waves of two blocks in 121 registers, the same 16 waves per CU.
// 2,146,689 points of a 2^22 x 16 x 8 float32 table, 256 hidden units: 3.18 ms as separate
// launches, 1.61 ms here; two passes of 131,072 and 524,288 points, bf16: 880 us
// and 610 us.
#include "hashgrid_dev.h"
#include "mfma.h"

namespace na {

constexpr int kSvPts = 64;

struct SdfValueParams {
  const float* x;
  int64_t n;
  float vmin, vrange;
  const void* table;
  int active;
  const void* W;  // [N, ldw]: encoder columns first, then the point's (see below)
  int64_t ldw;
  const float* b;
  const float* ws;
  const float* bs;
  float beta;
  float* out;
};

// LDS row of one point in a plane: K bf16 and 16 bytes of padding, so that eight
// consecutive rows put a 16-byte chunk on eight different bank groups
template <int K> struct SvRow { static constexpr int PITCH = K + 8; };

// Weight columns of the point, in float32: columns K .. K + 2, or in the bf16 layout
// [W_hi | W_hi | W_lo] at K, K + 3, K + 6 the sum W_hi + W_lo.
__device__ inline float sv_point_weight(const float* w, int K, int k) { return w[K + k]; }
__device__ inline float sv_point_weight(const bf16_t* w, int K, int k) {
  return bf16_to_f32(w[K + k]) + bf16_to_f32(w[K + 6 + k]);
}

// T: table and weight type (float: three planes and split weights; bf16: one plane).
// F features per level, L levels, K = L F (a multiple of 16); NB 32-column blocks per
// wave (hidden width 32 NB WAVES).
template <typename T, int F, int K, int NB, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 4) sdf_value_kernel(na_grid_desc d, SdfValueParams p) {
  constexpr bool F32 = sizeof(T) == 4;
  constexpr int Q = F32 ? 3 : 1, PITCH = SvRow<K>::PITCH, L = K / F, N = 32 * NB * WAVES;
  constexpr int kThreads = 64 * WAVES;
  __shared__ __attribute__((aligned(16))) bf16_t s_enc[Q][kSvPts][PITCH];
  __shared__ __attribute__((aligned(16))) float s_w[5][N];  // point weights x, y, z; bias; head
  __shared__ float s_x[kSvPts][3];
  __shared__ float s_sum[2 * WAVES][kSvPts];  // by wave and half of its lanes
  __shared__ int s_odd;  // a sum that is not finite
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5;
  const int64_t i0 = (int64_t)blockIdx.x * kSvPts;
  const T* table = (const T*)p.table;
  const T* W = (const T*)p.W;
  if (tid == 0) s_odd = 0;
  for (int n = tid; n < N; n += kThreads) {
#pragma unroll
    for (int k = 0; k < 3; ++k) s_w[k][n] = sv_point_weight(W + n * p.ldw, K, k);
    s_w[3][n] = p.b[n];
    s_w[4][n] = p.ws[n];
  }
  for (int k = tid; k < 3 * kSvPts; k += kThreads) {
    const int64_t g = i0 * 3 + k;
    (&s_x[0][0])[k] = p.x[g < p.n * 3 ? g : p.n * 3 - 3 + k % 3];  // past the end: the last point
  }
  __syncthreads();
  auto features = [&](int pt, int l, float (&v)[F]) {
    const LevelParams lp = level_params(d, l);
    uint32_t cell[3];
    float t[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pos_fract(normalize_coord_gather(s_x[pt][k], p.vmin, p.vrange), lp.scale, cell[k], t[k]);
    gather_cell<F, T>(table + (size_t)lp.off * F, lp, cell, t, v);
  };
#pragma unroll 2
  for (int u = 0; u < kSvPts * L / kThreads; ++u) {
    const int item = u * kThreads + tid, pt = item / L, l = item % L;
    float v[F];
#pragma unroll
    for (int f = 0; f < F; ++f) v[f] = 0.0f;
    if (l < p.active) features(pt, l, v);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      RowStore<F, bf16_t>::store(&s_enc[q][pt][l * F], v);
      if (q + 1 < Q) {
#pragma unroll
        for (int f = 0; f < F; ++f) v[f] -= bf16_to_f32(f32_to_bf16(v[f]));
      }
    }
  }
  __syncthreads();

  f32x16_t acc[2][NB], low[F32 ? 2 : 1][F32 ? NB : 1];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] = 0.0f;
        if constexpr (F32) low[i][j][r] = 0.0f;
      }
  const int n0 = wave * 32 * NB;
  const int steps = (p.active * F + 15) / 16;  // inactive levels are zero
  for (int s = 0; s < steps; ++s) {
    const int k = 16 * s + 8 * h;
    bf16x8_t a[2][Q];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < Q; ++q)
        a[i][q] = *reinterpret_cast<const bf16x8_t*>(&s_enc[q][32 * i + (lane & 31)][k]);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const T* w = W + (int64_t)(n0 + 32 * j + (lane & 31)) * p.ldw + k;
      if constexpr (F32) {
        const float4 w0 = *reinterpret_cast<const float4*>(w), w1 = *reinterpret_cast<const float4*>(w + 4);
        const f32x8_t wv = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
        bf16x8_t b[3];
        split3(wv, b);
        constexpr int kTerms[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            f32x16_t& c = t < 5 ? low[i][j] : acc[i][j];
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[kTerms[t][1]], a[i][kTerms[t][0]], c, 0, 0, 0);
          }
      } else {
        const bf16x8_t b = *reinterpret_cast<const bf16x8_t*>(w);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a[i][0], acc[i][j], 0, 0, 0);
      }
    }
  }
  // lane: point row 32 i + lane % 32; register r of block j: column n0 + 32 j + 8 (r / 4)
  // + 4 h + r % 4
  const float ib = 1.0f / p.beta;
  float px[2][3], sum[2] = {0.0f, 0.0f};
  bool odd = false;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k) px[i][k] = s_x[32 * i + (lane & 31)][k];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n = n0 + 32 * j + 8 * g + 4 * h;
      float w[5][4];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const float4 q = *reinterpret_cast<const float4*>(&s_w[k][n]);
        w[k][0] = q.x; w[k][1] = q.y; w[k][2] = q.z; w[k][3] = q.w;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float part = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          float z = acc[i][j][4 * g + c];
          if constexpr (F32) {
            z += low[i][j][4 * g + c];
            odd = odd || !(fabsf(z) < INFINITY);
          }
          z = fmaf(px[i][0], w[0][c], z);
          z = fmaf(px[i][1], w[1][c], z);
          z = fmaf(px[i][2], w[2][c], z) + w[3][c];
          part = fmaf(w[4][c], softplus_sel(z, p.beta, ib), part);
        }
        sum[i] += part;  // short chains: the head's rounding is most of the result's error
      }
    }
  if (odd) s_odd = 1;
#pragma unroll
  for (int i = 0; i < 2; ++i) s_sum[2 * wave + h][32 * i + (lane & 31)] = sum[i];
  __syncthreads();
  if constexpr (F32) {
    // values that are not finite, or too large to split into bf16 parts: the tile again
    // in float32, a thread per point and wave, which takes its own columns
    if (__builtin_expect(s_odd != 0, 0)) {
      const int pt = tid & 63;
      float total = 0.0f;
      for (int c0 = wave * 32 * NB; c0 < (wave + 1) * 32 * NB; c0 += 8) {
        float z[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) z[c] = 0.0f;
        for (int l = 0; l < p.active; ++l) {
          float v[F];
          features(pt, l, v);
#pragma unroll
          for (int f = 0; f < F; ++f)
#pragma unroll
            for (int c = 0; c < 8; ++c)
              z[c] = fmaf(v[f], (float)W[(int64_t)(c0 + c) * p.ldw + l * F + f], z[c]);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          float q = z[c];
#pragma unroll
          for (int k = 0; k < 3; ++k) q = fmaf(s_x[pt][k], s_w[k][c0 + c], q);
          total = fmaf(s_w[4][c0 + c], softplus_sel(q + s_w[3][c0 + c], p.beta, ib), total);
        }
      }
      __syncthreads();  // every thread has read s_odd's verdict and the shared rows
      s_sum[2 * wave][pt] = total;
      s_sum[2 * wave + 1][pt] = 0.0f;
      __syncthreads();
    }
  }
  if (tid < kSvPts && i0 + tid < p.n) {
    double v = p.bs[0];
#pragma unroll
    for (int q = 0; q < 2 * WAVES; ++q) v += s_sum[q][tid];
    p.out[i0 + tid] = (float)v;
  }
}

template <typename T, int F, int K>
static int launch_sdf_value(const na_grid_desc& d, const SdfValueParams& p, int64_t N, hipStream_t s) {
  constexpr int NB = sizeof(T) == 4 ? 1 : 2;
  const dim3 grid((unsigned)ceil_div(p.n, (int64_t)kSvPts));
  if (N == 256)
    hipLaunchKernelGGL((sdf_value_kernel<T, F, K, NB, 8 / NB>), grid, dim3(512 / NB), 0, s, d, p);
  else
    hipLaunchKernelGGL((sdf_value_kernel<T, F, K, 1, 4>), grid, dim3(256), 0, s, d, p);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

}  // namespace na

using namespace na;

// The shapes with an instantiation: the presets' 16 levels of 4 or 8 features (a K of 64 or
// 128, whole 16-wide steps, whose planes leave two workgroups' LDS per CU) and hidden
// widths of four or eight 32-column waves.  There one launch was faster at each measured
// count (64 points 12-16 us against 28-32, 131,072 points 1.3 to 1.7 times); other shapes take the three separate launches.
extern "C" int na_sdf_value_supported(const na_grid_desc* d, int32_t dtype, int64_t N) {
  return d && d->n_levels == 16 && (d->n_features == 4 || d->n_features == 8) &&
         (dtype == NA_F32 || dtype == NA_BF16) && (N == 128 || N == 256);
}

extern "C" int na_sdf_value(const na_grid_desc* desc, const float* points, int64_t n, float vmin,
                            float vmax, const void* table, int32_t dtype, int32_t active_levels,
                            const void* W, int64_t ldw, int64_t N, const float* b, const float* ws,
                            const float* bs, float beta, float* out, na_stream_t stream) {
  NA_CHECK_ARG(desc != nullptr, "desc is null");
  if (!na_sdf_value_supported(desc, dtype, N)) {
    set_error("na_sdf_value: 16 levels of 4 or 8 features and 128 or 256 hidden units, float32 or bf16");
    return NA_ERR_UNSUPPORTED;
  }
  NA_CHECK_ARG(n >= 0, "n < 0");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(points && table && W && b && ws && bs && out, "null pointer");
  NA_CHECK_ARG(vmax > vmin, "vmax must exceed vmin");
  const int64_t K = (int64_t)desc->n_levels * desc->n_features;
  const bool f32 = dtype == NA_F32;
  NA_CHECK_ARG(ldw >= K + (f32 ? 3 : 9) && ldw % (f32 ? 4 : 8) == 0 && ((uintptr_t)W & 15) == 0,
               "W rows must hold the encoder and point columns and keep 16-byte alignment");
  NA_CHECK_ARG(ceil_div(n, (int64_t)kSvPts) < 0x7fffffffLL, "n too large");
  int active = active_levels < desc->n_levels ? active_levels : desc->n_levels;
  if (active < 0) active = 0;
  SdfValueParams p{points, n, vmin, vmax - vmin, table, active, W, ldw, b, ws, bs, beta, out};
  hipStream_t s = (hipStream_t)stream;
  if (desc->n_features == 8)
    return f32 ? launch_sdf_value<float, 8, 128>(*desc, p, N, s)
               : launch_sdf_value<bf16_t, 8, 128>(*desc, p, N, s);
  return f32 ? launch_sdf_value<float, 4, 64>(*desc, p, N, s)
             : launch_sdf_value<bf16_t, 4, 64>(*desc, p, N, s);
}
