// Per-ray operators of the NeuS / Neuralangelo renderer.
//
// Everything here is memory- or latency-bound elementwise/scan work.  Scans
// along a ray (CDF, transmittance, merge) run one ray per lane with the
// ray's prefix data staged in LDS, in a fixed sequential order so that the
// discrete outputs (searchsorted indices, merge order) are reproducible
// bit-for-bit.  FMA contraction is disabled in this file so every float op
// rounds exactly where the reference formula rounds.
#include "common.h"

#pragma clang fp contract(off)

namespace na {

constexpr int kRayBlock = 64;  // rays per workgroup for the per-ray scan kernels
constexpr int kCompU = 8;      // samples whose loads a compositing thread issues together

__device__ inline float sigmoidf_(float x) { return 1.0f / (1.0f + expf(-x)); }

// torch.min over two values: NaN propagates.
__device__ inline float tmin(float a, float b) { return (a != a || a < b) ? a : b; }

// ---------------------------------------------------------------------------
// bounds + coarse sampling
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
ray_bounds_sample_kernel(const float* __restrict__ center, const float* __restrict__ ray,
                         const float* __restrict__ rands, int64_t R, int N,
                         float* __restrict__ near_out, float* __restrict__ far_out,
                         uint8_t* __restrict__ outside_out, float* __restrict__ dists) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R * N) return;
  int64_t r = t / N;
  int i = (int)(t % N);
  float c0 = center[r * 3], c1 = center[r * 3 + 1], c2 = center[r * 3 + 2];
  float v0 = ray[r * 3], v1 = ray[r * 3 + 1], v2 = ray[r * 3 + 2];
  float ctc = c0 * c0 + c1 * c1 + c2 * c2;
  float ctv = c0 * v0 + c1 * v1 + c2 * v2;
  float disc = ctv * ctv - (ctc - 1.0f);
  float sq = sqrtf(disc);
  float nr = -ctv - sq;
  float fr = -ctv + sq;
  nr = (nr != nr) ? nr : (nr > 0.0f ? nr : 0.0f);  // relu_, NaN kept
  bool out = nr != nr;
  if (out) {
    nr = 1.0f;
    fr = 1.2f;
  }
  if (i == 0) {
    near_out[r] = nr;
    far_out[r] = fr;
    outside_out[r] = out ? 1 : 0;
  }
  float u = rands ? rands[t] : 0.5f;
  float a = u + (float)i;
  float d = a / (float)N * (fr - nr) + nr;
  dists[t] = d;
}

// Raw sphere crossings, no clamping: t = -<c,v> -/+ sqrt(<c,v>^2 - (<c,c> - r^2)),
// NaN for a ray that misses.  One thread per ray.
__global__ void __launch_bounds__(256)
sphere_crossings_kernel(const float* __restrict__ center, const float* __restrict__ ray, int64_t R,
                        float r2, float* __restrict__ near_out, float* __restrict__ far_out) {
  int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  float c0 = center[r * 3], c1 = center[r * 3 + 1], c2 = center[r * 3 + 2];
  float v0 = ray[r * 3], v1 = ray[r * 3 + 1], v2 = ray[r * 3 + 2];
  float ctc = c0 * c0 + c1 * c1 + c2 * c2;
  float ctv = c0 * v0 + c1 * v1 + c2 * v2;
  float sq = sqrtf(ctv * ctv - (ctc - r2));
  near_out[r] = -ctv - sq;
  far_out[r] = -ctv + sq;
}

// Pixel-centre camera rays.  Pixel p of an H x W image sits at
// (x, y) = (p mod W + 0.5, p div W + 0.5); its camera-space point is
// K^-1 [x, y, 1]^T, and the inverse of the world-to-camera pose [R | t] maps it
// to the world: X_w = R^T X_c - R^T t.  center = -R^T t, ray = X_w - center
// (depth 1, not unit), ray_unit = ray / max(|ray|, 1e-12).  K^-1 comes from the
// adjugate in double precision.  One thread per (camera, ray); ray_idx [B, R]
// picks the pixels (NULL: pixel j for ray j).
__global__ void __launch_bounds__(256)
camera_rays_kernel(const float* __restrict__ pose, const float* __restrict__ intr, int64_t B,
                   int64_t W, const int64_t* __restrict__ ray_idx, int64_t R,
                   float* __restrict__ center, float* __restrict__ ray,
                   float* __restrict__ ray_unit) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= B * R) return;
  const int64_t b = t / R;
  const int64_t p = ray_idx ? ray_idx[t] : t - b * R;
  const float* K = intr + b * 9;
  const double k0 = K[0], k1 = K[1], k2 = K[2], k3 = K[3], k4 = K[4], k5 = K[5], k6 = K[6],
               k7 = K[7], k8 = K[8];
  const double c00 = k4 * k8 - k5 * k7, c01 = k5 * k6 - k3 * k8, c02 = k3 * k7 - k4 * k6;
  const double rdet = 1.0 / (k0 * c00 + k1 * c01 + k2 * c02);
  float Ki[9];
  Ki[0] = (float)(c00 * rdet);
  Ki[1] = (float)((k2 * k7 - k1 * k8) * rdet);
  Ki[2] = (float)((k1 * k5 - k2 * k4) * rdet);
  Ki[3] = (float)(c01 * rdet);
  Ki[4] = (float)((k0 * k8 - k2 * k6) * rdet);
  Ki[5] = (float)((k2 * k3 - k0 * k5) * rdet);
  Ki[6] = (float)(c02 * rdet);
  Ki[7] = (float)((k1 * k6 - k0 * k7) * rdet);
  Ki[8] = (float)((k0 * k4 - k1 * k3) * rdet);
  const float px = (float)(p % W) + 0.5f, py = (float)(p / W) + 0.5f;
  float xc[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) xc[k] = Ki[k * 3] * px + Ki[k * 3 + 1] * py + Ki[k * 3 + 2];
  const float* P = pose + b * 12;  // row-major [3, 4]: P[r*4 + c]
  float cw[3], rw[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    cw[k] = -(P[k] * P[3] + P[4 + k] * P[7] + P[8 + k] * P[11]);
    const float xw = P[k] * xc[0] + P[4 + k] * xc[1] + P[8 + k] * xc[2] + cw[k];
    rw[k] = xw - cw[k];
  }
  float nrm = sqrtf(rw[0] * rw[0] + rw[1] * rw[1] + rw[2] * rw[2]);
  nrm = nrm > 1e-12f ? nrm : 1e-12f;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    center[t * 3 + k] = cw[k];
    ray[t * 3 + k] = rw[k];
    if (ray_unit) ray_unit[t * 3 + k] = rw[k] / nrm;
  }
}

// Evenly stratified distances between per-ray bounds (a NULL bound array means
// the constant): d[r,i] = (i + u) / N * (hi - lo) + lo, u = rands[r,i] or 0.5.
__global__ void __launch_bounds__(256)
sample_dists_kernel(const float* __restrict__ lo, const float* __restrict__ hi, float lo_c,
                    float hi_c, const float* __restrict__ rands, int64_t R, int N,
                    float* __restrict__ dists) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R * N) return;
  int64_t r = t / N;
  int i = (int)(t % N);
  float a = lo ? lo[r] : lo_c;
  float b = hi ? hi[r] : hi_c;
  float u = rands ? rands[t] : 0.5f;
  dists[t] = (u + (float)i) / (float)N * (b - a) + a;
}

// ---------------------------------------------------------------------------
// inverse-CDF sampling (shared by na_sample_pdf and na_hier_resample)
// cdf: LDS row of N floats (cdf[0] = 0, cdf[i] = prefix of pdf[0..i-1])
// ---------------------------------------------------------------------------
__device__ inline float linspace_val(int idx, int steps) {
  // torch.linspace(0, 1, steps) in float32
  float step = (1.0f - 0.0f) / (float)(steps - 1);
  int halfway = steps / 2;
  if (idx < halfway) return 0.0f + step * (float)idx;
  return 1.0f - step * (float)(steps - idx - 1);
}

// sample j of Nf from the cdf of N - 1 intervals (element i at cdf[i * stride])
__device__ inline float pdf_sample(const float* cdf, int stride, int N, const float* bins, int j,
                                   int Nf) {
  float u = 0.5f * (linspace_val(j, Nf + 1) + linspace_val(j + 1, Nf + 1));
  // searchsorted right=True: first index with cdf > u
  int lo = 0, hi = N;
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (cdf[mid * stride] <= u) lo = mid + 1;
    else hi = mid;
  }
  int idx = lo;
  int low = idx - 1 > 0 ? idx - 1 : 0;
  int high = idx < N - 1 ? idx : N - 1;
  float cl = cdf[low * stride], ch = cdf[high * stride];
  float dmin = bins[low], dmax = bins[high];
  float t = (u - cl) / (ch - cl + 1e-8f);
  return dmin + t * (dmax - dmin);
}

__device__ inline void pdf_sample_row(const float* __restrict__ cdf, int stride, int N,
                                      const float* __restrict__ bins, int Nf,
                                      float* __restrict__ out) {
  for (int j = 0; j < Nf; ++j) out[j] = pdf_sample(cdf, stride, N, bins, j, Nf);
}

// cdf column layout in LDS: element i of lane l at s[i * kRayBlock + l]
__global__ void __launch_bounds__(kRayBlock)
sample_pdf_kernel(const float* __restrict__ bins, const float* __restrict__ weights, int64_t R,
                  int N, int Nf, float* __restrict__ out) {
  extern __shared__ float s_cdf[];
  const int l = threadIdx.x;
  const int64_t r = (int64_t)blockIdx.x * kRayBlock + l;
  if (r >= R) return;
  const float* w = weights + r * (N - 1);
  float l1 = 0.0f;
  for (int i = 0; i < N - 1; ++i) l1 = l1 + fabsf(w[i]);
  float denom = l1 > 1e-12f ? l1 : 1e-12f;
  float* cdf = s_cdf + l;
  float acc = 0.0f;
  cdf[0] = 0.0f;
  for (int i = 0; i < N - 1; ++i) {
    acc = acc + w[i] / denom;
    cdf[(i + 1) * kRayBlock] = acc;
  }
  pdf_sample_row(cdf, kRayBlock, N, bins + r * N, Nf, out + r * Nf);
}

// One hierarchical round per ray by a wave for kHierRays rays.  Everything that is
// independent per interval, sample or output runs over the lanes; only the three prefix
// chains (transmittance with the weights' sum, the cdf) run in one lane per ray, on
// LDS values, in the canonical order, so every bit is the lane-per-ray kernel's.
// That one walked 80 intervals and 96 merge steps of dependent memory and divisions
// per lane: 72 us at 1,024 and at 8,192 rays (64 + 16 samples); here 19 and 25 us.
// Rows that are sorted (as sampling makes them) merge by rank; others by the same
// two-pointer walk as before.
constexpr int kHierRays = 4, kHierMaxFine = 256;

__global__ void __launch_bounds__(64)
hier_resample_wave_kernel(const float* __restrict__ dists, const float* __restrict__ sdfs,
                          int64_t R, int N, float inv_s, int Nf, float* __restrict__ merged,
                          float* __restrict__ fine, int32_t* __restrict__ pos_coarse,
                          int32_t* __restrict__ pos_fine) {
  extern __shared__ float s_rows[];
  __shared__ float s_denom[kHierRays];
  __shared__ int s_unsorted[kHierRays];
  const int lane = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.x * kHierRays;
  const int nr = R - r0 < kHierRays ? (int)(R - r0) : kHierRays;
  float* s_d = s_rows;                      // [ray][N] distances
  float* s_c = s_d + kHierRays * N;         // [ray][N] alphas, weights, cdf
  float* s_f = s_c + kHierRays * N;         // [ray][Nf] fine distances
  if (lane < kHierRays) s_unsorted[lane] = 0;
  for (int k = lane; k < nr * N; k += 64) s_d[k] = dists[r0 * N + k];
  // interval alphas (model.py:251-264)
  for (int k = lane; k < nr * (N - 1); k += 64) {
    const int q = k / (N - 1), i = k % (N - 1);
    const float* d = dists + (r0 + q) * N + i;
    const float* s = sdfs + (r0 + q) * N + i;
    const float sp = s[0], sn = s[1], dp = d[0], dn = d[1];
    float prev_cos = 0.0f;
    if (i > 0) {
      const float s0 = s[-1], d0 = d[-1];
      prev_cos = (sp - s0) / (dp - d0 + 1e-5f);
    }
    float mid = (sp + sn) * 0.5f;
    float cosv = (sn - sp) / (dn - dp + 1e-5f);
    float cr = tmin(prev_cos, cosv);
    float intv = dn - dp;
    float est_prev = mid - cr * intv * 0.5f;
    float est_next = mid + cr * intv * 0.5f;
    float pc = sigmoidf_(est_prev * inv_s);
    float nc = sigmoidf_(est_next * inv_s);
    float a = (pc - nc) / (pc + 1e-5f);
    a = a < 0.0f ? 0.0f : (a > 1.0f ? 1.0f : a);
    s_c[q * N + i + 1] = a;
  }
  __syncthreads();
  // compositing weights (render.py:94-98) and their sum, in order
  if (lane < nr) {
    float* c = s_c + lane * N;
    float T = 1.0f, l1 = 0.0f;
    for (int i0 = 1; i0 < N; i0 += kCompU) {
      float av[kCompU];
#pragma unroll
      for (int u = 0; u < kCompU; ++u) av[u] = i0 + u < N ? c[i0 + u] : 0.0f;
#pragma unroll
      for (int u = 0; u < kCompU; ++u) {
        if (i0 + u >= N) break;
        const float a = av[u];
        float w = a * T;
        T = T * (1.0f - a);
        c[i0 + u] = w;
        l1 = l1 + fabsf(w);
      }
    }
    s_denom[lane] = l1 > 1e-12f ? l1 : 1e-12f;
  }
  __syncthreads();
  for (int k = lane; k < nr * (N - 1); k += 64) {
    const int q = k / (N - 1), i = k % (N - 1);
    s_c[q * N + i + 1] = s_c[q * N + i + 1] / s_denom[q];
  }
  __syncthreads();
  // pdf -> cdf in place (nerf_util.py:50-53)
  if (lane < nr) {
    float* c = s_c + lane * N;
    float acc = 0.0f;
    c[0] = 0.0f;
    for (int i0 = 1; i0 < N; i0 += kCompU) {
      float pv[kCompU];
#pragma unroll
      for (int u = 0; u < kCompU; ++u) pv[u] = i0 + u < N ? c[i0 + u] : 0.0f;
#pragma unroll
      for (int u = 0; u < kCompU; ++u) {
        if (i0 + u >= N) break;
        acc = acc + pv[u];
        c[i0 + u] = acc;
      }
    }
  }
  __syncthreads();
  for (int k = lane; k < nr * Nf; k += 64) {
    const int q = k / Nf, j = k % Nf;
    const float v = pdf_sample(s_c + q * N, 1, N, s_d + q * N, j, Nf);
    s_f[k] = v;
    fine[r0 * Nf + k] = v;
  }
  __syncthreads();
  for (int k = lane; k < nr * Nf; k += 64)
    if (k % Nf != 0 && !(s_f[k - 1] <= s_f[k])) s_unsorted[k / Nf] = 1;
  for (int k = lane; k < nr * N; k += 64)
    if (k % N != 0 && !(s_d[k - 1] <= s_d[k])) s_unsorted[k / N] = 1;
  __syncthreads();
  // stable merge, coarse first on ties
  const int W = N + Nf;
  for (int k = lane; k < nr * W; k += 64) {
    const int q = k / W, i = k % W;
    if (s_unsorted[q]) continue;
    const bool coarse = i < N;
    const float* d = s_d + q * N;
    const float* f = s_f + q * Nf;
    const float v = coarse ? d[i] : f[i - N];
    // coarse: the fine values below it; fine: the coarse values not above it
    int lo = 0, hi = coarse ? Nf : N;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (coarse ? f[mid] < v : !(v < d[mid])) lo = mid + 1;
      else hi = mid;
    }
    const int at = lo + (coarse ? i : i - N);
    merged[(r0 + q) * W + at] = v;
    if (coarse) pos_coarse[(r0 + q) * N + i] = at;
    else pos_fine[(r0 + q) * Nf + i - N] = at;
  }
  if (lane < nr && s_unsorted[lane]) {
    const float* d = s_d + lane * N;
    const float* f = s_f + lane * Nf;
    int i = 0, j = 0;
    for (int k = 0; k < W; ++k) {
      const bool take = (j >= Nf) || (i < N && !(f[j] < d[i]));
      merged[(r0 + lane) * W + k] = take ? d[i] : f[j];
      if (take) pos_coarse[(r0 + lane) * N + i++] = k;
      else pos_fine[(r0 + lane) * Nf + j++] = k;
    }
  }
}

// The same round with a lane per ray, where that is better or the only way: rows whose fine
// samples do not fit the wave kernel's LDS, and many rays of a few samples, which leave the
// wave kernel's lanes idle.
__global__ void __launch_bounds__(kRayBlock)
hier_resample_kernel(const float* __restrict__ dists, const float* __restrict__ sdfs, int64_t R,
                     int N, float inv_s, int Nf, float* __restrict__ merged,
                     float* __restrict__ fine, int32_t* __restrict__ pos_coarse,
                     int32_t* __restrict__ pos_fine) {
  extern __shared__ float s_cdf[];
  const int l = threadIdx.x;
  const int64_t r = (int64_t)blockIdx.x * kRayBlock + l;
  if (r >= R) return;
  const float* d = dists + r * N;
  const float* s = sdfs + r * N;
  float* cdf = s_cdf + l;
  // pass 1: interval alphas (model.py:251-264) and compositing weights
  // (render.py:94-98); the weights are parked in the cdf slots 1..N-1.
  float T = 1.0f;
  float prev_cos = 0.0f;
  float l1 = 0.0f;
  // (the loads of kCompU intervals go out before their sequential arithmetic)
  float sp = s[0], dp = d[0];
  for (int i0 = 0; i0 < N - 1; i0 += kCompU) {
    float sv[kCompU], dv[kCompU];
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int i = i0 + u + 1;
      sv[u] = i < N ? s[i] : 0.0f;
      dv[u] = i < N ? d[i] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int i = i0 + u;
      if (i >= N - 1) break;
      const float sn = sv[u], dn = dv[u];
      float mid = (sp + sn) * 0.5f;
      float cosv = (sn - sp) / (dn - dp + 1e-5f);
      float cr = tmin(prev_cos, cosv);
      prev_cos = cosv;
      float intv = dn - dp;
      float est_prev = mid - cr * intv * 0.5f;
      float est_next = mid + cr * intv * 0.5f;
      float pc = sigmoidf_(est_prev * inv_s);
      float nc = sigmoidf_(est_next * inv_s);
      float a = (pc - nc) / (pc + 1e-5f);
      a = a < 0.0f ? 0.0f : (a > 1.0f ? 1.0f : a);
      float w = a * T;
      T = T * (1.0f - a);
      cdf[(i + 1) * kRayBlock] = w;
      l1 = l1 + fabsf(w);
      sp = sn;
      dp = dn;
    }
  }
  // pass 2: pdf -> cdf in place (nerf_util.py:50-53)
  float denom = l1 > 1e-12f ? l1 : 1e-12f;
  float acc = 0.0f;
  cdf[0] = 0.0f;
  for (int i = 0; i < N - 1; ++i) {
    acc = acc + cdf[(i + 1) * kRayBlock] / denom;
    cdf[(i + 1) * kRayBlock] = acc;
  }
  float* f = fine + r * Nf;
  pdf_sample_row(cdf, kRayBlock, N, d, Nf, f);
  // stable merge of the sorted coarse row and the (sorted) fine row
  float* m = merged + r * (N + Nf);
  int i = 0, j = 0;
  for (int k = 0; k < N + Nf; ++k) {
    bool take_coarse = (j >= Nf) || (i < N && !(f[j] < d[i]));
    if (take_coarse) {
      m[k] = d[i];
      pos_coarse[r * N + i] = k;
      ++i;
    } else {
      m[k] = f[j];
      pos_fine[r * Nf + j] = k;
      ++j;
    }
  }
}

__global__ void __launch_bounds__(256)
scatter_merge_kernel(const float* __restrict__ a, const int32_t* __restrict__ pa, int Na,
                     const float* __restrict__ b, const int32_t* __restrict__ pb, int Nb,
                     int64_t R, float* __restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int M = Na + Nb;
  if (t >= R * M) return;
  int64_t r = t / M;
  int i = (int)(t % M);
  if (i < Na) out[r * M + pa[r * Na + i]] = a[r * Na + i];
  else out[r * M + pb[r * Nb + (i - Na)]] = b[r * Nb + (i - Na)];
}

// ---------------------------------------------------------------------------
// NeuS alpha
// ---------------------------------------------------------------------------
struct NeusIn {
  const float* ray;
  const float* sdfs;
  const float* grads;
  const float* dists;
  const float* far;
  const uint8_t* outside;
  float outside_val;
  const float* s_var;
  float anneal_ratio;
  int64_t R;  // rays (dense) or samples (packed)
  int N;      // samples per ray (dense) or 1 (packed)
  const int32_t* off;      // packed: ray r owns samples [off[r], off[r+1])
  const int32_t* ray_idx;  // packed: ray of each sample
};

struct NeusTerms {
  float sdf, cosv, intv, iter_cos, est_prev, est_next, inv_s, pc, nc, ratio;
  bool outside;
  int64_t r;
};

// Terms of sample t of ray r (has_next: t is not the ray's last sample).
__device__ inline NeusTerms neus_terms_of(const NeusIn& p, int64_t t, int64_t r, bool has_next) {
  NeusTerms q;
  q.r = r;
  q.outside = p.outside && p.outside[r];
  q.sdf = q.outside ? p.outside_val : p.sdfs[t];
  float v0 = p.ray[r * 3], v1 = p.ray[r * 3 + 1], v2 = p.ray[r * 3 + 2];
  float g0 = p.grads[t * 3], g1 = p.grads[t * 3 + 1], g2 = p.grads[t * 3 + 2];
  q.cosv = v0 * g0 + v1 * g1 + v2 * g2;
  float a = p.anneal_ratio;
  float u1 = -q.cosv * 0.5f + 0.5f;
  float u2 = -q.cosv;
  float r1 = u1 > 0.0f ? u1 : 0.0f;
  float r2 = u2 > 0.0f ? u2 : 0.0f;
  q.iter_cos = -(r1 * (1.0f - a) + r2 * a);
  float dnext = has_next ? p.dists[t + 1] : (p.far ? p.far[r] : 1e10f);
  q.intv = dnext - p.dists[t];
  q.est_prev = q.sdf - q.iter_cos * q.intv * 0.5f;
  q.est_next = q.sdf + q.iter_cos * q.intv * 0.5f;
  q.inv_s = expf(*p.s_var);
  q.pc = sigmoidf_(q.est_prev * q.inv_s);
  q.nc = sigmoidf_(q.est_next * q.inv_s);
  q.ratio = (q.pc - q.nc) / (q.pc + 1e-5f);
  return q;
}

__device__ inline NeusTerms neus_terms(const NeusIn& p, int64_t t) {
  int64_t r;
  bool has_next;
  if (p.off) {
    r = p.ray_idx[t];
    has_next = t + 1 < (int64_t)p.off[r + 1];
  } else {
    r = t / p.N;
    has_next = (int)(t % p.N) + 1 < p.N;
  }
  return neus_terms_of(p, t, r, has_next);
}

// Backward of one sample's alpha: dsdf, dgrad (3) and the sample's share of
// d(s_var) from dalpha (the clamp passes the gradient where 0 <= ratio <= 1).
__device__ inline float neus_sample_bwd(const NeusIn& p, const NeusTerms& q, float da, int64_t t,
                                        float* __restrict__ dsdf, float* __restrict__ dgrad) {
  float dr = (q.ratio >= 0.0f && q.ratio <= 1.0f) ? da : 0.0f;
  float num = q.pc - q.nc, den = q.pc + 1e-5f;
  float dnum = dr / den;
  float dden = -dr * num / (den * den);
  float dpc = dnum + dden;
  float dnc = -dnum;
  float dzp = dpc * q.pc * (1.0f - q.pc);  // d(est_prev * inv_s)
  float dzn = dnc * q.nc * (1.0f - q.nc);
  float dep = dzp * q.inv_s, den_ = dzn * q.inv_s;
  float dinv = dzp * q.est_prev + dzn * q.est_next;
  dsdf[t] = q.outside ? 0.0f : (dep + den_);
  float diter = (-dep + den_) * q.intv * 0.5f;
  float a = p.anneal_ratio;
  float u1 = -q.cosv * 0.5f + 0.5f;
  float u2 = -q.cosv;
  float dcos = diter * (0.5f * (1.0f - a) * (u1 > 0.0f ? 1.0f : 0.0f) + a * (u2 > 0.0f ? 1.0f : 0.0f));
  const int64_t r = q.r;
  dgrad[t * 3] = dcos * p.ray[r * 3];
  dgrad[t * 3 + 1] = dcos * p.ray[r * 3 + 1];
  dgrad[t * 3 + 2] = dcos * p.ray[r * 3 + 2];
  return dinv * q.inv_s;
}

__global__ void __launch_bounds__(256)
neus_alpha_fwd_kernel(NeusIn p, float* __restrict__ alpha) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= p.R * p.N) return;
  NeusTerms q = neus_terms(p, t);
  float a = q.ratio;
  alpha[t] = a < 0.0f ? 0.0f : (a > 1.0f ? 1.0f : a);  // clip_, NaN kept
}

__global__ void __launch_bounds__(256)
neus_alpha_bwd_kernel(NeusIn p, const float* __restrict__ dalpha, float* __restrict__ dsdf,
                      float* __restrict__ dgrad, float* __restrict__ ds_var) {
  __shared__ float red[4];
  // grid-stride over the samples: a few hundred workgroups, so that few atomics
  // meet on the one ds_var
  float dsv = 0.0f;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < p.R * p.N;
       t += (int64_t)gridDim.x * blockDim.x) {
    NeusTerms q = neus_terms(p, t);
    dsv += neus_sample_bwd(p, q, dalpha[t], t, dsdf, dgrad);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) dsv += __shfl_xor(dsv, o);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = dsv;
  __syncthreads();
  if (threadIdx.x == 0) atomic_add_f32(ds_var, red[0] + red[1] + red[2] + red[3]);
}

// ---------------------------------------------------------------------------
// alpha compositing + composite
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kRayBlock)
composite_fwd_kernel(const float* __restrict__ alpha, const float* __restrict__ q, int64_t R,
                     int N, int K, float* __restrict__ weights, float* __restrict__ out) {
  const int64_t r = (int64_t)blockIdx.x * kRayBlock + threadIdx.x;
  if (r >= R) return;
  float logT = 0.0f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  // the loads of kCompU samples go out before their (sequential) arithmetic
  for (int i0 = 0; i0 < N; i0 += kCompU) {
    float av[kCompU], qv[kCompU][4];
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int i = i0 + u;
      av[u] = i < N ? alpha[r * N + i] : 0.0f;
#pragma unroll
      for (int k = 0; k < 4; ++k) qv[u][k] = (i < N && k < K) ? q[(r * N + i) * K + k] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int i = i0 + u;
      if (i >= N) break;
      float a = av[u];
      float T = expf(logT);
      float w = a * T;
      weights[r * N + i] = w;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < K) acc[k] = acc[k] + qv[u][k] * w;
      logT = logT + log1pf(-a);
    }
  }
  for (int k = 0; k < K; ++k) out[r * K + k] = acc[k];
}

__global__ void __launch_bounds__(kRayBlock)
composite_bwd_kernel(const float* __restrict__ alpha, const float* __restrict__ q,
                     const float* __restrict__ weights, int64_t R, int N, int K,
                     const float* __restrict__ dout, const float* __restrict__ dweights,
                     float* __restrict__ dalpha, float* __restrict__ dq) {
  extern __shared__ float s_T[];
  const int l = threadIdx.x;
  const int64_t r = (int64_t)blockIdx.x * kRayBlock + l;
  if (r >= R) return;
  float* T = s_T + l;
  float logT = 0.0f;
  // (the loads of kCompU samples go out before their sequential arithmetic)
  for (int i0 = 0; i0 < N; i0 += kCompU) {
    float av[kCompU];
#pragma unroll
    for (int u = 0; u < kCompU; ++u) av[u] = i0 + u < N ? alpha[r * N + i0 + u] : 0.0f;
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      if (i0 + u >= N) break;
      T[(i0 + u) * kRayBlock] = expf(logT);
      logT = logT + log1pf(-av[u]);
    }
  }
  float d[4] = {0.f, 0.f, 0.f, 0.f};
  if (dout)
    for (int k = 0; k < K; ++k) d[k] = dout[r * K + k];
  // U_j = sum_{i>j} g_i a_i prod_{j<k<i}(1-a_k);  dalpha_j = T_j (g_j - U_j)
  float U = 0.0f;
  for (int j0 = N - 1; j0 >= 0; j0 -= kCompU) {
    float gv[kCompU], av[kCompU], wv[kCompU], qv[kCompU][4];
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int j = j0 - u;
      const bool ok = j >= 0;
      gv[u] = (ok && dweights) ? dweights[r * N + j] : 0.0f;
      av[u] = ok ? alpha[r * N + j] : 0.0f;
      wv[u] = (ok && dq) ? weights[r * N + j] : 0.0f;
#pragma unroll
      for (int k = 0; k < 4; ++k) qv[u][k] = (ok && k < K) ? q[(r * N + j) * K + k] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int j = j0 - u;
      if (j < 0) break;
      float g = gv[u];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < K) g = g + d[k] * qv[u][k];
      if (dq)
        for (int k = 0; k < K; ++k) dq[(r * N + j) * K + k] = wv[u] * d[k];
      float a = av[u];
      float Tj = T[j * kRayBlock];
      dalpha[r * N + j] = Tj * (g - U);
      U = g * a + (1.0f - a) * U;
    }
  }
}

// Packed rays (ragged sample counts): ray r owns samples [off[r], off[r+1]) of
// every per-sample array.  Same arithmetic and order as the dense kernels; the
// backward keeps the transmittance of the forward pass in dalpha until the
// reverse pass overwrites it, so a ray may hold any number of samples.
__global__ void __launch_bounds__(256)
composite_packed_fwd_kernel(const float* __restrict__ alpha, const float* __restrict__ q,
                            const int32_t* __restrict__ off, int64_t R, int K,
                            float* __restrict__ weights, float* __restrict__ out) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  const int64_t b = off[r], e = off[r + 1];
  float logT = 0.0f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int64_t i0 = b; i0 < e; i0 += kCompU) {
    float av[kCompU], qv[kCompU][4];
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int64_t i = i0 + u;
      av[u] = i < e ? alpha[i] : 0.0f;
#pragma unroll
      for (int k = 0; k < 4; ++k) qv[u][k] = (i < e && k < K) ? q[i * K + k] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int64_t i = i0 + u;
      if (i >= e) break;
      float a = av[u];
      float T = expf(logT);
      float w = a * T;
      weights[i] = w;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < K) acc[k] = acc[k] + qv[u][k] * w;
      logT = logT + log1pf(-a);
    }
  }
  for (int k = 0; k < K; ++k) out[r * K + k] = acc[k];
}

__global__ void __launch_bounds__(256)
composite_packed_bwd_kernel(const float* __restrict__ alpha, const float* __restrict__ q,
                            const float* __restrict__ weights, const int32_t* __restrict__ off,
                            int64_t R, int K, const float* __restrict__ dout,
                            const float* __restrict__ dweights, float* __restrict__ dalpha,
                            float* __restrict__ dq) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  const int64_t b = off[r], e = off[r + 1];
  float logT = 0.0f;
  for (int64_t i0 = b; i0 < e; i0 += kCompU) {
    float av[kCompU];
#pragma unroll
    for (int u = 0; u < kCompU; ++u) av[u] = i0 + u < e ? alpha[i0 + u] : 0.0f;
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      if (i0 + u >= e) break;
      dalpha[i0 + u] = expf(logT);  // T_i, replaced by the gradient below
      logT = logT + log1pf(-av[u]);
    }
  }
  float d[4] = {0.f, 0.f, 0.f, 0.f};
  if (dout)
    for (int k = 0; k < K; ++k) d[k] = dout[r * K + k];
  float U = 0.0f;
  for (int64_t j0 = e - 1; j0 >= b; j0 -= kCompU) {
    // each T_j is read here before this block overwrites it
    float gv[kCompU], av[kCompU], wv[kCompU], tv[kCompU], qv[kCompU][4];
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int64_t j = j0 - u;
      const bool ok = j >= b;
      gv[u] = (ok && dweights) ? dweights[j] : 0.0f;
      av[u] = ok ? alpha[j] : 0.0f;
      wv[u] = (ok && dq) ? weights[j] : 0.0f;
      tv[u] = ok ? dalpha[j] : 0.0f;
#pragma unroll
      for (int k = 0; k < 4; ++k) qv[u][k] = (ok && k < K) ? q[j * K + k] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kCompU; ++u) {
      const int64_t j = j0 - u;
      if (j < b) break;
      float g = gv[u];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < K) g = g + d[k] * qv[u][k];
      if (dq)
        for (int k = 0; k < K; ++k) dq[j * K + k] = wv[u] * d[k];
      float a = av[u];
      dalpha[j] = tv[u] * (g - U);
      U = g * a + (1.0f - a) * U;
    }
  }
}

__global__ void __launch_bounds__(256)
weighted_sum_packed_fwd_kernel(const float* __restrict__ q, const float* __restrict__ w,
                               const int32_t* __restrict__ off, int64_t R, int K,
                               float* __restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R * K) return;
  int64_t r = t / K;
  int k = (int)(t % K);
  float acc = 0.0f;
  for (int64_t i = off[r]; i < off[r + 1]; ++i) acc = acc + q[i * K + k] * w[i];
  out[t] = acc;
}

__global__ void __launch_bounds__(256)
weighted_sum_packed_bwd_kernel(const float* __restrict__ q, const float* __restrict__ w,
                               const int32_t* __restrict__ ray_idx, int64_t S, int K,
                               const float* __restrict__ dout, float* __restrict__ dq,
                               float* __restrict__ dw) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= S) return;
  int64_t r = ray_idx[t];
  float acc = 0.0f;
  for (int k = 0; k < K; ++k) {
    float d = dout[r * K + k];
    if (dq) dq[t * K + k] = w[t] * d;
    acc = acc + q[t * K + k] * d;
  }
  if (dw) dw[t] = acc;
}

// ray of every packed sample from the offsets (one thread per ray)
// ---------------------------------------------------------------------------
// Packed rays in one persistent launch each way: NeuS alpha + compositing.
// A persistent grid (a few workgroups per CU) whose waves take chunks of
// kPackedChunk consecutive rays from a work counter (queue, zero at launch)
// until every ray is done, so rays of uneven sample counts balance across the
// chip.  A wave renders one ray at a time, its 64 lanes over 64 consecutive
// samples (coalesced loads and stores):
//   forward: each sample's alpha (neus_alpha_fwd_kernel's terms, the ray's last
//   sample against its far distance), log T as the running sum of log(1 - alpha)
//   (a wave scan per 64 samples plus the carry of the earlier ones), the weights
//   and the composited q (K <= 4 channels, summed over the wave);
//   backward: the same transmittance pass (kept in dsdf until overwritten), then
//   the 64-sample groups from the ray's end: U_j = sum_{i>j} g_i a_i prod_{j<k<i}
//   (1 - a_k) is the composition of the affine maps x -> (1 - a_i) x + g_i a_i
//   of the later samples applied to the carry of the later groups (a suffix scan
//   of maps), dalpha_j = T_j (g_j - U_j) plus any direct dalpha, and from it
//   dsdf, dgrad and the s_var gradient (one atomic per wave).
// The sums run in wave-scan order, so values match the one-lane-per-ray kernels
// to float rounding.
// ---------------------------------------------------------------------------
constexpr int kPackedChunk = 8;  // rays per work-counter request

__device__ inline int64_t packed_next_chunk(int* queue) {
  int c = 0;
  if ((threadIdx.x & 63) == 0) c = atomicAdd(queue, 1);
  return (int64_t)__shfl(c, 0);
}

__device__ inline float wave_incl_sum(float x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  return x;
}

__device__ inline float wave_total(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

__global__ void __launch_bounds__(256)
neus_composite_packed_fwd_kernel(NeusIn p, const float* __restrict__ q, int K,
                                 float* __restrict__ alpha, float* __restrict__ weights,
                                 float* __restrict__ out, int* __restrict__ queue) {
  const int lane = threadIdx.x & 63;
  const int64_t R = p.R;
  for (int64_t ch = packed_next_chunk(queue); ch * kPackedChunk < R; ch = packed_next_chunk(queue)) {
    for (int rr = 0; rr < kPackedChunk; ++rr) {
      const int64_t r = ch * kPackedChunk + rr;
      if (r >= R) break;
      const int64_t b = p.off[r], e = p.off[r + 1];
      float carry = 0.0f;  // log T before this group's first sample
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
      for (int64_t base = b; base < e; base += 64) {
        const int64_t i = base + lane;
        const bool valid = i < e;
        float a = 0.0f;
        if (valid) {
          const NeusTerms t = neus_terms_of(p, i, r, i + 1 < e);
          const float ra = t.ratio;
          a = ra < 0.0f ? 0.0f : (ra > 1.0f ? 1.0f : ra);  // clip_, NaN kept
          alpha[i] = a;
        }
        const float l = valid ? log1pf(-a) : 0.0f;
        const float incl = wave_incl_sum(l);
        float ex = __shfl_up(incl, 1);
        if (lane == 0) ex = 0.0f;
        if (valid) {
          const float w = a * expf(carry + ex);
          weights[i] = w;
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (k < K) acc[k] = acc[k] + q[i * K + k] * w;
        }
        carry = carry + __shfl(incl, 63);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (k < K) {
          const float sk = wave_total(acc[k]);
          if (lane == 0) out[r * K + k] = sk;
        }
      }
    }
  }
}

__global__ void __launch_bounds__(256)
neus_composite_packed_bwd_kernel(NeusIn p, const float* __restrict__ q, int K,
                                 const float* __restrict__ alpha,
                                 const float* __restrict__ weights,
                                 const float* __restrict__ dout,
                                 const float* __restrict__ dweights,
                                 const float* __restrict__ dalpha_in, float* __restrict__ dsdf,
                                 float* __restrict__ dgrad, float* __restrict__ dq,
                                 float* __restrict__ ds_var, int* __restrict__ queue) {
  const int lane = threadIdx.x & 63;
  const int64_t R = p.R;
  float dsv = 0.0f;
  for (int64_t ch = packed_next_chunk(queue); ch * kPackedChunk < R; ch = packed_next_chunk(queue)) {
    for (int rr = 0; rr < kPackedChunk; ++rr) {
      const int64_t r = ch * kPackedChunk + rr;
      if (r >= R) break;
      const int64_t b = p.off[r], e = p.off[r + 1];
      // transmittance of every sample, kept in dsdf (as the forward formed it)
      float carry = 0.0f;
      for (int64_t base = b; base < e; base += 64) {
        const int64_t i = base + lane;
        const bool valid = i < e;
        const float l = valid ? log1pf(-alpha[i]) : 0.0f;
        const float incl = wave_incl_sum(l);
        float ex = __shfl_up(incl, 1);
        if (lane == 0) ex = 0.0f;
        if (valid) dsdf[i] = expf(carry + ex);
        carry = carry + __shfl(incl, 63);
      }
      float d[4] = {0.f, 0.f, 0.f, 0.f};
      if (dout)
        for (int k = 0; k < K; ++k) d[k] = dout[r * K + k];
      float uc = 0.0f;  // U of the sample before the later groups' first one
      const int64_t n = e - b;
      for (int64_t base = b + ((n - 1) / 64) * 64; n > 0 && base >= b; base -= 64) {
        const int64_t j = base + lane;
        const bool valid = j < e;
        float g = 0.0f, a = 0.0f, tj = 0.0f;
        if (valid) {
          g = dweights ? dweights[j] : 0.0f;
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (k < K) g = g + d[k] * q[j * K + k];
          if (dq) {
            const float wj = weights[j];
            for (int k = 0; k < K; ++k) dq[j * K + k] = wj * d[k];
          }
          a = alpha[j];
          tj = dsdf[j];
        }
        // suffix composition of x -> m x + c over lanes j .. 63 (identity past e)
        float m = valid ? 1.0f - a : 1.0f, c = valid ? g * a : 0.0f;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const float m2 = __shfl_down(m, o), c2 = __shfl_down(c, o);
          if (lane + o < 64) {
            c = m * c2 + c;
            m = m * m2;
          }
        }
        // exclusive: the maps of lanes j + 1 .. 63 applied to the carry
        float mx = __shfl_down(m, 1), cx = __shfl_down(c, 1);
        if (lane == 63) {
          mx = 1.0f;
          cx = 0.0f;
        }
        const float U = mx * uc + cx;
        const float u0 = __shfl(m, 0) * uc + __shfl(c, 0);  // U before this group
        if (valid) {
          float da = tj * (g - U);
          if (dalpha_in) da = da + dalpha_in[j];
          const NeusTerms t = neus_terms_of(p, j, r, j + 1 < e);
          dsv += neus_sample_bwd(p, t, da, j, dsdf, dgrad);
        }
        uc = u0;
      }
    }
  }
  dsv = wave_total(dsv);
  if (lane == 0 && dsv != 0.0f) atomic_add_f32(ds_var, dsv);
}

__global__ void __launch_bounds__(256)
packed_ray_index_kernel(const int32_t* __restrict__ off, int64_t R, int32_t* __restrict__ ray_idx) {
  int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  for (int64_t i = off[r]; i < off[r + 1]; ++i) ray_idx[i] = (int32_t)r;
}

__global__ void __launch_bounds__(256)
weighted_sum_fwd_kernel(const float* __restrict__ q, const float* __restrict__ w, int64_t R,
                        int N, int K, float* __restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R * K) return;
  int64_t r = t / K;
  int k = (int)(t % K);
  float acc = 0.0f;
  for (int i = 0; i < N; ++i) acc = acc + q[(r * N + i) * K + k] * w[r * N + i];
  out[t] = acc;
}

__global__ void __launch_bounds__(256)
weighted_sum_bwd_kernel(const float* __restrict__ q, const float* __restrict__ w, int64_t R,
                        int N, int K, const float* __restrict__ dout, float* __restrict__ dq,
                        float* __restrict__ dw) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R * N) return;
  int64_t r = t / N;
  float acc = 0.0f;
  for (int k = 0; k < K; ++k) {
    float d = dout[r * K + k];
    if (dq) dq[t * K + k] = w[t] * d;
    acc = acc + q[t * K + k] * d;
  }
  if (dw) dw[t] = acc;
}

// ---------------------------------------------------------------------------
// 4-tap numerical gradient
// ---------------------------------------------------------------------------
__constant__ float kTap[4][3] = {{1, -1, -1}, {-1, -1, 1}, {-1, 1, -1}, {1, 1, 1}};

__global__ void __launch_bounds__(256)
taps_points_kernel(const float* __restrict__ x, int64_t n, float eps, float* __restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * 3) return;
  int64_t p = t / 3;
  int d = (int)(t % 3);
  float xv = x[t];
#pragma unroll
  for (int k = 0; k < 4; ++k) out[(k * n + p) * 3 + d] = xv + kTap[k][d] * eps;
}

// Increment form of the 4-tap combination: ds[t] = sdf(x + eps k_t) - sdf(x),
// sc = sdf(x) as evaluated, sdf = the value the reference passes in (the outside
// fill included).  gradient = sum_t k_t ds_t / (4 eps) (sum k_t = 0);
// hessian trace h = (sum_t ds_t / 2 + 2 (sc - sdf)) / eps^2, returned as h/3 per
// component -- the reference's ((sum s_t)/2 - 2 sdf)/eps^2 without subtracting
// nearly equal numbers.
__global__ void __launch_bounds__(256)
taps_delta_fwd_kernel(const float* __restrict__ ds, const float* __restrict__ sc,
                      const float* __restrict__ sdf, int64_t n, float eps, float eps_sq,
                      float* __restrict__ grad, float* __restrict__ hess) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const float d1 = ds[p], d2 = ds[n + p], d3 = ds[2 * n + p], d4 = ds[3 * n + p];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float g = kTap[0][k] * d1 + kTap[1][k] * d2 + kTap[2][k] * d3 + kTap[3][k] * d4;
    grad[p * 3 + k] = g / (4.0f * eps);
  }
  if (hess) {
    const float h = ((d1 + d2 + d3 + d4) / 2.0f + 2.0f * (sc[p] - sdf[p])) / eps_sq;
    const float h3 = h / 3.0f;
    hess[p * 3] = h3;
    hess[p * 3 + 1] = h3;
    hess[p * 3 + 2] = h3;
  }
}

__global__ void __launch_bounds__(256)
taps_delta_bwd_kernel(int64_t n, float eps, float eps_sq, const float* __restrict__ dgrad,
                      const float* __restrict__ dhess, float* __restrict__ dds,
                      float* __restrict__ dsc, float* __restrict__ dsdf) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  float dh = 0.0f;
  if (dhess) dh = (dhess[p * 3] + dhess[p * 3 + 1] + dhess[p * 3 + 2]) / 3.0f / eps_sq;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    float v = 0.5f * dh;
    if (dgrad)
      v += (kTap[t][0] * dgrad[p * 3] + kTap[t][1] * dgrad[p * 3 + 1] +
            kTap[t][2] * dgrad[p * 3 + 2]) / (4.0f * eps);
    dds[t * n + p] = v;
  }
  if (dsc) dsc[p] = 2.0f * dh;
  if (dsdf) dsdf[p] = -2.0f * dh;
}

__global__ void __launch_bounds__(256)
taps_combine_fwd_kernel(const float* __restrict__ s, const float* __restrict__ sdf, int64_t n,
                        float eps, float eps_sq, float* __restrict__ grad,
                        float* __restrict__ hess) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  float s1 = s[p], s2 = s[n + p], s3 = s[2 * n + p], s4 = s[3 * n + p];
  float den = 4.0f * eps;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    float g = kTap[0][d] * s1 + kTap[1][d] * s2;
    g = g + kTap[2][d] * s3;
    g = g + kTap[3][d] * s4;
    grad[p * 3 + d] = g / den;
  }
  if (hess) {
    float sum = ((s1 + s2) + s3) + s4;
    float h = (sum / 2.0f - 2.0f * sdf[p]) / eps_sq;
    float h3 = h / 3.0f;
    hess[p * 3] = h3;
    hess[p * 3 + 1] = h3;
    hess[p * 3 + 2] = h3;
  }
}

__global__ void __launch_bounds__(256)
taps_combine_bwd_kernel(int64_t n, float eps, float eps_sq, const float* __restrict__ dgrad,
                        const float* __restrict__ dhess, float* __restrict__ ds,
                        float* __restrict__ dsdf, int add_dsdf) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  float den = 4.0f * eps;
  float g0 = dgrad ? dgrad[p * 3] / den : 0.0f;
  float g1 = dgrad ? dgrad[p * 3 + 1] / den : 0.0f;
  float g2 = dgrad ? dgrad[p * 3 + 2] / den : 0.0f;
  float dh = 0.0f;
  if (dhess) dh = ((dhess[p * 3] + dhess[p * 3 + 1]) + dhess[p * 3 + 2]) / 3.0f / eps_sq;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    ds[k * n + p] = kTap[k][0] * g0 + kTap[k][1] * g1 + kTap[k][2] * g2 + dh / 2.0f;
  if (dsdf) {
    float v = -2.0f * dh;
    dsdf[p] = add_dsdf ? dsdf[p] + v : v;
  }
}

// ---------------------------------------------------------------------------
// colour-MLP input: [feat | x | SH16 | normal | pad]
// ---------------------------------------------------------------------------
// Real SH constants (closed forms: C0 = 1/(2 sqrt(pi)), C1 = sqrt(3)/(2 sqrt(pi)), ...)
#define SH_C0 0.28209479177387814f
#define SH_C1 0.4886025119029199f
#define SH_C2_0 1.0925484305920792f
#define SH_C2_1 -1.0925484305920792f
#define SH_C2_2 0.31539156525252005f
#define SH_C2_3 -1.0925484305920792f
#define SH_C2_4 0.5462742152960396f
#define SH_C3_0 -0.5900435899266435f
#define SH_C3_1 2.890611442640554f
#define SH_C3_2 -0.4570457994644658f
#define SH_C3_3 0.3731763325901154f
#define SH_C3_4 -0.4570457994644658f
#define SH_C3_5 1.445305721320277f
#define SH_C3_6 -0.5900435899266435f

__device__ inline void sh3(float x, float y, float z, float v[16]) {
  v[0] = SH_C0;
  v[1] = -SH_C1 * y;
  v[2] = SH_C1 * z;
  v[3] = -SH_C1 * x;
  float xx = x * x, yy = y * y, zz = z * z;
  float xy = x * y, yz = y * z, xz = x * z;
  v[4] = SH_C2_0 * xy;
  v[5] = SH_C2_1 * yz;
  v[6] = SH_C2_2 * (2.0f * zz - xx - yy);
  v[7] = SH_C2_3 * xz;
  v[8] = SH_C2_4 * (xx - yy);
  v[9] = SH_C3_0 * y * (3.0f * xx - yy);
  v[10] = SH_C3_1 * xy * z;
  v[11] = SH_C3_2 * y * (4.0f * zz - xx - yy);
  v[12] = SH_C3_3 * z * (2.0f * zz - 3.0f * xx - 3.0f * yy);
  v[13] = SH_C3_4 * x * (4.0f * zz - xx - yy);
  v[14] = SH_C3_5 * z * (xx - yy);
  v[15] = SH_C3_6 * x * (xx - 3.0f * yy);
}

template <typename TO>
__global__ void __launch_bounds__(256)
rgb_input_fwd_kernel(const float* __restrict__ x, const float* __restrict__ ray,
                     int64_t n_per_ray, const float* __restrict__ grad, int normalize, int64_t n,
                     int col0, TO* __restrict__ out, int64_t ld, int vec24) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int64_t r = p / n_per_ray;
  float row[24];
  row[0] = x[p * 3];
  row[1] = x[p * 3 + 1];
  row[2] = x[p * 3 + 2];
  sh3(ray[r * 3], ray[r * 3 + 1], ray[r * 3 + 2], row + 3);
  float g0 = grad[p * 3], g1 = grad[p * 3 + 1], g2 = grad[p * 3 + 2];
  if (normalize) {
    float nrm = sqrtf(g0 * g0 + g1 * g1 + g2 * g2);
    float dn = nrm > 1e-12f ? nrm : 1e-12f;
    g0 = g0 / dn;
    g1 = g1 / dn;
    g2 = g2 / dn;
  }
  row[19] = g0;
  row[20] = g1;
  row[21] = g2;
  row[22] = row[23] = 0.0f;
  TO* o = out + p * ld + col0;
  if (vec24) {
    // the row's tail is exactly these 24 columns, 16-byte aligned: whole
    // 16-byte stores (same rounding as the element stores)
    if constexpr (sizeof(TO) == 2) {
      uint32_t w[12];
#pragma unroll
      for (int i = 0; i < 12; ++i)
        w[i] = (uint32_t)f32_to_bf16(row[2 * i]) | ((uint32_t)f32_to_bf16(row[2 * i + 1]) << 16);
      uint4* q = reinterpret_cast<uint4*>(o);
#pragma unroll
      for (int i = 0; i < 3; ++i) q[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    } else {
      float4* q = reinterpret_cast<float4*>(o);
#pragma unroll
      for (int i = 0; i < 6; ++i) q[i] = make_float4(row[4 * i], row[4 * i + 1], row[4 * i + 2], row[4 * i + 3]);
    }
    return;
  }
  for (int c = 0; c < 22; ++c) scalar_io<TO>::store(o + c, row[c]);
  for (int64_t c = col0 + 22; c < ld; ++c) scalar_io<TO>::store(out + p * ld + c, 0.0f);
}

// Standalone SH encoding of unit directions: the first (levels+1)^2 basis
// values per direction (degree <= 3), the same polynomials the colour input uses.
__global__ void __launch_bounds__(256)
sh_encode_kernel(const float* __restrict__ dirs, int64_t n, int nb, float* __restrict__ out) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  float v[16];
  sh3(dirs[p * 3], dirs[p * 3 + 1], dirs[p * 3 + 2], v);
  for (int k = 0; k < nb; ++k) out[p * nb + k] = v[k];
}

template <typename TD>
__global__ void __launch_bounds__(256)
rgb_input_bwd_kernel(const float* __restrict__ grad, int normalize, int64_t n, int col0,
                     const TD* __restrict__ dy, int64_t ld, float* __restrict__ dgrad, int add) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  float g0 = grad[p * 3], g1 = grad[p * 3 + 1], g2 = grad[p * 3 + 2];
  float nrm = sqrtf(g0 * g0 + g1 * g1 + g2 * g2);
  const TD* d = dy + p * ld + col0 + 19;
  float d0 = scalar_io<TD>::load(d), d1 = scalar_io<TD>::load(d + 1), d2 = scalar_io<TD>::load(d + 2);
  float o0, o1, o2;
  if (!normalize) {
    o0 = d0;
    o1 = d1;
    o2 = d2;
  } else if (nrm > 1e-12f) {
    float n0 = g0 / nrm, n1 = g1 / nrm, n2 = g2 / nrm;
    float dot = n0 * d0 + n1 * d1 + n2 * d2;
    o0 = (d0 - n0 * dot) / nrm;
    o1 = (d1 - n1 * dot) / nrm;
    o2 = (d2 - n2 * dot) / nrm;
  } else {
    o0 = d0 / 1e-12f;
    o1 = d1 / 1e-12f;
    o2 = d2 / 1e-12f;
  }
  if (add) {
    o0 += dgrad[p * 3];
    o1 += dgrad[p * 3 + 1];
    o2 += dgrad[p * 3 + 2];
  }
  dgrad[p * 3] = o0;
  dgrad[p * 3 + 1] = o1;
  dgrad[p * 3 + 2] = o2;
}

// ---------------------------------------------------------------------------
// eikonal + curvature losses
// ---------------------------------------------------------------------------
__device__ inline bool finitef_(float v) { return v == v && fabsf(v) != INFINITY; }

__global__ void __launch_bounds__(256)
sdf_losses_fwd_kernel(const float* __restrict__ grad, const float* __restrict__ hess,
                      const uint8_t* __restrict__ outside, int64_t n, int64_t n_per_ray,
                      float* __restrict__ sums) {
  __shared__ float red[2][4];
  // grid-stride: a few hundred workgroups, so that few atomics meet on the two sums
  // (NaN / Inf terms count as 0, as before the sum)
  float e = 0.0f, c = 0.0f;
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    float m = (outside && outside[p / n_per_ray]) ? 0.0f : 1.0f;
    if (grad) {
      float g0 = grad[p * 3], g1 = grad[p * 3 + 1], g2 = grad[p * 3 + 2];
      float nrm = sqrtf(g0 * g0 + g1 * g1 + g2 * g2);
      float ev = (nrm - 1.0f) * (nrm - 1.0f);
      e += (finitef_(ev) ? ev : 0.0f) * m;
    }
    if (hess) {
      float lap = fabsf((hess[p * 3] + hess[p * 3 + 1]) + hess[p * 3 + 2]);
      c += (finitef_(lap) ? lap : 0.0f) * m;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    e += __shfl_xor(e, o);
    c += __shfl_xor(c, o);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][w] = e;
    red[1][w] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomic_add_f32(sums, red[0][0] + red[0][1] + red[0][2] + red[0][3]);
    atomic_add_f32(sums + 1, red[1][0] + red[1][1] + red[1][2] + red[1][3]);
  }
}

__global__ void __launch_bounds__(256)
sdf_losses_bwd_kernel(const float* __restrict__ grad, const float* __restrict__ hess,
                      const uint8_t* __restrict__ outside, int64_t n, int64_t n_per_ray,
                      const float* __restrict__ wts, float* __restrict__ dgrad, int add_dgrad,
                      float* __restrict__ dhess) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const float w_eik = wts[0], w_curv = wts[1];
  float m = (outside && outside[p / n_per_ray]) ? 0.0f : 1.0f;
  float inv_n = 1.0f / (float)n;
  if (dgrad) {
    float g0 = grad[p * 3], g1 = grad[p * 3 + 1], g2 = grad[p * 3 + 2];
    float nrm = sqrtf(g0 * g0 + g1 * g1 + g2 * g2);
    float ev = (nrm - 1.0f) * (nrm - 1.0f);
    float s = (finitef_(ev) && nrm > 0.0f) ? w_eik * inv_n * m * 2.0f * (nrm - 1.0f) / nrm : 0.0f;
    float o0 = s * g0, o1 = s * g1, o2 = s * g2;
    if (add_dgrad) {
      o0 += dgrad[p * 3];
      o1 += dgrad[p * 3 + 1];
      o2 += dgrad[p * 3 + 2];
    }
    dgrad[p * 3] = o0;
    dgrad[p * 3 + 1] = o1;
    dgrad[p * 3 + 2] = o2;
  }
  if (dhess) {
    float lap = (hess[p * 3] + hess[p * 3 + 1]) + hess[p * 3 + 2];
    float sg = lap > 0.0f ? 1.0f : (lap < 0.0f ? -1.0f : 0.0f);
    float v = finitef_(fabsf(lap)) ? w_curv * inv_n * m * sg : 0.0f;
    dhess[p * 3] = v;
    dhess[p * 3 + 1] = v;
    dhess[p * 3 + 2] = v;
  }
}

static inline dim3 grid1d(int64_t n, int block = 256) { return dim3((unsigned)ceil_div(n, block)); }
// Grid of a grid-stride kernel that ends in one atomic per workgroup on a
// single address: at most 512 workgroups of 256 threads.
static inline dim3 grid_reduce(int64_t n) {
  const int64_t b = ceil_div(n, (int64_t)256);
  return dim3((unsigned)(b < 512 ? b : 512));
}

}  // namespace na

using namespace na;

extern "C" int na_ray_bounds_sample(const float* center, const float* ray_unit, const float* rands,
                                    int64_t R, int32_t N, float* near, float* far,
                                    uint8_t* outside, float* dists, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 1, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(center && ray_unit && near && far && outside && dists, "null pointer");
  hipLaunchKernelGGL(ray_bounds_sample_kernel, grid1d(R * N), dim3(256), 0, (hipStream_t)stream,
                     center, ray_unit, rands, R, N, near, far, outside, dists);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_sphere_crossings(const float* center, const float* ray_unit, int64_t R,
                                   float radius, float* near, float* far, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(center && ray_unit && near && far, "null pointer");
  hipLaunchKernelGGL(sphere_crossings_kernel, grid1d(R), dim3(256), 0, (hipStream_t)stream,
                     center, ray_unit, R, radius * radius, near, far);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_camera_rays(const float* pose, const float* intr, int64_t B, int64_t H,
                              int64_t W, const int64_t* ray_idx, int64_t R, float* center,
                              float* ray, float* ray_unit, na_stream_t stream) {
  NA_CHECK_ARG(B >= 0 && H >= 1 && W >= 1 && R >= 0, "bad sizes");
  NA_CHECK_ARG(ray_idx || R == H * W, "without ray_idx every pixel is a ray (R == H*W)");
  if (B == 0 || R == 0) return NA_OK;
  NA_CHECK_ARG(pose && intr && center && ray, "null pointer");
  hipLaunchKernelGGL(camera_rays_kernel, grid1d(B * R), dim3(256), 0, (hipStream_t)stream, pose,
                     intr, B, W, ray_idx, R, center, ray, ray_unit);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_sample_dists(const float* lo, const float* hi, float lo_const, float hi_const,
                               const float* rands, int64_t R, int32_t N, float* dists,
                               na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 1, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(dists, "null pointer");
  hipLaunchKernelGGL(sample_dists_kernel, grid1d(R * N), dim3(256), 0, (hipStream_t)stream, lo, hi,
                     lo_const, hi_const, rands, R, N, dists);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_sh_encode(const float* dirs, int64_t n, int32_t levels, float* out,
                            na_stream_t stream) {
  NA_CHECK_ARG(n >= 0, "bad sizes");
  if (levels < 0 || levels > 3) {
    set_error("na_sh_encode: degree must be 0..3");
    return NA_ERR_UNSUPPORTED;
  }
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(dirs && out, "null pointer");
  hipLaunchKernelGGL(sh_encode_kernel, grid1d(n), dim3(256), 0, (hipStream_t)stream, dirs, n,
                     (levels + 1) * (levels + 1), out);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

static size_t cdf_lds_bytes(int N) { return (size_t)(N + 1) * kRayBlock * sizeof(float); }

extern "C" int na_sample_pdf(const float* bins, const float* weights, int64_t R, int32_t N,
                             int32_t Nf, float* out, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 2 && Nf >= 1, "bad sizes");
  NA_CHECK_ARG(cdf_lds_bytes(N) <= 65536, "N too large (<= 255)");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(bins && weights && out, "null pointer");
  hipLaunchKernelGGL(sample_pdf_kernel, grid1d(R, kRayBlock), dim3(kRayBlock), cdf_lds_bytes(N),
                     (hipStream_t)stream, bins, weights, R, N, Nf, out);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_hier_resample(const float* dists, const float* sdfs, int64_t R, int32_t N,
                                float inv_s, int32_t Nf, float* merged, float* fine,
                                int32_t* pos_coarse, int32_t* pos_fine, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 2 && Nf >= 1, "bad sizes");
  NA_CHECK_ARG(cdf_lds_bytes(N) <= 65536, "N too large (<= 255)");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(dists && sdfs && merged && fine && pos_coarse && pos_fine, "null pointer");
  // Few samples: 131,072 rays of 4 + 4 take 13 us by lane and 27 by wave, of 8 + 4 23 and 28
  // (1,000,000 rays: 111 and 173, 268 and 182); up to 16,384 rays the wave kernel is as fast.
  const bool brief = N + 2 * Nf <= 12 && R > 16384;
  NA_CHECK_ARG(Nf > kHierMaxFine || R < ((int64_t)1 << 28),
               "too many rays for one launch (16 threads a ray, below 2^32)");
  if (Nf <= kHierMaxFine && !brief) {
    const size_t lds = (size_t)kHierRays * (2 * N + Nf) * sizeof(float);
    hipLaunchKernelGGL(hier_resample_wave_kernel, grid1d(R, kHierRays), dim3(64), lds,
                       (hipStream_t)stream, dists, sdfs, R, N, inv_s, Nf, merged, fine, pos_coarse,
                       pos_fine);
    NA_CHECK_LAUNCH();
    return NA_OK;
  }
  hipLaunchKernelGGL(hier_resample_kernel, grid1d(R, kRayBlock), dim3(kRayBlock),
                     cdf_lds_bytes(N), (hipStream_t)stream, dists, sdfs, R, N, inv_s, Nf, merged,
                     fine, pos_coarse, pos_fine);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_scatter_merge(const float* src_a, const int32_t* pos_a, int32_t Na,
                                const float* src_b, const int32_t* pos_b, int32_t Nb, int64_t R,
                                float* out, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && Na >= 0 && Nb >= 0, "bad sizes");
  if (R == 0 || Na + Nb == 0) return NA_OK;
  NA_CHECK_ARG(out && (Na == 0 || (src_a && pos_a)) && (Nb == 0 || (src_b && pos_b)), "null pointer");
  hipLaunchKernelGGL(scatter_merge_kernel, grid1d(R * (Na + Nb)), dim3(256), 0, (hipStream_t)stream,
                     src_a, pos_a, Na, src_b, pos_b, Nb, R, out);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

static NeusIn make_neus(const float* ray_unit, const float* sdfs, const float* grads,
                        const float* dists, const float* far, const uint8_t* outside,
                        float outside_val, const float* s_var, float progress, float anneal_end,
                        int64_t R, int32_t N) {
  NeusIn p;
  p.ray = ray_unit; p.sdfs = sdfs; p.grads = grads; p.dists = dists; p.far = far;
  p.outside = outside; p.outside_val = outside_val; p.s_var = s_var;
  float ratio = progress / anneal_end;  // _get_iter_cos: min(progress / anneal_end, 1)
  p.anneal_ratio = ratio < 1.0f ? ratio : 1.0f;
  p.R = R; p.N = N;
  p.off = nullptr; p.ray_idx = nullptr;
  return p;
}

extern "C" int na_neus_alpha_fwd(const float* ray_unit, const float* sdfs, const float* grads,
                                 const float* dists, const float* far, const uint8_t* outside,
                                 float outside_val, const float* s_var, float progress,
                                 float anneal_end, int64_t R, int32_t N, float* alpha,
                                 na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 1, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(ray_unit && sdfs && grads && dists && s_var && alpha, "null pointer");
  NA_CHECK_ARG(anneal_end > 0.0f, "anneal_end must be > 0");
  NeusIn p = make_neus(ray_unit, sdfs, grads, dists, far, outside, outside_val, s_var, progress,
                       anneal_end, R, N);
  hipLaunchKernelGGL(neus_alpha_fwd_kernel, grid1d(R * N), dim3(256), 0, (hipStream_t)stream, p, alpha);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_neus_alpha_bwd(const float* ray_unit, const float* sdfs, const float* grads,
                                 const float* dists, const float* far, const uint8_t* outside,
                                 float outside_val, const float* s_var, float progress,
                                 float anneal_end, int64_t R, int32_t N, const float* dalpha,
                                 float* dsdf, float* dgrad, float* ds_var, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 1, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(ray_unit && sdfs && grads && dists && s_var && dalpha && dsdf && dgrad && ds_var,
               "null pointer");
  NA_CHECK_ARG(anneal_end > 0.0f, "anneal_end must be > 0");
  NeusIn p = make_neus(ray_unit, sdfs, grads, dists, far, outside, outside_val, s_var, progress,
                       anneal_end, R, N);
  hipLaunchKernelGGL(neus_alpha_bwd_kernel, grid_reduce(R * N), dim3(256), 0, (hipStream_t)stream,
                     p, dalpha, dsdf, dgrad, ds_var);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_composite_fwd(const float* alpha, const float* q, int64_t R, int32_t N,
                                int32_t K, float* weights, float* out, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 1 && K >= 0 && K <= 4, "bad sizes (K <= 4)");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(alpha && weights && (K == 0 || (q && out)), "null pointer");
  hipLaunchKernelGGL(composite_fwd_kernel, grid1d(R, kRayBlock), dim3(kRayBlock), 0,
                     (hipStream_t)stream, alpha, q, R, N, K, weights, out);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_composite_bwd(const float* alpha, const float* q, const float* weights,
                                int64_t R, int32_t N, int32_t K, const float* dout,
                                const float* dweights, float* dalpha, float* dq,
                                na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 1 && K >= 0 && K <= 4, "bad sizes (K <= 4)");
  NA_CHECK_ARG((size_t)N * kRayBlock * sizeof(float) <= 65536, "N too large (<= 256)");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(alpha && weights && dalpha, "null pointer");
  NA_CHECK_ARG(K == 0 || q, "q needed when K > 0");
  hipLaunchKernelGGL(composite_bwd_kernel, grid1d(R, kRayBlock), dim3(kRayBlock),
                     (size_t)N * kRayBlock * sizeof(float), (hipStream_t)stream, alpha, q,
                     weights, R, N, K, dout, dweights, dalpha, dq);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_weighted_sum_fwd(const float* q, const float* w, int64_t R, int32_t N,
                                   int32_t K, float* out, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 1 && K >= 1, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(q && w && out, "null pointer");
  hipLaunchKernelGGL(weighted_sum_fwd_kernel, grid1d(R * K), dim3(256), 0, (hipStream_t)stream, q,
                     w, R, N, K, out);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_weighted_sum_bwd(const float* q, const float* w, int64_t R, int32_t N,
                                   int32_t K, const float* dout, float* dq, float* dw,
                                   na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && N >= 1 && K >= 1, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(q && w && dout, "null pointer");
  hipLaunchKernelGGL(weighted_sum_bwd_kernel, grid1d(R * N), dim3(256), 0, (hipStream_t)stream, q,
                     w, R, N, K, dout, dq, dw);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_taps_points(const float* x, int64_t n, float eps, float* out,
                              na_stream_t stream) {
  NA_CHECK_ARG(n >= 0, "bad size");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(x && out, "null pointer");
  hipLaunchKernelGGL(taps_points_kernel, grid1d(n * 3), dim3(256), 0, (hipStream_t)stream, x, n,
                     eps, out);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_taps_combine_fwd(const float* s_taps, const float* sdf, int64_t n, float eps,
                                   float eps_sq, float* grad, float* hess, na_stream_t stream) {
  NA_CHECK_ARG(n >= 0, "bad size");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(s_taps && grad && (!hess || sdf), "null pointer");
  hipLaunchKernelGGL(taps_combine_fwd_kernel, grid1d(n), dim3(256), 0, (hipStream_t)stream,
                     s_taps, sdf, n, eps, eps_sq, grad, hess);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_taps_combine_bwd(int64_t n, float eps, float eps_sq, const float* dgrad,
                                   const float* dhess, float* ds_taps, float* dsdf,
                                   int32_t add_dsdf, na_stream_t stream) {
  NA_CHECK_ARG(n >= 0, "bad size");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(ds_taps, "null pointer");
  hipLaunchKernelGGL(taps_combine_bwd_kernel, grid1d(n), dim3(256), 0, (hipStream_t)stream, n,
                     eps, eps_sq, dgrad, dhess, ds_taps, dsdf, add_dsdf);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_rgb_input_fwd(const float* x, const float* ray_unit, int64_t n_per_ray,
                                const float* grad, int32_t normalize, int64_t n, int32_t col0,
                                void* out, int32_t out_dtype, int64_t ld, na_stream_t stream) {
  NA_CHECK_ARG(n >= 0 && n_per_ray >= 1 && col0 >= 0 && ld >= col0 + 22, "bad sizes");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(x && ray_unit && grad && out, "null pointer");
  // a tail of exactly 24 columns on 16-byte boundaries goes out as vector stores
  const int64_t eb = out_dtype == NA_BF16 ? 2 : 4;
  const int vec24 = ld - col0 == 24 && ((uintptr_t)out % 16) == 0 && (ld * eb) % 16 == 0 &&
                    (col0 * eb) % 16 == 0;
  if (out_dtype == NA_BF16)
    hipLaunchKernelGGL(rgb_input_fwd_kernel<bf16_t>, grid1d(n), dim3(256), 0, (hipStream_t)stream,
                       x, ray_unit, n_per_ray, grad, normalize, n, col0, (bf16_t*)out, ld, vec24);
  else
    hipLaunchKernelGGL(rgb_input_fwd_kernel<float>, grid1d(n), dim3(256), 0, (hipStream_t)stream,
                       x, ray_unit, n_per_ray, grad, normalize, n, col0, (float*)out, ld, vec24);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_rgb_input_bwd(const float* grad, int32_t normalize, int64_t n, int32_t col0,
                                const void* dy, int32_t dy_dtype, int64_t ld, float* dgrad,
                                int32_t add, na_stream_t stream) {
  NA_CHECK_ARG(n >= 0 && ld >= col0 + 22, "bad sizes");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(grad && dy && dgrad, "null pointer");
  if (dy_dtype == NA_BF16)
    hipLaunchKernelGGL(rgb_input_bwd_kernel<bf16_t>, grid1d(n), dim3(256), 0, (hipStream_t)stream,
                       grad, normalize, n, col0, (const bf16_t*)dy, ld, dgrad, add);
  else
    hipLaunchKernelGGL(rgb_input_bwd_kernel<float>, grid1d(n), dim3(256), 0, (hipStream_t)stream,
                       grad, normalize, n, col0, (const float*)dy, ld, dgrad, add);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_sdf_losses_fwd(const float* grad, const float* hess, const uint8_t* outside,
                                 int64_t n, int64_t n_per_ray, float* sums, na_stream_t stream) {
  NA_CHECK_ARG(n >= 0 && n_per_ray >= 1, "bad sizes");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(sums, "null pointer");
  hipLaunchKernelGGL(sdf_losses_fwd_kernel, grid_reduce(n), dim3(256), 0, (hipStream_t)stream,
                     grad, hess, outside, n, n_per_ray, sums);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_sdf_losses_bwd(const float* grad, const float* hess, const uint8_t* outside,
                                 int64_t n, int64_t n_per_ray, const float* w, float* dgrad,
                                 int32_t add_dgrad, float* dhess, na_stream_t stream) {
  NA_CHECK_ARG(n >= 0 && n_per_ray >= 1, "bad sizes");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(w && (!dgrad || grad) && (!dhess || hess), "null pointer");
  hipLaunchKernelGGL(sdf_losses_bwd_kernel, grid1d(n), dim3(256), 0, (hipStream_t)stream, grad,
                     hess, outside, n, n_per_ray, w, dgrad, add_dgrad, dhess);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_taps_delta_fwd(const float* ds, const float* sc, const float* sdf, int64_t n,
                                 float eps, float eps_sq, float* grad, float* hess,
                                 na_stream_t stream) {
  NA_CHECK_ARG(n >= 0, "bad size");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(ds && grad && (!hess || (sc && sdf)), "null pointer");
  hipLaunchKernelGGL(taps_delta_fwd_kernel, grid1d(n), dim3(256), 0, (hipStream_t)stream, ds, sc,
                     sdf, n, eps, eps_sq, grad, hess);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_taps_delta_bwd(int64_t n, float eps, float eps_sq, const float* dgrad,
                                 const float* dhess, float* dds, float* dsc, float* dsdf,
                                 na_stream_t stream) {
  NA_CHECK_ARG(n >= 0, "bad size");
  if (n == 0) return NA_OK;
  NA_CHECK_ARG(dds, "null pointer");
  hipLaunchKernelGGL(taps_delta_bwd_kernel, grid1d(n), dim3(256), 0, (hipStream_t)stream, n, eps,
                     eps_sq, dgrad, dhess, dds, dsc, dsdf);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

// ---------------------------------------------------------------------------
// packed (ragged) rays
// ---------------------------------------------------------------------------
extern "C" int na_packed_ray_index(const int32_t* offsets, int64_t R, int32_t* ray_idx,
                                   na_stream_t stream) {
  NA_CHECK_ARG(R >= 0, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(offsets && ray_idx, "null pointer");
  hipLaunchKernelGGL(packed_ray_index_kernel, grid1d(R), dim3(256), 0, (hipStream_t)stream,
                     offsets, R, ray_idx);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_composite_packed_fwd(const float* alpha, const float* q, const int32_t* offsets,
                                       int64_t R, int32_t K, float* weights, float* out,
                                       na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && K >= 0 && K <= 4, "bad sizes (K <= 4)");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(offsets && alpha && weights && (K == 0 || (q && out)), "null pointer");
  const int rb = (int)tune_value(TUNE_PACKED_RAYS);
  hipLaunchKernelGGL(composite_packed_fwd_kernel, grid1d(R, rb), dim3(rb), 0,
                     (hipStream_t)stream, alpha, q, offsets, R, K, weights, out);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_composite_packed_bwd(const float* alpha, const float* q, const float* weights,
                                       const int32_t* offsets, int64_t R, int32_t K,
                                       const float* dout, const float* dweights, float* dalpha,
                                       float* dq, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && K >= 0 && K <= 4, "bad sizes (K <= 4)");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(offsets && alpha && weights && dalpha, "null pointer");
  NA_CHECK_ARG(K == 0 || q, "q needed when K > 0");
  const int rb = (int)tune_value(TUNE_PACKED_RAYS);
  hipLaunchKernelGGL(composite_packed_bwd_kernel, grid1d(R, rb), dim3(rb), 0,
                     (hipStream_t)stream, alpha, q, weights, offsets, R, K, dout, dweights, dalpha,
                     dq);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_weighted_sum_packed_fwd(const float* q, const float* w, const int32_t* offsets,
                                          int64_t R, int32_t K, float* out, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && K >= 1, "bad sizes");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(q && w && offsets && out, "null pointer");
  hipLaunchKernelGGL(weighted_sum_packed_fwd_kernel, grid1d(R * K), dim3(256), 0,
                     (hipStream_t)stream, q, w, offsets, R, K, out);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_weighted_sum_packed_bwd(const float* q, const float* w, const int32_t* ray_idx,
                                          int64_t S, int32_t K, const float* dout, float* dq,
                                          float* dw, na_stream_t stream) {
  NA_CHECK_ARG(S >= 0 && K >= 1, "bad sizes");
  if (S == 0) return NA_OK;
  NA_CHECK_ARG(q && w && ray_idx && dout, "null pointer");
  hipLaunchKernelGGL(weighted_sum_packed_bwd_kernel, grid1d(S), dim3(256), 0, (hipStream_t)stream,
                     q, w, ray_idx, S, K, dout, dq, dw);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_neus_alpha_packed_fwd(const float* ray_unit, const float* sdfs,
                                        const float* grads, const float* dists, const float* far,
                                        const uint8_t* outside, float outside_val,
                                        const float* s_var, float progress, float anneal_end,
                                        const int32_t* offsets, const int32_t* ray_idx, int64_t S,
                                        float* alpha, na_stream_t stream) {
  NA_CHECK_ARG(S >= 0, "bad sizes");
  if (S == 0) return NA_OK;
  NA_CHECK_ARG(ray_unit && sdfs && grads && dists && s_var && alpha && offsets && ray_idx,
               "null pointer");
  NA_CHECK_ARG(anneal_end > 0.0f, "anneal_end must be > 0");
  NeusIn p = make_neus(ray_unit, sdfs, grads, dists, far, outside, outside_val, s_var, progress,
                       anneal_end, S, 1);
  p.off = offsets; p.ray_idx = ray_idx;
  hipLaunchKernelGGL(neus_alpha_fwd_kernel, grid1d(S), dim3(256), 0, (hipStream_t)stream, p, alpha);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_neus_alpha_packed_bwd(const float* ray_unit, const float* sdfs,
                                        const float* grads, const float* dists, const float* far,
                                        const uint8_t* outside, float outside_val,
                                        const float* s_var, float progress, float anneal_end,
                                        const int32_t* offsets, const int32_t* ray_idx, int64_t S,
                                        const float* dalpha, float* dsdf, float* dgrad,
                                        float* ds_var, na_stream_t stream) {
  NA_CHECK_ARG(S >= 0, "bad sizes");
  if (S == 0) return NA_OK;
  NA_CHECK_ARG(ray_unit && sdfs && grads && dists && s_var && dalpha && dsdf && dgrad && ds_var &&
                   offsets && ray_idx,
               "null pointer");
  NA_CHECK_ARG(anneal_end > 0.0f, "anneal_end must be > 0");
  NeusIn p = make_neus(ray_unit, sdfs, grads, dists, far, outside, outside_val, s_var, progress,
                       anneal_end, S, 1);
  p.off = offsets; p.ray_idx = ray_idx;
  hipLaunchKernelGGL(neus_alpha_bwd_kernel, grid_reduce(S), dim3(256), 0, (hipStream_t)stream, p,
                     dalpha, dsdf, dgrad, ds_var);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

// Persistent grid of the fused packed kernels: rays_per_wg-thread workgroups,
// at most wg_per_cu of them per CU, never more than the ray chunks need.
static dim3 packed_persistent_grid(int64_t R, int rb) {
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    ncu = 256;
  const int64_t chunks = (R + kPackedChunk - 1) / kPackedChunk, waves = rb / 64;
  const int64_t want = (chunks + waves - 1) / waves;
  const int64_t cap = (int64_t)ncu * tune_value(TUNE_PACKED_WG_PER_CU);
  return dim3((unsigned)std::max<int64_t>(1, std::min(want, cap)));
}

extern "C" int na_neus_composite_packed_fwd(const float* ray_unit, const float* sdfs,
                                            const float* grads, const float* dists,
                                            const float* far, const uint8_t* outside,
                                            float outside_val, const float* s_var, float progress,
                                            float anneal_end, const int32_t* offsets, int64_t R,
                                            const float* q, int32_t K, float* alpha,
                                            float* weights, float* out, int32_t* queue,
                                            na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && K >= 0 && K <= 4, "bad sizes (K <= 4)");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(ray_unit && sdfs && grads && dists && s_var && offsets && alpha && weights && queue,
               "null pointer");
  NA_CHECK_ARG(K == 0 || (q && out), "q and out are needed when K > 0");
  NA_CHECK_ARG(anneal_end > 0.0f, "anneal_end must be > 0");
  NA_CHECK_ARG(R <= (int64_t)0x7fffffff * kPackedChunk, "too many rays");
  NeusIn p = make_neus(ray_unit, sdfs, grads, dists, far, outside, outside_val, s_var, progress,
                       anneal_end, R, 1);
  p.off = offsets;
  const int rb = (int)tune_value(TUNE_PACKED_RAYS);
  hipLaunchKernelGGL(neus_composite_packed_fwd_kernel, packed_persistent_grid(R, rb), dim3(rb), 0,
                     (hipStream_t)stream, p, q, (int)K, alpha, weights, out, (int*)queue);
  NA_CHECK_LAUNCH();
  return NA_OK;
}

extern "C" int na_neus_composite_packed_bwd(const float* ray_unit, const float* sdfs,
                                            const float* grads, const float* dists,
                                            const float* far, const uint8_t* outside,
                                            float outside_val, const float* s_var, float progress,
                                            float anneal_end, const int32_t* offsets, int64_t R,
                                            const float* q, int32_t K, const float* alpha,
                                            const float* weights, const float* dout,
                                            const float* dweights, const float* dalpha,
                                            float* dsdf, float* dgrad, float* dq, float* ds_var,
                                            int32_t* queue, na_stream_t stream) {
  NA_CHECK_ARG(R >= 0 && K >= 0 && K <= 4, "bad sizes (K <= 4)");
  if (R == 0) return NA_OK;
  NA_CHECK_ARG(ray_unit && sdfs && grads && dists && s_var && offsets && alpha && weights && dsdf &&
                   dgrad && ds_var && queue,
               "null pointer");
  NA_CHECK_ARG(K == 0 || q, "q is needed when K > 0");
  NA_CHECK_ARG(anneal_end > 0.0f, "anneal_end must be > 0");
  NA_CHECK_ARG(R <= (int64_t)0x7fffffff * kPackedChunk, "too many rays");
  NeusIn p = make_neus(ray_unit, sdfs, grads, dists, far, outside, outside_val, s_var, progress,
                       anneal_end, R, 1);
  p.off = offsets;
  const int rb = (int)tune_value(TUNE_PACKED_RAYS);
  hipLaunchKernelGGL(neus_composite_packed_bwd_kernel, packed_persistent_grid(R, rb), dim3(rb), 0,
                     (hipStream_t)stream, p, q, (int)K, alpha, weights, dout, dweights, dalpha,
                     dsdf, dgrad, dq, ds_var, (int*)queue);
  NA_CHECK_LAUNCH();
  return NA_OK;
}
