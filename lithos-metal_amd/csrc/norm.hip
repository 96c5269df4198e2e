// The decode layer's RMSNorm as standalone ops (ops/norm.py:11-12): rmsnorm_stat (stat[t] = Σ_k h[t][k]²,
// kernels/common/rmsnorm_stat.metal:18-40) and norm_apply (x = bf16(h·rsqrt(Σ stat / K + eps)·w), w the (1 + w)
// weight, norm_apply.metal:24-51) — for a lowered graph whose norm does not feed a GEMV directly (the GEMVs fuse it
// on load and never launch these).
//
// MI355X design: a workgroup per row, a thread per 8-column vector (16-byte loads and stores) of up to 8192 columns; a
// wave's 64 vectors are one slice of the statistic (vec_sumsq), the slices meet in LDS and every thread adds them in
// order, so the result does not depend on scheduling. What bounds it is latency: the row and its weights are loaded at
// once and stay in registers, one memory round trip from launch to store: 8 rows of 5120 2.83 → 2.43 us back to back,
// rows of 16384 4.8 → 3.6 (256 threads read the row twice, and the weights after the statistic). Wider rows loop, reading
// the row twice.
#include "mi_common.h"

#include <algorithm>

namespace {

constexpr int NT = 1024;                        // threads at most: a wave per slice of up to 8192 columns

struct NormArgs {
  int t, k, ldh, ldx, parts;
  const uint16_t* h;
  float* stat_out;          // rmsnorm_stat: [t][parts] (parts = 1 here)
  const float* stat_in;     // norm_apply: [t][parts] partial sums, or null
  const float* w;           // (1 + w) [k]
  uint16_t* x;
  float eps;
};

// Σ x² of the row (every thread's result); v: the thread's first vector (zeros past the row). A round of the workgroup's
// waves takes as many slices; the rounds alternate between two LDS rows
__device__ __forceinline__ float row_sumsq(const uint16_t* row, int k, const uint32_t (&v)[4]) {
  __shared__ float sl[2][NT / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int n = (k + STAT_SLICE - 1) / STAT_SLICE;
  float s = vec_sumsq(v), t = 0.0f;
  for (int base = 0, buf = 0;; buf ^= 1) {
    s = wave_sum(s);
    if (lane == 0) sl[buf][w] = s;
    __syncthreads();
    for (int i = 0; i < min(waves, n - base); ++i) t += sl[buf][i];
    base += waves;
    if (base >= n) return t;
    const int c = (base + w) * STAT_SLICE + 8 * lane;
    const uint4 q = c < k ? *reinterpret_cast<const uint4*>(row + c) : uint4{0u, 0u, 0u, 0u};
    const uint32_t u[4] = {q.x, q.y, q.z, q.w};
    s = vec_sumsq(u);
  }
}

__global__ __launch_bounds__(NT) void rmsnorm_stat(NormArgs a) {
  const int t = blockIdx.x, c = 8 * threadIdx.x;
  const uint16_t* row = a.h + (long long)t * a.ldh;
  const uint4 q = c < a.k ? *reinterpret_cast<const uint4*>(row + c) : uint4{0u, 0u, 0u, 0u};
  const uint32_t v[4] = {q.x, q.y, q.z, q.w};
  const float s = row_sumsq(row, a.k, v);
  if (threadIdx.x == 0) a.stat_out[t] = s;
}

__global__ __launch_bounds__(NT) void norm_apply(NormArgs a) {
  const int t = blockIdx.x, c0 = 8 * threadIdx.x, cc = min(c0, a.k - 8);
  const uint16_t* row = a.h + (long long)t * a.ldh;
  const uint4 q = *reinterpret_cast<const uint4*>(row + cc);
  float4 w0 = *reinterpret_cast<const float4*>(a.w + cc), w1 = *reinterpret_cast<const float4*>(a.w + cc + 4);
  uint32_t v[4] = {q.x, q.y, q.z, q.w};
  float ssq = 0.0f;
  if (a.stat_in) {
    for (int i = 0; i < a.parts; ++i) ssq += a.stat_in[t * a.parts + i];
  } else {
    const uint32_t u[4] = {c0 < a.k ? v[0] : 0u, c0 < a.k ? v[1] : 0u, c0 < a.k ? v[2] : 0u, c0 < a.k ? v[3] : 0u};
    ssq = row_sumsq(row, a.k, u);
  }
  const float r = 1.0f / sqrtf(ssq / (float)a.k + a.eps);
  uint16_t* out = a.x + (long long)t * a.ldx;
  for (int c = c0; c < a.k;) {
    uint32_t o[4];
    norm_vec(v, r, w0, w1, o);
    *reinterpret_cast<uint4*>(out + c) = uint4{o[0], o[1], o[2], o[3]};
    c += 8 * blockDim.x;
    if (c < a.k) {                              // a row wider than the workgroup
      const uint4 n = *reinterpret_cast<const uint4*>(row + c);
      v[0] = n.x; v[1] = n.y; v[2] = n.z; v[3] = n.w;
      w0 = *reinterpret_cast<const float4*>(a.w + c);
      w1 = *reinterpret_cast<const float4*>(a.w + c + 4);
    }
  }
}

// a thread per vector, whole waves. More rows than CUs share them: half the threads, so that four fit a CU, and the rows
// past 4096 columns in rounds (1000 rows of 8192 with 1024 / 512 threads 8.0 / 7.0 us, of 8200 9.0 / 7.7, of 5120 6.2 /
// 6.1; 300 rows 4.4 / 4.3, 5.0 / 4.8, 3.7 / 3.9)
int threads_of(int k, int t) { return std::min(t > 256 ? NT / 2 : NT, (k / 8 + 63) / 64 * 64); }

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int check(const mi_norm_desc* d, const char* name) {
  MI_REQUIRE(d, "%s: null descriptor", name);
  MI_REQUIRE(d->t >= 1 && d->t <= 4096, "%s: t=%d must be in 1..4096", name, d->t);
  MI_REQUIRE(d->k >= 8 && d->k % 8 == 0, "%s: k=%d must be a positive multiple of 8", name, d->k);
  MI_REQUIRE(d->h && al16(d->h) && d->ldh >= d->k && d->ldh % 8 == 0,
             "%s: h must be 16-byte aligned rows with a stride >= k, multiple of 8", name);
  return MI_OK;
}

}  // namespace

extern "C" int mi_rmsnorm_stat(const mi_norm_desc* d, void* stream) {
  if (int rc = check(d, "mi_rmsnorm_stat")) return rc;
  MI_REQUIRE(d->stat, "mi_rmsnorm_stat: null stat");
  NormArgs a{d->t, d->k, d->ldh, 0, 1, d->h, d->stat, nullptr, nullptr, nullptr, 0.0f};
  hipLaunchKernelGGL(rmsnorm_stat, dim3(d->t), dim3(threads_of(d->k, d->t)), 0, static_cast<hipStream_t>(stream), a);
  MI_TRY_HIP(hipGetLastError(), "rmsnorm_stat launch");
  return MI_OK;
}

extern "C" int mi_norm_apply(const mi_norm_desc* d, void* stream) {
  if (int rc = check(d, "mi_norm_apply")) return rc;
  MI_REQUIRE(d->w && al16(d->w), "mi_norm_apply: w must be a 16-byte aligned float32 [k]");
  MI_REQUIRE(d->x && al16(d->x) && d->ldx >= d->k && d->ldx % 8 == 0, "mi_norm_apply: bad output x");
  MI_REQUIRE(!d->stat || d->stat_parts >= 1, "mi_norm_apply: stat_parts >= 1 with a stat");
  NormArgs a{d->t, d->k, d->ldh, d->ldx, d->stat_parts, d->h, nullptr, d->stat, d->w, d->x, d->eps};
  hipLaunchKernelGGL(norm_apply, dim3(d->t), dim3(threads_of(d->k, d->t)), 0, static_cast<hipStream_t>(stream), a);
  MI_TRY_HIP(hipGetLastError(), "norm_apply launch");
  return MI_OK;
}
