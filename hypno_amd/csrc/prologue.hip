// The decode step's neighbours of the GEMV as device kernels: RMS norm
// (kernels.rs:592-625) and silu(gate) * up (transformer.rs:446-449,
// turbo.rs:235-237).  The streaming GEMV applies both as prologues of its
// activation staging (gemv_q4_0.hip); these stand-alone kernels serve the
// other paths (any K, batched rows) and the C ABI's hypno_hip_rms_norm_dev /
// hypno_hip_silu_mul_dev.
#include "common.hpp"

namespace hypno {

namespace {

constexpr int kNormThreads = 256;

// One work-group per row.  Sum of squares: per-thread FMA chains, wave sums,
// then the waves' sums in a fixed order.  Elements below n - n % 8 are
// x * inv_rms * w, the last n % 8 are x / sqrt(mean + eps) * w, the two forms
// of kernels.rs:611-616.
__global__ void __launch_bounds__(kNormThreads)
rms_norm_rows_kernel(float* out, const float* x, const float* __restrict__ weight, size_t n,
                     float eps) {
  __shared__ float wsum[kNormThreads / 64];
  const size_t row = blockIdx.x;
  const float* xr = x + row * n;
  float* orow = out + row * n;
  const int t = threadIdx.x;
  float ss = 0.0f;
  for (size_t i = t; i < n; i += kNormThreads) ss = fmaf(xr[i], xr[i], ss);
  ss = wave_sum(ss);
  if ((t & 63) == 0) wsum[t >> 6] = ss;
  __syncthreads();
  float tot = 0.0f;
#pragma unroll
  for (int w = 0; w < kNormThreads / 64; w++) tot += wsum[w];
  const float mean = tot / (float)n;
  const float root = sqrtf(mean + eps);
  const float inv = 1.0f / root;
  const size_t n8 = n - n % 8;
  // Every read of the row happens before any write (out may alias x): the
  // sum above is complete (barrier), and each element below is read and
  // written by the same thread.
  for (size_t i = t; i < n; i += kNormThreads) {
    const float v = xr[i];
    orow[i] = i < n8 ? v * inv * weight[i] : v / root * weight[i];
  }
}

// The same for rows that are whole 16-byte vectors: one work-group per row
// reads it once into registers (kV float4 per thread, all in flight
// together), so the row costs one memory latency instead of one per 256
// elements and is not read again for the output.  Bound by that latency for
// a few rows and by HBM for many.  Measured (one launch, before -> after):
// 8 x 4096 13.2 -> 3.4 us, 512 x 3072 11.7 -> 5.6, 2048 x 4096 23.4 -> 14.5
// (67 MB: 4.6 TB/s).
template <int kV>
__global__ void __launch_bounds__(kNormThreads)
rms_norm_rows_vec_kernel(float* out, const float* x, const float* __restrict__ weight, int n,
                         float eps) {
  __shared__ float wsum[kNormThreads / 64];
  const float4* xr = reinterpret_cast<const float4*>(x + (size_t)blockIdx.x * n);
  float4* orow = reinterpret_cast<float4*>(out + (size_t)blockIdx.x * n);
  const float4* wv = reinterpret_cast<const float4*>(weight);
  const int t = threadIdx.x, nv = n / 4;
  float4 v[kV], w[kV];
#pragma unroll
  for (int u = 0; u < kV; u++) {
    const int i = t + u * kNormThreads;
    v[u] = i < nv ? load_global<float4>(xr + i) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
#pragma unroll
  for (int u = 0; u < kV; u++) {
    const int i = t + u * kNormThreads;
    w[u] = load_global<float4>(wv + (i < nv ? i : 0));
  }
  float ss = 0.0f;
#pragma unroll
  for (int u = 0; u < kV; u++) {
    ss = fmaf(v[u].x, v[u].x, ss);
    ss = fmaf(v[u].y, v[u].y, ss);
    ss = fmaf(v[u].z, v[u].z, ss);
    ss = fmaf(v[u].w, v[u].w, ss);
  }
  ss = wave_sum(ss);
  if ((t & 63) == 0) wsum[t >> 6] = ss;
  __syncthreads();
  float tot = 0.0f;
#pragma unroll
  for (int k = 0; k < kNormThreads / 64; k++) tot += wsum[k];
  const float mean = tot / (float)n;
  const float root = sqrtf(mean + eps);
  const float inv = 1.0f / root;
  const int nv8 = n / 8 * 2;  // vectors below n - n % 8
#pragma unroll
  for (int u = 0; u < kV; u++) {
    const int i = t + u * kNormThreads;
    if (i >= nv) break;
    float4 o;
    if (i < nv8) {
      o = make_float4(v[u].x * inv * w[u].x, v[u].y * inv * w[u].y, v[u].z * inv * w[u].z,
                      v[u].w * inv * w[u].w);
    } else {
      o = make_float4(v[u].x / root * w[u].x, v[u].y / root * w[u].y, v[u].z / root * w[u].z,
                      v[u].w / root * w[u].w);
    }
    orow[i] = o;
  }
}

__device__ __forceinline__ float silu(float g) { return g / (1.0f + expf(-g)); }

__global__ void __launch_bounds__(256)
silu_mul_kernel(float* out, const float* gate, const float* __restrict__ up, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    out[i] = silu(gate[i]) * up[i];
  }
}

// The same on 16-byte vectors, kSiluVecs of gate and of up per thread in flight
// together; the last n % 4 elements one a thread.  Every vector is read before
// its place is written, so out may be gate or up.  Bound by HBM (by the launch
// for a few tokens): a 4-byte load a thread per grid step kept too few bytes in
// flight.  Per launch, before -> after: 2048 x 14336 68.0 -> 64.8 us (5.4 TB/s),
// 512 x 14336 14.9 -> 14.0, 333 x 7200 8.2 -> 7.6; one vector a thread 64.2,
// 14.3 and 7.7, four 65.8, 14.4 and 7.8.
constexpr int kSiluVecs = 2;
__global__ void __launch_bounds__(256)
silu_mul_vec_kernel(float* out, const float* gate, const float* up, size_t n) {
  const size_t nv = n / 4;
  const float4* gv = reinterpret_cast<const float4*>(gate);
  const float4* uv = reinterpret_cast<const float4*>(up);
  const size_t first = (size_t)blockIdx.x * (256 * kSiluVecs) + threadIdx.x;
  float4 g[kSiluVecs], v[kSiluVecs];
#pragma unroll
  for (int k = 0; k < kSiluVecs; k++) {
    const size_t i = first + k * 256;
    const size_t j = i < nv ? i : 0;
    g[k] = load_global<float4>(gv + j);
    v[k] = load_global<float4>(uv + j);
  }
#pragma unroll
  for (int k = 0; k < kSiluVecs; k++) {
    const size_t i = first + k * 256;
    if (i >= nv) break;
    reinterpret_cast<float4*>(out)[i] =
        make_float4(silu(g[k].x) * v[k].x, silu(g[k].y) * v[k].y, silu(g[k].z) * v[k].z,
                    silu(g[k].w) * v[k].w);
  }
  const size_t e = 4 * nv + threadIdx.x;
  if (blockIdx.x == 0 && e < n) out[e] = silu(gate[e]) * up[e];
}

}  // namespace

hipError_t launch_rms_norm(float* out, const float* x, const float* weight, size_t n,
                           size_t rows, float eps, hipStream_t s) {
  if (n == 0 || rows == 0) return hipSuccess;
  // Rows of whole 16-byte vectors that fit the work-group's registers go to
  // the one-read kernel; any other width or alignment to the element loop.
  const bool vec = n % 4 == 0 && n <= (size_t)kNormThreads * 4 * 16 &&
                   (((uintptr_t)out | (uintptr_t)x | (uintptr_t)weight) & 15) == 0;
  if (vec) {
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3(kNormThreads), 0, s, out, x, weight,
                         (int)n, eps);
      return hipGetLastError();
    };
    if (n <= (size_t)kNormThreads * 4 * 4) return go(rms_norm_rows_vec_kernel<4>);
    if (n <= (size_t)kNormThreads * 4 * 8) return go(rms_norm_rows_vec_kernel<8>);
    return go(rms_norm_rows_vec_kernel<16>);
  }
  hipLaunchKernelGGL(rms_norm_rows_kernel, dim3((unsigned)rows), dim3(kNormThreads), 0, s, out, x,
                     weight, n, eps);
  return hipGetLastError();
}

hipError_t launch_silu_mul(float* out, const float* gate, const float* up, size_t n,
                           hipStream_t s) {
  if (n == 0) return hipSuccess;
  const size_t groups = (n / 4 + 256 * kSiluVecs - 1) / (256 * kSiluVecs);
  if (n >= 4 && groups <= 0xFFFFFF &&
      (((uintptr_t)out | (uintptr_t)gate | (uintptr_t)up) & 15) == 0) {
    hipLaunchKernelGGL(silu_mul_vec_kernel, dim3((unsigned)groups), dim3(256), 0, s, out, gate, up,
                       n);
    return hipGetLastError();
  }
  size_t grid = (n + 255) / 256;
  if (grid > 4096) grid = 4096;
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)grid), dim3(256), 0, s, out, gate, up, n);
  return hipGetLastError();
}

}  // namespace hypno
