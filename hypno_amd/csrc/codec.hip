// Q4_0 and Q8_0 block codecs on the device: the quantizers that produce
// hypno's packed weights and the dequantizers, bit-exact with the reference
// code.
//
// Two kernels each way.  The wave kernels (16-byte aligned buffers) move whole
// lines: a wave takes 64 consecutive blocks, eight lanes a block, so every
// access to the fp32 side is 1 KB of consecutive addresses (16 bytes a lane)
// and the packed side goes through LDS in 16-byte pieces.  A thread per block
// instead strides the fp32 side by 128 bytes and the packed side by single
// bytes; those kernels remain for other alignments.  Both are bound by memory.
// 58.7M weights (268 MB at Q4_0), thread and wave kernels: quantize 48 / 42
// us, dequantize 79 / 41 us.  Loads are plain (non-temporal 45 us), the fp32
// stores non-temporal (plain ones 41 us at Q4_0, but 52 against 44 at Q8_0).
#include "common.hpp"

namespace hypno {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <bool Q8>
struct Codec {
  static constexpr int kBytes = Q8 ? kQ8BlockBytes : kBlockBytes;
  static constexpr int kWave = 64 * kBytes;  // packed bytes of a wave's 64 blocks
  static_assert(kWave % 16 == 0, "whole 16-byte pieces");
  static constexpr float kMax = Q8 ? 127.0f : 7.0f;
  static constexpr float kMin = Q8 ? -127.0f : -8.0f;
  static constexpr int kZero = Q8 ? 128 : 8;
};

// The quantised integer of v by the reference's own steps (an IEEE division).
template <bool Q8>
__device__ __forceinline__ int quant_exact(float v, float scale) {
  const float r = roundf(v / scale);
  return r == r ? (int)fminf(fmaxf(r, Codec<Q8>::kMin), Codec<Q8>::kMax) : 0;
}

// quantize_q4_0_kernel / quantize_q8_0_kernel on whole waves.  32 IEEE
// divisions a block would bound it by VALU; v times the reciprocal of the
// scale (relative error under 2^-22) decides the integer unless it lies within
// kEps of a rounding boundary, or is not a number: then the lane divides.
template <bool Q8>
__global__ void __launch_bounds__(256)
quantize_wave_kernel(uint8_t* __restrict__ out, const float* __restrict__ src, size_t n_blocks) {
  using C = Codec<Q8>;
  constexpr float kEps = Q8 ? 1e-4f : 1e-5f;  // over 127 2^-22, 7 2^-22
  __shared__ __align__(16) uint8_t lds[4 * C::kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t b0 = ((size_t)blockIdx.x * 4 + wave) * 64;
  if (b0 >= n_blocks) return;  // wave-uniform (no barrier below)
  uint8_t* buf = lds + wave * C::kWave;
  uint16_t* h = reinterpret_cast<uint16_t*>(buf);
  const int g = lane >> 3, i = lane & 7;
  const int nv = (int)(n_blocks - b0 < 64 ? n_blocks - b0 : 64);
  f32x4 v[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int b = 8 * k + g < nv ? 8 * k + g : nv - 1;
    v[k] = load_global<f32x4>(src + (b0 + b) * kBlockElems + 4 * i);
  }
#pragma unroll
  for (int k = 0; k < 8; k++) {
    // |v| folded with fmaxf (NaN ignored), then over the block's eight lanes
    // (DPP quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror)
    float m = fmaxf(fmaxf(fmaxf(fmaxf(0.0f, fabsf(v[k][0])), fabsf(v[k][1])), fabsf(v[k][2])),
                    fabsf(v[k][3]));
    m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0xB1, 0xF, 0xF, false)));
    m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x4E, 0xF, 0xF, false)));
    m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x141, 0xF, 0xF, false)));
    const float s = m > 0.0f ? m / C::kMax : 1.0f;
    const _Float16 dh = (_Float16)s;
    const float scale = Q8 ? (float)dh : s;  // Q8_0 divides by the rounded scale
    const float inv = __builtin_amdgcn_rcpf(scale);
    int q[4];
    bool near = false;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float a = fmaf(fabsf(v[k][e]), inv, 0.5f);
      const float fl = floorf(a), fr = a - fl;
      near = near || !(fr > kEps && fr < 1.0f - kEps);
      const int n = (int)fminf(fl, 127.0f);
      q[e] = v[k][e] < 0.0f ? -n : n;
    }
    if (near) {
#pragma unroll
      for (int e = 0; e < 4; e++) q[e] = quant_exact<Q8>(v[k][e], scale);
    }
    const int at = (8 * k + g) * (C::kBytes / 2);
    if (i == 0) h[at] = __builtin_bit_cast(uint16_t, dh);
    if (Q8) {
      h[at + 1 + 2 * i] = (uint16_t)((q[0] + 128) | (q[1] + 128) << 8);
      h[at + 2 + 2 * i] = (uint16_t)((q[2] + 128) | (q[3] + 128) << 8);
    } else {
      h[at + 1 + i] =
          (uint16_t)((q[0] + 8) | (q[1] + 8) << 4 | (q[2] + 8) << 8 | (q[3] + 8) << 12);
    }
  }
  // (the wave's own LDS: its reads below follow its writes)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  uint8_t* o = out + b0 * C::kBytes;
  const int bytes = nv * C::kBytes;
#pragma unroll
  for (int p = 0; p < (C::kWave + 1023) / 1024; p++) {
    const int at = 16 * (64 * p + lane);
    if (at + 16 <= bytes) {
      __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(buf + at),
                                  reinterpret_cast<u32x4*>(o + at));
    } else if (at < bytes) {
      for (int c = at; c < bytes; c += 2)
        *reinterpret_cast<uint16_t*>(o + c) = *reinterpret_cast<const uint16_t*>(buf + c);
    }
  }
}

// dequantize_q4_0_kernel / dequantize_q8_0_kernel on whole waves.
template <bool Q8>
__global__ void __launch_bounds__(256)
dequantize_wave_kernel(float* __restrict__ out, const uint8_t* __restrict__ q, size_t n_blocks) {
  using C = Codec<Q8>;
  __shared__ __align__(16) uint8_t lds[4 * C::kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t b0 = ((size_t)blockIdx.x * 4 + wave) * 64;
  if (b0 >= n_blocks) return;  // wave-uniform (no barrier below)
  uint8_t* buf = lds + wave * C::kWave;
  const int nv = (int)(n_blocks - b0 < 64 ? n_blocks - b0 : 64);
  const uint8_t* w = q + b0 * C::kBytes;
  const int bytes = nv * C::kBytes;
  u32x4 r[(C::kWave + 1023) / 1024];
#pragma unroll
  for (int p = 0; p < (C::kWave + 1023) / 1024; p++) {
    const int at = 16 * (64 * p + lane);
    if (at + 16 <= bytes) r[p] = load_global<u32x4>(w + at);
  }
#pragma unroll
  for (int p = 0; p < (C::kWave + 1023) / 1024; p++) {
    const int at = 16 * (64 * p + lane);
    if (at + 16 <= bytes) {
      *reinterpret_cast<u32x4*>(buf + at) = r[p];
    } else if (at < bytes) {
      for (int c = at; c < bytes; c += 2)
        *reinterpret_cast<uint16_t*>(buf + c) = *reinterpret_cast<const uint16_t*>(w + c);
    }
  }
  // (the wave's own LDS: its reads below follow its writes)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const uint16_t* h = reinterpret_cast<const uint16_t*>(buf);
  const int g = lane >> 3, i = lane & 7;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int b = 8 * k + g;
    if (b >= nv) break;
    const int at = b * (C::kBytes / 2);
    const float d = f16_bits_to_f32(h[at]);
    f32x4 f;
    if (Q8) {
      const uint32_t lo = h[at + 1 + 2 * i], hi = h[at + 2 + 2 * i];
      f[0] = (float)((int)(lo & 0xFF) - 128) * d;
      f[1] = (float)((int)(lo >> 8) - 128) * d;
      f[2] = (float)((int)(hi & 0xFF) - 128) * d;
      f[3] = (float)((int)(hi >> 8) - 128) * d;
    } else {
      const uint32_t x = h[at + 1 + i];
#pragma unroll
      for (int e = 0; e < 4; e++) f[e] = (float)((int)((x >> (4 * e)) & 0xF) - 8) * d;
    }
    __builtin_nontemporal_store(
        f, reinterpret_cast<f32x4*>(out + (b0 + b) * kBlockElems + 4 * i));
  }
}

bool aligned16(const void* a, const void* b) {
  return (((uintptr_t)a | (uintptr_t)b) & 15) == 0;
}

}  // namespace

// Q4_0Block::quantize (quant.rs:49-71), one thread per 32-element block.
// amax folds |v| with fmaxf (NaN ignored, like f32::max); s = amax/7 in f32
// with IEEE division (1.0 for an all-zero block); d = f16 RNE(s);
// q = clamp(round_half_away(v / s), -8, 7) with NaN -> 0.
__global__ void __launch_bounds__(256)
quantize_q4_0_kernel(uint8_t* __restrict__ out, const float* __restrict__ src, size_t n_blocks) {
  const size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n_blocks) return;
  const float* v = src + b * kBlockElems;
  float vals[kBlockElems];
  float max_abs = 0.0f;
#pragma unroll
  for (int i = 0; i < kBlockElems; i++) {
    vals[i] = v[i];
    max_abs = fmaxf(max_abs, fabsf(vals[i]));
  }
  const float scale = max_abs > 0.0f ? max_abs / 7.0f : 1.0f;
  const uint16_t d = __builtin_bit_cast(uint16_t, (_Float16)scale);
  uint8_t* o = out + b * kBlockBytes;
  o[0] = (uint8_t)(d & 0xFF);
  o[1] = (uint8_t)(d >> 8);
#pragma unroll
  for (int i = 0; i < 16; i++) {
    uint32_t nib[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const float r = roundf(vals[2 * i + j] / scale);
      int q = 0;
      if (r == r) q = (int)fminf(fmaxf(r, -8.0f), 7.0f);
      nib[j] = (uint32_t)(q + 8) & 0x0Fu;
    }
    o[2 + i] = (uint8_t)(nib[0] | (nib[1] << 4));
  }
}

// Q4_0Block::dequantize (quant.rs:25-34): element 2i = (lo - 8) * d,
// element 2i+1 = (hi - 8) * d.  The product of an integer in [-8, 7] and an
// fp16 value is exact in fp32, so the output is bit-exact.
__global__ void __launch_bounds__(256)
dequantize_q4_0_kernel(float* __restrict__ out, const uint8_t* __restrict__ q, size_t n_blocks) {
  const size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n_blocks) return;
  const uint8_t* blk = q + b * kBlockBytes;
  const float scale = f16_bits_to_f32((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
  float* o = out + b * kBlockElems;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const uint32_t byte = blk[2 + i];
    o[2 * i] = (float)((int)(byte & 0x0F) - 8) * scale;
    o[2 * i + 1] = (float)((int)(byte >> 4) - 8) * scale;
  }
}

// quantize_f32_to_q8_0 (quant.rs:177-191), one thread per block: amax as for
// Q4_0; d = f16 RNE(amax / 127) (1.0 for an all-zero block); unlike Q4_0 each
// value is divided by the ROUNDED scale f32(d); q = clamp(round_half_away(v /
// f32(d)), -127, 127) with NaN -> 0 and +-inf -> +-127 (Rust's saturating
// cast); byte = q + 128.
__global__ void __launch_bounds__(256)
quantize_q8_0_kernel(uint8_t* __restrict__ out, const float* __restrict__ src, size_t n_blocks) {
  const size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n_blocks) return;
  const float* v = src + b * kBlockElems;
  float vals[kBlockElems];
  float max_abs = 0.0f;
#pragma unroll
  for (int i = 0; i < kBlockElems; i++) {
    vals[i] = v[i];
    max_abs = fmaxf(max_abs, fabsf(vals[i]));
  }
  const _Float16 dh = (_Float16)(max_abs > 0.0f ? max_abs / 127.0f : 1.0f);
  const uint16_t d = __builtin_bit_cast(uint16_t, dh);
  const float scale = (float)dh;
  uint8_t* o = out + b * kQ8BlockBytes;
  o[0] = (uint8_t)(d & 0xFF);
  o[1] = (uint8_t)(d >> 8);
#pragma unroll
  for (int i = 0; i < kBlockElems; i++) {
    const float r = roundf(vals[i] / scale);
    int q = 0;
    if (r == r) q = (int)fminf(fmaxf(r, -127.0f), 127.0f);
    o[2 + i] = (uint8_t)(q + 128);
  }
}

// Q8_0Block::dequantize (quant.rs:90-95): (u - 128) * d, exact in fp32.
__global__ void __launch_bounds__(256)
dequantize_q8_0_kernel(float* __restrict__ out, const uint8_t* __restrict__ q, size_t n_blocks) {
  const size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n_blocks) return;
  const uint8_t* blk = q + b * kQ8BlockBytes;
  const float scale = f16_bits_to_f32((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
  float* o = out + b * kBlockElems;
#pragma unroll
  for (int i = 0; i < kBlockElems; i++) o[i] = (float)((int)blk[2 + i] - 128) * scale;
}

hipError_t launch_quantize_q8_0(uint8_t* out, const float* src, size_t n_blocks, hipStream_t s) {
  if (n_blocks == 0) return hipSuccess;
  const size_t grid = (n_blocks + 255) / 256;
  if (aligned16(out, src)) {
    hipLaunchKernelGGL(quantize_wave_kernel<true>, dim3((unsigned)grid), dim3(256), 0, s, out, src,
                       n_blocks);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned)grid), dim3(256), 0, s, out, src, n_blocks);
  return hipGetLastError();
}

hipError_t launch_dequantize_q8_0(float* out, const uint8_t* q, size_t n_blocks, hipStream_t s) {
  if (n_blocks == 0) return hipSuccess;
  const size_t grid = (n_blocks + 255) / 256;
  if (aligned16(out, q)) {
    hipLaunchKernelGGL(dequantize_wave_kernel<true>, dim3((unsigned)grid), dim3(256), 0, s, out, q,
                       n_blocks);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(dequantize_q8_0_kernel, dim3((unsigned)grid), dim3(256), 0, s, out, q, n_blocks);
  return hipGetLastError();
}

hipError_t launch_quantize_q4_0(uint8_t* out, const float* src, size_t n_blocks, hipStream_t s) {
  if (n_blocks == 0) return hipSuccess;
  const size_t grid = (n_blocks + 255) / 256;
  if (aligned16(out, src)) {
    hipLaunchKernelGGL(quantize_wave_kernel<false>, dim3((unsigned)grid), dim3(256), 0, s, out, src,
                       n_blocks);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(quantize_q4_0_kernel, dim3((unsigned)grid), dim3(256), 0, s, out, src, n_blocks);
  return hipGetLastError();
}

hipError_t launch_dequantize_q4_0(float* out, const uint8_t* q, size_t n_blocks, hipStream_t s) {
  if (n_blocks == 0) return hipSuccess;
  const size_t grid = (n_blocks + 255) / 256;
  if (aligned16(out, q)) {
    hipLaunchKernelGGL(dequantize_wave_kernel<false>, dim3((unsigned)grid), dim3(256), 0, s, out, q,
                       n_blocks);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(dequantize_q4_0_kernel, dim3((unsigned)grid), dim3(256), 0, s, out, q, n_blocks);
  return hipGetLastError();
}

}  // namespace hypno
