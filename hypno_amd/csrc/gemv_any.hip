// One-token matrix-vector product on Q4_0 or Q8_0 weights for rows that the
// streaming GEMV (gemv_q4_0.hip) does not take: any K % 32 == 0 up to 32768
// (so whole blocks per row, on any 2-byte boundary), any x alignment.  fp32
// throughout, as the any-shape kernel it stands in for: the integer weights
// as exact fp16 values, widened in the FMAs; each block's dot product times d
// added to the row's sum.  The dot product is four chains of eight FMAs, not
// one of 32, and for Q8_0, whose any-shape kernel adds single products over 64
// lanes, chains of four that add up in fp64, as do its rows: errors against 64
// bits (any-shape kernel, one chain of 32, this) Q4_0 K 1120 1.1e-7, 1.1e-7,
// 9.0e-8; Q8_0 K 288 8.0e-8, 1.2e-7, 4.9e-8.
//
// Bound by HBM.  The any-shape kernel reads single bytes, 18 bytes apart per
// lane, one dependent block at a time (4096 x 11008: 101 us, 0.25 TB/s).  Here
// a wave takes kR rows together, its lanes consecutive blocks (kL lanes per
// row, so short rows share a wave): each block comes as one 16-byte and one
// 4-byte load of the window that starts at the dword at or below it, kDeep
// steps ahead, and x sits in LDS as [quarter-block][block] vectors, where the
// lanes' reads of consecutive blocks hit distinct banks and serve all kR rows.
// Measured per call, any-shape kernel -> this one: Q4_0 4096 x 11008 98 -> 11.3
// us (2.2 TB/s), 4096 x 2880 28.5 -> 5.5, 4228 x 20096 217 -> 23.3; Q8_0 4096 x
// 11008 61.5 -> 17.0 (2.8 TB/s; 16.4 as one chain of 32).
#include <type_traits>

#include "common.hpp"

namespace hypno {

namespace {

constexpr int kAThreads = 512;
constexpr int kAWaves = kAThreads / 64;
constexpr int kAR = 2;  // rows per wave (and lane group)

template <int F>
struct AnyFmt {
  static constexpr int kBytes = F == kFmtQ8_0 ? kQ8BlockBytes : kBlockBytes;
  static constexpr int kDw = F == kFmtQ8_0 ? 9 : 5;  // window dwords
  static constexpr int kDeep = F == kFmtQ8_0 ? 2 : 3;
  // Sums of eight products (Q8_0: four) are chains of FMAs; what they add up in.
  using Sum = std::conditional_t<F == kFmtQ8_0, double, float>;
};

template <int F>
struct AnyWin {
  uint32_t v[AnyFmt<F>::kDw];
};

// (the loops keep kDeep windows per row in registers)
template <int F, int L>
__global__ void __launch_bounds__(kAThreads)
gemv_any_kernel(float* __restrict__ y, const uint8_t* __restrict__ w, size_t w_bytes,
                const uint16_t* __restrict__ tail, const float* __restrict__ x,
                const float* __restrict__ bias, int n, int B, size_t y_tok) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the buffer builtins exist only in the device pass)
  using FT = AnyFmt<F>;
  constexpr int kDw = FT::kDw, kDeep = FT::kDeep;
  using Sum = typename FT::Sum;
  constexpr int kGroups = 64 / L;
  extern __shared__ __align__(16) float4 xs[];  // [8][B]
  y += (size_t)blockIdx.y * y_tok;
  x += (size_t)blockIdx.y * B * kBlockElems;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l = lane & (L - 1);
  const int g = lane / L;
  // Rows row0 + g kAR .. + kAR - 1 belong to this lane's group.
  const int row0 = (blockIdx.x * kAWaves + wave) * kGroups * kAR;
  const size_t row_bytes = (size_t)B * FT::kBytes;
  // A buffer from the wave's first row to the end of W, from the dword at or
  // below it; rows past N aim past the buffer and read zeros.
  const size_t start = row0 < n ? (size_t)row0 * row_bytes : 0;
  const size_t left = w_bytes - (start & ~(size_t)3);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(w + (start & ~(size_t)3)), (short)0,
      (int)(uint32_t)(left < 0xFFFFFF00u ? left : 0xFFFFFF00u), 0x00020000);
  const uint32_t first = (uint32_t)(start & 3);
  uint32_t off[kAR];
  bool live[kAR];
#pragma unroll
  for (int r = 0; r < kAR; r++) {
    const int k = g * kAR + r;
    live[r] = row0 + k < n;
    off[r] = first + (uint32_t)k * (uint32_t)row_bytes + (uint32_t)l * FT::kBytes;
  }
  const int steps = (B + L - 1) / L;
  // W ends 2 bytes into its last block's last window dword, which the buffer's
  // whole dwords leave out: the lane of that block reads the 2 bytes.
  const bool has_tail = tail && row0 + kGroups * kAR >= n;  // wave-uniform
  auto load = [&](int s, int r) __attribute__((always_inline)) -> AnyWin<F> {
    AnyWin<F> o;
    const uint32_t byte = off[r] + (uint32_t)s * (uint32_t)(L * FT::kBytes);
    const uint32_t a = live[r] && s * L + l < B ? byte & ~3u : 0xFFFFFF00u;
#pragma unroll
    for (int i = 0; i < kDw / 4; i++) {
      const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(rs, a + 16 * i, 0, 2);
#pragma unroll
      for (int k = 0; k < 4; k++) o.v[4 * i + k] = q[k];
    }
    o.v[kDw - 1] = __builtin_amdgcn_raw_buffer_load_b32(rs, a + 4 * (kDw - 1), 0, 2);
    if (has_tail && s * L + l == B - 1 && row0 + g * kAR + r == n - 1) o.v[kDw - 1] = *tail;
    return o;
  };
  AnyWin<F> win[kDeep][kAR];
#pragma unroll
  for (int d = 0; d < kDeep; d++)
#pragma unroll
    for (int r = 0; r < kAR; r++) win[d][r] = load(d, r);
  // x, while the first weights are on their way
  if (((uintptr_t)x & 15) == 0) {
    for (int i = t; i < B * 8; i += kAThreads)
      xs[(i & 7) * B + (i >> 3)] = load_global<float4>(x + 4 * i);
  } else {
    for (int i = t; i < B * 8; i += kAThreads)
      xs[(i & 7) * B + (i >> 3)] = make_float4(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
  }
  __syncthreads();
  Sum acc[kAR];
#pragma unroll
  for (int r = 0; r < kAR; r++) acc[r] = 0;
  for (int s0 = 0; s0 < steps; s0 += kDeep) {
#pragma unroll
    for (int d = 0; d < kDeep; d++) {
      const int s = s0 + d;
      if (s < steps) {
        const int b = min(s * L + l, B - 1);
        Sum dot[kAR];
#pragma unroll
        for (int r = 0; r < kAR; r++) dot[r] = 0;
#pragma unroll
        for (int c = 0; c < 4; c++) {  // eight elements at a time
          const float4 p = xs[(2 * c) * B + b], q = xs[(2 * c + 1) * B + b];
#pragma unroll
          for (int r = 0; r < kAR; r++) {
            const uint32_t(&v)[kDw] = win[d][r].v;
            const bool odd = (off[r] + (uint32_t)s * (uint32_t)(L * FT::kBytes)) & 2;
            const uint32_t sel = odd ? 0x07060504u : 0x05040302u;
            u32x4 h;
            if constexpr (F == kFmtQ4_0) {
              // slots e0,e4,e1,e5,e2,e6,e3,e7
              h = unpack8(__builtin_amdgcn_perm(v[c + 1], v[c], sel));
            } else {
              const uint32_t lo = __builtin_amdgcn_perm(v[2 * c + 1], v[2 * c], sel);
              const uint32_t hi = __builtin_amdgcn_perm(v[2 * c + 2], v[2 * c + 1], sel);
              h = unpack8_bytes(lo, hi);
            }
            half2v e[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const uint32_t u = h[i];
              e[i] = __builtin_bit_cast(half2v, u);
            }
            float a = 0.0f;
            if constexpr (F == kFmtQ4_0) {
              a = fmaf((float)e[0][0], p.x, a);
              a = fmaf((float)e[1][0], p.y, a);
              a = fmaf((float)e[2][0], p.z, a);
              a = fmaf((float)e[3][0], p.w, a);
              a = fmaf((float)e[0][1], q.x, a);
              a = fmaf((float)e[1][1], q.y, a);
              a = fmaf((float)e[2][1], q.z, a);
              a = fmaf((float)e[3][1], q.w, a);
            } else {
              a = fmaf((float)e[0][0], p.x, a);
              a = fmaf((float)e[0][1], p.y, a);
              a = fmaf((float)e[1][0], p.z, a);
              a = fmaf((float)e[1][1], p.w, a);
              dot[r] += (Sum)a;
              a = (float)e[2][0] * q.x;
              a = fmaf((float)e[2][1], q.y, a);
              a = fmaf((float)e[3][0], q.z, a);
              a = fmaf((float)e[3][1], q.w, a);
            }
            dot[r] += (Sum)a;
          }
        }
#pragma unroll
        for (int r = 0; r < kAR; r++) {
          const bool odd = (off[r] + (uint32_t)s * (uint32_t)(L * FT::kBytes)) & 2;
          const float sc = f16_bits_to_f32(odd ? win[d][r].v[0] >> 16 : win[d][r].v[0] & 0xFFFFu);
          // (a lane past the row's blocks holds zeros, but x may hold inf or NaN)
          if (s * L + l < B) acc[r] = fma((Sum)sc, dot[r], acc[r]);
          win[d][r] = load(s + kDeep, r);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kAR; r++) {
    Sum v = acc[r];
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int row = row0 + g * kAR + r;
    // Integers times x leave fp32 where weights times x may not (|x| from 2^120
    // on): a row that is not finite is computed again from the weights.
    const bool again = live[r] && !(fabsf((float)v) < __builtin_inff());
    if (__any(again)) {
      float u = 0.0f;
      if (again) {
        for (int b = l; b < B; b += L) {
          const uint8_t* blk = w + (size_t)row * row_bytes + (size_t)b * FT::kBytes;
          const float d = f16_bits_to_f32((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
          for (int i = 0; i < kBlockElems; i++) {
            const int q = F == kFmtQ8_0 ? (int)blk[2 + i] - 128
                                        : (int)((blk[2 + i / 2] >> (4 * (i & 1))) & 15) - 8;
            u = fmaf((float)q * d, x[b * kBlockElems + i], u);
          }
        }
      }
#pragma unroll
      for (int o = L / 2; o > 0; o >>= 1) u += __shfl_xor(u, o, 64);
      if (again) v = u;
    }
    if (l == 0 && live[r]) y[row] = (float)v + (bias ? bias[row] : 0.0f);
  }
#endif
}

}  // namespace

// Whole blocks per row, x within LDS, w dword-aligned; a row group's offsets
// in 32 bits follow from K <= 32768.
bool gemv_any_ok(int fmt, const uint8_t* w, size_t w_len, size_t n, size_t m) {
  if (n == 0 || m == 0 || m % kBlockElems != 0 || m > 32768) return false;
  if (((uintptr_t)w & 3) != 0 || n > (size_t)0x7FFFFFF) return false;
  const size_t bytes = fmt == kFmtQ8_0 ? kQ8BlockBytes : kBlockBytes;
  return w_len / bytes >= n * (m / kBlockElems);
}

template <int F>
static hipError_t launch_any(float* y, const uint8_t* w, size_t w_bytes, const uint16_t* tail,
                             const float* x, const float* bias, size_t n, size_t m, size_t batch,
                             hipStream_t s) {
  const int B = (int)(m / kBlockElems);
  const size_t lds = (size_t)B * 128;
  auto go = [&](auto kernel, int L) -> hipError_t {
    hipError_t e = set_lds_limit(reinterpret_cast<const void*>(kernel), 32768 * 4);
    if (e != hipSuccess) return e;
    const size_t per = (size_t)kAWaves * (64 / L) * kAR;
    for (size_t t = 0; t < batch; t += 65535) {
      const unsigned cnt = (unsigned)(batch - t < 65535 ? batch - t : 65535);
      hipLaunchKernelGGL(kernel, dim3((unsigned)((n + per - 1) / per), cnt), dim3(kAThreads), lds,
                         s, y + t * n, w, w_bytes, tail, x + t * m, bias, (int)n, B, n);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
  };
  if (B <= 8) return go(gemv_any_kernel<F, 8>, 8);
  if (B <= 16) return go(gemv_any_kernel<F, 16>, 16);
  if (B <= 32) return go(gemv_any_kernel<F, 32>, 32);
  return go(gemv_any_kernel<F, 64>, 64);
}

hipError_t launch_gemv_any(int fmt, float* y, const uint8_t* w, size_t w_len, const float* x,
                           const float* bias, size_t n, size_t m, size_t batch, hipStream_t s) {
  const size_t row_bytes =
      m / kBlockElems * (size_t)(fmt == kFmtQ8_0 ? kQ8BlockBytes : kBlockBytes);
  // Whole dwords of W; where N rows end at 2 mod 4 and the buffer ends with
  // them, the last 2 bytes go apart.
  const size_t end = n * row_bytes;
  const bool cut = (end & 3) != 0 && w_len < end + 2;
  const size_t w_bytes = cut ? end - 2 : (end + 3) / 4 * 4;
  const uint16_t* tail = cut ? reinterpret_cast<const uint16_t*>(w + end - 2) : nullptr;
  return fmt == kFmtQ8_0 ? launch_any<kFmtQ8_0>(y, w, w_bytes, tail, x, bias, n, m, batch, s)
                         : launch_any<kFmtQ4_0>(y, w, w_bytes, tail, x, bias, n, m, batch, s);
}

}  // namespace hypno
