// fp32-accurate batched GEMM on bf16 operand parts, for gfx950:
// Y[M][N] = X[M][K] . W[N][K]^T (+ bias) with X = (x1 + x2 + x3) 2^e per token
// (all 24 bits, x_rows_split_kernel) and W = w1 + w2 (exact), and its users:
// column-major Q4_0 batches (kernels.rs:403-535, turbo.rs:322-326) and fp16
// batches whose rows are no multiple of 64.  All six products of the parts are
// exact and add up in fp32 on the matrix cores, smallest first.
//
// Column-major Q4_0: W_col[k][j] keeps 32 outputs j of one input k in a
// block, so the scale d changes with k inside an output's sum and cannot be
// applied to partial sums.  Each weight becomes a pair in registers instead:
// n d has at most 14 significant bits (3 of a 4-bit integer, 11 of d), w1 takes
// the first 8 and w2 the rest.  An fp16 weight (11 bits) splits the same way.
//
// A wave's 32 columns are one block column, so its stage of 64 K is 64 blocks,
// one a lane; they change hands inside the wave through 1.5 KB of LDS (16 byte
// writes and 10 16-byte reads a lane, no barrier).  An expansion pass before
// the GEMM (4 bytes written and read back per weight) took as long as the
// products; one pass over the weights per token, the other way to do it, 412 us
// a call for 128 tokens of 5632 x 2048 where this takes 35, 52 for 8 tokens
// of 14336 x 4096 (37).
//
// What bounds it: six MFMAs per product beside the pairs' VALU and LDS work
// on one issue port, and at few tokens the three launches of a call.  (Two fp16
// parts of x and three products: 28 us at 128 tokens of 5632 x 2048, but 22 bits
// of x, fewer beside an outlier.)
//
//  * Work-group = 8 waves on a 32 MT x 256 tile of Y, 32 columns a wave;
//    32x32x16 MFMAs.  fp16 weights: lane (n, h) loads the 64 bytes of its
//    column and lane half straight into registers, two stages of 64 K ahead;
//    column-major blocks are loaded three stages ahead.
//  * X: the parts' rows by DMA into a ring of LDS stages, 16-byte chunk c of
//    row r in slot c ^ ((r >> 1) & 7) (16 rows of an operand read hit distinct
//    banks); one barrier per stage publishes the stage two ahead.
//  * An infinity (or NaN) in a weight or token makes NaN of some products of
//    its parts: an output whose sum is NaN is computed again from the weights
//    and x as they came, in fp32.
#include <algorithm>

#include "common.hpp"

namespace hypno {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kPWaves = 8;
constexpr int kPThreads = 64 * kPWaves;
constexpr int kPBN = 32 * kPWaves;
constexpr int kPStageK = 64;
constexpr int kPRowBytes = kPStageK * 2;
constexpr int kPParts = 3;
constexpr int kPRing = 4;
// A wave's 64 column-major blocks in LDS: byte i of block k at i * kTPitch + k
// (16 rows whose 16-byte reads hit distinct banks), then the 64 scales.
[[maybe_unused]] constexpr int kTPitch = 80;
constexpr int kTBytes = 16 * kTPitch + 256;

struct PairArgs {
  float* y;
  const uint8_t* wh;   // fp16 [N][K] (not column-major)
  const uint8_t* xh;   // bf16 [M][Kp], a plane of M rows per part
  const float* bias;
  const int* xexp;     // [M]: row m of xh holds X row m times 2^-xexp[m]
  const uint8_t* col;  // column-major blocks
  size_t col_blocks;   // whole blocks in that buffer
  uint32_t col_bytes;  // its bytes
  const float* x;      // X as it came
  float* part;         // [splits][M][N] partial planes (splits > 1)
  uint32_t w_bytes;    // bytes of wh
  uint32_t x_bytes;    // bytes of one xh plane (rows past M read zeros)
  uint32_t y_bytes;    // M x N x 4
  int M, N, K;
  int steps;           // 64-K stages of a row (the last may be half)
  int tiles_m, tiles_n;
  int splits;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t prsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           0x00020000);
}

// kCol: column-major Q4_0 blocks (else fp16 rows).
template <int MT, bool kCol>
__global__ void __launch_bounds__(kPThreads, 1) gemm_pair_kernel(const PairArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the buffer builtins exist only in the device pass)
  constexpr int BM = 32 * MT;
  constexpr int kRows = (kPParts * BM + 63) / 64 * 64;  // whole DMAs of every wave
  constexpr int kTile = kRows * kPRowBytes;
  constexpr int kDx = kRows / 64;           // X DMAs per wave and stage
  constexpr int kWLoads = kCol ? 2 : 4;     // W loads per wave and stage
  extern __shared__ __align__(16) uint8_t smem[];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 31;
  const int h = lane >> 5;
  const int m0 = (blockIdx.x % a.tiles_m) * BM;
  const int n0 = (blockIdx.x / a.tiles_m) * kPBN;
  const int z = blockIdx.y;
  const int s0 = (int)((long long)a.steps * z / a.splits);
  const int s1 = (int)((long long)a.steps * (z + 1) / a.splits);
  const int steps = s1 - s0;

  // X DMA: instruction i of wave w fills LDS rows 8 (8 i + w) .. + 7 of the
  // slot (part p in rows BM p .. BM p + BM - 1; rows that only fill up the last
  // DMA read the last part again).
  const uint32_t x_row = (uint32_t)a.steps * kPRowBytes;
  uint32_t xvoff[kDx];
#pragma unroll
  for (int i = 0; i < kDx; i++) {
    const int row = 8 * (8 * i + wave) + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    xvoff[i] = (uint32_t)(m0 + row % BM) * x_row + (uint32_t)c * 16u;
  }
  auto issue_x = [&](int s) __attribute__((always_inline)) {  // stage min(s, steps-1) -> slot of s
    const int soff = (s0 + (s < steps ? s : steps - 1)) * kPRowBytes;
    uint8_t* slot = smem + (s % kPRing) * kTile;
#pragma unroll
    for (int i = 0; i < kDx; i++) {
      const int part = min(8 * (8 * i + wave) / BM, kPParts - 1);  // wave-uniform
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          prsrc(a.xh + (size_t)part * a.x_bytes, a.x_bytes),
          (__attribute__((address_space(3))) void*)(slot + 8 * (8 * i + wave) * kPRowBytes), 16,
          xvoff[i], soff, 0, 0);
    }
  };

  // W: lane (n, h) holds elements 32 h .. + 31 of column n's stage; MFMA j
  // takes 8 j .. + 7 of them.  fp16 rows: columns past N re-read column N - 1;
  // elements past K read as zeros (their own row's end is not the buffer's).
  const int ncol = n0 + 32 * wave + lr;
  const bool nvalid = ncol < a.N;
  const __amdgpu_buffer_rsrc_t whs = prsrc(a.wh, a.w_bytes);
  const uint32_t wvoff = (uint32_t)min(ncol, a.N - 1) * (uint32_t)a.K * 2u + 64u * h;
  struct Wreg {
    u32x4 h[4], l[4];  // w1 and w2 of elements 8 j .. + 7
  };
  // Two fp32 weights -> their first 8 bits and the rest, each two bf16.
  auto pair2 = [&](float p, float q, uint32_t& h, uint32_t& l) __attribute__((always_inline)) {
    const uint32_t ph = __float_as_uint(p) & 0xFFFF0000u, qh = __float_as_uint(q) & 0xFFFF0000u;
    h = __builtin_amdgcn_perm(qh, ph, 0x07060302u);
    l = __builtin_amdgcn_perm(__float_as_uint(q - __uint_as_float(qh)),
                              __float_as_uint(p - __uint_as_float(ph)), 0x07060302u);
  };
  struct Rows {
    u32x4 v[4];
  };
  auto load_w = [&](int s) __attribute__((always_inline)) -> Rows {
    const int sc = s0 + (s < steps ? s : steps - 1);
    const uint32_t v = sc * kPStageK + 32 * h < a.K ? wvoff : 0xFFFFFF00u;
    const uint32_t off = v == 0xFFFFFF00u ? v : v + (uint32_t)sc * kPRowBytes;
    Rows r;
#pragma unroll
    for (int j = 0; j < 4; j++) r.v[j] = __builtin_amdgcn_raw_buffer_load_b128(whs, off + 16 * j, 0, 0);
    return r;
  };
  auto split_rows = [&](const Rows& r) __attribute__((always_inline)) -> Wreg {
    Wreg w;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t u = r.v[j][i];
        uint32_t h2, l2;
        pair2(f16_bits_to_f32(u & 0xFFFFu), f16_bits_to_f32(u >> 16), h2, l2);
        w.h[j][i] = h2;
        w.l[j][i] = l2;
      }
    return w;
  };
  // Column-major: lane i loads block (k = 64 s + i, the wave's block column),
  // 18 bytes from an even address, as the five dwords around it; zeros past
  // K, past N and past a short buffer.
  const __amdgpu_buffer_rsrc_t cs = prsrc(a.col, a.col_bytes);
  const int nb = a.N / kBlockElems, bc = n0 / kBlockElems + wave;
  struct Raw {
    u32x4 v;
    uint32_t v4;
    uint32_t odd;  // 0: the block starts with v; 2: two bytes later; 4: no block
  };
  auto load_col = [&](int s) __attribute__((always_inline)) -> Raw {
    const int k = (s0 + (s < steps ? s : steps - 1)) * kPStageK + lane;
    const size_t g = (size_t)k * nb + bc;
    const bool ok = k < a.K && bc < nb && g < a.col_blocks;
    const uint32_t byte = (uint32_t)(g * kBlockBytes);
    const uint32_t off = ok ? byte & ~3u : 0xFFFFFF00u;
    Raw r;
    r.v = __builtin_amdgcn_raw_buffer_load_b128(cs, off, 0, 0);
    r.v4 = __builtin_amdgcn_raw_buffer_load_b32(cs, off + 16, 0, 0);
    r.odd = ok ? byte & 2u : 4u;
    return r;
  };
  uint8_t* const tb = smem + kPRing * kTile + wave * kTBytes;  // this wave's own
  auto expand = [&](const Raw& r) __attribute__((always_inline)) -> Wreg {
    const uint32_t sel = r.odd & 2u ? 0x07060504u : 0x05040302u;
    const uint32_t v[5] = {r.v[0], r.v[1], r.v[2], r.v[3], r.v4};
    const uint32_t d = r.odd & 2u ? v[0] >> 16 : r.odd ? 0u : v[0] & 0xFFFFu;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t q = __builtin_amdgcn_perm(v[j + 1], v[j], sel);
#pragma unroll
      for (int b = 0; b < 4; b++) tb[(4 * j + b) * kTPitch + lane] = (uint8_t)(q >> (8 * b));
    }
    // (16 d: v_cvt_off_f32_i4 below gives (nibble - 8) / 16)
    *reinterpret_cast<float*>(tb + 16 * kTPitch + 4 * lane) = 16.0f * f16_bits_to_f32(d);
    // (LDS keeps a wave's accesses in order: these reads follow the writes,
    // and the next stage's writes follow them)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    u32x4 qb[2], db[8];
#pragma unroll
    for (int j = 0; j < 2; j++)
      qb[j] = *reinterpret_cast<const u32x4*>(tb + (lr >> 1) * kTPitch + 32 * h + 16 * j);
#pragma unroll
    for (int j = 0; j < 8; j++)
      db[j] = *reinterpret_cast<const u32x4*>(tb + 16 * kTPitch + 128 * h + 16 * j);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int sh = 4 * (lr & 1);
    Wreg w;
#pragma unroll
    for (int e = 0; e < 32; e += 4) {  // four elements of a dword
      const uint32_t n4 = (qb[e / 16][e / 4 % 4] >> sh) ^ 0x88888888u;
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t di = db[e / 4][i];
        p[i] = __builtin_amdgcn_cvt_off_f32_i4(n4 >> (8 * i)) * __uint_as_float(di);
      }
      uint32_t h2, l2;
      pair2(p[0], p[1], h2, l2);
      w.h[e / 8][e / 2 % 4] = h2;
      w.l[e / 8][e / 2 % 4] = l2;
      pair2(p[2], p[3], h2, l2);
      w.h[e / 8][e / 2 % 4 + 1] = h2;
      w.l[e / 8][e / 2 % 4 + 1] = l2;
    }
    return w;
  };

  uint32_t aoff[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    aoff[j] = (uint32_t)lr * kPRowBytes + (((4 * h + j) ^ ((lr >> 1) & 7)) << 4);
  auto read_a = [&](int s, int i, int p, int j) __attribute__((always_inline)) -> u32x4 {
    return *reinterpret_cast<const u32x4*>(smem + (s % kPRing) * kTile + aoff[j] +
                                           (32 * i + BM * p) * kPRowBytes);
  };

  floatx16 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;

  // Prologue: X of stages 0..2 in flight, stages 0 and 1 landed and published.
  Wreg wa, wb;
  Raw r1, r2;  // blocks of the next two stages
  Rows rn;     // rows of the next stage
  if constexpr (kCol) {
    r1 = load_col(0);
    r2 = load_col(1);
  } else {
    rn = load_w(0);
  }
  asm volatile("" ::: "memory");
  for (int i = 0; i < kPRing - 1; i++) issue_x(i);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kDx) : "memory");
  if constexpr (kCol) {
    wa = expand(r1);
    r1 = r2;
    r2 = load_col(2);
  } else {
    wa = split_rows(rn);
    rn = load_w(1);
  }
  // A stage is 3 MT steps, step t part 2 - t % 3 of row tile t / 3; operands are
  // read kAhead steps ahead (fewer registers where MT = 2 needs them).
  constexpr int kSteps = kPParts * MT;
  constexpr int kAhead = MT == 2 ? 2 : 3;
  static_assert(kSteps % kAhead == 0, "a step's registers are the same in every stage");
  u32x4 fa[kAhead][4];
  auto read_step = [&](int s, int t) __attribute__((always_inline)) {
    const int u = t % kSteps;
#pragma unroll
    for (int j = 0; j < 4; j++)
      fa[t % kAhead][j] = read_a(s + t / kSteps, u / kPParts, kPParts - 1 - u % kPParts, j);
  };
#pragma unroll
  for (int t = 0; t < kAhead; t++) read_step(0, t);
  // The sum moves to `tot` every kGroup stages, so no output is a chain of one
  // rounding per stage (512 tokens, 14336 x 4096 in one piece: 1.6e-7 off 64 bits
  // as one chain, 9.3e-8 so, 1.1e-7 the one-token kernel).
  constexpr int kGroup = 8;
  floatx16 tot[MT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) tot[i][r] = 0.0f;

  // At the end of stage s X(s+2), which went out in the stage before, has
  // landed: this stage's X DMAs and W loads are all younger.
  auto stage = [&](int s, const Wreg& w, Wreg& wn) __attribute__((always_inline)) {
    issue_x(s + kPRing - 1);
    asm volatile("" ::: "memory");
    if constexpr (kCol) {
      wn = expand(r1);
      r1 = r2;
      r2 = load_col(s + 3);
    } else {
      wn = split_rows(rn);
      rn = load_w(s + 2);
    }
    auto mfma = [&](u32x4 x, u32x4 y, floatx16 c) __attribute__((always_inline)) {
      return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c, 0, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < MT; i++) {
      // The stage's products add up from zero and then to the tile's sum, so
      // that sum is rounded once per 64 columns; the small products go first,
      // so the roundings at the stage sum's own size are four, not 24.
      floatx16 p;
#pragma unroll
      for (int r = 0; r < 16; r++) p[r] = 0.0f;
#pragma unroll
      for (int q = 0; q < kPParts; q++) {
        const int t = kPParts * i + q;
#pragma unroll
        for (int j = 0; j < 4; j++) p = mfma(fa[t % kAhead][j], w.l[j], p);
#pragma unroll
        for (int j = 0; j < 4; j++) p = mfma(fa[t % kAhead][j], w.h[j], p);
        read_step(s, t + kAhead);
      }
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][r] += p[r];
      __builtin_amdgcn_sched_barrier(0);
    }
    if (s % kGroup == kGroup - 1) {
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          tot[i][r] += acc[i][r];
          acc[i][r] = 0.0f;
        }
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kDx + kWLoads) : "memory");
  };
  int s = 0;
  for (; s + 1 < steps; s += 2) {
    stage(s, wa, wb);
    stage(s + 1, wb, wa);
  }
  if (s < steps) stage(s, wa, wb);
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] += tot[i][r];
  // Every DMA into LDS (the trailing re-reads included) has landed before
  // the work-group's LDS is released.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // Register r of a lane holds output row m0 + 32 i + 8 (r / 4) + 4 h + r % 4,
  // column ncol: scaled back by 2^xexp[m] (exact).  Y goes out through a
  // buffer whose range is M x N, so rows past M drop out of range and lanes
  // past N aim past it.  K pieces write their partial plane instead; the
  // reduction adds the bias.
  const __amdgpu_buffer_rsrc_t ers = prsrc(a.xexp, (uint32_t)a.M * 4u);
  float* dst = a.splits > 1 ? a.part + (size_t)z * a.M * a.N : a.y;
  const __amdgpu_buffer_rsrc_t yrs = prsrc(dst, a.y_bytes);
  const float bv = (nvalid && a.bias && a.splits == 1) ? a.bias[ncol] : 0.0f;
  // An output in fp32 over this piece, straight from the weights.
  auto from_weights = [&](int m) -> float {
    float v = 0.0f;
    const int k1 = min(a.K, s1 * kPStageK);
    const float* x = a.x + (size_t)m * a.K;
    if constexpr (kCol) {
      for (int k = s0 * kPStageK; k < k1; k++) {
        const size_t g = (size_t)k * (a.N / kBlockElems) + ncol / kBlockElems;
        if (g >= a.col_blocks) continue;
        const uint8_t* b = a.col + g * kBlockBytes;
        const float d = f16_bits_to_f32((uint32_t)b[0] | ((uint32_t)b[1] << 8));
        const int o = ncol % kBlockElems;
        const int q = (b[2 + o / 2] >> (4 * (o & 1))) & 15;
        v = fmaf((float)(q - 8), d * x[k], v);
      }
    } else {
      const uint16_t* w = reinterpret_cast<const uint16_t*>(a.wh) + (size_t)ncol * a.K;
      for (int k = s0 * kPStageK; k < k1; k++) v = fmaf(f16_bits_to_f32(w[k]), x[k], v);
    }
    return v;
  };
#pragma unroll
  for (int i = 0; i < MT; i++) {
    uint32_t ex[16];
    uint32_t again = 0;  // registers that are NaN
#pragma unroll
    for (int r = 0; r < 16; r++) {
      ex[r] = __builtin_amdgcn_raw_buffer_load_b32(
          ers, (uint32_t)(m0 + 32 * i + 8 * (r / 4) + 4 * h + r % 4) * 4u, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const uint32_t m = (uint32_t)(m0 + 32 * i + 8 * (r / 4) + 4 * h + r % 4);
      const bool nan = acc[i][r] != acc[i][r];
      if (nan) again |= 1u << r;
      const uint32_t off = nvalid && !nan ? (m * (uint32_t)a.N + (uint32_t)ncol) * 4u : 0xFFFFFFF0u;
      const float v = ldexpf(acc[i][r], (int)ex[r]) + bv;
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yrs, off, 0, 0);
    }
    if (again && nvalid) {
      for (int r = 0; r < 16; r++) {
        const int m = m0 + 32 * i + 8 * (r / 4) + 4 * h + r % 4;
        if (m < a.M && (again >> r & 1)) dst[(size_t)m * a.N + ncol] = from_weights(m) + bv;
      }
    }
  }
#endif
}

size_t rup(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Rows per tile and K pieces.  Costs (microseconds, fitted to 30 shapes at every
// number of pieces; the plans they choose measured 1.6% above the best on
// average, 11% at most): a 64-K stage 1.0 / 1.7 on 32- / 64-row tiles, a round of
// work-groups ~3 more; K pieces add the reduction launch (~2.5), 0.15 each and
// the planes' traffic (~3 TB/s a way).
struct PairPlan {
  int mt, splits;
};
PairPlan pair_plan(size_t n, size_t m, size_t batch, int num_cus) {
  const size_t tn = (n + kPBN - 1) / kPBN;
  const size_t steps = rup(m, kPStageK) / kPStageK;
  PairPlan best{1, 1};
  double best_cost = 1e300;
  for (int mt : {1, 2}) {
    if (mt > 1 && (size_t)16 * mt >= batch) break;  // taller tiles than the rows
    const size_t tiles = (batch + 32 * mt - 1) / (32 * mt) * tn;
    const double stage_us = mt == 2 ? 1.7 : 1.0;
    for (size_t sp = 1; sp <= std::min<size_t>(steps, 64); sp++) {
      const size_t rounds = (tiles * sp + num_cus - 1) / num_cus;
      double cost = (double)rounds * ((double)((steps + sp - 1) / sp) * stage_us + 3.0);
      if (sp > 1) cost += 2.5 + (double)sp * (0.15 + (double)(batch * n * 4) / 3.0e6);
      if (cost < best_cost * 0.999) {
        best_cost = cost;
        best = PairPlan{mt, (int)sp};
      }
      if (rounds > 1 && sp > 1) break;  // more pieces only add rounds
    }
  }
  return best;
}

bool pair_shape_ok(size_t n, size_t m, size_t batch) {
  const size_t lim = ((size_t)1 << 32) - 4096;
  return n <= 0x7FFFFFF && m <= 0x7FFFFFF && batch <= 0x7FFFFFF && n * m * 2 < lim &&
         (batch + 256) * rup(m, kPStageK) * 2 < lim && (batch + 256) * n * 4 < lim;
}

// (X is already converted at xws.)  wh: fp16 rows, or NULL and `col` the
// column-major blocks.
hipError_t launch_pair(float* y, const void* wh, const uint8_t* col, size_t col_len,
                       const float* x, const float* bias, size_t n, size_t m, size_t batch,
                       uint8_t* xws, int num_cus, hipStream_t s) {
  const PairPlan p = pair_plan(n, m, batch, num_cus);
  const size_t kp = rup(m, kPStageK);
  const int* xexp = x_split_exponents(xws, batch, m);
  hipError_t e;
  PairArgs a;
  a.col = col;
  a.col_blocks = col_len / kBlockBytes;
  a.col_bytes = (uint32_t)col_len;
  a.x = x;
  a.y = y;
  a.wh = static_cast<const uint8_t*>(wh);
  a.xh = xws;
  a.bias = bias;
  a.xexp = xexp;
  a.part = reinterpret_cast<float*>(xws + x_split_bytes(batch, m));
  a.w_bytes = (uint32_t)(n * m * 2);
  a.x_bytes = (uint32_t)(batch * kp * 2);
  a.y_bytes = (uint32_t)(batch * n * 4);
  a.M = (int)batch;
  a.N = (int)n;
  a.K = (int)m;
  a.steps = (int)(kp / kPStageK);
  a.tiles_m = (int)((batch + 32 * p.mt - 1) / (32 * p.mt));
  a.tiles_n = (int)((n + kPBN - 1) / kPBN);
  a.splits = p.splits;
  auto go = [&](auto kernel) -> hipError_t {
    const int rows = (kPParts * 32 * p.mt + 63) / 64 * 64;
    const int lds = kPRing * rows * kPRowBytes + (wh ? 0 : kPWaves * kTBytes);
    hipError_t le = set_lds_limit(reinterpret_cast<const void*>(kernel), lds);
    if (le != hipSuccess) return le;
    hipLaunchKernelGGL(kernel, dim3(a.tiles_m * a.tiles_n, p.splits), dim3(kPThreads), lds, s, a);
    return hipGetLastError();
  };
  if (!wh)
    e = p.mt == 2 ? go(gemm_pair_kernel<2, true>) : go(gemm_pair_kernel<1, true>);
  else
    e = p.mt == 2 ? go(gemm_pair_kernel<2, false>) : go(gemm_pair_kernel<1, false>);
  if (e != hipSuccess || p.splits == 1) return e;
  return launch_split_reduce(y, a.part, bias, batch * n, n, p.splits, s);
}

size_t pair_bytes(size_t n, size_t m, size_t batch, int num_cus) {
  const PairPlan p = pair_plan(n, m, batch, num_cus);
  return x_split_bytes(batch, m) + (p.splits > 1 ? (size_t)p.splits * batch * n * 4 : 0);
}

}  // namespace

// Whole block columns and 64-K stages, windows as the one-token kernel reads
// them (dword-aligned, the last block's 2 bytes of over-read inside the
// buffer), 32-bit offsets.
bool q4_0_col_gemm_ok(const uint8_t* w, size_t w_len, size_t n, size_t m, size_t batch) {
  if (n == 0 || m == 0 || n % kBlockElems != 0 || m % kBlockElems != 0 || batch == 0) return false;
  if (((uintptr_t)w & 3) != 0 || w_len >= 0xFFFFFF00u || !pair_shape_ok(n, m, batch)) return false;
  const size_t avail = w_len / kBlockBytes;
  return avail > 0 && (avail % 2 == 0 || w_len >= avail * kBlockBytes + 2);
}

size_t q4_0_col_gemm_workspace_bytes(size_t n, size_t m, size_t batch, int num_cus) {
  return pair_bytes(n, m, batch, num_cus);
}

hipError_t launch_q4_0_col_gemm(float* y, const uint8_t* w, size_t w_len, const float* x,
                                const float* bias, size_t n, size_t m, size_t batch, void* ws,
                                int num_cus, hipStream_t s) {
  uint8_t* xws = static_cast<uint8_t*>(ws);
  hipError_t e = launch_x_split(xws, x, batch, m, s);
  if (e != hipSuccess) return e;
  return launch_pair(y, nullptr, w, w_len, x, bias, n, m, batch, xws, num_cus, s);
}

// fp16 weights [n][m] as they are: K % 32 == 0, w 16-byte aligned.
bool f16_pair_gemm_ok(const uint8_t* w, size_t n, size_t m, size_t batch) {
  return n != 0 && m != 0 && m % 32 == 0 && batch != 0 && ((uintptr_t)w & 15) == 0 &&
         pair_shape_ok(n, m, batch);
}

size_t f16_pair_gemm_workspace_bytes(size_t n, size_t m, size_t batch, int num_cus) {
  return pair_bytes(n, m, batch, num_cus);
}

hipError_t launch_f16_pair_gemm(float* y, const uint8_t* w, const float* x, const float* bias,
                                size_t n, size_t m, size_t batch, void* ws, int num_cus,
                                hipStream_t s) {
  uint8_t* xws = static_cast<uint8_t*>(ws);
  hipError_t e = launch_x_split(xws, x, batch, m, s);
  if (e != hipSuccess) return e;
  return launch_pair(y, w, nullptr, 0, x, bias, n, m, batch, xws, num_cus, s);
}

}  // namespace hypno
