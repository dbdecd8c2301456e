// fp32-accurate batched GEMM on fp16 operand pairs, for gfx950:
// Y[M][N] = X[M][K] . W[N][K]^T (+ bias) with X = (xh + xl) 2^e per token and
// W = wh (fp16 weights) or wh + wl, and its users: column-major Q4_0 batches
// (kernels.rs:403-535, turbo.rs:322-326) and fp16 batches whose rows are no
// multiple of 64.
//
// Column-major Q4_0: W_col[k][j] keeps 32 outputs j of one input k in a
// block, so the scale d changes with k inside an output's sum and cannot be
// applied to partial sums.  Each weight becomes a pair in registers instead:
// wh = fp16(n d) rounded to nearest and wl = n d - wh, which fp16 holds exactly
// (a 4-bit integer times an 11-bit d leaves at most 4 units of d's last place,
// and that place is at least 2^-24).  The GEMM adds xh wh + xl wh + xh wl in
// fp32 on the matrix cores; what it leaves out, xl wl, is 2^-24 of a product.
//
// A wave's 32 columns are one block column, so its stage of 64 K is 64 blocks,
// one a lane; they change hands inside the wave through 1.4 KB of LDS (16 byte
// writes and 6 16-byte reads a lane, no barrier), and 10 VALU ops make four
// pairs: 80 a stage against 48 MFMAs of 128 tokens.  An expansion pass before
// the GEMM (4 bytes written and read back per weight) took as long as the
// products: 128 tokens, 5632 x 2048, 41 us a call with it, 28 without (one
// pass over the weights per token, the other way to do it: 412); 8 tokens,
// 14336 x 4096, 28 (52).
//
// What bounds it: three MFMAs per product beside the pairs' VALU and LDS work
// on one issue port, and at few tokens the three launches of a call.
//
//  * Work-group = 8 waves on a 32 MT x 256 tile of Y, 32 columns a wave;
//    32x32x16 MFMAs.  fp16 weights: lane (n, h) loads the 64 bytes of its
//    column and lane half straight into registers, one stage of 64 K ahead;
//    column-major blocks are loaded three stages ahead.
//  * X: hi rows then lo rows by DMA into a ring of four LDS stages, 16-byte
//    chunk c of row r in slot c ^ ((r >> 1) & 7) (16 rows of an operand read
//    hit distinct banks); one barrier per stage publishes the stage two ahead.
#include <algorithm>

#include "common.hpp"

namespace hypno {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kPWaves = 8;
constexpr int kPThreads = 64 * kPWaves;
constexpr int kPBN = 32 * kPWaves;
constexpr int kPStageK = 64;
constexpr int kPRowBytes = kPStageK * 2;
constexpr int kPRing = 4;
// A wave's 64 column-major blocks in LDS: byte i of block k at i * kTPitch + k
// (16 rows whose 16-byte reads hit distinct banks), then the 64 scales.
[[maybe_unused]] constexpr int kTPitch = 80;
constexpr int kTBytes = 16 * kTPitch + 128;
[[maybe_unused]] constexpr uint32_t kBigScale = 0x6FFF;  // fp16 bits of 8188: 8 * 8188 is fp16's largest value
[[maybe_unused]] constexpr uint32_t kNotFinite = 0x80000000u;  // exponent of a token holding inf or NaN

struct PairArgs {
  float* y;
  const uint8_t* wh;   // fp16 [N][K] (not column-major)
  const uint8_t* xh;   // fp16 [M][Kp] hi parts, then a plane of M rows of lo parts
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
  constexpr int kTile = 2 * BM * kPRowBytes;
  constexpr int kDx = 2 * BM / 64;          // X DMAs per wave and stage
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
  // slot (rows BM .. 2 BM - 1 are the lo parts).
  const uint32_t x_row = (uint32_t)a.steps * kPRowBytes;
  const __amdgpu_buffer_rsrc_t xrs = prsrc(a.xh, a.x_bytes);
  const __amdgpu_buffer_rsrc_t xls = prsrc(a.xh + a.x_bytes, a.x_bytes);
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
      const bool lo = 8 * (8 * i + wave) >= BM;  // wave-uniform
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          lo ? xls : xrs,
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
    u32x4 h[4], l[4];
  };
  auto load_w = [&](int s) __attribute__((always_inline)) -> Wreg {
    const int sc = s0 + (s < steps ? s : steps - 1);
    const uint32_t v = sc * kPStageK + 32 * h < a.K ? wvoff : 0xFFFFFF00u;
    const uint32_t off = v == 0xFFFFFF00u ? v : v + (uint32_t)sc * kPRowBytes;
    Wreg r;
#pragma unroll
    for (int j = 0; j < 4; j++) r.h[j] = __builtin_amdgcn_raw_buffer_load_b128(whs, off + 16 * j, 0, 0);
    return r;
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
  uint32_t dmax = 0;  // largest |d| of this lane's blocks, as bits
  auto expand = [&](const Raw& r) __attribute__((always_inline)) -> Wreg {
    const uint32_t sel = r.odd & 2u ? 0x07060504u : 0x05040302u;
    const uint32_t v[5] = {r.v[0], r.v[1], r.v[2], r.v[3], r.v4};
    const uint32_t d = r.odd & 2u ? v[0] >> 16 : r.odd ? 0u : v[0] & 0xFFFFu;
    dmax = max(dmax, d & 0x7FFFu);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t q = __builtin_amdgcn_perm(v[j + 1], v[j], sel);
#pragma unroll
      for (int b = 0; b < 4; b++) tb[(4 * j + b) * kTPitch + lane] = (uint8_t)(q >> (8 * b));
    }
    *reinterpret_cast<uint16_t*>(tb + 16 * kTPitch + 2 * lane) = (uint16_t)d;
    // (LDS keeps a wave's accesses in order: these reads follow the writes,
    // and the next stage's writes follow them)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    u32x4 qb[2], db[4];
#pragma unroll
    for (int j = 0; j < 2; j++)
      qb[j] = *reinterpret_cast<const u32x4*>(tb + (lr >> 1) * kTPitch + 32 * h + 16 * j);
#pragma unroll
    for (int j = 0; j < 4; j++)
      db[j] = *reinterpret_cast<const u32x4*>(tb + 16 * kTPitch + 64 * h + 16 * j);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int sh = 4 * (lr & 1);
    const half2v off = {(_Float16)-1032.0f, (_Float16)-1032.0f};
    Wreg w;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) {  // elements 8 j + 2 i, + 1
        const uint32_t n4 = (qb[j >> 1][2 * (j & 1) + (i >> 1)] >> sh) & 0x0F0F0F0Fu;
        const uint32_t u = __builtin_amdgcn_perm(0x64646464u, n4, i & 1 ? 0x04030402u : 0x04010400u);
        const uint32_t db2 = db[j][i];
        const half2v n = __builtin_bit_cast(half2v, u) + off, dd = __builtin_bit_cast(half2v, db2);
        const half2v hi = n * dd;
        w.h[j][i] = __builtin_bit_cast(uint32_t, hi);
        w.l[j][i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(n, dd, -hi));
      }
    return w;
  };

  uint32_t aoff[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    aoff[j] = (uint32_t)lr * kPRowBytes + (((4 * h + j) ^ ((lr >> 1) & 7)) << 4);
  auto read_a = [&](int s, int i, int p, int j) __attribute__((always_inline)) -> half8 {
    return *reinterpret_cast<const half8*>(smem + (s % kPRing) * kTile + aoff[j] +
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
  if constexpr (kCol) {
    r1 = load_col(0);
    r2 = load_col(1);
  } else {
    wa = load_w(0);
  }
  asm volatile("" ::: "memory");
  for (int i = 0; i < kPRing - 1; i++) issue_x(i);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kDx) : "memory");
  if constexpr (kCol) {
    wa = expand(r1);
    r1 = r2;
    r2 = load_col(2);
  }
  half8 fa[2][4];  // hi and lo operands of the next row tile
#pragma unroll
  for (int p = 0; p < 2; p++)
#pragma unroll
    for (int j = 0; j < 4; j++) fa[p][j] = read_a(0, 0, p, j);

  floatx16 prev;  // the previous tile's stage sum
#pragma unroll
  for (int r = 0; r < 16; r++) prev[r] = 0.0f;

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
      wn = load_w(s + 1);
    }
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const int ns = i + 1 == MT ? s + 1 : s, ni = (i + 1) % MT;
      // The stage's products add up from zero and then to the tile's sum, so
      // that sum is rounded once per 64 columns; the lo products go first,
      // so the roundings at the stage sum's own size are four, not twelve.
      floatx16 p;
#pragma unroll
      for (int r = 0; r < 16; r++) p[r] = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if constexpr (kCol)
          p = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[0][j], __builtin_bit_cast(half8, w.l[j]),
                                                     p, 0, 0, 0);
        p = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[1][j], __builtin_bit_cast(half8, w.h[j]), p,
                                                   0, 0, 0);
        fa[1][j] = read_a(ns, ni, 1, j);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        p = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[0][j], __builtin_bit_cast(half8, w.h[j]), p,
                                                   0, 0, 0);
        fa[0][j] = read_a(ns, ni, 0, j);
      }
      const int pi = (i + MT - 1) % MT;
#pragma unroll
      for (int r = 0; r < 16; r++) acc[pi][r] += prev[r];
      prev = p;
      __builtin_amdgcn_sched_barrier(0);
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
  for (int r = 0; r < 16; r++) acc[MT - 1][r] += prev[r];
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
  // An output straight from the blocks, in fp32 over this piece: where a
  // product n d of the wave's blocks leaves fp16 (big) or a token holds inf or NaN (its exponent
  // says so), whose products with a zero wl would all be NaN.
  auto from_blocks = [&](int m) -> float {
    float v = 0.0f;
    const int k1 = min(a.K, s1 * kPStageK);
    for (int k = s0 * kPStageK; k < k1; k++) {
      const size_t g = (size_t)k * (a.N / kBlockElems) + ncol / kBlockElems;
      if (g >= a.col_blocks) continue;
      const uint8_t* b = a.col + g * kBlockBytes;
      const float d = f16_bits_to_f32((uint32_t)b[0] | ((uint32_t)b[1] << 8));
      const int o = ncol % kBlockElems;
      const int q = (b[2 + o / 2] >> (4 * (o & 1))) & 15;
      v = fmaf((float)(q - 8), d * a.x[(size_t)m * a.K + k], v);
    }
    return v;
  };
  // The same from fp16 rows: where the pairs' sum is NaN, which an infinity (in
  // the weights or the token) makes of finite neighbours (inf times a zero or
  // an opposite lo part).
  auto from_rows = [&](int m) -> float {
    float v = 0.0f;
    const int k1 = min(a.K, s1 * kPStageK);
    const uint16_t* w = reinterpret_cast<const uint16_t*>(a.wh) + (size_t)ncol * a.K;
    for (int k = s0 * kPStageK; k < k1; k++)
      v = fmaf(f16_bits_to_f32(w[k]), a.x[(size_t)m * a.K + k], v);
    return v;
  };
  const bool big = kCol && __any(dmax > kBigScale);
#pragma unroll
  for (int i = 0; i < MT; i++) {
    uint32_t ex[16];
    uint32_t redo = big ? 0xFFFFu : 0u;  // registers to compute from the source
#pragma unroll
    for (int r = 0; r < 16; r++) {
      ex[r] = __builtin_amdgcn_raw_buffer_load_b32(
          ers, (uint32_t)(m0 + 32 * i + 8 * (r / 4) + 4 * h + r % 4) * 4u, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const uint32_t m = (uint32_t)(m0 + 32 * i + 8 * (r / 4) + 4 * h + r % 4);
      const uint32_t off = nvalid ? (m * (uint32_t)a.N + (uint32_t)ncol) * 4u : 0xFFFFFFF0u;
      if (kCol ? ex[r] == kNotFinite : acc[i][r] != acc[i][r]) redo |= 1u << r;
      const float v = ldexpf(acc[i][r], (int)ex[r]) + bv;
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yrs, off, 0, 0);
    }
    if (redo && nvalid) {
      for (int r = 0; r < 16; r++) {
        const int m = m0 + 32 * i + 8 * (r / 4) + 4 * h + r % 4;
        if (m < a.M && (redo >> r & 1))
          dst[(size_t)m * a.N + ncol] = (kCol ? from_blocks(m) : from_rows(m)) + bv;
      }
    }
  }
#endif
}

size_t rup(size_t v, size_t a) { return (v + a - 1) / a * a; }

size_t pair_x_bytes(size_t batch, size_t m) {
  return rup(2 * batch * rup(m, kPStageK) * 2, 256) + rup(batch * 4, 256);
}

// Rows per tile and K pieces.  Costs (microseconds): a 64-K stage 0.8 / 1.0 /
// 1.5 on 32- / 64- / 128-row tiles of fp16 weights, 0.83 / 1.2 / 2.25 of
// column-major blocks (128 tokens, 2048 x 5632, whole K: 86 / 126 / 213 us a
// call), a round of work-groups ~3 more, the reduction of K pieces its launch
// (~2.5) and the planes' traffic (~4, column-major ~3 TB/s).
struct PairPlan {
  int mt, splits;
};
PairPlan pair_plan(bool col, size_t n, size_t m, size_t batch, int num_cus) {
  const size_t tn = (n + kPBN - 1) / kPBN;
  const size_t steps = rup(m, kPStageK) / kPStageK;
  PairPlan best{1, 1};
  double best_cost = 1e300;
  for (int mt : {1, 2, 4}) {
    if (mt > 1 && (size_t)16 * mt >= batch) break;  // taller tiles than the rows
    const size_t tiles = (batch + 32 * mt - 1) / (32 * mt) * tn;
    const double stage_us = mt == 4 ? (col ? 2.25 : 1.5) : mt == 2 ? (col ? 1.2 : 1.0)
                                                                   : (col ? 0.83 : 0.8);
    for (size_t sp = 1; sp <= std::min<size_t>(steps, 64); sp++) {
      const size_t rounds = (tiles * sp + num_cus - 1) / num_cus;
      double cost = (double)rounds * ((double)((steps + sp - 1) / sp) * stage_us + 3.0);
      if (sp > 1) cost += 2.5 + (double)sp * (double)(batch * n * 4) / (col ? 3.0e6 : 4.0e6);
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

int* pair_exponents(uint8_t* xws, size_t batch, size_t m) {
  return reinterpret_cast<int*>(xws + rup(2 * batch * rup(m, kPStageK) * 2, 256));
}

// (X is already converted at xws.)  wh: fp16 rows, or NULL and `col` the
// column-major blocks.
hipError_t launch_pair(float* y, const void* wh, const uint8_t* col, size_t col_len,
                       const float* x, const float* bias, size_t n, size_t m, size_t batch,
                       uint8_t* xws, int num_cus, hipStream_t s) {
  const PairPlan p = pair_plan(!wh, n, m, batch, num_cus);
  const size_t kp = rup(m, kPStageK);
  const int* xexp = pair_exponents(xws, batch, m);
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
  a.part = reinterpret_cast<float*>(xws + pair_x_bytes(batch, m));
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
    const int lds = kPRing * 2 * 32 * p.mt * kPRowBytes + (wh ? 0 : kPWaves * kTBytes);
    hipError_t le = set_lds_limit(reinterpret_cast<const void*>(kernel), lds);
    if (le != hipSuccess) return le;
    hipLaunchKernelGGL(kernel, dim3(a.tiles_m * a.tiles_n, p.splits), dim3(kPThreads), lds, s, a);
    return hipGetLastError();
  };
  if (!wh)
    e = p.mt == 4   ? go(gemm_pair_kernel<4, true>)
        : p.mt == 2 ? go(gemm_pair_kernel<2, true>)
                    : go(gemm_pair_kernel<1, true>);
  else
    e = p.mt == 4   ? go(gemm_pair_kernel<4, false>)
        : p.mt == 2 ? go(gemm_pair_kernel<2, false>)
                    : go(gemm_pair_kernel<1, false>);
  if (e != hipSuccess || p.splits == 1) return e;
  return launch_split_reduce(y, a.part, bias, batch * n, n, p.splits, s);
}

size_t pair_bytes(bool col, size_t n, size_t m, size_t batch, int num_cus) {
  const PairPlan p = pair_plan(col, n, m, batch, num_cus);
  return pair_x_bytes(batch, m) + (p.splits > 1 ? (size_t)p.splits * batch * n * 4 : 0);
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
  return 256 + pair_bytes(true, n, m, batch, num_cus);
}

hipError_t launch_q4_0_col_gemm(float* y, const uint8_t* w, size_t w_len, const float* x,
                                const float* bias, size_t n, size_t m, size_t batch, void* ws,
                                int num_cus, hipStream_t s) {
  // (the exponent of a token holding inf or NaN says so where a word to clear
  // is given; nothing else uses that word)
  uint8_t* xws = static_cast<uint8_t*>(ws) + 256;
  hipError_t e = launch_x_hilo(xws, pair_exponents(xws, batch, m), x, batch, m,
                               rup(m, kPStageK), static_cast<uint32_t*>(ws), s);
  if (e != hipSuccess) return e;
  return launch_pair(y, nullptr, w, w_len, x, bias, n, m, batch, xws, num_cus, s);
}

// fp16 weights [n][m] as they are: K % 32 == 0, w 16-byte aligned.
bool f16_pair_gemm_ok(const uint8_t* w, size_t n, size_t m, size_t batch) {
  return n != 0 && m != 0 && m % 32 == 0 && batch != 0 && ((uintptr_t)w & 15) == 0 &&
         pair_shape_ok(n, m, batch);
}

size_t f16_pair_gemm_workspace_bytes(size_t n, size_t m, size_t batch, int num_cus) {
  return pair_bytes(false, n, m, batch, num_cus);
}

hipError_t launch_f16_pair_gemm(float* y, const uint8_t* w, const float* x, const float* bias,
                                size_t n, size_t m, size_t batch, void* ws, int num_cus,
                                hipStream_t s) {
  uint8_t* xws = static_cast<uint8_t*>(ws);
  hipError_t e = launch_x_hilo(xws, pair_exponents(xws, batch, m), x, batch, m,
                               rup(m, kPStageK), nullptr, s);
  if (e != hipSuccess) return e;
  return launch_pair(y, w, nullptr, 0, x, bias, n, m, batch, xws, num_cus, s);
}

}  // namespace hypno
