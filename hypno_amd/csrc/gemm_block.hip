// Batched GEMM on block-quantised weights, accurate to fp32, for gfx950:
// Y[M][N] = X[M][K] . W[N][K]^T (+ bias), W in hypno's Q4_0 or Q8_0 blocks
// (quant.rs:10-22, :74-103), any K % 32 == 0.  It serves the batches that the
// tuned kernels do not take (rows that are no multiple of their stages), for
// which the alternative is one fp32 dot product per token and row.
//
// Arithmetic: the integer weights (nibble - 8, or byte - 128) go to the
// matrix cores as exact bf16 values.  Each token is three bf16 rows that hold
// all 24 bits of x (x 2^s = x1 + x2 + x3, each the next 8 bits; s a power of
// two per token that keeps every sum in range, undone exactly on output),
// whose products with a block, all exact, add up smallest first in one partial
// P (K = 32: six chained v_mfma_f32_32x32x16_bf16 from a zeroed accumulator);
// the block's d scales it in fp32, acc += d * P.
//
// What bounds it: the 16 scale FMAs per 32 x 32 output tile and block share
// the SIMD's issue port with the MFMAs, and every wave reads the whole X tile
// from LDS.  The 32x32x16 form issues half as many MFMAs per product as
// 16x16x32 and an A operand feeds 32 columns.  Measured: 333 tokens, N 2880,
// K 7200 (225 blocks a row): 74-81 us per call where the fp32 dot products took
// 14.5 ms, error against 64 bits 1.4e-7 (1.9e-7).  With two fp16 parts in place
// of three bf16 ones (60 us) x keeps 22 bits, fewer beside an outlier.
//
//  * Work-group = 8 waves (two per SIMD) on a 32 MT x 256 tile of Y; wave w
//    owns output columns 32 w .. 32 w + 31 for all 32 MT rows.  Its weights
//    reach its own LDS ring by DMA (4 bytes per lane; only the wave's own
//    load counter orders that ring) and are unpacked in registers, once per
//    block for MT tiles of rows.
//  * X: 16-bit rows by DMA into a ring of kRing stages of 64 K shared by the
//    waves, 16-byte chunk c of row r in slot c ^ ((r >> 1) & 7) (16 rows of
//    an operand read hit distinct banks).  One barrier per stage: it
//    publishes the stage two ahead.
//  * A stage is 2 MT slots (block 0 of every row tile, then block 1); slot j
//    issues its MFMAs, the reloads of the A registers they free for slot
//    j + 2, the 16 scale FMAs of slot j - 1 and a share of the next block's
//    unpack, in that order (a scheduling barrier between slots).
//  * One part: x rounded once to fp16 (the prefill GEMMs' arithmetic) takes
//    the same kernel on fp16 operands, a third of the MFMAs and of the LDS per
//    row, so tiles go up to 256 rows.  Per 256 x 256 x 64 stage 2.3 us with
//    every CU at work (930 TFLOP/s); copies without X and W DMA 13% faster,
//    without the barrier 4%, without the A reads no faster: what is left is
//    the MFMAs and FMAs of two waves on one issue port (a probe of 32x32x16
//    MFMAs with 8 FMAs each reaches 1560 TFLOP/s, with 10 ops 1460).
//  * K % 64 == 32: the X rows are padded with a zero block, and the scale of
//    the block past the row's end is taken as 0.  Rows of an odd number of
//    blocks start on 2-byte boundaries: each row's window then starts at the
//    dword below it and a lane's selectors depend on its row's parity (kOdd).
#include <algorithm>

#include "common.hpp"

namespace hypno {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kBWaves = 8;
constexpr int kBThreads = 64 * kBWaves;
constexpr int kBN = 32 * kBWaves;  // 256 output columns per work-group
constexpr int kBStageK = 64;       // two blocks per stage
constexpr int kBRowBytes = kBStageK * 2;

// FMT: weight format; MT: 32-row tiles per wave; ODD: an odd number of blocks
// per row.
template <int FMT, int MT, bool ODD, int PARTS = 3>
struct BlockGeom {
  static constexpr int kBlk = FMT == kFmtQ8_0 ? kQ8BlockBytes : kBlockBytes;
  static constexpr int kRowDw = 2 * kBlk / 4 + (ODD ? 1 : 0);  // a row's dwords per stage
  static constexpr int kDw = (32 * kRowDw + 63) / 64;          // W DMAs per wave and stage
  static constexpr int kWSlot = 256 * kDw;
  // X rows of the tile, part by part (padded to whole DMAs of every wave)
  static constexpr int kXRows = (32 * PARTS * MT + 63) / 64 * 64;
  static constexpr int kTile = kXRows * kBRowBytes;
  static constexpr int kDx = kXRows / 64;  // X DMAs per wave and stage
  static constexpr int kFree = 160 * 1024;
  static constexpr int kRing = kTile >= 24576 ? 3 : 4;
  static constexpr int kFit = (kFree - kRing * kTile) / (kBWaves * kWSlot);
  static constexpr int kMost = FMT == kFmtQ8_0 ? 4 : 6;  // (vmcnt counts to 63)
  static constexpr int kWRing = kFit > kMost ? kMost : kFit;
  static constexpr int kLds = kRing * kTile + kBWaves * kWRing * kWSlot;
  // The wait at the end of stage s leaves outstanding what went out after
  // X(s+2): the W DMAs of its stage and R-3 whole stages.
  static constexpr int kStageWait = kDw + (kRing - 3) * (kDx + kDw);
  static_assert(kWRing >= kRing && kWRing >= 3, "W(s+2) is older than X(s+2)");
  static_assert(kStageWait <= kDw * (kWRing - 3) + kDx + kDw, "W(2) landed in stage 0");
  static_assert((kRing - 1) * kDx + kWRing * kDw + kDx + kDw < 64, "vmcnt");
};

struct BlockArgs {
  float* y;
  const uint8_t* w;
  const uint8_t* xh;  // 16-bit [M][Kp], a plane of M rows per part
  const float* bias;
  const int* xexp;    // [M]: row m of xh holds X row m times 2^-xexp[m]
  float* part;        // [splits][M][N] partial planes (splits > 1)
  uint32_t w_bytes;   // W bytes (buffer range)
  uint32_t x_bytes;   // bytes of one xh plane (rows past M read zeros)
  uint32_t y_bytes;   // M x N x 4: the range of Y and of each partial plane
  int M, N, B;        // B: blocks per row
  int steps;          // 64-K stages of a row
  int tiles_m, tiles_n;
  int xcd_map;
  int splits;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t brsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           0x00020000);
}

// The matrix product of one operand pair: fp16 where x is rounded to one part,
// bf16 where it is three.
template <int PARTS>
__device__ __forceinline__ floatx16 block_mfma(u32x4 a, u32x4 b, floatx16 c) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (PARTS == 1)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a),
                                                  __builtin_bit_cast(half8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
#else
  return c;
#endif
}

// Eight packed integers -> eight exact bf16 values in order.  Q4_0: (nibble -
// 8) / 16, what v_cvt_off_f32_i4 makes of a nibble with its top bit flipped;
// the caller's scale carries the 16.  Q8_0: byte - 128.
__device__ __forceinline__ u32x4 unpack8_bf16(uint32_t q) {
  const uint32_t lo = q ^ 0x88888888u, hi = lo >> 4;
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t a = __float_as_uint(__builtin_amdgcn_cvt_off_f32_i4(lo >> (8 * i)));
    const uint32_t b = __float_as_uint(__builtin_amdgcn_cvt_off_f32_i4(hi >> (8 * i)));
    r[i] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  }
  return r;
}
__device__ __forceinline__ u32x4 unpack8_bytes_bf16(uint32_t lo, uint32_t hi) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t s = (i < 2 ? lo : hi) ^ 0x80808080u;
    const uint32_t a = __float_as_uint((float)(int8_t)(s >> (16 * (i & 1))));
    const uint32_t b = __float_as_uint((float)(int8_t)(s >> (16 * (i & 1) + 8)));
    r[i] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  }
  return r;
}

// One lane's weights of a block: the integers its two B operands hold (lane
// half h takes elements 16 h + 8 j .. + 7 for MFMA j), packed, and the scale
// bits.
template <int FMT>
struct RawBlock {
  uint32_t q[FMT == kFmtQ8_0 ? 4 : 2];
  uint32_t d;
};

template <int FMT, int MT, bool ODD, int PARTS>
__global__ void __launch_bounds__(kBThreads, 1) gemm_block_kernel(const BlockArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the buffer builtins exist only in the device pass)
  using G = BlockGeom<FMT, MT, ODD, PARTS>;
  constexpr int BM = 32 * MT;
  constexpr int kRing = G::kRing, kWRing = G::kWRing;
  constexpr int kParts = PARTS;  // x1, x2, x3; or the rounded x alone
  extern __shared__ __align__(16) uint8_t smem[];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 31;
  const int h = lane >> 5;

  // Tile of this work-group; with xcd_map the 8 XCDs (work-groups go round
  // robin over them) each get a contiguous range of tiles in (n-tile,
  // m-tile) order, so the m-tiles sharing W rows share an L2.
  int tile = blockIdx.x;
  const int ntiles = a.tiles_m * a.tiles_n;
  if (a.xcd_map) tile = (tile & 7) * (ntiles >> 3) + (tile >> 3);
  const int m0 = (tile % a.tiles_m) * BM;
  const int n0 = (tile / a.tiles_m) * kBN;
  // K range of this piece: stages [s0, s0 + steps).
  const int z = blockIdx.y;
  const int s0 = (int)((long long)a.steps * z / a.splits);
  const int s1 = (int)((long long)a.steps * (z + 1) / a.splits);
  const int steps = s1 - s0;

  // --- X DMA: instruction i of wave w fills LDS rows 8 (8 i + w) .. + 7 of
  // the slot (part p in rows BM p .. BM p + BM - 1); lane -> row
  // 8 (8 i + w) + (lane >> 3), slot chunk lane & 7, which holds logical chunk
  // (lane & 7) ^ ((row >> 1) & 7).
  const uint32_t x_row = (uint32_t)a.steps * kBRowBytes;
  uint32_t xvoff[G::kDx];
#pragma unroll
  for (int i = 0; i < G::kDx; i++) {
    const int row = 8 * (8 * i + wave) + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    // (a whole DMA lies in one part: BM is a multiple of its 8 rows)
    xvoff[i] = (uint32_t)(m0 + row % BM) * x_row + (uint32_t)c * 16u;
  }
  auto issue_x = [&](int s) __attribute__((always_inline)) {  // stage min(s, steps-1) -> slot of s
    const int sc = s < steps ? s : steps - 1;
    const int soff = (s0 + sc) * kBRowBytes;
    uint8_t* slot = smem + (s % kRing) * G::kTile;
#pragma unroll
    for (int i = 0; i < G::kDx; i++) {
      // (wave-uniform; rows that only fill up the last DMA read the last part again)
      const int part = min(8 * (8 * i + wave) / BM, PARTS - 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          brsrc(a.xh + (size_t)part * a.x_bytes, a.x_bytes),
          (__attribute__((address_space(3))) void*)(slot + 8 * (8 * i + wave) * kBRowBytes), 16,
          xvoff[i], soff, 0, 0);
    }
  };

  // --- W: each wave DMAs its own 32 rows' stage windows (kRowDw dwords from
  // the dword at or below the row's stage start) into its own ring and reads
  // them back per lane; rows past N re-read row N - 1.  A window dword past
  // the buffer reads 0.
  const int ncol = n0 + 32 * wave + lr;
  const bool nvalid = ncol < a.N;
  const __amdgpu_buffer_rsrc_t wrs = brsrc(a.w, a.w_bytes);
  const uint32_t w_row = (uint32_t)a.B * G::kBlk;
  uint32_t wvoff[G::kDw];
#pragma unroll
  for (int i = 0; i < G::kDw; i++) {
    const int l = min(64 * i + lane, 32 * G::kRowDw - 1);
    const int r = l / G::kRowDw, c = l % G::kRowDw;
    const uint32_t start = (uint32_t)min(n0 + 32 * wave + r, a.N - 1) * w_row;
    wvoff[i] = (start & ~3u) + 4u * (uint32_t)c;
  }
  const bool hi2 = ODD && (((uint32_t)min(ncol, a.N - 1) * w_row) & 2u) != 0;
  uint8_t* const wring = smem + kRing * G::kTile + wave * kWRing * G::kWSlot;
  auto issue_w = [&](int s) __attribute__((always_inline)) {
    const int sc = s < steps ? s : steps - 1;
    const int soff = (s0 + sc) * 2 * G::kBlk;
    uint8_t* slot = wring + (s % kWRing) * G::kWSlot;
#pragma unroll
    for (int i = 0; i < G::kDw; i++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          wrs, (__attribute__((address_space(3))) void*)(slot + 256 * i), 4, wvoff[i], soff, 0, 0);
  };
  // Block kb of stage s (its first byte is at window byte kb * kBlk, 2 more
  // for a row that starts 2 bytes past its window): raw window dwords, and
  // what they hold.  The integers of lane half h start 2 + (kQ h) bytes in.
  constexpr int kQ = FMT == kFmtQ8_0 ? 16 : 8;  // integer bytes per lane half
  constexpr int kQd = kQ / 4;
  struct Win {
    uint32_t v[kQd + 1];
    uint32_t d;
  };
  // Without ODD block 0's integers sit at 2 mod 4 and block 1's (36/18 and
  // 68/34: kBlk + 2 is a multiple of 4) at 0 mod 4; a row that starts 2 bytes
  // past its window swaps the two cases.
  auto read_win = [&](int s, int kb) __attribute__((always_inline)) -> Win {
    const uint32_t* p = reinterpret_cast<const uint32_t*>(wring + (s % kWRing) * G::kWSlot) +
                        lr * G::kRowDw;
    const int q0 = (kb * G::kBlk + 2) / 4;  // dword of the first integer byte (even rows)
    const int d0 = (kb * G::kBlk) / 4;
    Win r;
    if constexpr (ODD) {
      const uint32_t* pq = p + q0 + kQd * h + (kb == 0 && hi2 ? 1 : 0);
#pragma unroll
      for (int i = 0; i <= kQd; i++) r.v[i] = pq[i];
      r.d = p[d0 + (kb == 1 && hi2 ? 1 : 0)];
    } else {
#pragma unroll
      for (int i = 0; i <= kQd; i++) r.v[i] = (i < kQd || kb == 0) ? p[q0 + kQd * h + i] : 0u;
      r.d = p[d0];
    }
    return r;
  };
  // (sel: bytes 2..5 of a dword pair, or 0..3)
  auto take = [&](const Win& w, int kb, RawBlock<FMT>& o) __attribute__((always_inline)) {
    if constexpr (ODD) {
      const bool mis = (kb == 0) != hi2;  // integers at 2 mod 4
      const uint32_t sel = mis ? 0x05040302u : 0x03020100u;
#pragma unroll
      for (int i = 0; i < kQd; i++) o.q[i] = __builtin_amdgcn_perm(w.v[i + 1], w.v[i], sel);
      o.d = (kb == 0) != hi2 ? w.d & 0xFFFFu : w.d >> 16;
    } else {
#pragma unroll
      for (int i = 0; i < kQd; i++)
        o.q[i] = kb == 0 ? __builtin_amdgcn_perm(w.v[i + 1], w.v[i], 0x05040302u) : w.v[i];
      o.d = kb == 0 ? w.d & 0xFFFFu : w.d >> 16;
    }
  };
  auto unpack = [&](const RawBlock<FMT>& o, int j) __attribute__((always_inline)) -> u32x4 {
    if constexpr (FMT == kFmtQ8_0)
      return PARTS == 1 ? unpack8_bytes(o.q[2 * j], o.q[2 * j + 1])
                        : unpack8_bytes_bf16(o.q[2 * j], o.q[2 * j + 1]);
    else
      return PARTS == 1 ? unpack8(o.q[j]) : unpack8_bf16(o.q[j]);
  };
  // A block past the row's end (K % 64 == 32, block 1 of the last stage)
  // multiplies X's zero padding; its scale bits are not the row's: take 0.
  auto scale_of = [&](const RawBlock<FMT>& o, int s, int kb) __attribute__((always_inline)) {
    const bool ok = nvalid && (!ODD || kb == 0 || 2 * (s0 + s) + 1 < a.B);
    const float unit = FMT == kFmtQ4_0 && PARTS == 3 ? 16.0f : 1.0f;
    return ok ? f16_bits_to_f32(o.d) * unit : 0.0f;
  };

  // --- A operands: part p, block kb, MFMA j, row tile i: row
  // 32 i + lr (+ BM p), logical chunk 4 kb + 2 h + j.
  uint32_t aoff[2][2];
#pragma unroll
  for (int kb = 0; kb < 2; kb++)
#pragma unroll
    for (int j = 0; j < 2; j++)
      aoff[kb][j] = (uint32_t)lr * kBRowBytes + (((4 * kb + 2 * h + j) ^ ((lr >> 1) & 7)) << 4);
  auto read_a = [&](int s, int kb, int i, int p, int j) __attribute__((always_inline)) -> u32x4 {
    return *reinterpret_cast<const u32x4*>(smem + (s % kRing) * G::kTile + aoff[kb][j] +
                                           (32 * i + BM * p) * kBRowBytes);
  };

  floatx16 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;
  // Three parts: the sum moves to `tot` every kGroup stages, so no output is a
  // chain of one rounding per block (1000 tokens, K 2848 in one piece: rel-L2
  // 1.8e-7 as one chain, 1.0e-7 so, 1.4e-7 the fp32 dot products).
  constexpr int kGroup = 8;
  constexpr int kTot = PARTS == 3 ? MT : 1;
  floatx16 tot[kTot];
  if constexpr (PARTS == 3) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) tot[i][r] = 0.0f;
  }

  // Prologue: X of stages 0..R-2 and W of stages 0..P-1 in flight; X and W of
  // stages 0 and 1 landed and published; the A operands of slots 0 and 1 and
  // block 0 of stage 0 unpacked.
  for (int i = 0; i < kRing - 1; i++) issue_x(i);
  for (int i = 0; i < kWRing; i++) issue_w(i);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(G::kDw * (kWRing - 2)) : "memory");
  constexpr int kSlots = 2 * MT;
  u32x4 fa[2][kParts][2];  // slot j's operands: fa[j & 1]
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int p = 0; p < kParts; p++)
#pragma unroll
      for (int k = 0; k < 2; k++) fa[j][p][k] = read_a(0, j / MT, j % MT, p, k);
  u32x4 fb[2];
  float d;
  Win wodd = read_win(0, 1);
  {
    RawBlock<FMT> o;
    take(read_win(0, 0), 0, o);
    fb[0] = unpack(o, 0);
    fb[1] = unpack(o, 1);
    d = scale_of(o, 0, 0);
  }
  floatx16 prev;  // the previous slot's partial, its scale and row tile
  float dprev = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; r++) prev[r] = 0.0f;

  for (int s = 0; s < steps; s++) {
    const Win weven = read_win(s + 1, 0);
    Win wodd_next = wodd;
    u32x4 nb[2];
    float nd = 0.0f;
    RawBlock<FMT> raw;
#pragma unroll
    for (int j = 0; j < kSlots; j++) {
      const int kb = j / MT, i = j % MT;
      if (j == 1) {
        // Every wave is past the barrier that ended stage s - 1, so the X
        // slot of s - 1 is free; so is the W slot of s: its words are in this
        // wave's registers (slot 0 used the last of them).
        issue_x(s + kRing - 1);
        asm volatile("" ::: "memory");  // X DMAs before W DMAs (the wait counts on it)
        issue_w(s + kWRing);
      }
      floatx16 p;
#pragma unroll
      for (int r = 0; r < 16; r++) p[r] = 0.0f;
#pragma unroll
      for (int q = kParts - 1; q >= 0; q--)  // the smallest parts first
#pragma unroll
        for (int k = 0; k < 2; k++) p = block_mfma<PARTS>(fa[j & 1][q][k], fb[k], p);
      // operands of slot j + 2
      {
        const int nj = j + 2;
        const int ns = nj >= kSlots ? s + 1 : s;
        const int nk = nj % kSlots;
#pragma unroll
        for (int q = 0; q < kParts; q++)
#pragma unroll
          for (int k = 0; k < 2; k++) fa[j & 1][q][k] = read_a(ns, nk / MT, nk % MT, q, k);
      }
      // scale FMAs of the previous slot
      const int pi = (j + MT - 1) % MT;
#pragma unroll
      for (int r = 0; r < 16; r++) acc[pi][r] = fmaf(dprev, prev[r], acc[pi][r]);
      // the next block: window to integers, the two operands, the scale
      if (i == 0) {
        if (kb == 0) take(wodd, 1, raw);
        else take(weven, 0, raw);
        nb[0] = unpack(raw, 0);
        if (kb == 0) {
          asm volatile("" ::"v"(raw.d) : "memory");
#pragma unroll
          for (int k = 0; k < kQd; k++) asm volatile("" ::"v"(raw.q[k]) : "memory");
        }
      }
      if (i == (MT > 1 ? 1 : 0)) nb[1] = unpack(raw, 1);
      if (i == MT - 1) {
        nd = kb == 0 ? scale_of(raw, s, 1) : scale_of(raw, s + 1, 0);
        if (kb == 0) wodd_next = read_win(s + 1, 1);
      }
      prev = p;
      dprev = d;
      if (i == MT - 1) {
        fb[0] = nb[0];
        fb[1] = nb[1];
        d = nd;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (PARTS == 3) {
      if (s % kGroup == kGroup - 1) {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            tot[i][r] += acc[i][r];
            acc[i][r] = 0.0f;
          }
      }
    }
    wodd = wodd_next;
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(G::kStageWait) : "memory");
  }
#pragma unroll
  for (int r = 0; r < 16; r++) acc[MT - 1][r] = fmaf(dprev, prev[r], acc[MT - 1][r]);
  if constexpr (PARTS == 3) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][r] += tot[i][r];
  }
  // Every DMA into LDS (the trailing re-reads included) has landed before
  // the work-group's LDS is released.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // Register r of a lane holds output row m0 + 32 i + 8 (r / 4) + 4 h + r % 4,
  // column ncol: scaled back by 2^xexp[m] (exact).  Y goes out through a
  // buffer whose range is M x N, so rows past M drop out of range and lanes
  // past N aim past it.  K pieces write their partial plane instead; the
  // reduction adds the bias.
  const __amdgpu_buffer_rsrc_t ers = brsrc(a.xexp, (uint32_t)a.M * 4u);
  float* dst = a.splits > 1 ? a.part + (size_t)z * a.M * a.N : a.y;
  const __amdgpu_buffer_rsrc_t yrs = brsrc(dst, a.y_bytes);
  const float bv = (nvalid && a.bias && a.splits == 1) ? a.bias[ncol] : 0.0f;
#pragma unroll
  for (int i = 0; i < MT; i++) {
    uint32_t ex[16];
#pragma unroll
    for (int r = 0; r < 16; r++)
      ex[r] = __builtin_amdgcn_raw_buffer_load_b32(
          ers, (uint32_t)(m0 + 32 * i + 8 * (r / 4) + 4 * h + r % 4) * 4u, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const uint32_t m = (uint32_t)(m0 + 32 * i + 8 * (r / 4) + 4 * h + r % 4);
      const uint32_t off = nvalid ? (m * (uint32_t)a.N + (uint32_t)ncol) * 4u : 0xFFFFFFF0u;
      const float v = ldexpf(acc[i][r], (int)ex[r]) + bv;
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yrs, off, 0, 0);
    }
  }
#endif
}

// Y = the planes (+ bias): plane z in sum z % 4, the four then added, an order of
// its own that is the same on every run (up to 64 planes as one chain rounded
// more than the fp32 dot products: 16 tokens, column-major 2048 x 2048 in 32
// pieces 1.16e-7 against 1.15e-7).
__global__ void __launch_bounds__(256)
block_split_reduce_kernel(float* __restrict__ y, const float* __restrict__ part,
                          const float* __restrict__ bias, size_t mn, int n, int splits) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= mn) return;
  float v[4] = {part[i], 0.0f, 0.0f, 0.0f};
  for (int z = 1; z < 4 && z < splits; z++) v[z] = part[(size_t)z * mn + i];
  for (int z = 4; z < splits; z += 4) {
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (z + k < splits) v[k] += part[(size_t)(z + k) * mn + i];
  }
  y[i] = ((v[0] + v[1]) + (v[2] + v[3])) + (bias ? bias[i % n] : 0.0f);
}

// X fp32 [M][K] -> three bf16 planes [M][Kp], `plane` vectors apart, one
// work-group of 256 threads per row: x 2^sh = x1 + x2 + x3 exactly, each part
// the next 8 bits of x with its sign.  sh puts the row's largest finite |x| in
// [2^(kXTop - 1), 2^kXTop), where no sum of products overflows and the last
// part of an element is whole down to 2^-186 of that maximum; xexp[row] = -sh,
// columns K .. Kp - 1 zero.  An infinity or NaN is x1 alone.  The row is read
// once if it fits the registers (K <= 16384 and 16-byte aligned), twice
// otherwise.
constexpr int kXG = 8;
constexpr int kXTop = 76;
__global__ void __launch_bounds__(256)
x_rows_split_kernel(u32x4* __restrict__ xh, int* __restrict__ xexp, const float* __restrict__ x,
                    size_t plane, int K, int Kp) {
  __shared__ uint32_t red[4];
  const int row = blockIdx.x;
  const int t = threadIdx.x;
  const int groups = K / 8, gp = Kp / 8;
  u32x4* dst = xh + (size_t)row * gp;
  const float* src = x + (size_t)row * K;
  const bool al = ((uintptr_t)src & 15) == 0;
  const bool keep = al && groups <= 256 * kXG;
  float4 v[kXG][2];
  uint32_t mb = 0;  // largest finite |x| by bit pattern
  auto load8 = [&](int g, float4& lo, float4& hi) {
    const float* p = src + (size_t)g * 8;
    if (al) {
      lo = load_global<float4>(p);
      hi = load_global<float4>(p + 4);
    } else {
      lo = make_float4(p[0], p[1], p[2], p[3]);
      hi = make_float4(p[4], p[5], p[6], p[7]);
    }
  };
  auto amax8 = [&](const float4& lo, const float4& hi) {
    const float e[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const uint32_t b = __float_as_uint(e[i]) & 0x7FFFFFFFu;
      mb = max(mb, b < 0x7F800000u ? b : 0u);
    }
  };
  if (keep) {
#pragma unroll
    for (int u = 0; u < kXG; u++)
      if (t + 256 * u < groups) load8(t + 256 * u, v[u][0], v[u][1]);
#pragma unroll
    for (int u = 0; u < kXG; u++)
      if (t + 256 * u < groups) amax8(v[u][0], v[u][1]);
  } else {
    for (int g = t; g < groups; g += 256) {
      float4 lo, hi;
      load8(g, lo, hi);
      amax8(lo, hi);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mb = max(mb, (uint32_t)__shfl_xor((int)mb, off, 64));
  if ((t & 63) == 0) red[t >> 6] = mb;
  __syncthreads();
  mb = max(max(red[0], red[1]), max(red[2], red[3]));
  const int sh = mb ? kXTop - __builtin_amdgcn_frexp_expf(__uint_as_float(mb)) : 0;
  auto put = [&](int g, const float4& lo, const float4& hi) {
    const float e[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    uint32_t b[3][8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float s = ldexpf(e[i], sh);
      b[0][i] = __float_as_uint(s) & 0xFFFF0000u;
      const float r1 = s - __uint_as_float(b[0][i]);
      b[1][i] = __float_as_uint(r1) & 0xFFFF0000u;
      b[2][i] = __float_as_uint(r1 - __uint_as_float(b[1][i]));
      if (!(fabsf(s) < __builtin_inff())) {
        if (s != s) b[0][i] = 0x7FC00000u;
        b[1][i] = b[2][i] = 0u;
      }
    }
#pragma unroll
    for (int p = 0; p < 3; p++) {
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 4; j++)
        o[j] = __builtin_amdgcn_perm(b[p][2 * j + 1], b[p][2 * j], 0x07060302u);
      dst[p * plane + g] = o;
    }
  };
  if (keep) {
#pragma unroll
    for (int u = 0; u < kXG; u++)
      if (t + 256 * u < groups) put(t + 256 * u, v[u][0], v[u][1]);
  } else {
    for (int g = t; g < groups; g += 256) {
      float4 lo, hi;
      load8(g, lo, hi);
      put(g, lo, hi);
    }
  }
  if (t < gp - groups)
    for (int p = 0; p < 3; p++) dst[p * plane + groups + t] = u32x4{0u, 0u, 0u, 0u};
  if (t == 0) xexp[row] = -sh;
}

size_t rup(size_t v, size_t a) { return (v + a - 1) / a * a; }

}  // namespace

// Geometry chosen for a shape: 32-row tiles per wave and K pieces.
//
// Costs (microseconds, fitted to 26 shapes at every number of pieces; the plans
// they choose measured 0.2% above the best on average, 1% at most): a 64-K stage
// 0.95 / 1.2 on 32- / 64-row tiles, a round of work-groups (one per CU) ~3 more
// to fill and drain; K pieces add the reduction launch (~2.5), 0.3 each and the
// partial planes' traffic (~2 TB/s a way).
BlockPlan block_plan(size_t n, size_t m, size_t batch, int num_cus) {
  const size_t tn = (n + kBN - 1) / kBN;
  const size_t steps = rup(m, kBStageK) / kBStageK;
  BlockPlan best{1, 1, 0.0};
  double best_cost = 1e300;
  // (rows of an even number of blocks come with fewer than 16 tokens, or with
  // more than the prefill kernels' limits allow: 32-row tiles only)
  const bool odd = m / kBlockElems % 2 != 0;
  for (int mt : {1, 2}) {
    if (mt > 1 && (!odd || (size_t)16 * mt >= batch)) break;  // taller tiles than the rows
    const size_t tm = (batch + 32 * mt - 1) / (32 * mt);
    const size_t tiles = tm * tn;
    const double stage_us = mt == 2 ? 1.2 : 0.95;
    for (size_t sp = 1; sp <= std::min<size_t>(steps, 64); sp++) {
      const size_t wgs = tiles * sp;
      const size_t rounds = (wgs + num_cus - 1) / num_cus;
      double cost = (double)rounds * ((double)((steps + sp - 1) / sp) * stage_us + 3.0);
      if (sp > 1) cost += 2.5 + (double)sp * (0.3 + (double)(batch * n * 4) / 2.0e6);
      if (cost < best_cost * 0.999) {
        best_cost = cost;
        best = BlockPlan{mt, (int)sp, cost};
      }
      if (rounds > 1 && sp > 1) break;  // more pieces only add rounds
    }
  }
  return best;
}

// The same for x rounded once to fp16 (m % 64 == 0), with no more than
// `planes` bytes of partial planes.  A stage costs 1.0 / 1.42 / 2.35 on 64- /
// 128- / 256-row tiles of Q8_0; K pieces write planes that the reduction reads,
// ~3 TB/s in all.  Q4_0 has the 256-row tiles only (2.3): on lower ones the
// 16x16x32 kernel is as fast or faster (512 x 14336, K 4096: 90 us against 91;
// 2048 x 4096, K 4096: 98 / 100; 1024 x 4096, K 14336: 173 / 179; 400 x 14336, K
// 2048: 49.5 / 50.7).
BlockPlan block_plan_f16x(int fmt, size_t n, size_t m, size_t batch, int num_cus, size_t planes) {
  const size_t tn = (n + kBN - 1) / kBN;
  const size_t steps = m / kBStageK;
  const bool q8 = fmt == kFmtQ8_0;
  BlockPlan best{q8 ? 2 : 8, 1, 1e300};
  for (int mt : {2, 4, 8}) {
    if (!q8 && mt != 8) continue;
    if (mt > 2 && (size_t)16 * mt >= batch) break;  // taller tiles than the rows
    const size_t tm = (batch + 32 * mt - 1) / (32 * mt);
    const size_t tiles = tm * tn;
    const double stage_us = mt == 8 ? (q8 ? 2.35 : 2.3) : mt == 4 ? 1.42 : 1.0;
    for (size_t sp = 1; sp <= std::min<size_t>(steps, 64); sp++) {
      if (sp > 1 && sp * batch * n * 4 > planes) break;
      const size_t rounds = (tiles * sp + num_cus - 1) / num_cus;
      double cost = (double)rounds * ((double)((steps + sp - 1) / sp) * stage_us + 3.0);
      if (sp > 1) cost += 2.5 + (double)sp * (double)(batch * n * 4) / 3.0e6;
      if (cost < best.cost * 0.999) best = BlockPlan{mt, (int)sp, cost};
      if (rounds > 1 && sp > 1) break;  // more pieces only add rounds
    }
  }
  return best;
}

// K % 32 == 0, w 4-byte aligned and holding N whole rows in whole dwords
// (the last row's window ends on the buffer's last dword), W, X and Y under
// 4 GB (32-bit buffer offsets).
bool block_gemm_ok(int fmt, const uint8_t* w, size_t w_len, size_t n, size_t m, size_t batch) {
  if (m == 0 || m % 32 != 0 || n == 0 || batch == 0) return false;
  if (((uintptr_t)w & 3) != 0) return false;
  if (n > (size_t)0x7FFFFFF || m > (size_t)0x7FFFFFF || batch > (size_t)0x7FFFFFF) return false;
  const size_t wbytes =
      rup(n * (m / kBlockElems) * (fmt == kFmtQ8_0 ? kQ8BlockBytes : kBlockBytes), 4);
  if (wbytes >= ((size_t)1 << 32) - 4096) return false;
  if ((batch + 256) * rup(m, kBStageK) * 2 >= ((size_t)1 << 32)) return false;
  // Output offsets (row m < M + 256) stay below 2^32 - 16 (the lanes past N
  // aim at 2^32 - 16).
  if ((batch + 256) * n * 4 >= ((size_t)1 << 32) - 16) return false;
  return w_len >= wbytes;
}

size_t x_split_bytes(size_t batch, size_t m) {
  return rup(3 * batch * rup(m, kBStageK) * 2, 256) + rup(batch * 4, 256);
}

int* x_split_exponents(void* xs, size_t batch, size_t m) {
  return reinterpret_cast<int*>(static_cast<uint8_t*>(xs) +
                                rup(3 * batch * rup(m, kBStageK) * 2, 256));
}

hipError_t launch_x_split(void* xs, const float* x, size_t batch, size_t m, hipStream_t s) {
  const size_t kp = rup(m, kBStageK);
  hipLaunchKernelGGL(x_rows_split_kernel, dim3((unsigned)batch), dim3(256), 0, s,
                     static_cast<u32x4*>(xs), x_split_exponents(xs, batch, m), x, batch * kp / 8,
                     (int)m, (int)kp);
  return hipGetLastError();
}

size_t block_gemm_workspace_bytes(const BlockPlan& p, size_t n, size_t m, size_t batch) {
  return x_split_bytes(batch, m) + (p.splits > 1 ? (size_t)p.splits * batch * n * 4 : 0);
}

template <int FMT, bool ODD>
static hipError_t launch_block_mt(const BlockPlan& p, const BlockArgs& a, hipStream_t s) {
  auto go = [&](auto kernel, int lds) -> hipError_t {
    hipError_t e = set_lds_limit(reinterpret_cast<const void*>(kernel), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(a.tiles_m * a.tiles_n, p.splits), dim3(kBThreads), lds, s, a);
    return hipGetLastError();
  };
  if constexpr (ODD)
    if (p.mt == 2) return go(gemm_block_kernel<FMT, 2, ODD, 3>, BlockGeom<FMT, 2, ODD>::kLds);
  return go(gemm_block_kernel<FMT, 1, ODD, 3>, BlockGeom<FMT, 1, ODD>::kLds);
}

hipError_t launch_block_gemm(const BlockPlan& p, int fmt, float* y, const uint8_t* w,
                             const float* x, const float* bias, size_t n, size_t m, size_t batch,
                             void* ws, hipStream_t s) {
  const size_t kp = rup(m, kBStageK);
  BlockArgs a;
  a.y = y;
  a.w = w;
  a.xh = static_cast<const uint8_t*>(ws);
  a.bias = bias;
  a.xexp = x_split_exponents(ws, batch, m);
  a.part = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + x_split_bytes(batch, m));
  a.B = (int)(m / kBlockElems);
  a.w_bytes = (uint32_t)rup(n * a.B * (fmt == kFmtQ8_0 ? kQ8BlockBytes : kBlockBytes), 4);
  a.x_bytes = (uint32_t)(batch * kp * 2);
  a.y_bytes = (uint32_t)(batch * n * 4);
  a.M = (int)batch;
  a.N = (int)n;
  a.steps = (int)(kp / kBStageK);
  a.tiles_m = (int)((batch + 32 * p.mt - 1) / (32 * p.mt));
  a.tiles_n = (int)((n + kBN - 1) / kBN);
  a.xcd_map = (a.tiles_m * a.tiles_n) % 8 == 0 ? 1 : 0;
  a.splits = p.splits;

  const bool q8 = fmt == kFmtQ8_0, odd = a.B % 2 != 0;
  hipError_t e = launch_x_split(ws, x, batch, m, s);
  if (e != hipSuccess) return e;
  if (q8)
    e = odd ? launch_block_mt<kFmtQ8_0, true>(p, a, s) : launch_block_mt<kFmtQ8_0, false>(p, a, s);
  else
    e = odd ? launch_block_mt<kFmtQ4_0, true>(p, a, s) : launch_block_mt<kFmtQ4_0, false>(p, a, s);
  if (e != hipSuccess || p.splits == 1) return e;
  return launch_split_reduce(y, a.part, bias, batch * n, n, p.splits, s);
}

template <int FMT>
static hipError_t launch_block_single(const BlockPlan& p, const BlockArgs& a, hipStream_t s) {
  auto go = [&](auto kernel, int lds) -> hipError_t {
    hipError_t e = set_lds_limit(reinterpret_cast<const void*>(kernel), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(a.tiles_m * a.tiles_n, p.splits), dim3(kBThreads), lds, s, a);
    return hipGetLastError();
  };
  if (p.mt == 8) return go(gemm_block_kernel<FMT, 8, false, 1>, BlockGeom<FMT, 8, false, 1>::kLds);
  if constexpr (FMT == kFmtQ8_0) {
    if (p.mt == 4)
      return go(gemm_block_kernel<FMT, 4, false, 1>, BlockGeom<FMT, 4, false, 1>::kLds);
    if (p.mt == 2)
      return go(gemm_block_kernel<FMT, 2, false, 1>, BlockGeom<FMT, 2, false, 1>::kLds);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_block_gemm_f16x(const BlockPlan& p, int fmt, float* y, const uint8_t* w,
                                  const float* bias, size_t n, size_t m, size_t batch,
                                  const void* xh, size_t x_bytes, const int* xexp, float* part,
                                  hipStream_t s) {
  BlockArgs a;
  a.y = y;
  a.w = w;
  a.xh = static_cast<const uint8_t*>(xh);
  a.bias = bias;
  a.xexp = xexp;
  a.part = part;
  a.B = (int)(m / kBlockElems);
  a.w_bytes = (uint32_t)(n * a.B * (fmt == kFmtQ8_0 ? kQ8BlockBytes : kBlockBytes));
  a.x_bytes = (uint32_t)x_bytes;
  a.y_bytes = (uint32_t)(batch * n * 4);
  a.M = (int)batch;
  a.N = (int)n;
  a.steps = (int)(m / kBStageK);
  a.tiles_m = (int)((batch + 32 * p.mt - 1) / (32 * p.mt));
  a.tiles_n = (int)((n + kBN - 1) / kBN);
  a.xcd_map = (a.tiles_m * a.tiles_n) % 8 == 0 ? 1 : 0;
  a.splits = p.splits;
  hipError_t e = fmt == kFmtQ8_0 ? launch_block_single<kFmtQ8_0>(p, a, s)
                                 : launch_block_single<kFmtQ4_0>(p, a, s);
  if (e != hipSuccess || p.splits == 1) return e;
  return launch_split_reduce(y, part, bias, batch * n, n, p.splits, s);
}

hipError_t launch_split_reduce(float* y, const float* part, const float* bias, size_t mn, size_t n,
                               int splits, hipStream_t s) {
  hipLaunchKernelGGL(block_split_reduce_kernel, dim3((unsigned)((mn + 255) / 256)), dim3(256), 0,
                     s, y, part, bias, mn, (int)n, splits);
  return hipGetLastError();
}

}  // namespace hypno
