// Q4 projection of a short prompt's rows (17 .. 128, or a few times that where
// the tiles suit the chip; q4_rows_supported has the line):
// Y[M][N] = X[M][K] * dequant(W)^T with the GEMM's numerics (q4_gemm.hip):
// weights fp16(q*s + b), activations fp16, fp32 sums, bf16 output.
//
// At these sizes the weights' bytes and the products cost about the same (77
// rows: 36 us of HBM and 41 us of MFMA for the layer's set and down
// projection), and the GEMM's 256-row tiles spend most of their products on
// padding and their steps on a dequantise -> LDS -> read chain.  Here a tile is
// 32 MB rows (up to 96) by 192 W rows, and only packed weights pass LDS:
//
//  * Twelve waves as 3 (64 W rows each) x 4 (K parts).  A round is one
//    quantisation group for each K part: 128 contiguous bytes (a cache line) of
//    each of the 192 W rows.  Lane (n, h) of a wave takes half h (16 bytes, four words)
//    of its group of W row n, and word s of it, dequantised in registers, is
//    its B operand of MFMA step s: the k order of a group is then (h, s,
//    element), and X is stored to match.  Every W element is read and
//    dequantised once per row tile.
//  * X is converted once per call into fp16 blocks in MFMA operand order
//    (x_rows_kernel), so its part of a round is read back linearly.
//  * Both are DMAed to LDS NS - 1 rounds ahead, W as 128-byte runs of a row
//    into slots whose swizzle keeps the reads off each other's banks.  One
//    barrier a round.
//  * Scales and biases of eight groups are loaded by the waves that own the
//    rows, converted to fp16 and passed through LDS.
//  * The K parts meet in LDS at the end.  When the tiles alone leave the chip
//    idle, K is cut into slices whose fp32 tiles a second launch adds in slice
//    order (the sum does not depend on timing) before the epilogue.
//
// Measured for QKV 5120 -> 10240 with the gate/up pair 5120 -> 2 x 17408, and
// down 17408 -> 5120 (us; the GEMM's tiles before): 17 rows 50 + 27 (153 + 90),
// 77 rows 64 + 34 (150 + 96), 160 rows 120 + 52 (152 + 99), 300 rows 236 + 89
// (272 + 127).  What bounds it at 77 rows, by taking one part out: the
// dequantisation 5 us, the W loads 7, the X loads 10, the scale loads 4; the
// products alone are 28 us at the clock that random operands leave.  Three
// waves a SIMD (at most 168 registers) hide the rest better than two: 4 x 2
// waves on 256 W rows took 81 + 37 us, and with W loaded straight to registers
// (32-byte runs of 32 rows an instruction) 88 + 38.  192 rows a tile also
// leave fewer CUs idle than 256 at these widths (236 tiles of the set).
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace qm {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

constexpr int WN = 3, WK = 4;  // waves over the W rows of a tile (64 each), and over K
constexpr int kXcds = 8, kUnitGroups = 8;  // groups whose scales are passed together
constexpr uint32_t kMaxBlocks = 3;          // 32-row blocks of X in a tile

struct RowsArgs {
  Q4Job jobs[kMaxQ4Jobs];  // plain projections and gate/up pairs (kQ4OutSwiglu)
  int n_jobs;
  const uint16_t* xt;  // fp16 blocks [m tile][group][32-row block][step][64 lanes][8]
  uint32_t K, M;
  uint32_t m_tiles, tiles, slices;
  float* partials;  // [tile][slice][32 MB x 64 WN] fp32 in accumulator order
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint64_t bytes) {
  const uint32_t n = bytes > 0xFFFFFFF0ull ? 0xFFFFFFF0u : (uint32_t)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)n, 0x00020000);
}

// Lane i's 16 bytes land at lds + 16 i (the builtin exists only in the device pass).
#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}
#else
__device__ void dma16(__amdgpu_buffer_rsrc_t, void*, uint32_t, uint32_t);
#endif

// s_waitcnt vmcnt(n) lgkmcnt(0) (gfx9 encoding; expcnt left at its maximum):
// this wave's LDS reads are done, and all but its n latest loads.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 0xF) | ((N >> 4) << 14));
  __asm__ volatile("" ::: "memory");
}

__device__ __forceinline__ floatx16 mfma_f16(u32x4 a, u32x4 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0,
                                                0, 0);
}

__device__ __forceinline__ uint32_t dq_pair(uint32_t w, int j, half2v s2, half2v b2) {
  const uint32_t t = ((w >> (4 * j)) & 0x000F000Fu) | 0x64006400u;
  const half2v q = __builtin_bit_cast(half2v, t) - (half2v){(_Float16)1024.0f, (_Float16)1024.0f};
  return __builtin_bit_cast(uint32_t, q * s2 + b2);
}

// X -> xt: thread (block, lane) writes the 16 bytes of row 32 b + (lane & 31),
// chunk 4 (lane >> 5) + s of its group, elements in the order 0,4,1,5,2,6,3,7
// in which a packed word unpacks.  Rows past M are zero.
// Activations beyond the fp16 range saturate, as in the GEMM.
__global__ __launch_bounds__(256) void x_rows_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ xt,
                                                     uint32_t K, uint32_t M, uint32_t mb, size_t chunks) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= chunks) return;
  const uint32_t lane = i & 63, s = (i >> 6) & 3;
  const size_t blk = i >> 8;  // (m tile * groups + group) * mb + block
  const uint32_t b = blk % mb, G = K / 64, g = blk / mb % G, mt = blk / mb / G;
  const uint32_t row = (mt * mb + b) * 32 + (lane & 31), k = 64 * g + 8 * (4 * (lane >> 5) + s);
  u32x4 v = {0u, 0u, 0u, 0u};
  if (row < M) v = *(const u32x4*)(x + (size_t)row * K + k);
  uint32_t h[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float f = bf16_to_f32(e & 1 ? v[e >> 1] >> 16 : v[e >> 1] & 0xFFFFu);
    f = f > 65504.0f ? 65504.0f : (f < -65504.0f ? -65504.0f : f);
    const _Float16 c = (_Float16)f;
    h[e] = __builtin_bit_cast(uint16_t, c);
  }
  *(u32x4*)(xt + 8 * i) = u32x4{h[0] | (h[4] << 16), h[1] | (h[5] << 16), h[2] | (h[6] << 16), h[3] | (h[7] << 16)};
}

// One column's four rows m .. m + 3 (q: accumulator quad of the 32-row block).
__device__ __forceinline__ void store_quad(const Q4Job& jb, bool pair, uint32_t M, uint32_t m, uint32_t n0,
                                           uint32_t n1, floatx4 v0, floatx4 v1) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (m + e >= M) break;
    uint16_t* row = jb.out + (size_t)(m + e) * jb.rows;
    if (pair) {
      if (n0 < jb.rows) row[n0] = f32_to_bf16(silu_f(v0[e]) * v1[e]);
    } else {
      if (n0 < jb.rows) row[n0] = f32_to_bf16(v0[e]);
      if (n1 < jb.rows) row[n1] = f32_to_bf16(v1[e]);
    }
  }
}

// The tile's job and first row (of the gate, for a pair's 32 WN + 32 WN rows).
__device__ __forceinline__ const Q4Job& tile_job(const RowsArgs& args, uint32_t n_tile, bool* pair, uint32_t* n_first) {
  int jt = 0;
  while (jt + 1 < args.n_jobs && n_tile >= args.jobs[jt + 1].tile_begin) ++jt;
  const Q4Job& jb = args.jobs[jt];
  *pair = jb.mode == kQ4OutSwiglu;
  *n_first = (n_tile - jb.tile_begin) * (*pair ? 32u : 64u) * WN;
  return jb;
}

// Rounds in LDS (24 + 16 MB KB each, beside 12 KB of scales).
constexpr int rows_stages(int mb) { return mb == 1 ? 3 : 2; }

template <int MB>
__global__ __launch_bounds__(64 * WN * WK, WN * WK / 4) void q4_rows_kernel(RowsArgs args) {
  constexpr int NS = rows_stages(MB), kWaves = WN * WK;
  constexpr uint32_t kRowB = 32 * WK;                   // bytes of a W row in a round
  constexpr uint32_t kP = 2 * WK;                       // ... in 16-byte pieces
  constexpr uint32_t kW = 64 * WN * kRowB, kX = 4096 * MB * WK, kStage = kW + kX;
  constexpr uint32_t kScales = 64 * WN * 32;            // a unit's: per W row 8 scales and 8 biases, fp16
  constexpr uint32_t kUnit = kUnitGroups / WK;          // rounds of a unit
  constexpr uint32_t kRed = WN * MB * 2 * 4096;         // one K part's accumulators
  constexpr uint32_t kBytes = NS * kStage + 2 * kScales;
  constexpr uint32_t kRedParts = WK / 2;                // ... that meet in LDS at a time
  __shared__ __attribute__((aligned(16))) uint8_t lds[kBytes > kRed * kRedParts ? kBytes : kRed * kRedParts];

  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wn = wave % WN, wk = wave / WN;
  const uint32_t K = args.K, G = K / 64, R = G / WK;

  // Workgroups are dealt round-robin to the XCDs; an XCD takes a contiguous
  // run of (W tile, slice, row tile), so the row tiles of a slice share its L2.
  const uint32_t workers = args.tiles * args.slices;
  const uint32_t xcd = blockIdx.x % kXcds, wq = workers / kXcds, wrem = workers % kXcds;
  const uint32_t lw = xcd * wq + min(xcd, wrem) + blockIdx.x / kXcds;
  const uint32_t n_tile = lw / (args.slices * args.m_tiles), rest = lw % (args.slices * args.m_tiles);
  const uint32_t slice = rest / args.m_tiles, m_tile = rest % args.m_tiles;
  const uint32_t units = (G + kUnitGroups - 1) / kUnitGroups;
  const uint32_t r0 = units * slice / args.slices * kUnit, r1 = min(R, units * (slice + 1) / args.slices * kUnit);

  bool pair;
  uint32_t n_first;
  const Q4Job& jb = tile_job(args, n_tile, &pair, &n_first);

  // W rows of the tile as staged: 64 WN rows of a plain projection, or 32 WN
  // gate rows and their up rows.  Resources start at the tile's first row, so
  // 32-bit offsets suffice.
  const size_t rows_left = jb.rows - n_first;
  const uint32_t last_row = (uint32_t)min(rows_left, (size_t)64 * WN) - 1;
  constexpr uint32_t kRowsPer = 64 / kP;                // staged rows of one W DMA
  constexpr uint32_t kWDma = kW / 1024 / kWaves;        // W DMAs of a wave
  static_assert(kWDma * kWaves * 1024 == kW, "every wave stages the same share of W");
  // 16-byte piece p of staged row r lies in slot kP r + (p ^ swz(r)).
  auto swz = [](uint32_t row) { return (row >> 1) & 7; };
  uint32_t w_off[kWDma];
  __amdgpu_buffer_rsrc_t rw[kWDma];
#pragma unroll
  for (uint32_t k = 0; k < kWDma; ++k) {
    const uint32_t first = (wave * kWDma + k) * kRowsPer;  // uniform
    const bool up = pair && first >= 32 * WN;
    rw[k] = make_rsrc((up ? jb.uw : jb.w) + (size_t)n_first * (K / 8), rows_left * (K / 2));
    const uint32_t row = first + lane / kP, p = (lane % kP) ^ swz(row);
    w_off[k] = min(up ? row - 32 * WN : row, last_row) * (K / 2) + 16 * p;
  }
  // Scales of 64 staged rows by each of the waves 0 .. WN - 1, their biases by
  // the next WN.  A pair's boundary lies inside a wave's rows when WN is odd,
  // so up to two resources, one for each half of the lanes.
  const bool sc_wave = wave < 2 * WN;
  const uint32_t sc_first = 64 * (wave % WN);
  auto sc_rsrc = [&](bool up) {
    const uint16_t* t = wave < WN ? (up ? jb.us : jb.s) : (up ? jb.ub : jb.b);
    return make_rsrc(t + (size_t)n_first * G, rows_left * G * 2);
  };
  const bool up0 = pair && sc_first >= 32 * WN, up1 = pair && sc_first + 32 >= 32 * WN;
  const __amdgpu_buffer_rsrc_t rs0 = sc_rsrc(up0), rs1 = sc_rsrc(up1);
  const uint32_t sc_row = sc_first + lane, sc_up = lane < 32 ? up0 : up1;
  const uint32_t sc_off = min(sc_up ? sc_row - 32 * WN : sc_row, last_row) * G * 2;
  uint8_t* const scales = lds + NS * kStage;
  uint8_t* const sc_dst = scales + sc_row * 32 + (wave < WN ? 0 : 16);

  const __amdgpu_buffer_rsrc_t rx = make_rsrc(args.xt + (size_t)m_tile * G * (2048 * MB), (uint64_t)G * (4096 * MB));
  constexpr uint32_t kXDma = kX / 1024, kXMin = kXDma / kWaves;  // X DMAs of a round, and of a wave at least
  auto load = [&](uint32_t r) __attribute__((always_inline)) {
    const uint32_t src = min(r, r1 - 1);
    uint8_t* dst = lds + (r - r0) % NS * kStage;
#pragma unroll
    for (uint32_t k = 0; k < kWDma; ++k) dma16(rw[k], dst + (wave * kWDma + k) * 1024, w_off[k], src * kRowB);
#pragma unroll
    for (uint32_t k = 0; k * kWaves < kXDma; ++k) {
      const uint32_t x = k * kWaves + wave;
      if (x < kXDma) dma16(rx, dst + kW + x * 1024, lane * 16, src * kX + x * 1024);
    }
  };
  // Eight scales (or biases) of the lane's row; those of groups past K are not used.
  auto sc_load = [&](uint32_t u) __attribute__((always_inline)) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (sc_wave) {
      const uint32_t at = min(u, units - 1) * (2 * kUnitGroups);
      if (up0 == up1) {
        v = __builtin_amdgcn_raw_buffer_load_b128(rs0, sc_off, at, 0);
      } else if (lane < 32) {
        v = __builtin_amdgcn_raw_buffer_load_b128(rs0, sc_off, at, 0);
      } else {
        v = __builtin_amdgcn_raw_buffer_load_b128(rs1, sc_off, at, 0);
      }
    }
    return v;
  };
  auto sc_store = [&](uint32_t u, u32x4 v) __attribute__((always_inline)) {
    if (!sc_wave) return;
    uint32_t h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const half2v f = {(_Float16)bf16_to_f32(v[i] & 0xFFFFu), (_Float16)bf16_to_f32(v[i] >> 16)};
      h[i] = __builtin_bit_cast(uint32_t, f);
    }
    *(u32x4*)(sc_dst + (u & 1) * kScales) = u32x4{h[0], h[1], h[2], h[3]};
  };

  floatx16 acc[MB][2];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[m][j] = floatx16{};

  // Loads retire in order: a round's are followed by at least this many, those
  // of the NS - 2 rounds after it (and, now and then, by a scale load).
  constexpr int kAfter = (NS - 2) * (kWDma + kXMin);
  u32x4 sc = sc_load(r0 / kUnit);
#pragma unroll
  for (int r = 0; r < NS - 1; ++r) load(r0 + r);
  sc_store(r0 / kUnit, sc);

  uint32_t w_rd[2], s_rd[2], n[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t row = (pair ? 32 * WN * j + 32 * wn : 64 * wn + 32 * j) + (lane & 31);
    w_rd[j] = 16 * (kP * row + ((2 * wk + (lane >> 5)) ^ swz(row)));
    s_rd[j] = row * 32;
  }
  n[0] = n_first + (pair ? 32 : 64) * wn + (lane & 31);
  n[1] = pair ? n[0] : n[0] + 32;

  for (uint32_t r = r0; r < r1; ++r) {
    const uint32_t u = r / kUnit, i = r % kUnit;
    wait_vmcnt<kAfter>();
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
    load(r + NS - 1);  // into the stage that every wave left before the barrier
    if (i == 0) sc = sc_load(u + 1);
    const uint8_t* st = lds + (r - r0) % NS * kStage;
    const uint8_t* sp = scales + (u & 1) * kScales + 2 * (WK * i + wk);
    u32x4 w[2];
    half2v s2[2], b2[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      w[j] = *(const u32x4*)(st + w_rd[j]);
      const _Float16 s = *(const _Float16*)(sp + s_rd[j]), b = *(const _Float16*)(sp + s_rd[j] + 16);
      s2[j] = half2v{s, s};
      b2[j] = half2v{b, b};
    }
    const uint8_t* xs = st + kW + wk * (4096 * MB) + lane * 16;
    // A operands leave LDS kAhead steps early (all at once where the registers allow).
    constexpr int kAhead = MB == 3 ? 2 : 4;
    u32x4 a[4][MB];
    auto a_load = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int m = 0; m < MB; ++m) a[s][m] = *(const u32x4*)(xs + (m * 4 + s) * 1024);
    };
#pragma unroll
    for (int s = 0; s < kAhead; ++s) a_load(s);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      u32x4 b[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b[j] = u32x4{dq_pair(w[j][s], 0, s2[j], b2[j]), dq_pair(w[j][s], 1, s2[j], b2[j]),
                     dq_pair(w[j][s], 2, s2[j], b2[j]), dq_pair(w[j][s], 3, s2[j], b2[j])};
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[m][j] = mfma_f16(a[s][m], b[j], acc[m][j]);
      if (s + kAhead < 4) {
        a_load(s + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // The next unit's scales: their buffer was last read a unit ago.
    if (i == kUnit / 2) sc_store(u + 1, sc);
  }

  // The K parts' accumulators meet in LDS, which every load has to have left:
  // the upper half of the parts is added to the lower one, then again.
  wait_vmcnt<0>();
  __syncthreads();
#pragma unroll
  for (uint32_t h = WK / 2; h > 0; h /= 2) {
    floatx4* red = (floatx4*)lds + ((size_t)(wk % h) * WN + wn) * MB * 2 * 4 * 64 + lane;
    if (wk >= h && wk < 2 * h) {
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            red[((m * 2 + j) * 4 + q) * 64] =
                floatx4{acc[m][j][4 * q], acc[m][j][4 * q + 1], acc[m][j][4 * q + 2], acc[m][j][4 * q + 3]};
    }
    __syncthreads();
    if (wk < h) {
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const floatx4 v = red[((m * 2 + j) * 4 + q) * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[m][j][4 * q + e] += v[e];
          }
    }
    if (h > 1) __syncthreads();
  }
  if (wk > 0) return;
  const uint32_t tile = n_tile * args.m_tiles + m_tile;
  floatx4* po = (floatx4*)args.partials +
                (((size_t)tile * args.slices + slice) * WN + wn) * MB * 2 * 4 * 64 + lane;
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      floatx4 v[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        v[j] = floatx4{acc[m][j][4 * q], acc[m][j][4 * q + 1], acc[m][j][4 * q + 2], acc[m][j][4 * q + 3]};
      if (args.slices > 1) {
        po[((m * 2) * 4 + q) * 64] = v[0];
        po[((m * 2 + 1) * 4 + q) * 64] = v[1];
      } else {
        store_quad(jb, pair, args.M, (m_tile * MB + m) * 32 + 8 * q + 4 * (lane >> 5), n[0], n[1], v[0], v[1]);
      }
    }
}

// Adds a tile's slices in slice order and runs the epilogue: a thread per
// (W-row block pair, quad of rows).
template <int MB>
__global__ __launch_bounds__(256) void q4_rows_reduce_kernel(RowsArgs args) {
  const uint32_t lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const uint32_t m = blockIdx.x % MB, wn = blockIdx.x / MB % WN, tile = blockIdx.x / (WN * MB);
  const uint32_t n_tile = tile / args.m_tiles, m_tile = tile % args.m_tiles;
  const size_t piece = (size_t)WN * MB * 2 * 4 * 64;
  const floatx4* p = (const floatx4*)args.partials + (size_t)tile * args.slices * piece +
                     (size_t)wn * MB * 2 * 4 * 64 + lane;
  floatx4 v[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
  for (uint32_t s0 = 0; s0 < args.slices; s0 += 4) {
    floatx4 t[4][2];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const size_t s = min(s0 + k, args.slices - 1);
#pragma unroll
      for (int j = 0; j < 2; ++j) t[k][j] = p[s * piece + ((m * 2 + j) * 4 + q) * 64];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (s0 + k < args.slices) {
        v[0] += t[k][0];
        v[1] += t[k][1];
      }
  }
  bool pair;
  uint32_t n_first;
  const Q4Job& jb = tile_job(args, n_tile, &pair, &n_first);
  const uint32_t n0 = n_first + (pair ? 32 : 64) * wn + (lane & 31), n1 = pair ? n0 : n0 + 32;
  store_quad(jb, pair, args.M, (m_tile * MB + m) * 32 + 8 * q + 4 * (lane >> 5), n0, n1, v[0], v[1]);
}

struct RowsPlan {
  uint32_t mb, m_tiles, tiles, slices;
};

uint32_t job_tiles(const Q4Job& j) {
  constexpr uint32_t kPlain = 64 * WN;
  const uint32_t rows = j.mode == kQ4OutSwiglu ? kPlain / 2 : kPlain;
  return (j.rows + rows - 1) / rows;
}

// K slices: workgroups run in rounds of one per CU, at about 4.6, 4.8 or 5.9 us
// a unit (eight groups) with one to three row blocks and 3 us to start and end;
// slices cost a launch and their fp32 tiles' traffic.
RowsPlan rows_plan(const Q4Job* jobs, int n_jobs, uint32_t K, uint32_t M, const Tuning& tune) {
  RowsPlan p{};
  const uint32_t blocks = (M + 31) / 32, units = (K / 64 + kUnitGroups - 1) / kUnitGroups;
  const uint32_t cus = tune.cus > 0 ? (uint32_t)tune.cus : 256;
  p.m_tiles = (blocks + kMaxBlocks - 1) / kMaxBlocks;
  p.mb = (blocks + p.m_tiles - 1) / p.m_tiles;
  uint32_t n_tiles = 0;
  for (int i = 0; i < n_jobs; ++i) n_tiles += job_tiles(jobs[i]);
  p.tiles = n_tiles * p.m_tiles;
  const double unit_us = p.mb == 1 ? 4.6 : p.mb == 2 ? 4.8 : 5.9;
  double best = 0.0;
  for (uint32_t s = 1; s <= std::min(units, 16u); ++s) {
    const double rounds = (double)(((uint64_t)p.tiles * s + cus - 1) / cus);
    const double us =
        rounds * ((units + s - 1) / s * unit_us + 3.0) + (s > 1 ? 3.0 + 0.006 * p.tiles * s * p.mb : 0.0);
    if (p.slices == 0 || us < best) {
      best = us;
      p.slices = s;
    }
  }
  if (tune.rows_slices > 0) p.slices = std::min<uint32_t>(units, (uint32_t)tune.rows_slices);
  return p;
}

// The plan's time (median error 5 % over the calls that q4_gemm_us names).
double rows_us(const RowsPlan& p, uint32_t K, uint32_t cus) {
  const uint32_t units = (K / 64 + kUnitGroups - 1) / kUnitGroups, wgs = p.tiles * p.slices;
  const double work = (units + p.slices - 1) / p.slices * (p.mb == 1 ? 2.8 : p.mb == 2 ? 3.7 : 5.1);
  auto round = [&](double n) { return work * (0.81 + 0.19 * wave_fill(n, cus)) + 7.4; };
  double us = 6.7 + wgs / cus * round(cus);
  if (wgs % cus) us += round(wgs % cus);
  return p.slices > 1 ? us + 0.6 + 0.003 * wgs * p.mb : us;
}

template <int MB>
void launch_rows(const RowsArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(q4_rows_kernel<MB>, dim3(a.tiles * a.slices), dim3(64 * WN * WK), 0, st, a);
  if (a.slices > 1) hipLaunchKernelGGL(q4_rows_reduce_kernel<MB>, dim3(a.tiles * WN * MB), dim3(256), 0, st, a);
}

}  // namespace

bool q4_rows_supported(const Q4Job* jobs, int n_jobs, uint32_t K, uint32_t M, const Tuning& tune) {
  // A forced GEMM plan is for the GEMM.
  if (M <= 16 || K % (64 * WK) != 0 || tune.rows_max <= 16 || tune.gemm_splits > 0 || tune.gemm_q > 0) return false;
  if (M <= (uint32_t)tune.rows_max && tune.rows_slices > 0) return true;
  // While the tiles run in one round of the CUs, whatever the rows (4096 -> 4096
  // at 512 rows: 46 us against the GEMM's 57).
  const RowsPlan p = rows_plan(jobs, n_jobs, K, M, tune);
  const uint32_t cus = tune.cus > 0 ? (uint32_t)tune.cus : 256;
  if (p.tiles <= cus) return true;
  if (M > (uint32_t)tune.rows_max) return false;
  // Past that the tiles cross a round at other rows than the GEMM's (5120 -> 2 x
  // 17408: 108 us against 151 at 192 rows, 165 against 151 at 256, 167 against
  // 214 at 288; 1024 -> 65536: 45 each at 128, 80 against 46 at 224), so the
  // estimates decide.  A tenth in this kernel's favour is the best line over the
  // calls that q4_gemm_us names: up to 384 rows on average 0.1 % above the
  // faster of the two (2.4 % with this kernel always).
  return rows_us(p, K, cus) <= 1.1 * q4_gemm_us(jobs, n_jobs, K, M, tune);
}

void q4_rows_workspace(const Q4Job* jobs, int n_jobs, uint32_t K, uint32_t M, const Tuning& tune,
                       size_t* partial_bytes, size_t* xt_bytes) {
  const RowsPlan p = rows_plan(jobs, n_jobs, K, M, tune);
  *partial_bytes = p.slices > 1 ? (size_t)p.tiles * p.slices * p.mb * 32 * 64 * WN * sizeof(float) : 0;
  *xt_bytes = (size_t)p.m_tiles * (K / 64) * 4096 * p.mb;
}

hipError_t launch_q4_rows(const Q4Job* jobs, int n_jobs, const uint16_t* x, uint32_t K, uint32_t M,
                          const Workspace& ws, hipStream_t stream) {
  if (n_jobs < 1 || n_jobs > kMaxQ4Jobs || !ws.tune || !q4_rows_supported(jobs, n_jobs, K, M, *ws.tune))
    return hipErrorInvalidValue;
  for (int i = 0; i < n_jobs; ++i)
    if (jobs[i].mode != kQ4OutBf16 && jobs[i].mode != kQ4OutSwiglu) return hipErrorInvalidValue;
  const RowsPlan p = rows_plan(jobs, n_jobs, K, M, *ws.tune);
  size_t pbytes, xbytes;
  q4_rows_workspace(jobs, n_jobs, K, M, *ws.tune, &pbytes, &xbytes);
  if (!ws.xh || ws.xh_bytes < xbytes || ws.partial_bytes < pbytes) return hipErrorInvalidValue;
  RowsArgs a{};
  a.n_jobs = n_jobs;
  a.xt = ws.xh;
  a.K = K;
  a.M = M;
  a.m_tiles = p.m_tiles;
  a.tiles = p.tiles;
  a.slices = p.slices;
  a.partials = ws.partials;
  uint32_t n_tiles = 0;
  for (int i = 0; i < n_jobs; ++i) {
    a.jobs[i] = jobs[i];
    a.jobs[i].tile_begin = n_tiles;
    n_tiles += job_tiles(jobs[i]);
  }
  const size_t chunks = xbytes / 16;
  hipLaunchKernelGGL(x_rows_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, stream, x, ws.xh, K, M,
                     p.mb, chunks);
  switch (p.mb) {
    case 1: launch_rows<1>(a, stream); break;
    case 2: launch_rows<2>(a, stream); break;
    default: launch_rows<3>(a, stream); break;
  }
  return hipGetLastError();
}

}  // namespace qm
