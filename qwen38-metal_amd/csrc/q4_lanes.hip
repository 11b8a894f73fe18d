// Q4 projection of a few activation rows (up to 16): concurrent decode lanes or
// drafted tokens.  HBM-bound: Y[M][N] = X[M][K] * W^T with the decode kernels'
// arithmetic, exact weights and fp32 scales: per group of 64,
//   y += s * sum (128 + q) x  +  (b - 128 s) * sum x
// with the sums on bf16 MFMA (128 + q is exact in bf16) in fp32.
//
// The weights stream through LDS as in q4_rows.hip: a tile is 192 W rows, a
// workgroup twelve waves as 3 (64 W rows each) x 4 (K parts), a round one group
// for each K part, so the DMA reads 128 contiguous bytes (a cache line) of
// every W row; the slots are swizzled so that the reads that give every lane
// the two words of its column keep off each other's banks.  (Reading the words
// into registers in load order takes a transpose through LDS in every wave.)
// X rows are DMAed beside them, 16 bytes a lane in MFMA operand order, and the
// scales and biases of a unit of two rounds; the group sums of X come from an
// MFMA against ones.  Every load is a DMA: a table loaded to registers and
// stored to LDS waits, loads retiring in order, for every weight load before it
// (the set below 42 us).
//
// Measured: QKV 5120 -> 10240 with the gate/up pair 5120 -> 2 x 17408, one
// launch, 34.5 us at 3 rows and 36.2 at 16 (3.8 TB/s; 38 .. 39 on the MFMA
// streaming kernel at 3 and 4 rows, 43 .. 58 on the decode kernel's two launches
// at 5 .. 16).  The DMAs alone take 25 us (5.1 TB/s) and their X and tables 5;
// the rest is the arithmetic, 110 VALU operations a wave and round, that the
// waits on the full memory pipeline do not hide.
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace qm {
namespace {

constexpr int WN = 3, WK = 4, kWaves = WN * WK;
constexpr int kXcds = 8, kUnitGroups = 8;  // groups whose scales are passed together
constexpr uint32_t kTile = 64 * WN;        // W rows of a tile
constexpr int NS = 4;                      // rounds in LDS

struct LanesArgs {
  Q4Job jobs[kMaxQ4Jobs];  // plain projections and gate/up pairs (kQ4OutSwiglu)
  int n_jobs;
  const uint16_t* x;  // bf16 [M][K]
  uint32_t K, M;
  uint32_t tiles, slices;
  float* partials;  // [tile][slice][wave column][16-row block][64 lanes][4]
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

// The tile's job and first row (of the gate, for a pair's 96 + 96 rows).
__device__ __forceinline__ const Q4Job& tile_job(const LanesArgs& args, uint32_t tile, bool* pair, uint32_t* n_first) {
  int jt = 0;
  while (jt + 1 < args.n_jobs && tile >= args.jobs[jt + 1].tile_begin) ++jt;
  const Q4Job& jb = args.jobs[jt];
  *pair = jb.mode == kQ4OutSwiglu;
  *n_first = (tile - jb.tile_begin) * (*pair ? kTile / 2 : kTile);
  return jb;
}

// Rows 4 (lane >> 4) .. + 3 of a wave's four 16-column blocks (a pair: gate
// blocks 0, 1 and their up blocks 2, 3; b0 is the first block given).
__device__ __forceinline__ void store_blocks(const Q4Job& jb, bool pair, uint32_t M, uint32_t n_first, uint32_t wn,
                                             uint32_t lane, uint32_t b, floatx4 v0, floatx4 v2) {
  const uint32_t m0 = 4 * (lane >> 4), n = n_first + (pair ? 32 : 64) * wn + 16 * b + (lane & 15);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (m0 + i >= M) break;
    uint16_t* row = jb.out + (size_t)(m0 + i) * jb.rows;
    if (pair) {
      if (n < jb.rows) row[n] = f32_to_bf16(silu_f(v0[i]) * v2[i]);
    } else {
      if (n < jb.rows) row[n] = f32_to_bf16(v0[i]);
      if (n + 32 < jb.rows) row[n + 32] = f32_to_bf16(v2[i]);
    }
  }
}

__global__ __launch_bounds__(64 * kWaves, 3) void q4_lanes_kernel(LanesArgs args) {
  constexpr uint32_t kW = kTile * 128, kX = WK * 2 * 1024, kStage = kW + kX;
  constexpr uint32_t kTab = kTile * 16, kTabs = 4;  // a unit's scales (or biases), 8 a row; units of them in LDS
  constexpr uint32_t kUnit = kUnitGroups / WK;
  static_assert(kUnit == 2 && kTabs * kUnit >= NS + kUnit + 1, "a unit's tables outlive the loads behind them");
  __shared__ __attribute__((aligned(16))) uint8_t lds[NS * kStage + kTabs * 2 * kTab];

  const uint32_t lane = threadIdx.x & 63, q = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wn = wave % WN, wk = wave / WN;
  const uint32_t K = args.K, G = K / 64, R = G / WK;

  // Workgroups are dealt round-robin to the XCDs; an XCD takes a contiguous run.
  const uint32_t workers = args.tiles * args.slices;
  const uint32_t xcd = blockIdx.x % kXcds, wq = workers / kXcds, wrem = workers % kXcds;
  const uint32_t lw = xcd * wq + min(xcd, wrem) + blockIdx.x / kXcds;
  const uint32_t tile = lw / args.slices, slice = lw % args.slices;
  const uint32_t units = (G + kUnitGroups - 1) / kUnitGroups;
  const uint32_t r0 = units * slice / args.slices * kUnit, r1 = min(R, units * (slice + 1) / args.slices * kUnit);

  bool pair;
  uint32_t n_first;
  const Q4Job& jb = tile_job(args, tile, &pair, &n_first);
  const size_t rows_left = jb.rows - n_first;
  const uint32_t last_row = (uint32_t)min(rows_left, (size_t)kTile) - 1;

  // Each wave stages 16 of the 192 rows (a pair: rows 96.. are the up rows), 8
  // rows a DMA; 16-byte piece p of staged row r lies in slot 8 r + (p ^ swz(r)).
  auto swz = [](uint32_t row) { return (row >> 1) & 7; };
  const bool w_up = pair && wave * 16 >= kTile / 2;
  const __amdgpu_buffer_rsrc_t rw =
      make_rsrc((w_up ? jb.uw : jb.w) + (size_t)n_first * (K / 8), rows_left * (K / 2));
  uint32_t w_off[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t row = wave * 16 + k * 8 + (lane >> 3), p = (lane & 7) ^ swz(row);
    w_off[k] = min(w_up ? row - kTile / 2 : row, last_row) * (K / 2) + 16 * p;
  }
  // Waves 0..7 stage X: operand t = wave & 1 of K part wave / 2, lane (row, q)
  // the chunk 2 q + t of its group (rows past M repeat the last one).
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(args.x, (uint64_t)args.M * K * 2);
  const uint32_t x_off = min(lane & 15, args.M - 1) * K * 2 + 128 * (wave >> 1) + 16 * (2 * q + (wave & 1));
  // Waves 8..10 stage the scales and biases of 64 rows each, 16 bytes (a unit's
  // eight) a row: a round brings the scales (even) or biases (odd) of the unit
  // after its own.  A pair's boundary (row 96) lies inside wave 9's rows.
  const uint32_t t_row = 64 * (wave - 8) + lane;
  const bool t_up = pair && t_row >= kTile / 2;
  const uint32_t t_off = min(t_up ? t_row - kTile / 2 : t_row, last_row) * G * 2;
  uint8_t* const tabs = lds + NS * kStage;
  auto tab_load = [&](uint32_t u, bool bias) __attribute__((always_inline)) {
    uint8_t* dst = tabs + (u % kTabs * 2 + (bias ? 1 : 0)) * kTab + (wave - 8) * 1024;
    const uint32_t at = min(u, units - 1) * (2 * kUnitGroups);
    auto from = [&](bool up) __attribute__((always_inline)) {
      const uint16_t* t = bias ? (up ? jb.ub : jb.b) : (up ? jb.us : jb.s);
      dma16(make_rsrc(t + (size_t)n_first * G, rows_left * G * 2), dst, t_off, at);
    };
    if (!pair || wave != 9) {
      from(pair && wave == 10);
    } else {  // lanes 0..31 gate, 32..63 up: the DMA writes the active lanes' slots
      if (lane < 32) from(false);
      if (lane >= 32) from(true);
    }
  };
  auto load = [&](uint32_t r) __attribute__((always_inline)) {
    const uint32_t src = min(r, r1 - 1);
    uint8_t* dst = lds + (r - r0) % NS * kStage;
#pragma unroll
    for (int k = 0; k < 2; ++k) dma16(rw, dst + (wave * 2 + k) * 1024, w_off[k], src * 128);
    if (wave < 8)
      dma16(rx, dst + kW + wave * 1024, x_off, src * (128 * WK));
    else if (wave < 11)
      tab_load(r / kUnit + 1, r % kUnit);
  };

  floatx4 acc[4];
  uint32_t w_rd[4], s_rd[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    const uint32_t row = (pair ? kTile / 2 * (b >> 1) + 32 * wn + 16 * (b & 1) : 64 * wn + 16 * b) + (lane & 15);
    w_rd[b] = 16 * (8 * row + ((2 * wk + (q >> 1)) ^ swz(row))) + 8 * (q & 1);
    s_rd[b] = row * 16 + 2 * wk;
  }
  // A round's operands, read from LDS while the round before it is computed.
  struct Ops {
    u32x4 a[2];
    u32x2 w[4];
    uint16_t s[4], b[4];
  };
  auto read = [&](uint32_t r, Ops& o) __attribute__((always_inline)) {
    const uint8_t* st = lds + (r - r0) % NS * kStage;
    const uint8_t* sp = tabs + r / kUnit % kTabs * 2 * kTab + 2 * WK * (r % kUnit);
    const u32x4* xp = (const u32x4*)(st + kW + wk * 2048) + lane;
    o.a[0] = xp[0];
    o.a[1] = xp[64];
#pragma unroll
    for (int b = 0; b < 4; ++b) o.w[b] = *(const u32x2*)(st + w_rd[b]);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      o.s[b] = *(const uint16_t*)(sp + s_rd[b]);
      o.b[b] = *(const uint16_t*)(sp + kTab + s_rd[b]);
    }
  };
  const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const Ops& o) __attribute__((always_inline)) {
    const u32x4 a0 = interleave_bf16x8(o.a[0]), a1 = interleave_bf16x8(o.a[1]);
    const floatx4 xs = mfma16x16x32(a1, ones, mfma16x16x32(a0, ones, zero));
    floatx4 d[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) d[b] = mfma16x16x32(a0, q4_word_to_bf16x8(o.w[b].x), zero);
#pragma unroll
    for (int b = 0; b < 4; ++b) d[b] = mfma16x16x32(a1, q4_word_to_bf16x8(o.w[b].y), d[b]);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float sc = bf16_to_f32(o.s[b]), off = __builtin_fmaf(-128.0f, sc, bf16_to_f32(o.b[b]));
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[b][e] = __builtin_fmaf(sc, d[b][e], __builtin_fmaf(off, xs[e], acc[b][e]));
    }
  };
  // Loads retire in order: a round's are followed by those of the NS - 2 rounds
  // after it.  Past this every wave's part of the round is in LDS, and every
  // wave has read the round before it.
  auto arrive = [&]() __attribute__((always_inline)) {
    if (wave < 11)
      wait_vmcnt<3 * (NS - 2)>();
    else
      wait_vmcnt<2 * (NS - 2)>();
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
  };

  if (wave >= 8 && wave < 11) {
    tab_load(r0 / kUnit, false);
    tab_load(r0 / kUnit, true);
  }
#pragma unroll
  for (int r = 0; r < NS - 1; ++r) load(r0 + r);
  Ops o[2];
  arrive();
  load(r0 + NS - 1);
  read(r0, o[0]);
  // Computes round r from `cur` while round r + 1 (any past the end) is read
  // into `next`.  The loads come last: a wave stands still while the memory
  // pipeline is full, and the others compute (42 us against 45 with the loads
  // first).
  auto round = [&](uint32_t r, const Ops& cur, Ops& next) __attribute__((always_inline)) {
    arrive();
    read(r + 1, next);
    __builtin_amdgcn_sched_barrier(0);
    compute(cur);
    __builtin_amdgcn_sched_barrier(0);
    load(r + NS);  // into the stage of round r
  };
  for (uint32_t r = r0; r < r1; r += 2) {
    round(r, o[0], o[1]);
    if (r + 1 < r1) round(r + 1, o[1], o[0]);
  }

  // The K parts meet in LDS, which every load has to have left, in K order.
  wait_vmcnt<0>();
  __syncthreads();
  floatx4* red = (floatx4*)lds + (size_t)wn * 4 * 64 + lane;
  if (wk > 0) {
#pragma unroll
    for (int b = 0; b < 4; ++b) red[((size_t)(wk - 1) * WN * 4 + b) * 64] = acc[b];
  }
  __syncthreads();
  if (wk > 0) return;
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int k = 0; k < WK - 1; ++k) acc[b] += red[((size_t)k * WN * 4 + b) * 64];
  if (args.slices > 1) {
    floatx4* po = (floatx4*)args.partials + ((size_t)tile * args.slices + slice) * WN * 4 * 64 + wn * 4 * 64 + lane;
#pragma unroll
    for (int b = 0; b < 4; ++b) po[b * 64] = acc[b];
  } else {
    store_blocks(jb, pair, args.M, n_first, wn, lane, 0, acc[0], acc[2]);
    store_blocks(jb, pair, args.M, n_first, wn, lane, 1, acc[1], acc[3]);
  }
}

// Adds a tile's slices in slice order and runs the epilogue: one workgroup per
// tile and wave column, wave b takes blocks b and b + 2.
__global__ __launch_bounds__(128) void q4_lanes_reduce_kernel(LanesArgs args) {
  const uint32_t lane = threadIdx.x & 63, b = threadIdx.x >> 6;
  const uint32_t tile = blockIdx.x / WN, wn = blockIdx.x % WN;
  const floatx4* p = (const floatx4*)args.partials + ((size_t)tile * args.slices * WN + wn) * 4 * 64 + lane;
  floatx4 v0 = {0.f, 0.f, 0.f, 0.f}, v2 = v0;
  for (uint32_t s0 = 0; s0 < args.slices; s0 += 8) {
    floatx4 t[8][2];
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        t[k][j] = p[((size_t)min(s0 + k, args.slices - 1) * WN * 4 + b + 2 * j) * 64];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (s0 + k < args.slices) {
        v0 += t[k][0];
        v2 += t[k][1];
      }
  }
  bool pair;
  uint32_t n_first;
  const Q4Job& jb = tile_job(args, tile, &pair, &n_first);
  store_blocks(jb, pair, args.M, n_first, wn, lane, b, v0, v2);
}

struct LanesPlan {
  uint32_t tiles, slices;
};

uint32_t job_tiles(const Q4Job& j) {
  const uint32_t rows = j.mode == kQ4OutSwiglu ? kTile / 2 : kTile;
  return (j.rows + rows - 1) / rows;
}

// K slices: workgroups run in rounds of one per CU, at about 3 us a unit (eight
// groups) and 4 us to start and end; slices cost a launch.
LanesPlan lanes_plan(const Q4Job* jobs, int n_jobs, uint32_t K, const Tuning& tune) {
  LanesPlan p{};
  const uint32_t units = (K / 64 + kUnitGroups - 1) / kUnitGroups;
  const uint32_t cus = tune.cus > 0 ? (uint32_t)tune.cus : 256;
  for (int i = 0; i < n_jobs; ++i) p.tiles += job_tiles(jobs[i]);
  double best = 0.0;
  for (uint32_t s = 1; s <= std::min(units, 32u); ++s) {
    const double rounds = (double)(((uint64_t)p.tiles * s + cus - 1) / cus);
    const double us = rounds * ((units + s - 1) / s * 3.0 + 4.0) + (s > 1 ? 3.0 + 0.002 * p.tiles * s : 0.0);
    if (p.slices == 0 || us < best) {
      best = us;
      p.slices = s;
    }
  }
  if (tune.lanes_slices > 0) p.slices = std::min<uint32_t>(units, (uint32_t)tune.lanes_slices);
  return p;
}

// The plan's time, and what the call takes on the other kernels of these rows
// (one MFMA streaming launch, or the decode kernel's: the plain jobs together
// and each pair).  Fitted to 926 calls of 130 shapes (K 512 .. 17408, 16 .. 1444
// tiles): median error 3 %, and 9 and 6 % of the others'.
double lanes_us(const LanesPlan& p, uint32_t K, uint32_t M, uint32_t cus) {
  const uint32_t units = (K / 64 + kUnitGroups - 1) / kUnitGroups, wgs = p.tiles * p.slices;
  const double work = (units + p.slices - 1) / p.slices * 2.6 * (1.0 + 0.0044 * M);
  auto round = [&](uint32_t n) { return work * (0.72 + 0.28 * n / cus) + 4.6; };
  double us = 1.7 + wgs / cus * round(cus);
  if (wgs % cus) us += round(wgs % cus);
  return p.slices > 1 ? us + 3.3 + 0.0032 * wgs : us;
}

struct Others {
  double us;
  int launches;
};
Others others_us(const Q4Job* jobs, int n_jobs, uint32_t K, uint32_t M, const Tuning& tune) {
  double mb = 0.0;  // weights and tables
  int pairs = 0;
  for (int i = 0; i < n_jobs; ++i) {
    const bool pair = jobs[i].mode == kQ4OutSwiglu;
    mb += (double)jobs[i].rows * (pair ? 2 : 1) * K * 0.5625e-6;
    pairs += pair;
  }
  if (tune.q4_mma_lo > 0 && (int)M >= tune.q4_mma_lo && (int)M <= tune.q4_mma_hi)
    return {6.9 + mb / (pairs ? 3.9 : 4.28), 1};
  const bool long_k = tune.q4_mma_k > 0 && K > (uint32_t)tune.q4_mma_k;
  if (long_k && M <= 8) return {24.0 + mb / 3.6, 1};
  const int launches = pairs + (pairs < n_jobs);
  const double rate = (5.1 - 0.105 * M) / (long_k ? 1.49 - 0.03 * ((int)M - 8) : 1.0);
  return {5.6 + 5.1 * (launches - 1) + mb / rate, launches};
}

}  // namespace

bool q4_lanes_supported(const Q4Job* jobs, int n_jobs, uint32_t K, uint32_t M, const Tuning& tune) {
  if (M < (uint32_t)tune.lanes_lo || M > 16 || tune.lanes_lo <= 0 || K % (64 * WK) != 0) return false;
  // A forced plan of another kernel is for that kernel.
  if (tune.q4_nt > 0 || tune.q4_rpw > 0 || tune.q4_split > 0 || tune.q4_mma_c > 0 || !tune.q4_stream) return false;
  for (int i = 0; i < n_jobs; ++i)
    if (jobs[i].mode != kQ4OutBf16 && jobs[i].mode != kQ4OutSwiglu) return false;
  if (tune.lanes_slices > 0) return true;
  const LanesPlan p = lanes_plan(jobs, n_jobs, K, tune);
  const uint64_t cus = tune.cus > 0 ? (uint64_t)tune.cus : 256;
  const Others o = others_us(jobs, n_jobs, K, M, tune);
  // Where the tiles fill half of the CUs the estimates decide: a tile more than
  // a round's costs a round (5120 -> 192 rows a tile at 9 rows: 35 us for 256
  // tiles and 58 for 257, where the decode kernel takes 37 and 38; at 16 rows 37
  // and 60 against 44 and 47), and 5 to 9 rows of a round two thirds full lose
  // too (160 tiles 31 us against 25 .. 27).  On 926 timed calls of 130 shapes the
  // choice is on average 1.7 % above the faster kernel (16.9 with this one always).
  if (2 * (uint64_t)p.tiles >= cus) return lanes_us(p, K, M, (uint32_t)cus) <= 1.05 * o.us;
  // Smaller matrices need slices and their second launch, and the kernels that
  // cut finer stay ahead (4096 -> 4096: 6 .. 9 us against 11; QKV alone 13 .. 15
  // against 16 up to 9 rows) until the decode kernel's time grows with the rows:
  // QKV 17.2 us against 20.0 at 16; down 17408 -> 5120 28 us at 9 rows and 38 at
  // 16, 21 here (up to 8 rows the MFMA streaming kernel takes it in 17 .. 20).
  // One launch of narrow rows stays there (2560 -> 15674 at 12 rows 13 us, 15 here).
  return (M >= 9 && K > 8192 && 16 * (uint64_t)p.tiles >= cus) ||
         (M >= 12 && (K > 3072 || o.launches > 1) && 5 * (uint64_t)p.tiles >= cus);
}

void q4_lanes_workspace(const Q4Job* jobs, int n_jobs, uint32_t K, const Tuning& tune, size_t* partial_bytes) {
  const LanesPlan p = lanes_plan(jobs, n_jobs, K, tune);
  *partial_bytes = p.slices > 1 ? (size_t)p.tiles * p.slices * WN * 4 * 64 * sizeof(floatx4) : 0;
}

hipError_t launch_q4_lanes(const Q4Job* jobs, int n_jobs, const uint16_t* x, uint32_t K, uint32_t M,
                           const Workspace& ws, hipStream_t stream) {
  if (n_jobs < 1 || n_jobs > kMaxQ4Jobs || M == 0 || !ws.tune || !q4_lanes_supported(jobs, n_jobs, K, M, *ws.tune))
    return hipErrorInvalidValue;
  const LanesPlan p = lanes_plan(jobs, n_jobs, K, *ws.tune);
  size_t pbytes;
  q4_lanes_workspace(jobs, n_jobs, K, *ws.tune, &pbytes);
  if (ws.partial_bytes < pbytes) return hipErrorInvalidValue;
  LanesArgs a{};
  a.n_jobs = n_jobs;
  a.x = x;
  a.K = K;
  a.M = M;
  a.tiles = p.tiles;
  a.slices = p.slices;
  a.partials = ws.partials;
  uint32_t tiles = 0;
  for (int i = 0; i < n_jobs; ++i) {
    a.jobs[i] = jobs[i];
    a.jobs[i].tile_begin = tiles;
    tiles += job_tiles(jobs[i]);
  }
  hipLaunchKernelGGL(q4_lanes_kernel, dim3(p.tiles * p.slices), dim3(64 * kWaves), 0, stream, a);
  if (p.slices > 1) hipLaunchKernelGGL(q4_lanes_reduce_kernel, dim3(p.tiles * WN), dim3(128), 0, stream, a);
  return hipGetLastError();
}

}  // namespace qm
