// Prefill GEMM: tiles of at most 64 rows (dense; 80 in the expert-major merged
// list) x 256 weight columns (128 of gate and 128 of up), one block of 4 waves
// each, two blocks per CU; x 128 columns where that would leave the chip idle.
//
// What bounds it is the vector L1: a load whose neighbouring lanes read
// different weight rows (an MFMA operand's own layout: lane = column) costs
// one tag access per lane, 64 a load, and with weights and scales loaded that
// way the L1 was busy 93 % of the cycles. So every operand comes in by direct
// global -> LDS loads whose lanes run along k (4 lanes of 16 bytes per weight
// row and k-step), and the operand layout is made by the LDS read, of which
// there is plenty: an A fragment feeds TILES MFMAs.
// Measured in turn (us a call, before: the 8-wave kernels with weights loaded
// straight into registers): 2048 x 2304 x 12288 at G = 128 141 -> 121 (960
// TFLOP/s, MFMA 44 % and VALU 37 % of the SIMD cycles at 2.04 GHz), 1500 x 4096
// x 2304 at G = 32 152 -> 63, 333 x 2304 x 9216 MXFP4 on fp16 rows 111 -> 19, the
// MoE block of 2048 tokens at G = 128 466 -> 428, of 777 tokens at G = 32 (with
// its router) 1239 -> 409. At groups of 32 no unit is full at 1500 rows (VALU
// 30 %, LDS 29 %, MFMA 17 % of the cycles, 1.3 waves per SIMD): each k-step waits
// for the loads of the next, with few waves to fill the time. At 777 tokens the
// gate/up launch fetches 1.8 times its banks, at 4.7 TB/s.
// A k-step is 128 of k. The loads of step s + 1 are issued while step s
// computes; a wait and one barrier a step publish the next stage.

#include <algorithm>

#include "lk_gemm.hpp"
#include "tile_gemm.hpp"

namespace lk {
namespace {

constexpr int W = 4;  // waves per block

// Rows of the highest tile: the expert-major list joins an expert's last tile
// of at most 16 rows to the 64-row tile before it.
constexpr int tg_rows(bool dense) { return dense ? kTileRows : kTileRows + 16; }

// One stage in LDS (16-byte units): activations [row][16 slots], their
// -136 * sum(x) (G = 128: one float a row; G = 32, 64: four, one per 32 of k,
// of which G = 64 uses the first of each pair), then per wave its weights
// [16 column tiles][column][4 slots] and its scale dwords [dword][column].
constexpr int kTgRowU4 = 16;
constexpr int kTgStages = 2;
template <int TILES, int FMT, int ROWS>
struct TgStage {
  static constexpr int kRows = ROWS;
  static constexpr int kNegU4 = fmt_is_w4(FMT) ? (fmt_chain(FMT) < 4 ? kRows : kRows / 4) : 0;
  static constexpr int kScaleDwords = FMT == kFmtW4G32 ? 2 : 1;
  static constexpr int kNegAt = kRows * kTgRowU4;
  static constexpr int kWeightAt = kNegAt + kNegU4;
  static constexpr int kWeightU4 = TILES * 64;  // per wave
  static constexpr int kScaleAt = kWeightAt + W * kWeightU4;
  static constexpr int kScaleU4 = kScaleDwords * TILES * 4;  // per wave
  static constexpr int kU4 = kScaleAt + W * kScaleU4;
};

// Codes of output matrix i, chosen by masks: of pick3's branches on these
// pointers the compiler made a copy of all three in scratch memory, stored by
// every block and read back by index (32 bytes a lane of every launch).
__device__ inline const uint8_t* codes_of(const GemmArgs& g, int i) {
  const uint64_t one = -static_cast<uint64_t>(i == 1), two = -static_cast<uint64_t>(i == 2);
  return reinterpret_cast<const uint8_t*>(
      (reinterpret_cast<uint64_t>(g.wp[0]) & ~(one | two)) |
      (reinterpret_cast<uint64_t>(g.wp[1]) & one) | (reinterpret_cast<uint64_t>(g.wp[2]) & two));
}

template <int TILES, int FMT, int MATS, int MT, bool GATHER, bool SCATTER, bool DENSE>
__device__ __forceinline__ void tg_tile(const GemmArgs& g, uint4* const lds, const int expert,
                                        const int row0, const int rows, const int cb,
                                        const int osel) {
  constexpr bool kW4 = fmt_is_w4(FMT);
  constexpr int kChain = kW4 ? fmt_chain(FMT) : 4;
  constexpr bool kInOrder = kW4 && kChain < 4;  // MFMA t takes k = 32 t .. of the step
  constexpr int NT = TILES / MATS;
  constexpr int kBN = W * NT * 16;
  typedef TgStage<TILES, FMT, tg_rows(DENSE)> St;
  constexpr int kRowLoads = MT;  // 4-row loads per wave and k-step
  const int64_t N = g.n, K = g.k;
  // this block's k-steps: all, or the blockIdx.y-th run of a split product
  const int all_steps = static_cast<int>(K >> 7);
  const int first_step = DENSE ? static_cast<int>(blockIdx.y) * g.split_steps : 0;
  const int ksteps = DENSE ? min(g.split_steps, all_steps - first_step) : all_steps;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int jq = lane >> 4;
  const int ln = lane & 15;

  // activation rows of this lane's direct loads: load h fills the 4 rows of
  // block wv + W h (lane L: row + L / 16, slot L % 16); rows past the tile's
  // end read its first row (never stored)
  auto source_row = [&](int m) -> int64_t {
    const int mm = m < rows ? m : 0;
    if constexpr (GATHER) return g.perm[row0 + mm] / static_cast<int32_t>(g.routes);
    return row0 + mm;
  };
  auto swizzle = [](int m) { return kInOrder ? (m & 15) : row_swizzle(m); };
  const u32x4_t rs_a = buffer_rsrc(kW4 ? g.a_pair : g.a, g.a_rows * K * 2);
  uint32_t va[kRowLoads];
#pragma unroll
  for (int h = 0; h < kRowLoads; ++h) {
    const int m = 4 * (wv + W * h) + jq;
    va[h] = static_cast<uint32_t>(source_row(m) * K * 2 + ((ln ^ swizzle(m)) * 16));
  }
  constexpr int kNegBytes = kInOrder ? 16 : 4;  // per row and k-step
  constexpr int kNegRows = St::kRows / W;       // rows per wave
  u32x4_t rs_n = {0u, 0u, 0u, 0u};
  uint32_t vn = 0;
  if constexpr (kW4) {
    rs_n = buffer_rsrc(g.a_neg, g.a_rows * (K / 128) * kNegBytes);
    vn = static_cast<uint32_t>(source_row(kNegRows * wv + min(lane, kNegRows - 1)) * (K / 128) *
                               kNegBytes);
  }
  // weights: 16-column tile i of the wave (matrix i / NT, column tile i % NT).
  // Lane L loads slot L of the tile's 64: column row_swizzle(L / 4), 16-byte
  // chunk (L % 4) ^ (column % 4), so 4 lanes read a column's 64 bytes of the
  // step and the operand reads below are free of bank conflicts.
  const int64_t rowb = K / 2;
  const int64_t spr = K / (kW4 ? fmt_group(FMT) : 32);  // scales per column
  constexpr int kSb = kW4 ? 2 : 1;                      // bytes of one
  auto column = [&](int nt, int c) -> int64_t {
    const int64_t col = static_cast<int64_t>(cb) * kBN + (wv * NT + nt) * 16 + c;
    return col < N ? col : N - 1;
  };
  const int lcol = row_swizzle(lane >> 2);
  u32x4_t rs_w[MATS], rs_s[MATS];
#pragma unroll
  for (int mi = 0; mi < MATS; ++mi) {
    rs_w[mi] = buffer_rsrc(codes_of(g, osel + mi) + expert * g.wstride, N * rowb);
    // (an odd count of scales: the last dword's valid half must not read as
    // zero, so that dword is read whole, 2 bytes past the tensor)
    rs_s[mi] = buffer_rsrc(static_cast<const uint8_t*>(pick3(g.ws, osel + mi)) +
                               expert * g.sstride * kSb,
                           (N * spr * kSb + 3) & ~int64_t{3});
  }
  uint32_t vw[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    vw[nt] = static_cast<uint32_t>(column(nt, lcol) * rowb + ((lane & 3) ^ (lcol & 3)) * 16);
  // scales: lane L loads column L % 16 of the wave's column tile (L / 16) % NT
  // (TILES / MATS tiles; two matrices: one load each, of half the lanes).
  // G = 128: the dword that holds the step's scale, which half depends on the
  // column where its scales start on an odd one.
  const int64_t scol = column((lane >> 4) % NT, ln);
  const uint32_t vs = static_cast<uint32_t>(scol * spr * kSb);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_offset(lds));
  auto load_step = [&](int step_, int stage) {
    const int local = __builtin_amdgcn_readfirstlane(step_);
    // past the last k-step: descriptors of no bytes (zeros, no traffic)
    const bool live = local < ksteps;
    const int step = first_step + local;
    auto only = [&](u32x4_t r) {
      r[2] = live ? r[2] : 0u;
      return r;
    };
    const uint32_t base = lds0 + static_cast<uint32_t>(stage * St::kU4 * 16);
    const uint32_t st = static_cast<uint32_t>(step);
    const u32x4_t ra = only(rs_a);
#pragma unroll
    for (int h = 0; h < kRowLoads; ++h)
      lds_direct16(ra, base + static_cast<uint32_t>((wv + W * h) * 4 * kTgRowU4 * 16), va[h],
                  st * 256u);
    const uint32_t wbase = base + static_cast<uint32_t>((St::kWeightAt + wv * St::kWeightU4) * 16);
    const uint32_t sbase = base + static_cast<uint32_t>((St::kScaleAt + wv * St::kScaleU4) * 16);
#pragma unroll
    for (int mi = 0; mi < MATS; ++mi) {
      const u32x4_t rw = only(rs_w[mi]), rs = only(rs_s[mi]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        lds_direct16(rw, wbase + static_cast<uint32_t>((mi * NT + nt) * 1024), vw[nt], st * 64u);
      if (lane < NT * 16) {
#pragma unroll
        for (int d = 0; d < St::kScaleDwords; ++d) {
          const uint32_t to = sbase + static_cast<uint32_t>(d * TILES * 64 + mi * NT * 64);
          if constexpr (FMT == kFmtW4A16)
            lds_direct4(rs, to, (vs + st * 2u) & ~3u, 0u);
          else
            lds_direct4(rs, to, vs, st * (FMT == kFmtW4G32 ? 8u : 4u) + 4u * d);
        }
      }
    }
    if constexpr (kW4) {
      const u32x4_t rn = only(rs_n);
      const uint32_t nb = base + static_cast<uint32_t>(St::kNegAt * 16 + wv * kNegRows * kNegBytes);
      if (lane < kNegRows) {
        if constexpr (kInOrder) lds_direct16(rn, nb, vn, st * 16u);
        else lds_direct4(rn, nb, vn, st * 4u);
      }
    }
  };

  const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t tot[TILES][MT];  // column tile mi * NT + nt
#pragma unroll
  for (int i = 0; i < TILES; ++i)
#pragma unroll
    for (int ms = 0; ms < MT; ++ms) tot[i][ms] = zero4;

  // LDS slots of this lane's operands: A fragments (row ln of a subtile, MFMA t)
  int slot[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
    slot[t] = ln * kTgRowU4 + ((kInOrder ? 4 * t + jq : 4 * jq + t) ^ swizzle(ln));

  const int wslot = row_swizzle(ln) * 4 + (jq ^ (ln & 3));
  // G = 128: the first scale of each column is the high half of its dword
  [[maybe_unused]] int odd[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) odd[nt] = static_cast<int>(column(nt, ln) * spr) & 1;

  // 80-row tiles whose groups chain MFMAs take the column tiles in two halves,
  // reading the fragments twice: the chains' accumulators of all four do not
  // fit the registers beside the totals
  constexpr int kHalves = MT == 5 && kW4 && kChain > 1 ? 2 : 1;
  auto compute = [&](int step, int stage) {
    const uint4* const a = lds + stage * St::kU4;
    const float* const neg_lds = reinterpret_cast<const float*>(a + St::kNegAt);
    const uint4* const w_lds = a + St::kWeightAt + wv * St::kWeightU4;
    const uint32_t* const s_lds =
        reinterpret_cast<const uint32_t*>(a + St::kScaleAt + wv * St::kScaleU4);
#pragma unroll
    for (int half = 0; half < kHalves; ++half) {
      constexpr int kN = TILES / kHalves;
      uint32_t w[kN][4];
      uint32_t sd[kN][St::kScaleDwords];
#pragma unroll
      for (int i = 0; i < kN; ++i) {
        const int ti = half * kN + i;
        const uint4 v = w_lds[ti * 64 + wslot];
        w[i][0] = v.x;
        w[i][1] = v.y;
        w[i][2] = v.z;
        w[i][3] = v.w;
#pragma unroll
        for (int d = 0; d < St::kScaleDwords; ++d) sd[i][d] = s_lds[d * TILES * 16 + ti * 16 + ln];
        if constexpr (kInOrder) transpose4(w[i]);
      }
      f32x4_t acc[kN][MT];
      f32x4_t neg[MT];  // of the current group: the C rows 4 jq .. + 3 of each subtile
      // fragments one MFMA group ahead of their use
      u32x4_t afn[MT];
      auto read_a = [&](int t) {
#pragma unroll
        for (int ms = 0; ms < MT; ++ms) {
          const uint4 v = a[ms * 16 * kTgRowU4 + slot[t]];
          afn[ms] = u32x4_t{v.x, v.y, v.z, v.w};
        }
      };
      read_a(0);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        u32x4_t af[MT];
#pragma unroll
        for (int ms = 0; ms < MT; ++ms) {
          af[ms] = afn[ms];
          if constexpr (kW4) {
            if (t % kChain == 0) {
              const int r = ms * 16 + jq * 4;
              if constexpr (kInOrder) {
#pragma unroll
                for (int q = 0; q < 4; ++q) neg[ms][q] = neg_lds[(r + q) * 4 + t];
              } else {
                neg[ms] = *reinterpret_cast<const f32x4_t*>(neg_lds + r);
              }
            }
          }
        }
        if (t < 3) read_a(t + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kN; ++i) {
          const int ti = half * kN + i;
          if constexpr (!kW4) {
            const float sc = e8m0_to_f32((sd[i][0] >> (8 * jq)) & 0xFFu);
            if constexpr (FMT == kFmtMxF16) {
              const f16x8_t bv = __builtin_bit_cast(f16x8_t, unpack_fp4x8_f16(w[i][t], sc));
#pragma unroll
              for (int ms = 0; ms < MT; ++ms)
                tot[ti][ms] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(f16x8_t, af[ms]), bv, tot[ti][ms], 0, 0, 0);
            } else {
              const bf16x8_t bv = __builtin_bit_cast(bf16x8_t, unpack_fp4x8_bf16(w[i][t], sc));
#pragma unroll
              for (int ms = 0; ms < MT; ++ms)
                tot[ti][ms] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8_t, af[ms]), bv, tot[ti][ms], 0, 0, 0);
            }
          } else {
            const bf16x8_t bv = unpack_q8(w[i][t]);
            const bool first = t % kChain == 0, last = (t + 1) % kChain == 0;
            float sc;
            if constexpr (kInOrder) {  // the step's scales are pairs of bf16
              const int e = t / kChain;
              const uint32_t sw = sd[i][e >> 1];
              sc = __builtin_bit_cast(float, (e & 1) ? (sw & 0xFFFF0000u) : (sw << 16));
            } else {
              sc = __builtin_bit_cast(float,
                                      (sd[i][0] >> (((odd[ti % NT] ^ (first_step + step)) & 1) * 16)) << 16);
            }
#pragma unroll
            for (int ms = 0; ms < MT; ++ms) {
              acc[i][ms] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  __builtin_bit_cast(bf16x8_t, af[ms]), bv, first ? neg[ms] : acc[i][ms], 0, 0, 0);
              if (last) tot[ti][ms] += sc * acc[i][ms];
            }
          }
        }
      }
    }
  };

  // the stream: step s computes from stage s % 2 while the loads of step s + 1
  // are in flight. The wait is for all of them, so this wave's part of step
  // s + 1 has landed; the barrier publishes it and retires stage s % 2.
  load_step(0, 0);
  wait_vmcnt<0>();
  __syncthreads();
  auto one = [&](int s, int stage) {
    load_step(s + 1, stage ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    compute(s, stage);
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<0>();
    __syncthreads();
  };
  for (int s = 0;;) {
    one(s, 0);
    if (++s >= ksteps) break;
    one(s, 1);
    if (++s >= ksteps) break;
  }
  if constexpr (DENSE && MATS == 1) {
    if (g.part != nullptr) {  // a split product: this run's fp32 sums, [run][row][output][column]
      wait_vmcnt<0>();        // no direct load outlives the block
#pragma unroll
      for (int ms = 0; ms < MT; ++ms)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = ms * 16 + jq * 4 + i;
          if (m >= rows) continue;
          float* const prow = g.part + ((static_cast<int64_t>(blockIdx.y) * g.dense_rows + row0 + m) *
                                            g.outputs + osel) * N;
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            const int64_t col = static_cast<int64_t>(cb) * kBN + (wv * NT + nt) * 16 + ln;
            if (col < N) prow[col] = tot[nt][ms][i];
          }
        }
      return;
    }
  }
  wait_vmcnt<0>();  // the last direct loads (zeros) have written their slots
  __syncthreads();

  // the tile goes through LDS ([row][column], rows padded by 8 values) and out
  // as 16-byte chunks. Gate/up with out_neg: each chunk paired, and the group
  // sums written too (the block's 128 columns; the 16 chunks of a row sit in
  // one 16-lane DPP row), as the down GEMM's direct loads take them.
  constexpr int kPitch = kBN + 8;
  constexpr int kChunks = kBN / 8;
  uint16_t* const out = pick3(g.out, osel);
  uint16_t* const otile = reinterpret_cast<uint16_t*>(lds);
#pragma unroll
  for (int ms = 0; ms < MT; ++ms)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        uint16_t v;
        if constexpr (MATS == 2)
          v = g.act == kActSitu ? situ_bf16(tot[nt][ms][i], tot[NT + nt][ms][i], g.situ_beta,
                                            g.situ_linear_beta)
                                : swiglu_bf16(tot[nt][ms][i], tot[NT + nt][ms][i]);
        else
          v = store_value<FMT>(tot[nt][ms][i]);
        otile[(ms * 16 + jq * 4 + i) * kPitch + (wv * NT + nt) * 16 + ln] = v;
      }
  __syncthreads();
  for (int u = tid; u < MT * 16 * kChunks; u += W * kWave) {
    const int m = u / kChunks, c = u - m * kChunks;
    const uint4 v = *reinterpret_cast<const uint4*>(otile + m * kPitch + c * 8);
    const int64_t c0 = static_cast<int64_t>(cb) * kBN + c * 8;
    const bool live = m < rows && c0 < N;
    if constexpr (DENSE) {
      if (N & 7) {  // rows of any alignment: value by value (uniform)
        const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (m < rows && c0 + q < N)
            out[(row0 + m) * N + c0 + q] = static_cast<uint16_t>(d[q >> 1] >> (16 * (q & 1)));
        continue;
      }
    }
    int64_t orow = row0 + m;
    if constexpr (SCATTER) orow = live ? g.perm[row0 + m] : 0;
    if constexpr (kW4 && MATS == 2) {
      if (g.out_neg) {
        uint32_t q[4];
        pair_x8(v, q);
        const float sx = pair_group_sum<kChain>(v);
        if (live) {
          *reinterpret_cast<uint4*>(out + orow * N + c0) = make_uint4(q[0], q[1], q[2], q[3]);
          if ((c & (4 * kChain - 1)) == 0)
            g.out_neg[(orow * (N / 128) + cb) * (kInOrder ? 4 : 1) + (kInOrder ? c / 4 : 0)] =
                -kCodeOffset * sx;
        }
        continue;
      }
    }
    if (live) *reinterpret_cast<uint4*>(out + orow * N + c0) = v;
  }
}

template <int TILES, int FMT, int MATS, bool GATHER, bool SCATTER, bool DENSE>
__global__ void __launch_bounds__(W * kWave, TILES == 4 ? 2 : 3) tile_gemm_kernel(const GemmArgs g) {
  constexpr int kBN = W * (TILES / MATS) * 16;
  typedef TgStage<TILES, FMT, tg_rows(DENSE)> St;
  __shared__ uint4 lds[kTgStages * St::kU4];
  const int per_tile = g.col_blocks * g.outputs;
  const int id = blockIdx.x;
  int tile, cb_all;
  if (DENSE && per_tile % 8 == 0) {
    // XCD x (block ids are dealt round robin to the 8 XCDs) takes a band of
    // per_tile / 8 column blocks and walks the row tiles with it: the band's
    // weights stay in that XCD's L2
    const int band = per_tile >> 3;
    const int j = id >> 3;
    tile = j / band;
    cb_all = (id & 7) * band + (j - tile * band);
  } else {
    // XCD x takes an eighth of the list, a tile's column blocks together.
    // Schedule modes: whole tiles, consecutive ones, so tiles of one expert
    // meet in one L2 (an even split of the blocks measured 403 against 381 us
    // on the block of 777 tokens). Dense: an even split of the blocks (whole
    // tiles left XCDs idle where the tiles are few: 468 blocks 65 against 44 us).
    const int count = DENSE ? (g.dense_rows + kTileRows - 1) / kTileRows : *g.tile_count;
    const int j = id >> 3;
    if constexpr (DENSE) {
      const int units = count * per_tile, share = (units + 7) >> 3;
      const int unit = (id & 7) * share + j;
      if (j >= share || unit >= units) return;
      tile = unit / per_tile;
      cb_all = unit - tile * per_tile;
    } else {
      const int chunk = (count + 7) >> 3;
      if (j >= chunk * per_tile) return;
      tile = (id & 7) * chunk + j / per_tile;
      cb_all = j % per_tile;
    }
  }
  const int osel = cb_all / g.col_blocks;
  const int cb = cb_all - osel * g.col_blocks;
  int expert, row0, rows;
  if constexpr (DENSE) {
    row0 = tile * kTileRows;
    if (row0 >= g.dense_rows) return;
    rows = min(kTileRows, g.dense_rows - row0);
    expert = 0;
  } else {
    // the descriptor load does not wait for the count (the list holds max_tiles entries)
    const int4 d = reinterpret_cast<const int4*>(g.tiles)[tile];
    if (tile >= *g.tile_count) return;
    expert = __builtin_amdgcn_readfirstlane(d.x);
    row0 = __builtin_amdgcn_readfirstlane(d.y);
    rows = __builtin_amdgcn_readfirstlane(d.z);
  }
  // routes outside the bank produce zero rows (the MoE block routes itself and
  // has none; a guard against reading in front of the bank)
  if (expert < 0) {
    uint16_t* const out = pick3(g.out, osel);
    for (int i = threadIdx.x; i < rows * kBN; i += W * kWave) {
      const int m = i / kBN;
      const int64_t col = static_cast<int64_t>(cb) * kBN + (i - m * kBN);
      if (col < g.n) {
        const int64_t orow = SCATTER ? g.perm[row0 + m] : row0 + m;
        out[orow * g.n + col] = 0;
      }
    }
    return;
  }
  if constexpr (!DENSE) {
    if (rows > 64) {
      tg_tile<TILES, FMT, MATS, 5, GATHER, SCATTER, DENSE>(g, lds, expert, row0, rows, cb, osel);
      return;
    }
  }
  if (rows > 48)
    tg_tile<TILES, FMT, MATS, 4, GATHER, SCATTER, DENSE>(g, lds, expert, row0, rows, cb, osel);
  else if (rows > 32)
    tg_tile<TILES, FMT, MATS, 3, GATHER, SCATTER, DENSE>(g, lds, expert, row0, rows, cb, osel);
  else if (rows > 16)
    tg_tile<TILES, FMT, MATS, 2, GATHER, SCATTER, DENSE>(g, lds, expert, row0, rows, cb, osel);
  else
    tg_tile<TILES, FMT, MATS, 1, GATHER, SCATTER, DENSE>(g, lds, expert, row0, rows, cb, osel);
}

// The runs of a split product added in run order and rounded once: 4 columns a thread.
template <bool F16>
__global__ void __launch_bounds__(256)
tile_reduce_kernel(const float* __restrict__ part, const GemmArgs g, int runs) {
  const int64_t quads = (g.n + 3) / 4;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t ro = gid / quads;  // row * outputs + output
  if (ro >= static_cast<int64_t>(g.dense_rows) * g.outputs) return;
  const int64_t c = (gid - ro * quads) * 4;
  const int64_t row = ro / g.outputs;
  const int osel = static_cast<int>(ro - row * g.outputs);
  const int64_t stride = static_cast<int64_t>(g.dense_rows) * g.outputs * g.n;
  const float* p = part + ro * g.n + c;
  uint16_t* const y = pick3(g.out, osel) + row * g.n + c;
  if ((g.n & 3) == 0) {
    f32x4_t t = *reinterpret_cast<const f32x4_t*>(p);
#pragma unroll 4
    for (int z = 1; z < runs; ++z) t += *reinterpret_cast<const f32x4_t*>(p + z * stride);
    uint32_t v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = store_value<F16 ? kFmtMxF16 : kFmtMxBf16>(t[q]);
    *reinterpret_cast<uint2*>(y) = make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16));
  } else {
    for (int q = 0; q < 4 && c + q < g.n; ++q) {
      float t = p[q];
      for (int z = 1; z < runs; ++z) t += p[z * stride + q];
      y[q] = store_value<F16 ? kFmtMxF16 : kFmtMxBf16>(t);
    }
  }
}

template <int TILES, int FMT, int MATS>
int launch_mode(const GemmArgs& g, Mode mode, dim3 blocks, hipStream_t s) {
  switch (mode) {
    case Mode::Gather:
      if constexpr (MATS == 2 && FMT != kFmtMxF16) {
        tile_gemm_kernel<TILES, FMT, 2, true, false, false><<<blocks, W * kWave, 0, s>>>(g);
        return LK_OK;
      }
      break;
    case Mode::Scatter:
      if constexpr (TILES == 4 && MATS == 1 && FMT != kFmtMxF16) {
        tile_gemm_kernel<TILES, FMT, 1, false, true, false><<<blocks, W * kWave, 0, s>>>(g);
        return LK_OK;
      }
      break;
    case Mode::Dense:
      if constexpr (MATS == 1) {
        tile_gemm_kernel<TILES, FMT, 1, false, false, true><<<blocks, W * kWave, 0, s>>>(g);
        return LK_OK;
      }
      break;
    default: break;
  }
  return fail_arg("tile gemm: unsupported mode");
}

template <int TILES, int MATS>
int launch_fmt(int fmt, const GemmArgs& g, Mode mode, dim3 blocks, hipStream_t s) {
  switch (fmt) {
    case kFmtW4A16: return launch_mode<TILES, kFmtW4A16, MATS>(g, mode, blocks, s);
    case kFmtW4G32: return launch_mode<TILES, kFmtW4G32, MATS>(g, mode, blocks, s);
    case kFmtW4G64: return launch_mode<TILES, kFmtW4G64, MATS>(g, mode, blocks, s);
    case kFmtMxBf16: return launch_mode<TILES, kFmtMxBf16, MATS>(g, mode, blocks, s);
    case kFmtMxF16: return launch_mode<TILES, kFmtMxF16, MATS>(g, mode, blocks, s);
    default: return fail_arg("tile gemm: unsupported format");
  }
}

}  // namespace

namespace {

// Column blocks and k-split of a dense product of m rows. 256-column blocks
// where they fill their rounds of 512 (two fit a CU), else 128-column ones
// (three fit a CU, and their partial rounds cost less): r = blocks / 512,
// 256 against 128 columns in us: r = 0.7 40.9 : 38.9, 0.91 44.3 : 49.5, 1.13
// 64.5 : 56.7, 1.5 65 : 69, 1.97 80.6 : 87, 2.25 101.9 : 100.2, 3 118 : 129
// (k = 2304, G = 128); 333 x 2304 x 9216 MXFP4 (0.42) 25.3 : 19.4.
// K goes in runs of at least kTgRunSteps k-steps where even 128-column blocks
// leave CUs idle. Estimated microseconds, fitted to measurements at 16
// to 1500 rows: a k-step of one block alone on its CU takes 0.65 + 0.17 a
// 16-row subtile (MXFP4: 0.35 + 0.1), 0.6 of that more for each further block
// on the CU; runs cost the reduce launch (5, with its launch on the host) and
// their fp32 sums written and read at 6 TB/s; a split has to gain kTgGain.
// 64 x 9216 -> 2304 at G = 32: 32 us in 8 runs against 70; 1000 rows 97
// against 126; 200 x 2304 -> 9216 stays whole (31.4 against 34.2).
// At G = 128 (one closing FMA per four MFMAs) 256-column blocks split too, into
// at most kTgWideRuns runs of at least kTgWideRunSteps, where all of them are
// resident: estimated
// at 1.55 of a 128-column block's step, 0.55 of that for each further one, and
// taken where that is kTgWideGain of the other estimate. 9216 -> 2304, us, the
// 8-wave kernel before, 128 columns, these: 1100 rows 87, 93, 74; 1200 rows
// 89, 96, 90; 1400 rows 92, 99, 94; 2048 x 8192 -> 1024 74 against 61. Of 184
// products of 16 to 4096 rows it changed 20: 0.79 to 1.05 of the time. At
// groups of 32 and 64 the same estimate lost up to 16 % on some.
constexpr double kTgWideSlots = 512.0;
constexpr int64_t kTgRunSteps = 4;
// shorter products stay whole (little to gain, and their outputs stay the
// bits of the kernels without a workspace)
constexpr int64_t kTgSplitSteps = 24;
constexpr int64_t kTgMaxRuns = 16;
constexpr double kTgGain = 6.0;
constexpr int64_t kTgWideRunSteps = 16;
constexpr int64_t kTgWideRuns = 4;  // eight lost up to 6 % at 16384 -> 512
constexpr double kTgWideGain = 0.95;

struct DensePlan {
  bool narrow;
  int64_t steps, runs;  // k-steps per run, runs
};

DensePlan dense_plan(int fmt, int64_t m, int64_t n, int64_t k, int64_t outputs, bool may_split) {
  const int64_t tiles = (m + kTileRows - 1) / kTileRows, ksteps = k / 128;
  const double r = static_cast<double>(tiles * ((n + 255) / 256) * outputs) / kTgWideSlots;
  const double part = r - static_cast<double>(static_cast<int64_t>(r));
  const bool mx = !fmt_is_w4(fmt);
  const bool wide = r >= 3.0 || (r >= 0.8 && (part == 0.0 || part >= 0.4));
  DensePlan p{!wide, ksteps, 1};
  if (!p.narrow || !may_split || ksteps < kTgSplitSteps) return p;
  const double blocks = static_cast<double>(tiles * ((n + 127) / 128) * outputs);
  const double wide_blocks = static_cast<double>(tiles * ((n + 255) / 256) * outputs);
  const double subtiles = static_cast<double>((std::min<int64_t>(m, kTileRows) + 15) / 16);
  const double step = mx ? 0.35 + 0.1 * subtiles : 0.65 + 0.17 * subtiles;
  auto estimate_of = [&](double count, double one, double further, int64_t steps, int64_t runs) {
    const double per_cu = std::max(1.0, count * runs / 256.0);
    const double sums = runs > 1 ? 5.0 + 8e-6 / 6.0 * runs * m * n * outputs : 0.0;
    return steps * one * (1.0 + further * (per_cu - 1.0)) + sums;
  };
  auto estimate = [&](int64_t steps, int64_t runs) {
    return estimate_of(blocks, step, 0.6, steps, runs);
  };
  double best = estimate(ksteps, 1) - kTgGain;
  for (int64_t want = 2; want <= std::min(ksteps / kTgRunSteps, kTgMaxRuns); ++want) {
    const int64_t steps = (ksteps + want - 1) / want, runs = (ksteps + steps - 1) / steps;
    const double t = estimate(steps, runs);
    if (t < best) {
      best = t;
      p.steps = steps;
      p.runs = runs;
    }
  }
  if (fmt != kFmtW4A16) return p;
  double most = best * kTgWideGain;
  for (int64_t want = 2; want <= std::min(ksteps / kTgWideRunSteps, kTgWideRuns); ++want) {
    const int64_t steps = (ksteps + want - 1) / want, runs = (ksteps + steps - 1) / steps;
    if (wide_blocks * runs > kTgWideSlots) break;
    const double t = estimate_of(wide_blocks, 1.55 * step, 0.55, steps, runs);
    if (t < most) {
      most = t;
      p = {false, steps, runs};
    }
  }
  return p;
}

}  // namespace

int64_t tile_gemm_split_bytes(int fmt, int64_t m, int64_t n, int64_t k, int64_t outputs) {
  const DensePlan p = dense_plan(fmt, m, n, k, outputs, true);
  return p.runs > 1 ? p.runs * m * n * outputs * 4 : 0;
}

int tile_gemm_launch(int fmt, int mats, GemmArgs g, Mode mode, int64_t tiles, hipStream_t s,
                     const char* what) {
  const bool dense = mode == Mode::Dense;
  const bool split = dense && g.part != nullptr;
  const DensePlan plan = dense ? dense_plan(fmt, g.dense_rows, g.n, g.k, g.outputs, split)
                               : DensePlan{false, g.k / 128, 1};
  if (plan.runs == 1) g.part = nullptr;
  g.split_steps = static_cast<int>(plan.steps);
  const int bn = W * ((plan.narrow ? 2 : 4) / mats) * 16;
  g.col_blocks = static_cast<int>((g.n + bn - 1) / bn);
  const int64_t blocks = (tiles + 7) / 8 * 8 * g.col_blocks * g.outputs;
  LK_REQUIRE(blocks > 0 && blocks < (1LL << 31), "%s: too many blocks", what);
  const dim3 nb(static_cast<unsigned>(blocks), static_cast<unsigned>(plan.runs));
  if (int rc = mats == 2     ? launch_fmt<4, 2>(fmt, g, mode, nb, s)
               : plan.narrow ? launch_fmt<2, 1>(fmt, g, mode, nb, s)
                             : launch_fmt<4, 1>(fmt, g, mode, nb, s))
    return rc;
  if (int rc = check_launch(what)) return rc;
  if (plan.runs == 1) return LK_OK;
  const int64_t work = static_cast<int64_t>(g.dense_rows) * g.outputs * ((g.n + 3) / 4);
  auto* reduce = fmt == kFmtMxF16 ? &tile_reduce_kernel<true> : &tile_reduce_kernel<false>;
  reduce<<<static_cast<unsigned>((work + 255) / 256), 256, 0, s>>>(g.part, g,
                                                                   static_cast<int>(plan.runs));
  return check_launch(what);
}

}  // namespace lk
