// Shared device code of the matrix-core GEMMs (moe_gemm.hip, tile_gemm.hip):
// the launch arguments, the weight decodes, the direct global -> LDS loads
// and the epilogue arithmetic.

#pragma once

#include "lk_common.hpp"

namespace lk {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kTileRows = 64;  // rows per tile of the prefill GEMMs
constexpr int64_t kMaxDirectBytes = 0xFFFFFFFFll;  // direct-load sources: 32-bit byte offsets

// How a launch finds its rows: gathered through the permutation, scattered
// through it, both, or a dense product.
enum class Mode { Gather, Scatter, GatherScatter, Dense };

// weight format x activation type; kFmtMxF8: MXFP4 weights x activations
// split into fp8 hi + lo with per-32 E8M0 exponents (scaled fp4 MFMA)
// kFmtW4G32 / kFmtW4G64: W4A16 with groups of 32 / 64 on 16-byte weight loads
// (transpose4), in kernels whose kFmtW4A16 form takes G = 128 only
enum : int { kFmtW4A16 = 0, kFmtMxBf16 = 1, kFmtMxF16 = 2, kFmtMxF8 = 3, kFmtW4G32 = 4, kFmtW4G64 = 5 };
constexpr bool fmt_is_w4(int fmt) { return fmt == kFmtW4A16 || fmt == kFmtW4G32 || fmt == kFmtW4G64; }
// group width of the 16-byte-load W4A16 forms, and their MFMAs (32 of k) per group
constexpr int fmt_group(int fmt) { return fmt == kFmtW4G32 ? 32 : fmt == kFmtW4G64 ? 64 : 128; }
constexpr int fmt_chain(int fmt) { return fmt_group(fmt) / 32; }
enum : int { kActSwiglu = 0, kActSitu = 1 };                   // two-matrix epilogues

struct GemmArgs {
  const uint16_t* a;         // activations (bf16, or fp16 for kFmtMxF16), rows of k
  const uint8_t* a_hi;       // kFmtMxF8: fp8 hi codes, rows of k bytes
  const uint8_t* a_lo;       // kFmtMxF8: fp8 lo codes
  const uint16_t* a_sc;      // kFmtMxF8: per-32 exponents, byte 0 hi, byte 1 lo
  // the prefill GEMM (tile_gemm.hip) loads activations into LDS with direct
  // loads: W4A16 from a_pair (rows of a with every 8-value chunk in the weight
  // decode's k order) and a_neg (-136 * sum(x) per row and k-step: one float
  // at G = 128, four at G = 32 and 64), MXFP4 from a. a_rows bounds them.
  const uint16_t* a_pair;
  const float* a_neg;
  int64_t a_rows;
  // W4A16 gate/up on that GEMM: write the activations paired (the down
  // GEMM's a_pair) and their group sums here (its a_neg); null: plain rows
  float* out_neg;
  const int32_t* perm;       // sorted position -> entry (gather / scatter modes)
  const int32_t* tiles;      // [*, 4] tile list (schedule modes)
  const int32_t* tile_count;
  const uint8_t* wp[3];      // packed weights per output matrix (two-matrix: gate, up)
  const void* ws[3];         // scales: bf16 (W4A16) or E8M0 bytes (MXFP4)
  uint16_t* out[3];
  int64_t n, k, group;
  int64_t wstride;           // packed bytes per expert
  int64_t sstride;           // scale elements per expert
  int64_t routes;            // entries per token (gather: token = entry / routes)
  int dense_rows;            // rows of a dense product
  int split_steps;           // dense on the prefill GEMM: k-steps per run (blockIdx.y)
  float* part;               // the runs' fp32 sums (more than one run), else null
  int col_blocks;            // column blocks per output matrix
  int outputs;               // output matrices (3 for fused QKV, else 1)
  int act;                   // two-matrix epilogue (kActSwiglu / kActSitu)
  int tail16;                // 64-row launches: tiles of <= 16 rows take the 16-row path
  float situ_beta, situ_linear_beta;  // SiTU parameters; linear_beta <= 0: none
  // persistent gate/up launches of small batches that route and schedule the
  // batch themselves (no router or schedule launch before them): the
  // router's inputs, the outputs block 0 writes, and the batch
  const float* rt_logits;
  const float* rt_bias;
  int64_t* rt_idx;
  float* rt_w;
  int rt_tokens, rt_routed, rt_top_k, rt_renorm;
  float rt_scaling;
  // nonzero: the selections come from rt_idx (written by the router launch)
  // and the block only ranks them
  int rt_from_idx;
  // where block 0 also writes the schedule (perm, tiles, count) for a later
  // launch of the same block (the split SwiGLU's down GEMM); null: not needed
  int32_t* rt_perm_out;
  int32_t* rt_tiles_out;
  int32_t* rt_count_out;
};

template <typename T>
__device__ inline T pick3(const T (&v)[3], int i) {
  return i == 0 ? v[0] : (i == 1 ? v[1] : v[2]);
}

constexpr int kSub = 4;       // 16-row MFMA subtiles per 64-row tile
constexpr uint32_t kOnesBf16x2 = 0x3F803F80u;  // (1.0, 1.0) in bf16

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef int v8i32_t __attribute__((ext_vector_type(8)));

// ((w ^ 0x88888888) >> 4j) & 0x000F000F | 0x43004300 rewritten as
// ((w >> 4j) & 0x000F000F) ^ 0x43084308: every nibble of the flip is 8 and the
// flipped bit never overlaps the bf16 128.0 bits, so each output is one shift
// and one three-input bit op.
constexpr uint32_t kFlip128 = kBf16_128 | (kNibbleFlip & kPairMask);  // 0x43084308
__device__ inline bf16x8_t unpack_q8(uint32_t w) {
  const u32x4_t v = {(w & kPairMask) ^ kFlip128, ((w >> 4) & kPairMask) ^ kFlip128,
                     ((w >> 8) & kPairMask) ^ kFlip128, ((w >> 12) & kPairMask) ^ kFlip128};
  return __builtin_bit_cast(bf16x8_t, v);
}

// W4A16 groups narrower than a k-step on 16-byte loads: lane block jq = lane / 16
// loads codes 32 jq .. 32 jq + 31 of its column, but an MFMA must stay inside
// one group, so MFMA t takes codes 32 t .. 32 t + 31 and lane block jq needs
// dword jq of block t: a 4 x 4 transpose over (dword, lane block), two
// half-wave swaps and two row swaps. The four dwords loaded apart (and four
// 2-byte scales) are eight loads a k-step instead of two: at 16 tokens of the
// Kimi-Linear layer with G = 32 they held the block to 1.0 TB/s, 416 us with
// its norms and router, against 118 us on the persistent kernel in this form.
__device__ inline void transpose4(uint32_t (&w)[4]) {
  auto half = [](uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  };
  auto row = [](uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  };
  half(w[0], w[2]);
  half(w[1], w[3]);
  row(w[0], w[1]);
  row(w[2], w[3]);
}

// 2**(e - 127) as fp32 for an E8M0 byte (e = 0: the subnormal 2**-127, 255: inf)
__device__ inline float e8m0_to_f32(uint32_t e) {
  return __builtin_bit_cast(float, e == 0u ? 0x00400000u : e << 23);
}

// 8 E2M1 codes (natural order, low nibble first) times 2**(e - 127), exact in
// bf16 / fp16 within range: the gfx950 scaled convert, two codes per byte.
__device__ inline u32x4_t unpack_fp4x8_bf16(uint32_t w, float scale) {
  const u32x4_t v = {
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 0)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 1)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 2)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 3))};
  return v;
}
__device__ inline u32x4_t unpack_fp4x8_f16(uint32_t w, float scale) {
  const u32x4_t v = {
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, scale, 0)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, scale, 1)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, scale, 2)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, scale, 3))};
  return v;
}

// K3's SiTU (engine/kernels/moe_grouped.py:163-178): gate and up rounded to
// bf16 first (they are linear outputs), fp32 math, one rounding at the end.
__device__ inline uint16_t situ_bf16(float gate_acc, float up_acc, float beta, float lbeta) {
  const float g = round_bf16(gate_acc);
  float u = round_bf16(up_acc);
  const float ag = beta * tanhf(g / beta) * (1.0f / (1.0f + expf(-g)));
  if (lbeta > 0.f) u = lbeta * tanhf(u / lbeta);
  return f32_to_bf16(ag * u);
}

// fp32 sum of 8 bf16 activations: four dot2 against (1, 1), exact products
__device__ inline float sum_x8_dot(const uint4 v) {
  float s = dot2_bf16(v.x, kOnesBf16x2, 0.f);
  s = dot2_bf16(v.y, kOnesBf16x2, s);
  s = dot2_bf16(v.z, kOnesBf16x2, s);
  return dot2_bf16(v.w, kOnesBf16x2, s);
}

// The sum of a row's 32-, 64- or 128-wide group (CHAIN = 1, 2, 4 MFMAs) over
// the 16-lane row that holds the row's 16 chunks of a k-step, in every lane
// of the group: the fixed order of every staging, so its bits do not depend
// on which kernel summed it.
template <int CHAIN>
__device__ inline float pair_group_sum(const uint4 v) {
  float s = sum_x8_dot(v);
  if constexpr (CHAIN == 4) {
    s = sum8(s);
    s += dpp_f32<kRowMirror>(s);
  } else {
    s = sum4(s);
    if constexpr (CHAIN == 2) s += dpp_f32<kRowHalfMirror>(s);
  }
  return s;
}

// ---- direct global -> LDS loads (buffer_load ... lds)
// One wave-wide load: lane L's 16 (or 4) bytes at voff + soff of the buffer
// land in LDS at lds + 16 L (4 L); lds and soff are wave-uniform. Issued from
// inline asm so that the compiler does not order LDS reads behind it: the
// caller waits for it (s_waitcnt vmcnt) before the barrier that publishes
// the LDS buffer, and the "memory" clobber keeps the loads issued after it
// in program order (which that vmcnt count relies on).
__device__ inline uint32_t lds_offset(const void* p) {
  return static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)(p)));
}
// raw buffer descriptor of `bytes` bytes at `base` (stride 0; loads at or
// past `bytes` return zeros)
__device__ inline u32x4_t buffer_rsrc(const void* base, int64_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  const uint32_t n = bytes < 0xFFFFFFFFll ? static_cast<uint32_t>(bytes) : 0xFFFFFFFFu;
  return u32x4_t{static_cast<uint32_t>(a), static_cast<uint32_t>(a >> 32) & 0xFFFFu, n,
                 0x00020000u};
}
// The s_nop makes five wait states since the instruction before the block: a
// scalar operand that a vector instruction (v_readfirstlane) has just written
// is not ready for a load before that, and the compiler does not look into
// the block.
__device__ inline u32x4_t uniform_rsrc(u32x4_t r) {
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_readfirstlane(r[i]);
  return r;
}
__device__ inline void lds_direct16(u32x4_t rs, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               ::"s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(uniform_rsrc(rs)),
                 "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory");
}
__device__ inline void lds_direct4(u32x4_t rs, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dword %1, %2, %3 offen lds"
               ::"s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(uniform_rsrc(rs)),
                 "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory");
}

template <int FMT>
__device__ inline uint16_t store_value(float v) {
  if constexpr (FMT == kFmtMxF16) return __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
  else return f32_to_bf16(v);
}

// s_waitcnt vmcnt(N) from inline asm (the compiler does not count the
// direct loads, so it cannot place this wait itself)
template <int N>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N <= 63, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Slot swizzle of row m in the direct-load activation layout: (m & 15) with
// its two 2-bit halves swapped.
__device__ inline int row_swizzle(int m) { return ((m >> 2) & 3) | ((m & 3) << 2); }

}  // namespace lk
