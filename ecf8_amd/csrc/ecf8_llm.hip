// Consumer side of the decode path on gfx950: the block-scaled FP8 linear
// that reads the decoded e4m3fn weights, and the few fused kernels a
// Qwen3-shaped decoder layer needs around it (activation quantization,
// residual + RMSNorm, SiLU gating, per-head norm + rotary embedding + KV
// cache write, split-sequence decode attention).
//
// Numerics follow the fine-grained FP8 scheme of the FP8 checkpoints the
// reference runs (transformers' FP8Linear, used by dfloat/run/run.py's
// DFloatModel for Qwen3-8B-FP8): weights e4m3fn with one fp32 scale per
// 128x128 block, activations quantized on the fly to e4m3fn with one fp32
// scale per row and 128-column group (scale = amax / 448), products
// accumulated in fp32 per 128-column group and scaled by both scales.
//
// Every kernel is deterministic: reductions run in a fixed order, so a
// model decoded from ECF8 and the same model kept in FP8 produce identical
// logits.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "ecf8.h"
#include "ecf8_llm.h"

namespace {

constexpr int kGroup = 128;          // quantization group along K
constexpr float kFp8Max = 448.f;     // largest finite e4m3fn value
constexpr int kHeadDim = 128;
constexpr int kAttnChunk = 256;      // positions per attention workgroup

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Tile layout of FP8 operands (activations always, weights optionally; see
// ecf8_llm.h): per 16 rows and 128-column group one 2 KB block in the
// order the MFMA lanes take their operands -- lane l = 16 g + r holds row
// r's bytes [16 g, +16) at byte 16 l and [64 + 16 g, +16) at 1024 + 16 l,
// so each 16-byte load of a wave covers 1 KB contiguous.
// Byte offset of row m's lane-part (g = 0) of group kg:
__device__ __forceinline__ size_t tile_row_off(int m, int kg, int kgroups) {
  return ((size_t)(m >> 4) * kgroups + kg) * 2048 + (size_t)(m & 15) * 16;
}
// ... and of the 16 bytes [16 c, +16) of the group (c = 0..7):
__device__ __forceinline__ size_t tile_chunk_off(int m, int kg, int kgroups, int c) {
  return tile_row_off(m, kg, kgroups) + (size_t)(c >> 2) * 1024 + (size_t)(c & 3) * 256;
}
// Per-lane base of row m's operand bytes (lane part g), to which a group
// adds kg * 2048 and the second half 1024 more.
__device__ __forceinline__ const uint8_t *tile_lane_base(const uint8_t *p, int m, int kgroups,
                                                         int g) {
  return p + tile_row_off(m, 0, kgroups) + (size_t)g * 256;
}

// 16-byte streaming load (weights are read once per launch)
__device__ __forceinline__ uint4 load_stream16(const uint8_t *p) {
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ float bf16_f32(uint32_t h16) { return __uint_as_float(h16 << 16); }

// fp32 -> bf16, round to nearest even (the rounding torch uses)
__device__ __forceinline__ uint32_t f32_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}

// Four fp32 -> four e4m3fn codes, round to nearest even, with the signs of
// sg; |y| is clamped to 448 first (so is a NaN), the result is always finite
// (callers pass values already scaled into range).  Subnormals (|y| < 2^-6)
// have a step of 2^-9.  The hardware conversion, the same code for every
// fp32 pattern as clamping and rounding the bits by hand.
__device__ __forceinline__ uint32_t f32_e4m3x4(const float (&y)[4], const float (&sg)[4]) {
  float c[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = copysignf(fminf(fabsf(y[i]), kFp8Max), sg[i]);
  const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], lo, true);
}

// Sum over the wave, in every lane: halves, then 16, 8, 4, 2, 1 lanes apart,
// without LDS shuffles (after each step the values repeat with half the
// period, so a row rotation brings the same partner as an exclusive-or).
__device__ __forceinline__ float wave_sum(float v) {
  auto swap = [](uint32_t a, bool half) {
    const auto u = half ? __builtin_amdgcn_permlane32_swap(a, a, false, false)
                        : __builtin_amdgcn_permlane16_swap(a, a, false, false);
    return __uint_as_float(u[0]) + __uint_as_float(u[1]);
  };
  v = swap(__float_as_uint(v), true);
  v = swap(__float_as_uint(v), false);
#define ECF8_DPP_ADD(ctrl)                                                                 \
  v += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), ctrl, \
                                                             0xF, 0xF, true))
  ECF8_DPP_ADD(0x128);  // row_ror:8
  ECF8_DPP_ADD(0x124);  // row_ror:4
  ECF8_DPP_ADD(0x4E);   // quad_perm 2, 3, 0, 1
  ECF8_DPP_ADD(0xB1);   // quad_perm 1, 0, 3, 2
#undef ECF8_DPP_ADD
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

// The largest value of the wave, in every lane, through DPP row shifts and
// broadcasts (VALU latency; each __shfl_xor step is an LDS round trip).
// A lane without a source keeps its own value.
__device__ __forceinline__ float wave_max_dpp(float v) {
#define ECF8_DPP_MAX(ctrl)                                                                  \
  v = fmaxf(v, __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(                       \
                   (int)__float_as_uint(v), (int)__float_as_uint(v), ctrl, 0xF, 0xF, false)))
  ECF8_DPP_MAX(0x111);  // row_shr:1
  ECF8_DPP_MAX(0x112);  // row_shr:2
  ECF8_DPP_MAX(0x114);  // row_shr:4
  ECF8_DPP_MAX(0x118);  // row_shr:8
  ECF8_DPP_MAX(0x142);  // row_bcast:15
  ECF8_DPP_MAX(0x143);  // row_bcast:31
#undef ECF8_DPP_MAX
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), 63));
}

// Quantize 16 consecutive values held by one thread; the 8 threads of a
// 128-column group are 8 consecutive lanes.  Writes 16 e4m3fn bytes and,
// from the group's first thread, the group scale.
__device__ __forceinline__ void quant16(const float (&v)[16], uint8_t *q_out, float *s_out,
                                        bool first_of_group) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  amax = fmaxf(amax, __shfl_xor(amax, 4));
  const float s = amax > 0.f ? amax / kFp8Max : 1.f;
  // v / s, correctly rounded: with r = 1 / s correctly rounded and a quotient
  // within an ulp (q after one correction), q + r (v - q s) is (Markstein
  // 1990); s in this range keeps every quotient of 2^-11 or more (smaller
  // ones round to 0) and its remainder normal.  A zero's sign is lost on the
  // way and taken from v.
  const bool plain = s >= 0x1p-60f && s <= 0x1p60f;
  const float r = 1.f / s;
  uint32_t w[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float q[4], sg[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = v[4 * j + i];
      if (plain) {
        q[i] = x * r;
        q[i] = fmaf(fmaf(-q[i], s, x), r, q[i]);
        q[i] = fmaf(fmaf(-q[i], s, x), r, q[i]);
        sg[i] = x;
      } else {
        q[i] = sg[i] = x / s;
      }
    }
    w[j] = f32_e4m3x4(q, sg);
  }
  *reinterpret_cast<uint4 *>(q_out) = make_uint4(w[0], w[1], w[2], w[3]);
  if (first_of_group) *s_out = s;
}

__device__ __forceinline__ void load16_bf16(const uint16_t *p, float (&v)[16]) {
  const uint4 a = *reinterpret_cast<const uint4 *>(p);
  const uint4 b = *reinterpret_cast<const uint4 *>(p + 8);
  const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v[2 * i] = bf16_f32(w[i] & 0xffffu);
    v[2 * i + 1] = bf16_f32(w[i] >> 16);
  }
}

// ------------------------------------------------------------ FP8 linear

struct LinearSegs {
  const uint8_t *w[ECF8_LINEAR_MAX_SEGS];
  const float *ws[ECF8_LINEAR_MAX_SEGS];
  int n_end[ECF8_LINEAR_MAX_SEGS];  // cumulative output columns
  int col[ECF8_LINEAR_MAX_SEGS];    // first output column of the segment
  int tiled[ECF8_LINEAR_MAX_SEGS];  // weight in the tile layout (else row-major)
  int count;
};

// Buffer resources: a wave-uniform base and extent in scalar registers, so
// a load's address is that base + a scalar offset + one VGPR of 32-bit
// lane offset (a 64-bit address per lane per load would cost the registers
// of a whole batch of loads).  Raw buffer (stride 0); lane offsets at or
// past `bytes` read zero instead of faulting.
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc make_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}
// 16 bytes at lane offset voff + scalar offset soff (kNt: streamed,
// non-temporal -- data read once per launch)
template <bool kNt>
__device__ __forceinline__ uint4 buf_load16(Rsrc r, uint32_t voff, uint32_t soff) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, kNt ? 2 : 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float buf_load_f32(Rsrc r, uint32_t voff, uint32_t soff) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

// A 16-row panel's weight operand for the lane (r, g), in either weight
// layout: the panel's first byte (wave-uniform: n0 is a multiple of 16),
// the lane's 32-bit offset from it (r K + 16 g row-major, 16 l in the tile
// layout), the step between 128-column groups and the offset of the
// group's second half.  A uniform base and a 32-bit lane offset let each
// load take its address from scalar registers plus one VGPR.
struct WeightLane {
  const uint8_t *base;
  uint32_t lane;
  int step, half;
  __device__ __forceinline__ WeightLane(const uint8_t *w, bool tiled, int n0, int r, int g, int K)
      : base(tiled ? w + (size_t)(n0 >> 4) * (size_t)(K / kGroup) * 2048 : w + (size_t)n0 * K),
        lane(tiled ? 16u * (uint32_t)(16 * g + r) : (uint32_t)r * (uint32_t)K + 16u * (uint32_t)g),
        step(tiled ? 2048 : kGroup),
        half(tiled ? 1024 : 64) {}
  __device__ __forceinline__ const uint8_t *at(int kg) const {
    return base + (size_t)kg * step + lane;
  }
  // the panel as a buffer: 16 rows x K bytes in either layout
  __device__ __forceinline__ Rsrc rsrc(int K) const { return make_rsrc(base, 16u * (uint32_t)K); }
  // group kg's two 16-byte halves (kg wave-uniform), streamed
  __device__ __forceinline__ void load(Rsrc r, int kg, uint4 &lo, uint4 &hi) const {
    lo = buf_load16<true>(r, lane, (uint32_t)kg * (uint32_t)step);
    hi = buf_load16<true>(r, lane, (uint32_t)kg * (uint32_t)step + (uint32_t)half);
  }
};

// out[m, col + n] = sum_g (sum_{k in g} aq[m,k] * w[n,k]) * as[m,g] * ws[n/128, g]
//
// ------------------------------------------------ prompt-size GEMM (M > 16)
//
// out[m, col + n] = sum_g (sum_{k in g} aq[m,k] * w[n,k]) * as[m,g] * ws[n/128, g]
// for M > 16: 256 x 256 or 256 x 128 output tiles per workgroup of eight
// waves, one 128-column K group per step through a ring of two or three LDS
// stages.
//
// Every operand block -- 16 rows x one K group, 2 KB -- lands in LDS in
// the tile layout of ecf8_llm.h straight from global memory
// (global_load_lds_dwordx4: each lane's 16 bytes to LDS at 16 x lane, no
// register staging): the tile-layout activations and weights block by
// block, row-major weights gathered into the same order.  The MFMA is
// gfx950's v_mfma_f32_16x16x128_f8f6f4 (one instruction per 16 x 16 tile
// and K group): lane l = 16 g + r feeds it the 32 bytes of row r at block
// bytes 16 l and 1024 + 16 l of both operands -- the same K positions for
// both, so the dot product is that of the group -- and each LDS read is 16
// consecutive bytes per lane (conflict-free).  Each group's product is
// scaled by as[m, g] * ws[n/128, g] and added to the fp32 accumulators in
// group order.  Rows past M read the last valid 16-row block and are never
// stored.  Workgroups are ordered so each XCD (blockIdx.x mod 8) takes a
// contiguous run of tiles, column block by column block: the weight block
// a tile column reads stays in that XCD's L2 across its row blocks.
//
// Two waves share a SIMD.  They take turns, a barrier apart: four waves read
// their operands from LDS while the other four multiply, so the reads hide
// behind the MFMAs instead of all waves doing both in step.  LDS reads bound
// it (an operand is read by each wave that uses it): without the MFMAs a 256
// x 256 tile takes 0.82 of the time, without the loads to LDS 0.86.  Qwen3-8B
// prompt of 2048 rows, us, all waves in step on 256 x 128 tiles before and
// now: gate/up 262 -> 210, q/k/v 80 -> 69, o 47 -> 44, down 118 -> 110; M =
// 4096: gate/up 533 -> 427 (1.93 PFLOP/s), down 256 -> 207.  (The weights'
// operand straight from L2 into registers instead, a phase ahead: 1.1 to 1.3
// times as long.)
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const v2bf v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ void lds_load16(const uint8_t *g, void *lds) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}
__device__ __forceinline__ void lds_load4(const void *g, void *lds) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void *)lds, 4, 0, 0);
}
// Workgroup barrier without a memory fence (a fence on LDS would also wait
// for every stage's loads in flight: they write LDS and are counted by
// vmcnt).  Each wave waits for its own loads of the stage it is about to
// read with an explicit vmcnt first; the empty asm keeps the compiler from
// moving memory operations across the barrier.
__device__ __forceinline__ void gemm_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Workgroup barrier that waits for LDS only (a __syncthreads would also
// wait for the prefetched global loads).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt((0x3F & 15) | (0x3 << 14) | (0x7 << 4) | (0x0 << 8));  // lgkmcnt(0)
  gemm_barrier();
}

// LDS of one wave only: the writes of all its lanes before the reads after.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Waits for this wave's loads of group kg + 1; those of kg + 2 (with three
// stages), issued later, may stay in flight.
template <int kLoads, int kStages>
__device__ __forceinline__ void gemm_wait_loads(int kg, int kgroups) {
  if (kStages == 3 && kg + 2 < kgroups)
    __builtin_amdgcn_s_waitcnt((kLoads & 15) | ((kLoads >> 4) << 14) | (0x7 << 4) | (0xF << 8));
  else
    __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8));  // vmcnt(0)
}

// One load phase's operands from LDS: four A blocks at `a` (and, with kB,
// four B blocks at `b`) and the A rows' scales at `sc`, read and waited for
// in one asm block (no register is in flight past it).
struct GemmOps {
  u32x4 al[4], ah[4];
  float sv[4];
};
__device__ __forceinline__ void gemm_read_a(uint32_t a, uint32_t sc, GemmOps &o) {
  asm volatile(
      "ds_read_b128 %0, %12\n"
      "ds_read_b128 %1, %12 offset:1024\n"
      "ds_read_b128 %2, %12 offset:2048\n"
      "ds_read_b128 %3, %12 offset:3072\n"
      "ds_read_b128 %4, %12 offset:4096\n"
      "ds_read_b128 %5, %12 offset:5120\n"
      "ds_read_b128 %6, %12 offset:6144\n"
      "ds_read_b128 %7, %12 offset:7168\n"
      "ds_read_b32 %8, %13\n"
      "ds_read_b32 %9, %13 offset:64\n"
      "ds_read_b32 %10, %13 offset:128\n"
      "ds_read_b32 %11, %13 offset:192\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(o.al[0]), "=&v"(o.ah[0]), "=&v"(o.al[1]), "=&v"(o.ah[1]), "=&v"(o.al[2]),
        "=&v"(o.ah[2]), "=&v"(o.al[3]), "=&v"(o.ah[3]), "=&v"(o.sv[0]), "=&v"(o.sv[1]),
        "=&v"(o.sv[2]), "=&v"(o.sv[3])
      : "v"(a), "v"(sc)
      : "memory");
}
__device__ __forceinline__ void gemm_read_b(uint32_t b, u32x4 (&bl)[4], u32x4 (&bh)[4]) {
  asm volatile(
      "ds_read_b128 %0, %8\n"
      "ds_read_b128 %1, %8 offset:1024\n"
      "ds_read_b128 %2, %8 offset:2048\n"
      "ds_read_b128 %3, %8 offset:3072\n"
      "ds_read_b128 %4, %8 offset:4096\n"
      "ds_read_b128 %5, %8 offset:5120\n"
      "ds_read_b128 %6, %8 offset:6144\n"
      "ds_read_b128 %7, %8 offset:7168\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(bl[0]), "=&v"(bh[0]), "=&v"(bl[1]), "=&v"(bh[1]), "=&v"(bl[2]), "=&v"(bh[2]),
        "=&v"(bl[3]), "=&v"(bh[3])
      : "v"(b)
      : "memory");
}

__device__ __forceinline__ v8i join32(u32x4 lo, u32x4 hi) {
  return __builtin_shufflevector(__builtin_bit_cast(v4i, lo), __builtin_bit_cast(v4i, hi), 0, 1, 2,
                                 3, 4, 5, 6, 7);
}

// WM x WN = 8 waves of (64 kHalves) x 64 outputs each.
template <int WM, int WN, int kHalves, int kStages>
struct GemmShape {
  static constexpr int kBM = 64 * kHalves * WM, kBN = 64 * WN;
  static constexpr int kABlocks = kBM / 16, kBBlocks = kBN / 16;
  static constexpr int kStageBytes = (kABlocks + kBBlocks) * 2048 + kBM * 4;
  // loads per wave and stage: A and B block halves, and one of scales
  static constexpr int kLoads = 2 * (kABlocks + kBBlocks) / 8 + 1;
  static_assert(WM * WN == 8 && kABlocks % 8 == 0 && kBBlocks % 8 == 0, "blocks deal evenly");
  static_assert(kStages * kStageBytes <= 163840 && kBM % 8 == 0 && kBM <= 512, "LDS");
};

template <int WM, int WN, int kHalves, int kStages>
__global__ __launch_bounds__(512) void fp8_gemm_kernel(
    const uint8_t *__restrict__ aq, const float *__restrict__ as, int M, int K, LinearSegs segs,
    uint16_t *__restrict__ out, int ldo, int n_mb, int n_tiles) {
  using Sh = GemmShape<WM, WN, kHalves, kStages>;
  __shared__ __attribute__((aligned(16))) uint8_t s_ring[kStages * Sh::kStageBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int kgroups = K / kGroup;

  // tile order: XCD x = blockIdx.x % 8 takes tiles [x * per, (x + 1) * per)
  int tile = blockIdx.x;
  const int per = n_tiles / 8;
  if (tile < 8 * per) tile = (tile % 8) * per + tile / 8;
  const int mb = tile % n_mb, nb = tile / n_mb;
  const int m0 = mb * Sh::kBM;

  // each 128-column half of the tile lies in one segment; a wave loads
  // blocks of, and multiplies, one half
  auto segment = [&](int n, const uint8_t *&w, const float *&ws, int &col, int &wt) {
    w = segs.w[0];
    ws = segs.ws[0];
    col = segs.col[0];
    wt = segs.tiled[0];
    int start = 0;
#pragma unroll
    for (int s = 1; s < ECF8_LINEAR_MAX_SEGS; ++s) {
      if (s < segs.count && n >= segs.n_end[s - 1]) {
        w = segs.w[s];
        ws = segs.ws[s];
        col = segs.col[s];
        wt = segs.tiled[s];
        start = segs.n_end[s - 1];
      }
    }
    return n - start;
  };
  const int n_total = segs.n_end[segs.count - 1];
  // loading: wave v fills B blocks v B/8 .. of the tile (columns past the
  // last repeat its last 128)
  constexpr int kNA = Sh::kABlocks / 8, kNB = Sh::kBBlocks / 8;
  const uint8_t *lw;
  const float *lws;
  int lcol, lwt;
  const int ln = min(nb * Sh::kBN + 16 * kNB * wave, n_total - 128 + (16 * kNB * wave) % 128);
  const int ln0 = segment(ln, lw, lws, lcol, lwt);
  // multiplying: the wave's 64 columns
  const uint8_t *mw;
  const float *mws;
  int mcol, mwt;
  const int mn = nb * Sh::kBN + 64 * wn;
  const bool in = mn < n_total;
  const int mn0 = segment(in ? mn : n_total - 64, mw, mws, mcol, mwt);
  typedef const __attribute__((address_space(4))) float ConstF;  // scalar loads
  ConstF *const wsrow = (ConstF *)(mws + (size_t)(mn0 / kGroup) * kgroups);
  const int last_rb = (M + 15) / 16 - 1;  // the last 16-row block of aq
  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)s_ring;

  // group kg into its stage: A blocks, B blocks, A scales (lanes 0 .. of
  // each wave)
  auto issue = [&](int kg) {
    uint8_t *const sa = s_ring + (kg % kStages) * Sh::kStageBytes;
    uint8_t *const sb = sa + Sh::kABlocks * 2048;
    float *const ss = reinterpret_cast<float *>(sb + Sh::kBBlocks * 2048);
#pragma unroll
    for (int h = 0; h < kNA; ++h) {
      const int t = kNA * wave + h;
      const uint8_t *ab = aq + ((size_t)min(m0 / 16 + t, last_rb) * kgroups + kg) * 2048;
      lds_load16(ab + 16 * lane, sa + t * 2048);
      lds_load16(ab + 1024 + 16 * lane, sa + t * 2048 + 1024);
    }
#pragma unroll
    for (int h = 0; h < kNB; ++h) {
      const int t = kNB * wave + h;
      const uint8_t *b0, *b1;
      if (lwt) {
        const uint8_t *bb = lw + ((size_t)(ln0 / 16 + h) * kgroups + kg) * 2048;
        b0 = bb + 16 * lane;
        b1 = bb + 1024 + 16 * lane;
      } else {
        b0 = lw + (size_t)(ln0 + 16 * h + (lane & 15)) * K + kg * kGroup + 16 * (lane >> 4);
        b1 = b0 + 64;
      }
      lds_load16(b0, sb + t * 2048);
      lds_load16(b1, sb + t * 2048 + 1024);
    }
    constexpr int kRows = Sh::kBM / 8;  // rows of scales per wave
    if (lane < kRows) {
      const int row = min(m0 + kRows * wave + lane, M - 1);
      lds_load4(as + (size_t)row * kgroups + kg, ss + kRows * wave);
    }
  };

  v4f acc[kHalves][4][4];
#pragma unroll
  for (int h = 0; h < kHalves; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[h][i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // the lane's LDS offsets in a stage: its A, B and scale reads
  const uint32_t a_off = ring + (uint32_t)(4 * kHalves * wm) * 2048u + 16u * (uint32_t)lane;
  const uint32_t b_off = ring + (uint32_t)(Sh::kABlocks + 4 * wn) * 2048u + 16u * (uint32_t)lane;
  const uint32_t s_off = ring + (uint32_t)(Sh::kABlocks + Sh::kBBlocks) * 2048u +
                         4u * (uint32_t)(64 * kHalves * wm + (lane & 15));

#pragma unroll
  for (int s = 0; s < kStages - 1; ++s)
    if (s < kgroups) issue(s);
  gemm_wait_loads<Sh::kLoads, kStages>(-1, kgroups);
  gemm_barrier();
  if (wave >= 4) gemm_barrier();  // the second four waves run one phase behind
  u32x4 bl[4], bh[4];
  for (int kg = 0; kg < kgroups; ++kg) {
    const uint32_t base = (uint32_t)(kg % kStages) * Sh::kStageBytes;
    const float sw = wsrow[kg];
#pragma unroll
    for (int h = 0; h < kHalves; ++h) {
      // load phase (the other four waves multiply)
      GemmOps o;
      if (h == 0) {
        gemm_read_b(base + b_off, bl, bh);
      }
      gemm_read_a(base + a_off + 8192u * h, base + s_off + 256u * h, o);
      // the stage read in the group before is free: both halves of the waves
      // have passed their last load phase of it
      if (h == 0 && kg + kStages - 1 < kgroups) issue(kg + kStages - 1);
      // before the other four waves' first load phase of the next group, and
      // (below) before this wave's: its own loads of that group are in LDS
      if (h == kHalves - 1 && wave >= 4) gemm_wait_loads<Sh::kLoads, kStages>(kg, kgroups);
      gemm_barrier();
      // multiply phase (the other four waves load)
      // product n, then the sums of product n - 2, which is done by then
      // (the empty asm holds the compiler to this order: with all 16
      // products first, 64 registers more are live)
      v4f d[3];
#pragma unroll
      for (int n = 0; n < 18; ++n) {
        if (n < 16) {
          const v4f z = {0.f, 0.f, 0.f, 0.f};
          // scale operands 0: the unscaled e4m3 x e4m3 form
          d[n % 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
              join32(bl[n % 4], bh[n % 4]), join32(o.al[n / 4], o.ah[n / 4]), z, 0, 0, 0, 0, 0, 0);
        }
        if (n >= 2) {
          const int i = (n - 2) / 4, j = (n - 2) % 4;
          if (j == 0) o.sv[i] *= sw;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            acc[h][i][j][q] = fmaf(d[(n - 2) % 3][q], o.sv[i], acc[h][i][j][q]);
          asm volatile("" : "+v"(acc[h][i][j]));
        }
      }
      if (h == kHalves - 1 && wave < 4) gemm_wait_loads<Sh::kLoads, kStages>(kg, kgroups);
      gemm_barrier();
    }
  }
  if (wave < 4) gemm_barrier();
  if (!in) return;
  // Lane: columns 4 (l / 16) .. + 3 of each 16 x 16 tile, row l % 16.  Every
  // wave is done with the ring (the last barrier): through its own part of
  // it to whole lines, 64 rows of 128 bytes (+ 16: no bank conflicts) at a
  // time.  K = 896, 2048 rows, N = 12288: 40.2 us, with the lanes' own 8-byte
  // stores 47.5.
  const bool whole =
      (((uintptr_t)out | 2u * (uintptr_t)(uint32_t)ldo | 2u * (uintptr_t)(uint32_t)mcol) & 15) == 0;
  constexpr int kRow = 144;
  static_assert(8 * 64 * kRow <= kStages * Sh::kStageBytes, "output tiles fit the ring");
  uint8_t *const st = s_ring + wave * (64 * kRow);
#pragma unroll
  for (int h = 0; h < kHalves; ++h) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const v4f &c = acc[h][i][j];
        *reinterpret_cast<u32x2 *>(st + (16 * i + (lane & 15)) * kRow + 32 * j + 8 * (lane >> 4)) =
            u32x2{pack_bf16(c[0], c[1]), pack_bf16(c[2], c[3])};
      }
    wave_sync();
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int row = 8 * t + (lane >> 3), m = m0 + 64 * kHalves * wm + 64 * h + row;
      const u32x4 v = *reinterpret_cast<const u32x4 *>(st + row * kRow + 16 * (lane & 7));
      if (m < M) {
        uint16_t *o = out + (size_t)m * ldo + mcol + mn0 + 8 * (lane & 7);
        if (whole) {
          *reinterpret_cast<u32x4 *>(o) = v;
        } else {
#pragma unroll
          for (int q = 0; q < 8; ++q) o[q] = (uint16_t)(v[q / 2] >> (16 * (q & 1)));
        }
      }
    }
    wave_sync();
  }
}

// ------------------------------------------ middle form (16 < M, few tiles)
//
// The tile GEMM above has one workgroup per 256 x 128 outputs: a few dozen
// at the row counts of a served batch or a short prompt, most CUs idle.
// Here a workgroup of eight waves computes 16 kCh rows x 16 P columns, and
// wave w multiplies the K groups w, w + 8, ... straight from its registers,
// two of them ahead, so eight waves read a few dozen columns' weights at
// once.  The sums are the tile GEMM's, bit for bit: every eight groups the
// waves put their products into LDS, and each 16 x 16 tile of the strip has
// one wave that adds them to its sums in group order, with that kernel's
// scale and fma.  So a row's result does not depend on how many rows share
// the call (above 16).
//
// P trades the number of workgroups against re-reading the activations per
// column strip (from L2).  The latency of a round bounds it, ~3 us for 128 KB
// of operands at P = 4 (L2) and the products' way through LDS.  MI355X, tile
// layout, us, against the tile GEMM, and against waves that each add a run
// of K (another order, that differs with the row count): 64 rows, N = K =
// 4096 7.6 / 32.5 / 8.4, N = 4096, K = 12288 23.6 / 89.8 / 26.7; 256 rows
// 12.4 / 33.1 / 12.8 and 38.6 / 111 / 33.0; 512 rows 23.6 / 33.5 / 23.8 and
// 67 / 106 / 58.  16 tiles fill one LDS buffer, with two barriers a round and
// two tiles a wave; eight at a time in two buffers took 1.05 to 1.09 times as
// long.
template <int P, int kCh>
__global__ __launch_bounds__(512) void fp8_rows_kernel(const uint8_t *__restrict__ aq,
                                                       const float *__restrict__ as, int M, int K,
                                                       LinearSegs segs, uint16_t *__restrict__ out,
                                                       int ldo) {
  constexpr int kWaves = 8, kTiles = P * kCh;  // 16 x 16 tiles
  constexpr int kPer = (kTiles + kWaves - 1) / kWaves, kBufs = kPer > 1 ? 1 : 2;
  static_assert(kTiles <= kWaves || kTiles % kWaves == 0, "tiles deal evenly");
  // products of a round of eight groups
  __shared__ v4f s_d[kBufs][kWaves][kTiles][64];
  __shared__ float s_sc[2][kWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int kgroups = K / kGroup;
  const int m0 = blockIdx.y * 16 * kCh;

  int n0 = blockIdx.x * 16 * P;
  const uint8_t *w = segs.w[0];
  const float *ws = segs.ws[0];
  int col = segs.col[0], seg_start = 0, wt = segs.tiled[0];
#pragma unroll
  for (int s = 1; s < ECF8_LINEAR_MAX_SEGS; ++s) {
    if (s < segs.count && n0 >= segs.n_end[s - 1]) {
      w = segs.w[s];
      ws = segs.ws[s];
      col = segs.col[s];
      wt = segs.tiled[s];
      seg_start = segs.n_end[s - 1];
    }
  }
  n0 -= seg_start;  // 16 P divides 128, so the strip lies in one segment and scale row
  const float *wsrow = ws + (size_t)(n0 / kGroup) * kgroups;
  const WeightLane wl(w, wt != 0, n0, r, g, K);
  // the strip's 16 P rows x K bytes; panel p starts 16 K bytes after p - 1
  const Rsrc wr = make_rsrc(wl.base, 16u * P * (uint32_t)K);
  const int last_rb = (M + 15) / 16 - 1;  // rows past M read the last 16-row block
  const uint8_t *ab[kCh];
#pragma unroll
  for (int c = 0; c < kCh; ++c)
    ab[c] = aq + (size_t)min(m0 / 16 + c, last_rb) * kgroups * 2048 + 16 * lane;
  const float *asr = as + (size_t)min(m0 + min(lane, 16 * kCh - 1), M - 1) * kgroups;
  const int rounds = (kgroups + kWaves - 1) / kWaves;

  struct Stage {
    u32x4 wv[P][2], av[kCh][2];
    float sa, sw;
  };
  auto load = [&](int rd, Stage &s) {
    const int k = min(kWaves * rd + wave, kgroups - 1);  // past the last: loaded, unused
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const uint32_t at = (uint32_t)k * (uint32_t)wl.step + 16u * (uint32_t)p * (uint32_t)K;
      s.wv[p][0] = __builtin_amdgcn_raw_buffer_load_b128(wr, wl.lane, at, 0);
      s.wv[p][1] = __builtin_amdgcn_raw_buffer_load_b128(wr, wl.lane, at + (uint32_t)wl.half, 0);
    }
#pragma unroll
    for (int c = 0; c < kCh; ++c) {
      s.av[c][0] = *reinterpret_cast<const u32x4 *>(ab[c] + (size_t)k * 2048);
      s.av[c][1] = *reinterpret_cast<const u32x4 *>(ab[c] + (size_t)k * 2048 + 1024);
    }
    s.sa = asr[k];
    s.sw = wsrow[k];
  };
  // wave's tiles: wave + 8 h, tile i being panel i / kCh, rows 16 (i % kCh)..;
  // lane: columns 4 g .. + 3, row r
  v4f acc[kPer];
#pragma unroll
  for (int h = 0; h < kPer; ++h) acc[h] = v4f{0.f, 0.f, 0.f, 0.f};
  auto step = [&](Stage &s, int rd) {
    const int n = min(kWaves, kgroups - kWaves * rd);  // groups of this round
    const int buf = rd & (kBufs - 1);
    if (wave < n) {  // uniform
      s_sc[rd & 1][wave][lane] = s.sa * s.sw;
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int c = 0; c < kCh; ++c) {
          const v4f z = {0.f, 0.f, 0.f, 0.f};
          s_d[buf][wave][p * kCh + c][lane] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
              join32(s.wv[p][0], s.wv[p][1]), join32(s.av[c][0], s.av[c][1]), z, 0, 0, 0, 0, 0, 0);
        }
    }
    if (rd + 2 < rounds) load(rd + 2, s);
    // the products are in LDS; with two buffers the other one (and that of
    // the scales) was last read before every wave's arrival here
    lds_barrier();
    if (wave < kTiles) {  // uniform
      const float *sc = &s_sc[rd & 1][0][16 * (wave % kCh) + r];
      auto add = [&](int v) {
        const float f = sc[64 * v];
#pragma unroll
        for (int h = 0; h < kPer; ++h) {
          const v4f d = s_d[buf][v][wave + kWaves * h][lane];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[h][i] = fmaf(d[i], f, acc[h][i]);
        }
      };
      if (n == kWaves) {  // all reads in flight at once
#pragma unroll
        for (int v = 0; v < kWaves; ++v) add(v);
      } else {
        for (int v = 0; v < n; ++v) add(v);
      }
    }
    if (kBufs == 1) lds_barrier();
  };
  Stage s0, s1;
  load(0, s0);
  if (rounds > 1) load(1, s1);
  for (int rd = 0; rd < rounds; rd += 2) {
    step(s0, rd);
    if (rd + 1 < rounds) step(s1, rd + 1);  // uniform
  }
  if (wave >= kTiles) return;
  const int m = m0 + 16 * (wave % kCh) + r;  // 8 is a multiple of kCh
  if (m >= M) return;
  const bool whole =
      (((uintptr_t)out | 2u * (uintptr_t)(uint32_t)ldo | 2u * (uintptr_t)(uint32_t)col) & 7) == 0;
#pragma unroll
  for (int h = 0; h < kPer; ++h) {
    uint16_t *o = out + (size_t)m * ldo + col + n0 + 16 * ((wave + kWaves * h) / kCh) + 4 * g;
    const u32x2 v = {pack_bf16(acc[h][0], acc[h][1]), pack_bf16(acc[h][2], acc[h][3])};
    if (whole) {
      *reinterpret_cast<u32x2 *>(o) = v;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) o[q] = (uint16_t)(v[q / 2] >> (16 * (q & 1)));
    }
  }
}

// Small-M form (M <= 16, the decode step): one 16-row MFMA tile per
// workgroup of WAVES waves, wave w taking the K groups w, w + WAVES, ... in
// batches of 4 and summing each group with four v_mfma_f32_16x16x32_fp8_fp8:
// lane l = 16 g + r holds row r of both operands, bytes [16 g, +16) and
// [64 + 16 g, +16) of the group -- the 16-byte halves at block bytes 16 l
// and 1024 + 16 l of the tile layout -- so each 16-byte load feeds two
// MFMAs; the K order inside a group is a permutation shared by both
// operands, so the dot product is unchanged.  Every load a batch needs
// (weights from HBM, activations and both scales from L2) is issued before
// its first MFMA, so a batch costs one memory round trip; the loads are
// buffer loads from scalar bases (96 VGPRs for a batch, no spills).  The
// waves' sums meet in LDS and are added in wave order.
template <int WAVES>
__global__ __launch_bounds__(WAVES * 64) void fp8_linear16_kernel(
    const uint8_t *__restrict__ aq, const float *__restrict__ as, int M, int K, LinearSegs segs,
    uint16_t *__restrict__ out, int ldo) {
  static_assert(WAVES >= 4, "the final sums take one thread each of the first 256");
  __shared__ float red[WAVES][4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kgroups = K / kGroup;

  int n0 = blockIdx.x * 16;
  const uint8_t *w = segs.w[0];
  const float *ws = segs.ws[0];
  int col = segs.col[0], seg_start = 0, wt = segs.tiled[0];
#pragma unroll
  for (int s = 1; s < ECF8_LINEAR_MAX_SEGS; ++s) {
    if (s < segs.count && n0 >= segs.n_end[s - 1]) {
      w = segs.w[s];
      ws = segs.ws[s];
      col = segs.col[s];
      wt = segs.tiled[s];
      seg_start = segs.n_end[s - 1];
    }
  }
  n0 -= seg_start;

  const int r = lane & 15, g = lane >> 4;
  const WeightLane wl(w, wt != 0, n0, r, g, K);
  const float *wsrow = ws + (size_t)(n0 / kGroup) * kgroups;
  // An MFMA output row depends on its own A row and scale only, and rows
  // past M are never stored: the pad rows of the tile-layout activations
  // are multiplied as they are, and output rows past M take row M-1's
  // scale (an in-bounds read).
  // buffers: the panel's weights, the first 16-row tile of the
  // activations, their scales (M rows); lane offsets: the lane's activation
  // bytes in a group block, the scale rows it applies
  const Rsrc wr = wl.rsrc(K);
  const Rsrc ar = make_rsrc(aq, (uint32_t)kgroups * 2048u);
  const Rsrc sr = make_rsrc(as, 4u * (uint32_t)M * (uint32_t)kgroups);
  const uint32_t alane = 16u * (uint32_t)lane;
  uint32_t srow[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) srow[i] = 4u * (uint32_t)min(4 * g + i, M - 1) * (uint32_t)kgroups;

  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  constexpr int kU = 4;
  for (int kb = wave; kb < kgroups; kb += WAVES * kU) {
    uint4 wv[kU][2], av[kU][2];
    float wsv[kU], sav[kU][4];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int kg = kb + WAVES * u;
      if (kg < kgroups) {
        wl.load(wr, kg, wv[u][0], wv[u][1]);
        wsv[u] = wsrow[kg];
        av[u][0] = buf_load16<false>(ar, alane, (uint32_t)kg * 2048u);
        av[u][1] = buf_load16<false>(ar, alane, (uint32_t)kg * 2048u + 1024u);
#pragma unroll
        for (int i = 0; i < 4; ++i) sav[u][i] = buf_load_f32(sr, srow[i], 4u * (uint32_t)kg);
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int kg = kb + WAVES * u;
      if (kg >= kgroups) break;
      v4f d = {0.f, 0.f, 0.f, 0.f};
      d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
          (long)(((uint64_t)av[u][0].y << 32) | av[u][0].x),
          (long)(((uint64_t)wv[u][0].y << 32) | wv[u][0].x), d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
          (long)(((uint64_t)av[u][0].w << 32) | av[u][0].z),
          (long)(((uint64_t)wv[u][0].w << 32) | wv[u][0].z), d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
          (long)(((uint64_t)av[u][1].y << 32) | av[u][1].x),
          (long)(((uint64_t)wv[u][1].y << 32) | wv[u][1].x), d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
          (long)(((uint64_t)av[u][1].w << 32) | av[u][1].z),
          (long)(((uint64_t)wv[u][1].w << 32) | wv[u][1].z), d, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(d[i], sav[u][i] * wsv[u], acc[i]);
    }
  }

#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][i][lane] = acc[i];
  __syncthreads();
  if (threadIdx.x < 256) {
    const int i = threadIdx.x >> 6, l = threadIdx.x & 63;
    float sum = 0.f;
#pragma unroll
    for (int wv = 0; wv < WAVES; ++wv) sum += red[wv][i][l];
    const int m = 4 * (l >> 4) + i;
    if (m < M) out[(size_t)m * ldo + col + n0 + (l & 15)] = (uint16_t)f32_bf16(sum);
  }
}

// Persistent small-M form for K = 4096 (32 groups, 4 per wave): each
// workgroup keeps its waves' activation groups and scales in registers and
// walks the 16-column tiles blockIdx.x, + gridDim.x, ...; the next tile's
// weights are loaded while the current tile's MFMAs run.  Used when there
// are more tiles than resident workgroups (the gate/up projection).
template <int WAVES>
__global__ __launch_bounds__(WAVES * 64) void fp8_linear16p_kernel(
    const uint8_t *__restrict__ aq, const float *__restrict__ as, int M, LinearSegs segs,
    uint16_t *__restrict__ out, int ldo, int n_tiles) {
  constexpr int K = 4096, kgroups = K / kGroup, kU = kgroups / WAVES;
  static_assert(WAVES >= 4, "the final sums take one thread each of the first 256");
  __shared__ float red[WAVES][4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const bool row_ok = r < M;

  // this wave's groups: wave, wave + WAVES, ...
  uint4 av[kU][2];
  float sav[kU][4];
  {
    const uint8_t *arow = tile_lane_base(aq, r, kgroups, g);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int kg = wave + WAVES * u;
      av[u][0] = *reinterpret_cast<const uint4 *>(arow + (size_t)kg * 2048);
      av[u][1] = *reinterpret_cast<const uint4 *>(arow + (size_t)kg * 2048 + 1024);
      if (!row_ok) av[u][0] = av[u][1] = make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int mi = 4 * g + i;
        const float v = as[(size_t)(mi < M ? mi : 0) * kgroups + kg];
        sav[u][i] = mi < M ? v : 0.f;
      }
    }
  }

  auto tile_base = [&](int tile, const uint8_t *&w, const float *&ws, int &col, int &n0,
                       int &wt) {
    n0 = tile * 16;
    w = segs.w[0];
    ws = segs.ws[0];
    col = segs.col[0];
    wt = segs.tiled[0];
    int seg_start = 0;
#pragma unroll
    for (int s2 = 1; s2 < ECF8_LINEAR_MAX_SEGS; ++s2) {
      if (s2 < segs.count && n0 >= segs.n_end[s2 - 1]) {
        w = segs.w[s2];
        ws = segs.ws[s2];
        col = segs.col[s2];
        wt = segs.tiled[s2];
        seg_start = segs.n_end[s2 - 1];
      }
    }
    n0 -= seg_start;
  };
  auto load_w = [&](int tile, uint4 (&wv)[kU][2], float (&wsv)[kU]) {
    const uint8_t *w;
    const float *ws;
    int col, n0, wt;
    tile_base(tile, w, ws, col, n0, wt);
    const WeightLane wl(w, wt != 0, n0, r, g, K);
    const Rsrc wr = wl.rsrc(K);
    const float *wsrow = ws + (size_t)(n0 / kGroup) * kgroups;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int kg = wave + WAVES * u;
      wl.load(wr, kg, wv[u][0], wv[u][1]);
      wsv[u] = wsrow[kg];
    }
  };

  uint4 wcur[kU][2], wnxt[kU][2];
  float scur[kU], snxt[kU];
  int tile = blockIdx.x;
  if (tile >= n_tiles) return;  // uniform
  load_w(tile, wcur, scur);
  for (;;) {
    const int next = tile + (int)gridDim.x;
    const bool more = next < n_tiles;  // uniform
    if (more) load_w(next, wnxt, snxt);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      v4f d = {0.f, 0.f, 0.f, 0.f};
      d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
          (long)(((uint64_t)av[u][0].y << 32) | av[u][0].x),
          (long)(((uint64_t)wcur[u][0].y << 32) | wcur[u][0].x), d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
          (long)(((uint64_t)av[u][0].w << 32) | av[u][0].z),
          (long)(((uint64_t)wcur[u][0].w << 32) | wcur[u][0].z), d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
          (long)(((uint64_t)av[u][1].y << 32) | av[u][1].x),
          (long)(((uint64_t)wcur[u][1].y << 32) | wcur[u][1].x), d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
          (long)(((uint64_t)av[u][1].w << 32) | av[u][1].z),
          (long)(((uint64_t)wcur[u][1].w << 32) | wcur[u][1].z), d, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(d[i], sav[u][i] * scur[u], acc[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][i][lane] = acc[i];
    __syncthreads();
    if (threadIdx.x < 256) {
      const int i = threadIdx.x >> 6, l = threadIdx.x & 63;
      float sum = 0.f;
#pragma unroll
      for (int wv2 = 0; wv2 < WAVES; ++wv2) sum += red[wv2][i][l];
      const int m = 4 * (l >> 4) + i;
      const uint8_t *w;
      const float *ws;
      int col, n0, wt;
      tile_base(tile, w, ws, col, n0, wt);
      if (m < M) out[(size_t)m * ldo + col + n0 + (l & 15)] = (uint16_t)f32_bf16(sum);
    }
    if (!more) break;
    __syncthreads();  // red is rewritten by the next tile
    tile = next;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      wcur[u][0] = wnxt[u][0];
      wcur[u][1] = wnxt[u][1];
      scur[u] = snxt[u];
    }
  }
}

// ------------------------------------------------- quantizing row kernels

// residual += x (if x); y = residual * rsqrt(mean(residual^2) + eps) * w;
// y -> bf16 (ob), and/or -> e4m3fn + group scales (oq, os; from the
// bf16-rounded y when both are written).  One workgroup per row of
// K = 16 * kThreads (4096: 256 threads, 2048: 128), 16 values per thread.
template <int kThreads>
__global__ __launch_bounds__(kThreads) void rmsnorm_kernel(const uint16_t *__restrict__ x,
                                                           float *__restrict__ res,
                                                           const uint16_t *__restrict__ w,
                                                           float eps, int K,
                                                           uint8_t *__restrict__ oq,
                                                           float *__restrict__ os,
                                                           uint16_t *__restrict__ ob) {
  static_assert(kThreads == 128 || kThreads == 256, "rows of 2048 or 4096");
  __shared__ float part[kThreads / 64];
  const int m = blockIdx.x, t = threadIdx.x;
  const size_t base = (size_t)m * K + 16 * t;
  float v[16];
  float4 *rp = reinterpret_cast<float4 *>(res + base);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float4 f = rp[j];
    v[4 * j] = f.x;
    v[4 * j + 1] = f.y;
    v[4 * j + 2] = f.z;
    v[4 * j + 3] = f.w;
  }
  if (x) {
    float xv[16];
    load16_bf16(x + base, xv);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] += xv[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) rp[j] = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) ss = fmaf(v[i], v[i], ss);
  ss = wave_sum(ss);
  if ((t & 63) == 0) part[t >> 6] = ss;
  __syncthreads();
  float total;
  if constexpr (kThreads == 256)
    total = (part[0] + part[1]) + (part[2] + part[3]);
  else
    total = part[0] + part[1];
  const float rs = rsqrtf(total / (float)K + eps);
  float wv[16];
  load16_bf16(w + 16 * t, wv);
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = v[i] * rs * wv[i];
  if (ob) {
    uint32_t p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = f32_bf16(v[2 * i]) | (f32_bf16(v[2 * i + 1]) << 16);
    uint4 *op = reinterpret_cast<uint4 *>(ob + base);
    op[0] = make_uint4(p[0], p[1], p[2], p[3]);
    op[1] = make_uint4(p[4], p[5], p[6], p[7]);
    if (oq) {  // both outputs: quantize the bf16-rounded values
      float r[16];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        r[2 * i] = bf16_f32(p[i] & 0xffffu);
        r[2 * i + 1] = bf16_f32(p[i] >> 16);
      }
      quant16(r, oq + tile_chunk_off(m, t >> 3, K / kGroup, t & 7),
              os + (size_t)m * (K / kGroup) + (t >> 3), (t & 7) == 0);
    }
  } else {
    quant16(v, oq + tile_chunk_off(m, t >> 3, K / kGroup, t & 7),
            os + (size_t)m * (K / kGroup) + (t >> 3), (t & 7) == 0);
  }
}

// h = silu(gate) * up over [M, 2I] (gate columns [0, I), up [I, 2I)),
// quantized; grid (ceil(I / 4096), M).  I is a multiple of 128, so the 8
// threads of a group are all inside the row or all past it.
__global__ __launch_bounds__(256) void silu_mul_quant_kernel(const uint16_t *__restrict__ gu, int I,
                                                             uint8_t *__restrict__ oq,
                                                             float *__restrict__ os) {
  const int m = blockIdx.y, e = blockIdx.x * 4096 + 16 * threadIdx.x;
  if (e >= I) return;
  float g[16], u[16];
  load16_bf16(gu + (size_t)m * 2 * I + e, g);
  load16_bf16(gu + (size_t)m * 2 * I + I + e, u);
#pragma unroll
  for (int i = 0; i < 16; ++i) g[i] = g[i] / (1.f + expf(-g[i])) * u[i];
  quant16(g, oq + tile_chunk_off(m, e >> 7, I / kGroup, (e >> 4) & 7),
          os + (size_t)m * (I / kGroup) + (e >> 7), (threadIdx.x & 7) == 0);
}

// plain bf16 -> e4m3fn per 1x128 group; grid (ceil(K / 4096), M), K a
// multiple of 128
__global__ __launch_bounds__(256) void act_quant_kernel(const uint16_t *__restrict__ x, int K,
                                                        uint8_t *__restrict__ oq,
                                                        float *__restrict__ os) {
  const int m = blockIdx.y, e = blockIdx.x * 4096 + 16 * threadIdx.x;
  if (e >= K) return;
  float v[16];
  load16_bf16(x + (size_t)m * K + e, v);
  quant16(v, oq + tile_chunk_off(m, e >> 7, K / kGroup, (e >> 4) & 7),
          os + (size_t)m * (K / kGroup) + (e >> 7), (threadIdx.x & 7) == 0);
}

// --------------------------------------------- per-head norm + rotary + KV

// One wave, one head row of 128 bf16 values (lane l holds dims 2l, 2l+1):
// RMSNorm over the head (bf16 weights nw), then the rotary embedding at
// position p (rotate-half convention, cos/sin tables [Lmax, 64]); returns
// the lane's two results as packed bf16.  The loads are apart from the
// arithmetic, so a kernel can issue them ahead of longer ones.
struct RopeIn {
  uint32_t w2;   // the norm's weights
  float2 c, s;   // the rotary tables at p
};

__device__ __forceinline__ RopeIn rope_load(const uint16_t *__restrict__ nw,
                                            const float *__restrict__ cosv,
                                            const float *__restrict__ sinv, int p, int lane) {
  const int j = (2 * lane) & 63;
  return RopeIn{*reinterpret_cast<const uint32_t *>(nw + 2 * lane),
                make_float2(cosv[p * 64 + j], cosv[p * 64 + j + 1]),
                make_float2(sinv[p * 64 + j], sinv[p * 64 + j + 1])};
}

__device__ __forceinline__ uint32_t norm_rope(uint32_t x2, const RopeIn &in, float eps, int lane) {
  float x0 = bf16_f32(x2 & 0xffffu), x1 = bf16_f32(x2 >> 16);
  const float ss = wave_sum(x0 * x0 + x1 * x1);
  const float rs = rsqrtf(ss / (float)kHeadDim + eps);
  x0 = x0 * rs * bf16_f32(in.w2 & 0xffffu);
  x1 = x1 * rs * bf16_f32(in.w2 >> 16);
  // dims d +- 64 lie in the other half of the wave
  const auto s0 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x0), __float_as_uint(x0), false,
                                                   false);
  const auto s1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x1), __float_as_uint(x1), false,
                                                   false);
  const float y0 = __uint_as_float(lane < 32 ? s0[1] : s0[0]);
  const float y1 = __uint_as_float(lane < 32 ? s1[1] : s1[0]);
  const float sg = lane < 32 ? -1.f : 1.f;
  x0 = x0 * in.c.x + sg * y0 * in.s.x;
  x1 = x1 * in.c.y + sg * y1 * in.s.y;
  return f32_bf16(x0) | (f32_bf16(x1) << 16);
}

// The heads of the fused qkv projection output [B*T, (Hq + 2 Hkv) * 128]: q
// and k heads get RMSNorm over the head (weights qn / kn) and the rotary
// embedding at position pos[0] + t (rotate-half convention, cos/sin tables
// [Lmax, 64]); q goes to q_out [B, Hq, T, 128], k and v to the caches
// [B, Hkv, Lmax, 128].  Workgroup (token, 16 heads), four heads per wave, all
// loaded at once and sharing the token's rotary values.  Loads in
// flight bound it: 50 MB at 2048 tokens of 48 heads in 15.8 us, 3.2 TB/s
// where a copy moves 6.2 (one head per wave 29.5 us).
constexpr int kRopePer = 4;
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(
    const uint16_t *__restrict__ qkv, int T, int Hq, int Hkv, const uint16_t *__restrict__ qn,
    const uint16_t *__restrict__ kn, float eps, const float *__restrict__ cosv,
    const float *__restrict__ sinv, const int *__restrict__ pos, int Lmax,
    uint16_t *__restrict__ q_out, uint16_t *__restrict__ kc, uint16_t *__restrict__ vc) {
  const int lane = threadIdx.x & 63;
  const int H = Hq + 2 * Hkv;
  const int n_hb = (H + 4 * kRopePer - 1) / (4 * kRopePer);
  const int tok = (int)blockIdx.x / n_hb, b = tok / T, t = tok % T;
  const int h0 = ((int)blockIdx.x % n_hb * 4 +
                  __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * kRopePer;
  if (h0 >= H) return;
  const int p = pos[0] + t;
  if (p < 0 || p >= Lmax) return;
  uint32_t x2[kRopePer];
#pragma unroll
  for (int i = 0; i < kRopePer; ++i)
    x2[i] = *reinterpret_cast<const uint32_t *>(
        qkv + ((size_t)tok * H + min(h0 + i, H - 1)) * kHeadDim + 2 * lane);
  RopeIn in = rope_load(h0 < Hq ? qn : kn, cosv, sinv, p, lane);
  const uint32_t wk = *reinterpret_cast<const uint32_t *>(kn + 2 * lane);
#pragma unroll
  for (int i = 0; i < kRopePer; ++i) {
    const int hh = h0 + i;
    if (hh >= H) break;
    uint16_t *dst;
    if (hh < Hq) {
      dst = q_out + (((size_t)b * Hq + hh) * T + t) * kHeadDim;
    } else if (hh < Hq + Hkv) {
      in.w2 = wk;
      dst = kc + (((size_t)b * Hkv + (hh - Hq)) * Lmax + p) * kHeadDim;
    } else {
      dst = vc + (((size_t)b * Hkv + (hh - Hq - Hkv)) * Lmax + p) * kHeadDim;
    }
    *reinterpret_cast<uint32_t *>(dst + 2 * lane) =
        hh >= Hq + Hkv ? x2[i] : norm_rope(x2[i], in, eps, lane);
  }
}

// ------------------------------------------------------ decode attention

// Eight bytes at any dword: a v cache may start at any.
typedef uint32_t u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));

// What the fused form of the split kernel needs besides the caches.
struct AttnFused {
  const uint16_t *qkv;  // [B, (Hq + 2 Hkv) * 128], one new token per sequence
  const uint16_t *qn, *kn;
  float eps;
  const float *cosv, *sinv;
};

// Rows (16 lanes) 0..3 of x and y -> rows x0 + x1, y0 + y1, x2 + x3, y2 + y3.
__device__ __forceinline__ float add_swap16(float x, float y) {
  const auto v = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false,
                                                  false);
  return __uint_as_float(v[0]) + __uint_as_float(v[1]);
}
// -> rows x0 + x2, x1 + x3, y0 + y2, y1 + y3.
__device__ __forceinline__ float add_swap32(float x, float y) {
  const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false,
                                                  false);
  return __uint_as_float(v[0]) + __uint_as_float(v[1]);
}

// Split-sequence attention for one new token per sequence: workgroup
// (b * Hkv + kh, split) handles positions [split*256, +256) of the L =
// pos[0] + 1 cached ones for the G = Hq / Hkv query heads sharing kv head
// kh.  Scores: one lane per position, an FMA chain over the dims; softmax
// partials per head; PV: one thread per (head, dim) and position mod 4.
// Partials go to work: m, l [B*Hq, S] and acc [B*Hq, S, 128].
//
// Eight waves: wave v takes positions 64 (v mod 4).. and half of the heads
// for the scores, half of the dims for PV.  Keys and values are both loaded
// before q is prepared (one round trip); keys go to LDS in coalesced loads,
// 16-byte units exclusive-ored with their row so a lane reads its row
// without conflicts; a wave's sums use permlane swaps and DPP.
//
// kFused: q comes from the projection output through the per-head norm and
// rotary embedding (norm_rope), and the split holding position pos[0] writes
// the new token's k and v to the caches -- the work of qk_norm_rope_kernel,
// in the same arithmetic -- and takes them from LDS.  (Merging the splits in
// the last workgroup to finish would need device-scope fences, which on this
// multi-XCD part write back and invalidate the whole L2: the merge stays a
// kernel of its own.)
//
// HBM-bound for long contexts, the latency of one workgroup for short ones;
// MI355X, 16 sequences, with the merge, us before (each lane loading its own
// key row, values after the softmax, LDS shuffles) and now: 8192 positions
// 142.9 -> 118.4 (8 query heads per KV head 100.5 -> 79.4), 640 19.7 -> 18.8.
// (Scores from MFMAs took 108 and 67, but sum in another order: the FP8
// codes of a decode step then differ from those of the kernel it replaces.)
constexpr int kAttnWaves = 8;

template <int G, bool kFused>
__global__ __launch_bounds__(64 * kAttnWaves) void attn_split_kernel(
    const uint16_t *__restrict__ q, uint16_t *__restrict__ kc, uint16_t *__restrict__ vc,
    const int *__restrict__ pos, int Hkv, int Lmax, int S, float *__restrict__ wm,
    float *__restrict__ wl, float *__restrict__ wacc, AttnFused fu) {
  constexpr int kUnits = kHeadDim / 8;  // 16-byte units of a row
  __shared__ u32x4 s_k[kAttnChunk * kUnits];
  __shared__ __attribute__((aligned(16))) float qs[G][kHeadDim];
  // probability of position 64 w + j: [h][w][16 (j mod 4) + j / 4]
  __shared__ __attribute__((aligned(16))) float pw[G][4][64];
  __shared__ uint32_t s_new[kHeadDim / 2];  // the new token's v
  __shared__ float red[2][G][4];
  // PV partials [position group][head][dim], over the keys once they are read
  float(*part)[G][kHeadDim] = reinterpret_cast<float(*)[G][kHeadDim]>(s_k);
  const int bk = blockIdx.x, split = blockIdx.y;
  const int b = bk / Hkv, kh = bk % Hkv;
  const int Hq = Hkv * G;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int p = pos[0];
  int L = p + 1;
  L = L < 1 ? 1 : (L > Lmax ? Lmax : L);
  const int c0 = split * kAttnChunk;
  const size_t head0 = (size_t)b * Hq + kh * G;
  if (c0 >= L) return;  // the merge reads the splits in use only
  const int n = min(kAttnChunk, L - c0);
  // fused: the new token's position in this chunk; past every position
  // otherwise
  const int fresh = kFused && p >= c0 && p < c0 + kAttnChunk && p < Lmax ? p - c0 : kAttnChunk;
  const float scale = rsqrtf((float)kHeadDim);

  // The wave's head of q and the new token's k or v (the waves past the
  // heads, or the first two): loaded first, since loads return in order and
  // the keys take longest.
  constexpr int kNew = G < 8 ? 4 : 0;  // wave kNew: k, wave kNew + 1: v
  RopeIn qin, nin;
  uint32_t qx = 0, nx = 0;
  if constexpr (kFused) {
    const uint16_t *row = fu.qkv + (size_t)b * (Hq + 2 * Hkv) * kHeadDim + 2 * lane;
    // rotary row (p is in range for a valid call)
    qin = rope_load(fu.qn, fu.cosv, fu.sinv, min(max(p, 0), Lmax - 1), lane);
    nin = qin;
    nin.w2 = *reinterpret_cast<const uint32_t *>(fu.kn + 2 * lane);
    if (wave < G) qx = *reinterpret_cast<const uint32_t *>(row + (size_t)(kh * G + wave) * kHeadDim);
    if (wave == kNew || wave == kNew + 1)
      nx = *reinterpret_cast<const uint32_t *>(row +
                                               (size_t)(Hq + (wave - kNew) * Hkv + kh) * kHeadDim);
  }
  const size_t row0 = ((size_t)b * Hkv + kh) * Lmax + c0;
  const int pg = wave & 3, half = wave >> 2;
  const int dg = lane & 15, rr = lane >> 4;
  u32x4 kr[kAttnChunk * kUnits / 512];
#pragma unroll
  for (int i = 0; i < kAttnChunk * kUnits / 512; ++i) {
    const int row = (t + 512 * i) / kUnits, c = t % kUnits;
    if (row < n)
      kr[i] = *reinterpret_cast<const u32x4 *>(kc + (row0 + row) * kHeadDim + 8 * c);
  }
  // values: positions 64 pg + 4 st + rr, dims 64 half + 4 dg..; positions
  // past n read row n - 1 with weight 0
  u32x2 vv[16];
#pragma unroll
  for (int st = 0; st < 16; ++st)
    vv[st] = *reinterpret_cast<const u32x2a4 *>(
        vc + (row0 + min(64 * pg + 4 * st + rr, n - 1)) * kHeadDim + 64 * half + 4 * dg);

  if constexpr (kFused) {
    if (wave < G) {
      const uint32_t y2 = norm_rope(qx, qin, fu.eps, lane);
      qs[wave][2 * lane] = bf16_f32(y2 & 0xffffu) * scale;
      qs[wave][2 * lane + 1] = bf16_f32(y2 >> 16) * scale;
    }
    if (fresh < kAttnChunk && (wave == kNew || wave == kNew + 1)) {
      const uint32_t y2 = wave == kNew ? norm_rope(nx, nin, fu.eps, lane) : nx;
      uint16_t *cache = wave == kNew ? kc : vc;
      *reinterpret_cast<uint32_t *>(cache + (row0 + fresh) * kHeadDim + 2 * lane) = y2;
      if (wave == kNew)
        reinterpret_cast<uint32_t *>(
            &s_k[fresh * kUnits + ((lane >> 2) ^ (fresh & (kUnits - 1)))])[lane & 3] = y2;
      else
        s_new[lane] = y2;
    }
  } else {
    for (int i = t; i < G * kHeadDim; i += 512)
      qs[i / kHeadDim][i % kHeadDim] =
          bf16_f32(q[(head0 + i / kHeadDim) * kHeadDim + i % kHeadDim]) * scale;
  }
#pragma unroll
  for (int i = 0; i < kAttnChunk * kUnits / 512; ++i) {
    const int row = (t + 512 * i) / kUnits, c = t % kUnits;
    if (row < n && row != fresh) s_k[row * kUnits + (c ^ (row & (kUnits - 1)))] = kr[i];
  }
  lds_barrier();
  if (kFused && fresh < 64 * pg + 64) {  // uniform
    // the fresh row, also for the positions past it (their loads found the
    // row as it was before)
    const u32x2 nv = *reinterpret_cast<const u32x2 *>(&s_new[32 * half + 2 * dg]);
#pragma unroll
    for (int st = 0; st < 16; ++st)
      if (64 * pg + 4 * st + rr >= fresh) vv[st] = nv;
  }

  constexpr int kH = G / 2;  // heads of this wave's scores: half * kH..
  const int j = 64 * pg + lane;  // position within the chunk
  float s[kH];
#pragma unroll
  for (int h = 0; h < kH; ++h) s[h] = 0.f;
  const bool valid = j < n;
  if (valid) {
#pragma unroll
    for (int c = 0; c < kUnits; ++c) {
      const u32x4 kv = s_k[j * kUnits + (c ^ (j & (kUnits - 1)))];
      float kf[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kf[2 * e] = bf16_f32(kv[e] & 0xffffu);
        kf[2 * e + 1] = __uint_as_float(kv[e] & 0xffff0000u);
      }
#pragma unroll
      for (int h = 0; h < kH; ++h) {
        const float4 q0 = *reinterpret_cast<const float4 *>(&qs[half * kH + h][8 * c]);
        const float4 q1 = *reinterpret_cast<const float4 *>(&qs[half * kH + h][8 * c + 4]);
        s[h] = fmaf(q0.x, kf[0], s[h]);
        s[h] = fmaf(q0.y, kf[1], s[h]);
        s[h] = fmaf(q0.z, kf[2], s[h]);
        s[h] = fmaf(q0.w, kf[3], s[h]);
        s[h] = fmaf(q1.x, kf[4], s[h]);
        s[h] = fmaf(q1.y, kf[5], s[h]);
        s[h] = fmaf(q1.z, kf[6], s[h]);
        s[h] = fmaf(q1.w, kf[7], s[h]);
      }
    }
  }
#pragma unroll
  for (int h = 0; h < kH; ++h) {
    const float mw = wave_max_dpp(valid ? s[h] : -INFINITY);
    if (lane == 0) red[0][half * kH + h][pg] = mw;
  }
  lds_barrier();
#pragma unroll
  for (int h = 0; h < kH; ++h) {
    const float *rm = red[0][half * kH + h];
    const float mh = fmaxf(fmaxf(rm[0], rm[1]), fmaxf(rm[2], rm[3]));
    const float e = valid ? expf(s[h] - mh) : 0.f;
    pw[half * kH + h][pg][16 * (lane & 3) + (lane >> 2)] = e;
    const float sw = wave_sum(e);
    if (lane == 0) red[1][half * kH + h][pg] = sw;
  }
  lds_barrier();
  if (t < G) {
    wm[(head0 + t) * S + split] =
        fmaxf(fmaxf(red[0][t][0], red[0][t][1]), fmaxf(red[0][t][2], red[0][t][3]));
    wl[(head0 + t) * S + split] =
        (red[1][t][0] + red[1][t][1]) + (red[1][t][2] + red[1][t][3]);
  }
  float acc[G][4];
#pragma unroll
  for (int h = 0; h < G; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[h][e] = 0.f;
#pragma unroll
  for (int s4 = 0; s4 < 4; ++s4) {
    float4 pv[G];
#pragma unroll
    for (int h = 0; h < G; ++h)
      pv[h] = *reinterpret_cast<const float4 *>(&pw[h][pg][16 * rr + 4 * s4]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x2 wds = vv[4 * s4 + i];
      const float v0 = bf16_f32(wds[0] & 0xffffu), v1 = __uint_as_float(wds[0] & 0xffff0000u);
      const float v2 = bf16_f32(wds[1] & 0xffffu), v3 = __uint_as_float(wds[1] & 0xffff0000u);
#pragma unroll
      for (int h = 0; h < G; ++h) {
        const float pr = i == 0 ? pv[h].x : i == 1 ? pv[h].y : i == 2 ? pv[h].z : pv[h].w;
        acc[h][0] = fmaf(pr, v0, acc[h][0]);
        acc[h][1] = fmaf(pr, v1, acc[h][1]);
        acc[h][2] = fmaf(pr, v2, acc[h][2]);
        acc[h][3] = fmaf(pr, v3, acc[h][3]);
      }
    }
  }
  // every wave is past its keys (two barriers ago): part overlays them.  The
  // four lane rows' sums, (0 + 1) + (2 + 3), four accumulators at a time:
  // lane row g holds dim 4 dg + g's.
#pragma unroll
  for (int h = 0; h < G; ++h)
    part[pg][h][64 * half + 4 * dg + rr] =
        add_swap32(add_swap16(acc[h][0], acc[h][1]), add_swap16(acc[h][2], acc[h][3]));
  lds_barrier();
  for (int v = t; v < G * kHeadDim; v += 512) {
    const int h = v / kHeadDim, d = v % kHeadDim;
    wacc[((head0 + h) * S + split) * kHeadDim + d] =
        (part[0][h][d] + part[1][h][d]) + (part[2][h][d] + part[3][h][d]);
  }
}

// Merge the splits [0, used) of one (b, head) -- partials m, l [B*Hq, S] and
// acc [B*Hq, S, 128] -- in order, and write its 128 outputs: quantized as
// one o-projection group, and optionally as bf16.  One wave, two dims per
// lane.  Latency-bound, so eight splits' loads are in flight at a time (16 x
// 32 heads of 33 splits: 15.9 us one by one, 7.8 now).
__global__ __launch_bounds__(64) void attn_combine_kernel(const float *__restrict__ wm,
                                                          const float *__restrict__ wl,
                                                          const float *__restrict__ wacc,
                                                          const int *__restrict__ pos, int Lmax,
                                                          int S, int Hq, uint8_t *__restrict__ oq,
                                                          float *__restrict__ os,
                                                          uint16_t *__restrict__ ob) {
  const int lane = threadIdx.x;
  int L = pos[0] + 1;
  L = L < 1 ? 1 : (L > Lmax ? Lmax : L);
  const int used = (L + kAttnChunk - 1) / kAttnChunk;
  const size_t bh = blockIdx.x;
  const float *pm = wm + bh * S, *pl = wl + bh * S;
  const float2 *pa = reinterpret_cast<const float2 *>(wacc + bh * S * kHeadDim) + lane;
  constexpr int kU = 8;
  float2 a[kU];
  auto load = [&](int s0) {
#pragma unroll
    for (int u = 0; u < kU; ++u) a[u] = pa[(size_t)min(s0 + u, used - 1) * 64];
  };
  load(0);
  float mx = -INFINITY;
  for (int s = lane; s < used; s += 64) mx = fmaxf(mx, pm[s]);
  mx = wave_max_dpp(mx);
  float l = 0.f, a0 = 0.f, a1 = 0.f;
  for (int s0 = 0; s0 < used; s0 += kU) {
    float2 c[kU];
    float f[kU], ls[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int s = min(s0 + u, used - 1);
      c[u] = a[u];
      f[u] = pm[s];
      ls[u] = pl[s];
    }
    if (s0 + kU < used) load(s0 + kU);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (s0 + u < used) {  // uniform
        const float e = expf(f[u] - mx);
        l = fmaf(e, ls[u], l);
        a0 = fmaf(e, c[u].x, a0);
        a1 = fmaf(e, c[u].y, a1);
      }
    }
  }
  a0 /= l;
  a1 /= l;
  if (ob) reinterpret_cast<uint32_t *>(ob)[bh * 64 + lane] = f32_bf16(a0) | (f32_bf16(a1) << 16);
  const float amax = wave_max_dpp(fmaxf(fabsf(a0), fabsf(a1)));
  const float sc = amax > 0.f ? amax / kFp8Max : 1.f;
  const float qs[4] = {a0 / sc, a1 / sc, 0.f, 0.f};
  const uint32_t q2 = f32_e4m3x4(qs, qs);
  // row b = bh / Hq, group = head: bytes 2 lane, 2 lane + 1 of the group
  const int b = (int)(bh / (size_t)Hq), head = (int)(bh % (size_t)Hq);
  *reinterpret_cast<uint16_t *>(oq + tile_chunk_off(b, head, Hq, lane >> 3) + 2 * (lane & 7)) =
      (uint16_t)q2;
  if (lane == 0) os[bh] = sc;
}

// ---------------------------------------------------- FP8 block dequantize

// e4m3fn byte -> fp32 (exact; 0x7F / 0xFF, the NaN codes, become NaN)
__device__ __forceinline__ float e4m3_f32(uint32_t b) {
  const uint32_t sign = (b & 0x80u) << 24;
  const uint32_t e = (b >> 3) & 0xFu, m = b & 7u;
  if (e == 0) return __uint_as_float(sign | __float_as_uint((float)m * 0.001953125f));  // m * 2^-9
  if (e == 15 && m == 7) return __uint_as_float(sign | 0x7FC00000u);
  return __uint_as_float(sign | ((e + 120u) << 23) | (m << 20));
}

// out[r, c] = bf16(w[r, c] * scale[r / 128, c / 128]); one thread per 16
// consecutive bytes of a row (always inside one 128-column group).
__global__ __launch_bounds__(256) void dequant_fp8_block_kernel(const uint8_t *__restrict__ w,
                                                                const float *__restrict__ scale,
                                                                int64_t n, int64_t k,
                                                                uint16_t *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // 16-byte unit
  const int64_t units_per_row = k / 16;
  if (i >= n * units_per_row) return;
  const int64_t r = i / units_per_row, c = (i % units_per_row) * 16;
  const float sc = scale[(r / kGroup) * (k / kGroup) + c / kGroup];
  const uint4 b = *reinterpret_cast<const uint4 *>(w + r * k + c);
  const uint32_t wd[4] = {b.x, b.y, b.z, b.w};
  uint32_t o[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float v0 = e4m3_f32(wd[j] & 0xFFu) * sc, v1 = e4m3_f32((wd[j] >> 8) & 0xFFu) * sc;
    const float v2 = e4m3_f32((wd[j] >> 16) & 0xFFu) * sc, v3 = e4m3_f32(wd[j] >> 24) * sc;
    o[2 * j] = f32_bf16(v0) | (f32_bf16(v1) << 16);
    o[2 * j + 1] = f32_bf16(v2) | (f32_bf16(v3) << 16);
  }
  uint4 *op = reinterpret_cast<uint4 *>(out + r * k + c);
  op[0] = make_uint4(o[0], o[1], o[2], o[3]);
  op[1] = make_uint4(o[4], o[5], o[6], o[7]);
}

// ------------------------------------------------------------ MoE routing

// Router logits: logits[m, e] = x[m] . wr[e] over H (bf16 inputs, fp32
// products accumulated per lane in order, then summed across the wave in a
// fixed tree).  Workgroup (ex, tb): wave w takes expert 4 ex + w and tokens
// [4 tb, +4); every load of a 2048-column slice is issued before its FMAs.
// H a multiple of 512.
__global__ __launch_bounds__(256) void moe_logits_kernel(const uint16_t *__restrict__ x,
                                                         const uint16_t *__restrict__ wr, int M,
                                                         int H, int E,
                                                         float *__restrict__ logits) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = blockIdx.x * 4 + wave;
  const int m0 = blockIdx.y * 4;
  if (e >= E) return;  // uniform per wave; no barrier below
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int h0 = 0; h0 < H; h0 += 2048) {
    uint4 wv[4], xv[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = h0 + 512 * j + 8 * lane;
      const bool in = h0 + 512 * j < H;
      wv[j] = in ? *reinterpret_cast<const uint4 *>(wr + (size_t)e * H + c) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int m = min(m0 + t, M - 1);  // rows past M re-read row M - 1, unused
        xv[t][j] = in ? *reinterpret_cast<const uint4 *>(x + (size_t)m * H + c)
                      : make_uint4(0, 0, 0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t ww[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t xw[4] = {xv[t][j].x, xv[t][j].y, xv[t][j].z, xv[t][j].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[t] = fmaf(bf16_f32(xw[i] & 0xffffu), bf16_f32(ww[i] & 0xffffu), acc[t]);
          acc[t] = fmaf(bf16_f32(xw[i] >> 16), bf16_f32(ww[i] >> 16), acc[t]);
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const float v = wave_sum(acc[t]);
    if (lane == 0 && m0 + t < M) logits[(size_t)(m0 + t) * E + e] = v;
  }
}

// Top-k of one token per wave (4 tokens per 256-thread workgroup): softmax
// over the E <= 256 logits in fp32, the top_k largest probabilities (ties
// to the lower expert index), renormalized to sum 1.  One wave's latency
// bounds it: each pick is a DPP maximum and four ballots (16 tokens of 128
// experts, top 8: 6.9 -> 4.5 us against two shuffles per butterfly step).
__global__ __launch_bounds__(256) void moe_topk_kernel(const float *__restrict__ logits, int M,
                                                       int E, int top_k,
                                                       int *__restrict__ topk_idx,
                                                       float *__restrict__ topk_w) {
  const int lane = threadIdx.x & 63;
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;  // uniform per wave; no barrier below
  // lane l holds experts l, l + 64, l + 128, l + 192
  float p[4];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = lane + 64 * i;
    p[i] = e < E ? logits[(size_t)m * E + e] : -INFINITY;
    mx = fmaxf(mx, p[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    p[i] = lane + 64 * i < E ? expf(p[i] - mx) : 0.f;
    sum += p[i];
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = lane + 64 * i < E ? p[i] / sum : -1.f;  // -1: not a choice
  float my_w = 0.f, sel_sum = 0.f;
  int my_i = 0;
  for (int k = 0; k < top_k; ++k) {
    // the largest probability, then the lowest expert that has it (expert
    // lane + 64 i: the lowest i first, then the lowest lane)
    // (-2 if none is a number)
    const float bv = wave_max_dpp(fmaxf(fmaxf(fmaxf(fmaxf(-2.f, p[0]), p[1]), p[2]), p[3]));
    int bi = 0x7fffffff;
#pragma unroll
    for (int i = 3; i >= 0; --i) {
      const uint64_t at = __ballot(p[i] == bv);
      if (at) bi = 64 * i + __builtin_ctzll(at);  // uniform
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (lane + 64 * i == bi) p[i] = -1.f;
    sel_sum += bv;
    if (lane == k) {
      my_w = bv;
      my_i = bi;
    }
  }
  if (lane < top_k) {
    topk_idx[(size_t)m * top_k + lane] = my_i;
    topk_w[(size_t)m * top_k + lane] = my_w / sel_sum;
  }
}

// Group the P = M * top_k (token, expert) pairs by expert (one workgroup
// of 1024 threads, P <= 8192, E <= 256): pairs of expert e take sorted
// positions [offsets[e], offsets[e + 1]) in token order; pair_tok / pair_w
// give each sorted position's token and routing weight, pair_pos each
// pair's sorted position; active[0, n_active) lists the experts with pairs
// in increasing order; select[e] (optional) = 1 if expert e has pairs.
// Expert ids outside [0, E) are clamped into it.
//
// A stable counting sort.  Wave w owns a contiguous run of 64 x chunks
// pairs (chunks = ceil(P / 1024) <= 8); a lane's rank among the pairs of
// its expert in its 64-pair chunk is a popcount of the wave's match mask
// (eight ballots, one per bit of the expert), and the wave's own row of
// counts in LDS carries the rank over its chunks.  Latency of one
// workgroup bounds it: three barriers and 8 ballots per 64 pairs instead of
// a serial walk over 1024 pairs per chunk and pass (MI355X: 4096 pairs
// 168.9 -> 10.1 us, 128 pairs 8.2 -> 4.4 us).
__global__ __launch_bounds__(1024) void moe_group_kernel(
    const int *__restrict__ topk_idx, const float *__restrict__ topk_w, int P, int top_k, int E,
    int *__restrict__ offsets, int *__restrict__ active, int *__restrict__ n_active,
    int *__restrict__ pair_tok, float *__restrict__ pair_w, int *__restrict__ pair_pos,
    int *__restrict__ select) {
  constexpr int kWaves = 16, kMaxChunks = 8;
  __shared__ int s_cnt[kWaves][256];  // pairs per expert of each wave's run
  __shared__ int s_tot[256];
  __shared__ int s_off[256];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int chunks = (P + 1023) >> 10;
  const int base = wave * 64 * chunks;
  int ex[kMaxChunks], rank[kMaxChunks];
  float w[kMaxChunks];
#pragma unroll
  for (int c = 0; c < kMaxChunks; ++c) {
    const int p = base + 64 * c + lane;
    const bool in = c < chunks && p < P;
    ex[c] = in ? min(max(topk_idx[p], 0), E - 1) : -1;
    w[c] = in ? topk_w[p] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) s_cnt[wave][lane + 64 * i] = 0;
  // The wave's own row: LDS serves one wave in program order, so its later
  // reads follow these writes (wave barriers keep the compiler to it).
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int c = 0; c < kMaxChunks; ++c) {
    rank[c] = 0;
    if (c < chunks) {  // uniform
      const bool in = ex[c] >= 0;
      uint64_t peers = __ballot(in);
#pragma unroll
      for (int bit = 0; bit < 8; ++bit) {
        const bool one = (ex[c] >> bit) & 1;
        const uint64_t ones = __ballot(one);
        peers &= one ? ones : ~ones;
      }
      const int before = __popcll(peers & ((1ull << lane) - 1));
      if (in) {
        rank[c] = s_cnt[wave][ex[c]] + before;
        __builtin_amdgcn_wave_barrier();
        // the last pair of each expert writes the new count (all its peers
        // have read the old one: one wave, in program order)
        if ((peers >> lane) == 1) s_cnt[wave][ex[c]] = rank[c] + 1;
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  __syncthreads();
  if (t < 256) {  // counts of each wave -> pairs of that expert in earlier waves
    int run = 0;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) {
      const int n = s_cnt[v][t];
      s_cnt[v][t] = run;
      run += n;
    }
    s_tot[t] = run;
  }
  __syncthreads();
  if (t < 64) {
    // wave 0: exclusive prefix of the counts and of the active flags over
    // E <= 256 experts, 4 consecutive experts per lane
    int c[4], f[4], sc = 0, sf = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c[i] = s_tot[4 * t + i];  // zero from expert E on
      f[i] = c[i] > 0;
      sc += c[i];
      sf += f[i];
    }
    int ic = sc, jf = sf;  // inclusive scans across lanes
    for (int o = 1; o < 64; o <<= 1) {
      const int uc = __shfl_up(ic, o), uf = __shfl_up(jf, o);
      if (t >= o) {
        ic += uc;
        jf += uf;
      }
    }
    int off = ic - sc, na = jf - sf;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = 4 * t + i;
      s_off[e] = off;
      if (e < E) {
        offsets[e] = off;
        if (f[i]) active[na] = e;
        if (select) select[e] = f[i];
      }
      off += c[i];
      na += f[i];
    }
    if (t == 63) {
      offsets[E] = ic;
      *n_active = jf;
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kMaxChunks; ++c) {
    if (ex[c] >= 0) {
      const int p = base + 64 * c + lane;
      const int q = s_off[ex[c]] + s_cnt[wave][ex[c]] + rank[c];
      pair_tok[q] = p / top_k;
      pair_w[q] = w[c];
      pair_pos[p] = q;
    }
  }
}

// Grouped small-M FP8 linear over the active experts: workgroup (tile,
// slot) computes output columns [16 tile, +16) of expert e = active[slot]
// for its rows [offsets[e], offsets[e + 1]) in chunks of 16:
//   out[q, col] = sum_g (sum_{k in g} aq[row(q), k] * w_e[n, k]) * as[row(q), g] * ws_e[n/128, g]
// with row(q) = row_of[q] (a gather, e.g. the token of a sorted pair) or q.
// Segment s of an expert (e.g. gate, up) owns output columns
// [s * seg_n, +seg_n).  Slots past n_active exit at once, so the grid can
// be sized for every expert and captured in a graph.
struct MoeLinear {
  const uint8_t *aq;
  const float *as;
  const int *row_of;
  const int *offsets;
  const int *active;
  const int *n_active;
  const uint64_t *w;   // [E * n_segs] weight addresses
  const uint64_t *ws;  // [E * n_segs] scale addresses
  uint16_t *out;
  int n_segs, seg_n, K, ldo;
  int wtiled;  // expert weights in the tile layout (else row-major)
};

template <int WAVES, int kU>
__global__ __launch_bounds__(WAVES * 64) void moe_linear16_kernel(MoeLinear a) {
  __shared__ float red[WAVES][4][64];
  const int slot = blockIdx.y;
  if (slot >= a.n_active[0]) return;  // uniform
  const int e = a.active[slot];
  const int r0 = a.offsets[e], rows = a.offsets[e + 1] - r0;
  const int seg = (int)(blockIdx.x * 16) / a.seg_n;
  const int n0 = (int)(blockIdx.x * 16) - seg * a.seg_n;
  const uint8_t *w = reinterpret_cast<const uint8_t *>(a.w[(size_t)e * a.n_segs + seg]);
  const float *ws = reinterpret_cast<const float *>(a.ws[(size_t)e * a.n_segs + seg]);
  const int col = seg * a.seg_n;
  const int K = a.K, kgroups = K / kGroup;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const WeightLane wl(w, a.wtiled != 0, n0, r, g, K);
  const Rsrc wr = wl.rsrc(K);
  const float *wsrow = ws + (size_t)(n0 / kGroup) * kgroups;

  for (int rc = 0; rc < rows; rc += 16) {
    const int mrows = min(16, rows - rc);
    const bool row_ok = r < mrows;
    const int q = r0 + rc + (row_ok ? r : 0);
    const uint8_t *arow = tile_lane_base(a.aq, a.row_of ? a.row_of[q] : q, kgroups, g);
    bool srow_ok[4];
    const float *srow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      srow_ok[i] = 4 * g + i < mrows;
      const int qi = r0 + rc + (srow_ok[i] ? 4 * g + i : 0);
      srow[i] = a.as + (size_t)(a.row_of ? a.row_of[qi] : qi) * kgroups;
    }
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int kb = wave; kb < kgroups; kb += WAVES * kU) {
      uint4 wv[kU][2], av[kU][2];
      float wsv[kU], sav[kU][4];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int kg = kb + WAVES * u;
        if (kg < kgroups) {
          wl.load(wr, kg, wv[u][0], wv[u][1]);
          wsv[u] = wsrow[kg];
          av[u][0] = *reinterpret_cast<const uint4 *>(arow + (size_t)kg * 2048);
          av[u][1] = *reinterpret_cast<const uint4 *>(arow + (size_t)kg * 2048 + 1024);
#pragma unroll
          for (int i = 0; i < 4; ++i) sav[u][i] = srow[i][kg];
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int kg = kb + WAVES * u;
        if (kg >= kgroups) break;
        if (!row_ok) av[u][0] = av[u][1] = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) sav[u][i] = srow_ok[i] ? sav[u][i] : 0.f;
        v4f d = {0.f, 0.f, 0.f, 0.f};
        d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
            (long)(((uint64_t)av[u][0].y << 32) | av[u][0].x),
            (long)(((uint64_t)wv[u][0].y << 32) | wv[u][0].x), d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
            (long)(((uint64_t)av[u][0].w << 32) | av[u][0].z),
            (long)(((uint64_t)wv[u][0].w << 32) | wv[u][0].z), d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
            (long)(((uint64_t)av[u][1].y << 32) | av[u][1].x),
            (long)(((uint64_t)wv[u][1].y << 32) | wv[u][1].x), d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
            (long)(((uint64_t)av[u][1].w << 32) | av[u][1].z),
            (long)(((uint64_t)wv[u][1].w << 32) | wv[u][1].z), d, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(d[i], sav[u][i] * wsv[u], acc[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][i][lane] = acc[i];
    __syncthreads();
    // the 256 sums (4 accumulators x 64 lanes), over the threads
    for (int t = threadIdx.x; t < 256; t += WAVES * 64) {
      const int i = t >> 6, l = t & 63;
      float sum = 0.f;
#pragma unroll
      for (int wv2 = 0; wv2 < WAVES; ++wv2) sum += red[wv2][i][l];
      const int m = 4 * (l >> 4) + i;
      if (m < mrows)
        a.out[(size_t)(r0 + rc + m) * a.ldo + col + n0 + (l & 15)] = (uint16_t)f32_bf16(sum);
    }
    __syncthreads();  // red is rewritten by the next chunk
  }
}

// Block u of the rows that the active experts have past their first kRows, in
// turn, kRows rows (or the rest of an expert's) each: its expert and its
// number in it; false past the last.  Each wave finds it by itself, 256
// experts at a time, four per lane.
template <int kRows>
__device__ __forceinline__ bool moe_row_block(const MoeLinear &a, int n_active, int u, int &e,
                                              int &block) {
  const int lane = threadIdx.x & 63;
  for (int page = 0; page < n_active; page += 256) {
    int ex[4], n[4], sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int slot = page + 4 * lane + i;
      ex[i] = slot < n_active ? a.active[slot] : -1;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rows = ex[i] < 0 ? 0 : a.offsets[ex[i] + 1] - a.offsets[ex[i]];
      n[i] = max(rows - 1, 0) / kRows;
      sum += n[i];
    }
    int end = sum;  // inclusive scan over the lanes
#define ECF8_DPP_SCAN(ctrl, rows) \
  end += __builtin_amdgcn_update_dpp(0, end, ctrl, rows, 0xF, false)
    ECF8_DPP_SCAN(0x111, 0xF);  // row_shr:1
    ECF8_DPP_SCAN(0x112, 0xF);  // row_shr:2
    ECF8_DPP_SCAN(0x114, 0xF);  // row_shr:4
    ECF8_DPP_SCAN(0x118, 0xF);  // row_shr:8
    ECF8_DPP_SCAN(0x142, 0xA);  // row_bcast:15 to rows 1 and 3
    ECF8_DPP_SCAN(0x143, 0xC);  // row_bcast:31 to rows 2 and 3
#undef ECF8_DPP_SCAN
    const uint64_t past = __ballot(u < end);
    if (past) {
      int at = u - (end - sum), found = -1;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (found < 0 && at < n[i]) found = ex[i];
        if (found < 0) at -= n[i];
      }
      const int src = __builtin_ctzll(past);
      e = __builtin_amdgcn_readlane(found, src);
      block = __builtin_amdgcn_readlane(at, src) + 1;
      return true;
    }
    u -= __builtin_amdgcn_readlane(end, 63);
  }
  return false;
}

// The same grouped linear for many rows per expert (a prompt): a workgroup of
// eight waves computes a 128-column strip of a block of 16 kChunks rows, wave
// w its columns [16 w, +16), so an expert's weights are read once per 64 (or
// 32) rows instead of once per 16.  The rows' activations go to LDS in MFMA
// lane order (gathered 16-byte parts), shared by the eight waves and
// double-buffered; a wave's weight panel goes straight to its registers, one
// stage of PARTS groups ahead.  Workgroups (strip, slot < n_experts) take the
// active experts' first rows, those after them the blocks past these, one
// each (moe_row_block), so that the experts that most tokens pick do not hold
// up a few workgroups.
//
// The sums are moe_linear16_kernel's, bit for bit: group kg adds to partial
// sum kg mod PARTS (that kernel's wave), the partial sums are added in
// order.  The latency of a block's loads bounds it, one after the other:
// routing, scales and rows, then two to four stages of weights (2.9 to 3.6
// TB/s of weights where a copy reads and writes at 6.2).  MI355X, 128 experts,
// tile-layout weights, us, gate/up and down, 16-row form against this one:
// 512 tokens routed evenly 339 / 104 against 113 / 68; all on eight experts
// 172 / 92 against 62 / 47 (142 / 92 when an expert's workgroups walked all
// its rows); every token on one expert among others 318 / 104 against 113 /
// 60 (147 / 105).
template <int PARTS, int kChunks>
__global__ __launch_bounds__(512, 8 / kChunks) void moe_rows_kernel(MoeLinear a, int n_experts) {
  constexpr int kRows = 16 * kChunks, kMaxGroups = 16;
  constexpr int kCopies = 2 * kChunks < 8 ? 8 / (2 * kChunks) : 1;  // waves per 1 KB part
  __shared__ u32x4 s_a[2][PARTS][kChunks][2][64];
  __shared__ __attribute__((aligned(16))) float s_s[kMaxGroups][kRows];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int seg = (int)(blockIdx.x * 128) / a.seg_n;  // seg_n is a multiple of 128
  const int n0 = (int)(blockIdx.x * 128) - seg * a.seg_n + 16 * wave;
  const int K = a.K, kgroups = K / kGroup;
  const int stages = (kgroups + PARTS - 1) / PARTS;
  const int n_active = a.n_active[0];

  int u = (int)blockIdx.y - n_experts, e, block = 0;
  if (u < 0) {  // uniform
    if ((int)blockIdx.y >= n_active) return;
    e = a.active[blockIdx.y];
  } else if (!moe_row_block<kRows>(a, n_active, u, e, block)) {
    return;
  }
  do {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // nothing per lane is kept from block to block
    const int r = lane & 15, g = lane >> 4;
    const int r0 = a.offsets[e], rc = kRows * block;
    const int mrows = min(kRows, a.offsets[e + 1] - r0 - rc);
    const uint8_t *w = reinterpret_cast<const uint8_t *>(a.w[(size_t)e * a.n_segs + seg]);
    const float *wsrow =
        reinterpret_cast<const float *>(a.ws[(size_t)e * a.n_segs + seg]) +
        (size_t)(n0 / kGroup) * kgroups;
    const WeightLane wl(w, a.wtiled != 0, n0, r, g, K);
    const Rsrc wr = wl.rsrc(K);
    const int nch = (mrows + 15) >> 4;  // 16-row chunks in use (uniform)
    // scales, [group][row]; rows past the last take its values, unused
    for (int i = threadIdx.x; i < kRows * kgroups; i += 512) {
      const int row = i / kgroups, kg = i - row * kgroups;
      const int q = r0 + rc + min(row, mrows - 1);
      s_s[kg][row] = a.as[(size_t)(a.row_of ? a.row_of[q] : q) * kgroups + kg];
    }
    // wave v stages half (v / kCopies) & 1 of chunk v / kCopies / 2: groups
    // v % kCopies, + kCopies, ... of each stage
    const int lc = wave / kCopies >> 1, lh = wave / kCopies & 1, lu = wave % kCopies;
    const int lq = r0 + rc + min(16 * lc + r, mrows - 1);
    const uint8_t *arow =
        tile_lane_base(a.aq, a.row_of ? a.row_of[lq] : lq, kgroups, g) + 1024 * lh;
    constexpr int kA = (PARTS + kCopies - 1) / kCopies;
    u32x4 av[kA];
    uint4 wv[PARTS][2];
    float wsv[PARTS];
    // groups past the last load it again, unused
    auto load = [&](int s, u32x4 (&av)[kA], uint4 (&wv)[PARTS][2], float (&wsv)[PARTS]) {
#pragma unroll
      for (int u = 0; u < kA; ++u)
        av[u] = *reinterpret_cast<const u32x4 *>(
            arow + (size_t)min(s * PARTS + lu + kCopies * u, kgroups - 1) * 2048);
#pragma unroll
      for (int u = 0; u < PARTS; ++u) {
        const int kg = min(s * PARTS + u, kgroups - 1);
        wl.load(wr, kg, wv[u][0], wv[u][1]);
        wsv[u] = wsrow[kg];
      }
    };
    float acc[PARTS][kChunks][4];
#pragma unroll
    for (int u = 0; u < PARTS; ++u)
#pragma unroll
      for (int c = 0; c < kChunks; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u][c][i] = 0.f;
    load(0, av, wv, wsv);
    for (int s = 0; s < stages; ++s) {
      const int buf = s & 1;
      uint4 wc[PARTS][2];
      float wsc[PARTS];
#pragma unroll
      for (int u = 0; u < kA; ++u)
        if (lu + kCopies * u < PARTS) s_a[buf][lu + kCopies * u][lc][lh][lane] = av[u];
#pragma unroll
      for (int u = 0; u < PARTS; ++u) {
        wc[u][0] = wv[u][0];
        wc[u][1] = wv[u][1];
        wsc[u] = wsv[u];
      }
      // this stage is in LDS; the other buffer was last read in stage s - 1,
      // before every wave's arrival here
      lds_barrier();
      if (s + 1 < stages) load(s + 1, av, wv, wsv);
#pragma unroll
      for (int u = 0; u < PARTS; ++u) {
        const int kg = s * PARTS + u;
        if (kg >= kgroups) break;  // uniform
#pragma unroll
        for (int c = 0; c < kChunks; ++c) {
          if (c < nch) {  // uniform
            const u32x4 lo = s_a[buf][u][c][0][lane], hi = s_a[buf][u][c][1][lane];
            const float4 sc = *reinterpret_cast<const float4 *>(&s_s[kg][16 * c + 4 * g]);
            v4f d = {0.f, 0.f, 0.f, 0.f};
            d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
                (long)(((uint64_t)lo.y << 32) | lo.x),
                (long)(((uint64_t)wc[u][0].y << 32) | wc[u][0].x), d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
                (long)(((uint64_t)lo.w << 32) | lo.z),
                (long)(((uint64_t)wc[u][0].w << 32) | wc[u][0].z), d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
                (long)(((uint64_t)hi.y << 32) | hi.x),
                (long)(((uint64_t)wc[u][1].y << 32) | wc[u][1].x), d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
                (long)(((uint64_t)hi.w << 32) | hi.z),
                (long)(((uint64_t)wc[u][1].w << 32) | wc[u][1].z), d, 0, 0, 0);
            acc[u][c][0] = fmaf(d[0], sc.x * wsc[u], acc[u][c][0]);
            acc[u][c][1] = fmaf(d[1], sc.y * wsc[u], acc[u][c][1]);
            acc[u][c][2] = fmaf(d[2], sc.z * wsc[u], acc[u][c][2]);
            acc[u][c][3] = fmaf(d[3], sc.w * wsc[u], acc[u][c][3]);
          }
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kChunks; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = 16 * c + 4 * g + i;
        float sum = 0.f;
#pragma unroll
        for (int u = 0; u < PARTS; ++u) sum += acc[u][c][i];
        if (m < mrows)
          a.out[(size_t)(r0 + rc + m) * a.ldo + seg * a.seg_n + n0 + r] = (uint16_t)f32_bf16(sum);
      }
    if (u < 0) return;
    u += (int)gridDim.y - n_experts;
    lds_barrier();  // s_s and s_a are refilled for the next rows
  } while (moe_row_block<kRows>(a, n_active, u, e, block));
}

// y[m, :] = sum_k pair_w[q] * down[q, :] over q = pair_pos[m * top_k + k],
// k = 0 .. top_k - 1 in order, accumulated in fp32; bf16 out [M, H].  One
// workgroup per token, 8 columns per thread.
__global__ __launch_bounds__(256) void moe_combine_kernel(const uint16_t *__restrict__ down,
                                                          int ldd, const int *__restrict__ pair_pos,
                                                          const float *__restrict__ pair_w,
                                                          int top_k, int H,
                                                          uint16_t *__restrict__ out) {
  const int m = blockIdx.x;
  for (int c = 8 * threadIdx.x; c < H; c += 8 * 256) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < top_k; ++k) {
      const int q = pair_pos[(size_t)m * top_k + k];
      const float wq = pair_w[q];
      const uint4 v = *reinterpret_cast<const uint4 *>(down + (size_t)q * ldd + c);
      const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = fmaf(wq, bf16_f32(wd[i] & 0xffffu), acc[2 * i]);
        acc[2 * i + 1] = fmaf(wq, bf16_f32(wd[i] >> 16), acc[2 * i + 1]);
      }
    }
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = f32_bf16(acc[2 * i]) | (f32_bf16(acc[2 * i + 1]) << 16);
    *reinterpret_cast<uint4 *>(out + (size_t)m * H + c) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }
inline bool aligned(const void *p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }
inline int launched() { return hipGetLastError() == hipSuccess ? ECF8_OK : ECF8_ERR_HIP; }

}  // namespace

extern "C" int ecf8_fp8_linear(const void *aq, const float *as, int64_t M, int64_t K,
                               const ecf8_linear_seg *segs, int n_segs, void *out, int64_t ldo,
                               void *stream) {
  if (!aq || !as || !segs || !out || M <= 0 || K <= 0 || n_segs < 1 ||
      n_segs > ECF8_LINEAR_MAX_SEGS)
    return ECF8_ERR_INVALID_ARG;
  if (K % kGroup || M > (1 << 24) || K > (1 << 20)) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(aq, 16) || !aligned(out, 4) || !aligned(as, 4)) return ECF8_ERR_MISALIGNED;
  LinearSegs s{};
  int64_t n_total = 0;
  for (int i = 0; i < n_segs; ++i) {
    const ecf8_linear_seg &g = segs[i];
    if (!g.weight || !g.weight_scale || g.n <= 0 || g.out_col < 0) return ECF8_ERR_INVALID_ARG;
    if (g.weight_layout != ECF8_WEIGHT_ROWS && g.weight_layout != ECF8_WEIGHT_TILES)
      return ECF8_ERR_INVALID_ARG;
    if (g.n % kGroup) return ECF8_ERR_UNSUPPORTED;
    if (!aligned(g.weight, 16) || !aligned(g.weight_scale, 4)) return ECF8_ERR_MISALIGNED;
    if (g.out_col + g.n > ldo) return ECF8_ERR_CAPACITY;
    n_total += g.n;
    s.w[i] = static_cast<const uint8_t *>(g.weight);
    s.ws[i] = g.weight_scale;
    s.n_end[i] = (int)n_total;
    s.col[i] = (int)g.out_col;
    s.tiled[i] = g.weight_layout == ECF8_WEIGHT_TILES;
  }
  if (n_total > (1 << 24)) return ECF8_ERR_UNSUPPORTED;
  s.count = n_segs;
  const auto *a = static_cast<const uint8_t *>(aq);
  auto *o = static_cast<uint16_t *>(out);
  if (M <= 16) {
    const unsigned n_tiles = (unsigned)(n_total / 16);
    int dev = 0, cus = 0;
    // more tiles than two workgroups per CU at K = 4096: the persistent form
    if (K == 4096 && hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        n_tiles > 2u * (unsigned)cus) {
      fp8_linear16p_kernel<16><<<(unsigned)cus, 1024, 0, as_stream(stream)>>>(
          a, as, (int)M, s, o, (int)ldo, (int)n_tiles);
      return launched();
    }
    // long K: 16 waves, so each wave's share stays within two batches;
    // at most one tile per CU: 16 waves, so the fused linear summing in the
    // same order runs 16 waves per CU (Qwen3-8B o projection: fused 9.8 ->
    // 8.4 us, FP8 unchanged at 5.5)
    if (K / kGroup >= 64 ||
        (hipGetDevice(&dev) == hipSuccess &&
         hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
         n_tiles <= (unsigned)cus))
      fp8_linear16_kernel<16><<<n_tiles, 1024, 0, as_stream(stream)>>>(a, as, (int)M, (int)K, s,
                                                                       o, (int)ldo);
    else
      fp8_linear16_kernel<8><<<n_tiles, 512, 0, as_stream(stream)>>>(a, as, (int)M, (int)K, s, o,
                                                                     (int)ldo);
  } else {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return ECF8_ERR_HIP;
    // The middle form while its 64 x 64 blocks are at most two per CU.  Where
    // M fills the 256-row tiles, the tile GEMM then has a workgroup on a
    // quarter of the CUs at most; for few rows it can have one on each, and
    // the line rests on the times alone.  MI355X, us, middle form against
    // tile GEMM (weight copies rotated): N = K = 4096: M = 64 7.6 / 32.5, M =
    // 256 12.4 / 33.1, M = 512 (512 blocks) 23.6 / 33.5, M = 768 about 35 /
    // 33.8; N = 24576: M = 64 (384 blocks) 34.5 / 39.1, M = 128 (768) about
    // 50 / 40.1; N = 32768, M = 64 (512) 38.8 / 44.6; K = 512, M = 512, N =
    // 4096 6.9 / 8.5 (one K group: 6.1 / 5.5).
    const int64_t blocks = (M + 63) / 64 * (n_total / 64);
    if (blocks <= 2 * (int64_t)cus) {
      // The narrowest strips that need no second round of workgroups; for a
      // single block of rows, where the weights come from HBM once, three
      // workgroups per CU in turn (N = 24576, M = 64: two panels 34.3, four
      // 36 us; N = 28672: 43.8 and 36.6; N = 6144, M = 64: one 11.7, two 9.7,
      // four 12.9).  32 rows a block where that covers M: M = 32, N = 4096
      // 5.8 us.
      const bool narrow = M <= 32;
      const int64_t row_blocks = narrow ? 1 : (M + 63) / 64;
      const int64_t one = row_blocks * (n_total / 16);
      const int panels = one <= cus ? 1 : one / 2 <= (row_blocks == 1 ? 3 : 1) * cus ? 2 : 4;
      const dim3 grid((unsigned)(n_total / (16 * panels)), (unsigned)row_blocks);
#define ECF8_ROWS(P, CH)                                                                    \
  fp8_rows_kernel<P, CH><<<grid, 512, 0, as_stream(stream)>>>(a, as, (int)M, (int)K, s, o, \
                                                              (int)ldo)
      if (narrow) {
        if (panels == 1) ECF8_ROWS(1, 2);
        else if (panels == 2) ECF8_ROWS(2, 2);
        else ECF8_ROWS(4, 2);
      } else {
        if (panels == 1) ECF8_ROWS(1, 4);
        else if (panels == 2) ECF8_ROWS(2, 4);
        else ECF8_ROWS(4, 4);
      }
#undef ECF8_ROWS
      return launched();
    }
    // 256 x 256 tiles where they need fewer rounds of workgroups even at
    // 1.75 times the time of a 256 x 128 tile.  MI355X, K = 4096, M = 2048,
    // us, wide against slim: N = 24576 (3 rounds and 6) 227 and 257, N = 6144
    // (1 and 2) 72 and 80, N = 4096 (1 and 1) 67 and 45.
    const int n_mb = (int)((M + 255) / 256);
    const int64_t wide = n_mb * ((n_total + 255) / 256), slim = n_mb * (n_total / 128);
    if (slim > INT32_MAX) return ECF8_ERR_UNSUPPORTED;
    if (7 * ((wide + cus - 1) / cus) < 4 * ((slim + cus - 1) / cus))
      fp8_gemm_kernel<2, 4, 2, 2><<<(unsigned)wide, 512, 0, as_stream(stream)>>>(
          a, as, (int)M, (int)K, s, o, (int)ldo, n_mb, (int)wide);
    else
      fp8_gemm_kernel<4, 2, 1, 3><<<(unsigned)slim, 512, 0, as_stream(stream)>>>(
          a, as, (int)M, (int)K, s, o, (int)ldo, n_mb, (int)slim);
  }
  return launched();
}

extern "C" int ecf8_rmsnorm(const void *x, float *residual, const void *weight, float eps, int64_t M,
                            int64_t K, void *out_q, float *out_scale, void *out_bf16, void *stream) {
  if (!residual || !weight || M <= 0 || (!out_bf16 && !out_q) || (!out_q != !out_scale))
    return ECF8_ERR_INVALID_ARG;
  if ((K != 4096 && K != 2048) || M > 0x7fffffff) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(residual, 16) || (x && !aligned(x, 16)) || !aligned(weight, 16) ||
      (out_q && !aligned(out_q, 16)) || (out_bf16 && !aligned(out_bf16, 16)))
    return ECF8_ERR_MISALIGNED;
  const auto *xp = static_cast<const uint16_t *>(x);
  const auto *wp = static_cast<const uint16_t *>(weight);
  auto *qp = static_cast<uint8_t *>(out_q);
  auto *bp = static_cast<uint16_t *>(out_bf16);
  if (K == 4096)
    rmsnorm_kernel<256><<<(unsigned)M, 256, 0, as_stream(stream)>>>(xp, residual, wp, eps, (int)K,
                                                                    qp, out_scale, bp);
  else
    rmsnorm_kernel<128><<<(unsigned)M, 128, 0, as_stream(stream)>>>(xp, residual, wp, eps, (int)K,
                                                                    qp, out_scale, bp);
  return launched();
}

extern "C" int ecf8_silu_mul_quant(const void *gate_up, int64_t M, int64_t I, void *out_q,
                                   float *out_scale, void *stream) {
  if (!gate_up || !out_q || !out_scale || M <= 0 || I <= 0) return ECF8_ERR_INVALID_ARG;
  if (I % kGroup || I > (1 << 24) || M > 65535) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(gate_up, 16) || !aligned(out_q, 16)) return ECF8_ERR_MISALIGNED;
  silu_mul_quant_kernel<<<dim3((unsigned)((I + 4095) / 4096), (unsigned)M), 256, 0,
                          as_stream(stream)>>>(
      static_cast<const uint16_t *>(gate_up), (int)I, static_cast<uint8_t *>(out_q), out_scale);
  return launched();
}

extern "C" int ecf8_act_quant(const void *x, int64_t M, int64_t K, void *out_q, float *out_scale,
                              void *stream) {
  if (!x || !out_q || !out_scale || M <= 0 || K <= 0) return ECF8_ERR_INVALID_ARG;
  if (K % kGroup || K > (1 << 24) || M > 65535) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(x, 16) || !aligned(out_q, 16)) return ECF8_ERR_MISALIGNED;
  act_quant_kernel<<<dim3((unsigned)((K + 4095) / 4096), (unsigned)M), 256, 0,
                     as_stream(stream)>>>(
      static_cast<const uint16_t *>(x), (int)K, static_cast<uint8_t *>(out_q), out_scale);
  return launched();
}

extern "C" int ecf8_qk_norm_rope(const void *qkv, int64_t B, int64_t T, int Hq, int Hkv,
                                 const void *q_norm, const void *k_norm, float eps, const float *cos_t,
                                 const float *sin_t, const int *pos, int64_t Lmax, void *q_out,
                                 void *k_cache, void *v_cache, void *stream) {
  if (!qkv || !q_norm || !k_norm || !cos_t || !sin_t || !pos || !q_out || !k_cache || !v_cache ||
      B <= 0 || T <= 0 || Hq <= 0 || Hkv <= 0 || Lmax <= 0)
    return ECF8_ERR_INVALID_ARG;
  const int64_t items = B * T * (Hq + 2 * Hkv);
  if (items > (int64_t)1 << 30) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(qkv, 4) || !aligned(q_norm, 4) || !aligned(k_norm, 4) || !aligned(q_out, 4) ||
      !aligned(k_cache, 4) || !aligned(v_cache, 4))
    return ECF8_ERR_MISALIGNED;
  const int64_t per = 4 * kRopePer;  // heads per workgroup
  const int64_t blocks = B * T * ((Hq + 2 * Hkv + per - 1) / per);
  qk_norm_rope_kernel<<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t *>(qkv), (int)T, Hq, Hkv, static_cast<const uint16_t *>(q_norm),
      static_cast<const uint16_t *>(k_norm), eps, cos_t, sin_t, pos, (int)Lmax,
      static_cast<uint16_t *>(q_out), static_cast<uint16_t *>(k_cache),
      static_cast<uint16_t *>(v_cache));
  return launched();
}

extern "C" int ecf8_dequant_fp8_block(const void *weight, const float *weight_scale, int64_t n,
                                      int64_t k, void *out, void *stream) {
  if (!weight || !weight_scale || !out || n <= 0 || k <= 0) return ECF8_ERR_INVALID_ARG;
  if (n % kGroup || k % kGroup || n * k > ((int64_t)1 << 40)) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(weight, 16) || !aligned(out, 16) || !aligned(weight_scale, 4))
    return ECF8_ERR_MISALIGNED;
  const int64_t units = n * (k / 16);
  dequant_fp8_block_kernel<<<(unsigned)((units + 255) / 256), 256, 0, as_stream(stream)>>>(
      static_cast<const uint8_t *>(weight), weight_scale, n, k, static_cast<uint16_t *>(out));
  return launched();
}

extern "C" int64_t ecf8_attention_work_floats(int64_t B, int Hq, int64_t Lmax) {
  if (B <= 0 || Hq <= 0 || Lmax <= 0) return -1;
  const int64_t S = (Lmax + kAttnChunk - 1) / kAttnChunk;
  return B * Hq * S * (kHeadDim + 2);
}

extern "C" int ecf8_decode_attention(const void *q, const void *k_cache, const void *v_cache,
                                     const int *pos, int64_t B, int Hq, int Hkv, int64_t Lmax,
                                     float *work, int64_t work_floats, void *out_q,
                                     float *out_scale, void *out_bf16, void *stream) {
  if (!q || !k_cache || !v_cache || !pos || !work || !out_q || !out_scale || B <= 0 || Hq <= 0 ||
      Hkv <= 0 || Lmax <= 0)
    return ECF8_ERR_INVALID_ARG;
  if ((Hq != 4 * Hkv && Hq != 8 * Hkv) || B * Hkv > 65535 || Lmax > (1 << 24))
    return ECF8_ERR_UNSUPPORTED;
  const int64_t S = (Lmax + kAttnChunk - 1) / kAttnChunk;
  if (work_floats < B * Hq * S * (kHeadDim + 2)) return ECF8_ERR_CAPACITY;
  if (!aligned(q, 4) || !aligned(k_cache, 16) || !aligned(v_cache, 4) || !aligned(work, 8) ||
      !aligned(out_q, 2) || (out_bf16 && !aligned(out_bf16, 4)))
    return ECF8_ERR_MISALIGNED;
  float *wm = work, *wl = work + B * Hq * S, *wacc = work + 2 * B * Hq * S;
  const dim3 grid((unsigned)(B * Hkv), (unsigned)S);
  const auto *qp = static_cast<const uint16_t *>(q);
  auto *kp = static_cast<uint16_t *>(const_cast<void *>(k_cache));
  auto *vp = static_cast<uint16_t *>(const_cast<void *>(v_cache));
  const AttnFused none{};
  if (Hq == 4 * Hkv)
    attn_split_kernel<4, false><<<grid, 64 * kAttnWaves, 0, as_stream(stream)>>>(
        qp, kp, vp, pos, Hkv, (int)Lmax, (int)S, wm, wl, wacc, none);
  else
    attn_split_kernel<8, false><<<grid, 64 * kAttnWaves, 0, as_stream(stream)>>>(
        qp, kp, vp, pos, Hkv, (int)Lmax, (int)S, wm, wl, wacc, none);
  attn_combine_kernel<<<(unsigned)(B * Hq), 64, 0, as_stream(stream)>>>(
      wm, wl, wacc, pos, (int)Lmax, (int)S, Hq, static_cast<uint8_t *>(out_q), out_scale,
      static_cast<uint16_t *>(out_bf16));
  return launched();
}

extern "C" int ecf8_decode_attention_fused(const void *qkv, int64_t B, int Hq, int Hkv,
                                           const void *q_norm, const void *k_norm, float eps,
                                           const float *cos_t, const float *sin_t, const int *pos,
                                           int64_t Lmax, void *k_cache, void *v_cache,
                                           float *work, int64_t work_floats, void *out_q,
                                           float *out_scale, void *out_bf16, void *stream) {
  if (!qkv || !q_norm || !k_norm || !cos_t || !sin_t || !pos || !k_cache || !v_cache || !work ||
      !out_q || !out_scale || B <= 0 || Hq <= 0 || Hkv <= 0 || Lmax <= 0)
    return ECF8_ERR_INVALID_ARG;
  if ((Hq != 4 * Hkv && Hq != 8 * Hkv) || B * Hkv > 65535 || Lmax > (1 << 24))
    return ECF8_ERR_UNSUPPORTED;
  const int64_t S = (Lmax + kAttnChunk - 1) / kAttnChunk;
  if (work_floats < B * Hq * S * (kHeadDim + 2)) return ECF8_ERR_CAPACITY;
  if (!aligned(qkv, 4) || !aligned(q_norm, 4) || !aligned(k_norm, 4) || !aligned(k_cache, 16) ||
      !aligned(v_cache, 4) || !aligned(work, 8) || !aligned(out_q, 2) ||
      (out_bf16 && !aligned(out_bf16, 4)))
    return ECF8_ERR_MISALIGNED;
  float *wm = work, *wl = work + B * Hq * S, *wacc = work + 2 * B * Hq * S;
  const AttnFused fu{static_cast<const uint16_t *>(qkv), static_cast<const uint16_t *>(q_norm),
                     static_cast<const uint16_t *>(k_norm), eps, cos_t, sin_t};
  const dim3 grid((unsigned)(B * Hkv), (unsigned)S);
  auto *kp = static_cast<uint16_t *>(k_cache);
  auto *vp = static_cast<uint16_t *>(v_cache);
  if (Hq == 4 * Hkv)
    attn_split_kernel<4, true><<<grid, 64 * kAttnWaves, 0, as_stream(stream)>>>(
        nullptr, kp, vp, pos, Hkv, (int)Lmax, (int)S, wm, wl, wacc, fu);
  else
    attn_split_kernel<8, true><<<grid, 64 * kAttnWaves, 0, as_stream(stream)>>>(
        nullptr, kp, vp, pos, Hkv, (int)Lmax, (int)S, wm, wl, wacc, fu);
  attn_combine_kernel<<<(unsigned)(B * Hq), 64, 0, as_stream(stream)>>>(
      wm, wl, wacc, pos, (int)Lmax, (int)S, Hq, static_cast<uint8_t *>(out_q), out_scale,
      static_cast<uint16_t *>(out_bf16));
  return launched();
}

extern "C" int ecf8_moe_route(const void *x, const void *router_w, int64_t M, int64_t H, int E,
                              int top_k, float *logits, int *topk_idx, float *topk_w,
                              void *stream) {
  if (!x || !router_w || !logits || !topk_idx || !topk_w || M <= 0 || H <= 0 || E <= 0 ||
      top_k <= 0)
    return ECF8_ERR_INVALID_ARG;
  if (H % 512 || H > (1 << 20) || E > 256 || top_k > 16 || top_k > E || M > (1 << 16))
    return ECF8_ERR_UNSUPPORTED;
  if (!aligned(x, 16) || !aligned(router_w, 16) || !aligned(logits, 4) || !aligned(topk_idx, 4) ||
      !aligned(topk_w, 4))
    return ECF8_ERR_MISALIGNED;
  moe_logits_kernel<<<dim3((unsigned)((E + 3) / 4), (unsigned)((M + 3) / 4)), 256, 0,
                      as_stream(stream)>>>(static_cast<const uint16_t *>(x),
                                           static_cast<const uint16_t *>(router_w), (int)M,
                                           (int)H, E, logits);
  moe_topk_kernel<<<(unsigned)((M + 3) / 4), 256, 0, as_stream(stream)>>>(logits, (int)M, E,
                                                                          top_k, topk_idx, topk_w);
  return launched();
}

extern "C" int ecf8_moe_group(const int *topk_idx, const float *topk_w, int64_t M, int top_k, int E,
                              int *offsets, int *active, int *n_active, int *pair_tok,
                              float *pair_w, int *pair_pos, int *select, void *stream) {
  if (!topk_idx || !topk_w || !offsets || !active || !n_active || !pair_tok || !pair_w ||
      !pair_pos || M <= 0 || top_k <= 0 || E <= 0)
    return ECF8_ERR_INVALID_ARG;
  if (M * top_k > 8192 || E > 256) return ECF8_ERR_UNSUPPORTED;
  moe_group_kernel<<<1, 1024, 0, as_stream(stream)>>>(topk_idx, topk_w, (int)(M * top_k), top_k, E,
                                                     offsets, active, n_active, pair_tok, pair_w,
                                                     pair_pos, select);
  return launched();
}

extern "C" int ecf8_moe_linear_pairs(const void *aq, const float *as, const int *row_of,
                                     const int *offsets, const int *active, const int *n_active,
                                     int n_experts, const void *const *weights,
                                     const float *const *weight_scales, int n_segs,
                                     int64_t seg_n, int64_t K, int weight_layout, int64_t pairs,
                                     void *out, int64_t ldo, void *stream) {
  if (!aq || !as || !offsets || !active || !n_active || !weights || !weight_scales || !out ||
      n_experts <= 0 || n_segs < 1 || n_segs > ECF8_LINEAR_MAX_SEGS || seg_n <= 0 || K <= 0 ||
      (weight_layout != ECF8_WEIGHT_ROWS && weight_layout != ECF8_WEIGHT_TILES))
    return ECF8_ERR_INVALID_ARG;
  if (seg_n % kGroup || K % kGroup || K > (1 << 20) || n_segs * seg_n > (1 << 20) ||
      n_experts > 65535)
    return ECF8_ERR_UNSUPPORTED;
  if (ldo < n_segs * seg_n) return ECF8_ERR_CAPACITY;
  if (!aligned(aq, 16) || !aligned(as, 4) || !aligned(out, 4) || !aligned(weights, 8) ||
      !aligned(weight_scales, 8))
    return ECF8_ERR_MISALIGNED;
  MoeLinear a{static_cast<const uint8_t *>(aq), as, row_of, offsets, active, n_active,
              reinterpret_cast<const uint64_t *>(weights),
              reinterpret_cast<const uint64_t *>(weight_scales), static_cast<uint16_t *>(out),
              n_segs, (int)seg_n, (int)K, (int)ldo, weight_layout == ECF8_WEIGHT_TILES};
  const int64_t groups = K / kGroup;
  // Four rows per expert and more: the form that reads an expert's weights
  // once per 64 (32) rows, while its three or four partial sums fit the
  // registers.  MI355X, 128 experts, row-major weights, us for gate/up K =
  // 2048 and down K = 768, 16-row form against this one: 32 tokens (2 rows)
  // 88.2 / 40.8 against 99.4 / 42.9, 48 tokens 103.9 / 46.2 against 102.3 /
  // 45.7, 64 tokens 114.5 / 49.0 against 103.9 / 49.6, 128 tokens 144.7 /
  // 53.3 against 106.8 / 51.4, 1024 tokens 787 / 249 against 229 / 144.  64
  // tokens on eight experts (64 rows each): 26.3 / 16.6 against 23.3 / 16.6,
  // tile-layout weights 19.0 / 13.1 against 20.1 / 13.5.
  // 32 rows for down keep two workgroups per CU, its loads' latency being
  // most of its two stages (64 rows: 86.0 against 92.4 us at 512 tokens, but
  // 67.5 against 48.6 at 128); the four-part form spills at 128 VGPRs.
  if (pairs >= 4 * (int64_t)n_experts && groups <= ECF8_MOE_FOUR_WAVE_GROUPS) {
    // each expert's first rows, then at most pairs / 64 (32) blocks past them
    // (a few stand for more, in turns)
    const int64_t past = pairs / (groups == 6 ? 32 : 64), most = 65536 - n_experts;
    const dim3 strips((unsigned)(n_segs * seg_n / 128),
                      (unsigned)(n_experts + (past < 1 ? 1 : past > most ? most : past)));
    if (groups == 6)
      moe_rows_kernel<3, 2><<<strips, 512, 0, as_stream(stream)>>>(a, n_experts);
    else
      moe_rows_kernel<4, 4><<<strips, 512, 0, as_stream(stream)>>>(a, n_experts);
    return launched();
  }
  const dim3 grid((unsigned)(n_segs * seg_n / 16), (unsigned)n_experts);
  // each wave's share of the K groups in one batch of loads where it fits.
  // On MI355X, Qwen3-30B-A3B experts at 16 tokens (48 layers back to back):
  // gate/up (K = 2048) 48.5 us per layer at four waves of four groups
  // against 53.4 at eight of two; down (K = 768) 23.7 us at three waves of
  // two groups against 26.9 at four (two, two, one, one)
  static_assert(ECF8_MOE_FOUR_WAVE_GROUPS == 16, "four waves of at most four groups");
  if (groups == 6)
    moe_linear16_kernel<3, 2><<<grid, 192, 0, as_stream(stream)>>>(a);
  else if (groups <= 8)
    moe_linear16_kernel<4, 2><<<grid, 256, 0, as_stream(stream)>>>(a);
  else if (groups <= ECF8_MOE_FOUR_WAVE_GROUPS)
    moe_linear16_kernel<4, 4><<<grid, 256, 0, as_stream(stream)>>>(a);
  else
    moe_linear16_kernel<8, 4><<<grid, 512, 0, as_stream(stream)>>>(a);
  return launched();
}

extern "C" int ecf8_moe_linear(const void *aq, const float *as, const int *row_of,
                               const int *offsets, const int *active, const int *n_active,
                               int n_experts, const void *const *weights,
                               const float *const *weight_scales, int n_segs, int64_t seg_n,
                               int64_t K, int weight_layout, void *out, int64_t ldo,
                               void *stream) {
  return ecf8_moe_linear_pairs(aq, as, row_of, offsets, active, n_active, n_experts, weights,
                               weight_scales, n_segs, seg_n, K, weight_layout, 0, out, ldo,
                               stream);
}

extern "C" int ecf8_moe_combine(const void *down, int64_t ldd, const int *pair_pos,
                                const float *pair_w, int64_t M, int top_k, int64_t H, void *out,
                                void *stream) {
  if (!down || !pair_pos || !pair_w || !out || M <= 0 || top_k <= 0 || H <= 0 || ldd < H)
    return ECF8_ERR_INVALID_ARG;
  if (H % 8 || ldd % 8 || M > 0x7fffffff) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(down, 16) || !aligned(out, 16)) return ECF8_ERR_MISALIGNED;
  moe_combine_kernel<<<(unsigned)M, 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t *>(down), (int)ldd, pair_pos, pair_w, top_k, (int)H,
      static_cast<uint16_t *>(out));
  return launched();
}
