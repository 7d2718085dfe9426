// Attention of many queries per head on gfx950: the prompt's causal
// attention (grouped-query, over the KV caches) and the DiT's attention
// over text and image tokens, with the passes that prepare their operands.
// Head dimension 128, bf16 operands, fp32 scores, softmax and sums.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "ecf8.h"
#include "ecf8_attn.h"

namespace {

constexpr int kD = 128;      // head dimension
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kBlock = 64;   // keys per step of the attention kernel
constexpr int kQueries = 128;  // queries per workgroup: four waves of 32

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bf16_f32(uint32_t h16) { return __uint_as_float(h16 << 16); }
// two fp32 -> packed bf16, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const v2bf v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// Eight bf16 with their infinities and NaNs replaced by zeros.
__device__ __forceinline__ u32x4 finite_or_zero(u32x4 v) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if ((v[j] & 0x7f80u) == 0x7f80u) v[j] &= 0xffff0000u;
    if ((v[j] & 0x7f800000u) == 0x7f800000u) v[j] &= 0xffffu;
  }
  return v;
}

// Workgroup barrier that waits for LDS only (a __syncthreads would also
// wait for the prefetched global loads).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt((0x3F & 15) | (0x3 << 14) | (0x7 << 4) | (0x0 << 8));  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Packed keys and values.  Per (batch, kv head), tokens padded with zero
// rows to a multiple of 64:
//   keys:   per 32 tokens 8 KB: 16-byte unit kk * 64 + 32 h + r holds token
//           r's dims [16 kk + 8 h, +8) -- lane 32 h + r's A operand of the
//           kk-th v_mfma_f32_32x32x16_bf16;
//   values: per 16 tokens 4 KB: unit dt * 64 + 32 h + d holds dim 32 dt + d
//           of tokens 4 h + {0..3} and 8 + 4 h + {0..3} -- the A operand of
//           the transposed value tile, with its K order that of the score
//           tile's registers (row 8 (i / 4) + 4 h + i % 4), so the
//           probabilities feed the second product as they stand.
__device__ __forceinline__ size_t packed_key(int t, int kk, int h) {
  return (size_t)(t >> 5) * 4096 + (size_t)((kk * 64 + 32 * h + (t & 31)) * 8);
}

// Writes 32 tokens' values (s_v: [token][dim], kPad elements a row) as two
// packed 16-token blocks at dst.
constexpr int kPad = kD + 2;  // odd dword stride
__device__ __forceinline__ void store_values(const uint16_t (*s_v)[kPad], uint16_t *dst) {
  for (int u = threadIdx.x; u < 512; u += 256) {
    const int blk = u >> 8, d = 32 * ((u >> 6) & 3) + (u & 31), h = (u >> 5) & 1;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = 16 * blk + (j < 2 ? 4 * h + 2 * j : 8 + 4 * h + 2 * j - 4);
      w[j] = (uint32_t)s_v[t][d] | ((uint32_t)s_v[t + 1][d] << 16);
    }
    *reinterpret_cast<u32x4 *>(dst + (size_t)u * 8) = u32x4{w[0], w[1], w[2], w[3]};
  }
}

// ---------------------------------------------------------- attention

struct Attn {
  const uint16_t *q;        // bf16 [B * Hq, T, 128]
  const uint16_t *k, *v;    // packed, [B * Hkv, Tp, 128]
  uint16_t *out;            // bf16, row (b * T + t), head columns 128 head
  int64_t out_stride;       // elements per output row
  int T, Tp, Hq, group, tiles, heads;  // heads = B * Hq
  float scale;              // of the scores (base-2 exponent's factor included)
};

// One workgroup: 128 queries of one head, 32 per wave, all keys in blocks
// of 64.  Scores are computed transposed (S^T = K Q^T), so a lane holds one
// query's scores of 32 keys per block: the running maximum and sum need one
// exchange with lane ^ 32, and the exponentials are the second product's B
// operand in place (O^T += V^T P^T).  Keys and values come packed in MFMA
// order, so both the copies to LDS and the LDS reads are 16 consecutive
// bytes per lane.  A block's keys and values are loaded a block ahead into
// registers and written to the other LDS buffer: one barrier per block.
//
// kExact (the prompt): a probability enters the second product as the sum
// of three bf16 parts, which hold its 24 mantissa bits, so that product is
// that of the fp32 probabilities (an infinite value times a probability
// above zero is infinite, as there).  Otherwise probabilities are rounded to
// bf16, as the DiT's softmax does.
//
// Bound by the MFMA pipe and the exponentials (16 of each per 32 x 32 tile
// per wave: ~512 and ~450 cycles).  MI355X,
// causal with three parts: 1 x 32 heads x 2048 queries 136 us with the packing
// pass (fp32 library products, mask and softmax passes before: 1272 us),
// 16 x 32 x 128 23 us (219).
template <bool kCausal, bool kExact>
__global__ __launch_bounds__(256, 2) void flash_kernel(Attn a) {
  __shared__ u32x4 s_k[2][kBlock * 16];
  __shared__ u32x4 s_v[2][kBlock * 16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, h = lane >> 5;
  // workgroups are dealt to the 8 XCDs round robin: a head's query tiles
  // go to one XCD, whose L2 then holds the head's keys and values; long
  // causal tiles first
  int id = blockIdx.x;
  if (a.heads % 8 == 0) id = (id % 8) * (a.heads / 8 * a.tiles) + id / 8;
  const int head = id / a.tiles;
  int tile = id % a.tiles;
  if (kCausal) tile = a.tiles - 1 - tile;
  const int q0 = tile * kQueries + 32 * wave;
  const int qi = min(q0 + r, a.T - 1);  // rows past T repeat the last, unstored
  const int kvh = head / a.group;

  v8bf qf[8];
  {
    const uint16_t *qp = a.q + ((size_t)head * a.T + qi) * kD + 8 * h;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) qf[kk] = *reinterpret_cast<const v8bf *>(qp + 16 * kk);
  }
  const u32x4 *kp = reinterpret_cast<const u32x4 *>(a.k + (size_t)kvh * a.Tp * kD);
  const u32x4 *vp = reinterpret_cast<const u32x4 *>(a.v + (size_t)kvh * a.Tp * kD);
  const int last = kCausal ? min(tile * kQueries + kQueries, a.T) : a.T;  // keys in use
  const int blocks = (last + kBlock - 1) / kBlock;

  u32x4 kr[4], vr[4];
  auto load = [&](int b, u32x4 (&kr)[4], u32x4 (&vr)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      kr[i] = kp[(size_t)b * (kBlock * 16) + 256 * i + threadIdx.x];
      vr[i] = vp[(size_t)b * (kBlock * 16) + 256 * i + threadIdx.x];
    }
  };

  v16f o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  float m = -INFINITY, l = 0.f;  // of query r: both lanes hold the same m

  // one block's keys and values, in LDS or packed in memory
  auto step = [&](int b, const u32x4 *k, const u32x4 *v, auto careful) {
    const int key0 = b * kBlock;
    if (q0 >= a.T || (kCausal && key0 > q0 + 31)) return;  // uniform per wave

    v16f s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[t][i] = 0.f;
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        const v8bf kf = *reinterpret_cast<const v8bf *>(&k[t * 512 + kk * 64 + lane]);
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[kk], s[t], 0, 0, 0);
      }
    }
    if (key0 + kBlock > a.T || (kCausal && key0 + kBlock - 1 > q0)) {  // uniform
      const int lim = kCausal ? qi : a.T - 1;  // last key of this lane's query
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (key0 + 32 * t + 8 * (i >> 2) + 4 * h + (i & 3) > lim) s[t][i] = -INFINITY;
    }
    float bm = s[0][0];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) bm = fmaxf(bm, s[t][i]);
    const auto hm = __builtin_amdgcn_permlane32_swap(__float_as_uint(bm), __float_as_uint(bm),
                                                     false, false);
    const float mn = fmaxf(m, fmaxf(__uint_as_float(hm[0]), __uint_as_float(hm[1])));
    if (__any(mn > m)) {  // uniform: some query's maximum moved
      float f = __builtin_amdgcn_exp2f((m - mn) * a.scale);
      if (careful && m == mn) f = 1.f;  // both may be -inf
      l *= f;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] *= f;
      m = mn;
    }
    const float top = careful && m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[t][i] = __builtin_amdgcn_exp2f((s[t][i] - top) * a.scale);
        l += s[t][i];
      }
#pragma unroll
    for (int g = 0; g < 4; ++g) {  // 16 keys a step
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) p[j] = s[g >> 1][8 * (g & 1) + j];
      constexpr int kParts = kExact ? 3 : 1;
      u32x4 pf[kParts];
#pragma unroll
      for (int q = 0; q < kParts; ++q) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t w = pack_bf16(p[2 * j], p[2 * j + 1]);
          pf[q][j] = w;
          p[2 * j] -= bf16_f32(w & 0xffffu);      // exact
          p[2 * j + 1] -= __uint_as_float(w & 0xffff0000u);
        }
      }
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const u32x4 vf = v[g * 256 + d * 64 + lane];
        const u32x4 vs = careful ? finite_or_zero(vf) : vf;
#pragma unroll
        for (int q = kParts - 1; q >= 0; --q)  // small parts first
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(v8bf, q ? vs : vf), __builtin_bit_cast(v8bf, pf[q]), o[d], 0, 0,
              0);
      }
    }
  };

  load(0, kr, vr);
  for (int b = 0; b < blocks; ++b) {
    const int buf = b & 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s_k[buf][256 * i + threadIdx.x] = kr[i];
      s_v[buf][256 * i + threadIdx.x] = vr[i];
    }
    // this block is in LDS; the other buffer was last read in block b - 1,
    // before every wave's arrival here
    lds_barrier();
    if (b + 1 < blocks) load(b + 1, kr, vr);
    step(b, s_k[buf], s_v[buf], std::false_type());
  }
  if constexpr (kExact) {
    // The smaller parts of a probability, zero or below zero, make NaN of an
    // infinite value, and a block whose scores are all -inf makes NaN of the
    // sums.  Then once more, each wave by itself.
    bool nan = l != l;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) nan |= o[d][i] != o[d][i];
    if (__any(nan)) {  // uniform
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
      m = -INFINITY, l = 0.f;
      for (int b = 0; b < blocks; ++b)
        step(b, kp + (size_t)b * (kBlock * 16), vp + (size_t)b * (kBlock * 16), std::true_type());
    }
  }
  l += __shfl_xor(l, 32);
  if (q0 + r >= a.T) return;
  const float inv = 1.f / l;
  const int batch = head / a.Hq;
  uint16_t *op = a.out + ((size_t)batch * a.T + qi) * a.out_stride +
                 (size_t)(head % a.Hq) * kD + 4 * h;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x2 *>(op + 32 * d + 8 * i) =
          u32x2{pack_bf16(o[d][4 * i] * inv, o[d][4 * i + 1] * inv),
                pack_bf16(o[d][4 * i + 2] * inv, o[d][4 * i + 3] * inv)};
}

// ------------------------------------------- attention without a mask (DiT)

constexpr int kPairQueries = 256;  // queries per workgroup: eight waves of 32

// flash_kernel's computation (no mask, probabilities rounded to bf16) with
// the two waves of a SIMD taking turns, a barrier apart: one runs its
// products (the values' of the last block, then the scores' of this one;
// operands are read from LDS eight products ahead) while the other runs its
// softmax.
// Keys and values of a block go through registers to a ring of three LDS
// stages: block b + 1 is written in the phase in which the first four waves
// run block b's softmax and the others its products, when its stage was last
// read two phases before.
//
// Bound by the softmax phase (per wave and block 1024 cycles of MFMA, ~1100
// of exponentials and other vector instructions, which share the SIMD's
// issue).  MI355X, 24 heads x 4608 tokens: 261 us (the MFMAs alone 127 us at
// the clock it ran at; the grid's second round of workgroups is 0.69 full),
// flash_kernel 327 us.
__global__ __launch_bounds__(512) void pair_attention_kernel(Attn a) {
  __shared__ u32x4 s_k[3][kBlock * 16];
  __shared__ u32x4 s_v[3][kBlock * 16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool behind = wave >= 4;  // a phase behind the others
  const int r = lane & 31, h = lane >> 5;
  // a head's query tiles go to one XCD (see flash_kernel)
  int id = blockIdx.x;
  if (a.heads % 8 == 0) id = (id % 8) * (a.heads / 8 * a.tiles) + id / 8;
  const int head = id / a.tiles;
  const int q0 = (id % a.tiles) * kPairQueries + 32 * wave;
  const int qi = min(q0 + r, a.T - 1);  // rows past T repeat the last, unstored
  const bool used = q0 < a.T;           // uniform

  v8bf qf[8];
  {
    const uint16_t *qp = a.q + ((size_t)head * a.T + qi) * kD + 8 * h;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) qf[kk] = *reinterpret_cast<const v8bf *>(qp + 16 * kk);
  }
  const u32x4 *kp = reinterpret_cast<const u32x4 *>(a.k + (size_t)head * a.Tp * kD);
  const u32x4 *vp = reinterpret_cast<const u32x4 *>(a.v + (size_t)head * a.Tp * kD);
  const int blocks = (a.T + kBlock - 1) / kBlock;

  u32x4 kr[2], vr[2];
  auto load = [&](int b) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      kr[i] = kp[(size_t)b * (kBlock * 16) + 512 * i + threadIdx.x];
      vr[i] = vp[(size_t)b * (kBlock * 16) + 512 * i + threadIdx.x];
    }
  };
  auto write = [&](int st) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      s_k[st][512 * i + threadIdx.x] = kr[i];
      s_v[st][512 * i + threadIdx.x] = vr[i];
    }
  };
  auto phase = [] {
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  v16f o[4], s[2];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  float m = -INFINITY, l = 0.f;  // of query r: both lanes hold the same m
  u32x4 pf[4] = {};              // the probabilities of 16 keys each

  auto values = [&](int st) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const v8bf vf = *reinterpret_cast<const v8bf *>(&s_v[st][g * 256 + d * 64 + lane]);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, __builtin_bit_cast(v8bf, pf[g]), o[d],
                                                       0, 0, 0);
      }
  };
  auto scores = [&](int st) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[t][i] = 0.f;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const v8bf kf = *reinterpret_cast<const v8bf *>(&s_k[st][t * 512 + kk * 64 + lane]);
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[kk], s[t], 0, 0, 0);
      }
  };
  // n products whose operands are read from LDS kAhead products before
  auto order = [](auto n) {
    constexpr int kN = decltype(n)::value, kAhead = 8;
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);  // LDS reads
#pragma unroll
    for (int i = 0; i < kN - kAhead; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x8, kAhead, 0);
  };

  load(0);
  write(0);
  if (blocks > 1) load(1);
  phase();
  // block b + 1 to its stage, block b + 2 on its way
  auto stage = [&](int b, int st) {
    if (b + 1 < blocks) {
      write(st);
      if (b + 2 < blocks) load(b + 2);
    }
  };
  if (behind) {
    phase();
    stage(0, 1);
  }
  if (used) {
    scores(0);
    order(std::integral_constant<int, 16>());
  }
  phase();
  int st = 0;  // stage of block b
  for (int b = 0;; ++b) {
    const int st1 = st == 2 ? 0 : st + 1, st2 = st == 0 ? 2 : st - 1;  // of b + 1, b + 2
    // softmax (the other four waves: products)
    if (!behind) stage(b, st1);
    __builtin_amdgcn_s_setprio(1);
    if (used) {
      const int key0 = b * kBlock;
      if (key0 + kBlock > a.T) {  // uniform: keys past the last
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (key0 + 32 * t + 8 * (i >> 2) + 4 * h + (i & 3) >= a.T) s[t][i] = -INFINITY;
      }
      float bm = s[0][0];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) bm = fmaxf(bm, s[t][i]);
      const auto hm = __builtin_amdgcn_permlane32_swap(__float_as_uint(bm), __float_as_uint(bm),
                                                       false, false);
      const float mn = fmaxf(m, fmaxf(__uint_as_float(hm[0]), __uint_as_float(hm[1])));
      // uniform: some query's maximum moved by more than a factor 2^8 of its
      // exponentials.  Below that m stays (nothing overflows, the quotient
      // of the sums is the same); most blocks would rescale for a query.
      if (__any(mn > m + 8.f)) {
        const float f = __builtin_amdgcn_exp2f(m - mn);
        l *= f;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[d][i] *= f;
        m = mn;
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[t][i] = __builtin_amdgcn_exp2f(s[t][i] - m);
          l += s[t][i];
        }
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          pf[g][j] = pack_bf16(s[g >> 1][8 * (g & 1) + 2 * j], s[g >> 1][8 * (g & 1) + 2 * j + 1]);
    }
    __builtin_amdgcn_s_setprio(0);
    phase();
    if (b + 1 == blocks) break;
    // products (the other four waves: softmax)
    if (behind) stage(b + 1, st2);
    if (used) {
      values(st);
      scores(st1);
      order(std::integral_constant<int, 32>());
    }
    phase();
    st = st1;
  }
  if (!behind) phase();
  if (!used) return;
  values(st);
  order(std::integral_constant<int, 16>());
  l += __shfl_xor(l, 32);
  if (q0 + r >= a.T) return;
  const float inv = 1.f / l;
  uint16_t *op = a.out + ((size_t)(head / a.Hq) * a.T + qi) * a.out_stride +
                 (size_t)(head % a.Hq) * kD + 4 * h;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x2 *>(op + 32 * d + 8 * i) =
          u32x2{pack_bf16(o[d][4 * i] * inv, o[d][4 * i + 1] * inv),
                pack_bf16(o[d][4 * i + 2] * inv, o[d][4 * i + 3] * inv)};
}

// --------------------------------------------------- packing keys, values

// 32 tokens of one (batch, kv head): the caches' rows [Lmax, 128] -> packed
// keys and values; rows past T become zero.
__global__ __launch_bounds__(256) void pack_kv_kernel(const uint16_t *__restrict__ kc,
                                                      const uint16_t *__restrict__ vc, int T,
                                                      int Tp, int64_t Lmax,
                                                      uint16_t *__restrict__ ko,
                                                      uint16_t *__restrict__ vo) {
  __shared__ uint16_t s_v[32][kPad];
  const int tile = blockIdx.x % (Tp / 32);
  const size_t bh = blockIdx.x / (Tp / 32);
  const int row = threadIdx.x >> 3, c = threadIdx.x & 7;
  const int t = 32 * tile + row;
  u32x4 k0 = {}, k1 = {}, v0 = {}, v1 = {};
  if (t < T) {
    const size_t at = (bh * (size_t)Lmax + t) * kD + 16 * c;
    k0 = *reinterpret_cast<const u32x4 *>(kc + at);
    k1 = *reinterpret_cast<const u32x4 *>(kc + at + 8);
    v0 = *reinterpret_cast<const u32x4 *>(vc + at);
    v1 = *reinterpret_cast<const u32x4 *>(vc + at + 8);
  }
  uint16_t *kb = ko + bh * (size_t)Tp * kD;
  *reinterpret_cast<u32x4 *>(kb + packed_key(t, c, 0)) = k0;
  *reinterpret_cast<u32x4 *>(kb + packed_key(t, c, 1)) = k1;
  uint32_t *sv = reinterpret_cast<uint32_t *>(&s_v[row][16 * c]);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sv[j] = v0[j];
    sv[4 + j] = v1[j];
  }
  __syncthreads();
  store_values(s_v, vo + (bh * (size_t)Tp + 32 * (size_t)tile) * kD);
}

// ------------------------------------------------------------ DiT operands

__device__ __forceinline__ void load16(const uint16_t *p, float (&v)[16]) {
  const u32x4 a = *reinterpret_cast<const u32x4 *>(p), b = *reinterpret_cast<const u32x4 *>(p + 8);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[2 * j] = bf16_f32(a[j] & 0xffffu);
    v[2 * j + 1] = __uint_as_float(a[j] & 0xffff0000u);
    v[8 + 2 * j] = bf16_f32(b[j] & 0xffffu);
    v[8 + 2 * j + 1] = __uint_as_float(b[j] & 0xffff0000u);
  }
}

// One stream's rows of the joint attention: the projection output (q heads,
// then k heads, then v heads) and the head norms' weights.
struct Stream {
  const uint16_t *qkv;
  const uint16_t *qn, *kn;
  int64_t row, batch;  // elements between rows and between batches
  int tokens;
};

// 32 tokens of one (batch, head): RMSNorm of the q and k heads and the
// rotary embedding of interleaved pairs, in fp32; q scaled, rounded to bf16
// and stored as rows, k and v packed for flash_kernel.  Tokens of `first`
// come before those of `second`.  Eight threads a token, 16 dims each.
// HBM bounds it: 6 bytes read and written per element where separate passes
// moved fp32 copies of each.
__global__ __launch_bounds__(256) void dit_qkv_kernel(Stream first, Stream second, int H, int T,
                                                      int Tp, float eps, float scale,
                                                      const float *__restrict__ cosv,
                                                      const float *__restrict__ sinv,
                                                      uint16_t *__restrict__ qo,
                                                      uint16_t *__restrict__ ko,
                                                      uint16_t *__restrict__ vo) {
  __shared__ uint16_t s_v[32][kPad];
  const int tiles = Tp / 32;
  const int tile = blockIdx.x % tiles;
  const int bh = blockIdx.x / tiles, b = bh / H, head = bh % H;
  const int row = threadIdx.x >> 3, c = threadIdx.x & 7;
  const int t = 32 * tile + row;
  u32x4 k0 = {}, k1 = {}, v0 = {}, v1 = {};
  if (t < T) {
    const bool in = t < first.tokens;
    const Stream &s = in ? first : second;
    const uint16_t *p = s.qkv + (size_t)b * s.batch + (size_t)(in ? t : t - first.tokens) * s.row +
                        (size_t)head * kD + 16 * c;
    float q[16], k[16];
    load16(p, q);
    load16(p + (size_t)H * kD, k);
    const u32x4 *vp = reinterpret_cast<const u32x4 *>(p + (size_t)2 * H * kD);
    v0 = vp[0];
    v1 = vp[1];
    float co[8], si[8];
#pragma unroll
    for (int j = 0; j < 8; j += 4) {
      const float4 cv = *reinterpret_cast<const float4 *>(cosv + (size_t)t * 64 + 8 * c + j);
      const float4 sv = *reinterpret_cast<const float4 *>(sinv + (size_t)t * 64 + 8 * c + j);
      co[j] = cv.x, co[j + 1] = cv.y, co[j + 2] = cv.z, co[j + 3] = cv.w;
      si[j] = sv.x, si[j + 1] = sv.y, si[j + 2] = sv.z, si[j + 3] = sv.w;
    }
    auto norm_rope = [&](float (&x)[16], const uint16_t *nw, float sc) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) ss = fmaf(x[i], x[i], ss);
      ss += __shfl_xor(ss, 1);
      ss += __shfl_xor(ss, 2);
      ss += __shfl_xor(ss, 4);
      const float rs = rsqrtf(ss / (float)kD + eps);
      float w[16];
      load16(nw + 16 * c, w);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x0 = x[2 * j] * rs * w[2 * j], x1 = x[2 * j + 1] * rs * w[2 * j + 1];
        x[2 * j] = (x0 * co[j] - x1 * si[j]) * sc;
        x[2 * j + 1] = (x0 * si[j] + x1 * co[j]) * sc;
      }
    };
    norm_rope(q, s.qn, scale);
    norm_rope(k, s.kn, 1.f);
    u32x4 q0, q1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      q0[j] = pack_bf16(q[2 * j], q[2 * j + 1]);
      q1[j] = pack_bf16(q[8 + 2 * j], q[8 + 2 * j + 1]);
      k0[j] = pack_bf16(k[2 * j], k[2 * j + 1]);
      k1[j] = pack_bf16(k[8 + 2 * j], k[8 + 2 * j + 1]);
    }
    u32x4 *qp = reinterpret_cast<u32x4 *>(qo + ((size_t)bh * T + t) * kD + 16 * c);
    qp[0] = q0;
    qp[1] = q1;
  }
  uint16_t *kb = ko + (size_t)bh * Tp * kD;
  *reinterpret_cast<u32x4 *>(kb + packed_key(t, c, 0)) = k0;
  *reinterpret_cast<u32x4 *>(kb + packed_key(t, c, 1)) = k1;
  uint32_t *sv = reinterpret_cast<uint32_t *>(&s_v[row][16 * c]);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sv[j] = v0[j];
    sv[4 + j] = v1[j];
  }
  __syncthreads();
  store_values(s_v, vo + ((size_t)bh * Tp + 32 * (size_t)tile) * kD);
}

// ------------------------------------------------- DiT elementwise passes
//
// Each replaces several library passes over fp32 or bf16 copies by one that
// reads its inputs once and writes its output once (HBM-bound), with the
// roundings of the passes it replaces.

__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f[2 * j] = bf16_f32(v[j] & 0xffffu);
    f[2 * j + 1] = __uint_as_float(v[j] & 0xffff0000u);
  }
}

__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
  return u32x4{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]),
               pack_bf16(f[6], f[7])};
}

// The sum over the 256 threads, in every thread, in a fixed order.
__device__ __forceinline__ float block_sum(float v, float *part) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();  // part may still be read from the last sum
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  return (part[0] + part[1]) + (part[2] + part[3]);
}

// out = bf16(LayerNorm(x) * (1 + scale) + shift) per row of C <= 2048 kV,
// mean and variance in fp32 from the row held in registers.
template <int kV>
__global__ __launch_bounds__(256) void modulate_kernel(const uint16_t *__restrict__ x, int rows,
                                                       int C, const uint16_t *__restrict__ shift,
                                                       int64_t shift_batch,
                                                       const uint16_t *__restrict__ scale,
                                                       int64_t scale_batch, float eps,
                                                       uint16_t *__restrict__ out) {
  __shared__ float part[4];
  const size_t m = blockIdx.x;
  const size_t b = m / (size_t)rows;
  float v[kV][8];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    const int c = 2048 * i + 8 * threadIdx.x;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    if (c < C) unpack8(*reinterpret_cast<const u32x4 *>(x + m * C + c), v[i]);
#pragma unroll
    for (int j = 0; j < 8; ++j) sum += v[i][j];
  }
  const float mean = block_sum(sum, part) / (float)C;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    if (2048 * i + 8 * (int)threadIdx.x >= C) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[i][j] -= mean;
      sq = fmaf(v[i][j], v[i][j], sq);
    }
  }
  const float rs = rsqrtf(block_sum(sq, part) / (float)C + eps);
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    const int c = 2048 * i + 8 * threadIdx.x;
    if (c >= C) continue;
    float sh[8], sc[8];
    unpack8(*reinterpret_cast<const u32x4 *>(shift + b * shift_batch + c), sh);
    unpack8(*reinterpret_cast<const u32x4 *>(scale + b * scale_batch + c), sc);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = v[i][j] * rs * (1.f + sc[j]) + sh[j];
    *reinterpret_cast<u32x4 *>(out + m * C + c) = pack8(v[i]);
  }
}

// out = bf16(x + bf16(gate * y)) per row of C, gate per batch.
__global__ __launch_bounds__(256) void gated_add_kernel(const uint16_t *__restrict__ x,
                                                        const uint16_t *__restrict__ gate,
                                                        int64_t gate_batch,
                                                        const uint16_t *__restrict__ y,
                                                        int64_t units, int rows, int C,
                                                        uint16_t *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // 8 elements
  if (i >= units) return;
  const int64_t m = i / (C / 8);
  const int c = 8 * (int)(i - m * (C / 8));
  float xf[8], gf[8], yf[8];
  unpack8(*reinterpret_cast<const u32x4 *>(x + 8 * i), xf);
  unpack8(*reinterpret_cast<const u32x4 *>(y + 8 * i), yf);
  unpack8(*reinterpret_cast<const u32x4 *>(gate + (m / rows) * gate_batch + c), gf);
#pragma unroll
  for (int j = 0; j < 8; ++j) xf[j] += bf16_f32(pack_bf16(gf[j] * yf[j], 0.f) & 0xffffu);
  *reinterpret_cast<u32x4 *>(out + 8 * i) = pack8(xf);
}

// out[m, :C] = bf16(gelu_tanh(x[m, :C])), both with a row stride: 0.5 x (1 +
// tanh(u)) = x / (1 + exp(-2 u)), u = sqrt(2 / pi) (x + 0.044715 x^3).
__global__ __launch_bounds__(256) void gelu_kernel(const uint16_t *__restrict__ x, int64_t x_row,
                                                   int64_t units, int C,
                                                   uint16_t *__restrict__ out, int64_t out_row) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= units) return;
  const int64_t m = i / (C / 8);
  const int c = 8 * (int)(i - m * (C / 8));
  float v[8];
  unpack8(*reinterpret_cast<const u32x4 *>(x + m * x_row + c), v);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float u = 0.7978845608028654f * (v[j] + 0.044715f * v[j] * v[j] * v[j]);
    v[j] = v[j] * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-2.f * kLog2e * u));
  }
  *reinterpret_cast<u32x4 *>(out + m * out_row + c) = pack8(v);
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }
inline bool aligned(const void *p, uintptr_t a) {
  return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0;
}
inline int launched() { return hipGetLastError() == hipSuccess ? ECF8_OK : ECF8_ERR_HIP; }
inline int64_t padded(int64_t T) { return (T + kBlock - 1) / kBlock * kBlock; }

}  // namespace

extern "C" int64_t ecf8_packed_kv_elements(int64_t B, int Hkv, int64_t T) {
  if (B <= 0 || Hkv <= 0 || T <= 0 || T > (1 << 24) || B > (1 << 24)) return -1;
  return B * Hkv * padded(T) * kD;
}

extern "C" int ecf8_prompt_attention(const void *q, const void *k_cache, const void *v_cache,
                                     int64_t B, int Hq, int Hkv, int64_t T, int64_t Lmax,
                                     void *k_packed, void *v_packed, void *out, void *stream) {
  if (!q || !k_cache || !v_cache || !k_packed || !v_packed || !out || B <= 0 || Hq <= 0 ||
      Hkv <= 0 || T <= 0 || Lmax < T)
    return ECF8_ERR_INVALID_ARG;
  const int64_t tiles = (T + kQueries - 1) / kQueries;
  const int64_t Tp = padded(T);
  if (Hq % Hkv || T > (1 << 24) || B > (1 << 24) || B * Hq * tiles > INT32_MAX ||
      B * Hkv * (Tp / 32) > INT32_MAX)
    return ECF8_ERR_UNSUPPORTED;
  if (!aligned(q, 16) || !aligned(k_cache, 16) || !aligned(v_cache, 16) ||
      !aligned(k_packed, 16) || !aligned(v_packed, 16) || !aligned(out, 8))
    return ECF8_ERR_MISALIGNED;
  pack_kv_kernel<<<(unsigned)(B * Hkv * (Tp / 32)), 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t *>(k_cache), static_cast<const uint16_t *>(v_cache), (int)T,
      (int)Tp, Lmax, static_cast<uint16_t *>(k_packed), static_cast<uint16_t *>(v_packed));
  const Attn a{static_cast<const uint16_t *>(q), static_cast<const uint16_t *>(k_packed),
               static_cast<const uint16_t *>(v_packed), static_cast<uint16_t *>(out),
               (int64_t)Hq * kD, (int)T, (int)Tp, Hq, Hq / Hkv, (int)tiles, (int)(B * Hq),
               kLog2e / sqrtf((float)kD)};
  flash_kernel<true, true><<<(unsigned)(B * Hq * tiles), 256, 0, as_stream(stream)>>>(a);
  return launched();
}

extern "C" int ecf8_dit_qkv(const ecf8_dit_stream *streams, int n_streams, int64_t B, int H,
                            float eps, float scale, const float *cos_t, const float *sin_t,
                            void *q, void *k_packed, void *v_packed, void *stream) {
  if (!streams || n_streams < 1 || n_streams > 2 || B <= 0 || H <= 0 || !cos_t || !sin_t || !q ||
      !k_packed || !v_packed)
    return ECF8_ERR_INVALID_ARG;
  Stream s[2] = {};
  int64_t T = 0;
  for (int i = 0; i < n_streams; ++i) {
    const ecf8_dit_stream &g = streams[i];
    if (!g.qkv || !g.q_norm || !g.k_norm || g.tokens <= 0) return ECF8_ERR_INVALID_ARG;
    if (g.row_stride < 3 * (int64_t)H * kD || g.row_stride % 8 || g.batch_stride % 8 ||
        (B > 1 && g.batch_stride < g.row_stride))
      return ECF8_ERR_UNSUPPORTED;
    if (!aligned(g.qkv, 16) || !aligned(g.q_norm, 16) || !aligned(g.k_norm, 16))
      return ECF8_ERR_MISALIGNED;
    if (g.tokens > (1 << 24)) return ECF8_ERR_UNSUPPORTED;
    s[i] = Stream{static_cast<const uint16_t *>(g.qkv), static_cast<const uint16_t *>(g.q_norm),
                  static_cast<const uint16_t *>(g.k_norm), g.row_stride, g.batch_stride,
                  (int)g.tokens};
    T += g.tokens;
  }
  const int64_t Tp = padded(T);
  if (T > (1 << 24) || B > (1 << 24) || B * H * (Tp / 32) > INT32_MAX) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(cos_t, 16) || !aligned(sin_t, 16) || !aligned(q, 16) || !aligned(k_packed, 16) ||
      !aligned(v_packed, 16))
    return ECF8_ERR_MISALIGNED;
  dit_qkv_kernel<<<(unsigned)(B * H * (Tp / 32)), 256, 0, as_stream(stream)>>>(
      s[0], s[1], H, (int)T, (int)Tp, eps, scale, cos_t, sin_t, static_cast<uint16_t *>(q),
      static_cast<uint16_t *>(k_packed), static_cast<uint16_t *>(v_packed));
  return launched();
}

extern "C" int ecf8_packed_attention(const void *q, const void *k_packed, const void *v_packed,
                                     int64_t B, int H, int64_t T, void *out, int64_t out_stride,
                                     void *stream) {
  if (!q || !k_packed || !v_packed || !out || B <= 0 || H <= 0 || T <= 0)
    return ECF8_ERR_INVALID_ARG;
  if (T > (1 << 24) || B > (1 << 24) || B * H * ((T + kQueries - 1) / kQueries) > INT32_MAX ||
      out_stride % 4)
    return ECF8_ERR_UNSUPPORTED;
  if (out_stride < (int64_t)H * kD) return ECF8_ERR_CAPACITY;
  if (!aligned(q, 16) || !aligned(k_packed, 16) || !aligned(v_packed, 16) || !aligned(out, 8))
    return ECF8_ERR_MISALIGNED;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return ECF8_ERR_HIP;
  // While 128-query workgroups of four waves find a CU each, spreading the
  // waves (one a SIMD) beats pairing them: MI355X, 24 heads, with the packing
  // pass, us, four waves against eight: T = 1088 (216 workgroups) 43.3
  // against 45.9, T = 2304 (432) 101.6 against 82.2, two batches of T = 1500
  // (576) 117.5 against 113.6, T = 4608 354 against 288.
  const bool spread = B * H * ((T + kQueries - 1) / kQueries) <= cus;
  const int queries = spread ? kQueries : kPairQueries;
  const int tiles = (int)((T + queries - 1) / queries);
  const Attn a{static_cast<const uint16_t *>(q), static_cast<const uint16_t *>(k_packed),
               static_cast<const uint16_t *>(v_packed), static_cast<uint16_t *>(out), out_stride,
               (int)T, (int)padded(T), H, 1, tiles, (int)(B * H), 1.f};
  if (spread)
    flash_kernel<false, false><<<(unsigned)(B * H * tiles), 256, 0, as_stream(stream)>>>(a);
  else
    pair_attention_kernel<<<(unsigned)(B * H * tiles), 512, 0, as_stream(stream)>>>(a);
  return launched();
}

extern "C" int ecf8_dit_modulate(const void *x, int64_t B, int64_t rows, int64_t C,
                                 const void *shift, int64_t shift_batch, const void *scale,
                                 int64_t scale_batch, float eps, void *out, void *stream) {
  if (!x || !shift || !scale || !out || B <= 0 || rows <= 0 || C <= 0) return ECF8_ERR_INVALID_ARG;
  if (C % 8 || C > 8192 || shift_batch % 8 || scale_batch % 8 || rows > (1 << 24) ||
      B * rows > INT32_MAX)
    return ECF8_ERR_UNSUPPORTED;
  if (!aligned(x, 16) || !aligned(shift, 16) || !aligned(scale, 16) || !aligned(out, 16))
    return ECF8_ERR_MISALIGNED;
  const auto *xp = static_cast<const uint16_t *>(x), *sh = static_cast<const uint16_t *>(shift),
             *sc = static_cast<const uint16_t *>(scale);
  auto *op = static_cast<uint16_t *>(out);
  const unsigned grid = (unsigned)(B * rows);
#define ECF8_MODULATE(V)                                                                        \
  modulate_kernel<V><<<grid, 256, 0, as_stream(stream)>>>(xp, (int)rows, (int)C, sh, shift_batch, \
                                                          sc, scale_batch, eps, op)
  if (C <= 2048)
    ECF8_MODULATE(1);
  else if (C <= 4096)
    ECF8_MODULATE(2);
  else
    ECF8_MODULATE(4);
#undef ECF8_MODULATE
  return launched();
}

extern "C" int ecf8_dit_gated_add(const void *x, const void *gate, int64_t gate_batch,
                                  const void *y, int64_t B, int64_t rows, int64_t C, void *out,
                                  void *stream) {
  if (!x || !gate || !y || !out || B <= 0 || rows <= 0 || C <= 0) return ECF8_ERR_INVALID_ARG;
  const int64_t units = B * rows * (C / 8);
  if (C % 8 || C > (1 << 24) || gate_batch % 8 || rows > (1 << 24) || B > (1 << 24) ||
      (units + 255) / 256 > INT32_MAX)
    return ECF8_ERR_UNSUPPORTED;
  if (!aligned(x, 16) || !aligned(gate, 16) || !aligned(y, 16) || !aligned(out, 16))
    return ECF8_ERR_MISALIGNED;
  gated_add_kernel<<<(unsigned)((units + 255) / 256), 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(gate), gate_batch,
      static_cast<const uint16_t *>(y), units, (int)rows, (int)C, static_cast<uint16_t *>(out));
  return launched();
}

extern "C" int ecf8_dit_gelu(const void *x, int64_t x_row, int64_t rows, int64_t C, void *out,
                             int64_t out_row, void *stream) {
  if (!x || !out || rows <= 0 || C <= 0 || x_row < C || out_row < C) return ECF8_ERR_INVALID_ARG;
  const int64_t units = rows * (C / 8);
  if (C % 8 || C > (1 << 24) || x_row % 8 || out_row % 8 || rows > INT32_MAX ||
      (units + 255) / 256 > INT32_MAX)
    return ECF8_ERR_UNSUPPORTED;
  if (!aligned(x, 16) || !aligned(out, 16)) return ECF8_ERR_MISALIGNED;
  gelu_kernel<<<(unsigned)((units + 255) / 256), 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t *>(x), x_row, units, (int)C, static_cast<uint16_t *>(out),
      out_row);
  return launched();
}
