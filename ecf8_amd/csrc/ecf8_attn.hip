// Attention of many queries per head on gfx950: the prompt's causal
// attention (grouped-query, over the KV caches) and the DiT's attention
// over text and image tokens, with the passes that prepare their operands.
// Head dimension 128, bf16 operands, fp32 scores, softmax and sums.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "ecf8.h"
#include "ecf8_attn.h"

namespace {

constexpr int kD = 128;      // head dimension
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
// that of the fp32 probabilities.  Otherwise probabilities are rounded to
// bf16, as the DiT's softmax does.
//
// Bound by the MFMA pipe and the exponentials (16 of each per 32 x 32 tile
// per wave: ~512 and ~450 cycles).MI355X, causal
// with three parts: 1 x 32 heads x 2048 queries 136 us with the packing
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
    const int key0 = b * kBlock;
    if (q0 >= a.T || (kCausal && key0 > q0 + 31)) continue;  // uniform per wave

    v16f s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[t][i] = 0.f;
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        const v8bf kf = *reinterpret_cast<const v8bf *>(&s_k[buf][t * 512 + kk * 64 + lane]);
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
    bm = fmaxf(bm, __shfl_xor(bm, 32));
    const float mn = fmaxf(m, bm);
    if (__any(mn > m)) {  // uniform: some query's maximum moved
      const float f = __builtin_amdgcn_exp2f((m - mn) * a.scale);
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
        s[t][i] = __builtin_amdgcn_exp2f((s[t][i] - m) * a.scale);
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
        const v8bf vf = *reinterpret_cast<const v8bf *>(&s_v[buf][g * 256 + d * 64 + lane]);
#pragma unroll
        for (int q = kParts - 1; q >= 0; --q)  // small parts first
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, __builtin_bit_cast(v8bf, pf[q]), o[d],
                                                         0, 0, 0);
      }
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

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }
inline bool aligned(const void *p, uintptr_t a) {
  return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0;
}
inline int launched() { return hipGetLastError() == hipSuccess ? ECF8_OK : ECF8_ERR_HIP; }
inline int64_t padded(int64_t T) { return (T + kBlock - 1) / kBlock * kBlock; }

constexpr float kLog2e = 1.4426950408889634f;

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
