// The ends of a decode step on gfx950: the bf16 linear of a few rows (the
// vocabulary head, and the DiT's modulation Linears), the greedy choice of
// the next token, and its embedding.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ecf8.h"
#include "ecf8_head.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf16_f32(uint32_t h16) { return __uint_as_float(h16 << 16); }

// out[m, n] = bf16(sum_k x[m, k] w[n, k] (+ bias[n])), M <= 16, fp32 sums.
//
// The weights are read once and nothing else matters.  A persistent
// workgroup of 16 waves takes a contiguous run of 16-row panels of w; its
// waves split K (kS steps of 32 each), so a panel is read as one contiguous
// block, and each wave keeps its slice of x in registers in MFMA lane order.
// The next panel's loads are in flight while this one's sums meet in LDS
// (two buffers, one LDS-only barrier a panel) and are added in wave order.
// (Waves streaming a whole panel each, 65,000 rows open at once, read 4.7
// TB/s at 16 rows.)  HBM-bound; MI355X,
// 16 rows, us against the library's: 151936 x 4096 221 / 263 (5.6 TB/s),
// 151936 x 2048 121 / 208; one row: 18432 x 3072 28 / 67, 3072 x 3072 8.4 /
// 14.2.
constexpr int kWaves = 16;
constexpr int kMaxK = 4096;

// Workgroup barrier that waits for LDS only (a __syncthreads would also
// wait for the prefetched global loads).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt((0x3F & 15) | (0x3 << 14) | (0x7 << 4) | (0x0 << 8));  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int kS>
__global__ __launch_bounds__(kWaves * 64) void bf16_rows_kernel(
    const uint16_t *__restrict__ x, int64_t ldx, int M, int K, const uint16_t *__restrict__ w,
    int panels, const uint16_t *__restrict__ bias, uint16_t *__restrict__ out, int64_t ldo) {
  __shared__ float s_red[2][kWaves][4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int last = K / 32 - 1;
  // this workgroup's run of panels
  const int p0 = (int)((int64_t)panels * blockIdx.x / gridDim.x);
  const int p1 = (int)((int64_t)panels * (blockIdx.x + 1) / gridDim.x);

  // steps past K's end load the last one again, unused
  u32x4 xf[kS], next[kS];
  auto load = [&](int pn, u32x4 (&v)[kS]) {
    const uint16_t *row = w + (size_t)(16 * pn + r) * K + 8 * g;
#pragma unroll
    for (int u = 0; u < kS; ++u)
      v[u] = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4 *>(row + 32 * min(wave * kS + u, last)));
  };
  load(p0, next);
#pragma unroll
  for (int u = 0; u < kS; ++u) {
    const int st = wave * kS + u;
    xf[u] = r < M && st <= last
                ? *reinterpret_cast<const u32x4 *>(x + (size_t)r * ldx + 32 * st + 8 * g)
                : u32x4{0, 0, 0, 0};
  }
  for (int panel = p0; panel < p1; ++panel) {
    u32x4 cur[kS];
#pragma unroll
    for (int u = 0; u < kS; ++u) cur[u] = next[u];
    if (panel + 1 < p1) load(panel + 1, next);
    v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kS; ++u) {
      if (wave * kS + u > last) break;  // uniform: zero times an infinite weight is not zero
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, xf[u]),
                                                    __builtin_bit_cast(v8bf, cur[u]), acc, 0, 0, 0);
    }
    const int buf = panel & 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) s_red[buf][wave][i][lane] = acc[i];
    // the other buffer is rewritten after the next barrier, by when its
    // readers have passed this one
    lds_barrier();
    if (threadIdx.x < 256) {
      const int i = threadIdx.x >> 6, m = 4 * g + i, n = 16 * panel + r;
      float sum = 0.f;
#pragma unroll
      for (int v = 0; v < kWaves; ++v) sum += s_red[buf][v][i][lane];
      if (bias) sum += bf16_f32(bias[n]);
      if (m < M) out[(size_t)m * ldo + n] = __builtin_bit_cast(uint16_t, (__bf16)sum);
    }
  }
}

// ------------------------------------------------------- greedy next token

// Sort key of a logit at index i: larger is better, NaN above everything,
// equal values (either zero) to the lower index.
__device__ __forceinline__ uint64_t logit_key(uint32_t h, uint32_t i) {
  uint32_t k;
  if ((h & 0x7fffu) > 0x7f80u)
    k = 0x1ffffu;
  else if ((h & 0x7fffu) == 0)
    k = 0x8000u;
  else
    k = h & 0x8000u ? 0x8000u - (h & 0x7fffu) : 0x8000u + h;
  return ((uint64_t)k << 32) | (uint32_t)~i;
}

__device__ __forceinline__ uint64_t wave_max64(uint64_t v) {
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t u = __shfl_xor(v, o);
    v = u > v ? u : v;
  }
  return v;
}

// Best key of each of `chunks` runs of a row's logits (bf16; `vec`: rows are
// 16-byte aligned, 8 per load): 64
// workgroups a row and a small second kernel where the library's reduction
// took 57 us for 16 rows of 151936 (9 us both).
__global__ __launch_bounds__(256) void argmax_chunk_kernel(const uint16_t *__restrict__ logits,
                                                           int64_t ld, int V, int chunks,
                                                           int vec, uint64_t *__restrict__ keys) {
  __shared__ uint64_t s_k[4];
  const int chunk = blockIdx.x, b = blockIdx.y;
  const int units = (V + 7) / 8, per = (units + chunks - 1) / chunks;
  const uint16_t *row = logits + (size_t)b * ld;
  uint64_t best = 0;
  for (int u = chunk * per + threadIdx.x; u < min((chunk + 1) * per, units); u += 256) {
    if (vec && 8 * u + 8 <= V) {
      const u32x4 v = *reinterpret_cast<const u32x4 *>(row + 8 * u);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint64_t k = logit_key((v[j >> 1] >> (16 * (j & 1))) & 0xffffu, 8 * u + j);
        best = k > best ? k : best;
      }
    } else {
      for (int i = 8 * u; i < min(8 * u + 8, V); ++i) {
        const uint64_t k = logit_key(row[i], i);
        best = k > best ? k : best;
      }
    }
  }
  best = wave_max64(best);
  if ((threadIdx.x & 63) == 0) s_k[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 4; ++i) best = s_k[i] > best ? s_k[i] : best;
    keys[(size_t)b * chunks + chunk] = best;
  }
}

// Each row's token -> next[b] and tokens[b, step[0]]; then step += 1 and
// pos += advance.  One workgroup, a wave per row in turn.  A step outside
// the rows writes no token and sets *refused (where there is one).
__global__ __launch_bounds__(1024) void emit_kernel(const uint64_t *__restrict__ keys, int chunks,
                                                    int B, int64_t *__restrict__ tokens,
                                                    int64_t ldt, int64_t *__restrict__ next,
                                                    int64_t *__restrict__ step,
                                                    int *__restrict__ pos, int advance,
                                                    int *__restrict__ refused) {
  const int lane = threadIdx.x & 63;
  const int64_t at = step[0];
  for (int b = threadIdx.x >> 6; b < B; b += 16) {
    uint64_t best = 0;
    for (int c = lane; c < chunks; c += 64) {
      const uint64_t k = keys[(size_t)b * chunks + c];
      best = k > best ? k : best;
    }
    best = wave_max64(best);
    if (lane == 0) {
      const int64_t tok = (int64_t)(uint32_t)~(uint32_t)best;
      next[b] = tok;
      if (at >= 0 && at < ldt) tokens[(size_t)b * ldt + at] = tok;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    step[0] = at + 1;
    if (advance) pos[0] += advance;
    if (refused && (at < 0 || at >= ldt)) *refused = 1;
  }
}

// out[b, :] = float(table[token[b], :]); a token outside the table writes
// zeros and sets *refused (where there is one)
__global__ __launch_bounds__(256) void embed_kernel(const int64_t *__restrict__ token,
                                                    const uint16_t *__restrict__ table, int64_t V,
                                                    int H, float *__restrict__ out,
                                                    int *__restrict__ refused) {
  const int b = blockIdx.y, c = 8 * (blockIdx.x * 256 + threadIdx.x);
  if (c >= H) return;
  const int64_t t = token[b];
  u32x4 v = {0, 0, 0, 0};
  if (t >= 0 && t < V)
    v = *reinterpret_cast<const u32x4 *>(table + (size_t)t * H + c);
  else if (refused)
    *refused = 1;
  float4 *o = reinterpret_cast<float4 *>(out + (size_t)b * H + c);
  o[0] = make_float4(bf16_f32(v[0] & 0xffffu), bf16_f32(v[0] >> 16), bf16_f32(v[1] & 0xffffu),
                     bf16_f32(v[1] >> 16));
  o[1] = make_float4(bf16_f32(v[2] & 0xffffu), bf16_f32(v[2] >> 16), bf16_f32(v[3] & 0xffffu),
                     bf16_f32(v[3] >> 16));
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }
inline bool aligned(const void *p, uintptr_t a) {
  return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0;
}
inline int launched() { return hipGetLastError() == hipSuccess ? ECF8_OK : ECF8_ERR_HIP; }

}  // namespace

extern "C" int ecf8_bf16_linear16(const void *x, int64_t ldx, int64_t M, int64_t K, const void *w,
                                  int64_t N, const void *bias, void *out, int64_t ldo,
                                  void *stream) {
  if (!x || !w || !out || M <= 0 || K <= 0 || N <= 0) return ECF8_ERR_INVALID_ARG;
  if (M > 16 || K % 32 || K > kMaxK || N % 16 || N > (1 << 27) || ldx % 8 || (M > 1 && ldx < K))
    return ECF8_ERR_UNSUPPORTED;
  if (ldo < N && M > 1) return ECF8_ERR_CAPACITY;
  if (!aligned(x, 16) || !aligned(w, 16) || !aligned(out, 2) || (bias && !aligned(bias, 2)))
    return ECF8_ERR_MISALIGNED;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return ECF8_ERR_HIP;
  const int64_t panels = N / 16;
  const unsigned grid = (unsigned)(panels < cus ? panels : cus);
  const auto *xp = static_cast<const uint16_t *>(x), *wp = static_cast<const uint16_t *>(w),
             *bp = static_cast<const uint16_t *>(bias);
  auto *op = static_cast<uint16_t *>(out);
#define ECF8_BF16_ROWS(S)                                                                      \
  bf16_rows_kernel<S><<<grid, kWaves * 64, 0, as_stream(stream)>>>(xp, ldx, (int)M, (int)K, wp, \
                                                                   (int)panels, bp, op, ldo)
  const int64_t per_wave = (K / 32 + kWaves - 1) / kWaves;
  if (per_wave <= 2)
    ECF8_BF16_ROWS(2);
  else if (per_wave <= 4)
    ECF8_BF16_ROWS(4);
  else if (per_wave <= 6)
    ECF8_BF16_ROWS(6);
  else
    ECF8_BF16_ROWS(8);
#undef ECF8_BF16_ROWS
  return launched();
}

extern "C" int64_t ecf8_greedy_work_bytes(int64_t B) {
  return B <= 0 ? -1 : B * ECF8_GREEDY_CHUNKS * 8;
}

extern "C" int ecf8_greedy_emit_checked(const void *logits, int64_t ld, int64_t B, int64_t V,
                                        void *work, int64_t work_bytes, int64_t *tokens,
                                        int64_t ld_tokens, int64_t *next_token, int64_t *step,
                                        int *pos, int advance, int *refused, void *stream) {
  if (!logits || !work || !tokens || !next_token || !step || (advance && !pos) || B <= 0 ||
      V <= 0 || ld < V || ld_tokens <= 0)
    return ECF8_ERR_INVALID_ARG;
  if (B > 65535 || V > (1 << 30)) return ECF8_ERR_UNSUPPORTED;
  if (work_bytes < ecf8_greedy_work_bytes(B)) return ECF8_ERR_CAPACITY;
  if (!aligned(logits, 2) || !aligned(work, 8) || !aligned(tokens, 8) ||
      !aligned(next_token, 8) || !aligned(step, 8) || !aligned(refused, 4))
    return ECF8_ERR_MISALIGNED;
  auto *keys = static_cast<uint64_t *>(work);
  argmax_chunk_kernel<<<dim3(ECF8_GREEDY_CHUNKS, (unsigned)B), 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t *>(logits), ld, (int)V, ECF8_GREEDY_CHUNKS,
      ld % 8 == 0 && aligned(logits, 16), keys);
  emit_kernel<<<1, 1024, 0, as_stream(stream)>>>(keys, ECF8_GREEDY_CHUNKS, (int)B, tokens,
                                                 ld_tokens, next_token, step, pos, advance,
                                                 refused);
  return launched();
}

extern "C" int ecf8_greedy_emit(const void *logits, int64_t ld, int64_t B, int64_t V, void *work,
                                int64_t work_bytes, int64_t *tokens, int64_t ld_tokens,
                                int64_t *next_token, int64_t *step, int *pos, int advance,
                                void *stream) {
  return ecf8_greedy_emit_checked(logits, ld, B, V, work, work_bytes, tokens, ld_tokens,
                                  next_token, step, pos, advance, nullptr, stream);
}

extern "C" int ecf8_embed_rows_checked(const int64_t *token, int64_t B, const void *table,
                                       int64_t V, int64_t H, float *out, int *refused,
                                       void *stream) {
  if (!token || !table || !out || B <= 0 || V <= 0 || H <= 0) return ECF8_ERR_INVALID_ARG;
  if (H % 8 || H > (1 << 24) || B > 65535) return ECF8_ERR_UNSUPPORTED;
  if (!aligned(token, 8) || !aligned(table, 16) || !aligned(out, 16) || !aligned(refused, 4))
    return ECF8_ERR_MISALIGNED;
  embed_kernel<<<dim3((unsigned)((H + 2047) / 2048), (unsigned)B), 256, 0, as_stream(stream)>>>(
      token, static_cast<const uint16_t *>(table), V, (int)H, out, refused);
  return launched();
}

extern "C" int ecf8_embed_rows(const int64_t *token, int64_t B, const void *table, int64_t V,
                               int64_t H, float *out, void *stream) {
  return ecf8_embed_rows_checked(token, B, table, V, H, out, nullptr, stream);
}
