// Host-side part of libecf8: the bitstream encoder (the producer of the
// decoder's input, run offline on the CPU as in the reference), encoder
// output sizing, and the compressed-block format validator.  Declared in
// include/ecf8.h.

#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <memory>
#include <new>
#include <thread>
#include <vector>

#include "ecf8.h"

namespace {

constexpr int kMaxThreads = 64;

// Encoder core shared by sizing and encoding.  The per-symbol bookkeeping
// follows the reference's rule exactly (dfloat/utils.py:387-463): a chunk gap
// is recorded whenever the running bit count enters a chunk with no gap yet
// (total_bits / chunk_bits + 1 > gaps recorded), a format-block position
// whenever it enters a format-block with none yet, and after the last symbol
// the same two checks run once more at the EOF pad position when a partial
// byte remains.  Bits are accumulated 32 at a time and written big-endian.
struct Sink {
  uint8_t *encoded;
  int64_t enc_cap;
  uint8_t *gaps;  // packed nibbles, even chunk high
  int64_t gaps_cap;
  uint64_t *op;
  int64_t op_cap;
  bool write;
  bool overflow = false;
  int64_t n_enc = 0, n_gaps = 0, n_op = 0;

  void put_byte(uint8_t b) {
    if (write) {
      if (n_enc < enc_cap) encoded[n_enc] = b;
      else overflow = true;
    }
    ++n_enc;
  }
  void put_gap(uint32_t gap) {
    if (write) {
      const int64_t byte = n_gaps >> 1;
      if (byte < gaps_cap) {
        if (n_gaps & 1) gaps[byte] = (uint8_t)(gaps[byte] | (gap & 0xF));
        else gaps[byte] = (uint8_t)((gap & 0xF) << 4);
      } else {
        overflow = true;
      }
    }
    ++n_gaps;
  }
  void put_op(uint64_t v) {
    if (write) {
      if (n_op < op_cap) op[n_op] = v;
      else overflow = true;
    }
    ++n_op;
  }
};

int encode_core(const uint8_t *exps, int64_t n, const uint8_t *code_bits, const uint32_t *code_vals,
                int eof_bits, uint32_t eof_value, int bpt, int tpb, Sink &sink) {
  const int64_t chunk_bits = 8LL * bpt;
  const int64_t block_bits = chunk_bits * tpb;
  uint64_t acc = 0;  // pending bits, right-aligned
  int nacc = 0;      // < 32 between symbols
  int64_t total = 0;
  for (int64_t i = 0; i < n; ++i) {
    const uint32_t s = exps[i];
    if (s > 15 || code_bits[s] == 0 || code_bits[s] > 16) return ECF8_ERR_FORMAT;
    if (total / chunk_bits + 1 > sink.n_gaps) sink.put_gap((uint32_t)(total % chunk_bits));
    if (total / block_bits + 1 > sink.n_op) sink.put_op((uint64_t)i);
    const int len = code_bits[s];
    acc = (acc << len) | (code_vals ? (code_vals[s] & ((1u << len) - 1)) : 0u);
    nacc += len;
    total += len;
    if (nacc >= 32) {
      const uint32_t word = (uint32_t)(acc >> (nacc - 32));
      sink.put_byte((uint8_t)(word >> 24));
      sink.put_byte((uint8_t)(word >> 16));
      sink.put_byte((uint8_t)(word >> 8));
      sink.put_byte((uint8_t)word);
      nacc -= 32;
      acc &= (nacc ? ((1ull << nacc) - 1) : 0ull);
    }
  }
  while (nacc >= 8) {
    sink.put_byte((uint8_t)(acc >> (nacc - 8)));
    nacc -= 8;
    acc &= (1ull << nacc) - 1;
  }
  if (nacc > 0) {  // final partial byte, padded with the EOF code's leading bits
    if (total / chunk_bits + 1 > sink.n_gaps) sink.put_gap((uint32_t)(total % chunk_bits));
    if (total / block_bits + 1 > sink.n_op) sink.put_op((uint64_t)n);
    if (eof_bits < 1 || eof_bits > 24) return ECF8_ERR_FORMAT;
    const uint64_t v = (acc << eof_bits) | (eof_value & ((1u << eof_bits) - 1));
    const int size = nacc + eof_bits;
    sink.put_byte((uint8_t)(size >= 8 ? v >> (size - 8) : v << (8 - size)));
  }
  sink.put_op((uint64_t)n);
  const int64_t fb_bytes = (int64_t)bpt * tpb;
  const int64_t n_fb = (sink.n_enc + fb_bytes - 1) / fb_bytes;
  while (sink.n_gaps < n_fb * tpb) sink.put_gap(0);
  return sink.overflow ? ECF8_ERR_CAPACITY : ECF8_OK;
}

// f(0) .. f(n - 1) on a thread each; where a thread cannot be had, here.
template <typename F>
void run_parallel(int n, F f) {
  std::thread th[kMaxThreads];
  int started = 0;
  try {
    for (; started < n - 1; ++started) th[started] = std::thread(f, started);
  } catch (...) {  // no thread, or no memory for its state
  }
  for (int i = started; i < n; ++i) f(i);
  for (int i = 0; i < started; ++i) th[i].join();
}

// Parts of n items for at most n_threads threads, `least` items or more each.
int parts_of(int64_t n, int n_threads, int64_t least) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(std::min(n_threads, kMaxThreads), n / least));
}

// Code bits of exps[a..b), or -1 if one has no code.
int64_t code_bits_of(const uint8_t *exps, int64_t a, int64_t b, const uint8_t *code_bits) {
  uint32_t len[256];
  for (int v = 0; v < 256; ++v)
    len[v] = v < 16 && code_bits[v] >= 1 && code_bits[v] <= 16 ? code_bits[v] : 1u << 24;
  int64_t sum = 0;
  while (a < b) {  // a run's bits stay below the flag
    const int64_t e = std::min<int64_t>(b, a + (1 << 16));
    uint64_t run = 0;
    for (; a < e; ++a) run += len[exps[a]];
    if (run >> 24) return -1;
    sum += (int64_t)run;
  }
  return sum;
}

// What encode_core writes, from the number of code bits and the bits at
// which the last symbol starts (a code is at most 16 bits and a chunk at
// least 16, so every chunk and format-block up to the last holds a start).
struct Sizes {
  int64_t enc, gaps, op, chunks, blocks;  // chunks, blocks: with a start or the pad
};
Sizes sizes_of(int64_t n, int64_t bits, int last_len, int bpt, int tpb) {
  const int64_t chunk_bits = 8LL * bpt, block_bits = chunk_bits * tpb;
  Sizes z{(bits + 7) / 8, 0, 1, 0, 0};
  if (n == 0) return z;
  const int64_t end = bits % 8 ? bits : bits - last_len;
  z.chunks = end / chunk_bits + 1;
  z.blocks = end / block_bits + 1;
  z.op = z.blocks + 1;
  const int64_t fb = (int64_t)bpt * tpb;
  z.gaps = std::max(z.chunks, (z.enc + fb - 1) / fb * tpb);
  return z;
}

// encode_core over `parts` runs of symbols at once, the same bytes.  Each run
// starts at the bit where the codes before it end (a first pass adds up the
// code lengths); a byte that two runs share is put together at the end.
// Bound by the symbol loop; a 4096 x 4096 Linear compresses in 14 ms on 16
// threads, where two passes of encode_core (sizes, bytes) and torch's split
// and count took 94.
int encode_parallel(const uint8_t *exps, int64_t n, const uint8_t *code_bits,
                    const uint32_t *code_vals, int eof_bits, uint32_t eof_value, int bpt, int tpb,
                    uint8_t *encoded, int64_t enc_cap, uint8_t *gaps, int64_t gaps_cap,
                    uint64_t *op, int64_t op_cap, int parts) {
  const int64_t chunk_bits = 8LL * bpt, block_bits = chunk_bits * tpb;
  int64_t bits[kMaxThreads], start[kMaxThreads + 1];
  auto first = [&](int i) { return n * i / parts; };
  run_parallel(parts, [&](int i) { bits[i] = code_bits_of(exps, first(i), first(i + 1), code_bits); });
  start[0] = 0;
  for (int i = 0; i < parts; ++i) {
    if (bits[i] < 0) return ECF8_ERR_FORMAT;
    start[i + 1] = start[i] + bits[i];
  }
  const int64_t total = start[parts];
  if (total % 8 && (eof_bits < 1 || eof_bits > 24)) return ECF8_ERR_FORMAT;
  const Sizes z = sizes_of(n, total, code_bits[exps[n - 1]], bpt, tpb);
  if (z.enc > enc_cap || (z.gaps + 1) / 2 > gaps_cap || z.op > op_cap) return ECF8_ERR_CAPACITY;
  std::unique_ptr<uint8_t[]> gap(new (std::nothrow) uint8_t[z.gaps + 1]);
  if (!gap) return -1;
  memset(gap.get() + z.chunks, 0, z.gaps + 1 - z.chunks);
  uint8_t head[kMaxThreads] = {};  // a run's bits of the byte it starts inside
  uint64_t tail[kMaxThreads];      // its bits past the last whole byte
  run_parallel(parts, [&](int i) {
    const int64_t a = first(i), b = first(i + 1);
    int64_t at = start[i];  // bit of the next symbol
    const int64_t before = a ? at - code_bits[exps[a - 1]] : -1;  // where the last one started
    int64_t chunk = a ? before / chunk_bits + 1 : 0, block = a ? before / block_bits + 1 : 0;
    int64_t next_chunk = chunk * chunk_bits, next_block = block * block_bits;
    uint32_t len[16], val[16];
    for (int v = 0; v < 16; ++v) {
      len[v] = code_bits[v];
      val[v] = len[v] && len[v] <= 16 ? code_vals[v] & ((1u << len[v]) - 1) : 0;
    }
    uint64_t acc = 0;
    int nacc = (int)(at % 8);
    uint8_t *out = encoded + at / 8;
    bool shared = nacc > 0;  // the first byte waits for the run before
    for (int64_t k = a; k < b; ++k) {
      const uint32_t s = exps[k];
      if (at >= next_chunk) {
        gap[chunk++] = (uint8_t)((at - next_chunk) & 0xF);
        next_chunk += chunk_bits;
        if (at >= next_block) {
          op[block++] = (uint64_t)k;
          next_block += block_bits;
        }
      }
      acc = (acc << len[s]) | val[s];
      nacc += (int)len[s];
      at += len[s];
      if (nacc >= 32) {
        nacc -= 32;
        const uint32_t word = (uint32_t)(acc >> nacc);
        if (shared) {
          head[i] = (uint8_t)(word >> 24);
          shared = false;
        } else {
          out[0] = (uint8_t)(word >> 24);
        }
        out[1] = (uint8_t)(word >> 16);
        out[2] = (uint8_t)(word >> 8);
        out[3] = (uint8_t)word;
        out += 4;
        acc &= (1ull << nacc) - 1;
      }
    }
    while (nacc >= 8) {
      nacc -= 8;
      *out++ = (uint8_t)(acc >> nacc);
      acc &= (1ull << nacc) - 1;
    }
    tail[i] = acc;
  });
  for (int i = 1; i < parts; ++i)
    if (const int r = (int)(start[i] % 8))
      encoded[start[i] / 8] = (uint8_t)(head[i] | (tail[i - 1] << (8 - r)));
  if (const int r = (int)(total % 8)) {  // padded with the EOF code's leading bits
    const uint64_t v = (tail[parts - 1] << eof_bits) | (eof_value & ((1u << eof_bits) - 1));
    const int size = r + eof_bits;
    encoded[total / 8] = (uint8_t)(size >= 8 ? v >> (size - 8) : v << (8 - size));
    // the pad counts as a start where no symbol starts in its chunk, block
    const int64_t last = total - code_bits[exps[n - 1]];
    if (total / chunk_bits > last / chunk_bits)
      gap[total / chunk_bits] = (uint8_t)(total % chunk_bits & 0xF);
    if (total / block_bits > last / block_bits) op[total / block_bits] = (uint64_t)n;
  }
  op[z.op - 1] = (uint64_t)n;
  for (int64_t k = 0; k < (z.gaps + 1) / 2; ++k)
    gaps[k] = (uint8_t)(gap[2 * k] << 4 | gap[2 * k + 1]);
  return ECF8_OK;
}

bool geometry_ok(int bpt, int tpb) {
  return bpt >= 2 && bpt <= 64 && tpb >= 2 && tpb <= 4096 && (tpb % 2) == 0;
}

}  // namespace

extern "C" const char *ecf8_version(void) { return "ecf8_amd 0.1.0 (gfx950)"; }

extern "C" const char *ecf8_status_string(int status) {
  switch (status) {
    case ECF8_OK: return "ok";
    case ECF8_ERR_INVALID_ARG: return "invalid argument";
    case ECF8_ERR_UNSUPPORTED: return "unsupported format geometry";
    case ECF8_ERR_MISALIGNED: return "misaligned device buffer";
    case ECF8_ERR_FORMAT: return "malformed compressed block";
    case ECF8_ERR_HIP: return "HIP runtime error";
    case ECF8_ERR_CAPACITY: return "output buffer too small";
    default: return "unknown status";
  }
}

extern "C" int ecf8_encoded_sizes(const uint8_t *exponents, int64_t n, const uint8_t *code_bits,
                                  int bytes_per_thread, int threads_per_block, int64_t *n_bytes,
                                  int64_t *gaps_bytes, int64_t *n_output_positions) {
  if ((n > 0 && !exponents) || !code_bits || n < 0 || !n_bytes || !gaps_bytes ||
      !n_output_positions)
    return ECF8_ERR_INVALID_ARG;
  if (!geometry_ok(bytes_per_thread, threads_per_block)) return ECF8_ERR_UNSUPPORTED;
  Sink sink{nullptr, 0, nullptr, 0, nullptr, 0, false};
  // the EOF code only affects the pad byte's value, not the sizes
  const int rc = encode_core(exponents, n, code_bits, nullptr, 1, 0, bytes_per_thread,
                             threads_per_block, sink);
  if (rc != ECF8_OK) return rc;
  *n_bytes = sink.n_enc;
  *gaps_bytes = (sink.n_gaps + 1) / 2;
  *n_output_positions = sink.n_op;
  return ECF8_OK;
}

extern "C" int ecf8_encode_exponents(const uint8_t *exponents, int64_t n, const uint8_t *code_bits,
                                     const uint32_t *code_vals, int eof_bits, uint32_t eof_value,
                                     int bytes_per_thread, int threads_per_block, uint8_t *encoded,
                                     int64_t encoded_capacity, uint8_t *gaps, int64_t gaps_capacity,
                                     uint64_t *output_positions,
                                     int64_t output_positions_capacity) {
  if ((n > 0 && !exponents) || !code_bits || !code_vals || n < 0 || !output_positions ||
      (encoded_capacity > 0 && !encoded) || (gaps_capacity > 0 && !gaps))
    return ECF8_ERR_INVALID_ARG;
  if (!geometry_ok(bytes_per_thread, threads_per_block)) return ECF8_ERR_UNSUPPORTED;
  Sink sink{encoded, encoded_capacity, gaps, gaps_capacity, output_positions,
            output_positions_capacity, true};
  return encode_core(exponents, n, code_bits, code_vals, eof_bits, eof_value, bytes_per_thread,
                     threads_per_block, sink);
}

extern "C" int ecf8_encoded_sizes_threads(const uint8_t *exponents, int64_t n,
                                          const uint8_t *code_bits, int bytes_per_thread,
                                          int threads_per_block, int n_threads, int64_t *n_bytes,
                                          int64_t *gaps_bytes, int64_t *n_output_positions) {
  if ((n > 0 && !exponents) || !code_bits || n < 0 || !n_bytes || !gaps_bytes ||
      !n_output_positions)
    return ECF8_ERR_INVALID_ARG;
  if (!geometry_ok(bytes_per_thread, threads_per_block)) return ECF8_ERR_UNSUPPORTED;
  int64_t bits[kMaxThreads], total = 0;
  const int parts = parts_of(n, n_threads, 1 << 16);
  run_parallel(parts, [&](int i) {
    bits[i] = code_bits_of(exponents, n * i / parts, n * (i + 1) / parts, code_bits);
  });
  for (int i = 0; i < parts; ++i) {
    if (bits[i] < 0) return ECF8_ERR_FORMAT;
    total += bits[i];
  }
  const Sizes z = sizes_of(n, total, n ? code_bits[exponents[n - 1]] : 0, bytes_per_thread,
                           threads_per_block);
  *n_bytes = z.enc;
  *gaps_bytes = (z.gaps + 1) / 2;
  *n_output_positions = z.op;
  return ECF8_OK;
}

extern "C" int ecf8_encode_exponents_threads(
    const uint8_t *exponents, int64_t n, const uint8_t *code_bits, const uint32_t *code_vals,
    int eof_bits, uint32_t eof_value, int bytes_per_thread, int threads_per_block, int n_threads,
    uint8_t *encoded, int64_t encoded_capacity, uint8_t *gaps, int64_t gaps_capacity,
    uint64_t *output_positions, int64_t output_positions_capacity) {
  if ((n > 0 && !exponents) || !code_bits || !code_vals || n < 0 || !output_positions ||
      (encoded_capacity > 0 && !encoded) || (gaps_capacity > 0 && !gaps))
    return ECF8_ERR_INVALID_ARG;
  if (!geometry_ok(bytes_per_thread, threads_per_block)) return ECF8_ERR_UNSUPPORTED;
  const int parts = parts_of(n, n_threads, 1 << 16);
  if (parts > 1) {
    const int rc = encode_parallel(exponents, n, code_bits, code_vals, eof_bits, eof_value,
                                   bytes_per_thread, threads_per_block, encoded, encoded_capacity,
                                   gaps, gaps_capacity, output_positions,
                                   output_positions_capacity, parts);
    if (rc >= 0) return rc;  // else: no memory for the gaps, encode here
  }
  return ecf8_encode_exponents(exponents, n, code_bits, code_vals, eof_bits, eof_value,
                               bytes_per_thread, threads_per_block, encoded, encoded_capacity,
                               gaps, gaps_capacity, output_positions, output_positions_capacity);
}

extern "C" int ecf8_split_fp8(const uint8_t *weights, int64_t n, uint8_t *exponents,
                              uint8_t *packed, int64_t *counts, int n_threads) {
  if ((n > 0 && (!weights || !exponents || !packed)) || !counts || n < 0)
    return ECF8_ERR_INVALID_ARG;
  if (n % 2) return ECF8_ERR_UNSUPPORTED;
  int64_t count[kMaxThreads][16] = {};
  const int parts = parts_of(n / 2, n_threads, 1 << 16);
  run_parallel(parts, [&](int i) {
    const int64_t a = n / 2 * i / parts, b = n / 2 * (i + 1) / parts;
    for (int64_t k = 2 * a; k < 2 * b; ++k) exponents[k] = (weights[k] >> 3) & 0xF;
    for (int64_t k = a; k < b; ++k) {
      const uint8_t e = weights[2 * k], o = weights[2 * k + 1];
      packed[k] = (uint8_t)((e & 0x80) | (e & 7) << 4 | (o >> 4 & 8) | (o & 7));
    }
    int64_t c[4][256] = {};  // neighbours in tables of their own
    for (int64_t k = a; k < b; ++k) {
      ++c[k & 1][weights[2 * k]];
      ++c[2 + (k & 1)][weights[2 * k + 1]];
    }
    for (int v = 0; v < 256; ++v) count[i][v >> 3 & 0xF] += c[0][v] + c[1][v] + c[2][v] + c[3][v];
  });
  for (int v = 0; v < 16; ++v) {
    counts[v] = 0;
    for (int i = 0; i < parts; ++i) counts[v] += count[i][v];
  }
  return ECF8_OK;
}

extern "C" int ecf8_validate_format(const uint8_t *luts, int n_luts, int64_t n_bytes,
                                    int64_t packed_bytes, const uint64_t *output_positions,
                                    int64_t n_output_positions, int64_t gaps_bytes,
                                    int64_t n_elements, int threads_per_block,
                                    int bytes_per_thread, char *msg, size_t msg_len) {
  auto fail = [&](int rc, const char *fmt, long long a, long long b) {
    if (msg && msg_len) snprintf(msg, msg_len, fmt, a, b);
    return rc;
  };
  if (!luts || !output_positions)
    return fail(ECF8_ERR_INVALID_ARG, "null luts (%lld) or output_positions (%lld)", !luts,
                !output_positions);
  if (!geometry_ok(bytes_per_thread, threads_per_block))
    return fail(ECF8_ERR_UNSUPPORTED, "geometry %lld x %lld unsupported", bytes_per_thread,
                threads_per_block);
  if (n_luts < 2 || n_luts > ECF8_MAX_LUTS)
    return fail(ECF8_ERR_FORMAT, "n_luts=%lld outside [2, %lld]", n_luts, ECF8_MAX_LUTS);
  if (n_elements != 2 * packed_bytes)
    return fail(ECF8_ERR_FORMAT, "n_elements=%lld != 2 * packed bytes %lld", n_elements,
                packed_bytes);
  const uint8_t *lens = luts + 256 * (n_luts - 1);
  // first-level and second-level entries: a symbol with a code length, or
  // (first level only) a pointer to an existing second-level row
  for (int r = 0; r < n_luts - 1; ++r) {
    for (int k = 0; k < 256; ++k) {
      const int v = luts[256 * r + k];
      if (v >= 240) {
        if (r != 0) return fail(ECF8_ERR_FORMAT, "pointer in second-level row %lld at %lld", r, k);
        const int row = 256 - v;
        if (row > n_luts - 2)
          return fail(ECF8_ERR_FORMAT, "pointer to row %lld of %lld rows", row, n_luts - 2);
      } else if (v > 15) {
        return fail(ECF8_ERR_FORMAT, "entry %lld is not an exponent (row %lld)", v, r);
      }
    }
  }
  // Entries of symbols without a code (length 0) are legal: the builder's
  // forward fill starts from 0 (utils.py:352), so keys before the first code
  // in a row read as symbol 0, reachable only through the EOF code's bits.
  for (int v = 0; v < 16; ++v)
    if (lens[v] > 16) return fail(ECF8_ERR_FORMAT, "symbol %lld has code length %lld", v, lens[v]);
  const int64_t fb_bytes = (int64_t)bytes_per_thread * threads_per_block;
  const int64_t n_fb = (n_bytes + fb_bytes - 1) / fb_bytes;
  if (n_output_positions != n_fb + 1)
    return fail(ECF8_ERR_FORMAT, "%lld output positions for %lld format-blocks", n_output_positions,
                n_fb);
  if (gaps_bytes != n_fb * threads_per_block / 2)
    return fail(ECF8_ERR_FORMAT, "%lld gap bytes for %lld format-blocks", gaps_bytes, n_fb);
  if (output_positions[0] != 0 && n_fb > 0)
    return fail(ECF8_ERR_FORMAT, "output_positions[0]=%lld, expected %lld",
                (long long)output_positions[0], 0);
  for (int64_t b = 0; b < n_fb; ++b)
    if (output_positions[b + 1] < output_positions[b])
      return fail(ECF8_ERR_FORMAT, "output_positions decrease at %lld (%lld)", b,
                  (long long)output_positions[b + 1]);
  if ((int64_t)output_positions[n_fb] != n_elements)
    return fail(ECF8_ERR_FORMAT, "last output position %lld != n_elements %lld",
                (long long)output_positions[n_fb], n_elements);
  const int64_t max_syms = (int64_t)threads_per_block * 8 * bytes_per_thread;
  for (int64_t b = 0; b < n_fb; ++b)
    if ((int64_t)(output_positions[b + 1] - output_positions[b]) > max_syms)
      return fail(ECF8_ERR_FORMAT, "format-block %lld holds more than %lld symbols", b, max_syms);
  return ECF8_OK;
}
