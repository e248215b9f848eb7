// GGUF block decoding shared by the dequantizer (gguf.hip) and the fused
// dequantize + requantize converter (gguf_requant.hip).
//
// Reference: the per-type block decoders of src/gguf/dequant.rs (:228-719).
// decode_run<TAG, N>(block, j, v) is elements j .. j + N - 1 of a block (N =
// 4, 8, 16 or 32, j a multiple of N), with exactly the IEEE f32 operations,
// operand order and roundings the reference uses for each.  Every file that
// includes this header is compiled with -ffp-contract=off so no mul+add/sub
// is fused.
//
// A run shares what its elements have in common: the f16 block scales (one
// v_cvt_f32_f16 each, exact for every encoding), the sub-block scale, the
// nibble half; codes are masked four at a time in their words and converted
// with one instruction each.  Blocks are read from LDS at 2-byte alignment.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "iq_tables.h"

namespace mlxq {
namespace {  // internal linkage: each including file has its own copy

__device__ __forceinline__ float f16_to_f32(uint32_t h) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(h)));
}
// 2-byte aligned reads (every block size and field offset used here is even)
__device__ __forceinline__ uint32_t rd_u16(const uint8_t* b) { return *reinterpret_cast<const uint16_t*>(b); }
__device__ __forceinline__ float rd_f16(const uint8_t* b, int i) { return f16_to_f32(rd_u16(b + i)); }
__device__ __forceinline__ uint32_t rd_u32(const uint8_t* b) { return rd_u16(b) | (rd_u16(b + 2) << 16); }
// N bytes at alignment A as words
template <int N, int A>
__device__ __forceinline__ void rd_words(const uint8_t* b, uint32_t (&w)[N / 4]) {
  __builtin_memcpy(w, __builtin_assume_aligned(b, A), N);
}

// float of unsigned byte k of a word (v_cvt_f32_ubyte)
__device__ __forceinline__ float ubyte(uint32_t w, int k) { return static_cast<float>((w >> (8 * k)) & 0xFFu); }
// float of signed byte k
__device__ __forceinline__ float sbyte(uint32_t w, int k) {
  return static_cast<float>(static_cast<int8_t>((w >> (8 * k)) & 0xFFu));
}

// f(i, w) for the N/4 words w of a run whose four codes sit in the nibbles of
// four bytes: 16 bytes at p hold elements 0-15 in the low nibbles and 16-31
// in the high ones (Q4_0 and its kin)
template <int N, int A, typename F>
__device__ __forceinline__ void nibbles16(const uint8_t* p, int j, F&& f) {
  if constexpr (N == 32) {
    uint32_t w[4];
    rd_words<16, A>(p, w);
#pragma unroll
    for (int i = 0; i < 8; i++) f(i, (i < 4 ? w[i & 3] : w[i & 3] >> 4) & 0x0F0F0F0Fu);
  } else {
    uint32_t w[N / 4];
    rd_words<N, (A < N ? A : N)>(p + (j & 15), w);
    const int sh = (j >> 2) & 4;
#pragma unroll
    for (int i = 0; i < N / 4; i++) f(i, (w[i] >> sh) & 0x0F0F0F0Fu);
  }
}

// bits 0-3 of x as the low bits of four bytes
__device__ __forceinline__ uint32_t spread4(uint32_t x) { return __umul24(x & 0xFu, 0x204081u) & 0x01010101u; }

// IQ4_NL codebook, four lookups at once: v_perm picks byte q & 7 of each
// 8-byte half of the table, and a byte mask of the codes' bit 3 (selectors
// 8-11 of v_perm replicate a sign bit) selects between the halves.
constexpr int8_t kIq4nl[16] = {-127, -104, -83, -65, -49, -35, -22, -10,
                               1,    13,   25,  38,  53,  69,  89,  113};
constexpr uint32_t iq4nl_word(int w) {
  return static_cast<uint32_t>(static_cast<uint8_t>(kIq4nl[4 * w])) |
         (static_cast<uint32_t>(static_cast<uint8_t>(kIq4nl[4 * w + 1])) << 8) |
         (static_cast<uint32_t>(static_cast<uint8_t>(kIq4nl[4 * w + 2])) << 16) |
         (static_cast<uint32_t>(static_cast<uint8_t>(kIq4nl[4 * w + 3])) << 24);
}
__device__ __forceinline__ uint32_t iq4nl_values(uint32_t q) {  // four codes in bytes -> four signed bytes
  const uint32_t sel = q & 0x07070707u, y = q << 4;
  const uint32_t lo = __builtin_amdgcn_perm(iq4nl_word(1), iq4nl_word(0), sel);
  const uint32_t hi = __builtin_amdgcn_perm(iq4nl_word(3), iq4nl_word(2), sel);
  const uint32_t mask = __builtin_amdgcn_perm(y << 8, y, 0x090B080Au);
  return (hi & mask) | (lo & ~mask);
}

// get_scale_min_k4 (dequant.rs:375-383).  Branch-free (j differs between
// the lanes of a wave, so a branch would run both sides): with a = q[j & 3],
// b = q[(j & 3) + 4], c = q[(j & 3) + 8], sub-blocks 0-3 take the low 6 bits
// of a / b, sub-blocks 4-7 the nibbles of c plus the top 2 bits of a / b.
__device__ __forceinline__ void scale_min_k4(int j, const uint8_t* q, uint32_t& d, uint32_t& m) {
  const int j3 = j & 3;
  const uint32_t a = q[j3], b = q[j3 + 4], c = q[j3 + 8];
  const uint32_t hd = (c & 0x0Fu) | ((a >> 6) << 4), hm = (c >> 4) | ((b >> 6) << 4);
  const uint32_t low = j < 4 ? 0xFFu : 0u;
  d = (a & 63u & low) | (hd & ~low);
  m = (b & 63u & low) | (hm & ~low);
}

// One element j of a block at b (LDS): the IQ grid types.
template <int TAG>
__device__ __forceinline__ float decode(const uint8_t* b, int j);

// ---- IQ grid types (dequant.rs:505-719).  Codebooks: the format's fixed
// tables (iq_tables.h).  ksigns_iq2xs is computed: entry i is i with bit 7 =
// parity of i.
__constant__ uint64_t kIq2xxs[256] = {MLXQ_IQ2XXS_GRID};
__constant__ uint64_t kIq2xs[512] = {MLXQ_IQ2XS_GRID};
__constant__ uint64_t kIq2s[1024] = {MLXQ_IQ2S_GRID};
__constant__ uint32_t kIq3xxs[256] = {MLXQ_IQ3XXS_GRID};
__constant__ uint32_t kIq3s[512] = {MLXQ_IQ3S_GRID};
__constant__ uint64_t kIq1s[2048] = {MLXQ_IQ1S_GRID};
constexpr float kIq1sDelta = 0.125f;  // dequant.rs:26-27

__device__ __forceinline__ uint32_t ksigns(uint32_t i) {
  i &= 127u;
  return i | ((__popc(i) & 1u) << 7);
}
// output lane jj's sign: -1 where bit jj of the sign byte is set (dequant.rs:508-516)
__device__ __forceinline__ float iq_sign(uint32_t s, int jj) { return (s >> jj) & 1u ? -1.0f : 1.0f; }
__device__ __forceinline__ uint32_t grid_byte(uint64_t g, int jj) {
  return static_cast<uint32_t>(g >> (8 * jj)) & 0xFFu;
}

// IQ2_XXS (dequant.rs:521-539): 32-block ib32, 8-lane group l, lane jj
template <>
__device__ __forceinline__ float decode<16>(const uint8_t* b, int j) {
  const int ib32 = j >> 5, l = (j >> 3) & 3, jj = j & 7;
  const float d = rd_f16(b, 0);
  const uint8_t* q = b + 2 + 8 * ib32;
  const uint32_t aux1 = rd_u32(q + 4);
  const float db = d * (0.5f + static_cast<float>(aux1 >> 28)) * 0.25f;
  const uint64_t g = kIq2xxs[q[l]];
  return db * static_cast<float>(grid_byte(g, jj)) * iq_sign(ksigns(aux1 >> (7 * l)), jj);
}
// IQ2_XS (dequant.rs:543-564)
template <>
__device__ __forceinline__ float decode<17>(const uint8_t* b, int j) {
  const int ib32 = j >> 5, l = (j >> 3) & 3, jj = j & 7;
  const float d = rd_f16(b, 0);
  const uint32_t sc = b[66 + ib32];
  const float db = d * (0.5f + static_cast<float>(l < 2 ? (sc & 0xFu) : (sc >> 4))) * 0.25f;
  const int qo = 2 + 2 * (4 * ib32 + l);
  const uint32_t q = static_cast<uint32_t>(b[qo]) | (static_cast<uint32_t>(b[qo + 1]) << 8);
  const uint64_t g = kIq2xs[q & 511u];
  return db * static_cast<float>(grid_byte(g, jj)) * iq_sign(ksigns(q >> 9), jj);
}
// IQ2_S (dequant.rs:568-591)
template <>
__device__ __forceinline__ float decode<22>(const uint8_t* b, int j) {
  const int ib32 = j >> 5, l = (j >> 3) & 3, jj = j & 7;
  const float d = rd_f16(b, 0);
  const uint32_t sc = b[74 + ib32];
  const float db = d * (0.5f + static_cast<float>(l < 2 ? (sc & 0xFu) : (sc >> 4))) * 0.25f;
  const uint32_t idx = b[2 + 4 * ib32 + l] | ((static_cast<uint32_t>(b[66 + ib32]) << (8 - 2 * l)) & 0x300u);
  const uint64_t g = kIq2s[idx];
  return db * static_cast<float>(grid_byte(g, jj)) * iq_sign(b[34 + 4 * ib32 + l], jj);
}
// IQ3_XXS (dequant.rs:596-615): lanes 0-3 from grid point 2l, 4-7 from 2l+1
template <>
__device__ __forceinline__ float decode<18>(const uint8_t* b, int j) {
  const int ib32 = j >> 5, l = (j >> 3) & 3, jj = j & 7;
  const float d = rd_f16(b, 0);
  const uint32_t aux = rd_u32(b + 66 + 4 * ib32);
  const float db = d * (0.5f + static_cast<float>(aux >> 28)) * 0.5f;
  const uint32_t g = kIq3xxs[b[2 + 8 * ib32 + 2 * l + (jj >> 2)]];
  return db * static_cast<float>(grid_byte(g, jj & 3)) * iq_sign(ksigns(aux >> (7 * l)), jj);
}
// IQ3_S (dequant.rs:619-651): 64-element pair k, its half, 8-lane group l
template <>
__device__ __forceinline__ float decode<21>(const uint8_t* b, int j) {
  const int k = j >> 6, half = (j >> 5) & 1, l = (j >> 3) & 3, jj = j & 7;
  const float d = rd_f16(b, 0);
  const uint32_t sc = b[106 + k];
  const float db = d * static_cast<float>(1 + 2 * static_cast<int>(half ? (sc >> 4) : (sc & 0xFu)));
  const uint32_t qhb = b[66 + 2 * k + half];
  const uint8_t* q = b + 2 + 16 * k + 8 * half;
  const uint32_t idx = jj < 4 ? (q[2 * l] | ((qhb << (8 - 2 * l)) & 256u))
                              : (q[2 * l + 1] | ((qhb << (7 - 2 * l)) & 256u));
  const uint32_t g = kIq3s[idx];
  return db * static_cast<float>(grid_byte(g, jj & 3)) * iq_sign(b[74 + 8 * k + 4 * half + l], jj);
}
// IQ1_S (dequant.rs:655-673): signed grid plus a +-delta offset
template <>
__device__ __forceinline__ float decode<19>(const uint8_t* b, int j) {
  const int ib = j >> 5, l = (j >> 3) & 3, jj = j & 7;
  const float d = rd_f16(b, 0);
  const uint32_t h = static_cast<uint32_t>(b[34 + 2 * ib]) | (static_cast<uint32_t>(b[35 + 2 * ib]) << 8);
  const float dl = d * static_cast<float>(2 * static_cast<int>((h >> 12) & 7u) + 1);
  const float delta = (h & 0x8000u) ? -kIq1sDelta : kIq1sDelta;
  const uint32_t idx = b[2 + 4 * ib + l] | (((h >> (3 * l)) & 7u) << 8);
  const int v = static_cast<int8_t>(grid_byte(kIq1s[idx], jj));
  return dl * (static_cast<float>(v) + delta);
}
// IQ1_M (dequant.rs:678-719): f16 scale from the top nibbles of the four
// scale words, two 3-bit sub-scales per 32-block
template <>
__device__ __forceinline__ float decode<29>(const uint8_t* b, int j) {
  const int ib = j >> 5, l = (j >> 3) & 3, jj = j & 7;
  uint32_t sc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) sc[i] = static_cast<uint32_t>(b[48 + 2 * i]) | (static_cast<uint32_t>(b[49 + 2 * i]) << 8);
  const uint32_t bits = (sc[0] >> 12) | ((sc[1] >> 8) & 0x00F0u) | ((sc[2] >> 4) & 0x0F00u) | (sc[3] & 0xF000u);
  const float d = f16_to_f32(bits);
  const uint32_t w = sc[ib >> 1];
  const int shift = 6 * (ib & 1) + (l < 2 ? 0 : 3);
  const float dl = d * static_cast<float>(2 * static_cast<int>((w >> shift) & 7u) + 1);
  const uint32_t qh = b[32 + 2 * ib + (l >> 1)];
  const uint32_t idx = b[4 * ib + l] | ((l & 1) ? ((qh << 4) & 0x700u) : ((qh << 8) & 0x700u));
  const float delta = (qh & ((l & 1) ? 0x80u : 0x08u)) ? -kIq1sDelta : kIq1sDelta;
  const int v = static_cast<int8_t>(grid_byte(kIq1s[idx], jj));
  return dl * (static_cast<float>(v) + delta);
}

template <int TAG, int N>
__device__ __forceinline__ void decode_run(const uint8_t* b, int j, float (&v)[N]) {
  static_assert(N == 4 || N == 8 || N == 16 || N == 32, "run length");
  if constexpr (TAG == 2) {  // Q4_0 (dequant.rs:228-237): (q - 8) * d
    const float d = rd_f16(b, 0);
    nibbles16<N, 2>(b + 2, j, [&](int i, uint32_t w) {
#pragma unroll
      for (int k = 0; k < 4; k++) v[4 * i + k] = (ubyte(w, k) - 8.f) * d;
    });
  } else if constexpr (TAG == 3) {  // Q4_1 (dequant.rs:239-247): q * d + m
    const float d = rd_f16(b, 0), m = rd_f16(b, 2);
    nibbles16<N, 4>(b + 4, j, [&](int i, uint32_t w) {
#pragma unroll
      for (int k = 0; k < 4; k++) v[4 * i + k] = ubyte(w, k) * d + m;
    });
  } else if constexpr (TAG == 6) {  // Q5_0 (dequant.rs:249-261): (q - 16) * d, fifth bits in qh
    const float d = rd_f16(b, 0);
    const uint32_t qh = rd_u32(b + 2) >> (j & 31);
    nibbles16<N, 2>(b + 6, j, [&](int i, uint32_t w) {
      const uint32_t x = w | (spread4(qh >> (4 * i)) << 4);
#pragma unroll
      for (int k = 0; k < 4; k++) v[4 * i + k] = (ubyte(x, k) - 16.f) * d;
    });
  } else if constexpr (TAG == 7) {  // Q5_1 (dequant.rs:263-276): q * d + m
    const float d = rd_f16(b, 0), m = rd_f16(b, 2);
    const uint32_t qh = rd_u32(b + 4) >> (j & 31);
    nibbles16<N, 8>(b + 8, j, [&](int i, uint32_t w) {
      const uint32_t x = w | (spread4(qh >> (4 * i)) << 4);
#pragma unroll
      for (int k = 0; k < 4; k++) v[4 * i + k] = ubyte(x, k) * d + m;
    });
  } else if constexpr (TAG == 8) {  // Q8_0 (dequant.rs:278-284)
    const float d = rd_f16(b, 0);
    uint32_t w[N / 4];
    rd_words<N, 2>(b + 2 + j, w);
#pragma unroll
    for (int e = 0; e < N; e++) v[e] = sbyte(w[e >> 2], e & 3) * d;
  } else if constexpr (TAG == 10 || TAG == 11 || TAG == 14) {
    // 16 elements a scale: half h (128 elements), 32-run r, byte l of the run
    constexpr int S = N < 16 ? N : 16;
    const int h = j >> 7, r = (j >> 5) & 3;
    const float d = rd_f16(b, TAG == 10 ? 80 : TAG == 11 ? 108 : 208);
    const float dmin = TAG == 10 ? rd_f16(b, 82) : 0.f;
#pragma unroll
    for (int g = 0; g < N / S; g++) {
      const int l = (j & 31) + g * S, is = 8 * h + 2 * r + (l >> 4);
      float (&o)[N] = v;
      uint32_t w[S / 4];
      if constexpr (TAG == 10) {  // Q2_K (dequant.rs:288-318): dl * q - ml
        const uint32_t sc = b[is];
        const float dl = d * static_cast<float>(sc & 0xFu), ml = dmin * static_cast<float>(sc >> 4);
        rd_words<S, 4>(b + 16 + 32 * h + l, w);
#pragma unroll
        for (int i = 0; i < S / 4; i++) {
          const uint32_t x = (w[i] >> (2 * r)) & 0x03030303u;
#pragma unroll
          for (int k = 0; k < 4; k++) o[g * S + 4 * i + k] = dl * ubyte(x, k) - ml;
        }
      } else if constexpr (TAG == 11) {  // Q3_K (dequant.rs:320-371): dl * (2-bit code - 4 where the mask bit is clear)
        const int sc = static_cast<int>(((b[96 + (is & 7)] >> (4 * (is >> 3))) & 0xFu) |
                                        (((b[104 + (is & 3)] >> (2 * (is >> 2))) & 3u) << 4));
        const float dl = d * static_cast<float>(sc - 32);
        uint32_t m[S / 4];
        rd_words<S, 2>(b + 32 + 32 * h + l, w);
        rd_words<S, 2>(b + l, m);
#pragma unroll
        for (int i = 0; i < S / 4; i++) {
          const uint32_t x = ((w[i] >> (2 * r)) & 0x03030303u) | (((m[i] >> (4 * h + r)) & 0x01010101u) << 2);
#pragma unroll
          for (int k = 0; k < 4; k++) o[g * S + 4 * i + k] = dl * (ubyte(x, k) - 4.f);
        }
      } else {  // Q6_K (dequant.rs:446-468): (d * scale) * (q - 32)
        const float ds = d * static_cast<float>(static_cast<int8_t>(b[192 + is]));
        uint32_t u[S / 4];
        rd_words<S, 2>(b + 64 * h + 32 * (r & 1) + l, w);
        rd_words<S, 2>(b + 128 + 32 * h + l, u);
#pragma unroll
        for (int i = 0; i < S / 4; i++) {
          const uint32_t x = ((w[i] >> (4 * (r >> 1))) & 0x0F0F0F0Fu) | (((u[i] >> (2 * r)) & 0x03030303u) << 4);
#pragma unroll
          for (int k = 0; k < 4; k++) o[g * S + 4 * i + k] = ds * (ubyte(x, k) - 32.f);
        }
      }
    }
  } else if constexpr (TAG == 12 || TAG == 13) {  // Q4_K, Q5_K (dequant.rs:385-444): d1 * q - m1
    const int c = j >> 6, hi = (j >> 5) & 1, l = j & 31;
    uint32_t sc, m;
    scale_min_k4(2 * c + hi, b + 4, sc, m);
    const float d1 = rd_f16(b, 0) * static_cast<float>(sc), m1 = rd_f16(b, 2) * static_cast<float>(m);
    uint32_t w[N / 4];
    rd_words<N, (N < 16 ? N : 16)>(b + (TAG == 12 ? 16 : 48) + 32 * c + l, w);
#pragma unroll
    for (int i = 0; i < N / 4; i++) w[i] = (w[i] >> (4 * hi)) & 0x0F0F0F0Fu;
    if constexpr (TAG == 13) {  // fifth bits: bit 2c + hi of byte l
      uint32_t h[N / 4];
      rd_words<N, (N < 16 ? N : 16)>(b + 16 + l, h);
#pragma unroll
      for (int i = 0; i < N / 4; i++) w[i] |= ((h[i] >> (2 * c + hi)) & 0x01010101u) << 4;
    }
#pragma unroll
    for (int e = 0; e < N; e++) v[e] = d1 * ubyte(w[e >> 2], e & 3) - m1;
  } else if constexpr (TAG == 20) {  // IQ4_NL (dequant.rs:472-479)
    const float d = rd_f16(b, 0);
    nibbles16<N, 2>(b + 2, j, [&](int i, uint32_t w) {
      const uint32_t x = iq4nl_values(w);
#pragma unroll
      for (int k = 0; k < 4; k++) v[4 * i + k] = d * sbyte(x, k);
    });
  } else if constexpr (TAG == 23) {  // IQ4_XS (dequant.rs:481-497)
    const int ib = j >> 5;
    const int ls = static_cast<int>(((b[4 + (ib >> 1)] >> (4 * (ib & 1))) & 0xFu) | (((rd_u16(b + 2) >> (2 * ib)) & 3u) << 4));
    const float dl = rd_f16(b, 0) * static_cast<float>(ls - 32);
    nibbles16<N, 8>(b + 8 + 16 * ib, j & 31, [&](int i, uint32_t w) {
      const uint32_t x = iq4nl_values(w);
#pragma unroll
      for (int k = 0; k < 4; k++) v[4 * i + k] = dl * sbyte(x, k);
    });
  } else {
#pragma unroll
    for (int e = 0; e < N; e++) v[e] = decode<TAG>(b, j + e);
  }
}

template <int TAG> struct Geo;
template <> struct Geo<2> { static constexpr int E = 32, B = 18; };
template <> struct Geo<3> { static constexpr int E = 32, B = 20; };
template <> struct Geo<6> { static constexpr int E = 32, B = 22; };
template <> struct Geo<7> { static constexpr int E = 32, B = 24; };
template <> struct Geo<8> { static constexpr int E = 32, B = 34; };
template <> struct Geo<10> { static constexpr int E = 256, B = 84; };
template <> struct Geo<11> { static constexpr int E = 256, B = 110; };
template <> struct Geo<12> { static constexpr int E = 256, B = 144; };
template <> struct Geo<13> { static constexpr int E = 256, B = 176; };
template <> struct Geo<14> { static constexpr int E = 256, B = 210; };
template <> struct Geo<20> { static constexpr int E = 32, B = 18; };
template <> struct Geo<23> { static constexpr int E = 256, B = 136; };
template <> struct Geo<16> { static constexpr int E = 256, B = 66; };
template <> struct Geo<17> { static constexpr int E = 256, B = 74; };
template <> struct Geo<22> { static constexpr int E = 256, B = 82; };
template <> struct Geo<18> { static constexpr int E = 256, B = 98; };
template <> struct Geo<21> { static constexpr int E = 256, B = 110; };
template <> struct Geo<19> { static constexpr int E = 256, B = 50; };
template <> struct Geo<29> { static constexpr int E = 256, B = 56; };

}  // namespace
}  // namespace mlxq
