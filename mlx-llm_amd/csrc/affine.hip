// Group-wise affine quantize / dequantize for gfx950.
//
// Reference: QuantizedLinear::quantize / dequantize_weight
// (src/primitives/quant.rs:38-53, :73-81) -> mlx_rs::ops::{quantize,dequantize}
// (MLX 0.31.2); the per-group arithmetic is in affine_group.hpp.
// Layout: every lane owns 8 (f32) or 16 (bf16) consecutive elements; the lanes
// of a group reduce min/max with lane moves, then each lane packs its own
// codes into whole uint32 words.  This file is compiled with
// -ffp-contract=off: codes must be bit-identical with the CPU restatement.
#include <hip/hip_runtime.h>

#include <string>

#include "affine_group.hpp"
#include "common.hpp"

namespace mlxq {
namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// code words: any 4-byte alignment (one instruction each all the same)
typedef u32x2 u32x2_words __attribute__((aligned(4)));
typedef u32x4 u32x4_words __attribute__((aligned(4)));

constexpr int kThreads = 256;

// EPL consecutive elements (16-byte loads)
template <int DT, int EPL>
__device__ __forceinline__ void load_elems(const void* w, int64_t lane, float (&v)[EPL]) {
  constexpr int P = EPL * (DT == MLXQ_F32 ? 4 : 2) / 16;
  u32x4 p[P];
#pragma unroll
  for (int i = 0; i < P; i++) p[i] = reinterpret_cast<const u32x4*>(w)[lane * P + i];
#pragma unroll
  for (int i = 0; i < EPL; i++) {
    if constexpr (DT == MLXQ_F32) v[i] = bits_to_f32(p[i >> 2][i & 3]);
    else v[i] = bits_to_f32((i & 1) ? p[i >> 3][(i >> 1) & 3] & 0xFFFF0000u : p[i >> 3][(i >> 1) & 3] << 16);
  }
}

template <int DT>
__device__ __forceinline__ void store1(void* p, int64_t i, float v) {
  if constexpr (DT == MLXQ_F32) static_cast<float*>(p)[i] = v;
  else static_cast<uint16_t*>(p)[i] = static_cast<uint16_t>(f32_to_bf16_bits(v));
}

template <int DT>
__device__ __forceinline__ float load1(const void* p, int64_t i) {
  if constexpr (DT == MLXQ_F32) return static_cast<const float*>(p)[i];
  else return bf16_bits_to_f32(static_cast<const uint16_t*>(p)[i]);
}

// One lane per EPL elements, LPG lanes per group.  Bound by HBM (bf16 in,
// Q4 out: 2.6 bytes per element) once the per-group arithmetic is shared by
// enough elements: every lane of a group repeats it, so bf16 takes 16
// elements per lane (14336 x 4096, Q4 / Q8: 45.9 / 45.8 us with 8 elements
// and the general division, 36.3 / 37.5 with the shorter quotient, 29.6 /
// 33.1 = 5.1 / 5.4 TB/s with 16; those copies come from HBM in turn, a single
// one repeated stays partly in the 256 MB cache: 23.9 / 26.0 against 28.5 /
// 32.3).  f32 input is bound by its loads and takes
// 8 (Q4 51 -> 47.9 us; 49.7 with 16, whose loads cover a quarter of each
// line per instruction).  Two and four runs of lanes per workgroup measured
// slower (bf16 Q4 30.9, f32 Q4 51.3 us with two).
template <int DT, int BITS, int LPG, int EPL>
__global__ __launch_bounds__(kThreads) void affine_quantize_kernel(const void* __restrict__ w, int64_t n_lanes,
                                                                    uint32_t* __restrict__ wq,
                                                                    void* __restrict__ scales,
                                                                    void* __restrict__ biases) {
  constexpr int W = EPL * BITS / 32;  // words per lane
  const int64_t lane = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  float v[EPL];
  load_elems<DT, EPL>(w, min(lane, n_lanes - 1), v);  // clamped: no branch around the load
  uint32_t words[W];
  float scale, bias;
  quantize_group<BITS, LPG, EPL>(v, words, scale, bias);  // n_lanes is a multiple of LPG: a group's lanes are all real or all clamped
  if (lane >= n_lanes) return;
  if constexpr (W == 1) wq[lane] = words[0];
  else if constexpr (W == 2) *reinterpret_cast<u32x2_words*>(wq + lane * W) = u32x2{words[0], words[1]};
  else *reinterpret_cast<u32x4_words*>(wq + lane * W) = u32x4{words[0], words[1], words[2], words[3]};
  if ((threadIdx.x & (LPG - 1)) == 0) {
    const int64_t g = lane / LPG;
    store1<DT>(scales, g, scale);
    store1<DT>(biases, g, bias);
  }
}

// out = scale*q + bias in f32, then stored in DT.  Bound by HBM (4 bits or a
// byte in, 2 or 4 bytes out per element).  A unit is one 16-byte store (8
// bf16 or 4 f32 outputs) and its codes; a workgroup covers U runs of 256
// units, every run's loads first.  Each wave instruction stores 1 KB
// contiguously, so the outputs, which the kernel never reads back, go out
// non-temporal and leave the caches to the codes: 14336 x 4096, bf16 Q4 / Q8
// 31.0 / 35.0 -> 22.5 / 33.0 us, f32 Q4 / Q8 54.4 / 56.3 -> 39.2 / 52.9 (U =
// 4: 22.8 / 32.5, 39.3 / 54.1; plain stores at U = 2: 30.7 / 34.2, 56.4 /
// 53.9), on copies that come from HBM in turn; a single one repeated, whose
// codes the non-temporal stores leave in the cache, takes 22.2 / 26.3, 39.2 /
// 42.7.
template <int DT, int BITS, int U>
__global__ __launch_bounds__(kThreads) void affine_dequantize_kernel(const uint32_t* __restrict__ wq,
                                                                      const void* __restrict__ scales,
                                                                      const void* __restrict__ biases,
                                                                      int64_t n_units, int gshift,
                                                                      u32x4* __restrict__ out) {
  constexpr int E = DT == MLXQ_F32 ? 4 : 8;  // elements per unit
  constexpr int CB = E * BITS / 8;           // code bytes per unit: 2, 4 or 8
  const int64_t u0 = static_cast<int64_t>(blockIdx.x) * (kThreads * U) + threadIdx.x;
  uint32_t q[U][2];
  float s[U], b[U];
#pragma unroll
  for (int j = 0; j < U; j++) {
    const int64_t u = min(u0 + j * kThreads, n_units - 1);  // clamped: no branch around the loads
    if constexpr (CB == 2) {
      q[j][0] = reinterpret_cast<const uint16_t*>(wq)[u];
    } else if constexpr (CB == 4) {
      q[j][0] = wq[u];
    } else {
      const uint2 t = reinterpret_cast<const uint2*>(wq)[u];
      q[j][0] = t.x;
      q[j][1] = t.y;
    }
    const int64_t g = u >> gshift;
    s[j] = load1<DT>(scales, g);
    b[j] = load1<DT>(biases, g);
  }
#pragma unroll
  for (int j = 0; j < U; j++) {
    const int64_t u = u0 + j * kThreads;
    if (u >= n_units) return;
    float r[E];
#pragma unroll
    for (int i = 0; i < E; i++) {
      const uint32_t c = (q[j][i * BITS / 32] >> (i * BITS % 32)) & ((1u << BITS) - 1);
      r[i] = s[j] * static_cast<float>(c) + b[j];
    }
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if constexpr (DT == MLXQ_F32) {
        o[i] = __float_as_uint(r[i]);
      } else {
        // v_cvt_pk_bf16_f32: two values per instruction, round to nearest even
        const bf16x2_t v = {static_cast<__bf16>(r[2 * i]), static_cast<__bf16>(r[2 * i + 1])};
        o[i] = __builtin_bit_cast(uint32_t, v);
      }
    }
    __builtin_nontemporal_store(o, out + u);
  }
}

int check_args(int dtype, int64_t rows, int64_t cols, int group_size, int bits) {
  if (bits != 4 && bits != 8)
    return fail(MLXQ_ERR_UNSUPPORTED, "unsupported: bits=" + std::to_string(bits) + " (4 or 8)");
  if (group_size != 32 && group_size != 64 && group_size != 128)
    return fail(MLXQ_ERR_UNSUPPORTED, "unsupported: group_size=" + std::to_string(group_size) + " (32, 64, 128)");
  if (dtype != MLXQ_F32 && dtype != MLXQ_BF16)
    return fail(MLXQ_ERR_UNSUPPORTED, "unsupported: dtype " + std::to_string(dtype) + " (f32 or bf16)");
  if (rows < 0 || cols <= 0) return fail(MLXQ_ERR_INVALID, "quantize: bad shape");
  if (cols % group_size)
    return fail(MLXQ_ERR_SHAPE, "quantize: last dimension " + std::to_string(cols) +
                                    " is not divisible by group_size " + std::to_string(group_size));
  return MLXQ_OK;
}

template <int DT, int BITS>
void launch_quant(const void* w, int64_t n, int group_size, uint32_t* wq, void* s, void* b, hipStream_t st) {
  constexpr int EPL = DT == MLXQ_F32 ? 8 : 16;
  const int64_t lanes = n / EPL;
  const dim3 grid(ceil_div(lanes, kThreads));
  switch (group_size) {
    case 32: MLXQ_LAUNCH((affine_quantize_kernel<DT, BITS, 32 / EPL, EPL>), grid, dim3(kThreads), 0, st, w, lanes, wq, s, b); break;
    case 64: MLXQ_LAUNCH((affine_quantize_kernel<DT, BITS, 64 / EPL, EPL>), grid, dim3(kThreads), 0, st, w, lanes, wq, s, b); break;
    default: MLXQ_LAUNCH((affine_quantize_kernel<DT, BITS, 128 / EPL, EPL>), grid, dim3(kThreads), 0, st, w, lanes, wq, s, b); break;
  }
}

template <int DT, int BITS>
void launch_dequant(const uint32_t* wq, const void* s, const void* b, int64_t n, int group_size, void* out,
                    hipStream_t st) {
  constexpr int U = 2, E = DT == MLXQ_F32 ? 4 : 8;
  const int64_t units = n / E;
  MLXQ_LAUNCH((affine_dequantize_kernel<DT, BITS, U>), dim3(ceil_div(units, kThreads * U)), dim3(kThreads), 0, st, wq, s,
              b, units, __builtin_ctz(static_cast<unsigned>(group_size / E)), static_cast<u32x4*>(out));
}

}  // namespace
}  // namespace mlxq

using namespace mlxq;

extern "C" int mlxq_quantize(const void* w, int dtype, int64_t rows, int64_t cols, int group_size, int bits,
                             uint32_t* wq, void* scales, void* biases, void* stream) {
  clear_error();
  int rc = check_args(dtype, rows, cols, group_size, bits);
  if (rc) return rc;
  const int64_t n = rows * cols;
  if (n == 0) return MLXQ_OK;
  if (!w || !wq || !scales || !biases) return fail(MLXQ_ERR_INVALID, "quantize: null pointer");
  hipStream_t st = as_stream(stream);
  if (dtype == MLXQ_F32) {
    if (bits == 4) launch_quant<MLXQ_F32, 4>(w, n, group_size, wq, scales, biases, st);
    else launch_quant<MLXQ_F32, 8>(w, n, group_size, wq, scales, biases, st);
  } else {
    if (bits == 4) launch_quant<MLXQ_BF16, 4>(w, n, group_size, wq, scales, biases, st);
    else launch_quant<MLXQ_BF16, 8>(w, n, group_size, wq, scales, biases, st);
  }
  return check_launch("quantize");
}

extern "C" int mlxq_dequantize(const uint32_t* wq, const void* scales, const void* biases, int dtype, int64_t rows,
                               int64_t cols, int group_size, int bits, void* out, void* stream) {
  clear_error();
  int rc = check_args(dtype, rows, cols, group_size, bits);
  if (rc) return rc;
  const int64_t n = rows * cols;
  if (n == 0) return MLXQ_OK;
  if (!wq || !scales || !biases || !out) return fail(MLXQ_ERR_INVALID, "dequantize: null pointer");
  hipStream_t st = as_stream(stream);
  if (dtype == MLXQ_F32) {
    if (bits == 4) launch_dequant<MLXQ_F32, 4>(wq, scales, biases, n, group_size, out, st);
    else launch_dequant<MLXQ_F32, 8>(wq, scales, biases, n, group_size, out, st);
  } else {
    if (bits == 4) launch_dequant<MLXQ_BF16, 4>(wq, scales, biases, n, group_size, out, st);
    else launch_dequant<MLXQ_BF16, 8>(wq, scales, biases, n, group_size, out, st);
  }
  return check_launch("dequantize");
}
