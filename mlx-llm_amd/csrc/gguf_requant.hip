// Fused GGUF -> MLX affine requantization of a projection weight, on device.
//
// Reference: the convert chain of src/gguf/convert.rs for a projection
// tensor: dequantize (:131, dequant.rs:156-211), the llama q/k row
// un-permute (:133-137, permute_inverse_qk :232-256), the cast to bf16
// (:156, as_dtype(bf16): round to nearest even) and the snapshot writer's
// requant (:176 -> snapshot.rs:100-107 -> quant.rs:44, mlx quantize of the
// bf16 tensor).  The reference materializes the whole f32 tensor on the host
// and then the bf16 copy; here every lane decodes consecutive elements of its
// output row straight from the GGUF blocks (un-permuted source row), rounds
// them to bf16 and quantizes its share of the group in registers, so the only
// HBM traffic is the GGUF bytes in and the packed MLX tensor out.
//
// Bit-exactness: the element decode (gguf_decode.hpp) and the group
// quantization (affine_group.hpp) are the ones of mlxq_gguf_dequantize and
// mlxq_quantize; this file is compiled with -ffp-contract=off.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "affine_group.hpp"
#include "common.hpp"
#include "gguf_decode.hpp"

namespace mlxq {
namespace {

constexpr int kThreads = 256;
constexpr int kUnit = 32;  // block formats: elements per lane
constexpr int kFloatUnit = 16;  // float tensors: elements per lane

template <int TAG>
constexpr bool is_float_tag() {
  return TAG == 0 || TAG == 1 || TAG == 30;
}

// 16 bytes per lane from global memory straight into LDS: a wave's active
// lanes fill lane * 16 bytes from `l` (no registers held while in flight)
__device__ __forceinline__ void lds_dma16(const uint8_t* g, uint8_t* l) {
  __builtin_amdgcn_global_load_lds(g, l, 16, 0, 0);
}

// Source row of output row r: perm_hd > 0 un-permutes llama.cpp's q/k head
// interleave -- within head h = r / perm_hd, output row rr = r % perm_hd
// reads source row h * perm_hd + 2 * (rr % half) + rr / half (half =
// perm_hd / 2).
__device__ __forceinline__ int source_row(int r, int perm_hd) {
  if (perm_hd <= 0) return r;
  const int h = r / perm_hd, rr = r - h * perm_hd, half = perm_hd / 2;
  return h * perm_hd + 2 * (rr % half) + rr / half;
}

// as_dtype(bf16): v_cvt_pk_bf16_f32, round to nearest even (a NaN payload
// cannot reach a code: max/min skip NaN and a NaN quotient clamps to 0)
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
template <int N>
__device__ __forceinline__ void round_bf16(float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; i += 2) {
    const bf16x2_t t = {static_cast<__bf16>(v[i]), static_cast<__bf16>(v[i + 1])};
    const uint32_t u = __builtin_bit_cast(uint32_t, t);
    v[i] = bits_to_f32(u << 16);
    v[i + 1] = bits_to_f32(u & 0xFFFF0000u);
  }
}

// the words of a lane's codes (16-byte stores, wq at any 8-byte alignment),
// and its group's scale and bias from the group's first lane
typedef uint32_t u32x4_words __attribute__((ext_vector_type(4), aligned(8)));
template <int BITS, int LPG, int EPL>
__device__ __forceinline__ void store_group(const uint32_t (&words)[EPL * BITS / 32], float scale, float bias,
                                            int64_t lane, uint32_t* wq, uint16_t* scales, uint16_t* biases) {
  constexpr int W = EPL * BITS / 32;
  if constexpr (W == 2) {
    reinterpret_cast<uint2*>(wq)[lane] = make_uint2(words[0], words[1]);
  } else {
#pragma unroll
    for (int j = 0; j < W / 4; j++)
      *reinterpret_cast<u32x4_words*>(wq + lane * W + 4 * j) =
          u32x4_words{words[4 * j], words[4 * j + 1], words[4 * j + 2], words[4 * j + 3]};
  }
  if ((threadIdx.x & (LPG - 1)) == 0) {
    const int64_t g = lane / LPG;
    scales[g] = static_cast<uint16_t>(f32_to_bf16_bits(scale));
    biases[g] = static_cast<uint16_t>(f32_to_bf16_bits(bias));
  }
}

// A workgroup converts `rpw` consecutive output rows of a block format.  All
// of their source rows' GGUF bytes are requested up front (direct global ->
// LDS loads when 16-byte aligned), then every lane decodes 32 consecutive
// elements of a row from LDS, rounds them to bf16 and quantizes its share of
// the group.  Bound by the VALU (instructions per element: Q8_0 15.3, IQ4_NL
// 17.3, Q4_K 18.3, Q6_K 19.0): a lane repeats its block's header decode and
// its group's scale arithmetic, so 32 elements share them.  14336 x 4096 to
// Q4 g64, 16 elements per lane with a
// generic decode -> here (us): Q4_0 45.1 -> 30.5, Q5_0 53.4 -> 32.8, Q8_0
// 42.9 -> 31.5, Q2_K 46.1 -> 28.9, Q3_K 76.3 -> 33.9, Q4_K 48.4 -> 32.4, Q5_K
// 55.1 -> 29.2, Q6_K 54.4 -> 34.1, IQ4_NL 48.2 -> 30.7, IQ4_XS 49.7 -> 31.6.
template <int TAG, int BITS, int LPG>
__global__ __launch_bounds__(kThreads) void gguf_requant_kernel(const uint8_t* __restrict__ data, int rows, int K,
                                                                 int row_bytes, int perm_hd, int rpw, int aligned16,
                                                                 float rcp_lpr, uint32_t* __restrict__ wq,
                                                                 uint16_t* __restrict__ scales,
                                                                 uint16_t* __restrict__ biases) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int r0 = blockIdx.x * rpw;
  const int nr = min(rpw, rows - r0);
  const int tid = threadIdx.x;
  if (aligned16) {
    const int n16 = row_bytes >> 4;
    const int pieces = (n16 + 63) >> 6;  // 1 KB wave loads per row
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    for (int t = wave; t < nr * pieces; t += kThreads / 64) {
      const int i = t / pieces, p = t - i * pieces, q = p * 64 + lane;
      const uint8_t* src = data + static_cast<int64_t>(source_row(r0 + i, perm_hd)) * row_bytes;
      if (q < n16) lds_dma16(src + q * 16, lds + i * row_bytes + p * 1024);
    }
    __builtin_amdgcn_s_waitcnt(0);
  } else {
    for (int i = 0; i < nr; i++) {
      const uint8_t* src = data + static_cast<int64_t>(source_row(r0 + i, perm_hd)) * row_bytes;
      for (int j = tid; j < row_bytes; j += kThreads) lds[i * row_bytes + j] = src[j];
    }
  }
  __syncthreads();
  // the rows' units in one run: a group's lanes are adjacent (units per row
  // and kThreads are multiples of LPG), lanes past the end repeat the last
  // unit and store nothing
  constexpr int E = Geo<TAG>::E, B = Geo<TAG>::B;
  const int lpr = K / kUnit, units = nr * lpr;
  for (int u0 = 0; u0 < units; u0 += kThreads) {
    const int u = min(u0 + tid, units - 1);
    // u / lpr: below 2^20 the f32 quotient of u + 1/2 cannot cross an integer
    const int i = static_cast<int>((static_cast<float>(u) + 0.5f) * rcp_lpr);
    const int l = u - i * lpr;
    const uint8_t* b = lds + i * row_bytes + (E == 32 ? l : l >> 3) * B;
    float v[kUnit];
    decode_run<TAG, kUnit>(b, E == 32 ? 0 : (l & 7) * kUnit, v);
    round_bf16(v);
    uint32_t words[kUnit * BITS / 32];
    float scale, bias;
    quantize_group<BITS, LPG, kUnit>(v, words, scale, bias);
    if (u0 + tid < units)
      store_group<BITS, LPG, kUnit>(words, scale, bias, static_cast<int64_t>(r0) * lpr + u, wq, scales, biases);
  }
}

// F32 / F16 / BF16 tensors: nothing is shared between lanes, so each lane
// takes its 16 elements straight from global memory (any alignment).  Bound
// by HBM; through LDS with a per-element decode -> here (us, 14336 x 4096 to
// Q4 g64): F16 72.2 -> 30.5, BF16 41.8 -> 28.1, F32 54.6 -> 48.9.
template <int TAG, int BITS, int LPG>
__global__ __launch_bounds__(kThreads) void float_requant_kernel(const uint8_t* __restrict__ data, int64_t n_lanes,
                                                                  int lpr, int perm_hd, uint32_t* __restrict__ wq,
                                                                  uint16_t* __restrict__ scales,
                                                                  uint16_t* __restrict__ biases) {
  constexpr int B = kFloatUnit * (TAG == 0 ? 4 : 2);  // source bytes per lane
  const int64_t lane = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  int64_t src = min(lane, n_lanes - 1);
  if (perm_hd > 0) {
    int64_t r;
    if (n_lanes <= UINT32_MAX) r = static_cast<uint32_t>(src) / static_cast<uint32_t>(lpr);
    else r = src / lpr;
    src += (static_cast<int64_t>(source_row(static_cast<int>(r), perm_hd)) - r) * lpr;
  }
  uint32_t w[B / 4];
  __builtin_memcpy(w, data + src * B, B);
  float v[kFloatUnit];
#pragma unroll
  for (int i = 0; i < kFloatUnit; i++) {
    if constexpr (TAG == 0) v[i] = bits_to_f32(w[i]);
    else if constexpr (TAG == 1) v[i] = f16_to_f32((w[i >> 1] >> (16 * (i & 1))) & 0xFFFFu);
    else v[i] = bits_to_f32((i & 1) ? w[i >> 1] & 0xFFFF0000u : w[i >> 1] << 16);
  }
  if constexpr (TAG != 30) round_bf16(v);
  uint32_t words[kFloatUnit * BITS / 32];
  float scale, bias;
  quantize_group<BITS, LPG, kFloatUnit>(v, words, scale, bias);
  if (lane < n_lanes) store_group<BITS, LPG, kFloatUnit>(words, scale, bias, lane, wq, scales, biases);
}

// Rows per workgroup: one 32-element unit for each of the 256 threads, so
// that a CU holds several workgroups in different phases and one's loads run
// beside another's arithmetic (14336 x 4096, 2 rows against 8: Q4_K 32.4 /
// 33.2 us, Q5_K 29.2 / 30.9, Q8_0 31.5 / 35.3; 16 rows: 35.8 / 38.7 / 35.4),
// at most 32 KB of LDS.
inline int rows_per_workgroup(int units_per_row, int row_bytes) {
  return std::max(1, std::min(static_cast<int>(ceil_div(kThreads, units_per_row)), (32 * 1024) / std::max(row_bytes, 1)));
}

template <int TAG, int BITS, int GS>
int launch_gs(int rows, int K, int row_bytes, int perm_hd, const uint8_t* d, uint32_t* wq, uint16_t* s, uint16_t* b,
              hipStream_t st) {
  if constexpr (is_float_tag<TAG>()) {
    const int lpr = K / kFloatUnit;
    const int64_t lanes = static_cast<int64_t>(rows) * lpr;
    MLXQ_LAUNCH((float_requant_kernel<TAG, BITS, GS / kFloatUnit>), dim3(static_cast<unsigned>(ceil_div(lanes, kThreads))),
                dim3(kThreads), 0, st, d, lanes, lpr, perm_hd, wq, s, b);
  } else {
    const bool al = (reinterpret_cast<uintptr_t>(d) & 15u) == 0 && row_bytes % 16 == 0;
    const int rpw = rows_per_workgroup(K / kUnit, row_bytes);
    const size_t lds = static_cast<size_t>(rpw) * row_bytes;
    const dim3 grid(static_cast<unsigned>((rows + rpw - 1) / rpw));
    auto kern = gguf_requant_kernel<TAG, BITS, GS / kUnit>;
    if (lds > 64 * 1024) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
      if (e != hipSuccess)
        return fail(MLXQ_ERR_DEVICE, std::string("gguf_requantize: LDS size: ") + hipGetErrorString(e));
    }
    MLXQ_LAUNCH(kern, grid, dim3(kThreads), lds, st, d, rows, K, row_bytes, perm_hd, rpw, static_cast<int>(al),
                1.0f / static_cast<float>(K / kUnit), wq, s, b);
  }
  return check_launch("gguf_requantize");
}

template <int TAG, int BITS>
int launch_bits(int group_size, int rows, int K, int row_bytes, int perm_hd, const uint8_t* d, uint32_t* wq,
                uint16_t* s, uint16_t* b, hipStream_t st) {
  if (group_size == 32) return launch_gs<TAG, BITS, 32>(rows, K, row_bytes, perm_hd, d, wq, s, b, st);
  if (group_size == 64) return launch_gs<TAG, BITS, 64>(rows, K, row_bytes, perm_hd, d, wq, s, b, st);
  return launch_gs<TAG, BITS, 128>(rows, K, row_bytes, perm_hd, d, wq, s, b, st);
}

template <int TAG>
int launch_tag(int bits, int group_size, int rows, int K, int row_bytes, int perm_hd, const uint8_t* d,
               uint32_t* wq, uint16_t* s, uint16_t* b, hipStream_t st) {
  if (bits == 4) return launch_bits<TAG, 4>(group_size, rows, K, row_bytes, perm_hd, d, wq, s, b, st);
  return launch_bits<TAG, 8>(group_size, rows, K, row_bytes, perm_hd, d, wq, s, b, st);
}

}  // namespace
}  // namespace mlxq

using namespace mlxq;

extern "C" int mlxq_gguf_requantize(uint32_t tag, const void* data, int64_t data_len, int64_t rows, int64_t cols,
                                    int permute_heads, int group_size, int bits, uint32_t* wq, void* scales,
                                    void* biases, void* stream) {
  clear_error();
  if (bits != 4 && bits != 8) return fail(MLXQ_ERR_UNSUPPORTED, "gguf_requantize: bits must be 4 or 8");
  if (group_size != 32 && group_size != 64 && group_size != 128)
    return fail(MLXQ_ERR_UNSUPPORTED, "gguf_requantize: group_size must be 32, 64 or 128");
  if (rows < 0 || cols <= 0 || permute_heads < 0) return fail(MLXQ_ERR_INVALID, "gguf_requantize: bad shape");
  if (cols % group_size)
    return fail(MLXQ_ERR_SHAPE, "gguf_requantize: cols=" + std::to_string(cols) + " not divisible by group_size");
  if (cols > INT32_MAX / 2 || rows > INT32_MAX) return fail(MLXQ_ERR_INVALID, "gguf_requantize: too large");
  int64_t elems = 0, bbytes = 0;
  if (int rc = mlxq_gguf_block(tag, &elems, &bbytes)) return rc;
  const bool device_tag = tag == 0 || tag == 1 || tag == 30 || tag == 2 || tag == 3 || tag == 6 || tag == 7 ||
                          tag == 8 || tag == 10 || tag == 11 || tag == 12 || tag == 13 || tag == 14 || tag == 20 ||
                          tag == 23 || tag == 16 || tag == 17 || tag == 22 || tag == 18 || tag == 21 || tag == 19 ||
                          tag == 29;
  if (!device_tag) return fail(MLXQ_ERR_UNSUPPORTED, "gguf_requantize: GGUF type " + std::to_string(tag) +
                                                         " has no device decoder");
  if (cols % elems) return fail(MLXQ_ERR_SHAPE, "gguf_requantize: rows must hold whole blocks");
  const int64_t n = rows * cols;
  const int64_t need = n / elems * bbytes;
  if (data_len < need)
    return fail(MLXQ_ERR_SHORT_BUFFER, "gguf_requantize: need " + std::to_string(need) + " bytes of blocks, got " +
                                           std::to_string(data_len));
  int perm_hd = 0;
  if (permute_heads > 0) {
    if (rows % permute_heads) return fail(MLXQ_ERR_SHAPE, "gguf_requantize: rows not divisible by the head count");
    perm_hd = static_cast<int>(rows / permute_heads);
    if (perm_hd % 2) return fail(MLXQ_ERR_SHAPE, "gguf_requantize: odd head_dim");
  }
  if (n == 0) return MLXQ_OK;
  if (!data || !wq || !scales || !biases) return fail(MLXQ_ERR_INVALID, "gguf_requantize: null pointer");
  if ((reinterpret_cast<uintptr_t>(wq) & 7u)) return fail(MLXQ_ERR_INVALID, "gguf_requantize: wq must be 8-byte aligned");
  const int64_t row_bytes = cols / elems * bbytes;
  if (row_bytes > 160 * 1024) return fail(MLXQ_ERR_UNSUPPORTED, "gguf_requantize: row larger than LDS");
  const int K = static_cast<int>(cols), R = static_cast<int>(rows), RB = static_cast<int>(row_bytes);
  const uint8_t* d = static_cast<const uint8_t*>(data);
  uint16_t* s = static_cast<uint16_t*>(scales);
  uint16_t* b = static_cast<uint16_t*>(biases);
  hipStream_t st = as_stream(stream);
  switch (tag) {
    case 0: return launch_tag<0>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 1: return launch_tag<1>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 30: return launch_tag<30>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 2: return launch_tag<2>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 3: return launch_tag<3>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 6: return launch_tag<6>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 7: return launch_tag<7>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 8: return launch_tag<8>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 10: return launch_tag<10>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 11: return launch_tag<11>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 12: return launch_tag<12>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 13: return launch_tag<13>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 14: return launch_tag<14>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 20: return launch_tag<20>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 16: return launch_tag<16>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 17: return launch_tag<17>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 22: return launch_tag<22>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 18: return launch_tag<18>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 21: return launch_tag<21>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 19: return launch_tag<19>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    case 29: return launch_tag<29>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
    default: return launch_tag<23>(bits, group_size, R, K, RB, perm_hd, d, wq, s, b, st);
  }
}
