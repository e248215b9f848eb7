// MLX group-wise affine quantization of one group, shared by the quantizer
// (affine.hip) and the fused GGUF converter (gguf_requant.hip).
//
// Reference: QuantizedLinear::quantize (src/primitives/quant.rs:38-53) ->
// mlx_rs::ops::quantize (MLX 0.31.2 semantics, restated):
//   scale = max((max - min) / n_bins, 1e-7); the edge with the larger
//   magnitude becomes the bias and the scale is snapped so that 0 is exactly
//   on the grid; code = clamp(rint((w - bias) / scale), 0, n_bins).
// Every file including this header is compiled with -ffp-contract=off: codes
// must be bit-identical with the CPU restatement.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace mlxq {
namespace {  // internal linkage: each including file has its own copy

// Correctly rounded x / n for finite x of ordinary magnitude (the quotient's
// residual is then exact): the quotient estimate and one residual step.  For
// n = 1 .. 257 and r within one ulp of 1/n (v_rcp_f32, and RN(1/n) for the
// constants 15 and 255) this equals the f32 division for every mantissa of x
// (tests/cpp/quotient_sweep.cpp); the compiler's general division is 11
// instructions.  Larger n can be off by an ulp: with x = 0x1.b5b6b2p-1 and n =
// x / 1e-7, a constant group, one of the reciprocals within an ulp of 1/n
// gives another quotient.
__device__ __forceinline__ float div_by(float x, float n, float r) {
  const float q = x * r;
  return fmaf(fmaf(-n, q, x), r, q);
}

// max / min with the value of another lane of the group, without a zeroed
// destination for the move (every lane is active)
template <int CTRL>
__device__ __forceinline__ float dpp_all(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Lane owns EPL consecutive elements v of a group of EPL * LPG; the LPG
// lanes of the group (aligned, within one wavefront) reduce min/max with
// DPP moves.  Every lane of the group must call it.  `words`: the lane's
// codes packed LSB-first.
//
// What bounds it: VALU work.  Per element: the subtraction, two instructions
// of quotient, one clamp, one rounding add and one pack.
template <int BITS, int LPG, int EPL = 8>
__device__ __forceinline__ void quantize_group(const float (&v)[EPL], uint32_t (&words)[EPL * BITS / 32], float& scale,
                                               float& bias) {
  float w_max = v[0], w_min = v[0];
#pragma unroll
  for (int i = 1; i < EPL; i++) {
    w_max = fmaxf(w_max, v[i]);
    w_min = fminf(w_min, v[i]);
  }
  // All-reduce within the LPG lanes of this group (groups never straddle a
  // 16-lane row: LPG is 1 .. 16 and the lane index is group-aligned) with
  // DPP moves: quad swaps, then the other quad of 8 (lane i <-> 7 - i), then
  // the other 8 of 16 (i <-> 15 - i).  Exact for max/min in any order.
  static_assert(LPG == 1 || LPG == 2 || LPG == 4 || LPG == 8 || LPG == 16, "lanes per group");
  if constexpr (LPG >= 2) {
    w_max = fmaxf(w_max, dpp_all<kDppQuadXor1>(w_max));
    w_min = fminf(w_min, dpp_all<kDppQuadXor1>(w_min));
  }
  if constexpr (LPG >= 4) {
    w_max = fmaxf(w_max, dpp_all<kDppQuadXor2>(w_max));
    w_min = fminf(w_min, dpp_all<kDppQuadXor2>(w_min));
  }
  if constexpr (LPG >= 8) {
    w_max = fmaxf(w_max, dpp_all<kDppRowHalfMirror>(w_max));
    w_min = fminf(w_min, dpp_all<kDppRowHalfMirror>(w_min));
  }
  if constexpr (LPG >= 16) {
    w_max = fmaxf(w_max, dpp_all<kDppRowMirror>(w_max));
    w_min = fminf(w_min, dpp_all<kDppRowMirror>(w_min));
  }

  constexpr float n_bins = static_cast<float>((1 << BITS) - 1);
  constexpr int CPW = 32 / BITS;  // codes per word
  const float eps = 1e-7f;
  const bool mask = fabsf(w_min) > fabsf(w_max);
  const float edge = mask ? w_min : w_max;
  scale = fmaxf(div_by(w_max - w_min, n_bins, 1.0f / n_bins), eps);
  scale = mask ? scale : -scale;
  // rint(fl(x / s)), fl the correctly rounded f32 division, is rint of
  // fma(x, r1, x r2) with r1 + r2 = 1/s to about 48 bits: the two quotients
  // can only round apart next to a half-integer, and there they were compared
  // on gfx950 for every mantissa of s, every half-integer up to 256.5 and the
  // nine x around their product (on the CPU, with every reciprocal within an
  // ulp and most of those mantissas: tests/cpp/quotient_sweep.cpp); the one
  // mantissa that differs (all ones, x/s next to 0.5) takes the division
  // below.  The comparison carries over to any scale whose products neither
  // overflow nor lose their residuals: s is at least 0.5e-7, and |x| at most
  // 2^60 is tested.
  auto recip = [](float s, float& r1, float& r2) {
    const float r0 = __builtin_amdgcn_rcpf(s);
    r1 = fmaf(fmaf(-s, r0, 1.0f), r0, r0);
    r2 = fmaf(-s, r1, 1.0f) * r1;
  };
  float r1, r2;
  recip(scale, r1, r2);
  const float q0 = __builtin_rintf(fmaf(edge, r1, edge * r2));
  bias = 0.f;
  if (q0 != 0.f) {
    scale = div_by(edge, q0, __builtin_amdgcn_rcpf(q0));
    bias = edge;
  }
  recip(scale, r1, r2);
  // false for an infinite or NaN edge too (a finite edge bounds the group).
  // |q0| is at most n_bins + 1 in a group with values of both signs, but edge
  // / scale, up to 2^60 / 1e-7, in a narrow one of one sign: past 256 neither
  // quotient above was compared.
  const bool ordinary = fabsf(edge) <= 0x1p60f && fabsf(q0) <= 256.f &&
                        (__float_as_uint(scale) & 0x7FFFFFu) != 0x7FFFFFu;
  // The quotient lies in [0, n_bins + 1] (bias is the group's edge and scale
  // of the sign that makes it positive; with bias 0 it rounds to 0); a NaN
  // element clamps to 0.  Adding 2^23 rounds it to the nearest integer, ties
  // to even, into the low mantissa bits; the words collect those bits, the
  // exponent bits that the shifts leave behind are a constant.
#pragma unroll
  for (int w = 0; w < EPL / CPW; w++) {
    uint32_t acc = 0;
#pragma unroll
    for (int i = CPW - 1; i >= 0; i--) {
      const float d = v[w * CPW + i] - bias;
      const float q = __builtin_amdgcn_fmed3f(fmaf(d, r1, d * r2), 0.f, n_bins);
      acc = (acc << BITS) + __float_as_uint(q + 0x1p23f);
    }
    words[w] = acc - (BITS == 4 ? 0xFB000000u : 0x4B000000u);  // sum of 0x4B000000 << BITS i
  }
  if (!ordinary) {  // the whole group takes it: the divisions themselves
    scale = fmaxf((w_max - w_min) / n_bins, eps);
    scale = mask ? scale : -scale;
    const float qe = __builtin_rintf(edge / scale);
    bias = 0.f;
    if (qe != 0.f) {
      scale = edge / qe;
      bias = edge;
    }
#pragma unroll
    for (int w = 0; w < EPL / CPW; w++) {
      words[w] = 0;
#pragma unroll
      for (int i = 0; i < CPW; i++) {
        const float q = fminf(fmaxf(__builtin_rintf((v[w * CPW + i] - bias) / scale), 0.f), n_bins);
        words[w] |= static_cast<uint32_t>(q) << (BITS * i);
      }
    }
  }
}

}  // namespace
}  // namespace mlxq
