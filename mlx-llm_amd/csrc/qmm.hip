// Prefill-shaped quantized matmul (qmm) for gfx950: y[M,N] = x[M,K] . W^T,
// W group-wise affine quantized (Q4 / Q8), any M; K a multiple of 512 and
// of 8 groups.
//
// Reference: QuantizedLinear::forward (src/primitives/quant.rs:56-70) ->
// mlx_rs::ops::quantized_matmul, which MLX serves with its qmm kernels when M
// is large (prefill, batched decode).
//
// Design (MFMA-bound at prefill sizes):
//  * Workgroup tile BM x 256 (BM = 256 or 128), four waves side by side
//    along N; each wave owns BM x 64 of the output as (BM/32) x 2 tiles of
//    v_mfma_f32_32x32x16_bf16 with f32 accumulators (up to 256 per lane, in
//    the accumulator registers).  K advances 64 per step.
//  * Everything arrives by LDS DMA (global_load_lds_dwordx4: no VGPRs, no
//    VALU), in whole 128-byte lines: the memory path pays per line touched,
//    so a 32-byte slice of a code row costs as much as a full line.
//      - activations: the BM x 64 bf16 tile of one step (one line per row),
//        four stages (128-row tiles; short Q8 slices of group size 32 two) or
//        two, requested that many steps ahead;
//      - codes: 128 bytes of each of the 256 weight rows (4 steps at Q4, 2
//        at Q8), two buffers, requested a few at a time over the steps;
//      - scales and biases: 16 bytes per row and array (8 steps of groups),
//        two buffers.
//    Rows are stored with their 16-byte chunks permuted (chunk c of row r at
//    c ^ swz(r)), which makes the 16-byte fragment reads bank-conflict free.
//  * Weights are dequantized straight into the MFMA B-operand layout in
//    registers, by the wave that multiplies them: lane (n, h) of a 32-column
//    tile takes the 32 codes k0 + 32h .. +32 of weight row n (one 16-byte LDS
//    read at Q4), and for sub-step j the 8 codes 32h + 8j .. +8 become its
//    bf16x8 operand (bf16(s * q + b): f32 FMA, round to nearest even).  The
//    activation fragment of sub-step j is the 16-byte chunk 4h + j of the
//    row: both operands follow the same k order, which the MFMA sums over.
//    No weight tile is written to LDS.
//  * Measured (us, M = 2048 on 4096 x 14336, M = 512 and 1024 on 14336 x
//    4096, Q4): 202.4, 67.2, 127.8 -> 192.9, 63.7, 118.4 with the mixed FMA
//    decode, paired requests, one wait per sub-step, four activation stages
//    and spread code requests (Q8 the same: 218.1 -> 211.2, 74.9 -> 71.9).
//    256 MFMA streams of random data draw enough power to run at 1.8 GHz (18
//    ns per MFMA, 13.6 on up to 128 CUs): 147 us of the 193; the decode costs
//    about 25, the LDS reads and requests the rest.
//  * Step k's MFMAs use the operands decoded during step k-1: the wave
//    alternates one MFMA (32 cycles on the matrix core) with a few decode
//    instructions and LDS reads, in a fixed per-step schedule.
//  * Tiles are ordered so that each XCD (workgroups round-robin over the 8
//    XCDs) takes a contiguous, M-major run of tiles: the workgroups of one
//    XCD share activation rows in that XCD's L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <utility>

#include "common.hpp"
#include "qmatmul.hpp"

namespace mlxq {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int BK = 64;      // K per step
constexpr int PERIOD = 8;   // steps per unrolled period (one scale batch)

template <int BITS, int GS, int TM, int TN, int ST>
struct QmmGeom {
  static constexpr int WAVES = 4, THREADS = 64 * WAVES;
  static constexpr int BN = 256;               // weight rows per workgroup
  static constexpr int WN = BN / (32 * TN);    // waves along N (each TN 32-column tiles)
  static constexpr int WM = WAVES / WN;        // waves along M (each TM 32-row tiles)
  static constexpr int BM = WM * TM * 32;
  static constexpr int A_BYTES = BM * BK * 2;  // activation tile of one step
  static constexpr int CROW = BK * BITS / 8;   // code bytes per weight row per step
  static constexpr int CB = 128 / CROW;        // steps per code batch (one 128-byte line per row)
  static constexpr int C_BYTES = BN * 128;
  static constexpr int SROW = GS == 32 ? 32 : 16;  // scale bytes per row per batch (and bias bytes)
  static constexpr int S_BYTES = BN * 2 * SROW;
  static constexpr int AST = ST;  // activation stages
  static constexpr int A_OFF = 0, C_OFF = AST * A_BYTES, S_OFF = C_OFF + 2 * C_BYTES;
  static constexpr int LDS_BYTES = S_OFF + 2 * S_BYTES;
  // DMA instructions per wave: activations per step, codes / scales per batch
  static constexpr int A_DMA = A_BYTES / 1024 / WAVES;
  static constexpr int C_DMA = C_BYTES / 1024 / WAVES;
  static constexpr int S_DMA = S_BYTES / 1024 / WAVES;
  static constexpr int CW = BITS == 4 ? 1 : 2;  // 16-byte code reads per lane per tile per step
  static_assert(A_BYTES % (1024 * WAVES) == 0 && C_BYTES % (1024 * WAVES) == 0 && S_BYTES % (1024 * WAVES) == 0,
                "whole DMA chunks");
  static_assert(PERIOD % CB == 0, "code batches tile the period");
  static_assert(WM * WN == WAVES && TM % 2 == 0 && TN % 2 == 0, "wave grid");
  // activation fragments: two register sets where they fit (128-row tiles)
  static constexpr int ASETS = TM <= 4 ? 2 : 1;
  // slot of the step boundary, where every activation read of the step has
  // been issued: with two sets those of the last sub-step go out in the first
  // TM slots of the third, with one at its end
  static constexpr int BOUNDARY = ASETS == 2 ? 2 * TM * TN + TM + 2 : 3 * TM * TN + 1;
  static_assert(A_DMA % 2 == 0 && C_DMA % 4 == 0, "DMA pairs");
  static_assert(LDS_BYTES <= 160 * 1024, "fits in LDS");
  static_assert(CB == 2 || CB == 4, "code batch schedule");
  // Requests of step u (mod PERIOD), in issue order: after its boundary the
  // activations of step u + AST into the stage that the boundary freed; then,
  // in the next step's first slots, pairs [c_lo, c_hi) of a code batch and the
  // scale batch two periods on.  Batch b is last read right after boundary CB
  // b + CB - 3, so its buffer is free from the next boundary on: batch b + 2
  // is requested by steps 4b + 2 and 4b + 3 (Q4) or 2b (Q8).  Codes come from
  // HBM: spread out, so that they do not fill the miss queues at once, and
  // waited for three (Q4) or two (Q8) steps after their request.
  static constexpr int mod(int u, int n) { return ((u % PERIOD) + PERIOD) % n; }
  static constexpr int C_PAIRS = C_DMA / 2;
  static constexpr int c_lo(int u) { return CB == 4 && mod(u, 4) == 3 ? C_PAIRS / 2 : 0; }
  static constexpr int c_hi(int u) {
    if (CB == 2) return mod(u, 2) == 0 ? C_PAIRS : 0;
    return mod(u, 4) == 2 ? C_PAIRS / 2 : mod(u, 4) == 3 ? C_PAIRS : 0;
  }
  static constexpr int C_AHEAD = CB == 2 ? 4 : 8;  // step kt requests from batch (kt + C_AHEAD) / CB
  static constexpr int s_num(int u) { return mod(u, PERIOD) == PERIOD - 2 ? S_DMA : 0; }
  static constexpr int step_num(int u) { return A_DMA + 2 * (c_hi(u) - c_lo(u)) + s_num(u); }
  // Requests that may still be in flight at boundary u: those issued after the
  // activations of step u + 1 and, where step u + 2 opens a code batch, after
  // that batch's last pair (scale batches are older than either).
  static constexpr int in_flight(int u) {
    int a = step_num(u + 1 - AST) - A_DMA;
    for (int v = u + 2 - AST; v < u; v++) a += step_num(v);
    if ((u + 2) % CB == 0) {
      const int w = u - (CB == 2 ? 2 : 3);
      int c = s_num(w);
      for (int v = w + 1; v < u; v++) c += step_num(v);
      a = c < a ? c : a;
    }
    return a;
  }
  static_assert(4 * TM * TN > BOUNDARY + A_DMA / 2 && BOUNDARY > 2 * C_PAIRS + S_DMA, "DMA slots");
};

// LDS DMA of 16 bytes per lane (global_load_lds_dwordx4): lane l's bytes
// land at lds + 16 l.  Written out rather than through the compiler's
// builtin: the builtin only emits the 64-bit per-lane address form, while
// the SGPR-base form (wave-uniform base + 32-bit per-lane offset) carries
// half the per-lane address data, which the issuing wave pays for.  Every
// LDS DMA of this kernel goes through these functions, so M0 (the LDS
// destination) is only ever written here, right before its use; the caller
// accounts for them in its own s_waitcnt vmcnt (the compiler does not count
// inline assembly).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// Two requests for consecutive KB of LDS: the instruction's offset moves the
// LDS destination and the memory address alike, so one M0 serves both, and
// off1 is the second request's offset less 1024 (from a base 1024 lower, so
// that it cannot be negative).  Every first offset is then 1024 more than the
// byte it names and has to fit 32 bits all the same.
constexpr uint32_t kDmaBias = 1024;
__device__ __forceinline__ void dma16x2_to_lds_sbase(const void* base, uint32_t off0, uint32_t off1,
                                                     unsigned char* lds) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds)));
  asm volatile(
      "s_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024" ::"v"(
          off0),
      "v"(off1), "s"(base), "s"(m0)
      : "memory", "m0");
}
__device__ __forceinline__ void dma16_to_lds(const void* g, unsigned char* lds) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds)));
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(m0) : "memory", "m0");
}
#pragma clang diagnostic pop

// s_waitcnt with only the vector-memory counter limited to n (gfx9 encoding)
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
// ... with only the LDS counter limited to n
template <int N>
__device__ __forceinline__ void wait_lgkm() {
  static_assert(N >= 0 && N < 16, "lgkmcnt range");
  __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8));
}
__device__ __forceinline__ void wait_lgkm0() { wait_lgkm<0>(); }

// 16-byte chunk position of logical chunk c in 128-byte LDS row r is
// c ^ swz(r): a bijection within the row under which rows 0..15 at one c
// hit distinct banks
__device__ __forceinline__ int swz(int r) { return (r ^ (r >> 3)) & 7; }

// f(integral_constant<int, I>) for I = 0 .. N-1, unrolled at compile time
template <typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
  (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  bf16x2 v;
  v[0] = static_cast<__bf16>(a);  // v_cvt_pk_bf16_f32: round to nearest even
  v[1] = static_cast<__bf16>(b);
  return __builtin_bit_cast(uint32_t, v);
}

template <int BITS, int GS, int TM, int TN, int ST>
__device__ __forceinline__ void qmm_tile(const uint16_t* __restrict__ x, int M, const uint32_t* __restrict__ wq,
                                         const uint16_t* __restrict__ scales, const uint16_t* __restrict__ biases,
                                         const uint16_t* __restrict__ bias_vec, int N, int K,
                                         uint16_t* __restrict__ y, float* __restrict__ part, int grain,
                                         int slice_grains, int longer) {
  using Gm = QmmGeom<BITS, GS, TM, TN, ST>;
  constexpr int BM = Gm::BM, BN = Gm::BN, CB = Gm::CB;
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % Gm::WN, wm = wave / Gm::WN;  // this wave's column / row block

  // tile of this workgroup: XCD blockIdx.x % 8 takes tiles [xcd * per, (xcd + 1) * per)
  const int nbn = (N + BN - 1) / BN, nbm = (M + BM - 1) / BM;
  const int tiles = nbn * nbm, per = (tiles + 7) / 8;
  const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (t >= tiles) return;
  const int m0 = (t / nbn) * BM, n0 = (t % nbn) * BN;
  // split K: the first `longer` slices take slice_grains + 1 grains of K, the
  // others slice_grains
  const int sl = blockIdx.y;
  const int kb = (sl * slice_grains + min(sl, longer)) * grain;            // first K of this slice
  const int KT = (slice_grains + (sl < longer ? 1 : 0)) * (grain / BK);    // a multiple of PERIOD
  const int G = K / GS;
  const uint32_t row_bytes = static_cast<uint32_t>(K) * BITS / 8;

  // ---- DMA sources: per-lane byte offsets (32-bit: the host checks sizes)
  // activations: 1 KB chunk q = 8 rows; lane -> row 8q + lane/8, chunk position
  // lane % 8 (at most M K 2 + 112, K a multiple of 512: it fits wherever the
  // activations are below 4 GiB)
  uint32_t a_off[Gm::A_DMA];
#pragma unroll
  for (int i = 0; i < Gm::A_DMA; i++) {
    const int r = 8 * (wave * Gm::A_DMA + i) + (lane >> 3), c = (lane & 7) ^ swz(r);
    a_off[i] = (static_cast<uint32_t>(min(m0 + r, M - 1)) * K + kb + 8 * c) * 2 + (i & 1 ? 0 : kDmaBias);
  }
  // codes: the same row / chunk mapping over 128-byte code lines.  From nine
  // rows of weights on, a second request's row is at least row 8, and no base
  // has to be lowered: codes of up to 4 GiB, whose last rows have no room for
  // a larger offset.
  const uint32_t code_bias = N > 8 ? 0 : kDmaBias;
  uint32_t c_off[Gm::C_DMA];
#pragma unroll
  for (int i = 0; i < Gm::C_DMA; i++) {
    const int r = 8 * (wave * Gm::C_DMA + i) + (lane >> 3), c = (lane & 7) ^ swz(r);
    c_off[i] = static_cast<uint32_t>(min(n0 + r, N - 1)) * row_bytes + kb * BITS / 8 + 16 * c +
               (i & 1 ? code_bias - kDmaBias : code_bias);
  }
  // scales / biases: per row [scales SROW bytes][biases SROW bytes]; lanes
  // (row, array, 16-byte part)
  constexpr int SPR = 2 * Gm::SROW / 16;  // lanes per row
  uint32_t s_off[Gm::S_DMA];
#pragma unroll
  for (int i = 0; i < Gm::S_DMA; i++) {
    const int r = (wave * Gm::S_DMA + i) * (64 / SPR) + lane / SPR;
    const int part = lane % (Gm::SROW / 16);
    s_off[i] = (static_cast<uint32_t>(min(n0 + r, N - 1)) * G + kb / GS) * 2 + 16 * part;
  }
  const char* sb_base = reinterpret_cast<const char*>((lane % SPR) >= SPR / 2 ? biases : scales);

  // DMA of the activations of step kt / code batch c / scale batch sb into
  // stage / buffer `buf` (the index is clamped past the end, the buffer not)
  // pair i of this wave's share of a DMA (the offsets carry the bias)
  auto dma_a1 = [&](int kt, int buf, int i) __attribute__((always_inline)) {
    dma16x2_to_lds_sbase(reinterpret_cast<const char*>(x) + kt * (BK * 2) - kDmaBias, a_off[2 * i], a_off[2 * i + 1],
                         lds + Gm::A_OFF + buf * Gm::A_BYTES + (wave * Gm::A_DMA + 2 * i) * 1024);
  };
  auto dma_c1 = [&](int c, int buf, int i) __attribute__((always_inline)) {  // steps CB c .. CB c + CB - 1
    dma16x2_to_lds_sbase(reinterpret_cast<const char*>(wq) + c * 128 - code_bias, c_off[2 * i], c_off[2 * i + 1],
                         lds + Gm::C_OFF + buf * Gm::C_BYTES + (wave * Gm::C_DMA + 2 * i) * 1024);
  };
  auto dma_s1 = [&](int sb, int buf, int i) __attribute__((always_inline)) {  // steps 8 sb .. 8 sb + 7
    // groups from 8 * floor(first group / 8): 16 bytes of 8 groups (GS = 128:
    // the batch's 4 groups are one half of them)
    dma16_to_lds(sb_base + ((sb * PERIOD * BK / GS) & ~7) * 2 + s_off[i],
                 lds + Gm::S_OFF + buf * Gm::S_BYTES + (wave * Gm::S_DMA + i) * 1024);
  };
  auto dma_a = [&](int kt, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < Gm::A_DMA / 2; i++) dma_a1(kt, buf, i);
  };
  auto dma_c = [&](int c, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < Gm::C_DMA / 2; i++) dma_c1(c, buf, i);
  };
  auto dma_s = [&](int sb, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < Gm::S_DMA; i++) dma_s1(sb, buf, i);
  };

  // ---- fragment addressing (bytes within a stage / buffer)
  const int fr = lane & 31, h = lane >> 5;
  const int sw0 = (fr & 7) ^ (fr >> 3);  // swz(32 i + fr) = sw0 ^ 4 (i & 1)
  int a_rd[4][2];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int p = 0; p < 2; p++) a_rd[j][p] = (wm * TM * 32 + fr) * 128 + 16 * ((4 * h + j) ^ sw0 ^ (4 * p));
  // codes of step s (s % CB = u) for tile tt: logical chunks CW (u * 2 + h) + v
  int c_rd[CB][TN][Gm::CW];
#pragma unroll
  for (int u = 0; u < CB; u++)
#pragma unroll
    for (int tt = 0; tt < TN; tt++)
#pragma unroll
      for (int v = 0; v < Gm::CW; v++)
        c_rd[u][tt][v] = (wn * TN * 32 + tt * 32 + fr) * 128 +
                         16 * ((Gm::CW * (2 * u + h) + v) ^ swz(wn * TN * 32 + tt * 32 + fr));
  const int s_rd = (wn * TN * 32 + fr) * 2 * Gm::SROW;  // + tt * 32 rows

  bf16x8 bop[2][TN][4];  // decoded weight operands, double-buffered over steps
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int tt = 0; tt < TN; tt++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][tt][v] = 0.f;

  // codes and scale/bias bits of one step for this lane, read from LDS
  struct Raw {
    uint32_t w[TN][4 * Gm::CW];
    uint32_t s[TN], z[TN];
  };
  // step s = k0 + u (k0 % PERIOD == 0, u compile-time, may reach PERIOD + 1)
  auto read_raw = [&](int k0, auto uc, Raw& r) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    const unsigned char* cs = lds + Gm::C_OFF + ((u / CB) & 1) * Gm::C_BYTES;  // k0 / CB is even
    const int sbuf = ((k0 / PERIOD + u / PERIOD) & 1);
    const unsigned char* ss = lds + Gm::S_OFF + sbuf * Gm::S_BYTES + s_rd;
    // element of this step's group within the row's 16 / 32 bytes
    int e;
    if constexpr (GS == 32) e = 2 * (u % PERIOD) + h;
    else if constexpr (GS == 64) e = u % PERIOD;
    else e = 4 * ((k0 / PERIOD + u / PERIOD) & 1) + (u % PERIOD) / 2;
#pragma unroll
    for (int tt = 0; tt < TN; tt++) {
      r.s[tt] = *reinterpret_cast<const uint16_t*>(ss + tt * 32 * 2 * Gm::SROW + 2 * e);
      r.z[tt] = *reinterpret_cast<const uint16_t*>(ss + tt * 32 * 2 * Gm::SROW + Gm::SROW + 2 * e);
#pragma unroll
      for (int v = 0; v < Gm::CW; v++) {
        const u32x4 q = *reinterpret_cast<const u32x4*>(cs + c_rd[u % CB][tt][v]);
        r.w[tt][4 * v] = q[0];
        r.w[tt][4 * v + 1] = q[1];
        r.w[tt][4 * v + 2] = q[2];
        r.w[tt][4 * v + 3] = q[3];
      }
    }
  };
  auto read_a = [&](const unsigned char* as, int j, int i) __attribute__((always_inline)) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(as + i * 32 * 128 + a_rd[j][i & 1]));
  };
  // Decode piece p (0..31) of raw codes into `dst`: word w = p / 4 (tile
  // w / 4, sub-step w % 4), bf16 pair p % 4 of its operand.  A masked code in
  // the low bits of a half word is the subnormal half q * 2^-24 (times 16 for
  // a nibble in bits 4-7: still below 2^11 units, where halves are linear),
  // which v_fma_mix_f32 takes as it is: with the scale times 2^24 (2^20) the
  // product is the exact s * q, one instruction per code and one mask per
  // two (a scale of 2^104 and above overflows there: see the end of the loop).
  float sc[TN], zz[TN], sc16[TN];
  uint32_t h0 = 0, h1 = 0, h2 = 0, h3 = 0, d[4];
  auto half = [](uint32_t w, int i) __attribute__((always_inline)) {
    return static_cast<float>(__builtin_bit_cast(f16x2, w)[i]);
  };
  float f0 = 0.f, f1 = 0.f;
  auto piece_fma = [&](const Raw& r, auto pc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
    constexpr int w = p >> 2, tt = w >> 2, jj = w & 3, pp = p & 3;
    if constexpr (jj == 0 && pp == 0) {
      const float s0 = __uint_as_float(r.s[tt] << 16);
      zz[tt] = __uint_as_float(r.z[tt] << 16);
      sc[tt] = s0 * 0x1p24f;
      sc16[tt] = s0 * 0x1p20f;
    }
    if constexpr (BITS == 4) {
      // halves (q0, q4), (q1, q5), (q2, q6), (q3, q7)
      if constexpr (pp == 0) {
        h0 = r.w[tt][jj] & 0x000F000Fu;
        h1 = r.w[tt][jj] & 0x00F000F0u;
      }
      if constexpr (pp == 1) {
        h2 = (r.w[tt][jj] >> 8) & 0x000F000Fu;
        h3 = (r.w[tt][jj] >> 8) & 0x00F000F0u;
      }
      f0 = __builtin_fmaf(half(pp & 1 ? h2 : h0, pp >> 1), sc[tt], zz[tt]);
      f1 = __builtin_fmaf(half(pp & 1 ? h3 : h1, pp >> 1), sc16[tt], zz[tt]);
    } else {
      // word v = pp / 2: halves (q0, q2), (q1, q3)
      if constexpr ((pp & 1) == 0) {
        h0 = r.w[tt][2 * jj + (pp >> 1)] & 0x00FF00FFu;
        h1 = (r.w[tt][2 * jj + (pp >> 1)] >> 8) & 0x00FF00FFu;
      }
      f0 = __builtin_fmaf(half(h0, pp & 1), sc[tt], zz[tt]);
      f1 = __builtin_fmaf(half(h1, pp & 1), sc[tt], zz[tt]);
    }
  };
  // The pair of piece p packed and, with the fourth, the operand assembled:
  // issued one piece later (a convert right after the mixed FMA it reads costs
  // a wait state).
  auto piece_pack = [&](float g0, float g1, auto pc, bf16x8 (&dst)[TN][4]) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
    constexpr int w = p >> 2, tt = w >> 2, jj = w & 3, pp = p & 3;
    d[pp] = pack_bf16(g0, g1);
    if constexpr (pp == 3) dst[tt][jj] = __builtin_bit_cast(bf16x8, u32x4{d[0], d[1], d[2], d[3]});
  };

  // One K step (kt = k0 + u) as a fixed instruction schedule: slot s issues
  // MFMA s (sub-step j = s / (TM TN), row tile i, column tile tt); the LDS
  // reads of the next sub-step's activation fragments (for j = 3: the next
  // step's first), with two register sets in the first TM slots of a sub-step
  // (one wait per sub-step), with one after the last MFMA of each row tile
  // (two waits); then decode pieces of the next step's operands.  Each slot is fenced, so the wave alternates between the
  // matrix core and the vector ALU.  What bounds it is the issue rate of one
  // wave per SIMD, about five cycles an instruction of any kind, so the loop
  // is kept short: 7.2 instructions per MFMA at TM = 4 (9.2 with one wait per
  // fragment, one M0 write per request and a convert per code).
  // Once every activation read of the step has been issued, sits the step
  // boundary: wait for this wave's DMA of the next
  // step's activations, barrier, issue the DMA that the schedule places here,
  // read the codes of the step after next.  With 256-row tiles the decode
  // pieces all come before the boundary, so one set of raw-code registers
  // serves (the boundary refills it); with 128-row tiles they spread over the
  // whole step and the raw codes are double-buffered.
  constexpr int S = 4 * TM * TN, NP = 4 * 4 * TN, BOUNDARY = Gm::BOUNDARY;
  constexpr bool ONE_RAW = NP <= BOUNDARY;
  constexpr int PIECE_SLOTS = ONE_RAW ? BOUNDARY : S;
  constexpr int NRAW = ONE_RAW ? 1 : 2;
  constexpr int ASETS = Gm::ASETS, AST = Gm::AST;
  const int KTL = KT - 1;
  auto step = [&](int k0, auto uc, const bf16x8 (&cur)[TN][4], bf16x8 (&nxt)[TN][4], const Raw& rcur, Raw& rnext,
                  bf16x8 (&a)[Gm::ASETS][TM]) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    const int kt = k0 + u;
    const unsigned char* as = lds + Gm::A_OFF + u % AST * Gm::A_BYTES;
    const unsigned char* an = lds + Gm::A_OFF + (u + 1) % AST * Gm::A_BYTES;
    static_for<S>([&](auto sc_) __attribute__((always_inline)) {
      constexpr int s = decltype(sc_)::value;
      constexpr int j = s / (TM * TN), r = s % (TM * TN), i = r / TN, tt = r % TN;
      if constexpr (s == BOUNDARY) {
        wait_lgkm0();  // this wave's reads of step kt's stage are done
        // activations of step kt + 1 and the codes and scales of step kt + 2
        wait_vm<Gm::in_flight(u)>();
        __builtin_amdgcn_s_barrier();
        read_raw(k0, std::integral_constant<int, u + 2>{}, rnext);
        __builtin_amdgcn_sched_barrier(0);
      }
      constexpr int TH = TM / 2 * TN;
      if constexpr (ASETS == 2 ? r == 0 && j < 3 : r % TH == 0 && s < BOUNDARY) {
        // this (half) sub-step's fragments; after the boundary, its wait covers them
        if constexpr (ASETS == 2) wait_lgkm0();
        else wait_lgkm<TM / 2>();
        __builtin_amdgcn_sched_barrier(0);
      }
      constexpr int set = ASETS == 2 ? j & 1 : 0, other = ASETS == 2 ? (j + 1) & 1 : 0;
      // weights as the first operand: the output tile comes out transposed,
      // lane = activation row, 4 consecutive output columns per register quad
      acc[i][tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[tt][j], a[set][i], acc[i][tt], 0, 0, 0);
      if constexpr (ASETS == 2 ? r < TM : tt == TN - 1) {
        constexpr int ri = ASETS == 2 ? r : i;
        a[other][ri] = read_a(j < 3 ? as : an, (j + 1) & 3, ri);
      }
      // DMA: after the boundary the activations of step kt + AST into the
      // stage of step kt (read by every wave before the barrier); in the
      // first slots what step kt - 1 left to do (see QmmGeom): a pair every
      // other slot, then the scales.  Past the end: the last step / batch
      // again, into buffers nobody reads.
      constexpr int up = (u + PERIOD - 1) % PERIOD, CP = Gm::c_hi(up) - Gm::c_lo(up);
      if constexpr (s > BOUNDARY && s <= BOUNDARY + Gm::A_DMA / 2)
        dma_a1(min(kt + AST, KTL), u % AST, s - BOUNDARY - 1);
      if constexpr (s % 2 == 1 && s / 2 < CP)
        dma_c1(min((kt - 1 + Gm::C_AHEAD) / CB, KTL / CB), (u + PERIOD - 1 + Gm::C_AHEAD) / CB & 1, Gm::c_lo(up) + s / 2);
      if constexpr (s >= 2 * CP && s < 2 * CP + Gm::s_num(up))
        dma_s1(min((kt - 1) / PERIOD + 2, KTL / PERIOD), (k0 / PERIOD) & 1, s - 2 * CP);
      // pieces p with p * PIECE_SLOTS / NP == s
      constexpr int P_LO = (s * NP + PIECE_SLOTS - 1) / PIECE_SLOTS;
      constexpr int P_HI = ((s + 1) * NP + PIECE_SLOTS - 1) / PIECE_SLOTS;
      static_for<(NP + PIECE_SLOTS - 1) / PIECE_SLOTS>([&](auto qc) __attribute__((always_inline)) {
        constexpr int p = P_LO + decltype(qc)::value;
        if constexpr (p < P_HI && p < NP) {
          const float g0 = f0, g1 = f1;
          piece_fma(rcur, std::integral_constant<int, p>{});
          if constexpr (p > 0) piece_pack(g0, g1, std::integral_constant<int, p - 1>{}, nxt);
        }
      });
      // the last pair of the step
      if constexpr (s == (PIECE_SLOTS < S ? PIECE_SLOTS : S - 1))
        piece_pack(f0, f1, std::integral_constant<int, NP - 1>{}, nxt);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // ---- prologue: code batch 0, scale batch 0 and the activations of step 0,
  // whose operands are decoded here; then what the steps before it would have
  // requested, in their order (the counted waits of the loop hold from its
  // first boundary on).  Only the former are waited for: waiting for all of
  // them, up to 140 KB per workgroup, cost 0.1 to 0.4 us per launch (Q4 4096 x
  // 4096 M = 256 / 333 28.8 / 28.5 -> 28.3 / 28.1, Q8 5120 x 13824 M = 333 80.4 ->
  // 79.3).
  bf16x8 a[ASETS][TM];
  Raw raw[NRAW];
  constexpr int C1 = CB == 4 ? Gm::C_PAIRS / 2 : Gm::C_PAIRS;  // of code batch 1 what no step of the loop requests
  dma_c(0, 0);
  dma_s(0, 0);
#pragma unroll
  for (int v = 0; v < AST; v++) {
    dma_a(min(v, KTL), v);
    if (v == AST - 2) {
#pragma unroll
      for (int i = 0; i < C1; i++) dma_c1(min(1, KTL / CB), 1, i);
      dma_s(min(1, KTL / PERIOD), 1);
    }
  }
  wait_vm<(AST - 1) * Gm::A_DMA + 2 * C1 + Gm::S_DMA>();
  __builtin_amdgcn_s_barrier();
  read_raw(0, std::integral_constant<int, 0>{}, raw[0]);
#pragma unroll
  for (int i = 0; i < TM; i++) a[0][i] = read_a(lds + Gm::A_OFF, 0, i);
  static_for<NP>([&](auto pc) __attribute__((always_inline)) {
    piece_fma(raw[0], pc);
    piece_pack(f0, f1, pc, bop[0]);
  });
  read_raw(0, std::integral_constant<int, 1>{}, raw[NRAW - 1]);

  for (int k0 = 0; k0 < KT; k0 += PERIOD) {
    static_for<PERIOD / 2>([&](auto vc) __attribute__((always_inline)) {
      constexpr int u = 2 * decltype(vc)::value;
      step(k0, std::integral_constant<int, u>{}, bop[0], bop[1], raw[NRAW - 1], raw[0], a);
      step(k0, std::integral_constant<int, u + 1>{}, bop[1], bop[0], raw[0], raw[NRAW - 1], a);
    });
  }
  wait_vm<0>();  // no DMA may land after the workgroup's LDS is released

  // A finite scale of 2^104 and above became infinite in the decode's scaled
  // multiply, and its weights infinite or (code 0) NaN, and with them every
  // row of its column.  A wave with a sum in its first rows that is not finite
  // (16 fused multiply-adds cover the 32 of a lane; a large one that overflows
  // there costs the look at the scales) and such a scale forms its sums again
  // with the unscaled multiply, in the same order, from global memory (never
  // for weights of ordinary magnitude).  A maximum of the scales kept in the
  // loop, one instruction per step, took 0.2 us of the 48.2 of 333 rows x
  // 14336 x 4096 and 0.4 of the 54.4 of 4096 x 14336.
  float probe = 0.f;
#pragma unroll
  for (int tt = 0; tt < TN; tt++)
#pragma unroll
    for (int v = 0; v < 16; v += 2) probe = __builtin_fmaf(acc[0][tt][v], acc[0][tt][v + 1], probe);
  if (__builtin_expect(__any(!(fabsf(probe) < __builtin_inff())), 0)) {
    static_assert(TN == 2, "a column per lane, sc[0] and sc[1]");
    const uint16_t* sr = scales + static_cast<int64_t>(min(n0 + wn * 64 + lane, N - 1)) * G;
    bool large = false;
    for (int g = kb / GS; g < (kb + KT * BK) / GS; g++) {
      const uint32_t e = sr[g] & 0x7FFFu;
      large |= e >= 0x7380u && e < 0x7F80u;  // bf16 of 2^104; infinity
    }
    if (__any(large)) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int tt = 0; tt < TN; tt++)
#pragma unroll
          for (int v = 0; v < 16; v++) acc[i][tt][v] = 0.f;
#pragma unroll 1
      for (int kt = 0; kt < KT; kt++) {
        const int k = kb + kt * BK + 32 * h;  // this lane's 32 k of the step
        bf16x8 wv[TN][4];
#pragma unroll
        for (int tt = 0; tt < TN; tt++) {
          const int64_t n = min(n0 + (wn * TN + tt) * 32 + fr, N - 1);
          const float s0 = bf16_bits_to_f32(scales[n * G + k / GS]), z0 = bf16_bits_to_f32(biases[n * G + k / GS]);
          const u32x4* wr = reinterpret_cast<const u32x4*>(wq) + (n * K + k) * BITS / 128;
          uint32_t w[4 * Gm::CW];
#pragma unroll
          for (int v = 0; v < Gm::CW; v++) {
            const u32x4 q = wr[v];
#pragma unroll
            for (int e = 0; e < 4; e++) w[4 * v + e] = q[e];
          }
#pragma unroll
          for (int j = 0; j < 4; j++) {
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
              auto value = [&](int c) {  // code c of the lane's 32
                const uint32_t q = (w[c * BITS / 32] >> (c * BITS % 32)) & ((1u << BITS) - 1);
                return __builtin_fmaf(s0, static_cast<float>(q), z0);
              };
              o[e] = pack_bf16(value(8 * j + 2 * e), value(8 * j + 2 * e + 1));
            }
            wv[tt][j] = __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
          }
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int i = 0; i < TM; i++) {
            const int64_t m = min(m0 + (wm * TM + i) * 32 + fr, M - 1);
            const bf16x8 av = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(x + m * K + k + 8 * j));
#pragma unroll
            for (int tt = 0; tt < TN; tt++)
              acc[i][tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[tt][j], av, acc[i][tt], 0, 0, 0);
          }
      }
    }
  }

  // Output layout of a 32x32 tile (weights x activations^T): lane holds
  // activation row m = lane % 32 and output columns n = 8 (v / 4) + 4 (lane /
  // 32) + v % 4 for accumulator v.  Pairs of column groups are exchanged
  // between the wave halves (permlane32 swap) so that every lane ends with 8
  // consecutive columns: one 16-byte store (bf16) or two (f32 partials).
  const int mrow0 = m0 + wm * TM * 32 + fr;
  const int ncol0 = n0 + wn * TN * 32;
  if (part) {  // split K: this slice's f32 partial sums, added by the reduce kernel
    float* dst = part + static_cast<int64_t>(blockIdx.y) * M * N;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int m = mrow0 + i * 32;
      if (m >= M) continue;
#pragma unroll
      for (int tt = 0; tt < TN; tt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int n = ncol0 + tt * 32 + 8 * g + 4 * h;
          float* q = dst + static_cast<int64_t>(m) * N + n;
          if (n + 3 < N && (N & 3) == 0) {
            *reinterpret_cast<f32x4*>(q) = f32x4{acc[i][tt][4 * g], acc[i][tt][4 * g + 1], acc[i][tt][4 * g + 2],
                                                 acc[i][tt][4 * g + 3]};
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < N) q[e] = acc[i][tt][4 * g + e];
          }
        }
    }
  } else {
#pragma unroll
    for (int tt = 0; tt < TN; tt++) {
#pragma unroll
      for (int gp = 0; gp < 2; gp++) {
        // columns ncol0 + tt 32 + 16 gp + 8 h + [0, 8) after the exchange;
        // before it this lane holds groups 2 gp + q (q = 0, 1) at columns
        // ncol0 + tt 32 + 16 gp + 8 q + 4 h + [0, 4)
        const int n = ncol0 + tt * 32 + 16 * gp + 8 * h;
        float bb[2][4];
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const int nb = ncol0 + tt * 32 + 16 * gp + 8 * q + 4 * h + e;
            bb[q][e] = bias_vec && nb < N ? bf16_bits_to_f32(bias_vec[nb]) : 0.f;
          }
#pragma unroll
        for (int i = 0; i < TM; i++) {
          const f32x16& c = acc[i][tt];
          const uint32_t lo0 = pack_bf16(c[8 * gp + 0] + bb[0][0], c[8 * gp + 1] + bb[0][1]);
          const uint32_t lo1 = pack_bf16(c[8 * gp + 2] + bb[0][2], c[8 * gp + 3] + bb[0][3]);
          const uint32_t hi0 = pack_bf16(c[8 * gp + 4] + bb[1][0], c[8 * gp + 5] + bb[1][1]);
          const uint32_t hi1 = pack_bf16(c[8 * gp + 6] + bb[1][2], c[8 * gp + 7] + bb[1][3]);
          // lanes 0-31 keep group 2 gp and receive the other half's group
          // 2 gp; lanes 32-63 keep group 2 gp + 1 and receive the first
          // half's group 2 gp + 1
          const auto s0 = __builtin_amdgcn_permlane32_swap(lo0, hi0, false, false);
          const auto s1 = __builtin_amdgcn_permlane32_swap(lo1, hi1, false, false);
          const uint32_t w0 = s0[0], w1 = s1[0], w2 = s0[1], w3 = s1[1];
          const int m = mrow0 + i * 32;
          if (m >= M) continue;
          uint16_t* q = y + static_cast<int64_t>(m) * N + n;
          if (n + 7 < N && (N & 7) == 0) {
            *reinterpret_cast<u32x4*>(q) = u32x4{w0, w1, w2, w3};
          } else {
            const uint32_t ww[4] = {w0, w1, w2, w3};
#pragma unroll
            for (int e = 0; e < 8; e++)
              if (n + e < N) q[e] = static_cast<uint16_t>(ww[e >> 1] >> (16 * (e & 1)));
          }
        }
      }
    }
  }
}

// As many activation stages as fit; two for short slices (see launch_cfg).
template <int BITS, int GS, int TM, int TN>
__global__ __launch_bounds__(256, 1) void qmm_kernel(const uint16_t* __restrict__ x, int M,
                                                     const uint32_t* __restrict__ wq,
                                                     const uint16_t* __restrict__ scales,
                                                     const uint16_t* __restrict__ biases,
                                                     const uint16_t* __restrict__ bias_vec, int N, int K,
                                                     uint16_t* __restrict__ y, float* __restrict__ part, int grain,
                                                     int slice_grains, int longer) {
  qmm_tile<BITS, GS, TM, TN, TM <= 4 ? 4 : 2>(x, M, wq, scales, biases, bias_vec, N, K, y, part, grain, slice_grains,
                                              longer);
}
template <int BITS, int GS, int TM, int TN>
__global__ __launch_bounds__(256, 1) void qmm_short_kernel(const uint16_t* __restrict__ x, int M,
                                                           const uint32_t* __restrict__ wq,
                                                           const uint16_t* __restrict__ scales,
                                                           const uint16_t* __restrict__ biases,
                                                           const uint16_t* __restrict__ bias_vec, int N, int K,
                                                           uint16_t* __restrict__ y, float* __restrict__ part,
                                                           int grain, int slice_grains, int longer) {
  qmm_tile<BITS, GS, TM, TN, 2>(x, M, wq, scales, biases, bias_vec, N, K, y, part, grain, slice_grains, longer);
}

template <int BITS, int GS, int TM, int TN, bool SHORT = false>
int launch(const uint16_t* x, int M, const uint32_t* wq, const uint16_t* s, const uint16_t* b, const uint16_t* bias,
           int N, int K, uint16_t* y, float* part, int splits, hipStream_t st) {
  using Gm = QmmGeom<BITS, GS, TM, TN, (SHORT || TM > 4) ? 2 : 4>;
  auto kern = [] {
    if constexpr (SHORT) return &qmm_short_kernel<BITS, GS, TM, TN>;
    else return &qmm_kernel<BITS, GS, TM, TN>;
  }();
  static bool attr_set = false;  // once per process; the attribute is per function
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       Gm::LDS_BYTES);
    if (e != hipSuccess) return fail(MLXQ_ERR_DEVICE, std::string("qmm: set LDS size: ") + hipGetErrorString(e));
    attr_set = true;
  }
  const int64_t tiles = ceil_div(N, Gm::BN) * ceil_div(M, Gm::BM);
  constexpr int grain = GS > PERIOD * BK / 8 ? 8 * GS : PERIOD * BK;
  dim3 grid(static_cast<unsigned>(8 * ceil_div(tiles, 8)), splits);
  MLXQ_LAUNCH(kern, grid, dim3(Gm::THREADS), Gm::LDS_BYTES, st, x, M, wq, s, b, bias, N, K, y,
                     splits > 1 ? part : nullptr, grain, K / grain / splits, K / grain % splits);
  if (int rc = check_launch("qmm")) return rc;
  if (splits == 1) return MLXQ_OK;
  return launch_split_reduce(part, bias, y, M, N, splits, st);
}

int cu_count() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      return 256;
    return n;
  }();
  return cus;
}

// Workgroup tile of a launch: 256 rows (four waves of 256 x 64) when those
// tiles give at least one full round of workgroups, else 128 rows (four
// waves of 128 x 64: half the MFMAs per decoded code, twice the workgroups).
// MLXQ_QMM_CFG = 82 / 42 forces one (tests, tuning).  Measured and not kept
// (Llama-3-8B prefill, M = 2048): 2 x 2 waves of 128 x 128 (each column
// decoded twice), and two 128-row workgroups per CU.
int qmm_cfg(int64_t M, int64_t N, int splits) {
  if (const int c = overrides().qmm_cfg) return c == 42 ? 42 : 82;
  return ceil_div(N, 256) * ceil_div(M, 256) * splits >= cu_count() ? 82 : 42;
}

template <int BITS, int GS>
int launch_cfg(const uint16_t* x, int M, const uint32_t* wq, const uint16_t* s, const uint16_t* b, const uint16_t* bias,
               int N, int K, uint16_t* y, float* part, int splits, hipStream_t st) {
  if (qmm_cfg(M, N, splits) == 42) {
    // Q8 of group size 32 has the most bytes per step, and slices of up to 16
    // steps end before the deeper prefetch pays for what it requests past
    // their end: two activation stages (us with four / two; K steps per slice
    // in brackets): 300 x 1024 x 1024 (8) 17.6 / 16.7, 64 x 17408 x 1024 (16)
    // 19.6 / 19.4, 300 x 4096 x 4096 (16) 29.7 / 29.5, 300 x 4096 x 6144 (24)
    // 36.5 / 36.8, 333 x 4096 x 14336 (48) 67.3 / 70.0.
    if constexpr (BITS == 8 && GS == 32)
      if (ceil_div(K / (PERIOD * BK), splits) <= 2)
        return launch<BITS, GS, 4, 2, true>(x, M, wq, s, b, bias, N, K, y, part, splits, st);
    return launch<BITS, GS, 4, 2>(x, M, wq, s, b, bias, N, K, y, part, splits, st);
  }
  return launch<BITS, GS, 8, 2>(x, M, wq, s, b, bias, N, K, y, part, splits, st);
}

}  // namespace

bool qmm_eligible(int64_t K, int group_size) { return K % (PERIOD * BK) == 0 && K % (8 * group_size) == 0; }

int qmm_split_k(int64_t M, int64_t N, int64_t K, int group_size) {
  // split K when even 128-row tiles leave most CUs idle; every slice is a
  // whole number of grains (unrolled periods and 8-group scale batches), as
  // even as they divide: the fewest slices that make the longest one as short
  // as one round of workgroups allows.  Against slices of one length, us: K =
  // 5632 (11 grains, not split before) 2048 x 5632 M = 118 / 692 Q4 61.9 / 63.5
  // -> 23.1 / 32.6, Q8 72.1 / 70.7 -> 25.3 / 36.7; K = 13824 (27) 5120 x 13824 M
  // = 118 / 692 Q4 64.5 / 160 -> 39.6 / 114; K = 14336 (28) 4096 x 14336 M = 333
  // 61.7 -> 58.0 (five slices for four); K = 5120 (10) 5120 x 5120 M = 333 44.1
  // -> 36.9 (four for two).
  // MLXQ_QMM_SPLIT overrides (tests, tuning).
  const int64_t grains = K / std::max<int64_t>(PERIOD * BK, 8 * group_size);
  if (const int sp = overrides().qmm_split) return sp >= 1 && sp <= kQmmMaxSplits && sp <= grains ? sp : 1;
  const int64_t cus = cu_count();
  const int64_t t128 = ceil_div(N, 256) * ceil_div(M, 128);
  if (t128 * 4 >= cus * 3) return 1;
  const int64_t most = std::min(std::min<int64_t>(kQmmMaxSplits, grains), cus / t128);
  return most > 1 ? static_cast<int>(ceil_div(grains, ceil_div(grains, most))) : 1;
}

size_t qmm_workspace_bytes(int64_t M, int64_t N, int64_t K, int group_size) {
  const int sp = qmm_split_k(M, N, K, group_size);
  return sp > 1 ? static_cast<size_t>(sp) * M * N * sizeof(float) : 0;
}

int launch_qmm(const uint16_t* x, int64_t M, const uint32_t* wq, const uint16_t* s, const uint16_t* b,
               const uint16_t* bias, int64_t N, int64_t K, int group_size, int bits, uint16_t* y, void* workspace,
               size_t workspace_bytes, hipStream_t st) {
  // the DMA offsets are 32-bit byte offsets from the array bases
  if (M * K * 2 >= (int64_t(1) << 32) || N * K * bits / 8 >= (int64_t(1) << 32) || !qmm_eligible(K, group_size))
    return fail(MLXQ_ERR_UNSUPPORTED, "qmm: activations and codes must each be below 4 GiB, K a multiple of " +
                                          std::to_string(PERIOD * BK) + " and of 8 groups");
  const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
  // split K only when the caller's workspace holds the partials
  int splits = qmm_split_k(M, N, K, group_size);
  if (splits > 1 && (!workspace || workspace_bytes < static_cast<size_t>(splits) * M * N * sizeof(float) ||
                     (reinterpret_cast<uintptr_t>(workspace) & 255u)))
    splits = 1;
  float* part = static_cast<float*>(workspace);
  if (bits == 4) {
    if (group_size == 32) return launch_cfg<4, 32>(x, m, wq, s, b, bias, n, k, y, part, splits, st);
    if (group_size == 64) return launch_cfg<4, 64>(x, m, wq, s, b, bias, n, k, y, part, splits, st);
    return launch_cfg<4, 128>(x, m, wq, s, b, bias, n, k, y, part, splits, st);
  }
  if (group_size == 32) return launch_cfg<8, 32>(x, m, wq, s, b, bias, n, k, y, part, splits, st);
  if (group_size == 64) return launch_cfg<8, 64>(x, m, wq, s, b, bias, n, k, y, part, splits, st);
  return launch_cfg<8, 128>(x, m, wq, s, b, bias, n, k, y, part, splits, st);
}

}  // namespace mlxq
