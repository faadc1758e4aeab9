#pragma once

// Prefill GEMM Y[t][n] = sum_k W[n][k] x[t][k] over Q4_K r1 / Q6_K r1 weights with f16 activations
// and f32 accumulation, for MI355X (gfx950 / CDNA4): the attention's q / k / v / output
// projections of a prefill chunk (src/engine/weights.hip:306-330 gemm_input / gemm, called from
// src/engine/attention.hip:125-146). The interface is miso's kernels/qgemm.hpp -- QFormat,
// QGemmActParams, qgemm_act_op / qgemm_act_kernel, QGemmParams, qgemm_op<F>, qgemm_tiles and
// qgemm_kernel<F> keep their names, fields and launch contract (qgemm_act_kernel on
// ceil(n_tok k / 32 / 256) workgroups of 256 threads, qgemm_kernel<F> on qgemm_tiles(n, n_tok)
// workgroups of 256 threads). The design is this file's own.
//
// Activations: qgemm_act rounds x to f16 (xh) and sums each 32-element group of the rounded
// values (xs, f32, in the reference's order), 8 elements per thread, the four threads of a quad
// combining a group's sum with DPP.
//
// GEMM: a workgroup computes a 64-token x 64-row tile with v_mfma_f32_32x32x16_f16, each of its 4
// waves a 32 x 32 quarter (the lane's accumulator column is one weight row, so per-row scales are
// per-lane scalars). K advances in stages of 128. Per stage every thread fetches (two stages
// ahead, into registers) 64 bytes of the x tile and one 16-byte run of one row's quantized
// weights, and expands the weights into LDS as exact f16 integers:
//   Q4_K: q sc (<= 945) per weight through the 1024-exponent convert and one fused v_pk_fma_f16;
//         a block's partial C (16 MFMAs over its 256 k) is scaled by the row's d, and the block's
//         dmin m term is one more MFMA: A = the tokens' 8 sub-block sums of the block, each split
//         into f16 hi and lo parts (xs 2^-6 = hi + lo 2^-11), against B = m and m 2^-11.
//   Q6_K: c - 32 (low nibble set) and 16 (c - 32) (high set), exact; each 16-element scale group
//         is one MFMA whose result the lane scales by d sc (d sc / 16 for the high set).
// LDS tiles are double-buffered by stage (one barrier per stage) and their 16-byte chunks are
// XOR-swizzled by row, so the 32 rows an MFMA operand read touches spread over the banks.
// Workgroups are mapped to tiles in groups of 8 token tiles swept across the row tiles, each XCD
// a contiguous part of that order, so an XCD's activations and weights are read from the memory
// side about once and reused through its L2.
//
// The layer wiring and the C ABI run qgemm_wide_kernel instead (no reference counterpart): wide
// tiles fed by LDS DMA in four shapes, up to three products in one launch; qgemm_launch picks the
// shape. Results are bit-identical to qgemm_kernel's.

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>

#include "cdna4_wave.hpp"
#include "q6k_gemv.hpp"

namespace miso::kernels {

enum class QFormat { Q4K, Q6K };

struct QGemmActParams {
  const float* x;  // n_tok x k
  _Float16* xh;    // n_tok x k, x rounded to FP16
  float* xs;       // n_tok x k / 32, sums of the rounded values of each 32-group
  unsigned k, n_tok;
};

struct QGemmParams {
  const std::uint8_t* w;  // n_rows rows in the format's r1 layout
  const _Float16* xh;     // n_tok x k
  const float* xs;        // n_tok x k / 32 (Q4_K only)
  float* y;               // n_tok rows of stride ldy
  unsigned k, n_rows, n_tok, ldy;
};

// 8 consecutive elements of a thread, the four threads of a quad holding one 32-element group: f16
// into h, the group's sum of the rounded values returned. The sum is the reference's association
// (tests/test_qgemm.hip:92-104): the chunk sums ((h0 + h1) + h2) + h3 of the 8 four-element chunks
// added in order to 0; every lane gathers the quad's chunk sums by DPP broadcast.
__device__ __attribute__((always_inline)) inline float qgemm_act_group(const float (&x)[8],
                                                                      _Float16 (&h)[8]) {
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    h[j] = static_cast<_Float16>(x[j]);
    v[j] = static_cast<float>(h[j]);
  }
  const float c0 = ((v[0] + v[1]) + v[2]) + v[3];
  const float c1 = ((v[4] + v[5]) + v[6]) + v[7];
  // Chunk sums 2 l and 2 l + 1 come from quad lane l (DPP quad_perm broadcasts of lane l).
  using cdna4::as_float;
  using cdna4::as_uint;
  auto from = [](float y, auto ctrl) {
    return as_float(__builtin_amdgcn_update_dpp(0u, as_uint(y), decltype(ctrl)::value, 0xF, 0xF,
                                                true));
  };
  using L0 = std::integral_constant<int, 0x00>;
  using L1 = std::integral_constant<int, 0x55>;
  using L2 = std::integral_constant<int, 0xAA>;
  using L3 = std::integral_constant<int, 0xFF>;
  float sum = 0.0f + from(c0, L0{});
  sum += from(c1, L0{});
  sum += from(c0, L1{});
  sum += from(c1, L1{});
  sum += from(c0, L2{});
  sum += from(c1, L2{});
  sum += from(c0, L3{});
  sum += from(c1, L3{});
  return sum;
}

// Groups [first, first + count) of n_tok k / 32 (group g: elements 32 g .. 32 g + 31 of x, row
// major), grid-stride: thread i of the launch takes elements 8 (i % 4) .. + 7 of group
// first + i / 4. xs is bit-identical to the reference's (qgemm_act_group).
__device__ inline void qgemm_act_op(const QGemmActParams& p, unsigned first, unsigned count) {
  const unsigned stride = gridDim.x * blockDim.x;  // a multiple of 4: quads stay whole
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i / 4 < count; i += stride) {
    const std::size_t e = (std::size_t{first} + i / 4) * 32 + 8 * (i % 4);
    const float4 a = *reinterpret_cast<const float4*>(p.x + e);
    const float4 b = *reinterpret_cast<const float4*>(p.x + e + 4);
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    _Float16 h[8];
    const float sum = qgemm_act_group(x, h);
    *reinterpret_cast<uint4*>(p.xh + e) = __builtin_bit_cast(uint4, h);
    if (i % 4 == 0)
      p.xs[first + i / 4] = sum;
  }
}

// A template with a defaulted parameter: launches keep the reference's qgemm_act_kernel<<<...>>>
// form, and several translation units may include this header without clashing symbols.
template <int = 0>
__global__ void __launch_bounds__(256) qgemm_act_kernel(QGemmActParams p) {
  qgemm_act_op(p, 0, p.n_tok * (p.k / 32));
}

namespace qgemm_detail {

using cdna4::float16_t;
using cdna4::half2_t;
using cdna4::half8_t;
using q4k_gemv_detail::u32x4;

constexpr int kThreads = 256;
constexpr unsigned kBM = 64, kBN = 64, kBK = 128;  // tokens, rows, k per stage
constexpr unsigned kChunks = kBK / 8;              // 16-byte chunks per tile row

template <QFormat F>
constexpr unsigned row_bytes(unsigned k) {
  return F == QFormat::Q4K ? k / 256 * 144 : (k / 256 * 210 + 15) / 16 * 16;
}

// Half offset of chunk c of row r in a [rows][kBK] f16 tile (swizzled).
__device__ __attribute__((always_inline)) inline unsigned chunk_at(unsigned r, unsigned c) {
  return 8u * (kChunks * r + (c ^ (r & (kChunks - 1))));
}

struct alignas(16) Lds {
  _Float16 x[2][kBM * kBK];  // activations of the stage, by stage parity
  _Float16 w[2][kBN * kBK];  // expanded weights of the stage
  _Float16 xm[2][kBM][16];   // Q4_K, by block parity: sub-block sums as (hi, lo) pairs
  _Float16 wm[2][kBN][16];   // Q4_K: (m, m 2^-11) per sub-block
  float dd[2][kBN][4];       // Q4_K: d, dmin 2^6 (two unused slots: every quad lane writes one)
  float sc[2][kBN][8];       // Q6_K, by stage parity: d sc of the stage's 8 scale groups
};

// One thread's global data for a stage: x chunks 4q .. 4q + 3 of token tok, and 16 bytes of row
// tok's (as a weight row) quantized weights. q = thread % 4, tok = thread / 4. The loads have no
// control flow around them (a token or row past the end reads the last one, a stage past the end
// the last stage; store() zeroes what is out of range), so nothing waits for them before store()
// consumes them two stages later.
template <QFormat F>
struct Fetch;

template <>
struct Fetch<QFormat::Q4K> {
  u32x4 x[4];
  u32x4 head;  // block header
  u32x4 nib;   // nibble bytes 16 (q % 2) .. of group 2 (s % 2) + q / 2
  float2 xs;   // sums of sub-blocks 2q, 2q + 1 of the stage's block for token tok
};

template <>
struct Fetch<QFormat::Q6K> {
  u32x4 x[4];
  u32x4 ql;         // ql bytes 16 q .. 16 q + 15 of the stage's half-block
  u32x4 qh;         // qh bytes 16 (q % 2) ..
  unsigned short sc_lo, sc_hi;  // scale bytes 2 (q / 2), + 1 and 4 + 2 (q / 2), + 1 of the stage
  unsigned short d_bits;        // f16 d
};

template <QFormat F>
__device__ inline Fetch<F> fetch(const QGemmParams& p, unsigned n0, unsigned m0, unsigned s,
                                 unsigned t) {
  Fetch<F> f;
  const unsigned tok = t >> 2, q = t & 3u;
  const unsigned n_stages = p.k / kBK;
  s = s < n_stages ? s : n_stages - 1;
  const unsigned tk = m0 + tok < p.n_tok ? m0 + tok : p.n_tok - 1;
  const _Float16* xr = p.xh + std::size_t{tk} * p.k + kBK * s + 32 * q;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    f.x[i] = *reinterpret_cast<const u32x4*>(xr + 8 * i);
  const unsigned row = n0 + tok < p.n_rows ? n0 + tok : p.n_rows - 1;
  const std::uint8_t* wr = p.w + std::size_t{row} * row_bytes<F>(p.k);
  const unsigned b = s / 2, part = s % 2;
  if constexpr (F == QFormat::Q4K) {
    const std::uint8_t* blk = wr + 144 * b;
    f.head = *reinterpret_cast<const u32x4*>(blk);
    f.nib = *reinterpret_cast<const u32x4*>(blk + 16 + 64 * part + 16 * q);
    f.xs = *reinterpret_cast<const float2*>(p.xs + std::size_t{tk} * (p.k / 32) + 8 * b + 2 * q);
  } else {
    const unsigned nb = p.k / 256;
    f.ql = *reinterpret_cast<const u32x4*>(wr + 128 * b + 64 * part + 16 * q);
    f.qh = *reinterpret_cast<const u32x4*>(wr + nb * 128 + 64 * b + 32 * part + 16 * (q & 1u));
    const std::uint8_t* sc = wr + nb * 192 + 16 * b + 8 * part + 2 * (q / 2);
    f.sc_lo = *reinterpret_cast<const unsigned short*>(sc);
    f.sc_hi = *reinterpret_cast<const unsigned short*>(sc + 4);
    f.d_bits = *reinterpret_cast<const unsigned short*>(wr + nb * 208 + 2 * b);
  }
  return f;
}

__device__ __attribute__((always_inline)) inline void put(_Float16* tile, unsigned r, unsigned c,
                                                          u32x4 v) {
  *reinterpret_cast<u32x4*>(tile + chunk_at(r, c)) = v;
}

// (hi, lo) with v 2^-6 = hi + lo 2^-11 up to f16 rounding of lo; |v| < 2^21 keeps hi finite.
__device__ __attribute__((always_inline)) inline half2_t split(float v) {
  const float s = v * 0x1p-6f;
  const _Float16 hi = static_cast<_Float16>(s);
  return half2_t{hi, static_cast<_Float16>((s - static_cast<float>(hi)) * 0x1p11f)};
}

// Writes a fetched stage into the stage-parity buffers (and, for Q4_K, its block's min-term
// operands and scales into the block-parity ones; both stages of a block write the same values,
// which are read only after the block's second barrier). The thread's token and row go to tile
// row t / 4.
template <QFormat F>
__device__ inline void store(const Fetch<F>& f, Lds& sm, unsigned s, unsigned t, bool tok_ok,
                             bool row_ok) {
  using q4k_gemv_detail::spread_bytes;
  const unsigned tok = t >> 2, q = t & 3u, buf = s & 1u;
  const u32x4 zero{0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    put(sm.x[buf], tok, 4 * q + i, tok_ok ? f.x[i] : zero);
  if constexpr (F == QFormat::Q4K) {
    using q4k_gemv_detail::int_pair;
    using q4k_gemv_detail::splat;
    const unsigned w[4] = {f.nib.x, f.nib.y, f.nib.z, f.nib.w};
    const unsigned j = 2 * (s % 2) + q / 2, hb = q & 1u;
    const u32x4 head = row_ok ? f.head : zero;  // a row past the end: all scales zero
    const unsigned fld = q4k_gemv_detail::scale_field(head, j);
    const float sc_lo = static_cast<float>(fld & 63u), sc_hi = static_cast<float>((fld >> 12) & 63u);
    const half2_t s_lo = splat(sc_lo), c_lo = splat(-1024.0f * sc_lo);
    const half2_t s_hi = splat(sc_hi * 0.0625f), c_hi = splat(-64.0f * sc_hi);
    unsigned lo[8], hi[8];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const unsigned b = spread_bytes(w[d], i);
        lo[2 * d + i] = cdna4::as_uint(int_pair(b, 0x000F000Fu, s_lo, c_lo));
        hi[2 * d + i] = cdna4::as_uint(int_pair(b, 0x00F000F0u, s_hi, c_hi));
      }
    // Local k of the low set: 64 (q / 2) + 16 hb + i; of the high set 32 more.
    const unsigned c0 = 8 * (q / 2) + 2 * hb;
    put(sm.w[buf], tok, c0, u32x4{lo[0], lo[1], lo[2], lo[3]});
    put(sm.w[buf], tok, c0 + 1, u32x4{lo[4], lo[5], lo[6], lo[7]});
    put(sm.w[buf], tok, c0 + 4, u32x4{hi[0], hi[1], hi[2], hi[3]});
    put(sm.w[buf], tok, c0 + 5, u32x4{hi[4], hi[5], hi[6], hi[7]});
    {  // both stages of a block write the same block data (read after the block's second barrier)
      const unsigned bb = (s / 2) & 1u;
      const unsigned g = q4k_gemv_detail::scale_field(head, q);  // sub-blocks 2q, 2q + 1
      const float m0 = static_cast<float>((g >> 6) & 63u), m1 = static_cast<float>(g >> 18);
      const half2_t wm0{static_cast<_Float16>(m0), static_cast<_Float16>(m0 * 0x1p-11f)};
      const half2_t wm1{static_cast<_Float16>(m1), static_cast<_Float16>(m1 * 0x1p-11f)};
      *reinterpret_cast<uint2*>(&sm.wm[bb][tok][4 * q]) =
          uint2{cdna4::as_uint(wm0), cdna4::as_uint(wm1)};
      const float2 xs = tok_ok ? f.xs : float2{0.0f, 0.0f};
      *reinterpret_cast<uint2*>(&sm.xm[bb][tok][4 * q]) =
          uint2{cdna4::as_uint(split(xs.x)), cdna4::as_uint(split(xs.y))};
      const float dq = q == 0 ? q4k_gemv_detail::f16_bits(head.x & 0xFFFFu)
                              : q4k_gemv_detail::f16_bits(head.x >> 16) * 0x1p6f;
      sm.dd[bb][tok][q] = dq;  // slot 0: d, 1: dmin 2^6 (slots 2, 3 unused)
    }
  } else {
    using q6k_gemv_detail::code_pairs;
    const unsigned l[4] = {f.ql.x, f.ql.y, f.ql.z, f.ql.w};
    const unsigned h[4] = {f.qh.x, f.qh.y, f.qh.z, f.qh.w};
    unsigned lo[8], hi[8];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const q6k_gemv_detail::CodePairs c = code_pairs(l[d], h[d], i, 2 * (q / 2));
        lo[2 * d + i] = cdna4::as_uint(c.lo);
        hi[2 * d + i] = cdna4::as_uint(c.hi16);
      }
    // Elements 16 q + i (low set) and 64 + 16 q + i (high set) of the half-block.
    put(sm.w[buf], tok, 2 * q, u32x4{lo[0], lo[1], lo[2], lo[3]});
    put(sm.w[buf], tok, 2 * q + 1, u32x4{lo[4], lo[5], lo[6], lo[7]});
    put(sm.w[buf], tok, 8 + 2 * q, u32x4{hi[0], hi[1], hi[2], hi[3]});
    put(sm.w[buf], tok, 9 + 2 * q, u32x4{hi[4], hi[5], hi[6], hi[7]});
    const float d = row_ok ? q4k_gemv_detail::f16_bits(f.d_bits) : 0.0f;
    const unsigned at = 8 * (q & 1u);  // scale bytes q and 4 + q of the stage
    sm.sc[buf][tok][q] = d * static_cast<float>(static_cast<signed char>((f.sc_lo >> at) & 0xFFu));
    sm.sc[buf][tok][4 + q] =
        d * 0.0625f * static_cast<float>(static_cast<signed char>((f.sc_hi >> at) & 0xFFu));
  }
}

__device__ __attribute__((always_inline)) inline float16_t mfma(half8_t a, half8_t b,
                                                                float16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Tile index for workgroup b of a launch of `count` workgroups: workgroups are dealt round-robin
// to the 8 XCDs, so XCD x's workgroups b = x, x + 8, ... take the contiguous range
// [x q + min(x, r), ...) (q = count / 8, r = count % 8) of the tile order below.
__device__ __attribute__((always_inline)) inline unsigned xcd_tile(unsigned b, unsigned count) {
  const unsigned q = count / 8, r = count % 8, x = b % 8;
  return x * q + (x < r ? x : r) + b / 8;
}

// The tile order: groups of kGroupTok token tiles, and inside a group the row tiles in order, the
// group's token tiles fastest. The ~64 workgroups an XCD runs at once then cover 8 token tiles x 8
// row tiles, and a group's activations (8 x 64 tokens x k f16: 2 MiB at k = 2048) stay in that
// XCD's L2 while its row tiles pass -- each XCD reads its activations once and each weight row
// once per group, where a row tile swept across all token tiles would re-read the whole activation
// matrix from the memory side for every row tile.
constexpr unsigned kGroupTok = 8;
template <unsigned kGroup = kGroupTok>
__device__ __attribute__((always_inline)) inline void grouped_tile(unsigned t, unsigned n_ttiles,
                                                                  unsigned n_rtiles,
                                                                  unsigned& ttile,
                                                                  unsigned& rtile) {
  const unsigned per_group = kGroup * n_rtiles;
  const unsigned first_tok = t / per_group * kGroup, in = t % per_group;
  const unsigned width = n_ttiles - first_tok < kGroup ? n_ttiles - first_tok : kGroup;
  ttile = first_tok + in % width;
  rtile = in / width;
}

}  // namespace qgemm_detail

namespace qgemm_detail {

// One 64 x 64 output tile at tokens m0, rows n0. kStages: the stage count k / kBK when it is a
// compile-time constant (then the stage loop unrolls and the compiler's wait counts see the
// two-stage prefetch in straight-line code), 0 for any other k.
template <QFormat F, unsigned kStages>
__device__ __attribute__((always_inline)) inline void gemm_tile(const QGemmParams& p, Lds& sm,
                                                                unsigned m0, unsigned n0) {
  const unsigned t = threadIdx.x, lane = t % 64, wave = t / 64;
  const unsigned wt = wave >> 1, wr = wave & 1u;  // the wave's token half and row half
  const unsigned ar = 32 * wt + lane % 32, br = 32 * wr + lane % 32, kq = lane / 32;
  const unsigned n_stages = kStages ? kStages : p.k / kBK;
  float16_t acc = {}, c = {};
  // Two register sets, even and odd stages: stage s's data is requested two stages ahead.
  Fetch<F> fa = fetch<F>(p, n0, m0, 0, t);
  asm volatile("" : : : "memory");  // stage 0's loads are issued before stage 1's
  Fetch<F> fb = fetch<F>(p, n0, m0, 1, t);
  const bool tok_ok = m0 + t / 4 < p.n_tok, row_ok = n0 + t / 4 < p.n_rows;
  auto step = [&](Fetch<F>& f, unsigned s) __attribute__((always_inline)) {
    // Nothing crosses a stage boundary: the scheduler would otherwise hoist arithmetic on the
    // newest loads into the stage before, and the wait for them with it.
    __builtin_amdgcn_sched_barrier(0);
    store<F>(f, sm, s, t, tok_ok, row_ok);
    f = fetch<F>(p, n0, m0, s + 2, t);  // past the last stage: re-reads it, never stored
    __syncthreads();
    const unsigned buf = s & 1u;
#pragma unroll
    for (unsigned kk = 0; kk < kBK / 16; ++kk) {
      const half8_t a = *reinterpret_cast<const half8_t*>(sm.x[buf] + chunk_at(ar, 2 * kk + kq));
      const half8_t b = *reinterpret_cast<const half8_t*>(sm.w[buf] + chunk_at(br, 2 * kk + kq));
      if constexpr (F == QFormat::Q4K) {
        c = mfma(a, b, c);
      } else {
        const float16_t g = mfma(a, b, float16_t{});
        const float scale = sm.sc[buf][br][kk];
#pragma unroll
        for (int r = 0; r < 16; ++r)
          acc[r] = __builtin_fmaf(scale, g[r], acc[r]);
      }
    }
    if constexpr (F == QFormat::Q4K) {
      if (s % 2 == 1) {  // the block's last stage: its dmin m term, then its d scale
        const unsigned bb = (s / 2) & 1u;
        const half8_t am = *reinterpret_cast<const half8_t*>(&sm.xm[bb][ar][8 * kq]);
        const half8_t bm = *reinterpret_cast<const half8_t*>(&sm.wm[bb][br][8 * kq]);
        const float16_t mins = mfma(am, bm, float16_t{});
        const float d = sm.dd[bb][br][0], dmin = sm.dd[bb][br][1];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          acc[r] = __builtin_fmaf(d, c[r], acc[r]);
          acc[r] = __builtin_fmaf(-dmin, mins[r], acc[r]);
        }
        c = float16_t{};
      }
    }
  };
  for (unsigned s = 0; s < n_stages; s += 2) {  // n_stages is even (k % 256 == 0)
    step(fa, s);
    step(fb, s + 1);
  }
  // Lane (row br, half kq) holds tokens 8 (r / 4) + 4 kq + r % 4 of the wave's 32.
  const unsigned n = n0 + br;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const unsigned tok = m0 + 32 * wt + 8 * (r / 4) + 4 * kq + r % 4;
    if (tok < p.n_tok && n < p.n_rows)
      p.y[std::size_t{tok} * p.ldy + n] = acc[r];
  }
}

// ---- Wide tiles (no reference counterpart) ----
// A workgroup of WM x WN waves computes kTok tokens x kRow rows, each wave a (kTok / WM) x
// (kRow / WN) part of it in 32 x 32 MFMA blocks. K advances in stages of 64 (Q4_K: a nibble group
// of a block; Q6_K: one of the two 64-element sets of a block half).
//
// What bounds it: per stage, a wave's LDS operand reads, its share of expanding the weights, its
// MFMAs and one barrier. Activations (and Q4_K's nibbles, headers and activation sums) come in by
// LDS DMA, each instruction 1 KiB of whole row segments: fetched into registers row by row, as
// gemm_tile does, a wave's loads touch 64 separate segments each, which the address unit takes
// one per cycle -- that was the bound of the 128 x 128 tiles these replace. Two workgroups per CU
// (or two waves per SIMD in the 256 x 128 tile) let one's expansion and barrier run beside the
// other's MFMAs. Measured, Q4_K, before and after on one box: 8192 rows x 2048, 4096 tokens 354 ->
// 196 us (389 -> 702 TFLOP/s), 2048 x 4096, 4096 tokens 158 -> 85 us (435 -> 804); matrix units
// 40% busy, VALU 38%, LDS 32% (256 x 128): what is left is the lock step of one barrier per stage.
//
// Stage s: the MFMAs read activations and expanded weights of stage s while the same threads
// expand stage s + 1 into the other weight buffer. kRing 3 keeps two stages of activations in
// flight, with counted waits (the waves then have no other loads), kRing 4 three; kRing 2 one stage.
// Per output element the arithmetic is gemm_tile's in the same order: all tile shapes give
// bit-identical results.
//
// LDS tiles are rows of 64 f16 (128 bytes, 8 chunks); chunk c of row r is at position
// c ^ ((r / 2) % 8), so the 16 rows an operand read takes at once (two rows span the 64 banks) are
// 16 distinct chunk positions.
constexpr unsigned kWideK = 64;

template <unsigned kTok, unsigned kRow, unsigned kRing>
struct alignas(1024) LdsWide {
  _Float16 x[kRing][kTok * kWideK];
  _Float16 w[2][kRow * kWideK];
  std::uint8_t nib[kRing][kRow][32];  // Q4_K nibbles of a stage
  std::uint8_t head[2][kRow][16];     // Q4_K block headers; Q6_K by stage parity, 4 f32 scales
  float xs[kTok][8];                  // Q4_K activation sums of a block
};

template <QFormat F, unsigned kTok, unsigned kRow, unsigned WM, unsigned WN, unsigned kRing>
__device__ __attribute__((always_inline)) inline void gemm_tile_wide(
    const QGemmParams& p, LdsWide<kTok, kRow, kRing>& sm, unsigned m0, unsigned n0) {
  constexpr bool kQ4 = F == QFormat::Q4K;
  constexpr unsigned kWaves = WM * WN, MB = kTok / 32 / WM, NB = kRow / 32 / WN;
  constexpr unsigned kXInstr = kTok / 8 / kWaves;  // activation DMAs per wave and stage
  static_assert(kRow * 4 == 64 * kWaves, "four threads expand a row's stage");
  static_assert(kTok / 32 <= kWaves && kXInstr >= 1 && MB >= 1 && NB >= 1);
  static_assert(kRing >= 2 && kRing <= 4);
  const unsigned t = threadIdx.x, lane = t % 64;
  const unsigned wave = __builtin_amdgcn_readfirstlane(t / 64);
  const unsigned wt = wave / WN, wr = wave % WN, col = lane % 32, kq = lane / 32;
  const unsigned n_stages = p.k / kWideK;
  const std::size_t row_b = row_bytes<F>(p.k);

  // This lane's sources (rows and tokens past the end read the last one; their results are not
  // stored). Activations: instruction i of the wave moves tile rows 8 (kXInstr wave + i) .. + 7,
  // lane l chunk (l % 8) ^ ((row / 2) % 8) of row l / 8.
  const _Float16* xsrc[kXInstr];
#pragma unroll
  for (unsigned i = 0; i < kXInstr; ++i) {
    const unsigned r = 8 * (kXInstr * wave + i) + lane / 8;
    const unsigned tok = m0 + r < p.n_tok ? m0 + r : p.n_tok - 1;
    xsrc[i] = p.xh + std::size_t{tok} * p.k + 8 * ((lane % 8) ^ ((r / 2) % 8));
  }
  auto w_row = [&](unsigned r) __attribute__((always_inline)) {
    const unsigned row = n0 + r < p.n_rows ? n0 + r : p.n_rows - 1;
    return p.w + row * row_b;
  };
  const unsigned x_lds = cdna4::lds_offset(sm.x);
  // Stages and blocks past the end re-read the last one into a buffer that nothing reads again.
  auto load_x = [&](unsigned s, unsigned slot) __attribute__((always_inline)) {
    const unsigned at = kWideK * (s < n_stages ? s : n_stages - 1);
#pragma unroll
    for (unsigned i = 0; i < kXInstr; ++i)
      cdna4::lds_load16(xsrc[i] + at,
                        x_lds + slot * (kTok * kWideK * 2) + 1024 * (kXInstr * wave + i));
  };
  auto barrier = []() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  // Q4_K: nibbles (32 rows an instruction), headers (64 rows) and activation sums (32 tokens) by
  // the first waves, one instruction each; with kRing 4 the headers and sums by the last ones, so that
  // the waves of the nibbles issue the same in every stage.
  constexpr unsigned kHead0 = kRing == 4 ? kWaves - kRow / 64 : 0;
  constexpr unsigned kXs0 = kRing == 4 ? kWaves - kTok / 32 : 0;
  static_assert(kRing != 4 || (kHead0 >= kRow / 32 && kXs0 >= kRow / 32));
  const bool nib_wave = wave < kRow / 32, head_wave = wave - kHead0 < kRow / 64;
  const bool xs_wave = wave - kXs0 < kTok / 32;
  const std::uint8_t* nsrc = w_row(32 * (wave % (kRow / 32)) + lane / 2) + 16 + 16 * (lane % 2);
  const std::uint8_t* hsrc = w_row(64 * (wave % (kRow / 64)) + lane);
  const float* ssrc = nullptr;
  if constexpr (kQ4) {
    const unsigned r = 32 * (wave % (kTok / 32)) + lane / 2;
    const unsigned tok = m0 + r < p.n_tok ? m0 + r : p.n_tok - 1;
    ssrc = p.xs + std::size_t{tok} * (p.k / 32) + 4 * (lane % 2);
  }
  const unsigned nib_lds = cdna4::lds_offset(sm.nib), head_lds = cdna4::lds_offset(sm.head);
  const unsigned xs_lds = cdna4::lds_offset(sm.xs);
  auto load_nib = [&](unsigned s, unsigned slot) __attribute__((always_inline)) {
    s = s < n_stages ? s : n_stages - 1;
    cdna4::lds_load16(nsrc + 144 * (s / 4) + 32 * (s % 4),
                      nib_lds + slot * (kRow * 32) + 1024 * wave);
  };
  auto load_head = [&](unsigned b) __attribute__((always_inline)) {
    const unsigned at = 4 * b < n_stages ? b : n_stages / 4 - 1;
    cdna4::lds_load16(hsrc + 144 * at, head_lds + (b & 1u) * (kRow * 16) + 1024 * (wave - kHead0));
  };
  auto load_xs = [&](unsigned b) __attribute__((always_inline)) {
    cdna4::lds_load16(ssrc + 8 * b, xs_lds + 1024 * (wave - kXs0));
  };
  // Stage s needs every DMA of stage s - kRing + 1 and before; outstanding may be those of the
  // kRing - 2 stages since: their activations' and `extra` more. With kRing 2 (and Q6_K) all have to be
  // in.
  auto wait = [&](unsigned extra) __attribute__((always_inline)) {
    constexpr unsigned kX = (kRing - 2) * kXInstr;
    if (kRing == 2 || !kQ4)
      cdna4::wait_vmcnt<0>();
    else if (extra == 0)
      cdna4::wait_vmcnt<kX>();
    else if (extra == 1)
      cdna4::wait_vmcnt<kX + 1>();
    else
      cdna4::wait_vmcnt<kX + 2>();
  };

  // Expansion of a stage into weight buffer s % 2 by thread (row er = t / 4, quarter eq = t % 4).
  const unsigned er = t / 4, eq = t % 4, eswz = (er / 2) % 8;
  auto put_w = [&](unsigned s, unsigned c, u32x4 v) __attribute__((always_inline)) {
    *reinterpret_cast<u32x4*>(sm.w[s & 1u] + kWideK * er + 8 * (c ^ eswz)) = v;
  };
  // Q4_K: bytes 8 eq .. 8 eq + 7 of the group's 32: weights 8 eq + i (low), 32 + 8 eq + i (high).
  auto expand_q4 = [&](unsigned s, unsigned slot) __attribute__((always_inline)) {
    using namespace q4k_gemv_detail;
    const uint2 raw = *reinterpret_cast<const uint2*>(&sm.nib[slot][er][8 * eq]);
    const u32x4 head = *reinterpret_cast<const u32x4*>(&sm.head[(s / 4) & 1u][er][0]);
    const unsigned fld = scale_field(head, s % 4);
    const float sc_lo = static_cast<float>(fld & 63u), sc_hi = static_cast<float>((fld >> 12) & 63u);
    const half2_t s_lo = splat(sc_lo), c_lo = splat(-1024.0f * sc_lo);
    const half2_t s_hi = splat(sc_hi * 0.0625f), c_hi = splat(-64.0f * sc_hi);
    unsigned lo[4], hi[4];
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const unsigned b = spread_bytes(d == 0 ? raw.x : raw.y, i);
        lo[2 * d + i] = cdna4::as_uint(int_pair(b, 0x000F000Fu, s_lo, c_lo));
        hi[2 * d + i] = cdna4::as_uint(int_pair(b, 0x00F000F0u, s_hi, c_hi));
      }
    put_w(s, eq, u32x4{lo[0], lo[1], lo[2], lo[3]});
    put_w(s, 4 + eq, u32x4{hi[0], hi[1], hi[2], hi[3]});
  };
  // Q6_K: elements 16 eq .. 16 eq + 15 of the set (stage 2 h': low nibbles, 2 h' + 1: high), one
  // scale group. A block half's bytes serve both of its stages; they are fetched into registers
  // one half ahead.
  struct Half {
    u32x4 ql, qh;
    unsigned sc[2], d;  // scale bytes of the two sets' groups, f16 d
  };
  const std::uint8_t* qrow = w_row(er);
  const unsigned nb = p.k / 256;
  auto fetch_half = [&](unsigned h) __attribute__((always_inline)) {
    h = h < 2 * nb ? h : 2 * nb - 1;
    Half f;
    f.ql = *reinterpret_cast<const u32x4*>(qrow + 64 * h + 16 * eq);
    f.qh = *reinterpret_cast<const u32x4*>(qrow + nb * 128 + 32 * h + 16 * (eq & 1u));
    const std::uint8_t* sc = qrow + nb * 192 + 8 * h + eq;
    f.sc[0] = sc[0];
    f.sc[1] = sc[4];
    f.d = *reinterpret_cast<const unsigned short*>(qrow + nb * 208 + 2 * (h / 2));
    return f;
  };
  auto expand_q6 = [&](unsigned s, const Half& f) __attribute__((always_inline)) {
    const unsigned l[4] = {f.ql.x, f.ql.y, f.ql.z, f.ql.w};
    const unsigned h[4] = {f.qh.x, f.qh.y, f.qh.z, f.qh.w};
    unsigned v[8];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const q6k_gemv_detail::CodePairs c =
            q6k_gemv_detail::code_pairs(l[d], h[d], i, 2 * (eq / 2));
        v[2 * d + i] = cdna4::as_uint((s & 1u) == 0 ? c.lo : c.hi16);
      }
    put_w(s, 2 * eq, u32x4{v[0], v[1], v[2], v[3]});
    put_w(s, 2 * eq + 1, u32x4{v[4], v[5], v[6], v[7]});
    const float d = q4k_gemv_detail::f16_bits(f.d) * ((s & 1u) == 0 ? 1.0f : 0.0625f);
    reinterpret_cast<float*>(sm.head[s & 1u][er])[eq] =
        d * static_cast<float>(static_cast<signed char>(f.sc[s & 1u]));
  };

  float16_t acc[MB][NB], c[MB][NB];
#pragma unroll
  for (unsigned i = 0; i < MB; ++i)
#pragma unroll
    for (unsigned j = 0; j < NB; ++j)
      acc[i][j] = c[i][j] = float16_t{};

  Half raw{}, ahead{};
  // In the order in which they are waited for: what expands stage 0, stage 0 itself, then what the
  // stages since would have issued.
  if constexpr (kQ4) {
    if (head_wave)
      load_head(0);
    if (nib_wave) {
      load_nib(0, 0);
      load_nib(1, 1);
    }
    for (unsigned s = 0; s + 1 < kRing; ++s) {
      load_x(s, s);
      if (s != 0 && nib_wave)
        load_nib(s + 1, s + 1);
    }
    if (nib_wave)
      cdna4::wait_vmcnt<(kRing - 1) * (kXInstr + 1)>();
    else
      cdna4::wait_vmcnt<(kRing - 1) * kXInstr>();
    barrier();
    expand_q4(0, 0);
  } else {
    raw = fetch_half(0);
    for (unsigned s = 0; s + 1 < kRing; ++s)
      load_x(s, s);
    cdna4::wait_vmcnt<0>();
    barrier();
    expand_q6(0, raw);
  }

  // Operand addresses: row 32 i + col of a tile, chunk 2 kk + kq.
  unsigned at[4];
#pragma unroll
  for (unsigned kk = 0; kk < 4; ++kk)
    at[kk] = kWideK * col + 8 * ((2 * kk + kq) ^ ((col / 2) % 8));
  unsigned cur = 0, nxt = 1, spare = kRing - 1;  // ring slots of stages s, s + 1, s + kRing - 1
  for (unsigned s4 = 0; s4 < n_stages; s4 += 4) {
#pragma unroll
    for (unsigned j = 0; j < 4; ++j) {
      const unsigned s = s4 + j;
      // What the last kRing - 2 stages (the prologue's among them) issued besides activations; with
      // kRing 4 not the headers and sums (once a block their waves wait for a little more).
      if constexpr (kRing == 4)
        wait(nib_wave ? 2u : 0u);
      else
        wait((nib_wave ? 1u : 0u) + (j == 1 && xs_wave ? 1u : 0u) + (j == 2 && head_wave ? 1u : 0u));
      barrier();  // stage s complete for every wave, and every wave done with stage s - 1
      load_x(s + kRing - 1, spare);
      if constexpr (kQ4) {
        if (nib_wave)
          load_nib(s + kRing, cur);  // slot of stage s, expanded in stage s - 1
        if (j == 0 && xs_wave)
          load_xs(s4 / 4);  // read at j == 3; the last block's were read before this barrier
        if (j == (kRing == 4 ? 0 : 1) && head_wave)
          load_head(s4 / 4 + 1);  // expanded from at j == 3
      } else if (j % 2 == 0) {
        ahead = fetch_half(s / 2 + 1);
      }
      const _Float16* xt = sm.x[0] + cur * (kTok * kWideK) + 32 * kWideK * MB * wt;
      const _Float16* wtile = sm.w[j & 1u] + 32 * kWideK * NB * wr;
      float4 scale[NB];
      if constexpr (!kQ4)
#pragma unroll
        for (unsigned n = 0; n < NB; ++n)
          scale[n] =
              *reinterpret_cast<const float4*>(sm.head[j & 1u][32 * (NB * wr + n) + col]);
#pragma unroll
      for (unsigned kk = 0; kk < 4; ++kk) {
        half8_t a[MB], b[NB];
#pragma unroll
        for (unsigned i = 0; i < MB; ++i)
          a[i] = *reinterpret_cast<const half8_t*>(xt + 32 * kWideK * i + at[kk]);
#pragma unroll
        for (unsigned i = 0; i < NB; ++i)
          b[i] = *reinterpret_cast<const half8_t*>(wtile + 32 * kWideK * i + at[kk]);
#pragma unroll
        for (unsigned i = 0; i < MB; ++i)
#pragma unroll
          for (unsigned n = 0; n < NB; ++n) {
            if constexpr (kQ4) {
              c[i][n] = mfma(a[i], b[n], c[i][n]);
            } else {  // one scale group per k-step
              const float16_t g = mfma(a[i], b[n], float16_t{});
              const float sc = kk == 0   ? scale[n].x
                               : kk == 1 ? scale[n].y
                               : kk == 2 ? scale[n].z
                                         : scale[n].w;
#pragma unroll
              for (int r = 0; r < 16; ++r)
                acc[i][n][r] = __builtin_fmaf(sc, g[r], acc[i][n][r]);
            }
          }
      }
      // Past the last stage: into the buffer that nothing reads again.
      if constexpr (kQ4) {
        expand_q4(s + 1, nxt);
      } else {
        if (j % 2 == 1)
          raw = ahead;
        expand_q6(s + 1, raw);
      }
      if (kQ4 && j == 3) {  // the block's dmin m term, then its d scale
#pragma unroll
        for (unsigned n = 0; n < NB; ++n) {
          const u32x4 head = *reinterpret_cast<const u32x4*>(
              &sm.head[(s4 / 4) & 1u][32 * (NB * wr + n) + col][0]);
          half8_t bm;
#pragma unroll
          for (unsigned g = 0; g < 2; ++g) {
            const unsigned f = q4k_gemv_detail::scale_field(head, 2 * kq + g);
            const float me = static_cast<float>((f >> 6) & 63u), mo = static_cast<float>(f >> 18);
            bm[4 * g] = static_cast<_Float16>(me);
            bm[4 * g + 1] = static_cast<_Float16>(me * 0x1p-11f);
            bm[4 * g + 2] = static_cast<_Float16>(mo);
            bm[4 * g + 3] = static_cast<_Float16>(mo * 0x1p-11f);
          }
          const float d = q4k_gemv_detail::f16_bits(head.x & 0xFFFFu);
          const float dmin = q4k_gemv_detail::f16_bits(head.x >> 16) * 0x1p6f;
#pragma unroll
          for (unsigned i = 0; i < MB; ++i) {
            const float4 v =
                *reinterpret_cast<const float4*>(&sm.xs[32 * (MB * wt + i) + col][4 * kq]);
            const half2_t h[4] = {split(v.x), split(v.y), split(v.z), split(v.w)};
            const half8_t am = {h[0][0], h[0][1], h[1][0], h[1][1],
                                h[2][0], h[2][1], h[3][0], h[3][1]};
            const float16_t mins = mfma(am, bm, float16_t{});
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              acc[i][n][r] = __builtin_fmaf(d, c[i][n][r], acc[i][n][r]);
              acc[i][n][r] = __builtin_fmaf(-dmin, mins[r], acc[i][n][r]);
            }
            c[i][n] = float16_t{};
          }
        }
      }
      if constexpr (kRing == 4) {  // stage s is in slot s % 4
        cur = (j + 1) % 4, nxt = (j + 2) % 4, spare = j;
      } else {
        const unsigned tmp = cur;
        cur = nxt;
        nxt = kRing == 2 ? tmp : spare;
        spare = kRing == 2 ? nxt : tmp;
      }
    }
  }
  // Lane (row col of block n, half kq) holds tokens 8 (r / 4) + 4 kq + r % 4 of token block i.
#pragma unroll
  for (unsigned n = 0; n < NB; ++n) {
    const unsigned row = n0 + 32 * (NB * wr + n) + col;
#pragma unroll
    for (unsigned i = 0; i < MB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const unsigned tok = m0 + 32 * (MB * wt + i) + 8 * (r / 4) + 4 * kq + r % 4;
        if (tok < p.n_tok && row < p.n_rows)
          p.y[std::size_t{tok} * p.ldy + row] = acc[i][n][r];
      }
  }
  cdna4::wait_vmcnt<0>();  // every DMA has landed before the workgroup's LDS is given away
}

// The 64 x 64 tiles [first, first + count), in grouped_tile's order.
template <QFormat F>
__device__ inline void gemm_small(const QGemmParams& p, unsigned first, unsigned count, Lds& sm) {
  const unsigned n_ttiles = (p.n_tok + kBM - 1) / kBM, n_rtiles = (p.n_rows + kBN - 1) / kBN;
  for (unsigned i = blockIdx.x; i < count; i += gridDim.x) {
    const unsigned tile = first + (gridDim.x == count ? xcd_tile(i, count) : i);
    unsigned ttile, rtile;
    grouped_tile(tile, n_ttiles, n_rtiles, ttile, rtile);
    gemm_tile<F, 0>(p, sm, ttile * kBM, rtile * kBN);
    __syncthreads();  // the next tile's first stores reuse buffer 0
  }
}

}  // namespace qgemm_detail

// Output tiles [first, first + count) of 64 tokens x 64 rows, in grouped_tile's order.
template <QFormat F>
__device__ void qgemm_op(const QGemmParams& p, unsigned first, unsigned count) {
  __shared__ qgemm_detail::Lds sm;
  qgemm_detail::gemm_small<F>(p, first, count, sm);
}

__host__ __device__ inline unsigned qgemm_tiles(unsigned n_rows, unsigned n_tok) {
  using namespace qgemm_detail;
  return (n_rows + kBN - 1) / kBN * ((n_tok + kBM - 1) / kBM);
}

template <QFormat F>
__global__ void __launch_bounds__(qgemm_detail::kThreads) qgemm_kernel(QGemmParams p) {
  qgemm_op<F>(p, 0, qgemm_tiles(p.n_rows, p.n_tok));
}

// Up to three products over one prepared chunk (the q, k and v projections) in one launch: the
// same xh, xs, k and n_tok, each its own weights, format, rows and output.
struct QGemmBatch {
  QGemmParams m[3];
  QFormat format[3];
  unsigned count;
};

// One workgroup per kTok x kRow tile of every product. The row tiles of products 1 and 2 are
// spread evenly among product 0's, so every XCD (a contiguous part of the tile order, see xcd_tile)
// gets its share of each format.
template <unsigned kTok, unsigned kRow, unsigned WM, unsigned WN, unsigned kRing,
          unsigned kWavesPerSimd, unsigned kGroup>
__global__ void __launch_bounds__(64 * WM * WN, kWavesPerSimd) qgemm_wide_kernel(QGemmBatch p) {
  using namespace qgemm_detail;
  __shared__ LdsWide<kTok, kRow, kRing> sm;
  const unsigned n_tok = p.m[0].n_tok;
  unsigned rt[3], all = 0;
#pragma unroll
  for (unsigned i = 0; i < 3; ++i) {
    rt[i] = i < p.count ? (p.m[i].n_rows + kRow - 1) / kRow : 0;
    all += rt[i];
  }
  const unsigned n_ttiles = (n_tok + kTok - 1) / kTok;
  unsigned ttile, r;
  grouped_tile<kGroup>(xcd_tile(blockIdx.x, n_ttiles * all), n_ttiles, all, ttile, r);
  unsigned which = 0;
#pragma unroll
  for (unsigned i = 2; i > 0; --i) {  // is place r of `all` one of product i's rt[i]?
    if (which == 0 && rt[i] != 0) {
      const unsigned before = r * rt[i] / all;
      if ((r + 1) * rt[i] / all > before)
        which = i, r = before;
      else
        r -= before, all -= rt[i];
    }
  }
  const QGemmParams q = which == 0 ? p.m[0] : which == 1 ? p.m[1] : p.m[2];
  const QFormat f = which == 0 ? p.format[0] : which == 1 ? p.format[1] : p.format[2];
  if (f == QFormat::Q4K)
    gemm_tile_wide<QFormat::Q4K, kTok, kRow, WM, WN, kRing>(q, sm, ttile * kTok, r * kRow);
  else
    gemm_tile_wide<QFormat::Q6K, kTok, kRow, WM, WN, kRing>(q, sm, ttile * kTok, r * kRow);
}

// The tile shape with the least estimated time: a CU's tiles, in rounds of as many workgroups as
// fit on it together. Times of a round by workgroups per CU, in us per 2048 of k (one MI355X,
// Q4_K, HBM-resident weights):
//   64 x 64     13, 18, 24 (three together)     128 x 64    17, 28
//   128 x 128   24, 50                          256 x 128   48 (one fills the CU)
// so small launches take small tiles (more CUs, shorter stages) and full chips large ones (fewer
// LDS bytes and expansions per MFMA): 512 tokens x 8192 rows 38 / 34 / 33 / 40 us in this order,
// 200 tokens 22 / 20 / 27 / 37, 4096 tokens 263 / 229 / 199 / 196.
// kGroup (token tiles swept across the row tiles) keeps the ~32 to 96 tiles an XCD runs at once
// within its 4 MiB of L2 also at k = 4096: 2048 rows x 4096, 512 tokens in 64 x 64 tiles 36 us
// in groups of 8, 31 in groups of 4.
// 64 x 64 tiles, one workgroup per CU: nothing hides a stage's wait, and weights come from memory
// (a model's layers do not stay in the L2s), so Q4_K takes four stages in the ring. Weights of 80
// matrices in turn, with two stages and four: 2048 rows x 4096, 13 tokens 30.8 / 26.4 us, 512
// tokens 34.8 / 27.3; 8192 rows x 2048, 64 tokens 19.6 / 15.8; a whole layer over 512 tokens 125 /
// 118. Q6_K waits for its weights' registers at every other stage, and stays with two: 512 rows x
// 2048 19.5 / 20.9.
struct QGemmShape {
  unsigned index;  // 0 .. 3: 64 x 64, 128 x 64, 128 x 128, 256 x 128
  unsigned tiles;  // the launch's workgroups
  bool deep;       // four stages in the ring (64 x 64)
};
inline QGemmShape qgemm_shape(const QGemmBatch& p) {
  auto tiles = [&](unsigned tok, unsigned row) {
    unsigned rows = 0;
    for (unsigned i = 0; i < p.count; ++i)
      rows += (p.m[i].n_rows + row - 1) / row;
    return rows * ((p.m[0].n_tok + tok - 1) / tok);
  };
  constexpr unsigned kShapes = 4;
  const unsigned count[kShapes] = {tiles(64, 64), tiles(128, 64), tiles(128, 128),
                                   tiles(256, 128)};
  constexpr unsigned kTogether[kShapes] = {3, 2, 2, 1};
  constexpr unsigned kRound[kShapes][4] = {{0, 13, 18, 24}, {0, 17, 28}, {0, 24, 50}, {0, 48}};
  unsigned best = 0;
  std::uint64_t least = ~std::uint64_t{0};
  for (unsigned i = 0; i < kShapes; ++i) {
    const unsigned per_cu = (count[i] + 255) / 256, full = per_cu / kTogether[i];
    const std::uint64_t t = std::uint64_t{full} * kRound[i][kTogether[i]] +
                            kRound[i][per_cu % kTogether[i]];
    if (t < least)
      best = i, least = t;
  }
  return {best, count[best], best == 0 && count[0] <= 256 && p.format[0] == QFormat::Q4K};
}

inline void qgemm_launch(const QGemmBatch& p, hipStream_t stream) {
  const QGemmShape s = qgemm_shape(p);
  switch (s.index) {
    case 0:
      if (s.deep)
        qgemm_wide_kernel<64, 64, 2, 2, 4, 2, 4><<<s.tiles, 256, 0, stream>>>(p);
      else
        qgemm_wide_kernel<64, 64, 2, 2, 2, 2, 4><<<s.tiles, 256, 0, stream>>>(p);
      break;
    case 1: qgemm_wide_kernel<128, 64, 2, 2, 2, 2, 2><<<s.tiles, 256, 0, stream>>>(p); break;
    case 2: qgemm_wide_kernel<128, 128, 2, 4, 2, 4, 2><<<s.tiles, 512, 0, stream>>>(p); break;
    default: qgemm_wide_kernel<256, 128, 4, 2, 3, 2, 4><<<s.tiles, 512, 0, stream>>>(p); break;
  }
}

}  // namespace miso::kernels
