// Quantised matmul for a few tokens (2 up to a medium prompt) on the matrix cores:
// OUT[t][r] = sum_e W[r][e] * X[t][e].
//
// A few tokens read every weight once and do little with it, so a call is bound by
// the latency of one pass (load, decode, multiply, combine) and, as rows and tokens
// add up, by the vector instructions that decode the weights. One launch does it all,
// with nothing prepared beforehand:
//   * a workgroup takes a K slice of up to 8 to 20 half blocks (by its shape) and walks
//     tiles of 16 weight rows; its waves split the slice, each keeping its half blocks
//     of all the tokens in registers, so the activations are read and split once per
//     workgroup and a weight is decoded once per 16 or 32 tokens;
//   * within a half block K runs in four steps of 32 columns, one Q4_K sub-block or
//     Q6_K quarter each: lane (r, kg) = (lane % 16, lane / 16) holds columns 32 s +
//     8 kg .. + 7 of token r (A of v_mfma_f32_16x16x32_f16) and of weight row r (B);
//   * the activations are split in registers: per (token, half block) a power of two
//     brings max |x| into [2^13, 2^14) and x becomes two fp16 terms hi + lo (~2^-22
//     |x|), whose products accumulate apart (the lo sums are small, so only the hi
//     sums round);
//   * Q4_K weights enter centred, sc_j (q - 8), an exact fp16 integer: the partial
//     sums are half of those of sc_j q, and so is their rounding. The rest, (8 d sc_j -
//     dmin m_j) times the sub-block's sum of x, comes from one double-precision
//     matrix product per half block and joins in double. (A column far larger than the
//     others whose quant is near 0 is the other way round: it rounds by 8 d sc_j of it.)
//   * Q6_K weights enter as w = sc (q - 32) in two exact fp16 terms (w rounded, and
//     the remainder, nonzero only for |w| > 2048); the matrix cores form x_hi w_hi,
//     x_lo w_hi and x_hi w_lo; x_lo w_lo is below 2^-22 |x w|.
// Relative error against 64 bits at 2048 columns: 1.0e-7 (Q4_K), 1.1e-7 (Q6_K), where the
// tiled kernel has 1.2e-7 and the prefill GEMM 3.2e-7 and 1.9e-7.
//
// Measured on MI355X (graph replay, weights rotated past the Infinity Cache), against
// the tiled kernel (below 16 or 32 tokens) and the prefill GEMM that ran these sizes:
// q / k / v of a 1.7B layer, 21 tokens 46.6 -> 9.4 us, 128 tokens 69.8 -> 19.0; gate / up
// with SwiGLU 43.6 -> 17.8 and 71.6 -> 36.7; ffn_down 40.8 -> 16.9 and 39.8 -> 28.5;
// the 151936-row output projection at 21 tokens 350 -> 104. What a tile of 16 rows costs
// now is mostly its ~130 vector instructions per wave and half block, of which the
// decode is 40; loading x in the matrix core's own layout (4 us more per call: one cache
// line per lane instead of one per four) and the weights one lane's bytes at a time
// (22 instead of 16 us for gate / up) were the largest costs taken out on the way.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "dev_util.h"
#include "kernels_gpu.h"
#include "launch.h"
#include "matmul_mfma.h"
#include "matmul_small.h"
#include "quant_dev.h"

namespace rpg {
namespace {

typedef _Float16 F16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 H2 __attribute__((ext_vector_type(2)));
typedef float F32x4 __attribute__((ext_vector_type(4)));
typedef double F64x4 __attribute__((ext_vector_type(4)));
typedef unsigned int U32x4 __attribute__((ext_vector_type(4)));

constexpr int kCUs = 256;
constexpr int kUnit = 128;  // columns of a half block, the unit of work along K
constexpr int kSteps = 4;   // its 32-column steps

__device__ __forceinline__ H2 Half2(uint32_t w) { return __builtin_bit_cast(H2, w); }
__device__ __forceinline__ H2 Both(float f) {
  const _Float16 h = static_cast<_Float16>(f);
  return H2{h, h};
}
__device__ __forceinline__ F16x8 Join(H2 a, H2 b, H2 c, H2 d) {
  F16x8 v;
  v[0] = a[0]; v[1] = a[1]; v[2] = b[0]; v[3] = b[1];
  v[4] = c[0]; v[5] = c[1]; v[6] = d[0]; v[7] = d[1];
  return v;
}
__device__ __forceinline__ float HalfF(uint32_t bits) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits)));
}

// fp16(x0 s), fp16(x1 s) packed, and the fp16 remainders x s - fp16(x s), each
// one mixed-precision FMA (exact product, one rounding).
__device__ __forceinline__ uint32_t ScaledPair(float x0, float x1, float s) {
  uint32_t d;
  asm("v_fma_mixlo_f16 %0, %1, %3, 0\n\t"
      "v_fma_mixhi_f16 %0, %2, %3, 0"
      : "=&v"(d)
      : "v"(x0), "v"(x1), "v"(s));
  return d;
}
__device__ __forceinline__ uint32_t RemainderPair(float x0, float x1, float s, uint32_t h) {
  uint32_t d;
  asm("v_fma_mixlo_f16 %0, %1, %3, -%4 op_sel_hi:[0,0,1]\n\t"
      "v_fma_mixhi_f16 %0, %2, %3, -%4 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
      : "=&v"(d)
      : "v"(x0), "v"(x1), "v"(s), "v"(h));
  return d;
}

// The power of two 2^e that brings m into [2^13, 2^14), e at most 120 (and 0 for a
// non-finite m), and its inverse.
__device__ __forceinline__ float FitScale(float m, float* inv) {
  const int xe = static_cast<int>((__float_as_uint(m) >> 23) & 0xFFu);
  const int e = xe == 255 ? 0 : (140 - xe < 120 ? 140 - xe : 120);
  *inv = __uint_as_float(static_cast<uint32_t>(127 - e) << 23);
  return __uint_as_float(static_cast<uint32_t>(127 + e) << 23);
}

// ---------------------------------------------------------------- activations

// A unit's columns of a 16-token tile as loaded: lane l holds columns 32 s + 8 (l
// % 4) .. + 7 of token l / 4, so four lanes read one cache line. (Loading the
// matrix core's layout directly, token l % 16, touches four lines per four
// lanes and took as long as the rest of the kernel.)
struct XRaw {
  float4 v[kSteps][2];
};

__device__ __forceinline__ void LoadX(XRaw& x, const float* __restrict__ p) {
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    x.v[s][0] = *reinterpret_cast<const float4*>(p + 32 * s);
    x.v[s][1] = *reinterpret_cast<const float4*>(p + 32 * s + 4);
  }
}

// The same through a buffer, at (the lane's) + base (the wave's) bytes: one register for
// the addresses instead of two.
__device__ __forceinline__ void LoadX(XRaw& x, __amdgpu_buffer_rsrc_t rows, uint32_t at, uint32_t base) {
#pragma unroll
  for (int s = 0; s < kSteps; ++s)
#pragma unroll
    for (int k = 0; k < 2; ++k)
      x.v[s][k] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rows, static_cast<int>(at), static_cast<int>(base + 128 * s + 16 * k), 0));
}

// The value of the lane whose index differs in bit 0 / bit 1.
__device__ __forceinline__ float Xor1(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float Xor2(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));
}

// The matrix core's operands: lane (r, kg) holds columns 32 s + 8 kg .. + 7 of token
// r as two fp16 terms hi and lo, elements in the order 0, 2, 1, 3, 4, 6, 5, 7 (that of
// the decoded weights); sum: over step kg's 32 columns, for the double-precision matrix
// product of the sub-blocks' offsets.
struct XSplit {
  F16x8 hi[kSteps], lo[kSteps];
  double sum;
};

// inv: the wave's LDS area for the tokens' inverse scales. Whether a value is infinite.
__device__ __forceinline__ bool SplitX(const XRaw& x, XSplit& o, float* inv, int lane, bool want_sums) {
  float mx = 0.0f;
#pragma unroll
  for (int s = 0; s < kSteps; ++s)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float4 f = x.v[s][k];
      mx = fmaxf(fmaxf(mx, fabsf(f.x)), fabsf(f.y));
      mx = fmaxf(fmaxf(mx, fabsf(f.z)), fabsf(f.w));
    }
  mx = fmaxf(mx, Xor1(mx));
  mx = fmaxf(mx, Xor2(mx));
  float is;
  const float sc = FitScale(mx, &is);
  if ((lane & 3) == 0) inv[lane >> 2] = is;
  // lane (r, kg) takes what lane 4 r + kg holds
  const int from = 4 * (4 * (lane & 15) + (lane >> 4));
  auto move = [&](uint32_t v) { return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from, static_cast<int>(v))); };
  float sum[kSteps];
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    const float4 a = x.v[s][0], b = x.v[s][1];
    if (want_sums) sum[s] = ((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w));
    const U32x4 h = {ScaledPair(a.x, a.z, sc), ScaledPair(a.y, a.w, sc), ScaledPair(b.x, b.z, sc), ScaledPair(b.y, b.w, sc)};
    const U32x4 l = {RemainderPair(a.x, a.z, sc, h.x), RemainderPair(a.y, a.w, sc, h.y),
                     RemainderPair(b.x, b.z, sc, h.z), RemainderPair(b.y, b.w, sc, h.w)};
    U32x4 hm, lm;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      hm[k] = move(h[k]);
      lm[k] = move(l[k]);
    }
    o.hi[s] = __builtin_bit_cast(F16x8, hm);
    o.lo[s] = __builtin_bit_cast(F16x8, lm);
  }
  const bool infinite = __builtin_amdgcn_ballot_w64(mx > FLT_MAX) != 0;
  if (!want_sums) return infinite;
  // sums over a token's four lanes, transposed on the way: after two exchanges lane
  // 4 r + k holds the sum of step k
  const bool up2 = (lane & 2) != 0, up1 = (lane & 1) != 0;
  float p[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) p[k] = (up2 ? sum[2 + k] : sum[k]) + Xor2(up2 ? sum[k] : sum[2 + k]);
  const float total = (up1 ? p[1] : p[0]) + Xor1(up1 ? p[0] : p[1]);
  // (its result's rows 4 i + kg belong to tokens 4 kg + i of the other products, hence
  // the token of lane r here)
  const int from_sum = 4 * (4 * (4 * (lane & 3) + ((lane >> 2) & 3)) + (lane >> 4));
  o.sum = __int_as_float(__builtin_amdgcn_ds_bpermute(from_sum, __float_as_int(total)));
  return infinite;
}

// ---------------------------------------------------------------- weights

// The bytes lane (r, kg) needs of half hb of a block of weight row r.
template <bool kQ6>
struct WRaw;
template <>
struct WRaw<false> {
  uint4 hdr;   // d | dmin | 12 scale bytes
  uint2 q[2];  // qs bytes 32 g + 8 kg .. + 7 of the sub-block pairs g = 2 hb, 2 hb + 1
};
template <>
struct WRaw<true> {
  uint3 ql[2], qh;  // 8-byte windows (the aligned dwords around them)
  uint3 sc;         // the window of the half's 8 scale bytes
  uint16_t d;
  uint32_t sh;      // the block's offset inside its aligned dword (0 or 2)
};

// Both read from LDS, where a tile's rows are copied as they lie in memory.
__device__ __forceinline__ void ReadW(WRaw<false>& o, const uint8_t* blk, int hb, int kg) {
  o.hdr = *reinterpret_cast<const uint4*>(blk);
#pragma unroll
  for (int g = 0; g < 2; ++g) o.q[g] = *reinterpret_cast<const uint2*>(blk + 16 + 64 * hb + 32 * g + 8 * kg);
}

// Q6_K blocks are 2-byte aligned: every window starts at the aligned dword at or
// before its field. sh: the block's offset inside its aligned dword (0 or 2).
__device__ __forceinline__ void ReadW(WRaw<true>& o, const uint8_t* blk, uint32_t sh, int hb, int kg) {
  o.sh = sh;
  const uint8_t* ab = blk - sh;
  auto window = [](const uint8_t* p) {
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
    return make_uint3(q[0], q[1], q[2]);
  };
  o.ql[0] = window(ab + 64 * hb + 8 * kg);
  o.ql[1] = window(ab + 64 * hb + 32 + 8 * kg);
  o.qh = window(ab + 128 + 32 * hb + 8 * kg);
  o.sc = window(ab + 192 + 8 * hb);
  o.d = *reinterpret_cast<const uint16_t*>(blk + 208);
}

__device__ __forceinline__ uint2 Window8(uint3 w, uint32_t sh) {
  return make_uint2(__builtin_amdgcn_alignbyte(w.y, w.x, sh), __builtin_amdgcn_alignbyte(w.z, w.y, sh));
}

__device__ __forceinline__ float ByteF(uint32_t w, int k) { return static_cast<float>((w >> (8 * k)) & 0xFFu); }

// (q - 8) sc 2^-14 for four quants of a dword (bytes 0, 2 and 1, 3), exact: the
// masked bits, read as fp16 subnormals, are q 2^-24 (low nibbles) or q 2^-20
// (high nibbles), so one FMA against sc 2^10 or sc 2^6 and -8 sc 2^-14 decodes a pair.
template <bool kHigh>
__device__ __forceinline__ void PairsQ4(uint32_t v, H2 mul, H2 off, H2* a, H2* b) {
  constexpr uint32_t kMask = kHigh ? 0x00F000F0u : 0x000F000Fu;
  *a = __builtin_elementwise_fma(Half2(v & kMask), mul, off);
  *b = __builtin_elementwise_fma(Half2((v >> 8) & kMask), mul, off);
}

// acc += a half block's products of one 16-row tile with every token tile.
template <int kNT>
__device__ __forceinline__ void TileQ4(const WRaw<false>& w, int hb, const XSplit (&x)[kNT], const F32x4 (&inv)[kNT],
                                       int kg, F32x4 (&acc)[kNT]) {
  const float d = HalfF(w.hdr.x & 0xFFFFu);
  const float dmin = HalfF(w.hdr.x >> 16);
  // the 6-bit scales and mins of the half's four sub-blocks, one per byte
  const uint32_t s0 = w.hdr.y, s1 = w.hdr.z, s2 = w.hdr.w;
  const uint32_t sc4 = hb == 0 ? s0 & 0x3F3F3F3Fu : (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
  const uint32_t m4 = hb == 0 ? s1 & 0x3F3F3F3Fu : ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
  F32x4 hi[kNT], lo[kNT];
  const F32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int g = 0; g < 2; ++g) {
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int s = 2 * g + n;
      const float sc = ByteF(sc4, s);
      const H2 mul = Both(sc * (n == 0 ? 0x1p10f : 0x1p6f));
      const H2 sub = Both(sc * -0x1p-11f);
      H2 p[4];
      if (n == 0) {
        PairsQ4<false>(w.q[g].x, mul, sub, &p[0], &p[1]);
        PairsQ4<false>(w.q[g].y, mul, sub, &p[2], &p[3]);
      } else {
        PairsQ4<true>(w.q[g].x, mul, sub, &p[0], &p[1]);
        PairsQ4<true>(w.q[g].y, mul, sub, &p[2], &p[3]);
      }
      const F16x8 b = Join(p[0], p[1], p[2], p[3]);
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        hi[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[nt].hi[s], b, s == 0 ? zero : hi[nt], 0, 0, 0);
        lo[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[nt].lo[s], b, s == 0 ? zero : lo[nt], 0, 0, 0);
      }
    }
  }
  // What the centring took, less the mins: lane (r, kg) has c = 8 d sc - dmin m of
  // sub-block kg, exact in double, against the sub-blocks' sums. The rest joins in
  // double too, so for a single x the result rounds once, as the dequantised weight.
  const double c = __builtin_fma(8.0 * d, static_cast<double>((sc4 >> (8 * kg)) & 0xFFu),
                                 -(static_cast<double>(dmin) * static_cast<double>((m4 >> (8 * kg)) & 0xFFu)));
  const double dd = d * 0x1p14f;
  const F64x4 zero64 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt) {
    const F64x4 off = __builtin_amdgcn_mfma_f64_16x16x4f64(x[nt].sum, c, zero64, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      acc[nt][i] += static_cast<float>(__builtin_fma(dd, static_cast<double>((hi[nt][i] + lo[nt][i]) * inv[nt][i]), off[i]));
  }
}

// Quants q6 of quarter kQ for two bytes of a dword (shifted by 8 for the odd
// ones), as the low bits of 16-bit lanes: q6 (kQ < 2) or 16 q6.
template <int kQ>
__device__ __forceinline__ H2 PairQ6(uint32_t ql, uint32_t qh_up4, uint32_t qh_up2) {
  constexpr uint32_t kLo = kQ < 2 ? 0x000F000Fu : 0x00F000F0u;
  constexpr uint32_t kHi = kQ < 2 ? 0x00300030u : 0x03000300u;
  const H2 t = Half2((ql & kLo) | ((kQ & 1 ? qh_up2 : qh_up4) & kHi));
  // (q6 - 32) 2^-9, exact
  return __builtin_elementwise_fma(t, Both(kQ < 2 ? 0x1p15f : 0x1p11f), Both(-0x1p-4f));
}

template <int kNT>
__device__ __forceinline__ void TileQ6(const WRaw<true>& w, const XSplit (&x)[kNT], const F32x4 (&inv)[kNT], int kg,
                                       F32x4 (&acc)[kNT]) {
  const float d = HalfF(w.d) * 0x1p9f;
  // scale bytes 0-3 and 4-7 of the half; lane kg uses bytes 2 q + kg / 2
  const uint2 scb = Window8(w.sc, w.sh);
  const uint32_t ks = 4u * (static_cast<uint32_t>(kg) & 2u);
  const uint32_t sw[2] = {scb.x >> ks, scb.y >> ks};
  // signed bytes 0 and 2 as an fp16 pair: sc + 128 above 0x64 is 1024 + sc + 128
  H2 scp[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) scp[k] = Half2(((sw[k] ^ 0x00800080u) & 0x00FF00FFu) | 0x64006400u) + Both(-1152.0f);
  const uint2 qh = Window8(w.qh, w.sh);
  const uint2 ql[2] = {Window8(w.ql[0], w.sh), Window8(w.ql[1], w.sh)};
  F32x4 hi[kNT], lo[kNT];
  const F32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  auto step = [&](auto qc) {
    constexpr int q = decltype(qc)::value;  // columns 32 q + 8 kg .. + 7 of the half
    const uint2 l = ql[q & 1];
    const H2 t[4] = {PairQ6<q>(l.x, qh.x << 4, qh.x << 2), PairQ6<q>(l.x >> 8, qh.x >> 4, qh.x >> 6),
                     PairQ6<q>(l.y, qh.y << 4, qh.y << 2), PairQ6<q>(l.y >> 8, qh.y >> 4, qh.y >> 6)};
    const H2 s2 = {scp[q >> 1][q & 1], scp[q >> 1][q & 1]};
    H2 wh[4], wl[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      wh[k] = t[k] * s2;                                     // rounded to fp16
      wl[k] = __builtin_elementwise_fma(t[k], s2, -wh[k]);  // the exact remainder
    }
    const F16x8 bh = Join(wh[0], wh[1], wh[2], wh[3]);
    const F16x8 bl = Join(wl[0], wl[1], wl[2], wl[3]);
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      hi[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[nt].hi[q], bh, q == 0 ? zero : hi[nt], 0, 0, 0);
      lo[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[nt].lo[q], bh, q == 0 ? zero : lo[nt], 0, 0, 0);
      lo[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[nt].hi[q], bl, lo[nt], 0, 0, 0);
    }
  };
  step(std::integral_constant<int, 0>{});
  step(std::integral_constant<int, 1>{});
  step(std::integral_constant<int, 2>{});
  step(std::integral_constant<int, 3>{});
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[nt][i] += (d * inv[nt][i]) * (hi[nt][i] + lo[nt][i]);
}

// ---------------------------------------------------------------- values that are not finite

// Row `row` of a matrix times token t, each weight dequantised and added with one fused
// multiply-add: what the tiled kernel of the smallest calls gives for infinities and NaNs.
__device__ __forceinline__ float RowDot(bool q6, const uint8_t* w, int64_t row, int32_t nb, const float* x, int64_t t, int lane) {
  const uint32_t type = q6 ? kGgmlQ6_K : kGgmlQ4_K;
  const int32_t bytes = q6 ? kQ6KBlockBytes : kQ4KBlockBytes;
  const uint8_t* wr = w + row * nb * bytes;
  const float* xr = x + t * nb * kQK_K;
  float acc = 0.0f;
  for (int32_t b = 0; b < nb; ++b)
#pragma unroll 1
    for (int e = lane; e < kQK_K; e += 64)
      acc = __builtin_fmaf(dev::DeqElemAny(type, wr + static_cast<int64_t>(b) * bytes, e), xr[static_cast<int64_t>(b) * kQK_K + e], acc);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  return acc;
}

// ---------------------------------------------------------------- kernel

// From this many tokens on a call stands for one of the prefill GEMM: the slices of a K
// that is too long for a workgroup's registers become workgroups of their own, whose
// partial results a second launch sums, and a token with a value that is not finite
// gives NaNs. Below, a call stands for one of the tiled kernel: a workgroup walks the
// slices itself, which needs no buffer (such calls never had one, so they may overlap on
// several streams and be captured without a first run), and the results for infinities
// are the tiled kernel's.
constexpr int64_t kSliceMinTokens = 32;

struct SmallArgs {
  const uint8_t* w[kSmallMaxMats];
  float* out[kSmallMaxMats];
  int32_t rows[kSmallMaxMats];
  int32_t tile_end[kSmallMaxMats];  // row tiles of matrices 0 .. i
  uint32_t q6_mask;
  int32_t tiles;
  int32_t nb;
  int32_t bps;    // blocks per K slice
  int32_t loops;  // slices that a workgroup walks itself (1: slice blockIdx.z)
  const float* x;
  int32_t n_tokens;
  float* partial;  // more than one K slice: [slice][token][row] of each matrix, one matrix after the other
  int64_t slice_elems;
};

// Wave w holds half blocks kU w .. + kU - 1 of its workgroup's K slice, for every
// token of the workgroup's token tiles, split in registers; the workgroup walks
// row tiles blockIdx.x, blockIdx.x + gridDim.x, .... A tile's 16 rows of the slice are
// copied to LDS byte for byte (whole lines; each lane then picks its fields
// there), the tile after next's bytes in flight meanwhile. Its partial sums meet in
// LDS too: thread e sums output e over the waves. Both areas are double, so a tile
// takes one barrier. kSwiGLU: tile 2 p is gate's row tile p, tile 2 p + 1 up's, and
// a workgroup walks pairs.
template <int kW, int kU, int kNT, bool kAnyQ4, bool kAnyQ6, bool kSwiGLU>
struct SmallCfg {
  static constexpr int kToks = 16 * kNT;
  static constexpr int kMaxBlocks = kW * kU / 2;
  // 16-byte pieces of a staged row: the slice's blocks from the aligned piece
  // before the first byte to the one after the last; odd, so that the rows fall
  // on different banks
  static constexpr int kPieces = ((kMaxBlocks * (kAnyQ6 ? kQ6KBlockBytes + 0 : kQ4KBlockBytes) + (kAnyQ6 ? 29 : 0)) / 16) | 1;
  static constexpr int kWBytes = 16 * kPieces * 16;
  static constexpr int kStride = 20;
  // floats of a wave's sums; the padding puts the parts that neighbouring threads
  // read on different banks
  static constexpr int kRedWave = kToks * kStride + 4;
  static constexpr int kRedFloats = kW * kRedWave;
  static constexpr int kSum = kW / (4 * kNT);  // threads per output (rounded down)
  static_assert((kSum == 1 || kSum == 2 || kSum == 4) && kW % kSum == 0, "an output's threads lie in one quad");
  static constexpr int kInvFloats = kW * kU * kToks;
  // LDS: tile buffer 0 | tile buffer 1 | sums 0 | sums 1 | inverse scales
  static constexpr int kBytes = 2 * kWBytes + 8 * kRedFloats + 4 * kInvFloats;
  static constexpr int kRowsPerWave = (16 + kW - 1) / kW;
  static constexpr int kLoads = (kPieces + 63) / 64;
};

template <int kW, int kU, int kNT, bool kAnyQ4, bool kAnyQ6, bool kSwiGLU, bool kLoop>
__global__ __launch_bounds__(64 * kW, kW == 8 ? 2 : kW == 10 ? 3 : 4) void MatMulSmallKernel(SmallArgs a) {
  using C = SmallCfg<kW, kU, kNT, kAnyQ4, kAnyQ6, kSwiGLU>;
  constexpr int kToks = C::kToks;
  __shared__ __attribute__((aligned(16))) uint8_t lds[C::kBytes];
  __shared__ uint32_t lds_infinite[kW];
  int tid = threadIdx.x;
  int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int r = lane & 15;
  int kg = lane >> 4;
  // The lane counted again, so that what follows from it isn't kept in registers until
  // then: kLoop's 16 waves have 128 each, and a spilled address read back waits for all
  // of the weights on their way.
  auto lane_again = [&] {
    uint32_t all = ~0u;
    asm volatile("" : "+s"(all));
    lane = static_cast<int>(__builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0u)));
    tid = 64 * wave + lane;
    r = lane & 15;
    kg = lane >> 4;
  };
  const int t0 = static_cast<int>(blockIdx.y) * kToks;
  const int n_here = a.n_tokens - t0 < kToks ? a.n_tokens - t0 : kToks;
  auto first_block = [&](int z) { return (static_cast<int>(blockIdx.z) + z) * a.bps; };
  auto blocks_of = [&](int z) { return a.nb - first_block(z) < a.bps ? a.nb - first_block(z) : a.bps; };
  float* invs = reinterpret_cast<float*>(lds + 2 * C::kWBytes + 8 * C::kRedFloats) + wave * kU * kToks;

  // matrix and first row of a tile
  auto locate = [&](int tile, int* mi, int* r0) {
    *mi = 0;
    int first = 0;
    if constexpr (kSwiGLU) {
      *mi = tile & 1;
      *r0 = 16 * (tile >> 1);
      return;
    }
#pragma unroll
    for (int i = 0; i + 1 < kSmallMaxMats; ++i)
      if (tile >= a.tile_end[i]) {
        *mi = i + 1;
        first = a.tile_end[i];
      }
    *r0 = 16 * (tile - first);
  };
  auto is_q6 = [&](int mi) { return kAnyQ6 && (!kAnyQ4 || ((a.q6_mask >> mi) & 1u) != 0); };
  // first byte of row `row` of slice z
  auto row_ptr = [&](int mi, int row, int z) {
    const int64_t bb = is_q6(mi) ? kQ6KBlockBytes : kQ4KBlockBytes;
    return a.w[mi] + (static_cast<int64_t>(row) * a.nb + first_block(z)) * bb;
  };
  // A step of the workgroup: slice z of its k-th tile.
  struct Step {
    int k, z;
  };
  auto after = [&](Step s) { return kLoop && s.z + 1 < a.loops ? Step{s.k, s.z + 1} : Step{s.k + 1, 0}; };
  const int step = static_cast<int>(gridDim.x);
  auto tile_at = [&](int k) {
    return kSwiGLU ? 2 * (static_cast<int>(blockIdx.x) + (k >> 1) * step) + (k & 1) : static_cast<int>(blockIdx.x) + k * step;
  };
  // this wave's rows of a step: the aligned 16-byte pieces that hold the slice
  // (past the last step: the first tile's again, never used)
  U32x4 held[C::kRowsPerWave][C::kLoads];
  auto load = [&](Step s) {
    const int tile = tile_at(s.k) < a.tiles ? tile_at(s.k) : tile_at(0);
    const int z = s.z;
    int mi, r0;
    locate(tile, &mi, &r0);
    const int seg = blocks_of(z) * (is_q6(mi) ? kQ6KBlockBytes : kQ4KBlockBytes);
#pragma unroll
    for (int k = 0; k < C::kRowsPerWave; ++k) {
      const int row = r0 + wave + kW * k;  // past the tile's 16 rows: loaded, not staged
      const uint8_t* p = row_ptr(mi, row < a.rows[mi] ? row : a.rows[mi] - 1, z);  // clamped: loads stay in bounds
      const int sh = static_cast<int>(reinterpret_cast<uintptr_t>(p) & 15u);
      const int last = (sh + seg - 1) >> 4;
#pragma unroll
      for (int j = 0; j < C::kLoads; ++j) {
        const int piece = lane + 64 * j < last ? lane + 64 * j : last;
        held[k][j] = *reinterpret_cast<const U32x4*>(p - sh + 16 * piece);
      }
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int k = 0; k < C::kRowsPerWave; ++k)
#pragma unroll
      for (int j = 0; j < C::kLoads; ++j)
        if (wave + kW * k < 16 && lane + 64 * j < C::kPieces)
          *reinterpret_cast<U32x4*>(lds + buf * C::kWBytes + 16 * ((wave + kW * k) * C::kPieces + lane + 64 * j)) = held[k][j];
  };

  XSplit xs[kU][kNT];
  float gate = 0.0f, sum = 0.0f;
  Step now{0, 0}, next = after(now);
  // the slice's activations of this wave; past the slice: loaded, never used
  XRaw xr[kU][kNT];
  const int64_t cols = static_cast<int64_t>(a.nb) * kQK_K;
  // kLoop: n_tokens cols floats are less than 2^32 bytes
  const __amdgpu_buffer_rsrc_t xrows = dev::OutResource(const_cast<float*>(a.x), 4u * static_cast<uint32_t>(a.n_tokens * cols));
  auto load_x = [&](int z) {
    const int units = 2 * blocks_of(z);
#pragma unroll
    for (int k = 0; k < kU; ++k)
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        const int u = kU * wave + k < units ? kU * wave + k : units - 1;
        const int t = t0 + 16 * nt + (lane >> 2);
        const int64_t lane_at = (t < a.n_tokens ? t : a.n_tokens - 1) * cols + 8 * (lane & 3);
        const int64_t wave_at = static_cast<int64_t>(kQK_K) * first_block(z) + kUnit * u;
        if constexpr (kLoop) {
          LoadX(xr[k][nt], xrows, 4u * static_cast<uint32_t>(lane_at), 4u * static_cast<uint32_t>(wave_at));
        } else {
          LoadX(xr[k][nt], a.x + (lane_at + wave_at));
        }
      }
  };
  bool infinite = false;  // among this wave's activations so far
  if (lane == 0) lds_infinite[wave] = 0;
  // waves that have a unit of slice z; the others copy and sum
  auto waves_of = [&](int z) { return (2 * blocks_of(z) + kU - 1) / kU; };
  auto split_x = [&](int z) {
    if (wave >= waves_of(z)) return;
#pragma unroll
    for (int k = 0; k < kU; ++k)
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) infinite |= SplitX(xr[k][nt], xs[k][nt], invs + kToks * k + 16 * nt, lane, kAnyQ4);
    if (infinite) lds_infinite[wave] = 1;
  };
  load_x(0);
  load(now);
  split_x(0);
  if constexpr (kLoop) load_x(next.z);
  stage(0);
  load(next);
  __syncthreads();
  uint32_t flag = lds_infinite[lane % kW];  // (kLoop: of the first slice)
  for (int i = 0;; ++i, now = next, next = after(next)) {
    const int tile = tile_at(now.k);
    if (tile >= a.tiles) break;
    const int z = now.z;
    const int waves = waves_of(z);
    if constexpr (kLoop) {
      if constexpr (kAnyQ6) lane_again();
      if (i > 0) {
        split_x(z);
        load_x(next.z);
      }
    }
    int mi, r0;
    locate(tile, &mi, &r0);
    const int rows = a.rows[mi];
    const bool q6 = is_q6(mi);
    float* red = reinterpret_cast<float*>(lds + 2 * C::kWBytes) + (i & 1) * C::kRedFloats;
    F32x4 acc[kNT];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) acc[nt] = F32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (wave < waves) {
      const uint32_t sh = q6 ? static_cast<uint32_t>(reinterpret_cast<uintptr_t>(row_ptr(mi, r0 + r < rows ? r0 + r : rows - 1, z)) & 15u) : 0u;
      const uint8_t* wrow = lds + (i & 1) * C::kWBytes + 16 * C::kPieces * r;
#pragma unroll
      for (int k = 0; k < kU; ++k) {
        const int u = kU * wave + k;
        const int hb = u & 1;
        F32x4 inv[kNT];  // of tokens 4 kg .. + 3
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) inv[nt] = *reinterpret_cast<const F32x4*>(invs + kToks * k + 16 * nt + 4 * kg);
        if (q6) {
          if constexpr (kAnyQ6) {
            const uint32_t off = sh + kQ6KBlockBytes * static_cast<uint32_t>(u >> 1);
            WRaw<true> w;
            ReadW(w, wrow + off, off & 3u, hb, kg);
            TileQ6<kNT>(w, xs[k], inv, kg, acc);
          }
        } else {
          if constexpr (kAnyQ4) {
            WRaw<false> w;
            ReadW(w, wrow + kQ4KBlockBytes * (u >> 1), hb, kg);
            TileQ4<kNT>(w, hb, xs[k], inv, kg, acc);
          }
        }
      }
    }
    // D of the matrix core: column (lane % 16) is the weight row, rows 4 kg + i are tokens
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[wave * C::kRedWave + (16 * nt + 4 * kg + j) * C::kStride + r] = acc[nt][j];
    stage((i + 1) & 1);
    __syncthreads();
    load(after(next));
    // kSum threads share an output, each summing kW / kSum waves' parts
    const int t = tid / (16 * C::kSum), c = (tid / C::kSum) & 15, part = tid % C::kSum;
    if (t < n_here) {
      const float* p = red + part * (kW / C::kSum) * C::kRedWave + t * C::kStride + c;
      float w[kW / C::kSum];
#pragma unroll
      for (int k = 0; k < kW / C::kSum; ++k) w[k] = p[k * C::kRedWave];
      // pairwise: for 8 blocks the same tree whatever the shape
#pragma unroll
      for (int n = kW / C::kSum; n > 1; n = (n + 1) / 2)
#pragma unroll
        for (int k = 0; 2 * k < n; ++k) w[k] = 2 * k + 1 < n ? w[2 * k] + w[2 * k + 1] : w[2 * k];
      float v = w[0];
      if (C::kSum > 1) v += Xor1(v);
      if (C::kSum > 2) v += Xor2(v);
      if constexpr (kLoop) {
        v = z == 0 ? v : sum + v;
        sum = v;
        if (z + 1 < a.loops) continue;
      }
      const int64_t at = static_cast<int64_t>(t0 + t) * rows + r0 + c;
      const bool mine = part == 0 && r0 + c < rows;
      if (a.partial != nullptr) {
        if (mine) {
          int64_t first = static_cast<int64_t>(blockIdx.z) * a.slice_elems;
          for (int k = 0; k < mi; ++k) first += static_cast<int64_t>(a.n_tokens) * a.rows[k];
          a.partial[first + at] = v;
        }
      } else if (!kSwiGLU) {
        if (mine) a.out[mi][at] = v;
      } else if (mi == 0) {
        gate = v;
      } else if (mine) {
        a.out[0][at] = dev::SiluMul(gate, v);
        a.out[1][at] = v;
      }
    }
  }
  // An infinity's second term and 0 times it are NaNs that the sum of the weights' own
  // products does not have: the outputs that are not finite again, each by its wave
  if (a.n_tokens >= kSliceMinTokens) return;
  lane_again();
  if (kLoop) flag = lds_infinite[lane % kW];
  if (__builtin_amdgcn_ballot_w64(flag != 0) == 0) return;
  const int t = tid / (16 * C::kSum), c = (tid / C::kSum) & 15, part = tid % C::kSum;
  for (int k = 0; tile_at(k) < a.tiles; k += kSwiGLU ? 2 : 1) {
    int mi, r0;
    locate(tile_at(k), &mi, &r0);
    const bool mine = t < n_here && part == 0 && r0 + c < a.rows[mi];
    const int64_t at = static_cast<int64_t>(t0 + t) * a.rows[mi] + r0 + c;
    bool wrong = mine && !(fabsf(a.out[mi][at]) <= FLT_MAX);
    if (kSwiGLU) wrong = wrong || (mine && !(fabsf(a.out[1][at]) <= FLT_MAX));
    for (uint64_t left = __builtin_amdgcn_ballot_w64(wrong); left != 0; left &= left - 1) {
      const int from = __builtin_ctzll(left);
      const int row = r0 + __builtin_amdgcn_readlane(c, from), token = t0 + __builtin_amdgcn_readlane(t, from);
      const float v = RowDot(is_q6(mi), a.w[mi], row, a.nb, a.x, token, lane);
      if constexpr (kSwiGLU) {
        const float u = RowDot(is_q6(1), a.w[1], row, a.nb, a.x, token, lane);
        if (lane == from) {
          a.out[0][at] = dev::SiluMul(v, u);
          a.out[1][at] = u;
        }
      } else {
        if (lane == from) a.out[mi][at] = v;
      }
    }
  }
}

// The sum of the K slices, in order. kSwiGLU: out[0] = silu(matrix 0) * matrix 1, out[1] = matrix 1.
template <bool kSwiGLU>
__global__ __launch_bounds__(256) void SmallReduceKernel(SmallArgs a, int32_t slices) {
  const int64_t per_mat = static_cast<int64_t>(a.n_tokens) * a.rows[0];
  const int64_t n = kSwiGLU ? per_mat : a.slice_elems;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= n) return;
  const float* p = a.partial + e;
  float v = p[0];
  for (int z = 1; z < slices; ++z) v += p[z * a.slice_elems];
  if constexpr (kSwiGLU) {
    p += per_mat;
    float u = p[0];
    for (int z = 1; z < slices; ++z) u += p[z * a.slice_elems];
    a.out[0][e] = dev::SiluMul(v, u);
    a.out[1][e] = u;
  } else {
    int64_t at = e;
    int mi = 0;
#pragma unroll
    for (int i = 0; i + 1 < kSmallMaxMats; ++i) {
      const int64_t elems = static_cast<int64_t>(a.n_tokens) * a.rows[i];
      if (mi == i && at >= elems && a.out[i + 1] != nullptr) {
        at -= elems;
        mi = i + 1;
      }
    }
    a.out[mi][at] = v;
  }
}

// Workgroup shapes (waves, half blocks per wave, token tiles) and what they cost:
// a fixed part (launch, activations, first and last tile) and a part per row tile
// that a workgroup walks, by weight type: us = fixed + tiles * step, fitted to every
// shape's MI355X times (graph replay, weights from memory) at 1196 sizes of 32 .. 511
// tokens, 129 .. 32000 rows of 1 .. 56 blocks. From 8 blocks on it gives 0.88 to 1.1 of
// them (less work per tile is done below), and the shape chosen is within 0.2% of the
// best: 2048 x 2048 Q4_K at 448 tokens 27 us, 2048 x 6144 Q6_K at 21 tokens 14 (16
// measured). 16 waves and one token tile are quickest for few tokens and few tiles; two
// token tiles share a decode and win as the tiles add up; 10 waves fit rows of 10 blocks
// in two slices.
struct Shape {
  int w, u, nt;
  double fixed, step4, step6;
};
constexpr Shape kShapes[] = {{16, 1, 1, 4.9, 1.73, 1.83}, {8, 2, 2, 8.2, 2.2, 2.27}, {8, 1, 2, 5.9, 1.36, 1.47},
                             {10, 1, 2, 7.45, 1.64, 1.76}, {10, 2, 1, 6.4, 2.14, 2.7}};
constexpr double kLoopX = 1.2;  // splitting a slice's activations again for each step
constexpr int kShapeCount = sizeof(kShapes) / sizeof(kShapes[0]);

// How a launch of one workgroup shape covers a call: K slices of bps blocks,
// groups of token tiles, row tiles per workgroup.
struct Plan {
  int bps, slices, loops, groups, grid, iters;
};

Plan PlanFor(int shape, int nb, int64_t n_tokens, int want) {
  const Shape& s = kShapes[shape];
  const int nt = s.nt, blocks = s.w * s.u / 2;
  Plan p;
  p.slices = (nb + blocks - 1) / blocks;
  p.bps = (nb + p.slices - 1) / p.slices;
  p.slices = (nb + p.bps - 1) / p.bps;
  p.loops = 1;
  if (n_tokens < kSliceMinTokens) {
    p.loops = p.slices;
    p.slices = 1;
  }
  p.groups = static_cast<int>((n_tokens + 16 * nt - 1) / (16 * nt));
  const int cap = kCUs / (p.groups * p.slices) > 0 ? kCUs / (p.groups * p.slices) : 1;  // one workgroup per CU
  p.iters = (want + cap - 1) / cap;
  p.grid = (want + p.iters - 1) / p.iters;
  return p;
}

// us of a matrix on shape s, the launch that sums its K slices included.
double ShapeCost(int shape, int nb, int64_t n_tokens, int64_t rows, bool q6) {
  const Shape& s = kShapes[shape];
  const Plan p = PlanFor(shape, nb, n_tokens, static_cast<int>((rows + 15) / 16));
  if (p.loops > 1 && shape != 0) return 1e9;  // built for the first shape only
  const double reduce = p.slices > 1 ? 2.2 + 8.0 * p.slices * static_cast<double>(n_tokens) * static_cast<double>(rows) / 5e6 : 0.0;
  // rows of 1 to 3 blocks leave waves without work (12000 x 512 Q4_K, 224 tokens: 26 us
  // on the third shape, 37 on the second; 35 on the GEMM)
  const double share = nb < 4 ? 0.5 + nb / static_cast<double>(s.w * s.u) : 1.0;
  const double step = share * (q6 ? s.step6 : s.step4) + (p.loops > 1 ? kLoopX : 0.0);
  return s.fixed + p.iters * p.loops * step + reduce;
}

template <int kShape, bool kSwiGLU, bool kLoop>
void LaunchTyped(const char* name, SmallArgs a, int32_t n_mats, bool any4, bool any6) {
  constexpr int kW = kShapes[kShape].w, kU = kShapes[kShape].u, kNT = kShapes[kShape].nt;
  const Plan p = PlanFor(kShape, a.nb, a.n_tokens, kSwiGLU ? a.tiles / 2 : a.tiles);
  RPG_CHECK(p.groups <= 65535 && p.slices <= 65535, "small-batch matmul grid too large");
  a.bps = p.bps;
  a.loops = p.loops;
  const dim3 grid(static_cast<unsigned>(p.grid), static_cast<unsigned>(p.groups), static_cast<unsigned>(p.slices));
  const dim3 block(64 * kW);
  a.slice_elems = 0;
  for (int i = 0; i < n_mats; ++i) a.slice_elems += static_cast<int64_t>(a.n_tokens) * a.rows[i];
  if (p.slices > 1) a.partial = SplitPartials(static_cast<size_t>(p.slices) * static_cast<size_t>(a.slice_elems) * sizeof(float));
  if (any4 && any6) {
    if constexpr (!kSwiGLU) Launch(name, MatMulSmallKernel<kW, kU, kNT, true, true, false, kLoop>, grid, block, a);
  } else if (any6) {
    Launch(name, MatMulSmallKernel<kW, kU, kNT, false, true, kSwiGLU, kLoop>, grid, block, a);
  } else {
    Launch(name, MatMulSmallKernel<kW, kU, kNT, true, false, kSwiGLU, kLoop>, grid, block, a);
  }
  if (p.slices > 1) {
    const int64_t n = kSwiGLU ? static_cast<int64_t>(a.n_tokens) * a.rows[0] : a.slice_elems;
    Launch("MatMulSmallReduceKernel", SmallReduceKernel<kSwiGLU>, dim3(GridFor(n, 256)), dim3(256), a,
           static_cast<int32_t>(p.slices));
  }
}

// One launch of a group whose matrices all take shape `shape`.
template <bool kSwiGLU>
void LaunchShaped(int shape, const SmallMat* mats, int32_t n_mats, int32_t nb, const float* x, int64_t n_tokens) {
  SmallArgs a{};
  a.nb = nb;
  a.x = x;
  a.n_tokens = static_cast<int32_t>(n_tokens);
  bool any4 = false, any6 = false;
  for (int i = 0; i < kSmallMaxMats; ++i) {
    if (i < n_mats) {
      a.w[i] = mats[i].w;
      a.out[i] = mats[i].out;
      a.rows[i] = static_cast<int32_t>(mats[i].rows);
      a.tiles += (a.rows[i] + 15) / 16;
      if (mats[i].q6) a.q6_mask |= 1u << i;
      any4 = any4 || !mats[i].q6;
      any6 = any6 || mats[i].q6;
    }
    a.tile_end[i] = i + 1 < n_mats ? a.tiles : INT32_MAX;
  }
  const char* name = kSwiGLU        ? (any6 ? "MatMulSmallSwiGLUQ6KKernel" : "MatMulSmallSwiGLUQ4KKernel")
                     : any4 && any6 ? "MatMulSmallQ4KQ6KKernel"
                     : any6         ? "MatMulSmallQ6KKernel"
                                    : "MatMulSmallQ4KKernel";
  switch (shape) {
    case 0:
      if (PlanFor(0, nb, n_tokens, a.tiles).loops > 1) return LaunchTyped<0, kSwiGLU, true>(name, a, n_mats, any4, any6);
      return LaunchTyped<0, kSwiGLU, false>(name, a, n_mats, any4, any6);
    case 1: return LaunchTyped<1, kSwiGLU, false>(name, a, n_mats, any4, any6);
    case 2: return LaunchTyped<2, kSwiGLU, false>(name, a, n_mats, any4, any6);
    case 3: return LaunchTyped<3, kSwiGLU, false>(name, a, n_mats, any4, any6);
    default: return LaunchTyped<4, kSwiGLU, false>(name, a, n_mats, any4, any6);
  }
}

// The shape for `rows` rows, and its cost. Up to 8 blocks (4 for the third shape) the
// first shapes hold whole rows and sum in one order, so a group may take the shape of
// its rows together; a longer row's order depends on the shape, which then comes from
// the matrix's own rows.
int ShapeOf(int64_t rows, bool q6, int32_t nb, int64_t n_tokens, double* us) {
  int best = 0;
  for (int i = 0; i < (nb <= 4 ? 3 : nb <= 8 ? 2 : kShapeCount); ++i) {
    const double c = ShapeCost(i, nb, n_tokens, rows, q6);
    if (i == 0 || c < *us) {
      best = i;
      *us = c;
    }
  }
  return best;
}

}  // namespace

bool MatMulSmallWins(const SmallMat& m, int32_t nb, int64_t n_tokens) {
  double us = 0.0;
  ShapeOf(m.rows, m.q6, nb, n_tokens, &us);
  const double mega = static_cast<double>(m.rows) * 256e-6 * nb;  // weights, in millions
  // The tiled kernel: 2.4 us and 0.26 (Q4_K) or 0.17 us per token and million weights
  // (2048 x 2048 Q4_K: 4.8 us at 2 tokens, 11.4 at 8, against 6.7 here; 2048 x 6144
  // Q6_K: 8.5 and 18.9 against 15).
  if (n_tokens < 32) return us <= 1.1 * (2.4 + (m.q6 ? 0.17 : 0.26) * static_cast<double>(n_tokens) * mega);
  // The prefill kernels. (Of 2288 sizes of 2 to 511 tokens, 13 take 3 to 9% longer than on
  // the GEMM: 5120 x 5120 Q6_K at 333 tokens 123 us and 113, 2560 x 9728 Q4_K at 256 78
  // and 74.)
  return us <= std::min(MfmaUs(m.q6, m.rows, nb, n_tokens), PlanesUs(m.q6, m.rows, nb, n_tokens));
}

void LaunchMatMulSmall(const SmallMat* mats, int32_t n_mats, int32_t nb, const float* x, int64_t n_tokens) {
  int shape_of_all = -1;
  if (nb <= 8) {
    int64_t rows = 0;
    bool any6 = false;
    for (int i = 0; i < n_mats; ++i) {
      rows += mats[i].rows;
      any6 = any6 || mats[i].q6;
    }
    double us = 0.0;
    shape_of_all = ShapeOf(rows, any6, nb, n_tokens, &us);
  }
  for (int shape = 0; shape < kShapeCount; ++shape) {
    SmallMat same[kSmallMaxMats];
    int n = 0;
    for (int i = 0; i < n_mats; ++i) {
      double us = 0.0;
      const int s = shape_of_all >= 0 ? shape_of_all : ShapeOf(mats[i].rows, mats[i].q6, nb, n_tokens, &us);
      if (s == shape) same[n++] = mats[i];
      if (n == kSmallMaxMats || (i + 1 == n_mats && n > 0)) {
        LaunchShaped<false>(shape, same, n, nb, x, n_tokens);
        n = 0;
      }
    }
  }
}

void LaunchMatMulSmallSwiGLU(const SmallMat& gate, const SmallMat& up, int32_t nb, const float* x, int64_t n_tokens) {
  const SmallMat mats[2] = {gate, up};
  double us = 0.0;
  LaunchShaped<true>(ShapeOf((nb <= 8 ? 2 : 1) * gate.rows, gate.q6, nb, n_tokens, &us), mats, 2, nb, x, n_tokens);
}

}  // namespace rpg
