// The arithmetic of one lane's chunk of consecutive elements: rotation, group scales, E2M1 codes.  Used by the
// quantizers (fpq_quantize.hip) and by the GEMM that quantizes its few activation rows itself (fpq_gemm_stream.hip).
#pragma once
#include <type_traits>

#include "fpq_device.h"

namespace fpq {

constexpr int kFmtMx = 0;
constexpr int kFmtNv = 1;

__device__ __forceinline__ void unpack8(const uint4& raw, float (&p)[8]) {
  p[0] = bf16_lo(raw.x); p[1] = bf16_hi(raw.x);
  p[2] = bf16_lo(raw.y); p[3] = bf16_hi(raw.y);
  p[4] = bf16_lo(raw.z); p[5] = bf16_hi(raw.z);
  p[6] = bf16_lo(raw.w); p[7] = bf16_hi(raw.w);
}

constexpr float kKappa = -0x1.8p-26f;  // fma(x, 0.75, x * kKappa) rounds to the E2M1 code of x / fl(4/3)

// SiLU by lookup: an LDS copy of the busy part of a 65536-entry table of bf16(silu(g)), |g| in [2^-14, 128), held as fp32;
// the two table offsets of a pair of gates are formed with packed 16-bit arithmetic.  Smaller magnitudes are g / 2 exactly
// (the relative deviation, |g| / 2, is below half a bf16 step) and larger ones come from the global table: a wave that
// holds any redoes those lanes.
constexpr uint32_t kSiluLdsFirst = 113u << 7;         // bf16 magnitude bits of 2^-14
constexpr uint32_t kSiluLdsCount = 21u * 128u;        // magnitudes up to (not including) 2^7
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) const float lds_f32;

template <int THREADS>
__device__ __forceinline__ void silu_table_to_lds(float* lds, const uint16_t* __restrict__ table) {
  for (uint32_t i = threadIdx.x; i < 2u * kSiluLdsCount / 4u; i += THREADS) {
    const uint32_t first = 4u * i, sgn = first >= kSiluLdsCount ? 1u : 0u;
    const uint2 e = *(const uint2*)&table[(sgn << 15) | (kSiluLdsFirst + first - sgn * kSiluLdsCount)];
    *(float4*)&lds[first] = make_float4(bf16_lo(e.x), bf16_hi(e.x), bf16_lo(e.y), bf16_hi(e.y));
  }
}

// sv[i]: bf16(silu(.)) of the i-th of the bf16 values in `w`.  live: whether anybody reads this lane's (other lanes get some
// value of the table, and do not send the wave round again).
template <int N>
__device__ __forceinline__ void silu_lookup(const uint32_t (&w)[N], float (&sv)[2 * N], lds_f32* table,
                                            const uint16_t* __restrict__ global, bool live) {
  u16x2 most = u16x2{0, 0};
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const u16x2 bits = __builtin_bit_cast(u16x2, w[k]);
    const u16x2 idx = __builtin_bit_cast(u16x2, w[k] & 0x7fff7fffu) - (unsigned short)kSiluLdsFirst;
    most = __builtin_elementwise_max(most, idx);
    const u16x2 in = __builtin_elementwise_min(idx, u16x2{kSiluLdsCount - 1, kSiluLdsCount - 1});
    const u16x2 at = (bits >> (unsigned short)15) * (unsigned short)kSiluLdsCount + in;
    sv[2 * k] = table[at.x];
    sv[2 * k + 1] = table[at.y];
  }
  const bool outside = live && (most.x >= kSiluLdsCount || most.y >= kSiluLdsCount);
  if (__builtin_amdgcn_ballot_w64(outside) != 0ull) {
#pragma unroll
    for (int e = 0; e < 2 * N; ++e) {
      const uint32_t bits = (e & 1) ? w[e >> 1] >> 16 : w[e >> 1] & 0xffffu, mag = bits & 0x7fffu;
      if (mag < kSiluLdsFirst) {
        uint32_t b = __float_as_uint(__uint_as_float(bits << 16) * 0.5f);   // rounded to bf16, to nearest even
        b += 0x7fffu + ((b >> 16) & 1u);
        sv[e] = __uint_as_float(b & 0xffff0000u);
      } else if (mag >= kSiluLdsFirst + kSiluLdsCount) {
        sv[e] = __uint_as_float((uint32_t)global[bits] << 16);
      }
    }
  }
}

// Hadamard output index that sequency-ordered output k of a g-block takes: bitreverse(k ^ (k >> 1))
__host__ __device__ constexpr int gsr_source(int k, int g) {
  int gray = k ^ (k >> 1), r = 0;
  for (int b = 1; b < g; b <<= 1) {
    r = (r << 1) | (gray & 1);
    gray >>= 1;
  }
  return r;
}

template <int ZERO>
__device__ __forceinline__ uint32_t fix_zero_nibbles(uint32_t w) {
  if (ZERO == kZeroReference) {
    const uint32_t nz = ((w & 0x77777777u) + 0x77777777u) & 0x88888888u;  // bit 3 set where magnitude != 0
    w |= nz ^ 0x88888888u;
  }
  return w;
}

// v[i] += sign * (v[i] of the lane that the quad permutation CTRL names), one instruction each.  Written as assembly
// because the compiler keeps the lane move apart; a DPP operand may be read two wait states after it was written,
// which the leading s_nop grants whatever comes before.
template <int CTRL>
__device__ __forceinline__ void fma_exchange8(float (&v)[8], float sign) {
#define FPQ_FMAC_DPP(QP)                                                                                            \
  asm volatile("s_nop 1\n\t"                                                                                        \
               "v_fmac_f32_dpp %0, %0, %8 " QP "\n\tv_fmac_f32_dpp %1, %1, %8 " QP "\n\t"                           \
               "v_fmac_f32_dpp %2, %2, %8 " QP "\n\tv_fmac_f32_dpp %3, %3, %8 " QP "\n\t"                           \
               "v_fmac_f32_dpp %4, %4, %8 " QP "\n\tv_fmac_f32_dpp %5, %5, %8 " QP "\n\t"                           \
               "v_fmac_f32_dpp %6, %6, %8 " QP "\n\tv_fmac_f32_dpp %7, %7, %8 " QP                                  \
               : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])     \
               : "v"(sign))
  static_assert(CTRL == 0xB1 || CTRL == 0x4E, "lane ^ 1 or lane ^ 2");
  if (CTRL == 0xB1) FPQ_FMAC_DPP("quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf");
  else FPQ_FMAC_DPP("quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf");
#undef FPQ_FMAC_DPP
}

// One lane's chunk of EPL consecutive elements, rotated in place: the butterflies with stride < EPL stay in the
// lane's registers, a wider rotation takes one or two exchanges with the neighbouring lanes that hold the rest
// of the block (lane % (G / EPL) is the chunk's place in it).
//
// An exchange gives the lower lane a + b and the upper one a - b.  With KEEP_ZERO_SIGN the upper lane negates its own
// value and both add (two instructions and a wait between them); otherwise a lane holds its values negated through
// the stages before an exchange in which it is the upper one (the norm's sign: a rotation of negated values is the
// negated rotation), and the exchange is ONE fused multiply-add with +-1, own + sign * other, whose product is exact.
// The only differences are the sign of a zero, which the reference's zero policy does not look at, and the sign of a NaN.
template <int EPL, int G, int ROT, bool KEEP_ZERO_SIGN>
__device__ __forceinline__ void rotate_chunk(float (&v)[EPL], float norm, uint32_t lane) {
  if (ROT == FPQ_ROT_HADAMARD || ROT == FPQ_ROT_GSR) {
    static_assert(G <= 4 * EPL, "at most two exchanges between lanes");
    constexpr bool kNegate = !KEEP_ZERO_SIGN && G > EPL;
    const uint32_t upper1 = (lane & 1u) << 31, upper2 = G > 2 * EPL ? (lane & 2u) << 30 : 0u;
    const float n = kNegate ? __uint_as_float(__float_as_uint(norm) ^ upper1 ^ upper2) : norm;
#pragma unroll
    for (int i = 0; i < EPL; ++i) v[i] *= n;
#pragma unroll
    for (int s = 1; s < (G < EPL ? G : EPL); s *= 2) {
      __builtin_amdgcn_sched_barrier(0);  // keep the stages in place: EPL live values, no more
#pragma unroll
      for (int i = 0; i < EPL; ++i) {
        if ((i & s) == 0) {
          const float a = v[i], b = v[i + s];
          v[i] = a + b;
          v[i + s] = a - b;
        }
      }
    }
    auto exchange = [&](auto ctrl, uint32_t upper) __attribute__((always_inline)) {
      constexpr int kCtrl = decltype(ctrl)::value;
      __builtin_amdgcn_sched_barrier(0);
      const float sign = __uint_as_float(0xbf800000u ^ upper);   // lower lane -1 (its partner holds -b), upper lane +1
      if (kNegate) {
#pragma unroll
        for (int i = 0; i < EPL; i += 8) fma_exchange8<kCtrl>(*(float (*)[8])&v[i], sign);
      } else {
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
          const float other = __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v[i]), kCtrl, 0xF,
                                                                                 0xF, true));
          v[i] = other + __uint_as_float(__float_as_uint(v[i]) ^ upper);
        }
      }
    };
    // stride EPL: the two halves of a rotation block sit in lanes 2u and 2u + 1; stride 2 EPL (a 128-wide rotation
    // with EPL = 32): the quarters sit in lanes 4u .. 4u + 3 and the partner is lane ^ 2
    if (G > EPL) exchange(std::integral_constant<int, 0xB1 /* quad_perm [1,0,3,2] */>{}, upper1);
    if (G > 2 * EPL) exchange(std::integral_constant<int, 0x4E /* quad_perm [2,3,0,1] */>{}, upper2);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (ROT == FPQ_ROT_GSR) {
    // sequency order inside every G-block (G <= EPL here): a compile-time renaming of registers
    static_assert(ROT != FPQ_ROT_GSR || G <= EPL, "GSR blocks must fit in one lane");
    float w[EPL];
#pragma unroll
    for (int k = 0; k < EPL; ++k) w[k] = v[(k & ~(G - 1)) | gsr_source(k & (G - 1), G)];
#pragma unroll
    for (int k = 0; k < EPL; ++k) v[k] = w[k];
  }
}

// Whether a rotated chunk holds a NaN or an infinity.  quantize_chunk gives a NaN element the code of its sign and the
// largest magnitude, and an infinite NVFP4 group the scale byte of a NaN; quantize_chunk_slow, as the generic kernel, leaves
// a NaN element out (code of zero) and clamps the group's scale.  Kernels that took calls over from the generic one send
// such chunks there: one NaN in a decode row must not depend on how many rows are quantized with it.  (Not the norm's tile
// kernel, 2-5 % slower with the check: a NaN there is the whole block's, and meets a scale of 2^-126 or zero.)  It costs a
// few rows' GEMM 0-1 % (4 x 4096 x 4096 5.87 -> 5.95 us) and ragged rows 1-4 % (2000 x 3200 4.63 -> 4.70, NVFP4 5.45 -> 5.66).
template <int EPL>
__device__ __forceinline__ bool chunk_not_finite(const float (&v)[EPL]) {
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < EPL; ++i) m = __builtin_elementwise_maximum(m, __builtin_fabsf(v[i]));   // (keeps a NaN)
  return !(m <= 3.402823466e+38f);
}

// E2M1 codes and scale bytes of one lane's rotated chunk (cw: CW dwords of codes; sbytes: the scale bytes, with
// eight of them the first four in sb_lo).  Returns whether a group left the range in which the two-operation
// division is proven: the caller then redoes the chunk with quantize_chunk_slow.
template <int EPL, int FMT, int ZERO, bool QUEST>
__device__ __forceinline__ bool quantize_chunk(const float (&v)[EPL], float gs, bool nv_fast,
                                               const float2* __restrict__ lut, uint32_t (&cw)[EPL / 8],
                                               uint32_t& sbytes, uint32_t& sb_lo) {
  constexpr int GROUP = FMT == kFmtMx ? 32 : 16;
  constexpr int NG = EPL / GROUP;
  bool need_slow = false;
#pragma unroll
  for (int gi = 0; gi < NG; ++gi) {
    float a = 0.0f;
    if (!QUEST) {
#pragma unroll
      for (int i = 0; i < GROUP; ++i) a = __builtin_fmaxf(a, __builtin_fabsf(v[gi * GROUP + i]));
    }
    uint32_t byte;
    bool fast;
    float k1, k2, cvt_scale;
    if (QUEST) {
      float os[4], oq[4];
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        const float* p = &v[gi * GROUP + 8 * o];
        float sum = p[0], sq = p[0] * p[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) {
          sum = sum + p[i];
          sq = sq + p[i] * p[i];
        }
        os[o] = sum;
        oq[o] = sq;
      }
      const float sum = (os[0] + os[1]) + (os[2] + os[3]), sq = (oq[0] + oq[1]) + (oq[2] + oq[3]);
      const float mean = sum * 0.03125f, msq = sq * 0.03125f;
      float var = msq - mean * mean;
      var = var > 0.0f ? var : 0.0f;
      const float sc = __builtin_sqrtf(var) * 0.48707976f + 1e-8f;   // fl32(2.92247856 / 6); >= 1e-8: normal
      byte = (__float_as_uint(sc) >> 23) & 0xffu;
      fast = true;
      k1 = k2 = 0.0f;
      cvt_scale = __uint_as_float(byte << 23);                         // s = 2^floor(log2(sc))
    } else if (FMT == kFmtMx) {
      const uint32_t bits = __float_as_uint(a);
      byte = bits >> 23;
      fast = (byte - 29u) <= 198u || bits == 0u;                       // -98 <= e <= 100, or all zero
      k1 = 0.75f;
      k2 = kKappa;
      cvt_scale = __uint_as_float((bits & 0x7f800000u) - (2u << 23));  // 2^(e-2)
      if (bits == 0u) {  // a zero group stores 2^-126 and zero codes
        byte = 1u;
        cvt_scale = 1.0f;
      }
    } else {
      float t = div6_rn(a) * gs;
      t = t > 448.0f ? 448.0f : t;
      byte = e4m3_encode(t);
      fast = nv_fast;
      const float2 e = lut[byte & 0x7fu];
      k1 = e.x;
      k2 = e.y;
      cvt_scale = 1.0f;
    }
    need_slow |= !fast;
#pragma unroll
    for (int d = 0; d < GROUP / 8; ++d) {
      uint32_t w = 0u;
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const float x0 = v[gi * GROUP + d * 8 + 2 * h], x1 = v[gi * GROUP + d * 8 + 2 * h + 1];
        float q0 = QUEST ? x0 : __builtin_fmaf(x0, k1, x0 * k2);
        float q1 = QUEST ? x1 : __builtin_fmaf(x1, k1, x1 * k2);
        if (ZERO == kZeroSigned && !QUEST) {  // x / s keeps the sign of x, also for -0
          q0 = __builtin_copysignf(q0, x0);
          q1 = __builtin_copysignf(q1, x1);
        }
        if (h == 0) w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, q0, q1, cvt_scale, 0);
        if (h == 1) w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, q0, q1, cvt_scale, 1);
        if (h == 2) w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, q0, q1, cvt_scale, 2);
        if (h == 3) w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, q0, q1, cvt_scale, 3);
      }
      if (FMT == kFmtNv && ZERO == kZeroSigned) w = byte == 0u ? 0u : w;  // zero scale: +0 codes
      cw[gi * (GROUP / 8) + d] = fix_zero_nibbles<ZERO>(w);
    }
    sbytes |= (byte & 0xffu) << (8 * (gi & 3));
    if (NG == 8 && gi == 3) {  // eight scale bytes per chunk: park the first four
      sb_lo = sbytes;
      sbytes = 0u;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  return need_slow;
}

// UNROLL: for kernels that may not have an array in scratch memory (v and cw, indexed by a loop's group): setting it up
// costs every launch, although hardly any takes this path.  The streaming kernels, larger and longer, measured the same
// either way (NVFP4 8192 x 4096 16.4 us) or worse unrolled (MXFP4 4096 x 5120, 64-wide, 11.3 -> 13.0) and keep the loop.
template <int EPL, int FMT, int ZERO, bool UNROLL = false>
__device__ __forceinline__ void quantize_chunk_slow(const float (&u)[EPL], float gs, float rg,
                                                    uint32_t (&cw)[EPL / 8], uint32_t& sbytes) {
  constexpr int GROUP = FMT == kFmtMx ? 32 : 16;
  constexpr int NG = EPL / GROUP;
  sbytes = 0u;
#pragma unroll UNROLL ? NG : 1
  for (int gi = 0; gi < NG; ++gi) {
    float a = 0.0f;
#pragma unroll
    for (int i = 0; i < GROUP; ++i) a = __builtin_fmaxf(a, __builtin_fabsf(u[gi * GROUP + i]));
    const GroupScale g = FMT == kFmtMx ? mx_group_scale(a) : nv_group_scale(a, gs, rg);
#pragma unroll
    for (int d = 0; d < GROUP / 8; ++d) {
      uint32_t w = 0u;
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        const float xv = u[gi * GROUP + d * 8 + h];
        float q = scale_element(xv, g);
        if (ZERO == kZeroSigned) q = __builtin_copysignf(q, xv);
        if (FMT == kFmtNv) q = g.zero ? 0.0f : q;
        w |= e2m1_code<ZERO>(q) << (4 * h);
      }
      cw[gi * (GROUP / 8) + d] = w;
    }
    sbytes |= (g.byte & 0xffu) << (8 * gi);
  }
}

// Entry `byte` of the NVFP4 division table quantize_chunk reads: RN(1/s) and RN((1 - s RN(1/s)) / s) for the group
// scale s that the E4M3 byte stands for (rg: 1 / global scale).
__device__ __forceinline__ float2 nv_division(uint32_t byte, float rg, bool nv_fast) {
  const float s = e4m3_decode(byte) * rg;
  float2 e = make_float2(0.0f, 0.0f);
  if (s != 0.0f && nv_fast) {
    const float y = 1.0f / s;
    e = make_float2(y, __builtin_fmaf(-s, y, 1.0f) / s);
  }
  return e;
}
// The global scales for which every table entry is proven.
__device__ __forceinline__ bool nv_global_scale_fast(float gs) {
  return gs >= 8.673617379884035e-19f && gs <= 1.152921504606847e18f;
}

}  // namespace fpq
