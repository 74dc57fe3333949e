// A GEMM that quantizes its few activation rows itself: a part of the weight-streaming kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/fpq.h"
#include "fpq_device.h"
#include "fpq_gemm_epilogue.h"
#include "fpq_quantize_chunk.h"

namespace fpq {

typedef unsigned v4u_s __attribute__((ext_vector_type(4)));

struct Packed {};
struct PackedSlabs {};
struct PackedSlabsInARow {};
struct FewRows {
  const uint4* x;            // bf16 [M, xk]; SiLU*up: gate
  const uint4* up;           // SiLU*up: the multiplier; RMSNorm: the norm's weight [xk]
  const uint16_t* silu;      // ... and the table of bf16(silu(g))
  const float* gs;           // NVFP4: the activations' global scale
  uint8_t *codes, *scales;   // optional: the quantized rows, in the packed layout (rows past M are not written)
  float norm;
  int xk;                    // a multiple of 32 and of the rotation's size; K is padded to whole blocks
  float eps;                 // RMSNorm
};
enum { kFewPlain = 0, kFewSilu = 1, kFewNorm = 2 };   // what a few rows' chunk goes through before it is rotated
// 32-element chunks a wave quantizes at most: one per lane and pass
constexpr int few_rows_passes(int pro) { return pro == kFewPlain ? 2 : 1; }
constexpr int few_rows_chunks(int pro) { return 64 * few_rows_passes(pro); }
constexpr int kFewNormRows = 4;   // at most, with a norm (see norm_rows_multi)

// The quantization of a few activation rows inside a GEMM: a wave's 32-element chunks in lane order, row by row (the eight
// chunks of a 256-K block are neighbours, so the lanes of a rotation block are), of the blocks first, first + NW, ... that
// the wave multiplies.
//
// SiLU*up looks its values up in LDS, where every workgroup puts the busy part of the table (silu_lookup) while its rows and
// weights are on their way: 32 gathers per lane from the global table, most of a line each, kept the texture path busy for
// three microseconds ahead of the weights (us, global / LDS: MXFP4 1 x 4096 x 14336 12.5 / 11.5, 1 x 2048 x 8192 8.1 / 7.8,
// NVFP4 1 x 4096 x 12288 13.7 / 13.3).
template <bool NV, int XG, int XROT, int XPRO, int NW>
struct FewChunks {
  static constexpr int kPasses = few_rows_passes(XPRO), kChunks = few_rows_chunks(XPRO), FMT = NV ? kFmtNv : kFmtMx;
  static constexpr int kOctets = few_rows_chunks(kFewNorm) * 4 * NW;   // of a workgroup's rows, at most
  static constexpr int kTableLoads = (2 * (int)kSiluLdsCount / 4 + 64 * NW - 1) / (64 * NW);
  struct Shared {
    // a wave's quantized chunks, 16 bytes of codes each, and their scale bytes in the order the matrix instruction takes
    // them: [block][K half][K step]
    uint8_t codes[NW][kChunks * 16];
    uint8_t scales[NW][kChunks * (NV ? 2 : 1)];
    float2 lut[NV ? 128 : 1];
    float octets[XPRO == kFewNorm ? kOctets : 4];
    float silu[XPRO == kFewSilu ? 2 * kSiluLdsCount : 4];
  };
  uint4 xr[kPasses][4], ur[XPRO != kFewPlain ? kPasses : 1][4];
  uint2 table[XPRO == kFewSilu ? kTableLoads : 1];
  int col[kPasses], at[kPasses];
  int chunks;

  // Asked for before the weights, since loads complete in order.
  __device__ __forceinline__ void load(const FewRows& in, int M, int first, int nblk, int lane) {
    chunks = M * nblk * 8;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int ci = min(p * 64 + lane, max(chunks - 1, 0)), blk = ci >> 3, row = nblk > 0 ? blk / nblk : 0;
      const int kb = nblk > 0 ? first + NW * (blk - row * nblk) : 0;
      col[p] = kb * 256 + (ci & 7) * 32;
      at[p] = row * 0x10000 + kb;
      // (a chunk in the padding of the last block reads the row's start and is replaced by zeros)
      const size_t from = ((size_t)row * in.xk + (col[p] < in.xk ? col[p] : 0)) >> 3;
      if (p == 0 || chunks > 64) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          xr[p][i] = in.x[from + i];
          if constexpr (XPRO == kFewSilu) ur[p][i] = in.up[from + i];
          if constexpr (XPRO == kFewNorm) ur[p][i] = in.up[col[p] / 8 + i];   // (xk is whole blocks there)
        }
      }
    }
    if constexpr (XPRO == kFewSilu) {
#pragma unroll
      for (int i = 0; i < kTableLoads; ++i) {
        const uint32_t first4 = 4u * min((uint32_t)(threadIdx.x + 64 * NW * i), 2u * kSiluLdsCount / 4u - 1u);
        const uint32_t sgn = first4 >= kSiluLdsCount ? 1u : 0u;
        table[i] = *(const uint2*)&in.silu[(sgn << 15) | (kSiluLdsFirst + first4 - sgn * kSiluLdsCount)];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  // hand_on: the quantized rows also go to in.codes and in.scales.
  __device__ __forceinline__ void quantize(const FewRows& in, int M, Shared& sh, int wave, int lane, bool hand_on) {
    float gs = 1.0f, rg = 1.0f;
    bool nv_fast = true;
    if constexpr (NV) {
      gs = *in.gs;
      rg = gs == 0.0f ? 0.0f : 1.0f / gs;
      nv_fast = nv_global_scale_fast(gs);
      if (threadIdx.x < 128) sh.lut[threadIdx.x] = nv_division(threadIdx.x, rg, nv_fast);
    }
    // RMSNorm: the octets' sums of squares of all rows, added by every wave in row_inv_rms_kernel's order
    float row_rs[kFewNormRows] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (XPRO == kFewNorm) {
#pragma unroll
      for (int p = 0; p < kPasses; ++p) {
        if (p * 64 + lane < chunks) {
          float s[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float e[8];
            unpack8(xr[p][i], e);
            s[i] = e[0] * e[0];
#pragma unroll
            for (int k = 1; k < 8; ++k) s[i] = s[i] + e[k] * e[k];
          }
          // (A 24-bit product.  The 64-bit multiply-add that the compiler takes otherwise reads a register pair whose upper half
          // it had given to a weight scale on its way: the wave waited for all its weights here.  us, a token's norm with q, k
          // and v / gate and up: 7.8 / 16.6 -> 7.1 / 15.5; 7.0 / 15.0 with other code around it, by whose chance
          // the pair was free.)
          *(v4f*)&sh.octets[(__umul24(at[p] >> 16, in.xk) + col[p]) / 8] = v4f{s[0], s[1], s[2], s[3]};
        }
      }
    }
    if constexpr (XPRO == kFewSilu) {
#pragma unroll
      for (int i = 0; i < kTableLoads; ++i) {
        const uint32_t at4 = threadIdx.x + 64 * NW * i;
        if (at4 < 2u * kSiluLdsCount / 4u)
          *(float4*)&sh.silu[4 * at4] = make_float4(bf16_lo(table[i].x), bf16_hi(table[i].x), bf16_lo(table[i].y), bf16_hi(table[i].y));
      }
    }
    // (the weights' loads stay in flight: a barrier for LDS only)
    if constexpr (NV || XPRO != kFewPlain) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (XPRO == kFewNorm) {
      const int cpr = in.xk / 8;
      const float cols_f = (float)in.xk;
#pragma unroll
      for (int r = 0; r < kFewNormRows; ++r) {
        if (r >= M) break;   // (uniform)
        float a = 0.0f;
        for (int c0 = 0; c0 < cpr; c0 += 512) {   // eight reads at a time (adding zero is adding nothing: a >= 0)
          float t[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) t[i] = c0 + 64 * i + lane < cpr ? sh.octets[r * cpr + c0 + 64 * i + lane] : 0.0f;
#pragma unroll
          for (int i = 0; i < 8; ++i) a = a + t[i];
        }
        // the butterfly a += a[lane ^ m], m = 1, 2, ..., 32 (mirrors are lane ^ 4 and ^ 8 once a quad's lanes agree)
        auto dpp = [](float v, auto ctrl) __attribute__((always_inline)) {
          return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v), decltype(ctrl)::value, 0xF, 0xF, true));
        };
        a = a + dpp(a, std::integral_constant<int, 0xB1>{});    // quad_perm [1,0,3,2]
        a = a + dpp(a, std::integral_constant<int, 0x4E>{});    // quad_perm [2,3,0,1]
        a = a + dpp(a, std::integral_constant<int, 0x141>{});   // row_half_mirror
        a = a + dpp(a, std::integral_constant<int, 0x140>{});   // row_mirror
        a = a + __shfl_xor(a, 16, 64);
        a = a + __shfl_xor(a, 32, 64);
        row_rs[r] = 1.0f / __builtin_sqrtf(a / cols_f + in.eps);
      }
    }
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      if (p * 64 < chunks) {   // (wave-uniform)
        const int few_r = at[p] >> 16;
        const float rs = few_r == 0 ? row_rs[0] : few_r == 1 ? row_rs[1] : few_r == 2 ? row_rs[2] : row_rs[3];
        auto load_rotate = [&](float (&v)[32]) __attribute__((always_inline)) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float e[8];
            unpack8(xr[p][i], e);
            if constexpr (XPRO == kFewNorm) {
              float q[8];
              unpack8(ur[p][i], q);
#pragma unroll
              for (int k = 0; k < 8; k += 2) {
                const uint32_t t = pack_bf16x2(e[k] * rs, e[k + 1] * rs);
                const uint32_t pr = pack_bf16x2(bf16_lo(t) * q[k], bf16_hi(t) * q[k + 1]);
                e[k] = bf16_lo(pr);
                e[k + 1] = bf16_hi(pr);
              }
            }
            if constexpr (XPRO == kFewSilu) {
              float q[8];
              unpack8(ur[p][i], q);
              const uint32_t w[4] = {xr[p][i].x, xr[p][i].y, xr[p][i].z, xr[p][i].w};
              silu_lookup(w, e, (lds_f32*)sh.silu, in.silu, p * 64 + lane < chunks);
#pragma unroll
              for (int k = 0; k < 8; k += 2) {
                const uint32_t pr = pack_bf16x2(e[k] * q[k], e[k + 1] * q[k + 1]);
                e[k] = bf16_lo(pr);
                e[k + 1] = bf16_hi(pr);
              }
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) v[8 * i + k] = e[k];
          }
          rotate_chunk<32, XG, XROT, false>(v, in.norm, lane);
        };
        float v[32];
        load_rotate(v);
        uint32_t cw[4], sbytes = 0u, sb_lo = 0u;
        bool need_slow = chunk_not_finite<32>(v);
        need_slow |= quantize_chunk<32, FMT, kZeroReference, false>(v, gs, nv_fast, sh.lut, cw, sbytes, sb_lo);
        if (__builtin_amdgcn_ballot_w64(need_slow) != 0ull) {
          float u[32];
          load_rotate(u);
          quantize_chunk_slow<32, FMT, kZeroReference, true>(u, gs, rg, cw, sbytes);
        }
        if (col[p] >= in.xk) {
          cw[0] = cw[1] = cw[2] = cw[3] = 0u;
          sbytes = 0u;
        }
        const int ci = p * 64 + lane, g8 = ci & 7;
        if (ci < chunks) {
          const uint4 c4 = make_uint4(cw[0], cw[1], cw[2], cw[3]);
          *(uint4*)&sh.codes[wave][ci * 16] = c4;
          const int sc = (ci & ~7) + (g8 & 1) * 4 + (g8 >> 1);
          if constexpr (NV) *(uint16_t*)&sh.scales[wave][sc * 2] = (uint16_t)sbytes;
          else sh.scales[wave][sc] = (uint8_t)sbytes;
          if (hand_on) {
            const int row = at[p] >> 16, kb = at[p] & 0xffff, slot = (g8 & 1) * 32 + row;
            *(uint4*)(in.codes + ((size_t)(kb * 4 + (g8 >> 1)) * 64 + slot) * 16) = c4;
            if constexpr (NV) *(uint16_t*)(in.scales + (size_t)kb * 512 + slot * 8 + 2 * (g8 >> 1)) = (uint16_t)sbytes;
            else in.scales[(size_t)kb * 256 + slot * 4 + (g8 >> 1)] = (uint8_t)sbytes;
          }
        }
      }
    }
    asm volatile("" ::: "memory");   // (a wave's LDS accesses complete in order: its chunks are there when it reads them)
  }
};

}  // namespace fpq
