// Weight-streaming FP4 GEMM on packed operands for at most 128 activation rows (MXFP4; NVFP4 with the
// operands dequantized in registers to exact fp16, as in the NVFP4 tile kernel).
//
// With so few rows the time is the one pass over the weights (31 MB for the Llama-3-8B up/gate
// projection: 3.9 us at 8 TB/s), so the kernel is built around bytes in flight, not around tiles:
//   * a workgroup owns one 32-row weight tile (up to four: stream_plan) and a range of K; nothing is staged through LDS:
//     in the packed layout one operand of one 32x32x64 matrix instruction is one contiguous
//     kilobyte, lane by lane, so a wave loads it straight into the registers the instruction reads;
//   * the four waves take the 256-K blocks of the range in turn (wave w: blocks w, w + 4, ...) and
//     every wave issues the loads of up to DB blocks before its first matrix instruction, so for
//     K = 4096 and 32 rows the whole weight tile is requested at once;
//   * activations (at most four 32-row tiles, padded rows are zero) are re-read by every workgroup
//     and come from the L2;
//   * the four partial tiles meet in LDS and are summed in the fixed order (w0 + w2) + (w1 + w3), every
//     wave a quarter of each tile; the rounded tile goes through LDS once more so that a store writes 64
//     contiguous bytes per row, and the four waves share the stores.
// Shapes with few weight tiles (N = 4096: 128 workgroups for 256 CUs) or long K also split K
// ACROSS workgroups: each stores its fp32 partial tile into a workspace, a per-tile counter tells
// the last one to arrive, and that one adds the partials of all splits in split order (its own
// included, read back from the workspace), so the result does not depend on the arrival order.
// Counters are left at zero for the next launch.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

#include "../../include/fpq.h"
#include "fpq_device.h"
#include "fpq_few_rows.h"
#include "fpq_gemm_epilogue.h"

namespace fpq {

constexpr int kStreamCounters = 4096;                        // one per weight tile group
constexpr int64_t kStreamCounterBytes = kStreamCounters * 4;  // they open the workspace
constexpr int kStreamMaxRows = 128;

// Dynamic LDS of a workgroup with more than four output tiles (0: the kernel's own arrays hold them)
constexpr int stream_dynamic_lds(int nt, int mt) {
  return nt * mt > 4 ? 4 * nt * mt * 3 * 64 * 16 + nt * mt * 32 * 20 * 4 : 0;
}

// NT weight row tiles per workgroup, MT activation row tiles (exactly ceil(M / 32)), DB 256-K blocks
// of loads in flight per wave, NW waves.  Every workgroup re-reads all activations (NT = 2 halves
// that, at a register cost that stream_plan explains).  Two weight tiles per workgroup are compiled for
// two workgroups per CU (at most 256 registers).
//
// What bounds it.  A CU takes in about 60 bytes per nanosecond of a mix of weights from HBM and activations from the L2,
// whatever number of loads a wave has outstanding (one or two blocks per wave, measured the same): they complete in order,
// so an activation that the L2 would serve at once waits behind a weight, and some 64 KB are under way at a time (the
// activations and weights of 512 x 4096 x 14336 take 26 us with the matrix instructions left out and 14 us the other way
// round).  So the time follows the kilobytes that a workgroup loads per K step, NT + MT, as long as one round of the
// CUs holds all workgroups; and MXFP4 with several weight tiles per workgroup (kUnits) streams K step by K step: a step's
// registers are asked for again, one load behind each matrix instruction of the step after it, and not a whole block
// at a time, which left the matrix pipes idle while the loads went out.  us, weights from HBM, block by block with one
// weight tile per workgroup or two (or the tile kernels) / step by step: 64 x 14336 x 4096 11.2 / 10.3, 64 x 24576 x 4096
// 15.8 / 13.0, 96 x 14336 x 4096 13.4 / 11.8, 32 x 28672 x 4096 15.2 / 12.9.
// NV: NVFP4 operands (two E4M3 scale bytes per lane and K step, 512-byte scale blocks): a lane's dword s
// of a 64-K unit, times its group's scale, is its fp16 operand of the s-th 32x32x16 matrix instruction
// of the unit on both sides, so the K order is permuted consistently and the sum is complete.
//
// IN = FewRows: the activations come as bf16 rows (few of them) and every wave rotates and quantizes the 256-K blocks it
// multiplies, while its weights are on their way.  See few_rows_plan.
// IN = PackedSlabs: more than 32 MT activation rows in slabs of that many.  Dispatch goes round the XCDs workgroup by
// workgroup: in a grid of 8 x slabs x eighths of the groups of weight tiles the slabs (blockIdx.y) of a group
// (8 blockIdx.z + blockIdx.x) run on one XCD at about the same time, and all but one find the weights in its L2.
// IN = PackedSlabsInARow: where that grid would give an XCD more workgroups than CUs (groups rounded up to eights), every XCD
// takes a row of the workgroups numbered slab by slab within a group: most groups are still one XCD's.  Slabs by a grid of
// groups x slabs, on eight XCDs, / this (two weight tiles per workgroup; us, weights from HBM): 400 x 3200 x 4096 11.5 / 9.7,
// 280 x 5400 x 10240 22.5 / 18.7, 1100 x 700 x 4096 11.2 / 8.9, 500 x 2688 x 14336 28.8 / 23.9.
// IN = RowMajor: both operands as the quantize operators write them, codes [rows, k / 2] and scales [rows, stride] with the
// strides multiples of four.  A lane takes the same 16 bytes of codes of a row, and the same scale bytes, as from the
// packed layout, so the sums are the same bit for bit; only the addresses differ.  See launch_rows.
// RAGGED: k is no multiple of 256 (but one of 32).  The last block's groups past k read the row's start and are replaced.
template <bool RAGGED>
struct RowMajor {
  int k;
  uint32_t xs_stride, ws_stride;
};

template <int NT, int MT, int DB, int NW, bool NV = false, class IN = Packed, int XG = 32, int XROT = FPQ_ROT_IDENTITY,
          int XPRO = kFewPlain>
__global__ __launch_bounds__(64 * NW, NT == 2 && NT * MT <= 4 ? 2 : 1) void gemm_fp4_stream_kernel(
    const uint8_t* __restrict__ xq_all, const uint8_t* __restrict__ xs_all, const uint8_t* __restrict__ wq,
    const uint8_t* __restrict__ ws, const float* __restrict__ alpha_p, const uint16_t* __restrict__ bias,
    const uint16_t* residual_all, uint16_t* y, int M_all, int N, int K, int bps, int ksplit,
    float* partial, unsigned* counters, const OutSegments seg, const IN in) {
  constexpr bool kFew = std::is_same_v<IN, FewRows>;
  constexpr bool kRagged = std::is_same_v<IN, RowMajor<true>>, kRow = kRagged || std::is_same_v<IN, RowMajor<false>>;
  constexpr bool kSlabsInARow = std::is_same_v<IN, PackedSlabsInARow>, kSlabs = kSlabsInARow || std::is_same_v<IN, PackedSlabs>;
  static_assert(!kFew || MT == 1, "few rows: one activation tile");
  // The arguments lie in four cache lines, and none of them is near when a kernel starts: what the rows and the weights are asked
  // for with comes from all four at once.  Left alone, the compiler asks for the weights' addresses behind the rows (us, a
  // line later / at once, weights from HBM, rows not handed on: 1 x 4096 x 4096 5.7 / 5.5, 1 x 6144 x 4096 6.1 / 5.9, 1 x 14336 x
  // 4096 8.0 / 7.7; handed on 5.6 / 5.6, 6.0 / 6.0, 8.0 / 7.9).  With a norm or SiLU*up, whose rows take longer than the line,
  // and with two weight tiles a token's block measured 0.2 slower that way.
  if constexpr (kFew && XPRO == kFewPlain && NT == 1)
    asm volatile("" :: "s"(wq), "s"(ws), "s"(M_all), "s"(N), "s"(K), "s"(bps), "s"(in.x), "s"(in.up), "s"(in.xk));
  constexpr bool kUnits = !NV && NT >= 2;   // K step by K step (see above)
  static_assert(NW == 4, "a wave owns a quarter of every tile");
  // Slabs of 32 MT rows, each a product of its own (the last may have fewer rows, even fewer row tiles).
  int slab = kSlabs ? blockIdx.y : 0, rtg = kSlabs ? blockIdx.z * 8 + blockIdx.x : blockIdx.x;
  if constexpr (kSlabsInARow) {
    const unsigned slabs = (unsigned)(M_all + MT * 32 - 1) / (MT * 32), each = gridDim.x >> 3, xcd = blockIdx.x & 7;
    const unsigned at = xcd * each + min(xcd, gridDim.x & 7) + (blockIdx.x >> 3);   // (the first XCDs have one more)
    rtg = at / slabs;
    slab = at - rtg * slabs;
  }
  const int m0 = slab * (MT * 32), split = kSlabs ? 0 : blockIdx.y;
  const int M = min(M_all - m0, MT * 32);
  const uint8_t* xq = xq_all + (size_t)slab * MT * (K >> 6) * 1024;
  const uint8_t* xs = xs_all + (size_t)slab * MT * (K >> 8) * (NV ? 512 : 256);
  const uint16_t* residual = residual_all ? residual_all + (size_t)m0 * N : nullptr;
  const int tile_id = rtg;   // numbers the output tile groups for the K split (slabs never come with one)
  constexpr int kStageRow = 20;             // dwords: 16 of a row's 32 bf16 + 4, rows stay 16-byte aligned
  constexpr int kStageTile = 32 * kStageRow;
  // part: [owning wave][tile][the other waves in order][lane]; stage: the rounded tiles on their way out.  More
  // than four tiles per workgroup need more than the 64 KB a kernel may declare: those take them from the
  // launch's dynamic LDS.
  typedef v4f PartOf[NT * MT][3][64];
  typedef uint32_t StageOf[kStageTile];
  constexpr bool kDynLds = stream_dynamic_lds(NT, MT) > 0;
  __shared__ v4f part_fixed[kDynLds ? 1 : 4][kDynLds ? 1 : NT * MT][3][64];
  __shared__ __attribute__((aligned(16))) uint32_t stage_fixed[kDynLds ? 1 : NT * MT][kStageTile];
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_dynamic[];
  PartOf* const part = kDynLds ? (PartOf*)lds_dynamic : (PartOf*)part_fixed;
  StageOf* const stage = kDynLds ? (StageOf*)(lds_dynamic + 4 * sizeof(PartOf)) : (StageOf*)stage_fixed;
  __shared__ unsigned arrival;
  constexpr int kSB = NV ? 512 : 256;    // scale bytes per row tile and 256-K block
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nu = K >> 6, nkb = K >> 8;
  const float alpha = *alpha_p;   // asked for now: the epilogue, on the critical path of every workgroup, finds it there
  const int rt_n = (N + 31) >> 5;
  const int kb_begin = split * bps, kb_end = min(nkb, kb_begin + bps);
  const int first = kb_begin + wave;                                   // this wave: first, first + NW, ...
  // (Slabs: the groups of weight tiles may be rounded up to eights.  The ones past the last have no blocks and store nothing;
  // a return at the top would have every workgroup wait for N before it asks for its other arguments, 0.2 us.)
  const bool exists = !kSlabs || rtg * (NT * 32) < N;
  const int nblk = kb_end > first && exists ? (kb_end - first + NW - 1) / NW : 0;

  // A weight tile past the last one (odd tile count, NT = 2) re-reads the last: nothing of it is stored.
  const uint8_t* wcode[NT];
  const uint8_t* wscale[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int rt = min(rtg * NT + i, rt_n - 1);
    if constexpr (kRow) {
      const int row = min(rt * 32 + (lane & 31), N - 1);
      wcode[i] = wq + (size_t)row * (in.k >> 1) + (lane >> 5) * 16;
      wscale[i] = ws + (size_t)row * in.ws_stride;
      continue;
    }
    wcode[i] = wq + (size_t)rt * nu * 1024 + lane * 16;
    wscale[i] = ws + (size_t)rt * nkb * kSB + lane * (kSB / 64);
  }
  // Lanes whose activation row lies past M read what the lane of row 0 in their K half reads: no further
  // cache line is touched for rows that are never stored.  A row tile past the last one (a short last
  // slab) re-reads the last: the operand ends there.
  const uint8_t* xcode[MT];
  const uint8_t* xscale[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    if constexpr (kFew) break;
    if constexpr (kRow) {
      const int row = 32 * j + (lane & 31) < M ? 32 * j + (lane & 31) : 0;
      xcode[j] = xq_all + (size_t)row * (in.k >> 1) + (lane >> 5) * 16;
      xscale[j] = xs_all + (size_t)row * in.xs_stride;
      continue;
    }
    const int l = (lane & 31) < M - 32 * j ? lane : (lane & 32);
    const int jt = min(j, (M - 1) >> 5);
    xcode[j] = xq + (size_t)jt * nu * 1024 + l * 16;
    xscale[j] = xs + (size_t)jt * nkb * kSB + l * (kSB / 64);
  }

  v16f acc[NT * MT];
#pragma unroll
  for (int j = 0; j < NT * MT; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;

  // A ring of DB blocks in registers.  Every load is unconditional (a block index past the wave's
  // last one is clamped to it and its matrix instructions are skipped): with loads under branches
  // the compiler can no longer count which of them are still in flight and waits for all.
  uint4 a[DB][4][NT], b[DB][4][MT];
  uint2 sa[DB][NT], sb[DB][MT];   // MXFP4 uses .x only
  // Row-major: a row's scale bytes of a block as they lie (MXFP4: .x and .y), of which run_block takes the lane's
  uint4 sa_row[kRow ? DB : 1][NT], sb_row[kRow ? DB : 1][MT];
  int tail_steps = 4;   // K steps of the last block in which this lane has a group
  if constexpr (kRagged) tail_steps = ((in.k >> 5) - (nkb - 1) * 8 - (lane >> 5) + 1) >> 1;
  auto row_scales = [&](const uint8_t* row, int kb, uint32_t stride) __attribute__((always_inline)) {
    typedef uint32_t v2u_4 __attribute__((ext_vector_type(2), aligned(4)));
    typedef uint32_t v4u_4 __attribute__((ext_vector_type(4), aligned(4)));
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if constexpr (kRagged) {   // dword by dword: the last ones of the block may lie past the row
      const uint32_t last = stride - 4, at = (uint32_t)kb * (NV ? 16 : 8);
      v.x = *(const uint32_t*)(row + min(at, last));
      v.y = *(const uint32_t*)(row + min(at + 4, last));
      if constexpr (NV) {
        v.z = *(const uint32_t*)(row + min(at + 8, last));
        v.w = *(const uint32_t*)(row + min(at + 12, last));
      }
    } else if constexpr (NV) {
      const v4u_4 d = *(const v4u_4*)(row + (size_t)kb * 16);
      v = make_uint4(d.x, d.y, d.z, d.w);
    } else {
      const v2u_4 d = *(const v2u_4*)(row + (size_t)kb * 8);
      v.x = d.x;
      v.y = d.y;
    }
    return v;
  };
  auto row_offset = [&](int kb, int u) __attribute__((always_inline)) {   // of the lane's codes of K step u
    if constexpr (kRagged) return kb < nkb - 1 || u < tail_steps ? kb * 128 + u * 32 : -(lane >> 5) * 16;
    else return kb * 128 + u * 32;
  };
  const int t_last = nblk > 0 ? nblk - 1 : 0;
  auto load_weights = [&](const uint8_t* from) __attribute__((always_inline)) {
    const v4u_s ld = __builtin_nontemporal_load((const v4u_s*)from);
    return make_uint4(ld.x, ld.y, ld.z, ld.w);
  };
  // (the lambdas must be inlined whatever their size: a call would pin the register arrays they capture
  // to memory)
  auto load_block = [&](auto slot, int t) __attribute__((always_inline)) {
    constexpr int s = decltype(slot)::value;
    const int kb = min(first + NW * min(t, t_last), nkb - 1);
    if constexpr (kRow) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
#pragma unroll
        for (int u = 0; u < 4; ++u) a[s][u][i] = *(const uint4*)(wcode[i] + row_offset(kb, u));
        sa_row[s][i] = row_scales(wscale[i], kb, in.ws_stride);
      }
#pragma unroll
      for (int j = 0; j < MT; ++j) {
#pragma unroll
        for (int u = 0; u < 4; ++u) b[s][u][j] = *(const uint4*)(xcode[j] + row_offset(kb, u));
        sb_row[s][j] = row_scales(xscale[j], kb, in.xs_stride);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[s][u][i] = load_weights(wcode[i] + (size_t)(kb * 4 + u) * 1024);
      }
      if constexpr (NV) sa[s][i] = *(const uint2*)(wscale[i] + (size_t)kb * kSB);
      else sa[s][i].x = *(const uint32_t*)(wscale[i] + (size_t)kb * kSB);
    }
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      if constexpr (kFew) break;
#pragma unroll
      for (int u = 0; u < 4; ++u) b[s][u][j] = *(const uint4*)(xcode[j] + (size_t)(kb * 4 + u) * 1024);
      if constexpr (NV) sb[s][j] = *(const uint2*)(xscale[j] + (size_t)kb * kSB);
      else sb[s][j].x = *(const uint32_t*)(xscale[j] + (size_t)kb * kSB);
    }
  };
  // NVFP4: activation row tiles whose fp16 operands are held at a time (four tiles: two and two, the
  // weight operand is converted once more; all four at once left the register file)
  constexpr int kJB = (MT == 4) ? 2 : MT;
  auto scale_f16 = [](uint32_t d, int byte) __attribute__((always_inline)) {
    if constexpr (kRow) return e4m3_signed_f16(d, byte);
    else return e4m3_byte_f16(d, byte);
  };
  auto compute_block = [&](auto slot) __attribute__((always_inline)) {
    constexpr int s = decltype(slot)::value;
#define FPQ_STREAM_STEP(U)                                                                              \
  if constexpr (NV) {                                                                                   \
    _Pragma("unroll") for (int j0 = 0; j0 < MT; j0 += kJB) {                                            \
      v8h bh[kJB][4];                                                                                   \
      _Pragma("unroll") for (int j = 0; j < kJB; ++j) {                                                 \
        const uint4 bq = b[s][U][j0 + j];                                                               \
        const uint32_t bw[4] = {bq.x, bq.y, bq.z, bq.w};                                                \
        const uint32_t bsc = (U) < 2 ? sb[s][j0 + j].x : sb[s][j0 + j].y;                               \
        const _Float16 bsh[2] = {scale_f16(bsc, 2 * ((U) & 1)), scale_f16(bsc, 2 * ((U) & 1) + 1)};           \
        _Pragma("unroll") for (int s4 = 0; s4 < 4; ++s4)                                                \
          bh[j][s4] = dequant8_f16_h(bw[s4], bsh[s4 >> 1]);                                             \
      }                                                                                                 \
      _Pragma("unroll") for (int i = 0; i < NT; ++i) {                                                  \
        const uint4 aq = a[s][U][i];                                                                    \
        const uint32_t aw[4] = {aq.x, aq.y, aq.z, aq.w};                                                \
        const uint32_t asc = (U) < 2 ? sa[s][i].x : sa[s][i].y;                                         \
        const _Float16 ash[2] = {scale_f16(asc, 2 * ((U) & 1)), scale_f16(asc, 2 * ((U) & 1) + 1)};           \
        _Pragma("unroll") for (int s4 = 0; s4 < 4; ++s4) {                                              \
          const v8h ah = dequant8_f16_h(aw[s4], ash[s4 >> 1]);                                          \
          _Pragma("unroll") for (int j = 0; j < kJB; ++j)                                               \
            acc[i * MT + j0 + j] =                                                                      \
                __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh[j][s4], acc[i * MT + j0 + j], 0, 0, 0);   \
        }                                                                                               \
      }                                                                                                 \
    }                                                                                                   \
  } else {                                                                                              \
    _Pragma("unroll") for (int i = 0; i < NT; ++i) {                                                    \
      const uint4 aq = a[s][U][i];                                                                      \
      const v8i av = v8i{(int)aq.x, (int)aq.y, (int)aq.z, (int)aq.w, 0, 0, 0, 0};                       \
      _Pragma("unroll") for (int j = 0; j < MT; ++j) {                                                  \
        const uint4 bq = b[s][U][j];                                                                    \
        const v8i bv = v8i{(int)bq.x, (int)bq.y, (int)bq.z, (int)bq.w, 0, 0, 0, 0};                     \
        acc[i * MT + j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(                              \
            av, bv, acc[i * MT + j], 4, 4, U, (int)sa[s][i].x, U, (int)sb[s][j].x);                     \
      }                                                                                                 \
    }                                                                                                   \
  }
    FPQ_STREAM_STEP(0)
    FPQ_STREAM_STEP(1)
    FPQ_STREAM_STEP(2)
    FPQ_STREAM_STEP(3)
#undef FPQ_STREAM_STEP
  };
  // NVFP4 with three activation row tiles: the 16 K steps of a block (one 32x32x16 matrix instruction per output
  // tile each) as a software pipeline -- while the matrix instructions of step t issue, the operands of step
  // t + 1 are converted, and the instruction order is pinned to one matrix instruction followed by its share of
  // the conversions.  Only a step's operands are held as fp16 (32 registers, not the 48 of a whole unit's
  // activations), which brings the kernel under 256 registers: two workgroups per CU, whose waves fill each
  // other's gaps (a wave alone on its SIMD issues a conversion every 8 cycles, measured).  96 rows, K = 4096,
  // weights from HBM: N = 14336 22.5 -> 20.5 us, N = 24576 33.7 -> 28.9, N = 28672 44.7 -> 36.0.  One, two and
  // four row tiles measured the same or up to 5 % slower this way and keep the unit-by-unit order above.
  constexpr bool kPipelined = NV && MT == 3;
  auto a_op = [&](auto slot, int t, int i) __attribute__((always_inline)) {
    constexpr int s = decltype(slot)::value;
    const int U = t >> 2, s4 = t & 3;
    const uint4 q = a[s][U][i];
    const uint32_t cd = s4 == 0 ? q.x : s4 == 1 ? q.y : s4 == 2 ? q.z : q.w;
    return dequant8_f16_h(cd, e4m3_byte_f16(U < 2 ? sa[s][i].x : sa[s][i].y, 2 * (U & 1) + (s4 >> 1)));
  };
  auto b_op = [&](auto slot, int t, int j) __attribute__((always_inline)) {
    constexpr int s = decltype(slot)::value;
    const int U = t >> 2, s4 = t & 3;
    const uint4 q = b[s][U][j];
    const uint32_t cd = s4 == 0 ? q.x : s4 == 1 ? q.y : s4 == 2 ? q.z : q.w;
    return dequant8_f16_h(cd, e4m3_byte_f16(U < 2 ? sb[s][j].x : sb[s][j].y, 2 * (U & 1) + (s4 >> 1)));
  };
  auto compute_block_nv = [&](auto slot) __attribute__((always_inline)) {
    v8h ah[NT], bh[MT];
#pragma unroll
    for (int i = 0; i < NT; ++i) ah[i] = a_op(slot, 0, i);
#pragma unroll
    for (int j = 0; j < MT; ++j) bh[j] = b_op(slot, 0, j);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      v8h an[NT], bn[MT];
      if (t < 15) {
#pragma unroll
        for (int i = 0; i < NT; ++i) an[i] = a_op(slot, t + 1, i);
#pragma unroll
        for (int j = 0; j < MT; ++j) bn[j] = b_op(slot, t + 1, j);
      }
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[i * MT + j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], bh[j], acc[i * MT + j], 0, 0, 0);
      constexpr int kValu = ((NT + MT) * 9 + NT * MT - 1) / (NT * MT);   // 8 conversions + the scale's share, per operand
#pragma unroll
      for (int m = 0; m < NT * MT; ++m) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (t < 15) {
#pragma unroll
        for (int i = 0; i < NT; ++i) ah[i] = an[i];
#pragma unroll
        for (int j = 0; j < MT; ++j) bh[j] = bn[j];
      }
    }
  };
  // (lanes past the last row read row 0's chunks, as above)
  typedef std::conditional_t<kFew, typename FewChunks<NV, XG, XROT, XPRO, NW>::Shared, Packed> FewShared;
  __shared__ __attribute__((aligned(16))) FewShared few_shared;
  const int few_row = (lane & 31) < M ? (lane & 31) * nblk : 0;   // first block of the lane's row
  auto run_block = [&](auto slot, int t) __attribute__((always_inline)) {
    if constexpr (kFew) {
      constexpr int s = decltype(slot)::value;
      const int blk = few_row + t, kh = lane >> 5;
#pragma unroll
      for (int u = 0; u < 4; ++u) b[s][u][0] = *(const uint4*)&few_shared.codes[wave][(blk * 8 + 2 * u + kh) * 16];
      if constexpr (NV) sb[s][0] = *(const uint2*)&few_shared.scales[wave][blk * 16 + kh * 8];
      else sb[s][0].x = *(const uint32_t*)&few_shared.scales[wave][blk * 8 + kh * 4];
    }
    if constexpr (kRow) {
      constexpr int s = decltype(slot)::value;
      const int kh = lane >> 5;
      const uint32_t sel = NV ? (kh ? 0x07060302u : 0x05040100u) : (kh ? 0x07050301u : 0x06040200u);
      auto take = [&](const uint4& v) __attribute__((always_inline)) {
        return make_uint2(__builtin_amdgcn_perm(v.y, v.x, sel), NV ? __builtin_amdgcn_perm(v.w, v.z, sel) : 0u);
      };
#pragma unroll
      for (int i = 0; i < NT; ++i) sa[s][i] = take(sa_row[s][i]);
#pragma unroll
      for (int j = 0; j < MT; ++j) sb[s][j] = take(sb_row[s][j]);
      if (kRagged && first + NW * t == nkb - 1) {
        // Past k: zero codes on the activations' side, and scale bytes that are no NaN on both (an E8M0 0xff beyond the
        // end would make NaN of them; the E4M3 bytes are taken as finite whatever they are).
        const uint32_t keep = tail_steps >= 4 ? 0xffffffffu : (1u << (8 * tail_steps)) - 1u;
#pragma unroll
        for (int i = 0; i < NT; ++i)
          if constexpr (!NV) sa[s][i].x &= keep;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          if constexpr (!NV) sb[s][j].x &= keep;
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (u >= tail_steps) b[s][u][j] = make_uint4(0u, 0u, 0u, 0u);
        }
      }
    }
    if constexpr (kPipelined) compute_block_nv(slot);
    else compute_block(slot);
  };
  auto for_slots = [&](auto&& f) __attribute__((always_inline)) {
    f(std::integral_constant<int, 0>{});
    if constexpr (DB > 1) f(std::integral_constant<int, 1>{});
    if constexpr (DB > 2) f(std::integral_constant<int, 2>{});
    if constexpr (DB > 3) f(std::integral_constant<int, 3>{});
  };
  static_assert(DB >= 1 && DB <= 4, "at most four blocks in flight");

  // With a ring of two or more blocks the loads of a slot and the matrix instructions of the next must stay
  // in program order: left alone, the instruction scheduler groups the loads of all slots (weights first,
  // then scales and activations), and since loads complete in order the wait for one slot's last operand
  // then covers the other slots' weights as well -- the ring degenerates into load everything, wait for
  // everything, compute everything (M = 1, N = 14336: 8.4 against 7.8 us from HBM; it also takes 40 registers
  // more).  With three or four activation row tiles the effect is within +-4 % either way; only four tiles
  // of NVFP4 gain throughout (128 rows, N = 4096: 15.1 -> 14.6 us).  One block in flight has nothing to order.
  constexpr bool kOrdered = NT == 1 && DB >= 2 && (MT <= 2 || (NV && MT == 4));
  // K step by K step (kUnits): the steps of the blocks in flight are a ring of 4 DB steps in a[] and b[].  While the matrix
  // instructions of a step issue, the step before it is asked for again, 4 DB - 1 steps ahead; a block's scales go with its
  // first step and are taken into registers of their own when the block begins.  Few rows: theirs come from LDS then.
  constexpr int kLoads = NT + (kFew ? 0 : MT);     // operands loaded per step: the weights' first
  uint32_t now_a[NT], now_b[MT];
  auto block_at = [&](int t) __attribute__((always_inline)) { return min(first + NW * min(t, t_last), nkb - 1); };
  auto load_operand = [&](auto slot, int u, int l, int kb) __attribute__((always_inline)) {
    constexpr int s = decltype(slot)::value;
    const size_t at = (size_t)(kb * 4 + u) * 1024;
    if (l < NT) a[s][u][l] = load_weights(wcode[l] + at);
    else b[s][u][l - NT] = *(const uint4*)(xcode[l - NT] + at);
  };
  auto load_scale = [&](auto slot, int l, int kb) __attribute__((always_inline)) {
    constexpr int s = decltype(slot)::value;
    if (l < NT) sa[s][l].x = *(const uint32_t*)(wscale[l] + (size_t)kb * kSB);
    else sb[s][l - NT].x = *(const uint32_t*)(xscale[l - NT] + (size_t)kb * kSB);
  };
  // Block t of the wave; the first ASK of its steps ask for one further ahead (which has to exist: the last blocks ask for less)
  auto run_units = [&](auto slot, int t, auto ask) __attribute__((always_inline)) {
    constexpr int s = decltype(slot)::value, ASK = decltype(ask)::value;
    if constexpr (kFew) {
      const int blk = few_row + t, kh = lane >> 5;
#pragma unroll
      for (int u = 0; u < 4; ++u) b[s][u][0] = *(const uint4*)&few_shared.codes[wave][(blk * 8 + 2 * u + kh) * 16];
      now_b[0] = *(const uint32_t*)&few_shared.scales[wave][blk * 8 + kh * 4];
    }
    // (moves that the compiler may not turn into copies at the end of the loop, where it would wait for every load)
#pragma unroll
    for (int l = 0; l < kLoads; ++l) {
      if (l < NT) asm volatile("v_mov_b32 %0, %1" : "=v"(now_a[l]) : "v"(sa[s][l].x));
      else asm volatile("v_mov_b32 %0, %1" : "=v"(now_b[l - NT]) : "v"(sb[s][l - NT].x));
    }
    wait_states_before_mfma([&](auto&& pass) __attribute__((always_inline)) {
#pragma unroll
      for (int l = 0; l < kLoads; ++l) pass(l < NT ? now_a[l] : now_b[l - NT]);
    });
    const int kb_before = block_at(t - 1 + DB), kb_next = block_at(t + DB);
    auto step = [&](auto step_u) __attribute__((always_inline)) {   // (which byte of the scales an instruction takes is a constant)
      constexpr int U = decltype(step_u)::value;
#pragma unroll
      for (int p = 0; p < NT * MT; ++p) {
        const int i = p / MT, j = p % MT;
        const uint4 aq = a[s][U][i], bq = b[s][U][j];
        acc[p] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            v8i{(int)aq.x, (int)aq.y, (int)aq.z, (int)aq.w, 0, 0, 0, 0}, v8i{(int)bq.x, (int)bq.y, (int)bq.z, (int)bq.w, 0, 0, 0, 0},
            acc[p], 4, 4, U, (int)now_a[i], U, (int)now_b[j]);
        if constexpr (U < ASK) {
#pragma unroll
          for (int l = p * kLoads / (NT * MT); l < (p + 1) * kLoads / (NT * MT); ++l) {
            if constexpr (U == 0) {
              load_operand(std::integral_constant<int, (s + DB - 1) % DB>{}, 3, l, kb_before);
            } else {
              if constexpr (U == 1) load_scale(slot, l, kb_next);
              load_operand(slot, U - 1, l, kb_next);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
  };
  FewChunks<NV, XG, XROT, XPRO, NW> few;
  if constexpr (kFew) few.load(in, M, first, nblk, lane);
  for_slots([&](auto slot) {
    if constexpr (kUnits) {
      constexpr int s = decltype(slot)::value;
      const int kb = block_at(s);
#pragma unroll
      for (int l = 0; l < kLoads; ++l) load_scale(slot, l, kb);
#pragma unroll
      for (int u = 0; u < (s == DB - 1 ? 3 : 4); ++u) {
#pragma unroll
        for (int l = 0; l < kLoads; ++l) load_operand(slot, u, l, kb);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      load_block(slot, decltype(slot)::value);
      if constexpr (kOrdered || kFew) __builtin_amdgcn_sched_barrier(0);
    }
  });
  if constexpr (kFew) few.quantize(in, M, few_shared, wave, lane, in.codes && blockIdx.x == 0);
  // Where the epilogue will store, worked out while the first loads are in flight (after the reduction
  // every instruction delays the workgroup's end).  The epilogue's lane layout: 8 consecutive columns
  // (16 bytes) of row lane / 4 and of that row + 16.  16-byte accesses need the whole tile inside N and
  // aligned rows and bases (a residual never comes with segments: one output, its rows N long).
  const int row16 = lane >> 2, c = lane & 3;
  int res_rows = __builtin_amdgcn_readfirstlane(residual && (N & 7) == 0 && ((uintptr_t)residual & 15) == 0);
  const uint16_t* res_src = residual + (size_t)row16 * N + rtg * NT * 32 + 8 * c;
  uint16_t* out_dst[NT];
  int out_ld[NT], out_whole[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int tn0 = (rtg * NT + i) * 32;
    const OutView out = out_view(seg, y, nullptr, tn0, N);   // the matrix this tile's columns go to (unused past N)
    out_ld[i] = __builtin_amdgcn_readfirstlane(out.N);
    out_dst[i] = out.y + (size_t)(m0 + row16) * out.N + out.n0 + 8 * c;
    out_whole[i] = __builtin_amdgcn_readfirstlane(tn0 + 32 <= N && (out.N & 7) == 0 && ((uintptr_t)out.y & 15) == 0 &&
                                                  (!residual || res_rows));
    // (values the compiler may not look through: it would otherwise move their computation, kernel
    // argument loads included, to their first use behind the reduction)
    if constexpr (NT == 1) asm volatile("" : "+s"(out_ld[i]), "+s"(out_whole[i]), "+v"(out_dst[i]));
  }
  if constexpr (NT == 1) asm volatile("" : "+s"(res_rows), "+v"(res_src));
  int t0 = 0;
  if constexpr (kUnits) {
    static_assert(DB <= 2, "one or two blocks of K steps in flight");
    typedef std::integral_constant<int, 0> S0;
    typedef std::integral_constant<int, DB - 1> S1;
    typedef std::integral_constant<int, 1> Ask1;   // (the step that completes the ring)
    typedef std::integral_constant<int, 4> Ask4;
    for (; t0 + 2 * DB <= nblk; t0 += DB)
      for_slots([&](auto slot) { run_units(slot, t0 + decltype(slot)::value, Ask4{}); });
    if constexpr (DB == 1) {
      if (t0 < nblk) run_units(S0{}, t0, Ask1{});
    } else {
      if (nblk - t0 == 3) {
        run_units(S0{}, t0, Ask4{});
        run_units(S1{}, t0 + 1, Ask1{});
        run_units(S0{}, t0 + 2, std::integral_constant<int, 0>{});
      } else if (nblk - t0 == 2) {
        run_units(S0{}, t0, Ask1{});
        run_units(S1{}, t0 + 1, std::integral_constant<int, 0>{});
      } else if (nblk - t0 == 1) {
        run_units(S0{}, t0, std::integral_constant<int, 0>{});
      }
    }
    t0 = nblk;
  }
  for (; !kUnits && t0 + 2 * DB <= nblk; t0 += DB) {   // steady state: the block DB ahead exists
    for_slots([&](auto slot) {
      run_block(slot, t0 + decltype(slot)::value);
      if constexpr (kOrdered) __builtin_amdgcn_sched_barrier(0);
      load_block(slot, t0 + DB + decltype(slot)::value);
      if constexpr (kOrdered) __builtin_amdgcn_sched_barrier(0);
    });
  }
  if constexpr (!kUnits) for_slots([&](auto slot) {   // the ring's last full or partial content
    if (t0 + decltype(slot)::value < nblk) run_block(slot, t0 + decltype(slot)::value);
    if constexpr (kOrdered) __builtin_amdgcn_sched_barrier(0);
  });
  if (!kUnits && nblk - t0 > DB) {          // up to DB - 1 blocks more
    for_slots([&](auto slot) { load_block(slot, t0 + DB + decltype(slot)::value); });
    for_slots([&](auto slot) {
      if (t0 + DB + decltype(slot)::value < nblk) run_block(slot, t0 + DB + decltype(slot)::value);
    });
  }

  // ---- the four K parts of the workgroup, summed in the fixed order (w0 + w2) + (w1 + w3).
  // Whatever follows the last matrix instruction delays the workgroup's end, so all four waves share it:
  // wave g owns quarter g of every tile (registers 4g .. 4g + 3: columns 8g .. 8g + 7), gets that
  // quarter from the three others through LDS and carries it through the rest of the kernel.
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    if (g == wave) continue;
    const int from = wave < g ? wave : wave - 1;
#pragma unroll
    for (int t = 0; t < NT * MT; ++t)
      part[g][t][from][lane] = v4f{acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]};
  }
  // The rows of the residual this wave will add are asked for now: they arrive during the reduction.
  // (Store pass 2 t + p -- rows 16 p .. 16 p + 15 of tile t -- belongs to wave (2 t + p) % 4.)
  uint4 rv[(2 * NT * MT + 3) / 4];
  if (res_rows) {
#pragma unroll
    for (int pass = 0; pass < 2 * NT * MT; ++pass) {
      if ((pass & 3) != wave) continue;
      const int i = (pass >> 1) / MT, j = (pass >> 1) % MT, p = pass & 1;
      const int m = j * 32 + 16 * p + row16, n = (rtg * NT + i) * 32 + 8 * c;
      rv[pass >> 2] = m < M && n < N ? *(const uint4*)(res_src + (size_t)(j * 32 + 16 * p) * N + 32 * i)
                                     : make_uint4(0, 0, 0, 0);
    }
  }
  __syncthreads();
  v4f sum[NT * MT];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    if (g != wave) continue;
#pragma unroll
    for (int t = 0; t < NT * MT; ++t) {
      v4f k[4];   // the quarter as each wave computed it
#pragma unroll
      for (int w = 0; w < 4; ++w)
        k[w] = w == g ? v4f{acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]}
                      : part[g][t][w < g ? w : w - 1][lane];
#pragma unroll
      for (int q = 0; q < 4; ++q) sum[t][q] = (k[0][q] + k[2][q]) + (k[1][q] + k[3][q]);
    }
  }

  // ---- K split across workgroups: partial tiles through the workspace, last arrival finishes
  if (ksplit > 1) {
    // The parts of a tile run on different XCDs, whose L2 caches are not coherent with each other
    // for ordinary accesses.  Device-scope fences would write back and invalidate whole caches
    // (measured: 55 us for a 6 us kernel); instead every access to the workspace is a relaxed
    // device-scope atomic, which the hardware performs at the point all XCDs agree on, and every
    // wave waits for its stores to be acknowledged before the workgroup moves the counter.
    constexpr int kTile = NT * MT * 16 * 64;  // floats per partial: register v of tile t at (16 t + v) * 64 + lane
    float* mine = partial + ((size_t)tile_id * ksplit + split) * kTile + wave * 256 + lane;
#pragma unroll
    for (int t = 0; t < NT * MT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        __hip_atomic_store(mine + (t * 16 + q) * 64, sum[t][q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // (ksplit is the same for the whole grid: every wave of the workgroup is here)
    // One arrival per workgroup: a counter that every wave moved made the exchange 1.5 us slower (its
    // updates from different XCDs are served one after the other).
    if (threadIdx.x == 0)
      arrival = __hip_atomic_fetch_add(counters + tile_id, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    // (one value for the workgroup: all its waves leave or all stay for the barrier further down)
    if (__builtin_amdgcn_readfirstlane(arrival) != (unsigned)(ksplit - 1)) return;
    const float* all = partial + (size_t)tile_id * ksplit * kTile + wave * 256 + lane;
    for (int s = 0; s < ksplit; ++s) {
#pragma unroll
      for (int t = 0; t < NT * MT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float p = __hip_atomic_load(all + (size_t)s * kTile + (t * 16 + q) * 64, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
          sum[t][q] = s == 0 ? p : sum[t][q] + p;
        }
    }
    if (threadIdx.x == 0) __hip_atomic_store(counters + tile_id, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // ---- y[m][n] = bf16(alpha * sum) (+ bias) (+ residual, a further bf16 add): element q of this wave's
  // quarter of tile (i, j) is m = 32 j + lane % 32, n = 32 (NT rtg + i) + 8 wave + 4 (lane / 32) + q.
  // Stored from there, an instruction would write 16 bytes into each of 32 rows; so many small pieces
  // cost 5-8 % of the whole kernel (M = 16, N = 14336: 8.0 -> 7.6 us; M = 64: 11.3 -> 10.4 us).  The
  // rounded tile goes through LDS instead and comes back with a lane holding 8 consecutive columns: 64
  // contiguous bytes per row and store.
  const int r32 = lane & 31, kh = lane >> 5;
  uint32_t* lane_stage = &stage[0][r32 * kStageRow + 4 * wave + 2 * kh];
  if (!bias) {   // (a code path of its own rather than a select after the additions)
#pragma unroll
    for (int t = 0; t < NT * MT; ++t)
      *(uint2*)(lane_stage + t * kStageTile) = make_uint2(pack_bf16x2(sum[t][0] * alpha, sum[t][1] * alpha),
                                                          pack_bf16x2(sum[t][2] * alpha, sum[t][3] * alpha));
  } else {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int n = (rtg * NT + i) * 32 + 8 * wave + 4 * kh;   // bias is indexed by the product's column
      float bv[4];   // (columns past N are not stored: no branch around a load)
#pragma unroll
      for (int q = 0; q < 4; ++q) bv[q] = __uint_as_float((uint32_t)bias[min(n + q, N - 1)] << 16);
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const v4f& t = sum[i * MT + j];
        const uint32_t lo = pack_bf16x2(t[0] * alpha, t[1] * alpha), hi = pack_bf16x2(t[2] * alpha, t[3] * alpha);
        *(uint2*)(lane_stage + (i * MT + j) * kStageTile) =
            make_uint2(pack_bf16x2(__uint_as_float(lo << 16) + bv[0], __uint_as_float(lo & 0xffff0000u) + bv[1]),
                       pack_bf16x2(__uint_as_float(hi << 16) + bv[2], __uint_as_float(hi & 0xffff0000u) + bv[3]));
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < 2 * NT * MT; ++pass) {
    if ((pass & 3) != wave) continue;
    const int i = (pass >> 1) / MT, j = (pass >> 1) % MT, p = pass & 1;
    const int n = (rtg * NT + i) * 32 + 8 * c, m = j * 32 + 16 * p + row16;
    if (m >= M || n >= N) continue;
    const uint4 v = *(const uint4*)&stage[pass >> 1][(16 * p + row16) * kStageRow + 4 * c];
    uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint16_t* dst = out_dst[i] + (size_t)(j * 32 + 16 * p) * out_ld[i];
    if (out_whole[i]) {   // the same for every lane
      if (residual) {
        const uint32_t r[4] = {rv[pass >> 2].x, rv[pass >> 2].y, rv[pass >> 2].z, rv[pass >> 2].w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
          w[q] = pack_bf16x2(__uint_as_float(w[q] << 16) + __uint_as_float(r[q] << 16),
                             __uint_as_float(w[q] & 0xffff0000u) + __uint_as_float(r[q] & 0xffff0000u));
      }
      *(uint4*)dst = make_uint4(w[0], w[1], w[2], w[3]);
      continue;
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {   // N's last tile, or an unaligned output: element by element
      if (n + q >= N) continue;
      uint32_t h = (w[q >> 1] >> (16 * (q & 1))) & 0xffffu;
      if (residual)
        h = pack_bf16x2(__uint_as_float(h << 16) + __uint_as_float((uint32_t)residual[(size_t)m * N + n + q] << 16), 0.0f) & 0xffffu;
      dst[q] = (uint16_t)h;
    }
  }
}

struct StreamPlan {
  bool use;    // false: the tile kernels of fpq_gemm_packed.hip serve the shape better
  int nt;      // weight row tiles per workgroup
  int ksplit;  // K parts (workgroups per group of weight tiles)
  int bps;     // 256-K blocks per part
};

// Which shapes run here and how (all thresholds are measured break-even points on Llama-3-8B and
// Qwen3-8B layer shapes).  Up to 64 activation rows: always.  More
// rows: up to a number of weight tiles beyond which the 128x128 tile kernel, which shares activations
// through LDS, is faster -- 65-96 rows: 512 tiles for MXFP4, one round of this kernel's workgroups (with the
// weights from HBM, this kernel against the tiles: N = 14336 12.0 / 12.3 us, N = 16384 12.5 / 12.5, N = 18432
// 15.6 / 14.3, N = 24576 17.1 / 15.3, N = 28672 20.7 / 16.5, N = 32768 21.9 / 18.0), any number for NVFP4 (N = 14336: 22.1
// against 35.9 us, N = 128256: 165 against 215); 97-128 rows (276-346 registers, one workgroup per
// CU): one round of the 256 CUs for both formats (NVFP4 took two until its tile kernels ran eight waves per
// workgroup: N = 8192 15.0 against 22.9 us for the tiles, N = 10240 26.7 against 22.7, N = 16384 27.7 against 23.9).  (One tile per workgroup with two blocks in flight, two workgroups per CU, is the
// better one for NVFP4 at 33-64 rows -- except from 384 weight tiles on, where two tiles per workgroup with ONE block in
// flight, held to 256 registers, share the activations' conversion to fp16: N = 28672 26.2 -> 22.6 us, N = 57344 45.6 ->
// 40.8, 1-4 % up to 767 tiles.  MXFP4: see below.)
// K is split across workgroups when the weight tiles leave at least half of the CUs idle and every
// part keeps at least 4096 of K (the exchange of partial tiles through the workspace costs about as
// much as streaming 16 blocks); fewer parts if the workspace is small.  (While one wave did the
// exchange alone the split paid for at most 32 rows; shared by the four waves it pays at every row
// count: N = 4096, K = 14336: 64 rows 14.4 -> 11.7 us, 128 rows 19.8 -> 15.4 us, NVFP4 39.0 -> 24.6 us.)
static StreamPlan stream_plan(int64_t M, int64_t N, int64_t K, int64_t workspace_bytes, bool nv = false) {
  StreamPlan plan{false, 1, 1, 0};
  if (M < 1 || M > kStreamMaxRows || N < 1 || K < 256 || K % 256 != 0) return plan;
  const int64_t rt_m = (M + 31) / 32, tiles = (N + 31) / 32, nkb = K / 256;
  // (weight-tile counts in units of the device's compute units: 256 on the part the figures above were measured on)
  const int64_t cus = device_cus();
  if (rt_m == 3 && !nv && tiles > 2 * cus) return plan;
  if (rt_m == 4 && tiles > cus) return plan;
  plan.use = true;
  // MXFP4: as many weight tiles per workgroup as bring the workgroups into one round of the CUs, up to four.  A second
  // round, full or not, costs its start and its end, and all activations once more per weight tile (us, weights from HBM,
  // K = 4096, one tile per workgroup, from 768 tiles at 33-64 rows two / this: 32 rows: N = 10240 8.5 / 7.6, N = 14336 9.5 /
  // 8.6, N = 28672 15.2 / 12.9; 64 rows: N = 10240 10.5 / 9.1, N = 16384 12.3 / 10.6, N = 20480 15.0 / 12.0, N = 24576
  // 15.8 / 13.0, N = 28672 16.7 / 15.3; 96 rows: N = 10240 12.2 / 10.7, N = 16384 13.6 / 12.3).
  // Not where one tile per workgroup fills its rounds to the last sixteenth, its waves have whole pairs of blocks, as many as
  // they keep in flight, and up to 16 rows (24 in place of four tiles) leave few activations to load again (one tile / this: 16 x
  // 24576 x 8192 18.0 / 19.1, 5 x 32768 x 4096 13.3 / 14.4; 24 x 24576 x 8192 18.9 / 19.2; 5 x 15360 x 5120 9.7 / 8.8); nor four in place
  // of a single pair (8 x 28672 x 2048 8.2 / 8.7), nor three for a single block (5 x 16640 x 256 4.8 / 5.1).  33-64 rows: two instead of four for a short K, with two workgroups to a CU (four / two: 64 x
  // 24832 x 1024 7.7 / 6.7, 33 x 32768 x 2048 11.1 / 10.1, 64 x 30720 x 3072 12.9 / 12.6).
  if (!nv && tiles > cus && tiles <= 4 * cus) {
    plan.nt = (int)((tiles + cus - 1) / cus);
    if (rt_m == 2 && plan.nt == 4 && K <= 3072) plan.nt = 2;
    if (M <= (plan.nt == 4 ? 24 : 16) && nkb % 8 == 0 && (16 * tiles >= 15 * plan.nt * cus || (plan.nt == 4 && nkb == 8)))
      plan.nt = 1;
    if (rt_m == 1 && plan.nt == 3 && nkb == 1) plan.nt = 1;
  } else if (rt_m == 2 && tiles >= (nv ? 3 * cus / 2 : 3 * cus)) plan.nt = 2;
  // NVFP4, 33-64 rows, between two and three weight tiles per CU: three per workgroup, one workgroup per CU in
  // a single round instead of a round and a half of pairs (N = 24576: K = 4096 22.2 -> 21.2 us, K = 12288 56.0 ->
  // 48.0; N = 20480 21.0 -> 19.7; four tiles per workgroup for the next range measured 4 % slower than pairs).
  // With one workgroup per CU anyway it keeps two blocks in flight per wave (N = 24576: 20.9 -> 20.1 us, K = 12288
  // 48.2 -> 45.2; N = 20480 19.8 -> 18.8; three measured 15-20 % slower).
  if (nv && rt_m == 2 && tiles > 2 * cus && tiles <= 3 * cus) plan.nt = 3;
  const int64_t groups = (tiles + plan.nt - 1) / plan.nt;
  int64_t ksplit = 1;
  if (workspace_bytes > kStreamCounterBytes && groups <= kStreamCounters) {
    ksplit = cus / groups;
    if (ksplit > nkb / 16) ksplit = nkb / 16;
    if (ksplit < 1) ksplit = 1;
    while (ksplit > 1 && kStreamCounterBytes + ksplit * groups * plan.nt * rt_m * 4096 > workspace_bytes) --ksplit;
  }
  const int64_t bps = (nkb + ksplit - 1) / ksplit;
  plan.ksplit = (int)((nkb + bps - 1) / bps);  // no empty part
  plan.bps = (int)bps;
  return plan;
}

bool stream_eligible(bool nv, int64_t M, int64_t N, int64_t K) { return stream_plan(M, N, K, 0, nv).use; }

int64_t gemm_mxf4_stream_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  const StreamPlan plan = stream_plan(M, N, K, (int64_t)1 << 62);
  if (!plan.use || plan.ksplit <= 1) return 0;
  const int64_t groups = ((N + 31) / 32 + plan.nt - 1) / plan.nt;
  return kStreamCounterBytes + (int64_t)plan.ksplit * groups * plan.nt * ((M + 31) / 32) * 4096;
}

// Arguments are validated by the caller (gemm_packed); `workspace` is null or 256-byte aligned with
// its first kStreamCounterBytes zero.  NV: NVFP4 operands.  slab_rows > 0 (a multiple of 32, at most 128):
// M exceeds what one workgroup takes and is cut into slabs of that many rows, slab_nt weight tiles per workgroup, K whole.
template <bool NV>
static int launch_stream(const void* xq, const void* xs, const void* wq, const void* ws, const float* alpha,
                         const void* bias, const void* residual, void* y, int64_t M, int64_t N, int64_t K,
                         void* workspace, int64_t workspace_bytes, const OutSegments& seg, hipStream_t stream,
                         int64_t slab_rows = 0, int slab_nt = 1) {
  if (slab_rows) workspace = nullptr;
  const int64_t rows = slab_rows ? slab_rows : M;   // what one workgroup sees
  StreamPlan plan = stream_plan(rows, N, K, workspace ? workspace_bytes : 0, NV);
  if (!plan.use) return FPQ_E_UNSUPPORTED;
  if (slab_rows) plan.nt = slab_nt;
  const unsigned groups = (unsigned)(((N + 31) / 32 + plan.nt - 1) / plan.nt);
  const unsigned slabs = (unsigned)(slab_rows ? (M + slab_rows - 1) / slab_rows : 1);
  // Slabs: eights of groups unless that gives an XCD more workgroups than CUs, two on one of them; then in a row.  A multiple of
  // four groups has each on two XCDs at most in a grid of groups x slabs, which measured the same or better (us, that / in a row:
  // 590 x 2304 x 10240 17.8 / 18.4, 1300 x 768 x 10240 14.9 / 15.8), and the weights of few groups are little to share.
  // MXFP4 with one tile and up to one block per wave: not eights either that are half empty or more, whose workgroups without a
  // tile cost 0.2 to 0.5 (eights / groups x slabs: 34 x 2112 x 512 4.6 / 4.2, 84 x 128 x 256 4.2 / 4.0, 132 x 3336 x 768 5.8 / 5.5; 100 x 1470 x
  // 1024, 46 groups, 4.7 / 5.1; 34 x 2112 x 1280 4.7 / 4.8; NVFP4 level).
  const bool half_empty = !NV && plan.nt == 1 && K <= 1024 && groups % 8 >= 1 && groups % 8 <= 4;
  const bool eights = !half_empty && 8u * ((groups + 7) / 8) * slabs <= (unsigned)device_cus();
  const bool in_a_row = !NV && slab_rows && plan.nt == 2 && !eights && groups > 8 && groups % 4 != 0;
  const dim3 grid = !slab_rows ? dim3(groups, (unsigned)plan.ksplit)
                    : eights   ? dim3(8, slabs, (groups + 7) / 8)
                    : in_a_row ? dim3(groups * slabs) : dim3(groups, slabs);
  unsigned* counters = (unsigned*)workspace;
  float* partial = workspace ? (float*)((uint8_t*)workspace + kStreamCounterBytes) : nullptr;
  auto go = [&](auto nt, auto mt, auto db, auto in) {
    constexpr int NT = decltype(nt)::value, MT = decltype(mt)::value, DB = decltype(db)::value;
    constexpr int kLds = stream_dynamic_lds(NT, MT);
    constexpr auto kernel = &gemm_fp4_stream_kernel<NT, MT, DB, 4, NV, decltype(in)>;
    if constexpr (kLds > 0) {
      static LdsLimitOnce lds_limit;
      if (const int st = lds_limit.ensure((const void*)kernel, kLds)) return st;
    }
    hipLaunchKernelGGL(kernel, grid, dim3(256), kLds, stream, (const uint8_t*)xq, (const uint8_t*)xs, (const uint8_t*)wq,
                       (const uint8_t*)ws, alpha, (const uint16_t*)bias, (const uint16_t*)residual, (uint16_t*)y, (int)M,
                       (int)N, (int)K, plan.bps, plan.ksplit, partial, counters, seg, in);
    return (int)hipGetLastError();
  };
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 3> I3;
  typedef std::integral_constant<int, 4> I4;
  const int mt = (int)((rows + 31) / 32);
  // enough workgroups for three per CU: two blocks in flight per wave beat four by 3-5 %; with fewer
  // workgroups the deeper ring of each wave is what keeps the memory system busy
  const bool many = (int64_t)groups * plan.ksplit * slabs >= 3 * device_cus() / 2;
  // (65-128 rows: one block in flight per wave, which fits two workgroups into a CU, measured 1-2 %
  // slower for MXFP4 and 6-12 % slower for NVFP4 than two blocks -- 96 rows of NVFP4, N = 4096:
  // K = 4096 12.4 against 11.5 us, K = 14336 33.7 against 29.5 us)
  if (slab_rows) {
    if (plan.nt == 1) {
      if (mt == 1) return many ? go(I1{}, I1{}, I2{}, PackedSlabs{}) : go(I1{}, I1{}, I4{}, PackedSlabs{});
      if (mt == 2) return go(I1{}, I2{}, I2{}, PackedSlabs{});
      if (mt == 3) return go(I1{}, I3{}, I2{}, PackedSlabs{});
      if (mt == 4) return go(I1{}, I4{}, I2{}, PackedSlabs{});
    }
    if constexpr (!NV) {
      auto go_slabs = [&](auto mt_c) { return in_a_row ? go(I2{}, mt_c, I1{}, PackedSlabsInARow{}) : go(I2{}, mt_c, I1{}, PackedSlabs{}); };
      if (plan.nt == 2 && mt == 2) return go_slabs(I2{});
      if (plan.nt == 2 && mt == 3) return go_slabs(I3{});
      if (plan.nt == 2 && mt == 4) return go_slabs(I4{});
    }
    return FPQ_E_UNSUPPORTED;
  }
  if (plan.nt == 1) {
    if (mt == 1) return many ? go(I1{}, I1{}, I2{}, Packed{}) : go(I1{}, I1{}, I4{}, Packed{});
    if (mt == 2) return go(I1{}, I2{}, I2{}, Packed{});
    if (mt == 3) return go(I1{}, I3{}, I2{}, Packed{});
    return go(I1{}, I4{}, I2{}, Packed{});
  }
  if constexpr (NV) {   // 33-64 rows
    if (mt != 2) return FPQ_E_UNSUPPORTED;
    if (plan.nt == 3) return go(I3{}, I2{}, I2{}, Packed{});
    return go(I2{}, I2{}, I1{}, Packed{});
  } else {
    if (plan.nt == 2) {
      if (mt == 1) return go(I2{}, I1{}, I2{}, Packed{});
      return mt == 2 ? go(I2{}, I2{}, I1{}, Packed{}) : mt == 3 ? go(I2{}, I3{}, I1{}, Packed{}) : (int)FPQ_E_UNSUPPORTED;
    }
    if (plan.nt == 3)
      return mt == 1 ? go(I3{}, I1{}, I2{}, Packed{}) : mt == 2 ? go(I3{}, I2{}, I1{}, Packed{}) : (int)FPQ_E_UNSUPPORTED;
    return mt == 1 ? go(I4{}, I1{}, I1{}, Packed{}) : mt == 2 ? go(I4{}, I2{}, I1{}, Packed{}) : (int)FPQ_E_UNSUPPORTED;
  }
}

int gemm_fp4_stream(bool nv, const void* xq, const void* xs, const void* wq, const void* ws, const float* alpha,
                    const void* bias, const void* residual, void* y, int64_t M, int64_t N, int64_t K,
                    void* workspace, int64_t workspace_bytes, const OutSegments& seg, hipStream_t stream) {
  return nv ? launch_stream<true>(xq, xs, wq, ws, alpha, bias, residual, y, M, N, K, workspace, workspace_bytes, seg,
                                  stream)
            : launch_stream<false>(xq, xs, wq, ws, alpha, bias, residual, y, M, N, K, workspace, workspace_bytes, seg,
                                   stream);
}

// M rows in slabs of slab_rows (a multiple of 32 for which stream_eligible holds), all in one launch; nt weight tiles per
// workgroup (NVFP4: one).
int gemm_fp4_stream_slabs(bool nv, const void* xq, const void* xs, const void* wq, const void* ws,
                          const float* alpha, const void* bias, const void* residual, void* y, int64_t M, int64_t N,
                          int64_t K, int64_t slab_rows, int nt, const OutSegments& seg, hipStream_t stream) {
  if (slab_rows < 32 || slab_rows > kStreamMaxRows || slab_rows % 32 != 0 || M <= slab_rows) return FPQ_E_UNSUPPORTED;
  return nv ? launch_stream<true>(xq, xs, wq, ws, alpha, bias, residual, y, M, N, K, nullptr, 0, seg, stream, slab_rows, nt)
            : launch_stream<false>(xq, xs, wq, ws, alpha, bias, residual, y, M, N, K, nullptr, 0, seg, stream, slab_rows, nt);
}


// At most 64 activation rows, both operands row-major (the GEMM operators): the kernel above on rows instead of packed
// blocks, without a K split across workgroups (there is no workspace).  An operand load touches the lines of 32 rows, 32
// bytes each, where a packed one reads a kilobyte end to end, and the texture path bounds it (about 38 cycles per load;
// NVFP4: the conversions, like the packed kernel's).  The kernels that it replaced took K in whole multiples of 2048 with
// every load of a wave's quarter ahead of its matrix instructions but none across them, any other K a step at a time
// (us, before / now, weights from HBM): NVFP4 64 x 6144 x 4096 15.7 / 11.1, 20 x 28672 x 14336 96 / 69, 4 x 23552 x 6656 62 /
// 23, 40 x 2440 x 6784 94 / 18; MXFP4 64 x 6144 x 4096 13.3 / 9.7, 32 x 4096 x 14336 22.6 / 16.7, 1 x 10240 x 8704 42.7 /
// 16.1, 64 x 4096 x 1280 12.9 / 4.9.  Two blocks in flight per wave; one where a wave has hardly two (below eight blocks:
// 64 x 4096 x 1280 4.9 against 5.6, 14 x 28672 x 1024 6.1 against 9.1; at eight, 64 x 28672 x 2048 16.5 against 15.9).
// Four, eight waves per workgroup, and two weight tiles per workgroup measured slower over most of the range.
constexpr int64_t kRowMajorMaxRows = 64;
template <bool NV>
static int launch_rows(const void* xq, const void* xs, int64_t xs_stride, const void* wq, const void* ws, int64_t ws_stride,
                       const float* alpha, const void* bias, void* y, int64_t M, int64_t N, int64_t K, hipStream_t stream) {
  const int64_t nkb = (K + 255) / 256, tiles = (N + 31) / 32;
  auto go = [&](auto ragged) {
    typedef RowMajor<decltype(ragged)::value> In;
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(256), 0, stream, (const uint8_t*)xq, (const uint8_t*)xs,
                         (const uint8_t*)wq, (const uint8_t*)ws, alpha, (const uint16_t*)bias, (const uint16_t*)nullptr,
                         (uint16_t*)y, (int)M, (int)N, (int)(nkb * 256), (int)nkb, 1, (float*)nullptr, (unsigned*)nullptr,
                         OutSegments{}, In{(int)K, (uint32_t)xs_stride, (uint32_t)ws_stride});
    };
    if (M > 32) nkb < 8 ? launch(gemm_fp4_stream_kernel<1, 2, 1, 4, NV, In>) : launch(gemm_fp4_stream_kernel<1, 2, 2, 4, NV, In>);
    else nkb < 8 ? launch(gemm_fp4_stream_kernel<1, 1, 1, 4, NV, In>) : launch(gemm_fp4_stream_kernel<1, 1, 2, 4, NV, In>);
    return (int)hipGetLastError();
  };
  return K % 256 != 0 ? go(std::true_type{}) : go(std::false_type{});
}

// Arguments are validated by the caller (fpq_gemm.hip); FPQ_E_UNSUPPORTED, with nothing launched: a shape or an alignment
// that this kernel does not take.
int gemm_fp4_rows(bool nv, const void* xq, const void* xs, int64_t xs_stride, const void* wq, const void* ws,
                  int64_t ws_stride, const float* alpha, const void* bias, void* y, int64_t M, int64_t N, int64_t K,
                  hipStream_t stream) {
  if (M > kRowMajorMaxRows || K % 32 != 0 || ((xs_stride | ws_stride) & 3) || (((uintptr_t)xs | (uintptr_t)ws) & 3u) ||
      xs_stride >= ((int64_t)1 << 31) || ws_stride >= ((int64_t)1 << 31))
    return FPQ_E_UNSUPPORTED;
  return nv ? launch_rows<true>(xq, xs, xs_stride, wq, ws, ws_stride, alpha, bias, y, M, N, K, stream)
            : launch_rows<false>(xq, xs, xs_stride, wq, ws, ws_stride, alpha, bias, y, M, N, K, stream);
}

// Few activation rows quantized by the GEMM itself.  A layer of one token is two kernels of about 4 us each, of which
// most is the start and the end of a kernel, and two launches of 3.3 us host time; here every workgroup repeats the
// quantization of the blocks it multiplies (each wave its own, no exchange between them) behind the loads of its
// weights, in the same arithmetic and with the same order of sums: the same bits as the two kernels.
//
// The vector work grows with rows x K and is repeated per weight tile, so it is taken for one or two passes of a
// wave's lanes over its 32-element chunks (rows x 256-K blocks of a wave <= 8 or 16) and, since it does not hide
// behind the loads once the workgroups fill the CUs over and over, up to a number of weight tiles.  Measured (us, two
// kernels / one; graph replays, weights in the last-level cache):
//   MXFP4 1 row:  4096 x 4096 7.1 / 4.8, N = 14336 10.2 / 6.3, N = 28672 14.8 / 12.2, N = 128256 44.4 / 42.1;
//                 K = 14336, N = 4096 11.6 / 9.2; 8192 x 8192 10.7 / 6.8
//   MXFP4 4 rows (two passes):  4096 x 4096 7.2 / 5.7, N = 14336 10.2 / 8.1, N = 28672 14.9 / 14.5, N = 128256 45.5 / 49.0
//   NVFP4 1 row:  4096 x 4096 9.4 / 7.2, N = 14336 12.6 / 9.8, N = 28672 19.6 / 17.9, N = 128256 59.8 / 65.3
//   NVFP4 4 rows: 4096 x 4096 9.4 / 8.2, N = 14336 12.5 / 11.5, N = 28672 19.5 / 19.9
// SiLU*up (two more lookups per element) gains in one pass only (weights from HBM, two passes built for it): MXFP4, N = 4096, K =
// 14336: 1 row 13.8 / 12.1, 2 rows (two passes) 13.9 / 13.7; K = 12288: 13.2 / 11.4, 13.3 / 13.6; K = 4096: 1 row 8.7 / 6.6, 2 rows
// 8.7 / 7.1, 4 rows (two) 8.8 / 9.2; NVFP4, K = 14336: 16.5 / 15.8, 16.7 / 17.8; K = 4096: 10.8 / 10.1, 4 rows 10.9 / 12.1.
static bool few_rows_plan(const StreamPlan& plan, bool nv, int pro, int64_t M, int64_t N, int64_t K, int64_t xk) {
  const int64_t chunks = M * ((plan.bps + 3) / 4) * 8;   // of the wave with the most
  if (!plan.use || (nv && plan.nt != 1) || M > 32 || chunks > few_rows_chunks(pro) || K >= ((int64_t)1 << 22) || xk > K) return false;
  const int64_t tiles = (N + 31) / 32, cus = device_cus();
  return chunks <= 64 ? !nv || tiles <= 4 * cus : tiles <= (nv ? 2 : 4) * cus;
}

int silu_table_address(hipStream_t stream, const uint16_t** out);   // fpq_quantize.hip

// (`plan`, and what it takes, are the caller's)
template <bool NV, int PRO>
static int launch_few_rows(const FewRows& in, const StreamPlan& plan, int rot_kind, int g, const void* wq, const void* ws,
                           const float* alpha, const void* bias, const void* residual, void* y, int64_t M, int64_t N, int64_t K,
                           void* workspace, const OutSegments& seg, hipStream_t stream) {
  if (rot_kind == FPQ_ROT_IDENTITY) g = 32;
  else if (rot_kind != FPQ_ROT_HADAMARD || in.xk % g != 0) return FPQ_E_UNSUPPORTED;
  // Two weight tiles per workgroup: the rows are quantized, and a norm's sums added up, half as often; the sums of the products
  // are those of any plan.nt.  There are no activations to load, so that it pays for the vector work alone: with three to four
  // weight tiles per CU, of which a CU holds three at a time; with two to three where a wave has two passes, of two rows
  // over up to five blocks or of three and more, or, in one pass for three to five blocks, a norm in front or blocks that the
  // waves do not share evenly.  us, one
  // / two tiles, weights from HBM: 1 row, K = 4096: N = 24832 12.2 / 12.1, N = 32768 14.5 / 13.7, N = 20480 10.5 / 11.5; N = 20480: 1 row,
  // K = 8192 16.8 / 18.8, K = 2560 9.2 / 8.7, 2 rows, K = 8192 17.5 / 18.4, 4 rows, K = 4096 11.4 / 10.9; with a norm, 1 row: N = 28672, K =
  // 4096 14.8 / 12.5, N = 24576, K = 4096 12.0 / 11.4, N = 20480: K = 2048 9.2 / 9.6, K = 3072 11.3 / 10.1, K = 6144 13.8 / 14.9.  Four tiles
  // measured as one does, and 448 tiles lose (1 x 14336 x 4096 8.2 / 8.7).  SiLU*up's projections have a hidden size of features,
  // too few for it.
  const int64_t nkb = K / 256, blocks = (nkb + 3) / 4, tiles = (N + 31) / 32, cus = device_cus();
  const bool three_to_five = blocks >= 3 && blocks <= 5;
  const bool pays = tiles > 3 * cus ? tiles <= 4 * cus
                                    : tiles > 2 * cus && (PRO == kFewNorm ? three_to_five
                                                          : (M * blocks > 8 && (M >= 3 || three_to_five)) ||
                                                            (three_to_five && nkb % 4 != 0));
  const int nt = !NV && PRO != kFewSilu && pays ? 2 : 1;
  const dim3 grid((unsigned)(((N + 31) / 32 + nt - 1) / nt), (unsigned)plan.ksplit);
  const bool many = (int64_t)grid.x * grid.y >= 3 * device_cus() / 2;   // (as launch_stream)
  unsigned* counters = (unsigned*)workspace;
  float* partial = workspace ? (float*)((uint8_t*)workspace + kStreamCounterBytes) : nullptr;
  auto go = [&](auto rows_g, auto rows_rot) {
    constexpr int G = decltype(rows_g)::value, ROT = decltype(rows_rot)::value;
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, nullptr, nullptr, (const uint8_t*)wq, (const uint8_t*)ws, alpha,
                         (const uint16_t*)bias, (const uint16_t*)residual, (uint16_t*)y, (int)M, (int)N, (int)K, plan.bps,
                         plan.ksplit, partial, counters, seg, in);
    };
    if constexpr (!NV && PRO != kFewSilu) {
      if (nt == 2) {
        launch(gemm_fp4_stream_kernel<2, 1, 2, 4, NV, FewRows, G, ROT, PRO>);
        return (int)hipGetLastError();
      }
    }
    if (many) launch(gemm_fp4_stream_kernel<1, 1, 2, 4, NV, FewRows, G, ROT, PRO>);
    else launch(gemm_fp4_stream_kernel<1, 1, 4, 4, NV, FewRows, G, ROT, PRO>);
    return (int)hipGetLastError();
  };
  typedef std::integral_constant<int, FPQ_ROT_HADAMARD> Had;
  if (rot_kind == FPQ_ROT_IDENTITY)
    return go(std::integral_constant<int, 32>{}, std::integral_constant<int, FPQ_ROT_IDENTITY>{});
  if constexpr (NV) {
    if (g == 16) return go(std::integral_constant<int, 16>{}, Had{});
  }
  if (g == 32) return go(std::integral_constant<int, 32>{}, Had{});
  if (g == 64) return go(std::integral_constant<int, 64>{}, Had{});
  if (g == 128) return go(std::integral_constant<int, 128>{}, Had{});
  return FPQ_E_UNSUPPORTED;
}

template <bool NV>
static int linear_rows(const FewRows& in, int rot_kind, int g, const void* wq, const void* ws, const float* alpha,
                       const void* bias, const void* residual, void* y, int64_t M, int64_t N, int64_t xk, void* workspace,
                       int64_t workspace_bytes, int zero_policy, hipStream_t stream) {
  const int64_t K = (xk + 255) / 256 * 256;
  if (M < 1 || N < 1 || xk < 256 || workspace_bytes < 0) return FPQ_E_SHAPE;
  if (!in.x || !wq || !ws || !alpha || !y || (NV && !in.gs)) return FPQ_E_NULL;
  if (xk % 32 != 0 || N > (1 << 24) || xk > (1 << 24)) return FPQ_E_SHAPE;
  if (((uintptr_t)wq & 15u) || ((uintptr_t)ws & 15u) || ((uintptr_t)y & 15u) || ((uintptr_t)residual & 15u) ||
      ((uintptr_t)workspace & 255u) || ((uintptr_t)in.codes & 15u) || ((uintptr_t)in.scales & 15u))
    return FPQ_E_ALIGN;
  if (((uintptr_t)in.x & 15u) || ((uintptr_t)in.up & 15u) || zero_policy != FPQ_ZERO_REFERENCE) return FPQ_E_UNSUPPORTED;
  if (!workspace) workspace_bytes = 0;
  // The plan that fpq_gemm_*_packed_splitk follows for these rows: the same parts of K, the same sums.
  const StreamPlan plan = stream_plan(M, N, K, workspace_bytes, NV);
  if (!few_rows_plan(plan, NV, in.up ? kFewSilu : kFewPlain, M, N, K, xk)) return FPQ_E_UNSUPPORTED;
  return in.up ? launch_few_rows<NV, kFewSilu>(in, plan, rot_kind, g, wq, ws, alpha, bias, residual, y, M, N, K, workspace,
                                               OutSegments{}, stream)
               : launch_few_rows<NV, kFewPlain>(in, plan, rot_kind, g, wq, ws, alpha, bias, residual, y, M, N, K, workspace,
                                                OutSegments{}, stream);
}

// RMSNorm in front of a group of projections, for a token or a few: one launch instead of the norm's (a workgroup per row,
// 4.7 us for any row) and the GEMM's.  Every workgroup has its rows' chunks in registers anyway; the octets' sums of squares
// go through LDS, each wave adds them up in row_inv_rms_kernel's order, and the normalised bf16 values stay in registers.
// (the by-product that the norm's own kernel writes is not written: for callers that need the projections only)
// K is whole (no split across workgroups: a row has to be in one workgroup), as for these rows in
// fpq_gemm_*_packed_multi: the same sums.
//
// Up to four rows, in one pass of a wave's lanes over its chunks (rows x 256-K blocks of a wave <= 8).  Measured (us, two
// kernels / one; graph replays, weights from HBM), the launch that a caller saves besides not counted:
//   MXFP4 1 row:  K = 4096, N = 6144 9.8 / 6.8, N = 28672 16.5 / 14.5; K = 1024, N = 1536 7.6 / 5.9
//   MXFP4 2 rows: 9.5 / 7.2, 16.6 / 15.7; 4 rows: K = 2048, N = 2560 8.5 / 7.2, N = 14336 9.5 / 9.4
//   NVFP4 1 row:  12.2 / 9.2, 21.8 / 20.6; 2 rows 11.8 / 9.7, 21.3 / 21.6; 4 rows: K = 2048 9.4 / 8.4
// Two passes (twice the registers for rows and weight) took 10.7 and 24.9 for 4 MXFP4 rows of K = 4096 (9.8, 16.8 in two kernels).
static bool norm_rows_plan(bool nv, int64_t M, int64_t N, int64_t K, StreamPlan& plan) {
  if (M > kFewNormRows || K > (1 << 20)) return false;
  plan = stream_plan(M, N, K, 0, nv);
  return few_rows_plan(plan, nv, kFewNorm, M, N, K, K);
}

template <bool NV>
static int norm_rows_multi(const FewRows& in, int rot_kind, int g, const void* wq, const void* ws, const float* alpha,
                           const void* bias, const OutSegments& seg, int64_t M, int64_t N, int64_t K, int zero_policy,
                           hipStream_t stream) {
  StreamPlan plan;
  if (zero_policy != FPQ_ZERO_REFERENCE || !norm_rows_plan(NV, M, N, K, plan)) return FPQ_E_UNSUPPORTED;
  return launch_few_rows<NV, kFewNorm>(in, plan, rot_kind, g, wq, ws, alpha, bias, nullptr, seg.y[0], M, N, K, nullptr, seg,
                                       stream);
}

// ---- the entry point that allocates nothing -------------------------------------------------------
// Counters and partial tiles of a split K live in this file-scope array instead of a caller-provided
// workspace.  Every GPU the library runs on holds its own copy at its own address until the process
// ends; the array's name is only a host-side handle, the device address comes from
// hipGetSymbolAddress, once per device, and that address is what kernels and host code use.
// A split needs at most 1024 partial tiles of 4 KB on a device of 256 compute units (stream_plan: parts x
// weight tiles <= compute units, times up to four activation row tiles).
constexpr int64_t kScratchBytes = kStreamCounterBytes + 1024 * 4096;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
static std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (looked up on the first call per device; two
// threads racing on that first call store the same address).
int scratch_address(void** out) {   // also called by fpq_prepare_device (fpq_capi.hip)
  int device = -1;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return (int)err;
  if (device < 0 || device >= kMaxDevices) return FPQ_E_UNSUPPORTED;
  void* ptr = g_scratch_ptr[device].load(std::memory_order_acquire);
  if (!ptr) {
    err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (err != hipSuccess) return (int)err;
    if (!ptr) return FPQ_E_UNSUPPORTED;
    g_scratch_ptr[device].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return FPQ_OK;
}

// fpq_gemm_packed.hip: argument checks and dispatch shared with fpq_gemm_mxf4_packed_splitk
int gemm_mxf4_packed_any(const void* xq, const void* xs, const void* wq, const void* ws, const float* alpha,
                         const void* bias, const void* residual, void* y, int64_t M, int64_t N, int64_t K,
                         void* workspace, int64_t workspace_bytes, void* stream);

}  // namespace fpq

extern "C" int64_t fpq_gemm_mxf4_packed_noalloc_max_rows(void) { return fpq::kStreamMaxRows; }

extern "C" int fpq_gemm_mxf4_packed_noalloc(const void* xq, const void* xs, const void* wq, const void* ws,
                                            const float* alpha, const void* bias, const void* residual,
                                            void* y, int64_t M, int64_t N, int64_t K, void* stream) {
  if (M > fpq::kStreamMaxRows) return FPQ_E_LIMIT;
  // (a shape that could use more than the array holds -- none on a device of 256 compute units -- splits K
  // into as many parts as fit: stream_plan sizes the split to the workspace it is given)
  void* ptr = nullptr;
  const int st = fpq::scratch_address(&ptr);
  if (st != FPQ_OK) return st;
  return fpq::gemm_mxf4_packed_any(xq, xs, wq, ws, alpha, bias, residual, y, M, N, K, ptr, fpq::kScratchBytes,
                                   stream);
}

// Test hook: the split-K counters at the head of the current device's scratch array (16 KB), copied to
// `out` (device memory) in stream order; they must read zero between calls.
extern "C" int fpq_test_noalloc_counters(void* out, int64_t bytes, void* stream) {
  if (!out) return FPQ_E_NULL;
  if (bytes < 0 || bytes > fpq::kStreamCounterBytes) return FPQ_E_SHAPE;
  void* ptr = nullptr;
  const int st = fpq::scratch_address(&ptr);
  if (st != FPQ_OK) return st;
  if (bytes == 0) return FPQ_OK;
  return (int)hipMemcpyAsync(out, ptr, (size_t)bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream);
}

extern "C" int fpq_linear_rows(int nv, const void* x, const void* up, int64_t M, int64_t K, int rot_kind, int g, float norm,
                               const float* global_scale, const void* wq, const void* ws, const float* alpha,
                               const void* bias, const void* residual, void* y, int64_t N, void* packed_codes,
                               void* packed_scales, void* workspace, int64_t workspace_bytes, int zero_policy,
                               void* stream) {
  fpq::FewRows in{(const uint4*)x, (const uint4*)up, nullptr, global_scale, (uint8_t*)packed_codes,
                  (uint8_t*)packed_scales, norm, (int)K, 0.0f};
  if (!packed_codes != !packed_scales) return FPQ_E_NULL;
  if (K < 0 || K > (1 << 24)) return FPQ_E_SHAPE;
  if (up) {
    if (const int st = fpq::silu_table_address((hipStream_t)stream, &in.silu)) return st;
  }
  return nv ? fpq::linear_rows<true>(in, rot_kind, g, wq, ws, alpha, bias, residual, y, M, N, K, workspace,
                                     workspace_bytes, zero_policy, (hipStream_t)stream)
            : fpq::linear_rows<false>(in, rot_kind, g, wq, ws, alpha, bias, residual, y, M, N, K, workspace,
                                      workspace_bytes, zero_policy, (hipStream_t)stream);
}

extern "C" int fpq_norm_rows_multi(int nv, const void* x, const void* norm_weight, float eps, int64_t M, int64_t K,
                                   int rot_kind, int g, float norm, const float* global_scale, const void* wq,
                                   const void* ws, const float* alpha, const void* bias, void* const* ys,
                                   const int64_t* ns, int64_t count, int zero_policy, void* stream) {
  if (count < 1 || count > fpq::kMaxSegments || M < 0 || K < 256 || K % 256 != 0 || K > (1 << 24)) return FPQ_E_SHAPE;
  if (M == 0) return FPQ_OK;
  if (!x || !norm_weight || !wq || !ws || !alpha || !ys || !ns || (nv && !global_scale)) return FPQ_E_NULL;
  if (((uintptr_t)x & 15u) || ((uintptr_t)norm_weight & 15u) || ((uintptr_t)wq & 15u) || ((uintptr_t)ws & 15u))
    return FPQ_E_ALIGN;
  fpq::OutSegments seg{};
  int64_t N = 0;
  for (int64_t i = 0; i < count; ++i) {   // (as fpq_gemm_*_packed_multi)
    if (ns[i] < 1 || ns[i] % fpq::kSegmentAlign != 0 || N + ns[i] > (1 << 24)) return FPQ_E_SHAPE;
    if (!ys[i]) return FPQ_E_NULL;
    if ((uintptr_t)ys[i] & 15u) return FPQ_E_ALIGN;
    N += ns[i];
    seg.end[i] = (int)N;
    seg.y[i] = (uint16_t*)ys[i];
  }
  seg.count = (int)count;
  const fpq::FewRows in{(const uint4*)x, (const uint4*)norm_weight, nullptr, global_scale, nullptr, nullptr, norm, (int)K, eps};
  return nv ? fpq::norm_rows_multi<true>(in, rot_kind, g, wq, ws, alpha, bias, seg, M, N, K, zero_policy, (hipStream_t)stream)
            : fpq::norm_rows_multi<false>(in, rot_kind, g, wq, ws, alpha, bias, seg, M, N, K, zero_policy, (hipStream_t)stream);
}

extern "C" int fpq_norm_rows_takes(int nv, int64_t M, int64_t N, int64_t K) {
  fpq::StreamPlan plan;
  return M > 0 && N > 0 && N <= (1 << 24) && fpq::norm_rows_plan(nv != 0, M, N, K, plan);
}
