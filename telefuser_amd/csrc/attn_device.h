// Shared by the attention kernels (attn.hip: FP8 P.V and the streaming forms; attn_half.hip: half P.V): the launch
// parameters, LDS DMA, the softmax and epilogue pieces, and the in-kernel Q quantizer.
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.h"

namespace qattn {

constexpr int kD = 128;
constexpr int kBQ = 128;  // query quantization block
constexpr int kWavesPerSimd = 2;  // occupancy target: 2 workgroups of 4 waves per CU
constexpr int kPrefetch = 2;      // K/V tiles in flight ahead of the one being computed
constexpr int kNBuf = kPrefetch + 1;
// k_scales staged in LDS per workgroup (floats).  Sized so that two workgroups per CU still fit in the
// 160 KiB of LDS next to the K/V buffers: 24 + 24 + 30 KiB.
constexpr int kKsLdsFloats = 7680;
// multi-block launches (one workgroup streams up to kMqMaxBlocks query blocks of one head through one
// K/V pipeline): short key ranges only, so their k_scales and q_scales are staged whole in LDS
constexpr int kMqMaxTiles = 64;
// the automatic rule picks multi-block launches below this many key tiles: from 32 tiles on the ping-pong
// kernel is 4-12 % faster (32760 x 2048 x 12, 8192 x 4096 x 16), at 12 and 16 tiles the two tie
constexpr int kMqAutoMaxTiles = 24;
constexpr int kMqMaxBlocks = 64;
// per-thread K scales: 4 per 64-key tile (one per mma lane-pair class), otherwise 1
constexpr int ks_per_tile(bool kt) { return kt ? 4 : 1; }
constexpr int kBK = 64;
constexpr int kThreads = 256;
constexpr float kFp8Offset = 8.807f;  // attn_utils.cuh:35 S_FP8_OFFSET
constexpr float kMInit = -3.0e38f;
// Lazy-rescale threshold (log2 units), see the softmax below.  After a move of the running max the largest p of
// the row is 448 / 2^kLazyTau.  Measured against 1 (C4, text cross attention over 512 keys: a few tiles per
// row, so the max moves on most of them at 1): 8 % faster at 3, RMS error against float64 truth 3.84 % ->
// 3.90 % (cosine 0.99926 -> 0.99924); C2 / C5 within 1 %, error unchanged.
constexpr float kLazyTau = 3.0f;
// The QK accumulators start at kAccBiasBits instead of 0: the int32 result bias + s, read as fp32,
// is exactly kAccBias + s for |s| < 2^22 (here |s| <= 2^21), so the logits reach the softmax as floats
// without an int -> float conversion per element; the bias is folded into the exp2 offset.
constexpr int kAccBiasBits = 0x4B400000;
constexpr float kAccBias = 12582912.0f;
// a masked logit as -inf: as int32 (-2^23) it lies below every biased logit, as fp32 its exp2 is 0
constexpr int kMaskedLogitBits = (int)0xFF800000u;

struct AttnParams {
  const int8_t* q8;
  int64_t qsb, qsl, qsh;
  const int8_t* k8;
  int64_t ksb, ksl, ksh;
  const void* v;  // tile-layout V: e4m3 (PV_FP8) or the half dtype, [B, Hkv, D, Lpad]
  int64_t Lpad;
  const float* q_scale;  // [B, Hq, nQS]: per 128-row block, per 32-row warp block, or per thread class
  const float* k_scale;  // [B, Hkv, nKS]: per 64-key tile, or 4 lane-pair classes per tile
  const float* v_scale;  // [B, Hkv, D] (FP8 P.V only)
  const float* v_mean;   // [B, Hkv, D] or null: added to the output (smoothed V, FP8 P.V only)
  void* o;
  int64_t osb, osl, osh;
  float* lse;  // [B, Hq, Lq] or null
  const int32_t* kv_valid;
  const int8_t* tile_mask;  // block-sparse: [B, Hkv, nQB, nKB] (strides tm_s1 per (b, kv head), tm_s2 per Q block)
  int64_t tm_s1, tm_s2;
  float* ws_o;   // split partials [split][B][Hq][Lq][D]
  float* ws_ml;  // [split][B][Hq][Lq][2]
  int64_t B, Lq, Lk, Hq, Hkv, nQB, nKB;
  int64_t nQS, nKS;  // scale entries per (b, h)
  int qgran;         // QATTN_GRAN_BLOCK / _WARP / _THREAD (q_scale indexing)
  float q_sm_scale;  // Q quantized per block inside the kernel: the factor multiplied into Q first
  int qrs;           // log2 of the rows of a warp cell of q_scale: 5 (sm89 tables) or 4 (sm90 tables)
  int kts;           // key tiles (64 keys) per k_scale block, as a shift: 0 (64-key blocks) or 1 (128)
  int64_t q_offset;
  int group;
  int nsplit;
  int tiles_per_split;
  int qpw;       // multi-block launches: query blocks per workgroup
  int64_t nQC;   // multi-block launches: workgroups per (batch, head)
  int causal;
  float qk_mult;
  // packed variable-length batches (null otherwise): sequence b has query rows cu_q[b] .. cu_q[b + 1] and key
  // rows cu_k[b] .. cu_k[b + 1] of the packed [1, total, H, D] tensors, its scales start at block cu_qs[b] /
  // cu_ks[b] of [total_blocks, H] tables, and its V tiles at tile cu_vt[b] of the [1, Hkv, D, Lpad] tile layout
  const int32_t* cu_q;
  const int32_t* cu_k;
  const int32_t* cu_qs;
  const int32_t* cu_ks;
  const int32_t* cu_vt;
  int64_t var_tq, var_tk;  // rows of the packed Q / K tensors
  // resident-K/V launches: each workgroup takes wb_per_wg consecutive 32-row wave blocks of one head,
  // n_chunk workgroups per (batch, head)
  int64_t wb_per_wg;
  int64_t n_chunk;
};

__device__ __forceinline__ int64_t xcd_remap(int64_t bid, int64_t n) {
  const int64_t q = n / 8, r = n % 8;
  const int64_t xcd = bid % 8, idx = bid / 8;
  return xcd * q + (xcd < r ? xcd : r) + idx;
}

// The KV split, (batch, head) and pair of query blocks of a workgroup.
//   * Dense: consecutive pairs of one head on one XCD, sharing its K/V in the XCD's L2; splits outermost, so the
//     workgroups of one key range of a head run next to each other.  (64-bit divisions: with 32-bit ones the start-up
//     is shorter, and 32760 x 32760 x 12 measured 0.8 % slower in every one of twelve interleaved rounds.)
//   * Causal, unsplit (CAUSAL): the longest pairs of all heads first.  Pair i costs about i + 1 key ranges; dealt in
//     ascending order the long ones started last and the launch ended on a few CUs.  Heads run innermost, so with a
//     multiple of 8 of them a head still stays on one XCD.
template <bool SPLIT, bool CAUSAL>
__device__ __forceinline__ void pair_of_workgroup(const AttnParams& p, int& split, int64_t& b, int64_t& h, int64_t& qp) {
  const int64_t nQP = (p.nQB + 1) / 2;
  if constexpr (CAUSAL && !SPLIT) {
    const uint32_t BH = (uint32_t)(p.B * p.Hq), i = blockIdx.x / BH, bh = blockIdx.x - i * BH;
    split = 0;
    qp = nQP - 1 - i;
    const uint32_t bb = bh / (uint32_t)p.Hq;
    b = bb;
    h = bh - bb * (uint32_t)p.Hq;
    return;
  }
  const int64_t wg_id = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t n_pairs = p.B * p.Hq * nQP;
  split = SPLIT ? (int)(wg_id / n_pairs) : 0;
  const int64_t tile_id = SPLIT ? wg_id - (int64_t)split * n_pairs : wg_id;
  qp = tile_id % nQP;
  const int64_t rest = tile_id / nQP;
  h = rest % p.Hq;
  b = rest / p.Hq;
}

// Buffer resource (V#) for raw, unswizzled byte addressing of [base, base + bytes): loads whose offset
// is at or past `bytes` return zeros instead of touching memory.
// q_scale entry of query row `row` (< nQB * 128): one per 128-row block, per warp cell of 2^qrs rows, or
// per row class (rows of a warp cell with equal row % 8: the reference's per-thread grouping).  Clamped
// to the table: the sm90 tables cover ceil(Lq / 64) * 64 rows, and the rows past that are masked.
__device__ __forceinline__ int64_t q_scale_index(const AttnParams& p, int64_t row) {
  const int64_t i = p.qgran == QATTN_GRAN_THREAD ? ((row >> p.qrs) << 3) + (row & 7)
                    : p.qgran == QATTN_GRAN_WARP ? row >> p.qrs
                                                 : row >> 7;
  return i < p.nQS ? i : p.nQS - 1;
}

// k_scale entry c (< ks) of key tile t in a table of ks entries per k_scale block
__device__ __forceinline__ int64_t k_scale_index(const AttnParams& p, int64_t t, int c, int ks) {
  return (t >> p.kts) * ks + c;
}

__device__ __forceinline__ v4u make_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  v4u r;
  r[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;  // raw buffer, 32-bit data format
  return r;
}

// One 16-byte-per-lane buffer -> LDS DMA (buffer_load_dwordx4 ... lds): lane j's 16 bytes, read at
// base + soff + voff_j, land at LDS address lds + 16 j.  The per-lane offsets are loop-invariant
// VGPRs and the tile advance is a scalar offset, so issuing a tile costs no VALU work.  Issued through
// inline asm so the compiler does not treat every later LDS read as a possible alias of the in-flight
// DMA (it would otherwise put an s_waitcnt vmcnt(0) in front of them and serialise the prefetch);
// completion is tracked with explicit vmcnt waits instead.
__device__ __forceinline__ void lds_dma16(uint32_t voff, v4u rsrc, uint32_t soff, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %0, %1, %2 offen lds"
      :
      : "v"(voff), "s"(rsrc), "s"(soff), "s"(lds)
      : "memory", "m0");
}

// The 4-byte form (buffer_load_dword ... lds): lane j's dword lands at lds + 4 j.
__device__ __forceinline__ void lds_dma4(uint32_t voff, v4u rsrc, uint32_t soff, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "buffer_load_dword %0, %1, %2 offen lds"
      :
      : "v"(voff), "s"(rsrc), "s"(soff), "s"(lds)
      : "memory", "m0");
}

// two floats -> two round-to-nearest-even halves (bf16: v_cvt_pk_bf16_f32), low word first
template <bool IS_FP16>
__device__ __forceinline__ uint32_t pack_half2(float a, float b) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  uint32_t r;
  if constexpr (IS_FP16) {
    const h2 v = __builtin_convertvector(f2{a, b}, h2);
    __builtin_memcpy(&r, &v, 4);
  } else {
    const b2 v = __builtin_convertvector(f2{a, b}, b2);
    __builtin_memcpy(&r, &v, 4);
  }
  return r;
}

// One output value: O / l * v_scale (+ v_mean for smoothed V), rounded after every operation (no fused
// multiply-add), so that every kernel and the split combine produce the same bits.
template <bool ADD_MEAN>
__device__ __forceinline__ float epilogue_value(float o, float inv_l, float sc, float vm) {
#pragma clang fp contract(off)
  const float x = o * inv_l * sc;
  if constexpr (ADD_MEAN) return x + vm;
  else return x;
}

// P of the FP8 P.V without an exponential.  u = 8 (x - kPLinShift) + 56, rounded to an integer k (RNE) and
// clamped to [0, 255] by v_cvt_pk_u8_f32, is read as the e4m3 byte of P: exponent field floor(y) + 7 and
// mantissa round(8 frac(y)) for y = x - kPLinShift, i.e. 2^floor(y) (1 + frac(y)) rounded to the e4m3 grid.
// This is Schraudolph's exponential ("A fast, compact approximation of the exponential function", Neural
// Computation 11, 1999: the argument scaled into the exponent field, the mantissa interpolating 2^f
// linearly) at e4m3 precision.  (1 + f) / 2^f lies in [1, 1.0861] with mean 1.040685 over f in [0, 1); the
// shift kPLinShift = log2(1.040685) removes that mean, so P is unbiased against exp2(x) on average and within
// -4.0 % / +4.4 % of it before the e4m3 rounding (RMS 3.15 % relative including the rounding, against
// 2.66 % for exp2(x) rounded to e4m3).  x <= 8.807 (the FP8 offset) gives k <= 126 (448); k = 127 would
// be NaN.  x < -7 gives 0; k < 8 are the e4m3 subnormals (P < 2^-6, linear in k).  Costs one full-rate
// conversion per element against a quarter-rate v_exp_f32 plus half a quarter-rate fp8 pack (measured:
// 10.3 against 23.9 cycles per element with the fma, two waves per SIMD).
constexpr float kPLinShift = 0.057539f;
constexpr float kPLinBias = 56.0f - 8.0f * kPLinShift;  // e4m3 exponent bias 7, in units of 1/8
__device__ __forceinline__ int p_e4m3_x4(float u0, float u1, float u2, float u3) {
  uint32_t t = __builtin_amdgcn_cvt_pk_u8_f32(u0, 0, 0u);
  t = __builtin_amdgcn_cvt_pk_u8_f32(u1, 1, t);
  t = __builtin_amdgcn_cvt_pk_u8_f32(u2, 2, t);
  return (int)__builtin_amdgcn_cvt_pk_u8_f32(u3, 3, t);
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}

// Row sums of P on the matrix pipe (FP8 P.V): one v_mfma_scale_f32_16x16x128_f8f6f4 per tile, D += A . B with
// B the e4m3 P^T operand of the P.V MFMA read in the 16 x 16 x 128 layout (lane l feeds column l % 16; its 32
// bytes are, in the 32 x 32 layout, 32 keys of query l % 32, so columns collect query c from lanes c and
// c + 32 and query c + 16 from lanes c + 16 and c + 48) and A an fp4 (e2m1) selector.  In this layout fp4
// nibbles 0-15 of A lane 16 a + r meet bytes 0-15 (a = 0, 1: of B lane groups 0, 2) or 16-31 (a = 2, 3) of
// lane groups 0 / 2, and nibbles 16-31 the same bytes of lane groups 1 / 3 (measured on gfx950).  So row 0 of
// A is 1.0 on nibbles 0-15 of lanes 0, 16, 32, 48 and row 1 on nibbles 16-31 of lanes 1, 17, 33, 49: row 0
// of the result is the running sum l of queries 0..15, row 1 that of queries 16..31, and lane c < 16 holds
// them in elements 0 and 1.  l is thus the sum of the e4m3-rounded P (the reference's accumulate_d sums p
// before rounding; the difference is the mean FP8 rounding error of P, far inside the attention tolerance);
// the row sums leave the softmax's VALU stream, and the MFMA costs half the 32 x 32 x 64 form.
__device__ __forceinline__ v8i row_sum_selector() {
  const int r = threadIdx.x & 15;
  const int lo = r == 0 ? 0x22222222 : 0, hi = r == 1 ? 0x22222222 : 0;
  return v8i{lo, lo, hi, hi, 0, 0, 0, 0};
}
__device__ __forceinline__ v4f row_sum_mfma(const v4f& acc, const v8i& pf, const v8i& sel) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(sel, pf, acc, 4, 0, 0, 0, 0, 0);
}
// online-softmax rescale of the row sums: element 0 of lane c belongs to query c (the lane's own), element 1
// to query c + 16, whose factor lane c + 16 holds
__device__ __forceinline__ void row_sum_rescale(v4f& acc, float alpha) {
  const int lane = threadIdx.x & 63;
  const float a_hi = __int_as_float(__builtin_amdgcn_ds_bpermute(((lane & 15) + 16) * 4, __float_as_int(alpha)));
  acc[0] *= alpha;
  acc[1] *= a_hi;
}
// the row sum of query lq (lanes lq and lq + 32 both get it)
__device__ __forceinline__ float row_sum_value(const v4f& acc, int lq) {
  const int src = (lq & 15) * 4;
  const float v0 = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(acc[0])));
  const float v1 = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(acc[1])));
  return lq < 16 ? v0 : v1;
}

// P.V flavours: e4m3 P x e4m3 V (the reference's fp8 kernel, with the 8.807 offset and v_scale), or
// P rounded to the half dtype of V x V as given (the Triton / SAGE_ATTN_2_8_16 style), fp32 accumulation.
enum PvKind { PV_FP8 = 0, PV_BF16 = 1, PV_FP16 = 2 };

// QF: Q as int8 with its scale table (0), or Q in the output's half type quantized inside the attention
// kernel: with the per-thread classes of the Triton quantizer (QF_THREAD: rows with equal row % 8 of a wave's
// 32 share a scale, round half away from x / scale), the per-warp blocks of the CUDA one (QF_WARP: a wave's
// 32 rows share a scale, RNE of x * 127 / amax), or its per-block form (QF_BLOCK: the
// 128 rows of a query block, held by four waves of one workgroup, share a scale, x multiplied by
// sm_scale * log2(e) first) -- the codes and
// scales of per_thread_int8 / per_warp_int8 / per_block_int8 bit for bit, without writing int8 Q out and
// reading it back.
constexpr int QF_INT8 = 0, QF_THREAD = 1, QF_WARP = 2, QF_BLOCK = 3;

// Lane (lq, hf) of a wave whose 32 query rows are lq = lane % 32: the raw half words of its row (row
// pointer rowp; zeros when !valid) at 32 m + 16 hf .. + 16, m < NQF.
template <int NQF>
__device__ __forceinline__ void quant_q_raw(const uint16_t* rowp, bool valid, int hf, v4u (&r)[NQF][2]) {
#pragma unroll
  for (int m = 0; m < NQF; m++) {
    r[m][0] = r[m][1] = v4u{0, 0, 0, 0};
    if (valid) {
      r[m][0] = *reinterpret_cast<const v4u*>(rowp + m * 32 + hf * 16);
      r[m][1] = *reinterpret_cast<const v4u*>(rowp + m * 32 + hf * 16 + 8);
    }
  }
}

// Those values as fp32, times mul when MUL.
template <bool IS_FP16, int NQF, bool MUL>
__device__ __forceinline__ void quant_q_unpack(const v4u (&r)[NQF][2], float mul, float (&x)[NQF][16]) {
#pragma unroll
  for (int m = 0; m < NQF; m++) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      x[m][2 * e] = half_to_f32<IS_FP16>((uint16_t)(r[m][0][e] & 0xffffu));
      x[m][2 * e + 1] = half_to_f32<IS_FP16>((uint16_t)(r[m][0][e] >> 16));
      x[m][8 + 2 * e] = half_to_f32<IS_FP16>((uint16_t)(r[m][1][e] & 0xffffu));
      x[m][8 + 2 * e + 1] = half_to_f32<IS_FP16>((uint16_t)(r[m][1][e] >> 16));
    }
    if constexpr (MUL) {
#pragma unroll
      for (int e = 0; e < 16; e++) x[m][e] = x[m][e] * mul;
    }
  }
}

// The |x| maximum over the lane's scale group within the wave (per-thread class: lanes lq ^ 8, lq ^ 16 and
// the other half-row; per-warp / per-block: all 64 lanes, from the CUDA quantizer's 1e-7 floor).
template <int QF, int NQF>
__device__ __forceinline__ float quant_q_amax(const float (&x)[NQF][16]) {
  float am = QF == QF_THREAD ? 0.f : 0.0000001f;
#pragma unroll
  for (int m = 0; m < NQF; m++)
#pragma unroll
    for (int e = 0; e < 16; e++) am = fmaxf(am, fabsf(x[m][e]));
  if constexpr (QF != QF_THREAD) {
    am = fmaxf(am, __shfl_xor(am, 1, 64));
    am = fmaxf(am, __shfl_xor(am, 2, 64));
    am = fmaxf(am, __shfl_xor(am, 4, 64));
  }
  am = fmaxf(am, __shfl_xor(am, 8, 64));
  am = fmaxf(am, __shfl_xor(am, 16, 64));
  am = fmaxf(am, __shfl_xor(am, 32, 64));
  return am;
}

// The three steps at once: the lane's values x (times mul when MUL) and their group maximum.
template <bool IS_FP16, int QF, int NQF, bool MUL = false>
__device__ __forceinline__ float quant_q_load(const uint16_t* rowp, bool valid, int hf, float mul, float (&x)[NQF][16]) {
  v4u r[NQF][2];
  quant_q_raw<NQF>(rowp, valid, hf, r);
  quant_q_unpack<IS_FP16, NQF, MUL>(r, mul, x);
  return quant_q_amax<QF, NQF>(x);
}

// The scale of a group with |x| maximum am (returned) and the int8 codes as the MFMA B fragments qf.
template <int QF, int NQF>
__device__ __forceinline__ float quant_q_codes(const float (&x)[NQF][16], float am, v4i (&qf)[NQF]) {
  constexpr bool TRITON = QF == QF_THREAD;
  const float sc = TRITON ? quant_scale_triton(am) : quant_scale_cuda(am);
  const float iv = TRITON ? refined_rcp(sc) : quant_recip_cuda(am);
#pragma unroll
  for (int m = 0; m < NQF; m++) {
    int c[16];
#pragma unroll
    for (int e = 0; e < 16; e++) c[e] = TRITON ? quant_code_triton<true>(x[m][e], sc, iv) : quant_code_cuda(x[m][e], iv);
#pragma unroll
    for (int g = 0; g < 4; g++)
      // (the low bytes of a pair by one v_perm_b32, then lshl_or: 3 instructions)
      qf[m][g] = (int)(__builtin_amdgcn_perm((uint32_t)c[4 * g + 1], (uint32_t)c[4 * g], 0x0c0c0400u) |
                       (__builtin_amdgcn_perm((uint32_t)c[4 * g + 3], (uint32_t)c[4 * g + 2], 0x0c0c0400u) << 16));
  }
  return sc;
}

// per-thread / per-warp: both steps within the wave
template <bool IS_FP16, int QF, int NQF>
__device__ __forceinline__ float quant_q_rows(const uint16_t* rowp, bool valid, int hf, v4i (&qf)[NQF]) {
  static_assert(QF == QF_THREAD || QF == QF_WARP, "wave-local scale groups");
  float x[NQF][16];
  const float am = quant_q_load<IS_FP16, QF, NQF>(rowp, valid, hf, 1.f, x);
  return quant_q_codes<QF, NQF>(x, am, qf);
}

// workgroup barrier that the compiler neither crosses with memory operations nor schedules around
__device__ __forceinline__ void pp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// the KV-split combine of a launch with p.nsplit > 1 (attn.hip)
void launch_combine(const AttnParams& p, int out_dtype, int64_t D, hipStream_t st);

// half P.V launches (attn_half.hip): dense and block-sparse, packed varlen; key tiles one split can cover, and the
// split count of a dense launch
int launch_half(AttnParams& p, bool kt, bool f16v, bool sparse, int out_dtype, int ns, hipStream_t st);
int launch_half_varlen(AttnParams& p, int out_dtype, hipStream_t st);
int64_t half_max_tiles(bool kt, bool sparse);
int half_num_splits(int64_t bh, int64_t nqb, int64_t nkb, bool kt);

}  // namespace qattn
