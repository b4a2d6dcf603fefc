// Quantized attention forward for gfx950: INT8 Q.K^T and FP8 P.V on MFMA, fp32 online softmax.
//
// Math (the reference's sm89 kernel, tf-kernel/csrc/sageattn2/qattn/qk_int_sv_f8_cuda_sm89.cuh:342-840,
// attn_utils.cuh:362-452 update_mdo, :469-481 RS_32_to_8, :711-756 normalize_d):
//   s    = int32(Q8 . K8^T) * (q_scale * k_scale * qk_mult)          (log2 domain)
//   m'   = max(m, rowmax(s) - 8.807);   p = exp2(s - m')  in (0, 448]
//          (here with a lazy update rule: m' = rowmax(s) - 5.807 only if that exceeds m by > 3, which
//          keeps p <= 448 and skips the O rescale on almost every tile; oracle/ restates the rule)
//   l    = l * exp2(m - m') + sum(p)
//   O    = O * exp2(m - m') + e4m3(p) . e4m3(V)                        (fp32 accumulation)
//   out  = O / l * v_scale[d]
//   (the FP8 P.V kernels form e4m3(p) straight from s - m' without an exponential, p_e4m3_x4 below,
//   and sum that rounded P; the half P.V kernels use exp2)
//
// MI355X design (not a translation of the NVIDIA tiling):
//   * qattn_fwd_kernel: workgroup = 4 wave64s = 128 query rows (one Q quantization block, so one q_scale);
//     each wave owns 32 rows.  Key tiles of 64 keys (one K quantization block, one k_scale).
//   * S^T = K . Q^T with v_mfma_i32_32x32x32_i8 (A = K from LDS, B = Q held in VGPRs for the whole
//     loop).  In the 32x32 result each lane owns one query column and 16 key rows, so the row max
//     is an in-lane max plus one lane^32 exchange, and the running sum stays per lane until the end.
//   * O^T = V^T . P^T with v_mfma_f32_32x32x64_f8f6f4 (A = V^T from LDS, B = P^T straight from the
//     softmax registers).  The FP8 V quantizer stores every 64-key tile in exactly the key order the
//     B operand inherits from the S^T layout, so P never goes through LDS.
//   * K/V tiles are multi-buffered in LDS, fragment-major (each 1 KiB block holds one MFMA operand
//     fragment of all 64 lanes), and fetched by LDS DMA (buffer_load_dwordx4 ... lds) issued before the
//     current tile's MFMA/softmax work, so staging costs neither VGPRs nor VALU slots and a lane reads
//     its fragments from one base address plus constant offsets.
//   * Large dense launches run the ping-pong kernel (two 4-wave groups per workgroup, 256 rows, whose
//     waves alternate matrix and vector stages on each SIMD); the per-element arithmetic is the same.
//   * blockIdx -> tile mapping is XCD-aware: the hardware deals workgroups round-robin over the 8
//     XCDs, so consecutive tiles of one (batch, head) are gathered onto one XCD and share its L2.
//   * Optional KV split (flash-decoding style) for grids that cannot fill 256 CUs; a combine kernel
//     merges the partial (O, m, l) triples.
#include <mutex>

#include "attn_device.h"

namespace qattn {

template <bool IS_FP16_OUT, bool SPLIT, bool KT, bool MQ = false>
__global__ __launch_bounds__(kThreads, kWavesPerSimd) void qattn_fwd_kernel(AttnParams p) {
  static_assert(!MQ || !SPLIT, "multi-block launches: no split");
  constexpr int KS = ks_per_tile(KT);
  __shared__ __align__(16) uint8_t lds_k[kNBuf][kBK * kD];
  __shared__ __align__(16) uint8_t lds_v[kNBuf][kD * kBK];
  __shared__ float lds_ks[MQ ? kMqMaxTiles * 4 : kKsLdsFloats];  // k_scales of its key tiles
  // multi-block launches: a wave-private 4 KiB region per wave that receives the next query block's Q
  // rows by DMA and then stages the finished block's O rows; and the q_scales of all its blocks
  __shared__ __align__(16) uint8_t lds_qo[MQ ? 4 * 4096 : 16];
  __shared__ float lds_qs[MQ ? kMqMaxBlocks * 32 : 1];
  __shared__ __align__(16) float lds_vs[kD];  // v_scale of this head (epilogue)
  __shared__ __align__(16) float lds_vm[kD];  // v_mean of this head (smoothed V)

  const int64_t tile_id = xcd_remap(blockIdx.x, gridDim.x);
  int64_t qb, qb_end;  // query blocks [qb, qb_end) of this workgroup
  int64_t rest;
  int split = 0;
  if constexpr (MQ) {
    qb = (tile_id % p.nQC) * p.qpw;
    qb_end = min(p.nQB, qb + p.qpw);
    rest = tile_id / p.nQC;
  } else {
    qb = tile_id % p.nQB;
    qb_end = qb + 1;
    rest = tile_id / p.nQB;
    split = (int)(rest % p.nsplit);
    rest /= p.nsplit;
  }
  const int64_t qb0 = qb;
  const int64_t h = rest % p.Hq;
  const int64_t b = rest / p.Hq;
  const int64_t hk = h / p.group;

  const int64_t Lq = p.Lq, Lk = p.Lk;
  const int8_t* q8b = p.q8 + b * p.qsb;
  const int8_t* k8b = p.k8 + b * p.ksb;
  const float* qs_tab = p.q_scale + (b * p.Hq + h) * p.nQS;
  const float* ks_ptr = p.k_scale + (b * p.Hkv + hk) * p.nKS;
  uint16_t* ob = static_cast<uint16_t*>(p.o) + b * p.osb;

  const int tid = threadIdx.x;
  // (wave index in a scalar register, so that every per-wave quantity and branch stays scalar)
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, hf = lane >> 5;

  // key range of this workgroup
  int64_t q_first = qb * kBQ;
  int64_t kv_end = Lk;
  if (p.kv_valid) kv_end = min(kv_end, (int64_t)p.kv_valid[b]);
  if (p.causal) kv_end = min(kv_end, q_first + kBQ + p.q_offset);
  const int64_t n_tiles = kv_end > 0 ? (kv_end + kBK - 1) / kBK : 0;
  const int64_t t_begin = SPLIT ? (int64_t)split * p.tiles_per_split : 0;
  const int64_t t_end = SPLIT ? min(n_tiles, t_begin + p.tiles_per_split) : n_tiles;

  // Q fragment (B operand of S^T = K.Q^T): lane owns query row lq of this wave, bytes
  // d = 32*m + 16*hf .. +16 for m = 0..3
  int64_t wrow0 = q_first + w * 32;
  int64_t qrow = wrow0 + lq;
  // Q fragments: the wave's 32 rows are read row-contiguously (8 lanes x 16 B per 128-byte row, full
  // cache lines) into a wave-private LDS stage, then each lane picks its MFMA B-operand bytes
  // d = 32 m + 16 hf .. +16 of row lq.  Stage rows are 128 B with the 16-byte chunk c stored at
  // chunk c ^ (row & 7), so both the row writes and the fragment reads are bank-conflict free.
  uint8_t* stage = (MQ ? &lds_qo[0] : &lds_k[0][0]) + w * 4096;  // 32 rows x 128 B per wave (lds_k is free here)
  v4i qf[4];
  {
    const int8_t* qbase = q8b + h * p.qsh;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = i * 8 + (lane >> 3), c = lane & 7;
      const int64_t row = wrow0 + r;
      const v4i val = row < Lq ? *reinterpret_cast<const v4i*>(qbase + row * p.qsl + c * 16) : v4i{0, 0, 0, 0};
      *reinterpret_cast<v4i*>(stage + r * 128 + ((c ^ (r & 7)) << 4)) = val;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const int c = 2 * m + hf;
      qf[m] = *reinterpret_cast<const v4i*>(stage + lq * 128 + ((c ^ (lq & 7)) << 4));
    }
    // consume the loads here: otherwise the compiler's wait for them lands at their first use inside
    // the key loop
#pragma unroll
    for (int m = 0; m < 4; m++) asm volatile("" ::"v"(qf[m]));
  }
  // q_scale of this lane's query row
  float qs = qs_tab[q_scale_index(p, qb * kBQ + w * 32 + lq)] * p.qk_mult;
  // q_scale entries per query block, and this lane's entry within its block
  const int qs_per = p.qgran == QATTN_GRAN_THREAD ? (kBQ >> p.qrs) * 8 : p.qgran == QATTN_GRAN_WARP ? kBQ >> p.qrs : 1;
  const int qs_sub = p.qgran == QATTN_GRAN_BLOCK ? 0 : (int)q_scale_index(p, w * 32 + lq);

  // global -> LDS copies go through the LDS-DMA path (buffer_load_dwordx4 ... lds): lane j of a wave
  // writes the 16 bytes at LDS slot (wave base + 16 j).  The tiles are fragment-major: 1 KiB block f holds
  // MFMA operand fragment f of all 64 lanes (lane l at 16 l), so a lane reads its fragments at one base
  // address plus constant offsets, each read a contiguous, conflict-free 1 KiB:
  //   K block j (0..7): lane l gets K row (j & 1) * 32 + l % 32, bytes 16 (2 (j >> 1) + l / 32) .. + 16
  //   V block 2 dblk + h: lane l gets V^T row dblk * 32 + l % 32, bytes 16 (2 (l / 32) + h) .. + 16
  // DMA instruction i of wave w fills block 4 i + w.  Each wave moves 2 x 1 KiB of K and 2 x 1 KiB of V
  // per tile; no VGPRs are spent on staging.
  // The K resource of a tile starts at the tile's first row, so K rows at or past Lk fall outside its
  // range and arrive as zeros (masked anyway) without being read (the range check covers the
  // per-lane offset, not the scalar one).
  const int8_t* kbase = k8b + hk * p.ksh;
  const uint8_t* vbase = static_cast<const uint8_t*>(p.v) + (b * p.Hkv + hk) * (int64_t)kD * p.Lpad;
  const int64_t kbytes = (Lk - 1) * p.ksl + kD;
  const v4u vrsrc = make_rsrc(vbase, (uint32_t)((int64_t)kD * p.Lpad));
  // per-lane byte offsets relative to the tile start (first K row / first V column)
  uint32_t koff[2], voff[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int j = i * 4 + w;
    koff[i] = (uint32_t)(((j & 1) * 32 + lq) * p.ksl + (2 * (j >> 1) + hf) * 16);
  }
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int f = i * 4 + w;
    voff[i] = (uint32_t)(((f >> 1) * 32 + lq) * p.Lpad + (2 * hf + (f & 1)) * 16);
  }
  const int64_t k_step = kBK * p.ksl;
  const uint32_t lds_k0 = lds_addr(&lds_k[0][0]) + __builtin_amdgcn_readfirstlane(w) * 1024;
  const uint32_t lds_v0 = lds_addr(&lds_v[0][0]) + __builtin_amdgcn_readfirstlane(w) * 1024;
  auto dma_tile = [&](int64_t t, int buf) {
    const int64_t kso = t * k_step;
    const v4u krsrc = make_rsrc(kbase + kso, (uint32_t)(kbytes - kso));
    const uint32_t vso = (uint32_t)t * kBK;
    const uint32_t kl = lds_k0 + buf * (kBK * kD), vl = lds_v0 + buf * (kD * kBK);
#pragma unroll
    for (int i = 0; i < 2; i++) lds_dma16(koff[i], krsrc, 0, kl + i * 4096);
#pragma unroll
    for (int i = 0; i < 2; i++) lds_dma16(voff[i], vrsrc, vso, vl + i * 4096);
  };
  // multi-block launches: the wave's 32 rows of the next query block go by DMA into its region of
  // lds_qo, in the stage layout (LDS slot (r, c') receives global chunk c' ^ (r & 7)); the resource
  // covers exactly the rows below Lq, the others arrive as zeros
  uint32_t qoff[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int slot = i * 64 + lane, r = slot >> 3;
    qoff[i] = (uint32_t)(r * p.qsl + (((slot & 7) ^ (r & 7)) << 4));
  }
  const int8_t* qhead = q8b + h * p.qsh;
  const int wu = __builtin_amdgcn_readfirstlane(w);
  auto dma_q = [&](int64_t blk) {
    const int64_t r0 = blk * kBQ + wu * 32;
    const int64_t nr = min((int64_t)32, Lq - r0);
    const v4u qr = make_rsrc(qhead + (nr > 0 ? r0 * p.qsl : 0), nr > 0 ? (uint32_t)((nr - 1) * p.qsl + kD) : 0u);
    const uint32_t ql = lds_addr(&lds_qo[0]) + wu * 4096;
#pragma unroll
    for (int i = 0; i < 4; i++) lds_dma16(qoff[i], qr, 0, ql + i * 1024);
  };

  v16f o[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[i][r] = 0.f;
  float m_run = kMInit;
  v4f lacc = {0.f, 0.f, 0.f, 0.f};  // row sums of P on the matrix pipe (row_sum_mfma)
  const v8i rs_sel = row_sum_selector();
  v16i kbias;
#pragma unroll
  for (int r = 0; r < 16; r++) kbias[r] = kAccBiasBits;

  // K/V tiles run kPrefetch tiles ahead of the compute through kNBuf = kPrefetch + 1 LDS buffers:
  // iteration t issues tile t + kPrefetch into buffer (t + kPrefetch) % kNBuf, which was last read in
  // iteration t - 1.  The k_scales of all tiles are staged in LDS once, so the only VMEM traffic in the
  // loop is the 4 DMA instructions per tile and the vmcnt accounting below is exact.
  __syncthreads();  // every wave has its Q fragments out of the LDS stage before the DMA reuses it
  for (int64_t i = tid; i < (t_end - t_begin) * KS; i += kThreads) lds_ks[i] = ks_ptr[k_scale_index(p, t_begin + i / KS, i % KS, KS)];
  if constexpr (!SPLIT)
    if (tid < kD) {
      lds_vs[tid] = p.v_scale[(b * p.Hkv + hk) * kD + tid];
      lds_vm[tid] = p.v_mean ? p.v_mean[(b * p.Hkv + hk) * kD + tid] : 0.f;
    }
  if constexpr (MQ) {
    const float* qsp = p.q_scale + (b * p.Hq + h) * p.nQS + qb0 * qs_per;
    const int64_t n_qs = std::min<int64_t>((qb_end - qb0) * qs_per, p.nQS - qb0 * qs_per);
    for (int64_t i = tid; i < n_qs; i += kThreads) lds_qs[i] = qsp[i];
  }
  // The loop runs over (query block, key tile) pairs: a multi-block launch walks the same key tiles once
  // per query block, and its DMA stream runs on across the block boundaries.
  const int64_t n_kt = t_end - t_begin;
  const int64_t total = MQ ? (qb_end - qb0) * n_kt : n_kt;
#pragma unroll
  for (int d = 0; d < kPrefetch; d++)
    if (d < total) dma_tile(t_begin + (MQ ? d % n_kt : d), d);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // ---- epilogue of the current query block: O / l * v_scale out through the wave's LDS stage ----
  auto finish = [&]() {
    const float l_tot = row_sum_value(lacc, lq);
    if (SPLIT) {
      if (qrow >= Lq) return;
      const int64_t row = (((int64_t)split * p.B + b) * p.Hq + h) * p.Lq + qrow;
      float* wo = p.ws_o + row * kD;
#pragma unroll
      for (int dblk = 0; dblk < 4; dblk++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int d = dblk * 32 + g * 8 + hf * 4;
          *reinterpret_cast<v4f*>(wo + d) =
              v4f{o[dblk][g * 4 + 0], o[dblk][g * 4 + 1], o[dblk][g * 4 + 2], o[dblk][g * 4 + 3]};
        }
      if (hf == 0) {
        p.ws_ml[row * 2 + 0] = m_run;
        p.ws_ml[row * 2 + 1] = l_tot;
      }
      return;
    }
    const float inv_l = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    // O goes out through the wave-private LDS stage (the K/V buffers are idle after the loop's last
    // barrier; multi-block launches use their own region), 64 channels per pass, so that every row is
    // stored as whole 128-byte lines
    uint16_t* obase = ob + h * p.osh;
    auto store = [&](auto mean_t) {
    constexpr bool kMean = decltype(mean_t)::value;
#pragma unroll
    for (int pass = 0; pass < 2; pass++) {
#pragma unroll
      for (int db = 0; db < 2; db++) {
        const int dblk = pass * 2 + db;
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int d = dblk * 32 + g * 8 + hf * 4;
          const v4f sc = *reinterpret_cast<const v4f*>(&lds_vs[d]);
          float f[4];
          const v4f vm = kMean ? *reinterpret_cast<const v4f*>(&lds_vm[d]) : v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; e++) f[e] = epilogue_value<kMean>(o[dblk][g * 4 + e], inv_l, sc[e], vm[e]);
          const v2u packed{pack_half2<IS_FP16_OUT>(f[0], f[1]), pack_half2<IS_FP16_OUT>(f[2], f[3])};
          const int c = db * 4 + g;  // 16-byte chunk of the staged 128-byte row (8 channels)
          *reinterpret_cast<v2u*>(stage + lq * 128 + ((c ^ (lq & 7)) << 4) + hf * 8) = packed;
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int r = i * 8 + (lane >> 3), c = lane & 7;
        const v4u val = *reinterpret_cast<const v4u*>(stage + r * 128 + ((c ^ (r & 7)) << 4));
        const int64_t row = wrow0 + r;
        if (row < Lq) *reinterpret_cast<v4u*>(obase + row * p.osl + pass * 64 + c * 8) = val;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    };
    if (p.v_mean) store(std::true_type{});
    else store(std::false_type{});
    if (p.lse && hf == 0 && qrow < Lq)
      p.lse[(b * p.Hq + h) * p.Lq + qrow] = l_tot > 0.f ? __builtin_log2f(l_tot) + m_run : -INFINITY;
  };
  [[maybe_unused]] auto next_block = [&]() {
    qb++;
    q_first = qb * kBQ;
    wrow0 = q_first + w * 32;
    qrow = wrow0 + lq;
    qs = lds_qs[(qb - qb0) * qs_per + qs_sub] * p.qk_mult;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[i][r] = 0.f;
    m_run = kMInit;
    lacc = v4f{0.f, 0.f, 0.f, 0.f};
  };

  int buf = 0;
  int64_t t = t_begin;                            // key slot being computed
  int64_t pt = t_begin + (MQ && total > 0 ? kPrefetch % n_kt : kPrefetch);  // next slot to fetch
  for (int64_t it = 0; it < total; it++) {
    const bool issue = it + kPrefetch < total;
    // (issued before this iteration's K/V DMA, so the iteration's final vmcnt wait covers it)
    if constexpr (MQ)
      if (t == 0 && qb + 1 < qb_end) dma_q(qb + 1);
    if (issue) {
      dma_tile(pt, buf == 0 ? kNBuf - 1 : buf - 1);
      pt++;
      if (MQ && pt == t_end) pt = t_begin;
    }
    // logit scale(s) of this lane: with per-thread K scales, key kappa of the tile belongs to class
    // (kappa % 8) / 2 = 2 hf + (r & 3) / 2 for accumulator element r, so a lane needs two of them
    float cs_a, cs_b;
    if constexpr (KT) {
      cs_a = qs * lds_ks[(t - t_begin) * 4 + 2 * hf];
      cs_b = qs * lds_ks[(t - t_begin) * 4 + 2 * hf + 1];
    } else {
      cs_a = cs_b = qs * lds_ks[t - t_begin];
    }

    // ---- S^T = K . Q^T: two 32-key blocks x 4 MFMAs over D = 128; K fragments streamed from LDS ----
    v16i s[2];
    {
      v4i kf[8];  // all K fragments first: the LDS latency is paid once per tile
#pragma unroll
      for (int j = 0; j < 8; j++)
        kf[j] = *reinterpret_cast<const v4i*>(&lds_k[buf][j * 1024 + lane * 16]);
      // The QK MFMAs run at raised wave priority: when the other wave of the SIMD is in its softmax
      // VALU phase, the scheduler then keeps the matrix pipe fed from this wave (measured ~6 % faster
      // than equal priorities).
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int m = j >> 1, kb = j & 1;
        s[kb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[j], qf[m], m == 0 ? kbias : s[kb], 0, 0, 0);
      }
      __builtin_amdgcn_s_setprio(0);
    }

    // ---- masking (tail tile, key padding, causal diagonal) ----
    const int64_t k0 = t * kBK;
    const bool masked = (k0 + kBK > kv_end) || (p.causal && k0 + kBK - 1 > wrow0 + p.q_offset);
    if (masked) {
      // element r of block kb holds key k0 + c + 4 hf with c = 32 kb + 8 (r / 4) + r % 4; it is masked
      // when key >= kv_end or (causal) key > qrow + q_offset, i.e. when c >= lim for this lane's lim
      int lim = (int)min(kv_end - k0, (int64_t)kBK);
      if (p.causal) lim = min(lim, (int)max(min(qrow + p.q_offset + 1 - k0, (int64_t)kBK), (int64_t)-1));
      lim -= hf * 4;
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (kb * 32 + (r >> 2) * 8 + (r & 3) >= lim) s[kb][r] = INT32_MIN;
    }

    // ---- online softmax ----
    float m_tile;
    if constexpr (!KT) {
      int mx = max(s[0][0], s[0][1]);
#pragma unroll
      for (int r = 2; r < 16; r++) mx = max(mx, s[0][r]);
#pragma unroll
      for (int r = 0; r < 16; r++) mx = max(mx, s[1][r]);
      {  // lanes l and l^32 hold the two key halves of the same query row
        const auto sw = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
        mx = max((int)sw[0], (int)sw[1]);
      }
      // Lazy rescale: the running max m is only moved when the tile max exceeds it by more than
      // kLazyTau (log2 units), per row.  With the offset lowered by the same tau, p = exp2(s - m) stays
      // <= 2^8.807 = 448 (the e4m3 maximum), so the FP8 range is honoured while the O rescale (64
      // multiplies per lane) is skipped on almost every tile.  A row whose keys in this tile are all
      // masked never moves m.
      m_tile = mx == INT32_MIN ? kMInit : fmaf(__int_as_float(mx), cs_a, -fmaf(kAccBias, cs_a, kFp8Offset - kLazyTau));
    } else {  // two scale classes per lane: max per class, scaled, then across the lane pair
      int ma = INT32_MIN, mb = INT32_MIN;
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          if ((r & 3) < 2) ma = max(ma, s[kb][r]);
          else mb = max(mb, s[kb][r]);
        }
      const float fa = ma == INT32_MIN ? kMInit : fmaf(__int_as_float(ma), cs_a, -fmaf(kAccBias, cs_a, kFp8Offset - kLazyTau));
      const float fb = mb == INT32_MIN ? kMInit : fmaf(__int_as_float(mb), cs_b, -fmaf(kAccBias, cs_b, kFp8Offset - kLazyTau));
      float mt = fmaxf(fa, fb);
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
      m_tile = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    const bool grow = m_tile > m_run + kLazyTau;
    if (__any(grow)) {
      const float m_new = grow ? m_tile : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] *= alpha;
      row_sum_rescale(lacc, alpha);
      m_run = m_new;
    }
    v8i pf;  // P^T as the e4m3 B operand: byte s of the lane = slot s = 16 kb + r
    // u = 8 (s * cs - m - kPLinShift) + 56 (p_e4m3_x4); masked logits give u = -1, P = 0
    const float cs8_a = 8.0f * cs_a, cs8_b = 8.0f * cs_b;
    const float nu_a = fmaf(-8.0f, fmaf(kAccBias, cs_a, m_run), kPLinBias);
    const float nu_b = fmaf(-8.0f, fmaf(kAccBias, cs_b, m_run), kPLinBias);
    auto body = [&](auto mk) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int kb = j >> 2, r0 = (j & 3) * 4;
        float u[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int sv = s[kb][r0 + e];
          u[e] = fmaf(__int_as_float(sv), e < 2 ? cs8_a : cs8_b, e < 2 ? nu_a : nu_b);
          if constexpr (decltype(mk)::value) u[e] = sv == INT32_MIN ? -1.f : u[e];
        }
        pf[j] = p_e4m3_x4(u[0], u[1], u[2], u[3]);
      }
    };
    if (masked) body(std::true_type{});
    else body(std::false_type{});

    // ---- O^T += V^T . P^T (FP8 MFMA, K = 64 keys) ----
    v8i vf[4];
#pragma unroll
    for (int dblk = 0; dblk < 4; dblk++) {
      const v4i a0 = *reinterpret_cast<const v4i*>(&lds_v[buf][(2 * dblk) * 1024 + lane * 16]);
      const v4i a1 = *reinterpret_cast<const v4i*>(&lds_v[buf][(2 * dblk + 1) * 1024 + lane * 16]);
      vf[dblk] = v8i{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
    }
#pragma unroll
    for (int dblk = 0; dblk < 4; dblk++)
      o[dblk] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf[dblk], pf, o[dblk], 0, 0, 0, 0, 0, 0);
    lacc = row_sum_mfma(lacc, pf, rs_sel);

    // tile t+1 must have landed; the DMAs of the tiles after it may stay in flight
    if (issue) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (kPrefetch - 1)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    buf = buf + 1 == kNBuf ? 0 : buf + 1;
    t++;
    if constexpr (MQ) {
      if (t == t_end && qb + 1 < qb_end) {
        // block boundary: the next block's Q rows (landed with this iteration's wait) leave the region
        // before the finished block's O goes out through it
        v4i qn[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
          const int c = 2 * m + hf;
          qn[m] = *reinterpret_cast<const v4i*>(stage + lq * 128 + ((c ^ (lq & 7)) << 4));
        }
        finish();
#pragma unroll
        for (int m = 0; m < 4; m++) qf[m] = qn[m];
        next_block();
        t = t_begin;
      }
    }
  }
  if constexpr (MQ) {
    // no key tiles at all (kv_valid 0): every block of the workgroup gets the empty-row output
    if (total == 0)
      while (qb + 1 < qb_end) {
        finish();
        next_block();
      }
  }
  finish();
}

// ---- ping-pong workgroups: two groups of four waves, one wave of each group per SIMD ----
//
// In qattn_fwd_kernel the two waves of a SIMD belong to different workgroups and fall into step with
// each other: both run their softmax on the VALU, then both run their MFMAs, so a SIMD spends the sum
// of the two phases per tile.  Here one workgroup holds two query blocks of the same head (group 0 =
// waves 0-3, group 1 = waves 4-7; wave w runs on SIMD w % 4) and the groups alternate through workgroup
// barriers, half a tile apart:
//
//   group 0:  M(0) | V(0) | M(1) | V(1) | ...        M(t) = P(t-1).V(t-1), row sum, Q.K(t)^T (matrix pipe)
//   group 1:    -  | M(0) | V(0) | M(1) | ...        V(t) = mask, softmax, P(t) to e4m3  (VALU)
//
// so at every step one wave of a SIMD feeds the matrix pipe while the other runs the VALU softmax, and
// a SIMD spends about max(MFMA, VALU) per step instead of their sum.  Per element the arithmetic is
// that of qattn_fwd_kernel (32 rows per wave, same MFMA chains, lazy running max, FP8 offset, row sums
// on the matrix pipe), so both kernels give identical results.
//
// K/V tiles come in by LDS DMA, four buffers, two tiles ahead: every wave moves 1 KiB of K and 1 KiB of
// V of tile t + 2 at the start of its stage M(t) and has its share of tile t + 1 landed by the end of
// M(t); tile t is read as K in M(t) and as V during V(t) (operands of M(t + 1)), so its buffer is free
// once both groups have finished M(t + 1).
constexpr int kPPThreads = 512;
constexpr int kPPNBuf = 4;

// CA: unsplit causal launches (KV-split ones decide by p.causal)
template <bool IS_FP16_OUT, bool KT, bool SPLIT, int HD, int QF, bool CA>
__device__ __forceinline__ void qattn_fwd_pp(const AttnParams& p) {
  // HD: head dimension, 128 or 64.  Per 64-key tile a wave runs HD / 16 Q.K^T MFMAs (two key blocks x HD / 32
  // k-steps) and HD / 32 P.V MFMAs; K and V tiles are HD / 16 fragments of 1 KiB each.
  static_assert(HD == 128 || HD == 64, "head_dim 128 or 64");
  constexpr int NQF = HD / 32;  // Q fragments (k-steps of 32) = P.V output blocks of 32 dims
  constexpr int NKF = HD / 16;  // K fragments per tile = V fragments per tile
  constexpr int ROWB = HD;      // bytes of one int8 Q row
  constexpr int KS = ks_per_tile(KT);
  constexpr int NB = kPPNBuf;
  // the K buffers double as the waves' Q / O stage (4 KiB per wave), so they span at least 32 KiB
  constexpr int kKBytes = NB * kBK * HD > 8 * 4096 ? NB * kBK * HD : 8 * 4096;
  __shared__ __align__(16) uint8_t lds_kbuf[kKBytes];
  auto lds_k = reinterpret_cast<uint8_t (*)[kBK * HD]>(lds_kbuf);
  __shared__ __align__(16) uint8_t lds_v[NB][HD * kBK];
  auto buf_of = [](int t) { return (int)((unsigned)t % (unsigned)NB); };
  __shared__ float lds_ks[kKsLdsFloats];
  __shared__ __align__(16) float lds_vs[HD];
  __shared__ __align__(16) float lds_vm[HD];

  int split;
  int64_t b, h, qp;
  pair_of_workgroup<SPLIT, CA>(p, split, b, h, qp);
  // (the non-causal form keeps p.causal as a run-time value, false there: with the diagonal compiled out, another
  // schedule of the loop measured 1 - 2 % slower at 32760 x 32760 x 12 and on 64-wide heads)
  const bool causal = CA && !SPLIT ? true : p.causal != 0;
  const int64_t hk = h / p.group;

  const int tid = threadIdx.x;
  // (wave index in a scalar register, so that every per-wave quantity and branch stays scalar)
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, hf = lane >> 5;
  const int grp = w >> 2, wl = w & 3;
  const int64_t qb = qp * 2 + grp;  // == nQB for the empty second group of an odd block count
  const int64_t q_first = qb * kBQ;
  const int64_t wrow0 = q_first + wl * 32;
  const int64_t qrow = wrow0 + lq;

  // key range of this group, and of the workgroup (its last non-empty group)
  int64_t kv_lim = p.Lk;
  if (p.kv_valid) kv_lim = min(kv_lim, (int64_t)p.kv_valid[b]);
  int64_t kv_end = kv_lim, kv_end_wg = kv_lim;
  if (causal) {
    kv_end = min(kv_lim, q_first + kBQ + p.q_offset);
    kv_end_wg = min(kv_lim, min(qp * 2 + 1, p.nQB - 1) * kBQ + kBQ + p.q_offset);
  }
  // (wave-uniform values in scalar registers: kv_valid comes through a vector load)
  const int kv_end_s = __builtin_amdgcn_readfirstlane((int)kv_end);
  // last key that the wave's first row may see (causal), clamped so that adding a row index stays in range
  constexpr int kNoDiag = INT32_MAX - 128;
  const int diag_s = causal ? __builtin_amdgcn_readfirstlane((int)min(wrow0 + p.q_offset, (int64_t)kNoDiag)) : kNoDiag;
  const int n_tiles = __builtin_amdgcn_readfirstlane(kv_end_wg > 0 ? (int)((kv_end_wg + kBK - 1) / kBK) : 0);
  // this workgroup's key tiles t_lo .. t_end - 1 (the split's run, as in qattn_fwd_kernel)
  const int t_lo = SPLIT ? split * p.tiles_per_split : 0;
  const int t_end = SPLIT ? min(n_tiles, t_lo + p.tiles_per_split) : n_tiles;

  // Q fragments through the wave-private LDS stage (rows row-contiguous, 16-byte chunk c of row r at
  // c ^ (r % chunks per row))
  constexpr int QC = ROWB / 16;  // 16-byte chunks per Q row
  uint8_t* stage = &lds_k[0][0] + w * 4096;
  v4i qf[NQF];
  float qs;
  auto load_q = [&]() {
  if constexpr (QF == QF_BLOCK) {
    // half Q quantized per 128-row block: the four waves of a group exchange their maxima through LDS
    // (q_sm_scale = sm_scale * log2(e) multiplied in first; the logits then take qk_mult = 1)
    __shared__ float lds_qam[8];
    const uint16_t* qh16 = reinterpret_cast<const uint16_t*>(p.q8) + b * p.qsb + h * p.qsh;
    float x[NQF][16];
    const float am_w = quant_q_load<IS_FP16_OUT, QF, NQF, true>(qh16 + qrow * p.qsl, qrow < p.Lq, hf, p.q_sm_scale, x);
    if (lane == 0) lds_qam[w] = am_w;
    __syncthreads();
    const float am = fmaxf(fmaxf(lds_qam[grp * 4], lds_qam[grp * 4 + 1]), fmaxf(lds_qam[grp * 4 + 2], lds_qam[grp * 4 + 3]));
    qs = quant_q_codes<QF, NQF>(x, am, qf) * p.qk_mult;
  } else if constexpr (QF != QF_INT8) {
    // half Q quantized by the wave itself (see quant_q_rows)
    const uint16_t* qh16 = reinterpret_cast<const uint16_t*>(p.q8) + b * p.qsb + h * p.qsh;
    qs = quant_q_rows<IS_FP16_OUT, QF, NQF>(qh16 + qrow * p.qsl, qrow < p.Lq, hf, qf) * p.qk_mult;
  } else {
    const int8_t* qbase = p.q8 + b * p.qsb + h * p.qsh;
#pragma unroll
    for (int i = 0; i < 32 * QC / 64; i++) {
      const int r = i * (64 / QC) + lane / QC, c = lane % QC;
      const int64_t row = wrow0 + r;
      const v4i val = row < p.Lq ? *reinterpret_cast<const v4i*>(qbase + row * p.qsl + c * 16) : v4i{0, 0, 0, 0};
      *reinterpret_cast<v4i*>(stage + r * ROWB + ((c ^ (r % QC)) << 4)) = val;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int m = 0; m < NQF; m++) {
      const int c = 2 * m + hf;
      qf[m] = *reinterpret_cast<const v4i*>(stage + lq * ROWB + ((c ^ (lq % QC)) << 4));
    }
#pragma unroll
    for (int m = 0; m < NQF; m++) asm volatile("" ::"v"(qf[m]));
    const int64_t qbs = min(qb, p.nQB - 1);
    const int64_t qsi = q_scale_index(p, qbs * kBQ + wl * 32 + lq);
    qs = p.q_scale[(b * p.Hq + h) * p.nQS + qsi] * p.qk_mult;
  }
  };
  // int8 Q goes through the LDS stage, which the first DMAs overwrite: it is loaded first.  Half Q is
  // quantized in registers, so its loads are issued behind the first DMAs and their latencies overlap.
  if constexpr (QF == QF_INT8) load_q();
  const float* ks_ptr = p.k_scale + (b * p.Hkv + hk) * p.nKS;

  // K/V tiles in LDS, fragment-major: 1 KiB block j holds MFMA operand fragment j of all 64 lanes (lane l
  // at 16 l), so a lane reads its fragments at one per-tile base address plus constant offsets (no
  // per-fragment address arithmetic) and every read is a contiguous, conflict-free 1 KiB.
  //   K block j (0..7): lane l gets K row (j & 1) * 32 + l % 32, bytes 16 (2 (j >> 1) + l / 32) .. + 16
  //   V block 2 dblk + h (h = 0, 1): lane l gets V^T row dblk * 32 + l % 32, bytes 16 (2 (l / 32) + h) .. + 16
  //     of the tile (the two halves of the lane's P.V A operand)
  // LDS DMA: with HD = 128 wave w fills block w of the K tile and block w of the V tile (two DMAs per wave
  // and tile); with HD = 64 the tiles have four blocks each, waves 0-3 fill the K blocks and waves 4-7 the
  // V blocks (one DMA per wave and tile).
  constexpr int kDmaPerTile = HD == 128 ? 2 : 1;
  const int8_t* kbase = p.k8 + b * p.ksb + hk * p.ksh;
  const uint8_t* vbase = static_cast<const uint8_t*>(p.v) + (b * p.Hkv + hk) * (int64_t)HD * p.Lpad;
  const int64_t kbytes = (p.Lk - 1) * p.ksl + HD;
  const v4u vrsrc = make_rsrc(vbase, (uint32_t)((int64_t)HD * p.Lpad));
  const int wu = __builtin_amdgcn_readfirstlane(w);
  const int kblk = HD == 128 ? wu : wu & 3;  // the K block and V block this wave fills
  uint32_t koff, voff;
  {
    const int kr = (kblk & 1) * 32 + lq, kc = 2 * (kblk >> 1) + hf;
    koff = (uint32_t)(kr * p.ksl + kc * 16);
    const int vd = (kblk >> 1) * 32 + lq, vc = 2 * hf + (kblk & 1);
    voff = (uint32_t)(vd * p.Lpad + vc * 16);
  }
  const int64_t k_step = kBK * p.ksl;
  const uint32_t lds_k0 = lds_addr(&lds_k[0][0]) + kblk * 1024;
  const uint32_t lds_v0 = lds_addr(&lds_v[0][0]) + kblk * 1024;
  const bool dma_k = HD == 128 || wu < 4, dma_v = HD == 128 || wu >= 4;
  auto dma_tile = [&](int t) {
    const int buf = buf_of(t);
    const int64_t kso = (int64_t)t * k_step;
    if (dma_k) lds_dma16(koff, make_rsrc(kbase + kso, (uint32_t)(kbytes - kso)), 0, lds_k0 + buf * (kBK * HD));
    if (dma_v) lds_dma16(voff, vrsrc, (uint32_t)t * kBK, lds_v0 + buf * (HD * kBK));
  };

  v16f o[NQF];
#pragma unroll
  for (int i = 0; i < NQF; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[i][r] = 0.f;
  float m_run = kMInit;
  v4f lacc = {0.f, 0.f, 0.f, 0.f};
  const v8i rs_sel = row_sum_selector();
  v16i kbias;
#pragma unroll
  for (int r = 0; r < 16; r++) kbias[r] = kAccBiasBits;

  if constexpr (QF == QF_INT8) __syncthreads();  // Q fragments are out of the LDS stage before the DMA reuses it
  // the key scales of tiles t_lo .. t_end - 1, from lds_ks[0]
  for (int i = tid; i < (t_end - t_lo) * KS; i += kPPThreads) lds_ks[i] = ks_ptr[k_scale_index(p, t_lo + i / KS, i % KS, KS)];
  if (tid < HD) {
    lds_vs[tid] = p.v_scale[(b * p.Hkv + hk) * HD + tid];
    lds_vm[tid] = p.v_mean ? p.v_mean[(b * p.Hkv + hk) * HD + tid] : 0.f;
  }
  for (int t = t_lo; t < min(t_end, t_lo + 2); t++) dma_tile(t);
  if constexpr (QF != QF_INT8) load_q();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  v16i s[2];
  v8i pf, vf[NQF];
  v4i kf[NKF];
  float cs_a, cs_b;  // logit scales of the tile in the softmax
  auto read_k = [&](int t) {
    const uint8_t* kb = &lds_k[buf_of(t)][lane * 16];
#pragma unroll
    for (int j = 0; j < NKF; j++) kf[j] = *reinterpret_cast<const v4i*>(kb + j * 1024);
  };
  auto read_cs = [&](int t) {
    if constexpr (KT) {
      cs_a = qs * lds_ks[(t - t_lo) * 4 + 2 * hf];
      cs_b = qs * lds_ks[(t - t_lo) * 4 + 2 * hf + 1];
    } else {
      cs_a = cs_b = qs * lds_ks[t - t_lo];
    }
  };
  auto read_v = [&](int t) {
    const uint8_t* vb = &lds_v[buf_of(t)][lane * 16];
#pragma unroll
    for (int dblk = 0; dblk < NQF; dblk++) {
      const v4i a0 = *reinterpret_cast<const v4i*>(vb + (2 * dblk) * 1024);
      const v4i a1 = *reinterpret_cast<const v4i*>(vb + (2 * dblk + 1) * 1024);
      vf[dblk] = v8i{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
    }
  };
  // stage M: P(t-1).V(t-1) and its row sum (operands from the previous stage V), then S^T(t) = K(t).Q^T
  auto pv = [&]() {
#pragma unroll
    for (int dblk = 0; dblk < NQF; dblk++)
      o[dblk] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf[dblk], pf, o[dblk], 0, 0, 0, 0, 0, 0);
    lacc = row_sum_mfma(lacc, pf, rs_sel);
  };
  auto qk = [&]() {
#pragma unroll
    for (int j = 0; j < NKF; j++) {
      const int m = j >> 1, kb = j & 1;
      s[kb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[j], qf[m], m == 0 ? kbias : s[kb], 0, 0, 0);
    }
  };
  auto stage_m = [&](int t, auto first_t) {
    constexpr bool kFirst = decltype(first_t)::value;
    if (!kFirst) read_v(t - 1);
    if constexpr (HD == 128) read_k(t);
    if (!kFirst) pv();
    if constexpr (HD == 64) {
      // (K's fragments behind P.V: V's registers are free by then, which is what fits 128 VGPRs; their latency is
      // covered by the queued MFMAs and the SIMD's other pair)
      __builtin_amdgcn_sched_barrier(0);
      read_k(t);
    }
    qk();
    // the logit scales of the tile, for the softmax of the next stage
    read_cs(t);
    if constexpr (!kFirst && HD == 128) {
      // LDS reads three ahead of the MFMA that consumes them: 3 reads, then (1 MFMA, 2 reads) x 7,
      // then the remaining MFMAs (16 fragment reads + the key-scale read; 13 MFMAs with the row sum)
      __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
      for (int i = 0; i < 7; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
    }
  };
  // stage V: V(t) fragments out of LDS (operands of the next stage M), mask, online softmax, P(t) to e4m3
  auto stage_v = [&](int t) {
    const int k0 = t * kBK;
    const bool masked = (k0 + kBK > kv_end_s) || (k0 + kBK - 1 > diag_s);
    if (masked) {
      int lim = max(min(kv_end_s - k0, kBK), -1);
      lim = min(lim, max(min(diag_s + lq + 1 - k0, kBK), -1));
      lim -= hf * 4;
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (kb * 32 + (r >> 2) * 8 + (r & 3) >= lim) s[kb][r] = INT32_MIN;
    }
    float m_tile;
    if constexpr (!KT) {
      int mx = max(s[0][0], s[0][1]);
#pragma unroll
      for (int r = 2; r < 16; r++) mx = max(mx, s[0][r]);
#pragma unroll
      for (int r = 0; r < 16; r++) mx = max(mx, s[1][r]);
      const auto sw = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
      mx = max((int)sw[0], (int)sw[1]);
      m_tile = mx == INT32_MIN ? kMInit : fmaf(__int_as_float(mx), cs_a, -fmaf(kAccBias, cs_a, kFp8Offset - kLazyTau));
    } else {
      int ma = INT32_MIN, mb = INT32_MIN;
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          if ((r & 3) < 2) ma = max(ma, s[kb][r]);
          else mb = max(mb, s[kb][r]);
        }
      const float fa = ma == INT32_MIN ? kMInit : fmaf(__int_as_float(ma), cs_a, -fmaf(kAccBias, cs_a, kFp8Offset - kLazyTau));
      const float fb = mb == INT32_MIN ? kMInit : fmaf(__int_as_float(mb), cs_b, -fmaf(kAccBias, cs_b, kFp8Offset - kLazyTau));
      const float mt = fmaxf(fa, fb);
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
      m_tile = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    const bool grow = m_tile > m_run + kLazyTau;
    if (__any(grow)) {
      const float m_new = grow ? m_tile : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
#pragma unroll
      for (int i = 0; i < NQF; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] *= alpha;
      row_sum_rescale(lacc, alpha);
      m_run = m_new;
    }
    // u = 8 (s * cs - m - kPLinShift) + 56 (p_e4m3_x4); masked logits give u = -1, P = 0
    const float cs8_a = 8.0f * cs_a, cs8_b = 8.0f * cs_b;
    const float nu_a = fmaf(-8.0f, fmaf(kAccBias, cs_a, m_run), kPLinBias);
    const float nu_b = fmaf(-8.0f, fmaf(kAccBias, cs_b, m_run), kPLinBias);
    auto body = [&](auto mk) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int kb = j >> 2, r0 = (j & 3) * 4;
        float u[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int sv = s[kb][r0 + e];
          u[e] = fmaf(__int_as_float(sv), e < 2 ? cs8_a : cs8_b, e < 2 ? nu_a : nu_b);
          if constexpr (decltype(mk)::value) u[e] = sv == INT32_MIN ? -1.f : u[e];
        }
        pf[j] = p_e4m3_x4(u[0], u[1], u[2], u[3]);
      }
    };
    if (masked) body(std::true_type{});
    else body(std::false_type{});
  };

  auto step = [&](int t, auto first_t) {
    const bool issue = t + 2 < t_end;
    if (issue) dma_tile(t + 2);
    // the matrix stage runs at raised wave priority: the vector-stage wave of the SIMD then cannot
    // delay the issue of its MFMAs (measured faster than equal priorities)
    __builtin_amdgcn_s_setprio(1);
    stage_m(t, first_t);
    __builtin_amdgcn_s_setprio(0);
    // this wave's share of tile t + 1 has landed (tile t + 2 may stay in flight)
    if (issue) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kDmaPerTile) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    pp_barrier();
    stage_v(t);
    pp_barrier();
  };
  if (grp == 1) pp_barrier();
  // the first tile has no P.V of a previous one: peeled, so the loop body has no branch on it
  if (t_lo < t_end) step(t_lo, std::true_type{});
  for (int t = t_lo + 1; t < t_end; t++) step(t, std::false_type{});
  if (grp == 0) pp_barrier();
  if (t_end > t_lo) {
    read_v(t_end - 1);
#pragma unroll
    for (int dblk = 0; dblk < NQF; dblk++)
      o[dblk] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf[dblk], pf, o[dblk], 0, 0, 0, 0, 0, 0);
    lacc = row_sum_mfma(lacc, pf, rs_sel);
  }

  const float l_tot = row_sum_value(lacc, lq);
  if constexpr (SPLIT) {
    // the split's partial (unnormalised O, m, l) for the combine kernel, in qattn_fwd_kernel's layout
    if (qrow >= p.Lq) return;
    const int64_t row = (((int64_t)split * p.B + b) * p.Hq + h) * p.Lq + qrow;
    float* wo = p.ws_o + row * HD;
#pragma unroll
    for (int dblk = 0; dblk < NQF; dblk++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int d = dblk * 32 + g * 8 + hf * 4;
        *reinterpret_cast<v4f*>(wo + d) = v4f{o[dblk][g * 4 + 0], o[dblk][g * 4 + 1], o[dblk][g * 4 + 2], o[dblk][g * 4 + 3]};
      }
    if (hf == 0) {
      p.ws_ml[row * 2 + 0] = m_run;
      p.ws_ml[row * 2 + 1] = l_tot;
    }
    return;
  }

  // ---- epilogue: O / l * v_scale out through the wave's LDS stage (the K buffers are idle now) ----
  const float inv_l = l_tot > 0.f ? 1.0f / l_tot : 0.f;
  uint16_t* obase = static_cast<uint16_t*>(p.o) + b * p.osb + h * p.osh;
  auto store = [&](auto mean_t) {
  constexpr bool kMean = decltype(mean_t)::value;
#pragma unroll
  for (int pass = 0; pass < HD / 64; pass++) {
#pragma unroll
    for (int db = 0; db < 2; db++) {
      const int dblk = pass * 2 + db;
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int d = dblk * 32 + g * 8 + hf * 4;
        const v4f sc = *reinterpret_cast<const v4f*>(&lds_vs[d]);
        float f[4];
        const v4f vm = kMean ? *reinterpret_cast<const v4f*>(&lds_vm[d]) : v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = epilogue_value<kMean>(o[dblk][g * 4 + e], inv_l, sc[e], vm[e]);
        const v2u packed{pack_half2<IS_FP16_OUT>(f[0], f[1]), pack_half2<IS_FP16_OUT>(f[2], f[3])};
        const int c = db * 4 + g;
        *reinterpret_cast<v2u*>(stage + lq * 128 + ((c ^ (lq & 7)) << 4) + hf * 8) = packed;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = i * 8 + (lane >> 3), c = lane & 7;
      const v4u val = *reinterpret_cast<const v4u*>(stage + r * 128 + ((c ^ (r & 7)) << 4));
      const int64_t row = wrow0 + r;
      if (row < p.Lq) *reinterpret_cast<v4u*>(obase + row * p.osl + pass * 64 + c * 8) = val;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  };
  if (p.v_mean) store(std::true_type{});
  else store(std::false_type{});
  if (p.lse && hf == 0 && qrow < p.Lq)
    p.lse[(b * p.Hq + h) * p.Lq + qrow] = l_tot > 0.f ? __builtin_log2f(l_tot) + m_run : -INFINITY;
}

// Head dim 64: the softmax per query-key pair does not shrink with the head dimension (~450 VALU cycles a tile against
// 288 MFMA ones), so one pair of waves per SIMD left both pipes waiting.  Unsplit launches are held to 128 VGPRs: two
// workgroups per CU (80 KiB of LDS each), two pairs per SIMD.  2 x 4680 x 4680 x 24 292 -> 238 us a call, 16000 x
// 16000 x 12 608 -> 513, 30000 x 300 x 16 98 -> 62.  (Three waves per SIMD as three groups of one workgroup, the
// softmax cut in two stages by a barrier: 285 us, and 4096 x 4096 x 24 slower, 160 against 136 us.  The KV-split form
// spills 30 registers at 128 and keeps one workgroup per CU.)
template <bool IS_FP16_OUT, bool KT, bool SPLIT, int HD, int QF, bool CA>
__global__ __launch_bounds__(kPPThreads, HD == 64 && !SPLIT ? 4 : 1) void qattn_fwd_pp_kernel(AttnParams p) {
  qattn_fwd_pp<IS_FP16_OUT, KT, SPLIT, HD, QF, CA>(p);
}

// ---- resident K/V: short key ranges (at most kResMaxTiles tiles, e.g. text cross-attention) ----
//
// The whole key range of a head (K int8 and e4m3 V, fragment-major as in the streaming kernels) is
// loaded into LDS once per workgroup; then each of the 12 waves walks its own 32-row query blocks over
// the resident tiles with no workgroup barrier at all: Q fragments come straight from global memory, the
// three waves of a SIMD drift apart freely so that one's softmax and Q loads overlap the others' MFMAs,
// and O leaves through a 2 KiB wave-private LDS stage as whole 64-byte row segments.  Twelve waves leave
// each 168 VGPRs: K and V fragments are read from LDS next to their MFMAs, and the next block's Q is not
// prefetched into registers (three waves per SIMD hide its latency better than two waves with prefetch:
// C4 0.63 -> 0.615 ms).  Per element the arithmetic is that of qattn_fwd_kernel
// (same MFMA chains, masking, lazy running max, FP8 offset, row sums on the matrix pipe), so the
// results are identical to it.
constexpr int kResMaxTiles = 8;
constexpr int kResThreads = 768;
constexpr int kResWaves = kResThreads / 64;

template <bool IS_FP16_OUT, bool KT, int QF = QF_INT8>
__global__ __launch_bounds__(kResThreads) void qattn_fwd_res_kernel(AttnParams p) {
  constexpr int KS = ks_per_tile(KT);
  constexpr int NW = kResThreads / 64;
  __shared__ __align__(16) uint8_t lds_k[kResMaxTiles][kBK * kD];
  __shared__ __align__(16) uint8_t lds_v[kResMaxTiles][kD * kBK];
  __shared__ __align__(16) uint8_t lds_o[NW][32 * 64];
  __shared__ __align__(16) uint8_t lds_pf[QF == QF_BLOCK ? NW : 1][256];  // landing slots of the Q prefetch, never read
  __shared__ float lds_ks[kResMaxTiles * 4];
  __shared__ __align__(16) float lds_vs[kD];
  __shared__ __align__(16) float lds_vm[kD];

  const int64_t wg = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t chunk = wg % p.n_chunk;
  const int64_t h = (wg / p.n_chunk) % p.Hq;
  const int64_t b = wg / (p.n_chunk * p.Hq);
  const int64_t hk = h / p.group;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, hf = lane >> 5;
  const v8i rs_sel = row_sum_selector();

  // key range (wave-uniform, in scalar registers: kv_valid comes through a vector load)
  int64_t kv_lim = p.Lk;
  if (p.kv_valid) kv_lim = min(kv_lim, (int64_t)p.kv_valid[b]);
  const int64_t kv_end = __builtin_amdgcn_readfirstlane((int)max(kv_lim, (int64_t)0));
  const int n_tiles = (int)((kv_end + kBK - 1) / kBK);

  // ---- the key range into LDS: tile t of K / V in lds_k[t] / lds_v[t], fragment-major ----
  {
    const int8_t* kbase = p.k8 + b * p.ksb + hk * p.ksh;
    const uint8_t* vbase = static_cast<const uint8_t*>(p.v) + (b * p.Hkv + hk) * (int64_t)kD * p.Lpad;
    const int64_t kbytes = (p.Lk - 1) * p.ksl + kD;
    const v4u vrsrc = make_rsrc(vbase, (uint32_t)((int64_t)kD * p.Lpad));
    // per tile, wave w < 8 fills 1 KiB block w of the K tile and block w of the V tile (one DMA
    // instruction each), so waves 0-7 cover both tiles
    const int j = w;
    const uint32_t koff = (uint32_t)(((j & 1) * 32 + lq) * p.ksl + (2 * (j >> 1) + hf) * 16);
    const uint32_t voff = (uint32_t)(((j >> 1) * 32 + lq) * p.Lpad + (2 * hf + (j & 1)) * 16);
    const uint32_t lk0 = lds_addr(&lds_k[0][0]) + w * 1024, lv0 = lds_addr(&lds_v[0][0]) + w * 1024;
    if (w < 8) {
      for (int t = 0; t < n_tiles; t++) {
        const int64_t kso = (int64_t)t * kBK * p.ksl;
        const v4u krsrc = make_rsrc(kbase + kso, (uint32_t)(kbytes - kso));
        lds_dma16(koff, krsrc, 0, lk0 + t * (kBK * kD));
        lds_dma16(voff, vrsrc, (uint32_t)t * kBK, lv0 + t * (kD * kBK));
      }
    }
    const float* ks_ptr = p.k_scale + (b * p.Hkv + hk) * p.nKS;
    if (tid < n_tiles * KS) lds_ks[tid] = ks_ptr[k_scale_index(p, tid / KS, tid % KS, KS)];
    if (tid < kD) {
      lds_vs[tid] = p.v_scale[(b * p.Hkv + hk) * kD + tid];
      lds_vm[tid] = p.v_mean ? p.v_mean[(b * p.Hkv + hk) * kD + tid] : 0.f;
    }
  }

  // this wave's 32-row blocks: wb = wb0 + w, wb0 + w + NW, ... below wb_end
  const int64_t n_wb = (p.Lq + 31) / 32;
  const int64_t wb0 = chunk * p.wb_per_wg;
  const int64_t wb_end = min(n_wb, wb0 + p.wb_per_wg);
  const int8_t* qhead = p.q8 + b * p.qsb + h * p.qsh;
  const float* qs_tab = p.q_scale + (b * p.Hq + h) * p.nQS;
  // lane (lq, hf) holds bytes 32 m + 16 hf .. + 16 of query row lq (the MFMA B operand)
  auto load_q = [&](int64_t wb, v4i (&qf)[4]) {
    const int64_t row = wb * 32 + lq;
#pragma unroll
    for (int m = 0; m < 4; m++)
      qf[m] = row < p.Lq ? *reinterpret_cast<const v4i*>(qhead + row * p.qsl + m * 32 + hf * 16) : v4i{0, 0, 0, 0};
  };
  const uint16_t* qhead16 = reinterpret_cast<const uint16_t*>(p.q8) + b * p.qsb + h * p.qsh;
  v4i qf[4];
  int64_t wb = wb0 + w;
  v16i kbias;
#pragma unroll
  for (int r = 0; r < 16; r++) kbias[r] = kAccBiasBits;
  uint8_t* stage = &lds_o[w][0];
  uint16_t* obase = static_cast<uint16_t*>(p.o) + b * p.osb + h * p.osh;

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // every wave's share of the key range has landed

  // per-block Q (QF_BLOCK): the layout starts every chunk on a 128-row block, so in each round waves 4 g ..
  // 4 g + 3 hold the four 32-row blocks of one Q block and exchange their maxima through LDS; every wave
  // runs all rounds of the chunk (a wave past the chunk's end takes zero rows, contributes 0 to the maxima,
  // joins the barrier and stores nothing)
  const int64_t wb_lim = QF == QF_BLOCK ? wb0 + (wb_end - wb0 + NW - 1) / NW * NW : wb_end;
  for (int rnd = 0; wb < wb_lim; rnd++, wb += NW) {
    const bool live = QF != QF_BLOCK || wb < wb_end;
    float qs;
    if constexpr (QF == QF_INT8) {
      load_q(wb, qf);
      qs = qs_tab[q_scale_index(p, wb * 32 + lq)] * p.qk_mult;
    } else if constexpr (QF == QF_BLOCK) {
      // (double-buffered by round: a wave writes round r + 2's maximum only after the barrier of round r + 1,
      // which every wave reaches after reading round r's)
      // (only the raw half words stay live across the barrier, and the values are formed again after it:
      // 64 fp32 values per lane would not fit beside the kernel's other registers)
      __shared__ float lds_qam[2][NW];
      const int64_t row = wb * 32 + lq;
      v4u raw[4][2];
      quant_q_raw<4>(qhead16 + row * p.qsl, live && row < p.Lq, hf, raw);
      float am_w;
      {
        float x[4][16];
        quant_q_unpack<IS_FP16_OUT, 4, true>(raw, p.q_sm_scale, x);
        am_w = quant_q_amax<QF, 4>(x);
      }
      if (lane == 0) lds_qam[rnd & 1][w] = am_w;
      __syncthreads();
      const float* g4 = &lds_qam[rnd & 1][w & ~3];
      const float am = fmaxf(fmaxf(g4[0], g4[1]), fmaxf(g4[2], g4[3]));
#pragma unroll
      for (int m = 0; m < 4; m++) asm volatile("" : "+v"(raw[m][0]), "+v"(raw[m][1]));  // (no reuse of the first unpack)
      float x[4][16];
      quant_q_unpack<IS_FP16_OUT, 4, true>(raw, p.q_sm_scale, x);
      qs = quant_q_codes<QF, 4>(x, am, qf) * p.qk_mult;
    } else {
      const int64_t row = wb * 32 + lq;
      qs = quant_q_rows<IS_FP16_OUT, QF, 4>(qhead16 + row * p.qsl, row < p.Lq, hf, qf) * p.qk_mult;
    }
    const int64_t wrow0 = wb * 32, qrow = wrow0 + lq;
    // Per block, the round barrier lines the waves up, so all of them would load their next Q rows at once
    // and wait out the HBM latency together: the wave's next 32 rows go into L2 while this block runs, one
    // dword of every 128-byte line (lane (lq, hf): row lq, line hf) DMA'd into the wave's landing slot so
    // that no register waits for it.  (The free-running forms stagger their loads by themselves: the
    // prefetch measured no gain there.)
    if constexpr (QF == QF_BLOCK) {
      if (wb + NW < wb_end) {
        constexpr int kQB = 2;  // bytes per Q element
        const int64_t nrow0 = (wb + NW) * 32;
        const uint8_t* nbase = reinterpret_cast<const uint8_t*>(p.q8) + (b * p.qsb + h * p.qsh + nrow0 * p.qsl) * kQB;
        const int64_t rem = ((p.Lq - 1 - nrow0) * p.qsl + kD) * kQB;  // bytes to the end of the last row
        lds_dma4((uint32_t)((lq * p.qsl + hf * 64) * kQB), make_rsrc(nbase, (uint32_t)min(rem, (int64_t)UINT32_MAX)), 0,
                 lds_addr(&lds_pf[w][0]));
      }
    }

    v16f o[4];
    v4f lacc;
    float m_run = kMInit;
    // One key tile.  The first tile of a block is peeled: its running max is the tile max and its P.V
    // starts from zero accumulators, which is what the general step computes there (the rescale factor
    // exp2(kMInit - m) is 0 while O and l are still 0, and a first tile always holds a valid key),
    // without zeroing O and l and without the O rescale.
    auto tile = [&](int t, auto first_t) {
      constexpr bool kFirst = decltype(first_t)::value;
      float cs_a, cs_b;
      if constexpr (KT) {
        cs_a = qs * lds_ks[t * 4 + 2 * hf];
        cs_b = qs * lds_ks[t * 4 + 2 * hf + 1];
      } else {
        cs_a = cs_b = qs * lds_ks[t];
      }
      v16i s[2];
      {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const int m = j >> 1, kb = j & 1;
          const v4i kf = *reinterpret_cast<const v4i*>(&lds_k[t][j * 1024 + lane * 16]);
          s[kb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[m], m == 0 ? kbias : s[kb], 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
      }
      const int64_t k0 = (int64_t)t * kBK;
      const bool masked = k0 + kBK > kv_end;
      // Masked logits become -inf (as int32 below every biased logit, so the max skips them), whose
      // exp2 is exactly 0: no per-logit select in the softmax.  A zero logit scale (an all-zero block
      // under the Triton rounding) would turn -inf into NaN there, so a wave with one falls back to
      // INT32_MIN and the select.
      bool select_mask = false;
      if (masked) {
        select_mask = !__all(cs_a > 0.f && cs_b > 0.f);
        const int mval = select_mask ? INT32_MIN : kMaskedLogitBits;
        int lim = (int)min(kv_end - k0, (int64_t)kBK) - hf * 4;
        asm volatile("" : "+v"(lim));  // (compared here, not as 32 lane masks kept in registers across the loops)
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
          for (int r = 0; r < 16; r++)
            if (kb * 32 + (r >> 2) * 8 + (r & 3) >= lim) s[kb][r] = mval;
      }
      auto all_masked = [](int x) { return x == INT32_MIN || x == kMaskedLogitBits; };
      float m_tile;
      if constexpr (!KT) {
        int mx = max(s[0][0], s[0][1]);
#pragma unroll
        for (int r = 2; r < 16; r++) mx = max(mx, s[0][r]);
#pragma unroll
        for (int r = 0; r < 16; r++) mx = max(mx, s[1][r]);
        const auto sw = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
        mx = max((int)sw[0], (int)sw[1]);
        m_tile = all_masked(mx) ? kMInit : fmaf(__int_as_float(mx), cs_a, -fmaf(kAccBias, cs_a, kFp8Offset - kLazyTau));
      } else {
        int ma = INT32_MIN, mb = INT32_MIN;
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            if ((r & 3) < 2) ma = max(ma, s[kb][r]);
            else mb = max(mb, s[kb][r]);
          }
        const float fa = all_masked(ma) ? kMInit : fmaf(__int_as_float(ma), cs_a, -fmaf(kAccBias, cs_a, kFp8Offset - kLazyTau));
        const float fb = all_masked(mb) ? kMInit : fmaf(__int_as_float(mb), cs_b, -fmaf(kAccBias, cs_b, kFp8Offset - kLazyTau));
        const float mt = fmaxf(fa, fb);
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
        m_tile = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      }
      if constexpr (kFirst) {
        m_run = m_tile;
      } else {
        const bool grow = m_tile > m_run + kLazyTau;
        if (__any(grow)) {
          const float m_new = grow ? m_tile : m_run;
          const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
#pragma unroll
          for (int i = 0; i < 4; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[i][r] *= alpha;
          row_sum_rescale(lacc, alpha);
          m_run = m_new;
        }
      }
      // u = 8 (s * cs - m - kPLinShift) + 56 (p_e4m3_x4); masked logits give u = -1, P = 0
      const float cs8_a = 8.0f * cs_a, cs8_b = 8.0f * cs_b;
      const float nu_a = fmaf(-8.0f, fmaf(kAccBias, cs_a, m_run), kPLinBias);
      const float nu_b = fmaf(-8.0f, fmaf(kAccBias, cs_b, m_run), kPLinBias);
      v8i pf;
      auto body = [&](auto mk) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const int kb = j >> 2, r0 = (j & 3) * 4;
          float u[4];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const int sv = s[kb][r0 + e];
            u[e] = fmaf(__int_as_float(sv), e < 2 ? cs8_a : cs8_b, e < 2 ? nu_a : nu_b);
            if constexpr (decltype(mk)::value) u[e] = sv == INT32_MIN ? -1.f : u[e];
          }
          pf[j] = p_e4m3_x4(u[0], u[1], u[2], u[3]);
        }
      };
      if (select_mask) body(std::true_type{});
      else body(std::false_type{});
      const v16f zero = {};
#pragma unroll
      for (int dblk = 0; dblk < 4; dblk++) {
        const v4i a0 = *reinterpret_cast<const v4i*>(&lds_v[t][(2 * dblk) * 1024 + lane * 16]);
        const v4i a1 = *reinterpret_cast<const v4i*>(&lds_v[t][(2 * dblk + 1) * 1024 + lane * 16]);
        const v8i vf = v8i{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
        o[dblk] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf, pf, kFirst ? zero : o[dblk], 0, 0, 0, 0, 0, 0);
      }
      lacc = row_sum_mfma(kFirst ? v4f{0.f, 0.f, 0.f, 0.f} : lacc, pf, rs_sel);
    };
    if (n_tiles > 0) {
      tile(0, std::true_type{});
      for (int t = 1; t < n_tiles; t++) tile(t, std::false_type{});
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] = 0.f;
      lacc = v4f{0.f, 0.f, 0.f, 0.f};
    }

    // ---- epilogue: O / l * v_scale (+ v_mean), 32 channels per pass through the 2 KiB stage ----
    const float l_tot = row_sum_value(lacc, lq);
    const float inv_l = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    auto store = [&](auto mean_t) {
    constexpr bool kMean = decltype(mean_t)::value;
#pragma unroll
    for (int dblk = 0; dblk < 4; dblk++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int d = dblk * 32 + g * 8 + hf * 4;
        const v4f sc = *reinterpret_cast<const v4f*>(&lds_vs[d]);
        const v4f vm = kMean ? *reinterpret_cast<const v4f*>(&lds_vm[d]) : v4f{0.f, 0.f, 0.f, 0.f};
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = epilogue_value<kMean>(o[dblk][g * 4 + e], inv_l, sc[e], vm[e]);
        const v2u packed{pack_half2<IS_FP16_OUT>(f[0], f[1]), pack_half2<IS_FP16_OUT>(f[2], f[3])};
        // stage row lq: 4 chunks of 16 B (8 channels), chunk g stored at g ^ (lq & 3)
        *reinterpret_cast<v2u*>(stage + lq * 64 + ((g ^ (lq & 3)) << 4) + hf * 8) = packed;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int id = i * 64 + lane, r = id >> 2, c = id & 3;
        const v4u val = *reinterpret_cast<const v4u*>(stage + r * 64 + ((c ^ (r & 3)) << 4));
        const int64_t row = wrow0 + r;
        if (live && row < p.Lq) *reinterpret_cast<v4u*>(obase + row * p.osl + dblk * 32 + c * 8) = val;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    };
    if (p.v_mean) store(std::true_type{});
    else store(std::false_type{});
    if (p.lse && hf == 0 && live && qrow < p.Lq)
      p.lse[(b * p.Hq + h) * p.Lq + qrow] = l_tot > 0.f ? __builtin_log2f(l_tot) + m_run : -INFINITY;
  }
  if constexpr (QF == QF_BLOCK) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no prefetch left in flight
}

// Merge the KV-split partials: four channels per lane, so a wave reads 1 KiB of whole rows of each split.  HBM- and
// latency-bound ((D + 2) 4 bytes per row and split): the partials of four splits are loaded at once, the first four ahead
// of the maxima, and the row is split into (batch, head, query) by 32-bit divisions where the rows fit them (one row per
// wave, a split at a time and 64-bit divisions: 1560 x 12 rows 12.9 us, 10.0 now; a call at 300 x 20000 x 8 116 -> 110).
template <bool IS_FP16_OUT, int HD = kD>
__global__ __launch_bounds__(256) void qattn_combine_kernel(AttnParams p) {
  constexpr int E = 4, TPR = HD / E;  // channels per lane, lanes per row
  constexpr int NS = 4;               // splits loaded together
  const int64_t row = (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;  // over B*Hq*Lq
  const int d0 = (threadIdx.x % TPR) * E;
  const int64_t total = p.B * p.Hq * p.Lq;
  if (row >= total) return;
  int64_t b, h, qrow;
  if (total <= (int64_t)UINT32_MAX) {
    const uint32_t r = (uint32_t)row, lq = (uint32_t)p.Lq, hq = (uint32_t)p.Hq;
    const uint32_t bh = r / lq;
    qrow = r - bh * lq;
    b = bh / hq;
    h = bh - (uint32_t)b * hq;
  } else {
    qrow = row % p.Lq;
    h = (row / p.Lq) % p.Hq;
    b = row / (p.Lq * p.Hq);
  }
  const int64_t hk = h / p.group;
  const int ns = p.nsplit;
  // (past the last split the loads repeat it and are not used)
  v4f part[NS];
  auto load = [&](int s0) {
#pragma unroll
    for (int i = 0; i < NS; i++)
      part[i] = *reinterpret_cast<const v4f*>(p.ws_o + (min(s0 + i, ns - 1) * total + row) * HD + d0);
  };
  load(0);
  float M = kMInit;
  for (int s0 = 0; s0 < ns; s0 += NS) {
    float m[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) m[i] = p.ws_ml[(min(s0 + i, ns - 1) * total + row) * 2];
#pragma unroll
    for (int i = 0; i < NS; i++) M = fmaxf(M, m[i]);
  }
  float L = 0.f, a[E];
#pragma unroll
  for (int e = 0; e < E; e++) a[e] = 0.f;
  for (int s0 = 0; s0 < ns; s0 += NS) {
    if (s0) load(s0);
    float m[NS], l[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) {
      const float* ml = p.ws_ml + (min(s0 + i, ns - 1) * total + row) * 2;
      m[i] = ml[0];
      l[i] = ml[1];
    }
#pragma unroll
    for (int i = 0; i < NS; i++) {
      if (s0 + i >= ns) break;
      const float f = __builtin_amdgcn_exp2f(m[i] - M);
      L += l[i] * f;
#pragma unroll
      for (int e = 0; e < E; e++) a[e] += part[i][e] * f;
    }
  }
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  const float* vs = p.v_scale ? p.v_scale + (b * p.Hkv + hk) * HD + d0 : nullptr;
  const float* vm = p.v_mean ? p.v_mean + (b * p.Hkv + hk) * HD + d0 : nullptr;
  float r[E];
#pragma unroll
  for (int e = 0; e < E; e++)
    r[e] = vm ? epilogue_value<true>(a[e], inv, vs ? vs[e] : 1.f, vm[e])
              : epilogue_value<false>(a[e], inv, vs ? vs[e] : 1.f, 0.f);
  const v2u packed{pack_half2<IS_FP16_OUT>(r[0], r[1]), pack_half2<IS_FP16_OUT>(r[2], r[3])};
  uint16_t* orow = static_cast<uint16_t*>(p.o) + b * p.osb + qrow * p.osl + h * p.osh + d0;
  *reinterpret_cast<v2u*>(orow) = packed;
  if (p.lse && d0 == 0) p.lse[(b * p.Hq + h) * p.Lq + qrow] = L > 0.f ? __builtin_log2f(L) + M : -INFINITY;
}

// Natural-log LSE of the original K from the kernels' log2-domain LSE against K - km: lse * ln 2 + (q . km) sm_scale,
// in place.  One pass over Q (HBM-bound: 2 B per element), 16 bytes of a row per lane and the rows in Q's memory order
// (torch's form took six launches, 70 us of them next to a 140 us attention at 2 x 4096 x 16: the matvec alone 45).
template <bool IS_FP16, int D>
__global__ __launch_bounds__(256) void lse_finish_kernel(float* lse, const uint16_t* q, int64_t sb, int64_t sl, int64_t sh,
                                                         const uint16_t* km, int64_t L, int64_t Hq, int group,
                                                         int64_t rows, float sm_scale) {
  constexpr int TPR = D / 8;  // lanes per row
  const int64_t r = (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  const int dc = threadIdx.x % TPR;
  if (r >= rows) return;  // (whole rows: their lanes leave together)
  // r counts rows with the smaller of the sequence and head strides innermost
  int64_t b, h, l;
  if (sh < sl) {
    h = r % Hq;
    l = (r / Hq) % L;
  } else {
    l = r % L;
    h = (r / L) % Hq;
  }
  b = r / (Hq * L);
  const v4u x = *reinterpret_cast<const v4u*>(q + b * sb + l * sl + h * sh + dc * 8);
  const v4u m = *reinterpret_cast<const v4u*>(km + (b * (Hq / group) + h / group) * D + dc * 8);
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    s = fmaf(half_to_f32<IS_FP16>((uint16_t)(x[e] & 0xffffu)), half_to_f32<IS_FP16>((uint16_t)(m[e] & 0xffffu)), s);
    s = fmaf(half_to_f32<IS_FP16>((uint16_t)(x[e] >> 16)), half_to_f32<IS_FP16>((uint16_t)(m[e] >> 16)), s);
  }
#pragma unroll
  for (int o = 1; o < TPR; o <<= 1) s += __shfl_xor(s, o, 64);
  if (dc == 0) {
    float* p = lse + (b * Hq + h) * L + l;
    *p = *p / 1.44269504f + s * sm_scale;
  }
}

void launch_combine(const AttnParams& p, int out_dtype, int64_t D, hipStream_t st) {
  const int64_t per = 256 / (D / 4), g = (p.B * p.Hq * p.Lq + per - 1) / per;
  if (D == 64) {
    if (out_dtype == QATTN_BF16) qattn_combine_kernel<false, 64><<<g, 256, 0, st>>>(p);
    else qattn_combine_kernel<true, 64><<<g, 256, 0, st>>>(p);
  } else {
    if (out_dtype == QATTN_BF16) qattn_combine_kernel<false><<<g, 256, 0, st>>>(p);
    else qattn_combine_kernel<true><<<g, 256, 0, st>>>(p);
  }
}

}  // namespace qattn

using namespace qattn;

static bool is_thread_gran(int g) { return g == QATTN_GRAN_THREAD || g == QATTN_GRAN_THREAD_SM90; }

// key tiles one workgroup can cover (its k_scales are staged in LDS)
static int64_t max_tiles_per_split(bool kt) { return kKsLdsFloats / ks_per_tile(kt); }

// Ping-pong KV-split launches take whole pairs of query blocks; an odd block count leaves the last pair's
// second wave group idle, allowed when that is at most 1/6 of the groups.
static bool pp_split_fits(int64_t nqb) { return nqb % 2 == 0 || nqb >= 5; }

static int num_splits_for(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int64_t max_tiles, bool pp) {
  const int64_t nqb = (Lq + kBQ - 1) / kBQ;
  const int64_t wgs = B * Hq * nqb;
  const int64_t nkb = (Lk + kBK - 1) / kBK;
  if (wgs <= 0 || nkb <= 0) return 1;
  // 256 CUs x 2 resident workgroups.  Split only when the grid leaves CUs without any workgroup: at
  // 256 or more workgroups the combine traffic of a split costs more than the idle half-slots it fills
  // (C5, 444 workgroups: 0.63 ms unsplit against 0.79 ms with 3 splits); every split still gets at least
  // 8 key tiles.  (Block-sparse launches, pp = false, keep this count of one-block workgroups and all key tiles, though
  // theirs hold two blocks, one to a CU, and a split takes its share of the kept tiles' list as if all were kept: how
  // many are is not known here, and no count for them was measured.)
  const int64_t target = 1024;
  const int64_t min_s = (nkb + max_tiles - 1) / max_tiles;
  if (wgs >= target / 4) return (int)min_s;
  if (pp && pp_split_fits(nqb)) {
    // FP8 dense launches: splits for one round of at most 256 ping-pong workgroups (one per CU).  Against
    // the earlier count (about 1024 one-block workgroups) 5-27 % faster at 512-4680 queries over 8k-32k keys,
    // with either kernel (fewer splits, less combine traffic)
    const int64_t pairs = B * Hq * ((nqb + 1) / 2);
    const int64_t s = std::min<int64_t>(std::min<int64_t>(256 / pairs, nkb / 8), 32);
    return (int)std::max<int64_t>(min_s, std::max<int64_t>(s, 1));
  }
  int64_t s = (target + wgs - 1) / wgs;
  s = std::min<int64_t>(s, nkb / 8);
  return (int)std::max<int64_t>(min_s, std::min<int64_t>(s, 32));
}

extern "C" int qattn_fwd_num_splits(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq) {
  return num_splits_for(B, Lq, Lk, Hq, max_tiles_per_split(false), true);
}

// the split count of a dense launch (pv: PvKind)
static int dense_num_splits(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int pv, int gran) {
  if (pv == PV_FP8) return num_splits_for(B, Lq, Lk, Hq, max_tiles_per_split(is_thread_gran(gran)), true);
  return half_num_splits(B * Hq, (Lq + kBQ - 1) / kBQ, (Lk + kBK - 1) / kBK, is_thread_gran(gran));
}

extern "C" int qattn_fwd_ex_num_splits(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int v_kind, int qk_quant_gran) {
  return dense_num_splits(B, Lq, Lk, Hq, v_kind == QATTN_V_FP8 ? PV_FP8 : PV_BF16, qk_quant_gran);
}

static int blocks_per_workgroup(int64_t bh, int64_t nqb, int64_t nkb);

extern "C" int qattn_fwd_ex_blocks_per_workgroup(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int v_kind,
                                                 int qk_quant_gran, int causal) {
  if (v_kind != QATTN_V_FP8 || causal || B <= 0 || Lq <= 0 || Lk <= 0 || Hq <= 0) return 1;
  const int64_t nkb = (Lk + kBK - 1) / kBK, nqb = (Lq + kBQ - 1) / kBQ;
  if (nkb >= kMqAutoMaxTiles) return 1;
  if (num_splits_for(B, Lq, Lk, Hq, max_tiles_per_split(is_thread_gran(qk_quant_gran)), true) != 1)
    return 1;
  return blocks_per_workgroup(B * Hq, nqb, nkb);
}

extern "C" size_t qattn_fwd_workspace_size(int64_t B, int64_t Lq, int64_t Hq, int64_t D, int num_splits) {
  if (num_splits <= 1) return 0;
  return (size_t)num_splits * B * Hq * Lq * (D + 2) * sizeof(float);
}

// Kernel selection.  Dense FP8 launches without a KV split run the ping-pong kernel when its grid (one
// workgroup per two query blocks, one workgroup per CU) fills the 256 CUs, the multi-block variant of
// qattn_fwd_kernel for short key ranges (blocks_per_workgroup > 1), and qattn_fwd_kernel otherwise.
// Half-P.V launches (dense, block-sparse, varlen) have one kernel of their own (attn_half.hip) and report
// QATTN_KERNEL_ONE_BLOCK whatever the override.  A thread-local override
// (qattn_set_kernel) forces one of the applicable kernels, so tests can compare them on small shapes.
static thread_local int t_kernel_override = QATTN_KERNEL_AUTO;
static thread_local int t_last_kernel = QATTN_KERNEL_AUTO;

extern "C" int qattn_set_kernel(int kernel) {
  const int prev = t_kernel_override;
  if (kernel >= QATTN_KERNEL_AUTO && kernel <= QATTN_KERNEL_RESIDENT) t_kernel_override = kernel;
  return prev;
}

extern "C" int qattn_last_kernel(void) { return t_last_kernel; }

// the kernel a launch runs, given its split count and whether the multi-block / resident layouts apply
static int pick_kernel(int pv, bool sparse, int ns, int causal, int64_t B, int64_t Hq, int64_t nQB, int qpw_auto,
                       bool mq_ok, bool res_ok) {
  if (pv != PV_FP8 || sparse) return QATTN_KERNEL_ONE_BLOCK;
  const int ov = t_kernel_override;
  // KV-split launches: the ping-pong kernel when its grid of pairs x splits is one round of 128 to 256
  // workgroups over whole pairs (the split count the automatic rule picks for it: 3-5 % faster than the
  // one-block kernel with the same splits), else the one-block kernel (also for tiny grids such as C1's
  // 16 ping-pong workgroups, where its 32 run 1 us faster)
  if (ns > 1) {
    if (ov == QATTN_KERNEL_PINGPONG) return QATTN_KERNEL_PINGPONG;
    const int64_t g = B * Hq * ((nQB + 1) / 2) * ns;
    const bool pp = ov == QATTN_KERNEL_AUTO && pp_split_fits(nQB) && g >= 128 && g <= 256;
    return pp ? QATTN_KERNEL_PINGPONG : QATTN_KERNEL_ONE_BLOCK;
  }
  if (ov == QATTN_KERNEL_PINGPONG || ov == QATTN_KERNEL_ONE_BLOCK) return ov;
  if (ov == QATTN_KERNEL_MULTI_BLOCK && mq_ok && !causal) return QATTN_KERNEL_MULTI_BLOCK;
  if (ov == QATTN_KERNEL_RESIDENT && res_ok) return QATTN_KERNEL_RESIDENT;
  if (res_ok) return QATTN_KERNEL_RESIDENT;
  if (qpw_auto > 1) return QATTN_KERNEL_MULTI_BLOCK;
  // The ping-pong kernel (one workgroup of two 128-row query blocks per CU) against one-block workgroups
  // (one query block, two per CU), in rounds of the 256 CUs: a ping-pong round takes about T (one pair
  // over the whole key range), a full round of one-block workgroups ~1.1 T (C2: 3.9 against 3.45 ms for
  // the same rounds), a last round with a single one-block workgroup on a CU ~0.9 T (one wave per SIMD:
  // 0.454 against 0.512 ms at 2048 x 32760 x 12).  At the C5 chunk shape with 8, 10, 11 and 12 heads (152
  // to 228 pairs) the ping-pong grid is 4-9 % faster.
  const int64_t pairs = B * Hq * ((nQB + 1) / 2), blocks = B * Hq * nQB;
  const double pp_cost = (double)((pairs + 255) / 256);
  const int64_t rem = blocks % 512;
  const double ob_cost = (double)(blocks / 512) * 1.1 + (rem == 0 ? 0.0 : rem > 256 ? 1.1 : 0.9);
  return pp_cost <= ob_cost ? QATTN_KERNEL_PINGPONG : QATTN_KERNEL_ONE_BLOCK;
}

// Resident-K/V launches: the 32-row wave blocks of each (batch, head) are cut into n_chunk workgroups
// of wb_per_wg blocks.  One workgroup runs per CU (its LDS holds the key range), its kResWaves waves each
// taking every kResWaves-th block; the cut minimises full rounds of 256 workgroups x (wave rounds per
// workgroup + one round of start-up for the key-range load).
static void resident_layout(int64_t bh, int64_t n_wb, int64_t& wb_per_wg, int64_t& n_chunk, int64_t align = 1) {
  double best = 1e300;
  wb_per_wg = (n_wb + align - 1) / align * align;
  n_chunk = 1;
  for (int64_t c = 1; c <= std::max<int64_t>(1, (n_wb + kResWaves - 1) / kResWaves); c++) {
    const int64_t per = ((n_wb + c - 1) / c + align - 1) / align * align;
    const int64_t chunks = (n_wb + per - 1) / per;
    const int64_t rounds = (bh * chunks + 255) / 256;
    const double cost = (double)rounds * (double)((per + kResWaves - 1) / kResWaves + 1);
    if (cost < best) {
      best = cost;
      wb_per_wg = per;
      n_chunk = chunks;
    }
  }
}

// the ping-pong kernel of a launch: KV-split (and the combine), causal or neither
template <bool KT, int HD, int QF>
static void launch_pp(AttnParams& p, int dtype, int ns, hipStream_t st) {
  const int64_t g = p.B * p.Hq * ((p.nQB + 1) / 2) * ns;
#define QATTN_PP(SPLIT, CA)                                                                                      \
  do {                                                                                                           \
    if (dtype == QATTN_BF16) qattn_fwd_pp_kernel<false, KT, SPLIT, HD, QF, CA><<<g, kPPThreads, 0, st>>>(p);     \
    else qattn_fwd_pp_kernel<true, KT, SPLIT, HD, QF, CA><<<g, kPPThreads, 0, st>>>(p);                          \
  } while (0)
  if (ns > 1) {
    QATTN_PP(true, true);
    launch_combine(p, dtype, HD, st);
  } else if (p.causal) {
    QATTN_PP(false, true);
  } else {
    QATTN_PP(false, false);
  }
#undef QATTN_PP
}

template <bool KT>
static int launch_fwd(AttnParams& p, int out_dtype, int ns, void* workspace, size_t workspace_bytes, hipStream_t st,
                      int64_t D, int kernel) {
  t_last_kernel = kernel;
  if (kernel == QATTN_KERNEL_MULTI_BLOCK) {
    p.nsplit = 1;
    p.tiles_per_split = (int)p.nKB;
    p.nQC = (p.nQB + p.qpw - 1) / p.qpw;
    const int64_t g = p.B * p.Hq * p.nQC;
    QATTN_REQUIRE(g < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
    if (out_dtype == QATTN_BF16) qattn_fwd_kernel<false, false, KT, true><<<g, kThreads, 0, st>>>(p);
    else qattn_fwd_kernel<true, false, KT, true><<<g, kThreads, 0, st>>>(p);
    return check_launch("qattn_fwd");
  }
  if (kernel == QATTN_KERNEL_RESIDENT) {
    p.nsplit = 1;
    p.tiles_per_split = (int)p.nKB;
    resident_layout(p.B * p.Hq, (p.Lq + 31) / 32, p.wb_per_wg, p.n_chunk);
    const int64_t g = p.B * p.Hq * p.n_chunk;
    QATTN_REQUIRE(g < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
    if (out_dtype == QATTN_BF16) qattn_fwd_res_kernel<false, KT><<<g, kResThreads, 0, st>>>(p);
    else qattn_fwd_res_kernel<true, KT><<<g, kResThreads, 0, st>>>(p);
    return check_launch("qattn_fwd");
  }
  if (kernel == QATTN_KERNEL_PINGPONG) {
    const int64_t g = p.B * p.Hq * ((p.nQB + 1) / 2) * ns;
    QATTN_REQUIRE(g < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
    p.nsplit = ns;
    p.tiles_per_split = (int)((p.nKB + ns - 1) / ns);
    if (ns > 1) {
      QATTN_REQUIRE(workspace && workspace_bytes >= qattn_fwd_workspace_size(p.B, p.Lq, p.Hq, D, ns),
                    QATTN_ERR_WORKSPACE, "qattn_fwd with %d KV splits needs %zu workspace bytes", ns,
                    qattn_fwd_workspace_size(p.B, p.Lq, p.Hq, D, ns));
      p.ws_o = static_cast<float*>(workspace);
      p.ws_ml = p.ws_o + (int64_t)ns * p.B * p.Hq * p.Lq * D;
    }
    if (D == 64) launch_pp<KT, 64, QF_INT8>(p, out_dtype, ns, st);
    else launch_pp<KT, kD, QF_INT8>(p, out_dtype, ns, st);
    return check_launch("qattn_fwd");
  }
  const int64_t grid = p.B * p.Hq * p.nQB * ns;
  QATTN_REQUIRE(grid < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
  p.nsplit = ns;
  p.tiles_per_split = (int)((p.nKB + ns - 1) / ns);
  if (ns > 1) {
    QATTN_REQUIRE(workspace && workspace_bytes >= qattn_fwd_workspace_size(p.B, p.Lq, p.Hq, D, ns), QATTN_ERR_WORKSPACE,
                  "qattn_fwd with %d KV splits needs %zu workspace bytes", ns,
                  qattn_fwd_workspace_size(p.B, p.Lq, p.Hq, D, ns));
    p.ws_o = static_cast<float*>(workspace);
    p.ws_ml = p.ws_o + (int64_t)ns * p.B * p.Hq * p.Lq * D;
    if (out_dtype == QATTN_BF16) qattn_fwd_kernel<false, true, KT><<<grid, kThreads, 0, st>>>(p);
    else qattn_fwd_kernel<true, true, KT><<<grid, kThreads, 0, st>>>(p);
    launch_combine(p, out_dtype, D, st);
  } else {
    if (out_dtype == QATTN_BF16) qattn_fwd_kernel<false, false, KT><<<grid, kThreads, 0, st>>>(p);
    else qattn_fwd_kernel<true, false, KT><<<grid, kThreads, 0, st>>>(p);
  }
  return check_launch("qattn_fwd");
}

// Short key ranges: one workgroup streams several query blocks of a head through one K/V pipeline, so
// the per-workgroup start-up (Q load, scale staging, first DMA round trip) and the epilogue overlap the
// next block's work.  Picks the blocks per workgroup that minimise the modelled makespan: full rounds
// of 512 resident workgroups (256 CUs x 2), each block costing its key tiles plus about one tile of
// epilogue, each workgroup about four tiles of start-up.
static int blocks_per_workgroup(int64_t bh, int64_t nqb, int64_t nkb) {
  int best = 1;
  double best_cost = 1e300;
  for (int64_t q = 1; q <= std::min<int64_t>(nqb, kMqMaxBlocks); q++) {
    const int64_t wgs = bh * ((nqb + q - 1) / q);
    const int64_t rounds = (wgs + 511) / 512;
    const double cost = (double)rounds * (double)(q * (nkb + 1) + 4);
    if (cost < best_cost) {
      best_cost = cost;
      best = (int)q;
    }
  }
  return best;
}

// Split count, query blocks per workgroup and kernel of a launch (rows of 128 queries, tiles of 64 keys).
static void plan_fwd(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int pv, int gran, int causal, bool sparse,
                     int num_splits, int& ns, int& qpw, int& kernel) {
  const int64_t nQB = (Lq + kBQ - 1) / kBQ, nKB = (Lk + kBK - 1) / kBK;
  const int64_t max_tiles = pv == PV_FP8 ? max_tiles_per_split(is_thread_gran(gran))
                                         : half_max_tiles(is_thread_gran(gran), sparse);
  ns = num_splits > 0 ? num_splits
       : sparse       ? num_splits_for(B, Lq, Lk, Hq, max_tiles, false)
                      : dense_num_splits(B, Lq, Lk, Hq, pv, gran);
  ns = (int)std::min<int64_t>(ns, nKB);
  if (ns < 1) ns = 1;
  // a workgroup stages the k_scales of at most max_tiles key tiles
  ns = (int)std::max<int64_t>(ns, (nKB + max_tiles - 1) / max_tiles);
  // (the multi-block kernel stages at most 32 q_scales per query block)
  const bool mq_ok = ns == 1 && !sparse && !causal && pv == PV_FP8 && nKB <= kMqMaxTiles &&
                     gran != QATTN_GRAN_THREAD_SM90;
  const bool res_ok = ns == 1 && !sparse && !causal && pv == PV_FP8 && nKB <= kResMaxTiles;
  const int qpw_mq = mq_ok ? blocks_per_workgroup(B * Hq, nQB, nKB) : 1;
  const int qpw_auto = nKB < kMqAutoMaxTiles ? qpw_mq : 1;
  kernel = pick_kernel(pv, sparse, ns, causal, B, Hq, nQB, qpw_auto, mq_ok, res_ok);
  qpw = kernel == QATTN_KERNEL_MULTI_BLOCK ? qpw_mq : 1;
}

extern "C" int qattn_fwd_ex_kernel(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int v_kind, int qk_quant_gran,
                                   int causal, int num_splits) {
  if (B <= 0 || Lq <= 0 || Lk <= 0 || Hq <= 0) return QATTN_KERNEL_AUTO;
  const int pv = v_kind == QATTN_V_FP8 ? PV_FP8 : v_kind == QATTN_V_BF16 ? PV_BF16 : PV_FP16;
  int ns, qpw, kernel;
  plan_fwd(B, Lq, Lk, Hq, pv, qk_quant_gran, causal, false, num_splits, ns, qpw, kernel);
  return kernel;
}

static int setup_fwd(AttnParams& p, int& ns, qattn_seq q8, const float* q_scale, qattn_seq k8, const float* k_scale,
                     const void* v, int64_t Lpad, qattn_seq o, int out_dtype, int64_t B, int64_t Lq, int64_t Lk,
                     int64_t Hq, int64_t Hkv, int64_t D, float qk_mult, int causal, int64_t q_offset,
                     const int32_t* kv_valid, float* lse, int num_splits, int pv, int gran, int& kernel,
                     bool sparse = false) {
  QATTN_REQUIRE(out_dtype == QATTN_BF16 || out_dtype == QATTN_FP16, QATTN_ERR_DTYPE, "out dtype must be bf16 or fp16");
  QATTN_REQUIRE(D == kD || (D == 64 && pv == PV_FP8 && !sparse), QATTN_ERR_HEAD_DIM,
                "qattn_fwd needs head_dim 128, or 64 with FP8 V on a dense launch (pad other heads), got %lld",
                (long long)D);
  QATTN_REQUIRE(gran >= QATTN_GRAN_BLOCK && gran <= QATTN_GRAN_THREAD_SM90, QATTN_ERR_ARG,
                "qk_quant_gran must be 1 (per block), 2 (per warp), 3 (per thread), 4 (per warp, sm90 tables) or "
                "5 (per thread, sm90 tables), got %d", gran);
  QATTN_REQUIRE(B >= 0 && Lq >= 0 && Lk >= 0 && Hq > 0 && Hkv > 0, QATTN_ERR_SHAPE, "bad sizes");
  QATTN_REQUIRE(Hq % Hkv == 0, QATTN_ERR_HEAD_RATIO, "num_qo_heads (%lld) must be divisible by num_kv_heads (%lld)",
                (long long)Hq, (long long)Hkv);
  if (B * Lq == 0) return -1;  // nothing to do
  QATTN_REQUIRE(Lk > 0, QATTN_ERR_SHAPE, "kv_len must be positive");
  QATTN_REQUIRE(Lpad % kBK == 0 && Lpad >= (Lk + kBK - 1) / kBK * kBK, QATTN_ERR_SHAPE,
                "Lpad must be a multiple of 64 covering kv_len");
  for (const qattn_seq* sq : {&q8, &k8}) {
    QATTN_REQUIRE(sq->data && aligned16(sq->data), QATTN_ERR_ALIGN, "q8/k8 must be 16-byte aligned");
    QATTN_REQUIRE(sq->sb % 16 == 0 && sq->sl % 16 == 0 && sq->sh % 16 == 0, QATTN_ERR_STRIDE,
                  "q8/k8 strides must be multiples of 16 bytes");
  }
  QATTN_REQUIRE(o.data && aligned16(o.data), QATTN_ERR_ALIGN, "output must be 16-byte aligned");
  QATTN_REQUIRE(o.sb % 8 == 0 && o.sl % 8 == 0 && o.sh % 8 == 0, QATTN_ERR_STRIDE,
                "output strides must be multiples of 16 bytes");
  QATTN_REQUIRE(v && aligned16(v) && q_scale && k_scale, QATTN_ERR_ARG, "null scale or V pointer");
  QATTN_REQUIRE(!causal || q_offset >= 0, QATTN_ERR_ARG, "q_offset must be >= 0");
  // the kernel addresses one (batch, kv head) of K and V through 32-bit buffer offsets
  QATTN_REQUIRE((Lk - 1) * k8.sl + D < (1ll << 32) && D * Lpad * 2 < (1ll << 32), QATTN_ERR_SHAPE,
                "K/V of one (batch, head) must span less than 4 GiB");

  p = AttnParams{};
  p.q8 = static_cast<const int8_t*>(q8.data);
  p.qsb = q8.sb; p.qsl = q8.sl; p.qsh = q8.sh;
  p.k8 = static_cast<const int8_t*>(k8.data);
  p.ksb = k8.sb; p.ksl = k8.sl; p.ksh = k8.sh;
  p.v = v; p.Lpad = Lpad;
  p.q_scale = q_scale; p.k_scale = k_scale;
  p.o = o.data; p.osb = o.sb; p.osl = o.sl; p.osh = o.sh;
  p.lse = lse; p.kv_valid = kv_valid;
  p.B = B; p.Lq = Lq; p.Lk = Lk; p.Hq = Hq; p.Hkv = Hkv;
  p.nQB = (Lq + kBQ - 1) / kBQ;
  p.nKB = (Lk + kBK - 1) / kBK;
  const bool sm90 = gran == QATTN_GRAN_WARP_SM90 || gran == QATTN_GRAN_THREAD_SM90;
  p.qgran = sm90 ? gran - 2 : gran;
  p.qrs = sm90 ? 4 : 5;
  p.kts = sm90 ? 1 : 0;
  if (sm90) {
    // 64-row Q blocks of four 16-row warps, 128-key K blocks
    const int64_t nq64 = (Lq + 63) / 64, nk128 = (Lk + 127) / 128;
    p.nQS = p.qgran == QATTN_GRAN_THREAD ? nq64 * 32 : nq64 * 4;
    p.nKS = p.qgran == QATTN_GRAN_THREAD ? nk128 * 4 : nk128;
  } else {
    p.nQS = gran == QATTN_GRAN_THREAD ? p.nQB * 32 : gran == QATTN_GRAN_WARP ? p.nQB * 4 : p.nQB;
    p.nKS = gran == QATTN_GRAN_THREAD ? p.nKB * 4 : p.nKB;
  }
  p.q_offset = q_offset;
  p.group = (int)(Hq / Hkv);
  p.causal = causal ? 1 : 0;
  p.qk_mult = qk_mult;

  plan_fwd(B, Lq, Lk, Hq, pv, gran, causal, sparse, num_splits, ns, p.qpw, kernel);
  if (D == 64) {
    // head_dim 64 runs the ping-pong kernel only (its unsplit and KV-split forms)
    QATTN_REQUIRE(t_kernel_override == QATTN_KERNEL_AUTO || t_kernel_override == QATTN_KERNEL_PINGPONG,
                  QATTN_ERR_HEAD_DIM, "head_dim 64 runs the ping-pong kernel only (kernel override %d)",
                  t_kernel_override);
    kernel = QATTN_KERNEL_PINGPONG;
    p.qpw = 1;
  }
  return QATTN_OK;
}

static int launch_gran(AttnParams& p, int gran, int out_dtype, int ns, void* ws, size_t wsb, hipStream_t st,
                       int64_t D, int kernel) {
  if (is_thread_gran(gran)) return launch_fwd<true>(p, out_dtype, ns, ws, wsb, st, D, kernel);
  return launch_fwd<false>(p, out_dtype, ns, ws, wsb, st, D, kernel);
}

// half P.V: the automatic split count evens out the rounds of workgroups and takes its partials (520 bytes per row and
// split, hundreds of MB for long calls) for granted; where the workspace holds fewer, the launch splits less, down to
// what the staged k_scales need
static int half_fit_splits(const AttnParams& p, int ns, bool kt, size_t bytes) {
  const int64_t tiles = half_max_tiles(kt, false), min_ns = (p.nKB + tiles - 1) / tiles;
  while (ns > min_ns && qattn_fwd_workspace_size(p.B, p.Lq, p.Hq, kD, ns) > bytes) ns--;
  return ns;
}

// half P.V: the workspace of a KV split, then the launch (attn_half.hip)
static int launch_half_ws(AttnParams& p, bool kt, bool f16v, bool sparse, int out_dtype, int ns, void* ws, size_t wsb,
                          hipStream_t st) {
  t_last_kernel = QATTN_KERNEL_ONE_BLOCK;
  if (ns > 1) {
    const size_t need = qattn_fwd_workspace_size(p.B, p.Lq, p.Hq, kD, ns);
    QATTN_REQUIRE(ws && wsb >= need, QATTN_ERR_WORKSPACE, "qattn_fwd with %d KV splits needs %zu workspace bytes", ns,
                  need);
    p.ws_o = static_cast<float*>(ws);
    p.ws_ml = p.ws_o + (int64_t)ns * p.B * p.Hq * p.Lq * kD;
  }
  return launch_half(p, kt, f16v, sparse, out_dtype, ns, st);
}

extern "C" int qattn_fwd_ex(qattn_seq q8, const float* q_scale, qattn_seq k8, const float* k_scale, const void* v,
                            int v_kind, int64_t Lpad, const float* v_scale, qattn_seq o, int out_dtype, int64_t B,
                            int64_t Lq, int64_t Lk, int64_t Hq, int64_t Hkv, int64_t D, float qk_mult,
                            int qk_quant_gran, int causal, int64_t q_offset, const int32_t* kv_valid, float* lse,
                            int num_splits, void* workspace, size_t workspace_bytes, qattn_stream_t stream) {
  return qattn_fwd_ex2(q8, q_scale, k8, k_scale, v, v_kind, Lpad, v_scale, nullptr, o, out_dtype, B, Lq, Lk, Hq, Hkv,
                       D, qk_mult, qk_quant_gran, causal, q_offset, kv_valid, lse, num_splits, workspace,
                       workspace_bytes, stream);
}

extern "C" int qattn_fwd_ex2(qattn_seq q8, const float* q_scale, qattn_seq k8, const float* k_scale, const void* v,
                             int v_kind, int64_t Lpad, const float* v_scale, const float* v_mean, qattn_seq o,
                             int out_dtype, int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int64_t Hkv, int64_t D,
                             float qk_mult, int qk_quant_gran, int causal, int64_t q_offset, const int32_t* kv_valid,
                             float* lse, int num_splits, void* workspace, size_t workspace_bytes,
                             qattn_stream_t stream) {
  QATTN_REQUIRE(!v_mean || v_kind == QATTN_V_FP8, QATTN_ERR_ARG, "v_mean needs the FP8 V path");
  QATTN_REQUIRE(v_kind == QATTN_V_FP8 || v_kind == QATTN_V_BF16 || v_kind == QATTN_V_FP16, QATTN_ERR_DTYPE,
                "v_kind must be 0 (fp8), 1 (bf16) or 2 (fp16), got %d", v_kind);
  AttnParams p;
  int ns = 1, kernel = QATTN_KERNEL_AUTO;
  const int pv = v_kind == QATTN_V_FP8 ? PV_FP8 : v_kind == QATTN_V_BF16 ? PV_BF16 : PV_FP16;
  const int rc = setup_fwd(p, ns, q8, q_scale, k8, k_scale, v, Lpad, o, out_dtype, B, Lq, Lk, Hq, Hkv, D, qk_mult,
                           causal, q_offset, kv_valid, lse, num_splits, pv, qk_quant_gran, kernel);
  if (rc < 0) return QATTN_OK;
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (pv == PV_FP8) {
    QATTN_REQUIRE(v_scale, QATTN_ERR_ARG, "v_scale is null");
    p.v_scale = v_scale;
    p.v_mean = v_mean;
    return launch_gran(p, qk_quant_gran, out_dtype, ns, workspace, workspace_bytes, st, D, kernel);
  }
  p.v_scale = nullptr;
  if (num_splits <= 0) ns = half_fit_splits(p, ns, is_thread_gran(qk_quant_gran), workspace ? workspace_bytes : 0);
  return launch_half_ws(p, is_thread_gran(qk_quant_gran), pv == PV_FP16, false, out_dtype, ns, workspace,
                        workspace_bytes, st);
}

// ---- half Q quantized inside the attention kernel (resident or ping-pong) ----
// the kernel a qattn_fwd_q16 launch runs: the automatic rule's, when it is one of the two with a fused-Q form
static int q16_kernel(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int64_t D, int gran, int causal) {
  if ((D != kD && D != 64) || B <= 0 || Lq <= 0 || Lk <= 0 || Hq <= 0) return QATTN_KERNEL_AUTO;
  if (D == 64) return QATTN_KERNEL_PINGPONG;  // (head_dim 64 runs the ping-pong kernel only)
  int ns, qpw, kernel;
  plan_fwd(B, Lq, Lk, Hq, PV_FP8, gran, causal, false, 0, ns, qpw, kernel);
  return kernel == QATTN_KERNEL_RESIDENT || kernel == QATTN_KERNEL_PINGPONG ? kernel : QATTN_KERNEL_AUTO;
}

extern "C" int qattn_fwd_q16_supported(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int64_t D, int qk_quant_gran,
                                       int causal) {
  if (qk_quant_gran < QATTN_GRAN_BLOCK || qk_quant_gran > QATTN_GRAN_THREAD) return 0;
  return q16_kernel(B, Lq, Lk, Hq, D, qk_quant_gran, causal) != QATTN_KERNEL_AUTO ? 1 : 0;
}

extern "C" int qattn_fwd_q16(qattn_seq q, qattn_seq k8, const float* k_scale, const uint8_t* v8, int64_t Lpad,
                             const float* v_scale, const float* v_mean, qattn_seq o, int dtype, int64_t B,
                             int64_t Lq, int64_t Lk, int64_t Hq, int64_t Hkv, int64_t D, float qk_mult,
                             int qk_quant_gran, int causal, int64_t q_offset, const int32_t* kv_valid, float* lse,
                             int num_splits, void* workspace, size_t workspace_bytes, qattn_stream_t stream) {
  QATTN_REQUIRE(qk_quant_gran >= QATTN_GRAN_BLOCK && qk_quant_gran <= QATTN_GRAN_THREAD, QATTN_ERR_ARG,
                "qattn_fwd_q16 quantizes Q per block (1), per warp (2) or per thread (3), got %d", qk_quant_gran);
  QATTN_REQUIRE(v8 && v_scale, QATTN_ERR_ARG, "null V or v_scale");
  if (B * Lq == 0) return QATTN_OK;
  const int kernel = q16_kernel(B, Lq, Lk, Hq, D, qk_quant_gran, causal);
  QATTN_REQUIRE(kernel != QATTN_KERNEL_AUTO, QATTN_ERR_SHAPE,
                "qattn_fwd_q16 runs the resident or ping-pong kernel: head_dim 64, or 128 and a launch the automatic "
                "rule gives one of them (see qattn_fwd_q16_supported)");
  AttnParams p;
  int ns = 1, kplan = QATTN_KERNEL_AUTO;
  // (q's scale table is formed inside the kernel: k_scale stands in for the pointer setup_fwd checks)
  const int rc = setup_fwd(p, ns, q, k_scale, k8, k_scale, v8, Lpad, o, dtype, B, Lq, Lk, Hq, Hkv, D, qk_mult, causal,
                           q_offset, kv_valid, lse, num_splits, PV_FP8, qk_quant_gran, kplan);
  if (rc < 0) return QATTN_OK;
  if (rc) return rc;
  QATTN_REQUIRE(kplan == kernel, QATTN_ERR_ARG, "qattn_fwd_q16: num_splits %d moves the launch off its kernel",
                num_splits);
  p.v_scale = v_scale;
  p.v_mean = v_mean;
  if (qk_quant_gran == QATTN_GRAN_BLOCK) {
    // per-block scales carry sm_scale * log2(e): it is multiplied into Q, the logits take 1
    p.q_sm_scale = qk_mult;
    p.qk_mult = 1.0f;
  }
  hipStream_t st = (hipStream_t)stream;
  t_last_kernel = kernel;
  if (kernel == QATTN_KERNEL_RESIDENT) {
    p.nsplit = 1;
    p.tiles_per_split = (int)p.nKB;
    // (chunks of whole 128-row Q blocks for per-block scales)
    resident_layout(p.B * p.Hq, (p.Lq + 31) / 32, p.wb_per_wg, p.n_chunk, qk_quant_gran == QATTN_GRAN_BLOCK ? 4 : 1);
    const int64_t g = p.B * p.Hq * p.n_chunk;
    QATTN_REQUIRE(g < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
    if (qk_quant_gran == QATTN_GRAN_BLOCK) {
      if (dtype == QATTN_BF16) qattn_fwd_res_kernel<false, false, QF_BLOCK><<<g, kResThreads, 0, st>>>(p);
      else qattn_fwd_res_kernel<true, false, QF_BLOCK><<<g, kResThreads, 0, st>>>(p);
    } else if (qk_quant_gran == QATTN_GRAN_THREAD) {
      if (dtype == QATTN_BF16) qattn_fwd_res_kernel<false, true, QF_THREAD><<<g, kResThreads, 0, st>>>(p);
      else qattn_fwd_res_kernel<true, true, QF_THREAD><<<g, kResThreads, 0, st>>>(p);
    } else {
      if (dtype == QATTN_BF16) qattn_fwd_res_kernel<false, false, QF_WARP><<<g, kResThreads, 0, st>>>(p);
      else qattn_fwd_res_kernel<true, false, QF_WARP><<<g, kResThreads, 0, st>>>(p);
    }
    return check_launch("qattn_fwd_q16");
  }
  const int64_t g = p.B * p.Hq * ((p.nQB + 1) / 2) * ns;
  QATTN_REQUIRE(g < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
  p.nsplit = ns;
  p.tiles_per_split = (int)((p.nKB + ns - 1) / ns);
  if (ns > 1) {
    QATTN_REQUIRE(workspace && workspace_bytes >= qattn_fwd_workspace_size(p.B, p.Lq, p.Hq, D, ns),
                  QATTN_ERR_WORKSPACE, "qattn_fwd_q16 with %d KV splits needs %zu workspace bytes", ns,
                  qattn_fwd_workspace_size(p.B, p.Lq, p.Hq, D, ns));
    p.ws_o = static_cast<float*>(workspace);
    p.ws_ml = p.ws_o + (int64_t)ns * p.B * p.Hq * p.Lq * D;
  }
  if (D == 64) {
    if (qk_quant_gran == QATTN_GRAN_THREAD) launch_pp<true, 64, QF_THREAD>(p, dtype, ns, st);
    else if (qk_quant_gran == QATTN_GRAN_WARP) launch_pp<false, 64, QF_WARP>(p, dtype, ns, st);
    else launch_pp<false, 64, QF_BLOCK>(p, dtype, ns, st);
  } else {
    if (qk_quant_gran == QATTN_GRAN_THREAD) launch_pp<true, kD, QF_THREAD>(p, dtype, ns, st);
    else if (qk_quant_gran == QATTN_GRAN_WARP) launch_pp<false, kD, QF_WARP>(p, dtype, ns, st);
    else launch_pp<false, kD, QF_BLOCK>(p, dtype, ns, st);
  }
  return check_launch("qattn_fwd_q16");
}

// ---- packed variable-length batches ----
// One launch over every sequence of a packed batch (attn_qk_int8_block_varlen.py:68-155): the grid is a bound, from the
// packed lengths alone, on the pairs of query blocks of all sequences and heads; each workgroup finds its sequence, head
// and pair in the device tables (attn_half.hip), so the host never reads cu_seqlens.
extern "C" int qattn_fwd_varlen(qattn_seq q8, const float* q_scale, qattn_seq k8, const float* k_scale,
                                const uint16_t* v16, int64_t Lpad, qattn_seq o, int out_dtype, int64_t B,
                                int64_t total_q, int64_t total_k, int64_t max_lq, int64_t max_lk, int64_t Hq,
                                int64_t Hkv, int64_t D, float qk_mult,
                                int causal, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                const int32_t* cu_qs, const int32_t* cu_ks, const int32_t* cu_vt,
                                qattn_stream_t stream) {
  QATTN_REQUIRE(cu_seqlens_q && cu_seqlens_k && cu_qs && cu_ks && cu_vt, QATTN_ERR_ARG, "null sequence table");
  QATTN_REQUIRE(total_q >= 0 && total_k >= 0, QATTN_ERR_SHAPE, "negative packed size");
  AttnParams p;
  int ns = 1, kernel = QATTN_KERNEL_AUTO;
  const int rc = setup_fwd(p, ns, q8, q_scale, k8, k_scale, v16, Lpad, o, out_dtype, B, max_lq, max_lk, Hq, Hkv, D,
                           qk_mult, causal, 0, nullptr, nullptr, 1, PV_FP16, QATTN_GRAN_BLOCK, kernel);
  if (rc < 0) return QATTN_OK;
  if (rc) return rc;
  p.cu_q = cu_seqlens_q;
  p.cu_k = cu_seqlens_k;
  p.cu_qs = cu_qs;
  p.cu_ks = cu_ks;
  p.cu_vt = cu_vt;
  p.var_tq = total_q;
  p.var_tk = total_k;
  p.v_scale = nullptr;
  p.qpw = 1;
  t_last_kernel = QATTN_KERNEL_ONE_BLOCK;
  return launch_half_varlen(p, out_dtype, (hipStream_t)stream);
}

// ---- allocation-free form of qattn_fwd_ex ----
// KV-split launches keep their partial (O, m, l) rows in this file-scope device array instead of a caller
// workspace.  Every GPU the library runs on holds its own copy for the life of the process; host code
// reaches it only through the address hipGetSymbolAddress returns on that device (the array's name is a
// host-side stand-in, not a device address).
constexpr size_t kScratchBytes = 128ull << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;  // guards the per-device tables and orders the scratch users (below)
static void* g_scratch_ptr[kMaxDevices];
// Completion of the last launch that used a device's scratch.  Each launch that uses the scratch first makes
// its stream wait for this event and then records it again, so launches from different streams (or threads)
// take the array one after the other in the order the host issued them (hipStreamWaitEvent is asynchronous:
// no host wait).  Created with the symbol lookup on the first call that needs the scratch on the device.
static hipEvent_t g_scratch_done[kMaxDevices];

// the scratch address and its ordering event on the calling thread's current device, set up once per device;
// the caller holds g_scratch_mu
static int scratch_on_current_device(void** out, int* dev_out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  QATTN_REQUIRE(e == hipSuccess && dev >= 0 && dev < kMaxDevices, QATTN_ERR_LAUNCH, "hipGetDevice failed: %s",
                hipGetErrorString(e));
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    QATTN_REQUIRE(e == hipSuccess && ptr, QATTN_ERR_LAUNCH, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                  hipGetErrorString(e));
    hipEvent_t ev = nullptr;
    e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    QATTN_REQUIRE(e == hipSuccess && ev, QATTN_ERR_LAUNCH, "hipEventCreate failed on device %d: %s", dev,
                  hipGetErrorString(e));
    g_scratch_done[dev] = ev;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  *dev_out = dev;
  return QATTN_OK;
}

extern "C" size_t qattn_fwd_noalloc_max_scratch(void) { return kScratchBytes; }

extern "C" int qattn_fwd_ex_noalloc(qattn_seq q8, const float* q_scale, qattn_seq k8, const float* k_scale,
                                    const void* v, int v_kind, int64_t Lpad, const float* v_scale, qattn_seq o,
                                    int out_dtype, int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int64_t Hkv,
                                    int64_t D, float qk_mult, int qk_quant_gran, int causal, int64_t q_offset,
                                    const int32_t* kv_valid, float* lse, int num_splits, qattn_stream_t stream) {
  QATTN_REQUIRE(v_kind == QATTN_V_FP8 || v_kind == QATTN_V_BF16 || v_kind == QATTN_V_FP16, QATTN_ERR_DTYPE,
                "v_kind must be 0 (fp8), 1 (bf16) or 2 (fp16), got %d", v_kind);
  AttnParams p;
  int ns = 1, kernel = QATTN_KERNEL_AUTO;
  const int pv = v_kind == QATTN_V_FP8 ? PV_FP8 : v_kind == QATTN_V_BF16 ? PV_BF16 : PV_FP16;
  const int rc = setup_fwd(p, ns, q8, q_scale, k8, k_scale, v, Lpad, o, out_dtype, B, Lq, Lk, Hq, Hkv, D, qk_mult,
                           causal, q_offset, kv_valid, lse, num_splits, pv, qk_quant_gran, kernel);
  if (rc < 0) return QATTN_OK;
  if (rc) return rc;
  if (pv != PV_FP8 && num_splits <= 0) ns = half_fit_splits(p, ns, is_thread_gran(qk_quant_gran), kScratchBytes);
  const size_t need = qattn_fwd_workspace_size(B, Lq, Hq, D, ns);
  QATTN_REQUIRE(need <= kScratchBytes, QATTN_ERR_WORKSPACE,
                "qattn_fwd_ex_noalloc: %d KV splits need %zu bytes of scratch, more than its %zu-byte limit "
                "(use qattn_fwd_ex with a workspace, or fewer splits)", ns, need, kScratchBytes);
  if (need == 0)  // no KV split: nothing of the scratch is used
    return qattn_fwd_ex(q8, q_scale, k8, k_scale, v, v_kind, Lpad, v_scale, o, out_dtype, B, Lq, Lk, Hq, Hkv, D,
                        qk_mult, qk_quant_gran, causal, q_offset, kv_valid, lse, ns, nullptr, 0, stream);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  void* ws = nullptr;
  int dev = -1;
  int e = scratch_on_current_device(&ws, &dev);
  if (e) return e;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // Order this launch after the previous scratch user on the device.  A stream under graph capture is left
  // to the graph's own order (waiting there on an event recorded outside the capture is not allowed):
  // replays of a captured graph must not overlap other users of the scratch.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  hipError_t he = hipStreamIsCapturing(st, &cap);
  QATTN_REQUIRE(he == hipSuccess, QATTN_ERR_LAUNCH, "hipStreamIsCapturing failed: %s", hipGetErrorString(he));
  const bool order = cap == hipStreamCaptureStatusNone;
  if (order) {
    he = hipStreamWaitEvent(st, g_scratch_done[dev], 0);
    QATTN_REQUIRE(he == hipSuccess, QATTN_ERR_LAUNCH, "hipStreamWaitEvent failed: %s", hipGetErrorString(he));
  }
  // the same launch as qattn_fwd_ex with this split count and the device array as its workspace
  e = qattn_fwd_ex(q8, q_scale, k8, k_scale, v, v_kind, Lpad, v_scale, o, out_dtype, B, Lq, Lk, Hq, Hkv, D, qk_mult,
                   qk_quant_gran, causal, q_offset, kv_valid, lse, ns, ws, need, stream);
  if (e) return e;
  if (order) {
    he = hipEventRecord(g_scratch_done[dev], st);
    QATTN_REQUIRE(he == hipSuccess, QATTN_ERR_LAUNCH, "hipEventRecord failed: %s", hipGetErrorString(he));
  }
  return QATTN_OK;
}

extern "C" int qattn_lse_finish(float* lse, qattn_seq q, int dtype, const void* k_mean, int64_t B, int64_t Lq,
                                int64_t Hq, int64_t Hkv, int64_t D, float sm_scale, qattn_stream_t stream) {
  QATTN_REQUIRE(dtype == QATTN_BF16 || dtype == QATTN_FP16, QATTN_ERR_DTYPE, "dtype must be bf16 (0) or fp16 (1)");
  QATTN_REQUIRE(D == 64 || D == 128, QATTN_ERR_HEAD_DIM, "head_dim must be 64 or 128, got %lld", (long long)D);
  QATTN_REQUIRE(B >= 0 && Lq >= 0 && Hq > 0 && Hkv > 0, QATTN_ERR_SHAPE, "bad sizes");
  QATTN_REQUIRE(Hq % Hkv == 0, QATTN_ERR_HEAD_RATIO, "num_qo_heads (%lld) must be divisible by num_kv_heads (%lld)",
                (long long)Hq, (long long)Hkv);
  if (B * Lq == 0) return QATTN_OK;
  QATTN_REQUIRE(lse && k_mean && aligned16(k_mean) && q.data && aligned16(q.data), QATTN_ERR_ALIGN,
                "null or misaligned pointer");
  QATTN_REQUIRE(q.sb % 8 == 0 && q.sl % 8 == 0 && q.sh % 8 == 0, QATTN_ERR_STRIDE,
                "q strides must be multiples of 16 bytes");
  const int64_t rows = B * Lq * Hq, per = 256 / (D / 8), g = (rows + per - 1) / per;
  QATTN_REQUIRE(g < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
  hipStream_t st = (hipStream_t)stream;
  const uint16_t *qp = static_cast<const uint16_t*>(q.data), *km = static_cast<const uint16_t*>(k_mean);
#define QATTN_LF(F16, DD) \
  lse_finish_kernel<F16, DD><<<g, 256, 0, st>>>(lse, qp, q.sb, q.sl, q.sh, km, Lq, Hq, (int)(Hq / Hkv), rows, sm_scale)
  if (dtype == QATTN_BF16) {
    if (D == 128) QATTN_LF(false, 128);
    else QATTN_LF(false, 64);
  } else {
    if (D == 128) QATTN_LF(true, 128);
    else QATTN_LF(true, 64);
  }
#undef QATTN_LF
  return check_launch("qattn_lse_finish");
}

extern "C" int qattn_fwd(qattn_seq q8, const float* q_scale, qattn_seq k8, const float* k_scale, const uint8_t* v8,
                         int64_t Lpad, const float* v_scale, qattn_seq o, int out_dtype, int64_t B, int64_t Lq,
                         int64_t Lk, int64_t Hq, int64_t Hkv, int64_t D, float qk_mult, int causal,
                         int64_t q_offset, const int32_t* kv_valid, float* lse, int num_splits, void* workspace,
                         size_t workspace_bytes, qattn_stream_t stream) {
  return qattn_fwd_ex(q8, q_scale, k8, k_scale, v8, QATTN_V_FP8, Lpad, v_scale, o, out_dtype, B, Lq, Lk, Hq, Hkv, D,
                      qk_mult, QATTN_GRAN_BLOCK, causal, q_offset, kv_valid, lse, num_splits, workspace,
                      workspace_bytes, stream);
}

extern "C" int qattn_fwd_pv16(qattn_seq q8, const float* q_scale, qattn_seq k8, const float* k_scale,
                              const uint16_t* v16, int v_dtype, int64_t Lpad, qattn_seq o, int out_dtype, int64_t B,
                              int64_t Lq, int64_t Lk, int64_t Hq, int64_t Hkv, int64_t D, float qk_mult, int causal,
                              int64_t q_offset, const int32_t* kv_valid, float* lse, int num_splits, void* workspace,
                              size_t workspace_bytes, qattn_stream_t stream) {
  QATTN_REQUIRE(v_dtype == QATTN_BF16 || v_dtype == QATTN_FP16, QATTN_ERR_DTYPE, "V dtype must be bf16 or fp16");
  return qattn_fwd_ex(q8, q_scale, k8, k_scale, v16, v_dtype == QATTN_BF16 ? QATTN_V_BF16 : QATTN_V_FP16, Lpad,
                      nullptr, o, out_dtype, B, Lq, Lk, Hq, Hkv, D, qk_mult, QATTN_GRAN_BLOCK, causal, q_offset,
                      kv_valid, lse, num_splits, workspace, workspace_bytes, stream);
}

extern "C" int qattn_fwd_block_sparse_num_splits(int64_t B, int64_t Lq, int64_t Lk, int64_t Hq) {
  return num_splits_for(B, Lq, Lk, Hq, half_max_tiles(false, true), false);
}

extern "C" int qattn_fwd_block_sparse(qattn_seq q8, const float* q_scale, qattn_seq k8, const float* k_scale,
                                      const uint16_t* v16, int v_dtype, int64_t Lpad, qattn_seq o, int out_dtype,
                                      int64_t B, int64_t Lq, int64_t Lk, int64_t Hq, int64_t Hkv, int64_t D,
                                      float qk_mult, int causal, const int8_t* tile_mask, int64_t mask_sbh,
                                      int64_t mask_sq, float* lse, int num_splits, void* workspace,
                                      size_t workspace_bytes, qattn_stream_t stream) {
  QATTN_REQUIRE(v_dtype == QATTN_BF16 || v_dtype == QATTN_FP16, QATTN_ERR_DTYPE, "V dtype must be bf16 or fp16");
  QATTN_REQUIRE(tile_mask != nullptr, QATTN_ERR_ARG, "tile_mask is null");
  QATTN_REQUIRE(mask_sbh >= 0 && mask_sq >= 0, QATTN_ERR_STRIDE, "negative mask stride");
  AttnParams p;
  int ns = 1, kernel = QATTN_KERNEL_AUTO;
  const int pv = v_dtype == QATTN_BF16 ? PV_BF16 : PV_FP16;
  const int rc = setup_fwd(p, ns, q8, q_scale, k8, k_scale, v16, Lpad, o, out_dtype, B, Lq, Lk, Hq, Hkv, D, qk_mult,
                           causal, 0, nullptr, lse, num_splits, pv, QATTN_GRAN_BLOCK, kernel, true);
  if (rc < 0) return QATTN_OK;
  if (rc) return rc;
  p.v_scale = nullptr;
  p.tile_mask = tile_mask;
  p.tm_s1 = mask_sbh;
  p.tm_s2 = mask_sq;
  hipStream_t st = (hipStream_t)stream;
  return launch_half_ws(p, false, pv == PV_FP16, true, out_dtype, ns, workspace, workspace_bytes, st);
}
