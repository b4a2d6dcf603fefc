// INT8 Q.K^T attention with P.V in the half dtype of V (SAGE_ATTN_2_8_16, the Triton entries, packed varlen
// batches and block-sparse masks) for gfx950.  Per element the math is the FP8 kernels' (attn.hip) except that
// p = exp2(s - m) is rounded to V's half type, multiplied with V as given on v_mfma_f32_32x32x16_{bf16,f16}, and
// summed in fp32 before rounding (the reference's Triton kernels, attn_qk_int8_per_block.py:46-101).
//
// What bounds it, per wave (32 query rows) and 64-key tile: 768 matrix cycles (8 INT8 and 16 half MFMAs of 32),
// ~700 VALU cycles (32 v_exp_f32 at a quarter rate, 32 fma, 32 adds, 16 max3, 16 packs), 24 KiB of LDS fragment
// reads (768 cycles of the CU's 128 B/clk for the four waves that run a matrix stage together).  So the matrix
// stage of one wave has to run beside the softmax of another: two groups of four waves per workgroup (one wave of
// each per SIMD) alternate through workgroup barriers, half a tile apart, as in the FP8 ping-pong kernel:
//
//   group 0:  M(0) | V(0) | M(1) | V(1) | ...        M(t) = P(t-1).V(t-1), Q.K(t)^T  (matrix pipe)
//   group 1:    -  | M(0) | V(0) | M(1) | ...        V(t) = mask, softmax, P(t) to half  (VALU)
//
// Measured against a kernel with one 128-row block and four waves per workgroup, two workgroups per CU, whose waves
// fell into step (MFMAs, then softmax): 32760 x 32760 x 12 heads per-thread scales 5.40 (with the combine of the two
// splits that it needed) -> 4.60 ms (1.43 PFLOP/s; matrix pipe busy 55 %, VALU 62 %), 8 sequences of 257 .. 6240
// tokens, 12 heads 1475 -> 433 us (mostly HF_VAR's order of the work), block-sparse 32760 x 32760 x 12 at a quarter of
// the tiles 1555 -> 1475 us.
//
// Forms (one template axis):
//   HF_PAIR  the groups are two adjacent 128-row query blocks of a head: each K/V tile is fetched once for both
//   HF_VAR   the same over a packed variable-length batch: the workgroups find their (sequence, head, pair) in
//            the device tables, longest key ranges first up to 64 sequences
//   HF_OWN   each group takes a query block of its own (block-sparse masks, whose rows differ, and dense launches
//            with one or three query blocks per head, where a pair would be half empty, up to half_own_tiles).  The
//            tiles that both blocks visit come first, fetched once for both and five tiles ahead (their order follows
//            the mask: 30 % of the requests miss L2, against 4 % of HF_PAIR's); then each group streams what only its
//            block visits.
#include "attn_device.h"

namespace qattn {

constexpr int kHFThreads = 512;
// K and V tiles in LDS: K(t) is read in M(t), V(t) in M(t + 1).  With NB buffers of each, M(t) issues K(t + NB - 1)
// (where K(t - 1) was) and V(t + NB - 2) (where V(t - 2) was): both were last read in a stage that ended before
// M(t) began, for both groups.  A tile stream of a group's own has kHFBuf buffers, a shared one all of them.
constexpr int kHFBuf = 3;
constexpr int HF_PAIR = 0, HF_VAR = 1, HF_OWN = 2;
// k_scales (and tile ids, HF_OWN) of a workgroup's key range staged in LDS
constexpr int kHFKsPair = 4096;  // floats, next to 32 + 48 KiB of K / V buffers
constexpr int kHFKsOwn = 1024;   // floats per group, next to 2 x (24 + 48) KiB

template <bool F16V>
struct HalfVec {
  typedef __attribute__((ext_vector_type(8))) __bf16 vec;
  typedef __bf16 elem;
};
template <>
struct HalfVec<true> {
  typedef __attribute__((ext_vector_type(8))) _Float16 vec;
  typedef _Float16 elem;
};

// A sequence of a packed batch: its pairs of query blocks and its key count, none and -1 where it has no keys or its V
// tile range runs past Lpad (a too small Lpad leaves the sequence's rows untouched).
__device__ __forceinline__ void varlen_pairs(const AttnParams& p, int b, int& n, int& key) {
  int64_t r0, lq, lk;
  varlen_range(p.cu_k, b, p.var_tk, p.Lk, r0, lk);
  varlen_range(p.cu_q, b, p.var_tq, p.Lq, r0, lq);
  n = 0;
  key = -1;
  if (lk > 0 && ((int64_t)p.cu_vt[b] + (lk + kBK - 1) / kBK) * kBK <= p.Lpad) {
    n = (int)((lq + 2 * kBQ - 1) / (2 * kBQ));
    key = (int)lk;
  }
}

// Work item of workgroup g of a packed batch.  Every lane of the wave gets the same answer; false if g has none.
//   * Up to kVarSorted sequences: in order of decreasing key count (ties by index), each as head-major pairs of query
//     blocks, so the longest workgroups start first and the launch ends evenly.  (Dealt by sequence, one long sequence
//     kept a single XCD busy for most of the launch.)
//   * More: in sequence order with the heads innermost.  Sequence b starts at slot (cu_qs[b] + b) / 2 of each head, which
//     leaves room for its ceil(blocks / 2) pairs and at most one slot more, so that the block offsets are all the
//     search needs: 64 of them at a time, two loads up to 4096 sequences.  Ordered in runs of 64, every workgroup went
//     through all runs before its own (a call over 1000 sequences of 64 tokens, 12 heads, 3469 -> 1132 us; 200 of 32 .. 400
//     tokens 750 -> 533; 100 of 64 .. 8192 tokens, where the order counts most, 4308 -> 4067).
constexpr int kVarSorted = 64;
__device__ __forceinline__ int varlen_slot(const AttnParams& p, int b) { return (int)(((uint32_t)p.cu_qs[b] + (uint32_t)b) >> 1); }
__device__ __forceinline__ bool varlen_item(const AttnParams& p, int g, int& b_out, int& h_out, int& qp_out) {
  const int lane = threadIdx.x & 63, B = (int)p.B, H = (int)p.Hq;
  if (B <= kVarSorted) {
    int n = 0, key = -1;
    if (lane < B) varlen_pairs(p, lane, n, key);
    int before = 0, total = 0;
    for (int j = 0; j < B; j++) {
      const int nj = __builtin_amdgcn_readlane(n, j), kj = __builtin_amdgcn_readlane(key, j);
      total += nj;
      if (kj > key || (kj == key && j < lane)) before += nj;
    }
    const uint64_t hit = __ballot(n > 0 && g >= before * H && g < (before + n) * H);
    if (hit == 0) return false;
    const int src = __builtin_ctzll(hit);
    const int ns = __builtin_amdgcn_readlane(n, src), r = g - __builtin_amdgcn_readlane(before, src) * H;
    b_out = src;
    h_out = r / ns;
    qp_out = p.causal ? ns - 1 - r % ns : r % ns;
    return true;
  }
  const int slot = g / H;
  int lo = 0, hi = B;  // the last sequence of lo .. hi - 1 that starts at or before the slot
  while (hi - lo > 1) {
    const int step = (hi - lo + 63) / 64, at = lo + lane * step;
    const int n_ok = __popcll(__ballot(at < hi && varlen_slot(p, at) <= slot));
    lo += max(n_ok - 1, 0) * step;
    hi = min(hi, lo + step);
  }
  int n, key;
  varlen_pairs(p, lo, n, key);
  n = __builtin_amdgcn_readfirstlane(n);
  const int qp = slot - __builtin_amdgcn_readfirstlane(varlen_slot(p, lo));
  if (qp < 0 || qp >= n) return false;
  b_out = lo;
  h_out = g - slot * H;
  qp_out = p.causal ? n - 1 - qp : qp;
  return true;
}

template <bool F16OUT, bool F16V, bool KT, bool SPLIT, int FORM>
__global__ __launch_bounds__(kHFThreads) void qattn_fwd_half_kernel(AttnParams p) {
  constexpr bool OWN = FORM == HF_OWN, VAR = FORM == HF_VAR;
  static_assert(!VAR || (!KT && !SPLIT), "varlen launches: per-block scales, no split");
  using HV = typename HalfVec<F16V>::vec;
  using HS = typename HalfVec<F16V>::elem;
  constexpr int KS = ks_per_tile(KT);
  constexpr int kKTile = kBK * kD, kVTile = kD * kBK * 2;
  constexpr int NBS = OWN ? 2 * kHFBuf : kHFBuf;  // K (and V) buffers of the workgroup
  // the K buffers double as the waves' O stage (4 KiB per wave)
  constexpr int kKBytes = NBS * kKTile > 8 * 4096 ? NBS * kKTile : 8 * 4096;
  __shared__ __align__(16) uint8_t lds_k[kKBytes];
  __shared__ __align__(16) uint8_t lds_v[NBS * kVTile];
  __shared__ float lds_ksc[OWN ? 2 * kHFKsOwn : kHFKsPair];
  __shared__ int16_t lds_tid[OWN ? 2 * kHFKsOwn : 2];  // HF_OWN with a mask: ids of each group's tiles
  __shared__ int lds_n[4];

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 31, hf = lane >> 5;
  const int grp = w >> 2, wl = w & 3;

  // ---- this group's query block ----
  int64_t b, h, qb;
  int split = 0;
  bool live = true;
  [[maybe_unused]] uint32_t unit0 = 0;  // HF_OWN: group 0's (batch, head, query block)
  int64_t Lq = p.Lq, Lk = p.Lk;
  int64_t nqb_wg_last;  // last query block of the workgroup (its key range bounds the shared stream)
  if constexpr (VAR) {
    int vb, vh, vq;
    if (!varlen_item(p, (int)blockIdx.x, vb, vh, vq)) return;
    b = vb;
    h = vh;
    qb = (int64_t)vq * 2 + grp;
    nqb_wg_last = (int64_t)vq * 2 + 1;
  } else if constexpr (OWN) {
    const uint32_t units = (uint32_t)(p.B * p.Hq * p.nQB), wgs = (units + 1) / 2;
    const uint32_t wg = (uint32_t)xcd_remap(blockIdx.x, gridDim.x);
    split = SPLIT ? (int)(wg / wgs) : 0;
    unit0 = (wg - (uint32_t)split * wgs) * 2;
    const uint32_t u = unit0 + grp;
    live = u < units;
    const uint32_t uc = live ? u : units - 1, bh = uc / (uint32_t)p.nQB;
    qb = uc - bh * (uint32_t)p.nQB;
    b = bh / (uint32_t)p.Hq;
    h = bh - (uint32_t)b * (uint32_t)p.Hq;
    nqb_wg_last = qb;
  } else {
    int64_t qp;
    if (!SPLIT && p.causal) pair_of_workgroup<SPLIT, true>(p, split, b, h, qp);
    else pair_of_workgroup<SPLIT, false>(p, split, b, h, qp);
    qb = qp * 2 + grp;  // == nQB for the empty second group of an odd block count
    nqb_wg_last = min(qp * 2 + 1, p.nQB - 1);
  }
  const int64_t hk = (uint32_t)h / (uint32_t)p.group;

  const int8_t* q8b = p.q8 + b * p.qsb;
  const int8_t* k8b = p.k8 + b * p.ksb;
  int64_t vcol0 = 0;  // first key column of this entry in the V tile layout
  const float* qs_tab = p.q_scale + (b * p.Hq + h) * p.nQS;
  const float* ks_tab = p.k_scale + (b * p.Hkv + hk) * p.nKS;
  int64_t qs_stride = 1, ks_stride = 1;
  uint16_t* ob = static_cast<uint16_t*>(p.o) + b * p.osb;
  int64_t n_qs = p.nQS;
  if constexpr (VAR) {
    int64_t q0, k0s;
    varlen_range(p.cu_q, b, p.var_tq, p.Lq, q0, Lq);
    varlen_range(p.cu_k, b, p.var_tk, p.Lk, k0s, Lk);
    q8b = p.q8 + q0 * p.qsl;
    k8b = p.k8 + k0s * p.ksl;
    vcol0 = (int64_t)p.cu_vt[b] * kBK;
    qs_tab = p.q_scale + (int64_t)p.cu_qs[b] * p.Hq + h;
    ks_tab = p.k_scale + (int64_t)p.cu_ks[b] * p.Hkv + hk;
    qs_stride = p.Hq;
    ks_stride = p.Hkv;
    ob = static_cast<uint16_t*>(p.o) + q0 * p.osl;
    n_qs = (Lq + kBQ - 1) / kBQ;
    nqb_wg_last = min(nqb_wg_last, n_qs - 1);
  }
  const int64_t q_first = qb * kBQ;
  const int64_t wrow0 = q_first + wl * 32;
  const int64_t qrow = wrow0 + lq;

  // key range of this group, and of its tile stream (the workgroup's last non-empty block)
  int64_t kv_lim = Lk;
  if (p.kv_valid) kv_lim = min(kv_lim, (int64_t)p.kv_valid[b]);
  int64_t kv_end = kv_lim, kv_end_wg = kv_lim;
  if (p.causal) {
    kv_end = min(kv_lim, q_first + kBQ + p.q_offset);
    kv_end_wg = min(kv_lim, nqb_wg_last * kBQ + kBQ + p.q_offset);
  }
  const int kv_end_s = __builtin_amdgcn_readfirstlane((int)kv_end);
  // last key that the wave's first row may see (causal), clamped so that adding a row index stays in range
  constexpr int kNoDiag = INT32_MAX - 128;
  const int diag_s = p.causal ? __builtin_amdgcn_readfirstlane((int)min(wrow0 + p.q_offset, (int64_t)kNoDiag)) : kNoDiag;
  int n_slots = __builtin_amdgcn_readfirstlane(kv_end_wg > 0 && live ? (int)((kv_end_wg + kBK - 1) / kBK) : 0);
  const int t_lo = SPLIT ? split * p.tiles_per_split : 0;
  // Q rows on their way while the tile list is formed and the first tiles are fetched: 8 lanes x 16 B per row
  v4i qraw[4];
  {
    const int8_t* qbase = q8b + h * p.qsh;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int64_t row = wrow0 + i * 8 + (lane >> 3);
      qraw[i] = live && row < Lq ? *reinterpret_cast<const v4i*>(qbase + row * p.qsl + (lane & 7) * 16) : v4i{0, 0, 0, 0};
    }
  }
  // HF_OWN slots: the key tiles of this group's block (block-sparse: those the mask keeps,
  // sparse_int8_attn.py:57-58) with the tiles that the other group's block visits too in the first n_sh slots, in
  // the same slots for both.  A split takes its run of the slots.
  const bool sparse = OWN && p.tile_mask != nullptr;
  int n_sh = 0;
  if constexpr (OWN) {
    const uint32_t u2 = unit0 + (grp ^ 1), bh2 = u2 / (uint32_t)p.nQB;
    const int64_t qb2 = u2 - bh2 * (uint32_t)p.nQB;
    const uint32_t b2 = bh2 / (uint32_t)p.Hq, h2 = bh2 - b2 * (uint32_t)p.Hq;
    const bool same = live && b2 == (uint32_t)b && h2 / (uint32_t)p.group == (uint32_t)hk;  // (b2 == p.B past the end)
    int64_t kv_end2 = kv_lim;
    if (p.causal) kv_end2 = min(kv_lim, qb2 * kBQ + kBQ + p.q_offset);
    const int n2 = __builtin_amdgcn_readfirstlane(same && kv_end2 > 0 ? (int)((kv_end2 + kBK - 1) / kBK) : 0);
    n_sh = min(n_slots, n2);
    if (sparse) {
      if (wl == 0) {  // one wave of the group compacts the mask row with ballots; only this split's slots are stored
        const int8_t* mbase = p.tile_mask + (b * p.Hkv + hk) * p.tm_s1;
        const int8_t *mrow = mbase + qb * p.tm_s2, *mrow2 = n2 > 0 ? mbase + qb2 * p.tm_s2 : mrow;
        const int cap = SPLIT ? p.tiles_per_split : kHFKsOwn;
        int cnt = 0, both = 0;
        for (int pass = 0; pass < 2; pass++) {  // the shared tiles, then this block's own
          for (int base = 0; base < n_slots; base += 512) {  // (eight loads of each row in flight)
            int8_t m1[8], m2[8];
            bool act[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
              const int t = base + u * 64 + lane;
              m1[u] = mrow[min(t, n_slots - 1)];
              m2[u] = mrow2[min(t, max(n2 - 1, 0))];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
              const int t = base + u * 64 + lane;
              act[u] = t < n_slots && m1[u] != 0 && (t < n2 && m2[u] != 0) == (pass == 0);
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
              const uint64_t bal = __ballot(act[u]);
              const int slot = cnt + __popcll(bal & ((1ull << lane) - 1ull));
              if (act[u] && slot >= t_lo && slot < t_lo + cap)
                lds_tid[grp * kHFKsOwn + slot - t_lo] = (int16_t)(base + u * 64 + lane);
              cnt += __popcll(bal);
            }
          }
          if (pass == 0) both = cnt;
        }
        if (lane == 0) {
          lds_n[grp] = cnt;
          lds_n[2 + grp] = both;
        }
      }
      __syncthreads();
      n_slots = __builtin_amdgcn_readfirstlane(lds_n[grp]);
      n_sh = __builtin_amdgcn_readfirstlane(lds_n[2 + grp]);
    }
  }
  const int t_end = SPLIT ? min(n_slots, t_lo + p.tiles_per_split) : n_slots;
  const int n_kt = max(t_end - t_lo, 0);  // slots 0 .. n_kt - 1 of this group, from here on
  // A pair streams the tiles of its last block; those past this block's own diagonal are not multiplied (their p is 0, but
  // a V that is not finite would make NaN of it, in rows that may not see its key).
  const int n_live = OWN ? n_kt : max(min((kv_end_s + kBK - 1) / kBK, t_end) - t_lo, 0);
  int n_own = 0;  // slots after the shared ones, of the longer group
  if constexpr (OWN) {
    n_sh = max(min(n_sh, t_end) - t_lo, 0);
    __syncthreads();  // (lds_n is read above)
    if (wl == 0 && lane == 0) lds_n[grp] = n_kt;
    __syncthreads();
    n_own = __builtin_amdgcn_readfirstlane(max(lds_n[0], lds_n[1])) - n_sh;
  } else {
    n_sh = n_kt;
  }
  auto tile_of = [&](int i) -> int {  // key tile of slot i (wave-uniform)
    if constexpr (OWN) {
      if (sparse) return __builtin_amdgcn_readfirstlane((int)lds_tid[grp * kHFKsOwn + i]);
    }
    return t_lo + i;
  };
  // (clamped to the entry's table: the empty second group of an odd block count reads its neighbour's scale)
  const int64_t qsi = min(q_scale_index(p, min(qb * kBQ + wl * 32 + lq, (int64_t)INT32_MAX)), n_qs - 1);
  const float qs = qs_tab[qsi * qs_stride] * p.qk_mult;

  // ---- K/V tiles by LDS DMA, fragment-major ----
  //   K block j (0..7): lane l gets K row (j & 1) * 32 + l % 32, bytes 16 (2 (j >> 1) + l / 32) .. + 16
  //   V block 4 dblk + c (0..15): lane l gets V^T row dblk * 32 + l % 32, bytes 16 (4 (l / 32) + c) .. + 16
  // A shared tile is fetched by all eight waves (one K and two V blocks each), a group's own by its four (two and
  // four): wave wl's blocks wl + 4 i are its group's share of both, i = grp of K and i = grp, grp + 2 of V.
  const int8_t* kbase = k8b + hk * p.ksh;
  const uint8_t* vbase = static_cast<const uint8_t*>(p.v) + ((VAR ? 0 : b) * p.Hkv + hk) * (int64_t)kD * p.Lpad * 2 + vcol0 * 2;
  const int64_t kbytes = (Lk - 1) * p.ksl + kD;
  const v4u vrsrc = make_rsrc(vbase, (uint32_t)(((int64_t)kD * p.Lpad - vcol0) * 2));
  constexpr int NKO = OWN ? 2 : 1, NVO = OWN ? 4 : 2;  // blocks whose offsets a wave holds
  uint32_t koff[NKO], voff[NVO];
#pragma unroll
  for (int i = 0; i < NKO; i++) {
    const int j = (OWN ? i : grp) * 4 + wl;
    koff[i] = (uint32_t)(((j & 1) * 32 + lq) * p.ksl + (2 * (j >> 1) + hf) * 16);
  }
#pragma unroll
  for (int i = 0; i < NVO; i++) {
    const int f = (OWN ? i : grp + 2 * i) * 4 + wl;
    voff[i] = (uint32_t)(((f >> 2) * 32 + lq) * p.Lpad * 2 + (4 * hf + (f & 3)) * 16);
  }
  const int64_t k_step = kBK * p.ksl;
  const uint32_t lds_k0 = lds_addr(lds_k) + wl * 1024, lds_v0 = lds_addr(lds_v) + wl * 1024;
  // K / V of a tile into buffer buf of the shared stream or of the group's own (buffers grp * kHFBuf ..)
  auto dma_k = [&](auto sh_t, int tile, int buf) __attribute__((always_inline)) {
    const int64_t kso = (int64_t)__builtin_amdgcn_readfirstlane(tile) * k_step;
    const v4u krsrc = make_rsrc(kbase + kso, (uint32_t)(kbytes - kso));
    if constexpr (decltype(sh_t)::value) {
      const uint32_t kl = __builtin_amdgcn_readfirstlane(lds_k0 + buf * kKTile + grp * 4096);
      lds_dma16(OWN && grp ? koff[NKO - 1] : koff[0], krsrc, 0, kl);
    } else {
      const uint32_t kl = __builtin_amdgcn_readfirstlane(lds_k0 + (grp * kHFBuf + buf) * kKTile);
#pragma unroll
      for (int d = 0; d < NKO; d++) lds_dma16(koff[d], krsrc, 0, kl + d * 4096);
    }
  };
  auto dma_v = [&](auto sh_t, int tile, int buf) __attribute__((always_inline)) {
    const uint32_t vso = (uint32_t)__builtin_amdgcn_readfirstlane(tile) * (kBK * 2);
    if constexpr (decltype(sh_t)::value) {
      const uint32_t vl = __builtin_amdgcn_readfirstlane(lds_v0 + buf * kVTile + grp * 4096);
#pragma unroll
      for (int d = 0; d < 2; d++)
        lds_dma16(OWN ? (grp ? voff[(2 * d + 1) % NVO] : voff[(2 * d) % NVO]) : voff[d % NVO], vrsrc, vso, vl + d * 8192);
    } else {
      const uint32_t vl = __builtin_amdgcn_readfirstlane(lds_v0 + (grp * kHFBuf + buf) * kVTile);
#pragma unroll
      for (int d = 0; d < NVO; d++) lds_dma16(voff[d], vrsrc, vso, vl + d * 4096);
    }
  };

  v16f o[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[i][r] = 0.f;
  float m_run = kMInit, l_run = 0.f;
  v16i kbias;
#pragma unroll
  for (int r = 0; r < 16; r++) kbias[r] = kAccBiasBits;

  // The first tiles of a stream, in the order that the steps go on with: K(0), then V(d), K(d + 1).
  // tq[d] is the tile of slot i + d of the step being run (i = 0 here): the ids of a mask come out of LDS one step
  // ahead, so that no DMA waits for its id.
  constexpr int kDKS = NBS - 1, kDKO = kHFBuf - 1;
  int tq_sh[kDKS + 1];
  [[maybe_unused]] int tq_own[kDKO + 1];
  auto fetch_first = [&](auto sh_t, int s0, int n, auto& tq) __attribute__((always_inline)) {
    constexpr int DK = decltype(sh_t)::value ? kDKS : kDKO;
    if (n > 0) {
#pragma unroll
      for (int d = 0; d <= DK; d++) tq[d] = sparse ? tile_of(s0 + min(d, n - 1)) : t_lo + s0 + d;
      dma_k(sh_t, tq[0], 0);
#pragma unroll
      for (int d = 0; d < DK - 1; d++) {
        if (d < n) dma_v(sh_t, tq[d], d);
        if (d + 1 < n) dma_k(sh_t, tq[d + 1], d + 1);
      }
    }
  };
  // K(0) has landed when all but the DK - 1 (V, K) pairs behind it have
  fetch_first(std::true_type{}, 0, n_sh, tq_sh);

  // Q fragments through a wave-private LDS stage (rows of 128 B, the 16-byte chunk c of row r at c ^ (r & 7)) in the
  // two V buffers that the first tiles leave free
  v4i qf[4];
  {
    uint8_t* qstage = lds_v + (NBS - 2) * kVTile + w * 4096;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = i * 8 + (lane >> 3), c = lane & 7;
      *reinterpret_cast<v4i*>(qstage + r * 128 + ((c ^ (r & 7)) << 4)) = qraw[i];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const int c = 2 * m + hf;
      qf[m] = *reinterpret_cast<const v4i*>(qstage + lq * 128 + ((c ^ (lq & 7)) << 4));
    }
#pragma unroll
    for (int m = 0; m < 4; m++) asm volatile("" ::"v"(qf[m]));
  }
  float* ksl = lds_ksc + (OWN ? grp * kHFKsOwn : 0);
  {
    const int step = OWN ? 256 : kHFThreads, first = OWN ? (tid & 255) : tid;
    for (int i = first; i < n_kt * KS; i += step) {
      int t = t_lo + i / KS;
      if (sparse) t = lds_tid[grp * kHFKsOwn + i / KS];
      ksl[i] = ks_tab[k_scale_index(p, t, i % KS, KS) * ks_stride];
    }
  }

  v16i s[2];
  HV ph[4];
  float cs_a, cs_b;
  auto pv = [&](int buf) __attribute__((always_inline)) {  // O^T += V^T . P^T, V from its buffer
    const uint8_t* vb = lds_v + buf * kVTile + lane * 16;
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int dblk = 0; dblk < 4; dblk++) {
        const HV vf = *reinterpret_cast<const HV*>(vb + (4 * dblk + c) * 1024);
        if constexpr (F16V) o[dblk] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, ph[c], o[dblk], 0, 0, 0);
        else o[dblk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, ph[c], o[dblk], 0, 0, 0);
      }
  };
  // slot i with K in buffer kbuf; the previous slot's V in buffer vbuf
  auto stage_m = [&](int i, int kbuf, int vbuf, auto first_t) __attribute__((always_inline)) {
    constexpr bool kFirst = decltype(first_t)::value;
    if constexpr (!kFirst) pv(vbuf);
    const uint8_t* kb_ = lds_k + kbuf * kKTile + lane * 16;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int m = j >> 1, kb = j & 1;
      const v4i kf = *reinterpret_cast<const v4i*>(kb_ + j * 1024);
      s[kb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[m], m == 0 ? kbias : s[kb], 0, 0, 0);
    }
    // the logit scales of the tile, for the softmax of the next stage
    if constexpr (KT) {
      cs_a = qs * ksl[i * 4 + 2 * hf];
      cs_b = qs * ksl[i * 4 + 2 * hf + 1];
    } else {
      cs_a = cs_b = qs * ksl[i];
    }
    if constexpr (!kFirst) {
      // LDS reads four ahead of the MFMA that consumes them (24 fragment reads and the key scale; 24 MFMAs)
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int r = 0; r < 20; r++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    }
  };
  auto stage_v = [&](int tile) __attribute__((always_inline)) {
    const int k0 = tile * kBK;
    const bool masked = (k0 + kBK > kv_end_s) || (k0 + kBK - 1 > diag_s);
    if (masked) {
      int lim = max(min(kv_end_s - k0, kBK), -1);
      lim = min(lim, max(min(diag_s + lq + 1 - k0, kBK), -1));
      lim -= hf * 4;
      asm volatile("" : "+v"(lim));  // (compared here, not as 32 lane masks kept in scalar registers)
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (kb * 32 + (r >> 2) * 8 + (r & 3) >= lim) s[kb][r] = INT32_MIN;
    }
    // p <= 1: the running max is kept kLazyTau above the tile max that moved it (see qattn_fwd_kernel)
    float m_tile;
    if constexpr (!KT) {
      int mx = max(s[0][0], s[0][1]);
#pragma unroll
      for (int r = 2; r < 16; r++) mx = max(mx, s[0][r]);
#pragma unroll
      for (int r = 0; r < 16; r++) mx = max(mx, s[1][r]);
      const auto sw = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
      mx = max((int)sw[0], (int)sw[1]);
      m_tile = mx == INT32_MIN ? kMInit : fmaf(__int_as_float(mx), cs_a, -fmaf(kAccBias, cs_a, -kLazyTau));
    } else {
      int ma = INT32_MIN, mb = INT32_MIN;
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          if ((r & 3) < 2) ma = max(ma, s[kb][r]);
          else mb = max(mb, s[kb][r]);
        }
      const float fa = ma == INT32_MIN ? kMInit : fmaf(__int_as_float(ma), cs_a, -fmaf(kAccBias, cs_a, -kLazyTau));
      const float fb = mb == INT32_MIN ? kMInit : fmaf(__int_as_float(mb), cs_b, -fmaf(kAccBias, cs_b, -kLazyTau));
      const float mt = fmaxf(fa, fb);
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
      m_tile = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    const bool grow = m_tile > m_run + kLazyTau;
    if (__any(grow)) {
      const float m_new = grow ? m_tile : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < 4; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[d][r] *= alpha;
      m_run = m_new;
    }
    const float nc_a = -fmaf(kAccBias, cs_a, m_run), nc_b = -fmaf(kAccBias, cs_b, m_run);
    auto body = [&](auto mk) {
      float lsum = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int kb = j >> 2, r0 = (j & 3) * 4;
        float pv4[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int sv = s[kb][r0 + e];
          pv4[e] = __builtin_amdgcn_exp2f(fmaf(__int_as_float(sv), e < 2 ? cs_a : cs_b, e < 2 ? nc_a : nc_b));
          // (masked logits become p = 0 exactly: the sentinel times a tiny scale is not necessarily very negative)
          if constexpr (decltype(mk)::value) pv4[e] = sv == INT32_MIN ? 0.f : pv4[e];
        }
        lsum += (pv4[0] + pv4[1]) + (pv4[2] + pv4[3]);
#pragma unroll
        for (int e = 0; e < 4; e++) ph[j >> 1][(j & 1) * 4 + e] = (HS)pv4[e];  // RNE
      }
      l_run += lsum;
    };
    if (masked) body(std::true_type{});
    else body(std::false_type{});
  };

  // Slots s0 .. s0 + n - 1 of a tile stream whose first tiles are on their way, in `steps` >= n steps (the longer
  // group's count): shared by the groups, or the group's own.
  auto phase = [&](auto sh_t, int s0, int n, int steps, auto& tq) __attribute__((always_inline)) {
    constexpr bool SH = decltype(sh_t)::value;
    constexpr int NB = SH ? NBS : kHFBuf, DK = NB - 1, DV = NB - 2;
    constexpr int kPer = SH ? 3 : 6, kPerK = SH ? 1 : 2;  // a wave's DMA instructions per tile, and those for K
    const int b0 = SH ? 0 : grp * kHFBuf;
    if (n > DK) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DV * kPer) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const int live = OWN ? steps : min(n_live, steps);
    int buf = 0;  // slot i's buffer, i % NB
    // live_t: false for the steps past the block's own tiles, which only fetch; the first of them still owes the last P.V
    auto step = [&](int i, auto first_t, auto live_t) __attribute__((always_inline)) {
      constexpr bool kLive = decltype(live_t)::value;
      const int prev = buf == 0 ? NB - 1 : buf - 1, prev2 = prev == 0 ? NB - 1 : prev - 1;
      if (SH || i < n) {
        const int left = n - DK - i;  // <= 0 at the stream's end: no K to issue, < 0: no V either
        if (left > 0) dma_k(sh_t, tq[DK], prev);
        if (left >= 0) dma_v(sh_t, tq[DV], prev2);
        if constexpr (kLive) {
          // (raised wave priority: the vector-stage wave of the SIMD cannot delay the issue of the MFMAs)
          __builtin_amdgcn_s_setprio(1);
          stage_m(s0 + i, b0 + buf, b0 + prev, first_t);
          __builtin_amdgcn_s_setprio(0);
        } else if (i == live && i > 0) {
          pv(b0 + prev);
        }
        // This wave's share of K(i + 1) and V(i), issued DV steps ago, has landed; what the last DV steps issued may
        // stay in flight (nothing was issued for slots past the end).
        if (left > 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DV * kPer) : "memory");
        else if (left == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DV * kPer - kPerK) : "memory");
        else if (DV > 1 && left == -1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DV > 1 ? (DV - 1) * kPer - kPerK : 0) : "memory");
        else if (DV > 2 && left == -2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DV > 2 ? (DV - 2) * kPer - kPerK : 0) : "memory");
        else if (DV > 3 && left == -3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DV > 3 ? (DV - 3) * kPer - kPerK : 0) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      pp_barrier();
      if (SH || i < n) {
        int nxt = tq[DK] + 1;
        if constexpr (OWN) {
          if (sparse) nxt = lds_tid[grp * kHFKsOwn + s0 + min(i + DK + 1, n - 1)];
        }
        if constexpr (kLive) stage_v(tq[0]);
#pragma unroll
        for (int d = 0; d < DK; d++) tq[d] = tq[d + 1];
        tq[DK] = OWN ? __builtin_amdgcn_readfirstlane(nxt) : nxt;
        buf = buf == NB - 1 ? 0 : buf + 1;
      }
      pp_barrier();
    };
    static_assert(DV <= 4, "vmcnt cases");
    if (grp == 1) pp_barrier();
    if (live > 0) step(0, std::true_type{}, std::true_type{});
    for (int i = 1; i < live; i++) step(i, std::false_type{}, std::true_type{});
    if constexpr (!OWN)
      for (int i = live; i < steps; i++) step(i, std::false_type{}, std::false_type{});
    if (grp == 0) pp_barrier();
    if (n > 0 && live == steps) pv(b0 + (buf == 0 ? NB - 1 : buf - 1));
  };
  phase(std::true_type{}, 0, n_sh, n_sh, tq_sh);
  if constexpr (OWN) {
    if (n_own > 0) {
      __syncthreads();  // both groups are done with the shared stream's buffers
      fetch_first(std::false_type{}, n_sh, n_kt - n_sh, tq_own);
      phase(std::false_type{}, n_sh, n_kt - n_sh, n_own, tq_own);
    }
  }

  const auto lsw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
  const float l_tot = __uint_as_float(lsw[0]) + __uint_as_float(lsw[1]);
  if constexpr (SPLIT) {
    // the split's partial (unnormalised O, m, l) for the combine kernel
    if (qrow >= Lq || !live) return;
    const int64_t row = (((int64_t)split * p.B + b) * p.Hq + h) * p.Lq + qrow;
    float* wo = p.ws_o + row * kD;
#pragma unroll
    for (int dblk = 0; dblk < 4; dblk++)
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

  // ---- epilogue: O / l out through a wave-private LDS stage (the K buffers are idle now) ----
  uint8_t* stage = lds_k + w * 4096;
  const float inv_l = l_tot > 0.f ? 1.0f / l_tot : 0.f;
  uint16_t* obase = ob + h * p.osh;
#pragma unroll
  for (int pass = 0; pass < 2; pass++) {
#pragma unroll
    for (int db = 0; db < 2; db++) {
      const int dblk = pass * 2 + db;
#pragma unroll
      for (int g = 0; g < 4; g++) {
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = epilogue_value<false>(o[dblk][g * 4 + e], inv_l, 1.f, 0.f);
        const v2u packed{pack_half2<F16OUT>(f[0], f[1]), pack_half2<F16OUT>(f[2], f[3])};
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
      if (live && row < Lq) *reinterpret_cast<v4u*>(obase + row * p.osl + pass * 64 + c * 8) = val;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  if (p.lse && hf == 0 && live && qrow < Lq)
    p.lse[(b * p.Hq + h) * p.Lq + qrow] = l_tot > 0.f ? __builtin_log2f(l_tot) + m_run : -INFINITY;
}

// A pair of query blocks per workgroup needs an even block count, or enough blocks that the idle second group of
// the last pair does not matter (at most 1/6 of the groups); other launches give each group a block of its own.
// A group of its own stages a quarter of a pair's k_scales, so key ranges past that (half_own_tiles) are pairs too.
static bool half_even(int64_t nqb) { return nqb % 2 == 0 || nqb >= 5; }
static int64_t half_own_tiles(bool kt) { return kHFKsOwn / ks_per_tile(kt); }
static bool half_pairs(int64_t nqb, bool kt, bool sparse, int64_t tiles) {
  return !sparse && (half_even(nqb) || tiles > half_own_tiles(kt));
}

int64_t half_max_tiles(bool kt, bool sparse) { return sparse ? half_own_tiles(kt) : kHFKsPair / ks_per_tile(kt); }

static int64_t half_workgroups(int64_t bh, int64_t nqb, bool pairs) {
  return pairs ? bh * ((nqb + 1) / 2) : (bh * nqb + 1) / 2;
}

// KV splits of a dense launch: the count that makes rounds of 256 workgroups (one per CU) x (key tiles + start-up
// and epilogue, about six tiles' worth) plus the combine cheapest.  A workgroup step is ~1.1 us per key tile (two
// wave-tiles per SIMD); a split writes and the combine reads 520 bytes per query row, at ~4 TB/s together, and costs
// a launch (~4 us).
int half_num_splits(int64_t bh, int64_t nqb, int64_t nkb, bool kt) {
  if (bh <= 0 || nqb <= 0 || nkb <= 0) return 1;
  const bool pairs = half_even(nqb);
  const int64_t max_tiles = pairs ? half_max_tiles(kt, false) : half_own_tiles(kt), min_s = (nkb + max_tiles - 1) / max_tiles;
  const int64_t wgs = half_workgroups(bh, nqb, pairs);
  int64_t best = min_s;
  double best_cost = 1e300;
  for (int64_t s = min_s; s <= std::max<int64_t>(min_s, std::min<int64_t>(32, nkb / 8)); s++) {
    const double rounds = (double)((wgs * s + 255) / 256), tiles = (double)((nkb + s - 1) / s);
    const double combine = s > 1 ? 4.0 + (double)(bh * nqb * kBQ) * s * 1040.0 / 4.0e6 : 0.0;  // us
    const double cost = rounds * (tiles + 6.0) * 1.1 + combine;
    if (cost < best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  return (int)best;
}

template <bool KT, bool SPLIT, int FORM>
static void launch_form(const AttnParams& p, int64_t g, int out_dtype, bool f16v, hipStream_t st) {
  if (out_dtype == QATTN_BF16) {
    if (f16v) qattn_fwd_half_kernel<false, true, KT, SPLIT, FORM><<<g, kHFThreads, 0, st>>>(p);
    else qattn_fwd_half_kernel<false, false, KT, SPLIT, FORM><<<g, kHFThreads, 0, st>>>(p);
  } else {
    if (f16v) qattn_fwd_half_kernel<true, true, KT, SPLIT, FORM><<<g, kHFThreads, 0, st>>>(p);
    else qattn_fwd_half_kernel<true, false, KT, SPLIT, FORM><<<g, kHFThreads, 0, st>>>(p);
  }
}

int launch_half(AttnParams& p, bool kt, bool f16v, bool sparse, int out_dtype, int ns, hipStream_t st) {
  p.nsplit = ns;
  p.tiles_per_split = (int)((p.nKB + ns - 1) / ns);
  const bool pairs = half_pairs(p.nQB, kt, sparse, p.tiles_per_split);
  const int64_t g = half_workgroups(p.B * p.Hq, p.nQB, pairs) * ns;
  QATTN_REQUIRE(g < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
  QATTN_REQUIRE(p.tiles_per_split <= half_max_tiles(kt, sparse), QATTN_ERR_SHAPE, "too many key tiles per workgroup");
  if (pairs) {
    if (ns > 1) {
      if (kt) launch_form<true, true, HF_PAIR>(p, g, out_dtype, f16v, st);
      else launch_form<false, true, HF_PAIR>(p, g, out_dtype, f16v, st);
    } else {
      if (kt) launch_form<true, false, HF_PAIR>(p, g, out_dtype, f16v, st);
      else launch_form<false, false, HF_PAIR>(p, g, out_dtype, f16v, st);
    }
  } else {
    if (ns > 1) {
      if (kt) launch_form<true, true, HF_OWN>(p, g, out_dtype, f16v, st);
      else launch_form<false, true, HF_OWN>(p, g, out_dtype, f16v, st);
    } else {
      if (kt) launch_form<true, false, HF_OWN>(p, g, out_dtype, f16v, st);
      else launch_form<false, false, HF_OWN>(p, g, out_dtype, f16v, st);
    }
  }
  if (ns > 1) launch_combine(p, out_dtype, kD, st);
  return check_launch("qattn_fwd");
}

int launch_half_varlen(AttnParams& p, int out_dtype, hipStream_t st) {
  p.nsplit = 1;
  p.tiles_per_split = (int)p.nKB;
  QATTN_REQUIRE(p.nKB <= kHFKsPair, QATTN_ERR_SHAPE, "varlen sequences hold at most %d keys", kHFKsPair * kBK);
  // pairs of the batch, bounded on the host without reading the lengths: sum of ceil(len / 256), or the slots of a
  // batch past kVarSorted, half the sum of ceil(len / 128) + 1
  const int64_t pairs = p.B <= kVarSorted
                            ? std::min((p.var_tq + 2 * kBQ - 1) / (2 * kBQ) + p.B, p.B * ((p.nQB + 1) / 2))
                            : std::min(p.var_tq / kBQ + 2 * p.B, p.B * (p.nQB + 1)) / 2;
  const int64_t g = p.Hq * pairs;
  QATTN_REQUIRE(g < (1ll << 31), QATTN_ERR_SHAPE, "grid too large");
  if (out_dtype == QATTN_BF16) qattn_fwd_half_kernel<false, true, false, false, HF_VAR><<<g, kHFThreads, 0, st>>>(p);
  else qattn_fwd_half_kernel<true, true, false, false, HF_VAR><<<g, kHFThreads, 0, st>>>(p);
  return check_launch("qattn_fwd_varlen");
}

}  // namespace qattn
