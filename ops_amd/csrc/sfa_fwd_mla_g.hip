// gfx950 MFMA forward of latent attention (d_qk = 576, d_v = 512, V the first
// 512 dims of the K rows) for up to 64 query heads per latent row: what one
// rank of a head-parallel group holds (16, 32 or 64 of 128 heads).  bf16 in,
// fp32 accumulate, paged or contiguous rows.
//
// Reference: `_attn_fwd` / `_inner_fwd` (lilac-me/ops SFA.py:309-587); the math
// is the one of the 128-head kernel in sfa_fwd_mfma.hip (masked base-2 online
// softmax with a lazy rescale, P V, sink, LSE, split-k partials).  With few
// heads a gathered row is used for few products (30 FLOP per byte at 16 heads),
// so the kernel is built around the gather:
//  * one workgroup of 4 waves per (batch, query, kv head[, split]) and all its
//    heads (up to 32, NG groups of 16, the MFMA's N; more take a workgroup per
//    32); 32-key tiles of whole 1152-byte
//    rows straight into LDS (RowGather), double buffered, 78 KB, so that two
//    workgroups share a CU and one's products cover the other's waits;
//  * S^T = K Q^T is divided over the waves by key half and, with 16 heads, by
//    halves of the 576 dims, with 32 by head group: a tile row is read once or
//    twice from LDS, not once per wave, and a wave keeps 36 or 72 Q registers;
//  * the scores go through LDS in the accumulator layout (lane-linear 16-byte
//    slots, conflict free); every wave forms the whole tile's softmax (the
//    same values in each) and P^T in the B-operand layout;
//  * O^T = V^T P^T is divided by dims, 128 per wave (32 NG accumulators).
// P keeps its 24 bits, as three bf16 terms (three MFMAs per operand), and
// split-k partials are fp32: the scalar kernel that these shapes ran on held
// both in fp32.  Share of outputs that are not the bf16 value nearest to the
// float64 result, over prefills and decodes of 16 to 64 heads: 1.8e-4 to 3.0e-4
// (scalar kernel 1.7e-4 to 5.5e-4; with two terms 1.7e-3 to 2.3e-3, at 450
// against 485 us for 2048 queries of 16 heads, 1110 against 1290 us of 64).
// Bound: with 16 heads the gather (4.8 GB in 0.44 ms, 11 TB/s, three quarters of
// it from L2 on ascending index rows, the rest from the Infinity Cache) and the
// serial chain of a tile, the matrix cores with 64.  2048 queries on 16384 keys,
// top-k 2048, 16 heads: 0.52 ms, 0.44 ms on ascending rows, 64.5 ms on the
// scalar kernel (one workgroup per query and head); 64 heads 1.28 ms.
// Up to 4 queries of 65 to 128 heads with 16384 slots in all (a few sequences'
// decode step) take it too, 16 heads per workgroup: the 128-head kernel loads all 147 KB of Q in
// every split before its first product.

#include "sfa_common.h"
#include "sfa_generic_row.h"
#include "sfa_lds.h"
#include "sfa_mfma.h"

namespace sfa {
namespace {

constexpr int kDqk = 576, kDv = 512;
constexpr int kCh = kDqk / 8;         // 16-byte chunks per row
constexpr int kKeys = 32;             // keys per tile
constexpr int kHalf = 256;            // slots per half of the staged index ring
constexpr int kOT = kDv / 4 / 16;     // 16-dim O^T tiles per wave
constexpr float kSlack = 8.0f;        // lazy-rescale slack (base-2 units)

// Base-2 log-sum-exp of 2^m2 l.  The logarithm is taken of l's mantissa: that of
// l itself, ~11 for 2048 slots below a lazy maximum, carries the rounding of
// its whole part (relative error of the LSE against float64 6e-8, now 4e-8).
__device__ __forceinline__ float lse2_of(float m2, float l) {
  int e;
  const float f = frexpf(l, &e);
  return m2 + ((float)e + log2f(f));
}
// ... and the natural one
__device__ __forceinline__ float lse_of(float m2, float l) {
  int e;
  const float f = frexpf(l, &e);
  return fmaf(m2, kLn2, fmaf((float)e, kLn2, logf(f)));
}

// LDS-only barrier: the DMA in flight (vmcnt) is not waited for.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// ... and with every DMA and load of this wave landed
__device__ __forceinline__ void full_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int NG, bool PAGED>
__global__ __launch_bounds__(256, 2) void fwd_mla_g_kernel(Params p) {
  using M = Mfma<16>;
  typedef M::acc_t acc_t;
  typedef typename std::conditional<PAGED, PoolRows, BufRowsOffUT>::type Src;
  typedef RowGather<kKeys, kCh, 4, true, Src, TileSwz16> RG;
  static_assert(NG == 1 || NG == 2, "S^T is divided over the wave pairs by dims (16 heads) or by head group (32)");
  constexpr int KS = NG == 1 ? 9 : 18;             // contraction steps (32 dims) of a wave's S^T
  constexpr int TILE = kKeys * kCh;                // 16-byte slots

  __shared__ u32x4 s_k[2 * TILE];                  // two tiles (the scalar fallback's scratch at the end)
  __shared__ f32x4 s_x[4][64];                     // [role][key half][lane]
  __shared__ int s_idx[2 * kHalf];                 // ring of staged slots: row offsets, < 0 invalid
  __shared__ int s_red[4];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lt = lane & 15, hq = lane >> 4;
  const int kt = wave & 1, role = wave >> 1;       // S^T: key half; dims half (NG = 1) or head group

  // ---- work item: its splits and head groups on one XCD (workgroup id % 8:
  // they share its Q or its rows), unsplit items in runs of 32 consecutive
  // queries on one XCD (shared keys meet in its L2); the last items, fewer than
  // 8, spread theirs over the XCDs (all of a small decode step: more CUs) ------
  const int64_t nitems = (int64_t)p.B * p.Sq * p.Hkv;
  const int nhg = (p.G + 16 * NG - 1) / (16 * NG), nsub = p.num_splits * nhg;
  const int runs = p.num_splits == 1 ? (int)(nitems / 256 * 256) : 0;  // items placed in runs
  const int eights = (int)((nitems - runs) / 8 * 8);                   // then items placed by eights
  int wi = blockIdx.x, sub;
  if (wi < runs * nsub) {
    const int x = wi % 8, r = wi / 8 / nsub;
    sub = wi / 8 % nsub;
    wi = ((r / 32) * 8 + x) * 32 + r % 32;
  } else {
    const int id = wi - runs * nsub, x = id % 8;
    if (id < eights * nsub) {
      sub = id / 8 % nsub;
      wi = runs + id / 8 / nsub * 8 + x;
    } else {
      sub = (id - eights * nsub) % nsub;
      wi = runs + eights + (id - eights * nsub) / nsub;
    }
  }
  const int split = sub / nhg, hg0 = (sub % nhg) * 16 * NG;  // split, first head of the group
  const int gheads = min(p.G - hg0, 16 * NG);
  const int g = wi % p.Hkv;
  wi /= p.Hkv;
  const int t = wi % p.Sq;
  const int b = wi / p.Sq;
  const int slot0 = split * p.split_len;
  const int nslots = max(0, min(p.topk - slot0, p.split_len));
  const int32_t* irow = p.idx + b * p.i_sb + t * p.i_ss + g * p.i_sh + slot0;
  const int bound = bound_of(p, b);

  // ---- Q^T B operands: lane holds head 16 ng + lt, dims 32 s + 8 hq ----------
  bf16x8 qb[KS];
  {
    const int hl = (NG == 1 ? 0 : 16 * role) + lt;
    const bf16* qrow = reinterpret_cast<const bf16*>(p.q) + b * p.q_sb + t * p.q_ss +
                       (int64_t)(g * p.G + hg0 + min(hl, gheads - 1)) * p.q_sh + 8 * hq + (NG == 1 ? role * 288 : 0);
#pragma unroll
    for (int s = 0; s < KS; ++s) qb[s] = *reinterpret_cast<const bf16x8*>(qrow + 32 * s);
  }

  // ---- rows ------------------------------------------------------------------
  Src src;
  const int64_t kbyte0 = 2 * ((PAGED ? 0 : b * p.k_sb) + g * p.k_sh);
  if constexpr (PAGED) {
    src.base = reinterpret_cast<const char*>(p.k) + kbyte0;
    src.shift = p.pool_shift;
  } else {
    src.rs = make_rsrc(reinterpret_cast<const char*>(p.k) + kbyte0, (uint32_t)(2 * ((int64_t)(p.Skv - 1) * p.k_ss + kDqk)));
    src.row_bytes = (uint32_t)(2 * p.k_ss);
  }
  // A slot is staged in steps, so that the loads of one are in flight over
  // several tiles: its key id, (paged) the page of that id, its row's offset
  // (negative: invalid).
  auto slot_id = [&](int i) { return i < nslots ? irow[i] : -1; };
  const uint32_t tbytes =
      PAGED ? (uint32_t)(4 * ((int64_t)(p.B - 1) * p.bt_sb + (((int64_t)p.Skv + (1 << p.page_shift) - 1) >> p.page_shift))) : 0u;
  const __amdgpu_buffer_rsrc_t rt = make_rsrc(p.block_table, tbytes);
  auto page_of = [&](int id) -> int {
    if constexpr (!PAGED) return 0;
    const bool ok = id >= 0 && id < bound;
    return (int)__builtin_amdgcn_raw_buffer_load_b32(
        rt, ok ? 4u * (uint32_t)((int64_t)b * p.bt_sb + (id >> p.page_shift)) : tbytes, 0, 0);
  };
  auto row_off = [&](int id, int pg) -> int {
    const bool ok = id >= 0 && id < bound;
    if constexpr (PAGED) {
      const uint32_t r = ((uint32_t)pg << p.page_shift) | (uint32_t)(id & ((1 << p.page_shift) - 1));
      return ok && pg >= 0 && pg < p.num_pages
                 ? (int)(pool_row_offset(r, p.page_shift, (uint64_t)(2 * p.k_sb), (uint32_t)(2 * p.k_ss)) >> p.pool_shift)
                 : -1;
    } else {
      return ok ? (int)__umul24((uint32_t)id, src.row_bytes) : (int)kOOBRow;
    }
  };

  // tiles past the last valid slot (trailing padding) contribute nothing
  int used = 0;
#pragma unroll 8
  for (int i = tid; i < nslots; i += 256) {
    const int id = irow[i];
    if (id >= 0 && id < bound) used = i + 1;
  }
  used = wave_max_int(used);
  if (lane == 0) s_red[wave] = used;
  int next_id = slot_id(tid), next_pg = page_of(next_id);  // the slots of the half that is staged next
  s_idx[tid] = row_off(next_id, next_pg);
  __syncthreads();
  const int ntiles = (max(max(s_red[0], s_red[1]), max(s_red[2], s_red[3])) + kKeys - 1) / kKeys;

  RG rg;
  auto fetch_ids = [&](int j, int (&raw)[RG::RPW]) { RG::fetch(s_idx + (j * kKeys) % (2 * kHalf), wave, raw); };
  auto gather = [&](const int (&raw)[RG::RPW], u32x4* dst) {
    rg.set(raw, true, src);
#pragma unroll
    for (int k = 0; k < RG::NI; ++k) rg.issue(k, src, dst, wave, lane);
  };
  if (ntiles > 0) {
    int raw[RG::RPW];
    fetch_ids(0, raw);
    gather(raw, s_k);
  }

  // ---- operand addresses ------------------------------------------------------
  // K A operand (16 keys x 32 dims): row 16 kt + lt, chunk 4 s + hq; the
  // swizzle moves a chunk within its aligned 8, so two lane offsets serve
  const int krow = 16 * kt + lt;
  const int kc0 = NG == 1 ? role * 36 : 0;  // the wave's first chunk
  uint32_t ka[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int c = kc0 + 4 * e;
    ka[e] = (uint32_t)(krow * kCh + (c & ~7) + (((c & 7) + hq) ^ TileSwz16::at(krow))) * 16u;
  }
  // V^T A operand (16 dims x 32 keys): transposing reads of 4-row runs at keys
  // 4 hq and 16 + 4 hq (the P^T order of the exchanged scores), lane's piece
  // cc of 4 dims; dims 128 wave + 16 ot
  const int gi = lane & 15, rr = gi >> 2, cc = gi & 3;
  const int vrow = 4 * hq + rr;
  uint32_t va[4];
#pragma unroll
  for (int o = 0; o < 4; ++o)
    va[o] = (uint32_t)(vrow * kCh + 16 * wave + ((2 * o + (cc >> 1)) ^ TileSwz16::at(vrow))) * 16u + (uint32_t)(cc & 1) * 8u;

  acc_t oacc[NG][kOT];
  float m_used[NG], l_part[NG];
#pragma unroll
  for (int n = 0; n < NG; ++n) {
    m_used[n] = kNegInf;
    l_part[n] = 0.f;
#pragma unroll
    for (int i = 0; i < kOT; ++i) oacc[n][i] = acc_t{};
  }

  auto step = [&](int j, const u32x4* kb, u32x4* kn) {
    full_barrier();  // tile j has landed for all waves; the other buffer and the scores of tile j - 1 are read
    // the next half of the ring: its slots' loads go out at tiles 0 and 3 of
    // this half and have landed by a later tile's barrier; stored at tile 6
    // (its last readers were a half behind, its first is tile 7's gather)
    const int half = j / (kHalf / kKeys), ph = j % (kHalf / kKeys);
    if ((half + 1) * kHalf < nslots) {
      if (ph == 0) next_id = slot_id((half + 1) * kHalf + tid);
      if (ph == 3) next_pg = page_of(next_id);
      if (ph == 6) s_idx[((half + 1) & 1) * kHalf + tid] = row_off(next_id, next_pg);
    }
    // Operand reads are issued a phase ahead of their use (the scheduling
    // barriers keep them there): ids and K operands before the next gather's
    // address arithmetic, V^T operands before the softmax (32 heads: two of
    // them, paged one: more spill, 1590 and 1875 against 1455 us for paged
    // prefills of 64 heads with two and four).  With each read next to its MFMA a tile of
    // 16 heads took 1.4 us, now 1.28.
    int raw[RG::RPW];
    if (j + 1 < ntiles) fetch_ids(j + 1, raw);
    const int vid = s_idx[(j * kKeys) % (2 * kHalf) + (lane & 31)];
    bf16x8 ko[9];
#pragma unroll
    for (int s = 0; s < 9; ++s) ko[s] = lds_read_b128(kb, ka[s & 1] + (uint32_t)(s >> 1) * 128u);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t vmask = (uint32_t)__ballot(vid >= 0);
    if (j + 1 < ntiles) gather(raw, kn);
    __builtin_amdgcn_sched_barrier(0);

    // S^T of this wave's keys (two chains)
    acc_t sacc[2] = {};
#pragma unroll
    for (int s = 0; s < 9; ++s) {
      sacc[s & 1] = M::mma(ko[s], qb[s], sacc[s & 1]);
      if constexpr (KS == 18) ko[s] = lds_read_b128(kb, ka[(s + 9) & 1] + (uint32_t)((s + 9) >> 1) * 128u);
    }
    if constexpr (KS == 18) {
#pragma unroll
      for (int s = 0; s < 9; ++s) sacc[s & 1] = M::mma(ko[s], qb[KS == 18 ? 9 + s : s], sacc[s & 1]);
    }
    s_x[role * 2 + kt][lane] = sacc[0] + sacc[1];
    lds_barrier();

    f32x4 x[NG][2];
#pragma unroll
    for (int n = 0; n < NG; ++n)
#pragma unroll
      for (int h = 0; h < 2; ++h) x[n][h] = s_x[n * 2 + h][lane];
    if constexpr (NG == 1) {
      x[0][0] += s_x[2][lane];
      x[0][1] += s_x[3][lane];
    }
    constexpr int PRE = NG == 1 ? kOT : PAGED ? 1 : 2;
    bf16x4 vo[kOT][2];
    auto read_v = [&](int ot) {
      const uint32_t off = va[ot & 3] + (uint32_t)(ot >> 2) * 128u;
      vo[ot][0] = lds_read_tr16(kb, off);
      vo[ot][1] = lds_read_tr16(kb, off + 16u * kCh * 16u);
    };
#pragma unroll
    for (int ot = 0; ot < PRE; ++ot) read_v(ot);
    __builtin_amdgcn_sched_barrier(0);

    // softmax of head group n over this lane's 8 keys: key(kt, e) = 16 kt + 4 hq + e
    bf16x8 phi[NG], pmid[NG], plo[NG];
#pragma unroll
    for (int n = 0; n < NG; ++n) {
      float sv[8];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = 16 * h + 4 * hq + e;
          sv[4 * h + e] = (vmask == 0xffffffffu || ((vmask >> key) & 1u)) ? x[n][h][e] * p.scale_log2 : kNegInf;
        }
      }
      float tmax = fmaxf(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])), fmaxf(fmaxf(sv[4], sv[5]), fmaxf(sv[6], sv[7])));
      tmax = xor32_max(xor16_max(tmax));
      const float m_new = fmaxf(m_used[n], tmax);
      if (__any(m_new > m_used[n] + kSlack)) {
        const float alpha = (m_new == kNegInf) ? 1.f : exp2f(m_used[n] - m_new);
        l_part[n] *= alpha;
#pragma unroll
        for (int i = 0; i < kOT; ++i) oacc[n][i] *= alpha;
        m_used[n] = m_new;
      }
      const float moff = (m_used[n] == kNegInf) ? 0.f : m_used[n];
      float ex[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        ex[i] = __builtin_amdgcn_exp2f(sv[i] - moff);
        phi[n][i] = (bf16)ex[i];
        const float rest = ex[i] - (float)phi[n][i];
        pmid[n][i] = (bf16)rest;
        plo[n][i] = (bf16)(rest - (float)pmid[n][i]);
      }
      l_part[n] += ((ex[0] + ex[1]) + (ex[2] + ex[3])) + ((ex[4] + ex[5]) + (ex[6] + ex[7]));
    }

    // O^T += V^T P^T
#pragma unroll
    for (int ot = 0; ot < kOT; ++ot) {
      if (ot + PRE < kOT) read_v(ot + PRE);
      const bf16x4 lo = vo[ot][0], hi = vo[ot][1];
      const bf16x8 a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
      for (int n = 0; n < NG; ++n) {
        oacc[n][ot] = M::mma(a, phi[n], oacc[n][ot]);
        oacc[n][ot] = M::mma(a, pmid[n], oacc[n][ot]);
        oacc[n][ot] = M::mma(a, plo[n], oacc[n][ot]);
      }
    }
  };
  for (int j = 0; j < ntiles; j += 2) {
    step(j, s_k, s_k + TILE);
    if (j + 1 < ntiles) step(j + 1, s_k + TILE, s_k);
  }

  // ---- finish -------------------------------------------------------------------
  const bool partial = p.num_splits > 1;
  const int64_t nrows = (int64_t)p.B * p.Sq * p.Hq;
  bool nan = false;
#pragma unroll
  for (int n = 0; n < NG; ++n) {
    float l_sum = l_part[n];
    l_sum += __shfl_xor(l_sum, 16, 64);
    l_sum = xor32_sum(l_sum);
    const int hl = 16 * n + lt;
    if (hl >= gheads) continue;
    const int h = g * p.G + hg0 + hl;
    const int64_t row = ((int64_t)b * p.Sq + t) * p.Hq + h;
    const float m_fin = m_used[n];
    float scale_o, lse;  // lse: base 2 in a partial
    if (partial) {
      scale_o = l_sum > 0.f ? 1.f / l_sum : 0.f;
      lse = l_sum > 0.f ? lse2_of(m_fin, l_sum) : kNegInf;
    } else {
      const float sink2 = p.sink ? p.sink[h] * kLog2e : kNegInf;
      const float mm = fmaxf(m_fin, sink2);
      const float fo = (m_fin == kNegInf) ? 0.f : exp2f(m_fin - mm);
      float l = l_sum * fo;
      if (p.sink && mm != kNegInf) l += exp2f(sink2 - mm);
      scale_o = l > 0.f ? fo / l : 0.f;
      lse = l > 0.f ? lse_of(mm, l) : kNegInf;
    }
    if (wave == 0 && hq == 0) {
      if (partial)
        p.part_lse[split * nrows + row] = lse;
      else
        p.lse[b * p.l_sb + t * p.l_ss + (int64_t)h * p.l_sh] = lse;
    }
    nan |= l_sum != l_sum;
    // C layout: head lt, dims 128 wave + 16 ot + 4 hq + e
    const int d0 = 128 * wave + 4 * hq;
#pragma unroll
    for (int ot = 0; ot < kOT; ++ot) {
      const f32x4 v = oacc[n][ot] * scale_o;
      nan |= v[0] != v[0] || v[1] != v[1] || v[2] != v[2] || v[3] != v[3];
      if (partial) {
        *reinterpret_cast<f32x4*>(p.part_of + (split * nrows + row) * kDv + d0 + 16 * ot) = v;
      } else {
        const bf16x4 v4 = {(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
        *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(p.out) + b * p.o_sb + t * p.o_ss + (int64_t)h * p.o_sh + d0 +
                                   16 * ot) = v4;
      }
    }
  }
  // rows with infinities: the scalar loop's answer (see sfa_generic_row.h),
  // over the stores above
  full_barrier();
  if (lane == 0) s_red[wave] = 0;
  if (__any(nan) && lane == 0) s_red[wave] = 1;
  __syncthreads();
  if (s_red[0] | s_red[1] | s_red[2] | s_red[3]) {
    static_assert((kDqk + kMlaGMaxTopk + kRowWaves) * 4 <= 2 * TILE * 16, "the scalar loop's scratch fits the tiles");
    float* smem = reinterpret_cast<float*>(s_k);
    for (int hl = 0; hl < gheads; ++hl) {
      const int h = g * p.G + hg0 + hl;
      const int64_t row = ((int64_t)b * p.Sq + t) * p.Hq + h;
      __syncthreads();
      const float lse2 = generic_fwd_row<bf16>(p, b, t, h, slot0, nslots, !partial, smem, [&](int d, float x) {
        if (partial)
          p.part_of[(split * nrows + row) * kDv + d] = x;
        else
          reinterpret_cast<bf16*>(p.out)[b * p.o_sb + t * p.o_ss + (int64_t)h * p.o_sh + d] = (bf16)x;
      });
      if (tid == 0) {
        if (partial)
          p.part_lse[split * nrows + row] = lse2;
        else
          p.lse[b * p.l_sb + t * p.l_ss + (int64_t)h * p.l_sh] = lse2 * kLn2;
      }
    }
  }
}

// Merge of the fp32 split partials: one wave per row, lane s holds split s's
// weight, a lane's 8 dims of up to 8 splits are loaded together.  A split whose
// sum is not a number says so in its log-sum-exp: the row's weights, and with
// them the row, are then NaN whatever the other splits hold (a max drops a NaN,
// so it is looked at itself).  A sink that is not finite only takes the sum: it
// leaves zeros, as in the unsplit kernel.
__global__ __launch_bounds__(256) void combine_f32_kernel(Params p) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t nrows = (int64_t)p.B * p.Sq * p.Hq;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= nrows) return;
  const int h = row % p.Hq;
  const int t = (row / p.Hq) % p.Sq;
  const int b = row / ((int64_t)p.Hq * p.Sq);
  const float* part = p.part_of + row * kDv + 8 * lane;
  const int64_t stride = nrows * kDv;
  constexpr int U = 8;
  f32x4 x0[U], x1[U];
  auto load = [&](int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = min(s0 + u, p.num_splits - 1);
      x0[u] = *reinterpret_cast<const f32x4*>(part + s * stride);
      x1[u] = *reinterpret_cast<const f32x4*>(part + s * stride + 4);
    }
  };
  load(0);
  const float ls = lane < p.num_splits ? p.part_lse[lane * nrows + row] : kNegInf;
  const float sink2 = p.sink ? p.sink[h] * kLog2e : kNegInf;
  const float mm = fmaxf(wave_max(ls), sink2);
  const float e = ls != ls ? ls : (ls == kNegInf || mm == kNegInf) ? 0.f : exp2f(ls - mm);
  const float le = wave_sum(e);
  float l = le;
  if (p.sink && mm != kNegInf) l += exp2f(sink2 - mm);
  const float wl = l > 0.f ? e / l : (le != le ? le : 0.f);  // weight of split `lane`
  f32x4 a0{}, a1{};
  for (int s0 = 0; s0 < p.num_splits; s0 += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float w = s0 + u < p.num_splits ? __shfl(wl, s0 + u, 64) : 0.f;
      if (w != 0.f) {
        a0 += w * x0[u];
        a1 += w * x1[u];
      }
    }
    if (s0 + U < p.num_splits) load(s0 + U);
  }
  const bf16x8 o = {(bf16)a0[0], (bf16)a0[1], (bf16)a0[2], (bf16)a0[3], (bf16)a1[0], (bf16)a1[1], (bf16)a1[2], (bf16)a1[3]};
  *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16*>(p.out) + b * p.o_sb + t * p.o_ss + (int64_t)h * p.o_sh + 8 * lane) = o;
  if (lane == 0) p.lse[b * p.l_sb + t * p.l_ss + (int64_t)h * p.l_sh] = (l > 0.f) ? lse_of(mm, l) : kNegInf;
}

template <int NG>
void launch_ng(const Params& p, dim3 grid, hipStream_t s) {
  if (p.block_table)
    hipLaunchKernelGGL((fwd_mla_g_kernel<NG, true>), grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((fwd_mla_g_kernel<NG, false>), grid, dim3(256), 0, s, p);
}

}  // namespace

// Heads per workgroup: 16 for a few queries of many heads, else 32.  Four
// groups (64 heads in one workgroup, one wave per SIMD) keep each row's gather
// single but leave the products nothing to overlap with: 2048 queries of 64
// heads 1.57 against 1.18 ms in two workgroups that meet in their XCD's L2.
int fwd_mla_g_groups(const Params& p) { return p.G <= 64 ? (p.G + 31) / 32 : (p.G + 15) / 16; }

hipError_t launch_fwd_mla_g(const Params& p, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)p.B * p.Sq * p.Hkv * p.num_splits * fwd_mla_g_groups(p)));
  if (p.G <= 16 || p.G > 64)
    launch_ng<1>(p, grid, s);
  else
    launch_ng<2>(p, grid, s);
  return hipGetLastError();
}

hipError_t launch_combine_f32(const Params& p, hipStream_t s) {
  const int64_t rows = (int64_t)p.B * p.Sq * p.Hq;
  hipLaunchKernelGGL(combine_f32_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, p);
  return hipGetLastError();
}

}  // namespace sfa
