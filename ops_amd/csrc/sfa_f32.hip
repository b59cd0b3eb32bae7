// float32 sparse flash attention on the fp32 matrix instructions, d_qk = d_v =
// 64 or 128, any number of heads (16 per workgroup), contiguous or paged rows.
//
// Reference: SFA.py:309-587 (forward), 613-1145 (backward).  The scalar kernels
// of sfa_generic.hip, which keep the other widths, take one workgroup per
// (query, head): its slots one after another, a dependent load and a wave
// reduction each, rows gathered again and dK / dV rows added again for every
// head.  Here a workgroup of 4 waves owns a query and up to 16 heads
// (v_mfma_f32_16x16x4_f32, exact fp32 products, fp32 sums), in windows of 256
// slots:
//  * S^T = K Q^T (and dP^T = V dO^T): a wave takes 16 keys at a time straight
//    from global memory into the A operand; lane (key, hq) loads dims 16 j +
//    4 hq .. +3 as one float4, whose elements are four contraction steps (Q has
//    the same order);
//  * the scores meet in LDS ([head][slot]), where 16 lanes per head form the
//    softmax (forward) or each lane its P and dS (backward);
//  * O = P V (dQ = dS K): a wave takes every fourth group of 4 slots; a load
//    instruction reads 4 whole rows, float4 per lane, whose elements are four
//    16-dim tiles of the result (dims 4 n + e); the waves' sums meet in LDS;
//  * dK = dS^T Q (+ P^T dO when the rows are shared): contraction over the
//    heads, so a (key, dim) takes one fp32 atomic per query, not one per query
//    and head, added into the caller's gradient itself.
// Bound by latency at the sizes fp32 is used at (a chain of index, row, score,
// row loads per query); S = 256, 4 heads, d = 64, top-k 64: forward 26 -> 7 us,
// backward 52 -> 12 us against the scalar kernels.

#include "sfa_common.h"
#include "sfa_generic_row.h"

namespace sfa {
namespace {

constexpr int kW = 256;       // slots per window (one per thread)
constexpr int kPP = kW + 4;   // LDS pitch of a head's window (floats): operand reads hit distinct banks
constexpr int kHeads = 16;    // heads per workgroup
constexpr int kMaxTopkF32 = 8192;  // (the scalar fallback's scores fit the kernel's LDS)

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Contraction over the J float4 of a row: products of 4 dims per instruction,
// added as a tree.  (2-norm error against float64, S = 64 to 838, 4 to 16 heads,
// top-k 16 to 192: with one running sum over all 16 J dims out 1.8e-7 to 3.1e-7
// and dq 2.8e-7 to 4.4e-7, the scalar kernel's lanes and their tree 1.2e-7 to
// 2.1e-7 and 2.0e-7 to 3.2e-7, this 1.1e-7 to 1.5e-7 and 2.0e-7 to 3.1e-7.  B = 1, S
// = 2048, 32 heads on 8, d = 128, top-k 1024: forward 1802 -> 1859 us, backward
// 13.2 -> 13.1 ms.)
template <int J>
__device__ __forceinline__ f32x4 dot(const f32x4 (&a)[J], const f32x4 (&b)[J]) {
  f32x4 t[J];  // t[j]: the sum of the last 2^k, k the trailing ones of j
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const f32x4 z = {};
    t[j] = (mma4(a[j][0], b[j][0], z) + mma4(a[j][1], b[j][1], z)) + (mma4(a[j][2], b[j][2], z) + mma4(a[j][3], b[j][3], z));
#pragma unroll
    for (int n = 1; j & n; n *= 2) t[j] += t[j - n];
    asm volatile("" : "+v"(t[j]));  // (in this order: all products before the first sum take 4 J registers more)
  }
  return t[J - 1];
}

// sum / max over the 16 lanes of a group
__device__ __forceinline__ float sum16(float x) {
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) x += __shfl_xor(x, o, 16);
  return x;
}
__device__ __forceinline__ float max16(float x) {
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, 16));
  return x;
}

// Work item: (batch, query, kv head) and its group of 16 heads.
struct Item {
  int b, t, g, h0, nh;  // first query head, heads of the group
};
__device__ __forceinline__ Item item_at(const Params& p, int wi) {
  const int nhg = (p.G + kHeads - 1) / kHeads;
  Item it;
  const int hg = wi % nhg;
  wi /= nhg;
  it.g = wi % p.Hkv;
  wi /= p.Hkv;
  it.t = wi % p.Sq;
  it.b = wi / p.Sq;
  it.h0 = it.g * p.G + hg * kHeads;
  it.nh = min(kHeads, p.G - hg * kHeads);
  return it;
}

// Rows of k or v by staged id (key, or pool row when paged); negative: zeros.
struct Rows {
  const float* base;
  int64_t sb, ss;
  int shift, mask;
  __device__ __forceinline__ Rows(const Params& p, const void* ptr, int64_t sb_, int64_t ss_, int64_t sh, int b, int g) {
    const bool paged = p.block_table != nullptr;
    base = reinterpret_cast<const float*>(ptr) + (paged ? 0 : b * sb_) + g * sh;
    sb = sb_;
    ss = ss_;
    shift = paged ? p.page_shift : 31;
    mask = paged ? (1 << p.page_shift) - 1 : 0x7fffffff;
  }
  __device__ __forceinline__ const float* at(int r) const {
    return r < 0 ? reinterpret_cast<const float*>(kZeroRow)
                 : base + (int64_t)((uint32_t)r >> shift) * sb + (int64_t)(r & mask) * ss;
  }
};

__device__ __forceinline__ int staged_row(const Params& p, int b, int id, int bound) {
  if (p.block_table) return paged_row(p, b, id, bound);
  return id >= 0 && id < bound ? id : -1;
}

template <int D>
__global__ __launch_bounds__(256) void fwd_f32_kernel(Params p) {
  constexpr int J = D / 16;  // float4 per lane of a row in the S^T operand order
  constexpr int V = D / 64;  // float4 per lane of a whole-row load
  constexpr int kScratch = D + kMaxTopkF32 + kRowWaves;
  constexpr int kLds = kHeads * kPP + 4 * kHeads * D;
  __shared__ __attribute__((aligned(16))) float s_mem[kLds > kScratch ? kLds : kScratch];
  __shared__ __attribute__((aligned(16))) int s_row[kW];
  __shared__ float s_alpha[kHeads];
  float* const s_p = s_mem;                   // [16][kPP]
  float* const s_red = s_mem + kHeads * kPP;  // [4][16][D]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, hq = lane >> 4;
  const int hs = tid >> 4, c = tid & 15;  // softmax: head, lane of its 16
  const Item it = item_at(p, blockIdx.x);
  const int32_t* irow = p.idx + it.b * p.i_sb + it.t * p.i_ss + it.g * p.i_sh;
  const int bound = bound_of(p, it.b);
  const Rows kr(p, p.k, p.k_sb, p.k_ss, p.k_sh, it.b, it.g), vr(p, p.v, p.v_sb, p.v_ss, p.v_sh, it.b, it.g);

  f32x4 q[J];
  {
    const float* qrow = reinterpret_cast<const float*>(p.q) + it.b * p.q_sb + it.t * p.q_ss +
                        (int64_t)(it.h0 + min(n, it.nh - 1)) * p.q_sh + 4 * hq;
#pragma unroll
    for (int j = 0; j < J; ++j) q[j] = *reinterpret_cast<const f32x4*>(qrow + 16 * j);
  }

  f32x4 o[V][4];
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[v][e] = f32x4{};
  float m_run = kNegInf, l_run = 0.f;

  for (int w0 = 0; w0 < p.topk; w0 += kW) {
    const int wn = min(kW, p.topk - w0);
    __syncthreads();  // the previous window's reads
    s_row[tid] = tid < wn ? staged_row(p, it.b, irow[w0 + tid], bound) : -1;
    __syncthreads();

    for (int kt = wave; 16 * kt < wn; kt += 4) {
      const float* row = kr.at(s_row[16 * kt + n]) + 4 * hq;
      f32x4 a[J];
#pragma unroll
      for (int j = 0; j < J; ++j) a[j] = *reinterpret_cast<const f32x4*>(row + 16 * j);
      f32x4 s = dot(a, q);
      // C layout: head n, keys 16 kt + 4 hq + e
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = s_row[16 * kt + 4 * hq + e] >= 0 ? s[e] * p.scale_log2 : kNegInf;
      *reinterpret_cast<f32x4*>(s_p + n * kPP + 16 * kt + 4 * hq) = s;
    }
    // the V rows of the wave's first steps, in flight over the softmax
    constexpr int PRE = 4;
    f32x4 pv[PRE][V];
#pragma unroll
    for (int i = 0; i < PRE; ++i) {
      const int key = 4 * (wave + 4 * i) + hq;
      const float* row = vr.at(key < wn ? s_row[key] : -1) + 4 * n;
#pragma unroll
      for (int v = 0; v < V; ++v) pv[i][v] = *reinterpret_cast<const f32x4*>(row + 64 * v);
    }
    __syncthreads();

    // softmax of head hs over the window
    {
      float x[kW / 16], mx = kNegInf, sum = 0.f;
      float* ph = s_p + hs * kPP + c;
#pragma unroll
      for (int i = 0; i < kW / 16; ++i) x[i] = 16 * i < wn ? ph[16 * i] : kNegInf;
#pragma unroll
      for (int i = 0; i < kW / 16; ++i) mx = fmaxf(mx, x[i]);
      const float m_new = fmaxf(m_run, max16(mx));
      const float alpha = m_run == kNegInf ? (m_new == kNegInf ? 1.f : 0.f) : exp2f(m_run - m_new);
#pragma unroll
      for (int i = 0; i < kW / 16; ++i) {
        if (16 * i >= wn) break;
        const float e = x[i] == kNegInf ? 0.f : exp2f(x[i] - m_new);
        sum += e;
        ph[16 * i] = e;
      }
      l_run = l_run * alpha + sum16(sum);
      m_run = m_new;
      if (c == 0) s_alpha[hs] = alpha;
    }
    __syncthreads();

    if (w0 > 0) {
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        const float al = s_alpha[4 * hq + e2];
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[v][e][e2] *= al;
      }
    }
    // O += P V: step i takes keys 4 (wave + 4 i) + hq
    auto pv_step = [&](int key, const f32x4 (&x)[V]) {
      const float a = s_p[n * kPP + key];
#pragma unroll
      for (int v = 0; v < V; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[v][e] = mma4(a, x[v][e], o[v][e]);
    };
#pragma unroll
    for (int i = 0; i < PRE; ++i)
      if (4 * (wave + 4 * i) < wn) pv_step(4 * (wave + 4 * i) + hq, pv[i]);
#pragma unroll 4
    for (int k0 = 4 * (wave + 4 * PRE); k0 < wn; k0 += 16) {
      f32x4 x[V];
      const float* row = vr.at(s_row[k0 + hq]) + 4 * n;
#pragma unroll
      for (int v = 0; v < V; ++v) x[v] = *reinterpret_cast<const f32x4*>(row + 64 * v);
      pv_step(k0 + hq, x);
    }
  }

  // head hs's denominator; the waves' sums (C layout: head 4 hq + e2, dims 64 v + 4 n + e)
  const int h = it.h0 + min(hs, it.nh - 1);
  float scale_o, lse2;
  {
    const float sink2 = p.sink ? p.sink[h] * kLog2e : kNegInf;
    const float mm = fmaxf(m_run, sink2);
    const float fo = m_run == kNegInf ? 0.f : exp2f(m_run - mm);
    float l = l_run * fo;
    if (p.sink && mm != kNegInf) l += exp2f(sink2 - mm);
    scale_o = l > 0.f ? fo / l : 0.f;
    lse2 = l > 0.f ? mm + log2f(l) : kNegInf;
  }
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int e2 = 0; e2 < 4; ++e2)
      *reinterpret_cast<f32x4*>(s_red + (wave * kHeads + 4 * hq + e2) * D + 64 * v + 4 * n) =
          f32x4{o[v][0][e2], o[v][1][e2], o[v][2][e2], o[v][3][e2]};
  __syncthreads();
  bool nan = l_run != l_run;
  const bool live = hs < it.nh;
  float* orow = reinterpret_cast<float*>(p.out) + it.b * p.o_sb + it.t * p.o_ss + (int64_t)h * p.o_sh;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int d = 64 * v + 4 * c;
    f32x4 x = *reinterpret_cast<const f32x4*>(s_red + hs * D + d);
#pragma unroll
    for (int w = 1; w < 4; ++w) x += *reinterpret_cast<const f32x4*>(s_red + (w * kHeads + hs) * D + d);
    x *= scale_o;
    nan |= x[0] != x[0] || x[1] != x[1] || x[2] != x[2] || x[3] != x[3];
    if (live) *reinterpret_cast<f32x4*>(orow + d) = x;
  }
  if (live && c == 0) p.lse[it.b * p.l_sb + it.t * p.l_ss + (int64_t)h * p.l_sh] = lse2 * kLn2;
  // rows with infinities: the scalar loop's answer, over the stores above
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (__syncthreads_or(nan && live)) {
    for (int i = 0; i < it.nh; ++i) {
      __syncthreads();
      float* out = reinterpret_cast<float*>(p.out) + it.b * p.o_sb + it.t * p.o_ss + (int64_t)(it.h0 + i) * p.o_sh;
      const float l2 = generic_fwd_row<float>(p, it.b, it.t, it.h0 + i, 0, p.topk, true, s_mem,
                                              [&](int d, float x) { out[d] = x; });
      if (tid == 0) p.lse[it.b * p.l_sb + it.t * p.l_ss + (int64_t)(it.h0 + i) * p.l_sh] = l2 * kLn2;
    }
  }
}

// Gradients of one query and 16 heads; MERGE: v is k (their one gradient, dK +
// dV, goes to dk_acc).  dk_acc / dv_acc are the caller's gradient tensors,
// zeroed before, with their strides.
template <int D, bool MERGE>
__global__ __launch_bounds__(256, 2) void bwd_f32_kernel(Params p, F32Grads gr) {
  constexpr int J = D / 16, V = D / 64;
  __shared__ __attribute__((aligned(16))) float s_mem[2 * kHeads * kPP];
  __shared__ __attribute__((aligned(16))) int s_row[kW];
  static_assert(4 * kHeads * D <= 2 * kHeads * kPP, "the waves' dQ sums fit the score windows");
  float* const s_p = s_mem;
  float* const s_ds = s_mem + kHeads * kPP;  // scale dS

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, hq = lane >> 4;
  const Item it = item_at(p, blockIdx.x);
  const int32_t* irow = p.idx + it.b * p.i_sb + it.t * p.i_ss + it.g * p.i_sh;
  const int bound = bound_of(p, it.b);
  const Rows kr(p, p.k, p.k_sb, p.k_ss, p.k_sh, it.b, it.g), vr(p, p.v, p.v_sb, p.v_ss, p.v_sh, it.b, it.g);
  const float* const q0 = reinterpret_cast<const float*>(p.q) + it.b * p.q_sb + it.t * p.q_ss + (int64_t)it.h0 * p.q_sh;
  const float* const d0 = reinterpret_cast<const float*>(p.dout) + it.b * p.do_sb + it.t * p.do_ss + (int64_t)it.h0 * p.do_sh;
  const float* const o0 = reinterpret_cast<const float*>(p.out) + it.b * p.o_sb + it.t * p.o_ss + (int64_t)it.h0 * p.o_sh;

  // B operands over dims (head n, dims 16 j + 4 hq + e) and over heads (head
  // 4 s + hq, dim 16 j + n; rows without a gradient zero), δ and the softmax's constants
  const bool live = n < it.nh;
  const int64_t hn = live ? n : it.nh - 1;
  f32x4 q[J], dob[J], od[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    q[j] = *reinterpret_cast<const f32x4*>(q0 + hn * p.q_sh + 16 * j + 4 * hq);
    dob[j] = *reinterpret_cast<const f32x4*>(d0 + hn * p.do_sh + 16 * j + 4 * hq);
    const f32x4 ov = *reinterpret_cast<const f32x4*>(o0 + hn * p.o_sh + 16 * j + 4 * hq);
    od[j] = dob[j] * ov;
  }
#pragma unroll
  for (int n2 = J / 2; n2 > 0; n2 /= 2)
#pragma unroll
    for (int j = 0; j < n2; ++j) od[j] += od[j + n2];
  float delta = (od[0][0] + od[0][1]) + (od[0][2] + od[0][3]);
  delta += __shfl_xor(delta, 16, 64);
  delta += __shfl_xor(delta, 32, 64);
  const int64_t lofs = it.b * p.l_sb + it.t * p.l_ss + (it.h0 + hn) * p.l_sh;
  if (p.dlse) delta -= p.dlse[lofs];
  if (wave == 0 && hq == 0 && live) p.delta[((int64_t)it.b * p.Sq + it.t) * p.Hq + it.h0 + n] = delta;
  const float lse = p.lse[lofs];
  // (a row with no valid slot and no sink, or an absent head, has no gradient:
  // its operands are zeros and its dQ is written as zeros, since 0 x inf is not 0)
  const bool row_live = live && lse != kNegInf;
  const float lse2 = lse * kLog2e;
  float qh[4][J], doh[4][J];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int64_t hh = 4 * s + hq;
    const bool on = __shfl((int)row_live, 4 * s + hq, 64);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      qh[s][j] = on ? q0[hh * p.q_sh + 16 * j + n] : 0.f;
      doh[s][j] = on ? d0[hh * p.do_sh + 16 * j + n] : 0.f;
    }
  }

  f32x4 dq[V][4];
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) dq[v][e] = f32x4{};

  for (int w0 = 0; w0 < p.topk; w0 += kW) {
    const int wn = min(kW, p.topk - w0);
    __syncthreads();
    s_row[tid] = tid < wn ? staged_row(p, it.b, irow[w0 + tid], bound) : -1;
    __syncthreads();

    for (int kt = wave; 16 * kt < wn; kt += 4) {
      const int r = s_row[16 * kt + n];
      const float* krow = kr.at(r) + 4 * hq;
      f32x4 a[J], b[MERGE ? 1 : J];
#pragma unroll
      for (int j = 0; j < J; ++j) a[j] = *reinterpret_cast<const f32x4*>(krow + 16 * j);
      if constexpr (!MERGE) {
        const float* vrow = vr.at(r) + 4 * hq;
#pragma unroll
        for (int j = 0; j < J; ++j) b[j] = *reinterpret_cast<const f32x4*>(vrow + 16 * j);
      }
      const f32x4 s = dot(a, q);
      f32x4 dp;
      if constexpr (MERGE)
        dp = dot(a, dob);
      else
        dp = dot(b, dob);
      f32x4 pr, ds;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = row_live && s_row[16 * kt + 4 * hq + e] >= 0;
        pr[e] = ok ? exp2f(s[e] * p.scale_log2 - lse2) : 0.f;
        ds[e] = ok ? p.scale * (pr[e] * (dp[e] - delta)) : 0.f;
      }
      *reinterpret_cast<f32x4*>(s_p + n * kPP + 16 * kt + 4 * hq) = pr;
      *reinterpret_cast<f32x4*>(s_ds + n * kPP + 16 * kt + 4 * hq) = ds;
    }
    __syncthreads();

    // dQ += dS K, step i: keys 4 (wave + 4 i) + hq (rows just read: L1 / L2)
#pragma unroll 4
    for (int k0 = 4 * wave; k0 < wn; k0 += 16) {
      const float* row = kr.at(s_row[k0 + hq]) + 4 * n;
      const float a = s_ds[n * kPP + k0 + hq];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(row + 64 * v);
#pragma unroll
        for (int e = 0; e < 4; ++e) dq[v][e] = mma4(a, x[e], dq[v][e]);
      }
    }
    // dK, dV of 16 keys: contraction over the heads (C layout: dim 16 j + n,
    // key 16 kt + 4 hq + e: an atomic instruction covers 64 bytes of 4 rows)
    for (int kt = wave; 16 * kt < wn; kt += 4) {
      float ads[4], ap[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        ads[s] = s_ds[(4 * s + hq) * kPP + 16 * kt + n];
        ap[s] = s_p[(4 * s + hq) * kPP + 16 * kt + n];
      }
      int r[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = s_row[16 * kt + 4 * hq + e];
      float *dk[4], *dv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        dk[e] = gr.dk + it.b * gr.dk_sb + (int64_t)r[e] * gr.dk_ss + it.g * gr.dk_sh + n;
        dv[e] = MERGE ? nullptr : gr.dv + it.b * gr.dv_sb + (int64_t)r[e] * gr.dv_ss + it.g * gr.dv_sh + n;
      }
#pragma unroll
      for (int j = 0; j < J; ++j) {
        f32x4 k4 = {}, v4 = {};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (4 * s >= it.nh) break;
          k4 = mma4(ads[s], qh[s][j], k4);
          if constexpr (MERGE)
            k4 = mma4(ap[s], doh[s][j], k4);
          else
            v4 = mma4(ap[s], doh[s][j], v4);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (r[e] < 0) continue;
          atomicAdd(dk[e] + 16 * j, k4[e]);
          if constexpr (!MERGE) atomicAdd(dv[e] + 16 * j, v4[e]);
        }
      }
    }
  }

  // the waves' dQ sums (head 4 hq + e2, dims 64 v + 4 n + e)
  __syncthreads();
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int e2 = 0; e2 < 4; ++e2)
      *reinterpret_cast<f32x4*>(s_mem + (wave * kHeads + 4 * hq + e2) * D + 64 * v + 4 * n) =
          f32x4{dq[v][0][e2], dq[v][1][e2], dq[v][2][e2], dq[v][3][e2]};
  __syncthreads();
  const int hs = tid >> 4, c = tid & 15;
  const bool on = __shfl((int)row_live, hs, 64);
  if (hs >= it.nh) return;
  float* dqrow = reinterpret_cast<float*>(p.dq) + it.b * p.dq_sb + it.t * p.dq_ss + (int64_t)(it.h0 + hs) * p.dq_sh;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int d = 64 * v + 4 * c;
    f32x4 x = *reinterpret_cast<const f32x4*>(s_mem + hs * D + d);
#pragma unroll
    for (int w = 1; w < 4; ++w) x += *reinterpret_cast<const f32x4*>(s_mem + (w * kHeads + hs) * D + d);
    *reinterpret_cast<f32x4*>(dqrow + d) = on ? x : f32x4{};
  }
}

// zeros into dk (and dv) rows of D floats with the caller's strides
__global__ void zero_grads_kernel(F32Grads gr, int B, int Skv, int Hkv, int D) {
  const int64_t n = (int64_t)B * Skv * Hkv * D;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int d = (int)(i % D);
    int64_t r = i / D;
    const int h = (int)(r % Hkv);
    r /= Hkv;
    const int64_t s = r % Skv, b = r / Skv;
    gr.dk[b * gr.dk_sb + s * gr.dk_ss + h * gr.dk_sh + d] = 0.f;
    if (gr.dv) gr.dv[b * gr.dv_sb + s * gr.dv_ss + h * gr.dv_sh + d] = 0.f;
  }
}

}  // namespace

// (the 16-byte row loads need aligned rows: checked by the caller, which
// knows which tensors the call has)
bool f32_mfma_supported(const Params& p) {
  return p.Dqk == p.Dv && (p.Dqk == 64 || p.Dqk == 128) && p.topk <= kMaxTopkF32;
}

hipError_t launch_fwd_f32(const Params& p, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)p.B * p.Sq * p.Hkv * ((p.G + kHeads - 1) / kHeads)));
  if (p.Dqk == 64)
    hipLaunchKernelGGL(fwd_f32_kernel<64>, grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL(fwd_f32_kernel<128>, grid, dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_bwd_f32(const Params& p, const F32Grads& gr, hipStream_t s) {
  const int64_t n = (int64_t)p.B * p.Skv * p.Hkv * p.Dqk, blocks = (n + 1023) / 1024;
  hipLaunchKernelGGL(zero_grads_kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)), dim3(256), 0, s, gr, p.B, p.Skv,
                     p.Hkv, p.Dqk);
  const dim3 grid((unsigned)((int64_t)p.B * p.Sq * p.Hkv * ((p.G + kHeads - 1) / kHeads)));
#define SFA_BWD_F32(D, M) hipLaunchKernelGGL((bwd_f32_kernel<D, M>), grid, dim3(256), 0, s, p, gr)
  if (p.Dqk == 64) {
    if (gr.dv) SFA_BWD_F32(64, false);
    else SFA_BWD_F32(64, true);
  } else {
    if (gr.dv) SFA_BWD_F32(128, false);
    else SFA_BWD_F32(128, true);
  }
#undef SFA_BWD_F32
  return hipGetLastError();
}

}  // namespace sfa
