// One (batch, query, head) row of the forward over a range of its slots, by a
// whole workgroup of 256 threads with scalar float32 arithmetic: the generic
// forward kernel's row, and what the MFMA kernels that replace it fall back
// to for a work item whose result is not a number (a gathered row with
// infinities: 0 * inf in a matrix product is NaN where this loop leaves a
// slot of zero weight out).
#pragma once

#include "sfa_common.h"

namespace sfa {

constexpr int kRowThreads = 256;
constexpr int kRowWaves = kRowThreads / 64;

__device__ __forceinline__ float block_reduce_max(float x, float* red) {
  x = wave_max(x);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = x;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int i = 1; i < kRowWaves; ++i) r = fmaxf(r, red[i]);
  return r;
}

__device__ __forceinline__ float block_reduce_sum(float x, float* red) {
  x = wave_sum(x);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = x;
  __syncthreads();
  float r = 0.f;
#pragma unroll
  for (int i = 0; i < kRowWaves; ++i) r += red[i];
  return r;
}

// smem: q row [Dqk] | per-slot score / probability [nslots] | reduce [kRowWaves].
// put(d, value) receives the normalised output, the return value is the
// row's base-2 log-sum-exp (-inf: no valid slot); with_sink: the sink joins
// the denominator.
template <typename T, class Put>
__device__ __forceinline__ float generic_fwd_row(const Params& p, int b, int t, int h, int slot0, int nslots,
                                                 bool with_sink, float* smem, Put put) {
  float* qs = smem;
  float* sc = smem + p.Dqk;
  float* red = sc + nslots;
  const int g = h / p.G;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  const T* qrow = reinterpret_cast<const T*>(p.q) + b * p.q_sb + t * p.q_ss + h * p.q_sh;
  for (int d = tid; d < p.Dqk; d += kRowThreads) qs[d] = to_f32(qrow[d]);
  __syncthreads();

  const int32_t* irow = p.idx + b * p.i_sb + t * p.i_ss + g * p.i_sh + slot0;
  const int bound = bound_of(p, b);
  // paged KV: k / v are pools and the slot's pool row comes from the block
  // table (-1 for an invalid slot or an unmapped page)
  const bool paged = p.block_table != nullptr;
  const T* kb = reinterpret_cast<const T*>(p.k) + (paged ? 0 : b * p.k_sb) + g * p.k_sh;
  const T* vb = reinterpret_cast<const T*>(p.v) + (paged ? 0 : b * p.v_sb) + g * p.v_sh;
  const int pmask = (1 << p.page_shift) - 1;
  auto key_row = [&](const T* base, int id, int64_t sb, int64_t ss) -> const T* {
    if (paged) {
      const int r = paged_row(p, b, id, bound);
      return r < 0 ? nullptr : base + (int64_t)(r >> p.page_shift) * sb + (int64_t)(r & pmask) * ss;
    }
    return (id >= 0 && id < bound) ? base + (int64_t)id * ss : nullptr;
  };

  for (int j = wave; j < nslots; j += kRowWaves) {
    const T* kr = key_row(kb, irow[j], p.k_sb, p.k_ss);
    float s = kNegInf;
    if (kr != nullptr) {
      float acc = 0.f;
      for (int d = lane; d < p.Dqk; d += 64) acc += qs[d] * to_f32(kr[d]);
      s = wave_sum(acc) * p.scale_log2;
    }
    if (lane == 0) sc[j] = s;
  }
  __syncthreads();

  float m = kNegInf;
  for (int j = tid; j < nslots; j += kRowThreads) m = fmaxf(m, sc[j]);
  m = block_reduce_max(m, red);
  const bool sink = with_sink && p.sink;
  const float sink2 = sink ? p.sink[h] * kLog2e : kNegInf;
  const float mm = fmaxf(m, sink2);

  float l = 0.f;
  for (int j = tid; j < nslots; j += kRowThreads) {
    const float s = sc[j];
    const float e = (s == kNegInf) ? 0.f : exp2f(s - mm);
    sc[j] = e;
    l += e;
  }
  l = block_reduce_sum(l, red);  // contains the barrier that publishes sc[]
  if (sink && mm != kNegInf) l += exp2f(sink2 - mm);
  const float inv = l > 0.f ? 1.f / l : 0.f;

  for (int d = tid; d < p.Dv; d += kRowThreads) {
    float acc = 0.f;
    for (int j = 0; j < nslots; ++j) {
      const float e = sc[j];
      if (e != 0.f) acc += e * to_f32(key_row(vb, irow[j], p.v_sb, p.v_ss)[d]);
    }
    put(d, acc * inv);
  }
  // (a partial, merged later without the sink, hands on a sum that is not a
  // number; a final row has always reported -inf for one)
  return l > 0.f ? mm + log2f(l) : (l != l && !with_sink) ? l : kNegInf;
}

}  // namespace sfa
