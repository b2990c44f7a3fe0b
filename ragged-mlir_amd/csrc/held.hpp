// Softmax of a whole segment held in a workgroup's registers, for the
// block-per-segment schedule.
//
// Reading a segment twice (statistics, then the rows again) makes two chains
// of rounds, each of a few loads, and two or more exponentials per element. A
// segment of up to kHeldRows vectors (rows) per thread -- 64 KiB where rows take
// 16-byte accesses and their lanes are a power of two, less elsewhere; 32 KiB
// flat -- is read once, every load in flight together; column max and column
// sum are exact passes over the registers, and the output is written from
// them. The registers cost half the waves per SIMD, so the plan takes this
// kernel only where segments fit (holds_segments; bf16 D=64, 4 MiB in segments
// of about 32 rows: 0.65 of the streaming kernel's time, of twice the
// capacity: 1.06).
#pragma once

#include "fused.hpp"

namespace rg {

template <bool FLAT> constexpr int kHeldRows = FLAT ? 8 : 16;      // vectors (rows) per thread

template <class T, int VEC, bool FLAT>
__device__ __forceinline__ bool held_softmax(const Params& p, int64_t start, int64_t end, int tile, float* lds) {
  using In = Words<T, VEC>;
  constexpr int K = kHeldRows<FLAT>;
  const int t = threadIdx.x, d = p.d;
  const RowGeo g = row_geo<VEC>(FLAT ? VEC : d, kBlock, t, tile);
  // Vector i of this thread: FLAT, vector j0 + t + i * kBlock of the array;
  // else the features of row start + row_lane + i * rows_step.
  const int64_t lo = FLAT ? start * d : start, hi = FLAT ? end * d : end;
  const int64_t j0 = FLAT ? lo / VEC : lo, j1 = FLAT ? (hi - 1) / VEC : hi - 1;     // first and last vector / row
  const int step = FLAT ? kBlock : g.rows_step;
  if (hi <= lo || j1 - j0 >= (int64_t)K * step) return false;
  if (FLAT && j1 >= p.n * d / VEC) return false;        // the array's partial last vector
  const int count = (int)(j1 - j0) + 1;
  const int own = FLAT ? t : g.row_lane;
  const T* in = static_cast<const T*>(p.values);
  uint32_t w[K][In::kCount];
  // Vectors past the segment re-read its last one (in cache).
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (i * step >= count) break;
    const int64_t j = own + i * step < count ? j0 + own + i * step : j1;
    const int64_t e = FLAT ? j * VEC : j * d + (g.active ? g.feature : 0);
    if constexpr (In::kBytes == 16) {
      const uint4 q = *reinterpret_cast<const uint4*>(in + e);
      w[i][0] = q.x; w[i][1] = q.y; w[i][2] = q.z; w[i][3] = q.w;
    } else if constexpr (In::kBytes == 8) {
      const uint2 q = *reinterpret_cast<const uint2*>(in + e);
      w[i][0] = q.x; w[i][1] = q.y;
    } else if constexpr (In::kBytes == 4) {
      w[i][0] = *reinterpret_cast<const uint32_t*>(in + e);
    } else {
      w[i][0] = *reinterpret_cast<const uint16_t*>(in + e);
    }
  }
  // Component v of vector i inside the segment.
  auto inside = [&](int i, int v) {
    if (own + i * step >= count) return false;
    if (!FLAT) return g.active;
    const int64_t e = (j0 + own + (int64_t)i * step) * VEC + v;
    return e >= lo && e < hi;
  };
  auto value = [&](int i, int v) {
#pragma clang fp contract(off)
    return In::get(w[i], v) * p.scale;       // (x * 1 is x)
  };
  float m[VEC], sum[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) m[v] = neg_inf();
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (i * step >= count) break;
#pragma unroll
    for (int v = 0; v < VEC; ++v) m[v] = inside(i, v) ? fmax_nan(m[v], value(i, v)) : m[v];
  }
  if constexpr (FLAT) fold_residues<true, VEC>(m, d);      // component c is feature c % D
  block_allreduce<true, VEC>(m, g.lpr, g.feat_lane, lds);
  ExpSum<T> acc[VEC];
  float ref[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) ref[v] = m[v] == neg_inf() ? 0.f : m[v];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (i * step >= count) break;
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      const float e = exp_out<T>(value(i, v) - ref[v]);
      acc[v].add(inside(i, v) ? e : 0.f);
      if constexpr (std::is_same<T, float>::value) w[i][v] = __float_as_uint(e);     // f32 keeps it for the output
    }
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v) sum[v] = acc[v].s;
  if constexpr (FLAT) fold_residues<false, VEC>(sum, d);
  block_allreduce<false, VEC>(sum, g.lpr, g.feat_lane, lds);
  float inv[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) inv[v] = fast_exp(m[v] - m[v]) / sum[v];     // 1 / sum, or NaN for an all -inf column
  T* out = static_cast<T*>(p.out);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (i * step >= count) break;
    if (own + i * step >= count || !g.active) continue;
    const int64_t j = j0 + own + i * step;
    float y[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      y[v] = (std::is_same<T, float>::value ? __uint_as_float(w[i][v]) : exp_out<T>(value(i, v) - ref[v])) * inv[v];
    const int64_t e = FLAT ? j * VEC : j * d + g.feature;
    if (!FLAT || (e >= lo && e + VEC <= hi)) {
      Elem<T>::template store<VEC>(out + e, y);
    } else {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        if (e + v >= lo && e + v < hi) Elem<T>::put(out + e + v, y[v]);
      }
    }
  }
  __syncthreads();       // lds is free for the next segment
  return true;
}

}  // namespace rg
