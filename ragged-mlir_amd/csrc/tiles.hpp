// Sum / max over equal tiles of the input.
//
// The classified schedule spends a launch on binning segments, and its worker
// starts with a chain of dependent round trips (class counts, queue, offsets,
// rows, tickets). Here the input itself is cut, whatever the segments are:
// rows and segment ends are laid on one axis (segment s ends at position
// offsets[s+1] + W s and its end takes W positions, the rows that cost as
// much as finishing a segment), each wave takes one run of V positions, and a
// search of 64 probes per step finds its first and last segment. So every wave
// has the same work for any lengths, needs no queue, ticket or counter, and
// reads one contiguous span.
//
// A segment inside a tile is written at once. A tile that holds the end of a
// segment begun in an earlier tile writes its share as the tile's head
// partial, one that a segment leaves writes a tail partial, and k_tiles_fold
// adds tails and head in row order (deterministic: it depends on N, B and V
// only). Nothing in the workspace outlives the call and nothing is waited
// for: invalid offsets give wrong values, but every loop is bounded by the
// tile and every access by the clamped rows and segments.
//
// Bound by memory: 539 MB f32 D=128 (4,096 segments of up to 512 rows) 107 ->
// 91 us a call against the classified schedule, 5.9 TB/s, what a plain read
// reaches; 1.07 GB bf16 D=128 long tail 235 -> 185 us (5.8 TB/s); 168 MB bf16
// D=84 49 -> 40 us; 102 MB f32 D=2 29 -> 26 us; 100 MB f32 D=5 99 -> 49 us.
// 128 KB: 12.7 -> 8.5 us of kernels, latency (launches, search, one batch).
#pragma once

#include "fused.hpp"

namespace rg {

constexpr int kTileStage = 4096;      // bytes a wave stages in LDS per batch of rows
constexpr int kTileLoads = kTileStage / (kWave * 16);
// Cache policy of the tile loads: non-temporal, as the rows are read once
// (539 MB f32 D=128: 103 -> 90 us; 1.07 GB bf16 D=128: 205 -> 183 us).
constexpr int kTileAux = kStreamAux;
constexpr int kTileThreads = 1024;    // largest workgroup of k_tiles
constexpr int kFoldFlight = 8;        // k_tiles_fold: partials in flight per lane
constexpr int kFoldParts = 32;        // k_tiles_fold: longest chain one lane per feature folds
constexpr int kFoldWave = 64;         // k_tiles_fold: parts per lane up to which a wave folds a chain
constexpr int kFoldFeatures = 16;     // k_tiles_fold: features per workgroup
constexpr int kFoldLong = kTileThreads / kFoldParts;      // longer chains one workgroup's tiles can end
constexpr int kTileFoldBytes = 4 * (kTileThreads + kFoldLong + 1);   // LDS of a fold: a float per thread, the list
constexpr int kGroupSteps = 32;       // rows per lane up to which segments of a batch are reduced side by side

// Lanes per tile in k_tiles_fold: a power of two, at most kFoldFeatures.
__host__ __device__ inline int tile_fold_lanes(int d) {
  int lanes = 1;
  while (lanes < d && lanes < kFoldFeatures) lanes <<= 1;
  return lanes;
}

__device__ __forceinline__ void tile_load(Rsrc r, int voffset, uint32_t (&w)[4]) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voffset, 0, kTileAux);
  w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
}

// First segments s0, s1 of [0, B] whose end position offsets[s+1] + W s is at
// least v0, v1 (B: none): 64 probes per step, both searches at once.
template <class OffT>
__device__ __forceinline__ void tile_search(const Params& p, int lane, int64_t v0, int64_t v1, int64_t& s0,
                                            int64_t& s1) {
  const int64_t w = p.marker_rows;
  int64_t lo0 = 0, hi0 = p.b, lo1 = 0, hi1 = p.b;
  while (lo0 < hi0 || lo1 < hi1) {
    const int64_t step0 = (hi0 - lo0 + kWave - 1) / kWave, step1 = (hi1 - lo1 + kWave - 1) / kWave;
    const int64_t i0 = lo0 + lane * step0, i1 = lo1 + lane * step1;
    bool at0 = i0 >= hi0, at1 = i1 >= hi1;      // past the range: taken as found
    if (!at0) at0 = offset_at<OffT>(p, i0 + 1) + w * i0 >= v0;
    if (!at1) at1 = offset_at<OffT>(p, i1 + 1) + w * i1 >= v1;
    const uint64_t m0 = __ballot(at0), m1 = __ballot(at1);
    auto narrow = [](int64_t& lo, int64_t& hi, int64_t step, uint64_t m) {
      if (lo >= hi) return;
      const int first = m ? __ffsll((unsigned long long)m) - 1 : kWave;
      const int64_t top = lo + first * step;     // the first probe found
      const int64_t below = first ? lo + (first - 1) * step + 1 : lo;
      hi = top < hi ? top : hi;
      lo = below < hi ? below : hi;
    };
    narrow(lo0, hi0, step0, m0);
    narrow(lo1, hi1, step1, m1);
  }
  s0 = lo0;
  s1 = lo1;
}

// Butterfly over the lane masks from `lo` up to, and not including, `hi`.
template <class Step>
__device__ __forceinline__ void xor_butterfly_range(int lo, int hi, Step&& step) {
  if (lo <= 1 && hi > 1) step(std::integral_constant<int, 1>{});
  if (lo <= 2 && hi > 2) step(std::integral_constant<int, 2>{});
  if (lo <= 4 && hi > 4) step(std::integral_constant<int, 4>{});
  if (lo <= 8 && hi > 8) step(std::integral_constant<int, 8>{});
  if (lo <= 16 && hi > 16) step(std::integral_constant<int, 16>{});
  if (lo <= 32 && hi > 32) step(std::integral_constant<int, 32>{});
}

// The chain of partials of tile w's head: out[s] = tail[first .. w-1], head[w]
// in order, features f0 .. of `lanes` lanes per tile. Called by whole
// workgroups of `threads` threads (it contains barriers).
template <int OP, class T>
__device__ __forceinline__ void fold_tiles(const Params& p, int64_t tile0, int lanes, int64_t f0, int threads,
                                           float* lds, int* list) {
  const int t = threadIdx.x;
  const int fl = t & (lanes - 1);
  const int64_t w = tile0 + t / lanes, f = f0 + fl;
  const int64_t d = p.d;
  const float* part = p.partials;      // [tiles][2][D]: head, tail
  T* out = static_cast<T*>(p.out);
  auto add = [](State<OP>& acc, float x) {
    if constexpr (OP == OP_SUM) {
      acc.fold(x);
    } else {
      State<OP> o;
      o.m = x;
      acc.merge(o);
    }
  };
  // Chain of tile w: parts first .. w - 1 (tails), then its head; first is the
  // tile that holds the segment's first row.
  auto first_of = [&](int64_t tile) {
    const int64_t q = p.part_begin[tile] / p.tile_items;
    return q < tile ? q : tile;
  };
  // Tails [q, stop) into acc, in order, kFoldFlight loads in flight.
  auto add_tails = [&](State<OP>& acc, int64_t q, int64_t stop) {
    for (; q < stop; q += kFoldFlight) {
      float x[kFoldFlight];
#pragma unroll
      for (int u = 0; u < kFoldFlight; ++u) x[u] = part[((q + u < stop ? q + u : q) * 2 + 1) * d + f];
#pragma unroll
      for (int u = 0; u < kFoldFlight; ++u) {
        if (q + u < stop) add(acc, x[u]);
      }
    }
  };
  if (t == 0) *list = 0;
  __syncthreads();
  const int64_t s = w < p.tile_count ? p.item_pos[w] : -1;
  if (s >= 0) {
    const int64_t first = first_of(w);
    if (w - first > kFoldParts) {
      if (fl == 0) {
        const int k = atomicAdd(list, 1);
        if (k < kFoldLong) list[1 + k] = (int)(w - tile0);
      }
    } else if (f < d) {
      const float head = part[w * 2 * d + f];
      State<OP> acc;
      acc.init();
      add_tails(acc, first, w);
      add(acc, head);
      Elem<T>::put(out + s * d + f, exact_value<OP>(acc));
    }
  }
  __syncthreads();
  // Longer chains: a wave each, its lanes on contiguous runs of parts; those
  // too long for a wave the whole workgroup.
  const int many = *list < kFoldLong ? *list : kFoldLong;
  const int in_wave = kWave / lanes;
  auto shared = [&](State<OP>& acc, int k, int pl, int pl_count) {
    const int64_t w2 = tile0 + list[1 + k], first2 = first_of(w2), count = w2 - first2;
    acc.init();
    if (f < d) add_tails(acc, first2 + count * pl / pl_count, first2 + count * (pl + 1) / pl_count);
  };
  auto parts_of = [&](int k) { return tile0 + list[1 + k] - first_of(tile0 + list[1 + k]); };
  auto finish = [&](State<OP>& acc, int k) {
    const int64_t w2 = tile0 + list[1 + k];
    add(acc, part[w2 * 2 * d + f]);
    Elem<T>::put(out + p.item_pos[w2] * d + f, exact_value<OP>(acc));
  };
  for (int k = t / kWave; k < many; k += threads / kWave) {
    if (parts_of(k) > kFoldWave * in_wave) continue;
    State<OP> acc;
    shared(acc, k, (t & (kWave - 1)) / lanes, in_wave);
    State<OP> one[1] = {acc};
    merge_lanes<OP, 1, true>(one, [&](auto&& step) { xor_butterfly_range(lanes, kWave, step); });
    acc = one[0];
    if ((t & (kWave - 1)) < lanes && f < d) finish(acc, k);
  }
  for (int k = 0; k < many; ++k) {
    if (parts_of(k) <= kFoldWave * in_wave) continue;
    State<OP> acc;
    shared(acc, k, t / lanes, threads / lanes);
    __syncthreads();
    lds[t] = exact_value<OP>(acc);
    __syncthreads();
    if (t < lanes && f < d) {
      acc.init();
      for (int q = 0; q < threads / lanes; ++q) add(acc, lds[q * lanes + fl]);
      finish(acc, k);
    }
  }
  __syncthreads();      // before the list is used again
}

// A call's partials overlap what a register-resident softmax plan keeps at
// zero in a shared workspace: record its state as unknown.
__device__ __forceinline__ void mark_arena_unknown(const Params& p) {
  if (p.counters && threadIdx.x == 0) p.counters[kCleanSlot] = 1;
}

template <int OP, class T>
__global__ __launch_bounds__(kBlock) void k_tiles_fold(Params p) {
  __shared__ float lds[kBlock];
  __shared__ int list[1 + kFoldLong];
  const int lanes = tile_fold_lanes(p.d);
  if (blockIdx.x == 0 && blockIdx.y == 0) mark_arena_unknown(p);
  fold_tiles<OP, T>(p, (int64_t)blockIdx.x * (kBlock / lanes), lanes, (int64_t)blockIdx.y * lanes, kBlock, lds, list);
}

// One wave per tile. Rows are D elements of VEC-element lanes (at most a
// wave's): lane (row lane, feature lane) as in row_geo; D below 16 bytes has
// one lane per row. The tile's bytes come in batches of whole rows, read as
// 16-byte vectors whatever D is, straight into the wave's LDS.
template <int OP, class T, class OffT, int VEC>
__global__ __launch_bounds__(kTileThreads) void k_tiles(Params p) {
  constexpr int K = VEC * (int)sizeof(T) == 16 ? 4 : 8;      // rows in flight per lane
  extern __shared__ __align__(16) unsigned char tile_lds[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t w = (int64_t)blockIdx.x * (blockDim.x / kWave) + wave;
  const int d = p.d;
  if (w < p.tile_count) {
    const int64_t v0 = w * p.tile_items;
    const int64_t axis = p.n + p.marker_rows * p.b;
    const int64_t v1 = v0 + p.tile_items < axis ? v0 + p.tile_items : axis;
    int64_t s0, s1;
    tile_search<OffT>(p, lane, v0, v1, s0, s1);
    // Rows of the tile: the position without the ends before it, kept
    // inside the segment's rows (a position within an end, or offsets that
    // break the contract) and inside the array.
    auto row_at = [&](int64_t v, int64_t s) {
      const int64_t a = offset_at<OffT>(p, s), e = s < p.b ? offset_at<OffT>(p, s + 1) : p.n;
      int64_t r = v - p.marker_rows * s;
      r = r > e ? e : r;
      r = r < a ? a : r;
      return r < 0 ? 0 : (r > p.n ? p.n : r);
    };
    const int64_t r0 = row_at(v0, s0);
    int64_t r1 = row_at(v1, s1);
    r1 = r1 < r0 ? r0 : (r1 > r0 + p.tile_items ? r0 + p.tile_items : r1);
    int64_t begin0 = s0 < p.b ? offset_at<OffT>(p, s0) : r0;
    begin0 = begin0 < 0 ? 0 : begin0;
    const bool head_open = w > 0 && begin0 < r0;
    const RowGeo g = row_geo<VEC>(d, kWave, lane, 0);
    const int lpr = g.lpr, row_lanes = g.rows_step;
    const int row_bytes = d * (int)sizeof(T);
    const int to = (int)(r1 - r0);                 // rows of the tile
    const int batch = p.tile_batch;                // rows staged at once
    // The 16-byte granules that hold the tile's bytes.
    const uintptr_t first_byte = (uintptr_t)p.values + (uintptr_t)(r0 * row_bytes);
    const int shift = (int)(first_byte & 15);
    const Rsrc in = make_rsrc((const void*)(first_byte - shift), ((int64_t)to * row_bytes + shift + 15) & ~15ll);
    unsigned char* stage = tile_lds + wave * kTileStage;

    // Ends of 64 segments at a time, as rows of the tile (past it: to + 1).
    int64_t window = s0;
    int ends = 0;
    auto load_window = [&](int64_t first) {
      window = first;
      const int64_t i = first + lane + 1;
      int64_t e = offset_at<OffT>(p, i < p.b ? i : p.b);
      e = e < r0 ? r0 : (e > r1 ? r1 + 1 : e);
      ends = (int)(e - r0);
    };
    load_window(s0);
    int64_t s = s0;
    State<OP> st[VEC];
    init_all<OP, VEC>(st);
    int pos = 0;
    bool open = head_open, head_done = false;
    T* out = static_cast<T*>(p.out);

    // The states of `lanes` row lanes into one.
    auto reduce = [&](int lanes) {
      if (lanes > 1) merge_lanes<OP, VEC, true>(st, [&](auto&& step) { xor_butterfly_range(lpr, lpr * lanes, step); });
    };
    auto put_partial = [&](int which) {
      if (!p.partials) return;      // a single tile has none (valid offsets)
      float* dst = p.partials + (w * 2 + which) * d + g.feature;
      if (g.row_lane == 0 && g.active) {
#pragma unroll
        for (int v = 0; v < VEC; ++v) dst[v] = exact_value<OP>(st[v]);
      }
    };

    // Batch of rows from x0: its first granule, and the bytes it reads there.
    auto granule_of = [&](int x) { return (shift + x * row_bytes) & ~15; };
    // The next batch loads into registers while this one is reduced from LDS.
    uint32_t next[kTileLoads][4];
    auto load = [&](int x) {
      const int granule = granule_of(x);
      const int last = x + batch < to ? x + batch : to;
      const int bytes = shift + last * row_bytes - granule;
#pragma unroll
      for (int u = 0; u < kTileLoads; ++u) {
        const int at = u * kWave * 16 + lane * 16;
        tile_load(in, at < bytes ? granule + at : kOutOfRange, next[u]);
      }
    };
    load(0);
    int x0 = 0;
    do {
      const int limit = x0 + batch < to ? x0 + batch : to;
      const unsigned char* rows = stage + (shift + x0 * row_bytes - granule_of(x0));      // row x0
      // (One wave: its LDS operations complete in order.)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < kTileLoads; ++u)
        *reinterpret_cast<uint4*>(stage + (u * kWave + lane) * 16) = make_uint4(next[u][0], next[u][1], next[u][2], next[u][3]);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      load(x0 + batch);
      for (;;) {
        if (s - window >= kWave) load_window(s);
        const int k0 = (int)(s - window);
        int e = s < s1 ? __builtin_amdgcn_readlane(ends, k0) : to + 1;
        const bool fin = e <= limit;
        e = fin ? e : limit;
        int m = 1, lanes = row_lanes, i = 0, a_i = pos, e_i = e;
        if (fin && !open && row_lanes > 1) {
          // Whole segments inside the batch, side by side: a group of
          // `lanes` row lanes each, while none takes over kGroupSteps rows
          // per lane.
          const int64_t left = s1 - window;
          m = (int)__popcll(__ballot(lane >= k0 && lane < left && ends <= limit));
          m = m < row_lanes ? m : row_lanes;
          if (m > 1) {
            while (lanes > 1 && lanes * m > row_lanes) lanes >>= 1;
            i = g.row_lane >> (31 - __builtin_clz(lanes));
            const int at = k0 + (i < m ? i : 0);
            // (Clamped: offsets that break the contract stay inside the batch.)
            e_i = __shfl(ends, at, kWave);
            a_i = __shfl(ends, at > 0 ? at - 1 : 0, kWave);
            a_i = i == 0 || a_i < pos ? pos : (a_i > limit ? limit : a_i);
            e_i = e_i < a_i ? a_i : (e_i > limit ? limit : e_i);
            const uint64_t wide = __ballot(i < m && e_i - a_i > kGroupSteps * lanes);
            if (wide) m = (__ffsll((unsigned long long)wide) - 1) >> (31 - __builtin_clz(lpr * lanes));
            if (m < 2) {
              m = 1;
              lanes = row_lanes;
              i = 0;
              a_i = pos;
              e_i = e;
            }
          }
        }
        if (i < m && g.active) {
          const int k = g.row_lane & (lanes - 1);
          int r = a_i + k;
          const T* at = reinterpret_cast<const T*>(rows) + g.feature;
          for (; r + (K - 1) * lanes < e_i; r += K * lanes) {
            float x[K][VEC];
#pragma unroll
            for (int u = 0; u < K; ++u) Elem<T>::template load<VEC>(at + (r - x0 + u * lanes) * d, x[u]);
            bool folded = false;
            if constexpr (OP == OP_SUM && sizeof(T) == 2) {
              // bf16 has twice the additions per byte: K rows are added
              // without the check for an infinite sum after each, and once
              // more with it where the result is not finite (the same bits).
              State<OP> acc[VEC];
              folded = true;
#pragma unroll
              for (int v = 0; v < VEC; ++v) {
                acc[v] = st[v];
#pragma unroll
                for (int u = 0; u < K; ++u) acc[v].fold_finite(x[u][v]);
                folded = folded && __builtin_fabsf(acc[v].s) < pos_inf();
              }
              if (folded) {
#pragma unroll
                for (int v = 0; v < VEC; ++v) st[v] = acc[v];
              }
            }
            if (!folded) {
#pragma unroll
              for (int u = 0; u < K; ++u) {
#pragma unroll
                for (int v = 0; v < VEC; ++v) st[v].fold(x[u][v]);
              }
            }
          }
          for (; r < e_i; r += lanes) {
            float x[VEC];
            Elem<T>::template load<VEC>(at + (r - x0) * d, x);
#pragma unroll
            for (int v = 0; v < VEC; ++v) st[v].fold(x[v]);
          }
        }
        bool tail = false;
        if (!fin) {
          open = open || pos < limit;
          pos = limit;
          tail = limit == to && open && s1 < p.b;     // the segment goes on in the next tile
          if (!tail) break;
        } else {
          const int last = __builtin_amdgcn_readlane(ends, k0 + m - 1);
          pos = last > pos ? (last < limit ? last : limit) : pos;
        }
        // Segments s .. s + m - 1 end: their results, or the tile's partials.
        reduce(lanes);
        if (tail || (s == s0 && head_open)) {
          put_partial(tail ? 1 : 0);
          head_done = head_done || !tail;
          if (tail) break;
        } else if (i < m && (g.row_lane & (lanes - 1)) == 0 && g.active) {
          float x[VEC];
#pragma unroll
          for (int v = 0; v < VEC; ++v) x[v] = exact_value<OP>(st[v]);
          Elem<T>::template store<VEC>(out + (s + i) * d + g.feature, x);
        }
        init_all<OP, VEC>(st);
        open = false;
        s += m;
      }
      x0 += batch;
    } while (x0 < to);
    if (lane == 0 && p.item_pos) {
      // The head's segment, and the position of its first row.
      p.item_pos[w] = head_done ? s0 : -1;
      p.part_begin[w] = begin0 + p.marker_rows * s0;
    }
  }
  if (p.tile_single) {
    // One workgroup holds every tile: it folds the chains itself, in the
    // staging memory, which no wave uses any more. (Doing this for more
    // workgroups, the last one out folding, took 11.4 us where the two
    // launches take 7.8 and 8.8: the release, the count and the fold follow
    // one another.)
    __threadfence_block();
    __syncthreads();
    float* lds = reinterpret_cast<float*>(tile_lds);
    int* list = reinterpret_cast<int*>(tile_lds) + kTileThreads;
    mark_arena_unknown(p);
    const int lanes = tile_fold_lanes(d);
    for (int64_t f0 = 0; f0 < d; f0 += lanes) {
      for (int64_t t0 = 0; t0 < p.tile_count; t0 += blockDim.x / lanes)
        fold_tiles<OP, T>(p, t0, lanes, f0, blockDim.x, lds, list);
    }
  }
}

}  // namespace rg
