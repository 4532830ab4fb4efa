// LayerNorm backward of few rows in one launch: some workgroups take rows and write dx, the others take
// columns and write dgamma / dbeta; neither waits for the other.
//
// The row kernels give every workgroup a partial dgamma / dbeta row, 8 bytes a column, for a second launch
// to fold.  With few rows to a workgroup those rows outweigh the data ([241, 13845] fp16: 14 MB written and
// read back for 13 MB of x and dy), and with very few the second launch is most of the time.  The column
// sums need nothing but x, dy and the saved statistics: here x and dy are read twice instead, the second
// time from a cache that has just seen them, and nothing is left to fold.
//   rows:    a wave or a workgroup of 512 threads per row, VPT vectors per lane, one pass
//   columns: STRIP lanes to a strip of as many vectors, 512 / STRIP rows at a time, eight steps in flight
// Bound by the launch (4.7 us, the two launches 7.6) up to some 100 rows, then by the column workgroups'
// loads, a cache line or half of one a row: fp16 [256, 13845] 11.0 us (22.2) for 42 MB.
// dx may alias neither x nor dy (the column workgroups may read them later).
#pragma once

#include "norm_common.hip.h"

namespace atexn {

constexpr int kPairThreads = 512;
constexpr int kPairBatch = 8;  // a column workgroup's steps in flight

template <typename T, int V, int TPR, int VPT>
__device__ __forceinline__ void pair_rows(const T* dy, const T* x, const float* gamma, const float* mean_in,
                                          const float* rstd_in, T* dx, int64_t n_rows, int d_elems, int block,
                                          float2* buf) {
  const int t = static_cast<int>(threadIdx.x);
  const int64_t row = static_cast<int64_t>(block) * (kPairThreads / TPR) + t / TPR;
  const int lane = t % TPR;
  const bool row_ok = row < n_rows;
  const int64_t at = (row_ok ? row : n_rows - 1) * d_elems;
  Pack<T, V> px[VPT], pd[VPT];
  float g[VPT][V];
  int cnt[VPT];
  const float mean = mean_in[row_ok ? row : n_rows - 1], rstd = rstd_in[row_ok ? row : n_rows - 1];
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int e = (lane + k * TPR) * V;
    const int left = d_elems - e;
    cnt[k] = left <= 0 ? 0 : (left < V ? left : V);
    if (cnt[k] == V) {
      px[k] = load_pack_last<T, V>(x + at + e);
      pd[k] = load_pack_last<T, V>(dy + at + e);
      load_f32<V>(gamma + e, g[k]);
    } else {  // (dy = 0 adds nothing)
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const bool ok = i < cnt[k];
        px[k].v[i] = ok ? x[at + e + i] : T(0);
        pd[k].v[i] = ok ? dy[at + e + i] : T(0);
        g[k][i] = ok ? gamma[e + i] : 0.f;
      }
    }
  }
  float s1 = 0.f, s2 = 0.f;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float w = to_f32(pd[k].v[i]) * g[k][i];
      s1 += w;
      s2 += w * ((to_f32(px[k].v[i]) - mean) * rstd);
    }
  }
  if constexpr (TPR == kWave) {
    s1 = group_sum<kWave>(s1);
    s2 = group_sum<kWave>(s2);
  } else {
    const float2 s = block_sum2(s1, s2, buf, kPairThreads / kWave);
    s1 = s.x;
    s2 = s.y;
  }
  if (!row_ok) return;
  const float inv_d = 1.0f / static_cast<float>(d_elems);
  const float ca = -rstd * (s2 * inv_d), cb = -rstd * (s1 * inv_d);
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    if (cnt[k] == 0) continue;
    Pack<T, V> o;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float xh = (to_f32(px[k].v[i]) - mean) * rstd;
      o.v[i] = from_f32<T>(rstd * (to_f32(pd[k].v[i]) * g[k][i]) + (ca * xh + cb));
    }
    store_pack_n<T, V>(dx + at + (lane + k * TPR) * V, o, cnt[k]);
  }
}

// dgamma / dbeta of vectors block * STRIP .. + STRIP - 1.  The last vector of a ragged row starts at D - V
// and writes its own columns only.  A thread adds up a few rows; the threads' sums are added in double,
// which costs nothing beside the loads and leaves the result a rounding.
template <typename T, int V, int STRIP>
__device__ __forceinline__ void pair_columns(const T* dy, const T* x, const float* mean_in, const float* rstd_in,
                                             int64_t n_rows, int d_elems, float* dgamma, float* dbeta, int block,
                                             float* lds, double* wide) {
  constexpr int AT_ONCE = kPairThreads / STRIP;
  const int t = static_cast<int>(threadIdx.x);
  const int n_vec = (d_elems + V - 1) / V;
  const int vec = block * STRIP + t % STRIP;
  const int nominal = (vec < n_vec ? vec : n_vec - 1) * V;
  const int col = nominal + V <= d_elems ? nominal : d_elems - V;
  float acc[2 * V];
#pragma unroll
  for (int i = 0; i < 2 * V; ++i) acc[i] = 0.f;
  for (int64_t n0 = t / STRIP; n0 < n_rows; n0 += AT_ONCE * kPairBatch) {
    Pack<T, V> px[kPairBatch], pd[kPairBatch];
    float m[kPairBatch], r[kPairBatch];
#pragma unroll
    for (int b = 0; b < kPairBatch; ++b) {
      const int64_t n = n0 + b * AT_ONCE;
      const int64_t at = n < n_rows ? n : n0;
      m[b] = mean_in[at];
      r[b] = rstd_in[at];
      px[b] = load_pack<T, V>(x + at * d_elems + col);
      pd[b] = load_pack<T, V>(dy + at * d_elems + col);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < kPairBatch; ++b) {
      if (n0 + b * AT_ONCE < n_rows) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float d = to_f32(pd[b].v[i]);
          acc[i] += d * ((to_f32(px[b].v[i]) - m[b]) * r[b]);
          acc[V + i] += d;
        }
      }
    }
  }
  constexpr int OUT = STRIP * 2 * V;           // sums of the strip
  constexpr int PARTS = kPairThreads / OUT;    // threads to each
  constexpr int EACH = AT_ONCE / PARTS;
  store_f32<2 * V>(lds + t * 2 * V, acc);
  __syncthreads();
  const int o = t % OUT, part = t / OUT;
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < EACH; ++k) s += static_cast<double>(lds[(part * EACH + k) * OUT + o]);
  wide[t] = s;
  __syncthreads();
  if (t < OUT) {
#pragma unroll
    for (int k = 1; k < PARTS; ++k) s += wide[k * OUT + t];
    const int v = block * STRIP + t / (2 * V);
    const int base = v * V + V <= d_elems ? v * V : d_elems - V;
    const int c = base + t % V;
    if (v < n_vec && c >= v * V) (t % (2 * V) < V ? dgamma : dbeta)[c] = static_cast<float>(s);
  }
}

template <typename T, int V, int TPR, int VPT, int STRIP>
__global__ void __launch_bounds__(kPairThreads, 4)
rows_bwd_pair(const T* __restrict__ dy, const T* __restrict__ x, const float* __restrict__ gamma,
              const float* __restrict__ mean_in, const float* __restrict__ rstd_in, T* __restrict__ dx,
              float* __restrict__ dgamma, float* __restrict__ dbeta, int64_t n_rows, int d_elems, int row_blocks) {
  __shared__ __attribute__((aligned(16))) float lds[kPairThreads * 2 * V];
  __shared__ double wide[kPairThreads];
  __shared__ float2 buf[16];
  const int b = static_cast<int>(blockIdx.x);
  if (b < row_blocks) {
    pair_rows<T, V, TPR, VPT>(dy, x, gamma, mean_in, rstd_in, dx, n_rows, d_elems, b, buf);
  } else {
    pair_columns<T, V, STRIP>(dy, x, mean_in, rstd_in, n_rows, d_elems, dgamma, dbeta, b - row_blocks, lds, wide);
  }
}

}  // namespace atexn
