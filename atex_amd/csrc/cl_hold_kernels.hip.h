// Channels-last InstanceNorm of instances larger than the flat kernels hold (cl_flat_kernels.hip.h), on the
// same layout and exchange: 512 threads of 256 registers per CU, in one workgroup or two, keep what registers
// and LDS take of their slabs (forward 60 vectors per thread, 480 KB per CU and 126 MB of the chip's; backward
// 30 of x and of dy), and only the rest is read a second time.
//
// Bound by memory: against two stages, which read everything twice, [2, 128*128*128, 32] fp16 forward 118 us
// (130) and backward 190 (217), [8, 524288, 32] 107 (137) and 173 (221), [3, 703459, 23] 42 (52) and 72 (163); a read
// of 134 MB and its write alone take 48 us, held ones 56: reads and writes of one instance do not overlap, and
// the exchange between them costs 8 us, 5 of them after the last slab's sums.
//
// A thread's U vectors are, in the order in which they are summed up: the HA first, held in registers; passes
// of Q through Q more registers, of which the first one goes on to LDS where the kernel has a place for it and
// the others (R vectors) are read again; and the last Q, or some fewer, that stay in those registers.  A pass
// goes by batches: a batch is summed up and its registers asked for the next pass's, so that loads are in
// flight behind all arithmetic.  After the exchange the passes go the other way, and what was read last is
// read again first, while the caches behind the L2s still have some of it.
#pragma once

#include <type_traits>

#include "cl_flat_kernels.hip.h"

namespace atexn {

struct HoldArgs {
  int U, R;     // vectors per thread: all, read twice (a multiple of Q)
  int hold_at;  // where in LDS (floats, a multiple of 4) the held vectors are
};

// Mean and squared deviations of a thread's V streams over the vectors from, ..., B - 1 of a batch (the last
// one nv elements), an exact two-pass over the batch, merged into those of the n vectors before it (Chan).
template <typename T, int V, int B, int UNROLL, typename Vector>
__device__ __forceinline__ void hold_stats(int from, int nv, Vector&& vector, float& n, float (&m)[V], float (&q)[V]) {
#pragma clang fp contract(off)
  const float one = mix_one();
  float bm[V], bq[V];
#pragma unroll
  for (int i = 0; i < V; ++i) bm[i] = bq[i] = 0.f;
#pragma unroll UNROLL
  for (int u = 0; u < B; ++u) {
    if (u >= from) {
      const Pack<T, V> x = vector(u);
#pragma unroll
      for (int i = 0; i < V; ++i) bm[i] = add_f32<T>(bm[i], x.v[i], one);
    }
  }
  const float k = static_cast<float>(B - from);
  const float whole = 1.0f / k, less = k > 1.0f ? 1.0f / (k - 1.0f) : 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) bm[i] *= i < nv ? whole : less;
#pragma unroll UNROLL
  for (int u = 0; u < B; ++u) {
    if (u >= from) {
      const Pack<T, V> x = vector(u);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        float d = sub_f32<T>(x.v[i], bm[i], one);
        if (u == B - 1) d = i < nv ? d : 0.f;
        bq[i] = __builtin_fmaf(d, d, bq[i]);
      }
    }
  }
  const float fw = k / (n + k), fl = n + k > 1.0f ? (k - 1.0f) / (n + k - 1.0f) : 0.f;
  const float gw = n * fw, gl = n * fl;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const float d = bm[i] - m[i];
    m[i] = __builtin_fmaf(d, i < nv ? fw : fl, m[i]);
    q[i] += __builtin_fmaf(d * (i < nv ? gw : gl), d, bq[i]);
  }
  n += k;
}

// The sums so far are computed here, not where they are needed at last: vectors whose slots have been given
// away would have to be kept until then.
template <int V>
__device__ __forceinline__ void hold_now(float (&v)[V]) {
#pragma unroll
  for (int i = 0; i < V; ++i) asm volatile("" : "+v"(v[i]));
}

// The thread's index, anew at each use: an address in LDS made from it is not kept until it is needed again.
__device__ __forceinline__ unsigned hold_thread() {
  unsigned t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// A thread's way through its slab, in bytes from its start (a slab has less than 4 GiB: one register per
// address, a 64-bit base in scalars and a 32-bit offset).  No load is behind a branch (the compiler would make
// the next use of any vector wait for more than that vector): what the last pass has too much of, skip
// vectors, it reads again from before it.
template <typename T, int V, int HA, int Q, bool LDS, int B>
struct HoldLane {
  static constexpr int NB = Q / B;
  unsigned lane, step, end;  // end: where the slab's last whole vector starts
  int U, P;                  // vectors; passes before the last
  int skip, nv;              // of the last pass's vectors: not to be counted; elements of the very last one

  __device__ __forceinline__ HoldLane(const FlatArgs& a, const HoldArgs& h, int n_el) {
    U = h.U;
    P = h.R / Q + (LDS ? 1 : 0);
    step = static_cast<unsigned>(a.A) * 16u;
    lane = (static_cast<int>(threadIdx.x) < a.A ? threadIdx.x : 0u) * 16u;  // (a lane without data adds to nothing)
    end = static_cast<unsigned>(n_el) * sizeof(T) - 16u;
    skip = HA + (P + 1) * Q - U;
    const int left = n_el - static_cast<int>(((U - 1) * step + lane) / sizeof(T));
    nv = left <= 0 ? 0 : (left < V ? left : V);
  }
  // (Opaque to the compiler, which would otherwise keep the loads' addresses for the stores.)
  __device__ __forceinline__ unsigned from(int u) const {
    unsigned o = lane;
    asm volatile("" : "+v"(o));
    return o + static_cast<unsigned>(u) * step;
  }
  __device__ __forceinline__ unsigned at(int p, int b) const { return from((p < P ? HA + p * Q : U - Q) + b * B); }
  static __device__ __forceinline__ T* there(T* base, unsigned o) { return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + o); }
  static __device__ __forceinline__ const T* there(const T* base, unsigned o) {
    return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + o);
  }
  // the registers' own
  __device__ __forceinline__ void load(u32x4 (&own)[HA], const T* src) const {
    unsigned o = lane;
#pragma unroll
    for (int u = 0; u < HA; ++u) {
      own[u] = flat_bits(load_pack<T, V>(there(src, o)));
      flat_advance(o, step);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // batch b of pass p
  template <bool LAST>
  __device__ __forceinline__ void load(u32x4 (&ring)[Q], int p, int b, const T* src) const {
    load_from<LAST>(ring, p < P ? HA + p * Q : U - Q, b, src);
  }
  // batch b of the Q vectors from the u-th on
  template <bool LAST>
  __device__ __forceinline__ void load_from(u32x4 (&ring)[Q], int u, int b, const T* src) const {
    unsigned o = from(u + b * B);
#pragma unroll
    for (int i = 0; i < B; ++i) {
      if (b == NB - 1 && i == B - 1) o = o < end ? o : end;
      ring[b * B + i] = flat_bits(LAST ? load_pack_last<T, V>(there(src, o)) : load_pack<T, V>(there(src, o)));
      flat_advance(o, step);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // The last vector, taken from the slab's end, as the elements that it has, then zeros.
  __device__ __forceinline__ void settle(u32x4& v) const {
    const unsigned bits = static_cast<unsigned>(V - nv) * (8u * sizeof(T));
    uint64_t lo = v[0] | (uint64_t(v[1]) << 32), hi = v[2] | (uint64_t(v[3]) << 32);
    if (bits >= 64) {
      lo = hi;
      hi = 0;
    }
    const unsigned by = bits & 63;
    lo = (lo >> by) | ((hi << 1) << (63 - by));
    hi >>= by;
    if (bits >= 128) lo = hi = 0;
    v = u32x4{static_cast<unsigned>(lo), static_cast<unsigned>(lo >> 32), static_cast<unsigned>(hi), static_cast<unsigned>(hi >> 32)};
  }
  template <typename Value>
  __device__ __forceinline__ void store(int p, int b, T* dst, Value&& value) const {
    unsigned o = at(p, b);
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const int r = b * B + i;
      if (r == Q - 1) {
        const int cnt = p < P ? V : nv;
        if (cnt > 0) store_pack_n<T, V>(there(dst, o), value(r), cnt);
      } else if (p < P || r >= skip) {
        store_pack<T, V>(there(dst, o), value(r));
      }
      flat_advance(o, step);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // All U vectors in passes of Q, in order, through the registers of one: batch(u, b) has the b-th batch from
  // the u-th vector on, last(b) that of the last pass.  ring(f): f(registers, where they come from) for all arrays.
  template <bool LAST, typename Ring, typename Batch, typename Last>
  __device__ __forceinline__ void through(Ring&& ring, Batch&& batch, Last&& last) const {
    auto load = [&](int u, int b) { ring([&](u32x4 (&r)[Q], const T* src) { load_from<LAST>(r, u, b, src); }); };
    const int main = HA + P * Q;  // vectors before the last pass
#pragma unroll
    for (int b = 0; b < NB; ++b) load(0, b);
#pragma unroll 1
    for (int u = 0; u < main; u += Q) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        batch(u, b);
        load(u + Q < main ? u + Q : U - Q, b);
      }
    }
    ring([&](u32x4 (&r)[Q], const T*) { settle(r[Q - 1]); });
#pragma unroll
    for (int b = 0; b < NB; ++b) last(b);
  }
  // N vectors from the u-th on
  template <int N, typename Value>
  __device__ __forceinline__ void store_own(int u, T* dst, Value&& value) const {
    unsigned o = from(u);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      store_pack<T, V>(there(dst, o), value(i));
      flat_advance(o, step);
      if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
};

// ------------------------------------------------------------------------------ forward
// One batch after another.
template <typename T, int V, int B>
__device__ __forceinline__ void hold_stats_now(const u32x4* batch, int skip, int nv, float& n, float (&m)[V], float (&q)[V]) {
  hold_stats<T, V, B, B>(skip, nv, [&](int u) { return flat_pack<T, V>(batch[u]); }, n, m, q);
  hold_now(m);
  hold_now(q);
}

template <typename T, int V, int HA, int Q, bool LDS, int B>
struct HoldFwdOp : FlatFwdOp<T, V> {
  HoldArgs h;
  using Lane = HoldLane<T, V, HA, Q, LDS, B>;
  // in the kernel's order, in passes through one pass's registers
  __device__ __forceinline__ void sums(int64_t n, int l) const {
    const FlatArgs& a = this->a;
    const FlatSlab f = flat_slab<V>(a, l);
    const T* const src = this->x + n * a.E + f.e0;
    const Lane w(a, h, f.n_el);
    u32x4 r[Q];
    float m[V], q[V], cnt = 0.f;
#pragma unroll
    for (int i = 0; i < V; ++i) m[i] = q[i] = 0.f;
    w.template through<false>([&](auto&& f) { f(r, src); },
                              [&](int, int b) { hold_stats_now<T, V, B>(r + b * B, 0, V, cnt, m, q); },
                              [&](int b) {
                                const int skip = w.skip - b * B;
                                if (skip < B) hold_stats_now<T, V, B>(r + b * B, skip > 0 ? skip : 0, b == Lane::NB - 1 ? w.nv : V, cnt, m, q);
                              });
    flat_merge_stats<V>(a, f, flat_pixels(a, l), h.U, m, q, this->nt, this->lds,
                        [&](int c, float cm, float cq) { this->publish(n, l, c, cm, cq); });
  }
  __device__ __forceinline__ void apply(int64_t n, int l) const {
    const FlatArgs& a = this->a;
    const FlatSlab f = flat_slab<V>(a, l);
    const T* const src = this->x + n * a.E + f.e0;
    T* const dst = this->y + n * a.E + f.e0;
    const Lane w(a, h, f.n_el);
    const typename FlatFwdOp<T, V>::Coef coef = this->coef();
    if (static_cast<int>(threadIdx.x) >= a.A) return;
    u32x4 r[Q];
    auto value = [&](int i) { return coef(flat_pinned<T, V>(flat_pack<T, V>(r[i]))); };
    w.template through<true>([&](auto&& f) { f(r, src); },
                             [&](int u, int b) { w.template store_own<B>(u + b * B, dst, [&](int i) { return value(b * B + i); }); },
                             [&](int b) { w.store(w.P, b, dst, value); });
  }
};

template <typename Op>
__device__ __attribute__((noinline)) void hold_fwd_alone(const Op* op, FlatShared* sm, int64_t n, int s) {
  flat_alone<true>(op->a, *op, *sm, op->nt, op->tag, n, s);
}

template <typename T, int V, int HA, int Q, bool LDS, int B>
__global__ void __launch_bounds__(kFlatMaxThreads, 2)
cl_hold_fwd(const T* __restrict__ x, const float* __restrict__ gamma, const float* __restrict__ beta,
            T* __restrict__ y, float* __restrict__ mean_out, float* __restrict__ rstd_out, FlatArgs a, float eps,
            HoldArgs h) {
  static_assert(HA % B == 0 && Q % B == 0, "whole batches");
  constexpr int NB = Q / B;
  extern __shared__ __attribute__((aligned(16))) float flat_lds[];
  __shared__ FlatShared sm;
  const int nt = block_threads();
  const unsigned tag = a.ex.the_tag();
  const FlatFwdOp<T, V> op{a, x, gamma, beta, y, mean_out, rstd_out, eps, nt, h.U, tag, flat_lds};
  int64_t n;
  int s;
  if (!flat_place(a, n, s)) return;
  const typename FlatFwdOp<T, V>::Params params = op.fetch(n);
  const FlatSlab f = flat_slab<V>(a, s);
  const T* const src = x + n * a.E + f.e0;
  u32x4* const held = reinterpret_cast<u32x4*>(flat_lds + h.hold_at) + hold_thread();
  const HoldLane<T, V, HA, Q, LDS, B> w(a, h, f.n_el);

  u32x4 own[HA], ring[Q];
  w.load(own, src);
#pragma unroll
  for (int b = 0; b < NB; ++b) w.template load<false>(ring, 0, b, src);
  op.template keep<false>(n, params);
  float m[V], q[V], cnt = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) m[i] = q[i] = 0.f;
  auto stats = [&](const u32x4* batch, int skip, int nv) { hold_stats_now<T, V, B>(batch, skip, nv, cnt, m, q); };
#pragma unroll
  for (int u = 0; u < HA; u += B) stats(own + u, 0, V);
  if constexpr (LDS) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      stats(ring + b * B, 0, V);
#pragma unroll
      for (int i = 0; i < B; ++i) held[(b * B + i) * nt] = ring[b * B + i];
      w.template load<false>(ring, 1, b, src);
    }
#pragma unroll 1
    for (int p = 1; p < w.P; ++p) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        stats(ring + b * B, 0, V);
        w.template load<false>(ring, p + 1, b, src);
      }
    }
  }
  w.settle(ring[Q - 1]);
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int skip = w.skip - b * B;
    if (skip < B) stats(ring + b * B, skip > 0 ? skip : 0, b == NB - 1 ? w.nv : V);
  }
  flat_merge_stats<V>(a, f, flat_pixels(a, s), h.U, m, q, nt, flat_lds, [&](int c, float cm, float cq) { op.publish(n, s, c, cm, cq); });
  flat_exchange<true>(a, op, sm, nt, tag, n, s);
  if (flat_uniform(sm.fail) == 0) {
    flat_forget(own);
    flat_forget(ring);
    const typename FlatFwdOp<T, V>::Coef coef = op.coef();
    T* const dst = y + n * a.E + f.e0;
    auto value = [&](const u32x4& v) { return coef(flat_pinned<T, V>(flat_pack<T, V>(v))); };
    auto ringed = [&](int r) { return value(ring[r]); };
    if (static_cast<int>(threadIdx.x) < a.A) {
      if constexpr (LDS) {
#pragma unroll 1
        for (int p = w.P; p > 1; --p) {
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            w.store(p, b, dst, ringed);
            w.template load<true>(ring, p - 1, b, src);
          }
        }
      }
      w.template store_own<HA>(0, dst, [&](int u) { return value(own[u]); });
#pragma unroll
      for (int b = 0; b < NB; ++b) w.store(LDS ? 1 : 0, b, dst, ringed);
      if constexpr (LDS) {
        const u32x4* const again = reinterpret_cast<const u32x4*>(flat_lds + h.hold_at) + hold_thread();
        w.template store_own<Q>(HA, dst, [&](int u) { return value(again[u * nt]); });
      }
    }
  }
  asm volatile("" ::: "memory");  // (asked for again, so that nothing of the slab lives across the call)
  if (flat_uniform(sm.fail) != 0) {
    const FlatArgs args = a;
    const HoldFwdOp<T, V, HA, Q, LDS, B> copy{{args, x, gamma, beta, y, mean_out, rstd_out, eps, nt, h.U, tag, flat_lds}, h};
    hold_fwd_alone(&copy, &sm, n, s);
  }
}

// ----------------------------------------------------------------------------- backward
// One pair of vectors after another (flat_lane_sums).
template <typename T, int V>
__device__ __forceinline__ void hold_sums_now(const u32x4& bx, const u32x4& bd, const float (&mu)[V], float (&b)[V], float (&s)[V]) {
#pragma clang fp contract(off)
  const float one = mix_one();
  const Pack<T, V> vx = flat_pack<T, V>(bx), vd = flat_pack<T, V>(bd);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    b[i] = __builtin_fmaf(to_f32(vd.v[i]), sub_f32<T>(vx.v[i], mu[i], one), b[i]);
    s[i] = add_f32<T>(s[i], vd.v[i], one);
  }
  hold_now(b);
  hold_now(s);
}

template <typename T, int V, int HA, int Q, bool LDS, int B>
struct HoldBwdOp : FlatBwdOp<T, V> {
  HoldArgs h;
  using Lane = HoldLane<T, V, HA, Q, LDS, B>;
  // in the kernel's order, in passes through one pass's registers
  __device__ __forceinline__ void sums(int64_t n, int l) const {
    const FlatArgs& a = this->a;
    const FlatSlab f = flat_slab<V>(a, l);
    const T* const sx = this->x + n * a.E + f.e0;
    const T* const sd = this->dy + n * a.E + f.e0;
    const Lane w(a, h, f.n_el);
    u32x4 rx[Q], rd[Q];
    float mu[V], b[V], d[V];
    this->means(mu);
#pragma unroll
    for (int i = 0; i < V; ++i) b[i] = d[i] = 0.f;
    w.template through<false>([&](auto&& f) { f(rx, sx); f(rd, sd); },
                              [&](int, int k) {
#pragma unroll
                                for (int r = k * B; r < (k + 1) * B; ++r) hold_sums_now<T, V>(rx[r], rd[r], mu, b, d);
                              },
                              [&](int k) {
#pragma unroll
                                for (int r = k * B; r < (k + 1) * B; ++r) {
                                  if (r >= w.skip) hold_sums_now<T, V>(rx[r], rd[r], mu, b, d);
                                }
                              });
    flat_merge_sums<V>(a, b, d, this->nt, this->lds, [&](int c, float cb, float cd) { this->publish(n, l, c, cb, cd); });
  }
  __device__ __forceinline__ void apply(int64_t n, int l) const {
    const FlatArgs& a = this->a;
    const FlatSlab f = flat_slab<V>(a, l);
    const T* const sx = this->x + n * a.E + f.e0;
    const T* const sd = this->dy + n * a.E + f.e0;
    T* const dst = this->dx + n * a.E + f.e0;
    const Lane w(a, h, f.n_el);
    const typename FlatBwdOp<T, V>::Coef coef = this->coef();
    if (static_cast<int>(threadIdx.x) >= a.A) return;
    u32x4 rx[Q], rd[Q];
    auto value = [&](int i) { return coef(flat_pinned<T, V>(flat_pack<T, V>(rx[i])), flat_pinned<T, V>(flat_pack<T, V>(rd[i]))); };
    w.template through<true>([&](auto&& f) { f(rx, sx); f(rd, sd); },
                             [&](int u, int k) { w.template store_own<B>(u + k * B, dst, [&](int i) { return value(k * B + i); }); },
                             [&](int k) { w.store(w.P, k, dst, value); });
  }
};

template <typename Op>
__device__ __attribute__((noinline)) void hold_bwd_alone(const Op* op, FlatShared* sm, int64_t n, int s) {
  flat_alone<false>(op->a, *op, *sm, op->nt, op->tag, n, s);
}

template <typename T, int V, int HA, int Q, bool LDS, int B>
__global__ void __launch_bounds__(kFlatMaxThreads, 2)
cl_hold_bwd(const T* __restrict__ dy, const T* __restrict__ x, const float* __restrict__ gamma,
            const float* __restrict__ mean_in, const float* __restrict__ rstd_in, T* __restrict__ dx,
            float* __restrict__ o0, float* __restrict__ o1, int64_t o_stride, FlatArgs a, HoldArgs h) {
  static_assert(HA % B == 0 && Q % B == 0, "whole batches");
  constexpr int NB = Q / B;
  extern __shared__ __attribute__((aligned(16))) float flat_lds[];
  __shared__ FlatShared sm;
  const int nt = block_threads();
  const unsigned tag = a.ex.the_tag();
  const FlatBwdOp<T, V> op{a, dy, x, gamma, mean_in, rstd_in, dx, o0, o1, o_stride, nt, h.U, tag, flat_lds};
  int64_t n;
  int s;
  if (!flat_place(a, n, s)) return;
  const typename FlatBwdOp<T, V>::Params params = op.fetch(n);
  const FlatSlab f = flat_slab<V>(a, s);
  const T* const sx = x + n * a.E + f.e0;
  const T* const sd = dy + n * a.E + f.e0;
  u32x4* const held = reinterpret_cast<u32x4*>(flat_lds + h.hold_at) + hold_thread();
  const HoldLane<T, V, HA, Q, LDS, B> w(a, h, f.n_el);

  u32x4 ox[HA], od[HA], rx[Q], rd[Q];
  auto load = [&](int p, int b, auto last) {
    w.template load<decltype(last)::value>(rx, p, b, sx);
    w.template load<decltype(last)::value>(rd, p, b, sd);
  };
  w.load(ox, sx);
  w.load(od, sd);
#pragma unroll
  for (int b = 0; b < NB; ++b) load(0, b, std::false_type{});
  op.template keep<false>(n, params);
  __syncthreads();
  float mu[V], sb[V], ss[V];
  op.means(mu);
#pragma unroll
  for (int i = 0; i < V; ++i) sb[i] = ss[i] = 0.f;
  auto sums = [&](const u32x4& bx, const u32x4& bd) { hold_sums_now<T, V>(bx, bd, mu, sb, ss); };
#pragma unroll
  for (int u = 0; u < HA; ++u) sums(ox[u], od[u]);
  if constexpr (LDS) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int r = b * B; r < (b + 1) * B; ++r) {
        sums(rx[r], rd[r]);
        held[2 * r * nt] = rx[r];
        held[(2 * r + 1) * nt] = rd[r];
      }
      load(1, b, std::false_type{});
    }
#pragma unroll 1
    for (int p = 1; p < w.P; ++p) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int r = b * B; r < (b + 1) * B; ++r) sums(rx[r], rd[r]);
        load(p + 1, b, std::false_type{});
      }
    }
  }
  w.settle(rx[Q - 1]);
  w.settle(rd[Q - 1]);
#pragma unroll
  for (int r = 0; r < Q; ++r) {
    if (r >= w.skip) sums(rx[r], rd[r]);
  }
  flat_merge_sums<V>(a, sb, ss, nt, flat_lds, [&](int c, float cb, float cd) { op.publish(n, s, c, cb, cd); });
  flat_exchange<false>(a, op, sm, nt, tag, n, s);
  if (flat_uniform(sm.fail) == 0) {
    flat_forget(ox);
    flat_forget(od);
    flat_forget(rx);
    flat_forget(rd);
    const typename FlatBwdOp<T, V>::Coef coef = op.coef();
    T* const dst = dx + n * a.E + f.e0;
    auto value = [&](const u32x4& vx, const u32x4& vd) {
      return coef(flat_pinned<T, V>(flat_pack<T, V>(vx)), flat_pinned<T, V>(flat_pack<T, V>(vd)));
    };
    auto ringed = [&](int r) { return value(rx[r], rd[r]); };
    if (static_cast<int>(threadIdx.x) < a.A) {
      if constexpr (LDS) {
#pragma unroll 1
        for (int p = w.P; p > 1; --p) {
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            w.store(p, b, dst, ringed);
            load(p - 1, b, std::true_type{});
          }
        }
      }
      w.template store_own<HA>(0, dst, [&](int u) { return value(ox[u], od[u]); });
#pragma unroll
      for (int b = 0; b < NB; ++b) w.store(LDS ? 1 : 0, b, dst, ringed);
      if constexpr (LDS) {
        const u32x4* const again = reinterpret_cast<const u32x4*>(flat_lds + h.hold_at) + hold_thread();
        w.template store_own<Q>(HA, dst, [&](int u) { return value(again[2 * u * nt], again[(2 * u + 1) * nt]); });
      }
    }
  }
  asm volatile("" ::: "memory");  // (asked for again, so that nothing of the slab lives across the call)
  if (flat_uniform(sm.fail) != 0) {
    const FlatArgs args = a;
    const HoldBwdOp<T, V, HA, Q, LDS, B> copy{{args, dy, x, gamma, mean_in, rstd_in, dx, o0, o1, o_stride, nt, h.U, tag, flat_lds}, h};
    hold_bwd_alone(&copy, &sm, n, s);
  }
}

}  // namespace atexn
