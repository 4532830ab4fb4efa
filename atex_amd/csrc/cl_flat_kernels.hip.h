// Channels-last InstanceNorm in one launch per direction, for any channel count of at least one
// vector: an instance is taken as the flat array of D * C elements that it is in memory.
//
// The other channels-last kernels give a pixel a power of two of lanes and let the last vector of a
// pixel overlap its neighbour when C is no multiple of V: [59, 33*16*32, 17] fp16 moves 1.4 times its
// bytes in pieces of 34, on 3 of 4 lanes.  Here consecutive lanes hold consecutive 16-byte vectors
// whatever C is.  The channels of a vector's V elements repeat every P = C / gcd(C, V) vectors (a
// period; V / gcd(C, V) pixels), so a thread that steps by a whole number of periods meets the same V
// channels in every step: A = m * P of the workgroup's lanes hold data, thread t the vectors t, t + A,
// t + 2 A, ... of its workgroup's slab, U of them, in registers from the load to the store.
//
// A thread sums up its own V streams, and element e of the step's A * V lane sums belongs to channel
// e % C: the sums of a channel over the workgroup are every C-th entry of one array in LDS, for any C.
// With S > 1 slabs per instance the workgroups of an instance exchange their slabs' sums while they run,
// as tagged pairs (norm_common.hip.h): workgroup s folds the channels s, s + S, ... (a wave per channel,
// the lanes over the slabs) and publishes them, and every workgroup waits for all C of those.
//
// Bound by memory with data, by the exchange's two hops (about 4 us with the merges in LDS) without:
// forward [28, 13300, 29] bf16 13.7 us (two stages 26.7; 43 MB at 5.5 TB/s: 7.9), [36, 36288, 29] fp16 31.6
// (59.1; 27.6), backward [22, 14280, 17] fp16 14.3 (22.9; 5.8).  128 registers, four waves per SIMD: what a launch can hold at
// once counts for more than the next slab's loads in flight.
//
// Nothing depends on which workgroups are on the chip together.  A workgroup publishes its slab's sums
// before it waits for anything, and every wait is a bounded number of polls.  A workgroup whose wait runs
// out looks which slabs have no sums, all at once, claims one of them (an atomic exchange on a word per slab),
// computes its sums, to the same bits, and looks again until nothing is left to claim: every slab's sums are
// there or in the hands of a running workgroup.  It does the duties of the slabs that it has computed (the
// channels that they fold) besides its own, so that every channel's fold is a running workgroup's, waits for
// those, and reads its own slab a second time to normalise it.  That is code of its own, outside the kernel:
// compiled into it, it doubled the registers of the held vectors (the look and the claim alone, for workgroups
// that find nothing to claim to go on with theirs, spilled 25), and what a kernel runs only once in a while
// comes from memory cold, some microseconds of instruction fetches.  The outputs must not alias x (the slabs are
// read again).
#pragma once

#include "norm_common.hip.h"

namespace atexn {

constexpr int kFlatMaxThreads = 512;
constexpr int kFlatMaxSlabs = 512;
constexpr int kFlatFwdMost = 16, kFlatBwdMost = 8;  // vectors per thread
constexpr int kFlatOwnPolls = 1 << 16;  // for values known to be published: bounds the wait only
// How long a wait lasts, in polls of about 0.15 us (exchange_wait_pair), besides one for each vector of a thread:
// the slabs of an instance that is on the chip together end the further apart the larger they are.  After 24
// polls most workgroups of held instances took running peers for absent ones (fp16 [2, 128^3, 32], 64 vectors, on
// a free GPU with waits cut short: forward 121 us -> 570), 99 were enough there, 159 for 128 vectors, not 300 for
// 512 and 1024 (backward [1, 2^24, 64] bf16 2230 us, 1880 with 600), 600 were.
constexpr int kFlatHastyPolls = 112;

// A value that is the same in every thread, as the compiler's scalar: a branch on it keeps no copy of the
// held vectors for lanes that might not take it.
__device__ __forceinline__ int flat_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

struct FlatArgs {
  int64_t N, D, E;     // instances, pixels and elements (D * C) of one
  int C, P, A;         // channels; vectors per period; lanes that hold data
  int S, base, extra;  // slabs per instance; periods of a slab, the last `extra` have one more
  int pix;             // pixels per period
  int width;           // lanes that share the fold of a channel: a power of two, at least S if S < 64, else 64
  float inv_d;         // 1 / D
  float px_more, px_base, px_last;  // pixels of the last `extra` slabs, of the others, of the very last one
  int local;           // the slabs of an instance on one XCD
  int hasty;           // polls of a wait that is cut short
  int k_at;            // where in LDS the channels' parameters, then constants, are: behind the sums
  ExchangeArgs ex;
  cl_word* tagged;      // [N][S][C] pairs: the slabs' sums
  cl_word* finals;      // [N][C] pairs: the instances'
  unsigned* claims;     // [N][S]: tag: a workgroup that has given up waiting computes the slab's sums
};

// A slab: where it starts (elements from the instance's first), its elements and pixels.
struct FlatSlab {
  int64_t e0;
  int n_el;
};
template <int V>
__device__ __forceinline__ FlatSlab flat_slab(const FlatArgs& a, int s) {
  const int more = s - (a.S - a.extra);
  const int64_t p0 = static_cast<int64_t>(s) * a.base + (more > 0 ? more : 0);
  const int k = a.base + (more >= 0 ? 1 : 0);
  const int64_t px0 = p0 * a.pix, px1 = px0 + static_cast<int64_t>(k) * a.pix;
  const int64_t px = (px1 < a.D ? px1 : a.D) - px0;
  FlatSlab f;
  f.e0 = px0 * a.C;
  f.n_el = static_cast<int>(px) * a.C;
  return f;
}

__device__ __forceinline__ float flat_pixels(const FlatArgs& a, int s) {
  return s == a.S - 1 ? a.px_last : (s < a.S - a.extra ? a.px_base : a.px_more);
}

// Which slab of which instance the workgroup takes.  local: unit by unit on each XCD (cl_single_place
// has the order); else the slabs of all instances in turn, over all XCDs.
__device__ __forceinline__ bool flat_place(const FlatArgs& a, int64_t& n, int& s) {
  const unsigned b = blockIdx.x, S = static_cast<unsigned>(a.S);
  if (a.local) {
    const unsigned j = b / 8;
    n = static_cast<int64_t>(j / S) * 8 + b % 8;
    s = static_cast<int>(j % S);
    return n < a.N;
  }
  n = b / S;
  s = static_cast<int>(b % S);
  return true;
}

// A held vector is kept as its 16 bytes and taken apart at each use: a register quad whatever T is.
template <typename T, int V>
__device__ __forceinline__ u32x4 flat_bits(const Pack<T, V>& p) {
  u32x4 b;
  __builtin_memcpy(&b, &p, 16);
  return b;
}
template <typename T, int V>
__device__ __forceinline__ Pack<T, V> flat_pack(const u32x4& b) {
  Pack<T, V> p;
  __builtin_memcpy(&p, &b, 16);
  return p;
}
// A vector as its 16 bytes: the compiler rounds a multiply-add to half precision once or twice
// (v_fma_mixlo_f16 or a conversion) depending on where its operands come from and its result goes.
template <typename T, int V>
__device__ __forceinline__ Pack<T, V> flat_pinned(const Pack<T, V>& p) {
  u32x4 b = flat_bits(p);
  asm volatile("" : "+v"(b));
  return flat_pack<T, V>(b);
}
template <int U>
__device__ __forceinline__ void flat_forget(u32x4 (&raw)[U]) {  // no value derived from a vector outlives this
#pragma unroll
  for (int u = 0; u < U; ++u) asm volatile("" : "+v"(raw[u]));
}

// The next step's element offset.  (Opaque to the compiler, which would otherwise keep a 64-bit base for
// each of the U steps in scalar registers, U pairs for every array that is read or written.)
__device__ __forceinline__ void flat_advance(unsigned& at, unsigned step) {
  at += step;
  asm volatile("" : "+v"(at));
}
// The thread's U vectors of a slab (at most MAX; the last one in the last place).  All steps but the last are
// whole (the planner sees to it); nv: the thread's valid elements of the last one, the others read as zero.
template <typename T, int V, int MAX, bool LAST>
__device__ __forceinline__ void flat_load(const T* src, int A, int n_el, int U, u32x4 (&raw)[MAX], int& nv) {
  const int t = static_cast<int>(threadIdx.x);
  const unsigned step = static_cast<unsigned>(A) * V;
  unsigned at = static_cast<unsigned>(t) * V;
  const int left = n_el - static_cast<int>((U - 1) * step + at);
  nv = t >= A || left <= 0 ? 0 : (left < V ? left : V);
#pragma unroll
  for (int u = 0; u < MAX; ++u) raw[u] = u32x4{};
  if (t < A) {
#pragma unroll
    for (int u = 0; u < MAX - 1; ++u) {
      if (u < U - 1) {
        raw[u] = flat_bits(LAST ? load_pack_last<T, V>(src + at) : load_pack<T, V>(src + at));
        flat_advance(at, step);
      }
    }
    if (nv == V) {
      raw[MAX - 1] = flat_bits(LAST ? load_pack_last<T, V>(src + at) : load_pack<T, V>(src + at));
    }
    // (an `else` puts these loads, and the wait for them, ahead of the whole vector's)
    if (nv > 0 && nv < V) {
      Pack<T, V> part;
#pragma unroll
      for (int i = 0; i < V; ++i) part.v[i] = i < nv ? src[at + i] : T(0);
      raw[MAX - 1] = flat_bits(part);
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load is on its way before the first use
}
template <typename T, int V, int MAX, typename F>
__device__ __forceinline__ void flat_store(T* dst, int A, int U, int nv, F&& value) {
  const int t = static_cast<int>(threadIdx.x);
  const unsigned step = static_cast<unsigned>(A) * V;
  unsigned at = static_cast<unsigned>(t) * V;
  if (t >= A) return;
#pragma unroll
  for (int u = 0; u < MAX - 1; ++u) {
    if (u < U - 1) {
      store_pack<T, V>(dst + at, value(u));
      flat_advance(at, step);
    }
  }
  if (nv > 0) store_pack_n<T, V>(dst + at, value(MAX - 1), nv);
}

// How the workgroup's threads share the entries of the channels: thread (q, c) of Q * C, or with more
// channels than threads every thread some channels.
struct FlatShare {
  int Q, q, c0, step;
};
__device__ __forceinline__ FlatShare flat_share(int C, int nt) {
  const int t = static_cast<int>(threadIdx.x);
  FlatShare f;
  if (C > nt) {
    f.Q = 1;
    f.q = 0;
    f.c0 = t;
    f.step = nt;
  } else {
    f.Q = nt / C;
    f.q = t / C;
    f.c0 = f.q < f.Q ? t - f.q * C : C;  // (a thread beyond Q * C has no channel)
    f.step = C;  // (one channel)
  }
  return f;
}

// f(value of l[e], e) for e = first, first + stride, ... < end in that order, eight loads in flight.
template <typename F>
__device__ __forceinline__ void flat_each(const float* l, int first, int end, int stride, F&& f) {
  constexpr int B = 8;
#pragma unroll 1
  for (int e = first; e < end; e += B * stride) {
    float v[B];
#pragma unroll
    for (int k = 0; k < B; ++k) v[k] = l[e + k * stride < end ? e + k * stride : e];
#pragma unroll
    for (int k = 0; k < B; ++k) {
      if (e + k * stride < end) f(v[k], e + k * stride);
    }
  }
}

// The thread's V streams over its U vectors (placed as flat_load has them; the last one nv elements): mean and
// squared deviations, an exact two-pass over the registers.
template <typename T, int V, int MAX, typename Vector>
__device__ __forceinline__ void flat_lane_stats(int U, int nv, Vector&& vector, float (&m)[V], float (&q)[V]) {
#pragma clang fp contract(off)  // (a thread's sums have the same bits wherever they are computed)
  const float one = mix_one();
#pragma unroll
  for (int i = 0; i < V; ++i) m[i] = q[i] = 0.f;
#pragma unroll
  for (int u = 0; u < MAX; ++u) {
    if (u < U - 1 || u == MAX - 1) {
      const Pack<T, V> x = vector(u);
#pragma unroll
      for (int i = 0; i < V; ++i) m[i] = add_f32<T>(m[i], x.v[i], one);
    }
  }
  const float whole = 1.0f / static_cast<float>(U), less = U > 1 ? 1.0f / static_cast<float>(U - 1) : 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) m[i] *= i < nv ? whole : less;
#pragma unroll
  for (int u = 0; u < MAX; ++u) {
    if (u < U - 1 || u == MAX - 1) {
      const Pack<T, V> x = vector(u);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        float d = sub_f32<T>(x.v[i], m[i], one);
        if (u == MAX - 1) d = i < nv ? d : 0.f;
        q[i] = __builtin_fmaf(d, d, q[i]);
      }
    }
  }
}
// Statistics of the slab per channel from its threads': done(c, mean, m2) by one thread per channel, Chan's
// merge of all of the channel's entries at once.  lds: 2 * A * V + 2 * max(threads, C) floats, of which the
// first 2 * A * V are free when done is called.
template <int V, typename Done>
__device__ __forceinline__ void flat_merge_stats(const FlatArgs& a, const FlatSlab& f, float pixels, int U, const float (&m)[V],
                                                 const float (&q)[V], int nt, float* lds, Done&& done) {
#pragma clang fp contract(off)
  const int t = static_cast<int>(threadIdx.x);
  const int AV = a.A * V;
  float* em = lds;
  float* eq = lds + AV;
  float* l1 = lds + 2 * AV;
  float* l2 = l1 + (nt > a.C ? nt : a.C);
  if (t < a.A) {
    store_f32<V>(em + t * V, m);
    store_f32<V>(eq + t * V, q);
  }
  __syncthreads();
  const FlatShare sh = flat_share(a.C, nt);
  const int tail = f.n_el - (U - 1) * AV;  // entries below it have U values, the others U - 1
  const float inv = 1.0f / pixels;
  const float w1 = static_cast<float>(U), w0 = static_cast<float>(U - 1);
  const int stride = sh.Q * a.C;
  for (int c = sh.c0; c < a.C; c += sh.step) {
    float s = 0.f;
    flat_each(em, c + sh.q * a.C, AV, stride, [&](float v, int e) { s = __builtin_fmaf(e < tail ? w1 : w0, v, s); });
    l1[sh.q * a.C + c] = s;
  }
  __syncthreads();
  auto total = [&](const float* l, int c) {
    float s = 0.f;
    flat_each(l, c, stride, a.C, [&](float v, int) { s += v; });
    return s;
  };
  for (int c = sh.c0; c < a.C; c += sh.step) {
    const float mean = total(l1, c) * inv;
    float s = 0.f;
    flat_each(eq, c + sh.q * a.C, AV, stride, [&](float v, int) { s += v; });
    flat_each(em, c + sh.q * a.C, AV, stride, [&](float v, int e) {
      const float d = v - mean;
      s = __builtin_fmaf((e < tail ? w1 : w0) * d, d, s);
    });
    l2[sh.q * a.C + c] = s;
  }
  __syncthreads();
  for (int c = sh.q == 0 ? sh.c0 : a.C; c < a.C; c += sh.step) done(c, total(l1, c) * inv, total(l2, c));
}

// The same for the backward's sums: b = sum dy * (x - mu), s = sum dy.
template <typename T, int V, int MAX, typename Vx, typename Vd>
__device__ __forceinline__ void flat_lane_sums(int U, Vx&& vx, Vd&& vd, const float (&mu)[V], float (&b)[V],
                                               float (&s)[V]) {
#pragma clang fp contract(off)
  const float one = mix_one();
#pragma unroll
  for (int i = 0; i < V; ++i) b[i] = s[i] = 0.f;
#pragma unroll
  for (int u = 0; u < MAX; ++u) {
    if (u < U - 1 || u == MAX - 1) {
      const Pack<T, V> x = vx(u), d = vd(u);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        // (what the last step does not have reads as dy = 0)
        b[i] = __builtin_fmaf(to_f32(d.v[i]), sub_f32<T>(x.v[i], mu[i], one), b[i]);
        s[i] = add_f32<T>(s[i], d.v[i], one);
      }
    }
  }
}
template <int V, typename Done>
__device__ __forceinline__ void flat_merge_sums(const FlatArgs& a, const float (&b)[V], const float (&s)[V], int nt,
                                                float* lds, Done&& done) {
  const int t = static_cast<int>(threadIdx.x);
  const int AV = a.A * V;
  float* eb = lds;
  float* es = lds + AV;
  float* l1 = lds + 2 * AV;
  float* l2 = l1 + (nt > a.C ? nt : a.C);
  if (t < a.A) {
    store_f32<V>(eb + t * V, b);
    store_f32<V>(es + t * V, s);
  }
  __syncthreads();
  const FlatShare sh = flat_share(a.C, nt);
  const int stride = sh.Q * a.C;
  for (int c = sh.c0; c < a.C; c += sh.step) {
    float cb = 0.f, cs = 0.f;
    flat_each(eb, c + sh.q * a.C, AV, stride, [&](float v, int) { cb += v; });
    flat_each(es, c + sh.q * a.C, AV, stride, [&](float v, int) { cs += v; });
    l1[sh.q * a.C + c] = cb;
    l2[sh.q * a.C + c] = cs;
  }
  __syncthreads();
  for (int c = sh.q == 0 ? sh.c0 : a.C; c < a.C; c += sh.step) {
    float cb = 0.f, cs = 0.f;
    flat_each(l1, c, stride, a.C, [&](float v, int) { cb += v; });
    flat_each(l2, c, stride, a.C, [&](float v, int) { cs += v; });
    done(c, cb, cs);
  }
}

// group_sum over aligned groups of `width` lanes (uniform; a power of two).
__device__ __forceinline__ float flat_group_sum(float v, int width) {
  if (width >= 2) v += dpp_read<kDppQuadXor1>(v);
  if (width >= 4) v += dpp_read<kDppQuadXor2>(v);
  if (width >= 8) v += dpp_read<kDppRowHalfMirror>(v);
  if (width >= 16) v += dpp_read<kDppRowMirror>(v);
  if (width >= 32) v = swap_add<16>(v);
  if (width >= 64) v = swap_add<32>(v);
  return v;
}
// Channel c of instance n (want: there is one) from the pairs of at most 64 slabs, by a.width lanes; false
// when a wait of the wave runs out.  STATS: (mean, m2) by Chan's merge of all slabs at
// once; else sums.
template <bool STATS>
__device__ __forceinline__ bool flat_fold(const FlatArgs& a, unsigned tag, int64_t n, int c, bool want, int polls,
                                          unsigned* trouble, float& r0, float& r1) {
#pragma clang fp contract(off)
  const int sub = threadIdx.x & (a.width - 1);
  const unsigned stride = static_cast<unsigned>(a.C) * 2;
  const cl_word* const at = a.tagged + n * a.S * a.C * 2;
  const unsigned col = want ? 2u * c : 0u;
  const bool mine = want && sub < a.S;
  float p, q;
  if (!exchange_wait_pair(at + (mine ? sub * stride + col : 0u), mine, tag, polls, trouble, p, q, a.hasty)) return false;
  r0 = flat_group_sum(mine ? (STATS ? p * flat_pixels(a, sub) : p) : 0.f, a.width);
  if constexpr (STATS) {
    r0 *= a.inv_d;
    const float d = p - r0;
    q += flat_pixels(a, sub) * (d * d);
  }
  r1 = flat_group_sum(mine ? q : 0.f, a.width);
  return true;
}

// The same by the whole workgroup, for more slabs than a wave has lanes: thread t takes the slabs t, t +
// threads.  All threads call it, and all get the result; buf: 3 * 16 floats.
template <bool STATS>
__device__ __forceinline__ bool flat_fold_wide(const FlatArgs& a, unsigned tag, int64_t n, int c, int nt, int polls,
                                               unsigned* trouble, float* buf, float& r0, float& r1) {
#pragma clang fp contract(off)
  constexpr int R = kFlatMaxSlabs / 256;
  const unsigned stride = static_cast<unsigned>(a.C) * 2;
  const cl_word* const at = a.tagged + (n * a.S * a.C + c) * 2;
  const int wave = threadIdx.x / kWave, nw = nt / kWave;
  float p[R], q[R];
  float s0 = 0.f, s1 = 0.f;
  bool ok = true;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    p[r] = q[r] = 0.f;
    const int l = static_cast<int>(threadIdx.x) + r * nt;
    if (ok && r * nt < a.S) {  // (wave-uniform)
      ok = exchange_wait_pair(at + (l < a.S ? l * stride : 0u), l < a.S, tag, polls, trouble, p[r], q[r],
                              a.hasty);
      s0 += l < a.S ? (STATS ? p[r] * flat_pixels(a, l) : p[r]) : 0.f;
      if constexpr (!STATS) s1 += l < a.S ? q[r] : 0.f;
    }
  }
  s0 = group_sum<kWave>(s0);
  if constexpr (!STATS) s1 = group_sum<kWave>(s1);
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) {
    buf[wave] = s0;
    buf[16 + wave] = s1;
    buf[32 + wave] = ok ? 0.f : 1.f;
  }
  __syncthreads();
  r0 = buf[0];
  r1 = buf[16];
  float bad = buf[32];
  for (int w = 1; w < nw; ++w) {
    r0 += buf[w];
    r1 += buf[16 + w];
    bad += buf[32 + w];
  }
  if constexpr (STATS) {
    r0 *= a.inv_d;
    s1 = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int l = static_cast<int>(threadIdx.x) + r * nt;
      const float d = p[r] - r0;
      s1 += l < a.S ? q[r] + flat_pixels(a, l) * (d * d) : 0.f;
    }
    s1 = group_sum<kWave>(s1);
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) buf[wave] = s1;
    __syncthreads();
    r1 = buf[0];
    for (int w = 1; w < nw; ++w) r1 += buf[w];
  }
  return flat_uniform(bad > 0.f) == 0;
}

__device__ __forceinline__ void flat_publish(cl_word* pair, float v0, float v1, unsigned tag, bool local) {
  if (local) cl_publish(pair, v0, v1, tag);
  else cl_publish_device(pair, v0, v1, tag);
}

struct FlatShared {  // in LDS
  int fail;  // a wait has run out
  int pick;  // the slab that the workgroup has claimed then
  float buf[48];
  unsigned open[kFlatMaxSlabs / 32], mine[kFlatMaxSlabs / 32];  // slabs: nobody's, computed by this workgroup
};

// The fold of the channels of slab `sk` by the workgroup, published as the instance's; whether a wait of the
// wave ran out.  OP: result(n, c, r0, r1) (what the instance's folded pair means: outputs, and the pair to
// publish).  CERTAIN: for sums that are on their way; should they not show up after all, the results are
// marked (NaN).
template <bool STATS, bool CERTAIN, typename Op>
__device__ __forceinline__ bool flat_own(const FlatArgs& a, Op& op, FlatShared& sm, int nt, unsigned tag, int64_t n, int sk,
                                         int polls, unsigned* trouble) {
  const int lane = threadIdx.x & (kWave - 1), wave = flat_uniform(threadIdx.x / kWave), nw = nt / kWave;
  const int at_once = kWave / a.width;  // channels of a wave
  bool fail = false;
  auto done = [&](int c, bool mine, float r0, float r1) {
    if (CERTAIN && fail) {
      r0 = r1 = __builtin_nanf("");
      fail = false;
    }
    if (!fail && mine) {
      op.result(n, c, r0, r1);
      flat_publish(a.finals + (n * a.C + c) * 2, r0, r1, tag, a.local);
    }
  };
  if (a.S > kWave) {
#pragma unroll 1
    for (int c = sk; c < a.C && !fail; c += a.S) {  // (the same in every wave)
      float r0, r1;
      fail = !flat_fold_wide<STATS>(a, tag, n, c, nt, polls, trouble, sm.buf, r0, r1);
      done(c, threadIdx.x == 0, r0, r1);
    }
  } else {
#pragma unroll 1
    for (int c0 = sk + wave * at_once * a.S; c0 < a.C && !fail; c0 += nw * at_once * a.S) {
      const int c = c0 + lane / a.width * a.S;
      float r0, r1;
      fail = !flat_fold<STATS>(a, tag, n, c, c < a.C, polls, trouble, r0, r1);
      done(c, c < a.C && (lane & (a.width - 1)) == 0, r0, r1);
    }
  }
  return fail;
}
// The instance's pairs as constants(n, c, r0, r1) in LDS, a lane per channel; whether a wait of the wave ran out.
template <bool CERTAIN, typename Op>
__device__ __forceinline__ bool flat_finals(const FlatArgs& a, Op& op, int nt, unsigned tag, int64_t n, int polls,
                                            unsigned* trouble) {
  const int lane = threadIdx.x & (kWave - 1), wave = flat_uniform(threadIdx.x / kWave);
  bool fail = false;
#pragma unroll 1
  for (int c0 = wave * kWave; c0 < a.C && !fail; c0 += nt) {
    const int c = c0 + lane;
    float r0, r1;
    fail = !exchange_wait_pair(a.finals + (n * a.C + (c < a.C ? c : 0)) * 2, c < a.C, tag, polls, trouble, r0, r1,
                               a.hasty);
    if (CERTAIN && fail) {
      r0 = r1 = __builtin_nanf("");
      fail = false;
    }
    if (!fail && c < a.C) op.constants(n, c, r0, r1);
  }
  return fail;
}

// The exchange of instance n by its workgroup s; sm.fail: whether a wait ran out.
template <bool STATS, typename Op>
__device__ __forceinline__ void flat_exchange(const FlatArgs& a, Op& op, FlatShared& sm, int nt, unsigned tag, int64_t n,
                                              int s) {
  if (threadIdx.x == 0) sm.fail = 0;
  __syncthreads();
  const bool fail = flat_own<STATS, false>(a, op, sm, nt, tag, n, s, a.ex.max_polls, a.ex.trouble) ||
                    flat_finals<false>(a, op, nt, tag, n, a.ex.max_polls, a.ex.trouble);
  if (fail && (threadIdx.x & (kWave - 1)) == 0) sm.fail = 1;
  __syncthreads();
}

// A slab of instance n whose sums are neither there nor anybody's to compute, claimed for this workgroup; -1
// when there is none (left).  A slab's workgroup publishes all of its channels without waiting, so one of them
// tells.  Every round in which another workgroup was quicker claims a slab: there are at most S.  The claims
// of workgroups that look at the same time spread over the open slabs.  Contains barriers.
__device__ __forceinline__ int flat_claim(const FlatArgs& a, FlatShared& sm, int nt, unsigned tag, int64_t n, int s) {
  constexpr int WORDS = kFlatMaxSlabs / 32;
  const int t = static_cast<int>(threadIdx.x);
  unsigned* const claims = a.claims + n * a.S;
#pragma unroll 1
  for (int round = 0; round < a.S; ++round) {
    __syncthreads();
    if (t < WORDS) sm.open[t] = 0;
    __syncthreads();
#pragma unroll 1
    for (int l = t; l < a.S; l += nt) {
      const cl_word* const pair = a.tagged + ((n * a.S + l) * a.C + a.C - 1) * 2;
      const cl_word w0 = cl_peek(pair), w1 = cl_peek(pair + 1);
      const unsigned whose = __hip_atomic_load(claims + l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool there = static_cast<unsigned>(w0 >> 32) == tag && static_cast<unsigned>(w1 >> 32) == ~tag;
      if (l != s && !there && whose != tag) atomicOr(&sm.open[l / 32], 1u << l % 32);
    }
    __syncthreads();
    if (t == 0) {
      int total = 0;
#pragma unroll 1
      for (int w = 0; w < WORDS; ++w) total += __popc(sm.open[w]);
      int pick = -1;
      if (total > 0) {
        int k = s % total, w = 0;
#pragma unroll 1
        while (k >= __popc(sm.open[w])) k -= __popc(sm.open[w++]);
        unsigned bits = sm.open[w];
#pragma unroll 1
        for (; k > 0; --k) bits &= bits - 1;
        const int l = w * 32 + __ffs(bits) - 1;
        pick = atomicExch(claims + l, tag) != tag ? l : -2;
      }
      sm.pick = pick;
    }
    __syncthreads();
    const int pick = flat_uniform(sm.pick);
    if (pick != -2) return pick;
  }
  return -1;
}

// A workgroup whose wait has run out, to its end.  OP has also params(n) (the channels' parameters into LDS),
// sums(n, l) (slab l's, published) and apply(n, l).
template <bool STATS, typename Op>
__device__ __forceinline__ void flat_alone(const FlatArgs& a, Op& op, FlatShared& sm, int nt, unsigned tag, int64_t n, int s) {
  constexpr int WORDS = kFlatMaxSlabs / 32;
  if (threadIdx.x < WORDS) sm.mine[threadIdx.x] = 0;
  op.params(n);
#pragma unroll 1
  for (int l; (l = flat_claim(a, sm, nt, tag, n, s)) >= 0;) {
    if (threadIdx.x == 0) sm.mine[l / 32] |= 1u << l % 32;
    op.sums(n, l);
  }
  __syncthreads();
#pragma unroll 1
  for (int w = 0; w < WORDS; ++w) {
    unsigned bits = static_cast<unsigned>(flat_uniform(static_cast<int>(sm.mine[w] | (w == s / 32 ? 1u << s % 32 : 0u))));
#pragma unroll 1
    for (; bits != 0; bits &= bits - 1) {
      flat_own<STATS, true>(a, op, sm, nt, tag, n, w * 32 + __ffs(bits) - 1, kFlatOwnPolls, nullptr);
    }
  }
  flat_finals<true>(a, op, nt, tag, n, kFlatOwnPolls, nullptr);
  __syncthreads();
  op.apply(n, s);
}

// ------------------------------------------------------------------------------ forward
template <typename T, int V>
struct FlatFwdOp {
  const FlatArgs& a;
  const T* x;
  const float* gamma;
  const float* beta;
  T* y;
  float* mean_out;
  float* rstd_out;
  float eps;
  int nt, U;
  unsigned tag;
  float* lds;

  // (mean, m2) becomes (mean, inverse std)
  __device__ __forceinline__ void result(int64_t n, int c, float& m, float& q) const {
    q = rsqrtf(__builtin_fmaf(q, a.inv_d, eps));
    mean_out[n * a.C + c] = m;
    rstd_out[n * a.C + c] = q;
  }
  // the channels' parameters: asked for ahead of the slab, stored behind its loads
  struct Params {
    float g, b;
  };
  __device__ __forceinline__ Params fetch(int64_t) const {
    const int c = static_cast<int>(threadIdx.x) < a.C ? threadIdx.x : 0;
    return Params{gamma[c], beta[c]};
  }
  template <bool MANY = true>  // (more channels than threads)
  __device__ __forceinline__ void keep(int64_t, Params p) const {
    float* k = lds + a.k_at;
    const int mine = static_cast<int>(threadIdx.x) < a.C ? threadIdx.x : 0;  // (no branch: the others have channel 0's)
    k[a.C + mine] = p.g;
    k[2 * a.C + mine] = p.b;
    if (MANY && a.C > nt) {  // (a loop with loads waits for all others before it)
#pragma unroll 1
      for (int c = threadIdx.x + nt; c < a.C; c += nt) {
        k[a.C + c] = gamma[c];
        k[2 * a.C + c] = beta[c];
      }
    }
  }
  __device__ __forceinline__ void params(int64_t n) const { keep(n, fetch(n)); }
  __device__ __forceinline__ void constants(int64_t, int c, float m, float r) const {
    float* k = lds + a.k_at + c;
    k[0] = m;
    k[a.C] *= r;
  }
  struct Coef {
    float m[V], sc[V], bt[V];
    __device__ __forceinline__ Pack<T, V> operator()(const Pack<T, V>& v) const {
      const float one = mix_one();
      Pack<T, V> o;
#pragma unroll
      for (int i = 0; i < V; ++i) o.v[i] = from_f32<T>(__builtin_fmaf(sub_f32<T>(v.v[i], m[i], one), sc[i], bt[i]));
      return flat_pinned<T, V>(o);
    }
  };
  __device__ __forceinline__ Coef coef() const {
    const float* k = lds + a.k_at;
    Coef f;
    int c = static_cast<int>(threadIdx.x) * V % a.C;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      f.m[i] = k[c];
      f.sc[i] = k[a.C + c];
      f.bt[i] = k[2 * a.C + c];
      c = c + 1 == a.C ? 0 : c + 1;
    }
    return f;
  }
  __device__ __forceinline__ void publish(int64_t n, int l, int c, float m, float q) const {
    if (a.S > 1) {
      flat_publish(a.tagged + ((n * a.S + l) * a.C + c) * 2, m, q, tag, a.local);
    } else {
      result(n, c, m, q);
      constants(n, c, m, q);
    }
  }
  // as the kernel has them
  __device__ __forceinline__ void sums(int64_t n, int l) const {
    const FlatSlab f = flat_slab<V>(a, l);
    u32x4 raw[kFlatFwdMost];
    int nv;
    flat_load<T, V, kFlatFwdMost, false>(x + n * a.E + f.e0, a.A, f.n_el, U, raw, nv);
    float m[V], q[V];
    flat_lane_stats<T, V, kFlatFwdMost>(U, nv, [&](int u) { return flat_pack<T, V>(raw[u]); }, m, q);
    flat_merge_stats<V>(a, f, flat_pixels(a, l), U, m, q, nt, lds, [&](int c, float cm, float cq) { publish(n, l, c, cm, cq); });
  }
  __device__ __forceinline__ void apply(int64_t n, int l) const {
    const FlatSlab f = flat_slab<V>(a, l);
    const Coef k = coef();
    u32x4 raw[kFlatFwdMost];
    int nv;
    flat_load<T, V, kFlatFwdMost, true>(x + n * a.E + f.e0, a.A, f.n_el, U, raw, nv);
    flat_store<T, V, kFlatFwdMost>(y + n * a.E + f.e0, a.A, U, nv, [&](int u) { return k(flat_pinned<T, V>(flat_pack<T, V>(raw[u]))); });
  }
};

// (a function of its own: its registers and scalars stay out of the kernel's)
template <typename T, int V>
__device__ __attribute__((noinline)) void flat_fwd_alone(const FlatFwdOp<T, V>* op, FlatShared* sm, int64_t n, int s) {
  flat_alone<true>(op->a, *op, *sm, op->nt, op->tag, n, s);
}

template <typename T, int V, int U>
__global__ void __launch_bounds__(kFlatMaxThreads, 4)
cl_flat_fwd(const T* __restrict__ x, const float* __restrict__ gamma, const float* __restrict__ beta,
            T* __restrict__ y, float* __restrict__ mean_out, float* __restrict__ rstd_out, FlatArgs a, float eps) {
  extern __shared__ __attribute__((aligned(16))) float flat_lds[];
  __shared__ FlatShared sm;
  const int nt = block_threads();
  const unsigned tag = a.S > 1 ? a.ex.the_tag() : 0;
  const FlatFwdOp<T, V> op{a, x, gamma, beta, y, mean_out, rstd_out, eps, nt, U, tag, flat_lds};
  int64_t n;
  int s;
  if (!flat_place(a, n, s)) return;
  const typename FlatFwdOp<T, V>::Params params = op.fetch(n);
  const FlatSlab f = flat_slab<V>(a, s);
  u32x4 raw[U];
  int nv;
  flat_load<T, V, U, false>(x + n * a.E + f.e0, a.A, f.n_el, U, raw, nv);
  op.keep(n, params);
  {
    float m[V], q[V];
    flat_lane_stats<T, V, U>(U, nv, [&](int u) { return flat_pack<T, V>(raw[u]); }, m, q);
    flat_merge_stats<V>(a, f, flat_pixels(a, s), U, m, q, nt, flat_lds, [&](int c, float cm, float cq) { op.publish(n, s, c, cm, cq); });
  }
  if (a.S > 1) {
    flat_exchange<true>(a, op, sm, nt, tag, n, s);
  } else {
    if (threadIdx.x == 0) sm.fail = 0;
    __syncthreads();
  }
  if (flat_uniform(sm.fail) == 0) {
    flat_forget(raw);
    const typename FlatFwdOp<T, V>::Coef k = op.coef();
    flat_store<T, V, U>(y + n * a.E + f.e0, a.A, U, nv, [&](int u) { return k(flat_pack<T, V>(raw[u])); });
  }
  asm volatile("" ::: "memory");  // (asked for again, so that nothing of the slab lives across the call)
  if (flat_uniform(sm.fail) != 0) {
    const FlatArgs args = a;
    const FlatFwdOp<T, V> copy{args, x, gamma, beta, y, mean_out, rstd_out, eps, nt, U, tag, flat_lds};
    flat_fwd_alone<T, V>(&copy, &sm, n, s);
  }
}

// ----------------------------------------------------------------------------- backward
template <typename T, int V>
struct FlatBwdOp {
  const FlatArgs& a;
  const T* dy;
  const T* x;
  const float* gamma;
  const float* mean_in;
  const float* rstd_in;
  T* dx;
  float* o0;
  float* o1;
  int64_t o_stride;
  int nt, U;
  unsigned tag;
  float* lds;

  // the channels' parameters: asked for ahead of the slab, stored behind its loads
  struct Params {
    float m, g, r;
  };
  __device__ __forceinline__ Params fetch(int64_t n) const { return at(n, static_cast<int>(threadIdx.x) < a.C ? threadIdx.x : 0); }
  __device__ __forceinline__ Params at(int64_t n, int c) const { return Params{mean_in[n * a.C + c], gamma[c], rstd_in[n * a.C + c]}; }
  template <bool MANY = true>  // (more channels than threads)
  __device__ __forceinline__ void keep(int64_t n, Params p) const {
    float* k = lds + a.k_at;
    auto put = [&](int c, const Params& v) {
      k[c] = v.m;
      k[a.C + c] = v.g;
      k[2 * a.C + c] = v.r;
    };
    put(static_cast<int>(threadIdx.x) < a.C ? threadIdx.x : 0, p);  // (no branch: the others have channel 0's)
    if (MANY && a.C > nt) {  // (a loop with loads waits for all others before it)
#pragma unroll 1
      for (int c = threadIdx.x + nt; c < a.C; c += nt) put(c, at(n, c));
    }
  }
  __device__ __forceinline__ void params(int64_t n) const { keep(n, fetch(n)); }
  __device__ __forceinline__ void means(float (&mu)[V]) const {
    const float* k = lds + a.k_at;
    int c = static_cast<int>(threadIdx.x) * V % a.C;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      mu[i] = k[c];
      c = c + 1 == a.C ? 0 : c + 1;
    }
  }
  // dgamma / dbeta themselves for a single instance, else partial rows for a col_reduce launch
  __device__ __forceinline__ void result(int64_t n, int c, float b, float d) const {
    o0[n * o_stride + c] = b;
    o1[n * o_stride + c] = d;
  }
  // constants of dx = sc * dy + (ca * (x - mu) + cb)
  __device__ __forceinline__ void constants(int64_t n, int c, float b, float d) const {
#pragma clang fp contract(off)
    float* k = lds + a.k_at + c;
    const float r = k[2 * a.C];
    const float sc = k[a.C] * r;
    k[a.C] = sc;
    k[2 * a.C] = -(sc * r) * (b * a.inv_d);
    k[3 * a.C] = -sc * (d * a.inv_d);
  }
  struct Coef {
    float mu[V], sc[V], ca[V], cb[V];
    __device__ __forceinline__ Pack<T, V> operator()(const Pack<T, V>& vx, const Pack<T, V>& vd) const {
      const float one = mix_one();
      Pack<T, V> o;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        o.v[i] = from_f32<T>(__builtin_fmaf(sc[i], to_f32(vd.v[i]),
                                            __builtin_fmaf(ca[i], sub_f32<T>(vx.v[i], mu[i], one), cb[i])));
      }
      return flat_pinned<T, V>(o);
    }
  };
  __device__ __forceinline__ Coef coef() const {
    const float* k = lds + a.k_at;
    Coef f;
    int c = static_cast<int>(threadIdx.x) * V % a.C;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      f.mu[i] = k[c];
      f.sc[i] = k[a.C + c];
      f.ca[i] = k[2 * a.C + c];
      f.cb[i] = k[3 * a.C + c];
      c = c + 1 == a.C ? 0 : c + 1;
    }
    return f;
  }
  __device__ __forceinline__ void publish(int64_t n, int l, int c, float b, float d) const {
    b *= lds[a.k_at + 2 * a.C + c];
    if (a.S > 1) {
      flat_publish(a.tagged + ((n * a.S + l) * a.C + c) * 2, b, d, tag, a.local);
    } else {
      result(n, c, b, d);
      constants(n, c, b, d);
    }
  }
  // as the kernel has them
  __device__ __forceinline__ void sums(int64_t n, int l) const {
    const FlatSlab f = flat_slab<V>(a, l);
    u32x4 rx[kFlatBwdMost], rd[kFlatBwdMost];
    int nv;
    flat_load<T, V, kFlatBwdMost, false>(x + n * a.E + f.e0, a.A, f.n_el, U, rx, nv);
    flat_load<T, V, kFlatBwdMost, false>(dy + n * a.E + f.e0, a.A, f.n_el, U, rd, nv);
    float mu[V], b[V], d[V];
    means(mu);
    flat_lane_sums<T, V, kFlatBwdMost>(U, [&](int u) { return flat_pack<T, V>(rx[u]); },
                                       [&](int u) { return flat_pack<T, V>(rd[u]); }, mu, b, d);
    flat_merge_sums<V>(a, b, d, nt, lds, [&](int c, float cb, float cd) { publish(n, l, c, cb, cd); });
  }
  __device__ __forceinline__ void apply(int64_t n, int l) const {
    const FlatSlab f = flat_slab<V>(a, l);
    const Coef k = coef();
    u32x4 rx[kFlatBwdMost], rd[kFlatBwdMost];
    int nv;
    flat_load<T, V, kFlatBwdMost, true>(x + n * a.E + f.e0, a.A, f.n_el, U, rx, nv);
    flat_load<T, V, kFlatBwdMost, true>(dy + n * a.E + f.e0, a.A, f.n_el, U, rd, nv);
    flat_store<T, V, kFlatBwdMost>(dx + n * a.E + f.e0, a.A, U, nv, [&](int u) {
      return k(flat_pinned<T, V>(flat_pack<T, V>(rx[u])), flat_pinned<T, V>(flat_pack<T, V>(rd[u])));
    });
  }
};

template <typename T, int V>
__device__ __attribute__((noinline)) void flat_bwd_alone(const FlatBwdOp<T, V>* op, FlatShared* sm, int64_t n, int s) {
  flat_alone<false>(op->a, *op, *sm, op->nt, op->tag, n, s);
}

template <typename T, int V, int U>
__global__ void __launch_bounds__(kFlatMaxThreads, 4)
cl_flat_bwd(const T* __restrict__ dy, const T* __restrict__ x, const float* __restrict__ gamma,
            const float* __restrict__ mean_in, const float* __restrict__ rstd_in, T* __restrict__ dx,
            float* __restrict__ o0, float* __restrict__ o1, int64_t o_stride, FlatArgs a) {
  extern __shared__ __attribute__((aligned(16))) float flat_lds[];
  __shared__ FlatShared sm;
  const int nt = block_threads();
  const unsigned tag = a.S > 1 ? a.ex.the_tag() : 0;
  const FlatBwdOp<T, V> op{a, dy, x, gamma, mean_in, rstd_in, dx, o0, o1, o_stride, nt, U, tag, flat_lds};
  int64_t n;
  int s;
  if (!flat_place(a, n, s)) return;
  const typename FlatBwdOp<T, V>::Params params = op.fetch(n);
  const FlatSlab f = flat_slab<V>(a, s);
  u32x4 rx[U], rd[U];
  int nv;
  flat_load<T, V, U, true>(x + n * a.E + f.e0, a.A, f.n_el, U, rx, nv);
  flat_load<T, V, U, true>(dy + n * a.E + f.e0, a.A, f.n_el, U, rd, nv);
  op.keep(n, params);
  __syncthreads();
  {
    float mu[V], b[V], d[V];
    op.means(mu);
    flat_lane_sums<T, V, U>(U, [&](int u) { return flat_pack<T, V>(rx[u]); }, [&](int u) { return flat_pack<T, V>(rd[u]); },
                         mu, b, d);
    flat_merge_sums<V>(a, b, d, nt, flat_lds, [&](int c, float cb, float cd) { op.publish(n, s, c, cb, cd); });
  }
  if (a.S > 1) {
    flat_exchange<false>(a, op, sm, nt, tag, n, s);
  } else {
    if (threadIdx.x == 0) sm.fail = 0;
    __syncthreads();
  }
  if (flat_uniform(sm.fail) == 0) {
    flat_forget(rx);
    flat_forget(rd);
    const typename FlatBwdOp<T, V>::Coef k = op.coef();
    flat_store<T, V, U>(dx + n * a.E + f.e0, a.A, U, nv, [&](int u) { return k(flat_pack<T, V>(rx[u]), flat_pack<T, V>(rd[u])); });
  }
  asm volatile("" ::: "memory");  // (asked for again, so that nothing of the slab lives across the call)
  if (flat_uniform(sm.fail) != 0) {
    const FlatArgs args = a;
    const FlatBwdOp<T, V> copy{args, dy, x, gamma, mean_in, rstd_in, dx, o0, o1, o_stride, nt, U, tag, flat_lds};
    flat_bwd_alone<T, V>(&copy, &sm, n, s);
  }
}

}  // namespace atexn
