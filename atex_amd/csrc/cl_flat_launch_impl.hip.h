// Launchers of the flat channels-last kernels, templated on the storage type.
#pragma once

#include "cl_hold_kernels.hip.h"
#include "large_lds.h"
#include "plan.h"
#include "status.h"

namespace atexn {

static_assert(kPlanFlatMaxSlabs == kFlatMaxSlabs && kPlanFlatMaxThreads == kFlatMaxThreads,
              "the planner and the flat kernels must agree on their limits");

// float32 backwards go on the held kernels or stay on the slabs' (flat_may): the flat ones are built only where
// a switch can ask for them.
#ifdef ATEXN_BENCH_BUILD
constexpr bool kFlatBwdAnyWidth = true;
#else
constexpr bool kFlatBwdAnyWidth = false;
#endif

inline FlatArgs flat_args(const FlatPlan& p, int64_t N, int64_t C, int64_t D, void* ws, const ExchangeTag& e) {
  char* w = static_cast<char*>(ws);
  FlatArgs a;
  a.N = N;
  a.D = D;
  a.E = D * C;
  a.C = static_cast<int>(C);
  a.P = p.P;
  a.A = p.A;
  a.S = p.S;
  a.base = p.base;
  a.extra = p.extra;
  a.pix = p.pix;
  a.width = std::min(64, pow2_ceil(p.S));
  a.inv_d = 1.0f / static_cast<float>(D);
  a.px_base = static_cast<float>(int64_t(p.base) * p.pix);
  a.px_more = static_cast<float>((int64_t(p.base) + 1) * p.pix);
  a.px_last = static_cast<float>(D - (int64_t(p.S - 1) * p.base + std::max(p.extra - 1, 0)) * p.pix);
  a.local = p.local;
  a.k_at = p.k_at;
  const int polls = tuning().cl_flat_polls;
  a.ex = ExchangeArgs{e.tag, e.at, polls < kExchangePatientPolls ? polls : polls + p.U, e.trouble};
  a.hasty = kFlatHastyPolls + p.U;
  a.tagged = reinterpret_cast<cl_word*>(w + p.off_tagged);
  a.finals = reinterpret_cast<cl_word*>(w + p.off_finals);
  a.claims = reinterpret_cast<unsigned*>(w + p.off_claims);
  return a;
}

inline HoldArgs hold_args(const FlatPlan& p) { return HoldArgs{p.U, p.R, p.hold_at}; }

template <auto Kernel, typename... Args>
int hold_launch(const FlatPlan& p, hipStream_t st, const char* name, Args... args) {
  ATEXN_REQUIRE(allow_large_lds<Kernel>() == hipSuccess, "this device does not give a workgroup %zu bytes of LDS", p.lds);
  Kernel<<<static_cast<unsigned>(p.grid), p.threads, p.lds, st>>>(args..., hold_args(p));
  ATEXN_CHECK_LAUNCH(name);
  return ATEXN_OK;
}
// f(K): the kind of the plan's hold kernel as a constant.
template <size_t N, typename F, size_t... K>
int hold_kind(const HoldKind (&)[N], const FlatPlan& p, F&& f, std::index_sequence<K...>) {
  int rc = ATEXN_INVALID_ARGUMENT;
  (void)((static_cast<int>(K) == p.kind && ((rc = f(std::integral_constant<size_t, K>{})), true)) || ...);
  return rc;
}

// Launches the call's kernel unless its workgroups may not exchange results (taken: it did).
template <typename T, int V>
int flat_fwd_v(const FlatPlan& p, const T* x, const float* gamma, const float* beta, int64_t N, int64_t C, int64_t D,
               float eps, T* y, float* mean, float* rstd, void* ws, hipStream_t st, bool& taken) {
  ExchangeTag e;
  e.ok = true;
  if (p.S > 1) ATEXN_TRY(exchange_tag(st, static_cast<char*>(ws) + p.off_tag, e));
  taken = e.ok;
  if (!taken) return ATEXN_OK;
  const FlatArgs a = flat_args(p, N, C, D, ws, e);
  const unsigned grid = static_cast<unsigned>(p.grid);
  if (p.hold) {
    return hold_kind(kPlanHoldFwd, p, [&](auto k) {
      constexpr HoldKind h = kPlanHoldFwd[k];
      return hold_launch<cl_hold_fwd<T, V, h.HA, kPlanHoldFwdPass, h.lds, kPlanHoldFwdBatch>>(
          p, st, "cl_hold_fwd", x, gamma, beta, y, mean, rstd, a, eps);
    }, std::make_index_sequence<std::size(kPlanHoldFwd)>{});
  }
#define ATEXN_FLAT_FWD(U_) \
  case U_: cl_flat_fwd<T, V, U_><<<grid, p.threads, p.lds, st>>>(x, gamma, beta, y, mean, rstd, a, eps); break
  switch (p.U) {
    ATEXN_FLAT_FWD(1);
    ATEXN_FLAT_FWD(2);
    ATEXN_FLAT_FWD(3);
    ATEXN_FLAT_FWD(4);
    ATEXN_FLAT_FWD(6);
    ATEXN_FLAT_FWD(8);
    ATEXN_FLAT_FWD(12);
    ATEXN_FLAT_FWD(16);
    default: return set_error(ATEXN_INVALID_ARGUMENT, "no kernel for %d vectors per thread", p.U);
  }
#undef ATEXN_FLAT_FWD
  ATEXN_CHECK_LAUNCH("cl_flat_fwd");
  return ATEXN_OK;
}

template <typename T, int V>
int flat_bwd_v(const FlatPlan& p, const T* dy, const T* x, const float* gamma, const float* mean, const float* rstd,
               int64_t N, int64_t C, int64_t D, T* dx, float* dgamma, float* dbeta, void* ws, hipStream_t st,
               bool& taken) {
  ExchangeTag e;
  e.ok = true;
  if (p.S > 1) ATEXN_TRY(exchange_tag(st, static_cast<char*>(ws) + p.off_tag, e));
  taken = e.ok;
  if (!taken) return ATEXN_OK;
  const FlatArgs a = flat_args(p, N, C, D, ws, e);
  const unsigned grid = static_cast<unsigned>(p.grid);
  float* part = reinterpret_cast<float*>(static_cast<char*>(ws) + p.off_part);
  float* o0 = N == 1 ? dgamma : part;
  float* o1 = N == 1 ? dbeta : part + C;
  if (p.hold) {
    ATEXN_TRY(hold_kind(kPlanHoldBwd, p, [&](auto k) {
      constexpr HoldKind h = kPlanHoldBwd[k];
      return hold_launch<cl_hold_bwd<T, V, h.HA, kPlanHoldBwdPass, h.lds, kPlanHoldBwdBatch>>(
          p, st, "cl_hold_bwd", dy, x, gamma, mean, rstd, dx, o0, o1, 2 * C, a);
    }, std::make_index_sequence<std::size(kPlanHoldBwd)>{}));
    if (N > 1) return launch_col_reduce(part, dgamma, dbeta, static_cast<int>(N), C, st);
    return ATEXN_OK;
  }
  if constexpr (V == 8 || kFlatBwdAnyWidth) {
#define ATEXN_FLAT_BWD(U_) \
  case U_: cl_flat_bwd<T, V, U_><<<grid, p.threads, p.lds, st>>>(dy, x, gamma, mean, rstd, dx, o0, o1, 2 * C, a); break
    switch (p.U) {
      ATEXN_FLAT_BWD(1);
      ATEXN_FLAT_BWD(2);
      ATEXN_FLAT_BWD(3);
      ATEXN_FLAT_BWD(4);
      ATEXN_FLAT_BWD(6);
      ATEXN_FLAT_BWD(8);
      default: return set_error(ATEXN_INVALID_ARGUMENT, "no kernel for %d vectors per thread", p.U);
    }
#undef ATEXN_FLAT_BWD
  } else {
    return set_error(ATEXN_INVALID_ARGUMENT, "no flat backward for vectors of %d elements", V);
  }
  ATEXN_CHECK_LAUNCH("cl_flat_bwd");
  if (N > 1) return launch_col_reduce(part, dgamma, dbeta, static_cast<int>(N), C, st);
  return ATEXN_OK;
}

#define ATEXN_INSTANTIATE_FLAT(T)                                                                                \
  template int flat_fwd_v<T, VecOf<T>::value>(const FlatPlan&, const T*, const float*, const float*, int64_t,    \
                                              int64_t, int64_t, float, T*, float*, float*, void*, hipStream_t,   \
                                              bool&);                                                            \
  template int flat_bwd_v<T, VecOf<T>::value>(const FlatPlan&, const T*, const T*, const float*, const float*,   \
                                              const float*, int64_t, int64_t, int64_t, T*, float*, float*,       \
                                              void*, hipStream_t, bool&);

}  // namespace atexn
