// Error reporting shared by every translation unit of libatex_norms_hip.so.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/atex_norms.h"

namespace atexn {

// Records a printf-style message for atexn_last_error() of this thread; returns `code`.
int set_error(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
const char* last_error();

// Number of compute units of the current device (256 on MI355X); 256 if no device can be
// queried, so that the workspace queries stay usable on a host without a GPU.
int cu_count();

// A tag that no earlier call of this process has used (odd, so never 0): kernels whose workgroups
// exchange partial results mark them with it, so that whatever an earlier call left in the caller's
// workspace is never taken for data of this one.  A process-wide atomic counter, started from the clock.
unsigned next_call_tag();

// Whether a call on stream `st` may take the InstanceNorm kernels whose workgroups exchange partial
// results under a tag from the host.  Not while the stream is being captured (a graph replay would
// repeat the call's tag; LayerNorm's long rows, ragged planes and flat and held channels-last instances take
// theirs from exchange_tag below and are recorded as they are), and neither these nor those in a process started with ATEXN_NO_EXCHANGE set
// to anything but "0": such kernels need the workgroups of one instance / plane on the chip together, which a process that
// keeps other kernels resident on the same GPU (communication kernels overlapped with compute)
// may never give them; every wait then runs out and every workgroup recomputes its peers' share.
// The results are the same; the time is not.  The variable is read once, at the first call.
bool exchange_allowed(void* st);

// The current device's word for exchange_wait_pair (norm_common.hip.h): a static
// device variable of the library, looked up once per device.  nullptr if that fails (the kernels
// then always wait patiently).
unsigned* exchange_trouble_word();

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

#define ATEXN_REQUIRE(cond, ...)                                                  \
  do {                                                                            \
    if (!(cond)) return ::atexn::set_error(ATEXN_INVALID_ARGUMENT, __VA_ARGS__);  \
  } while (0)

#define ATEXN_TRY(expr)             \
  do {                              \
    const int rc_ = (expr);         \
    if (rc_ != ATEXN_OK) return rc_; \
  } while (0)

#define ATEXN_CHECK_LAUNCH(what)                                                           \
  do {                                                                                     \
    hipError_t e_ = hipGetLastError();                                                     \
    if (e_ != hipSuccess)                                                                  \
      return ::atexn::set_error(ATEXN_LAUNCH_ERROR, "%s: %s", what, hipGetErrorString(e_)); \
  } while (0)

// The tag of a launch whose workgroups exchange results.  ok: the launch may (not in a process with
// ATEXN_NO_EXCHANGE).  On an ordinary stream `tag` is next_call_tag() and `at` null.  A stream that
// is being captured gets no number of its own, since every replay would repeat it: a one-thread
// kernel is recorded ahead of the launch that takes the next number of a device-wide counter and
// leaves it at `word` (device memory, 4 bytes, part of the caller's workspace), and the launch reads
// its tag there (`at`).  Host tags are odd, recorded ones even and not 0 (call_tag.h).  Eager calls and replays thus run the
// same kernels, to the same bits.
struct ExchangeTag {
  bool ok = false;
  unsigned tag = 0;
  const unsigned* at = nullptr;
  unsigned* trouble = nullptr;  // see exchange_trouble_word; the ages it holds are those of eager calls
};
int exchange_tag(hipStream_t st, void* word, ExchangeTag& out);

// Flat entry points used by the C ABI (dtype already validated).
size_t rows_fwd_ws(int dtype, bool affine, int64_t n_rows, int64_t D, int C);
size_t rows_bwd_ws(int dtype, bool affine, int64_t n_rows, int64_t D, int C);
int rows_fwd(int dtype, bool affine, const void* x, const float* gamma, const float* beta,
             int64_t n_rows, int64_t D, int C, float eps, void* y, float* mean, float* rstd,
             void* ws, size_t ws_bytes, hipStream_t st);
int rows_bwd(int dtype, bool affine, const void* dy, const void* x, const float* gamma,
             const float* mean, const float* rstd, int64_t n_rows, int64_t D, int C, void* dx,
             float* dgamma, float* dbeta, void* ws, size_t ws_bytes, hipStream_t st);

size_t cl_fwd_ws(int dtype, int64_t N, int64_t C, int64_t D);
size_t cl_bwd_ws(int dtype, int64_t N, int64_t C, int64_t D);
int cl_fwd(int dtype, const void* x, const float* gamma, const float* beta, int64_t N, int64_t C,
           int64_t D, float eps, void* y, float* mean, float* rstd, void* ws, size_t ws_bytes,
           hipStream_t st);
int cl_bwd(int dtype, const void* dy, const void* x, const float* gamma, const float* mean,
           const float* rstd, int64_t N, int64_t C, int64_t D, void* dx, float* dgamma,
           float* dbeta, void* ws, size_t ws_bytes, hipStream_t st);

// out[0..n) = 0 on the stream (a kernel, so that callers may capture it in a HIP graph).
int fill_zero(float* out, int64_t n, hipStream_t st);

// Launches the deterministic column reduction out0[j] = sum_g part[g][0][j],
// out1[j] = sum_g part[g][1][j], j < W; `batch` independent problems at the given strides
// (in floats) in one launch.
int launch_col_reduce(const float* part, float* out0, float* out1, int G, int64_t W,
                      hipStream_t st, int batch = 1, int64_t part_stride = 0,
                      int64_t out_stride = 0);
// The same, summed in double.
int launch_col_reduce_double(const float* part, float* out0, float* out1, int G, int64_t W, hipStream_t st);

inline int elem_size(int dtype) { return dtype == ATEXN_F32 ? 4 : 2; }

}  // namespace atexn
