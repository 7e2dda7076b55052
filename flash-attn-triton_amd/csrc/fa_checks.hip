// fa_check_ranges: the range checks on device integer arrays that a call
// validates its arguments with (cache lengths, page tables, cache rows, left
// pads), reduced in one launch.
//
// Workgroup i reduces array i (plus an optional elementwise addend, or as the
// differences of adjacent elements) to its minimum and maximum as int64 and
// writes them to minmax[2i], minmax[2i + 1].
// minmax may be pinned host memory, so the host reads the results after an
// event on the stream without a separate device-to-host copy.
//
// fa_check_bounds is the form the Python layer uses: each workgroup also
// compares its range with bounds and writes a flag that later launches on the
// stream can be guarded with (they read nothing else when it is set), and
// marks its results done, so that fa_check_wait can poll pinned memory instead
// of recording and waiting for an event.  On one MI355X a torch event recorded
// and waited for behind the launch took 13 us of host time, its wait on a
// second stream 16 us; a one-token decode call went from 103 to 45 us, an
// append + rotary call from 258 to 82 us.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <sched.h>

#include "fa_api_internal.h"
#include "fa_gfx950.h"

namespace {

constexpr int kThreads = 256;

struct RangeJob {
  const void* a;   // int32 or int64 elements
  const void* b;   // nullable addend, int32 or int64
  int64_t n;       // values reduced: numel, or numel - 1 for differences
  int a_wide, b_wide, diff;
  int64_t lo, hi;  // fa_check_bounds
};

struct RangeJobs {
  RangeJob job[FA_MAX_RANGE_CHECKS];
  int64_t* minmax;   // {min, max} per array; with `done`, {min, max, done}
  int* guard;        // nullable: 1 where the range leaves [lo, hi], else 0
  int done;
};

__device__ inline int64_t load_int(const void* p, int wide, int64_t i) {
  return wide ? static_cast<const int64_t*>(p)[i]
              : static_cast<int64_t>(static_cast<const int32_t*>(p)[i]);
}

__global__ __launch_bounds__(kThreads) void range_minmax_kernel(RangeJobs jobs) {
  const RangeJob j = jobs.job[blockIdx.x];
  int64_t lo = INT64_MAX, hi = INT64_MIN;
  for (int64_t i = threadIdx.x; i < j.n; i += kThreads) {
    int64_t x = load_int(j.a, j.a_wide, i + (j.diff ? 1 : 0));
    if (j.diff)
      x -= load_int(j.a, j.a_wide, i);
    else if (j.b)
      x += load_int(j.b, j.b_wide, i);
    lo = x < lo ? x : lo;
    hi = x > hi ? x : hi;
  }
  for (int off = 32; off > 0; off >>= 1) {
    const int64_t ol = __shfl_xor(lo, off);
    const int64_t oh = __shfl_xor(hi, off);
    lo = ol < lo ? ol : lo;
    hi = oh > hi ? oh : hi;
  }
  __shared__ int64_t s_lo[kThreads / 64], s_hi[kThreads / 64];
  if ((threadIdx.x & 63) == 0) {
    s_lo[threadIdx.x >> 6] = lo;
    s_hi[threadIdx.x >> 6] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; ++w) {
      lo = s_lo[w] < lo ? s_lo[w] : lo;
      hi = s_hi[w] > hi ? s_hi[w] : hi;
    }
    const int i = blockIdx.x;
    if (jobs.guard) jobs.guard[i] = lo < j.lo || hi > j.hi;
    if (jobs.done) {
      // The results and, once those stores have completed, the mark, all
      // written through to host memory (system scope).  A release store would
      // also write back the XCD's whole L2, under an attention kernel that runs
      // beside this one.
      auto put = [&](int k, int64_t x) {
        __hip_atomic_store(jobs.minmax + 3 * i + k, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      };
      put(0, lo);
      put(1, hi);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      put(2, 1);
    } else {
      jobs.minmax[2 * i] = lo;
      jobs.minmax[2 * i + 1] = hi;
    }
  }
}

int run_checks(int n, const void* const* a, const int* a_bytes, const void* const* b,
               const int* b_bytes, const int* diff, const int64_t* numel, const int64_t* lo,
               const int64_t* hi, int64_t* minmax, int32_t* guard, bool done, hipStream_t stream) {
  if (n < 1 || n > FA_MAX_RANGE_CHECKS)
    return fa_set_error(FA_ERR_INVALID, "fa_check_ranges: n must be in [1, FA_MAX_RANGE_CHECKS]");
  if (!a || !a_bytes || !numel || !minmax)
    return fa_set_error(FA_ERR_INVALID, "fa_check_ranges: null pointer argument");
  if (reinterpret_cast<uintptr_t>(minmax) % 8 != 0)
    return fa_set_error(FA_ERR_INVALID, "fa_check_ranges: minmax must be 8-byte aligned");
  RangeJobs jobs{};
  for (int i = 0; i < n; ++i) {
    const bool dif = diff && diff[i];
    const bool has_b = !dif && b && b[i];
    if (!a[i] || numel[i] < 0 || (a_bytes[i] != 4 && a_bytes[i] != 8) ||
        (has_b && (!b_bytes || (b_bytes[i] != 4 && b_bytes[i] != 8))))
      return fa_set_error(FA_ERR_INVALID,
                          "fa_check_ranges: each array needs a pointer, a size >= 0 and 4- or "
                          "8-byte elements");
    jobs.job[i] = RangeJob{a[i], has_b ? b[i] : nullptr,
                           dif ? (numel[i] > 0 ? numel[i] - 1 : 0) : numel[i], a_bytes[i] == 8,
                           has_b && b_bytes[i] == 8, dif ? 1 : 0, lo ? lo[i] : INT64_MIN,
                           hi ? hi[i] : INT64_MAX};
  }
  // The results go to device memory or to pinned host memory, through the
  // address the device sees; pageable host memory would fault the kernel.
  hipPointerAttribute_t attr{};
  void* dst = minmax;
  hipError_t e = hipPointerGetAttributes(&attr, minmax);
  if (e == hipSuccess && attr.type == hipMemoryTypeHost)
    e = hipHostGetDevicePointer(&dst, minmax, 0);
  else if (e == hipSuccess && (done || attr.type != hipMemoryTypeDevice))
    e = hipErrorInvalidValue;
  if (e != hipSuccess || dst == nullptr) {
    (void)hipGetLastError();
    return fa_set_error(FA_ERR_INVALID,
                        "fa_check_ranges: minmax must be device memory or pinned host memory");
  }
  jobs.minmax = static_cast<int64_t*>(dst);
  jobs.guard = guard;
  jobs.done = done;
  if (done)
    for (int i = 0; i < n; ++i)
      __atomic_store_n(minmax + 3 * i + 2, (int64_t)0, __ATOMIC_RELEASE);
  hipLaunchKernelGGL(range_minmax_kernel, dim3(n), dim3(kThreads), 0, stream, jobs);
  e = hipGetLastError();
  if (e != hipSuccess) return fa_set_error(FA_ERR_HIP, hipGetErrorString(e));
  fa_set_error(FA_OK, "");
  return FA_OK;
}

}  // namespace

extern "C" int fa_check_ranges(int n, const void* const* a, const int* a_bytes,
                               const void* const* b, const int* b_bytes, const int* diff,
                               const int64_t* numel, int64_t* minmax, fa_stream_t stream) {
  return run_checks(n, a, a_bytes, b, b_bytes, diff, numel, nullptr, nullptr, minmax, nullptr,
                    false, (hipStream_t)stream);
}

extern "C" int fa_check_bounds(int n, const void* const* a, const int* a_bytes,
                               const void* const* b, const int* b_bytes, const int* diff,
                               const int64_t* numel, const int64_t* lo, const int64_t* hi,
                               int64_t* result, int32_t* guard, fa_stream_t stream) {
  if (!lo || !hi) return fa_set_error(FA_ERR_INVALID, "fa_check_bounds: null pointer argument");
  // The caller waits for the results, which a captured launch never writes.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &cap) != hipSuccess) (void)hipGetLastError();
  if (cap != hipStreamCaptureStatusNone)
    return fa_set_error(FA_ERR_UNSUPPORTED,
                        "fa_check_bounds: argument checks need a host wait and cannot be captured");
  return run_checks(n, a, a_bytes, b, b_bytes, diff, numel, lo, hi, result, guard, true,
                    (hipStream_t)stream);
}

extern "C" int fa_check_wait(const int64_t* result, int n, fa_stream_t stream) {
  if (!result || n < 0) return fa_set_error(FA_ERR_INVALID, "fa_check_wait: bad argument");
  int i = 0;
  auto advance = [&]() {
    while (i < n && __atomic_load_n(result + 3 * i + 2, __ATOMIC_ACQUIRE) != 0) ++i;
    return i == n;
  };
  for (unsigned spins = 1; !advance(); ++spins) {
    if (spins % 1024 != 0) {
      __builtin_ia32_pause();
      continue;
    }
    // Long waits: let other threads run, and every few ms end if the stream has
    // failed or has drained without the results (rarely: a query may put a
    // marker on the stream).
    sched_yield();
    if (spins % 65536 != 0) continue;
    const hipError_t e = hipStreamQuery((hipStream_t)stream);
    if (e == hipErrorNotReady) {
      (void)hipGetLastError();
      continue;
    }
    if (e != hipSuccess) return fa_set_error(FA_ERR_HIP, hipGetErrorString(e));
    if (!advance())
      return fa_set_error(FA_ERR_HIP, "fa_check_wait: the stream drained without the results");
    break;
  }
  fa_set_error(FA_OK, "");
  return FA_OK;
}
