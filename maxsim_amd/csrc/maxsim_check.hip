// Layout checks of a call's device-resident offsets, ids and lengths, with
// the verdict written straight into pinned host memory.
#include "maxsim_host.h"
#include "maxsim_internal.h"

#include <algorithm>

namespace maxsim {

// ---------------------------------------------------------------------------
// check_layout_kernel: each workgroup checks its share of up to four index
// arrays and stores one word (system scope) into `status`: bit 0 done, bit 1
// some value is bad, bits 32.. the longest segment it saw in the first array
// if that one is CSR offsets.  The host polls the words: no device-to-host
// copies (a blit kernel, a pinned buffer and an event each), no host pass
// over the values.  Bound by one launch and one trip over the bus, behind
// which the call's own kernels are queued: the whole public call 82 -> 18 us
// for 8 queries x 16 fp32 candidates (14 us of it the scoring kernel), 80 -> 30
// for 32 x 100 fp16 ones (25 us), 116 -> 32 for the same as packed pairs, and
// 1565 us before and after for 256 x 1000, all against copies on a side
// stream and numpy checks.
// ---------------------------------------------------------------------------
constexpr int kCheckThreads = 256;
constexpr int kCheckPerThread = 8;   // values per thread from which another workgroup is taken
constexpr int kCheckMaxWgs = 128;

struct CheckArray {
  const void* p;
  int64_t n;
  int64_t limit;   // CSR: the last value; ids: below it; lengths: at most it
  int kind;        // maxsim_check_kind
  bool is64;
};
struct CheckArgs {
  CheckArray a[MAXSIM_CHECK_ARRAYS];
  int count;
  uint64_t* status;
};

__global__ __launch_bounds__(kCheckThreads) void check_layout_kernel(CheckArgs c) {
  __shared__ int any_bad, longest;
  if (threadIdx.x == 0) any_bad = longest = 0;
  __syncthreads();
  bool bad = false;
  int64_t seg = 0;
  const int64_t first = (int64_t)blockIdx.x * kCheckThreads + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * kCheckThreads;
  for (int k = 0; k < c.count; ++k) {
    const CheckArray a = c.a[k];
    auto at = [&](int64_t i) __attribute__((always_inline)) -> int64_t {
      return a.is64 ? static_cast<const int64_t*>(a.p)[i] : static_cast<const int32_t*>(a.p)[i];
    };
    if (a.kind == MAXSIM_CHECK_CSR) {
      if (a.n < 2) bad = true;
#pragma unroll 4
      for (int64_t i = first; i + 1 < a.n; i += stride) {
        const int64_t lo = at(i), hi = at(i + 1);
        bad |= hi <= lo || (i == 0 && lo != 0) || (i + 2 == a.n && hi != a.limit);
        if (k == 0) seg = max(seg, hi - lo);
      }
    } else {
      const int64_t least = a.kind == MAXSIM_CHECK_IDS ? 0 : 1;
      const int64_t most = a.kind == MAXSIM_CHECK_IDS ? a.limit - 1 : a.limit;
#pragma unroll 4
      for (int64_t i = first; i < a.n; i += stride) {
        const int64_t v = at(i);
        bad |= v < least || v > most;
      }
    }
  }
  // segments beyond 2^31 - 1 belong to arrays that are bad anyway
  const int s = (int)(seg < 0x7fffffff ? seg : 0x7fffffff);
  if (bad) any_bad = 1;
  if (s > 0) atomicMax(&longest, s);
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(c.status + blockIdx.x,
                       1ull | (any_bad ? 2ull : 0ull) | ((uint64_t)(uint32_t)longest << 32),
                       __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace maxsim

using namespace maxsim;

extern "C" {

int maxsim_internal_check_words(const maxsim_check_array* arrays, int count) {
  int64_t n = 0;
  for (int k = 0; k < count; ++k) n += arrays[k].n;
  const int64_t per = (int64_t)kCheckThreads * kCheckPerThread;
  return (int)std::min<int64_t>(std::max<int64_t>((n + per - 1) / per, 1), kCheckMaxWgs);
}

int maxsim_internal_check_layout(const maxsim_check_array* arrays, int count, uint64_t* status,
                                 void* stream) {
  clear_error();
  if (count < 1 || count > MAXSIM_CHECK_ARRAYS || !status)
    return fail(MAXSIM_ERR_INVALID, "layout check: bad arguments");
  CheckArgs c{};
  for (int k = 0; k < count; ++k) {
    if (arrays[k].n > 0 && !arrays[k].values)
      return fail(MAXSIM_ERR_INVALID, "layout check: null array");
    c.a[k] = CheckArray{arrays[k].values, arrays[k].n, arrays[k].limit, arrays[k].kind,
                        arrays[k].is64 != 0};
  }
  c.count = count;
  c.status = status;
  const int wgs = maxsim_internal_check_words(arrays, count);
  hipLaunchKernelGGL(check_layout_kernel, dim3((unsigned)wgs), dim3(kCheckThreads), 0,
                     static_cast<hipStream_t>(stream), c);
  return check_launch("check_layout_kernel");
}

}  // extern "C"
