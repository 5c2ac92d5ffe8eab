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
constexpr int kCheckUnroll = 4;      // values in flight per thread
constexpr int kCheckMaxWgs = 128;

struct CheckArray {
  const void* p;
  int64_t n;
  int64_t limit;   // CSR: the last value; ids: below it; lengths: at most it
  int first_wg;    // its workgroups: first_wg .. the next array's
  int kind;        // maxsim_check_kind
  bool is64;
};
struct CheckArgs {
  CheckArray a[MAXSIM_CHECK_ARRAYS];
  int count;
  int64_t per_wg;  // values per workgroup, a multiple of kCheckThreads * kCheckUnroll
  uint64_t* status;
};

// A workgroup checks a run of one array, kCheckUnroll loads in flight per
// thread (clamped, so that no branch keeps one waiting for another): 57,000
// values of four arrays 5.7 us, 8.8 when every thread went through all of them.
template <typename I>
__device__ __forceinline__ bool check_run(const CheckArray& a, int64_t lo, int64_t hi,
                                          int64_t& longest) {
  const I* v = static_cast<const I*>(a.p);
  bool bad = false;
  if (a.kind == MAXSIM_CHECK_CSR) {
    // pair i: values i and i + 1
    for (int64_t i0 = lo + threadIdx.x; i0 < hi; i0 += kCheckThreads * kCheckUnroll) {
      int64_t x[kCheckUnroll], y[kCheckUnroll];
#pragma unroll
      for (int u = 0; u < kCheckUnroll; ++u) {
        const int64_t i = min(i0 + u * kCheckThreads, hi - 1);
        x[u] = v[i];
        y[u] = v[i + 1];
      }
#pragma unroll
      for (int u = 0; u < kCheckUnroll; ++u) {
        const int64_t i = min(i0 + u * kCheckThreads, hi - 1);
        bad |= y[u] <= x[u] || (i == 0 && x[u] != 0) || (i + 2 == a.n && y[u] != a.limit);
        longest = max(longest, y[u] - x[u]);
      }
    }
  } else {
    const int64_t least = a.kind == MAXSIM_CHECK_IDS ? 0 : 1;
    const int64_t most = a.kind == MAXSIM_CHECK_IDS ? a.limit - 1 : a.limit;
    for (int64_t i0 = lo + threadIdx.x; i0 < hi; i0 += kCheckThreads * kCheckUnroll) {
      int64_t x[kCheckUnroll];
#pragma unroll
      for (int u = 0; u < kCheckUnroll; ++u) x[u] = v[min(i0 + u * kCheckThreads, hi - 1)];
#pragma unroll
      for (int u = 0; u < kCheckUnroll; ++u) bad |= x[u] < least || x[u] > most;
    }
  }
  return bad;
}

__global__ __launch_bounds__(kCheckThreads) void check_layout_kernel(CheckArgs c) {
  __shared__ int any_bad, longest;
  if (threadIdx.x == 0) any_bad = longest = 0;
  __syncthreads();
  int k = 0;
  while (k + 1 < c.count && (int)blockIdx.x >= c.a[k + 1].first_wg) ++k;
  const CheckArray a = c.a[k];
  // entries: pairs of neighbours for CSR offsets, values otherwise
  const int64_t n = a.kind == MAXSIM_CHECK_CSR ? a.n - 1 : a.n;
  const int64_t lo = (int64_t)((int)blockIdx.x - a.first_wg) * c.per_wg;
  const int64_t hi = min(lo + c.per_wg, n);
  int64_t seg = 0;
  bool bad = a.kind == MAXSIM_CHECK_CSR && a.n < 2;
  if (lo < hi)
    bad |= a.is64 ? check_run<int64_t>(a, lo, hi, seg) : check_run<int32_t>(a, lo, hi, seg);
  // segments beyond 2^31 - 1 belong to arrays that are bad anyway
  const int s = k == 0 ? (int)(seg < 0x7fffffff ? seg : 0x7fffffff) : 0;
  if (bad) any_bad = 1;
  if (s > 0) atomicMax(&longest, s);
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(c.status + blockIdx.x,
                       1ull | (any_bad ? 2ull : 0ull) | ((uint64_t)(uint32_t)longest << 32),
                       __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Workgroups of each array (at least one) at `per_wg` values each.
static int array_wgs(int64_t n, int64_t per_wg) {
  return (int)std::max<int64_t>((n + per_wg - 1) / per_wg, 1);
}
static int64_t values_per_wg(const maxsim_check_array* arrays, int count, int* wgs) {
  for (int64_t per = kCheckThreads * kCheckUnroll;; per *= 2) {
    int64_t all = 0;
    for (int k = 0; k < count; ++k) all += (arrays[k].n + per - 1) / per + 1;
    if (all <= kCheckMaxWgs) {
      *wgs = 0;
      for (int k = 0; k < count; ++k) *wgs += array_wgs(arrays[k].n, per);
      return per;
    }
  }
}

}  // namespace maxsim

using namespace maxsim;

extern "C" {

int maxsim_internal_check_words(const maxsim_check_array* arrays, int count) {
  int wgs = 0;
  values_per_wg(arrays, count, &wgs);
  return wgs;
}

int maxsim_internal_check_layout(const maxsim_check_array* arrays, int count, uint64_t* status,
                                 void* stream) {
  clear_error();
  if (count < 1 || count > MAXSIM_CHECK_ARRAYS || !status)
    return fail(MAXSIM_ERR_INVALID, "layout check: bad arguments");
  CheckArgs c{};
  int wgs = 0;
  c.per_wg = values_per_wg(arrays, count, &wgs);
  int first = 0;
  for (int k = 0; k < count; ++k) {
    if (arrays[k].n > 0 && !arrays[k].values)
      return fail(MAXSIM_ERR_INVALID, "layout check: null array");
    c.a[k] = CheckArray{arrays[k].values, arrays[k].n, arrays[k].limit, first, arrays[k].kind,
                        arrays[k].is64 != 0};
    first += array_wgs(arrays[k].n, c.per_wg);
  }
  c.count = count;
  c.status = status;
  hipLaunchKernelGGL(check_layout_kernel, dim3((unsigned)wgs), dim3(kCheckThreads), 0,
                     static_cast<hipStream_t>(stream), c);
  return check_launch("check_layout_kernel");
}

}  // extern "C"
