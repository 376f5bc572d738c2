// validate.hip -- the device half of the validation: one launch reduces the
// lengths, offsets and used page-table entries that a call is to check
// (flashattn_tile/paging.py:84-130 validate_cache, as called by
// flashattn_tile/kernels/decode.py:503-522, and kernels/prefill.py:194-233)
// to a few numbers, instead of a dozen framework reductions.
//
// fat_check_begin / fat_check_wait: what the Python package runs.  The kernel
// writes its numbers into page-locked host memory and the host polls them, so
// a validated call neither copies nor synchronises.
//
// fat_cache_stats: the same numbers of a paged cache in device memory, for
// callers of the C library that have no page-locked words or copy them with
// other results.
#include <limits.h>

#include <algorithm>
#include <atomic>
#include <chrono>

#include "fat_common.h"

namespace fat {

constexpr int kStatsThreads = 1024;

// out[0..4] = min(seq_lens), max(seq_lens), min and max of page_table[b, c]
// over every row b and column c < min(ceil(max_len / P), max_pages) (INT_MAX
// and INT_MIN when no entry is used), sum_b ceil(max(seq_lens[b], 0) / P).
__global__ __launch_bounds__(kStatsThreads) void cache_stats_kernel(const int32_t* __restrict__ lens,
                                                                    const int32_t* __restrict__ pt, int B,
                                                                    int max_pages, int64_t pt_sb, int P,
                                                                    int64_t* __restrict__ out) {
  __shared__ int s_min[kStatsThreads / 64], s_max[kStatsThreads / 64];
  __shared__ long long s_sum[kStatsThreads / 64];
  __shared__ int s_need;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  int mn = INT_MAX, mx = INT_MIN;
  long long pages = 0;
  for (int b = tid; b < B; b += kStatsThreads) {
    const int l = lens[b];
    mn = min(mn, l);
    mx = max(mx, l);
    pages += (max(l, 0) + (long long)P - 1) / P;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mn = min(mn, __shfl_xor(mn, off));
    mx = max(mx, __shfl_xor(mx, off));
    pages += __shfl_xor(pages, off);
  }
  if (lane == 0) {
    s_min[w] = mn;
    s_max[w] = mx;
    s_sum[w] = pages;
  }
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < kStatsThreads / 64; ++i) {
      mn = min(mn, s_min[i]);
      mx = max(mx, s_max[i]);
      pages += s_sum[i];
    }
    out[0] = mn;
    out[1] = mx;
    out[4] = pages;
    // Columns the longest sequence uses (as the torch restatement: floor((max + P - 1) / P)).
    const long long need = mx > 0 ? ((long long)mx + P - 1) / P : 0;
    s_need = (int)min(need, (long long)max_pages);
  }
  __syncthreads();
  const int need = s_need;
  int pmn = INT_MAX, pmx = INT_MIN;
  const long long n = (long long)B * need;
  for (long long i = tid; i < n; i += kStatsThreads) {
    const int b = (int)(i / need);
    const int c = (int)(i - (long long)b * need);
    const int v = pt[b * pt_sb + c];
    pmn = min(pmn, v);
    pmx = max(pmx, v);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    pmn = min(pmn, __shfl_xor(pmn, off));
    pmx = max(pmx, __shfl_xor(pmx, off));
  }
  __syncthreads();  // s_min / s_max are reused
  if (lane == 0) {
    s_min[w] = pmn;
    s_max[w] = pmx;
  }
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < kStatsThreads / 64; ++i) {
      pmn = min(pmn, s_min[i]);
      pmx = max(pmx, s_max[i]);
    }
    out[2] = pmn;
    out[3] = pmx;
  }
}

constexpr int kCheckThreads = 256;
// Table entries per workgroup.  One workgroup of 1024 threads took 27.8 us
// for a table of 64 sequences of up to 1000 pages; 16 workgroups of 256 take
// 8.5 us, of which the lengths, the launch and the writes to the host are 4.3.
constexpr int64_t kCheckEntries = 4096;

struct CheckParams {
  const int32_t* cu_q;
  const int32_t* cu_k;
  const int32_t* lens;
  const int32_t* pt;
  int64_t pt_sb;
  int64_t* host;
  int64_t ticket;
  int32_t B, max_pages, P;
  const float* values;
  int64_t count;
};

struct RMin { template <typename T> static __device__ __forceinline__ T f(T a, T b) { return a < b ? a : b; } };
struct RMax { template <typename T> static __device__ __forceinline__ T f(T a, T b) { return a > b ? a : b; } };
struct RSum { template <typename T> static __device__ __forceinline__ T f(T a, T b) { return a + b; } };
struct ROr { template <typename T> static __device__ __forceinline__ T f(T a, T b) { return a | b; } };

// Reduction over the workgroup; every thread gets the result.
template <typename Op>
__device__ __forceinline__ long long check_reduce(long long x) {
  __shared__ long long s[kCheckThreads / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x = Op::f(x, __shfl_xor(x, off));
  __syncthreads();  // the previous reduction's reads are done
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = x;
  __syncthreads();
  x = s[0];
#pragma unroll
  for (int i = 1; i < kCheckThreads / 64; ++i) x = Op::f(x, s[i]);
  return x;
}

// Latency-bound: a few dependent loads, then a PCIe write per workgroup.  The
// stores are system-scope (written through to host memory) and each
// workgroup's ticket follows its results once they are complete (vmcnt(0)),
// so no cache is written back and the host needs no synchronisation.
template <int KIND>
__global__ __launch_bounds__(kCheckThreads) void check_kernel(const CheckParams p) {
  constexpr bool LENS = KIND == FAT_CHECK_CACHE || KIND == FAT_CHECK_PAGED || KIND == FAT_CHECK_APPEND;
  constexpr bool CU = KIND == FAT_CHECK_VARLEN || KIND == FAT_CHECK_PAGED;
  constexpr bool TABLE = KIND == FAT_CHECK_CACHE || KIND == FAT_CHECK_PAGED;
  const int tid = threadIdx.x;
  auto put = [&](int word, long long v) {
    __hip_atomic_store(p.host + word, (int64_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  };
  long long mn = INT_MAX, mx = INT_MIN, pages = 0, flags = 0, mq = INT_MIN, mk = INT_MIN, keyless = INT_MAX;
  int pmn = INT_MAX, pmx = INT_MIN;
  for (int b = tid; b < p.B; b += kCheckThreads) {
    long long len = 0, lq = 0, lk = 0;
    if constexpr (LENS) {
      len = p.lens[b];
      mn = min(mn, len);
      mx = max(mx, len);
      pages += (max(len, 0ll) + p.P - 1) / p.P;
      lk = len;
    }
    if constexpr (CU) {
      lq = (long long)p.cu_q[b + 1] - p.cu_q[b];
      if constexpr (KIND == FAT_CHECK_VARLEN) lk = (long long)p.cu_k[b + 1] - p.cu_k[b];
      flags |= (lq < 0 ? 1 : 0) | (KIND == FAT_CHECK_VARLEN && lk < 0 ? 2 : 0) | (lk < lq ? 4 : 0);
      mq = max(mq, lq);
      mk = max(mk, lk);
      // a packed sequence without keys, a cached one without tokens
      if (lq > 0 && (KIND == FAT_CHECK_VARLEN ? lk == 0 : lk <= 0)) keyless = min(keyless, (long long)b);
    }
    if constexpr (KIND == FAT_CHECK_APPEND) {
      const int block = len < 0 ? 0 : (int)min(len / p.P, (long long)p.max_pages - 1);
      const int id = p.pt[b * p.pt_sb + block];
      pmn = min(pmn, id);
      pmx = max(pmx, id);
    }
  }
  if constexpr (KIND == FAT_CHECK_RANGE) {
    // Order-preserving integers, so that the reductions below apply; a NaN is
    // tracked apart (bit 0 of flags).
    const int64_t step = (int64_t)gridDim.x * kCheckThreads;
#pragma unroll 4
    for (int64_t i = (int64_t)blockIdx.x * kCheckThreads + tid; i < p.count; i += step) {
      const float v = p.values[i];
      const int bits = __builtin_bit_cast(int, v);
      const int key = bits ^ ((bits >> 31) & 0x7fffffff);
      pmn = min(pmn, key);
      pmx = max(pmx, key);
      flags |= v != v ? 1 : 0;
    }
    pmn = (int)check_reduce<RMin>(pmn);
    pmx = (int)check_reduce<RMax>(pmx);
    const bool nan = check_reduce<ROr>(flags) != 0;
    pmn = nan ? INT_MIN : pmn;  // no float's key: the host sees a NaN
    pmx = nan ? INT_MAX : pmx;
  }
  if constexpr (LENS) mx = check_reduce<RMax>(mx);
  if constexpr (TABLE) {
    const long long need = mx > 0 ? min((mx + p.P - 1) / p.P, (long long)p.max_pages) : 0;
    const long long n = (long long)p.B * need;
    const uint32_t cols = (uint32_t)need;
    const long long step = (long long)gridDim.x * kCheckThreads;
#pragma unroll 4
    for (long long i = (long long)blockIdx.x * kCheckThreads + tid; i < n; i += step) {
      const long long b = n <= 0xffffffffll ? (long long)((uint32_t)i / cols) : i / need;
      const int id = p.pt[b * p.pt_sb + (i - b * need)];
      pmn = min(pmn, id);
      pmx = max(pmx, id);
    }
  }
  if constexpr (TABLE || KIND == FAT_CHECK_APPEND) {
    pmn = (int)check_reduce<RMin>(pmn);
    pmx = (int)check_reduce<RMax>(pmx);
  }
  if (blockIdx.x == 0) {  // uniform
    if constexpr (LENS) {
      mn = check_reduce<RMin>(mn);
      pages = check_reduce<RSum>(pages);
    }
    if constexpr (CU) {
      flags = check_reduce<ROr>(flags);
      mq = check_reduce<RMax>(mq);
      mk = check_reduce<RMax>(mk);
      keyless = check_reduce<RMin>(keyless);
    }
    if (tid == 0) {
      put(0, mn);
      put(1, mx);
      put(2, pages);
      if constexpr (CU) {
        put(3, p.cu_q[0]);
        put(4, p.cu_q[p.B]);
        if constexpr (KIND == FAT_CHECK_VARLEN) {
          put(5, p.cu_k[0]);
          put(6, p.cu_k[p.B]);
        }
        put(7, flags);
        put(8, mq);
        put(9, mk);
        const bool any = keyless != INT_MAX;
        put(10, any ? keyless : -1);
        put(11, any ? (long long)p.cu_q[keyless + 1] - p.cu_q[keyless] : 0);
      }
    }
  }
  if (tid == 0) {
    const int at = FAT_CHECK_RESULTS + 2 * blockIdx.x;
    put(at, (long long)(((unsigned long long)(uint32_t)pmx << 32) | (uint32_t)pmn));
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the results are complete
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    put(at + 1, p.ticket);
  }
}

}  // namespace fat

namespace {

int check_groups(const fat_check_args* a) {
  if (a->kind == FAT_CHECK_VARLEN || a->kind == FAT_CHECK_APPEND) return 1;
  const int64_t entries = a->kind == FAT_CHECK_RANGE ? a->count : (int64_t)a->batch * a->max_pages;
  const int64_t n = (entries + fat::kCheckEntries - 1) / fat::kCheckEntries;
  return (int)std::min<int64_t>(std::max<int64_t>(n, 1), FAT_CHECK_MAX_GROUPS);
}

bool check_args_ok(const fat_check_args* a, const char* who) {
  const bool cu = a && (a->kind == FAT_CHECK_VARLEN || a->kind == FAT_CHECK_PAGED);
  const bool range = a && a->kind == FAT_CHECK_RANGE;
  const bool lens = a && a->kind != FAT_CHECK_VARLEN && !range;
  if (!a || !a->host || (cu && !a->cu_q) || (a->kind == FAT_CHECK_VARLEN && !a->cu_k) || (lens && !a->seq_lens) ||
      (lens && !a->page_table) || (range && !a->values)) {
    fat_host::set_error("%s: a required pointer is NULL", who);
    return false;
  }
  if (a->kind < FAT_CHECK_CACHE || a->kind > FAT_CHECK_RANGE || (!range && a->batch <= 0) ||
      a->ticket <= 0 || (range && a->count <= 0) ||
      (lens && (a->max_pages <= 0 || a->page_size <= 0 || a->page_table_stride < 0)) ||
      (a->kind == FAT_CHECK_CACHE && a->page_table_stride < a->max_pages)) {
    fat_host::set_error("%s: kind %d, batch %d, ticket %lld, max_pages %d, page_size %d or page_table_stride %lld "
                        "invalid", who, a->kind, a->batch, (long long)a->ticket, a->max_pages, a->page_size,
                        (long long)a->page_table_stride);
    return false;
  }
  return true;
}

}  // namespace

extern "C" int fat_check_begin(const fat_check_args* a, void* stream_ptr) {
  fat_host::clear_error();
  if (!check_args_ok(a, "fat_check_begin")) return FAT_E_INVALID;
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(stream, &cap);
  if (e != hipSuccess || cap != hipStreamCaptureStatusNone) {
    if (e != hipSuccess) (void)hipGetLastError();
    fat_host::set_error("fat_check_begin: the stream is capturing: a validated call waits for the GPU (use the "
                        "launch functions below the validation under capture)");
    return FAT_E_LAUNCH;
  }
  const fat::CheckParams prm{a->cu_q, a->cu_k, a->seq_lens, a->page_table, a->page_table_stride, a->host,
                             a->ticket, a->batch, a->max_pages, a->page_size, a->values, a->count};
  const dim3 grid((unsigned)check_groups(a)), block(fat::kCheckThreads);
  switch (a->kind) {
    case FAT_CHECK_CACHE: hipLaunchKernelGGL((fat::check_kernel<FAT_CHECK_CACHE>), grid, block, 0, stream, prm); break;
    case FAT_CHECK_VARLEN: hipLaunchKernelGGL((fat::check_kernel<FAT_CHECK_VARLEN>), grid, block, 0, stream, prm); break;
    case FAT_CHECK_PAGED: hipLaunchKernelGGL((fat::check_kernel<FAT_CHECK_PAGED>), grid, block, 0, stream, prm); break;
    case FAT_CHECK_RANGE: hipLaunchKernelGGL((fat::check_kernel<FAT_CHECK_RANGE>), grid, block, 0, stream, prm); break;
    default: hipLaunchKernelGGL((fat::check_kernel<FAT_CHECK_APPEND>), grid, block, 0, stream, prm); break;
  }
  return fat_host::launch_status("check_kernel");
}

extern "C" int fat_check_wait(const fat_check_args* a, void* stream_ptr, int64_t* result) {
  fat_host::clear_error();
  if (!check_args_ok(a, "fat_check_wait")) return FAT_E_INVALID;
  if (!result) {
    fat_host::set_error("fat_check_wait: result is NULL");
    return FAT_E_INVALID;
  }
  const int n = check_groups(a);
  // Tickets arrive in any order; `done` are known to be here.
  int done = 0;
  auto arrived = [&] {
    while (done < n && __atomic_load_n(a->host + FAT_CHECK_RESULTS + 2 * done + 1, __ATOMIC_ACQUIRE) == a->ticket)
      ++done;
    return done == n;
  };
  const auto limit = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
  bool here = arrived();
  for (int spin = 1; !here; ++spin) {
    __builtin_ia32_pause();
    here = arrived();
    if (!here && (spin & 255) == 0 && std::chrono::steady_clock::now() > limit) break;
  }
  if (!here) {
    const hipError_t e = hipStreamSynchronize(static_cast<hipStream_t>(stream_ptr));
    if (e != hipSuccess) {
      (void)hipGetLastError();
      fat_host::set_error("fat_check_wait: the stream failed: %s", hipGetErrorString(e));
      return FAT_E_LAUNCH;
    }
    if (!arrived()) {
      fat_host::set_error("fat_check_wait: no result for ticket %lld (was it begun on this stream?)",
                          (long long)a->ticket);
      return FAT_E_INVALID;
    }
  }
  for (int i = 0; i < 12; ++i) result[i] = a->host[i];
  int32_t lo = INT_MAX, hi = INT_MIN;
  for (int i = 0; i < n; ++i) {
    const uint64_t w = (uint64_t)a->host[FAT_CHECK_RESULTS + 2 * i];
    lo = std::min(lo, (int32_t)(uint32_t)w);
    hi = std::max(hi, (int32_t)(uint32_t)(w >> 32));
  }
  if (a->kind == FAT_CHECK_RANGE) {
    const bool nan = lo == INT_MIN && hi == INT_MAX;
    lo = nan ? 0x7fc00000 : lo ^ ((lo >> 31) & 0x7fffffff);
    hi = nan ? 0x7fc00000 : hi ^ ((hi >> 31) & 0x7fffffff);
  }
  result[12] = lo;
  result[13] = hi;
  result[14] = result[15] = 0;
  return FAT_OK;
}

extern "C" int fat_cache_stats(const fat_cache_stats_args* a, void* stream_ptr) {
  fat_host::clear_error();
  if (!a || !a->seq_lens || !a->out || (a->batch > 0 && a->max_pages > 0 && !a->page_table)) {
    fat_host::set_error("fat_cache_stats: a required pointer is NULL");
    return FAT_E_INVALID;
  }
  if (a->batch < 0 || a->max_pages < 0 || a->page_size <= 0 || (a->max_pages > 0 && a->page_table_stride < a->max_pages)) {
    fat_host::set_error("fat_cache_stats: batch %d, max_pages %d, page_size %d or page_table_stride %lld invalid",
                        a->batch, a->max_pages, a->page_size, (long long)a->page_table_stride);
    return FAT_E_INVALID;
  }
  hipLaunchKernelGGL(fat::cache_stats_kernel, dim3(1), dim3(fat::kStatsThreads), 0,
                     static_cast<hipStream_t>(stream_ptr), a->seq_lens, a->page_table, a->batch, a->max_pages,
                     a->page_table_stride, a->page_size, a->out);
  return fat_host::launch_status("cache_stats_kernel");
}
