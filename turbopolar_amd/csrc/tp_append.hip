// tp_append.hip -- the per-append staging step of TurboPolarKVCacheRuntime.
//
// The reference validates every append with mx.isfinite(...).all() (one host
// synchronisation per input, turbo_polar_cache.py:69) and then concatenates
// the new tokens onto its dense tail (:114-115).  Here one launch does both:
// it scans every element of k and v for non-finite values and copies a token
// range of them into the caller's preallocated dense tail; the host then reads
// one 4-byte verdict.  Nothing else in the runtime's state changes, so a
// rejected append leaves the cache as it was (only tail slots past the valid
// length were written).
#include "tp_common.h"

namespace tp {

struct AppendArgs {
  const void* k;
  const void* v;
  void* tail_k;
  void* tail_v;
  int64_t bh;
  int64_t in_tokens;
  int64_t copy_begin;
  int64_t n_copy;
  int64_t scan_begin;   // tokens of each row that the launch reads: all of them
  int64_t scan_tokens;  // with a check, the copied ones without
  int64_t tail_tokens;  // token capacity of one (b, h) row of the tail
  int64_t tail_pos;
  uint32_t* flag;
  uint32_t epoch;
  int32_t check;
};

__device__ __forceinline__ bool all_finite(uint4 w, bool f32) {
  const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
  bool ok = true;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (f32) {
      ok = ok && ((ws[i] & 0x7f800000u) != 0x7f800000u);
    } else {
      ok = ok && ((ws[i] & 0x7c00u) != 0x7c00u) && ((ws[i] & 0x7c000000u) != 0x7c000000u);
    }
  }
  return ok;
}

// One thread per 16-byte chunk of k (and the same chunk of v).
template <bool kF32>
__global__ __launch_bounds__(256) void append_stage_kernel(AppendArgs a) {
  constexpr int kElems = kF32 ? 4 : 8;           // elements per 16-byte chunk
  constexpr int kChunks = kHeadDim / kElems;     // chunks per token row
  const int64_t n = a.bh * a.scan_tokens * kChunks;
  bool bad = false;
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = c / kChunks;             // (bh, scanned token)
    const int part = (int)(c - row * kChunks);
    const int64_t bh = row / a.scan_tokens;
    const int64_t tok = a.scan_begin + (row - bh * a.scan_tokens);
    const int64_t src = (bh * a.in_tokens + tok) * kChunks + part;
    const uint4 kw = reinterpret_cast<const uint4*>(a.k)[src];
    const uint4 vw = reinterpret_cast<const uint4*>(a.v)[src];
    if (a.check) bad = bad || !all_finite(kw, kF32) || !all_finite(vw, kF32);
    const int64_t rel = tok - a.copy_begin;
    if (rel >= 0 && rel < a.n_copy) {
      const int64_t dst = (bh * a.tail_tokens + a.tail_pos + rel) * kChunks + part;
      reinterpret_cast<uint4*>(a.tail_k)[dst] = kw;
      reinterpret_cast<uint4*>(a.tail_v)[dst] = vw;
    }
  }
  if (a.check == 2 && gridDim.x == 1) {
    // One workgroup: it reports completion itself, epoch (all finite) or
    // epoch + 1, once every thread's copies are issued and its verdict known;
    // the host polls the pinned word instead of synchronising the stream.
    const bool any_bad = __syncthreads_or(bad);
    if (threadIdx.x == 0)
      __hip_atomic_store(a.flag, any_bad ? a.epoch + 1u : a.epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  } else if (bad) {  // every writer stores the same value
    if (a.check >= 2)
      __hip_atomic_store(a.flag, a.epoch + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);  // pinned host flag
    else
      *a.flag = a.epoch;
  }
}

// ---- growth of a page store -------------------------------------------------------
//
// Bound by launches, not by bytes: a store of 512 pages x 8 heads was filled and
// copied buffer by buffer in 12 torch launches, most of them 2-4 us of kernel
// behind 10-20 us of host; here every buffer's kept and cleared bytes go out
// in one.  blockIdx.z is the buffer, y the (batch, head) row, x strides over the
// row's chunks; a buffer whose pointers, rows and bounds are all multiples of 16
// bytes moves 16 bytes a thread, any other (the fp16 page scales) 2, or 1.
constexpr int kGrowMax = 8;
struct GrowArgs {
  tp_grow b[kGrowMax];
  int64_t rows;
};

template <class T>
__device__ __forceinline__ void grow_row(const tp_grow& g, int64_t row) {
  const int64_t keep = g.keep / (int64_t)sizeof(T);
  const int64_t clear = g.clear_from / (int64_t)sizeof(T);
  const int64_t total = keep + g.dst_row / (int64_t)sizeof(T) - clear;
  const T* src = reinterpret_cast<const T*>(static_cast<const char*>(g.src) + row * g.src_row);
  T* dst = reinterpret_cast<T*>(static_cast<char*>(g.dst) + row * g.dst_row);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    if (i < keep)
      dst[i] = src[i];
    else
      dst[clear + i - keep] = T{};
  }
}

__global__ __launch_bounds__(256) void grow_rows_kernel(GrowArgs a) {
  const tp_grow& g = a.b[blockIdx.z];
  const uint64_t u = (uint64_t)(uintptr_t)g.src | (uint64_t)(uintptr_t)g.dst | (uint64_t)g.src_row |
                     (uint64_t)g.dst_row | (uint64_t)g.keep | (uint64_t)g.clear_from;
  for (int64_t row = blockIdx.y; row < a.rows; row += gridDim.y) {
    if ((u & 15u) == 0)
      grow_row<uint4>(g, row);
    else if ((u & 1u) == 0)
      grow_row<uint16_t>(g, row);
    else
      grow_row<uint8_t>(g, row);
  }
}

}  // namespace tp

using namespace tp;

extern "C" {

int32_t tp_grow_rows(const tp_grow* bufs, int32_t n_bufs, int64_t rows, void* stream) {
  clear_error();
  if (!bufs || n_bufs < 1 || n_bufs > kGrowMax || rows < 1) {
    set_error("tp_grow_rows takes 1 to %d buffers and at least one row, got %d and %lld", kGrowMax, n_bufs,
              (long long)rows);
    return TP_ERR_INVALID;
  }
  GrowArgs a{};
  a.rows = rows;
  int64_t most = 0;
  for (int i = 0; i < n_bufs; ++i) {
    const tp_grow& g = bufs[i];
    if (!g.dst || g.keep < 0 || g.keep > g.src_row || g.keep > g.clear_from || g.clear_from > g.dst_row ||
        (g.keep > 0 && !g.src)) {
      set_error("tp_grow_rows: buffer %d keeps %lld of %lld bytes and clears from %lld of %lld", i, (long long)g.keep,
                (long long)g.src_row, (long long)g.clear_from, (long long)g.dst_row);
      return TP_ERR_INVALID;
    }
    a.b[i] = g;
    most = std::max(most, g.keep + g.dst_row - g.clear_from);
  }
  if (most == 0) return TP_OK;
  // Four chunks of 16 bytes a thread, at most 64 workgroups a row.
  const unsigned x = (unsigned)std::min<int64_t>((most + 16383) / 16384, 64);
  const dim3 grid(x, (unsigned)std::min<int64_t>(rows, 65535), (unsigned)n_bufs);
  hipLaunchKernelGGL(grow_rows_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), a);
  return launch_status("tp_grow_rows");
}

int32_t tp_append_stage(const void* k, const void* v, int32_t in_dtype, int64_t bh, int64_t in_tokens,
                        int64_t copy_begin, int64_t n_copy, void* tail_k, void* tail_v, int64_t tail_tokens,
                        int64_t tail_pos, int32_t check, uint32_t* flag, uint32_t epoch, void* stream) {
  clear_error();
  if (in_dtype != 0 && in_dtype != 1) {
    set_error("in_dtype must be 0 (fp16) or 1 (fp32), got %d", in_dtype);
    return TP_ERR_INVALID;
  }
  if (!k || !v || bh < 1 || in_tokens < 1) {
    set_error("bad input: k=%p v=%p bh=%lld tokens=%lld", k, v, (long long)bh, (long long)in_tokens);
    return TP_ERR_INVALID;
  }
  if (copy_begin < 0 || n_copy < 0 || copy_begin + n_copy > in_tokens || tail_pos < 0 ||
      tail_pos + n_copy > tail_tokens || (n_copy > 0 && (!tail_k || !tail_v))) {
    set_error("bad copy range: begin=%lld n=%lld of %lld tokens into tail position %lld of %lld",
              (long long)copy_begin, (long long)n_copy, (long long)in_tokens, (long long)tail_pos,
              (long long)tail_tokens);
    return TP_ERR_INVALID;
  }
  if (check < 0 || check > 3 || (check && !flag) || (check >= 2 && (epoch & 1u))) {
    set_error("check must be 0, 1 (device flag), 2 (pinned host flag, even epoch) or 3 (deferred, pinned host "
              "flag, even epoch), with a flag when checking");
    return TP_ERR_INVALID;
  }
  const uintptr_t al = (uintptr_t)k | (uintptr_t)v | (uintptr_t)tail_k | (uintptr_t)tail_v;
  if (al & 15u) {
    set_error("k, v and the tail buffers must be 16-byte aligned");
    return TP_ERR_INVALID;
  }
  AppendArgs a;
  a.k = k;
  a.v = v;
  if (!check && n_copy == 0) return TP_OK;
  a.scan_begin = check ? 0 : copy_begin;
  a.scan_tokens = check ? in_tokens : n_copy;
  a.tail_k = tail_k;
  a.tail_v = tail_v;
  a.bh = bh;
  a.in_tokens = in_tokens;
  a.copy_begin = copy_begin;
  a.n_copy = n_copy;
  a.tail_tokens = tail_tokens;
  a.tail_pos = tail_pos;
  a.flag = flag;
  a.epoch = epoch;
  a.check = check;
  const int64_t chunks = bh * a.scan_tokens * (in_dtype ? kHeadDim / 4 : kHeadDim / 8);
  const unsigned blocks = (unsigned)std::min<int64_t>((chunks + 255) / 256, 1024);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (in_dtype)
    hipLaunchKernelGGL(append_stage_kernel<true>, dim3(blocks), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(append_stage_kernel<false>, dim3(blocks), dim3(256), 0, s, a);
  int32_t st = launch_status("tp_append_stage");
  if (st != TP_OK || !check || check == 3) return st;
  // The kernel writes the pinned host flag directly, no copy; one workgroup also
  // reports a finite input, so the host polls for it.
  if (check == 2) return wait_verdict(flag, epoch, s, blocks == 1, "tp_append_stage");
  uint32_t verdict = 0;
  if (hipMemcpyAsync(&verdict, flag, sizeof(verdict), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess) {
    set_error("tp_append_stage: reading the verdict failed");
    return TP_ERR_HIP;
  }
  if (verdict == epoch) {
    set_error("append() inputs must contain finite values");
    return TP_ERR_NONFINITE;
  }
  return TP_OK;
}

}  // extern "C"
