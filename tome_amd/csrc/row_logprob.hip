// Row kernel: logits[rows, V] -> log-prob of one target id per row (+ lse, entropy, argmax).
//
// Replaces local_compute_logprobs (mlx-impl/node.py:400-404) and the
// fused_log_softmax + host gather pair (mlx-impl/model.py:16-89, node.py:571,605).  The
// reference reads each row three times and writes a full [rows, V] matrix; here each
// element is read from HBM once with 16-byte loads and only per-row scalars are written.
//
// Grid: rows * splits workgroups of 4 wave64, or rows workgroups of 8 or 16 (row_waves_unsplit).  A workgroup owns a contiguous
// range of 16-byte load units of one row (RowSpan: units start at the row's first 16-byte boundary), every lane keeps an online (max, sum 2^(y-m))
// pair over the units it reads, lanes are merged by DPP and LDS-crossbar exchanges, the
// waves through LDS.  splits == 1 finishes in the same launch; otherwise per-split
// partials go to the workspace and row_combine_kernel merges them (no float atomics, so
// results do not depend on scheduling).
#include "row_common.hpp"

#include <atomic>
#include <mutex>

namespace tome {

// A launch scores `problems`: problem i reads row i of the logits - or, with a row list, row row_index[i] - and
// owns entry i of the targets, the mask, the outputs and the partials.
struct RowArgs {
  const void* logits;
  const int32_t* row_index;  // nullable: problem -> row of `logits` (a row outside [0, n_rows) scores NaN, argmax -1)
  int64_t n_rows;            // rows the logits matrix holds (only read with a row list)
  RowSel sel;
  float* out_lp;
  float* out_lse;
  float* out_entropy;
  int32_t* out_argmax;
  RowPartial* partials;
  int64_t V;
  int64_t row_stride;
  int splits;
  float scale;  // log2(e) / temperature
};

// First element of unit `unit` (RowSpan's numbering) that holds the row's maximum.
template <typename T>
__device__ __forceinline__ int argmax_in_unit(const T* row, int64_t V, int unit, float mx) {
  constexpr int kVec = Elem<T>::kVec;
  const RowSpan<T> sp(row, V);
  // No element above the floor was seen (all -inf / NaN row): report index 0, as a first-max scan would.
  if (unit < 0 || unit >= sp.head + sp.n_units + sp.tail) return 0;
  if (unit < sp.head) return unit;
  if (unit >= sp.head + sp.n_units) return (int)(sp.tail_start() + (unit - sp.head - sp.n_units));
  const int64_t first = sp.head + (int64_t)(unit - sp.head) * kVec;
  for (int i = 0; i < kVec; ++i)
    if (Elem<T>::load1(row + first + i) == mx) return (int)(first + i);
  return (int)first;
}

// The target's logit, or NaN when no log-prob is asked for or the id is outside [0, V).  Lane 0 issues
// this at the start of its workgroup, so the dependent load pair (id, then logit) is long finished
// when the row has been streamed.
template <typename T>
__device__ __forceinline__ float load_target_logit(const RowArgs& a, const T* row, int64_t r) {
  if (!a.out_lp || !a.sel.targets) return __builtin_nanf("");
  const int32_t t = a.sel.target(r);
  return (t >= 0 && t < a.V) ? Elem<T>::load1(row + t) : __builtin_nanf("");
}

template <typename T, bool ENT, bool AMAX>
__device__ __forceinline__ void finish_row(const RowArgs& a, const T* row, int64_t r, const RowStat& st, float x_t) {
  // Called by one lane.  lp = (y_t - m - log2 s) ln2 with the same fma that fed the sum, so
  // the target's own term is part of s and lp <= 0 up to the rounding of the merges.
  const float m = st.mx * a.scale;
  const float log2s = fast_log2(st.s);
  if (a.out_lp) a.out_lp[r] = (fmaf(x_t, a.scale, -m) - log2s) * kLn2;  // NaN in, NaN out
  if (a.out_lse) a.out_lse[r] = (m + log2s) * kLn2;
  if constexpr (ENT) a.out_entropy[r] = (log2s - st.w / st.s) * kLn2;  // w is relative to the maximum: no m here
  if constexpr (AMAX) a.out_argmax[r] = argmax_in_unit<T>(row, a.V, st.bi, st.mx);
}

// KEEP: the caller reads the rows again right away (the second pass of the full log-softmax matrix), so they are
// loaded with ordinary loads and stay in the caches; everyone else streams them past the caches.
template <typename T, bool ENT, bool AMAX, bool KEEP, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void row_logprob_kernel(RowArgs a) {
  constexpr int kVec = Elem<T>::kVec;
  constexpr int kWG = WAVES * 64;
  __shared__ RowLdsT<WAVES> lds;
  const int tid = threadIdx.x;
  // No division for rows that are not split, and a 32-bit one for those that are: batches of short rows are bound by what a
  // workgroup does around its few loads (32768 x 300 fp32 60.8 -> 49.8 us, bf16 61.8 -> 51.2; 32768 x 2048 78.4 -> 61.9 and 69.7 -> 56.7).
  int64_t r = blockIdx.x;  // problem index
  int split = 0;
  if (a.splits > 1) {
    r = blockIdx.x / a.splits;
    split = blockIdx.x % a.splits;
  }

  if (!a.sel.valid(r)) {  // masked row: not read, outputs zeroed
    if (split == 0 && tid == 0) {
      if (a.out_lp) a.out_lp[r] = 0.f;
      if (a.out_lse) a.out_lse[r] = 0.f;
      if (ENT) a.out_entropy[r] = 0.f;
      if (AMAX) a.out_argmax[r] = -1;
    }
    return;
  }
  const int64_t src = a.row_index ? (int64_t)a.row_index[r] : r;  // row of the logits matrix
  if (a.row_index && (uint64_t)src >= (uint64_t)a.n_rows) {        // a list entry that names no row: not read
    if (split == 0 && tid == 0) {
      if (a.out_lp) a.out_lp[r] = __builtin_nanf("");
      if (a.out_lse) a.out_lse[r] = __builtin_nanf("");
      if (ENT) a.out_entropy[r] = __builtin_nanf("");
      if (AMAX) a.out_argmax[r] = -1;
    }
    return;
  }

  const T* row = static_cast<const T*>(a.logits) + src * a.row_stride;
  const RowSpan<T> sp(row, a.V);
  int64_t u0 = 0, u1 = sp.n_units;
  if (a.splits > 1) {
    const int per_split = ((int)sp.n_units + a.splits - 1) / a.splits;  // (a row has fewer than 2^29 units)
    u0 = (int64_t)per_split * split;
    u1 = u0 + per_split < sp.n_units ? u0 + per_split : sp.n_units;
  }

  float x_t = 0.f;
  if (tid == 0 && a.splits == 1) x_t = load_target_logit<T>(a, row, r);
  RowStat st = stat_identity();
  if (split == 0 && tid < sp.head) {  // single elements in front of the first whole unit, one per lane
    float x[1] = {Elem<T>::load1(row + tid)};
    absorb<1, ENT, AMAX>(st, x, tid, a.scale);
  }
  const u32x4* p = sp.p;
  int64_t u = u0 + tid;
  for (; u + (kRowUnroll - 1) * kWG < u1; u += kRowUnroll * kWG) {  // several 16-byte loads in flight per lane
    u32x4 v[kRowUnroll];
#pragma unroll
    for (int k = 0; k < kRowUnroll; ++k) v[k] = KEEP ? p[u + k * kWG] : __builtin_nontemporal_load(p + u + k * kWG);
#pragma unroll
    for (int k = 0; k < kRowUnroll; ++k) {
      float x[kVec];
      Elem<T>::unpack(v[k], x);
      absorb<kVec, ENT, AMAX>(st, x, sp.head + (int)(u + k * kWG), a.scale);
    }
  }
  {  // leftover units of this lane, issued together so their latencies overlap
    u32x4 v[kRowUnroll - 1];
#pragma unroll
    for (int k = 0; k < kRowUnroll - 1; ++k)
      if (u + k * kWG < u1) v[k] = KEEP ? p[u + k * kWG] : __builtin_nontemporal_load(p + u + k * kWG);
#pragma unroll
    for (int k = 0; k < kRowUnroll - 1; ++k)
      if (u + k * kWG < u1) {
        float x[kVec];
        Elem<T>::unpack(v[k], x);
        absorb<kVec, ENT, AMAX>(st, x, sp.head + (int)(u + k * kWG), a.scale);
      }
  }
  if (split == a.splits - 1 && tid < sp.tail) {  // ... and after the last one
    const int64_t e = sp.tail_start() + tid;
    float x[1] = {Elem<T>::load1(row + e)};
    absorb<1, ENT, AMAX>(st, x, sp.head + (int)sp.n_units + tid, a.scale);
  }

  const RowStat tot = block_reduce(st, a.scale, lds);
  if (tid != 0) return;
  if (a.splits == 1) finish_row<T, ENT, AMAX>(a, row, r, tot, x_t);
  else a.partials[r * a.splits + split] = RowPartial{tot.mx, tot.s, tot.w, tot.bi};
}

// One wave per row merges the per-split partials (splits <= 64).
template <typename T, bool ENT, bool AMAX>
__global__ __launch_bounds__(64) void row_combine_kernel(RowArgs a) {
  touch_args(a);  // 8 x 151936 in a captured graph, both launches, 6.15 -> 6.06 us (whole calls: equal, 7.2); no gain in the kernel above
  const int64_t r = blockIdx.x;
  if (!a.sel.valid(r)) return;  // outputs already zeroed by the main kernel
  const int64_t src = a.row_index ? (int64_t)a.row_index[r] : r;
  if (a.row_index && (uint64_t)src >= (uint64_t)a.n_rows) return;  // outputs already written by the main kernel
  const int lane = threadIdx.x;
  const T* row = static_cast<const T*>(a.logits) + src * a.row_stride;
  float x_t = 0.f;
  if (lane == 0) x_t = load_target_logit<T>(a, row, r);
  RowStat st = stat_identity();
  if (lane < a.splits) {
    const RowPartial p = a.partials[r * a.splits + lane];
    st = RowStat{p.mx, p.s, p.w, p.bi};
  }
  stat_wave_reduce(st, a.scale);
  if (lane != 0) return;
  finish_row<T, ENT, AMAX>(a, row, r, st, x_t);
}

template <typename T, bool ENT, bool AMAX, bool KEEP, int WAVES>
static hipError_t launch_row(const RowArgs& a, int64_t rows, hipStream_t stream, bool skip_combine = false) {
  hipLaunchKernelGGL((row_logprob_kernel<T, ENT, AMAX, KEEP, WAVES>), dim3((unsigned)(rows * a.splits)),
                     dim3(WAVES * 64), 0, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.splits == 1 || skip_combine) return e;
  hipLaunchKernelGGL((row_combine_kernel<T, ENT, AMAX>), dim3((unsigned)rows), dim3(64), 0,
                     stream, a);
  return hipGetLastError();
}

template <typename T, bool ENT, bool AMAX>
static hipError_t launch_waves(const RowArgs& a, int64_t rows, int waves, hipStream_t stream) {
  if (waves == 16) return launch_row<T, ENT, AMAX, false, 16>(a, rows, stream);
  if (waves == 8) return launch_row<T, ENT, AMAX, false, 8>(a, rows, stream);
  return launch_row<T, ENT, AMAX, false, kRowWaves>(a, rows, stream);
}

template <typename T>
static hipError_t dispatch_flags(const RowArgs& a, int64_t rows, int waves, hipStream_t stream) {
  const bool ent = a.out_entropy != nullptr, amax = a.out_argmax != nullptr;
  if (ent && amax) return launch_waves<T, true, true>(a, rows, waves, stream);
  if (ent) return launch_waves<T, true, false>(a, rows, waves, stream);
  if (amax) return launch_waves<T, false, true>(a, rows, waves, stream);
  return launch_waves<T, false, false>(a, rows, waves, stream);
}

// How many workgroups share a row, where rows are split (and the bound the workspace is sized for).  From 512 rows on one workgroup per row; smaller batches (decode steps,
// the 64-row CPU-comparison case) are split so that ~2 workgroups per CU are in flight, as long as every
// split keeps a few loads per lane.  Measured: aiming at 512 to 2048 workgroups is equal within 0.5 us for
// 32-256 rows, and 512 spares the 512- and 1024-row batches the combine launch (27.0 against 30.6 us,
// 50.3 against 52.7 us); 3072 and more are slower everywhere.
int row_splits_for(int64_t rows, int64_t V, int vec) {
  const int64_t units = V / vec;
  // Short rows (up to 128 KB) in batches of 256 and more: one workgroup per CU is there already, and the combine launch
  // costs more than the second half of the chip brings (256 rows of 32000: fp32 10.6 against 12.0 us, bf16 7.8 against 9.9).
  if (rows >= 256 && units <= 8192) return 1;
  const int64_t want_wgs = 512;
  int64_t s = (want_wgs + rows - 1) / rows;
  const int64_t max_by_work = units / (2 * kRowWG);  // >= 2 loads per lane per split
  if (s > max_by_work) s = max_by_work;
  if (s > 64) s = 64;
  if (s < 1) s = 1;
  return (int)s;
}

// Workgroup size for a launch of `rows` rows, 0 = split the rows as above.  Splitting a row costs a second launch (2-3 us,
// as much as a decode-sized call's loads); a workgroup of 8 or 16 waves keeps enough loads of ONE row in flight that between
// about a row per thousand elements and 512 rows the single launch is the faster one, and always for rows of up to 24576
// elements.  Inside a captured graph, split / 16 waves a row (us): 64 x 32000 fp32 8.4 / 6.5, 128 x 32000 9.6 / 6.9, 200 x
// 100000 18.7 / 15.6, 200 x 151936 bf16 16.5 / 13.8; on the other side of the line 48 x 65536 8.6 / 8.9, 64 x 100000 9.8 /
// 11.9, 64 x 151936 12.0 / 16.1, 96 x 151936 bf16 11.6 / 12.9.  A little above one row per CU, long rows are dealt out more
// evenly in halves (300 x 151936: fp32 34.5 / 37.0, bf16 21.1 / 22.0; 393 rows 45.3 / 40.5 and 27.4 / 23.7).
// Above one row per CU 8 waves are as fast as 16 or faster (393 x 50257 bf16, all statistics: 4 / 8 / 16 waves 14.2 / 12.9 /
// 13.7); short rows do not fill more waves (4096 elements: 300 rows 4.4 / 5.2 / 6.3, 64 rows 8 / 16 waves 4.0 / 4.4).
static int row_waves_unsplit(int64_t rows, int64_t V, int vec) {
  const int64_t units = V / vec;
  if (rows >= 512 || units < 4 * kRowWG) return row_splits_for(rows, V, vec) == 1 ? kRowWaves : 0;
  if (rows > 256) {
    if (rows < 352 && V > 98304) return 0;
    return units < 16 * kRowWG ? kRowWaves : 8;
  }
  if (V > 24576 && rows * 1000 < V) return 0;
  return units < 12 * kRowWG ? 8 : 16;
}

// `rows` problems.  With `row_index` (device, one entry per problem) problem i reads row row_index[i] of a matrix
// of `n_rows` rows; without it, row i.
hipError_t row_logprob_launch_rows(const void* logits, int dtype, int64_t n_rows, const int32_t* row_index, int64_t rows,
                                   int64_t V, int64_t row_stride, const RowSel& sel, float temperature, float* out_lp, float* out_lse, float* out_entropy,
                                   int32_t* out_argmax, void* workspace, hipStream_t stream) {
  const int esize = dtype == 0 ? 4 : 2;
  const int vec = 16 / esize;
  RowArgs a;
  a.logits = logits;
  a.row_index = row_index;
  a.n_rows = n_rows;
  a.sel = sel;
  a.out_lp = out_lp;
  a.out_lse = out_lse;
  a.out_entropy = out_entropy;
  a.out_argmax = out_argmax;
  a.partials = static_cast<RowPartial*>(workspace);
  a.V = V;
  a.row_stride = row_stride;
  const int waves = row_waves_unsplit(rows, V, vec);
  a.splits = waves ? 1 : row_splits_for(rows, V, vec);
  a.scale = kLog2e / temperature;
  return dtype == 0 ? dispatch_flags<float>(a, rows, waves, stream) : dispatch_flags<uint16_t>(a, rows, waves, stream);
}

// The rows' logsumexp for a caller that merges split rows itself: only the main kernel is launched.  With
// *splits == 1 out_lse holds the result; otherwise the workspace holds *splits partials per row (RowPartial) and
// out_lse is untouched.
hipError_t row_lse_partials_launch(const void* logits, int dtype, int64_t rows, int64_t V, int64_t row_stride,
                                   float temperature, float* out_lse, void* workspace, int* splits, hipStream_t stream) {
  const int esize = dtype == 0 ? 4 : 2;
  const int vec = 16 / esize;
  RowArgs a{};
  a.logits = logits;
  a.n_rows = rows;
  a.out_lse = out_lse;
  a.partials = static_cast<RowPartial*>(workspace);
  a.V = V;
  a.row_stride = row_stride;
  a.splits = row_splits_for(rows, V, vec);
  a.scale = kLog2e / temperature;
  *splits = a.splits;
  // The caller's second pass reads the matrix again: up to ~3/4 GB it pays to leave the rows in the caches (measured, both
  // passes, fp32 rows of 151936: 64 rows 25.9 -> 24.4 us, 512 rows 155 -> 145, 1024 rows 312 -> 294; 2048 rows 628 -> 648).
  const bool keep = (double)rows * (double)V * esize <= 768.0 * 1024 * 1024;
  if (dtype == 0)
    return keep ? launch_row<float, false, false, true, kRowWaves>(a, rows, stream, true)
                : launch_row<float, false, false, false, kRowWaves>(a, rows, stream, true);
  return keep ? launch_row<uint16_t, false, false, true, kRowWaves>(a, rows, stream, true)
              : launch_row<uint16_t, false, false, false, kRowWaves>(a, rows, stream, true);
}

hipError_t row_logprob_launch(const void* logits, int dtype, int64_t rows, int64_t V, int64_t row_stride,
                              const RowSel& sel, float temperature, float* out_lp, float* out_lse, float* out_entropy,
                              int32_t* out_argmax, void* workspace, hipStream_t stream) {
  return row_logprob_launch_rows(logits, dtype, rows, nullptr, rows, V, row_stride, sel, temperature,
                                 out_lp, out_lse, out_entropy, out_argmax, workspace, stream);
}

// ---- allocation-free variant ---------------------------------------------------------------------
// The per-(row, split) partials of a split launch normally live in a caller-provided workspace.  For
// callers that cannot allocate one (code under graph capture, serving loops with a fixed memory plan)
// the same launches can use this array, which is part of the code object: every GPU the library runs on
// holds its own copy from the first launch until the process ends.  In host code the array's name is
// only a handle for hipGetSymbolAddress; kernels are given the address it returns for the current
// device.  Nothing in it has to start at zero: the combine kernel reads exactly the partials that the
// main kernel of the same call wrote.  All calls on one GPU share the array, so two calls that overlap
// in time on one GPU (different streams) race on it.
constexpr size_t kRowScratchBytes = 64 * 1024;
static __device__ __align__(256) unsigned char scratch[kRowScratchBytes];

constexpr int kMaxDevices = 64;
static std::atomic<void*> g_scratch_ptr[kMaxDevices];  // device address of `scratch`, per device ordinal
static std::mutex g_scratch_mutex;
// Bytes of the array a call may use: the whole array, unless a test lowered it to reach the error path.
static std::atomic<size_t> g_scratch_limit{kRowScratchBytes};

size_t row_scratch_capacity() { return kRowScratchBytes; }
size_t row_scratch_set_limit(size_t bytes) {
  const size_t lim = (bytes == 0 || bytes > kRowScratchBytes) ? kRowScratchBytes : bytes;
  g_scratch_limit.store(lim, std::memory_order_relaxed);
  return lim;
}

// Address of this device's copy of the scratch array; resolved once per device, with that device current.
// After that first call the address is read without taking the lock.
static hipError_t row_scratch_for_current_device(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (!p) {
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess) return e;
      if (!p) return hipErrorInvalidSymbol;
      g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return hipSuccess;
}

// Bytes of partials a call with these shapes writes (0 when every row is one workgroup).
size_t row_partials_bytes(int dtype, int64_t rows, int64_t V) {
  const int vec = 16 / (dtype == 0 ? 4 : 2);
  const int splits = row_splits_for(rows, V, vec);
  return splits <= 1 ? 0 : (size_t)rows * (size_t)splits * sizeof(RowPartial);
}

// row_logprob_launch with the partials in the library's own scratch array.  `too_big` is set (and nothing
// launched) when the call would need more than the array holds.
hipError_t row_logprob_noalloc_launch(const void* logits, int dtype, int64_t rows, int64_t V, int64_t row_stride,
                                      const RowSel& sel, float temperature, float* out_lp, float* out_lse, float* out_entropy, int32_t* out_argmax,
                                      bool* too_big, hipStream_t stream) {
  *too_big = row_partials_bytes(dtype, rows, V) > g_scratch_limit.load(std::memory_order_relaxed);
  if (*too_big) return hipSuccess;
  void* ptr = nullptr;
  const hipError_t e = row_scratch_for_current_device(&ptr);
  if (e != hipSuccess) return e;
  return row_logprob_launch(logits, dtype, rows, V, row_stride, sel, temperature, out_lp, out_lse,
                            out_entropy, out_argmax, ptr, stream);
}

}  // namespace tome
