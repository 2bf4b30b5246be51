// Decode-step sampler fused onto the logits pass: per row, the top-k logits, one categorical draw
// among them, the log-prob of the drawn token under the FULL softmax, and the greedy token.
//
// Replaces, per decode step, _sample_token (mlx-impl/node.py:894-907: argpartition top-k of
// logits / temperature, mx.random.categorical over them) together with
// fused_log_softmax(...)[b, token] (node.py:590,605 / 356,373) and int(mx.argmax(logits))
// (node.py:602,897) - B host round trips per step in the reference, one launch and one small
// copy here.
//
// The draw is specified without an RNG: the caller passes one uniform u in [0, 1) per row and the
// kernel takes the inverse CDF of softmax(top-k logits / T), the k candidates ordered by logit
// (descending; equal logits by ascending token id).  MLX's own random stream cannot be matched.
//
// Rows may start at any element (RowSpan): 1024 rows of 128258 fp32 / bf16 303 / 445 us on element-wise loads, 94 / 72 us here.
//
// Two forms.
//
// Decode batches (row_sample_cells_kernel + row_sample_pick_kernel): the first launch streams the rows from as many
// workgroups as fill the chip and leaves, besides the partial (max, sum 2^(y-m)), the maximum of every CELL of 8 consecutive
// load units (128 bytes: a cache line).  The second, a workgroup per row, takes the k best cells by (maximum, lower cell
// first) and reads only those again: as cells lie in the order of the ids, they hold the row's top k - were a top-k element
// in another cell, each of the k better cells would hold an element that precedes it.  Nothing but a maximum per lane
// and load unit is then paid per element, and the selection is done once a row instead of once a range (the form before:
// every workgroup ranked the candidates of its range, a second launch merged splits * k keys).
// Two launches either way; 64 x 151936 fp32 20.2 -> 15 us (6.5 streaming, 7 picking), 8 rows 14.6 -> 10, 64 x 50257 25 -> 11; bf16 64 x 151936
// 20.4 -> 13, 256 rows 40 -> 23, 700 rows 67 -> 47, 1024 x 50257 172 -> 31.  (Rows that the memory-side cache still holds; on
// rotating buffers the streaming launch takes 9.7 us, 38.9 MB at 4.0 TB/s.)  The other launch is a chain of some 12000 cycles: kernel
// arguments and first loads 1500, cell maxima 1700, the bound 1500, cells collected 1800, partial statistics 1200 (beside the elements' load), elements 1000, ranks 1100, draw 1000.
//
// Large batches (row_sample_kernel, one workgroup a row, no workspace): per row,
//   * the online (max, sum 2^(y-m)) for the full-vocabulary lse and every lane's own largest element;
//   * a lower bound `theta` of the k-th largest logit: the k-th largest of the lane maxima (four waves,
//     each extracting its ceil(k/4) largest);
//   * every element >= theta, as a candidate in an LDS buffer (typically k + a few entries).
// Short rows (a lane owns <= 8 load units) are loaded once and kept in registers for the candidate
// scan.  Long rows are streamed once: theta comes from the lanes' first units, is renewed after a
// quarter of the row, and candidates are collected as the row goes by; only when the buffer overflows
// is the row scanned a second time with the bound from all of it.
// Candidates are 64-bit keys (order-preserving image of the float, then ~index), so there are no
// ties and the top k is unique.  If a buffer overflows (adversarial orderings), theta is raised to
// the k-th largest of what was kept - still a lower bound - and the scan is repeated.  The final k are ranked by
// counting.
#include "row_common.hpp"
#include <type_traits>

namespace tome {

constexpr int kSampCap = 1024;      // candidate keys per buffer in the main kernel (2 x 8 KB of LDS: 8 workgroups per CU)
constexpr int kCellUnits = 8;       // load units per cell: consecutive, one 128-byte line
constexpr int kCellBlock = kCellUnits * kRowWG;  // load units a workgroup of the cells kernel takes at a time (256 cells)
// Keys per buffer of the pick kernel: k <= 32 cells of 8 units, and the single elements of the edges.
template <typename T>
constexpr int kSampPickCap = 32 * kCellUnits * Elem<T>::kVec + 64;
constexpr int kSampCached = 8;      // a lane keeps up to this many load units in registers between the passes
constexpr int kSampMaxK = 32;  // one tightening round is then sure to drop >= 32 of the 64 sampled keys

struct SampleArgs {
  const void* logits;
  const float* uniforms;      // one per row, or nullptr = greedy (candidate 0)
  RowSel sel;                 // its mask only
  int32_t* out_token;
  float* out_lp;              // nullable
  float* out_lse;             // nullable
  int32_t* out_argmax;        // nullable
  int32_t* out_topk_idx;      // nullable, [rows, top_k], -1 past the end of a short row
  float* out_topk_logit;      // nullable, [rows, top_k] raw logits
  // A decode loop's state (out_next set): `active` is also the mask `sel` reads, and loses the rows that draw stop_token;
  // out_next is the next step's input id, idle_token for rows that are done.
  int32_t* active;
  int64_t* out_next;
  int64_t idle_token;
  int32_t stop_token;
  float* cells;               // workspace: [rows, n_cells] cell maxima (splits > 0)
  float2* part_stat;          // workspace: [rows, splits * kRowWaves] (max, sum)
  int64_t V;
  int64_t row_stride;
  int top_k;
  int splits;                 // workgroups per row of the cells kernel
  int blocks_per_split;
  int64_t n_cells;            // a multiple of 256
  float scale;                // log2(e) / temperature
};

// Order-preserving map float -> uint32 (NaN never gets here: candidates pass a float compare first).
__device__ __forceinline__ uint32_t float_key(float x) {
  const uint32_t u = __float_as_uint(x + 0.0f);  // -0.0 -> +0.0
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}
__device__ __forceinline__ uint64_t make_key(float x, uint32_t idx) {
  return ((uint64_t)float_key(x) << 32) | (uint64_t)(0xFFFFFFFFu - idx);  // equal logits: lower id first
}
__device__ __forceinline__ uint32_t key_index(uint64_t k) { return 0xFFFFFFFFu - (uint32_t)k; }

template <int CAP>
struct SampleLds {
  uint64_t a[CAP];
  uint64_t b[CAP];
  uint64_t top[kSampMaxK];
  uint64_t thr4[kRowWaves];
  int cnt;
  int cnt2;
  int kept;       // select_top_k's own count
  int wave_cnt[kRowWaves];
  RowLds red;
};

// Keys of four wave regions (counts c[w], region w starting at base + w * stride) as one list: entry i.
__device__ __forceinline__ uint64_t region_entry(const uint64_t* base, int stride, const int* c, int i) {
  int w = 0;
#pragma unroll
  for (int q = 0; q < kRowWaves - 1; ++q)
    if (w == q && i >= c[q]) {
      i -= c[q];
      w = q + 1;
    }
  return base[w * stride + i];
}

// One wave sorts up to 64 keys held one per lane (0 = none; m = number of lanes that may hold one): returns in lane i
// the (i+1)-th largest key for i < k, 0 elsewhere.  Register traffic only (v_readlane broadcasts, one ds_permute pair).
__device__ __forceinline__ uint64_t wave_sorted_top_k(uint64_t key, int m, int k) {
  const uint32_t lo = (uint32_t)key, hi = (uint32_t)(key >> 32);
  int rank = 0;
  for (int j0 = 0; j0 < m; j0 += 8)  // (lanes from m on hold 0: counted by nobody)
#pragma unroll
    for (int j = j0; j < j0 + 8; ++j) {
      const uint64_t o = ((uint64_t)__builtin_amdgcn_readlane(hi, j) << 32) | (uint32_t)__builtin_amdgcn_readlane(lo, j);
      rank += o > key ? 1 : 0;
    }
  const bool keep = key != 0 && rank < k;           // k <= kSampMaxK = 32: lane 63 is never a destination
  const int dst = (keep ? rank : 63) * 4;
  const uint32_t slo = (uint32_t)__builtin_amdgcn_ds_permute(dst, (int)(keep ? lo : 0u));
  const uint32_t shi = (uint32_t)__builtin_amdgcn_ds_permute(dst, (int)(keep ? hi : 0u));
  return ((uint64_t)shi << 32) | slo;               // lanes nobody sends to read 0
}

// Number of lanes of this wave whose key is larger than this lane's.  v_readlane broadcasts (the lane
// index is uniform), not LDS-crossbar shuffles: 64 dependent ds_bpermute round trips cost microseconds.
__device__ __forceinline__ int wave_rank(uint64_t key, int m) {
  const uint32_t lo = (uint32_t)key, hi = (uint32_t)(key >> 32);
  int rank = 0;
#pragma unroll 8
  for (int j = 0; j < m; ++j) {
    const uint64_t o = ((uint64_t)__builtin_amdgcn_readlane(hi, j) << 32) | (uint32_t)__builtin_amdgcn_readlane(lo, j);
    rank += o > key ? 1 : 0;
  }
  return rank;
}

// Sorted top-k of the m keys in `cur` (m <= the buffer size; 0 = empty slot) into sh.top[0..k), the rest of
// sh.top zeroed; returns the k-th largest key (0 if there are fewer than k).  `cur` / `other` are
// the two LDS buffers; both are clobbered.  All lanes of the workgroup must call it.
//
// Up to 256 keys are ranked directly: lane i counts the keys larger than key i (uniform LDS
// addresses: broadcast reads; a wave none of whose lanes holds a key skips the count - the chain of a
// decode-sized launch is bound by the instructions its waves issue, not by their latencies).  More than that are first thinned by a lower bound of the k-th
// largest from a sample: every wave ranks 64 keys of its own (256 distinct positions spread over the
// buffer), and the smallest of the four ceil(k/4)-th largest has >= k sampled keys at or above it;
// at least 32 sampled keys fall below it, so every round makes progress.
//
// The rounds count in sh.kept and leave sh.cnt alone: callers pass an `m` that every wave has just read from sh.cnt, with no barrier
// in between, and a wave late at that read would see a cleared count, take another path and leave the others' barriers unpaired.
// (A barrier at the head of the round is as safe, but costs the pick kernel's usual path, which never gets here, 0.27 us.)
template <class Lds>
__device__ uint64_t select_top_k(Lds& sh, uint64_t* cur, uint64_t* other, int m, int k) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  while (m > kRowWG) {
    const uint64_t key = cur[(int)(((int64_t)tid * m) >> 8)];
    const int rank = wave_rank(key, 64);
    const int want = (k + kRowWaves - 1) / kRowWaves;
    if (lane == 0) sh.thr4[wave] = 0;  // stays 0 (no bound) when fewer than `want` sampled keys are real
    __builtin_amdgcn_wave_barrier();
    if (key != 0 && rank == want - 1) sh.thr4[wave] = key;
    if (tid == 0) sh.kept = 0;
    __syncthreads();
    uint64_t thr = sh.thr4[0];
#pragma unroll
    for (int w = 1; w < kRowWaves; ++w) thr = sh.thr4[w] < thr ? sh.thr4[w] : thr;
    for (int i = tid; i < m; i += kRowWG) {
      const uint64_t key2 = cur[i];
      if (key2 >= thr && key2 != 0) other[atomicAdd(&sh.kept, 1)] = key2;
    }
    __syncthreads();
    const int kept = sh.kept;
    __syncthreads();
    if (kept == m) break;  // cannot happen for k <= 32 (see kSampMaxK); guards against an endless loop
    m = kept;
    uint64_t* t = cur;
    cur = other;
    other = t;
  }
  if (m > kRowWG) m = kRowWG;  // unreachable, see above
  const uint64_t key = tid < m ? cur[tid] : 0;
  int rank = 0;
  if (wave * 64 < m)  // wave-uniform: a wave whose lanes hold no key has nothing to rank
    for (int j = 0; j < m; ++j) rank += cur[j] > key ? 1 : 0;
  if (tid < kSampMaxK) sh.top[tid] = 0;
  __syncthreads();
  if (key != 0 && rank < k) sh.top[rank] = key;
  __syncthreads();
  return sh.top[k - 1];
}

// Maximum of a value over the wave, as a uniform value: six v_max_f32 with DPP sources towards lane 63 (lanes without a source
// keep theirs; each DPP read of a register just written waits two slots).  All lanes of the wave must call it.
__device__ __forceinline__ float wave_max_uniform(float v) {
  asm volatile(
      "s_nop 1\n"
      "v_max_f32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n s_nop 1\n"
      "v_max_f32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf\n s_nop 1\n"
      "v_max_f32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf\n s_nop 1\n"
      "v_max_f32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n s_nop 1\n"
      "v_max_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n s_nop 1\n"
      "v_max_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n s_nop 1"
      : "+v"(v));
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), 63));
}

// Lower bound of the k-th largest element of this workgroup's range from the lanes' own maxima (-inf
// for a lane that saw nothing): each wave extracts its ceil(k/4) largest lane maxima one by one (a
// wave-wide max, then the first lane that holds it steps aside), and the smallest of the four results
// has at least k lane maxima at or above it.  Values only - any element with that value passes.
template <class Lds>
__device__ uint64_t bound_from_lane_maxima(Lds& sh, float lane_max, int k) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int want = (k + kRowWaves - 1) / kRowWaves;
  float v = lane_max, kth = -INFINITY;
  for (int t = 0; t < want; ++t) {
    const float m = wave_max_uniform(v);
    kth = m;
    const uint64_t holders = __ballot(v == m);
    if (holders == 0) break;  // cannot happen (lane maxima are never NaN); guards the ctz below
    if (lane == __builtin_ctzll(holders)) v = -INFINITY;
  }
  if (lane == 0) sh.thr4[wave] = (uint64_t)float_key(kth) << 32;
  __syncthreads();
  uint64_t thr = sh.thr4[0];
#pragma unroll
  for (int w = 1; w < kRowWaves; ++w) thr = sh.thr4[w] < thr ? sh.thr4[w] : thr;
  __syncthreads();
  return thr;
}

// Wave 0: draw among the sorted candidates (lane i < k holds the (i+1)-th largest key, 0 = none) and write the
// row's outputs.  `tot` holds the full-vocabulary (max, sum) in every lane.
__device__ __forceinline__ float read_lane(float v, int i) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), i));
}
__device__ __forceinline__ void finish_sample(const SampleArgs& a, uint64_t key, int64_t r, const RowStat& tot, int lane, float uniform) {
  const int k = a.top_k;
  const bool have = key != 0;
  const float x = have ? key_float((uint32_t)(key >> 32)) : -INFINITY;
  const int n_have = __builtin_popcountll(__ballot(have));
  const float x0 = read_lane(x, 0);
  // Inclusive scan over the first 32 lanes (k <= kSampMaxK), without leaving the VALU: inside the 16-lane rows, then the first
  // row's total to the second.
  float cdf = have ? fast_exp2((x - x0) * a.scale) : 0.f;
  cdf += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(cdf), 0x111, 0xF, 0xF, true));  // row_shr:1
  cdf += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(cdf), 0x112, 0xF, 0xF, true));
  cdf += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(cdf), 0x114, 0xF, 0xF, true));
  cdf += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(cdf), 0x118, 0xF, 0xF, true));
  cdf += lane >= 16 ? read_lane(cdf, 15) : 0.f;
  int chosen = 0;
  if (a.uniforms && n_have > 0) {
    const float target = uniform * read_lane(cdf, n_have - 1);
    chosen = __builtin_popcountll(__ballot(have && cdf <= target));
    chosen = chosen < n_have ? chosen : n_have - 1;
  }
  const float cx = read_lane(x, chosen);
  const int32_t cidx = (int32_t)__builtin_amdgcn_readlane((int)key_index(key), chosen);
  if (a.out_topk_idx && lane < k) a.out_topk_idx[r * k + lane] = have ? (int32_t)key_index(key) : -1;
  if (a.out_topk_logit && lane < k) a.out_topk_logit[r * k + lane] = have ? x : 0.f;
  if (lane != 0) return;
  if (a.out_next) {  // every lane of this workgroup has read the row's mask long ago
    const int32_t token = n_have == 0 ? -1 : cidx;
    const bool stop = token == a.stop_token;
    a.out_next[r] = stop ? a.idle_token : token;
    if (stop) a.active[r] = 0;
  }
  const float m2 = tot.mx * a.scale;
  const float log2s = fast_log2(tot.s);
  if (n_have == 0) {  // nothing above -inf in the row
    a.out_token[r] = -1;
    if (a.out_lp) a.out_lp[r] = __builtin_nanf("");
    if (a.out_argmax) a.out_argmax[r] = 0;
  } else {
    a.out_token[r] = cidx;
    if (a.out_lp) a.out_lp[r] = (fmaf(cx, a.scale, -m2) - log2s) * kLn2;
    if (a.out_argmax) a.out_argmax[r] = (int32_t)key_index(key);
  }
  if (a.out_lse) a.out_lse[r] = (m2 + log2s) * kLn2;
}

// A masked row: not read.
__device__ __forceinline__ void masked_sample(const SampleArgs& a, int64_t r, int tid) {
  if (tid == 0) {
    a.out_token[r] = -1;
    if (a.out_lp) a.out_lp[r] = 0.f;
    if (a.out_lse) a.out_lse[r] = 0.f;
    if (a.out_argmax) a.out_argmax[r] = -1;
    if (a.out_next) a.out_next[r] = a.idle_token;
  }
  if (tid < a.top_k) {
    if (a.out_topk_idx) a.out_topk_idx[r * a.top_k + tid] = -1;
    if (a.out_topk_logit) a.out_topk_logit[r * a.top_k + tid] = 0.f;
  }
}

// CACHED: the host promises that a lane owns at most kSampCached load units (short rows); they are loaded
// once and both passes run from registers.
template <typename T, bool CACHED>
__global__ __launch_bounds__(kRowWG) __attribute__((amdgpu_waves_per_eu(6, 8))) void row_sample_kernel(SampleArgs a) {
  constexpr int kVec = Elem<T>::kVec;
  __shared__ SampleLds<kSampCap> sh;
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k = a.top_k;

  if (!a.sel.valid(r)) {
    masked_sample(a, r, tid);
    return;
  }

  const T* row = static_cast<const T*>(a.logits) + r * a.row_stride;
  const RowSpan<T> sp(row, a.V);
  const int64_t u0 = 0, u1 = sp.n_units;
  // single elements in front of the first whole unit and after the last one, one per lane
  const int n_head = sp.head;
  const int n_tail = sp.tail;

  const bool big_range = (u1 - u0) * kVec + n_head + n_tail > kSampCap;
  if (tid == 0) sh.cnt = 0;  // published by the first barrier below, before any candidate is offered
  // A candidate: a logit above -inf (a -inf logit has probability zero and is never drawn; NaN fails every
  // compare) at or above the bound (value first, then the whole key).
  auto offer = [&](float x, int64_t idx, uint64_t thr, float thr_val) {
    if (x >= thr_val && x > -INFINITY) {
      const uint64_t key = make_key(x, (uint32_t)idx);
      if (key >= thr) {
        const int pos = atomicAdd(&sh.cnt, 1);
        if (pos < kSampCap) sh.a[pos] = key;
      }
    }
  };

  // ---- pass 1: full-vocabulary statistics and this lane's own maximum --------------------------
  RowStat st = stat_identity();
  u32x4 cached[CACHED ? kSampCached : 1];
  float lane_max = -INFINITY;  // this lane's largest element, or -inf when it saw nothing above -inf
  RowStat tot = stat_identity();
  uint64_t theta = 0;
  const u32x4* p = sp.p;
  const int64_t tail_e = sp.tail_start() + tid;
  const float x_head = tid < n_head ? Elem<T>::load1(row + tid) : -INFINITY;  // -inf: adds nothing, is no candidate
  const float x_tail = tid < n_tail ? Elem<T>::load1(row + tail_e) : -INFINITY;
  if constexpr (CACHED) {
    // Everything a lane owns is in registers, so the statistics take two sweeps over them instead of an online
    // update: the maxima first, then the sum of 2^(y - m) against one reference per wave (no rescaling chain).
#pragma unroll
    for (int q = 0; q < kSampCached; ++q) {  // unconditional (clamped) loads: all eight in flight together
      const int64_t u = u0 + tid + q * kRowWG;
      cached[q] = __builtin_nontemporal_load(p + (u < u1 ? u : 0));  // unit 0 exists (checked on the host)
    }
#pragma unroll
    for (int q = 0; q < kSampCached; ++q)
      if (u0 + tid + q * kRowWG < u1) {
        float x[kVec];
        Elem<T>::unpack(cached[q], x);
        lane_max = fmaxf(lane_max, max_of_raw<kVec>(x));
      }
    lane_max = fmaxf(lane_max, fmaxf(x_head, x_tail));
    float wmax = lane_max;  // maximum of the wave
    wmax = fmaxf(wmax, wave_exchange<0>(wmax));
    wmax = fmaxf(wmax, wave_exchange<1>(wmax));
    wmax = fmaxf(wmax, wave_exchange<2>(wmax));
    wmax = fmaxf(wmax, wave_exchange<3>(wmax));
    wmax = fmaxf(wmax, wave_exchange<4>(wmax));
    wmax = fmaxf(wmax, wave_exchange<5>(wmax));
    const float mref = fmaxf(wmax, kMaxFloor);
    const float mm = mref * a.scale;
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int q = 0; q < kSampCached; ++q)
      if (u0 + tid + q * kRowWG < u1) {
        float x[kVec];
        Elem<T>::unpack(cached[q], x);
#pragma unroll
        for (int i = 0; i < kVec; i += 2) {
          s0 += fast_exp2(fmaf(x[i], a.scale, -mm));
          s1 += fast_exp2(fmaf(x[i + 1], a.scale, -mm));
        }
      }
    s0 += fast_exp2(fmaf(x_head, a.scale, -mm)) + fast_exp2(fmaf(x_tail, a.scale, -mm));
    float ws = s0 + s1;
    ws += wave_exchange<0>(ws);
    ws += wave_exchange<1>(ws);
    ws += wave_exchange<2>(ws);
    ws += wave_exchange<3>(ws);
    ws += wave_exchange<4>(ws);
    ws += wave_exchange<5>(ws);
    if (lane == 0) {
      sh.red.mx[wave] = mref;
      sh.red.s[wave] = ws;
    }
    __syncthreads();  // also publishes sh.cnt == 0
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) stat_merge(tot, RowStat{sh.red.mx[w], sh.red.s[w], 0.f, 0x7fffffff}, a.scale);
    // theta: k-th largest lane maximum (ranges that fit the buffer skip the bound)
    if (big_range) theta = bound_from_lane_maxima(sh, lane_max, k);
  } else {
    // Streaming variant: candidates are collected during this one pass.  The k-th largest of the
    // lanes' maxima over their FIRST units is already a lower bound of the row's k-th largest, so
    // everything at or above it goes to the buffer as it streams by; after a quarter of the range
    // the bound is renewed from the maxima so far, which lets far less through (a few hundred
    // candidates per row in all).
    constexpr int kGroup = kRowUnroll * kRowWG;                    // units per workgroup and iteration
    const int64_t n_groups = (u1 > u0 ? u1 - u0 : 0) / kGroup;     // iterations in which every lane has all its units
    uint64_t early = 0;  // ranges that fit the buffer are collected whole
    float early_val = -INFINITY;
    auto consume = [&](const u32x4& v, int64_t unit) {
      float x[kVec];
      Elem<T>::unpack(v, x);
      if (absorb<kVec, false, true>(st, x, (int)unit, a.scale) >= early_val) {
#pragma unroll
        for (int i = 0; i < kVec; ++i) offer(x[i], sp.head + unit * kVec + i, early, early_val);
      }
    };
    auto renew_bound = [&]() {
      early = bound_from_lane_maxima(sh, st.bi != 0x7fffffff ? st.mx : -INFINITY, k);
      early_val = early == 0 ? -INFINITY : key_float((uint32_t)(early >> 32));
    };
    int64_t g0 = 0;
    if (n_groups > 0 && big_range) {  // first iteration: statistics, then the bound, then its candidates
      u32x4 first[kRowUnroll];
#pragma unroll
      for (int q = 0; q < kRowUnroll; ++q) first[q] = __builtin_nontemporal_load(p + u0 + tid + q * kRowWG);
#pragma unroll
      for (int q = 0; q < kRowUnroll; ++q) {
        float x[kVec];
        Elem<T>::unpack(first[q], x);
        absorb<kVec, false, true>(st, x, (int)(u0 + tid + q * kRowWG), a.scale);
      }
      renew_bound();  // its barriers also publish sh.cnt == 0
#pragma unroll
      for (int q = 0; q < kRowUnroll; ++q) {
        float x[kVec];
        Elem<T>::unpack(first[q], x);
        if (max_of_raw<kVec>(x) >= early_val) {
#pragma unroll
          for (int i = 0; i < kVec; ++i) offer(x[i], sp.head + (u0 + tid + q * kRowWG) * kVec + i, early, early_val);
        }
      }
      g0 = 1;
    } else {
      __syncthreads();  // sh.cnt == 0 is visible
    }
    const int64_t g_renew = n_groups >= 8 && big_range ? 1 + (n_groups - 1) / 4 : n_groups;
    for (int64_t gi = g0; gi < n_groups; ++gi) {
      if (gi == g_renew) renew_bound();  // uniform: every lane runs the same iterations
      u32x4 v[kRowUnroll];
#pragma unroll
      for (int q = 0; q < kRowUnroll; ++q) v[q] = __builtin_nontemporal_load(p + u0 + gi * kGroup + tid + q * kRowWG);
#pragma unroll
      for (int q = 0; q < kRowUnroll; ++q) consume(v[q], u0 + gi * kGroup + tid + q * kRowWG);
    }
    for (int64_t u = u0 + n_groups * kGroup + tid; u < u1; u += kRowWG) consume(__builtin_nontemporal_load(p + u), u);
    if (tid < n_head) {
      float x[1] = {x_head};
      absorb<1, false, true>(st, x, 0, a.scale);
      offer(x_head, tid, early, early_val);
    }
    if (tid < n_tail) {
      float x[1] = {x_tail};
      absorb<1, false, true>(st, x, 0, a.scale);
      offer(x_tail, tail_e, early, early_val);
    }
  }
  int m = 0;
  bool scan = true;
  if constexpr (!CACHED) {
    lane_max = st.bi != 0x7fffffff ? st.mx : -INFINITY;  // nothing above the floor seen: -inf
    tot = block_reduce(st, a.scale, sh.red);  // valid in wave 0; its barrier also ends the offers of pass 1
    const int offered = sh.cnt;
    if (offered <= kSampCap) {
      m = offered;
      scan = false;
    } else {  // the early bound let too much through: fall back to the bound from the whole range and rescan
      __syncthreads();
      if (tid == 0) sh.cnt = 0;
      // ---- theta: k-th largest lane maximum (ranges that fit the buffer skip the bound) --------------
      if (big_range) theta = bound_from_lane_maxima(sh, lane_max, k);
      else __syncthreads();
    }
  }

  // ---- pass 2: collect every element >= theta ---------------------------------------------------
  uint64_t sorted = 0;  // wave 0, lane i < k: the (i+1)-th largest key of this range
  if constexpr (CACHED) {
    // sh.cnt is zero here: cleared before the first barrier, and again after an overflow.
    for (;;) {
      const float theta_val = theta == 0 ? -INFINITY : key_float((uint32_t)(theta >> 32));
      // Opaque to the optimiser, so that the keys and element indices below are formed where they are
      // used (rarely) instead of being hoisted out of the retry loop into a hundred live registers.
      uint32_t first_elem = (uint32_t)(sp.head + (u0 + tid) * kVec);
      asm volatile("" : "+v"(first_elem));
#pragma unroll
      for (int q = 0; q < kSampCached; ++q)
        asm volatile("" : "+v"(cached[q].x), "+v"(cached[q].y), "+v"(cached[q].z), "+v"(cached[q].w));
#pragma unroll
      for (int q = 0; q < kSampCached; ++q)
        if (u0 + tid + q * kRowWG < u1) {
          float x[kVec];
          Elem<T>::unpack(cached[q], x);
          if (max_of_raw<kVec>(x) >= theta_val) {
#pragma unroll
            for (int i = 0; i < kVec; ++i) offer(x[i], first_elem + (uint32_t)(q * kRowWG * kVec + i), theta, theta_val);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      offer(x_head, tid, theta, theta_val);
      offer(x_tail, tail_e, theta, theta_val);
      __syncthreads();
      const int offered = sh.cnt;
      if (offered <= kSampCap) {
        m = offered;
        break;
      }
      // Overflow: the k-th largest of the kSampCap keys that were kept is a strictly higher lower bound.
      __syncthreads();
      theta = select_top_k(sh, sh.a, sh.b, kSampCap, k);
      if (tid == 0) sh.cnt = 0;
      __syncthreads();
    }
    if (m <= 64) {  // the usual case: wave 0 ranks them in registers, the other waves are done
      if (wave != 0) return;
      sorted = wave_sorted_top_k(lane < m ? sh.a[lane] : 0, m, k);
    } else {
      select_top_k(sh, sh.a, sh.b, m, k);
      if (wave != 0) return;
      sorted = lane < k ? sh.top[lane] : 0;
    }
  } else {
    // sh.cnt is zero here: cleared before the first barrier, and again after an overflow.
    while (scan) {
      const float theta_val = theta == 0 ? -INFINITY : key_float((uint32_t)(theta >> 32));
      auto offer2 = [&](float x, int64_t idx) { offer(x, idx, theta, theta_val); };
      int64_t u = u0 + tid;
      for (; u + (kRowUnroll - 1) * kRowWG < u1; u += kRowUnroll * kRowWG) {
        u32x4 v[kRowUnroll];
#pragma unroll
        for (int q = 0; q < kRowUnroll; ++q) v[q] = p[u + q * kRowWG];
#pragma unroll
        for (int q = 0; q < kRowUnroll; ++q) {
          float x[kVec];
          Elem<T>::unpack(v[q], x);
          if (max_of_raw<kVec>(x) >= theta_val) {
#pragma unroll
            for (int i = 0; i < kVec; ++i) offer2(x[i], sp.head + (u + q * kRowWG) * kVec + i);
          }
        }
      }
      for (; u < u1; u += kRowWG) {
        float x[kVec];
        Elem<T>::unpack(p[u], x);
        if (max_of_raw<kVec>(x) >= theta_val) {
#pragma unroll
          for (int i = 0; i < kVec; ++i) offer2(x[i], sp.head + u * kVec + i);
        }
      }
      offer2(x_head, tid);
      offer2(x_tail, tail_e);
      __syncthreads();
      const int offered = sh.cnt;
      if (offered <= kSampCap) {
        m = offered;
        break;
      }
      // Overflow: the k-th largest of the kSampCap keys that were kept is a strictly higher lower bound.
      __syncthreads();
      theta = select_top_k(sh, sh.a, sh.b, kSampCap, k);
      if (tid == 0) sh.cnt = 0;
      __syncthreads();
    }
    select_top_k(sh, sh.a, sh.b, m, k);
    if (wave != 0) return;
    sorted = lane < k ? sh.top[lane] : 0;
  }

  finish_sample(a, sorted, r, tot, lane, a.uniforms ? a.uniforms[r] : 0.f);  // wave 0
}

// First launch of the decode form: partial statistics and cell maxima of one row's blocks [b0, b1).  Edge elements (RowSpan's
// head and tail) are left to the second launch.
template <typename T>
__global__ __launch_bounds__(kRowWG) __attribute__((amdgpu_waves_per_eu(6, 8))) void row_sample_cells_kernel(SampleArgs a) {
  touch_args(a);  // 64 x 151936 fp32 in a captured graph, both launches, 13.23 -> 13.16 us (whole calls: equal); in the pick launch, which loads cells first, it costs 0.1
  constexpr int kVec = Elem<T>::kVec;
  const int64_t r = blockIdx.x / a.splits;
  const int split = blockIdx.x % a.splits;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (!a.sel.valid(r)) return;  // outputs are written by the second launch
  const T* row = static_cast<const T*>(a.logits) + r * a.row_stride;
  const RowSpan<T> sp(row, a.V);
  const int n_blocks = (int)(a.n_cells / kRowWG);
  const int b0 = split * a.blocks_per_split;
  const int b1 = b0 + a.blocks_per_split < n_blocks ? b0 + a.blocks_per_split : n_blocks;
  float* cells = a.cells + r * a.n_cells + wave * 8 + (lane >> 3) + (lane & 7) * (kRowWG / 8);
  const u32x4 none = sizeof(T) == 4 ? u32x4{0xff800000u, 0xff800000u, 0xff800000u, 0xff800000u}   // -inf
                                    : u32x4{0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
  float mx = kMaxFloor, s = 0.f;
  for (int b = b0; b < b1; ++b) {
    const int64_t u = (int64_t)b * kCellBlock + tid;
    u32x4 v[kCellUnits];
    if ((int64_t)(b + 1) * kCellBlock <= sp.n_units) {  // uniform
#pragma unroll
      for (int q = 0; q < kCellUnits; ++q) v[q] = __builtin_nontemporal_load(sp.p + u + q * kRowWG);
    } else {
#pragma unroll
      for (int q = 0; q < kCellUnits; ++q) v[q] = u + q * kRowWG < sp.n_units ? __builtin_nontemporal_load(sp.p + u + q * kRowWG) : none;
    }
    float m[kCellUnits];
#pragma unroll
    for (int q = 0; q < kCellUnits; ++q) {
      float x[kVec];
      Elem<T>::unpack(v[q], x);
      m[q] = max_of_raw<kVec>(x);
    }
    // Opaque to the optimiser: the second sweep unpacks again instead of keeping every element in a register of its own.
#pragma unroll
    for (int q = 0; q < kCellUnits; ++q) asm volatile("" : "+v"(v[q].x), "+v"(v[q].y), "+v"(v[q].z), "+v"(v[q].w));
    const float mx_new = raw_max3(raw_max3(raw_max3(mx, m[0], m[1]), m[2], m[3]), raw_max3(m[4], m[5], m[6]), m[7]);
    const float mm = mx_new * a.scale;
    float s0 = s * fast_exp2((mx - mx_new) * a.scale), s1 = 0.f;
#pragma unroll
    for (int q = 0; q < kCellUnits; ++q) {
      float x[kVec];
      Elem<T>::unpack(v[q], x);
#pragma unroll
      for (int i = 0; i < kVec; i += 2) {
        s0 += fast_exp2(fmaf(x[i], a.scale, -mm));
        s1 += fast_exp2(fmaf(x[i + 1], a.scale, -mm));
      }
    }
    s = s0 + s1;
    mx = mx_new;
    // Cell maxima: over groups of eight lanes, all eight units at once (each register is read through DPP eight
    // instructions after it was written; the s_nop covers the first one).
    asm volatile(
        "s_nop 1\n"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %3, %3, %3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %4, %4, %4 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %5, %5, %5 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %6, %6, %6 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %7, %7, %7 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %3, %3, %3 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %4, %4, %4 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %5, %5, %5 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %6, %6, %6 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %7, %7, %7 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %2, %2, %2 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %3, %3, %3 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %4, %4, %4 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %5, %5, %5 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %6, %6, %6 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %7, %7, %7 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "s_nop 1"
        : "+v"(m[0]), "+v"(m[1]), "+v"(m[2]), "+v"(m[3]), "+v"(m[4]), "+v"(m[5]), "+v"(m[6]), "+v"(m[7]));
    float mine = m[0];  // lane j of a group keeps unit row j's maximum: every lane stores one cell
#pragma unroll
    for (int q = 1; q < kCellUnits; ++q) mine = (lane & 7) == q ? m[q] : mine;
    cells[(int64_t)b * kRowWG] = mine;
  }
  float wm = mx;
  wm = raw_max(wm, wave_exchange<0>(wm));
  wm = raw_max(wm, wave_exchange<1>(wm));
  wm = raw_max(wm, wave_exchange<2>(wm));
  wm = raw_max(wm, wave_exchange<3>(wm));
  wm = raw_max(wm, wave_exchange<4>(wm));
  wm = raw_max(wm, wave_exchange<5>(wm));
  s *= fast_exp2((mx - wm) * a.scale);
  s += wave_exchange<0>(s);
  s += wave_exchange<1>(s);
  s += wave_exchange<2>(s);
  s += wave_exchange<3>(s);
  s += wave_exchange<4>(s);
  s += wave_exchange<5>(s);
  if (lane == 0) a.part_stat[(r * a.splits + split) * kRowWaves + wave] = float2{wm, s};
}

// Second launch: one workgroup per row takes the best cells, reads them, ranks their elements and draws.  Its time is that of
// one chain of dependent steps run once per workgroup, the code fetched cold: loads come first and unconditionally, the usual
// path is short and straight, whatever does not follow from the common case sits behind a branch at its end.
// In batches of 1000 rows and more it is bound by how many rows are in flight: rows of up to 8 blocks of cells take an
// instantiation that holds 8 maxima a lane instead of 32 (53 VGPRs instead of 90), and the candidate buffers have the size the
// element type needs (fp32 18 KB of LDS instead of 34): 8 workgroups a CU instead of 4 in fp32.  Both launches, us: fp32 65536
// elements x 1400 / 2000 rows 74.9 -> 71.8, 103.7 -> 99.8, 24000 x 6000 132.9 -> 121.3, 12000 x 1000 22.2 -> 21.3; bf16 24000 x 1000
// 24.0 -> 22.8, 65536 x 700 23.9 -> 23.0; rows above 8 blocks unchanged.
template <typename T, int kHold>                 // kHold: cell maxima a lane keeps (a multiple of 8)
__global__ __launch_bounds__(kRowWG) void row_sample_pick_kernel(SampleArgs a) {
  constexpr int kVec = Elem<T>::kVec;
  constexpr int kCap = kSampPickCap<T>;
  constexpr int kStats = 64 * kRowWaves / 64;    // partial statistics per lane of wave 0 (splits <= 64)
  constexpr int kWaveCap = kCap / kRowWaves;
  __shared__ SampleLds<kCap> sh;
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k = a.top_k;
  const float* cells = a.cells + r * a.n_cells;
  const int per_lane = (int)(a.n_cells / kRowWG);
  // A lane's cells: `slot` of every block.  In a row of a single block, which may be half empty, waves are dealt every fourth
  // cell, so that all four have maxima (the bound needs some in each): bf16 rows of 12000 19.6 -> 10.1 us.
  const int slot = per_lane > 1 ? tid : lane * kRowWaves + wave;
  float c[kHold];
#pragma unroll
  for (int q0 = 0; q0 < kHold; q0 += 8) {  // eight loads at a time: up to 7 past this row's cells (the workspace has room)
    if (q0 < per_lane) {
#pragma unroll
      for (int q = q0; q < q0 + 8; ++q) c[q] = cells[slot + q * kRowWG];
    } else {
#pragma unroll
      for (int q = q0; q < q0 + 8; ++q) c[q] = -INFINITY;
    }
  }
  const int n_part = a.splits * kRowWaves;
  const float2* stats = a.part_stat + r * n_part;
  float2 part[kStats];
#pragma unroll
  for (int q = 0; q < kStats; ++q) part[q] = stats[lane + q * 64 < n_part ? lane + q * 64 : 0];
  const float uniform = a.uniforms ? a.uniforms[r] : 0.f;
  if (!a.sel.valid(r)) {
    masked_sample(a, r, tid);
    return;
  }
  const T* row = static_cast<const T*>(a.logits) + r * a.row_stride;
  const RowSpan<T> sp(row, a.V);
  // The single elements of the edges (at most 7 on either side): lanes 0 .. 7 and 8 .. 15.
  const bool edge = tid < 8 ? tid < sp.head : tid - 8 < sp.tail;
  const int64_t edge_e = tid < 8 ? tid : sp.tail_start() + (tid - 8);
  const float x_edge = edge ? Elem<T>::load1(row + edge_e) : -INFINITY;  // -inf: no candidate
  if (tid < 64) sh.b[tid] = 0;  // the ranking below reads 64 entries; published by the barriers of the bound
  if (tid == 0) sh.cnt2 = 0;
  float lane_max = -INFINITY;  // fmaxf also drops the NaN of a cell that holds nothing else
#pragma unroll
  for (int q = 0; q < kHold; ++q) c[q] = q < per_lane ? c[q] : -INFINITY;
#pragma unroll
  for (int q = 0; q < kHold; q += 2) lane_max = fmaxf(lane_max, fmaxf(c[q], c[q + 1]));
  for (int q = kHold; q < per_lane; ++q) lane_max = fmaxf(lane_max, cells[(int64_t)q * kRowWG + slot]);

  // ---- the cells at or above a lower bound of the k-th best ----------------------------------------
  uint64_t theta = bound_from_lane_maxima(sh, lane_max, k);
  float least = fmaxf(key_float((uint32_t)(theta >> 32)), -__FLT_MAX__);  // -inf is never a candidate
  // Every wave owns a quarter of the buffer and a running count that is the same in all its lanes; the lanes that pass take
  // consecutive slots by their position among the passing lanes (an LDS atomic per candidate would queue up).
  int count = 0;
  auto offer_cell = [&](float w, int q) {
    const uint64_t b = __ballot(w >= least);
    if (__builtin_expect(b == 0, 1)) return;
    const int pos = count + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
    if (w >= least && pos < kWaveCap) sh.a[wave * kWaveCap + pos] = ((uint64_t)__float_as_uint(w) << 32) | (uint32_t)(q * kRowWG + slot);
    count += __builtin_popcountll(b);
  };
#pragma unroll
  for (int q0 = 0; q0 < kHold; q0 += 8)
    if (q0 < per_lane) {
#pragma unroll
      for (int q = q0; q < q0 + 8; ++q) offer_cell(c[q], q);
    }
  for (int q = kHold; q < per_lane; ++q) offer_cell(cells[(int64_t)q * kRowWG + slot], q);
  if (lane == 0) sh.wave_cnt[wave] = count;
  __syncthreads();
  int n_wave[kRowWaves], n_best = 0;
  bool fits = true;
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) {
    n_wave[w] = sh.wave_cnt[w];
    n_best += n_wave[w];
    fits = fits && n_wave[w] <= kWaveCap;
  }

  // ---- their elements: eight lanes a cell, one load unit each -----------------------------------------
  // cells_of(j): the cell of this lane's group in round j (32 groups a round), -1 = none.  Elements at or above `least` go to
  // sh.b, consecutive slots per wave by position among the passing lanes; sh.cnt2 counts what passed, stored or not.
  const u32x4 none = sizeof(T) == 4 ? u32x4{0xff800000u, 0xff800000u, 0xff800000u, 0xff800000u}   // -inf
                                    : u32x4{0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
  const int group = tid >> 3;
  auto load_unit = [&](int64_t cell) {
    const int64_t u = cell * kCellUnits + (lane & 7);
    return cell >= 0 && u < sp.n_units ? sp.p[u] : none;
  };
  auto offer_n = [&](const float* e, auto n, auto index_of) {
    uint64_t pass[decltype(n)::value];
    int total = 0;
#pragma unroll
    for (int i = 0; i < decltype(n)::value; ++i) {
      pass[i] = __ballot(e[i] >= least);
      total += __builtin_popcountll(pass[i]);
    }
    if (total == 0) return;  // wave-uniform
    int at = 0;
    if (lane == 0) at = atomicAdd(&sh.cnt2, total);
    at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
    for (int i = 0; i < decltype(n)::value; ++i) {
      if (pass[i] == 0) continue;
      const int pos = at + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(pass[i] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)pass[i], 0u));
      if (e[i] >= least && pos < kCap) sh.b[pos] = make_key(e[i], (uint32_t)index_of(i));
      at += __builtin_popcountll(pass[i]);
    }
  };
  auto offer_unit = [&](const u32x4& v, int64_t cell) {
    float x[kVec];
    Elem<T>::unpack(v, x);
    offer_n(x, std::integral_constant<int, kVec>(), [&](int i) { return sp.head + (cell * kCellUnits + (lane & 7)) * kVec + i; });
  };
  auto offer_edge = [&]() {
    if (wave == 0 && sp.head + sp.tail > 0) offer_n(&x_edge, std::integral_constant<int, 1>(), [&](int) { return edge_e; });
  };

  RowStat st = stat_identity();
  auto merge_stats = [&]() {  // the maximum first, then every partial sum moved to it
    float mx = fmaxf(x_edge, kMaxFloor);
#pragma unroll
    for (int q = 0; q < kStats; ++q) mx = fmaxf(mx, part[q].x);  // (lanes past the end hold a copy of entry 0)
    mx = fmaxf(mx, wave_exchange<0>(mx));
    mx = fmaxf(mx, wave_exchange<1>(mx));
    mx = fmaxf(mx, wave_exchange<2>(mx));
    mx = fmaxf(mx, wave_exchange<3>(mx));
    mx = fmaxf(mx, wave_exchange<4>(mx));
    mx = fmaxf(mx, wave_exchange<5>(mx));
    float sum = fast_exp2(fmaf(x_edge, a.scale, -mx * a.scale));
#pragma unroll
    for (int q = 0; q < kStats; ++q) sum += lane + q * 64 < n_part ? part[q].y * fast_exp2((part[q].x - mx) * a.scale) : 0.f;
    sum += wave_exchange<0>(sum);
    sum += wave_exchange<1>(sum);
    sum += wave_exchange<2>(sum);
    sum += wave_exchange<3>(sum);
    sum += wave_exchange<4>(sum);
    sum += wave_exchange<5>(sum);
    st.mx = mx;
    st.s = sum;
  };
  int m = kCap + 1;
  if (__builtin_expect(n_best <= 64, 1)) {
    const int64_t c0 = group < n_best ? (int64_t)(uint32_t)region_entry(sh.a, kWaveCap, n_wave, group) : -1;
    const u32x4 v0 = load_unit(c0);
    int64_t c1 = -1;
    u32x4 v1 = none;
    if (n_best > 32) {
      if (group + 32 < n_best) c1 = (int64_t)(uint32_t)region_entry(sh.a, kWaveCap, n_wave, group + 32);
      v1 = load_unit(c1);
    }
    if (wave == 0) merge_stats();  // while the loads are under way
    offer_unit(v0, c0);
    if (n_best > 32) offer_unit(v1, c1);
    offer_edge();
    __syncthreads();
    m = sh.cnt2;
  }
  if (__builtin_expect(m > kCap, 0)) {
    // Far more cells or elements than k at or above the bound (many equal ones, or the large ones all in a few lanes): the k
    // best cells by whole keys, and the elements of those alone, which always fit.
    if (wave == 0) merge_stats();
    if (n_best <= 64 || fits) {
      __syncthreads();
      for (int i = tid; i < n_best; i += kRowWG) {
        const uint64_t raw = region_entry(sh.a, kWaveCap, n_wave, i);
        sh.b[i] = make_key(__uint_as_float((uint32_t)(raw >> 32)), (uint32_t)raw);
      }
      __syncthreads();
    } else {
      for (;;) {
        __syncthreads();
        if (tid == 0) sh.cnt = 0;
        __syncthreads();
        for (int q = 0; q < per_lane; ++q) {
          const float w = cells[(int64_t)q * kRowWG + slot];
          const uint64_t key = make_key(w, (uint32_t)(q * kRowWG + slot));
          if (w > -INFINITY && key >= theta) {
            const int pos = atomicAdd(&sh.cnt, 1);
            if (pos < kCap) sh.b[pos] = key;
          }
        }
        __syncthreads();
        n_best = sh.cnt;
        if (n_best <= kCap) break;
        // Overflow: the k-th largest of the keys that were kept is a strictly higher lower bound.
        __syncthreads();
        theta = select_top_k(sh, sh.b, sh.a, kCap, k);
      }
    }
    select_top_k(sh, sh.b, sh.a, n_best, k);
    const uint64_t kth = sh.top[k - 1], mine = sh.top[group];  // kSampMaxK = 32 cells, 32 groups
    if (kth != 0) least = key_float((uint32_t)(kth >> 32));
    __syncthreads();
    if (tid < 64) sh.b[tid] = 0;
    if (tid == 0) sh.cnt2 = 0;
    __syncthreads();
    const int64_t cell = mine != 0 ? (int64_t)key_index(mine) : -1;
    offer_unit(load_unit(cell), cell);
    offer_edge();
    __syncthreads();
    m = sh.cnt2;
  }
  uint64_t sorted;
  if (__builtin_expect(m <= 64, 1)) {
    // Four lanes a key, each counting the larger ones among 16 entries (0 past the end).
    const uint64_t key = sh.b[tid >> 2];
    const int first = (tid & 3) * 16;
    int rank = 0;
    if ((tid & 3) * 16 < m)
#pragma unroll
      for (int j = 0; j < 16; ++j) rank += sh.b[first + j] > key ? 1 : 0;
    rank += __builtin_amdgcn_update_dpp(0, rank, 0xB1, 0xF, 0xF, true);
    rank += __builtin_amdgcn_update_dpp(0, rank, 0x4E, 0xF, 0xF, true);
    if (tid < kSampMaxK) sh.top[tid] = 0;
    __syncthreads();
    if ((tid & 3) == 0 && key != 0 && rank < k) sh.top[rank] = key;
    __syncthreads();
  } else {
    select_top_k(sh, sh.b, sh.a, m, k);
  }
  if (wave != 0) return;
  sorted = lane < k ? sh.top[lane] : 0;
  finish_sample(a, sorted, r, st, lane, uniform);
}

int row_splits_for(int64_t rows, int64_t V, int vec);

// Batches that need a workspace: those whose rows are worth more than one workgroup.  They always take the decode form.
bool row_sample_needs_workspace(int64_t rows, int64_t V, int vec) {
  int64_t s = (V + 8191) / 8192;
  const int64_t most_ranges = vec == 4 ? 18000 : 6500;   // rows * ranges: ~950 fp32 rows, ~340 bf16 rows at V = 151936
  if (rows * s > most_ranges) return row_splits_for(rows, V, vec) > 1;
  // fp32 rows of a block of cells and part of a second one, by the thousand: two launches and a nearly empty workgroup a row cost
  // more than one workgroup that streams the row.  Cells / streamed, us: 8200 elements 1500 rows 24.3 / 20.0, 12000 elements
  // 1000 / 1500 / 2000 / 4000 / 6000 rows 21.3 / 23.8, 27.7 / 27.5, 35.2 / 36.4, 56.4 / 53.0, 79.4 / 72.6, 13000 elements 1500 / 4000
  // rows 28.8 / 28.6, 59.8 / 53.8; 14000 elements 2000 / 4000 rows 36.6 / 38.2, 60.4 / 58.3; 16384 elements 4000 rows 58.8 / 63.2.
  // (Ranges of 8192 elements kept in registers, the form before the cells, took 12000 elements 21.8, 28.8, 33.3, 58.5, 84.0.)
  if (vec == 4 && V <= 13312 && rows >= 1500) return false;
  const int64_t fill = (512 + rows - 1) / rows;
  if (s < fill) s = fill;
  const int64_t max_by_work = (V / vec) / (2 * kRowWG);  // >= 2 load units per lane and split
  if (s > max_by_work) s = max_by_work;
  return s > 1;
}
// Batches that take the decode form if they are given its workspace: larger bf16 ones as well, up to the largest measured
// (rows of 151936: 700 / 1000 / 1500 67 / 76 / 97 us streamed, 47 / 63 / 93 in cells; 2500 x 65536
// 89 / 72, 8000 x 32000 150 / 131).  Rows shorter than that stream faster (4000 x 16384 39 / 47, 2500 x 20000 42 / 44).  fp32 rows stream as fast as they are read either way (1000 x 151936: 114 us in cells, 108 streamed).
static bool sample_prefers_cells(int64_t rows, int64_t V, int vec) {
  if (row_sample_needs_workspace(rows, V, vec)) return true;
  return vec == 8 && V >= 32000 && rows * V <= (int64_t)1 << 28;
}

// The decode form's work split: one block of 2048 load units (32 KB) per workgroup, more only where a row would take more than
// 64 workgroups.  Measured with 512 to 4096 workgroups in the launch: equal up to ~128 rows of 151936, from there on one block
// is the fastest (400 / 1000 rows fp32 51-55 / 122-124 us against 49.8 / 114, 700 rows bf16 50-61 against 46.5), also
// against a variant that requests the next block before it takes in the present one.
struct CellPlan {
  int splits, blocks_per_split;
  int64_t n_cells;
};
static CellPlan cell_plan(int64_t V, int vec) {
  const int64_t blocks = (V / vec + kCellBlock - 1) / kCellBlock;
  const int64_t per = (blocks + 63) / 64;
  return CellPlan{(int)((blocks + per - 1) / per), (int)per, blocks * kRowWG};
}

static size_t align256s(size_t b) { return (b + 255) & ~(size_t)255; }
size_t row_sample_workspace_bytes(int64_t rows, int64_t V, int dtype_vec, int top_k) {
  (void)top_k;
  if (!sample_prefers_cells(rows, V, dtype_vec)) return 0;
  const CellPlan p = cell_plan(V, dtype_vec);
  // (the second launch reads up to 7 x 256 cells past a row's own)
  return align256s((size_t)(rows * p.n_cells + 7 * kRowWG) * sizeof(float)) + align256s((size_t)rows * p.splits * kRowWaves * sizeof(float2));
}

hipError_t row_sample_launch(const void* logits, int dtype, int64_t rows, int64_t V, int64_t row_stride,
                             const float* uniforms, const RowSel& sel, float temperature, int top_k,
                             int32_t* out_token, float* out_lp, float* out_lse, int32_t* out_argmax,
                             int32_t* out_topk_idx, float* out_topk_logit, const DecodeState& state, void* workspace,
                             hipStream_t stream) {
  const int esize = dtype == 0 ? 4 : 2;
  const int vec = 16 / esize;
  SampleArgs a{};
  a.logits = logits;
  a.uniforms = uniforms;
  a.sel = sel;
  a.out_token = out_token;
  a.out_lp = out_lp;
  a.out_lse = out_lse;
  a.out_argmax = out_argmax;
  a.out_topk_idx = out_topk_idx;
  a.out_topk_logit = out_topk_logit;
  a.active = state.active;
  a.out_next = state.out_next;
  a.idle_token = state.idle_token;
  a.stop_token = state.stop_token;
  a.V = V;
  a.row_stride = row_stride;
  a.top_k = top_k;
  a.scale = kLog2e / temperature;
  const dim3 block(kRowWG);
  if (workspace && sample_prefers_cells(rows, V, vec)) {
    const CellPlan p = cell_plan(V, vec);
    a.cells = static_cast<float*>(workspace);
    a.part_stat = reinterpret_cast<float2*>(static_cast<char*>(workspace) + align256s((size_t)(rows * p.n_cells + 7 * kRowWG) * sizeof(float)));
    a.splits = p.splits;
    a.blocks_per_split = p.blocks_per_split;
    a.n_cells = p.n_cells;
    const dim3 grid((unsigned)(rows * p.splits));
    if (dtype == 0) hipLaunchKernelGGL((row_sample_cells_kernel<float>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((row_sample_cells_kernel<uint16_t>), grid, block, 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const bool few = p.n_cells <= 8 * kRowWG;
    const dim3 pick_grid((unsigned)rows);
    if (dtype == 0 && few) hipLaunchKernelGGL((row_sample_pick_kernel<float, 8>), pick_grid, block, 0, stream, a);
    else if (dtype == 0) hipLaunchKernelGGL((row_sample_pick_kernel<float, 32>), pick_grid, block, 0, stream, a);
    else if (few) hipLaunchKernelGGL((row_sample_pick_kernel<uint16_t, 8>), pick_grid, block, 0, stream, a);
    else hipLaunchKernelGGL((row_sample_pick_kernel<uint16_t, 32>), pick_grid, block, 0, stream, a);
    return hipGetLastError();
  }
  const dim3 grid((unsigned)rows);
  // (two units' worth of elements: every row then holds a whole unit at any phase)
  const bool cached = V >= 2 * vec && V / vec <= (int64_t)kSampCached * kRowWG;
  if (dtype == 0) {
    if (cached) hipLaunchKernelGGL((row_sample_kernel<float, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((row_sample_kernel<float, false>), grid, block, 0, stream, a);
  } else {
    if (cached) hipLaunchKernelGGL((row_sample_kernel<uint16_t, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((row_sample_kernel<uint16_t, false>), grid, block, 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace tome
