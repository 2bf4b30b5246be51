// Second pass of the full log-softmax matrix: out[r, j] = T(x[r, j] * inv_temp) - T(lse_r).
//
// The reference kernel (mlx-impl/model.py:57-65) computes the difference in the I/O dtype T:
// both operands are first cast to T, and for bf16 the result is rounded once more.  The row
// logsumexp comes from row_logprob_kernel, so the matrix is read twice and written once
// where the reference reads it three times.  Rows that row_logprob_kernel split over several
// workgroups are merged here, by every workgroup of the row for itself (a few partials), which
// saves the launch of a merge kernel between the two passes.
//
// Rows of 16384 elements and more need neither the second launch nor (most of) the second read, except in small batches: a
// 1024-lane workgroup holds a bf16 row of up to 155648 elements in its registers (full_log_softmax_onepass_kernel) and an
// fp32 row of up to 106496 in registers and LDS (full_log_softmax_row_kernel, which reads only the rest again).
#include "row_common.hpp"

#include <type_traits>

namespace tome {

constexpr int kFullWG = 256;
constexpr int kFullUnroll = 4;

struct FullArgs {
  const void* in;
  void* out;
  float* row_lse;              // read when splits == 1; written (by the row's first workgroup) otherwise
  const RowPartial* partials;  // [rows, splits] when splits > 1
  int splits;
  float scale;                 // log2(e) / temperature, as the pass that made the partials used it
  int64_t V;
  int64_t in_stride;
  int64_t out_stride;
  int chunks;  // workgroups per row
  float inv_temp;
};

__device__ __forceinline__ float bf16_rt(float f) { return bf16_bits_to_f32(f32_to_bf16_bits(f)); }

// Two elements: round the scaled logits to bf16, subtract, round again (v_cvt_pk_bf16_f32 twice; the
// software rounding this replaces cost more VALU time than the memory stream left room for).
__device__ __forceinline__ uint32_t sub_pack_bf16(uint32_t u, float inv_temp, float lse_t) {
  const uint32_t z = pack_bf16(__fmul_rn(bf16_lo(u), inv_temp), __fmul_rn(bf16_hi(u), inv_temp));
  return pack_bf16(__fsub_rn(bf16_lo(z), lse_t), __fsub_rn(bf16_hi(z), lse_t));
}

// 16-byte units are laid out from the OUTPUT row's first 16-byte boundary: stores are then whole aligned units at any
// vocabulary size and stride.  Input rows at another phase (a strided view) are read with the same loads at the alignment
// of their elements.  Against element-wise loads and stores, which every row off a 16-byte boundary took (1024 rows of
// 128258, both passes): fp32 508 -> 245 us, bf16 (now on the one-pass kernel) 458 -> 107 us.
typedef u32x4 u32x4_any __attribute__((aligned(2)));
template <typename Offset>
__device__ __forceinline__ u32x4 load_unit(const void* row, Offset byte) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(static_cast<const char*>(row) + byte));
}

// One load unit / one element of the result: T(x * inv_temp) - T(lse), rounded where T rounds.
template <typename T>
__device__ __forceinline__ u32x4 log_softmax_unit(const u32x4& v, float inv_temp, float lse_t) {
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (sizeof(T) == 2) o[i] = sub_pack_bf16(v[i], inv_temp, lse_t);
    else o[i] = __float_as_uint(__fsub_rn(__fmul_rn(__uint_as_float(v[i]), inv_temp), lse_t));
  }
  return o;
}
template <typename T>
__device__ __forceinline__ T log_softmax_one(T x, float inv_temp, float lse_t) {
  if constexpr (sizeof(T) == 2) return f32_to_bf16_bits(__fsub_rn(bf16_rt(__fmul_rn(bf16_bits_to_f32(x), inv_temp)), lse_t));
  else return __fsub_rn(__fmul_rn(x, inv_temp), lse_t);
}

template <bool BF16, int UNROLL = kFullUnroll>
__global__ __launch_bounds__(kFullWG) void full_log_softmax_kernel(FullArgs a) {
  int64_t r = blockIdx.x;  // (no division for short rows, as in the row kernel)
  int chunk = 0;
  if (a.chunks > 1) {
    r = blockIdx.x / a.chunks;
    chunk = blockIdx.x % a.chunks;
  }
  float lse;
  if (a.splits > 1) {  // merge the row's partials (at most 64: one per lane of wave 0)
    __shared__ float lse_sh;
    if (threadIdx.x < 64) {
      RowStat st = stat_identity();
      if ((int)threadIdx.x < a.splits) {
        const RowPartial p = a.partials[r * a.splits + threadIdx.x];
        st = RowStat{p.mx, p.s, p.w, p.bi};
      }
      stat_wave_reduce(st, a.scale);
      if (threadIdx.x == 0) {
        lse_sh = (st.mx * a.scale + fast_log2(st.s)) * kLn2;  // as finish_row forms it
        if (chunk == 0) a.row_lse[r] = lse_sh;
      }
    }
    __syncthreads();
    lse = lse_sh;
  } else {
    lse = a.row_lse[r];
  }
  typedef typename std::conditional<BF16, uint16_t, float>::type T;
  const T* in_row = static_cast<const T*>(a.in) + r * a.in_stride;
  T* out_row = static_cast<T*>(a.out) + r * a.out_stride;
  const RowSpan<T> sp(out_row, a.V);
  const int64_t n_units = sp.n_units;
  int64_t u0 = 0, u1 = n_units;
  if (a.chunks > 1) {
    const int per = ((int)n_units + a.chunks - 1) / a.chunks;
    u0 = (int64_t)per * chunk;
    u1 = u0 + per < n_units ? u0 + per : n_units;
  }
  const float lse_t = BF16 ? bf16_rt(lse) : lse;

  const T* src = in_row + sp.head;
  u32x4* dst = reinterpret_cast<u32x4*>(out_row + sp.head);
  auto convert = [&](const u32x4& v) { return log_softmax_unit<T>(v, a.inv_temp, lse_t); };
  int64_t u = u0 + threadIdx.x;
  for (; u + (UNROLL - 1) * kFullWG < u1; u += UNROLL * kFullWG) {  // several 16-byte loads in flight per lane
    u32x4 v[UNROLL];
#pragma unroll
    for (int q = 0; q < UNROLL; ++q) v[q] = load_unit(src, (u + q * kFullWG) * 16);
#pragma unroll
    for (int q = 0; q < UNROLL; ++q) __builtin_nontemporal_store(convert(v[q]), dst + u + q * kFullWG);
  }
  for (; u < u1; u += kFullWG) __builtin_nontemporal_store(convert(load_unit(src, u * 16)), dst + u);
  auto single = [&](int64_t e) { out_row[e] = log_softmax_one<T>(in_row[e], a.inv_temp, lse_t); };
  if (chunk == 0 && (int)threadIdx.x < sp.head) single(threadIdx.x);
  if (chunk == a.chunks - 1 && (int)threadIdx.x < sp.tail) single(sp.tail_start() + threadIdx.x);
}

// ---- one pass for bf16 rows that fit a workgroup's registers ----------------------------------------
// A 1024-lane workgroup (one per CU) holds a whole row in registers - up to CH 16-byte units per lane, all requested
// together - and writes T(x * inv_temp) - T(lse) from the same registers: the matrix is read ONCE and written once.
// With a single workgroup on the CU nothing else covers its arithmetic, so every lane keeps a running (maximum, sum) of
// its own and takes in each unit as it arrives (the row kernel's online update) instead of a sweep for the maximum, a
// barrier and a sweep for the sum after the last byte has landed; the lanes' states are merged through one barrier.
//
// Rows of up to 65536 elements need 64 registers a lane, so that two workgroups share a CU and one's loads run under the
// other's arithmetic: batches of more than 256 rows take an instantiation held to that (at 69 registers, one workgroup a CU:
// 512 / 1024 / 2048 rows of 32000 13.4 -> 11.1, 26.3 -> 23.9, 51.7 -> 44.9 us, 4096 x 16384 65.4 -> 51.2, 512 x 65536 25.2 -> 22.2).
// Smaller batches have a CU per row and are 0.1 us faster without the limit.
template <int CH, int WAVES>  // WAVES per SIMD: 4, or 8 for two workgroups on a CU
__global__ __launch_bounds__(1024, WAVES) void full_log_softmax_onepass_kernel(FullArgs a) {
  constexpr int kWaves = 16;
  __shared__ float red_m[kWaves], red_s[kWaves];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint16_t* in_row = static_cast<const uint16_t*>(a.in) + r * a.in_stride;
  uint16_t* out_row = static_cast<uint16_t*>(a.out) + r * a.out_stride;
  const RowSpan<uint16_t> sp(out_row, a.V);
  const uint16_t* src = in_row + sp.head;
  u32x4* dst = reinterpret_cast<u32x4*>(out_row + sp.head);
  const int n_units = (int)sp.n_units;
  // single elements in front of the first whole unit and after the last one: one per lane of the first wave
  const int n_edge = sp.head + sp.tail;
  const int edge = tid < sp.head ? tid : (int)sp.tail_start() + tid - sp.head;
  const float scale = a.scale;
  u32x4 v[CH];
#pragma unroll
  for (int q = 0; q < CH; ++q) {  // unconditional (clamped) loads; a whole unit exists (checked on the host)
    const int u = tid + q * 1024;
    if constexpr (WAVES == 8) v[q] = load_unit(src, (uint32_t)min(u, n_units - 1) * 16u);  // (64 registers without a spill)
    else v[q] = load_unit(src, (int64_t)(u < n_units ? u : 0) * 16);
  }
  // the lane's running maximum (floored like every kernel of this path) and sum of 2^((x - maximum) * scale)
  float lm = kMaxFloor, ls = 0.f;
#pragma unroll
  for (int q = 0; q < CH; ++q)
    if (tid + q * 1024 < n_units) {
      float x[8];
      Elem<uint16_t>::unpack(v[q], x);
      const float nm = raw_max3(raw_max3(x[0], x[1], x[2]), raw_max3(x[3], x[4], x[5]), raw_max3(lm, x[6], x[7]));
      const float m = nm * scale;
      float s0 = ls * fast_exp2((lm - nm) * scale), s1 = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        s0 += fast_exp2(fmaf(x[i], scale, -m));
        s1 += fast_exp2(fmaf(x[i + 1], scale, -m));
      }
      ls = s0 + s1;
      lm = nm;
    }
  if (tid < n_edge) {  // (V not a multiple of 8) fetched here, so that no wait stands in front of the sweep
    const float x = bf16_bits_to_f32(in_row[edge]);
    const float nm = fmaxf(lm, x);
    ls = ls * fast_exp2((lm - nm) * scale) + fast_exp2(fmaf(x, scale, -nm * scale));
    lm = nm;
  }
  auto merge = [&](float om, float os) {
    const float nm = fmaxf(lm, om);
    ls = ls * fast_exp2((lm - nm) * scale) + os * fast_exp2((om - nm) * scale);
    lm = nm;
  };
  merge(wave_exchange<0>(lm), wave_exchange<0>(ls));
  merge(wave_exchange<1>(lm), wave_exchange<1>(ls));
  merge(wave_exchange<2>(lm), wave_exchange<2>(ls));
  merge(wave_exchange<3>(lm), wave_exchange<3>(ls));
  merge(wave_exchange<4>(lm), wave_exchange<4>(ls));
  merge(wave_exchange<5>(lm), wave_exchange<5>(ls));
  if (lane == 0) {
    red_m[wave] = lm;
    red_s[wave] = ls;
  }
  __syncthreads();
  float mx = red_m[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, red_m[w]);
  float sum = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) sum += red_s[w] * fast_exp2((red_m[w] - mx) * scale);
  const float lse = (mx * scale + fast_log2(sum)) * kLn2;
  if (tid == 0) a.row_lse[r] = lse;
  const float lse_t = bf16_rt(lse);
  if (a.inv_temp == 1.0f) {  // the usual call: T(x * 1) is x itself, one rounding and two operations per pair fewer
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int u = tid + q * 1024;
      if (u < n_units) {
        u32x4 o;
        o.x = pack_bf16(__fsub_rn(bf16_lo(v[q].x), lse_t), __fsub_rn(bf16_hi(v[q].x), lse_t));
        o.y = pack_bf16(__fsub_rn(bf16_lo(v[q].y), lse_t), __fsub_rn(bf16_hi(v[q].y), lse_t));
        o.z = pack_bf16(__fsub_rn(bf16_lo(v[q].z), lse_t), __fsub_rn(bf16_hi(v[q].z), lse_t));
        o.w = pack_bf16(__fsub_rn(bf16_lo(v[q].w), lse_t), __fsub_rn(bf16_hi(v[q].w), lse_t));
        __builtin_nontemporal_store(o, dst + u);
      }
    }
  } else {
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int u = tid + q * 1024;
      if (u < n_units) {
        u32x4 o;
        o.x = sub_pack_bf16(v[q].x, a.inv_temp, lse_t);
        o.y = sub_pack_bf16(v[q].y, a.inv_temp, lse_t);
        o.z = sub_pack_bf16(v[q].z, a.inv_temp, lse_t);
        o.w = sub_pack_bf16(v[q].w, a.inv_temp, lse_t);
        __builtin_nontemporal_store(o, dst + u);
      }
    }
  }
  if (tid < n_edge) {
    out_row[edge] = log_softmax_one<uint16_t>(in_row[edge], a.inv_temp, lse_t);
  }
}

// ---- one launch for fp32 rows (and bf16 rows too long for the registers) -----------------------------
// As above, a 1024-lane workgroup owns a row and the CU; of the row's 16-byte units a lane keeps the first REG in registers
// and the next STASH in LDS, and only what is left over - 11 of 37 units a lane for a row of 151936 fp32 - is read a second
// time, right after it was first read: those loads come last in the first sweep and keep the default cache policy, so the
// L2 and the memory-side cache serve them again.  RING loads are in flight behind the register units.  HBM-bound: 1024 x 151936
// fp32 289 -> 235 us (5.3 TB/s of the 2 * V * 4 bytes a row cannot do without, where the two launches read the matrix twice),
// 2500 rows 720 -> 577, 128 rows 42 -> 29.4, 64 rows 24.6 -> 22.3; 1024 x 50256 102 -> 75; bf16 1024 x 160000 159 -> 123.
// 17 + 9 units is what 128 registers (no spills) and 160 KB of LDS hold; 18 + 8, 19 + 9 and 20 + 8 spill and measured 0-2 %
// slower.
template <typename T, int REG, int STASH, int RING>
__global__ __launch_bounds__(1024) void full_log_softmax_row_kernel(FullArgs a) {
  constexpr int kWaves = 16, kVec = Elem<T>::kVec;
  static_assert(STASH % RING == 0, "the ring of loads in flight is refilled in whole turns");
  __shared__ u32x4 stash[STASH > 0 ? STASH * 1024 : 1];
  __shared__ float red_m[kWaves], red_s[kWaves];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* in_row = static_cast<const T*>(a.in) + r * a.in_stride;
  T* out_row = static_cast<T*>(a.out) + r * a.out_stride;
  const RowSpan<T> sp(out_row, a.V);
  const T* src = in_row + sp.head;
  char* dst = reinterpret_cast<char*>(out_row + sp.head);
  const int n_units = (int)sp.n_units;
  const int n_edge = sp.head + sp.tail;  // single elements at the row's ends: one per lane of the first wave
  const int edge = tid < sp.head ? tid : (int)sp.tail_start() + tid - sp.head;
  const float scale = a.scale;
  auto unit_of = [&](int q) { return tid + q * 1024; };
  auto inside = [&](int u) { return (uint32_t)(u < n_units ? u : 0) * 16u; };  // unit 0 exists; rows below 4 GiB (host)

  float lm = kMaxFloor, ls = 0.f;  // the lane's running maximum and sum of 2^((x - maximum) * scale)
  auto take = [&](const u32x4& v) {
    float x[kVec];
    Elem<T>::unpack(v, x);
    float nm = lm;
#pragma unroll
    for (int i = 0; i < kVec; i += 2) nm = raw_max3(nm, x[i], x[i + 1]);
    const float m = nm * scale;
    float s0 = ls * fast_exp2((lm - nm) * scale), s1 = 0.f;
#pragma unroll
    for (int i = 0; i < kVec; i += 2) {
      s0 += fast_exp2(fmaf(x[i], scale, -m));
      s1 += fast_exp2(fmaf(x[i + 1], scale, -m));
    }
    ls = s0 + s1;
    lm = nm;
  };

  u32x4 v[REG];
#pragma unroll
  for (int q = 0; q < REG; ++q) v[q] = load_unit(src, inside(unit_of(q)));
  const int n_rounds = STASH > 0 ? (n_units - REG * 1024 + RING * 1024 - 1) / (RING * 1024) : 0;  // turns of the ring (<= 0: none)
  u32x4 t[RING];
  if constexpr (STASH > 0) {
#pragma unroll
    for (int j = 0; j < RING; ++j) t[j] = load_unit(src, inside(unit_of(REG + j)));
  }
#pragma unroll
  for (int q = 0; q < REG; ++q)
    if (unit_of(q) < n_units) take(v[q]);
  if constexpr (STASH > 0) {
    for (int g = 0; g < n_rounds; ++g) {
#pragma unroll
      for (int j = 0; j < RING; ++j) {
        const int q = REG + g * RING + j;
        if (unit_of(q) < n_units) take(t[j]);
        if (g < STASH / RING) stash[(g * RING + j) * 1024 + tid] = t[j];
        const uint32_t next = inside(unit_of(q + RING));
        if (g + 1 < STASH / RING) t[j] = load_unit(src, next);
        else t[j] = *reinterpret_cast<const u32x4_any*>(reinterpret_cast<const char*>(src) + next);
      }
    }
  }
  if (tid < n_edge) {
    const float x = Elem<T>::load1(in_row + edge);
    const float nm = fmaxf(lm, x);
    ls = ls * fast_exp2((lm - nm) * scale) + fast_exp2(fmaf(x, scale, -nm * scale));
    lm = nm;
  }
  auto merge = [&](float om, float os) {
    const float nm = fmaxf(lm, om);
    ls = ls * fast_exp2((lm - nm) * scale) + os * fast_exp2((om - nm) * scale);
    lm = nm;
  };
  merge(wave_exchange<0>(lm), wave_exchange<0>(ls));
  merge(wave_exchange<1>(lm), wave_exchange<1>(ls));
  merge(wave_exchange<2>(lm), wave_exchange<2>(ls));
  merge(wave_exchange<3>(lm), wave_exchange<3>(ls));
  merge(wave_exchange<4>(lm), wave_exchange<4>(ls));
  merge(wave_exchange<5>(lm), wave_exchange<5>(ls));
  if (lane == 0) {
    red_m[wave] = lm;
    red_s[wave] = ls;
  }
  // the first turn of the second read is on its way while the lanes meet
  constexpr int kKept = REG + STASH;
  const int n_again = STASH > 0 ? n_rounds - STASH / RING : 0;
  auto load_again = [&](int g) {
#pragma unroll
    for (int j = 0; j < RING; ++j) t[j] = load_unit(src, inside(unit_of(kKept + g * RING + j)));
  };
  if constexpr (STASH > 0) {
    if (n_again > 0) load_again(0);
  }
  __syncthreads();
  float mx = red_m[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, red_m[w]);
  float sum = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) sum += red_s[w] * fast_exp2((red_m[w] - mx) * scale);
  const float lse = (mx * scale + fast_log2(sum)) * kLn2;
  if (tid == 0) a.row_lse[r] = lse;
  const float lse_t = sizeof(T) == 2 ? bf16_rt(lse) : lse;
  auto put = [&](const u32x4& x, int u) {
    if (u < n_units) __builtin_nontemporal_store(log_softmax_unit<T>(x, a.inv_temp, lse_t), reinterpret_cast<u32x4*>(dst + (uint32_t)u * 16u));
  };
#pragma unroll
  for (int q = 0; q < REG; ++q) put(v[q], unit_of(q));
  if constexpr (STASH > 0) {
    for (int g = 0; g < n_again; ++g) {
#pragma unroll
      for (int j = 0; j < RING; ++j) put(t[j], unit_of(kKept + g * RING + j));
      if (g + 1 < n_again) load_again(g + 1);
    }
    const int n_stash = n_rounds < STASH / RING ? n_rounds * RING : STASH;
    for (int i = 0; i < n_stash; ++i) put(stash[i * 1024 + tid], unit_of(REG + i));
  }
  if (tid < n_edge) out_row[edge] = log_softmax_one<T>(in_row[edge], a.inv_temp, lse_t);
}

constexpr int kOnePassUnits = 19;  // 16-byte units per lane: 1024 lanes hold 155648 bf16 elements
constexpr int64_t kOneLaunchMaxV = 524288;

// Whether the one-launch kernels take this call: a row long enough to keep most of a workgroup's 1024 lanes busy, and enough
// rows.  One workgroup per row leaves most of the chip idle on a decode-sized batch, but it is ONE launch where the two-pass
// form is two: rows of up to 40960 elements always come here (16 rows of 16384 / 32000: 4.3 / 5.4 us against 6.8 / 7.9),
// longer ones from V / 3000 rows on.  Measured crossovers, bf16: 65536 elements ~24 rows (16 rows 7.5 against 7.0 us, 32 rows
// 7.5 against 8.0), 131072 ~60 rows (32 rows 12.1 against 8.7, 64 rows 12.4 against 12.8), 151936 ~44 rows (32 / 48 / 64 rows:
// 13.2 / 13.3 / 13.4 against 11.6 / 14.3 / 16.5); fp32: 65536 ~22 rows (24 rows 9.2 against 9.9), 100000 ~32 (13.3 against
// 13.5), 128256 ~42 (48 rows 18.1 against 18.8), 151936 ~54 (48 / 64 rows 21.5 / 22.2 against 20.4 / 24.6).  bf16 rows above the
// one-pass kernel's 155648 elements start lower down the same curve: 160000 ~66 rows (64 / 96 rows 17.4 / 18.1 against
// 17.1 / 22.3).  Above 262144 elements most of a row is read twice here as well, and an uneven last round of rows costs more:
// 500000 fp32, 300 / 1024 / 2500 rows 304 / 908 / 2210 against 292 / 988 / 2441 (bf16 157 / 433 / 1025 against 149 / 540 / 1480);
// 1000000 is equal, and left to the two passes.
bool full_log_softmax_one_pass(int dtype, int64_t rows, int64_t V) {
  if (V < 16384 || V > kOneLaunchMaxV) return false;
  int64_t per_row = 3000;
  if (dtype == 1 && V / 8 > (int64_t)kOnePassUnits * 1024) per_row = 2400;
  if (V > 262144) per_row = 1000;
  return V <= 40960 || rows * per_row >= V;
}

hipError_t full_log_softmax_onepass_launch(const void* in, void* out, int dtype, int64_t rows, int64_t V, int64_t in_stride,
                                           int64_t out_stride, float temperature, float* row_lse, hipStream_t stream) {
  FullArgs a{};
  a.in = in;
  a.out = out;
  a.row_lse = row_lse;
  a.splits = 1;
  a.scale = kLog2e / temperature;
  a.V = V;
  a.in_stride = in_stride;
  a.out_stride = out_stride;
  a.chunks = 1;
  a.inv_temp = 1.0f / temperature;
  const dim3 grid((unsigned)rows), block(1024);
  // Lanes hold 8, 13 or 20 units, or 17 + 9 and read the rest again.  13 instead of 20 where it fits spares the requests of the
  // units that are not there (64 / 128 / 300 rows of 40000 fp32: 7.3 / 8.5 / 19.8 against 8.2 / 9.3 / 21.2 us; 53248: 8.4 / 10.7 /
  // 25.3 against 9.0 / 11.2 / 25.9), but streams large batches slower (2500 x 53248: 186 against 181 us, 1024 rows 78.3 / 76.8).
  if (dtype == 0) {
    if (V / 4 <= 8 * 1024) hipLaunchKernelGGL((full_log_softmax_row_kernel<float, 8, 0, 1>), grid, block, 0, stream, a);
    else if (V / 4 <= 13 * 1024 && rows <= 512) hipLaunchKernelGGL((full_log_softmax_row_kernel<float, 13, 0, 1>), grid, block, 0, stream, a);
    else if (V / 4 <= 20 * 1024) hipLaunchKernelGGL((full_log_softmax_row_kernel<float, 20, 0, 1>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((full_log_softmax_row_kernel<float, 17, 9, 3>), grid, block, 0, stream, a);
  } else if (V / 8 > (int64_t)kOnePassUnits * 1024) {
    hipLaunchKernelGGL((full_log_softmax_row_kernel<uint16_t, 17, 9, 3>), grid, block, 0, stream, a);
  } else if (V / 8 > 8 * 1024) {
    hipLaunchKernelGGL((full_log_softmax_onepass_kernel<kOnePassUnits, 4>), grid, block, 0, stream, a);
  } else if (rows > 256) {
    hipLaunchKernelGGL((full_log_softmax_onepass_kernel<8, 8>), grid, block, 0, stream, a);
  } else {
    hipLaunchKernelGGL((full_log_softmax_onepass_kernel<8, 4>), grid, block, 0, stream, a);
  }
  return hipGetLastError();
}

// Second pass.  `splits` > 1: the rows' partials (RowPartial [rows, splits]) are merged here and the merged lse is
// also written to row_lse; splits == 1: row_lse already holds it.
hipError_t full_log_softmax_launch(const void* in, void* out, int dtype, int64_t rows, int64_t V,
                                   int64_t in_stride, int64_t out_stride, float temperature,
                                   float* row_lse, const void* partials, int splits, hipStream_t stream) {
  const int esize = dtype == 0 ? 4 : 2;
  const int vec = 16 / esize;
  FullArgs a;
  a.in = in;
  a.out = out;
  a.row_lse = row_lse;
  a.partials = static_cast<const RowPartial*>(partials);
  a.splits = splits;
  a.scale = kLog2e / temperature;
  a.V = V;
  a.in_stride = in_stride;
  a.out_stride = out_stride;
  a.inv_temp = 1.0f / temperature;  // the reference multiplies by 1/temp (model.py:27)
  const int64_t units = V / vec;
  // Many short workgroups stream a read + write mix best, as long as each still issues a few loads per lane.  bf16
  // rows (a batch too small or rows too long for the one-pass kernel): four loads per lane and pass, aiming at 65536
  // workgroups (against 4096: 4096 x 151936 bf16 655 -> 633 us, both passes included).  fp32 rows: workgroups of ONE pass
  // of two loads per lane - of one load per lane for matrices above 3/4 GB, the size up to which the first pass leaves the
  // rows in the caches (both passes, rows of 151936 fp32, four / two / one load: 64 rows 24.4 / 24.2 / 26.6 us, 1024 rows
  // 296 / 288 / 295, 2048 rows 629 / 618 / 588, 4096 rows 1370 / 1227 / 1168; rows of 32000: 4096 rows - / 248 / 253,
  // 8192 rows - / 503 / 491; rows of 65536: 2048 rows - / 254 / 256, 4096 rows - / 501 / 496).
  int64_t chunks = (65536 + rows - 1) / rows;
  int64_t by_work = units / (kFullUnroll * kFullWG);
  const int f32_unroll = (double)rows * (double)V * 4.0 > 768.0 * 1024 * 1024 ? 1 : 2;
  if (dtype == 0) {
    chunks = by_work = units / (f32_unroll * kFullWG);
  }
  if (chunks > by_work) chunks = by_work;
  if (chunks < 1) chunks = 1;
  a.chunks = (int)chunks;
  const dim3 grid((unsigned)(rows * chunks)), block(kFullWG);
  if (dtype != 0) hipLaunchKernelGGL(full_log_softmax_kernel<true>, grid, block, 0, stream, a);
  else if (f32_unroll == 1) hipLaunchKernelGGL((full_log_softmax_kernel<false, 1>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((full_log_softmax_kernel<false, 2>), grid, block, 0, stream, a);
  return hipGetLastError();
}

}  // namespace tome
