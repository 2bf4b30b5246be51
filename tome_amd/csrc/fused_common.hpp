// What the sweep kernels of the fused lm_head + log-softmax share: arguments, partial records, the work decomposition and
// the fold of a 16x16 MFMA accumulator tile into the running row states.
#pragma once
#include "common.hpp"
#include "fused_plan.hpp"
#include <atomic>
#include <type_traits>

namespace tome {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The same on the device, by one whole wave: lane i prices tile i, lane c c + 1 splits.
__device__ inline FusedSchedule fused_schedule_wave(int n_valid, const FusedShape& sh, int lane) {
  int tile = __builtin_ctz(sh.tiles);
  if (!fused_one_tile(sh)) {  // the DMA kernel's eight
    const int i = lane & 7;
    const float c = fused_tile_allowed(sh, n_valid, i) ? fused_tile_cost(sh, n_valid, i) : 3e38f;
    // positive floats order like their bits; the last three carry the tile
    unsigned key = (__float_as_uint(c) & ~7u) | (unsigned)i;
    const unsigned a = (unsigned)wave_exchange<0>((int)key);
    key = a < key ? a : key;
    const unsigned b = (unsigned)wave_exchange<1>((int)key);
    key = b < key ? b : key;
    const unsigned d = (unsigned)wave_exchange<2>((int)key);
    key = d < key ? d : key;
    tile = __builtin_amdgcn_readfirstlane((int)(key & 7u));
  }
  FusedSchedule s;
  if (fused_schedule_begin(s, n_valid, sh, tile)) {
    const int upt = s.unit32 == 1 ? 8 : 1, n_vtiles = (s.n_vunits + upt - 1) / upt, c = lane + 1;
    int64_t cost = c <= kSplitCandidates && c <= n_vtiles ? fused_split_cost(s.n_ttiles, c, sh.slots, s.n_vunits, upt) : INT64_MAX;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int64_t o = __shfl_xor(cost, off, 64);
      cost = o < cost ? o : cost;
    }
    s.n_splits = (int)(cost & 63);
    s.n_wg = s.n_ttiles * s.n_splits;
  }
  return s;
}

// Workgroup id -> (token tile, vocab split).  The hardware deals consecutive workgroup ids round-robin
// over the 8 XCDs, each with its own L2; XCD x is given the contiguous logical ids
// [x * per, (x + 1) * per), and logical ids run over blocks of <= 8 splits, token tile by token tile,
// so that the workgroups resident on an XCD at any time share token tiles AND vocab ranges.
__device__ __forceinline__ bool fused_locate(const FusedSchedule& s, int bid, int& ttile, int& split) {
  const int per = (s.n_wg + 7) >> 3;
  const int li = bid >> 3;
  int g = (bid & 7) * per + li;
  if (li >= per || g >= s.n_wg) return false;  // the grid is sized for the worst case over n_valid
  const int nb = (s.n_splits + 7) >> 3, base = s.n_splits / nb, rem = s.n_splits % nb;
  int s0 = 0, w = base;
  for (int sb = 0; sb < nb; ++sb) {
    w = base + (sb < rem ? 1 : 0);
    const int cnt = s.n_ttiles * w;
    if (g < cnt) break;
    g -= cnt;
    s0 += w;
  }
  ttile = g / w;
  split = s0 + g % w;
  return true;
}

struct FusedArgs {
  // What a workgroup needs to find its work comes first, in one cache line: a fresh launch misses on its arguments.
  const int32_t* n_valid;    // device scalar, or nullptr = n_tokens
  const FusedSchedule* sched_dev;  // written by compact_rows_kernel next to n_valid, or nullptr = `sched`
  FusedSchedule sched;       // host-computed schedule (no mask)
  int n_tokens;
  int H;
  int V;
  float scale;               // log2(e) / temperature
  const char* hidden;
  const char* weight;
  RowSel sel;                // its targets (the mask went into row_index)
  const int32_t* row_index;  // compacted valid rows (position -> row of targets / outputs), or nullptr = identity
  const int32_t* hidden_index;  // position -> row of `hidden`: row_index, the caller's row list, or nullptr when hidden is already compact
  int n_rows;                   // rows of `hidden`; an entry of a caller's list outside them reads a row inside (and scores NaN)
  FusedPartial* partials;
  uint32_t hidden_stride_b;  // bytes
  uint32_t weight_stride_b;
  uint32_t hidden_bytes;     // extent of the hidden matrix (< 4 GiB, checked on the host)
  // Two hidden matrices in one sweep: tokens [0, n) are rows of `hidden`, [n, 2 n) the same rows of
  // `hidden2`, n the number of valid tokens; n_tokens and the schedule count both.  nullptr: one matrix.
  const char* hidden2;
};

// ---- 16x16x32 MFMA accumulator layout --------------------------------------------------------------
// A 16x16 block lives in four registers: lane l holds token column l % 16 and vocab rows
// 4*(l/16) + e, e = 0..3.  A lane therefore owns one token per 16-token block, and the four lane
// groups l/16 share that token: they are merged once, at the end, over lane ^ 16 and lane ^ 32.
typedef float f32x4v __attribute__((ext_vector_type(4)));

// Fold one wave tile (NBV x NBT blocks of 16x16) into the per-token running states.  Element e of
// block i holds vocab row  vw0 + i*16 + 4*g + e  (g = lane / 16) for the token of block column j.
// NBV of the NBV_ALLOC block rows the array holds are folded (a short tile uses the first few).
template <bool ENT, bool AMAX, int NBV, int NBT, int NBV_ALLOC>
__device__ __forceinline__ void fold_tile16(f32x4v (&acc)[NBV_ALLOC][NBT], RowStat (&st)[NBT], float (&tx)[NBT],
                                            const int (&tgt)[NBT], int vw0, int g, bool partial_tile, int V,
                                            float scale) {
  if (partial_tile) {  // last vocab tile: rows past V do not exist
#pragma unroll
    for (int i = 0; i < NBV; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool dead = vw0 + i * 16 + 4 * g + e >= V;
#pragma unroll
        for (int j = 0; j < NBT; ++j) acc[i][j][e] = dead ? -INFINITY : acc[i][j][e];
      }
  }
  const int vlane = vw0 + 4 * g;  // first vocab row this lane holds in block 0
#pragma unroll
  for (int j = 0; j < NBT; ++j) {
    __builtin_amdgcn_sched_barrier(0);  // one scheduling region per token block (register pressure)
    // Target capture: rare (one tile in V/256 per token), so behind a wave-uniform test.
    const int rel = tgt[j] - vw0;
    const bool mine = tgt[j] >= 0 && rel >= 0 && rel < NBV * 16 && ((rel >> 2) & 3) == g;
    if (__any(mine)) {
      const int want = mine ? ((rel >> 4) * 4 + (rel & 3)) : -1;
#pragma unroll
      for (int i = 0; i < NBV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) tx[j] = (want == i * 4 + e) ? acc[i][j][e] : tx[j];
    }
    float cm = st[j].mx;
    int bi = st[j].bi;
#pragma unroll
    for (int i = 0; i < NBV; ++i) {
      if constexpr (AMAX) {
        // Seven more VALU operations per block, only when the argmax is asked for: the block maximum comes
        // with the position of its first holder, and the running maximum carries the vocab row of the
        // element that set it.  Only a strictly larger value replaces the holder and a lane meets its rows in
        // ascending order, so the sweep itself names the first maximum of the fp32 logits it computed.
        const float x0 = acc[i][j][0], x1 = acc[i][j][1], x2 = acc[i][j][2], x3 = acc[i][j][3];
        const float m01 = raw_max(x0, x1), m23 = raw_max(x2, x3);
        const int e01 = x1 > x0 ? 1 : 0, e23 = x3 > x2 ? 3 : 2;
        const int e = m23 > m01 ? e23 : e01;
        const float bm = raw_max(m01, m23);
        bi = bm > cm ? vlane + i * 16 + e : bi;
        cm = raw_max(cm, bm);
      } else {
        const float bm = raw_max3(acc[i][j][0], acc[i][j][1], raw_max(acc[i][j][2], acc[i][j][3]));
        cm = raw_max(cm, bm);
      }
    }
    const float dm = (st[j].mx - cm) * scale;
    const float resc = fast_exp2(dm);
    const float m = cm * scale;
    // w: sum (y - m) 2^(y - m), relative to the running maximum (stat_merge has the rule for moving it)
    float s0 = st[j].s * resc, s1 = 0.f, w0 = ENT ? fmaf(dm, st[j].s, st[j].w) * resc : 0.f, w1 = 0.f;
#pragma unroll
    for (int i = 0; i < NBV; ++i)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const float x0 = acc[i][j][e], x1 = acc[i][j][e + 1];
        const float t0 = fmaf(x0, scale, -m), t1 = fmaf(x1, scale, -m);
        const float e0 = fast_exp2(t0);
        const float e1 = fast_exp2(t1);
        s0 += e0;
        s1 += e1;
        if constexpr (ENT) {  // a masked row (-inf): floor * 0, not -inf * 0
          w0 = fmaf(clamp_below(t0), e0, w0);
          w1 = fmaf(clamp_below(t1), e1, w1);
        }
      }
    st[j].mx = cm;
    st[j].bi = bi;
    st[j].s = s0 + s1;
    if constexpr (ENT) st[j].w = w0 + w1;
  }
}

// Where position p of a sweep over n_valid tokens finds its hidden row and its target.
struct TokenSource {
  const char* hidden;
  int q;  // position among the valid tokens
};
__device__ __forceinline__ TokenSource token_source(const FusedArgs& a, int p, int n_valid) {
  const int n_one = a.hidden2 ? n_valid >> 1 : n_valid;
  const bool second = p >= n_one;
  return {second ? a.hidden2 : a.hidden, second ? p - n_one : p};
}

// Target id of position p, -1 past the last token or outside [0, V).  Without a branch: registers spilled inside one that only
// some lanes take are lost for the others (seen in a kernel at the limit of the register file: token positions stored under
// the mask of the last block's tokens).
__device__ __forceinline__ int token_target(const FusedArgs& a, int p, int n_valid) {
  const int q = token_source(a, p < n_valid ? p : n_valid - 1, n_valid).q;
  const int t = a.sel.target(a.row_index ? a.row_index[q] : q);
  return p < n_valid && t >= 0 && t < a.V ? t : -1;
}

// Merge the four lane groups that share a token and write one partial per (token, part).
template <int NBT>
__device__ __forceinline__ void write_partials16(RowStat (&st)[NBT], float (&tx)[NBT], FusedPartial* partials,
                                                 int p0, int n_valid, int part, int n_parts, int l16, int g,
                                                 float scale) {
#pragma unroll
  for (int j = 0; j < NBT; ++j) {
    stat_wave_step<4>(st[j], scale);
    stat_wave_step<5>(st[j], scale);
    tx[j] = fmaxf(tx[j], wave_exchange<4>(tx[j]));
    tx[j] = fmaxf(tx[j], wave_exchange<5>(tx[j]));
    const int p = p0 + j * 16 + l16;
    if (g == 0 && p < n_valid) {
      FusedPartial out;
      out.mx = st[j].mx;
      out.s = st[j].s;
      out.w = st[j].w;
      out.tx = tx[j];
      out.bi = st[j].bi;
      out.pad[0] = out.pad[1] = out.pad[2] = 0;
      partials[(int64_t)p * n_parts + part] = out;
    }
  }
}

// Opt in to more than 64 KB of dynamic LDS.
template <typename K>
static bool allow_big_lds(K kernel, int bytes) {
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess)
    return true;
  (void)hipGetLastError();  // the launch that follows reports its own error
  return false;
}

}  // namespace tome
