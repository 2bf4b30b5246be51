// Fused lm_head + log-softmax: hidden[n, H] x weight[V, H]^T -> per-token log-prob of the
// target id (+ lse, entropy), with the [n, V] logits living only in MFMA accumulators.
//
// Replaces `logits = x @ embed_tokens.weight.T` (mlx-impl/model.py:538) followed by
// local_compute_logprobs (mlx-impl/node.py:400-404); the reference materialises the logits in
// bf16 and upcasts them again, here bf16 x bf16 products are accumulated in fp32 and consumed
// in place.
//
// Decomposition
//   * The GEMM is computed transposed: MFMA "A" rows are vocab entries (W is [V, H], K
//     contiguous), MFMA "B" columns are tokens (hidden is [n, H], K contiguous).  In the
//     accumulator layouts a lane then owns ONE token per block column (lane % 32 with the 32x32
//     MFMA, lane % 16 with the 16x16 one) and a few vocab rows per block, so the softmax row
//     statistics are per-lane registers that persist across the whole vocab sweep; the lanes
//     that share a token are merged once at the end.
//   * A workgroup owns one token tile and a contiguous range of 256-row vocab tiles.  Per vocab
//     tile it runs the K loop, then folds the accumulator tile into the running
//     (max, sum 2^(y-m), sum y 2^(y-m)) states.  Two kernels share this shape; a third,
//     fused_lmhead_small_kernel (<= 64 tokens, W streamed once, K split across waves), is
//     described where it is defined:
//       fused_lmhead_dma_kernel  (H % 64 == 0) 512 lanes, 256 vocab rows x 64 .. 256 tokens,
//                                16x16x32 MFMA, K slabs DMA'd into LDS - described at the kernel;
//       fused_lmhead_kernel      (any H % 8) 256 lanes, 256 x 128 tile, 32x32x16 MFMA, 64-wide
//                                slabs staged through registers into padded LDS.
//   * The vocab axis is split over workgroups (fused_schedule); each writes one partial per
//     (token, split, vocab-wave) and fused_combine_kernel merges them deterministically.
//   * Masked tokens are compacted first (compact_rows_kernel); token tiles are built from
//     the compacted index list, so masked rows cost no FLOPs and no HBM traffic.
#include "fused_common.hpp"

namespace tome {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBT = 128;                 // tokens per tile (generic kernel; kBV = 256 vocab rows)
constexpr int kBK = 64;                  // K slab
constexpr int kPitch = kBK * 2 + 16;     // LDS row pitch in bytes: 16 B pad -> conflict-free b128 reads
constexpr int kFusedWG = 256;
constexpr int kWaveT = 64;               // per-wave tile: kWaveV = 128 vocab rows x 64 tokens
constexpr int kNBV = kWaveV / 32, kNBT = kWaveT / 32;
constexpr int kALoads = kBV * 8 / kFusedWG;  // 16-byte chunks per lane per slab (W)
constexpr int kBLoads = kBT * 8 / kFusedWG;  // (hidden)

// Raw buffer descriptors: 16-byte loads addressed by a 32-bit per-lane byte offset plus a
// uniform (scalar) offset.  A per-lane offset at or past num_bytes reads as zero, which is how
// vocab rows past V are handled; the scalar offset is not range-checked.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const char* base, uint32_t num_bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, num_bytes, 0x00020000);
}
__device__ __forceinline__ u32x4 ld16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, uniform_off, 0);
}


// Fold one wave tile of logits (NBV x NBT blocks of 32x32 accumulators) into the per-token
// running states.  Accumulator element e of block i holds vocab row
//   vw0 + i*32 + 8*(e/4) + 4*lh + e%4        (vw0 = first vocab row of this wave's tile)
// for the token this lane owns in block column j.
template <bool ENT, bool AMAX, int NBV, int NBT>
__device__ __forceinline__ void fold_tile(f32x16 (&acc)[NBV][NBT], RowStat (&st)[NBT], float (&tx)[NBT],
                                          const int (&tgt)[NBT], int vw0, int lh, bool partial_tile, int V,
                                          float scale) {
  if (partial_tile) {  // last vocab tile: rows past V do not exist
#pragma unroll
    for (int i = 0; i < NBV; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const bool dead = vw0 + 4 * lh + i * 32 + 8 * (e / 4) + (e % 4) >= V;
#pragma unroll
        for (int j = 0; j < NBT; ++j) acc[i][j][e] = dead ? -INFINITY : acc[i][j][e];
      }
  }
  const int vlane = vw0 + 4 * lh;  // first vocab row this lane holds in block 0
#pragma unroll
  for (int j = 0; j < NBT; ++j) {
    // One scheduling region per token block: otherwise all accumulator reads of all blocks are
    // hoisted to the top and the register file overflows.
    __builtin_amdgcn_sched_barrier(0);
    // Target capture: rare (one tile in V/256 per token), so behind a wave-uniform test.
    const int rel = tgt[j] - vw0;
    const bool mine = tgt[j] >= 0 && rel >= 0 && rel < NBV * 32 && ((rel >> 2) & 1) == lh;
    if (__any(mine)) {
      const int want = mine ? ((rel >> 5) * 16 + ((rel & 31) >> 3) * 4 + (rel & 3)) : -1;
#pragma unroll
      for (int i = 0; i < NBV; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) tx[j] = (want == i * 16 + e) ? acc[i][j][e] : tx[j];
    }
    float cm = st[j].mx;
    int bi = st[j].bi;
#pragma unroll
    for (int i = 0; i < NBV; ++i) {
      if constexpr (AMAX) {
        // The running maximum carries the vocab row of the element that set it.  A lane meets its rows in
        // ascending order and only a strictly larger value replaces the holder, so the first maximum stays.
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float x = acc[i][j][e];
          bi = x > cm ? vlane + i * 32 + 8 * (e / 4) + (e % 4) : bi;
          cm = raw_max(cm, x);
        }
      } else {
        float m = acc[i][j][0];
#pragma unroll
        for (int e = 1; e < 16; e += 2) m = raw_max3(m, acc[i][j][e], e + 1 < 16 ? acc[i][j][e + 1] : acc[i][j][e]);
        cm = raw_max(cm, m);
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
      for (int e = 0; e < 16; e += 2) {
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

// Merge the two lane halves that share a token and write one partial per (token, part).
template <int NBT>
__device__ __forceinline__ void write_partials(RowStat (&st)[NBT], float (&tx)[NBT], FusedPartial* partials,
                                               int p0, int n_valid, int part, int n_parts, int l32, int lh,
                                               float scale) {
#pragma unroll
  for (int j = 0; j < NBT; ++j) {
    stat_wave_step<5>(st[j], scale);
    const float txo = wave_exchange<5>(tx[j]);
    tx[j] = fmaxf(tx[j], txo);
    const int p = p0 + j * 32 + l32;
    if (lh == 0 && p < n_valid) {
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

template <bool ENT, bool AMAX>
__global__ __launch_bounds__(kFusedWG, 2) void fused_lmhead_kernel(FusedArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[(kBV + kBT) * kPitch];
  char* ldsA = lds;
  char* ldsB = lds + kBV * kPitch;

  const int n_valid = a.n_valid ? *a.n_valid : a.n_tokens;
  const FusedSchedule sch = a.sched_dev ? *a.sched_dev : a.sched;
  int ttile, split;
  if (n_valid <= 0 || !fused_locate(sch, blockIdx.x, ttile, split)) return;
  const int t0 = ttile * kBT;
  const int vt0 = (int)((int64_t)split * sch.n_vunits / sch.n_splits);  // one unit = one 256-row tile here
  const int vt1 = (int)((int64_t)(split + 1) * sch.n_vunits / sch.n_splits);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wave_v = wave & 1, wave_t = wave >> 1;
  const int l32 = lane & 31, lh = lane >> 5;

  // ---- global -> LDS staging assignment: 8 lanes cover one 128-byte row segment ----------
  const int ld_row = tid >> 3, ld_c = tid & 7;
  const __amdgpu_buffer_rsrc_t rsrcB = make_rsrc(a.hidden, a.hidden_bytes);
  uint32_t boff[kBLoads];
#pragma unroll
  for (int j = 0; j < kBLoads; ++j) {
    int p = t0 + ld_row + 32 * j;
    p = p < n_valid ? p : n_valid - 1;
    const int tok = a.hidden_index ? min(max(a.hidden_index[p], 0), a.n_rows - 1) : p;
    boff[j] = (uint32_t)tok * a.hidden_stride_b + ld_c * 16;
  }
  uint32_t aoff[kALoads];
#pragma unroll
  for (int j = 0; j < kALoads; ++j) aoff[j] = (uint32_t)(ld_row + 32 * j) * a.weight_stride_b + ld_c * 16;
  const int st_off = ld_row * kPitch + ld_c * 16;

  // ---- per-lane token state ---------------------------------------------------------------
  RowStat st[kNBT];
  float tx[kNBT];
  int tgt[kNBT];
#pragma unroll
  for (int bt = 0; bt < kNBT; ++bt) {
    st[bt] = stat_identity();
    tx[bt] = -INFINITY;
    tgt[bt] = token_target(a, t0 + wave_t * kWaveT + bt * 32 + l32, n_valid);
  }

  const int nk = (a.H + kBK - 1) / kBK;
  const char* rdA = ldsA + (wave_v * kWaveV + l32) * kPitch + lh * 16;
  const char* rdB = ldsB + (wave_t * kWaveT + l32) * kPitch + lh * 16;

  for (int vt = vt0; vt < vt1; ++vt) {
    const int v0 = vt * kBV;
    // Descriptor rebased to this tile: per-lane offsets stay constant and rows past V fall
    // outside num_bytes (read as zero, then masked to -inf in the epilogue).
    const __amdgpu_buffer_rsrc_t rsrcA =
        make_rsrc(a.weight + (int64_t)v0 * a.weight_stride_b, (uint32_t)(a.V - v0) * a.weight_stride_b);

    f32x16 acc[kNBV][kNBT];
#pragma unroll
    for (int i = 0; i < kNBV; ++i)
#pragma unroll
      for (int j = 0; j < kNBT; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    u32x4 ra[kALoads], rb[kBLoads];
    const bool in0 = ld_c * 8 < a.H;
#pragma unroll
    for (int j = 0; j < kALoads; ++j) ra[j] = in0 ? ld16(rsrcA, aoff[j], 0) : u32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < kBLoads; ++j) rb[j] = in0 ? ld16(rsrcB, boff[j], 0) : u32x4{0, 0, 0, 0};

    for (int kt = 0; kt < nk; ++kt) {
      __syncthreads();  // every wave has finished reading the previous slab
#pragma unroll
      for (int j = 0; j < kALoads; ++j) *reinterpret_cast<u32x4*>(ldsA + st_off + j * 32 * kPitch) = ra[j];
#pragma unroll
      for (int j = 0; j < kBLoads; ++j) *reinterpret_cast<u32x4*>(ldsB + st_off + j * 32 * kPitch) = rb[j];
      __syncthreads();
      if (kt + 1 < nk) {  // prefetch the next slab while this one is multiplied
        const int koff = (kt + 1) * kBK * 2;
        const bool in = (kt + 1) * kBK + ld_c * 8 < a.H;
#pragma unroll
        for (int j = 0; j < kALoads; ++j) ra[j] = in ? ld16(rsrcA, aoff[j], koff) : u32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < kBLoads; ++j) rb[j] = in ? ld16(rsrcB, boff[j], koff) : u32x4{0, 0, 0, 0};
      }
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks) {
        bf16x8 fa[kNBV], fb[kNBT];
#pragma unroll
        for (int i = 0; i < kNBV; ++i)
          fa[i] = *reinterpret_cast<const bf16x8*>(rdA + i * 32 * kPitch + ks * 32);
#pragma unroll
        for (int j = 0; j < kNBT; ++j)
          fb[j] = *reinterpret_cast<const bf16x8*>(rdB + j * 32 * kPitch + ks * 32);
#pragma unroll
        for (int i = 0; i < kNBV; ++i)
#pragma unroll
          for (int j = 0; j < kNBT; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
    }

    fold_tile<ENT, AMAX>(acc, st, tx, tgt, v0 + wave_v * kWaveV, lh, v0 + kBV > a.V, a.V, a.scale);
  }

  write_partials(st, tx, a.partials, t0 + wave_t * kWaveT, n_valid, split * kPartsPerSplit + wave_v,
                 sch.n_splits * kPartsPerSplit, l32, lh, a.scale);
}



// ===============================================================================================
// Small batches (<= 64 tokens, the decode-step regime): W streams from HBM exactly once and nothing is
// reused, so the kernel is built like a streaming reduction, not like a GEMM.
//
//   * K is split across the waves of a workgroup (256 or 512 columns each).  A wave's slice of the
//     hidden states - all tokens - then fits its registers as MFMA B fragments for the whole launch,
//     and W goes from global memory into registers and through a wave-private LDS tile into A
//     fragments: no barrier on the load path.
//   * Each wave keeps 16 sixteen-byte loads in flight (two 16-row tiles of its K slice, refilled in
//     place right after the MFMA that consumed them); one workgroup per CU owns one contiguous range of
//     16-row vocab tiles.
//   * Per tile the waves' partial sums (16 rows x 16*NBT tokens, MFMA layout) meet in LDS; wave j sums
//     them in wave order and folds token block j into its online-softmax state.  One barrier per tile:
//     the buffer of tile t is rewritten at tile t + 2, after the barrier of tile t + 1, which the
//     folding waves only reach once tile t is folded.
//   * One partial per (token, workgroup); the combine kernel is shared with the other paths.
// ===============================================================================================
template <bool ENT, bool AMAX, int NBT, int KSTEPS>
__global__ __launch_bounds__(512) void fused_lmhead_small_kernel(FusedArgs a) {
  extern __shared__ __attribute__((aligned(16))) char small_mem[];  // [2][waves][NBT][64 lanes] f32x4, then [waves] 4 KB tiles
  constexpr int kBuf = 16 / KSTEPS;                                 // tile buffers in flight (registers): 16 loads per lane
  constexpr int kRed = 2;                                           // reduction buffers (LDS)
  touch_args(a);
  const int n_valid = a.n_valid ? *a.n_valid << (a.hidden2 ? 1 : 0) : a.n_tokens;
  if (n_valid <= 0) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_waves = blockDim.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int n_tiles = (a.V + 15) >> 4;
  const int t0 = (int)((int64_t)blockIdx.x * n_tiles / gridDim.x);
  const int t1 = (int)((int64_t)(blockIdx.x + 1) * n_tiles / gridDim.x);
  const int kb0 = (wave * KSTEPS * 32 + 8 * g) * 2;  // byte offset of this lane's first K chunk in a row

  // Hidden-state fragments of this wave's K slice: lane (token l16, group g) holds K = 32 ks + 8 g .. + 7.
  bf16x8 fb[KSTEPS][NBT];
#pragma unroll
  for (int j = 0; j < NBT; ++j) {
    int p = j * 16 + l16;
    p = p < n_valid ? p : n_valid - 1;
    const TokenSource src = token_source(a, p, n_valid);
    const int tok = a.hidden_index ? min(max(a.hidden_index[src.q], 0), a.n_rows - 1) : src.q;
    const char* hp = src.hidden + (int64_t)tok * a.hidden_stride_b + kb0;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) fb[ks][j] = *reinterpret_cast<const bf16x8*>(hp + ks * 64);
  }
  // Token state of the block this wave folds (waves >= NBT fold nothing).
  RowStat st[1] = {stat_identity()};
  float tx[1] = {-INFINITY};
  int tgt[1] = {-1};
  if (wave < NBT) {
    tgt[0] = token_target(a, wave * 16 + l16, n_valid);
  }

  // W loads are shaped for HBM, not for the MFMA: one instruction fetches 4 rows x 256 bytes (lane = row
  // lane/16 of the group, 16-byte chunk lane%16), which streams 17 % faster than the operand shape of 16
  // rows x 64 bytes (6.85 against 5.84 TB/s in a copy kernel with this kernel's structure).  A unit of
  // 16 rows x 256 bytes (four K steps) then changes layout through a wave-private 4 KB LDS tile: chunk c
  // of row r is stored at position c ^ r, so the contiguous writes and the fragment reads (16 rows, one
  // chunk) are both free of bank conflicts.
  constexpr int kUnits = KSTEPS / 4;  // units per tile and wave
  const int lr = lane >> 4, lc = lane & 15;
  auto w_ptr = [&](int t, int q) {  // rows past V (last tile only) read the last row; masked in the fold
    int row = t * 16 + 4 * q + lr;
    row = row < a.V ? row : a.V - 1;
    return a.weight + (int64_t)row * a.weight_stride_b + wave * (KSTEPS * 64) + lc * 16;
  };
  char* stage = small_mem + (size_t)kRed * n_waves * NBT * 1024 + wave * 4096;
  u32x4 wb[kBuf][kUnits][4];
#pragma unroll
  for (int b = 0; b < kBuf && t0 < t1; ++b) {
    const int t = t0 + b < t1 ? t0 + b : t1 - 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const char* wp = w_ptr(t, q);
#pragma unroll
      for (int u = 0; u < kUnits; ++u) wb[b][u][q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp + u * 256));
    }
  }

  for (int tb = t0; tb < t1; tb += kBuf) {
#pragma unroll
    for (int b = 0; b < kBuf; ++b) {
      const int t = tb + b;
      if (t >= t1) break;  // uniform
      // The refill is unconditional (past the range it re-reads the tile just consumed, an L2 hit that is
      // never used): with a load behind a branch the compiler cannot count the loads in flight and waits
      // for far more of them than the one it needs.
      const int tn = t + kBuf < t1 ? t + kBuf : t;
      f32x4v acc[NBT];
#pragma unroll
      for (int j = 0; j < NBT; ++j) acc[j] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < kUnits; ++u) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<u32x4*>(stage + (4 * q + lr) * 256 + ((lc ^ (4 * q + lr)) << 4)) = wb[b][u][q];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          wb[b][u][q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w_ptr(tn, q) + u * 256));
        // The tile is private to this wave and LDS serves a wave's requests in order.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        bf16x8 fa[4];
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4)
          fa[k4] = *reinterpret_cast<const bf16x8*>(stage + l16 * 256 + (((4 * k4 + g) ^ l16) << 4));
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4)
#pragma unroll
          for (int j = 0; j < NBT; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[k4], fb[4 * u + k4][j], acc[j], 0, 0, 0);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // the next unit overwrites what was just read
        __builtin_amdgcn_wave_barrier();
      }
      char* red = small_mem + (size_t)(((t & (kRed - 1)) * n_waves + wave) * NBT) * 1024 + lane * 16;
#pragma unroll
      for (int j = 0; j < NBT; ++j) *reinterpret_cast<f32x4v*>(red + j * 1024) = acc[j];
      __syncthreads();
      if (wave < NBT) {
        f32x4v sum[1][1] = {{f32x4v{0.f, 0.f, 0.f, 0.f}}};
        const char* src = small_mem + (size_t)((t & (kRed - 1)) * n_waves * NBT + wave) * 1024 + lane * 16;
        for (int w = 0; w < n_waves; ++w) sum[0][0] += *reinterpret_cast<const f32x4v*>(src + (size_t)w * NBT * 1024);
        fold_tile16<ENT, AMAX, 1>(sum, st, tx, tgt, t * 16, g, t * 16 + 16 > a.V, a.V, a.scale);
      }
    }
  }
  // One partial per (token, workgroup): part index = workgroup id.
  // (the lane derived afresh: kept across the loop it is one register too many for two token blocks of 512 columns, and the loop's
  // loads are then scheduled around a spill, 1-4 % at 17 .. 32 tokens x H = 4096)
  int ln = (int)threadIdx.x;
  asm volatile("" : "+v"(ln));
  if (wave < NBT)
    write_partials16<1>(st, tx, a.partials, wave * 16, n_valid, (int)blockIdx.x, (int)gridDim.x, ln & 15, (ln & 63) >> 4, a.scale);
}

// ---- compaction of valid rows ----------------------------------------------------------------
// One workgroup: row_index[0 .. n_valid) = ascending indices of the valid rows.
// Outputs of masked rows are zeroed here.
struct CompactArgs {
  RowSel sel;
  int32_t* row_index;
  int32_t* n_valid;
  float* out0;
  float* out1;
  float* out2;
  float* out3;
  float* out4;
  int32_t* out_argmax;
  int n;
  FusedShape shape;              // of the schedule, which this kernel derives from n_valid
  int joint;                     // 1: every valid token is swept twice (two hidden matrices)
};

// Rows are taken in batches of up to 8192: each of the 16 waves owns a run of consecutive rows of a batch (a
// sixteenth of the rows, at most 512) and reads their mask values with 8 independent coalesced loads (lane
// l of chunk c reads row first + 64 c + l), which stay in registers for the second sweep; counts come from ballots,
// the waves' offsets from a scan through LDS.  One workgroup between two launches is bound by its chain of misses - arguments,
// instructions, mask, LDS - so there is little code, and wave 15 works out the schedule of an unmasked batch while the mask
// is on its way: that fetches the instructions, and it is the answer if all rows turn out to count.
template <typename V>
__device__ __forceinline__ void load_mask_chunks(int (&v)[8], int rows_left, int lane, V&& value) {
#pragma unroll
  for (int c = 0; c < 8; ++c) {  // unconditional (clamped) loads: all of them in flight together
    const int r = c * 64 + lane;
    v[c] = value(r < rows_left ? r : rows_left - 1);
  }
}
__global__ __launch_bounds__(1024) void compact_rows_kernel(CompactArgs a) {
  constexpr int kChunks = 8;                        // 64-row chunks per wave and batch, at most
  __shared__ int wave_tot[16];
  touch_args(a);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t below = (1ull << lane) - 1;        // lanes in front of this one
  int n_chunks = (int)((((int64_t)a.n + 15) / 16 + 63) / 64);  // per wave, so that small batches use all 16 waves
  n_chunks = n_chunks > kChunks ? kChunks : n_chunks;
  const int wave_rows = n_chunks * 64;
  const int64_t batch_rows = 16 * (int64_t)wave_rows;
  FusedSchedule sch;
  int done = 0;                                     // valid rows of earlier batches
  for (int64_t b0 = 0; b0 < a.n; b0 += batch_rows) {
    const int64_t first = b0 + (int64_t)wave * wave_rows;
    int left = (int)(a.n - first < wave_rows ? a.n - first : wave_rows);  // rows of this wave's run that exist
    left = left < 0 ? 0 : left;
    int v[kChunks];
    if (left > 0) {
      const char* mask = static_cast<const char*>(a.sel.row_valid) + first * a.sel.valid_bytes;
      if (!a.sel.row_valid) load_mask_chunks(v, left, lane, [&](int r) { return a.sel.inside_length((uint32_t)(first + r)) ? 1 : 0; });
      else if (a.sel.valid_bytes == 1) load_mask_chunks(v, left, lane, [&](int r) { return (int)reinterpret_cast<const uint8_t*>(mask)[(unsigned)r]; });
      else load_mask_chunks(v, left, lane, [&](int r) { return *reinterpret_cast<const int32_t*>(mask + (unsigned)(r * a.sel.valid_bytes)); });
    }
    if (wave == 15 && b0 == 0) sch = fused_schedule_wave(a.n << a.joint, a.shape, lane);
    int cnt = 0;
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      v[c] = c * 64 + lane < left ? v[c] : 0;
      cnt += __builtin_popcountll(__ballot(v[c] != 0));
    }
    if (lane == 0) wave_tot[wave] = cnt;
    __syncthreads();
    const int tot = wave_tot[lane & 15];
    __syncthreads();                                // wave_tot is rewritten by the next batch
    int pos = done;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int t = __builtin_amdgcn_readlane(tot, w);
      pos += w < wave ? t : 0;
      done += t;
    }
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      if (c >= n_chunks) break;
      const int64_t r = first + c * 64 + lane;
      const uint64_t mask = __ballot(v[c] != 0);    // zero for chunks past the end
      if (v[c] != 0) {
        a.row_index[pos + __builtin_popcountll(mask & below)] = (int32_t)r;
      } else if (c * 64 + lane < left) {
        if (a.out0) a.out0[r] = 0.f;
        if (a.out1) a.out1[r] = 0.f;
        if (a.out2) a.out2[r] = 0.f;
        if (a.out3) a.out3[r] = 0.f;
        if (a.out4) a.out4[r] = 0.f;
        if (a.out_argmax) a.out_argmax[r] = -1;
      }
      pos += __builtin_popcountll(mask);
    }
  }
  if (threadIdx.x == 0) *a.n_valid = done;
  if (wave == 15) {  // one wave also fixes the work decomposition, which depends on the total
    if (done != a.n) sch = fused_schedule_wave(done << a.joint, a.shape, lane);
    if (lane == 0) *reinterpret_cast<FusedSchedule*>(a.n_valid + 4) = sch;
  }
}

// ---- final RMSNorm of the rows that will be multiplied ------------------------------------------
// y = w * T(x * rsqrt(mean(x^2) + eps)) in bf16 with fp32 statistics: mx.fast.rms_norm as
// mlx-impl/model.py:343 calls it on the last hidden states (model.py:536).  Only valid rows are
// normalised, and they are written compactly: position p of the output is row row_index[p] of x.
struct NormArgs {
  const char* x[2];          // bf16 [n, H]; the second for blockIdx.y = 1
  const uint16_t* w;         // bf16 [H]
  char* y[2];                // bf16 [n_valid, H], dense
  const int32_t* row_index;  // or nullptr = identity; entries outside [0, n_rows) read a row inside
  const int32_t* n_valid;    // or nullptr = n
  uint32_t x_stride_b;
  int n, n_rows, H;
  float eps;
};

// What bounds it below some thousand rows is a chain of misses (arguments, row list, row, weights), not bytes: everything that does
// not depend on another load is requested at once, and a row of up to kNormHeld x 512 elements stays in the registers of its wave,
// where it was read twice and the weights were only asked for behind the sum; the two roundings are one v_cvt_pk_bf16_f32 each for two
// elements (the same bits for every float).  64 x 4096 8.3 -> 4.7 us, 512 x 2560 7.8 -> 5.0, 2048 x 2560 10.4 -> 7.9, 16384 x 2560
// 39.2 -> 27.3 (168 MB: 6.1 TB/s, what a copy reaches), 8192 x 6144 46.5 -> 35.3, 64 x 1024 4.1 -> 3.4, 4096 x 1024 8.4 -> 7.7.
constexpr int kNormHeld = 8;  // 16-byte units a lane holds (H = 4096); longer rows read the rest a second time
__device__ __forceinline__ void norm_add(const u32x4& v, float& ss) {
  const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float lo = bf16_lo(u[k]), hi = bf16_hi(u[k]);
    ss = fmaf(lo, lo, ss);
    ss = fmaf(hi, hi, ss);
  }
}
__device__ __forceinline__ u32x4 norm_scale(const u32x4& v, const u32x4& g, float inv) {
  const uint32_t u[4] = {v.x, v.y, v.z, v.w}, gw[4] = {g.x, g.y, g.z, g.w};
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t n = pack_bf16(bf16_lo(u[k]) * inv, bf16_hi(u[k]) * inv);
    o[k] = pack_bf16(bf16_lo(gw[k]) * bf16_lo(n), bf16_hi(gw[k]) * bf16_hi(n));
  }
  return u32x4{o[0], o[1], o[2], o[3]};
}
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(NormArgs a) {
  touch_args(a);
  const int lane = threadIdx.x & 63;
  const int p = blockIdx.x * 4 + (threadIdx.x >> 6);  // one wave per row
  const int n_chunks = a.H / 8;
  const u32x4* w = reinterpret_cast<const u32x4*>(a.w);
  u32x4 g[kNormHeld], v[kNormHeld];
#pragma unroll
  for (int q = 0; q < kNormHeld; ++q)
    if (q * 64 < n_chunks) g[q] = w[min(q * 64 + lane, n_chunks - 1)];
  const int n_valid = a.n_valid ? *a.n_valid : a.n;
  if (p >= n_valid) return;
  const int row = a.row_index ? min(max(a.row_index[p], 0), a.n_rows - 1) : p;
  const u32x4* x = reinterpret_cast<const u32x4*>((blockIdx.y ? a.x[1] : a.x[0]) + (int64_t)row * a.x_stride_b);
  u32x4* y = reinterpret_cast<u32x4*>((blockIdx.y ? a.y[1] : a.y[0]) + (int64_t)p * a.H * 2);
#pragma unroll
  for (int q = 0; q < kNormHeld; ++q)
    if (q * 64 < n_chunks) v[q] = x[min(q * 64 + lane, n_chunks - 1)];
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < kNormHeld; ++q)
    if (q * 64 + lane < n_chunks) norm_add(v[q], ss);
  for (int c = kNormHeld * 64 + lane; c < n_chunks; c += 64) norm_add(x[c], ss);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  const float inv = 1.0f / sqrtf(ss / (float)a.H + a.eps);
#pragma unroll
  for (int q = 0; q < kNormHeld; ++q)
    if (q * 64 + lane < n_chunks) y[q * 64 + lane] = norm_scale(v[q], g[q], inv);
  for (int c = kNormHeld * 64 + lane; c < n_chunks; c += 64) y[c] = norm_scale(x[c], w[c], inv);  // from the caches
}

// ---- combine -----------------------------------------------------------------------------------
struct CombineArgs {
  const FusedPartial* partials;      // policy (or the only) weight set
  const FusedPartial* partials_ref;  // second sweep, or nullptr
  int joint;                         // 1: the second half of `partials` is the second matrix of a joint sweep
  const int32_t* row_index;
  const int32_t* n_valid;
  float* out_lp;
  float* out_lse;
  float* out_entropy;
  float* out_ref_lp;
  float* out_k3;
  int32_t* out_argmax;
  const int32_t* hidden_rows;  // the caller's row list, or nullptr: an entry outside [0, n_rows) scores NaN (argmax -1)
  int n_rows;
  int n_tokens;
  const FusedSchedule* sched_dev;  // as in FusedArgs
  FusedSchedule sched;
  float scale;
};

__device__ __forceinline__ void combine_one(const FusedPartial* parts, int n_parts, int lane, float scale,
                                            RowStat& st, float& tx) {
  st = stat_identity();
  tx = -INFINITY;
  // A lane's partials are fetched eight at a time before the first is merged (clamped, unconditional loads: all in
  // flight together): the merges form a chain, and a load inside it costs a trip to memory per partial - the previous
  // launch wrote these records on other dies.  Same merge order as a plain loop.
  constexpr int kBatch = 8;
  for (int base = 0; base < n_parts; base += 64 * kBatch) {
    f32x4 head[kBatch];
    int bi[kBatch];
#pragma unroll
    for (int q = 0; q < kBatch; ++q) {
      const int i = base + lane + 64 * q;
      const FusedPartial* src = parts + (i < n_parts ? i : n_parts - 1);
      head[q] = *reinterpret_cast<const f32x4*>(src);  // mx, s, w, tx
      bi[q] = src->bi;
    }
#pragma unroll
    for (int q = 0; q < kBatch; ++q) {
      if (base + lane + 64 * q < n_parts) {
        RowStat o{head[q][0], head[q][1], head[q][2], bi[q]};
        stat_merge(st, o, scale);
        tx = fmaxf(tx, head[q][3]);
      }
    }
  }
  stat_wave_reduce(st, scale);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) tx = fmaxf(tx, __shfl_xor(tx, off, 64));
}

__global__ __launch_bounds__(256) void fused_combine_kernel(CombineArgs a) {
  touch_args(a);
  const int lane = threadIdx.x & 63;
  const int p = blockIdx.x * 4 + (threadIdx.x >> 6);  // compacted position, one wave each
  const int n_valid = a.n_valid ? *a.n_valid : a.n_tokens;
  if (p >= n_valid) return;
  const int tok = a.row_index ? a.row_index[p] : p;
  const int n_parts = (a.sched_dev ? a.sched_dev->n_splits : a.sched.n_splits) * kPartsPerSplit;
  RowStat st;
  float tx;
  combine_one(a.partials + (int64_t)p * n_parts, n_parts, lane, a.scale, st, tx);
  const float m = st.mx * a.scale;
  const float log2s = fast_log2(st.s);
  // tx stays -inf only when the target id was outside [0, V).
  const float lp = tx == -INFINITY ? __builtin_nanf("") : (fmaf(tx, a.scale, -m) - log2s) * kLn2;
  float ref_lp = 0.f;
  const FusedPartial* second = a.joint ? a.partials + (int64_t)n_valid * n_parts : a.partials_ref;
  if (second) {
    RowStat sr;
    float txr;
    combine_one(second + (int64_t)p * n_parts, n_parts, lane, a.scale, sr, txr);
    const float mr = sr.mx * a.scale;
    ref_lp = txr == -INFINITY ? __builtin_nanf("") : (fmaf(txr, a.scale, -mr) - fast_log2(sr.s)) * kLn2;
  }
  if (lane != 0) return;
  if (a.hidden_rows && (uint32_t)a.hidden_rows[p] >= (uint32_t)a.n_rows) {  // (never with a second weight set)
    if (a.out_argmax) a.out_argmax[tok] = -1;
    if (a.out_lp) a.out_lp[tok] = __builtin_nanf("");
    if (a.out_lse) a.out_lse[tok] = __builtin_nanf("");
    if (a.out_entropy) a.out_entropy[tok] = __builtin_nanf("");
    return;
  }
  // The sweep kernels name the element themselves: bi is the vocab row of the first maximum among the fp32
  // logits they accumulated (0 when nothing above the floor was seen, as a first-maximum scan would say).
  if (a.out_argmax) a.out_argmax[tok] = st.bi == 0x7fffffff ? 0 : st.bi;
  if (a.out_lp) a.out_lp[tok] = lp;
  if (a.out_lse) a.out_lse[tok] = (m + log2s) * kLn2;
  if (a.out_entropy) a.out_entropy[tok] = (log2s - st.w / st.s) * kLn2;
  if (a.out_ref_lp) a.out_ref_lp[tok] = ref_lp;
  if (a.out_k3) {
    const float d = ref_lp - lp;
    a.out_k3[tok] = expm1f(d) - d;
  }
}

// ---- host side -----------------------------------------------------------------------------------
// The DMA kernel needs whole 64-wide K slabs (ragged H goes to the generic kernel); its token tile shrinks
// with the batch.  Decode-sized batches whose hidden states fit the waves' registers take the streaming kernel.

// Kernel selector for tests and tuning runs: -1 (the default) picks by shape, kGeneric / kDma force that
// sweep kernel wherever its shape rules allow.  Process-wide; set it while no call is in flight.
static std::atomic<int> g_forced_kind{-1};
void fused_force_kernel(int kind) { g_forced_kind.store(kind, std::memory_order_relaxed); }

// The DMA kernels' launches (fused_dma.hpp), instantiated in the fused_dma_*.hip files: one token tile, or the tile of the schedule
// on the device; the 160 KB of LDS their largest form asks for.
template <bool ENT, bool AMAX>
bool launch_dma(const FusedArgs& a, int tile, bool deep, bool w_nt, int grid, hipStream_t stream);
template <bool ENT, bool AMAX>
void launch_dma_any(const FusedArgs& a, bool deep, bool w_nt, int grid, hipStream_t stream);
bool dma_allow_deep_lds();

// Does the current device grant the 160 KB of dynamic LDS that the third W buffer asks for - all of a CU's LDS, which a
// driver may not hand out whole?  Where it does not, plans keep to the tiles and the ring depth that do without.
static bool deep_lds_granted() {
  static std::atomic<uint64_t> known{0}, refused{0};  // bit per device ordinal
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDeviceOrdinals) {
    (void)hipGetLastError();  // no device: a workspace is being sized
    return true;
  }
  const uint64_t bit = 1ull << dev;
  if (!(known.load(std::memory_order_acquire) & bit)) {
    if (!dma_allow_deep_lds()) refused.fetch_or(bit, std::memory_order_relaxed);
    known.fetch_or(bit, std::memory_order_release);
  }
  return !(refused.load(std::memory_order_relaxed) & bit);
}

// Workgroups of the small-batch kernel: one per CU.  Measured at 16 and 64 tokens, H = 1024: 256 workgroups
// 59 us, 512 66 us, 1024 (all that fit) 71 us, 2048 (queued) 95 us; a deeper load ring changes nothing.
// The stream is bound by the 16-rows-by-64-bytes shape of an MFMA operand load, which a plain copy
// kernel of the same shape and lifetime moves at 5.6 TB/s, and more concurrent streams lower that.
static int small_wg_count() {
  static std::atomic<int> cached[kMaxDeviceOrdinals];  // per device ordinal: GPUs of one process may differ
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDeviceOrdinals) return 0;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 2) return 0;
    if (cus > 512) cus = 512;  // the workspace holds 512 parts per token
    n = cus & ~1;              // even: the combine kernel counts parts in pairs
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

static FusedEnv fused_env() { return FusedEnv{g_forced_kind.load(std::memory_order_relaxed), small_wg_count()}; }

// The generic kernel addresses both matrices through buffer descriptors with 32-bit byte offsets.
bool fused_needs_32bit_extents(int64_t n_tokens, int64_t H, int64_t V) { return fused_kernel(fused_env(), n_tokens, H, V).kind == kGeneric; }

FusedLayout fused_call_layout(int64_t n_tokens, int64_t H, int64_t V, int n_sweeps, int n_normed) {
  return fused_layout(fused_env(), n_tokens, H, V, n_sweeps, n_normed);
}

template <bool ENT, bool AMAX, int NBT, int KSTEPS>
static int launch_small(const FusedArgs& a, int waves, hipStream_t stream) {
  int n_wg = small_wg_count();
  const int n_tiles = (a.V + 15) / 16;
  if (n_wg > n_tiles) n_wg = n_tiles & ~1;  // no empty vocab ranges
  if (n_wg < 2) return 0;
  const size_t lds = (size_t)2 * waves * NBT * 1024 + (size_t)waves * 4096;
  static DeviceOnce attr_set;  // opt in to > 64 KB of dynamic LDS once per instantiation and device
  if (lds > 65536 && attr_set.first_on_current_device())
    allow_big_lds(&fused_lmhead_small_kernel<ENT, AMAX, NBT, KSTEPS>, 2 * 8 * 4 * 1024 + 8 * 4096);
  hipLaunchKernelGGL((fused_lmhead_small_kernel<ENT, AMAX, NBT, KSTEPS>), dim3((unsigned)n_wg), dim3((unsigned)waves * 64),
                     lds, stream, a);
  return n_wg;
}

// Launches the sweep kernel of `plan`.  Returns the number of partials per token it leaves (0 = the
// schedule's own count, -1 = no kernel for the plan, nothing launched).
template <bool ENT>
static int launch_main(const FusedArgs& a, const FusedPlan& plan, bool want_argmax, hipStream_t stream) {
  if (plan.kind == kSmall) {
    int n = 0;
    const int w = plan.small_waves;
#define TOME_SMALL(NBT, KS)                                                 \
  n = want_argmax ? launch_small<ENT, true, NBT, KS>(a, w, stream) : launch_small<ENT, false, NBT, KS>(a, w, stream)
    if (plan.small_ksteps == 8 && plan.small_nbt == 1) TOME_SMALL(1, 8);
    else if (plan.small_ksteps == 8) TOME_SMALL(4, 8);
    else if (plan.small_nbt == 1) TOME_SMALL(1, 16);
    else TOME_SMALL(2, 16);
#undef TOME_SMALL
    return n;  // >= 2: fused_plan only picks this kernel when it can be placed
  }
  if (plan.kind == kDma) {
    const bool deep = ENT ? plan.deep : plan.deep_lp;
    if (a.sched_dev && plan.any_tile) {
      if (want_argmax) launch_dma_any<ENT, true>(a, plan.any_deep, plan.w_nt, plan.grid, stream);
      else launch_dma_any<ENT, false>(a, plan.any_deep, plan.w_nt, plan.grid, stream);
    } else if (!(want_argmax ? launch_dma<ENT, true>(a, a.sched.tile, deep, plan.w_nt, plan.grid, stream)
                             : launch_dma<ENT, false>(a, a.sched.tile, deep, plan.w_nt, plan.grid, stream))) {
      return -1;
    }
  } else {
    if (want_argmax) hipLaunchKernelGGL((fused_lmhead_kernel<ENT, true>), dim3((unsigned)plan.grid), dim3(kFusedWG), 0, stream, a);
    else hipLaunchKernelGGL((fused_lmhead_kernel<ENT, false>), dim3((unsigned)plan.grid), dim3(kFusedWG), 0, stream, a);
  }
  return 0;
}

// One sweep per (hidden, weight) pair: the policy pair always, and a reference pair when a second weight
// set (`w1`) or a second hidden-state matrix (`hidden_ref`) is given; either may repeat the policy's.
// `hidden_rows` (nullable): token p is row hidden_rows[p] of a hidden matrix of `n_rows` rows, ids and outputs packed.
static hipError_t fused_launch_impl(const void* hidden, const int32_t* hidden_rows, int64_t n_rows, const void* hidden_ref, const void* norm_weight,
                                    float norm_eps, const void* w0, const void* w1, int64_t n_tokens, int64_t H,
                                    int64_t V, int64_t hidden_stride, int64_t weight_stride, const RowSel& sel,
                                    float temperature, float* out_lp, float* out_lse,
                                    float* out_entropy, int32_t* out_argmax, float* out_ref_lp, float* out_k3,
                                    const FusedLayout& layout, void* workspace, hipStream_t stream) {
  const bool second = w1 != nullptr || hidden_ref != nullptr;
  if (!w1) w1 = w0;
  if (!hidden_ref) hidden_ref = hidden;
  char* ws = static_cast<char*>(workspace);
  const FusedEnv env = fused_env();
  const bool joint = second && w1 == w0 && hidden_ref != hidden && joint_fits(n_tokens, H, sel.masked()) && env.forced != kGeneric;
  const int swept = (int)n_tokens << (joint ? 1 : 0);
  const FusedPlan plan = fused_plan(env, swept, H, V, deep_lds_granted(), out_entropy != nullptr, out_argmax != nullptr, sel.masked());
  int32_t* n_valid = nullptr;
  int32_t* row_index = nullptr;
  if (sel.masked()) {
    n_valid = reinterpret_cast<int32_t*>(ws);
    row_index = reinterpret_cast<int32_t*>(ws + kFusedIndexOffset);
    CompactArgs c{sel, row_index, n_valid, out_lp, out_lse, out_entropy, out_ref_lp, out_k3, out_argmax,
                  (int)n_tokens, plan.shape, joint ? 1 : 0};
    hipLaunchKernelGGL(compact_rows_kernel, dim3(1), dim3(1024), 0, stream, c);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  FusedArgs a;
  a.hidden = static_cast<const char*>(hidden);
  a.sel = sel;
  a.row_index = row_index;
  a.hidden_index = hidden_rows ? hidden_rows : row_index;
  a.n_rows = (int)n_rows;
  a.n_valid = n_valid;
  a.hidden_stride_b = (uint32_t)(hidden_stride * 2);
  a.weight_stride_b = (uint32_t)(weight_stride * 2);
  a.hidden_bytes = (uint32_t)(((n_rows - 1) * hidden_stride + H) * 2);  // read by the generic kernel only (< 4 GiB there)
  const char* second_hidden = static_cast<const char*>(hidden_ref);
  if (norm_weight) {  // normalise the valid rows into a dense buffer and multiply that
    char* normed = ws + layout.normed;
    char* normed_ref = hidden_ref != hidden ? ws + layout.normed_second : normed;
    NormArgs na{{a.hidden, second_hidden}, static_cast<const uint16_t*>(norm_weight), {normed, normed_ref}, a.hidden_index, n_valid,
                a.hidden_stride_b, (int)n_tokens, (int)n_rows, (int)H, norm_eps};
    hipLaunchKernelGGL(rmsnorm_rows_kernel, dim3((unsigned)((n_tokens + 3) / 4), hidden_ref != hidden ? 2 : 1), dim3(256), 0, stream, na);
    second_hidden = normed_ref;
    a.hidden = normed;
    a.hidden_index = nullptr;
    a.hidden_stride_b = (uint32_t)(H * 2);
    a.hidden_bytes = (uint32_t)(n_tokens * H * 2);
  }
  a.hidden2 = joint ? second_hidden : nullptr;
  a.n_tokens = swept;
  a.H = (int)H;
  a.V = (int)V;
  // Workspace header: [0] n_valid, [16..40) the schedule derived from it on the device.
  a.sched_dev = sel.masked() ? reinterpret_cast<const FusedSchedule*>(n_valid + 4) : nullptr;
  a.sched = plan.full;
  a.scale = kLog2e / temperature;
  FusedPartial* p0 = reinterpret_cast<FusedPartial*>(ws + layout.partials);
  FusedPartial* p1 = reinterpret_cast<FusedPartial*>(ws + layout.partials_second);

  a.weight = static_cast<const char*>(w0);
  a.partials = p0;
  int n_parts = out_entropy ? launch_main<true>(a, plan, out_argmax != nullptr, stream)
                            : launch_main<false>(a, plan, out_argmax != nullptr, stream);
  if (n_parts < 0) return hipErrorInvalidConfiguration;
  if (n_parts > 0) {  // small-batch kernel: one part per workgroup, whatever the mask
    a.sched = FusedSchedule{1, n_parts / kPartsPerSplit, n_parts, kTileGeneric, 0, 0};
    a.sched_dev = nullptr;
  }
  const char* first_hidden = a.hidden;
  if (second && !joint) {
    a.weight = static_cast<const char*>(w1);
    a.hidden = second_hidden;
    a.partials = p1;
    if (launch_main<false>(a, plan, false, stream) < 0) return hipErrorInvalidConfiguration;
    a.hidden = first_hidden;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;

  CombineArgs c;
  c.partials = p0;
  c.partials_ref = second && !joint ? p1 : nullptr;
  c.joint = joint ? 1 : 0;
  c.row_index = row_index;
  c.n_valid = n_valid;
  c.out_lp = out_lp;
  c.out_lse = out_lse;
  c.out_entropy = out_entropy;
  c.out_ref_lp = out_ref_lp;
  c.out_k3 = out_k3;
  c.out_argmax = out_argmax;
  c.hidden_rows = hidden_rows;
  c.n_rows = (int)n_rows;
  c.n_tokens = (int)n_tokens;
  c.sched_dev = a.sched_dev;
  c.sched = a.sched;
  c.scale = a.scale;
  hipLaunchKernelGGL(fused_combine_kernel, dim3((unsigned)((n_tokens + 3) / 4)), dim3(256), 0, stream, c);
  return hipGetLastError();
}

hipError_t fused_lmhead_launch(const void* hidden, const int32_t* hidden_rows, int64_t n_rows, const void* norm_weight, float norm_eps, const void* w0,
                               const void* w1, int64_t n_tokens, int64_t H, int64_t V, int64_t hidden_stride,
                               int64_t weight_stride, const RowSel& sel, float temperature, float* out_lp, float* out_lse,
                               float* out_entropy, int32_t* out_argmax, float* out_ref_lp, float* out_k3,
                               const FusedLayout& layout, void* workspace, hipStream_t stream) {
  return fused_launch_impl(hidden, hidden_rows, n_rows, nullptr, norm_weight, norm_eps, w0, w1, n_tokens, H, V, hidden_stride, weight_stride,
                           sel, temperature, out_lp, out_lse, out_entropy, out_argmax, out_ref_lp, out_k3,
                           layout, workspace, stream);
}

hipError_t fused_pair_launch(const void* hidden, const void* hidden_ref, const void* norm_weight, float norm_eps,
                             const void* w0, const void* w1, int64_t n_tokens, int64_t H, int64_t V,
                             int64_t hidden_stride, int64_t weight_stride, const RowSel& sel, float temperature, float* out_lp, float* out_entropy,
                             float* out_ref_lp, float* out_k3, const FusedLayout& layout, void* workspace, hipStream_t stream) {
  return fused_launch_impl(hidden, nullptr, n_tokens, hidden_ref, norm_weight, norm_eps, w0, w1, n_tokens, H, V, hidden_stride,
                           weight_stride, sel, temperature, out_lp, nullptr, out_entropy, nullptr,
                           out_ref_lp, out_k3, layout, workspace, stream);
}

}  // namespace tome
