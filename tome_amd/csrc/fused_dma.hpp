// The DMA sweep kernel of the fused lm_head + log-softmax and its launch.  Included by the fused_dma_*.hip files, one per
// combination of optional outputs, which instantiate launch_dma or launch_dma_any and are compiled side by side.
#pragma once
#include "fused_common.hpp"

namespace tome {

// ===============================================================================================
// Fast path (H % 64 == 0): 512 lanes, 256 x 256 tile, v_mfma_f32_16x16x32_bf16, K slabs DMA'd straight
// into LDS, double-buffered (a third W buffer in the DEEP form, below).
//
//   * 8 waves as 2 (vocab) x 4 (token), 128 vocab x 64 tokens per wave as 8 x 4 blocks of 16x16.  The
//     16x16x32 MFMA moves half the accumulator bytes per FLOP of the 32x32x16 one; on this
//     power-limited part that alone is worth 12-16 % (measured with the instruction swapped in place).
//     The partial layout is shared with the other kernels.
//   * global_load_lds_dwordx4: every lane fetches 16 bytes and the wave's 1 KB lands contiguously
//     in LDS, bypassing registers.  No staging registers are needed, which leaves room to
//     double-buffer the MFMA fragments.
//   * What this kernel pays for beside its MFMAs is the L2 -> LDS fill (64 KB per 256x256x64 MACs and CU: the
//     requests cost in proportion to their number, wherever the data lands and whether or not it hits in L2 -
//     mostly as engine clock, which this power-limited part lowers under the added load, not as issue slots),
//     and the L2 serves it by the request, not by the byte: a slab row is therefore one whole 128-byte
//     cache line (K = 64), which streams 1.5x faster than 64-byte rows.  Two 64 KB slabs (W 256 rows +
//     hidden 256 rows each) fill the LDS; one is computed on while the other is in flight.  Step s (one
//     slab = two K = 32 MFMA sub-steps of 32 MFMAs per wave, each in two halves by vocab block) runs
//         MFMA(s, k0, blocks 0-3) | reads (s, k0, blocks 4-7), requests 5-6 of slab s+1
//         MFMA(s, k0, blocks 4-7) | reads (s, k1, blocks 0-3 and hidden), requests 7-8 of slab s+1
//         MFMA(s, k1, blocks 0-3) | reads (s, k1, blocks 4-7)
//         own reads and own share of slab s+1 complete; barrier
//         MFMA(s, k1, blocks 4-7) | reads (s+1, k0, blocks 0-3 and hidden), requests 1-4 of slab s+2
//     After the barrier everybody has read all of slab s, so it can be refilled, and slab s+1 is
//     visible before its first fragments are read, which happens under the last quarter of the
//     MFMAs - the MFMA stream has no bubble at step or vocab-tile boundaries.
//   * Bank conflicts are avoided by an XOR swizzle instead of padding (DMA writes are dense).
//     The LDS has 64 four-byte banks, so a 16-lane phase of a 128-bit read is conflict-free when
//     its 16 rows hit 16 different 16-byte bank groups.  A 128-byte row r covers groups
//     8*(r&1) .. +7, so chunk c of row r is stored at chunk position c ^ ((r >> 1) & 7); the
//     lane that DMA-writes position p of row r fetches global chunk p ^ ((r >> 1) & 7).
// ===============================================================================================
//
// The token tile is a template parameter, 64 .. 256 tokens: of the four token waves two own NA and two own NB blocks of
// 16 tokens, NA = NB or NB + 1.  (4, 4) is the shape described above; (4, 3), (3, 3), (2, 2), (2, 1) and (1, 1) are tiles of
// 224, 192, 128, 96 and 64 tokens.  Waves w and w + 4 share a SIMD and own NA and NB blocks, so an uneven pair still loads
// all four SIMDs alike; the two widths are two bodies of one kernel that meet at the same barriers.  A tile costs its full
// MFMA work and fill however few of its tokens exist, and at up to ~1500 tokens that padding was what most shapes were
// furthest from their floor by (V = 151936, us before -> now, H = 1024 / 2560: 130 tokens 82 -> 70 / 183 -> 163, 200:
// 83 -> 77 / 189 -> 181, 300: 131 -> 109 / 330 -> 262, 384: 132 -> 109 / 338 -> 256, 600: 193 -> 178 / 454 -> 425, 1300: 376 -> 351 /
// 883 -> 817).  160 = (3, 2) was built too: equal to 192 where it could be used.  fused_tile_cost holds the choice.
constexpr int k2BV = 256, k2WG = 512;
constexpr int k2BK = kDmaSlab;
constexpr int k2RowBytes = k2BK * 2;                     // 128: one cache line
// Slab buffers, as many as fit the 160 KB of LDS: two for the tiles of 192 tokens and more (56-64 KB per slab), three
// otherwise.  The W halves and the hidden halves form two rings of that depth.
constexpr int dma_bufs(int tokens) { return tokens > 128 ? 2 : 3; }
// With two buffers a slab's request is issued in three portions - in the last quarter of the step that frees
// its buffer, and in the first two quarters of the next step - instead of all at once: right after a barrier
// all eight waves are at the same point, and 64 requests issued together queue up in the memory pipeline
// while the waves that issued them cannot issue their MFMAs.
constexpr int kIssueQ4 = 4, kIssueQ1 = 2;   // instructions of the eight in the last / first quarter; the rest in the second
constexpr int k2Loads = k2BV * (k2RowBytes / 16) / k2WG; // DMA instructions per lane and slab for W (4)
constexpr int k2NBV = kWaveV / 16;                       // 16x16 vocab blocks per wave tile: 8
static_assert(k2Loads == 4 && k2NBV == 8, "the MFMA/DMA interleave is written for this shape");
constexpr int dma_tile_tokens(int na, int nb) { return (na + nb) * 32; }                       // two token waves of na and two of nb blocks of 16
constexpr int dma_w_bytes() { return k2BV * k2RowBytes; }                                      // 32768
constexpr int dma_h_bytes(int tokens) { return tokens * k2RowBytes; }                          // 32768 at 256 tokens
// DEEP (tiles of 192 tokens and more): a third W buffer, with 256 tokens all of the CU's LDS; see the kernel.
constexpr int dma_w_bufs(int tokens, bool deep) { return deep ? 3 : dma_bufs(tokens); }
constexpr int dma_lds_bytes(int tokens, bool deep = false) {  // 131072 at 256 tokens, 163840 with the third W buffer
  return dma_w_bufs(tokens, deep) * dma_w_bytes() + dma_bufs(tokens) * dma_h_bytes(tokens);
}

// AUX: the request's cache policy bits (0 = default, 2 = non-temporal).  Hidden rows always go with the default; W rows
// do wherever several token tiles read them (there non-temporal requests for either operand measured 1.5-5 % slower),
// see WNT at the kernel.
template <int AUX = 0>
__device__ __forceinline__ void dma16(const char* gptr, char* lds_wave_base) {
  __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t*>(gptr),
                                   (__attribute__((address_space(3))) uint32_t*)lds_wave_base, 16, 0, AUX);
}

// Scheduling pattern: N_READS times (N_MFMA MFMAs, then one LDS read).
template <int N_MFMA, int N_READS>
__device__ __forceinline__ void pair_reads() {
#pragma unroll
  for (int q = 0; q < N_READS; ++q) {
    __builtin_amdgcn_sched_group_barrier(0x008, N_MFMA, 0);  // MFMA
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // DS read
  }
}

// Vocab ranges are dealt in units of 32 rows and a workgroup cuts its range into the fewest tiles of at most 256 rows,
// all of the same height or one unit apart (the taller ones first): V = 151936 over 16 splits is 297 units per
// workgroup = 31 tiles of 256 rows + 7 of 224, where whole 256-row tiles would give some workgroups 38 tiles and others
// 37 - and a tile costs its full MFMA work however few of its rows count.  A tile of nb blocks of 16 rows per wave
// (nb = 1 .. 8) runs the same pipeline with 8 * nb MFMAs per wave and step.  Its slab keeps the LDS layout of a whole
// tile (rows 0..127 for the waves of vocab half 0, 128..255 for half 1, so fragment addresses do not change); each
// half holds 16 * nb rows of W and the rest of its LDS rows are requested as copies of its last row and never multiplied.
//
// DEEP: the tiles of 192 tokens and more with THREE W buffers and two hidden buffers (at 256 tokens 160 KB, the whole LDS of a CU).  The W half of
// a slab is requested two steps ahead - in the first two quarters of a step, its buffer free since the previous step's
// barrier - and the hidden half, which comes from L2, one step ahead, after the step's own barrier; before a barrier
// the four W instructions of the newest request stay in flight.  Faster wherever a step waits for its fill: 10-15 %
// where every workgroup streams W rows of its own (one token tile), 2-3 % at 4096 x 1024 tokens x hidden, nothing from
// 8192 x 4096 on; with the entropy its fold spills and it only pays up to 1024 tokens, behind a mask also beyond where a tile has the
// K steps for it (fused_plan, FusedPlan::any_deep: rules and figures).
//
// WNT: W is requested non-temporally.  Where W streams through once or a few times (up to four token tiles) its rows have
// no business in the caches that the hidden rows and the partials live in: 64 x 4096 tokens x hidden 221 -> 205 us,
// 256 x 1024 88 -> 84, 128 x 4096 234 -> 230, 512 x 1024 138 -> 135.5, 1024 x 4096 924 -> 917; from 2048 tokens on the
// workgroups of an XCD that share a W tile want it kept (4096 x 1024: 936 -> 951), and so do three 128-token tiles
// (384 x 1024: 130 -> 138).
//
// ROT (tiles of up to 128 tokens, W requested non-temporally, no argmax): where one token tile streams W and its rows lie a multiple of
// 8 KB apart, the workgroups start their K loops at different slabs (the sums just begin elsewhere).  Not with the argmax: rows of W
// that are equal bit for bit must have equal logits wherever they lie, or the first of them is not the one that is named.  In step, all of them would ask
// the same few memory channels for the same columns of their rows: V = 50257 / 64001 / 100000 / 128256 / 151936 x H = 4096, 64 tokens
// 94 -> 68, 119 -> 86, 143 -> 130, 197 -> 165, 201 -> 190 us, 96 tokens 96 -> 75, 121 -> 87, 152 -> 135, 198 -> 162, 221 -> 197, 128 tokens
// 98 -> 81, 122 -> 91, 155 -> 151, 204 -> 174, 222 -> 218 (to the kernels before it; 42 shapes up to H = 8192 0.72 .. 0.98).  Row pitches
// of 2 and 5 KB gain nothing, nor does a W that the memory-side cache holds (32000 x 4096: 50.0 -> 50.5).
__device__ __host__ inline bool dma_rotates(const FusedArgs& a) { return (a.weight_stride_b & 8191) == 0; }
// NBT: this wave's token blocks; BT: the workgroup's token tile; tok0: this wave's first token in it.
template <bool ENT, bool AMAX, int NBT, int BT, int HI, bool DEEP, bool WNT, bool ROT>
__device__ __forceinline__ void dma_sweep(const FusedArgs& a, const FusedSchedule& sch, int n_valid, int ttile, int split, int wave,
                                          int tok0) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];  // (handed down as a pointer it costs the sweep 2-4 %)
  static_assert((BT >= 224 && (HI == 4 || HI == 3)) || (BT < 224 && HI == 0), "tiles of 224 / 256 tokens: every vocab tile 256 (HI = 4) or 224 rows; others: mixed heights");
  static_assert(!DEEP || BT > 128, "the third W buffer is for the tiles with two buffers");
  // Waves of four token blocks run at the limit of the register file: their kernels keep ONE tile height per launch (4 + HI
  // blocks per wave, the host picks 256 or 224 rows), because the code for two or more heights in one kernel costs it 60 and more spilled
  // registers whose reloads, at every tile change, wait for memory behind the W stream (measured with heights of 224 and
  // 256 rows mixed: +8 % at 4096 x 1024 instead of the 1.7 % that the even shares would save).  The smaller token tiles
  // have registers to spare and mix heights as described above.
  constexpr bool kMixed = HI == 0;
  constexpr int kMaxBlocks = kMixed ? 8 : 4 + HI;   // 16-row vocab blocks per wave in the tallest tile
  constexpr int kNBVw = 8;                          // accumulator block rows per wave
  constexpr int k2NBT = NBT;                        // 16-token blocks per wave
  constexpr int kBufs = dma_bufs(BT);               // hidden buffers
  constexpr int kBufsW = dma_w_bufs(BT, DEEP);      // W buffers
  constexpr int kWBytes = dma_w_bytes(), kHBytes = dma_h_bytes(BT);
  constexpr int kHBase = kBufsW * kWBytes;          // the hidden ring starts behind the W ring
  constexpr int kBLoads = NBT;                      // DMA instructions per lane and slab for the hidden rows (an uneven
                                                    // tile's last 32 rows are fetched by waves 0-3, the ones with NA blocks)
  constexpr int k2DmaPerSlab = k2Loads + kBLoads;   // 8 at NBT = 4
  // Portions of a request (see kIssueQ4): with three buffers everything goes out in the last quarter.
  constexpr int kP4 = kBufs == 2 ? kIssueQ4 : k2DmaPerSlab;
  constexpr int kP1 = kBufs == 2 ? kIssueQ1 : 0;
  constexpr int kP2 = k2DmaPerSlab - kP4 - kP1;
  static_assert(kP4 >= 1 && kP1 >= 0 && kP2 >= 0 && kP1 <= 8 && kP2 <= 8, "portions of the eight instructions");
  static_assert(kBufs == 2 || kP4 == k2DmaPerSlab, "split requests are written for two buffers");
  // Which of the eight instructions (0-3: W, 4-7: hidden) go out in the first, second and last quarter of a step.
  // Two buffers: a request starts in the last quarter of the step that frees its buffers (W first: it has furthest to
  // come) and ends in the second quarter of the next.  DEEP: request step + 2 as a whole inside one step, W in the first
  // two quarters (its buffer was freed by the previous step's barrier), hidden after this step's barrier.
  constexpr int kQ1Lo = DEEP ? 0 : kP4, kQ1Hi = DEEP ? 2 : kP4 + kP1;
  constexpr int kQ2Lo = kQ1Hi, kQ2Hi = DEEP ? 4 : k2DmaPerSlab;
  constexpr int kQ4Lo = DEEP ? 4 : 0, kQ4Hi = DEEP ? k2DmaPerSlab : kP4;
  constexpr bool kDoneAfterQ4 = DEEP || kP4 == k2DmaPerSlab;
  // Requests complete in the order they were issued, so "slab s has landed" is a count of newer instructions that
  // may still be in flight.  Before a step's barrier (slab step + 1 must be there) those are the whole requests
  // of the slabs after it (DEEP: the W instructions of request step + 2); before the loop (slab 0) also the first
  // portion of the newest request (DEEP: the whole request for slab 1).
  constexpr int kInFlightAtStep = DEEP ? k2Loads : (kBufs - 2) * k2DmaPerSlab;
  constexpr int kInFlightAtStart = DEEP ? k2DmaPerSlab : (kBufs - 2) * k2DmaPerSlab + kP4;

  const int t0 = ttile * BT;
  // This workgroup's vocab range in 32-row blocks (unit32 blocks per unit: 1, or 7 / 8 when ranges are whole tiles).
  const int u0 = (int)((int64_t)split * sch.n_vunits / sch.n_splits) * sch.unit32;
  const int u1 = (int)((int64_t)(split + 1) * sch.n_vunits / sch.n_splits) * sch.unit32;
  const int n_units = u1 - u0;                      // >= 1: every split holds at least one unit
  // With mixed heights every workgroup of a launch cuts its range into the SAME number of tiles (the longest range's), so
  // that all of them step through tiles of (nearly) the same heights at the same time: the workgroups that share a
  // hidden-state or W stream in an XCD's L2 only hit there while they stay in step.
  const int n_tiles = kMixed ? ((sch.n_vunits + sch.n_splits - 1) / sch.n_splits * sch.unit32 + 7) >> 3 : n_units / kMaxBlocks;
  const int nb_short = kMixed ? n_units / n_tiles : kMaxBlocks;  // 16-row blocks per wave of the shorter tiles (1 .. 8)
  const int n_tall = kMixed ? n_units - nb_short * n_tiles : 0;  // tiles with one block more: they come first
  const int row0 = u0 * 32;
  auto tile_blocks = [&](int tile) { return nb_short + (tile < n_tall ? 1 : 0); };
  auto tile_row0 = [&](int tile) {
    if constexpr (!kMixed) return row0 + tile * (32 * kMaxBlocks);
    else return row0 + 32 * (tile * nb_short + (tile < n_tall ? tile : n_tall));
  };

  const int lane = threadIdx.x & 63;
  const int wave_v = wave & 1;
  const int l16 = lane & 15, g = lane >> 4;  // 16x16 MFMA: token column, lane group

  // ---- DMA assignment: instruction j of wave w fills LDS rows (j*8 + w)*8 .. +7 of an operand ----
  // All address arithmetic is incremental: per-lane pointers advance by one slab (128 bytes) per
  // request and are rebased at vocab-tile changes, so a step carries no multiplies or divides.
  const int dr = lane >> 3;                                   // row inside the 8-row group
  const int dc = (lane & 7) ^ (4 * (wave & 1) + (dr >> 1));   // global chunk: position ^ ((row >> 1) & 7)
  const int nk = a.H / k2BK;
  const int k0 = ROT && sch.n_ttiles == 1 && dma_rotates(a) ? split % nk : 0;
  const char* pa[k2Loads];  // next W slab to request, per DMA instruction
  const char* pb[kBLoads];  // next hidden slab
  // Mixed heights: LDS row r of a W slab holds vocab row  base + (r / 128) * wr + min(r % 128, wr - 1)  of tile `tile`,
  // wr = rows per wave of that tile.  One height: LDS row r is tile row r; the 32 LDS rows past a 224-row tile are requested
  // as copies of rows that waves 0-3 fetch with the same instruction.  Rows past V (last tile only) read the last row
  // and are masked in the epilogue.
  auto point_a = [&](int tile) {
    const int64_t base = tile_row0(tile);
    const int wr = kMixed ? tile_blocks(tile) * 16 : kMaxBlocks * 16;
    // The lane's row and chunk are derived afresh here (the empty asm hides that they are loop invariants): hoisted
    // out of the sweep, the 64-bit per-lane address terms built from them would stay live across every step, and this
    // kernel has no register left for them.
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int dr = ln >> 3;
    const int dc = (ln & 7) ^ (4 * (wave & 1) + (dr >> 1));
#pragma unroll
    for (int j = 0; j < k2Loads; ++j) {
      const int r = (j * 8 + wave) * 8 + dr;
      int64_t v;
      if constexpr (kMixed) {
        const int in_half = (r & 127) < wr ? (r & 127) : wr - 1;
        v = base + (r >> 7) * wr + in_half;
      } else {
        v = base + ((HI == 4 || r < 2 * wr) ? r : r - 32);
      }
      v = v < a.V ? v : a.V - 1;
      pa[j] = a.weight + v * a.weight_stride_b + dc * 16 + (ROT ? k0 * k2RowBytes : 0);
    }
  };
  point_a(0);
#pragma unroll
  for (int j = 0; j < kBLoads; ++j) {
    int p = t0 + (j * 8 + wave) * 8 + dr;
    p = p < n_valid ? p : n_valid - 1;
    const TokenSource src = token_source(a, p, n_valid);
    const int tok = a.hidden_index ? min(max(a.hidden_index[src.q], 0), a.n_rows - 1) : src.q;
    pb[j] = src.hidden + (int64_t)tok * a.hidden_stride_b + dc * 16 + (ROT ? k0 * k2RowBytes : 0);
  }

  // ---- per-lane token state: one token per 16-token block, shared by the four lane groups ---------
  RowStat st[k2NBT];
  float tx[k2NBT];
  int tgt[k2NBT];
#pragma unroll
  for (int bt = 0; bt < k2NBT; ++bt) {
    st[bt] = stat_identity();
    tx[bt] = -INFINITY;
    tgt[bt] = token_target(a, t0 + tok0 + bt * 16 + l16, n_valid);
  }

  // ---- fragment read offsets inside a slab (swizzled): lane group g reads chunk 4*ks + g ----------
  const int swz = (g ^ ((l16 >> 1) & 7)) * 16;  // sub-step k0; k1 is this ^ 64
  // the wave's first LDS row (128 with mixed heights) is a multiple of 16: the swizzle term stays l16's
  const int rdA = (wave_v * (kMixed ? 128 : kMaxBlocks * 16) + l16) * k2RowBytes + swz;
  const int rdB = (tok0 + l16) * k2RowBytes + swz;

  const int n_steps = n_tiles * nk;
  const int64_t slab_rewind = (int64_t)(nk - 1) * k2RowBytes;
  int i_kt = 0, i_tile = 0;  // slab the next request fetches
  int i_col = k0;            // its place in the row (ROT)
  int issued = 0;            // slabs requested so far; request q lands in buffers q % kBufs

  // One of the DMA instructions of the next request (0-3: W rows; the others: hidden rows).  Past the last slab
  // the request is repeated (same addresses, same buffer, identical bytes): it is issued on every step so that
  // the code has no branch and the wait counts stay static.
  auto issue_piece = [&](int piece) {
    const unsigned slab = (unsigned)(issued < n_steps ? issued : n_steps - 1);
    if (piece < k2Loads) dma16<WNT ? 2 : 0>(pa[piece], smem + (slab % kBufsW) * kWBytes + wave * 1024 + piece * 8192);
    else dma16(pb[piece - k2Loads], smem + kHBase + (slab % kBufs) * kHBytes + wave * 1024 + (piece - k2Loads) * 8192);
  };
  auto issue_done = [&]() {
    ++issued;
    if (issued >= n_steps) return;  // the stream stays on the last slab
    if constexpr (ROT) {
      int64_t on = k2RowBytes;
      if (++i_col == nk) {
        i_col = 0;
        on = -slab_rewind;
      }
#pragma unroll
      for (int j = 0; j < kBLoads; ++j) pb[j] += on;
      if (++i_kt < nk) {
#pragma unroll
        for (int j = 0; j < k2Loads; ++j) pa[j] += on;
      } else {
        i_kt = 0;
        ++i_tile;
        if (i_tile < n_tiles) point_a(i_tile);
      }
      return;
    }
    if (++i_kt < nk) {
#pragma unroll
      for (int j = 0; j < k2Loads; ++j) pa[j] += k2RowBytes;
#pragma unroll
      for (int j = 0; j < kBLoads; ++j) pb[j] += k2RowBytes;
    } else {
      i_kt = 0;
      ++i_tile;
#pragma unroll
      for (int j = 0; j < kBLoads; ++j) pb[j] -= slab_rewind;
      if (i_tile < n_tiles) point_a(i_tile);
    }
  };
  // Fragments of one K = 32 sub-step of a slab: W blocks [i0, i0 + n) or the hidden blocks.
  // DEEP: the offsets of the second sub-step (rdA ^ 64, rdB ^ 64) are formed where they are used (the empty asm hides
  // that they are loop invariants).  Kept in registers across the sweep they are spilled, and a reload inside a step
  // makes the compiler wait for EVERY outstanding memory operation - the requests two slabs ahead included.
  auto read_a = [&](int slot, int ks, int i0, bf16x8 (&fa)[4], auto n) {
    const char* slab = smem + ((unsigned)slot % kBufsW) * kWBytes;
    int rd = rdA;
    if constexpr (DEEP) asm volatile("" : "+v"(rd));
#pragma unroll
    for (int i = 0; i < decltype(n)::value; ++i)
      fa[i] = *reinterpret_cast<const bf16x8*>(slab + (rd ^ (ks * 64)) + (i0 + i) * 16 * k2RowBytes);
  };
  auto read_b = [&](int slot, int ks, bf16x8 (&fb)[k2NBT]) {
    const char* slab = smem + kHBase + ((unsigned)slot % kBufs) * kHBytes;
    int rd = rdB;
    if constexpr (DEEP) asm volatile("" : "+v"(rd));
#pragma unroll
    for (int j = 0; j < k2NBT; ++j)
      fb[j] = *reinterpret_cast<const bf16x8*>(slab + (rd ^ (ks * 64)) + j * 16 * k2RowBytes);
  };

  // Prologue: whole requests for all buffers but the last, and the first portion of the last one's (DEEP: slabs 0 and 1).
#pragma unroll
  for (int q = 0; q < (DEEP ? 2 : kBufs - 1); ++q) {
#pragma unroll
    for (int piece = 0; piece < k2DmaPerSlab; ++piece) issue_piece(piece);
    issue_done();
  }
  if constexpr (!DEEP) {
#pragma unroll
    for (int piece = 0; piece < kP4; ++piece) issue_piece(piece);
    if constexpr (kP4 == k2DmaPerSlab) issue_done();
  }
  // Slab 0 has landed (this wave's share): only the requests of the later slabs may still be in flight.
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kInFlightAtStart) : "memory");
  __builtin_amdgcn_s_barrier();

  constexpr std::integral_constant<int, 4> kFour{};
  bf16x8 fa_lo[4], fa_hi[4], fb0[k2NBT], fb1[k2NBT];
  read_a(0, 0, 0, fa_lo, kFour);
  read_b(0, 0, fb0);

  f32x4v acc[kNBVw][k2NBT];
#pragma unroll
  for (int i = 0; i < kNBVw; ++i)
#pragma unroll
    for (int j = 0; j < k2NBT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.f;

  // 4 * n MFMAs on n vocab blocks; in a whole tile the group barriers then put one LDS read or DMA request behind
  // every MFMA (or every second one), so that its issue hides under the MFMA's execution.
  // `fresh`: the first K sub-step of a vocab tile starts from a zero C operand, which saves clearing
  // the 128 accumulator registers after every fold.
  auto mfma_half = [&](int i0, bf16x8 (&fa)[4], bf16x8 (&fb)[k2NBT], auto fresh, auto n) {
    const f32x4v zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < decltype(n)::value; ++i)
#pragma unroll
      for (int j = 0; j < k2NBT; ++j)
        acc[i0 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], decltype(fresh)::value ? zero : acc[i0 + i][j],
                                                                   0, 0, 0);
  };
  // The two waves of a SIMD (w and w + 4) at different priorities: they fall out of step between barriers, one's fragment reads under
  // the other's MFMAs (1 % at 96 .. 600 tokens, nothing where power decides: 200 x 2560 182.5 -> 180.7 us, 96 x 2560 142.6 -> 141.1).
  if (wave >= 4) __builtin_amdgcn_s_setprio(1);
  int step = 0;
  // N times (one MFMA, then one DMA request).
  auto pair_dma = [](auto n) {
#pragma unroll
    for (int q = 0; q < decltype(n)::value; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // VMEM (DMA request)
    }
  };
  // One K slab on a tile of `lo` + `hi` vocab blocks per wave: lo = min(nb, 4), hi = nb - lo.  The fragments of the
  // NEXT step's first quarter are always read for four blocks (the next step may belong to a taller tile).
  auto do_step = [&](auto fresh, auto lo, auto hi) {
    constexpr int LO = decltype(lo)::value, HIB = decltype(hi)::value;
    constexpr bool kTuned = NBT >= 3 && LO == 4 && HIB >= 3;  // the interleave below is written for tiles of 224 and 256 rows
    __builtin_amdgcn_sched_barrier(0);
    read_a(step, 0, 4, fa_hi, hi);
#pragma unroll
    for (int piece = kQ1Lo; piece < kQ1Hi; ++piece) issue_piece(piece);  // two buffers: second portion of the request for slab step + 1
    mfma_half(0, fa_lo, fb0, fresh, lo);
    if constexpr (kTuned) {
      pair_reads<2, HIB>();
      pair_dma(std::integral_constant<int, kQ1Hi - kQ1Lo>{});
    }
    __builtin_amdgcn_sched_barrier(0);
    read_a(step, 1, 0, fa_lo, lo);
    read_b(step, 1, fb1);
#pragma unroll
    for (int piece = kQ2Lo; piece < kQ2Hi; ++piece) issue_piece(piece);  // third portion
    mfma_half(4, fa_hi, fb0, fresh, hi);
    if constexpr (kTuned) {
      if constexpr (kQ2Hi == kQ2Lo) {
        pair_reads<NBT == 4 ? 2 : 1, 4 + NBT>();
      } else {
        pair_reads<1, 4 + NBT>();
        pair_dma(std::integral_constant<int, kQ2Hi - kQ2Lo>{});
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!kDoneAfterQ4) issue_done();
    read_a(step, 1, 4, fa_hi, hi);
    mfma_half(0, fa_lo, fb1, std::false_type{}, lo);
    if constexpr (kTuned) pair_reads<2, HIB>();
    __builtin_amdgcn_sched_barrier(0);
    // This wave has read all it needs of slab `step` and its share of slab step+1 has landed; after
    // the (fence-less) barrier both hold for everyone.  (With three buffers the request of slab step+2
    // stays in flight across the barrier.)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kInFlightAtStep) : "memory");
    __builtin_amdgcn_s_barrier();
    // Last quarter: first fragments of slab step+1 (after the last step a stale buffer, unused) and the
    // first portion of the next request, which refills the buffers of slab `step`.  The DMA requests write
    // LDS, so they keep their program order after the fragment reads.
    __builtin_amdgcn_sched_barrier(0);
    read_a(step + 1, 0, 0, fa_lo, kFour);
    read_b(step + 1, 0, fb0);
#pragma unroll
    for (int piece = kQ4Lo; piece < kQ4Hi; ++piece) issue_piece(piece);
    mfma_half(4, fa_hi, fb1, std::false_type{}, hi);
    if constexpr (kTuned) {
      pair_reads<1, 4 + NBT>();
      pair_dma(std::integral_constant<int, kQ4Hi - kQ4Lo>{});
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kDoneAfterQ4) issue_done();
    ++step;
  };

  // Two runs of tiles: n_tall tiles of nb_short + 1 blocks, then the others of nb_short blocks.
  auto run_tiles = [&](int first, int last, auto lo, auto hi) {
    constexpr int NB = decltype(lo)::value + decltype(hi)::value;
    for (int tile = first; tile < last; ++tile) {
      do_step(std::true_type{}, lo, hi);
      for (int kt = 1; kt < nk; ++kt) do_step(std::false_type{}, lo, hi);
      const int v0 = tile_row0(tile);
      fold_tile16<ENT, AMAX, NB>(acc, st, tx, tgt, v0 + wave_v * NB * 16, g, v0 + 2 * NB * 16 > a.V, a.V, a.scale);
    }
  };
  using std::integral_constant;
  if constexpr (!kMixed) {
    constexpr integral_constant<int, HI == 0 ? 4 : HI> kHi{};
    for (int tile = 0; tile < n_tiles; ++tile) {
      do_step(std::true_type{}, kFour, kHi);
      for (int kt = 1; kt < nk; ++kt) do_step(std::false_type{}, kFour, kHi);
      const int v0 = row0 + tile * (32 * kMaxBlocks);
      fold_tile16<ENT, AMAX, kMaxBlocks>(acc, st, tx, tgt, v0 + wave_v * kMaxBlocks * 16, g, v0 + 32 * kMaxBlocks > a.V, a.V, a.scale);
    }
  } else {
    for (int run = 0; run < 2; ++run) {
      const int first = run == 0 ? 0 : n_tall, last = run == 0 ? n_tall : n_tiles;
      if (first >= last) continue;
      const int nb = nb_short + (run == 0 ? 1 : 0);
      switch (nb) {
        case 1: run_tiles(first, last, integral_constant<int, 1>{}, integral_constant<int, 0>{}); break;
        case 2: run_tiles(first, last, integral_constant<int, 2>{}, integral_constant<int, 0>{}); break;
        case 3: run_tiles(first, last, integral_constant<int, 3>{}, integral_constant<int, 0>{}); break;
        case 4: run_tiles(first, last, integral_constant<int, 4>{}, integral_constant<int, 0>{}); break;
        case 5: run_tiles(first, last, integral_constant<int, 4>{}, integral_constant<int, 1>{}); break;
        case 6: run_tiles(first, last, integral_constant<int, 4>{}, integral_constant<int, 2>{}); break;
        case 7: run_tiles(first, last, integral_constant<int, 4>{}, integral_constant<int, 3>{}); break;
        default: run_tiles(first, last, kFour, kFour); break;
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no request may outlive the workgroup's LDS

  write_partials16(st, tx, a.partials, t0 + tok0, n_valid, split * kPartsPerSplit + wave_v,
                   sch.n_splits * kPartsPerSplit, l16, g, a.scale);
}

// TILE: the token tile (index of FusedTile), or kAnyTile: one kernel with the bodies of all of them, which takes the one that the
// schedule names.  Behind a mask the number of tokens, and so the tile, is only known on the device.  The combined kernel
// costs about 1 us a launch more and runs the 256-token tile 1-2 % slower than the kernels of one tile each.
constexpr int kAnyTile = -1;
template <bool ENT, bool AMAX, int TILE, bool DEEP, bool WNT, bool ROT = false>
__global__ __launch_bounds__(k2WG) void fused_lmhead_dma_kernel(FusedArgs a) {
  touch_args(a);
  int n_valid = a.n_tokens;
  FusedSchedule sch = a.sched;
  if (a.sched_dev) {  // behind a mask, next to the count
    n_valid = *a.n_valid << (a.hidden2 ? 1 : 0);
    sch = *a.sched_dev;
  }
  int ttile, split;
  if (n_valid <= 0 || !fused_locate(sch, blockIdx.x, ttile, split)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: keeps LDS bases scalar
  auto sweep = [&](auto tile) {
    constexpr FusedTile kTile = fused_tile(decltype(tile)::value);
    constexpr int BT = kTile.tokens, NA = (BT + 32) / 64, NB = BT / 32 - NA, HI = kTile.unit32 == 1 ? 0 : kTile.unit32 - 4;
    constexpr bool kDeep = BT > 128 && (DEEP || BT < 256);
    constexpr bool kRot = BT <= 128 && !AMAX && (TILE == kAnyTile ? WNT : ROT);
    static_assert(BT == dma_tile_tokens(NA, NB), "two token waves of NA blocks, two of NB");
    const int wave_t = wave >> 1;
    if (NA == NB || wave_t < 2) {
      dma_sweep<ENT, AMAX, NA, BT, HI, kDeep, WNT, kRot>(a, sch, n_valid, ttile, split, wave, wave_t * NA * 16);
    } else if constexpr (NA != NB) {  // the same steps, so the same barriers
      dma_sweep<ENT, AMAX, NB, BT, HI, kDeep, WNT, kRot>(a, sch, n_valid, ttile, split, wave, 2 * NA * 16 + (wave_t - 2) * NB * 16);
    }
  };
  if constexpr (TILE != kAnyTile) {
    sweep(std::integral_constant<int, TILE>{});
  } else {
    switch (__builtin_amdgcn_readfirstlane(sch.tile)) {
      case 0: sweep(std::integral_constant<int, 0>{}); break;
      case 1: sweep(std::integral_constant<int, 1>{}); break;
      case 2: sweep(std::integral_constant<int, 2>{}); break;
      case 3: sweep(std::integral_constant<int, 3>{}); break;
      case 4: sweep(std::integral_constant<int, 4>{}); break;
      case 5: sweep(std::integral_constant<int, 5>{}); break;
      case 6: sweep(std::integral_constant<int, 6>{}); break;
      default: sweep(std::integral_constant<int, 7>{}); break;
    }
  }
}

template <bool ENT, bool AMAX, int TILE, bool DEEP, bool WNT, bool ROT = false>
static void launch_dma_form(const FusedArgs& a, int grid, hipStream_t stream) {
  constexpr int kTokens = fused_tile(TILE < 0 ? 0 : TILE).tokens;
  constexpr int kLds = TILE != kAnyTile ? dma_lds_bytes(kTokens, DEEP) : DEEP ? dma_lds_bytes(256, true) : dma_lds_bytes(224, true);
  static_assert(dma_lds_bytes(224, true) >= dma_lds_bytes(256), "the largest body of the combined kernel");
  static DeviceOnce attr_set;  // opt in to > 64 KB of dynamic LDS once per instantiation and device
  if (attr_set.first_on_current_device()) allow_big_lds(&fused_lmhead_dma_kernel<ENT, AMAX, TILE, DEEP, WNT, ROT>, kLds);
  hipLaunchKernelGGL((fused_lmhead_dma_kernel<ENT, AMAX, TILE, DEEP, WNT, ROT>), dim3((unsigned)grid), dim3(k2WG), kLds, stream, a);
}
// deep: three W buffers for the 256-token tile too (FusedPlan::any_deep); w_nt: non-temporal W requests (the kernel's WNT), which up to four
// token tiles take and so never without `deep`.
template <bool ENT, bool AMAX>
void launch_dma_any(const FusedArgs& a, bool deep, bool w_nt, int grid, hipStream_t stream) {
  if (w_nt) return launch_dma_form<ENT, AMAX, kAnyTile, true, true>(a, grid, stream);
  if constexpr (ENT) {
    if (!deep) return launch_dma_form<ENT, AMAX, kAnyTile, false, false>(a, grid, stream);
  }
  launch_dma_form<ENT, AMAX, kAnyTile, true, false>(a, grid, stream);
}
// False, and nothing launched, for a tile without the form asked for.
template <bool ENT, bool AMAX>
bool launch_dma(const FusedArgs& a, int tile, bool deep, bool w_nt, int grid, hipStream_t stream) {
  if (tile < 0 || tile >= kTileGeneric || !dma_has_form(tile, deep)) return false;
  auto go = [&](auto t) {
    constexpr int TILE = decltype(t)::value;
    constexpr bool kBig = fused_tile(TILE).tokens > 128;
    if constexpr (!kBig && !AMAX) {
      if (w_nt && dma_rotates(a)) return launch_dma_form<ENT, AMAX, TILE, false, true, true>(a, grid, stream);
    }
    if (w_nt && (deep || !kBig)) launch_dma_form<ENT, AMAX, TILE, kBig, true>(a, grid, stream);
    else if (deep || !kBig) launch_dma_form<ENT, AMAX, TILE, kBig, false>(a, grid, stream);
    else if constexpr (dma_has_form(TILE, false)) launch_dma_form<ENT, AMAX, TILE, false, false>(a, grid, stream);
  };
  switch (tile) {
    case 0: go(std::integral_constant<int, 0>{}); break;
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    default: go(std::integral_constant<int, 7>{}); break;
  }
  return true;
}

}  // namespace tome
