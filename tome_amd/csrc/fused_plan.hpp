// Planning of a fused lm_head call: which sweep kernel, token tiles, how the vocab axis is dealt, grid and workspace.  Host code, and
// the parts of it that a mask leaves to the device; nothing here needs a GPU.
#pragma once
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace tome {

constexpr int kBV = 256;                 // vocab rows per tile
constexpr int kWaveV = 128;              // vocab rows per wave
constexpr int kPartsPerSplit = kBV / kWaveV;
constexpr int kDmaSlab = 64;             // K columns per step of the DMA kernel

struct FusedPartial {  // 32 bytes per (token, part)
  float mx, s, w, tx;
  int bi;
  int pad[3];
};

// Work decomposition: token tiles x vocab splits.  It depends on the number of valid tokens, which is
// known on the host without a mask and only on the device with one, so it is computed by the host (and
// passed by value) or by compact_rows_kernel (and read from the workspace header); both run the
// same code.  Every kernel of a launch uses the same numbers.
//
// A workgroup owns one token tile and one contiguous range of vocab tiles.
//   * Few token tiles (n_ttiles * 8 <= slots): as many splits as fill the chip in ONE round, rounded
//     down - one workgroup too many would cost a whole extra round.
//   * Many token tiles: several rounds.  The candidates 1..32 are priced as
//         rounds * (longest vocab range + half a tile of prologue) * L2 penalty
//     where the penalty prefers >= 8 splits: the workgroups resident on an XCD are then a block of
//     ~4 token tiles x ~8 splits, which read 12 distinct slab streams through its L2 instead of 33
//     (measured on MI355X: 65536 tokens, H = 4096: 1 split 1.09 PFLOP/s, 8-9 splits 1.4).
struct FusedSchedule {
  int n_ttiles, n_splits, n_wg;
  int tile;              // index of FusedTile
  int n_vunits, unit32;  // vocab units the splits share out, and 32-row blocks per unit
};
// A token tile and how the vocab axis is dealt to the splits with it: in whole tiles of 256 or 224 rows (unit32 = 8 / 7), or in
// 32-row units, of which a workgroup makes tiles of up to 256 rows, all within one unit of each other.
struct FusedTile {
  int tokens, unit32;
};
constexpr int kFusedTiles = 9, kTileGeneric = 8;  // 0 .. 7: the DMA kernel's; 8: the generic kernel's
__host__ __device__ constexpr FusedTile fused_tile(int i) {
  return i == 0 ? FusedTile{256, 8} : i == 1 ? FusedTile{256, 7} : i == 2 ? FusedTile{224, 8} : i == 3 ? FusedTile{224, 7} :
         i == 4 ? FusedTile{192, 1} : i == 5 ? FusedTile{128, 1} : i == 6 ? FusedTile{96, 1} : i == 7 ? FusedTile{64, 1} : FusedTile{128, 8};
}
// What the decomposition depends on beside the number of valid tokens.
struct FusedShape {
  int H, V;
  int slots;       // workgroups that fit the chip at once
  uint32_t tiles;  // bit i: FusedTile i may be taken
  int vunits32, vunits224, vunits256;  // the vocab axis in 32-row units, 224-row and 256-row tiles
  int whole;       // 1: vocab ranges in whole 256-row tiles whatever the token tile
  int named;       // 1: the selector names the token tile, which is then taken for any number of tokens
};
inline FusedShape fused_shape(int64_t H, int64_t V, int slots, uint32_t tiles, bool whole, bool named) {
  return FusedShape{(int)H, (int)V, slots, tiles, (int)((V + 31) / 32), (int)((V + 223) / 224), (int)((V + 255) / 256), whole ? 1 : 0, named ? 1 : 0};
}
__host__ __device__ inline bool fused_one_tile(const FusedShape& sh) { return (sh.tiles & (sh.tiles - 1)) == 0; }
// The tiles below 256 tokens save padding where there are few of them; they are not taken beyond these numbers of valid tokens
// (5074 tokens: 256 a tile 1148 us, 224 1207; the tiles up to 128 tokens are no better than 192 from two of those on).
__host__ __device__ constexpr int fused_tile_most(int i) { return i >= 5 && i < kTileGeneric ? 256 : i >= 2 && i < 5 ? 2560 : 0x7fffffff; }
__host__ __device__ inline bool fused_tile_allowed(const FusedShape& sh, int n_valid, int i) {
  return ((sh.tiles >> i) & 1) && (n_valid <= fused_tile_most(i) || sh.named);
}
// The forms the DMA kernel is built in: two W buffers for 256 tokens, three for 192 .. 256, and the tiles of up to 128 tokens.
__host__ __device__ constexpr bool dma_has_form(int i, bool deep) { return fused_tile(i).tokens <= 128 || deep || fused_tile(i).tokens == 256; }
__host__ __device__ inline int fused_unit32(const FusedShape& sh, int i) { return sh.whole ? 8 : fused_tile(i).unit32; }
__host__ __device__ inline int fused_vunits(const FusedShape& sh, int i) {
  const int u = fused_unit32(sh, i);
  return u == 1 ? sh.vunits32 : u == 7 ? sh.vunits224 : sh.vunits256;
}
__host__ __device__ inline int fused_ttiles(int n_valid, int bt) {
  const int t = (n_valid + bt - 1) / bt;
  return t < 1 ? 1 : t;
}
__host__ __device__ inline int fused_one_round_splits(int n_ttiles, int slots, int n_vtiles) {
  int sp = slots / n_ttiles;
  if (sp > n_vtiles) sp = n_vtiles;  // every split keeps at least one tile's worth of rows
  return sp < 1 ? 1 : sp;
}
// What a batch costs on tile i where one round of workgroups holds it: the longest vocab range bounds the launch.  Fitted to 2300
// timings (V = 32000 .. 151936, H = 768 .. 4096, 33 .. 4096 tokens, every tile): per K slab and vocab tile a constant, the tile's
// MFMA work and the hidden rows' fill, and per vocab tile the fold.  Choosing by it is 0.1 % slower than choosing the measured
// best in the mean, at most 6 % at any of the 290 shapes (32000 x 2560, 640 tokens: 192 a tile 102.5 us, 224 96.9).  Tiles of 224 and
// 192 tokens are only taken for a gain of 3 %: below that the optional outputs and the sharing of W in L2 decide, which are not
// priced (50257 x 2048, 1024 tokens, as five tiles of 224 instead of four of 256: 165 -> 174 us).
// 224-row vocab tiles pay where they shorten the longest range: whole 256-row tiles deal V = 151936 as three tiles to 82
// workgroups and two to the others, 224-row tiles as three to 167 and two to 89, an eighth less for the longest.
// (In floats, quotients of whole numbers with half a unit to spare before the rounding: integer divisions by a lane's own divisor
// are 40 instructions each, and behind a mask one wave prices the tiles between two launches.)
__host__ __device__ inline float fused_tile_cost(const FusedShape& sh, int n_valid, int i) {
  const float tokens = (float)fused_tile(i).tokens, unit32 = (float)fused_unit32(sh, i), units = (float)fused_vunits(sh, i);
  const float vtiles = unit32 == 1.f ? (float)sh.vunits256 : units, nk = (float)(sh.H / kDmaSlab);
  const float ttiles = floorf(((float)n_valid + tokens - 0.5f) / tokens);
  float splits = floorf(((float)sh.slots + 0.5f) / (ttiles < 1.f ? 1.f : ttiles));
  splits = splits > vtiles ? vtiles : splits < 1.f ? 1.f : splits;
  const float longest = floorf((units + splits - 0.5f) / splits);
  const float tiles = unit32 == 1.f ? floorf((longest + 7.f) * 0.125f) : longest, rows = longest * unit32 * 32.f;
  const float cost = tiles * nk * (61.f * 65536.f + 39.f * 256.f * tokens) + rows * (nk * (100.f * tokens + 3.f * 256.f) + 143.f * tokens);
  return i >= 2 && i < 5 ? cost * 1.03f : cost;
}
__host__ __device__ inline int fused_split_round_cost(int n_splits, int n_vunits, int upt) {
  const int longest = (n_vunits + n_splits - 1) / n_splits;  // in units
  const int pen64 = 60 + 32 / (n_splits < 8 ? n_splits : 8);
  return (2 * longest + upt) * pen64;
}
__host__ __device__ inline int64_t fused_split_cost(int n_ttiles, int n_splits, int slots, int n_vunits, int upt) {
  const int rounds = (n_ttiles * n_splits + slots - 1) / slots;
  return (int64_t)rounds * fused_split_round_cost(n_splits, n_vunits, upt) * 64 + n_splits;  // ties go to fewer splits
}
constexpr int kSplitCandidates = 32;
// The schedule but for the number of splits where several rounds are needed; returns whether that is so.
__host__ __device__ inline bool fused_schedule_begin(FusedSchedule& s, int n_valid, const FusedShape& sh, int tile) {
  s.tile = tile;
  s.unit32 = fused_unit32(sh, tile);
  s.n_vunits = fused_vunits(sh, tile);
  s.n_ttiles = fused_ttiles(n_valid, fused_tile(tile).tokens);
  if (s.n_ttiles * 8 > sh.slots) return true;
  s.n_splits = fused_one_round_splits(s.n_ttiles, sh.slots, s.unit32 == 1 ? (s.n_vunits + 7) / 8 : s.n_vunits);
  s.n_wg = s.n_ttiles * s.n_splits;
  return false;
}
inline FusedSchedule fused_schedule_on(int n_valid, const FusedShape& sh, int tile) {  // host
  FusedSchedule s;
  if (fused_schedule_begin(s, n_valid, sh, tile)) {
    const int upt = s.unit32 == 1 ? 8 : 1, n_vtiles = (s.n_vunits + upt - 1) / upt;
    int64_t best = INT64_MAX;
    for (int c = 1; c <= kSplitCandidates && c <= n_vtiles; ++c) {
      const int64_t cost = fused_split_cost(s.n_ttiles, c, sh.slots, s.n_vunits, upt);
      if (cost < best) best = cost;
    }
    s.n_splits = (int)(best & 63);
    s.n_wg = s.n_ttiles * s.n_splits;
  }
  return s;
}
// The most workgroups that any number of valid tokens up to `most` can ask for on one tile.  One round holds at most `slots` of them;
// where several are needed the splits do not follow the number of token tiles in order, and every number is looked at.
inline int fused_most_workgroups(const FusedShape& sh, int tile, int64_t most) {  // host
  const int upt = fused_unit32(sh, tile) == 1 ? 8 : 1, n_vunits = fused_vunits(sh, tile), n_vtiles = (n_vunits + upt - 1) / upt;
  const int64_t ttiles = fused_ttiles((int)most, fused_tile(tile).tokens), one_round = sh.slots / 8;
  const int64_t splits = (ttiles < one_round ? ttiles : one_round) * n_vtiles;
  int best = (int)(splits < sh.slots ? splits : sh.slots);
  if (ttiles <= one_round) return best;
  const int candidates = n_vtiles < kSplitCandidates ? n_vtiles : kSplitCandidates, shift = __builtin_ctz((unsigned)sh.slots);  // slots: a power of two
  int64_t round_cost[kSplitCandidates];
  for (int c = 1; c <= candidates; ++c) round_cost[c - 1] = (int64_t)fused_split_round_cost(c, n_vunits, upt) * 64;
  for (int64_t tt = ttiles; tt > one_round && tt * candidates > best; --tt) {
    int64_t cheapest = INT64_MAX;
    for (int c = 1; c <= candidates; ++c) {
      const int64_t cost = ((tt * c + sh.slots - 1) >> shift) * round_cost[c - 1] + c;
      cheapest = cost < cheapest ? cost : cheapest;
    }
    const int n_wg = (int)(tt * (cheapest & 63));
    best = n_wg > best ? n_wg : best;
  }
  return best;
}
inline FusedSchedule fused_schedule(int n_valid, const FusedShape& sh) {  // host
  float best = INFINITY;
  int tile = __builtin_ctz(sh.tiles);
  for (int i = 0; i < kFusedTiles; ++i) {
    if (!fused_tile_allowed(sh, n_valid, i)) continue;
    const float c = fused_tile_cost(sh, n_valid, i);
    if (c < best) best = c, tile = i;
  }
  return fused_schedule_on(n_valid, sh, tile);
}
enum FusedKind { kGeneric = 0, kDma = 1, kSmall = 2 };
constexpr int kForceDmaWholeTiles = 3;  // selector value: the DMA kernel with vocab ranges cut at whole 256-row tiles
constexpr int kForceDmaTwoWBuffers = 4, kForceDmaThreeWBuffers = 5;  // the DMA kernel, its 256-token tile with two / three W buffers
constexpr int kForceDmaTile = 64;       // 64, 96 .. 256: the DMA kernel with token tiles of that size

// What a plan depends on beside the call.
struct FusedEnv {
  int forced;     // tome_select_fused_kernel, or -1
  int small_wgs;  // workgroups of the streaming kernel, 0 where no device says how many
};

struct FusedPlan {
  FusedKind kind;
  bool deep, deep_lp;                        // kDma only: three W buffers, for the first sweep / one without optional outputs
  bool w_nt;                                 // kDma only: W requested non-temporally (few token tiles: see the kernel's WNT)
  int small_nbt, small_ksteps, small_waves;  // kSmall only
  FusedShape shape;
  FusedSchedule full;  // of all tokens
  bool any_tile;       // kDma: behind a mask the device picks the token tile
  bool any_deep;       // ... with three W buffers for 256 tokens too (sweeps with the entropy; the others always)
  int grid;            // workgroups to launch: behind a mask the most that any number of valid tokens can ask for
};

// Shape rules of the small-batch kernel: <= 64 tokens, K split over 2..8 waves in slices of 256 or 512
// (slices of 128 on twice the waves measured 2 us slower at H = 1024).  At H = 1024 it keeps up to 16 tokens only: since
// the tiled kernel requests W non-temporally where it streams through once, its 64- and 128-token tiles are faster there
// from 17 tokens on (17..64 tokens: 53.3-54.8 against 54.7-59 us; 65..128, which this kernel served with eight token blocks
// on K slices of 128: 61-64 against 67-72 us); at 1280, 1536 and 1792 the two are within 3 % of each other either way, at
// 2048 and above this kernel wins (64 x 2048: 108 against 125 us).
inline bool small_shape(int64_t n_tokens, int64_t H, int64_t V, int& nbt, int& ksteps, int& waves) {
  if (n_tokens > 64 || V < 64) return false;
  if (H == 1024 && n_tokens > 16) return false;
  nbt = n_tokens <= 16 ? 1 : (n_tokens <= 32 ? 2 : 4);
  if (H % 256 == 0 && H / 256 <= 8 && H / 256 >= 2) {
    ksteps = 8;
    waves = (int)(H / 256);
  } else if (H % 512 == 0 && H / 512 <= 8 && H / 512 >= 2 && nbt <= 2) {
    ksteps = 16;
    waves = (int)(H / 512);
  } else {
    return false;
  }
  if (ksteps == 8 && nbt == 2) nbt = 4;  // instantiated token-block counts: 1 and 4 (K 256), 1 and 2 (K 512)
  return waves >= nbt;
}

// Behind a mask of up to this many tokens the device picks the token tile from the valid ones (60 % valid of 200 / 384 / 600 tokens, V =
// 151936, H = 2560: 185 -> 170, 246 -> 197, 331 -> 269 us); the tiles that more tokens fill evenly enough are run by a
// kernel of their own (2100 tokens: 0.975 .. 1.08 with the choice).
constexpr int64_t kAnyTileTokens = 2048;

struct FusedKernel {
  FusedKind kind;
  int nbt, ksteps, waves;  // of the streaming kernel; nbt = 0 for shapes that it does not take
};
inline FusedKernel fused_kernel(const FusedEnv& env, int64_t n_tokens, int64_t H, int64_t V) {
  FusedKernel k{H % kDmaSlab == 0 ? kDma : kGeneric, 0, 0, 0};
  // The streaming kernel runs one workgroup per CU: without a CU count (no device) the tiled kernels serve.
  if (!small_shape(n_tokens, H, V, k.nbt, k.ksteps, k.waves)) k.nbt = 0;
  else if (env.small_wgs >= 2) k.kind = kSmall;
  if (env.forced == kGeneric) k.kind = kGeneric;
  if ((env.forced == kDma || env.forced >= kForceDmaWholeTiles) && H % kDmaSlab == 0) k.kind = kDma;
  return k;
}
// Token tiles that the selector names; 192 and 224 exist with three W buffers only.
inline uint32_t fused_named_tiles(const FusedEnv& env, bool deep_lds) {
  uint32_t named = 0;
  if (env.forced >= kForceDmaTile)
    for (int i = 0; i < kTileGeneric; ++i) named |= (uint32_t)(fused_tile(i).tokens == env.forced && dma_has_form(i, deep_lds)) << i;
  return named;
}
// resident workgroups on 256 CUs: 2 per CU, or 1 for the DMA path's LDS (two 64-token workgroups of 80 KB per CU measured
// slower than one: 288 against 277 us at 64 x 4096)
inline FusedShape fused_shape_on(const FusedEnv& env, FusedKind kind, int64_t H, int64_t V, uint32_t tiles, bool named) {
  if (kind != kDma) return fused_shape(H, V, 512, 1u << kTileGeneric, env.forced == kForceDmaWholeTiles, false);
  return fused_shape(H, V, 256, tiles, env.forced == kForceDmaWholeTiles, named);
}

// One plan a call.  The host's planning of a whole call, the workspace's size asked for twice (by the caller and in the check), us: 200
// tokens 1.8 -> 0.3, 4096 3.5 -> 0.2, 16384 117 -> 2.6, 65536 797 -> 2.9, against walking every number of token tiles of every tile, seven
// times a call.
inline FusedPlan fused_plan(const FusedEnv& env, int64_t n_tokens, int64_t H, int64_t V, bool deep_lds, bool entropy, bool argmax, bool masked) {
  FusedPlan p;
  const int forced = env.forced;
  const FusedKernel kernel = fused_kernel(env, n_tokens, H, V);
  p.kind = kernel.kind;
  p.small_nbt = kernel.nbt;
  p.small_ksteps = kernel.ksteps;
  p.small_waves = kernel.waves;
  // The third W buffer (see the kernel), measured against the two-buffer form in the same runs.  One or two token tiles:
  // 6-13 % faster with any outputs (256 x 1024: 96 -> 87 us, 256 x 4096: 338 -> 297, 512 x 4096: 534 -> 503).  More token
  // tiles, log-probs only: 4096 x 1024 -2.3 %, 8192 x 1024 -1.5 %, 1024 x 4096 -5 %, 4096 x 4096 -1.7 %, 16384 x 2560 -2.6 %,
  // 8192 x 4096 -1.6..+0.2 % over boxes, but 32768 x 4096 +0.7 %, 65536 x 4096 +0.5..2 %.  With the argmax alone it follows
  // (1024 x 4096 -4 %, 4096 x 1024 equal, 8192 x 4096 -1 %); with the entropy the fold of the deeper form spills 29-37
  // registers around every tile change: 1024 x 4096 -3 %, but 4096 x 1024 +2.6 % and 8192 x 4096 +2.3 %.
  p.deep_lp = deep_lds && (H < 4096 || n_tokens <= 8192);
  p.deep = deep_lds && n_tokens <= 1024;
  if (forced == kForceDmaTwoWBuffers) p.deep = p.deep_lp = false;
  if (forced == kForceDmaThreeWBuffers) p.deep = p.deep_lp = deep_lds;
  // Token tiles.  The two-buffer form has 256 tokens only, and a call of two sweeps one schedule for both.
  const uint32_t named = fused_named_tiles(env, deep_lds);
  if (named && !dma_has_form(__builtin_ctz(named), false)) p.deep = p.deep_lp = true;
  const bool any = masked && n_tokens <= kAnyTileTokens && n_tokens > 64;
  const bool all_deep = p.deep_lp && (p.deep || !entropy || any);
  p.shape = fused_shape_on(env, p.kind, H, V, named ? named : all_deep ? 0xffu : 3u, named != 0);
  if (p.kind == kDma) {
    if (forced == kForceDmaTwoWBuffers || forced == kForceDmaThreeWBuffers) p.shape.tiles = 3;
    if (p.shape.whole) p.shape.tiles &= ~((1u << 1) | (1u << 3));  // no vocab tiles of 224 rows
    if (masked && n_tokens > kAnyTileTokens && !named) p.shape.tiles &= 3u;
    // 224 tokens and both optional outputs: the fold's spills outweigh the padding saved (660 of 1100 x 512 1.06 -> 0.98, 1.0 = 256 tokens)
    if (any && n_tokens > 1024 && entropy && argmax && H < 1024 && !named) p.shape.tiles &= ~((1u << 2) | (1u << 3));
  }
  p.full = fused_schedule((int)n_tokens, p.shape);
  const bool w_streams = V * H * 2 >= (int64_t)288 << 20;  // larger than the 256 MB memory-side cache
  // A mask of up to 64 tokens leaves the smallest tile; beyond kAnyTileTokens the 256-token tile serves.
  if (masked && (n_tokens <= 64 || n_tokens > kAnyTileTokens || !all_deep)) p.shape.tiles = 1u << p.full.tile;
  p.any_tile = masked && !fused_one_tile(p.shape);
  // The combined kernel's 256-token body on three W buffers spills 67 registers with the entropy, 87 with the argmax too, most of them around every fold.
  // Up to 1024 tokens, where few token tiles wait for the W stream, it wins all the same; beyond, where W does not stay in the caches and a
  // tile has the K steps to pay for its fold.  To the 256-token kernel without a choice, three | two W buffers, 1280 .. 2048 tokens of which
  // 25 .. 100 % count.  Entropy: H = 256 1.10 .. 1.14 | 1.00, 512 1.10 .. 1.18 | 1.01, 1024 1.01 .. 1.04 | 1.01, 1536 0.95 .. 1.03 | 1.01,
  // 2048 0.93 .. 1.02 | 0.99.  Both: 512 1.19 .. 1.25 | 1.00, 1024 1.04 .. 1.10 | 1.00, 1536 0.97 .. 1.05 | 1.00, 2048 0.94 .. 1.02 | 1.00.  A W of
  // 164 MB, H = 2560: up to 1536 tokens 0.57 .. 1.02 | 0.58 .. 1.01 (pairs 0.80 | 0.84), 1800 and 2048 1.00 .. 1.06 | 0.99 .. 1.01.
  p.any_deep = n_tokens <= 1024 || forced == kForceDmaThreeWBuffers || (H >= (argmax ? 2048 : 1536) && (w_streams || (!argmax && n_tokens <= 1536)));
  p.w_nt = false;
  p.grid = 0;
  if (p.kind == kSmall) return p;  // a grid of its own; the schedule is ignored
  // Non-temporal W (the kernel's WNT): few token tiles, and a W larger than the 256 MB memory-side cache - a smaller one is
  // found there again by the next call as long as it is requested normally (repeated calls, 64 tokens: V = 32000, H = 4096,
  // 262 MB: 48 us against 71 non-temporally; V = 50257, H = 768, 77 MB: 21.0 against 23.3).  Five token tiles already want
  // it kept (50257 x 4096, 1024 tokens as five tiles of 224: 396 us non-temporally, 354 normally).
  p.w_nt = w_streams && p.full.n_ttiles <= (fused_tile(p.full.tile).tokens > 128 ? 4 : 1);
  p.grid = p.full.n_wg;
  if (masked) {  // whatever number of valid tokens and tile the device may end up with
    for (int i = 0; i < kFusedTiles; ++i) {
      if (!((p.shape.tiles >> i) & 1)) continue;
      const int n_wg = fused_most_workgroups(p.shape, i, n_tokens < fused_tile_most(i) || named ? n_tokens : fused_tile_most(i));
      p.grid = n_wg > p.grid ? n_wg : p.grid;
    }
  }
  p.grid = 8 * ((p.grid + 7) / 8);  // fused_locate deals whole rows of 8 workgroup ids
  return p;
}

// Partials that a sweep over up to n_tokens can leave: the same on every device, with and without a mask and for every output, whichever
// plan that makes.
inline size_t partial_bytes(const FusedEnv& env, int64_t n_tokens, int64_t H, int64_t V) {
  const FusedKernel kernel = fused_kernel(env, n_tokens, H, V);
  size_t most = kernel.nbt ? (size_t)64 * 512 : 0;  // the streaming kernel: one partial per (token, workgroup), at most 512
  if (kernel.kind != kSmall) {
    const uint32_t named = fused_named_tiles(env, true);
    const FusedShape shape = fused_shape_on(env, kernel.kind, H, V, named | 3u | (named ? 0u : 0xffu), named != 0);
    for (int i = 0; i < kFusedTiles; ++i) {
      if (!((shape.tiles >> i) & 1)) continue;
      const int64_t tokens = named || n_tokens < fused_tile_most(i) ? n_tokens : fused_tile_most(i);
      const size_t records = (size_t)fused_most_workgroups(shape, i, tokens) * fused_tile(i).tokens * kPartsPerSplit;
      most = records > most ? records : most;
    }
  }
  return most * sizeof(FusedPartial);
}

// Two hidden matrices against one weight are ONE sweep over both where that is a batch of up to this many tokens: W is streamed once
// instead of twice and half-filled token tiles meet.  The sweep computes the entropy for the second matrix too, which at more tokens
// costs what the sharing gives.  Two sweeps / one, us, V = 151936, H = 1024 | 2560: 16 tokens 104 / 56 | 239 / 124, 128: 126 / 90 |
// 314 / 198, 512: 281 / 277 | 645 / 611, 768: 400 / 418 | 921 / 980; behind a mask that leaves 56 %, 128: 121 / 86 | 285 / 185, 512:
// 170 / 140 | 380 / 301, 768: 236 / 222 | 538 / 471, 1024: 369 / 383 | 868 / 845.  All tokens valid behind a mask, 640: 406 / 358 | 956 / 772,
// 704 .. 768: 412 / 416 | 946 / 940 (H = 512: 221 / 219, 2048: 754 / 767), on the combined kernel's two W buffers (FusedPlan::any_deep; on three
// 6 % more than two sweeps at H = 512, 4 at 1024).
inline bool joint_fits(int64_t n_tokens, int64_t H, bool masked) { return n_tokens <= (masked ? 768 : 512) && H % kDmaSlab == 0; }

// Layout of the workspace: [n_valid + schedule: 256 B][row_index: n_tokens int32, 256-aligned][partials of the first sweep, of the
// second][normalised hidden rows, per matrix, only with a norm weight].  Offsets in bytes.
constexpr size_t kFusedIndexOffset = 256;
struct FusedLayout {
  size_t partials, partials_second, normed, normed_second, total;
};
inline size_t fused_align(size_t n) { return (n + 255) & ~(size_t)255; }
inline FusedLayout fused_layout(const FusedEnv& env, int64_t n_tokens, int64_t H, int64_t V, int n_sweeps, int n_normed) {
  FusedLayout l;
  const size_t each = partial_bytes(env, n_tokens, H, V);
  const size_t joint = n_sweeps == 2 && joint_fits(n_tokens, H, true) ? partial_bytes(env, 2 * n_tokens, H, V) : 0;
  const size_t normed = fused_align((size_t)n_tokens * H * 2);
  l.partials = kFusedIndexOffset + fused_align((size_t)n_tokens * 4);
  l.partials_second = l.partials + each;
  l.normed = l.partials + (each * n_sweeps > joint ? each * n_sweeps : joint);
  l.normed_second = l.normed + normed;
  l.total = fused_align(l.normed + normed * n_normed);
  return l;
}

}  // namespace tome
