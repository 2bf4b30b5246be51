// Checks the planning of fused lm_head calls (tome_amd/csrc/fused_plan.hpp) over random calls, without a GPU: whatever tile and number
// of valid tokens a call may end up with, a kernel form exists for it, the grid holds its workgroups, the workspace its partials, and
// every vocab range is one that the kernels can cut into tiles.  Prints the first faults and their number; `time N ...`: what one
// call of N tokens plans on the host, in us.
#include "fused_plan.hpp"
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

using namespace tome;

static int faults = 0;
static void fault(const char* what, const FusedEnv& env, int64_t n, int64_t H, int64_t V, bool ent, bool masked, bool deep, int64_t n_valid, int tile) {
  if (++faults <= 20)
    std::printf("%s: selector %d, %lld tokens, H %lld, V %lld, entropy %d, masked %d, deep %d, valid %lld, tile %d\n", what, env.forced,
                (long long)n, (long long)H, (long long)V, ent, masked, deep, (long long)n_valid, tile);
}

static void check_call(const FusedEnv& env, int64_t n, int64_t H, int64_t V, bool ent, bool amax, bool masked, bool deep) {
  const FusedPlan p = fused_plan(env, n, H, V, deep, ent, amax, masked);
  const size_t records = partial_bytes(env, n, H, V) / sizeof(FusedPartial);
#define FAULT(what, n_valid, tile) fault(what, env, n, H, V, ent, masked, deep, n_valid, tile)
  if (p.kind == kSmall) {
    if (n > 64 || (size_t)64 * 512 > records) FAULT("streaming kernel", n, -1);
    return;
  }
  if (p.kind == kDma && H % kDmaSlab != 0) FAULT("ragged H on the DMA kernel", n, -1);
  const int host_tile = p.full.tile;
  if (fused_schedule((int)n, p.shape).tile != host_tile) FAULT("the plan's schedule", n, host_tile);
  const bool tile_holds = env.forced <= 128 || env.forced == 256 || deep;  // 192 and 224 need the third W buffer
  if (p.kind == kDma && env.forced >= 64 && tile_holds && fused_tile(host_tile).tokens != env.forced) FAULT("selected token tile not taken", n, host_tile);
  auto on_tile = [&](int64_t n_valid, int tile) {
    if (!((p.shape.tiles >> tile) & 1)) FAULT("tile outside the plan", n_valid, tile);
    if (p.kind == kDma && !p.any_tile) {  // launched by tile; a second sweep is one without the entropy
      if (!dma_has_form(tile, ent ? p.deep : p.deep_lp) || !dma_has_form(tile, p.deep_lp)) FAULT("no kernel form", n_valid, tile);
    }
    if (p.any_tile && ent && !p.any_deep && p.w_nt) FAULT("non-temporal W without the third W buffer", n_valid, tile);
    if (p.any_tile && env.forced == kForceDmaThreeWBuffers && !p.any_deep) FAULT("selected third W buffer not taken", n_valid, tile);
    if (p.any_tile && !deep) FAULT("device-chosen tile without the third W buffer", n_valid, tile);
    const FusedSchedule s = fused_schedule_on((int)n_valid, p.shape, tile);
    if (s.tile != tile || s.n_wg != s.n_ttiles * s.n_splits || s.n_splits < 1 || (int64_t)s.n_ttiles * fused_tile(tile).tokens < n_valid) FAULT("schedule", n_valid, tile);
    if (8 * ((s.n_wg + 7) / 8) > p.grid) FAULT("grid too small", n_valid, tile);
    if ((size_t)n_valid * s.n_splits * kPartsPerSplit > records) FAULT("workspace too small", n_valid, tile);
    const bool mixed = p.kind == kDma && fused_tile(tile).tokens <= 192;
    const int longest_tiles = ((s.n_vunits + s.n_splits - 1) / s.n_splits * s.unit32 + 7) >> 3;
    int64_t end = 0;
    for (int k = 0; k < s.n_splits; ++k) {
      const int64_t u0 = (int64_t)k * s.n_vunits / s.n_splits, u1 = (int64_t)(k + 1) * s.n_vunits / s.n_splits;
      const int64_t blocks = (u1 - u0) * s.unit32;
      const int64_t height = mixed ? blocks / longest_tiles : s.unit32;
      if (u0 != end || u1 <= u0 || (mixed && (height < 1 || height + (blocks > height * longest_tiles) > 8))) FAULT("vocab range", n_valid, tile);
      end = u1;
    }
    if (end != s.n_vunits || (int64_t)s.n_vunits * s.unit32 * 32 < V) FAULT("vocabulary not covered", n_valid, tile);
  };
  if (!masked) return on_tile(n, host_tile);
  for (int64_t n_valid = 1; n_valid <= n; n_valid = n_valid == n ? n + 1 : std::min(n, n_valid + 32 * (1 + n_valid / 4096))) {
    bool any = false;
    for (int i = 0; i < kFusedTiles; ++i)
      if (fused_tile_allowed(p.shape, (int)n_valid, i)) any = true, on_tile(n_valid, i);
    if (!any) FAULT("no tile", n_valid, -1);
    if (!p.any_tile && fused_schedule((int)n_valid, p.shape).tile != host_tile) FAULT("device and host on different tiles", n_valid, host_tile);
  }
}

// The workspace's size (the caller's, and the check's), the choice of the kernel, the plan.
static size_t plan_one_call(const FusedEnv& env, int64_t n, int64_t H, int64_t V) {
  size_t sum = fused_layout(env, n, H, V, 1, 0).total;
  sum += fused_kernel(env, n, H, V).kind + fused_layout(env, n, H, V, 1, 0).normed;
  const FusedPlan p = fused_plan(env, n, H, V, true, false, false, false);
  return sum + p.grid + p.full.n_wg;
}

int main(int argc, char** argv) {
  if (argc > 1 && !std::strcmp(argv[1], "time")) {  // one call's planning, best of several runs, us
    for (int i = 2; i < argc; ++i) {
      const int64_t n = std::atoll(argv[i]);
      double best = 1e9;
      size_t sink = 0;
      for (int r = 0; r < 200; ++r) {
        const auto t0 = std::chrono::steady_clock::now();
        for (int k = 0; k < 4; ++k) sink += plan_one_call(FusedEnv{-1, 256}, n, 1024, 151936 + (int)(sink & 1));
        best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 4);
      }
      std::printf("%lld %.3f\n", (long long)n, sink ? best : 0.0);
    }
    return 0;
  }
  std::mt19937_64 rng(argc > 1 ? std::strtoull(argv[1], nullptr, 10) : 1);
  auto spread = [&](double lo, double hi) { return std::exp(std::uniform_real_distribution<double>(std::log(lo), std::log(hi))(rng)); };
  const int selectors[] = {-1, -1, -1, -1, 0, 1, 3, 4, 5, 64, 96, 128, 192, 224, 256};
  int calls = 0;
  for (; calls < 6000; ++calls) {
    const FusedEnv env{selectors[rng() % 15], rng() % 8 ? 256 : 0};
    const int64_t n = (int64_t)spread(1, rng() % 4 ? 4000 : 70000), H = rng() % 8 ? 64 * (1 + (int64_t)(spread(1, 100))) : 8 * (1 + rng() % 500);
    const int64_t V = (int64_t)spread(16, 260000);
    check_call(env, n, H, V, rng() & 1, rng() & 1, rng() & 1, rng() % 8 != 0);
  }
  for (const int selector : selectors)  // sizes at the rules' own lines
    for (const int64_t n : {1, 64, 65, 256, 257, 1024, 1025, 1452, 2048, 2049, 2560, 2561, 8192, 8193, 15580})
      for (const int64_t V : {223, 1068, 32000, 151936})
        for (int bits = 0; bits < 24; ++bits, ++calls)
          check_call(FusedEnv{selector, 256}, n, bits >= 16 ? 4864 : bits >= 8 ? 1024 : 512, V, bits & 1, bits & 2, bits & 4, true);
  std::printf("%d calls, %d faults\n", calls, faults);
  return faults != 0;
}
