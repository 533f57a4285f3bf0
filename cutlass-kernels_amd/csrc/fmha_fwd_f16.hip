// FMHA forward, fp16 operands: tile shapes and dispatch.  The kernels are in fmha_fwd_kernel.h (32x32 MFMAs) and
// fmha_fwd_kernel16.h (16x16x32 MFMAs).
#include "fmha_fwd_kernel16p.h"
#include "fmha_fwd_kernel_ks.h"

namespace cfk {
namespace {

constexpr int kCus = 256;

// <head dim, keys per tile, waves, waves per SIMD, e4m3 Q/K, e4m3 P/V, V transposed, score tap, tiles per barrier,
//  K fragments read ahead of the barrier, 16x16x32 build>.  4 waves = 128 query rows (two workgroups share a CU),
// 8 waves = 256 rows (one workgroup per CU, half the K/V traffic per query row).  Two waves per SIMD, except head dim
// 64, whose 128-row tile fits three (the faster choice there).  Head dim 256 (one wave per SIMD) is built in
// fmha_fwd_f16_d256.hip, under a machine-scheduler strategy of its own; only its score-tap build is here.
using C64_128x64 = FmhaCfg<64, 64, 4, 3, false, false>;
using C64_256x64 = FmhaCfg<64, 64, 8, 2, false, false>;
using C64_128x128 = FmhaCfg<64, 64, 4, 2, false, false, false, false, 2>;
using C64_256x128 = FmhaCfg<64, 64, 8, 2, false, false, false, false, 2>;
using C128_128x64 = FmhaCfg<128, 64, 4, 2, false, false>;
using C128_256x64 = FmhaCfg<128, 64, 8, 2, false, false>;
using C128_256x64P = FmhaCfg<128, 64, 8, 2, false, false, false, false, 1, 4>;  // key length a multiple of 256
using C128_128x128 = FmhaCfg<128, 64, 4, 2, false, false, false, false, 2>;
using C128_256x128 = FmhaCfg<128, 64, 8, 2, false, false, false, false, 2>;
// The builds on 16x16x32 MFMAs, the automatic choice for big problems at head dims 64 and 128 (+6..10 % on N(0,1)
// data).  Head dim 128: two key tiles per barrier when the key length allows (+1..2 %: 1145-1157 against 1134
// TFLOP/s on B=8 H=16 S=2048).  Not built: the K fragment prefetch (registers spill), at head dim 64 256 rows (880
// against 919 TFLOP/s for 128 rows) and two tiles per barrier (950 against 1030: the LDS then holds two workgroups
// per CU, not three), head dim 256 (929 against 932 for the 32x32 build).
using N64_128x64 = FmhaCfg<64, 64, 4, 3, false, false, false, false, 1, 0, true>;
using N128_128x64 = FmhaCfg<128, 64, 4, 2, false, false, false, false, 1, 0, true>;
using N128_256x64 = FmhaCfg<128, 64, 8, 2, false, false, false, false, 1, 0, true>;
using N128_256x128 = FmhaCfg<128, 64, 8, 2, false, false, false, false, 2, 0, true>;
using N128_128x128 = FmhaCfg<128, 64, 4, 2, false, false, false, false, 2, 0, true>;
// ... and with the hand-scheduled main loop (key length a multiple of 256, at least 512)
using A128_256x128 = FmhaCfg<128, 64, 8, 2, false, false, false, false, 2, 0, true, true>;
using A64_256x128 = FmhaCfg<64, 64, 8, 2, false, false, false, false, 2, 0, true, true>;
using A128_128x128 = FmhaCfg<128, 64, 4, 1, false, false, false, false, 2, 0, true, true>;   // the same loops, 4 waves, one per SIMD
using A64_128x128 = FmhaCfg<64, 64, 4, 1, false, false, false, false, 2, 0, true, true>;

// ... and for small grids: 32 query rows per workgroup, the eight waves split the keys (fmha_fwd_kernel_ks.h)
using K64_32x64 = KsCfg<64, 8>;
using K128_32x64 = KsCfg<128, 8>;

// builds that also write the score tap (debug): 128-row tile only
using C64Tap = FmhaCfg<64, 64, 4, 2, false, false, false, true>;
using C128Tap = FmhaCfg<128, 64, 4, 2, false, false, false, true>;
using C256Tap = FmhaCfg<256, 32, 4, 1, false, false, false, true>;

using All64 = CfgList<C64_128x64, N64_128x64, C64_256x64, C64_128x128, C64_256x128, A64_256x128, A64_128x128, K64_32x64>;
using All128 = CfgList<C128_128x64, N128_128x64, C128_256x64P, C128_256x64, N128_256x64, C128_128x128, C128_256x128, N128_128x128, A128_256x128, A128_128x128, N128_256x128, K128_32x64>;

template <class F>
bool dispatch(int head_dim, int sq, int skv, int bh, bool tap_s, F &&f) {
  if (tap_s) {
    switch (head_dim) {
      case 64: f(C64Tap{}); return true;
      case 128: f(C128Tap{}); return true;
      case 256: f(C256Tap{}); return true;
      default: return false;
    }
  }
  switch (head_dim) {
    case 64: select_tile<All64, CfgList<K64_32x64, A64_256x128, A64_128x128, N64_128x64, C64_128x64>, C64_128x64>(sq, skv, bh, f); return true;
    case 128: select_tile<All128, CfgList<K128_32x64, A128_256x128, A128_128x128, N128_256x128, N128_256x64, N128_128x64, C128_256x64P, C128_256x64, C128_128x64>, C128_128x64>(sq, skv, bh, f); return true;
    default: return false;
  }
}

}  // namespace

bool plan_fmha_f16(int head_dim, int sq, int skv, int bh, bool tap_s, FmhaPlan *p) {
  if (head_dim == 256 && !tap_s) { plan_fmha_f16_d256(sq, skv, bh, p); return true; }
  return dispatch(head_dim, sq, skv, bh, tap_s, [&](auto cfg) { fill_fmha_plan<decltype(cfg)>(sq, skv, bh, p); });
}

hipError_t launch_fmha_f16(const FmhaArgs &a, int head_dim, hipStream_t s) {
  if (head_dim == 256 && !a.s_tap) return launch_fmha_f16_d256(a, s);
  if (a.n_split > 1 && a.split_bm == 256) return head_dim == 64 ? launch_fmha_split<A64_256x128>(a, s) : launch_fmha_split<A128_256x128>(a, s);
  if (a.n_split > 1 && a.split_bm == 128) return head_dim == 64 ? launch_fmha_split<A64_128x128>(a, s) : launch_fmha_split<A128_128x128>(a, s);
  hipError_t e = hipErrorInvalidValue;
  dispatch(head_dim, a.Sq, a.Skv, a.B * a.H, a.s_tap != nullptr, [&](auto cfg) { e = launch_fmha_cfg<decltype(cfg)>(a, s); });
  return e;
}

// The hand-scheduled builds run one workgroup per CU in rounds of 256 units of work.  The whole rounds take items as they are; the
// items left over -- all of them, where there are fewer than CUs -- are cut into n units along the keys, at least two groups
// of four key tiles each, as many as still make one round.  n, and the rows per item, are what the times below add up to least
// for; the call is cut if that is less than its time otherwise by a twentieth.  Times, us, by head dim: a key tile of a unit while
// all CUs work and while at most half do (the clock is higher then), a unit's start and end, tiles behind the last group of four
// as two and a half, the merge 5 and 4 TB/s for the partial results.  That is short of what a cut costs where the whole call is
// short, so a call stays whole unless a second sum says less time as well: with 5 us for a cut behind whole rounds, else 6 for one of
// 128-row items, 13.5 at head dim 256, and of 256-row items 10.5, or 12.5 where a head has more than two of them.  (1442 drawn calls that
// the first sum alone would cut, each side 0.1 s at a time in turn, whole -> cut: head dim 64 52 of 1102 slower by more than a hundredth, up
// to 1.37 -- 25 heads of 512 rows, 2048 keys 19.0 -> 26.0 us --, head dim 128 1 of 168, head dim 256 8 of 172, up to 1.06.  With both 9 of
// 1041, 0 of 167 and 3 of 156; of the 78 calls that the second sum keeps whole 14 would gain more than three hundredths cut.)  Measured, N(0,1), us before -> after: D=128, 36 heads of 256
// rows, 10176 keys 127.6 -> 65.5 (3 units); 16 heads of 1024 rows, 8192 keys 99.2 -> 71.0; 20 heads of 6528 rows, 6144 keys (520
// items of 256 rows) 399 -> 334; D=64, 16 heads of 4512 rows, 6976 keys 174.0 -> 132.4; 160 heads of 1216 rows, 4864 keys 259 -> 234;
// D=256, 36 heads of 256 rows, 8192 keys 225.8 -> 114.4; 15 heads of 2976 rows, 4096 keys 202.1 -> 181.7.  No gain, and the rule
// keeps off: 256 items of 128 rows, D=128, 4096 keys 64.0 / 70.5.
// (Only calls that run a hand-scheduled build anyway: its Q is rounded once more, rms error of O 3.6e-4 of its size against
// 2.9e-4 of the compiler-scheduled builds.)
bool plan_fmha_f16_split(int head_dim, int sq, int skv, int bh, const FmhaPlan &plan, KeySplit *out) {
  const TileWish w = tile_wish();
  const int bn = head_dim == 256 ? 32 : 64, tiles = skv / bn, groups = tiles / 4, left = tiles % 4;
  if (!plan.hand || w.bm || w.bn || groups < 4) return false;
  struct Build { int bm; float full, low, fixed; };
  const Build b256 = head_dim == 64 ? Build{256, 0.885f, 0.62f, 3.f} : Build{256, 1.66f, 1.05f, 5.f};
  const Build b128 = head_dim == 64 ? Build{128, 0.48f, 0.45f, 4.f} : head_dim == 128 ? Build{128, 0.95f, 0.74f, 4.f} : Build{128, 0.884f, 0.67f, 4.f};
  const auto round_us = [&](const Build &b, int units, int loop_tiles, int tail) {
    const float busy = 2.f * units / kCus - 1.f, tile = b.low + (b.full - b.low) * (busy > 0.f ? busy : 0.f);
    return units ? b.fixed + (loop_tiles + 2.5f * tail) * tile : 0.f;
  };
  const auto rounds_us = [&](const Build &b, int items) {
    return items / kCus * round_us(b, kCus, 4 * groups, left) + round_us(b, items % kCus, 4 * groups, left);
  };
  const float call_us = rounds_us(plan.block_m == 256 ? b256 : b128, plan.grid);
  float best_us = 0.95f * call_us;
  KeySplit best{};
  bool pays = false;
  for (const Build &b : {b256, b128}) {
    if (head_dim == 256 && b.bm == 256) continue;
    const int items = bh * ((sq + b.bm - 1) / b.bm), from = items / kCus * kCus, cut = items - from;
    const float whole_us = rounds_us(b, from);
    for (int n = 2; n * cut <= kCus && 2 * n <= groups && cut; ++n) {
      const float units_us = whole_us + round_us(b, n * cut, 4 * ((groups + n - 1) / n), left);
      const float us = units_us + 5.f + (float)n * cut * b.bm * head_dim * 4.f / 4e6f;
      if (us >= best_us) continue;
      const float cut_us = from ? 5.f : head_dim == 256 ? 13.5f : b.bm == 128 ? 6.f : sq <= 512 ? 10.5f : 12.5f;
      best_us = us, best = KeySplit{n, b.bm, from}, pays = units_us + cut_us < call_us;
    }
  }
  if (pays) *out = best;
  return pays;
}

hipError_t prepare_fmha_f16() {
  hipError_t e = prepare_all(All64{});
  if (e == hipSuccess) e = prepare_all(All128{});
  if (e == hipSuccess) e = prepare_fmha_f16_d256();
  const hipError_t split[] = {prepare_fmha_split<A64_256x128>(), prepare_fmha_split<A64_128x128>(), prepare_fmha_split<A128_256x128>(), prepare_fmha_split<A128_128x128>()};
  for (hipError_t x : split)
    if (e == hipSuccess) e = x;
  if (e == hipSuccess) e = prepare_all(CfgList<C64Tap, C128Tap, C256Tap>{});
  return e;
}

}  // namespace cfk
