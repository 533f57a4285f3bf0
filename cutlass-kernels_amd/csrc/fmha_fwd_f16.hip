// FMHA forward, fp16 operands: tile shapes and dispatch.  The kernels are in fmha_fwd_kernel.h (32x32 MFMAs) and
// fmha_fwd_kernel16.h (16x16x32 MFMAs).
#include "fmha_fwd_kernel16p.h"
#include "fmha_fwd_kernel_ks.h"
#include "fmha_split_choice.h"

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
// ... and with the hand-scheduled main loop (any key length from 512 on)
using A128_256x128 = FmhaCfg<128, 64, 8, 2, false, false, false, false, 2, 0, true, true>;
using A64_256x128 = FmhaCfg<64, 64, 8, 2, false, false, false, false, 2, 0, true, true>;
using A128_128x128 = FmhaCfg<128, 64, 4, 1, false, false, false, false, 2, 0, true, true>;   // the same loops, 4 waves, one per SIMD
using A64_128x128 = FmhaCfg<64, 64, 4, 1, false, false, false, false, 2, 0, true, true>;
// ... and a multiply-add per score
using F128_256x128 = FmaCfg<A128_256x128>;
using F64_256x128 = FmaCfg<A64_256x128>;
using F128_128x128 = FmaCfg<A128_128x128>;
using F64_128x128 = FmaCfg<A64_128x128>;

// ... and for small grids: 32 query rows per workgroup, the eight waves split the keys (fmha_fwd_kernel_ks.h)
using K64_32x64 = KsCfg<64, 8>;
using K128_32x64 = KsCfg<128, 8>;

// builds that also write the score tap (debug): 128-row tile only
using C64Tap = FmhaCfg<64, 64, 4, 2, false, false, false, true>;
using C128Tap = FmhaCfg<128, 64, 4, 2, false, false, false, true>;
using C256Tap = FmhaCfg<256, 32, 4, 1, false, false, false, true>;

using All64 = CfgList<C64_128x64, N64_128x64, C64_256x64, C64_128x128, C64_256x128, A64_256x128, A64_128x128, F64_256x128, F64_128x128, K64_32x64>;
using All128 = CfgList<C128_128x64, N128_128x64, C128_256x64P, C128_256x64, N128_256x64, C128_128x128, C128_256x128, N128_128x128, A128_256x128, A128_128x128, F128_256x128, F128_128x128, N128_256x128, K128_32x64>;

// ---- What a call of head dim 64 or 128 takes that no rule above gives a hand-scheduled build with the scale folded into Q: a
// compiler-scheduled build or a FmaCfg one, whichever the sums below make less time of.  They follow how the rounds of workgroups fill:
// a compiler-scheduled build has places for three (head dim 64) or two workgroups on a CU and deals them out one by one, a
// hand-scheduled one walks rounds of 256 items, in which a tile takes `low` us while at most half of the CUs work and more the more do,
// up to `full`; either may instead be bound by reading K and V.  Fitted to 299 drawn calls of at least 512 keys, N(0,1) (rms of
// the error: 3 to 4 % at head dim 64, 5 to 7 % at 128; where one sum is off, the other mostly is by as much).  The choice takes 0.947 of the
// time of the compiler-scheduled builds (geometric mean; the best choice for each 0.940); kinds of call on which it was wrong: fma_rows.  us, compiler-scheduled -> chosen:
// head dim 64, 80 heads of 1696 rows, 3520 keys 144.9 -> 135.1; 161 of 192, 6400 keys 113.4 -> 94.5; head dim 128, 108 of 2560, 1856 keys
// 277.5 -> 243.3; 168 of 704, 1664 keys 125.2 -> 107.8; 36 of 2016, 3200 keys 146.4 -> 117.3 (last round cut along the keys).
struct Call {
  int head_dim, sq, skv, bh;
  int items(int bm) const { return bh * ((sq + bm - 1) / bm); }
  int tiles() const { return skv / 64; }
  float mbytes() const { return 4e-6f * head_dim * bh * ((float)sq + skv); }
};
struct HandTimes {
  int bm;
  float full, low, first, round;   // us: a tile; what a call and what each of its rounds takes besides
};
HandTimes fma_times(int head_dim, int bm) {
  if (head_dim == 64) return bm == 256 ? HandTimes{256, 0.942f, 0.753f, 2.f, 2.9f} : HandTimes{128, 0.572f, 0.527f, 2.3f, 1.9f};
  return bm == 256 ? HandTimes{256, 1.709f, 1.135f, 4.6f, 3.5f} : HandTimes{128, 0.973f, 0.815f, 3.1f, 3.5f};
}
float round_us(const HandTimes &h, int units, int tiles) {
  const float busy = 2.f * units / kCus - 1.f;
  return units ? h.round + tiles * (h.low + (h.full - h.low) * (busy > 0.f ? busy : 0.f)) : 0.f;
}
float fma_issue_us(const Call &c, const HandTimes &h) {
  const int items = c.items(h.bm);
  return h.first + items / kCus * round_us(h, kCus, c.tiles()) + round_us(h, items % kCus, c.tiles());
}
float fma_us(const Call &c, const HandTimes &h) { return either(fma_issue_us(c, h), c.mbytes() / 3.4f); }
// the same with the items from `from` on cut into n units along the keys, and the merge of their results
float fma_cut_us(const Call &c, const HandTimes &h, int n, int from) {
  const int units = n * (c.items(h.bm) - from);
  const float part = 4e-6f * units * h.bm * c.head_dim;   // MB
  const float us = h.first + from / kCus * round_us(h, kCus, c.tiles()) + round_us(h, units, (c.tiles() + n - 1) / n);
  return either(us, (c.mbytes() + part) / 3.4f) + 3.f + part / 4.f;
}
float compiled_us(const Call &c, bool m16) {
  const float x = (float)c.items(128) / kCus;
  const float t = c.head_dim == 64 ? (x <= 1 ? 0.625f + 0.006f * x : x <= 2 ? 0.98f + 0.206f * (x - 1) : x <= 3 ? 1.482f + 0.448f * (x - 2) : 0.327f + 0.562f * x)
                                   : (x <= 1 ? 0.935f + 0.205f * x : x <= 2 ? 1.571f + 0.744f * (x - 1) : 0.545f + 0.928f * x);
  const float per_tile = !m16 ? t : t * (c.head_dim == 64 ? 0.933f : 0.972f);
  return c.head_dim == 64 ? 3.33f * ceilf(x / 3) - 0.2f + either(c.tiles() * per_tile, c.mbytes() / 3.42f)
                          : 6.57f * ceilf(x / 2) - 2.73f + either(c.tiles() * per_tile, c.mbytes() / 3.93f);
}
// rows of the FmaCfg build to take instead of a compiler-scheduled one, 0: none; *us: the least of the sums, *rows_of_sum: whose it is
int fma_rows(const Call &c, bool m16, float *us, int *rows_of_sum) {
  int bm = *rows_of_sum = 0;
  *us = compiled_us(c, m16);
  float best = 0.97f * *us;
  for (int rows : {256, 128}) {
    if (rows == 128 && c.skv < 1024) continue;   // (0.98 to 1.06 of the time there)
    // (a last 256-row tile that is filled to half or less in every other tile -- 320, 352, 384 rows -- gained nothing: 0.99 to 1.08)
    if (rows == 256 && 2 * c.items(128) <= 3 * c.items(256)) continue;
    const HandTimes h = fma_times(c.head_dim, rows);
    const float t = fma_us(c, h);
    if (t >= best) continue;
    best = *us = t, *rows_of_sum = rows;
    // Where the sum says less and the calls took more (540 drawn calls, time relative to the compiler-scheduled build):
    // 128 rows: more than a round of items 0.99 to 1.37 (300 heads of 128 rows, 1152 keys, head dim 64 24.0 -> 32.8 us; 96 heads of 608, 2048 keys, head dim 128
    // 72.8 -> 75.3); a round or less: head dim 128 below 1216 keys 0.99 to 1.02; head dim 64 below 1600 keys and few rows a head, so that reading K and V
    // takes as long as the multiplies, 0.98 to 1.16 (222 heads of 128 rows, 1216 keys 16.1 -> 18.6).  The others 0.92 to 1.00.
    // 256 rows: head dim 128, up to half a round behind one whole round, below 896 keys 0.99 to 1.13 (336 heads of 224 rows, 768 keys 51.7 -> 57.1; 32 of 2912,
    // 704 keys 39.8 -> 41.6), with more 0.93 to 1.01; head dim 64, a round or less below 768 keys, reading K and V, 0.96 to 1.05.  The others 0.73 to 1.02.
    const int items = c.items(rows);
    const bool reading = c.mbytes() / 3.4f > 0.8f * fma_issue_us(c, h);   // (or nearly as long)
    const bool slower = rows == 128           ? items > kCus || (c.head_dim == 128 ? c.skv < 1216 : reading && c.skv < 1600)
                        : c.head_dim == 128 ? items > kCus && 2 * items <= 3 * kCus && c.skv < 896
                                            : items <= kCus && reading && c.skv < 768;
    bm = slower ? 0 : rows;
  }
  return bm;
}

template <class Auto, class Fallback, class F256, class F128, class F>
void select_f16(int head_dim, int sq, int skv, int bh, F &&f) {
  tile_by_rule<Auto, Fallback>(sq, skv, bh, [&](auto cfg) {
    using C = decltype(cfg);
    if constexpr (!C::KSPLIT && !C::ASM) {
      // (time relative to the compiler-scheduled build, drawn calls with what fma_rows leaves out left out: head dim 128, 512 and 576 keys 0.87 to 1.04; 640 keys 0.90 to
      // 0.99, but with at least 512 whole 256-row tiles, which fmha_fwd_kernel16 takes otherwise, 0.90 to 1.03; from 704 on 0.78 to 0.97 there.  Head dim 64,
      // as many tiles, up to 1216 keys 0.93 to 1.00, 0.977 in the geometric mean: not worth a time that depends on the data)
      const bool big = problem_size(sq, bh) == 2;
      if (hand_loops_allowed() && fits<F256>(sq, skv) && skv >= (head_dim == 128 ? big ? 704 : 640 : big ? 1280 : 512)) {
        float us;
        int sum;
        const int rows = fma_rows(Call{head_dim, sq, skv, bh}, C::M16, &us, &sum);
        if (rows == 256) return f(F256{});
        if (rows == 128) return f(F128{});
      }
    }
    f(cfg);
  });
}

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
    case 64:
      if (!tile_by_wish<All64>(sq, skv, bh, f))
        select_f16<CfgList<K64_32x64, A64_256x128, A64_128x128, N64_128x64, C64_128x64>, C64_128x64, F64_256x128, F64_128x128>(64, sq, skv, bh, f);
      return true;
    case 128:
      if (!tile_by_wish<All128>(sq, skv, bh, f))
        select_f16<CfgList<K128_32x64, A128_256x128, A128_128x128, N128_256x128, N128_256x64, N128_128x64, C128_256x64P, C128_256x64, C128_128x64>, C128_128x64,
                   F128_256x128, F128_128x128>(128, sq, skv, bh, f);
      return true;
    default: return false;
  }
}

template <class A256, class A128>
hipError_t launch_split(const FmhaArgs &a, bool fma, hipStream_t s) {
  if (fma) return a.split_bm == 256 ? launch_fmha_split<FmaCfg<A256>>(a, s) : launch_fmha_split<FmaCfg<A128>>(a, s);
  return a.split_bm == 256 ? launch_fmha_split<A256>(a, s) : launch_fmha_split<A128>(a, s);
}

}  // namespace

bool plan_fmha_f16(int head_dim, int sq, int skv, int bh, bool tap_s, FmhaPlan *p) {
  if (head_dim == 256 && !tap_s) { plan_fmha_f16_d256(sq, skv, bh, p); return true; }
  return dispatch(head_dim, sq, skv, bh, tap_s, [&](auto cfg) { fill_fmha_plan<decltype(cfg)>(sq, skv, bh, p); });
}

hipError_t launch_fmha_f16(const FmhaArgs &a, int head_dim, hipStream_t s) {
  if (head_dim == 256 && !a.s_tap) return launch_fmha_f16_d256(a, s);
  if (a.n_split > 1 && a.split_bm != 32) {
    FmhaPlan plan{};   // (the scale is folded into Q in calls that have it so without a workspace)
    plan_fmha_f16(head_dim, a.Sq, a.Skv, a.B * a.H, false, &plan);
    const bool fma = !plan.hand || plan.fma;
    return head_dim == 64 ? launch_split<A64_256x128, A64_128x128>(a, fma, s) : launch_split<A128_256x128, A128_128x128>(a, fma, s);
  }
  hipError_t e = hipErrorInvalidValue;
  dispatch(head_dim, a.Sq, a.Skv, a.B * a.H, a.s_tap != nullptr, [&](auto cfg) { e = launch_fmha_cfg<decltype(cfg)>(a, s); });
  return e;
}

// The hand-scheduled builds run one workgroup per CU in rounds of 256 units of work.  The whole rounds take items as they are; the
// items left over -- all of them, where there are fewer than CUs -- are cut into n units along the keys, at least eight key
// tiles each, as many as still make one round.  n, and the rows per item, are what the times below add up to least
// for; the call is cut if that is less than its time otherwise by a twentieth.  Times, us, by head dim: a key tile of a unit while
// all CUs work and while at most half do (the clock is higher then), a unit's start and end, the merge 5 and 4 TB/s for the partial
// results.  That is short of what a cut costs where the whole call is
// short, so a call stays whole unless a second sum says less time as well: with 5 us for a cut behind whole rounds, else 6 for one of
// 128-row items, 13.5 at head dim 256, and of 256-row items 10.5, or 12.5 where a head has more than two of them.  (1442 drawn calls that
// the first sum alone would cut, each side 0.1 s at a time in turn, whole -> cut: head dim 64 52 of 1102 slower by more than a hundredth, up
// to 1.37 -- 25 heads of 512 rows, 2048 keys 19.0 -> 26.0 us --, head dim 128 1 of 168, head dim 256 8 of 172, up to 1.06.  With both 9 of
// 1041, 0 of 167 and 3 of 156; of the 78 calls that the second sum keeps whole 14 would gain more than three hundredths cut.)  Measured, N(0,1), us before -> after: D=128, 36 heads of 256
// rows, 10176 keys 127.6 -> 65.5 (3 units); 16 heads of 1024 rows, 8192 keys 99.2 -> 71.0; 20 heads of 6528 rows, 6144 keys (520
// items of 256 rows) 399 -> 334; D=64, 16 heads of 4512 rows, 6976 keys 174.0 -> 132.4; 160 heads of 1216 rows, 4864 keys 259 -> 234;
// D=256, 36 heads of 256 rows, 8192 keys 225.8 -> 114.4; 15 heads of 2976 rows, 4096 keys 202.1 -> 181.7.  No gain, and the rule
// keeps off: 256 items of 128 rows, D=128, 4096 keys 64.0 / 70.5.
// (Calls of a FmaCfg or a compiler-scheduled build are cut, as a FmaCfg build, where the sums above say less time by a twentieth.  At
// head dim 256 all go by the sums here.)
bool plan_fmha_f16_split(int head_dim, int sq, int skv, int bh, const FmhaPlan &plan, KeySplit *out) {
  const TileWish w = tile_wish();
  const int bn = head_dim == 256 ? 32 : 64, tiles = skv / bn, groups = tiles / 4, left = tiles % 4;
  if (w.bm || w.bn || tiles < 16 || plan.split_tiles || !(plan.hand || (head_dim != 256 && hand_loops_allowed()))) return false;
  if (head_dim != 256 && !(plan.hand && !plan.fma)) {
    const Call call{head_dim, sq, skv, bh};
    float us;
    int rows;
    fma_rows(call, plan.mfma == 16, &us, &rows);
    if (rows) fma_rows(call, true, &us, &rows);   // (where a FmaCfg sum is the least, cuts were fitted beside the sum of fmha_fwd_kernel16)
    us *= 0.95f;
    KeySplit best{};
    for (int bm : {256, 128}) {
      const int items = call.items(bm), from = items / kCus * kCus, cut = items - from;
      for (int n = 2; n * cut <= kCus && 8 * n <= tiles && cut; ++n) {
        const float t = fma_cut_us(call, fma_times(head_dim, bm), n, from);
        if (t < us) us = t, best = KeySplit{n, bm, from};
      }
    }
    if (best.n) *out = best;
    return best.n != 0;
  }
  struct Build { int bm; float full, low, fixed; };
  const Build b256 = head_dim == 64 ? Build{256, 0.885f, 0.62f, 3.f} : Build{256, 1.66f, 1.05f, 5.f};
  const Build b128 = head_dim == 64 ? Build{128, 0.48f, 0.45f, 4.f} : head_dim == 128 ? Build{128, 0.95f, 0.74f, 4.f} : Build{128, 0.884f, 0.67f, 4.f};
  const auto unit_us = [&](const Build &b, int units, int unit_tiles) {
    const float busy = 2.f * units / kCus - 1.f, tile = b.low + (b.full - b.low) * (busy > 0.f ? busy : 0.f);
    return units ? b.fixed + unit_tiles * tile : 0.f;
  };
  const auto rounds_us = [&](const Build &b, int items) {
    return items / kCus * unit_us(b, kCus, tiles) + unit_us(b, items % kCus, tiles);
  };
  const float call_us = rounds_us(plan.block_m == 256 ? b256 : b128, plan.grid);
  float best_us = 0.95f * call_us;
  KeySplit best{};
  bool pays = false;
  for (const Build &b : {b256, b128}) {
    if (head_dim == 256 && b.bm == 256) continue;
    const int items = bh * ((sq + b.bm - 1) / b.bm), from = items / kCus * kCus, cut = items - from;
    const float whole_us = rounds_us(b, from);
    for (int n = 2; n * cut <= kCus && 8 * n <= tiles && cut; ++n) {
      const float units_us = whole_us + unit_us(b, n * cut, 4 * ((groups + n - 1) / n) + left);
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
  const hipError_t split[] = {prepare_fmha_split<A64_256x128>(), prepare_fmha_split<A64_128x128>(), prepare_fmha_split<A128_256x128>(), prepare_fmha_split<A128_128x128>(),
                              prepare_fmha_split<F64_256x128>(), prepare_fmha_split<F64_128x128>(), prepare_fmha_split<F128_256x128>(), prepare_fmha_split<F128_128x128>()};
  for (hipError_t x : split)
    if (e == hipSuccess) e = x;
  if (e == hipSuccess) e = prepare_all(CfgList<C64Tap, C128Tap, C256Tap>{});
  return e;
}

}  // namespace cfk
