// FMHA forward, e4m3 operands for both GEMMs (the reference's -DGEMM2FP8 build): tile shapes and dispatch.
// The kernel, including the fp8 V-tile layout transform, is in fmha_fwd_kernel.h.
#include "fmha_fwd_kernel.h"
#include "fmha_fwd_kernel8p.h"
#include "fmha_fwd_kernel_ks.h"
#include "fmha_split_choice.h"

namespace cfk {
namespace {

// template arguments as in fmha_fwd_f16.hip.  Head dim 64 runs three waves per SIMD (the VALU-bound softmax gains from
// every extra wave); head dim 256 one (O 128 + S 64 + Q 32 registers).
using C64_128x64 = FmhaCfg<64, 64, 4, 3, true, true>;
using C64_128x128 = FmhaCfg<64, 64, 4, 2, true, true, false, false, 2>;
using C128_128x64 = FmhaCfg<128, 64, 4, 2, true, true>;
using C128_256x64 = FmhaCfg<128, 64, 8, 2, true, true>;
using C128_128x128 = FmhaCfg<128, 64, 4, 2, true, true, false, false, 2>;
using C128_256x128 = FmhaCfg<128, 64, 8, 2, true, true, false, false, 2>;
// ... with the hand-scheduled main loop and persistent workgroups (fmha_fwd_kernel8p.h); key sequences from 3072 (by wish
// from 512): below, e4m3 weights run the max-tracking pass only (cfk_api.hip, hand_loop_pays in fmha_fwd_kernel.h),
// which this build would do in a loop that is not pipelined
using A128_256x128 = FmhaCfg<128, 64, 8, 2, true, true, false, false, 2, 0, false, true>;
using A128_128x128 = FmhaCfg<128, 64, 4, 2, true, true, false, false, 2, 0, false, true>;   // the same loop, 4 waves, one per SIMD
using C256_128x64 = FmhaCfg<256, 64, 4, 1, true, true>;
using C256_128x128 = FmhaCfg<256, 64, 4, 1, true, true, false, false, 2>;

// few query rows: the waves of a workgroup split the keys (fmha_fwd_kernel_ks.h; not by wish)
using K64 = KsCfg8<64, 8, true, false>;
using K128 = KsCfg8<128, 8, true, false>;
using K256 = KsCfg8<256, 4, true, false>;
using K64T = KsCfg8<64, 8, true, true>;
using K128T = KsCfg8<128, 8, true, true>;
using K256T = KsCfg8<256, 4, true, true>;

// V pre-transposed to [B,D,H,S] (the reference's offline transpose, src/fmha-pipeline/fmha_forward.cu:514-532)
// Head dim 64: three waves per SIMD once there are more than two workgroups for every CU (B=8 H=16 S=1024 36.7 -> 34.5 us, B=4
// H=16 S=4096 180 -> 173, 8 x 32 heads of 544 rows, 384 keys 20.3 -> 18.8; up to 512 workgroups a tie, 31.3 at B=2 H=16 S=2048;
// two key tiles per barrier at two waves 36.3, 174 and 20.0).
using C64T3 = FmhaCfg<64, 64, 4, 3, true, true, true>;
using C64T = FmhaCfg<64, 64, 4, 2, true, true, true>;
using C128T = FmhaCfg<128, 64, 4, 2, true, true, true>;
using C256T = FmhaCfg<256, 64, 4, 1, true, true, true>;

// builds that also write the score tap (debug)
using C64Tap = FmhaCfg<64, 64, 4, 2, true, true, false, true>;
using C128Tap = FmhaCfg<128, 64, 4, 2, true, true, false, true>;
using C256Tap = FmhaCfg<256, 64, 4, 1, true, true, false, true>;
using C64TTap = FmhaCfg<64, 64, 4, 2, true, true, true, true>;
using C128TTap = FmhaCfg<128, 64, 4, 2, true, true, true, true>;
using C256TTap = FmhaCfg<256, 64, 4, 1, true, true, true, true>;

using All64 = CfgList<C64_128x64, C64_128x128>;
using All128 = CfgList<C128_128x64, C128_256x64, C128_128x128, C128_256x128, A128_256x128, A128_128x128>;
using All256 = CfgList<C256_128x64, C256_128x128>;

template <class F>
bool dispatch(int head_dim, int sq, int skv, int bh, int v_layout, bool tap_s, F &&f) {
  if (tap_s) {
    const bool t = v_layout == 1;
    switch (head_dim) {
      case 64: t ? f(C64TTap{}) : f(C64Tap{}); return true;
      case 128: t ? f(C128TTap{}) : f(C128Tap{}); return true;
      case 256: t ? f(C256TTap{}) : f(C256Tap{}); return true;
      default: return false;
    }
  }
  if (v_layout == 1) {
    switch (head_dim) {
      case 64: 
      if ((long long)bh * ((sq + 127) / 128) > 512) select_tile<CfgList<C64T3>, CfgList<K64T, C64T3>, C64T3>(sq, skv, bh, f);
      else select_tile<CfgList<C64T>, CfgList<K64T, C64T>, C64T>(sq, skv, bh, f);
      return true;
      case 128: select_tile<CfgList<C128T>, CfgList<K128T, C128T>, C128T>(sq, skv, bh, f); return true;
      case 256: select_tile<CfgList<C256T>, CfgList<K256T, C256T>, C256T>(sq, skv, bh, f); return true;
      default: return false;
    }
  }
  switch (head_dim) {
    case 64: select_tile<All64, CfgList<K64, C64_128x64>, C64_128x64>(sq, skv, bh, f); return true;
    // big problems: 256 rows with one barrier per 128 keys (+4 % on N(0,1) data over the 128x64 tile)
    case 128: select_tile<All128, CfgList<K128, A128_256x128, A128_128x128, C128_256x128, C128_128x64>, C128_128x64>(sq, skv, bh, f); return true;
    // one barrier per 128 keys: +11 % at head dim 256 (1604 against 1439 TFLOP/s, B=4 H=8 S=4096)
    case 256: select_tile<All256, CfgList<K256, C256_128x128, C256_128x64>, C256_128x64>(sq, skv, bh, f); return true;
    default: return false;
  }
}

// the SplitCfg build of a call: compiler-scheduled, 128 rows
template <class F>
void split_build(int head_dim, int skv, int v_layout, int units, F &&f) {
  if (head_dim == 64) return v_layout != 1 ? f(C64_128x64{}) : units > 512 ? f(C64T3{}) : f(C64T{});
  if (head_dim == 128) return v_layout != 1 ? f(C128_128x64{}) : f(C128T{});
  return v_layout == 1 ? f(C256T{}) : skv % 128 == 0 ? f(C256_128x128{}) : f(C256_128x64{});
}

}  // namespace

bool plan_fmha_fp8(int head_dim, int sq, int skv, int bh, int v_layout, bool tap_s, FmhaPlan *p) {
  return dispatch(head_dim, sq, skv, bh, v_layout, tap_s, [&](auto cfg) { fill_fmha_plan<decltype(cfg)>(sq, skv, bh, p); });
}

// The pass that tracks the row max (key lengths below 3072; cfk_api.hip) is slower in a way of its own.
bool plan_fmha_fp8_split(int head_dim, int sq, int skv, int bh, const FmhaPlan &plan, KeySplit *out) {
  const TileWish w = tile_wish();
  const bool first_pass = skv >= 3072 && !predictable_latency();
  if (plan.split_tiles || w.bm || w.bn || fast_e4m3_weights() || (!first_pass && head_dim != 256)) return false;
  static constexpr CutTimes k64{3, {0.234f, 0.393f, 0.662f, 0.827f}, 8.67f, 1.06f, 0.f, 2.52f}, k128{2, {0.424f, 0.491f, 0.935f}, 0.f, 11.f, 1.95f, 4.43f},
      k256{1, {0.895f, 1.023f}, 0.f, 2.84f, 0.f, 1.92f}, k256_tracked{1, {1.665f, 1.782f}, 4.66f, 0.83f, 6.07f, 4.32f};
  const CutTimes &c = head_dim == 64 ? k64 : head_dim == 128 ? k128 : first_pass ? k256 : k256_tracked;
  const float mbytes = 1e-6f * bh * head_dim * (3.f * sq + 2.f * skv);
  return choose_cut(c, bh * ((sq + 127) / 128), skv, head_dim == 256 && skv % 128 == 0 ? 128 : 64, mbytes,
                    head_dim, plan, out);
}

hipError_t launch_fmha_fp8(const FmhaArgs &a, int head_dim, hipStream_t s) {
  hipError_t e = hipErrorNotSupported;
  if (a.n_split > 1 && a.split_bm == 128) {
    const int items = a.B * a.H * ((a.Sq + 127) / 128);
    split_build(head_dim, a.Skv, a.v_layout, a.split_from + (items - a.split_from) * a.n_split, [&](auto cfg) { e = launch_fmha_split<decltype(cfg)>(a, s); });
    return e;
  }
  dispatch(head_dim, a.Sq, a.Skv, a.B * a.H, a.v_layout, a.s_tap != nullptr, [&](auto cfg) { e = launch_fmha_cfg<decltype(cfg)>(a, s); });
  return e;
}

hipError_t prepare_fmha_fp8() {
  hipError_t e = prepare_all(All64{});
  if (e == hipSuccess) e = prepare_all(All128{});
  if (e == hipSuccess) e = prepare_all(All256{});
  if (e == hipSuccess) e = prepare_all(CfgList<K64, K128, K256, K64T, K128T, K256T>{});
  const hipError_t split[] = {prepare_fmha_split<C64_128x64>(), prepare_fmha_split<C64T3>(), prepare_fmha_split<C64T>(), prepare_fmha_split<C128_128x64>(),
                              prepare_fmha_split<C128T>(), prepare_fmha_split<C256T>(), prepare_fmha_split<C256_128x128>(), prepare_fmha_split<C256_128x64>()};
  for (hipError_t x : split)
    if (e == hipSuccess) e = x;
  if (e == hipSuccess) e = prepare_all(CfgList<C64T, C64T3, C128T, C256T, C64Tap, C128Tap, C256Tap, C64TTap, C128TTap, C256TTap>{});
  return e;
}

}  // namespace cfk
