// FMHA forward, hybrid precision: Q, K e4m3 (GEMM-I on the fp8 MFMA), P and V fp16 (GEMM-II on the fp16 MFMA) --
// what the reference's --prec-type=2 computes when built without -DGEMM2FP8 (src/fmha-pipeline/fmha_forward.cu:
// 446-450).  Tile shapes and dispatch; the kernel is in fmha_fwd_kernel.h.
#include "fmha_fwd_kernel.h"
#include "fmha_fwd_kernel_ks.h"
#include "fmha_split_choice.h"

namespace cfk {
namespace {

// template arguments as in fmha_fwd_f16.hip
using C64_128x64 = FmhaCfg<64, 64, 4, 3, true, false>;
using C64_128x128 = FmhaCfg<64, 64, 4, 2, true, false, false, false, 2>;
using C128_128x64 = FmhaCfg<128, 64, 4, 2, true, false>;
using C128_256x64 = FmhaCfg<128, 64, 8, 2, true, false>;
using C128_256x128 = FmhaCfg<128, 64, 8, 2, true, false, false, false, 2>;
using C256_128x32 = FmhaCfg<256, 32, 4, 1, true, false>;
// (No 16x16-MFMA build for this mode.  With S on v_mfma_f32_16x16x128_f8f6f4 and the reference point found by the row sum, as in
// fmha_fwd_kernel16.h, its time depends on the scores, which that of a hybrid call is not to do: B=4 H=16 S=4096 D=128 684 us against
// 406 where they climb along the keys.  On N(0,1) data, time relative to this build, medians of 420 drawn calls, each side 0.1 s at a
// time in turn: head dim 128 1.09 at 192 keys, 1.05 at 256 to 361, 1.03 to 511, 0.97..0.98 at 512 to 1447, 0.99..1.00 beyond
// (B=4 H=16 S=4096 398 us here, 383 there); head dim 64 1.01..1.02.)

// few query rows: the waves of a workgroup split the keys (fmha_fwd_kernel_ks.h; not by wish)
using K64 = KsCfg8<64, 8, false, false>;
using K128 = KsCfg8<128, 8, false, false>;
using K256 = KsCfg8<256, 4, false, false>;

// builds that also write the score tap (debug): 128-row tile only
using C64Tap = FmhaCfg<64, 64, 4, 2, true, false, false, true>;
using C128Tap = FmhaCfg<128, 64, 4, 2, true, false, false, true>;
using C256Tap = FmhaCfg<256, 32, 4, 1, true, false, false, true>;

using All64 = CfgList<C64_128x64, C64_128x128>;
using All128 = CfgList<C128_128x64, C128_256x64, C128_256x128>;
using All256 = CfgList<C256_128x32>;

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
    case 64: select_tile<All64, CfgList<K64, C64_128x64>, C64_128x64>(sq, skv, bh, f); return true;
    case 128: select_tile<All128, CfgList<K128, C128_256x64, C128_128x64>, C128_128x64>(sq, skv, bh, f); return true;
    case 256: select_tile<All256, CfgList<K256, C256_128x32>, C256_128x32>(sq, skv, bh, f); return true;
    default: return false;
  }
}

}  // namespace

bool plan_fmha_hybrid(int head_dim, int sq, int skv, int bh, bool tap_s, FmhaPlan *p) {
  return dispatch(head_dim, sq, skv, bh, tap_s, [&](auto cfg) { fill_fmha_plan<decltype(cfg)>(sq, skv, bh, p); });
}

bool plan_fmha_hybrid_split(int head_dim, int sq, int skv, int bh, const FmhaPlan &plan, KeySplit *out) {
  const TileWish w = tile_wish();
  if (plan.split_tiles || w.bm || w.bn) return false;
  static constexpr CutTimes k64{3, {0.404f, 0.609f, 1.039f, 1.314f}, 1.3f, 3.61f, 2.42f, 2.44f}, k128{2, {0.606f, 0.841f, 1.51f}, 2.74f, 2.1f, 3.65f, 3.16f},
      k256{1, {1.207f, 1.481f}, 5.35f, 0.75f, 0.f, 2.31f};
  const float mbytes = 1e-6f * bh * head_dim * 3.f * ((float)sq + skv);
  return choose_cut(head_dim == 64 ? k64 : head_dim == 128 ? k128 : k256, bh * ((sq + 127) / 128), skv,
                    head_dim == 256 ? 32 : 64, mbytes, head_dim, plan, out);
}

hipError_t launch_fmha_hybrid(const FmhaArgs &a, int head_dim, hipStream_t s) {
  hipError_t e = hipErrorNotSupported;
  if (a.n_split > 1 && a.split_bm == 128) return head_dim == 64 ? launch_fmha_split<C64_128x64>(a, s) : head_dim == 128 ? launch_fmha_split<C128_128x64>(a, s) : launch_fmha_split<C256_128x32>(a, s);
  dispatch(head_dim, a.Sq, a.Skv, a.B * a.H, a.s_tap != nullptr, [&](auto cfg) { e = launch_fmha_cfg<decltype(cfg)>(a, s); });
  return e;
}

hipError_t prepare_fmha_hybrid() {
  hipError_t e = prepare_all(All64{});
  if (e == hipSuccess) e = prepare_all(All128{});
  if (e == hipSuccess) e = prepare_all(All256{});
  if (e == hipSuccess) e = prepare_all(CfgList<K64, K128, K256>{});
  const hipError_t split[] = {prepare_fmha_split<C64_128x64>(), prepare_fmha_split<C128_128x64>(), prepare_fmha_split<C256_128x32>()};
  for (hipError_t x : split)
    if (e == hipSuccess) e = x;
  if (e == hipSuccess) e = prepare_all(CfgList<C64Tap, C128Tap, C256Tap>{});
  return e;
}

}  // namespace cfk
