// Merges the partial results of a call whose keys were split over workgroups (a.n_split of them per query block): the merge
// of online_softmax.h:123-165 across key ranges.  One thread per eight consecutive d of a query row.
// Bound by latency: a few waves a CU, each of which needs the parts' reference points, then the partial O, from the caches (n_split x 4
// bytes per element of O).  Up to eight parts everything is asked for before anything is waited for; with a loop over the parts, whose
// first turns waited for one reference point after the other, the kernel took 6.4 us for 48 blocks of 256 rows, head dim 64, in five
// parts (now 5.2), and 2 x 16 heads of 64 rows, 16384 keys, head dim 128 (four parts) 63.6 us as a whole call (now 61.7).
#include <type_traits>

#include "fmha_common.h"

namespace cfk {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;

template <int D>
__global__ void __launch_bounds__(kThreads) fmha_combine(const FmhaArgs a) {
  const int bm = __builtin_ctz(a.split_bm), q_blocks = (a.Sq + a.split_bm - 1) >> bm;   // (32, 128 or 256 rows)
  const int64_t rows = (int64_t)(a.B * a.H * q_blocks - a.split_from) * a.split_bm;
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t row = e / (D / 8);
  if (row >= rows) return;
  const int d8 = (int)(e % (D / 8));
  const int block = (int)(row >> bm), bh = (a.split_from + block) / q_blocks;
  const int q = (a.split_from + block - bh * q_blocks) * a.split_bm + (int)(row - (int64_t)block * a.split_bm);
  if (q >= a.Sq) return;   // (behind the last row of a partly filled block)
  const f32x2 *ml = (const f32x2 *)a.part_ml + row;
  const float *part_o = a.part_o + row * D + d8 * 8;
  float m_all = -INFINITY, l_all = 0.f;
  f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = o0;
  const auto add = [&](f32x2 x, f32x4 p0, f32x4 p1) __attribute__((always_inline)) {
    const float w = x[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(x[0] - m_all);   // (no finite score among the part's keys)
    l_all += x[1] * w;
    o0 += p0 * w;
    o1 += p1 * w;
  };
  const auto all = [&](auto n) __attribute__((always_inline)) {
    constexpr int N = decltype(n)::value;
    f32x2 x[N];
    f32x4 p0[N], p1[N];
#pragma unroll
    for (int s = 0; s < N; ++s) x[s] = ml[s * rows];
#pragma unroll
    for (int s = 0; s < N; ++s) p0[s] = ((const f32x4 *)(part_o + s * rows * D))[0], p1[s] = ((const f32x4 *)(part_o + s * rows * D))[1];
#pragma unroll
    for (int s = 0; s < N; ++s) m_all = fmaxf(m_all, x[s][0]);
#pragma unroll
    for (int s = 0; s < N; ++s) add(x[s], p0[s], p1[s]);
  };
  switch (a.n_split) {
    case 2: all(std::integral_constant<int, 2>{}); break;
    case 3: all(std::integral_constant<int, 3>{}); break;
    case 4: all(std::integral_constant<int, 4>{}); break;
    case 5: all(std::integral_constant<int, 5>{}); break;
    case 6: all(std::integral_constant<int, 6>{}); break;
    case 7: all(std::integral_constant<int, 7>{}); break;
    case 8: all(std::integral_constant<int, 8>{}); break;
    default:
#pragma unroll 8
      for (int s = 0; s < a.n_split; ++s) m_all = fmaxf(m_all, ml[s * rows][0]);
#pragma unroll 8
      for (int s = 0; s < a.n_split; ++s) add(ml[s * rows], ((const f32x4 *)(part_o + s * rows * D))[0], ((const f32x4 *)(part_o + s * rows * D))[1]);
  }
  const float inv = a.out_scale / l_all;
  half8 o8;
#pragma unroll
  for (int t = 0; t < 4; ++t) o8[t] = (_Float16)(o0[t] * inv), o8[4 + t] = (_Float16)(o1[t] * inv);
  const int b = bh / a.H, h = bh - b * a.H;
  *(half8 *)((_Float16 *)a.o + (((int64_t)b * a.Sq + q) * a.H + h) * D + d8 * 8) = o8;
  if (d8 == 0) {   // (the parts' reference points are the row maxima of their keys)
    const int64_t si = (int64_t)bh * a.Sq + q;
    if (a.row_max) a.row_max[si] = m_all;
    if (a.row_sum) a.row_sum[si] = l_all;
  }
}

}  // namespace

hipError_t launch_fmha_combine(const FmhaArgs &a, int head_dim, hipStream_t s) {
  const int blocks = a.B * a.H * ((a.Sq + a.split_bm - 1) / a.split_bm) - a.split_from;
  const int64_t threads = (int64_t)blocks * a.split_bm * (head_dim / 8);
  const dim3 grid((unsigned)((threads + kThreads - 1) / kThreads)), block(kThreads);
  switch (head_dim) {
    case 64: hipLaunchKernelGGL(fmha_combine<64>, grid, block, 0, s, a); break;
    case 128: hipLaunchKernelGGL(fmha_combine<128>, grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL(fmha_combine<256>, grid, block, 0, s, a); break;
  }
  return hipGetLastError();
}

}  // namespace cfk
