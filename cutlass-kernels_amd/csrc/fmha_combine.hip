// Merges the partial results of a call whose keys were split over workgroups (a.n_split of them per query block): the merge
// of online_softmax.h:123-165 across key ranges.  One thread per eight consecutive d of a query row.
// Bound by reading the partial O, n_split x 4 bytes per element of O, from the caches.
#include "fmha_common.h"

namespace cfk {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;

template <int D>
__global__ void __launch_bounds__(kThreads) fmha_combine(const FmhaArgs a) {
  const int q_blocks = (a.Sq + a.split_bm - 1) / a.split_bm;
  const int64_t rows = (int64_t)(a.B * a.H * q_blocks - a.split_from) * a.split_bm;
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t row = e / (D / 8);
  if (row >= rows) return;
  const int d8 = (int)(e % (D / 8));
  const int block = (int)(row / a.split_bm), bh = (a.split_from + block) / q_blocks;
  const int q = (a.split_from + block - bh * q_blocks) * a.split_bm + (int)(row - (int64_t)block * a.split_bm);
  if (q >= a.Sq) return;   // (behind the last row of a partly filled block)
  const f32x2 *ml = (const f32x2 *)a.part_ml;
  float m_all = -INFINITY;
  for (int s = 0; s < a.n_split; ++s) m_all = fmaxf(m_all, ml[s * rows + row][0]);
  float l_all = 0.f;
  f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = o0;
#pragma unroll 4
  for (int s = 0; s < a.n_split; ++s) {
    const f32x2 x = ml[s * rows + row];
    const float w = x[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(x[0] - m_all);   // (no finite score among the part's keys)
    const f32x4 *po = (const f32x4 *)(a.part_o + (s * rows + row) * D + d8 * 8);
    l_all += x[1] * w;
    o0 += po[0] * w;
    o1 += po[1] * w;
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
