// The FMHA forward kernel for few query rows (KsCfg, KsCfg8 below): the waves of a workgroup split the KEYS, not the query
// rows.  A problem like B=1 H=8 S=512 D=64 gives the 128-row tile 32 workgroups for 256 CUs, each of which walks its
// eight key tiles one after the other: the run time is that chain of dependent steps (copy, barrier, S = K.Q^T, softmax,
// O += P.V), not arithmetic.  Here a workgroup owns 32 query rows (four times as many workgroups) and its NWAVES waves
// take the key tiles round-robin (tile j goes to wave j % NWAVES), each with its own running max, row sum and O; the
// partial results meet in the LDS at the end (the merge of online_softmax.h:123-165 across waves instead of across
// tiles).  The chain per wave is then one eighth as long, and no barrier sits inside it.
//
// A query block's keys can further be split over a.n_split workgroups: each leaves its unnormalised fp32 O, reference point
// and row sum in the caller's workspace, and fmha_combine (fmha_combine.hip) merges them the same way.
//
// What bounds it: with few workgroups the latency of that chain, with long key sequences the stream of K and V.  Both are
// copied global -> LDS into tiles of the wave's own, 1 KB of whole rows per instruction: loading K fragments straight into
// registers in operand order (16 rows, 16 bytes a lane) runs at 16 bytes per clock and CU, a quarter of the copies' 64.  K of
// the next tile is requested as soon as this tile's fragments have left the LDS, V behind the second GEMM, so one buffer of
// each keeps 12 to 16 KB (head dim 256: 24 to 32 KB) per wave in flight for most of a turn.
// Mathematics, accumulator layout and key order are those of fmha_fwd_kernel16.h (16x16 MFMAs; lane (c, g) holds keys
// 16 kb + 4 g .. +3 of query 16 qb + c).  e4m3 Q and K multiply on v_mfma_f32_16x16x32_fp8_fp8: half the rate of the
// f8f6f4 form, which does not show here, and the same lane layout with 8 bytes in place of 8 halves.  e4m3 V is turned into
// halves (exactly) as it leaves the LDS and meets fp16 weights: the conversions fit beside the waits for memory, the weights are
// spared their rounding to e4m3 (rms error of O 2.4e-2 -> 3e-4 of its size), and one softmax serves all modes.
#pragma once
#include "fmha_fwd_kernel16.h"

namespace cfk {

// What the dispatch and the kernel want to know of a key-split build.  TK: keys per wave tile; BN: what the key length has to
// be a multiple of; the other names as in FmhaCfg.
template <int D_, int NWAVES_, bool QK8_, bool PV8_, bool VT_, int TK_, int BN_>
struct KsTiles {
  static constexpr int D = D_, NWAVES = NWAVES_, TK = TK_, BN = BN_, BM = 32, T = NWAVES * 64, WPE = 1, SUB = 1, KPRE = 0;
  static constexpr bool QK8 = QK8_, PV8 = PV8_, VT = VT_, TAP_S = false, M16 = true, ASM = false, FMA = false, DIRECT = false, KSPLIT = true;
  static constexpr int K_PITCH = D * (QK8 ? 1 : 2), V_PITCH = VT ? TK : D * (PV8 ? 1 : 2);
  static constexpr int K_BYTES = TK * K_PITCH, V_BYTES = (VT ? D : TK) * V_PITCH, WAVE_BYTES = K_BYTES + V_BYTES;
  static constexpr int K_IPW = K_BYTES / 1024, V_IPW = V_BYTES / 1024;   // 1 KB copies of a tile, all by the wave that owns it
  static constexpr int Q_BYTES = 32 * K_PITCH;
  // LDS: the waves' K and V tiles, later their partial O (32 fp32 rows each); Q; m[NWAVES][32] and l[NWAVES][32]
  static constexpr int Q_ST = NWAVES * (WAVE_BYTES > 32 * D * 4 ? WAVE_BYTES : 32 * D * 4);
  static constexpr int STATS = Q_ST + Q_BYTES;
  static constexpr int LDS_BYTES = STATS + 2 * NWAVES * 32 * 4;
  // about how long a turn of the waves takes while memory keeps up, in us (measured: 64 to 16384 keys, 8 workgroups)
  static constexpr float TURN_US = D == 256 ? (PV8 ? 2.2f : 1.6f) : PV8 && D == 128 ? 1.6f : 1.1f;
  static_assert(K_IPW * 1024 == K_BYTES && V_IPW * 1024 == V_BYTES && Q_BYTES % 1024 == 0 && BN % TK == 0 && TK % 32 == 0, "whole copies and K-steps");
  static_assert(K_IPW + V_IPW < 64 && LDS_BYTES <= 160 * 1024 && !(VT && TK != 64), "");
};
// fp16.  (Head dim 64: 64-key tiles, so that 512 keys are one tile per wave.)
template <int D_, int NWAVES_>
struct KsCfg : KsTiles<D_, NWAVES_, false, false, false, D_ == 64 ? 64 : 32, D_ == 256 ? 32 : 64> {};
// e4m3 Q and K; PV8: e4m3 P and V too, VT: V pre-transposed
template <int D_, int NWAVES_, bool PV8_, bool VT_>
struct KsCfg8 : KsTiles<D_, NWAVES_, true, PV8_, VT_, PV8_ || D_ == 64 ? 64 : 32, PV8_ || D_ != 256 ? 64 : 32> {};

template <class C>
__global__ void __launch_bounds__(C::T) fmha_fwd_kernel_ks(const FmhaArgs a) {
  static_assert(C::KSPLIT && !C::TAP_S, "");
  constexpr bool QK8 = C::QK8, PV8 = C::PV8, VT = C::VT;
  constexpr int D = C::D, TK = C::TK, W = C::NWAVES;
  constexpr int QB = 2, KB = TK / 16, DB = D / 16, PS = TK / 32;
  constexpr int KF = C::K_PITCH / 64;            // 16-byte fragments of a K row per lane (e4m3: two K-steps of 8 bytes each)
  constexpr int QES = QK8 ? 1 : 2, VES = PV8 ? 1 : 2;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;

  // (the query blocks that read the same keys next to each other: one XCD's L2)
  const int q_blocks = a.Sq / 32;
  const int unit = xcd_remap(blockIdx.x, gridDim.x);
  const int part = unit / q_blocks;
  const int q0 = (unit - part * q_blocks) * 32;
  const int bh = part / a.n_split, split = part - bh * a.n_split;
  const int b = bh / a.H, h = bh - b * a.H;
  const int64_t ld = (int64_t)a.H * D;  // row stride in elements
  const char *Qp = (const char *)a.q + ((((int64_t)b * a.Sq + q0) * a.H + h) * D) * QES;
  const char *Kp = (const char *)a.k + (((int64_t)b * a.Skv * a.H + h) * D) * QES;
  const char *Vp = VT ? (const char *)a.v + ((int64_t)b * D * a.H + h) * a.Skv : (const char *)a.v + (((int64_t)b * a.Skv * a.H + h) * D) * VES;
  const int tiles = a.Skv / TK;
  const int t_first = (int)((int64_t)tiles * split / a.n_split), t_end = (int)((int64_t)tiles * (split + 1) / a.n_split);
  const float c_log2 = a.scale_log2;
  const uint32_t k_ld = (uint32_t)(ld * QES), v_ld = VT ? (uint32_t)a.H * (uint32_t)a.Skv : (uint32_t)(ld * VES);  // global row pitch in bytes
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

  // ---- this wave's K and V tile: copied by the wave itself, 1 KB per instruction; chunk position ^ swizzle on the global side
  const uint32_t lds_base = (uint32_t)(uintptr_t)LDS_PTR(char, smem);
  const uint32_t k_tile = lds_base + wave * C::WAVE_BYTES, v_tile = k_tile + C::K_BYTES;
  auto swz_k = [](int row) { return QK8 ? swz_row<C::K_PITCH>(row) : swz_k16n<C::K_PITCH>(row); };
  auto swz_v = [](int row) { return PV8 ? swz_row<C::V_PITCH>(row) : swz_v16n<C::V_PITCH>(row); };
  constexpr int K_CPR = C::K_PITCH / 16, V_CPR = C::V_PITCH / 16;
  uint32_t goff_k[C::K_IPW], goff_v[C::V_IPW];
#pragma unroll
  for (int i = 0; i < C::K_IPW; ++i) {
    const int row = i * (64 / K_CPR) + lane / K_CPR;
    // pre-transposed V: a lane's eight P slots of a 32-key step are to be eight contiguous keys, so row 16 kb + 4 g + j of the
    // step holds key 8 g + 4 kb + j
    const int key = VT ? (row & ~31) + 8 * ((row >> 2) & 3) + 4 * ((row >> 4) & 1) + (row & 3) : row;
    goff_k[i] = (uint32_t)key * k_ld + (uint32_t)(((lane % K_CPR) ^ swz_k(row)) * 16);
  }
#pragma unroll
  for (int i = 0; i < C::V_IPW; ++i) {
    const int row = i * (64 / V_CPR) + lane / V_CPR;
    goff_v[i] = (uint32_t)row * v_ld + (uint32_t)(((lane % V_CPR) ^ swz_v(row)) * 16);
  }
  auto load_k = [&](int j) __attribute__((always_inline)) {
    const char *kt = Kp + (size_t)j * ((size_t)TK * k_ld);
#pragma unroll
    for (int i = 0; i < C::K_IPW; ++i) lds_dma16(kt, goff_k[i], k_tile, i * 1024);
  };
  auto load_v = [&](int j) __attribute__((always_inline)) {
    const char *vt = VT ? Vp + (size_t)j * TK : Vp + (size_t)j * ((size_t)TK * v_ld);
#pragma unroll
    for (int i = 0; i < C::V_IPW; ++i) lds_dma16(vt, goff_v[i], v_tile, i * 1024);
  };
  uint32_t k_rd[KF], v_rd[DB];
#pragma unroll
  for (int f = 0; f < KF; ++f) k_rd[f] = k_tile + c * C::K_PITCH + (((4 * f + g) ^ swz_k(c)) * 16);   // + 16 rows per key block
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    if constexpr (VT) {          // row d = 16 db + c, keys 8 g .. +7 of a step
      v_rd[db] = v_tile + (16 * db + c) * C::V_PITCH + (((g >> 1) ^ swz_v(c)) * 16) + 8 * (g & 1);
    } else if constexpr (PV8) {  // lane L of 16 hands the transposing read row L/2 of its eight keys, columns 8 (L%2) .. +7
      const int e = c >> 1, v_key = 16 * (e >> 2) + 4 * g + (e & 3);
      v_rd[db] = v_tile + v_key * C::V_PITCH + ((db ^ swz_v(v_key)) * 16) + 8 * (c & 1);
    } else {
      const int v_key = 4 * g + (c >> 2), cg = c & 3;
      v_rd[db] = v_tile + v_key * C::V_PITCH + (((2 * db + (cg >> 1)) ^ swz_v(v_key)) * 16) + (cg & 1) * 8;
    }
  }

  // ---- Q: 32 rows through the LDS once for all waves, in K's row format
  int j = t_first + wave;
#pragma unroll
  for (int i = 0; i < (C::Q_BYTES / 1024 + W - 1) / W; ++i) {
    const int p = i * W + wave;
    if (p < C::Q_BYTES / 1024) {
      const int row = p * (64 / K_CPR) + lane / K_CPR;
      lds_dma16(Qp, (uint32_t)row * k_ld + (uint32_t)(((lane % K_CPR) ^ swz_k(row)) * 16), lds_base + C::Q_ST, p * 1024);
    }
  }
  if (j < t_end) {
    load_k(j);
    load_v(j);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(C::K_IPW + C::V_IPW) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }
  int4v qreg[QB][KF];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int f = 0; f < KF; ++f) qreg[qb][f] = *LDS_AT(int4v, lds_base + C::Q_ST + (16 * qb + c) * C::K_PITCH + (((4 * f + g) ^ swz_k(c)) * 16));

  f32x4 oacc[DB][QB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) oacc[db][qb] = zero4;
  float m_ref[QB], l_run[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) m_ref[qb] = -INFINITY, l_run[qb] = 0.f;

  auto as_long = [](int lo, int hi) { return (long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo); };
  for (; j < t_end; j += W) {
    const bool more = j + W < t_end;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::V_IPW) : "memory");   // K has landed (V, requested behind it, may be on its way)
    f32x4 s_[KB][QB];
#pragma unroll
    for (int f = 0; f < KF; ++f)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int4v ka = *LDS_AT(int4v, k_rd[f] + kb * 16 * C::K_PITCH);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          f32x4 acc = f == 0 ? zero4 : s_[kb][qb];
          if constexpr (QK8) {
            acc = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(as_long(ka[0], ka[1]), as_long(qreg[qb][f][0], qreg[qb][f][1]), acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(as_long(ka[2], ka[3]), as_long(qreg[qb][f][2], qreg[qb][f][3]), acc, 0, 0, 0);
          } else {
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, ka), __builtin_bit_cast(half8, qreg[qb][f]), acc, 0, 0, 0);
          }
          s_[kb][qb] = acc;
        }
      }
    // the fragments have left the tile: K of the next turn
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) load_k(j + W);
    // online softmax, reference point = running max (online_softmax.h:123-165)
    half8 pb[QB][PS];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const float m_old = m_ref[qb];
      float mx = s_[0][qb][0];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int t = 0; t < 4; ++t) mx = __builtin_fmaxf(mx, s_[kb][qb][t]);
      // (while all of a row's scores are -inf -- keys masked by an infinite K -- the point stays there and the weights, taken
      // against 0, are 0: which keys a wave meets first is this kernel's choice, and -inf minus -inf would be NaN)
      m_ref[qb] = fmaxf(m_old, quad_max(mx) * c_log2);
      const float m_new = m_ref[qb] == -INFINITY ? 0.f : m_ref[qb];
      const float alpha = __builtin_amdgcn_exp2f(m_old - m_new);
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[db][qb] *= alpha;
      float rs = 0.f;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s_[kb][qb][t], c_log2, -m_new));
          rs += p;   // summed in fp32 before the cast (online_softmax.h:173-206)
          pb[qb][kb / 2][4 * (kb % 2) + t] = (_Float16)p;
        }
      l_run[qb] = l_run[qb] * alpha + rs;
    }
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::K_IPW) : "memory");   // V has landed
    else wait_lds_dma();
#pragma unroll
    for (int ps = 0; ps < PS; ++ps)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        half8 va;
        if constexpr (PV8) {
          int2v x;
          // (pre-transposed: 32 keys further are 32 bytes, chunk 2 of the row's four: the swizzle leaves its bit 1 to the XOR)
          if constexpr (VT) x = *LDS_AT(int2v, v_rd[db] ^ (ps * 32));
          else x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_AT(int2v, v_rd[db] + ps * 32 * C::V_PITCH));
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const half2v lo = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(x[t], 1.0f, false), hi = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(x[t], 1.0f, true);
            va[4 * t] = lo[0], va[4 * t + 1] = lo[1], va[4 * t + 2] = hi[0], va[4 * t + 3] = hi[1];
          }
        } else {
          const uint32_t vp = v_rd[db] + ps * 32 * C::V_PITCH;
          union {
            struct { short4v lo, hi; } s2;
            half8 h;
          } u;
          u.s2.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_AT(short4v, vp));
          u.s2.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_AT(short4v, vp + 16 * C::V_PITCH));
          va = u.h;
        }
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) oacc[db][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb[qb][ps], oacc[db][qb], 0, 0, 0);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the fragments have left the tile: V of the next turn
    if (more) load_v(j + W);
  }

  // ---- the partial results meet: wave u leaves O_u as fp32 rows (chunks of 4 XOR-swizzled by the row) and per query its
  // reference point m_u and row sum l_u; a wave without tiles leaves m = -inf, l = 0, O = 0
  __syncthreads();   // (the rows lie over other waves' tiles)
  {
    char *op = smem + wave * (32 * D * 4);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) *(f32x4 *)(op + (16 * qb + c) * (D * 4) + (((4 * db + g) ^ c) * 16)) = oacc[db][qb];
    float *st = (float *)(smem + C::STATS);
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const float l_tot = quad_sum(l_run[qb]);
      if (g == 0) {
        st[wave * 32 + 16 * qb + c] = m_ref[qb];
        st[(W + wave) * 32 + 16 * qb + c] = l_tot;
      }
    }
  }
  __syncthreads();
  // a thread takes eight consecutive d of a row
  const float *st = (const float *)(smem + C::STATS);
  for (int e = tid; e < 32 * (D / 8); e += C::T) {
    const int row = e / (D / 8), d8 = e % (D / 8);
    float m_all = -INFINITY;
#pragma unroll
    for (int u = 0; u < W; ++u) m_all = fmaxf(m_all, st[u * 32 + row]);
    float l_all = 0.f;
    f32x4 o_all[2] = {zero4, zero4};
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const float m_u = st[u * 32 + row];
      const float w_u = m_u == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_u - m_all);
      l_all += st[(W + u) * 32 + row] * w_u;
#pragma unroll
      for (int i = 0; i < 2; ++i) o_all[i] += *(const f32x4 *)(smem + u * (32 * D * 4) + row * (D * 4) + (((2 * d8 + i) ^ (row & 15)) * 16)) * w_u;
    }
    const int64_t si = (int64_t)bh * a.Sq + q0 + row;
    if (a.n_split > 1) {
      const int64_t pi = (int64_t)split * a.B * a.H * a.Sq + si;
      f32x4 *po = (f32x4 *)(a.part_o + pi * D + d8 * 8);
      po[0] = o_all[0];
      po[1] = o_all[1];
      if (d8 == 0) {
        a.part_ml[2 * pi] = m_all;
        a.part_ml[2 * pi + 1] = l_all;
      }
      continue;
    }
    const float inv = a.out_scale / l_all;
    half8 o8;
#pragma unroll
    for (int t = 0; t < 8; ++t) o8[t] = (_Float16)(o_all[t / 4][t % 4] * inv);
    *(half8 *)((_Float16 *)a.o + (((int64_t)b * a.Sq + q0 + row) * a.H + h) * D + d8 * 8) = o8;
    if (d8 == 0) {
      // the reference point follows the running max in every wave: the merged one is the true row max
      if (a.row_max) a.row_max[si] = m_all;
      if (a.row_sum) a.row_sum[si] = l_all;
    }
  }
}

}  // namespace cfk
