// Dense (batched) GEMM D = alpha * A.B + beta * C with fp32 accumulation and an fp32 epilogue, D row-major M x N, for
// fp16 operands (v_mfma_f32_16x16x32_f16) and fp32 operands (v_mfma_f32_32x32x2_f32) -- gfx950 only.
//
// Secondary bench beside the attention kernels, with their XOR-swizzled LDS rows and transpose reads.
// Takes the place of gemm_device/gemm of the reference's CuTe example (src/cute-gemm-tma-gma/gemm.cu:57-463: TMA load
// of one A and one B tile, one synchronous WGMMA batch per K-tile, no pipelining; its type 1 is float, type 3 half,
// :677-684; batch count L with packed strides, :519-521) and of the CUTLASS-API example with its alpha / beta
// epilogue (src/cutlass-gemm/gemm.cu:87-140, 318-324).  Layouts: TN = A is M x K and B is N x K, both K-contiguous
// (the reference's form, :362-380); NN (fp16 only) = B is K x N, N-contiguous (the literal C = A.B), whose B operand is
// read with ds_read_b64_tr_b16 exactly as V is in the attention kernel.  The reference writes C column-major
// (:386-389); C and D are row-major here.  gfx950 has no tf32/xf32 MFMA: fp32 operands multiply in full fp32.
//
// gemm_kernel16 (fp16): 8 waves, two per SIMD, on a 256 x 256 macro tile, for as many of those as fill the CUs
// in whole rounds; wave (wm, wn) of a 2 x 4 grid owns 128 x 64 of C, its 128 accumulator registers in the AGPR half of the
// register file, 8 x 4 blocks of 16x16x32 MFMAs (the power-efficient shape on this board).  K tiles are 128 bytes deep and go
// global -> registers -> LDS: 16-byte buffer loads a tile ahead (scalar resource + 32-bit lane offset, no vector address
// arithmetic), parked in one of two 64 KB LDS stages by ds_write_b128 while the other stage multiplies, one barrier per tile;
// every multiply is followed by at most one fragment read or one store/load pair, see the pipeline comment at BlockCfg.
// gemm_kernel16_rows, gemm_kernel16<NN, 3>: the same kernel on 192 x 192, 192 x 256, 256 x 192 and 320 x 256 macro tiles, for products whose
// rounds these fill better (choose_gemm_f16).
// gemm_tile (gemm_kernel16_tile, gemm_kernel_f32): the smaller macro tiles, for what 256 x 256 blocks leave over and for all
// fp32 products (v_mfma_f32_32x32x2_f32), whose 16 times slower multiplies any tile can feed.
// The MFMA computes the TRANSPOSED block (rows = n, columns = m); the epilogue stages blocks through LDS and stores whole
// rows, 16 bytes per lane.
// Measured on MI355X, M=N=K=8192 fp16 TN: 1.33-1.42 PFLOP/s by box on U(-1,1) operands, where the board is power-limited
// (the vendor library's kernel for this shape, also on 16x16x32 MFMAs: 1.55); fp32: 150 TFLOP/s.
#include <type_traits>

#include <mutex>

#include "fmha_common.h"
#include "gemm_choice.h"

namespace cfk {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int BM = 256, BN = 256;

// K-contiguous rows of PITCH bytes (128: two rows per 256-byte bank period; 64: four): 16 consecutive rows at one
// 16-byte chunk index must spread over all banks -> rows at the same place in the period get distinct XOR values
template <int PITCH>
__device__ __forceinline__ int swz_k(int row) { return PITCH == 128 ? (row >> 1) & 7 : (row >> 2) & 3; }

// B rows [k][n] of PITCH bytes read with ds_read_b64_tr_b16 in the 16x16x32 lane map: a 32-lane half of the wave touches rows 8g .. 8g+3
// of two k groups g x 32 contiguous bytes, which spread over the 256-byte bank period (of which 256/PITCH rows share one); bit 0 stays
// clear so that the 32 bytes stay contiguous
template <int PITCH>
__device__ __forceinline__ int swz_bn(int row) {
  if (PITCH % 256 == 0) return ((row & 3) | (((row >> 3) & 1) << 2)) << 1;
  if (PITCH % 128 == 0) return (((row >> 1) & 1) | (((row >> 3) & 1) << 1)) << 1;
  return ((row >> 3) & 1) << 1;
}

// beta * C + alpha * acc, the latter as rounded to fp32, rounded to fp32 once: left to itself the compiler rounds some elements of a row to fp16
// right away (v_fma_mixlo_f16) and others not, by kernel, and a result would depend on the tile that it lies in.
template <class T>
__device__ __forceinline__ float add_c(float x, float beta, T c) {
  x = __builtin_fmaf(beta, (float)c, x);
  asm("" : "+v"(x));
  return x;
}

// The fp16 kernel on 16x16x32 MFMAs (v_mfma_f32_16x16x32_f16).  8 waves, two per SIMD, in a 2 x 4 grid; a wave owns MB x NB blocks of
// 16 x 16 of C (8 x 4: 128 x 64 of a 256 x 256 macro tile).  Measured, 8192^3 TN, one session, 4 waves of 128 x 128: 1401 TFLOP/s on
// U(-1,1) operands against 1309 for the same kernel on 32x32x16 MFMAs; on constant operands 1837 against 2048 (LDS writes between the
// short multiplies hold the MFMA pipe up for about 20 cycles each).  On U(-1,1) operands this board is power-limited and the deeper,
// narrower MFMA moves half the accumulator bits per FLOP: a register-only loop sustains 1.90 PFLOP/s with it against 1.69 with 32x32x16.
// 8 waves read a half more from the LDS than 4 waves of 128 x 128, but with two on a SIMD one multiplies while the other waits for
// memory, which shows wherever the time is not all main loop (us, 4 -> 8 waves, one session, three sets of operands and results in turn):
// M=N=4096 with K=64 12.4 -> 10.8, K=192 and C 24.6 -> 20.4, K=1024 33.8 -> 32.5, K=4096 108.1 -> 105.5; two of 4096 x 2048 x 512 NN and C 31.6 ->
// 27.5; 8192^3 the same (816 and 820).  (The same tile by 8 waves in two groups half a step
// apart, copies straight into the LDS through a ring of five 32 KB slots: 812.7 beside 808.5, with K=192 and C 19.7; without those copies 691, so
// what is left at large K is the 64 KB that every 8.4 MFLOP take from L2.)
// Lane (c = lane % 16, g = lane / 16) holds, of an operand fragment, row c and contraction slots 8g .. 8g+7 (16 bytes), and of an
// accumulator block column c, rows 4g .. 4g+3.  The MFMA computes the transposed block (rows = n, columns = m), so a lane owns 4
// consecutive n of one row m of C.
//
// Pipeline: two LDS stages and one K tile in registers.  While tile kt multiplies out of stage kt % 2, the registers (tile kt+1, loaded a
// tile ago) are written to the other stage -- whose readers passed the barrier that opened this tile -- and refilled with tile kt+2, all
// before the tile's one barrier.  A run of LDS and memory instructions between two multiplies stalls the MFMA pipe, so a tile is laid
// out as slots of one multiply each (K-step major, then m block, then n block) with at most one piece of other work behind each, pinned
// in that order.  The n-side fragments of a K-step are live throughout it and double-buffered; the m-side fragments, needed for NB
// multiplies only, live in a ring of four and are read LOOK blocks ahead; a load is issued two staging pieces behind the store that frees
// its register (right behind it, it waits for that store to have read it).
template <int MB, int NB>
struct BlockCfg {
  static constexpr int BMT = 32 * MB, BNT = 64 * NB, S = MB * NB;
  static constexpr int A_PPW = MB / 2, CPT = MB / 2 + NB;   // 16-byte pieces per lane of an A tile, of both
  static constexpr int A_TILE = BMT * 128, STAGE = (BMT + BNT) * 128;
  static constexpr int LOOK = NB >= 4 ? 2 : 3;              // m-side fragments are read so many blocks ahead
  static constexpr int E_PITCH = NB * 64 + 16;
  static constexpr int LDS_BYTES = 2 * STAGE > 8 * 16 * E_PITCH ? 2 * STAGE : 8 * 16 * E_PITCH;
  static_assert(MB % 2 == 0 && LDS_BYTES <= 160 * 1024, "pieces, stages");
  static constexpr int LD_LAG = 2;
  // Per slot of a tile (two K-steps of S): the m-side fragment (its block, counted through both K-steps), the n-side fragment of K-step 1,
  // the staging piece to store and the one to load that lie behind its multiply, or -1.  From `barrier` on the slots carry the first
  // fragments of the next tile: every read of this tile's stage and every store of the next one's is in front of it.
  struct Slots {
    int m_frag[2 * S], n_frag[2 * S], store[2 * S], load[2 * S], barrier;
    bool fits;
  };
  static constexpr Slots slots() {
    Slots r{};
    bool used[2 * S] = {};
    for (int i = 0; i < 2 * S; ++i) r.m_frag[i] = r.n_frag[i] = r.store[i] = r.load[i] = -1;
    r.barrier = S + (MB - 2) * NB;
    r.fits = (2 * MB - 1 - LOOK) * NB < r.barrier && NB + LOOK <= 2 * NB;
    for (int x = 0; x < 2 * MB - LOOK; ++x) {
      r.m_frag[x * NB] = x + LOOK;
      used[x * NB] = true;
    }
    for (int j = 0; j < NB; ++j) {
      int i = j * (S - 2) / NB + NB / 2;
      while (used[i]) ++i;
      r.n_frag[i] = j;
      used[i] = true;
      r.fits = r.fits && i < S - 2;
    }
    for (int q = 0, last = 0; q < CPT + LD_LAG; ++q) {
      int i = q * S / CPT + 1;
      while (i < r.barrier && (used[i] || i <= last)) ++i;
      if (i >= r.barrier) {
        r.fits = false;
        break;
      }
      if (q < CPT) r.store[i] = q;
      if (q >= LD_LAG) r.load[i] = q - LD_LAG;
      used[i] = true;
      last = i;
    }
    return r;
  }
};

template <bool NN, int MB, int NB>
__device__ __forceinline__ void gemm_block(const _Float16 *__restrict__ A, const _Float16 *__restrict__ B, const _Float16 *__restrict__ Cin,
                                           _Float16 *__restrict__ D, int M, int N, int K, float alpha, float beta) {
  using T = _Float16;
  using C = BlockCfg<MB, NB>;
  constexpr int PITCH = 128, BK = PITCH / 2, S = C::S, CPT = C::CPT, A_PPW = C::A_PPW, A_TILE = C::A_TILE, STAGE = C::STAGE;
  constexpr int BPITCH = C::BNT * 2;   // NN: bytes of a k row of the B tile
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int wm = wave / 4, wn = wave % 4;

  // tile order: groups of 8 tile rows, column-major inside a group, so concurrently running workgroups share A and
  // B panels in L2; workgroup ids are first remapped so that each XCD owns a contiguous range of that order (the problems
  // of a batch one after the other)
  const int tiles_n = (N + C::BNT - 1) / C::BNT, tiles_m = (M + C::BMT - 1) / C::BMT;
  int t = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t batch = t / (tiles_m * tiles_n);  // packed strides M*K, N*K, M*N (reference: gemm.cu:519-521)
  const int batches = ((int)gridDim.x + tiles_m * tiles_n - 1) / (tiles_m * tiles_n);
  t -= (int)batch * tiles_m * tiles_n;
  constexpr int GROUP = 8;
  const int per_group = GROUP * tiles_n;
  const int grp = t / per_group;
  const int first_m = grp * GROUP;
  const int rows_in_group = tiles_m - first_m < GROUP ? tiles_m - first_m : GROUP;
  const int in_grp = t - grp * per_group;
  const int m_own = (first_m + in_grp % rows_in_group) * C::BMT, n_own = in_grp / rows_in_group * C::BNT;
  // a last tile that would reach beyond the edge lies against it instead, and leaves out what its neighbour stores
  const int m0 = m_own + C::BMT <= M ? m_own : M - C::BMT, n0 = n_own + C::BNT <= N ? n_own : N - C::BNT;

  A += batch * M * K;
  B += batch * N * K;
  D += batch * M * N;
  if (Cin) Cin += batch * M * N;
  const char *Ap = (const char *)(A + (int64_t)m0 * K);
  const char *Bp = NN ? (const char *)(B + n0) : (const char *)(B + (int64_t)n0 * K);

  // ---- global -> register -> LDS staging, 16 B per lane and piece.  Piece i of wave w covers the 8 tile rows from (8 i + w) * 8 on;
  // lane l owns LDS slot (row l / 8, chunk position l % 8) of the piece and fetches chunk position ^ swz(row) of that row: the
  // XOR swizzle is applied on the global side, LDS writes are linear.  (NN: the B tile is 64 k rows of BPITCH bytes, cut into
  // pieces of 1 KB.)  The pieces lie 64 rows apart, but one lane offset plus a scalar offset per piece is slower than a lane
  // offset for each: 8192^3 797.0 us against 787.5.  The loads are ordinary loads into registers
  // (compiler-tracked), issued a tile ahead of the ds_write that parks them in LDS.
  constexpr int KP = NN || A_PPW > NB ? A_PPW : NB;
  uint32_t goff_k[KP];
#pragma unroll
  for (int i = 0; i < KP; ++i) {
    const int row = (i * 8 + wave) * 8 + lane / 8;
    goff_k[i] = (uint32_t)row * (uint32_t)(K * 2) + (uint32_t)(((lane % 8) ^ swz_k<PITCH>(row)) * 16);
  }
  // (320 rows NN: registers for one lane offset of B only, which serves all pieces, 16 k rows apart, with a scalar offset)
  constexpr bool ONE_B = NN && MB > 8;
  static_assert(!ONE_B || BPITCH == 512, "pieces a multiple of 16 rows apart");
  constexpr int BPN = ONE_B ? 1 : NB;
  uint32_t goff_b[BPN];
  if constexpr (NN) {
#pragma unroll
    for (int i = 0; i < BPN; ++i) {
      constexpr int CPR = BPITCH / 16;
      const int idx = (i * 8 + wave) * 64 + lane, krow = idx / CPR;
      goff_b[i] = (uint32_t)krow * (uint32_t)(N * 2) + (uint32_t)(((idx % CPR) ^ swz_bn<BPITCH>(krow)) * 16);
    }
  }
  const uint32_t st_off = wave * 1024 + lane * 16;
  int4v stg[CPT];
  using Rsrc = __amdgpu_buffer_rsrc_t;
  auto tile_ptrs = [&](int kt, Rsrc &ga, Rsrc &gb) {
    const char *pa = Ap + (size_t)kt * PITCH;
    const char *pb = NN ? Bp + (size_t)kt * BK * (size_t)(N * 2) : Bp + (size_t)kt * PITCH;
    ga = __builtin_amdgcn_make_buffer_rsrc((void *)pa, 0, -1, 0x00020000);
    gb = __builtin_amdgcn_make_buffer_rsrc((void *)pb, 0, -1, 0x00020000);
  };
  auto load_piece = [&](Rsrc ga, Rsrc gb, int p) {
    u32x4 x;
    if (p < A_PPW) x = __builtin_amdgcn_raw_buffer_load_b128(ga, (int)goff_k[p], 0, 0);
    else if (NN) x = __builtin_amdgcn_raw_buffer_load_b128(gb, (int)goff_b[ONE_B ? 0 : p - A_PPW], ONE_B ? (int)(32u * (uint32_t)N * (uint32_t)(p - A_PPW)) : 0, 0);
    else x = __builtin_amdgcn_raw_buffer_load_b128(gb, (int)goff_k[p - A_PPW], 0, 0);
    stg[p] = __builtin_bit_cast(int4v, x);
  };
  auto store_piece = [&](int stage, int p) {
    char *dst = smem + stage * STAGE + st_off + (p < A_PPW ? p * 8192 : A_TILE + (p - A_PPW) * 8192);
    *(int4v *)dst = stg[p];
  };

  // ---- LDS read addresses.  K-step s: lane (c, g) needs bytes 64s + 16g .. +16 of its row (k = 32s + 8g .. +8).
  // swz_k<128> depends on the row within its group of 16 only, so blocks are immediates.
  int a_rd[2], b_rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    a_rd[s] = (wm * MB * 16 + c) * PITCH + (((4 * s + g) ^ swz_k<PITCH>(c)) * 16);
    b_rd[s] = A_TILE + (wn * NB * 16 + c) * PITCH + (((4 * s + g) ^ swz_k<PITCH>(c)) * 16);
  }
  // NN: the n-side operand via two ds_read_b64_tr_b16 from [k][n] rows: within its block of 16 lanes, lane L hands
  // the read the address of (k row L/4, columns 4(L%4) .. +3) and receives k rows 0..3 of column L; block g reads k
  // rows 8g .. 8g+3, the second read 4 further
  const int bk_row = 8 * g + (c >> 2);          // + 32 s (+ 4)
  const int cg = c & 3;
  int bt_rd[NB];
  if constexpr (NN) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int chunk = (wn * NB * 16 + 16 * nb) / 8 + (cg >> 1);
      bt_rd[nb] = A_TILE + bk_row * BPITCH + ((chunk ^ swz_bn<BPITCH>(bk_row)) * 16) + (cg & 1) * 8;
    }
  }

  f32x4 acc[MB][NB];  // [m block][n block]
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int k_tiles = K / BK;
  auto fetch_a = [&](const char *st, int s, int blk) -> half8 { return *(const half8 *)(st + a_rd[s] + blk * 16 * PITCH); };
  auto fetch_b = [&](const char *st, int s, int blk) -> half8 {
    if constexpr (!NN) {
      return *(const half8 *)(st + b_rd[s] + blk * 16 * PITCH);
    } else {
      union {
        struct { short4v lo, hi; } p;
        half8 h;
      } u;
      const char *bp = st + bt_rd[blk] + s * 32 * BPITCH;
      u.p.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(short4v, bp));
      u.p.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(short4v, bp + 4 * BPITCH));
      return u.h;
    }
  };
  constexpr typename C::Slots sl = C::slots();
  static_assert(sl.fits, "slot layout");
  // The multiplies are asm statements with in-place accumulators: the compiler's hazard recognizer does not see the
  // matrix-pipe write -> accumulate-read dependency between two of them, so the distance between two multiplies into
  // one accumulator is this layout's business.  Every accumulator block is used once per K-step: MB * NB multiplies
  // lie between two uses, each holding the pipe for the 4 passes of v_mfma_f32_16x16x32_f16; back-to-back
  // dependent MFMAs of this shape need 4 passes + 2 wait states.
  static_assert(S >= 8, "distance between two multiplies into one accumulator: at least the MFMA's passes plus its wait states");
  Rsrc ga, gb;
  tile_ptrs(0, ga, gb);
#pragma unroll
  for (int p = 0; p < CPT; ++p) load_piece(ga, gb, p);
#pragma unroll
  for (int p = 0; p < CPT; ++p) store_piece(0, p);
  tile_ptrs(k_tiles > 1 ? 1 : 0, ga, gb);
#pragma unroll
  for (int p = 0; p < CPT; ++p) load_piece(ga, gb, p);
  __syncthreads();
  half8 aop[4], bop[2][NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) bop[0][nb] = fetch_b(smem, 0, nb);
#pragma unroll
  for (int x = 0; x < C::LOOK; ++x) aop[x] = fetch_a(smem, 0, x);
  int stage = 0;
  for (int kt = 0; kt < k_tiles; ++kt) {
    const char *st = smem + stage * STAGE;
    const char *nx = smem + (stage ^ 1) * STAGE;
    const int nstage = stage ^ 1;
    tile_ptrs(kt + 2 < k_tiles ? kt + 2 : k_tiles - 1, ga, gb);  // clamped at the end: a surplus tile is loaded and dropped
#pragma unroll
    for (int i = 0; i < 2 * S; ++i) {
      // x: the m block, counted through both K-steps.  The n blocks are walked there and back, so that from one multiply to the next only
      // one operand changes: an operand that stays costs less power (register-only loops on U(-1,1) operands: 1893 TFLOP/s with one
      // operand changing, 1815 with both; 8192^3 819.0 -> 815.9 us, 8192 x 8192 x 4096 NN 436.4 -> 431.4).
      const int x = i / NB, nb = x & 1 ? NB - 1 - i % NB : i % NB, s2 = i / S, mb = x % MB;
      if (i == sl.barrier) __syncthreads();
      // written out so that the accumulator is updated in place: through the builtin the register allocator moves the small
      // accumulators between the two halves of the register file.  Nothing but these multiplies touches the accumulators inside the
      // loop, so no hazard is hidden from the compiler here.  (The compiler gives a wave 128 AGPRs: 32 blocks.)
      if (mb * NB + nb < 32) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[mb][nb]) : "v"(bop[s2][nb]), "v"(aop[x % 4]));
      else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc[mb][nb]) : "v"(bop[s2][nb]), "v"(aop[x % 4]));
      if (sl.m_frag[i] >= 0) aop[sl.m_frag[i] % 4] = fetch_a(st, sl.m_frag[i] / MB, sl.m_frag[i] % MB);
      if (sl.n_frag[i] >= 0) bop[1][sl.n_frag[i]] = fetch_b(st, 1, sl.n_frag[i]);
      if (i >= sl.barrier) {
        const int j = i - sl.barrier;   // n 0, m 0, n 1, m 1, .., then the rest of the n side
        if (j < 2 * C::LOOK && j % 2 == 1) aop[j / 2] = fetch_a(nx, 0, j / 2);
        else if (j < NB + C::LOOK) {
          const int n = j < 2 * C::LOOK ? j / 2 : j - C::LOOK;
          bop[0][n] = fetch_b(nx, 0, n);
        }
      }
      if (sl.store[i] >= 0) store_piece(nstage, sl.store[i]);
      if (sl.load[i] >= 0) load_piece(ga, gb, sl.load[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
    stage = nstage;
  }

  // the last multiplies have left the pipe before the epilogue reads their accumulators (the compiler does not see
  // the dependency through the asm statements)
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  // ---- epilogue: D = alpha * acc + beta * C in fp32, each row of blocks staged through the wave's own LDS region and stored as
  // whole rows, 16 bytes per lane, through the L2 to memory: a round of tiles writes as much as the L2s hold, and left there as dirty
  // lines it has to be written out before the operands of the next round find room.  us, left in the L2 / through it, where D is the same in
  // every call, and where three take turns: 8192 x 4096 x 320 38.2 / 31.4, 37.9 / 31.4; 4096 x 4096 x 512 20.6 / 19.3, the same; 7936 x 7936 x 320
  // 66.1 / 55.9, 62.6 / 59.7; 8192 x 8192 with K=320 73.8 / 60.2, 71.9 / 77.2, NN 68.9 / 61.2, 72.1 / 72.9, with K=512 84.1 / 76.9, 87.5 / 89.8.  (The last
  // are the largest: three D of 134 MB do not fit the 256 MB behind the L2s.  Past the caches they take 70.5, 70.6 with K=320 and 60.6, 60.1 with
  // K=192, where through the L2 they take 54.9, 77.0; 4096 x 8192 x 320 36.4, 36.3, where 32.5, 32.0.)
  constexpr int EPL = 8, LPR = NB * 2, CHUNKS = 16 * LPR;   // halves per lane and store, lanes per row
  constexpr int PASSES = (CHUNKS + 63) / 64;
  char *et = smem + wave * (16 * C::E_PITCH);
  const int el = fresh_lane();   // (no register is kept for it across the main loop: 320 rows NN have none)
  // Three forms, so that a call without C meets no wait for it.
  enum { NO_C, C_CACHED, C_STREAMED };
  // C is asked for in front of the first store, into the registers that the main loop has left: a load per store had its latency in every
  // pass (us: M=N=4096 K=192 20.1 -> 18.3; two of 4096 x 2048 x 512 NN 28.0 -> 26.4; 8192 x 8192 x 2048 286.0 -> 271.0).  Up to 256 rows all of it.
  // With 320 rows 160 accumulators leave no room for its 80 registers: five rows of blocks ahead of the one that is stored (5 or 6: the same;
  // all of it, through scratch memory: two of 4352 x 4096 x 192 50.2 -> 41.3, 5120 x 4096 x 512 36.5 -> 32.1, x 4096 138.5 -> 135.6).
  constexpr int C_AHEAD = MB > 8 ? 5 : MB;
  half8 cv[C_AHEAD][PASSES];
  const auto read_c = [&](auto form, int mb, int pass) __attribute__((always_inline)) {
    int idx = pass * 64 + el;
    int gm = m0 + (wm * MB + mb) * 16 + idx / LPR, gn = n0 + wn * NB * 16 + idx % LPR * EPL;
    if constexpr (C_AHEAD == MB) {
      // (asked for by the lanes that use it, behind a branch each: without, the compiler moves the first piece into the branch around its
      // store, behind the wait for the others, or, kept from that, calls of one round take longer: 4096 x 4096 x 192 17.0 -> 17.7)
      if ((CHUNKS % 64 != 0 && idx >= CHUNKS) || gm < m_own || gn < n_own) return;
    } else {
      // (by every lane, so that the compiler can count what is on its way: some line that is read anyway instead of what a neighbour stores)
      static_assert(CHUNKS % 64 == 0, "no lane beyond the row of blocks");
      gm = gm < m_own ? m_own : gm;
      gn = gn < n_own ? n_own : gn;
    }
    const half8 *p = (const half8 *)(Cin + (int64_t)gm * N + gn);
    cv[mb % C_AHEAD][pass] = form.value == C_STREAMED ? __builtin_nontemporal_load(p) : *p;
  };
  const auto epilogue = [&](auto form) __attribute__((always_inline)) {
    constexpr bool WITH_C = form.value != NO_C;
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the surplus tile, whose registers are used anew (asked for a tile ago: it is there)
    if constexpr (WITH_C) {
#pragma unroll
      for (int mb = 0; mb < C_AHEAD; ++mb)
#pragma unroll
        for (int pass = 0; pass < PASSES; ++pass) read_c(form, mb, pass);
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) *(f32x4 *)(et + (el & 15) * C::E_PITCH + (nb * 16 + 4 * (el >> 4)) * 4) = acc[mb][nb];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int pass = 0; pass < PASSES; ++pass) {
        half8 cm{};
        if constexpr (WITH_C) {
          cm = cv[mb % C_AHEAD][pass];
          if (mb + C_AHEAD < MB) read_c(form, mb + C_AHEAD, pass);
        }
        const int idx = pass * 64 + el, row = idx / LPR, col = idx % LPR * EPL;
        const int gm = m0 + (wm * MB + mb) * 16 + row, gn = n0 + wn * NB * 16 + col;
        if ((CHUNKS % 64 != 0 && idx >= CHUNKS) || gm < m_own || gn < n_own) continue;
        float v[EPL];
#pragma unroll
        for (int q = 0; q < EPL / 4; ++q) {
          const f32x4 x = *(const f32x4 *)(et + row * C::E_PITCH + (col + 4 * q) * 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) v[4 * q + j] = alpha * x[j];
        }
        if constexpr (WITH_C) {
#pragma unroll
          for (int j = 0; j < EPL; ++j) v[j] = add_c(v[j], beta, cm[j]);
        }
        half8 o;
#pragma unroll
        for (int j = 0; j < EPL; ++j) o[j] = (T)v[j];
        store16_through(D + (int64_t)gm * N + gn, o);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the region is rewritten by the next row of blocks
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  };
  // From 64 MB on C is read past the caches, where a C of that size is not anyway and its lines would take the place of others; smaller
  // ones often lie in the 256 MB behind the L2s, written by the call before.  us, past the caches / through them, K=512, three sets of
  // operands in turn: 33 MB 27.6 / 25.1, 50 MB 43.2 / 36.6, 67 MB 54.5 / 55.3, 101 MB 74.5 / 81.1, 134 MB 101.5 / 123.3.  (64 MB are two rounds of
  // 256 x 256 blocks.  A call of more than that whose last ones run as small tiles has two whole rounds here, and one of less has not.)
  const bool big_c = (int64_t)M * N * batches * 2 >= (64 << 20);
  if (Cin == nullptr || beta == 0.f) {
    epilogue(std::integral_constant<int, NO_C>{});
    return;
  }
  if (big_c) {
    asm volatile("; C past the caches");   // (or the compiler makes one branch of the two)
    epilogue(std::integral_constant<int, C_STREAMED>{});
    asm volatile("; C past the caches");
    return;
  }
  epilogue(std::integral_constant<int, C_CACHED>{});
}

template <bool NN, int NB>   // 256 rows
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_kernel16(const _Float16 *__restrict__ A, const _Float16 *__restrict__ B, const _Float16 *__restrict__ Cin,
              _Float16 *__restrict__ D, int M, int N, int K, float alpha, float beta) {
  gemm_block<NN, 8, NB>(A, B, Cin, D, M, N, K, alpha, beta);
}
template <bool NN, int MB, int NB>   // 32 MB rows
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_kernel16_rows(const _Float16 *__restrict__ A, const _Float16 *__restrict__ B, const _Float16 *__restrict__ Cin,
                   _Float16 *__restrict__ D, int M, int N, int K, float alpha, float beta) {
  gemm_block<NN, MB, NB>(A, B, Cin, D, M, N, K, alpha, beta);
}

// ---- Smaller macro tiles (which of them a call takes: gemm_choice.h).
// 8 waves (two per SIMD) or 4: WM x WN of them share a tile of K, each with TM x TN of C, and KG such groups take the
// 128-byte deep K tiles in turn; their partial sums meet in the LDS.  Splitting the waves over K instead of over C keeps
// the wave tile large -- an operand fragment feeds TM/16 or TN/16 multiplies -- where the macro tile is small, and puts KG
// times the bytes in flight.  Tiles go global -> LDS by copy instructions (1 KB a wave, whole 128-byte row pieces: a
// lane-per-row load of operand fragments straight into registers runs at 16 bytes per clock and CU, a quarter of this)
// through ST stages, waited for by count.
// FB: block edge of the MFMA (fp32: 32 or 16).  SETS (fp32): accumulators of a block that its multiplies take in turn, added up at the end: as
// many partial sums as SETS groups over K would make, without the groups.
// SHARE: the two groups take the two K-steps of one K tile instead of a K tile each.  All waves fill a stage, half the size, so twice as
// many of them are in flight, for a barrier every K-step (which tiles: gemm_choice.h; M=N=2048 K=4096 TN 39.4 -> 36.9 us).
template <class T_, bool NN_, int WM_, int WN_, int TM_, int TN_, int KG_, int ST_, int FB_ = sizeof(T_) == 2 ? 16 : 32, int SETS_ = 1, bool SHARE_ = false>
struct TileCfg {
  using T = T_;
  static constexpr bool NN = NN_;
  static constexpr int ES = sizeof(T), WM = WM_, WN = WN_, TM = TM_, TN = TN_, KG = KG_, ST = ST_;
  static constexpr int BMT = WM * TM, BNT = WN * TN, SUB = (BM / BMT) * (BN / BNT);  // tiles of a 256 x 256 block
  static constexpr int WPG = WM * WN, NW = WPG * KG, THREADS = NW * 64;
  static constexpr int BK = 128 / ES;
  static constexpr bool SHARE = SHARE_;
  static constexpr int A_BYTES = BMT * 128, G_BYTES = (BMT + BNT) * 128, STAGE = (SHARE ? 1 : KG) * G_BYTES;
  static constexpr int CW = SHARE ? NW : WPG;                                 // waves that fill a group's part of a stage
  static constexpr int A_PIECES = BMT / 8, PIECES = (BMT + BNT) / 8, PPW = (PIECES + CW - 1) / CW;   // 1 KB copies of a stage, per wave
  static constexpr int E_PITCH = BNT * 4 + 16, E_BYTES = KG * BMT * E_PITCH;  // epilogue: fp32 sums, rows padded
  static constexpr int LDS_BYTES = ST * STAGE > E_BYTES ? ST * STAGE : E_BYTES;
  static constexpr int SETS = SETS_;
  static constexpr int FB = FB_;                                              // block edge of the MFMA
  static constexpr bool EDGES = BM % BMT || BN % BNT;                          // tiles of M x N instead of a 256 x 256 block's
  static constexpr int RPP = THREADS / (BNT * ES / 16), PASSES = (BMT + RPP - 1) / RPP;   // epilogue: rows per pass
  // what piece i of a wave copies: a part of A, a part of B, or the one or the other by wave, some of them a part that another wave copies too
  static constexpr int A_PART = 0, B_PART = 1, BY_WAVE = 2;
  static constexpr int part(int i) { return (i + 1) * CW <= A_PIECES ? A_PART : i * CW >= A_PIECES && (i + 1) * CW <= PIECES ? B_PART : BY_WAVE; }
  static_assert(A_PIECES * 8 == BMT && PIECES * 8 == BMT + BNT && (SHARE || PIECES % CW == 0), "whole 1 KB copies");
  static_assert(!SHARE || (ES == 2 && KG == 2), "two groups, two K-steps");
  static_assert(LDS_BYTES <= 160 * 1024 && ST >= 2, "stages");
};

// AHEAD: there is a C, and all of it that a lane needs is asked for before the sums meet, not pass by pass (us: 2048 x 2048 x 512 NN 11.1 ->
// 9.4, 2048 x 4096 x 512 15.4 -> 13.0, fp32 4096 x 4096 x 512 140.2 -> 131.5; in front of the main loop 10.3, 15.0 and 133.4).  For tiles
// of several passes, in kernels of their own: with both epilogues in one kernel a call without C takes 1 % longer.
template <class C, bool AHEAD = false>
__device__ __forceinline__ void gemm_tile(const typename C::T *__restrict__ A, const typename C::T *__restrict__ B,
                                          const typename C::T *__restrict__ Cin, typename C::T *__restrict__ D, int M, int N, int K,
                                          float alpha, float beta, int block0, int wg, int wgs) {
  using T = typename C::T;
  constexpr bool F16 = C::ES == 2, NN = C::NN;
  constexpr int ES = C::ES, FB = C::FB, MB = C::TM / FB, NB = C::TN / FB;
  constexpr int BPITCH = C::BNT * 2;               // NN: bytes of a k row of the B tile
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / C::WPG, wi = wave % C::WPG, wm = wi / C::WN, wn = wi % C::WN;
  const int c = lane % FB, g = lane / FB;

  // tile order: the 256 x 256 blocks in the order of the kernels above (from block0 on, the batch's problems one after the
  // other), the tiles of a block next to each other; EDGES: the tiles themselves in that order, and a last one that would reach beyond the edge
  // lies against it instead and leaves out what its neighbour stores
  const int tiles_n = C::EDGES ? (N + C::BNT - 1) / C::BNT : N / BN, tiles_m = C::EDGES ? (M + C::BMT - 1) / C::BMT : M / BM;
  const int w = xcd_remap(wg, wgs);
  int t = C::EDGES ? w : block0 + w / C::SUB;
  const int s_idx = C::EDGES ? 0 : w % C::SUB;
  const int64_t batch = t / (tiles_m * tiles_n);
  t -= (int)batch * tiles_m * tiles_n;
  constexpr int GROUP = 8;
  const int per_group = GROUP * tiles_n;
  const int grp = t / per_group;
  const int first_m = grp * GROUP;
  const int rows_in_group = tiles_m - first_m < GROUP ? tiles_m - first_m : GROUP;
  const int in_grp = t - grp * per_group;
  const int m_own = (first_m + in_grp % rows_in_group) * (C::EDGES ? C::BMT : BM) + (C::EDGES ? 0 : s_idx / (BN / C::BNT) * C::BMT);
  const int n_own = in_grp / rows_in_group * (C::EDGES ? C::BNT : BN) + (C::EDGES ? 0 : s_idx % (BN / C::BNT) * C::BNT);
  const int m0 = !C::EDGES || m_own + C::BMT <= M ? m_own : M - C::BMT, n0 = !C::EDGES || n_own + C::BNT <= N ? n_own : N - C::BNT;
  A += batch * M * K;
  B += batch * N * K;
  D += batch * M * N;
  if (Cin) Cin += batch * M * N;
  const char *Ap = (const char *)(A + (int64_t)m0 * K);
  const char *Bp = NN ? (const char *)(B + n0) : (const char *)(B + (int64_t)n0 * K);

  // ---- copies: group kg fills its own part of a stage; piece i of a wave is 8 rows of A or B (NN: 1 KB of k rows of B)
  const int ci = C::SHARE ? wave : wi;
  const uint32_t lds_base = (uint32_t)(uintptr_t)LDS_PTR(char, smem);
  const uint32_t lds_wave = lds_base + (C::SHARE ? 0 : kg * C::G_BYTES) + ci * 1024;
  uint32_t goff[C::PPW];
  bool of_a[C::PPW], again[C::PPW];
#pragma unroll
  for (int i = 0; i < C::PPW; ++i) {
    int q = i * C::CW + ci;
    again[i] = C::part(i) == C::BY_WAVE && q >= C::PIECES;
    if (again[i]) q -= C::PIECES;
    of_a[i] = C::part(i) == C::BY_WAVE ? q < C::A_PIECES : C::part(i) == C::A_PART;
    const int p = of_a[i] ? q : q - C::A_PIECES;
    if (!NN || of_a[i]) {
      const int row = p * 8 + lane / 8;
      goff[i] = (uint32_t)row * (uint32_t)(K * ES) + (uint32_t)(((lane % 8) ^ swz_k<128>(row)) * 16);
    } else {
      constexpr int CPR = BPITCH / 16;
      const int idx = p * 64 + lane, krow = idx / CPR;
      goff[i] = (uint32_t)krow * (uint32_t)(N * 2) + (uint32_t)(((idx % CPR) ^ swz_bn<BPITCH>(krow)) * 16);
    }
  }
  const int chunks = K / C::BK, n_st = C::SHARE ? chunks : (chunks + C::KG - 1) / C::KG;
  auto load_piece = [&](int j, int slot, int i) __attribute__((always_inline)) {
    int ch = C::SHARE ? j : j * C::KG + kg;
    ch = ch < chunks ? ch : chunks - 1;   // (a group without a tile in the last turn copies one it does not multiply)
    const char *gp = of_a[i] ? Ap + (size_t)ch * 128 : NN ? Bp + (size_t)ch * ((size_t)C::BK * N * 2) : Bp + (size_t)ch * 128;
    lds_dma16(gp, goff[i], lds_wave + slot * C::STAGE, (uint32_t)(i * C::CW - (again[i] ? C::PIECES : 0)) * 1024u);
  };
  auto load_stage = [&](int j, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::PPW; ++i) load_piece(j, slot, i);
  };

  // ---- LDS read addresses, relative to the group's part of a stage (see gemm_kernel16; fp32: lane (c, g) needs bytes
  // 32s + 16g .. +16 of its row, k = 8s + 4g .. +4, used one element per 32x32x2 MFMA: which contraction slot means which k
  // is free as long as A and B agree)
  constexpr int KS = C::SHARE ? 1 : FB == 16 ? 2 : 4;   // K-steps (one 16-byte fragment per operand block) of a tile
  constexpr int FPS = FB == 16 ? 4 : 2;            // fragments of a row in a K-step
  int a_rd[KS], b_rd[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int ks = C::SHARE ? kg : s;
    a_rd[s] = (wm * C::TM + c) * 128 + (((FPS * ks + g) ^ swz_k<128>(c)) * 16);
    b_rd[s] = C::A_BYTES + (wn * C::TN + c) * 128 + (((FPS * ks + g) ^ swz_k<128>(c)) * 16);
  }
  int bt_rd[NB];
  if constexpr (NN) {
    const int bk_row = 8 * g + (c >> 2), cg = c & 3;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int chunk = (wn * C::TN + 16 * nb) / 8 + (cg >> 1);
      bt_rd[nb] = C::A_BYTES + (C::SHARE ? kg * 32 * BPITCH : 0) + bk_row * BPITCH + ((chunk ^ swz_bn<BPITCH>(bk_row)) * 16) + (cg & 1) * 8;
    }
  }
  using Frag = std::conditional_t<F16, half8, f32x4>;
  using Acc = std::conditional_t<FB == 16, f32x4, f32x16>;
  constexpr int AV = FB == 16 ? 4 : 16;
  Acc accs[C::SETS][MB][NB];
  auto &acc = accs[0];
#pragma unroll
  for (int x = 0; x < C::SETS; ++x)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < AV; ++v) accs[x][mb][nb][v] = 0.f;

  Frag af[2][MB], bf[2][NB];
  // fragment i of K-step s of the stage in `slot`, in the order the multiplies want them: B 0, A 0, B 1 .., A 1 ..
  constexpr int FRAGS = MB + NB;
  auto fetch_piece = [&](int slot, int s, int i, Frag (&fa)[MB], Frag (&fb)[NB]) __attribute__((always_inline)) {
    const char *st = smem + slot * C::STAGE + (C::SHARE ? 0 : kg * C::G_BYTES);
    if (i == 1 || i > NB) {
      const int mb = i == 1 ? 0 : i - NB;
      fa[mb] = *(const Frag *)(st + a_rd[s] + mb * FB * 128);
      return;
    }
    const int nb = i == 0 ? 0 : i - 1;
    if constexpr (!NN) {
      fb[nb] = *(const Frag *)(st + b_rd[s] + nb * FB * 128);
    } else {
      union {
        struct { short4v lo, hi; } p;
        half8 h;
      } u;
      const char *bp = st + bt_rd[nb] + s * 32 * BPITCH;
      u.p.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(short4v, bp));
      u.p.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(short4v, bp + 4 * BPITCH));
      fb[nb] = u.h;
    }
  };
  auto multiply_block = [&](int mb, int nb, const Frag (&fa)[MB], const Frag (&fb)[NB]) __attribute__((always_inline)) {
    if constexpr (F16) {
      acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[nb], fa[mb], acc[mb][nb], 0, 0, 0);
    } else if constexpr (FB == 16) {
#pragma unroll
      for (int e = 0; e < 4; ++e) accs[e % C::SETS][mb][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[nb][e], fa[mb][e], accs[e % C::SETS][mb][nb], 0, 0, 0);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) accs[e % C::SETS][mb][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[nb][e], fa[mb][e], accs[e % C::SETS][mb][nb], 0, 0, 0);
    }
  };
  // The multiplies of one K-step with the other work (fragment reads of the next, copies).  Where all waves work on one tile
  // of K it is spread between them, order pinned: a run of LDS reads in front of the multiplies leaves the matrix cores idle
  // while all eight waves queue for the LDS (256 x 128, M=4096 N=2048 K=4096: 60.5 us against 62.7).  With several groups
  // the compiler's order is the faster one (128 x 128, M=N=2048 K=8192: 68.7 us against 71.9).
  auto multiply_with = [&](const Frag (&fa)[MB], const Frag (&fb)[NB], auto n_pieces, auto &&piece) __attribute__((always_inline)) {
    constexpr int P = decltype(n_pieces)::value, NS = MB * NB;
    if constexpr (C::KG > 1) {
#pragma unroll
      for (int k = 0; k < P; ++k) piece(k);
    }
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      multiply_block(i / NB, i % NB, fa, fb);
      if constexpr (C::KG == 1) {
#pragma unroll
        for (int k = 0; k < P; ++k)
          if (k * NS / (P ? P : 1) == i) piece(k);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // Waits until all but this wave's copies of the `behind` newest stages have landed and its LDS reads have returned, and
  // meets the others: then everybody's copies have, and a slot whose reads lie in front of the barrier is free.
  static_assert(C::ST <= 8 && (C::ST - 1) * C::PPW < 64, "copies that can be waited for by count");
  auto arrive = [&](int behind) __attribute__((always_inline)) {
    if (C::ST >= 8 && behind >= 6) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::ST >= 8 ? 6 * C::PPW : 0) : "memory");
    else if (C::ST >= 7 && behind >= 5) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::ST >= 7 ? 5 * C::PPW : 0) : "memory");
    else if (C::ST >= 6 && behind >= 4) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::ST >= 6 ? 4 * C::PPW : 0) : "memory");
    else if (C::ST >= 5 && behind >= 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(3 * C::PPW) : "memory");
    else if (C::ST >= 4 && behind >= 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * C::PPW) : "memory");
    else if (C::ST >= 3 && behind >= 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::PPW) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  // Fragments are read one K-step ahead, across the barrier too, so that the reads of one step lie beside the multiplies
  // of the one before.
#pragma unroll
  for (int j = 0; j < C::ST; ++j)
    if (j < n_st) load_stage(j, j);
  if (n_st >= C::ST) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((C::ST - 1) * C::PPW) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int i = 0; i < FRAGS; ++i) fetch_piece(0, 0, i, af[0], bf[0]);
  using std::integral_constant;
  int slot = 0;
  if constexpr (C::SHARE) {
    auto step = [&](auto parity, int j) __attribute__((always_inline)) {   // one K-step of a stage: the fragments change places every stage
      constexpr int P = decltype(parity)::value;
      const int next = slot == C::ST - 1 ? 0 : slot + 1, behind = n_st - 2 - j;
      arrive(behind < C::ST - 2 ? behind : C::ST - 2);
      const bool more = j + C::ST < n_st;
      multiply_with(af[P], bf[P], integral_constant<int, FRAGS + C::PPW>{}, [&](int k) __attribute__((always_inline)) {
        if (k < FRAGS) fetch_piece(next, 0, k, af[P ^ 1], bf[P ^ 1]);
        else if (more) load_piece(j + C::ST, slot, k - FRAGS);
      });
      slot = next;
    };
    int j = 0;
    for (; j + 2 < n_st; j += 2) {
      step(integral_constant<int, 0>{}, j);
      step(integral_constant<int, 1>{}, j + 1);
    }
    if (j + 1 < n_st) step(integral_constant<int, 0>{}, j);
    if (n_st % 2 == 0) multiply_with(af[1], bf[1], integral_constant<int, 0>{}, [](int) {});
    else multiply_with(af[0], bf[0], integral_constant<int, 0>{}, [](int) {});
  } else {
    for (int j = 0; j + 1 < n_st; ++j) {
      const int next = slot == C::ST - 1 ? 0 : slot + 1;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (s + 1 < KS) {
          multiply_with(af[s & 1], bf[s & 1], integral_constant<int, FRAGS>{},
                        [&](int k) __attribute__((always_inline)) { fetch_piece(slot, s + 1, k, af[(s + 1) & 1], bf[(s + 1) & 1]); });
        } else {
          const int behind = n_st - 2 - j;
          arrive(behind < C::ST - 2 ? behind : C::ST - 2);
          const bool more = j + C::ST < n_st;
          multiply_with(af[s & 1], bf[s & 1], integral_constant<int, FRAGS + C::PPW>{}, [&](int k) __attribute__((always_inline)) {
            if (k < FRAGS) fetch_piece(next, 0, k, af[0], bf[0]);
            else if (more) load_piece(j + C::ST, slot, k - FRAGS);
          });
        }
      }
      slot = next;
    }
    if (C::KG == 1 || (n_st - 1) * C::KG + kg < chunks) {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (s + 1 < KS)
          multiply_with(af[s & 1], bf[s & 1], integral_constant<int, FRAGS>{},
                        [&](int k) __attribute__((always_inline)) { fetch_piece(slot, s + 1, k, af[(s + 1) & 1], bf[(s + 1) & 1]); });
        else multiply_with(af[s & 1], bf[s & 1], integral_constant<int, 0>{}, [](int) {});
      }
    }
  }

#pragma unroll
  for (int x = 1; x < C::SETS; x *= 2)
#pragma unroll
    for (int y = 0; y < C::SETS; y += 2 * x)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) accs[y][mb][nb] += accs[y + x][mb][nb];
  // ---- epilogue: every group leaves its fp32 sums in the LDS as rows of C; they are added up, scaled and rounded once on
  // the way out, 16 bytes per lane of whole tile rows
  constexpr int PASSES = C::PASSES;
  std::conditional_t<F16, half8, f32x4> c_ahead[AHEAD ? PASSES : 1];
  if constexpr (AHEAD) {
    constexpr int EPL = 16 / ES, LPR = C::BNT / EPL, RPP = C::RPP;
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
      int row = pass * RPP + tid / LPR;
      if (C::BMT % RPP && row >= C::BMT) row = C::BMT - 1;   // (not stored)
      c_ahead[pass] = *(const decltype(&c_ahead[0]))(Cin + (int64_t)(m0 + row) * N + n0 + (tid % LPR) * EPL);
    }
  }
  __syncthreads();
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < AV / 4; ++i) {
        f32x4 v4;
#pragma unroll
        for (int x = 0; x < 4; ++x) v4[x] = acc[mb][nb][4 * i + x];
        // lane (m = c, g): n = 4 g .. +3 of a 16-wide block, 8 i + 4 g .. +3 of a 32-wide one
        *(f32x4 *)(smem + (kg * C::BMT + wm * C::TM + mb * FB + c) * C::E_PITCH + (wn * C::TN + nb * FB + 8 * i + 4 * g) * 4) = v4;
      }
  __syncthreads();
  constexpr int EPL = 16 / ES, LPR = C::BNT / EPL, RPP = C::RPP;
  using OutV = std::conditional_t<F16, half8, f32x4>;
  const bool with_c = AHEAD || (PASSES == 1 && Cin != nullptr && beta != 0.f);   // (several passes meet a C in the AHEAD kernels only)
  const int e_row = tid / LPR, e_col = (tid % LPR) * EPL;
  static_assert(C::BMT % RPP == 0 || RPP > C::BMT || C::EDGES, "whole passes");
#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) {
    const int row = pass * RPP + e_row;
    if (C::BMT % RPP && row >= C::BMT) break;
    if (C::EDGES && (e_row >= RPP || m0 + row < m_own || n0 + e_col < n_own)) continue;
    const int64_t off = (int64_t)(m0 + row) * N + n0 + e_col;
    float v[EPL];
#pragma unroll
    for (int q = 0; q < EPL / 4; ++q) {
      f32x4 x = *(const f32x4 *)(smem + row * C::E_PITCH + (e_col + 4 * q) * 4);
#pragma unroll
      for (int k = 1; k < C::KG; ++k) x += *(const f32x4 *)(smem + (k * C::BMT + row) * C::E_PITCH + (e_col + 4 * q) * 4);
#pragma unroll
      for (int x2 = 0; x2 < 4; ++x2) v[4 * q + x2] = alpha * x[x2];
    }
    if (with_c) {
      const OutV cv = AHEAD ? c_ahead[AHEAD ? pass : 0] : *(const OutV *)(Cin + off);
#pragma unroll
      for (int x = 0; x < EPL; ++x) v[x] = add_c(v[x], beta, cv[x]);
    }
    OutV o;
#pragma unroll
    for (int x = 0; x < EPL; ++x) o[x] = (T)v[x];
    // (through the L2 as in gemm_block, but for the smallest tiles, whose calls end with these stores: M=N=K=1024 NN 6.69 -> 6.79 us, three
    // fp32 problems of 1024 x 768 x 1536 61.7 -> 62.0; 2048 x 4096 x 512 12.2 -> 11.2)
    if constexpr (PASSES > 1) store16_through(D + off, o);
    else *(OutV *)(D + off) = o;
  }
}

// The macro tiles built: <operand type, NN, waves along m and n, rows and columns per wave, wave groups over K, stages>.
// Measured and not built (fp16, TN): 128 x 128 by 8 waves on one K tile, 4 stages, 67.8 us against 68.7 at M=N=2048 K=8192 but
// 90 against 73.5 for NN; 64 x 64 by four K groups of two waves, 31.9 us against 27.7 at M=N=1024 K=8192 (two stages, half
// the bytes in flight).
template <bool NN, int ROWS, int COLS> struct HTile;
template <bool NN> struct HTile<NN, 256, 128> : TileCfg<_Float16, NN, 4, 2, 64, 64, 1, 3> {};
template <bool NN> struct HTile<NN, 192, 128> : TileCfg<_Float16, NN, 4, 2, 48, 64, 1, 3> {};
template <bool NN> struct HTile<NN, 128, 192> : TileCfg<_Float16, NN, 2, 4, 64, 48, 1, 3> {};
template <bool NN> struct HTile<NN, 96, 128> : TileCfg<_Float16, NN, 2, 2, 48, 64, 2, 2> {};
template <bool NN> struct HTile<NN, 96, 96> : TileCfg<_Float16, NN, 2, 2, 48, 48, 2, 3> {};
template <bool NN> struct HTile<NN, 96, 64> : TileCfg<_Float16, NN, 2, 2, 48, 32, 2, 4> {};
template <bool NN> struct HTile<NN, 64, 32> : TileCfg<_Float16, NN, 2, 1, 32, 32, 4, 3> {};
template <bool NN> struct HTile<NN, 128, 128> : TileCfg<_Float16, NN, 2, 2, 64, 64, 2, 2> {};
template <bool NN> struct HTile<NN, 128, 64> : TileCfg<_Float16, NN, 2, 2, 64, 32, 2, 3> {};
template <bool NN> struct HTile<NN, 64, 64> : TileCfg<_Float16, NN, 2, 2, 32, 32, 2, 4> {};
template <bool NN> struct HTile<NN, 32, 32> : TileCfg<_Float16, NN, 1, 1, 32, 32, 4, 4> {};
// ... and those whose two groups share K tiles
template <bool NN, int ROWS> struct HShared;
template <bool NN> struct HShared<NN, 128> : TileCfg<_Float16, NN, 2, 2, 64, 64, 2, 5, 16, 1, true> {};
template <bool NN> struct HShared<NN, 96> : TileCfg<_Float16, NN, 2, 2, 48, 64, 2, 5, 16, 1, true> {};
template <int EDGE> struct FTile;
// ... and the two tiles of gemm_kernel_f32_mix, 32 KB of LDS each: 4 waves of 32 x 32 and of 16 x 16
template <int SETS> struct FMix64 : TileCfg<float, false, 2, 2, 32, 32, 1, 2, 32, SETS> {};
template <int SETS> struct FMix32 : TileCfg<float, false, 2, 2, 16, 16, 1, 4, 16, SETS> {};
template <> struct FTile<128> : TileCfg<float, false, 2, 2, 64, 64, 1, 2> {};
template <> struct FTile<64> : TileCfg<float, false, 2, 2, 32, 32, 2, 2> {};
template <> struct FTile<32> : TileCfg<float, false, 1, 1, 32, 32, 4, 2> {};

template <bool NN, int ROWS, int COLS>
__global__ void __launch_bounds__((HTile<NN, ROWS, COLS>::THREADS))
gemm_kernel16_tile(const _Float16 *__restrict__ A, const _Float16 *__restrict__ B, const _Float16 *__restrict__ Cin,
                   _Float16 *__restrict__ D, int M, int N, int K, float alpha, float beta, int block0) {
  gemm_tile<HTile<NN, ROWS, COLS>>(A, B, Cin, D, M, N, K, alpha, beta, block0, blockIdx.x, gridDim.x);
}

template <bool NN, int ROWS, int COLS>
__global__ void __launch_bounds__((HTile<NN, ROWS, COLS>::THREADS))
gemm_kernel16_tile_c(const _Float16 *__restrict__ A, const _Float16 *__restrict__ B, const _Float16 *__restrict__ Cin,
                     _Float16 *__restrict__ D, int M, int N, int K, float alpha, float beta, int block0) {
  gemm_tile<HTile<NN, ROWS, COLS>, true>(A, B, Cin, D, M, N, K, alpha, beta, block0, blockIdx.x, gridDim.x);
}

// ROWS x 128
template <bool NN, int ROWS>
__global__ void __launch_bounds__((HShared<NN, ROWS>::THREADS))
gemm_kernel16_shared(const _Float16 *__restrict__ A, const _Float16 *__restrict__ B, const _Float16 *__restrict__ Cin,
                     _Float16 *__restrict__ D, int M, int N, int K, float alpha, float beta, int block0) {
  gemm_tile<HShared<NN, ROWS>>(A, B, Cin, D, M, N, K, alpha, beta, block0, blockIdx.x, gridDim.x);
}

template <bool NN, int ROWS>
__global__ void __launch_bounds__((HShared<NN, ROWS>::THREADS))
gemm_kernel16_shared_c(const _Float16 *__restrict__ A, const _Float16 *__restrict__ B, const _Float16 *__restrict__ Cin,
                       _Float16 *__restrict__ D, int M, int N, int K, float alpha, float beta, int block0) {
  gemm_tile<HShared<NN, ROWS>, true>(A, B, Cin, D, M, N, K, alpha, beta, block0, blockIdx.x, gridDim.x);
}

template <int EDGE>
__global__ void __launch_bounds__(FTile<EDGE>::THREADS)
gemm_kernel_f32_c(const float *__restrict__ A, const float *__restrict__ B, const float *__restrict__ Cin, float *__restrict__ D,
                  int M, int N, int K, float alpha, float beta, int block0) {
  gemm_tile<FTile<EDGE>, true>(A, B, Cin, D, M, N, K, alpha, beta, block0, blockIdx.x, gridDim.x);
}

template <int EDGE>
__global__ void __launch_bounds__(FTile<EDGE>::THREADS)
gemm_kernel_f32(const float *__restrict__ A, const float *__restrict__ B, const float *__restrict__ Cin, float *__restrict__ D,
                int M, int N, int K, float alpha, float beta, int block0) {
  gemm_tile<FTile<EDGE>>(A, B, Cin, D, M, N, K, alpha, beta, block0, blockIdx.x, gridDim.x);
}

// Tiles of 64 x 64 for the first blocks64 blocks and of 32 x 32 for the others, in one launch of workgroups of 4 waves, five of which share a
// CU.  What bounds fp32 products is how evenly the multiplies go round the CUs and what of a workgroup's life is not multiplies (first
// copies, sums through the LDS, stores: some 4 us): in whole rounds of one tile size three problems of 1024 x 768 x 1536 took nine 32 x 32
// tiles on each CU, two at a time, 63.1 us -- now two of 64 x 64 and one of 32 x 32 beside each other 56.6; without the small ones, where some CUs
// have three of 64 x 64, 73.4; the small ones first 57.2; three stages, so that three share a CU, 55.9, but 2304 x 768 x 3072 101.1 instead of 87.0.
template <int SETS, bool AHEAD>
__device__ __forceinline__ void gemm_f32_mix(const float *__restrict__ A, const float *__restrict__ B, const float *__restrict__ Cin, float *__restrict__ D,
                                             int M, int N, int K, float alpha, float beta, int blocks64) {
  const int n64 = blocks64 * FMix64<SETS>::SUB, wg = blockIdx.x;
  if (wg < n64) gemm_tile<FMix64<SETS>, AHEAD>(A, B, Cin, D, M, N, K, alpha, beta, 0, wg, n64);
  else gemm_tile<FMix32<SETS>>(A, B, Cin, D, M, N, K, alpha, beta, blocks64, wg - n64, (int)gridDim.x - n64);
}
template <int SETS>
__global__ void __launch_bounds__(256)
gemm_kernel_f32_mix(const float *__restrict__ A, const float *__restrict__ B, const float *__restrict__ Cin, float *__restrict__ D, int M, int N,
                    int K, float alpha, float beta, int blocks64) {
  gemm_f32_mix<SETS, false>(A, B, Cin, D, M, N, K, alpha, beta, blocks64);
}
template <int SETS>
__global__ void __launch_bounds__(256)
gemm_kernel_f32_mix_c(const float *__restrict__ A, const float *__restrict__ B, const float *__restrict__ Cin, float *__restrict__ D, int M, int N,
                      int K, float alpha, float beta, int blocks64) {
  gemm_f32_mix<SETS, true>(A, B, Cin, D, M, N, K, alpha, beta, blocks64);
}

// one-time set-up of a kernel (its dynamic-LDS limit), thread-safe and callable ahead of any launch
template <auto Kern, int Lds>
hipError_t prepare_kernel() {
  static std::once_flag once;
  static hipError_t status = hipSuccess;
  std::call_once(once, [] { status = hipFuncSetAttribute((const void *)Kern, hipFuncAttributeMaxDynamicSharedMemorySize, Lds); });
  return status;
}

template <bool NN, int MB, int NB>
constexpr auto block_kernel() {
  if constexpr (MB == 8) return &gemm_kernel16<NN, NB>;
  else return &gemm_kernel16_rows<NN, MB, NB>;
}
// the macro tiles 0 .. tiles-1 of the batch
template <bool NN, int MB, int NB>
hipError_t launch_blocks(const GemmArgs &g, hipStream_t s, int tiles) {
  using C = BlockCfg<MB, NB>;
  constexpr auto kern = block_kernel<NN, MB, NB>();
  const hipError_t e = prepare_kernel<kern, C::LDS_BYTES>();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(512), C::LDS_BYTES, s, (const _Float16 *)g.A, (const _Float16 *)g.B, (const _Float16 *)g.C,
                     (_Float16 *)g.D, g.M, g.N, g.K, g.alpha, g.beta);
  return hipGetLastError();
}

// tiles of configuration C by kernel Kern, of the 256 x 256 blocks from block0 on (EDGES: all that there are)
template <class C, auto Kern>
hipError_t launch_tiles(const GemmArgs &g, hipStream_t s, int block0, int tiles) {
  const hipError_t e = prepare_kernel<Kern, C::LDS_BYTES>();
  if (e != hipSuccess) return e;
  using T = typename C::T;
  hipLaunchKernelGGL(Kern, dim3(tiles), dim3(C::THREADS), C::LDS_BYTES, s, (const T *)g.A, (const T *)g.B, (const T *)g.C,
                     (T *)g.D, g.M, g.N, g.K, g.alpha, g.beta, block0);
  return hipGetLastError();
}
template <bool NN, int ROWS, int COLS>
hipError_t launch_edge16(const GemmArgs &g, hipStream_t s, int tiles, int block0 = 0) {
  using C = HTile<NN, ROWS, COLS>;
  if constexpr (C::PASSES > 1) {
    if (g.C && g.beta != 0.f) return launch_tiles<C, gemm_kernel16_tile_c<NN, ROWS, COLS>>(g, s, block0, tiles);
  }
  return launch_tiles<C, gemm_kernel16_tile<NN, ROWS, COLS>>(g, s, block0, tiles);
}
template <bool NN, int ROWS, int COLS>
hipError_t launch_tiles16(const GemmArgs &g, hipStream_t s, int block0, int blocks) {
  return launch_edge16<NN, ROWS, COLS>(g, s, blocks * HTile<NN, ROWS, COLS>::SUB, block0);
}
template <bool NN, int ROWS>
hipError_t launch_shared(const GemmArgs &g, hipStream_t s, int tiles, int block0) {
  using C = HShared<NN, ROWS>;
  if (g.C && g.beta != 0.f) return launch_tiles<C, gemm_kernel16_shared_c<NN, ROWS>>(g, s, block0, tiles);
  return launch_tiles<C, gemm_kernel16_shared<NN, ROWS>>(g, s, block0, tiles);
}
template <int EDGE>
hipError_t launch_tiles32(const GemmArgs &g, hipStream_t s, int blocks) {
  using C = FTile<EDGE>;
  if constexpr (C::PASSES > 1) {
    if (g.C && g.beta != 0.f) return launch_tiles<C, gemm_kernel_f32_c<EDGE>>(g, s, 0, blocks * C::SUB);
  }
  return launch_tiles<C, gemm_kernel_f32<EDGE>>(g, s, 0, blocks * C::SUB);
}

// What the choice names (gemm_choice.h).
template <bool NN>
hipError_t launch_f16(const GemmArgs &g, hipStream_t s) {
  const GemmChoice c = choose_gemm_f16(g.M, g.N, g.K, g.batch);
  hipError_t e = hipSuccess;
  if (c.rows == 96) return c.cols == 64 ? launch_edge16<NN, 96, 64>(g, s, c.tiles) : c.cols == 96 ? launch_edge16<NN, 96, 96>(g, s, c.tiles) : g.K >= kSharedFrom ? launch_shared<NN, 96>(g, s, c.tiles, 0) : launch_edge16<NN, 96, 128>(g, s, c.tiles);
  if (c.rows == 128) return launch_edge16<NN, 128, 192>(g, s, c.tiles);
  if (c.rows == 192 && c.cols == 128) return launch_edge16<NN, 192, 128>(g, s, c.tiles);
  if (c.rows == 256 && c.cols == 256) e = launch_blocks<NN, 8, 4>(g, s, c.tiles);
  else if (c.rows == 256) e = launch_blocks<NN, 8, 3>(g, s, c.tiles);
  else if (c.rows == 320) e = launch_blocks<NN, 10, 4>(g, s, c.tiles);
  else if (c.cols == 256) e = launch_blocks<NN, 6, 4>(g, s, c.tiles);
  else if (c.rows == 192) e = launch_blocks<NN, 6, 3>(g, s, c.tiles);
  if (e != hipSuccess || !c.tail_blocks) return e;
  const int from = c.tiles, left = c.tail_blocks;
  if (c.tail_rows == 32) return launch_tiles16<NN, 32, 32>(g, s, from, left);
  if (c.tail_rows == 64 && c.tail_cols == 32) return launch_tiles16<NN, 64, 32>(g, s, from, left);
  if (c.tail_rows == 64) return launch_tiles16<NN, 64, 64>(g, s, from, left);
  if (c.tail_rows == 256) return launch_tiles16<NN, 256, 128>(g, s, from, left);
  if (c.tail_cols == 64) return launch_tiles16<NN, 128, 64>(g, s, from, left);
  return g.K >= kSharedFrom ? launch_shared<NN, 128>(g, s, left * HShared<NN, 128>::SUB, from) : launch_tiles16<NN, 128, 128>(g, s, from, left);
}

template <int SETS> constexpr int kMixLds = FMix64<SETS>::LDS_BYTES > FMix32<SETS>::LDS_BYTES ? FMix64<SETS>::LDS_BYTES : FMix32<SETS>::LDS_BYTES;
template <int SETS>
hipError_t launch_mix(const GemmArgs &g, hipStream_t s, int blocks, int blocks64) {
  const bool with_c = g.C && g.beta != 0.f;
  const hipError_t e = with_c ? prepare_kernel<gemm_kernel_f32_mix_c<SETS>, kMixLds<SETS>>() : prepare_kernel<gemm_kernel_f32_mix<SETS>, kMixLds<SETS>>();
  if (e != hipSuccess) return e;
  const int tiles = blocks64 * FMix64<SETS>::SUB + (blocks - blocks64) * FMix32<SETS>::SUB;
  hipLaunchKernelGGL(with_c ? &gemm_kernel_f32_mix_c<SETS> : &gemm_kernel_f32_mix<SETS>, dim3(tiles), dim3(256), kMixLds<SETS>, s, (const float *)g.A, (const float *)g.B,
                     (const float *)g.C, (float *)g.D, g.M, g.N, g.K, g.alpha, g.beta, blocks64);
  return hipGetLastError();
}

hipError_t launch_f32(const GemmArgs &g, hipStream_t s) {
  const int blocks = (g.M / BM) * (g.N / BN) * g.batch, edge = choose_gemm_f32(blocks);
  const GemmMix mix = choose_gemm_f32_mix(blocks, g.K);
  if (mix.sums == 1) return launch_mix<1>(g, s, blocks, mix.blocks64);
  if (mix.sums == 2) return launch_mix<2>(g, s, blocks, mix.blocks64);
  if (mix.sums == 4) return launch_mix<4>(g, s, blocks, mix.blocks64);
  if (edge == 128) return launch_tiles32<128>(g, s, blocks);
  return edge == 64 ? launch_tiles32<64>(g, s, blocks) : launch_tiles32<32>(g, s, blocks);
}

template <bool NN, int ROWS, int COLS>
hipError_t prepare_tile() {
  constexpr int lds = HTile<NN, ROWS, COLS>::LDS_BYTES;
  const hipError_t e = prepare_kernel<gemm_kernel16_tile<NN, ROWS, COLS>, lds>();
  return e != hipSuccess ? e : prepare_kernel<gemm_kernel16_tile_c<NN, ROWS, COLS>, lds>();
}
template <bool NN>
hipError_t prepare_f16() {
  const hipError_t e[] = {prepare_kernel<block_kernel<NN, 8, 4>(), BlockCfg<8, 4>::LDS_BYTES>(),
                          prepare_kernel<block_kernel<NN, 8, 3>(), BlockCfg<8, 3>::LDS_BYTES>(),
                          prepare_kernel<block_kernel<NN, 6, 4>(), BlockCfg<6, 4>::LDS_BYTES>(),
                          prepare_kernel<block_kernel<NN, 6, 3>(), BlockCfg<6, 3>::LDS_BYTES>(),
                          prepare_kernel<block_kernel<NN, 10, 4>(), BlockCfg<10, 4>::LDS_BYTES>(),
                          prepare_tile<NN, 256, 128>(), prepare_tile<NN, 128, 128>(), prepare_tile<NN, 128, 64>(),
                          prepare_tile<NN, 192, 128>(), prepare_tile<NN, 128, 192>(), prepare_tile<NN, 96, 128>(), prepare_tile<NN, 96, 96>(), prepare_tile<NN, 96, 64>(),
                          prepare_kernel<gemm_kernel16_shared<NN, 128>, HShared<NN, 128>::LDS_BYTES>(), prepare_kernel<gemm_kernel16_shared_c<NN, 128>, HShared<NN, 128>::LDS_BYTES>(),
                          prepare_kernel<gemm_kernel16_shared<NN, 96>, HShared<NN, 96>::LDS_BYTES>(), prepare_kernel<gemm_kernel16_shared_c<NN, 96>, HShared<NN, 96>::LDS_BYTES>(),
                          prepare_kernel<gemm_kernel16_tile<NN, 64, 32>, HTile<NN, 64, 32>::LDS_BYTES>(),
                          prepare_kernel<gemm_kernel16_tile<NN, 64, 64>, HTile<NN, 64, 64>::LDS_BYTES>(),
                          prepare_kernel<gemm_kernel16_tile<NN, 32, 32>, HTile<NN, 32, 32>::LDS_BYTES>()};
  for (hipError_t x : e)
    if (x != hipSuccess) return x;
  return hipSuccess;
}

}  // namespace

hipError_t launch_gemm(const GemmArgs &g, hipStream_t s) {
  if (g.f32) return g.layout == 0 ? launch_f32(g, s) : hipErrorNotSupported;
  return g.layout == 0 ? launch_f16<false>(g, s) : launch_f16<true>(g, s);
}

hipError_t prepare_gemm() {
  hipError_t e = prepare_f16<false>();
  if (e == hipSuccess) e = prepare_f16<true>();
  if (e == hipSuccess) e = prepare_kernel<gemm_kernel_f32<128>, FTile<128>::LDS_BYTES>();
  if (e == hipSuccess) e = prepare_kernel<gemm_kernel_f32<64>, FTile<64>::LDS_BYTES>();
  if (e == hipSuccess) e = prepare_kernel<gemm_kernel_f32<32>, FTile<32>::LDS_BYTES>();
  if (e == hipSuccess) e = prepare_kernel<gemm_kernel_f32_c<128>, FTile<128>::LDS_BYTES>();
  if (e == hipSuccess) e = prepare_kernel<gemm_kernel_f32_c<64>, FTile<64>::LDS_BYTES>();
  const hipError_t mix[] = {prepare_kernel<gemm_kernel_f32_mix<1>, kMixLds<1>>(), prepare_kernel<gemm_kernel_f32_mix_c<1>, kMixLds<1>>(),
                            prepare_kernel<gemm_kernel_f32_mix<2>, kMixLds<2>>(), prepare_kernel<gemm_kernel_f32_mix_c<2>, kMixLds<2>>(),
                            prepare_kernel<gemm_kernel_f32_mix<4>, kMixLds<4>>(), prepare_kernel<gemm_kernel_f32_mix_c<4>, kMixLds<4>>()};
  for (hipError_t x : mix)
    if (e == hipSuccess) e = x;
  return e;
}

}  // namespace cfk
