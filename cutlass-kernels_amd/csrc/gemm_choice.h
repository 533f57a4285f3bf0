// Which macro tiles a product of cfk_gemm runs in.  Host code without HIP: gemm.hip launches what stands here, and
// tests/test_gemm_choice.py asks it which kernels a shape takes.
#pragma once

namespace cfk {

constexpr int kCus = 256;
constexpr int kSharedFrom = 1088;   // K from which tiles of 96 x 128 and 128 x 128 run with groups that share K tiles (below)

// A first launch of `tiles` macro tiles of rows x cols, and a second one of `tail_blocks` blocks of 256 x 256, the last ones of the batch, in
// tiles of tail_rows x tail_cols; either may be missing (0).
struct GemmChoice {
  int rows, cols, tiles, tail_rows, tail_cols, tail_blocks;
};

// 256 x 256 blocks run in whole rounds of the CUs, one to a CU; the blocks of a last round that at most half fills the CUs are cut into the
// smallest tiles that still go round the CUs once.  Such a round takes, at K=4096 (1024), of one of 256 x 256 blocks, 105 (32.4) us: 256 x 128
// 0.58 (0.61), 128 x 128 0.38 (0.41), 128 x 64 0.22 (0.26), 64 x 64 0.14 (0.19), 32 x 32 0.08 (0.17).
// Behind whole rounds the tiles are a second launch.  Time relative to whole blocks alone, batches of 256 x 256 problems, with and without
// C, TN and NN (range of the four; three sets of operands and results in turn), behind one and behind three rounds:
//   K=64    8 left 0.81..0.91, 0.95..0.97    40 0.90, 0.98..1.00        72 0.94..0.95, 0.98..1.02  104 0.96..0.98, 1.01..1.03  128 0.96..1.00, 1.03..1.04
//   K=256          0.83..0.88, 0.94..0.96       0.91, 0.96..0.99           0.94..0.97, 0.98..1.01      0.95..1.01, 0.99..1.01      1.05..1.11, 1.05..1.08
//   K=512          0.82..0.87, 0.92..0.93       0.91..0.97, 0.94..0.98     0.94..0.97, 0.96..0.99      0.96..1.01, 0.96..0.98      0.97..1.01, 0.97..1.00
//   K=2048         0.80..0.83, 0.91..0.92       0.91..0.95, 0.95..0.98     0.95..0.99, 0.98..1.01      0.97..1.01, 0.98..1.04      1.00..1.03, 0.99..1.06
inline GemmChoice gemm_blocks_and_tiles(int blocks) {
  const int left = blocks % kCus, whole = left > kCus / 2 ? blocks : blocks - left;
  GemmChoice c{};
  if (whole) c.rows = c.cols = 256, c.tiles = whole;
  if (whole == blocks) return c;
  c.tail_blocks = left;
  if (left * 64 <= kCus) c.tail_rows = c.tail_cols = 32;
  else if (left * 16 <= kCus) c.tail_rows = c.tail_cols = 64;
  else if (left * 8 <= kCus) c.tail_rows = 128, c.tail_cols = 64;
  else if (left * 4 <= kCus) c.tail_rows = c.tail_cols = 128;
  else c.tail_rows = 256, c.tail_cols = 128;
  return c;
}

// fp16, up to half a round of 256 x 256 blocks: one round of tiles, the smaller the better.  Between the sizes that divide a block lie others (the
// last ones against the edges of M x N), taken from 512 of K on where the CUs hold them all at once.  Time relative to the next larger
// size that divides a block, K=512 to 8192, TN and NN, with and without C, 500 drawn products: 64 x 32 0.89 to 0.93 (5 to 8 blocks), 96 x 64 0.90 to
// 0.95 (17 to 24), 96 x 96 0.69 to 0.78, 96 x 128 0.92 to 0.94 (33 to 48), 128 x 192 and 192 x 128 0.89 to 0.95 (65 to 96).  us: 768 x 3072 x 4800 NN with C
// 41.6 -> 29.7; M=N=1536 K=2048 TN 19.7 -> 13.6; 512 x 1024 x 2240 8.4 -> 6.8; 3840 x 1024 x 2048 21.3 -> 20.1.  (Measured and not built: 128 x 96 0.94 to 0.99, 64 x 96 0.95 to 0.99 of the larger size.)
// What bounds the smaller ones: 3.2 to 3.4 us of launch, first stage, sums and stores, and then the bytes that a CU gets from the L2, of 154 a nanosecond that the copies
// could bring.  M=N=1024 NN in tiles of 64 x 64, us at K=512, 1024, 2048, 4096: 4.5, 5.9, 8.3, 15.7 on one set of operands, 4.6, 6.3, 9.4, 15.7 on three in turn:
// 105 and 85 bytes a nanosecond between 1024 and 2048, where eight turns and more come out of the L2 or the memory behind it, 71 and 83 between 2048 and 4096.
// The two with 128 columns, of which two K tiles a turn leave room for one turn ahead in the LDS, waited for them.  With both groups at one K tile and four ahead,
// K=1088 to 2048, 185 products of 33 to 64 blocks, operands changing from call to call 0.85 to 0.96 of the time (0.918 in the geometric mean); the same operands
// again and again 0.84 to 0.99, but 1.02 to 1.10 in 18 of 145 whose share of the operands lies in each XCD's L2 from the call before (up to about 3.9 of its 4 MB:
// 1024 x 2304 x 1280 TN 9.8 -> 10.7 us), where there is no way to hide and the barrier every K-step is left.  A line drawn by that size gave
// those back and cost the same products 0.06 to 0.12 on operands that change.  1.05 to 1.10 at K=512 to 768.  The other tiles have three
// or four turns in the LDS and lose by it: 128 x 64 0.99 to 1.09, 96 x 96 1.01 to 1.03, 64 x 64 and 96 x 64 1.03 to 1.21.
inline GemmChoice choose_gemm_f16_round(int M, int N, int K, int batch, int blocks) {
  const auto tiles = [&](int r, int c) { return (int)((long long)((M + r - 1) / r) * ((N + c - 1) / c) * batch); };
  const auto in = [&](int from, int to) { return blocks >= from && blocks <= to; };
  if (K >= 512) {
    if (in(5, 8)) return GemmChoice{0, 0, 0, 64, 32, blocks};
    if (in(17, 24) && tiles(96, 64) <= kCus) return GemmChoice{96, 64, tiles(96, 64), 0, 0, 0};
    if (in(33, 48) && tiles(96, 96) <= kCus) return GemmChoice{96, 96, tiles(96, 96), 0, 0, 0};
    if (in(33, 48) && tiles(96, 128) <= kCus) return GemmChoice{96, 128, tiles(96, 128), 0, 0, 0};
    if (in(65, 96)) {
      const int wide = tiles(128, 192), high = tiles(192, 128);
      if (wide <= high && wide <= kCus) return GemmChoice{128, 192, wide, 0, 0, 0};
      if (high <= kCus) return GemmChoice{192, 128, high, 0, 0, 0};
    }
  }
  return gemm_blocks_and_tiles(blocks);
}

// fp16.  From half a round of 256 x 256 blocks on: rounds of other macro tiles where these waste less of the chip.  Times in rounds of 256 x 256
// tiles; one of which a share f is filled takes (1 + f)/2, because the idle CUs leave the others their power.
// Measured, every tile for 842 drawn products of 129 to 1040 blocks, TN and NN, with and without C, D the same and three in turn; a full round,
// relative to 256 x 256: 192 x 256 0.77 at K=192 to 0.82 from 768 on, with C 0.78 to 0.82; 192 x 192 0.66 to 0.69; 320 x 256 1.12 to 1.23, with C
// 1.19 to 1.21; 256 x 192 0.89 up to K=1536 and 0.84 from 3072 on, with C 0.86 and 0.85.  (The 192-column tiles write rows of 96 bytes, parts of lines.)
// The choice is 1.001 of the best tile for each in the geometric mean, and 0.950 of 256 x 256 blocks with small tiles behind them; worst 1.04 of
// those (5632 x 3840 x 2880 NN: 121 -> 126).  With 0.792 for 256 x 192 at every K and 0.622 for 192 x 192, 30 of them went to these two at 1.05 of the
// time that they take now: 7 x 1024 x 5120 x 640 60 -> 76 us, 6 x 512 x 7168 x 1024 53 -> 61, 4 x 768 x 6144 x 1856 NN with C 79 -> 84.
// us, blocks and small tiles / the choice: 5120 x 4096 x 4096 TN 149 / 128 and with C 158 / 135 (256 tiles of 320 x 256); M=N=3072 K=512 15.3 / 13.7 (256 of
// 192 x 192).  Not built: 320 x 192 and 192 x 320 (103.6 against 102.7 and 100.7 against 102.0 for 240 blocks), 256 x 128 and less by the block kernel
// (64.3 against 61.8 for a round of 256 x 128).
inline GemmChoice choose_gemm_f16(int M, int N, int K, int batch) {
  const int blocks = (M / 256) * (N / 256) * batch;
  if (blocks <= kCus / 2) return choose_gemm_f16_round(M, N, K, batch, blocks);
  GemmChoice choice = gemm_blocks_and_tiles(blocks);
  const auto rounds = [](long long tiles) {
    const int part = (int)(tiles % kCus);
    return (double)(tiles / kCus) + (part ? 0.5 + 0.5 * part / kCus : 0.0);
  };
  double best = rounds(blocks);
  if (choice.tail_blocks) {
    const int sub = 256 / choice.tail_rows * (256 / choice.tail_cols);
    const double full = sub == 64 ? 0.06 : sub == 16 ? 0.14 : sub == 8 ? 0.22 : sub == 4 ? 0.40 : 0.55;
    best = blocks / kCus + full * (0.6 + 0.4 * choice.tail_blocks * sub / kCus) + 0.03;
  }
  const auto offer = [&](int r, int c, double round) {
    // (a tile against the edge needs a whole one; 32-bit byte offsets within a tile's rows)
    if (M < r || N < c || (long long)r * K * 2 >= (1LL << 32)) return;
    const long long n = (long long)((M + r - 1) / r) * ((N + c - 1) / c) * batch;
    const double t = round * rounds(n);
    if (t < best) best = t, choice = GemmChoice{r, c, (int)n, 0, 0, 0};
  };
  offer(192, 256, 0.772);
  offer(256, 192, 0.85 + 40.0 / K);
  offer(192, 192, 0.65);
  offer(320, 256, 1.192);
  return choice;
}

// fp32, the edge of the square tiles: the multiplies bound every tile size, so what counts is how full the last round of the CUs is: the tile
// whose rounds, at their measured times relative to 128 x 128 (66 us per 1024 of K), add up to least.  Three problems of M=1024 N=768 K=1536
// (576 tiles of 64 x 64, 2304 of 32 x 32) 64.6 us by 32 x 32 against 76.3 and 97; M=N=5120 K=4096 1532 us by 64 x 64 against
// 1615 and 1717; M=N=K=8192 7.31 ms by 128 x 128.  (256 x 256 blocks, 4 waves of 128 x 128 with registers between global memory
// and LDS: 345 us, 1989 us and 7.89 ms for the three.)
inline int choose_gemm_f32(int blocks) {
  const auto rounds = [&](int sub) { return (double)(((long long)blocks * sub + kCus - 1) / kCus); };
  const double t128 = rounds(4), t64 = 0.267 * rounds(16), t32 = 0.072 * rounds(64);
  if (t128 <= t64 && t128 <= t32) return 128;
  return t64 <= t32 ? 64 : 32;
}

// ... or, where sums > 0, tiles of 64 x 64 for the first blocks64 blocks, whole rounds of the CUs, and of 32 x 32 for the others beside them in one
// launch (gemm_kernel_f32_mix).  An element is added up from as many partial sums as in the tile above, `sums`: with fewer it would be
// further off, with more the time is up to 4 % longer (1, 2 and 4 at 3072 x 3328 x 384: 0.954, 0.978 and 0.995 of it).
// Time relative to the tile above, one problem, K=256 to 4096: 17 to 28 blocks 0.78 to 0.98, 33 to 44 0.70 to 0.96, 49 to 60 0.81 to 0.98, 66 to 168
// 0.84 to 0.99; with more than 12 blocks behind whole rounds, which would be a whole round themselves, 1.05 to 1.15; whole rounds
// alone 1.01 up to 64 blocks and 0.98 to 0.99 beyond; 124 of two rounds of 64 blocks 1.00, 120 0.99, 561 of nine 1.025.  9 to 12 blocks in 32 x 32 tiles
// alone: 0.92 at K=256, 0.95 at 768, 1.00 at 2048; fewer 1.03 to 1.28.
struct GemmMix {
  int blocks64, sums;
};
inline GemmMix choose_gemm_f32_mix(int blocks, int K) {
  const int edge = choose_gemm_f32(blocks), left = blocks % 16, sums = edge == 128 ? 1 : edge == 64 ? 2 : 4;
  if (blocks <= 16) return GemmMix{0, blocks >= 9 && blocks <= 12 && K <= 1024 ? 4 : 0};
  if (left > 12 || (left == 0 && blocks <= 64)) return GemmMix{0, 0};
  if (edge == 128 && blocks > 61 * ((blocks + 63) / 64)) return GemmMix{0, 0};   // (its rounds nearly full)
  return GemmMix{blocks - left, sums};
}

}  // namespace cfk
