// Which kernel a call's bf16 linears run, and the height of the tiled GEMMs'
// tiles: host rules on sizes alone, free of HIP so that they can be checked
// without a GPU.
#pragma once
#include <stdint.h>

namespace w4a16 {

// A shared-MLP linear (M rows, N output columns, K deep) as the tiled GEMM
// instead of the stream (k_linear_bf16, its weights once per 64 rows).  A
// launch of few tiles takes a tile's time, about 20 us at K = 2816, whatever
// its size; the stream's grows with the 64-row passes and the weights of each.

// The stream on rows in fragment order.  Two passes were never slower; from
// the third on the line is passes times weights.  The FFN block (H = 2816),
// streamed / tiled, in us, at 128, 129, 193..208, 257..288 rows: Im = 512
// 158/173, 164/175, 194/202, 265/259; 1056 163/181, 169/182, 207/209, 240/236;
// 1600 167/183, 201/207, 218/212, 253/238; 2112 176/189, 214/214, 229/217,
// 273/244; 4096 199/208, 225/210, 276/235, 331/266; 12288 300/299, 360/322.
inline bool linear_tiled_frag(int64_t M, int64_t N, int64_t K) {
  return M > 128 && ((M + 63) / 64 - 2) * (N * K) > 4600000;
}

// The stream on row-major rows (16 x 64 bytes a load): tiled earlier.  Im =
// 1056 at 96 / 128 / 160 rows 170/182, 218/219, 228/223; 1600 at 81 / 96
// 178/179, 185/183; 2112 at 65 / 81 / 300 181/187, 187/186, 331/246; 4096 at
// 65 211/204.
inline bool linear_tiled_rows(int64_t M, int64_t N, int64_t K) {
  return (M > 64 && M * N * K > 420000000) || linear_tiled_frag(M, N, K);
}

// The block's two linears (H x Im) stream fragment-order rows: from 17 rows
// on, one row tile gains nothing; `fits`: the padded rows fit in the place
// they are held.
inline bool ffn_fragment_rows(int64_t M, int64_t H, int64_t Im, bool fits, bool tiles_supported) {
  return M > 16 && fits && !(tiles_supported && linear_tiled_frag(M, Im, H));
}

// The tile height, in 32-row blocks, of a launch whose tiles (256 weight rows
// each) are all alike and run one per CU: the time is the rounds of tiles times
// a tile's, cost[blocks - 1].
inline int cheapest_blocks(int64_t M, int64_t wrows, int cus, int max_blocks, const int* cost) {
  const int64_t n_nt = (wrows + 255) / 256;
  int best = 0;
  int64_t least = 0;
  for (int mb = 1; mb <= max_blocks; ++mb) {
    const int64_t tiles = (M + 32 * mb - 1) / (32 * mb) * n_nt;
    const int64_t c = (tiles + cus - 1) / cus * cost[mb - 1];
    if (best == 0 || c < least) {
      best = mb;
      least = c;
    }
  }
  return best;
}

// Dense bf16 GEMM: a tile's time is close to (blocks + 1), its MFMAs and a
// stage's weights, barrier and waits whatever the height.  The FFN block (Im =
// 2112, flat routing) with 1 .. 5 blocks: 287 / 265 / 270 / 283 / 288 us at 512
// rows (2 picked), 399 / 354 / 336 / 346 / 353 at 1024 (3), 572 / 521 / 480 /
// 490 / 468 at 2048 (gate/up 5, down 3: 464).
constexpr int kGemmMaxBlocks = 5;
inline int gemm_bf16_blocks(int64_t M, int64_t wrows, int cus) {
  constexpr int cost[kGemmMaxBlocks] = {2, 3, 4, 5, 6};
  return cheapest_blocks(M, wrows, cus, kGemmMaxBlocks, cost);
}

// The decode streamer's shape for K: k tiles (128 wide) per wavefront in a row
// and wavefronts per sum.  It is also what a sum is: wavefront w's fp32 chain
// over the tiles w tpw .. w tpw + tpw - 1, and those a multiple of ksplit tpw
// behind them, the wavefronts' chains added in order.
struct DecodeShape {
  int tpw;
  int ksplit;
};
inline DecodeShape decode_shape(int64_t K) {
  const int64_t ntiles = (K + 127) / 128;
  if (ntiles <= 2) return {2, 1};
  if (ntiles <= 4) return {4, 1};
  if (ntiles <= 6) return {6, 1};   // down, K = 704: 6 tiles, 4 column groups
  if (ntiles <= 8) return {2, 4};
  if (ntiles <= 16) return {4, 4};
  return {6, 4};                    // gate_up, K = 2816: 22 tiles over 4 wavefronts
}
// whether a chain's tiles lie apart (more than ksplit tpw tiles)
inline bool decode_ranges_interleave(int64_t K) {
  const DecodeShape s = decode_shape(K);
  return (K + 127) / 128 > s.tpw * s.ksplit;
}

// Linear4Bit tiles of at most max_blocks: one round of tiles of 1 .. 6 blocks
// measured 31, 37, 44, 52, 61, 72 us at K = 2816, 11.0 .. 25.4 at K = 704 (a
// stage's barrier and waits dominate few blocks).
constexpr int kLinearW4MaxBlocks = 6;
inline int linear_w4_blocks(int64_t M, int64_t N, int cus, int max_blocks) {
  constexpr int cost[kLinearW4MaxBlocks] = {31, 37, 44, 52, 61, 72};
  return cheapest_blocks(M, N, cus, max_blocks, cost);
}

}  // namespace w4a16
