// Host rules of the GEMM dispatch: which tiles a product runs on.
#pragma once
#include <stdint.h>

namespace ghip {

// Grids of at most this many 128 x 128 tiles run 64 x 64 tiles of the register-staged
// core instead (any layout): four times the workgroups, each with four k-tiles of
// loads in flight.  Graph-replayed, us, 128 x 128 DMA core / 64 x 64: bf16 [256,512,256]
// 5.8 / 4.3, [512,512,512] 8.0 / 5.4, [1024,1024,1024] 12.6 / 8.1, [1024,2048,1024] (128
// tiles) 12.8 / 11.3, but 14.2 / 14.8 at 144 tiles and 14.6 / 18.8 at 256; fp32, bound
// by a CU's MFMA rate, [256,512,256] 20.9 / 8.2, [1024,1024,256] 21.8 / 9.4,
// [1536,2048,512] (192 tiles) 40.2 / 32.4, 270 / 277 at 224 tiles.
constexpr bool gemm_small_tiles(int64_t batch, int64_t M, int64_t N, int es) {
  return batch * ((M + 127) / 128) * ((N + 127) / 128) <= (es == 4 ? 192 : 128);
}
// fp32 grids of at most 128 tiles of 64 x 64: 32 x 32 tiles with the contraction spread
// over a workgroup's waves.  us, 64 x 64 / 32 x 32: [256,512,256] 8.1 / 4.9, [256,256,512]
// 13.0 / 6.5, [512,1024,1024] (128 tiles) 23.7 / 16.7, but 24.7 / 27.0 at 256.
constexpr bool gemm_f32_tiny(int64_t batch, int64_t M, int64_t N) {
  return batch * ((M + 63) / 64) * ((N + 63) / 64) <= 128;
}
// 16-bit products for 256 x 128 tiles (gemm_bf16_body4h): grids that are one round of
// them but more than one 128 x 128 tile per CU, with a contraction long enough to pay for
// a prologue and an epilogue that no second workgroup hides.  Graph-replayed, us, 128 x
// 128 core / 256 x 128: [4096,2048,8192] 127 / 108, [2304,2304,4096] 55.3 / 48.0,
// [2048,3072,4096] 55 / 49, [4096,2048,2048] 35.0 / 33.0, but [2,2048,2048,1024] 20.4 /
// 20.7; at 256 tiles of 128 x 128 [2048,2048,2048] 27.5 / 28.5; where 256 x 256 tiles are
// more than 128 their cores win ([4096,4096,4096] 97 / 112).  Ragged tiles pay for the
// masks of their loads, more so on an MN-contiguous A: [3080,2056,4096] 60.2 / 56.2, A
// MN-contiguous 65.0 / 64.0 ([2056,2184,4096] 58.6 / 60.6), [3080,2056,2048] 33.5 / 34.6.
constexpr bool gemm_half_whole(int64_t M, int64_t N, int64_t K) { return M % 256 == 0 && N % 128 == 0 && K % 64 == 0; }
constexpr bool gemm_half_tiles(int64_t batch, int64_t M, int64_t N, int64_t K, bool a_k) {
  const int64_t t128 = batch * ((M + 127) / 128) * ((N + 127) / 128);
  const int64_t half = batch * ((M + 255) / 256) * ((N + 127) / 128);
  return M >= 256 && t128 > 256 && half <= 256 && (gemm_half_whole(M, N, K) ? K >= 2048 : a_k && K >= 4096);
}
// Tiles of a product that only the register-staged cores can address: 64 x 64 (fp32
// 32 x 32) for grids of few tiles, else the size whose grid is modelled fastest, since a
// tile's cost hardly depends on how much of it lies inside the output: ns a tile of a full
// chip, 128 x 128 5.3 + 3.6 per 64-step k-tile (fp32 6 + 7.6 per 32 steps), 64 x 64 2.8 +
// 1.5 (2.6 + 2.1), fp32 32 x 32 1.6 + 0.85; 16 (the 16 x 16 kernel, which takes any
// layout): 0.56 per 16 steps, one workgroup's at least 420.  Batches of products, us,
// 16 x 16 / 32 / 64 / 128: bf16 512 of [63,1001,63] 292 / - / 24 / 33, 4096 of [5,7,5]
// 12.3 / - / 16.4 / 34.7, of [33,33,33] 64 / - / 22 / 47, 512 of [100,65,100] 69 / - /
// 14.4 / 11.9; fp32 4096 of [5,1001,5] 150 / 86 / 278 / 1018, of [33,65,33] 104 / 65 /
// 42 / 123, 30000 of [5,7,5] 18 / 63 / 123 / 346; [1999,1001,1999] bf16 - / - / 28 / 22.
constexpr int gemm_staged_tile(int64_t batch, int64_t M, int64_t N, int64_t K, int es) {
  if (es == 4 && gemm_f32_tiny(batch, M, N)) return 32;
  if (gemm_small_tiles(batch, M, N, es)) return 64;
  auto tiles = [&](int64_t t) { return static_cast<double>(batch) * ((M + t - 1) / t) * ((N + t - 1) / t); };
  const double kt = static_cast<double>(es == 4 ? (K + 31) / 32 : (K + 63) / 64), k16 = static_cast<double>((K + 15) / 16);
  int best = 128;
  double cost = tiles(128) * (es == 4 ? 6.0 + 7.6 * kt : 5.3 + 3.6 * kt);
  const double c64 = tiles(64) * (es == 4 ? 2.6 + 2.1 * kt : 2.8 + 1.5 * kt);
  if (c64 < cost) best = 64, cost = c64;
  const double c32 = tiles(32) * (1.6 + 0.85 * kt);
  if (es == 4 && c32 < cost) best = 32, cost = c32;
  const double c16 = tiles(16) * 0.56 * k16, serial = 420.0 * k16;
  if (batch <= 65535 && (M + 15) / 16 <= 65535 && (c16 > serial ? c16 : serial) < cost) best = 16;
  return best;
}

}  // namespace ghip
