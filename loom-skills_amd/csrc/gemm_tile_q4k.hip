// The tile GEMM (gemm_tile_kernel.hpp) of one weight format.
#include "gemm_tile_kernel.hpp"

int qmm::tile_gemm_q4k(int kind, int shape, const TileArgs &a, hipStream_t s) {
  return tile::dispatch<tile::kQ4K>(kind, shape, a, s);
}
