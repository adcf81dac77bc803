// The tile GEMM (gemm_tile_kernel.hpp) of one weight format.
#include "gemm_tile_kernel.hpp"

int qmm::tile_gemm_q40(int kind, int shape, const TileArgs &a, hipStream_t s) {
  return tile::dispatch<tile::kQ40>(kind, shape, a, s);
}
