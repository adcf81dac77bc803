// The tile GEMM (gemm_tile_kernel.hpp) of one weight format.
#include "gemm_tile_kernel.hpp"

int qmm::tile_gemm_q6k(int kind, int shape, const TileArgs &a, hipStream_t s) {
  return tile::dispatch<tile::kQ6K>(kind, shape, a, s);
}
