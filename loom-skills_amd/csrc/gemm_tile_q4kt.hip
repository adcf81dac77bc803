// The tile GEMM (gemm_tile_kernel.hpp) of one weight format.
#include "gemm_tile_kernel.hpp"

int qmm::tile_gemm_q4kt(int kind, int shape, const TileArgs &a, hipStream_t s) {
  return tile::dispatch<tile::kQ4KT>(kind, shape, a, s);
}
