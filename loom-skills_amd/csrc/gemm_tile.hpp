// The tile GEMM on the f16 MFMA for GGUF-block weights (Q4_K, tiled Q4_K, Q6_K, Q4_0): arguments and launchers. The
// kernel is in gemm_tile_kernel.hpp, one translation unit a weight format (gemm_tile_*.hip).
#pragma once

#include "common.hpp"

namespace qmm {

// kTDense: Y (+)= X W^T; kTSwiglu: Y = silu(X Wg^T inv) (X Wu^T inv) over dense rows; kTGU / kTDN: the grouped gate/up
// and down GEMMs over bucketed 64-row expert tiles
enum TileKind { kTDense = 0, kTSwiglu = 1, kTGU = 2, kTDN = 3 };
// the workgroup: rows x waves along N x K-parts (a wave holds 64 weight columns)
enum TileShape { kT128x4x1 = 0, kT128x4x2 = 1, kT64x4x1 = 2, kT64x2x4 = 3 };

struct TileArgs {
  int M, N, K;                 // dense: rows; grouped: rows of the sorted output (max_tiles * 64)
  const _Float16 *x16;         // activation rows (dense / dn: [M, K]; gu: token rows [x_rows, K])
  const float *scales;         // [rows of x16, 2] or NULL
  int x_rows;                  // rows of x16
  const u8 *w, *w2;            // dense: W (swiglu: gate, up); grouped: expert tensors (gu: gate, up; fused: w only)
  int64_t ebytes, ebytes2;     // grouped: bytes of one expert's matrix (gu: gate / up)
  int64_t up_off;              // gu, fused: bytes from an expert's gate matrix to its up matrix
  const int32_t *tile_info, *rowmap;
  const float *bias, *bias2;   // grouped: per-expert output biases [E, N] (gu: gate, up; dn: bias only) or NULL
  int KU, E, act;
  void *y;
  int acc, y_bf16;             // dense: Y += ..., bf16 output rows
  int tiles_m, tiles_n;
};

int tile_gemm_q4k(int kind, int shape, const TileArgs &a, hipStream_t s);
int tile_gemm_q4kt(int kind, int shape, const TileArgs &a, hipStream_t s);
int tile_gemm_q6k(int kind, int shape, const TileArgs &a, hipStream_t s);
int tile_gemm_q40(int kind, int shape, const TileArgs &a, hipStream_t s);

}  // namespace qmm
