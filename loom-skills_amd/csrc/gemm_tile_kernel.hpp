// GGUF-block matmuls on the f16 MFMA for many rows: the prefill GEMM g_gemm_{fmt}_{store|acc|swiglu}
// (S/gen_gemm.py:535-703) and the MoE grouped expert GEMMs g_moe_ggu_{fmt}[_fused]_k{H} / g_moe_gdn_{fmt}_k{FE}
// (S/gen_moe.py:1126-1228; the Q4_0 expert staging of S/moe_q4_0.py:11-61).
//
//   dense   Y[r, c]   = (acc ? Y[r, c] : 0) + inv[r] sum_k X16[r, k] W[c, k]
//   swiglu  Y[r, c]   = silu(inv[r] sum_k X16[r, k] Wg[c, k]) (inv[r] sum_k X16[r, k] Wu[c, k])
//   gu      act[r, c] = act_fn(inv[t] sum_k X16[t, k] Wg[e][c, k] + bg[e, c], inv[t] sum_k X16[t, k] Wu[e][c, k]
//                       + bu[e, c]),  t = rowmap[r] / KU  (rows gathered from the token rows)
//   dn      ys[r, c]  = inv[r] sum_k A16[r, k] Wd[e][c, k] + bd[e, c]            (rows already sorted)
//
// X16 / A16 are the row-scaled f16 operands of g_row_scale_f16[_tiles] (S/gen_llm.py:1843-1915, S/gen_moe.py:503-527),
// inv = scales[row, 1]; W is dequantized to f16 in registers with the reference's roundings (deq_f16.hpp: Q4_K
// fma_f16(f16(q), f16(d sc), f16(-dmin m)), Q6_K f16(f16(d sc) (q - 32)), Q4_0 f16(d (q - 8)));
// fp32 accumulation.
//
// Design (gfx950: wave64, v_mfma_f32_32x32x16_f16, 160 KB LDS, 256 CUs in 8 XCDs). A workgroup is NW waves along N by
// KS parts of K over a tile of BM rows x 64 NW weight columns (gate/up: 32 NW columns of both matrices, a wave's first
// 32-column block from the gate matrix and its second from the up matrix, so the activation is applied in registers).
//   - A wave streams its own 64 weight columns of its K-part straight into registers, half a super-block (128 values)
//     a step and one step ahead, and dequantizes each fragment there once: it feeds BM / 32 MFMAs, and no weight
//     touches LDS.
//   - The activation rows of a step (BM x 128 values a K-part) go straight into LDS (buffer_load ... lds, no
//     registers), double-buffered, one barrier a step. A row is 256 bytes; its 16-byte chunk c lies at chunk
//     c ^ (row % 16), so the 32 rows a fragment read covers spread over every bank.
//   - Two waves a SIMD (eight waves, or two workgroups of four a CU): a wave issues one vector instruction in about 8
//     cycles, so it takes a second wave to dequantize at the SIMD's rate beside the first one's MFMAs.
//   - The K-parts meet through LDS at the end: each part finishes the accumulator registers r of [16 p / KS,
//     16 (p + 1) / KS) of every 32 x 32 block, adding the parts in order.
// MFMA operand order: lane (lc, h) = (lane % 32, lane / 32) of a K16 step holds 8 K values of row / column lc. Q4_K and
// Q6_K: lane half h takes code bytes 16 h .. 16 h + 15 of a 64-value page, so K16 step (jh, gl, s2) of a 128-value step
// is K positions 64 jh + 32 gl + 16 h + 8 s2 ..; Q4_0: lane half h takes block 2 jh + h of the step, positions
// 64 jh + 32 h + 16 gl + 8 s2 .. . The activation fragment is read from LDS at the same K.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "deq_f16.hpp"
#include "gemm_tile.hpp"

namespace qmm {
namespace tile {

constexpr int kGroupM = 8;   // row tiles of a group in the dense tile order

typedef __attribute__((ext_vector_type(4))) u32 u32x4;

enum { kQ4K = 0, kQ4KT = 1, kQ6K = 2, kQ40 = 3 };

// 16 bytes a lane from a buffer resource into LDS at lds + 16 lane (wave-uniform lds, soff); lanes past the resource's
// end write zeros. Written out so that the compiler's wait counting stays with the register loads: it would drain every
// load before each LDS read. Nothing is returned in registers; the caller waits with wait_vm0 before the barrier.
__device__ __forceinline__ void lds_load16(u32x4 rsrc, u32 voff, u32 soff, u32 lds) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(voff), "s"(rsrc), "s"(soff), "s"(lds)
               : "m0", "memory");
}
__device__ __forceinline__ void wait_vm0() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// One column's registers of a 128-value step (the lane's half of the codes).
template <int WF>
struct Raw;

template <>
struct Raw<kQ4K> {   // two pages' 16 code bytes and the super-block header
  uint4 q[2], hd;
};
template <>
struct Raw<kQ6K> {   // ql of the even / odd groups, qh, the half's 8 scales, d (in the high half)
  uint4 qa, qb, qh;
  u32 s0, s1, d;
};
template <>
struct Raw<kQ40> {   // two blocks' 16 code bytes and d
  uint4 q[2];
  u32 d[2];
};

constexpr int raw_of(int wf) { return wf == kQ4KT ? kQ4K : wf; }
constexpr int64_t row_bytes_of(int wf, int64_t k) {
  return wf == kQ40 ? k / 32 * 18 : k / 256 * (wf == kQ6K ? 210 : 144);
}

// The wave's weight stream: load(hs) issues the loads of half super-block hs of the wave's two 32-column blocks, and
// take(j, lds) turns block j's into Raw registers. A GGUF row is thousands of bytes long, so a load in which every lane
// reads its own column touches 64 lines and takes the CU's address unit 64 cycles or more (twice that at Q6_K's 2-byte
// alignment: the unit was busy 9.8 k cycles a step beside 4.1 k of MFMAs). The GGUF formats therefore load a column's
// contiguous bytes with neighbouring lanes (four lanes a 64-byte code run) and pass them to the lanes that multiply
// them through kXpose bytes of the wave's own LDS (its reads and writes there are in order, so nothing waits for
// another wave). A 16-byte piece p of column c is written at c 4 + (p ^ (c / 4 % 4)) (two pieces a column:
// c 2 + (p ^ (c / 8 % 2))) so that the 16 columns a read covers at a time lie in different banks.
constexpr int xpose_bytes(int wf) { return wf == kQ4KT ? 0 : wf == kQ4K ? 2048 : wf == kQ6K ? 3072 : 2304; }
__device__ __forceinline__ int slot4(int c, int p) { return 4 * c + (p ^ ((c >> 2) & 3)); }
__device__ __forceinline__ int slot2(int c, int p) { return 2 * c + (p ^ ((c >> 3) & 1)); }
// dword v of lane l % 32 (lo) and of lane 32 + l % 32 (hi), in every lane
__device__ __forceinline__ void both_halves(u32 v, u32 &lo, u32 &hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  lo = r[0];
  hi = r[1];
}

// Matrix of block j at m[j] (first byte of column n0), the block's first column j0[j] from it, nc columns from n0 on
// (columns past them read the last one)
template <int WF>
struct Stream {
  const u8 *m[2];
  u32 oc[2][2], oh[2], os[2];   // per-lane byte offsets: codes, qh / d, scales
  uint4 rc[2][2], rh[2];
  u32 rs[2][2];
  uint4 hd;

  __device__ __forceinline__ void init(const u8 *m0, const u8 *m1, int j0, int j1, int nc, u32 RB, int lane) {
    m[0] = m0;
    m[1] = m1;
    const int h = lane >> 5, lc = lane & 31;
    const int jb[2] = {j0, j1};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      auto at = [&](int c) { return (u32)min(jb[j] + c, nc - 1) * RB; };
      if constexpr (WF == kQ4KT) {
        // tiled: n0 is a multiple of 16; 16-column block at 16 RB, column c % 16's codes at 512 + 1024 h + 64 (c % 16)
        const int c = min(jb[j] + lc, nc - 1);
        oc[j][0] = (u32)(c >> 4) * 16u * RB + 512u + 1024u * (u32)h + 64u * (u32)(c & 15);
        os[j] = (u32)(c >> 4) * 16u * RB + 32u * (u32)(c & 15);
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
          oc[j][i] = at(16 * i + (lane >> 2)) + (u32)(lane & 3) * (WF == kQ40 ? 18u : 16u);
        if constexpr (WF == kQ6K) {
          oh[j] = at(lane >> 1) + 128u + 16u * (u32)(lane & 1);
          os[j] = at(lc);
        }
      }
    }
    if constexpr (WF == kQ4K) os[0] = (u32)min((h ? j1 : j0) + lc, nc - 1) * RB;
  }
  // the loads of half super-block hs, in kLoads pieces so that the caller can spread them between other instructions
  static constexpr int kLoads = WF == kQ4K ? 5 : WF == kQ4KT ? 6 : 8;
  __device__ __forceinline__ void load(int hs, int lane, int piece) {
    const int sb = hs >> 1, hb = hs & 1;
    if (WF == kQ4K && piece == 4) {
      // lane l the header of column l of the wave's 64 (lanes 32 .. 63: block 1, in its own matrix for gate/up)
      hd = ld16((lane < 32 ? m[0] : m[1]) + sb * 144 + os[0]);
      return;
    }
    constexpr int per = kLoads / 2;
    const int j = piece / per, i = piece % per;
    if constexpr (WF == kQ4KT) {
      // unit sb / 2 (4608 bytes): page p's bytes 16 h .. in plane 2 (p % 2) + h, 32 (sb % 2) + 16 (p / 2) in the column
      if (i < 2) rc[j][i] = ld16(m[j] + (sb >> 1) * 4608 + 32 * (sb & 1) + 16 * hb + 2048 * i + oc[j][0]);
      else rh[j] = ld16(m[j] + (sb >> 1) * 4608 + 16 * (sb & 1) + os[j]);
    } else if constexpr (WF == kQ4K) {
      rc[j][i] = ld16(m[j] + sb * 144 + 16 + 64 * hb + oc[j][i]);
    } else if constexpr (WF == kQ6K) {
      const u8 *b = m[j] + sb * 210;
      if (i < 2) rc[j][i] = ld16u(b + 64 * hb + oc[j][i]);
      else if (i == 2) rh[j] = ld16u(b + 32 * hb + oh[j]);
      else {
        // lanes 0 .. 31 the half's 8 scales, lanes 32 .. 63 the block's last 8 bytes (d in the last two)
        const u8 *q = b + (lane < 32 ? 192 + 8 * hb : 202) + os[j];
        rs[j][0] = ld4u(q);
        rs[j][1] = ld4u(q + 4);
      }
    } else {
      const u8 *b = m[j] + hs * 72 + oc[j][i & 1];
      if (i < 2) rc[j][i] = ld16u(b + 2);
      else rs[j][i & 1] = *reinterpret_cast<const u16 *>(b);
    }
  }
  __device__ __forceinline__ void take(Raw<raw_of(WF)> (&r)[2], u8 *lds, int lane) {
    const int h = lane >> 5, lc = lane & 31;
    uint4 *c4 = reinterpret_cast<uint4 *>(lds);
    uint4 *c2 = reinterpret_cast<uint4 *>(lds + 2048);
    if constexpr (WF == kQ4K) {
      const u32 v[4] = {hd.x, hd.y, hd.z, hd.w};
      u32 lo[4], hi[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) both_halves(v[q], lo[q], hi[q]);
      r[0].hd = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      r[1].hd = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (WF == kQ4KT) {
        r[j].q[0] = rc[j][0];
        r[j].q[1] = rc[j][1];
        r[j].hd = rh[j];
        continue;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) c4[slot4(16 * i + (lane >> 2), lane & 3)] = rc[j][i];
      if constexpr (WF == kQ6K) c2[slot2(lane >> 1, lane & 1)] = rh[j];
      if constexpr (WF == kQ40) {
        u16 *d = reinterpret_cast<u16 *>(lds + 2048);
#pragma unroll
        for (int i = 0; i < 2; ++i) d[64 * i + lane] = (u16)rs[j][i];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if constexpr (WF == kQ4K || WF == kQ40) {   // Q4_K: page p's bytes 16 h ..; Q4_0: block 2 p + h
        r[j].q[0] = c4[slot4(lc, h)];
        r[j].q[1] = c4[slot4(lc, 2 + h)];
      }
      if constexpr (WF == kQ40) {
        const u16 *d = reinterpret_cast<const u16 *>(lds + 2048);
        r[j].d[0] = d[4 * lc + h];
        r[j].d[1] = d[4 * lc + 2 + h];
      }
      if constexpr (WF == kQ6K) {
        r[j].qa = c4[slot4(lc, h)];
        r[j].qb = c4[slot4(lc, 2 + h)];
        r[j].qh = c2[slot2(lc, h)];
        u32 x;
        both_halves(rs[j][0], r[j].s0, x);
        both_halves(rs[j][1], r[j].s1, r[j].d);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
};

// a column's f16 scale pairs (d sc, -dmin m) of the step's four 32-value runs (jh, gl), as (dsc | nmn << 16); Q6_K's are
// the lane half's 16-value runs, Q4_0's is d
template <int WF>
__device__ __forceinline__ void decode_pairs(const Raw<raw_of(WF)> &r, int hb, int h, u32 (&pr)[4]) {
  if constexpr (WF == kQ4K || WF == kQ4KT) {
    // the 6-bit (scale, minimum) bytes of sub-blocks 4 hb .. 4 hb + 3 (ggml get_scale_min_k4)
    const u32 scw = hb ? (r.hd.w & 0x0F0F0F0Fu) | ((r.hd.y >> 2) & 0x30303030u) : r.hd.y & 0x3F3F3F3Fu;
    const u32 mnw = hb ? ((r.hd.w >> 4) & 0x0F0F0F0Fu) | ((r.hd.z >> 2) & 0x30303030u) : r.hd.z & 0x3F3F3F3Fu;
    const h2 dm = as_h2(r.hd.x ^ 0x80000000u);   // (d, -dmin)
    const h2 m1024 = as_h2(0xE400E400u);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      // (1024 + sc, 1024 + m) as an f16 pair: bytes (sc, 0x64, m, 0x64); less 1024 is exact; one rounding multiply
      const u32 sel = (u32)(g | 0x0C00u | ((4 + g) << 16) | 0x0C000000u);
      const u32 p = __builtin_amdgcn_perm(mnw, scw, sel) | 0x64006400u;
      pr[g] = as_u32((as_h2(p) + m1024) * dm);
    }
  } else if constexpr (WF == kQ6K) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {   // f16(d sc): d sc is exact in f32 (S/gen_gemm.py:435-444)
      const u32 s = g < 2 ? r.s0 : r.s1;
      const float sv = f16_to_f32(r.d >> 16) * (float)(signed char)((s >> (8 * (2 * (g & 1) + h))) & 0xFFu);
      pr[g] = (u32)__builtin_bit_cast(u16, (_Float16)sv);
    }
  } else {
#pragma unroll
    for (int g = 0; g < 4; ++g) pr[g] = r.d[g >> 1];
  }
}

// weights 2 d, 2 d + 1 of the 8 of K16 step (jh, gl, s2) of a 128-value step, from the step's scale pair
template <int WF>
__device__ __forceinline__ u32 dequant2(const Raw<raw_of(WF)> &r, u32 pr, int jh, int gl, int s2, int d) {
  const h2 pv = as_h2(pr);
  const h2 dsc = h2{pv[0], pv[0]};   // splats fold into the packed instructions' operand selects
  const bool hi = d & 1;
  const u32 sel = hi ? 0x04030402u : 0x04010400u;   // bytes (0, 1) or (2, 3) as (1024 + code) f16 pairs
  if constexpr (WF == kQ6K) {
    // codes ((ql >> 4 jh) & 15) | (((qh >> (4 jh + 2 gl)) & 3) << 4)
    const uint4 &ql = gl ? r.qb : r.qa;
    const u32 l = d < 2 ? (s2 ? ql.z : ql.x) : (s2 ? ql.w : ql.y);
    const u32 q = d < 2 ? (s2 ? r.qh.z : r.qh.x) : (s2 ? r.qh.w : r.qh.y);
    const int hs = 4 * jh + 2 * gl;
    const u32 c = ((l >> (4 * jh)) & 0x0F0F0F0Fu) | ((hs < 4 ? q << (4 - hs) : q >> (hs - 4)) & 0x30303030u);
    // less 1024 + 32 is exact, then one rounding multiply
    return as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, c, sel)) + as_h2(0xE420E420u)) * dsc);
  } else {
    const uint4 &q = r.q[jh];
    const u32 w = d < 2 ? (s2 ? q.z : q.x) : (s2 ? q.w : q.y);
    const u32 n = (gl ? w >> 4 : w) & 0x0F0F0F0Fu;
    if constexpr (WF == kQ40)   // (1024 + q) - 1032 = q - 8 exactly, then one rounding multiply
      return as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, n, sel)) + as_h2(0xE408E408u)) * dsc);
    // a code byte 0000qqqq read as OCP E4M3 is q 2^-9 exactly; one rounding fma
    const h2 c = hi ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(n, 512.0f, true)
                    : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(n, 512.0f, false);
    return as_u32(__builtin_elementwise_fma(c, dsc, h2{pv[1], pv[1]}));
  }
}

template <int WF, int KIND, int BM, int NW, int KS>
__global__ __launch_bounds__(64 * NW * KS, 2) void gemm_tile_kernel(TileArgs a) {
  constexpr int NI = BM / 32;
  constexpr bool kTwoW = KIND == kTGU || KIND == kTSwiglu;
  constexpr bool kDenseRows = KIND == kTDense || KIND == kTSwiglu;
  constexpr int BN = (kTwoW ? 32 : 64) * NW;   // output columns
  constexpr int kPart = BM * 256;              // LDS bytes of a K-part's staged step
  static_assert(BM <= 64 * NW * KS && BM % (4 * NW) == 0 && 16 % KS == 0, "prologue and staging maps");
  extern __shared__ __align__(1024) u8 smem[];   // [2][KS][BM][256], then a wave's kXpose; at the end the K-part exchange
  constexpr int kXpose = xpose_bytes(WF);
  __shared__ int src_row[BM];
  __shared__ float rinv[BM];                     // the row's inverse activation scale (1 without scales)
  __shared__ unsigned long long live_rows[BM / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % NW, kp = wave / NW;
  const int h = lane >> 5, lc = lane & 31;
  const int M = a.M, N = a.N, K = a.K;

  int m0, n0, expert = 0;
  if constexpr (kDenseRows) {
    // XCD-aware order: workgroup b runs on XCD b % 8, which gets a contiguous range of tiles in groups of kGroupM row
    // tiles (rows fastest inside a group), so that the tiles of an XCD at a time share activation rows and weight
    // columns in its L2
    const int per = (int)(gridDim.x / 8);
    const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (t >= a.tiles_m * a.tiles_n) return;
    const int g = t / (kGroupM * a.tiles_n), gm = min(kGroupM, a.tiles_m - g * kGroupM), gt = t - g * kGroupM * a.tiles_n;
    m0 = (g * kGroupM + gt % gm) * BM;
    n0 = gt / gm * BN;
  } else {
    // expert tiles dealt to the XCDs round-robin: the bucket writes the live tiles first, so a contiguous range per
    // XCD would leave the XCDs holding the trailing unused tiles idle; a tile's column blocks share one XCD's L2
    const int xcd = (int)(blockIdx.x & 7), xi = (int)(blockIdx.x >> 3);
    const int tile = xcd + 8 * (xi / a.tiles_n);
    if (tile >= a.tiles_m) return;
    n0 = (xi % a.tiles_n) * BN;
    m0 = tile * BM;
    expert = a.tile_info[2 * tile];
    if (expert < 0) return;
    expert = expert >= a.E ? a.E - 1 : expert;
  }
  // activation row of each tile row (-1: a dead row, read as zeros and not written)
  if (tid < BM) {
    int src;
    if constexpr (kDenseRows) {
      src = m0 + tid < M ? m0 + tid : -1;
      // skip-padding: 64 rows that all have scale 0 (padding rows) are not written
      if (a.scales && __ballot(src >= 0 && a.scales[2 * (src >= 0 ? src : 0)] != 0.f) == 0) src = -1;
    } else if constexpr (KIND == kTGU) {
      const int rm = a.rowmap[m0 + tid];
      src = rm >= 0 ? rm / a.KU : -1;
      src = src < a.x_rows ? src : -1;
    } else {
      src = a.rowmap[m0 + tid] >= 0 ? m0 + tid : -1;
    }
    src_row[tid] = src;
    rinv[tid] = (a.scales && src >= 0) ? a.scales[2 * src + 1] : 1.f;
    const unsigned long long b = __ballot(src >= 0);
    if (lane == 0) live_rows[wave] = b;
  }
  __syncthreads();
  // 32-row blocks up to the last one with a live row; the blocks past it take no MFMAs
  int nlive = 0;
#pragma unroll
  for (int i = 0; i < BM / 64; ++i) {
    const unsigned long long b = live_rows[i];
    nlive = (u32)b ? 2 * i + 1 : nlive;
    nlive = (u32)(b >> 32) ? 2 * i + 2 : nlive;
  }
  nlive = __builtin_amdgcn_readfirstlane(nlive);
  if (nlive == 0) return;

  // ---- the K-part's steps of 128 values
  const int H = K / 128;
  const int h0 = kp * H / KS, np = (kp + 1) * H / KS - h0, S = (H + KS - 1) / KS;
  const int64_t RB = row_bytes_of(WF, K);

  // ---- activation staging: load i of a step writes rows 4 (i NW + wn) .. + 3 of the part
  constexpr int ND = BM / (4 * NW);
  const uint64_t xa = (uint64_t)a.x16;
  const u32x4 xrs = {(u32)xa, (u32)(xa >> 32) & 0xFFFFu, (u32)((int64_t)a.x_rows * K * 2), 0x00020000u};
  u32 aoff[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int row = 4 * (i * NW + wn) + (lane >> 4);
    const int src = src_row[row];
    aoff[i] = src >= 0 ? (u32)src * (u32)K * 2u + (u32)(((lane & 15) ^ (row & 15)) * 16) : 0x80000000u;
  }
  const u32 lds0 = (u32)(uintptr_t)(__attribute__((address_space(3))) u8 *)smem;
  auto stage = [&](int buf, int hs, int i) __attribute__((always_inline)) {
    const u32 dst = __builtin_amdgcn_readfirstlane(lds0 + (u32)((buf * KS + kp) * kPart + wn * 1024));
    lds_load16(xrs, aoff[i], (u32)(hs * 256), dst + (u32)(i * NW * 1024));
  };

  // ---- the wave's weight columns: blocks j = 0, 1 of 32 (gate/up: gate and up of the same columns)
  Stream<WF> st;
  {
    const u8 *mg = a.w, *mu = a.w;
    if constexpr (KIND == kTSwiglu) mu = a.w2;
    if constexpr (!kDenseRows) mg = mu = a.w + (int64_t)expert * a.ebytes;
    if constexpr (KIND == kTGU) mu = a.w2 ? a.w2 + (int64_t)expert * a.ebytes2 : mg + a.up_off;
    const int64_t nb = (int64_t)n0 * RB;   // n0 is a multiple of 16: tiled columns too
    const int c0 = kTwoW ? 32 * wn : 64 * wn;
    st.init(mg + nb, mu + nb, c0, kTwoW ? c0 : c0 + 32, N - n0, (u32)RB, lane);
  }
  u8 *xp = smem + 2 * KS * kPart + wave * kXpose;

  f32x16 acc[NI][2];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  Raw<raw_of(WF)> now[2];
  const u32 axor = (u32)(lc * 256 + (((WF == kQ40 ? 4 * h : 2 * h) ^ (lc & 15)) << 4));

  // K16 step kk of a 128-value step (Q6_K: jh innermost, the two uses of a masked qh dword)
  auto jh_of = [](int kk) { return WF == kQ6K ? kk & 1 : kk >> 2; };
  auto gl_of = [](int kk) { return WF == kQ6K ? kk >> 2 : (kk >> 1) & 1; };
  auto s2_of = [](int kk) { return WF == kQ6K ? (kk >> 1) & 1 : kk & 1; };

  // A step's vector memory instructions (activation pieces, then weight pieces) are spread over its first half, one every
  // kEvery MFMAs: issued together behind the barrier they would fill the CU's address unit for as long as half the
  // step's MFMAs take while every wave waits to issue its own.
  auto run = [&](auto nlc) __attribute__((always_inline)) {
    constexpr int NL = decltype(nlc)::value;
    constexpr int kVm = ND + Stream<WF>::kLoads;
    constexpr int kEvery = 8 * NL / kVm > 0 ? 8 * NL / kVm : 1;   // one every kEvery of the 8 NL MFMAs, or
    constexpr int kPer = (kVm + 8 * NL - 1) / (8 * NL);           // kPer behind each
    auto fetch = [&](int buf, int hs, int v) __attribute__((always_inline)) {
      if (v < ND) stage(buf, hs, v);
      else st.load(hs, lane, v - ND);
    };
    u32 pr[2][4];
    f16x8 af[NL];
    u32 bf[2][2][4];   // weight fragments [step parity][block][dword]
    auto part = [&](int kk, int q) __attribute__((always_inline)) {   // dword q % 4 of block q / 4 of K16 step kk
      const int jh = jh_of(kk), gl = gl_of(kk), j = q >> 2;
      bf[kk & 1][j][q & 3] = dequant2<WF>(now[j], pr[j][2 * jh + gl], jh, gl, s2_of(kk), q & 3);
    };
    // the loaded weights of half super-block hs into place
    auto take = [&](int hs) __attribute__((always_inline)) {
      wait_vm0();
      st.take(now, xp, lane);
#pragma unroll
      for (int j = 0; j < 2; ++j) decode_pairs<WF>(now[j], hs & 1, h, pr[j]);
    };
    {
      const int hs = min(h0, H - 1);
#pragma unroll
      for (int v = 0; v < kVm; ++v) fetch(0, hs, v);
      take(hs);
#pragma unroll
      for (int q = 0; q < 8; ++q) part(0, q);
    }
    __syncthreads();
    for (int s = 0; s < S; ++s) {
      if (s < np) {
        const int buf = s & 1, hn = min(h0 + s + 1, H - 1);   // past the part's end: the last half again, not multiplied
        const u8 *ab = smem + (buf * KS + kp) * kPart;
        auto read_a = [&](int i, int kk) __attribute__((always_inline)) {
          const int jh = jh_of(kk), gl = gl_of(kk), s2 = s2_of(kk);
          const u32 kc = (u32)(WF == kQ40 ? 8 * jh + 2 * gl + s2 : 8 * jh + 4 * gl + s2) << 4;
          af[i] = *reinterpret_cast<const f16x8 *>(ab + (axor ^ kc) + i * 8192);
        };
#pragma unroll
        for (int i = 0; i < NL; ++i) read_a(i, 0);
        // K16 step kk issues its MFMAs on fragments prepared by the step before, and between them dequantizes the next
        // K16 step's weights (two values a part; the last one's: the next step's first) and reloads each activation
        // fragment after its last use: the matrix pipe runs while the vector pipe works a step ahead. Scheduling
        // barriers keep that order.
        constexpr int kPin = 0x0004;   // only scalar instructions cross the barriers
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
          if (kk == 7) take(hn);
#pragma unroll
          for (int i = 0; i < NL; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const u32x4 b = {bf[kk & 1][j][0], bf[kk & 1][j][1], bf[kk & 1][j][2], bf[kk & 1][j][3]};
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], __builtin_bit_cast(f16x8, b), acc[i][j], 0, 0, 0);
              __builtin_amdgcn_sched_barrier(kPin);
              if (j == 1 && kk < 7) read_a(i, kk + 1);
#pragma unroll
              for (int q = 0; q < 4 / NL; ++q) part((kk + 1) & 7, (4 / NL) * (2 * i + j) + q);
              constexpr int kSlots = 2 * NL;
              const int slot = kk * kSlots + 2 * i + j;
              if (slot % kEvery == 0) {
#pragma unroll
                for (int v = slot / kEvery * kPer; v < (slot / kEvery + 1) * kPer; ++v)
                  if (v < kVm) fetch(buf ^ 1, hn, v);
              }
              __builtin_amdgcn_sched_barrier(kPin);
            }
          }
        }
      }
      __syncthreads();
    }
  };
  if (nlive > NI / 2) run(std::integral_constant<int, NI>{});
  else run(std::integral_constant<int, NI / 2>{});

  // ---- the K-parts meet: part p keeps registers r of [p RK, (p + 1) RK) of every block and hands the others on
  constexpr int RK = 16 / KS;
  float out[NI][2][RK];
  if constexpr (KS > 1) {
    float *red = reinterpret_cast<float *>(smem);
    constexpr int kSlot = NI * 2 * RK * 64;   // floats a (wave, receiver, sender) slot
    auto slot = [&](int to, int from) { return red + ((wn * KS + to) * (KS - 1) + (from < to ? from : from - 1)) * kSlot + lane; };
#pragma unroll
    for (int p = 0; p < KS; ++p) {
      if (p == kp) continue;
      float *d = slot(p, kp);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < RK; ++r) d[((i * 2 + j) * RK + r) * 64] = acc[i][j][p * RK + r];
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < KS; ++p) {
      if (p == kp) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < RK; ++r) out[i][j][r] = acc[i][j][p * RK + r];
      }
    }
    float sum[NI][2][RK];
#pragma unroll
    for (int p = 0; p < KS; ++p) {
      const float *d = p == kp ? nullptr : slot(kp, p);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < RK; ++r) {
            const float v = d ? d[((i * 2 + j) * RK + r) * 64] : out[i][j][r];
            sum[i][j][r] = p ? sum[i][j][r] + v : v;
          }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < RK; ++r) out[i][j][r] = sum[i][j][r];
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < RK; ++r) out[i][j][r] = acc[i][j][r];
  }

  // ---- epilogue: accumulator register r of a block is row 8 (r / 4) + 4 h + r % 4, column lc
  float *yf = static_cast<float *>(a.y);
  u16 *yb = static_cast<u16 *>(a.y);
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int r = 0; r < RK; ++r) {
      const int rr = kp * RK + r;
      const int lr = 32 * i + 8 * (rr >> 2) + 4 * h + (rr & 3);
      if (src_row[lr] < 0) continue;
      const float inv = rinv[lr];
#pragma unroll
      for (int j = 0; j < (kTwoW ? 1 : 2); ++j) {
        const int c = n0 + (kTwoW ? 32 * wn : 64 * wn + 32 * j) + lc;
        if (c >= N) continue;
        const int64_t o = (int64_t)(m0 + lr) * N + c;
        float v = out[i][j][r] * inv;
        if constexpr (!kDenseRows) {
          const int64_t bo = (int64_t)expert * N + c;
          v += a.bias ? a.bias[bo] : 0.f;
          if constexpr (KIND == kTGU) v = act_fn(a.act, v, out[i][1][r] * inv + (a.bias2 ? a.bias2[bo] : 0.f));
          yf[o] = v;
        } else {
          if constexpr (KIND == kTSwiglu) v = act_fn(QMM_ACT_SILU, v, out[i][1][r] * inv);
          if (a.y_bf16) {
            if (a.acc) v += bf16_to_f32(yb[o]);
            yb[o] = (u16)f32_to_bf16_rne(v);
          } else {
            if (a.acc) v += yf[o];
            yf[o] = v;
          }
        }
      }
    }
}

template <int WF, int KIND, int BM, int NW, int KS>
int launch(TileArgs a, hipStream_t s) {
  constexpr bool kTwoW = KIND == kTGU || KIND == kTSwiglu;
  constexpr bool kDenseRows = KIND == kTDense || KIND == kTSwiglu;
  constexpr int BN = (kTwoW ? 32 : 64) * NW;
  constexpr int kLds = 2 * KS * BM * 256 + NW * KS * xpose_bytes(WF);
  if constexpr (kDenseRows) a.tiles_m = (a.M + BM - 1) / BM;   // grouped: the caller's 64-row expert tiles
  a.tiles_n = (a.N + BN - 1) / BN;
  const int64_t tiles = kDenseRows ? (int64_t)a.tiles_m * a.tiles_n : (int64_t)((a.tiles_m + 7) / 8) * 8 * a.tiles_n;
  const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)));
  static std::atomic<unsigned> raised{0};
  const void *fn = reinterpret_cast<const void *>(&gemm_tile_kernel<WF, KIND, BM, NW, KS>);
  if (int st = raise_dyn_lds(fn, kLds, raised)) return st;
  gemm_tile_kernel<WF, KIND, BM, NW, KS><<<grid, 64 * NW * KS, kLds, s>>>(a);
  return launch_status();
}

template <int WF>
int dispatch(int kind, int shape, const TileArgs &a, hipStream_t s) {
  if (kind == kTGU) return launch<WF, kTGU, 64, 4, 1>(a, s);
  if (kind == kTDN) return launch<WF, kTDN, 64, 4, 1>(a, s);
  if (kind == kTSwiglu) {
    if (shape == kT128x4x1) return launch<WF, kTSwiglu, 128, 4, 1>(a, s);
    if (shape == kT128x4x2) return launch<WF, kTSwiglu, 128, 4, 2>(a, s);
    if (shape == kT64x4x1) return launch<WF, kTSwiglu, 64, 4, 1>(a, s);
    return launch<WF, kTSwiglu, 64, 2, 4>(a, s);
  }
  if (shape == kT128x4x1) return launch<WF, kTDense, 128, 4, 1>(a, s);
  if (shape == kT128x4x2) return launch<WF, kTDense, 128, 4, 2>(a, s);
  if (shape == kT64x4x1) return launch<WF, kTDense, 64, 4, 1>(a, s);
  return launch<WF, kTDense, 64, 2, 4>(a, s);
}

}  // namespace tile
}  // namespace qmm
