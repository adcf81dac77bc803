// Decode matvecs on Q8_1 activations for 9 tokens and more (Q4_K, GGUF or tiled): g_mv_{fmt}_k{K}[_swiglu|_pair]_q8 of a
// batch of decoding sequences (S/gen_llm.py:1159-1197, :1288-1301), on the int8 MFMA.
//
//   y[t, r] (+)= sum over 32-value groups g of (di sc - xs mn) da,   di = sum q_w q_x (exact), sc = d sc_g,
//                                                                     mn = dmin m_g, (da, xs) the group's Q8_1 pair
//   swiglu: y (+)= silu(gate) up;  pair: y (+)= x W^T, y2 (+)= x W2^T (one launch, a matrix a grid layer)
//
// Every output has the bits of the same token's call with fewer tokens (a multi-token call equals one-token calls,
// make_kernel_tests.py:264-268): di is an exact integer, a group's term takes the roundings of q4k_q8_term (xs mn as a
// product of one MFMA step, so rounded once, then one fma), and the terms meet in the tree of the kernel that takes the
// call at one token:
//   kItems   (gemv_q8.hip, the item walk: every GGUF call but the next) an item is a page, two groups; item lane l sums
//            page l % 4 of super-blocks l / 4, l / 4 + 16, ..., then the 64 lanes meet in a butterfly (xor 32 .. 1)
//   kSlices  (gemv_q4kt.hip; gemv_q8.hip's K-sliced kernel, GGUF at K = 4096 / 8192) a wave's slice of K: chains of four
//            groups (half a super-block) are summed over the units of the slice (tiled), the halves in a butterfly, the
//            slices in order
//
// The matvec kernels read every weight once per two tokens (GGUF) or eight (tiled) and spend a v_dot4 per four products.
// Here a weight is read once per 16 tokens and 16 x 16 products of a group take one v_mfma_i32_16x16x32_i8 a wave: what is
// left is the fixup of each group's 256 sums (convert, two fma; kItems half a multiply and half an add more: 12 - 14 vector
// instructions of a wave's 30 a group), which bounds it: 24 tokens through 2 x 12288 x 4096 keep the vector pipes busy 80 %
// of the time a CU holds a wave, the address unit 73 %, the LDS 48 %. That call: 112 us in the matvec kernel, 30.4 here, with the quantizer's
// launch (8 us of weights).
//
// A workgroup: 16 weight rows (swiglu: of each matrix) x 16 tokens, eight waves. A wave takes whole super-blocks of all rows
// (kItems: v, v + 16, ... and then v + 8, v + 24, ...; kSlices: slice v): it brings the super-block's codes and pairs of its
// tokens into its own LDS (coalesced: a load in which every lane reads its own token takes the address unit 64 cycles), then
// the rows' super-block past them, the next loads in flight. The waves' sums meet in LDS at the end. That takes up to 128
// registers, so four waves a SIMD. Measured and slower at 24 tokens through 2 x 12288 x 4096: the gate matrix, then the up
// matrix (35.7; kept where an item lane sums several super-blocks, whose sums would not fit), 32 tokens a workgroup (36.4
// at two waves a SIMD; at four it spills), half super-blocks (41.7), workgroups that stay for several tiles (38.7).
//
// MFMA operands: lane (c, q) = (lane % 16, lane / 16) holds 8 K values of weight row / token c; which 8 does not matter
// while both agree. A page's 32 code bytes are two groups (low and high nibbles). Lane (c, q) loads bytes 16 q .. of two
// pages (64 bytes of a row from four lanes); exchanging register halves between lanes 0-31 and 32-63 (v_permlane32_swap)
// leaves bytes 16 (q % 2) + 8 (q / 2) .. + 7 of the one page in the first two registers and of the other in the last
// two; a token's codes of a group are read at those bytes, so they meet the weights at the same K.
// The sums of 16 tokens x 16 rows lie in four registers: lane (c, q), register i is token 4 q + i, row c, so that a row's
// scale is one register. The products xs mn of four groups are the four blocks of a v_mfma_f32_16x16x1_4b_f32: lane (c, q)
// holds row / token c of group q, and register 4 b + i of the result is block b's.
#include "common.hpp"

using namespace qmm;

namespace {

typedef __attribute__((ext_vector_type(4))) u32 u32x4;

enum Order { kItems = 0, kSlices = 1 };
constexpr int kWaves = 8;

struct MArgs {
  int n, tokens, nsb;           // rows of a matrix, tokens, super-blocks a row
  int chains, units;            // kSlices: slice v is super-blocks v chains units .. ; chain j sums units of them, two apart
  const u8 *codes;              // planar Q8_1: codes [tokens][K], then pairs f32 [tokens][K / 32][2]
  const float *meta;
  const u8 *w, *w2;             // swiglu: gate, up; pair: the matrices of blockIdx.z = 0 and 1
  float *y, *y2;
  int accumulate;
};

// a 16-byte piece's registers (0, 2) and (1, 3): halves of the wave exchanged so that 0 and 1 belong to one page, 2 and 3
// to the other
__device__ __forceinline__ u32x4 page_swap(u32x4 v) {
  const auto a = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
  return u32x4{a[0], b[0], a[1], b[1]};
}
__device__ __forceinline__ long pack8(u32 a, u32 b) { return (long)(((uint64_t)b << 32) | a); }

// LONG (kItems): more than 16 super-blocks, so an item lane sums several
template <bool TL, bool SWIGLU, int ORDER, bool LONG>
__global__ __launch_bounds__(64 * kWaves, 4) void mv_q8_mfma_kernel(MArgs a) {
  constexpr int NV = ORDER == kItems ? 4 : 2;                             // sums of a super-block: pages, or halves
  // LDS bytes a wave: the codes of 16 tokens, their da and xs [group][token]
  constexpr int kCode = 16 * 256, kMeta = 1024;
  constexpr int kOwn = kCode + kMeta;
  static_assert(kOwn >= 4 * 256 * 4, "a wave's share of the meeting");
  // swiglu: the gate's meeting has its own room
  __shared__ __align__(16) u8 smem[kWaves * (kOwn + (SWIGLU ? (ORDER == kItems ? 4 : 1) * 256 * 4 : 0))];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, q = lane >> 4;
  const u32 K = (u32)a.nsb * 256u, RB = (u32)a.nsb * 144u;   // all byte offsets fit 32 bits (qmm_mv_q8_mfma_fits)
  // workgroup b runs on XCD b % 8 = blockIdx.x % 8: the token tiles of a row block follow each other there and share its
  // weights in L2
  const int row0 = ((int)blockIdx.y * 8 + (int)(blockIdx.x & 7)) * 16, t0 = (int)(blockIdx.x >> 3) * 16;
  if (row0 >= a.n) return;
  // Matrices that a pass over the super-blocks sums, and passes: both swiglu matrices at once, one after the other where
  // LONG's sums would not fit the registers. kAheadX: the next super-block's tokens are loaded with its weights (else, for
  // the same reason, late in the pass over the present one)
  constexpr int R = SWIGLU && !LONG ? 2 : 1, kPasses = SWIGLU && LONG ? 2 : 1;
  constexpr bool kAheadX = !LONG && R == 1;
  u8 *own = smem + wave * kOwn;
  float *md = reinterpret_cast<float *>(own + kCode);

  // The loads go through buffer resources, whose wave-uniform offset is the super-block's: byte offsets of the lane's row in
  // its matrix (rows past n read row n - 1 and are not stored; tiled: the lane's plane q of its 16-row block, whose header
  // lies 512 + 1024 q + 32 (row % 16) before it), of its tokens' codes (16 lanes a token, four tokens a load) and pairs
  // (four lanes a token); tokens past the last read it
  const int row = min(row0 + c, a.n - 1);
  const u32 wr = TL ? (u32)(row >> 4) * 16u * RB + 32u * (u32)(row & 15) : (u32)row * RB;
  const u32 wc = TL ? wr + 512u + 1024u * (u32)q + 32u * (u32)(row & 15) : wr + 16u * (u32)q;
  u32 xo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) xo[i] = (u32)min(t0 + 4 * i + q, a.tokens - 1) * K + 16u * (u32)c;
  const u32 po = (u32)min(t0 + (lane >> 2), a.tokens - 1) * (K / 4u) + 16u * (u32)(lane & 3);
  auto load = [](const void *p, u32 bytes, u32 off, u32 soff) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, 0));
  };

  // ---- the wave's super-blocks in order, the next one's weights and tokens loaded while one is summed
  struct Pos { int pass, sb, j, u; };   // kItems: j = 0 (v, v + 16, ..) or 1 (v + 8, ..); kSlices: chain j, its unit u
  const int per = a.chains * a.units;   // kSlices: super-blocks of a slice
  const int first = ORDER == kItems ? wave : wave * per;
  auto next = [&](Pos p) __attribute__((always_inline)) {
    if constexpr (ORDER == kItems) {
      p.sb += 2 * kWaves;
      if (p.sb >= a.nsb && p.j == 0 && wave + kWaves < a.nsb) { p.j = 1; p.sb = wave + kWaves; }
    } else {
      if (++p.u == a.units) { p.u = 0; ++p.j; }
      p.sb = p.j == a.chains ? a.nsb : first + p.j + 2 * p.u;
    }
    if (p.sb >= a.nsb) p = Pos{p.pass + 1, first, 0, 0};
    return p;
  };
  u32x4 c0, c1, h, v[4], pr;
  auto load_w = [&](Pos at, int r) __attribute__((always_inline)) {
    const u8 *m = SWIGLU ? (r + at.pass ? a.w2 : a.w) : blockIdx.z ? a.w2 : a.w;
    const u32 sb = (u32)at.sb, bytes = at.pass < kPasses ? (u32)a.n * RB : 0;   // past the last super-block: no memory
    // tiled: unit sb / 2 (4608 bytes), page p's bytes 16 h .. in plane 2 (p % 2) + h, at 64 row + 32 (sb % 2) + 16 (p / 2):
    // lane q reads page q / 2 (and 2 + q / 2), half q % 2, plane q
    const u32 uc = TL ? (sb >> 1) * 4608u + 32u * (sb & 1) : 144u * sb, uh = TL ? (sb >> 1) * 4608u + 16u * (sb & 1) : 144u * sb;
    c0 = load(m, bytes, wc + (TL ? 0u : 16u), uc);
    c1 = load(m, bytes, wc + (TL ? 16u : 80u), uc);
    h = load(m, bytes, wr, uh);
  };
  auto load_x = [&](Pos at) __attribute__((always_inline)) {
    const u32 bytes = at.pass < kPasses ? (u32)a.tokens * K : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = load(a.codes, bytes, xo[i], 256u * (u32)at.sb);
    pr = load(a.meta, bytes / 4u, po, 64u * (u32)at.sb);
  };

  f32x4 sum[R][NV], held[R][NV];   // held: kItems the first class's sums (LONG); kSlices 0 a pair of chains, 1 the slice
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int i = 0; i < NV; ++i) sum[r][i] = held[r][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float *meet = reinterpret_cast<float *>(smem);                      // [wave][NM][token][row]
  float *meet_gate = reinterpret_cast<float *>(smem + kWaves * kOwn);
  constexpr int NM = ORDER == kItems ? 4 : 1;                         // sums a wave hands on
  auto hand = [&](float *to, int r) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) to[(wave * NM + i) * 256 + 16 * (4 * q + j) + c] = ORDER == kItems ? sum[r][i][j] : held[r][1][j];
  };

  Pos at{first < a.nsb ? 0 : kPasses, first, 0, 0};
  load_w(at, 0);
  load_x(at);
  if (kPasses == 2 && at.pass == 2) hand(meet_gate, 0);   // no super-block: zeros
#pragma unroll 1
  while (at.pass < kPasses) {
    const Pos nx = next(at);
    // piece i of token k at i ^ k: the 16 tokens of a read lie in different banks
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x4 *>(own + (4 * i + q) * 256 + 16 * (c ^ (4 * i + q))) = v[i];
    float *mt = md + 32 * (lane & 3) + (lane >> 2);   // groups 2 (lane % 4) and + 1, token lane / 4
    mt[0] = u32_as_f32(pr.x);
    mt[16] = u32_as_f32(pr.z);
    mt[128] = u32_as_f32(pr.y);
    mt[144] = u32_as_f32(pr.w);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // row c's minima of groups q and q + 4, and its 8 scales (ggml get_scale_min_k4)
      const u32 sh = 8u * (u32)q;
      const u32 hz = h.z >> sh, hw = h.w >> sh;
      const float d = f16_to_f32(h.x), dmin = f16_to_f32(h.x >> 16);
      const float mn[2] = {dmin * (float)(hz & 63u), dmin * (float)(((hw >> 4) & 15u) | ((hz >> 2) & 48u))};
      const u32 sc[2] = {h.y & 0x3F3F3F3Fu, (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u)};
      const u32x4 wq[2] = {page_swap(c0), page_swap(c1)};
      if (r + 1 < R) load_w(at, r + 1);
      else if (R == 2 || nx.pass < kPasses) {
        load_w(nx, 0);
        if (kAheadX) load_x(nx);
      }
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        // -xs mn of groups 4 hf .. 4 hf + 3 where their sums lie: xs of token c, mn of row c, group 4 hf + q
        const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        const f32x16 xm = __builtin_amdgcn_mfma_f32_16x16x1f32(md[128 + 64 * hf + 16 * q + c], -mn[hf], zero16, 0, 0, 0);
        f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int pi = 0; pi < 2; ++pi) {   // page p: groups 2 p (low nibbles) and 2 p + 1
          const int p = 2 * hf + pi;
          f32x4 term[2], da[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            da[e] = *reinterpret_cast<const f32x4 *>(md + 16 * (2 * p + e) + 4 * q);   // of tokens 4 q .. 4 q + 3
            const float s = d * (float)((sc[hf] >> (8 * (2 * pi + e))) & 0xFFu);
            const u32 b0 = pi ? wq[hf].z : wq[hf].x, b1 = pi ? wq[hf].w : wq[hf].y;
            const long wa = pack8((b0 >> (4 * e)) & 0x0F0F0F0Fu, (b1 >> (4 * e)) & 0x0F0F0F0Fu);
            // the token's codes of group 2 p + e, bytes 16 (q % 2) + 8 (q / 2) ..
            const long xa = *reinterpret_cast<const long *>(own + c * 256 + 16 * ((4 * p + 2 * e + (q & 1)) ^ c) + 8 * (q >> 1));
            const i32x4 di = __builtin_amdgcn_mfma_i32_16x16x32_i8(xa, wa, i32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) term[e][i] = __builtin_fmaf((float)di[i], s, xm[8 * pi + 4 * e + i]);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if constexpr (ORDER == kItems) {
              sum[r][p][i] += q4k_q8_item(term[0][i], da[0][i], term[1][i], da[1][i]);
            } else {
              part[i] = __builtin_fmaf(term[0][i], da[0][i], part[i]);
              part[i] = __builtin_fmaf(term[1][i], da[1][i], part[i]);
            }
          }
          if (R > 1) __builtin_amdgcn_sched_barrier(0);   // keeps the pages' LDS reads from piling up in registers
        }
        if constexpr (ORDER == kSlices) sum[r][hf] += part;
        if (R == 2 && r == 1 && hf == 0) load_x(nx);
      }
      if constexpr (ORDER == kItems) {
        // item lanes 4 v + p and 4 (v + 8) + p meet, the butterfly's first step (!LONG: one super-block each, the second
        // joins the first by itself)
        if (LONG && nx.j != at.j) {
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            if (at.j == 0) { held[r][p] = sum[r][p]; sum[r][p] = f32x4{0.f, 0.f, 0.f, 0.f}; }
            else sum[r][p] += held[r][p];
          }
        }
      } else if (nx.j != at.j) {   // a chain is done, its halves' sum: (chain 0 + chain 1) + (chain 2 + chain 3)
        const f32x4 one = sum[r][0] + sum[r][1];
        sum[r][0] = sum[r][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        held[r][0] = at.j & 1 ? held[r][0] + one : one;
        if (at.j == 1) held[r][1] = held[r][0];
        if (at.j == 3) held[r][1] += held[r][0];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (kPasses == 2 && nx.pass == 1 && at.pass == 0) {
      hand(meet_gate, 0);
#pragma unroll
      for (int p = 0; p < NV; ++p) sum[0][p] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (LONG && nx.pass < kPasses) load_x(nx);
    at = nx;
  }
  if (R == 2) hand(meet_gate, 0);

  // ---- the waves' sums meet, in place of their own areas
  __syncthreads();
  hand(meet, R - 1);
  __syncthreads();
  auto total = [&](const float *from, int o) __attribute__((always_inline)) {
    if constexpr (ORDER == kItems) {   // the butterfly's steps 16 .. 1
      float pv[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        auto w = [&](int k) { return from[(k * 4 + p) * 256 + o]; };
        pv[p] = ((w(0) + w(4)) + (w(2) + w(6))) + ((w(1) + w(5)) + (w(3) + w(7)));
      }
      return 0.f + ((pv[0] + pv[2]) + (pv[1] + pv[3]));
    } else {                           // the slices in order
      float s = 0.f;
      for (int k = 0; k < a.nsb / per; ++k) s += from[k * 256 + o];
      return s;
    }
  };
  const int o = tid & 255, tok = t0 + o / 16, rw = row0 + (o & 15);
  const bool in = tok < a.tokens && rw < a.n;
  if constexpr (SWIGLU) {   // threads 0 .. 255 the gate, the others the up total
    const float s = total(tid < 256 ? meet_gate : meet, o);
    __syncthreads();
    if (tid >= 256) meet[o] = s;
    __syncthreads();
    if (tid < 256 && in) {
      float *p = a.y + (int64_t)tok * a.n + rw;
      const float y = act_fn(QMM_ACT_SILU, s, meet[o]);
      *p = a.accumulate ? *p + y : y;
    }
  } else if (tid < 256 && in) {
    float *p = (blockIdx.z ? a.y2 : a.y) + (int64_t)tok * a.n + rw;
    const float y = total(meet, o);
    *p = a.accumulate ? *p + y : y;
  }
}

template <bool TL, int ORDER, bool LONG>
int launch(int swiglu, const MArgs &a, hipStream_t s) {
  const dim3 grid((unsigned)(8 * ((a.tokens + 15) / 16)), (unsigned)((a.n + 127) / 128), a.y2 ? 2u : 1u);
  if (swiglu) mv_q8_mfma_kernel<TL, true, ORDER, LONG><<<grid, 64 * kWaves, 0, s>>>(a);
  else mv_q8_mfma_kernel<TL, false, ORDER, LONG><<<grid, 64 * kWaves, 0, s>>>(a);
  return launch_status();
}

// slices a wave of the tiled matvec kernel: K = 512 U NW, the least U <= 4 with NW <= 8 (qmm_mv_q4kt_q8); 0: none
int tiled_slices(int64_t k) {
  for (int u = 1; u <= 4; ++u)
    if (k / 512 % u == 0 && k / 512 / u <= 8) return u;
  return 0;
}

}  // namespace

// Whether qmm_mv_q8_mfma takes a call (the int8 matvec entry points ask; their argument checks hold). Nine tokens and
// more, and enough outputs for the grid: 1024 x 4096 at 24 tokens takes 9.7 us here, 9.5 in the matvec kernel; 4096 x 4096
// 7.9 against 14.0 at nine tokens and 15.5 against 71.8 at 63; 12288 x 4096 gate / up 18.7 against 52.7 and 54.9 against
// 284 (Q4_K blocks; the tiled layout 19.3 against 34.8 and 48.8 against 153). Tiled rows of K = 512 have one slice, so one
// wave works: 12288 gate / up at 33 tokens 25.0 against 22.7, at K = 1024 25.6 against 27.6.
// Shapes that the matvec kernels refuse (tiled: a K that does not split over their waves; too many rows) stay theirs.
bool qmm_mv_q8_mfma_fits(int fmt, int64_t k, int64_t n, int64_t tokens) {
  if (fmt != QMM_Q4_K && fmt != QMM_Q4_KT) return false;
  if (k % 256 || tokens < 9 || n * tokens < 32768 || tokens > 65535 || n > 65535 * 8) return false;
  if (tokens * k >= (1ll << 31) || n * (k / 256 * 144) >= (1ll << 32)) return false;   // 32-bit byte offsets
  if (fmt == QMM_Q4_K) return true;
  return n % 16 == 0 && k % 512 == 0 && k >= 1024 && tiled_slices(k) > 0;
}

// y2: a pair call (swiglu = 0). sliced: the call's one-token kernel is the K-sliced one (GGUF, K = 4096 or 8192).
int qmm_mv_q8_mfma(int fmt, int swiglu, int sliced, int64_t k, int64_t n, int64_t tokens, int accumulate, const void *xq,
                   const void *w, const void *w2, float *y, float *y2, hipStream_t s) {
  MArgs a{};
  a.n = (int)n; a.tokens = (int)tokens; a.nsb = (int)(k / 256);
  a.codes = static_cast<const u8 *>(xq);
  a.meta = reinterpret_cast<const float *>(a.codes + tokens * k);
  a.w = static_cast<const u8 *>(w); a.w2 = static_cast<const u8 *>(w2);
  a.y = y; a.y2 = y2; a.accumulate = accumulate;
  if (fmt == QMM_Q4_KT) {
    a.chains = 2; a.units = tiled_slices(k);
    return launch<true, kSlices, false>(swiglu, a, s);
  }
  if (sliced) {   // eight slices of 2 (K = 4096) or 4 super-blocks, a chain each
    a.chains = (int)(k / 2048); a.units = 1;
    return launch<false, kSlices, false>(swiglu, a, s);
  }
  return a.nsb > 2 * kWaves ? launch<false, kItems, true>(swiglu, a, s) : launch<false, kItems, false>(swiglu, a, s);
}
