// Decode matvecs on Q8_1 activations for 9 tokens and more (Q4_K, GGUF or tiled): g_mv_{fmt}_k{K}[_swiglu]_q8 of a
// batch of decoding sequences (S/gen_llm.py:1159-1197, :1288-1301), on the int8 MFMA.
//
//   y[t, r] (+)= sum over 32-value groups g of (di sc - xs mn) da,   di = sum q_w q_x (exact), sc = d sc_g,
//                                                                     mn = dmin m_g, (da, xs) the group's Q8_1 pair
//   swiglu: y (+)= silu(gate) up
//
// The matvec kernels read every weight once per two tokens (GGUF) or eight (tiled) and spend a v_dot4 per four products;
// 24 tokens through 2 x 12288 x 4096 took 122 us, against 7 us of weight bytes (here 26.5). Here a weight is read once per 32 tokens
// and 16 x 16 products of a group take one v_mfma_i32_16x16x32_i8 a wave: what is left is the fixup of each group's
// 256 sums (convert, scale, fma: 12 vector instructions a wave), which bounds it. The codes are taken as 16 (q - 8), so
// a group adds (16 di - 128 xs) (sc / 16) da - xs (mn - 8 sc) da: the first sums are free of the codes' common offset (with
// unsigned codes the two terms cancel, and the result was twice as far from 64 bits), and the second term,
// small, is a product of f32 matrices over the groups: two v_mfma_f32_16x16x4_f32 a super-block.
//
// A workgroup: 16 weight rows (swiglu: 16 of each matrix) x 16 NT tokens, kWaves waves. Wave v takes super-blocks v,
// v + kWaves, ... of all rows: it brings the super-block's codes and pairs of its tokens into registers (coalesced through its own
// LDS: a load in which every lane reads its own token or row takes the address unit 64 cycles), then streams the
// super-block of the rows past them. The waves' sums meet in LDS at the end, in wave order.
//
// MFMA operands: lane (c, q) = (lane % 16, lane / 16) holds 8 K values of weight row / token c; which 8 does not matter
// while both agree. A page's 32 code bytes are two groups (low and high nibbles). Lane (c, q) loads bytes 16 q .. of two
// pages (64 bytes of a row from four lanes); exchanging register halves between lanes 0-31 and 32-63 (v_permlane32_swap)
// leaves bytes 16 (q % 2) + 8 (q / 2) .. + 7 of the one page in the first two registers and of the other in the last
// two. A token's 64 codes of a page's two groups go through the same exchange, so they meet the weights at the same K.
#include "common.hpp"

using namespace qmm;

namespace {

typedef __attribute__((ext_vector_type(4))) u32 u32x4;


struct MArgs {
  int n, tokens, nsb;           // rows of a matrix, tokens, super-blocks a row
  const u8 *codes;              // planar Q8_1: codes [tokens][K], then pairs f32 [tokens][K / 32][2]
  const float *meta;
  const u8 *w, *w2;
  float *y;
  int accumulate;
};

// registers (a, b) of a 16-byte piece: halves of the wave exchanged so that a belongs to one page, b to the other
__device__ __forceinline__ void page_swap(u32 &a, u32 &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ long pack8(u32 a, u32 b) { return (long)(((uint64_t)b << 32) | a); }

template <bool TL, bool SWIGLU, int NT, int kRowBlocks, int kWaves>
__global__ __launch_bounds__(64 * kWaves, kWaves == 8 ? 4 : 3) void mv_q8_mfma_kernel(MArgs a) {
  // LDS bytes a wave: the codes of 16 tokens, per 16 tokens da and xs da [group][token], d sc of 16 rows [group][row]
  constexpr int kCode = 16 * 256, kMeta = NT * 1024, kScale = 8 * 16 * 4;
  constexpr int kOwn = kCode + kMeta + kScale;
  constexpr int kPair = kRowBlocks > 1 ? 2 : 1;                           // row blocks that meet in LDS at a time
  constexpr int kRed = kPair * NT * 256 * 4;
  __shared__ __align__(16) u8 smem[kWaves * (kOwn > kRed ? kOwn : kRed)];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, q = lane >> 4;
  const u32 K = (u32)a.nsb * 256u, RB = (u32)a.nsb * 144u;   // all byte offsets fit 32 bits (qmm_mv_q8_mfma_fits)
  constexpr int kOut = 16 * (SWIGLU ? kRowBlocks / 2 : kRowBlocks);       // output rows a workgroup
  const int row0 = (int)blockIdx.x * kOut, t0 = (int)blockIdx.y * 16 * NT;
  u8 *own = smem + wave * kOwn;

  // the lane's row of each row block (rows past n read row n - 1 and are not stored)
  u32 wr[kRowBlocks];   // byte offset in its matrix
#pragma unroll
  for (int r = 0; r < kRowBlocks; ++r) {
    const bool up = SWIGLU && r >= kRowBlocks / 2;   // swiglu: gate blocks, then their up blocks
    const int row = min(row0 + 16 * (up ? r - kRowBlocks / 2 : r) + c, a.n - 1);
    // tiled: the lane's plane q of its 16-row block (the header lies 512 + 1024 q + 32 (row % 16) before it)
    wr[r] = TL ? (u32)(row >> 4) * 16u * RB + 512u + 1024u * (u32)q + 64u * (u32)(row & 15) : (u32)row * RB;
  }
  const u32 hoff = 512u + 1024u * (u32)q + 32u * (u32)c;   // tiled: rows of a block are the lanes c (row0 % 16 = 0)
  constexpr bool kTwoSums = !SWIGLU && NT == 1;   // a wave's even and odd super-blocks summed apart, where registers allow
  f32x4 acc[kRowBlocks][NT], alt[kRowBlocks][NT];
#pragma unroll
  for (int r = 0; r < kRowBlocks; ++r)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[r][t] = alt[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int sb = wave; sb < a.nsb; sb += kWaves) {
    // ---- the super-block's weights of the first row block, then the tokens
    uint4 c0[2], c1[2], hd[2];
    auto load_w = [&](int r) __attribute__((always_inline)) {
      const u8 *m = SWIGLU && r >= kRowBlocks / 2 ? a.w2 : a.w;
      if constexpr (TL) {
        // unit sb / 2 (4608 bytes): page p's bytes 16 h .. in plane 2 (p % 2) + h, at 64 row + 32 (sb % 2) + 16 (p / 2);
        // lane q reads page q / 2 (and 2 + q / 2), half q % 2: plane q
        const u8 *u = m + (int64_t)(sb >> 1) * 4608;
        c0[r & 1] = *reinterpret_cast<const uint4 *>(u + 32 * (sb & 1) + wr[r]);
        c1[r & 1] = *reinterpret_cast<const uint4 *>(u + 32 * (sb & 1) + 16 + wr[r]);
        hd[r & 1] = *reinterpret_cast<const uint4 *>(u + 16 * (sb & 1) + (wr[r] - hoff));
      } else {
        const u8 *b = m + (int64_t)sb * 144;
        c0[r & 1] = *reinterpret_cast<const uint4 *>(b + 16 + (wr[r] + 16u * (u32)q));
        c1[r & 1] = *reinterpret_cast<const uint4 *>(b + 80 + (wr[r] + 16u * (u32)q));
        hd[r & 1] = *reinterpret_cast<const uint4 *>(b + wr[r]);
      }
    };
    load_w(0);
    u32 xb[NT][8][2];      // token codes of group g: two dwords
    float sx[NT][2];       // xs da of the lane's token, groups q and q + 4
    float *md = reinterpret_cast<float *>(own + kCode);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint4 v[4], m;
#pragma unroll
      for (int i = 0; i < 4; ++i) {   // 16 lanes a token: its 256 codes
        const int tok = min(t0 + 16 * t + 4 * i + q, a.tokens - 1);
        v[i] = *reinterpret_cast<const uint4 *>(a.codes + sb * 256 + ((u32)tok * K + 16u * (u32)c));
      }
      {                               // four lanes a token: its 8 pairs
        const int tok = min(t0 + 16 * t + (lane >> 2), a.tokens - 1);
        m = *reinterpret_cast<const uint4 *>(reinterpret_cast<const u8 *>(a.meta) + sb * 64 +
                                             ((u32)tok * (K / 4u) + 16u * (u32)(lane & 3)));
      }
      // piece i of token k at i ^ k: the 16 tokens of a read lie in different banks
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<uint4 *>(own + (4 * i + q) * 256 + 16 * (c ^ (4 * i + q))) = v[i];
      float *mt = md + 256 * t + 32 * (lane & 3) + (lane >> 2);   // groups 2 (lane % 4) and + 1, token lane / 4
      const float d0 = u32_as_f32(m.x), d1 = u32_as_f32(m.z);
      mt[0] = d0;
      mt[16] = d1;
      mt[128] = d0 * u32_as_f32(m.y);   // exact: 11 x 12 bits
      mt[144] = d1 * u32_as_f32(m.w);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        uint4 x = *reinterpret_cast<const uint4 *>(own + c * 256 + 16 * ((4 * p + q) ^ c));
        page_swap(x.x, x.z);
        page_swap(x.y, x.w);
        xb[t][2 * p][0] = x.x; xb[t][2 * p][1] = x.y;
        xb[t][2 * p + 1][0] = x.z; xb[t][2 * p + 1][1] = x.w;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) sx[t][j] = md[256 * t + 128 + 16 * (q + 4 * j) + c];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    // ---- the row blocks, the next one's loads in flight
#pragma unroll
    for (int r = 0; r < kRowBlocks; ++r) {
      if (r + 1 < kRowBlocks) load_w(r + 1);
      uint4 x = c0[r & 1], z = c1[r & 1];
      const uint4 h = hd[r & 1];
      page_swap(x.x, x.z);
      page_swap(x.y, x.w);
      page_swap(z.x, z.z);
      page_swap(z.y, z.w);
      const u32 pg[4][2] = {{x.x, x.y}, {x.z, x.w}, {z.x, z.y}, {z.z, z.w}};
      // row c's scales of groups q and q + 4 (ggml get_scale_min_k4); the d sc go to the lanes that hold its sums
      const u32 sh = 8u * (u32)q;
      const u32 y0 = h.y >> sh, z0 = h.z >> sh, w0 = h.w >> sh;
      const float d = f16_to_f32(h.x), dmin = f16_to_f32(h.x >> 16);
      const float sc0 = d * (float)(y0 & 63u), sc1 = d * (float)((w0 & 15u) | ((y0 >> 2) & 48u));
      const float mn0 = dmin * (float)(z0 & 63u) - 8.f * sc0, mn1 = dmin * (float)(((w0 >> 4) & 15u) | ((z0 >> 2) & 48u)) - 8.f * sc1;
      float *sl = reinterpret_cast<float *>(own + kCode + kMeta);
      sl[lane] = sc0 * 0.0625f;
      sl[64 + lane] = sc1 * 0.0625f;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      // a super-block's sum in two chains of four groups before it joins the wave's: short chains, and so rounding
      // errors, as the matvec kernels' trees have them
      f32x4 part[2][NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        part[0][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(-mn0, sx[t][0], zero, 0, 0, 0);
        part[1][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(-mn1, sx[t][1], zero, 0, 0, 0);
      }
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        const f32x4 s = *reinterpret_cast<const f32x4 *>(sl + 16 * g + 4 * q);   // rows 4 q .. 4 q + 3 of group g
        const u32 e0 = pg[g >> 1][0], e1 = pg[g >> 1][1];
        // 16 (q - 8) as int8: the nibble in the high half, its top bit flipped
        const long wa = (g & 1) ? pack8((e0 & 0xF0F0F0F0u) ^ 0x80808080u, (e1 & 0xF0F0F0F0u) ^ 0x80808080u)
                                : pack8(((e0 << 4) & 0xF0F0F0F0u) ^ 0x80808080u, ((e1 << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const float da = md[256 * t + 16 * g + c];
          const i32x4 di = __builtin_amdgcn_mfma_i32_16x16x32_i8(wa, pack8(xb[t][g][0], xb[t][g][1]), i32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) part[g >> 2][t][i] = __builtin_fmaf((float)di[i], s[i] * da, part[g >> 2][t][i]);
        }
        if (g & 1) __builtin_amdgcn_sched_barrier(0);   // keeps the groups' LDS reads from piling up in registers
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const f32x4 v = acc[r][t] + (part[0][t] + part[1][t]);
        if constexpr (!kTwoSums) {
          acc[r][t] = v;
        } else {   // the two swap places after every super-block
          acc[r][t] = alt[r][t];
          alt[r][t] = v;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }

  // ---- the waves' sums meet, two row blocks at a time (swiglu: a gate and its up block): [wave][block][token][row]
  float *red = reinterpret_cast<float *>(smem);
#pragma unroll
  for (int rr = 0; rr < kRowBlocks / kPair; ++rr) {
    __syncthreads();   // the waves' own areas (or the sums before) are done with
#pragma unroll
    for (int u = 0; u < kPair; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        *reinterpret_cast<f32x4 *>(&red[((wave * kPair + u) * NT + t) * 256 + 16 * c + 4 * q]) =
            SWIGLU ? acc[rr + kRowBlocks / 2 * u][t] : kTwoSums ? acc[kPair * rr + u][t] + alt[kPair * rr + u][t] : acc[kPair * rr + u][t];
    __syncthreads();
    for (int o = tid; o < (SWIGLU ? 1 : kPair) * NT * 256; o += 64 * kWaves) {
      auto total = [&](int at) {   // of the waves, as a tree
        float e[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) e[w] = red[w * kPair * NT * 256 + at];
        if constexpr (kWaves == 4) return (e[0] + e[1]) + (e[2] + e[3]);
        else return ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
      };
      float v = total(o);
      const int u = o / (NT * 256), tok = t0 + (o % (NT * 256)) / 16;
      const int row = row0 + 16 * (SWIGLU ? rr : kPair * rr + u) + (o & 15);
      if (tok < a.tokens && row < a.n) {
        if constexpr (SWIGLU) v = act_fn(QMM_ACT_SILU, v, total(NT * 256 + o));
        float *p = a.y + (int64_t)tok * a.n + row;
        *p = a.accumulate ? *p + v : v;
      }
    }
  }
}

template <bool TL, bool SWIGLU, int NT, int R, int W>
int launch(const MArgs &a, hipStream_t s) {
  constexpr int kOut = 16 * (SWIGLU ? R / 2 : R);
  const dim3 grid((unsigned)((a.n + kOut - 1) / kOut), (unsigned)((a.tokens + 16 * NT - 1) / (16 * NT)));
  mv_q8_mfma_kernel<TL, SWIGLU, NT, R, W><<<grid, 64 * W, 0, s>>>(a);
  return launch_status();
}
// Eight waves a workgroup of 16 rows (swiglu: 16 of each matrix), so that 4096 rows fill the chip (with 64 rows a
// workgroup 4096 x 4096 at 9 tokens took 15.2 us, with 16 7.9); swiglu past 16 tokens four waves, whose registers hold
// both matrices' sums (eight would spill: 24 tokens 44.9 -> 26.5 us at 12288 x 4096; plain 20.6 us with eight waves, 28.4
// with four at 4096 x 12288).
template <bool TL, bool SWIGLU>
int launch_nt(const MArgs &a, hipStream_t s) {
  constexpr int R = SWIGLU ? 2 : 1;
  return a.tokens <= 16 ? launch<TL, SWIGLU, 1, R, 8>(a, s) : launch<TL, SWIGLU, 2, R, SWIGLU ? 4 : 8>(a, s);
}

}  // namespace

// Whether qmm_mv_q8_mfma takes a call (the int8 matvec entry points ask; their argument checks hold). Nine tokens and
// more, and enough outputs for the grid: 1024 x 4096 at 24 tokens takes 9.4 us here, 9.0 in the matvec kernel; 4096 x 4096
// 7.9 against 11.9 at nine tokens and 14.4 against 46.6 at 63; 12288 x 4096 gate / up 19.6 against 57.7 and 49 against 287
// (Q4_K blocks; the tiled layout 17.5 against 36 and 45 against 160).
// Shapes that the matvec kernels refuse (tiled: a K that does not split over their waves; too many rows) stay theirs.
bool qmm_mv_q8_mfma_fits(int fmt, int64_t k, int64_t n, int64_t tokens) {
  if (fmt != QMM_Q4_K && fmt != QMM_Q4_KT) return false;
  if (k % 256 || tokens < 9 || n * tokens < 32768 || tokens > 65535 || n > 65535 * 8) return false;
  if (tokens * k >= (1ll << 31) || n * (k / 256 * 144) >= (1ll << 32)) return false;   // 32-bit byte offsets
  if (fmt == QMM_Q4_K) return true;
  bool split = false;   // K = 512 U NW, U <= 4 slices a wave, NW <= 8 waves (qmm_mv_q4kt_q8)
  for (int u = 1; u <= 4; ++u) split = split || (k / 512 % u == 0 && k / 512 / u <= 8);
  return n % 16 == 0 && k % 512 == 0 && split;
}

int qmm_mv_q8_mfma(int fmt, int swiglu, int64_t k, int64_t n, int64_t tokens, int accumulate, const void *xq,
                   const void *w, const void *w2, float *y, hipStream_t s) {
  MArgs a{};
  a.n = (int)n; a.tokens = (int)tokens; a.nsb = (int)(k / 256);
  a.codes = static_cast<const u8 *>(xq);
  a.meta = reinterpret_cast<const float *>(a.codes + tokens * k);
  a.w = static_cast<const u8 *>(w); a.w2 = static_cast<const u8 *>(w2);
  a.y = y; a.accumulate = accumulate;
  if (fmt == QMM_Q4_KT) return swiglu ? launch_nt<true, true>(a, s) : launch_nt<true, false>(a, s);
  return swiglu ? launch_nt<false, true>(a, s) : launch_nt<false, false>(a, s);
}
