// SPDX-License-Identifier: Apache-2.0
// MFMA decode attention over pages of one byte per element, for gfx950: INT8
// codes with per-channel scales (kind-0 work items of a plan), and E4M3 codes
// with a scale per (token, head), planned on the device.
//
// Reference: the fused decode with per-channel antiquant of
// pkg/methods/int8_dynamic/attention_backend.py:173-205 (antiquant_mode 0,
// offset 0): K = code * k_aq, V = code * v_aq per (kv head, dim), softmax in
// fp32; and the values of Fp8PerTokenHeadSemantics.dequantize
// (pkg/methods/fp8_per_token_head/semantics.py:63-65), K = code * k_scale per
// (token, kv head), which the reference has no device read path for.  Cache
// layout [NB, Bs, KVH, D] bytes: one token of one kv head is a D-byte row, the
// rows of a token's heads are adjacent.
//
// One wave per (work item, kv head), 32-token tiles double-buffered in the
// wave's 16 KB of LDS (32 KB at D = 256): global_load_lds DMA with 16-byte lanes
// brings whole rows (cache lines) while the previous tile computes.  On
// config 2 this ran 117 us against 126 us for register tiles loaded 32 bytes
// a lane (two requests per line), at 118 instead of 232 VGPRs.
//
// QK^T (v_mfma_f32_16x16x32_f16, S^T = K * Q'^T), per 16-token group j:
//   A = key codes, row = token, k = dim.  Lane (g, n) = (lane / 16, lane % 16)
//       reads the D/4 contiguous bytes from D/4 g on of token row n and takes
//       dims D/4 g + 8s + i at k-step s.  INT8: a byte b becomes the exact fp16
//       code: v_perm places (b ^ 0x80) under the exponent byte 0x64 (fp16
//       1024 + b + 128) and one packed subtract of 1152 leaves b.
//   B = Q' = q * k_aq (exact in fp32 for bf16 / fp16 activations) scaled by a
//       power of two per head into fp16 range, split into hi + lo fp16 parts
//       (~22 bits): two MFMAs, or with GQA groups of at most 8 heads one MFMA
//       whose columns n and n + 8 carry the two parts (FOLD).  The softmax
//       scale * log2(e) and the inverse power of two multiply the fp32 scores.
//   E4M3: A is the dense row the gather would leave, code * scale rounded to the
//       query's dtype (e4m3_rows); B is the query as it is, one MFMA.
// PV (O = P * V), one 32-token k-step per tile:
//   A = P (fp16), row = query head, k = token: lane (g, n) already holds p of
//       tokens 16j + 4g + r (j = 0, 1; r = 0..3) for head n from the QK
//       output layout, and uses exactly those tokens as its 8 k-values.
//   B = value codes, column n of tile t = dim (D/16) n + t: the lane reads bytes
//       [(D/16) n, (D/16) (n + 1)) of its 8 token rows and builds code pairs from
//       byte t of two rows (v_perm + or + packed subtract, exact).
//   v_aq multiplies the output per dim at the end.
//   E4M3: the rows' 4 x 4 byte blocks are transposed (v_perm) and become the
//       gather's dense rows likewise; A is p as hi + lo parts of the query's
//       dtype (16 bits of it at least), two MFMAs.
// Online softmax in the log2 domain; each item leaves (m, l, o) per query head
// for the log-sum-exp combine.
//
// Tiles start on the 16-aligned position at or below the item's start, so
// with block_size % 16 == 0 every 16-token group lies in one page (one
// uniform page lookup per group).  Positions outside [start, end) are masked;
// their addresses are clamped to the group holding end - 1 and page ids to
// [0, num_blocks), so every load stays inside the cache and the table row.
#include <algorithm>

#include "kvq_common.h"
#include "kvq_decode.h"

namespace {

using namespace kvq;

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));

constexpr int kTile = 32;  // tokens per tile: two groups of 16
constexpr uint32_t kExp64 = 0x64646464u;  // 0x64: high byte of fp16 1024 + u, u < 256
constexpr uint32_t kFlip = 0x80808080u;   // int8 code -> excess-128 byte

__device__ __forceinline__ h8 as_h8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  u4v v = {a, b, c, d};
  return __builtin_bit_cast(h8, v);
}
__device__ __forceinline__ uint32_t minus1152(uint32_t pair) {
  const h2 v = __builtin_bit_cast(h2, pair) - h2{1152.0f16, 1152.0f16};
  return __builtin_bit_cast(uint32_t, v);
}

// Two fp32 values as a bf16 / fp16 pair (round to nearest even), and the pair back.
__device__ __forceinline__ uint32_t pack2(float lo, float hi, bf16) { return bf16x2_bits(lo, hi); }
__device__ __forceinline__ uint32_t pack2(float lo, float hi, f16) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{lo, hi}), h2));
}
__device__ __forceinline__ f2 widen2(uint32_t w, bf16) {
  return f2{__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)};
}
__device__ __forceinline__ f2 widen2(uint32_t w, f16) {
  const h2 v = __builtin_bit_cast(h2, w);
  return f2{static_cast<float>(v[0]), static_cast<float>(v[1])};
}

// E4M3 codes (bytes 0, 1 or 2, 3 of x) times their scales, as a pair of dense
// values in T: fp32 product, one rounding, to the bit what the gather leaves.
// (Exact codes with the scales on the fp32 scores and probabilities take 66.5 us
// a step of 32 requests of 0.5K-8K positions, 32 heads on 8 kv heads, and these
// 74.5; but the decode would then answer otherwise than the same rows gathered:
// 0.0047 apart, 0.06 at the worst element.)
template <bool HI, typename T>
__device__ __forceinline__ uint32_t e4m3_rows(uint32_t x, float s0, float s1, T) {
  const auto v = __builtin_amdgcn_cvt_pk_f32_fp8(x, HI);
  return pack2(v[0] * s0, v[1] * s1, T{});
}
__device__ __forceinline__ f4 mfma_q(u4v a, u4v b, f4 c, bf16) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a),
                                                 __builtin_bit_cast(b8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma_q(u4v a, u4v b, f4 c, f16) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a),
                                                __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

// Exact fp16 codes (bytes 2u, 2u + 1 of the excess-128 word x).
template <int U>
__device__ __forceinline__ uint32_t key_pair(uint32_t x) {
  // byte0 = x.b[2U], byte1 = 0x64, byte2 = x.b[2U + 1], byte3 = 0x64
  constexpr uint32_t sel = (2u * U) | (4u << 8) | ((2u * U + 1u) << 16) | (4u << 24);
  return minus1152(__builtin_amdgcn_perm(kExp64, x, sel));
}

// Exact fp16 codes (byte K of excess-128 word lo, byte K of word hi).
template <int K>
__device__ __forceinline__ uint32_t value_pair(uint32_t lo, uint32_t hi) {
  // byte0 = lo.b[K], byte1 = 0, byte2 = hi.b[K], byte3 = 0
  constexpr uint32_t sel = 0x0c000c00u | K | ((4u + K) << 16);
  return minus1152(__builtin_amdgcn_perm(hi, lo, sel) | 0x64006400u);
}

__device__ __forceinline__ uint32_t h2_bits(_Float16 a, _Float16 b) {
  return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, a)) |
         (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, b)) << 16);
}

// One tile's codes in registers.  k[j][u]: the 16 bytes from D/4 g + 16 u on of
// token 16j + n; v[j][r][w]: word w of bytes [D/16 n, D/16 (n + 1)) of token
// 16j + 4g + r; ksc (E4M3): scale of token 16j + n, vsc: of tokens 16j + 4g + r.
template <int D, bool FP8>
struct TileRegs {
  uint4 k[2][D / 64];
  uint32_t v[2][4][D / 64];
  float ksc[FP8 ? 2 : 1];
  f4 vsc[FP8 ? 2 : 1];
};

struct WaveCtx {
  const int8_t* kc;
  const int8_t* vc;
  const float* ks;    // E4M3 scales [NB, Bs, KVH]
  const float* vs;
  const void* bt;     // this request's table row
  int bt64;           // its entries are int64
  int64_t nb;
  int bs, kvh, h, g, n;
  int last_group;     // 16-aligned start of the group holding end - 1
  __device__ __forceinline__ int64_t page(int i) const {
    const int64_t b0 = bt64 ? static_cast<const int64_t*>(bt)[i]
                            : static_cast<int64_t>(static_cast<const int32_t*>(bt)[i]);
    return b0 < 0 ? 0 : (b0 >= nb ? nb - 1 : b0);
  }
};

// ---- LDS-staged tiles -------------------------------------------------------
// The tile's 32 key rows and 32 value rows (D bytes each) arrive by DMA in the
// wave's LDS, 16-byte lanes, D/16 lanes per row, so every request is a whole
// line.  Chunk c of row t (16 bytes) sits at position c ^ (t % (D/16)): the
// operand reads of 16 rows spread over the banks.  The operand registers are
// then filled from LDS in the layout compute_tile reads.  E4M3: one more DMA
// brings the 32 key scales and the 32 value scales behind the rows.
template <int D, bool FP8>
constexpr int tile_bytes() { return 2 * kTile * D + (FP8 ? 8 * kTile : 0); }
template <int D, bool FP8>
constexpr int tile_dmas() { return D / 16 + (FP8 ? 1 : 0); }

template <int D, bool FP8>
__device__ __forceinline__ void issue_tile_dma(char* buf, const WaveCtx& c, int p, int lane) {
  constexpr int CH = D / 16;   // chunks per row
  constexpr int RPI = 64 / CH; // rows per instruction
  int64_t first[2];            // first token row of each group
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    int gt = p + 16 * j;
    gt = gt < c.last_group ? gt : c.last_group;
    const int64_t row0 = c.page(gt / c.bs) * c.bs + gt % c.bs;
    first[j] = row0;
#pragma unroll
    for (int part = 0; part < 16 / RPI; ++part) {
      const int r = RPI * part + lane / CH;        // row of the group
      const int chunk = (lane % CH) ^ (r % CH);    // global chunk for LDS position lane % CH
      const int64_t off = ((row0 + r) * c.kvh + c.h) * D + 16 * chunk;
      char* dst = buf + (16 * j + RPI * part) * D;  // the DMA adds 16 * lane
      dma16(c.kc + off, dst);
      dma16(c.vc + off, dst + kTile * D);
    }
  }
  if constexpr (FP8) {
    const int64_t row = (lane & 16 ? first[1] : first[0]) + (lane & 15);
    dma4((lane & 32 ? c.vs : c.ks) + row * c.kvh + c.h, buf + 2 * kTile * D);
  }
}

template <int D, bool FP8>
__device__ __forceinline__ void read_tile_lds(TileRegs<D, FP8>& t, const char* buf, int g, int n) {
  constexpr int CH = D / 16;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const char* kr = buf + (16 * j + n) * D;  // row % CH == n % CH
#pragma unroll
    for (int u = 0; u < D / 64; ++u)
      t.k[j][u] = *reinterpret_cast<const uint4*>(kr + 16 * (((D / 64) * g + u) ^ (n % CH)));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int vrow = 16 * j + 4 * g + r;
      const char* vr = buf + kTile * D + vrow * D;
      if constexpr (D == 128) {
        const uint2 x =
            *reinterpret_cast<const uint2*>(vr + 16 * ((n / 2) ^ (vrow % 8)) + 8 * (n % 2));
        t.v[j][r][0] = x.x;
        t.v[j][r][1] = x.y;
      } else {
        const uint4 x = *reinterpret_cast<const uint4*>(vr + 16 * (n ^ (vrow % 16)));
        t.v[j][r][0] = x.x;
        t.v[j][r][1] = x.y;
        t.v[j][r][2] = x.z;
        t.v[j][r][3] = x.w;
      }
    }
    if constexpr (FP8) {
      const float* sc = reinterpret_cast<const float*>(buf + 2 * kTile * D) + 16 * j;
      t.ksc[j] = sc[n];
      t.vsc[j] = *reinterpret_cast<const f4*>(sc + kTile + 4 * g);
    }
  }
}

// INT8 at 256 dims: p's (and o's) lift on the way through fp16, so that the two
// parts of a p down to 2^-28 keep their bits and one is lost only below 2^-39.
// (Against 64 bits, fp32 activations, 300 - 16K positions: 1.4e-7 - 2.1e-7, where the
// fp32 kernel these calls had before was 2.7e-7 - 3.3e-7 off.)
template <int D>
constexpr float kLift = D == 256 ? 16384.0f : 1.0f;

template <int D>
struct SoftmaxState {
  float m;    // running max of head n (log2 domain), same in the 4 lane groups
  float l;    // this lane's partial sum of p
  f4 o[D / 16];  // o[t][r]: head 4g + r, dim (D/16) n + t
};

// x + (x of lane n ^ 8 in the same 16-lane row): v_add_f32 with a DPP
// row_ror:8 operand.
__device__ __forceinline__ float add_ror8(float x) {
  const int y = __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false);
  return x + __int_as_float(y);
}

// pb, pe: the item's positions; pen: where those of the lane's column end.
// FOLD (GQA groups of at most 8 heads): qh carries the hi part of head n in
// columns n < 8 and the lo part of head n - 8 in columns n >= 8, so one MFMA
// per k-step gives both partial scores and a rotate-by-8 add sums them (both
// lanes then hold head n % 8's score; ql unused).
template <typename TQ, int D, bool FOLD, bool FP8>
__device__ __forceinline__ void compute_tile(const TileRegs<D, FP8>& t, int p, int pb, int pe,
                                             int pen, const u4v (&qh)[D / 32], const u4v (&ql)[D / 32],
                                             float sc, int g, SoftmaxState<D>& st) {
  // ---- S^T = K * Q'^T: 2 groups of 16 tokens ----
  f4 s[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    s[j] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      const uint4& kw = t.k[j][ks / 2];
      const uint32_t w0 = ks % 2 ? kw.z : kw.x, w1 = ks % 2 ? kw.w : kw.y;
      if constexpr (FP8) {
        const float k = t.ksc[j];
        const u4v a = {e4m3_rows<false>(w0, k, k, TQ{}), e4m3_rows<true>(w0, k, k, TQ{}),
                       e4m3_rows<false>(w1, k, k, TQ{}), e4m3_rows<true>(w1, k, k, TQ{})};
        s[j] = mfma_q(a, qh[ks], s[j], TQ{});
      } else {
        const uint32_t x0 = w0 ^ kFlip, x1 = w1 ^ kFlip;
        const h8 a = as_h8(key_pair<0>(x0), key_pair<1>(x0), key_pair<0>(x1), key_pair<1>(x1));
        s[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, __builtin_bit_cast(h8, qh[ks]), s[j], 0,
                                                      0, 0);
        if (!FOLD)
          s[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, __builtin_bit_cast(h8, ql[ks]), s[j],
                                                        0, 0, 0);
      }
    }
  }
  if (FOLD) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[j][r] = add_ror8(s[j][r]);
  }
  // ---- online softmax for head n over tokens 16j + 4g + r ----
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = p + 16 * j + 4 * g + r;
      const float x = s[j][r] * sc;
      const float v = (tok >= pb && tok < pen) ? x : -INFINITY;
      s[j][r] = v;
      mx = fmaxf(mx, v);
    }
  mx = max_rows4(mx);
  const float m_new = fmaxf(st.m, mx);
  // a fully masked prefix keeps m = -inf: nothing to rescale, p = 0
  const float m_use = m_new == -INFINITY ? 0.0f : m_new;
  const float alpha = st.m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(st.m - m_use);
  st.m = m_new;
  float psum = 0.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float pv = __builtin_amdgcn_exp2f(s[j][r] - m_use);  // exp2(-inf) = 0
      s[j][r] = pv;
      psum += pv;
    }
  st.l = st.l * alpha + psum;
  // o rows are heads 4g + r: their alphas live in lanes 4g + r
  if (__any(alpha != 1.0f)) {
    float a[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = __shfl(alpha, 4 * g + r, 64);
#pragma unroll
    for (int tt = 0; tt < D / 16; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) st.o[tt][r] *= a[r];
  }
  // ---- O += P * V: one k-step of 32 tokens ----
  if constexpr (FP8) {
    uint32_t ph[4], pl[4];  // p of the lane's 8 tokens, hi and lo parts
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = u / 2, r = 2 * (u % 2);
      ph[u] = pack2(s[j][r], s[j][r + 1], TQ{});
      const f2 hi = widen2(ph[u], TQ{});
      pl[u] = pack2(s[j][r] - hi[0], s[j][r + 1] - hi[1], TQ{});
    }
    const u4v ah = {ph[0], ph[1], ph[2], ph[3]}, al = {pl[0], pl[1], pl[2], pl[3]};
    // rows past the item may hold NaN codes and scales (their p is 0)
    const bool whole = p >= pb && p + kTile <= pe;  // uniform
    f4 vsc[2] = {t.vsc[0], t.vsc[1]};
    if (!whole) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int tok = p + 16 * j + 4 * g + r;
          vsc[j][r] = tok >= pb && tok < pe ? vsc[j][r] : 0.0f;
        }
    }
#pragma unroll
    for (int w = 0; w < D / 64; ++w) {
      uint32_t tr[4][2];  // byte b of the 8 tokens' words, tokens 4j .. 4j + 3 in [b][j]
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        uint32_t x[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = t.v[j][r][w];
        if (!whole) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int tok = p + 16 * j + 4 * g + r;
            x[r] = tok >= pb && tok < pe ? x[r] : 0u;
          }
        }
        const uint32_t l01 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400u);
        const uint32_t h01 = __builtin_amdgcn_perm(x[1], x[0], 0x07030602u);
        const uint32_t l23 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400u);
        const uint32_t h23 = __builtin_amdgcn_perm(x[3], x[2], 0x07030602u);
        tr[0][j] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
        tr[1][j] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
        tr[2][j] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
        tr[3][j] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const u4v v = {e4m3_rows<false>(tr[b][0], vsc[0][0], vsc[0][1], TQ{}),
                       e4m3_rows<true>(tr[b][0], vsc[0][2], vsc[0][3], TQ{}),
                       e4m3_rows<false>(tr[b][1], vsc[1][0], vsc[1][1], TQ{}),
                       e4m3_rows<true>(tr[b][1], vsc[1][2], vsc[1][3], TQ{})};
        f4& o = st.o[4 * w + b];
        o = mfma_q(ah, v, o, TQ{});
        o = mfma_q(al, v, o, TQ{});
      }
    }
  } else {
    // at 256 dims p goes as fp16 hi + lo parts, at 128 as one fp16
    constexpr bool kSplitP = kLift<D> != 1.0f;
    auto halves = [](const f4 (&x)[2]) {
      return as_h8(h2_bits(static_cast<_Float16>(x[0][0]), static_cast<_Float16>(x[0][1])),
                   h2_bits(static_cast<_Float16>(x[0][2]), static_cast<_Float16>(x[0][3])),
                   h2_bits(static_cast<_Float16>(x[1][0]), static_cast<_Float16>(x[1][1])),
                   h2_bits(static_cast<_Float16>(x[1][2]), static_cast<_Float16>(x[1][3])));
    };
    if constexpr (kSplitP) {
#pragma unroll
      for (int j = 0; j < 2; ++j) s[j] *= kLift<D>;
    }
    const h8 a = halves(s);
    h8 al = a;
    if constexpr (kSplitP) {
      f4 rest[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          rest[j][r] = s[j][r] - static_cast<float>(static_cast<_Float16>(s[j][r]));
      al = halves(rest);
    }
    // the lane's 8 tokens (i = 4j + r), four dims per word
#pragma unroll
    for (int w = 0; w < D / 64; ++w) {
      uint32_t x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = t.v[i / 4][i % 4][w] ^ kFlip;
#define KVQ_PV_TILE(K)                                                                       \
  {                                                                                          \
    const h8 b = as_h8(value_pair<K>(x[0], x[1]), value_pair<K>(x[2], x[3]),                 \
                       value_pair<K>(x[4], x[5]), value_pair<K>(x[6], x[7]));                \
    st.o[4 * w + K] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, st.o[4 * w + K], 0, 0, 0); \
    if constexpr (kSplitP)                                                                   \
      st.o[4 * w + K] =                                                                      \
          __builtin_amdgcn_mfma_f32_16x16x32_f16(al, b, st.o[4 * w + K], 0, 0, 0);           \
  }
      KVQ_PV_TILE(0)
      KVQ_PV_TILE(1)
      KVQ_PV_TILE(2)
      KVQ_PV_TILE(3)
#undef KVQ_PV_TILE
    }
  }
}

// ---- E4M3 plan on the device --------------------------------------------------
// The requests' lengths travel as a kernel argument (no copy to the device): a
// call is launched for up to kMaxLens requests at a time.  Request b is cut into
// ceil(len / split) items, laid end to end.
constexpr int kMaxLens = 768;
struct SeqLens {
  int32_t n, split;
  int32_t len[kMaxLens];
};

// The lens argument (the kernel's first) read in place: passed on by value the
// compiler would copy it to scratch for the indexed reads.
typedef const __attribute__((address_space(4))) int32_t cint32;
__device__ __forceinline__ cint32* lens_arg() {
  return (cint32*)__builtin_amdgcn_kernarg_segment_ptr();
}

// Inclusive sum over the wave's lanes 0..lane.
__device__ __forceinline__ int wave_prefix(int x, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int y = __shfl_up(x, d, 64);
    x += lane >= d ? y : 0;
  }
  return x;
}

// Request, its length and the positions of item wi; false past the last one
// (wave-uniform).
__device__ __forceinline__ bool find_item(int wi, int lane, int& b, int& l, int& pb, int& pe) {
  cint32* a = lens_arg();
  const int n = a[0], split = a[1];
  int base = 0;
  for (int c = 0; c < n; c += 64) {
    const int len = c + lane < n ? a[2 + c + lane] : 0;
    const int items = (len + split - 1) / split;
    const int upto = base + wave_prefix(items, lane);
    const uint64_t past = __builtin_amdgcn_ballot_w64(upto > wi);
    if (past) {
      const int at = __builtin_ctzll(past);
      l = __builtin_amdgcn_readlane(len, at);
      const int first = __builtin_amdgcn_readlane(upto - items, at);
      b = c + at;
      pb = (wi - first) * split;
      pe = split < l - pb ? pb + split : l;  // no sum past l
      return true;
    }
    base = __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

// (first item, items) of every request, for the combine: one wave.
__device__ __forceinline__ void write_meta(int lane, int32_t* __restrict__ meta) {
  cint32* a = lens_arg();
  const int n = a[0], split = a[1];
  int base = 0;
  for (int c = 0; c < n; c += 64) {
    const int len = c + lane < n ? a[2 + c + lane] : 0;
    const int items = (len + split - 1) / split;
    const int upto = base + wave_prefix(items, lane);
    if (c + lane < n) {
      meta[2 * (c + lane)] = upto - items;
      meta[2 * (c + lane) + 1] = items;
    }
    base = __builtin_amdgcn_readlane(upto, 63);
  }
}

// A workgroup holds hpw waves: kv heads q*hpw .. q*hpw + hpw - 1 of one work
// item, one wave per head, each with its own two tile buffers.  With hpw = kvh
// (the launcher's choice whenever the LDS allows) a barrier after every tile
// keeps the item's heads in step, so that the rows of one token, which the
// heads' K and V lines interleave in HBM, are requested together: the DRAM
// pages open once for all heads instead of once per head (config-2 decode
// 111.5 -> 101 us, one 8-wave workgroup per CU).
//
// E4M3 with several query rows per request (RowCols): the columns of the score
// MFMA are the rows' heads, each with its own last position, so that 16 / rep
// rows share one pass over the codes.  32 requests of 0.5K-8K positions, 32 heads
// on 8 kv heads: 75 us for 4 rows, 139 for 8 (two passes), 267 for 16 (four);
// gathered to dense rows first they take 286, 294 and 302.
struct RowCols {
  int rows;   // query rows of a request
  int first;  // first of them in this pass
  int take;   // rows of this pass, take * rep <= 16
  int limit;  // positions the first row of the request sees; one more per row if step
  int step;
};
template <typename TQ, int D, bool FOLD, bool FP8>
__device__ __forceinline__ void decode_item(
    const TQ* __restrict__ query, RowCols rc, int hq, int kvh, int hpw, int h, float qscale,
    const int8_t* __restrict__ kc, const int8_t* __restrict__ vc, const float* __restrict__ ks,
    const float* __restrict__ vs, int bs, int64_t nb, const TQ* __restrict__ k_aq,
    const TQ* __restrict__ v_aq, const void* __restrict__ table_row, int bt64, int wi, int b,
    int pb, int pe, char* lds_i8, int lane, float* __restrict__ ws_o,
    float* __restrict__ ws_ml) {
  const int rep = hq / kvh;
  const int n = lane & 15;
  const int g = lane >> 4;
  u4v qh[D / 32], ql[D / 32];
  float sc = qscale;
  // column c's row among the request's rows * hq (E4M3), and the end of its positions
  const int cols = FP8 ? rep * rc.take : rep;
  auto col_head = [&](int c) {
    const int j = FP8 ? c / rep : 0;
    return (FP8 ? rc.first + j : 0) * hq + h * rep + (c - j * rep);
  };
  const int heads = FP8 ? rc.rows * hq : hq;
  int pen = pe;
  if constexpr (FP8) {
    const bool live = n < cols;
    pen = min(pe, rc.limit + rc.step * (rc.first + (live ? n / rep : 0)));
    const TQ* qrow = query + (static_cast<int64_t>(b) * heads + col_head(live ? n : 0)) * D;
#pragma unroll
    for (int s = 0; s < D / 32; ++s) {
      const u4v x = *reinterpret_cast<const u4v*>(qrow + (D / 4) * g + 8 * s);
      qh[s] = live ? x : u4v{0, 0, 0, 0};
    }
  } else {
    // ---- Q' = q * k_aq for head n, dims D/4 g + 8s + i, scaled by 2^e ----
    float qf[D / 4];
    float amax = 0.0f;
    {
      const int hn = FOLD ? (n & 7) : n;  // folded: columns n and n + 8 carry head n % 8
      const bool live = hn < rep;
      const TQ* qrow = query + (static_cast<int64_t>(b) * hq + h * rep + (live ? hn : 0)) * D;
      const TQ* arow = k_aq + static_cast<int64_t>(h) * D;
#pragma unroll
      for (int i = 0; i < D / 4; ++i) {
        const int dim = (D / 4) * g + i;
        const float x = to_f32(qrow[dim]) * to_f32(arow[dim]);
        qf[i] = live ? x : 0.0f;
        amax = fmaxf(amax, fabsf(qf[i]));
      }
    }
    amax = max_rows4(amax);
    int ex = 0;
    if (amax > 0.0f) (void)frexpf(amax, &ex);
    const int e = amax > 0.0f ? 15 - ex : 0;  // max |Q' * 2^e| in [2^14, 2^15)
#pragma unroll
    for (int s = 0; s < D / 32; ++s) {
      uint32_t hw[4], lw[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        _Float16 hh[2], ll[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const float x = ldexpf(qf[8 * s + 2 * u + k], e);
          hh[k] = static_cast<_Float16>(x);
          ll[k] = static_cast<_Float16>(x - static_cast<float>(hh[k]));
        }
        hw[u] = h2_bits(hh[0], hh[1]);
        lw[u] = h2_bits(ll[0], ll[1]);
      }
      if (FOLD) {
        const bool lo_col = n >= 8;
        qh[s] = u4v{lo_col ? lw[0] : hw[0], lo_col ? lw[1] : hw[1], lo_col ? lw[2] : hw[2],
                    lo_col ? lw[3] : hw[3]};
      } else {
        qh[s] = u4v{hw[0], hw[1], hw[2], hw[3]};
        ql[s] = u4v{lw[0], lw[1], lw[2], lw[3]};
      }
    }
    sc = ldexpf(qscale, -e);
  }

  WaveCtx c;
  c.kc = kc;
  c.vc = vc;
  c.ks = ks;
  c.vs = vs;
  c.bt = table_row;
  c.bt64 = bt64;
  c.nb = nb;
  c.bs = bs;
  c.kvh = kvh;
  c.h = h;
  c.g = g;
  c.n = n;
  c.last_group = (pe - 1) & ~15;

  SoftmaxState<D> st;
  st.m = -INFINITY;
  st.l = 0.0f;
#pragma unroll
  for (int tt = 0; tt < D / 16; ++tt) st.o[tt] = f4{0.f, 0.f, 0.f, 0.f};

  // two LDS buffers: tile i + 1's DMA is in flight while tile i computes.
  // Both are __restrict__ within a step, so the compiler's wait-count pass
  // knows the reads of `cur` cannot alias the DMA into `nxt`; the wait for
  // tile i itself is explicit.
  constexpr int kBuf = tile_bytes<D, FP8>();
  const int p0 = pb & ~15;
  auto step = [&](const char* __restrict__ cur, char* __restrict__ nxt, int p) {
    if (p + kTile < pe) {
      issue_tile_dma<D, FP8>(nxt, c, p + kTile, lane);
      wait_vmcnt<tile_dmas<D, FP8>()>();  // the DMAs of tile i + 1 may stay in flight
    } else {
      wait_vmcnt<0>();
    }
    TileRegs<D, FP8> t;
    read_tile_lds<D, FP8>(t, cur, g, n);
    compute_tile<TQ, D, FOLD, FP8>(t, p, pb, pe, pen, qh, ql, sc, g, st);
  };
  if (p0 < pe) issue_tile_dma<D, FP8>(lds_i8, c, p0, lane);  // an empty range leaves m = -inf, l = 0
  int cur = 0;
  for (int p = p0; p < pe; p += kTile) {
    step(lds_i8 + cur * kBuf, lds_i8 + (cur ^ 1) * kBuf, p);
    // every LDS read of this buffer is consumed before the next DMA into it
    asm volatile("" ::: "memory");
    cur ^= 1;
    if (hpw > 1) __syncthreads();  // uniform: the workgroup's heads share the item
  }

  // ---- epilogue ----
  constexpr int DPL = D / 16;  // dims per lane
  float l = st.l;
  l = sum_rows4(l);
  float va[DPL];
#pragma unroll
  for (int tt = 0; tt < DPL; ++tt)
    va[tt] = FP8 ? 1.0f
                 : to_f32(v_aq[static_cast<int64_t>(h) * D + DPL * n + tt]) * (1.0f / kLift<D>);
  const int64_t head0 = static_cast<int64_t>(wi) * heads;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int hh = 4 * g + r;
    if (hh < cols) {
      float* dst = ws_o + (head0 + col_head(hh)) * D + DPL * n;
#pragma unroll
      for (int w = 0; w < D / 64; ++w) {
        float4 x;
        x.x = st.o[4 * w][r] * va[4 * w];
        x.y = st.o[4 * w + 1][r] * va[4 * w + 1];
        x.z = st.o[4 * w + 2][r] * va[4 * w + 2];
        x.w = st.o[4 * w + 3][r] * va[4 * w + 3];
        *reinterpret_cast<float4*>(dst + 4 * w) = x;
      }
    }
  }
  if (g == 0 && n < cols) {
    const int64_t hh = head0 + col_head(n);
    // E4M3: a NaN score (a NaN query or code) leaves m without it; m = inf then
    // makes the combine's weights and its result NaN, as the gathered rows give
    ws_ml[2 * hh] = FP8 && l != l ? INFINITY : st.m;
    ws_ml[2 * hh + 1] = l;
  }
}

template <typename TQ, int D, bool FOLD>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
int8_decode_mfma_kernel(const TQ* __restrict__ query, int hq, int kvh, int hpw, float qscale,
                        const int8_t* __restrict__ kc, const int8_t* __restrict__ vc, int bs,
                        int64_t nb, const TQ* __restrict__ k_aq, const TQ* __restrict__ v_aq,
                        const int32_t* __restrict__ block_table, int64_t maxb,
                        const int32_t* __restrict__ work, float* __restrict__ ws_o,
                        float* __restrict__ ws_ml) {
  extern __shared__ __align__(16) char lds_wg[];
  const int groups = kvh / hpw;
  const int wi = blockIdx.x / groups;
  // wave-uniform; saying so keeps the DMA destinations in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = (blockIdx.x - wi * groups) * hpw + wave;
  const int lane = threadIdx.x & 63;
  const int32_t* wk = work + 4 * static_cast<int64_t>(wi);
  const int rep = hq / kvh;
  if (wk[3] != 0) {
    // an empty request's item: m = -inf, l = 0 (the combine gives it weight 0
    // and writes zeros when a request has nothing else)
    if (lane < rep) {
      const int64_t hh = static_cast<int64_t>(wi) * hq + static_cast<int64_t>(h) * rep + lane;
      ws_ml[2 * hh] = -INFINITY;
      ws_ml[2 * hh + 1] = 0.0f;
    }
    return;
  }
  const int b = wk[0];
  decode_item<TQ, D, FOLD, false>(query, RowCols{}, hq, kvh, hpw, h, qscale, kc, vc, nullptr, nullptr, bs, nb,
                                  k_aq, v_aq, block_table + static_cast<int64_t>(b) * maxb, 0, wi,
                                  b, wk[1], wk[2], lds_wg + wave * 2 * tile_bytes<D, false>(), lane,
                                  ws_o, ws_ml);
}

// E4M3: the work list follows from the lengths (find_item); the first workgroup
// leaves the combine's (first item, items) per request in meta.
template <typename TQ, int D>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
fp8_decode_mfma_kernel(SeqLens lens, const TQ* __restrict__ query, int rows, int take, int causal,
                       int hq, int kvh, int hpw,
                       float qscale, const uint8_t* __restrict__ kc, const float* __restrict__ ks,
                       const uint8_t* __restrict__ vc, const float* __restrict__ vs, int bs,
                       int64_t nb, const void* __restrict__ block_table, int bt64, int64_t maxb,
                       float* __restrict__ ws_o, float* __restrict__ ws_ml,
                       int32_t* __restrict__ meta) {
  extern __shared__ __align__(16) char lds_wg[];
  const int groups = kvh / hpw;
  const int wi = blockIdx.x / groups;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = (blockIdx.x - wi * groups) * hpw + wave;
  const int lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && blockIdx.y == 0 && wave == 0) write_meta(lane, meta);
  int b, len, pb, pe;
  if (!find_item(wi, lane, b, len, pb, pe)) return;  // workgroup-uniform
  // blockIdx.y: the pass, `take` of the request's rows
  const int first = static_cast<int>(blockIdx.y) * take;
  const RowCols rc{rows, first, min(take, rows - first), causal ? len - rows + 1 : len,
                   causal ? 1 : 0};
  const char* row = static_cast<const char*>(block_table) + b * maxb * (bt64 ? 8 : 4);
  decode_item<TQ, D, false, true>(query, rc, hq, kvh, hpw, h, qscale,
                                  reinterpret_cast<const int8_t*>(kc),
                                  reinterpret_cast<const int8_t*>(vc), ks, vs, bs, nb, nullptr,
                                  nullptr, row, bt64, wi, b, pb, pe,
                                  lds_wg + wave * 2 * tile_bytes<D, true>(), lane, ws_o, ws_ml);
}

}  // namespace

namespace kvq {

int launch_int8_decode_mfma(const void* query, int dtype, int hq, int kvh, int d, float qscale,
                            const int8_t* kc, const int8_t* vc, int bs, int64_t nb,
                            const void* k_aq, const void* v_aq, const int32_t* block_table,
                            int64_t maxb, const int32_t* work, int64_t num_work, float* ws_o,
                            float* ws_ml, hipStream_t s, bool* launched) {
  *launched = false;
  if ((d != 128 && d != 256) || hq / kvh > 16 || bs % 16) return KVQ_OK;
  // rows off the DMA's 16-byte lanes run the generic kernel
  if (!aligned16(kc, vc)) return KVQ_OK;
  if (num_work * kvh > 0x7fffffff) return KVQ_ERR_INVALID;
  // all kv heads of an item in one workgroup when they fit (at most 8 waves
  // and their tile buffers in the workgroup's LDS), else one wave per head
  int64_t lds_max = 0;
  const int lrc = device_lds_max(&lds_max);
  if (lrc != KVQ_OK) return lrc;
  const int wave_lds = 2 * (d == 128 ? tile_bytes<128, false>() : tile_bytes<256, false>());
  const int hpw = kvh <= 8 && kvh * wave_lds <= lds_max ? kvh : 1;
  const dim3 grid(static_cast<unsigned>(num_work * (kvh / hpw)));
  // GQA groups of at most 8 heads fold the hi/lo score parts into one MFMA
  const bool fold = hq / kvh <= 8;
#define KVQ_LAUNCH_I8(TQ, D, F)                                                               \
  hipLaunchKernelGGL((int8_decode_mfma_kernel<TQ, D, F>), grid, dim3(64 * hpw), hpw * wave_lds, \
                     s, static_cast<const TQ*>(query), hq, kvh, hpw, qscale, kc, vc, bs, nb,  \
                     static_cast<const TQ*>(k_aq), static_cast<const TQ*>(v_aq), block_table, \
                     maxb, work, ws_o, ws_ml)
#define KVQ_LAUNCH_I8_F(TQ, D) \
  if (fold) KVQ_LAUNCH_I8(TQ, D, true); else KVQ_LAUNCH_I8(TQ, D, false);
  KVQ_DISPATCH_FLOAT(dtype, TQ,
    if (d == 128) { KVQ_LAUNCH_I8_F(TQ, 128) } else { KVQ_LAUNCH_I8_F(TQ, 256) });
#undef KVQ_LAUNCH_I8_F
#undef KVQ_LAUNCH_I8
  KVQ_LAUNCH_CHECK();
  *launched = true;
  return KVQ_OK;
}

}  // namespace kvq

// ---- E4M3 decode ---------------------------------------------------------------
namespace {

// Positions per item: one workgroup of an item's heads per slot of the chip (two
// waves per SIMD, or as many as the LDS holds), a multiple of 128, grown until
// the requests, each cut on its own, fit: a partial second round of workgroups
// costs more than longer items.
int64_t fp8_split(const int64_t* lens, int64_t n, int kvh, int d, int cus) {
  const int64_t waves = d == 128 ? 8 : 4;
  const int64_t target = std::max<int64_t>(1, cus * waves / std::max(1, kvh));
  int64_t total = 0;
  for (int64_t b = 0; b < n; ++b) total += lens[b];
  int64_t split = std::max<int64_t>(128, ((total + target - 1) / target + 127) / 128 * 128);
  auto items = [&](int64_t s) {
    int64_t c = 0;
    for (int64_t b = 0; b < n; ++b) c += (lens[b] + s - 1) / s;
    return c;
  };
  while (split < 16384 && items(split) > std::max<int64_t>(target, n)) split += 128;
  return split;
}

constexpr int64_t kMaxLen = 0x7fff0000;  // positions of a request
constexpr int64_t kMaxRowHeads = 65536;  // rows * query heads of a request (the combine's grid)

struct Fp8Plan {
  int64_t first, n, split, items;  // requests [first, first + n) of one launch
};

// The launches of a batch: up to kMaxLens requests each.
template <typename F>
int fp8_launches(const int64_t* lens, int64_t batch, int kvh, int d, F f) {
  int cus = 0;
  const int rc = kvq::device_cu_count(&cus);
  if (rc != KVQ_OK) return rc;
  if (cus <= 0) cus = 256;
  for (int64_t b = 0; b < batch; b += kMaxLens) {
    Fp8Plan p{b, std::min<int64_t>(kMaxLens, batch - b), 0, 0};
    p.split = fp8_split(lens + b, p.n, kvh, d, cus);
    for (int64_t i = 0; i < p.n; ++i) p.items += (lens[b + i] + p.split - 1) / p.split;
    const int frc = f(p);
    if (frc != KVQ_OK) return frc;
  }
  return KVQ_OK;
}

bool fp8_decode_geometry(int hq, int kvh, int d, int bs) {
  return kvh > 0 && hq > 0 && hq % kvh == 0 && hq / kvh <= 16 && (d == 128 || d == 256) &&
         bs > 0 && bs % 16 == 0;
}

// Bytes of one launch's partials, then its (first item, items) table.
int64_t fp8_ws_bytes(int64_t items, int64_t n, int hq, int d) {
  return kvq::decode_workspace_bytes(items, hq, d) + 8 * n;
}

}  // namespace

extern "C" int64_t kvq_fp8_pth_decode_workspace_bytes(const int64_t* seq_lens, int64_t batch,
                                                      int64_t rows, int num_heads,
                                                      int num_kv_heads, int head_size,
                                                      int block_size) {
  if (rows <= 0 || rows * std::max(1, num_heads) > kMaxRowHeads) return KVQ_ERR_INVALID;
  if (batch < 0 || (batch > 0 && !seq_lens)) return KVQ_ERR_INVALID;
  if (!fp8_decode_geometry(num_heads, num_kv_heads, head_size, block_size))
    return KVQ_ERR_GEOMETRY;
  for (int64_t b = 0; b < batch; ++b)
    if (seq_lens[b] < 0 || seq_lens[b] > kMaxLen) return KVQ_ERR_INVALID;
  int64_t most = 0;  // launches run one after another on one stream and share it
  const int rc = fp8_launches(seq_lens, batch, num_kv_heads, head_size, [&](const Fp8Plan& p) {
    most = std::max(most, fp8_ws_bytes(p.items, p.n, rows * num_heads, head_size));
    return KVQ_OK;
  });
  return rc != KVQ_OK ? KVQ_ERR_INVALID : most;
}

extern "C" int kvq_fp8_pth_decode_attn(const void* query, int dtype, int64_t batch, int64_t rows,
                                       int causal, int num_heads, int num_kv_heads,
                                       int head_size, float scale,
                                       const uint8_t* k_data, const float* k_scale,
                                       const uint8_t* v_data, const float* v_scale,
                                       int64_t num_blocks, int block_size,
                                       const void* block_table, int block_index_type,
                                       int64_t max_blocks, const int64_t* seq_lens,
                                       void* workspace, int64_t workspace_bytes, void* out,
                                       void* stream) {
  if (batch == 0) return KVQ_OK;
  if (!query || !k_data || !k_scale || !v_data || !v_scale || !block_table || !seq_lens || !out ||
      !workspace || batch < 0 || num_blocks <= 0 || max_blocks <= 0)
    return KVQ_ERR_INVALID;
  if (block_index_type != KVQ_INDEX_I32 && block_index_type != KVQ_INDEX_I64)
    return KVQ_ERR_INVALID;
  if (!(scale > 0.0f)) return KVQ_ERR_INVALID;
  if (rows <= 0 || rows * std::max(1, num_heads) > kMaxRowHeads) return KVQ_ERR_INVALID;
  if ((dtype != KVQ_DTYPE_BF16 && dtype != KVQ_DTYPE_F16) ||
      !fp8_decode_geometry(num_heads, num_kv_heads, head_size, block_size) ||
      !kvq::aligned16(k_data, v_data))  // 16-byte DMA lanes
    return KVQ_ERR_GEOMETRY;
  for (int64_t b = 0; b < batch; ++b)
    if (seq_lens[b] < 0 || seq_lens[b] > kMaxLen || seq_lens[b] > max_blocks * block_size)
      return KVQ_ERR_INVALID;
  int64_t lds_max = 0;
  const int lrc = kvq::device_lds_max(&lds_max);
  if (lrc != KVQ_OK) return lrc;
  const int d = head_size, kvh = num_kv_heads;
  const int wave_lds = 2 * (d == 128 ? tile_bytes<128, true>() : tile_bytes<256, true>());
  if (wave_lds > lds_max) return KVQ_ERR_GEOMETRY;
  const int hpw = kvh <= 8 && kvh * wave_lds <= lds_max ? kvh : 1;
  const float qscale = scale * 1.4426950408889634f;
  const int bt64 = block_index_type == KVQ_INDEX_I64;
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* ws_o = static_cast<float*>(workspace);
  const int heads = static_cast<int>(rows) * num_heads;  // of a request
  const int64_t row = static_cast<int64_t>(heads) * d * 2;  // bytes of its 16-bit query rows
  const int take = std::min<int>(static_cast<int>(rows), 16 / (num_heads / kvh));
  const unsigned passes = static_cast<unsigned>((rows + take - 1) / take);
  // the launches' items follow from the lengths and the device: every one has to
  // fit before the first writes
  const int wrc = fp8_launches(seq_lens, batch, kvh, d, [&](const Fp8Plan& p) -> int {
    return fp8_ws_bytes(p.items, p.n, heads, d) <= workspace_bytes ? KVQ_OK : KVQ_ERR_INVALID;
  });
  if (wrc != KVQ_OK) return wrc;
  return fp8_launches(seq_lens, batch, kvh, d, [&](const Fp8Plan& p) -> int {
    float* ws_ml = ws_o + p.items * heads * d;
    int32_t* meta = reinterpret_cast<int32_t*>(ws_ml + 2 * p.items * heads);
    // a launch with nothing to read still writes the table (and the zeros)
    const int64_t blocks = std::max<int64_t>(1, p.items) * (kvh / hpw);
    if (blocks > 0x7fffffff) return KVQ_ERR_INVALID;
    SeqLens lens;
    lens.n = static_cast<int32_t>(p.n);
    lens.split = static_cast<int32_t>(p.split);
    for (int64_t i = 0; i < p.n; ++i) lens.len[i] = static_cast<int32_t>(seq_lens[p.first + i]);
    const char* q = static_cast<const char*>(query) + p.first * row;
    const char* bt = static_cast<const char*>(block_table) + p.first * max_blocks * (bt64 ? 8 : 4);
#define KVQ_LAUNCH_FP8(TQ, D)                                                                  \
  hipLaunchKernelGGL((fp8_decode_mfma_kernel<TQ, D>),                                          \
                     dim3(static_cast<unsigned>(blocks), passes), dim3(64 * hpw),              \
                     hpw * wave_lds, s, lens, reinterpret_cast<const TQ*>(q),                  \
                     static_cast<int>(rows), take, causal, num_heads, kvh, hpw, qscale, k_data, k_scale, v_data, v_scale, block_size, \
                     num_blocks, bt, bt64, max_blocks, ws_o, ws_ml, meta)
    if (dtype == KVQ_DTYPE_BF16) {
      if (d == 128) KVQ_LAUNCH_FP8(kvq::bf16, 128); else KVQ_LAUNCH_FP8(kvq::bf16, 256);
    } else {
      if (d == 128) KVQ_LAUNCH_FP8(kvq::f16, 128); else KVQ_LAUNCH_FP8(kvq::f16, 256);
    }
#undef KVQ_LAUNCH_FP8
    KVQ_LAUNCH_CHECK();
    return kvq::launch_decode_combine(dtype, p.n, heads, d, meta, 2, 0, ws_o, ws_ml,
                                      static_cast<char*>(out) + p.first * row, s);
  });
}
