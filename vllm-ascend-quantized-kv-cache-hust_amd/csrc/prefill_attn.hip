// SPDX-License-Identifier: Apache-2.0
// Causal (or full) attention over dense TND K/V on MFMA, for prefill and the
// prompt rows of a chunked batch.
//
// Replaces the NPU fused-attention calls with input_layout "TND":
// pkg/methods/kivi_int4/attention_backend.py:1248-1262 (PrefillNoCache),
// :1320-1334 (chunked prompt rows), the dense fallback :1341-1392, and the
// INT8 prefill paths pkg/methods/int8_dynamic/attention_backend.py:282-296,
// 350-364.  Query row i of a request with lq queries and lk keys sits at
// position lk - lq + i; with `causal`, key positions past it are masked
// (pkg/methods/kivi_int4/semantics.py:285-299).
//
// bf16/fp16 inputs with head_size 64, 128 or 256 run prefill_attn_fa_kernel
// (64-key blocks, DMA-staged K, transposed V, described at the kernel).  The
// kernel below covers the rest (fp32 inputs, head_size 32):
// one workgroup = 4 waves = 64 query rows of one query head; each wave owns
// 16 rows.  Keys/values stream through LDS in 32-token blocks.
//   S^T = K * Q^T   (v_mfma_f32_16x16x32_{bf16,f16}): A = K rows from LDS
//                   (16-byte reads), B = Q^T from registers (loaded once).
//   O^T += V^T * P^T: B = P^T straight from the S^T result registers (each
//                   lane already holds its query row's 8 probabilities);
//                   A = V^T read from the LDS block.
// Online softmax in the log2 domain, fp32 accumulation, output in the input
// dtype (fp32 inputs run through bf16 operands).
#include <algorithm>
#include <vector>

#include "kvq_common.h"

namespace {

using namespace kvq;

typedef float f4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef uint16_t u8v __attribute__((ext_vector_type(8)));

constexpr int kRowsPerWave = 16;
constexpr int kWaves = 4;
constexpr int kKvBlock = 32;

// Operand element type of the MFMA for an input type.
template <typename T> struct Op { using type = bf16; };
template <> struct Op<f16> { using type = f16; };

__device__ __forceinline__ uint16_t op_bits(float x, bf16) { return f32_to_bf16_bits(x); }
__device__ __forceinline__ uint16_t op_bits(float x, f16) {
  return __builtin_bit_cast(uint16_t, static_cast<_Float16>(x));
}
template <typename T>
__device__ __forceinline__ uint16_t raw_bits(T v) {
  return op_bits(to_f32(v), typename Op<T>::type{});
}
template <>
__device__ __forceinline__ uint16_t raw_bits<bf16>(bf16 v) { return v.bits; }
template <>
__device__ __forceinline__ uint16_t raw_bits<f16>(f16 v) { return __builtin_bit_cast(uint16_t, v); }

__device__ __forceinline__ float op_to_f32(uint16_t bits, bf16) {
  return __uint_as_float(static_cast<uint32_t>(bits) << 16);
}
__device__ __forceinline__ float op_to_f32(uint16_t bits, f16) {
  return static_cast<float>(__builtin_bit_cast(_Float16, bits));
}

// Two fp32 values as an operand pair (round to nearest even), and back.
__device__ __forceinline__ uint32_t pack_op2(float lo, float hi, bf16) { return bf16x2_bits(lo, hi); }
__device__ __forceinline__ uint32_t pack_op2(float lo, float hi, f16) {
  typedef float f2v __attribute__((ext_vector_type(2)));
  typedef _Float16 h2v __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2v{lo, hi}), h2v));
}
__device__ __forceinline__ float op_lo_f32(uint32_t w, bf16) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float op_hi_f32(uint32_t w, bf16) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float op_lo_f32(uint32_t w, f16) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w)));
}
__device__ __forceinline__ float op_hi_f32(uint32_t w, f16) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w >> 16)));
}

__device__ __forceinline__ f4 mfma16(u8v a, u8v b, f4 c, bf16) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b),
                                                 c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma16(u8v a, u8v b, f4 c, f16) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b),
                                                c, 0, 0, 0);
}

// Eight consecutive elements as operand bits (one 16-byte load for 16-bit types).
template <typename T>
__device__ __forceinline__ u8v load_op8(const T* p) {
  u8v r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = raw_bits(p[i]);
  return r;
}
template <>
__device__ __forceinline__ u8v load_op8<bf16>(const bf16* p) {
  return *reinterpret_cast<const u8v*>(p);
}
template <>
__device__ __forceinline__ u8v load_op8<f16>(const f16* p) {
  return *reinterpret_cast<const u8v*>(p);
}

template <typename T, int D>
__global__ void __launch_bounds__(256)
prefill_attn_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ cu_k, int hq,
                    int kvh, float qscale, int causal, T* __restrict__ out) {
  using O = typename Op<T>::type;
  constexpr int KS = D / 32;   // k-steps of the score MFMA
  constexpr int DB = D / 16;   // 16-dim output blocks
  __shared__ uint16_t s_k[kKvBlock * D];
  __shared__ uint16_t s_v[kKvBlock * D];

  const int b = blockIdx.z;
  const int head = blockIdx.y;
  const int kvhead = head / (hq / kvh);
  const int q_start = cu_q[b];
  const int lq = cu_q[b + 1] - q_start;
  const int k_start = cu_k[b];
  const int lk = cu_k[b + 1] - k_start;
  const int row0 = blockIdx.x * (kRowsPerWave * kWaves);
  if (row0 >= lq) return;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int n = lane & 15;
  const int kg = lane >> 4;
  const int wrow0 = row0 + wave * kRowsPerWave;
  const int my_row = wrow0 + n;           // query row of the lane's column
  const bool row_live = my_row < lq;
  const int my_pos = lk - lq + my_row;    // its kv position
  // kv range the workgroup needs
  const int last_row = min(row0 + kRowsPerWave * kWaves, lq) - 1;
  const int kv_end = causal ? min(lk, lk - lq + last_row + 1) : lk;

  // Q^T operand: lane (col n = query row, k-group kg) holds dims 32*s + 8*kg + i
  u8v qop[KS];
  {
    const T* qrow = q + (static_cast<int64_t>(q_start + (row_live ? my_row : 0)) * hq + head) * D;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i)  // unscaled: exact in the operand type
        qop[s][i] = row_live ? raw_bits(qrow[32 * s + 8 * kg + i]) : uint16_t(0);
  }

  float m_run = -INFINITY, l_run = 0.0f;
  f4 o[DB];
#pragma unroll
  for (int j = 0; j < DB; ++j) o[j] = f4{0.f, 0.f, 0.f, 0.f};

  for (int kb = 0; kb < kv_end; kb += kKvBlock) {
    __syncthreads();
    // stage K and V rows [kb, kb + 32) of this kv head (16-byte loads)
    constexpr int QPR = D / 8;  // 8-element pieces per row
    for (int e = tid; e < kKvBlock * QPR; e += 256) {
      const int t = e / QPR;
      const int c = (e - t * QPR) * 8;
      const int pos = kb + t;
      u8v kvv, vvv;
      if (pos < lk) {
        const int64_t src = (static_cast<int64_t>(k_start + pos) * kvh + kvhead) * D + c;
        kvv = load_op8(k + src);
        vvv = load_op8(v + src);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          kvv[i] = 0;
          vvv[i] = 0;
        }
      }
      *reinterpret_cast<u8v*>(s_k + t * D + c) = kvv;
      *reinterpret_cast<u8v*>(s_v + t * D + c) = vvv;
    }
    __syncthreads();
    // waves whose rows are all before this block under the causal mask skip it
    const int wave_last_pos = lk - lq + min(wrow0 + kRowsPerWave, lq) - 1;
    if (wrow0 >= lq || (causal && kb > wave_last_pos)) continue;

    // scores: two 16-token halves; lane holds query row n, tokens 4*kg + r (+16)
    f4 s0 = f4{0.f, 0.f, 0.f, 0.f}, s1 = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u8v a0 = *reinterpret_cast<const u8v*>(s_k + n * D + 32 * s + 8 * kg);
      const u8v a1 = *reinterpret_cast<const u8v*>(s_k + (16 + n) * D + 32 * s + 8 * kg);
      s0 = mfma16(a0, qop[s], s0, O{});
      s1 = mfma16(a1, qop[s], s1, O{});
    }
    float sc[8];
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int p0 = kb + 4 * kg + r;
      const int p1 = p0 + 16;
      const bool ok0 = p0 < lk && (!causal || p0 <= my_pos);
      const bool ok1 = p1 < lk && (!causal || p1 <= my_pos);
      sc[r] = ok0 ? s0[r] * qscale : -INFINITY;
      sc[4 + r] = ok1 ? s1[r] * qscale : -INFINITY;
      tmax = fmaxf(tmax, fmaxf(sc[r], sc[4 + r]));
    }
    tmax = max_rows4(tmax);
    const float m_new = fmaxf(m_run, tmax);
    const float alpha = m_run == -INFINITY ? (m_new == -INFINITY ? 1.0f : 0.0f)
                                           : exp2f(m_run - m_new);
    float psum = 0.0f;
    u8v pop;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = m_new == -INFINITY ? 0.0f : exp2f(sc[i] - m_new);
      pop[i] = op_bits(p, O{});
      // normalise by the probabilities the MFMA actually sees
      psum += op_to_f32(pop[i], O{});
    }
    psum = sum_rows4(psum);
    l_run = l_run * alpha + psum;
    m_run = m_new;
    // PV: A = V^T rows (dims), 8 tokens {4*kg + r, 16 + 4*kg + r}
#pragma unroll
    for (int j = 0; j < DB; ++j) {
      const int dim = 16 * j + n;
      u8v a;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        a[r] = s_v[(4 * kg + r) * D + dim];
        a[4 + r] = s_v[(16 + 4 * kg + r) * D + dim];
      }
      o[j] *= alpha;
      o[j] = mfma16(a, pop, o[j], O{});
    }
  }
  if (!row_live) return;
  // o[j][r] = O^T[dim 16*j + 4*kg + r][row n]
  const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
  T* orow = out + (static_cast<int64_t>(q_start + my_row) * hq + head) * D;
#pragma unroll
  for (int j = 0; j < DB; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) orow[16 * j + 4 * kg + r] = from_f32<T>(o[j][r] * inv);
}

// ---- 64-key-block kernel for 16-bit inputs, D in {64, 128, 256} -------------
// One workgroup = 4 waves x 32 rows (two 16-row MFMA column groups) of one
// request and kv head; key/value blocks of 64 tokens, double-buffered in LDS
// with one barrier per block.  Row R of a (request, kv head) is query R / rep
// of query head kvhead * rep + R % rep: the GQA group's heads share a tile, so
// the tile's queries sit rep times closer together (fewer keys masked along
// the diagonal), a short prompt fills its tile, and each key block is staged
// once for the group instead of once per head.
//   K  [64][D]    written by global_load_lds (16-byte lanes); the 16-byte
//                 column of each row is XOR-swizzled by the row so that the
//                 16 rows one score MFMA reads sit in different banks;
//   V  [64][D]    written by global_load_lds too, row-major; 16-byte column
//                 c of row r stored at c ^ (2*(r % 4) + 8*((r / 4) % 2)) (the
//                 second term at D >= 128), so that the rows the transposing
//                 reads of one LDS cycle cover sit in different banks.
// Keys run one block ahead of values: the step of block i computes block i's
// softmax and PV and block i+1's scores, whose MFMAs interleave with block
// i's exponentials (independent work, one basic block); block i+2's keys and
// block i+1's values are in flight (DMA) meanwhile.
//   S^T = K * Q^T: A = 16 keys x 32 dims (one 16-byte read per lane), B = the
//                  wave's Q^T (registers), each A feeding both column groups.
//   O^T += V^T * P^T: B = P^T straight from the S^T registers (the lane's
//                  keys 16*(2ks + i/4) + 4*kg + i%4 of its query column),
//                  A = the same 8 keys of one dim, gathered out of the
//                  row-major V by two transposing LDS reads
//                  (ds_read_b64_tr_b16: within each 16-lane group, lane l gets
//                  element l % 4 of the 8-byte runs that lanes l / 4 + 4k
//                  address, k = 0..3).
// The rescale needs no shuffles: S^T and O^T both put the lane's query in
// its column.
// The common step's softmax is the row maxima, one compare per column, and an
// fma and exp2 per score; the offset bookkeeping (new offset, rescale factor)
// sits in the branch that the lazy offset rarely takes.

constexpr int kFaBlock = 64;  // keys per block
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s* lds_v4s_ptr;

// LDS DMA of 16 bytes per lane from base + voff (base uniform, in SGPRs;
// voff the lane's 32-bit byte offset) to LDS bytes m0 + 16 * lane (m0
// uniform), so no 64-bit address is formed per lane.  The s_nop covers the
// M0-write hazard.  Inline asm, outside the compiler's wait counting: the
// kernel waits for every block's DMA explicitly (wait_vmcnt<0> before the
// barrier that publishes it).
__device__ __forceinline__ void dma16_so(const char* base, uint32_t voff, uint32_t m0) {
  m0 = __builtin_amdgcn_readfirstlane(m0);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(voff), "s"(base), "{m0}"(m0)
               : "memory");
}
__device__ __forceinline__ uint32_t lds_addr(const char* p) {
  return static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char*)(p)));
}

template <int D>
struct FaLds {
  static constexpr int K_BYTES = kFaBlock * D * 2;
  static constexpr int V_BYTES = kFaBlock * D * 2;
  static constexpr int BUF = K_BYTES + V_BYTES;
  static constexpr int BYTES = 2 * BUF;
};

// NG 16-row column groups per wave; the workgroup's 8 / NG waves cover 128 rows
// and share the LDS blocks, at two waves per SIMD (fa_ng below):
//   D <= 128: NG = 2 (4 waves of 32 rows, two workgroups a CU): each LDS operand
//     feeds two MFMAs.  NG = 1 measured 26% slower on 8 x 2048 queries over
//     10240 keys (twice the LDS reads per MFMA, and spills at the 128-VGPR limit
//     of 4 waves per SIMD).
//   D = 256: NG = 1 (8 waves of 16 rows; the blocks take 128 KB, one workgroup
//     a CU): 240 VGPRs, 254 us on 6 ragged prompts of 200 - 2048 rows with 3000
//     keys of history (8 heads on 1 kv head); the fallback kernel took 1612.
//     NG = 2 needs about 400 registers, one wave per SIMD and accumulator moves:
//     322 us, and 335 with its operand reads a step ahead.
template <int D>
constexpr int fa_ng() { return D == 256 ? 1 : 2; }

// A launch's tiles, as a kernel argument when they fit (small calls then copy
// nothing to the device): int32 cu_q [batch + 1], cu_k [batch + 1], and the
// units request | tile << 16 in dispatch order.
constexpr int kPlanArgWords = 500;
struct PlanArg {
  int32_t w[kPlanArgWords];
};
// Read-only tables: uniform reads through the constant address space are
// scalar loads.  The plan argument is the kernel's first and is read in place
// (indexed by value, the compiler would copy it to scratch).
typedef const __attribute__((address_space(4))) int32_t cint32;
__device__ __forceinline__ cint32* as_const(const int32_t* p) { return (cint32*)(p); }

// Where a call's keys are cut into `segs` segments per tile (few tiles, long
// keys): the partial results, o [unit][kv head][seg][row of the tile][D] and
// (m, l) per row, m in the log2 domain.
struct SegWs {
  float* o;
  float* ml;
  int segs;
};

template <typename T, int D, int NG>
__global__ void __launch_bounds__(64 * (8 / NG))
__attribute__((amdgpu_waves_per_eu(2, 2)))
prefill_attn_fa_kernel(PlanArg plan_arg, const int32_t* __restrict__ plan, int batch,
                       const T* __restrict__ q, const T* __restrict__ k,
                       const T* __restrict__ v, const int32_t* __restrict__ cu_q,
                       const int32_t* __restrict__ cu_k, int tiles, int hq, int kvh,
                       FastDiv rep_div, float qscale, int causal, T* __restrict__ out, SegWs seg) {
  using O = typename Op<T>::type;
  using L = FaLds<D>;
  constexpr int kFaWaves = 8 / NG;
  constexpr int kFaRows = 16 * NG;  // query rows per wave
  constexpr int KS = D / 32;      // score k-steps
  constexpr int DB = D / 16;      // output dim blocks
  constexpr int PPR = D / 8;      // 16-byte pieces per row
  constexpr int RPI = 64 / PPR;   // K rows per DMA instruction
  constexpr int KINST = kFaBlock / RPI / kFaWaves;  // DMA instructions per wave per block
  static_assert(KINST >= 1 && kFaBlock % (RPI * kFaWaves) == 0, "K / V DMA split");
  static_assert(PPR >= 8, "V swizzle 2 * (r % 4) stays inside the row");
  // V's 16-byte column c of row r sits at c ^ vswz(r): 2 (r % 4) spreads the
  // four rows one transposing read covers over the banks, and with 16 columns
  // a row (D = 128) 8 ((r / 4) % 2) also parts the rows 4 apart that the two
  // 16-lane groups of one LDS cycle read
  auto vswz = [](int r) { return 2 * (r % 4) + (PPR >= 16 ? 8 * ((r / 4) % 2) : 0); };
  extern __shared__ __align__(16) char lds[];
  const uint32_t lds0 = lds_addr(lds);  // LDS byte address of the buffers (DMA M0)

  // Workgroup ids go to the XCDs round-robin: with 8 kv heads each XCD runs one
  // kv head of every tile, in the order of the unit list (a request's tiles
  // one after another where its keys outgrow an L2, so that the XCD's L2 keeps
  // them between its tiles); with fewer kv heads a request's tiles spread over
  // all XCDs.
  const int rep = static_cast<int>(rep_div.d);
  const int unit = static_cast<int>(blockIdx.x) / kvh;
  const int kvhead = static_cast<int>(blockIdx.x) - unit * kvh;
  // without a unit list (cu_q): every request's `tiles` tiles, the last (most
  // keys under the causal mask) first
  int b, tile;
  cint32 *cq, *ck;
  if (cu_q) {
    b = unit / tiles;
    tile = tiles - 1 - unit % tiles;
    cq = as_const(cu_q);
    ck = as_const(cu_k);
  } else {
    cq = plan ? as_const(plan) : (cint32*)__builtin_amdgcn_kernarg_segment_ptr();
    ck = cq + batch + 1;
    const uint32_t u = static_cast<uint32_t>(ck[batch + 1 + unit]);
    b = static_cast<int>(u & 0xffffu);
    tile = static_cast<int>(u >> 16);
  }
  const int q_start = cq[b];
  const int lq = cq[b + 1] - q_start;
  const int k_start = ck[b];
  const int lk = ck[b + 1] - k_start;
  const int rows = lq * rep;  // rows of this (request, kv head)
  const int row0 = tile * (kFaRows * kFaWaves);
  if (row0 >= rows) return;  // uniform over the workgroup
  const int tid = threadIdx.x;
  // wave-uniform; saying so keeps the DMA destinations in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int n = lane & 15;
  const int kg = lane >> 4;
  const int wrow0 = row0 + wave * kFaRows;
  auto query_of = [&](int row) { return static_cast<int>(rep_div.div(static_cast<uint32_t>(row))); };
  const int last_row = min(row0 + kFaRows * kFaWaves, rows) - 1;
  const int kv_end = causal ? min(lk, lk - lq + query_of(last_row) + 1) : lk;
  int blk0 = 0, nblk = (kv_end + kFaBlock - 1) / kFaBlock;  // this workgroup's blocks [blk0, nblk)
  if (seg.segs > 1) {
    const int all = nblk > 0 ? nblk : 0, sg = static_cast<int>(blockIdx.y);
    blk0 = static_cast<int>(static_cast<int64_t>(all) * sg / seg.segs);
    nblk = static_cast<int>(static_cast<int64_t>(all) * (sg + 1) / seg.segs);
  }
  const int wave_last = min(wrow0 + kFaRows, rows) - 1;  // < wrow0 when the wave has no rows
  // kv positions of the wave's first and last query
  const int wave_first_pos = lk - lq + query_of(wrow0);
  const int wave_last_pos = lk - lq + query_of(wave_last);

  // element offset of row R in q and out
  auto row_offset = [&](int row) -> int64_t {
    const int i = query_of(row);
    return (static_cast<int64_t>(q_start + i) * hq + kvhead * rep + (row - i * rep)) * D;
  };
  // row of this workgroup's first row in the segments' partial results
  const int64_t seg_row0 =
      (static_cast<int64_t>(blockIdx.x) * seg.segs + blockIdx.y) * (kFaRows * kFaWaves);
  if (seg.segs > 1 && blk0 >= nblk) {  // uniform: a segment without keys
    for (int r = tid; r < kFaRows * kFaWaves; r += 64 * kFaWaves) {
      seg.ml[2 * (seg_row0 + r)] = -INFINITY;
      seg.ml[2 * (seg_row0 + r) + 1] = 0.0f;
    }
    return;
  }
  if (lk <= 0) {  // uniform: nothing to attend to
    for (int r = tid >> 4; r < kFaRows * kFaWaves; r += 4 * kFaWaves)
      if (row0 + r < rows)
        for (int c = tid & 15; c < D; c += 16) out[row_offset(row0 + r) + c] = from_f32<T>(0.0f);
    return;
  }

  // Q^T operands: group g2, k-step s: row wrow0 + 16*g2 + n, dims 32s + 8kg + i
  // (unscaled: exact in the operand type; loaded with the first blocks below)
  u8v qop[NG][KS];
  int my_pos[NG];
  bool live[NG];
#pragma unroll
  for (int g2 = 0; g2 < NG; ++g2) {
    const int row = wrow0 + 16 * g2 + n;
    live[g2] = row < rows;
    my_pos[g2] = lk - lq + query_of(row);
  }

  // ---- staging ----
  const T* kbase = k + (static_cast<int64_t>(k_start) * kvh + kvhead) * D;
  const T* vbase = v + (static_cast<int64_t>(k_start) * kvh + kvhead) * D;
  const int64_t row_stride = static_cast<int64_t>(kvh) * D;
  // DMA instruction i of a wave moves block rows c .. c + RPI - 1, c = RPI *
  // (wave * KINST + i): lane l the 16-byte column (l % PPR) ^ swz(row) of row
  // c + l / PPR.  Both swizzles split over the bits of the row, swz(c + l / PPR)
  // = swz(c) ^ swz(l / PPR), and a row's columns are the low bits of its
  // offset, so one offset per lane and side serves every instruction: the
  // instruction adds row c to the uniform base and xors 16 * swz(c).
  auto kswz = [](int r) { return r % PPR; };
  const uint32_t row_bytes = static_cast<uint32_t>(row_stride * 2);
  const int lane_row = lane / PPR;
  const uint32_t koff = lane_row * row_bytes + 16 * ((lane % PPR) ^ kswz(lane_row));
  const uint32_t voff = lane_row * row_bytes + 16 * ((lane % PPR) ^ vswz(lane_row));
  // DMA of block rows kb .. kb + 63 of `base` into `dst`; in the last block
  // rows past the end read the last row (masked later)
  auto issue_rows = [&](const T* base, uint32_t off, auto swz, char* dst, int kb) {
    const char* gb = reinterpret_cast<const char*>(base + static_cast<int64_t>(kb) * row_stride);
    if (kb + kFaBlock <= lk) {  // uniform: only the last block clamps
#pragma unroll
      for (int i = 0; i < KINST; ++i) {
        const int c = RPI * (wave * KINST + i);
        dma16_so(gb + static_cast<uint32_t>(c) * row_bytes, off ^ (16u * swz(c)),
                 lds0 + static_cast<uint32_t>(dst - lds) + 1024u * (wave * KINST + i));
      }
    } else {
#pragma unroll
      for (int i = 0; i < KINST; ++i) {
        // rows past the end step back to row lk - 1 - kb of the block (>= 0),
        // so the offset from the block's first row stays non-negative
        const int c = RPI * (wave * KINST + i);
        const int over = kb + c + lane_row - (lk - 1);
        const int r = c - (over > 0 ? over : 0);
        dma16_so(gb, (off ^ (16u * swz(c))) + static_cast<uint32_t>(r) * row_bytes,
                 lds0 + static_cast<uint32_t>(dst - lds) + 1024u * (wave * KINST + i));
      }
    }
  };
  // PV operand reads: lane s of a 16-lane group addresses V row keybase + s / 4,
  // dims 16j + 4 (s % 4) .. + 3 (swizzled 16-byte column), so that lane n of
  // the group receives V[keybase + k][16j + n], k = 0..3
  const int tr_row = lane % 16 / 4;
  const int tr_chunk = (lane % 4) / 2;  // + 2j
  const int tr_half = 8 * (lane % 2);   // byte offset inside the 16-byte column

  // Per query column: m_run, the raw score the exponent offset stands for
  // (-inf before the first finite score); m_off = -qscale * m_run (0 while
  // m_run is -inf), so p = 2^(qscale * s + m_off); m_thr = m_run + 8 / qscale,
  // the raw score past which the offset moves (lazy offset, below).
  // At D = 256 the offset follows every new maximum: the largest p is then 1
  // exactly, where the rounding of a p past 1 costs 3 - 8% more error in the
  // output (254 against 244 us on the prompts of fa_ng above).
  const float lazy_thr = D == 256 ? 0.0f : 8.0f / qscale;  // qscale > 0
  float m_run[NG], m_off[NG], m_thr[NG];
#pragma unroll
  for (int g2 = 0; g2 < NG; ++g2) {
    m_run[g2] = -INFINITY;
    m_off[g2] = 0.0f;
    m_thr[g2] = -INFINITY;
  }
  // l_acc[g2]: every row holds the running sum of the (rounded) P of query
  // column n, accumulated by an MFMA with an all-ones A, so it is the exact sum
  // of what the PV MFMAs saw and rescales together with o
  f4 l_acc[NG];
  f4 o[DB][NG];
#pragma unroll
  for (int g2 = 0; g2 < NG; ++g2) {
    l_acc[g2] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < DB; ++j) o[j][g2] = f4{0.f, 0.f, 0.f, 0.f};
  }
  const uint16_t one = op_bits(1.0f, O{});
  const u8v ones = u8v{one, one, one, one, one, one, one, one};

  // LDS: two key buffers and two value buffers.  Keys run one block ahead of
  // values: step i computes block i's softmax and PV and block i + 1's scores
  // (the score MFMAs interleaved with the softmax's exponentials, which do not
  // depend on them), while block i + 2's keys and block i + 1's values arrive.
  char* const kbuf0 = lds;
  char* const kbuf1 = lds + L::K_BYTES;
  char* const vbuf0 = lds + 2 * L::K_BYTES;
  char* const vbuf1 = lds + 2 * L::K_BYTES + L::V_BYTES;
  // waves whose rows all precede block i under the causal mask skip it (and
  // every later block)
  auto active = [&](int i) {
    return wrow0 <= wave_last && !(causal && i * kFaBlock > wave_last_pos);
  };
  // the K operands of 16-key group kb2 of the block at `sk`
  auto k_reads = [&](const uint16_t* sk, int kb2, u8v (&a)[KS]) {
    const int r = 16 * kb2 + n;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int piece = (4 * s + kg) ^ (r % PPR);
      a[s] = *reinterpret_cast<const u8v*>(sk + r * D + 8 * piece);
    }
  };
  // the V^T operands of k-step ks, half jh of the dim blocks
  auto v_reads = [&](const char* sv, int ks, int jh, u8v (&a)[DB / 2]) {
#pragma unroll
    for (int jj = 0; jj < DB / 2; ++jj) {
      const int j = jh * (DB / 2) + jj;
      v4s part[2];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        // keys 32 ks + 16 hh + 4 kg + k, k = 0..3
        const int r = 32 * ks + 16 * hh + 4 * kg + tr_row;
        const int pos = (2 * j + tr_chunk) ^ vswz(r);
        part[hh] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_v4s_ptr)(sv + r * (2 * D) + 16 * pos + tr_half));
      }
      a[jj] = u8v{static_cast<uint16_t>(part[0][0]), static_cast<uint16_t>(part[0][1]),
                  static_cast<uint16_t>(part[0][2]), static_cast<uint16_t>(part[0][3]),
                  static_cast<uint16_t>(part[1][0]), static_cast<uint16_t>(part[1][1]),
                  static_cast<uint16_t>(part[1][2]), static_cast<uint16_t>(part[1][3])};
    }
  };
  auto k_mfmas = [&](const u8v (&a)[KS], f4 (&acc)[NG]) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int g2 = 0; g2 < NG; ++g2) acc[g2] = mfma16(a[s], qop[g2][s], acc[g2], O{});
  };

  // prologue: keys of the first two blocks, values and scores of the first
  issue_rows(kbase, koff, kswz, kbuf0, blk0 * kFaBlock);
  if (blk0 + 1 < nblk) issue_rows(kbase, koff, kswz, kbuf1, (blk0 + 1) * kFaBlock);
  issue_rows(vbase, voff, vswz, vbuf0, blk0 * kFaBlock);
  // the query rows go out behind the DMAs, so that one wait covers both
#pragma unroll
  for (int g2 = 0; g2 < NG; ++g2) {
    const T* qrow = q + row_offset(live[g2] ? wrow0 + 16 * g2 + n : 0);
#pragma unroll
    for (int s = 0; s < KS; ++s) qop[g2][s] = load_op8(qrow + 32 * s + 8 * kg);
  }
#pragma unroll
  for (int g2 = 0; g2 < NG; ++g2)
#pragma unroll
    for (int s = 0; s < KS; ++s)
      if (!live[g2]) qop[g2][s] = u8v{0, 0, 0, 0, 0, 0, 0, 0};
  wait_vmcnt<0>();  // landed in LDS
  __syncthreads();
  f4 sacc[4][NG];
#pragma unroll
  for (int kb2 = 0; kb2 < 4; ++kb2)
#pragma unroll
    for (int g2 = 0; g2 < NG; ++g2) sacc[kb2][g2] = f4{0.f, 0.f, 0.f, 0.f};
  if (active(blk0)) {
#pragma unroll
    for (int kb2 = 0; kb2 < 4; ++kb2) {
      u8v a[KS];
      k_reads(reinterpret_cast<const uint16_t*>(kbuf0), kb2, a);
      k_mfmas(a, sacc[kb2]);
    }
  }
  __syncthreads();  // block 0's keys are read before block 2's overwrite them

  // One block step.  The four buffers are __restrict__ within the step, so
  // the compiler's wait-count pass knows that the LDS reads of `kn` (block
  // i + 1's keys) and `vc` (block i's values) cannot alias the DMA in flight
  // into `kd` and `vd` (otherwise it waits for that DMA before the first read).
  auto step = [&](const char* __restrict__ kn, const char* __restrict__ vc,
                  char* __restrict__ kd, char* __restrict__ vd, int i) {
    const int kb = i * kFaBlock;
    if (i + 2 < nblk) issue_rows(kbase, koff, kswz, kd, kb + 2 * kFaBlock);
    if (i + 1 < nblk) issue_rows(vbase, voff, vswz, vd, kb + kFaBlock);
    if (active(i)) {
      // ---- online softmax of block i per query column ----
      // the max runs over raw scores (qscale > 0), the exponent is one fma:
      // p = 2^(qscale * s + m_off)
      const bool full = kb + kFaBlock <= lk && (!causal || kb + kFaBlock - 1 <= wave_first_pos);
      if (!full) {  // uniform: one branch, then a compare per score
#pragma unroll
        for (int g2 = 0; g2 < NG; ++g2) {
          // key kb + 16 kb2 + 4 kg + r is live when 16 kb2 + r <= rel
          const int rel = (causal ? min(lk - 1, my_pos[g2]) : lk - 1) - kb - 4 * kg;
#pragma unroll
          for (int e = 0; e < 16; ++e)
            sacc[e / 4][g2][e % 4] = 16 * (e / 4) + e % 4 <= rel ? sacc[e / 4][g2][e % 4] : -INFINITY;
        }
      }
      float tmax[NG];
      // row maxima: two chains per column group, the groups side by side,
      // then the cross-row steps of both groups together
#pragma unroll
      for (int g2 = 0; g2 < NG; ++g2) {
        // med3(a, b, FLT_MAX) = max(a, b) for scores (never +inf or NaN),
        // without the canonicalizing moves a two-operand fmaxf gets
        constexpr float kBig = 0x1.fffffep127f;
        float ta = __builtin_amdgcn_fmed3f(sacc[0][g2][0], sacc[0][g2][1], kBig);
        float tb = __builtin_amdgcn_fmed3f(sacc[2][g2][0], sacc[2][g2][1], kBig);
#pragma unroll
        for (int e = 2; e < 8; ++e) {
          ta = fmaxf(ta, sacc[e / 4][g2][e % 4]);
          tb = fmaxf(tb, sacc[2 + e / 4][g2][e % 4]);
        }
        tmax[g2] = fmaxf(ta, tb);
      }
      if constexpr (NG == 2) {
        max_rows4_pair(tmax[0], tmax[1]);
      } else {
#pragma unroll
        for (int g2 = 0; g2 < NG; ++g2) tmax[g2] = max_rows4(tmax[g2]);
      }
      // lazy offset: a column's offset moves only when its max grows past
      // m_run by more than 8 (log2 units), so p <= 2^8 and most blocks skip
      // the branch (o, l and the offsets stay); the normalisation by l makes
      // the result the same softmax whatever offset the column settled on
      bool grow[NG], rescale = false;
#pragma unroll
      for (int g2 = 0; g2 < NG; ++g2) {
        grow[g2] = tmax[g2] > m_thr[g2];
        rescale = rescale || grow[g2];
      }
      if (__any(rescale)) {
#pragma unroll
        for (int g2 = 0; g2 < NG; ++g2) {
          const float m_new = grow[g2] ? tmax[g2] : m_run[g2];
          // the first finite max finds o and l still zero
          const float alpha =
              !grow[g2] ? 1.0f
                        : (m_run[g2] == -INFINITY
                               ? 0.0f
                               : __builtin_amdgcn_exp2f(qscale * (m_run[g2] - m_new)));
          l_acc[g2] *= alpha;
#pragma unroll
          for (int j = 0; j < DB; ++j) o[j][g2] *= alpha;
          m_run[g2] = m_new;
          m_off[g2] = m_new == -INFINITY ? 0.0f : -qscale * m_new;
          m_thr[g2] = m_new + lazy_thr;
        }
      }
      // raised wave priority from here to the end of the PV MFMAs: the SIMD's
      // arbiter then issues this wave's MFMAs first and fills their cycles
      // with the other wave's row maxima, which pulls the two waves into
      // alternating phases (+1-3% on config-4 attention)
      __builtin_amdgcn_s_setprio(1);
      // ---- P of block i, with block i + 1's score MFMAs in between ----------
      // 16-key group c: its exponentials (pop[g2][c / 2], half c % 2) beside
      // the score MFMAs of the next block's group c
      // (the last step computes scores of stale keys it never uses: one
      // branch-free block keeps the MFMAs and the exponentials interleavable;
      // the last step as code of its own spills 55 registers)
      f4 snext[4][NG];
#pragma unroll
      for (int kb2 = 0; kb2 < 4; ++kb2)
#pragma unroll
        for (int g2 = 0; g2 < NG; ++g2) snext[kb2][g2] = f4{0.f, 0.f, 0.f, 0.f};
      uint32_t pw[NG][2][4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        u8v a[KS];
        k_reads(reinterpret_cast<const uint16_t*>(kn), c, a);
#pragma unroll
        for (int g2 = 0; g2 < NG; ++g2)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(qscale, sacc[c][g2][2 * h], m_off[g2]));
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(qscale, sacc[c][g2][2 * h + 1], m_off[g2]));
            pw[g2][c / 2][2 * (c % 2) + h] = pack_op2(p0, p1, O{});
          }
        k_mfmas(a, snext[c]);
      }
      u8v pop[NG][2];  // [g2][ks]
#pragma unroll
      for (int g2 = 0; g2 < NG; ++g2)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
          pop[g2][ks] = __builtin_bit_cast(u8v, make_uint4(pw[g2][ks][0], pw[g2][ks][1],
                                                           pw[g2][ks][2], pw[g2][ks][3]));
      // ---- O^T += V^T * P^T ----
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int jh = 0; jh < 2; ++jh) {
          u8v a[DB / 2];  // half the dim blocks' V^T operands of this k-step, then the MFMAs
          v_reads(vc, ks, jh, a);
          __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of the MFMAs
#pragma unroll
          for (int jj = 0; jj < DB / 2; ++jj)
#pragma unroll
            for (int g2 = 0; g2 < NG; ++g2)
              o[jh * (DB / 2) + jj][g2] =
                  mfma16(a[jj], pop[g2][ks], o[jh * (DB / 2) + jj][g2], O{});
          if (jh == 1) {
#pragma unroll
            for (int g2 = 0; g2 < NG; ++g2) l_acc[g2] = mfma16(ones, pop[g2][ks], l_acc[g2], O{});
          }
        }
      __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int kb2 = 0; kb2 < 4; ++kb2)
#pragma unroll
        for (int g2 = 0; g2 < NG; ++g2) sacc[kb2][g2] = snext[kb2][g2];
    }
    if (i + 1 < nblk) wait_vmcnt<0>();  // block i + 2's keys and i + 1's values landed
  };
  // two steps per iteration, so that each step's buffers are compile-time
  // LDS offsets (folded into the reads' immediates instead of per-read adds)
  int i = blk0;
  for (; i + 1 < nblk; i += 2) {
    step(kbuf1, vbuf0, kbuf0, vbuf1, i);
    __syncthreads();
    step(kbuf0, vbuf1, kbuf1, vbuf0, i + 1);
    __syncthreads();
  }
  if (i < nblk) {
    step(kbuf1, vbuf0, kbuf0, vbuf1, i);
    __syncthreads();
  }

  if (seg.segs > 1) {  // uniform: this segment's partial, merged by the kernel below
#pragma unroll
    for (int g2 = 0; g2 < NG; ++g2) {
      if (!live[g2]) continue;
      const int64_t r = seg_row0 + wave * kFaRows + 16 * g2 + n;
#pragma unroll
      for (int j = 0; j < DB; ++j)
        *reinterpret_cast<f4*>(seg.o + r * D + 16 * j + 4 * kg) = o[j][g2];
      if (kg == 0) {
        // a NaN score reaches l but not the maximum: m = inf then makes the merge's
        // weights NaN, where a small m's would drop the segment from the sum
        const float l = l_acc[g2][0];
        seg.ml[2 * r] = l != l                    ? INFINITY
                        : m_run[g2] == -INFINITY ? -INFINITY
                                                  : qscale * m_run[g2];
        seg.ml[2 * r + 1] = l;
      }
    }
    return;
  }
  // o[j][g2][r] = O^T[dim 16j + 4kg + r][query 16*g2 + n]
#pragma unroll
  for (int g2 = 0; g2 < NG; ++g2) {
    const float l = l_acc[g2][0];
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    T* orow = out + row_offset(live[g2] ? wrow0 + 16 * g2 + n : 0);
    // two dim blocks' 8-byte pieces trade places between the lanes of a row's
    // 16-lane groups, so that a lane stores 16 bytes: group kg the dims 16 (j +
    // kg % 2) + 8 (kg / 2) .. + 7
    // (8-byte stores: 106 against 103 us on 12 ragged prompts of 17 - 1500 rows,
    // 32 heads on 8 kv heads; a tile's end took 2.7 us of its 29)
#pragma unroll
    for (int j = 0; j < DB; j += 2) {
      uint32_t w[2][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const auto r = __builtin_amdgcn_permlane16_swap(
            pack_op2(o[j][g2][2 * h] * inv, o[j][g2][2 * h + 1] * inv, O{}),
            pack_op2(o[j + 1][g2][2 * h] * inv, o[j + 1][g2][2 * h + 1] * inv, O{}), false, false);
        w[0][h] = r[0];
        w[1][h] = r[1];
      }
      if (live[g2])
        *reinterpret_cast<uint4*>(orow + 16 * (j + kg % 2) + 8 * (kg / 2)) =
            make_uint4(w[0][0], w[0][1], w[1][0], w[1][1]);
    }
  }
}

constexpr int kFaTileRows = 128;  // rows (queries x heads of a GQA group) per workgroup

// Merge of the segments of a tile's rows: one wave per row, 8 waves a workgroup,
// blockIdx.y the tile's group of 8 rows.  A segment without keys for the row
// (m = -inf) has its o, possibly unwritten, selected out; one whose weight
// underflows takes part (a NaN or inf among its values has to show).
constexpr int kMergeRows = 8;
template <typename T, int D>
__global__ void __launch_bounds__(64 * kMergeRows)
prefill_merge_kernel(PlanArg plan_arg, int batch, int hq, int kvh, FastDiv rep_div,
                     T* __restrict__ out, SegWs seg) {
  const int unit = static_cast<int>(blockIdx.x) / kvh;
  const int kvhead = static_cast<int>(blockIdx.x) - unit * kvh;
  cint32* cq = (cint32*)__builtin_amdgcn_kernarg_segment_ptr();
  const uint32_t u = static_cast<uint32_t>(cq[2 * (batch + 1) + unit]);
  const int b = static_cast<int>(u & 0xffffu), tile = static_cast<int>(u >> 16);
  const int rep = static_cast<int>(rep_div.d);
  const int q_start = cq[b];
  const int rows = (cq[b + 1] - q_start) * rep;
  const int lane = threadIdx.x & 63;
  const int r = kMergeRows * blockIdx.y + (threadIdx.x >> 6);  // of the tile
  const int row = tile * kFaTileRows + r;
  if (row >= rows) return;  // whole wave: no barrier below
  const int64_t first = static_cast<int64_t>(blockIdx.x) * seg.segs * kFaTileRows + r;
  // lane s: segment s's (m, l); at most 32 segments
  float m = -INFINITY, l = 0.0f;
  if (lane < seg.segs) {
    const float2 x = *reinterpret_cast<const float2*>(
        seg.ml + 2 * (first + static_cast<int64_t>(lane) * kFaTileRows));
    m = x.x;
    l = x.y;
  }
  const uint64_t written = __builtin_amdgcn_ballot_w64(m != -INFINITY);
  const float mx = max_wave64(m);
  const float w = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mx);
  const float lsum = sum_wave64(w * l);
  constexpr int PL = D / 64;  // dims per lane
  float acc[PL];
#pragma unroll
  for (int i = 0; i < PL; ++i) acc[i] = 0.0f;
#pragma unroll 4
  for (int s = 0; s < seg.segs; ++s) {
    const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), s));
    const float* o = seg.o + (first + static_cast<int64_t>(s) * kFaTileRows) * D + PL * lane;
#pragma unroll
    for (int i = 0; i < PL; ++i) acc[i] += (written >> s) & 1 ? ws * o[i] : 0.0f;
  }
  const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
  const int i = static_cast<int>(rep_div.div(static_cast<uint32_t>(row)));
  T* orow = out + (static_cast<int64_t>(q_start + i) * hq + kvhead * rep + (row - i * rep)) * D;
#pragma unroll
  for (int k = 0; k < PL; ++k) orow[PL * lane + k] = from_f32<T>(acc[k] * inv);
}

// The 64-key-block kernel: 16-bit inputs, head sizes 64, 128 and 256, on a
// device with its LDS.  The tiles come from `arg` (num_units units; the only
// form that may be cut into segments), from a plan on the device, or from
// cu_q / cu_k: num_units = batch * tiles, every request's `tiles` tiles.
// *launched: false when another kernel has to run.
struct FaTiles {
  const PlanArg* arg;
  const int32_t* plan;
  const int32_t* cu_q;
  const int32_t* cu_k;
  int64_t batch, num_units, tiles;
};

// The keys and values are on 16-byte bounds, which their DMA into LDS takes in
// 16-byte lanes; views off them run prefill_attn_kernel.
int fa_applies(const void* key, const void* value, int dtype, int head_size, bool* applies) {
  *applies = false;
  if (dtype != KVQ_DTYPE_BF16 && dtype != KVQ_DTYPE_F16) return KVQ_OK;
  if (head_size != 64 && head_size != 128 && head_size != 256) return KVQ_OK;
  if (!aligned16(key, value)) return KVQ_OK;
  int64_t lds_max = 0;  // LDS one workgroup may use on this device
  const int lrc = device_lds_max(&lds_max);
  if (lrc != KVQ_OK) return lrc;
  *applies = lds_max >= (head_size == 64    ? FaLds<64>::BYTES
                         : head_size == 128 ? FaLds<128>::BYTES
                                            : FaLds<256>::BYTES);
  return KVQ_OK;
}

int launch_fa(const void* query, const void* key, const void* value, int dtype, const FaTiles& t,
              int num_heads, int num_kv_heads, int head_size, float qscale, int causal, void* out,
              SegWs seg, hipStream_t s, bool* launched) {
  *launched = false;
  bool applies = false;
  const int arc = fa_applies(key, value, dtype, head_size, &applies);
  if (arc != KVQ_OK || !applies) return arc;
  if (t.num_units * num_kv_heads > 0x7fffffff || t.tiles > 0x7fffffff / kFaTileRows)
    return KVQ_ERR_INVALID;
  const unsigned wgs = static_cast<unsigned>(t.num_units * num_kv_heads);
  const dim3 grid(wgs, static_cast<unsigned>(seg.segs));
  const FastDiv rep_div = FastDiv::make(static_cast<uint32_t>(num_heads / num_kv_heads));
  static const PlanArg none{};
  const PlanArg& arg = t.arg ? *t.arg : none;
#define KVQ_PREFILL_FA(TT, DD)                                                              \
  {                                                                                          \
    hipLaunchKernelGGL((prefill_attn_fa_kernel<TT, DD, fa_ng<DD>()>), grid,                  \
                       dim3(64 * (8 / fa_ng<DD>())), FaLds<DD>::BYTES, s, arg, t.plan,       \
                       static_cast<int>(t.batch), static_cast<const TT*>(query),             \
                       static_cast<const TT*>(key), static_cast<const TT*>(value), t.cu_q,   \
                       t.cu_k, static_cast<int>(t.tiles), num_heads, num_kv_heads, rep_div,  \
                       qscale, causal, static_cast<TT*>(out), seg);                          \
    if (seg.segs > 1)                                                                        \
      hipLaunchKernelGGL((prefill_merge_kernel<TT, DD>),                                     \
                         dim3(wgs, kFaTileRows / kMergeRows), dim3(64 * kMergeRows), 0, s,   \
                         arg, static_cast<int>(t.batch), num_heads, num_kv_heads, rep_div,   \
                         static_cast<TT*>(out), seg);                                        \
    break;                                                                                   \
  }
#define KVQ_PREFILL_FA_D(TT)              \
  switch (head_size) {                    \
    case 64: KVQ_PREFILL_FA(TT, 64)       \
    case 128: KVQ_PREFILL_FA(TT, 128)     \
    default: KVQ_PREFILL_FA(TT, 256)      \
  }
  if (dtype == KVQ_DTYPE_BF16) {
    KVQ_PREFILL_FA_D(kvq::bf16)
  } else {
    KVQ_PREFILL_FA_D(kvq::f16)
  }
#undef KVQ_PREFILL_FA_D
#undef KVQ_PREFILL_FA
  KVQ_LAUNCH_CHECK();
  *launched = true;
  return KVQ_OK;
}

}  // namespace

extern "C" int kvq_prefill_attn(const void* query, const void* key, const void* value, int dtype,
                                const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                int64_t batch, int64_t max_q_len, int num_heads,
                                int num_kv_heads, int head_size, float scale, int causal,
                                void* out, void* stream) {
  if (batch == 0 || max_q_len == 0) return KVQ_OK;
  if (!query || !key || !value || !cu_seqlens_q || !cu_seqlens_k || !out || batch < 0 ||
      max_q_len < 0 || batch > 65535 || num_heads > 65535)
    return KVQ_ERR_INVALID;
  if (num_kv_heads <= 0 || num_heads % num_kv_heads) return KVQ_ERR_GEOMETRY;
  if (head_size != 64 && head_size != 128 && head_size != 256 && head_size != 32)
    return KVQ_ERR_GEOMETRY;
  if (!(scale > 0.0f)) return KVQ_ERR_INVALID;  // the softmax max runs over raw scores
  hipStream_t s = static_cast<hipStream_t>(stream);
  const float qscale = scale * 1.4426950408889634f;
  const int64_t rows = max_q_len * (num_heads / num_kv_heads);
  const int64_t tiles = (rows + kFaTileRows - 1) / kFaTileRows;
  bool launched = false;
  const FaTiles t{nullptr, nullptr, cu_seqlens_q, cu_seqlens_k, batch, batch * tiles, tiles};
  const int frc = launch_fa(query, key, value, dtype, t, num_heads, num_kv_heads, head_size,
                            qscale, causal, out, SegWs{nullptr, nullptr, 1}, s, &launched);
  if (frc != KVQ_OK || launched) return frc;
  const int64_t qblocks = (max_q_len + 63) / 64;
  if (qblocks > 0x7fffffff) return KVQ_ERR_INVALID;
  const dim3 grid(static_cast<unsigned>(qblocks), num_heads, static_cast<unsigned>(batch));
#define KVQ_PREFILL(DD)                                                                  \
  KVQ_DISPATCH_FLOAT(dtype, T,                                                           \
    hipLaunchKernelGGL((prefill_attn_kernel<T, DD>), grid, dim3(256), 0, s,              \
                       static_cast<const T*>(query), static_cast<const T*>(key),          \
                       static_cast<const T*>(value), cu_seqlens_q, cu_seqlens_k,          \
                       num_heads, num_kv_heads, qscale, causal, static_cast<T*>(out)))
  switch (head_size) {
    case 32: KVQ_PREFILL(32); break;
    case 64: KVQ_PREFILL(64); break;
    case 128: KVQ_PREFILL(128); break;
    default: KVQ_PREFILL(256); break;
  }
#undef KVQ_PREFILL
  KVQ_LAUNCH_CHECK();
  return KVQ_OK;
}

namespace {

struct Unit {
  int64_t group, cost;  // descending sort keys
  uint32_t unit;        // request | tile << 16
};

// The tiles of a batch with their cost in key blocks; *most the largest cost.
// KVQ_ERR_CAPACITY past `cap` tiles or outside the packed unit's range.
int64_t plan_units(const int64_t* q_lens, const int64_t* kv_lens, int64_t batch, int64_t rep,
                   int causal, int64_t cap, int64_t* most, std::vector<Unit>* all) {
  int64_t nq = 0, nk = 0, n = 0;
  *most = 0;
  for (int64_t b = 0; b < batch; ++b) {
    const int64_t lq = q_lens[b], lk = kv_lens[b];
    if (lq < 0 || lk < 0) return KVQ_ERR_INVALID;
    nq += lq;
    nk += lk;
    if (nq * rep > 0x7fffffff || nk > 0x7fffffff) return KVQ_ERR_INVALID;
    const int64_t rows = lq * rep, tiles = (rows + kFaTileRows - 1) / kFaTileRows;
    if (n + tiles > cap || tiles > 0x10000 || b > 0xffff) return KVQ_ERR_CAPACITY;
    n += tiles;
    for (int64_t t = 0; t < tiles; ++t) {
      const int64_t last = (std::min<int64_t>((t + 1) * kFaTileRows, rows) - 1) / rep;
      const int64_t end = causal ? std::min(lk, lk - lq + last + 1) : lk;
      const int64_t cost = end <= 0 ? 0 : (end + kFaBlock - 1) / kFaBlock;
      *most = std::max(*most, cost);
      if (all) all->push_back({0, cost, static_cast<uint32_t>(b | (t << 16))});
    }
  }
  return n;
}

// Segments per tile.  A launch of fewer tiles than the chip holds workgroups
// leaves the rest of it idle while each tile walks its keys alone (8 query
// heads on 1 kv head, 16 rows over 8K keys: 128 blocks on 1 of 256 CUs), so its
// keys are cut, into segments of at least 4 blocks (a segment's start and end
// cost about 3) that fit the chip at once, where the blocks this takes off the
// longest tile outweigh the partials' way through memory.  In microseconds, as
// measured on 1 - 256 tiles of 4 - 128 rows over 768 - 12K keys: a block of the
// longest tile 1.05 (1.5 at 256 dims, 0.85 at 64), 1.4 times that where two workgroups
// share a CU, the merge 3.5 + 0.2 a segment + 0.5 a MB of partials.  8 requests
// of 60 rows over 1K keys, 64 heads on 8 kv heads: 27.8 whole, 41.1 in two
// segments; 3 of them over 2K keys 41.7, 35.6 in three; 1 over 3K on 1 kv head 58,
// 18 in ten.
int64_t plan_segs(int64_t units, int64_t most, int64_t rows, int kvh, int head_size, int cus) {
  if (cus <= 0) return 1;
  const double wgs = static_cast<double>(std::max<int64_t>(1, units * kvh));
  const int64_t slots = static_cast<int64_t>(cus) * (head_size == 256 ? 1 : 2);
  const int64_t fit =
      std::min<int64_t>({slots / std::max<int64_t>(1, units * kvh), most / 4, 32});
  const double block = head_size == 256 ? 1.5 : head_size == 128 ? 1.05 : 0.85;
  const double row_mb = static_cast<double>(rows) * kvh * (head_size + 2) * 4e-6;
  int64_t best = 1;
  double least = block * static_cast<double>(most) - 1.5;  // whole, and what a cut has to save
  for (int64_t segs = 2; segs <= fit; ++segs) {
    const double share = std::min(1.0, std::max(0.0, wgs * static_cast<double>(segs) / cus - 1.0));
    const double us = block * static_cast<double>((most + segs - 1) / segs) * (1.0 + 0.4 * share) +
                      3.5 + static_cast<double>(segs) * (0.2 + 0.5 * row_mb);
    if (us < least) {
      least = us;
      best = segs;
    }
  }
  return best;
}

int64_t plan_segs(int64_t units, int64_t most, int64_t rows, int kvh, int head_size) {
  int cus = 0;
  if (device_cu_count(&cus) != KVQ_OK) return 1;
  return plan_segs(units, most, rows, kvh, head_size, cus);
}

// Rows of one kv head of a batch whose lengths plan_units accepts.
int64_t head_rows(const int64_t* q_lens, int64_t batch, int64_t rep) {
  int64_t n = 0;
  for (int64_t b = 0; b < batch; ++b) n += q_lens[b];
  return n * rep;
}

int64_t seg_rows(int64_t units, int kvh, int64_t segs) { return units * kvh * segs * kFaTileRows; }

bool plan_args_ok(const int64_t* q_lens, const int64_t* kv_lens, int64_t batch, int num_heads,
                  int num_kv_heads, int head_size) {
  return batch >= 0 && (batch == 0 || (q_lens && kv_lens)) && num_kv_heads > 0 && num_heads > 0 &&
         num_heads % num_kv_heads == 0 && head_size > 0;
}

// Host side of a planned call: the cumulative lengths and the tiles in the
// order they should start.  Long tiles start first, so that the last to end are
// short.  Where the keys and values an XCD streams outgrow its 4 MB L2 twice
// over, a request's tiles stay together (the requests by falling cost), so that
// one request's keys are in use at a time.
int64_t write_plan(const int64_t* q_lens, const int64_t* kv_lens, int64_t batch, int num_heads,
                   int num_kv_heads, int head_size, int causal, int32_t* plan, int64_t cap_units,
                   int64_t* most) {
  std::vector<Unit> all;
  const int64_t n = plan_units(q_lens, kv_lens, batch, num_heads / num_kv_heads, causal,
                               cap_units, most, &all);
  if (n < 0) return n;
  int32_t* cu_q = plan;
  int32_t* cu_k = plan + batch + 1;
  cu_q[0] = cu_k[0] = 0;
  for (int64_t b = 0; b < batch; ++b) {
    cu_q[b + 1] = cu_q[b] + static_cast<int32_t>(q_lens[b]);
    cu_k[b + 1] = cu_k[b] + static_cast<int32_t>(kv_lens[b]);
  }
  const int64_t xcd_bytes =
      static_cast<int64_t>(cu_k[batch]) * head_size * 4 * std::max(1, num_kv_heads / 8);
  if (xcd_bytes > (int64_t{8} << 20))
    for (auto& u : all) u.group = q_lens[u.unit & 0xffff] * kv_lens[u.unit & 0xffff];
  std::stable_sort(all.begin(), all.end(), [](const Unit& x, const Unit& y) {
    if (x.group != y.group) return x.group > y.group;
    if (x.group != 0 && (x.unit & 0xffff) != (y.unit & 0xffff))
      return (x.unit & 0xffff) < (y.unit & 0xffff);
    return x.cost > y.cost;
  });
  int32_t* units = plan + 2 * (batch + 1);
  for (int64_t i = 0; i < n; ++i) units[i] = static_cast<int32_t>(all[static_cast<size_t>(i)].unit);
  return n;
}

int64_t plan_arg_cap(int64_t batch) { return kPlanArgWords - 2 * (batch + 1); }

}  // namespace

extern "C" int64_t kvq_plan_prefill_attn(const int64_t* q_lens, const int64_t* kv_lens,
                                         int64_t batch, int num_heads, int num_kv_heads,
                                         int head_size, int causal, int32_t* plan,
                                         int64_t cap_units) {
  if (!plan || !plan_args_ok(q_lens, kv_lens, batch, num_heads, num_kv_heads, head_size))
    return KVQ_ERR_INVALID;
  int64_t most = 0;
  return write_plan(q_lens, kv_lens, batch, num_heads, num_kv_heads, head_size, causal, plan,
                    cap_units, &most);
}

extern "C" int kvq_prefill_attn_planned(const void* query, const void* key, const void* value,
                                        int dtype, const int32_t* plan, int64_t batch,
                                        int64_t num_units, int num_heads, int num_kv_heads,
                                        int head_size, float scale, int causal, void* out,
                                        void* stream) {
  if (batch == 0 || num_units == 0) return KVQ_OK;
  if (!query || !key || !value || !plan || !out || batch < 0 || num_units < 0)
    return KVQ_ERR_INVALID;
  if (num_kv_heads <= 0 || num_heads % num_kv_heads) return KVQ_ERR_GEOMETRY;
  if (!(scale > 0.0f)) return KVQ_ERR_INVALID;
  bool launched = false;
  const FaTiles t{nullptr, plan, nullptr, nullptr, batch, num_units, 0};
  const int rc = launch_fa(query, key, value, dtype, t, num_heads, num_kv_heads, head_size,
                           scale * 1.4426950408889634f, causal, out, SegWs{nullptr, nullptr, 1},
                           static_cast<hipStream_t>(stream), &launched);
  if (rc != KVQ_OK) return rc;
  return launched ? KVQ_OK : KVQ_ERR_GEOMETRY;
}

extern "C" int64_t kvq_prefill_attn_segments(const int64_t* q_lens, const int64_t* kv_lens,
                                             int64_t batch, int num_heads, int num_kv_heads,
                                             int head_size, int causal, int cu_count) {
  if (!plan_args_ok(q_lens, kv_lens, batch, num_heads, num_kv_heads, head_size))
    return KVQ_ERR_INVALID;
  if (plan_arg_cap(batch) <= 0) return KVQ_ERR_CAPACITY;
  int64_t most = 0;
  const int64_t n = plan_units(q_lens, kv_lens, batch, num_heads / num_kv_heads, causal,
                               plan_arg_cap(batch), &most, nullptr);
  return n < 0 ? n
               : plan_segs(n, most, head_rows(q_lens, batch, num_heads / num_kv_heads),
                           num_kv_heads, head_size, cu_count);
}

extern "C" int64_t kvq_prefill_attn_lens_workspace_bytes(const int64_t* q_lens,
                                                         const int64_t* kv_lens, int64_t batch,
                                                         int num_heads, int num_kv_heads,
                                                         int head_size, int causal) {
  if (!plan_args_ok(q_lens, kv_lens, batch, num_heads, num_kv_heads, head_size))
    return KVQ_ERR_INVALID;
  if (plan_arg_cap(batch) <= 0) return KVQ_ERR_CAPACITY;
  int64_t most = 0;
  const int64_t n = plan_units(q_lens, kv_lens, batch, num_heads / num_kv_heads, causal,
                               plan_arg_cap(batch), &most, nullptr);
  if (n <= 0) return n;
  const int64_t segs = plan_segs(n, most, head_rows(q_lens, batch, num_heads / num_kv_heads),
                                 num_kv_heads, head_size);
  return segs == 1 ? 0 : seg_rows(n, num_kv_heads, segs) * (head_size + 2) * 4;
}

extern "C" int kvq_prefill_attn_lens(const void* query, const void* key, const void* value,
                                     int dtype, const int64_t* q_lens, const int64_t* kv_lens,
                                     int64_t batch, int num_heads, int num_kv_heads,
                                     int head_size, float scale, int causal, void* workspace,
                                     int64_t workspace_bytes, void* out, void* stream) {
  if (!plan_args_ok(q_lens, kv_lens, batch, num_heads, num_kv_heads, head_size))
    return KVQ_ERR_INVALID;
  if (batch == 0) return KVQ_OK;
  if (!query || !key || !value || !out || !(scale > 0.0f)) return KVQ_ERR_INVALID;
  bool applies = false;
  const int arc = fa_applies(key, value, dtype, head_size, &applies);
  if (arc != KVQ_OK) return arc;
  if (!applies) return KVQ_ERR_GEOMETRY;
  if (plan_arg_cap(batch) <= 0) return KVQ_ERR_CAPACITY;
  PlanArg arg;
  int64_t most = 0;
  const int64_t n = write_plan(q_lens, kv_lens, batch, num_heads, num_kv_heads, head_size, causal,
                               arg.w, plan_arg_cap(batch), &most);
  if (n <= 0) return static_cast<int>(n);
  // without the workspace (or on another device than it was sized on) the keys
  // stay whole
  SegWs seg{nullptr, nullptr, 1};
  const int64_t segs = plan_segs(n, most, head_rows(q_lens, batch, num_heads / num_kv_heads),
                                 num_kv_heads, head_size);
  const int64_t rows = seg_rows(n, num_kv_heads, segs);
  if (segs > 1 && workspace && workspace_bytes >= rows * (head_size + 2) * 4) {
    seg.o = static_cast<float*>(workspace);
    seg.ml = seg.o + rows * head_size;
    seg.segs = static_cast<int>(segs);
  }
  bool launched = false;
  const FaTiles t{&arg, nullptr, nullptr, nullptr, batch, n, 0};
  return launch_fa(query, key, value, dtype, t, num_heads, num_kv_heads, head_size,
                   scale * 1.4426950408889634f, causal, out, seg,
                   static_cast<hipStream_t>(stream), &launched);
}
