// SPDX-License-Identifier: Apache-2.0
// KIVI INT4 decode of a plan's pieces, one wave per (pieces, kv head), the waves
// of a workgroup merging their partial results on the chip, for MI355X (gfx950).
//
// Why: the page-streaming kernel (decode_coop.hip) lives on the 8 kv heads of a
// page; one rank of a tensor-parallel layer holds 1, 2 or 4 of them (1 with 256
// dims in the reference's serving geometry).  A wave per (piece, kv head) fills
// the chip with 2048 / kvh pieces, and as every one leaves a split-K partial (o
// per query head in fp32, written and read back) the partials rival the int4
// pages and the combine walks tens of items per request.  Consecutive pieces
// are consecutive positions, so a workgroup of NW waves takes NW * ppw of them:
// its waves run free, each over its own pieces, and where they end in the same
// request they leave one partial between them.
//
// Head size 256 had no MFMA path (the generic fp32 kernel: 4650 us for 64
// requests of 1K-16K positions on 1 kv head, against 32 us for its 166 MB at
// the copy rate; 69 here, its combine included).
//
// Tiles: 64 positions, decode_tr.h's layout and compute, double-buffered in the
// wave's own LDS: the DMA of the next tile is in flight while one computes.  The
// DMAs are inline asm from a uniform base plus lane offsets that are fixed for
// the kernel, so the waits are explicit: vector memory operations complete in
// issue order, and the NINST DMAs of the next tile are the youngest.  NW = 4:
//   D = 128: 2 workgroups a CU (8 x 19-20 KB of LDS), one piece a wave;
//   D = 256: 1 workgroup a CU (4 x 38-40 KB), two pieces a wave where the plan
//            has more of them than the chip holds waves.
// What bounds it: at D = 256 the issue of one wave per SIMD (a tile's 1600 vector,
// 128 matrix and 270 scalar instructions take some 6 us, of them 0.95 waiting for
// its DMA; the wave issues vector instructions in 45% of its cycles), at
// D = 128 the start: every wave's first tile, 20 MB over the chip, takes 5 - 6 of
// 22 us on 40 requests of 1K-10K positions and 2 kv heads.  Hence the query rows
// through LDS (the second tile leaves before the first is there), the key
// group's operands kept over its two tiles, and MFMA results in ordinary
// registers (a build flag): 69.1 -> 62.0 us on the 64 requests above, 58.4 ->
// 52.6 on 20 of 0.5K-10K with 2 kv heads of 256, 40.5 -> 38.7 on the 40.  (What
// keeps fp32's bits at 256 dims then added 6 us: P' 4, the tails 2.)
#include <algorithm>

#include "decode_tail.h"
#include "decode_tr.h"
#include "kvq_common.h"
#include "kvq_decode.h"

namespace {

using namespace kvq;
using tr::f4;

// The plan's tables are read-only for the kernel's lifetime: through the
// constant address space their uniform reads are scalar loads, which do not
// count among the vector memory operations in flight.
typedef const __attribute__((address_space(4))) int32_t cint32;
__device__ __forceinline__ cint32* as_const(const int32_t* p) { return (cint32*)(p); }

// 16 (4) bytes per lane from base + voff (base uniform, voff the lane's byte
// offset) to LDS byte address m0 + 16 (4) * lane (m0 uniform).  The s_nop
// covers the M0-write hazard.
__device__ __forceinline__ void sdma16(const char* base, uint32_t voff, uint32_t m0) {
  m0 = __builtin_amdgcn_readfirstlane(m0);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(voff), "s"(base), "{m0}"(m0)
               : "memory");
}
__device__ __forceinline__ void sdma4(const char* base, uint32_t voff, uint32_t m0) {
  m0 = __builtin_amdgcn_readfirstlane(m0);
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1"
               :
               : "v"(voff), "s"(base), "{m0}"(m0)
               : "memory");
}

// This wave's LDS accesses are done (its vector memory operations need not be).
__device__ __forceinline__ void wait_lds() {
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8));
  asm volatile("" ::: "memory");
}
constexpr int kSplitWaves = 4;

// LDS of one wave: two tile buffers, at least the tail path's staging.
template <int D, int NVG, bool KSV>
constexpr int wave_bytes() {
  constexpr int two = 2 * tr::Tile<NVG, KSV, D>::BYTES;
  constexpr int tail = D == 256 ? tail::kLdsBytesWide : tail::kLdsBytes;
  return two > tail ? two : tail;
}

template <typename TQ, int D, int NVG, bool KSV, bool FOLD>
__global__ void __launch_bounds__(64 * kSplitWaves, D == 256 ? 1 : 2)
kivi_decode_split_kernel(const TQ* __restrict__ query, int hq, int kvh, float qscale,
                         const uint32_t* __restrict__ kq, const float* __restrict__ ks,
                         const float* __restrict__ km, const uint32_t* __restrict__ vq,
                         const float* __restrict__ vs, const float* __restrict__ vm, int bs,
                         int g, int64_t nb, const int32_t* __restrict__ block_table, int64_t maxb,
                         const int32_t* __restrict__ seq_meta, const int32_t* __restrict__ work,
                         const int32_t* __restrict__ pieces, int num_pieces, int ppw,
                         const TQ* __restrict__ ring_k, const TQ* __restrict__ ring_v,
                         int ring_len, float* __restrict__ ws_o, float* __restrict__ ws_ml) {
  using T = tr::Tile<NVG, KSV, D>;
  constexpr int NW = kSplitWaves;
  constexpr int DB = D / 16;
  constexpr int WAVE = wave_bytes<D, NVG, KSV>();
  constexpr int DEP = DB * 1024;  // a wave's partial: o, then m and l of 16 heads, then two ints
  static_assert(DEP + 136 <= WAVE, "a partial fits the wave's LDS");
  extern __shared__ __align__(128) char lds_raw[];
  const int groups = (num_pieces + NW * ppw - 1) / (NW * ppw);
  int gi, h;
  if (!xcd_item_head(blockIdx.x, kvh, groups, gi, h)) return;  // workgroup-uniform
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 15;
  const int kg = lane >> 4;
  const int rep = hq / kvh;
  const int bsh = __builtin_ctz(static_cast<unsigned>(bs));
  const int gsh = __builtin_ctz(static_cast<unsigned>(g));
  const int gpb = bs >> gsh;
  const int wpd = bs >> 3;
  cint32* cwork = as_const(work);
  cint32* ctable = as_const(block_table);
  // the wave's items: those of its ppw pieces (none past the plan's end)
  const int k0 = (gi * NW + w) * ppw;
  const int k1 = k0 + ppw < num_pieces ? k0 + ppw : num_pieces;
  int it0 = 0, it1 = 0;
  if (k0 < num_pieces) {
    it0 = pieces ? as_const(pieces)[k0] : k0;
    it1 = pieces ? as_const(pieces)[k1] : k1;
  }
  char* const my_lds = lds_raw + w * WAVE;
  const uint32_t my_off = tr::lds_off(my_lds);

  // ---- tile DMA: lane offsets of decode_tr.h's layout ---------------------------
  // keys: instruction i copies dims 32 i .. 32 i + 31, lane dim lane >> 1, half
  // (lane & 1) ^ ((lane >> 3) & 1) of its 32 bytes
  const uint32_t k_lane =
      4u * static_cast<uint32_t>((lane >> 1) * wpd + 4 * ((lane & 1) ^ ((lane >> 3) & 1)));
  // values: instruction i copies TPI tokens, lane token lane / CPT, its 16-byte
  // chunk xor-ed with the token's pi, whose instruction part is uniform
  constexpr int CPT = D / 32;      // 16-byte chunks per token row
  constexpr int TPI = 64 / CPT;    // tokens per instruction
  const int v_tok = lane / CPT;
  const uint32_t v_row = static_cast<uint32_t>(v_tok * kvh * (D / 2));
  const uint32_t v_chunk = static_cast<uint32_t>((lane % CPT) ^ ((v_tok >> 1) & 1));
  const uint32_t ks_lane = static_cast<uint32_t>(KSV ? 16 * (lane % (D / 4)) : 4 * lane * gpb);
  const uint32_t vs_lane = static_cast<uint32_t>(
      4 * tr::tau((lane >> 3) & 3, 8 * (lane >> 5) + tr::slot_nib(lane & 7)) * kvh * NVG);
  // DMA of the tile at position p of a request whose page there is blk.  At D =
  // 128 the loops stay rolled: unrolled, their bases spill scalar registers
  // (104 requests of 384 - 506 positions on 4 kv heads 37.7 us, rolled 37.0); at
  // D = 256 rolled costs more than the spills (62.3 against 63.5).
  constexpr int DMA_UNROLL = D == 256 ? 8 : 1;
  auto issue = [&](int64_t blk, int p, int buf) {
    const uint32_t m0 = my_off + static_cast<uint32_t>(buf * T::BYTES);
    const int off0 = p & (bs - 1);
    const int64_t krow = (blk * kvh + h) * D;
    const int64_t vtok = ((blk << bsh) + off0) * kvh + h;
    const char* kb = reinterpret_cast<const char*>(kq + krow * wpd + (off0 >> 3));
    const uint32_t kstep = 128u * static_cast<uint32_t>(wpd);
#pragma unroll DMA_UNROLL
    for (int i = 0; i < T::KW_INST; ++i, kb += kstep)
      sdma16(kb, k_lane, m0 + 4 * T::KW + 1024 * i);
    const char* sb = reinterpret_cast<const char*>(ks + krow * gpb + (off0 >> gsh));
    const char* mb = reinterpret_cast<const char*>(km + krow * gpb + (off0 >> gsh));
    if constexpr (KSV && D == 256) {
      sdma16(sb, ks_lane, m0 + 4 * T::KS);
      sdma16(mb, ks_lane, m0 + 4 * T::KM);
    } else if constexpr (KSV) {
      // lanes 0..31 the scales; 32..63 the minima, which land right after them
      const uint32_t far = static_cast<uint32_t>(mb - sb);
      sdma16(sb, ks_lane + (lane & 32 ? far : 0u), m0 + 4 * T::KS);
    } else {
#pragma unroll
      for (int i = 0; i < D / 64; ++i) {
        sdma4(sb + static_cast<int64_t>(256 * i) * gpb, ks_lane, m0 + 4 * (T::KS + 64 * i));
        sdma4(mb + static_cast<int64_t>(256 * i) * gpb, ks_lane, m0 + 4 * (T::KM + 64 * i));
      }
    }
    const char* vb = reinterpret_cast<const char*>(vq + vtok * (D / 8));
    const uint32_t vstep = static_cast<uint32_t>(TPI * kvh * (D / 2));
#pragma unroll DMA_UNROLL
    for (int i = 0; i < T::VW_INST; ++i, vb += vstep) {
      const uint32_t pi = D == 128 ? i : 2 * (i >> 1);  // of token TPI * i
      sdma16(vb, v_row + 16 * (v_chunk ^ pi), m0 + 4 * T::VW + 1024 * i);
    }
    const char* vsb = reinterpret_cast<const char*>(vs + vtok * NVG);
    const char* vmb = reinterpret_cast<const char*>(vm + vtok * NVG);
#pragma unroll
    for (int vg = 0; vg < NVG; ++vg) {
      sdma4(vsb + 4 * vg, vs_lane, m0 + 4 * (T::VS + 64 * vg));
      sdma4(vmb + 4 * vg, vs_lane, m0 + 4 * (T::VM + 64 * vg));
    }
  };
  // The query rows of request b and this kv head into the second buffer: row r's
  // 16-byte chunk c in its slot c ^ (r % 16), over the banks.
  constexpr int QCH = D / 8;  // chunks per row
  const bool q_aligned = (reinterpret_cast<uintptr_t>(query) & 15) == 0;
  auto stage_q = [&](int b) {
    const char* src = reinterpret_cast<const char*>(
        query + (static_cast<int64_t>(b) * hq + h * rep) * D);
#pragma unroll 1
    for (int i = 0; i * 64 < rep * QCH; ++i) {
      const int r = (64 * i + lane) / QCH, c = (lane % QCH) ^ (r & 15 & (QCH - 1));
      sdma16(src, static_cast<uint32_t>(2 * D * min(r, rep - 1) + 16 * c),
             my_off + static_cast<uint32_t>(T::BYTES) + 1024u * i);
    }
  };
  static_assert(T::BYTES >= 16 * 2 * D, "16 query rows fit a tile buffer");
  auto page_of = [&](int b, int p) -> int64_t {
    const int64_t v = ctable[static_cast<int64_t>(b) * maxb + (p >> bsh)];
    return v < 0 ? 0 : (v >= nb ? nb - 1 : v);  // never leave the cache
  };
  // an item whose positions another item's partial carries: weight 0
  auto mark_merged = [&](int it) {
    if (lane < rep) {
      const int64_t hh = static_cast<int64_t>(it) * hq + h * rep + lane;
      ws_ml[2 * hh] = -INFINITY;
      ws_ml[2 * hh + 1] = 0.0f;
    }
  };

  // ---- the wave's items ------------------------------------------------------------
  // A run is one request's consecutive int4 items (kind 0), or one other item.
  // Every run but the last is stored as it ends, at its first item; the last one
  // meets the other waves' below.
  tail::PartialT<DB> part;
  int run_b = -1, run_first = 0;
  for (int it = it0; it < it1;) {
    if (run_b >= 0) tail::store_o<DB>(part, run_first, hq, h, rep, lane, ws_o, ws_ml);
    run_first = it;
    run_b = cwork[4 * static_cast<int64_t>(it)];
    const int kind = cwork[4 * static_cast<int64_t>(it) + 3];
    if (kind == 1) {
      part = tail::tail_item<TQ, D / 128>(my_lds, query, hq, kvh, qscale, kq, ks, km, vq, vs, vm,
                                          bs, g, nb, block_table, maxb, seq_meta,
                                          work + 4 * static_cast<int64_t>(it), it, h, ring_k,
                                          ring_v, ring_len, 0, 1);
      wait_lds();
      ++it;
      continue;
    }
    // the run's tiles: [pb, pe) of item `it`, then of the next while it continues
    // the request (kinds 2 / 3: every second tile, from the first / second on);
    // tile p is in buffer cb, the next one is issued into the other
    const int st = kind >= 2 ? 128 : 64;
    int pb = cwork[4 * static_cast<int64_t>(it) + 1], pe = cwork[4 * static_cast<int64_t>(it) + 2];
    int p = kind >= 2 ? pb + 64 * (kind - 2) : pb & ~63;
    int64_t ahead = 0;  // page of the tile after the one issued last, in its item
    // the query rows go ahead of the first tile, through the other buffer: a
    // load to registers would be waited for with the tile behind it, and the
    // second tile could not leave before the first is there
    if (q_aligned) stage_q(run_b);
    if (p < pe) {
      issue(page_of(run_b, p), p, 0);
      ahead = page_of(run_b, p + st < pe ? p + st : pe - 1);
    }
    tr::QLane<TQ, D> ql;
    if (q_aligned) {
      if (p < pe)
        wait_vmcnt<T::NINST>();
      else
        wait_vmcnt<0>();
      ql = tr::load_q_at<TQ, D>(
          [&](int hn, int c) {
            return reinterpret_cast<const TQ*>(my_lds + T::BYTES) + hn * D +
                   8 * (c ^ (hn & 15 & (QCH - 1)));
          },
          rep, n, kg, FOLD);
    } else {
      ql = tr::load_q<TQ, D>(query, run_b, hq, h, rep, n, kg, FOLD);
    }
    tr::Acc<NVG, DB> acc;
    acc.init();
    tr::QGroup<D> qg;
    int again = -1;  // the tile that shares the last prepared key group
    int cb = 0;
    while (p < pe) {
      // the tile after p: in this item, or the first of the item that continues it
      const int tb = pb, te = pe;
      int np = p + st;
      if (np >= pe) {
        ++it;
        if (kind == 0 && it < it1 && cwork[4 * static_cast<int64_t>(it) + 3] == 0 &&
            cwork[4 * static_cast<int64_t>(it)] == run_b) {
          mark_merged(it);
          pb = cwork[4 * static_cast<int64_t>(it) + 1];
          pe = cwork[4 * static_cast<int64_t>(it) + 2];
          np = pb & ~63;
          ahead = page_of(run_b, np < pe ? np : pe > 0 ? pe - 1 : 0);
        } else {
          pe = np;  // the run ends
        }
      }
      wait_lds();  // the other buffer's last reads are done
      if (np < pe) {
        issue(ahead, np, cb ^ 1);
        ahead = page_of(run_b, np + st < pe ? np + st : pe - 1);
        wait_vmcnt<T::NINST>();
      } else {
        wait_vmcnt<0>();
      }
      const uint32_t* W = reinterpret_cast<const uint32_t*>(my_lds + cb * T::BYTES);
      // the second tile of a 128-position key group runs on the first one's
      // operands (unfolded, twice the operands, they spill if kept)
      if (!FOLD || p != again) tr::prepare_group<TQ, NVG, KSV, FOLD>(W, n, kg, ql, qscale, qg);
      again = ((p + 64) & (g - 1)) != 0 ? p + 64 : -1;
      const uint32_t off = my_off + static_cast<uint32_t>(cb * T::BYTES);
      if (p >= tb && p + 64 <= te)
        tr::compute_tile<NVG, KSV, FOLD, true, D>(W, off, p, tb, te, n, kg, qg, qscale, acc);
      else
        tr::compute_tile<NVG, KSV, FOLD, false, D>(W, off, p, tb, te, n, kg, qg, qscale, acc);
      asm volatile("" ::: "memory");
      cb ^= 1;
      p = np;
    }
    if (it < it1 && it == run_first) ++it;  // an item without a tile
    tr::finish<NVG, DB>(acc, kg, part.o);
    part.m = acc.m_run;
    part.l = acc.l_run;
    wait_lds();
  }

  // ---- the waves' last runs ---------------------------------------------------------
  // Each wave leaves its run in its LDS; runs of one request merge into the first
  // one's item, wave x writing dims blocks x DB / NW .. of every merged partial.
  {
    char* dep = my_lds;
    if (run_b >= 0) {
      f4* xo = reinterpret_cast<f4*>(dep);
#pragma unroll
      for (int v = 0; v < DB; ++v) xo[v * 64 + lane] = part.o[v];
      float* xml = reinterpret_cast<float*>(dep + DEP);
      if (kg == 0) {
        xml[n] = part.m;
        xml[16 + n] = part.l;
      }
    }
    if (lane == 0) {
      int* info = reinterpret_cast<int*>(dep + DEP + 128);
      info[0] = run_b;
      info[1] = run_first;
    }
  }
  wait_lds();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int rb[NW], rf[NW];
#pragma unroll
  for (int x = 0; x < NW; ++x) {
    const int* info = reinterpret_cast<const int*>(lds_raw + x * WAVE + DEP + 128);
    rb[x] = __builtin_amdgcn_readfirstlane(info[0]);
    rf[x] = __builtin_amdgcn_readfirstlane(info[1]);
  }
#pragma unroll
  for (int x = 0; x < NW; ++x) {
    bool first = rb[x] >= 0;
#pragma unroll
    for (int y = 0; y < x; ++y) first = first && rb[y] != rb[x];
    if (!first) {  // uniform: wave x has no run, or an earlier wave's item carries it
      if (rb[x] >= 0 && w == x) mark_merged(rf[x]);
      continue;
    }
    f4 mx = f4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    f4 wt[NW], ls = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int y = x; y < NW; ++y) {
      if (rb[y] != rb[x]) continue;
      wt[y] = *reinterpret_cast<const f4*>(lds_raw + y * WAVE + DEP + 16 * kg);
#pragma unroll
      for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], wt[y][r]);
    }
    f4 sum[DB / NW];
#pragma unroll
    for (int vi = 0; vi < DB / NW; ++vi) sum[vi] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int y = x; y < NW; ++y) {
      if (rb[y] != rb[x]) continue;
      const f4 ly = *reinterpret_cast<const f4*>(lds_raw + y * WAVE + DEP + 64 + 16 * kg);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // a run without positions has m = -inf, l = 0, o = 0: weight 0
        wt[y][r] = wt[y][r] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(wt[y][r] - mx[r]);
        ls[r] += wt[y][r] * ly[r];
      }
#pragma unroll
      for (int vi = 0; vi < DB / NW; ++vi) {
        const f4 oy =
            reinterpret_cast<const f4*>(lds_raw + y * WAVE)[(w * (DB / NW) + vi) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[vi][r] += wt[y][r] * oy[r];
      }
    }
    const int64_t head0 = static_cast<int64_t>(rf[x]) * hq + h * rep;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int hh = 4 * kg + r;
      if (hh < rep) {
#pragma unroll
        for (int vi = 0; vi < DB / NW; ++vi)
          ws_o[(head0 + hh) * D + 16 * (w * (DB / NW) + vi) + n] = sum[vi][r];
        if (w == 0 && n == 0) {
          ws_ml[2 * (head0 + hh)] = mx[r];
          ws_ml[2 * (head0 + hh) + 1] = ls[r];
        }
      }
    }
  }
}

}  // namespace

namespace kvq {

bool split_decode_applies(int q_dtype, int hq, int kvh, int d, int ring_dtype, int bs, int g) {
  return (d == 128 || d == 256) && (g == 64 || g == 128) && hq % kvh == 0 && hq / kvh <= 16 &&
         ring_dtype == q_dtype && (q_dtype == KVQ_DTYPE_BF16 || q_dtype == KVQ_DTYPE_F16) &&
         bs >= 64 && (bs & (bs - 1)) == 0 && bs % g == 0;
}

int launch_kivi_decode_split(const void* query, int q_dtype, int hq, int kvh, int d, float qscale,
                             const int32_t* kq, const float* ks, const float* km,
                             const int32_t* vq, const float* vs, const float* vm, int bs, int g,
                             int64_t nb, const int32_t* block_table, int64_t maxb,
                             const int32_t* seq_meta, const int32_t* work,
                             int64_t num_work, const int32_t* pieces, int64_t num_pieces,
                             const void* ring_k,
                             const void* ring_v, int ring_dtype, int ring_len, float* ws_o,
                             float* ws_ml, hipStream_t s, bool* launched) {
  *launched = false;
  if (!split_decode_applies(q_dtype, hq, kvh, d, ring_dtype, bs, g)) return KVQ_OK;
  // caches off the DMA's 16-byte lanes: the generic kernel
  if (!(aligned16(kq, vq) && aligned16(ks, km))) return KVQ_OK;
  // a plan without pieces: every item is one (its tail items too)
  if (!pieces) num_pieces = num_work;
  // the lane offsets of a tile's DMAs are 32-bit: a page of all heads, and (in
  // the one-instruction form) the way from the scales to the minima
  if (static_cast<int64_t>(bs) * kvh * d > (int64_t{1} << 30)) return KVQ_OK;
  const bool ksv = bs == g && (d == 256 || (static_cast<int64_t>(km - ks) >= 0 &&
                                            static_cast<int64_t>(km - ks) < (int64_t{1} << 29)));
  int64_t lds_max = 0;
  const int lrc = device_lds_max(&lds_max);
  if (lrc != KVQ_OK) return lrc;
  // one piece a wave, or at D = 256 as many as put the plan's pieces on the
  // waves the chip holds (4 a CU) at once
  int ppw = 1;
  if (d == 256) {
    int cus = 0;
    const int crc = device_cu_count(&cus);
    if (crc != KVQ_OK) return crc;
    const int64_t waves = static_cast<int64_t>(kSplitWaves) * (cus > 0 ? cus : 256);
    ppw = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(2, num_pieces * kvh / waves)));
  }
  const int64_t groups = (num_pieces + kSplitWaves * ppw - 1) / (kSplitWaves * ppw);
  const int64_t blocks = xcd_grid_size(groups, kvh);
  if (blocks > 0x7fffffff) return KVQ_ERR_INVALID;
  const dim3 grid(static_cast<unsigned>(blocks));
  const bool fold = hq / kvh <= 8;
  const uint32_t* kqu = reinterpret_cast<const uint32_t*>(kq);
  const uint32_t* vqu = reinterpret_cast<const uint32_t*>(vq);
#define KVQ_LAUNCH_SPLIT(TQ, D, V, KV, F)                                                      \
  {                                                                                            \
    constexpr int lds = kSplitWaves * wave_bytes<D, V, KV>();                                 \
    if (lds > lds_max) return KVQ_OK; /* not this device: the other kernels run */             \
    hipLaunchKernelGGL((kivi_decode_split_kernel<TQ, D, V, KV, F>), grid,                      \
                       dim3(64 * kSplitWaves), lds, s, static_cast<const TQ*>(query), hq, \
                       kvh, qscale, kqu, ks, km, vqu, vs, vm, bs, g, nb, block_table, maxb,    \
                       seq_meta, work, pieces, static_cast<int>(num_pieces), ppw,              \
                       static_cast<const TQ*>(ring_k), static_cast<const TQ*>(ring_v),         \
                       ring_len, ws_o, ws_ml);                                                 \
  }
#define KVQ_LAUNCH_SPLIT_F(TQ, D, V, KV) \
  if (fold) KVQ_LAUNCH_SPLIT(TQ, D, V, KV, true) else KVQ_LAUNCH_SPLIT(TQ, D, V, KV, false)
#define KVQ_LAUNCH_SPLIT_D(TQ, D)                                                  \
  if (g == 128) {                                                                  \
    if (ksv) { KVQ_LAUNCH_SPLIT_F(TQ, D, D / 128, true) }                          \
    else { KVQ_LAUNCH_SPLIT_F(TQ, D, D / 128, false) }                             \
  } else {                                                                         \
    if (ksv) { KVQ_LAUNCH_SPLIT_F(TQ, D, D / 64, true) }                           \
    else { KVQ_LAUNCH_SPLIT_F(TQ, D, D / 64, false) }                              \
  }
#define KVQ_LAUNCH_SPLIT_T(TQ) \
  if (d == 128) { KVQ_LAUNCH_SPLIT_D(TQ, 128) } else { KVQ_LAUNCH_SPLIT_D(TQ, 256) }
  if (q_dtype == KVQ_DTYPE_BF16) {
    KVQ_LAUNCH_SPLIT_T(bf16)
  } else {
    KVQ_LAUNCH_SPLIT_T(f16)
  }
#undef KVQ_LAUNCH_SPLIT_T
#undef KVQ_LAUNCH_SPLIT_D
#undef KVQ_LAUNCH_SPLIT_F
#undef KVQ_LAUNCH_SPLIT
  KVQ_LAUNCH_CHECK();
  *launched = true;
  return KVQ_OK;
}

}  // namespace kvq
