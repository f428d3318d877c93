// BF16 skinny GEMM / GEMV (M <= 32): y = x . w^T in fp32. Weights row-major, or tiled: the FP8
// tile permutation of include/krq.h applied to the [N, 2K] byte matrix (16 rows x 32 bf16).
// A step is 64 bf16 of K per weight row (two 32-element tiles, one v_mfma_f32_16x16x32_bf16 each);
// M == 1 runs on the vector ALUs with cross-lane sums. Conventions: gemv_common.h.
#include "gemv_common.h"

#include <stdlib.h>

#include <algorithm>
#include <type_traits>

using namespace krq;

namespace {

// How a block's operands are loaded: in the tiles' lane order (64 bytes of sixteen rows per load), in
// whole lines of eight rows that lanes exchange into the tiles' operands (row-major weights too), or so
// with one activation load per step (at most eight rows).
constexpr int kTileLoads = 0, kLineLoads = 1, kOneLine = 2;

// PB = 2 or 4: adjacent row blocks per block sharing the activation loads (as in gemv_fp8.hip;
// 4 for the multi-row lm_head, where every 16-column block re-reads the bf16 rows from L2).
// bx: the column block this workgroup owns (its two-matrix, paired or single row block, or with
// MODE kOutSwiGluHalf its half-pair block).
// CHAIN (the chained BF16 MLP, k_mlp_chain_bf16): a SwiGLU block writes act through to memory and
// counts itself into the first-stage counters; a split-K (partials) block is a second-stage block
// on act, which issues its weight loads, waits for the first stage's done flag (chain_wait; a wait
// that gives up makes the block's partials NaN) and then reads act with agent-scope (sc1) loads,
// and counts its exit. sy >= 0 / nwo > 0: the block's K split and its wave count, given (the
// chained kernel's one-dimensional grid and common block size); waves past nwo end at once.
template <int MT, int MODE, int LAYOUT, int ALGO, int U, int PB, int XM, bool CHAIN = false>
KRQ_DEV void gemv_bf16_body(const uint8_t* __restrict__ x, const uint8_t* __restrict__ w, int M, int64_t NO,
                            int64_t K, int kts, void* __restrict__ out, void* __restrict__ aux, int64_t bx,
                            int sy = -1, int nwo = 0, const FusedArgs* fa = nullptr) {
  extern __shared__ __align__(16) float red[];
  __shared__ float ones[32];
  static_assert(PB == 1 || (MODE != KRQ_OUT_SWIGLU && ALGO != 2), "paired row blocks: MFMA, no SwiGLU");
  static_assert(PB == 1 || PB == 2 || PB == 4, "one, two or four row blocks per block");
  constexpr bool XO = XM == kOneLine;
  static_assert(!XO || MT == 1, "one activation load per step: at most eight rows");
  static_assert(ALGO != 2 || XM == kTileLoads || (XO && LAYOUT == KRQ_W_ROWMAJOR), "one row: no lines on packed weights");
  static_assert(!CHAIN || (PB == 1 && (MODE == KRQ_OUT_SWIGLU || MODE == kOutSwiGluHalf || MODE == KRQ_OUT_PARTIAL)),
                "chained MLP: SwiGLU first stage, partials second stage");
  constexpr bool WAITS = CHAIN && MODE == KRQ_OUT_PARTIAL;  // (second stage)
  constexpr int P = MODE == KRQ_OUT_SWIGLU ? 2 : PB;  // weight row blocks streamed per step
  constexpr int NV = MT * 256;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = nwo > 0 ? nwo : blockDim.x >> 6;
  if (CHAIN && __builtin_amdgcn_readfirstlane(wave) >= nw) return;
  const int r = lane & 15, g = lane >> 4;
  const int64_t rb = bx * PB;
  const int sidx = sy >= 0 ? sy : static_cast<int>(blockIdx.y);
  const int nsteps = (kts + 1) >> 1;
  const int64_t tbase = (int64_t)sidx * kts;
  const int64_t rowb = 2 * K;
  const int jcount = wave < nsteps ? (nsteps - wave + nw - 1) / nw : 0;
  constexpr bool RM = LAYOUT == KRQ_W_ROWMAJOR && XM != kTileLoads;  // weights in whole lines (w_line_chunk)
  if (threadIdx.x < 32) ones[threadIdx.x] = 1.0f;
  // weight set p: the up half of the SwiGLU, else the p-th row block of this block
  auto rbp = [&](int p) -> int64_t { return MODE == KRQ_OUT_SWIGLU && p == 1 ? rb + (NO >> 4) : rb + p; };

  v4f acc[P][MT];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[p][mt] = v4f{0.f, 0.f, 0.f, 0.f};
  float sv[P][2];  // vector-ALU partial sums (ALGO 2) of the low and high tile of each step
#pragma unroll
  for (int p = 0; p < P; ++p) sv[p][0] = sv[p][1] = 0.f;
  // a ring of U step slots: consume slot u (step cc), then refill it with step cc + U
  uint4 wl[P][U], wh[P][U], xl[U][MT], xh[U][MT];
  // Every slot load is issued unconditionally (a branch around a load makes the compiler drain all
  // outstanding loads at the join): a slot past this wave's last step reloads that step (already
  // in flight or cached) and is masked where consumed; rows m >= M read row M - 1, whose products
  // land in accumulator rows the epilogue never writes.
  // (WAITS: act, written in this launch on every XCD, read with sc1 loads through a buffer resource)
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(x), (short)0, WAITS ? static_cast<int>(M * rowb) : 0, 0x00020000);
  auto load_w = [&](int u, int cc) {
    const int j = jcount > 0 ? wave + min(cc, jcount - 1) * nw : 0;
    const int64_t t0 = tbase + 2 * j;
    const int64_t t1 = (2 * j + 1 < kts) ? t0 + 1 : t0;
    if constexpr (RM) {
      const int64_t o = t0 * 64 + 16 * w_line_chunk(lane, 2 * j + 1 >= kts);
#pragma unroll
      for (int p = 0; p < P; ++p) {  // (a half-pair block: its eight gate rows, then the up rows)
        const int64_t row = (MODE == kOutSwiGluHalf ? 8 * rb : 16 * rbp(p)) + (r & 7);
        wl[p][u] = ld16nt(w + row * rowb + o);
        wh[p][u] = ld16nt(w + (row + (MODE == kOutSwiGluHalf ? NO : 8)) * rowb + o);
      }
    } else if constexpr (MODE == kOutSwiGluHalf) {
      wl[0][u] = ld16nt(w_addr_hp<LAYOUT>(w, rb, NO, t0, rowb, lane));
      wh[0][u] = ld16nt(w_addr_hp<LAYOUT>(w, rb, NO, t1, rowb, lane));
    } else {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        wl[p][u] = ld16nt(w_addr<LAYOUT>(w, rbp(p), t0, rowb, lane));
        wh[p][u] = ld16nt(w_addr<LAYOUT>(w, rbp(p), t1, rowb, lane));
      }
    }
  };
  // The activations in whole lines too, row by row as row-major weights; XO: one load per step, the lane
  // columns c and c + 8 taking the two halves of row c's line.
  constexpr bool XL = XM != kTileLoads;
  auto load_x = [&](int u, int cc) {
    const int j = jcount > 0 ? wave + min(cc, jcount - 1) * nw : 0;
    const int64_t t0 = tbase + 2 * j;
    const int64_t t1 = (2 * j + 1 < kts) ? t0 + 1 : t0;
    const int64_t o = t0 * 64 + 16 * w_line_chunk(lane, 2 * j + 1 >= kts);
    auto ld = [&](int m, int64_t a) -> uint4 {
      if constexpr (WAITS)
        return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                             xrs, static_cast<int>(m * rowb) + static_cast<int>(a), 0, 16));
      else
        return ld16(x + m * rowb + a);
    };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if constexpr (!XL) {
        const int m = ALGO == 2 ? 0 : min(mt * 16 + r, M - 1);
        xl[u][mt] = ld(m, t0 * 64 + g * 16);
        xh[u][mt] = ld(m, t1 * 64 + g * 16);
      } else {
        const int m = ALGO == 2 ? 0 : mt * 16 + (r & 7);
        xl[u][mt] = ld(min(m, M - 1), o);
        if constexpr (!XO) xh[u][mt] = ld(min(m + 8, M - 1), o);
      }
    }
  };
  auto load_slot = [&](int u, int cc) {
    load_w(u, cc);
    load_x(u, cc);
  };
  // LAST: the step may be past this wave's last one, or the split's half step (one tile of two). On the
  // vector ALUs what is not there is skipped (four layers row-major at M = 1 183.0 us, 188.7 masked);
  // on the matrix cores, which ignore the execution mask, the activations are zeroed with the
  // weights, since an infinite one times zero is NaN.
  const int jlast = __builtin_amdgcn_readfirstlane(jcount), wv = __builtin_amdgcn_readfirstlane(wave);
  auto consume_slot = [&](auto last, int u, int cc) {
    constexpr bool LAST = decltype(last)::value, SKIP = LAST && ALGO == 2;
    const int cs = __builtin_amdgcn_readfirstlane(cc);
    if (SKIP && cs >= jlast) return;
    const int j = SKIP ? wv + cs * nw : jcount > 0 ? wave + min(cc, jcount - 1) * nw : 0;
    const bool ok = SKIP || cc < jcount, hi = ok && (2 * j + 1 < kts);
    uint4 al[MT], ah[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      al[mt] = xl[u][mt];
      ah[mt] = xh[u][mt];
      if constexpr (XL) lines_to_tiles(xl[u][mt], XO ? xl[u][mt] : xh[u][mt], &al[mt], &ah[mt]);
      if constexpr (LAST && !SKIP) {
        al[mt] = sel4(ok, al[mt]);
        ah[mt] = sel4(hi, ah[mt]);
      }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      uint4 bl = wl[p][u], bh = wh[p][u];
      if constexpr (RM) lines_to_tiles(wl[p][u], wh[p][u], &bl, &bh);
      if constexpr (LAST && !SKIP) {
        bl = sel4(ok, bl);
        bh = sel4(hi, bh);
      }
      if (ALGO == 2) {
        sv[p][0] = dot8_bf16(bl, al[0], sv[p][0]);
        if (!SKIP || hi) sv[p][1] = dot8_bf16(bh, ah[0], sv[p][1]);
      } else {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          acc[p][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(al[mt]), as_v8bf(bl), acc[p][mt], 0, 0, 0);
          acc[p][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(ah[mt]), as_v8bf(bh), acc[p][mt], 0, 0, 0);
        }
      }
    }
  };
  bool chain_bad = false;
  if constexpr (WAITS) {  // the weights first, then the wait, then act
#pragma unroll
    for (int u = 0; u < U; ++u) load_w(u, u);
    chain_bad = !chain_wait(*fa);
#pragma unroll
    for (int u = 0; u < U; ++u) load_x(u, u);
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) load_slot(u, u);
  }
  __builtin_amdgcn_sched_barrier(0);
  // the last batch is peeled off (consume only), so no load sits behind a branch and the first
  // batch's loads stay ahead of everything else
  int base = 0;
  if constexpr (WAITS) {
    // One batch peeled off, unconditionally (past jcount it reloads the last step and consumes
    // nothing): the first batch's loads went out weights first, act after the wait, and a loop
    // entered with them in that order waits for every load on its first pass.
#pragma unroll
    for (int u = 0; u < U; ++u) {
      consume_slot(std::true_type{}, u, u);
      load_slot(u, u + U);
    }
    base = U;
  }
  // One-row single-matrix blocks pin each slot's refill right behind its products: left to itself
  // the compiler moves the batch's loads to its end and waits for the whole ring on every pass.
  // Measured (M = 1, split 1, graph-timed, two alternating runs on one box): QKV 9.37 -> 8.75 us,
  // O 8.35 -> 6.89, the BF16 lm_head 125.5 -> 122.6, down (split 4) and gate_up unchanged within
  // the runs' spread; pinning every slot of the two-matrix SwiGLU block and of the matrix-core
  // rings (M > 1) as well measured slower (gate_up 18.5 -> 19.8 us, M = 16 lm_head 139 -> 152).
  constexpr bool PIN = ALGO == 2 && P == 1;
  for (; base + U < jcount; base += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      consume_slot(std::false_type{}, u, base + u);
      load_slot(u, base + u + U);
      if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
    }
  }
  // (a last batch of U whole steps needs none of it: a scalar branch, and the shapes of the projections
  // pay nothing for the others)
  const int bs = __builtin_amdgcn_readfirstlane(base);
  if (ALGO != 2 && bs + U == jlast && (kts & 1) == 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) consume_slot(std::false_type{}, u, bs + u);
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) consume_slot(std::true_type{}, u, bs + u);
  }
  if (ALGO == 2) {
    // the four lanes of row r (g = 0..3) hold partial sums of disjoint k: add them; lanes 0..15
    // then carry columns 16 rb + lane in MFMA slot (mt 0, i 0), i.e. output row m = 0
#pragma unroll
    for (int p = 0; p < P; ++p) {
      float a = sv[p][0] + sv[p][1];
      a += __shfl_xor(a, 16, kWave);
      a += __shfl_xor(a, 32, kWave);
      acc[p][0] = v4f{g == 0 ? a : 0.f, 0.f, 0.f, 0.f};
    }
  }
  if (WAITS && chain_bad) {  // (the wait gave up: every partial of the block is NaN)
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[p][mt] = v4f{NAN, NAN, NAN, NAN};
  }
  // the P accumulator sets of each wave, in the layout epilogue() reads
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[(wave * P + p) * NV + mt * 256 + i * 64 + lane] = acc[p][mt][i];
  __syncthreads();
  if (MODE == KRQ_OUT_SWIGLU) {
    epilogue<MT, MODE, P, CHAIN>(red, 0, nw, M, NO, rb, sidx, ones, ColScales{1.0f, 1.0f}, out, aux,
                                 CHAIN ? nw * kWave : 0);
  } else {
#pragma unroll
    for (int p = 0; p < PB; ++p)
      epilogue<MT, MODE, P, CHAIN>(red, p, nw, M, NO, rb + p, sidx, ones, ColScales{1.0f, 1.0f}, out, aux,
                                   CHAIN ? nw * kWave : 0);
  }
  if constexpr (CHAIN) chain_tail<!WAITS>(*fa);
}

template <int MT, int MODE, int LAYOUT, int ALGO, int U, int PB, int XM>
__global__ __launch_bounds__(512) void k_gemv_bf16(const uint8_t* __restrict__ x,
                                                  const uint8_t* __restrict__ w, int M, int64_t NO,
                                                  int64_t K, int kts, void* __restrict__ out,
                                                  void* __restrict__ aux) {
  gemv_bf16_body<MT, MODE, LAYOUT, ALGO, U, PB, XM>(x, w, M, NO, K, kts, out, aux, blockIdx.x);
}

// Wide blocks at 4 < M <= 32: a workgroup of four waves owns four adjacent row blocks (one per wave, 64
// output columns; P = 2: of both halves of the SwiGLU) of one K split. A 16-column block brings as
// many activation bytes from L2 as weight bytes at M = 16 (twice as many at M = 32); here the split's
// activation rows go to LDS once for the four, by direct-to-LDS loads of whole lines, and each wave
// streams only its weights through a ring of U step slots. Steps, products and sums are those of the
// NS-wave launch it replaces: step j goes to accumulator set j % NS, the sets are added from zero in
// wave order, so the results are the same bit for bit.
// (The two sets on two waves, eight waves a workgroup with the sets added through LDS, measured
// slower: four layers row-major, M = 16 221.5 -> 226 us, M = 32 247.5 -> 254.8; packed M = 32 229 -> 242.)
// LDS: step j of row group h (rows 8 h .. 8 h + 7 of the HV in use) is 1 KiB at (j HV + h) KiB, entry
// 8 (c ^ (h % 2)) + row the row's 16-byte chunk c: a wave's operand read (rows 0-7 of one group, 8-15 of
// the next, one chunk) then covers 256 consecutive bytes modulo the banks.
constexpr int kWideRb = 4;

KRQ_DEV void wide_dma(const uint8_t* base, uint32_t voff, uint32_t l) {
  // (waited for by hand: issued before every other load, and vector memory loads complete in order)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(l), "v"(voff), "s"(base)
               : "memory", "m0");
}

template <int MODE, int LAYOUT, int MT, int U, int NS, int TL>
__global__ __launch_bounds__(kWideRb * 64) void k_gemv_bf16_wide(const uint8_t* __restrict__ x,
                                                                 const uint8_t* __restrict__ w, int M, int64_t NO,
                                                                 int64_t K, int kts, void* __restrict__ out) {
  constexpr int P = MODE == KRQ_OUT_SWIGLU ? 2 : 1;
  constexpr bool RM = LAYOUT == KRQ_W_ROWMAJOR;
  static_assert(U % NS == 0 && 2 * P * U < 64, "slot u feeds set u % NS; vmcnt range");
  __shared__ __align__(1024) uint8_t xt[TL * 1024];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  const int sidx = blockIdx.y;
  const int64_t rb = (int64_t)blockIdx.x * kWideRb + wave;
  const int nsteps = (kts + 1) >> 1, hv = (M + 7) >> 3;
  const int64_t tbase = (int64_t)sidx * kts, rowb = 2 * K;

  const uint32_t lx = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint8_t*)xt)));
  for (int i = wave; i < nsteps * hv; i += kWideRb) {
    const int j = i / hv, h = i - j * hv;
    int c = (lane >> 3) ^ (h & 1);
    if (2 * j + 1 >= kts) c &= 3;  // (a half last step: the high chunks repeat the low ones, masked below)
    wide_dma(x, static_cast<uint32_t>(min(8 * h + (lane & 7), M - 1) * rowb + (tbase + 2 * j) * 64 + 16 * c),
             lx + 1024u * static_cast<uint32_t>(i));
  }
  uint4 wl[P][U], wh[P][U];
  auto load_slot = [&](int u, int cc) {  // (a slot past the last step reloads it and is not consumed)
    const int j = min(cc, nsteps - 1);
    const int64_t t0 = tbase + 2 * j, t1 = (2 * j + 1 < kts) ? t0 + 1 : t0;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int64_t rr = p == 1 ? rb + (NO >> 4) : rb;
      if constexpr (RM) {
        const uint8_t* a = w + (16 * rr + (r & 7)) * rowb + t0 * 64 + 16 * w_line_chunk(lane, 2 * j + 1 >= kts);
        wl[p][u] = ld16nt(a);
        wh[p][u] = ld16nt(a + 8 * rowb);
      } else {
        wl[p][u] = ld16nt(w_addr<LAYOUT>(w, rr, t0, rowb, lane));
        wh[p][u] = ld16nt(w_addr<LAYOUT>(w, rr, t1, rowb, lane));
      }
    }
  };
#pragma unroll
  for (int u = 0; u < U; ++u) {
    load_slot(u, u);
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * P * U) : "memory");  // (the activation rows have landed)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");

  v4f acc[P][NS][MT];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int q = 0; q < NS; ++q)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[p][q][mt] = v4f{0.f, 0.f, 0.f, 0.f};
  auto consume = [&](auto last, int u, int j) {  // (last: as in gemv_bf16_body)
    const bool hi = 2 * j + 1 < kts;
    uint4 al[MT], ah[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {  // (rows past the groups in use read the last group)
      const int h = min(2 * mt + (r >> 3), hv - 1);
      const uint8_t* xr = xt + (j * hv + h) * 1024 + 16 * (r & 7);
      al[mt] = *reinterpret_cast<const uint4*>(xr + 128 * (g ^ (h & 1)));
      ah[mt] = *reinterpret_cast<const uint4*>(xr + 128 * ((g + 4) ^ (h & 1)));
      if constexpr (decltype(last)::value) ah[mt] = sel4(hi, ah[mt]);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      uint4 bl = wl[p][u], bh = wh[p][u];
      if constexpr (RM) lines_to_tiles(wl[p][u], wh[p][u], &bl, &bh);
      bh = sel4(hi, bh);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        v4f& c = acc[p][u % NS][mt];
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(al[mt]), as_v8bf(bl), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(ah[mt]), as_v8bf(bh), c, 0, 0, 0);
      }
    }
  };
  int base = 0;
  for (; base + U < nsteps; base += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      consume(std::false_type{}, u, base + u);
      load_slot(u, base + u + U);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (base + U == nsteps && (kts & 1) == 0) {  // (whole steps, as in gemv_bf16_body)
#pragma unroll
    for (int u = 0; u < U; ++u) consume(std::false_type{}, u, base + u);
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (base + u < nsteps) consume(std::true_type{}, u, base + u);
  }

  // element i of lane l: row 16 mt + 4 (l / 16) + i, column 16 rb + l % 16
  const int64_t n = rb * 16 + r;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float a[P];
#pragma unroll
      for (int p = 0; p < P; ++p) {
        a[p] = 0.0f;
#pragma unroll
        for (int q = 0; q < NS; ++q) a[p] += acc[p][q][mt][i];
      }
      const int m = mt * 16 + 4 * g + i;
      if (m >= M) continue;
      if constexpr (MODE == KRQ_OUT_PARTIAL) {
        reinterpret_cast<float*>(out)[((int64_t)sidx * M + m) * NO + n] = a[0];
      } else if constexpr (MODE == KRQ_OUT_BF16) {
        reinterpret_cast<uint16_t*>(out)[(int64_t)m * NO + n] = f32_to_bf16(a[0]);
      } else {
        const float gg = round_bf16(a[0]), uu = round_bf16(a[P - 1]);
        const float sl = round_bf16(gg / (1.0f + expf(-gg)));
        reinterpret_cast<uint16_t*>(out)[(int64_t)m * NO + n] = f32_to_bf16(sl * uu);
      }
    }
}

// The SwiGLU with its last column blocks split in half, as k_gemv_fp8_swiglu_mixed: workgroups
// below nfull are two-matrix blocks, workgroup nfull + j is half-pair block 2 nfull + j (the same
// steps per wave, so the same output bits).
template <int LAYOUT, int ALGO, int U, int XM>
__global__ __launch_bounds__(512) void k_gemv_bf16_swiglu_mixed(const uint8_t* __restrict__ x,
                                                               const uint8_t* __restrict__ w, int M, int64_t NO,
                                                               int64_t K, int kts, void* __restrict__ out,
                                                               void* __restrict__ aux, int nfull) {
  if (static_cast<int>(blockIdx.x) < nfull)
    gemv_bf16_body<1, KRQ_OUT_SWIGLU, LAYOUT, ALGO, U, 1, XM>(x, w, M, NO, K, kts, out, aux, blockIdx.x);
  else
    gemv_bf16_body<1, kOutSwiGluHalf, LAYOUT, ALGO, U, 1, XM>(x, w, M, NO, K, kts, out, aux,
                                                          (int64_t)blockIdx.x + nfull);
}

// The chained BF16 MLP (krq_mlp_chain_bf16): act = SwiGLU(x . Wgu^T) and the split-K partials of
// act . Wd^T in one launch. Workgroups below fa.n_first are the SwiGLU launch's blocks (two-matrix
// blocks below nfull, then half-pair blocks, as k_gemv_bf16_swiglu_mixed, when MT == 1), with
// NWG waves; the rest are the down launch's blocks with NWD waves, block p at row block p % nrb2
// of K split p / nrb2. Each stage keeps the standalone launch's plan, so act and the partials are
// those of the two launches, bit for bit. The block holds max(NWG, NWD) waves; the waves a stage
// does not use end at once (a barrier waits only for the waves that have not ended).
template <int MT, int LAYOUT, int ALGO, int U, int XM>
__global__ __launch_bounds__(512) void k_mlp_chain_bf16(const uint8_t* __restrict__ x, const uint8_t* __restrict__ wgu,
                                                       const uint8_t* __restrict__ wd, int M, int64_t I, int64_t H,
                                                       int kts_g, int kts_d, int nfull, int nrb2, int nwg, int nwd,
                                                       uint16_t* __restrict__ act, float* __restrict__ part,
                                                       FusedArgs fa) {
  const int w = static_cast<int>(blockIdx.x);
  if (w < nfull) {
    gemv_bf16_body<MT, KRQ_OUT_SWIGLU, LAYOUT, ALGO, U, 1, XM, true>(x, wgu, M, I, H, kts_g, act, nullptr, w, 0, nwg, &fa);
  } else if (w < fa.n_first) {
    if constexpr (MT == 1)
      gemv_bf16_body<1, kOutSwiGluHalf, LAYOUT, ALGO, U, 1, XM, true>(x, wgu, M, I, H, kts_g, act, nullptr,
                                                                  (int64_t)w + nfull, 0, nwg, &fa);
  } else {
    const int p = w - fa.n_first;
    gemv_bf16_body<MT, KRQ_OUT_PARTIAL, LAYOUT, ALGO, U, 1, XM, true>(reinterpret_cast<const uint8_t*>(act), wd, M, H, I,
                                                                  kts_d, part, nullptr, p % nrb2, p / nrb2, nwd, &fa);
  }
}

// Persistent row partition (the reference's gemv_rows, engine/kernels/gemv.py:270-348): exactly
// G = gridDim.x workgroups; workgroup p owns output rows [p N / G, (p + 1) N / G) over the full K
// and walks them in 16-row chunks, chunk c to wave c mod nw. A chunk streams its rows' whole K
// through a ring of U step slots on the BF16 matrix cores (row-major weights: a chunk may start
// on any row) and writes the rows it owns straight from its accumulators; lanes of rows past the
// workgroup's range reload its last row and store nothing. One wave sums each output row, in one
// order, so the result does not depend on G. P = 2 (SwiGLU): gate rows n, up rows N + n of the
// [2N, K] matrix, bf16(bf16(silu(bf16 g)) * bf16 u) as gemv.py:125-130.
template <int MT, int P, int U>
__global__ __launch_bounds__(512) void k_gemv_bf16_rows(const uint8_t* __restrict__ x,
                                                       const uint8_t* __restrict__ w, int M, int64_t N,
                                                       int64_t K, void* __restrict__ out) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int64_t G = gridDim.x, pid = blockIdx.x;
  const int64_t r0 = pid * N / G, r1 = (pid + 1) * N / G;
  const int64_t rowb = 2 * K;
  const int kts = static_cast<int>(K >> 5);  // 64-byte (32-element) tiles of a row
  const int nsteps = (kts + 1) >> 1;
  const int64_t nchunks = (r1 - r0 + 15) >> 4;
  const uint8_t* xr[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) xr[mt] = x + (int64_t)min(mt * 16 + r, M - 1) * rowb + g * 16;
  for (int64_t c = wave; c < nchunks; c += nw) {
    const int64_t n0 = r0 + 16 * c, nrow = min(n0 + r, r1 - 1);
    const uint8_t* wg = w + nrow * rowb + g * 16;
    const uint8_t* wu = w + (N + nrow) * rowb + g * 16;  // (P == 2)
    v4f acc[MT], accu[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc[mt] = v4f{0.f, 0.f, 0.f, 0.f};
      accu[mt] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    uint4 wl[U], wh[U], ul[U], uh[U], xl[U][MT], xh[U][MT];
    // every slot load is issued (a slot past the last step reloads it and is zeroed where consumed)
    auto load_slot = [&](int u, int cc) {
      const int j = min(cc, nsteps - 1);
      const int64_t t0 = 2 * j, t1 = (2 * j + 1 < kts) ? t0 + 1 : t0;
      wl[u] = ld16nt(wg + t0 * 64);
      wh[u] = ld16nt(wg + t1 * 64);
      if (P == 2) {
        ul[u] = ld16nt(wu + t0 * 64);
        uh[u] = ld16nt(wu + t1 * 64);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        xl[u][mt] = ld16(xr[mt] + t0 * 64);
        xh[u][mt] = ld16(xr[mt] + t1 * 64);
      }
    };
    auto consume_slot = [&](auto last, int u, int cc) {  // (last: as in gemv_bf16_body)
      const int j = min(cc, nsteps - 1);
      const bool ok = cc < nsteps, hi = ok && (2 * j + 1 < kts);
      const uint4 bl = sel4(ok, wl[u]), bh = sel4(hi, wh[u]);
      if constexpr (decltype(last)::value) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          xl[u][mt] = sel4(ok, xl[u][mt]);
          xh[u][mt] = sel4(hi, xh[u][mt]);
        }
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(xl[u][mt]), as_v8bf(bl), acc[mt], 0, 0, 0);
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(xh[u][mt]), as_v8bf(bh), acc[mt], 0, 0, 0);
      }
      if (P == 2) {
        const uint4 cl = sel4(ok, ul[u]), ch = sel4(hi, uh[u]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          accu[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(xl[u][mt]), as_v8bf(cl), accu[mt], 0, 0, 0);
          accu[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(xh[u][mt]), as_v8bf(ch), accu[mt], 0, 0, 0);
        }
      }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) load_slot(u, u);
    __builtin_amdgcn_sched_barrier(0);
    int base = 0;
    for (; base + U < nsteps; base += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        consume_slot(std::false_type{}, u, base + u);
        load_slot(u, base + u + U);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) consume_slot(std::true_type{}, u, base + u);
    // lane (g, r), element i of tile mt: output row m = 16 mt + 4 g + i, column n0 + r
    const int64_t n = n0 + r;
    if (n < r1) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = mt * 16 + 4 * g + i;
          if (m >= M) continue;
          uint16_t y;
          if (P == 2) {
            const float gg = round_bf16(acc[mt][i]), uu = round_bf16(accu[mt][i]);
            const float sl = round_bf16(gg / (1.0f + expf(-gg)));
            y = f32_to_bf16(sl * uu);
          } else {
            y = f32_to_bf16(acc[mt][i]);
          }
          reinterpret_cast<uint16_t*>(out)[(int64_t)m * N + n] = y;
        }
    }
  }
}

template <int MODE, int LAYOUT, bool LINES>
void launch(int M, int pb, dim3 grid, int nw, size_t smem, hipStream_t s, const uint8_t* x,
            const uint8_t* w, int m, int64_t NO, int64_t K, int kts, void* out, void* aux) {
  const dim3 block(nw * 64);
  constexpr int PB2 = MODE == KRQ_OUT_SWIGLU ? 1 : 2;
  constexpr int PB4 = MODE == kOutArgmax ? 4 : 1;  // (pb is 4 only for the argmax epilogue)
  constexpr bool RM = LAYOUT == KRQ_W_ROWMAJOR;
  constexpr int ONE = LINES ? kOneLine : kTileLoads, X = LINES ? kLineLoads : kTileLoads;
#define KRQ_BF16(MT_, ALGO_, U_, PB_, XM_)                                                                           \
  hipLaunchKernelGGL((k_gemv_bf16<MT_, MODE, LAYOUT, ALGO_, U_, PB_, XM_>), grid, block, smem, s, x, w, m, NO, K, kts, \
                     out, aux)
  if (M == 1) KRQ_BF16(1, 2, 4, 1, (RM ? ONE : kTileLoads));
  else if (M <= 4) KRQ_BF16(1, 1, 4, 1, ONE);
  else if (M <= 16 && pb == 4) KRQ_BF16(1, 1, 2, PB4, (RM ? X : kTileLoads));
  else if (M <= 16 && pb == 2) KRQ_BF16(1, 1, 2, PB2, X);
  else if (M <= 16) KRQ_BF16(1, 1, 2, 1, X);
  else if (pb == 2) KRQ_BF16(2, 1, 2, PB2, X);
  else KRQ_BF16(2, 1, 2, 1, X);
#undef KRQ_BF16
}

template <int MODE>
void launch_layout(int layout, bool lines, int M, int pb, dim3 grid, int nw, size_t smem, hipStream_t s, const uint8_t* x,
                   const uint8_t* w, int m, int64_t NO, int64_t K, int kts, void* out, void* aux) {
#define KRQ_BF16_LAYOUT(LAYOUT_)                                                                        \
  if (lines) launch<MODE, LAYOUT_, true>(M, pb, grid, nw, smem, s, x, w, m, NO, K, kts, out, aux);       \
  else launch<MODE, LAYOUT_, false>(M, pb, grid, nw, smem, s, x, w, m, NO, K, kts, out, aux)
  if (layout == KRQ_W_TILED) {
    KRQ_BF16_LAYOUT(KRQ_W_TILED);
  } else {
    KRQ_BF16_LAYOUT(KRQ_W_ROWMAJOR);
  }
#undef KRQ_BF16_LAYOUT
}

constexpr int64_t kCUs = 256;  // compute units of the MI355X (workgroup b runs on CU b mod 256)

// k_gemv_bf16_swiglu_mixed for M <= 16 when the SwiGLU's column blocks number a little over a
// multiple of the CUs (gate_up: 608 = 2 x 256 + 96), with the variant launch() would pick; false
// otherwise.
bool launch_swiglu_mixed(int layout, bool lines, int M, int64_t NO, int nw, size_t smem, hipStream_t s, const uint8_t* x,
                         const uint8_t* w, int64_t K, int kts, void* out) {
  const int64_t nrbs = NO / 16, rem = nrbs % kCUs;
  if (M > 16 || nrbs <= 2 * kCUs || rem == 0 || 2 * rem > kCUs) return false;
  const int nfull = static_cast<int>(nrbs - rem);
  const dim3 grid(static_cast<unsigned>(nfull + 2 * rem), 1), block(nw * 64);
#define KRQ_MIXED(LAYOUT_, ALGO_, U_, XM_)                                                                          \
  hipLaunchKernelGGL((k_gemv_bf16_swiglu_mixed<LAYOUT_, ALGO_, U_, XM_>), grid, block, smem, s, x, w, M, NO, K, kts, out, \
                     nullptr, nfull)
#define KRQ_MIXED_M(LAYOUT_, ONE_, ONE1_, X_)      \
  if (M == 1) KRQ_MIXED(LAYOUT_, 2, 4, ONE1_);     \
  else if (M <= 4) KRQ_MIXED(LAYOUT_, 1, 4, ONE_); \
  else KRQ_MIXED(LAYOUT_, 1, 2, X_)
  if (layout == KRQ_W_TILED) {
    if (lines) { KRQ_MIXED_M(KRQ_W_TILED, kOneLine, kTileLoads, kLineLoads); }
    else { KRQ_MIXED_M(KRQ_W_TILED, kTileLoads, kTileLoads, kTileLoads); }
  } else {
    if (lines) { KRQ_MIXED_M(KRQ_W_ROWMAJOR, kOneLine, kOneLine, kLineLoads); }
    else { KRQ_MIXED_M(KRQ_W_ROWMAJOR, kTileLoads, kTileLoads, kTileLoads); }
  }
#undef KRQ_MIXED_M
#undef KRQ_MIXED
  return true;
}

// Whether 16-column blocks (`blocks` of them, ks elements of K each) load whole lines. On row-major weights
// a line then goes through the caches once instead of twice, on packed ones the activations do, but
// the lanes' exchange lengthens every step of a block: it pays where the caches bound a unit's blocks,
// not where one or two blocks' own chain does. Measured, us, tile loads / lines:
//   row-major  QKV in two M = 1 10.7 / 8.3; 1,024 x 1,024 in four M = 1 3.33 / 3.53 (short chains); 5,120 x
//              5,120 M = 6 22.0 / 16.6, but 4,096 x 4,096, one block per unit, 9.84 / 11.0
//   SwiGLU     (two matrices a block) 8,192 x 8,192, 256 blocks, M = 6 33.4 / 36.9; gate_up M = 1 26.6 / 19.1;
//              5,120 x 5,120, 160 blocks, M = 1 23.3 / 22.6, M = 24 27.6 / 26.5, M = 32 30.6 / 26.9;
//              4,096 x 11,008, 128 blocks, M = 24 49.4 / 50.8, M = 32 55.1 / 51.8
//   packed     up to 9 rows no gain (4,096 x 4,096 M = 6 8.9 / 9.7); 5,120 x 5,120 M = 12 15.7 / 14.8, M = 16
//              18.2 / 16.6; one block per unit 4,096 x 4,096 M = 16 9.1 / 9.9, 4,096 x 11,008 M = 32 31.1 / 28.4;
//              SwiGLU 4,096 x 4,096 M = 16 15.1 / 16.7, gate_up M = 12 19.2 / 18.5, 28,672 x 4,096 M = 8 40.2 /
//              39.4, 11,008 x 4,096 (344 blocks) M = 24 25.2 / 24.4
bool line_loads(int layout, int M, int mode, int64_t blocks, int64_t ks) {
  const bool even = blocks == kCUs || blocks == 2 * kCUs;
  if (layout == KRQ_W_ROWMAJOR) {
    if (mode == KRQ_OUT_SWIGLU) return blocks >= (M > 24 ? 128 : M > 16 || M == 1 ? 160 : kCUs + 1);
    return (ks >= 1280 || blocks >= 2 * kCUs) && !(even && M > 4 && M <= 8);
  }
  if (mode == KRQ_OUT_SWIGLU) return M >= 8 && blocks > (M > 16 ? kCUs : 2 * kCUs);
  return M >= 10 && (M > 16 || !even);
}

// k_gemv_bf16_wide where it applies (false otherwise): launches of more than four rows whose replaced
// plan has two waves, whole groups of four row blocks on half the compute units or more, the split's
// activation rows within LDS. Four Qwen3-4B layers in one graph, us, 16-column blocks / wide, row-major
// weights: M = 3 194.1 / 195.5 and M = 4 199.1 / 197.6 (left narrow), M = 6 202 / 190, M = 16 246 / 221,
// M = 32 336 / 256; packed: M = 16 205 / 189, M = 32 291 / 229. Four slots: two measured 254 at M = 16
// row-major, six 228, eight 234. The two-matrix SwiGLU block (152 workgroups for gate_up) is wide above
// 16 rows only: at M = 16 23.8 us against 25.2 wide, at M = 32 34.0 against 21.
// Fewer rows bring fewer activation bytes to share, and a grid a little over the units leaves most of a
// second round empty. Packed up to 16 rows: not on half the units (4,096 x 4,096 in two M = 16 9.0 / 9.8, but
// 8,192 x 1,024 M = 24 8.02 / 6.86), splits of at most 48 steps (LDS for two workgroups a unit; 8,192 x
// 8,192 in two M = 6 22.7 / 25.9), and up to 12 within one round or on short splits (4,096 x 4,096 in four
// M = 6 7.8 / 9.0, QKV in four 8.55 / 7.72). Row-major up to eight rows: not on half the units (8,192 x 8,192 M = 6 31.0 / 35.8) nor a
// little over them (19,456 x 2,560, 304 workgroups, M = 6 22.4 / 25.0).
bool launch_wide(int layout, int M, int mode, int pb, int nw, int64_t NO, int split, hipStream_t s, const uint8_t* x,
                 const uint8_t* w, int64_t K, int kts, void* out) {
  const int64_t groups = NO / 16 / kWideRb, wgs = groups * split;
  const int steps = (kts + 1) / 2, kib = steps * ((M + 7) / 8);  // LDS for the split's activation rows
  if (M <= 4 || pb != 1 || nw != 2 || (NO / 16) % kWideRb != 0 || 2 * wgs < kCUs || kib > 160) return false;
  if (layout == KRQ_W_TILED) {
    if (M <= 16 && (wgs < 144 || steps > 48 || (M <= 12 && wgs > 240 && steps > 10))) return false;
  } else if (M <= 8 && (wgs < 144 || (wgs > kCUs && wgs < 344))) {
    return false;
  }
  if (M * 2 * K > 0x7fffffff) return false;  // (32-bit activation offsets)
  const dim3 grid(static_cast<unsigned>(groups), static_cast<unsigned>(split)), block(kWideRb * 64);
#define KRQ_WIDE(MODE_, LAYOUT_, MT_, TL_) \
  hipLaunchKernelGGL((k_gemv_bf16_wide<MODE_, LAYOUT_, MT_, 4, 2, TL_>), grid, block, 0, s, x, w, M, NO, K, kts, out)
#define KRQ_WIDE_TL(MODE_, LAYOUT_, MT_)                     \
  if (kib <= 40) { KRQ_WIDE(MODE_, LAYOUT_, MT_, 40); }      \
  else if (kib <= 80) { KRQ_WIDE(MODE_, LAYOUT_, MT_, 80); } \
  else { KRQ_WIDE(MODE_, LAYOUT_, MT_, 160); }
#define KRQ_WIDE_M(MODE_, LAYOUT_) \
  if (M <= 16) { KRQ_WIDE_TL(MODE_, LAYOUT_, 1) } else { KRQ_WIDE_TL(MODE_, LAYOUT_, 2) }
#define KRQ_WIDE_L(MODE_)                                                    \
  if (layout == KRQ_W_TILED) { KRQ_WIDE_M(MODE_, KRQ_W_TILED) } else { KRQ_WIDE_M(MODE_, KRQ_W_ROWMAJOR) }
  if (mode == KRQ_OUT_PARTIAL) {
    KRQ_WIDE_L(KRQ_OUT_PARTIAL)
  } else if (mode == KRQ_OUT_BF16) {
    KRQ_WIDE_L(KRQ_OUT_BF16)
  } else if (mode == KRQ_OUT_SWIGLU && M > 16) {
    if (layout == KRQ_W_TILED) { KRQ_WIDE_TL(KRQ_OUT_SWIGLU, KRQ_W_TILED, 2) }
    else { KRQ_WIDE_TL(KRQ_OUT_SWIGLU, KRQ_W_ROWMAJOR, 2) }
  } else {
    return false;
  }
#undef KRQ_WIDE_L
#undef KRQ_WIDE_M
#undef KRQ_WIDE_TL
#undef KRQ_WIDE
  return true;
}

}  // namespace

int krq::gemv_bf16_run(const void* x, const void* w, int w_layout, int64_t M, int64_t N, int64_t K,
                       int split, int mode, void* out, void* aux, void* stream) {
  KRQ_REQUIRE(x && w && (out || mode == kOutArgmax) && (aux || mode != kOutArgmax),
              "gemv_bf16: null pointer");
  KRQ_REQUIRE(aligned16(x) && aligned16(w), "gemv_bf16: x and w must be 16-byte aligned");
  KRQ_REQUIRE(M >= 1 && M <= 32, "gemv_bf16: M=%lld outside 1..32", (long long)M);
  KRQ_REQUIRE(N > 0 && K > 0 && split >= 1, "gemv_bf16: bad shape N=%lld K=%lld split=%d",
              (long long)N, (long long)K, split);
  KRQ_REQUIRE(K % split == 0 && (K / split) % 32 == 0,
              "gemv_bf16: no tiling divides K_SPLIT (K=%lld split=%d; K/split must be a multiple of 32)",
              (long long)K, split);
  KRQ_REQUIRE(mode >= KRQ_OUT_BF16 && mode <= kOutArgmax, "gemv_bf16: bad mode %d", mode);
  KRQ_REQUIRE(w_layout == KRQ_W_ROWMAJOR || w_layout == KRQ_W_TILED, "gemv_bf16: bad layout %d", w_layout);
  KRQ_REQUIRE(mode == KRQ_OUT_PARTIAL || split == 1, "gemv_bf16: split %d needs the partials output", split);
  const int64_t NO = mode == KRQ_OUT_SWIGLU ? N / 2 : N;
  KRQ_REQUIRE(NO % 16 == 0 && (mode != KRQ_OUT_SWIGLU || N % 2 == 0),
              "gemv_bf16: no tiling divides N=%lld (output columns must be a multiple of 16)", (long long)N);
  KRQ_REQUIRE(NO / 16 <= 0x7fffffff && split <= 65535, "gemv_bf16: grid too large");
  const int kts = static_cast<int>(K / split / 32);
  // paired only where halving the blocks still leaves thousands (the lm_head), as in gemv_fp8.hip;
  // the lm_head's argmax launch at 4 < M <= 16 takes four row blocks per block
  int pb = (mode != KRQ_OUT_SWIGLU && M > 4 && (NO / 16) % 2 == 0 &&
            (NO / 16) * split >= 4096) ? 2 : 1;
  if (pb == 2 && mode == kOutArgmax && M <= 16 && (NO / 16) % 4 == 0) pb = 4;
  const int P = mode == KRQ_OUT_SWIGLU ? 2 : pb;
  const int MT = M <= 16 ? 1 : 2;
  const int nw = plan_waves((kts + 1) / 2, P, M <= 4 ? 4 : 2, NO / 16 / pb * split);  // U of launch()'s variant
  const size_t smem = (size_t)nw * P * MT * 256 * sizeof(float);
  const dim3 grid(static_cast<unsigned>(NO / 16 / pb), static_cast<unsigned>(split));
  const uint8_t* xb = (const uint8_t*)x;
  const uint8_t* wb = (const uint8_t*)w;
  const int m = static_cast<int>(M);
  hipStream_t s = (hipStream_t)stream;
  const bool lines = line_loads(w_layout, m, mode, NO / 16 * split, K / split);
  if (launch_wide(w_layout, m, mode, pb, nw, NO, split, s, xb, wb, K, kts, out)) return krq_check_launch("gemv_bf16");
  if (mode == KRQ_OUT_BF16) launch_layout<KRQ_OUT_BF16>(w_layout, lines, m, pb, grid, nw, smem, s, xb, wb, m, NO, K, kts, out, aux);
  else if (mode == KRQ_OUT_PARTIAL) launch_layout<KRQ_OUT_PARTIAL>(w_layout, lines, m, pb, grid, nw, smem, s, xb, wb, m, NO, K, kts, out, aux);
  else if (mode == KRQ_OUT_SWIGLU && launch_swiglu_mixed(w_layout, lines, m, NO, nw, smem, s, xb, wb, K, kts, out))
    ;  // the mixed launch below 17 rows on grids a little over a multiple of the CUs
  else if (mode == KRQ_OUT_SWIGLU) launch_layout<KRQ_OUT_SWIGLU>(w_layout, lines, m, pb, grid, nw, smem, s, xb, wb, m, NO, K, kts, out, aux);
  else launch_layout<kOutArgmax>(w_layout, lines, m, pb, grid, nw, smem, s, xb, wb, m, NO, K, kts, out, aux);
  return krq_check_launch("gemv_bf16");
}

extern "C" int krq_gemv_bf16(const void* x, const void* w, int w_layout, int64_t M, int64_t N, int64_t K,
                             int split, int mode, void* out, void* stream) {
  KRQ_REQUIRE(mode >= KRQ_OUT_BF16 && mode <= KRQ_OUT_SWIGLU, "gemv_bf16: bad mode %d", mode);
  return gemv_bf16_run(x, w, w_layout, M, N, K, split, mode, out, nullptr, stream);
}

extern "C" int krq_gemv_bf16_rows(const void* x, const void* w, int64_t M, int64_t N, int64_t K, int programs,
                                  int swiglu, void* out, void* stream) {
  KRQ_REQUIRE(x && w && out, "gemv_rows: null pointer");
  KRQ_REQUIRE(aligned16(x) && aligned16(w), "gemv_rows: x and w must be 16-byte aligned");
  KRQ_REQUIRE(M >= 1 && M <= 32, "gemv_rows: M=%lld outside 1..32", (long long)M);
  KRQ_REQUIRE(N > 0 && K > 0 && K % 32 == 0,
              "gemv_rows: bad shape N=%lld K=%lld (K must be a positive multiple of 32)", (long long)N,
              (long long)K);
  KRQ_REQUIRE(programs >= 1, "gemv_rows: programs=%d must be at least 1", programs);
  KRQ_REQUIRE(N <= 0x3fffffffffffll / programs, "gemv_rows: N=%lld too large", (long long)N);
  // waves: the most 16-row chunks any workgroup owns (at most 8; more chunks loop)
  const int64_t maxrows = (N + programs - 1) / programs;
  const int nw = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(8, (maxrows + 15) / 16)));
  const dim3 grid(static_cast<unsigned>(programs)), block(nw * 64);
  const uint8_t* xb = (const uint8_t*)x;
  const uint8_t* wb = (const uint8_t*)w;
  const int m = static_cast<int>(M);
  hipStream_t s = (hipStream_t)stream;
  if (swiglu) {
    if (M <= 16)
      hipLaunchKernelGGL((k_gemv_bf16_rows<1, 2, 4>), grid, block, 0, s, xb, wb, m, N, K, out);
    else
      hipLaunchKernelGGL((k_gemv_bf16_rows<2, 2, 4>), grid, block, 0, s, xb, wb, m, N, K, out);
  } else {
    if (M <= 16)
      hipLaunchKernelGGL((k_gemv_bf16_rows<1, 1, 4>), grid, block, 0, s, xb, wb, m, N, K, out);
    else
      hipLaunchKernelGGL((k_gemv_bf16_rows<2, 1, 4>), grid, block, 0, s, xb, wb, m, N, K, out);
  }
  return krq_check_launch("gemv_rows");
}

// The chained BF16 MLP (k_mlp_chain_bf16): both stages of the decode MLP in one launch, each with
// the plan krq_gemv_bf16 gives it (the SwiGLU launch and the split-K partials launch).
extern "C" int krq_mlp_chain_bf16(const void* x, const void* w_gu, const void* w_down, int w_layout, int64_t M,
                                  int64_t H, int64_t I, int split, void* act, uint32_t* ctl, uint32_t max_polls,
                                  void* out, void* stream) {
  KRQ_REQUIRE(x && w_gu && w_down && act && ctl && out, "mlp_chain_bf16: null pointer");
  KRQ_REQUIRE(aligned16(x) && aligned16(w_gu) && aligned16(w_down) && aligned16(act),
              "mlp_chain_bf16: x, weights and act must be 16-byte aligned");
  KRQ_REQUIRE(w_layout == KRQ_W_ROWMAJOR || w_layout == KRQ_W_TILED, "mlp_chain_bf16: bad layout %d", w_layout);
  KRQ_REQUIRE(M >= 1 && M <= 32, "mlp_chain_bf16: M=%lld outside 1..32", (long long)M);
  KRQ_REQUIRE(H > 0 && I > 0 && H % 32 == 0 && I % 16 == 0 && split >= 1 && I % split == 0 &&
                  (I / split) % 32 == 0,
              "mlp_chain_bf16: shape H=%lld I=%lld split=%d (H and I/split multiples of 32, I of 16)",
              (long long)H, (long long)I, split);
  KRQ_REQUIRE(M * 2 * I <= 0x7fffffff && I / 16 <= 0x7fffffff && split <= 65535,
              "mlp_chain_bf16: shape too large");
  KRQ_REQUIRE(max_polls > 0, "mlp_chain_bf16: max_polls must be positive");
  const int64_t nrb2 = H / 16, n_second = nrb2 * split;
  // the down launch pairs row blocks on grids of thousands of blocks above 4 rows; the chained
  // kernel keeps one row block per block, so it takes only the unpaired plan
  KRQ_REQUIRE(!(M > 4 && nrb2 % 2 == 0 && n_second >= 4096),
              "mlp_chain_bf16: %lld down blocks at M=%lld (the chained form takes fewer than 4096 above 4 rows)",
              (long long)n_second, (long long)M);
  const int U = M <= 4 ? 4 : 2, MT = M <= 16 ? 1 : 2;  // (launch()'s variant)
  const int kts_g = static_cast<int>(H / 32), kts_d = static_cast<int>(I / split / 32);
  // gate_up: the SwiGLU launch's plan (two-matrix blocks, the last ones as half-pair blocks)
  const int64_t nrbs = I / 16, rem = nrbs % kCUs;
  const bool mixed = M <= 16 && nrbs > 2 * kCUs && rem != 0 && 2 * rem <= kCUs;
  const int64_t nfull = mixed ? nrbs - rem : nrbs, n_first = mixed ? nfull + 2 * rem : nrbs;
  KRQ_REQUIRE(n_first + n_second <= 0x7fffffff, "mlp_chain_bf16: grid too large");
  const int nwg = plan_waves((kts_g + 1) / 2, 2, U, nrbs), nwd = plan_waves((kts_d + 1) / 2, 1, U, n_second);
  const int nwb = std::max(nwg, nwd);
  const size_t smem = std::max((size_t)nwg * 2, (size_t)nwd) * MT * 256 * sizeof(float);
  FusedArgs fa{};
  fa.cnt = ctl;
  fa.max_polls = max_polls;
  fa.n_first = static_cast<int>(n_first);
  fa.n_second = static_cast<int>(n_second);
  const dim3 grid(static_cast<unsigned>(n_first + n_second)), block(nwb * 64);
  hipStream_t s = (hipStream_t)stream;
  const uint8_t* xb = (const uint8_t*)x;
  const uint8_t* gb = (const uint8_t*)w_gu;
  const uint8_t* db = (const uint8_t*)w_down;
  const int m = static_cast<int>(M);
#define KRQ_CHAIN(MT_, LAYOUT, ALGO, U_, XM_)                                                                        \
  hipLaunchKernelGGL((k_mlp_chain_bf16<MT_, LAYOUT, ALGO, U_, XM_>), grid, block, smem, s, xb, gb, db, m, I, H, kts_g, \
                     kts_d, static_cast<int>(nfull), static_cast<int>(nrb2), nwg, nwd, (uint16_t*)act, (float*)out, fa)
#define KRQ_CHAIN_M(LAYOUT)                                                                     \
  if (M == 1) KRQ_CHAIN(1, LAYOUT, 2, 4, (LAYOUT == KRQ_W_ROWMAJOR ? kOneLine : kTileLoads));   \
  else if (M <= 4) KRQ_CHAIN(1, LAYOUT, 1, 4, kOneLine);                                        \
  else if (M <= 16) KRQ_CHAIN(1, LAYOUT, 1, 2, kLineLoads);                                     \
  else KRQ_CHAIN(2, LAYOUT, 1, 2, kLineLoads);
  if (w_layout == KRQ_W_TILED) {
    KRQ_CHAIN_M(KRQ_W_TILED)
  } else {
    KRQ_CHAIN_M(KRQ_W_ROWMAJOR)
  }
#undef KRQ_CHAIN_M
#undef KRQ_CHAIN
  return krq_check_launch("mlp_chain_bf16");
}
