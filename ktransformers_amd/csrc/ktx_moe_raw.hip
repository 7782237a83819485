// ktx_moe_raw.hip — prompt GEMM of RAWINT4 experts (its own translation unit: it takes as long to compile as ktx_moe.hip).
#include <hip/hip_runtime.h>
#include <type_traits>

#include "ktx_common.h"
#include "ktx_moe_dec.inc"
#include "ktx_moe_raw.h"

// =====================================================================================================
// RAWINT4 prompt chunks: the same products on the 16x16x32 f16 MFMA, one MFMA per (32-k group) x (16 rows) x (16 tokens).
//
// The exact kernel (ktx_moe.hip) keeps the reference's SIXTEEN fp32 lane accumulators per output.  A prompt chunk does not need that
// association: the terms of an output are the per-group sums  as[t][g] * bs[n][g] * sum_{k in g} a[t][k] * q[n][k]  — the reference adds
// them as 16 interleaved chains + a tree, this kernel as ONE chain over the groups in k order, held to the bound of the FP8 / BF16 formats
// (tests/test_moe_gpu.py::test_rawint4_prompt_chunks).  Decode and short batches (qlen < 64) keep the exact kernels; dev knob 29 = 1
// forces them for every size.
//
// The vector ALU's and the matrix pipe's instructions bound it, which take turns more than they overlap (128 experts of 7168 x 2048 with 64 rows each: 60 and 40 % busy), so the
// operands are what costs them least: codes and nibbles as f16 integers, whose sum over a group the f16 MFMA gives exactly and in fp32 already (below 2^15), and scale
// products by the fp32 MFMA of four 16 x 16 outer products, so that the vector ALU is left with one fma an output and group (with an int8 MFMA, a conversion as well): the
// terms are the reference's, with any scale.
// (The weight's scale inside the f16 operand is exact for magnitudes of 2^-23 .. 4 and saves the scale products, but the terms are then rounded once where the
// reference's are twice, the sums reach only 2^119, and experts with another scale need a path of their own.)
//
// No second copy of the weights: the RAW tiles are read as they lie in HBM.  MFMA lane (i = lane & 15, kc = lane >> 4) needs
// row i's eight nibbles k = 64 kb + 32 h + 8 kc + [0, 8) of group (kb, h): those are the pieces (L, j) = (8h + 2kc + o, i & 3),
// o = 0 / 1, of RAW tile rg = i >> 2 — so the lane loads exactly its four pieces q = (h, o) of the strip's four tiles and nothing moves
// between lanes; inside 8 k the pairs come out as (0,2) (1,3) (4,6) (5,7), the order in which the activation codes are stored.
//   workgroup = 4 wavefronts = 4 strips of 16 weight rows x (gate, up), or 8 strips of down, x 64 rows of the expert, two workgroups per CU (one
//   multiplies while the other waits: 8 wavefronts on 128 rows are 2 to 20 % slower, though no expert of 65 .. 128 rows is widened twice).  K walks in the RAW
//   step of 512: its weights go through the LDS into registers (the LDS holds the next step's meanwhile: two steps in registers leave none for
//   the sums of two rounds), the activations in quarters of it, all by LDS-DMA.
// At Kimi-K2's sizes, us for the whole forward, scale products on the vector ALU, their activations' scales by a 4-byte gather a group, rows' addresses read from the LDS in
// front of each request -> here (the same bits): 64 tokens 986 -> 896, 200 1453 -> 1329, 500 1973 -> 1808, 2048 4177 -> 3770; 64 experts of 2048 x 1024, top-8: 130 tokens 113 ->
// 109, 360 163 -> 156, 2048 557 -> 512; 8 of 4096 x 1536, top-2: 64 tokens 76 -> 72, 300 111 -> 106, 1200 247 -> 219.  Of 2048 tokens' 400 us the scale products gave 160, with one
// group of k a set in every tile; that cost tiles of up to 16 rows 10 %, where sets of 4 groups save 6.  Nibbles left 1032 or 72 too large, which an MFMA of the activations with that constant
// takes off each group's sum (4 vector instructions in 20 saved a widened fragment): no change at 16 rows an expert, 1 % slower at 64.
// =====================================================================================================
// the pairs (byte 0, byte 2) and (byte 1, byte 3) of the low (par 0) or high nibbles of x as q; x: two's complement nibbles.
// A nibble (its top bit turned: q + 8) becomes mantissa bits 0..3 or 4..7 of an f16 of exponent 2^10 where it lies, or after a shift by a byte:
// 1024 + (q + 8), or 1024 + 16 (q + 8).
template <int PAR>
__device__ __forceinline__ void raw_widen(uint32_t x, const uint32_t (&mask)[2], const uint32_t (&top)[2], uint32_t& o0, uint32_t& o1) {
  auto value = [&](uint32_t e) {
    const raw_h2 v = __builtin_bit_cast(raw_h2, (e & mask[PAR]) ^ top[PAR]);
    if constexpr (PAR == 0) return raw_h2_bits(v + raw_h2{(_Float16)-1032.0f, (_Float16)-1032.0f});
    else return raw_h2_bits(__builtin_elementwise_fma(v, raw_h2{(_Float16)0.0625f, (_Float16)0.0625f}, raw_h2{(_Float16)-72.0f, (_Float16)-72.0f}));
  };
  o0 = value(x);
  o1 = value(x >> 8);
}

// A step's weights of a wavefront: w[u][h * 2 + o] the piece L = 8 h + 2 kc + o of unit u; s[u]: 8 bf16 scales (kb = 0 .. 7) of the row and h that the lane's
// scale products take (NH = 2: of both h).
template <int NU, int NH>
struct RawStep { uint4 w[NU][4]; uint4 s[NU][NH]; };

// 4 wavefronts of one strip (x gate, up; or two strips of down) each, up to RAW_ROWS rows of one expert.
template <bool GATE_UP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void moe_rawint4_chunk_kernel(RawGemmParams p) {
  constexpr int NW = 4, NU = 2;                     // weight operands per wavefront that share one activation fragment: (gate, up) of a
                                                    // strip, or two strips of down
  constexpr int TOK = NW * 16, MT = NW;
  // activations: codes (f16) in quarter steps (128 k), two buffers of up to TOK rows or four of up to TOK / 2; the scales of a step, two buffers of [rows][16 groups]
  constexpr int XBYTES = 2 * TOK * 256, AB = TOK * 64, ABYTES = 2 * AB;
  constexpr int WB = NU * 4096 + NU * 512;          // a wavefront's weights of a step: [u][q] pieces of 1 KB, [u][row][h] scales of 16 B
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];   // XBYTES | ABYTES | [NW][WB]
  __shared__ int s_src[TOK];

  const int tile_idx = blockIdx.y, sgroup = blockIdx.x;
  if (tile_idx >= p.counters[0]) return;
  const Tile tile = p.tiles[tile_idx];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nstrips = p.N / 16;
  const int NS = p.K / 512, G = p.K / 32;
  const int i = lane & 15, kc = lane >> 4, rg = i >> 2, j = i & 3;
  int ustrip[NU];
#pragma unroll
  for (int u = 0; u < NU; u++) ustrip[u] = GATE_UP ? sgroup * NW + wave : (sgroup * NW + wave) * 2 + u;
  const bool wave_ok = ustrip[0] < nstrips;

  // rows past the tile read its first row again (their outputs are never stored)
  if (tid < TOK) {
    const int r = tile.row0 + (tid < tile.nrows ? tid : 0);
    s_src[tid] = p.row_src ? p.row_src[r] : r;
  }
  __syncthreads();
  const int mt_live = (tile.nrows + 15) >> 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

  // ---- weights: this lane's four pieces of each unit's four RAW tiles, and a row's scales (a strip past N aliases strip 0, not stored)
  const uint8_t* wb[NU];
  const uint8_t* sb;            // lanes 0..31 bring unit 0's scales, 32..63 unit 1's: row (lane >> 1) & 15, h = lane & 1
  const uint32_t wo = (uint32_t)(rg * NS * 1024 + ((2 * kc) * 4 + j) * 16);
  {
    const uint8_t* sbu[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int st = ustrip[u] < nstrips ? ustrip[u] : 0;
      wb[u] = ((GATE_UP && u) ? p.w1 : p.w0) + (size_t)tile.expert * p.expert_stride + (size_t)(st * 4) * NS * 1024;
      sbu[u] = reinterpret_cast<const uint8_t*>(((GATE_UP && u) ? p.s1 : p.s0) + (size_t)tile.expert * p.scale_stride + (size_t)(st * 4) * NS * 64);
    }
    const int row = (lane >> 1) & 15;
    sb = (lane < 32 ? sbu[0] : sbu[1]) + (size_t)((row >> 2) * NS * 128 + (row & 3) * 32 + (lane & 1) * 16);
  }
  // the activations' scales of a step: a row's 16 groups lie together, 4 lanes bring them, group quad q of row r to place q ^ (r >> 2 & 3) (16 rows' reads of one quad:
  // 16 places of a bank row)
  const uint8_t* ga = reinterpret_cast<const uint8_t*>(p.act_d + (size_t)s_src[wave * 16 + (lane >> 2)] * G) + ((lane ^ (lane >> 4)) & 3) * 16;
  const uint32_t lds_w = lds0 + XBYTES + ABYTES + wave * WB;
  const uint8_t* my_w = smem + XBYTES + ABYTES + wave * WB;
  constexpr int WDMA = NU * 4 + 2;
  auto stage_w = [&](int st, int par) __attribute__((always_inline)) {   // par: the scales' buffer
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        moe_dma(wb[u] + (size_t)st * 1024 + wo + ((q >> 1) * 8 + (q & 1)) * 64, lds_w + (u * 4 + q) * 1024);
    moe_dma(sb + (size_t)st * 128, lds_w + NU * 4096);
    moe_dma(ga + (size_t)st * 64, lds0 + XBYTES + par * AB + wave * 1024);
  };
  const uint32_t xo0 = i * 256 + ((kc ^ i) * 16);   // row i's piece kc; piece 4 g + kc: ^ 64 g
  // constants the compiler cannot see through: and + xor become one v_bitop3_b32
  uint32_t mask[2], top[2];
  asm("s_mov_b32 %0, 0x000F000F" : "=s"(mask[0]));
  asm("s_mov_b32 %0, 0x00F000F0" : "=s"(mask[1]));
  asm("v_mov_b32 %0, 0x64086408" : "=v"(top[0]));   // 1024 = 0x6400, and the nibble's top bit turned
  asm("v_mov_b32 %0, 0x64806480" : "=v"(top[1]));

  // MTL = 16-row groups of the tile that hold rows; one instantiation per count, chosen once per workgroup.
  auto run = [&](auto mtl) __attribute__((always_inline)) {
    constexpr int MTL = decltype(mtl)::value;
    constexpr int TB = MTL < 2 ? MTL : 2, NP = (MTL + TB - 1) / TB;   // fragments whose sums are in registers at once; rounds of them
    float acc[NU][MTL][4];
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
      for (int t = 0; t < MTL; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[u][t][r] = 0.0f;

    // A quarter step: four groups (kb = 2 Q, 2 Q + 1; h) in rounds of TB fragments.  A round's MFMAs are issued before the sums of the round before it, with
    // the operands' loads and the next group's widening between, so that a wavefront by itself keeps both units busy.  Rounds are fenced from each
    // other: left alone, the compiler widens a whole step's weights up front and spills them.
    constexpr int R = 4 * NP, NBUF = MTL * 2 > MT ? 2 : 4, XB = XBYTES / NBUF;
    // Scale products by the 4-block fp32 MFMA (16x16x1: an outer product a block, each product rounded once, as the vector ALU's): its four blocks are the tile's
    // row groups, and where there are one or two of them four or two groups of k as well.  Block kc: rows 16 (kc % SB) + i, group GS set + kc / SB.
    constexpr int SB = MTL > 2 ? 4 : MTL, GS = 4 / SB, NH = SB == 4 ? 2 : 1;
    using WStep = RawStep<NU, NH>;
    auto fetch_w = [&](WStep& d) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < NU; u++) {
#pragma unroll
        for (int q = 0; q < 4; q++) d.w[u][q] = *reinterpret_cast<const uint4*>(my_w + (u * 4 + q) * 1024 + lane * 16);
#pragma unroll
        for (int h = 0; h < NH; h++) d.s[u][h] = *reinterpret_cast<const uint4*>(my_w + NU * 4096 + u * 512 + i * 32 + (SB == 4 ? h : SB == 2 ? kc >> 1 : kc & 1) * 16);
      }
      // read before the next step's DMAs may overwrite them
#pragma unroll
      for (int u = 0; u < NU; u++) {
#pragma unroll
        for (int q = 0; q < 4; q++) asm volatile("" : "+v"(d.w[u][q].x), "+v"(d.w[u][q].y), "+v"(d.w[u][q].z), "+v"(d.w[u][q].w)::"memory");
#pragma unroll
        for (int h = 0; h < NH; h++) asm volatile("" : "+v"(d.s[u][h].x), "+v"(d.s[u][h].y), "+v"(d.s[u][h].z), "+v"(d.s[u][h].w)::"memory");
      }
    };
    raw_h8 bop[2][NU];
    auto scale = [&](const WStep& w, auto qc, auto sc, int u) __attribute__((always_inline)) {
      constexpr int Q = decltype(qc)::value, set = decltype(sc)::value;
      const uint4& sv = w.s[u][SB == 4 ? set & 1 : 0];
      const uint32_t S = Q == 0 ? sv.x : Q == 1 ? sv.y : Q == 2 ? sv.z : sv.w;
      if constexpr (SB == 1) return __uint_as_float(kc >> 1 ? S & 0xffff0000u : S << 16);
      else return __uint_as_float((SB == 4 ? set >> 1 : set) ? S & 0xffff0000u : S << 16);
    };
    auto widen = [&](const WStep& w, auto qc, auto gc) __attribute__((always_inline)) {
      constexpr int Q = decltype(qc)::value, g = decltype(gc)::value, par = g >> 1, h = g & 1;
#pragma unroll
      for (int u = 0; u < NU; u++) {
        const uint4 &w0 = w.w[u][h * 2], &w1 = w.w[u][h * 2 + 1];
        const uint32_t P0 = Q == 0 ? w0.x : Q == 1 ? w0.y : Q == 2 ? w0.z : w0.w;
        const uint32_t P1 = Q == 0 ? w1.x : Q == 1 ? w1.y : Q == 2 ? w1.z : w1.w;
        uint32_t o[4];
        raw_widen<par>(P0, mask, top, o[0], o[1]);
        raw_widen<par>(P1, mask, top, o[2], o[3]);
        bop[g & 1][u] = __builtin_bit_cast(raw_h8, make_uint4(o[0], o[1], o[2], o[3]));
      }
    };
    auto compute = [&](auto qc, int st, const WStep& w) __attribute__((always_inline)) {
      constexpr int Q = decltype(qc)::value, buf = Q % NBUF;
      const uint8_t* xb = smem + buf * XB;
      float as[SB];   // set: of the lane's row and group
      {
        const uint8_t* sp = smem + XBYTES + (st & 1) * AB + ((Q ^ (i >> 2)) & 3) * 16;   // (r >> 2 & 3 = i >> 2)
        if constexpr (SB == 4) {
          const float4 v = *reinterpret_cast<const float4*>(sp + lane * 64);
          as[0] = v.x; as[1] = v.y; as[2] = v.z; as[3] = v.w;
        } else {
#pragma unroll
          for (int set = 0; set < SB; set++) as[set] = *reinterpret_cast<const float*>(sp + ((kc % SB) * 16 + i) * 64 + (GS * set + kc / SB) * 4);
        }
      }
      raw_h8 af[2][TB];
      v16f S[NU];
      v4f d[2][TB][NU];
      auto load_a = [&](int r) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TB; t++)
          if ((r % NP) * TB + t < MTL) af[r & 1][t] = *reinterpret_cast<const raw_h8*>(xb + (xo0 ^ ((r / NP) * 64)) + ((r % NP) * TB + t) * 4096);
      };
      auto scales = [&](auto sc) __attribute__((always_inline)) {
        constexpr int set = decltype(sc)::value;
#pragma unroll
        for (int u = 0; u < NU; u++) S[u] = __builtin_amdgcn_mfma_f32_16x16x1f32(as[set], scale(w, qc, sc, u), v16f{}, 0, 0, 0);
      };
      auto mul = [&](int r) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TB; t++)
          if ((r % NP) * TB + t < MTL)
#pragma unroll
            for (int u = 0; u < NU; u++) d[r & 1][t][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[r & 1][t], bop[(r / NP) & 1][u], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      };
      load_a(0);
      if constexpr (Q == 0) widen(w, qc, std::integral_constant<int, 0>{});
      if constexpr (NP == 1) widen(w, qc, std::integral_constant<int, 1>{});
      scales(std::integral_constant<int, 0>{});
      mul(0);
      load_a(1);
      __builtin_amdgcn_sched_barrier(0);
      static_for<R>([&](auto rc) __attribute__((always_inline)) {
        constexpr int r = decltype(rc)::value;
        constexpr bool next = r + 1 < R && (r + 1) % (NP * GS) == 0;   // the first round of a set of groups
        if constexpr (r + 1 < R) mul(r + 1);
        if constexpr (r + 2 < R) load_a(r + 2);
        // the group of round r + 2 if that is its first (its operands' buffer was last read by the MFMAs two groups before it)
        if constexpr (r + 2 < R && (r + 2) % NP == 0) widen(w, qc, std::integral_constant<int, ((r + 2) / NP) & 3>{});
        if constexpr (r + 1 == R && Q < 3) widen(w, std::integral_constant<int, (Q + 1) & 3>{}, std::integral_constant<int, 0>{});
#pragma unroll
        for (int t = 0; t < TB; t++) {
          if ((r % NP) * TB + t >= MTL) continue;
#pragma unroll
          for (int u = 0; u < NU; u++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
              float& o = acc[u][(r % NP) * TB + t][e];
              o = fmaf(S[u][((r / NP % GS) * SB + (r % NP) * TB + t) * 4 + e], d[r & 1][t][u][e], o);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (next) scales(std::integral_constant<int, ((r + 1) / (NP * GS)) & 3>{});
      });
    };

    // activations of a quarter step: one DMA instruction per four rows of 256 B (LDS slot s of row r holds the row's 16-byte piece s ^ (r & 15)), dealt
    // over the wavefronts.  The rows' addresses stay in registers: read from s_src in front of each request, an LDS round trip per instruction.
    const int8_t* ax[MTL];
#pragma unroll
    for (int c = 0; c < MTL; c++) {
      const int row = (c * NW + wave) * 4 + (lane >> 4);
      ax[c] = p.act_q + (size_t)s_src[row] * (size_t)(p.K * 2) + ((lane ^ row) & 15) * 16;
    }
    auto stage = [&](int qs, int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < MTL; c++) moe_dma(ax[c] + (size_t)qs * 256, lds0 + buf * XB + (c * NW + wave) * 1024);
    };

    // A step of 512 k: its weights come from the LDS into registers, then the next step's are requested; a quarter's activations are requested NBUF - 1 quarters
    // ahead.  The waits leave what was requested after the quarter needed next: SD requests a quarter, WDMA of weights in the first one.  Requests
    // past the end repeat the last ones.  (Wavefronts of their own for the weights' and the activations' requests, so that neither waits for the
    // other's: 4 % slower, the four are no longer even.)
    constexpr int SD = MTL;
    auto quarter = [&](auto qc, int st, const WStep& w) __attribute__((always_inline)) {
      constexpr int Q = decltype(qc)::value;
      stage(min(4 * st + Q + NBUF - 1, 4 * NS - 1), (Q + NBUF - 1) % NBUF);
      if constexpr (Q == 0) stage_w(min(st + 1, NS - 1), (st + 1) & 1);
      if (wave_ok) compute(qc, st, w);
      // needed next: quarter Q + 1's activations, requested NBUF - 2 quarters ago (before that quarter's weights, if it was the first); at the end of the
      // step the weights as well
      constexpr int younger = (NBUF - 2) * SD, left = Q == 3 ? (younger < 2 * SD ? younger : 2 * SD) : Q <= NBUF - 2 ? younger + WDMA : younger;
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(left) : "memory");
      __syncthreads();
    };
    stage_w(0, 0);
#pragma unroll
    for (int q = 0; q < NBUF - 1; q++) stage(q, q);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 2) * SD) : "memory");
    __syncthreads();
    for (int st = 0; st < NS; st++) {
      WStep w;
      fetch_w(w);
      quarter(std::integral_constant<int, 0>{}, st, w);
      quarter(std::integral_constant<int, 1>{}, st, w);
      quarter(std::integral_constant<int, 2>{}, st, w);
      quarter(std::integral_constant<int, 3>{}, st, w);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no request may outlive the workgroup's LDS

    if (!wave_ok) return;
    if constexpr (GATE_UP) {
      const int n = ustrip[0] * 16 + i;
#pragma unroll
      for (int t = 0; t < MTL; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int row = t * 16 + kc * 4 + r;
          if (row < tile.nrows) {
            const bf16_t gv = f32_to_bf16(acc[0][t][r]), uv = f32_to_bf16(acc[1][t][r]);
            p.out[(size_t)(tile.row0 + row) * p.N + n] = f32_to_bf16(act_fn(bf16_to_f32(gv), bf16_to_f32(uv)));
          }
        }
    } else {
#pragma unroll
      for (int u = 0; u < NU; u++) {
        if (ustrip[u] >= nstrips) continue;
        const int n = ustrip[u] * 16 + i;
#pragma unroll
        for (int t = 0; t < MTL; t++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const int row = t * 16 + kc * 4 + r;
            if (row < tile.nrows) p.out[(size_t)(tile.row0 + row) * p.N + n] = f32_to_bf16(acc[u][t][r]);
          }
      }
    }
  };
#define KTX_RAW_CASE(m) case m: run(std::integral_constant<int, m>{}); break;
  switch (mt_live) {
    KTX_RAW_CASE(1) KTX_RAW_CASE(2) KTX_RAW_CASE(3) KTX_RAW_CASE(4)
  }
#undef KTX_RAW_CASE
}

template <bool GATE_UP>
static int launch_rawint4_chunk(const RawGemmParams& p, int max_tiles, hipStream_t st) {
  constexpr size_t lds = 4 * (2 * 16 * 256 + 2 * 16 * 64 + 2 * 4608);
  const hipError_t err = ktx_set_max_lds(reinterpret_cast<const void*>(moe_rawint4_chunk_kernel<GATE_UP>), (int)lds);
  KTX_HIP(err);
  const int per_wg = GATE_UP ? 4 : 8;       // strips per workgroup (down: two strips per wavefront)
  hipLaunchKernelGGL((moe_rawint4_chunk_kernel<GATE_UP>), dim3((p.N / 16 + per_wg - 1) / per_wg, max_tiles), dim3(256), lds, st, p);
  KTX_HIP(hipGetLastError());
  return 0;
}

int moe_launch_rawint4_chunk(bool gate_up, const RawGemmParams& p, int max_tiles, hipStream_t st) {
  return gate_up ? launch_rawint4_chunk<true>(p, max_tiles, st) : launch_rawint4_chunk<false>(p, max_tiles, st);
}
