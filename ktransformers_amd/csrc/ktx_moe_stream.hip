// ktx_moe_stream.hip — prompt GEMM of AMXINT4 / AMXINT8 experts (its own translation unit, compiled beside ktx_moe.hip).
#include <hip/hip_runtime.h>
#include <type_traits>

#include "ktx_common.h"
#include "ktx_internal.h"
#include "ktx_moe_dec.inc"
#include "ktx_moe_stream.h"

// =====================================================================================================
// Grouped GEMM of AMXINT4 / AMXINT8 prompts on tiles of 64 rows.  What bounds it is the memory's way in while experts have few rows (256 of 7168 x 2048, gate|up
// of 31 rows each: 5.2 TB/s) and, with more, the power that MFMAs beside that stream draw: the clock falls to 1.65 GHz of 2.4 as the cycles go down.  So it does
// no work that no row needs and keeps both units fed:
//   * a tile multiplies the 16-row groups that hold rows, by an instantiation for each count (a quarter of a 64-row tile is absent at 64 rows an expert);
//   * each wavefront owns four 16-row weight strips (gate|up: two strips of both; down: four), so a fragment of activations feeds 4 MFMAs; weights stream
//     through a ring of registers, 4 k-steps deep.  That is 128 KB a CU, as much as its share of the L2 holds; 8 deep is slower (31 rows an expert: 1151 us against 1131);
//   * activations come by LDS-DMA into one of two buffers of 4 or 8 k-steps while the other is multiplied.  Before, 2048 columns were staged at once, and nothing
//     multiplied meanwhile: a fifth of the time of a 64-row tile.
// NW = 8: one workgroup a CU.  NW = 4: two, of half the strips and half the LDS each, so that one starts or ends beside the other's MFMAs, and a job is half as
// large; the activations cross from L2 twice as often.  The caller's rule says which, with figures.
// Whole forward, AMXINT4, us, staged at once with all groups multiplied -> here: 256 experts of 7168 x 2048, 2048 tokens 1594 -> 1553, 4096 2450 -> 2316; 64 of 6144 x 3072,
// 1000, top-6: 591 -> 568; 32 of them, 700, top-4: 358 -> 314 (moe_gemm_kernel before); 64 of 3072 x 3072, 2000, top-4: 466 -> 433.
// Integer arithmetic and epilogue are those of moe_gemm_kernel, so results are bit-identical.
// =====================================================================================================
template <int WBITS, int NW, bool GATE_UP>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void moe_gemm_stream_kernel(GemmParams p) {
  constexpr int NJ = 4;                              // (strip, matrix) units per wavefront
  constexpr int SPW = GATE_UP ? 2 : 4;               // strips per wavefront
  constexpr int TOK = STREAM_ROWS, MT = TOK / 16;
  constexpr int TILE_BYTES = (WBITS == 4) ? 1024 : 2048;
  constexpr int XB = TOK * 128 * NW;                 // a chunk's activations: 64 rows of NW k-steps, or 32 rows of 8
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];   // [2][XB]
  __shared__ float s_ad[TOK];

  Tile tile;
  int bx;
  if (!moe_pick_job(p.tiles, p.counters[0], (p.N / 16 + NW * SPW - 1) / (NW * SPW), tile, bx)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int strip0 = (bx * NW + wave) * SPW;
  const int nstrips = p.N / 16, NKS = p.K / 128, ncol = p.K / 16;

  // strips past N alias strip 0 and are not stored
  const uint8_t* wb[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int st = strip0 + (GATE_UP ? (j >> 1) : j);
    const uint8_t* base = (GATE_UP && (j & 1)) ? p.w1 : p.w0;
    wb[j] = base + (size_t)tile.expert * p.expert_stride + (size_t)(st < nstrips ? st : 0) * NKS * TILE_BYTES;
  }

  // B fragment of k-step s of a chunk, half hh, row group t: column s*8 + kc*2 + hh of row t*16 + i.  A row's 16-byte column c lies in slot c ^ (row & 15):
  // ds_read_b128 takes lanes {0-3,12-15,20-27} together, whose slots are distinct modulo 16 (rows {0-3,12-15} of one kc, {4-11} of the next), and a
  // write's 8 lanes keep to 8 slots of one 128-byte line.
  const int i = lane & 15, kc = lane >> 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

  auto run = [&](auto mtl) __attribute__((always_inline)) {
    constexpr int MTL = decltype(mtl)::value;
    constexpr int SC = NW == 8 || MTL <= MT / 2 ? 8 : 4, ROWB = SC * 128;             // k-steps of a chunk; its bytes per row
    constexpr int D = 16 / WBITS;                                          // k-steps of weights in flight
    int xo[2][2];
#pragma unroll
    for (int par = 0; par < 2; par++)
#pragma unroll
      for (int hh = 0; hh < 2; hh++) xo[par][hh] = i * ROWB + (((par * 8 + kc * 2 + hh) ^ i) << 4);
    WFrag<WBITS> ring[D][NJ];
    int wlane = lane;
    asm volatile("" : "+v"(wlane));   // (the instantiations' first loads are the same: merged, they would be held across each other's loops)
    auto load_w = [&](int d, int ks) __attribute__((always_inline)) {
      const int kn = ks < NKS ? ks : NKS - 1;
#pragma unroll
      for (int j = 0; j < NJ; j++) ring[d][j] = load_wfrag<WBITS>(wb[j] + (size_t)kn * TILE_BYTES, wlane);
    };
#pragma unroll
    for (int d = 0; d < D; d++) load_w(d, d);
    // A chunk's rows: requests of 1 KB, one row of 8 k-steps or two of 4, dealt over the wavefronts.  A row past the tile reads its first one (its outputs
    // are not stored).
    constexpr int RP = 8 / SC, NQ = MTL * 16 / (NW * RP);
    auto row_of = [&](int q) __attribute__((always_inline)) { return (q * NW + wave) * RP + (RP == 2 ? lane >> 5 : 0); };
    int src[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const int row = row_of(q), r = tile.row0 + (row < tile.nrows ? row : 0);
      src[q] = p.row_src ? p.row_src[r] : r;
    }
    if (tid < MTL * 16) {
      const int r = tile.row0 + (tid < tile.nrows ? tid : 0);
      s_ad[tid] = p.act_d[p.row_src ? p.row_src[r] : r];
    }
    auto stage = [&](int q, int chunk) __attribute__((always_inline)) {
      const int col = chunk * (ROWB / 16) + ((lane & (ROWB / 16 - 1)) ^ (row_of(q) & 15));
      int r = src[q];
      asm volatile("" : "+v"(r));   // (the compiler otherwise keeps every row's address in registers that the loop has not got)
      moe_dma(p.act_q + (size_t)r * p.K + min(col, ncol - 1) * 16, lds0 + (chunk & 1) * XB + (q * NW + wave) * 1024);
    };
#pragma unroll
    for (int q = 0; q < NQ; q++) stage(q, 0);

    v4i acc[NJ][MTL];
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int t = 0; t < MTL; t++) acc[j][t] = v4i{0, 0, 0, 0};
    v4i a[2][NJ], b[2][MTL];   // operands of a k-step's halves
    auto read_b = [&](auto sc, auto hc, int chunk) __attribute__((always_inline)) {
      constexpr int s = decltype(sc)::value, hh = decltype(hc)::value;
      const uint8_t* xb = smem + (chunk & 1) * XB + (s >> 1) * 256 + xo[s & 1][hh];
#pragma unroll
      for (int t = 0; t < MTL; t++) b[hh][t] = *reinterpret_cast<const v4i*>(xb + t * (16 * ROWB));
    };
    auto unpack = [&](int d, auto hc) __attribute__((always_inline)) {
      constexpr int hh = decltype(hc)::value;
#pragma unroll
      for (int j = 0; j < NJ; j++) a[hh][j] = unpack_whalf<WBITS, hh>(ring[d][j]);
    };
    auto mul = [&](auto hc) __attribute__((always_inline)) {
      constexpr int hh = decltype(hc)::value;
#pragma unroll
      for (int t = 0; t < MTL; t++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[j][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[hh][j], b[hh][t], acc[j][t], 0, 0, 0);
    };
    const std::integral_constant<int, 0> h0{};
    const std::integral_constant<int, 1> h1{};
    // A k-step in two halves.  Beside a half's MFMAs: the reads and the unpacking of the next half's operands; the step's weights are refilled D steps ahead as soon
    // as they are unpacked.  The fences keep the compiler from unpacking further ahead than there are registers.
    auto step = [&](auto sc, auto mc, int chunk) __attribute__((always_inline)) {
      constexpr int s = decltype(sc)::value, d = s % D, dn = (s + 1) % D;
      constexpr bool more = decltype(mc)::value;
      read_b(sc, h1, chunk);
      unpack(d, h1);
      mul(h0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (more && s < SC / 2)   // the next chunk's rows, in the first half of this one
#pragma unroll
        for (int q = s; q < NQ; q += SC / 2) stage(q, chunk + 1);
      if constexpr (more || D < SC) load_w(d, chunk * SC + s + D);
      if constexpr (s + 1 < SC) read_b(std::integral_constant<int, (s + 1) % SC>{}, h0, chunk);
      unpack(dn, h0);
      mul(h1);
      __builtin_amdgcn_sched_barrier(0);
    };
    unpack(0, h0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int chunk = 0;
    for (; (chunk + 1) * SC <= NKS; chunk++) {
      read_b(h0, h0, chunk);
      static_for<SC>([&](auto sc) __attribute__((always_inline)) { step(sc, std::true_type{}, chunk); });
      // the next chunk is in the LDS (what was requested after its rows: SC / 2 + 1 steps of weights), and no one reads this one any more
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SC / 2 + 1) * NJ * (WBITS / 4)) : "memory");
      __syncthreads();
    }
    if (chunk * SC < NKS) {
      read_b(h0, h0, chunk);
      static_for<SC>([&](auto sc) __attribute__((always_inline)) {
        if (chunk * SC + decltype(sc)::value < NKS) step(sc, std::false_type{}, chunk);
      });
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no request may outlive the workgroup's LDS

    // ---- epilogue: the arithmetic of moe_gemm_kernel's (GemmKernel224Int4::apply_scale, la/amx_kernels.hpp:1808-1846)
    const int ld = GATE_UP ? 2 * p.N : p.N;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      const int st = strip0 + (GATE_UP ? (j >> 1) : j);
      if (st >= nstrips) continue;
      const int n0 = st * 16 + kc * 4;
      const float* sp = (GATE_UP && (j & 1)) ? p.s1 : p.s0;
      const float4 sc = *reinterpret_cast<const float4*>(sp + (size_t)tile.expert * p.N + n0);
      const float sv[4] = {sc.x, sc.y, sc.z, sc.w};
      const int coff = (GATE_UP && (j & 1)) ? p.N : 0;
#pragma unroll
      for (int t = 0; t < MTL; t++) {
        const int row = t * 16 + i;
        if (row < tile.nrows) {
          const float ad = s_ad[row];
          bf16_t o[4];
#pragma unroll
          for (int r = 0; r < 4; r++) o[r] = f32_to_bf16((ad * sv[r]) * (float)acc[j][t][r]);
          *reinterpret_cast<uint2*>(p.out + (size_t)(tile.row0 + row) * ld + coff + n0) =
              make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
        }
      }
    }
  };
  switch ((tile.nrows + 15) >> 4) {
    case 1: run(std::integral_constant<int, 1>{}); break;
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;
    default: run(std::integral_constant<int, MT>{}); break;
  }
}

template <int WBITS, int NW, bool GATE_UP>
static int launch_gemm_stream(const GemmParams& p, int max_tiles, hipStream_t st) {
  constexpr int per_wg = NW * (GATE_UP ? 2 : 4), lds = 2 * STREAM_ROWS * 128 * NW;   // strips; bytes
  const hipError_t err = ktx_set_max_lds(reinterpret_cast<const void*>(moe_gemm_stream_kernel<WBITS, NW, GATE_UP>), lds);
  KTX_HIP(err);
  hipLaunchKernelGGL((moe_gemm_stream_kernel<WBITS, NW, GATE_UP>), moe_job_grid(max_tiles, (p.N / 16 + per_wg - 1) / per_wg), dim3(NW * 64), lds, st, p);
  KTX_HIP(hipGetLastError());
  return 0;
}

template <int WBITS, int NW>
static int launch_gemm_stream(bool gate_up, const GemmParams& p, int max_tiles, hipStream_t st) {
  return gate_up ? launch_gemm_stream<WBITS, NW, true>(p, max_tiles, st) : launch_gemm_stream<WBITS, NW, false>(p, max_tiles, st);
}

int moe_launch_gemm_stream(int wbits, int nw, bool gate_up, const GemmParams& p, int max_tiles, hipStream_t st) {
  if (wbits == 4) return nw == 4 ? launch_gemm_stream<4, 4>(gate_up, p, max_tiles, st) : launch_gemm_stream<4, 8>(gate_up, p, max_tiles, st);
  return nw == 4 ? launch_gemm_stream<8, 4>(gate_up, p, max_tiles, st) : launch_gemm_stream<8, 8>(gate_up, p, max_tiles, st);
}
