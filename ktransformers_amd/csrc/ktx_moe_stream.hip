// ktx_moe_stream.hip — streaming prompt GEMMs of AMXINT4 / AMXINT8 and of FP8 experts (a translation unit of its own, compiled beside ktx_moe.hip).
#include <hip/hip_runtime.h>
#include <type_traits>

#include "ktx_common.h"
#include "ktx_internal.h"
#include "ktx_moe_dec.inc"
#include "ktx_moe_stream.h"

// =====================================================================================================
// Grouped GEMM of AMXINT4 / AMXINT8 prompts on tiles of 64 rows.  What bounds it is the memory's way in while experts have few rows (256 of 7168 x 2048, gate|up
// of 31 rows each: 5.2 TB/s) and, with more, the power that MFMAs beside that stream draw: the clock falls as the cycles go down (64 rows each: 1.73 M cycles at 1.87 GHz, with 4
// wavefronts 1.54 M at 1.65).  So it does no work that no row needs and keeps both units fed:
//   * a tile multiplies the 16-row groups that hold rows, by an instantiation for each count (a quarter of a 64-row tile is absent at 64 rows an expert);
//   * each wavefront owns four 16-row weight strips (gate|up: two strips of both; down: four), so a fragment of activations feeds 4 MFMAs; weights stream
//     through a ring of registers, 4 k-steps deep (AMXINT8: 2).  That is 128 KB a CU, as much as its share of the L2 holds; AMXINT4 8 deep is slower (31 rows an expert: 1151 us against
//     1131; at 94 rows, 64 of 6144 x 3072, it was 1 % faster, 570 against 576);
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

// =====================================================================================================
// The same for FP8 experts, on tiles of 32 rows, 4 wavefronts, two workgroups a CU; bf16 activations, 4 k-steps a buffer; weights 2 k-steps ahead, widened to bf16 a
// quarter k-step before their MFMAs.  Gate|up of 256 experts of 7168 x 2048, 1000 tokens: 177 M vector instructions beside 36 M MFMAs (234 M beside 45 M in
// moe_gemm_fp_kernel, which waits for a chunk's weights at the end of the chunk before it).  4 k-steps ahead, 256 KB a CU, are more than the L2 holds: 1000 tokens 2216 us against 2185.  8 wavefronts, one workgroup a CU: 2223.  Arithmetic, summation order and epilogue are moe_gemm_fp_kernel's: results are bit-identical.
// Whole forward, us, moe_gemm_fp_kernel -> here: 256 experts of 7168 x 2048, top-8: 1000 tokens 2298 -> 2185, 2048 3338 -> 3012, 8192 8697 -> 8131; 64 of 2048 x 1408, top-6, 800: 225
// -> 197; 64 of 6144 x 3072, top-6, 1000: 1243 -> 1175.  At fewer rows than the caller's rule asks for, more wavefronts of few registers stream better.
// =====================================================================================================
template <bool GATE_UP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void moe_fp8_stream_kernel(FpGemmParams p) {
  constexpr int NW = 4, NJ = 4, SPW = GATE_UP ? 2 : 4, SC = 4, D = 2;
  constexpr int ROWB = SC * 256, XB = FP_STREAM_ROWS * ROWB, TILE_BYTES = 2048;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];   // [2][XB] | scales [NW][2][NKS]

  Tile tile;
  int bx;
  if (!moe_pick_job(p.tiles, p.counters[0], (p.N / 16 + NW * SPW - 1) / (NW * SPW), tile, bx)) return;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, kc = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int strip0 = (bx * NW + wave) * SPW, nstrips = p.N / 16, NKS = p.K / 128;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

  const uint8_t* wb[NJ];   // strips past N alias strip 0 and are not stored
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int st = strip0 + (GATE_UP ? (j >> 1) : j);
    wb[j] = ((GATE_UP && (j & 1)) ? p.w1 : p.w0) + (size_t)tile.expert * p.expert_stride + (size_t)(st < nstrips ? st : 0) * NKS * TILE_BYTES;
  }
  float* s_sc = reinterpret_cast<float*>(smem + 2 * XB) + wave * 2 * NKS;   // a wavefront's strips lie in one block of 128 rows

  auto run = [&](auto mtl) __attribute__((always_inline)) {
    constexpr int MTL = decltype(mtl)::value;
    uint4 ring[D][NJ][2];
    int wlane = lane;
    asm volatile("" : "+v"(wlane));   // (the instantiations' first loads are the same: merged, they would be held across each other's loops)
    auto load_w = [&](int d, int ks) __attribute__((always_inline)) {
      const int kn = ks < NKS ? ks : NKS - 1;
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int q = 0; q < 2; q++) ring[d][j][q] = *reinterpret_cast<const uint4*>(wb[j] + (size_t)kn * TILE_BYTES + q * 1024 + wlane * 16);
    };
#pragma unroll
    for (int d = 0; d < D; d++) load_w(d, d);
    // A chunk's rows, one a request, dealt over the wavefronts.  A row past the tile reads its first one (not stored).
    constexpr int NQ = MTL * 16 / NW;
    int src[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const int row = q * NW + wave, r = tile.row0 + (row < tile.nrows ? row : 0);
      src[q] = __builtin_amdgcn_readfirstlane(p.row_src ? p.row_src[r] : r);
    }
    auto stage = [&](int q, int chunk) __attribute__((always_inline)) {
      const int row = q * NW + wave;
      int l = wlane;
      asm volatile("" : "+v"(l));   // (the compiler otherwise keeps every request's offset in registers that the loop has not got)
      const int piece = chunk * (ROWB / 16) + (l ^ fp_swz(row & 15));
      moe_dma(p.act + (size_t)src[q] * p.K + min(piece, p.K / 8 - 1) * 8, lds0 + (chunk & 1) * XB + row * ROWB);
    };
#pragma unroll
    for (int q = 0; q < NQ; q++) stage(q, 0);
    for (int ks = lane; ks < NKS; ks += 64)
#pragma unroll
      for (int m = 0; m < (GATE_UP ? 2 : 1); m++) {
        const int st = strip0 < nstrips ? strip0 : 0;
        s_sc[m * NKS + ks] = (m ? p.s1 : p.s0)[(size_t)tile.expert * p.scale_stride + (size_t)(st / 8) * NKS + ks];
      }

    int xo[4];
#pragma unroll
    for (int j = 0; j < 4; j++) xo[j] = i * ROWB + (((kc * 4 + j) ^ fp_swz(i)) << 4);
    v4f acc[NJ][MTL], tmp[NJ][MTL];
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int t = 0; t < MTL; t++) acc[j][t] = v4f{0.f, 0.f, 0.f, 0.f};
    v8bf a[2][NJ], b[2][MTL];   // operands of two quarters
    auto read_b = [&](auto sc, auto qc, int chunk) __attribute__((always_inline)) {
      constexpr int s = decltype(sc)::value, q = decltype(qc)::value;
      const uint8_t* xb = smem + (chunk & 1) * XB + s * 256 + xo[q];
#pragma unroll
      for (int t = 0; t < MTL; t++) b[q & 1][t] = u4_as_v8bf(*reinterpret_cast<const uint4*>(xb + t * (16 * ROWB)));
    };
    auto widen = [&](int d, auto qc) __attribute__((always_inline)) {
      constexpr int q = decltype(qc)::value;
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const uint4& w = ring[d][j][q >> 1];
        const uint2 e0 = fp8x4_to_bf16x4(q & 1 ? w.z : w.x), e1 = fp8x4_to_bf16x4(q & 1 ? w.w : w.y);
        a[q & 1][j] = u4_as_v8bf(make_uint4(e0.x, e0.y, e1.x, e1.y));
      }
    };
    auto mul = [&](auto qc) __attribute__((always_inline)) {
      constexpr int q = decltype(qc)::value;
#pragma unroll
      for (int t = 0; t < MTL; t++)
#pragma unroll
        for (int j = 0; j < NJ; j++) tmp[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q & 1][j], b[q & 1][t], q ? tmp[j][t] : v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    };
    const std::integral_constant<int, 0> q0{};
    // A k-step in quarters.  Beside a quarter's MFMAs: the reads and the widening of the next one's operands.
    auto step = [&](auto sc, auto mc, int chunk) __attribute__((always_inline)) {
      constexpr int s = decltype(sc)::value, d = s % D;
      constexpr bool more = decltype(mc)::value;
      static_for<3>([&](auto qc) __attribute__((always_inline)) {
        constexpr std::integral_constant<int, decltype(qc)::value + 1> next{};
        read_b(sc, next, chunk);
        widen(d, next);
        mul(qc);
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (more && s < SC / 2)   // the next chunk's rows, in the first half of this one
#pragma unroll
        for (int q = s; q < NQ; q += SC / 2) stage(q, chunk + 1);
      load_w(d, chunk * SC + s + D);
      if constexpr (s + 1 < SC) read_b(std::integral_constant<int, (s + 1) % SC>{}, q0, chunk);
      float scale[2];
#pragma unroll
      for (int m = 0; m < (GATE_UP ? 2 : 1); m++) scale[m] = s_sc[m * NKS + chunk * SC + s];
      widen((s + 1) % D, q0);
      mul(std::integral_constant<int, 3>{});
#pragma unroll
      for (int t = 0; t < MTL; t++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) acc[j][t][r] = fmaf(tmp[j][t][r], scale[GATE_UP ? j & 1 : 0], acc[j][t][r]);   // apply_scale_kgroup
      __builtin_amdgcn_sched_barrier(0);
    };
    widen(0, q0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int chunk = 0;
    for (; (chunk + 1) * SC <= NKS; chunk++) {
      read_b(q0, q0, chunk);
      static_for<SC>([&](auto sc) __attribute__((always_inline)) { step(sc, std::true_type{}, chunk); });
      // the next chunk is in the LDS (what was requested after its rows: SC / 2 + 1 steps of weights), and no one reads this one any more
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SC / 2 + 1) * NJ * 2) : "memory");
      __syncthreads();
    }
    if (chunk * SC < NKS) {
      read_b(q0, q0, chunk);
      static_for<SC>([&](auto sc) __attribute__((always_inline)) {
        if (chunk * SC + decltype(sc)::value < NKS) step(sc, std::false_type{}, chunk);
      });
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no request may outlive the workgroup's LDS

#pragma unroll
    for (int u = 0; u < SPW; u++) {
      const int st = strip0 + u;
      if (st >= nstrips) continue;
      const int n0 = st * 16 + kc * 4;
      // FP8_PERCHANNEL: the whole-K sum times the row's scale; x * 1.0f is exact, so the block-scaled format is untouched.  Asked for ahead of the stores, which the compiler
      // takes for writes to them, row by row: 64 experts of 2048 x 1024, top-8, 450 tokens 165 -> 137 us (moe_gemm_fp_kernel 156), of 2048 x 1408, top-6, 580 206 -> 181 (202).
      float rs0[4] = {1.f, 1.f, 1.f, 1.f}, rs1[4] = {1.f, 1.f, 1.f, 1.f};
      if (p.r0) {
        const float4 v = *reinterpret_cast<const float4*>(p.r0 + (size_t)tile.expert * p.N + n0);
        rs0[0] = v.x; rs0[1] = v.y; rs0[2] = v.z; rs0[3] = v.w;
      }
      if (GATE_UP && p.r1) {
        const float4 v = *reinterpret_cast<const float4*>(p.r1 + (size_t)tile.expert * p.N + n0);
        rs1[0] = v.x; rs1[1] = v.y; rs1[2] = v.z; rs1[3] = v.w;
      }
#pragma unroll
      for (int t = 0; t < MTL; t++) {
        const int row = t * 16 + i;
        if (row < tile.nrows) {
          bf16_t o[4];
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const bf16_t g = f32_to_bf16(acc[GATE_UP ? 2 * u : u][t][r] * rs0[r]);
            if constexpr (GATE_UP) {
              const bf16_t up = f32_to_bf16(acc[2 * u + 1][t][r] * rs1[r]);
              o[r] = f32_to_bf16(act_fn(bf16_to_f32(g), bf16_to_f32(up)));
            } else {
              o[r] = g;
            }
          }
          *reinterpret_cast<uint2*>(p.out + (size_t)(tile.row0 + row) * p.N + n0) =
              make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
        }
      }
    }
  };
  if (tile.nrows <= 16) run(std::integral_constant<int, 1>{});
  else run(std::integral_constant<int, 2>{});
}

template <bool GATE_UP>
static int launch_fp8_stream(const FpGemmParams& p, int max_tiles, hipStream_t st) {
  constexpr int per_wg = 4 * (GATE_UP ? 2 : 4);   // strips
  const int lds = (int)fp8_stream_lds(p.K);
  const hipError_t err = ktx_set_max_lds(reinterpret_cast<const void*>(moe_fp8_stream_kernel<GATE_UP>), 160 * 1024);
  KTX_HIP(err);
  hipLaunchKernelGGL((moe_fp8_stream_kernel<GATE_UP>), moe_job_grid(max_tiles, (p.N / 16 + per_wg - 1) / per_wg), dim3(256), lds, st, p);
  KTX_HIP(hipGetLastError());
  return 0;
}

int moe_launch_fp8_stream(bool gate_up, const FpGemmParams& p, int max_tiles, hipStream_t st) {
  return gate_up ? launch_fp8_stream<true>(p, max_tiles, st) : launch_fp8_stream<false>(p, max_tiles, st);
}
