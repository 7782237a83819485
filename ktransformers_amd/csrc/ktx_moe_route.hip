// ktx_moe_route.hip — bucketing of (token, expert) pairs, int8 rows of the tokens, and the weighted combine of the experts' rows.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ktx_common.h"
#include "ktx_moe_dec.inc"
#include "ktx_moe_route.h"

// =====================================================================================================
// K0: prep — workgroups 0 .. E-1 bucket the (t,j) pairs, one expert each; the others quantise tokens' activations (a5, a6)
// =====================================================================================================
constexpr int PREP_THREADS = 1024;

// per row: d = amax/127, id = d ? 1/d : 0, q = sat8(rne(x*id))   (amx_buffers.hpp:47-98).  The row stays in registers between the two passes (K <= 8192).
// Every thread of the workgroup comes here; red: LDS, one float per wavefront.
__device__ __forceinline__ void quant_row_256(bool live, const bf16_t* __restrict__ src, int K, int8_t* __restrict__ dst, float* __restrict__ d_out, float* red) {
  const int g = threadIdx.x & 255;
  constexpr int HELD = 4, STEP = 256 * 8;
  uint4 v[HELD];
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < HELD; i++) {
    const int j = g * 8 + i * STEP;
    v[i] = live && j < K ? *reinterpret_cast<const uint4*>(src + j) : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < HELD; i++) amax = amax8(v[i], amax);
  for (int j = g * 8 + HELD * STEP; live && j < K; j += STEP) amax = amax8(*reinterpret_cast<const uint4*>(src + j), amax);
  amax = wave_max(amax);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[w] = amax;
  __syncthreads();
  if (!live) return;
  const float* r = red + (w & ~3);
  const float d = fmaxf(fmaxf(r[0], r[1]), fmaxf(r[2], r[3])) / 127.0f;
  const float id = d ? 1.0f / d : 0.0f;
#pragma unroll
  for (int i = 0; i < HELD; i++) {
    const int j = g * 8 + i * STEP;
    if (j < K) *reinterpret_cast<uint2*>(dst + j) = quant8(v[i], id);
  }
  for (int j = g * 8 + HELD * STEP; j < K; j += STEP) *reinterpret_cast<uint2*>(dst + j) = quant8(*reinterpret_cast<const uint4*>(src + j), id);
  if (g == 0) *d_out = d;
}

// Rows of an expert lie in (token, slot) order — the reference's m_local_pos_ (moe_base.hpp:208-227): the row of a pair depends on the routing table only.
// A workgroup reads the whole table: it counts all experts' pairs (LDS), which gives its expert's first row and first tile, then ranks its own expert's pairs, a
// stretch of the table per wavefront, by ballots; a stretch of up to 512 pairs is read once.  No workgroup waits for another.  Us, one workgroup for all experts (a CU's vector ALU and
// LDS, three passes) -> E of them that read the table twice -> here: 256 experts, top-8, 2048 tokens 45 -> 19.6 -> 19.6, 1000 24.1 -> 12.1 -> 10.9, 32 10.5 -> 4.7 -> 4.2; 64, top-6, 300
// 7.7 -> 7.4 -> 6.2; 8, top-2, 1000 8.0 -> 8.3 -> 7.4, 500 5.9 -> 6.6 -> 6.2, 100 4.6 -> 5.0 -> 4.3 (with the tokens' int8 rows beside).
__global__ __launch_bounds__(PREP_THREADS) void moe_prep_kernel(PrepParams p) {
  __shared__ int s_cnt[KTX_EMAX];
  __shared__ float s_red[PREP_THREADS / 64];
  __shared__ int s_sum[4][PREP_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = blockDim.x >> 6;
  int T = p.qlen;
  if (p.d_bsz) T = min(max(*p.d_bsz, 0), p.qlen);
  const int E = p.E;

  if ((int)blockIdx.x >= E) {
    const int t = (blockIdx.x - E) * (blockDim.x >> 8) + (tid >> 8);
    quant_row_256(t < T, p.x + (size_t)t * p.H, p.H, p.x_q + (size_t)t * p.H, p.x_d + t, s_red);
    return;
  }

  const int me = blockIdx.x, npairs = T * p.k;
  const int per_wave = ((npairs + nwaves - 1) / nwaves + 63) & ~63, i0 = min(wave * per_wave, npairs), i1 = min(i0 + per_wave, npairs);
  auto expert = [&](long long id) -> int {
    id -= p.expert_begin;
    return (id >= 0 && id < E && !(p.mask && p.mask[id])) ? (int)id : -1;
  };
  constexpr int U = 8;
  int ex[U];   // of 64 pairs each: the expert, -1: none, -2: no pair
  auto fetch = [&](int base) {
    long long id[U];
#pragma unroll
    for (int u = 0; u < U; u++) id[u] = p.ids[min(base + u * 64 + lane, npairs - 1)];
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (base + u * 64 >= i1) break;
      ex[u] = base + u * 64 + lane < i1 ? expert(id[u]) : -2;
    }
  };
  for (int e = tid; e < E; e += blockDim.x) s_cnt[e] = 0;
  __syncthreads();
  int mine = 0;   // this wavefront's pairs of this workgroup's expert
  for (int base = i0; base < i1; base += U * 64) {
    fetch(base);
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (base + u * 64 >= i1) break;
      if (ex[u] >= 0) atomicAdd(&s_cnt[ex[u]], 1);   // (an integer sum: the order of the adds does not matter)
      mine += __popcll(__ballot(ex[u] == me));
    }
  }
  __syncthreads();
  auto tiles_of = [&](int c) { return (c + p.rows_per_tile - 1) / p.rows_per_tile; };
  const int mine_all = s_cnt[me];
  {   // rows of the experts before this one, tiles of those whose tiles lie before its own, and rows and tiles of all
    int v[4] = {0, 0, 0, 0};
    for (int e = tid; e < E; e += blockDim.x) {
      const int c = s_cnt[e], tl = tiles_of(c);
      v[2] += c; v[3] += tl;
      if (e < me) v[0] += c;
      if (p.by_size && c != mine_all ? c > mine_all : e < me) v[1] += tl;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) v[q] += __shfl_xor(v[q], o, 64);
      if (lane == 0) s_sum[q][wave] = v[q];
    }
  }
  __shared__ int s_mine[PREP_THREADS / 64];
  if (lane == 0) s_mine[wave] = mine;
  __syncthreads();
  int sum[4] = {0, 0, 0, 0}, run = 0;
  for (int w = 0; w < nwaves; w++) {
#pragma unroll
    for (int q = 0; q < 4; q++) sum[q] += s_sum[q][w];
    if (w < wave) run += s_mine[w];
  }
  const int row0 = sum[0], cnt = mine_all, ntiles = tiles_of(cnt);
  if (me == 0 && tid == 0) { p.counters[0] = sum[3]; p.counters[1] = sum[2]; }
  run += row0;
  if (mine || me == 0)
    for (int base = i0; base < i1; base += U * 64) {
      if (per_wave > U * 64) fetch(base);   // (a stretch of one step is still there)
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (base + u * 64 >= i1) break;
        const int i = base + u * 64 + lane;
        const unsigned long long m = __ballot(ex[u] == me);
        if (ex[u] == me) {
          const int r = run + __popcll(m & ((1ull << lane) - 1ull));
          p.src_of_row[r] = i / p.k;
          p.row_of_pair[i] = r;
        } else if (me == 0 && ex[u] == -1) {
          p.row_of_pair[i] = -1;
        }
        run += __popcll(m);
      }
    }
  for (int i = tid; i < ntiles; i += blockDim.x) {
    Tile t;
    t.expert = me; t.row0 = row0 + i * p.rows_per_tile; t.nrows = min(p.rows_per_tile, cnt - i * p.rows_per_tile); t.idx = i; t.cnt = ntiles;
    p.tiles[sum[1] + i] = t;
  }
}

hipError_t moe_launch_prep(const PrepParams& p, bool quantise, hipStream_t st) {
  const int threads = (size_t)p.qlen * p.k <= 2048 ? 256 : PREP_THREADS, tokens = threads / 256;   // a few pairs: little to share, and more workgroups for the tokens
  hipLaunchKernelGGL(moe_prep_kernel, dim3(p.E + (quantise ? (p.qlen + tokens - 1) / tokens : 0)), dim3(threads), 0, st, p);
  return hipGetLastError();
}

// =====================================================================================================
// K3: weighted combine in slot order (a12) + merge/incremental + bf16 (a4)
// =====================================================================================================
// What it costs is the rows' way in, so a thread's loads are V elements wide and U experts of a token are asked for before the first is used.  Us, 4 elements a thread, one expert
// after the other -> here: 2048 rows of 7168, top-8, 52 -> 43 (6.1 TB/s); 1000 23.4 -> 21.9; 2048 of 4096, top-2, 11.6 -> 10.4.
template <int V, bool F32, int U>
__global__ __launch_bounds__(128) void moe_combine_kernel(CombineParams p) {
  int T = p.qlen;
  if (p.d_bsz) T = min(max(*p.d_bsz, 0), p.qlen);
  const int t = blockIdx.y;
  if (t >= T) return;
  const int h = (blockIdx.x * blockDim.x + threadIdx.x) * V;
  if (h >= p.H) return;
  const int32_t* rows = p.row_of_pair + (size_t)t * p.k;
  const float* weights = p.weights + (size_t)t * p.k;
  constexpr int NQ = V * (F32 ? 4 : 2) / 8;   // pieces of 8 bytes
  float acc[V];
#pragma unroll
  for (int e = 0; e < V; e++) acc[e] = 0.f;
  for (int j0 = 0; j0 < p.k; j0 += U) {
    int r[U];
    float ws[U];
    uint2 v[U][NQ];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int j = min(j0 + u, p.k - 1), row = rows[j];
      ws[u] = weights[j];
      r[u] = j0 + u < p.k ? row : -1;
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (r[u] < 0) continue;
      const uint8_t* src = reinterpret_cast<const uint8_t*>(p.dn) + ((size_t)r[u] * p.H + h) * (F32 ? 4 : 2);
      if constexpr (NQ >= 2) {
#pragma unroll
        for (int q = 0; q < NQ; q += 2) {
          const uint4 f = *reinterpret_cast<const uint4*>(src + q * 8);
          v[u][q] = make_uint2(f.x, f.y);
          v[u][q + 1] = make_uint2(f.z, f.w);
        }
      } else {
        v[u][0] = *reinterpret_cast<const uint2*>(src);
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (r[u] < 0) continue;
      const float w = ws[u];
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        if constexpr (F32) {
          acc[2 * q] = acc[2 * q] + __uint_as_float(v[u][q].x) * w;
          acc[2 * q + 1] = acc[2 * q + 1] + __uint_as_float(v[u][q].y) * w;
        } else {
          const uint32_t d[2] = {v[u][q].x, v[u][q].y};
#pragma unroll
          for (int e = 0; e < 2; e++) {
            acc[4 * q + 2 * e] = fmaf(bf16_to_f32((bf16_t)(d[e] & 0xffffu)), w, acc[4 * q + 2 * e]);
            acc[4 * q + 2 * e + 1] = fmaf(bf16_to_f32((bf16_t)(d[e] >> 16)), w, acc[4 * q + 2 * e + 1]);
          }
        }
      }
    }
  }
  if (p.partial_f32) {  // expert-parallel partial: un-rounded fp32 sums, reduced across ranks by the caller
    float* fp = reinterpret_cast<float*>(p.y) + (size_t)t * p.H + h;
#pragma unroll
    for (int e = 0; e < V; e += 4) *reinterpret_cast<float4*>(fp + e) = make_float4(acc[e], acc[e + 1], acc[e + 2], acc[e + 3]);
    return;
  }
  bf16_t* yp = p.y + (size_t)t * p.H + h;
#pragma unroll
  for (int e = 0; e < V; e += 4) {
    if (p.incremental) {
      const uint2 o = *reinterpret_cast<const uint2*>(yp + e);
      acc[e] = acc[e] + bf16_to_f32((bf16_t)(o.x & 0xffffu));
      acc[e + 1] = acc[e + 1] + bf16_to_f32((bf16_t)(o.x >> 16));
      acc[e + 2] = acc[e + 2] + bf16_to_f32((bf16_t)(o.y & 0xffffu));
      acc[e + 3] = acc[e + 3] + bf16_to_f32((bf16_t)(o.y >> 16));
    }
    const uint32_t lo = (uint32_t)f32_to_bf16(acc[e]) | ((uint32_t)f32_to_bf16(acc[e + 1]) << 16);
    const uint32_t hi = (uint32_t)f32_to_bf16(acc[e + 2]) | ((uint32_t)f32_to_bf16(acc[e + 3]) << 16);
    *reinterpret_cast<uint2*>(yp + e) = make_uint2(lo, hi);
  }
}

// U: the experts of a token, as 2, 4 or 8 (what is asked for in vain, and its code, shows in short calls: 500 tokens of 4096, top-2, U 8 4.8 us, 2: 4.4)
template <int V, bool F32>
static void launch_combine(const CombineParams& p, hipStream_t st) {
  const dim3 g((p.H / V + 127) / 128, p.qlen);
  if (p.k <= 2) hipLaunchKernelGGL((moe_combine_kernel<V, F32, 2>), g, dim3(128), 0, st, p);
  else if (p.k <= 4) hipLaunchKernelGGL((moe_combine_kernel<V, F32, 4>), g, dim3(128), 0, st, p);
  else hipLaunchKernelGGL((moe_combine_kernel<V, F32, 8>), g, dim3(128), 0, st, p);
}

// 8 elements a thread where rows lie on 16 bytes (H a multiple of 8 and the rows' address) and there are enough of them for the CUs, 4 otherwise (100 tokens of 4096, top-2, 8 | 4 elements:
// 3.6 | 3.2 us, 64 of 2048, top-6: 4.6 | 4.0; 300 of 4096, top-2 about even); fp32 rows of 4 elements are 16 bytes wide as well
hipError_t moe_launch_combine(const CombineParams& p, hipStream_t st) {
  if (p.dn_f32) launch_combine<4, true>(p, st);
  else if ((size_t)p.qlen * p.H >= ((size_t)1 << 20) && p.H % 8 == 0 && (reinterpret_cast<uintptr_t>(p.dn) & 15) == 0) launch_combine<8, false>(p, st);
  else launch_combine<4, false>(p, st);
  return hipGetLastError();
}
