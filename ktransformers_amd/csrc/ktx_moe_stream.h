// ktx_moe_stream.h — what ktx_moe.hip and ktx_moe_stream.hip (the streaming prompt GEMMs of AMXINT4 / AMXINT8 and FP8 experts) share.
#ifndef KTX_MOE_STREAM_H
#define KTX_MOE_STREAM_H
#include "ktx_common.h"
#include "ktx_moe_tile.h"

// Workgroup -> (tile, strip group) of a grouped GEMM, from a one-dimensional grid: ids are dealt round-robin to the 8 XCDs, so id % 8 is the
// XCD.  The jobs lie expert after expert, within an expert strip group by strip group, the group's tiles side by side; each XCD takes an
// eighth of them.  So the XCDs end together whatever the number of tiles, an expert's weights go into one L2 and are read there once for all
// its tiles, and its rows (the operand every strip group re-reads) stay there too.  False: nothing to do.
// SHARE false: launch order, for tiles so low that an expert mostly has one (256 experts of 7168 x 2048, AMXINT4, 114 tokens: shares cost 1 %).
template <bool SHARE = true>
__device__ __forceinline__ bool moe_pick_job(const Tile* tiles, int ntiles, int nsg, Tile& tile, int& sgroup) {
  if constexpr (!SHARE) {
    const int t = blockIdx.x / nsg;
    if (t >= ntiles) return false;
    tile = tiles[t];
    sgroup = blockIdx.x - t * nsg;
    return true;
  }
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int total = ntiles * nsg, per = (total + 7) / 8, job = xcd * per + seq;
  if (seq >= per || job >= total) return false;
  tile = tiles[job / nsg];
  const int first = job / nsg - tile.idx, ofs = job - first * nsg;
  sgroup = ofs / tile.cnt;
  if (tile.cnt > 1) tile = tiles[first + ofs % tile.cnt];
  return true;
}
// The same by strip groups: an XCD takes every eighth one, of all experts, so that the XCDs end together whatever their experts' tiles hold.  With the experts from the most
// rows on (PrepParams.by_size) what ends last is small.  The groups past the last eight are dealt job by job, and go first.
__device__ __forceinline__ bool moe_pick_strips(const Tile* tiles, int ntiles, int nsg, Tile& tile, int& sgroup) {
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3, main = nsg >> 3, rest = nsg & 7;
  const int dealt = (ntiles * rest + 7 - xcd) >> 3;
  if (seq < dealt) {
    const int u = seq * 8 + xcd, t = u / rest;
    tile = tiles[t];
    sgroup = main * 8 + u - t * rest;
    return true;
  }
  const int j = seq - dealt;
  if (j >= ntiles * main) return false;
  const int t = j / main;
  tile = tiles[t];
  const int first = t - tile.idx, ofs = j - first * main;
  sgroup = ofs / tile.cnt * 8 + xcd;
  if (tile.cnt > 1) tile = tiles[first + ofs % tile.cnt];
  return true;
}
static dim3 moe_strip_grid(int max_tiles, int nsg) { return dim3((unsigned)((size_t)max_tiles * (nsg >> 3) + ((size_t)max_tiles * (nsg & 7) + 7) / 8) * 8); }
static dim3 moe_job_grid(int max_tiles, int nsg) { return dim3((unsigned)(((size_t)max_tiles * nsg + 7) / 8 * 8)); }

struct GemmParams {
  const uint8_t* w0;   // gate (GATE_UP) or down
  const uint8_t* w1;   // up   (GATE_UP) or nullptr
  const float* s0;     // scales [E][N]
  const float* s1;
  size_t expert_stride;  // bytes of one expert's matrix
  int N, K;
  const int8_t* act_q;      // [src rows][K]
  const float* act_d;       // [src rows]
  const int32_t* row_src;   // sorted row -> source row (nullptr: identity)
  const Tile* tiles;
  const int32_t* counters;
  bf16_t* out;  // [sorted rows][N]
};

constexpr int STREAM_ROWS = 64;   // rows of a tile
// One grouped GEMM of a prompt on tiles of STREAM_ROWS rows; wbits 4 or 8; nw: 8 wavefronts in a workgroup that has a CU to itself, or 4 in one of two.
int moe_launch_gemm_stream(int wbits, int nw, bool gate_up, const GemmParams& p, int max_tiles, hipStream_t st);

// ---- FP8 (and BF16) experts: the layout of their weights is at moe_gemm_fp_kernel
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ v8bf u4_as_v8bf(const uint4& u) {
  union { uint4 u; v8bf v; } c;
  c.u = u;
  return c.v;
}

// 4 e4m3 bytes -> 4 bf16 (two dwords): v_cvt_pk_f32_fp8 is exact, and every e4m3 value is exact in bf16, so taking the
// upper halves of the fp32 results is exact (OCP e4m3fn on gfx950; 0x7F/0xFF are NaN here, +-480 in the reference's LUT).
__device__ __forceinline__ uint2 fp8x4_to_bf16x4(uint32_t v) {
  // gfx950: v_cvt_scalef32_pk_bf16_fp8 converts two e4m3 bytes straight to two bf16 (scale 1.0): 2 VALU instructions per four weights
  // instead of two converts + two packs (scripts/fp8_cvt_probe.hip: the same bits as the two-step path for all 256 codes)
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  union { bf2 v; uint32_t u; } lo, hi;
  lo.v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, false);
  hi.v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, true);
  return make_uint2(lo.u, hi.u);
}

struct FpGemmParams {
  const uint8_t *w0, *w1;     // tiled weights (gate | down, up)
  const float *s0, *s1;       // FP8: scale_inv [E][N/128][K/128]; BF16: nullptr
  const float *r0, *r1;       // FP8_PERCHANNEL: scale per output row [E][N] (the block scales are then all 1), else nullptr
  size_t expert_stride;       // bytes per expert matrix
  size_t scale_stride;        // floats per expert
  int N, K;
  const bf16_t* act;          // [src rows][K] bf16
  const int32_t* row_src;     // sorted row -> source row (nullptr: identity)
  const Tile* tiles;
  const int32_t* counters;
  bf16_t* out;                // [sorted rows][N]
};

// the places of a row's pieces: distinct for 16 rows, also with rows 4 .. 11 flipped by 4 (ds_read_b128 takes lanes 0-3, 12-15, 20-23, 24-27 together)
__device__ __forceinline__ int fp_swz(int row) { return (row & 3) | (int)((0x3102u >> (((row >> 2) & 3) * 4)) & 3u) << 2; }
constexpr int FP_STREAM_ROWS = 32;
static inline size_t fp8_stream_lds(int K) { return 2 * FP_STREAM_ROWS * 4 * 256 + (size_t)4 * 2 * (K / 128) * sizeof(float); }   // two buffers of activations, scales
// One grouped GEMM of an FP8 batch on tiles of FP_STREAM_ROWS rows.
int moe_launch_fp8_stream(bool gate_up, const FpGemmParams& p, int max_tiles, hipStream_t st);
#endif
