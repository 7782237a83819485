// ktx_moe_stream.h — what ktx_moe.hip (which buckets, quantises and combines) and ktx_moe_stream.hip (the prompt GEMM of AMXINT4 / AMXINT8 experts) share.
#ifndef KTX_MOE_STREAM_H
#define KTX_MOE_STREAM_H
#include "ktx_common.h"
#include "ktx_moe_raw.h"

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
#endif
