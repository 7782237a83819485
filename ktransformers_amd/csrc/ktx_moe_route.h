// ktx_moe_route.h — a batch's way to its experts and back: ktx_moe_route.hip has the kernels, ktx_moe.hip calls them for every weight format.
#ifndef KTX_MOE_ROUTE_H
#define KTX_MOE_ROUTE_H
#include "ktx_common.h"
#include "ktx_moe_tile.h"

#define KTX_EMAX 1024   // experts of a handle

struct PrepParams {
  const int32_t* d_bsz;
  int qlen, k, E, expert_begin, H;
  int rows_per_tile;  // 16*MT
  bool by_size;       // the experts' tiles: from the expert of the most rows on, not in the experts' order (their rows lie in that in any case)
  const int64_t* ids;
  const uint8_t* mask;
  const bf16_t* x;
  int8_t* x_q;
  float* x_d;
  int32_t* row_of_pair;  // [qlen*k]  -> sorted row or -1
  int32_t* src_of_row;   // [qlen*k]  sorted row -> token index
  Tile* tiles;
  int32_t* counters;  // [0] = num_tiles, [1] = num_rows
};
// Buckets the pairs by expert and, if quantise, turns the tokens into int8 rows (x_q, x_d).
hipError_t moe_launch_prep(const PrepParams& p, bool quantise, hipStream_t st);

struct CombineParams {
  const int32_t* d_bsz;
  int qlen, k, H;
  const bf16_t* dn;            // [sorted rows][H]
  const int32_t* row_of_pair;  // [qlen*k]
  const float* weights;        // [qlen][k]
  bf16_t* y;                   // [qlen][H]  (float* when partial_f32)
  int incremental;
  int partial_f32;
  int dn_f32;                  // GGUF path: dn is fp32 and the sum is `out += dn * w` (llamafile/moe.hpp:447-449)
};
hipError_t moe_launch_combine(const CombineParams& p, hipStream_t st);
#endif
