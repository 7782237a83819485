// ktx_moe_raw.h — what ktx_moe.hip (which buckets, quantises and combines) and ktx_moe_raw.hip (the prompt GEMM of RAWINT4 experts) share.
#ifndef KTX_MOE_RAW_H
#define KTX_MOE_RAW_H
#include "ktx_common.h"
#include "ktx_moe_tile.h"

struct RawGemmParams {
  const uint8_t *w0, *w1;      // RAW tiles (gate | down, up)
  const bf16_t *s0, *s1;       // bf16 scales, [row group][step][row][half][8 blocks] (pack_rawint4_scales_kernel)
  size_t expert_stride;        // bytes of weights per expert matrix
  size_t scale_stride;         // bf16 elements of scales per expert matrix
  int N, K;
  const int8_t* act_q;         // [src rows][K] int8 codes, or f16 ones (prompts: 2 K bytes a row)
  const float* act_d;          // [src rows][K/32]
  const int32_t* row_src;
  const Tile* tiles;           // rows per tile: 4, of a prompt RAW_ROWS
  const int32_t* counters;
  bf16_t* out;                 // [sorted rows][N]
};

typedef _Float16 raw_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 raw_h8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ uint32_t raw_h2_bits(raw_h2 v) { return __builtin_bit_cast(uint32_t, v); }

constexpr int RAW_ROWS = 64;   // rows of a prompt tile
// One grouped GEMM of a RAWINT4 prompt on tiles of RAW_ROWS rows.
int moe_launch_rawint4_chunk(bool gate_up, const RawGemmParams& p, int max_tiles, hipStream_t st);
#endif
