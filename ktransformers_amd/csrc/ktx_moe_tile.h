// ktx_moe_tile.h — what every grouped expert kernel takes: the tiles that ktx_moe_route.hip lays out.
#ifndef KTX_MOE_TILE_H
#define KTX_MOE_TILE_H
#include "ktx_common.h"

struct Tile {
  int expert;  // local expert index
  int row0;    // first sorted row
  int nrows;   // <= 16*MT
  int idx;     // place among its expert's tiles
  int cnt;     // the expert's tiles
};
#endif
