// ktx_moe_tile.h — what every grouped expert kernel takes: the tiles that ktx_moe_route.hip lays out; and a loop over constants.
#ifndef KTX_MOE_TILE_H
#define KTX_MOE_TILE_H
#include <type_traits>

template <int N, class F, int I = 0>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, F, I + 1>(static_cast<F&&>(f));
  }
}

struct Tile {
  int expert;  // local expert index
  int row0;    // first sorted row
  int nrows;   // <= 16*MT
  int idx;     // place among its expert's tiles
  int cnt;     // the expert's tiles
};
#endif
