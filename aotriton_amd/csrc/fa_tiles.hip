// Compile-time tile/occupancy table keyed on (element type, head dim, causal / windowed) and, where a kernel's
// variants differ, on the options; reported through fa_query_*_config.
#include "fa_fwd_impl.h"
#include "fa_bwd_pair.h"
#include "fa_bwd_wide.h"
#include "fa_fwd_wide.h"
#include "fa_kernels.h"

namespace fa {

template <typename T, int D> static TileShape fwd_shape_of(bool windowed, int half) {
  auto shape = [](auto tile, int per_cu) {
    using Tile = decltype(tile);
    return TileShape{Tile::BM, Tile::BN, Tile::NW, Tile::LDS, per_cu};
  };
  if constexpr (D <= 128) {
    if (D == 64 && half == 3) return shape(FwdThirdTile{}, 3);
    if (half) return shape(FwdHalfTile<D>{}, 2);
  }
  return windowed ? shape(FwdTile<T, D, true>{}, 1) : shape(FwdTile<T, D, false>{}, 1);
}

template <typename T, int D> static TileShape bwd_shape_of(bool windowed, bool bias, bool dropout, int slot, bool stored) {
  switch ((windowed ? 4 : 0) | (bias ? 2 : 0) | (dropout ? 1 : 0)) {
    case 0: return bwd_shape<T, D, false, false, false>(slot, stored);
    case 1: return bwd_shape<T, D, false, false, true>(slot, stored);
    case 2: return bwd_shape<T, D, false, true, false>(slot, stored);
    case 3: return bwd_shape<T, D, false, true, true>(slot, stored);
    case 4: return bwd_shape<T, D, true, false, false>(slot, stored);
    case 5: return bwd_shape<T, D, true, false, true>(slot, stored);
    case 6: return bwd_shape<T, D, true, true, false>(slot, stored);
    default: return bwd_shape<T, D, true, true, true>(slot, stored);
  }
}

TileShape fwd_tile_shape(int dtype, int head_dim, bool windowed, int half_tiles) {
  const bool bf = dtype == kDtypeBF16;
  switch (head_dim) {
    case 64: return bf ? fwd_shape_of<bf16_t, 64>(windowed, half_tiles) : fwd_shape_of<f16_t, 64>(windowed, half_tiles);
    case 128: return bf ? fwd_shape_of<bf16_t, 128>(windowed, half_tiles) : fwd_shape_of<f16_t, 128>(windowed, half_tiles);
    default: return bf ? fwd_shape_of<bf16_t, 256>(windowed, half_tiles) : fwd_shape_of<f16_t, 256>(windowed, half_tiles);
  }
}

TileShape bwd_tile_shape(int dtype, int head_dim, bool windowed, bool bias, bool dropout, int slot, bool stored) {
  const bool bf = dtype == kDtypeBF16;
  switch (head_dim) {
    case 64: return bf ? bwd_shape_of<bf16_t, 64>(windowed, bias, dropout, slot, stored) : bwd_shape_of<f16_t, 64>(windowed, bias, dropout, slot, stored);
    case 128: return bf ? bwd_shape_of<bf16_t, 128>(windowed, bias, dropout, slot, stored) : bwd_shape_of<f16_t, 128>(windowed, bias, dropout, slot, stored);
    default: return bf ? bwd_shape_of<bf16_t, 256>(windowed, bias, dropout, slot, stored) : bwd_shape_of<f16_t, 256>(windowed, bias, dropout, slot, stored);
  }
}

TileShape fwd_wide_shape() { return TileShape{256, 64, 4, WideFwdSmem::BYTES + kLevelBytes, 1}; }

TileShape bwd_pair_shape(bool bias) { return TileShape{32, 128, 8, bias ? PairSmem<true>::BYTES : PairSmem<false>::BYTES, 1}; }

TileShape bwd_wide_shape(bool dkdv) {
  return dkdv ? TileShape{kWideBM, kWideBN, 4, WideDkDvSmem::BYTES + kLevelBytes, 1} : TileShape{kWideBN, kWideBM, 4, WideDqSmem::BYTES + kLevelBytes, 1};
}

}  // namespace fa
