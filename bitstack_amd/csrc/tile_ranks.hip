// The kernels of tile.hip for ranks 8 to 15 (a translation unit of its own: the two compile side by side).
#define TILE_RANKS
#include "tile.hip"
