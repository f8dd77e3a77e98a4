// The kernels of tile.hip for ranks 8 to 15 (a translation unit of its own: they compile side by side).
#define TILE_RANKS 8
#define TILE_LAUNCH bs_launch_tile_ranks
#include "tile.hip"
