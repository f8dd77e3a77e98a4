// The kernels of tile.hip for ranks 4 to 7 (a translation unit of its own: they compile side by side).
#define TILE_RANKS 4
#define TILE_LAUNCH bs_launch_tile_few_ranks
#include "tile.hip"
