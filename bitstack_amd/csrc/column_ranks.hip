// The kernels of column.hip for ranks 4 to 15 (a translation unit of its own: the two compile side by side).
#define COLUMN_RANKS
#include "column.hip"
