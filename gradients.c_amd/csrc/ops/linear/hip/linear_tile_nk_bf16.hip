/* linear_tile_nk.hip compiled over BF16 operands (linear_elem.h). */
#define GD_LINEAR_BF16 1
#include "linear_tile_nk.hip"
