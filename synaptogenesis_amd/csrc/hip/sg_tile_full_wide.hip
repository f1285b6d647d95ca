// sg_tile_full.hip's passes with sixteen wavefronts a tile.
#define SG_COMPACT 0
#define SG_WIDE 1
#include "sg_tile_iz.h"
