// sg_tile_compact.hip's passes with sixteen wavefronts a tile.
#define SG_COMPACT 1
#define SG_WIDE 1
#include "sg_tile_iz.h"
