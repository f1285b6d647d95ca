// Tile kernels, compact records (sg_hip.h: SG_IZC_*): the Izhikevich
// passes whose presynaptic trace and short-term plasticity are kept per
// source.
#define SG_COMPACT 1
#include "sg_tile_iz.h"
