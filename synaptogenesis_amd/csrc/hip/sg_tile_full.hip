// Tile kernels, full records: the Izhikevich passes over records with every
// per-synapse field.
#define SG_COMPACT 0
#include "sg_tile_iz.h"
