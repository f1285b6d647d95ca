// The Izhikevich tile passes of one record form (SG_COMPACT) and block width
// (SG_WIDE), a translation unit each: the instantiations take minutes to
// compile, side by side.
#include "sg_tile_kernels.h"

#ifndef SG_WIDE
#define SG_WIDE 0
#endif
#define SG_PASTE(a, b, c) a##b##c
#define SG_LAUNCHER(c, w) SG_PASTE(launch_iz_tile_, c, w)

namespace sg {

hipError_t SG_LAUNCHER(SG_COMPACT, SG_WIDE)(
        const sg_conn &c, const sg_iz_syn &s, const sg_iz_dest &d, int kind,
        int sub, int upd, int act, const float *st_, const float *dt_,
        hipStream_t st) {
    if (upd && act)
        return launch_iz_tile_t<1, 1, SG_COMPACT, SG_WIDE>(c, s, d, kind, sub,
                                                           st_, dt_, st);
    if (upd)
        return launch_iz_tile_t<1, 0, SG_COMPACT, SG_WIDE>(
            c, s, d, sub ? SG_IZ_SUB : SG_IZ_ADD, sub, st_, dt_, st);
    return launch_iz_tile_t<0, 1, SG_COMPACT, SG_WIDE>(c, s, d, kind, 0, st_,
                                                       dt_, st);
}

}  // namespace sg
