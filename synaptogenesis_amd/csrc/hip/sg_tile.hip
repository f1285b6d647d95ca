// Launchers of the tile kernels: the base activator, and the choice of the
// Izhikevich passes' translation unit.
#include "sg_tile_kernels.h"

namespace sg {

template <int TYPE, int D, int WAVES>
static void launch_tile_type(const sg_conn &c, hipStream_t st) {
    dim3 g((c.num_dest + D - 1) / D), b(64 * WAVES);
    switch (c.out_type) {
        case SG_OUT_BIT:
            hipLaunchKernelGGL((tile_base_kernel<TYPE, SG_OUT_BIT, D, WAVES>),
                               g, b, 0, st, c);
            break;
        case SG_OUT_INT:
            hipLaunchKernelGGL((tile_base_kernel<TYPE, SG_OUT_INT, D, WAVES>),
                               g, b, 0, st, c);
            break;
        default:
            hipLaunchKernelGGL((tile_base_kernel<TYPE, SG_OUT_FLOAT, D,
                                WAVES>), g, b, 0, st, c);
    }
}

template <int TYPE>
static void launch_lane_type(const sg_conn &c, hipStream_t st) {
    dim3 g((c.num_dest + 63) / 64), b(64);
    switch (c.out_type) {
        case SG_OUT_BIT:
            hipLaunchKernelGGL((lane_base_kernel<TYPE, SG_OUT_BIT>), g, b, 0,
                               st, c);
            break;
        case SG_OUT_INT:
            hipLaunchKernelGGL((lane_base_kernel<TYPE, SG_OUT_INT>), g, b, 0,
                               st, c);
            break;
        default:
            hipLaunchKernelGGL((lane_base_kernel<TYPE, SG_OUT_FLOAT>), g, b,
                               0, st, c);
    }
}

// Which form of the base activator (all three give the same bits), from one
// sweep of sizes:
// * lanes alone where a tile's visits would leave most of a block idle, up to
//   16 of them past two tiles a CU: 1 x 1 on 230 x 230 3.9 us against 6.7,
//   10 -> 1000000 fully connected 15 against 43;
// * and once the layer's own wavefronts fill the GPU and the visits' sources
//   have to be walked: convergent 5 x 5 on 256 x 256 (1024 tiles) 6.3 us
//   against 6.8, on 420 x 420 7.4 against 16, 9 x 9 on 420 x 420 17.8 against
//   28 (on 300 x 300: 15.9 against 15.6).  Fully connected layers need no walk
//   and keep the tile kernel past 32 visits (20 -> 131072 5.2 us against 6.9,
//   48 -> 131072 8.3 against 7.1); a sparse one's lists are better read by
//   whole blocks (64 visits, 2188 tiles: 31 us against 33, 600 visits 319
//   against 502);
// * 16 destinations a block while that gives every block a CU of its own
//   (64 tiles): 784 -> 1024 5.7 us against 11, 4096 -> 4096 24 against 55,
//   784 -> 8192 (128 tiles) 13.3 against 12.5; not for up to 64 visits,
//   which fill an eighth of its chunk: 5 x 5 into 576 3.7 us against 6.5.
template <int TYPE>
static hipError_t launch_base_type(const sg_conn &c, hipStream_t st) {
    const int tiles = (c.num_dest + 63) / 64;
    const int count = cursor<TYPE>(c, 0).count;
    const bool lanes =
        count <= 16 ? tiles > 512
        : TYPE == SG_FULLY_CONNECTED ? count <= 32 && tiles >= 2048
        : TYPE == SG_SPARSE ? false
                            : tiles >= (count <= 64 ? 1024 : 2048);
    if (lanes)
        launch_lane_type<TYPE>(c, st);
    else if (count > 64 && tiles <= 64)
        launch_tile_type<TYPE, 16, 16>(c, st);
    else
        launch_tile_type<TYPE, 64, 8>(c, st);
    return hipGetLastError();
}

hipError_t launch_tile_base(const sg_conn &c, hipStream_t st) {
    switch (c.type) {
        case SG_FULLY_CONNECTED:
            return launch_base_type<SG_FULLY_CONNECTED>(c, st);
        case SG_SUBSET: return launch_base_type<SG_SUBSET>(c, st);
        case SG_CONVERGENT: return launch_base_type<SG_CONVERGENT>(c, st);
        case SG_DIVERGENT: return launch_base_type<SG_DIVERGENT>(c, st);
        case SG_SPARSE: return launch_base_type<SG_SPARSE>(c, st);
    }
    return hipErrorInvalidValue;
}

// launch_iz_tile_<compact record><sixteen wavefronts a tile> (sg_tile_iz.h)
#define SG_DECLARE(N)                                                        \
    hipError_t launch_iz_tile_##N(const sg_conn &c, const sg_iz_syn &s,      \
                                  const sg_iz_dest &d, int kind, int sub,    \
                                  int upd, int act, const float *st_,        \
                                  const float *dt_, hipStream_t st);
SG_DECLARE(00)
SG_DECLARE(01)
SG_DECLARE(10)
SG_DECLARE(11)
#undef SG_DECLARE

hipError_t launch_iz_tile(const sg_conn &c, const sg_iz_syn &s,
                          const sg_iz_dest &d, int kind, int sub, int upd,
                          int act, const float *st_, const float *dt_,
                          hipStream_t st) {
    const bool wide = wide_tiles((c.num_dest + 63) / 64);
    auto *launch = s.src_stp ? (wide ? launch_iz_tile_11 : launch_iz_tile_10)
                             : (wide ? launch_iz_tile_01 : launch_iz_tile_00);
    return launch(c, s, d, kind, sub, upd, act, st_, dt_, st);
}

}  // namespace sg
