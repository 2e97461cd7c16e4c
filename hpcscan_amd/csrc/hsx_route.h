// Which 3D grids the entry points send to the tiled kernels.
#ifndef HSX_ROUTE_H
#define HSX_ROUTE_H

#include "hsx_internal.h"

namespace hsx {

// Rows that are not whole 16-byte vectors (odd sizes, odd halo widths): the
// tiled kernels take them, one thread per point does as well on small grids,
// where a launch lasts as long as one workgroup's chunk of planes.  FP32 order
// 8, step / Laplacian / D2 along n3, one thread per point against tiled (us):
// 101^3 8.6 / 7.1 / 4.9 against 22.1 / 17.1 / 10.6; 151^3 24.6 / 18.6 / 15.4
// against 38.4 / 17.7 / 15.9; 201 x 203 x 199 48.6 / 39.2 / 27.7 against 41.7 /
// 23.3 / 16.1; 301 x 299 x 303 197 / 138 / 141 against 115 / 64 / 38.
constexpr int64_t UNALIGNED_TILED_POINTS = 6000000;
bool tile_shape_forced(void);   // hsx_set_tile asks for a shape (hsx_tiled_ac2.hip)
inline bool tiled_pays(const hsx_grid *g)
{
    if (kernel_family() == HSX_KERNEL_TILED || tile_shape_forced()) return true;
    if (g->n1 % (g->storage == HSX_FP64 ? 2 : 4) == 0) return true;
    return g->n1 * g->n2 * g->n3 >= UNALIGNED_TILED_POINTS;
}

} // namespace hsx

#endif
