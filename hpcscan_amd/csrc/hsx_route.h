// Which 3D grids the entry points send to the tiled kernels.
#ifndef HSX_ROUTE_H
#define HSX_ROUTE_H

#include "hsx_internal.h"

namespace hsx {

// Grids of up to 5 MB an array run one thread per point: a launch of the tiled
// kernels lasts as long as a workgroup's chunk of planes takes one after the
// other, one thread per point has no such chain.  Step, Laplacian and D2 along
// n3, one thread per point against tiled (us): FP32 order 8 61^3 3.8 / 3.7 / 3.9
// against 17 / 15 / 9, 80^3 5.5 (step) against 5.8, 100^3 8.0 / 6.9 / 5.1 against
// 7.4 / 7.0 / 5.7, 128^3 13.0 / 11.2 / 10.1 against 8.4 / - / -; FP64 100^3 (10
// MB) 15.7 (step) against 9.5.
constexpr int64_t TILED_LEAST_BYTES = 5200000;
bool tile_shape_forced(void);   // hsx_set_tile asks for a shape (hsx_tiled_ac2.hip)
// the library's own choice, where no shape is asked for
inline bool tiled_own(const hsx_grid *g)
{
    // (the contracted arithmetic exists in the tiled kernels only)
    if (kernel_family() == HSX_KERNEL_TILED || contract_mode()) return true;
    // one thread per point has a plane per workgroup along z: 65535 at most
    if (g->inner[5] - g->inner[4] >= 65535) return true;
    return g->n1 * g->n2 * g->n3 * (g->storage == HSX_FP64 ? 8 : 4) >= TILED_LEAST_BYTES;
}
inline bool tiled_pays(const hsx_grid *g)
{
    return tile_shape_forced() || tiled_own(g);
}
// the fused step: also where hsx_autotune found a tile shape faster than the own choice
bool step_shape_tuned(const hsx_grid *g);   // hsx_tiled_ac2.hip
inline bool step_tiled(const hsx_grid *g)
{
    return tiled_pays(g) || step_shape_tuned(g);
}

} // namespace hsx

#endif
