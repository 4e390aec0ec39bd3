// Fused level kernels of the V-cycle (mg_fused.hip): the start of a
// smoothing with its first sweep, and the residuum with its restriction.
#pragma once

#include <hip/hip_runtime.h>

#include "device.h"

namespace artss {
namespace k {

// the map and the items (MgFill) of a fill; n_items: its fill items in the
// form of dev::bc_items_grid, then the ghost cells if the fill leaves some
void build_mg_fill(hipStream_t s, const LevelDesc &L, const BCView &V, int32_t *map, int32_t *items, int n_items);

// one weighted-Jacobi sweep of a level
struct MgSweep {
    double ax, ay, az, beta, dsign, w;
};

// dst = one sweep, with its fill, of the iterate x carrying its fill
// (x nullptr: the result of a sweep from zero, w beta dsign b on the fluid
// cells).  The filled iterate is not stored.  Every cell of dst is written:
// cells off the fluid that the fill does not write get the iterate's value.
// dst must not be x or b.
template <typename T, typename TB>
void smooth_first(hipStream_t s, const LevelDesc &L, const MgFill &F, const MgSweep &c, T *dst, const T *x,
                  const TB *b);
// the same for the iterate x + prolongate(coarse); dst must not be coarse
// (x nullptr: in FP32 only)
template <typename T, typename TB, typename Tc>
void smooth_corrected(hipStream_t s, const LevelDesc &L, const MgFill &F, const MgSweep &c, T *dst, const T *x,
                      const TB *b, const LevelDesc &Lc, const MgFill &Fc, const Tc *coarse);
// out = restrict(b - lap(x)) on the coarse fluid cells, err (unless nullptr)
// = 0 on the whole coarse array.  x carries its fill; nullptr: x is the sweep
// from zero of b with the fill, evaluated from b, in FP32 only.  The
// restriction must not read the fine ghost layer.
template <typename T, typename TB, typename Tout>
void residuum_restrict(hipStream_t s, const LevelDesc &Lc, const LevelDesc &Lf, const MgFill &F, const MgSweep &c,
                       Tout *out, Tout *err, const T *x, const TB *b);

}  // namespace k
}  // namespace artss
