// Solo launches of the face/update tile kernel for cells of STRIDE slots (the Makefile compiles
// this file once per stride, so the instantiations build in parallel).
#include "face_tiles.hpp"
#include "tile_launch.hpp"

namespace ebb {

template <int S, int FLUX, int VISC, int ORDER, int LP, int MIX>
__global__ __launch_bounds__(BLK) void k_face_tile(DevMesh m, PhysParams p, StageArgs a, FaceTileArgs t)
{
    extern __shared__ double fsd[];
    const uint32_t tile = (a.order & 1) ? xcdBlockBack(blockIdx.x, gridDim.x) : xcdBlock(blockIdx.x, gridDim.x);
    faceTileBody<S, FLUX, VISC, ORDER, LP, MIX>(m, p, a, t, tile, blockIdx.x, fsd);
}

template <int S, int FLUX, int VISC>
static void faceTileO(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, hipStream_t st)
{
    const bool lp = p.order > 1 && p.limited && p.lpThresh > 0;
    const dim3 g(t.nTiles), b(BLK);
    if (p.mixed) {   // no LP vector limiter on the mixed path (rejected at set-up)
        if (p.order == 1) hipLaunchKernelGGL((k_face_tile<S, FLUX, VISC, 1, 0, 1>), g, b, t.ldsBytes, st, m, p, a, t);
        else if (!(p.limited && a.limit))
            hipLaunchKernelGGL((k_face_tile<S, FLUX, VISC, 2, 2, 1>), g, b, t.ldsBytes, st, m, p, a, t);
        else hipLaunchKernelGGL((k_face_tile<S, FLUX, VISC, 2, 0, 1>), g, b, t.ldsBytes, st, m, p, a, t);
        return;
    }
    if (p.order == 1) hipLaunchKernelGGL((k_face_tile<S, FLUX, VISC, 1, 0, 0>), g, b, t.ldsBytes, st, m, p, a, t);
    else if (!(p.limited && a.limit))
        hipLaunchKernelGGL((k_face_tile<S, FLUX, VISC, 2, 2, 0>), g, b, t.ldsBytes, st, m, p, a, t);
    else if (lp) hipLaunchKernelGGL((k_face_tile<S, FLUX, VISC, 2, 1, 0>), g, b, t.ldsBytes, st, m, p, a, t);
    else hipLaunchKernelGGL((k_face_tile<S, FLUX, VISC, 2, 0, 0>), g, b, t.ldsBytes, st, m, p, a, t);
}

template <int S>
void faceTileS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, hipStream_t st)
{
    if (p.flux == 1) {
        if (p.viscous) faceTileO<S, 1, 1>(m, p, a, t, st); else faceTileO<S, 1, 0>(m, p, a, t, st);
    } else {
        if (p.viscous) faceTileO<S, 0, 1>(m, p, a, t, st); else faceTileO<S, 0, 0>(m, p, a, t, st);
    }
}

template void faceTileS<STRIDE>(const DevMesh&, const PhysParams&, const StageArgs&, const FaceTileArgs&, hipStream_t);

}  // namespace ebb
