// Batched launches of the face/update tile kernel for cells of STRIDE slots (compiled once per
// stride).
#include "face_tiles.hpp"
#include "tile_launch.hpp"

namespace ebb {

template <int S, int FLUX, int VISC, int ORDER, int LP, int MIX>
__global__ __launch_bounds__(BLK) void k_face_tile_batch(const MemberArgs* __restrict__ mem,
                                                         const uint2* __restrict__ items, uint32_t parity, uint32_t stage)
{
    extern __shared__ double fsd[];
    const uint2 it = items[xcdBlock(blockIdx.x, gridDim.x)];
    const MemberArgs& M = mem[it.x];
    faceTileBody<S, FLUX, VISC, ORDER, LP, MIX>(M.m, M.p, M.st[parity ^ M.parityFlip][stage], M.t, it.y, it.y, fsd);
}

template <int S, int FLUX, int VISC, int MIX>
static void faceBatchO(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items, uint32_t n,
                       uint32_t lds, uint32_t par, uint32_t stg, hipStream_t s)
{
    const dim3 g(n), b(BLK);
    if (gs.order == 1) hipLaunchKernelGGL((k_face_tile_batch<S, FLUX, VISC, 1, 0, MIX>), g, b, lds, s, mem, items, par, stg);
    else if (!(gs.limited && limitStage))
        hipLaunchKernelGGL((k_face_tile_batch<S, FLUX, VISC, 2, 2, MIX>), g, b, lds, s, mem, items, par, stg);
    else hipLaunchKernelGGL((k_face_tile_batch<S, FLUX, VISC, 2, 0, MIX>), g, b, lds, s, mem, items, par, stg);
}

template <int S, int MIX>
void faceBatchS(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items, uint32_t n,
                       uint32_t lds, uint32_t par, uint32_t stg, hipStream_t s)
{
    if (gs.flux == 1) {
        if (gs.viscous) faceBatchO<S, 1, 1, MIX>(gs, limitStage, mem, items, n, lds, par, stg, s);
        else faceBatchO<S, 1, 0, MIX>(gs, limitStage, mem, items, n, lds, par, stg, s);
    } else {
        if (gs.viscous) faceBatchO<S, 0, 1, MIX>(gs, limitStage, mem, items, n, lds, par, stg, s);
        else faceBatchO<S, 0, 0, MIX>(gs, limitStage, mem, items, n, lds, par, stg, s);
    }
}

template void faceBatchS<STRIDE, 0>(const GroupShape&, int, const MemberArgs*, const uint2*, uint32_t, uint32_t,
                                    uint32_t, uint32_t, hipStream_t);
template void faceBatchS<STRIDE, 1>(const GroupShape&, int, const MemberArgs*, const uint2*, uint32_t, uint32_t,
                                    uint32_t, uint32_t, hipStream_t);

}  // namespace ebb
