// The gradient kernel, solo and batched, for cells of STRIDE slots (the Makefile compiles this file
// once per stride, so the instantiations build in parallel).
#include "epilogue.hpp"
#include "tile_launch.hpp"

namespace ebb {

// LDS of a gradient workgroup or of an epilogue workgroup riding in its kernel
template <int MODE>
union GradShared {
    GradLds<MODE> g;
    struct {
        double staging[2 * FORCE_LDS];
        EpiLds e;
    } x;
};

// The first epiPad workgroups (dispatched first) carry the epilogue of the step before; the
// others are the cell blocks.  The epilogue used to be two launches after each step, both bound
// by the latency of a few dependent round trips: 14 us of a 74 us step on 8,192 cells, 20 us of
// 250 us on 299,266; beside the gradients it costs nothing that the step waits for.
template <int S, int MODE, int MIX>
__global__ __launch_bounds__(BLK) void k_gradient(DevMesh m, PhysParams p, StageArgs a, DiagArgs d, uint32_t epiPad)
{
    __shared__ GradShared<MODE> L;
    if (blockIdx.x < epiPad) {
        if (blockIdx.x < d.nEpi) epilogueBody(d, blockIdx.x, L.x.e, L.x.staging);
        return;
    }
    const uint32_t b = blockIdx.x - epiPad, nb = gridDim.x - epiPad;
    gradientBody<S, MODE, MIX>(m, p, a, (a.order & 2) ? xcdBlockBack(b, nb) : xcdBlock(b, nb), L.g);
}

template <int S, int MODE, int MIX, int LANES>
__global__ __launch_bounds__(BLK) void k_gradient_split(DevMesh m, PhysParams p, StageArgs a, DiagArgs d, uint32_t epiPad)
{
    __shared__ GradShared<0> L;   // the epilogue's
    if (blockIdx.x < epiPad) {
        if (blockIdx.x < d.nEpi) epilogueBody(d, blockIdx.x, L.x.e, L.x.staging);
        return;
    }
    const uint32_t b = blockIdx.x - epiPad, nb = gridDim.x - epiPad;
    gradientSplitBody<S, MODE, MIX, LANES>(m, p, a, (a.order & 2) ? xcdBlockBack(b, nb) : xcdBlock(b, nb));
}

template <int S, int MODE, int MIX>
__global__ __launch_bounds__(BLK) void k_gradient_batch(const MemberArgs* __restrict__ mem, const uint2* __restrict__ items,
                                                        uint32_t parity, uint32_t stage, const uint2* __restrict__ epi,
                                                        uint32_t nEpi, uint32_t epiPad)
{
    __shared__ GradShared<MODE> L;
    if (blockIdx.x < epiPad) {
        if (blockIdx.x >= nEpi) return;
        const uint2 it = epi[blockIdx.x];
        const DiagArgs d = mem[it.x].d[parity ^ 1u ^ mem[it.x].parityFlip];   // scalar loads, before any store
        epilogueBody(d, it.y, L.x.e, L.x.staging);
        return;
    }
    const uint2 it = items[xcdBlock(blockIdx.x - epiPad, gridDim.x - epiPad)];
    const MemberArgs& M = mem[it.x];
    gradientBody<S, MODE, MIX>(M.m, M.p, M.st[parity ^ M.parityFlip][stage], it.y, L.g);
}

// Lanes per cell.  The LP limiter's simplex is most of its kernel and its four problems are serial in
// one lane: always four (Euler runs of 1,040 cells 1.87x faster, 10,414 1.73x, 42,496 1.44x, 540,000
// 1.15x).  The other limiters' lanes repeat the cell's ids and weights, which the shorter chain and
// the smaller register count outweigh until the chip is full several times over.  Runs of one / two /
// four lanes, us: FP64 8,192 cells 1873 / - / 1687, 32,400: 721 / 706 / 708, 42,496: 1358 / 1281 /
// 1299, 99,856: 971 / 961 / 1011, 299,266: 3202 / 3037 / - (its limited gradient kernel 16.4 / 13.9),
// 698,368: 6479 / 6300 / -, 1,048,576: 4551 / 4576 / -; mixed precision 32,400: 675 / 682 / 661,
// 81,900: 1552 / 1509 / 1553, 698,368: 4639 / 4527 / -, 1,048,576: 3351 / 3401 / -.
static int gradLanes(int mode, uint32_t cells) { return mode == 3 || cells <= 40000 ? 4 : cells <= 800000 ? 2 : 1; }

template <int S, int LANES>
static void gradSplit(int mode, const DevMesh& m, const PhysParams& p, const StageArgs& a, const DiagArgs& d,
                      uint32_t pad, hipStream_t st)
{
    const dim3 g((m.N + BLK / LANES - 1) / (BLK / LANES) + pad), b(BLK);
#define EBB_SPLIT(MODE, MIX) \
    hipLaunchKernelGGL((k_gradient_split<S, MODE, MIX, LANES>), g, b, 0, st, m, p, a, d, pad); break
    switch (mode + 8 * p.mixed) {
    case 1: EBB_SPLIT(1, 0);
    case 2: EBB_SPLIT(2, 0);
    case 4: EBB_SPLIT(4, 0);
    case 9: EBB_SPLIT(1, 1);
    case 10: EBB_SPLIT(2, 1);
    case 12: EBB_SPLIT(4, 1);
    default:
        if constexpr (LANES == 4) EBB_SPLIT(3, 0);
    }
#undef EBB_SPLIT
}

template <int S>
void gradS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const DiagArgs& d, hipStream_t st)
{
    const uint32_t pad = epiPadding(d.nEpi);
    const uint32_t g = (m.N + BLK - 1) / BLK + pad;
    if (g == 0) return;
    const int mode = p.order == 1 ? 0 : (!(p.limited && a.limit) ? 1 : (p.venkat ? 4 : (p.lpThresh > 0 ? 3 : 2)));
    const int lanes = mode ? gradLanes(mode, m.N) : 1;
    if (lanes == 4) { gradSplit<S, 4>(mode, m, p, a, d, pad, st); return; }
    if (lanes == 2) { gradSplit<S, 2>(mode, m, p, a, d, pad, st); return; }
#define EBB_GRAD(MODE, MIX) hipLaunchKernelGGL((k_gradient<S, MODE, MIX>), dim3(g), dim3(BLK), 0, st, m, p, a, d, pad); break
    if (p.mixed) {
        switch (mode) {
        case 0: EBB_GRAD(0, 1);
        case 1: EBB_GRAD(1, 1);
        case 4: EBB_GRAD(4, 1);
        default: EBB_GRAD(2, 1);
        }
        return;
    }
    switch (mode) {
    case 0: EBB_GRAD(0, 0);
    case 1: EBB_GRAD(1, 0);
    case 4: EBB_GRAD(4, 0);
    default: EBB_GRAD(2, 0);
    }
#undef EBB_GRAD
}

template <int S, int MIX>
void gradBatchS(int mode, const MemberArgs* mem, const uint2* items, uint32_t n, uint32_t par, uint32_t st,
                       const uint2* epi, uint32_t nEpi, hipStream_t s)
{
    const uint32_t pad = epiPadding(nEpi);
    const dim3 g(n + pad), b(BLK);
    switch (mode) {
    case 0: hipLaunchKernelGGL((k_gradient_batch<S, 0, MIX>), g, b, 0, s, mem, items, par, st, epi, nEpi, pad); break;
    case 1: hipLaunchKernelGGL((k_gradient_batch<S, 1, MIX>), g, b, 0, s, mem, items, par, st, epi, nEpi, pad); break;
    case 4: hipLaunchKernelGGL((k_gradient_batch<S, 4, MIX>), g, b, 0, s, mem, items, par, st, epi, nEpi, pad); break;
    default: hipLaunchKernelGGL((k_gradient_batch<S, 2, MIX>), g, b, 0, s, mem, items, par, st, epi, nEpi, pad); break;
    }
}

template void gradS<STRIDE>(const DevMesh&, const PhysParams&, const StageArgs&, const DiagArgs&, hipStream_t);
template void gradBatchS<STRIDE, 0>(int, const MemberArgs*, const uint2*, uint32_t, uint32_t, uint32_t, const uint2*,
                                    uint32_t, hipStream_t);
template void gradBatchS<STRIDE, 1>(int, const MemberArgs*, const uint2*, uint32_t, uint32_t, uint32_t, const uint2*,
                                    uint32_t, hipStream_t);

}  // namespace ebb
