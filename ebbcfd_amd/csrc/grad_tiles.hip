// The gradient-tile stage kernels (extensions.stagePath = "gradTiles") for cells of STRIDE slots
// (compiled once per stride).
#include "epilogue.hpp"
#include "face_tiles.hpp"
#include "tile_launch.hpp"

namespace ebb {

// ---------------------------------------------------------------- gradient tiles
// A stage in two launches that keeps most gradient and limiter rows on chip.
//   k_border_grad  per ring cell (a cell across a face of some other tile): its gradient
//                  and limiter rows to HBM; it also carries the gradient kernel's other
//                  duties (the epilogue of the step before, a call's first scalars);
//   k_grad_tile    per tile: its own cells' ghosts, gradients and limiters into LDS, the
//                  ring cells' rows copied in from the border kernel's output, then every
//                  face of the tile and the cells' update as in k_face_tile.
// Gradients come from cellGradient and faces from interiorFace/boundaryFace, the code of
// the split kernels, on the same inputs, so the stage's results are bit-identical to the
// other paths.  A boundary face takes its ghost state from its owner's row (ghostState)
// instead of reading back the row this launch's gradient phase wrote.

// LDS row of one cell: gradient (x,y per variable) then the 4 scalar limiters
constexpr int GROW = 12;

// One workgroup of the border kernel on border block `bid` of its mesh (the solo and the
// batched kernels run this same code); block 0 also sets what a call starts with (stageBegin).
template <int S, int MODE, int MIX>
DEV void borderGradBody(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, uint32_t bid)
{
    using R = RealOf<MIX>;
    if (!stageRuns(a)) return;
    if (bid == 0 && threadIdx.x == 0) stageBegin(a);
    const uint32_t k = bid * BLK + threadIdx.x;
    if (k >= t.nBorder) return;
    const uint32_t i = t.border[k];
    R g[4][2], lx[4], ly[4];
    cellGradient<S, MODE, MIX>(m, p, a, i, m.nbr + size_t(i) * S, false, g, lx, ly);   // the owning tile stores the ghosts
    if constexpr (MIX == 1) {
        float4* gd = reinterpret_cast<float4*>(a.grad32 + size_t(i) * 8);
        gd[0] = make_float4(g[0][0], g[0][1], g[1][0], g[1][1]);
        gd[1] = make_float4(g[2][0], g[2][1], g[3][0], g[3][1]);
        if (MODE != 1) *reinterpret_cast<float4*>(a.lim32 + size_t(i) * 4) = make_float4(lx[0], lx[1], lx[2], lx[3]);
    } else {
        double4* gd = reinterpret_cast<double4*>(a.grad + size_t(i) * 8);
        gd[0] = make_double4(g[0][0], g[0][1], g[1][0], g[1][1]);
        gd[1] = make_double4(g[2][0], g[2][1], g[3][0], g[3][1]);
        if (MODE != 1) *reinterpret_cast<double4*>(a.lim + size_t(i) * 4) = make_double4(lx[0], lx[1], lx[2], lx[3]);
    }
}

// The first epiPad workgroups carry the epilogue of the step before (as the gradient kernel's);
// the others are border blocks.
template <int S, int MODE, int MIX>
__global__ __launch_bounds__(BLK) void k_border_grad(DevMesh m, PhysParams p, StageArgs a, FaceTileArgs t, DiagArgs d,
                                                     uint32_t epiPad)
{
    if (blockIdx.x < epiPad) {
        __shared__ double staging[2 * FORCE_LDS];
        __shared__ EpiLds E;
        if (blockIdx.x < d.nEpi) epilogueBody(d, blockIdx.x, E, staging);
        return;
    }
    borderGradBody<S, MODE, MIX>(m, p, a, t, xcdBlock(blockIdx.x - epiPad, gridDim.x - epiPad));
}

// One workgroup of the gradient-tile kernel on tile `tile`.  MODE 1: an unlimited stage
// (no limiter rows; the faces take unit limiters); 2: the scalar limiter; 4: Venkatakrishnan.
template <int S, int FLUX, int VISC, int MODE, int MIX>
DEV void gradTileBody(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t,
                      uint32_t tile, uint32_t pslot, double* lds)
{
    using R = RealOf<MIX>;
    constexpr int LP = MODE == 1 ? 2 : 0;
    const FaceSrc<MIX> src{a};
    const uint32_t tid = threadIdx.x;
    // first loads beside the descriptor's (fixed strides; lanes past the counts read padding)
    const uint32_t gi0 = t.ids[size_t(tile) * t.cellStride + tid];
    uint4 rNext = t.fref[size_t(tile) * t.faceStride + tid];
    uint32_t sNext = t.fslot[size_t(tile) * t.faceStride + tid];
    const uint4 d = t.desc[tile];
    const uint32_t nH = t.nHalo[tile];
    if (!fluxRuns(a, pslot == 0 && tid == 0)) return;
    const uint32_t nC = d.x, nF = d.y;
    R* gl = reinterpret_cast<R*>(lds);
    const FaceLds<MIX> fl(lds + t.glDoubles, t.faceStride + 1);
    // the ring's rows first: their loads are in flight while the own gradients compute
    for (uint32_t h = tid; h < nH; h += BLK) {
        const uint32_t y = t.halo[size_t(tile) * t.haloStride + h];
        R gg[8];
        src.grad(y, gg);
        R* row = gl + GROW * (nC + h);
#pragma unroll
        for (int c = 0; c < 8; c++) row[c] = gg[c];
        if (MODE != 1) {
            R lx[4], ly[4];
            src.template lim<0>(y, lx, ly);
#pragma unroll
            for (int c = 0; c < 4; c++) row[8 + c] = lx[c];
        }
    }
    // own cells (ghosts stored: this tile owns them), neighbour ids from the tile's copy of
    // their rows, whose addresses do not wait for the cell ids
    for (uint32_t k = tid; k < nC; k += BLK) {
        const uint32_t i = k == tid ? gi0 : t.ids[d.z + k];
        R g[4][2], lx[4], ly[4];
        cellGradient<S, MODE, MIX>(m, p, a, i, t.nbrT + size_t(d.z + k) * S, true, g, lx, ly);
        R* row = gl + GROW * k;
#pragma unroll
        for (int c = 0; c < 4; c++) { row[2 * c] = g[c][0]; row[2 * c + 1] = g[c][1]; }
        if (MODE != 1) {
#pragma unroll
            for (int c = 0; c < 4; c++) row[8 + c] = lx[c];
        }
    }
    // the first cell rounds' ids for the cell phase
    const uint32_t giNext = gi0;
    const uint32_t giNext2 = t.ids[size_t(tile) * t.cellStride + tid + BLK];
    ldsBarrier();
    // face phase: as k_face_tile, with the rows from LDS
    for (uint32_t k = tid; k < nF; k += BLK) {
        const uint4 r = rNext;   // cell a, cell b, node 0, node 1
        const uint32_t sl = sNext;
        if (k + BLK < nF) { rNext = t.fref[d.w + k + BLK]; sNext = t.fslot[d.w + k + BLK]; }
        const bool interior = r.y < m.N;
        const double2 p0 = m.node[r.z], p1 = m.node[r.w];
        R qa[4], qb[4];
        src.q(r.x, qa);
        src.q(r.y, qb);   // a boundary face: the ghost row, whose TempPresInflow components carry over
        const double2 ca = m.cen[r.x], cb = m.cen[r.y];
        const R* ra = gl + GROW * (sl & 0xffffu);
        const R* rb = gl + GROW * (sl >> 16);
        R ga[8], gb[8], lxa[4], lya[4], lxb[4], lyb[4];
#pragma unroll
        for (int c = 0; c < 8; c++) { ga[c] = ra[c]; gb[c] = rb[c]; }
#pragma unroll
        for (int c = 0; c < 4; c++) {
            lxa[c] = lya[c] = MODE == 1 ? R(1.0) : ra[8 + c];
            lxb[c] = lyb[c] = MODE == 1 ? R(1.0) : rb[8 + c];
        }
        double2 n, mid;
        double len;
        edgeGeometry(interior, p0, p1, n, mid, len);
        R qL[4], qR[4], Fr[4], sMr;
        bool isB = false;
        uint32_t b = 0;
        if (interior) {
            interiorFace<FLUX, VISC, 2, LP, R>(qa, ga, lxa, lya, ca, qb, gb, lxb, lyb, cb, n, mid, p, qL, qR, Fr, sMr);
        } else {
            isB = true;
            b = r.y - m.N;
            const BFace& bf = m.bface[b];
            R qg[4];
            ghostState<R>(bf, qa, qg, qb);   // a failure was recorded by the gradient phase
            boundaryFace<FLUX, VISC, 2, LP, R>(qa, ga, lxa, lya, ca, qg, bf, n, mid, p, qL, qR, Fr, sMr);
        }
        const double F[4] = {double(Fr[0]), double(Fr[1]), double(Fr[2]), double(Fr[3])}, sMax = double(sMr);
        if (isB) {
            const uint32_t f = m.Fi + b;
            *reinterpret_cast<double4*>(a.lenF + size_t(f) * 4) =
                make_double4(len * F[0], len * F[1], len * F[2], len * F[3]);
            a.lenS[f] = len * sMax;
        }
        if (a.recordErrors && (isnan(F[0]) || isnan(F[1]) || isnan(F[2]) || isnan(F[3])))
            atomicMin(&a.sc->errEdge,
                      (uint64_t(a.stageId) << 32) | (isB ? uint64_t(b) : uint64_t(m.Fb) + t.fid[d.w + k]));
        if constexpr (MIX == 1) fl.put(k, len, Fr, sMr);
        else fl.put(k, len, F, sMax);
    }
    fl.zero(nF, tid);   // padding face
    tileCellPhase<S, MIX>(m, p, a, t, d, pslot, fl, giNext, giNext2);
}

// FP64: at most 168 VGPRs, three waves per SIMD (the LDS of three workgroups fits a CU)
template <int S, int FLUX, int VISC, int MODE, int MIX>
__global__ __launch_bounds__(BLK, 3) void k_grad_tile(DevMesh m, PhysParams p, StageArgs a, FaceTileArgs t)
{
    extern __shared__ double glds[];
    gradTileBody<S, FLUX, VISC, MODE, MIX>(m, p, a, t, xcdBlock(blockIdx.x, gridDim.x), blockIdx.x, glds);
}

template <int S, int FLUX, int VISC, int MIX>
static void gradTileM(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, int mode,
                      int parts, const DiagArgs* epi, hipStream_t st)
{
    const dim3 g(t.nTiles), b(BLK);
    const uint32_t nb = (t.nBorder + BLK - 1) / BLK;
    const DiagArgs d = epi ? *epi : DiagArgs{};
    const uint32_t pad = epiPadding(d.nEpi);
    const dim3 gb((nb ? nb : 1u) + pad);   // at least one workgroup: the Rmax reset
    const bool border = parts & 1, tiles = parts & 2;
    switch (mode) {
    case 1:
        if (border) hipLaunchKernelGGL((k_border_grad<S, 1, MIX>), gb, b, 0, st, m, p, a, t, d, pad);
        if (tiles) hipLaunchKernelGGL((k_grad_tile<S, FLUX, VISC, 1, MIX>), g, b, t.ldsBytes, st, m, p, a, t);
        break;
    case 4:
        if (border) hipLaunchKernelGGL((k_border_grad<S, 4, MIX>), gb, b, 0, st, m, p, a, t, d, pad);
        if (tiles) hipLaunchKernelGGL((k_grad_tile<S, FLUX, VISC, 4, MIX>), g, b, t.ldsBytes, st, m, p, a, t);
        break;
    default:
        if (border) hipLaunchKernelGGL((k_border_grad<S, 2, MIX>), gb, b, 0, st, m, p, a, t, d, pad);
        if (tiles) hipLaunchKernelGGL((k_grad_tile<S, FLUX, VISC, 2, MIX>), g, b, t.ldsBytes, st, m, p, a, t);
        break;
    }
}

template <int S>
void gradTileS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, int mode,
                      int parts, const DiagArgs* epi, hipStream_t st)
{
#define EBB_GT(F, V)                                                      \
    do {                                                                  \
        if (p.mixed) gradTileM<S, F, V, 1>(m, p, a, t, mode, parts, epi, st);  \
        else gradTileM<S, F, V, 0>(m, p, a, t, mode, parts, epi, st);          \
    } while (0)
    if (p.flux == 1) {
        if (p.viscous) EBB_GT(1, 1); else EBB_GT(1, 0);
    } else {
        if (p.viscous) EBB_GT(0, 1); else EBB_GT(0, 0);
    }
#undef EBB_GT
}

template <int S, int MODE, int MIX>
__global__ __launch_bounds__(BLK) void k_border_grad_batch(const MemberArgs* __restrict__ mem,
                                                           const uint2* __restrict__ items, uint32_t parity, uint32_t stage,
                                                           const uint2* __restrict__ epi, uint32_t nEpi, uint32_t epiPad)
{
    if (blockIdx.x < epiPad) {
        __shared__ double staging[2 * FORCE_LDS];
        __shared__ EpiLds E;
        if (blockIdx.x >= nEpi) return;
        const uint2 it = epi[blockIdx.x];
        const DiagArgs d = mem[it.x].d[parity ^ 1u ^ mem[it.x].parityFlip];   // scalar loads, before any store
        epilogueBody(d, it.y, E, staging);
        return;
    }
    const uint2 it = items[xcdBlock(blockIdx.x - epiPad, gridDim.x - epiPad)];
    const MemberArgs& M = mem[it.x];
    borderGradBody<S, MODE, MIX>(M.m, M.p, M.st[parity ^ M.parityFlip][stage], M.t, it.y);
}

template <int S, int FLUX, int VISC, int MODE, int MIX>
__global__ __launch_bounds__(BLK, 3) void k_grad_tile_batch(const MemberArgs* __restrict__ mem,
                                                         const uint2* __restrict__ items, uint32_t parity, uint32_t stage)
{
    extern __shared__ double glds[];
    const uint2 it = items[xcdBlock(blockIdx.x, gridDim.x)];
    const MemberArgs& M = mem[it.x];
    gradTileBody<S, FLUX, VISC, MODE, MIX>(M.m, M.p, M.st[parity ^ M.parityFlip][stage], M.t, it.y, it.y, glds);
}

template <int S, int MIX>
void borderBatchS(int mode, const MemberArgs* mem, const uint2* items, uint32_t n, uint32_t par, uint32_t st,
                  const uint2* epi, uint32_t nEpi, hipStream_t s)
{
    const uint32_t pad = epiPadding(nEpi);
    const dim3 g(n + pad), b(BLK);
    switch (mode) {
    case 1: hipLaunchKernelGGL((k_border_grad_batch<S, 1, MIX>), g, b, 0, s, mem, items, par, st, epi, nEpi, pad); break;
    case 4: hipLaunchKernelGGL((k_border_grad_batch<S, 4, MIX>), g, b, 0, s, mem, items, par, st, epi, nEpi, pad); break;
    default: hipLaunchKernelGGL((k_border_grad_batch<S, 2, MIX>), g, b, 0, s, mem, items, par, st, epi, nEpi, pad); break;
    }
}

template <int S, int FLUX, int VISC, int MIX>
static void gradTileBatchM(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items, uint32_t n,
                           uint32_t lds, uint32_t par, uint32_t stg, hipStream_t s)
{
    const dim3 g(n), b(BLK);
    const int mode = !(gs.limited && limitStage) ? 1 : (gs.venkat ? 4 : 2);
    if (mode == 1) hipLaunchKernelGGL((k_grad_tile_batch<S, FLUX, VISC, 1, MIX>), g, b, lds, s, mem, items, par, stg);
    else if (mode == 4) hipLaunchKernelGGL((k_grad_tile_batch<S, FLUX, VISC, 4, MIX>), g, b, lds, s, mem, items, par, stg);
    else hipLaunchKernelGGL((k_grad_tile_batch<S, FLUX, VISC, 2, MIX>), g, b, lds, s, mem, items, par, stg);
}

template <int S, int MIX>
void gradTileBatchS(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items, uint32_t n,
                    uint32_t lds, uint32_t par, uint32_t stg, hipStream_t s)
{
    if (gs.flux == 1) {
        if (gs.viscous) gradTileBatchM<S, 1, 1, MIX>(gs, limitStage, mem, items, n, lds, par, stg, s);
        else gradTileBatchM<S, 1, 0, MIX>(gs, limitStage, mem, items, n, lds, par, stg, s);
    } else {
        if (gs.viscous) gradTileBatchM<S, 0, 1, MIX>(gs, limitStage, mem, items, n, lds, par, stg, s);
        else gradTileBatchM<S, 0, 0, MIX>(gs, limitStage, mem, items, n, lds, par, stg, s);
    }
}

template void gradTileS<STRIDE>(const DevMesh&, const PhysParams&, const StageArgs&, const FaceTileArgs&, int, int,
                                const DiagArgs*, hipStream_t);
template void borderBatchS<STRIDE, 0>(int, const MemberArgs*, const uint2*, uint32_t, uint32_t, uint32_t, const uint2*,
                                      uint32_t, hipStream_t);
template void borderBatchS<STRIDE, 1>(int, const MemberArgs*, const uint2*, uint32_t, uint32_t, uint32_t, const uint2*,
                                      uint32_t, hipStream_t);
template void gradTileBatchS<STRIDE, 0>(const GroupShape&, int, const MemberArgs*, const uint2*, uint32_t, uint32_t,
                                        uint32_t, uint32_t, hipStream_t);
template void gradTileBatchS<STRIDE, 1>(const GroupShape&, int, const MemberArgs*, const uint2*, uint32_t, uint32_t,
                                        uint32_t, uint32_t, hipStream_t);

}  // namespace ebb
