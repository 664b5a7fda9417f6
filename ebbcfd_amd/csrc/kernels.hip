// HIP kernels for the explicit residual-and-update loop, FP64, gfx950.
//
// One residual evaluation (source/solve.d:322-1122) on the split path is three launches:
//   k_gradient  per interior cell: ghost states of its boundary faces
//               (solve.d:520-689), LSQ gradient, min/max bounds and the scalar
//               limiter at neighbour centroids (solve.d:324-403), LP vector
//               limiter (solve.d:404-497);
//   k_faces     per face, each computed once: reconstruction at the midpoint with
//               the p<0 fallback (solve.d:283-319, 970-1011), Roe/Rusanov flux
//               (flux.d:66-303), viscous flux (flux.d:28-64), boundary fluxes
//               (solve.d:769-968); stores len*flux and len*sMax per face;
//   k_update    per interior cell: gathers its faces in the cell's own edge
//               order with the owner sign (solve.d:1082-1118), CFL time step
//               and Rmax (one pair of partials per block, reduced by the step's
//               epilogue or the call's last kernel; exact because min/max are order
//               independent), the MMS source (app/ms.d:131-141) and the integrator
//               stage update (source/integrators.d:22-270) fused in.
// The default path is two: k_gradient and k_face_tile, which does the work of the other two
// for a tile of cells with the faces in LDS.
// No atomics touch the residual: each cell sums its own faces in a fixed order,
// so results are deterministic and bit-identical to the edge-loop form.
// Built with -ffp-contract=off: every product and sum rounds as written.
// This file holds the split-path and step epilogue kernels and the launchers; the gradient
// kernels are in gradient.hip, the tile kernels in face_tiles.hpp, grad_tiles.hip and fused.hip.
#include "epilogue.hpp"
#include "tile_launch.hpp"

namespace ebb {

template <int FLUX, int VISC, int ORDER, int LP, int STORE, int MIX>
__global__ __launch_bounds__(BLK) void k_faces(DevMesh m, PhysParams p, StageArgs a, uint32_t nbi)
{
    using R = typename std::conditional<MIX == 1, float, double>::type;
    if (!fluxRuns(a, blockIdx.x == 0 && threadIdx.x == 0)) return;
    const FaceSrc<MIX> src{a};
    R qL[4], qR[4], F[4], sMax;
    uint32_t f;
    double len;
    uint64_t errKey;
    if (blockIdx.x < nbi) {
        f = xcdBlock(blockIdx.x, nbi) * BLK + threadIdx.x;
        if (f >= m.Fi) return;
        const uint2 c = m.fcell[f];
        len = m.flen[f];
        R qa[4], qb[4], ga[8], gb[8], lxa[4], lya[4], lxb[4], lyb[4];
        src.q(c.x, qa);
        src.q(c.y, qb);
        if (ORDER > 1 || VISC) { src.grad(c.x, ga); src.grad(c.y, gb); }
        double2 ca = make_double2(0, 0), cb = make_double2(0, 0), mid = make_double2(0, 0);
        if (ORDER > 1) {
            src.template lim<LP>(c.x, lxa, lya);
            src.template lim<LP>(c.y, lxb, lyb);
            ca = m.cen[c.x]; cb = m.cen[c.y]; mid = m.fmid[f];
        }
        interiorFace<FLUX, VISC, ORDER, LP, R>(qa, ga, lxa, lya, ca, qb, gb, lxb, lyb, cb, m.fn[f], mid, p, qL, qR, F,
                                              sMax);
        errKey = uint64_t(m.Fb) + f;   // boundary edges are checked first in the reference
    } else {
        const uint32_t b = (blockIdx.x - nbi) * BLK + threadIdx.x;
        if (b >= m.Fb) return;
        f = m.Fi + b;
        const uint32_t o = m.fcell[f].x;
        len = m.flen[f];
        R qo[4], qg[4], gO[8], lx[4], ly[4];
        src.q(o, qo);
        src.q(m.N + b, qg);
        if (ORDER > 1 || VISC) src.grad(o, gO);
        double2 co = make_double2(0, 0), mid = make_double2(0, 0);
        if (ORDER > 1) {
            src.template lim<LP>(o, lx, ly);
            co = m.cen[o]; mid = m.fmid[f];
        }
        boundaryFace<FLUX, VISC, ORDER, LP, R>(qo, gO, lx, ly, co, qg, m.bface[b], m.fn[f], mid, p, qL, qR, F, sMax);
        errKey = b;
    }
    if (a.recordErrors && (isnan(F[0]) || isnan(F[1]) || isnan(F[2]) || isnan(F[3])))
        atomicMin(&a.sc->errEdge, (uint64_t(a.stageId) << 32) | errKey);
    *reinterpret_cast<double4*>(a.lenF + size_t(f) * 4) =
        make_double4(len * double(F[0]), len * double(F[1]), len * double(F[2]), len * double(F[3]));
    a.lenS[f] = len * double(sMax);
    if (STORE) {
        a.estate[2 * f] = make_double4(qL[0], qL[1], qL[2], qL[3]);
        a.estate[2 * f + 1] = make_double4(qR[0], qR[1], qR[2], qR[3]);
    }
}

template <int S, int KIND>
__global__ __launch_bounds__(BLK) void k_update(DevMesh m, PhysParams p, StageArgs a)
{
    if (a.checkActive && !a.sc->active) return;
    const uint32_t i = xcdBlock(blockIdx.x, gridDim.x) * BLK + threadIdx.x;
    double dtCand = INFINITY, rCand = 0.0;
    double qNew[4] = {0, 0, 0, 0}, qOld[4] = {0, 0, 0, 0};
    if (i < m.N) {
        double r[4] = {0.0, 0.0, 0.0, 0.0};
        double sAve = 0;
#pragma unroll
        for (int j = 0; j < S; j++) {
            const uint32_t fe = m.cface[i * S + j];
            const uint32_t f = fe & 0x7fffffffu;
            const double4 lf = *reinterpret_cast<const double4*>(a.lenF + size_t(f) * 4);
            if (fe >> 31) { r[0] = r[0] - lf.x; r[1] = r[1] - lf.y; r[2] = r[2] - lf.z; r[3] = r[3] - lf.w; }
            else { r[0] = r[0] + lf.x; r[1] = r[1] + lf.y; r[2] = r[2] + lf.z; r[3] = r[3] + lf.w; }
            sAve += a.lenS[f];
        }
        cellStage<KIND>(m, p, a, i, r, sAve, nullptr, nullptr, dtCand, rCand, qNew, qOld);
    }
    if ((KIND == SK_EULER || KIND == SK_RK2_2 || KIND == SK_TVD_2 || KIND == SK_RK4_4) && a.rmsBlocks)
        rmsBlockLeaf(i < m.N, qNew, qOld, i < m.N ? m.refId[i] : 0u, a.rmsBlocks);
    blockPartial(dtCand, rCand, a.partial, blockIdx.x);
}

void launchFaceTiles(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, int S,
                     hipStream_t st)
{
    if (t.nTiles == 0) return;
    if (S == 3) faceTileS<3>(m, p, a, t, st);
    else if (S == 4) faceTileS<4>(m, p, a, t, st);
    else faceTileS<6>(m, p, a, t, st);
    if (!a.deferReduce) launchReduceStage(a.partial, t.nTiles, a.sc, a.checkActive, st);
}

void launchGradTiles(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, int S,
                     hipStream_t st, int parts, const DiagArgs* epi)
{
    if (t.nTiles == 0) return;
    // order 2 and no LP vector limiter (the set-up keeps other configurations on face tiles)
    const int mode = !(p.limited && a.limit) ? 1 : (p.venkat ? 4 : 2);
    if (S == 3) gradTileS<3>(m, p, a, t, mode, parts, epi, st);
    else if (S == 4) gradTileS<4>(m, p, a, t, mode, parts, epi, st);
    else gradTileS<6>(m, p, a, t, mode, parts, epi, st);
    if ((parts & 2) && !a.deferReduce)
        launchReduceStage(a.partial, t.nTiles, a.sc, a.checkActive, st);
}

// newDt = min over the stage's workgroup partials; Rmax = max with the step's running value
__global__ __launch_bounds__(1024) void k_reduce_stage(const double* __restrict__ partial, uint32_t n,
                                                       DevScalars* sc, int checkActive)
{
    if (checkActive && !sc->active) return;
    __shared__ double sMin[16], sMax_[16];
    double a0 = INFINITY, b0 = 0.0;
    for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
        a0 = fmin(a0, partial[2 * k]);
        b0 = fmax(b0, partial[2 * k + 1]);
    }
    a0 = warpMin(a0);
    b0 = warpMax(b0);
    const int w = threadIdx.x / 64, l = threadIdx.x % 64;
    if (l == 0) { sMin[w] = a0; sMax_[w] = b0; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t k = 1; k < blockDim.x / 64; k++) { a0 = fmin(a0, sMin[k]); b0 = fmax(b0, sMax_[k]); }
        a0 = fmin(a0, sMin[0]);
        b0 = fmax(b0, sMax_[0]);
        sc->newDtBits = (unsigned long long)__double_as_longlong(a0);
        const double prev = __longlong_as_double((long long)sc->rmaxBits);
        if (b0 > prev) sc->rmaxBits = (unsigned long long)__double_as_longlong(b0);
    }
}

void launchReduceStage(const double* partial, uint32_t n, DevScalars* sc, int checkActive, hipStream_t st)
{
    hipLaunchKernelGGL(k_reduce_stage, dim3(1), dim3(1024), 0, st, partial, n, sc, checkActive);
}

// ---------------------------------------------------------------- diagnostics
// Leaf sums of the RMS residuals (rmsBlockLeaf) from the states, in the reference's numbering, for
// the paths whose last stage does not leave them: 16 consecutive lanes own one block.
__global__ __launch_bounds__(BLK) void k_rms_leaves(DiagArgs d, double* blockSums)
{
    if (!d.sc->active) return;
    const uint32_t e = blockIdx.x * BLK + threadIdx.x;
    const bool have = e < d.N;
    double qa[4] = {0, 0, 0, 0}, qb[4] = {0, 0, 0, 0};
    if (have) {
        const uint32_t dv = d.perm ? d.perm[e] : e;
        ld4(d.qnew, dv, qa);
        ld4(d.qold, dv, qb);
    }
    rmsBlockLeaf(have, qa, qb, e, blockSums);
}

__global__ __launch_bounds__(EPT) void k_epilogue(DiagArgs d)
{
    __shared__ double staging[2 * FORCE_LDS];
    __shared__ EpiLds E;
    epilogueBody(d, blockIdx.x, E, staging);
}

__global__ __launch_bounds__(BLK) void k_restore_ghosts(double4* q, float4* q32, const double4* save, uint32_t n)
{
    const uint32_t i = blockIdx.x * BLK + threadIdx.x;
    if (i >= n) return;
    const double4 v = save[i];
    q[i] = v;
    if (q32) q32[i] = make_float4(float(v.x), float(v.y), float(v.z), float(v.w));
}

void launchRestoreGhosts(double4* q, float4* q32, const double4* save, uint32_t n, hipStream_t st)
{
    if (n) hipLaunchKernelGGL(k_restore_ghosts, dim3((n + BLK - 1) / BLK), dim3(BLK), 0, st, q, q32, save, n);
}

// FP32 shadow of a state array (mixed path): after set-up, an upload or a load
__global__ __launch_bounds__(BLK) void k_shadow(const double4* __restrict__ q, float4* __restrict__ q32, uint32_t n)
{
    const uint32_t i = blockIdx.x * BLK + threadIdx.x;
    if (i >= n) return;
    const double4 v = q[i];
    q32[i] = make_float4(float(v.x), float(v.y), float(v.z), float(v.w));
}

void launchShadow(const double4* q, float4* q32, uint32_t n, hipStream_t st)
{
    if (n) hipLaunchKernelGGL(k_shadow, dim3((n + BLK - 1) / BLK), dim3(BLK), 0, st, q, q32, n);
}

// Rows of 4 doubles into another numbering: out[i] = in[src[i]], a lane per half row
__global__ __launch_bounds__(BLK) void k_permute_rows(const double2* __restrict__ in, double2* __restrict__ out,
                                                      const uint32_t* __restrict__ src, uint32_t n)
{
    const uint64_t g = uint64_t(blockIdx.x) * BLK + threadIdx.x;
    const uint32_t i = uint32_t(g >> 1), h = uint32_t(g & 1u);
    if (i < n) out[g] = in[size_t(src[i]) * 2 + h];
}

void launchPermuteRows(const double4* in, double4* out, const uint32_t* src, uint32_t n, hipStream_t st)
{
    if (n)
        hipLaunchKernelGGL(k_permute_rows, dim3((2 * uint64_t(n) + BLK - 1) / BLK), dim3(BLK), 0, st,
                           reinterpret_cast<const double2*>(in), reinterpret_cast<double2*>(out), src, n);
}

__global__ void k_init_scalars(DevScalars* sc, double dt, double t, double CFL)
{
    sc->newDtBits = 0x7FF0000000000000ull;
    sc->rmaxBits = 0;
    sc->errEdge = ~0ull;
    sc->errCell = ~0ull;
    sc->errBC = ~0ull;
    sc->dt = dt;
    sc->t = t;
    sc->CFL = CFL;
    sc->residLast = INFINITY;
    sc->incIters = 0;
    sc->steps = 0;
    sc->active = 1;
    sc->specActive = 1;
    sc->ticket = 0;
    sc->converged = 0;
    sc->rms0 = 0;
    sc->loopDt = 0;
    for (int v = 0; v < 4; v++) sc->rms[v] = 0;
    sc->force[0] = sc->force[1] = 0;
    sc->fsum[0] = sc->fsum[1] = 0;
    sc->stageSum[0] = sc->stageSum[1] = 0;
}

__global__ void k_begin_call(DevScalars* sc, unsigned long long rmaxBits, double dt, int setDt)
{
    sc->rmaxBits = rmaxBits;
    sc->errEdge = ~0ull;
    sc->errCell = ~0ull;
    sc->errBC = ~0ull;
    if (setDt) {
        sc->loopDt = sc->dt;
        sc->dt = dt;
    }
}

// The end of a call: newDt of its last stage and Rmax of all from their partials (nPart pairs per
// stage), the run loop's dt put back, and the scalars straight into the host's page-locked copy.  A
// reduction per stage, a kernel for dt and a copy of the scalars were three to six dependent launches.
__global__ __launch_bounds__(1024) void k_finish_call(const double* __restrict__ partial, uint32_t nPart, uint32_t nStages,
                                                      DevScalars* sc, int putDt, DevScalars* host)
{
    __shared__ double sMin[16], sMax_[16];
    __shared__ DevScalars out;
    double a0 = INFINITY, b0 = 0.0;
    const uint32_t n = nStages * nPart, lastStage = n - nPart;
    for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
        const double2 v = reinterpret_cast<const double2*>(partial)[k];
        if (k >= lastStage) a0 = fmin(a0, v.x);
        b0 = fmax(b0, v.y);
    }
    a0 = warpMin(a0);
    b0 = warpMax(b0);
    const int w = threadIdx.x / 64, l = threadIdx.x % 64;
    if (l == 0) { sMin[w] = a0; sMax_[w] = b0; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t k = 0; k < blockDim.x / 64; k++) { a0 = fmin(a0, sMin[k]); b0 = fmax(b0, sMax_[k]); }
        DevScalars v = *sc;
        v.newDtBits = (unsigned long long)__double_as_longlong(a0);
        if (b0 > __longlong_as_double((long long)v.rmaxBits)) v.rmaxBits = (unsigned long long)__double_as_longlong(b0);
        if (putDt) v.dt = v.loopDt;
        sc->newDtBits = v.newDtBits;
        sc->rmaxBits = v.rmaxBits;
        sc->dt = v.dt;
        out = v;
    }
    __syncthreads();
    static_assert(sizeof(DevScalars) % 8 == 0 && sizeof(DevScalars) / 8 <= 1024, "copied as words by one workgroup");
    if (threadIdx.x < sizeof(DevScalars) / 8)
        reinterpret_cast<unsigned long long*>(host)[threadIdx.x] =
            reinterpret_cast<const unsigned long long*>(&out)[threadIdx.x];
}

// ---------------------------------------------------------------- launchers
static uint32_t nblk(uint64_t n) { return uint32_t((n + BLK - 1) / BLK); }

void launchGradient(const DevMesh& m, const PhysParams& p, const StageArgs& a, int S, hipStream_t st, const DiagArgs* epi)
{
    const DiagArgs d = epi ? *epi : DiagArgs{};
    if (S == 3) gradS<3>(m, p, a, d, st);
    else if (S == 4) gradS<4>(m, p, a, d, st);
    else gradS<6>(m, p, a, d, st);
}

template <int FLUX, int VISC, int ORDER, int LP, int MIX>
static void facesT(const DevMesh& m, const PhysParams& p, const StageArgs& a, hipStream_t st)
{
    const uint32_t nbi = nblk(m.Fi), nbb = nblk(m.Fb);
    if (nbi + nbb == 0) return;
    if (a.estate)
        hipLaunchKernelGGL((k_faces<FLUX, VISC, ORDER, LP, 1, MIX>), dim3(nbi + nbb), dim3(BLK), 0, st, m, p, a, nbi);
    else
        hipLaunchKernelGGL((k_faces<FLUX, VISC, ORDER, LP, 0, MIX>), dim3(nbi + nbb), dim3(BLK), 0, st, m, p, a, nbi);
}

template <int FLUX, int VISC>
static void facesO(const DevMesh& m, const PhysParams& p, const StageArgs& a, hipStream_t st)
{
    const bool lp = p.order > 1 && p.limited && p.lpThresh > 0;
    if (p.mixed) {
        if (p.order == 1) facesT<FLUX, VISC, 1, 0, 1>(m, p, a, st);
        else if (!(p.limited && a.limit)) facesT<FLUX, VISC, 2, 2, 1>(m, p, a, st);
        else facesT<FLUX, VISC, 2, 0, 1>(m, p, a, st);
        return;
    }
    if (p.order == 1) facesT<FLUX, VISC, 1, 0, 0>(m, p, a, st);
    else if (!(p.limited && a.limit)) facesT<FLUX, VISC, 2, 2, 0>(m, p, a, st);
    else if (lp) facesT<FLUX, VISC, 2, 1, 0>(m, p, a, st);
    else facesT<FLUX, VISC, 2, 0, 0>(m, p, a, st);
}

void launchFaces(const DevMesh& m, const PhysParams& p, const StageArgs& a, hipStream_t st)
{
    if (p.flux == 1) {
        if (p.viscous) facesO<1, 1>(m, p, a, st); else facesO<1, 0>(m, p, a, st);
    } else {
        if (p.viscous) facesO<0, 1>(m, p, a, st); else facesO<0, 0>(m, p, a, st);
    }
}

template <int S>
static void updS(const DevMesh& m, const PhysParams& p, const StageArgs& a, hipStream_t st)
{
    const uint32_t g = nblk(m.N);
    if (g == 0) return;
#define UPD(K) case K: hipLaunchKernelGGL((k_update<S, K>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
    switch (a.kind) {
        UPD(SK_RESIDUAL) UPD(SK_EULER) UPD(SK_RK2_1) UPD(SK_RK2_2) UPD(SK_TVD_1) UPD(SK_TVD_2)
        UPD(SK_RK4_1) UPD(SK_RK4_2) UPD(SK_RK4_3) UPD(SK_RK4_4)
    }
#undef UPD
}

void launchUpdate(const DevMesh& m, const PhysParams& p, const StageArgs& a, int S, hipStream_t st)
{
    if (S == 3) updS<3>(m, p, a, st);
    else if (S == 4) updS<4>(m, p, a, st);
    else updS<6>(m, p, a, st);
    const uint32_t g = nblk(m.N);
    if (g && !a.deferReduce) launchReduceStage(a.partial, g, a.sc, a.checkActive, st);
}

void launchRmsLeaves(const DiagArgs& d, double* blockSums, hipStream_t st)
{
    if (d.N) hipLaunchKernelGGL(k_rms_leaves, dim3(nblk(d.N)), dim3(BLK), 0, st, d, blockSums);
}

void launchEpilogue(const DiagArgs& d, hipStream_t st)
{
    hipLaunchKernelGGL(k_epilogue, dim3(d.nEpi), dim3(EPT), 0, st, d);
}

void launchBeginCall(DevScalars* sc, unsigned long long rmaxBits, const double* dt, hipStream_t st)
{
    hipLaunchKernelGGL(k_begin_call, dim3(1), dim3(1), 0, st, sc, rmaxBits, dt ? *dt : 0.0, dt ? 1 : 0);
}

void launchFinishCall(const double* partial, uint32_t nPart, uint32_t nStages, DevScalars* sc, int putDt,
                      DevScalars* host, hipStream_t st)
{
    hipLaunchKernelGGL(k_finish_call, dim3(1), dim3(1024), 0, st, partial, nPart, nStages, sc, putDt, host);
}

void launchInitScalars(DevScalars* sc, double dt, double t, double CFL, hipStream_t st)
{
    hipLaunchKernelGGL(k_init_scalars, dim3(1), dim3(1), 0, st, sc, dt, t, CFL);
}

// ---------------------------------------------------------------- batched launches
// One launch per kernel for many meshes.  Workgroup w takes item xcdBlock(w), so each
// XCD gets a contiguous run of items (items are listed mesh by mesh, cell blocks and tiles
// in order); the item names the mesh record and the block, tile or RMS workgroup, and the
// workgroup runs the solo kernel's code on it.
__global__ __launch_bounds__(EPT) void k_epilogue_batch(const MemberArgs* __restrict__ mem, const uint2* __restrict__ epi,
                                                        uint32_t parity)
{
    __shared__ double staging[2 * FORCE_LDS];
    __shared__ EpiLds E;
    const uint2 it = epi[blockIdx.x];
    const DiagArgs d = mem[it.x].d[parity ^ mem[it.x].parityFlip];
    epilogueBody(d, it.y, E, staging);
}

__global__ void k_gather_scalars(const MemberArgs* __restrict__ mem, const uint32_t* __restrict__ members, uint32_t n,
                                 DevScalars* __restrict__ out)
{
    // one thread per 8-byte word of a DevScalars record
    constexpr uint32_t W = sizeof(DevScalars) / 8;
    static_assert(sizeof(DevScalars) % 8 == 0, "DevScalars is copied in 8-byte words");
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n * W) return;
    const uint32_t k = g / W, w = g % W;
    const uint64_t* src = reinterpret_cast<const uint64_t*>(mem[members[k]].d[0].sc);
    reinterpret_cast<uint64_t*>(out + k)[w] = src[w];
}

void launchGradientBatch(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items,
                         uint32_t nItems, uint32_t parity, uint32_t stage, const uint2* epi, uint32_t nEpi,
                         hipStream_t st)
{
    if (nItems == 0) return;
    if (gs.gradTiles) {   // border blocks; order 2, no LP vector limiter
        const int mode = !(gs.limited && limitStage) ? 1 : (gs.venkat ? 4 : 2);
        if (gs.mixed) {
            if (gs.S == 3) borderBatchS<3, 1>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
            else if (gs.S == 4) borderBatchS<4, 1>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
            else borderBatchS<6, 1>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
        } else {
            if (gs.S == 3) borderBatchS<3, 0>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
            else if (gs.S == 4) borderBatchS<4, 0>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
            else borderBatchS<6, 0>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
        }
        return;
    }
    // batched groups run without the LP vector limiter (mode 3)
    const int mode = gs.order == 1 ? 0 : (!(gs.limited && limitStage) ? 1 : (gs.venkat ? 4 : 2));
    if (gs.mixed) {
        if (gs.S == 3) gradBatchS<3, 1>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
        else if (gs.S == 4) gradBatchS<4, 1>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
        else gradBatchS<6, 1>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
    } else {
        if (gs.S == 3) gradBatchS<3, 0>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
        else if (gs.S == 4) gradBatchS<4, 0>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
        else gradBatchS<6, 0>(mode, mem, items, nItems, parity, stage, epi, nEpi, st);
    }
}

void launchFaceTilesBatch(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items,
                          uint32_t nItems, uint32_t ldsBytes, uint32_t parity, uint32_t stage, hipStream_t st)
{
    if (nItems == 0) return;
    if (gs.gradTiles) {
#define EBB_GTB(S, MIX) gradTileBatchS<S, MIX>(gs, limitStage, mem, items, nItems, ldsBytes, parity, stage, st)
        if (gs.mixed) {
            if (gs.S == 3) EBB_GTB(3, 1); else if (gs.S == 4) EBB_GTB(4, 1); else EBB_GTB(6, 1);
        } else {
            if (gs.S == 3) EBB_GTB(3, 0); else if (gs.S == 4) EBB_GTB(4, 0); else EBB_GTB(6, 0);
        }
#undef EBB_GTB
        return;
    }
    if (gs.mixed) {
        if (gs.S == 3) faceBatchS<3, 1>(gs, limitStage, mem, items, nItems, ldsBytes, parity, stage, st);
        else if (gs.S == 4) faceBatchS<4, 1>(gs, limitStage, mem, items, nItems, ldsBytes, parity, stage, st);
        else faceBatchS<6, 1>(gs, limitStage, mem, items, nItems, ldsBytes, parity, stage, st);
    } else {
        if (gs.S == 3) faceBatchS<3, 0>(gs, limitStage, mem, items, nItems, ldsBytes, parity, stage, st);
        else if (gs.S == 4) faceBatchS<4, 0>(gs, limitStage, mem, items, nItems, ldsBytes, parity, stage, st);
        else faceBatchS<6, 0>(gs, limitStage, mem, items, nItems, ldsBytes, parity, stage, st);
    }
}

void launchEpilogueBatch(const MemberArgs* mem, const uint2* epi, uint32_t nEpi, uint32_t parity, hipStream_t st)
{
    if (nEpi) hipLaunchKernelGGL(k_epilogue_batch, dim3(nEpi), dim3(EPT), 0, st, mem, epi, parity);
}

void launchGatherScalars(const MemberArgs* mem, const uint32_t* members, uint32_t n, DevScalars* out, hipStream_t st)
{
    const uint32_t words = n * uint32_t(sizeof(DevScalars) / 8);
    if (words) hipLaunchKernelGGL(k_gather_scalars, dim3((words + 255) / 256), dim3(256), 0, st, mem, members, n, out);
}

}  // namespace ebb
