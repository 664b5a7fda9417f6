// HIP kernels for the explicit residual-and-update loop, FP64, gfx950.
//
// One residual evaluation (source/solve.d:322-1122) is three launches:
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
//               and Rmax (block reduction + one ordered-bits atomic per block,
//               exact because min/max are order independent), the MMS source
//               (app/ms.d:131-141) and the integrator stage update
//               (source/integrators.d:22-270) fused in.
// No atomics touch the residual: each cell sums its own faces in a fixed order,
// so results are deterministic and bit-identical to the edge-loop form.
// Built with -ffp-contract=off: every product and sum rounds as written.
// This file holds the gradient, split-path and step epilogue kernels and the launchers; the
// tile kernels are in face_tiles.hpp, grad_tiles.hip and fused.hip.
#include "device.hpp"
#include "tile_launch.hpp"

namespace ebb {

template <int S, int MODE, int MIX>
__global__ __launch_bounds__(BLK) void k_gradient(DevMesh m, PhysParams p, StageArgs a)
{
    static_assert(BLK * 9 >= 2 * FORCE_LDS, "force staging exceeds the gradient staging rows");
    __shared__ GradLds<MODE> L;
    // with a force boundary, workgroup 0 (dispatched first) sums a pending boundary force
    // of the previous step, whether or not the loop is still active; the others are the
    // cell blocks
    const uint32_t fw = a.force.n ? 1u : 0u;
    if (fw && blockIdx.x == 0) {
        pendingForce<BLK, FORCE_LDS>(a.force, a.sc, reinterpret_cast<double2*>(&L.sg[0][0]));
        return;
    }
    const uint32_t b = blockIdx.x - fw, nb = gridDim.x - fw;
    gradientBody<S, MODE, MIX>(m, p, a, (a.order & 2) ? xcdBlockBack(b, nb) : xcdBlock(b, nb), L);
}

template <int FLUX, int VISC, int ORDER, int LP, int STORE, int MIX>
__global__ __launch_bounds__(BLK) void k_faces(DevMesh m, PhysParams p, StageArgs a, uint32_t nbi)
{
    using R = typename std::conditional<MIX == 1, float, double>::type;
    if (a.checkActive && !a.sc->active) return;
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
                     hipStream_t st, int parts)
{
    if (t.nTiles == 0) return;
    // order 2 and no LP vector limiter (the set-up keeps other configurations on face tiles)
    const int mode = !(p.limited && a.limit) ? 1 : (p.venkat ? 4 : 2);
    if (S == 3) gradTileS<3>(m, p, a, t, mode, parts, st);
    else if (S == 4) gradTileS<4>(m, p, a, t, mode, parts, st);
    else gradTileS<6>(m, p, a, t, mode, parts, st);
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
// Phobos std.algorithm.sum over double[] (app/solver.d:153-168): 16-element
// blocks summed by a fixed tree, blocks merged by a binary counter (perfect
// pairwise trees over aligned power-of-two runs), remainder elements likewise,
// and the stack folded from the top.  A workgroup reduces an aligned chunk of
// RMS_CHUNK_BLOCKS blocks level by level; the finalize kernel replays the
// counter over the chunk trees.  Quantities 0..3: sum of (now-last)^2 per
// variable; 4..7: sum of now.
DEV void rmsElement(const DiagArgs& d, uint64_t e, double out[8])
{
    if (e < d.N) {
        const uint32_t dv = d.perm ? d.perm[e] : uint32_t(e);
        double qa[4], qb[4];
        ld4(d.qnew, dv, qa);
        ld4(d.qold, dv, qb);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const double x = qa[v] - qb[v];
            out[v] = x * x;
            out[4 + v] = qa[v];
        }
    } else {
#pragma unroll
        for (int v = 0; v < 8; v++) out[v] = 0.0;   // ghost slots hold 0 in both arrays
    }
}

constexpr int RBLK = 1024;   // threads per chunk workgroup (element path)
constexpr int FTILE = 2048;   // force faces staged per pass (RMS kernels)

// Pairwise levels of one chunk: v[q][0..cnt) holds its 16-element block sums.
// Level l's odd leftover is stored as tree l of the chunk (the binary counter's
// stack), mask marks the levels present.  NT threads.
template <int NT>
DEV void chunkLevels(double (*v)[RMS_CHUNK_BLOCKS], uint32_t cnt, double* out, uint32_t* maskOut)
{
    // NT/8 threads per quantity; slot u of a thread is pair l + u * G (registers, no
    // divisions by the level's length)
    constexpr uint32_t G = NT / 8;
    constexpr int PER = int((RMS_CHUNK_BLOCKS / 2 + G - 1) / G);
    const uint32_t qq = threadIdx.x / G, l = threadIdx.x % G;
    uint32_t c = cnt;
    int level = 0;
    uint32_t mask = 0;
    while (c > 0) {
        if (c & 1) {
            if (threadIdx.x < 8) out[threadIdx.x * 16 + level] = v[threadIdx.x][c - 1];
            mask |= 1u << level;
        }
        const uint32_t half = c / 2;
        double tmp[PER];
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const uint32_t j = l + uint32_t(u) * G;
            tmp[u] = j < half ? v[qq][2 * j] + v[qq][2 * j + 1] : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const uint32_t j = l + uint32_t(u) * G;
            if (j < half) v[qq][j] = tmp[u];
        }
        __syncthreads();
        c = half;
        level++;
    }
    if (threadIdx.x < 8) maskOut[threadIdx.x] = mask;
}

// The boundary force (mesh.d:645-671): len*flux of the force faces summed in the
// reference's edge order by one lane, from LDS-staged values; NT threads stage.
// The stage reductions of a time-loop step, done here instead of after each stage:
// newDt is the last stage's minimum (every stage overwrites it), Rmax the maximum
// over the step's stages; min and max are exact in any order.
template <int NT>
DEV void stageReduce(const DiagArgs& d, double* lds)
{
    // each pass issues all of a thread's loads before using any (the partials were
    // written on all XCDs: every load is a round trip past this XCD's L2)
    constexpr int SLOTS = 24;
    double a0 = INFINITY, b0 = 0.0;
    for (uint32_t s = 0; s < d.nStages; s++) {
        const double2* pp = reinterpret_cast<const double2*>(d.partial + size_t(s) * d.pstride);
        const bool lastStage = s + 1 == d.nStages;
        for (uint32_t base = 0; base < d.nPart; base += NT * SLOTS) {
            double2 pv[SLOTS];
#pragma unroll
            for (int u = 0; u < SLOTS; u++) {
                const uint32_t k = base + threadIdx.x + uint32_t(u) * NT;
                pv[u] = k < d.nPart ? pp[k] : make_double2(INFINITY, 0.0);
            }
#pragma unroll
            for (int u = 0; u < SLOTS; u++) {
                if (lastStage) a0 = fmin(a0, pv[u].x);
                b0 = fmax(b0, pv[u].y);
            }
        }
    }
    a0 = warpMin(a0);
    b0 = warpMax(b0);
    const uint32_t w = threadIdx.x / 64;
    if ((threadIdx.x & 63) == 0) { lds[2 * w] = a0; lds[2 * w + 1] = b0; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t k = 1; k < NT / 64; k++) { a0 = fmin(a0, lds[2 * k]); b0 = fmax(b0, lds[2 * k + 1]); }
        d.sc->newDtBits = (unsigned long long)__double_as_longlong(a0);
        const double prev = __longlong_as_double((long long)d.sc->rmaxBits);
        if (b0 > prev) d.sc->rmaxBits = (unsigned long long)__double_as_longlong(b0);
    }
}
// force workgroup of the RMS kernels: the step's force sums for k_finalize (unless
// they are left to the next gradient kernel)
template <int NT>
DEV void forceSum(const DiagArgs& d, double* fb)
{
    if (d.deferForce) return;
    double f0, f1;
    orderedForce<NT, FTILE>(d.forceFaces, d.nForce, d.lenF, reinterpret_cast<double2*>(fb), f0, f1);
    if (threadIdx.x == 0) { d.sc->fsum[0] = f0; d.sc->fsum[1] = f1; }
}


// RMS sums from the states (element path): one workgroup per chunk of
// RMS_CHUNK_BLOCKS 16-element blocks; 16 consecutive lanes own one block, and
// the xor butterfly over them adds exactly like the fixed tree
// (((r0+r1)+(r2+r3))+...).  The last workgroup sums the boundary force.
__global__ __launch_bounds__(RBLK) void k_rms_chunks(DiagArgs d)
{
    if (!d.sc->active) return;
    __shared__ double v[8][RMS_CHUNK_BLOCKS];
    if (blockIdx.x == gridDim.x - 2) { forceSum<RBLK>(d, &v[0][0]); return; }
    if (blockIdx.x == gridDim.x - 1) { if (d.nStages) stageReduce<RBLK>(d, &v[0][0]); return; }
    const uint64_t nb = uint64_t(d.L) / 16;
    const uint64_t c0 = uint64_t(blockIdx.x) * RMS_CHUNK_BLOCKS;
    const uint32_t cnt = uint32_t((nb - c0) < RMS_CHUNK_BLOCKS ? (nb - c0) : RMS_CHUNK_BLOCKS);
    constexpr uint32_t BPI = RBLK / 16;
    for (uint32_t it = 0; it < RMS_CHUNK_BLOCKS / BPI; it++) {
        const uint32_t lb = it * BPI + threadIdx.x / 16;
        double o[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (lb < cnt) rmsElement(d, (c0 + lb) * 16 + (threadIdx.x % 16), o);
#pragma unroll
        for (int m = 1; m < 16; m <<= 1)
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = o[q] + __shfl_xor(o[q], m, 64);
        if ((threadIdx.x % 16) == 0 && lb < cnt)
#pragma unroll
            for (int q = 0; q < 8; q++) v[q][lb] = o[q];
    }
    __syncthreads();
    chunkLevels<RBLK>(v, cnt, d.chunkTrees + size_t(blockIdx.x) * 8 * 16, d.chunkMask + blockIdx.x * 8);
}

// RMS sums from the leaf sums the last stage stored (blockSums, 8 per block;
// blocks wholly past the interior cells are zero).  Workgroups [0, nfull): one
// full chunk each, only its top tree is needed: each lane adds 4 consecutive
// blocks pairwise, the 64-lane xor butterfly adds levels 3..8 exactly as the
// pairwise tree does (the two orders of each sum are equal), the 4 waves levels
// 9 and 10.  Workgroup nfull: the partial last chunk; nfull+1: the boundary force.
constexpr int RFB = 256;
DEV void rmsBlocksBody(const DiagArgs& d, uint32_t nfull, uint32_t wg, double (*v)[RMS_CHUNK_BLOCKS])
{
    if (!d.sc->active) return;
    const uint64_t nb = uint64_t(d.L) / 16;
    if (wg == nfull + 1) { forceSum<RFB>(d, &v[0][0]); return; }
    if (wg == nfull + 2) { if (d.nStages) stageReduce<RFB>(d, &v[0][0]); return; }
    const uint64_t c0 = uint64_t(wg) * RMS_CHUNK_BLOCKS;
    auto leaf = [&](uint64_t b, double o[8]) {
        if (b * 16 < d.N) {
            const double4 x = *reinterpret_cast<const double4*>(d.blockSums + b * 8);
            const double4 y = *reinterpret_cast<const double4*>(d.blockSums + b * 8 + 4);
            o[0] = x.x; o[1] = x.y; o[2] = x.z; o[3] = x.w; o[4] = y.x; o[5] = y.y; o[6] = y.z; o[7] = y.w;
        } else {
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = 0.0;
        }
    };
    if (wg == nfull) {   // partial chunk
        const uint32_t cnt = uint32_t(nb - c0);
        for (uint32_t lb = threadIdx.x; lb < cnt; lb += RFB) {
            double o[8];
            leaf(c0 + lb, o);
#pragma unroll
            for (int q = 0; q < 8; q++) v[q][lb] = o[q];
        }
        __syncthreads();
        chunkLevels<RFB>(v, cnt, d.chunkTrees + size_t(nfull) * 8 * 16, d.chunkMask + nfull * 8);
        return;
    }
    double b[4][8], t[8];
#pragma unroll
    for (int u = 0; u < 4; u++) leaf(c0 + 4 * threadIdx.x + u, b[u]);
#pragma unroll
    for (int q = 0; q < 8; q++) t[q] = (b[0][q] + b[1][q]) + (b[2][q] + b[3][q]);
#pragma unroll
    for (int m = 1; m < 64; m <<= 1)
#pragma unroll
        for (int q = 0; q < 8; q++) t[q] = t[q] + __shfl_xor(t[q], m, 64);
    const int w = threadIdx.x / 64;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int q = 0; q < 8; q++) v[q][w] = t[q];
    __syncthreads();
    if (threadIdx.x < 8) {
        const int q = threadIdx.x;
        d.chunkTrees[size_t(wg) * 128 + q * 16 + 10] = (v[q][0] + v[q][1]) + (v[q][2] + v[q][3]);
    }
}

__global__ __launch_bounds__(RFB) void k_rms_blocks(DiagArgs d, uint32_t nfull)
{
    __shared__ double v[8][RMS_CHUNK_BLOCKS];
    rmsBlocksBody(d, nfull, blockIdx.x, v);
}

// Step epilogue (app/solver.d:122-247), one workgroup.  The chunk trees are
// merged level by level in LDS (a perfect tree over each aligned power-of-two
// run of chunks is exactly the binary counter's merge); the boundary force comes
// summed from the RMS kernel.
constexpr int FIN_T = 256;
constexpr int FIN_CHUNKS = 1024;     // chunk trees merged in LDS per quantity

struct FinLds {
    double v[8][FIN_CHUNKS];
    double trees[8][48];
    int ntree[8];
    double tot[8];
};

DEV void finalizeBody(const DiagArgs& d, FinLds& L)
{
    DevScalars* sc = d.sc;
    auto& v = L.v;
    auto& trees = L.trees;
    auto& ntree = L.ntree;
    auto& tot = L.tot;
    const int tid = threadIdx.x;
    const uint64_t nb = uint64_t(d.L) / 16;
    const uint64_t nfull = nb / RMS_CHUNK_BLOCKS, part = nb % RMS_CHUNK_BLOCKS;
    // Every global read of the kernel is issued here, before the first is used (the
    // active flag included): the previous kernels wrote this data on all XCDs, so each
    // read is a round trip past this XCD's L2, and a chain of them set the kernel's length.
    // FIN_T/8 threads per quantity; slot u of a thread is chunk l + u * G.
    constexpr uint32_t G = FIN_T / 8;
    constexpr int PER = int(FIN_CHUNKS / G), HPER = int(FIN_CHUNKS / 2 / G);
    const uint32_t qq = uint32_t(tid) / G, l = uint32_t(tid) % G;
    const uint32_t n = nfull <= FIN_CHUNKS ? uint32_t(nfull) : 0u;
    double tv[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const uint32_t k = l + uint32_t(u) * G;
        tv[u] = k < n ? d.chunkTrees[size_t(k) * 128 + qq * 16 + 10] : 0.0;
    }
    uint32_t pmask = 0;   // the partial chunk's level trees (thread q < 8: quantity q)
    double ptree[16];
#pragma unroll
    for (int b2 = 0; b2 < 16; b2++) ptree[b2] = 0.0;
    if (tid < 8 && part) {
        pmask = d.chunkMask[nfull * 8 + tid];
#pragma unroll
        for (int b2 = 0; b2 < 16; b2++) ptree[b2] = d.chunkTrees[nfull * 128 + tid * 16 + b2];
    }
    const DevScalars s0 = *sc;
    if (!s0.active) return;
    if (tid < 8) ntree[tid] = 0;
    __syncthreads();
    if (nfull <= FIN_CHUNKS) {
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const uint32_t k = l + uint32_t(u) * G;
            if (k < n) v[qq][k] = tv[u];
        }
        __syncthreads();
        uint32_t c = n;
        int level = 0;
        uint32_t lmask = 0;
        while (c > 0) {
            if (c & 1) {
                if (tid < 8) trees[tid][47 - level] = v[tid][c - 1];
                lmask |= 1u << level;
            }
            const uint32_t half = c / 2;
            double tmp[HPER];
#pragma unroll
            for (int u = 0; u < HPER; u++) {
                const uint32_t j = l + uint32_t(u) * G;
                tmp[u] = j < half ? v[qq][2 * j] + v[qq][2 * j + 1] : 0.0;
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < HPER; u++) {
                const uint32_t j = l + uint32_t(u) * G;
                if (j < half) v[qq][j] = tmp[u];
            }
            __syncthreads();
            c = half;
            level++;
        }
        // chunk-level trees, largest first
        if (tid < 8) {
            int t = 0;
            for (int l = 31; l >= 0; l--)
                if (lmask & (1u << l)) trees[tid][t++] = trees[tid][47 - l];
            ntree[tid] = t;
        }
    } else if (tid < 8) {
        // very large meshes: replay the binary counter over the chunk trees directly, on
        // the quantity's LDS stack (no scratch)
        double* st = trees[tid];
        int idx = 0;
        for (uint64_t k = 0; k < nfull; k++) {
            st[idx] = d.chunkTrees[k * 128 + tid * 16 + 10];
            const int last = idx - __builtin_ctzll(k + 1);
            while (idx > last) { st[idx - 1] += st[idx]; --idx; }
            ++idx;
        }
        ntree[tid] = idx;
    }
    __syncthreads();
    if (tid < 8) {
        const int q = tid;
        int idx = ntree[q];
        double* st = trees[q];
        if (part) {
#pragma unroll
            for (int b2 = 15; b2 >= 0; b2--)
                if (pmask & (1u << b2)) st[idx++] = ptree[b2];
        }
        const uint64_t rem = uint64_t(d.L) - nb * 16;
        for (uint64_t i = 0; i < rem; i++) {
            double o[8];
            rmsElement(d, nb * 16 + i, o);
            double oq = o[0];   // o[q] by selects, so o stays in registers
#pragma unroll
            for (int k = 1; k < 8; k++) oq = q == k ? o[k] : oq;
            st[idx] = oq;
            const int last = idx - __builtin_ctzll(i + 1);
            while (idx > last) { st[idx - 1] += st[idx]; --idx; }
            ++idx;
        }
        double s = 0.0;
        if (idx > 0) {
            s = st[idx - 1];
            for (int j2 = idx - 2; j2 >= 0; j2--) s += st[j2];
        }
        tot[q] = 0.0 + s;
    }
    __syncthreads();
    if (tid != 0) return;
    const double f0 = s0.fsum[0], f1 = s0.fsum[1];   // summed by the RMS kernel's force workgroup (unless deferred)
    double rms[4];
    for (int q = 0; q < 4; q++) rms[q] = sqrt(double(d.N) * tot[q]) / tot[4 + q];
    const double newDt = __longlong_as_double((long long)s0.newDtBits);
    const double Rmax = __longlong_as_double((long long)s0.rmaxBits);
    const double dt = d.dynamicDt ? newDt : s0.dt;
    const double ld0 = 0.0 + d.rot[0] * f0 + d.rot[1] * f1;
    const double ld1 = 0.0 + d.rot[2] * f0 + d.rot[3] * f1;
    const double residMax = dmax(dmax(dmax(rms[0], rms[1]), rms[2]), rms[3]);
    int64_t inc = s0.incIters;
    double CFL = s0.CFL;
    if (d.cflAdjust) {
        if (s0.residLast < residMax) inc++;
        else if (inc >= 1) inc--;
        if (inc >= 2000) { CFL *= 0.99; inc = 0; }
    }
    // the history row: by absolute step within the host's batch, or a ring (batched runs)
    const int64_t slot = d.histRing ? s0.steps % d.histCap : s0.steps - d.histBase;
    if (slot >= 0 && slot < d.histCap) {
        double* h = d.hist + slot * HIST_FIELDS;
        h[0] = s0.t; h[1] = dt; h[2] = rms[0]; h[3] = rms[1]; h[4] = rms[2]; h[5] = rms[3];
        h[6] = Rmax; h[9] = CFL;
        if (!d.deferForce) { h[7] = ld0; h[8] = ld1; }
    }
    const double t1 = s0.t + dt;
    const int64_t steps1 = s0.steps + 1;
    sc->dt = dt;
    sc->incIters = inc;
    sc->CFL = CFL;
    sc->residLast = residMax;
    for (int q = 0; q < 4; q++) sc->rms[q] = rms[q];
    if (d.deferForce) {
        // drag and lift of this step are summed by the next gradient kernel (or at the end of
        // the batch), which writes them into this row and sc->force
        sc->forcePending = 1;
        sc->forceSlot = (slot >= 0 && slot < d.histCap) ? slot : -1;
    } else {
        sc->force[0] = ld0; sc->force[1] = ld1;
    }
    sc->t = t1;
    sc->steps = steps1;
    // convergence stop (extensions.rmsDrop): the rho RMS residual of app/solver.d:153-168 has
    // dropped by the given factor below its value on the first step
    const double rms0 = s0.steps == 0 ? rms[0] : s0.rms0;
    sc->rms0 = rms0;
    const bool converged = d.rmsDrop > 0 && rms[0] <= d.rmsDrop * rms0;
    if (converged) sc->converged = 1;
    if (!(t1 < d.tEnd) || (d.maxSteps >= 0 && steps1 >= d.maxSteps) || s0.errEdge != ~0ull || s0.errCell != ~0ull ||
        s0.errBC != ~0ull || converged)
        sc->active = 0;
}

__global__ __launch_bounds__(FIN_T) void k_finalize(DiagArgs d)
{
    __shared__ FinLds L;
    finalizeBody(d, L);
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
    sc->converged = 0;
    sc->rms0 = 0;
    for (int v = 0; v < 4; v++) sc->rms[v] = 0;
    sc->force[0] = sc->force[1] = 0;
    sc->fsum[0] = sc->fsum[1] = 0;
    sc->forcePending = 0;
    sc->pad2 = 0;
    sc->forceSlot = -1;
}

// ---------------------------------------------------------------- launchers
static uint32_t nblk(uint64_t n) { return uint32_t((n + BLK - 1) / BLK); }

template <int S>
static void gradS(const DevMesh& m, const PhysParams& p, const StageArgs& a, hipStream_t st)
{
    const uint32_t g = nblk(m.N) + (a.force.n ? 1u : 0u);   // + the force workgroup
    if (g == 0) return;
    const int mode = p.order == 1 ? 0 : (!(p.limited && a.limit) ? 1 : (p.venkat ? 4 : (p.lpThresh > 0 ? 3 : 2)));
    if (p.mixed) {
        switch (mode) {
        case 0: hipLaunchKernelGGL((k_gradient<S, 0, 1>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
        case 1: hipLaunchKernelGGL((k_gradient<S, 1, 1>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
        case 4: hipLaunchKernelGGL((k_gradient<S, 4, 1>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
        default: hipLaunchKernelGGL((k_gradient<S, 2, 1>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
        }
        return;
    }
    switch (mode) {
    case 0: hipLaunchKernelGGL((k_gradient<S, 0, 0>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
    case 1: hipLaunchKernelGGL((k_gradient<S, 1, 0>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
    case 2: hipLaunchKernelGGL((k_gradient<S, 2, 0>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
    case 4: hipLaunchKernelGGL((k_gradient<S, 4, 0>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
    default: hipLaunchKernelGGL((k_gradient<S, 3, 0>), dim3(g), dim3(BLK), 0, st, m, p, a); break;
    }
}

void launchGradient(const DevMesh& m, const PhysParams& p, const StageArgs& a, int S, hipStream_t st)
{
    if (S == 3) gradS<3>(m, p, a, st);
    else if (S == 4) gradS<4>(m, p, a, st);
    else gradS<6>(m, p, a, st);
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

void launchRmsChunks(const DiagArgs& d, hipStream_t st)
{
    const uint64_t nb = uint64_t(d.L) / 16;
    const uint32_t nc = uint32_t((nb + RMS_CHUNK_BLOCKS - 1) / RMS_CHUNK_BLOCKS);
    if (d.blockSums) {
        // full chunks, the partial chunk (its workgroup returns at once when there is none), the
        // force, the stage reductions
        const uint32_t nfull = uint32_t(nb / RMS_CHUNK_BLOCKS);
        hipLaunchKernelGGL(k_rms_blocks, dim3(nfull + 3), dim3(RFB), 0, st, d, nfull);
    } else {
        hipLaunchKernelGGL(k_rms_chunks, dim3(nc + 2), dim3(RBLK), 0, st, d);
    }
}

__global__ __launch_bounds__(BLK) void k_pending_force(ForceArgs f, DevScalars* sc)
{
    __shared__ double2 fsh[FORCE_LDS];
    pendingForce<BLK, FORCE_LDS>(f, sc, fsh);
}

void launchPendingForce(const ForceArgs& f, DevScalars* sc, hipStream_t st)
{
    if (f.n) hipLaunchKernelGGL(k_pending_force, dim3(1), dim3(BLK), 0, st, f, sc);
}

void launchFinalize(const DiagArgs& d, hipStream_t st)
{
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(FIN_T), 0, st, d);
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
template <int S, int MODE, int MIX>
__global__ __launch_bounds__(BLK) void k_gradient_batch(const MemberArgs* __restrict__ mem, const uint2* __restrict__ items,
                                                        uint32_t parity, uint32_t stage)
{
    __shared__ GradLds<MODE> L;
    const uint2 it = items[xcdBlock(blockIdx.x, gridDim.x)];
    const MemberArgs& M = mem[it.x];
    const StageArgs& a = M.st[parity ^ M.parityFlip][stage];
    if (it.y == FORCE_ITEM) {
        pendingForce<BLK, FORCE_LDS>(a.force, a.sc, reinterpret_cast<double2*>(&L.sg[0][0]));
        return;
    }
    gradientBody<S, MODE, MIX>(M.m, M.p, a, it.y, L);
}

__global__ __launch_bounds__(RFB) void k_rms_batch(const MemberArgs* __restrict__ mem, const uint2* __restrict__ items,
                                                   uint32_t parity)
{
    __shared__ double v[8][RMS_CHUNK_BLOCKS];
    const uint2 it = items[blockIdx.x];
    const MemberArgs& M = mem[it.x];
    rmsBlocksBody(M.d[parity ^ M.parityFlip], M.nRmsFull, it.y, v);
}

__global__ __launch_bounds__(FIN_T) void k_finalize_batch(const MemberArgs* __restrict__ mem,
                                                          const uint32_t* __restrict__ members, uint32_t parity)
{
    __shared__ FinLds L;
    const MemberArgs& M = mem[members[blockIdx.x]];
    finalizeBody(M.d[parity ^ M.parityFlip], L);
}

__global__ __launch_bounds__(BLK) void k_pending_force_batch(const MemberArgs* __restrict__ mem,
                                                             const uint32_t* __restrict__ members)
{
    __shared__ double2 fsh[FORCE_LDS];
    const MemberArgs& M = mem[members[blockIdx.x]];
    pendingForce<BLK, FORCE_LDS>(M.f, M.d[0].sc, fsh);
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

template <int S, int MIX>
static void gradBatchS(int mode, const MemberArgs* mem, const uint2* items, uint32_t n, uint32_t par, uint32_t st,
                       hipStream_t s)
{
    const dim3 g(n), b(BLK);
    switch (mode) {
    case 0: hipLaunchKernelGGL((k_gradient_batch<S, 0, MIX>), g, b, 0, s, mem, items, par, st); break;
    case 1: hipLaunchKernelGGL((k_gradient_batch<S, 1, MIX>), g, b, 0, s, mem, items, par, st); break;
    case 4: hipLaunchKernelGGL((k_gradient_batch<S, 4, MIX>), g, b, 0, s, mem, items, par, st); break;
    default: hipLaunchKernelGGL((k_gradient_batch<S, 2, MIX>), g, b, 0, s, mem, items, par, st); break;
    }
}

void launchGradientBatch(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items,
                         uint32_t nItems, uint32_t parity, uint32_t stage, hipStream_t st)
{
    if (nItems == 0) return;
    if (gs.gradTiles) {   // border blocks; order 2, no LP vector limiter
        const int mode = !(gs.limited && limitStage) ? 1 : (gs.venkat ? 4 : 2);
        if (gs.mixed) {
            if (gs.S == 3) borderBatchS<3, 1>(mode, mem, items, nItems, parity, stage, st);
            else if (gs.S == 4) borderBatchS<4, 1>(mode, mem, items, nItems, parity, stage, st);
            else borderBatchS<6, 1>(mode, mem, items, nItems, parity, stage, st);
        } else {
            if (gs.S == 3) borderBatchS<3, 0>(mode, mem, items, nItems, parity, stage, st);
            else if (gs.S == 4) borderBatchS<4, 0>(mode, mem, items, nItems, parity, stage, st);
            else borderBatchS<6, 0>(mode, mem, items, nItems, parity, stage, st);
        }
        return;
    }
    // batched groups run without the LP vector limiter (mode 3)
    const int mode = gs.order == 1 ? 0 : (!(gs.limited && limitStage) ? 1 : (gs.venkat ? 4 : 2));
    if (gs.mixed) {
        if (gs.S == 3) gradBatchS<3, 1>(mode, mem, items, nItems, parity, stage, st);
        else if (gs.S == 4) gradBatchS<4, 1>(mode, mem, items, nItems, parity, stage, st);
        else gradBatchS<6, 1>(mode, mem, items, nItems, parity, stage, st);
    } else {
        if (gs.S == 3) gradBatchS<3, 0>(mode, mem, items, nItems, parity, stage, st);
        else if (gs.S == 4) gradBatchS<4, 0>(mode, mem, items, nItems, parity, stage, st);
        else gradBatchS<6, 0>(mode, mem, items, nItems, parity, stage, st);
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

void launchRmsBatch(const MemberArgs* mem, const uint2* items, uint32_t nItems, uint32_t parity, hipStream_t st)
{
    if (nItems) hipLaunchKernelGGL(k_rms_batch, dim3(nItems), dim3(RFB), 0, st, mem, items, parity);
}

void launchFinalizeBatch(const MemberArgs* mem, const uint32_t* members, uint32_t n, uint32_t parity, hipStream_t st)
{
    if (n) hipLaunchKernelGGL(k_finalize_batch, dim3(n), dim3(FIN_T), 0, st, mem, members, parity);
}

void launchPendingForceBatch(const MemberArgs* mem, const uint32_t* members, uint32_t n, hipStream_t st)
{
    if (n) hipLaunchKernelGGL(k_pending_force_batch, dim3(n), dim3(BLK), 0, st, mem, members);
}

void launchGatherScalars(const MemberArgs* mem, const uint32_t* members, uint32_t n, DevScalars* out, hipStream_t st)
{
    const uint32_t words = n * uint32_t(sizeof(DevScalars) / 8);
    if (words) hipLaunchKernelGGL(k_gather_scalars, dim3((words + 255) / 256), dim3(256), 0, st, mem, members, n, out);
}

}  // namespace ebb
