// The single fused stage kernel (extensions.stagePath = "fused").
#include "device.hpp"

namespace ebb {

// ---------------------------------------------------------------- fused stage
// One workgroup per tile: load the states of own + 2 halo rings into LDS, fill
// the ghosts, compute gradients/limiters for own + ring 1, every face flux of the
// own cells, and the own cells' residual + stage update -- one pass over HBM.
// The per-cell and per-face arithmetic is the same device code as the split
// kernels above, so results are bit-identical.
constexpr int TBLK = 256;

// Persistent form: a workgroup walks a contiguous run of tiles.  Two LDS buffers
// alternate: while the workgroup computes one tile, the next tile's blob is
// copied into the other buffer by direct global-to-LDS loads.
typedef __attribute__((address_space(3))) void* LdsPtr;

DEV void dmaBlob(const TileArgs& t, const uint4& d1, uint8_t* slot)
{
    const uint32_t n = d1.z, lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint4* src = t.blob + d1.y;
    for (uint32_t g = w; g * 64 < n; g += TBLK / 64) {
        const uint32_t c = g * 64 + lane;
        if (c < n) __builtin_amdgcn_global_load_lds((const void*)(src + c), (LdsPtr)(slot + g * 1024), 16, 0, 0);
    }
}

template <int S, int FLUX, int VISC, int LP>
__global__ __launch_bounds__(TBLK, 2) void k_stage_tile(DevMesh m, PhysParams p, StageArgs a, TileArgs t)
{
    if (a.checkActive && !a.sc->active) return;
    extern __shared__ uint4 ldsv[];
    uint8_t* lds = reinterpret_cast<uint8_t*>(ldsv);
    uint8_t* dyn = lds + 2 * t.slotBytes;
    const uint32_t bid = xcdBlock(blockIdx.x, gridDim.x);
    if (bid == 0 && threadIdx.x == 0 && a.first) a.sc->rmaxBits = 0;   // Rmax is per step
    const uint32_t per = t.nTiles / gridDim.x, rem = t.nTiles % gridDim.x;
    const uint32_t tBeg = bid * per + (bid < rem ? bid : rem), tEnd = tBeg + per + (bid < rem ? 1 : 0);
    constexpr int LW = LP ? 8 : 4;
    const uint32_t tid = threadIdx.x;
    double dtCand = INFINITY, rCand = 0.0;
    uint4 d0 = make_uint4(0, 0, 0, 0), d1 = make_uint4(0, 0, 0, 0);
    if (tBeg < tEnd) {
        d0 = t.desc[2 * tBeg];
        d1 = t.desc[2 * tBeg + 1];
        dmaBlob(t, d1, lds);
    }
    uint32_t par = 0;
    for (uint32_t tile = tBeg; tile < tEnd; tile++) {
        const uint32_t nC = d0.x, nG = d0.y, nQ = d0.z, nL = d0.w, nF = d1.x;
        const TileImg I = tileImage(nC, nG, nQ, nL, nF, S);
        const TileDyn D = tileDyn(nG, nL, LW);
        uint8_t* base = lds + par * t.slotBytes;
        __builtin_amdgcn_s_waitcnt(0);   // this wave's copies of the blob have landed
        ldsBarrier();
        const uint32_t* ids = reinterpret_cast<const uint32_t*>(base + I.ids);
        double* qs = reinterpret_cast<double*>(dyn + D.qs);
        for (uint32_t k = tid; k < nQ; k += TBLK) {
            const double4 v = a.qin[ids[k]];
            qs[4 * k] = v.x; qs[4 * k + 1] = v.y; qs[4 * k + 2] = v.z; qs[4 * k + 3] = v.w;
        }
        const uint4 n0 = reinterpret_cast<const uint4*>(base + I.hdr)[0];
        const uint4 n1 = reinterpret_cast<const uint4*>(base + I.hdr)[1];
        if (tile + 1 < tEnd) dmaBlob(t, n1, lds + (par ^ 1u) * t.slotBytes);   // overlaps the compute below
        ldsBarrier();
        if (nL > nQ) {
            const uint16_t* gown = reinterpret_cast<const uint16_t*>(base + I.gown);
            for (uint32_t k = nQ + tid; k < nL; k += TBLK) {
                const uint32_t g = ids[k], own = gown[k - nQ];
                double qg[4];
                if (!ghostFromOwner(m.bface[g - m.N], qs + 4 * own, a.qin, g, qg) && a.recordErrors)
                    atomicMin(&a.sc->errBC, (uint64_t(a.stageId) << 32) | (g - m.N));
#pragma unroll
                for (int c = 0; c < 4; c++) qs[4 * k + c] = qg[c];
                if (own < nC) st4(a.qin, g, qg);   // one writer per ghost: the tile owning its cell
            }
            ldsBarrier();
        }
        const double2* cs = reinterpret_cast<const double2*>(base + I.cs);
        double* gs = reinterpret_cast<double*>(dyn + D.gs);
        double* ls = reinterpret_cast<double*>(dyn + D.ls);
        if (p.order > 1) {
            const bool lim = p.limited && a.limit;
            const uint16_t* nbS = reinterpret_cast<const uint16_t*>(base + I.nb);
            const double* gmS = reinterpret_cast<const double*>(base + I.gm);
            for (uint32_t k = tid; k < nG; k += TBLK) {
                double qn[S][4];
                double2 cn[S];
                bool real[S];
#pragma unroll
                for (int j = 0; j < S; j++) {
                    const uint32_t nb = nbS[k * S + j];
#pragma unroll
                    for (int c = 0; c < 4; c++) qn[j][c] = qs[4 * nb + c];
                    cn[j] = cs[nb];
                    real[j] = nb != k;
                }
                double g[4][2], lx[4], ly[4];
                const double* gmi = gmS + k;
                if (!lim) gradLimit<S, 1, double>(qs + 4 * k, qn, gmi, nG, cs[k], cn, real, 0, p.lpThresh, g, lx, ly);
                else if (LP) gradLimit<S, 3, double>(qs + 4 * k, qn, gmi, nG, cs[k], cn, real, 1, p.lpThresh, g, lx, ly);
                else gradLimit<S, 2, double>(qs + 4 * k, qn, gmi, nG, cs[k], cn, real, 1, p.lpThresh, g, lx, ly);
#pragma unroll
                for (int c = 0; c < 4; c++) { gs[8 * k + 2 * c] = g[c][0]; gs[8 * k + 2 * c + 1] = g[c][1]; }
                if (LP) {
#pragma unroll
                    for (int c = 0; c < 4; c++) { ls[8 * k + 2 * c] = lx[c]; ls[8 * k + 2 * c + 1] = ly[c]; }
                } else {
#pragma unroll
                    for (int c = 0; c < 4; c++) ls[4 * k + c] = lx[c];
                }
            }
        } else if (VISC) {
            for (uint32_t k = tid; k < 8 * nG; k += TBLK) gs[k] = 0.0;   // order 1: zero gradients
        }
        ldsBarrier();
        double* fs = reinterpret_cast<double*>(base + I.fs);
        const uint2* fcS = reinterpret_cast<const uint2*>(base + I.fc);
        for (uint32_t k = tid; k < nF; k += TBLK) {
            const uint2 fe = fcS[k];
            const uint32_t f = fe.x, la = fe.y & 0xffffu, lb = fe.y >> 16;
            double* slot = fs + 5 * k;
            const double2 n = make_double2(slot[0], slot[1]);
            const double2 mid = make_double2(slot[2], slot[3]);
            const double len = slot[4];
            double qL[4], qR[4], F[4], sMax;
            double la_x[4], la_y[4], lb_x[4], lb_y[4];
            if (p.order > 1) {
                if (LP) {
#pragma unroll
                    for (int c = 0; c < 4; c++) { la_x[c] = ls[8 * la + 2 * c]; la_y[c] = ls[8 * la + 2 * c + 1]; }
                } else {
#pragma unroll
                    for (int c = 0; c < 4; c++) { la_x[c] = ls[4 * la + c]; la_y[c] = la_x[c]; }
                }
            }
            uint64_t errKey;
            if (f < m.Fi) {
                if (p.order > 1) {
                    if (LP) {
#pragma unroll
                        for (int c = 0; c < 4; c++) { lb_x[c] = ls[8 * lb + 2 * c]; lb_y[c] = ls[8 * lb + 2 * c + 1]; }
                    } else {
#pragma unroll
                        for (int c = 0; c < 4; c++) { lb_x[c] = ls[4 * lb + c]; lb_y[c] = lb_x[c]; }
                    }
                }
                const double2 ca = cs[la], cb = cs[lb];
                if (p.order > 1)
                    interiorFace<FLUX, VISC, 2, LP>(qs + 4 * la, gs + 8 * la, la_x, la_y, ca, qs + 4 * lb, gs + 8 * lb,
                                                    lb_x, lb_y, cb, n, mid, p, qL, qR, F, sMax);
                else
                    interiorFace<FLUX, VISC, 1, LP>(qs + 4 * la, gs + 8 * la, la_x, la_y, ca, qs + 4 * lb, gs + 8 * lb,
                                                    lb_x, lb_y, cb, n, mid, p, qL, qR, F, sMax);
                errKey = uint64_t(m.Fb) + f;
            } else {
                const uint32_t b = f - m.Fi;
                const double2 co = cs[la];
                if (p.order > 1)
                    boundaryFace<FLUX, VISC, 2, LP>(qs + 4 * la, gs + 8 * la, la_x, la_y, co, qs + 4 * lb, m.bface[b],
                                                    n, mid, p, qL, qR, F, sMax);
                else
                    boundaryFace<FLUX, VISC, 1, LP>(qs + 4 * la, gs + 8 * la, la_x, la_y, co, qs + 4 * lb, m.bface[b],
                                                    n, mid, p, qL, qR, F, sMax);
                errKey = b;
            }
            if (a.recordErrors && (isnan(F[0]) || isnan(F[1]) || isnan(F[2]) || isnan(F[3])))
                atomicMin(&a.sc->errEdge, (uint64_t(a.stageId) << 32) | errKey);
            slot[0] = len * F[0]; slot[1] = len * F[1]; slot[2] = len * F[2]; slot[3] = len * F[3];
            slot[4] = len * sMax;
            if (f >= m.Fi) {   // boundary faces (each in exactly one tile) feed the force integral
                *reinterpret_cast<double4*>(a.lenF + size_t(f) * 4) =
                    make_double4(len * F[0], len * F[1], len * F[2], len * F[3]);
                a.lenS[f] = len * sMax;
            }
        }
        ldsBarrier();
        const uint16_t* cfS = reinterpret_cast<const uint16_t*>(base + I.cf);
        const double* met = reinterpret_cast<const double*>(base + I.met);
        for (uint32_t k = tid; k < nC; k += TBLK) {
            double r[4] = {0.0, 0.0, 0.0, 0.0};
            double sAve = 0;
#pragma unroll
            for (int j = 0; j < S; j++) {
                const uint32_t fe = cfS[k * S + j];
                const double* lf = fs + 5 * (fe & 0x7fffu);
                if (fe >> 15) { r[0] = r[0] - lf[0]; r[1] = r[1] - lf[1]; r[2] = r[2] - lf[2]; r[3] = r[3] - lf[3]; }
                else { r[0] = r[0] + lf[0]; r[1] = r[1] + lf[1]; r[2] = r[2] + lf[2]; r[3] = r[3] + lf[3]; }
                sAve += lf[4];
            }
            const uint32_t gi = ids[k];
            const double* qi = qs + 4 * k;
            const double* mk = met + 3 * k;
            switch (a.kind) {
            case SK_EULER: cellStage<SK_EULER>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            case SK_RK2_1: cellStage<SK_RK2_1>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            case SK_RK2_2: cellStage<SK_RK2_2>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            case SK_TVD_1: cellStage<SK_TVD_1>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            case SK_TVD_2: cellStage<SK_TVD_2>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            case SK_RK4_1: cellStage<SK_RK4_1>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            case SK_RK4_2: cellStage<SK_RK4_2>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            case SK_RK4_3: cellStage<SK_RK4_3>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            case SK_RK4_4: cellStage<SK_RK4_4>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            default: cellStage<SK_RESIDUAL>(m, p, a, gi, r, sAve, qi, mk, dtCand, rCand); break;
            }
        }
        ldsBarrier();   // the next tile overwrites the LDS image
        d0 = n0;
        d1 = n1;
        par ^= 1u;
    }
    blockPartial(dtCand, rCand, a.partial, blockIdx.x);
}

template <int S, int FLUX, int VISC, int LP>
static void tileLaunch(const DevMesh& m, const PhysParams& p, const StageArgs& a, const TileArgs& t, hipStream_t st)
{
    hipLaunchKernelGGL((k_stage_tile<S, FLUX, VISC, LP>), dim3(t.nBlocks), dim3(TBLK), t.ldsBytes, st, m, p, a, t);
}

template <int S>
static void tileS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const TileArgs& t, hipStream_t st)
{
    const bool lp = p.order > 1 && p.limited && p.lpThresh > 0;
    if (p.flux == 1) {
        if (p.viscous) { if (lp) tileLaunch<S, 1, 1, 1>(m, p, a, t, st); else tileLaunch<S, 1, 1, 0>(m, p, a, t, st); }
        else { if (lp) tileLaunch<S, 1, 0, 1>(m, p, a, t, st); else tileLaunch<S, 1, 0, 0>(m, p, a, t, st); }
    } else {
        if (p.viscous) { if (lp) tileLaunch<S, 0, 1, 1>(m, p, a, t, st); else tileLaunch<S, 0, 1, 0>(m, p, a, t, st); }
        else { if (lp) tileLaunch<S, 0, 0, 1>(m, p, a, t, st); else tileLaunch<S, 0, 0, 0>(m, p, a, t, st); }
    }
}

void launchStageTiles(const DevMesh& m, const PhysParams& p, const StageArgs& a, const TileArgs& t, int S,
                      hipStream_t st)
{
    if (t.nTiles == 0) return;
    if (S == 3) tileS<3>(m, p, a, t, st);
    else if (S == 4) tileS<4>(m, p, a, t, st);
    else tileS<6>(m, p, a, t, st);
    if (!a.deferReduce) launchReduceStage(a.partial, t.nBlocks, a.sc, a.checkActive, st);
}

}  // namespace ebb
