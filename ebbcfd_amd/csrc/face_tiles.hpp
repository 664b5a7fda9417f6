// The face/update tile kernel: every face of a tile's cells, then the cells' stage update.
#pragma once
#include "device.hpp"

namespace ebb {

// ---------------------------------------------------------------- faces + update
// One workgroup per face tile: every face of the tile's cells (states,
// gradients, limiters and ghosts as the gradient kernel left them) into LDS,
// then the cells' residual and stage update from LDS.  Same device code as
// k_faces and k_update, so bit-identical to them.
// Edge length, unit normal and midpoint from the two nodes, in the operation order
// of the mesh set-up (source/mesh.d; mesh.cpp), so they equal the stored ones bit
// for bit.  Interior edges: normal = (y1-y0, x0-x1)/|.|, whose norm is the length
// (the same squares summed in the other order); boundary edges: (1/len) * (...).
// FAST: the interior normals by Div's short form.  The length is always the IEEE root, since boundary
// faces use it too and root<1> loses the last place of edges below 1e-100: with root<1> and a flag for
// such meshes, 50 RK2 steps on 130,143 quadrilaterals took 3.02 ms and now take 3.00, other cases the
// same.
template <int FAST = 0>
DEV void edgeGeometry(bool interior, double2 p0, double2 p1, double2& n, double2& mid, double& len)
{
    const double ddx = p0.x - p1.x, ddy = p0.y - p1.y;
    len = sqrt(ddx * ddx + ddy * ddy);
    const double vx = p1.y - p0.y, vy = p0.x - p1.x;
    if (interior) {
        const Div<FAST, double> byLen(len);
        n = make_double2(byLen(vx), byLen(vy));
    } else {
        const double inv = 1.0 / len;
        n = make_double2(inv * vx, inv * vy);
    }
    mid = make_double2(0.5 * (p0.x + p1.x), 0.5 * (p0.y + p1.y));
}

// A tile's face results in LDS.  FP64 path: len*flux and len*sMax per face (40 B).  Mixed
// path: the FP32 flux and sMax and the FP64 length (28 B per face); the cell phase forms the
// same FP64 products len*F, so its sums are those of the 40-byte layout bit for bit, in
// 30 % less LDS (four workgroups per CU at 768-cell tiles instead of three).  `cap`: face
// slots of the largest tile plus the padding face.
template <int MIX>
struct FaceLds;
template <>
struct FaceLds<0> {
    double* v;
    DEV FaceLds(double* base, uint32_t) : v(base) {}
    DEV void put(uint32_t k, double len, const double F[4], double sMax) const
    {
        double* slot = v + 5 * k;
        slot[0] = len * F[0]; slot[1] = len * F[1]; slot[2] = len * F[2]; slot[3] = len * F[3];
        slot[4] = len * sMax;
    }
    DEV void zero(uint32_t k, uint32_t tid) const { if (tid < 5) v[5 * k + tid] = 0.0; }
    DEV void get(uint32_t k, double o[5]) const
    {
        const double* slot = v + 5 * k;
        o[0] = slot[0]; o[1] = slot[1]; o[2] = slot[2]; o[3] = slot[3]; o[4] = slot[4];
    }
};
template <>
struct FaceLds<1> {
    float4* f;
    double* len;
    float* s;
    DEV FaceLds(double* base, uint32_t cap)
        : f(reinterpret_cast<float4*>(base)), len(reinterpret_cast<double*>(f + cap)), s(reinterpret_cast<float*>(len + cap))
    {
    }
    DEV void put(uint32_t k, double l, const float F[4], float sMax) const
    {
        f[k] = make_float4(F[0], F[1], F[2], F[3]);
        len[k] = l;
        s[k] = sMax;
    }
    DEV void zero(uint32_t k, uint32_t tid) const
    {
        if (tid == 0) { f[k] = make_float4(0.f, 0.f, 0.f, 0.f); len[k] = 0.0; s[k] = 0.f; }
    }
    DEV void get(uint32_t k, double o[5]) const
    {
        const float4 F = f[k];
        const double l = len[k];
        o[0] = l * double(F.x); o[1] = l * double(F.y); o[2] = l * double(F.z); o[3] = l * double(F.w);
        o[4] = l * double(s[k]);
    }
};
// The cell phase of a face tile: each own cell sums its faces' results from LDS in its own
// face order and applies the stage update; the workgroup's (min dt, max |R|) pair goes to
// partial slot `pslot`.  giNext/giNext2: the device ids of the first two cell rounds.
template <int S, int MIX>
DEV void tileCellPhase(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, const uint4& d,
                       uint32_t pslot, const FaceLds<MIX>& fl, uint32_t giNext, uint32_t giNext2)
{
    const uint32_t tid = threadIdx.x;
    const uint32_t nC = d.x;
    // each cell round's per-cell inputs are loaded one round ahead (the first round's
    // before the barrier, which waits for LDS only), from ids loaded two rounds ahead
    // (a load issued after the next round's would wait for it: loads complete in order)
    double metN[3] = {0, 0, 0}, qnN[4] = {0, 0, 0, 0}, qiN[4] = {0, 0, 0, 0}, acN[4] = {0, 0, 0, 0};
    uint32_t refN = 0;
    const bool wantQn = a.kind != SK_RESIDUAL, wantQi = a.kind == SK_TVD_2;
    const bool wantAcc = a.kind == SK_RK2_2 || a.kind == SK_RK4_2 || a.kind == SK_RK4_3 || a.kind == SK_RK4_4;
    const bool wantRef = a.rmsBlocks != nullptr;
    // the other stages leave the two quotients and 16 of the ~270 bytes per cell out
    const bool wantDt = stageWantsDt(p, a);
    uint32_t cfN[S] = {};
    auto loadCellIn = [&](uint32_t c) {
        if (wantDt) { metN[0] = m.cper[c]; metN[1] = m.cd[c]; }
        metN[2] = m.nia[c];
        if (wantQn) ld4(a.qn, c, qnN);
        if (wantQi) ld4(a.qin, c, qiN);
        if (wantAcc) ld4(a.acc, c, acN);
        if (wantRef) refN = m.refId[c];
    };
    auto loadCf = [&](uint32_t k) {
#pragma unroll
        for (int j = 0; j < S; j++) cfN[j] = t.cf[size_t(d.z + k) * S + j];
    };
    if (tid < nC) { loadCellIn(giNext); loadCf(tid); }
    ldsBarrier();
    double dtCand = INFINITY, rCand = 0.0;
    // uniform trip count: the RMS leaf sums need every lane of a 16-lane group
    for (uint32_t k0 = 0; k0 < nC; k0 += BLK) {
        const uint32_t k = k0 + tid;
        const bool have = k < nC;
        double qNew[4] = {0, 0, 0, 0}, qOld[4] = {0, 0, 0, 0};
        uint32_t gi = giNext;
        double met[3], qnC[4], qiC[4], acC[4];
#pragma unroll
        for (int x = 0; x < 3; x++) met[x] = metN[x];
#pragma unroll
        for (int x = 0; x < 4; x++) { qnC[x] = qnN[x]; qiC[x] = qiN[x]; acC[x] = acN[x]; }
        const uint32_t refC = refN;
        uint32_t cfC[S];
#pragma unroll
        for (int j = 0; j < S; j++) cfC[j] = cfN[j];
        if (k + BLK < nC) {
            giNext = giNext2;
            if (k + 2 * BLK < nC) giNext2 = t.ids[d.z + k + 2 * BLK];
            loadCellIn(giNext);
            loadCf(k + BLK);
        }
        if (have) {
            double r[4] = {0.0, 0.0, 0.0, 0.0};
            double sAve = 0;
#pragma unroll
            for (int j = 0; j < S; j++) {
                const uint32_t fe = cfC[j];
                double lf[5];
                fl.get(fe & 0x7fffu, lf);
                if (fe >> 15) { r[0] = r[0] - lf[0]; r[1] = r[1] - lf[1]; r[2] = r[2] - lf[2]; r[3] = r[3] - lf[3]; }
                else { r[0] = r[0] + lf[0]; r[1] = r[1] + lf[1]; r[2] = r[2] + lf[2]; r[3] = r[3] + lf[3]; }
                sAve += lf[4];
            }
            switch (a.kind) {
            case SK_EULER: cellStage<SK_EULER>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, qNew, qOld, qnC, acC, wantDt); break;
            case SK_RK2_1: cellStage<SK_RK2_1>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, nullptr, nullptr, qnC, acC, wantDt); break;
            case SK_RK2_2: cellStage<SK_RK2_2>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, qNew, qOld, qnC, acC, wantDt); break;
            case SK_TVD_1: cellStage<SK_TVD_1>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, nullptr, nullptr, qnC, acC, wantDt); break;
            case SK_TVD_2: cellStage<SK_TVD_2>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, qNew, qOld, qnC, acC, wantDt); break;
            case SK_RK4_1: cellStage<SK_RK4_1>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, nullptr, nullptr, qnC, acC, wantDt); break;
            case SK_RK4_2: cellStage<SK_RK4_2>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, nullptr, nullptr, qnC, acC, wantDt); break;
            case SK_RK4_3: cellStage<SK_RK4_3>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, nullptr, nullptr, qnC, acC, wantDt); break;
            case SK_RK4_4: cellStage<SK_RK4_4>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, qNew, qOld, qnC, acC, wantDt); break;
            default: cellStage<SK_RESIDUAL>(m, p, a, gi, r, sAve, qiC, met, dtCand, rCand, nullptr, nullptr, qnC, nullptr, wantDt); break;
            }
        }
        if (a.rmsBlocks) rmsBlockLeaf(have, qNew, qOld, have ? refC : 0u, a.rmsBlocks);
    }
    blockPartial(dtCand, rCand, a.partial, pslot);
}

// Whether a face's flux by the FAST forms stands: what is outside their range (a zero or infinite
// denominator, a density or sound speed below FastRange's) has reached it as a NaN or as a value
// beyond any flow's.  The forms with a guard on every quotient took longer than plain
// divisions; this one test took the 4.2M-cell viscous Rusanov launches from 295 to 265-278 us
// (VALU issue was ~155 us of them; they take 245 and 265 now, with 108 and 122 us of issue) and a
// 299,266-cell Roe launch from 33.6 to 32.4 us (26.5 now).
template <typename R>
DEV bool fluxInRange(const R F[4])
{
    constexpr R big = sizeof(R) == 8 ? R(1e100) : R(1e18);
    return fabs(F[0]) < big && fabs(F[1]) < big && fabs(F[2]) < big && fabs(F[3]) < big;
}

// An interior face by the IEEE forms, its rows loaded again: the fast path's registers do not
// keep them for it (the opaque record stops the compiler from doing so).
template <int FLUX, int VISC, int ORDER, int LP, int MIX>
DEV void exactFace(const DevMesh& m, const PhysParams& p, const FaceSrc<MIX>& src, uint4 r,
                   typename FaceSrc<MIX>::R F[4], typename FaceSrc<MIX>::R& sMax)
{
    using R = typename FaceSrc<MIX>::R;
    asm volatile("" : "+v"(r.x), "+v"(r.y), "+v"(r.z), "+v"(r.w));
    double2 n, mid, ca = make_double2(0, 0), cb = make_double2(0, 0);
    double len;
    edgeGeometry(true, m.node[r.z], m.node[r.w], n, mid, len);
    R qa[4], qb[4], ga[8], gb[8], lxa[4], lya[4], lxb[4], lyb[4], qL[4], qR[4];
    src.q(r.x, qa);
    src.q(r.y, qb);
    if (ORDER > 1 || VISC) { src.grad(r.x, ga); src.grad(r.y, gb); }
    if (ORDER > 1) {
        src.template lim<LP>(r.x, lxa, lya);
        src.template lim<LP>(r.y, lxb, lyb);
        ca = m.cen[r.x];
        cb = m.cen[r.y];
    }
    interiorFace<FLUX, VISC, ORDER, LP, R>(qa, ga, lxa, lya, ca, qb, gb, lxb, lyb, cb, n, mid, p, qL, qR, F, sMax);
}

// One workgroup of the face/update kernel on tile `tile` of its mesh, leaving its (min dt,
// max |R|) pair in partial slot `pslot` (the solo and the batched kernels run this same code).
template <int S, int FLUX, int VISC, int ORDER, int LP, int MIX>
DEV void faceTileBody(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t,
                      uint32_t tile, uint32_t pslot, double* fsd)
{
    using R = typename std::conditional<MIX == 1, float, double>::type;
    const FaceSrc<MIX> src{a};
    const FaceLds<MIX> fl(fsd, t.faceStride + 1);
    const uint32_t tid = threadIdx.x;
    // The first two cell rounds' ids are loaded ahead of the faces; the next round's
    // face record is loaded one round ahead, so each round waits for one memory latency
    // (cell data) instead of two (record, then cell data).  The tile's arrays start at
    // fixed strides, so these first loads are issued beside the descriptor's instead of
    // after it (lanes past the tile's counts read padding and do not use it).
    uint32_t giNext = t.ids[size_t(tile) * t.cellStride + tid];
    uint32_t giNext2 = t.ids[size_t(tile) * t.cellStride + tid + BLK];
    uint4 rNext = t.fref[size_t(tile) * t.faceStride + tid];
    const uint4 d = t.desc[tile];
    // the loop's active flag is read after those loads are issued (all in bounds)
    if (!fluxRuns(a, pslot == 0 && tid == 0)) return;
    const uint32_t nF = d.y;
    for (uint32_t k = tid; k < nF; k += BLK) {
        const uint4 r = rNext;   // cell a, cell b, node 0, node 1
        if (k + BLK < nF) rNext = t.fref[d.w + k + BLK];
        const bool interior = r.y < m.N;
        // every load of the face is issued before its arithmetic, with no branch between
        // them, so the round waits for one memory latency.  Side b of a boundary face is
        // its ghost (cell N + b), which has a state and a centroid but no gradient or
        // limiter row: the owner's row is read in its place and not used.
        const double2 p0 = m.node[r.z], p1 = m.node[r.w];
        const uint32_t rb = interior ? r.y : r.x;
        R qa[4], qb[4], ga[8], gb[8], lxa[4], lya[4], lxb[4], lyb[4];
        src.q(r.x, qa);
        src.q(r.y, qb);
        if (ORDER > 1 || VISC) { src.grad(r.x, ga); src.grad(rb, gb); }
        double2 ca = make_double2(0, 0), cb = make_double2(0, 0);
        if (ORDER > 1) {
            src.template lim<LP>(r.x, lxa, lya);
            src.template lim<LP>(rb, lxb, lyb);
            ca = m.cen[r.x]; cb = m.cen[r.y];
        }
        double2 n, mid;
        double len;
        edgeGeometry<1>(interior, p0, p1, n, mid, len);
        R qL[4], qR[4], Fr[4], sMr;
        bool isB = false;
        uint32_t b = 0;
        if (interior) {
            interiorFace<FLUX, VISC, ORDER, LP, R, 1>(qa, ga, lxa, lya, ca, qb, gb, lxb, lyb, cb, n, mid, p, qL, qR,
                                                     Fr, sMr);
            if (!fluxInRange(Fr)) exactFace<FLUX, VISC, ORDER, LP, MIX>(m, p, src, r, Fr, sMr);
        } else {
            isB = true;
            b = r.y - m.N;   // the ghost of boundary face b is cell N + b
            boundaryFace<FLUX, VISC, ORDER, LP, R>(qa, ga, lxa, lya, ca, qb, m.bface[b], n, mid, p, qL, qR, Fr, sMr);
        }
        // the residual is accumulated in FP64 from len * flux on either path
        const double F[4] = {double(Fr[0]), double(Fr[1]), double(Fr[2]), double(Fr[3])}, sMax = double(sMr);
        if (isB) {
            // boundary faces (each in exactly one tile) feed the force integral
            const uint32_t f = m.Fi + b;
            *reinterpret_cast<double4*>(a.lenF + size_t(f) * 4) =
                make_double4(len * F[0], len * F[1], len * F[2], len * F[3]);
            a.lenS[f] = len * sMax;
        }
        // boundary edges are checked first in the reference: their keys come first
        if (a.recordErrors && (isnan(F[0]) || isnan(F[1]) || isnan(F[2]) || isnan(F[3])))
            atomicMin(&a.sc->errEdge,
                      (uint64_t(a.stageId) << 32) | (isB ? uint64_t(b) : uint64_t(m.Fb) + t.fid[d.w + k]));
        if constexpr (MIX == 1) fl.put(k, len, Fr, sMr);
        else fl.put(k, len, F, sMax);
    }
    fl.zero(nF, tid);   // padding face
    tileCellPhase<S, MIX>(m, p, a, t, d, pslot, fl, giNext, giNext2);
}

}  // namespace ebb
