// The epilogue of a time-loop step (app/solver.d:122-247): RMS residuals, newDt and Rmax, the
// boundary force, cflAdjust, dt, the history row and the stop conditions.  It runs as a few
// extra workgroups of the next step's first gradient kernel (or as a launch of its own at the
// end of a run): nothing in that kernel needs its results, only the tile kernel after it does.
#pragma once
#include "device.hpp"

namespace ebb {

// Phobos std.algorithm.sum over double[] (app/solver.d:153-168): 16-element blocks summed by a
// fixed tree (the leaf blocks, left by the step's last stage), blocks merged by a binary counter
// (perfect pairwise trees over aligned power-of-two runs), remainder elements likewise, and the
// counter's stack folded from the top, which is smallest tree first.  Quantities 0..3: sum of
// (now-last)^2 per variable; 4..7: sum of now.
//
// The code runs once per step in a handful of workgroups, so its length counts: straight-line it
// took 36 KB and 10-20 us, mostly waiting for instructions.  Each of the four waves takes two
// quantities, a lane sixteen consecutive items, and the levels above are loops over shuffles.
constexpr int EPT = 256;                        // threads of an epilogue workgroup
typedef double sum2 __attribute__((ext_vector_type(2)));   // a wave's two quantities

struct EpiLds {
    double stack[8][16];                        // meshes of more than 1,024 full chunks
    double tot[8];
    double red[EPT / 64][2];
    double fsum[2];
    int last;
};
// The force staging shares its LDS with the gradient rows of the kernel it runs in.
constexpr int FORCE_LDS = 1024;                 // force faces staged per pass

DEV void agentStore(double* p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
DEV double agentLoad(const double* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

DEV sum2 shfl2(sum2 v, int lane) { return sum2{__shfl(v.x, lane, 64), __shfl(v.y, lane, 64)}; }

// the fold of the binary counter's stack (empty until `any`)
struct Fold {
    sum2 s = {0, 0};
    bool any = false;
    DEV void add(sum2 v)
    {
        s = any ? s + v : v;
        any = true;
    }
};

template <int CTRL>
DEV sum2 rowSwap2(sum2 v) { return sum2{rowSwap<CTRL>(v.x), rowSwap<CTRL>(v.y)}; }

// The perfect trees of n items (lane l holds item l, n < 2^levels or all 2^levels), smallest
// first: for every set bit j of n, the tree over the aligned run of 2^j items that the binary
// counter keeps at level j.  The xor butterfly adds exactly as the pairwise tree does (the two
// orders of each sum are equal); within a row it runs on DPP moves, and a tree's value is read from
// its lane (n is the same in every lane): LDS permutes took 0.1 us a level in this chain.
DEV void foldLanes(sum2 x, uint32_t n, int levels, Fold& f)
{
    if (n == 0) return;
    auto take = [&](int j) {
        const int l = int((n >> (j + 1)) << (j + 1));
        if (n >> j & 1u) f.add(sum2{laneValue(x.x, l), laneValue(x.y, l)});
    };
    take(0);
    x += rowSwap2<ROW_X1>(x);
    take(1);
    x += rowSwap2<ROW_X2>(x);
    take(2);
    x += rowSwap2<ROW_X4>(x);
    take(3);
    x += rowSwap2<ROW_X8>(x);
#pragma unroll 1
    for (int j = 4; j < levels && n >> j; j++) {
        take(j);
        x += shfl2(x, int((threadIdx.x & 63u) ^ (1u << j)));
    }
    if (n >> levels) f.add(x);
}

// The trees of cnt <= 1,024 items of 8 quantities each, for this wave's two quantities.  AGENT: the
// items were written in this launch.
template <bool AGENT>
DEV void foldItems(const double* items, uint32_t cnt, Fold& f)
{
    const uint32_t lane = threadIdx.x & 63u, n16 = cnt >> 4, tail = cnt & 15u;
    items += threadIdx.x / 64 * 2;
    auto load = [](const double* p) {
        if (AGENT) return sum2{agentLoad(p), agentLoad(p + 1)};
        return *reinterpret_cast<const sum2*>(p);
    };
    sum2 y = {0, 0}, g = {0, 0};
    if (lane < tail) y = load(items + size_t(n16) * 128 + lane * 8);
    if (n16 == 0) {
        foldLanes(y, tail, 4, f);
        return;
    }
    // a lane's sixteen items, eight at a time: the registers of sixteen would cost the gradient
    // kernel waves in mixed precision (94 registers, set by this code)
#pragma unroll 1
    for (int h = 0; h < 2; h++) {
        sum2 x[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) x[u] = sum2{0, 0};
        if (lane < n16) {
#pragma unroll
            for (uint32_t u = 0; u < 8; u++) x[u] = load(items + size_t(lane) * 128 + h * 64 + u * 8);
        }
        x[0] = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
        g = h ? g + x[0] : x[0];
    }
    foldLanes(y, tail, 4, f);
    foldLanes(g, n16, 6, f);
}

// The boundary force sum of mesh.d:645-671: (len*flux) momentum components of the force faces
// added in order, x in lane 0 and y in lane 1 (their result), so each addition of a chain waits
// only for its own predecessor.  fp: LDS staging, FORCE_LDS values per component.
// fi: the first pass's ids, loaded (forceIds) before anything else of the epilogue was waited for.
constexpr int FS = FORCE_LDS / EPT;
DEV void forceIds(const uint32_t* faces, uint32_t nF, uint32_t k0, uint32_t fi[FS])
{
#pragma unroll
    for (int u = 0; u < FS; u++) {
        const uint32_t x = k0 + threadIdx.x + uint32_t(u) * EPT;
        fi[u] = x < nF ? faces[x] : 0u;
    }
}
DEV double orderedForce(const uint32_t* faces, uint32_t nF, const double* lenF, double* fp, uint32_t fi[FS])
{
    double f = 0;
    for (uint32_t k0 = 0; k0 < nF; k0 += FORCE_LDS) {
        const uint32_t cnt = (nF - k0) < uint32_t(FORCE_LDS) ? (nF - k0) : uint32_t(FORCE_LDS);
        __syncthreads();
        // all of a thread's face ids, then all of their fluxes, are loaded before any is
        // used: two round trips per pass instead of two per face
        if (k0) forceIds(faces, nF, k0, fi);
        double2 fv[FS];
#pragma unroll
        for (int u = 0; u < FS; u++) {
            const uint32_t x = threadIdx.x + uint32_t(u) * EPT;
            fv[u] = x < cnt ? make_double2(lenF[size_t(fi[u]) * 4 + 1], lenF[size_t(fi[u]) * 4 + 2])
                            : make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int u = 0; u < FS; u++) {
            const uint32_t x = threadIdx.x + uint32_t(u) * EPT;
            if (x < cnt) { fp[x] = fv[u].x; fp[FORCE_LDS + x] = fv[u].y; }
        }
        __syncthreads();
        if (threadIdx.x < 2) {
            const double* v = fp + threadIdx.x * FORCE_LDS;
            uint32_t x = 0;
            for (; x + 24 <= cnt; x += 24) {   // 24 LDS reads are in flight ahead of the adds
                double a[24];
#pragma unroll
                for (int u = 0; u < 24; u++) a[u] = v[x + u];
#pragma unroll
                for (int u = 0; u < 24; u++) f += a[u];
            }
            for (; x < cnt; x++) f += v[x];
        }
    }
    return f;
}

// newDt is the last stage's minimum (every stage overwrites it), Rmax the maximum over the
// step's stages; min and max are exact in any order.  Thread 0 gets the result.
DEV void stageReduce(const DiagArgs& d, double (*red)[2], double& newDt, double& rmax)
{
    // each pass issues all of a thread's loads before using any (the partials were written on all
    // XCDs: every load is a round trip past this XCD's L2)
    constexpr int SLOTS = 8;
    double a0 = INFINITY, b0 = 0.0;
    const uint32_t n = d.nPart * d.nStages, lastStage = n - d.nPart;
    for (uint32_t base = threadIdx.x; base < n; base += EPT * SLOTS) {
        sum2 pv[SLOTS];
#pragma unroll
        for (int u = 0; u < SLOTS; u++) {
            pv[u] = sum2{INFINITY, 0.0};
            if (base + u * EPT < n) pv[u] = reinterpret_cast<const sum2*>(d.partial)[base + u * EPT];
        }
#pragma unroll
        for (int u = 0; u < SLOTS; u++) {
            if (base + u * EPT >= lastStage) a0 = fmin(a0, pv[u].x);
            b0 = fmax(b0, pv[u].y);
        }
    }
    a0 = warpMin(a0);
    b0 = warpMax(b0);
    const uint32_t w = threadIdx.x / 64;
    if ((threadIdx.x & 63) == 0) { red[w][0] = a0; red[w][1] = b0; }
    __syncthreads();
    if (threadIdx.x == 0)
        for (uint32_t k = 1; k < EPT / 64; k++) { a0 = fmin(a0, red[k][0]); b0 = fmax(b0, red[k][1]); }
    newDt = a0;
    rmax = b0;
}

// the loop's scalars as the step's stages left them
struct StepScalars {
    double t, dt, CFL, residLast, rms0;
    int64_t steps, incIters;
    bool failed;
};
DEV StepScalars loadScalars(const DevScalars* sc)
{
    return {sc->t, sc->dt, sc->CFL, sc->residLast, sc->rms0, sc->steps, sc->incIters,
            sc->errEdge != ~0ull || sc->errCell != ~0ull || sc->errBC != ~0ull};
}

// the same in every lane: in scalar registers, not in the vector registers that set the gradient
// kernel's occupancy
DEV double uniform(double v) { return laneValue(v, 0); }
DEV int64_t uniform(int64_t v)
{
    return int64_t(uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint64_t(v) >> 32)))) << 32 |
                   uint32_t(__builtin_amdgcn_readfirstlane(int(v))));
}
DEV StepScalars uniform(const StepScalars& s)
{
    return {uniform(s.t), uniform(s.dt), uniform(s.CFL), uniform(s.residLast), uniform(s.rms0), uniform(s.steps),
            uniform(s.incIters), __builtin_amdgcn_readfirstlane(int(s.failed)) != 0};
}

// The remainder's and the partial chunk's trees (ghost slots hold zeros in both states).
DEV void foldTail(const DiagArgs& d, Fold& f)
{
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x / 64, v = (w & 1u) * 2;
    const uint64_t nb = uint64_t(d.L) / 16, full = nb / RMS_CHUNK_BLOCKS * RMS_CHUNK_BLOCKS, e = nb * 16 + lane;
    const uint32_t rem = uint32_t(uint64_t(d.L) - nb * 16);
    sum2 x = {0, 0};
    if (lane < rem && e < d.N) {
        const uint32_t dv = d.perm ? d.perm[e] : uint32_t(e);
        x = *reinterpret_cast<const sum2*>(reinterpret_cast<const double*>(d.qnew + dv) + v);
        if (w < 2) {
            x -= *reinterpret_cast<const sum2*>(reinterpret_cast<const double*>(d.qold + dv) + v);
            x *= x;
        }
    }
    foldLanes(x, rem, 4, f);
    foldItems<false>(d.blockSums + full * 8, uint32_t(nb - full), f);
}

// One workgroup, with the step's newDt, Rmax and force sums at hand and f folded over the
// remainder and the partial chunk: folds the full chunks' tops, writes the history row and the
// loop's scalars and applies the stop conditions.
DEV void finishStep(const DiagArgs& d, const StepScalars& s0, EpiLds& L, Fold f, double newDt, double Rmax, double f0, double f1)
{
    DevScalars* sc = d.sc;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, q0 = tid / 64 * 2;
    const uint32_t nfull = uint32_t(uint64_t(d.L) / 16 / RMS_CHUNK_BLOCKS);
    if (nfull && nfull <= 1024) {
        foldItems<true>(d.chunkTops, nfull, f);
    } else if (nfull && lane < 2) {
        // very large meshes: the counter replayed over the chunk tops
        double* st = L.stack[q0 + lane];
        int idx = 0;
        for (uint32_t k = 0; k < nfull; k++) {
            st[idx] = agentLoad(d.chunkTops + size_t(k) * 8 + q0 + lane);
            const int last = idx - __builtin_ctz(k + 1);
            while (idx > last) { st[idx - 1] += st[idx]; --idx; }
            ++idx;
        }
        while (idx > 0) { --idx; f.add(sum2{st[idx], st[idx]}); }   // this lane's quantity in its own component
    }
    if (lane < 2) L.tot[q0 + lane] = 0.0 + (lane ? f.s.y : f.s.x);
    __syncthreads();
    if (tid >= 64) return;
    const double r = sqrt(double(d.N) * L.tot[lane & 3u]) / L.tot[4 + (lane & 3u)];
    const double rms[4] = {__shfl(r, 0, 64), __shfl(r, 1, 64), __shfl(r, 2, 64), __shfl(r, 3, 64)};
    if (tid != 0) return;
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
        h[6] = Rmax; h[7] = ld0; h[8] = ld1; h[9] = CFL;
    }
    const double t1 = s0.t + dt;
    const int64_t steps1 = s0.steps + 1;
    sc->newDtBits = (unsigned long long)__double_as_longlong(newDt);
    sc->rmaxBits = (unsigned long long)__double_as_longlong(Rmax);
    sc->dt = dt;
    sc->incIters = inc;
    sc->CFL = CFL;
    sc->residLast = residMax;
#pragma unroll
    for (int q = 0; q < 4; q++) sc->rms[q] = rms[q];
    sc->force[0] = ld0; sc->force[1] = ld1;
    sc->t = t1;
    sc->steps = steps1;
    // convergence stop (extensions.rmsDrop): the rho RMS residual of app/solver.d:153-168 has
    // dropped by the given factor below its value on the first step
    const double rms0 = s0.steps == 0 ? rms[0] : s0.rms0;
    sc->rms0 = rms0;
    const bool converged = d.rmsDrop > 0 && rms[0] <= d.rmsDrop * rms0;
    if (converged) sc->converged = 1;
    if (!(t1 < d.tEnd) || (d.maxSteps >= 0 && steps1 >= d.maxSteps) || s0.failed || converged)
        sc->active = 0;
}

// Workgroup wg of a step's epilogue (d.nEpi of them).  No full chunk of leaf blocks: a single
// workgroup does all of it.  Otherwise workgroup 0 sums the force, 1 reduces the stage partials,
// 2 folds the remainder and the partial chunk, 3.. one full chunk each, and the last of them to
// finish merges the results.  What they hand over goes through agent-scope stores and loads, which
// pass the XCDs' own L2s, and each wave waits for its stores before the workgroup draws its
// ticket; a __threadfence() instead would write back an L2 full of the gradients of the workgroups
// beside it (6 us longer under the 27 us gradient launch of 1M cells in mixed precision).
// staging: 2 * FORCE_LDS doubles of LDS.
DEV void epilogueBody(const DiagArgs& d, uint32_t wg, EpiLds& L, double* staging)
{
    DevScalars* sc = d.sc;
    const bool single = d.nEpi == 1;
    uint32_t fi[FS] = {};
    if (single || wg == 0) forceIds(d.forceFaces, d.nForce, 0, fi);
    if (!sc->active) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, q0 = tid / 64 * 2;
    const uint64_t nb = uint64_t(d.L) / 16;
    const uint32_t nfull = uint32_t(nb / RMS_CHUNK_BLOCKS);
    double newDt = 0, rmax = 0;
    Fold f;
    if (single || wg == 1) stageReduce(d, L.red, newDt, rmax);
    if (single || wg == 2) foldTail(d, f);
    else if (wg > 2) foldItems<false>(d.blockSums + size_t(wg - 3) * RMS_CHUNK_BLOCKS * 8, RMS_CHUNK_BLOCKS, f);
    StepScalars s0{};
    if (single) s0 = loadScalars(sc);
    if (single || wg == 0) {
        const double s = orderedForce(d.forceFaces, d.nForce, d.lenF, staging, fi);
        if (tid < 2) L.fsum[tid] = s;
        __syncthreads();
    }
    if (!single) {
        double* tops = d.chunkTops + size_t(wg == 2 ? nfull : wg - 3) * 8;
        if (wg >= 2 && lane < 2) agentStore(tops + q0 + lane, lane ? f.s.y : f.s.x);
        if (wg == 0 && tid < 2) agentStore(&sc->fsum[tid], L.fsum[tid]);
        if (wg == 1 && tid == 0) { agentStore(&sc->stageSum[0], newDt); agentStore(&sc->stageSum[1], rmax); }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's agent-scope stores have completed
        __syncthreads();
        if (tid == 0)
            L.last = __hip_atomic_fetch_add(&sc->ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == d.nEpi;
        __syncthreads();
        if (!L.last) return;
        if (tid == 0) sc->ticket = 0;
        // the scalars and what the others handed over arrive together
        s0 = loadScalars(sc);
        const double* tail = d.chunkTops + size_t(nfull) * 8 + q0;
        f.s = sum2{agentLoad(tail), agentLoad(tail + 1)};
        f.any = uint64_t(nfull) * RMS_CHUNK_BLOCKS * 16 != d.L;
        newDt = agentLoad(&sc->stageSum[0]);
        rmax = agentLoad(&sc->stageSum[1]);
        if (tid < 2) L.fsum[tid] = agentLoad(&sc->fsum[tid]);
        __syncthreads();
    }
    s0 = uniform(s0);
    finishStep(d, s0, L, f, newDt, rmax, L.fsum[0], L.fsum[1]);
}

}  // namespace ebb
