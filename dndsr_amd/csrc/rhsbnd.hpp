// rhsbnd.hpp -- the inviscid boundary-face fluxes of EvaluateRHS, shared by its face kernels.
#pragma once
#include "gas.hpp"
#include "internal.hpp"

namespace dndsr
{
// the stage's time step (StageUpdate), in two steps: the lane's loads, and the minimum over the
// wavefront, whose lanes all take part
__device__ __forceinline__ real stageDtLane(const StageUpdate &st)
{
    if (st.nPart == 0)
        return st.dtDev ? st.dtDev[0] : 1.0;
    real d = 3e200;
    for (int q = threadIdx.x & 63; q < st.nPart; q += 64)
        d = fmin(d, st.dtDev[q]);
    return d;
}
__device__ __forceinline__ real stageDtJoin(const StageUpdate &st, real d)
{
    if (st.nPart == 0)
        return d;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1)
        d = fmin(d, __shfl_xor(d, s));
    return d;
}
struct StageIn
{
    real x, y;
};
__device__ __forceinline__ StageIn stageLoad(const StageUpdate &st, size_t o)
{
    return {st.u ? st.u[o] : 0.0, st.u && st.y ? st.y[o] : 0.0};
}
// same arithmetic as kAxpby(a, u, b, y, cdt, rhs, dt) at offset o
__device__ __forceinline__ void stageStore(const StageUpdate &st, size_t o, const StageIn &in, real rhs, real dt)
{
    if (st.save)
        st.save[o] = in.x;
    real r = st.a * in.x;
    if (st.y)
        r += st.b * in.y;
    r += st.cdt * (rhs * dt);
    st.out[o] = r;
}

// Boundary faces (EvaluateRHS.hxx:194-207, 336-345), run after the tile kernel and overwriting the
// tile kernel's flux of that face.  The Roe average takes the cell mean and its ghost at the face
// centre (mean normal); every point takes the reconstructed state and its ghost at the point normal;
// dLambda is the owner cell's.  A few thousand faces leave most of the device idle and the pass is
// one chain of dependent loads and flux arithmetic, so a block is 64 faces with one wavefront per
// point (the face constants formed by each); the point fluxes meet in LDS and are summed in point
// order as in the tile kernels.
template <int DIM, int NDOF, int G, int RS, bool BATCH>
__global__ void __launch_bounds__(64 * G) kRHSBoundary(DevMesh m, GasParams gp, const real *__restrict__ u,
                                                       const real *__restrict__ uRec, const real *__restrict__ dlc,
                                                       real *__restrict__ fflux)
{
    constexpr int M = NDOF - 1;
    __shared__ real sF[G * 5][64];
    const int lane = threadIdx.x % 64, g = waveIndex(64);
    const idx t = blockIdx.x * 64 + lane;
    const bool valid = t < m.nBnd;
    const idx f = m.bndFace[valid ? t : m.nBnd - 1];
    const FacePts fp = bndPts(m, valid ? t : m.nBnd - 1);
    const size_t N = m.N, F = m.F;
    const idx cL = m.f2c[f];
    const int zone = m.fzone[f];
    real ULm[5], URm[5], UL[5], UR[5], nm[3], n[3], x[3];
#pragma unroll
    for (int r = 0; r < 3; r++)
    {
        nm[r] = m.fmeanN[(size_t)r * F + f];
        n[r] = fp.n(g, r);
        x[r] = fp.x(g, r);
    }
    const real wj = fp.w(g);
    const int type = m.bcType[zone];
    const real *far = m.bcVal + (size_t)zone * 5;
#pragma unroll
    for (int v = 0; v < 5; v++)
        UL[v] = ULm[v] = u[(size_t)v * N + cL];
    const real dLambda = dlc ? dlc[cL] : 0.0;
    if (uRec)
    {
        real xs[3], mom[M > 0 ? M : 1], phi[M > 0 ? M : 1];
#pragma unroll
        for (int j = 0; j < M; j++)
            mom[j] = m.moment[(size_t)j * N + cL];
        const real isc = m.iscale[cL];
#pragma unroll
        for (int r = 0; r < 3; r++)
        {
            xs[r] = x[r] - m.cent[(size_t)r * N + cL];
            if (DIM == 3 || r < 2)
                xs[r] *= isc;
        }
        basisRow0<DIM, NDOF>(xs, mom, phi);
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            real sacc = 0;
#pragma unroll
            for (int j = 0; j < M; j++)
                sacc += phi[j] * uRec[((size_t)v * M + j) * N + cL];
            UL[v] += sacc;
        }
    }
    bcGhost(type, ULm, nm, far, gp.gamma, URm);
    bcGhost(type, UL, n, far, gp.gamma, UR);
    real Fl[5];
    if constexpr (BATCH)
    {
        RoeBatchFace bf;
        roeBatchSetup<RS>(ULm, URm, nm, gp, dLambda, bf);
        roeBatchPoint<RS>(UL, UR, n, gp, bf, Fl);
    }
    else
    {
        RoeAve ra;
        real l0, l1, l4;
        roeAverage(ULm, URm, gp.gamma, ra);
        riemannFluxR<RS>(UL, UR, ra, n, gp, dLambda, Fl, l0, l1, l4);
    }
#pragma unroll
    for (int v = 0; v < 5; v++)
        sF[g * 5 + v][lane] = (-Fl[v]) * wj;
    __syncthreads();
    for (int v = g; v < 5; v += G)
    {
        real acc = 0;
#pragma unroll
        for (int q = 0; q < G; q++)
            acc += sF[q * 5 + v][lane];
        if (valid)
            fflux[(size_t)v * F + f] = acc;
    }
}
template <int DIM, int NDOF, int G, int RS, bool BATCH>
static void rhsBoundaryLaunch(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc, real *ff)
{
    if (c.m.nBnd == 0)
        return;
    kRHSBoundary<DIM, NDOF, G, RS, BATCH><<<gridFor(c.m.nBnd, 64), 64 * G, 0, c.stream>>>(c.m, gp, u, uRec, dlc, ff);
    DNDSR_HIP_CHECK(hipGetLastError());
}
} // namespace dndsr
