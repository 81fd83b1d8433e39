// facelin.hip -- face fluxes of EvaluateRHS with a linear (or no) reconstruction, one pass over the
// interior faces: the Riemann flux and, in a viscous run with one normal per face, the Navier-Stokes flux
// (EulerEvaluator_EvaluateRHS.hxx:171-662, EvaluateDt.hxx:1163-1215).
//
// One thread per face (lane = face), no LDS and no barrier.  A linear reconstruction needs few values
// per side: the basis row times the coefficients is G (x - cent - scale moment), G = uRec / scale, so a
// side is its mean u, the gradient G and the offset (26 values in 3-D, 23 on tetrahedra), read once and
// reduced at once to its states at the face's points (on a triangle, whose points are affine
// combinations of its vertices, to the mean, the offset at one vertex and the changes along two sides: the
// mean is added point by point, a state rounded once for all six points shifted the whole face's flux and
// raised the residual's error by half); of the gradients only the mean of the two sides lives on, for the
// viscous flux.  The tile kernels of the higher orders, one wavefront per point
// and the sides staged in LDS, re-read 80 rows of it there and left the viscous flux to a second pass
// with all its gathers.
//
// On a triangle the unit normal is one for the face, its six weights are two values, and the points come
// from the vertices, so 14 values per face replace the 42 of the point tables (normal and weights are
// read from those tables: the mean normal and the area carry a rounding of their own).  Each side's rows of
// u and uRec are read as they stand: 160-byte cell records written by a pass of their own before were
// slower in every cell order (384k tetrahedra, viscous residual: Morton order 151 us with records, 121
// with rows; grouped by colour 178 / 165; reverse Cuthill-McKee 166 / 131).
//
// Measured: 945k tetrahedra (1.9M faces), viscous Roe: 199 us, against 288 us (tile kernel) + 424 us
// (viscous pass); 333k faces of a mixed 2-D mesh, viscous Roe: 26 us against 33 + 37 us; 744k hexahedral
// faces, inviscid Roe: 77 us against 84 us.
#include "geom.hpp"
#include "rhsbnd.hpp"

namespace dndsr
{
struct ViscGas
{
    real g1, Cp, kOverMu;
};
// Navier-Stokes flux at a point (viscousPointFlux of gas.hpp with the mean gradient given and its
// quotients by the density taken as products with one reciprocal): Gm + n (UR - UL) idist is the
// gradient, Gm the mean of the two sides'
template <int DIM>
__device__ __forceinline__ void viscousPointLin(const GasParams &gp, const ViscGas &vg, const real *UL, const real *UR,
                                                const real (&Gm)[DIM][5], const real *n, real idist, real *Fv)
{
    real U[5], jump[5];
#pragma unroll
    for (int v = 0; v < 5; v++)
        U[v] = 0.5 * (UL[v] + UR[v]), jump[v] = (UR[v] - UL[v]) * idist;
    const real ri = rcpN(U[0]);
    const real vel[3] = {U[1] * ri, U[2] * ri, U[3] * ri};
    const real vSqr = dot3(vel, vel);
    const real p = vg.g1 * (U[4] - 0.5 * U[0] * vSqr);
    // velocity and temperature gradients: dv = (d(rho v) - v d rho) / rho,
    // dp = (gamma - 1) (dE - v . d(rho v) + |v|^2 d rho / 2), dT = c (rho dp - p d rho)
    real gv[3][3], gT[3];
    const real c = gp.gamma * ri * ri / (vg.g1 * vg.Cp);
#pragma unroll
    for (int d = 0; d < 3; d++)
    {
        real g[5];
#pragma unroll
        for (int v = 0; v < 5; v++)
            g[v] = (d < DIM ? Gm[d < DIM ? d : 0][v] : 0.0) + n[d] * jump[v];
        real vm = 0;
#pragma unroll
        for (int j = 0; j < 3; j++)
        {
            gv[d][j] = (g[1 + j] - vel[j] * g[0]) * ri;
            vm += vel[j] * g[1 + j];
        }
        const real dp = vg.g1 * (g[4] - vm + 0.5 * vSqr * g[0]);
        gT[d] = c * (U[0] * dp - p * g[0]);
    }
    const real mu = muEff(gp, U, gasTemperature(gp, p, U[0]));
    const real k = vg.kOverMu * mu;
    const real tr = (-2. / 3.) * mu * (gv[0][0] + gv[1][1] + gv[2][2]);
    real e = 0;
    Fv[0] = 0;
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        real s = tr * n[i];
#pragma unroll
        for (int j = 0; j < 3; j++)
            s += mu * (gv[i][j] + gv[j][i]) * n[j];
        Fv[1 + i] = s;
        e += s * vel[i] + k * gT[i] * n[i];
    }
    Fv[4] = e;
}

// the cells' constants: rows of 4 (tetrahedra, whose vertex mean is their barycentre: centre, 1 / scale) or
// of 8 (centre, 1 / scale, scale times moment, 0)
__global__ void __launch_bounds__(256) kLinCentre(DevMesh m, real *__restrict__ linC, int row)
{
    const idx i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m.N)
        return;
    const size_t N = m.N;
    real *o = linC + (size_t)i * row;
    for (int r = 0; r < 3; r++)
        o[r] = m.cent[r * N + i];
    o[3] = m.iscale[i];
    for (int r = 4; r < row; r++)
        o[r] = r < 4 + m.dim ? m.scale[i] * m.moment[(size_t)(r - 4) * N + i] : 0.0;
}
// distGRP of an interior face with one normal (EvaluateRHS.hxx:346-424)
__global__ void __launch_bounds__(256) kLinDist(DevMesh m, real *__restrict__ out)
{
    const idx f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= m.F)
        return;
    const size_t N = m.N, F = m.F;
    const idx cL = m.f2c[f], cR = m.f2c[F + f];
    out[f] = 1;
    if (cR < 0)
        return;
    real dn = 0;
    for (int r = 0; r < 3; r++)
        dn += ((m.bary[r * N + cR] - m.fshift[r * F + f]) - m.bary[r * N + cL]) * m.fmeanN[r * F + f];
    const real d0 = fmin(m.vol[cL], m.vol[cR]) / m.farea[f] * 2;
    out[f] = 1.0 / fmax(fmin(fabs(dn), d0 * 2), d0 * 0.25);
}

template <int DIM, bool TRI>
struct LinSide
{
    real u[5], G[DIM][5], c[3], d[DIM];
    __device__ __forceinline__ void load(const DevMesh &m, idx i, const real *__restrict__ u_,
                                         const real *__restrict__ uRec)
    {
        const size_t N = m.N;
#pragma unroll
        for (int r = 0; r < DIM; r++)
            d[r] = 0;
        if (uRec)
        {
            const double2 *q = reinterpret_cast<const double2 *>(m.linC + (size_t)i * (TRI ? 4 : 8));
            const double2 a = q[0], b = q[1];
            c[0] = a.x, c[1] = a.y, c[2] = b.x;
            if constexpr (!TRI)
            {
                const double2 e = q[2];
                d[0] = e.x, d[1] = e.y;
                if constexpr (DIM == 3)
                    d[DIM - 1] = reinterpret_cast<const real *>(q)[6];
            }
#pragma unroll
            for (int v = 0; v < 5; v++)
            {
                u[v] = ldu(u_ + (size_t)v * N, (uint32_t)i);
#pragma unroll
                for (int k = 0; k < DIM; k++)
                    G[k][v] = ldu(uRec + ((size_t)v * DIM + k) * N, (uint32_t)i) * b.y;
            }
            return;
        }
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            u[v] = ldu(u_ + (size_t)v * N, (uint32_t)i);
#pragma unroll
            for (int k = 0; k < DIM; k++)
                G[k][v] = 0;
        }
        c[0] = c[1] = c[2] = 0;
    }
    // the state at x: u + off, off = G (x - centre - scale moment), the small difference formed first
    __device__ __forceinline__ void off(const real *x, real *U) const
    {
        real e[DIM];
#pragma unroll
        for (int k = 0; k < DIM; k++)
            e[k] = (x[k] - c[k]) - d[k];
        along(e, U);
    }
    __device__ __forceinline__ void at(const real *x, real *U) const
    {
        off(x, U);
#pragma unroll
        for (int v = 0; v < 5; v++)
            U[v] += u[v];
    }
    __device__ __forceinline__ void along(const real *e, real *dU) const
    {
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            real a = 0;
#pragma unroll
            for (int k = 0; k < DIM; k++)
                a += G[k][v] * e[k];
            dU[v] = a;
        }
    }
};

static_assert(kTri6[2][0] == kTri6[2][1] && kTri6[2][0] == kTri6[2][2] && kTri6[2][3] == kTri6[2][4] &&
                  kTri6[2][3] == kTri6[2][5],
              "the weights of points 0-2 and 3-5");

// flux forms that read deltaLambdaCell (the H-correction fixes and HLLE+)
constexpr bool readsDeltaLambda(int rs) { return rs == RS_HLLEP || rs == RS_HLLEP_V1 || rs == RS_Roe_M6 || rs == RS_Roe_M8; }

// the flux of face f, times -1 and the area, summed over its points; false for a boundary face
template <int DIM, int G, int RS, bool BATCH, bool VIS, bool TRI>
__device__ __forceinline__ bool linFace(const DevMesh &m, const GasParams &gp, const real *__restrict__ u,
                                        const real *__restrict__ uRec, const real *__restrict__ dlc, idx f, idx cL, idx cR, real (&acc)[5])
{
    constexpr bool ONE_N = TRI || DIM == 2; // one normal per face
    static_assert(ONE_N || !VIS, "quadrilateral faces keep their own viscous pass");
    constexpr int NS = TRI ? 3 : G;
    const size_t F = m.F;
    const uint32_t fu = (uint32_t)f;
    // the points (or the vertices of a triangle), the (first point's) normal and the shift into the right
    // cell's frame
    real x[NS][3], n[3], sh[3];
    if constexpr (TRI)
    {
        idx nd[3];
#pragma unroll
        for (int k = 0; k < 3; k++)
            nd[k] = ldu(m.face2node + (size_t)k * F, fu);
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int r = 0; r < 3; r++)
                x[k][r] = ldu(m.coords + (size_t)r * m.nNode, (uint32_t)nd[k]);
    }
    else
#pragma unroll
        for (int k = 0; k < NS; k++)
#pragma unroll
            for (int r = 0; r < DIM; r++)
                x[k][r] = ldu(m.fpts + ((size_t)k * 3 + r) * F, fu);
#pragma unroll
    for (int r = 0; r < 3; r++)
    {
        sh[r] = ldu(m.fshift + (size_t)r * F, fu);
        if constexpr (ONE_N || BATCH)
            n[r] = ldu((ONE_N ? m.fnorm : m.fmeanN) + (size_t)r * F, fu);
    }
    real w0 = 0, w1 = 0, idist = 0;
    if constexpr (TRI)
        w0 = ldu(m.fwj, fu), w1 = ldu(m.fwj + (size_t)3 * F, fu);
    if constexpr (VIS)
        idist = ldu(m.linDist, fu);
    if (cR < 0) // boundary faces: kRHSBoundary and the viscous pass over the boundary list
        return false;
    real SL[NS][5], SR[NS][5], Gm[DIM][5], mL[5], mR[5];
    RoeBatchFace bf;
    {
        LinSide<DIM, TRI> L, R;
        L.load(m, cL, u, uRec);
        R.load(m, cR, u, uRec);
#pragma unroll
        for (int k = 0; k < NS; k++)
        {
            if (TRI && k > 0) // a triangle: the offset at its first vertex and the changes along two sides
            {
                const real e[3] = {x[k][0] - x[0][0], x[k][1] - x[0][1], x[k][2] - x[0][2]};
                L.along(e, SL[k]);
                R.along(e, SR[k]);
                continue;
            }
            real xr[3];
#pragma unroll
            for (int r = 0; r < DIM; r++)
                xr[r] = x[k][r] + sh[r];
            if constexpr (TRI)
            {
                L.off(x[k], SL[k]);
                R.off(xr, SR[k]);
#pragma unroll
                for (int v = 0; v < 5; v++)
                    mL[v] = L.u[v], mR[v] = R.u[v];
            }
            else
            {
                L.at(x[k], SL[k]);
                R.at(xr, SR[k]);
            }
        }
        if constexpr (VIS)
#pragma unroll
            for (int d = 0; d < DIM; d++)
#pragma unroll
                for (int v = 0; v < 5; v++)
                    Gm[d][v] = 0.5 * (L.G[d][v] + R.G[d][v]);
        if constexpr (BATCH)
            roeBatchSetup<RS>(L.u, R.u, n, gp,
                              dlc && readsDeltaLambda(RS) ? fmax(dlc[cL], dlc[cR]) : 0.0, bf);
        else
            roeAverage(L.u, R.u, gp.gamma, bf.r);
    }
    real dLambda = 0;
    if constexpr (!BATCH && readsDeltaLambda(RS))
        if (dlc)
            dLambda = fmax(dlc[cL], dlc[cR]);
    const real Cp = cpGas(gp);
    const ViscGas vg{gp.gamma - 1, Cp, Cp / gp.prGas};
    // state, weight and (where it varies) normal of point g
    auto point = [&](int g, real *UL, real *UR, real &wj) {
        if constexpr (TRI)
        {
            const real b1 = kTri6[0][g], b2 = kTri6[1][g];
#pragma unroll
            for (int v = 0; v < 5; v++)
            {
                UL[v] = mL[v] + (SL[0][v] + (b1 * SL[1][v] + b2 * SL[2][v]));
                UR[v] = mR[v] + (SR[0][v] + (b1 * SR[1][v] + b2 * SR[2][v]));
            }
            wj = g < 3 ? w0 : w1;
        }
        else
        {
#pragma unroll
            for (int v = 0; v < 5; v++)
                UL[v] = SL[g < NS ? g : 0][v], UR[v] = SR[g < NS ? g : 0][v];
            wj = ldu(m.fwj + (size_t)g * F, fu);
            if constexpr (!ONE_N)
#pragma unroll
                for (int r = 0; r < 3; r++)
                    n[r] = ldu(m.fnorm + ((size_t)g * 3 + r) * F, fu);
        }
    };
#pragma unroll
    for (int v = 0; v < 5; v++)
        acc[v] = 0;
    // a triangle's points differ by three constants only: a loop (unrolled, six interleaved fluxes spill)
#pragma unroll TRI ? 1 : G
    for (int g = 0; g < G; g++)
    {
        real UL[5], UR[5], wj, Fl[5];
        point(g, UL, UR, wj);
        if constexpr (BATCH)
            roeBatchPoint<RS>(UL, UR, n, gp, bf, Fl);
        else
        {
            real l0, l1, l4;
            riemannFluxR<RS>(UL, UR, bf.r, n, gp, dLambda, Fl, l0, l1, l4);
        }
        if constexpr (VIS)
        {
            real Fv[5];
            viscousPointLin<DIM>(gp, vg, UL, UR, Gm, n, idist, Fv);
#pragma unroll
            for (int v = 1; v < 5; v++)
                Fl[v] -= Fv[v];
        }
#pragma unroll
        for (int v = 0; v < 5; v++)
            acc[v] -= Fl[v] * wj;
    }
    return true;
}

template <int DIM, int G, int RS, bool BATCH, bool VIS, bool TRI>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
kRHSFaceLin(DevMesh m, GasParams gp, const real *__restrict__ u, const real *__restrict__ uRec,
            const real *__restrict__ dlc, real *__restrict__ fflux)
{
    const idx f = xcdTile(blockIdx.x, gridDim.x) * 64 + (idx)threadIdx.x;
    if (f >= m.F)
        return;
    const idx cL = ldu(m.f2c, (uint32_t)f), cR = ldu(m.f2c + m.F, (uint32_t)f);
    real acc[5];
    if (!linFace<DIM, G, RS, BATCH, VIS, TRI>(m, gp, u, uRec, dlc, f, cL, cR, acc))
        return;
#pragma unroll
    for (int v = 0; v < 5; v++)
        stu(fflux + (size_t)v * m.F, (uint32_t)f, acc[v]);
}

// Small meshes: face fluxes, gather and stage combination in one pass.  Four lanes per cell, one per
// face slot, evaluate the cell's faces themselves (each face twice, by the same code from the same
// values, so both sides see the same flux) and combine the slots in order by shuffles, as kRHSGather
// does; boundary faces' fluxes come from the boundary passes before it.  Blocks read their neighbours'
// u, so the stage result goes to another array (st.out).  Bound by one chain of loads and flux arithmetic
// (6.5 us at 4 096 quadrilaterals, against 4.5 + 4.4 us and a launch gap for face pass and gather).
template <int DIM, int G, int RS, bool BATCH, bool VIS, bool TRI>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
kRHSCellLin(DevMesh m, GasParams gp, const real *__restrict__ u, const real *__restrict__ uRec,
            const real *__restrict__ dlc, const real *__restrict__ fflux, real *__restrict__ rhs, StageUpdate st,
            int *__restrict__ nonFinite)
{
    const int k = threadIdx.x & 3;
    const idx i = (idx)xcdTile(blockIdx.x, gridDim.x) * 16 + (threadIdx.x >> 2);
    const size_t N = m.N, F = m.F;
    const bool in = i < m.N && k < m.K;
    const size_t q = in ? (size_t)k * N + i : 0;
    const idx f = in ? m.c2f[q] : idx(-1), o = m.c2c[q];
    const bool right = (m.c2flag[q] & 1) != 0; // the cell is the face's right side
    // the lanes of a cell store one variable each, the first one also the fifth; what they need at the
    // end is loaded with the first loads, so that it is there when the flux chain ends
    const size_t own = i < m.N ? i : 0, o0 = (size_t)k * N + own, o4 = 4 * N + own;
    const real vol = m.vol[own];
    const StageIn s0 = stageLoad(st, o0), s4 = stageLoad(st, o4);
    real dt = st.u ? stageDtLane(st) : 1.0;
    real t[5] = {0, 0, 0, 0, 0}, w = 0;
    if (f >= 0)
    {
        w = right ? -1.0 : 1.0;
        if (!linFace<DIM, G, RS, BATCH, VIS, TRI>(m, gp, u, uRec, dlc, f, right ? o : i, right ? i : o, t))
#pragma unroll
            for (int v = 0; v < 5; v++)
                t[v] = fflux[v * F + f];
    }
    if (st.u)
        dt = stageDtJoin(st, dt);
    real acc[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++)
    {
        const real ws = __shfl(w, s, 4);
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            const real ts = __shfl(t[v], s, 4);
            if (ws != 0)
                acc[v] += ws * ts;
        }
    }
    if (i >= m.N)
        return;
#pragma unroll
    for (int v = 0; v < 5; v++)
        acc[v] /= vol;
    if (k == 0 && nonFinite &&
        !(isfinite(acc[0]) && isfinite(acc[1]) && isfinite(acc[2]) && isfinite(acc[3]) && isfinite(acc[4])))
        atomicOr(nonFinite, 1);
    const real a = k == 0 ? acc[0] : k == 1 ? acc[1] : k == 2 ? acc[2] : acc[3];
    if (rhs)
        rhs[o0] = a;
    if (st.u)
        stageStore(st, o0, s0, a, dt);
    if (k != 0)
        return;
    if (rhs)
        rhs[o4] = acc[4];
    if (st.u)
        stageStore(st, o4, s4, acc[4], dt);
}

// with one normal per face the linear pass includes the viscous flux; on a quadrilateral, whose normal
// and viscous distance vary, the two together need more registers than there are
bool rhsLinearViscous(const DevMesh &m) { return m.dim == 2 || m.faceType == E_TRI3; }
bool rhsLinearRule(const DevMesh &m)
{
    return m.dim == 2 ? (m.G == 2 || m.G == 3) : (m.faceType == E_TRI3 ? m.G == 6 : m.G == 4);
}

// mesh constants, with the metrics
void setupLinear(Ctx &c)
{
    DevMesh &m = c.m;
    if (!rhsLinearRule(m))
        return;
    if (m.P == 1)
    {
        const int row = m.faceType == E_TRI3 ? 4 : 8;
        m.linC = devAlloc<real>(c, row * (size_t)m.N);
        kLinCentre<<<gridFor(m.N, 256), 256, 0, c.stream>>>(m, m.linC, row);
    }
    if (rhsLinearViscous(m))
    {
        m.linDist = devAlloc<real>(c, m.F);
        kLinDist<<<gridFor(m.F, 256), 256, 0, c.stream>>>(m, m.linDist);
    }
    DNDSR_HIP_CHECK(hipGetLastError());
}

struct LinArgs
{
    const real *u, *uRec, *dlc;
    real *ff;
    // the one-pass form of small meshes
    real *rhs = nullptr;
    const StageUpdate *stage = nullptr;
    int *nonFinite = nullptr;
};
template <int DIM, int G, bool TRI, int RS, bool BATCH>
static void linLaunch(Ctx &c, const GasParams &gp, const LinArgs &a)
{
    if constexpr (TRI || DIM == 2)
        if (a.stage)
        {
            if (c.m.nBnd > 0)
            {
                rhsBoundaryLaunch<DIM, DIM + 1, G, RS, BATCH>(c, gp, a.u, a.uRec, a.dlc, a.ff);
                if (gp.viscous)
                    launchRHSViscous(c, gp, a.u, a.uRec, a.ff, true);
            }
            KernelTimer kt(c, K_RHS_FACE);
            auto cell = gp.viscous ? kRHSCellLin<DIM, G, RS, BATCH, true, TRI> : kRHSCellLin<DIM, G, RS, BATCH, false, TRI>;
            cell<<<gridFor(c.m.N, 16), 64, 0, c.stream>>>(c.m, gp, a.u, a.uRec, a.dlc, a.ff, a.rhs, *a.stage,
                                                          a.nonFinite);
            DNDSR_HIP_CHECK(hipGetLastError());
            return;
        }
    auto kern = kRHSFaceLin<DIM, G, RS, BATCH, false, TRI>;
    if constexpr (TRI || DIM == 2)
        if (gp.viscous)
            kern = kRHSFaceLin<DIM, G, RS, BATCH, true, TRI>;
    kern<<<gridFor(c.m.F, 64), 64, 0, c.stream>>>(c.m, gp, a.u, a.uRec, a.dlc, a.ff);
    DNDSR_HIP_CHECK(hipGetLastError());
    rhsBoundaryLaunch<DIM, DIM + 1, G, RS, BATCH>(c, gp, a.u, a.uRec, a.dlc, a.ff);
}
template <int DIM, int G, bool TRI>
static void linDispatch(Ctx &c, const GasParams &gp, const LinArgs &a)
{
    const bool batch = gp.rsMeanValueEig != 0 && gp.rsType >= RS_Roe_M1 && gp.rsType <= RS_Roe_M5;
#define DNDSR_LIN_CASE(RSV, B)                              \
    case RSV:                                              \
        linLaunch<DIM, G, TRI, RSV, B>(c, gp, a);          \
        break;
    if (batch)
        switch (gp.rsType)
        {
            DNDSR_LIN_CASE(RS_Roe_M1, true)
            DNDSR_LIN_CASE(RS_Roe_M2, true)
            DNDSR_LIN_CASE(RS_Roe_M3, true)
            DNDSR_LIN_CASE(RS_Roe_M4, true)
            DNDSR_LIN_CASE(RS_Roe_M5, true)
        default: throw std::runtime_error("invalid batched Riemann solver");
        }
    else
        switch (gp.rsType)
        {
            DNDSR_LIN_CASE(RS_Roe, false)
            DNDSR_LIN_CASE(RS_HLLC, false)
            DNDSR_LIN_CASE(RS_HLLEP, false)
            DNDSR_LIN_CASE(RS_HLLEP_V1, false)
            DNDSR_LIN_CASE(RS_Roe_M1, false)
            DNDSR_LIN_CASE(RS_Roe_M2, false)
            DNDSR_LIN_CASE(RS_Roe_M3, false)
            DNDSR_LIN_CASE(RS_Roe_M4, false)
            DNDSR_LIN_CASE(RS_Roe_M5, false)
            DNDSR_LIN_CASE(RS_Roe_M6, false)
            DNDSR_LIN_CASE(RS_Roe_M7, false)
            DNDSR_LIN_CASE(RS_Roe_M8, false)
        default: throw std::runtime_error("the rs type is invalid");
        }
#undef DNDSR_LIN_CASE
}

static void linRule(Ctx &c, const GasParams &gp, const LinArgs &a)
{
    const DevMesh &m = c.m;
    if (m.dim == 2 && m.G == 2)
        linDispatch<2, 2, false>(c, gp, a);
    else if (m.dim == 2)
        linDispatch<2, 3, false>(c, gp, a);
    else if (m.faceType == E_TRI3)
        linDispatch<3, 6, true>(c, gp, a);
    else
        linDispatch<3, 4, false>(c, gp, a);
}

void launchRHSFaceLinear(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc, real *ff)
{
    linRule(c, gp, LinArgs{u, uRec, dlc, ff});
}

// Cells up to which the one-pass residual is taken (up to four faces per cell, the viscous flux in the
// linear pass).  Ten SSP-RK3 steps, face pass and gather against one pass: 9 000 quadrilaterals
// 503 / 459 us, 16 384 508 / 520, 24 000 584 / 615, 32 400 648 / 620, 65 536 963 / 1208; 16 256 triangles
// 515 / 478, 32 512 629 / 584; three steps on tetrahedra: 1 296 201 / 169, 10 368 224 / 196, 29 478
// 306 / 294.  In 2-D the viscous flux moves the crossover by no more than the spread of the mesh kinds (single
// residuals: 18 200 quadrilaterals 11.1 / 9.7 us, 24 000 10.5 / 11.8; 24 576 triangles 10.5 / 9.9, 32 512
// 10.5 / 10.9; mixed bounded cells 9 000 21.2 / 19.5, 25 500 23.7 / 24.5).  On tetrahedra, whose viscous
// one-pass kernel fills the registers, the line is one wavefront (16 cells) per SIMD: 13 182 cells
// 13.0 / 13.1, 16 464 13.5 / 17.4, 29 478 16.5 / 21.1; bounded 16 464 38.6 / 42.2.
constexpr idx kSmallRHS = 32768, kSmallRHSTetVisc = 16384;
bool rhsCellSize(const DevMesh &m)
{
    return m.N <= kSmallRHS && m.K <= 4 && rhsLinearRule(m) && rhsLinearViscous(m);
}
bool rhsCellRule(const Ctx &c, bool viscous, const real *u, const real *uRec, const real *dlc, const real *rhs,
                 const StageUpdate *stage)
{
    const DevMesh &m = c.m;
    if (!rhsCellSize(m) || (viscous && m.dim == 3 && m.N > kSmallRHSTetVisc) || (stage && stage->u && (!stage->out || stage->out == stage->u)))
        return false;
    // an array that is read must not be written before every block has read it
    const size_t N = m.N;
    auto apart = [&](const real *w, const real *r, size_t n) { return !w || !r || w + 5 * N <= r || r + n <= w; };
    return apart(rhs, u, 5 * N) && apart(rhs, uRec, 5 * (size_t)m.M * N) && apart(rhs, dlc, N);
}
void launchRHSCellLinear(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc, real *ff,
                         real *rhs, const StageUpdate &stage, int *nonFinite)
{
    linRule(c, gp, LinArgs{u, uRec, dlc, ff, rhs, &stage, nonFinite});
}

} // namespace dndsr
