// adjoint.hip -- discrete adjoint of the compact-FV residual: vector-Jacobian
// products of EvaluateRHS and of the VR Jacobi sweep.
//
// The reference has no adjoint; these kernels differentiate exactly the discrete
// operators of vr.hip / euler.hip:
//   EvaluateRHS:  rhs_i = sum_{f in i} s_if / V_i sum_g w_g (-F(U_L, U_R, uL, uR, n_g) + Fv(U_L, U_R, G_L, G_R, n_g))
//                 with U_side(x) = u_side + phi_side(x) . uRec_side, G_side(x) = D1phi_side(x) . uRec_side,
//                 deltaLambdaCell frozen; a boundary face takes U_R = ghost(U_L), u_R = ghost(u_L) (at
//                 the mean normal), G_R = G_L;
//   VR sweep:     y_i = c0 x_i + c1 sum_k [A^-1B_{i,k} x_j + A^-1b_{i,k} (u_j - u_i)].
// Derivatives of fluxes and ghost states are the reverse passes of gasadj.hpp; every branch is
// differentiated as executed.  Reconstruction is not
// stored: the caller passes the same uRec the forward pass used (the Python wrapper recomputes it).
#include <algorithm>

#include "gasadj.hpp"
#include "internal.hpp"

namespace dndsr
{
// zero-mean basis of cell c at the point x (+ shift, the periodic translation into
// the cell's frame); same arithmetic as the face kernel
template <int DIM, int NDOF>
__device__ inline void cellBasisAt(const DevMesh &m, idx c, const real *x, const real *shift, real *phi)
{
    constexpr int M = NDOF - 1;
    const size_t N = m.N;
    const real isc = ldu(m.iscale, (uint32_t)c);
    real xs[3], mom[M > 0 ? M : 1];
#pragma unroll
    for (int r = 0; r < 3; r++)
    {
        real p = x[r] + (shift ? shift[r] : 0.0);
        xs[r] = p - ldu(m.cent + (size_t)r * N, (uint32_t)c);
        if (DIM == 3 || r < 2)
            xs[r] *= isc;
    }
#pragma unroll
    for (int j = 0; j < M; j++)
        mom[j] = ldu(m.moment + (size_t)j * N, (uint32_t)c);
    basisRow0<DIM, NDOF>(xs, mom, phi);
}

// zero-mean basis and its gradient rows of cell c at x (+ shift), as the viscous pass
// evaluates them (scaled coordinates divided by the cell scale)
template <int DIM, int NDOF>
__device__ inline void cellBasisGradAt(const DevMesh &m, idx c, const real *x, const real *shift, real *phi,
                                       real (*dphi)[NDOF > 1 ? NDOF - 1 : 1])
{
    constexpr int M = NDOF - 1;
    const size_t N = m.N;
    const real s = ldu(m.scale, (uint32_t)c);
    real xs[3];
#pragma unroll
    for (int r = 0; r < 3; r++)
        xs[r] = (x[r] + (shift ? shift[r] : 0.0)) - ldu(m.cent + (size_t)r * N, (uint32_t)c);
    xs[0] /= s, xs[1] /= s;
    if (DIM == 3)
        xs[2] /= s;
#pragma unroll
    for (int j = 0; j < M; j++)
    {
        phi[j] = basisDiff(DIM, 0, j + 1, xs, s) - ldu(m.moment + (size_t)j * N, (uint32_t)c);
#pragma unroll
        for (int d = 0; d < DIM; d++)
            dphi[d][j] = basisDiff(DIM, 1 + d, j + 1, xs, s);
    }
}

// value, gradient and geometry of an interior face point, shared by the point and face kernels
template <int DIM, int NDOF>
struct AdjSide
{
    real U[5], phi[NDOF > 1 ? NDOF - 1 : 1], G[3][5];
    __device__ __forceinline__ void load(const DevMesh &m, idx c, const real *x, const real *shift, const real *um,
                                         const real *__restrict__ uRec, bool grad)
    {
        constexpr int M = NDOF - 1;
        const size_t N = m.N;
#pragma unroll
        for (int v = 0; v < 5; v++)
            U[v] = um[v];
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int v = 0; v < 5; v++)
                G[d][v] = 0;
        if (!uRec)
            return;
        cellBasisAt<DIM, NDOF>(m, c, x, shift, phi);
        real dphi[DIM][M > 0 ? M : 1], p2[M > 0 ? M : 1];
        if (grad)
        {
            if constexpr (M == DIM) // linear: d phi_j / d x_d = delta / scale
            {
                const real isc = ldu(m.iscale, (uint32_t)c);
#pragma unroll
                for (int d = 0; d < DIM; d++)
#pragma unroll
                    for (int j = 0; j < M; j++)
                        dphi[d][j] = d == j ? isc : 0.0;
            }
            else
                cellBasisGradAt<DIM, NDOF>(m, c, x, shift, p2, dphi);
        }
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            real s = 0;
#pragma unroll
            for (int j = 0; j < M; j++)
            {
                const real r = ldu(uRec + (size_t)(v * M + j) * N, (uint32_t)c);
                s += phi[j] * r;
                if (grad)
                {
                    if constexpr (M == DIM)
                        G[j][v] = dphi[j][j] * r;
                    else
#pragma unroll
                        for (int d = 0; d < DIM; d++)
                            G[d][v] += dphi[d][j] * r;
                }
            }
            U[v] += s;
        }
    }
};

// Sensitivities of an interior face point: Fbar . F(U_L, U_R, u_L, u_R) with respect to the point states
// (ULb, URb) and the cell means (mLb, mRb)
template <int RS, bool BATCH>
__device__ __forceinline__ void facePointBar(const GasParams &gp, const real *uL, const real *uR, const real *UL,
                                             const real *UR, const real *n, const real *nm, real dLambda,
                                             const real *Fbar, real *ULb, real *URb, real *mLb, real *mRb)
{
#pragma unroll
    for (int v = 0; v < 5; v++)
        ULb[v] = URb[v] = mLb[v] = mRb[v] = 0;
    RoeAve r;
    RoeBar rb;
    roeAverage(uL, uR, gp.gamma, r);
    riemannFluxBar<RS, BATCH>(UL, UR, r, n, nm, gp, dLambda, Fbar, ULb, URb, rb);
    roeAverageBar(uL, uR, gp.gamma, r, rb, mLb, mRb);
}
// -Fbar . Fv with respect to the point states (added) and the mean gradient of the two sides (Gb)
__device__ __forceinline__ void facePointVisBar(const DevMesh &m, const GasParams &gp, idx f, idx cL, idx cR,
                                                const real *sh, const real *UL, const real *UR, const real (*GL)[5],
                                                const real (*GR)[5], const real *n, const real *Fbar, real *ULb,
                                                real *URb, real (*Gb)[5])
{
    const size_t N = m.N;
    real dn = 0, Ga[3][5], Fvb[5];
#pragma unroll
    for (int q = 0; q < 3; q++)
        dn += ((ldu(m.bary + (size_t)q * N, (uint32_t)cR) - sh[q]) - ldu(m.bary + (size_t)q * N, (uint32_t)cL)) * n[q];
    const real d0 = fmin(ldu(m.vol, (uint32_t)cL), ldu(m.vol, (uint32_t)cR)) / ldu(m.farea, (uint32_t)f) * 2;
    const real idist = 1.0 / fmax(fmin(fabs(dn), d0 * 2), d0 * 0.25);
#pragma unroll
    for (int v = 0; v < 5; v++)
    {
        Fvb[v] = -Fbar[v];
#pragma unroll
        for (int d = 0; d < 3; d++)
            Ga[d][v] = 0.5 * (GL[d][v] + GR[d][v]);
    }
    viscousPointBar(gp, UL, UR, Ga, n, idist, false, Fvb, ULb, URb, Gb);
}

// The same for a boundary point: the right states are the ghosts of the left ones (the mean's at nm), GR = GL
template <int RS, bool BATCH>
__device__ __forceinline__ void bndPointBar(const DevMesh &m, const GasParams &gp, idx f, idx cL, const real *uL,
                                            const real *UL, const real (*GL)[5], const real *n, const real *nm,
                                            real dLambda, const real *Fbar, int vis, real *ULb, real *mLb,
                                            real (*Gb)[5])
{
    const int zone = m.fzone[f], type = m.bcType[zone];
    const real *far = m.bcVal + (size_t)zone * 5;
    real UR[5], uR[5], URb[5], mRb[5];
    bcGhost(type, UL, n, far, gp.gamma, UR);
    bcGhost(type, uL, nm, far, gp.gamma, uR);
#pragma unroll
    for (int v = 0; v < 5; v++)
        ULb[v] = URb[v] = mLb[v] = mRb[v] = 0;
    RoeAve r;
    RoeBar rb;
    roeAverage(uL, uR, gp.gamma, r);
    riemannFluxBar<RS, BATCH>(UL, UR, r, n, nm, gp, dLambda, Fbar, ULb, URb, rb);
    roeAverageBar(uL, uR, gp.gamma, r, rb, mLb, mRb);
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int v = 0; v < 5; v++)
            Gb[d][v] = 0;
    if (vis && !(type == BC_WALL_INVIS || type == BC_SYM || type == BC_FAR || type == BC_OUT))
    {
        const size_t N = m.N, F = m.F;
        real dn = 0, Fvb[5];
#pragma unroll
        for (int q = 0; q < 3; q++)
            dn += (m.fcent[(size_t)q * F + f] - ldu(m.bary + (size_t)q * N, (uint32_t)cL)) * n[q];
        const real d0 = ldu(m.vol, (uint32_t)cL) / ldu(m.farea, (uint32_t)f) * 2;
        const real idist = 1.0 / fmax(fmin(fabs(dn) * 2.0, d0 * 2), d0 * 0.25);
#pragma unroll
        for (int v = 0; v < 5; v++)
            Fvb[v] = -Fbar[v];
        viscousPointBar(gp, UL, UR, GL, n, idist, type == BC_WALL, Fvb, ULb, URb, Gb);
    }
    bcGhostBar(type, UL, n, far, gp.gamma, URb, ULb);
    bcGhostBar(type, uL, nm, far, gp.gamma, mRb, mLb);
}

// Point-sensitivity rows (of the buffer pbuf[row][G F]): 0-4 d/dU_L, 5-9 d/dU_R, 10-14 d/du_L (cell mean),
// 15-19 d/du_R, and with viscous fluxes 20-34 d/dG[d][v] of the two sides' mean gradient (row 20 + 5 d + v;
// each side takes half, and a boundary face, whose sides share one gradient, stores twice its value).
// One thread per (face, point), point-major: t = g F + f.
template <int DIM, int NDOF, int RS, bool BATCH>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1)))
kRHSPointAdj(DevMesh m, GasParams gp, const real *__restrict__ u, const real *__restrict__ uRec,
             const real *__restrict__ dlc, const real *__restrict__ fbar, real *__restrict__ pbuf, int vis)
{
    const size_t N = m.N, F = m.F, GF = (size_t)m.G * F;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= GF)
        return;
    const idx f = (idx)(t % F);
    const int g = (int)(t / F);
    const idx cL = m.f2c[f], cR = m.f2c[F + f];
    if (cR < 0) // boundary faces: kRHSBndPointAdj
        return;
    real x[3], n[3], nm[3], sh[3], uL[5], uR[5], Fbar[5];
#pragma unroll
    for (int r = 0; r < 3; r++)
    {
        x[r] = ldu(m.fpts + ((size_t)g * 3 + r) * F, (uint32_t)f);
        n[r] = ldu(m.fnorm + ((size_t)g * 3 + r) * F, (uint32_t)f);
        sh[r] = ldu(m.fshift + (size_t)r * F, (uint32_t)f);
        nm[r] = BATCH ? ldu(m.fmeanN + (size_t)r * F, (uint32_t)f) : 0.0;
    }
    const real wj = ldu(m.fwj + (size_t)g * F, (uint32_t)f);
#pragma unroll
    for (int v = 0; v < 5; v++)
    {
        uL[v] = ldu(u + (size_t)v * N, (uint32_t)cL), uR[v] = ldu(u + (size_t)v * N, (uint32_t)cR);
        Fbar[v] = -wj * ldu(fbar + (size_t)v * F, (uint32_t)f);
    }
    const real dLambda = dlc ? fmax(dlc[cL], dlc[cR]) : 0.0;
    AdjSide<DIM, NDOF> L, R;
    L.load(m, cL, x, nullptr, uL, uRec, vis != 0);
    R.load(m, cR, x, sh, uR, uRec, vis != 0);
    real a[5], b[5], c[5], d[5], Gb[3][5];
    facePointBar<RS, BATCH>(gp, uL, uR, L.U, R.U, n, nm, dLambda, Fbar, a, b, c, d);
    if (vis)
        facePointVisBar(m, gp, f, cL, cR, sh, L.U, R.U, L.G, R.G, n, Fbar, a, b, Gb);
#pragma unroll
    for (int v = 0; v < 5; v++)
    {
        pbuf[(size_t)v * GF + t] = a[v], pbuf[(size_t)(5 + v) * GF + t] = b[v];
        pbuf[(size_t)(10 + v) * GF + t] = c[v], pbuf[(size_t)(15 + v) * GF + t] = d[v];
    }
    if (vis)
#pragma unroll
        for (int q = 0; q < DIM; q++)
#pragma unroll
            for (int v = 0; v < 5; v++)
                pbuf[(size_t)(20 + 5 * q + v) * GF + t] = Gb[q][v];
}

// One thread per (boundary face, point): the rows of the back side (the front side has no state of its own)
template <int DIM, int NDOF, int RS, bool BATCH>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1)))
kRHSBndPointAdj(DevMesh m, GasParams gp, const real *__restrict__ u, const real *__restrict__ uRec,
                const real *__restrict__ dlc, const real *__restrict__ fbar, real *__restrict__ pbuf, int vis)
{
    const size_t N = m.N, F = m.F, GF = (size_t)m.G * F;
    const size_t tb = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tb >= (size_t)m.nBnd * m.G)
        return;
    const idx f = m.bndFace[tb % m.nBnd];
    const int g = (int)(tb / m.nBnd);
    const size_t t = (size_t)g * F + f;
    const idx cL = m.f2c[f];
    real x[3], n[3], nm[3], uL[5], Fbar[5];
#pragma unroll
    for (int r = 0; r < 3; r++)
    {
        x[r] = ldu(m.fpts + ((size_t)g * 3 + r) * F, (uint32_t)f);
        n[r] = ldu(m.fnorm + ((size_t)g * 3 + r) * F, (uint32_t)f);
        nm[r] = ldu(m.fmeanN + (size_t)r * F, (uint32_t)f);
    }
    const real wj = ldu(m.fwj + (size_t)g * F, (uint32_t)f);
#pragma unroll
    for (int v = 0; v < 5; v++)
        uL[v] = ldu(u + (size_t)v * N, (uint32_t)cL), Fbar[v] = -wj * ldu(fbar + (size_t)v * F, (uint32_t)f);
    AdjSide<DIM, NDOF> L;
    L.load(m, cL, x, nullptr, uL, uRec, vis != 0);
    real a[5], c[5], Gb[3][5];
    bndPointBar<RS, BATCH>(m, gp, f, cL, uL, L.U, L.G, n, nm, dlc ? dlc[cL] : 0.0, Fbar, vis, a, c, Gb);
#pragma unroll
    for (int v = 0; v < 5; v++)
        pbuf[(size_t)v * GF + t] = a[v], pbuf[(size_t)(10 + v) * GF + t] = c[v];
    if (vis)
#pragma unroll
        for (int q = 0; q < DIM; q++)
#pragma unroll
            for (int v = 0; v < 5; v++)
                pbuf[(size_t)(20 + 5 * q + v) * GF + t] = 2 * Gb[q][v];
}

// ---------------------------------------------------------------------------
// Linear reconstruction: the point sensitivities of a face are contracted with the basis where they are
// formed, so a face stores 5 + 5 DIM values per side (30 in 2-D, against 2 x 35 per point) and the cells
// only add their faces' rows.  A block is 64 faces; wavefront w takes the points w, w + NW, ... and sums
// them in its own LDS rows (the reverse pass leaves no registers for 30 accumulators), which are then added in
// wavefront order.  fbuf [2][5 + 5 DIM][F].
// Bound by FP64 issue and registers: at one wavefront per SIMD what does not fit stays in accumulation
// registers (143 us on the 333k faces of the mixed 2-D mesh, viscous); two per SIMD spill to scratch (328),
// and inviscid and viscous parts in kernels of their own measured 178.
// ---------------------------------------------------------------------------
template <int DIM>
constexpr int adjFaceWaves() { return DIM == 2 ? 2 : 3; }
template <int DIM, int RS, bool BATCH, bool VIS>
__global__ void __launch_bounds__(64 * adjFaceWaves<DIM>()) __attribute__((amdgpu_waves_per_eu(1)))
kRHSFaceAdj(DevMesh m, GasParams gp, const real *__restrict__ u, const real *__restrict__ uRec,
            const real *__restrict__ dlc, const real *__restrict__ fbar, real *__restrict__ fbuf)
{
    constexpr int NW = adjFaceWaves<DIM>(), Q = 5 + 5 * DIM;
    __shared__ real sm[NW][2 * Q][64];
    const int lane = threadIdx.x % 64, w = waveIndex(64);
    const size_t N = m.N, F = m.F;
    const idx f0 = xcdTile(blockIdx.x, gridDim.x) * 64, f = f0 + lane;
    const idx cL = f < m.F ? m.f2c[f] : -1, cR = f < m.F ? m.f2c[F + f] : -1;
    const bool on = cR >= 0; // boundary faces: kRHSBndFaceAdj
    for (int g = w; g < m.G && on; g += NW)
    {
        real x[3], n[3], nm[3], sh[3], uL[5], uR[5], Fbar[5];
#pragma unroll
        for (int r = 0; r < 3; r++)
        {
            x[r] = ldu(m.fpts + ((size_t)g * 3 + r) * F, (uint32_t)f);
            n[r] = ldu(m.fnorm + ((size_t)g * 3 + r) * F, (uint32_t)f);
            sh[r] = ldu(m.fshift + (size_t)r * F, (uint32_t)f);
            nm[r] = BATCH ? ldu(m.fmeanN + (size_t)r * F, (uint32_t)f) : 0.0;
        }
        const real wj = ldu(m.fwj + (size_t)g * F, (uint32_t)f);
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            uL[v] = ldu(u + (size_t)v * N, (uint32_t)cL), uR[v] = ldu(u + (size_t)v * N, (uint32_t)cR);
            Fbar[v] = -wj * ldu(fbar + (size_t)v * F, (uint32_t)f);
        }
        const real dLambda = dlc ? fmax(dlc[cL], dlc[cR]) : 0.0;
        AdjSide<DIM, DIM + 1> L, R;
        L.load(m, cL, x, nullptr, uL, uRec, VIS);
        R.load(m, cR, x, sh, uR, uRec, VIS);
        real a[5], b[5], c[5], d[5], Gb[3][5];
        facePointBar<RS, BATCH>(gp, uL, uR, L.U, R.U, n, nm, dLambda, Fbar, a, b, c, d);
        if constexpr (VIS)
            facePointVisBar(m, gp, f, cL, cR, sh, L.U, R.U, L.G, R.G, n, Fbar, a, b, Gb);
        const real hL = 0.5 * ldu(m.iscale, (uint32_t)cL), hR = 0.5 * ldu(m.iscale, (uint32_t)cR);
        auto put = [&](int q, real val) { sm[w][q][lane] = g == w ? val : sm[w][q][lane] + val; };
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            put(v, a[v] + c[v]);
            put(Q + v, b[v] + d[v]);
            if (uRec)
#pragma unroll
                for (int j = 0; j < DIM; j++)
                {
                    put(5 + v * DIM + j, L.phi[j] * a[v] + (VIS ? hL * Gb[j][v] : 0.0));
                    put(Q + 5 + v * DIM + j, R.phi[j] * b[v] + (VIS ? hR * Gb[j][v] : 0.0));
                }
        }
    }
    __syncthreads();
    if (!on)
        return;
    const int nw = m.G < NW ? m.G : NW;
    for (int q = w; q < 2 * Q; q += NW)
    {
        if (!uRec && q % Q >= 5)
            continue;
        real s = sm[0][q][lane];
        for (int k = 1; k < nw; k++)
            s += sm[k][q][lane];
        fbuf[(size_t)q * F + f] = s;
    }
}

// the boundary faces' rows of the back side: a block is 64 faces, wavefront w the points w, w + NW, ...
template <int DIM, int RS, bool BATCH>
__global__ void __launch_bounds__(64 * adjFaceWaves<DIM>()) __attribute__((amdgpu_waves_per_eu(1)))
kRHSBndFaceAdj(DevMesh m, GasParams gp, const real *__restrict__ u, const real *__restrict__ uRec,
               const real *__restrict__ dlc, const real *__restrict__ fbar, real *__restrict__ fbuf, int vis)
{
    constexpr int NW = adjFaceWaves<DIM>(), Q = 5 + 5 * DIM;
    __shared__ real sm[NW][Q][64];
    const int lane = threadIdx.x % 64, w = waveIndex(64);
    const idx t = blockIdx.x * 64 + lane;
    const bool on = t < m.nBnd;
    const size_t N = m.N, F = m.F;
    const idx f = m.bndFace[on ? t : m.nBnd - 1];
    const idx cL = m.f2c[f];
    const real isc = ldu(m.iscale, (uint32_t)cL);
    real nm[3], uL[5];
#pragma unroll
    for (int r = 0; r < 3; r++)
        nm[r] = ldu(m.fmeanN + (size_t)r * F, (uint32_t)f);
#pragma unroll
    for (int v = 0; v < 5; v++)
        uL[v] = ldu(u + (size_t)v * N, (uint32_t)cL);
    const real dLambda = dlc ? dlc[cL] : 0.0;
    for (int g = w; g < m.G; g += NW)
    {
        real x[3], n[3], Fbar[5];
#pragma unroll
        for (int r = 0; r < 3; r++)
        {
            x[r] = ldu(m.fpts + ((size_t)g * 3 + r) * F, (uint32_t)f);
            n[r] = ldu(m.fnorm + ((size_t)g * 3 + r) * F, (uint32_t)f);
        }
        const real wj = ldu(m.fwj + (size_t)g * F, (uint32_t)f);
#pragma unroll
        for (int v = 0; v < 5; v++)
            Fbar[v] = -wj * ldu(fbar + (size_t)v * F, (uint32_t)f);
        AdjSide<DIM, DIM + 1> L;
        L.load(m, cL, x, nullptr, uL, uRec, vis != 0);
        real a[5], c[5], Gb[3][5];
        bndPointBar<RS, BATCH>(m, gp, f, cL, uL, L.U, L.G, n, nm, dLambda, Fbar, vis, a, c, Gb);
        auto put = [&](int q, real val) { sm[w][q][lane] = g == w ? val : sm[w][q][lane] + val; };
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            put(v, a[v] + c[v]);
            if (uRec)
#pragma unroll
                for (int j = 0; j < DIM; j++)
                    put(5 + v * DIM + j, L.phi[j] * a[v] + isc * Gb[j][v]);
        }
    }
    __syncthreads();
    if (!on)
        return;
    const int nw = m.G < NW ? m.G : NW;
    for (int q = w; q < (uRec ? Q : 5); q += NW)
    {
        real s = sm[0][q][lane];
        for (int k = 1; k < nw; k++)
            s += sm[k][q][lane];
        fbuf[(size_t)q * F + f] = s;
    }
}

// one thread per cell: the sum of its faces' rows (in slot order)
template <int DIM, int KM>
__global__ void __launch_bounds__(256) kRHSGatherAdjLin(DevMesh m, const real *__restrict__ fbuf,
                                                        real *__restrict__ ubar, real *__restrict__ urecbar)
{
    constexpr int Q = 5 + 5 * DIM;
    const idx i = xcdTile(blockIdx.x, gridDim.x) * (idx)blockDim.x + threadIdx.x;
    if (i >= m.N)
        return;
    const size_t N = m.N, F = m.F;
    idx f[KM];
    bool on[KM];
    size_t base[KM];
#pragma unroll
    for (int k = 0; k < KM; k++)
    {
        const size_t q = (size_t)(k < m.K ? k : 0) * N + i;
        f[k] = m.c2f[q];
        on[k] = k < m.K && f[k] >= 0;
        base[k] = on[k] ? ((m.c2flag[q] & 1) ? (size_t)Q * F : 0) + f[k] : 0;
    }
    const int nq = urecbar ? Q : 5;
    for (int q = 0; q < nq; q++)
    {
        real r[KM], s = 0;
#pragma unroll
        for (int k = 0; k < KM; k++)
            r[k] = fbuf[base[k] + (size_t)q * F];
#pragma unroll
        for (int k = 0; k < KM; k++)
            s += on[k] ? r[k] : 0.0;
        (q < 5 ? ubar + (size_t)q * N : urecbar + (size_t)(q - 5) * N)[i] = s;
    }
}

// One thread per cell and variable (blockIdx.y): collect the point sensitivities of the cell's faces into
// uBar (N x 5) and uRecBar (5 M x N), evaluating the cell's basis at each point.
template <int DIM, int NDOF>
__global__ void __launch_bounds__(64) kRHSGatherAdj(DevMesh m, const real *__restrict__ pbuf,
                                                    real *__restrict__ ubar, real *__restrict__ urecbar, int vis)
{
    constexpr int M = NDOF - 1;
    const idx i = blockIdx.x * blockDim.x + threadIdx.x;
    const int v = blockIdx.y;
    if (i >= m.N)
        return;
    const size_t N = m.N, F = m.F, GF = (size_t)m.G * F;
    real au = 0, ar[M > 0 ? M : 1];
#pragma unroll
    for (int j = 0; j < M; j++)
        ar[j] = 0;
    for (int k = 0; k < m.K; k++)
    {
        const idx f = m.c2f[(size_t)k * N + i];
        if (f < 0)
            continue;
        const bool back = (m.c2flag[(size_t)k * N + i] & 1) == 0;
        const int rowU = (back ? 0 : 5) + v, rowM = (back ? 10 : 15) + v;
        real sh[3];
#pragma unroll
        for (int r = 0; r < 3; r++)
            sh[r] = m.fshift[(size_t)r * F + f];
        for (int g = 0; g < m.G; g++)
        {
            const size_t t = (size_t)g * F + f;
            const real gU = pbuf[(size_t)rowU * GF + t];
            au += gU + pbuf[(size_t)rowM * GF + t];
            if (urecbar)
            {
                real x[3], phi[M > 0 ? M : 1];
#pragma unroll
                for (int r = 0; r < 3; r++)
                    x[r] = m.fpts[((size_t)g * 3 + r) * F + f];
                cellBasisAt<DIM, NDOF>(m, i, x, back ? nullptr : sh, phi);
#pragma unroll
                for (int j = 0; j < M; j++)
                    ar[j] += phi[j] * gU;
                if (vis)
                {
                    real phi2[M > 0 ? M : 1], dphi[DIM][M > 0 ? M : 1];
                    cellBasisGradAt<DIM, NDOF>(m, i, x, back ? nullptr : sh, phi2, dphi);
#pragma unroll
                    for (int d = 0; d < DIM; d++)
                    {
                        const real gg = 0.5 * pbuf[(size_t)(20 + 5 * d + v) * GF + t];
#pragma unroll
                        for (int j = 0; j < M; j++)
                            ar[j] += dphi[d][j] * gg;
                    }
                }
            }
        }
    }
    ubar[(size_t)v * N + i] = au;
    if (urecbar)
#pragma unroll
        for (int j = 0; j < M; j++)
            urecbar[(size_t)(v * M + j) * N + i] = ar[j];
}

// adjoint of the face flux from the adjoint of the residual (the gather rhs_L += ff / V_L,
// rhs_R -= ff / V_R): fbar_f = rbar_L / V_L - rbar_R / V_R
__global__ void __launch_bounds__(256) kFaceBar(DevMesh m, const real *__restrict__ rbar, real *__restrict__ fbar)
{
    const idx f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= m.F)
        return;
    const size_t N = m.N, F = m.F;
    const idx cL = m.f2c[f], cR = m.f2c[F + f];
#pragma unroll
    for (int v = 0; v < 5; v++)
        fbar[(size_t)v * F + f] = cR >= 0 ? rbar[(size_t)v * N + cL] / m.vol[cL] - rbar[(size_t)v * N + cR] / m.vol[cR]
                                          : rbar[(size_t)v * N + cL] / m.vol[cL];
}

// values of the sensitivity buffer for this mesh
size_t adjBufferSize(const DevMesh &m, bool viscous)
{
    const size_t point = (size_t)(viscous ? 35 : 20) * m.G, face = 2 * (5 + 5 * m.dim);
    return std::max(point, face) * m.F;
}

// rbar: the face-flux adjoint [5][F], formed by launchEvalRHSVJP
template <int DIM, int NDOF, int RS, bool BATCH>
static void rhsAdjLaunch(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc,
                         const real *rbar, real *ubar, real *urecbar)
{
    const DevMesh &m = c.m;
    const int vis = gp.viscous ? 1 : 0;
    if constexpr (NDOF == DIM + 1)
    {
        const int g = gridFor(m.F, 64), bs = 64 * adjFaceWaves<DIM>();
        if (vis)
            kRHSFaceAdj<DIM, RS, BATCH, true><<<g, bs, 0, c.stream>>>(m, gp, u, uRec, dlc, rbar, c.adjPoint);
        else
            kRHSFaceAdj<DIM, RS, BATCH, false><<<g, bs, 0, c.stream>>>(m, gp, u, uRec, dlc, rbar, c.adjPoint);
        DNDSR_HIP_CHECK(hipGetLastError());
        if (m.nBnd > 0)
        {
            kRHSBndFaceAdj<DIM, RS, BATCH><<<gridFor(m.nBnd, 64), bs, 0, c.stream>>>(m, gp, u, uRec, dlc, rbar,
                                                                                     c.adjPoint, vis);
            DNDSR_HIP_CHECK(hipGetLastError());
        }
        const int cb = cellBlock(m.N), gc = gridFor(m.N, cb);
        if (m.K <= 4)
            kRHSGatherAdjLin<DIM, 4><<<gc, cb, 0, c.stream>>>(m, c.adjPoint, ubar, uRec ? urecbar : nullptr);
        else
            kRHSGatherAdjLin<DIM, kMaxFC><<<gc, cb, 0, c.stream>>>(m, c.adjPoint, ubar, uRec ? urecbar : nullptr);
        DNDSR_HIP_CHECK(hipGetLastError());
        return;
    }
    const size_t GF = (size_t)m.G * m.F;
    kRHSPointAdj<DIM, NDOF, RS, BATCH><<<(unsigned)((GF + 127) / 128), 128, 0, c.stream>>>(m, gp, u, uRec, dlc, rbar,
                                                                                          c.adjPoint, vis);
    DNDSR_HIP_CHECK(hipGetLastError());
    if (m.nBnd > 0)
    {
        const size_t nb = (size_t)m.nBnd * m.G;
        kRHSBndPointAdj<DIM, NDOF, RS, BATCH><<<(unsigned)((nb + 127) / 128), 128, 0, c.stream>>>(
            m, gp, u, uRec, dlc, rbar, c.adjPoint, vis);
        DNDSR_HIP_CHECK(hipGetLastError());
    }
    kRHSGatherAdj<DIM, NDOF><<<dim3(gridFor(m.N, 64), 5), 64, 0, c.stream>>>(m, c.adjPoint, ubar, urecbar,
                                                                             vis && uRec != nullptr);
    DNDSR_HIP_CHECK(hipGetLastError());
}

template <int DIM, int NDOF>
static void rhsAdjRS(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc, const real *rbar,
                     real *ubar, real *urecbar)
{
    const bool batch = gp.rsMeanValueEig != 0 && gp.rsType >= RS_Roe_M1 && gp.rsType <= RS_Roe_M5;
#define DNDSR_ADJ_CASE(RSV, B)                                                                    \
    case RSV:                                                                                     \
        rhsAdjLaunch<DIM, NDOF, RSV, B>(c, gp, u, uRec, dlc, rbar, ubar, urecbar);               \
        break;
    if (batch)
    {
        switch (gp.rsType)
        {
            DNDSR_ADJ_CASE(RS_Roe_M1, true)
            DNDSR_ADJ_CASE(RS_Roe_M2, true)
            DNDSR_ADJ_CASE(RS_Roe_M3, true)
            DNDSR_ADJ_CASE(RS_Roe_M4, true)
            DNDSR_ADJ_CASE(RS_Roe_M5, true)
        default: throw std::runtime_error("invalid batched Riemann solver");
        }
    }
    else
    {
        switch (gp.rsType)
        {
            DNDSR_ADJ_CASE(RS_Roe, false)
            DNDSR_ADJ_CASE(RS_HLLC, false)
            DNDSR_ADJ_CASE(RS_HLLEP, false)
            DNDSR_ADJ_CASE(RS_HLLEP_V1, false)
            DNDSR_ADJ_CASE(RS_Roe_M1, false)
            DNDSR_ADJ_CASE(RS_Roe_M2, false)
            DNDSR_ADJ_CASE(RS_Roe_M3, false)
            DNDSR_ADJ_CASE(RS_Roe_M4, false)
            DNDSR_ADJ_CASE(RS_Roe_M5, false)
            DNDSR_ADJ_CASE(RS_Roe_M6, false)
            DNDSR_ADJ_CASE(RS_Roe_M7, false)
            DNDSR_ADJ_CASE(RS_Roe_M8, false)
        default: throw std::runtime_error("the rs type is invalid");
        }
    }
#undef DNDSR_ADJ_CASE
}

void launchEvalRHSVJP(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc,
                      const real *rbar, real *ubar, real *urecbar, const real *faceBar)
{
    DevMesh &m = c.m;
    KernelTimer kt(c, K_ADJOINT);
    if (!faceBar)
    {
        kFaceBar<<<gridFor(m.F, 256), 256, 0, c.stream>>>(m, rbar, c.adjFaceBar);
        DNDSR_HIP_CHECK(hipGetLastError());
        faceBar = c.adjFaceBar;
    }
    rbar = faceBar; // the point kernels read the face-flux adjoint
    if (m.dim == 2)
    {
        if (!uRec || m.P == 1)
            rhsAdjRS<2, 3>(c, gp, u, uRec, dlc, rbar, ubar, urecbar);
        else if (m.P == 2)
            rhsAdjRS<2, 6>(c, gp, u, uRec, dlc, rbar, ubar, urecbar);
        else
            rhsAdjRS<2, 10>(c, gp, u, uRec, dlc, rbar, ubar, urecbar);
    }
    else
    {
        if (!uRec || m.P == 1)
            rhsAdjRS<3, 4>(c, gp, u, uRec, dlc, rbar, ubar, urecbar);
        else if (m.P == 2)
            rhsAdjRS<3, 10>(c, gp, u, uRec, dlc, rbar, ubar, urecbar);
        else
            rhsAdjRS<3, 20>(c, gp, u, uRec, dlc, rbar, ubar, urecbar);
    }
}

// ---------------------------------------------------------------------------
// Transposed VR sweep.  Forward: y_i = c0 x_i + c1 sum_k [B_{i,k} x_{j(i,k)} + b_{i,k}(u_j - u_i)]
// (c0, c1) = (1 - w, w) Jacobi, (1, -1) recordInc, (0, -1) recordInc with uRecIsZero,
// (1, -1) without the b term for IterDiff.  Gather form for cell j: its neighbours
// i across slots kj see j across their slot ki = c2s[kj][j], so
//   xbar_j = c0 ybar_j + c1 sum_kj B_{i,ki}^T ybar_i
//   ubar_j = c1 sum_kj b_{i,ki} . ybar_i - c1 sum_k b_{j,k} . ybar_j     (per variable)
// Tile kernel as the forward sweep's (kVRIter, vr.hip): 64 cells per block, one wavefront per output row r
// (two rows above 16), the neighbour's ybar block staged in LDS once per slot and shared by the row
// wavefronts, each matrix entry (column r of the neighbour's block) read once.  The ubar rows are spread over
// the wavefronts.  One thread per cell, which this replaces, re-read the block for every variable at one
// wavefront per SIMD: 430 us on 10.6k p2 hexahedra, against 52.
// ---------------------------------------------------------------------------
template <int M>
struct VRTRows
{
    static constexpr int RW = M <= 16 ? M : (M + 1) / 2; // wavefronts per block
    static constexpr int RPT = (M + RW - 1) / RW;        // rows per thread
};
template <int M, int NV>
__global__ void __launch_bounds__(64 * VRTRows<M>::RW)
kVRIterT(DevMesh m, const real *__restrict__ ybar, real *__restrict__ xbar, real *__restrict__ ubar, real c0, real c1,
         int useB, int useb)
{
    constexpr int RW = VRTRows<M>::RW, RPT = VRTRows<M>::RPT, NR = NV * M;
    constexpr int PER = (NR + RW - 1) / RW, VPT = (NV + RW - 1) / RW;
    __shared__ real sY[2][PER * RW][64];
    const int lane = threadIdx.x % 64, w = waveIndex(64);
    const idx jc = xcdTile(blockIdx.x, gridDim.x) * 64 + lane;
    const bool valid = jc < m.N;
    const size_t N = m.N;
    const idx j = valid ? jc : m.N - 1;
    const bool rowsU = ubar && useb;
    real ax[RPT][NV], au[VPT];
#pragma unroll
    for (int t = 0; t < RPT; t++)
    {
        const int r = w + t * RW < M ? w + t * RW : M - 1;
#pragma unroll
        for (int v = 0; v < NV; v++)
            ax[t][v] = c0 * ldu(ybar + (size_t)(v * M + r) * N, (uint32_t)j);
    }
#pragma unroll
    for (int t = 0; t < VPT; t++)
        au[t] = 0;
    auto stage = [&](int buf, idx o) {
        real nb[PER];
#pragma unroll
        for (int t = 0; t < PER; t++)
        {
            const int q = w + t * RW < NR ? w + t * RW : NR - 1;
            nb[t] = ldu(ybar + (size_t)q * N, (uint32_t)(o >= 0 ? o : j));
        }
#pragma unroll
        for (int t = 0; t < PER; t++)
            sY[buf][w + t * RW][lane] = nb[t];
    };
    idx on = m.c2c[j];
    for (int k = 0; k < m.K; k++)
    {
        const idx o = on;
        const int ki = o >= 0 ? m.c2s[(size_t)k * N + j] : 0;
        const size_t i = o >= 0 ? o : j;
        const real *B = m.AinvB + (size_t)(1 + ki) * M * M * N + i;
        const real *b = m.Ainvb + (size_t)ki * M * N + i;
        const real *bj = m.Ainvb + (size_t)k * M * N;
        real bc[RPT][M];
        if (useB)
#pragma unroll
            for (int t = 0; t < RPT; t++)
            {
                const int r = w + t * RW < M ? w + t * RW : M - 1;
#pragma unroll
                for (int q = 0; q < M; q++)
                    bc[t][q] = B[(size_t)(q * M + r) * N];
            }
        stage(k & 1, o);
        on = k + 1 < m.K ? m.c2c[(size_t)(k + 1) * N + j] : idx(-1);
        __syncthreads(); // sY[k & 1] complete; the other buffer no longer read
        if (o < 0)
            continue;
        if (useB)
#pragma unroll
            for (int t = 0; t < RPT; t++)
#pragma unroll
                for (int v = 0; v < NV; v++)
                {
                    real s = 0;
#pragma unroll
                    for (int q = 0; q < M; q++)
                        s += bc[t][q] * sY[k & 1][v * M + q][lane];
                    ax[t][v] += c1 * s;
                }
        if (rowsU)
#pragma unroll
            for (int t = 0; t < VPT; t++)
            {
                const int v = w + t * RW;
                if (v >= NV)
                    continue;
                real s = 0, sj = 0;
#pragma unroll
                for (int q = 0; q < M; q++)
                {
                    s += b[(size_t)q * N] * sY[k & 1][v * M + q][lane];
                    sj += ldu(bj + (size_t)q * N, (uint32_t)j) * ldu(ybar + (size_t)(v * M + q) * N, (uint32_t)j);
                }
                au[t] += c1 * (s - sj);
            }
    }
    if (!valid)
        return;
    if (xbar)
#pragma unroll
        for (int t = 0; t < RPT; t++)
        {
            const int r = w + t * RW;
            if (r < M)
#pragma unroll
                for (int v = 0; v < NV; v++)
                    stu(xbar + (size_t)(v * M + r) * N, (uint32_t)j, ax[t][v]);
        }
    if (ubar)
#pragma unroll
        for (int t = 0; t < VPT; t++)
        {
            const int v = w + t * RW;
            if (v < NV)
                stu(ubar + (size_t)v * N, (uint32_t)j, au[t]);
        }
}

// Transposed boundary term of the VR sweep (forward: uRecNew_i += scale A_i^-1 BCC_i,
// BCC_i = sum_{boundary faces, g} phi(x_g) (w0^2 (u_B(x_g) - u_i)) w_g JDet_g, u_B the ghost
// of the compressed point state u_i + phi . uRec_i, or the given point value).  One
// thread per boundary cell; BCCbar = scale A^-T ybar, then per point the adjoint of u_B - u_i and
// through the ghost (bcGhostBar) of the point state, i.e. of the cell's mean and coefficients (point
// values given: of the mean only), added to ubar / xbar.
template <int DIM, int NDOF, int NV>
__global__ void __launch_bounds__(64) kVRBoundaryT(DevMesh m, const real *__restrict__ uRec,
                                                   const real *__restrict__ u, const real *__restrict__ ybar,
                                                   real scale, real *__restrict__ xbar, real *__restrict__ ubar)
{
    constexpr int M = NDOF - 1;
    const idx t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= m.nBndCell)
        return;
    const idx i = m.bndCell[t];
    const size_t N = m.N, F = m.F;
    real Bb[M][NV];
#pragma unroll
    for (int j = 0; j < M; j++)
#pragma unroll
        for (int v = 0; v < NV; v++)
        {
            real a = 0;
#pragma unroll
            for (int r = 0; r < M; r++)
                a += m.AinvB[((size_t)r * M + j) * N + i] * ybar[((size_t)v * M + r) * N + i];
            Bb[j][v] = scale * a;
        }
    real mom[M], cen[3], um[NV];
#pragma unroll
    for (int j = 0; j < M; j++)
        mom[j] = m.moment[(size_t)j * N + i];
#pragma unroll
    for (int r = 0; r < 3; r++)
        cen[r] = m.cent[(size_t)r * N + i];
    const real isc = m.iscale[i];
#pragma unroll
    for (int v = 0; v < NV; v++)
        um[v] = u[(size_t)v * N + i];
    const bool euler = NV == 5 && m.bcType != nullptr;
    real ub[NV], xb[NV][M];
#pragma unroll
    for (int v = 0; v < NV; v++)
    {
        ub[v] = 0;
#pragma unroll
        for (int j = 0; j < M; j++)
            xb[v][j] = 0;
    }
    for (int k = 0; k < m.K; k++)
    {
        const idx f = m.c2f[(size_t)k * N + i];
        if (f < 0 || m.c2c[(size_t)k * N + i] >= 0)
            continue;
        const int zone = m.fzone[f];
        const real w0 = m.faceW[f];
        for (int g = 0; g < m.G; g++)
        {
            real xs[3], phi[M], tv[NV];
#pragma unroll
            for (int r = 0; r < 3; r++)
            {
                xs[r] = m.fpts[((size_t)g * 3 + r) * F + f] - cen[r];
                if (DIM == 3 || r < 2)
                    xs[r] *= isc;
            }
            basisRow0<DIM, NDOF>(xs, mom, phi);
            const real fac = m.fwj[(size_t)g * F + f] * (w0 * w0);
            // BCC_j += phi_j inc fac: the adjoint of inc
#pragma unroll
            for (int v = 0; v < NV; v++)
            {
                real q = 0;
#pragma unroll
                for (int j = 0; j < M; j++)
                    q += Bb[j][v] * phi[j];
                tv[v] = q * fac;
                ub[v] -= tv[v]; // inc = uB - u_i (given point values: value - u_i)
            }
            if (!euler)
                continue;
            real uBL[5], ULf[5], n[3];
#pragma unroll
            for (int v = 0; v < 5; v++)
            {
                real r = 0;
#pragma unroll
                for (int j = 0; j < M; j++)
                    r += phi[j] * uRec[((size_t)v * M + j) * N + i];
                uBL[v] = r;
            }
#pragma unroll
            for (int r = 0; r < 3; r++)
                n[r] = m.fnorm[((size_t)g * 3 + r) * F + f];
            // compressRecPart keeps the point state or falls back to the mean
            real full[5];
#pragma unroll
            for (int v = 0; v < 5; v++)
                full[v] = um[v] + uBL[v];
            compressRecPart(um, uBL, ULf);
            bool kept = true;
#pragma unroll
            for (int v = 0; v < 5; v++)
                kept = kept && !(ULf[v] != full[v]);
            real sb[5] = {0, 0, 0, 0, 0}, tb[5];
#pragma unroll
            for (int v = 0; v < 5; v++)
                tb[v] = tv[v < NV ? v : 0];
            bcGhostBar(m.bcType[zone], ULf, n, m.bcVal + (size_t)zone * 5, m.bcGamma, tb, sb);
#pragma unroll
            for (int v = 0; v < NV; v++)
            {
                ub[v] += sb[v];
#pragma unroll
                for (int j = 0; j < M; j++)
                    xb[v][j] += kept ? phi[j] * sb[v] : 0.0;
            }
        }
    }
#pragma unroll
    for (int v = 0; v < NV; v++)
    {
        if (ubar)
            ubar[(size_t)v * N + i] += ub[v];
        if (xbar && euler)
#pragma unroll
            for (int j = 0; j < M; j++)
                xbar[((size_t)v * M + j) * N + i] += xb[v][j];
    }
}

template <int DIM, int NDOF>
static void vrBndTLaunch(Ctx &c, int nVars, const real *uRec, const real *u, const real *ybar, real scale, real *xbar,
                         real *ubar)
{
    const int g = gridFor(c.m.nBndCell, 64);
    if (nVars == 5)
        kVRBoundaryT<DIM, NDOF, 5><<<g, 64, 0, c.stream>>>(c.m, uRec, u, ybar, scale, xbar, ubar);
    else
        kVRBoundaryT<DIM, NDOF, 1><<<g, 64, 0, c.stream>>>(c.m, uRec, u, ybar, scale, xbar, ubar);
    DNDSR_HIP_CHECK(hipGetLastError());
}

template <int M>
static void vrTLaunch(Ctx &c, int nVars, const real *ybar, real *xbar, real *ubar, real c0, real c1, int useB,
                      int useb)
{
    const int g = gridFor(c.m.N, 64), bs = 64 * VRTRows<M>::RW;
    if (nVars == 5)
        kVRIterT<M, 5><<<g, bs, 0, c.stream>>>(c.m, ybar, xbar, ubar, c0, c1, useB, useb);
    else if (nVars == 1)
        kVRIterT<M, 1><<<g, bs, 0, c.stream>>>(c.m, ybar, xbar, ubar, c0, c1, useB, useb);
    else
        throw std::runtime_error("nVars must be 1 or 5");
    DNDSR_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Transpose of the second-order substitute (kVR2nd): uRec_i = G_i(u) with
//   Gauss rule:     uRec_i[v][d] = 1/(V_i isc_i) sum_k c_ik[d] (u_k[v] - u_i[v]),
//                   c_ik = lThis/(lThis + lThat) A n sgn (boundary: A n / 2, u_k the ghost)
//   least squares:  uRec_i[v][d] = 1/isc_i (S_i^-1 sum_k dc_ik du_ik[v])[d], S_i = sum_k dc_ik dc_ik^T
// which is linear in u but for the boundary ghosts.  Pass 1 forms per cell the weight of its
// differences, q_i[v] = recBar_i[v] / (V_i isc_i) or S_i^-T recBar_i[v] / isc_i; pass 2 gathers
// per cell j: sum over its faces of c_ik . q_i from the neighbour i's side, minus its own
// c_jk . q_j, plus the ghosts' Jacobian (dual numbers) transposed.
// ---------------------------------------------------------------------------
template <int DIM>
__device__ inline void vr2ndFaceWeight(const DevMesh &m, idx i, int k, int method, bool plain, real *w)
{
    const size_t N = m.N, F = m.F;
    const idx f = m.c2f[(size_t)k * N + i];
    const idx o = m.c2c[(size_t)k * N + i];
    const bool back = m.f2c[f] == i;
    real bi[3], xf[3], n[3], ob[3] = {0, 0, 0};
    for (int r = 0; r < 3; r++)
    {
        bi[r] = m.bary[(size_t)r * N + i];
        xf[r] = m.fcent[(size_t)r * F + f] + (back ? 0.0 : m.fshift[(size_t)r * F + f]);
        n[r] = m.fmeanN[(size_t)r * F + f];
        if (o >= 0)
            ob[r] = m.bary[(size_t)r * N + o] + (back ? -m.fshift[(size_t)r * F + f] : m.fshift[(size_t)r * F + f]);
    }
    const real A = m.farea[f];
    if (method == 1)
    {
        if (o < 0)
        {
            for (int d = 0; d < DIM; d++)
                w[d] = 0.5 * A * n[d];
            return;
        }
        real lThis = 0, lThat = 0;
        for (int r = 0; r < 3; r++)
            lThis += (xf[r] - bi[r]) * (xf[r] - bi[r]), lThat += (ob[r] - xf[r]) * (ob[r] - xf[r]);
        lThis = plain ? 1.0 : sqrt(lThis);
        lThat = plain ? 1.0 : sqrt(lThat);
        const real sgn = back ? 1.0 : -1.0;
        for (int d = 0; d < DIM; d++)
            w[d] = lThis / (lThis + lThat + kVerySmall) * A * (n[d] * sgn);
        return;
    }
    if (o >= 0)
        for (int d = 0; d < DIM; d++)
            w[d] = ob[d] - bi[d];
    else
    {
        real pr = 0;
        for (int r = 0; r < 3; r++)
            pr += (bi[r] - m.fcent[(size_t)r * F + f]) * n[r];
        for (int d = 0; d < DIM; d++)
            w[d] = pr * -2.0 * n[d];
    }
}

template <int DIM, int NV>
__global__ void __launch_bounds__(64) kVR2ndTq(DevMesh m, const real *__restrict__ ybar, real *__restrict__ q)
{
    const idx i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m.N)
        return;
    const size_t N = m.N;
    const int method = m.s.subs2ndOrder;
    const bool plain = m.s.subs2ndOrderGGScheme == 0;
    const real isc = m.iscale[i];
    real gb[NV][DIM];
    for (int v = 0; v < NV; v++)
        for (int d = 0; d < DIM; d++)
            gb[v][d] = ybar[((size_t)v * DIM + d) * N + i] / isc;
    if (method == 1)
    {
        const real V = m.vol[i];
        for (int v = 0; v < NV; v++)
            for (int d = 0; d < DIM; d++)
                q[((size_t)v * DIM + d) * N + i] = gb[v][d] / V;
        return;
    }
    real S[DIM][DIM];
    for (int d = 0; d < DIM; d++)
        for (int e = 0; e < DIM; e++)
            S[d][e] = 0;
    for (int k = 0; k < m.K; k++)
    {
        if (m.c2f[(size_t)k * N + i] < 0)
            continue;
        real w[3];
        vr2ndFaceWeight<DIM>(m, i, k, method, plain, w);
        for (int d = 0; d < DIM; d++)
            for (int e = 0; e < DIM; e++)
                S[d][e] += w[d] * w[e];
    }
    real Si[DIM][DIM];
    if constexpr (DIM == 2)
    {
        const real det = S[0][0] * S[1][1] - S[0][1] * S[1][0];
        Si[0][0] = S[1][1] / det, Si[0][1] = -S[0][1] / det, Si[1][0] = -S[1][0] / det, Si[1][1] = S[0][0] / det;
    }
    else
    {
        real C[3][3];
        C[0][0] = S[1][1] * S[2][2] - S[1][2] * S[2][1];
        C[0][1] = S[0][2] * S[2][1] - S[0][1] * S[2][2];
        C[0][2] = S[0][1] * S[1][2] - S[0][2] * S[1][1];
        C[1][0] = S[1][2] * S[2][0] - S[1][0] * S[2][2];
        C[1][1] = S[0][0] * S[2][2] - S[0][2] * S[2][0];
        C[1][2] = S[0][2] * S[1][0] - S[0][0] * S[1][2];
        C[2][0] = S[1][0] * S[2][1] - S[1][1] * S[2][0];
        C[2][1] = S[0][1] * S[2][0] - S[0][0] * S[2][1];
        C[2][2] = S[0][0] * S[1][1] - S[0][1] * S[1][0];
        const real det = S[0][0] * C[0][0] + S[0][1] * C[1][0] + S[0][2] * C[2][0];
        for (int d = 0; d < 3; d++)
            for (int e = 0; e < 3; e++)
                Si[d][e] = C[d][e] / det;
    }
    for (int v = 0; v < NV; v++)
        for (int e = 0; e < DIM; e++)
        {
            real a = 0;
            for (int d = 0; d < DIM; d++)
                a += Si[d][e] * gb[v][d];
            q[((size_t)v * DIM + e) * N + i] = a;
        }
}

template <int DIM, int NV>
__global__ void __launch_bounds__(64) kVR2ndTGather(DevMesh m, const real *__restrict__ u,
                                                    const real *__restrict__ q, real *__restrict__ ubar)
{
    const idx j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= m.N)
        return;
    const size_t N = m.N, F = m.F;
    const int method = m.s.subs2ndOrder;
    const bool plain = m.s.subs2ndOrderGGScheme == 0;
    real qj[NV][DIM], acc[NV];
    for (int v = 0; v < NV; v++)
    {
        acc[v] = 0;
        for (int d = 0; d < DIM; d++)
            qj[v][d] = q[((size_t)v * DIM + d) * N + j];
    }
    for (int k = 0; k < m.K; k++)
    {
        const idx f = m.c2f[(size_t)k * N + j];
        if (f < 0)
            continue;
        const idx o = m.c2c[(size_t)k * N + j];
        real w[3];
        vr2ndFaceWeight<DIM>(m, j, k, method, plain, w);
        real s[NV]; // this face's own term: -c_jk . q_j
        for (int v = 0; v < NV; v++)
        {
            s[v] = 0;
            for (int d = 0; d < DIM; d++)
                s[v] += w[d] * qj[v][d];
            acc[v] -= s[v];
        }
        if (o >= 0)
        {
            // u_j as the neighbour of o, across o's slot of this face
            const int ko = m.c2s[(size_t)k * N + j];
            real wo[3];
            vr2ndFaceWeight<DIM>(m, o, ko, method, plain, wo);
            for (int v = 0; v < NV; v++)
                for (int d = 0; d < DIM; d++)
                    acc[v] += wo[d] * q[((size_t)v * DIM + d) * N + o];
        }
        else if constexpr (NV == 5)
        {
            // the ghost of u_j at the face centre (mean normal): its Jacobian transposed
            const int zone = m.fzone[f];
            real n[3];
            for (int r = 0; r < 3; r++)
                n[r] = m.fmeanN[(size_t)r * F + f];
            for (int cc = 0; cc < 5; cc++)
            {
                Dual U[5], G[5];
                for (int v = 0; v < 5; v++)
                    U[v] = Dual(u[(size_t)v * N + j], v == cc ? 1.0 : 0.0);
                bcGhost(m.bcType[zone], U, n, m.bcVal + (size_t)zone * 5, m.bcGamma, G);
                real a = 0;
                for (int v = 0; v < 5; v++)
                    a += G[v].d * s[v];
                acc[cc] += a;
            }
        }
    }
    for (int v = 0; v < NV; v++)
        ubar[(size_t)v * N + j] = acc[v];
}

void launchVRIterVJP(Ctx &c, int nVars, int mode, real relax, const real *uRec, const real *u, const real *ybar,
                     real *xbar, real *ubar)
{
    if (usesSubs2nd(c.m))
    {
        // every mode writes G(u): nothing flows back to uRec; IterDiff (mode 3) is zero
        KernelTimer kt(c, K_ADJOINT);
        const DevMesh &m = c.m;
        const size_t nR = (size_t)nVars * m.M * m.N;
        if (xbar)
            DNDSR_HIP_CHECK(hipMemsetAsync(xbar, 0, nR * sizeof(real), c.stream));
        if (mode == 3 || !ubar)
            return;
        if (nVars != 5 && nVars != 1)
            throw std::runtime_error("nVars must be 1 or 5");
        if (m.nBnd > 0 && !(nVars == 5 && m.bcType != nullptr && u != nullptr))
            throw std::runtime_error("the transposed second-order substitute on a mesh with boundary faces needs the "
                                     "Euler boundary table (nVars 5) and the base state u");
        if (!c.adj2ndQ)
            c.adj2ndQ = devAlloc<real>(c, (size_t)5 * 3 * m.N);
        const int g = gridFor(m.N, 64);
        if (m.dim == 2)
        {
            if (nVars == 5)
                kVR2ndTq<2, 5><<<g, 64, 0, c.stream>>>(m, ybar, c.adj2ndQ),
                    kVR2ndTGather<2, 5><<<g, 64, 0, c.stream>>>(m, u, c.adj2ndQ, ubar);
            else
                kVR2ndTq<2, 1><<<g, 64, 0, c.stream>>>(m, ybar, c.adj2ndQ),
                    kVR2ndTGather<2, 1><<<g, 64, 0, c.stream>>>(m, u, c.adj2ndQ, ubar);
        }
        else
        {
            if (nVars == 5)
                kVR2ndTq<3, 5><<<g, 64, 0, c.stream>>>(m, ybar, c.adj2ndQ),
                    kVR2ndTGather<3, 5><<<g, 64, 0, c.stream>>>(m, u, c.adj2ndQ, ubar);
            else
                kVR2ndTq<3, 1><<<g, 64, 0, c.stream>>>(m, ybar, c.adj2ndQ),
                    kVR2ndTGather<3, 1><<<g, 64, 0, c.stream>>>(m, u, c.adj2ndQ, ubar);
        }
        DNDSR_HIP_CHECK(hipGetLastError());
        return;
    }
    // mode 0 Jacobi (relax), 1 recordInc, 2 recordInc + uRecIsZero, 3 IterDiff
    real c0 = 1, c1 = -1;
    int useB = 1, useb = 1;
    if (mode == 0)
        c0 = 1 - relax, c1 = relax;
    else if (mode == 2)
        c0 = 0, useB = 0;
    else if (mode == 3)
        useb = 0;
    KernelTimer kt(c, K_ADJOINT);
    switch (c.m.M)
    {
    case 2: vrTLaunch<2>(c, nVars, ybar, xbar, ubar, c0, c1, useB, useb); break;
    case 3: vrTLaunch<3>(c, nVars, ybar, xbar, ubar, c0, c1, useB, useb); break;
    case 5: vrTLaunch<5>(c, nVars, ybar, xbar, ubar, c0, c1, useB, useb); break;
    case 9: vrTLaunch<9>(c, nVars, ybar, xbar, ubar, c0, c1, useB, useb); break;
    case 19: vrTLaunch<19>(c, nVars, ybar, xbar, ubar, c0, c1, useB, useb); break;
    default: throw std::runtime_error("unsupported number of reconstruction modes");
    }
    // boundary term (Jacobi: relax A^-1 BCC; recordInc: -A^-1 BCC; none with uRecIsZero)
    const DevMesh &m = c.m;
    if (m.nBnd == 0 || mode == 2)
        return;
    if (mode == 3)
        throw std::runtime_error("the transposed VR Jacobian (IterDiff) covers meshes without boundary faces");
    const bool euler = nVars == 5 && m.bcType != nullptr;
    if (!euler && !(m.dirVal && m.dirNV == nVars))
        throw std::runtime_error("the mesh has boundary faces: set the boundary conditions first");
    if (!u || (euler && !uRec))
        throw std::runtime_error("the transposed VR sweep on a mesh with boundary faces needs the base state uRec, u");
    const real scale = mode == 0 ? relax : -1.0;
    if (m.dim == 2)
    {
        if (m.P == 1)
            vrBndTLaunch<2, 3>(c, nVars, uRec, u, ybar, scale, xbar, ubar);
        else if (m.P == 2)
            vrBndTLaunch<2, 6>(c, nVars, uRec, u, ybar, scale, xbar, ubar);
        else
            vrBndTLaunch<2, 10>(c, nVars, uRec, u, ybar, scale, xbar, ubar);
    }
    else
    {
        if (m.P == 1)
            vrBndTLaunch<3, 4>(c, nVars, uRec, u, ybar, scale, xbar, ubar);
        else if (m.P == 2)
            vrBndTLaunch<3, 10>(c, nVars, uRec, u, ybar, scale, xbar, ubar);
        else
            vrBndTLaunch<3, 20>(c, nVars, uRec, u, ybar, scale, xbar, ubar);
    }
}

} // namespace dndsr
