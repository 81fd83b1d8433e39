// sgs.hip -- the LU-SGS solve of the device implicit loop with the scalar Jacobian: symmetric
// multicolour Gauss-Seidel (or Jacobi) sweeps from a zero increment, FP64 or FP32, on a
// colour-major copy of what they read.
//
// LUSGSMatrixInit (EulerEvaluator.hxx:37-159) and UpdateSGS (:550-693) with the same arithmetic as
// kLUSGSInit / kSGSColour.  The neighbour term is
//   0.5 alpha A_f / V_i (A(u_j) du_j . n - lambda_f du_j)
// and needs of u_j only the velocity v and the total enthalpy H: with the scaled normal
// q = n A_f / (2 V_i) and m, E the momentum and energy increments,
//   r = m . q - (v . q) drho,  dp = (gamma - 1) (dE - v . m + |v|^2 drho / 2),
//   dF = (m . q,  m (v . q) + v r + q dp,  (dE + dp) (v . q) + H r).
//
// Layout (position p holds cell colorCells[p], so a colour pass reads and writes one contiguous range
// whatever the caller's cell order; a neighbour precedes in the forward sweep exactly when its
// position is lower, the colouring having no neighbours of one colour):
//   inc [N][8]   the increment (5) and three zeros: a row is written whole, never part of a sector
//   st  [N][4]   v and H of the state
//   rec [N][12]  rhs (5), 1 / D, then lambda_f A_f / (2 V_i) per slot (6 at most)
//   nq  [3 K][N] q per slot, nbr [K][N] the neighbours' positions (both mesh-only)
// A pass is bound by the cache lines of its neighbour gathers and, on a mesh of up to a few hundred
// thousand cells per colour, by the latency of the chain neighbour index -> neighbour row (the whole
// pass is about one round of waves).  So a neighbour costs 64 + 32 bytes in 16-byte loads, everything
// a cell reads of its own is one record and coalesced rows, all K neighbour rows are in flight at
// once, and the blocks of one XCD take a contiguous range of positions (its L2 then serves the rows
// that several of them gather).  With three colours or more a visit gathers one side's neighbours only
// (SGSVisit).  Average pass, in place: 945k tetrahedra (5 colours) 20.5 us (23.4 with all neighbours,
// 4.9 TB/s of cache-line misses), 246k hexahedra (2 colours) 12.1 us (15.2 at three waves per SIMD, with
// 16 registers in scratch).
#include <utility>

#include "internal.hpp"

namespace dndsr
{
constexpr int kIncRow = 8, kStRow = 4, kRecRow = 12;

template <typename T>
struct SGSVec;
template <>
struct SGSVec<real>
{
    typedef double2 V;
    static constexpr int L = 2;
};
template <>
struct SGSVec<float>
{
    typedef float4 V;
    static constexpr int L = 4;
};
// n values at p (aligned to the vector) as vector loads
template <typename T, int n>
__device__ __forceinline__ void rowLoad(const T *p, T *out)
{
    using V = typename SGSVec<T>::V;
    constexpr int L = SGSVec<T>::L;
    static_assert(n % L == 0, "whole vectors");
#pragma unroll
    for (int q = 0; q < n / L; q++)
    {
        const V v = reinterpret_cast<const V *>(p)[q];
        const T *e = reinterpret_cast<const T *>(&v);
#pragma unroll
        for (int k = 0; k < L; k++)
            out[q * L + k] = e[k];
    }
}
template <typename T, int n>
__device__ __forceinline__ void rowStore(T *p, const T *in)
{
    using V = typename SGSVec<T>::V;
    constexpr int L = SGSVec<T>::L;
    static_assert(n % L == 0, "whole vectors");
#pragma unroll
    for (int q = 0; q < n / L; q++)
    {
        V v;
        T *e = reinterpret_cast<T *>(&v);
#pragma unroll
        for (int k = 0; k < L; k++)
            e[k] = in[q * L + k];
        reinterpret_cast<V *>(p)[q] = v;
    }
}

// the mesh-only part: scaled normals and neighbour positions per position, A_f / (2 V_i) per cell
template <typename T>
__global__ void __launch_bounds__(256) kSGSMesh(DevMesh m, T *__restrict__ nq, idx *__restrict__ nbr,
                                                idx *__restrict__ face, real *__restrict__ half)
{
    const idx p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= m.N)
        return;
    const size_t N = m.N, F = m.F;
    const idx i = m.colorCells[p];
    const real vol = m.vol[i];
    const uint32_t ranks = slotRanks(m, i, p);
    for (int k = 0; k < m.K; k++)
    {
        const idx f = m.c2f[(size_t)k * N + i];
        const idx o = m.c2c[(size_t)k * N + i];
        const real h = f >= 0 ? 0.5 * m.farea[f] / vol : 0.0;
        const real s = (m.c2flag[(size_t)k * N + i] & 1) ? -h : h;
        const uint32_t to = (ranks >> (4 * k)) & 15;
#pragma unroll
        for (int r = 0; r < 3; r++)
            nq[((size_t)to * 3 + r) * N + p] = f >= 0 ? (T)(m.fmeanN[r * F + f] * s) : T(0);
        nbr[(size_t)to * N + p] = (f < 0 || o < 0 || o == i) ? idx(-1) : m.cellPos[o];
        face[(size_t)to * N + i] = f;
        half[(size_t)to * N + i] = h;
    }
}

// The per-iteration part, one thread per cell in the caller's order (its reads are coalesced and each
// position's rows are written whole): the unsteady residual
//   rhs = sum_j a_j x_j - x / dt + alpha frhs(x)      (ODE.hpp:80-98, :440-451)
// with its L1 partial sums (as kDualResidual), LUSGSMatrixInit's diagonal
//   D = 1 / dTau + 1 / dt + alpha sum_f lambda_f A_f / (2 V_i),
// and the state's v and H.
template <typename T, int KM>
__global__ void __launch_bounds__(256) kSGSPrep(DevMesh m, real gamma, real alpha, BDFTerms bt, real rdt,
                                                const real *__restrict__ u, const real *__restrict__ rhsF,
                                                const real *__restrict__ dTau, const real *__restrict__ lam,
                                                const idx *__restrict__ face, const real *__restrict__ half,
                                                T *__restrict__ st, T *__restrict__ rec, real *__restrict__ part)
{
    __shared__ real sm[5][4];
    const idx i = blockIdx.x * blockDim.x + threadIdx.x;
    real loc[5] = {0, 0, 0, 0, 0};
    if (i < m.N)
    {
        const size_t N = m.N;
        idx f[KM];
        real h[KM], l[KM], U[5], r[kRecRow];
#pragma unroll
        for (int k = 0; k < KM; k++)
        {
            const size_t q = (size_t)(k < m.K ? k : 0) * N + i;
            f[k] = face[q];
            h[k] = half[q];
            if (k >= m.K || f[k] < 0)
                f[k] = 0, h[k] = 0;
        }
        const size_t p = m.cellPos[i];
        const real dtau = dTau[i];
#pragma unroll
        for (int v = 0; v < 5; v++)
            U[v] = u[v * N + i];
#pragma unroll
        for (int k = 0; k < KM; k++)
            l[k] = lam[f[k]];
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            const size_t k = (size_t)v * N + i;
            real a = bt.x[0][k] * bt.a[0];
            for (int j = 1; j < bt.n; j++)
                a += bt.x[j][k] * bt.a[j];
            a += U[v] * (-rdt);
            a += rhsF[k] * alpha;
            r[v] = a;
            loc[v] = fabs(a);
        }
        real D = 1.0 / dtau + rdt;
#pragma unroll
        for (int k = 0; k < kRecRow - 6; k++)
        {
            const real s = k < KM && h[k < KM ? k : 0] != 0 ? l[k < KM ? k : 0] * h[k < KM ? k : 0] : 0.0;
            r[6 + k] = s;
            D += alpha * s;
        }
        r[5] = 1.0 / D;
        const real ri = 1.0 / U[0];
        const real v[3] = {U[1] * ri, U[2] * ri, U[3] * ri};
        const real pr = (gamma - 1) * (U[4] - 0.5 * U[0] * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]));
        const T s4[4] = {(T)v[0], (T)v[1], (T)v[2], (T)((U[4] + pr) * ri)};
        T rT[kRecRow];
#pragma unroll
        for (int q = 0; q < kRecRow; q++)
            rT[q] = (T)r[q];
        rowStore<T, kStRow>(st + p * kStRow, s4);
        rowStore<T, kRecRow>(rec + p * kRecRow, rT);
    }
#pragma unroll
    for (int v = 0; v < 5; v++)
    {
        real a = loc[v];
#pragma unroll
        for (int s = 32; s > 0; s >>= 1)
            a += __shfl_xor(a, s);
        if ((threadIdx.x & 63) == 0)
            sm[v][threadIdx.x >> 6] = a;
    }
    __syncthreads();
    if (threadIdx.x < 5)
        part[(size_t)blockIdx.x * 5 + threadIdx.x] =
            (sm[threadIdx.x][0] + sm[threadIdx.x][1]) + (sm[threadIdx.x][2] + sm[threadIdx.x][3]);
}

// The positions [begin, end): xw = (rhs - alpha sum_k dF_k(x)) / D.  Gauss-Seidel: x and xw are the
// same array, one colour per launch, so a neighbour's row is its newest value; the neighbours of one
// side are summed (side) and, with HALF, the other side's sum is the one the cell's last visit kept
// (if any: read).  Jacobi: the whole mesh in one launch from the other array, all neighbours,
// or none in the sweep that starts from zero.
template <typename T, int K>
constexpr int sgsPassWaves()
{
    return sizeof(T) == 8 ? (K <= 4 ? 3 : 2) : 1; // FP64: the rows of 4 (6) slots in 168 (256) VGPRs, no scratch
}
template <typename T, int K, bool HALF>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(sgsPassWaves<T, K>())))
kSGSPass(size_t N, real gammaD, T alpha, const T *x, T *xw, const T *__restrict__ st, const T *__restrict__ rec,
         const T *__restrict__ nq, const idx *__restrict__ nbr, T *half, int read, int side, idx begin, idx end)
{
    const idx p = begin + xcdTile(blockIdx.x, gridDim.x) * 64 + (idx)threadIdx.x;
    if (p >= end)
        return;
    const T g1 = (T)gammaD - T(1);
    idx po[K];
#pragma unroll
    for (int k = 0; k < K; k++)
        po[k] = nbr[(size_t)k * N + p];
    bool use[K];
#pragma unroll
    for (int k = 0; k < K; k++)
        use[k] = po[k] >= 0 && (side & (po[k] < p ? SGS_BEFORE : SGS_AFTER));
    T q[K][3], r[kRecRow];
    rowLoad<T, kRecRow>(rec + (size_t)p * kRecRow, r);
#pragma unroll
    for (int k = 0; k < K; k++)
    {
        const size_t qp = !HALF || use[k] ? p : begin; // the slots not used share one line
#pragma unroll
        for (int d = 0; d < 3; d++)
            q[k][d] = nq[((size_t)k * 3 + d) * N + qp];
    }
    // the gathers are unconditional (the slots not used all read one row, of another colour if there is
    // one): a load under a branch makes the compiler wait for every earlier load at the join
    const size_t none = begin > 0 ? 0 : N - 1;
    T du[K][5], s[K][4], hs[5];
    if constexpr (HALF)
#pragma unroll
        for (int v = 0; v < 5; v++)
            hs[v] = half[(size_t)v * N + p];
#pragma unroll
    for (int k = 0; k < K; k++)
    {
        const size_t o = use[k] ? po[k] : none;
        T row[kIncRow];
        rowLoad<T, 4>(x + o * kIncRow, row);
        row[4] = x[o * kIncRow + 4];
#pragma unroll
        for (int v = 0; v < 5; v++)
            du[k][v] = row[v];
        rowLoad<T, kStRow>(st + o * kStRow, s[k]);
    }
    T acc[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < K; k++)
    {
        if (!use[k])
            continue;
        const T *v = s[k], *d = du[k];
        const T vq = v[0] * q[k][0] + v[1] * q[k][1] + v[2] * q[k][2];
        const T mq = d[1] * q[k][0] + d[2] * q[k][1] + d[3] * q[k][2];
        const T rr = mq - vq * d[0];
        const T v2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
        const T dp = g1 * (d[4] - (v[0] * d[1] + v[1] * d[2] + v[2] * d[3]) + T(0.5) * v2 * d[0]);
        const T l = r[6 + k];
        acc[0] += mq - l * d[0];
#pragma unroll
        for (int c = 0; c < 3; c++)
            acc[1 + c] += d[1 + c] * vq + v[c] * rr + q[k][c] * dp - l * d[1 + c];
        acc[4] += (d[4] + dp) * vq + v[3] * rr - l * d[4];
    }
    if constexpr (HALF)
#pragma unroll
        for (int v = 0; v < 5; v++)
        {
            half[(size_t)v * N + p] = acc[v];
            acc[v] += read ? hs[v] : T(0);
        }
    T out[kIncRow];
#pragma unroll
    for (int v = 0; v < kIncRow; v++)
        out[v] = v < 5 ? (r[v < 5 ? v : 0] - alpha * acc[v < 5 ? v : 0]) * r[5] : T(0);
    rowStore<T, kIncRow>(xw + (size_t)p * kIncRow, out);
}

template <typename T>
static void sgsPass(Ctx &c, const GasParams &gp, T alpha, SGSWork<T> &w, const T *x, T *xw, const SGSVisit &sv, idx b,
                    idx e)
{
    DevMesh &m = c.m;
    if (e <= b)
        return;
    KernelTimer kt(c, K_SGS);
    const int g = gridFor(e - b, 64);
    const bool half = sv.read || sv.keep;
    auto go = [&](auto kHalf, auto kWhole) {
        auto kern = half ? kHalf : kWhole;
        kern<<<g, 64, 0, c.stream>>>((size_t)m.N, gp.gamma, alpha, x, xw, w.st, w.rec, w.nq, w.nbr,
                                      w.half, sv.read, sv.side, b, e);
    };
    switch (m.K)
    {
    case 3: go(kSGSPass<T, 3, true>, kSGSPass<T, 3, false>); break;
    case 4: go(kSGSPass<T, 4, true>, kSGSPass<T, 4, false>); break;
    case 5: go(kSGSPass<T, 5, true>, kSGSPass<T, 5, false>); break;
    case 6: go(kSGSPass<T, 6, true>, kSGSPass<T, 6, false>); break;
    case 2: go(kSGSPass<T, 2, true>, kSGSPass<T, 2, false>); break;
    default: throw std::runtime_error("unsupported number of faces per cell");
    }
    DNDSR_HIP_CHECK(hipGetLastError());
}

template <typename T>
static void sgsSolve(Ctx &c, const GasParams &gp, real alphaD, const BDFTerms &bt, real dt, const real *u,
                     const real *rhsF, const real *dTau, const real *lam, SGSWork<T> &w, real *&half, int sgsIter,
                     int gsUpdate, real *resDev, T **result)
{
    DevMesh &m = c.m;
    const size_t N = m.N;
    const int nb = gridFor(m.N, 256);
    if (!w.st)
    {
        if (!half)
            half = devAlloc<real>(c, (size_t)m.K * N);
        w.x[0] = devAlloc<T>(c, kIncRow * N);
        w.rec = devAlloc<T>(c, kRecRow * N);
        w.nq = devAlloc<T>(c, (size_t)3 * m.K * N);
        w.nbr = devAlloc<idx>(c, (size_t)m.K * N);
        w.face = devAlloc<idx>(c, (size_t)m.K * N);
        if (m.nColor > 2)
            w.half = devAlloc<T>(c, 5 * N);
        w.st = devAlloc<T>(c, kStRow * N);
        kSGSMesh<T><<<nb, 256, 0, c.stream>>>(m, w.nq, w.nbr, w.face, half);
        DNDSR_HIP_CHECK(hipGetLastError());
    }
    if (!gsUpdate && !w.x[1])
        w.x[1] = devAlloc<T>(c, kIncRow * N);
    {
        KernelTimer kt(c, K_LUSGS_INIT);
        if (m.K <= 4)
            kSGSPrep<T, 4><<<nb, 256, 0, c.stream>>>(m, gp.gamma, alphaD, bt, 1.0 / dt, u, rhsF, dTau, lam, w.face, half,
                                                     w.st, w.rec, c.red);
        else
            kSGSPrep<T, kMaxFC><<<nb, 256, 0, c.stream>>>(m, gp.gamma, alphaD, bt, 1.0 / dt, u, rhsF, dTau, lam, w.face,
                                                          half, w.st, w.rec, c.red);
        DNDSR_HIP_CHECK(hipGetLastError());
        launchReduceSum5(c, nb, resDev);
    }
    const T alpha = (T)alphaD;
    T *x = w.x[0];
    if (!gsUpdate)
    {
        T *y = w.x[1];
        for (int s = 0; s < 2 * (1 + sgsIter); s++)
        {
            sgsPass<T>(c, gp, alpha, w, x, y, {s == 0 ? SGS_NONE : SGS_ALL, false, false}, 0, m.N);
            std::swap(x, y);
        }
    }
    else
        for (int s = 0; s <= sgsIter; s++)
            for (int dir = 1; dir >= 0; dir--)
            {
                // a sweep after the first begins with the colour the previous one ended with: that
                // pass would read the same increments and write the same values
                const bool first = s == 0 && dir == 1;
                for (int q = first || m.nColor < 2 ? 0 : 1; q < m.nColor; q++)
                {
                    const int col = dir ? q : m.nColor - 1 - q;
                    sgsPass<T>(c, gp, alpha, w, x, x, sgsVisit(m, col, dir, first, s == sgsIter && !dir),
                               m.colorPtrHost[col], m.colorPtrHost[col + 1]);
                }
            }
    *result = x;
}
void launchSGSSolve64(Ctx &c, const GasParams &gp, real alpha, const BDFTerms &bt, real dt, const real *u,
                      const real *rhsF, const real *dTau, const real *lam, SGSWork<real> &w, real *&half, int sgsIter,
                      int gsUpdate, real *resDev, real **result)
{
    sgsSolve<real>(c, gp, alpha, bt, dt, u, rhsF, dTau, lam, w, half, sgsIter, gsUpdate, resDev, result);
}
void launchSGSSolve32(Ctx &c, const GasParams &gp, real alpha, const BDFTerms &bt, real dt, const real *u,
                      const real *rhsF, const real *dTau, const real *lam, SGSWork<float> &w, real *&half,
                      int sgsIter, int gsUpdate, real *resDev, float **result)
{
    sgsSolve<float>(c, gp, alpha, bt, dt, u, rhsF, dTau, lam, w, half, sgsIter, gsUpdate, resDev, result);
}

} // namespace dndsr
