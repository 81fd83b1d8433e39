// internal.hpp -- context, device mesh and launcher declarations shared by the
// HIP translation units of libdndsr_amd.so (not part of the C-ABI).
#pragma once
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>
#include <vector>

#include "dev_common.hpp"

#define DNDSR_HIP_CHECK(x)                                                                          \
    do                                                                                              \
    {                                                                                               \
        hipError_t e_ = (x);                                                                        \
        if (e_ != hipSuccess)                                                                       \
            throw std::runtime_error(std::string(#x) + " failed: " + hipGetErrorString(e_));        \
    } while (0)

namespace dndsr
{
enum ElemType : int
{
    E_LINE2 = 1,
    E_QUAD4 = 2,
    E_HEX8 = 3,
    E_TRI3 = 4,
    E_TET4 = 5,
};

struct VRSettingsDev
{
    int maxOrder;
    int intOrder;
    int dirWeightScheme;  // 0 Factorial, 1 HQM_OPT
    int geomWeightScheme; // 0 GWNone, 1 HQM_SD
    real geomWeightBias;
    real geomWeightPower;
    real scaleMultiplier;
    real jacobiRelax;
    int nIterCellSmoothScale;
    real bcWeight;
    bool SORInstead; // solver loops sweep the reconstruction in place (multicolour SOR)
    int subs2ndOrder;         // maxOrder 1: 0 VR, 1 Gauss rule, 2 least squares
    int subs2ndOrderGGScheme; // 1 distance-weighted face value, 0 plain average
};

// Device-resident mesh, metrics and VR coefficients (all arrays SoA, see dev_common.hpp).
struct DevMesh
{
    int dim = 0, P = 0, NDOF = 0, M = 0;
    idx N = 0, F = 0, nNode = 0;
    int K = 0;      // max faces per cell
    int G = 0;      // face quadrature points
    int Gc = 0;     // cell quadrature points
    int cellType = 0, faceType = 0; // cellType: the type of every cell, or 0 on a mixed mesh
    int8_t *ctype = nullptr;         // [N] per-cell type on a mixed (Tri3 + Quad4) mesh
    VRSettingsDev s{};
    // connectivity
    idx *f2c = nullptr;     // [2][F], -1 = boundary
    idx *c2f = nullptr;     // [K][N], -1 = absent
    idx *c2c = nullptr;     // [K][N] cell across face slot k, -1 = absent
    int32_t *c2s = nullptr; // [K][N] slot of the same face in that neighbour cell
    uint8_t *c2flag = nullptr; // [K][N] bit 0: the cell is the face's front (R) side;
                               //        bit 1: the neighbour's colour precedes the cell's;
                               //        bits 2, 3: the neighbour is in the first, last colour
    float *fareaF = nullptr, *fmeanNF = nullptr, *volF = nullptr; // FP32 copies for the FP32 sweeps
    idx *cell2node = nullptr; // [nnc][N] (nnc = the most nodes of a cell type present)
    idx *face2node = nullptr; // [nnf][F]
    real *coords = nullptr;   // [3][nNode]
    // geometry
    real *fshift = nullptr;   // [3][F]
    real *fpts = nullptr;     // [G][3][F]
    real *fnorm = nullptr;    // [G][3][F]
    real *fwj = nullptr;      // [G][F]   w * (JDet + tiny)
    // the boundary faces' rows of these, in bndFace order ([.][nBnd]): in the face tables every value of a
    // boundary face is in a cache line of its own (42 values a face on triangles, 5 KB of lines; two
    // iterations on 945k tetrahedra 3203 us with the face tables, 3131 with these, on 83k 941 / 896)
    real *bpts = nullptr, *bnorm = nullptr, *bwj = nullptr;
    real *farea = nullptr;    // [F]
    real *fmeanN = nullptr;   // [3][F]
    real *fcent = nullptr;    // [3][F]
    real *faceL = nullptr;    // [F]
    real *faceW = nullptr;    // [P+1][F]
    real *vol = nullptr, *cent = nullptr, *bary = nullptr, *scale = nullptr, *smooth = nullptr;
    real *iscale = nullptr;   // [N] 1 / scale
    real *moment = nullptr;   // [M][N]
    real *cpts = nullptr;     // [Gc][3][N]
    real *cwj = nullptr;      // [Gc][N]
    // linear reconstruction (facelin.hip): [N][4] or [N][8] cell constants; [F] the inverse viscous distance
    // of interior faces with one normal
    real *linC = nullptr, *linDist = nullptr;
    // VR
    real *AinvB = nullptr;    // [(K+1)*M*M][N]
    real *Ainvb = nullptr;    // [K*M][N]
    // multicolour ordering of cells for the Gauss-Seidel sweeps
    int nColor = 0;
    std::vector<idx> colorPtrHost;
    idx *colorCells = nullptr; // [N] cells grouped by colour (the cell at each colour-major position)
    idx *cellPos = nullptr;    // [N] the colour-major position of each cell (inverse of colorCells)
    // the SOR sweep's cell lists: per colour (the ranges of colorPtrHost) the cells without a
    // boundary face first, then those with one, from sorSplitHost[colour] on
    idx *sorCells = nullptr;
    std::vector<idx> sorSplitHost;
    int32_t *color = nullptr;  // [N]
    real globalVol = 0;
    // boundary faces (face2cell[f][1] = -1) and their zones
    int nBCZone = 0;
    bool gasBC = false; // a zone of the boundary table is BCWallIsothermal or BCInPsTs
    idx nBnd = 0, nBndCell = 0;
    int32_t *fzone = nullptr;   // [F] zone of a boundary face, -1 elsewhere
    idx *bndFace = nullptr;     // [nBnd]
    idx *bndCell = nullptr;     // [nBndCell] cells with at least one boundary face
    int32_t *bndSlot = nullptr; // [K][nBndCell] index in bndFace of the face at slot k of bndCell[j], -1 elsewhere
    real *zoneW = nullptr;      // [nBCZone][P+1] boundary direction weights (setup only)
    // boundary-condition table (dndsr_set_bc) and VR boundary point values (dndsr_set_vr_dirichlet)
    int32_t *bcType = nullptr;  // [nBCZone]
    real *bcVal = nullptr;      // [nBCZone][5]
    real bcGamma = 1.4;
    int dirNV = 0;
    const real *dirVal = nullptr; // [dirNV][G][F]
};

struct Ctx
{
    int device = 0;
    hipStream_t stream = nullptr;
    DevMesh m;
    bool haveMesh = false;
    // scratch owned by the context (grown on demand, freed at destroy)
    real *faceFlux = nullptr;   // [5][F]
    real *vrBnd = nullptr;      // [nVars][M][nBnd] A^-1 BCC of each boundary face (VR sweep boundary term)
    // the SOR sweep's matrices in list order (vr.hip, prepareSOR): sweeps before it was asked for, whether it
    // was, and the copy, null without the memory for it
    int sorUse = 0;
    bool sorTried = false;
    real *sorB = nullptr;
    size_t faceFluxCap = 0;
    real *red = nullptr;        // reduction partials
    size_t redCap = 0;
    real *hostRed = nullptr;    // pinned host mirror of reductions
    real *faceLamTmp = nullptr; // [2][F] (lambdaFace, deltaLambdaFace)
    real *adjPoint = nullptr;   // point or face sensitivities of the RHS adjoint (adjBufferSize values)
    size_t adjPointCap = 0;
    real *adjFaceBar = nullptr; // [5][F] face-flux adjoint
    real *adj2ndQ = nullptr;    // [5][3][N] per-cell weights of the transposed second-order substitute
    real *adjRhs = nullptr;     // [5][N] residual of a functional's forward evaluation
    size_t faceLamCap = 0;
    int *nonFinite = nullptr;   // set by the residual gather when a cell's residual is not finite
    std::vector<void *> owned;  // device allocations freed at destroy
    // optional per-kernel timing with HIP events on the launch stream
    bool timing = false;
    struct TimedRec
    {
        int id;
        hipEvent_t a, b;
    };
    std::vector<TimedRec> recs;
    std::vector<hipEvent_t> evPool;
    double kernMs[16] = {0};
    long long kernCount[16] = {0};
};

// kernel ids reported by dndsr_get_timing
enum KernelId : int
{
    K_VR_ITER = 0,
    K_RHS_FACE = 1,
    K_RHS_GATHER = 2,
    K_DT_FACE = 3,
    K_DT_CELL = 4,
    K_AXPBY = 5,
    K_SGS = 6,
    K_LUSGS_INIT = 7,
    K_DUAL_RES = 8,
    K_INCREMENT = 9,
    K_CONVERT = 10,
    K_ADJOINT = 11,
    K_LINSOLVE = 12,
    K_RHS_VISCOUS = 13,
    K_NUM = 14,
};

// Records a HIP event pair around the launches in its scope when timing is on.
struct KernelTimer
{
    Ctx &c;
    int id;
    hipEvent_t b = nullptr;
    KernelTimer(Ctx &cc, int kid) : c(cc), id(kid)
    {
        if (!c.timing)
            return;
        hipEvent_t a = take();
        b = take();
        DNDSR_HIP_CHECK(hipEventRecord(a, c.stream));
        c.recs.push_back({id, a, b});
    }
    ~KernelTimer()
    {
        if (b)
            (void)hipEventRecord(b, c.stream);
    }
    hipEvent_t take()
    {
        if (!c.evPool.empty())
        {
            hipEvent_t e = c.evPool.back();
            c.evPool.pop_back();
            return e;
        }
        hipEvent_t e;
        DNDSR_HIP_CHECK(hipEventCreate(&e));
        return e;
    }
};

// ---- launchers (setup.hip)
void setupMetricsAndVR(Ctx &c);
// ---- launchers (vr.hip)
void launchVRIter(Ctx &c, int nVars, const real *uRec, real *uRecNew, const real *u, int mode, real relax);
void launchVRSOR(Ctx &c, int nVars, real *uRec, const real *u, real relax);
void prepareSOR(Ctx &c);
void refreshSOR(Ctx &c);
bool usesSubs2nd(const DevMesh &m);
void launchVR2nd(Ctx &c, int nVars, const real *u, real *out);
void launchVRIterDiff(Ctx &c, int nVars, const real *uRec, const real *u, const real *uRecDiff, real *uRecNew);
// ---- launchers (euler.hip)
// partials: dtMinDev may be left unwritten; the return value is then the number of partial minima in
// the context's reduction buffer (0: dtMinDev holds the minimum)
int launchEvalDt(Ctx &c, const GasParams &gp, const real *u, real CFL, real maxDt, int useLocalDt, real *dt,
                 real *lambdaFace, real *deltaLambdaCell, real *dtMinDev, bool partials = false);
// Optional stage combination fused into the RHS gather: out = a u + b y + cdt dt RHS (y optional; save
// receives u first).  dt is dtDev[0], the least of the nPart values at dtDev where nPart > 0, or 1.
// out null or u: in place, the face pass reading u before the gather starts; the one-pass form of small
// meshes (rhsCellRule) needs another array.
struct StageUpdate
{
    real a = 0, b = 0, cdt = 0;
    const real *y = nullptr, *dtDev = nullptr;
    const real *u = nullptr;
    real *out = nullptr, *save = nullptr;
    int nPart = 0;
};
// faceFluxBuf: the [5][F] face-flux scratch (NULL = the context's); flagNonFinite: raise the
// context's non-finite flag from the gather
void launchEvalRHS(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *deltaLambdaCell,
                   real *rhs, const StageUpdate *stage = nullptr, real *faceFluxBuf = nullptr,
                   bool flagNonFinite = true);
// ---- launchers (facelin.hip): fluxes (inviscid and viscous) of the interior faces and inviscid boundary
// fluxes with a linear or no reconstruction, for the face rules rhsLinearRule names
bool rhsLinearRule(const DevMesh &m);
bool rhsLinearViscous(const DevMesh &m);
void setupLinear(Ctx &c);
// the one-pass form of small meshes: whether the mesh may take it, whether a call does (its flux and its
// output apart from what it reads), and the launch
bool rhsCellSize(const DevMesh &m);
bool rhsCellRule(const Ctx &c, bool viscous, const real *u, const real *uRec, const real *dlc, const real *rhs,
                 const StageUpdate *stage);
void launchRHSCellLinear(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc, real *ff,
                         real *rhs, const StageUpdate &stage, int *nonFinite);
// the viscous flux (euler.hip) of all faces, or of the boundary faces only
void launchRHSViscous(Ctx &c, const GasParams &gp, const real *u, const real *uRec, real *ff, bool bndOnly);
void launchRHSFaceLinear(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc, real *ff);
void launchLUSGSInit(Ctx &c, const real *dTau, real dt, real alphaDiag, const real *lambdaFace, real *jdiag);
// a sweep of the transposed scalar LU-SGS matrix (the adjoint preconditioner), FP64
void launchSGSSweepT64(Ctx &c, const GasParams &gp, real alphaDiag, const real *rhs, const real *u, const real *uInc,
                       real *uIncNew, const real *jdiag, const real *lambdaFace, int forward, int gsUpdate,
                       int uIncIsZero, real *sumIncDev, int fCol = -1, int lCol = -1);
real *launchSGSSymmetric64(Ctx &c, const GasParams &gp, real alphaDiag, const real *rhs, const real *u, real *a,
                           real *b, const real *jd, const real *lam, int nSweep, int gsUpdate, real *sumIncDev);
float *launchSGSSymmetric32(Ctx &c, const GasParams &gp, float alphaDiag, const float *rhs, const float *u, float *a,
                            float *b, const float *jd, const float *lam, int nSweep, int gsUpdate, real *sumIncDev);
void launchSGSSweep64(Ctx &c, const GasParams &gp, real alphaDiag, const real *rhs, const real *u, const real *uInc,
                      real *uIncNew, const real *jdiag, const real *lambdaFace, int forward, int gsUpdate,
                      int uIncIsZero, real *sumIncDev);
void launchSGSSweep32(Ctx &c, const GasParams &gp, float alphaDiag, const float *rhs, const float *u,
                      const float *uInc, float *uIncNew, const float *jdiag, const float *lambdaFace, int forward,
                      int gsUpdate, int uIncIsZero, real *sumIncDev);
// out = a x + b y + cdt dt z (y, z, dtDev optional); save, when given, receives x first
// Roe-Jacobian block LU-SGS (useRoeJacobian): face eigenvalues lamRoe [3][F], block JDiag and its
// inverse [25][N] (bad set when a block cannot be inverted), block sweeps
void launchFaceRoeLambda(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc, real *lamRoe);
void launchLUSGSInitBlock(Ctx &c, const GasParams &gp, const real *dTau, real dt, real alphaDiag, const real *u,
                          const real *lam, const real *lamRoe, real *jd, real *jinv, int *bad);
// Half sums of the symmetric Gauss-Seidel solves (sgs.hip, roejac.hip; Conrad & Wallach 1979).  A cell's
// neighbours before it (in colour-major position) change between a backward visit and the next forward
// one, those after it between a forward visit and the next backward one; so a forward visit sums the
// former only, a backward visit the latter, and the other half is the sum its last visit kept (half).
// The first and the last colour have neighbours on one side only and keep nothing.  Two implicit
// iterations, all neighbours in each visit against one side (5 colours on tetrahedra, 3 on the mixed 2-D
// mesh, 5 extra sweeps there): 24 576 tetrahedra 457 / 442 us, 279 936 1141 / 1120 us, 944 784 in FP32
// 2401 / 2318 us; blocks on 50k cells of the 2-D mesh 652 / 596 us, on 97k 795 / 729 us; the scalar solve
// on 200k cells of it, where they do not pay, 746 / 747 us.
enum SGSSide { SGS_NONE = 0, SGS_BEFORE = 1, SGS_AFTER = 2, SGS_ALL = 3 };
struct SGSVisit
{
    int side;           // the neighbours summed
    bool read, keep;    // the half sum
};
inline SGSVisit sgsVisit(const DevMesh &m, int col, bool forward, bool first, bool last)
{
    const bool inner = col > 0 && col < m.nColor - 1;
    return {forward ? SGS_BEFORE : SGS_AFTER, inner && !first, inner && !last};
}
// the implicit loop's block solve (roejac.hip): workspace per precision, allocated at its first use;
// *result: the increment, rows of 8 in colour-major position order; bad set when a block is singular
template <typename T>
struct SGSBlockWork
{
    T *x[2] = {nullptr, nullptr}, *C = nullptr, *b = nullptr;
    T *half = nullptr; // [5][N] the kept half sums (SGSVisit)
    idx *nbr = nullptr;
};
void launchSGSBlockSolve64(Ctx &c, const GasParams &gp, real alphaDiag, const real *rhs, real dt, const real *u,
                           const real *dTau, const real *lam, const real *lamRoe, SGSBlockWork<real> &w, int sgsIter,
                           int gsUpdate, int *bad, real **result);
void launchSGSBlockSolve32(Ctx &c, const GasParams &gp, real alphaDiag, const real *rhs, real dt, const real *u,
                           const real *dTau, const real *lam, const real *lamRoe, SGSBlockWork<float> &w, int sgsIter,
                           int gsUpdate, int *bad, float **result);
void launchSGSSweepBlock64(Ctx &c, const GasParams &gp, real alphaDiag, const real *rhs, const real *u,
                           const real *uInc, real *uIncNew, const real *jinv, const real *lam, const real *lamRoe,
                           int forward, int gsUpdate, int uIncIsZero, real *sumIncDev);
void launchSGSSweepBlockT64(Ctx &c, const GasParams &gp, real alphaDiag, const real *rhs, const real *u,
                            const real *uInc, real *uIncNew, const real *jinv, const real *lam, const real *lamRoe,
                            int forward, int gsUpdate, int uIncIsZero, real *sumIncDev, int fCol = -1,
                            int lCol = -1);
void launchCopyColourInc64(Ctx &c, int col, const real *from, real *to);
void launchSGSSweepBlock32(Ctx &c, const GasParams &gp, float alphaDiag, const float *rhs, const float *u,
                           const float *uInc, float *uIncNew, const float *jinv, const float *lam,
                           const float *lamRoe, int forward, int gsUpdate, int uIncIsZero, real *sumIncDev);
// device bandwidth self-test (probe.hip): mode 0 read stream, 1 copy; average ms per pass
double streamProbe(Ctx &c, int mode, const double *src, double *dst, size_t n, int reps);
int streamProbeBlocks(Ctx &c);
// sum of nPart 5-wide partials in c.red into out[5]
void launchReduceSum5(Ctx &c, int nPart, real *out);
void launchAxpby(Ctx &c, idx n, real a, const real *x, real b, const real *y, real cdt, const real *z,
                 const real *dtDev, real *out, real *save = nullptr);
// dst[0:n) = src[0:n) on the library's stream
void launchCopy(Ctx &c, size_t n, const real *src, real *dst);
// the BDF unsteady residual: sum_j coef_j / dt xs_j - x / dt + alpha rhsF, nx in 1..4 (xs[0] = xLast)
void launchDualResidualBDF(Ctx &c, real dt, const real *const *xs, const real *coef, int nx, real alpha,
                           const real *x, const real *rhsF, real *rhs, real *resDev);
void launchScale(Ctx &c, idx n, real s, real *x);
void launchDualResidual(Ctx &c, real dt, const real *xLast, const real *x, const real *rhsF, real *rhs,
                        real *resDev);
// statistics of the positivity-preserving increment: limited cells, smallest alpha (as the bits
// of a positive double), and a flag for states the reference asserts against
struct PPStat
{
    unsigned long long alphaMinBits;
    int nLim;
    int bad;
};
void launchPPStatReset(Ctx &c, PPStat *stat);
// fincrement: u += CompressInc(u, alpha du) with alpha from EvaluateCellRHSAlpha, per cell
void launchAddIncrement64(Ctx &c, real gamma, real relax, real rhoEps, real pEps, real *u, const real *du,
                          PPStat *stat);
void launchToF32(Ctx &c, size_t n, const real *in, float *out);
// the sum of a dual-time residual: sum_j a_j x_j over xLast and up to three earlier states
struct BDFTerms
{
    const real *x[4];
    real a[4];
    int n;
};
// the implicit loop's LU-SGS solve (sgs.hip): workspace per precision, allocated at its first use
template <typename T>
struct SGSWork
{
    T *x[2] = {nullptr, nullptr}; // increments [N][8] in colour-major position order (the second: Jacobi)
    T *rec = nullptr, *nq = nullptr, *st = nullptr;
    T *half = nullptr; // [5][N] the kept half sums (SGSVisit)
    idx *nbr = nullptr, *face = nullptr;
};
// rhs = bt - u / dt + alpha rhsF with its L1 norm into resDev, LUSGSMatrixInit's scalar diagonal, and
// (1 + sgsIter) forward/backward sweeps from a zero increment; *result: the increment, rows of 8 in
// colour-major position order.  half: [K][N] mesh constants shared by the precisions
void launchSGSSolve64(Ctx &c, const GasParams &gp, real alpha, const BDFTerms &bt, real dt, const real *u,
                      const real *rhsF, const real *dTau, const real *lam, SGSWork<real> &w, real *&half, int sgsIter,
                      int gsUpdate, real *resDev, real **result);
void launchSGSSolve32(Ctx &c, const GasParams &gp, real alpha, const BDFTerms &bt, real dt, const real *u,
                      const real *rhsF, const real *dTau, const real *lam, SGSWork<float> &w, real *&half,
                      int sgsIter, int gsUpdate, real *resDev, float **result);
// u += du with du the LU-SGS solve's increment, rows of 8 in colour-major position order (exactly one
// of du64 / du32 non-null)
void launchAddIncrementCellMajor(Ctx &c, real gamma, real relax, real rhoEps, real pEps, real *u, const real *du64,
                                 const float *du32, PPStat *stat);
// ---- launchers (model.hip): ModelEvaluator::EvaluateRHS, scalar advection-diffusion (2-D)
void launchModelRHS(Ctx &c, int nVars, real ax, real ay, real sigma, const real *u, const real *uRec, real *rhs);
// ---- linear solver (linsolve.hip)
struct LinWork
{
    // operator: LU-SGS matrix at the state u (FP64) and its FP32 copies for FP32 sweeps
    const real *u = nullptr, *jd = nullptr, *lam = nullptr;
    const float *fU = nullptr, *fJd = nullptr, *fLam = nullptr;
    real alphaDiag = 1.0;
    int sgsIter = 0, gsUpdate = 1, fp32 = 0;
    // scratch: FP32 sweep vectors, FP64 sweep vector, Krylov basis [(k+1)][5N], temporaries
    float *fR = nullptr, *fX = nullptr, *fT = nullptr;
    real *dT = nullptr, *V = nullptr, *Vt = nullptr, *MLb = nullptr, *h = nullptr, *part = nullptr,
         *scal = nullptr, *coef = nullptr;
};
void launchLUSGSMatVec(Ctx &c, const GasParams &gp, real alphaDiag, const real *u, const real *x, const real *jd,
                       const real *lam, real *Ax);
void applyLUSGSPrecond(Ctx &c, const GasParams &gp, const LinWork &w, const real *r, real *out);
int gmresSolve(Ctx &c, const GasParams &gp, const LinWork &w, const real *b, real *x, int kSub, int nRestart,
               double *residualOut);
// ---- launchers (adjoint.hip)
size_t adjBufferSize(const DevMesh &m, bool viscous);
// faceBar (optional, [5][F]): the adjoint of the face fluxes instead of the residual's
// (rbar unused then); without it the face adjoint is formed from rbar
void launchEvalRHSVJP(Ctx &c, const GasParams &gp, const real *u, const real *uRec, const real *dlc,
                      const real *rbar, real *ubar, real *urecbar, const real *faceBar = nullptr);
// force on the boundary faces of a zone from the last EvaluateRHS's face fluxes:
// forceDev[d] = - sum_f ff[1 + d][f] (the momentum flux out of the domain)
void launchZoneForce(Ctx &c, int zone, real *forceDev);
// face-flux adjoint of that force: fbar[1 + d][f] = -forceBar[d] on the zone's faces, 0 elsewhere
void launchZoneForceBar(Ctx &c, int zone, const real *forceBarDev, real *fbar);
void launchVRIterVJP(Ctx &c, int nVars, int mode, real relax, const real *uRec, const real *u, const real *ybar,
                     real *xbar, real *ubar);

template <typename T>
T *devAlloc(Ctx &c, size_t n)
{
    void *p = nullptr;
    if (n == 0)
        n = 1;
    DNDSR_HIP_CHECK(hipMalloc(&p, n * sizeof(T)));
    c.owned.push_back(p);
    return static_cast<T *>(p);
}

// The quadrature points, normals and weights of one face: a column of the face tables, or of the
// boundary faces' own
struct FacePts
{
    const real *pts, *norm, *wj;
    size_t S;
    idx q;
    __device__ __forceinline__ real x(int g, int r) const { return pts[((size_t)g * 3 + r) * S + q]; }
    __device__ __forceinline__ real n(int g, int r) const { return norm[((size_t)g * 3 + r) * S + q]; }
    __device__ __forceinline__ real w(int g) const { return wj[(size_t)g * S + q]; }
};
__device__ __forceinline__ FacePts facePts(const DevMesh &m, idx f) { return {m.fpts, m.fnorm, m.fwj, (size_t)m.F, f}; }
__device__ __forceinline__ FacePts bndPts(const DevMesh &m, idx t) { return {m.bpts, m.bnorm, m.bwj, (size_t)m.nBnd, t}; }
inline int gridFor(idx n, int block) { return (int)((n + block - 1) / block); }
// Block size of the one-thread-per-cell gathers: one wavefront while 256-thread blocks would leave
// CUs without any (fewer than 512 of them), so that a small mesh spreads over the device
inline int cellBlock(idx n) { return n < 512 * 256 ? 64 : 256; }

// Where the slots of the cell at position p go among its K (4 bits each): by the neighbour's position,
// those before p first, those after it last, slots without a neighbour between them.  The lanes of a
// wavefront, one colour, then need mostly the same slots in a visit that sums one side.
__device__ inline uint32_t slotRanks(const DevMesh &m, idx i, idx p)
{
    idx key[kMaxFC];
#pragma unroll
    for (int k = 0; k < kMaxFC; k++)
    {
        const size_t q = (size_t)(k < m.K ? k : 0) * m.N + i;
        const idx o = m.c2c[q];
        key[k] = m.c2f[q] >= 0 && o >= 0 && o != i ? m.cellPos[o] : p;
    }
    uint32_t to = 0;
#pragma unroll
    for (int k = 0; k < kMaxFC; k++)
    {
        uint32_t r = 0;
#pragma unroll
        for (int j = 0; j < kMaxFC; j++)
            r += j < m.K && (key[j] < key[k] || (key[j] == key[k] && j < k));
        to |= r << (4 * k);
    }
    return to;
}

// Skipped colour passes of the symmetric Gauss-Seidel sweeps: a sweep may skip its first colour
// (fCol; its current values stay in the array the sweep reads) and read the colour the previous
// sweep skipped (lCol) from the array it writes.  Both are the first or the last colour, which
// the slot flags mark (bits 2, 3); -1 names none.
__device__ __forceinline__ bool nbrInColour(uint8_t fl, int col, int nColor)
{
    return (col == 0 && (fl & 4)) || (col >= 0 && col == nColor - 1 && (fl & 8));
}
__device__ __forceinline__ bool sweepReadNew(uint8_t fl, int fCol, int lCol, int nColor, bool useNew)
{
    if (nbrInColour(fl, fCol, nColor))
        return false;
    if (nbrInColour(fl, lCol, nColor))
        return true;
    return useNew;
}

} // namespace dndsr
