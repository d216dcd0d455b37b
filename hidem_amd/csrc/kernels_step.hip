// Per-timestep kernels for gfx950: force gather, time integration, link
// break and the rebuild (skin) reductions.
//
// Force gather (CombinedAccel::iterateCombined, CombinedAccel.h:121-197):
// one lane per particle, 64 consecutive particles per wavefront (states of few
// particles: six waves per 64 particles, k_step_tile).  A lane
// zeroes its force, applies the contact law to every neighbour-list entry in
// list order, then the beam law to each of its link sides in ascending link
// id, updating that side's CT0..CT5 in place, and finally overwrites its
// force.  Each particle owns its sides, so there are no atomics and the
// summation order is fixed: results are deterministic and, in the FP64 form,
// bit-identical to the sequential CPU order (this translation unit is built
// with -ffp-contract=off; FP64 sqrt and division are correctly rounded).
//
// The neighbour list and the link sides live in wave tiles: slot k of the 64
// particles of a tile is one contiguous run, so every list/CT access of a
// wavefront is a single coalesced 256 B / 512 B transaction.  Partner state
// (coordinates, Diff, radius) is gathered through L2; particles are stored in
// spatial (Morton) order, so partners of a tile mostly lie in its own or a
// neighbouring workgroup (which take the tiles in launch order or in a range
// per XCD: step_form).  A link's broken flag rides in the sign bit of its slot
// words (no per-link gather), and contact pairs beyond the attraction range are
// skipped when that provably leaves the force unchanged (pair_in_contact).
#include <cmath>
#include <type_traits>

#include "hdm_context.h"
#include "kernel_common.h"

namespace hdm {

namespace {

constexpr int TPB = 256;

template <class R>
struct ForceParams {
    R invDt, attractDistance, attractScaleForce, damping, dampingRotation, scaleE;
    R E, W2, W4, G;
    int32_t skipInert;  // contact constants small enough for pair_in_contact's argument
};

// The inert-contact skip relies on every term of the contact law staying
// finite in R for radius sums up to 1e6; these bounds on the law's constants
// guarantee it (Cnst <= sqrt(1e18) * 1e15 or 1e12 * 1e6 * 1e15 < FLT_MAX).
inline bool inert_skip_allowed(const hdm_force_params &f) {
    return std::fabs(f.attractDistance) <= 1e6 && std::fabs(f.attractScaleForce) <= 1e12 &&
           std::fabs(f.scaleE) <= 1e15;
}

template <class R>
ForceParams<R> cast_params(const hdm_force_params &f) {
    return ForceParams<R>{(R)f.invDt, (R)f.attractDistance, (R)f.attractScaleForce, (R)f.damping,
                          (R)f.dampingRotation, (R)f.scaleE, (R)f.E, (R)f.W2, (R)f.W4, (R)f.G,
                          inert_skip_allowed(f) ? 1 : 0};
}

// Diff differences of a pair, s - o: in the FP64 form exactly the law's own
// (self[c] - other[c]).  In the FP32 form the partner's Diff is the FP32 value
// its gather record carries, and the difference with the particle's own FP64
// Diff is formed in FP64 and rounded once: neighbouring Diffs are nearly
// equal, and rounding both to FP32 before subtracting would cancel most of the
// significant bits of their difference.
template <class R>
__device__ __forceinline__ void diff_delta(const double s[6], const double o[6], R d[6]) {
#pragma unroll
    for (int c = 0; c < 6; c++) d[c] = (R)(s[c] - (sizeof(R) == 4 ? (double)(float)o[c] : o[c]));
}

// HiDEMDefNeighForceFunc::operator() (HiDEMDefaultFunctions.h:38-86); the
// damping terms take the Diff differences d (diff_delta).  t: what the law adds
// to each force component.
template <class R>
__device__ __forceinline__ void contact_terms(R mask, R xDist, R yDist, R zDist, const R self[7], const R other[7],
                                              const R d[6], const ForceParams<R> &fp, R t[6]) {
    R xDist2 = xDist * xDist;
    R yDist2 = yDist * yDist;
    R zDist2 = zDist * zDist;
    R particleDistance2 = xDist2 + yDist2 + zDist2;
    R radSum = self[6] + other[6];
    R activeDist2 = (radSum + fp.attractDistance) * (radSum + fp.attractDistance);
    mask = (particleDistance2 >= activeDist2) ? R(0) : mask;
    R particleDistance = sqrt(particleDistance2);
    R invDist = R(1) / particleDistance;
    R xComp = xDist * invDist;
    R yComp = yDist * invDist;
    R zComp = zDist * invDist;
    R Cnst = 0;
    R dimDist = radSum - particleDistance;
    Cnst = (particleDistance < radSum) ? R(sqrt(dimDist * dimDist * dimDist)) : Cnst;
    Cnst = (particleDistance >= radSum && particleDistance < radSum + fp.attractDistance)
               ? fp.attractScaleForce * dimDist : Cnst;
    Cnst *= fp.scaleE;
    t[0] = mask * ((-fp.damping) * (d[0] * fp.invDt) + (Cnst * xComp));
    t[1] = mask * ((-fp.damping) * (d[1] * fp.invDt) + (Cnst * yComp));
    t[2] = mask * ((-fp.damping) * (d[2] * fp.invDt) + (Cnst * zComp));
    t[3] = mask * ((-fp.dampingRotation) * (d[3] * fp.invDt));
    t[4] = mask * ((-fp.dampingRotation) * (d[4] * fp.invDt));
    t[5] = mask * ((-fp.dampingRotation) * (d[5] * fp.invDt));
}

template <class R>
__device__ __forceinline__ void contact_law(R mask, R xDist, R yDist, R zDist, const R self[7], const R other[7],
                                            const R d[6], const ForceParams<R> &fp, R F[6]) {
    R t[6];
    contact_terms<R>(mask, xDist, yDist, zDist, self, other, d, fp, t);
#pragma unroll
    for (int c = 0; c < 6; c++) F[c] += t[c];
}

template <class R> __device__ __forceinline__ R huge_value();
template <> __device__ __forceinline__ double huge_value<double>() { return 1e300; }
template <> __device__ __forceinline__ float huge_value<float>() { return 1e37f; }

// HiDEMDefLinkForceFunc::operator() (HiDEMDefaultFunctions.h:105-203).  The
// FP64 form evaluates the reference expressions in their order.  The FP32
// form groups the same terms by pair differences, B0 - B6 = T0 . (s - o) etc.,
// with s - o = d from diff_delta, so the CT increments keep the relative
// motion of the two ends instead of the difference of two rounded values.
// add(c, j, v): the law adds v to force component c, its damping (j = 0)
// before its elastic term (j = 1).
template <class R, bool GROW = true, class Add>
__device__ __forceinline__ void beam_terms(R mask, R xDist, R yDist, R zDist, const R s[7], const R o[7],
                                           const R d[6], const ForceParams<R> &fp, R ct[6], Add add) {
    add(0, 0, (-fp.damping * (d[0] * fp.invDt)) * mask);
    add(1, 0, (-fp.damping * (d[1] * fp.invDt)) * mask);
    add(2, 0, (-fp.damping * (d[2] * fp.invDt)) * mask);
    add(3, 0, (-fp.dampingRotation * (d[3] * fp.invDt)) * mask);
    add(4, 0, (-fp.dampingRotation * (d[4] * fp.invDt)) * mask);
    add(5, 0, (-fp.dampingRotation * (d[5] * fp.invDt)) * mask);

    R xDist2 = xDist * xDist;
    R yDist2 = yDist * yDist;
    if (xDist == R(0) && yDist == R(0)) {
        xDist2 = R(1e-10);
        yDist2 = R(1e-10);
    }
    R zDist2 = zDist * zDist;
    R distSum = xDist2 + yDist2 + zDist2;
    R invLI = R(1) / sqrt(distSum);
    R invLP = R(1) / sqrt(xDist2 + yDist2);
    R invLILP = invLI * invLP;
    R LI = invLI * distSum;

    R T00 = xDist * invLI, T01 = yDist * invLI, T02 = zDist * invLI;
    R T10 = -yDist * invLP, T11 = xDist * invLP;
    R T20 = -(zDist * xDist) * invLILP;
    R T21 = -(zDist * yDist) * invLILP;
    R T22 = (xDist2 + yDist2) * invLILP;

    R L2 = LI * LI;
    R L3 = LI * LI * LI;
    R LIDiv6 = (R(1) / R(6)) * invLI;

    R K0 = fp.E * fp.W2 * invLI;
    R K1 = fp.E * fp.W4 / L3;
    R K5 = fp.E * fp.W4 / (R(2) * L2);
    R K2 = fp.G * fp.W4 * LIDiv6;
    R K3 = fp.E * fp.W4 * LIDiv6 * R(2);
    R K4 = fp.E * fp.W4 * LIDiv6;

    R B4 = T10 * s[3] + T11 * s[4];
    R B5 = T20 * s[3] + T21 * s[4] + T22 * s[5];
    R B10 = T10 * o[3] + T11 * o[4];
    R B11 = T20 * o[3] + T21 * o[4] + T22 * o[5];

    if constexpr (sizeof(R) == 8) {
        R B0 = T00 * s[0] + T01 * s[1] + T02 * s[2];
        R B1 = T10 * s[0] + T11 * s[1];
        R B2 = T20 * s[0] + T21 * s[1] + T22 * s[2];
        R B6 = T00 * o[0] + T01 * o[1] + T02 * o[2];
        R B7 = T10 * o[0] + T11 * o[1];
        R B8 = T20 * o[0] + T21 * o[1] + T22 * o[2];

        if constexpr (GROW) {
            ct[0] += K0 * B0 + (-K0) * B6;
            ct[1] += K1 * B1 + K5 * B5 + (-K1) * B7 + K5 * B11;
            ct[2] += K1 * B2 + (-K5) * B4 + (-K1) * B8 + (-K5) * B10;
        }

        add(0, 1, (-(T00 * ct[0] + T10 * ct[1] + T20 * ct[2])) * mask);
        add(1, 1, (-(T01 * ct[0] + T11 * ct[1] + T21 * ct[2])) * mask);
        add(2, 1, (-(T02 * ct[0] + T22 * ct[2])) * mask);

        R B3 = T00 * s[3] + T01 * s[4] + T02 * s[5];
        R B9 = T00 * o[3] + T01 * o[4] + T02 * o[5];

        if constexpr (GROW) {
            ct[3] += K2 * B3 + (-K2) * B9;
            ct[4] += (-K5) * B2 + K3 * B4 + K5 * B8 + K4 * B10;
            ct[5] += K5 * B1 + K3 * B5 + (-K5) * B7 + K4 * B11;
        }
    } else {
        R D0 = T00 * d[0] + T01 * d[1] + T02 * d[2];   // B0 - B6
        R D1 = T10 * d[0] + T11 * d[1];                 // B1 - B7
        R D2 = T20 * d[0] + T21 * d[1] + T22 * d[2];   // B2 - B8
        R D3 = T00 * d[3] + T01 * d[4] + T02 * d[5];   // B3 - B9

        if constexpr (GROW) {
            ct[0] += K0 * D0;
            ct[1] += K1 * D1 + K5 * (B5 + B11);
            ct[2] += K1 * D2 + (-K5) * (B4 + B10);
        }

        add(0, 1, (-(T00 * ct[0] + T10 * ct[1] + T20 * ct[2])) * mask);
        add(1, 1, (-(T01 * ct[0] + T11 * ct[1] + T21 * ct[2])) * mask);
        add(2, 1, (-(T02 * ct[0] + T22 * ct[2])) * mask);

        if constexpr (GROW) {
            ct[3] += K2 * D3;
            ct[4] += (-K5) * D2 + K3 * B4 + K4 * B10;
            ct[5] += K5 * D1 + K3 * B5 + K4 * B11;
        }
    }

    add(3, 1, (-(T00 * ct[3] + T10 * ct[4] + T20 * ct[5])) * mask);
    add(4, 1, (-(T01 * ct[3] + T11 * ct[4] + T21 * ct[5])) * mask);
    add(5, 1, (-(T02 * ct[3] + T22 * ct[5])) * mask);
}

template <class R, bool GROW = true>
__device__ __forceinline__ void beam_law(R mask, R xDist, R yDist, R zDist, const R s[7], const R o[7],
                                         const R d[6], const ForceParams<R> &fp, R ct[6], R F[6]) {
    beam_terms<R, GROW>(mask, xDist, yDist, zDist, s, o, d, fp, ct, [&](int c, int, R v) { F[c] += v; });
}

template <class R, class CT, class FO>
struct ForceArgs {
    using CTType = CT;
    const double *radius;
    int64_t n;
    const int32_t *nbrCount, *nbr;
    int32_t nbrWidth;
    const uint32_t *linkCount;
    const int32_t *slotLink, *slotOther;
    int32_t linkWidth;
    CT *ct;  // side store (ct_offset layout)
    FO *f0, *f1, *f2, *f3, *f4, *f5;
    ForceParams<R> fp;
    // Fused link break of the previous timestep (fused step only; breakCheck
    // = 0 elsewhere): before its beam law, every intact side evaluates
    // HiDEMDefLinkBreakFunc on the current state, exactly as k_break does
    // after the previous integration.
    int32_t breakCheck;
    // The neighbour list leaves out link partners (Context::nbrExcludesLinked,
    // FP32 only): the link loop applies the contact law of each side's pair,
    // before its beam law.
    int32_t linkedContacts;
    int32_t *slotLinkW, *slotOtherW;
    const double *tx, *ty, *tz, *initialLen, *maxLoad;
    uint8_t *state;
    double bendBreak, scalarMaxLoad;
    uint64_t *brokenCount;  // fused break: links broken are added here (nullptr: not counted)
};

// HiDEMDefLinkBreakFunc (HiDEMDefaultFunctions.h:217-241) for link l seen
// from one end: d = this end's coordinates minus the other's, t = this end's
// rotations, q = the other end.  Both ends compute the same bits: IEEE
// subtraction is antisymmetric (a - b == -(b - a)), so the squared distances
// and the absolute rotation differences do not depend on which end asks.
template <class R, class CT, class FO>
__device__ __forceinline__ bool link_breaks(const ForceArgs<R, CT, FO> &a, int32_t l, int32_t q, double xDist,
                                            double yDist, double zDist, const double t[3]) {
    double stretchLength = sqrt((xDist * xDist) + (yDist * yDist) + (zDist * zDist));
    double bx = fabs(t[0] - a.tx[q]);
    double by = fabs(t[1] - a.ty[q]);
    double bz = fabs(t[2] - a.tz[q]);
    double inner = (by < bz) ? bz : by;
    double maxBend = (bx < inner) ? inner : bx;
    double initialLen = a.initialLen[l];
    double load = (stretchLength - initialLen) / initialLen + a.bendBreak * maxBend;
    double maxLoad = a.maxLoad ? a.maxLoad[l] : a.scalarMaxLoad;
    return load >= maxLoad;
}

template <class R, class CT, class FO>
__device__ __forceinline__ void store_force(const ForceArgs<R, CT, FO> &a, int64_t p, const R F[6]) {
    a.f0[p] = (FO)F[0];
    a.f1[p] = (FO)F[1];
    a.f2[p] = (FO)F[2];
    a.f3[p] = (FO)F[3];
    a.f4[p] = (FO)F[4];
    a.f5[p] = (FO)F[5];
}

// ---- time integration --------------------------------------------------------
// Particle state read by the integrator (in) and written by it (out).  The
// standalone integrator updates in place (out == in); the fused step kernel
// writes the other buffer of a ping-pong pair, because other lanes of the same
// launch still gather the old state for their forces.
struct IntegArgs {
    const double *x, *y, *z, *tx, *ty, *tz, *d0, *d1, *d2, *d3, *d4, *d5;
    double *ox, *oy, *oz, *otx, *oty, *otz, *od0, *od1, *od2, *od3, *od4, *od5;
    const double *radius;
    const uint8_t *type;
    int64_t n;
    hdm_integ_params ip;
    // rebuild-test reductions of the new state (nullptr: none): one row of 3
    // doubles per workgroup, max(0, max Diff) per axis (HiDEMLib.h:424-461),
    // folded by k_skin_finalize
    double *partials;
    // exact-test guard (nullptr: off; see StepGuard): a launch that finds
    // *guard (the trip word of its input records) set does nothing but set
    // *guardOut; otherwise a particle whose new position trips the exact test
    // sets *guardOut, and workgroup 0 counts the executed launch in
    // *stepsDone.
    const uint32_t *guard;
    uint32_t *guardOut, *stepsDone;
    double guardThr;
    const double *x0, *y0, *z0;   // the rebuild snapshot
    const float *x0f, *y0f, *z0f; // the snapshot rounded to FP32 (guard_trips)
    const int32_t *blockId;       // batched form: waterline of the particle's block
    const double *blockWater;     // (nullptr: ip.waterLevel for every particle)
    const MapDev *maps;           // GlacierDem map inputs, slot k valid when bit k of mapMask
    int32_t mapMask;
};

// Damped central difference (HiDEMDefTimeIntegration, HiDEMDefaultFunctions.h
// :317-370; same expressions as the inline IceBlock form).
__device__ __forceinline__ void central_difference(double dragCoeff, double mass, double inertia,
                                                   const hdm_integ_params &ip, const double F[6],
                                                   const double diff[6], double cord[3], double cordPrev[3],
                                                   double theta[3], double thetaPrev[3], double vel[6]) {
    double dragInvDt2 = dragCoeff * ip.invDt2;
    double massDtSqr = mass * ip.invDtSqr;
    double pMassDtSqr = mass / ip.dtSqr;
    double pMemDtSqr = inertia / ip.dtSqr;
    double invC1 = 1.0 / (pMassDtSqr + dragCoeff * ip.invDt2);
    double invC2 = 1.0 / (pMemDtSqr + dragCoeff * ip.invDt2);
    double interDtSqr = inertia * ip.invDtSqr;
    double next[6];
#pragma unroll
    for (int c = 0; c < 3; c++) next[c] = (F[c] + massDtSqr * diff[c] + dragInvDt2 * -diff[c]) * invC1;
#pragma unroll
    for (int c = 3; c < 6; c++) next[c] = (F[c] + interDtSqr * diff[c] + dragInvDt2 * -diff[c]) * invC2;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        cordPrev[c] = cord[c];
        thetaPrev[c] = theta[c];
        cord[c] = cord[c] + next[c];
        theta[c] = theta[c] + next[3 + c];
        vel[c] = next[c] * ip.invDt;
        vel[3 + c] = (theta[c] - thetaPrev[c]) * ip.invDt;
    }
}

// Map2d::getIndexes (Map2d.h:92-108) for one axis: floor of the scaled
// coordinate, held within [-1, n] before the int conversion (so NaN and huge
// coordinates stay defined; the clamp to [0, n - 1] below treats them as the
// reference does any value beyond the grid).
__device__ __forceinline__ int32_t map_floor(float f, int32_t n) {
    f = floorf(f);
    if (!(f >= -1.0f)) f = -1.0f;
    if (f > (float)n) f = (float)n;
    return (int32_t)f;
}

__device__ __forceinline__ int32_t map_clamp(int32_t v, int32_t lo, int32_t hi) {
    return v < lo ? lo : (v > hi ? hi : v);
}

// Map2d::interp (Map2d.h:110-145): FP32 bilinear interpolation in the
// reference's expression order; the grid value itself where both axes clamp
// to one point.
__device__ double map_interp(const MapDev &m, float x, float y) {
    x += m.xOffset;
    y += m.yOffset;
    const int32_t xPoint = map_floor(((x - m.xMin) * m.invXMaxMin) * (float)(m.xPoints - 1), m.xPoints);
    const int32_t yPoint = map_floor(((y - m.yMin) * m.invYMaxMin) * (float)(m.yPoints - 1), m.yPoints);
    const int32_t xLow = map_clamp(xPoint, 0, m.xPoints - 1), yLow = map_clamp(yPoint, 0, m.yPoints - 1);
    const int32_t xHigh = map_clamp(xPoint + 1, 0, m.xPoints - 1), yHigh = map_clamp(yPoint + 1, 0, m.yPoints - 1);
    if (xLow == xHigh && yLow == yHigh) return m.data[xLow + yLow * m.xPoints];
    const float v00 = (float)m.data[xLow + yLow * m.xPoints];
    const float v01 = (float)m.data[xLow + yHigh * m.xPoints];
    const float v10 = (float)m.data[xHigh + yLow * m.xPoints];
    const float v11 = (float)m.data[xHigh + yHigh * m.xPoints];
    const float x0 = x - m.xMin;
    const float y0 = y - m.yMin;
    const float x1 = (float)xLow * m.xRes;
    const float x2 = (float)xHigh * m.xRes;
    const float y1 = (float)yLow * m.yRes;
    const float y2 = (float)yHigh * m.yRes;
    const float invX21 = 1.0f / (x2 - x1);
    const float c1 = (x2 - x0) * invX21;
    const float c2 = (x0 - x1) * invX21;
    float fxy1 = (c1 * v00) + (c2 * v10);
    float fxy2 = (c1 * v01) + (c2 * v11);
    if (xLow == xHigh) {
        fxy1 = v00;
        fxy2 = v01;
    } else if (yLow == yHigh) {
        return fxy1;
    }
    const float invY21 = 1.0f / (y2 - y1);
    return (((y2 - y0) * invY21) * fxy1) + (((y0 - y1) * invY21) * fxy2);
}

// applyForce: IceBlock (MainIceBlock.cpp:299-400, clamp = HDM_TYPE_FIXED) or
// GlacierDem (MainDem.cpp:145-259: bed height, friction and external force
// from maps (bit k of mapMask: maps[k]) or the analytic bed and constant
// force of ip, HiDEMDefVelocityLimit and HiDEMDefBoundaryCondition), on one
// particle's state in registers: cord/theta/diff are replaced by the new
// coordinates, rotations and Diff.
__device__ __forceinline__ void integrate_state(const hdm_integ_params &ip, const MapDev *maps, int32_t mapMask,
                                                bool fixed, double radius, double waterLevel, const double Fin[6],
                                                double cord[3], double theta[3], double diff[6]) {
    if (ip.variant == HDM_INTEG_ICEBLOCK && fixed) {
#pragma unroll
        for (int c = 0; c < 6; c++) diff[c] = 0;
        return;
    }
    double F[6] = {Fin[0], Fin[1], Fin[2], Fin[3], Fin[4], Fin[5]};
    double cordPrev[3], thetaPrev[3], vel[6];
    const double diameter = radius * 2.0;
    const double zCord = cord[2];
    const double particleMass = ip.rhoIce * diameter * diameter * diameter;
    const double particleMomentInertia = particleMass * diameter * diameter / 6.0;
    double dragCoeff;
    if (ip.variant == HDM_INTEG_ICEBLOCK) {
        dragCoeff = (zCord > waterLevel) ? ip.airDrag : ip.waterDrag;
        if (zCord > waterLevel) F[2] += -ip.g * particleMass;
        if (zCord <= waterLevel) F[2] += ip.lift * particleMass;
        central_difference(dragCoeff, particleMass, particleMomentInertia, ip, F, diff, cord, cordPrev, theta,
                           thetaPrev, vel);
    } else {
        // InputBed::getHeight / getFric (InputGeometry.h:57-67): the
        // coordinates go to Map2d::interp as float
        const float fx = (float)cord[0], fy = (float)cord[1];
        const double bedzCord = (mapMask & (1 << HDM_MAP_BED)) ? map_interp(maps[HDM_MAP_BED], fx, fy)
                                                               : ((cord[0] < ip.bedXEnd) ? ip.bedZ : ip.deepZ);
        const double fric = (mapMask & (1 << HDM_MAP_FRICTION)) ? map_interp(maps[HDM_MAP_FRICTION], fx, fy)
                                                                : ((cord[0] < ip.frictionXEnd) ? 1.0 : 0.0);
        if ((zCord + radius) - bedzCord < ip.bedInteract) {
            double d = ip.bedDrag * fric;
            dragCoeff = (ip.frictionCap < d) ? ip.frictionCap : d;
        } else if (zCord > waterLevel) {
            dragCoeff = ip.airDrag;
        } else {
            dragCoeff = ip.waterDrag;
        }
        if (zCord > waterLevel) F[2] += -ip.g * particleMass;
        if (zCord <= waterLevel) F[2] += ip.lift * particleMass;
        if (zCord + radius < bedzCord) F[2] += ip.bedStiffness * (bedzCord - (zCord + radius));
        if (mapMask >> HDM_MAP_EXT) {
            for (int c = 0; c < 6; c++)
                F[c] += (mapMask & (1 << (HDM_MAP_EXT + c))) ? map_interp(maps[HDM_MAP_EXT + c], fx, fy) : ip.ext[c];
        } else {
#pragma unroll
            for (int c = 0; c < 6; c++) F[c] += ip.ext[c];
        }
        central_difference(dragCoeff, particleMass, particleMomentInertia, ip, F, diff, cord, cordPrev, theta,
                           thetaPrev, vel);
        if (ip.velocityLimit) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (vel[c] > ip.maxVel) cord[c] = ip.dt * ip.maxVel + cordPrev[c];
                if (vel[3 + c] > ip.maxRot) theta[c] = ip.dt * ip.maxRot + thetaPrev[c];
            }
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (vel[c] < -ip.maxVel) cord[c] = ip.dt * -ip.maxVel + cordPrev[c];
                if (vel[3 + c] < -ip.maxRot) theta[c] = ip.dt * -ip.maxRot + thetaPrev[c];
            }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            if (cord[c] + radius < ip.lower[c] && ip.bound[2 * c]) cord[c] = cordPrev[c];
            if (cord[c] - radius > ip.upper[c] && ip.bound[2 * c + 1]) cord[c] = cordPrev[c];
        }
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
        diff[c] = cord[c] - cordPrev[c];
        diff[3 + c] = theta[c] - thetaPrev[c];
    }
}

// Integrates particle i under force Fin from the IntegArgs state arrays;
// returns its new state.
__device__ __forceinline__ void integrate_particle(const IntegArgs &a, int64_t i, const double Fin[6],
                                                   double cord[3], double theta[3], double diff[6],
                                                   double &radius) {
    const double *cordIn[3] = {a.x, a.y, a.z}, *thetaIn[3] = {a.tx, a.ty, a.tz};
    const double *diffIn[6] = {a.d0, a.d1, a.d2, a.d3, a.d4, a.d5};
#pragma unroll
    for (int c = 0; c < 3; c++) {
        cord[c] = cordIn[c][i];
        theta[c] = thetaIn[c][i];
    }
#pragma unroll
    for (int c = 0; c < 6; c++) diff[c] = diffIn[c][i];
    radius = a.radius[i];
    const bool fixed = (a.type[i] & HDM_TYPE_FIXED) != 0;
    const double waterLevel = a.blockWater ? a.blockWater[a.blockId[i]] : a.ip.waterLevel;
    integrate_state(a.ip, a.maps, a.mapMask, fixed, radius, waterLevel, Fin, cord, theta, diff);
    a.ox[i] = cord[0];
    a.oy[i] = cord[1];
    a.oz[i] = cord[2];
    a.otx[i] = theta[0];
    a.oty[i] = theta[1];
    a.otz[i] = theta[2];
    a.od0[i] = diff[0];
    a.od1[i] = diff[1];
    a.od2[i] = diff[2];
    a.od3[i] = diff[3];
    a.od4[i] = diff[4];
    a.od5[i] = diff[5];
}

// Largest positive Diff per axis of the particles this workgroup integrated
// (HiDEMLib.h:424-461; from 0, to which inactive lanes contribute), written as
// one row of a.partials; the rows are folded by k_skin_finalize after the
// launch.
template <int BLOCK>
__device__ __forceinline__ void skin_partials(const IntegArgs &a, bool active, const double diff[3]) {
    __shared__ double rows[BLOCK / 64][3];
    double m[3];
#pragma unroll
    for (int c = 0; c < 3; c++) m[c] = wave_max(active && diff[c] > 0.0 ? diff[c] : 0.0);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int c = 0; c < 3; c++) rows[w][c] = m[c];
    __syncthreads();
    if (threadIdx.x < 3) {
        double v = rows[0][threadIdx.x];
        for (int k = 1; k < BLOCK / 64; k++) v = rows[k][threadIdx.x] > v ? rows[k][threadIdx.x] : v;
        a.partials[(int64_t)blockIdx.x * 3 + threadIdx.x] = v;
    }
}

struct FinalizeArgs {
    const double *partials;
    int64_t rows;
    double *stage;        // [gridDim.x][3]
    uint32_t *ticket;
    uint64_t *skin;
};

// Largest value per axis over a workgroup's threads, left in m of thread 0.
__device__ __forceinline__ void block_max3(double m[3]) {
    __shared__ double part[TPB / 64][3];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 3; c++) m[c] = wave_max(m[c]);
    if ((threadIdx.x & 63) == 0)
        for (int c = 0; c < 3; c++) part[threadIdx.x >> 6][c] = m[c];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 1; k < TPB / 64; k++)
            for (int c = 0; c < 3; c++) m[c] = part[k][c] > m[c] ? part[k][c] : m[c];
}

// Folds the rows of the integrating launch: each workgroup reduces a slice
// into stage, and the last one (a ticket after a release fence: one fence
// per workgroup of this small launch) stores skin[0..2] as ordered keys for
// the host-checked rebuild policy.  Its workgroup reads the stage at once (a
// single thread reading one value after the other took most of the 11 us).
__global__ void __launch_bounds__(TPB) k_skin_finalize(FinalizeArgs a) {
    __shared__ int last;
    double m[3] = {0.0, 0.0, 0.0};
    for (int64_t r = (int64_t)blockIdx.x * TPB + threadIdx.x; r < a.rows; r += (int64_t)gridDim.x * TPB)
        for (int c = 0; c < 3; c++) {
            const double v = a.partials[r * 3 + c];
            m[c] = v > m[c] ? v : m[c];
        }
    block_max3(m);
    if (threadIdx.x == 0) {
        for (int c = 0; c < 3; c++) a.stage[blockIdx.x * 3 + c] = m[c];
        __threadfence();
        last = atomicAdd(a.ticket, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    const unsigned long long *st = reinterpret_cast<const unsigned long long *>(a.stage);
    for (int c = 0; c < 3; c++) m[c] = 0.0;
    for (uint32_t b = threadIdx.x; b < gridDim.x; b += TPB)
        for (int c = 0; c < 3; c++) {
            const double v = __longlong_as_double(
                (long long)__hip_atomic_load(st + b * 3 + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            m[c] = v > m[c] ? v : m[c];
        }
    block_max3(m);
    if (threadIdx.x != 0) return;
    for (int c = 0; c < 3; c++) a.skin[c] = ordered_key(m[c]);
    *a.ticket = 0;
}

// ---- fused step ------------------------------------------------------------------
// Gather records: MixedRec (kernel_common.h) in the FP32 form; the FP64 form
// gathers rec = double4 {x, y, z, radius} and the FP64 Diff from drec.
template <class R> struct RecOf { using type = double4; };
template <> struct RecOf<float> { using type = MixedRec; };
__device__ __forceinline__ double rec_radius(const double4 &P) { return P.w; }
__device__ __forceinline__ float rec_radius(const MixedRec &P) { return P.radius; }

// Gather records (see Context::rec / drec) and the break prefilter inputs.
template <class R>
struct StepRecs {
    using Real = R;
    using Rec = typename RecOf<R>::type;
    const Rec *rec;            // current state
    const double *drec;        // FP64 form: every particle's FP64 Diff; FP32 form: the escapes
    const MixedTail *tail;     // FP32 form: rest of the own Diff (split_diff3)
    Rec *recOut;               // integrated state
    double *drecOut;
    MixedTail *tailOut;
    double tame;               // Diff bound behind the radius flag of rec
    // Break prefilter inputs: per side a 16-bit code, code * thrScale at most
    // L0 (1 + maxLoad) with per-link maxLoad (perLinkMaxLoad) else L0, 0 when
    // L0 < 1e-30 or not finite; the largest L0 of the state (rounded up)
    const uint16_t *slotThr;
    float thrScale;
    int32_t prefilter;         // 0: every intact side takes the exact break test
    int32_t perLinkMaxLoad;
    float scalarMaxLoad, bendBreak, l0Max;
    int32_t storeForce;        // write x..wForce (the last step of a run; earlier ones are overwritten unseen)
};

// Upper bound of max |theta_p - theta_q| over components, as a float: the sum
// of absolute values, NaN/inf when any component is (then the prefilter
// defers to the exact test).
__device__ __forceinline__ float rotation_bound(const double t[3]) {
    return (float)(fabs(t[0]) + fabs(t[1]) + fabs(t[2]));
}

// Doubles per particle in drec: the FP64 form's partners gather it (Diff0..5,
// rotation bound, 0); in the FP32 form it is the escape array of
// split_diff3 (Diff0..2, written and read only for particles whose
// translation Diff does not split exactly), the rest travelling in the
// MixedRec and the MixedTail.
inline int64_t drec_stride(int32_t prec) { return prec == HDM_PREC_FP64 ? 8 : 3; }

__device__ __forceinline__ void load_drec(const double *drec, int64_t q, double o[6], float &rot) {
    const double4 *v = reinterpret_cast<const double4 *>(drec + q * 8);
    const double4 a = v[0], b = v[1];
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y;
    rot = (float)b.z;
}

template <class R>
__device__ __forceinline__ void store_records(const StepRecs<R> &r, int64_t p, const double cord[3],
                                              const double theta[3], const double diff[6], double radius) {
    bool tame = fabs(radius) <= 5e5;
#pragma unroll
    for (int c = 0; c < 6; c++) tame &= fabs(diff[c]) <= r.tame;
    if constexpr (sizeof(R) == 4) {
        MixedRec m;
        m.x = cord[0];
        m.y = cord[1];
        m.z = cord[2];
        float lo[3];
        const bool exact = split_diff3(diff, m.d, lo);
#pragma unroll
        for (int c = 3; c < 6; c++) m.d[c] = (float)diff[c];
        m.rot = rotation_bound(theta);
        m.radius = tame ? (float)radius : __builtin_nanf("");
        m.lo[0] = lo[0];
        m.lo[1] = lo[1];
        r.recOut[p] = m;
        MixedTail t;
#pragma unroll
        for (int c = 0; c < 3; c++) t.dr[c] = diff[3 + c];
        t.lo2 = lo[2];
        t.pad = 0.0f;
        r.tailOut[p] = t;
        if (!exact) {
#pragma unroll
            for (int c = 0; c < 3; c++) r.drecOut[p * 3 + c] = diff[c];
        }
    } else {
        r.recOut[p] = make_double4(cord[0], cord[1], cord[2], tame ? radius : __builtin_nan(""));
        double4 *d = reinterpret_cast<double4 *>(r.drecOut + p * 8);
        d[0] = make_double4(diff[0], diff[1], diff[2], diff[3]);
        d[1] = make_double4(diff[4], diff[5], (double)rotation_bound(theta), 0.0);
    }
}

// A partner's Diff (as the laws take it) and the pair differences, from its
// gathered record: FP32 from the record itself, FP64 from drec.
template <class R>
__device__ __forceinline__ void partner_diff(const StepRecs<R> &r, int32_t q, const typename RecOf<R>::type &Q,
                                             const double diff[6], R other[6], R d[6], float &rot) {
    if constexpr (sizeof(R) == 4) {
#pragma unroll
        for (int c = 0; c < 6; c++) {
            other[c] = Q.d[c];
            d[c] = (R)(diff[c] - (double)Q.d[c]);
        }
        rot = Q.rot;
    } else {
        double od[6];
        load_drec(r.drec, q, od, rot);
#pragma unroll
        for (int c = 0; c < 6; c++) other[c] = (R)od[c];
        diff_delta<R>(diff, od, d);
    }
}

// Records of the particles of one workgroup in LDS, 16 B chunks by [chunk][particle]
// (a lane's chunk reads fall on random 16 B slots of the banks, where the
// records' own stride would leave them on a quarter of the slots).
template <class R, int BLOCK>
struct BlockRecs {
    static constexpr int REC = (int)sizeof(typename RecOf<R>::type) / 16;   // chunks of rec
    static constexpr int CHUNKS = sizeof(R) == 8 ? REC + 4 : REC;           // and of drec (FP64 form)
    // four more columns: 16 lanes that write the four chunks of four particles hit 16 different bank slots
    double2 c[CHUNKS][BLOCK + 4];
    double2 out[BLOCK / 64][32 * 5];   // half a wave's new records on their way to contiguous stores
};

typedef double d2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double2 lds_load(const double2 *p) {
    const d2v v = *(const __attribute__((address_space(3))) d2v *)p;
    return make_double2(v.x, v.y);
}

// A partner's record fields (first `chunks` chunks) from the workgroup's LDS
// copy when it is one of the workgroup's own particles, else from memory.
template <class R, int BLOCK, int CHUNKS>
__device__ __forceinline__ void load_partner(const StepRecs<R> &r, const BlockRecs<R, BLOCK> &own, int32_t p0,
                                             int32_t q, double2 (&c)[CHUNKS]) {
    constexpr int REC = BlockRecs<R, BLOCK>::REC;
    const uint32_t at = (uint32_t)(q - p0);
    if (at < (uint32_t)BLOCK) {
        // as LDS loads: merged with the other branch's they would be flat ones
#pragma unroll
        for (int j = 0; j < CHUNKS; j++) c[j] = lds_load(&own.c[j][at]);
    } else {
        const double2 *a = reinterpret_cast<const double2 *>(r.rec + q);
#pragma unroll
        for (int j = 0; j < (CHUNKS < REC ? CHUNKS : REC); j++) c[j] = a[j];
        if constexpr (CHUNKS > REC) {
            const double2 *b = reinterpret_cast<const double2 *>(r.drec + (int64_t)q * 8);
#pragma unroll
            for (int j = 0; j < CHUNKS - REC; j++) c[REC + j] = b[j];
        }
    }
}

// The fields of a loaded record: coordinates and radius flag (contact test),
// then Diff as the laws take it, the pair differences and the rotation bound.
__device__ __forceinline__ float low_float(double v) { return __uint_as_float((uint32_t)__double_as_longlong(v)); }
__device__ __forceinline__ float high_float(double v) {
    return __uint_as_float((uint32_t)((uint64_t)__double_as_longlong(v) >> 32));
}
__device__ __forceinline__ float chunk_radius(const double2 &c1, float) { return low_float(c1.y); }
__device__ __forceinline__ double chunk_radius(const double2 &c1, double) { return c1.y; }

template <class R, int CHUNKS>
__device__ __forceinline__ void chunk_diff(const double2 (&c)[CHUNKS], const double diff[6], R other[6], R d[6],
                                           float &rot) {
    if constexpr (sizeof(R) == 4) {
        const float o[6] = {low_float(c[2].x), high_float(c[2].x), low_float(c[2].y),
                            high_float(c[2].y), low_float(c[3].x), high_float(c[3].x)};
#pragma unroll
        for (int k = 0; k < 6; k++) {
            other[k] = o[k];
            d[k] = (R)(diff[k] - (double)o[k]);
        }
        rot = high_float(c[1].y);
    } else {
        const double od[6] = {c[2].x, c[2].y, c[3].x, c[3].y, c[4].x, c[4].y};
#pragma unroll
        for (int k = 0; k < 6; k++) other[k] = (R)od[k];
        diff_delta<R>(diff, od, d);
        rot = (float)c[5].x;
    }
}

// Break prefilter: true when the link certainly stays intact.  The exact test
// (s - L0) / L0 + bendBreak * maxBend >= maxLoad, with L0 > 0, is
// s + bendBreak * maxBend * L0 >= L0 (1 + maxLoad) =: T.  In float, with the
// rotation bound (at least maxBend) and the largest L0 standing in for the
// link's own, the left side can only grow, and T comes from a 16-bit code
// that rounds it down (k_side_codes); the link passes when that estimate is
// below T by more than 1e-5 of the magnitudes.  Float rounding of the inputs
// and operations is below 1e-6 of those magnitudes and bendBreak >= 0 (the
// host disables the prefilter otherwise), so a link the exact FP64 test would
// break never passes.  NaN/inf inputs and code 0 (L0 < 1e-30) fail the
// comparison and go to the exact test.
__device__ __forceinline__ bool certainly_intact(float T, float bendBreak, float l0Max, double dx, double dy,
                                                 double dz, float rotBound) {
    const float fx = (float)dx, fy = (float)dy, fz = (float)dz;
    const float s = __builtin_amdgcn_sqrtf(fx * fx + fy * fy + fz * fz);
    const float lhs = s + bendBreak * rotBound * l0Max;
    const float margin = 1e-5f * (lhs + fabsf(T));
    return lhs + margin < T;
}

// Streaming accesses of the fused step: every CT value, slot word, list entry
// and per-particle SoA field is touched once per launch, so it is loaded and
// stored non-temporally and leaves L2 to the gathered partner records, which
// each particle's neighbours fetch again.
template <class T>
__device__ __forceinline__ T ld_stream(const T *p) {
    return __builtin_nontemporal_load(p);
}
template <class T>
__device__ __forceinline__ void st_stream(T *p, T v) {
    __builtin_nontemporal_store(v, p);
}
__device__ __forceinline__ float2 ld_stream(const float2 *p) {
    const unsigned long long u = __builtin_nontemporal_load(reinterpret_cast<const unsigned long long *>(p));
    float2 r;
    __builtin_memcpy(&r, &u, sizeof(r));
    return r;
}

// Contacts of the linked pairs flagged in `sides` (bit k: side k's pair is
// not provably inert), after every beam, in side order: outside the link
// loop, so that loop does not carry the contact law's registers.
template <class R, class CT>
__device__ __forceinline__ void contact_sides(const ForceArgs<R, CT, R> &f, const StepRecs<R> &r,
                                                        uint64_t sides, int64_t base, int64_t p, double xCord,
                                              double yCord, double zCord, const double diff[6], R self[7], R F[6]) {
    self[6] = (R)f.radius[p];
    while (sides) {
        const int k = __builtin_ctzll(sides);
        sides &= sides - 1;
        const int32_t q = f.slotOther[base + (int64_t)k * 64] & SLOT_LINK_MASK;
        const auto Q = r.rec[q];
        R other[7], d[6];
        float rot;
        partner_diff<R>(r, q, Q, diff, other, d, rot);
        other[6] = (R)f.radius[q];
        contact_law<R>(R(1), (R)(xCord - Q.x), (R)(yCord - Q.y), (R)(zCord - Q.z), self, other, d, f.fp, F);
    }
}

// One timestep of hdm_run in one launch: the link break of the previous
// timestep (when f.breakCheck), force on particle p from the current state
// (CombinedAccel::iterateCombined, as k_force), then its integration (as
// k_integrate), with the rebuild-test partials.
//
// The records are the state: a particle's coordinates and Diff are read from
// its own records (the lines its neighbours gather) and the integrated ones
// are written to the other record buffers only; the SoA coordinates and Diff
// are unpacked from the records when something else needs them (sync_state).
// The rotations stay SoA (ping-pong), read at integration and by the rare
// exact break test; the prefilter takes their bound from the records.
//
// Partner state comes from the records too.  FP64 form: 32 B of rec decide a
// contact pair that is provably inert (pair_in_contact: beyond radSum +
// attractDistance with every Diff bounded by tame, so every term the law adds
// is +-0); only other pairs, and link partners, take drec.  FP32 form: one
// 64 B MixedRec per partner.  Particles lie along a space-filling curve, so
// about three quarters of a particle's partners belong to its own workgroup of
// 256: those come from a copy of the workgroup's records in LDS (BlockRecs),
// the others from memory.  With every partner gathered through L1 (a 16 B load
// touches a cache line per lane) the address and data units of L1 were busy
// 83-100% of the time.  The walk holds no exact break test (walk_sides), and
// the new records leave through LDS as contiguous stores, which together
// bring the registers to 128 (FP64, four waves per SIMD) and 94 (FP32, five).
// 8M-particle slab, before and now: FP64 3.11 -> 2.42 ms, 5.4 TB/s of HBM
// traffic; FP32 1.71 -> 1.40 ms, 5.9 TB/s; a copy reaches 6.2 TB/s.
// Leaving out a quarter of the FP32 form's arithmetic changes nothing, so
// what bounds both is HBM.
//
// The break test of an intact side runs exactly (FP64, as k_break) unless the
// float prefilter proves the link stays intact.
// BLOCK (workgroup size), XCD (the per-XCD contiguous renumbering of
// workgroups) and OCC (one more wave per SIMD than the register count allows,
// bought with a few spills) are the autotuned launch shape; every shape
// computes the same per-particle arithmetic, so results do not depend on it.
template <class R>
constexpr int step_waves(bool occ) {
    return sizeof(R) == 4 ? (occ ? 5 : 4) : (occ ? 4 : 3);
}

// The device guard's test for particle p at its new position c: the exact
// test 2 |c - x0| >= guardThr in FP64, decided first from the snapshot
// rounded to FP32 (12 B instead of 24 B read per particle).  Rounding to
// nearest moves a component by less than 2^-23 of its FP32 value (and by
// less than 1e-30 below the normal range), so the FP64 distance lies within
// e = (|x0f| + |y0f| + |z0f|) 2^-23 + 1e-30 of the distance d to the FP32
// snapshot.  With a margin of 1e-12 (d + e) for the rounding of both
// evaluations, d outside [thr/2 - e, thr/2 + e] decides the test as the FP64
// evaluation would; only the rest (and non-finite values, which fail both
// comparisons) read the FP64 snapshot.
__device__ __forceinline__ bool guard_trips(const IntegArgs &g, int64_t p, const double c[3], float fx, float fy,
                                            float fz) {
    const double ax = c[0] - (double)fx, ay = c[1] - (double)fy, az = c[2] - (double)fz;
    const double d = sqrt(ax * ax + ay * ay + az * az);
    const double e = (fabs((double)fx) + fabs((double)fy) + fabs((double)fz)) * 0x1p-23 + 1e-30;
    const double m = (d + e) * 1e-12;
    if (2.0 * (d + e + m) < g.guardThr) return false;
    if (d - e - m > 0.0 && 2.0 * (d - e - m) >= g.guardThr) return true;
    const double ddx = c[0] - g.x0[p], ddy = c[1] - g.y0[p], ddz = c[2] - g.z0[p];
    return 2.0 * sqrt(ddx * ddx + ddy * ddy + ddz * ddz) >= g.guardThr;
}

__device__ __forceinline__ bool guard_trips(const IntegArgs &g, int64_t p, const double c[3]) {
    return guard_trips(g, p, c, ld_stream(g.x0f + p), ld_stream(g.y0f + p), ld_stream(g.z0f + p));
}

// LDS written by some lanes of the wave, read by others of it.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// C chunks of each of the wave's 64 particles, contiguous in memory at src,
// into rows row.. of the workgroup's copy: every load moves 1 KB of the wave's
// contiguous run (a lane reading its own particle's chunks would touch a line
// per one or two lanes).  left: particles from the wave's first one on.
template <int C, int PITCH>
__device__ __forceinline__ void stage_chunks(const double2 *src, double2 (*rows)[PITCH], int col0, int64_t left) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < C; i++) {
        const int u = i * 64 + lane, pl = u / C;
        if (pl < left) rows[u % C][col0 + pl] = src[u];
    }
}

// The wave's particles into the workgroup's LDS copy (wave0: its first one).
template <class R, int BLOCK>
__device__ __forceinline__ void stage_records(const StepRecs<R> &r, int64_t wave0, int64_t n,
                                              BlockRecs<R, BLOCK> &own) {
    constexpr int REC = BlockRecs<R, BLOCK>::REC;
    const int col0 = threadIdx.x & ~63;
    stage_chunks<REC>(reinterpret_cast<const double2 *>(r.rec + wave0), own.c, col0, n - wave0);
    if constexpr (sizeof(R) == 8)
        stage_chunks<4>(reinterpret_cast<const double2 *>(r.drec + wave0 * 8), own.c + REC, col0, n - wave0);
}

// C chunks per lane (v) to the wave's contiguous run at dst, through LDS: a
// lane storing its own chunks would write 16 B of 64 different lines.  Half
// the wave at a time (the stage then leaves room for the resident workgroups
// the registers allow), C + 1 chunks per particle, which keeps writes and
// reads off shared bank slots.  Every lane of the wave takes part.
template <int C>
__device__ __forceinline__ void store_chunks(double2 *dst, const double2 (&v)[C], double2 *stage, int lane) {
    constexpr int P = C + 1;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        if ((lane >> 5) == half) {
#pragma unroll
            for (int j = 0; j < C; j++) stage[(lane & 31) * P + j] = v[j];
        }
        wave_lds_fence();
#pragma unroll
        for (int i = 0; i < C / 2; i++) {
            const int u = i * 64 + lane;
            dst[half * 32 * C + u] = stage[u / C * P + u % C];
        }
        wave_lds_fence();
    }
}

// store_records for a whole wave, with contiguous stores.
template <class R>
__device__ __forceinline__ void store_records_wave(const StepRecs<R> &r, int64_t wave0, int lane, const double cord[3],
                                                   const double theta[3], const double diff[6], double radius,
                                                   double2 *stage) {
    bool tame = fabs(radius) <= 5e5;
#pragma unroll
    for (int c = 0; c < 6; c++) tame &= fabs(diff[c]) <= r.tame;
    if constexpr (sizeof(R) == 4) {
        float hi[3], lo[3];
        const bool exact = split_diff3(diff, hi, lo);
        const float2 rr = make_float2(tame ? (float)radius : __builtin_nanf(""), rotation_bound(theta));
        const float4 a = make_float4(hi[0], hi[1], hi[2], (float)diff[3]);
        const float4 b = make_float4((float)diff[4], (float)diff[5], lo[0], lo[1]);
        const double2 v[4] = {make_double2(cord[0], cord[1]), make_double2(cord[2], __builtin_bit_cast(double, rr)),
                              __builtin_bit_cast(double2, a), __builtin_bit_cast(double2, b)};
        store_chunks(reinterpret_cast<double2 *>(r.recOut + wave0), v, stage, lane);
        const float2 l2 = make_float2(lo[2], 0.0f);
        const double2 t[2] = {make_double2(diff[3], diff[4]), make_double2(diff[5], __builtin_bit_cast(double, l2))};
        store_chunks(reinterpret_cast<double2 *>(r.tailOut + wave0), t, stage, lane);
        if (!exact) {
            const int64_t p = wave0 + lane;
#pragma unroll
            for (int c = 0; c < 3; c++) r.drecOut[p * 3 + c] = diff[c];
        }
    } else {
        const double2 v[2] = {make_double2(cord[0], cord[1]),
                              make_double2(cord[2], tame ? radius : __builtin_nan(""))};
        store_chunks(reinterpret_cast<double2 *>(r.recOut + wave0), v, stage, lane);
        const double2 d[4] = {make_double2(diff[0], diff[1]), make_double2(diff[2], diff[3]),
                              make_double2(diff[4], diff[5]), make_double2((double)rotation_bound(theta), 0.0)};
        store_chunks(reinterpret_cast<double2 *>(r.drecOut + wave0 * 8), d, stage, lane);
    }
}

// False when contact_law would add exactly +-0 to every force component, so the
// pair can be skipped without changing a bit of the result: beyond
// radSum + attractDistance the law multiplies its terms by mask = 0, and while
// those terms are finite the product is +-0.  Adding +-0 leaves F unchanged,
// because F starts at +0 and round-to-nearest sums never yield -0.  The terms
// are finite when the distance is positive and at most sqrt(huge), the radius
// sum at most 1e6, the constants within inert_skip_allowed and the damping
// terms at most huge: the records' radius reads NaN, and with it radSum, unless
// both Diff and both radii are within their bounds (tame_bound).  Other pairs
// take the full path, so NaN/inf propagate exactly as in the sequential order
// of CombinedAccel::iterateCombined.
template <class R>
__device__ __forceinline__ bool pair_in_contact(R xDist, R yDist, R zDist, R radSum, R attractDistance) {
    const R particleDistance2 = xDist * xDist + yDist * yDist + zDist * zDist;
    const R activeDist = radSum + attractDistance;
    return !(particleDistance2 >= activeDist * activeDist && particleDistance2 <= huge_value<R>() &&
             particleDistance2 > R(0));
}

// What one particle's walks over its contacts and link sides share.
template <class R>
struct Walker {
    double xCord, yCord, zCord;
    double diff[6];
    R self[7];
    R radiusFlag;
    float rotSelf;
};

// Contacts of the neighbour list, added to F in list order.
template <class R, class CT, int BLOCK>
__device__ __forceinline__ void walk_contacts(const ForceArgs<R, CT, R> &f, const StepRecs<R> &r, int64_t p,
                                              int64_t tile, int lane, int32_t p0, const BlockRecs<R, BLOCK> &blk,
                                              const Walker<R> &me, R F[6]) {
    const int32_t cnt = ld_stream(f.nbrCount + p);
    const int32_t *nl = f.nbr + tile * 64 * f.nbrWidth + lane;
    // each entry's index is loaded one iteration ahead, so only the
    // record gather waits inside the iteration
    int32_t qNext = cnt > 0 ? ld_stream(nl) : 0;
    for (int32_t k = 0; k < cnt; k++) {
        const int32_t q = qNext;
        if (k + 1 < cnt) qNext = ld_stream(nl + (int64_t)(k + 1) * 64);
        double2 Q[2];
        load_partner(r, blk, p0, q, Q);
        const R xDist = (R)(me.xCord - Q[0].x);
        const R yDist = (R)(me.yCord - Q[0].y);
        const R zDist = (R)(me.zCord - Q[1].x);
        if (!pair_in_contact<R>(xDist, yDist, zDist, me.radiusFlag + chunk_radius(Q[1], R(0)), f.fp.attractDistance))
            continue;
        R other[7], d[6];
        float rotOther;
        partner_diff<R>(r, q, r.rec[q], me.diff, other, d, rotOther);
        other[6] = (R)f.radius[q];
        R self[7];
#pragma unroll
        for (int c = 0; c < 6; c++) self[c] = me.self[c];
        self[6] = (R)f.radius[p];
        contact_law<R>(R(1), xDist, yDist, zDist, self, other, d, f.fp, F);
    }
}

// Link sides in ascending link id, added to F.  GROW: the step's walk, which
// advances CT; else a second walk of it, which takes the CT already advanced.
// undecided: sides (bit k % 64) whose link the prefilter cannot prove intact;
// activeSides: linked pairs in contact (FP32, merged list; cnt <= 64).
template <bool GROW, class R, class CT, int BLOCK>
__device__ __forceinline__ void walk_sides(const ForceArgs<R, CT, R> &f, const StepRecs<R> &r, int64_t p,
                                           int64_t tile, int lane, int32_t p0, const BlockRecs<R, BLOCK> &blk,
                                           const Walker<R> &me, R F[6], uint64_t &undecidedOut,
                                           uint64_t &activeOut) {
    uint64_t undecided = 0, activeSides = 0;
    const int32_t cnt = (int32_t)ld_stream(f.linkCount + p);
    const int64_t base = tile * 64 * f.linkWidth + lane;
    // Software-pipelined: a side's partner word is loaded one
    // iteration ahead, and its record, CT and threshold code are
    // issued together, so a side waits for one memory latency (the
    // slowest of them) instead of a chain of dependent ones.
    int32_t owNext = cnt > 0 ? ld_stream(f.slotOther + base) : 0;  // partner; sign bit: broken
    // vmcnt(0) here: nothing loaded before the loop is still pending
    // at its header, so the header needs no wait (which, with the
    // previous side's CT stores outstanding, would drain them too).
    // gfx9 s_waitcnt immediate: vmcnt in bits 3:0 and 15:14 (0),
    // expcnt in 6:4 and lgkmcnt in 11:8 at their maxima (no wait).
    __builtin_amdgcn_s_waitcnt(0x0F70);
    for (int32_t k = 0; k < cnt; k++) {
        // FP64 form: the wave issues the side's loads at raised
        // priority, so the loads of all waves get in flight before
        // any returns to its arithmetic (measured 2-3% faster; the
        // FP32 form measured 1% slower with it)
        if constexpr (sizeof(R) == 8) __builtin_amdgcn_s_setprio(1);
        const int64_t sidx = base + (int64_t)k * 64;
        const int32_t ow = owNext;
        const int32_t q = ow & SLOT_LINK_MASK;
        CT cs[6];
        ct_load(f.ct, sidx, cs);
        // both loads unconditional (slotThr has the slot arrays'
        // extent; the last side re-reads its own word), so no branch
        // splits the issue from the one wait
        const uint16_t code = ld_stream(r.slotThr + sidx);
        owNext = ld_stream(f.slotOther + (k + 1 < cnt ? sidx + 64 : sidx));
        double2 Q[BlockRecs<R, BLOCK>::CHUNKS];
        load_partner(r, blk, p0, q, Q);
        if constexpr (sizeof(R) == 8) __builtin_amdgcn_s_setprio(0);
        R other[7], d[6];
        float rotOther;
        chunk_diff<R>(Q, me.diff, other, d, rotOther);
        other[6] = R(0);  // no radius needed
        const double dx = me.xCord - Q[0].x, dy = me.yCord - Q[0].y, dz = me.zCord - Q[1].x;
        // The prefilter is evaluated for every side and folded into
        // one branch condition, so the code's load cannot be sunk
        // into the break branch (where its wait would come late).
        const float thr = (float)code * r.thrScale;
        const float T = r.perLinkMaxLoad ? thr : thr * (1.0f + r.scalarMaxLoad);
        const bool skip =
            (r.prefilter != 0) & certainly_intact(T, r.bendBreak, r.l0Max, dx, dy, dz, me.rotSelf + rotOther);
        if (GROW && ((ow >= 0) & (f.breakCheck != 0) & !skip)) {
            undecided |= 1ull << (k & 63);
        }
        const R mask = ow < 0 ? R(0) : R(1);  // broken link (state == 0)
        R ct[6] = {(R)cs[0], (R)cs[1], (R)cs[2], (R)cs[3], (R)cs[4], (R)cs[5]};
        beam_law<R, GROW>(mask, (R)dx, (R)dy, (R)dz, me.self, other, d, f.fp, ct, F);
        if (sizeof(R) == 4 && f.linkedContacts) {
            // the pair's contact test (the contact loop's record test);
            // the rare active ones are applied after the loop, which
            // keeps the contact law out of this loop's registers
            // (placed after the beam law, where it does not delay the
            // side's loads)
            if (pair_in_contact<R>((R)dx, (R)dy, (R)dz, me.radiusFlag + chunk_radius(Q[1], R(0)),
                                   f.fp.attractDistance))
                activeSides |= 1ull << k;
        }
        if (GROW) {
#pragma unroll
            for (int c = 0; c < 6; c++) cs[c] = (CT)ct[c];
            ct_store(f.ct, sidx, cs);
        }
    }
    undecidedOut = undecided;
    activeOut = activeSides;
}

// One particle of the fused step (the body of k_step, k_step_loop and, up to
// the force, k_force: MOVE = false):
// break of the previous step, force, integration and the new records;
// cordN / diffN receive the integrated coordinates and translation Diff, and
// broke counts the links it broke at their smaller-index end.
template <class R, class CT, int BLOCK, bool MOVE = true>
__device__ __forceinline__ void step_particle(const ForceArgs<R, CT, R> &f, const IntegArgs &g, const StepRecs<R> &r,
                                              const int64_t p, const BlockRecs<R, BLOCK> &blk, double2 *stage,
                                              double cordN[3], double diffN[3], uint32_t &broke) {
    {
        double2 P[BlockRecs<R, BLOCK>::CHUNKS];   // own record, as staged
#pragma unroll
        for (int j = 0; j < BlockRecs<R, BLOCK>::CHUNKS; j++) P[j] = blk.c[j][threadIdx.x];
        Walker<R> me;
        me.xCord = P[0].x;
        me.yCord = P[0].y;
        me.zCord = P[1].x;
        me.radiusFlag = (R)chunk_radius(P[1], R(0));
        if constexpr (sizeof(R) == 4) {
            MixedRec m;
            __builtin_memcpy(&m, P, sizeof(m));
            join_diff6(m, r.tail[p], r.drec, p, me.diff);
            me.rotSelf = m.rot;
        } else {
            const double v[6] = {P[2].x, P[2].y, P[3].x, P[3].y, P[4].x, P[4].y};
#pragma unroll
            for (int c = 0; c < 6; c++) me.diff[c] = v[c];
            me.rotSelf = (float)P[5].x;
        }
        // the contact law takes the radius; it is read where that runs
#pragma unroll
        for (int c = 0; c < 6; c++) me.self[c] = (R)me.diff[c];
        me.self[6] = 0;
        R F[6] = {0, 0, 0, 0, 0, 0};
        const int lane = threadIdx.x & 63;
        // the wave's tile, as a scalar: the streams' addresses are then one
        // scalar base per access and a fixed offset per lane
        const int64_t tile = __builtin_amdgcn_readfirstlane((int32_t)(p >> 6));
        const int32_t p0 = (int32_t)(p - threadIdx.x);   // the workgroup's first particle
        walk_contacts(f, r, p, tile, lane, p0, blk, me, F);
        uint64_t undecided, activeSides;
        walk_sides<true>(f, r, p, tile, lane, p0, blk, me, F, undecided, activeSides);
        // What follows takes its addresses as scalar bases plus the lane, anew:
        // none of them is held over the walk.
        int l = threadIdx.x & 63;
        asm volatile("" : "+v"(l));
        const int64_t t0 = tile * 64;
        // The exact break test of the sides that the prefilter cannot decide
        // runs after the walk, where it holds none of the walk's registers
        // (inside it set the kernel's register count).  Undecided links
        // count as intact until then; the few particles whose link does break
        // sum their force again, with the updated slot words.
        if (MOVE && undecided) {
            bool redo = false;
            const int32_t cnt = (int32_t)f.linkCount[t0 + l];
            const int64_t base = tile * 64 * f.linkWidth + l;
            const double theta[3] = {g.tx[t0 + l], g.ty[t0 + l], g.tz[t0 + l]};
            for (int32_t k = 0; k < cnt; k++) {
                if (!((undecided >> (k & 63)) & 1)) continue;
                const int64_t sidx = base + (int64_t)k * 64;
                const int32_t ow = f.slotOther[sidx];
                if (ow < 0) continue;
                const auto Q = r.rec[ow];
                const int32_t word = f.slotLink[sidx];  // link id (intact: sign bit clear)
                if (link_breaks(f, word, ow, me.xCord - Q.x, me.yCord - Q.y, me.zCord - Q.z, theta)) {
                    // both ends reach the same verdict; each flags its own slot
                    f.slotLinkW[sidx] = word | SLOT_BROKEN;
                    f.slotOtherW[sidx] = ow | SLOT_BROKEN;
                    f.state[word] = 0;
                    broke += t0 + l < ow ? 1u : 0u;
                    redo = true;
                }
            }
            if (redo) {
#pragma unroll
                for (int c = 0; c < 6; c++) F[c] = 0;
                walk_contacts(f, r, t0 + l, tile, l, p0, blk, me, F);
                walk_sides<false>(f, r, t0 + l, tile, l, p0, blk, me, F, undecided, activeSides);
            }
        }
        if (sizeof(R) == 4 && activeSides)
            contact_sides(f, r, activeSides, tile * 64 * f.linkWidth + l, t0 + l, me.xCord, me.yCord, me.zCord, me.diff,
                          me.self, F);
        if (!MOVE || r.storeForce) store_force(f, t0 + l, F);
        if constexpr (!MOVE) return;
        const double radius = ld_stream(g.radius + t0 + l);
        const double Fd[6] = {(double)F[0], (double)F[1], (double)F[2], (double)F[3], (double)F[4], (double)F[5]};
        double cord[3] = {me.xCord, me.yCord, me.zCord};
        double theta[3] = {ld_stream(g.tx + t0 + l), ld_stream(g.ty + t0 + l), ld_stream(g.tz + t0 + l)};
        const bool fixed = (ld_stream(g.type + t0 + l) & HDM_TYPE_FIXED) != 0;
        const double waterLevel = g.blockWater ? g.blockWater[g.blockId[t0 + l]] : g.ip.waterLevel;
        integrate_state(g.ip, g.maps, g.mapMask, fixed, radius, waterLevel, Fd, cord, theta, me.diff);
        st_stream(g.otx + t0 + l, theta[0]);
        st_stream(g.oty + t0 + l, theta[1]);
        st_stream(g.otz + t0 + l, theta[2]);
        // a full wave stores its records contiguously, the last one lane by lane
        if (t0 + 64 <= f.n) store_records_wave(r, t0, l, cord, theta, me.diff, radius, stage);
        else store_records(r, t0 + l, cord, theta, me.diff, radius);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            cordN[c] = cord[c];
            diffN[c] = me.diff[c];
        }
    }
}

template <class R, class CT, int BLOCK, bool XCD, bool OCC>
__global__ void __launch_bounds__(BLOCK, step_waves<R>(OCC)) k_step(ForceArgs<R, CT, R> f, IntegArgs g,
                                                                    StepRecs<R> r) {
    fetch_arguments<sizeof(f) + sizeof(g) + sizeof(r)>();
    if (g.guard && *g.guard) {  // an earlier step found the neighbour list stale
        if (blockIdx.x == 0 && threadIdx.x == 0) *g.guardOut = 1u;
        return;
    }
    const int64_t wg = XCD ? xcd_block_index(gridDim.x) : (int64_t)blockIdx.x;
    uint32_t broke = 0;  // links this lane's particle broke (counted at its smaller-index end)
    const int64_t p = wg * BLOCK + threadIdx.x;
    const bool active = p < f.n;
    __shared__ BlockRecs<R, BLOCK> blk;
    const int64_t wave0 = wg * BLOCK + (threadIdx.x & ~63);
    stage_records(r, wave0, f.n, blk);
    __syncthreads();
    double cordN[3] = {0, 0, 0}, diffN[3] = {0, 0, 0};
    if (active) step_particle<R, CT, BLOCK>(f, g, r, p, blk, blk.out[threadIdx.x >> 6], cordN, diffN, broke);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // the particle's index anew (see step_particle)
    const int64_t pl = wg * BLOCK + tid;
    if (f.brokenCount) {
        broke = wave_sum_u32(broke);
        if ((threadIdx.x & 63) == 0 && broke) atomicAdd((unsigned long long *)f.brokenCount, (unsigned long long)broke);
    }
    if (g.guardOut) {
        if (pl < f.n && guard_trips(g, pl, cordN)) *g.guardOut = 1u;
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(g.stepsDone, 1u);
    } else if (g.partials) {
        skin_partials<BLOCK>(g, pl < f.n, diffN);
    }
}

// CombinedAccel::iterateCombined (CombinedAccel.h:121-197) alone (hdm_force):
// the fused step up to the force, on the same records.  2M-particle slab, FP32
// form: 294 us; the previous form, which gathered ten SoA fields per partner,
// 715 us (FP64, 2.1M: 601 and 1,044).  Records that are not current are packed
// first (k_pack_records); hdm_integrate keeps them current between calls.
template <class R, class CT>
__global__ void __launch_bounds__(TPB, step_waves<R>(false)) k_force(ForceArgs<R, CT, R> f, StepRecs<R> r) {
    __shared__ BlockRecs<R, TPB> blk;
    fetch_arguments<sizeof(f) + sizeof(r)>();
    // launch order, as the step of large states (step_form): 300 -> 294 us FP32,
    // 607 -> 600 FP64 on slabs of 2M particles
    const int64_t wg = blockIdx.x, p = wg * TPB + threadIdx.x;
    stage_records(r, wg * TPB + (threadIdx.x & ~63), f.n, blk);
    __syncthreads();
    if (p >= f.n) return;
    double cordN[3], diffN[3];
    uint32_t broke = 0;
    step_particle<R, CT, TPB, false>(f, IntegArgs{}, r, p, blk, nullptr, cordN, diffN, broke);
}

// ---- tile step -------------------------------------------------------------------
// One of three kernel arguments by a wave-uniform index.  The values pass
// through registers first: a select between members of an argument struct
// becomes a load at a selected address, and the struct goes to scratch.
template <class T>
__device__ __forceinline__ T pick3(int c, T a, T b, T d) {
    asm volatile("" : "+s"(a), "+s"(b), "+s"(d));
    return c == 0 ? a : c == 1 ? b : d;
}

// One component (c = 0..2: coordinate c, 3..5: rotation c - 3) of
// integrate_state: the same expressions on the same operands, for a wave that
// holds that component of 64 particles.  q / diff: the component's coordinate
// or rotation and its Diff, replaced by the new ones; cord: the particle's
// coordinates before the step.
__device__ __forceinline__ void integrate_component(const hdm_integ_params &ip, const MapDev *maps, int32_t mapMask,
                                                    bool fixed, double radius, double waterLevel, int c, double F,
                                                    const double cord[3], double &q, double &diff) {
    if (ip.variant == HDM_INTEG_ICEBLOCK && fixed) {
        diff = 0;
        return;
    }
    const double diameter = radius * 2.0;
    const double zCord = cord[2];
    const double particleMass = ip.rhoIce * diameter * diameter * diameter;
    const double particleMomentInertia = particleMass * diameter * diameter / 6.0;
    double dragCoeff;
    if (ip.variant == HDM_INTEG_ICEBLOCK) {
        dragCoeff = (zCord > waterLevel) ? ip.airDrag : ip.waterDrag;
        if (c == 2) {
            if (zCord > waterLevel) F += -ip.g * particleMass;
            if (zCord <= waterLevel) F += ip.lift * particleMass;
        }
    } else {
        const float fx = (float)cord[0], fy = (float)cord[1];
        const double bedzCord = (mapMask & (1 << HDM_MAP_BED)) ? map_interp(maps[HDM_MAP_BED], fx, fy)
                                                               : ((cord[0] < ip.bedXEnd) ? ip.bedZ : ip.deepZ);
        const double fric = (mapMask & (1 << HDM_MAP_FRICTION)) ? map_interp(maps[HDM_MAP_FRICTION], fx, fy)
                                                                : ((cord[0] < ip.frictionXEnd) ? 1.0 : 0.0);
        if ((zCord + radius) - bedzCord < ip.bedInteract) {
            double d = ip.bedDrag * fric;
            dragCoeff = (ip.frictionCap < d) ? ip.frictionCap : d;
        } else if (zCord > waterLevel) {
            dragCoeff = ip.airDrag;
        } else {
            dragCoeff = ip.waterDrag;
        }
        if (c == 2) {
            if (zCord > waterLevel) F += -ip.g * particleMass;
            if (zCord <= waterLevel) F += ip.lift * particleMass;
            if (zCord + radius < bedzCord) F += ip.bedStiffness * (bedzCord - (zCord + radius));
        }
        const double ext = c < 3 ? pick3(c, ip.ext[0], ip.ext[1], ip.ext[2])
                                 : pick3(c - 3, ip.ext[3], ip.ext[4], ip.ext[5]);
        F += (mapMask & (1 << (HDM_MAP_EXT + c))) ? map_interp(maps[HDM_MAP_EXT + c], fx, fy) : ext;
    }
    // central_difference
    const double inert = c < 3 ? particleMass : particleMomentInertia;
    const double dragInvDt2 = dragCoeff * ip.invDt2;
    const double inertDtSqr = inert * ip.invDtSqr;
    const double pInertDtSqr = inert / ip.dtSqr;
    const double invC = 1.0 / (pInertDtSqr + dragCoeff * ip.invDt2);
    const double next = (F + inertDtSqr * diff + dragInvDt2 * -diff) * invC;
    const double prev = q;
    q = q + next;
    if (ip.variant != HDM_INTEG_ICEBLOCK) {
        if (ip.velocityLimit) {
            const double vel = c < 3 ? next * ip.invDt : (q - prev) * ip.invDt;
            const double lim = c < 3 ? ip.maxVel : ip.maxRot;
            if (vel > lim) q = ip.dt * lim + prev;
            if (vel < -lim) q = ip.dt * -lim + prev;
        }
        if (c < 3) {
            const double lower = pick3(c, ip.lower[0], ip.lower[1], ip.lower[2]);
            const double upper = pick3(c, ip.upper[0], ip.upper[1], ip.upper[2]);
            const int32_t boundLo = pick3(c, ip.bound[0], ip.bound[2], ip.bound[4]);
            const int32_t boundHi = pick3(c, ip.bound[1], ip.bound[3], ip.bound[5]);
            if (q + radius < lower && boundLo) q = prev;
            if (q - radius > upper && boundHi) q = prev;
        }
    }
    diff = q - prev;
}

// The fused step with the work of 64 particles (one wave tile) spread over
// the six waves of a workgroup, for states of too few particles to fill the
// chip with one lane each (tile_step_pays).  There a step takes as long as one
// lane's walk, a chain of some 24 memory latencies; here wave w takes the
// list entries and link sides w, w + 6, ... of all 64 particles, so those of a
// round are in flight at once.  What the laws add to each force component goes
// to LDS, and wave c sums component c of every particle in the sequential
// order (contacts in list order, then per side damping and elastic term): the
// sums of step_particle bit for bit.  Wave c then integrates component c.
constexpr int TILE_WAVES = 6;
constexpr int TILE_THREADS = TILE_WAVES * 64;
constexpr int OUT_PITCH = 66;   // doubles per row of the output stage (8 B shifts between rows: no bank conflicts)

template <class R>
struct TileShared {
    union {
        R part[TILE_WAVES][12][64];     // terms of a round: [side][component, damping then elastic][particle]
        double out[12][OUT_PITCH];      // new coordinates, rotations and Diff
    };
    double2 own[TILE_THREADS];          // records of the tile's particles, as stored
    // what the end of the step reads, loaded at its start, as is the guard word:
    // each was a wait of its own in a kernel that is one chain of waits (step
    // of the 16k block, FP32 form: 11.4 -> 10.5 us; 960 particles, FP64: 12.8
    // -> 12.4)
    double radius[64], theta[3][64];
    float snapshot[3][64];
    uint8_t type[64];
    int32_t contacts;                   // some pair of the tile is in contact
};

// The tile's own records in LDS read as particle p's fields (Walker).
template <class R>
__device__ __forceinline__ Walker<R> read_own(const TileShared<R> &sm, const StepRecs<R> &r, int lane, int64_t p) {
    Walker<R> me;
    if constexpr (sizeof(R) == 4) {
        MixedRec P;
        MixedTail T;
        double2 a[4], b[2];
#pragma unroll
        for (int j = 0; j < 4; j++) a[j] = sm.own[lane * 4 + j];
#pragma unroll
        for (int j = 0; j < 2; j++) b[j] = sm.own[256 + lane * 2 + j];
        __builtin_memcpy(&P, a, sizeof(P));
        __builtin_memcpy(&T, b, sizeof(T));
        me.xCord = P.x;
        me.yCord = P.y;
        me.zCord = P.z;
        join_diff6(P, T, r.drec, p, me.diff);
        me.radiusFlag = P.radius;
        me.rotSelf = P.rot;
    } else {
        const double2 a = sm.own[lane * 2], b = sm.own[lane * 2 + 1];
        me.xCord = a.x;
        me.yCord = a.y;
        me.zCord = b.x;
        me.radiusFlag = b.y;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const double2 d = sm.own[128 + lane * 4 + j];
            me.diff[2 * j] = d.x;
            me.diff[2 * j + 1] = d.y;
        }
        me.rotSelf = (float)sm.own[128 + lane * 4 + 3].x;
    }
#pragma unroll
    for (int c = 0; c < 6; c++) me.self[c] = (R)me.diff[c];
    me.self[6] = 0;
    return me;
}

// What the contact law adds for particle and partner q.
template <class R, class CT>
__device__ __forceinline__ void contact_pair(const ForceArgs<R, CT, R> &f, const StepRecs<R> &r, int64_t p, int32_t q,
                                             const Walker<R> &me, R t[6]) {
    const auto Q = r.rec[q];
    R self[7], other[7], d[6];
#pragma unroll
    for (int c = 0; c < 6; c++) self[c] = me.self[c];
    self[6] = (R)f.radius[p];
    float rot;
    partner_diff<R>(r, q, Q, me.diff, other, d, rot);
    other[6] = (R)f.radius[q];
    contact_terms<R>(R(1), (R)(me.xCord - Q.x), (R)(me.yCord - Q.y), (R)(me.zCord - Q.z), self, other, d, f.fp, t);
}

// A side's loads in flight.
template <class R, class CT>
struct SideLoads {
    double2 rec[sizeof(R) == 8 ? 6 : 4];
    CT ct[6];
    uint16_t code;
    int32_t ow;
};

// broke: links this wave's lanes broke, counted at their smaller-index end.
// Returns false when an earlier step found the neighbour list stale (nothing
// is stored then).
template <class R, class CT, bool MOVE = true>
__device__ __forceinline__ bool step_tile(const ForceArgs<R, CT, R> &f, const IntegArgs &g, const StepRecs<R> &r,
                                          int64_t tile, TileShared<R> &sm, uint32_t &broke) {
    constexpr int W = TILE_WAVES;
    const int t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const int64_t p0 = tile * 64, p = p0 + lane;
    const bool act = p < f.n;
    // the tile's records, 16 B per thread: rec first, then drec / tail
    constexpr int RC = (int)sizeof(typename RecOf<R>::type) / 16, SC = 6 - RC;
    const bool first = t < 64 * RC;
    const int u = first ? t : t - 64 * RC, pl = first ? u / RC : u / SC, j = first ? u % RC : u % SC;
    const bool here = p0 + pl < f.n;
    double2 mine = {};
    if (here) {
        const void *second = sizeof(R) == 4 ? (const void *)(r.tail + p0) : (const void *)(r.drec + p0 * 8);
        mine = first ? reinterpret_cast<const double2 *>(r.rec + p0)[u] : reinterpret_cast<const double2 *>(second)[u];
    }
    const int32_t nc = act ? ld_stream(f.nbrCount + p) : 0;
    const int32_t lc = act ? (int32_t)ld_stream(f.linkCount + p) : 0;
    // side k of the tile's particles: row row0 + k of 64 slots (scalar row addresses, a fixed offset per lane)
    const int64_t row0 = tile * f.linkWidth;
    auto word = [&](int32_t k) { return k < f.linkWidth ? ld_stream(f.slotOther + (row0 + k) * 64 + lane) : 0; };
    int32_t owNext = word(w);
    const int32_t *nl = f.nbr + tile * (int64_t)64 * f.nbrWidth + lane;
    int32_t entry = w < f.nbrWidth ? ld_stream(nl + (int64_t)w * 64) : 0;
    auto load_side = [&](int32_t k, SideLoads<R, CT> &v) {
        v.ow = owNext;
        owNext = word(k + W);
        if (k < lc) {
            const int32_t q = v.ow & SLOT_LINK_MASK;
            const double2 *a = reinterpret_cast<const double2 *>(r.rec + q);
#pragma unroll
            for (int i = 0; i < RC; i++) v.rec[i] = a[i];
            if constexpr (sizeof(R) == 8) {
                const double2 *d = reinterpret_cast<const double2 *>(r.drec + (int64_t)q * 8);
#pragma unroll
                for (int i = 0; i < 4; i++) v.rec[2 + i] = d[i];
            }
            ct_load(f.ct + (row0 + k) * 384, lane, v.ct);
            v.code = ld_stream(r.slotThr + (row0 + k) * 64 + lane);
        }
    };
    uint32_t stale = 0;
    if constexpr (MOVE) {
        stale = g.guard ? *g.guard : 0;
        if (act) {
            if (w >= 3) sm.theta[w - 3][lane] = ld_stream(pick3(w - 3, g.tx, g.ty, g.tz) + p);
            else if (g.guardOut) sm.snapshot[w][lane] = ld_stream((w == 0 ? g.x0f : w == 1 ? g.y0f : g.z0f) + p);
            if (w == 0) sm.radius[lane] = ld_stream(g.radius + p);
            if (w == 1) sm.type[lane] = ld_stream(g.type + p);
        }
    }
    sm.own[t] = mine;
    if (t == 0) sm.contacts = 0;
    __syncthreads();
    if (MOVE && stale) return false;
    // the own state is read from LDS where it is used: it isn't held over the rounds
    R F = 0;   // component w of the force on particle p

    if (__any(nc > 0)) {
        const Walker<R> me = read_own(sm, r, lane, p);
        auto in_contact = [&](int32_t q) {
            const auto Q = r.rec[q];
            return pair_in_contact<R>((R)(me.xCord - Q.x), (R)(me.yCord - Q.y), (R)(me.zCord - Q.z),
                                      me.radiusFlag + (R)rec_radius(Q), f.fp.attractDistance);
        };
        bool some = false;
        for (int32_t b = 0; __any(nc > b); b += W) {
            const int32_t q = entry;
            if (b + W + w < f.nbrWidth) entry = ld_stream(nl + (int64_t)(b + W + w) * 64);
            if (b + w < nc) some |= in_contact(q);
        }
        if (__any(some) && lane == 0) sm.contacts = 1;
        __syncthreads();
        if (sm.contacts) {
            for (int32_t b = 0; __any(nc > b); b += W) {
                if (b + w < nc) {
                    const int32_t q = nl[(int64_t)(b + w) * 64];
                    R tm[6] = {0, 0, 0, 0, 0, 0};   // adding +0 leaves F (never -0) as it is
                    if (in_contact(q)) contact_pair(f, r, p, q, me, tm);
#pragma unroll
                    for (int c = 0; c < 6; c++) sm.part[w][c][lane] = tm[c];
                }
                __syncthreads();
#pragma unroll
                for (int s = 0; s < W; s++)
                    if (b + s < nc) F += sm.part[s][w][lane];
                __syncthreads();
            }
        }
    }

    uint64_t pairs = 0;   // bit i: the pair of this wave's side in round i is in contact (FP32, merged list)
    int round = 0;
    for (int32_t b = 0; __any(lc > b); b += W, round++) {
        const int32_t k = b + w;
        SideLoads<R, CT> v;
        load_side(k, v);
        if (k < lc) {
            const Walker<R> me = read_own(sm, r, lane, p);
            const int32_t ow = v.ow, q = ow & SLOT_LINK_MASK;
            R other[7], d[6];
            float rotOther;
            chunk_diff<R>(v.rec, me.diff, other, d, rotOther);
            other[6] = R(0);
            const double dx = me.xCord - v.rec[0].x, dy = me.yCord - v.rec[0].y, dz = me.zCord - v.rec[1].x;
            const float thr = (float)v.code * r.thrScale;
            const float T = r.perLinkMaxLoad ? thr : thr * (1.0f + r.scalarMaxLoad);
            const bool skip =
                (r.prefilter != 0) & certainly_intact(T, r.bendBreak, r.l0Max, dx, dy, dz, me.rotSelf + rotOther);
            const R mask = ow < 0 ? R(0) : R(1);  // broken link (state == 0)
            if (sizeof(R) == 4 && f.linkedContacts &&
                pair_in_contact<R>((R)dx, (R)dy, (R)dz, me.radiusFlag + chunk_radius(v.rec[1], R(0)),
                                   f.fp.attractDistance))
                pairs |= 1ull << round;
            R ct[6];
#pragma unroll
            for (int c = 0; c < 6; c++) ct[c] = (R)v.ct[c];
            beam_terms<R>(mask, (R)dx, (R)dy, (R)dz, me.self, other, d, f.fp, ct,
                          [&](int c, int h, R x) { sm.part[w][6 * h + c][lane] = x; });
            CT cs[6];
#pragma unroll
            for (int c = 0; c < 6; c++) cs[c] = (CT)ct[c];
            ct_store(f.ct + (row0 + k) * 384, lane, cs);
            // The rare exact test after the law, where none of its registers
            // are live: a link found broken has its terms multiplied by 0, as
            // the law multiplies them by the mask (x * 1 * 0 == x * 0).
            if (MOVE && ((ow >= 0) & (f.breakCheck != 0) & !skip)) {
                const auto Q2 = r.rec[q];
                const int64_t sidx = (row0 + k) * 64 + lane;
                const int32_t link = f.slotLink[sidx];  // link id (intact: sign bit clear)
                const double theta[3] = {g.tx[p], g.ty[p], g.tz[p]};
                const Walker<R> own = read_own(sm, r, lane, p);
                if (link_breaks(f, link, q, own.xCord - Q2.x, own.yCord - Q2.y, own.zCord - Q2.z, theta)) {
                    // both ends reach the same verdict; each flags its own slot
                    for (int c = 0; c < 12; c++) sm.part[w][c][lane] *= R(0);
                    f.slotLinkW[sidx] = link | SLOT_BROKEN;
                    f.slotOtherW[sidx] = ow | SLOT_BROKEN;
                    f.state[link] = 0;
                    broke += p < q ? 1u : 0u;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < W; s++)
            if (b + s < lc) {
                F += sm.part[s][w][lane];
                F += sm.part[s][6 + w][lane];
            }
        __syncthreads();
    }

    // the contacts of linked pairs, after every beam, in side order
    if (sizeof(R) == 4 && f.linkedContacts) {
        if (t == 0) sm.contacts = 0;
        __syncthreads();
        if (__any(pairs != 0) && lane == 0) sm.contacts = 1;
        __syncthreads();
        if (sm.contacts) {
            const Walker<R> me = read_own(sm, r, lane, p);
            round = 0;
            for (int32_t b = 0; __any(lc > b); b += W, round++) {
                R tm[6] = {0, 0, 0, 0, 0, 0};
                if ((pairs >> round) & 1ull)
                    contact_pair(f, r, p, f.slotOther[(row0 + b + w) * 64 + lane] & SLOT_LINK_MASK, me, tm);
                if (b + w < lc)
#pragma unroll
                    for (int c = 0; c < 6; c++) sm.part[w][c][lane] = tm[c];
                __syncthreads();
#pragma unroll
                for (int s = 0; s < W; s++)
                    if (b + s < lc) F += sm.part[s][w][lane];
                __syncthreads();
            }
        }
    }

    // the wave's component of the new state
    if (act && (!MOVE || r.storeForce)) (w < 3 ? pick3(w, f.f0, f.f1, f.f2) : pick3(w - 3, f.f3, f.f4, f.f5))[p] = F;
    if constexpr (!MOVE) return true;
    if (act) {
        const bool fixed = (sm.type[lane] & HDM_TYPE_FIXED) != 0;
        const double waterLevel = g.blockWater ? g.blockWater[g.blockId[p]] : g.ip.waterLevel;
        const double radius = sm.radius[lane];
        const Walker<R> me = read_own(sm, r, lane, p);
        const double cord[3] = {me.xCord, me.yCord, me.zCord};
        double q, diff;
        if (w < 3) {
            q = w == 0 ? cord[0] : w == 1 ? cord[1] : cord[2];
            diff = w == 0 ? me.diff[0] : w == 1 ? me.diff[1] : me.diff[2];
        } else {
            q = sm.theta[w - 3][lane];
            diff = w == 3 ? me.diff[3] : w == 4 ? me.diff[4] : me.diff[5];
        }
        integrate_component(g.ip, g.maps, g.mapMask, fixed, radius, waterLevel, w, (double)F, cord, q, diff);
        if (w >= 3) st_stream(pick3(w - 3, g.otx, g.oty, g.otz) + p, q);
        sm.out[w][lane] = q;
        sm.out[6 + w][lane] = diff;
    }
    __syncthreads();
    // the new records, one 16 B chunk per thread
    if (here) {
        double D[6];
#pragma unroll
        for (int c = 0; c < 6; c++) D[c] = sm.out[6 + c][pl];
        auto tame_radius = [&]() {
            const double rad = sm.radius[pl];
            bool tame = fabs(rad) <= 5e5;
#pragma unroll
            for (int c = 0; c < 6; c++) tame &= fabs(D[c]) <= r.tame;
            return tame ? rad : __builtin_nan("");
        };
        auto rot = [&]() {
            const double th[3] = {sm.out[3][pl], sm.out[4][pl], sm.out[5][pl]};
            return rotation_bound(th);
        };
        double2 v;
        if constexpr (sizeof(R) == 8) {
            if (first) {
                v = j == 0 ? make_double2(sm.out[0][pl], sm.out[1][pl]) : make_double2(sm.out[2][pl], tame_radius());
                reinterpret_cast<double2 *>(r.recOut + p0)[u] = v;
            } else {
                v = j == 0 ? make_double2(D[0], D[1])
                           : j == 1 ? make_double2(D[2], D[3])
                                    : j == 2 ? make_double2(D[4], D[5]) : make_double2((double)rot(), 0.0);
                reinterpret_cast<double2 *>(r.drecOut + p0 * 8)[u] = v;
            }
        } else {
            float hi[3], lo[3];
            const bool exact = split_diff3(D, hi, lo);
            if (first) {
                if (j == 0) {
                    v = make_double2(sm.out[0][pl], sm.out[1][pl]);
                } else if (j == 1) {
                    const float2 rr = make_float2((float)tame_radius(), rot());
                    v = make_double2(sm.out[2][pl], __builtin_bit_cast(double, rr));
                } else {
                    const float4 m = j == 2 ? make_float4(hi[0], hi[1], hi[2], (float)D[3])
                                            : make_float4((float)D[4], (float)D[5], lo[0], lo[1]);
                    v = __builtin_bit_cast(double2, m);
                }
                reinterpret_cast<double2 *>(r.recOut + p0)[u] = v;
            } else {
                const float2 l2 = make_float2(lo[2], 0.0f);
                v = j == 0 ? make_double2(D[3], D[4]) : make_double2(D[5], __builtin_bit_cast(double, l2));
                reinterpret_cast<double2 *>(r.tailOut + p0)[u] = v;
                if (j == 1 && !exact) {
#pragma unroll
                    for (int c = 0; c < 3; c++) r.drecOut[(p0 + pl) * 3 + c] = D[c];
                }
            }
        }
    }
    return true;
}

template <class R, class CT>
__global__ void __launch_bounds__(TILE_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
k_step_tile(ForceArgs<R, CT, R> f, IntegArgs g, StepRecs<R> r) {
    __shared__ TileShared<R> sm;
    fetch_arguments<sizeof(f) + sizeof(g) + sizeof(r)>();
    const int64_t tile = xcd_block_index(gridDim.x);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t broke = 0;
    if (!step_tile<R, CT>(f, g, r, tile, sm, broke)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *g.guardOut = 1u;
        return;
    }
    const int64_t p = tile * 64 + lane;
    const bool act = p < f.n;
    if (f.brokenCount && __any(broke != 0)) {
        broke = wave_sum_u32(broke);
        if (lane == 0) atomicAdd((unsigned long long *)f.brokenCount, (unsigned long long)broke);
    }
    if (g.guardOut) {
        if (w == 0 && act) {
            const double c[3] = {sm.out[0][lane], sm.out[1][lane], sm.out[2][lane]};
            if (guard_trips(g, p, c, sm.snapshot[0][lane], sm.snapshot[1][lane], sm.snapshot[2][lane]))
                *g.guardOut = 1u;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(g.stepsDone, 1u);
    } else if (g.partials) {
        // the tile's row of the rebuild-test maxima (skin_partials)
        if (w < 3) {
            double m = 0.0;
            if (act) {
                const double d = sm.out[6 + w][lane];
                m = d > 0.0 ? d : 0.0;
            }
            m = wave_max(m);
            if (lane == 0) g.partials[(int64_t)blockIdx.x * 3 + w] = m;
        }
    }
}

// k_force for the states k_step_tile serves.
template <class R, class CT>
__global__ void __launch_bounds__(TILE_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
k_force_tile(ForceArgs<R, CT, R> f, StepRecs<R> r) {
    __shared__ TileShared<R> sm;
    uint32_t broke = 0;
    fetch_arguments<sizeof(f) + sizeof(r)>();
    (void)step_tile<R, CT, false>(f, IntegArgs{}, r, xcd_block_index(gridDim.x), sm, broke);
}

// Sides whose words, codes and partners a lane loads together in the link break.
constexpr int BREAK_BATCH = 4;

// The link break on the records (the end of a run, and hdm_break while the
// records are current): linkUpdate (HiDEMLib.h:256-269,
// HiDEMDefLinkBreakFunc) per particle, as the next fused step would apply it,
// so the SoA state need not be unpacked first.  Every intact side of p takes
// the float prefilter and, when that cannot prove the link intact, the exact
// FP64 test; both ends reach the same verdict (the pair differences are
// antisymmetric) and flag their own slot, and the end with the smaller index
// counts the link.  The links broken are those k_break would break.
//
// A link needs 6 B of slot word and code per side and its ends' coordinates,
// about 1.1 GB on the 8M-particle slab, so the walk is latency bound: partners
// of the same workgroup come from LDS, BREAK_BATCH sides are in flight at
// once, and the exact tests run after the walk.  Slab: FP32 0.30 ms (0.61 with
// one side in flight at a time, every partner from memory), FP64 0.42 ms (0.67
// with a thread per slot).
template <class R>
__global__ void __launch_bounds__(TPB) k_break_recs(ForceArgs<R, R, R> f, StepRecs<R> r, uint64_t *counter,
                                                    const uint32_t *stepsDone, uint32_t steps) {
    constexpr int B = BREAK_BATCH;
    constexpr int REC = BlockRecs<R, TPB>::REC;
    __shared__ double2 own[2][TPB];   // x, y | z, radius (FP32 form: and rotation bound)
    __shared__ float ownRot[TPB];
    fetch_arguments<sizeof(f) + sizeof(r)>();
    if (stepsDone && *stepsDone != steps) return;   // a step before it was skipped
    const int64_t wg0 = xcd_block_index(gridDim.x) * TPB, p = wg0 + threadIdx.x;
    uint32_t broke = 0;
    double2 P[2] = {};
    float rotSelf = 0.0f;
    // chunks 0 and 1 of a record and the rotation bound
    auto load = [&](int64_t q, double2 (&c)[2], float &rot) {
        const double2 *a = reinterpret_cast<const double2 *>(r.rec) + q * REC;
        c[0] = a[0];
        c[1] = a[1];
        if constexpr (sizeof(R) == 8) rot = (float)r.drec[q * 8 + 6];
        else rot = high_float(c[1].y);
    };
    if (p < f.n) {
        load(p, P, rotSelf);
        own[0][threadIdx.x] = P[0];
        own[1][threadIdx.x] = P[1];
        ownRot[threadIdx.x] = rotSelf;
    }
    __syncthreads();
    if (p < f.n) {
        const int lane = threadIdx.x & 63;
        const int64_t row0 = (int64_t)__builtin_amdgcn_readfirstlane((int32_t)(p >> 6)) * f.linkWidth;
        const int32_t cnt = (int32_t)f.linkCount[p];
        uint64_t undecided = 0;   // bit k % 64: side k
        int32_t ow[B];
        uint16_t code[B];
        auto fetch = [&](int32_t k0) {   // past the last side: its own word again
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int64_t s = (row0 + (k0 + j < cnt ? k0 + j : cnt - 1)) * 64 + lane;
                ow[j] = ld_stream(f.slotOther + s);
                code[j] = ld_stream(r.slotThr + s);
            }
        };
        if (cnt > 0) fetch(0);
        for (int32_t k = 0; k < cnt; k += B) {
            double2 Q[B][2];
            float rot[B], thr[B];
            bool intact[B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int32_t q = ow[j] & SLOT_LINK_MASK;
                const uint32_t at = (uint32_t)(q - (int32_t)wg0);
                intact[j] = ow[j] >= 0 && k + j < cnt;
                thr[j] = (float)code[j] * r.thrScale;
                if (at < (uint32_t)TPB) {
                    Q[j][0] = lds_load(&own[0][at]);
                    Q[j][1] = lds_load(&own[1][at]);
                    rot[j] = ownRot[at];
                } else {
                    load(q, Q[j], rot[j]);
                }
            }
            if (k + B < cnt) fetch(k + B);
#pragma unroll
            for (int j = 0; j < B; j++) {
                const float T = r.perLinkMaxLoad ? thr[j] : thr[j] * (1.0f + r.scalarMaxLoad);
                const bool sure = (r.prefilter != 0) &
                                  certainly_intact(T, r.bendBreak, r.l0Max, P[0].x - Q[j][0].x, P[0].y - Q[j][0].y,
                                                   P[1].x - Q[j][1].x, rotSelf + rot[j]);
                if (intact[j] && !sure) undecided |= 1ull << ((k + j) & 63);
            }
        }
        if (undecided) {
            const double theta[3] = {f.tx[p], f.ty[p], f.tz[p]};
            for (int32_t k = 0; k < cnt; k++) {
                if (!((undecided >> (k & 63)) & 1)) continue;
                const int64_t s = (row0 + k) * 64 + lane;
                const int32_t q = f.slotOther[s];
                if (q < 0) continue;   // broken already
                const auto Q = r.rec[q];
                const int32_t word = f.slotLink[s];
                if (link_breaks(f, word, q, P[0].x - Q.x, P[0].y - Q.y, P[1].x - Q.z, theta)) {
                    f.slotLinkW[s] = word | SLOT_BROKEN;
                    f.slotOtherW[s] = q | SLOT_BROKEN;
                    f.state[word] = 0;
                    broke += p < q ? 1u : 0u;
                }
            }
        }
    }
    broke = wave_sum_u32(broke);
    if ((threadIdx.x & 63) == 0 && broke) {
        if (counter) atomicAdd((unsigned long long *)counter, (unsigned long long)broke);
        if (f.brokenCount) atomicAdd((unsigned long long *)f.brokenCount, (unsigned long long)broke);
    }
}

// ---- persistent timestep ------------------------------------------------------
// Grid barrier of a co-resident (cooperative) launch, in two levels so no
// word takes more than a few dozen arrivals: workgroup b arrives at group
// b % GRID_GROUPS, the last arrival of a group at the top word, and the last
// arrival there re-arms the counters and advances the generation the others
// wait on.  The words sit 128 B apart (their own L2 lines).  Only the first
// thread of a workgroup fences: the workgroup barrier before it has every
// wave's stores in its XCD's L2, which its release fence writes back; its
// acquire fence invalidates the L2 and the CU's L1 that the workgroup's
// waves read through after the closing workgroup barrier.  (Agent-scope
// fences write back and invalidate a whole XCD's L2, so one per workgroup
// and barrier rather than one per wave.)  A wait that outlasts maxSpins sets
// *error and returns, so a launch that could not make every workgroup
// resident ends instead of hanging (the host then fails the run).
constexpr int GRID_GROUPS = 64;
constexpr int BARRIER_STRIDE = 32;   // u32 words between counters
constexpr int BARRIER_WORDS = (GRID_GROUPS + 2) * BARRIER_STRIDE;

__device__ __forceinline__ void grid_barrier(uint32_t *bar, uint32_t *error, uint32_t maxSpins) {
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t *top = bar + GRID_GROUPS * BARRIER_STRIDE;
        uint32_t *gen = top + BARRIER_STRIDE;
        const uint32_t g = blockIdx.x % GRID_GROUPS;
        const uint32_t groups = gridDim.x < GRID_GROUPS ? gridDim.x : GRID_GROUPS;
        const uint32_t members = gridDim.x / GRID_GROUPS + (g < gridDim.x % GRID_GROUPS ? 1u : 0u);
        // the generation cannot advance before this workgroup arrives
        const uint32_t seen = __hip_atomic_load(gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        if (atomicAdd(bar + g * BARRIER_STRIDE, 1u) == members - 1) {
            __hip_atomic_store(bar + g * BARRIER_STRIDE, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__hip_atomic_fetch_add(top, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == groups - 1) {
                __hip_atomic_store(top, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_fetch_add(gen, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        uint32_t spins = 0;
        while (__hip_atomic_load(gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == seen) {
            __builtin_amdgcn_s_sleep(1);
            if (++spins > maxSpins) {
                atomicOr(error, 1u);
                break;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
}

// Tile of the k-th visit of workgroup b in a grid of G workgroups (G a
// multiple of 8) over T tiles: visit v = b + k G is dispatched on XCD v % 8,
// and each XCD's visits cover one contiguous range of tiles (the numbering
// of xcd_block_index over the T visits).
__device__ __forceinline__ int64_t xcd_tile(int64_t v, int64_t T) {
    const int64_t q = T / 8, rem = T % 8, xcd = v % 8, local = v / 8;
    return (xcd < rem) ? xcd * (q + 1) + local : rem * (q + 1) + (xcd - rem) * q + local;
}

struct LoopArgs {
    int32_t steps;        // steps to run; fewer when one trips the exact test
    uint32_t *barrier;    // BARRIER_WORDS, zero before the first launch
    uint32_t *error;      // set when a barrier wait timed out
    uint32_t maxSpins;
};

// The arguments of one step of k_step_loop.  Two sets sit in device memory:
// the first step's and the one with the ping-pong roles swapped, and step s
// reads set s % 2.  Loading a field from the set of the step's parity at its
// point of use keeps it out of the registers between uses; roles swapped in
// registers stay live across the whole loop and spill (and two sets passed
// as kernel arguments and selected by parity are copied to scratch).
template <class R, class CT>
struct LoopSet {
    ForceArgs<R, CT, R> f;
    IntegArgs g;
    StepRecs<R> r;
};

// Several fused steps in one co-resident launch (HDM_REBUILD_LEARNED with
// hdm_exec_params.persistent): every workgroup runs the particles of its
// tiles through step_particle, the grid synchronises, and the next step
// starts on the other argument set -- unless the step just done tripped the
// exact test (its output trip word, read after the barrier by every
// workgroup alike), in which case the launch ends there as the guarded
// per-step launches would have ended.  Same arithmetic per particle as
// k_step, so the same bits.
template <class R, class CT, int BLOCK>
__global__ void __launch_bounds__(BLOCK, sizeof(R) == 4 ? 4 : 3) k_step_loop(const LoopSet<R, CT> *__restrict__ sets,
                                                                            LoopArgs la) {
    const int64_t T = (sets[0].f.n + BLOCK - 1) / BLOCK;
    __shared__ BlockRecs<R, BLOCK> blk;
    for (int32_t s = 0; s < la.steps; s++) {
        const LoopSet<R, CT> &a = sets[s & 1];
        if (__hip_atomic_load(a.g.guard, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            if (blockIdx.x == 0 && threadIdx.x == 0) *a.g.guardOut = 1u;
            return;
        }
        uint32_t broke = 0;
        bool trip = false;
        for (int64_t v = blockIdx.x; v < T; v += gridDim.x) {
            const int64_t p = xcd_tile(v, T) * BLOCK + threadIdx.x;
            __syncthreads();   // the previous tile's records are read
            const int64_t wave0 = p - (threadIdx.x & 63);
            stage_records(a.r, wave0, a.f.n, blk);
            __syncthreads();
            if (p < a.f.n) {
                double cordN[3], diffN[3];
                step_particle<R, CT, BLOCK>(a.f, a.g, a.r, p, blk, blk.out[threadIdx.x >> 6], cordN, diffN, broke);
                trip |= guard_trips(a.g, p, cordN);
            }
        }
        if (trip) *a.g.guardOut = 1u;
        if (a.f.brokenCount) {
            broke = wave_sum_u32(broke);
            if ((threadIdx.x & 63) == 0 && broke)
                atomicAdd((unsigned long long *)a.f.brokenCount, (unsigned long long)broke);
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(a.g.stepsDone, 1u);
        grid_barrier(la.barrier, la.error, la.maxSpins);
        if (__hip_atomic_load(la.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    }
}

// Stores the two argument sets of a k_step_loop launch.
template <class R, class CT>
__global__ void k_store_loop_sets(LoopSet<R, CT> even, LoopSet<R, CT> odd, LoopSet<R, CT> *out) {
    if (threadIdx.x == 0) {
        out[0] = even;
        out[1] = odd;
    }
}

// The argument set of the step after `a`: the integrated state becomes the
// input, the trip words change roles.
template <class R, class CT>
LoopSet<R, CT> swapped_roles(const LoopSet<R, CT> &a) {
    LoopSet<R, CT> b = a;
    b.r.rec = a.r.recOut;
    b.r.recOut = const_cast<typename StepRecs<R>::Rec *>(a.r.rec);
    b.r.drec = a.r.drecOut;
    b.r.drecOut = const_cast<double *>(a.r.drec);
    b.r.tail = a.r.tailOut;
    b.r.tailOut = const_cast<MixedTail *>(a.r.tail);
    b.g.tx = a.g.otx;
    b.g.ty = a.g.oty;
    b.g.tz = a.g.otz;
    b.g.otx = const_cast<double *>(a.g.tx);
    b.g.oty = const_cast<double *>(a.g.ty);
    b.g.otz = const_cast<double *>(a.g.tz);
    b.f.tx = b.g.tx;
    b.f.ty = b.g.ty;
    b.f.tz = b.g.tz;
    b.g.guard = a.g.guardOut;
    b.g.guardOut = const_cast<uint32_t *>(a.g.guard);
    return b;
}

// SoA coordinates and Diff from the records (launch_unpack; an array that is
// not wanted is nullptr).  The tests also part the stores from the loads of the
// tail: without them the 1.7M particles of 256 blocks take 53.8 us, with them 49.4.
template <class Rec>
__global__ void __launch_bounds__(TPB) k_unpack_records(const Rec *__restrict__ rec,
                                                         const double *__restrict__ drec,
                                                         const MixedTail *__restrict__ tail, int64_t n, double *x,
                                                         double *y, double *z, double *d0, double *d1, double *d2,
                                                         double *d3, double *d4, double *d5) {
    const int64_t p = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (p >= n) return;
    const Rec P = rec[p];
    if (x) x[p] = P.x;
    if (y) y[p] = P.y;
    if (z) z[p] = P.z;
    double v[6];
    if constexpr (std::is_same<Rec, MixedRec>::value) {
        join_diff6(P, tail[p], drec, p, v);
    } else {
#pragma unroll
        for (int c = 0; c < 6; c++) v[c] = drec[p * 8 + c];
    }
    if (d0) d0[p] = v[0];
    if (d1) d1[p] = v[1];
    if (d2) d2[p] = v[2];
    if (d3) d3[p] = v[3];
    if (d4) d4[p] = v[4];
    if (d5) d5[p] = v[5];
}

// applyForce alone (hdm_integrate).  RECS: the records hold the state the
// particles come from and take the new one too, so that the next force and
// link break find them current (a pass that packs them again reads the whole
// state once more).
template <class R, bool RECS>
__global__ void __launch_bounds__(TPB) k_integrate(IntegArgs a, StepRecs<R> r, const R *__restrict__ f0,
                                                   const R *__restrict__ f1, const R *__restrict__ f2,
                                                   const R *__restrict__ f3, const R *__restrict__ f4,
                                                   const R *__restrict__ f5) {
    fetch_arguments<sizeof(a) + sizeof(r) + 6 * sizeof(f0)>();
    const int64_t i = xcd_block_index(gridDim.x) * TPB + threadIdx.x;
    __shared__ double2 stage[TPB / 64][32 * 5];
    if (i < a.n) {
        const double F[6] = {(double)f0[i], (double)f1[i], (double)f2[i], (double)f3[i], (double)f4[i], (double)f5[i]};
        double cord[3], theta[3], diff[6], radius;
        integrate_particle(a, i, F, cord, theta, diff, radius);
        if constexpr (RECS) {
            const int64_t wave0 = i - (threadIdx.x & 63);
            if (wave0 + 64 <= a.n)
                store_records_wave(r, wave0, threadIdx.x & 63, cord, theta, diff, radius, stage[threadIdx.x >> 6]);
            else
                store_records(r, i, cord, theta, diff, radius);
        }
    }
}

// Gather records of the current SoA state (hdm_run entry).
template <class R>
__global__ void __launch_bounds__(TPB) k_pack_records(const double *__restrict__ x, const double *__restrict__ y,
                                                       const double *__restrict__ z, const double *__restrict__ tx,
                                                       const double *__restrict__ ty, const double *__restrict__ tz,
                                                       const double *__restrict__ d0, const double *__restrict__ d1,
                                                       const double *__restrict__ d2, const double *__restrict__ d3,
                                                       const double *__restrict__ d4, const double *__restrict__ d5,
                                                       const double *__restrict__ radius, int64_t n,
                                                       StepRecs<R> r) {
    const int64_t p = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (p >= n) return;
    const double cord[3] = {x[p], y[p], z[p]};
    const double theta[3] = {tx[p], ty[p], tz[p]};
    const double diff[6] = {d0[p], d1[p], d2[p], d3[p], d4[p], d5[p]};
    store_records(r, p, cord, theta, diff, radius[p]);
}


// ---- link break --------------------------------------------------------------
struct BreakArgs {
    const double *x, *y, *z, *tx, *ty, *tz;
    const int32_t *A, *B;
    uint8_t *state;
    int32_t *slotLink, *slotOther;  // broken flag mirrored into both of the link's slots
    const int32_t *sidePos;
    const double *initialLen, *maxLoad;
    int64_t L;
    double bendBreak, scalarMaxLoad;
    uint64_t *counter;
};

// CombinedAccel::iterateLinks (CombinedAccel.h:200-235) applying
// HiDEMDefLinkBreakFunc (HiDEMDefaultFunctions.h:217-241); the strain is FP64
// in every precision form.
__global__ void __launch_bounds__(TPB) k_break(BreakArgs a) {
    fetch_arguments<sizeof(a)>();
    const int64_t l = (int64_t)blockIdx.x * TPB + threadIdx.x;
    uint32_t broke = 0;
    if (l < a.L && a.state[l] != 0) {
        const int32_t i = a.A[l], j = a.B[l];
        double xDist = a.x[i] - a.x[j];
        double yDist = a.y[i] - a.y[j];
        double zDist = a.z[i] - a.z[j];
        double stretchLength = sqrt((xDist * xDist) + (yDist * yDist) + (zDist * zDist));
        double bx = fabs(a.tx[i] - a.tx[j]);
        double by = fabs(a.ty[i] - a.ty[j]);
        double bz = fabs(a.tz[i] - a.tz[j]);
        double inner = (by < bz) ? bz : by;
        double maxBend = (bx < inner) ? inner : bx;
        double initialLen = a.initialLen[l];
        double load = (stretchLength - initialLen) / initialLen + a.bendBreak * maxBend;
        double maxLoad = a.maxLoad ? a.maxLoad[l] : a.scalarMaxLoad;
        if (load >= maxLoad) {
            a.state[l] = 0;
            const int32_t s0 = a.sidePos[2 * l], s1 = a.sidePos[2 * l + 1];
            a.slotLink[s0] |= SLOT_BROKEN;
            a.slotLink[s1] |= SLOT_BROKEN;
            a.slotOther[s0] |= SLOT_BROKEN;
            a.slotOther[s1] |= SLOT_BROKEN;
            broke = 1;
        }
    }
    broke = wave_sum_u32(broke);
    if ((threadIdx.x & 63) == 0 && broke && a.counter)
        atomicAdd((unsigned long long *)a.counter, (unsigned long long)broke);
}

// ---- skin reductions -----------------------------------------------------------
// HiDEMLib::getMaxDistOwned (HiDEMLib.h:424-461): max over particles of the
// signed Diff, starting from 0.0.  Bound by the read of the three arrays; three
// atomics per wave took 150 us at 2.1M particles, the workgroups' results and a
// fold 20.
__global__ void __launch_bounds__(TPB) k_skin_heuristic(const double *__restrict__ dx, const double *__restrict__ dy,
                                                         const double *__restrict__ dz, int64_t n, uint64_t *part) {
    double m[3] = {0.0, 0.0, 0.0};
    for (int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x; i < n; i += (int64_t)gridDim.x * TPB) {
        double v[3] = {dx[i], dy[i], dz[i]};
#pragma unroll
        for (int c = 0; c < 3; c++) m[c] = v[c] > m[c] ? v[c] : m[c];
    }
    block_max3(m);
    if (threadIdx.x == 0)
        for (int c = 0; c < 3; c++) part[c * RED_BLOCKS + blockIdx.x] = ordered_key(m[c]);
}

// Rebuild snapshot: the positions in FP64 and rounded to FP32.
__global__ void __launch_bounds__(TPB) k_snapshot(const double *__restrict__ x, const double *__restrict__ y,
                                                   const double *__restrict__ z, int64_t n, double *__restrict__ x0,
                                                   double *__restrict__ y0, double *__restrict__ z0,
                                                   float *__restrict__ x0f, float *__restrict__ y0f,
                                                   float *__restrict__ z0f) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const double a = x[i], b = y[i], c = z[i];
    x0[i] = a;
    y0[i] = b;
    z0[i] = c;
    x0f[i] = (float)a;
    y0f[i] = (float)b;
    z0f[i] = (float)c;
}

// Exact test: max over particles of |x - x0|^2 (FP64).
__global__ void __launch_bounds__(TPB) k_skin_exact(const double *__restrict__ x, const double *__restrict__ y,
                                                     const double *__restrict__ z, const double *__restrict__ x0,
                                                     const double *__restrict__ y0, const double *__restrict__ z0,
                                                     int64_t n, uint64_t *part) {
    double m2 = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x; i < n; i += (int64_t)gridDim.x * TPB) {
        double ddx = x[i] - x0[i], ddy = y[i] - y0[i], ddz = z[i] - z0[i];
        double d2 = ddx * ddx + ddy * ddy + ddz * ddz;
        m2 = d2 > m2 ? d2 : m2;
    }
    double m[3] = {m2, 0.0, 0.0};
    block_max3(m);
    if (threadIdx.x == 0) part[blockIdx.x] = ordered_key(m[0]);
}

inline int blocks_for(int64_t n) { return (int)((n + TPB - 1) / TPB); }
// State pointers for the integrator: in place (alt == nullptr) or from the
// current buffers into alt[0..11] (x, y, z, xTheta.., Diff0..5).
IntegArgs integ_args(Context &c, const hdm_integ_params &ip, bool partials, DevBuf *alt) {
    IntegArgs a;
    a.x = c.x.as<double>(); a.y = c.y.as<double>(); a.z = c.z.as<double>();
    a.tx = c.tx.as<double>(); a.ty = c.ty.as<double>(); a.tz = c.tz.as<double>();
    a.d0 = c.diff[0].as<double>(); a.d1 = c.diff[1].as<double>(); a.d2 = c.diff[2].as<double>();
    a.d3 = c.diff[3].as<double>(); a.d4 = c.diff[4].as<double>(); a.d5 = c.diff[5].as<double>();
    double *o[12];
    const double *in[12] = {a.x, a.y, a.z, a.tx, a.ty, a.tz, a.d0, a.d1, a.d2, a.d3, a.d4, a.d5};
    for (int k = 0; k < 12; k++) o[k] = alt ? alt[k].as<double>() : const_cast<double *>(in[k]);
    a.ox = o[0]; a.oy = o[1]; a.oz = o[2]; a.otx = o[3]; a.oty = o[4]; a.otz = o[5];
    a.od0 = o[6]; a.od1 = o[7]; a.od2 = o[8]; a.od3 = o[9]; a.od4 = o[10]; a.od5 = o[11];
    a.radius = c.radius.as<double>();
    a.type = c.type.as<uint8_t>();
    a.n = c.n;
    a.ip = ip;
    a.partials = partials ? c.skinPartials.as<double>() : nullptr;
    a.guard = nullptr;
    a.guardOut = nullptr;
    a.stepsDone = nullptr;
    a.guardThr = 0.0;
    a.x0 = c.x0.as<double>();
    a.y0 = c.y0.as<double>();
    a.z0 = c.z0.as<double>();
    a.x0f = c.x0f.as<float>();
    a.y0f = c.y0f.as<float>();
    a.z0f = c.z0f.as<float>();
    a.blockId = c.nBlocks > 0 ? c.blockId.as<int32_t>() : nullptr;
    a.blockWater = c.nBlocks > 0 ? c.blockWater.as<double>() : nullptr;
    a.mapMask = ip.variant == HDM_INTEG_GLACIER ? c.mapMask : 0;
    a.maps = a.mapMask ? c.mapDesc.as<MapDev>() : nullptr;
    return a;
}

template <class R, class CT, class FO>
ForceArgs<R, CT, FO> force_args(Context &c, const hdm_force_params &fp) {
    ForceArgs<R, CT, FO> a;
    a.radius = c.radius.as<double>();
    a.n = c.n;
    a.nbrCount = c.nbrCount.as<int32_t>(); a.nbr = c.nbr.as<int32_t>(); a.nbrWidth = c.maxNeigh;
    a.linkCount = c.linkCount.as<uint32_t>(); a.slotLink = c.slotLink.as<int32_t>();
    a.slotOther = c.slotOther.as<int32_t>(); a.linkWidth = c.maxLinks;
    a.ct = c.ct.as<CT>();
    a.f0 = c.force[0].as<FO>(); a.f1 = c.force[1].as<FO>(); a.f2 = c.force[2].as<FO>();
    a.f3 = c.force[3].as<FO>(); a.f4 = c.force[4].as<FO>(); a.f5 = c.force[5].as<FO>();
    a.fp = cast_params<R>(fp);
    a.breakCheck = 0;
    a.linkedContacts = c.nbrExcludesLinked ? 1 : 0;
    a.slotLinkW = c.slotLink.as<int32_t>();
    a.slotOtherW = c.slotOther.as<int32_t>();
    a.tx = c.tx.as<double>(); a.ty = c.ty.as<double>(); a.tz = c.tz.as<double>();
    a.initialLen = c.initialLen.as<double>();
    a.maxLoad = c.hasMaxLoad ? c.maxLoad.as<double>() : nullptr;
    a.state = c.state.as<uint8_t>();
    a.bendBreak = 0;
    a.scalarMaxLoad = 0;
    a.brokenCount = c.brokenCount.as<uint64_t>();
    return a;
}

constexpr int FINALIZE_BLOCKS = 32;

// Launch shapes of the fused step the autotuner chooses from.
struct StepShape {
    int block;
    const char *name;
};
constexpr StepShape kShapes[STEP_VARIANTS] = {
    {256, "wg256-xcd"},     {128, "wg128-xcd"},     {512, "wg512-xcd"}, {256, "wg256-linear"},
    {128, "wg128-xcd-occ"}, {256, "wg256-xcd-occ"}, {64, "wg64-xcd"}};
constexpr int kMinBlock = 64;

// States of at most two wave tiles per compute unit (32,768 particles on 256)
// run k_step_tile, unless the caller chose a shape: two of its six-wave
// workgroups are resident per CU.  Step time, tile form / workgroups of 64 of
// the lane form, us: intact block of 16,000 particles 12.7 / 23.6 FP64, 10.4 /
// 20.1 FP32; 31,200: 19.7 / 29.1, 12.5 / 19.6; with 20% of the links broken
// 23.5 / 34.3, 15.5 / 24.8.  Past the line a second round of tiles begins: 39,600
// 27.3 / 31.8, 18.0 / 20.5 (33.2 / 36.6, 23.7 / 27.1), 62,400 42.0 / 35.4, 29.2 /
// 25.5, so up to three tiles per unit the tile form would still be the faster
// one by 9-14%.
bool tile_step_pays(const Context &c) { return c.tiles() <= 2 * (int64_t)c.numCU; }

int64_t rows_for(int64_t n, int block) { return (n + block - 1) / block; }

// Rows for the rebuild-test partials (plus the finalize stage), and the guard
// words (zeroed once; the folding workgroup re-arms the ticket).
hipError_t ensure_partials(Context &c) {
    hipError_t e = c.skinPartials.ensure(sizeof(double) * 3 * ((size_t)rows_for(c.n, kMinBlock) + FINALIZE_BLOCKS));
    if (e != hipSuccess || c.guardState.ptr) return e;
    e = c.guardState.ensure(sizeof(uint32_t) * GUARD_WORDS);
    if (e != hipSuccess) return e;
    return launch_fill_u32(c.stream, c.guardState.as<uint32_t>(), 0u, GUARD_WORDS);
}

// k_skin_finalize over the rows of a launch of rows_for(n, block) workgroups.
hipError_t skin_finalize(Context &c, uint64_t *skin, int block) {
    FinalizeArgs f;
    f.rows = rows_for(c.n, block);
    f.partials = c.skinPartials.as<double>();
    f.stage = c.skinPartials.as<double>() + 3 * f.rows;
    f.ticket = c.guardState.as<uint32_t>() + GUARD_TICKET;
    f.skin = skin;
    hipLaunchKernelGGL(k_skin_finalize, dim3(FINALIZE_BLOCKS), dim3(TPB), 0, c.stream, f);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_guard_reset(Context &c) {
    hipError_t e = ensure_partials(c);
    if (e != hipSuccess) return e;
    return launch_fill_u32(c.stream, c.guardState.as<uint32_t>() + GUARD_FLAG, 0u, 3);
}

namespace {

// Bound on every Diff component under which a pair beyond the attraction
// range provably adds +-0 (pair_in_contact): the damping terms then stay
// below 1e300 (FP64) / 1e37 (FP32) in magnitude.  -1: no Diff qualifies.
double tame_bound(const Context &c, const hdm_force_params &fp) {
    if (!inert_skip_allowed(fp)) return -1.0;  // no Diff is tame: no pair is skipped
    double k = 1.0;
    const double a = fabs(fp.damping * fp.invDt), b = fabs(fp.dampingRotation * fp.invDt);
    k = a > k ? a : k;
    k = b > k ? b : k;
    if (!(k < 1e30)) return -1.0;  // also NaN
    return (c.prec == HDM_PREC_FP64 ? 1e299 : 1e36) / (4.0 * k);
}

template <class R>
StepRecs<R> step_recs(Context &c, double tame, const hdm_break_params *brk) {
    StepRecs<R> r;
    using Rec = typename StepRecs<R>::Rec;
    r.rec = c.rec.as<Rec>();
    r.drec = c.drec.as<double>();
    r.tail = c.dtail.as<MixedTail>();
    r.recOut = c.recAlt.as<Rec>();
    r.drecOut = c.drecAlt.as<double>();
    r.tailOut = c.dtailAlt.as<MixedTail>();
    r.tame = tame;
    r.slotThr = c.slotThr.as<uint16_t>();
    r.thrScale = c.thrScale;
    r.l0Max = c.l0Max;
    r.perLinkMaxLoad = c.hasMaxLoad ? 1 : 0;
    r.scalarMaxLoad = brk ? (float)brk->maxLoad : 0.0f;
    r.bendBreak = brk ? (float)brk->bendBreak : 0.0f;
    r.prefilter = (brk && brk->bendBreak >= 0.0 && brk->bendBreak < 1e30) ? 1 : 0;
    r.storeForce = 1;
    return r;
}

// The current records' buffers; alt: the other copy too (the fused step's).
hipError_t ensure_records(Context &c, bool alt) {
    const size_t n = (size_t)(c.n > 0 ? c.n : 1);
    const size_t recBytes = c.prec == HDM_PREC_FP64 ? sizeof(double4) : sizeof(MixedRec);
    const size_t drecBytes = sizeof(double) * (size_t)drec_stride(c.prec);
    hipError_t e = c.rec.ensure(recBytes * n);
    if (e == hipSuccess) e = c.drec.ensure(drecBytes * n);
    if (e == hipSuccess && c.prec != HDM_PREC_FP64) e = c.dtail.ensure(sizeof(MixedTail) * n);
    if (e != hipSuccess || !alt) return e;
    e = c.recAlt.ensure(recBytes * n);
    if (e == hipSuccess) e = c.drecAlt.ensure(drecBytes * n);
    if (e == hipSuccess && c.prec != HDM_PREC_FP64) e = c.dtailAlt.ensure(sizeof(MixedTail) * n);
    return e;
}

// step_recs whose output is the current records.
template <class R>
StepRecs<R> records_in_place(Context &c, double tame) {
    StepRecs<R> r = step_recs<R>(c, tame, nullptr);
    r.recOut = c.rec.as<typename StepRecs<R>::Rec>();
    r.drecOut = c.drec.as<double>();
    r.tailOut = c.dtail.as<MixedTail>();
    return r;
}

}  // namespace

hipError_t launch_pack_records(Context &c, double tame) {
    if (hipError_t se = sync_state(c); se != hipSuccess) return se;
    hipError_t e = ensure_records(c, false);
    if (e != hipSuccess || c.n == 0) return e;
    auto go = [&](auto r) {
        hipLaunchKernelGGL(k_pack_records, dim3(blocks_for(c.n)), dim3(TPB), 0, c.stream, c.x.as<double>(),
                           c.y.as<double>(), c.z.as<double>(), c.tx.as<double>(), c.ty.as<double>(),
                           c.tz.as<double>(), c.diff[0].as<double>(), c.diff[1].as<double>(), c.diff[2].as<double>(),
                           c.diff[3].as<double>(), c.diff[4].as<double>(), c.diff[5].as<double>(),
                           c.radius.as<double>(), c.n, r);
    };
    if (c.prec == HDM_PREC_FP64) go(records_in_place<double>(c, tame));
    else go(records_in_place<float>(c, tame));
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    c.recCurrent = true;
    c.recTame = tame;
    return hipSuccess;
}

hipError_t launch_force(Context &c, const hdm_force_params &fp) {
    if (c.n == 0) return hipSuccess;
    const double tame = tame_bound(c, fp);
    if (!c.recCurrent || c.recTame != tame) {
        hipError_t e = launch_pack_records(c, tame);
        if (e != hipSuccess) return e;
    }
    auto go = [&](auto f, auto r) {
        using R = typename decltype(r)::Real;
        if (tile_step_pays(c))
            hipLaunchKernelGGL((k_force_tile<R, R>), dim3((unsigned)c.tiles()), dim3(TILE_THREADS), 0, c.stream, f, r);
        else
            hipLaunchKernelGGL((k_force<R, R>), dim3(blocks_for(c.n)), dim3(TPB), 0, c.stream, f, r);
    };
    if (c.prec == HDM_PREC_FP64) go(force_args<double, double, double>(c, fp), step_recs<double>(c, tame, nullptr));
    else go(force_args<float, float, float>(c, fp), step_recs<float>(c, tame, nullptr));
    return hipGetLastError();
}

hipError_t launch_integrate(Context &c, const hdm_integ_params &ip) {
    if (hipError_t se = sync_state(c); se != hipSuccess) return se;
    if (c.n == 0) return hipSuccess;
    IntegArgs a = integ_args(c, ip, false, nullptr);
    auto go = [&](auto r) {
        using R = typename decltype(r)::Real;
        const dim3 grid(blocks_for(c.n));
        const R *fo[6];
        for (int k = 0; k < 6; k++) fo[k] = c.force[k].as<R>();
        if (c.recCurrent)
            hipLaunchKernelGGL((k_integrate<R, true>), grid, dim3(TPB), 0, c.stream, a, r, fo[0], fo[1], fo[2], fo[3],
                               fo[4], fo[5]);
        else
            hipLaunchKernelGGL((k_integrate<R, false>), grid, dim3(TPB), 0, c.stream, a, r, fo[0], fo[1], fo[2],
                               fo[3], fo[4], fo[5]);
    };
    if (c.prec == HDM_PREC_FP64) go(records_in_place<double>(c, c.recTame));
    else go(records_in_place<float>(c, c.recTame));
    return hipGetLastError();
}

void swap_step_state(Context &c) {
    c.guardCur ^= 1;
    swap_buf(c.tx, c.alt[3]);
    swap_buf(c.ty, c.alt[4]);
    swap_buf(c.tz, c.alt[5]);
    swap_buf(c.rec, c.recAlt);
    swap_buf(c.drec, c.drecAlt);
    swap_buf(c.dtail, c.dtailAlt);
}

hipError_t sync_state(Context &c) {
    if (!c.soaStale) return hipSuccess;
    c.soaStale = false;
    double *const own[9] = {c.x.as<double>(), c.y.as<double>(), c.z.as<double>(),
                            c.diff[0].as<double>(), c.diff[1].as<double>(), c.diff[2].as<double>(),
                            c.diff[3].as<double>(), c.diff[4].as<double>(), c.diff[5].as<double>()};
    return launch_unpack(c, own);
}

hipError_t launch_unpack(Context &c, double *const out[9]) {
    if (c.n == 0) return hipSuccess;
    auto go = [&](auto *rec) {
        using Rec = typename std::remove_pointer<decltype(rec)>::type;
        hipLaunchKernelGGL((k_unpack_records<Rec>), dim3(blocks_for(c.n)), dim3(TPB), 0, c.stream, rec,
                           c.drec.as<double>(), c.dtail.as<MixedTail>(), c.n, out[0], out[1], out[2], out[3], out[4], out[5],
                           out[6], out[7], out[8]);
    };
    if (c.prec == HDM_PREC_FP64) go(c.rec.as<double4>());
    else go(c.rec.as<MixedRec>());
    return hipGetLastError();
}

hipError_t launch_step(Context &c, const hdm_force_params &fp, const hdm_integ_params &ip, uint64_t *skin,
                       const hdm_break_params *brk, bool storeForce, const StepGuard *guard) {
    if (c.n == 0) return hipSuccess;
    const size_t b = sizeof(double) * (size_t)c.n;
    for (int k = 3; k < 6; k++) {
        hipError_t e = c.alt[k].ensure(b);
        if (e != hipSuccess) return e;
    }
    if (skin || guard) {
        hipError_t e = ensure_partials(c);
        if (e != hipSuccess) return e;
    }
    const double tame = tame_bound(c, fp);
    if (!c.recCurrent || c.recTame != tame) {
        hipError_t e = launch_pack_records(c, tame);
        if (e != hipSuccess) return e;
    }
    if (hipError_t e = ensure_records(c, true); e != hipSuccess) return e;
    IntegArgs g = integ_args(c, ip, skin && !guard, c.alt);
    if (guard) {
        uint32_t *words = c.guardState.as<uint32_t>();
        g.guard = words + GUARD_FLAG + c.guardCur;
        g.guardOut = words + GUARD_FLAG + (c.guardCur ^ 1);
        g.stepsDone = words + GUARD_STEPS;
        g.guardThr = guard->threshold;
    }
    const int v = step_form(c);
    const bool small = v == TILE_FORM;
    const int rowParticles = small ? 64 : kShapes[v].block;   // particles of a workgroup
    auto launch = [&](auto f, auto r) {
        r.storeForce = storeForce ? 1 : 0;
        if (brk && c.L > 0) {
            f.breakCheck = 1;
            f.bendBreak = brk->bendBreak;
            f.scalarMaxLoad = brk->maxLoad;
        }
        using A = decltype(f);
        using R = typename std::conditional<std::is_same<A, ForceArgs<double, double, double>>::value, double,
                                            float>::type;
        const dim3 grid((unsigned)rows_for(c.n, rowParticles));
        if (small) {
            hipLaunchKernelGGL((k_step_tile<R, R>), grid, dim3(TILE_THREADS), 0, c.stream, f, g, r);
            return;
        }
        switch (v) {
        case 0: hipLaunchKernelGGL((k_step<R, R, 256, true, false>), grid, dim3(256), 0, c.stream, f, g, r); break;
        case 1: hipLaunchKernelGGL((k_step<R, R, 128, true, false>), grid, dim3(128), 0, c.stream, f, g, r); break;
        case 2: hipLaunchKernelGGL((k_step<R, R, 512, true, false>), grid, dim3(512), 0, c.stream, f, g, r); break;
        case 3: hipLaunchKernelGGL((k_step<R, R, 256, false, false>), grid, dim3(256), 0, c.stream, f, g, r); break;
        case 4: hipLaunchKernelGGL((k_step<R, R, 128, true, true>), grid, dim3(128), 0, c.stream, f, g, r); break;
        case 5: hipLaunchKernelGGL((k_step<R, R, 256, true, true>), grid, dim3(256), 0, c.stream, f, g, r); break;
        default: hipLaunchKernelGGL((k_step<R, R, 64, true, false>), grid, dim3(64), 0, c.stream, f, g, r); break;
        }
    };
    if (c.prec == HDM_PREC_FP64) launch(force_args<double, double, double>(c, fp), step_recs<double>(c, tame, brk));
    else launch(force_args<float, float, float>(c, fp), step_recs<float>(c, tame, brk));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // the new state becomes current (records and rotations); the SoA
    // coordinates and Diff are unpacked on demand
    swap_step_state(c);
    c.soaStale = true;
    if (!skin || guard) return hipSuccess;
    return skin_finalize(c, skin, rowParticles);
}

hipError_t launch_break_records(Context &c, const hdm_break_params &bp, uint64_t *counter, int64_t guardedSteps) {
    if (counter) {
        hipError_t e = launch_fill_u64(c.stream, counter, 0ull, 1);
        if (e != hipSuccess) return e;
    }
    if (c.L == 0 || c.n == 0) return hipSuccess;
    // few particles: a thread per link (3.5 us on the 16k block, this walk 7.9),
    // where the SoA state is current too
    const bool guarded = guardedSteps >= 0;   // right after steps, so the records are current
    if (!guarded && (!c.recCurrent || (tile_step_pays(c) && !c.soaStale))) return launch_break(c, bp, counter);
    const uint32_t *done = guarded ? c.guardState.as<uint32_t>() + GUARD_STEPS : nullptr;
    hdm_force_params fp{};
    auto go = [&](auto f, auto r) {
        using A = decltype(f);
        using R = typename std::conditional<std::is_same<A, ForceArgs<double, double, double>>::value, double,
                                            float>::type;
        f.bendBreak = bp.bendBreak;
        f.scalarMaxLoad = bp.maxLoad;
        hipLaunchKernelGGL((k_break_recs<R>), dim3(blocks_for(c.n)), dim3(TPB), 0, c.stream, f, r, counter, done,
                           (uint32_t)(guarded ? guardedSteps : 0));
    };
    if (c.prec == HDM_PREC_FP64) go(force_args<double, double, double>(c, fp), step_recs<double>(c, c.recTame, &bp));
    else go(force_args<float, float, float>(c, fp), step_recs<float>(c, c.recTame, &bp));
    return hipGetLastError();
}

hipError_t launch_step_loop(Context &c, const hdm_force_params &fp, const hdm_integ_params &ip,
                            const hdm_break_params &brk, const StepGuard &guard, int32_t steps, bool *barrierFailed) {
    *barrierFailed = false;
    if (c.n == 0 || steps <= 0) return hipSuccess;
    if (!c.coopLaunch) return hipErrorNotSupported;
    const size_t b = sizeof(double) * (size_t)c.n;
    for (int k = 3; k < 6; k++) {
        hipError_t e = c.alt[k].ensure(b);
        if (e != hipSuccess) return e;
    }
    hipError_t e = ensure_partials(c);
    if (e != hipSuccess) return e;
    if (!c.loopBarrier.ptr) {
        e = c.loopBarrier.ensure(sizeof(uint32_t) * (BARRIER_WORDS + 1));
        if (e == hipSuccess) e = launch_fill_u32(c.stream, c.loopBarrier.as<uint32_t>(), 0u, BARRIER_WORDS + 1);
        if (e != hipSuccess) return e;
    }
    const double tame = tame_bound(c, fp);
    if (!c.recCurrent || c.recTame != tame) {
        e = launch_pack_records(c, tame);
        if (e != hipSuccess) return e;
    }
    e = ensure_records(c, true);
    if (e != hipSuccess) return e;
    IntegArgs g = integ_args(c, ip, false, c.alt);
    uint32_t *words = c.guardState.as<uint32_t>();
    g.guard = words + GUARD_FLAG + c.guardCur;
    g.guardOut = words + GUARD_FLAG + (c.guardCur ^ 1);
    g.stepsDone = words + GUARD_STEPS;
    g.guardThr = guard.threshold;
    LoopArgs la;
    la.steps = steps;
    la.barrier = c.loopBarrier.as<uint32_t>();
    la.error = la.barrier + BARRIER_WORDS;
    la.maxSpins = 1u << 22;   // seconds of waiting; a step takes milliseconds
    auto go = [&](auto f, auto r, const void *kernel) -> hipError_t {
        r.storeForce = 0;
        f.breakCheck = c.L > 0 ? 1 : 0;
        f.bendBreak = brk.bendBreak;
        f.scalarMaxLoad = brk.maxLoad;
        int perCU = 0;
        hipError_t e2 = hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, kernel, TPB, 0);
        if (e2 != hipSuccess) return e2;
        const int64_t tiles = (c.n + TPB - 1) / TPB;
        int64_t grid = (int64_t)perCU * (c.numCU > 0 ? c.numCU : 1);
        if (grid > tiles) grid = tiles;
        grid -= grid % 8;
        if (grid < 8) return hipErrorInvalidConfiguration;
        using Real = typename decltype(r)::Real;
        using CTT = typename decltype(f)::CTType;
        using Set = LoopSet<Real, CTT>;
        e2 = c.loopSets.ensure(2 * sizeof(Set));
        if (e2 != hipSuccess) return e2;
        Set *sets = static_cast<Set *>(c.loopSets.ptr);
        const Set even{f, g, r};
        hipLaunchKernelGGL((k_store_loop_sets<Real, CTT>), dim3(1), dim3(64), 0, c.stream, even, swapped_roles(even),
                           sets);
        e2 = hipGetLastError();
        if (e2 != hipSuccess) return e2;
        void *args[] = {&sets, &la};
        return hipLaunchCooperativeKernel(kernel, dim3((unsigned)grid), dim3(TPB), args, 0, c.stream);
    };
    if (c.prec == HDM_PREC_FP64)
        e = go(force_args<double, double, double>(c, fp), step_recs<double>(c, tame, &brk),
               reinterpret_cast<const void *>(&k_step_loop<double, double, TPB>));
    else
        e = go(force_args<float, float, float>(c, fp), step_recs<float>(c, tame, &brk),
               reinterpret_cast<const void *>(&k_step_loop<float, float, TPB>));
    if (e != hipSuccess) return e;
    // the launch swapped the roles `steps` times (the host undoes the ones a
    // trip skipped, as for skipped per-step launches)
    if (steps & 1) swap_step_state(c);
    c.soaStale = true;
    uint32_t err = 0;
    e = hipMemcpyAsync(&err, la.error, sizeof(err), hipMemcpyDeviceToHost, c.stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c.stream);
    if (e != hipSuccess) return e;
    if (err) {   // re-arm the barrier words for the next launch
        *barrierFailed = true;
        return launch_fill_u32(c.stream, c.loopBarrier.as<uint32_t>(), 0u, BARRIER_WORDS + 1);
    }
    return hipSuccess;
}

// Without a shape from the caller or the autotuner: 64 particles per workgroup
// while 256 would leave a compute unit at most four of them (262,144 particles
// on 256), so that what is there spreads evenly; above, 256, which share more
// records in LDS.  64 / 256, us per step: rubble of 134k particles 68.9 / 74.2
// FP64, 48.4 / 49.8 FP32; intact block of 50k 34.5 / 34.8, 24.9 / 25.3; of 291k
// 116.7 / 116.2, 63.4 / 63.6.  The larger states take their workgroups in
// launch order: all XCDs then stream neighbouring lines at a time, which is
// worth more than the 8% of traffic that ranges of their own save.  Launch
// order / a range per XCD, us: 8M slab 1403 / 1433 FP32, FP64 equal (2423 / 2440
// and 2436 / 2432); 256 blocks of 1.7M particles 322 / 329 FP32; 2M slab 362 /
// 372 FP32; 291k equal.
int step_form(const Context &c) {
    if (!c.shapeGiven && c.n > 0 && tile_step_pays(c)) return TILE_FORM;
    if (c.shapeChosen && c.stepVariant >= 0 && c.stepVariant < STEP_VARIANTS) return c.stepVariant;
    return c.n <= 4 * 256 * (int64_t)c.numCU ? 6 : 3;
}

const char *step_variant_name(int v) {
    if (v == TILE_FORM) return "tile64";
    return (v >= 0 && v < STEP_VARIANTS) ? kShapes[v].name : "?";
}

// The fastest shape.
int pick_step_variant(const double ms[STEP_VARIANTS]) {
    int best = 0;
    for (int v = 1; v < STEP_VARIANTS; v++)
        if (ms[v] < ms[best]) best = v;
    return best;
}

hipError_t launch_break(Context &c, const hdm_break_params &bp, uint64_t *counter) {
    if (hipError_t se = sync_state(c); se != hipSuccess) return se;
    if (c.L == 0) return hipSuccess;
    BreakArgs a;
    a.x = c.x.as<double>(); a.y = c.y.as<double>(); a.z = c.z.as<double>();
    a.tx = c.tx.as<double>(); a.ty = c.ty.as<double>(); a.tz = c.tz.as<double>();
    a.A = c.la.as<int32_t>(); a.B = c.lb.as<int32_t>();
    a.state = c.state.as<uint8_t>();
    a.initialLen = c.initialLen.as<double>();
    a.maxLoad = c.hasMaxLoad ? c.maxLoad.as<double>() : nullptr;
    a.slotLink = c.slotLink.as<int32_t>();
    a.slotOther = c.slotOther.as<int32_t>();
    a.sidePos = c.sidePos.as<int32_t>();
    a.L = c.L;
    a.bendBreak = bp.bendBreak;
    a.scalarMaxLoad = bp.maxLoad;
    a.counter = counter;
    hipLaunchKernelGGL(k_break, dim3(blocks_for(c.L)), dim3(TPB), 0, c.stream, a);
    return hipGetLastError();
}

hipError_t launch_skin_heuristic(Context &c, uint64_t *out3) {
    if (hipError_t se = sync_state(c); se != hipSuccess) return se;
    const int grid = reduce_blocks(c, c.n);
    hipLaunchKernelGGL(k_skin_heuristic, dim3(grid), dim3(TPB), 0, c.stream, c.diff[0].as<double>(),
                       c.diff[1].as<double>(), c.diff[2].as<double>(), c.n, c.red.as<uint64_t>() + RED_PARTS);
    return launch_fold(c, grid, 3, 0u, out3);
}

hipError_t launch_skin_exact(Context &c, uint64_t *out1) {
    if (hipError_t se = sync_state(c); se != hipSuccess) return se;
    const int grid = reduce_blocks(c, c.n);
    hipLaunchKernelGGL(k_skin_exact, dim3(grid), dim3(TPB), 0, c.stream, c.x.as<double>(), c.y.as<double>(),
                       c.z.as<double>(), c.x0.as<double>(), c.y0.as<double>(), c.z0.as<double>(), c.n,
                       c.red.as<uint64_t>() + RED_PARTS);
    return launch_fold(c, grid, 1, 0u, out1);
}

hipError_t launch_snapshot(Context &c) {
    if (hipError_t se = sync_state(c); se != hipSuccess) return se;
    if (c.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_snapshot, dim3(blocks_for(c.n)), dim3(TPB), 0, c.stream, c.x.as<double>(), c.y.as<double>(),
                       c.z.as<double>(), c.n, c.x0.as<double>(), c.y0.as<double>(), c.z0.as<double>(),
                       c.x0f.as<float>(), c.y0f.as<float>(), c.z0f.as<float>());
    return hipGetLastError();
}

}  // namespace hdm
