/*
 * What lies between two lattice steps for the particles of the device-resident host (lbm_harness.hip): the leapfrog update
 * of the step that ends, the reflection at solid nodes that begins the next one and its other forces, as the work of some
 * work-groups of a launch: a kernel of their own, or those in front of the lattice pass or of the bounce-back, which touch
 * other memory.  It reads one set of particle arrays and writes the other: a bonded particle needs its partners' new
 * positions, which it forms again from their old values.
 */
#pragma once

#include "lbm_coupling.h"

namespace lbm {

/* The forces of the System other than the LBMForce. */
struct OtherForces {
    int wall;
    double eps, sigma, zlo, zhi;
    const int* partners;          // [particle][2], -1: none; nullptr without bonds
    double k, r0;
    double box[3];
};

struct BetweenSteps {
    const double* pos = nullptr;
    const double* vel = nullptr;
    const double* force = nullptr;
    const double* invMass = nullptr;
    int n = 0;
    double dt = 0;
    OtherForces other;
    StepReflection reflection;
    int busyOffset = 0, busyCount = 0;      // wall partial sums that the launch's other work-groups write
    double* posOut = nullptr;
    double* velOut = nullptr;
    double* forceOut = nullptr;
    bool taken = false;                     // host: a launch of the lattice step included it
};

/* Those on particle i at x: the repulsive walls U = eps[(s/d1)^12 + (s/d2)^12] along z (when set) plus the harmonic bonds
   to the (at most two) chain partners, in that order.  partnerAt(j, xj): the position of particle j. */
template <typename F>
__device__ __forceinline__ void otherForcesOn(int i, const double x[3], const OtherForces& o, F&& partnerAt, double acc[3]) {
    acc[0] = acc[1] = acc[2] = 0;
    if (o.wall) {
        double z = x[2];
        double d1 = z - o.zlo, d2 = o.zhi - z;
        // -dU/dz = 12 eps s^12/d1^13 - 12 eps s^12/d2^13.
        double s1 = o.sigma/d1, s2 = o.sigma/d2;
        double s1_12 = s1*s1*s1*s1*s1*s1*s1*s1*s1*s1*s1*s1, s2_12 = s2*s2*s2*s2*s2*s2*s2*s2*s2*s2*s2*s2;
        acc[2] = 12.0*o.eps*(s1_12/d1 - s2_12/d2);
    }
    if (o.partners != nullptr) {
        double b[3] = {0, 0, 0};
        for (int p = 0; p < 2; p++) {
            int j = o.partners[2*i + p];
            if (j < 0)
                continue;
            double d[3], xj[3];
            partnerAt(j, xj);
            for (int a = 0; a < 3; a++) {
                d[a] = xj[a] - x[a];
                d[a] -= o.box[a]*rint(d[a]/o.box[a]);
            }
            double r = sqrt(d[0]*d[0] + d[1]*d[1] + d[2]*d[2]);
            double s = r > 0 ? o.k*(r - o.r0)/r : 0.0;
            for (int a = 0; a < 3; a++)
                b[a] += s*d[a];
        }
        for (int a = 0; a < 3; a++)
            acc[a] += b[a];
    }
}

/* One component of the leapfrog update, its roundings written out: a partner's new position is formed again, and every
   copy has to have the same bits. */
__device__ __forceinline__ double newVelocity(double v, double f, double invMass, double dt) {
    return fma(dt*f, invMass, v);
}
__device__ __forceinline__ double newPosition(double x, double v, double dt) {
    return fma(dt, v, x);
}

/* Work-group blockIdx.x of the first `blocks` of a launch, THREADS particles; every thread of it calls this. */
template <bool REFLECT, int THREADS>
__device__ __forceinline__ void betweenSteps(const BetweenSteps& b, int blocks) {
    if constexpr (REFLECT)
        clearOtherPartials<THREADS>(b.reflection.partials, b.reflection.count, b.reflection.ownOffset, blocks, b.busyOffset,
                b.busyCount);
    const int i = blockIdx.x*THREADS + threadIdx.x;
    double wallAcc[3] = {0, 0, 0};
    if (i < b.n) {
        auto moved = [&](int j, double x[3], double v[3]) {
            for (int a = 0; a < 3; a++) {
                const size_t k = 3*(size_t) j + a;
                v[a] = newVelocity(b.vel[k], b.force[k], b.invMass[j], b.dt);
                x[a] = newPosition(b.pos[k], v[a], b.dt);
            }
        };
        double x[3], v[3], acc[3];
        moved(i, x, v);
        if constexpr (REFLECT)
            reflectParticle(x, v, b.reflection.mass[i], b.reflection.mask, b.reflection.args, wallAcc);
        otherForcesOn(i, x, b.other, [&](int j, double xj[3]) {
            double vj[3];
            moved(j, xj, vj);
        }, acc);
        for (int a = 0; a < 3; a++) {
            const size_t k = 3*(size_t) i + a;
            b.posOut[k] = x[a];
            b.velOut[k] = v[a];
            b.forceOut[k] = acc[a];
        }
    }
    if constexpr (REFLECT)
        storeWallPartial<THREADS>(wallAcc, b.reflection.partials + 3*(size_t) b.reflection.ownOffset);
}

}  // namespace lbm

/* For the particle host: offers the work between step and step + 1 to the next lbm_execute_device, which sets b->taken when
   one of its launches includes it, and forgets it. */
void lbm_internal_offer_between(lbm_context* c, lbm::BetweenSteps* b);
