/*
 * Device-resident particle host for benchmarks and long runs: what OpenMM's Context and
 * VerletIntegrator do around the LBMForce kernel in the reference, kept on the GPU so that
 * a coupled step crosses no PCIe.  Per step, on the context's stream:
 *   lbm_begin_step_device -> zero forces -> extra forces (wall potential, harmonic bonds)
 *   -> lbm_execute_device (adds the coupling forces) -> leapfrog Verlet update
 *      v(t+dt/2) = v(t-dt/2) + dt F(t)/m,  x(t+dt) = x(t) + dt v(t+dt/2).
 * Between two steps of one call the update, the next step's reflection and its other forces are work-groups of a launch of
 * the lattice step, or one launch (lbm_between.h).
 * The extra forces are those of the benchmark configurations: a repulsive wall potential
 * eps[(sigma/d1)^12 + (sigma/d2)^12] between two planes z = zlo and z = zhi (the pattern of
 * the reference's examples/cocomo/shear.py:291-310), and harmonic bonds k/2 (r - r0)^2 with the
 * minimum image (bead chains, at most two bonds per particle), summed per particle in a fixed order.
 */
#include "lbm_between.h"
#include <stdexcept>
#include <utility>
#include <vector>

extern "C" hipStream_t lbm_internal_stream(lbm_context* c);

namespace {

struct MD {
    int n = 0;
    double dt = 0;
    double* pos = nullptr;
    double* vel = nullptr;
    double* force = nullptr;
    // The arrays that the merged launch between two steps writes (it reads the others); the two sets swap there.
    double* nextPos = nullptr;
    double* nextVel = nullptr;
    double* nextForce = nullptr;
    double* invMass = nullptr;
    bool wall = false;
    double eps = 0, sigma = 0, zlo = 0, zhi = 0;
    int numBonds = 0;
    int* bonds = nullptr;
    double bondK = 0, bondR0 = 0;
    double box[3] = {0, 0, 0};
};

thread_local std::string g_err;

using lbm::OtherForces;
using lbm::BetweenSteps;

/* The other forces, written (not added) for every particle. */
__global__ void __launch_bounds__(lbm::BLOCK) otherForces(const double* __restrict__ pos, double* __restrict__ f, int n,
        OtherForces o) {
    int i = blockIdx.x*lbm::BLOCK + threadIdx.x;
    if (i >= n)
        return;
    double x[3] = {pos[3*(size_t) i], pos[3*(size_t) i + 1], pos[3*(size_t) i + 2]}, acc[3];
    lbm::otherForcesOn(i, x, o, [&](int j, double xj[3]) {
        for (int a = 0; a < 3; a++)
            xj[a] = pos[3*(size_t) j + a];
    }, acc);
    for (int a = 0; a < 3; a++)
        f[3*(size_t) i + a] = acc[a];
}

__global__ void __launch_bounds__(lbm::BLOCK) verlet(double* __restrict__ pos, double* __restrict__ vel,
        const double* __restrict__ f, const double* __restrict__ invMass, int n, double dt) {
    int i = blockIdx.x*lbm::BLOCK + threadIdx.x;
    if (i >= n)
        return;
    for (int a = 0; a < 3; a++) {
        size_t k = 3*(size_t) i + a;
        double v = lbm::newVelocity(vel[k], f[k], invMass[i], dt);
        vel[k] = v;
        pos[k] = lbm::newPosition(pos[k], v, dt);
    }
}

/*
 * The work between two steps in a launch of its own, where no launch of the lattice step takes it.  The update, the
 * reflection and the other forces are each bound by their launch (~5 us beside a large lattice pass, 2 us beside a small one),
 * not by their work: in one launch, a step of 64 beads in 32^3 22.4 -> 20.0 us, of 100,000 chain beads in 128^3 318 -> 310 us.
 */
template <bool REFLECT>
__global__ void __launch_bounds__(lbm::BLOCK) particlesBetween(BetweenSteps b) {
    lbm::betweenSteps<REFLECT, lbm::BLOCK>(b, (int) gridDim.x);
}

void hipCheck(hipError_t e) {
    if (e != hipSuccess)
        throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e));
}

}  // namespace

extern "C" {

typedef struct lbm_md_system lbm_md_system;

const char* lbm_md_last_error(void) {
    return g_err.c_str();
}

int lbm_md_create(int n, const double* masses, const double* positions, const double* velocities, double dt,
        lbm_md_system** out) {
    MD* md = new MD();
    try {
        md->n = n;
        md->dt = dt;
        size_t bytes = 3*sizeof(double)*(size_t) n;
        hipCheck(hipMalloc(&md->pos, bytes));
        hipCheck(hipMalloc(&md->vel, bytes));
        hipCheck(hipMalloc(&md->force, bytes));
        hipCheck(hipMalloc(&md->nextPos, bytes));
        hipCheck(hipMalloc(&md->nextVel, bytes));
        hipCheck(hipMalloc(&md->nextForce, bytes));
        hipCheck(hipMalloc(&md->invMass, sizeof(double)*(size_t) n));
        std::vector<double> inv(n);
        for (int i = 0; i < n; i++)
            inv[i] = masses[i] > 0 ? 1.0/masses[i] : 0.0;
        hipCheck(hipMemcpy(md->pos, positions, bytes, hipMemcpyHostToDevice));
        hipCheck(hipMemcpy(md->vel, velocities, bytes, hipMemcpyHostToDevice));
        hipCheck(hipMemcpy(md->invMass, inv.data(), sizeof(double)*(size_t) n, hipMemcpyHostToDevice));
    }
    catch (const std::exception& e) {
        g_err = e.what();
        delete md;
        return LBM_ERROR_RUNTIME;
    }
    *out = (lbm_md_system*) md;
    return LBM_OK;
}

int lbm_md_set_wall_potential(lbm_md_system* s, double eps, double sigma, double zlo, double zhi) {
    MD* md = (MD*) s;
    md->wall = true;
    md->eps = eps;
    md->sigma = sigma;
    md->zlo = zlo;
    md->zhi = zhi;
    return LBM_OK;
}

int lbm_md_set_bonds(lbm_md_system* s, const int* pairs, int numBonds, double k, double r0, const double box[3]) {
    MD* md = (MD*) s;
    try {
        if (md->bonds)
            hipCheck(hipFree(md->bonds));
        md->bonds = nullptr;
        md->numBonds = numBonds;
        if (numBonds > 0) {
            std::vector<int> partners(2*(size_t) md->n, -1);
            for (int b = 0; b < numBonds; b++) {
                int i = pairs[2*b], j = pairs[2*b + 1];
                if (i < 0 || j < 0 || i >= md->n || j >= md->n)
                    throw std::runtime_error("lbm_md_set_bonds: particle index out of range");
                for (int end = 0; end < 2; end++) {
                    int a = end == 0 ? i : j, other = end == 0 ? j : i;
                    int slot = partners[2*(size_t) a] < 0 ? 0 : partners[2*(size_t) a + 1] < 0 ? 1 : -1;
                    if (slot < 0)
                        throw std::runtime_error("lbm_md_set_bonds: a particle has more than two bonds (chains only)");
                    partners[2*(size_t) a + slot] = other;
                }
            }
            hipCheck(hipMalloc(&md->bonds, partners.size()*sizeof(int)));
            hipCheck(hipMemcpy(md->bonds, partners.data(), partners.size()*sizeof(int), hipMemcpyHostToDevice));
        }
        md->bondK = k;
        md->bondR0 = r0;
        for (int a = 0; a < 3; a++)
            md->box[a] = box[a];
    }
    catch (const std::exception& e) {
        g_err = e.what();
        return LBM_ERROR_RUNTIME;
    }
    return LBM_OK;
}

/* Run numSteps integration steps starting at step count step0. */
int lbm_md_step(lbm_md_system* s, lbm_context* ctx, int64_t step0, int numSteps) {
    MD* md = (MD*) s;
    hipStream_t stream = lbm_internal_stream(ctx);
    const int grid = (md->n + lbm::BLOCK - 1)/lbm::BLOCK;
    OtherForces other = {md->wall ? 1 : 0, md->eps, md->sigma, md->zlo, md->zhi, md->numBonds > 0 ? md->bonds : nullptr,
                         md->bondK, md->bondR0, {md->box[0], md->box[1], md->box[2]}};
    bool begun = false;              // the merged launch of the previous step has begun this one
    for (int t = 0; t < numSteps; t++) {
        int64_t step = step0 + t;
        int status = LBM_OK;
        if (begun)
            lbm_internal_begin_reflected(ctx, step);
        else {
            status = lbm_begin_step_device(ctx, step, md->pos, md->vel);
            if (status != LBM_OK) {
                g_err = lbm_last_error();
                return status;
            }
            otherForces<<<grid, lbm::BLOCK, 0, stream>>>(md->pos, md->force, md->n, other);
        }
        BetweenSteps between;
        begun = t + 1 < numSteps && lbm_internal_reflection(ctx, step + 1, md->n, between.reflection);
        if (begun) {
            between.pos = md->pos;
            between.vel = md->vel;
            between.force = md->force;
            between.invMass = md->invMass;
            between.n = md->n;
            between.dt = md->dt;
            between.other = other;
            between.posOut = md->nextPos;
            between.velOut = md->nextVel;
            between.forceOut = md->nextForce;
            lbm_internal_offer_between(ctx, &between);
        }
        status = lbm_execute_device(ctx, step, 1, md->pos, md->vel, md->force);
        if (status != LBM_OK) {
            g_err = lbm_last_error();
            return status;
        }
        if (begun) {
            if (!between.taken) {
                if (between.reflection.mask != nullptr)
                    particlesBetween<true><<<grid, lbm::BLOCK, 0, stream>>>(between);
                else
                    particlesBetween<false><<<grid, lbm::BLOCK, 0, stream>>>(between);
            }
            std::swap(md->pos, md->nextPos);
            std::swap(md->vel, md->nextVel);
            std::swap(md->force, md->nextForce);
        }
        else
            verlet<<<grid, lbm::BLOCK, 0, stream>>>(md->pos, md->vel, md->force, md->invMass, md->n, md->dt);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            g_err = hipGetErrorString(e);
            return LBM_ERROR_RUNTIME;
        }
    }
    return LBM_OK;
}

int lbm_md_get(lbm_md_system* s, lbm_context* ctx, double* positions, double* velocities) {
    MD* md = (MD*) s;
    hipStream_t stream = lbm_internal_stream(ctx);
    size_t bytes = 3*sizeof(double)*(size_t) md->n;
    if (hipStreamSynchronize(stream) != hipSuccess)
        return LBM_ERROR_RUNTIME;
    if (positions && hipMemcpy(positions, md->pos, bytes, hipMemcpyDeviceToHost) != hipSuccess)
        return LBM_ERROR_RUNTIME;
    if (velocities && hipMemcpy(velocities, md->vel, bytes, hipMemcpyDeviceToHost) != hipSuccess)
        return LBM_ERROR_RUNTIME;
    return LBM_OK;
}

int lbm_md_destroy(lbm_md_system* s) {
    MD* md = (MD*) s;
    if (!md)
        return LBM_OK;
    void* bufs[] = {md->pos, md->vel, md->force, md->nextPos, md->nextVel, md->nextForce, md->invMass, md->bonds};
    for (void* b : bufs)
        if (b)
            (void) hipFree(b);
    delete md;
    return LBM_OK;
}

}  // extern "C"
