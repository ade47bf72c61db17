/*
 * The centred drag (LBMForce::Centered) on gfx950.
 *
 * With h = 1/2, a = gamma h, the velocity of a particle at the time of the force v~ = v(t - h)/(dx/dt) + h Fc/m (Fc:
 * the other forces of the System, read from the force array before the coupling adds to it) and the fluid velocity
 * u~ = (j + h rho g)/rho of a node:
 *
 *  - nearest node (ReferenceLBMKernels.cpp:555-641): the particles of one node are coupled to each other only.  With M,
 *    P~ = sum m v~ and R the sums of their masses, momenta and random forces,
 *        S = [-gamma (P~ - M u~) + R]/(1 + a + a M/rho),  u_c = u~ - h S/rho,  F_k = [-gamma m_k (v~_k - u_c) + R_k]/(1 + a),
 *    and the node receives -S (a solid node is a wall at rest: u_c = 0).  The particles are sorted by node (a stable
 *    radix sort of the node keys, so a node's particles stay in particle order) and the first particle of each run
 *    sums them in that order and solves its node: the sums have the reference's order.
 *  - stencil (ReferenceLBMKernels.cpp:726-901): (1 + a)/m_k F_k + a sum_l K_kl F_l = b_k/m_k with
 *    K_kl = sum_j xi_jk xi_jl/rho_j and b_k = -gamma m_k (v~_k - sum_j xi_jk u~_j) + R_k, solved per component by
 *    conjugate gradients preconditioned with the diagonal, from the diagonal solution, to a residual of 1e-13 of the
 *    right-hand side.  A product spreads the vector onto the nodes and interpolates it back; the spread accumulates in
 *    64-bit fixed point with a scale set from the largest entry of the vector (2^52 / that entry), so the sums are
 *    exact to 2^-52 of it and independent of the order of the atomics.  With sparse particles only the slots at nodes
 *    that several slots share are spread; a slot alone at its node takes its own particle's w x directly.  Two arrays
 *    of node sums serve the products in turn, each gather clearing the previous product's.  Dot products reduce over a fixed grid in a
 *    fixed order.  The device tests the residual after every iteration and the kernels of later iterations then skip
 *    their work; the host enqueues as many iterations as the previous solve took before it reads the residual, then
 *    one at a time, so the iterations and results are those of a check after every iteration without a round trip
 *    to the host for each.
 *
 *    Where the lattice is periodic and the particles have few neighbours (CgRows) the matrix is formed instead, once per
 *    solve: row k holds K_kl of the particles l whose stencils share a node with k's, 11 on average for 56,320 Keys
 *    particles in 120^3 against 64 slots, and a product reads its row and its neighbours' entries, no node sums.
 *
 * The reaction goes into the same fixed-point accumulators as the explicit drag (consumed by the fused pass; with the
 * split, stored where no other slot reaches the node, since those accumulators are zero, and added atomically where
 * several do), and into the wall partial sums at solid nodes.
 */
#include "lbm_coupling.h"
#include <hipcub/hipcub.hpp>
#include <cmath>
#include <stdexcept>

namespace lbm {

namespace {

constexpr int RED_BLOCKS = 256;          // fixed grid of the CG reductions
constexpr double CG_TOLERANCE = 1e-13;
constexpr int CG_MAX_ITERATIONS = 1000;

/* Device scalars of the conjugate gradients. */
enum Scalar {
    RZ = 0, RZ_NEW = 3, RR = 6, NORM = 9, DAD = 12, ALPHA = 15, BETA = 18, SCALE = 21, INV_SCALE = 22,
    RZ_SLOT = RZ_NEW - RZ,   // with matrix rows r.z of iteration t is at RZ + RZ_SLOT (t mod 2)
    DONE = 23,        // 1 once the residual is within tolerance: the remaining iterations' kernels return at once
    ITERS = 24,       // iterations run in this solve
    OVERFLOWED = 25,  // the host's copy of CgRows::overflow
    NUM_SCALARS = 26
};

void check(hipError_t e, const char* what) {
    if (e != hipSuccess)
        throw std::runtime_error(std::string("centred drag: ") + what + ": " + hipGetErrorString(e));
}

template <typename T>
T* alloc(size_t count) {
    void* p = nullptr;
    check(hipMalloc(&p, std::max<size_t>(count, 1)*sizeof(T)), "hipMalloc");
    return (T*) p;
}

/* v~ and the random force R of coupled particle i, lattice units (ReferenceLBMKernels.cpp:577-585). */
__device__ __forceinline__ void particleKnowns(const double* vel, const double* fc, double m, uint32_t i,
        const ParticleArgs& a, double known[3], double random[3]) {
    double noise[4] = {0, 0, 0, 0};
    if (a.randomForce)
        particleNoise(i, a, noise);
    double amp = sqrt(2.0*a.gamma*m*a.kT);
    for (int k = 0; k < 3; k++) {
        known[k] = vel[k]*(1.0/a.velocityScale) + (fc ? fc[k] : 0.0)*(0.5/(m*a.forceScale));
        random[k] = a.randomForce ? noise[k]*amp : 0.0;
    }
}

/* The reaction r on a node: into its fixed-point accumulators, or to the wall on a solid node.  Returns whether an
   accumulator changed (the node is then flagged in the touched mask by markTouched). */
__device__ __forceinline__ bool addReaction(uint32_t node, bool solid, const double r[3], const ParticleArgs& a,
        unsigned long long* reactionFixed, double wallAcc[3]) {
    if (solid) {
        for (int k = 0; k < 3; k++)
            wallAcc[k] += r[k];          // lattice momentum; the host converts the wall partials
        return false;
    }
    bool any = false;
    for (int k = 0; k < 3; k++) {
        if (!reactionInRange(r[k], a.overflow))
            continue;
        long long fixed = llrint(r[k]*FIXED_SCALE);
        if (fixed != 0) {
            atomicAdd(reactionFixed + reactionIndex(node, k, a.g.n, a.reactionPlanes), (unsigned long long) fixed);
            any = true;
        }
    }
    return any;
}

/* addReaction for a fluid node that no other slot of the step reaches (the CG split's unshared nodes): its
   accumulators are zero (the lattice pass consumed and cleared them), so a store puts the same bits as the atomic add. */
__device__ __forceinline__ bool storeReaction(uint32_t node, const double r[3], const ParticleArgs& a,
        unsigned long long* reactionFixed) {
    bool any = false;
    for (int k = 0; k < 3; k++) {
        if (!reactionInRange(r[k], a.overflow))
            continue;
        long long fixed = llrint(r[k]*FIXED_SCALE);
        if (fixed != 0) {
            reactionFixed[reactionIndex(node, k, a.g.n, a.reactionPlanes)] = (unsigned long long) fixed;
            any = true;
        }
    }
    return any;
}

__device__ __forceinline__ void blockPartials(const double acc[3], double* partials) {
    if (partials != nullptr)
        storeWallPartial<BLOCK>(acc, partials);
}

/* ---------------------------------------------------------------------------------------------------------------- */
/* Nearest node.                                                                                                     */
/* ---------------------------------------------------------------------------------------------------------------- */
__global__ void __launch_bounds__(BLOCK) centredKeys(const double* __restrict__ positions,
        const int* __restrict__ particles, ParticleArgs a, uint32_t* __restrict__ keys, int* __restrict__ values) {
    int i = blockIdx.x*BLOCK + threadIdx.x;
    if (i >= a.numParticles)
        return;
    keys[i] = nearestNodeOf(positions + 3*(size_t) particles[i], a);
    values[i] = i;
}

template <typename S>
__global__ void __launch_bounds__(BLOCK) centredNearest(const S* __restrict__ src, const uint32_t* __restrict__ mask,
        const double* __restrict__ velocities, const double* __restrict__ otherForces, const int* __restrict__ particles,
        const double* __restrict__ mass, const double* __restrict__ ucm, ParticleArgs a, double gx, double gy, double gz,
        const uint32_t* __restrict__ sortedKeys, const int* __restrict__ sortedIdx, double* __restrict__ particleForce,
        unsigned long long* __restrict__ reactionFixed, uint32_t* __restrict__ touched, double* __restrict__ partials) {
    const double h = 0.5, gamma = a.gamma, aa = a.gamma*h;
    double wallAcc[3] = {0, 0, 0};
    int s = blockIdx.x*BLOCK + threadIdx.x;
    if (s < a.numParticles && (s == 0 || sortedKeys[s] != sortedKeys[s - 1])) {
        uint32_t node = sortedKeys[s];
        double M = 0, P[3] = {0, 0, 0}, R[3] = {0, 0, 0};
        int e = s;
        for (; e < a.numParticles && sortedKeys[e] == node; e++) {
            int i = sortedIdx[e];
            int part = particles[i];
            double known[3], random[3];
            particleKnowns(velocities + 3*(size_t) part, otherForces ? otherForces + 3*(size_t) part : nullptr, mass[i],
                    (uint32_t) i, a, known, random);
            M += mass[i];
            for (int k = 0; k < 3; k++) {
                P[k] += known[k]*mass[i];
                R[k] += random[k];
            }
        }
        bool solid = solidAt(mask, node);
        double rho = 0, j[3] = {0, 0, 0};
        if (!solid)
            rho = nodeMoments(src, a.g, node, ucm, a.removal, j);
        double g[3] = {gx, gy, gz};
        double u[3] = {0, 0, 0}, sum[3];
        if (rho > 0) {
            for (int k = 0; k < 3; k++) {
                double knownFluid = (j[k] + h*(rho*g[k]))*(1.0/rho);
                sum[k] = ((P[k] - knownFluid*M)*(-gamma) + R[k])*(1.0/(1.0 + aa + aa*M/rho));
                u[k] = knownFluid - sum[k]*(h/rho);
            }
        }
        else
            for (int k = 0; k < 3; k++)
                sum[k] = ((P[k] - u[k]*M)*(-gamma) + R[k])*(1.0/(1.0 + aa));
        for (int t = s; t < e; t++) {
            int i = sortedIdx[t];
            int part = particles[i];
            double known[3], random[3];
            particleKnowns(velocities + 3*(size_t) part, otherForces ? otherForces + 3*(size_t) part : nullptr, mass[i],
                    (uint32_t) i, a, known, random);
            for (int k = 0; k < 3; k++)
                particleForce[3*(size_t) i + k] = ((known[k] - u[k])*(-gamma*mass[i]) + random[k])*(1.0/(1.0 + aa))*
                        a.forceScale;
        }
        if (a.isStep) {
            double r[3] = {-sum[0], -sum[1], -sum[2]};
            markTouched<1>(touched, node, addReaction(node, solid, r, a, reactionFixed, wallAcc), 0);
        }
    }
    blockPartials(wallAcc, partials);
}

/* ---------------------------------------------------------------------------------------------------------------- */
/* Stencils: conjugate gradients.                                                                                    */
/* ---------------------------------------------------------------------------------------------------------------- */
struct CgArgs {
    double* rhs;
    double* diag;
    double* F;
    double* r;
    double* z;
    double* d;
    int stride;              // of z and d from one particle to the next
    double* Ad;
    uint32_t* slotNode;
    double* slotW;
    double* slotWInvRho;     // w/rho, 0 at solid nodes
    uint8_t* slotSolid;
    uint8_t* slotSpreads;    // 1 where the slot takes part in the spread of a product (set by the solve's first one)
    unsigned long long* spread;        // [node][3] fixed point: the node sums of the current product
    unsigned long long* spreadOther;   // the other of the two arrays: the previous product's, cleared by the gather
    double* partials;        // [RED_BLOCKS][8]
    double* scalars;
    int slots;               // w^3
    const int* order;        // the particles in processing order (their slots are kept in that order), or nullptr
    // Sparse particles (split = 1): a product spreads only the slots at nodes that several slots share (spreadsAt); a
    // slot alone at its node contributes (w/rho) w x of its own particle directly.  seen/shared: node bits set by
    // cgMarkShared and cleared by cgForces.
    int split;
    uint32_t* seen;
    uint32_t* shared;
};

/*
 * The matrix of the solve by rows.  The particles are binned by the node their stencil starts at in cells of 4 x 4 x 4
 * nodes (the last cell of an axis takes the remainder, up to 7 nodes), so that those whose stencils reach a particle's lie in
 * the 27 cells around its own.  A row's entries are in the order of their particle, whatever the order in which the bins
 * were filled, so a solve is reproducible.  More than CELL_CAP particles in a cell or ROW_CAP in a row raise
 * `overflow`, which ends the solve by rows before its first iteration; the spread then takes it from what cgSetup left.
 * Each solve tries the rows anew: which of the two it takes depends on the particles alone, never on earlier solves, so
 * that a restarted run takes the same.  A step of 5,000 Keys particles and a crowd of 140 in 48^3, the rows' attempt
 * included: 403 us, 367 by the spread at once, 532 before there were rows.
 */
constexpr int CELL_CAP = 64, ROW_CAP = 128;
constexpr double ROWS_MEAN_NEIGHBOURS = 64.0;      // half of ROW_CAP
struct CellEntry {
    int particle, rank;
    uint32_t offset;         // of its first stencil node within the cell, x | y << 3 | z << 6
};
struct CgRows {
    int cells[3] = {0, 0, 0};
    int* cellCount = nullptr;        // cleared by cgInit
    CellEntry* cell = nullptr;       // [cell][CELL_CAP]
    uint32_t* home = nullptr;        // [rank][4]: the particle's cell along each axis, and its offset there
    double* axisWeight = nullptr;    // [rank][3][3w - 2]: the weights along each axis between w - 1 zeros on either side
    int* rowCount = nullptr;         // [particle]
    int* rowParticle = nullptr;      // [particle][ROW_CAP]
    double* rowValue = nullptr;
    int* overflow = nullptr;
};

/* Whether a slot's node takes part in the spread of a product: every node without the split, else the shared ones. */
__device__ __forceinline__ bool spreadsAt(const CgArgs& c, uint32_t node) {
    return !c.split || ((c.shared[node >> 5] >> (node & 31)) & 1u);
}

/*
 * The work-group's place in the processing order: each XCD takes a contiguous run of the particles, sorted by node, so
 * that the node sums that neighbouring stencils share are read through one L2.  For dense particles only (56,320 Keys
 * particles in 120^3: a gather 58.6 -> 39.1 us; 20,000 in 256^3 share few nodes and keep the index order).
 */
__device__ __forceinline__ uint32_t placeOf(const CgArgs& c) {
    return c.order != nullptr ? xcdContiguousTile(blockIdx.x, gridDim.x) : blockIdx.x;
}

/* The particle at place `rank` of the processing order. */
__device__ __forceinline__ int particleAt(const CgArgs& c, int rank) {
    return c.order != nullptr ? c.order[rank] : rank;
}

/* One group of LANES lanes per particle, one lane per stencil slot: the slot's node, weight and w/rho, the particle's
   right-hand side, diagonal and F = rhs/diagonal. */
template <typename S, int LANES>
__global__ void __launch_bounds__(BLOCK) cgSetup(const S* __restrict__ src, const uint32_t* __restrict__ mask,
        const double* __restrict__ positions, const double* __restrict__ velocities,
        const double* __restrict__ otherForces, const int* __restrict__ particles, const double* __restrict__ mass,
        const double* __restrict__ ucm, ParticleArgs a, double gx, double gy, double gz, CgArgs c,
        const double4* __restrict__ field, CgRows rows) {
    constexpr int GROUPS = BLOCK/LANES;
    const double h = 0.5, aa = a.gamma*h;
    int lane = threadIdx.x % LANES;
    const int rank = (int) placeOf(c)*GROUPS + threadIdx.x/LANES;
    bool active = rank < a.numParticles;
    const int i = active ? particleAt(c, rank) : 0;
    int part = active ? particles[i] : 0;
    const double* x = positions + 3*(size_t) part;
    // The stencil of the lanes (groupStencil), its slots along the axes formed by the group's first 3 w lanes as in
    // interpolateGroup.
    constexpr int STENCIL = groupStencil<LANES>();
    constexpr int w = STENCIL == LBM_STENCIL_KEYS ? 4 : STENCIL == LBM_STENCIL_THREE_POINT ? 3 : 2;
    bool inStencil = active && lane < c.slots;
    double ux = 0, uy = 0, uz = 0, self = 0;
    const int nx = (int) a.g.nx, ny = (int) a.g.ny, nz = (int) a.g.nz;
    const int openX = a.g.openX, openY = a.g.openY, openZ = a.g.openZ;
    int axisIndex;
    double axisWeight;
    {
        const int axis = lane < w ? 0 : (lane < 2*w ? 1 : 2);
        const int size = axis == 0 ? nx : (axis == 1 ? ny : nz);
        const int open = axis == 0 ? openX : (axis == 1 ? openY : openZ);
        axisSlot<STENCIL>(wrapCoordinate(x[axis], a.dx, size), size, open != 0, min(lane - axis*w, w - 1), axisIndex,
                axisWeight);
    }
    const int sub[3] = {lane % w, (lane/w) % w, min(lane/(w*w), w - 1)};
    int nodeIdx[3], first[3];
    double weight = 1.0;
    for (int k = 0; k < 3; k++) {
        nodeIdx[k] = __shfl(axisIndex, k*w + sub[k], LANES);
        first[k] = __shfl(axisIndex, k*w, LANES);
        weight *= __shfl(axisWeight, k*w + sub[k], LANES);
    }
    if (rows.cell != nullptr && active) {
        if (lane < 3*w)
            rows.axisWeight[((size_t) rank*3 + lane/w)*(3*w - 2) + w - 1 + lane % w] = axisWeight;
        if (lane == 0) {
            int cell[3];
            uint32_t offset = 0;
            for (int k = 0; k < 3; k++) {
                cell[k] = min(first[k] >> 2, rows.cells[k] - 1);
                offset |= (uint32_t) (first[k] - 4*cell[k]) << (3*k);
                rows.home[4*(size_t) rank + k] = (uint32_t) cell[k];
            }
            rows.home[4*(size_t) rank + 3] = offset;
            const size_t at = (size_t) cell[0] + (size_t) rows.cells[0]*(cell[1] + (size_t) rows.cells[1]*cell[2]);
            const int entry = atomicAdd(rows.cellCount + at, 1);
            if (entry < CELL_CAP)
                rows.cell[at*CELL_CAP + entry] = CellEntry{i, rank, offset};
            else
                *rows.overflow = 1;
        }
    }
    if (inStencil) {
        uint32_t node = (uint32_t) (nodeIdx[0] + (int) a.g.nx*(nodeIdx[1] + (int) a.g.ny*nodeIdx[2]));
        bool solid = solidAt(mask, node);
        double winv = 0.0;
        if (!solid) {
            double j[3], rho;
            if (field != nullptr) {
                const double4 m = field[node];
                j[0] = m.x;
                j[1] = m.y;
                j[2] = m.z;
                rho = m.w;
            }
            else
                rho = nodeMoments(src, a.g, node, ucm, a.removal, j);
            if (rho > 0) {
                ux = (j[0] + h*(rho*gx))*(weight/rho);
                uy = (j[1] + h*(rho*gy))*(weight/rho);
                uz = (j[2] + h*(rho*gz))*(weight/rho);
                self = weight*weight/rho;
                winv = weight/rho;
            }
        }
        size_t sl = (size_t) rank*c.slots + lane;
        c.slotNode[sl] = node;
        c.slotW[sl] = weight;
        c.slotWInvRho[sl] = winv;
        c.slotSolid[sl] = solid ? 1 : 0;
    }
    ux = groupSum<LANES>(ux);
    uy = groupSum<LANES>(uy);
    uz = groupSum<LANES>(uz);
    self = groupSum<LANES>(self);
    if (active && lane == 0) {
        double m = mass[i];
        double known[3], random[3];
        particleKnowns(velocities + 3*(size_t) part, otherForces ? otherForces + 3*(size_t) part : nullptr, m, (uint32_t) i,
                a, known, random);
        double u[3] = {ux, uy, uz};
        double diag = (1.0 + aa)/m + aa*self;
        c.diag[i] = diag;
        for (int k = 0; k < 3; k++) {
            double b = ((known[k] - u[k])*(-a.gamma*m) + random[k])*(1.0/m);
            c.rhs[3*(size_t) i + k] = b;
            c.F[3*(size_t) i + k] = b*(1.0/diag);
        }
    }
}

/*
 * The matrix row of each particle, one wavefront per particle, and the first product Ad = A F.  Pairs of lanes search a
 * cell each, the particles found are sorted by index, and then a lane takes a neighbour l: K_kl = sum over k's slots of
 * (w_k/rho) w_l, its own weights along the axes shifted by the distance of the two stencils (zero outside).  Forming the
 * row by lanes that are neighbours takes 84 FP64 operations for up to 64 of them; by lanes that are slots it takes a
 * sum over the wavefront for each.  56,320 Keys particles in 120^3: 96 us, bound by the chain of loads (cell, entries, weights),
 * and a product then takes 17 us (cgRowsStep) where spread and gather took 145.
 */
template <int W>
__global__ void __launch_bounds__(BLOCK) cgRows(int n, int nx, int ny, int nz, CgArgs c, CgRows rows,
        const double* __restrict__ mass, double aa) {
    constexpr int WAVES = BLOCK/64, SLOTS = W*W*W;
    struct Found {
        int particle[ROW_CAP], rank[ROW_CAP];
        uint16_t shift[ROW_CAP];             // the distance of the stencils + 3 along each axis, 3 bits each
        uint8_t sorted[ROW_CAP];
    };
    __shared__ Found all[WAVES];
    const int lane = (int) threadIdx.x & 63;
    const int rank = __builtin_amdgcn_readfirstlane((int) placeOf(c)*WAVES + (int) threadIdx.x/64);
    if (rank >= n || *rows.overflow != 0)
        return;
    // w/rho of the particle's slots: the same for every lane, so operands from scalar registers.
    const auto* own = (const __attribute__((address_space(4))) double*) (uintptr_t) (c.slotWInvRho + (size_t) rank*SLOTS);
    Found& f = all[threadIdx.x/64];
    const int size[3] = {nx, ny, nz};
    int origin[3] = {0, 0, 0};               // of the lane's cell, from the own cell's
    size_t at = 0;
    const uint4 home = *(const uint4*) (rows.home + 4*(size_t) rank);
    const uint32_t offset = home.w;
    int count = 0;
    if (lane < 54) {
        const int c27 = lane >> 1;
        const int step[3] = {c27 % 3 - 1, c27/3 % 3 - 1, c27/9 - 1};
        const int own[3] = {(int) home.x, (int) home.y, (int) home.z};
        int cell[3];
        for (int k = 0; k < 3; k++) {
            const int last = rows.cells[k] - 1;
            cell[k] = own[k] + step[k] < 0 ? last : (own[k] + step[k] > last ? 0 : own[k] + step[k]);
            const int widthOfLast = size[k] - 4*last;
            if (step[k] > 0)
                origin[k] = own[k] == last ? widthOfLast : 4;
            else if (step[k] < 0)
                origin[k] = cell[k] == last ? -widthOfLast : -4;
        }
        at = (size_t) cell[0] + (size_t) rows.cells[0]*(cell[1] + (size_t) rows.cells[1]*cell[2]);
        count = min(rows.cellCount[at], CELL_CAP);
    }
    int found = 0;
    // Two lanes per cell, two entries each per turn, their loads in one wait.
    for (int first = lane & 1; __ballot(first < count) != 0; first += 4) {
        CellEntry entries[2];
        for (int u = 0; u < 2; u++)
            entries[u] = first + 2*u < count ? rows.cell[at*CELL_CAP + first + 2*u] : CellEntry{0, 0, 0};
        for (int u = 0; u < 2; u++) {
            const CellEntry entry = entries[u];
            bool hit = first + 2*u < count;
            int d[3];
            for (int k = 0; k < 3; k++) {
                d[k] = origin[k] + (int) ((entry.offset >> (3*k)) & 7u) - (int) ((offset >> (3*k)) & 7u);
                hit = hit && d[k] > -W && d[k] < W;
            }
            const uint64_t hits = __ballot(hit);
            const int place = found + (int) __popcll(hits & ((1ull << lane) - 1ull));
            if (hit && place < ROW_CAP) {
                f.particle[place] = entry.particle;
                f.rank[place] = entry.rank;
                f.shift[place] = (uint16_t) ((d[0] + 3) | (d[1] + 3) << 3 | (d[2] + 3) << 6);
            }
            found += (int) __popcll(hits);
        }
    }
    if (found > ROW_CAP) {
        if (lane == 0)
            *rows.overflow = 1;
        found = ROW_CAP;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int e = lane; e < found; e += 64) {
        const int own = f.particle[e];
        int place = 0;
        for (int o = 0; o < found; o++)
            place += f.particle[o] < own ? 1 : 0;
        f.sorted[place] = (uint8_t) e;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const size_t i = (size_t) particleAt(c, rank);
    double acc[3] = {0, 0, 0};
    for (int e = lane; e < found; e += 64) {
        const int from = f.sorted[e], l = f.particle[from];
        const uint32_t shift = f.shift[from];
        const double* weights = rows.axisWeight + (size_t) f.rank[from]*(3*(3*W - 2)) + W - 1;
        double wl[3][W];
        for (int k = 0; k < 3; k++) {
            const int d = (int) ((shift >> (3*k)) & 7u) - 3;
            for (int sl = 0; sl < W; sl++)
                wl[k][sl] = weights[k*(3*W - 2) + sl - d];
        }
        double value = 0.0;
        for (int z = 0; z < W; z++) {
            double plane = 0.0;
            for (int y = 0; y < W; y++) {
                double row = 0.0;
                for (int xs = 0; xs < W; xs++)
                    row = fma(own[xs + W*(y + W*z)], wl[0][xs], row);
                plane = fma(row, wl[1][y], plane);
            }
            value = fma(plane, wl[2][z], value);
        }
        rows.rowParticle[i*ROW_CAP + e] = l;
        rows.rowValue[i*ROW_CAP + e] = value;
        for (int k = 0; k < 3; k++)
            acc[k] = fma(value, c.F[3*(size_t) l + k], acc[k]);
    }
    for (int k = 0; k < 3; k++)
        acc[k] = groupSum<64>(acc[k]);
    if (lane == 0)
        rows.rowCount[i] = found;
    if (lane < 3) {
        const double own = lane == 0 ? acc[0] : (lane == 1 ? acc[1] : acc[2]);
        c.Ad[3*i + lane] = c.F[3*i + lane]*((1.0 + aa)/mass[i]) + own*aa;
    }
}

/* The nodes that several fluid slots share (with the split), one group of LANES lanes per particle, one lane per slot
   (markSharedRun: one atomic OR per run of a stencil row's lanes on one word). */
template <int LANES>
__global__ void __launch_bounds__(BLOCK) cgMarkShared(int n, CgArgs c) {
    constexpr int GROUPS = BLOCK/LANES;
    constexpr int W = LANES == 64 ? 4 : LANES == 32 ? 3 : 2;    // slots per stencil row
    const int lane = threadIdx.x % LANES;
    const int i = blockIdx.x*GROUPS + threadIdx.x/LANES;
    uint32_t node = 0;
    bool live = false;
    if (i < n && lane < c.slots) {
        size_t sl = (size_t) i*c.slots + lane;
        live = c.slotWInvRho[sl] != 0.0;
        node = c.slotNode[sl];
    }
    markSharedRun<W>(c.seen, c.shared, node, live, lane);
}

/* Every component's residual within CG_TOLERANCE of its right-hand side (the host's test and the device's). */
__host__ __device__ inline bool residualConverged(const double* s) {
    for (int k = 0; k < 3; k++)
        if (s[RR + k] > CG_TOLERANCE*CG_TOLERANCE*s[NORM + k])
            return false;
    return true;
}

/* Largest |x| over the particles and components -> partials[block][0]. */
__global__ void __launch_bounds__(BLOCK) cgMaxAbs(const double* __restrict__ x, int n, double* __restrict__ partials,
        const double* done) {
    if (done != nullptr && *done != 0.0)
        return;
    double m = 0.0;
    for (int i = blockIdx.x*BLOCK + threadIdx.x; i < 3*n; i += gridDim.x*BLOCK)
        m = fmax(m, fabs(x[i]));
    __shared__ double lds[BLOCK];
    lds[threadIdx.x] = m;
    __syncthreads();
    for (int s = BLOCK/2; s > 0; s >>= 1) {
        if ((int) threadIdx.x < s)
            lds[threadIdx.x] = fmax(lds[threadIdx.x], lds[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0)
        partials[8*blockIdx.x] = lds[0];
}

/* The partial rows of the RED_BLOCKS blocks of a reduction, combined by one wavefront (launched with 64 threads):
   lane l takes the rows l, l + 64, ... in order, then the lanes combine in a fixed butterfly, so the result is the same
   in every run.  MAX takes the largest value instead of the sum.  Every lane returns the result. */
template <int COUNT, bool MAX = false>
__device__ __forceinline__ void combinePartials(const double* __restrict__ partials, double v[COUNT]) {
    static_assert(RED_BLOCKS % 64 == 0, "whole rows per lane");
    for (int q = 0; q < COUNT; q++)
        v[q] = 0.0;
    for (int b = threadIdx.x; b < RED_BLOCKS; b += 64)
        for (int q = 0; q < COUNT; q++)
            v[q] = MAX ? fmax(v[q], partials[8*b + q]) : v[q] + partials[8*b + q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        for (int q = 0; q < COUNT; q++) {
            double o = __shfl_xor(v[q], off, 64);
            v[q] = MAX ? fmax(v[q], o) : v[q] + o;
        }
}

/* spread[node] += w x (fixed point), one thread per particle slot and component: consecutive lanes add to consecutive
   words, 12 for a Keys row, so a wavefront's atomics, which run at the memory side and are bound by the requests, reach it
   as a third of those that three strided adds per slot made (56,320 Keys particles in 120^3: 255 -> 105 us).  The fixed-point scale, 2^(52 - e) with
   2^e >= max |x| (1 if x is zero), is formed by the first wavefront of every work-group from the largest |x| of the
   blocks in c.partials (one fixed combination, so every work-group has the same value); work-group 0 keeps it and its
   inverse in the scalars for the gather.  The solve's first product (first = 1) records which slots spread.
   firstBlock: of the launch; a launch holds SPREAD_BLOCKS at most, as its threads are counted in 32 bits. */
constexpr uint32_t SPREAD_BLOCKS = 1u << 20;
template <int SLOTS>
__global__ void __launch_bounds__(BLOCK) cgSpread(const double* __restrict__ x, int n, CgArgs c,
        const double* done, int first, uint32_t firstBlock) {
    if (done != nullptr && *done != 0.0)
        return;
    __shared__ double sharedScale;
    if (threadIdx.x < 64) {
        double m[1];
        combinePartials<1, true>(c.partials, m);
        if (threadIdx.x == 0) {
            int e = m[0] > 0 ? ilogb(m[0]) + 1 : 0;
            sharedScale = ldexp(1.0, 52 - e);
            if (blockIdx.x == 0) {
                c.scalars[SCALE] = sharedScale;
                c.scalars[INV_SCALE] = ldexp(1.0, e - 52);
            }
        }
    }
    __syncthreads();
    const uint64_t item = (uint64_t) (firstBlock + placeOf(c))*BLOCK + threadIdx.x;
    const uint64_t t = item/3;
    const int k = (int) (item - 3*t);
    const uint64_t rank = t/SLOTS;
    if (rank >= (uint64_t) n)
        return;
    double w = c.slotW[t];
    uint32_t node = c.slotNode[t];
    bool spreads;
    if (first) {
        spreads = w != 0.0 && spreadsAt(c, node);
        if (k == 0)
            c.slotSpreads[t] = spreads ? 1 : 0;
    }
    else
        spreads = c.slotSpreads[t] != 0;
    if (!spreads)
        return;
    const size_t i = (size_t) particleAt(c, (int) rank);
    long long v = llrint(w*x[3*i + k]*sharedScale);
    if (v != 0)
        atomicAdd(c.spread + 3*(size_t) node + k, (unsigned long long) v);
}

/* Ax = x (1 + a)/m + a sum_slots (w/rho) spread[node], one group of LANES lanes per particle. */
template <int LANES>
__global__ void __launch_bounds__(BLOCK) cgGather(const double* __restrict__ x, double* __restrict__ Ax,
        const double* __restrict__ mass, int n, double aa, CgArgs c, const double* done) {
    if (done != nullptr && *done != 0.0)
        return;
    constexpr int GROUPS = BLOCK/LANES;
    int lane = threadIdx.x % LANES;
    const int rank = (int) placeOf(c)*GROUPS + threadIdx.x/LANES;
    bool active = rank < n;
    const int i = active ? particleAt(c, rank) : 0;
    double s[3] = {0, 0, 0};
    if (active && lane < c.slots) {
        size_t sl = (size_t) rank*c.slots + lane;
        double winv = c.slotWInvRho[sl];
        const bool spreads = c.slotSpreads[sl] != 0;
        const uint32_t node = c.slotNode[sl];
        // The previous product's node sums, which every reader has read, cleared for the next product.
        if (spreads && c.spreadOther != nullptr)
            for (int k = 0; k < 3; k++)
                c.spreadOther[3*(size_t) node + k] = 0ull;
        if (winv != 0.0) {
            if (spreads) {
                double inv = c.scalars[INV_SCALE];
                for (int k = 0; k < 3; k++)
                    s[k] = (double) (long long) c.spread[3*(size_t) node + k]*inv*winv;
            }
            else {
                // Alone at its node: the node's sum is this slot's own w x.
                double ww = c.slotW[sl]*winv;
                for (int k = 0; k < 3; k++)
                    s[k] = ww*x[3*(size_t) i + k];
            }
        }
    }
    for (int k = 0; k < 3; k++)
        s[k] = groupSum<LANES>(s[k]);
    if (active && lane == 0)
        for (int k = 0; k < 3; k++)
            Ax[3*(size_t) i + k] = x[3*(size_t) i + k]*((1.0 + aa)/mass[i]) + s[k]*aa;
}

/* Block sums of up to 8 per-particle quantities into partials[block][0..7], fixed order. */
__device__ __forceinline__ void reduceBlock(double v[8], int count, double* partials) {
    __shared__ double lds[8][BLOCK];
    for (int q = 0; q < count; q++)
        lds[q][threadIdx.x] = v[q];
    __syncthreads();
    for (int s = BLOCK/2; s > 0; s >>= 1) {
        if ((int) threadIdx.x < s)
            for (int q = 0; q < count; q++)
                lds[q][threadIdx.x] += lds[q][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int q = 0; q < count; q++)
            partials[8*blockIdx.x + q] = lds[q][0];
}

/* r = rhs - Ax, z = r/diag, d = z; partials: r.z, rhs.rhs, r.r (3 each -> 9 values in two reductions). */
__global__ void __launch_bounds__(BLOCK) cgInit(int n, CgArgs c, double* partialsB, int* cellCount, int numCells) {
    for (int cell = blockIdx.x*BLOCK + threadIdx.x; cell < numCells; cell += gridDim.x*BLOCK)
        cellCount[cell] = 0;
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0}, w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int i = blockIdx.x*BLOCK + threadIdx.x; i < n; i += gridDim.x*BLOCK)
        for (int k = 0; k < 3; k++) {
            size_t t = 3*(size_t) i + k;
            double r = c.rhs[t] - c.Ad[t];
            double z = r*(1.0/c.diag[i]);
            c.r[t] = r;
            c.z[(size_t) i*c.stride + k] = z;
            c.d[(size_t) i*c.stride + k] = z;
            v[k] += r*z;
            v[3 + k] += c.rhs[t]*c.rhs[t];
            w[k] += r*r;
        }
    reduceBlock(v, 6, c.partials);
    __syncthreads();
    reduceBlock(w, 3, partialsB);
}

/* overflow: CgRows::overflow, or nullptr; with it set no iteration runs. */
__global__ void __launch_bounds__(64) cgFinishInit(const double* __restrict__ partials,
        const double* __restrict__ partialsB, double* __restrict__ scalars, const int* __restrict__ overflow) {
    double v[6], w[3];
    combinePartials<6>(partials, v);
    combinePartials<3>(partialsB, w);
    if (threadIdx.x != 0)
        return;
    for (int k = 0; k < 3; k++) {
        scalars[RZ + k] = v[k];
        scalars[NORM + k] = v[3 + k];
        scalars[RR + k] = w[k];
    }
    scalars[DONE] = residualConverged(scalars) || (overflow != nullptr && *overflow != 0) ? 1.0 : 0.0;
    scalars[ITERS] = 0.0;
}

/* d . Ad into c.partials (alpha = r.z/(d.Ad) follows in cgUpdate). */
__global__ void __launch_bounds__(BLOCK) cgDot(int n, CgArgs c, const double* done) {
    if (done != nullptr && *done != 0.0)
        return;
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int i = blockIdx.x*BLOCK + threadIdx.x; i < n; i += gridDim.x*BLOCK)
        for (int k = 0; k < 3; k++)
            v[k] += c.d[3*(size_t) i + k]*c.Ad[3*(size_t) i + k];
    reduceBlock(v, 3, c.partials);
}

/* alpha = r.z/(d.Ad), from the blocks' d.Ad in c.partials (formed by the first wavefront of every work-group, one
   fixed combination; work-group 0 keeps it in the scalars); F += alpha d, r -= alpha Ad, z = r/diag; partialsOut:
   r.z (new), r.r (a buffer of its own: other work-groups may still be reading c.partials). */
__global__ void __launch_bounds__(BLOCK) cgUpdate(int n, CgArgs c, double* __restrict__ partialsOut,
        const double* done, int rz) {
    if (done != nullptr && *done != 0.0)
        return;
    __shared__ double sharedAlpha[3];
    if (threadIdx.x < 64) {
        double dad[3];
        combinePartials<3>(c.partials, dad);
        if (threadIdx.x == 0)
            for (int k = 0; k < 3; k++) {
                sharedAlpha[k] = dad[k] > 0 ? c.scalars[rz + k]/dad[k] : 0.0;
                if (blockIdx.x == 0) {
                    c.scalars[DAD + k] = dad[k];
                    c.scalars[ALPHA + k] = sharedAlpha[k];
                }
            }
    }
    __syncthreads();
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    double alpha[3] = {sharedAlpha[0], sharedAlpha[1], sharedAlpha[2]};
    for (int i = blockIdx.x*BLOCK + threadIdx.x; i < n; i += gridDim.x*BLOCK)
        for (int k = 0; k < 3; k++) {
            size_t t = 3*(size_t) i + k;
            c.F[t] += alpha[k]*c.d[(size_t) i*c.stride + k];
            double r = c.r[t] - alpha[k]*c.Ad[t];
            double z = r*(1.0/c.diag[i]);
            c.r[t] = r;
            c.z[(size_t) i*c.stride + k] = z;
            v[k] += r*z;
            v[3 + k] += r*r;
        }
    reduceBlock(v, 6, partialsOut);
}

/* beta = r.z(new)/r.z(old), r.z <- r.z(new), r.r. */
__global__ void __launch_bounds__(64) cgFinishBeta(const double* __restrict__ partials, double* __restrict__ scalars,
        const double* done) {
    if (done != nullptr && *done != 0.0)
        return;
    double v[6];
    combinePartials<6>(partials, v);
    if (threadIdx.x != 0)
        return;
    for (int k = 0; k < 3; k++) {
        double rz = scalars[RZ + k];
        scalars[BETA + k] = rz > 0 ? v[k]/rz : 0.0;
        scalars[RZ + k] = v[k];
        scalars[RZ_NEW + k] = v[k];
        scalars[RR + k] = v[3 + k];
    }
    scalars[DONE] = residualConverged(scalars) ? 1.0 : 0.0;
    scalars[ITERS] += 1.0;
}

/* d = z + beta d, and the largest |d| of each block -> partials[block][0] (for the scale of the next spread). */
__global__ void __launch_bounds__(BLOCK) cgDirection(int n, CgArgs c, const double* done) {
    if (done != nullptr && *done != 0.0)
        return;
    double beta[3] = {c.scalars[BETA], c.scalars[BETA + 1], c.scalars[BETA + 2]};
    double m = 0.0;
    for (int i = blockIdx.x*BLOCK + threadIdx.x; i < n; i += gridDim.x*BLOCK)
        for (int k = 0; k < 3; k++) {
            size_t t = 3*(size_t) i + k;
            double d = c.z[t] + beta[k]*c.d[t];
            c.d[t] = d;
            m = fmax(m, fabs(d));
        }
    __shared__ double lds[BLOCK];
    lds[threadIdx.x] = m;
    __syncthreads();
    for (int s = BLOCK/2; s > 0; s >>= 1) {
        if ((int) threadIdx.x < s)
            lds[threadIdx.x] = fmax(lds[threadIdx.x], lds[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0)
        c.partials[8*blockIdx.x] = lds[0];
}

/*
 * One iteration's direction and product with the matrix rows, ROW_LANES lanes per particle: beta = r.z(new)/r.z(old) from
 * the update's partial sums (formed by the first wavefront of every work-group, one fixed combination), d = z + beta d and
 * Ad = A d with the neighbours' new d formed on the way, and d.Ad of each work-group.  A particle's z and old d are side by
 * side, [particle][z, d], one gather for both (20.7 -> 16.8 us for 56,320 Keys particles, bound by these gathers); d goes to
 * the other of two such arrays, since the neighbours read the old one, and the update puts the new z beside it.  Tests the
 * residual first, as the direction after a converged iteration is not needed.  With cgUpdate, two launches per iteration
 * where the spread takes six.  The particles are taken by index, not by their place in the processing order, which depends
 * on when it was last sorted: d.Ad must be the same sum in a run that was restarted (a step of 56,320 Keys particles in
 * 120^3 508 us by place, 503 by index; of 1,000,000 in 320^3 8.38 and 8.57 ms).
 */
constexpr int ROW_LANES = 8, ROW_THREADS_CG = 1024;
__global__ void __launch_bounds__(ROW_THREADS_CG) cgRowsStep(int n, CgArgs c, CgRows rows, const double* __restrict__ old,
        double* __restrict__ next, const double* __restrict__ mass, double aa, const double* __restrict__ partialsB,
        int iteration) {
    __shared__ double sharedBeta[3];
    __shared__ int sharedDone;
    __shared__ double sums[ROW_THREADS_CG/64][3];
    const int t = (int) threadIdx.x;
    if (t < 64) {
        double v[6] = {0, 0, 0, 0, 0, 0};
        if (iteration > 0)
            combinePartials<6>(partialsB, v);
        if (t == 0) {
            bool done = c.scalars[DONE] != 0.0;
            double beta[3] = {0, 0, 0};
            if (!done && iteration > 0) {
                double test[NUM_SCALARS];
                for (int k = 0; k < 3; k++) {
                    test[RR + k] = v[3 + k];
                    test[NORM + k] = c.scalars[NORM + k];
                    const double rz = c.scalars[RZ + RZ_SLOT*((iteration - 1) & 1) + k];
                    beta[k] = rz > 0 ? v[k]/rz : 0.0;
                }
                done = residualConverged(test);
                if (blockIdx.x == 0) {
                    for (int k = 0; k < 3; k++)
                        c.scalars[RZ + RZ_SLOT*(iteration & 1) + k] = v[k];
                    if (done) {
                        c.scalars[ITERS] = (double) iteration;
                        c.scalars[DONE] = 1.0;
                    }
                }
            }
            for (int k = 0; k < 3; k++)
                sharedBeta[k] = beta[k];
            sharedDone = done ? 1 : 0;
        }
    }
    __syncthreads();
    if (sharedDone)
        return;
    const double beta[3] = {sharedBeta[0], sharedBeta[1], sharedBeta[2]};
    const int lane = t % ROW_LANES;
    constexpr int PARTICLES = ROW_THREADS_CG/ROW_LANES;
    double dot = 0.0;                        // of component `lane`
    for (int base = (int) blockIdx.x*PARTICLES; base < n; base += RED_BLOCKS*PARTICLES) {
        const int i = base + t/ROW_LANES;
        double s[3] = {0, 0, 0};
        if (i < n) {
            const int count = rows.rowCount[i];
            for (int e = lane; e < count; e += ROW_LANES) {
                const double2* from = (const double2*) (old + 6*(size_t) rows.rowParticle[(size_t) i*ROW_CAP + e]);
                const double value = rows.rowValue[(size_t) i*ROW_CAP + e];
                const double2 a01 = from[0], a23 = from[1], a45 = from[2];
                s[0] = fma(value, fma(beta[0], a23.y, a01.x), s[0]);
                s[1] = fma(value, fma(beta[1], a45.x, a01.y), s[1]);
                s[2] = fma(value, fma(beta[2], a45.y, a23.x), s[2]);
            }
        }
        for (int k = 0; k < 3; k++)
            s[k] = groupSum<ROW_LANES>(s[k]);
        if (i < n && lane < 3) {
            const size_t at = 6*(size_t) i + lane;
            const double d = fma(lane == 0 ? beta[0] : (lane == 1 ? beta[1] : beta[2]), old[at + 3], old[at]);
            const double Ad = d*((1.0 + aa)/mass[i]) + (lane == 0 ? s[0] : (lane == 1 ? s[1] : s[2]))*aa;
            next[at + 3] = d;
            c.Ad[3*(size_t) i + lane] = Ad;
            dot = fma(d, Ad, dot);
        }
    }
    for (int off = ROW_LANES; off < 64; off *= 2)
        dot += __shfl_xor(dot, off, 64);
    if ((t & 63) < 3)
        sums[t/64][t & 63] = dot;
    __syncthreads();
    if (t < 3) {
        double v = 0.0;
        for (int w = 0; w < ROW_THREADS_CG/64; w++)
            v += sums[w][t];
        c.partials[8*blockIdx.x + t] = v;
    }
}

/* The state of the solve after `iterations` iterations with the matrix rows, to the device scalars and to the host's
   (page-locked): whether it has converged, and whether the rows overflowed, in which case nothing of it counts. */
__global__ void __launch_bounds__(64) cgRowsCheck(const double* __restrict__ partialsB, double* __restrict__ scalars,
        const int* __restrict__ overflow, int iterations, double* __restrict__ host) {
    double v[6];
    combinePartials<6>(partialsB, v);
    if (threadIdx.x != 0)
        return;
    bool done = scalars[DONE] != 0.0;
    if (!done && iterations > 0) {
        double test[NUM_SCALARS];
        for (int k = 0; k < 3; k++) {
            test[RR + k] = v[3 + k];
            test[NORM + k] = scalars[NORM + k];
        }
        done = residualConverged(test);
        scalars[ITERS] = (double) iterations;
    }
    const bool over = *overflow != 0;
    scalars[DONE] = done && !over ? 1.0 : 0.0;
    host[DONE] = scalars[DONE];
    host[ITERS] = scalars[ITERS];
    host[OVERFLOWED] = over ? 1.0 : 0.0;
}

/* The forces and the reactions -w F of the solution, one group of LANES lanes per particle (block layout of the explicit
   coupling, so the wall partials fit the same slots).  BINNED: in a step each particle goes into the bin of its first
   node's tile for spreadTiles, with the slots' weights where cgSetup left them; one whose bin is full spreads here (56,320
   Keys particles in 120^3: 46 us and 38 us for the tiles against 118 with the atomics).  wall: with a processing order, each
   particle's wall momentum goes to wall[particle][3] for cgWall, whose sums do not depend on the order; else the work-group's
   into partials. */
template <int LANES, bool BINNED>
__global__ void __launch_bounds__(BLOCK) cgForces(int n, ParticleArgs a, CgArgs c, double* __restrict__ particleForce,
        unsigned long long* __restrict__ reactionFixed, uint32_t* __restrict__ touched, double* __restrict__ partials,
        double* __restrict__ wall, const int* __restrict__ rowCount, SpreadBins bins, const int* __restrict__ particles,
        double* __restrict__ systemForce) {
    // With matrix rows the host launches this before it knows whether the solve has converged.
    if (rowCount != nullptr && c.scalars[DONE] == 0.0)
        return;
    constexpr int GROUPS = BLOCK/LANES;
    int lane = threadIdx.x % LANES;
    const int rank = (int) placeOf(c)*GROUPS + threadIdx.x/LANES;
    double wallAcc[3] = {0, 0, 0};
    uint32_t node = 0;
    bool flagged = false;
    __shared__ StagedReactions<BLOCK> staged;
    staged.clear();
    bool atomics = true;
    if (rank < n) {
        const int i = particleAt(c, rank);
        double F[3] = {c.F[3*(size_t) i], c.F[3*(size_t) i + 1], c.F[3*(size_t) i + 2]};
        if (lane < 3) {
            const double f = (lane == 0 ? F[0] : (lane == 1 ? F[1] : F[2]))*a.forceScale;
            particleForce[3*(size_t) i + lane] = f;
            // As groupForce: atomically, in case a particle were coupled twice.
            if (systemForce != nullptr)
                atomicAdd(systemForce + 3*(size_t) particles[i] + lane, f);
        }
        if constexpr (BINNED) {
            int full = 0;
            if (a.isStep && lane == 0) {
                uint32_t x[3];
                nodeCoords(a.g, c.slotNode[(size_t) rank*c.slots], x[0], x[1], x[2]);
                const uint32_t tx = tileOf(x[0], bins.ntx, bins.perNode[0]), ty = tileOf(x[1], bins.nty, bins.perNode[1]);
                const uint32_t tz = tileOf(x[2], bins.ntz, bins.perNode[2]);
                const uint32_t tile = tx + bins.ntx*(ty + bins.nty*tz);
                const int slot = atomicAdd(bins.count + tile, 1);
                if (slot < bins.cap) {
                    const size_t entry = (size_t) tile*bins.cap + slot;
                    bins.beads[entry] = rank;
                    bins.anchor[entry] = (uint16_t) ((x[0] - tileStart(tx, a.g.nx, bins.perTile[0])) |
                            (x[1] - tileStart(ty, a.g.ny, bins.perTile[1])) << 5 | (x[2] - tileStart(tz, a.g.nz, bins.perTile[2])) << 7);
                    for (int k = 0; k < 3; k++)
                        bins.force[3*entry + k] = F[k];
                }
                else {
                    full = 1;
                    atomicOr(bins.spilled, 1);
                }
            }
            atomics = __shfl(full, 0, LANES) != 0;
        }
        if (a.isStep && lane < c.slots) {
            size_t sl = (size_t) rank*c.slots + lane;
            double w = c.slotW[sl];
            node = c.slotNode[sl];
            if (w != 0.0) {
                double r[3] = {-w*F[0], -w*F[1], -w*F[2]};
                bool solid = c.slotSolid[sl] != 0;
                // With the split, a fluid slot that spreads nothing is alone at its node, and with matrix rows so is
                // every slot of a particle without neighbours: a store, not an atomic.
                const bool alone = BINNED ? false : rowCount != nullptr ? rowCount[particleAt(c, rank)] == 1 : c.split && c.slotSpreads[sl] == 0;
                if (alone && !solid && c.slotWInvRho[sl] != 0.0)
                    flagged = storeReaction(node, r, a, reactionFixed);
                else if (solid)
                    for (int k = 0; k < 3; k++)
                        wallAcc[k] = r[k];               // lattice momentum; the host converts the wall partials
                else if (atomics)
                    flagged = staged.put(node, r, a);
            }
        }
        // Both arrays of node sums and the node bits of the split, cleared for the next solve (every word that a
        // spread or cgMarkShared set belongs to one of these slots; nothing reads them after the solve).
        if (rowCount == nullptr && lane < c.slots) {
            size_t sl = (size_t) rank*c.slots + lane;
            uint32_t at = c.slotNode[sl];
            if (c.slotSpreads[sl] != 0)
                for (int k = 0; k < 3; k++) {
                    c.spread[3*(size_t) at + k] = 0ull;
                    c.spreadOther[3*(size_t) at + k] = 0ull;
                }
            if (c.split && c.slotWInvRho[sl] != 0.0) {
                c.seen[at >> 5] = 0u;
                c.shared[at >> 5] = 0u;
            }
        }
    }
    // The slots of a particle are its lanes, x fastest, as in the explicit coupling: one OR per run of a row's lanes.
    if (a.isStep)
        staged.add(a, reactionFixed);
    if (a.isStep)
        markTouched<LANES == 64 ? 4 : LANES == 32 ? 3 : 2>(touched, node, flagged, lane);
    if (wall == nullptr)
        blockPartials(wallAcc, partials);
    else
        for (int k = 0; k < 3; k++) {
            const double sum = groupSum<LANES>(wallAcc[k]);
            if (rank < n && lane == 0)
                wall[3*(size_t) particleAt(c, rank) + k] = sum;
        }
}

/* The wall partial sums of particles that cgForces took in a processing order: by index, `group` particles to each of the
   coupling's slots (5,000 Keys particles between walls in 64^3: 145 -> 147 us a step).  done: as cgForces, nothing before the
   solve has converged. */
__global__ void __launch_bounds__(BLOCK) cgWall(const double* __restrict__ wall, int n, int group, int slots,
        double* __restrict__ partials, const double* done) {
    if (done != nullptr && *done == 0.0)
        return;
    const int item = blockIdx.x*BLOCK + threadIdx.x, slot = item/3, k = item - 3*slot;
    if (slot >= slots)
        return;
    double sum = 0.0;
    for (int i = slot*group; i < n && i < (slot + 1)*group; i++)
        sum += wall[3*(size_t) i + k];
    partials[3*(size_t) slot + k] = sum;
}

unsigned blocksOf(size_t items, int perBlock) {
    return (unsigned) ((items + perBlock - 1)/perBlock);
}

}  // namespace

struct CentredState {
    int n = 0, stencil = 0, slots = 1, lanes = 1;
    uint32_t numNodes = 0;
    // Nearest node: the radix sort of the node keys.
    uint32_t* keys = nullptr;
    uint32_t* sortedKeys = nullptr;
    int* values = nullptr;
    int* sortedValues = nullptr;
    void* sortTemp = nullptr;
    size_t sortBytes = 0;
    int sortBits = 1;
    // Stencils: conjugate gradients.
    CgArgs cg{};
    unsigned long long* sums[2] = {nullptr, nullptr};   // the two arrays of node sums, used in turn by the products
    double* partialsB = nullptr;
    double* hostScalars = nullptr;        // pinned: the convergence check reads the scalars
    int lastIterations = 1;               // iterations of the previous solve: enqueued before the first check
    bool planned = true;                  // false (LBM_AMD_CG_PLANNED=0): the host reads the residual after each
    // The matrix rows and their two arrays of directions.
    CgRows rows;
    int numCells = 0;
    double* directions[2] = {nullptr, nullptr};      // [particle][z, d]
    bool crowded = false;                            // the previous solve's rows overflowed: look before the iterations
    hipEvent_t checked = nullptr;
    std::vector<void*> buffers;
};

CentredState* centredCreate(int numParticles, int stencil, const Geometry& g) {
    CentredState* st = new CentredState();
    try {
        const uint32_t numNodes = g.n;
        int n = std::max(numParticles, 1);
        st->n = numParticles;
        st->stencil = stencil;
        st->numNodes = numNodes;
        if (const char* plannedEnv = getenv("LBM_AMD_CG_PLANNED"))
            st->planned = plannedEnv[0] != '0';
        int w = stencilWidth(stencil);
        st->slots = w*w*w;
        st->lanes = coupleLanes(stencil);
        if (stencil == LBM_STENCIL_NEAREST) {
            st->keys = alloc<uint32_t>(n);
            st->sortedKeys = alloc<uint32_t>(n);
            st->values = alloc<int>(n);
            st->sortedValues = alloc<int>(n);
            while ((1ull << st->sortBits) < numNodes)
                st->sortBits++;
            check(hipcub::DeviceRadixSort::SortPairs(nullptr, st->sortBytes, st->keys, st->sortedKeys, st->values,
                    st->sortedValues, n, 0, st->sortBits, (hipStream_t) 0), "radix sort size");
            st->sortTemp = alloc<char>(st->sortBytes);
            st->buffers = {st->keys, st->sortedKeys, st->values, st->sortedValues, st->sortTemp};
        }
        else {
            CgArgs& c = st->cg;
            c.slots = st->slots;
            c.stride = 3;
            c.rhs = alloc<double>(3*(size_t) n);
            c.diag = alloc<double>(n);
            c.F = alloc<double>(3*(size_t) n);
            c.r = alloc<double>(3*(size_t) n);
            c.z = alloc<double>(3*(size_t) n);
            c.d = alloc<double>(3*(size_t) n);
            c.Ad = alloc<double>(3*(size_t) n);
            c.slotNode = alloc<uint32_t>((size_t) n*st->slots);
            c.slotW = alloc<double>((size_t) n*st->slots);
            c.slotWInvRho = alloc<double>((size_t) n*st->slots);
            c.slotSolid = alloc<uint8_t>((size_t) n*st->slots);
            c.slotSpreads = alloc<uint8_t>((size_t) n*st->slots);
            st->sums[0] = alloc<unsigned long long>(3*(size_t) numNodes);
            st->sums[1] = alloc<unsigned long long>(3*(size_t) numNodes);
            c.spread = st->sums[0];
            c.spreadOther = st->sums[1];
            // The split for sparse particles (stencil slots under a quarter of the nodes: few share a node);
            // LBM_AMD_CG_SPLIT=0 or 1 forces the choice.
            bool sparse = (uint64_t) numParticles*(uint64_t) st->slots*4 <= (uint64_t) numNodes;
            const char* splitEnv = getenv("LBM_AMD_CG_SPLIT");
            c.split = (splitEnv ? splitEnv[0] == '1' : sparse) ? 1 : 0;
            c.seen = nullptr;
            c.shared = nullptr;
            if (c.split) {
                size_t words = ((size_t) numNodes + 31)/32;
                c.seen = alloc<uint32_t>(words);
                c.shared = alloc<uint32_t>(words);
                check(hipMemset(c.seen, 0, words*sizeof(uint32_t)), "memset");
                check(hipMemset(c.shared, 0, words*sizeof(uint32_t)), "memset");
            }
            c.partials = alloc<double>(8*RED_BLOCKS);
            c.scalars = alloc<double>(NUM_SCALARS);
            st->partialsB = alloc<double>(8*RED_BLOCKS);
            check(hipMemset(st->sums[0], 0, 3*(size_t) numNodes*sizeof(unsigned long long)), "memset");
            check(hipMemset(st->sums[1], 0, 3*(size_t) numNodes*sizeof(unsigned long long)), "memset");
            st->buffers = {c.rhs, c.diag, c.F, c.r, c.z, c.d, c.Ad, c.slotNode, c.slotW, c.slotWInvRho, c.slotSolid,
                           c.slotSpreads, st->sums[0], st->sums[1], c.partials, c.scalars, st->partialsB, c.seen,
                           c.shared};
            check(hipHostMalloc((void**) &st->hostScalars, NUM_SCALARS*sizeof(double), hipHostMallocDefault),
                    "pinned scalars");
            // The matrix rows: periodic axes of at least three cells (no stencil meets another from both sides), and rows
            // that are expected at most half full, as are the cells.  There a step by the rows was the faster one at every
            // size measured: 56,320 Keys particles in 120^3 (11 neighbours) 620 us against 1,330, 20,000 in 256^3 (0.4) 781
            // against 938, 20,000 in 48^3 (62) 310 against 546, 2,000 trilinear ones in 128^3 148 against 193.
            // LBM_AMD_CG_ROWS=0 or 1 forces the choice where the lattice allows it; LBM_AMD_CG_SPLIT chooses a spread.
            const double reach = (2.0*w - 1)*(2.0*w - 1)*(2.0*w - 1);
            const char* rowsEnv = getenv("LBM_AMD_CG_ROWS");
            const bool periodic = !g.openX && !g.openY && !g.openZ && g.nx >= 12 && g.ny >= 12 && g.nz >= 12;
            const bool want = rowsEnv ? rowsEnv[0] == '1' : splitEnv == nullptr &&
                    reach*numParticles <= ROWS_MEAN_NEIGHBOURS*numNodes && numParticles <= (4 << 20) &&
                    64.0*numParticles <= 0.5*CELL_CAP*numNodes;
            if (periodic && want) {
                CgRows& r = st->rows;
                r.cells[0] = (int) g.nx/4;
                r.cells[1] = (int) g.ny/4;
                r.cells[2] = (int) g.nz/4;
                st->numCells = r.cells[0]*r.cells[1]*r.cells[2];
                const size_t rowEntries = (size_t) n*ROW_CAP, weights = 3*(3*(size_t) w - 2)*n;
                // Without the memory for them the solves take the spread.
                if (allocateOptional({{(void**) &r.cellCount, st->numCells*sizeof(int)},
                        {(void**) &r.cell, (size_t) st->numCells*CELL_CAP*sizeof(CellEntry)},
                        {(void**) &r.home, 4*(size_t) n*sizeof(uint32_t)}, {(void**) &r.axisWeight, weights*sizeof(double)},
                        {(void**) &r.rowCount, n*sizeof(int)}, {(void**) &r.rowParticle, rowEntries*sizeof(int)},
                        {(void**) &r.rowValue, rowEntries*sizeof(double)}, {(void**) &r.overflow, sizeof(int)},
                        {(void**) &st->directions[0], 6*(size_t) n*sizeof(double)},
                        {(void**) &st->directions[1], 6*(size_t) n*sizeof(double)}}, reservedBytes(numNodes))) {
                    for (void* b : {(void*) r.cellCount, (void*) r.cell, (void*) r.home, (void*) r.axisWeight, (void*) r.rowCount,
                                    (void*) r.rowParticle, (void*) r.rowValue, (void*) r.overflow, (void*) st->directions[0],
                                    (void*) st->directions[1]})
                        st->buffers.push_back(b);
                    check(hipMemset(r.cellCount, 0, st->numCells*sizeof(int)), "memset");
                    check(hipMemset(r.axisWeight, 0, weights*sizeof(double)), "memset");
                    check(hipMemset(r.overflow, 0, sizeof(int)), "memset");
                    check(hipEventCreateWithFlags(&st->checked, hipEventDisableTiming), "event");
                }
            }
        }
    }
    catch (...) {
        centredDestroy(st);
        throw;
    }
    return st;
}

void centredDestroy(CentredState* st) {
    if (!st)
        return;
    for (void* p : st->buffers)
        if (p)
            (void) hipFree(p);
    if (st->checked)
        (void) hipEventDestroy(st->checked);
    if (st->hostScalars)
        (void) hipHostFree(st->hostScalars);
    delete st;
}

namespace {

/* Ax = A x, with the node sums in array `sums` (the gather clears the other, the previous product's).  The largest |x|
   of each block must be in c.partials (cgMaxAbs, or cgDirection for x = d).  done: the solve's convergence flag inside
   the iteration loop (nullptr outside it); first: the solve's first product. */
template <typename S>
void multiply(CentredState* st, const double* x, double* Ax, const double* mass, double aa, const double* done,
        int sums, bool first, hipStream_t stream) {
    CgArgs c = st->cg;
    c.spread = st->sums[sums];
    c.spreadOther = st->sums[1 - sums];
    int n = st->n;
    const uint32_t spreadGroups = blocksOf(3*(size_t) n*c.slots, BLOCK);
    for (uint32_t at = 0; at < spreadGroups; at += SPREAD_BLOCKS) {
        const unsigned groups = std::min(spreadGroups - at, SPREAD_BLOCKS);
        switch (st->lanes) {
        case 8: cgSpread<8><<<groups, BLOCK, 0, stream>>>(x, n, c, done, first ? 1 : 0, at); break;
        case 32: cgSpread<27><<<groups, BLOCK, 0, stream>>>(x, n, c, done, first ? 1 : 0, at); break;
        default: cgSpread<64><<<groups, BLOCK, 0, stream>>>(x, n, c, done, first ? 1 : 0, at); break;
        }
    }
    switch (st->lanes) {
    case 8: cgGather<8><<<blocksOf(n, BLOCK/8), BLOCK, 0, stream>>>(x, Ax, mass, n, aa, c, done); break;
    case 32: cgGather<32><<<blocksOf(n, BLOCK/32), BLOCK, 0, stream>>>(x, Ax, mass, n, aa, c, done); break;
    default: cgGather<64><<<blocksOf(n, BLOCK/64), BLOCK, 0, stream>>>(x, Ax, mass, n, aa, c, done); break;
    }
}

bool converged(CentredState* st, hipStream_t stream) {
    double* s = st->hostScalars;
    check(hipMemcpyAsync(s, st->cg.scalars, NUM_SCALARS*sizeof(double), hipMemcpyDeviceToHost, stream), "download");
    check(hipStreamSynchronize(stream), "sync");
    return residualConverged(s);
}

const char* const NOT_CONVERGED = "LBMForce: the centred drag with the interpolation stencil did not converge in 1000 "
        "iterations of the conjugate gradients";

/*
 * The solve with the matrix rows, after cgSetup has binned the particles.  The forces (a launch that does nothing before the
 * solve has converged) go onto the stream ahead of the host's wait for the residual, so that the device works meanwhile.
 * Returns false if a bin or a row was too small; c.F and the slots are then as cgSetup left them.  After such a solve the
 * host looks for that before it enqueues iterations that would do nothing.
 */
template <typename Forces>
bool solveRows(CentredState* st, const Geometry& g, const double* mass, double aa, hipStream_t stream, Forces&& forces) {
    CgArgs c = st->cg;
    const CgRows& r = st->rows;
    const int n = st->n, nx = (int) g.nx, ny = (int) g.ny, nz = (int) g.nz;
    const unsigned waves = blocksOf(n, BLOCK/64);
    switch (st->lanes) {
    case 8: cgRows<2><<<waves, BLOCK, 0, stream>>>(n, nx, ny, nz, c, r, mass, aa); break;
    case 32: cgRows<3><<<waves, BLOCK, 0, stream>>>(n, nx, ny, nz, c, r, mass, aa); break;
    default: cgRows<4><<<waves, BLOCK, 0, stream>>>(n, nx, ny, nz, c, r, mass, aa); break;
    }
    c.stride = 6;
    c.z = st->directions[0];
    c.d = c.z + 3;
    cgInit<<<RED_BLOCKS, BLOCK, 0, stream>>>(n, c, st->partialsB, r.cellCount, st->numCells);
    cgFinishInit<<<1, 64, 0, stream>>>(c.partials, st->partialsB, c.scalars, r.overflow);
    int iteration = 0;
    const int planned = st->planned ? std::max(st->lastIterations, 1) : 1;
    for (int batch = st->crowded ? 0 : planned;; batch = iteration == 0 ? planned : 1) {
        for (int b = 0; b < batch; b++, iteration++) {
            c.z = st->directions[(iteration + 1) & 1];
            c.d = c.z + 3;
            cgRowsStep<<<RED_BLOCKS, ROW_THREADS_CG, 0, stream>>>(n, c, r, st->directions[iteration & 1], c.z, mass, aa,
                    st->partialsB, iteration);
            cgUpdate<<<RED_BLOCKS, BLOCK, 0, stream>>>(n, c, st->partialsB, c.scalars + DONE, RZ + RZ_SLOT*(iteration & 1));
        }
        cgRowsCheck<<<1, 64, 0, stream>>>(st->partialsB, c.scalars, r.overflow, iteration, st->hostScalars);
        check(hipEventRecord(st->checked, stream), "event");
        forces();
        check(hipGetLastError(), "launch");
        check(hipEventSynchronize(st->checked), "sync");
        st->crowded = st->hostScalars[OVERFLOWED] != 0.0;
        if (st->crowded) {
            check(hipMemsetAsync(r.overflow, 0, sizeof(int), stream), "memset");
            return false;
        }
        if (st->hostScalars[DONE] != 0.0)
            break;
        if (iteration >= CG_MAX_ITERATIONS)
            throw std::runtime_error(NOT_CONVERGED);
    }
    st->lastIterations = (int) st->hostScalars[ITERS];
    return true;
}

template <typename S>
void centredCoupleT(CentredState* st, const S* src, const uint32_t* mask, const double* positions,
        const double* velocities, const double* otherForces, const int* particles, const double* mass,
        const double* ucm, const ParticleArgs& a, const double g[3], const double4* field, const int* order,
        const SpreadBins* bins, double* particleForce, double* systemForce, unsigned long long* reactionFixed, uint32_t* touched,
        double* partials, hipStream_t stream) {
    int n = a.numParticles;
    if (n == 0)
        return;
    if (st->stencil == LBM_STENCIL_NEAREST) {
        centredKeys<<<blocksOf(n, BLOCK), BLOCK, 0, stream>>>(positions, particles, a, st->keys, st->values);
        size_t bytes = st->sortBytes;
        check(hipcub::DeviceRadixSort::SortPairs(st->sortTemp, bytes, st->keys, st->sortedKeys, st->values,
                st->sortedValues, n, 0, st->sortBits, stream), "radix sort");
        centredNearest<S><<<blocksOf(n, BLOCK), BLOCK, 0, stream>>>(src, mask, velocities, otherForces, particles, mass,
                ucm, a, g[0], g[1], g[2], st->sortedKeys, st->sortedValues, particleForce, reactionFixed, touched, partials);
        check(hipGetLastError(), "launch");
        return;
    }
    CgArgs& c = st->cg;
    c.order = order;
    double aa = 0.5*a.gamma;
    unsigned groups = blocksOf(n, BLOCK/st->lanes);
    auto setup = [&](const CgRows& rows) {
        switch (st->lanes) {
        case 8:
            cgSetup<S, 8><<<groups, BLOCK, 0, stream>>>(src, mask, positions, velocities, otherForces, particles, mass, ucm, a,
                    g[0], g[1], g[2], c, field, rows);
            break;
        case 32:
            cgSetup<S, 32><<<groups, BLOCK, 0, stream>>>(src, mask, positions, velocities, otherForces, particles, mass, ucm,
                    a, g[0], g[1], g[2], c, field, rows);
            break;
        default:
            cgSetup<S, 64><<<groups, BLOCK, 0, stream>>>(src, mask, positions, velocities, otherForces, particles, mass, ucm,
                    a, g[0], g[1], g[2], c, field, rows);
            break;
        }
    };
    SpreadBins spread;
    if (bins != nullptr && a.isStep) {
        spread = *bins;
        spread.slotWeight = c.slotW;
        spread.weightStride = c.slots;
    }
    // The particles' wall momentum, where their places in the launch depend on the order: in c.Ad, which a solve is done with.
    double* wall = order != nullptr && partials != nullptr ? c.Ad : nullptr;
    auto forces = [&](const int* rowCount) {
        auto launch = [&](auto binned) {
            constexpr bool B = decltype(binned)::value;
            switch (st->lanes) {
            case 8:
                cgForces<8, B><<<groups, BLOCK, 0, stream>>>(n, a, c, particleForce, reactionFixed, touched, partials, wall, rowCount,
                        spread, particles, systemForce);
                break;
            case 32:
                cgForces<32, B><<<groups, BLOCK, 0, stream>>>(n, a, c, particleForce, reactionFixed, touched, partials, wall, rowCount,
                        spread, particles, systemForce);
                break;
            default:
                cgForces<64, B><<<groups, BLOCK, 0, stream>>>(n, a, c, particleForce, reactionFixed, touched, partials, wall, rowCount,
                        spread, particles, systemForce);
                break;
            }
        };
        if (spread.count == nullptr)
            launch(std::false_type());
        else {
            launch(std::true_type());
            launchSpreadTiles(mask, a, spread, reactionFixed, touched, stream);
        }
        if (wall != nullptr)
            cgWall<<<blocksOf(3*(size_t) groups, BLOCK), BLOCK, 0, stream>>>(wall, n, BLOCK/st->lanes, (int) groups, partials,
                    rowCount != nullptr ? c.scalars + DONE : nullptr);
    };
    setup(st->rows);
    if (st->rows.cell != nullptr && solveRows(st, a.g, mass, aa, stream, [&] { forces(st->rows.rowCount); }))
        return;
    if (c.split)
        switch (st->lanes) {
        case 8: cgMarkShared<8><<<groups, BLOCK, 0, stream>>>(n, c); break;
        case 32: cgMarkShared<32><<<groups, BLOCK, 0, stream>>>(n, c); break;
        default: cgMarkShared<64><<<groups, BLOCK, 0, stream>>>(n, c); break;
        }
    cgMaxAbs<<<RED_BLOCKS, BLOCK, 0, stream>>>(c.F, n, c.partials, nullptr);
    multiply<S>(st, c.F, c.Ad, mass, aa, nullptr, 1, true, stream);
    cgInit<<<RED_BLOCKS, BLOCK, 0, stream>>>(n, c, st->partialsB, nullptr, 0);
    cgFinishInit<<<1, 64, 0, stream>>>(c.partials, st->partialsB, c.scalars, nullptr);
    check(hipGetLastError(), "launch");
    // Each iteration starts with the new direction (d = z after cgInit), so that the last one computes none.  The
    // previous solve's count of iterations is enqueued at once (those after convergence do nothing), then the host
    // reads the residual and adds one iteration at a time until it has converged.
    const double* done = c.scalars + DONE;
    int iteration = 0;
    for (int batch = st->planned ? std::max(st->lastIterations, 1) : 1;; batch = 1) {
        for (int b = 0; b < batch; b++, iteration++) {
            if (iteration == 0)
                cgMaxAbs<<<RED_BLOCKS, BLOCK, 0, stream>>>(c.d, n, c.partials, done);
            else
                cgDirection<<<RED_BLOCKS, BLOCK, 0, stream>>>(n, c, done);
            multiply<S>(st, c.d, c.Ad, mass, aa, done, iteration & 1, false, stream);
            cgDot<<<RED_BLOCKS, BLOCK, 0, stream>>>(n, c, done);
            cgUpdate<<<RED_BLOCKS, BLOCK, 0, stream>>>(n, c, st->partialsB, done, RZ);
            cgFinishBeta<<<1, 64, 0, stream>>>(st->partialsB, c.scalars, done);
            check(hipGetLastError(), "launch");
        }
        if (converged(st, stream))
            break;
        if (iteration >= CG_MAX_ITERATIONS) {
            // cgForces, which clears the node sums and bits after a solve, does not run: clear them here, so that a
            // caller who goes on after the error starts the next solve from zero.
            const size_t sumBytes = 3*(size_t) st->numNodes*sizeof(unsigned long long);
            check(hipMemsetAsync(st->sums[0], 0, sumBytes, stream), "memset");
            check(hipMemsetAsync(st->sums[1], 0, sumBytes, stream), "memset");
            if (c.split) {
                const size_t bitBytes = (((size_t) st->numNodes + 31)/32)*sizeof(uint32_t);
                check(hipMemsetAsync(c.seen, 0, bitBytes, stream), "memset");
                check(hipMemsetAsync(c.shared, 0, bitBytes, stream), "memset");
            }
            throw std::runtime_error(NOT_CONVERGED);
        }
    }
    st->lastIterations = (int) st->hostScalars[ITERS];
    forces(nullptr);
    check(hipGetLastError(), "launch");
}

}  // namespace

void centredCouple(CentredState* st, int storage, const void* src, const uint32_t* mask, const double* positions,
        const double* velocities, const double* otherForces, const int* particles, const double* mass,
        const double* ucm, const ParticleArgs& a, const double g[3], const double4* field, const int* order,
        const SpreadBins* bins, double* particleForce, double* systemForce, unsigned long long* reactionFixed, uint32_t* touched,
        double* partials, hipStream_t stream) {
    switch (storage) {
    case LBM_STORAGE_FP16:
        centredCoupleT<__half>(st, (const __half*) src, mask, positions, velocities, otherForces, particles, mass, ucm, a,
                g, field, order, bins, particleForce, systemForce, reactionFixed, touched, partials, stream);
        break;
    case LBM_STORAGE_BF16:
        centredCoupleT<__hip_bfloat16>(st, (const __hip_bfloat16*) src, mask, positions, velocities, otherForces,
                particles, mass, ucm, a, g, field, order, bins, particleForce, systemForce, reactionFixed, touched, partials, stream);
        break;
    case LBM_STORAGE_FP64:
        centredCoupleT<double>(st, (const double*) src, mask, positions, velocities, otherForces, particles, mass, ucm, a,
                g, field, order, bins, particleForce, systemForce, reactionFixed, touched, partials, stream);
        break;
    default:
        centredCoupleT<float>(st, (const float*) src, mask, positions, velocities, otherForces, particles, mass, ucm, a,
                g, field, order, bins, particleForce, systemForce, reactionFixed, touched, partials, stream);
        break;
    }
}

}  // namespace lbm
