/*
 * Coupling kernels of the learned closure (include/lbm_amd_closure.h).
 *
 *  closureStep      one wave per 16 particles: the network's inputs, built in LDS in the particle's frame (below) from the
 *                   27 nodes around the nearest node (u = j/rho in FP64, as the stencil coupling forms it), the sub-node
 *                   offset and the particle's velocity; the network on them (FP16 MFMA); the nearest-node drag with
 *                   u(nearest) + du (du turned back from the frame) and its reaction on the nearest node, exactly as the
 *                   nearest-node stencil coupling computes them (ReferenceLBMKernels.cpp:503-553): with du = 0 the two are
 *                   identical bit for bit.  A particle is out of distribution if a normalized velocity exceeds its bound,
 *                   a neighbour is solid, or the neighbourhood leaves the lattice at an open face: it is flagged and left.
 *  closureFallback  the Keys coupling of the flagged particles (ReferenceLBMKernels.cpp:643-697): fixed grid, each wave
 *                   scans the flags of 64 particles at a time with a fixed stride, so the wall partial sums have a fixed
 *                   order.
 *  closureField     u of every node, for closureStep where the particles are dense.
 *  closureFeatures  the same inputs for training pairs, raw, one group of 32 lanes per particle.
 *  closureTargets   u_Keys(x) - u(nearest) with the stencil interpolation of the coupling, in the particle's frame
 *                   (training pairs).
 *
 * The particle's frame: the Keys stencil and the lattice are symmetric under the 48 reflections and axis permutations
 * of the cube, so the network sees every particle after the one that makes its sub-node offset o non-negative and
 * sorted, o'_0 >= o'_1 >= o'_2 >= 0: frame axis i is lattice axis p_i, reflected where o_(p_i) < 0 (sign s_i = -1).
 * A vector w of the lattice frame has w'_i = s_i w_(p_i) there, and the node nearest + d sits at d'_i = s_i d_(p_i) of
 * the 3x3x3 block.  The network then learns on a 48th of the offsets' cube.
 */
#include "lbm_coupling.h"
#include "lbm_mlp.h"

namespace lbm {

namespace {

constexpr int FEATURE_LANES = 32;
constexpr int FALLBACK_MAX_BLOCKS = 512;

/* The frame of a particle whose sub-node offset is o (FP64): bit k set where lattice axis k is reflected (o_k < 0);
   bits 3-4 and 5-6 hold p_0 and p_1, the lattice axes of frame axes 0 and 1 (p_2 = 3 - p_0 - p_1), ordered by |o|
   from the largest, equal values in axis order. */
__device__ __forceinline__ uint8_t frameCode(const double o[3]) {
    double m[3];
    unsigned code = 0;
    for (int k = 0; k < 3; k++) {
        m[k] = fabs(o[k]);
        if (o[k] < 0)
            code |= 1u << k;
    }
    // Rank of each axis: the axes that precede it.
    int r0 = (m[1] > m[0]) + (m[2] > m[0]);
    int r1 = (m[0] >= m[1]) + (m[2] > m[1]);
    int p0 = r0 == 0 ? 0 : (r1 == 0 ? 1 : 2);
    int p1 = r0 == 1 ? 0 : (r1 == 1 ? 1 : 2);
    return (uint8_t) (code | (unsigned) p0 << 3 | (unsigned) p1 << 5);
}

struct Frame {
    int axis[3];      // p_i: the lattice axis of frame axis i
    double sign[3];   // s_i: -1 where that lattice axis is reflected
};

__device__ __forceinline__ Frame frameOf(unsigned code) {
    Frame f;
    f.axis[0] = (int) (code >> 3) & 3;
    f.axis[1] = (int) (code >> 5) & 3;
    f.axis[2] = 3 - f.axis[0] - f.axis[1];
    for (int i = 0; i < 3; i++)
        f.sign[i] = (code >> f.axis[i]) & 1u ? -1.0 : 1.0;
    return f;
}

/* v[k] for a lane-varying k, by selects (no indexed private array). */
template <typename T>
__device__ __forceinline__ T pick(const T v[3], int k) {
    return k == 0 ? v[0] : (k == 1 ? v[1] : v[2]);
}

template <typename S>
__global__ void __launch_bounds__(BLOCK) closureFeatures(const S* __restrict__ src, const uint32_t* __restrict__ mask,
        const double* __restrict__ positions, const double* __restrict__ velocities, const int* __restrict__ particles,
        const double* __restrict__ ucm, ParticleArgs a, float* __restrict__ raw, double* __restrict__ centreVelocity,
        uint8_t* __restrict__ frame) {
    constexpr int GROUPS = BLOCK/FEATURE_LANES;
    int lane = threadIdx.x % FEATURE_LANES;
    int i = blockIdx.x*GROUPS + threadIdx.x/FEATURE_LANES;
    bool active = i < a.numParticles;
    int part = active ? particles[i] : 0;
    const double* x = positions + 3*(size_t) part;
    int size[3] = {(int) a.g.nx, (int) a.g.ny, (int) a.g.nz};
    // The wrapped coordinate and the nearest node of axis k (FP64, as the coupling computes them) by the group's lane k,
    // shared with the others; every lane then forms the particle's frame from the three offsets.  The axis length is
    // selected, not indexed by the lane (a lane-varying index into the kernel argument's fields would be read once for
    // the whole wavefront).
    double swLane = 0.0;
    int nearLane = 0;
    if (active && lane < 3) {
        const int axisSize = lane == 0 ? size[0] : (lane == 1 ? size[1] : size[2]);
        swLane = wrapCoordinate(x[lane], a.dx, axisSize);
        nearLane = nearestIndex(swLane, axisSize);
    }
    double sw[3], o[3];
    int near[3];
    for (int k = 0; k < 3; k++) {
        sw[k] = __shfl(swLane, k, FEATURE_LANES);
        near[k] = __shfl(nearLane, k, FEATURE_LANES);
        o[k] = sw[k] - floor(sw[k] + 0.5);
    }
    const int code = frameCode(o);
    if (active && lane == 0)
        frame[i] = (uint8_t) code;
    const Frame fr = frameOf((unsigned) code);
    if (active) {
        float* ri = raw + (size_t) i*MLP_IN;
        if (lane < 27) {
            int d[3] = {lane % 3 - 1, (lane/3) % 3 - 1, lane/9 - 1};
            int idx[3];
            for (int k = 0; k < 3; k++) {
                int t = near[k] + d[k];
                if (t < 0 || t >= size[k])
                    t = (t + size[k]) % size[k];
                idx[k] = t;
            }
            uint32_t node = (uint32_t) (idx[0] + (int) a.g.nx*(idx[1] + (int) a.g.ny*idx[2]));
            double u[3] = {0, 0, 0};
            if (!solidAt(mask, node))
                nodeVelocity(src, a.g, node, ucm, a.removal, 1.0, u);
            if (lane == 13)
                for (int c = 0; c < 3; c++)
                    centreVelocity[3*(size_t) i + c] = u[c];
            // This node's place in the particle's frame, and its velocity there.
            int slot = 13;
            for (int k = 0, stride = 1; k < 3; k++, stride *= 3)
                slot += stride*(fr.sign[k] < 0 ? -pick(d, fr.axis[k]) : pick(d, fr.axis[k]));
            for (int c = 0; c < 3; c++)
                ri[3 + 3*slot + c] = (float) (fr.sign[c]*pick(u, fr.axis[c]));
        }
        else if (lane == 27) {
            float r[3];
            for (int k = 0; k < 3; k++)
                r[k] = (float) (2.0*(sw[k] - floor(sw[k] + 0.5)));
            for (int c = 0; c < 3; c++)
                ri[c] = fabsf(pick(r, fr.axis[c]));
        }
        else if (lane == 28) {
            const double* v = velocities + 3*(size_t) part;
            for (int c = 0; c < 3; c++)
                ri[84 + c] = (float) (fr.sign[c]*pick(v, fr.axis[c])/a.velocityScale);
        }
    }
}

/* u = j/rho of every fluid node (zero at solid nodes), FP64, [node][3]: one coalesced pass over the populations that
   replaces the 27 scattered pulls per particle when the particles are dense. */
template <typename S>
__global__ void __launch_bounds__(BLOCK) closureField(const S* __restrict__ src, const uint32_t* __restrict__ mask,
        const double* __restrict__ ucm, ParticleArgs a, double* __restrict__ field) {
    uint32_t node = blockIdx.x*BLOCK + threadIdx.x;
    if (node >= a.g.n)
        return;
    double u[3] = {0, 0, 0};
    if (!solidAt(mask, node))
        nodeVelocity(src, a.g, node, ucm, a.removal, 1.0, u);
    for (int c = 0; c < 3; c++)
        field[3*(size_t) node + c] = u[c];
}

template <typename S>
__global__ void __launch_bounds__(BLOCK) closureTargets(const S* __restrict__ src, const uint32_t* __restrict__ mask,
        const double* __restrict__ positions, const int* __restrict__ particles, const double* __restrict__ ucm,
        ParticleArgs a, const double* __restrict__ centreVelocity, const uint8_t* __restrict__ frame,
        float* __restrict__ targets) {
    constexpr int LANES = 64, GROUPS = BLOCK/LANES;
    int lane = threadIdx.x % LANES;
    int i = blockIdx.x*GROUPS + threadIdx.x/LANES;
    bool active = i < a.numParticles;
    int part = active ? particles[i] : 0;
    double u[3];
    interpolateGroup<S, LANES>(src, mask, positions + 3*(size_t) part, active, lane, ucm, a, u);
    if (active && lane == 0) {
        const Frame fr = frameOf(frame[i]);
        double du[3];
        for (int c = 0; c < 3; c++)
            du[c] = u[c] - centreVelocity[3*(size_t) i + c];
        for (int c = 0; c < 3; c++)
            targets[3*(size_t) i + c] = (float) (fr.sign[c]*pick(du, fr.axis[c]));
    }
}

constexpr int CLOSURE_WAVES = 8;          // waves per work-group of closureStep, 16 particles each
constexpr int CLOSURE_TILE = 16;
// Halves per row of the operands in LDS: 8-byte aligned, and the 16 rows x 4 quads of an operand spread over the banks.
constexpr int CLOSURE_X = MLP_IN_PAD + 4, CLOSURE_H = MLP_H + 8;

struct ClosureWeights {
    _Float16 w1[MLP_H*CLOSURE_X], w2[MLP_H*CLOSURE_H], w3[MLP_OUT_PAD*CLOSURE_H];
    float b1[MLP_H], b2[MLP_H], b3[MLP_OUT_PAD];
};

struct ClosureTile {
    _Float16 x[CLOSURE_TILE][CLOSURE_X];     // normalized inputs
    double u[CLOSURE_TILE][3];               // u(nearest)
    int near[CLOSURE_TILE][3];               // the nearest node along each axis
    float du[CLOSURE_TILE][3];               // the network's output
    uint32_t node[CLOSURE_TILE];             // the nearest node
    int code[CLOSURE_TILE];                  // the frame
    int ood[CLOSURE_TILE];
};

/* LDS written by other lanes of this wavefront, visible from here on. */
__device__ __forceinline__ void waveFence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/* Node `d` (0 .. 26, x fastest) of the block around particle b's nearest node; returns whether the particle may use it. */
__device__ __forceinline__ bool blockNode(const ClosureTile& tile, int b, const int d[3], const uint32_t* mask,
        const ParticleArgs& a, uint32_t& node) {
    const int size[3] = {(int) a.g.nx, (int) a.g.ny, (int) a.g.nz}, open[3] = {a.g.openX, a.g.openY, a.g.openZ};
    bool inside = true;
    int idx[3];
    for (int k = 0; k < 3; k++) {
        int t = tile.near[b][k] + d[k];
        if (t < 0 || t >= size[k]) {
            if (open[k])
                inside = false;
            t = (t + size[k]) % size[k];
        }
        idx[k] = t;
    }
    node = (uint32_t) (idx[0] + (int) a.g.nx*(idx[1] + (int) a.g.ny*idx[2]));
    return inside && !solidAt(mask, node);
}

/*
 * The whole coupling of the particles in distribution.  Bound by the latency of its gathers (27 node velocities per
 * particle) and, beside them, by the issue of the 128 divisions and exponentials per particle; nothing of a particle leaves
 * the wave between its position and its force.  In four kernels (inputs, network, drag, addition to the caller's forces),
 * which passed 192 B of inputs and 70 B of results per particle through memory, 100,000 chain beads in 128^3 took 37 + 18 +
 * 21 + 5 us; this takes 49 us.  FIELD: node velocities from closureField, all of a wave's in flight at once.  SHARED: the
 * work-group's waves share one tile's nodes and its first wave takes the rest (closureShares).
 */
template <typename S, bool FIELD, bool SHARED>
__global__ void __launch_bounds__(64*CLOSURE_WAVES) closureStep(const S* __restrict__ src, const uint32_t* __restrict__ mask,
        const double* __restrict__ positions, const double* __restrict__ velocities, const int* __restrict__ particles,
        const double* __restrict__ mass, const double* __restrict__ ucm, ParticleArgs a, ClosureNorm norm, float outInv,
        const MlpDevice* __restrict__ weights, const double* __restrict__ field, uint8_t* __restrict__ ood,
        double* __restrict__ particleForce, double* __restrict__ systemForces,
        unsigned long long* __restrict__ reactionFixed, uint32_t* __restrict__ touched,
        unsigned long long* __restrict__ counters) {
    __shared__ __align__(16) ClosureWeights w;
    constexpr int TILES = SHARED ? 1 : CLOSURE_WAVES;
    __shared__ __align__(16) ClosureTile tiles[TILES];
    __shared__ unsigned counts[TILES][2];
    constexpr int THREADS = 64*CLOSURE_WAVES;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    ClosureTile& tile = tiles[SHARED ? 0 : wave];
    const bool mine = !SHARED || wave == 0;        // this wave takes the tile's particles, not only their nodes
    for (int j = threadIdx.x; j < MLP_H*MLP_IN_PAD/4; j += THREADS)
        *(half4_t*) (w.w1 + j/(MLP_IN_PAD/4)*CLOSURE_X + 4*(j % (MLP_IN_PAD/4))) = load4(weights->w1t + 4*j);
    for (int j = threadIdx.x; j < MLP_H*MLP_H/4; j += THREADS)
        *(half4_t*) (w.w2 + j/(MLP_H/4)*CLOSURE_H + 4*(j % (MLP_H/4))) = load4(weights->w2t + 4*j);
    for (int j = threadIdx.x; j < MLP_OUT_PAD*MLP_H/4; j += THREADS)
        *(half4_t*) (w.w3 + j/(MLP_H/4)*CLOSURE_H + 4*(j % (MLP_H/4))) = load4(weights->w3t + 4*j);
    if (threadIdx.x < MLP_H) {
        w.b1[threadIdx.x] = weights->b1[threadIdx.x];
        w.b2[threadIdx.x] = weights->b2[threadIdx.x];
    }
    if (threadIdx.x < MLP_OUT_PAD)
        w.b3[threadIdx.x] = weights->b3[threadIdx.x];
    // Four lanes per particle, lane k < 3 for axis k: coordinate, nearest node, frame, offset and particle velocity (the
    // axis length is selected, not indexed by the lane: a lane-varying index into the kernel argument's fields would be
    // read once for the whole wavefront).
    const int first = ((int) blockIdx.x*TILES + (SHARED ? 0 : wave))*CLOSURE_TILE;
    const int b = lane >> 2, k = lane & 3, i = first + b;
    const bool active = mine && i < a.numParticles;
    const int part = active ? particles[i] : 0;
    double sw = 0.0, offset = 0.0, velocity = 0.0;
    int near = 0;
    if (active && k < 3) {
        const int nx = (int) a.g.nx, ny = (int) a.g.ny, nz = (int) a.g.nz;
        const int size = k == 0 ? nx : (k == 1 ? ny : nz);
        velocity = velocities[3*(size_t) part + k];
        sw = wrapCoordinate(positions[3*(size_t) part + k], a.dx, size);
        near = nearestIndex(sw, size);
        offset = sw - floor(sw + 0.5);
    }
    double o[3];
    for (int c = 0; c < 3; c++)
        o[c] = __shfl(offset, (lane & ~3) + c, 64);
    const int code = frameCode(o);
    const Frame fr = frameOf((unsigned) code);
    const int at = fr.axis[0] == k ? 0 : (fr.axis[1] == k ? 1 : 2);      // the frame axis of lattice axis k
    const double sign = (code >> k) & 1 ? -1.0 : 1.0;                    // and its reflection
    if (mine && k == 3) {
        tile.code[b] = code;
        tile.ood[b] = 0;
        for (int c = MLP_IN; c < MLP_IN_PAD; c++)
            tile.x[b][c] = (_Float16) 0.0f;
    }
    waveFence();
    if (mine && k < 3) {
        tile.near[b][k] = near;
        tile.x[b][at] = toHalf(fabsf((float) (2.0*(sw - floor(sw + 0.5)))));
        const float r = (float) (sign*velocity/a.velocityScale);
        if (!(fabsf(r*norm.vScale) <= norm.vBound))
            tile.ood[b] = 1;
        tile.x[b][84 + at] = productToHalf(r, norm.vScale);
    }
    if constexpr (SHARED)
        __syncthreads();
    else
        waveFence();
    // The velocities of the 27 nodes of each particle, one lane per node.
    constexpr int ITEMS = 27*CLOSURE_TILE, LANES = SHARED ? THREADS : 64, ROUNDS = (ITEMS + LANES - 1)/LANES;
    const int place = SHARED ? (int) threadIdx.x : lane;
    constexpr int BATCH = FIELD ? ROUNDS : 1;
    for (int base = 0; base < ROUNDS; base += BATCH) {
        double u[BATCH][3];
        uint32_t node[BATCH];
        bool good[BATCH];
#pragma unroll
        for (int q = 0; q < BATCH; q++) {
            const int item = place + LANES*(base + q), p = item/27, j = item - 27*p;
            const int d[3] = {j % 3 - 1, (j/3) % 3 - 1, j/9 - 1};
            u[q][0] = u[q][1] = u[q][2] = 0.0;
            node[q] = 0;
            good[q] = true;
            if (item < ITEMS && first + p < a.numParticles) {
                good[q] = blockNode(tile, p, d, mask, a, node[q]);
                if (!solidAt(mask, node[q])) {
                    if constexpr (FIELD) {
                        for (int c = 0; c < 3; c++)
                            u[q][c] = field[3*(size_t) node[q] + c];
                    }
                    else
                        nodeVelocity(src, a.g, node[q], ucm, a.removal, 1.0, u[q]);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < BATCH; q++) {
            const int item = place + LANES*(base + q), p = item/27, j = item - 27*p;
            if (item >= ITEMS || first + p >= a.numParticles)
                continue;
            const int d[3] = {j % 3 - 1, (j/3) % 3 - 1, j/9 - 1};
            if (j == 13) {
                tile.node[p] = node[q];
                for (int c = 0; c < 3; c++)
                    tile.u[p][c] = u[q][c];
            }
            // This node's place in the particle's frame, and its velocity there.
            const Frame f = frameOf((unsigned) tile.code[p]);
            int slot = 13;
            for (int c = 0, stride = 1; c < 3; c++, stride *= 3)
                slot += stride*(f.sign[c] < 0 ? -pick(d, f.axis[c]) : pick(d, f.axis[c]));
            bool out = !good[q];
            for (int c = 0; c < 3; c++) {
                const float r = (float) (f.sign[c]*pick(u[q], f.axis[c]));
                if (!(fabsf(r*norm.uScale) <= norm.uBound))
                    out = true;
                tile.x[p][3 + 3*slot + c] = productToHalf(r, norm.uScale);
            }
            if (out)
                tile.ood[p] = 1;
        }
    }
    __syncthreads();                         // the weights; the tile
    if (!mine)
        return;
    // The network (the sums of forwardTile, lbm_mlp.hip).
    const int row = lane & 15, quad = (lane >> 4)*4;
    half4_t h1[4], h2[4];
    {
        half4_t x[6];
#pragma unroll
        for (int s = 0; s < 6; s++)
            x[s] = load4(&tile.x[row][16*s + quad]);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            float4_t acc = *(const float4_t*) (w.b1 + 16*t + quad);
#pragma unroll
            for (int s = 0; s < 6; s++)
                acc = mfma16(load4(w.w1 + (16*t + row)*CLOSURE_X + 16*s + quad), x[s], acc);
#pragma unroll
            for (int r = 0; r < 4; r++)
                h1[t][r] = toHalf(siluf(acc[r]));
        }
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        float4_t acc = *(const float4_t*) (w.b2 + 16*t + quad);
#pragma unroll
        for (int s = 0; s < 4; s++)
            acc = mfma16(load4(w.w2 + (16*t + row)*CLOSURE_H + 16*s + quad), h1[s], acc);
#pragma unroll
        for (int r = 0; r < 4; r++)
            h2[t][r] = toHalf(siluf(acc[r]));
    }
    float4_t y = *(const float4_t*) (w.b3 + quad);
#pragma unroll
    for (int s = 0; s < 4; s++)
        y = mfma16(load4(w.w3 + row*CLOSURE_H + 16*s + quad), h2[s], y);
    if (quad == 0)
        for (int r = 0; r < MLP_OUT; r++)
            tile.du[row][r] = y[r]*outInv;
    waveFence();
    // The drag, lane k < 3 for component k, in the terms of dragForce: du is in the particle's frame, lattice component p_c
    // is s_c du_c.
    const bool fallback = active && tile.ood[b] != 0, network = active && !fallback;
    long long fixed = 0;
    uint32_t node = 0;
    if (network && k < 3) {
        const double u = tile.u[b][k] + sign*(double) tile.du[b][at];
        const double m = mass[i];
        const double v = velocity/a.velocityScale;
        double f = (v - u)*(-a.gamma*m);
        if (a.randomForce)
            f += particleNormal((uint32_t) i, k, a)*sqrt(2.0*a.gamma*m*a.kT);
        particleForce[3*(size_t) i + k] = f*a.forceScale;
        if (systemForces != nullptr)
            atomicAdd(systemForces + 3*(size_t) part + k, f*a.forceScale);
        node = tile.node[b];
        if (a.isStep && reactionInRange(-f, a.overflow)) {
            fixed = llrint(-f*FIXED_SCALE);
            if (fixed != 0)
                __hip_atomic_fetch_add(asGlobal(reactionFixed + reactionIndex(node, k, a.g.n, a.reactionPlanes)),
                        (unsigned long long) fixed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    const unsigned long long moved = __ballot(fixed != 0);
    if (k == 0 && ((moved >> lane) & 7ull) != 0ull)
        __hip_atomic_fetch_or(asGlobal(touched + (node >> 5)), 1u << (node & 31), __ATOMIC_RELAXED,
                __HIP_MEMORY_SCOPE_AGENT);
    if (active && k == 0)
        ood[i] = fallback ? 1 : 0;
    // The work-group's counts, added to its own pair of counters (one writer each: no atomics on a shared word).
    const unsigned long long net = __ballot(network && k == 0), fall = __ballot(fallback && k == 0);
    if (lane == 0) {
        counts[SHARED ? 0 : wave][0] = (unsigned) __popcll(net);
        counts[SHARED ? 0 : wave][1] = (unsigned) __popcll(fall);
    }
    if constexpr (SHARED)
        waveFence();
    else
        __syncthreads();
    if (threadIdx.x < 2) {
        unsigned sum = 0;
        for (int v = 0; v < TILES; v++)
            sum += counts[v][threadIdx.x];
        counters[2*blockIdx.x + threadIdx.x] += sum;
    }
}

template <typename S>
__global__ void __launch_bounds__(BLOCK) closureFallback(const S* __restrict__ src, const uint32_t* __restrict__ mask,
        const double* __restrict__ positions, const double* __restrict__ velocities, const int* __restrict__ particles,
        const double* __restrict__ mass, const double* __restrict__ ucm, ParticleArgs a, const uint8_t* __restrict__ ood,
        double* __restrict__ particleForce, double* __restrict__ systemForces,
        unsigned long long* __restrict__ reactionFixed, uint32_t* __restrict__ touched, double* __restrict__ partials) {
    constexpr int LANES = 64;
    int lane = threadIdx.x % LANES;
    int wave = blockIdx.x*(BLOCK/LANES) + threadIdx.x/LANES;
    int waves = gridDim.x*(BLOCK/LANES);
    double acc[3] = {0, 0, 0};
    // Each wave reads the flags of 64 particles at a time and couples the flagged ones one after another, all 64 lanes
    // on the 64 slots of the Keys stencil: a fixed assignment and order, so the wall partial sums are reproducible.
    for (int base = wave*LANES; base < a.numParticles; base += waves*LANES) {
        int j = base + lane;
        unsigned long long votes = __ballot(j < a.numParticles && ood[j] != 0);
        while (votes != 0ull) {
            int i = base + __ffsll((long long) votes) - 1;
            votes &= votes - 1ull;
            int part = particles[i];
            double wallAcc[3] = {0, 0, 0};
            coupleGroup<S, LANES>(src, mask, positions + 3*(size_t) part, velocities + 3*(size_t) part, (uint32_t) i,
                    mass[i], true, lane, ucm, a, particleForce + 3*(size_t) i, reactionFixed, touched, wallAcc, nullptr,
                    systemForces != nullptr ? systemForces + 3*(size_t) part : nullptr);
            for (int k = 0; k < 3; k++)
                acc[k] += wallAcc[k];
        }
    }
    if (partials != nullptr)
        storeWallPartial<BLOCK>(acc, partials);
}

unsigned gridOf(int64_t items, int perBlock) {
    return (unsigned) ((items + perBlock - 1)/perBlock);
}

}  // namespace

#define LBM_CLOSURE_STORAGE(storage, CALL) \
    switch (storage) { \
    case LBM_STORAGE_FP16: { using S = __half; CALL; break; } \
    case LBM_STORAGE_BF16: { using S = __hip_bfloat16; CALL; break; } \
    case LBM_STORAGE_FP64: { using S = double; CALL; break; } \
    default: { using S = float; CALL; break; } \
    }

void launchClosureFeatures(int storage, const void* src, const uint32_t* mask, const double* positions,
        const double* velocities, const int* particles, const double* ucm, const ParticleArgs& a, float* raw,
        double* centreVelocity, uint8_t* frame, hipStream_t stream) {
    if (a.numParticles == 0)
        return;
    unsigned grid = gridOf(a.numParticles, BLOCK/FEATURE_LANES);
    LBM_CLOSURE_STORAGE(storage, (closureFeatures<S><<<grid, BLOCK, 0, stream>>>((const S*) src, mask, positions,
            velocities, particles, ucm, a, raw, centreVelocity, frame)))
}

void launchClosureField(int storage, const void* src, const uint32_t* mask, const double* ucm, const ParticleArgs& a,
        double* field, hipStream_t stream) {
    unsigned grid = gridOf(a.g.n, BLOCK);
    LBM_CLOSURE_STORAGE(storage, (closureField<S><<<grid, BLOCK, 0, stream>>>((const S*) src, mask, ucm, a, field)))
}

void launchClosureTargets(int storage, const void* src, const uint32_t* mask, const double* positions,
        const int* particles, const double* ucm, const ParticleArgs& a, const double* centreVelocity,
        const uint8_t* frame, float* targets, hipStream_t stream) {
    if (a.numParticles == 0)
        return;
    unsigned grid = gridOf(a.numParticles, BLOCK/64);
    LBM_CLOSURE_STORAGE(storage, (closureTargets<S><<<grid, BLOCK, 0, stream>>>((const S*) src, mask, positions,
            particles, ucm, a, centreVelocity, frame, targets)))
}

/*
 * Whether a work-group shares one tile (eight waves on its nodes) instead of taking one per wave.  Pulls (no field) are 19
 * loads per node: always, so that a wave makes one round of them and not seven (a step of 5,000 chain beads in 128^3 104 ->
 * 79 us, 40,000 in 160^3 181 -> 167, 100,000 there 234 either way).  Node velocities from a field: up to 32,768 particles,
 * where tiles per wave leave compute units idle (10,000 in 64^3 41.4 -> 35.3 us, 20,000 42.9 -> 39.9, 40,000 48.2 -> 50.6).
 */
static bool closureShares(int numParticles, bool field) {
    return !field || numParticles <= 32768;
}

int closureStepBlocks(int numParticles, bool field) {
    return (int) gridOf(std::max(numParticles, 1), (closureShares(numParticles, field) ? 1 : CLOSURE_WAVES)*CLOSURE_TILE);
}

void launchClosureStep(int storage, const void* src, const uint32_t* mask, const double* positions,
        const double* velocities, const int* particles, const double* mass, const double* ucm, const ParticleArgs& a,
        const ClosureNorm& norm, const MlpDevice* weights, const double* field, uint8_t* ood, double* particleForce,
        double* systemForces, unsigned long long* reactionFixed, uint32_t* touched, unsigned long long* counters,
        hipStream_t stream) {
    if (a.numParticles == 0)
        return;
    const unsigned grid = (unsigned) closureStepBlocks(a.numParticles, field != nullptr);
    const float outInv = 1.0f/norm.outScale;
#define LBM_CLOSURE_STEP(S, FIELD, SHARED) \
    closureStep<S, FIELD, SHARED><<<grid, 64*CLOSURE_WAVES, 0, stream>>>((const S*) src, mask, positions, velocities, \
            particles, mass, ucm, a, norm, outInv, weights, field, ood, particleForce, systemForces, reactionFixed, touched, \
            counters)
    if (field == nullptr)
        LBM_CLOSURE_STORAGE(storage, (LBM_CLOSURE_STEP(S, false, true)))
    else if (closureShares(a.numParticles, true))      // the velocities replace the pulls: the storage does not matter
        LBM_CLOSURE_STEP(float, true, true);
    else
        LBM_CLOSURE_STEP(float, true, false);
#undef LBM_CLOSURE_STEP
}

int closureFallbackBlocks(int numParticles) {
    return std::max(1, std::min((int) gridOf(numParticles, BLOCK), FALLBACK_MAX_BLOCKS));
}

void launchClosureFallback(int storage, const void* src, const uint32_t* mask, const double* positions,
        const double* velocities, const int* particles, const double* mass, const double* ucm, const ParticleArgs& a,
        const uint8_t* ood, double* particleForce, double* systemForces, unsigned long long* reactionFixed, uint32_t* touched,
        double* partials, hipStream_t stream) {
    if (a.numParticles == 0)
        return;
    unsigned grid = (unsigned) closureFallbackBlocks(a.numParticles);
    LBM_CLOSURE_STORAGE(storage, (closureFallback<S><<<grid, BLOCK, 0, stream>>>((const S*) src, mask, positions,
            velocities, particles, mass, ucm, a, ood, particleForce, systemForces, reactionFixed, touched, partials)))
}

}  // namespace lbm
