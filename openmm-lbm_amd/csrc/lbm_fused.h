/*
 * The per-node body of the fused pull-stream + regularized collision + Guo forcing (+ Philox noise) pass,
 * shared by the single-lattice kernel (lbm_fluid.hip) and the batched-replica kernel (lbm_batch.hip).
 * Reference counterparts: computeFluidMoments + collideAndStream (lbmFluid.cc:89-139, 230-310;
 * ReferenceLBMKernels.cpp:430-469, 1066-1120).
 */
#pragma once

#include "lbm_internal.h"

namespace lbm {

/*
 * The touched-mask word of a node, read from the step's mask; the word's first node clears it in the next step's mask (the
 * two masks alternate, so that no thread can clear a word that another has yet to read).
 */
template <bool REACTION>
__device__ __forceinline__ uint32_t takeTouchedWord(const uint32_t* __restrict__ touched, uint32_t* __restrict__ nextTouched,
        uint32_t node) {
    uint32_t touchedWord = 0;
    if constexpr (REACTION) {
        touchedWord = *asGlobal(touched + (node >> 5));
        if ((node & 31) == 0)
            *asGlobal(nextTouched + (node >> 5)) = 0;
    }
    return touchedWord;
}

/*
 * One fluid node from its pulled pre-collision deviations fr[q] = C_q(x - c_q): form the moments, subtract the removal
 * velocity, add the body force and the particle reaction (consumed from the fixed-point accumulators where the
 * touched bit is set), collide, add the fluctuating part, store C_q(x) to dst at element e of x.
 */
template <typename S, bool REACTION, bool FLUCT, bool WIDE = false>
__device__ __forceinline__ void collideNode(const typename StorageTraits<S>::Real fr[NQ], S* __restrict__ dst,
        unsigned long long* __restrict__ reactionFixed, uint32_t touchedWord, const double* __restrict__ ucm,
        const StepArgs& a, uint32_t node, ElementIndex<WIDE> e) {
    using R = typename StorageTraits<S>::Real;
    using C = typename StorageTraits<S>::Compute;
    C f[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++)
        f[q] = (C) fr[q];
    Moments<C> m = nodeMoments(f);
    C pi[6];
    piNeq(m, pi);
    C rho = C(1) + m.dr;
    C jx = m.jx, jy = m.jy, jz = m.jz;
    if (a.removal) {
        jx -= rho*C(ucm[0]);
        jy -= rho*C(ucm[1]);
        jz -= rho*C(ucm[2]);
    }
    C fx = rho*C(a.gx), fy = rho*C(a.gy), fz = rho*C(a.gz);
    if constexpr (REACTION) {
        if ((touchedWord >> (node & 31)) & 1u) {
            // Reaction of the coupled particles on this node (fixed point), consumed and cleared: with FP16/BF16
            // populations by one atomic exchange per word (coupled step of 256^3 with 20,000 Keys beads 0.403 ->
            // 0.401 ms), with FP32 or FP64 by a load and a store (the exchange costs 0.627 -> 0.634 ms there).
            C r[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                unsigned long long* p = reactionFixed + reactionIndex(node, c, a.g.n, a.reactionPlanes);
                unsigned long long v;
                if constexpr (isReduced<S>())
                    v = __hip_atomic_exchange(p, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else {
                    v = *asGlobal(p);
                    *asGlobal(p) = 0ull;
                }
                r[c] = C((double) (long long) v*(1.0/FIXED_SCALE));
            }
            fx += r[0];
            fy += r[1];
            fz += r[2];
        }
    }
    C stress[6] = {C(0), C(0), C(0), C(0), C(0), C(0)};
    C omega = C(a.omega);
    // The random part is formed in the storage's load type R (FP32, or FP64 with FP64 storage): its precision is
    // that of a random number.  Its stress modes join P; its ghost modes, weighted, are added after the collision.
    R noise[NQ];
    if constexpr (FLUCT) {
        R r[16], s[6];
        drawNormals<R, 16>(a.seed, TAG_FLUID, node, a.step, r);
        R mu = R(a.mu), rhoR = R(rho), om = R(a.omega);
        R stressAmp, ghostAmp;
        if constexpr (std::is_same<R, float>::value) {
            stressAmp = __builtin_amdgcn_sqrtf(mu*rhoR*om*(2.0f - om));
            ghostAmp = __builtin_amdgcn_sqrtf(mu*rhoR);
        }
        else {
            stressAmp = sqrt(mu*rhoR*om*(R(2) - om));
            ghostAmp = sqrt(mu*rhoR);
        }
        stressNoise(r, stressAmp, s);
        ghostNoiseWeighted(r, ghostAmp, noise);
#pragma unroll
        for (int c = 0; c < 6; c++)
            stress[c] = C(s[c]);
    }
    C out[NQ];
    // The exact weights matter where the storage keeps FP32 or FP64 precision; FP16/BF16 rounding is far coarser.
    collide<C, false, !isReduced<S>()>(m.dr, jx, jy, jz, pi, fx, fy, fz, omega, stress, nullptr, out);
    uint32_t rnd = 0;
    if constexpr (isReduced<S>())
        rnd = mixBits(node ^ a.roundSeed);
    auto* base = asGlobal(dst);
    [[maybe_unused]] uint32_t offset = (uint32_t) e*(uint32_t) sizeof(S);
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        uint32_t r = 0;
        if constexpr (isReduced<S>())
            r = roundingBits<S>(rnd, q);
        R v = (R) out[q];
        if constexpr (FLUCT)
            v += noise[q];
        if constexpr (WIDE)
            storePopStream<S>(base + (uint64_t) q*a.g.qstride + e, v, r);
        else {
            // With FP16/BF16 storage and fluctuations the pass is bound by the issue of its instructions (a wavefront's 767
            // vector ones, 684 with this, Philox's three-input xors and no idle halves in the roundings: 256^3 FP16
            // 287 -> 256 us, 128^3 39.6 -> 37.4 us; FP32 734 -> 673, 433 -> 432 us, bound by memory).
            // The node's byte offset, opaque from one population to the next: each store then takes it beside a scalar
            // base.  Seen as one value, it made the compiler step a 64-bit vector address instead.
            asm("" : "+v"(offset));
            using Byte = __attribute__((address_space(1))) char;
            using Pop = __attribute__((address_space(1))) S;
            storePopStream<S>((Pop*) ((Byte*) (base + (size_t) q*a.g.qstride) + offset), v, r);
        }
    }
}

/*
 * Thread t of the pass: one node (chunkedNode), pull C_q(x - c_q) from src and collide (collideNode).  Writes nothing for
 * solid nodes.  A lane past the end of a padded row repeats the row's last node into the padding, so that the row's last
 * lines are written whole.
 */
template <typename S, bool SOLIDS, bool REACTION, bool FLUCT, bool WIDE = false>
__device__ __forceinline__ void fusedNode(const S* __restrict__ src, S* __restrict__ dst, const uint32_t* __restrict__ mask,
        unsigned long long* __restrict__ reactionFixed, const uint32_t* __restrict__ touched,
        uint32_t* __restrict__ nextTouched, const double* __restrict__ ucm, const StepArgs& a, uint32_t t) {
    uint32_t i, j, k;
    if (!chunkedNode(a.g, t, i, j, k))
        return;
    const uint32_t past = i < a.g.nx ? 0u : i - (a.g.nx - 1u);
    if (past != 0u && !a.g.padded)
        return;
    i -= past;
    const uint32_t node = (k*a.g.ny + j)*a.g.nx + i;
    uint32_t touchedWord = 0;
    if (past == 0u)
        touchedWord = takeTouchedWord<REACTION>(touched, nextTouched, node);
    if constexpr (SOLIDS)
        if (isSolid(mask, node))
            return;
    using Offset = typename std::conditional<WIDE, long long, int>::type;
    const ElementIndex<WIDE> e = elementOf<ElementIndex<WIDE>>(a.g, i, j, k);
    typename StorageTraits<S>::Real fr[NQ];
    pullNodeStream<S, WIDE>(src, a.g.qstride, e, elementNeighbours<Offset>(a.g, i, j, k), fr);
    collideNode<S, REACTION, FLUCT, WIDE>(fr, dst, reactionFixed, touchedWord, ucm, a, node, e + past);
}

}  // namespace lbm
