/*
 * Host-side rules of device memory: the memory that a lattice can do without, and that which the calls that read fields out
 * share.
 */
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <initializer_list>
#include <mutex>

namespace lbm {

/* Device memory of `bytes`, or nullptr where there is not as much; the error that this leaves is not the next call's. */
inline void* tryAllocate(size_t bytes) {
    void* p = nullptr;
    if (hipMalloc(&p, bytes) == hipSuccess)
        return p;
    (void) hipGetLastError();
    return nullptr;
}

/*
 * What stays free beside memory that a lattice of n nodes can do without (padded rows, a moment field, the tile spread's
 * bins, matrix rows): its reaction accumulators and masks, a state of 19 FP64 values per node and the fields on their way to
 * the host.  A lattice that fits without that memory then keeps fitting, and is read out, with it.
 */
inline uint64_t reservedBytes(uint64_t n) {
    return (24 + 1 + 19*8 + 4*8)*n;
}

/* The device's free memory beyond `reserve` bytes. */
inline uint64_t spareBytes(uint64_t reserve) {
    size_t free = 0, total = 0;
    return hipMemGetInfo(&free, &total) == hipSuccess && free > reserve ? free - reserve : 0;
}

/* Memory of up to this size is tried without a question to the device, which takes 0.15 ms. */
constexpr uint64_t SMALL_BYTES = 64ull << 20;

/* The bytes that an array of padded rows may take, of two arrays for each of the lattices (`nodes` in all) that share the
   room; the device is asked once, when an array is large. */
struct PaddingRoom {
    uint64_t nodes;
    bool asked = false;
    uint64_t spare = 0;
    bool holds(uint64_t bytes, uint64_t n) {
        if (bytes <= SMALL_BYTES)
            return true;
        if (!asked)
            spare = spareBytes(reservedBytes(nodes));
        asked = true;
        return (double) bytes <= (double) spare/2*((double) n/(double) nodes);
    }
};

/* One part of a set of arrays that are all there or not needed at all. */
struct OptionalPart {
    void** to;
    size_t bytes;
};

/* All the parts, or none (nullptr): where they would take more than the spare memory, or an allocation fails. */
inline bool allocateOptional(std::initializer_list<OptionalPart> parts, uint64_t reserve) {
    uint64_t total = 0;
    for (const OptionalPart& part : parts)
        total += part.bytes;
    bool all = total <= SMALL_BYTES || total <= spareBytes(reserve);
    for (const OptionalPart& part : parts) {
        *part.to = all ? tryAllocate(part.bytes) : nullptr;
        all = all && *part.to != nullptr;
    }
    if (!all)
        for (const OptionalPart& part : parts) {
            if (*part.to != nullptr)
                (void) hipFree(*part.to);
            *part.to = nullptr;
        }
    return all;
}

/*
 * Device memory that the calls which read fields out share, one after the other: kept from call to call up to KEEP bytes and
 * freed with its owner, allocated for the call beyond.  The lock is held until the call has what it wants on the host.
 */
struct FieldStage {
    static constexpr size_t KEEP = 1ull << 30;
    std::mutex lock;
    void* kept = nullptr;
    size_t bytes = 0;
    /* Memory for a call that needs `need` bytes, or nullptr; give it back with done(). */
    void* get(size_t need) {
        if (need <= bytes)
            return kept;
        if (need <= KEEP) {
            free();                         // no one else has it: the calls take turns
            kept = tryAllocate(need);
            bytes = kept != nullptr ? need : 0;
            return kept;
        }
        void* p = tryAllocate(need);
        if (p == nullptr && kept != nullptr) {
            free();                         // what a smaller call left may be what is missing
            p = tryAllocate(need);
        }
        return p;
    }
    hipError_t done(void* p) {
        return p == kept ? hipSuccess : hipFree(p);
    }
    void free() {
        if (kept != nullptr)
            (void) hipFree(kept);
        kept = nullptr;
        bytes = 0;
    }
};

}  // namespace lbm
