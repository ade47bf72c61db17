/*
 * Host-side rules of device memory: the memory that the calls which read fields out share.
 */
#pragma once

#include <hip/hip_runtime_api.h>
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
