// Tagged words: how the work-groups of a cooperative launch exchange values
// while they run. A 64-bit store carries a tag beside a 32-bit value, and the
// receiver polls the word itself until the tag is the one it waits for, so that
// no flag, fence or cache flush orders the exchange.
#pragma once

#include <mutex>

#include "mh_common.h"

namespace mh {

typedef unsigned long long Word;

constexpr int kWaitSpins = 1 << 16;  // loads of a word that does not come: tens of milliseconds

// Largest device index that has a lock for launches whose work-groups wait for
// one another: two of them at once could each hold a part of the device and
// wait for the other part for good.
constexpr int kMaxDevices = 64;
std::mutex &device_lock(int device);  // cmf_onchip.hip

// Compute units that plans for such launches count on: the device's, or what
// mh_cmf_set_chip_units says; 0 if they are not known.
int compute_units(mh_ctx *ctx);

template <int G>
struct alignas(4 * G) Vec {
    float v[G];
};

// Words are addressed by 32-bit byte offsets from the inbox (a few megabytes).
__device__ __forceinline__ Word *word_at(Word *base, unsigned byte)
{
    return reinterpret_cast<Word *>(reinterpret_cast<char *>(base) + size_t(byte));
}
__device__ __forceinline__ Word ld_word(const Word *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_word(Word *p, unsigned tag, float v)
{
    __hip_atomic_store(p, (Word(tag) << 32) | __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Orders LDS accesses of the work-group around the barrier; global stores (the
// words under way to other bricks) are not waited for.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Whether a wait ends without its word: every 16th load, when another
// work-group gave up or after kWaitSpins loads. Raises both flags.
__device__ __forceinline__ bool give_up(int spin, int *abort, int *fail)
{
    if ((spin & 15) != 15) return false;
    if (spin <= kWaitSpins && !__hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        return false;
    __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *fail = 1;
    return true;
}

// After the loop that polls: no load is under way on any path here, which the
// compiler does not see where the loop is left between its loads; it would wait
// at the registers' next use, for whatever was loaded in between as well.
__device__ __forceinline__ void words_arrived() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)

// A value the compiler cannot move computations on out of the loop (address
// arithmetic hoisted out of it would hold a register per address).
__device__ __forceinline__ unsigned here(unsigned v)
{
    asm volatile("" : "+v"(v));
    return v;
}

__device__ __forceinline__ int here_s(int v)  // the same for a uniform value
{
    asm volatile("" : "+s"(v));
    return v;
}

}  // namespace mh
