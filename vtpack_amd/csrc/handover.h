// Query counts handed from workgroup to workgroup of one launch, in launch order.  Plain enough to be compiled for the host
// too, where threads play the lanes: what it needs beside the language is wave_sum, wait_vmcnt and the builtins below.
#pragma once

namespace vtdge {

// status[0]: error flag, status[1 + w]: what workgroup w has to say: a flag bit and its count, the last of every 64
// workgroups the count of them all.  All zero at launch.
constexpr int CHAIN_GROUP = 64;
constexpr unsigned long long CHAIN_KNOWN = 1ull << 62;
constexpr int CHAIN_SPIN_LIMIT = 1 << 20;

template <typename T> __device__ __forceinline__ T chain_load(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ void chain_store(T *p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// what this wave has stored is there for every workgroup before anything behind this
__device__ __forceinline__ void chain_stored()
{
    asm volatile("" ::: "memory");
    wait_vmcnt<0>();
    asm volatile("" ::: "memory");
}

// the queries of workgroup `wg`; one wave
__device__ __forceinline__ void chain_publish(unsigned long long *words, int wg, int agg)
{
    if ((threadIdx.x & 63) == 0 && wg % CHAIN_GROUP != CHAIN_GROUP - 1) chain_store(words + wg, CHAIN_KNOWN | (unsigned long long)agg);
}

// `*total`, the rows of the whole launch, as its last workgroup knows them (one lane); past the capacity if a workgroup gave up
// waiting.  Whoever does raises the flag, then stores capacity + 1 in the total's place: behind this it stays, and before this
// the exchange brings it back.  (What else may have lain there is told by the flag.)  One trip to memory where all went well: a store
// that has to be there before a look at the flag would be two.
__device__ __forceinline__ void chain_total(unsigned long long *status, int64_t *total, int64_t rows, int64_t capacity)
{
    const int64_t was = __hip_atomic_exchange(total, rows, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (was == capacity + 1 && rows <= capacity && chain_load(status) != 0) chain_store(total, capacity + 1);
}

// The queries of all workgroups before `wg`, whose own are `agg`.  One wave, the value in every lane; `capacity`, with *total past
// it, where the wait was given up.  A lane takes a workgroup of wg's own group and every 64th of the groups before it, and asks again
// only for what it still lacks: two trips to memory once all have spoken, however many they are.  Looking back 64 words at a time
// took 52.1 us for the scatter-back of 1024 workgroups (256 x 16 x 16 tokens of 384 channels) and 96.6 of 2048, this 49.1 and 88.8;
// without any wait the first takes 48.3.  A group's sum made by atomic additions of all 64 instead: 58.9 us.
__device__ __forceinline__ long long chain_rows_before(unsigned long long *status, int wg, int agg, int64_t capacity, int64_t *total,
                                                       int spin_limit = CHAIN_SPIN_LIMIT)
{
    const int lane = threadIdx.x & 63;
    unsigned long long *st = status + 1;
    const int groups = wg / CHAIN_GROUP, place = wg % CHAIN_GROUP;
    int spins = 0, own = 0, before = 0, g = lane;
    bool want_own = lane < place, to_say = place == CHAIN_GROUP - 1;
    while (true) {
        unsigned long long vo = 0, vg = 0;
        if (want_own) vo = chain_load(st + groups * CHAIN_GROUP + lane);
        if (g < groups) vg = chain_load(st + (int64_t)g * CHAIN_GROUP + CHAIN_GROUP - 1);
        if (vo & CHAIN_KNOWN) {
            own = (int)(vo & 0xffffffffull);
            want_own = false;
        }
        if (vg & CHAIN_KNOWN) {
            before += (int)(vg & 0xffffffffull);
            g += WAVE;
        }
        const bool own_done = __builtin_amdgcn_ballot_w64(want_own) == 0;
        if (own_done && to_say) {
            to_say = false;
            const int all = agg + (int)wave_sum((float)own);                  // small integers: exact
            if (lane == 0) chain_store(st + wg, CHAIN_KNOWN | (unsigned long long)all);
        }
        if (own_done && __builtin_amdgcn_ballot_w64(g < groups) == 0) return (long long)wave_sum((float)(own + before));
        if (++spins > spin_limit) {
            // every row of this workgroup falls past the capacity, and of those that build on its group's count
            if (lane == 0) {
                chain_store(status, 1ull);
                chain_stored();
                chain_store(total, capacity + 1);
                if (to_say) chain_store(st + wg, CHAIN_KNOWN | (unsigned long long)capacity);
            }
            return capacity;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

}  // namespace vtdge
