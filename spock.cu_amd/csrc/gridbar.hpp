// The barrier of the workgroups that share one instance (grid mode of the fused engine): the protocol
// alone, over a memory policy, so that the kernels and a model on the host run the same code.
//
// Mem has, on the barrier's words: add(word, n), an atomic that returns the word's new value; load(word);
// store(word, v), which may become visible late; pause(), called while waiting.  release() makes everything
// this workgroup wrote before it visible to whoever sees a later write of it, acquire() drops what this
// workgroup may have cached, acqRel() is both.
#pragma once

#if defined(__HIP__)
#define SPK_BAR __device__ __forceinline__
#else
#define SPK_BAR inline
#endif

namespace spk {

// A counter for each of up to GRID_GROUPS groups of workgroups, one for the groups (the root) and a release
// flag for each group, every one in a 256-byte piece of its own.
constexpr unsigned GRID_GROUPS = 8;
constexpr unsigned GRID_BAR_STEP = 64;
constexpr unsigned GRID_BAR_WORDS = GRID_BAR_STEP * (2 * GRID_GROUPS + 1);

// What a counter grows by at every barrier, however many arrive: the first of them adds what the others leave, so
// the last is the one that finds a multiple of it.  Counters are never set back: a store that does so can
// become visible after the arrivals of the next barrier and wipe them out.  Between launches every
// counter is at a multiple, whatever the numbers of workgroups were.  More than arrive at one counter, and
// a power of two, so that the counters may overflow.
constexpr unsigned GRID_BAR_ROUND = 256;

constexpr unsigned GRID_BAR_ROOT = 0;
SPK_BAR unsigned gridCount(unsigned group) { return GRID_BAR_STEP * (1 + group); }
SPK_BAR unsigned gridFlag(unsigned group) { return GRID_BAR_STEP * (GRID_GROUPS + 1 + group); }

// The release value of the last barrier, before the first one of a launch by workgroup `wg`: no flag moves
// before this workgroup has arrived for the first time.
template <typename Mem>
SPK_BAR unsigned gridPassed(Mem &m, unsigned wg) {
    return m.load(gridFlag(wg % GRID_GROUPS));
}

// The barrier behind release value `passed`, by workgroup wg of n; returns its own release value.  Workgroups
// arrive in groups, the last of each group at the root, and the last there releases the flags.  Each of
// them passes on what it has seen by a fence between the atomic it read and the one it writes.  All
// flags move, also those of groups without a workgroup: a later launch of more workgroups starts from them, and
// its groups have to agree on the next release value.
template <typename Mem>
SPK_BAR unsigned gridPass(Mem &m, unsigned wg, unsigned n, unsigned passed) {
    const unsigned next = passed + 1, group = wg % GRID_GROUPS;
    const unsigned size = (n - group + GRID_GROUPS - 1) / GRID_GROUPS, groups = n < GRID_GROUPS ? n : GRID_GROUPS;
    m.release();
    if (m.add(gridCount(group), wg < GRID_GROUPS ? GRID_BAR_ROUND - (size - 1) : 1) % GRID_BAR_ROUND == 0) {
        m.acqRel();
        if (m.add(GRID_BAR_ROOT, group == 0 ? GRID_BAR_ROUND - (groups - 1) : 1) % GRID_BAR_ROUND == 0) {
            m.acqRel();
            for (unsigned q = 0; q < GRID_GROUPS; q++) m.store(gridFlag(q), next);
        }
    }
    while (m.load(gridFlag(group)) != next) m.pause();
    m.acquire();
    return next;
}

#if defined(__HIP__)
// The policy on the device.  Relaxed accesses at agent scope act in the coherent memory behind the XCDs' L2
// caches; the fences write back and drop what a workgroup's caches hold.  A write-back has to be waited for
// explicitly: hipcc (ROCm 7.2) drops the wait that belongs to a release fence where no other access is under way, and
// the next atomic could then overtake it.
struct GridMem {
    unsigned *words;
    __device__ __forceinline__ unsigned add(unsigned w, unsigned k) {
        return __hip_atomic_fetch_add(words + w, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + k;
    }
    __device__ __forceinline__ unsigned load(unsigned w) {
        return __hip_atomic_load(words + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void store(unsigned w, unsigned v) {
        __hip_atomic_store(words + w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void pause() { __builtin_amdgcn_s_sleep(1); }
    __device__ __forceinline__ void release() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __builtin_amdgcn_s_waitcnt(0);
    }
    __device__ __forceinline__ void acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }
    __device__ __forceinline__ void acqRel() {
        release();
        acquire();
    }
};
#endif

}  // namespace spk
