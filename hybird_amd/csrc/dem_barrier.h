// How the workgroups of one launch meet (dem_run.hip): the protocol on the words in memory, apart from the memory
// itself, so that it also runs on the host with one thread per workgroup.
//
// A word per workgroup and meeting: each workgroup stores its value into its own word, then reads all of them, and so
// knows that all have arrived and the maximum of their values. Three sets of words rotate: a set is empty again
// before it comes next, since nobody reaches meeting n + 1 before everybody has left meeting n - 1.
//
// M: the memory of the words, with load, store, now (in ticks) and pause.
#pragma once

namespace hyb {

typedef unsigned long long u64;

constexpr u64 SLOT_EMPTY = ~0ull;
constexpr u64 SLOT_TIMEOUT = ~0ull - 1;  // above every value

template <class M>
struct Meeting {
    u64* slots;  // [3][workgroups]
    unsigned n;  // meetings so far
    int nwg;

    __host__ __device__ __forceinline__ u64* set(unsigned k) const { return slots + (size_t)(k % 3u) * (size_t)nwg; }

    __host__ __device__ __forceinline__ void arrive(int wg, u64 value) const { M::store(&set(n)[wg], value); }

    // The value of one word, SLOT_TIMEOUT if it stays empty for `ticks`.
    __host__ __device__ __forceinline__ u64 wait(u64* word, u64 ticks) const {
        u64 s = M::load(word);
        if (s == SLOT_EMPTY) {
            const u64 t0 = M::now();
            do {
                M::pause();
                s = M::load(word);
            } while (s == SLOT_EMPTY && M::now() - t0 < ticks);
            if (s == SLOT_EMPTY) s = SLOT_TIMEOUT;
        }
        return s;
    }

    // The maximum of every lanes-th word from `lane` on.
    __host__ __device__ __forceinline__ u64 wait_all(int lane, int lanes, u64 ticks) const {
        u64 m = 0;
        for (int i = lane; i < nwg; i += lanes) {
            const u64 s = wait(&set(n)[i], ticks);
            m = s > m ? s : m;
        }
        return m;
    }

    // Everybody has arrived, hence left the meeting before: its word is free again.
    __host__ __device__ __forceinline__ void free_last(int wg) const { M::store(&set(n + 2u)[wg], SLOT_EMPTY); }
};

// What a workgroup says at the end of a launch: its failure, whichever one it is (nobody else sees that its wait ended
// without the others), and the first one what the next launch starts from.
enum Leaving { LEAVE_QUIETLY, LEAVE_STATE, LEAVE_ERROR };
__host__ __device__ __forceinline__ Leaving leaving(int wg, int err) {
    return err ? LEAVE_ERROR : (wg == 0 ? LEAVE_STATE : LEAVE_QUIETLY);
}

}  // namespace hyb
