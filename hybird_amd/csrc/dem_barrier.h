// How the workgroups of one launch meet (dem_run.hip): the protocol on the words in memory, apart from the memory
// itself, so that it also runs on the host with one thread per workgroup.
//
// A word per workgroup and meeting: each workgroup stores its value into its own word, then reads all of them, and so
// knows that all have arrived and the maximum of their values. Three sets of words rotate: a set is empty again
// before it comes next, since nobody reaches meeting n + 1 before everybody has left meeting n - 1.
//
// A launch begins with a roll call, since nothing promises that its workgroups are on the device together: another
// process's work, or a mask, may leave too few CUs, and two such launches of two processes can each hold a part and
// wait for the other. Each workgroup has one more word, 2 g after g launches, and checks in before the first meeting:
// 2 g + 2. At that meeting, a workgroup that has waited long enough for another refuses it, by making that word
// 2 g + 1, unless the other has checked in and is only on its way. A word changes once, so the launch meets if all have
// checked in, and otherwise nobody sees everybody arrive: one that was refused says so when it comes. Then all leave,
// and the last to leave does the work alone.
//
// M: the memory of the words, with load, store, swap (compare and swap; the old value), add (the old value), now (in
// ticks) and pause.
#pragma once

namespace hyb {

typedef unsigned long long u64;

constexpr u64 SLOT_EMPTY = ~0ull;
constexpr u64 SLOT_TIMEOUT = ~0ull - 1;  // above every value
constexpr u64 SLOT_PRESENT = 0, SLOT_REFUSED = 1;  // verdicts of the roll call

template <class M>
struct Meeting {
    u64* slots;  // [4][workgroups]: three sets and the words of the roll call
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

    __host__ __device__ __forceinline__ u64* roll(int wg) const { return &slots[3 * (size_t)nwg + (size_t)wg]; }

    // Before the first meeting, after g launches; the value to arrive with there. ticks 0: nobody is present, whoever is
    // on the device.
    __host__ __device__ __forceinline__ u64 check_in(int wg, u64 g, u64 ticks) const {
        const u64 was = M::swap(roll(wg), 2 * g, ticks ? 2 * g + 2 : 2 * g + 1);
        return was == 2 * g && ticks ? SLOT_PRESENT : SLOT_REFUSED;
    }
    // The first meeting, after arrive() with the value of check_in: the verdict from every lanes-th word, SLOT_PRESENT,
    // SLOT_REFUSED or, for a workgroup that checked in and stopped coming, SLOT_TIMEOUT.
    __host__ __device__ __forceinline__ u64 call(int lane, int lanes, u64 g, u64 ticks, u64 most) const {
        u64 m = SLOT_PRESENT;
        for (int i = lane; i < nwg; i += lanes) {
            u64 s = M::load(&set(n)[i]);
            if (s == SLOT_EMPTY) {
                const u64 t0 = M::now();
                u64 limit = ticks;
                do {
                    M::pause();
                    s = M::load(&set(n)[i]);
                    if (s == SLOT_EMPTY && M::now() - t0 >= limit) {
                        if (limit == most) s = SLOT_TIMEOUT;
                        else if (M::swap(roll(i), 2 * g, 2 * g + 1) != 2 * g + 2) s = SLOT_REFUSED;
                        limit = most;
                    }
                } while (s == SLOT_EMPTY);
            }
            m = s > m ? s : m;
        }
        return m;
    }
    // After a refused roll call: whether this workgroup is the last to leave.
    __host__ __device__ __forceinline__ bool last_out(unsigned* left) const {
        return M::add(left, 1u) == (unsigned)nwg - 1u;
    }
    // By the last to leave: the words as a launch that met leaves them.
    __host__ __device__ __forceinline__ void clear_all(int lane, int lanes, u64 g) const {
        for (int i = lane; i < 3 * nwg; i += lanes) M::store(&slots[i], SLOT_EMPTY);
        for (int i = lane; i < nwg; i += lanes) M::store(roll(i), 2 * g + 2);
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
