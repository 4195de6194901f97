// Allocations of one size that are made ahead and cleared together (mlel_hip_arena_alloc); nothing here knows the device.
#pragma once

namespace mlel {
// As many as share one wait (8 us).  A 4 KiB allocation: 13 us alone, 5.8 with four, 5.4 with six, 8.8 with eight.  Where the blocks lie moves
// what the runtime allocates for itself: instantiating a recorded graph of 38 launches afterwards took 44 us with six, 58 with four, 62
// with three, 50 with two.
constexpr int kFreshBlocks = 6;

struct FreshBlocks {
    void *fresh[kFreshBlocks], *clearing[kFreshBlocks];  // cleared and not handed out yet; those whose clearing nobody has waited for
    int n_fresh = 0, n_clearing = 0;

    // Hands out a cleared block.  make(&block) allocates one and starts its clearing, wait() waits for every clearing that was
    // started, drop(block) frees one; both return 0 or an error, of which `no_memory` says that there is none left.  Every call makes
    // at least one, so that what else refuses an allocation refuses every call; without memory, what was made before is handed out.
    template <typename Error, typename Make, typename Wait, typename Drop>
    Error take(void **out, Error no_memory, Make make, Wait wait, Drop drop) {
        Error e = make(&clearing[n_clearing]);
        if (e == Error(0)) n_clearing++;
        else if (e != no_memory || n_fresh + n_clearing == 0) return e;
        if (n_fresh == 0) {  // (n_clearing is at most the number that were handed out since, and one)
            while (n_clearing < kFreshBlocks && make(&clearing[n_clearing]) == Error(0)) n_clearing++;
            e = wait();
            if (e != Error(0)) {
                while (n_clearing > 0) drop(clearing[--n_clearing]);
                return e;
            }
            while (n_clearing > 0) fresh[n_fresh++] = clearing[--n_clearing];
        }
        *out = fresh[--n_fresh];
        return Error(0);
    }
    template <typename Drop>
    void clear(Drop drop) {
        while (n_fresh > 0) drop(fresh[--n_fresh]);
        while (n_clearing > 0) drop(clearing[--n_clearing]);
    }
};
}  // namespace mlel
