// The host's side of a result on its way to a caller's buffer: waiting for a
// piece's flag in pinned memory.  Plain C++, no runtime calls of its own.
#pragma once

#include <cstdint>

namespace qwn {

enum class Landing {
    kLanded,   // the flag holds the epoch: the piece is in the window
    kMissing,  // the stream has finished and the flag was never raised
    kFailed,   // the stream reported an error
};

enum class StreamState { kBusy, kDone, kFailed };

// Polls until *flag == epoch.  idle() fills the wait, state() asks the
// stream every `every` turns: a kernel that failed raises no flag, and the
// window then still holds what an earlier transfer left there.  A piece that
// lands between the last poll and the question is found by looking once more.
template <typename Idle, typename State>
Landing await_piece(const uint32_t *flag, uint32_t epoch, Idle &&idle, State &&state, uint32_t every = 16384) {
    for (uint32_t turn = 1; __atomic_load_n(flag, __ATOMIC_ACQUIRE) != epoch; ++turn) {
        idle();
        if (turn % every) continue;
        const StreamState s = state();
        if (s == StreamState::kBusy) continue;
        if (s == StreamState::kFailed) return Landing::kFailed;
        return __atomic_load_n(flag, __ATOMIC_ACQUIRE) == epoch ? Landing::kLanded : Landing::kMissing;
    }
    return Landing::kLanded;
}

// Has the page of *p mapped for writing without changing what it holds: one
// locked add of zero to the aligned word there, which another thread's store
// cannot be lost to.
inline void map_for_writing(float *p) {
    auto *word = reinterpret_cast<uint32_t *>(reinterpret_cast<uintptr_t>(p) & ~uintptr_t{3});
    __asm__ volatile("lock; addl $0, %0" : "+m"(*word) : : "cc");
}

}  // namespace qwn
