// pinned.h -- words of pinned host memory that kernels write and the host
// reads at any time, without a copy, an event or a wait.
//
// hipHostFree waits until every stream of the device has drained, so the
// words of a finished scene are kept for the next one, as its device blocks
// are (devcache.h): in blocks of 64 words, at most kBlocks of them, which go
// back to the driver on mpm_release_cache() if no word is taken.  All
// functions are thread-safe.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <vector>

namespace mpm {
namespace pinned {

constexpr size_t kBlocks = 64, kWords = 64, kStride = 8;  // a word per 64-byte line

struct State {
    std::mutex mu;
    std::vector<uint64_t*> blocks, idle;
};
inline State& state() {
    static State* s = new State;  // never destroyed: releases may come during process exit
    return *s;
}

// A zeroed word, or null if there is none.
inline uint64_t* take() {
    State& st = state();
    std::lock_guard<std::mutex> g(st.mu);
    if (st.idle.empty()) {
        void* p = nullptr;
        if (st.blocks.size() >= kBlocks) return nullptr;
        if (hipHostMalloc(&p, kWords * kStride * sizeof(uint64_t), 
                          hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        st.blocks.push_back(static_cast<uint64_t*>(p));
        for (size_t i = kWords; i-- > 0;) st.idle.push_back(st.blocks.back() + i * kStride);
    }
    uint64_t* w = st.idle.back();
    st.idle.pop_back();
    *w = 0;
    return w;
}

// The streams whose kernels write the word must be done.
inline void give(uint64_t* w) {
    if (!w) return;
    State& st = state();
    std::lock_guard<std::mutex> g(st.mu);
    st.idle.push_back(w);
}

inline void release_all() {
    State& st = state();
    std::lock_guard<std::mutex> g(st.mu);
    if (st.idle.size() != st.blocks.size() * kWords) return;
    for (uint64_t* p : st.blocks) (void)hipHostFree(p);
    st.blocks.clear();
    st.idle.clear();
}

}  // namespace pinned
}  // namespace mpm
