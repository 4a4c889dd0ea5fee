#pragma once
// A workspace that the library holds for callers who bring none: memory that grows on demand.
#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace saetta {

struct OwnedWorkspace {
    void *ptr = nullptr;
    size_t bytes = 0;
    size_t refused = SIZE_MAX;  // the least that could not be had
    // Holds at least the first of `wants` (in falling order) that can be had; false: not even the last, and nothing is held.  What was
    // once refused is asked for again only where nothing smaller does: a try gives up what is held, which waits for the stream.
    // alloc(bytes): null where there is none.
    template <class Alloc, class Release>
    bool take(std::initializer_list<size_t> wants, Alloc &&alloc, Release &&release) {
        for (const size_t &want : wants) {
            if (bytes >= want) return true;
            if (want >= refused && &want + 1 != wants.end()) continue;
            if (ptr) release(ptr);
            ptr = nullptr, bytes = 0;
            if ((ptr = alloc(want)) != nullptr) {
                bytes = want;
                if (want >= refused) refused = SIZE_MAX;
                return true;
            }
            if (want < refused) refused = want;
        }
        return false;
    }
};

}  // namespace saetta
