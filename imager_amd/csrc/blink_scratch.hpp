// Scratch of the stage calls that a caller may capture into a graph of its own
// (host code, and no HIP, so that the host tests run the same code).
#pragma once

#include <cstddef>
#include <vector>

namespace blink {

// A grow-only buffer.  A call made under a caller's capture leaves the address in a
// graph that may be replayed at any later time, and nothing tells when that graph
// is gone: an address handed out under capture therefore stays allocated until
// destroy(), also when a later call needs a larger buffer or release() gives the
// others back.
struct StageBuffer {
    void* ptr = nullptr;
    size_t bytes = 0;
    bool captured = false;    // a caller's graph may hold ptr
    std::vector<void*> kept;  // earlier buffers that callers' graphs may hold

    // At least `need` bytes.  Null when the buffer is smaller and may not grow, or
    // alloc returns null.  alloc(bytes) -> pointer, dealloc(pointer) once no queued
    // work uses it.
    template <class Alloc, class Dealloc>
    void* take(size_t need, bool capturing, bool may_grow, Alloc alloc, Dealloc dealloc) {
        if (bytes < need) {
            if (!may_grow) return nullptr;
            release(dealloc);
            ptr = alloc(need);
            if (!ptr) return nullptr;
            bytes = need;
        }
        captured = captured || capturing;
        return ptr;
    }

    template <class Dealloc>
    void release(Dealloc dealloc) {
        if (ptr && captured) kept.push_back(ptr);
        else if (ptr) dealloc(ptr);
        ptr = nullptr;
        bytes = 0;
        captured = false;
    }

    template <class Dealloc>
    void destroy(Dealloc dealloc) {
        release(dealloc);
        for (void* p : kept) dealloc(p);
        kept.clear();
    }
};

}  // namespace blink
