// blink::StageBuffer, the scratch of the stage calls: an address handed out under a
// caller's capture is freed by destroy() alone, whatever grows or is released
// before; without captures at most one buffer is held.
#include <cstdio>
#include <cstdlib>
#include <set>

#include "../../imager_amd/csrc/blink_scratch.hpp"

static int g_failed = 0;
static void check(bool ok, const char* what) {
    if (!ok) std::printf("FAILED: %s\n", what), g_failed++;
}

int main() {
    std::set<void*> live;
    bool full = false;
    auto alloc = [&](size_t n) -> void* {
        void* p = full ? nullptr : std::malloc(n);
        if (p) live.insert(p);
        return p;
    };
    auto dealloc = [&](void* p) {
        check(live.erase(p) == 1, "freed once, and only what was allocated");
        std::free(p);
    };

    {  // no capture: grows by replacing, gives everything back
        blink::StageBuffer b;
        void* p = b.take(100, false, true, alloc, dealloc);
        check(p && b.take(50, false, true, alloc, dealloc) == p, "a smaller call keeps the buffer");
        check(b.take(200, false, true, alloc, dealloc) && live.size() == 1, "growth replaces it");
        check(!b.take(300, false, false, alloc, dealloc) && live.size() == 1, "may not grow: null");
        b.release(dealloc);
        check(live.empty(), "release gives it back");
        check(!b.take(1, false, false, alloc, dealloc), "nothing left after release");
        full = true;
        check(!b.take(1, false, true, alloc, dealloc) && b.bytes == 0, "allocation failure: null");
        full = false;
        check(b.take(1, false, true, alloc, dealloc), "and the next call allocates");
        b.destroy(dealloc);
        check(live.empty(), "destroy gives it back");
    }
    {  // handed out under capture, then larger calls and release
        blink::StageBuffer b;
        b.take(100, false, true, alloc, dealloc);
        void* p = b.take(100, true, false, alloc, dealloc);
        check(p && b.captured, "a capture takes the buffer that is there");
        check(!b.take(101, true, false, alloc, dealloc), "a capture does not allocate");
        void* q = b.take(1000, false, true, alloc, dealloc);
        check(q && q != p && live.count(p), "a larger call leaves the captured buffer");
        void* r = b.take(2000, false, true, alloc, dealloc);
        check(r && live.count(p) && live.size() == 2, "the one in between is freed");
        b.take(2000, true, false, alloc, dealloc);
        b.take(10, false, true, alloc, dealloc);  // an eager call on a captured buffer
        b.release(dealloc);
        check(live.count(p) && live.count(r) && live.size() == 2, "release keeps what was captured");
        void* s = b.take(10, false, true, alloc, dealloc);
        check(s != p && s != r, "and does not hand it out again");
        b.destroy(dealloc);
        check(live.empty(), "destroy frees them all");
    }
    if (g_failed) return 1;
    std::printf("All tests passed.\n");
    return 0;
}
