// A device buffer that calls can do without: it grows when it can, and what it
// holds stays until something larger is there.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace sl {

struct Slots {
    void* p = nullptr;
    size_t bytes = 0;
    size_t limit = SIZE_MAX;  // bytes past which a request has been refused
};

// Grows s to `bytes`, or as much as alloc(size) gives (null: refused), down to
// `least`.  A size that was refused is not asked for again.  The old buffer is
// released once the new one is there.
template <typename Alloc, typename Release>
void grow(Slots* s, size_t bytes, size_t least, Alloc alloc, Release release) {
    for (;;) {
        const size_t want = std::min(bytes, s->limit);
        if (want <= s->bytes || want < least) return;
        if (void* p = alloc(want)) {
            if (s->p) release(s->p);
            s->p = p;
            s->bytes = want;
            return;
        }
        s->limit = want / 2;
    }
}

}  // namespace sl
