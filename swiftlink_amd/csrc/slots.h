// A device buffer that calls can do without: it grows when it can, and what it
// holds stays until something larger is there.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace sl {

// Share of the free memory one such buffer may take, so that contexts made one
// after another leave room for the buffers they cannot do without.
constexpr size_t kOptionalShare = 8;

struct Slots {
    void* p = nullptr;
    size_t bytes = 0;
    size_t limit = SIZE_MAX;  // bytes past which a request has been refused or cut
};

// Grows s to `bytes`, or as much as alloc(size) (null when refused) and a share
// of free_bytes() give, down to `least`.  A size that was refused is not asked
// for again.  The old buffer is released once the new one is there.
template <typename Alloc, typename Release, typename Free>
void grow(Slots* s, size_t bytes, size_t least, Alloc alloc, Release release, Free free_bytes) {
    if (std::min(bytes, s->limit) <= s->bytes) return;
    const size_t share = free_bytes() / kOptionalShare;
    if (bytes > share) s->limit = std::min(s->limit, share);
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

// alloc(n) for a buffer a call cannot do without: where it is refused and s holds
// one that calls can do without, that one is released first.
template <typename Alloc, typename Release>
void* take(Slots* s, size_t n, Alloc alloc, Release release) {
    void* p = alloc(n);
    if (p || !s->p) return p;
    release(s->p);
    s->p = nullptr;
    s->bytes = 0;
    return alloc(n);
}

// Replaces the buffer *p of *cap elements by one of n; alloc(p, n) is 0 when given.
// Refused, it leaves none, of no elements, so that the next request asks again.
template <typename T, typename Alloc, typename Release>
int replace(T** p, size_t* cap, size_t n, Alloc alloc, Release release) {
    if (*p) release(*p);
    *p = nullptr;
    *cap = 0;
    const int rc = alloc(p, n);
    if (rc == 0) *cap = n;
    return rc;
}

}  // namespace sl
