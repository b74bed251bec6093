// alloc_set.h — device buffers that are only of use together.
#pragma once
#include <stddef.h>

struct BufferReq {
    void** ptr;
    size_t bytes;
};

// Allocates every buffer with alloc(void**, bytes), or, if one cannot be had,
// none: those made so far go back to release(void*) and all pointers are null,
// so that a later call starts over.  Returns the first failing status, or 0.
template <size_t N, class Alloc, class Release>
int alloc_set(const BufferReq (&req)[N], Alloc alloc, Release release) {
    for (size_t i = 0; i < N; i++) {
        *req[i].ptr = nullptr;
        const int e = (int)alloc(req[i].ptr, req[i].bytes);
        if (e == 0) continue;
        *req[i].ptr = nullptr;
        for (size_t k = 0; k < i; k++) {
            release(*req[k].ptr);
            *req[k].ptr = nullptr;
        }
        return e;
    }
    return 0;
}
