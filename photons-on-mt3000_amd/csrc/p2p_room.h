// How much to reserve ahead of need (host only; tested without a device).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

namespace pp2p {

// attempt(want), then half as much each time it runs out of memory, down to
// `least`.  Its last result.
template <class Attempt>
inline hipError_t reserve_down(long long want, long long least, const Attempt &attempt)
{
    for (long long n = std::max(want, least);; n = std::max(n / 2, least)) {
        const hipError_t e = attempt(n);
        if (e != hipErrorOutOfMemory || n <= least)
            return e;
    }
}

// `want` elements of `each` bytes, or as many as a quarter of the free memory
// holds: what follows (the list itself, another context) needs room too.
inline long long modest(long long want, size_t each, size_t free_bytes)
{
    return std::min(want, (long long)(free_bytes / 4 / each));
}

}  // namespace pp2p
