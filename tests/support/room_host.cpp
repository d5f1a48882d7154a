// Host build of the reservation rule (photons-on-mt3000_amd/csrc/p2p_room.h) for
// tests/test_room.py.  No device is used.
#include "../../photons-on-mt3000_amd/csrc/p2p_room.h"

extern "C" {

// attempts on `room` elements (fails otherwise, with `error`); the sizes asked for go to asked[0 .. *n)
int room_reserve(long long want, long long least, long long room, int error, long long *asked, int *n)
{
    *n = 0;
    return pp2p::reserve_down(want, least, [&](long long k) {
        asked[(*n)++] = k;
        return k <= room ? hipSuccess : static_cast<hipError_t>(error);
    });
}

long long room_modest(long long want, long long each, long long free_bytes)
{
    return pp2p::modest(want, (size_t)each, (size_t)free_bytes);
}

}  // extern "C"
