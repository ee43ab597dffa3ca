// optional_buffers.hpp -- device buffers that make a call faster and that it
// can do without: plain C++, checked without a device.
#pragma once
#include <stddef.h>

namespace lqcd {

// Both buffers of p, kept from before or allocated now (alloc(double**, bytes)
// is true on success), or neither: false, and what p held is given back
// (release(double*)).
template <class Alloc, class Release>
bool both_or_neither(double* (&p)[2], size_t bytes, Alloc alloc, Release release)
{
    for (int k = 0; k < 2; ++k) {
        if (p[k] || alloc(&p[k], bytes)) continue;
        p[k] = nullptr;
        if (p[1 - k]) release(p[1 - k]);
        p[1 - k] = nullptr;
        return false;
    }
    return true;
}

} // namespace lqcd
