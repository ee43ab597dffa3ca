// limits.hpp -- lattice geometry, the sizes the device can address and those of
// launches: plain C++, so that the choices made from them can be checked without
// a device.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace lqcd {

constexpr int kMaxDim = 4;
// threads of a workgroup, where a kernel has no number of its own, and the most
// workgroups of a reduction
constexpr int kBlock = 256;
constexpr int kMaxReduceBlocks = 4096;
// the planes behind one buffer resource span less than 2^32 bytes: the device
// addresses them with 32-bit offsets
constexpr uint64_t kMaxPlaneBytes = 0xFFFFFFFFull;

struct Geom {
    int dim;
    int extent[kMaxDim];
    int64_t stride[kMaxDim];
    int64_t nsite;   // number of sites
    int64_t npad;    // row length of every SoA plane (>= nsite, multiple of 256)
};

// bytes of the link planes of one direction: 9 complex entries of two reals
// of `elem` bytes for every site
inline uint64_t link_direction_bytes(int64_t npad, size_t elem) { return (uint64_t)npad * 9 * 2 * elem; }

// whether one resource reaches the links of a direction; a lattice or chain
// past this is refused
inline bool direction_addressable(int64_t npad, size_t elem)
{
    return link_direction_bytes(npad, elem) <= kMaxPlaneBytes;
}

// whether one resource reaches the links of all D directions (AllLinks in
// k_clover.hip); kernels that need it leave larger lattices to the ones with
// a resource per direction
inline bool all_links_addressable(const Geom& g, size_t elem)
{
    return link_direction_bytes(g.npad, elem) * (uint64_t)g.dim <= kMaxPlaneBytes;
}

} // namespace lqcd
