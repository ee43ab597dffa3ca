// geometry.hpp -- periodic lattice geometry shared by host and device code.
//
// Sites are numbered as the reference's LatticePoint::to_index
// (src/lattice.rs:909-915): s = sum_i x_i * prod_{k<i} L_k, x_0 fastest.  The
// device stores each field as a structure of arrays over sites (see
// fields.hpp), so a wavefront of 64 consecutive sites reads 64 consecutive
// values of the same matrix element: coalesced.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch_order.hpp"
#include "limits.hpp"

namespace lqcd {

// Offsets to the +dir and -dir neighbours of site s (periodic wrap).  Site
// indices of one lattice fit in 31 bits (the device field access uses 32-bit
// byte offsets), so the offsets are 32-bit.
template <int D>
struct Neighbours {
    int32_t up[D];   // s + up[d]   = site + d_hat
    int32_t dn[D];   // s + dn[d]   = site - d_hat
};

template <int D>
__device__ __forceinline__ Neighbours<D> neighbours(const Geom& g, int64_t s)
{
    Neighbours<D> n;
    uint32_t r = (uint32_t)s;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const uint32_t L = (uint32_t)g.extent[d];
        const uint32_t x = (d == D - 1) ? r : r % L;
        r /= L;
        const int32_t st = (int32_t)g.stride[d];
        n.up[d] = (x == L - 1) ? -(int32_t)(L - 1) * st : st;
        n.dn[d] = (x == 0) ? (int32_t)(L - 1) * st : -st;
    }
    return n;
}

// Workgroups are dispatched round robin over the 8 XCDs (workgroup b runs on
// XCD b mod 8).  Give XCD k the contiguous logical range
// [k q + min(k, r), ...) of n = 8 q + r blocks.
__device__ __forceinline__ int64_t xcd_remap(int64_t b, int64_t n)
{
    const int64_t k = b & 7, i = b >> 3, q = n >> 3, r = n & 7;
    return k * q + (k < r ? k : r) + i;
}

// Site block of logical block j for the slab order: P blocks per slice of the
// slowest direction, G slices per XCD slab; within a slab the slice index runs
// fastest.
__device__ __forceinline__ int64_t slab_block(int64_t j, int64_t P, int64_t G)
{
    const int64_t q = j / (G * P), r = j % (G * P);
    return (q * G + r % G) * P + r / G;
}

// Coordinates of site s, and the offsets to its neighbours along a direction
// that is known at run time only (uniform over the wave: the extents come
// through scalar registers and the coordinate through a few selects, where an
// indexed Neighbours would go through LDS).
template <int D>
struct SiteCoords {
    uint32_t x[D];

    __device__ __forceinline__ SiteCoords(const Geom& g, int64_t s)
    {
        uint32_t r = (uint32_t)s;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const uint32_t L = (uint32_t)g.extent[d];
            x[d] = (d == D - 1) ? r : r % L;
            r /= L;
        }
    }
    __device__ __forceinline__ uint32_t at(int d) const
    {
        uint32_t v = x[0];
#pragma unroll
        for (int k = 1; k < D; ++k) v = d == k ? x[k] : v;
        return v;
    }
    __device__ __forceinline__ void extent(const Geom& g, int d, int32_t& L, int32_t& st) const
    {
        L = g.extent[0];
        st = 1;
#pragma unroll
        for (int k = 1; k < D; ++k) {
            L = d == k ? g.extent[k] : L;
            st = d == k ? (int32_t)g.stride[k] : st;
        }
    }
    __device__ __forceinline__ int32_t up(const Geom& g, int d) const
    {
        int32_t L, st;
        extent(g, d, L, st);
        return (int32_t)at(d) == L - 1 ? -(L - 1) * st : st;
    }
    __device__ __forceinline__ int32_t dn(const Geom& g, int d) const
    {
        int32_t L, st;
        extent(g, d, L, st);
        return at(d) == 0 ? (L - 1) * st : -st;
    }
};

// Site block of a workgroup in the order that P and G stand for
// (launch_order.hpp).
__device__ __forceinline__ int64_t ordered_block(int64_t P, int64_t G)
{
    if (P < 0) return blockIdx.x;
    const int64_t b = xcd_remap(blockIdx.x, gridDim.x);
    return P > 0 ? slab_block(b, P, G) : b;
}

template <int D>
__device__ __forceinline__ int site_parity(const Geom& g, int64_t s);

// Index of a site in a link plane, from its site index and its number of steps
// from site s.  Site order: the site index.  Parity order (PO, lattices of
// even extents): the sites of even parity first, then the odd ones, each in
// site order; of sites 2k and 2k + 1 one has either parity, so site s is word
// s / 2 of its half.
template <int D, bool PO>
struct SiteMap {
    int64_t off[2] = {0, 0};   // first word of the half of s, and of the other

    __device__ __forceinline__ SiteMap(const Geom& g, int64_t s) : SiteMap(g, PO ? site_parity<D>(g, s) : 0) {}
    __device__ __forceinline__ SiteMap(const Geom& g, int parity)
    {
        if constexpr (PO) {
            off[0] = parity ? g.nsite / 2 : 0;
            off[1] = g.nsite / 2 - off[0];
        }
    }
    template <int STEPS>
    __device__ __forceinline__ int64_t at(int64_t s) const
    {
        if constexpr (PO) return (s >> 1) + off[STEPS & 1];
        return s;
    }
};

template <int D>
__device__ __forceinline__ int site_parity(const Geom& g, int64_t s)
{
    uint32_t r = (uint32_t)s;
    uint32_t p = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const uint32_t L = (uint32_t)g.extent[d];
        const uint32_t x = (d == D - 1) ? r : r % L;
        r /= L;
        p += x;
    }
    return (int)(p & 1);
}

} // namespace lqcd
