// launch_order.hpp -- the order in which the workgroups of a stencil kernel take
// the blocks of sites: plain C++, checked without a device.
//
// Workgroup b runs on XCD b mod 8, so in storage order the blocks around a
// block run on the other XCDs and its links come from memory once for each.  An
// order is given by P and G:
//   P < 0   storage order;
//   P = 0   each XCD a contiguous eighth of the blocks (xcd_remap);
//   P > 0   the same, walked in slabs of the slowest direction (slab_block): P
//           blocks per slice, G slices, the slice index fastest.
#pragma once
#include "limits.hpp"

namespace lqcd {

// Slabs for workgroups of `block` sites, or P = G = 0 where the lattice does not
// allow them (whole workgroups per slice of the slowest direction, 8 | its
// extent).
inline void slab_shape(const Geom& g, int64_t block, int64_t& P, int64_t& G)
{
    const int64_t Ls = g.extent[g.dim - 1], slice = g.nsite / Ls;
    const bool fits = slice % block == 0 && Ls % 8 == 0;
    P = fits ? slice / block : 0;
    G = fits ? Ls / 8 : 0;
}

// The plaquette sums: at most kMaxReduceBlocks workgroups of kBlock sites, which
// take several passes over lattices past 2^20 sites.
// D = 4 (us, storage -> this order): f32 32^4 154 -> 115 (contiguous 117), 24^4 55
// -> 41, 48^3 x 96 1726 -> 1608; f64 16^4 19.6 -> 16.7, 24^4 86 -> 69 (contiguous
// 75), 32^4 223 -> 213 (contiguous 256).
// D = 2 and 3: contiguous where the lattice is more than a block per CU and one
// pass covers it: f64 48^3 19.2 -> 16.9, 64^3 39.4 -> 29.2, 100^3 132 -> 125, 512^2
// 28.0 -> 21.4, 1024^2 90 -> 63; f32 96^3 58.6 -> 47.2, 1024^2 43.7 -> 29.3.  Slabs are
// level or behind (f32 1024^2 59.5).  With more passes the XCDs are an eighth of
// a pass apart and storage order is ahead: f64 104^3 143 against 177, 128^3 234 against
// 281, 1200^2 101 against 113, 2048^2 260 against 280; f64 256^2, one block per CU, 7.0
// against 7.6.
inline void plaquette_order(const Geom& g, int64_t& P, int64_t& G)
{
    const int64_t blocks = (g.nsite + kBlock - 1) / kBlock;
    const bool one_pass = blocks <= kMaxReduceBlocks;
    P = G = 0;
    if (g.dim == 4) {
        if (one_pass) slab_shape(g, kBlock, P, G);
    } else if (!one_pass || blocks <= 256) {
        P = -1;
    }
}

// The force kernel, workgroups of `block` sites.
// D = 3 and 4 in slabs (us, storage -> this order, same bits): f64 16^4 47.6 -> 36.3,
// 24^4 255 -> 180 (contiguous 219), 32^4 596 -> 560, 15x13x11x17 33.1 -> 26.5, 128^3
// 743 -> 658; f32 24^4 128 -> 86, 32^4 348 -> 276.
// D = 2 contiguous: a slice is one row, and slabs walk down the rows.  f64 512^2
// 53 -> 36 (slabs 38), 1024^2 194 -> 130 (178), 1500^2 352 -> 265, 2500^2 988 -> 742;
// f32 1024^2 80 -> 71 (106), 2500^2 610 -> 464.  Storage order where the ranges of the
// XCDs start a multiple of 2^18 sites (4 MiB of a plane) apart, so that all eight
// read the same channels: f64 2048^2 494 against 651 (slabs 515), 1024 x 4096 499
// against 658, 2048 x 1024 246 against 256; f32 2048^2 304 against 312 (363).
inline void force_order(const Geom& g, int64_t block, int64_t& P, int64_t& G)
{
    slab_shape(g, block, P, G);
    if (g.dim != 2) return;
    G = 0;
    P = g.nsite % (8LL << 18) == 0 ? -1 : 0;
}

} // namespace lqcd
