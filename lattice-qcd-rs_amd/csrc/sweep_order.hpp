// sweep_order.hpp -- when the checkerboard sweeps of a lattice put its links
// in parity order (SiteMap in geometry.hpp): plain C++, checked without a
// device.
#pragma once
#include <stddef.h>

namespace lqcd {

enum SweepKind { SWEEP_METROPOLIS, SWEEP_HEAT_BATH, SWEEP_OVERRELAX };

// What a sweep gains in parity order, in units of the two reorderings that it
// costs to go there and back; 0: not worth it.  The least that was measured
// (us per sweep and per two reorderings, site -> parity order, f64 first):
//                two     Metropolis,   Metropolis,    heat bath     overrelaxation
//                        1 update      10 updates                   (either kind: the lesser gain)
//   16^4          31      197 ->  188   396 ->  384    281 ->  247    314 ->  281
//   20^4          64      350 ->  291   711 ->  657    526 ->  412    586 ->  496
//   24^4         130      594 ->  437  1090 ->  966    912 ->  622    952 ->  710
//   32^4         536     1587 -> 1096  2571 -> 2413   2635 -> 1562   2556 -> 1703
//   40^4        1102     3621 -> 2543  5958 -> 5601   6297 -> 3497   6028 -> 3978
//   44^3          31      145 ->  142   287 ->  289    201 ->  183    218 ->  202
//   64^3          85      296 ->  224   569 ->  511    426 ->  330    505 ->  427
//   96^3         273      721 ->  531  1471 -> 1383   1137 ->  786   1181 ->  877
//   128^3        762     1662 -> 1267  3258 -> 3163   2894 -> 1741   2887 -> 1970
//   342^2         29      102 ->   97   202 ->  204    137 ->  131    158 ->  151
//   512^2         56      151 ->  130   344 ->  316    222 ->  184    510 ->  474
//   2048^2       939     1631 -> 1216  3726 -> 3730   2391 -> 1551   2452 -> 2190
//   f32:
//   20^4          37      277 ->  268   650 ->  633    370 ->  335    428 ->  401
//   24^4          67      353 ->  343   888 ->  874    532 ->  455    629 ->  538
//   32^4         221      730 ->  683  2122 -> 2077   1199 ->  986   1362 -> 1197
//   40^4         503     1935 -> 1783  5258 -> 5151   2791 -> 2334   3177 -> 2866
//   128^3        343      938 ->  899  2950 -> 3042   1329 -> 1235   1628 -> 1580
// Links that fit in the 32 MiB of the eight L2s stay in site order.  In f32 only
// the heat bath and overrelaxation of D = 4 gain more than plaquette, force and
// normalisation lose in this order (32^4 113 -> 141, 275 -> 306, 78 -> 88 us).
constexpr size_t kParityOrderBytes = (size_t)32 << 20;

// whether the kernels read links in parity order (LQCD_DISPATCH_DS_PO)
inline bool parity_order_built(bool f64, int dim) { return f64 || dim == 4; }

inline double parity_order_gain(SweepKind kind, bool f64, int dim, size_t link_bytes, size_t n_update)
{
    if (link_bytes < kParityOrderBytes) return 0.0;
    if (!f64) return dim == 4 && kind != SWEEP_METROPOLIS ? 0.6 : 0.0;
    const bool large = link_bytes >= 2 * kParityOrderBytes;
    if (kind != SWEEP_METROPOLIS) {
        if (dim == 4) return large ? 1.3 : 1.0;
        if (dim == 3) return large ? 0.9 : 0.5;
        return 0.2;
    }
    double gain = dim == 4 ? (large ? 0.9 : 0.3) : dim == 3 ? (large ? 0.5 : 0.1) : (large ? 0.35 : 0.15);
    // more updates per link: the loads are a smaller part
    if (n_update > 1) gain = dim == 4 ? gain * 0.3 : dim == 3 ? gain * 0.2 : 0.0;
    return gain;
}

// A lattice whose links are in parity order is put back by the first call that
// needs site order, so the order pays when the sweeps up to that call gain
// more than the two reorderings.  That is known of a sweep that outweighs
// them by itself; otherwise it is taken from the sweeps between the last two
// such calls, and of a longer stretch once it has passed the cost.  A program
// that repeats itself is then never slower than in site order, but for at most
// one round trip at its start: 32^4 Metropolis sweeps each followed by F_mu_nu
// or a download would lose 45 us a sweep, 128^3 ones 367 us.
struct SweepOrder {
    double run = 0.0;    // gains of the sweeps since the last call in site order
    double last = 0.0;   // and between the two calls before

    bool pays(double gain) const { return gain > 0.0 && (gain >= 1.0 || run >= 1.0 || last >= 1.0); }
    void swept(double gain) { run += gain; }
    // a call that needs site order, or that replaces the links
    void site_call()
    {
        if (run > 0.0) last = run;
        run = 0.0;
    }
};

} // namespace lqcd
