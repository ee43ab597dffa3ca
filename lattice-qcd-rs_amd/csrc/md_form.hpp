// md_form.hpp -- the forms of an MD launch: plain C++, checked without a device.
#pragma once

namespace lqcd {

// What an MD launch does besides its kick (+ drift).  The Hamiltonian sums it
// can produce on the way: the plaquette sum as
// sum_mu Re Tr(U_mu(x) Sigma_mu(x)) over the links it reads (each plaquette
// enters through each of its 4 links: sum over links = 4 sum over plaquettes)
// and the momentum sum sum_mu,a e^a_mu(x)^2 of E before the kick
// (SUMS_BEFORE_KICK: the first launch of a trajectory, H_old) or after it
// (SUMS_AFTER_KICK: the final kick, H_new).  KICK_TWICE: no sums, two kicks
// (kick_link in md_device.hpp).
enum MdSums { SUMS_NONE = 0, SUMS_BEFORE_KICK = 1, SUMS_AFTER_KICK = 2, KICK_TWICE = 3 };
constexpr bool md_sums(int form) { return form == SUMS_BEFORE_KICK || form == SUMS_AFTER_KICK; }

// whether a launch with or without a drift, of a work decomposition that sums
// or does not, is built in this form and has what it writes to
inline bool md_form_valid(int form, bool drift, bool can_sum, bool has_partials)
{
    switch (form) {
    case SUMS_NONE: return true;
    case SUMS_BEFORE_KICK: return drift && can_sum && has_partials;
    case SUMS_AFTER_KICK: return !drift && can_sum && has_partials;
    case KICK_TWICE: return drift;
    default: return false;
    }
}

} // namespace lqcd
