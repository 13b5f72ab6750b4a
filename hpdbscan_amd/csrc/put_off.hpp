// What a wave of k_border_heavy may leave out.
#pragma once

#include <cstdint>

namespace hpd {

// A put-off border row keeps the smallest and the largest cluster found next
// to it in two words (INT_MAX and -1: none), which several waves lower and
// raise by one atomic each and read one after the other.  Whether a walk for
// cluster cl can change nothing any more: cl lies between the two, or is
// larger than the smallest of two clusters that differ.
// `best < worst`, not `best != worst`: between the two atomics of a first hit
// the words read (cl, -1), which differ without two clusters being known.  The
// smallest only falls and the largest only rises, so best < worst, read in any
// order, means that two different clusters were published; and cl between the
// two words is never outside the final ones.
constexpr bool cluster_settled(int32_t best, int32_t worst, int32_t cl) {
    return (cl >= best && cl <= worst) || (cl > best && best < worst);
}

}  // namespace hpd
