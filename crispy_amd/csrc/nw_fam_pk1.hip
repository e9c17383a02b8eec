// Packed NW family 1: its slice widths (kPkFamilies), one launch for the
// ACGT-only read sets and one with the upper code bits.
#include "nw_pk.hpp"

namespace crispy {

void launch_nw_pk_family1(hipStream_t s, unsigned slots, const NwFusedArgs &a, const PkLaunchArgs &k) {
  launch_nw_pk_family<1>(s, slots, a, k);
}

}  // namespace crispy
