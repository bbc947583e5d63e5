// The neighbour stages (density and nearest-higher, every metric and kernel) of
// one dimension, CLUE_NEIGHBOUR_D, in one precision, CLUE_NEIGHBOUR_T. The Makefile
// compiles this file once per dimension and precision so that the heaviest
// instantiations build in parallel.
#include "clue_stages_impl.h"

#if !defined(CLUE_NEIGHBOUR_D) || !defined(CLUE_NEIGHBOUR_T)
#error "CLUE_NEIGHBOUR_D (1..10) and CLUE_NEIGHBOUR_T (float, double) must be defined"
#endif

namespace clue_dev {

template void launch_neighbour_d<CLUE_NEIGHBOUR_D, CLUE_NEIGHBOUR_T>(
    const NeighbourLaunch<CLUE_NEIGHBOUR_T>&, bool);

}  // namespace clue_dev
