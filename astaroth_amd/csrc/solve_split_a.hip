// solve_split_a.hip -- the role-split solve kernels of 32 x 4 column blocks.
#define AC_SPLIT_INSTANTIATE
#include "solve_split.h"

namespace acamd {

template void launch_split_tile<AcRealT, 32, 4>(const SolveArgs<AcRealT>&, bool, bool, int, int, hipStream_t);

}  // namespace acamd
