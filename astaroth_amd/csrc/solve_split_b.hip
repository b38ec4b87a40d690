// solve_split_b.hip -- the role-split solve kernels of 16 x 8 column blocks.
#define AC_SPLIT_INSTANTIATE
#include "solve_split.h"

namespace acamd {

template void launch_split_tile<AcRealT, 16, 8>(const SolveArgs<AcRealT>&, bool, bool, int, int, hipStream_t);

}  // namespace acamd
