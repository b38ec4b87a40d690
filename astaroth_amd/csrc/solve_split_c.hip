// solve_split_c.hip -- the role-split solve kernels of 64 x 4 column blocks (FP32).
#define AC_SPLIT_INSTANTIATE
#include "solve_split.h"

namespace acamd {

#if !AC_DOUBLE_PRECISION
template void launch_split_tile<AcRealT, 64, 4>(const SolveArgs<AcRealT>&, bool, bool, int, int, hipStream_t);
#endif

}  // namespace acamd
