// Instantiations of the pair kernels: soft repulsion.
#include "pdx_pair_kernels.hpp"

namespace pdx {
namespace pairk {
template void launch_model<PDX_PAIR_SOFT>(bool, bool, int, int, dim3, hipStream_t, const PairArgs &);
template void launch_cells<PDX_PAIR_SOFT>(bool, bool, int, dim3, hipStream_t, const PairArgs &, const CellArgs &);
template void launch_acc<PDX_PAIR_SOFT>(int, bool, int, dim3, hipStream_t, const PairArgs &, int);
}  // namespace pairk
}  // namespace pdx
