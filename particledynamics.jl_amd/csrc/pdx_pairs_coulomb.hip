// Instantiations of the pair kernels: Coulomb alone.
#include "pdx_pair_kernels.hpp"

namespace pdx {
namespace pairk {
template void launch_model<PDX_PAIR_NONE>(bool, bool, int, int, dim3, hipStream_t, const PairArgs &);
template void launch_cells<PDX_PAIR_NONE>(bool, bool, int, dim3, hipStream_t, const PairArgs &, const CellArgs &);
}  // namespace pairk
}  // namespace pdx
