// Instantiations of the pair kernels: the typed models.
#include "pdx_pair_kernels.hpp"

namespace pdx {
namespace pairk {
template void launch_typed<PDX_PAIR_MIXED_LJ>(bool, bool, int, int, dim3, hipStream_t, const PairArgs &);
template void launch_typed<PDX_PAIR_MIXED_WCA>(bool, bool, int, int, dim3, hipStream_t, const PairArgs &);
template void launch_typed<PDX_PAIR_MATRIX_LJ>(bool, bool, int, int, dim3, hipStream_t, const PairArgs &);
template void launch_typed<PDX_PAIR_MATRIX_WCA>(bool, bool, int, int, dim3, hipStream_t, const PairArgs &);
}  // namespace pairk
}  // namespace pdx
