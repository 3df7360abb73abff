// Instantiations of the J kernels with bra Hermite order 2.
#include "coulomb_impl.hpp"

namespace lsjk {
template void launch_j_l12<2>(int, int, const JQuartetArgs&, const JTask*, int, unsigned int*, hipStream_t);
}  // namespace lsjk
