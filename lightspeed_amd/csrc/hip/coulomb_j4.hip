// Instantiations of the J kernels with bra Hermite order 4.
#include "coulomb_impl.hpp"

namespace lsjk {
template void launch_j_l12<4>(int, int, const JQuartetArgs&, const JTask*, int, unsigned int*, hipStream_t);
}  // namespace lsjk
