// Instantiations of the K build kernels with bra row and partner angular momenta 0 and 0, any operator terms.
#include "exchange_impl.hpp"

namespace lsjk {
template void launch_k_ket_l12<0, 0, false>(int, int, int, const KArgs&, const KGroups&, const KUnitG*, int, hipStream_t);
}  // namespace lsjk
