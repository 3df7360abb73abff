// Instantiations of the exchange-gradient kernels with the lane's pair of class (0 0).
#include "exchange_grad_impl.hpp"

namespace lsjk {
template void launch_k_grad_l12<0, 0>(int, int, const KGradArgs&, hipStream_t);
}  // namespace lsjk
