// Instantiations of the exchange-gradient kernels with the lane's pair of class (2 2).
#include "exchange_grad_impl.hpp"

namespace lsjk {
template void launch_k_grad_l12<2, 2>(int, int, const KGradArgs&, hipStream_t);
}  // namespace lsjk
