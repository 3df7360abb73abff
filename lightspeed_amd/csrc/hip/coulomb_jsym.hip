// Instantiations of the symmetric J kernels (js_enabled).
#include "coulomb_impl.hpp"

namespace lsjk {

void launch_j_quartets_sym(int L12, int L34, int route, const JQuartetArgs& a, const JTask* tasks, int ntask,
                           unsigned int* qctr, hipStream_t s)
{
    if (ntask <= 0) return;
#define ONE(X, Y, R)                                                                                     \
    {                                                                                                    \
        auto* kernel = a.ew.plain ? j_quartets_sym<X, Y, R, true> : j_quartets_sym<X, Y, R, false>;      \
        const size_t lds = JLds<X, Y, R>::kBytes;                                                        \
        const int grid = persistent_grid((const void*)kernel, 256, lds, ((long long)ntask + 3) / 4);     \
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), lds, s, a, tasks, ntask, qctr);                \
        return;                                                                                          \
    }
#define CASE(X, Y)                                                                                       \
    if (L12 == X && L34 == Y) {                                                                          \
        if (route == kRouteMixed) ONE(X, Y, kRouteMixed) else ONE(X, Y, kRoutePlain)                    \
    }
    CASE(0, 0) CASE(1, 0) CASE(2, 0) CASE(3, 0) CASE(4, 0)
#undef CASE
#undef ONE
    throw std::runtime_error("lsjk: j_quartets_sym class not instantiated");
}

}  // namespace lsjk
