// Direct Coulomb (J) build on gfx950: Hermite (McMurchie-Davidson) J-engine.
//
// Behaviour follows IntBox::coulombCPU (reference src/cpp/intbox/cpu/coulomb.cpp:14-196):
//   * ket truncation  B34' = float(B34 * max|D block|) kept if > thresp/max12
//     (PairListUtil::truncate_ket, src/cpp/core/pair_list_util.cpp:60-123),
//   * bra truncation  B12 >= thresp/max34 (truncate_bra, pair_list_util.cpp:32-58),
//   * quartet sieve   float(B12 * B34') >= thresp (coulomb.cpp:115),
//   * Hermite densities with (-1)^|t| phases (HermiteL::cart_to_herm, hermite.cpp:9-206) and
//     the transposed bra transform (herm_to_cart, hermite.cpp:207-411).
// The same set of primitive quartets is evaluated; only the order of evaluation differs.
//
// Kernels:
//   j_ket_prep           one thread per ket pair, all classes: truncated bound, Hermite density d_u.
//   j_quartets<L12,L34>  one wave per (64 bra pairs x ket chunk) task: each lane owns one bra
//                        pair and sweeps the chunk's kets (scalar loads); Hermite integrals R_{t+u}
//                        from Boys functions or by Rys quadrature; jp_t += sum_u R_{t+u} d_u in
//                        registers (coulomb_impl.hpp).
//   j_bra_scatter        one thread per bra pair, all classes: J_ab += K sum_t E E E jp_t
//                        (symmetrised).
#include "internal.hpp"
#include "kernels.hpp"

namespace lsjk {

// ------------------------------------------------------------------ ket preparation
// One pair k of class (LA, LB), whose Hermite group starts at pair hstart and buffer offset hoff.
template <int LA, int LB>
__device__ __forceinline__ void ket_prep(const JPrepArgs& a, int k, int hstart, size_t hoff)
{
    constexpr int NA = ncart(LA), NB = ncart(LB), L = LA + LB, H = nherm(L);
    const int ia = a.p1[k], ib = a.p2[k];
    const int ca = a.cartA[ia], cb = a.cartB[ib];
    const int pos = a.hpos[k];
    double Dt[NA][NB];
    double val = 0.0;
#pragma unroll
    for (int p = 0; p < NA; p++)
#pragma unroll
        for (int q = 0; q < NB; q++) {
            double v = a.D[(size_t)(ca + p) * a.ldD + (cb + q)];
            Dt[p][q] = v;
            val = fmax(val, fabs(v));
        }
    if (a.symmetric) {
        const double scale = (ia == ib) ? 0.5 : 1.0;
#pragma unroll
        for (int p = 0; p < NA; p++)
#pragma unroll
            for (int q = 0; q < NB; q++) {
                double v = a.D[(size_t)(cb + q) * a.ldD + (ca + p)];
                val = fmax(val, fabs(v));
                Dt[p][q] = (Dt[p][q] + v) * scale;
            }
    }
    atomicMax(&a.sc->dmax_bits, (unsigned long long)__double_as_longlong(val));
    const float B2 = (float)(val * (double)a.bound[k]);
    const bool keep = B2 > a.thre_ket;
    a.kb[pos] = keep ? B2 : -1.0f;
    double* dst = a.kd + hoff + (size_t)(pos - hstart) * H;
    float* dst32 = a.kd32 ? a.kd32 + hoff + (size_t)(pos - hstart) * H : nullptr;
    if (!keep) {
#pragma unroll
        for (int t = 0; t < H; t++) dst[t] = 0.0;
        if (dst32)
#pragma unroll
            for (int t = 0; t < H; t++) dst32[t] = 0.0f;
        return;
    }
    atomicMax(&a.sc->max34_bits, __float_as_uint(B2));
    const double eA = a.eA[ia], eB = a.eB[ib];
    const double p = eA + eB, ip = 1.0 / p;
    const double Ax = a.xA[ia], Ay = a.yA[ia], Az = a.zA[ia];
    const double Bx = a.xB[ib], By = a.yB[ib], Bz = a.zB[ib];
    const double Px = (eA * Ax + eB * Bx) * ip, Py = (eA * Ay + eB * By) * ip, Pz = (eA * Az + eB * Bz) * ip;
    HermE<LA, LB> Ex, Ey, Ez;
    hermite_E<LA, LB>(0.5 * ip, Px - Ax, Px - Bx, Ex);
    hermite_E<LA, LB>(0.5 * ip, Py - Ay, Py - By, Ey);
    hermite_E<LA, LB>(0.5 * ip, Pz - Az, Pz - Bz, Ez);
    const double Kab = a.K[k];
    static_for<H>([&](auto T_) {
        constexpr int t = decltype(T_)::value;
        constexpr int tx = herm_tx(t), ty = herm_ty(t), tz = herm_tz(t);
        double s = 0.0;
        static_for<NA>([&](auto P_) {
            constexpr int p = decltype(P_)::value;
            constexpr int ax = cart_lx(LA, p), ay = cart_ly(LA, p), az = cart_lz(LA, p);
            static_for<NB>([&](auto Q_) {
                constexpr int q = decltype(Q_)::value;
                constexpr int bx = cart_lx(LB, q), by = cart_ly(LB, q), bz = cart_lz(LB, q);
                if constexpr (tx <= ax + bx && ty <= ay + by && tz <= az + bz)
                    s += Ex.v[tx][ax][bx] * Ey.v[ty][ay][by] * Ez.v[tz][az][bz] * Dt[p][q];
            });
        });
        const double v = (((tx + ty + tz) & 1) ? -Kab : Kab) * s;
        dst[t] = v;
        if (dst32) dst32[t] = (float)v;
    });
}

// ------------------------------------------------------------------ gradient (bra centres)
// dE/dA_x = sum_ab Dsym_ab K_ab sum_t [2 alpha E^{a+1x,b}_tx - a_x E^{a-1x,b}_tx] E_ty E_tz V_t, the
// derivative of the primitive, d phi_a / dA_x = 2 alpha phi_{a+1x} - a_x phi_{a-1x}, expanded in
// Hermite Gaussians at P (t <= L12 + 1); likewise dE/dB with beta and b.  Dsym is the bra density
// block symmetrised as in the J bra transform (both triangles, 1/2 for a primitive with itself).
// The sum over both bra and ket roles gives the full gradient (reference coulomb_grad.cpp:19-563).
template <int LA, int LB>
__global__ __launch_bounds__(256) void j_grad_scatter(JGradArgs a, int k0, int nk, int hstart, size_t hoff)
{
    constexpr int NA = ncart(LA), NB = ncart(LB), L = LA + LB, H = nherm(L + 1);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nk) return;
    const int k = k0 + i;
    const float max34 = __uint_as_float(a.sc->max34_bits);
    const float thre_bra = a.thresp / max34;
    if (!(a.bound[k] >= thre_bra)) return;
    const int ia = a.p1[k], ib = a.p2[k];
    const double* vp = a.vp + hoff + (size_t)(a.hpos[k] - hstart) * H;
    double V[H];
#pragma unroll
    for (int t = 0; t < H; t++) V[t] = vp[t];
    const double eA = a.eA[ia], eB = a.eB[ib];
    const double p = eA + eB, ip = 1.0 / p;
    const double Ax = a.xA[ia], Ay = a.yA[ia], Az = a.zA[ia];
    const double Bx = a.xB[ib], By = a.yB[ib], Bz = a.zB[ib];
    const double Px = (eA * Ax + eB * Bx) * ip, Py = (eA * Ay + eB * By) * ip, Pz = (eA * Az + eB * Bz) * ip;
    HermE<LA + 1, LB + 1> Ex, Ey, Ez;
    hermite_E<LA + 1, LB + 1>(0.5 * ip, Px - Ax, Px - Bx, Ex);
    hermite_E<LA + 1, LB + 1>(0.5 * ip, Py - Ay, Py - By, Ey);
    hermite_E<LA + 1, LB + 1>(0.5 * ip, Pz - Az, Pz - Bz, Ez);
    const double scale = (a.symmetric && ia == ib) ? 0.5 : 1.0;
    const int ca = a.cartA[ia], cb = a.cartB[ib];
    double gA[3] = {0.0, 0.0, 0.0}, gB[3] = {0.0, 0.0, 0.0};
    // one-axis factor of the shifted function: sum over t of the axis, for exponents (i1, j1)
    static_for<NA>([&](auto P_) {
        constexpr int pa = decltype(P_)::value;
        constexpr int ax = cart_lx(LA, pa), ay = cart_ly(LA, pa), az = cart_lz(LA, pa);
        static_for<NB>([&](auto Q_) {
            constexpr int qb = decltype(Q_)::value;
            constexpr int bx = cart_lx(LB, qb), by = cart_ly(LB, qb), bz = cart_lz(LB, qb);
            double Dv = a.D[(size_t)(ca + pa) * a.ldD + (cb + qb)];
            if (a.symmetric) Dv = (Dv + a.D[(size_t)(cb + qb) * a.ldD + (ca + pa)]) * scale;
            if (Dv == 0.0) return;
            double dA[3] = {0.0, 0.0, 0.0}, dB[3] = {0.0, 0.0, 0.0};
            static_for<H>([&](auto T_) {
                constexpr int t = decltype(T_)::value;
                constexpr int tx = herm_tx(t), ty = herm_ty(t), tz = herm_tz(t);
                const double v = V[t];
                // plain factors (t within reach of the unshifted exponents)
                const double ex = (tx <= ax + bx) ? Ex.v[tx][ax][bx] : 0.0;
                const double ey = (ty <= ay + by) ? Ey.v[ty][ay][by] : 0.0;
                const double ez = (tz <= az + bz) ? Ez.v[tz][az][bz] : 0.0;
                // shifted factors: 2 alpha E^{a+1,b} - a E^{a-1,b} (bra A) and 2 beta E^{a,b+1} - b E^{a,b-1}
                auto shiftA = [&](const HermE<LA + 1, LB + 1>& E, int tt, int i1, int j1) __attribute__((always_inline)) {
                    double s = (tt <= i1 + 1 + j1) ? 2.0 * eA * E.v[tt][i1 + 1][j1] : 0.0;
                    if (i1 > 0 && tt <= i1 - 1 + j1) s -= i1 * E.v[tt][i1 - 1][j1];
                    return s;
                };
                auto shiftB = [&](const HermE<LA + 1, LB + 1>& E, int tt, int i1, int j1) __attribute__((always_inline)) {
                    double s = (tt <= i1 + j1 + 1) ? 2.0 * eB * E.v[tt][i1][j1 + 1] : 0.0;
                    if (j1 > 0 && tt <= i1 + j1 - 1) s -= j1 * E.v[tt][i1][j1 - 1];
                    return s;
                };
                dA[0] += shiftA(Ex, tx, ax, bx) * ey * ez * v;
                dA[1] += ex * shiftA(Ey, ty, ay, by) * ez * v;
                dA[2] += ex * ey * shiftA(Ez, tz, az, bz) * v;
                dB[0] += shiftB(Ex, tx, ax, bx) * ey * ez * v;
                dB[1] += ex * shiftB(Ey, ty, ay, by) * ez * v;
                dB[2] += ex * ey * shiftB(Ez, tz, az, bz) * v;
            });
#pragma unroll
            for (int d = 0; d < 3; d++) {
                gA[d] += Dv * dA[d];
                gB[d] += Dv * dB[d];
            }
        });
    });
    const double Kab = a.K[k];
    const int atA = a.atomA[ia], atB = a.atomB[ib];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        atomic_add(a.G + 3 * atA + d, Kab * gA[d]);
        atomic_add(a.G + 3 * atB + d, Kab * gB[d]);
    }
}

// ------------------------------------------------------------------ bra scatter
template <int LA, int LB>
__device__ __forceinline__ void bra_scatter(const JScatterArgs& a, int k, int hstart, size_t hoff)
{
    constexpr int NA = ncart(LA), NB = ncart(LB), L = LA + LB, H = nherm(L);
    if (a.screen) {
        const float max34 = __uint_as_float(a.sc->max34_bits);
        const float thre_bra = a.thresp / max34;
        if (!(a.bound[k] >= thre_bra)) return;
    }
    const int ia = a.p1[k], ib = a.p2[k];
    const int pos = a.hpos[k];
    const double* jp = a.jp + hoff + (size_t)(pos - hstart) * H;
    double jt[H];
    bool any = false;
#pragma unroll
    for (int t = 0; t < H; t++) {
        jt[t] = jp[t];
        any |= (jt[t] != 0.0);
    }
    if (!any) return;
    const double eA = a.eA[ia], eB = a.eB[ib];
    const double p = eA + eB, ip = 1.0 / p;
    const double Ax = a.xA[ia], Ay = a.yA[ia], Az = a.zA[ia];
    const double Bx = a.xB[ib], By = a.yB[ib], Bz = a.zB[ib];
    const double Px = (eA * Ax + eB * Bx) * ip, Py = (eA * Ay + eB * By) * ip, Pz = (eA * Az + eB * Bz) * ip;
    HermE<LA, LB> Ex, Ey, Ez;
    hermite_E<LA, LB>(0.5 * ip, Px - Ax, Px - Bx, Ex);
    hermite_E<LA, LB>(0.5 * ip, Py - Ay, Py - By, Ey);
    hermite_E<LA, LB>(0.5 * ip, Pz - Az, Pz - Bz, Ez);
    double Kab = a.K[k];
    if (a.symmetric && ia == ib) Kab *= 0.5;
    const int ca = a.cartA[ia], cb = a.cartB[ib];
    static_for<NA>([&](auto P_) {
        constexpr int p = decltype(P_)::value;
        constexpr int ax = cart_lx(LA, p), ay = cart_ly(LA, p), az = cart_lz(LA, p);
        static_for<NB>([&](auto Q_) {
            constexpr int q = decltype(Q_)::value;
            constexpr int bx = cart_lx(LB, q), by = cart_ly(LB, q), bz = cart_lz(LB, q);
            double s = 0.0;
            static_for<H>([&](auto T_) {
                constexpr int t = decltype(T_)::value;
                constexpr int tx = herm_tx(t), ty = herm_ty(t), tz = herm_tz(t);
                if constexpr (tx <= ax + bx && ty <= ay + by && tz <= az + bz)
                    s += Ex.v[tx][ax][bx] * Ey.v[ty][ay][by] * Ez.v[tz][az][bz] * jt[t];
            });
            s *= Kab;
            atomic_add(a.J + (size_t)(ca + p) * a.ldJ + (cb + q), s);
            if (a.symmetric) atomic_add(a.J + (size_t)(cb + q) * a.ldJ + (ca + p), s);
        });
    });
}

// ------------------------------------------------------------------ launchers
#define LSJK_L2_CASES(F) F(0, 0) F(0, 1) F(0, 2) F(1, 0) F(1, 1) F(1, 2) F(2, 0) F(2, 1) F(2, 2)

// All classes of a list in one launch: a workgroup finds its class among the (at most 9) segments.  One
// launch per class cost more than the classes' own time on small lists (5 us each against 2-9 us).
// The registers are those of the heaviest class in the list's maximum angular momentum (MAXL), which
// leaves fewer waves per SIMD for the light ones; a list of 100,000 pairs still fits the device at once.
template <int MAXL, typename F>
__device__ __forceinline__ void for_segment(const JSegments& seg, F&& f)
{
    int c = 0;
    while (c + 1 < seg.n && (int)blockIdx.x >= seg.block0[c + 1]) c++;
    const int i = ((int)blockIdx.x - seg.block0[c]) * 256 + (int)threadIdx.x;
    if (i >= seg.nk[c]) return;
    const int k = seg.k0[c] + i, L1 = seg.L1[c], L2 = seg.L2[c];
#define CASE(X, Y)                                                                  \
    if constexpr (X <= MAXL && Y <= MAXL)                                           \
        if (L1 == X && L2 == Y)                                                     \
            return f(std::integral_constant<int, X>{}, std::integral_constant<int, Y>{}, k, seg.hstart[c], seg.hoff[c]);
    LSJK_L2_CASES(CASE)
#undef CASE
}

template <int MAXL>
__global__ __launch_bounds__(256) void j_ket_prep(JPrepArgs a, JSegments seg)
{
    for_segment<MAXL>(seg, [&](auto A_, auto B_, int k, int hstart, size_t hoff) __attribute__((always_inline)) {
        ket_prep<decltype(A_)::value, decltype(B_)::value>(a, k, hstart, hoff);
    });
}

template <int MAXL>
__global__ __launch_bounds__(256) void j_bra_scatter(JScatterArgs a, JSegments seg)
{
    for_segment<MAXL>(seg, [&](auto A_, auto B_, int k, int hstart, size_t hoff) __attribute__((always_inline)) {
        bra_scatter<decltype(A_)::value, decltype(B_)::value>(a, k, hstart, hoff);
    });
}

void launch_j_ket_prep(const JPrepArgs& a, const JSegments& seg, hipStream_t s)
{
    if (seg.nblock <= 0) return;
    auto* kernel = seg.maxL == 0 ? j_ket_prep<0> : seg.maxL == 1 ? j_ket_prep<1> : j_ket_prep<2>;
    hipLaunchKernelGGL(kernel, dim3(seg.nblock), dim3(256), 0, s, a, seg);
}

void launch_j_bra_scatter(const JScatterArgs& a, const JSegments& seg, hipStream_t s)
{
    if (seg.nblock <= 0) return;
    auto* kernel = seg.maxL == 0 ? j_bra_scatter<0> : seg.maxL == 1 ? j_bra_scatter<1> : j_bra_scatter<2>;
    hipLaunchKernelGGL(kernel, dim3(seg.nblock), dim3(256), 0, s, a, seg);
}

void launch_j_grad_scatter(int LA, int LB, const JGradArgs& a, int k0, int nk, int hstart, size_t hoff,
                           hipStream_t s)
{
    if (nk <= 0) return;
    dim3 grid((nk + 255) / 256), block(256);
#define CASE(X, Y)                                                                                  \
    if (LA == X && LB == Y) {                                                                       \
        hipLaunchKernelGGL((j_grad_scatter<X, Y>), grid, block, 0, s, a, k0, nk, hstart, hoff);     \
        return;                                                                                     \
    }
    CASE(0, 0) CASE(0, 1) CASE(0, 2) CASE(1, 0) CASE(1, 1) CASE(1, 2) CASE(2, 0) CASE(2, 1) CASE(2, 2)
#undef CASE
}

template <int L12>
void launch_j_l12(int L34, int route, const JQuartetArgs& a, const JTask* tasks, int ntask, unsigned int* qctr,
                  hipStream_t s);
#define LSJK_J_EXTERN(X)                                                                                   \
    extern template void launch_j_l12<X>(int, int, const JQuartetArgs&, const JTask*, int, unsigned int*, \
                                         hipStream_t);
LSJK_J_EXTERN(0) LSJK_J_EXTERN(1) LSJK_J_EXTERN(2) LSJK_J_EXTERN(3) LSJK_J_EXTERN(4) LSJK_J_EXTERN(5)
#undef LSJK_J_EXTERN

void launch_j_quartets(int L12, int L34, int route, const JQuartetArgs& a, const JTask* tasks, int ntask,
                       unsigned int* qctr, hipStream_t s)
{
    if (ntask <= 0) return;
#define CASE(X) \
    if (L12 == X) return launch_j_l12<X>(L34, route, a, tasks, ntask, qctr, s);
    CASE(0) CASE(1) CASE(2) CASE(3) CASE(4) CASE(5)
#undef CASE
}

}  // namespace lsjk
