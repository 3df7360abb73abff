// Exchange gradient on gfx950: G (natom x 3) += d/dR sum D13_ac D24_bd (ab|cd) over a symmetric pair
// list (reference src/cpp/intbox/cpu/exchange_grad.cpp), shared by the translation units that
// instantiate it (exchange_grad_<L1><L2>.hip: one per class of the lane's pair).
//
// Each unordered primitive pair P = (a, b), its shell of higher angular momentum first, is held by a
// lane; the wave walks the pairs Q = (c, d) of one class at wave-uniform addresses, in bound order.
// With E = sum_P sum_Q sum_abcd (ab|cd) [D13_ac D24_bd + D13_bc D24_ad + D13_ad D24_bc + D13_bd D24_ac]
// (a pair of one primitive with itself counted half), the part of dE at P's own centres collects the
// same weight with P and Q exchanged, so over the full square of pairs a lane needs
//   dE/dA, dE/dB of P = sum_Q sum_abcd Gamma_abcd d(ab|cd)/dA, d(ab|cd)/dB,
//   Gamma = 2 [X13_ac X24_bd + X13_bc X24_ad + X13_ad X24_bc + X13_bd X24_ac],
// once with X the symmetric parts of D13 and D24 and, when both have one, once with their
// antisymmetric parts (the cross terms cancel).  Six registers per lane take the sums; there is no
// atomic per quartet, and each derivative integral of a pair of pairs is formed once per side
// instead of once for each of its eight orderings.
//
// What bounds it: FP64 VALU where classes are large (the derivative integrals and their weights, a
// few hundred FMAs per quartet), latency below that.
#pragma once
#include "exchange_impl.hpp"

namespace lsjk {

// One pair of the gradient's lists: p, Kp (as the K entries; halved for a primitive with itself), P,
// P - A, A - B, 1/(2p), 2 alpha, 2 beta, {cart A, cart B}, {block A, block B}.
struct GPair {
    double p, K, P[3], PA[3], AB[3], i2p, alpha2, beta2;
    int cartA, cartB, blkA, blkB;
};

template <bool UNIFORM>
__device__ __forceinline__ GPair load_gpair(const double* __restrict__ g)
{
    auto ld = [&](int i) __attribute__((always_inline)) {
        if constexpr (UNIFORM)
            return ld_const(g + i);
        else
            return g[i];
    };
    GPair e;
    e.p = ld(0);
    e.K = ld(1);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        e.P[k] = ld(2 + k);
        e.PA[k] = ld(5 + k);
        e.AB[k] = ld(8 + k);
    }
    e.i2p = ld(11);
    e.alpha2 = ld(12);
    e.beta2 = ld(13);
    const long long a = __double_as_longlong(ld(14)), b = __double_as_longlong(ld(15));
    e.cartA = (int)a;
    e.cartB = (int)(a >> 32);
    e.blkA = (int)b;
    e.blkB = (int)(b >> 32);
    return e;
}

// One quartet's contribution to dE/dA and dE/dB of the lane's pair e12, from 2-D Rys integrals with
// L1 and L2 raised by one:
//   d/dA_x (ab|cd) = 2 alpha (a+1x b|cd) - a_x (a-1x b|cd), likewise B with beta.
// nslice > 1 (classes with a (c, d) loop only): this wave takes the (c, d) components slice, slice +
// nslice, ...  gac..gbd: whether the ordering that takes X24 between those two shells passes the sieve; one that
// fails gets no weight.
template <int L1, int L2, int L3, int L4>
__device__ __forceinline__ void k_quartet_grad(const RysTable& tab, const double* s_tab, const Ewald& ew,
                                               const GPair& e12, const GPair& e34, const double* __restrict__ X13,
                                               const double* __restrict__ X24, int ldx, bool gac, bool gad,
                                               bool gbc, bool gbd, int slice, int nslice,
                                               double (&gA)[3], double (&gB)[3])
{
    constexpr int N1 = ncart(L1), N2 = ncart(L2), N3 = ncart(L3), N4 = ncart(L4);
    constexpr int NR = (L1 + L2 + L3 + L4 + 1) / 2 + 1;
    constexpr bool kExpand = grad_expanded(L1, L2, L3, L4);
    const double p = e12.p, q = e34.p;
    const double pq = p + q;
    const double rpq = rsqrt_pos(pq);
    const double ipq = rpq * rpq;
    const double rho = p * q * ipq;
    double PQ[3];
#pragma unroll
    for (int k = 0; k < 3; k++) PQ[k] = e12.P[k] - e34.P[k];
    const double r2 = PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2];
    const double base = e12.K * e34.K * rpq;  // 2 pi^(5/2) K_AB K_CD / (p q sqrt(p + q))
    const double qf = q * ipq, pf = p * ipq;
    // rows of the four weight blocks
    const double *x13a = X13 + (size_t)e12.cartA * ldx, *x13b = X13 + (size_t)e12.cartB * ldx;
    const double *x24a = X24 + (size_t)e12.cartA * ldx, *x24b = X24 + (size_t)e12.cartB * ldx;
    const int oc = e34.cartA, od = e34.cartB;
    // weight blocks in registers for the expanded classes
    double w13ac[kExpand ? N1 : 1][kExpand ? N3 : 1], w13ad[kExpand ? N1 : 1][kExpand ? N4 : 1];
    double w13bc[kExpand ? N2 : 1][kExpand ? N3 : 1], w13bd[kExpand ? N2 : 1][kExpand ? N4 : 1];
    double w24ac[kExpand ? N1 : 1][kExpand ? N3 : 1], w24ad[kExpand ? N1 : 1][kExpand ? N4 : 1];
    double w24bc[kExpand ? N2 : 1][kExpand ? N3 : 1], w24bd[kExpand ? N2 : 1][kExpand ? N4 : 1];
    if constexpr (kExpand) {
#pragma unroll
        for (int a = 0; a < N1; a++) {
#pragma unroll
            for (int c = 0; c < N3; c++) {
                w13ac[a][c] = x13a[(size_t)a * ldx + oc + c];
                w24ac[a][c] = gac ? x24a[(size_t)a * ldx + oc + c] : 0.0;
            }
#pragma unroll
            for (int d = 0; d < N4; d++) {
                w13ad[a][d] = x13a[(size_t)a * ldx + od + d];
                w24ad[a][d] = gad ? x24a[(size_t)a * ldx + od + d] : 0.0;
            }
        }
#pragma unroll
        for (int b = 0; b < N2; b++) {
#pragma unroll
            for (int c = 0; c < N3; c++) {
                w13bc[b][c] = x13b[(size_t)b * ldx + oc + c];
                w24bc[b][c] = gbc ? x24b[(size_t)b * ldx + oc + c] : 0.0;
            }
#pragma unroll
            for (int d = 0; d < N4; d++) {
                w13bd[b][d] = x13b[(size_t)b * ldx + od + d];
                w24bd[b][d] = gbd ? x24b[(size_t)b * ldx + od + d] : 0.0;
            }
        }
    }
    for (int it = 0; it < ew.n; it++) {
        const double om = ew.omega[it];
        double d2 = 1.0;
        double pref = 2.0 * ew.alpha[it] * base;  // the 2 of Gamma
        if (__double_as_longlong(om) != __double_as_longlong(-1.0)) {  // erf-attenuated term (bit test: scalar)
            d2 = om * om / (rho + om * om);
            pref *= sqrt(d2);
        }
        double x[NR], w[NR];
        rys_roots_any<NR>(tab, s_tab, rho * d2 * r2, x, w);
        // roots one after another (not unrolled): one copy of the assembly
#pragma unroll 1
        for (int i = 0; i < NR; i++) {
            const double u = x[i] * d2;
            const double B00 = 0.5 * u * ipq;
            const double B10 = e12.i2p * (1.0 - u * qf);
            const double B01 = e34.i2p * (1.0 - u * pf);
            const double cq = u * qf, cp = u * pf;
            Axis4<double, L1 + 1, L2 + 1, L3, L4> I[3];
            rys_axis<double, L1 + 1, L2 + 1, L3, L4>(pref * w[i], e12.PA[0] - cq * PQ[0], e34.PA[0] + cp * PQ[0], B10,
                                                     B01, B00, e12.AB[0], e34.AB[0], I[0]);
            rys_axis<double, L1 + 1, L2 + 1, L3, L4>(1.0, e12.PA[1] - cq * PQ[1], e34.PA[1] + cp * PQ[1], B10, B01,
                                                     B00, e12.AB[1], e34.AB[1], I[1]);
            rys_axis<double, L1 + 1, L2 + 1, L3, L4>(1.0, e12.PA[2] - cq * PQ[2], e34.PA[2] + cp * PQ[2], B10, B01,
                                                     B00, e12.AB[2], e34.AB[2], I[2]);
            // the (a, b) components of one (c, d): V(k, i, j) is axis k's integral at powers (i, j)
            auto bra = [&](auto&& V, auto&& gamma) __attribute__((always_inline)) {
                static_for<N1>([&](auto A_) {
                    constexpr int a = decltype(A_)::value;
                    static_for<N2>([&](auto B_) {
                        constexpr int b = decltype(B_)::value;
                        const double wgt = gamma(a, b);
                        double v[3], dA[3], dB[3];
                        static_for<3>([&](auto K_) {
                            constexpr int k = decltype(K_)::value;
                            constexpr int ia = cart_lk(L1, a, k), ib = cart_lk(L2, b, k);
                            v[k] = V(K_, std::integral_constant<int, ia>{}, std::integral_constant<int, ib>{});
                            dA[k] = e12.alpha2 * V(K_, std::integral_constant<int, ia + 1>{}, std::integral_constant<int, ib>{});
                            if constexpr (ia > 0)
                                dA[k] -= double(ia) * V(K_, std::integral_constant<int, ia - 1>{}, std::integral_constant<int, ib>{});
                            dB[k] = e12.beta2 * V(K_, std::integral_constant<int, ia>{}, std::integral_constant<int, ib + 1>{});
                            if constexpr (ib > 0)
                                dB[k] -= double(ib) * V(K_, std::integral_constant<int, ia>{}, std::integral_constant<int, ib - 1>{});
                        });
                        const double wx = wgt * v[0], yz = wgt * v[1] * v[2], xz = wx * v[2], xy = wx * v[1];
                        gA[0] = fma(yz, dA[0], gA[0]);
                        gA[1] = fma(xz, dA[1], gA[1]);
                        gA[2] = fma(xy, dA[2], gA[2]);
                        gB[0] = fma(yz, dB[0], gB[0]);
                        gB[1] = fma(xz, dB[1], gB[1]);
                        gB[2] = fma(xy, dB[2], gB[2]);
                    });
                });
            };
            if constexpr (kExpand) {
                static_for<N3>([&](auto C_) {
                    constexpr int c = decltype(C_)::value;
                    static_for<N4>([&](auto D_) {
                        constexpr int d = decltype(D_)::value;
                        bra(
                            [&](auto K_, auto I_, auto J_) __attribute__((always_inline)) {
                                constexpr int k = decltype(K_)::value;
                                constexpr int ic = cart_lk(L3, c, k), id = cart_lk(L4, d, k);
                                return I[k].v[decltype(I_)::value][decltype(J_)::value][ic][id];
                            },
                            [&](int a, int b) __attribute__((always_inline)) {
                                return w13ac[a][c] * w24bd[b][d] + w13bc[b][c] * w24ad[a][d] +
                                       w13ad[a][d] * w24bc[b][c] + w13bd[b][d] * w24ac[a][c];
                            });
                    });
                });
            } else {
                // one (c, d): its 2-D integrals S(k, i, j) and the weights of the four blocks
                auto component = [&](int c, int d, auto&& S) __attribute__((always_inline)) {
                    double a3c[N1], a3d[N1], a4c[N1], a4d[N1];
#pragma unroll
                    for (int a = 0; a < N1; a++) {
                        a3c[a] = x13a[(size_t)a * ldx + oc + c];
                        a3d[a] = x13a[(size_t)a * ldx + od + d];
                        a4c[a] = gac ? x24a[(size_t)a * ldx + oc + c] : 0.0;
                        a4d[a] = gad ? x24a[(size_t)a * ldx + od + d] : 0.0;
                    }
                    double b3c[N2], b3d[N2], b4c[N2], b4d[N2];
#pragma unroll
                    for (int b = 0; b < N2; b++) {
                        b3c[b] = x13b[(size_t)b * ldx + oc + c];
                        b3d[b] = x13b[(size_t)b * ldx + od + d];
                        b4c[b] = gbc ? x24b[(size_t)b * ldx + oc + c] : 0.0;
                        b4d[b] = gbd ? x24b[(size_t)b * ldx + od + d] : 0.0;
                    }
                    bra(S, [&](int a, int b) __attribute__((always_inline)) {
                        return a3c[a] * b4d[b] + b3c[b] * a4d[a] + a3d[a] * b4c[b] + b3d[b] * a4c[a];
                    });
                };
                if constexpr (grad_unrolled(L1, L2, L3, L4)) {
                    static_for<N3 * N4>([&](auto CD_) {
                        constexpr int cd = decltype(CD_)::value, c = cd / N4, d = cd - c * N4;
                        if (nslice > 1 && cd % nslice != slice) return;
                        component(c, d, [&](auto K_, auto I_, auto J_) __attribute__((always_inline)) {
                            constexpr int k = decltype(K_)::value;
                            constexpr int ic = cart_lk(L3, c, k), id = cart_lk(L4, d, k);
                            return I[k].v[decltype(I_)::value][decltype(J_)::value][ic][id];
                        });
                    });
                } else {
#pragma unroll 1
                    for (int cd = slice; cd < N3 * N4; cd += nslice) {
                        const int c = cd / N4, d = cd - c * N4;
                        double S[3][L1 + 2][L2 + 2];
#pragma unroll
                        for (int k = 0; k < 3; k++) {
                            const int ic = cart_lk(L3, c, k), id = cart_lk(L4, d, k);
#pragma unroll
                            for (int ia = 0; ia < L1 + 2; ia++)
#pragma unroll
                                for (int ib = 0; ib < L2 + 2; ib++) S[k][ia][ib] = I[k].v[ia][ib][ic][id];
                        }
                        component(c, d, [&](auto K_, auto I_, auto J_) __attribute__((always_inline)) {
                            return S[decltype(K_)::value][decltype(I_)::value][decltype(J_)::value];
                        });
                    }
                }
            }
        }
    }
}

// Lanes hold pairs of class (L1 L2) (64 per tile, bound order); each wave walks one chunk of the
// pairs of class (L3 L4) for one tile and adds its lanes' six derivatives to the pairs' sums with one
// atomic each.  Each ordering of a quartet is tested by the reference's sieve on its own,
// float(b12 b34) max|D24 block| >= thresp with the D24 block it multiplies (Dsh: the larger of the two
// triangles' maxima, so a symmetric D24 keeps the reference's set exactly); the quartet is evaluated
// when any of them passes.
template <int L1, int L2, int L3, int L4>
__global__ __launch_bounds__(256) void k_grad(KGradArgs a)
{
    constexpr int NR = (L1 + L2 + L3 + L4 + 1) / 2 + 1;
    extern __shared__ double s_dyn[];
    if constexpr (rys_staged(NR)) {
        rys_stage_lds<NR>(a.rys, s_dyn);
        __syncthreads();
    }
    const int lane = threadIdx.x & 63;
    const long long wid = (long long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ntile = (a.n1 + 63) / 64;
    // wave -> (chunk, slice of the (c, d) components, tile)
    const long long row = wid / ntile;
    const int tile = (int)(wid - row * ntile);
    const int chunk = (int)(row / a.nslice), slice = (int)(row - (long long)chunk * a.nslice);
    const long long k0 = (long long)chunk * a.chunk;
    if (k0 >= a.n2) return;
    const int k1 = (int)min((long long)a.n2, k0 + a.chunk);
    const int i = tile * 64 + lane;
    const bool active = i < a.n1;
    const int ii = active ? i : a.n1 - 1;
    const GPair e12 = load_gpair<false>(a.g1 + (size_t)ii * kGPairDoubles);
    const float b12 = active ? a.b1[ii] : 0.0f;
    const float b12top = ld_const(a.b1 + tile * 64);
    const double thr = (double)a.thresp;
    const double dmax = __longlong_as_double((long long)a.sc->dmax_bits);
    const double *dshA = a.Dsh + (size_t)e12.blkA * a.nblk, *dshB = a.Dsh + (size_t)e12.blkB * a.nblk;
    double gA[3] = {0.0, 0.0, 0.0}, gB[3] = {0.0, 0.0, 0.0};
    bool hit = false;
    for (int k = (int)k0; k < k1; k++) {
        const float b34 = ld_const(a.b2 + k);
        if ((double)(b12top * b34) * dmax < thr) break;  // bounds are sorted: no later pair passes
        const GPair e34 = load_gpair<true>(a.g2 + (size_t)k * kGPairDoubles);
        const double bb = (double)(b12 * b34);
        const bool gac = active && bb * dshA[e34.blkA] >= thr, gad = active && bb * dshA[e34.blkB] >= thr;
        const bool gbc = active && bb * dshB[e34.blkA] >= thr, gbd = active && bb * dshB[e34.blkB] >= thr;
        if (gac || gad || gbc || gbd) {
            k_quartet_grad<L1, L2, L3, L4>(a.rys, s_dyn, a.ew, e12, e34, a.X13, a.X24, a.ldx, gac, gad, gbc, gbd, slice,
                                           a.nslice, gA, gB);
            hit = true;
        }
    }
    if (hit) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            atomic_add(a.gp + (size_t)i * 6 + d, gA[d]);
            atomic_add(a.gp + (size_t)i * 6 + 3 + d, gB[d]);
        }
    }
}

template <int L1, int L2>
void launch_k_grad_l12(int L3, int L4, const KGradArgs& a, hipStream_t s)
{
    const long long waves = (long long)((a.n1 + 63) / 64) * ((a.n2 + a.chunk - 1) / a.chunk) * a.nslice;
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
#define CASE(C, D)                                                                               \
    if (L3 == C && L4 == D) {                                                                    \
        constexpr int NR = (L1 + L2 + C + D + 1) / 2 + 1;                                        \
        const size_t lds = rys_staged(NR) ? rys_lds_doubles(NR) * sizeof(double) : 0; \
        hipLaunchKernelGGL((k_grad<L1, L2, C, D>), grid, block, lds, s, a);                      \
        return;                                                                                  \
    }
    CASE(0, 0) CASE(1, 0) CASE(1, 1) CASE(2, 0) CASE(2, 1) CASE(2, 2)
#undef CASE
}

}  // namespace lsjk
