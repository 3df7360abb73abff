// Coulomb (J) quartet kernel templates, shared by the translation units that instantiate them
// (coulomb_j<L12>.hip: one per bra Hermite order; coulomb_jsym.hip: the symmetric kernels).  See
// coulomb.hip for the build they belong to.
#pragma once
#include "internal.hpp"
#include "kernels.hpp"

namespace lsjk {

// ------------------------------------------------------------------ quartets
// Arithmetic of the two routes: Real = double (FP64 route) or float (FP32 route).  The FP32 route
// forms T in FP64 (from FP64 centre differences) and uses the FP32 Rys rule; everything else of
// the quartet is FP32; the caller accumulates in FP64.
template <typename Real>
__device__ __forceinline__ Real rdiv(Real a, Real b)
{
    if constexpr (std::is_same<Real, float>::value)
        return __fdividef(a, b);
    else
        return a / b;
}

template <typename Real>
__device__ __forceinline__ Real rrsqrt(Real x)
{
    if constexpr (std::is_same<Real, float>::value)
        return __frsqrt_rn(x);
    else
        return rsqrt_pos(x);
}

template <typename Real, int NR>
__device__ __forceinline__ void roots_real(const RysTable& tab, const void* s_tab, double T, Real* x, Real* w)
{
    if constexpr (std::is_same<Real, float>::value)
        rys_roots_f32<NR, true>(static_cast<const float*>(s_tab), T, x, w);
    else
        rys_roots_any<NR>(tab, static_cast<const double*>(s_tab), T, x, w);
}

// Per-root one-dimensional Hermite factors of one bra-ket pair and operator term:
// H_0 = 1 (x: pref w_i), H_1 = U X, H_{n+1} = U (X H_n + n H_{n-1}), U = -2 rho d^2 x_i
// (coulomb.cpp:138-158).
template <typename Real, int L>
struct HermRoot {
    Real x[L + 1], y[L + 1], z[L + 1];
};

template <typename Real, int L>
__device__ __forceinline__ void herm_factors(Real pref_w, Real U, Real X, Real Y, Real Z, HermRoot<Real, L>& H)
{
    H.x[0] = pref_w;
    H.y[0] = Real(1);
    H.z[0] = Real(1);
    if constexpr (L > 0) {
        H.x[1] = U * X * H.x[0];
        H.y[1] = U * Y;
        H.z[1] = U * Z;
    }
#pragma unroll
    for (int u = 1; u < L; u++) {
        H.x[u + 1] = U * (X * H.x[u] + Real(u) * H.x[u - 1]);
        H.y[u + 1] = U * (Y * H.y[u] + Real(u) * H.y[u - 1]);
        H.z[u + 1] = U * (Z * H.z[u] + Real(u) * H.z[u - 1]);
    }
}

// Calls f(HermRoot) for every Rys root of every operator term of one bra-ket pair (BARE: of one bare 1/r
// term, its scale in c12).
// c12, c34: sqrt(2 pi^(5/2)) / p of each pair, so that c12 c34 (p + q)^(-1/2) = 2 pi^(5/2) / (p q sqrt(p + q)).
template <typename Real, int L, bool BARE, typename F>
__device__ __forceinline__ void for_each_root(const RysTable& tab, const void* s_tab, const Ewald& ew, double p12,
                                              double c12, double p34, double c34, double X, double Y, double Z, F&& f)
{
    constexpr int NR = L / 2 + 1;
    const Real p = (Real)p12, q = (Real)p34;
    const Real psum = p + q;
    const Real rs = rrsqrt(psum);
    const Real rho = p * q * (rs * rs);
    const Real base = (Real)c12 * (Real)c34 * rs;  // 2 pi^{5/2} / (p q sqrt(p+q))
    const double r2 = X * X + Y * Y + Z * Z;
    const Real Xr = (Real)X, Yr = (Real)Y, Zr = (Real)Z;
    // one operator term: Rys roots at T = rho d2 r2, Hermite factors with prefactor pref
    auto term = [&](Real pref, auto d2_) __attribute__((always_inline)) {
        const Real d2 = (Real)d2_;
        const double T = (double)(rho * d2) * r2;
        Real x[NR], w[NR];
        roots_real<Real, NR>(tab, s_tab, T, x, w);
#pragma unroll
        for (int i = 0; i < NR; i++) {
            HermRoot<Real, L> H;
            herm_factors<Real, L>(pref * w[i], Real(-2) * rho * d2 * x[i], Xr, Yr, Zr, H);
            f(H);
        }
    };
    if constexpr (BARE) {
        // one bare 1/r term, its scale in c12: no term loop
        term(base, std::integral_constant<int, 1>{});
        return;
    }
    for (int it = 0; it < ew.n; it++) {
        const double om = ew.omega[it];
        Real d2 = Real(1);
        Real pref = (Real)ew.alpha[it] * base;
        if (__double_as_longlong(om) != __double_as_longlong(-1.0)) {  // erf-attenuated term (bit test: scalar)
            const Real o = (Real)om;
            d2 = rdiv(o * o, rho + o * o);
            pref *= sqrt(d2);
        }
        term(pref, d2);
    }
}

// FP64 Hermite integrals of total order 2 .. 4 come from Boys functions by the McMurchie-Davidson
// recursion (J. Comput. Phys. 26, 218 (1978)): one polynomial (F_L) and an exponential instead of one
// polynomial per root and weight, and no sum over roots (order 4: about 130 FP64 operations against
// 340, order 2: 50 against 108), with 13 table doubles per bin against 24 nrys.  Order 0 and 1 cost the
// same either way; orders above 4 keep the factorised root sum (their recursion does not fit the
// registers).
constexpr bool j_md(int L) { return L >= 2 && L <= 4; }

template <int L, int N>
__device__ __forceinline__ void md_level(const double (&b)[L + 1], double X, double Y, double Z,
                                         double (&out)[nherm(L - N)])
{
    // R^(N)_t, |t| <= L - N, from R^(N+1): R^(n)_{t + 1_i} = X_i R^(n+1)_t + t_i R^(n+1)_{t - 1_i}
    out[0] = b[N];
    if constexpr (N < L) {
        double prev[nherm(L - N - 1)];
        md_level<L, N + 1>(b, X, Y, Z, prev);
        static_for<nherm(L - N) - 1>([&](auto I_) {
            constexpr int t = decltype(I_)::value + 1;
            constexpr int tx = herm_tx(t), ty = herm_ty(t), tz = herm_tz(t);
            // an axis of power one where there is one: its step has no second term
            constexpr int ax = tx == 1 ? 0 : ty == 1 ? 1 : tz == 1 ? 2 : tx > 0 ? 0 : ty > 0 ? 1 : 2;
            constexpr int n = ax == 0 ? tx : ax == 1 ? ty : tz;
            constexpr int lx = tx - (ax == 0), ly = ty - (ax == 1), lz = tz - (ax == 2);
            const double D = ax == 0 ? X : ax == 1 ? Y : Z;
            if constexpr (n > 1)
                out[t] = fma(D, prev[herm_index(lx, ly, lz)],
                             double(n - 1) * prev[herm_index(lx - (ax == 0), ly - (ax == 1), lz - (ax == 2))]);
            else
                out[t] = D * prev[herm_index(lx, ly, lz)];
        });
    }
}

template <int L, bool BARE>
__device__ __forceinline__ void hermite_R_md(const double* s_boys, const Ewald& ew, double p, double c12, double q,
                                             double c34, double X, double Y, double Z, double (&R)[nherm(L)])
{
    const double psum = p + q;
    const double rs = rsqrt_pos(psum);
    const double rho = p * q * (rs * rs);
    const double base = c12 * c34 * rs;  // 2 pi^{5/2} / (p q sqrt(p+q))
    const double r2 = X * X + Y * Y + Z * Z;
    double b[L + 1], F[L + 1];
    if constexpr (BARE) {
        boys_lds<L>(s_boys, rho * r2, F);
        double f = base;
#pragma unroll
        for (int n = 0; n <= L; n++) {
            b[n] = f * F[n];
            f *= -2.0 * rho;
        }
    } else {
        // the operator's terms differ in the Boys argument and the powers of d^2 only: one recursion
#pragma unroll
        for (int n = 0; n <= L; n++) b[n] = 0.0;
        for (int it = 0; it < ew.n; it++) {
            const double om = ew.omega[it];
            double d2 = 1.0, f = ew.alpha[it] * base;
            if (__double_as_longlong(om) != __double_as_longlong(-1.0)) {  // erf-attenuated term (bit test: scalar)
                d2 = om * om / (rho + om * om);
                f *= sqrt(d2);
            }
            const double rd = rho * d2;
            boys_lds<L>(s_boys, rd * r2, F);
#pragma unroll
            for (int n = 0; n <= L; n++) {
                b[n] = fma(f, F[n], b[n]);
                f *= -2.0 * rd;
            }
        }
    }
    md_level<L, 0>(b, X, Y, Z, R);
}

// Hermite Coulomb integrals R_{tuv} (t+u+v <= L) of one bra-ket pair, by Rys quadrature
// (R_{tuv} = pref * sum_i w_i Hx_t Hy_u Hz_v) or from Boys functions (j_md).
template <typename Real, int L, bool BARE>
__device__ __forceinline__ void hermite_R(const RysTable& tab, const void* s_tab, const Ewald& ew, double p12,
                                          double c12, double p34, double c34, double X, double Y, double Z,
                                          Real (&R)[nherm(L)])
{
    constexpr int HL = nherm(L);
    if constexpr (std::is_same<Real, double>::value && j_md(L))
        return hermite_R_md<L, BARE>(static_cast<const double*>(s_tab), ew, p12, c12, p34, c34, X, Y, Z, R);
#pragma unroll
    for (int t = 0; t < HL; t++) R[t] = Real(0);
    for_each_root<Real, L, BARE>(tab, s_tab, ew, p12, c12, p34, c34, X, Y, Z, [&](const HermRoot<Real, L>& H) __attribute__((always_inline)) {
        static_for<HL>([&](auto T_) {
            constexpr int t = decltype(T_)::value;
            constexpr int tx = herm_tx(t), ty = herm_ty(t), tz = herm_tz(t);
            R[t] += H.x[tx] * H.y[ty] * H.z[tz];
        });
    });
}

// High angular momentum: the same contraction factorised per Rys root, so the (L+1)(L+2)(L+3)/6
// Hermite integrals are never held at once:
//   A[uy][tz] = sum_uz Hz[tz+uz] d[ux,uy,uz];  B[ty][tz] = sum_uy Hy[ty+uy] A[uy][tz];
//   jp[tx,ty,tz] += Hx[tx+ux] B[ty][tz]   (for each ux).
template <typename Real, int L12, int L34, bool BARE, typename Acc>
__device__ __forceinline__ void hermite_contract_factorized(const RysTable& tab, const void* s_tab, const Ewald& ew,
                                                            double p12, double c12, double p34, double c34, double X,
                                                            double Y, double Z, const Real (&d)[nherm(L34)], Acc& jp)
{
    constexpr int L = L12 + L34;
    for_each_root<Real, L, BARE>(tab, s_tab, ew, p12, c12, p34, c34, X, Y, Z, [&](const HermRoot<Real, L>& H) __attribute__((always_inline)) {
        static_for<L34 + 1>([&](auto UX_) {
            constexpr int ux = decltype(UX_)::value;
            Real A[L34 + 1 - ux][L12 + 1];
            static_for<L34 + 1 - ux>([&](auto UY_) {
                constexpr int uy = decltype(UY_)::value;
                static_for<L12 + 1>([&](auto TZ_) {
                    constexpr int tz = decltype(TZ_)::value;
                    Real s = Real(0);
                    static_for<L34 + 1 - ux - uy>([&](auto UZ_) {
                        constexpr int uz = decltype(UZ_)::value;
                        constexpr int iu = herm_index(ux, uy, uz);
                        s = fma(H.z[tz + uz], d[iu], s);
                    });
                    A[uy][tz] = s;
                });
            });
            static_for<L12 + 1>([&](auto TY_) {
                constexpr int ty = decltype(TY_)::value;
                static_for<L12 + 1 - ty>([&](auto TZ_) {
                    constexpr int tz = decltype(TZ_)::value;
                    Real s = Real(0);
                    static_for<L34 + 1 - ux>([&](auto UY_) {
                        constexpr int uy = decltype(UY_)::value;
                        s = fma(H.y[ty + uy], A[uy][tz], s);
                    });
                    static_for<L12 + 1 - ty - tz>([&](auto TX_) {
                        constexpr int tx = decltype(TX_)::value;
                        constexpr int it = herm_index(tx, ty, tz);
                        jp[it] = fma(H.x[tx + ux], s, jp[it]);
                    });
                });
            });
        });
    });
}

// LDS of one j_quartets workgroup: the FP64 table (the Boys table of the class's order for j_md, the
// Rys block for nrys <= 3), then the FP32 Rys block on the mixed route.
template <int L12, int L34, int ROUTE>
struct JLds {
    static constexpr int L = L12 + L34, NR = L / 2 + 1;
    static constexpr bool HAS32 = ROUTE == kRouteMixed;
    static constexpr bool STAGED64 = j_md(L) || rys_staged(NR);
    static constexpr size_t kBytes64 =
        j_md(L) ? boys_lds_doubles(L) * sizeof(double) : rys_staged(NR) ? rys_lds_doubles(NR) * sizeof(double) : 0;
    static constexpr size_t kBytes = kBytes64 + (HAS32 ? rys32_lds_floats(NR) * sizeof(float) : 0);
    static __device__ __forceinline__ void stage(const RysTable& tab, double* s64, float* s32)
    {
        if constexpr (j_md(L))
            boys_stage_lds<L>(tab, s64);
        else if constexpr (rys_staged(NR))
            rys_stage_lds<NR>(tab, s64);
        if constexpr (HAS32) rys32_stage_lds<NR>(tab, s32);
        if constexpr (STAGED64 || HAS32) __syncthreads();
    }
};

// One ket pair's geometry at a wave-uniform index (scalar loads).
struct JKet {
    double q, c, x, y, z;
};
__device__ __forceinline__ JKet load_ket(const double* __restrict__ rec, int k)
{
    const double* g = rec + (size_t)k * kJKetDoubles;
    return {ld_const(g), ld_const(g + 1), ld_const(g + 2), ld_const(g + 3), ld_const(g + 4)};
}

// Waves per SIMD asked of the compiler (register budget 512 / waves) for the bare 1/r FP64 kernels that
// sit one to three registers above an occupancy step and reach it without spilling ((1|3) and the
// symmetric (3|0) spill when held, and measured 0.21 against 0.18 ms and no faster); 1 = no constraint.
constexpr int j_waves(int L12, int L34, int route, bool bare)
{
    if (route != kRoutePlain || !bare) return 1;
    if (L12 == 1 && (L34 == 1 || L34 == 2)) return 5;  // 97, 99 registers; step at 96
    if (L12 == 2 && L34 == 3) return 4;                // 129; step at 128
    return 1;
}

// Persistent kernel: each wave takes (64 bra pairs x ket range) tasks from a queue until it is
// empty.  The workgroup's waves share an LDS copy of the tables (JLds).  Lanes own bra pairs; the
// kets are read at wave-uniform addresses (scalar loads) one ket ahead of their use, in bound order
// (the lists are padded by one ket; behind the per-call buffers lies more of the same scratch).  Quartets with est = B12 * B34' at or above
// thresp are evaluated in FP64 (kRoutePlain), or on the mixed route (kRouteMixed) a ket step with any
// quartet at or above thredp in FP64 and the others in FP32.
template <int L12, int L34, int ROUTE, bool BARE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(j_waves(L12, L34, ROUTE, BARE)))) void j_quartets(JQuartetArgs a, const JTask* __restrict__ tasks, int ntask,
                                                  unsigned int* qctr)
{
    using Lds = JLds<L12, L34, ROUTE>;
    constexpr int H12 = nherm(L12), H34 = nherm(L34), L = L12 + L34, HL = nherm(L);
    constexpr bool MIXED = ROUTE == kRouteMixed;
    constexpr int DN = H34 <= 4 ? H34 : 1;  // ket densities loaded ahead (coulomb_call's scratch: at most 4)
    extern __shared__ double s_dyn[];
    double* s_tab64 = s_dyn;
    float* s_tab32 = reinterpret_cast<float*>(reinterpret_cast<char*>(s_dyn) + Lds::kBytes64);
    Lds::stage(a.rys, s_tab64, s_tab32);

    const int lane = threadIdx.x & 63;
    const float thresp = a.thresp;
    const float max34 = __uint_as_float(a.sc->max34_bits);
    const float thre_bra = thresp / max34;
    const double dmax = __longlong_as_double((long long)a.sc->dmax_bits);
    // evaluated quartets and wave steps with one (scalar registers)
    unsigned long long nq = 0, nq32 = 0;
    unsigned int nsteps = 0;

    for (;;) {
        const int t = (int)wave_take(qctr);
        if (t >= ntask) break;
        JTask task;
        task.bra0 = ld_const(&tasks[t].bra0);
        task.nbra = ld_const(&tasks[t].nbra);
        task.ket0 = ld_const(&tasks[t].ket0);
        task.ket1 = ld_const(&tasks[t].ket1);
        // largest bra bound of the tile (sorted, descending): its first pair
        const float B12max = ld_const(a.bra_b + task.bra0);
        if (!(B12max >= thre_bra)) continue;  // no bra of the tile survives truncation
        const int bra = task.bra0 + lane;
        const bool active = lane < task.nbra;
        float B12 = 0.0f;
        double p12 = 1.0, c12 = 0.0, Px = 0.0, Py = 0.0, Pz = 0.0;
        if (active) {
            B12 = a.bra_b[bra];
            p12 = a.bra_geom[bra];
            Px = a.bra_geom[a.bra_n + bra];
            Py = a.bra_geom[2 * a.bra_n + bra];
            Pz = a.bra_geom[3 * a.bra_n + bra];
            c12 = a.bra_geom[4 * a.bra_n + bra];
            if constexpr (BARE) c12 *= a.ew.alpha[0];
        }
        const bool bra_ok = active && (B12 >= thre_bra);
        if (!bra_ok) B12 = __builtin_nanf("");  // no estimate of the lane passes
        double jp[H12];
#pragma unroll
        for (int u = 0; u < H12; u++) jp[u] = 0.0;

        // Early exit: B34' <= float(dmax * B34) and the static ket bounds are sorted, so no ket with
        // static bound below kstop = thresp / (B12max dmax) (1 - 2^-21) can pass with a bra of the
        // tile; the test compares bit patterns (non-negative floats) on the scalar unit.
        const float kstop = (float)((double)thresp / ((double)B12max * dmax)) * (1.0f - 4.0f * 1.1920929e-7f);
        const unsigned int kstop_bits = __builtin_amdgcn_readfirstlane(__float_as_uint(kstop));
        float bsn = ld_const(a.ket_static_b + task.ket0), kbn = ld_const(a.ket_b + task.ket0);
        JKet kn = load_ket(a.ket_rec, task.ket0);
        double dn[DN];
        const double* __restrict__ kd = a.ket_d + (size_t)(task.ket0 - a.ket_hstart) * H34;
#pragma unroll
        for (int u = 0; u < DN; u++) dn[u] = ld_const(kd + u);
        for (int k = task.ket0; k < task.ket1; k++) {
            const float bs = bsn, kb = kbn;
            if (__float_as_uint(bs) < kstop_bits) break;
            const JKet ket = kn;
            double d0[DN];
#pragma unroll
            for (int u = 0; u < DN; u++) d0[u] = dn[u];
            bsn = ld_const(a.ket_static_b + k + 1);
            kbn = ld_const(a.ket_b + k + 1);
            kn = load_ket(a.ket_rec, k + 1);
            const size_t dofs = (size_t)(k - a.ket_hstart) * H34;
#pragma unroll
            for (int u = 0; u < DN; u++) dn[u] = ld_const(a.ket_d + dofs + H34 + u);
            const float est = B12 * kb;
            const bool take = est >= thresp;
            const unsigned long long m = __ballot(take);
            if (m == 0ull) continue;
            nsteps++;
            nq += __popcll(m);
            const bool step32 = MIXED && __ballot(take && est >= a.thredp) == 0ull;
            if (MIXED && step32) nq32 += __popcll(m);
            if (!take) continue;
            const double X = Px - ket.x, Y = Py - ket.y, Z = Pz - ket.z;
            // one quartet in the arithmetic of `acc`'s element type, with the ket density of that
            // precision and the matching table
            auto contract = [&](auto& acc, const auto* dsrc, const void* tab) __attribute__((always_inline)) {
                using Real = typename std::remove_reference<decltype(acc[0])>::type;
                Real dreg[H34];
#pragma unroll
                for (int u = 0; u < H34; u++)
                    dreg[u] = (std::is_same<Real, double>::value && DN == H34) ? (Real)d0[u] : (Real)ld_const(dsrc + dofs + u);
                if constexpr (L >= 5) {
                    hermite_contract_factorized<Real, L12, L34, BARE>(a.rys, tab, a.ew, p12, c12, ket.q, ket.c, X, Y, Z, dreg, acc);
                } else {
                    Real R[HL];
                    hermite_R<Real, L, BARE>(a.rys, tab, a.ew, p12, c12, ket.q, ket.c, X, Y, Z, R);
                    static_for<H34>([&](auto U_) {
                        constexpr int u = decltype(U_)::value;
                        constexpr int ux = herm_tx(u), uy = herm_ty(u), uz = herm_tz(u);
                        static_for<H12>([&](auto T_) {
                            constexpr int tt = decltype(T_)::value;
                            constexpr int idx = herm_index(herm_tx(tt) + ux, herm_ty(tt) + uy, herm_tz(tt) + uz);
                            acc[tt] = fma(R[idx], dreg[u], acc[tt]);
                        });
                    });
                }
            };
            if (MIXED && step32) {
                // FP32 quartet, FP64 accumulation
                float jq[H12];
#pragma unroll
                for (int u = 0; u < H12; u++) jq[u] = 0.0f;
                contract(jq, a.ket_d32, s_tab32);
#pragma unroll
                for (int u = 0; u < H12; u++) jp[u] += (double)jq[u];
            } else {
                contract(jp, a.ket_d, s_tab64);
            }
        }
        if (bra_ok) {
            double* dst = a.jp + (size_t)(bra - a.bra_hstart) * H12;
#pragma unroll
            for (int u = 0; u < H12; u++)
                if (jp[u] != 0.0) atomic_add(dst + u, jp[u]);
        }
    }
    if (a.count && lane == 0 && nq) {
        atomicAdd(&a.sc->counts[a.count_cls], nq);
        if (nq32) atomicAdd(&a.sc->counts32[a.count_cls], nq32);
        atomicAdd(&a.sc->wsteps[a.count_cls], (unsigned long long)nsteps);
        atomicAdd(&a.sc->wlanes[a.count_cls], nq);
    }
}

// Symmetric J (one list on both sides): each integral (x|y) of bra group L12 and ket group
// L34 (L12 >= L34; y < x by Hermite position within one group) is evaluated once and used twice,
// as the reference's two quartets:
//   A. J_x += (x|y) d_y  when x passes the bra truncation and float(B_x B'_y) >= thresp;
//   B. J_y += (y|x) d_x  when y passes the bra truncation and float(B_y B'_x) >= thresp
//      (not for y = x, where it is A again),
// B' being the truncated (D-weighted) bounds.  Lanes own bra pairs x as in j_quartets; the B
// contributions of a ket step are summed over the wave and added to J_y by one lane.  ROUTE
// kRoutePlain: FP64; kRouteMixed: a ket step in which no lane's estimate reaches thredp, in either
// use, is evaluated in FP32 (table, R, contraction; FP64 accumulation), the others in FP64.
template <int L12, int L34, int ROUTE, bool BARE>
__global__ __launch_bounds__(256) void j_quartets_sym(JQuartetArgs a, const JTask* __restrict__ tasks, int ntask,
                                                      unsigned int* qctr)
{
    using Lds = JLds<L12, L34, ROUTE>;
    constexpr bool MIXED = ROUTE == kRouteMixed;
    constexpr int H12 = nherm(L12), H34 = nherm(L34), L = L12 + L34, HL = nherm(L);
    constexpr bool SAME = L12 == L34;
    extern __shared__ double s_dyn[];
    double* s_tab64 = s_dyn;
    float* s_tab32 = reinterpret_cast<float*>(reinterpret_cast<char*>(s_dyn) + Lds::kBytes64);
    Lds::stage(a.rys, s_tab64, s_tab32);
    const int lane = threadIdx.x & 63;
    const float thre_lo = a.thresp;
    const float max34 = __uint_as_float(a.sc->max34_bits);
    const float thre_bra = a.thresp / max34;
    const double dmax = __longlong_as_double((long long)a.sc->dmax_bits);
    // evaluated quartets of each use, integrals (one serves both uses), wave steps (scalar registers)
    unsigned long long nqa = 0, nqb = 0, nq32a = 0, nq32b = 0, nlanes = 0;
    unsigned int nsteps = 0;

    for (;;) {
        const int t = (int)wave_take(qctr);
        if (t >= ntask) break;
        JTask task;
        task.bra0 = ld_const(&tasks[t].bra0);
        task.nbra = ld_const(&tasks[t].nbra);
        task.ket0 = ld_const(&tasks[t].ket0);
        task.ket1 = ld_const(&tasks[t].ket1);
        const float B12max = ld_const(a.bra_b + task.bra0);
        const int x = task.bra0 + lane;
        const bool active = lane < task.nbra;
        float Bx = 0.0f, kbx = -1.0f;
        double p12 = 1.0, c12 = 0.0, Px = 0.0, Py = 0.0, Pz = 0.0;
        double dx[H12];
#pragma unroll
        for (int u = 0; u < H12; u++) dx[u] = 0.0;
        if (active) {
            Bx = a.bra_b[x];
            kbx = a.ket_b[x];
            p12 = a.bra_geom[x];
            Px = a.bra_geom[a.bra_n + x];
            Py = a.bra_geom[2 * a.bra_n + x];
            Pz = a.bra_geom[3 * a.bra_n + x];
            c12 = a.bra_geom[4 * a.bra_n + x];
            if constexpr (BARE) c12 *= a.ew.alpha[0];
#pragma unroll
            for (int u = 0; u < H12; u++) dx[u] = a.bra_d[(size_t)(x - a.bra_hstart) * H12 + u];
        }
        const bool bra_ok = active && (Bx >= thre_bra);
        if (!bra_ok) Bx = __builtin_nanf("");    // no estimate of the lane passes in the first use,
        if (!active) kbx = __builtin_nanf("");  // or in the second
        double jp[H12];
#pragma unroll
        for (int u = 0; u < H12; u++) jp[u] = 0.0;

        // As in j_quartets, no ket with static bound below kstop passes with any bra of the tile,
        // in either use: B'_x <= float(dmax B_x) too (margin 2^-20 for the two roundings).
        const float kstop = (float)((double)thre_lo / ((double)B12max * dmax)) * (1.0f - 8.0f * 1.1920929e-7f);
        const unsigned int kstop_bits = __builtin_amdgcn_readfirstlane(__float_as_uint(kstop));
        float bsn = ld_const(a.ket_static_b + task.ket0), kbn = ld_const(a.ket_b + task.ket0);
        JKet kn = load_ket(a.ket_rec, task.ket0);
        for (int k = task.ket0; k < task.ket1; k++) {
            const float By = bsn, kby = kbn;
            if (__float_as_uint(By) < kstop_bits) break;
            const JKet ket = kn;
            const size_t dofs = (size_t)(k - a.ket_hstart) * H34;
            double dy[H34];
#pragma unroll
            for (int u = 0; u < H34; u++) dy[u] = ld_const(a.ket_d + dofs + u);
            bsn = ld_const(a.ket_static_b + k + 1);
            kbn = ld_const(a.ket_b + k + 1);
            kn = load_ket(a.ket_rec, k + 1);
            const float ea = Bx * kby, eb = By * kbx;
            const bool takeA = (!SAME || k <= x) && ea >= thre_lo;
            const bool takeB = (By >= thre_bra) && (!SAME || k < x) && eb >= thre_lo;
            const unsigned long long mA = __ballot(takeA), mB = __ballot(takeB);
            if ((mA | mB) == 0ull) continue;
            nsteps++;
            nqa += __popcll(mA);
            nqb += __popcll(mB);
            nlanes += __popcll(mA | mB);
            bool step32 = false;
            if constexpr (MIXED) {
                step32 = __ballot((takeA && ea >= a.thredp) || (takeB && eb >= a.thredp)) == 0ull;
                if (step32) {
                    nq32a += __popcll(mA);
                    nq32b += __popcll(mB);
                }
            }
            const double X = Px - ket.x, Y = Py - ket.y, Z = Pz - ket.z;
            double jy[H34];
#pragma unroll
            for (int u = 0; u < H34; u++) jy[u] = 0.0;
            if (takeA || takeB) {
                // one integral in the arithmetic Real, both uses; the A part lands in accA
                auto both = [&](auto* R, auto* accA, const void* tab) __attribute__((always_inline)) {
                    using Real = typename std::remove_reference<decltype(R[0])>::type;
                    hermite_R<Real, L, BARE>(a.rys, tab, a.ew, p12, c12, ket.q, ket.c, X, Y, Z,
                                       *reinterpret_cast<Real(*)[HL]>(R));
                    const Real wa = takeA ? Real(1) : Real(0), wb = takeB ? Real(1) : Real(0);
                    static_for<H34>([&](auto U_) {
                        constexpr int u = decltype(U_)::value;
                        constexpr int ux = herm_tx(u), uy = herm_ty(u), uz = herm_tz(u);
                        const Real du = wa * (Real)dy[u];
                        Real s = Real(0);
                        static_for<H12>([&](auto T_) {
                            constexpr int tt = decltype(T_)::value;
                            constexpr int idx = herm_index(herm_tx(tt) + ux, herm_ty(tt) + uy, herm_tz(tt) + uz);
                            accA[tt] = fma(R[idx], du, accA[tt]);
                            // (y|x) at Q - P = -(P - Q): R_{t+u}(-X) = (-1)^{|t|+|u|} R_{t+u}(X)
                            if constexpr (((herm_tx(tt) + herm_ty(tt) + herm_tz(tt) + ux + uy + uz) & 1) != 0)
                                s = fma(-R[idx], (Real)dx[tt], s);
                            else
                                s = fma(R[idx], (Real)dx[tt], s);
                        });
                        jy[u] = (double)(wb * s);
                    });
                };
                if (MIXED && step32) {
                    float R[HL], ja[H12];
#pragma unroll
                    for (int u = 0; u < H12; u++) ja[u] = 0.0f;
                    both(R, ja, s_tab32);
#pragma unroll
                    for (int u = 0; u < H12; u++) jp[u] += (double)ja[u];
                } else {
                    double R[HL];
                    both(R, jp, s_tab64);
                }
            }
            if (mB != 0ull) {
                // sum of the B contributions over the wave (all lanes active here: the ket loop
                // and this test are wave-uniform); lane 63 adds them to J_y
#pragma unroll
                for (int u = 0; u < H34; u++) jy[u] = wave_sum_last(jy[u]);
                if (lane == 63) {
                    double* dst = a.jq + dofs;
#pragma unroll
                    for (int u = 0; u < H34; u++)
                        if (jy[u] != 0.0) atomic_add(dst + u, jy[u]);
                }
            }
        }
        if (bra_ok) {
            double* dst = a.jp + (size_t)(x - a.bra_hstart) * H12;
#pragma unroll
            for (int u = 0; u < H12; u++)
                if (jp[u] != 0.0) atomic_add(dst + u, jp[u]);
        }
    }
    if (a.count && lane == 0) {
        if (nqa) atomicAdd(&a.sc->counts[a.count_cls], nqa);
        if (nqb) atomicAdd(&a.sc->counts[a.count_cls2], nqb);
        if (nlanes) {
            atomicAdd(&a.sc->wsteps[a.count_cls], (unsigned long long)nsteps);
            atomicAdd(&a.sc->wlanes[a.count_cls], nlanes);
        }
        if (nq32a) atomicAdd(&a.sc->counts32[a.count_cls], nq32a);
        if (nq32b) atomicAdd(&a.sc->counts32[a.count_cls2], nq32b);
    }
}

template <int L12, int L34, int ROUTE>
void launch_jq(const JQuartetArgs& a, const JTask* tasks, int ntask, unsigned int* qctr, hipStream_t s)
{
    // one bare 1/r term (the common case) has kernels without the operator-term loop
    auto* kernel = a.ew.plain ? j_quartets<L12, L34, ROUTE, true> : j_quartets<L12, L34, ROUTE, false>;
    const size_t lds = JLds<L12, L34, ROUTE>::kBytes;
    const int grid = persistent_grid((const void*)kernel, 256, lds, ((long long)ntask + 3) / 4);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), lds, s, a, tasks, ntask, qctr);
}

// All ket orders of one bra order: both routes, or the FP64 route only (order 5: gradients).
template <int L12>
void launch_j_l12(int L34, int route, const JQuartetArgs& a, const JTask* tasks, int ntask, unsigned int* qctr,
                  hipStream_t s)
{
#define CASE(Y)                                                                        \
    if (L34 == Y) {                                                                    \
        if constexpr (L12 <= 2 * kMaxL)                                                \
            if (route == kRouteMixed) return launch_jq<L12, Y, kRouteMixed>(a, tasks, ntask, qctr, s); \
        return launch_jq<L12, Y, kRoutePlain>(a, tasks, ntask, qctr, s);              \
    }
    CASE(0) CASE(1) CASE(2) CASE(3) CASE(4)
#undef CASE
}

}  // namespace lsjk
