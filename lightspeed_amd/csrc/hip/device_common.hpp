// Shared device-side definitions for the J/K kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

namespace lsjk {

constexpr int kMaxL = 2;            // per-primitive angular momentum supported by the kernels
constexpr int kMaxHerm = 35;        // Hermite functions of a d-d pair (L = 4)
constexpr int kMaxEwald = 8;        // operator terms per call
constexpr double kPi = 3.14159265358979323846;

__host__ __device__ constexpr int ncart(int L) { return (L + 1) * (L + 2) / 2; }
__host__ __device__ constexpr int nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }

// Cartesian component k of shell L in lexical order (xx, xy, xz, yy, yz, zz ...):
// exponent of x, y, z.
__host__ __device__ constexpr int cart_lx(int L, int k)
{
    int idx = 0;
    for (int i = 0; i <= L; i++)
        for (int j = 0; j <= i; j++, idx++)
            if (idx == k) return L - i;
    return 0;
}
__host__ __device__ constexpr int cart_ly(int L, int k)
{
    int idx = 0;
    for (int i = 0; i <= L; i++)
        for (int j = 0; j <= i; j++, idx++)
            if (idx == k) return i - j;
    return 0;
}
__host__ __device__ constexpr int cart_lz(int L, int k)
{
    int idx = 0;
    for (int i = 0; i <= L; i++)
        for (int j = 0; j <= i; j++, idx++)
            if (idx == k) return j;
    return 0;
}

// Exponent of axis k (0 = x, 1 = y, 2 = z) of Cartesian component idx of shell L.
__host__ __device__ constexpr int cart_lk(int L, int idx, int k)
{
    return k == 0 ? cart_lx(L, idx) : (k == 1 ? cart_ly(L, idx) : cart_lz(L, idx));
}

// Hermite index t of total order <= L in the nested (L, lexical) order: components.
__host__ __device__ constexpr int herm_tx(int t)
{
    int idx = 0;
    for (int L = 0; L <= 12; L++)
        for (int i = 0; i <= L; i++)
            for (int j = 0; j <= i; j++, idx++)
                if (idx == t) return L - i;
    return 0;
}
__host__ __device__ constexpr int herm_ty(int t)
{
    int idx = 0;
    for (int L = 0; L <= 12; L++)
        for (int i = 0; i <= L; i++)
            for (int j = 0; j <= i; j++, idx++)
                if (idx == t) return i - j;
    return 0;
}
__host__ __device__ constexpr int herm_tz(int t)
{
    int idx = 0;
    for (int L = 0; L <= 12; L++)
        for (int i = 0; i <= L; i++)
            for (int j = 0; j <= i; j++, idx++)
                if (idx == t) return j;
    return 0;
}
// Index of Hermite tuple (tx, ty, tz) in the same order.
__host__ __device__ constexpr int herm_index(int tx, int ty, int tz)
{
    int L = tx + ty + tz;
    int base = nherm(L - 1);
    if (L == 0) base = 0;
    // within shell L: i = L - tx, j = tz
    int i = L - tx;
    int off = i * (i + 1) / 2 + tz;
    return base + off;
}

// Compile-time loop: f(std::integral_constant<int, I>) for I = 0..N-1, fully expanded, so every
// index derived from I (Hermite / Cartesian tuples, table offsets) is a constant expression.
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

#include "../common/rys_asym.inc"

// Rys table in device memory, set up by the library at init: per nrys n, root and bin the
// coefficients of x = t^2 and of the weight in v = T - b - 1/2 on [b, b + 1), FP64 at
// rys_offset(n) + bin n 2 kRysNcoef + root 2 kRysNcoef + {x|w} kRysNcoef + k, and the FP32 rule for
// the single-precision route (same bins, kRysNcoef32 coefficients per polynomial).
struct RysTable {
    const double* coef;
    const float* coef32;
    const double* boys;  // Boys tables of orders 2 .. 4 (boys_offset)
};
constexpr int kRysNcoef = 12;
// Coefficients per polynomial of the FP32 rule: a degree-5 Chebyshev interpolant of the FP64
// polynomial on each bin reaches the FP32 rounding floor (1.2e-7 relative to F0).
constexpr int kRysNcoef32 = 6;
__host__ __device__ constexpr int rys_offset(int n, int ncoef = kRysNcoef)
{
    int o = 0;
    for (int k = 1; k < n; k++) o += kRysNbin[k] * k * 2 * ncoef;
    return o;
}

// Bin b of T in [0, Tc) and v = T - b - 1/2: adding 1.5 2^52 rounds T - 1/2 to an integer in the low
// word of the sum, which is the bin (at a bin's edge either neighbour, whose polynomials both hold
// there).  Four FP64 additions, where a conversion to an integer and back takes two quarter-rate
// instructions.  The bin is clamped, so the table is never read out of bounds.
template <int NRYS>
__device__ __forceinline__ int rys_bin(double T, double& v)
{
    constexpr double kRound = 6755399441055744.0;
    const double a = T - 0.5, t = a + kRound;
    v = a - (t - kRound);
    return (int)min((unsigned int)__double2loint(t), (unsigned int)(kRysNbin[NRYS] - 1));
}

// Large-T rule: x_i = r2_i / T, w_i = W_i / sqrt(T), 1/T and T^(-1/2) from one rsqrt; the constants
// are compile-time.
template <int NRYS, typename Real>
__device__ __forceinline__ void rys_asym(double T, Real* x, Real* w)
{
    const double s = rsqrt(T);
    const double iT = s * s;
#pragma unroll
    for (int i = 0; i < NRYS; i++) {
        x[i] = (Real)(kRysAsymR2[NRYS * (NRYS - 1) / 2 + i] * iT);
        w[i] = (Real)(kRysAsymW[NRYS * (NRYS - 1) / 2 + i] * s);
    }
}

// The bin polynomials of all roots at v; c: the bin's NRYS x {x|w} x NC coefficients.
template <int NRYS, int NC, typename Real>
__device__ __forceinline__ void rys_poly(const Real* c, Real v, Real* x, Real* w)
{
#pragma unroll
    for (int i = 0; i < NRYS; i++) {
        const Real* cx = c + i * 2 * NC;
        const Real* cw = cx + NC;
        Real px = cx[NC - 1], pw = cw[NC - 1];
#pragma unroll
        for (int k = NC - 2; k >= 0; k--) {
            px = fma(px, v, cx[k]);
            pw = fma(pw, v, cw[k]);
        }
        x[i] = px;
        w[i] = pw;
    }
}

// Evaluate the nrys-root rule from the global table: x_i = t_i^2, w_i (the oracle's rys_eval evaluates
// the same rule).  A non-finite T takes the asymptotic branch (no table access).
template <int NRYS>
__device__ __forceinline__ void rys_roots(const RysTable& tab, double T, double* x, double* w)
{
    if (!(T < (double)kRysNbin[NRYS])) return rys_asym<NRYS>(T, x, w);
    double v;
    const int b = rys_bin<NRYS>(T, v);
    rys_poly<NRYS, kRysNcoef>(tab.coef + rys_offset(NRYS) + (size_t)b * NRYS * 2 * kRysNcoef, v, x, w);
}

// LDS copy of the table block of one nrys: [bin][root][x|w][12] doubles with one pad double per
// bin, so that lanes reading the same coefficient of different bins hit different LDS banks (an
// unpadded bin of 24 nrys doubles puts every bin on the same few banks).
__host__ __device__ constexpr int rys_lds_stride(int nrys) { return nrys * 2 * 12 + 1; }
__host__ __device__ constexpr size_t rys_lds_doubles(int nrys) { return (size_t)kRysNbin[nrys] * rys_lds_stride(nrys); }

// Kernels stage the table block in LDS for nrys <= 3 (at most 27.6 KB, so several workgroups
// share a CU); for more roots they read it from global memory (rys_roots).
__host__ __device__ constexpr bool rys_staged(int nrys) { return nrys <= 3; }

// Upper limit of the dynamic LDS one workgroup of these kernels requests.
constexpr size_t kMaxLdsPerGroup = 65536;

// Roots from the LDS copy when the kernel staged one, else from the global table.
template <int NRYS>
__device__ __forceinline__ void rys_roots_any(const RysTable& tab, const double* s_coef, double T, double* x,
                                              double* w);

// Cooperative copy of the nrys block of the table into LDS, bins padded to rys_lds_stride (all
// threads of the workgroup; the caller synchronises the workgroup afterwards).
template <int NRYS>
__device__ __forceinline__ void rys_stage_lds(const RysTable& tab, double* s_coef)
{
    constexpr int B = NRYS * 2 * kRysNcoef, S = rys_lds_stride(NRYS);
    constexpr int n = kRysNbin[NRYS] * B;
    const double* src = tab.coef + rys_offset(NRYS);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int b = i / B;
        s_coef[b * S + (i - b * B)] = src[i];
    }
}

// rys_roots with the coefficients of this nrys read from LDS (staged by rys_stage_lds).
template <int NRYS>
__device__ __forceinline__ void rys_roots_lds(const double* s_coef, double T, double* x, double* w)
{
    if (!(T < (double)kRysNbin[NRYS])) return rys_asym<NRYS>(T, x, w);
    double v;
    const int b = rys_bin<NRYS>(T, v);
    rys_poly<NRYS, kRysNcoef>(s_coef + __umul24(b, rys_lds_stride(NRYS)), v, x, w);
}

template <int NRYS>
__device__ __forceinline__ void rys_roots_any(const RysTable& tab, const double* s_coef, double T, double* x,
                                              double* w)
{
    if constexpr (rys_staged(NRYS))
        rys_roots_lds<NRYS>(s_coef, T, x, w);
    else
        rys_roots<NRYS>(tab, T, x, w);
}

// Boys table of order L (2 .. 4): on the Rys bins of L / 2 + 1 roots the coefficients of F_L in
// v = T - b - 1/2 (degree 11) and exp(-(b + 1/2)), 13 doubles per bin (odd: lanes in different bins
// fall on different LDS banks).
constexpr int kBoysDoubles = kRysNcoef + 1;
__host__ __device__ constexpr size_t boys_lds_doubles(int L) { return (size_t)kRysNbin[L / 2 + 1] * kBoysDoubles; }
__host__ __device__ constexpr size_t boys_offset(int L)
{
    size_t o = 0;
    for (int k = 2; k < L; k++) o += boys_lds_doubles(k);
    return o;
}
template <int L>
__device__ __forceinline__ void boys_stage_lds(const RysTable& tab, double* s)
{
    for (int i = threadIdx.x; i < (int)boys_lds_doubles(L); i += blockDim.x) s[i] = tab.boys[boys_offset(L) + i];
}

// F_0 .. F_L at T from the staged table: F_L by its polynomial, exp(-T) = exp(-(b + 1/2)) exp(-v) with
// the degree-12 Chebyshev interpolant of exp(-v) on |v| <= 1/2 (5e-18), then downward,
// F_{n-1} = (2 T F_n + exp(-T)) / (2 n - 1), which is stable.  From T = Tc on (where exp(-T) is below
// rounding) F_n = F_{n-1} (n - 1/2) / T.
template <int L>
__device__ __forceinline__ void boys_lds(const double* s, double T, double (&F)[L + 1])
{
    constexpr int NR = L / 2 + 1;
    if (!(T < (double)kRysNbin[NR])) {
        const double r = rsqrt(T), iT = r * r;
        F[0] = kRysAsymW[0] * r;
#pragma unroll
        for (int n = 1; n <= L; n++) F[n] = F[n - 1] * ((n - 0.5) * iT);
        return;
    }
    double v;
    const double* c = s + __umul24(rys_bin<NR>(T, v), kBoysDoubles);
    constexpr double kExp[13] = {1.0,
                                 -9.99999999999999889e-01,
                                 5.00000000000000000e-01,
                                 -1.66666666666680646e-01,
                                 4.16666666666676636e-02,
                                 -8.33333333288569476e-03,
                                 1.38888888885692970e-03,
                                 -1.98412704550513576e-04,
                                 2.48015877398097512e-05,
                                 -2.75569101863640885e-06,
                                 2.75570271694439541e-07,
                                 -2.51828992381847868e-08,
                                 2.09701512151694754e-09};
    double f = c[kRysNcoef - 1], e = kExp[12];
#pragma unroll
    for (int k = kRysNcoef - 2; k >= 0; k--) f = fma(f, v, c[k]);
#pragma unroll
    for (int k = 11; k >= 0; k--) e = fma(e, v, kExp[k]);
    e *= c[kRysNcoef];
    F[L] = f;
    const double T2 = T + T;
#pragma unroll
    for (int n = L; n >= 1; n--) F[n - 1] = fma(T2, F[n], e) * (1.0 / (2 * n - 1));
}

// LDS copy of the FP32 table block of one nrys: bins of nrys 2 kRysNcoef32 floats plus one pad.
__host__ __device__ constexpr int rys32_lds_stride(int nrys) { return nrys * 2 * kRysNcoef32 + 1; }

// FP32 Rys rule for the single-precision route.  T is formed in FP64 by the caller; for T >= Tc
// the asymptotic roots are formed in FP64 and rounded; otherwise the FP32 bin polynomial is read
// from `c32`: the global table (LDS = false) or an LDS copy of this nrys block with padded bins
// (LDS = true).
template <int NRYS, bool LDS>
__device__ __forceinline__ void rys_roots_f32(const float* c32, double T, float* x, float* w)
{
    if (!(T < (double)kRysNbin[NRYS])) return rys_asym<NRYS>(T, x, w);
    double v;
    const int b = rys_bin<NRYS>(T, v);
    rys_poly<NRYS, kRysNcoef32>(c32 + __umul24(b, LDS ? rys32_lds_stride(NRYS) : NRYS * 2 * kRysNcoef32), (float)v, x, w);
}

__host__ __device__ constexpr size_t rys32_lds_floats(int nrys) { return (size_t)kRysNbin[nrys] * rys32_lds_stride(nrys); }

// Kernels of the FP32 route stage the FP32 block in LDS for nrys <= 5 (at most 14.2 KB).
__host__ __device__ constexpr bool rys32_staged(int nrys) { return nrys <= 5; }

// Cooperative copy of the FP32 nrys block into LDS, bins padded to rys32_lds_stride.
template <int NRYS>
__device__ __forceinline__ void rys32_stage_lds(const RysTable& tab, float* s_coef)
{
    constexpr int B = NRYS * 2 * kRysNcoef32, S = rys32_lds_stride(NRYS);
    constexpr int n = kRysNbin[NRYS] * B;
    const float* src = tab.coef32 + rys_offset(NRYS, kRysNcoef32);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int b = i / B;
        s_coef[b * S + (i - b * B)] = src[i];
    }
}

// 1/sqrt(x) for finite x > 0 (sums of Gaussian exponents): the hardware estimate y refined by one
// second-order step, 1/sqrt(x) = y (1 - e)^(-1/2) ~ y (1 + e/2 + 3 e^2 / 8) with e = 1 - x y^2.
// These are the operations the device library's rsqrt performs, without its selection of
// special values (zero, infinity, denormals), so for such x the two agree bit for bit.
__device__ __forceinline__ double rsqrt_pos(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// Load through the constant address space: a wave-uniform address becomes a scalar (SMEM) load,
// a divergent one an ordinary vector load.  Only for data no kernel of the launch writes.
template <typename T>
__device__ __forceinline__ T ld_const(const T* p)
{
    return *(const __attribute__((address_space(4))) T*)(p);
}

// Next work item of a dynamic queue for the calling wave (lane 0 takes it; all lanes get it).
__device__ __forceinline__ unsigned int wave_take(unsigned int* ctr)
{
    unsigned int t = 0;
    if ((threadIdx.x & 63) == 0) t = atomicAdd(ctr, 1u);
    return __builtin_amdgcn_readfirstlane(__shfl(t, 0));
}

// v + (v moved across lanes by the DPP control CTRL in the rows of ROW_MASK; 0 elsewhere), the
// double moved as its two 32-bit halves
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_add(double v)
{
    const long long b = __double_as_longlong(v);
    int lo, hi;
    if constexpr (ROW_MASK == 0xf) {  // every lane written from a valid source: no initial value
        lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, ROW_MASK, 0xf, false);
        hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, ROW_MASK, 0xf, false);
    } else {
        lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROW_MASK, 0xf, false);
        hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROW_MASK, 0xf, false);
    }
    return v + __longlong_as_double((long long)(((unsigned long long)(unsigned int)hi << 32) | (unsigned int)lo));
}

// Sum of v over the 64 lanes of a wave with every lane active, complete in lane 63: DPP moves
// within 16-lane rows (swap neighbours, swap pairs, half-row mirror, row mirror: each lane then
// holds its row's sum), then row broadcasts (lane 15 into rows 1 and 3, lane 31 into rows 2 and
// 3).  No LDS traffic.
__device__ __forceinline__ double wave_sum_last(double v)
{
    v = dpp_add<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
    v = dpp_add<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
    v = dpp_add<0x141, 0xf>(v);  // row_half_mirror
    v = dpp_add<0x140, 0xf>(v);  // row_mirror
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15
    v = dpp_add<0x143, 0xc>(v);  // row_bcast:31
    return v;
}

// Largest of the 64 lanes' values (every lane active), as a wave-uniform value: the moves of
// wave_sum_last with max in place of the sum.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ unsigned int dpp_umax(unsigned int v)
{
    return max(v, (unsigned int)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROW_MASK, 0xf, false));
}
__device__ __forceinline__ unsigned int wave_umax(unsigned int v)
{
    v = dpp_umax<0xB1, 0xf>(v);
    v = dpp_umax<0x4E, 0xf>(v);
    v = dpp_umax<0x141, 0xf>(v);
    v = dpp_umax<0x140, 0xf>(v);
    v = dpp_umax<0x142, 0xa>(v);
    v = dpp_umax<0x143, 0xc>(v);
    return (unsigned int)__builtin_amdgcn_readlane((int)v, 63);
}

// McMurchie-Davidson Hermite expansion coefficients for one axis:
// E[t][i][j] for i <= LA, j <= LB, t <= i + j (Helgaker, Jorgensen & Olsen eqs. 9.5.6-9.5.7):
//   E^{i+1,j}_t = E^{ij}_{t-1}/(2p) + X_PA E^{ij}_t + (t+1) E^{ij}_{t+1}
//   E^{i,j+1}_t = E^{ij}_{t-1}/(2p) + X_PB E^{ij}_t + (t+1) E^{ij}_{t+1}
template <int LA, int LB>
struct HermE {
    double v[LA + LB + 1][LA + 1][LB + 1];
};

template <int LA, int LB>
__device__ __forceinline__ void hermite_E(double oo2p, double XPA, double XPB, HermE<LA, LB>& E)
{
#pragma unroll
    for (int t = 0; t <= LA + LB; t++)
#pragma unroll
        for (int i = 0; i <= LA; i++)
#pragma unroll
            for (int j = 0; j <= LB; j++) E.v[t][i][j] = 0.0;
    E.v[0][0][0] = 1.0;
#pragma unroll
    for (int i = 0; i < LA; i++) {
#pragma unroll
        for (int t = 0; t <= i + 1; t++) {
            double a = (t > 0) ? E.v[t - 1][i][0] * oo2p : 0.0;
            double b = (t <= i) ? XPA * E.v[t][i][0] : 0.0;
            double c = (t + 1 <= i) ? (t + 1) * E.v[t + 1][i][0] : 0.0;
            E.v[t][i + 1][0] = a + b + c;
        }
    }
#pragma unroll
    for (int i = 0; i <= LA; i++) {
#pragma unroll
        for (int j = 0; j < LB; j++) {
#pragma unroll
            for (int t = 0; t <= i + j + 1; t++) {
                double a = (t > 0) ? E.v[t - 1][i][j] * oo2p : 0.0;
                double b = (t <= i + j) ? XPB * E.v[t][i][j] : 0.0;
                double c = (t + 1 <= i + j) ? (t + 1) * E.v[t + 1][i][j] : 0.0;
                E.v[t][i][j + 1] = a + b + c;
            }
        }
    }
}

// Double-precision atomic add that maps to the hardware global FP64 atomic.
__device__ __forceinline__ void atomic_add(double* p, double v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace lsjk
