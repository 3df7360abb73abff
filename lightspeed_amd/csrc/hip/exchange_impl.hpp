// Exchange (K) quartet kernel templates, shared by the translation units that instantiate them
// (exchange_k<L1><L2>.hip for one bare 1/r term and exchange_kt<L1><L2>.hip for any terms: one per bra
// row and partner angular momentum, so the 324 instantiations compile in parallel, and a process
// loads the code of the operators it uses: a unit's code goes to the device at the first launch
// from it, about 2.8 ms per MB.  The first exchange call of a process with one term, s to d
// functions, took 24.5 ms with both in one unit).
// Direct exchange (K) build on gfx950.
//
// K13 += sum_{2,4} (12|34) D24 over the quartets the reference evaluates
// (IntBox::exchangeCPU, reference src/cpp/intbox/cpu/exchange.cpp:17-355):
//   * pairs (1,2) and (3,4) taken from the K-invert partner lists with b >= thresp/(maxb*D24max)
//     (KBlock::build21 / build_symmetric, src/cpp/core/kvec.cpp:128-232; exchange.cpp:54-71),
//   * quartet sieve float(b12*b34) * max|D24 block| >= thresp (exchange.cpp:145-152, 186).
// The reference loops pivot pairs (2,4) and scatters each quartet's (1,3) block with atomics; here a
// wave holds 64 ket pairs and walks one bra row's partners (see k_ket).  With a symmetric D24 and one
// list on both sides K = K^T halves the work, the same 2x the reference's D24symm half-sieve
// (exchange.cpp:138-139, 326-336) obtains.
//
// Integrals: Rys quadrature with the 2-D integrals built by the vertical recurrence on centres
// A and C and the horizontal transfer to B and D (Rys, Dupuis & King, J. Comput. Chem. 4, 154
// (1983)), in registers, for each root x_i = t_i^2 (attenuated as t^2 d^2 for erf operators).
#pragma once
#include "internal.hpp"
#include "kernels.hpp"

namespace lsjk {

template <typename Real, int L1, int L2, int L3, int L4>
struct Axis4 {
    Real v[L1 + 1][L2 + 1][L3 + 1][L4 + 1];
};

// 2-D Rys integrals of one axis and one root: vertical recurrence on centres A and C
// (G[n][m] = (n 0 | m 0)), then the horizontal transfers to D and B.  All loops are compile-time
// expansions, so every array index is a constant and the arrays live in registers.
template <typename Real, int L1, int L2, int L3, int L4>
__device__ __forceinline__ void rys_axis(Real g00, Real C00, Real D00, Real B10, Real B01, Real B00, Real AB, Real CD,
                                         Axis4<Real, L1, L2, L3, L4>& I)
{
    constexpr int NX = L1 + L2 + 1, MX = L3 + L4 + 1;
    Real G[NX][MX];
    G[0][0] = g00;
    if constexpr (NX > 1) G[1][0] = C00 * g00;
    static_for<(NX > 2 ? NX - 2 : 0)>([&](auto N_) {
        constexpr int n = decltype(N_)::value + 1;
        G[n + 1][0] = C00 * G[n][0] + Real(n) * B10 * G[n - 1][0];
    });
    static_for<MX - 1>([&](auto M_) {
        constexpr int m = decltype(M_)::value;
        static_for<NX>([&](auto N_) {
            constexpr int n = decltype(N_)::value;
            Real v = D00 * G[n][m];
            if constexpr (m > 0) v += Real(m) * B01 * G[n][m - 1];
            if constexpr (n > 0) v += Real(n) * B00 * G[n - 1][m];
            G[n][m + 1] = v;
        });
    });
    // ket transfer: T[n][c][d] = (n 0 | c d)
    Real T[NX][MX][L4 + 1];
    static_for<NX>([&](auto N_) {
        constexpr int n = decltype(N_)::value;
        static_for<MX>([&](auto C_) {
            constexpr int c = decltype(C_)::value;
            T[n][c][0] = G[n][c];
        });
    });
    static_for<L4>([&](auto D_) {
        constexpr int d = decltype(D_)::value;
        static_for<NX>([&](auto N_) {
            constexpr int n = decltype(N_)::value;
            static_for<MX - 1 - d>([&](auto C_) {
                constexpr int c = decltype(C_)::value;
                T[n][c][d + 1] = T[n][c + 1][d] + CD * T[n][c][d];
            });
        });
    });
    // bra transfer
    static_for<L3 + 1>([&](auto C_) {
        constexpr int c = decltype(C_)::value;
        static_for<L4 + 1>([&](auto D_) {
            constexpr int d = decltype(D_)::value;
            Real U[NX][L2 + 1];
            static_for<NX>([&](auto A_) {
                constexpr int a = decltype(A_)::value;
                U[a][0] = T[a][c][d];
            });
            static_for<L2>([&](auto B_) {
                constexpr int b = decltype(B_)::value;
                static_for<NX - 1 - b>([&](auto A_) {
                    constexpr int a = decltype(A_)::value;
                    U[a][b + 1] = U[a + 1][b] + AB * U[a][b];
                });
            });
            static_for<L1 + 1>([&](auto A_) {
                constexpr int a = decltype(A_)::value;
                static_for<L2 + 1>([&](auto B_) {
                    constexpr int b = decltype(B_)::value;
                    I.v[a][b][c][d] = U[a][b];
                });
            });
        });
    });
}

// A partner entry in the arithmetic of a route: the centre P stays FP64 on both routes (P - Q is
// formed in FP64); the other fields are Real.
template <typename Real>
struct KEnt {
    double Px, Py, Pz;
    Real p, K, PAx, PAy, PAz, ABx, ABy, ABz, i2p;  // K: Kp of the packed entry
    int cart, blk;
};

// One packed FP64 entry: a 128-byte, 16-byte aligned record (p, K, P, P - A, A - B, {cart, blk}, 1/(2p),
// K view {cart, blk}); KV: take the K view ids.
template <bool KV = false>
__device__ __forceinline__ KEnt<double> load_ent(const double* __restrict__ eg, int i)
{
    const double* g = static_cast<const double*>(__builtin_assume_aligned(eg + (size_t)i * kKEntDoubles, 16));
    KEnt<double> e;
    e.p = g[0];
    e.K = g[1];
    e.Px = g[2];
    e.Py = g[3];
    e.Pz = g[4];
    e.PAx = g[5];
    e.PAy = g[6];
    e.PAz = g[7];
    e.ABx = g[8];
    e.ABy = g[9];
    e.ABz = g[10];
    const int* ids = reinterpret_cast<const int*>(g + (KV ? 13 : 11));
    e.cart = ids[0];
    e.blk = ids[1];
    e.i2p = g[12];
    return e;
}

template <typename Real>
__device__ __forceinline__ Real kdiv(Real a, Real b)
{
    if constexpr (std::is_same<Real, float>::value)
        return __fdividef(a, b);
    else
        return a / b;
}

template <typename Real>
__device__ __forceinline__ Real krsqrt(Real x)
{
    if constexpr (std::is_same<Real, float>::value)
        return __frsqrt_rn(x);
    else
        return rsqrt_pos(x);
}

// One primitive quartet: acc[a][c] += sum_{b,d} (ab|cd) Db[b][d], evaluated in the route's
// arithmetic (Real) and added to the FP64 accumulator.  STAGED: the table block of this nrys was
// copied to LDS at s_tab (FP64 block for Real = double, FP32 block for Real = float); otherwise
// the global table is read.  KETD (L3 = 0 only): e34's P - A holds Q - D, and the ket's 2-D
// integrals (ab|0d) are recurred at D directly, as (ab|d0) with D in the place of C (the same
// integrals; no transfer from C, so C - D is not needed).  BARE: the operator is one bare 1/r term
// whose scale the caller has put into e34's Kp; otherwise the terms of ew are summed.
template <typename Real, int L1, int L2, int L3, int L4, bool STAGED, bool KETD = false, bool BARE = false>
__device__ __forceinline__ void k_quartet(const RysTable& tab, const void* s_tab, const Ewald& ew,
                                          const KEnt<Real>& e12, const KEnt<Real>& e34,
                                          const Real (&Db)[ncart(L2)][ncart(L4)], double (&acc)[ncart(L1)][ncart(L3)])
{
    constexpr int N1 = ncart(L1), N2 = ncart(L2), N3 = ncart(L3), N4 = ncart(L4);
    constexpr int NR = (L1 + L2 + L3 + L4) / 2 + 1;
    const Real p = e12.p, q = e34.p;
    const Real pq = p + q;
    const Real rpq = krsqrt(pq);
    const Real ipq = rpq * rpq;
    const Real rho = p * q * ipq;
    const double PQxd = e12.Px - e34.Px, PQyd = e12.Py - e34.Py, PQzd = e12.Pz - e34.Pz;
    const double r2 = PQxd * PQxd + PQyd * PQyd + PQzd * PQzd;
    const Real PQx = (Real)PQxd, PQy = (Real)PQyd, PQz = (Real)PQzd;
    // 2 pi^(5/2) K_AB K_CD / (p q sqrt(p + q))
    const Real base = e12.K * e34.K * rpq;
    const Real PAx = e12.PAx, PAy = e12.PAy, PAz = e12.PAz;
    const Real QCx = e34.PAx, QCy = e34.PAy, QCz = e34.PAz;
    const Real ABx = e12.ABx, ABy = e12.ABy, ABz = e12.ABz;
    const Real CDx = e34.ABx, CDy = e34.ABy, CDz = e34.ABz;
    const Real qf = q * ipq, pf = p * ipq;  // rho/p, rho/q
    const Real i2p = e12.i2p, i2q = e34.i2p;
    // FP32 quartets: the roots' sum is formed in FP32 and added to the FP64 accumulator once
    constexpr bool FP32 = std::is_same<Real, float>::value;
    Real qacc[N1][N3];
    if constexpr (FP32) {
#pragma unroll
        for (int a = 0; a < N1; a++)
#pragma unroll
            for (int c = 0; c < N3; c++) qacc[a][c] = Real(0);
    }
    // one operator term: Rys roots at T = rho d2 |PQ|^2, assembly with prefactor pref (d2: the number,
    // or the constant one for a bare term)
    auto term = [&](Real pref, auto d2_) __attribute__((always_inline)) {
        const Real d2 = (Real)d2_;
        Real x[NR], w[NR];
        if constexpr (std::is_same<Real, float>::value)
            rys_roots_f32<NR, STAGED>(STAGED ? static_cast<const float*>(s_tab) : tab.coef32 + rys_offset(NR, kRysNcoef32),
                                      (double)(rho * d2) * r2, x, w);
        else if constexpr (STAGED)
            rys_roots_lds<NR>(static_cast<const double*>(s_tab), rho * d2 * r2, x, w);
        else
            rys_roots<NR>(tab, rho * d2 * r2, x, w);
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const Real u = x[i] * d2;
            const Real B00 = Real(0.5) * u * ipq;
            const Real B10 = i2p * (Real(1) - u * qf);
            const Real B01 = i2q * (Real(1) - u * pf);
            const Real cq = u * qf, cp = u * pf;
            static_assert(!KETD || L3 == 0, "KETD: no angular momentum on C");
            using AX = std::conditional_t<KETD, Axis4<Real, L1, L2, L4, 0>, Axis4<Real, L1, L2, L3, L4>>;
            AX Ix, Iy, Iz;
            if constexpr (KETD) {
                rys_axis<Real, L1, L2, L4, 0>(pref * w[i], PAx - cq * PQx, QCx + cp * PQx, B10, B01, B00, ABx, CDx, Ix);
                rys_axis<Real, L1, L2, L4, 0>(Real(1), PAy - cq * PQy, QCy + cp * PQy, B10, B01, B00, ABy, CDy, Iy);
                rys_axis<Real, L1, L2, L4, 0>(Real(1), PAz - cq * PQz, QCz + cp * PQz, B10, B01, B00, ABz, CDz, Iz);
            } else {
                rys_axis<Real, L1, L2, L3, L4>(pref * w[i], PAx - cq * PQx, QCx + cp * PQx, B10, B01, B00, ABx, CDx, Ix);
                rys_axis<Real, L1, L2, L3, L4>(Real(1), PAy - cq * PQy, QCy + cp * PQy, B10, B01, B00, ABy, CDy, Iy);
                rys_axis<Real, L1, L2, L3, L4>(Real(1), PAz - cq * PQz, QCz + cp * PQz, B10, B01, B00, ABz, CDz, Iz);
            }
            // (a b | c d) of one axis from either layout (indices are compile-time constants)
            auto at = [](const AX& I, int a_, int b_, int c_, int d_) __attribute__((always_inline)) {
                if constexpr (KETD)
                    return I.v[a_][b_][d_][0];
                else
                    return I.v[a_][b_][c_][d_];
            };
            static_for<N1>([&](auto A_) {
                constexpr int a = decltype(A_)::value;
                constexpr int ax = cart_lx(L1, a), ay = cart_ly(L1, a), az = cart_lz(L1, a);
                static_for<N3>([&](auto C_) {
                    constexpr int c = decltype(C_)::value;
                    constexpr int cx = cart_lx(L3, c), cy = cart_ly(L3, c), cz = cart_lz(L3, c);
                    Real s = Real(0);
                    static_for<N2>([&](auto B_) {
                        constexpr int b = decltype(B_)::value;
                        constexpr int bx = cart_lx(L2, b), by = cart_ly(L2, b), bz = cart_lz(L2, b);
                        static_for<N4>([&](auto D_) {
                            constexpr int d = decltype(D_)::value;
                            constexpr int dx = cart_lx(L4, d), dy = cart_ly(L4, d), dz = cart_lz(L4, d);
                            s = fma(at(Ix, ax, bx, cx, dx) * at(Iy, ay, by, cy, dy) * at(Iz, az, bz, cz, dz), Db[b][d], s);
                        });
                    });
                    if constexpr (FP32)
                        qacc[a][c] += s;
                    else
                        acc[a][c] += s;
                });
            });
        }
    };
    if constexpr (BARE) {
        term(base, std::integral_constant<int, 1>{});
    } else {
        for (int it = 0; it < ew.n; it++) {
            const double om = ew.omega[it];
            Real d2 = Real(1);
            Real pref = (Real)ew.alpha[it] * base;
            if (__double_as_longlong(om) != __double_as_longlong(-1.0)) {  // erf-attenuated term (bit test: scalar)
                const Real o = (Real)om;
                d2 = kdiv(o * o, rho + o * o);
                pref *= sqrt(d2);
            }
            term(pref, d2);
        }
    }
    if constexpr (FP32) {
#pragma unroll
        for (int a = 0; a < N1; a++)
#pragma unroll
            for (int c = 0; c < N3; c++) acc[a][c] += (double)qacc[a][c];
    }
}

// The entry of one ket slot from the group's fields in slot order (KGroups::ent; K view ids): a wave's
// slots are mostly consecutive, so each field is a few cache lines, where a 128-byte record per lane
// is one line per lane and load.
__device__ __forceinline__ KEnt<double> load_slot(const double* __restrict__ ent, int nslot, int s)
{
    auto f = [&](int i) __attribute__((always_inline)) { return (ent + (size_t)i * nslot)[s]; };
    KEnt<double> e;
    e.p = f(0);
    e.K = f(1);
    e.Px = f(2);
    e.Py = f(3);
    e.Pz = f(4);
    e.PAx = f(5);
    e.PAy = f(6);
    e.PAz = f(7);
    e.ABx = f(8);
    e.ABy = f(9);
    e.ABz = f(10);
    e.i2p = f(11);
    e.cart = (int)__double_as_longlong(f(12));
    e.blk = 0;
    return e;
}

// One packed FP64 entry at a wave-uniform index, through scalar loads (K view ids).
__device__ __forceinline__ KEnt<double> load_ent_uniform(const double* __restrict__ eg, int i)
{
    const double* g = eg + (size_t)i * kKEntDoubles;
    KEnt<double> e;
    e.p = ld_const(g + 0);
    e.K = ld_const(g + 1);
    e.Px = ld_const(g + 2);
    e.Py = ld_const(g + 3);
    e.Pz = ld_const(g + 4);
    e.PAx = ld_const(g + 5);
    e.PAy = ld_const(g + 6);
    e.PAz = ld_const(g + 7);
    e.ABx = ld_const(g + 8);
    e.ABy = ld_const(g + 9);
    e.ABz = ld_const(g + 10);
    const int* ids = reinterpret_cast<const int*>(g + 13);
    e.cart = ld_const(ids);
    e.blk = ld_const(ids + 1);
    e.i2p = ld_const(g + 12);
    return e;
}

// One packed FP32-route entry at a wave-uniform index, through scalar loads (K view ids).
__device__ __forceinline__ KEnt<float> load_ent32_uniform(const double* __restrict__ eg32, int i)
{
    const double* g = eg32 + (size_t)i * kKEnt32Doubles;
    KEnt<float> e;
    e.Px = ld_const(g + 0);
    e.Py = ld_const(g + 1);
    e.Pz = ld_const(g + 2);
    const float* f = reinterpret_cast<const float*>(g + 3);
    e.p = ld_const(f + 0);
    e.K = ld_const(f + 1);
    e.PAx = ld_const(f + 2);
    e.PAy = ld_const(f + 3);
    e.PAz = ld_const(f + 4);
    e.ABx = ld_const(f + 5);
    e.ABy = ld_const(f + 6);
    e.ABz = ld_const(f + 7);
    e.i2p = ld_const(f + 8);
    const int* ids = reinterpret_cast<const int*>(g + 9);
    e.cart = ld_const(ids);
    e.blk = ld_const(ids + 1);
    return e;
}

// LDS of one k_ket workgroup: the staged table blocks first, FP64 (routes with FP64 quartets,
// nrys <= 3) then FP32 (routes with FP32 quartets, nrys <= 5), then kKWaves group accumulators
// (gsize x N1 x N3 doubles each, gsize = rows per ket group) and kKWaves slot queues.  The FP64 table at
// address 0 keeps a bin's coefficient offsets (0..8 nrys * 24 bytes) inside the immediate offset field of the paired LDS reads, so the table
// lookup needs one address per bin.
template <int L1, int L2, int L3, int L4, int ROUTE>
struct KKetLds {
    static constexpr int NR = (L1 + L2 + L3 + L4) / 2 + 1;
    static constexpr bool STAGED64 = rys_staged(NR);
    static constexpr bool STAGED32 = ROUTE == kRouteMixed && rys32_staged(NR);
    static constexpr int N13 = ncart(L1) * ncart(L3);  // accumulator doubles per group row
    static __host__ __device__ size_t bytes64(const RysTable& tab)
    {
        return STAGED64 ? rys_lds_doubles(NR) * sizeof(double) : 0;
    }
    // byte offset of the accumulators: after both tables, 8-byte aligned
    static __host__ __device__ size_t acc_offset(const RysTable& tab)
    {
        const size_t b = bytes64(tab) + (STAGED32 ? rys32_lds_floats(NR) * sizeof(float) : 0);
        return (b + 7) & ~(size_t)7;
    }
    static size_t bytes(const RysTable& tab, int gsize)
    {
        return acc_offset(tab) + (size_t)kKWaves * (gsize * N13 * sizeof(double) + kKQueueBytes);
    }
};

// An FP64 entry rounded to the FP32 route's arithmetic (the values of its FP32 record).
__device__ __forceinline__ KEnt<float> ent_to_f32(const KEnt<double>& e)
{
    KEnt<float> f;
    f.Px = e.Px;
    f.Py = e.Py;
    f.Pz = e.Pz;
    f.p = (float)e.p;
    f.K = (float)e.K;
    f.PAx = (float)e.PAx;
    f.PAy = (float)e.PAy;
    f.PAz = (float)e.PAz;
    f.ABx = (float)e.ABx;
    f.ABy = (float)e.ABy;
    f.ABz = (float)e.ABz;
    f.i2p = (float)e.i2p;
    f.cart = e.cart;
    f.blk = e.blk;
    return f;
}

// Waves per SIMD the compiler is asked to keep room for (register budget 512 / waves): FP64 classes
// with an operator-term loop whose register count sits just above an occupancy step are held below it
// where that costs at most a few spilled dwords and measured faster (classes that already spill, or
// spill more, ran 15-55 % slower when held).  The bare 1/r kernels need no hold ((ss|ss) 48 registers,
// (ss|sp) 78; steps at 64 and 80).  1 = no constraint.
constexpr int kket_class(int L1, int L2, int L3, int L4) { return ((L1 * 3 + L2) * 3 + L3) * 3 + L4; }
constexpr int kket_waves(int L1, int L2, int L3, int L4, int route, bool bare)
{
    if (route != kRoutePlain || bare) return 1;
    switch (kket_class(L1, L2, L3, L4)) {
    case kket_class(0, 0, 0, 0):
        return 8;
    case kket_class(0, 0, 0, 1):
    case kket_class(0, 0, 2, 0):
    case kket_class(0, 0, 1, 1):
        return 5;
    default:
        return 1;
    }
}

// The lane's number, formed anew at each use: the address arithmetic that depends on it stays inside
// the loop that uses it instead of holding registers through the bra walk.
__device__ __forceinline__ int lane_id()
{
    int z = 0;
    asm volatile("" : "+s"(z));
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, (unsigned int)z));
}

// The kernel's arguments (KArgs, then KGroups) in constant memory, through a pointer formed anew at
// each call: what only the sieve and the ends of a walk read is then loaded there, instead of
// holding scalar registers (and, once those run out, vector registers) through the bra walk.
struct KKernArgs {
    KArgs a;
    KGroups kg;
};
__device__ __forceinline__ const __attribute__((address_space(4))) KKernArgs* kernel_args()
{
    auto p = (const __attribute__((address_space(4))) KKernArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// K build over ket groups.  Each wave of the workgroup takes one unit (bra row r1, chunks of ket
// group g).  It first sieves the unit's ket slots: a slot (r3, 4) can pass with some partner 2 of r1
// only if b34 max_2(b12 max|D24 block|) >= thresp, and the maximum over r1's partners per ket block is
// formed once per call (KArgs::rw).  Slots that can are packed into a queue in LDS; 64 at a time, lane
// l holds one ket pair in registers and the wave walks r1's partners 2 in bound order (wave-uniform,
// scalar loads) down to the smallest bound with which any of the 64 can pass.  Each lane tests the
// reference's sieve float(b12 b34) max|D24 block| >= thresp for its (2, 4) and, where it passes,
// evaluates the quartet into FP64 register accumulators for (r1, r3) (reference
// exchange.cpp:145-152, 186).  Without the packing a chunk of 64 slots was walked whenever its largest
// bound passed with the largest |D| anywhere: with a density that decays over distance most chunks
// then held no quartet ((H2O)128 / 6-31G*, (ss|ss): 451 k walk steps for 39 k with a quartet in a
// sample of rows, 35 k steps packed), and in the triangle mode chunks of earlier rows were walked too.
// On the mixed route (one launch) quartets with est >= thredp are evaluated in FP64 and the others in
// FP32, except that a wave step holding any FP64 quartet evaluates all of its quartets in FP64
// (never less precision than the route asks for, and one evaluation per step).  After a walk the
// lanes add their accumulators into the wave's LDS block of the group (row position t); at the end of
// the unit the block is added to K with one atomic per element, plus the transposed block in the
// symmetric mode (K = K^T) for r3 != r1.
template <int L1, int L2, int L3, int L4, int ROUTE, bool BARE>
__global__ __launch_bounds__(64 * kKWaves) __attribute__((amdgpu_waves_per_eu(kket_waves(L1, L2, L3, L4, ROUTE, BARE)))) void k_ket(KArgs a, KGroups kg, const KUnitG* __restrict__ units, int nunits)
{
    using Lds = KKetLds<L1, L2, L3, L4, ROUTE>;
    constexpr bool SPLIT = ROUTE == kRouteMixed;  // FP64 and FP32 in one launch
    // D24 blocks of up to three values are loaded ahead and sieved themselves; larger ones are sieved
    // by their block maxima first and loaded where they pass.  The walk's gathers are what bounds the
    // light classes (the vector cache looks up one line per clock: 90-98 % of its cycles on (ss|ss) and
    // (ss|sp) with a gather of the maximum and one of the value per step).
    constexpr bool DIRECT = ncart(L2) * ncart(L4) <= 3;
    constexpr int NR = Lds::NR;
    constexpr int N1 = ncart(L1), N2 = ncart(L2), N3 = ncart(L3), N4 = ncart(L4), N13 = N1 * N3;
    extern __shared__ double s_dyn[];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double* s_tab64 = s_dyn;
    float* s_tab32 = reinterpret_cast<float*>(reinterpret_cast<char*>(s_dyn) + Lds::bytes64(a.rys));
    const int G = kg.gsize;  // rows per ket group
    const int ACC = G * N13;  // accumulator doubles per wave
    double* s_acc0 = reinterpret_cast<double*>(reinterpret_cast<char*>(s_dyn) + Lds::acc_offset(a.rys));
    double* s_acc = s_acc0 + w * ACC;
    // the wave's queue: slots and their largest b34 max|D24 block| (bits), kKQueue of each
    int* q_wave = reinterpret_cast<int*>(s_acc0 + kKWaves * ACC) + w * (2 * kKQueue);
    if constexpr (Lds::STAGED64) rys_stage_lds<NR>(a.rys, s_tab64);
    if constexpr (Lds::STAGED32) rys32_stage_lds<NR>(a.rys, s_tab32);
    for (int q = lane; q < ACC; q += 64) s_acc[q] = 0.0;
    __syncthreads();
    // no workgroup barrier after this point: the waves are independent
    const int u = blockIdx.x * kKWaves + w;
    if (u >= nunits) return;
    const int i1 = ld_const(&units[u].i1), g = ld_const(&units[u].g), rank1 = ld_const(&units[u].rank1);
    const int crange = ld_const(&units[u].crange);
    const int r1 = ld_const(a.s12.rows + i1);
    int a0 = ld_const(a.s12.row_start + r1 * (a.s12.maxLp + 1) + L2);
    int a1 = ld_const(a.s12.row_start + r1 * (a.s12.maxLp + 1) + L2 + 1);
    const int prange = ld_const(&units[u].prange);
    if (prange != 0) {  // a piece of the row's partner walk
        a0 = min(a1, a0 + (prange & 0xffff));
        if (prange >> 16) a1 = min(a1, a0 + (prange >> 16));
    }
    if (a0 >= a1) return;
    const int s0 = ld_const(kg.grp_slot + g) + 64 * (crange & 0xffff);
    const int s1 = min(ld_const(kg.grp_slot + g + 1), s0 + 64 * (crange >> 16));

    const float thresp = a.thresp;
    const double dmax = __longlong_as_double((long long)a.sc->dmax_bits);
    // learned route: the unit's certified factor tau <= 1 (est tau bounds every quartet's
    // contribution), so the thresholds scale by 1 / tau.  It holds for quartets whose Schwarz
    // product is at least tau_smin; quartets below that fail the plain test whenever
    // thresp >= tau_smin max|D|, else the factor is not applied.
    const double tau = (a.tau && (double)thresp >= (double)a.tau_smin * dmax) ? (double)ld_const(a.tau + u) : 1.0;
    const double thr = (double)thresp / tau;
    const double thredp = (double)a.thredp / tau;
    const float thre12 = (float)(thr / ((double)a.maxb34 * dmax));
    const float thre34 = (float)(thr / ((double)a.maxb12 * dmax));
    const float b12top = __int_as_float(ld_const(&a.s12.ebk[a0].x));

    // evaluated quartets of the wave and the FP32 part of them, wave steps with one (scalar registers)
    unsigned long long nq = 0, nq32 = 0;
    unsigned int nsteps = 0;
    bool any = false;
    int c0 = s0, qn = 0;  // next slot to sieve; queue length (wave-uniform)
    for (;;) {
        int s4 = 0;             // the lane's slot
        unsigned int x4 = 0u;   // its largest b34 max|D24 block| (bits; 0: none)
        bool valid = false, direct = false;
        while (qn < 64 && c0 < s1) {
            const auto* A = kernel_args();
            const float b34max = ld_const(A->kg.chunk_b + (c0 >> 6));
            // no quartet of this chunk can pass, and the later chunks of the group hold smaller bounds
            if (!(b34max >= thre34) || (double)(b12top * b34max) * dmax < thr) {
                c0 = s1;
                break;
            }
            const int4* slots = A->kg.slot;
            const int4 sl = slots[c0 + lane_id()];
            const float b34 = __int_as_float(sl.z);
            bool can = sl.x >= 0 && b34 >= thre34;
            if (rank1 >= 0) {
                const int* ranks = A->kg.grp_rank;
                can = can && ranks[g * G + sl.y] >= rank1;
            }
            // x: the largest b34 max|D24 block| of the slot
            float x;
            if (const unsigned int* rw = A->a.rw) {
                // the row's maxima over its partners
                rw += (size_t)(r1 * (A->a.s12.maxLp + 1) + L2) * A->a.ldrw;
                if (const int* lo = A->a.rwlo) rw -= ld_const(lo + r1);
                const unsigned int wd = can ? rw[sl.w] : 0u;
                // margin for the rounding of float(b12 b34) and of the products here
                can = can && (double)b34 * (double)__uint_as_float(wd & 0xffff0000u) * (1.0 + 1.0e-6) >= thr;
                x = b34 * __uint_as_float(wd << 16);
            } else {
                x = (float)((double)b34 * dmax);
            }
            const unsigned long long m = __ballot(can);
            // a full chunk, or the unit's last one with nothing queued, goes as it is
            if (qn == 0 && m != 0ull && (m == ~0ull || c0 + 64 >= s1)) {
                direct = true;
                valid = can;
                s4 = c0 + lane_id();
                x4 = can ? __float_as_uint(x) : 0u;
                c0 += 64;
                break;
            }
            if (can) {
                int* q = q_wave + qn + __builtin_amdgcn_mbcnt_hi((unsigned int)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)m, 0));
                q[0] = c0 + lane_id();
                q[kKQueue] = __float_as_int(x);
            }
            qn += __popcll(m);
            c0 += 64;
        }
        if (!direct) {
            if (qn == 0) break;
            // LDS of one wave: its reads below follow its writes above in order
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int ln = lane_id();
            valid = ln < qn;
            int* q = q_wave + ln;
            // an empty lane takes the first queued slot, so that its loads stay in range
            s4 = valid ? q[0] : q_wave[0];
            x4 = valid ? (unsigned int)q[kKQueue] : 0u;
            // the slots left over move to the front
            const int me = q[64], mx = q[kKQueue + 64];
            __builtin_amdgcn_wave_barrier();
            qn = max(qn - 64, 0);
            if (ln < qn) {
                q[0] = me;
                q[kKQueue] = mx;
            }
        }
        const auto* A = kernel_args();
        const int4* slots = A->kg.slot;
        const int4 sl = slots[s4];
        const int t4 = sl.y;
        // an empty lane's bound is not a number: no estimate of it passes
        const float b34 = valid ? __int_as_float(sl.z) : __builtin_nanf("");
        // the slot's entry, from the fields in slot order (neighbouring lanes, neighbouring addresses)
        KEnt<double> E34 = load_slot(A->kg.ent, A->kg.nslot, s4);
        // s-type C with a higher D: the quartets recur at D (k_quartet KETD), from Q - D = (Q - C) + (C - D)
        constexpr bool KETD = L3 == 0 && L4 > 0;
        if constexpr (KETD) {
            E34.PAx += E34.ABx;
            E34.PAy += E34.ABy;
            E34.PAz += E34.ABz;
        }
        if constexpr (BARE) E34.K *= A->a.ew.alpha[0];
        KEnt<float> E34f;
        if constexpr (SPLIT) E34f = ent_to_f32(E34);
        const double* __restrict__ dsh = A->a.Dsh + sl.w;
        const double* __restrict__ dcol = A->a.D + E34.cart;
        double acc[N1][N3];
#pragma unroll
        for (int i = 0; i < N1; i++)
#pragma unroll
            for (int j = 0; j < N3; j++) acc[i][j] = 0.0;
        bool hit = false;
        // Bra partners below bstop cannot pass with any of the 64 slots: float(b12 b34) max|D24 block| <
        // thr for b12 < thr / x (1 - 2^-20) with the largest x of the slots (rounding of the bound
        // product and of x), and below thre12 the partner fails the truncation.  The partners are
        // sorted, so the walk stops at the first one below bstop (compared as bit patterns: the bounds
        // are non-negative floats).
        const float xmax = __uint_as_float(wave_umax(x4));
        const float bstop = fmaxf(thre12, (float)(thr / (double)xmax) * (1.0f - 8.0f * 1.1920929e-7f));
        const unsigned int bstop_bits = __builtin_amdgcn_readfirstlane(__float_as_uint(bstop));
        // Loads run ahead of their use: a partner's bound and ids two steps (the list is padded), its D
        // block maximum (or D block) one step.
        const int4* __restrict__ ebk12 = a.s12.ebk;
        auto load_block = [&](int cart, auto& Db) __attribute__((always_inline)) {
            using Real = typename std::remove_reference<decltype(Db[0][0])>::type;
#pragma unroll
            for (int b = 0; b < N2; b++)
#pragma unroll
                for (int d = 0; d < N4; d++) Db[b][d] = (Real)dcol[(size_t)(cart + b) * a.ldD + d];
        };
        int bn = ld_const(&ebk12[a0].x), bn2 = ld_const(&ebk12[a0 + 1].x);
        int id1 = ld_const(DIRECT ? &ebk12[a0].z : &ebk12[a0].y);
        int id2 = ld_const(DIRECT ? &ebk12[a0 + 1].z : &ebk12[a0 + 1].y);
        double dnext = 0.0, Dnext[DIRECT ? N2 : 1][DIRECT ? N4 : 1];
        if constexpr (DIRECT)
            load_block(id1, Dnext);
        else
            dnext = dsh[(size_t)id1 * a.ldDsh];
        for (int k = a0; k < a1; k++) {
            const float b12 = __int_as_float(bn);
            if ((unsigned int)bn < bstop_bits) break;
            double dblk = dnext, Db[DIRECT ? N2 : 1][DIRECT ? N4 : 1];
            if constexpr (DIRECT) {
                // the block's own maximum; the block past the row's last partner may be of another
                // size: the last one is loaded again in its place
                if (k + 1 < a1) id1 = id2;
                dblk = 0.0;
#pragma unroll
                for (int b = 0; b < N2; b++)
#pragma unroll
                    for (int d = 0; d < N4; d++) {
                        Db[b][d] = Dnext[b][d];
                        dblk = (N2 * N4 == 1) ? fabs(Db[b][d]) : fmax(dblk, fabs(Db[b][d]));
                    }
                load_block(id1, Dnext);
                id2 = ld_const(&ebk12[k + 2].z);
            } else {
                dnext = dsh[(size_t)id2 * a.ldDsh];
                id2 = ld_const(&ebk12[k + 2].y);
            }
            bn = bn2;
            bn2 = ld_const(&ebk12[k + 2].x);
            const double est = (double)(b12 * b34) * dblk;
            const bool pass = est >= thr;
            const unsigned long long m = __ballot(pass);
            if (m == 0ull) continue;
            nsteps++;
            nq += __popcll(m);
            // mixed route: a wave step with any quartet at or above thredp evaluates all its
            // quartets in FP64 (at least the precision the route asks for); the other steps in FP32
            const bool step32 = SPLIT && __ballot(pass && est >= thredp) == 0ull;
            if (!SPLIT || !step32) {
                const KEnt<double> E12 = load_ent_uniform(a.s12.eg, k);
                if (pass) {
                    if constexpr (DIRECT) {
                        k_quartet<double, L1, L2, L3, L4, Lds::STAGED64, KETD, BARE>(a.rys, s_tab64, a.ew, E12, E34, Db, acc);
                    } else {
                        double Dq[N2][N4];
                        load_block(E12.cart, Dq);
                        k_quartet<double, L1, L2, L3, L4, Lds::STAGED64, KETD, BARE>(a.rys, s_tab64, a.ew, E12, E34, Dq, acc);
                    }
                }
            } else if constexpr (SPLIT) {
                nq32 += __popcll(m);
                const KEnt<float> E12f = load_ent32_uniform(a.s12.eg32, k);
                if (pass) {
                    float Dq[N2][N4];
                    if constexpr (DIRECT) {
#pragma unroll
                        for (int b = 0; b < N2; b++)
#pragma unroll
                            for (int d = 0; d < N4; d++) Dq[b][d] = (float)Db[b][d];
                    } else {
                        load_block(E12f.cart, Dq);
                    }
                    k_quartet<float, L1, L2, L3, L4, Lds::STAGED32, KETD, BARE>(a.rys, s_tab32, a.ew, E12f, E34f, Dq, acc);
                }
            }
            hit = hit || pass;
        }
        if (hit) {
#pragma unroll
            for (int i = 0; i < N1; i++)
#pragma unroll
                for (int j = 0; j < N3; j++) atomicAdd(&s_acc[t4 * N13 + i * N3 + j], acc[i][j]);
        }
        any = any || (__ballot(hit) != 0ull);
    }
    if (any) {
        // the lanes' LDS additions above are complete before any lane reads the block
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const auto* A = kernel_args();
        const int *rows3 = A->kg.grp_rows, *cart3 = A->a.s34.cart;
        double* K = A->a.K;
        const int ldK = A->a.ldK;
        const bool sym = A->a.symmetric, diag = A->a.mirror_diag;
        const int o1 = ld_const(A->a.s12.cart + r1);
        for (int q = lane_id(); q < ACC; q += 64) {
            const double v = s_acc[q];
            if (v == 0.0) continue;
            const int t = q / N13, ij = q - t * N13, i = ij / N3, j = ij - i * N3;
            const int r3 = rows3[g * G + t];
            const int o3 = cart3[r3];
            atomic_add(K + (size_t)(o1 + i) * ldK + (o3 + j), v);
            if (sym && (r1 != r3 || diag)) atomic_add(K + (size_t)(o3 + j) * ldK + (o1 + i), v);
        }
    }
    if (a.count) {
        if (lane_id() == 0 && nq) {
            atomicAdd(&a.sc->counts[kcount_index(L1, L2, L3, L4)], nq);
            if (nq32) atomicAdd(&a.sc->counts32[kcount_index(L1, L2, L3, L4)], nq32);
            atomicAdd(&a.sc->wsteps[kcount_index(L1, L2, L3, L4)], (unsigned long long)nsteps);
            atomicAdd(&a.sc->wlanes[kcount_index(L1, L2, L3, L4)], nq);
        }
    }
}

// Training data of the learned screen: for each K work unit, the largest ratio M_q / (b12 b34)
// over the unit's quartets q with Schwarz product b12 b34 >= smin, M_q = max over the Cartesian
// components of |(ab|O|cd)| (the exact Rys evaluation of k_quartet, one component pair (b, d) at a
// time against a unit D block).  The unit's quartets are those k_ket would visit without any
// density screening: the bra row's partners (its walk piece) x the unit's slots (triangle rank
// rule included).  One wave per unit.
template <int L1, int L2, int L3, int L4>
__global__ __launch_bounds__(64 * kKWaves) void k_unit_mag(KArgs a, KGroups kg, const KUnitG* __restrict__ units,
                                                           int nunits, float smin, float* __restrict__ out)
{
    constexpr int N1 = ncart(L1), N2 = ncart(L2), N3 = ncart(L3), N4 = ncart(L4);
    const int G = kg.gsize;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int u = blockIdx.x * kKWaves + w;
    if (u >= nunits) return;
    const int i1 = ld_const(&units[u].i1), g = ld_const(&units[u].g), rank1 = ld_const(&units[u].rank1);
    const int crange = ld_const(&units[u].crange);
    const int r1 = ld_const(a.s12.rows + i1);
    int a0 = ld_const(a.s12.row_start + r1 * (a.s12.maxLp + 1) + L2);
    int a1 = ld_const(a.s12.row_start + r1 * (a.s12.maxLp + 1) + L2 + 1);
    const int prange = ld_const(&units[u].prange);
    if (prange != 0) {
        a0 = min(a1, a0 + (prange & 0xffff));
        if (prange >> 16) a1 = min(a1, a0 + (prange >> 16));
    }
    const int s0 = ld_const(kg.grp_slot + g) + 64 * (crange & 0xffff);
    const int s1 = min(ld_const(kg.grp_slot + g + 1), s0 + 64 * (crange >> 16));
    float best = 0.0f;
    for (int c0 = s0; c0 < s1; c0 += 64) {
        const int4 sl = kg.slot[c0 + lane];
        const int e4 = max(sl.x, 0);
        const bool valid = sl.x >= 0 && kg.grp_rank[g * G + sl.y] >= rank1;
        const double b34 = (double)__int_as_float(sl.z);
        const KEnt<double> E34 = load_ent(a.s34.eg, e4);
        for (int k = a0; k < a1; k++) {
            const double b12 = (double)__int_as_float(ld_const(&a.s12.ebk[k].x));
            const KEnt<double> E12 = load_ent_uniform(a.s12.eg, k);
            if (valid && b12 * b34 >= (double)smin) {
                double m = 0.0;
                for (int b = 0; b < N2; b++)
                    for (int d = 0; d < N4; d++) {
                        double Db[N2][N4];
#pragma unroll
                        for (int bb = 0; bb < N2; bb++)
#pragma unroll
                            for (int dd = 0; dd < N4; dd++) Db[bb][dd] = (bb == b && dd == d) ? 1.0 : 0.0;
                        double acc[N1][N3];
#pragma unroll
                        for (int i = 0; i < N1; i++)
#pragma unroll
                            for (int j = 0; j < N3; j++) acc[i][j] = 0.0;
                        k_quartet<double, L1, L2, L3, L4, false>(a.rys, nullptr, a.ew, E12, E34, Db, acc);
#pragma unroll
                        for (int i = 0; i < N1; i++)
#pragma unroll
                            for (int j = 0; j < N3; j++) m = fmax(m, fabs(acc[i][j]));
                    }
                best = fmaxf(best, (float)(m / (b12 * b34)));
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = fmaxf(best, __shfl_xor(best, o));
    if (lane == 0) out[u] = best;
}

// Launch of one K build class with bra row and partner angular momenta L1, L2 (instantiated in
// exchange_k<L1><L2>.hip, exchange_kt<L1><L2>.hip).
template <int L1, int L2, bool BARE>
void launch_k_ket_l12(int L3, int L4, int route, const KArgs& a, const KGroups& kg, const KUnitG* units, int nunits,
                      hipStream_t s)
{
    dim3 grid((unsigned)((nunits + kKWaves - 1) / kKWaves)), block(64 * kKWaves);
#define ONE(C, D, R)                                                                                \
    {                                                                                               \
        auto* kernel = k_ket<L1, L2, C, D, R, BARE>;                                                \
        const size_t lds = KKetLds<L1, L2, C, D, R>::bytes(a.rys, kg.gsize);                        \
        if (lds > kMaxLdsPerGroup || lds != kket_lds_bytes(a.rys, L1, L2, C, D, R, kg.gsize))      \
            throw std::runtime_error("lsjk: k_ket LDS request too large or inconsistent");         \
        hipLaunchKernelGGL(kernel, grid, block, lds, s, a, kg, units, nunits);                      \
    }
#define CASE(C, D)                                                                                  \
    if (L3 == C && L4 == D) {                                                                       \
        if (route == kRouteMixed)                                                                   \
            ONE(C, D, kRouteMixed)                                                                  \
        else if (route == kRoutePlain)                                                              \
            ONE(C, D, kRoutePlain)                                                                  \
        else                                                                                        \
            throw std::runtime_error("lsjk: k_ket route not instantiated");                         \
        return;                                                                                     \
    }
    CASE(0, 0) CASE(0, 1) CASE(0, 2) CASE(1, 0) CASE(1, 1) CASE(1, 2) CASE(2, 0) CASE(2, 1) CASE(2, 2)
#undef CASE
#undef ONE
}

}  // namespace lsjk
