// Exchange (K) build: small helper kernels (D block maxima, fills, copies) and the class
// dispatcher; the quartet kernels are in exchange_impl.hpp (instantiated by exchange_k<L1><L2>.hip and exchange_kt<L1><L2>.hip).
#include "internal.hpp"
#include "kernels.hpp"

namespace lsjk {

template <int L1, int L2, bool BARE>
void launch_k_ket_l12(int L3, int L4, int route, const KArgs& a, const KGroups& kg, const KUnitG* units, int nunits,
                      hipStream_t s);
#define LSJK_KET_EXTERN(X, Y)                                                                                \
    extern template void launch_k_ket_l12<X, Y, true>(int, int, int, const KArgs&, const KGroups&, const KUnitG*, \
                                                      int, hipStream_t);                                     \
    extern template void launch_k_ket_l12<X, Y, false>(int, int, int, const KArgs&, const KGroups&, const KUnitG*, \
                                                       int, hipStream_t);
LSJK_KET_EXTERN(0, 0) LSJK_KET_EXTERN(0, 1) LSJK_KET_EXTERN(0, 2)
LSJK_KET_EXTERN(1, 0) LSJK_KET_EXTERN(1, 1) LSJK_KET_EXTERN(1, 2)
LSJK_KET_EXTERN(2, 0) LSJK_KET_EXTERN(2, 1) LSJK_KET_EXTERN(2, 2)
#undef LSJK_KET_EXTERN

template <int L1, int L2>
void launch_k_grad_l12(int L3, int L4, const KGradArgs& a, hipStream_t s);
#define LSJK_GRAD_EXTERN(X, Y) extern template void launch_k_grad_l12<X, Y>(int, int, const KGradArgs&, hipStream_t);
LSJK_GRAD_EXTERN(0, 0) LSJK_GRAD_EXTERN(1, 0) LSJK_GRAD_EXTERN(1, 1)
LSJK_GRAD_EXTERN(2, 0) LSJK_GRAD_EXTERN(2, 1) LSJK_GRAD_EXTERN(2, 2)
#undef LSJK_GRAD_EXTERN

// Block maxima of |D24| per (block2, block4), Dsh[i2 * ldDsh + i4], and the global maximum.
// Dense: every (i2, i4), thread per pair.  Banded (blo != nullptr, a batch basis of independent
// molecules): only the pairs of one molecule, i4 in [blo[i2], bhi[i2]); thread (i2, j) takes
// i4 = blo[i2] + j, j < band (the largest molecule's block count).
__global__ void k_blockmax(const double* D, int ldD, const int* bc2, const int* bL2, int nb2, const int* bc4,
                           const int* bL4, int nb4, double* Dsh, int ldDsh, const int* blo, const int* bhi, int band,
                           CallScalars* sc)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int w = blo ? band : nb4;
    if (i >= (long long)nb2 * w) return;
    const int i2 = (int)(i / w);
    int i4 = (int)(i - (long long)i2 * w);
    if (blo) {
        i4 += blo[i2];
        if (i4 >= bhi[i2]) return;
    }
    const int o2 = bc2[i2], o4 = bc4[i4];
    const int n2 = ncart(bL2[i2]), n4 = ncart(bL4[i4]);
    double m = 0.0;
    for (int b = 0; b < n2; b++)
        for (int d = 0; d < n4; d++) m = fmax(m, fabs(D[(size_t)(o2 + b) * ldD + (o4 + d)]));
    Dsh[(size_t)i2 * ldDsh + i4] = m;
    atomicMax(&sc->dmax_bits, (unsigned long long)__double_as_longlong(m));
}

// One workgroup per (row, partner L) key, threads over the ket blocks (coalesced rows of the block
// maxima).  Bound by L2 reads of the maxima, 8 bytes per (partner, block).
__global__ __launch_bounds__(256) void k_rowmax(const int* __restrict__ row_start, int maxLp,
                                                const int4* __restrict__ ebk,
                                                const double* __restrict__ Dsh, int ldDsh, int ncol,
                                                const int* __restrict__ rwlo, const int* __restrict__ rwhi,
                                                float thresp, float maxb34, const CallScalars* __restrict__ sc,
                                                unsigned int* __restrict__ rw, int ldrw)
{
    const int key = blockIdx.x;
    const int a0 = ld_const(row_start + key);
    const int a1 = ld_const(row_start + key + 1);
    if (a0 == a1) return;
    const int row = key / (maxLp + 1);
    const int lo = rwlo ? ld_const(rwlo + row) : 0, hi = rwhi ? ld_const(rwhi + row) : ncol;
    const double dmax = __longlong_as_double((long long)sc->dmax_bits);
    const float thre12 = (float)((double)thresp / ((double)maxb34 * dmax));
    // the partners that count: sorted, so a prefix
    int n = a1 - a0;
    if (__int_as_float(ld_const(&ebk[a1 - 1].x)) < thre12) {
        int l = 0;
        while (l < n) {
            const int mid = (l + n) / 2;
            if (__int_as_float(ld_const(&ebk[a0 + mid].x)) < thre12)
                n = mid;
            else
                l = mid + 1;
        }
        n = l;
    }
    for (int c = lo + (int)threadIdx.x; c < hi; c += 256) {
        double w = 0.0, d = 0.0;
        // eight partners' loads in flight (the last one again past the end)
        for (int k = 0; k < n; k += 8) {
            double v[8];
            float b[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int e = a0 + min(k + q, n - 1);
                b[q] = __int_as_float(ld_const(&ebk[e].x));
                v[q] = Dsh[(size_t)ld_const(&ebk[e].y) * ldDsh + c];
            }
#pragma unroll
            for (int q = 0; q < 8; q++) {
                w = fmax(w, (double)b[q] * v[q]);
                d = fmax(d, v[q]);
            }
        }
        // upper halves, rounded up (values are finite or infinite and non-negative)
        auto up16 = [](double v) { return (unsigned int)min((__float_as_uint(__double2float_ru(v)) + 0xffffu) >> 16, 0x7f80u); };
        rw[(size_t)key * ldrw + (c - lo)] = up16(w) << 16 | up16(d);
    }
}

void launch_k_rowmax(const int* row_start, int nrow, int maxLp, const int4* ebk, const double* Dsh, int ldDsh, int ncol,
                     const int* rwlo, const int* rwhi, float thresp, float maxb34,
                     const CallScalars* sc, unsigned int* rw, int ldrw, hipStream_t s)
{
    const long long keys = (long long)nrow * (maxLp + 1);
    if (keys == 0 || ncol == 0) return;
    hipLaunchKernelGGL(k_rowmax, dim3((unsigned)keys), dim3(256), 0, s, row_start, maxLp, ebk, Dsh, ldDsh, ncol,
                       rwlo, rwhi, thresp, maxb34, sc, rw, ldrw);
}

// The K view of D24 in one pass: per (block2, block4) the block's values and its maximum, at the two
// blocks' places in the K view order (kc, kb: null for a basis that keeps its order), and the global
// maximum.  One thread per block pair: D is read once, coalesced along the ket blocks.
__global__ __launch_bounds__(256) void k_kview(KViewArgs a)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)a.nb2 * a.nb4) return;
    const int i2 = (int)(t / a.nb4), i4 = (int)(t - (long long)i2 * a.nb4);
    const int o2 = a.bc2[i2], o4 = a.bc4[i4], n2 = ncart(a.bL2[i2]), n4 = ncart(a.bL4[i4]);
    const int k2 = a.kc2 ? a.kc2[o2] : o2, k4 = a.kc4 ? a.kc4[o4] : o4;  // a block's functions stay together
    double m = 0.0;
    for (int b = 0; b < n2; b++)
        for (int d = 0; d < n4; d++) {
            const double v = a.D[(size_t)(o2 + b) * a.ld + (o4 + d)];
            a.Dk[(size_t)(k2 + b) * a.ld + (k4 + d)] = v;
            m = fmax(m, fabs(v));
        }
    a.Dshk[(size_t)(a.kb2 ? a.kb2[i2] : i2) * a.nb4 + (a.kb4 ? a.kb4[i4] : i4)] = m;
    atomicMax(&a.sc->dmax_bits, (unsigned long long)__double_as_longlong(m));
}

void launch_k_kview(const KViewArgs& a, hipStream_t s)
{
    const long long n = (long long)a.nb2 * a.nb4;
    if (n == 0) return;
    hipLaunchKernelGGL(k_kview, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
}

// n words and the ntail (at most 3) bytes behind them.
__global__ void fill_zero(unsigned int* p, size_t n, int ntail)
{
    const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t i = i0; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0u;
    if (i0 < (size_t)ntail) reinterpret_cast<unsigned char*>(p + n)[i0] = 0;
}

void launch_fill(void* p, size_t bytes, hipStream_t s)
{
    if (bytes == 0) return;
    const size_t n = bytes / 4;
    int blocks = (int)std::max<size_t>(1, std::min<size_t>((n + 255) / 256, 4096));
    hipLaunchKernelGGL(fill_zero, dim3(blocks), dim3(256), 0, s, (unsigned int*)p, n, (int)(bytes % 4));
}

// Plain copy, 16 bytes per lane per step (grid-stride); the tail below 16 bytes byte-wise.
__global__ void copy_bytes(uint4* __restrict__ dst, const uint4* __restrict__ src, size_t n16, unsigned char* dtail,
                           const unsigned char* stail, int ntail)
{
    const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t i = i0; i < n16; i += (size_t)gridDim.x * blockDim.x) dst[i] = src[i];
    if (i0 < (size_t)ntail) dtail[i0] = stail[i0];
}

void launch_copy(void* dst, const void* src, size_t bytes, hipStream_t s)
{
    if (bytes == 0) return;
    const size_t n16 = bytes / 16;
    const int ntail = (int)(bytes % 16);
    int blocks = (int)std::max<size_t>(1, std::min<size_t>((n16 + 255) / 256, 8192));
    hipLaunchKernelGGL(copy_bytes, dim3(blocks), dim3(256), 0, s, (uint4*)dst, (const uint4*)src, n16,
                       (unsigned char*)dst + n16 * 16, (const unsigned char*)src + n16 * 16, ntail);
}

void launch_k_blockmax(const double* D, int ldD, const int* bc2, const int* bL2, int nb2, const int* bc4,
                       const int* bL4, int nb4, double* Dsh, int ldDsh, const int* blo, const int* bhi, int band,
                       CallScalars* sc, hipStream_t s)
{
    long long n = (long long)nb2 * (blo ? band : nb4);
    if (n == 0) return;
    hipLaunchKernelGGL(k_blockmax, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, D, ldD, bc2, bL2, nb2, bc4,
                       bL4, nb4, Dsh, ldDsh, blo, bhi, band, sc);
}

__global__ __launch_bounds__(256) void k_grad_prep(KGradPrepArgs a)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double m = 0.0, m13 = 0.0, a13 = 0.0, a24 = 0.0;
    if (t < (long long)a.nblk * a.nblk) {
        const int bi = (int)(t / a.nblk), bj = (int)(t - (long long)bi * a.nblk);
        const int oi = a.blk_cart[bi], oj = a.blk_cart[bj], ni = ncart(a.blk_L[bi]), nj = ncart(a.blk_L[bj]);
        for (int i = oi; i < oi + ni; i++)
            for (int j = oj; j < oj + nj; j++) {
                const size_t ij = (size_t)i * a.n + j, ji = (size_t)j * a.n + i;
                const double u = a.D13[ij], v = a.D13[ji], x = a.D24[ij], y = a.D24[ji];
                a.S13[ij] = 0.5 * (u + v);
                a.A13[ij] = 0.5 * (u - v);
                a.S24[ij] = 0.5 * (x + y);
                a.A24[ij] = 0.5 * (x - y);
                m13 = fmax(m13, fmax(fabs(u), fabs(v)));
                a13 = fmax(a13, fabs(a.A13[ij]));
                a24 = fmax(a24, fabs(a.A24[ij]));
                m = fmax(m, fmax(fabs(x), fabs(y)));
            }
        a.Dsh[t] = m;
    }
    // one atomic per wave and maximum: all waves share the addresses
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        m = fmax(m, __shfl_xor(m, o));
        m13 = fmax(m13, __shfl_xor(m13, o));
        a13 = fmax(a13, __shfl_xor(a13, o));
        a24 = fmax(a24, __shfl_xor(a24, o));
    }
    if ((threadIdx.x & 63) == 0) {
        const double top[4] = {m13, a13, m, a24};
#pragma unroll
        for (int k = 0; k < 4; k++) atomicMax(a.maxima + k, (unsigned long long)__double_as_longlong(top[k]));
        atomicMax(&a.sc->dmax_bits, (unsigned long long)__double_as_longlong(m));
    }
}

void launch_k_grad_prep(const KGradPrepArgs& a, hipStream_t s)
{
    const long long n = (long long)a.nblk * a.nblk;
    if (n == 0) return;
    hipLaunchKernelGGL(k_grad_prep, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
}

// Atoms are few and pairs many, so each workgroup sums in LDS first (one global atomic per atom and
// axis) while the atoms fit kGradAtomsLds; above that the additions spread over enough addresses.
constexpr int kGradAtomsLds = 1024;
__global__ __launch_bounds__(256) void k_grad_atoms(const double* __restrict__ gp, const int2* __restrict__ prim,
                                                    const int* __restrict__ atom, int npair, int natom,
                                                    double* __restrict__ G)
{
    extern __shared__ double s_g[];
    const bool lds = natom <= kGradAtomsLds;
    if (lds) {
        for (int i = threadIdx.x; i < 3 * natom; i += blockDim.x) s_g[i] = 0.0;
        __syncthreads();
    }
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < npair; i += gridDim.x * blockDim.x) {
        const int2 pr = prim[i];
        const int2 at = make_int2(atom[pr.x], atom[pr.y]);
        for (int d = 0; d < 3; d++) {
            const double a = gp[(size_t)6 * i + d], b = gp[(size_t)6 * i + 3 + d];
            if (lds) {
                atomicAdd(&s_g[3 * at.x + d], a);
                atomicAdd(&s_g[3 * at.y + d], b);
            } else {
                atomic_add(G + 3 * (size_t)at.x + d, a);
                atomic_add(G + 3 * (size_t)at.y + d, b);
            }
        }
    }
    if (lds) {
        __syncthreads();
        for (int i = threadIdx.x; i < 3 * natom; i += blockDim.x)
            if (s_g[i] != 0.0) atomic_add(G + i, s_g[i]);
    }
}

void launch_k_grad_atoms(const double* gp, const int2* prim, const int* atom, int npair, int natom, double* G,
                         hipStream_t s)
{
    if (npair <= 0) return;
    const int grid = std::min((npair + 255) / 256, 256);
    const size_t lds = natom <= kGradAtomsLds ? (size_t)3 * natom * sizeof(double) : 0;
    hipLaunchKernelGGL(k_grad_atoms, dim3(grid), dim3(256), lds, s, gp, prim, atom, npair, natom, G);
}

void launch_k_grad(int L1, int L2, int L3, int L4, const KGradArgs& a, hipStream_t s)
{
    if (a.n1 <= 0 || a.n2 <= 0) return;
#define CASE(X, Y) \
    if (L1 == X && L2 == Y) return launch_k_grad_l12<X, Y>(L3, L4, a, s);
    CASE(0, 0) CASE(1, 0) CASE(1, 1) CASE(2, 0) CASE(2, 1) CASE(2, 2)
#undef CASE
}

void launch_k_ket(int L1, int L2, int L3, int L4, int route, const KArgs& a, const KGroups& kg, const KUnitG* units,
                  int nunits, hipStream_t s)
{
    if (nunits <= 0) return;
#define CASE(X, Y) \
    if (L1 == X && L2 == Y) {                                                                                \
        if (a.ew.plain) return launch_k_ket_l12<X, Y, true>(L3, L4, route, a, kg, units, nunits, s);         \
        return launch_k_ket_l12<X, Y, false>(L3, L4, route, a, kg, units, nunits, s);                        \
    }
    CASE(0, 0) CASE(0, 1) CASE(0, 2) CASE(1, 0) CASE(1, 1) CASE(1, 2) CASE(2, 0) CASE(2, 1) CASE(2, 2)
#undef CASE
}

}  // namespace lsjk
