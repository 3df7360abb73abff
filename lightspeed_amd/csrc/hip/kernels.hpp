// Kernel argument blocks and launcher declarations (library-internal).
#pragma once
#include "internal.hpp"

namespace lsjk {

// Index of the quartet counters in CallScalars::counts.
__host__ __device__ constexpr int jcount_index(int L12, int L34) { return L12 * 5 + L34; }
__host__ __device__ constexpr int kcount_index(int L1, int L2, int L3, int L4)
{
    return 256 + ((L1 * 5 + L2) * 5 + L3) * 5 + L4;
}

// Precision routes of a quartet kernel launch (the reference's documented mixed precision,
// intbox.hpp:736-742: FP64 when est >= thredp, FP32 when thresp <= est < thredp, else skipped).
constexpr int kRoutePlain = 0;  // est >= thresp, FP64 (thredp <= thresp)
constexpr int kRouteMixed = 4;  // est >= thredp in FP64 and thresp <= est < thredp in FP32, one launch

struct JPrepArgs {
    const int* p1;
    const int* p2;
    const float* bound;
    const int* hpos;
    const double* K;
    const double *eA, *xA, *yA, *zA;
    const int* cartA;
    const double *eB, *xB, *yB, *zB;
    const int* cartB;
    const double* D;
    int ldD;
    int symmetric;
    float thre_ket;
    float* kb;
    double* kd;
    float* kd32;  // FP32 copy of the densities for the FP32 route (nullptr: not needed)
    CallScalars* sc;
};

constexpr int kJKetDoubles = 6;
struct JQuartetArgs {
    RysTable rys;
    Ewald ew;
    float thresp;
    int count;
    int count_cls;
    // bra (Hermite order of the bra list)
    const float* bra_b;
    const double* bra_geom;  // SoA p, Px, Py, Pz, sqrt(2 pi^(5/2))/p, stride bra_n
    int bra_n;
    int bra_hstart;
    double* jp;  // accumulators of the bra group
    // ket (Hermite order of the ket list)
    const float* ket_b;         // truncated bounds (per call)
    const float* ket_static_b;  // Schwarz bounds
    const double* ket_rec;      // kJKetDoubles per pair: p, sqrt(2 pi^(5/2))/p, P (3), 0
    int ket_hstart;
    const double* ket_d;  // Hermite densities of the ket group
    const float* ket_d32; // their FP32 copy (FP32 route)
    float thredp;
    CallScalars* sc;
    // symmetric J (one list on both sides): the bra group's Hermite densities and the ket group's
    // accumulators, for the second use of each integral (the ket pair as bra)
    const double* bra_d;
    double* jq;
    int count_cls2;
};

struct JScatterArgs {
    const int* p1;
    const int* p2;
    const float* bound;
    const int* hpos;
    const double* K;
    const double *eA, *xA, *yA, *zA;
    const int* cartA;
    const double *eB, *xB, *yB, *zB;
    const int* cartB;
    const double* jp;
    double* J;
    int ldJ;
    int symmetric;
    int screen;  // 1: only bra pairs that survive truncate_bra (J); 0: every pair (potential)
    float thresp;
    CallScalars* sc;
};

// Coulomb gradient, bra-centre part: per bra pair, dE/dA and dE/dB from the potential V_t of the
// ket density at bra Hermite order L12 + 1 and the symmetrised bra density block.
struct JGradArgs {
    const int* p1;
    const int* p2;
    const float* bound;
    const int* hpos;
    const double* K;
    const double *eA, *xA, *yA, *zA;
    const int *cartA, *atomA;
    const double *eB, *xB, *yB, *zB;
    const int *cartB, *atomB;
    const double* vp;  // V_t, Hermite order, H(L12+1) per pair of group L12
    const double* D;   // bra density (Cartesian)
    int ldD;
    int symmetric;
    float thresp;
    double* G;  // natom x 3
    CallScalars* sc;
};
void launch_j_grad_scatter(int LA, int LB, const JGradArgs& a, int k0, int nk, int hstart, size_t hoff,
                           hipStream_t s);

// One-electron integrals (overlap, kinetic, potential) of one pair list.
struct OneEArgs {
    const int* p1;
    const int* p2;
    const int* hpos;
    const double* K;
    const double *eA, *xA, *yA, *zA;
    const int* cartA;
    const double *eB, *xB, *yB, *zB;
    const int* cartB;
    int symmetric;
    double* S;  // ncart1 x ncart2 outputs (nullptr: not wanted)
    double* T;
    int ld;
    // potential: point charges and operator
    RysTable rys;
    Ewald ew;
    const double* xyzc;  // nA x 4
    int nA;
    double* vp;  // Hermite accumulators (Hermite order, same layout as the J bra buffer)
};
void launch_one_e_st(int LA, int LB, const OneEArgs& a, int k0, int nk, hipStream_t s);
// nsplit: parts the charges are cut into (more than one: the accumulators are added to).
void launch_one_e_v(int LA, int LB, const OneEArgs& a, int k0, int nk, int nsplit, int hstart, size_t hoff,
                    hipStream_t s);

// Exchange gradient (exchange_grad_impl.hpp): the lanes' pairs (class 1, n1 of them) against chunks
// of `chunk` pairs of class 2; records of kGPairDoubles doubles and bounds, both in bound order.
constexpr int kGPairDoubles = 16;
struct KGradArgs {
    RysTable rys;
    Ewald ew;
    float thresp;
    const double *g1, *g2;
    const float *b1, *b2;
    int n1, n2, chunk, nslice;
    const double *X13, *X24;  // both symmetric or both antisymmetric, ncart x ncart
    int ldx;
    const double* Dsh;  // block maxima of |D24|, the larger of the two triangles', nblk x nblk
    int nblk;
    double* gp;  // the class-1 pairs' sums, 6 doubles each (dE/dA, dE/dB)
    CallScalars* sc;
};
void launch_k_grad(int L1, int L2, int L3, int L4, const KGradArgs& a, hipStream_t s);
// How a class's components are formed.  Expanded: every component at compile time with the weight
// blocks in registers, up to (pp|pp).  Unrolled: the (c, d) components at compile time, each loading
// its weights, up to (dd|pp); they can be cut over waves.  Above that (648 and 1296
// components) the (c, d) components run as a loop, the 2-D integrals indexed at run time in scratch,
// which bounds the code.
constexpr int grad_ncomp(int L1, int L2, int L3, int L4) { return ncart(L1) * ncart(L2) * ncart(L3) * ncart(L4); }
constexpr bool grad_expanded(int L1, int L2, int L3, int L4) { return grad_ncomp(L1, L2, L3, L4) <= 81; }
constexpr bool grad_unrolled(int L1, int L2, int L3, int L4) { return grad_ncomp(L1, L2, L3, L4) <= 324; }
// Per block pair: the symmetric and antisymmetric parts of D13 and D24, the block maxima of D24
// (the larger of the two triangles'), max|D24|, and maxima[0 .. 3] = max|D13|, max|A13|, max|D24|,
// max|A24| (bits of doubles).
struct KGradPrepArgs {
    const double *D13, *D24;
    int n, nblk;
    const int *blk_cart, *blk_L;
    double *S13, *S24, *A13, *A24, *Dsh;
    unsigned long long* maxima;
    CallScalars* sc;
};
void launch_k_grad_prep(const KGradPrepArgs& a, hipStream_t s);
// G[atom] += the pairs' sums (gp: 6 doubles each; prim: {primitive A, primitive B}; atom: of a primitive).
void launch_k_grad_atoms(const double* gp, const int2* prim, const int* atom, int npair, int natom, double* G,
                         hipStream_t s);

// K build: ket groups.  The rows of one (row L, partner L) class of the ket list are put in
// spatial (Morton) order and cut into groups of kgroup_size(L, Lp) consecutive rows; the partner
// entries of a group's rows are merged, sorted by bound (descending) and padded to a multiple of
// 64 slots.  A wave holds 64 slots (one ket pair per lane) in registers and streams the bra row's
// partners through scalar loads.  Rows with few partners per row (p or d partners) leave the
// bounds of a 16-row group's chunks spread wide, so that few lanes pass the sieve together;
// larger groups narrow each chunk's bound range: 64 rows for s rows with p or d partners, 32 for
// p rows with d partners (measured up to 42 % faster), 16 otherwise (larger groups measured
// slower there: longer units, and fewer ket rows of the bra row's triangle per group).
constexpr int kgroup_size(int L, int Lp) { return (L == 0 && Lp > 0) ? 64 : ((L == 1 && Lp == 2) ? 32 : 16); }
// These are the defaults: lsjk_autotune picks 16, 32 or 64 rows per (row L, partner L) of a list
// (KGroups::gsize), where every class over that ket pair fits the LDS limit (kket_lds_bytes).
constexpr int kKWaves = 4;  // waves (independent work units) per workgroup
// k_ket's queue of ket slots that can pass the sieve: slot and largest b34 max|D24 block|; at most 63
// left over + 64 new.
constexpr int kKQueue = 128;
constexpr size_t kKQueueBytes = kKQueue * 2 * sizeof(int);
struct KGroups {
    int gsize;             // rows per group
    // [nslot] {entry index or -1 (padding), position of the row in the group, bits of the entry's
    // bound, the partner's block id in the K view order}
    const int4* slot;
    // [13][nslot] the slots' entries by field: p, Kp, P (3), P - A (3), A - B (3), 1/(2p), the partner's
    // Cartesian offset in the K view order (zeros for padding)
    const double* ent;
    int nslot;
    const int* grp_slot;   // [ngroup + 1] first slot of each group
    const int* grp_rows;   // [ngroup * group size] row primitive at each position (-1: none)
    const int* grp_rank;   // [ngroup * group size] spatial rank of that row (INT_MAX: none)
    const float* chunk_b;  // [nslot / 64] largest bound of each 64-slot chunk
};
// A K work unit: bra row rows1[i1] against the 64-slot chunks [c0, c0 + nc) of ket group g
// (crange = c0 | nc << 16, chunks counted from the group's first slot).  rank1: in the triangle
// mode (one list, symmetric D24) only ket rows of spatial rank >= rank1 (the bra row's) take
// part; -1 otherwise.  prange = p0 | np << 16: the unit walks the row's partners from p0 on, np
// of them (np = 0: to the end); 0 = the whole walk.
struct KUnitG {
    int i1, g, rank1, crange, prange;
};
// A packed partner entry (row primitive A, partner primitive B), 128 bytes: p, Kp, P (3),
// P - A (3), A - B (3), {the partner's Cartesian offset, its block id} (two ints), 1/(2p), the
// same two ids in the partner basis's K view order (Basis::h_kcart, h_kblk), 2 zero pads.
// Kp = K_AB sqrt(2 pi^(5/2)) / p with K_AB = c_A c_B exp(-a b / p |A - B|^2).
constexpr int kKEntDoubles = 16;
// sqrt(2 pi^(5/2))
constexpr double kKPrefRoot = 5.914967172795613;
// The FP32-route copy, 80 bytes: P (3 doubles), p, Kp, P - A, A - B, 1/(2p), 0 (10 floats),
// {cart, blk}, {cart, blk} in the K view order.
constexpr int kKEnt32Doubles = 10;
struct KSide {
    const int* row_start;  // [nrow * (maxLp+1) + 1]
    int maxLp;
    // per entry {bits of the bound, the partner's block id and Cartesian offset in the K view order, 0}
    const int4* ebk;
    const double* eg;      // packed entries, kKEntDoubles doubles each (see KEnt)
    const double* eg32;    // FP32-route entries, kKEnt32Doubles doubles each
    int nent;
    const int* rows;       // rows of this class with partners of the class's partner L (primitive indices)
    int nrows;
    const double *x, *y, *z;  // row basis coordinates
    const int* cart;          // row basis Cartesian offsets
};

struct KArgs {
    RysTable rys;
    Ewald ew;
    float thresp;
    float thredp;
    int count;
    int symmetric;  // compute only row1 <= row3 and add the transposed block
    int mirror_diag;  // symmetric mode, a class evaluated for its mirror class as well: the
                      // transposed block is added on the diagonal (row1 == row3) too
    KSide s12, s34;
    const double* D;     // D24, ncart2 x ncart4
    int ldD;
    const double* Dsh;   // block maxima, nblk2 x nblk4
    int ldDsh;
    double* K;           // K13, ncart1 x ncart3
    int ldK;
    float maxb12, maxb34;  // max_bound of the two lists
    // Per bra row key r1 * (s12.maxLp + 1) + L2 and ket block: the largest b12 max|D24 block| over the
    // row's partners (upper 16 bits) and the largest max|D24 block| (lower 16), each the upper half
    // of a float, rounded up (launch_k_rowmax), at rw[key * ldrw + blk4 - (rwlo ? rwlo[r1] : 0)];
    // nullptr: not formed.  They only bound what a slot can reach, so 8 bits of mantissa do.
    const unsigned int* rw;
    int ldrw;
    const int* rwlo;
    // learned route (nullptr: none): per unit the certified factor tau in (0, 1] of the Schwarz
    // estimate, applied while thresp >= tau_smin max|D24|
    const float* tau;
    float tau_smin;
    CallScalars* sc;
};

struct CountJArgs {
    float thresp;
    const float* bra_bound;   // bra list bounds (list order)
    const float* ket_b;       // truncated ket bounds (Hermite order)
    const int* ket_hpos;      // list order -> Hermite order
    const int* ket_cls_start; // ket classes (list order)
    const int* ket_cls_L1;
    const int* ket_cls_L2;
    int ket_ncls;
    unsigned long long* out;
    CallScalars* sc;
};

struct CountKArgs {
    float thresp;
    int half;                 // D24symm half-sieve (same list): pivots i2 <= i4 only
    int n2, n4;               // pivot primitives of the two lists
    const int* rs12;          // pivot-view segment starts [n2 * (maxLa+1) + 1]
    const float* b12;         // pivot-view partner bounds
    int maxLa;
    const int* rs34;
    const float* b34;
    int maxLc;
    const int *L2, *L4, *blk2, *blk4;  // pivot angular momenta and block ids
    const double* Dsh;
    int ldDsh;
    float maxb12, maxb34;
    unsigned long long* out;
    CallScalars* sc;
};

void launch_count_j(const CountJArgs& a, int k0, int nk, int L1, int L2, hipStream_t s);
void launch_count_k(const CountKArgs& a, hipStream_t s);

// The classes of a pair list as segments of one launch: workgroups [block0[c], block0[c + 1]) take the
// pairs [k0[c], k0[c] + nk[c]) of class (L1[c], L2[c]).
struct JSegments {
    int n, nblock, maxL;
    int L1[9], L2[9], k0[9], nk[9], hstart[9], block0[9];
    size_t hoff[9];
};
void launch_j_ket_prep(const JPrepArgs& a, const JSegments& seg, hipStream_t s);
void launch_j_bra_scatter(const JScatterArgs& a, const JSegments& seg, hipStream_t s);
// Group pairs (L12 >= L34) of the symmetric J kernel: with one list on both sides it evaluates each
// bra-ket pair of the two groups once for both J blocks (the triangle within one group).  Used
// where measured faster than the two one-way launches: s-type kets (one Hermite component to
// reduce over the wave per ket); with p or d kets the per-ket reduction costs what it saves
// (measured again with the DPP reduction: (2, 1) 1.21 ms against 0.60 + 0.55 ms one-way).
__host__ __device__ constexpr bool js_enabled(int L12, int L34) { return L12 >= L34 && L34 == 0; }
void launch_j_quartets_sym(int L12, int L34, int route, const JQuartetArgs& a, const JTask* tasks, int ntask,
                           unsigned int* qctr, hipStream_t s);
// Bra order 5 (gradients: bra order L12 + 1) runs the FP64 route only.
void launch_j_quartets(int L12, int L34, int route, const JQuartetArgs& a, const JTask* tasks, int ntask,
                       unsigned int* qctr, hipStream_t s);

// Work-queue counters of one call (CallScalars::queue, zeroed with the call's scalars): J classes
// at jcount_index.

// Grid of a persistent kernel: as many workgroups as fit on the device at once (occupancy at
// this block size and LDS), but no more than the work needs.  Raises if the LDS request exceeds
// the device's per-workgroup limit.
int persistent_grid(const void* kernel, int block, size_t lds, long long nwork_groups);

// Dynamic LDS of one k_ket workgroup (as KKetLds lays it out): the staged Rys table blocks (FP64
// for nrys <= 3, FP32 on the mixed route for nrys <= 5), 8-byte aligned, then kKWaves accumulators
// of gsize x N1 x N3 doubles and kKWaves slot queues.
inline size_t kket_lds_bytes(const RysTable& tab, int L1, int L2, int L3, int L4, int route, int gsize)
{
    const int NR = (L1 + L2 + L3 + L4) / 2 + 1;
    size_t b = 0;
    if (rys_staged(NR)) b += rys_lds_doubles(NR) * sizeof(double);
    if (route == kRouteMixed && rys32_staged(NR)) b += rys32_lds_floats(NR) * sizeof(float);
    b = (b + 7) & ~(size_t)7;
    return b + (size_t)kKWaves * (gsize * ncart(L1) * ncart(L3) * sizeof(double) + kKQueueBytes);
}

// KArgs::rw of one exchange call: rows x (maxLp + 1) keys by ldrw ket blocks, from the block maxima
// (K view order) and the bra list's partner lists.  Partners below thresp / (maxb34 max|D24|) fail the
// sieve with every ket and are left out.
void launch_k_rowmax(const int* row_start, int nrow, int maxLp, const int4* ebk, const double* Dsh, int ldDsh, int ncol,
                     const int* rwlo, const int* rwhi, float thresp, float maxb34,
                     const CallScalars* sc, unsigned int* rw, int ldrw, hipStream_t s);

// The K view copies of D24 (ncart2 x ncart4, stride ld) and of its block maxima (nb2 x nb4), and max|D24|.
struct KViewArgs {
    const double* D;
    int ld;
    const int *bc2, *bL2, *bc4, *bL4;  // blocks' Cartesian offsets and angular momenta
    int nb2, nb4;
    const int *kc2, *kc4, *kb2, *kb4;  // K view places of Cartesian functions and blocks (null: unchanged)
    double *Dk, *Dshk;
    CallScalars* sc;
};
void launch_k_kview(const KViewArgs& a, hipStream_t s);
// blk_lo / blk_hi (nullptr: dense): per block 2, the range of blocks 4 of its molecule (batch
// basis); band = the largest such range.
void launch_k_blockmax(const double* D, int ldD, const int* blk_cart2, const int* blk_L2, int nblk2,
                       const int* blk_cart4, const int* blk_L4, int nblk4, double* Dsh, int ldDsh, const int* blk_lo,
                       const int* blk_hi, int band, CallScalars* sc, hipStream_t s);
// Learned-screen training data: per K unit, the largest M_q / (b12 b34) over its quartets with
// b12 b34 >= smin (classes with s and p functions only).
void launch_k_unit_mag_sp(int L1, int L2, int L3, int L4, const KArgs& a, const KGroups& kg, const KUnitG* units,
                          int nunits, float smin, float* out, hipStream_t s);
// K build classes (kRoutePlain or kRouteMixed) over ket-group units.
void launch_k_ket(int L1, int L2, int L3, int L4, int route, const KArgs& a, const KGroups& g, const KUnitG* units,
                  int nunits, hipStream_t s);
void launch_fill(void* p, size_t bytes, hipStream_t s);

// Boys functions F_0..F_nboys (nboys <= kBoysMax) of npoint arguments T, F row-major (npoint x
// (nboys + 1)), FP64 (boys.hip).
constexpr int kBoysMax = 16;
void launch_boys(int nboys, int npoint, const double* T, double* F, hipStream_t s);

// The learned screen's network (mlp.hip): ni <= kMlpMaxIn inputs, 3 hidden layers of kMlpHidden
// ReLU units, one linear output, FP32; kMlpTile samples per workgroup.
constexpr int kMlpHidden = 64;
constexpr int kMlpMaxIn = 32;
constexpr int kMlpTile = 64;
int mlp_nparam(int ni);
void launch_mlp_forward(const float* params, int ni, int n, const float* X, float* out, hipStream_t s);
// grad += d/dparams of (1/nb) sum_s sw_s r_s^2 (times wu where r_s < 0), r_s = f(X[idx[s]]) - y[idx[s]]
// (idx null: s itself; sw null: 1); loss[0] += that loss.
void launch_mlp_grad(const float* params, int ni, int nb, const int* idx, const float* X, const float* y,
                     const float* sw, float wu, float* grad, float* loss, hipStream_t s);
void launch_mlp_adam(int np, float* params, const float* grad, float* m, float* v, float lr, float b1, float b2,
                     float eps, int t, hipStream_t s);
void launch_copy(void* dst, const void* src, size_t bytes, hipStream_t s);

}  // namespace lsjk
