// pa_device.hpp -- device-side data layout shared by the host library and the kernels.
#pragma once

#include <utility>

#include "pa_numeric.hpp"

namespace pa {

// Per unique framework (FrameworkBatch's deduplicated per-framework storage).
constexpr int NBR_RADII = 3;  // radii at which a phase-0 near list can be cut short

struct FwDesc {
    double A[9];       // cell, column-major
    double invA[9];
    float Af[9];       // A * 2^-32 (maps a 32-bit fixed-point fractional offset to Å)
    double alpha;      // Ewald splitting parameter
    double const_off;  // constant_offset (eV)
    double volume;
    float alphaf;
    int atom_off, natoms;  // slice of the atom arrays
    int k_off, nk;         // slice of the k tables
    int upper;             // A is upper triangular (cell_matrix's form)
    int cg_off;            // hard-core cell grid: first entry of the framework in cell_start and nbr_range
    int cg_nc[3];          // cells per axis (fractional cell edge 1/cg_nc)
    int kn_max[3];         // largest |n_d| of the framework's k-vectors k = 2 pi A^-T n
    // phase-0 near lists: each hard-core cell lists every atom within nbr_r[2] (Å) of any point of it, found
    // by its distance to the cell's centre among the cells within nbr_reach. In shells of squared
    // distance nbr_thr2 (Å^2): those up to number 2 + i hold the atoms within nbr_r[i] of any point
    float nbr_r[NBR_RADII], nbr_thr2[2 + NBR_RADII];
    int nbr_reach[3];
};

// The guest, with compact type indices.
struct GuestDev {
    int nsites;
    int charged;
    double site[MAX_SITES][3];
    double q[MAX_SITES];
    float qke[MAX_SITES];   // KE * q_s in FP32
    int type[MAX_SITES];
    int mirror;             // 3 sites, sites 1 and 2 mirror images through site 0, equal charges
};

// True when a 3-site guest's sites 1 and 2 are mirror images through site 0 (site1 + site2 ==
// 2 site0 exactly) with equal charges: a linear symmetric molecule such as CO2 or a 3-site N2.
inline bool guest_mirror(const GuestDev &G)
{
    if (G.nsites != 3 || G.q[1] != G.q[2]) return false;
    for (int d = 0; d < 3; ++d)
        if (G.site[1][d] + G.site[2][d] != 2.0 * G.site[0][d]) return false;
    return true;
}

// Everything one energy launch needs. The flattened insertion index g runs system-major:
// system s owns g in [seg[s], seg[s+1]); insertion j of system s is g = seg[s] + j.
struct WidomArgs {
    const FwDesc *fw;
    const int *fw_of;          // nsys
    const int64_t *seg;        // nsys + 1
    int nsys;
    uint64_t seed;
    int64_t g0, g1;            // this launch covers g in [g0, g1)
    double *dU;                // indexed by g - out_base
    int64_t out_base;
    // FP64 plain path tables
    const double4 *atom64;     // x, y, z (Å), q
    const int *atype;          // compact type per atom
    const double4 *k64;        // kx, ky, kz, kprefactor
    const double2 *S64;        // host structure factor
    // mixed path tables
    const uint4 *atomfx;       // 32-bit fixed-point fractional x, y, z; q as float bits
    const int4 *kn;            // integer k coefficients n1, n2, n3
    const float2 *kc;          // 2 * kprefactor * (Re S, Im S); the guest charges carry KE
    // pair tables, [site][type] with ntypes_c compact types
    const double2 *pair64;     // sigma, epsilon
    const float2 *pair32;      // sigma^2, 4 epsilon
    int ntypes_c;
    double rc_lj2, rc_ew2;
    float rc_lj2f, rc_ew2f, rc_max2f;
    GuestDev guest;
};

// Spatial bins of one system's insertions (mixed path): the system's cell is cut into
// nb[0] x nb[1] x nb[2] parallelepipeds in fractional coordinates; every insertion is grouped
// with the others whose reference point lies in the same bin, and a bin's neighbour list holds
// every atom image within sqrt(rlist2) of the bin centre.
struct BinSys {
    int nb[3];
    int bin_base;   // first global bin id of the system
    float rlist2;   // (max cutoff + guest radius + bin circumradius + margin)^2, Å^2
    float alt[3];   // an atom with |fractional offset| >= alt[i] on axis i also gets the image
                    // across the cell boundary on that axis (alt >= 0.5: never)
    int hc_end;     // phase 0 runs over the cells' near lists up to this end of nbr_range (1..NBR_RADII); 0: no phase 0
    // radial classes of the neighbour list: class 0 holds the atoms closer than cls_d0 to the bin
    // centre, classes 1..BIN_NCLS-1 split [cls_d0, sqrt(rlist2)] into shells of width 1/cls_inv_w
    float cls_d0, cls_inv_w;
};

// The audit's from-scratch rebuild (audit_kernels.hip). Guest slot g of system n lies in
// [guest_off[n], guest_off[n + 1]); its live guests are the first occ[n].
struct AuditArgs {
    const FwDesc *fw;
    const int *fw_of;
    int nsys;
    const double4 *atom64;     // framework atoms, Cartesian (Å) and charge
    const int *atype;
    const double4 *k64;        // kx, ky, kz, kprefactor
    const double2 *S64;        // framework structure factor
    const int4 *kn;
    const double2 *pair64;     // sigma, epsilon per (site, compact type)
    int ntypes_c;
    double rc_lj2, rc_ew2;     // rc_ew2 = 0 for an uncharged guest
    GuestDev guest;
    const int *guest_off;      // nsys + 1
    const int *sk_off;         // nsys + 1: each system's slice of the running structure factor
    const int *occ;
    const double4 *pos, *quat; // per slot
    int nslots, nsk;
    int tw;                    // per-axis power table entries per site (largest over frameworks)
    double2 *tab;              // nslots * nsites * tw
    double2 *sk;               // rebuilt structure factor, nsk
    double *host_e;            // per slot: rebuilt host-guest energy (0 for an empty slot)
    double *sums;              // per system: host-guest sum, guest-guest pairs, reciprocal sum
};

struct BinnedArgs {
    const FwDesc *fw;
    const int *fw_of;
    const int64_t *seg;        // nsys + 1 flattened insertion offsets
    const BinSys *bins;        // nsys
    const int *bin_base;       // nsys + 1
    int nsys;
    int nbins;
    uint64_t seed;
    int64_t g0, g1;            // this chunk covers g in [g0, g1)
    uint32_t *sitefx;          // (g - g0) * 3 * NS fixed-point site coordinates
    int *key;                  // (g - g0) global bin id
    int *bin_count;            // nbins + 1
    int *bin_start;            // nbins + 1
    int *bin_perm;             // nbins: launch order of the energy kernel (most crowded bins first), or null
    int *bin_iota;             // nbins: 0, 1, 2, ... (the radix sort's input values, grids beyond one workgroup's)
    unsigned *bin_ksort;       // nbins: the sorted counts (the sort's key output)
    int sort_bits;             // bits of the largest possible count
    int *rank;                 // (g - g0) position of the insertion within its bin (from the count)
    int *order;                // chunk-relative insertion indices grouped by bin
    double *dU;                // indexed by g - out_base
    int64_t out_base;
    const uint4 *atomfx;       // the framework's atoms in Morton order: fixed point, q bits
    const int *atype;          // their compact types, same order
    const int4 *kn;
    const float2 *kc;
    const float2 *pair32;
    int ntypes_c;
    float rc_lj2f, rc_ew2f, rc_max2f;
    int listcap;               // neighbour-list capacity (entries) of one pass, >= BIN_WG
    int *extra_passes;         // max over bins of (passes - 1) of this call's energy launches
    int zero_passes;           // nonzero on the call's first chunk: bin_zero_kernel clears it
    GuestDev guest;
    // hard-core rejection (phase 0)
    const int4 *nbr_range;     // per hard-core cell: start of its list in nbr_atoms, and its end for each of nbr_r
    const uint4 *nbr_atoms;    // per cell, the atoms near it (fixed point and compact type), nearest to its centre first
    const float *rho2;         // nsys x NS x ntypes_c rejection radii^2 (Å^2), rounded down
};

// Gradient launches (widom_grad.hip): the weighted-insertion list, its per-insertion sites and
// weights, and the accumulators of the gather and k-space kernels.
struct GradArgs {
    const FwDesc *fw;
    const int *fw_of;
    const int64_t *seg;
    int nsys;
    uint64_t seed;
    const int64_t *list_g;      // flattened insertion index of each weighted insertion
    const double *dU;           // Delta U of every insertion of the run
    const double *msys;         // per system: max of -beta dU (the weight of insertion g is exp(-beta dU - m_s))
    double beta;
    int64_t nlist;
    const uint4 *atomfx;
    const int *atype;
    const int4 *kn;
    const float4 *pairg;        // [site][type]: sigma^2, 4 epsilon, 1/sigma, 0
    int ntypes_c;
    float rc_lj2f, rc_ew2f, rc_max2f;
    GuestDev guest;
    double *acc_lj;             // nsys x NS x ntc x 4: sum w dU/deps, sum wU dU/deps, sum w dU/dsig, sum wU dU/dsig
    double *acc_q;              // per system slice of 2 x natoms: sum w dU/dq_j, sum wU dU/dq_j
    const int64_t *qoff;        // nsys: first atom slot of the system in acc_q
    double *acc_k;              // per system slice of 4 x nk: w Re S_g, w Im S_g, wU Re S_g, wU Im S_g
    const int64_t *koff;        // nsys: first k slot of the system in acc_k
    // gather form
    const int64_t *loff;        // nsys + 1: each system's range of the weighted-insertion list
    uint32_t *lsite;            // per listed insertion: NS x 3 fixed-point site coordinates
    double2 *lw;                // per listed insertion: w, w dU
    const uint4 *corefx;        // atoms sorted by hard-core grid cell: fixed point + compact type
    const int *coreidx;         // original index of each sorted atom
    const int4 *blk;            // per gather workgroup: system, first sorted atom, list range (relative)
    const int4 *kblk;           // per k-space workgroup: system, first k-vector, list range (relative)
};

// Energy sums that need FP64 accuracy (~1e-14 relative) but no bit-for-bit agreement with
// another code path (test insertions into chains, the move path's host-guest sum) use the
// helpers below, which fuse multiply-adds; the helpers above keep every rounding step of the
// reference's formulas for the paths that need exact agreement.
// r^2 of the cell vector A (f - rint(f)) for a fractional offset f.
// UPPER: A[1] == A[2] == A[5] == 0 (every cell built from its parameters). The products with
// those exact zeros are dropped, which leaves every result bit for bit unchanged.
template <bool UPPER>
__device__ inline double cw_r2_t(const double A[9], double f0, double f1, double f2)
{
    f0 -= __builtin_rint(f0);
    f1 -= __builtin_rint(f1);
    f2 -= __builtin_rint(f2);
    const double m0 = __builtin_fma(A[0], f0, __builtin_fma(A[3], f1, A[6] * f2));
    const double m1 = UPPER ? __builtin_fma(A[4], f1, A[7] * f2) : __builtin_fma(A[1], f0, __builtin_fma(A[4], f1, A[7] * f2));
    const double m2 = UPPER ? A[8] * f2 : __builtin_fma(A[2], f0, __builtin_fma(A[5], f1, A[8] * f2));
    return __builtin_fma(m0, m0, __builtin_fma(m1, m1, m2 * m2));
}

// 1/x and 1/sqrt(x) of a positive normal x: the hardware's approximation (about 2^-24) and two
// Newton steps with fused residuals, which leave at most an ulp or two. The compiler's own FP64
// division and square root add the scaling and fix-up for zeros, subnormals and infinities that
// squared distances inside a cutoff never are (r2 = 0 still gives a non-finite pair energy).
__device__ inline double rcp64(double x)
{
    double y = __builtin_amdgcn_rcp(x);
    y = __builtin_fma(__builtin_fma(-x, y, 1.0), y, y);
    return __builtin_fma(__builtin_fma(-x, y, 1.0), y, y);
}

__device__ inline double rsqrt64(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    y = __builtin_fma(__builtin_fma(-x * y, y, 1.0), 0.5 * y, y);
    return __builtin_fma(__builtin_fma(-x * y, y, 1.0), 0.5 * y, y);
}

// The FP64 polynomials' coefficients in constant memory: FP64 instructions take no literals, so
// written as constants they are moved into registers once, outside every loop (60 doubles, 120
// registers). pair_coefs() hides the table's address at each use, and they come by scalar loads.
// exp(r) = sum r^k / k!, the erfc series' 17 coefficients, sincospi's 9 and 10.
struct PairCoefs {
    double exp_c[14], erfc_c[17], sin_c[9], cos_c[10];
};
typedef __attribute__((address_space(4))) const PairCoefs *PairCoefPtr;

template <int... K>
constexpr PairCoefs make_pair_coefs(std::integer_sequence<int, K...>)
{
    return PairCoefs{{1.0, 1.0, 1.0 / 2, 1.0 / 6, 1.0 / 24, 1.0 / 120, 1.0 / 720, 1.0 / 5040, 1.0 / 40320, 1.0 / 362880,
                      1.0 / 3628800, 1.0 / 39916800, 1.0 / 479001600, 1.0 / 6227020800.0},
                     {pair_erfc_mono64(K)...},
                     {SINCOSPI_S[0], SINCOSPI_S[1], SINCOSPI_S[2], SINCOSPI_S[3], SINCOSPI_S[4], SINCOSPI_S[5],
                      SINCOSPI_S[6], SINCOSPI_S[7], SINCOSPI_S[8]},
                     {SINCOSPI_C[0], SINCOSPI_C[1], SINCOSPI_C[2], SINCOSPI_C[3], SINCOSPI_C[4], SINCOSPI_C[5],
                      SINCOSPI_C[6], SINCOSPI_C[7], SINCOSPI_C[8], SINCOSPI_C[9]}};
}
static __constant__ const PairCoefs PAIR_COEFS = make_pair_coefs(std::make_integer_sequence<int, 17>{});

__device__ inline PairCoefPtr pair_coefs()
{
    PairCoefPtr p = (PairCoefPtr)&PAIR_COEFS;
    asm volatile("" : "+s"(p));
    return p;
}

// sum_{k=0..N} c_k x^k as two Horner chains in x^2, even and odd powers: half the dependent steps
// of one chain, which is what a wavefront alone on its SIMD waits for.
template <int N, class P>
__device__ inline double poly_even_odd(double x, const P &c)
{
    const double y = x * x;
    double e = c[N & ~1], o = c[(N - 1) | 1];
#pragma unroll
    for (int k = (N & ~1) - 2; k >= 0; k -= 2) e = __builtin_fma(e, y, c[k]);
#pragma unroll
    for (int k = ((N - 1) | 1) - 2; k >= 0; k -= 2) o = __builtin_fma(o, y, c[k]);
    return __builtin_fma(o, x, e);
}

// exp(x) for x in [-700, 1]: x = n ln2 + r with |r| <= ln2 / 2 (Cody-Waite: ln2 in two parts, so that n
// times the first is exact), the Taylor series of exp(r) to
// r^13 (remainder below 5e-18 of the value), scaled by 2^n.
__device__ inline double exp64_small(double x, PairCoefPtr C)
{
    const double n = __builtin_rint(x * 1.4426950408889634);
    const double r = __builtin_fma(-n, 1.9082149292705877e-10, __builtin_fma(-n, 0.6931471803691238, x));
    return __builtin_amdgcn_ldexp(poly_even_odd<13>(r, C->exp_c), (int)n);
}

// LJ inside rc_lj plus qq_ke erfc(alpha r)/r inside rc_ew. The value of pair_erfc_f64 through the
// same series as an ordinary polynomial (16 fused steps instead of 32 operations), one
// reciprocal square root for r and 1/r and one reciprocal for t: about 65 FP64 instructions
// where the Clenshaw form with the library's divisions, square root and exp takes about 250.
// An attempt of one chain evaluates some 1,100 pairs on four wavefronts.
// sg2 = sigma^2, ep4 = 4 epsilon. EXACT_LJ: the LJ term in site_pair_energy's own operations, so
// that a pair of overlapping guests (1e6 eV and more are allowed) has the same bits here and in
// the rebuilds that the running energy is audited against.
template <bool EXACT_LJ = false>
__device__ inline double cw_pair(double r2, double sg2, double ep4, double qq_ke, double alpha, double rc_lj2,
                                 double rc_ew2)
{
    const double ir = rsqrt64(r2);
    double e = 0.0;
    if (r2 < rc_lj2) {
#pragma clang fp contract(off)
        double x = EXACT_LJ ? sg2 / r2 : sg2 * (ir * ir);
        x = x * x * x;
        e = ep4 * (EXACT_LJ ? x * x - x : __builtin_fma(x, x, -x));
    }
    if (r2 < rc_ew2) {
        const double z = alpha * (r2 * ir);
        const double t = 2.0 * rcp64(2.0 + z);
        constexpr double XA = 4.0 / (1.0 - PAIR_ERFC_XLO), XB = -2.0 * (1.0 + PAIR_ERFC_XLO) / (1.0 - PAIR_ERFC_XLO) - 1.0;
        const double xi = __builtin_fma(XA, t, XB);
        // log(erfc(z)/t) + z^2
        const PairCoefPtr C = pair_coefs();
        const double p = poly_even_odd<16>(xi, C->erfc_c);
        e = __builtin_fma(qq_ke * (t * exp64_small(__builtin_fma(-z, z, p), C)), ir, e);
    }
    return e;
}

// One site pair of the move path (FP64): Lennard-Jones inside rc_lj plus the screened Coulomb
// qq_ke * erfc(alpha r)/r inside rc_ew (qq_ke = KE q_a q_b), on a minimum-image separation r^2.
__host__ __device__ inline double site_pair_energy(double r2, double sg, double ep, double qq_ke, double alpha,
                                                   double rc_lj2, double rc_ew2)
{
#pragma clang fp contract(off)
    double e = 0.0;
    if (r2 < rc_lj2) {
        double x = sg * sg / r2;
        x = x * x * x;
        e = 4.0 * ep * (x * x - x);
    }
    if (r2 < rc_ew2) {
        const double r = __builtin_sqrt(r2);
        e += qq_ke * pair_erfc_f64(alpha * r) / r;
    }
    return e;
}

// e^{i k.r} of a guest site for k = 2 pi A^-T n at the Cartesian point r = A f, as the product
// over axes of e^{2 pi i n_d f_d}. axis_power gives e^{2 pi i m f_d} (m >= 0), the phase m f_d
// reduced to one revolution with its rounding error carried along, so that a product of two
// powers agrees with the power of the sum to an ulp or two (the move kernel multiplies powers
// where the audit's rebuild takes one); cis_from_axes multiplies the three, conjugating the axes
// with negative n_d. The host's and the audit's structure-factor rebuilds evaluate both
// identically.
__host__ __device__ inline double axis_phase(double f, int m)
{
#pragma clang fp contract(off)
    f -= __builtin_rint(f);
    const double p = (double)m * f, lo = __builtin_fma((double)m, f, -p);
    return 2.0 * ((p - __builtin_rint(p)) + lo);
}

__host__ __device__ inline double2 axis_power(double f, int m)
{
    double sn, cs;
    sincospi(axis_phase(f, m), &sn, &cs);
    return make_double2(cs, sn);
}

// The same with the series' coefficients from constant memory (pair_coefs), same operations.
__device__ inline double2 axis_power_const(double f, int m)
{
    const PairCoefPtr C = pair_coefs();
    double sn, cs;
    sincospi_coefs(axis_phase(f, m), C->sin_c, C->cos_c, &sn, &cs);
    return make_double2(cs, sn);
}

__host__ __device__ inline double2 axis_power(const double *invA, const double r[3], int d, int m)
{
#pragma clang fp contract(off)
    return axis_power(invA[d] * r[0] + invA[d + 3] * r[1] + invA[d + 6] * r[2], m);
}

__host__ __device__ inline double2 cis_from_axes(double2 e0, double2 e1, double2 e2, int nx, int ny, int nz)
{
#pragma clang fp contract(off)
    const double i0 = nx < 0 ? -e0.y : e0.y, i1 = ny < 0 ? -e1.y : e1.y, i2 = nz < 0 ? -e2.y : e2.y;
    const double pr = e0.x * e1.x - i0 * i1, pi = e0.x * i1 + i0 * e1.x;
    return make_double2(pr * e2.x - pi * i2, pr * i2 + pi * e2.x);
}

// The k-vectors of a framework as runs of consecutive n3 at fixed (n1, n2), longest first, cut
// into blocks of 64 runs, one run per lane. A run of length L is walked from its middle outwards:
// step 0 is n3 = m, step j takes m + j (while 2j <= L) and m - j (while 2j + 1 <= L), so that both
// share the products of e^{2 pi i (n1 f1 + n2 f2 + m f3)} and e^{2 pi i j f3}. Lengths descend,
// so the runs still active at a step are the block's first lanes, and the k-vectors are stored in
// the order in which they are visited (block, step, +/-, lane) without gaps.
struct KRuns {
    const int4 *run;           // n1, n2, m, length; framework u's at [run_off[u], run_off[u + 1])
    const int *run_off;        // nfw + 1
    const int *base;           // per block of 64 runs: position of its first k-vector
    const int *blk_off;        // nfw + 1
    const double *kw;          // kprefactor by position (slices as the k tables)
};

// Ring of in-cutoff pairs of one wavefront in LDS: lanes append the pairs they found inside the
// cutoff (two numbers and a code), full wavefronts evaluate 64 at a time, so that LJ + erfc run
// on full wavefronts whatever the lanes' own pairs do. Up to 63 pending and 3 x 64 new.
constexpr int PAIR_RING = 256;
struct PairRing {
    double x[PAIR_RING], y[PAIR_RING];
    int code[PAIR_RING];
};
struct PairQueue {
    PairRing &r;
    int lane;
    unsigned head, tail;
    __device__ PairQueue(PairRing &ring, int l) : r(ring), lane(l), head(0), tail(0) {}
    __device__ inline unsigned pending() const { return tail - head; }
    __device__ inline void push(bool in, double x, double y, int code)
    {
        const uint64_t mask = __builtin_amdgcn_ballot_w64(in);
        if (in) {
            const unsigned below = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
            const unsigned i = (tail + below) & (PAIR_RING - 1);
            r.x[i] = x;
            r.y[i] = y;
            r.code[i] = code;
        }
        tail += (unsigned)__popcll(mask);
    }
    // evaluates the oldest cnt <= 64 pairs: eval(x, y, code)
    template <class E>
    __device__ inline void drain(unsigned cnt, E &&eval)
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if ((unsigned)lane < cnt) {
            const unsigned i = (head + lane) & (PAIR_RING - 1);
            eval(r.x[i], r.y[i], r.code[i]);
        }
        head += cnt;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
};

// Sum over the wavefront, in lane 63 (DPP shifts within rows of 16 lanes, then row broadcasts).
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v)
{
    const uint64_t b = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, true);
    return v + __longlong_as_double(((uint64_t)hi << 32) | lo);
}

__device__ inline double wave_sum63(double v)
{
    v = dpp_add<0x111, 0xf>(v);  // row_shr:1
    v = dpp_add<0x112, 0xf>(v);  // row_shr:2
    v = dpp_add<0x114, 0xf>(v);  // row_shr:4
    v = dpp_add<0x118, 0xf>(v);  // row_shr:8
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    return dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}

// Lists of the atoms near a point (batch_kernels.hip): bins of framework u's cell, and per bin the
// atoms that a guest with its reference point in the bin can have inside the cutoff. An entry is
// the atom's index (Morton order, framework-relative) and above it its compact type.
constexpr int NEAR_TYPE_SHIFT = 26;
constexpr uint32_t NEAR_INDEX = (1u << NEAR_TYPE_SHIFT) - 1u;
struct NearDesc {
    int nb[3];
    int bin_off;               // first bin of the framework in `start`
    double r2;                 // squared list radius, Å^2
    double close2;             // a list's first entries: the atoms within 2 Å of any site in the bin
    double reach[3];           // list radius over the perpendicular widths
};
struct NearLists {
    const double4 *atomf;      // fractional x, y, z in [0, 1) and charge, Morton order
    const NearDesc *desc;
    const int *start;          // per bin, one past the last included
    const uint32_t *ent;
};

// What the kernels share that build the lists (batch_kernels.hip).
struct NearBuild {
    const FwDesc *fw;
    const NearDesc *nd;
    const int *bin_fw;         // nfw + 1: first bin of every framework
    const int *run_off;        // nfw + 1: first run of 64 atoms of every framework
    int nfw, nbins, nruns;
    const double4 *atomf;
    const int *atype;          // in the same order
    double4 *run;              // per run of 64 atoms: centre (fractional), radius (Å)
    int *start;                // nbins + 1: counts (first pass), then offsets
    int *close;                // nbins: the atoms within close2 among them (first pass)
    uint32_t *ent;             // entries (second pass)
};

// The bin of a point with fractional coordinates f.
__device__ inline int near_bin(const NearDesc &D, const double f[3])
{
    int c[3];
    for (int d = 0; d < 3; ++d) {
        const double x = f[d] - __builtin_floor(f[d]);
        c[d] = min(D.nb[d] - 1, (int)(x * D.nb[d]));
    }
    return D.bin_off + c[0] + D.nb[0] * (c[1] + D.nb[1] * c[2]);
}

// One wavefront's host-guest pairs inside the cutoff, from the near list of `bin`: the guest's sites
// at fractional coordinates f in the cell A, pairs queued as (r^2, KE q_site q_atom, site * ntypes_c + type) and
// evaluated by `eval`. Several wavefronts share a list as the w-th of nw. With rho2 (squared radii by the same code) the first 64 entries, which hold
// the atoms close to the bin, are tested first: true if a site lies inside one, with nothing
// more evaluated.
template <int NS, bool UPPER, class E>
__device__ inline bool near_scan(const NearLists &L, int atom_off, const double *A, int bin, const double (&f)[NS][3],
                                 const double *q, int ntypes_c, double rc_max2, const double *rho2, PairQueue &Q,
                                 E &&eval, int w = 0, int nw = 1)
{
    const double nan = __builtin_nan("");
    const double4 *af = L.atomf + atom_off;
    const int e0 = L.start[bin], ne = L.start[bin + 1] - e0, lane = Q.lane, j0 = w * 64 + lane;
    const uint32_t *ent = L.ent + e0;
    // the next entry and its atom are loaded while the current one is evaluated; a lane past the
    // list's end takes a NaN position, which is inside nothing
    uint32_t en = j0 < ne ? ent[j0] : 0u;
    double4 hn = j0 < ne ? af[en & NEAR_INDEX] : make_double4(nan, nan, nan, 0.0);
#pragma unroll 1
    for (int jb = w * 64; jb < ne; jb += nw * 64) {
        const double4 h = hn;
        const int ht = (int)(en >> NEAR_TYPE_SHIFT), j = jb + lane + nw * 64;
        hn = make_double4(nan, nan, nan, 0.0);
        if (j < ne) {
            en = ent[j];
            hn = af[en & NEAR_INDEX];
        }
        double r2[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) r2[s] = cw_r2_t<UPPER>(A, f[s][0] - h.x, f[s][1] - h.y, f[s][2] - h.z);
        if (rho2 && jb == 0) {
            bool hit = false;
#pragma unroll
            for (int s = 0; s < NS; ++s) hit = hit || r2[s] < rho2[s * ntypes_c + ht];
            if (__builtin_amdgcn_ballot_w64(hit)) return true;
        }
        const double qh = KE * h.w;
#pragma unroll
        for (int s0 = 0; s0 < NS; s0 += 3) {
#pragma unroll
            for (int s = s0; s < (s0 + 3 < NS ? s0 + 3 : NS); ++s)
                Q.push(r2[s] < rc_max2, r2[s], q[s] * qh, s * ntypes_c + ht);
#pragma unroll 1
            while (Q.pending() >= 64) Q.drain(64, eval);
        }
    }
    Q.drain(Q.pending(), eval);
    return false;
}

// Move types of the move path: the reference's three NVT moves (src/moves.jl:69-71) and the two
// exchange moves.
constexpr int MOVE_TRANSLATION = 1, MOVE_ROTATION = 2, MOVE_REINSERTION = 3, MOVE_INSERTION = 4, MOVE_DELETION = 5;
constexpr int NMOVES = 5;

// Snapshots of the chains' states for the test insertions (nvt_kernels.hip). Slot c holds, per
// system n: occupancy at occ[c * nsys + n]; guests at pos/quat[c * nslots + guest_off[n] + i];
// the weighted structure factor c_k = kprefactor_k * S_k of every k-vector at
// csk[c * ctot + coff[n] + p] for the k-vector at position p (KRuns).
struct ChainSnap {
    int nsys, nslots;
    int64_t ctot;
    const int *coff;           // per system: first entry of its slice of csk
    int *occ;
    double4 *pos, *quat;
    double2 *csk;
};

// One launch of the move path: every chain (system) is one workgroup that runs its move attempts
// back to back (mc_kernels.hip).
struct McArgs {
    // framework tables: the FP64 layout with every k-vector (FULLK batch)
    const FwDesc *fw;
    const int *fw_of;
    NearLists near;             // the framework atoms near a pose
    KRuns kr;                   // the k-vectors; Sk is stored in their order
    int ktab_w;                 // max over frameworks of kn_max[0] + kn_max[1] + kn_max[2] + 3
    const double2 *pair64;      // [site][type]: sigma, epsilon
    int ntypes_c;
    double rc_lj2, rc_ew2;
    double rc_max2;             // max(rc_lj2, rc_ew2): the host-guest pair test
    GuestDev guest;
    int nsys;
    // chain state (SystemState, src/state.jl:89-104)
    const int *guest_off;       // nsys + 1: capacity blocks
    int *occupancy;
    double4 *refpos;            // per slot: x, y, z (Å), 0
    double4 *quat;              // per slot: x, y, z, w
    double *host_e;             // per slot: cached host-guest real-space energy
    double4 *gsite;             // scratch, per slot and site: Cartesian positions of the live guests' sites
    double2 *Sk;                // per system k slice, by position: host + every guest
    double *sk_abs;             // per system: accumulated rounding scale of every S_k
    const int *sk_off;          // nsys + 1
    double *energy, *energy_abs;
    const uint64_t *rng_seed;
    uint64_t *rng_counter;
    int *accepted, *attempted;  // nsys x NMOVES
    // what to run
    int mode;                   // 0: nmoves attempts of movetype; 1: ncycles GCMC cycles
    int movetype;
    int64_t nmoves;
    int64_t ncycles, min_cycle;
    double pcum[NMOVES];        // mode 1: cumulative probabilities of the move types
    const double *step_trans, *step_rot;   // per chain
    const double *log_fugV;     // per chain: log of fugacity (eV/Å^3) times volume
    const double *logn;         // log 1, log 2, ... up to the largest capacity + 1
    double log_kT;
    const double *const_p, *const_q;       // exchange constant term p + q N (src/moves.jl:728-773)
    double kT;
    int upper;                  // every framework's A has A[1] == A[2] == A[5] == 0
    // mode 1 sampling: after every cycle c of this launch, samp_*[n * samp_stride + samp_base + c]
    int sampling;
    int64_t samp_base, samp_stride;
    double *samp_e, *samp_n;
    int *max_occ;
    int *capacity_hits;         // per chain: accepted-by-Metropolis insertions refused at capacity
    double4 *trace;             // optional, per chain trace_cap entries: type, slot, dU, accepted
    int64_t trace_cap;
    // mode 1 snapshots: the state at the end of cycle c (0-based within the launch) for c < snap_n
    // (layout of ChainSnap)
    int64_t snap_n;
    ChainSnap snap;
};

// Test insertions into the chains' current configurations (nvt_kernels.hip). Insertion i of
// system s lies in [item_off[s], item_off[s+1]); local index l = i - item_off[s] is cycle slot
// l / nw, insertion l % nw of that cycle. Its pose is pose_pos/pose_quat[i] when given, else the
// Widom stream's pose of per-system index (cyc0 + slot) * nw + l % nw. Cycle slot c sees snapshot
// min(c, snap_n - 1).
struct ChainWidomArgs {
    const FwDesc *fw;
    const int *fw_of;
    NearLists near;             // the framework atoms near a pose
    KRuns kr;                   // the k-vectors
    int ktab_w;                 // max over frameworks of kn_max[0] + kn_max[1] + kn_max[2] + 3
    int upper;                  // every framework's A has A[1] == A[2] == A[5] == 0
    const double2 *pair64;
    int ntypes_c;
    double rc_lj2, rc_ew2;
    double rc_max2;             // max(rc_lj2, rc_ew2): the host-guest pair test
    GuestDev guest;
    int nsys;
    const int *guest_off;
    int64_t snap_n;
    ChainSnap snap;
    const int64_t *item_off;    // nsys + 1
    int64_t nitems, nw, cyc0;
    uint64_t widom_seed;
    const double *pose_pos, *pose_quat;
    double *dU;                 // nitems: energy without the insertion constant
};

}  // namespace pa
