// widom_kernels.hip -- gfx950 kernels of the Widom insertion path.
//
//  * widom_near_kernel     FP64 path of widom: one wavefront per insertion over the framework's
//                          near list, pairs inside the cutoff compacted through LDS, the
//                          reciprocal sum from per-axis phase tables.
//  * widom_f64_kernel      FP64 plain path: one work-item per insertion, every (site, atom)
//                          pair in FP64 with the reference's 17-term pair erfc and libm exp,
//                          minimum image per pair (src/energy.jl:42-82, src/reference.jl:39-56),
//                          bit for bit the oracle's energies: single energies and PA_SINGLE_PHASE.
//  (the mixed-precision pipeline is in widom_binned.hip)
//  * boltzmann_tiles_kernel per-tile log-sum-exp Boltzmann sums {max, sum w, sum U w} in FP64,
//                          deterministic (fixed per-thread order, wavefront butterfly,
//                          wavefronts merged in order).
//  * widom_pose_kernel     device-drawn poses, for bit-exact placement checks.
#include "pa_device.hpp"

namespace pa {

__device__ inline int find_system(const int64_t *seg, int nsys, int64_t g)
{
    // largest s with seg[s] <= g
    int lo = 0, hi = nsys - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (seg[mid] <= g) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// ------------------------------------------------------------------------------------------
// FP64 plain path
// ------------------------------------------------------------------------------------------
template <int NS, bool CHARGED>
__global__ __launch_bounds__(256) void widom_f64_kernel(WidomArgs a)
{
#pragma clang fp contract(off)
    const int64_t g = a.g0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= a.g1) return;
    const int s = find_system(a.seg, a.nsys, g);
    const int64_t j = g - a.seg[s];
    const FwDesc &F = a.fw[a.fw_of[s]];
    double f[3], q[4], pos[3];
    pose_uniforms(a.seed, s, j, f, q);
    matvec(F.A, f, pos);
    double gp[NS][3];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        double r[3];
        rotate(q, a.guest.site[t], r);
        for (int i = 0; i < 3; ++i) gp[t][i] = pos[i] + r[i];
    }
    double E_lj = 0.0, E_sr = 0.0;
    const double4 *atoms = a.atom64 + F.atom_off;
    const int *types = a.atype + F.atom_off;
    for (int n = 0; n < F.natoms; ++n) {
        const double4 h = atoms[n];
        const int ht = types[n];
#pragma unroll
        for (int t = 0; t < NS; ++t) {
            double d[3] = {gp[t][0] - h.x, gp[t][1] - h.y, gp[t][2] - h.z};
            double m[3];
            minimum_image(F.A, F.invA, d, m);
            double r2 = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
            if (!(r2 < a.rc_lj2 || r2 < a.rc_ew2)) continue;
            if (r2 < a.rc_lj2) {
                const double2 p = a.pair64[t * a.ntypes_c + ht];
                double x = p.x * p.x / r2;
                x = x * x * x;
                E_lj += 4.0 * p.y * (x * x - x);
            }
            if (CHARGED && r2 < a.rc_ew2) {
                double r = __builtin_sqrt(r2);
                E_sr += a.guest.q[t] * h.w * pair_erfc_f64(F.alpha * r) / r;
            }
        }
    }
    double E_lr = 0.0;
    if (CHARGED) {
        const double4 *ks = a.k64 + F.k_off;
        const double2 *S = a.S64 + F.k_off;
        for (int i = 0; i < F.nk; ++i) {
            const double4 k = ks[i];
            double re = 0.0, im = 0.0;
#pragma unroll
            for (int t = 0; t < NS; ++t) {
                double ph = k.x * gp[t][0] + k.y * gp[t][1] + k.z * gp[t][2];
                double sn, cs;
                sincos(ph, &sn, &cs);
                re += a.guest.q[t] * cs;
                im += a.guest.q[t] * sn;
            }
            E_lr += k.w * 2.0 * (S[i].x * re + S[i].y * im);
        }
    }
    a.dU[g - a.out_base] = (E_lj + KE * (E_sr + E_lr)) + F.const_off;
}

// ------------------------------------------------------------------------------------------
// FP64 path over the near lists
// ------------------------------------------------------------------------------------------
// One wavefront takes `per` consecutive insertions: it draws their poses one per lane, then
// evaluates them in turn. The plain kernel above tests all natoms x NS pairs and evaluates those
// inside the cutoff under divergence, a fifth of the lanes at a time, with some 250 instructions
// each; here an insertion reads the 790 of RUBTAK's 3,078 atoms near it and evaluates full
// wavefronts of pairs (cw_pair, some 65 instructions). With rho2, an insertion that the phase-0
// radii reject (Boltzmann weight exactly zero) gets Delta U = +inf after the first 64 atoms; a system
// where nothing binds is evaluated again without them (widom_core).
// FP64 issue bounds it. 100,000 insertions of CO2 into RUBTAK 3x3x3: 9.01 ms with the plain kernel,
// 0.77 ms here.
constexpr int WN_WAVES = 4, WN_BATCH = 32;

template <int NS, bool CHARGED, bool UPPER>
__global__ __launch_bounds__(64 * WN_WAVES, 4) void widom_near_kernel(WidomArgs a, NearLists L, const double *rho2, int per,
                                                                    int tab_w)
{
    __shared__ PairRing rings[WN_WAVES];
    __shared__ double wf[WN_WAVES][WN_BATCH][3 * NS];
    __shared__ int wsys[WN_WAVES][WN_BATCH], wbin[WN_WAVES][WN_BATCH];
    extern __shared__ double2 tabs[];  // per wavefront, with charges: (tab_w x NS) phases e^{2 pi i m f_d}
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t first = a.g0 + ((int64_t)blockIdx.x * WN_WAVES + wv) * per;
    if (first >= a.g1) return;  // whole wavefront; the kernel has no barrier
    const int cnt = (int)(a.g1 - first < per ? a.g1 - first : per);
    if (lane < cnt) {
#pragma clang fp contract(off)
        const int64_t g = first + lane;
        const int s = find_system(a.seg, a.nsys, g);
        const int u = a.fw_of[s];
        const FwDesc &F = a.fw[u];
        double f[3], q[4];
        pose_uniforms(a.seed, s, g - a.seg[s], f, q);
        for (int t = 0; t < NS; ++t) {
            double r[3], df[3];
            rotate(q, a.guest.site[t], r);
            matvec(F.invA, r, df);
            for (int d = 0; d < 3; ++d) wf[wv][lane][3 * t + d] = f[d] + df[d];
        }
        wsys[wv][lane] = s;
        wbin[wv][lane] = near_bin(L.desc[u], f);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    double2 *tab = tabs + (size_t)wv * NS * tab_w;
    PairQueue Q(rings[wv], lane);
#pragma unroll 1
    for (int i = 0; i < cnt; ++i) {
        const int s = __builtin_amdgcn_readfirstlane(wsys[wv][i]), bin = __builtin_amdgcn_readfirstlane(wbin[wv][i]);
        const FwDesc &F = a.fw[a.fw_of[s]];
        double f[NS][3];
#pragma unroll
        for (int t = 0; t < NS; ++t)
            for (int d = 0; d < 3; ++d) f[t][d] = wf[wv][i][3 * t + d];
        double e = 0.0;
        const double alpha = F.alpha, rc_ew2 = CHARGED ? a.rc_ew2 : 0.0;
        const bool out = near_scan<NS, UPPER>(
            L, F.atom_off, F.A, bin, f, a.guest.q, a.ntypes_c, fmax(a.rc_lj2, rc_ew2),
            rho2 ? rho2 + (size_t)s * NS * a.ntypes_c : nullptr, Q, [&](double r2, double qq, int code) {
                const double2 p = a.pair64[code];
                e += cw_pair(r2, p.x * p.x, 4.0 * p.y, qq, alpha, a.rc_lj2, rc_ew2);
            });
        if (out) {
            if (lane == 0) a.dU[first + i - a.out_base] = INFINITY;
            continue;
        }
        if (CHARGED) {
            const int m0 = F.kn_max[0] + 1, m1 = F.kn_max[1] + 1, tw = m0 + m1 + F.kn_max[2] + 1;
            const float inv_tw = 1.0f / (float)tw;
#pragma unroll 1
            for (int x = lane; x < NS * tw; x += 64) {
                const int t = (int)(((float)x + 0.5f) * inv_tw), c = x - t * tw;
                const int d = c < m0 ? 0 : (c < m0 + m1 ? 1 : 2);
                tab[c * NS + t] = axis_power_const(wf[wv][i][3 * t + d], c - (d == 0 ? 0 : (d == 1 ? m0 : m0 + m1)));
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int4 *kn = a.kn + F.k_off;
            const double4 *ks = a.k64 + F.k_off;
            const double2 *S64 = a.S64 + F.k_off;
            double acc = 0.0;
#pragma unroll 1
            for (int k = lane; k < F.nk; k += 64) {
                const int4 n = kn[k];
                const double w = ks[k].w;
                const double2 S = S64[k];
                const double2 *tx = tab + abs(n.x) * NS, *ty = tab + (m0 + abs(n.y)) * NS,
                              *tz = tab + (m0 + m1 + abs(n.z)) * NS;
                double re = 0.0, im = 0.0;
#pragma unroll
                for (int t = 0; t < NS; ++t) {
                    const double2 c = cis_from_axes(tx[t], ty[t], tz[t], n.x, n.y, n.z);
                    re = __builtin_fma(a.guest.q[t], c.x, re);
                    im = __builtin_fma(a.guest.q[t], c.y, im);
                }
                acc = __builtin_fma(w, __builtin_fma(S.x, re, S.y * im), acc);
            }
            e = __builtin_fma(2.0 * KE, acc, e);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        e = wave_sum63(e);
        if (lane == 63) a.dU[first + i - a.out_base] = e + F.const_off;
    }
}

// ------------------------------------------------------------------------------------------
// Boltzmann sums
// ------------------------------------------------------------------------------------------
struct Lse {
    double m, w, u;
};

__device__ inline void lse_add(Lse &acc, double lw, double du)
{
    if (lw == -INFINITY) return;  // w == 0 exactly: contributes 0 to both sums (src/widom.jl:80-84)
    if (lw > acc.m) {
        const double sc = exp(acc.m - lw);
        acc.w = acc.w * sc + 1.0;
        acc.u = acc.u * sc + du;
        acc.m = lw;
    } else {
        const double e = exp(lw - acc.m);
        acc.w += e;
        acc.u += du * e;
    }
}

__device__ inline Lse lse_merge(Lse x, Lse y)
{
    if (y.m == -INFINITY) return x;
    if (x.m == -INFINITY) return y;
    const double m = x.m > y.m ? x.m : y.m;
    const double ex = exp(x.m - m), ey = exp(y.m - m);
    Lse r;
    r.m = m;
    r.w = x.w * ex + y.w * ey;
    r.u = x.u * ex + y.u * ey;
    return r;
}

constexpr int TILE_THREADS = 256;

// One workgroup per tile of consecutive insertions (tiles never straddle a block). out[t] =
// {max log w, sum w e^-max, sum dU w e^-max, NaN count}. Each work-item accumulates its
// strided insertions with a running maximum, each wavefront merges its 64 partial sums with
// shuffles (butterfly, fixed order), and work-item 0 merges the wavefronts' results in order.
__global__ __launch_bounds__(TILE_THREADS) void boltzmann_tiles_kernel(const double *dU, const int64_t *tile_g0,
                                                                       const int *tile_n, double kT, double4 *out)
{
    constexpr int NW = TILE_THREADS / 64;
    __shared__ double4 part[NW];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t g0 = tile_g0[t];
    const int n = tile_n[t];
    Lse acc = {-INFINITY, 0.0, 0.0};
    int nan = 0;
    for (int i = tid; i < n; i += TILE_THREADS) {
        const double du = dU[g0 + i];
        const double lw = -du / kT;
        if (lw != lw) { ++nan; continue; }
        lse_add(acc, lw, du);
    }
    for (int off = 32; off >= 1; off >>= 1) {
        const Lse y = {__shfl_xor(acc.m, off, 64), __shfl_xor(acc.w, off, 64), __shfl_xor(acc.u, off, 64)};
        nan += __shfl_xor(nan, off, 64);
        // both lanes of a pair merge (lower lane's value first), so they hold the same result
        acc = (lane & off) ? lse_merge(y, acc) : lse_merge(acc, y);
    }
    if (lane == 0) part[w] = make_double4(acc.m, acc.w, acc.u, (double)nan);
    __syncthreads();
    if (tid == 0) {
        Lse r = {part[0].x, part[0].y, part[0].z};
        double nn = part[0].w;
        for (int i = 1; i < NW; ++i) {
            r = lse_merge(r, Lse{part[i].x, part[i].y, part[i].z});
            nn += part[i].w;
        }
        out[t] = make_double4(r.m, r.w, r.u, nn);
    }
}

// ------------------------------------------------------------------------------------------
// Poses
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void widom_pose_kernel(const FwDesc *fw, const int *fw_of, int sys, uint64_t seed,
                                                         int64_t j0, int64_t n, double *pos, double *quat)
{
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const FwDesc &F = fw[fw_of[sys]];
    double f[3], q[4], p[3];
    pose_uniforms(seed, sys, j0 + i, f, q);
    matvec(F.A, f, p);
    for (int d = 0; d < 3; ++d) pos[3 * i + d] = p[d];
    for (int d = 0; d < 4; ++d) quat[4 * i + d] = q[d];
}

// ------------------------------------------------------------------------------------------
// Host-side launchers
// ------------------------------------------------------------------------------------------
template <int NS>
static void launch_ns(const WidomArgs &a, hipStream_t st)
{
    const int64_t n = a.g1 - a.g0;
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    if (a.guest.charged) hipLaunchKernelGGL((widom_f64_kernel<NS, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((widom_f64_kernel<NS, false>), grid, block, 0, st, a);
}

// FP64 plain-path energy launch over g in [a.g0, a.g1).
hipError_t launch_energy(const WidomArgs &a, int precision, bool upper, hipStream_t st)
{
    (void)precision;
    (void)upper;
    if (a.g1 <= a.g0) return hipSuccess;
    switch (a.guest.nsites) {
    case 1: launch_ns<1>(a, st); break;
    case 2: launch_ns<2>(a, st); break;
    case 3: launch_ns<3>(a, st); break;
    case 4: launch_ns<4>(a, st); break;
    case 5: launch_ns<5>(a, st); break;
    case 6: launch_ns<6>(a, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int NS>
static void launch_near_ns(const WidomArgs &a, const NearLists &L, const double *rho2, bool upper, int per, int tab_w,
                           hipStream_t st)
{
    const int64_t waves = (a.g1 - a.g0 + per - 1) / per;
    const dim3 grid((unsigned)((waves + WN_WAVES - 1) / WN_WAVES)), block(64 * WN_WAVES);
    const size_t lds = a.guest.charged ? sizeof(double2) * WN_WAVES * NS * tab_w : 0;
    if (a.guest.charged) {
        if (upper) hipLaunchKernelGGL((widom_near_kernel<NS, true, true>), grid, block, lds, st, a, L, rho2, per, tab_w);
        else hipLaunchKernelGGL((widom_near_kernel<NS, true, false>), grid, block, lds, st, a, L, rho2, per, tab_w);
    } else {
        if (upper) hipLaunchKernelGGL((widom_near_kernel<NS, false, true>), grid, block, lds, st, a, L, rho2, per, tab_w);
        else hipLaunchKernelGGL((widom_near_kernel<NS, false, false>), grid, block, lds, st, a, L, rho2, per, tab_w);
    }
}

// Widest phase table (entries per site) that the near kernel's LDS holds for an ns-site guest.
int near_tab_max(int ns) { return 96 * 1024 / ((int)sizeof(double2) * WN_WAVES * ns); }

// FP64 energies of g in [a.g0, a.g1) over the near lists; rho2: nsys x NS x ntypes_c phase-0
// radii, or null. tab_w: largest kn_max[0] + kn_max[1] + kn_max[2] + 3 over the frameworks.
hipError_t launch_near(const WidomArgs &a, const NearLists &L, const double *rho2, bool upper, int tab_w, hipStream_t st)
{
    if (a.g1 <= a.g0) return hipSuccess;
    if (a.guest.charged && tab_w > near_tab_max(a.guest.nsites)) return hipErrorInvalidValue;
    // one insertion per wavefront until there are some 16 wavefronts for every SIMD, then up to
    // WN_BATCH, which shares the pose arithmetic among more lanes
    int per = 1;
    while (per < WN_BATCH && (a.g1 - a.g0) / (2 * per) >= 16384) per *= 2;
    switch (a.guest.nsites) {
    case 1: launch_near_ns<1>(a, L, rho2, upper, per, tab_w, st); break;
    case 2: launch_near_ns<2>(a, L, rho2, upper, per, tab_w, st); break;
    case 3: launch_near_ns<3>(a, L, rho2, upper, per, tab_w, st); break;
    case 4: launch_near_ns<4>(a, L, rho2, upper, per, tab_w, st); break;
    case 5: launch_near_ns<5>(a, L, rho2, upper, per, tab_w, st); break;
    case 6: launch_near_ns<6>(a, L, rho2, upper, per, tab_w, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_tiles(const double *dU, const int64_t *tile_g0, const int *tile_n, int ntiles, double kT, double4 *out,
                        hipStream_t st)
{
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(boltzmann_tiles_kernel, dim3((unsigned)ntiles), dim3(TILE_THREADS), 0, st, dU, tile_g0, tile_n, kT,
                       out);
    return hipGetLastError();
}

hipError_t launch_poses(const FwDesc *fw, const int *fw_of, int sys, uint64_t seed, int64_t j0, int64_t n, double *pos,
                        double *quat, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(widom_pose_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, fw, fw_of, sys, seed, j0, n,
                       pos, quat);
    return hipGetLastError();
}

}  // namespace pa
