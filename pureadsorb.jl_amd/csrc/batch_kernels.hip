// batch_kernels.hip -- FrameworkBatch tables on gfx950: the host structure factor at the
// k-vectors a framework keeps (src/batch.jl:173-195) and the 64-orientation guest self term
// over its full k table (src/batch.jl:360-389), both FP64, the phase-0 atom lists and
// the FP64 paths' near lists. k = 2 pi A^-T n, so e^{i k.r} = e^{2 pi i n.f}
// with f = A^-1 r; every phase is one own-sincospi of 2 n.f.
#include <hipcub/hipcub.hpp>

#include "pa_host.hpp"

namespace pa {

constexpr int BK_WG = 256;

// S(k_i) = sum_j q_j e^{2 pi i n_i.f_j} for the requested n_i (one work-item each); the atoms
// (fractional coordinates and charge) pass through LDS in tiles shared by the workgroup.
__global__ __launch_bounds__(BK_WG) void sk_kernel(const double4 *atoms, int natoms, const int4 *kreq, int nreq,
                                                   double2 *out)
{
    __shared__ double4 tile[BK_WG];
    const int i = blockIdx.x * BK_WG + threadIdx.x;
    const int4 n = i < nreq ? kreq[i] : make_int4(0, 0, 0, 0);
    const double n0 = (double)n.x, n1 = (double)n.y, n2 = (double)n.z;
    double re = 0.0, im = 0.0;
    for (int t0 = 0; t0 < natoms; t0 += BK_WG) {
        const int j = t0 + (int)threadIdx.x;
        tile[threadIdx.x] = j < natoms ? atoms[j] : make_double4(0, 0, 0, 0);
        __syncthreads();
        const int m = natoms - t0 < BK_WG ? natoms - t0 : BK_WG;
        for (int jj = 0; jj < m; ++jj) {
            const double4 a = tile[jj];
            double sn, cs;
            sincospi(2.0 * __builtin_fma(n2, a.z, __builtin_fma(n1, a.y, n0 * a.x)), &sn, &cs);
            re = __builtin_fma(a.w, cs, re);
            im = __builtin_fma(a.w, sn, im);
        }
        __syncthreads();
    }
    if (i < nreq) out[i] = make_double2(re, im);
}

// Partial sums of kprefactor_k |sum_s q_s e^{2 pi i n_k.g_os}|^2 over 64 consecutive k-vectors
// for each of the 64 orientations o (lane = orientation; the four wavefronts take every fourth
// k-vector). g_os: fractional coordinates of site s rotated by orientation o.
__global__ __launch_bounds__(BK_WG) void self_term_kernel(const int4 *kn, const double *kpref, int nk,
                                                         const double *gsf, const double *q, int ns, double *partial)
{
    __shared__ double red[BK_WG / 64][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int k0 = blockIdx.x * 64, k1 = k0 + 64 < nk ? k0 + 64 : nk;
    double acc = 0.0;
    for (int k = k0 + w; k < k1; k += BK_WG / 64) {
        const int4 n = kn[k];
        const double n0 = (double)n.x, n1 = (double)n.y, n2 = (double)n.z;
        double re = 0.0, im = 0.0;
        for (int s = 0; s < ns; ++s) {
            const double *g = gsf + 3 * (lane * ns + s);
            double sn, cs;
            sincospi(2.0 * __builtin_fma(n2, g[2], __builtin_fma(n1, g[1], n0 * g[0])), &sn, &cs);
            re = __builtin_fma(q[s], cs, re);
            im = __builtin_fma(q[s], sn, im);
        }
        acc = __builtin_fma(kpref[k], __builtin_fma(re, re, im * im), acc);
    }
    red[w][lane] = acc;
    __syncthreads();
    if (w == 0) partial[(int64_t)blockIdx.x * 64 + lane] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

// Squared length of A (x, y, z). A list kernel's counting and its filling instantiation have to agree
// on every atom, to the last bit, or an entry is left unwritten or written into the next list: the
// fused operations are spelt out, so that neither depends on what the compiler contracts.
template <class R>
__device__ inline R length2(const R A[9], R x, R y, R z)
{
#pragma clang fp contract(off)
    auto fma = [](R a, R b, R c) -> R {
        if constexpr (sizeof(R) == 8) return __builtin_fma(a, b, c);
        else return __builtin_fmaf(a, b, c);
    };
    const R ex = fma(A[6], z, fma(A[0], x, A[3] * y));
    const R ey = fma(A[7], z, fma(A[1], x, A[4] * y));
    const R ez = fma(A[8], z, fma(A[2], x, A[5] * y));
    return fma(ez, ez, fma(ex, ex, ey * ey));
}

// Phase-0 near lists: for every hard-core cell, the atoms within nbr_r of any point of it, by their
// minimum-image distance to the cell's centre. One wavefront per cell, its lanes over the cells
// within nbr_reach (each once where the reach goes around the axis). Without FILL the lists are
// counted into nbr_start (and their sum added to *sum); with it they are written in shells of growing
// distance, so that an insertion's overlap is usually found among the first entries and a call of smaller
// radii stops at the end of the last shell that can hold one, and nbr_range gets the start and those ends.
// cell_fw_off (nfw + 1) maps the global cell index to its framework.
template <bool FILL>
__global__ __launch_bounds__(BK_WG) void nbr_kernel(const FwDesc *fw, int nfw, const int *cell_fw_off, int ncells,
                                                   const int *cell_start, int *nbr_start, const uint4 *corefx,
                                                   uint4 *nbr_atoms, int4 *nbr_range, unsigned long long *sum)
{
    const int lane = threadIdx.x & 63;
    const int g = blockIdx.x * (BK_WG / 64) + (threadIdx.x >> 6);
    if (g >= ncells) return;
    int lo = 0, hi = nfw - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cell_fw_off[mid] <= g) lo = mid; else hi = mid - 1;
    }
    const FwDesc &D = fw[__builtin_amdgcn_readfirstlane(lo)];
    const int c = g - cell_fw_off[lo];
    const int nc[3] = {D.cg_nc[0], D.cg_nc[1], D.cg_nc[2]};
    const int h[3] = {c % nc[0], (c / nc[0]) % nc[1], c / (nc[0] * nc[1])};
    int k[3], first[3];
    uint32_t x[3];
    for (int d = 0; d < 3; ++d) {
        const int w = 2 * D.nbr_reach[d] + 1;
        k[d] = w < nc[d] ? w : nc[d];
        first[d] = w < nc[d] ? h[d] - D.nbr_reach[d] + nc[d] : 0;
        x[d] = to_fixed((h[d] + 0.5) / nc[d]);
    }
    const int ncand = k[0] * k[1] * k[2];
    const int *cs = cell_start + D.cg_off;
    const uint4 *src = corefx + D.atom_off;
    constexpr int SHELLS = 2 + NBR_RADII;
    // calls take(atom, its squared distance) for every atom of the cells in reach, one a lane
    auto each_atom = [&](auto &&take) {
        for (int i0 = 0; i0 < ncand; i0 += 64) {
            const int i = i0 + lane;
            int b0 = 0, len = 0;
            if (i < ncand) {
                const int c0 = (first[0] + i % k[0]) % nc[0], c1 = (first[1] + (i / k[0]) % k[1]) % nc[1],
                          c2 = (first[2] + i / (k[0] * k[1])) % nc[2];
                const int cc = c0 + nc[0] * (c1 + nc[1] * c2);
                b0 = cs[cc];
                len = cs[cc + 1] - b0;
            }
            for (int j = 0; __builtin_amdgcn_ballot_w64(j < len); ++j) {
                uint4 at = make_uint4(0u, 0u, 0u, 0u);
                float r2 = INFINITY;
                if (j < len) {
                    at = src[b0 + j];
                    r2 = length2(D.Af, (float)(int32_t)(x[0] - at.x), (float)(int32_t)(x[1] - at.y),
                                 (float)(int32_t)(x[2] - at.z));
                }
                take(at, r2);
            }
        }
    };
    auto atoms = [&](float r2, int sh) {  // the lanes whose atom is no farther than shell sh
        return __builtin_amdgcn_ballot_w64(r2 <= D.nbr_thr2[sh]);
    };
    int total = 0;
    if (!FILL) {
        each_atom([&](const uint4 &, float r2) { total += __popcll(atoms(r2, SHELLS - 1)); });
    } else {
        // the shells' sizes, then the atoms into all of them at once
        const int at0 = nbr_start[D.cg_off + c];
        int end[SHELLS], pos[SHELLS];
#pragma unroll
        for (int sh = 0; sh < SHELLS; ++sh) end[sh] = at0;
        each_atom([&](const uint4 &, float r2) {
#pragma unroll
            for (int sh = 0; sh < SHELLS; ++sh) end[sh] += __popcll(atoms(r2, sh));
        });
#pragma unroll
        for (int sh = 0; sh < SHELLS; ++sh) pos[sh] = sh ? end[sh - 1] : at0;
        each_atom([&](const uint4 &at, float r2) {
            uint64_t inner = 0;
#pragma unroll
            for (int sh = 0; sh < SHELLS; ++sh) {
                const uint64_t within = atoms(r2, sh), m = within & ~inner;
                if ((m >> lane) & 1) nbr_atoms[pos[sh] + __popcll(m & ((1ull << lane) - 1ull))] = at;
                pos[sh] += __popcll(m);
                inner = within;
            }
        });
        static_assert(NBR_RADII == 3, "a cell's start and ends are an int4");
        if (lane == 0) nbr_range[D.cg_off + c] = make_int4(at0, end[2], end[3], end[4]);
    }
    if (!FILL && lane == 0) nbr_start[D.cg_off + c] = total;
    if (!FILL && sum && lane == 0 && total) atomicAdd(sum, (unsigned long long)total);
    // the slot past a framework's last cell: no atoms
    if (!FILL && lane == 0 && g + 1 == cell_fw_off[lo + 1]) nbr_start[D.cg_off + c + 1] = 0;
}

// Exclusive scan of n counts in place (tmp == nullptr: only the temporary size).
hipError_t scan_counts(int *counts, int n, void *tmp, size_t *tmp_bytes, hipStream_t st)
{
    return hipcub::DeviceScan::ExclusiveSum(tmp, *tmp_bytes, counts, counts, n, st);
}

hipError_t launch_nbr(bool fill, const FwDesc *fw, int nfw, const int *cell_fw_off, int ncells, const int *cell_start,
                      int *nbr_start, const uint4 *corefx, uint4 *nbr_atoms, int4 *nbr_range, unsigned long long *sum,
                      hipStream_t st)
{
    if (ncells <= 0) return hipSuccess;
    const dim3 grid((unsigned)((ncells + BK_WG / 64 - 1) / (BK_WG / 64))), block(BK_WG);
    if (fill)
        hipLaunchKernelGGL(nbr_kernel<true>, grid, block, 0, st, fw, nfw, cell_fw_off, ncells, cell_start, nbr_start,
                           corefx, nbr_atoms, nbr_range, sum);
    else
        hipLaunchKernelGGL(nbr_kernel<false>, grid, block, 0, st, fw, nfw, cell_fw_off, ncells, cell_start, nbr_start,
                           corefx, nbr_atoms, nbr_range, sum);
    return hipGetLastError();
}

hipError_t launch_sk(const double4 *atoms, int natoms, const int4 *kreq, int nreq, double2 *out, hipStream_t st)
{
    if (nreq <= 0) return hipSuccess;
    hipLaunchKernelGGL(sk_kernel, dim3((unsigned)((nreq + BK_WG - 1) / BK_WG)), dim3(BK_WG), 0, st, atoms, natoms, kreq,
                       nreq, out);
    return hipGetLastError();
}

hipError_t launch_self_term(const int4 *kn, const double *kpref, int nk, const double *gsf, const double *q, int ns,
                            double *partial, hipStream_t st)
{
    if (nk <= 0) return hipSuccess;
    hipLaunchKernelGGL(self_term_kernel, dim3((unsigned)((nk + 63) / 64)), dim3(BK_WG), 0, st, kn, kpref, nk, gsf, q, ns,
                       partial);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Near lists: per-framework lists of the atoms near a point, for the FP64 paths.
//
// Every unique framework's cell is cut into bins of about NEAR_EDGE Å; a bin lists the atoms of
// which some image lies within R = max cutoff + largest site distance + bin circumradius of the
// bin's centre. The atoms that any site of a guest with its reference point in the bin can have
// inside the cutoff are then among them, whatever image is the nearest: the image that a site
// sees differs from the nearest one to the centre by at most one cell along each axis (both
// offsets are within half a cell, and the site within a small part of one of the centre), and
// all 27 are tried. Atoms are tried in runs of 64 neighbours in Morton order, and only the runs whose
// bounding sphere comes within R of the centre: trying every atom, the lists of a framework of 60,000
// took 100 ms, some 10 ms so. On RUBTAK 3x3x3 a list holds 790 of 3,078 atoms, of which a site has 360 inside
// its cutoff. Smaller bins have shorter lists (R falls with the circumradius) and more of them:
// 2.5 Å takes 11 MB on RUBTAK, and the edge grows until a batch's lists fit NEAR_MAX_ENTRIES.
// ------------------------------------------------------------------------------------------

constexpr double NEAR_EDGE = 2.5;
constexpr double NEAR_MAX_ENTRIES = 268435456.0;  // 1 GiB of 4-byte entries

// Centre (fractional) and radius (Å) of every run of 64 atoms, by each atom's nearest image to the run's
// first one. One wavefront per run.
__global__ __launch_bounds__(256) void near_run_kernel(NearBuild a)
{
    const int lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= a.nruns) return;
    int lo = 0, hi = a.nfw - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.run_off[mid] <= r) lo = mid; else hi = mid - 1;
    }
    const FwDesc &F = a.fw[__builtin_amdgcn_readfirstlane(lo)];
    const int i0 = (r - a.run_off[lo]) * 64, m = min(64, F.natoms - i0);
    const double4 *p = a.atomf + F.atom_off + i0;
    const double4 h = p[min(lane, m - 1)], h0 = p[0];
    double d[3] = {h.x - h0.x, h.y - h0.y, h.z - h0.z}, c[3];
    for (int e = 0; e < 3; ++e) {
        d[e] -= __builtin_rint(d[e]);
        c[e] = __shfl(wave_sum63(lane < m ? d[e] : 0.0), 63, 64) / m;
    }
    double rad2 = length2(F.A, d[0] - c[0], d[1] - c[1], d[2] - c[2]);
    for (int off = 32; off >= 1; off >>= 1) rad2 = fmax(rad2, __shfl_xor(rad2, off, 64));
    if (lane == 0) a.run[r] = make_double4(h0.x + c[0], h0.y + c[1], h0.z + c[2], __builtin_sqrt(rad2) + 1.0e-6);
}

// Squared distance (Å^2) of the nearest of 27 images of the fractional offset f, those left out whose
// component on an axis alone (reach: distance over the perpendicular widths) exceeds what is asked for:
// with a reach below half a cell that leaves an axis's nearest image alone.
__device__ inline double image_dist2(const FwDesc &F, double f0, double f1, double f2, double reach0, double reach1,
                                     double reach2)
{
    f0 -= __builtin_rint(f0);
    f1 -= __builtin_rint(f1);
    f2 -= __builtin_rint(f2);
    double best = INFINITY;
    const int n0 = reach0 < 0.5 ? 0 : 1, n1 = reach1 < 0.5 ? 0 : 1, n2 = reach2 < 0.5 ? 0 : 1;
    for (int s2 = -n2; s2 <= n2; ++s2) {
        const double g2 = f2 + s2;
        if (fabs(g2) > reach2) continue;
        for (int s1 = -n1; s1 <= n1; ++s1) {
            const double g1 = f1 + s1;
            if (fabs(g1) > reach1) continue;
            for (int s0 = -n0; s0 <= n0; ++s0) {
                const double g0 = f0 + s0;
                if (fabs(g0) <= reach0) best = fmin(best, length2(F.A, g0, g1, g2));
            }
        }
    }
    return best;
}

// One wavefront per bin. FILL: writes the entries at the bin's offset, else counts them.
template <bool FILL>
__global__ __launch_bounds__(256) void near_kernel(NearBuild a)
{
    const int lane = threadIdx.x & 63, b = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (b >= a.nbins) return;
    int lo = 0, hi = a.nfw - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.bin_fw[mid] <= b) lo = mid; else hi = mid - 1;
    }
    const int u = __builtin_amdgcn_readfirstlane(lo);
    const FwDesc &F = a.fw[u];
    const NearDesc D = a.nd[u];
    const int local = b - a.bin_fw[u];
    const int bx = local % D.nb[0], by = (local / D.nb[0]) % D.nb[1], bz = local / (D.nb[0] * D.nb[1]);
    const double c0 = (bx + 0.5) / D.nb[0], c1 = (by + 0.5) / D.nb[1], c2 = (bz + 0.5) / D.nb[2];
    const double R = __builtin_sqrt(D.r2);
    const double4 *run = a.run + a.run_off[u];
    const int nrun = a.run_off[u + 1] - a.run_off[u];
    // the atoms close to the bin come first, so that a caller that tests for overlaps finds them among
    // the first entries: where the next one of either kind goes, or how many there are
    int close = FILL ? a.start[b] : 0, others = FILL ? close + a.close[b] : 0;
    for (int q0 = 0; q0 < nrun; q0 += 64) {
        // 64 runs at once, one per lane: whether an atom of the run can be within R. A run wider than
        // the 27 images are sure to cover (an offset of up to a whole cell) is taken as it is.
        bool cand = false;
        if (q0 + lane < nrun) {
            const double4 c = run[q0 + lane];
            const double lim = R + c.w, k = lim / R * (1.0 + 1.0e-9);
            const double r0 = D.reach[0] * k, r1 = D.reach[1] * k, r2 = D.reach[2] * k;
            cand = fmax(r0, fmax(r1, r2)) > 1.0 ||
                   image_dist2(F, c.x - c0, c.y - c1, c.z - c2, r0, r1, r2) <= lim * lim * (1.0 + 1.0e-9);
        }
        for (uint64_t todo = __builtin_amdgcn_ballot_w64(cand); todo; todo &= todo - 1) {
            const int j = (q0 + __builtin_ctzll(todo)) * 64 + lane;
            double best = INFINITY;
            if (j < F.natoms) {
                const double4 h = a.atomf[F.atom_off + j];
                best = image_dist2(F, h.x - c0, h.y - c1, h.z - c2, D.reach[0], D.reach[1], D.reach[2]);
            }
            const bool in = best <= D.r2;
            const uint64_t mask = __builtin_amdgcn_ballot_w64(in), near = __builtin_amdgcn_ballot_w64(in && best <= D.close2);
            if (FILL && in) {
                const uint64_t below = (1ull << lane) - 1ull;
                const int at = (near >> lane) & 1 ? close + __popcll(near & below) : others + __popcll(mask & ~near & below);
                a.ent[at] = (uint32_t)j | ((uint32_t)a.atype[F.atom_off + j] << NEAR_TYPE_SHIFT);
            }
            close += __popcll(near);
            others += __popcll(mask & ~near);
        }
    }
    if (!FILL && lane == 0) {
        a.close[b] = close;
        a.start[b] = close + others;
        if (b + 1 == a.nbins) a.start[b + 1] = 0;  // the slot past the last bin
    }
}

hipError_t launch_near_runs(const NearBuild &a, hipStream_t st)
{
    if (a.nruns <= 0) return hipSuccess;
    hipLaunchKernelGGL(near_run_kernel, dim3((unsigned)((a.nruns + 3) / 4)), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_near_build(bool fill, const NearBuild &a, hipStream_t st)
{
    const dim3 grid((unsigned)((a.nbins + 3) / 4)), block(256);
    if (fill) hipLaunchKernelGGL(near_kernel<true>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(near_kernel<false>, grid, block, 0, st, a);
    return hipGetLastError();
}

// The near lists' bins of every framework, and what their kernels share. False: the batch has none, since a
// framework has more atoms than an entry can name, or the lists would not fit.
bool near_bins(const pa_batch *b, NearBuild &a, std::vector<NearDesc> &nd, std::vector<int> &bin_fw, std::vector<int> &run_off)
{
    const double rcmax = std::max(b->rc_lj, b->gdev.charged ? b->rc_ew : 0.0);
    nd.resize(b->nfw);
    bin_fw.assign(b->nfw + 1, 0);
    run_off.assign(b->nfw + 1, 0);
    for (int u = 0; u < b->nfw; ++u) {
        if (b->desc[u].natoms >= (1 << NEAR_TYPE_SHIFT)) return false;
        run_off[u + 1] = run_off[u] + (b->desc[u].natoms + 63) / 64;
    }
    for (double edge = NEAR_EDGE;; edge *= 1.26) {
        if (edge > 1000.0) return false;
        double entries = 0.0;
        int64_t nbins = 0;
        for (int u = 0; u < b->nfw; ++u) {
            const FwHost &h = b->info[u];
            const FwDesc &F = b->desc[u];
            NearDesc &D = nd[u];
            for (int d = 0; d < 3; ++d) D.nb[d] = std::max(1, std::min(512, (int)std::ceil(h.perp[d] / edge)));
            double rb = 0.0;  // circumradius: half the longest body diagonal
            for (int sy = -1; sy <= 1; sy += 2)
                for (int sz = -1; sz <= 1; sz += 2) {
                    const double f[3] = {0.5 / D.nb[0], 0.5 * sy / D.nb[1], 0.5 * sz / D.nb[2]};
                    double v[3];
                    matvec(F.A, f, v);
                    rb = std::max(rb, std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]));
                }
            const double R = rcmax + b->r_guest + rb + 1.0e-6;
            D.r2 = R * R;
            D.close2 = (rb + b->r_guest + 2.0) * (rb + b->r_guest + 2.0);
            for (int d = 0; d < 3; ++d) D.reach[d] = R / h.perp[d] * (1.0 + 1.0e-9);
            D.bin_off = (int)nbins;
            bin_fw[u] = (int)nbins;
            const int64_t n = (int64_t)D.nb[0] * D.nb[1] * D.nb[2];
            nbins += n;
            entries += (double)n * std::min<double>(F.natoms, F.natoms / h.volume * (4.0 / 3.0) * PI * R * R * R);
        }
        // an atom is in at most ((R + rb) / R)^3 < 8 times as many lists as the volume of its sphere
        // holds bins, so that lists of 2^28 entries by volume have offsets below 2^31
        if (entries > NEAR_MAX_ENTRIES || nbins >= (1 << 26)) continue;
        bin_fw[b->nfw] = (int)nbins;
        a.nfw = b->nfw;
        a.nbins = (int)nbins;
        a.nruns = run_off[b->nfw];
        return true;
    }
}

NearLists near_lists(const pa_batch *b)
{
    return NearLists{b->d_nearf.as<double4>(), b->d_near_desc.as<NearDesc>(), b->d_near_start.as<int>(),
                     b->d_near_ent.as<uint32_t>()};
}

}  // namespace pa
