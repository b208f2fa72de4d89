// batch_kernels.hip -- FrameworkBatch tables on gfx950: the host structure factor at the
// k-vectors a framework keeps (src/batch.jl:173-195) and the 64-orientation guest self term
// over its full k table (src/batch.jl:360-389), both FP64, and the phase-0 near-stencil atom
// lists. k = 2 pi A^-T n, so e^{i k.r} = e^{2 pi i n.f}
// with f = A^-1 r; every phase is one own-sincospi of 2 n.f.
#include <hipcub/hipcub.hpp>

#include "pa_device.hpp"

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

// Phase-0 near lists: for every hard-core cell, the atoms within nbr_r of any point of it, by their
// minimum-image distance to the cell's centre. One wavefront per cell, its lanes over the cells
// within nbr_reach (each once where the reach goes around the axis). Without FILL the lists are
// counted into nbr_start; with it they are written in three shells of growing distance, so that
// an insertion's overlap is usually found among the first entries. cell_fw_off (nfw + 1) maps the
// global cell index to its framework.
template <bool FILL>
__global__ __launch_bounds__(BK_WG) void nbr_kernel(const FwDesc *fw, int nfw, const int *cell_fw_off, int ncells,
                                                   const int *cell_start, int *nbr_start, const uint4 *corefx,
                                                   uint4 *nbr_atoms)
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
    const float shell[4] = {-1.0f, 0.36f * D.nbr_thr2, 0.64f * D.nbr_thr2, D.nbr_thr2};
    int total = 0;
    const int64_t at0 = FILL ? nbr_start[D.cg_off + c] : 0;
    for (int sh = 0; sh < (FILL ? 3 : 1); ++sh)
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
                bool in = false;
                uint4 at = make_uint4(0u, 0u, 0u, 0u);
                if (j < len) {
                    at = src[b0 + j];
                    const float dx = (float)(int32_t)(x[0] - at.x), dy = (float)(int32_t)(x[1] - at.y),
                                dz = (float)(int32_t)(x[2] - at.z);
                    const float ex = D.Af[0] * dx + D.Af[3] * dy + D.Af[6] * dz;
                    const float ey = D.Af[1] * dx + D.Af[4] * dy + D.Af[7] * dz;
                    const float ez = D.Af[2] * dx + D.Af[5] * dy + D.Af[8] * dz;
                    const float r2 = ex * ex + ey * ey + ez * ez;
                    in = FILL ? r2 > shell[sh] && r2 <= shell[sh + 1] : r2 <= D.nbr_thr2;
                }
                const uint64_t m = __builtin_amdgcn_ballot_w64(in);
                if (FILL && in) nbr_atoms[at0 + total + __popcll(m & ((1ull << lane) - 1ull))] = at;
                total += __popcll(m);
            }
        }
    if (!FILL && lane == 0) nbr_start[D.cg_off + c] = total;
    // the slot past a framework's last cell: no atoms
    if (!FILL && lane == 0 && g + 1 == cell_fw_off[lo + 1]) nbr_start[D.cg_off + c + 1] = 0;
}

// Exclusive scan of n counts in place (tmp == nullptr: only the temporary size).
hipError_t scan_counts(int *counts, int n, void *tmp, size_t *tmp_bytes, hipStream_t st)
{
    return hipcub::DeviceScan::ExclusiveSum(tmp, *tmp_bytes, counts, counts, n, st);
}

hipError_t launch_nbr(bool fill, const FwDesc *fw, int nfw, const int *cell_fw_off, int ncells, const int *cell_start,
                      int *nbr_start, const uint4 *corefx, uint4 *nbr_atoms, hipStream_t st)
{
    if (ncells <= 0) return hipSuccess;
    const dim3 grid((unsigned)((ncells + BK_WG / 64 - 1) / (BK_WG / 64))), block(BK_WG);
    if (fill)
        hipLaunchKernelGGL(nbr_kernel<true>, grid, block, 0, st, fw, nfw, cell_fw_off, ncells, cell_start, nbr_start,
                           corefx, nbr_atoms);
    else
        hipLaunchKernelGGL(nbr_kernel<false>, grid, block, 0, st, fw, nfw, cell_fw_off, ncells, cell_start, nbr_start,
                           corefx, nbr_atoms);
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

}  // namespace pa
