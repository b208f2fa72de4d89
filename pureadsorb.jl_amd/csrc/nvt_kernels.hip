// nvt_kernels.hip -- test-particle insertions into the chains' current configurations on gfx950
// (widom_chain_kernel!, src/nvt.jl:85-119), FP64.
//
// The energy of an insertion at pose (p, q) into system s holding guests G:
//   host-guest real space (LJ + KE q q' erfc(alpha r)/r, minimum image per site pair)
//   + KE * 2 sum_k kpref_k Re(conj(S_k) S_g,k)    against the chain's running S (host + G)
//   + guest-guest real space against every live guest of G
// (the host adds insertion_constant_term, src/nvt.jl:44-66).
//
// One wavefront per insertion:
//   * host-guest: the near list of the insertion's bin (batch_kernels.hip), pairs inside the cutoff
//     queued in LDS and evaluated 64 at a time;
//   * reciprocal: the chain's k-vectors in the order of the move kernel (KRuns), one run of
//     consecutive n3 per lane, walked from its middle. The pair m +- j of a run whose middle has
//     the phase x = e^{2 pi i (n1 f1 + n2 f2 + m f3)} adds, with z = e^{2 pi i j f3} and the
//     snapshot's c = kprefactor S,
//       x_r [z_r (c+_r + c-_r) + z_i (c+_i - c-_i)] + x_i [z_r (c+_i + c-_i) + z_i (c-_r - c+_r)],
//     so the brackets are summed over j first: 4 fused multiply-adds per site for two k-vectors
//     (a recurrence with one complex product per k-vector and site took 8 each). Phases come from
//     per-axis tables in LDS, or are evaluated where they are used in a cell so long that LDS does not
//     hold its tables;
//   * guest-guest: lanes take (guest, site) pairs against every site, through the same queue.
// The pose is drawn exactly as the Widom path draws it, `per` insertions of a wavefront one per
// lane; the energy terms use fused multiply-adds. FP64 issue bounds
// it: 40,960 insertions into RUBTAK 3x3x3 with some 30 CO2 take 0.67 ms (1.35 ms before).
#include "pa_device.hpp"

namespace pa {

constexpr int CW_NW = 4;
constexpr int CW_BATCH = 16;  // insertions of one wavefront

// Guests of up to three sites fit 4 wavefronts per SIMD without spilling; larger guests keep
// the compiler's own register budget. TAB: the phases come from tables in LDS.
template <int NS, bool UPPER, bool TAB>
__global__ __launch_bounds__(64 * CW_NW, (NS <= 3 ? 4 : 1)) void chain_widom_kernel(ChainWidomArgs a, int per)
{
    __shared__ PairRing rings[CW_NW];
    __shared__ double wf[CW_NW][CW_BATCH][3 * NS];
    __shared__ int wsys[CW_NW][CW_BATCH], wbin[CW_NW][CW_BATCH];
    extern __shared__ double2 tabs[];  // per wavefront, with charges: (ktab_w x NS) phases e^{2 pi i m f_d}
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwv = blockDim.x >> 6;
    const int64_t first = ((int64_t)blockIdx.x * nwv + wv) * per;
    if (first >= a.nitems) return;  // whole wavefront; the kernel has no barrier
    const int cnt = (int)(a.nitems - first < per ? a.nitems - first : per);
    const GuestDev &G = a.guest;
    const ChainSnap &S = a.snap;
    if (lane < cnt) {
        const int64_t item = first + lane;
        int lo = 0, hi = a.nsys - 1;
        while (lo < hi) {  // system of the item: item_off[s] <= item < item_off[s+1]
            const int mid = (lo + hi + 1) >> 1;
            if (a.item_off[mid] <= item) lo = mid; else hi = mid - 1;
        }
        const int u = a.fw_of[lo];
        const FwDesc &F = a.fw[u];
        double pos[3], q[4], pf[3];
        if (a.pose_pos) {
            for (int d = 0; d < 3; ++d) pos[d] = a.pose_pos[3 * item + d];
            for (int d = 0; d < 4; ++d) q[d] = a.pose_quat[4 * item + d];
        } else {
            double f[3];
            pose_uniforms(a.widom_seed, lo, a.cyc0 * a.nw + (item - a.item_off[lo]), f, q);
            matvec(F.A, f, pos);
        }
        matvec(F.invA, pos, pf);
        for (int t = 0; t < NS; ++t) {
            double r[3], x[3], f[3];
            rotate(q, G.site[t], r);
            for (int d = 0; d < 3; ++d) x[d] = pos[d] + r[d];
            matvec(F.invA, x, f);
            for (int d = 0; d < 3; ++d) wf[wv][lane][3 * t + d] = f[d];
        }
        wsys[wv][lane] = lo;
        wbin[wv][lane] = near_bin(a.near.desc[u], pf);
    }
    auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    fence();
    double2 *tab = tabs + (size_t)wv * NS * a.ktab_w;
    PairQueue Q(rings[wv], lane);
#pragma unroll 1
    for (int i = 0; i < cnt; ++i) {
        const int s = __builtin_amdgcn_readfirstlane(wsys[wv][i]), bin = __builtin_amdgcn_readfirstlane(wbin[wv][i]);
        const int u = a.fw_of[s];
        const FwDesc &F = a.fw[u];
        // the state this insertion sees: the snapshot of its cycle slot
        const int64_t cl = (first + i - a.item_off[s]) / a.nw;
        const int64_t slot = cl < a.snap_n ? cl : a.snap_n - 1;
        const int gr0 = a.guest_off[s], occ = S.occ[slot * S.nsys + s];
        double f[NS][3];
#pragma unroll
        for (int t = 0; t < NS; ++t)
            for (int d = 0; d < 3; ++d) f[t][d] = wf[wv][i][3 * t + d];
        double e = 0.0;
        const double alpha = F.alpha;
        auto eval = [&](double r2, double qq, int code) {
            const double2 p = a.pair64[code];
            e += cw_pair(r2, p.x * p.x, 4.0 * p.y, qq, alpha, a.rc_lj2, a.rc_ew2);
        };
        // (1) host-guest real space
        near_scan<NS, UPPER>(a.near, F.atom_off, F.A, bin, f, G.q, a.ntypes_c, a.rc_max2, nullptr, Q, eval);
        // (2) guest-guest real space
        const double4 *gpos = S.pos + slot * S.nslots + gr0, *gquat = S.quat + slot * S.nslots + gr0;
#pragma unroll 1
        for (int xb = 0; xb < occ * NS; xb += 64) {
            const int x = xb + lane, jj = x / NS, sb = x - jj * NS;
            const double nan = __builtin_nan("");
            double fb[3] = {nan, nan, nan};
            if (x < occ * NS) {
                const double4 p4 = gpos[jj], q4 = gquat[jj];
                const double qj[4] = {q4.x, q4.y, q4.z, q4.w};
                double r[3];
                rotate(qj, G.site[sb], r);
                const double pb[3] = {p4.x + r[0], p4.y + r[1], p4.z + r[2]};
                matvec(F.invA, pb, fb);
            }
            const double qb = KE * G.q[sb];
            const int tb = G.type[sb];
#pragma unroll
            for (int s0 = 0; s0 < NS; s0 += 3) {
#pragma unroll
                for (int sa = s0; sa < (s0 + 3 < NS ? s0 + 3 : NS); ++sa) {
                    const double r2 = cw_r2_t<UPPER>(F.A, f[sa][0] - fb[0], f[sa][1] - fb[1], f[sa][2] - fb[2]);
                    Q.push(r2 < a.rc_max2, r2, G.q[sa] * qb, sa * a.ntypes_c + tb);
                }
#pragma unroll 1
                while (Q.pending() >= 64) Q.drain(64, eval);
            }
        }
        Q.drain(Q.pending(), eval);
        // (3) reciprocal cross term
        if (G.charged) {
            const int m0 = F.kn_max[0] + 1, m1 = F.kn_max[1] + 1, tw = m0 + m1 + F.kn_max[2] + 1;
            if constexpr (TAB) {
                const float inv_tw = 1.0f / (float)tw;
#pragma unroll 1
                for (int x = lane; x < NS * tw; x += 64) {
                    const int t = (int)(((float)x + 0.5f) * inv_tw), c = x - t * tw;
                    const int d = c < m0 ? 0 : (c < m0 + m1 ? 1 : 2);
                    tab[c * NS + t] = axis_power_const(wf[wv][i][3 * t + d], c - (d == 0 ? 0 : (d == 1 ? m0 : m0 + m1)));
                }
                fence();
            }
            // e^{2 pi i m f_d} of site t, the table's row `at` of axis d
            auto phase = [&](const double2 *at, int d, int m, int t) {
                if constexpr (TAB) return at[t];
                else return axis_power_const(wf[wv][i][3 * t + d], m);
            };
            const int4 *runs = a.kr.run + a.kr.run_off[u];
            const int nruns = a.kr.run_off[u + 1] - a.kr.run_off[u];
            // c = kprefactor S through buffer loads: zero past the end, for lanes without a k-vector
            const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(S.csk + slot * S.ctot + S.coff[s]), (short)0, F.nk * 16, 0x00020000);
            auto load = [&](int p, int n) {
                const uint32_t at = lane < n ? (uint32_t)(p + lane) : 0x07FFFFFFu;
                return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rc, (int)(at * 16u), 0, 0));
            };
            double acc = 0.0;
            int pos = 0;
#pragma unroll 1
            for (int r0 = 0; r0 < nruns; r0 += 64) {
                const int4 run = r0 + lane < nruns ? runs[r0 + lane] : make_int4(0, 0, 0, 0);
                const int L = run.w;
                auto count = [&](int l) { return (int)__popcll(__builtin_amdgcn_ballot_w64(L >= l)); };
                const int n0 = count(1);
                const double2 c0 = load(pos, n0);
                pos += n0;
                int np = count(2), nm = count(3);
                double2 cp = load(pos, np), cm = load(pos + np, nm);
                double v1[NS], v2[NS];
#pragma unroll
                for (int t = 0; t < NS; ++t) {
                    v1[t] = c0.x;
                    v2[t] = c0.y;
                }
                const double2 *tj = tab + (m0 + m1 + 1) * NS;
#pragma unroll 1
                for (int j = 2; np > 0; ++j) {
                    double2 z[NS];
#pragma unroll
                    for (int t = 0; t < NS; ++t) z[t] = phase(tj, 2, j - 1, t);
                    tj += NS;
                    pos += np + nm;
                    np = count(2 * j);
                    nm = count(2 * j + 1);
                    const double2 cp2 = load(pos, np), cm2 = load(pos + np, nm);
                    __builtin_amdgcn_sched_barrier(0);
                    const double P = cp.x + cm.x, T = cp.y + cm.y, R = cp.y - cm.y, N = cm.x - cp.x;
#pragma unroll
                    for (int t = 0; t < NS; ++t) {
                        v1[t] = __builtin_fma(z[t].x, P, __builtin_fma(z[t].y, R, v1[t]));
                        v2[t] = __builtin_fma(z[t].x, T, __builtin_fma(z[t].y, N, v2[t]));
                    }
                    cp = cp2;
                    cm = cm2;
                }
                const double2 *tx = tab + abs(run.x) * NS, *ty = tab + (m0 + abs(run.y)) * NS,
                              *tz = tab + (m0 + m1 + abs(run.z)) * NS;
#pragma unroll
                for (int t = 0; t < NS; ++t) {
                    const double2 x = cis_from_axes(phase(tx, 0, abs(run.x), t), phase(ty, 1, abs(run.y), t),
                                                    phase(tz, 2, abs(run.z), t), run.x, run.y, run.z);
                    acc = __builtin_fma(G.q[t], __builtin_fma(x.x, v1[t], x.y * v2[t]), acc);
                }
            }
            e = __builtin_fma(2.0 * KE, acc, e);
            fence();
        }
        e = wave_sum63(e);
        if (lane == 63) a.dU[first + i] = e;
    }
}

// Snapshot slot `slot` of every system's live state (after an audit, or for insertions at
// caller poses): one workgroup per system.
__global__ __launch_bounds__(256) void chain_snapshot_kernel(ChainSnap S, int64_t slot, const FwDesc *fw,
                                                            const int *fw_of, const double *kw_all, const int *guest_off,
                                                            const int *sk_off, const int *occupancy,
                                                            const double4 *refpos, const double4 *quat,
                                                            const double2 *Sk)
{
    const int n = blockIdx.x, tid = threadIdx.x;
    const FwDesc &F = fw[fw_of[n]];
    const double *kw = kw_all + F.k_off;
    const double2 *sk = Sk + sk_off[n];
    double2 *dsk = S.csk + slot * S.ctot + S.coff[n];
    for (int k = tid; k < F.nk; k += 256) {
        const double w = kw[k];
        const double2 v = sk[k];
        dsk[k] = make_double2(w * v.x, w * v.y);
    }
    const int gr0 = guest_off[n], occ = occupancy[n];
    for (int i = tid; i < occ; i += 256) {
        S.pos[slot * S.nslots + gr0 + i] = refpos[gr0 + i];
        S.quat[slot * S.nslots + gr0 + i] = quat[gr0 + i];
    }
    if (tid == 0) S.occ[slot * S.nsys + n] = occ;
}

hipError_t launch_chain_snapshot(const ChainSnap &S, int64_t slot, const McArgs &m, hipStream_t st)
{
    hipLaunchKernelGGL(chain_snapshot_kernel, dim3((unsigned)S.nsys), dim3(256), 0, st, S, slot, m.fw, m.fw_of, m.kr.kw,
                       m.guest_off, m.sk_off, m.occupancy, m.refpos, m.quat, m.Sk);
    return hipGetLastError();
}

template <int NS>
static void launch_chain_widom_ns(const ChainWidomArgs &a, int per, int nwv, bool tab, hipStream_t st)
{
    const dim3 grid((unsigned)(((a.nitems + per - 1) / per + nwv - 1) / nwv)), block((unsigned)(64 * nwv));
    const size_t lds = a.guest.charged ? sizeof(double2) * nwv * NS * a.ktab_w : 0;
    if (!tab) hipLaunchKernelGGL((chain_widom_kernel<NS, false, false>), grid, block, 0, st, a, per);
    else if (a.upper) hipLaunchKernelGGL((chain_widom_kernel<NS, true, true>), grid, block, lds, st, a, per);
    else hipLaunchKernelGGL((chain_widom_kernel<NS, false, true>), grid, block, lds, st, a, per);
}

hipError_t launch_chain_widom(const ChainWidomArgs &a, hipStream_t st)
{
    if (a.nitems <= 0) return hipSuccess;
    // the wavefronts of a workgroup share nothing: one where the phase tables of four would not fit, and
    // no tables where one wavefront's would not (a six-site guest in a cell of 3,300 Å)
    const size_t bytes = a.guest.charged ? sizeof(double2) * a.guest.nsites * a.ktab_w : 0;
    const bool tab = bytes <= 100 * 1024;
    const int nwv = tab && CW_NW * bytes > 100 * 1024 ? 1 : CW_NW;
    // insertions per wavefront: one until there are some 16 wavefronts for every SIMD
    int per = 1;
    while (per < CW_BATCH && a.nitems / (2 * per) >= 16384) per *= 2;
    switch (a.guest.nsites) {
    case 1: launch_chain_widom_ns<1>(a, per, nwv, tab, st); break;
    case 2: launch_chain_widom_ns<2>(a, per, nwv, tab, st); break;
    case 3: launch_chain_widom_ns<3>(a, per, nwv, tab, st); break;
    case 4: launch_chain_widom_ns<4>(a, per, nwv, tab, st); break;
    case 5: launch_chain_widom_ns<5>(a, per, nwv, tab, st); break;
    case 6: launch_chain_widom_ns<6>(a, per, nwv, tab, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace pa
