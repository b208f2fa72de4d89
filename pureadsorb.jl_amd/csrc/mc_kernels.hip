// mc_kernels.hip -- the move-energy path (NVT and μVT Monte Carlo moves) on gfx950.
//
// One workgroup per chain runs that chain's move attempts back to back, so a run of many
// moves costs one launch instead of the reference's three launches per move
// (src/moves.jl:577-645). The random part of 64 attempts at a time is drawn with one attempt per
// lane from the chain's counter-based stream (select_and_propose, src/moves.jl:275-288). Four
// wavefronts evaluate an attempt, splitting the three sums a move needs across their lanes:
//   * the new pose's host-guest real-space energy over the framework atoms near it
//     (host_guest_realspace_energy_range, src/guest.jl:176-200; batch_kernels.hip), pairs inside the cutoff
//     compacted through LDS before the LJ + erfc evaluation (fused multiply-adds, FP64),
//   * the guest-guest real-space change over (other guest, site) pairs against the sites of the
//     old and the new pose (guest_guest_move_delta / guest_pair_realspace_energy_range,
//     src/guest.jl:112-156), from the live guests' site positions, pairs inside the cutoff
//     compacted the same way,
//   * the reciprocal change over the k-vectors against the running structure factor
//     (_reciprocal_move_delta_k, src/guest.jl:228-238), evaluated again for the update on
//     acceptance;
// reduces them through LDS, and every wavefront takes the same Metropolis decision
// (src/moves.jl:198-246). Work-item 0 commits poses and occupancy; the workgroup applies the
// changes to the running structure factor. Everything is FP64.
#include "pa_device.hpp"

namespace pa {

constexpr int MC_BATCH = 64;           // attempts whose random part is drawn at once

// Minimum-image squared distance between two points of the cell, minimum_image's operations.
// UPPER drops the products with the exact zeros of an upper-triangular cell and its inverse,
// which leaves every bit unchanged.
template <bool UPPER>
__device__ inline double mi_r2(const double *A, const double *I, const double a[3], const double b[3])
{
#pragma clang fp contract(off)
    const double d[3] = {a[0] - b[0], a[1] - b[1], a[2] - b[2]};
    double m[3];
    if (UPPER) {
        const double r0 = __builtin_rint(I[0] * d[0] + I[3] * d[1] + I[6] * d[2]);
        const double r1 = __builtin_rint(I[4] * d[1] + I[7] * d[2]);
        const double r2 = __builtin_rint(I[8] * d[2]);
        m[0] = d[0] - (A[0] * r0 + A[3] * r1 + A[6] * r2);
        m[1] = d[1] - (A[4] * r1 + A[7] * r2);
        m[2] = d[2] - A[8] * r2;
    } else {
        minimum_image(A, I, d, m);
    }
    return m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
}

// The random part of MC_BATCH attempts: move type, slot word, log of the acceptance uniform, and by
// type three normals, the turning quaternion, or a position and an orientation.
struct McDraws {
    int movetype;              // of every attempt, or 0: drawn from the cumulative probabilities
    double pcum[NMOVES], step_rot;
    int type[MC_BATCH];
    uint64_t slot[MC_BATCH];
    double lu[MC_BATCH], v[7][MC_BATCH];
};

// Draws the attempts from `first` on, one per lane of one wavefront: they depend on the attempt's
// counter alone. Not inlined, so that the constants of log, acos, sin and cos take no registers in
// the loop over rounds, which calls it once in 60 attempts.
__device__ __attribute__((noinline)) void mc_draw(uint64_t seed, uint64_t first, const double *cA, McDraws &D)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const uint64_t at = first + (uint64_t)lane;
    int type = D.movetype;
    if (type == 0) {
        Chain r1(seed, at, 1);
        const double v = unit_f64(r1.next());
        type = NMOVES;
        for (int i = NMOVES - 1; i >= 0; --i)
            if (v < D.pcum[i]) type = i + 1;
    }
    Chain rng(seed, at, 0);
    D.type[lane] = type;
    if (type != MOVE_INSERTION) D.slot[lane] = rng.next();
    if (type == MOVE_TRANSLATION) {
        for (int d = 0; d < 3; ++d) D.v[d][lane] = rand_normal(rng);
    } else if (type == MOVE_ROTATION) {
        double qr[4], qp[4];
        rand_quaternion(rng, qr);
        quaternion_pow(qr, D.step_rot, qp);
        for (int i = 0; i < 4; ++i) D.v[i][lane] = qp[i];
    } else if (type == MOVE_REINSERTION || type == MOVE_INSERTION) {
        double f[3], p[3], q[4];
        for (int d = 0; d < 3; ++d) f[d] = unit_f64(rng.next());
        matvec(cA, f, p);
        rand_quaternion(rng, q);
        for (int d = 0; d < 3; ++d) D.v[d][lane] = p[d];
        for (int i = 0; i < 4; ++i) D.v[3 + i][lane] = q[i];
    }
    D.lu[lane] = log(unit_f64(rng.next()));
}

// Speculative rounds: the workgroup holds SPEC groups of GNW wavefronts; group g evaluates attempt
// ctr + g against the state at the start of the round. Every attempt's proposal and acceptance
// draw come from its own counter (ChainRNG(chain seed, attempt, 0)), so until the first accepted
// attempt of the round each one is exactly what a sequential chain would evaluate: the round
// commits its first accepted attempt (if any), keeps the decisions of the attempts before it and
// discards the rest, which the next round evaluates again.
template <int NS, bool UPPER, int SPEC, int GNW>
__global__ __launch_bounds__(SPEC *GNW * 64) void mc_chain_kernel(McArgs a)
{
#pragma clang fp contract(off)
    constexpr int GW = 64 * GNW, WG = SPEC * GW, NW = SPEC * GNW;  // work-items and wavefronts
    __shared__ double red[2][NW];
    __shared__ PairRing rings[NW];
    // the round's attempts: type, slot, bin of the new pose's near list, log of the acceptance
    // uniform, cached host energy of the slot, proposed pose, and the sites of the old (0) and the
    // new (1) pose
    __shared__ int at_type[SPEC], at_slot[SPEC], at_bin[SPEC];
    __shared__ double at_lu[SPEC], at_he[SPEC], at_p[SPEC][3], at_q[SPEC][4];
    __shared__ double at_site[SPEC][2][NS][3], at_frac[SPEC][2][NS][3];
    __shared__ McDraws draws;  // attempts pbase .. pbase + MC_BATCH - 1
    // cell, inverse cell and guest, read from LDS so that no loop holds them in registers
    __shared__ double cA[9], cI[9], g_site[NS][3], g_q[NS];
    __shared__ int cnt_acc[NMOVES], cnt_att[NMOVES];
    // per-axis phase tables of the attempts' old and new sites: e^{2 pi i m f_d}, m = 0..kn_max[d]
    // (SPEC x 2 x NS x ktab_w with charges), then (sigma^2, 4 eps) of every (site, framework
    // type) and of every (site, site) pair, and KE q q' of the latter
    extern __shared__ double2 ktab[];
    // arguments of the rare paths (samples, snapshots, trace), read where they are used: held in
    // scalar registers over the whole loop they spill
    auto rare = []() {
        auto p = (__attribute__((address_space(4))) const McArgs *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(p));
        return p;
    };
    const int n = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gi = wid / GNW, gw = wid - gi * GNW, gt = tid - gi * GW;
    const int u = a.fw_of[n];
    const FwDesc &F = a.fw[u];
    const int gr0 = a.guest_off[n], cap = a.guest_off[n + 1] - gr0, nslots = a.guest_off[a.nsys];
    const double *kw = a.kr.kw + F.k_off;
    const int4 *runs = a.kr.run + a.kr.run_off[u];
    const int *kbase = a.kr.base + a.kr.blk_off[u];
    const int nruns = a.kr.run_off[u + 1] - a.kr.run_off[u], nkblk = a.kr.blk_off[u + 1] - a.kr.blk_off[u];
    double2 *Sk = a.Sk + a.sk_off[n];
    const int nk = F.nk;
    const bool charged = a.guest.charged;
    const double alpha = F.alpha;

    // chain scalars: identical copies in every work-item (every decision is taken by all)
    int occ = a.occupancy[n];
    double E = a.energy[n], Eabs = a.energy_abs[n], skabs = a.sk_abs[n];
    uint64_t ctr = a.rng_counter[n];
    const uint64_t seed = a.rng_seed[n];
    int maxocc = a.max_occ ? a.max_occ[n] : 0;
    int caphit = 0;
    int64_t ntrace = 0;
    const bool traced = a.trace != nullptr;
    const double log_fugV = a.log_fugV ? a.log_fugV[n] : 0.0;
    const double cp = a.const_p ? a.const_p[n] : 0.0, cq = a.const_q ? a.const_q[n] : 0.0;

    const int m0 = F.kn_max[0] + 1, m1 = F.kn_max[1] + 1, tw = m0 + m1 + F.kn_max[2] + 1;
    const float inv_tw = 1.0f / (float)tw;
    double2 *ptab = ktab + (charged ? (size_t)SPEC * 2 * NS * a.ktab_w : 0);
    const int gg0 = NS * a.ntypes_c;
    double *qgg = (double *)(ptab + gg0 + NS * NS);
    for (int i = tid; i < gg0; i += WG) {
        const double2 p = a.pair64[i];
        ptab[i] = make_double2(p.x * p.x, 4.0 * p.y);
    }
    for (int i = tid; i < NS * NS; i += WG) {
        const double2 p = a.pair64[(i / NS) * a.ntypes_c + a.guest.type[i % NS]];
        ptab[gg0 + i] = make_double2(p.x * p.x, 4.0 * p.y);
        qgg[i] = KE * a.guest.q[i / NS] * a.guest.q[i % NS];
    }
    if (tid < 9) {
        cA[tid] = F.A[tid];
        cI[tid] = F.invA[tid];
    }
    if (tid < NS) {
        for (int d = 0; d < 3; ++d) g_site[tid][d] = a.guest.site[tid][d];
        g_q[tid] = a.guest.q[tid];
    }
    if (tid < NMOVES) {
        cnt_acc[tid] = cnt_att[tid] = 0;
        draws.pcum[tid] = a.pcum[tid];
    }
    if (tid == 0) {
        draws.movetype = a.mode == 0 ? a.movetype : 0;
        draws.step_rot = a.step_rot ? a.step_rot[n] : 0.0;
    }
    __syncthreads();
    double ds_bound = 0.0;
    for (int s = 0; s < NS; ++s) ds_bound += fabs(g_q[s]);
    ds_bound *= 2.0;
    // positions of the live guests' sites, kept up to date by the commits
    double4 *gsite = a.gsite + (size_t)gr0 * NS;
    auto site_of = [&](const double p[3], const double q[4], int t, double out[3]) {
        double r[3];
        rotate(q, g_site[t], r);
        for (int d = 0; d < 3; ++d) out[d] = p[d] + r[d];
    };
    for (int i = tid; i < occ * NS; i += WG) {
        const double4 p4 = a.refpos[gr0 + i / NS], q4 = a.quat[gr0 + i / NS];
        const double p[3] = {p4.x, p4.y, p4.z}, q[4] = {q4.x, q4.y, q4.z, q4.w};
        double x[3];
        site_of(p, q, i % NS, x);
        gsite[i] = make_double4(x[0], x[1], x[2], 0.0);
    }
    __syncthreads();

    // Visits the k-vectors' structure-factor changes of one attempt (its phase tables at `tab`):
    // use(position, loaded, Re dS, Im dS), `loaded` being load(position) issued a step ahead; a
    // lane without a k-vector gets position KNONE. The blocks of 64 runs are dealt in snake order
    // (they get shorter) to nw / SPLIT teams of SPLIT wavefronts, which take every SPLIT-th step of
    // a block. One complex product of table entries per run and site starts a block; a pair of
    // k-vectors m +- j then takes 4 fused multiply-adds per site and pose for both. Per k-vector
    // that is 12 FP64 instructions for a 3-site guest's old and new pose, where two complex
    // products per site and k-vector took about 120. The tables interleave poses and sites, so
    // that a step's entries are neighbours, and the scheduling barriers keep each group of LDS
    // reads together: left to itself the compiler waits for every read in turn.
    constexpr int SPLIT = GNW / 4, PS = 2 * NS;
    constexpr uint32_t KNONE = 0x07FFFFFFu;  // times 16: past the end of every buffer
    auto visit_k = [&](const double2 *tab, bool ho, bool hn, int w, int nw, auto &&load, auto &&use) {
        const int sub = w % SPLIT, team = w / SPLIT, nt = nw / SPLIT;
#pragma unroll 1
        for (int r = 0; r * nt < nkblk; ++r) {
            const int blk = r * nt + ((r & 1) ? nt - 1 - team : team);
            if (blk >= nkblk) continue;
            const int ri = blk * 64 + lane;
            int pos = kbase[blk];
            const int4 run = ri < nruns ? runs[ri] : make_int4(0, 0, 0, 0);
            const int L = run.w;
            // runs of length >= l: the block's first lanes
            auto count = [&](int l) { return (int)__popcll(__builtin_amdgcn_ballot_w64(L >= l)); };
            auto at = [&](int p, int cnt) { return lane < cnt ? (uint32_t)(p + lane) : KNONE; };
            pos = __builtin_amdgcn_readfirstlane(pos);
            // this wavefront's first step
            int j = sub, np = count(1), nm = 0;
            if (SPLIT > 1 && sub > 0) {
                pos += np;
                for (int i = 1; i < sub; ++i) pos += count(2 * i) + count(2 * i + 1);
                np = count(2 * j);
                nm = count(2 * j + 1);
            }
            uint32_t ap = at(pos, np), am = at(pos + np, nm);
            auto lp = load(ap), lm = load(am);
            double er[PS], ei[PS];
            const double2 *tx = tab + abs(run.x) * PS, *ty = tab + (m0 + abs(run.y)) * PS,
                          *tz = tab + (m0 + m1 + abs(run.z)) * PS;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                double2 cx[NS], cy[NS], cz[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    cx[s] = tx[p * NS + s];
                    cy[s] = ty[p * NS + s];
                    cz[s] = tz[p * NS + s];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const double2 cc = cis_from_axes(cx[s], cy[s], cz[s], run.x, run.y, run.z);
                    // a pose that the move does not have counts zero times
                    const double q = p ? (hn ? g_q[s] : 0.0) : (ho ? -g_q[s] : 0.0);
                    er[p * NS + s] = q * cc.x;
                    ei[p * NS + s] = q * cc.y;
                }
            }
            const double2 *tj = tab + (m0 + m1 + j) * PS;
#pragma unroll 1
            while (np > 0) {
                double2 z[PS];
#pragma unroll
                for (int i = 0; i < PS; ++i) z[i] = tj[i];  // e^0 = 1 at step 0
                tj += SPLIT * PS;
                // the next step's positions and loads
                int pos2 = pos + np + nm;
                for (int i = j + 1; i < j + SPLIT; ++i) pos2 += count(2 * i) + count(2 * i + 1);
                j += SPLIT;
                const int np2 = count(2 * j), nm2 = count(2 * j + 1);
                const uint32_t ap2 = at(pos2, np2), am2 = at(pos2 + np2, nm2);
                auto lp2 = load(ap2), lm2 = load(am2);
                __builtin_amdgcn_sched_barrier(0);
                double A = er[0] * z[0].x, B = ei[0] * z[0].y, C = er[0] * z[0].y, D = ei[0] * z[0].x;
#pragma unroll
                for (int i = 1; i < PS; ++i) {
                    A = __builtin_fma(er[i], z[i].x, A);
                    B = __builtin_fma(ei[i], z[i].y, B);
                    C = __builtin_fma(er[i], z[i].y, C);
                    D = __builtin_fma(ei[i], z[i].x, D);
                }
                use(ap, lp, A - B, C + D);
                use(am, lm, A + B, D - C);
                pos = pos2;
                np = np2;
                nm = nm2;
                ap = ap2;
                am = am2;
                lp = lp2;
                lm = lm2;
            }
        }
    };
    // S_k and the weights through buffer loads (zero past the end; and the compiler does not move
    // them back to their use, as it does with plain loads that it can rematerialise)
    const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc((void *)Sk, (short)0, nk * 16, 0x00020000);
    const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc((void *)kw, (short)0, nk * 8, 0x00020000);
    auto load_S = [&](uint32_t p) {
        return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rS, (int)(p * 16u), 0, 0));
    };
    auto load_w = [&](uint32_t p) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rW, (int)(p * 8u), 0, 0));
    };

    // cycle mode: a cycle of chain n is max(occupancy at its start, min_cycle) attempts, and its
    // sample is taken at its end. Called before every attempt; false once the run is over.
    int64_t c = 0, m = 0, len = 0;
    bool finished = false;
    // cycles whose end-of-cycle snapshot is still to be written (npend of them from pend0): a
    // boundary only records the cycle, and the copy runs before the next commit (the state cannot
    // change before then)
    int64_t pend0 = 0;
    int npend = 0;
    auto cycle_boundary = [&]() -> bool {
        while (m == len) {
            if (c > 0) {
                if (occ > maxocc) maxocc = occ;
                const auto r = rare();
                if (r->sampling && tid == 0) {
                    const int64_t at = (int64_t)n * r->samp_stride + r->samp_base + c - 1;
                    r->samp_e[at] = E;
                    r->samp_n[at] = (double)occ;
                }
                if (c - 1 < r->snap_n && npend++ == 0) pend0 = c - 1;
            }
            const auto r = rare();
            if (c == r->ncycles) return false;
            if (occ > maxocc) maxocc = occ;
            len = occ > r->min_cycle ? occ : r->min_cycle;
            m = 0;
            ++c;
        }
        return true;
    };

    // writes the pending snapshots: the structure factor and the guests were last written before
    // a barrier
    auto flush_snapshots = [&]() {
        for (int64_t cs = pend0; cs < pend0 + npend; ++cs) {
            const auto &S = rare()->snap;
            double2 *dsk = S.csk + cs * S.ctot + S.coff[n];
            for (int k = tid; k < nk; k += WG) {
                const double w = kw[k];
                const double2 v = Sk[k];
                dsk[k] = make_double2(w * v.x, w * v.y);
            }
            double4 *dp = S.pos + cs * S.nslots + gr0, *dq = S.quat + cs * S.nslots + gr0;
            for (int i = tid; i < occ; i += WG) {
                dp[i] = a.refpos[gr0 + i];
                dq[i] = a.quat[gr0 + i];
            }
            if (tid == 0) S.occ[cs * S.nsys + n] = occ;
        }
        npend = 0;
    };

    // The attempt's slot, proposal and sites, into LDS: 2 NS lanes, one per (pose, site).
    auto propose = [&](int b) {
        const int type = draws.type[b], pose = gt / NS, t = gt - pose * NS;
        int slot = 0;
        double p[3] = {0, 0, 0}, q[4] = {0, 0, 0, 1}, x[3], f[3];
        if (type != MOVE_INSERTION) {
            const int64_t idx = (int64_t)mulhi64(draws.slot[b], (uint64_t)(occ > 0 ? occ : 1)) + 1;
            const int64_t sl = gr0 + idx - 1;
            slot = (int)(sl < nslots - 1 ? sl : nslots - 1);
            if (slot < 0) slot = 0;
            const double4 p4 = a.refpos[slot], q4 = a.quat[slot];
            p[0] = p4.x; p[1] = p4.y; p[2] = p4.z;
            q[0] = q4.x; q[1] = q4.y; q[2] = q4.z; q[3] = q4.w;
        }
        if (pose == 1) {
            if (type == MOVE_TRANSLATION) {
                const double st = a.step_trans ? a.step_trans[n] : 0.0;
                for (int d = 0; d < 3; ++d) p[d] = p[d] + st * draws.v[d][b];
            } else if (type == MOVE_ROTATION) {
                const double qp[4] = {draws.v[0][b], draws.v[1][b], draws.v[2][b], draws.v[3][b]}, oq[4] = {q[0], q[1], q[2], q[3]};
                qmul(qp, oq, q);
                qnormalize(q);
            } else if (type == MOVE_REINSERTION || type == MOVE_INSERTION) {
                for (int d = 0; d < 3; ++d) p[d] = draws.v[d][b];
                for (int i = 0; i < 4; ++i) q[i] = draws.v[3 + i][b];
            }
        }
        site_of(p, q, t, x);
        matvec(cI, x, f);
        for (int d = 0; d < 3; ++d) {
            at_site[gi][pose][t][d] = x[d];
            at_frac[gi][pose][t][d] = f[d];
        }
        if (gt == NS) {
            at_type[gi] = type;
            at_slot[gi] = slot;
            matvec(cI, p, f);
            at_bin[gi] = near_bin(a.near.desc[u], f);
            at_lu[gi] = draws.lu[b];
            at_he[gi] = type != MOVE_INSERTION ? a.host_e[slot] : 0.0;
            for (int d = 0; d < 3; ++d) at_p[gi][d] = p[d];
            for (int i = 0; i < 4; ++i) at_q[gi][i] = q[i];
        }
    };

    // The sums of the group's attempt over this wavefront's share: host-guest in lane 63's hsum,
    // the guest-guest and reciprocal change in its osum.
    auto evaluate = [&](double &hsum, double &osum) {
        const int type = __builtin_amdgcn_readfirstlane(at_type[gi]), slot = __builtin_amdgcn_readfirstlane(at_slot[gi]);
        const bool has_old = type != MOVE_INSERTION, has_new = type != MOVE_DELETION;
        double2 *mytab = ktab + (size_t)gi * 2 * NS * tw;
        if (charged)
            for (int e = gt; e < 2 * NS * tw; e += GW) {
                const int ps = (int)(((float)e + 0.5f) * inv_tw), x = e - ps * tw;  // exact for e < 2^22
                const int pose = ps / NS, t = ps - pose * NS;
                const int d = x < m0 ? 0 : (x < m0 + m1 ? 1 : 2);
                const int mm = x - (d == 0 ? 0 : (d == 1 ? m0 : m0 + m1));
                mytab[x * 2 * NS + ps] = axis_power_const(at_frac[gi][pose][t][d], mm);
            }
        // real space: the (site, site) pairs inside the cutoff go through the wavefront's ring in
        // LDS and are evaluated 64 at a time, so LJ + erfc run on full wavefronts
        PairQueue Q(rings[wid], lane);
        // (1) host-guest, the new pose: minimum images in fractional coordinates
        hsum = 0.0;
        auto host_pair = [&](double r2, double qq, int code) {
            const double2 p = ptab[code];
            hsum += cw_pair(r2, p.x, p.y, qq, alpha, a.rc_lj2, a.rc_ew2);
        };
        if (has_new) {
            double f[NS][3], A[9];
#pragma unroll
            for (int s = 0; s < NS; ++s)
                for (int d = 0; d < 3; ++d) f[s][d] = at_frac[gi][1][s][d];
            for (int i = 0; i < 9; ++i) A[i] = cA[i];
            near_scan<NS, UPPER>(a.near, F.atom_off, A, __builtin_amdgcn_readfirstlane(at_bin[gi]), f, g_q, a.ntypes_c,
                                 a.rc_max2, nullptr, Q, host_pair, gw, GNW);
        }
        // (2) guest-guest: the sites of the new pose (added) and of the old one (taken away by a
        // move, counted by a deletion) against every site of the other live guests. Both poses'
        // terms of a (site, other site) pair are taken in one lane: where guests overlap they are
        // large and nearly cancel.
        const double nan = __builtin_nan("");
        double gsum = 0.0;
        const double sg_old = type <= MOVE_REINSERTION ? -1.0 : 1.0;
        auto guest_pair = [&](double r2n, double r2o, int code) {
            const double2 p = ptab[gg0 + code];
            const double qq = qgg[code];
            gsum += cw_pair<true>(r2n, p.x, p.y, qq, alpha, a.rc_lj2, a.rc_ew2);
            gsum += sg_old * cw_pair<true>(r2o, p.x, p.y, qq, alpha, a.rc_lj2, a.rc_ew2);
        };
#pragma unroll 1
        for (int xb = gw * 64; xb < occ * NS; xb += GW) {
            const int x = xb + lane, jj = x / NS, sb = x - jj * NS;
            const bool on = x < occ * NS && !(has_old && gr0 + jj == slot);
            const double4 b4 = on ? gsite[x] : make_double4(nan, nan, nan, 0.0);
            const double pb[3] = {b4.x, b4.y, b4.z};
#pragma unroll
            for (int s0 = 0; s0 < NS; s0 += 3) {
#pragma unroll
                for (int sa = s0; sa < (s0 + 3 < NS ? s0 + 3 : NS); ++sa) {
                    const double r2n = has_new ? mi_r2<UPPER>(cA, cI, at_site[gi][1][sa], pb) : nan;
                    const double r2o = has_old ? mi_r2<UPPER>(cA, cI, at_site[gi][0][sa], pb) : nan;
                    Q.push(r2n < a.rc_max2 || r2o < a.rc_max2, r2n, r2o, sa * NS + sb);
                }
#pragma unroll 1
                while (Q.pending() >= 64) Q.drain(64, guest_pair);
            }
        }
        Q.drain(Q.pending(), guest_pair);
        osum = type == MOVE_DELETION ? -gsum : gsum;
    };

    // (3) The reciprocal change against the running structure factor. The guest term e^{i k.r} of
    // k = 2 pi A^-T n at r = A f is the product over axes of e^{2 pi i n_d f_d}, from the tables.
    auto reciprocal = [&]() -> double {
        const int type = __builtin_amdgcn_readfirstlane(at_type[gi]);
        double rsum = 0.0;
        struct Term {
            double2 S;
            double w;
        };
        visit_k(ktab + (size_t)gi * 2 * NS * tw, type != MOVE_INSERTION, type != MOVE_DELETION, gw, GNW,
                [&](uint32_t p) { return Term{load_S(p), load_w(p)}; },
                [&](uint32_t, const Term &t, double sre, double sim) {
                    const double e = __builtin_fma(sre, __builtin_fma(2.0, t.S.x, sre),
                                                   sim * __builtin_fma(2.0, t.S.y, sim));
                    rsum = __builtin_fma(t.w, e, rsum);
                });
        return KE * rsum;
    };

    // Both modes. In cycle mode a round may span cycle boundaries: the move types are drawn per
    // attempt counter, and a boundary only samples the state and, while no attempt has been
    // accepted, fixes the next cycle's length from the unchanged occupancy.
    uint64_t pbase = 0;
    bool have = false;
    for (;;) {
        int nv = SPEC;
        if (a.mode == 0) {
            if (m >= a.nmoves) break;
            if (a.nmoves - m < SPEC) nv = (int)(a.nmoves - m);
        } else if (!cycle_boundary()) {
            break;
        }
        if (!have || ctr + (uint64_t)nv > pbase + MC_BATCH) {
            if (wid == 0) mc_draw(seed, ctr, cA, draws);
            pbase = ctr;
            have = true;
            __syncthreads();
        }
        const bool active = gi < nv;
        if (active && gt < 2 * NS) propose((int)(ctr - pbase) + gi);
        __syncthreads();
        double hsum = 0.0, osum = 0.0;
        if (active) evaluate(hsum, osum);
        if (charged) {
            __syncthreads();
            if (active) osum += reciprocal();
        }
        hsum = wave_sum63(hsum);
        osum = wave_sum63(osum);
        if (lane == 63) {
            red[0][wid] = hsum;
            red[1][wid] = osum;
        }
        __syncthreads();

        // Metropolis tests of the round's attempts, one per lane, the same in every wavefront
        double d = 0.0, e_new = 0.0;
        bool accept = false, full = false;
        if (lane < nv) {
            double oth = 0.0;
            for (int w = lane * GNW; w < (lane + 1) * GNW; ++w) {
                e_new += red[0][w];
                oth += red[1][w];
            }
            const int ty = at_type[lane];
            const double lu = at_lu[lane], he = at_he[lane];
            if (ty <= MOVE_REINSERTION) {
                d = (e_new - he) + oth;
                accept = isfinite(d) && (-d / a.kT > lu) && occ > 0;
            } else {
                if (ty == MOVE_INSERTION) {
                    d = e_new + oth + (cp + cq * (double)occ);
                    const double lp = log_fugV - a.logn[occ] - a.log_kT;
                    const bool would = isfinite(d) && (lp - d / a.kT > lu);
                    accept = would && occ < cap;
                    full = would && occ >= cap;
                } else {
                    const int occ_eff = occ > 0 ? occ : 1;
                    d = oth - (he + (cp + cq * (double)(occ - 1)));
                    const double lp = -(log_fugV - a.logn[occ_eff - 1] - a.log_kT);
                    accept = isfinite(d) && (lp - d / a.kT > lu) && occ > 0;
                }
            }
        }
        const uint64_t acc_m = __builtin_amdgcn_ballot_w64(accept), full_m = __builtin_amdgcn_ballot_w64(full);
        // in order; the first accepted one ends the round
        int done = 0, first = -1;
        for (int g = 0; g < nv; ++g) {
            if (a.mode != 0 && !cycle_boundary()) {
                finished = true;
                break;
            }
            ++m;
            done = g + 1;
            const bool acc = (acc_m >> g) & 1;
            if ((full_m >> g) & 1) caphit = 1;
            if (traced) {
                const auto r = rare();
                const double dg = __shfl(d, g, 64);
                if (tid == 0 && ntrace < r->trace_cap)
                    r->trace[(int64_t)n * r->trace_cap + ntrace] =
                        make_double4((double)at_type[g], (double)(at_slot[g] - gr0), dg, acc ? 1.0 : 0.0);
            }
            ++ntrace;
            if (tid == 0) ++cnt_att[at_type[g] - 1];
            if (acc) {
                first = g;
                break;
            }
        }
        if (npend > 0) {
            flush_snapshots();
            __syncthreads();  // the commit below overwrites guests the copy read
        }
        if (first >= 0) {
            const int ty = __builtin_amdgcn_readfirstlane(at_type[first]);
            const int sl = __builtin_amdgcn_readfirstlane(at_slot[first]);
            const double dU = __shfl(d, first, 64), e_first = __shfl(e_new, first, 64);
            const int to = ty == MOVE_INSERTION ? gr0 + occ : sl;  // the slot written
            if (tid < NS) {
                const double *x = at_site[first][1][tid];
                gsite[(to - gr0) * NS + tid] =
                    ty == MOVE_DELETION ? gsite[(occ - 1) * NS + tid] : make_double4(x[0], x[1], x[2], 0.0);
            }
            if (tid == 0) {
                const double *pp = at_p[first], *qq = at_q[first];
                if (ty != MOVE_DELETION) {
                    a.refpos[to] = make_double4(pp[0], pp[1], pp[2], 0.0);
                    a.quat[to] = make_double4(qq[0], qq[1], qq[2], qq[3]);
                    a.host_e[to] = e_first;
                } else {
                    const int hi = gr0 + occ - 1;
                    if (sl != hi) {
                        a.refpos[sl] = a.refpos[hi];
                        a.quat[sl] = a.quat[hi];
                        a.host_e[sl] = a.host_e[hi];
                    }
                }
                ++cnt_acc[ty - 1];
            }
            if (ty == MOVE_INSERTION) ++occ;
            if (ty == MOVE_DELETION) --occ;
            E += dU;
            Eabs += fabs(dU);
            if (charged)
                // the accepted attempt's changes, evaluated again from its tables (cheaper than
                // writing and reading every attempt's)
                visit_k(ktab + (size_t)first * 2 * NS * tw, ty != MOVE_INSERTION, ty != MOVE_DELETION, wid, NW,
                        [&](uint32_t p) { return load_S(p); },
                        [&](uint32_t p, const double2 S, double sre, double sim) {
                            if (p != KNONE) Sk[p] = make_double2(S.x + sre, S.y + sim);
                        });
            skabs += ds_bound;
        }
        ctr += (uint64_t)done;
        __syncthreads();  // committed poses, red[] and the attempts' records reused by the next round
        if (finished) break;
    }
    flush_snapshots();
    if (tid == 0) {
        a.occupancy[n] = occ;
        a.energy[n] = E;
        a.energy_abs[n] = Eabs;
        a.sk_abs[n] = skabs;
        a.rng_counter[n] = ctr;
        for (int t = 0; t < NMOVES; ++t) {
            a.accepted[n * NMOVES + t] += cnt_acc[t];
            a.attempted[n * NMOVES + t] += cnt_att[t];
        }
        if (a.max_occ) a.max_occ[n] = maxocc;
        if (a.capacity_hits) a.capacity_hits[n] = caphit;
    }
}

template <int NS, bool UPPER>
static hipError_t launch_mc_ns(const McArgs &a, int spec, int gnw, size_t lds, hipStream_t st)
{
    const dim3 grid((unsigned)a.nsys), block((unsigned)(spec * gnw * 64));
    if constexpr (NS <= 4) {
        if (spec == 2) {
            hipLaunchKernelGGL((mc_chain_kernel<NS, UPPER, 2, 8>), grid, block, lds, st, a);
            return hipGetLastError();
        }
        if (spec == 4) {
            hipLaunchKernelGGL((mc_chain_kernel<NS, UPPER, 4, 4>), grid, block, lds, st, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((mc_chain_kernel<NS, UPPER, 1, 4>), grid, block, lds, st, a);
    return hipGetLastError();
}

hipError_t launch_mc(const McArgs &a, hipStream_t st)
{
    const int ns = a.guest.nsites;
    // the per-axis phase tables: old and new pose, every site, kn_max[d] + 1 powers per axis. A
    // guest and framework whose tables exceed the limit are refused whatever the split.
    const size_t tab = a.guest.charged ? (size_t)2 * ns * a.ktab_w * sizeof(double2) : 0;
    if (2 * tab > 72 * 1024) return hipErrorInvalidValue;
    const size_t pairs = sizeof(double2) * (size_t)ns * a.ntypes_c + (sizeof(double2) + sizeof(double)) * ns * ns;
    // Attempts at once and wavefronts for each. Up to one chain per CU (256) an attempt's latency
    // counts: two attempts on eight wavefronts each, or, where exchange moves make most attempts
    // fail, four on four. More chains share CUs and evaluate one attempt each, on four. Measured
    // (RUBTAK 3x3x3 + CO2; 2x8, 4x4, 1x4): 500 translations of one chain 6.6, 7.7, 8.5 ms; 24 GCMC
    // chains 5.8, 5.4, 8.0 ms; 60 translations of 512 chains 2.1, 2.8, 1.6 ms. Guests of five
    // and six sites spill registers with sixteen wavefronts in a workgroup.
    int spec = 1, gnw = 4;
    if (a.nsys <= 256 && ns <= 4) {
        const bool exchange = a.mode == 0 ? a.movetype >= MOVE_INSERTION : a.pcum[MOVE_REINSERTION - 1] < 1.0;
        spec = exchange ? 4 : 2;
        gnw = exchange ? 4 : 8;
        // LDS: tables, sixteen rings of 20-byte pairs, some 8 KB of draws and records
        if (spec * tab + pairs + 16 * sizeof(PairRing) + 8 * 1024 > 160 * 1024) spec = 1, gnw = 4;
    }
    const size_t lds = spec * tab + pairs;
    switch (ns * 2 + (a.upper ? 1 : 0)) {
    case 2: return launch_mc_ns<1, false>(a, spec, gnw, lds, st);
    case 3: return launch_mc_ns<1, true>(a, spec, gnw, lds, st);
    case 4: return launch_mc_ns<2, false>(a, spec, gnw, lds, st);
    case 5: return launch_mc_ns<2, true>(a, spec, gnw, lds, st);
    case 6: return launch_mc_ns<3, false>(a, spec, gnw, lds, st);
    case 7: return launch_mc_ns<3, true>(a, spec, gnw, lds, st);
    case 8: return launch_mc_ns<4, false>(a, spec, gnw, lds, st);
    case 9: return launch_mc_ns<4, true>(a, spec, gnw, lds, st);
    case 10: return launch_mc_ns<5, false>(a, spec, gnw, lds, st);
    case 11: return launch_mc_ns<5, true>(a, spec, gnw, lds, st);
    case 12: return launch_mc_ns<6, false>(a, spec, gnw, lds, st);
    case 13: return launch_mc_ns<6, true>(a, spec, gnw, lds, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pa
