// tp_map3.hip -- gfx950 kernels of the <Map^3> integrand path.
//
//  * the node (tp_device.h): BiHalofit (Takahashi et al. 2020, eqs. B4-B9) at one Limber
//    z-node, restating classed_version/bispectrum.cpp:166-236 (with F2 :614-633
//    and the Eisenstein & Hu P(k) :811-841) in terms of the dimensionless
//    wavenumbers q = k r_sigma.  Everything that depends on z only comes from a
//    per-node record (TpNodeT) that the table builder evaluated once in FP64.
//  * the 96-node Limber sum of classed_version/bispectrum.cpp: 238-286 /
//    1010-1020, accumulated in FP64.  T = double is the plain path;
//    T = float runs the bispectrum in FP32 (native v_exp_f32 / v_log_f32).
//  * point kernels (k_points, k_points_nodes): rows of B_kappa or of the <Map^3>
//    integrand, classed_version/apertureStatistics.cpp:16-28.
//  * region kernels: Genz-Malik degree-7/5 rule (classed_version/hcubature.cpp:
//    456-577) for many 3-D regions of many integrals per launch -- the points
//    (a thread or several waves per point, or P_E terms shared by a region's
//    points), then one thread per region for the rule sums, in the reference's
//    summation order.
#include <cmath>
#include <vector>

#include "tp_device.h"

namespace {

// --------------------------------------------------------------- kernels
// Points of the evaluation calls: B_kappa at (l1, l2, l3) rows, or the <Map^3> integrand at (l1, l2, phi) rows.
// Set-up of a point and its value from the z-sum, for the kernels below that split the sum differently.
struct PointTh {
    double t[3];  // aperture radii of the <Map^3> integrand
};
template <bool MAP3>
__device__ __forceinline__ int point_begin(const double *__restrict__ x, size_t i, int mode, int *flag, TpPointPre *P)
{
    const double a = x[3 * i], b = x[3 * i + 1], c = x[3 * i + 2];
    if (MAP3) return tp_map3_begin(a, b, c, mode, flag, P);
    P->l[0] = a;
    P->l[1] = b;
    P->l[2] = c;
    if (a == 0 || b == 0 || c == 0 || mode == TP_MODE_ANALYTIC) return TP_PT_NOSUM;
    tp_point_pre<double>(a, b, c, P);
    return TP_PT_SUM;
}
template <bool MAP3>
__device__ __forceinline__ double point_end(const TpPointPre &P, int kind, double sum, const PointTh &th, int mode,
                                            int *flag)
{
    if (MAP3) return tp_map3_end(P, kind, sum, th.t[0], th.t[1], th.t[2], flag);
    double v = sum;
    if (kind != TP_PT_SUM) v = mode == TP_MODE_ANALYTIC ? tp_bkappa_analytic(P.l[0], P.l[1], P.l[2]) : 0.0;
    if (!isfinite(v)) atomicOr(flag, 1);
    return v;
}

// A point's 96 nodes split over LPP waves (a power of two up to 8), the fixed summation tree of k_region_points: one thread per
// point takes ~100 us (FP32) to ~270 us (FP64) however few the points are, since its 96 nodes are one serial chain.
template <class T, int LPP, bool MAP3>
__global__ void __launch_bounds__(64 * (LPP < 4 ? 4 : LPP)) k_points(const TpNodeT<T> *__restrict__ nodes,
                                                                     const TpEHT<T> *__restrict__ eh, PointTh th,
                                                                     size_t npts, const double *__restrict__ x,
                                                                     double *__restrict__ f, int mode, int *flag)
{
    constexpr int GPB = LPP < 4 ? 4 / LPP : 1;  // groups of 64 points per workgroup
    __shared__ double part[GPB][LPP][64];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), g = wv / LPP,
              w = wv % LPP;
    const size_t i = ((size_t)blockIdx.x * GPB + g) * 64 + lane;
    TpPointPre P;
    int kind = TP_PT_DONE;
    double v = 0.0;
    if (i < npts) {
        kind = point_begin<MAP3>(x, i, mode, flag, &P);
        if (kind == TP_PT_SUM) v = tp_bkappa_parts<T, TP_NPART / LPP>(nodes, *eh, P, w * (TP_NPART / LPP));
    }
    if constexpr (LPP > 1) {
        part[g][w][lane] = v;
        __syncthreads();
        if (w != 0) return;
        double a[LPP];
#pragma unroll
        for (int k = 0; k < LPP; ++k) a[k] = part[g][k][lane];
#pragma unroll
        for (int s = 1; s < LPP; s <<= 1)
#pragma unroll
            for (int k = 0; k < LPP; k += 2 * s) a[k] = a[k] + a[k + s];
        v = a[0];
    }
    if (i < npts) f[i] = point_end<MAP3>(P, kind, v, th, mode, flag);
}

// The fewest points: one thread per (point, node), two points per workgroup of three waves.  Every thread of a point
// forms its set-up (no exchange, no barrier before the node), the node values go to LDS, eight threads add the
// partials in node order and one joins the tree -- the bits of every other split.  The chain is one node instead of
// twelve (8 waves per point); the set-up, repeated 96 times, is ~0.7 of a node's work, so it pays only while the
// launch leaves the chip idle.
constexpr int kNodePts = 2, kNodeBlock = kNodePts * TP_NNODES;  // 192 threads

// value of node `node` for the point, into val[node]; the sum over all nodes for the threads with node == 0
template <class T>
__device__ __forceinline__ double node_sum(const TpNodeT<T> *__restrict__ nodes, const TpEHT<T> &E, const TpPointPre &P,
                                           bool sum, int node, T *val, double *part)
{
    if (sum) {
        const TpNodeT<T> &N = nodes[node];
        const T ks = N.ks, lks = N.lnks;
        const T q[3] = {(T)P.l[0] * ks, (T)P.l[1] * ks, (T)P.l[2] * ks};
        const T lq[3] = {(T)P.ll[0] + lks, (T)P.ll[1] + lks, (T)P.ll[2] + lks};
        const T f2t[3] = {(T)P.f2t[0], (T)P.f2t[1], (T)P.f2t[2]};
        val[node] = tp_bispec_node<T>(N, E, q, lq, f2t, (T)P.lr1, (T)P.r2);
    }
    __syncthreads();
    if (sum && node < TP_NPART) {
        double acc = 0.0;
        for (int j = 0; j < TP_PART_NODES; ++j) {
            const int n = node * TP_PART_NODES + j;
            acc += (double)(nodes[n].wz * val[n]);
        }
        part[node] = acc;
    }
    __syncthreads();
    if (!sum || node != 0) return 0.0;
    return ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
}

template <class T, bool MAP3>
__global__ void __launch_bounds__(kNodeBlock) k_points_nodes(const TpNodeT<T> *__restrict__ nodes,
                                                             const TpEHT<T> *__restrict__ eh, PointTh th, size_t npts,
                                                             const double *__restrict__ x, double *__restrict__ f,
                                                             int mode, int *flag)
{
    __shared__ T val[kNodePts][TP_NNODES];
    __shared__ double part[kNodePts][TP_NPART];
    const int p = threadIdx.x / TP_NNODES, node = threadIdx.x - p * TP_NNODES;
    const size_t i = (size_t)blockIdx.x * kNodePts + p;
    TpPointPre P;
    const int kind = i < npts ? point_begin<MAP3>(x, i, mode, flag, &P) : TP_PT_DONE;
    const double v = node_sum<T>(nodes, *eh, P, kind == TP_PT_SUM, node, val[p], part[p]);
    if (i < npts && node == 0) f[i] = point_end<MAP3>(P, kind, v, th, mode, flag);
}

// The same split for the regions of a batch's smallest rounds.
template <class T>
__global__ void __launch_bounds__(kNodeBlock) k_region_nodes(const TpNodeT<T> *__restrict__ nodes,
                                                             const TpEHT<T> *__restrict__ eh, size_t nreg,
                                                             const TpRegion *__restrict__ reg,
                                                             const TpIntegralDesc *__restrict__ desc,
                                                             double *__restrict__ fvals, int mode, int *flag)
{
    __shared__ T val[kNodePts][TP_NNODES];
    __shared__ double part[kNodePts][TP_NPART];
    const int p = threadIdx.x / TP_NNODES, node = threadIdx.x - p * TP_NNODES;
    const size_t t = (size_t)blockIdx.x * kNodePts + p;
    const bool live = t < nreg * TP_NPTS_GM3;
    TpPointPre P;
    int kind = TP_PT_DONE;
    TpIntegralDesc D{};
    if (live) {
        const size_t r = t / TP_NPTS_GM3;
        const TpRegion R = reg[r];
        D = desc[R.integral];
        double x0, x1, x2;
        gm_point3(R, (int)(t - r * TP_NPTS_GM3), &x0, &x1, &x2);
        kind = tp_map3_begin(x0, x1, x2, mode, flag, &P);
    }
    const double v = node_sum<T>(nodes + (size_t)D.icosmo * TP_NNODES, eh[D.icosmo], P, kind == TP_PT_SUM, node, val[p],
                                 part[p]);
    if (live && node == 0) fvals[t] = tp_map3_end(P, kind, v, D.th[0], D.th[1], D.th[2], flag);
}

// Integrand values of the 33 Genz-Malik points of many regions of many integrals.  A point's 96
// z-nodes are split over LPP waves (1, 2, 4 or 8): wave w of a point group sums the partials
// [w 8/LPP, (w+1) 8/LPP) of the fixed summation tree with wave-uniform (scalar) node reads, and
// the group's first wave combines the waves' sums in tree order -- the same bits for every LPP.
// A workgroup holds max(1, 4/LPP) groups of 64 points.  nodes/eh are indexed by the integral's
// cosmology.
template <class T, int LPP>
__global__ void __launch_bounds__(64 * (LPP < 4 ? 4 : LPP)) k_region_points(
    const TpNodeT<T> *__restrict__ nodes, const TpEHT<T> *__restrict__ eh, size_t nreg,
    const TpRegion *__restrict__ reg, const TpIntegralDesc *__restrict__ desc, double *__restrict__ fvals, int mode,
    int *flag)
{
    constexpr int GPB = LPP < 4 ? 4 / LPP : 1;  // point groups per workgroup
    __shared__ double part[GPB][LPP][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = wv / LPP, w = wv % LPP;
    const size_t t = ((size_t)blockIdx.x * GPB + g) * 64 + lane;
    const bool live = t < nreg * TP_NPTS_GM3;
    TpPointPre P;
    int kind = TP_PT_DONE;
    double v = 0.0;
    TpIntegralDesc D{};
    if (live) {
        const size_t r = t / TP_NPTS_GM3;
        const int p = (int)(t - r * TP_NPTS_GM3);
        const TpRegion R = reg[r];
        D = desc[R.integral];
        double x0, x1, x2;
        gm_point3(R, p, &x0, &x1, &x2);
        kind = tp_map3_begin(x0, x1, x2, mode, flag, &P);
        if (kind == TP_PT_SUM)
            v = tp_bkappa_parts<T, TP_NPART / LPP>(nodes + (size_t)D.icosmo * TP_NNODES, eh[D.icosmo], P,
                                                   w * (TP_NPART / LPP));
    }
    if constexpr (LPP > 1) {
        part[g][w][lane] = v;
        __syncthreads();
        if (w != 0) return;
        double a[LPP];
#pragma unroll
        for (int k = 0; k < LPP; ++k) a[k] = part[g][k][lane];
#pragma unroll
        for (int s = 1; s < LPP; s <<= 1)
#pragma unroll
            for (int k = 0; k < LPP; k += 2 * s) a[k] = a[k] + a[k + s];
        v = a[0];
    }
    if (live) fvals[t] = tp_map3_end(P, kind, v, D.th[0], D.th[1], D.th[2], flag);
}

// Region-cached form of k_region_points (launch shapes 16, 32, 64).  Of a region's 33 points only 7
// distinct l1 (axis-0 codes -3..3) and 7 distinct l2 occur, and the P_E term of BiHalofit
// (tp_pse_node: the linear P(k), its exp/log and reciprocals) depends on one wavenumber only.  A
// workgroup takes kCacheReg regions with G groups of 256 threads; group g owns the partials
// [g 8/G, (g+1) 8/G) of the summation tree and, for each partial (12 z-nodes),
//   A. evaluates the P_E terms of the 47 multipoles per region (7 l1, 7 l2, 33 l3) at the 12 nodes
//      into its LDS block (work items of one node and 64 multipoles, and the remainders of all nodes
//      node records are read through wave-uniform loads);
//   B. lets each point add its 12 node values, the shape-dependent rest (tp_bispec_joint) with the
//      three P_E terms read from LDS, and push the partial into the group's subtree.
// The groups' subtrees are then joined in tree order.  Every value is formed by the same operations
// as in k_region_points, so every shape gives the same bits.  More groups shorten a thread's share
// of the work, which keeps launches of a few thousand regions from ending on a half-empty wave of
// workgroups.
constexpr int kCacheReg = 7, kCacheThreads = 256;  // regions per workgroup and threads per group
constexpr int kCacheSets = 2 * kCacheReg;          // (region, axis) sets of 7 multipoles l1 or l2
constexpr int kCacheN = 7 * kCacheSets + TP_NPTS_GM3 * kCacheReg;  // multipoles at most: 329
static_assert(kCacheSets <= 64 && TP_NPTS_GM3 * kCacheReg <= kCacheThreads && 7 * kCacheSets <= kCacheThreads, "");

// FP32: six waves per SIMD (80 VGPRs of the 93 it would take; 8 dwords spill, outside the node loops) against five,
// 74.2 -> 73.2 ms; FP64: four.
template <class T, int G>
__global__ void __launch_bounds__(kCacheThreads * G)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 6 : 4))) k_region_cached(const TpNodeT<T> *__restrict__ nodes,
                                                           const TpEHT<T> *__restrict__ eh, size_t nreg,
                                                           const TpRegion *__restrict__ reg,
                                                           const TpIntegralDesc *__restrict__ desc,
                                                           double *__restrict__ fvals, int mode, int *flag)
{
    constexpr int PPG = TP_NPART / G;                 // partials per group
    __shared__ T lv[kCacheN], llv[kCacheN];           // multipole and its log, as the points see them
    __shared__ T pse[G][TP_PART_NODES][kCacheN];      // P_E at (group, node of the partial, multipole)
    __shared__ double sub[G > 1 ? G : 1][kCacheReg * TP_NPTS_GM3];  // the groups' subtree values
    __shared__ double set_c[kCacheSets], set_h[kCacheSets];  // centre and half width of each (region, axis) set
    __shared__ int set_ic[kCacheSets];                // its cosmology (set 2 rr: of region rr)
    __shared__ int slot[kCacheSets], uset[kCacheSets];  // a set's place among the distinct ones; a place's set
    __shared__ int n_uset, one_cosmo;                 // distinct sets; all regions of the workgroup share a cosmology
    constexpr int NW = kCacheThreads / 64;
    const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kCacheThreads);
    const int t = threadIdx.x - g * kCacheThreads, lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const size_t r0 = (size_t)blockIdx.x * kCacheReg;
    const int nr = (int)((nreg - r0) < (size_t)kCacheReg ? (nreg - r0) : (size_t)kCacheReg);  // >= 1
    const int ns = 2 * nr;
    // distinct sets: wave 0 of group 0, one lane per set (lanes of one wave exchange through LDS, in order)
    if (threadIdx.x < 64) {
        double c = 0.0, h = 0.0;
        int ic = 0;
        if (lane < ns) {
            const TpRegion &R = reg[r0 + (lane >> 1)];
            c = R.c[lane & 1];
            h = R.hw[lane & 1];
            ic = desc[R.integral].icosmo;
            set_c[lane] = c;
            set_h[lane] = h;
            set_ic[lane] = ic;
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        int first = lane;
        for (int k = ns - 1; k >= 0; --k)
            if (k < lane && lane < ns && set_c[k] == c && set_h[k] == h && set_ic[k] == ic) first = k;
        const unsigned long long uniq = __ballot(lane < ns && first == lane);
        if (lane < ns) {
            const int at = __popcll(uniq & ((1ull << first) - 1));
            slot[lane] = at;
            if (first == lane) uset[at] = lane;
        }
        const unsigned long long other = __ballot(lane < ns && ic != __builtin_amdgcn_readfirstlane(ic));
        if (lane == 0) {
            n_uset = __popcll(uniq);
            one_cosmo = other == 0;
        }
    }
    // every group's point threads form their point
    const bool pt = t < nr * TP_NPTS_GM3;
    const int prr = t / TP_NPTS_GM3, pp = t - prr * TP_NPTS_GM3;
    TpPointPre P;
    int kind = TP_PT_DONE;
    TpIntegralDesc D{};
    if (pt) {
        const TpRegion R = reg[r0 + prr];
        D = desc[R.integral];
        double x0, x1, x2;
        gm_point3(R, pp, &x0, &x1, &x2);
        kind = tp_map3_begin(x0, x1, x2, mode, flag, &P);  // every group flags the same points: same bit
    }
    __syncthreads();
    // group 0 stores the multipoles: the distinct sets', then the points' l3
    const int nu7 = 7 * __builtin_amdgcn_readfirstlane(n_uset);
    const int ne = nu7 + nr * TP_NPTS_GM3;
    if (g == 0) {
        if (pt) {
            const int e = nu7 + t;
            lv[e] = kind == TP_PT_SUM ? (T)P.l[2] : T(1);
            llv[e] = kind == TP_PT_SUM ? (T)P.ll[2] : T(0);
        }
        if (t < nu7) {
            const int u = uset[t / 7];
            const double x = tp_gm_coord(set_c[u], set_h[u], t % 7 - 3);
            lv[t] = (T)x;
            llv[t] = x > 0 ? (T)TpMath<double>::lg(x) : T(0);  // non-positive: no summed point uses it
        }
    }
    __syncthreads();
    // block-uniform: with one cosmology the node and E&H records are read through scalar loads
    const int uni = __builtin_amdgcn_readfirstlane(one_cosmo);
    const int ic0 = __builtin_amdgcn_readfirstlane(set_ic[0]);
    const TpNodeT<T> *__restrict__ nodes0 = nodes + (size_t)ic0 * TP_NNODES;
    const bool sum = pt && kind == TP_PT_SUM;
    T L[3] = {T(1), T(1), T(1)}, LL[3] = {T(0), T(0), T(0)}, F2T[3] = {T(0), T(0), T(0)}, LR1 = T(0), R2 = T(0);
    int e0 = 0, e1 = 0, e2 = 0;
    const TpNodeT<T> *Np = nodes;
    if (sum) {
        for (int i = 0; i < 3; ++i) {
            L[i] = (T)P.l[i];
            LL[i] = (T)P.ll[i];
            F2T[i] = (T)P.f2t[i];
        }
        LR1 = (T)P.lr1;
        R2 = (T)P.r2;
        e0 = 7 * slot[2 * prr] + c_gm3_code[pp][0] + 3;
        e1 = 7 * slot[2 * prr + 1] + c_gm3_code[pp][1] + 3;
        e2 = nu7 + t;
        Np = nodes + (size_t)D.icosmo * TP_NNODES;
    }
    T(*ps_g)[kCacheN] = pse[g];
    // phase B body: the point's 12 node values of the partial starting at node n0, from records Nb
    auto node_block = [&](const TpNodeT<T> *__restrict__ Nb, int n0) {
        double acc = 0.0;
#pragma unroll 4  // FP32, 24 x 35 integrals: 76.4 ms rolled, 79.9 by 2, 76.8 by 3, 74.2 by 4, 74.5 by 6, 76.0 by 12
        for (int j = 0; j < TP_PART_NODES; ++j) {
            const TpNodeT<T> &N = Nb[n0 + j];
            const T ks = N.ks, lks = N.lnks;
            const T q[3] = {L[0] * ks, L[1] * ks, L[2] * ks};
            const T lq[3] = {LL[0] + lks, LL[1] + lks, LL[2] + lks};
            const T ps[3] = {ps_g[j][e0], ps_g[j][e1], ps_g[j][e2]};
            const T b = tp_bispec_joint<T>(N, q, lq, F2T, LR1, R2, ps);
            acc += (double)(N.wz * b);
        }
        return acc;
    };
    // phase A work items.  One cosmology: the full chunks of 64 multipoles, one node each (wave-uniform records, scalar
    // loads), then the last ne % 64 multipoles of all 12 nodes packed into chunks of 64 (records per lane).  More
    // cosmologies: one node and 64 multipoles, records per lane.
    const int nfull = uni ? ne >> 6 : 0, tail = ne - 64 * nfull, ntail = TP_PART_NODES * tail;
    const int nblk = (ne + 63) >> 6;
    double s1 = 0.0, s2 = 0.0, s4 = 0.0, v = 0.0;
    for (int k = 0; k < PPG; ++k) {
        const int n0 = (g * PPG + k) * TP_PART_NODES;
        if (uni) {
            int j = 0, c = wv;  // (node, chunk) of item wv, wv + NW, ...; past the last node c counts the tail's items
            for (; nfull; c += NW) {
                while (c >= nfull && j < TP_PART_NODES) {
                    c -= nfull;
                    ++j;
                }
                if (j >= TP_PART_NODES) break;
                const TpNodeT<T> &N = nodes0[n0 + j];
                const int e = c * 64 + lane;
                ps_g[j][e] = tp_pse_node<T>(N, eh[ic0], lv[e] * N.ks, llv[e] + N.lnks);
            }
            for (int f = c * 64 + lane; f < ntail; f += kCacheThreads) {
                const int jt = f / tail, e = 64 * nfull + f - jt * tail;
                const TpNodeT<T> &N = nodes0[n0 + jt];
                ps_g[jt][e] = tp_pse_node<T>(N, eh[ic0], lv[e] * N.ks, llv[e] + N.lnks);
            }
        } else {
            for (int it = wv; it < TP_PART_NODES * nblk; it += NW) {
                const int j = it / nblk, e = (it - j * nblk) * 64 + lane;
                if (e < ne) {
                    const int ic = set_ic[e < nu7 ? uset[e / 7] : 2 * ((e - nu7) / TP_NPTS_GM3)];
                    const TpNodeT<T> &N = nodes[(size_t)ic * TP_NNODES + n0 + j];
                    ps_g[j][e] = tp_pse_node<T>(N, eh[ic], lv[e] * N.ks, llv[e] + N.lnks);
                }
            }
        }
        __syncthreads();
        if (sum) v = tp_tree8_push(k, uni ? node_block(nodes0, n0) : node_block(Np, n0), s1, s2, s4);
        __syncthreads();
    }
    if constexpr (G > 1) {  // join the groups' subtrees: v0 + v1, or (v0 + v1) + (v2 + v3)
        if (pt) sub[g][t] = v;
        __syncthreads();
        if (g != 0) return;
        if (pt) {
            double a[G];
#pragma unroll
            for (int i = 0; i < G; ++i) a[i] = sub[i][t];
#pragma unroll
            for (int st = 1; st < G; st <<= 1)
#pragma unroll
                for (int i = 0; i < G; i += 2 * st) a[i] = a[i] + a[i + st];
            v = a[0];
        }
    }
    if (pt) fvals[(r0 + prr) * TP_NPTS_GM3 + pp] = tp_map3_end(P, kind, v, D.th[0], D.th[1], D.th[2], flag);
}

// Region r's flag: bit 0 = non-finite rule estimate.  Region 0 also carries the point
// kernel's flag word (non-finite ell: bit 1, non-finite B_kappa: bit 2), so one copy of
// the region outputs returns every error of the round.
__global__ void __launch_bounds__(256) k_region_rule(size_t nreg, const TpRegion *__restrict__ reg,
                                                     const double *__restrict__ fvals,
                                                     TpRegionOut *__restrict__ out, const int *__restrict__ flag)
{
    size_t r = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nreg) return;
    gm_rule3(reg[r].vol, fvals + r * TP_NPTS_GM3, &out[r]);
    if (r == 0) out[0].flag |= *flag << 1;
}

int grid_for(size_t n, int block) { return (int)((n + block - 1) / block); }

}  // namespace

// The split of a point's nodes by launch size, from calls of B_kappa in one launch (us; FP64, FP32 in brackets) with one
// thread per (point, node), 8, 2 and 1 waves per point:
//      33 points:  21 (20)   65 (35)  133 (57)  249 (95)     4 096:  45 (36)    68 (38)  136 (62)  254 (102)
//     8 192:       90 (68)   93 (61)  160 (84)  278 (126)   32 768: 224 (159)  170 (107) 195 (116) 307 (156)
//    65 536:                299 (174) 310 (183) 357 (204)  131 072:            555 (326) 546 (322) 576 (335)
// one thread per (point, node) while its repeated set-up costs less than the shorter chain gains, 8 waves until the
// launch fills the chip with fewer, then 2.  A call is cut into launches of ~65 536 points, at most 16 of them, so the
// last line is crossed by calls of 2.1 million points and more: 4 194 304 points in 16 launches 10.9 ms FP64 with 8 waves,
// 10.6 with 2 (FP32 6.15 and 6.15); 8 388 608: 21.6 and 20.8 (12.4 and 12.2).
constexpr size_t kNodePoints = 4096, kWidePoints = 131072;

template <class T, bool MAP3>
static void launch_points(hipStream_t st, const TpNodeT<T> *nodes, const TpEHT<T> *eh, const PointTh &th, size_t npts,
                          const double *d_x, double *d_f, int mode, int *d_flag)
{
    const size_t groups = (npts + 63) / 64;
    if (npts <= kNodePoints)
        hipLaunchKernelGGL((k_points_nodes<T, MAP3>), dim3((unsigned)((npts + kNodePts - 1) / kNodePts)),
                           dim3(kNodeBlock), 0, st, nodes, eh, th, npts, d_x, d_f, mode, d_flag);
    else if (npts < kWidePoints)
        hipLaunchKernelGGL((k_points<T, 8, MAP3>), dim3((unsigned)groups), dim3(512), 0, st, nodes, eh, th, npts, d_x,
                           d_f, mode, d_flag);
    else
        hipLaunchKernelGGL((k_points<T, 2, MAP3>), dim3((unsigned)((groups + 1) / 2)), dim3(256), 0, st, nodes, eh, th,
                           npts, d_x, d_f, mode, d_flag);
}

template <bool MAP3>
static int launch_points_mode(const tp_cosmo *c, int icosmo, const PointTh &th, size_t npts, const double *d_x,
                              double *d_f, int mode, int *d_flag, hipStream_t st)
{
    if (npts == 0) return 0;
    const size_t o = (size_t)icosmo * TP_NNODES;
    if (mode == TP_MODE_FP32)
        launch_points<float, MAP3>(st, c->d_node32 + o, c->d_eh32 + icosmo, th, npts, d_x, d_f, mode, d_flag);
    else
        launch_points<double, MAP3>(st, c->d_node64 + o, c->d_eh64 + icosmo, th, npts, d_x, d_f, mode, d_flag);
    TP_HIP(hipGetLastError());
    return 0;
}

int tp_launch_map3_points(const tp_cosmo *c, int icosmo, const double *th, size_t npts, const double *d_x, double *d_f,
                          int mode, int *d_flag, hipStream_t st)
{
    return launch_points_mode<true>(c, icosmo, PointTh{{th[0], th[1], th[2]}}, npts, d_x, d_f, mode, d_flag, st);
}

int tp_launch_bkappa_points(const tp_cosmo *c, int icosmo, size_t npts, const double *d_l, double *d_out, int mode,
                            int *d_flag, hipStream_t st)
{
    return launch_points_mode<false>(c, icosmo, PointTh{}, npts, d_l, d_out, mode, d_flag, st);
}

// The launch shape of k_region_nodes, taken by rounds of up to 32 regions: those read their region records from host
// memory, every wave its own, so the shape's many waves cost more there than in a point call (one FP32 integral:
// 1.91 ms without it, 1.48 up to 32 regions; 220 integrals: 24.6, 24.7, and 26.5 up to 124 regions).
constexpr int kShapeNodes = 96;
constexpr size_t kNodeRegionPoints = 32 * TP_NPTS_GM3;

// one launch of the region-point kernel with LPP waves per point group
template <class T>
static void launch_region_points(hipStream_t st, int lpp, const TpNodeT<T> *nodes, const TpEHT<T> *eh, size_t nreg,
                                 const TpRegion *d_reg, const TpIntegralDesc *d_desc, double *d_fvals, int mode,
                                 int *d_flag)
{
    const size_t np = nreg * TP_NPTS_GM3;
    const size_t groups = (np + 63) / 64;
    switch (lpp) {
    case kShapeNodes:
        hipLaunchKernelGGL((k_region_nodes<T>), dim3((unsigned)((np + kNodePts - 1) / kNodePts)), dim3(kNodeBlock), 0,
                           st, nodes, eh, nreg, d_reg, d_desc, d_fvals, mode, d_flag);
        break;
    case 2:
        hipLaunchKernelGGL((k_region_points<T, 2>), dim3((unsigned)((groups + 1) / 2)), dim3(256), 0, st, nodes, eh,
                           nreg, d_reg, d_desc, d_fvals, mode, d_flag);
        break;
    case 4:
        hipLaunchKernelGGL((k_region_points<T, 4>), dim3((unsigned)groups), dim3(256), 0, st, nodes, eh, nreg, d_reg,
                           d_desc, d_fvals, mode, d_flag);
        break;
    case 8:
        hipLaunchKernelGGL((k_region_points<T, 8>), dim3((unsigned)groups), dim3(512), 0, st, nodes, eh, nreg, d_reg,
                           d_desc, d_fvals, mode, d_flag);
        break;
    case 16:
        hipLaunchKernelGGL((k_region_cached<T, 1>), dim3((unsigned)((nreg + kCacheReg - 1) / kCacheReg)), dim3(kCacheThreads),
                           0, st, nodes, eh, nreg, d_reg, d_desc, d_fvals, mode, d_flag);
        break;
    case 32:
        hipLaunchKernelGGL((k_region_cached<T, 2>), dim3((unsigned)((nreg + kCacheReg - 1) / kCacheReg)), dim3(2 * kCacheThreads),
                           0, st, nodes, eh, nreg, d_reg, d_desc, d_fvals, mode, d_flag);
        break;
    case 64:
        hipLaunchKernelGGL((k_region_cached<T, 4>), dim3((unsigned)((nreg + kCacheReg - 1) / kCacheReg)), dim3(4 * kCacheThreads),
                           0, st, nodes, eh, nreg, d_reg, d_desc, d_fvals, mode, d_flag);
        break;
    default:
        hipLaunchKernelGGL((k_region_points<T, 1>), dim3((unsigned)((groups + 3) / 4)), dim3(256), 0, st, nodes, eh,
                           nreg, d_reg, d_desc, d_fvals, mode, d_flag);
    }
}

// size bucket of a launch for the launch-shape table (points: < 32k, < 160k, < 640k, more)
static int region_bucket(size_t np) { return np < 32768 ? 0 : np < 163840 ? 1 : np < 655360 ? 2 : 3; }

int tp_region_lanes(tp_ctx *ctx, const tp_cosmo *c, int mode, size_t np);  // tp_tune below

int tp_launch_regions(tp_ctx *ctx, const tp_cosmo *c, size_t nreg, const TpRegion *d_reg,
                      const TpIntegralDesc *d_desc, double *d_fvals, TpRegionOut *d_out, int mode, int *d_flag,
                      hipEvent_t evm, hipStream_t st)
{
    if (nreg == 0) return 0;
    const int B = 256;
    size_t np = nreg * TP_NPTS_GM3;
    const int lpp = tp_region_lanes(ctx, c, mode, np);
    if (lpp < 0) return TP_EHIP;
    if (mode == TP_MODE_FP32)
        launch_region_points<float>(st, lpp, c->d_node32, c->d_eh32, nreg, d_reg, d_desc, d_fvals, mode, d_flag);
    else
        launch_region_points<double>(st, lpp, c->d_node64, c->d_eh64, nreg, d_reg, d_desc, d_fvals, mode, d_flag);
    TP_HIP(hipGetLastError());
    TP_HIP(hipEventRecord(evm, st));
    hipLaunchKernelGGL(k_region_rule, dim3(grid_for(nreg, B)), dim3(B), 0, st, nreg, d_reg, d_fvals, d_out,
                       d_flag);
    TP_HIP(hipGetLastError());
    return 0;
}

// ------------------------------------------------------------------ graph rounds
// The round's kernels as (function, grid, block) for graph kernel nodes, the same choice as
// launch_region_points makes.
template <class T>
static void region_points_shape(int lpp, size_t nreg, void **func, dim3 *grid, dim3 *block)
{
    const size_t groups = (nreg * TP_NPTS_GM3 + 63) / 64;
    switch (lpp) {
    case kShapeNodes:
        *func = (void *)k_region_nodes<T>;
        *grid = dim3((unsigned)((nreg * TP_NPTS_GM3 + kNodePts - 1) / kNodePts));
        *block = dim3(kNodeBlock);
        break;
    case 2:
        *func = (void *)k_region_points<T, 2>;
        *grid = dim3((unsigned)((groups + 1) / 2));
        *block = dim3(256);
        break;
    case 4:
        *func = (void *)k_region_points<T, 4>;
        *grid = dim3((unsigned)groups);
        *block = dim3(256);
        break;
    case 8:
        *func = (void *)k_region_points<T, 8>;
        *grid = dim3((unsigned)groups);
        *block = dim3(512);
        break;
    case 16:
    case 32:
    case 64:
        *func = lpp == 16 ? (void *)k_region_cached<T, 1> : lpp == 32 ? (void *)k_region_cached<T, 2>
                                                                       : (void *)k_region_cached<T, 4>;
        *grid = dim3((unsigned)((nreg + kCacheReg - 1) / kCacheReg));
        *block = dim3(kCacheThreads * lpp / 16);
        break;
    default:
        *func = (void *)k_region_points<T, 1>;
        *grid = dim3((unsigned)((groups + 3) / 4));
        *block = dim3(256);
    }
}

int tp_graph_round(tp_ctx *ctx, const tp_cosmo *c, TpLane &L, size_t nreg, int mode, hipStream_t st)
{
    if (nreg == 0) return 0;
    const int lpp = tp_region_lanes(ctx, c, mode, nreg * TP_NPTS_GM3);
    if (lpp < 0) return TP_EHIP;
    const bool f32 = mode == TP_MODE_FP32;
    // kernel arguments (copied into the node at set-up / update)
    const void *nodes = f32 ? (const void *)c->d_node32 : (const void *)c->d_node64;
    const void *eh = f32 ? (const void *)c->d_eh32 : (const void *)c->d_eh64;
    const TpRegion *reg = (const TpRegion *)L.d_regions.p;
    const TpIntegralDesc *desc = (const TpIntegralDesc *)ctx->d_desc.p;
    double *fv = (double *)L.d_fvals.p;
    TpRegionOut *ro = (TpRegionOut *)L.d_rout.p;
    int *flag = (int *)L.d_flag.p;
    int md = mode;
    size_t n = nreg;
    void *pargs[] = {(void *)&nodes, (void *)&eh, (void *)&n, (void *)&reg, (void *)&desc, (void *)&fv, (void *)&md,
                     (void *)&flag};
    const int *cflag = flag;
    void *rargs[] = {(void *)&n, (void *)&reg, (void *)&fv, (void *)&ro, (void *)&cflag};
    hipKernelNodeParams kp{}, kr{};
    if (f32) region_points_shape<float>(lpp, nreg, &kp.func, &kp.gridDim, &kp.blockDim);
    else region_points_shape<double>(lpp, nreg, &kp.func, &kp.gridDim, &kp.blockDim);
    kp.kernelParams = pargs;
    kr.func = (void *)k_region_rule;
    kr.gridDim = dim3(grid_for(nreg, 256));
    kr.blockDim = dim3(256);
    kr.kernelParams = rargs;
    const size_t bin = sizeof(TpRegion) * nreg, bout = sizeof(TpRegionOut) * nreg;
    bool fresh = false;
    if (L.exec) {  // update the instantiated chain; an update the runtime refuses rebuilds it
        hipError_t u = hipGraphExecMemcpyNodeSetParams1D(L.exec, L.n_in, L.d_regions.p, L.h_regions.p, bin,
                                                         hipMemcpyHostToDevice);
        if (u == hipSuccess) u = hipGraphExecKernelNodeSetParams(L.exec, L.n_pts, &kp);
        if (u == hipSuccess) u = hipGraphExecKernelNodeSetParams(L.exec, L.n_rule, &kr);
        if (u == hipSuccess)
            u = hipGraphExecMemcpyNodeSetParams1D(L.exec, L.n_out, L.h_rout.p, L.d_rout.p, bout, hipMemcpyDeviceToHost);
        if (u != hipSuccess) {
            (void)hipGetLastError();
            (void)hipGraphExecDestroy(L.exec);
            (void)hipGraphDestroy(L.graph);
            L.exec = nullptr;
            L.graph = nullptr;
            ctx->stats.graph_rebuilds += 1;
        }
    }
    if (!L.exec) {  // build the chain
        TP_HIP(hipGraphCreate(&L.graph, 0));
        hipGraphNode_t e0, em, e1, ed;
        TP_HIP(hipGraphAddMemcpyNode1D(&L.n_in, L.graph, nullptr, 0, L.d_regions.p, L.h_regions.p, bin,
                                       hipMemcpyHostToDevice));
        TP_HIP(hipGraphAddEventRecordNode(&e0, L.graph, &L.n_in, 1, L.ev0));
        TP_HIP(hipGraphAddKernelNode(&L.n_pts, L.graph, &e0, 1, &kp));
        TP_HIP(hipGraphAddEventRecordNode(&em, L.graph, &L.n_pts, 1, L.evm));
        TP_HIP(hipGraphAddKernelNode(&L.n_rule, L.graph, &em, 1, &kr));
        TP_HIP(hipGraphAddEventRecordNode(&e1, L.graph, &L.n_rule, 1, L.ev1));
        TP_HIP(hipGraphAddMemcpyNode1D(&L.n_out, L.graph, &e1, 1, L.h_rout.p, L.d_rout.p, bout, hipMemcpyDeviceToHost));
        TP_HIP(hipGraphAddEventRecordNode(&ed, L.graph, &L.n_out, 1, L.done));
        TP_HIP(hipGraphInstantiate(&L.exec, L.graph, nullptr, nullptr, 0));
        fresh = true;
    }
    (void)fresh;
    TP_HIP(hipGraphLaunch(L.exec, st));
    return 0;
}

// ------------------------------------------------------------------ launch-shape autotuner
// The waves-per-point split of k_region_points is chosen per launch-size bucket by timing every
// shape on a synthetic batch of that size, once per context and precision, on the first batched
// call (a few tens of ms).  Small launches (the tail rounds of a batch) favour more waves per
// point, large ones one wave.  Every shape computes the same bits, so the choice never changes a
// result.  tp_set_region_lanes forces one shape (0 restores tuning).
int tp_region_lanes(tp_ctx *ctx, const tp_cosmo *c, int mode, size_t np)
{
    if (ctx->region_lpp_force) return ctx->region_lpp_force;
    const int im = mode == TP_MODE_FP32 ? 1 : 0;
    if (mode == TP_MODE_ANALYTIC) return 1;
    if (!ctx->region_tuned[im]) {
        ctx->region_tuned[im] = true;  // also when tuning fails: then the default shape stays
        const size_t sizes[4] = {256, 2048, 8192, 32768};  // regions per bucket probe
        const size_t nmax = sizes[3];
        TpRegion *d_reg = nullptr;
        TpIntegralDesc *d_desc = nullptr;
        double *d_f = nullptr;
        int *d_fl = nullptr;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        bool ok = hipMalloc(&d_reg, nmax * sizeof(TpRegion)) == hipSuccess &&
                  hipMalloc(&d_desc, sizeof(TpIntegralDesc)) == hipSuccess &&
                  hipMalloc(&d_f, nmax * TP_NPTS_GM3 * sizeof(double)) == hipSuccess &&
                  hipMalloc(&d_fl, sizeof(int)) == hipSuccess && hipEventCreate(&e0) == hipSuccess &&
                  hipEventCreate(&e1) == hipSuccess;
        if (ok) {
            // regions spread in log ell over [1, 7000]^2 x [0, 2 pi] for radii (2', 4', 8'), cosmology 0
            std::vector<TpRegion> hr(nmax);
            for (size_t k = 0; k < nmax; ++k) {
                const double u = (double)((k * 2654435761u) % 1000003) / 1000003.0;
                const double v = (double)((k * 40503u + 17) % 999983) / 999983.0;
                const double ph = (double)((k * 97u + 5) % 1009) / 1009.0;
                TpRegion &R = hr[k];
                R.c[0] = std::exp(8.85 * u);
                R.c[1] = std::exp(8.85 * v);
                R.c[2] = 2 * M_PI * ph;
                R.hw[0] = 0.05 * R.c[0];
                R.hw[1] = 0.05 * R.c[1];
                R.hw[2] = 0.05;
                R.vol = 8 * R.hw[0] * R.hw[1] * R.hw[2];
                R.integral = 0;
                R.pad = 0;
            }
            const double arcmin = 2.9088820866e-4;
            TpIntegralDesc hd{{2 * arcmin, 4 * arcmin, 8 * arcmin}, 0, 0};
            ok = hipMemcpy(d_reg, hr.data(), nmax * sizeof(TpRegion), hipMemcpyHostToDevice) == hipSuccess &&
                 hipMemcpy(d_desc, &hd, sizeof(hd), hipMemcpyHostToDevice) == hipSuccess &&
                 hipMemset(d_fl, 0, sizeof(int)) == hipSuccess;
        }
        const int shapes[7] = {1, 2, 4, 8, 16, 32, 64};
        for (int b = 0; ok && b < 4; ++b) {
            float best = 0;
            for (int s = 0; ok && s < 7; ++s) {
                float ms = 0;
                for (int rep = 0; rep < 3; ++rep) {  // first launch warms up
                    ok = hipEventRecord(e0, ctx->stream) == hipSuccess;
                    if (im)
                        launch_region_points<float>(ctx->stream, shapes[s], c->d_node32, c->d_eh32, sizes[b], d_reg,
                                                    d_desc, d_f, TP_MODE_FP32, d_fl);
                    else
                        launch_region_points<double>(ctx->stream, shapes[s], c->d_node64, c->d_eh64, sizes[b], d_reg,
                                                     d_desc, d_f, TP_MODE_FP64, d_fl);
                    ok = ok && hipGetLastError() == hipSuccess && hipEventRecord(e1, ctx->stream) == hipSuccess &&
                         hipEventSynchronize(e1) == hipSuccess;
                    float t = 0;
                    if (ok && rep > 0 && hipEventElapsedTime(&t, e0, e1) == hipSuccess) ms += t;
                }
                if (ok && (s == 0 || ms < best)) {
                    best = ms;
                    ctx->region_lpp[im][b] = shapes[s];
                }
            }
        }
        if (d_reg) (void)hipFree(d_reg);
        if (d_desc) (void)hipFree(d_desc);
        if (d_f) (void)hipFree(d_f);
        if (d_fl) (void)hipFree(d_fl);
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        if (!ok) return tp_set_error(TP_EHIP, "tp_launch_regions: launch-shape tuning failed"), -1;
    }
    return np <= kNodeRegionPoints ? kShapeNodes : ctx->region_lpp[im][region_bucket(np)];
}

extern "C" int tp_set_region_lanes(tp_ctx *ctx, int lanes)
{
    if (!ctx || !(lanes == 0 || lanes == 1 || lanes == 2 || lanes == 4 || lanes == 8 || lanes == 16 || lanes == 32 ||
                  lanes == 64))
        return tp_set_error(TP_EINVAL,
                            "tp_set_region_lanes: lanes must be 0 (tuned), 1, 2, 4, 8, or 16, 32, 64 (region-cached)");
    ctx->region_lpp_force = lanes;
    return 0;
}

extern "C" int tp_region_lanes_table(tp_ctx *ctx, int mode, int *lanes4)
{
    if (!ctx || !lanes4 || (mode != TP_MODE_FP64 && mode != TP_MODE_FP32))
        return tp_set_error(TP_EINVAL, "tp_region_lanes_table: bad arguments");
    const int im = mode == TP_MODE_FP32 ? 1 : 0;
    for (int b = 0; b < 4; ++b) lanes4[b] = ctx->region_tuned[im] ? ctx->region_lpp[im][b] : 0;
    return 0;
}
