// Batched NR: many scenarios (perturbed injections, optional warm start) of
// one or more topologies solved in one persistent launch per topology.
//
// One workgroup owns one scenario for its whole NR solve and pulls the next
// scenario from a per-topology work counter when done, so uneven scenario
// sizes and iteration counts balance themselves.  Small topologies keep the
// whole working set (state vectors, mismatch, step, 2x2-block LU) in LDS;
// larger ones use a per-workgroup slice of a global workspace (L2 resident).
// The topology (Ybus, symbolic factor program) is shared read-only.
//
// Per scenario the pass is the same as the single-network solver
// (CPU/newtonRaphson.cpp:180-305): P,Q -> limits trigger -> mismatch ->
// convergence / switch at convergence -> Jacobian -> FP32 block LU ->
// solves -> FP64 refinement -> update.  A start that diverges (non-finite or
// huge mismatch, singular pivot, or no convergence) is retried from the flat
// start inside the same workgroup.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <climits>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "kernels_decl.hpp"
#include "kernels_impl.hpp"
#include "pf_internal.hpp"
#include "transfer.hpp"

using namespace pf;

namespace pf {

struct BatchTopo {
    DevNet N;
    DevSym Y;
    const double *V0flat, *th0flat;     // flat start of this topology
    int nslot;                          // Jacobian slots
    int nblk;                           // factor blocks: slots, row-ordered L, chain inverse
    DevFlat F;                          // flat pair program of the narrow top (F.fl_ptr null: none)
    int ck_max;                         // without it: most chunks of a level of the narrow top
};

struct BatchJob {
    int nscen;                          // scenarios of this topology
    const int *nscen_dev;               // when set: the count, read on the device
    const int *scen;                    // global scenario index
    const long long *off;               // bus offset of scenario s in the packed arrays
    const double *Pliq, *Qliq, *Qload;  // packed [sum nB]
    const double *V0, *th0;             // packed warm start, may be null
    double *Vout, *thout;               // packed results
    int *iters, *conv;
    double *maxmis;
    const long long *pv_off;            // PV offset of scenario s in the packed limQ
    unsigned char *limQout;             // packed final limQ [sum nPV]
    int *flips;                         // PV<->PQ flips of the final solve, per scenario
    int *counter;                       // work queue head
    char *gws;                          // global workspace (per workgroup slice)
    long long ws_bytes;                 // bytes per workgroup slice
    int max_iter, lim, refine;
    double tol, diverge;
};

constexpr int GL = 16;   // lanes per node in the in-workgroup LU and solves
// dense top block: at most kBatchChain nodes when the working set sits in
// LDS (MODE 2), kBatchChainWide otherwise; S is inverted in register tiles
// of up to kBatchTile<T> x kBatchTile<T> blocks per thread, or where the
// working set lives when the workgroup cannot cover it
constexpr int kBatchChain = 32;
constexpr int kBatchChainWide = 64;
template <typename T> constexpr int kBatchTile = 2;   // wider tiles spill in the persistent kernel
// up to 512 threads (MODE 1): as wide as 64 nodes take, in FP32
template <typename T, int MAXT> constexpr int kLeanTile = sizeof(T) == 8 ? 2 : MAXT <= 256 ? 4 : 3;
template <int MODE> constexpr int batch_chain_cap() { return MODE == 2 ? kBatchChain : kBatchChainWide; }
// levels of at least kWideLevel nodes: a lane group per node; narrower ones:
// the whole workgroup on the level's destinations.  A constant, not the
// number of lane groups, so that every workgroup size sums in the same order.
constexpr int kWideLevel = 32;
// the narrow levels at the top of the tree (below the dense block), when
// their update pairs are chunked: chunks of kBatchChunkPairs pairs, one lane
// group of kBatchChunkLanes per chunk (one pair per lane), at most
// kBatchMaxChunks chunks on a level (LDS partial sums; kernels whose working
// set lives in global memory only)
constexpr int kBatchChunkPairs = 8, kBatchChunkLanes = 8, kBatchMaxChunks = 512;
static_assert(kWideLevel <= 4 * kBatchChain, "the narrow-level pivots pass through the dense-top LDS buffer");
// update pairs loaded per round in the factorisation (registers are tight
// in the persistent kernel)
constexpr int kBatchUnroll = 1;

// per-scenario working set, in LDS or in a global slice
template <typename T>
struct Work {
    double *V, *th, *P, *Q, *ql, *g, *x, *r;
    double2 *E, *I;
    unsigned char *isq, *limQ;
    T *blk;
};

// nblk: factor blocks (Jacobian slots and the row-ordered copy of L)
template <typename T>
__host__ __device__ inline long long work_bytes(int nB, int n, int nPV, int nblk) {
    long long b = 0;
    b += 8LL * nB * 5;                 // V th P Q ql
    b += 8LL * 2 * n * 3;              // g x r
    b = (b + 15) & ~15LL;              // E and I hold double2: 16-byte aligned
    b += 16LL * nB * 2;                // E I
    b += (long long)sizeof(T) * 4 * nblk;
    b += nB + nPV + 16;
    return (b + 255) & ~255LL;
}

template <typename T>
__device__ __forceinline__ Work<T> carve(char *base, int nB, int n, int nPV, int nblk) {
    Work<T> w;
    char *p = base;
    auto take = [&](size_t bytes) { char *q = p; p += bytes; return q; };
    w.V = (double *)take(8 * (size_t)nB);
    w.th = (double *)take(8 * (size_t)nB);
    w.P = (double *)take(8 * (size_t)nB);
    w.Q = (double *)take(8 * (size_t)nB);
    w.ql = (double *)take(8 * (size_t)nB);
    w.g = (double *)take(16 * (size_t)n);
    w.x = (double *)take(16 * (size_t)n);
    w.r = (double *)take(16 * (size_t)n);
    p = base + ((p - base + 15) & ~(size_t)15);   // 8 mod 16 when nB is odd
    w.E = (double2 *)take(16 * (size_t)nB);
    w.I = (double2 *)take(16 * (size_t)nB);
    w.blk = (T *)take(sizeof(T) * 4 * (size_t)nblk);
    w.isq = (unsigned char *)take(nB);
    w.limQ = (unsigned char *)take(nPV);
    return w;
}

template <typename T>
__device__ __forceinline__ void wg_factor_node(const DevSym &Y, T *blk, int j, int lane, int *bad) {
    const int d0 = Y.fd_ptr[j], nd = Y.fd_ptr[j + 1] - d0;
    const int L0 = Y.n, U0 = Y.n + Y.nnzL;
    B4<T> dinv{0, 0, 0, 0};
    for (int base = 0; base < nd; base += GL) {
        const int t = base + lane;
        B4<T> a{0, 0, 0, 0}, u{0, 0, 0, 0};
        int p = -1;
        if (t < nd) {
            const int d = d0 + t;
            B4<T> sa{0, 0, 0, 0}, su{0, 0, 0, 0};
            if (t == 0) {
                pairs_acc<T, false, kBatchUnroll>(Y, blk, Y.fc_ptr[d], Y.fc_ptr[d + 1], 1, sa, su);
                a = load_b4(blk, j);
            } else {
                pairs_acc<T, true, kBatchUnroll>(Y, blk, Y.fc_ptr[d], Y.fc_ptr[d + 1], 1, sa, su);
                p = Y.colptr[j] + t - 1;
                a = load_b4(blk, L0 + p);
                u = load_b4(blk, U0 + p);
            }
            a = B4<T>{a.a - sa.a, a.b - sa.b, a.c - sa.c, a.d - sa.d};
            u = B4<T>{u.a - su.a, u.b - su.b, u.c - su.c, u.d - su.d};
        }
        if (base == 0) {
            B4<T> di{0, 0, 0, 0};
            if (lane == 0) {
                T det = a.a * a.d - a.b * a.c;
                if (!(det != (T)0) || !isfinite((double)det)) {
                    *bad = 1;
                    det = (T)1;
                }
                di = B4<T>{a.d / det, -a.b / det, -a.c / det, a.a / det};
                store_b4(blk, Y.di0 + j, di);
            }
            dinv.a = __shfl(di.a, 0, GL);
            dinv.b = __shfl(di.b, 0, GL);
            dinv.c = __shfl(di.c, 0, GL);
            dinv.d = __shfl(di.d, 0, GL);
        }
        if (t < nd && t > 0) {
            const B4<T> l = mul(a, dinv);
            store_b4(blk, L0 + p, l);
            store_b4(blk, U0 + Y.nnzL + Y.lr_pos[p], l);
            store_b4(blk, U0 + p, u);
        }
    }
}

// Narrow elimination-tree levels [l0, l1) (fewer than kWideLevel nodes
// each) by the whole workgroup, two barriers per level, with the same
// arithmetic as coop_factor_range: groups of G lanes take the level's
// destination blocks, the lanes of a group split the destination's update
// pairs (pair q + G*i for lane q) and reduce them in a fixed order; after a
// barrier the pivot's inverse is stored and each column block is scaled by
// it.  What is loaded is arranged for latency: the indices of a group's
// first destination on the next level and of each lane's first pair are
// loaded one level ahead, a destination's current blocks are loaded with its
// first pair's blocks, the updated pivots pass through LDS (s_piv, one per
// node of the level) and the first updated column block stays in registers,
// so the second half of a level waits on no global load.
template <typename T, int G>
__device__ __forceinline__ void wg_factor_narrow(const DevSym &Y, T *blk, int l0, int l1, int *bad, B4<T> *s_piv) {
    const int L0 = Y.n, U0 = Y.n + Y.nnzL, LR0 = Y.n + 2 * Y.nnzL, DI = Y.di0;
    const int grp = (int)threadIdx.x / G, lane = (int)threadIdx.x % G, ng = (int)blockDim.x / G;
    struct Dest {
        int j, t, q, qe, pa, pb, p;   // p: the column block's position (t > 0)
    };
    auto dest = [&](int e0, int e) {
        Dest r;
        r.j = Y.ld_node[e0 + e];
        const int d = Y.ld_d[e0 + e];
        r.t = d - Y.fd_ptr[r.j];
        r.q = Y.fc_ptr[d] + lane;
        r.qe = Y.fc_ptr[d + 1];
        r.pa = r.pb = 0;
        if (r.q < r.qe) {
            r.pa = Y.fc_a[r.q];
            r.pb = Y.fc_b[r.q];
        }
        r.p = r.t ? Y.colptr[r.j] + r.t - 1 : 0;
        return r;
    };
    Dest cur{};
    cur.j = -1;
    if (l0 < l1 && grp < Y.ld_ptr[l0 + 1] - Y.ld_ptr[l0]) cur = dest(Y.ld_ptr[l0], grp);
    for (int l = l0; l < l1; l++) {
        const int e0 = Y.ld_ptr[l], ne = Y.ld_ptr[l + 1] - e0, s0 = Y.lvl_ptr[l];
        Dest nxt{};
        nxt.j = -1;
        if (l + 1 < l1 && grp < Y.ld_ptr[l + 2] - Y.ld_ptr[l + 1]) nxt = dest(Y.ld_ptr[l + 1], grp);
        B4<T> keep{0, 0, 0, 0};   // the first destination's updated column block
        int keep_lrp = 0;
        for (int e = grp; e < ne; e += ng) {
            const Dest D = (e == grp) ? cur : dest(e0, e);
            B4<T> a{0, 0, 0, 0}, u{0, 0, 0, 0};
            // the destination's own blocks, loaded with its first pair's
            B4<T> v0{0, 0, 0, 0}, v1{0, 0, 0, 0};
            if (lane == 0) {
                v0 = load_b4(blk, D.t ? L0 + D.p : D.j);
                if (D.t) v1 = load_b4(blk, U0 + D.p);
            }
            const int lrp = (lane == 0 && D.t) ? Y.lr_pos[D.p] : 0;
            if (D.q < D.qe) {
                mma2(a, load_b4(blk, L0 + D.pa), load_b4(blk, U0 + D.pb));
                if (D.t != 0) mma2(u, load_b4(blk, L0 + D.pb), load_b4(blk, U0 + D.pa));
            }
            if (D.t == 0) pairs_acc<T, false, 1>(Y, blk, D.q + G, D.qe, G, a, u);
            else pairs_acc<T, true, 1>(Y, blk, D.q + G, D.qe, G, a, u);
            a = group_sum<T, G>(a);
            u = group_sum<T, G>(u);
            if (lane == 0) {
                if (D.t == 0) {
                    const B4<T> P{v0.a - a.a, v0.b - a.b, v0.c - a.c, v0.d - a.d};
                    store_b4(blk, D.j, P);
                    s_piv[D.j - s0] = P;
                } else {
                    const B4<T> Lb{v0.a - a.a, v0.b - a.b, v0.c - a.c, v0.d - a.d};
                    store_b4(blk, L0 + D.p, Lb);
                    store_b4(blk, U0 + D.p, B4<T>{v1.a - u.a, v1.b - u.b, v1.c - u.c, v1.d - u.d});
                    if (e == grp) {
                        keep = Lb;
                        keep_lrp = lrp;
                    }
                }
            }
        }
        __syncthreads();
        if (lane == 0) {
            for (int e = grp; e < ne; e += ng) {
                int j, t, p, lrp;
                B4<T> Lb;
                if (e == grp) {
                    j = cur.j; t = cur.t; p = cur.p; lrp = keep_lrp; Lb = keep;
                } else {
                    j = Y.ld_node[e0 + e];
                    t = Y.ld_d[e0 + e] - Y.fd_ptr[j];
                    p = t ? Y.colptr[j] + t - 1 : 0;
                    lrp = t ? Y.lr_pos[p] : 0;
                    Lb = t ? load_b4(blk, L0 + p) : B4<T>{0, 0, 0, 0};
                }
                const B4<T> P = s_piv[j - s0];
                T det = P.a * P.d - P.b * P.c;
                const bool sing = !(det != (T)0) || !isfinite((double)det);
                if (sing) det = (T)1;
                const B4<T> Pi{P.d / det, -P.b / det, -P.c / det, P.a / det};
                if (t == 0) {
                    if (sing) atomicOr(bad, 1);
                    store_b4(blk, DI + j, Pi);
                } else {
                    const B4<T> lb = mul(Lb, Pi);
                    store_b4(blk, L0 + p, lb);
                    store_b4(blk, LR0 + lrp, lb);
                }
            }
        }
        __syncthreads();
        cur = nxt;
    }
}

// Forward and backward sweeps, GL lanes per node.  The first entry of the
// first node a lane group takes on a level (index and factor block, which do
// not depend on x) is loaded one level ahead, so its latency overlaps the
// previous level's arithmetic and barrier; the summation order is the same
// as without it.
template <typename T>
__device__ __forceinline__ void wg_solve(const DevSym &Y, const T *blk, double *x, double *s_r) {
    const int grp = (int)threadIdx.x / GL, lane = (int)threadIdx.x % GL, ng = (int)blockDim.x / GL;
    const int LR0 = Y.n + 2 * Y.nnzL, U0 = Y.n + Y.nnzL;
    const int nl = Y.nlev_s;
    auto fetch_fwd = [&](int l, int &k, B4<T> &L) {
        k = -1;
        const int s = Y.lvl_ptr[l];
        if (grp < Y.lvl_ptr[l + 1] - s) {
            const int j = s + grp, q = Y.rs_ptr[j] + lane;
            if (q < Y.rs_ptr[j + 1]) {
                k = Y.rs_k[q];
                L = load_b4(blk, LR0 + q);
            }
        }
    };
    int pk = -1;
    B4<T> pL{0, 0, 0, 0};
    if (nl > 0) fetch_fwd(0, pk, pL);
    for (int l = 0; l < nl; l++) {
        int nk = -1;
        B4<T> nL{0, 0, 0, 0};
        if (l + 1 < nl) fetch_fwd(l + 1, nk, nL);
        const int s = Y.lvl_ptr[l], c = Y.lvl_ptr[l + 1] - s;
        for (int i = grp; i < c; i += ng) {
            const int j = (s + i);
            double a0 = 0, a1 = 0;
            int q = Y.rs_ptr[j] + lane;
            if (i == grp) {
                if (pk >= 0) {
                    a0 += (double)pL.a * x[2 * pk] + (double)pL.b * x[2 * pk + 1];
                    a1 += (double)pL.c * x[2 * pk] + (double)pL.d * x[2 * pk + 1];
                }
                q += GL;
            }
            for (; q < Y.rs_ptr[j + 1]; q += GL) {
                B4<T> L = load_b4(blk, LR0 + q);
                const int k = Y.rs_k[q];
                a0 += (double)L.a * x[2 * k] + (double)L.b * x[2 * k + 1];
                a1 += (double)L.c * x[2 * k] + (double)L.d * x[2 * k + 1];
            }
            a0 = xor_sum<GL>(a0);
            a1 = xor_sum<GL>(a1);
            if (lane == 0) {
                x[2 * j] -= a0;
                x[2 * j + 1] -= a1;
            }
        }
        __syncthreads();
        pk = nk;
        pL = nL;
    }
    auto fetch_bwd = [&](int l, int &r, B4<T> &U, B4<T> &D) {
        r = -1;
        const int s = Y.lvl_ptr[l];
        if (grp < Y.lvl_ptr[l + 1] - s) {
            const int j = s + grp, p = Y.colptr[j] + lane;
            if (lane == 0) D = load_b4(blk, Y.di0 + j);
            if (p < Y.colptr[j + 1]) {
                r = Y.rowind[p];
                U = load_b4(blk, U0 + p);
            }
        }
    };
    int pr = -1;
    B4<T> pU{0, 0, 0, 0}, pD{0, 0, 0, 0};
    if (nl > 0) fetch_bwd(nl - 1, pr, pU, pD);
    if (Y.ch_m > 0) chain_solve<T, GL>(Y, blk, x, s_r, Y.rs_ptr);
    for (int l = nl - 1; l >= 0; l--) {
        int nr = -1;
        B4<T> nU{0, 0, 0, 0}, nD{0, 0, 0, 0};
        if (l > 0) fetch_bwd(l - 1, nr, nU, nD);
        const int s = Y.lvl_ptr[l], c = Y.lvl_ptr[l + 1] - s;
        for (int i = grp; i < c; i += ng) {
            const int j = (s + i);
            double a0 = 0, a1 = 0;
            int p = Y.colptr[j] + lane;
            if (i == grp) {
                if (pr >= 0) {
                    a0 += (double)pU.a * x[2 * pr] + (double)pU.b * x[2 * pr + 1];
                    a1 += (double)pU.c * x[2 * pr] + (double)pU.d * x[2 * pr + 1];
                }
                p += GL;
            }
            for (; p < Y.colptr[j + 1]; p += GL) {
                B4<T> U = load_b4(blk, U0 + p);
                const int r = Y.rowind[p];
                a0 += (double)U.a * x[2 * r] + (double)U.b * x[2 * r + 1];
                a1 += (double)U.c * x[2 * r] + (double)U.d * x[2 * r + 1];
            }
            a0 = xor_sum<GL>(a0);
            a1 = xor_sum<GL>(a1);
            if (lane == 0) {
                const double y0 = x[2 * j] - a0, y1 = x[2 * j + 1] - a1;
                const B4<T> D = (i == grp) ? pD : load_b4(blk, Y.di0 + j);
                x[2 * j] = (double)D.a * y0 + (double)D.b * y1;
                x[2 * j + 1] = (double)D.c * y0 + (double)D.d * y1;
            }
        }
        __syncthreads();
        pr = nr;
        pU = nU;
        pD = nD;
    }
}

// Row or column pointers of the sweeps in 16 bits in LDS, or, past 65,535
// entries, where they are in memory.
struct RowPtr16 {
    const unsigned short *h;
    const int *g;
    bool packed;
    __device__ __forceinline__ int operator[](int i) const { return packed ? (int)h[i] : g[i]; }
};

// Forward and backward sweeps whose factor entries are loaded a level
// ahead (they do not depend on x).  The entries of a level are contiguous
// (rs_ptr / colptr in node order, nodes numbered level by level).  A level's
// width alone says how many lanes a node gets, lane i taking entries i,
// i + g, ..., so every launch shape sums alike: 16 lanes up to
// kSweepGroupLevel nodes, 4 up to 4 kSweepGroupLevel (256 threads take either
// at once), one above.  A node's first kSweepAhead entries a lane come from
// registers filled during the level before; one barrier per level.  (Wide
// levels went through LDS, an entry's product a lane and two barriers a page
// of them: 512 x 1,888 buses 4,230 us, now 4,130; 2,048 x 944 9,790, 9,500.)
constexpr int kSweepGroupLevel = 16, kSweepAhead = 2;

// one direction: ptr, idx, B0: the rows and L by rows, or the columns and U
// (BWD, where the sum also meets the node's inverse pivot)
template <typename T, bool BWD, typename PTR>
__device__ __forceinline__ void wg_sweep(const DevSym &Y, const T *blk, double *x, const PTR ptr, const int *idx, int B0,
                                         int nl) {
    const int tid = (int)threadIdx.x, bd = (int)blockDim.x;
    constexpr int RA = kSweepAhead;
    int pk[RA];
    B4<T> pB[RA], pD{0, 0, 0, 0};
    // the coming level: its first node and width, log2 of its lanes a node,
    // the entries of this lane's node (from this lane's first on)
    int ns = 0, nc = 0, ng = 0, ne = 0, ne1 = 0;
    auto level = [&](int i) __attribute__((always_inline)) { return BWD ? nl - 1 - i : i; };
    auto ahead = [&](int l) __attribute__((always_inline)) {
        ns = Y.lvl_ptr[l];
        nc = Y.lvl_ptr[l + 1] - ns;
        ng = nc <= kSweepGroupLevel ? 4 : nc <= 4 * kSweepGroupLevel ? 2 : 0;
        const int me = tid >> ng, lane = tid & ((1 << ng) - 1);
#pragma unroll
        for (int r = 0; r < RA; r++) pk[r] = -1;
        if (me < nc) {
            const int j = ns + me;
            ne = ptr[j] + lane;
            ne1 = ptr[j + 1];
#pragma unroll
            for (int r = 0; r < RA; r++) {
                const int e = ne + (r << ng);
                if (e < ne1) {
                    pk[r] = idx[e];
                    pB[r] = load_b4(blk, B0 + e);
                }
            }
            if (BWD && lane == 0) pD = load_b4(blk, Y.di0 + j);
        }
    };
    auto put = [&](int j, double y0, double y1, const B4<T> &D) __attribute__((always_inline)) {
        if (BWD) {
            x[2 * j] = (double)D.a * y0 + (double)D.b * y1;
            x[2 * j + 1] = (double)D.c * y0 + (double)D.d * y1;
        } else {
            x[2 * j] = y0;
            x[2 * j + 1] = y1;
        }
    };
    if (nl > 0) ahead(level(0));
    for (int i = 0; i < nl; i++) {
        const int s = ns, c = nc, sh = ng, e0 = ne, e1 = ne1;
        const int me = tid >> sh, lane = tid & ((1 << sh) - 1);
        int ck[RA];
        B4<T> cB[RA];
        double xk[RA][2];   // x of the first entries, read before the next level's requests
#pragma unroll
        for (int r = 0; r < RA; r++) {
            ck[r] = pk[r];
            cB[r] = pB[r];
            const int k = ck[r] >= 0 ? ck[r] : 0;
            xk[r][0] = x[2 * k];
            xk[r][1] = x[2 * k + 1];
        }
        const B4<T> myD = pD;
        // the node's own x: no earlier level of this sweep writes it
        const int jo = s + (me < c ? me : 0);
        const double xj0 = x[2 * jo], xj1 = x[2 * jo + 1];
        if (i + 1 < nl) ahead(level(i + 1));
        if (me < c) {
            double a0 = 0, a1 = 0;
#pragma unroll
            for (int r = 0; r < RA; r++)
                if (ck[r] >= 0) {
                    a0 += (double)cB[r].a * xk[r][0] + (double)cB[r].b * xk[r][1];
                    a1 += (double)cB[r].c * xk[r][0] + (double)cB[r].d * xk[r][1];
                }
            for (int e = e0 + (RA << sh); e < e1; e += 1 << sh) {
                const B4<T> L = load_b4(blk, B0 + e);
                const int k = idx[e];
                const double x0 = x[2 * k], x1 = x[2 * k + 1];
                a0 += (double)L.a * x0 + (double)L.b * x1;
                a1 += (double)L.c * x0 + (double)L.d * x1;
            }
            if (sh == 4) {
                a0 = xor_sum<GL>(a0);
                a1 = xor_sum<GL>(a1);
            } else if (sh == 2) {
                a0 = quad_sum(a0);
                a1 = quad_sum(a1);
            }
            if (lane == 0) put(jo, xj0 - a0, xj1 - a1, myD);
            if (sh == 0)
                for (int j = s + me + bd; j < s + c; j += bd) {
                    double b0 = 0, b1 = 0;
                    for (int e = ptr[j], ee = ptr[j + 1]; e < ee; e++) {
                        const B4<T> L = load_b4(blk, B0 + e);
                        const int k = idx[e];
                        const double x0 = x[2 * k], x1 = x[2 * k + 1];
                        b0 += (double)L.a * x0 + (double)L.b * x1;
                        b1 += (double)L.c * x0 + (double)L.d * x1;
                    }
                    put(j, x[2 * j] - b0, x[2 * j + 1] - b1, BWD ? load_b4(blk, Y.di0 + j) : B4<T>{0, 0, 0, 0});
                }
        }
        __syncthreads();
    }
}

template <typename T, typename PTR>
__device__ __forceinline__ void wg_solve_flat(const DevSym &Y, const T *blk, double *x, double *s_r, const PTR rs,
                                              const PTR cl) {
    wg_sweep<T, false>(Y, blk, x, rs, Y.rs_k, Y.n + 2 * Y.nnzL, Y.nlev_s);
    if (Y.ch_m > 0) chain_solve<T, GL>(Y, blk, x, s_r, rs);
    wg_sweep<T, true>(Y, blk, x, cl, Y.rowind, Y.n + Y.nnzL, Y.nlev_s);
}

// I = Y E and S = E conj(I): 4 lanes per row
template <typename T>
__device__ __forceinline__ void wg_pq(const DevNet &N, Work<T> &w) {
    // two rows a lane group at a time (r and r + rows_per), their entries
    // walked together so that their loads are in flight together; each row
    // sums in the same order as alone
    const int rows_per = (int)blockDim.x / 4;
    const int lane = (int)threadIdx.x & 3;
    for (int r0 = 0; r0 < N.nB; r0 += 2 * rows_per) {
        int row[2], e[2], e1[2];
        double ar[2] = {0, 0}, ai[2] = {0, 0};
#pragma unroll
        for (int u = 0; u < 2; u++) {
            row[u] = r0 + u * rows_per + (int)threadIdx.x / 4;
            const bool ok = row[u] < N.nB;
            e[u] = ok ? N.rowptr[row[u]] + lane : 0;
            e1[u] = ok ? N.rowptr[row[u] + 1] : 0;
        }
        while (e[0] < e1[0] || e[1] < e1[1]) {
#pragma unroll
            for (int u = 0; u < 2; u++)
                if (e[u] < e1[u]) {
                    const double2 Em = w.E[N.colind[e[u]]];
                    const double2 y = N.y[e[u]];
                    ar[u] += y.x * Em.x - y.y * Em.y;
                    ai[u] += y.x * Em.y + y.y * Em.x;
                    e[u] += 4;
                }
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            ar[u] = quad_sum(ar[u]);
            ai[u] = quad_sum(ai[u]);
            if (row[u] < N.nB && lane == 0) {
                const double2 Ek = w.E[row[u]];
                w.I[row[u]] = make_double2(ar[u], ai[u]);
                w.P[row[u]] = Ek.x * ar[u] + Ek.y * ai[u];
                w.Q[row[u]] = Ek.y * ar[u] - Ek.x * ai[u];
            }
        }
    }
}

// r = g - J x (FP64, complex voltages)
template <typename T>
__device__ __forceinline__ void wg_residual(const DevNet &N, Work<T> &w) {
    // two rows a lane group at a time, as in wg_pq
    const int rows_per = (int)blockDim.x / 4;
    const int lane = (int)threadIdx.x & 3;
    for (int r0 = 0; r0 < N.nB; r0 += 2 * rows_per) {
        int row[2], e[2], e1[2];
        bool active[2];
        double ar[2] = {0, 0}, ai[2] = {0, 0};
#pragma unroll
        for (int u = 0; u < 2; u++) {
            row[u] = r0 + u * rows_per + (int)threadIdx.x / 4;
            active[u] = row[u] < N.nB && row[u] != N.slack;
            e[u] = active[u] ? N.rowptr[row[u]] + lane : 0;
            e1[u] = active[u] ? N.rowptr[row[u] + 1] : 0;
        }
        while (e[0] < e1[0] || e[1] < e1[1]) {
#pragma unroll
            for (int u = 0; u < 2; u++)
                if (e[u] < e1[u]) {
                    const int m = N.colind[e[u]];
                    if (m != N.slack) {
                        const int jm = N.node_of_bus[m];
                        const double dth = w.x[2 * jm];
                        const double dv = w.isq[m] ? w.x[2 * jm + 1] : 0.0;
                        const double2 Em = w.E[m];
                        const double f = dv / w.V[m];
                        const double dr = Em.x * f - Em.y * dth, di = Em.y * f + Em.x * dth;
                        const double2 y = N.y[e[u]];
                        ar[u] += y.x * dr - y.y * di;
                        ai[u] += y.x * di + y.y * dr;
                    }
                    e[u] += 4;
                }
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            ar[u] = quad_sum(ar[u]);
            ai[u] = quad_sum(ai[u]);
            if (active[u] && lane == 0) {
                const int k = row[u], j = N.node_of_bus[k];
                const double dth = w.x[2 * j];
                const bool q = w.isq[k];
                const double dv = q ? w.x[2 * j + 1] : 0.0;
                const double2 Ek = w.E[k], Ik = w.I[k];
                const double f = dv / w.V[k];
                const double dr = Ek.x * f - Ek.y * dth, di = Ek.y * f + Ek.x * dth;
                const double sr = dr * Ik.x + di * Ik.y + Ek.x * ar[u] + Ek.y * ai[u];
                const double si = di * Ik.x - dr * Ik.y + Ek.y * ar[u] - Ek.x * ai[u];
                w.r[2 * j] = w.g[2 * j] - sr;
                w.r[2 * j + 1] = q ? w.g[2 * j + 1] - si : -w.x[2 * j + 1];
            }
        }
    }
}

// limits pass: mode 0 chkLimQ (or undo when !chk), flips accumulated in *flips
template <typename T>
__device__ __forceinline__ void wg_limits(const DevNet &N, Work<T> &w, const double *Qliq, const double *Qload,
                          bool chk, int *flips) {
    int f = 0;
    for (int i = threadIdx.x; i < N.nPV; i += blockDim.x) {
        const int b = N.pv_bus[i];
        const double qload = Qload[b], qmin = N.qmin[i], qmax = N.qmax[i];
        unsigned char lq = w.limQ[i];
        double qll = w.ql[b];
        if (!lq) {
            if (chk) {
                const double qg = w.Q[b] + qload;
                if (qg < qmin - kFolga) { qll = qmin - qload; lq = 1; f++; }
                else if (qg > qmax + kFolga) { qll = qmax - qload; lq = 1; f++; }
            }
        } else {
            if (qll == qmax - qload) {
                if (w.V[b] > N.vset[i] + kFolga) { lq = 0; qll = Qliq[b]; f++; }
            } else {
                if (w.V[b] < N.vset[i] - kFolga) { lq = 0; qll = Qliq[b]; f++; }
            }
        }
        w.limQ[i] = lq;
        w.ql[b] = qll;
        w.isq[b] = lq;
    }
    if (f) atomicAdd(flips, f);
}

template <typename T>
__device__ __forceinline__ void wg_set_E(const DevNet &N, Work<T> &w) {
    for (int k = threadIdx.x; k < N.nB; k += blockDim.x) {
        double s, c;
        sincos(w.th[k], &s, &c);
        w.E[k] = make_double2(w.V[k] * c, w.V[k] * s);
    }
}

// Starting state of one scenario
template <typename T>
__device__ __forceinline__ void wg_start(const BatchTopo &tp, Work<T> &w, const double *Qliq, const double *V0,
                                         const double *th0) {
    const DevNet &N = tp.N;
    // a warm start sets |V| of the PQ buses and the angles of the non-slack
    // buses; PV buses start at their setpoint and the slack at its data
    for (int k = threadIdx.x; k < N.nB; k += blockDim.x) {
        const bool pq = N.pv_of_bus[k] < 0 && k != N.slack;
        w.V[k] = pq ? V0[k] : tp.V0flat[k];
        w.th[k] = (k == N.slack) ? tp.th0flat[k] : th0[k];
        w.ql[k] = Qliq[k];
        w.isq[k] = pq ? 1 : 0;                                   // initLim: PQ buses only
    }
    for (int i = threadIdx.x; i < N.nPV; i += blockDim.x) w.limQ[i] = 0;
}

// One NR solve of one scenario by the whole workgroup from the state in w.
// Returns (via shared result) iterations, converged flag, final max mismatch,
// flips and whether a pivot failed (s_end, may be null).
// s_chain: LDS of the dense top and of a narrow level's pivots; s_ck: of the
// chunked narrow top, null: level by level throughout; rs, cl: row and column
// pointers of the flat sweeps.
template <typename T, int TMAX, typename PTR>
__device__ __forceinline__ void wg_nr(const BatchTopo &tp, const BatchJob &J, Work<T> &w, const double *Pliq,
                      const double *Qliq, const double *Qload,
                      int *s_it, int *s_conv, double *s_maxg, int *s_fl, int *s_end, B4<T> *s_chain, B4<T> *s_ck, int ck_max,
                      const PTR rs, const PTR cl) {
    const DevNet &N = tp.N;
    const DevSym &Y = tp.Y;
    __shared__ unsigned long long s_maxG_bits, s_maxDx_bits;
    __shared__ int s_bad, s_flips, s_sing;
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_maxDx_bits = 0;
        s_flips = 0;
        s_sing = 0;
    }
    __syncthreads();
    wg_set_E(N, w);
    __syncthreads();
    int it = 0, conv = 0;
    double maxG = 0;
    while (it < J.max_iter) {
        wg_pq(N, w);
        if (tid == 0) { s_maxG_bits = 0; s_bad = 0; }
        __syncthreads();
        if (J.lim && it >= 1) {
            const bool chk = u64_as_double(s_maxDx_bits) < 0.1;
            int any = 0;
            if (!chk)
                for (int i = tid; i < N.nPV; i += blockDim.x) any |= w.limQ[i];
            any = __syncthreads_or(any);
            if (chk || any) wg_limits(N, w, Qliq, Qload, chk, &s_flips);
            __syncthreads();
        }
        // mismatch
        {
            double m = 0.0;
            int bad = 0;
            for (int k = tid; k < N.nB; k += blockDim.x) {
                if (k == N.slack) continue;
                const int j = N.node_of_bus[k];
                const double gp = Pliq[k] - w.P[k];
                const double gq = w.isq[k] ? w.ql[k] - w.Q[k] : 0.0;
                w.g[2 * j] = gp;
                w.g[2 * j + 1] = gq;
                m = dmax_nan(m, dmax_nan(fabs(gp), fabs(gq)));
                const int i = N.pv_of_bus[k];
                if (i >= 0) {
                    const double qg = w.Q[k] + Qload[k];
                    bad |= (qg < N.qmin[i] - kFolga) || (qg > N.qmax[i] + kFolga);
                }
            }
            m = wave_max(m);
            bad = __any(bad);
            if ((tid & 63) == 0) {
                atomicMax(&s_maxG_bits, double_as_u64(m));
                if (bad) atomicOr(&s_bad, 1);
            }
        }
        __syncthreads();
        maxG = u64_as_double(s_maxG_bits);
        const int simple_bad = s_bad;
        __syncthreads();
        if (maxG <= J.tol) {
            if (J.lim && simple_bad) {                    // switch taken at convergence
                wg_limits(N, w, Qliq, Qload, true, &s_flips);
                if (tid == 0) s_maxDx_bits = 0;
                __syncthreads();
                it++;
                continue;
            }
            conv = 1;
            break;
        }
        if (J.diverge > 0 && !(maxG < J.diverge)) break;  // NaN or diverging: give up this start
        // Jacobian blocks, four slots a thread at a time so that their index
        // loads are in flight together
        constexpr int JF = 4;
        for (int s0 = tid; s0 < tp.nslot; s0 += JF * blockDim.x) {
            int es[JF];
#pragma unroll
            for (int r = 0; r < JF; r++) {
                const int s = s0 + r * (int)blockDim.x;
                es[r] = s < tp.nslot ? Y.slot_e[s] : -1;
            }
            int ks[JF], ms[JF];
            double2 ys[JF];
#pragma unroll
            for (int r = 0; r < JF; r++) {
                const int e = es[r] >= 0 ? es[r] : 0;
                ks[r] = N.coorow[e];
                ms[r] = N.colind[e];
                ys[r] = N.y[e];
            }
#pragma unroll
            for (int r = 0; r < JF; r++) {
            const int s = s0 + r * (int)blockDim.x, e = es[r];
            if (s >= tp.nslot) break;
            B4<T> out{0, 0, 0, 0};
            if (e >= 0) {
                const int k = ks[r], m = ms[r];
                const double2 y = ys[r];
                double H, Nn, M, L;
                if (k != m) {
                    const double2 Em = w.E[m], Ek = w.E[k];
                    const double tr = y.x * Em.x - y.y * Em.y, ti = y.x * Em.y + y.y * Em.x;
                    const double cr = Ek.x * tr + Ek.y * ti, ci = Ek.y * tr - Ek.x * ti;
                    const double vm = w.V[m];
                    H = ci; Nn = cr / vm; M = -cr; L = ci / vm;
                } else {
                    const double v = w.V[k], v2 = v * v, p = w.P[k], q = w.Q[k];
                    H = -q - v2 * y.y; Nn = (p + v2 * y.x) / v; M = p - v2 * y.x; L = (q - v2 * y.y) / v;
                }
                if (!w.isq[m]) { Nn = 0; L = 0; }
                if (!w.isq[k]) { M = 0; L = (k == m) ? 1.0 : 0.0; }
                out = B4<T>{(T)H, (T)Nn, (T)M, (T)L};
            }
            store_b4(w.blk, s, out);
            }
        }
        if (tid == 0) s_maxDx_bits = 0;
        __syncthreads();
        // factor, level by level
        // wide levels: a lane group per node; narrow levels: the whole
        // workgroup on the level's destinations (coop_factor_range)
        {
            const int grp = tid / GL, lane = tid % GL, ng = (int)blockDim.x / GL;
            for (int l = 0; l < Y.nlev_s;) {
                if (s_ck && tp.F.fl_ptr && l == tp.F.lv0 && ((size_t)w.x & 15) == 0) {   // flat pair lists
                    T *pa = reinterpret_cast<T *>(w.x);   // x and r: free until the solve
                    flat_factor_levels<T, 1>(Y, tp.F, w.blk, 0, tp.F.nsteps, &s_sing, pa,
                                                pa + 4 * (size_t)tp.F.max_pairs);
                    break;
                }
                if (s_ck && Y.ck_lvl && l >= Y.tail_start) {   // the chunked narrow top
                    chunk_factor_levels<T, kBatchChunkLanes, 1>(Y, w.blk, l, Y.nlev_s, &s_sing, s_ck,
                                                                  s_ck + ck_max, s_chain);
                    break;
                }
                const int s = Y.lvl_ptr[l], c = Y.lvl_ptr[l + 1] - s;
                if (c >= kWideLevel) {
                    for (int i = grp; i < c; i += ng) wg_factor_node(Y, w.blk, (s + i), lane, &s_sing);
                    __syncthreads();
                    l++;
                } else {   // a run of narrow levels
                    int l1 = l + 1;
                    while (l1 < Y.nlev_s && Y.lvl_ptr[l1 + 1] - Y.lvl_ptr[l1] < kWideLevel) l1++;
                    wg_factor_narrow<T, kCoopLanes>(Y, w.blk, l, l1, &s_sing, s_chain);
                    l = l1;
                }
            }
            if (Y.ch_m > 0) {
                chain_factor_mem<T, GL, kBatchUnroll, TMAX>(Y, w.blk, &s_sing, s_chain);
                __syncthreads();
            }
        }
        if (s_sing) break;
        for (int i = tid; i < 2 * Y.n; i += blockDim.x) w.x[i] = w.g[i];
        __syncthreads();
        if (s_ck) wg_solve_flat(Y, (const T *)w.blk, w.x, (double *)s_chain, rs, cl);
        else wg_solve(Y, (const T *)w.blk, w.x, (double *)s_chain);
        for (int q = 0; q < J.refine; q++) {
            wg_residual(N, w);
            __syncthreads();
            if (s_ck) wg_solve_flat(Y, (const T *)w.blk, w.r, (double *)s_chain, rs, cl);
            else wg_solve(Y, (const T *)w.blk, w.r, (double *)s_chain);
            for (int i = tid; i < 2 * Y.n; i += blockDim.x) w.x[i] += w.r[i];
            __syncthreads();
        }
        // update
        {
            double m = 0.0;
            for (int k = tid; k < N.nB; k += blockDim.x) {
                if (k == N.slack) continue;
                const int j = N.node_of_bus[k];
                const double dth = w.x[2 * j];
                double v = w.V[k];
                const double th = w.th[k] + dth;
                m = dmax_nan(m, fabs(dth));
                if (w.isq[k]) {
                    const double dv = w.x[2 * j + 1];
                    v += dv;
                    m = dmax_nan(m, fabs(dv));
                }
                w.V[k] = v;
                w.th[k] = th;
                double sn, cs;
                sincos(th, &sn, &cs);
                w.E[k] = make_double2(v * cs, v * sn);
            }
            m = wave_max(m);
            if ((tid & 63) == 0) atomicMax(&s_maxDx_bits, double_as_u64(m));
        }
        __syncthreads();
        it++;
    }
    if (tid == 0) {
        *s_it = it;
        *s_conv = conv;
        *s_maxg = maxG;
        *s_fl = s_flips;
        if (s_end) *s_end = s_sing;
    }
    __syncthreads();
}

// bytes of LDS that MODE 1 uses: the step vectors g, x, r and the level /
// row-structure metadata the triangular solves and the factor walk
template <typename T>
__host__ __device__ inline long long partial_lds_bytes(int n, int nlev) {
    long long b = 16LL * n * 3;                              // g x r
    b += 4LL * ((nlev + 1) * 2 + 3 * (n + 1));               // lvl_ptr ld_ptr rs_ptr colptr fd_ptr
    return (b + 255) & ~255LL;
}

// blocks of LDS of the dense top, or of a narrow level's pivots
__host__ __device__ inline int chain_lds_blocks(int ch_m) {
    return 4 * ch_m + 2 > kWideLevel ? 4 * ch_m + 2 : kWideLevel;
}

// LDS of MODE 1 up to 512 threads, where several workgroups share a CU: the
// step vectors x and r, the dense top's staging, the level pointers and,
// packed, the row and column pointers, and the partial sums of a chunked
// narrow top.  The rest of MODE 1's arrays is read where it is in memory.
template <typename T>
struct LeanLds {
    long long buf, ck, lvl, rs, cl, bytes;   // offsets, and the whole
    bool packed;
    __host__ __device__ LeanLds(int n, int nnzL, int nlev, int ch_m, int chunks) {
        buf = 32LL * n;
        ck = buf + (long long)sizeof(B4<T>) * chain_lds_blocks(ch_m);
        lvl = ck + (long long)sizeof(B4<T>) * 2 * chunks;
        rs = lvl + 4LL * (nlev + 1);
        packed = nnzL <= 65535;
        cl = rs + (packed ? 2LL * (n + 1) : 0);
        bytes = (cl + (packed ? 2LL * (n + 1) : 0) + 255) & ~255LL;
    }
};

// MODE 2: the whole per-scenario working set in LDS.
// MODE 1: working set in a global slice, except the step vectors and the
//         level / row-structure metadata, staged in LDS (latency of the
//         level-by-level walk); MODE 0: everything in the global slice.
// The float LDS-resident kernel at 256 threads keeps three waves per SIMD
// (three workgroups per CU, within 168 VGPRs): small networks are latency
// bound, so more resident scenarios per CU beat the few registers it costs.
// MODE 1 keeps four (128 VGPRs) at every size, so that two workgroups of 512
// or four of 256 share a CU, and up to 512 threads it takes less LDS for it
// (LeanLds: x, r and 16-bit pointers; g in the slice).  A pass waits on loads
// and barriers, which one workgroup alone does not cover: 2,048 x 944 buses in
// FP32 9,840 us one of 1024, 7,090 two of 512; 2,048 x 354 buses 3,070 us two
// of 256 at 183 VGPRs, 2,090 four at 128.
// LEVELS: the level-by-level program of the sets in LDS, also where such a set
// is asked to run in MODE 1 or 0 (one instantiation each, of 1024 threads), so
// that a topology's answers do not depend on the placement.
template <typename T, int MODE, int MAXT>
constexpr int batch_min_waves() { return MODE == 1 ? 4 : (MODE == 2 && MAXT == 256 && sizeof(T) == 4) ? 3 : 1; }

template <typename T, int MODE, int MAXT, bool LEVELS = MODE == 2>   // MAXT: largest workgroup (register budget)
__global__ void __launch_bounds__(MAXT, (batch_min_waves<T, MODE, MAXT>())) k_batch(BatchTopo tp0, BatchJob J) {
    extern __shared__ __align__(16) char smem[];
    __shared__ int s_item, s_it, s_conv, s_fl;
    constexpr bool lean = MODE == 1 && MAXT < 1024;                // its buffers are in smem (LeanLds)
    __shared__ B4<T> s_chain_own[lean ? 1 : 4 * batch_chain_cap<MODE>() + 2];   // dense top: row / column / pivot staging
    __shared__ B4<T> s_ck_own[lean || LEVELS ? 1 : 2 * kBatchMaxChunks];        // chunk partial sums (a, u)
    __shared__ double s_maxg;
    B4<T> *s_chain = s_chain_own, *s_ck = LEVELS ? nullptr : s_ck_own;
    const int ck_max = lean ? tp0.ck_max : kBatchMaxChunks;
    BatchTopo tp = tp0;
    const DevNet &N = tp.N;
    char *base = (MODE == 2) ? smem : J.gws + (long long)blockIdx.x * J.ws_bytes;
    Work<T> w = carve<T>(base, N.nB, tp.Y.n, N.nPV, tp.nblk);
    using Ptr = std::conditional_t<lean, RowPtr16, const int *>;
    Ptr rs, cl;
    if constexpr (lean) {
        const int n = tp.Y.n, nlev = tp.Y.nlev;
        const LeanLds<T> o(n, tp.Y.nnzL, nlev, tp.Y.ch_m, tp.ck_max);
        w.x = reinterpret_cast<double *>(smem);
        w.r = w.x + 2 * n;
        s_chain = reinterpret_cast<B4<T> *>(smem + o.buf);
        s_ck = reinterpret_cast<B4<T> *>(smem + o.ck);
        int *lvl = reinterpret_cast<int *>(smem + o.lvl);
        for (int i = threadIdx.x; i <= nlev; i += blockDim.x) lvl[i] = tp0.Y.lvl_ptr[i];
        tp.Y.lvl_ptr = lvl;
        unsigned short *r16 = reinterpret_cast<unsigned short *>(smem + o.rs);
        unsigned short *c16 = reinterpret_cast<unsigned short *>(smem + o.cl);
        if (o.packed)
            for (int i = threadIdx.x; i <= n; i += blockDim.x) {
                r16[i] = (unsigned short)tp0.Y.rs_ptr[i];
                c16[i] = (unsigned short)tp0.Y.colptr[i];
            }
        rs = RowPtr16{r16, tp0.Y.rs_ptr, o.packed};
        cl = RowPtr16{c16, tp0.Y.colptr, o.packed};
        __syncthreads();
    } else if constexpr (MODE == 1) {
        const int n = tp.Y.n, nlev = tp.Y.nlev;
        double *v = reinterpret_cast<double *>(smem);
        w.g = v;
        w.x = v + 2 * n;
        w.r = v + 4 * n;
        int *ip = reinterpret_cast<int *>(v + 6 * n);
        auto stage = [&](const int *src, int cnt) {
            int *dst = ip;
            for (int i = threadIdx.x; i < cnt; i += blockDim.x) dst[i] = src[i];
            ip += cnt;
            return (const int *)dst;
        };
        tp.Y.lvl_ptr = stage(tp0.Y.lvl_ptr, nlev + 1);
        tp.Y.ld_ptr = stage(tp0.Y.ld_ptr, nlev + 1);
        tp.Y.rs_ptr = stage(tp0.Y.rs_ptr, n + 1);
        tp.Y.colptr = stage(tp0.Y.colptr, n + 1);
        tp.Y.fd_ptr = stage(tp0.Y.fd_ptr, n + 1);
        __syncthreads();
    }
    if constexpr (!lean) {
        rs = tp.Y.rs_ptr;
        cl = tp.Y.colptr;
    }
    const int nscen = J.nscen_dev ? *J.nscen_dev : J.nscen;
    for (;;) {
        if (threadIdx.x == 0) s_item = atomicAdd(J.counter, 1);
        __syncthreads();
        const int item = s_item;
        __syncthreads();
        if (item >= nscen) break;                           // every wave reaches this exit
        const int sc = J.scen[item];
        const long long off = J.off[sc];
        const double *Pl = J.Pliq + off, *Ql = J.Qliq + off, *Qd = J.Qload + off;
        const bool warm = J.V0 != nullptr;
        int total_it = 0;
        // one call site (the solve is inlined once): the warm start, then,
        // when it does not converge, the flat-start fallback
        for (int attempt = warm ? 0 : 1; attempt < 2; ++attempt) {
            const bool from_warm = attempt == 0;
            wg_start(tp, w, Ql, from_warm ? J.V0 + off : tp.V0flat, from_warm ? J.th0 + off : tp.th0flat);
            wg_nr<T, lean ? kLeanTile<T, MAXT> : kBatchTile<T>>(tp, J, w, Pl, Ql, Qd, &s_it, &s_conv, &s_maxg, &s_fl,
                                                                (int *)nullptr, s_chain, s_ck, ck_max, rs, cl);
            total_it += s_it;
            if (s_conv) break;                              // shared: uniform over the workgroup
        }
        for (int k = threadIdx.x; k < N.nB; k += blockDim.x) {
            J.Vout[off + k] = w.V[k];
            J.thout[off + k] = w.th[k];
        }
        const long long pvo = J.pv_off[sc];
        for (int i = threadIdx.x; i < N.nPV; i += blockDim.x) J.limQout[pvo + i] = w.limQ[i];
        if (threadIdx.x == 0) {
            J.iters[sc] = total_it;
            J.conv[sc] = s_conv;
            J.maxmis[sc] = s_maxg;
            J.flips[sc] = s_fl;
        }
        __syncthreads();
    }
}

// The whole NR loop of the single-network solver in one workgroup, the
// working set in LDS: from the solver's state and back to it, the outcome
// into *out (host memory).  A pass across the GPU is some twenty dependent
// launches, about 100 us whatever the size; here it is a barrier a step, 22 us
// at 14 buses and 50 at 118 (FP64), bound by the chain of levels.  A solve
// with its state read, FP64, 4 passes at 14 buses and 6 above, replayed graphs
// across the GPU -> one workgroup: 14 buses 431 -> 170 us, 57 buses
// 488 -> 212, 118 buses 704 -> 384, 236 buses 904 -> 635; mixed 354 buses
// 1,252 -> 949, the largest that fits.  The line is the LDS: all that fits is
// faster here.
template <typename T>
__global__ void __launch_bounds__(512) k_solve_wg(BatchTopo tp, BatchJob J, DevState S, Ctl *out) {
    extern __shared__ __align__(16) char smem[];
    __shared__ int s_it, s_conv, s_fl, s_end;
    __shared__ B4<T> s_chain[4 * kBatchChain + 2];
    __shared__ double s_maxg;
    const DevNet &N = tp.N;
    Work<T> w = carve<T>(smem, N.nB, tp.Y.n, N.nPV, tp.nblk);
    for (int k = threadIdx.x; k < N.nB; k += blockDim.x) {
        w.V[k] = S.V[k];
        w.th[k] = S.th[k];
        w.ql[k] = S.QliqLim[k];
        w.isq[k] = S.isq[k];
    }
    for (int i = threadIdx.x; i < N.nPV; i += blockDim.x) w.limQ[i] = S.limQ[i];
    wg_nr<T, kBatchTile<T>>(tp, J, w, S.Pliq, S.Qliq, S.Qload, &s_it, &s_conv, &s_maxg, &s_fl, &s_end, s_chain,
                            (B4<T> *)nullptr, 0, tp.Y.rs_ptr, tp.Y.colptr);
    for (int k = threadIdx.x; k < N.nB; k += blockDim.x) {
        S.V[k] = w.V[k];
        S.th[k] = w.th[k];
        S.E[k] = w.E[k];
        S.QliqLim[k] = w.ql[k];
        S.isq[k] = w.isq[k];
    }
    for (int i = threadIdx.x; i < N.nPV; i += blockDim.x) S.limQ[i] = w.limQ[i];
    if (threadIdx.x == 0) {
        out->it = s_it + s_end;   // a pass whose factors fail counts, its step is not taken
        out->done = s_conv;
        out->singular = s_end;
        out->maxG = s_maxg;
        out->flips = s_fl;
    }
}

// ------------------------------------------------------------ fixed scratch
// The allocation-free batch entry point keeps its per-call tables (packed
// offsets, per-network scenario lists, work counters) and the per-workgroup
// working-set slices in this fixed array, one copy per GPU, held until the
// process ends.  Host code must use the address hipGetSymbolAddress returns
// for the current device (noalloc_scratch), never the array's name.
constexpr long long kScratchBytes = 64LL << 20;
constexpr int kScratchHeader = 1024;        // counts [64], counters [64], invalid flag
static __device__ __align__(256) char scratch[kScratchBytes];

struct NoallocNets {
    int n_nets;
    int nB[64], nPV[64];
};

// exclusive prefix of v over the workgroup (1024 threads at most); *total:
// the sum over all threads
__device__ long long block_scan_excl(long long v, long long *total) {
    __shared__ long long buf[1024];
    const int t = threadIdx.x;
    buf[t] = v;
    __syncthreads();
    for (int d = 1; d < (int)blockDim.x; d <<= 1) {
        const long long a = t >= d ? buf[t - d] : 0;
        __syncthreads();
        buf[t] += a;
        __syncthreads();
    }
    const long long incl = buf[t];
    *total = buf[blockDim.x - 1];
    __syncthreads();
    return incl - v;
}

// One workgroup: the packed bus / PV offsets of every scenario, the list of
// scenarios of network i (in order) at scen + i * n_scen with its length in
// count[i], the work counters cleared, and a flag for net_of entries outside
// [0, n_nets) (those scenarios are left unsolved).
__global__ void __launch_bounds__(1024) k_noalloc_tables(const int *net_of, int n_scen, NoallocNets nn,
                                                         long long *off, long long *pvoff, int *scen,
                                                         int *count, int *counter, int *invalid) {
    const int T = blockDim.x, t = threadIdx.x;
    const int per = (n_scen + T - 1) / T;
    const int s0 = min(n_scen, t * per), s1 = min(n_scen, s0 + per);
    long long a = 0, b = 0;
    int bad = 0;
    for (int s = s0; s < s1; s++) {
        const int k = net_of[s];
        if (k < 0 || k >= nn.n_nets) { bad = 1; continue; }
        a += nn.nB[k];
        b += nn.nPV[k];
    }
    long long ta, tb;
    long long ea = block_scan_excl(a, &ta), eb = block_scan_excl(b, &tb);
    for (int s = s0; s < s1; s++) {
        const int k = net_of[s];
        off[s] = ea;
        pvoff[s] = eb;
        if (k < 0 || k >= nn.n_nets) continue;
        ea += nn.nB[k];
        eb += nn.nPV[k];
    }
    bad = __syncthreads_or(bad);
    for (int i = 0; i < nn.n_nets; i++) {
        long long c = 0, tot;
        for (int s = s0; s < s1; s++) c += net_of[s] == i;
        long long e = block_scan_excl(c, &tot);
        for (int s = s0; s < s1; s++)
            if (net_of[s] == i) scen[(long long)i * n_scen + e++] = s;
        if (t == 0) {
            count[i] = (int)tot;
            counter[i] = 0;
        }
    }
    if (t == 0) *invalid = bad;
}

__global__ void k_zero_int(int *p, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// The instantiation for a precision, working-set placement, workgroup size and
// program (levels: of a set that fits in LDS): compiled for at most 256, 512 or 1024 threads, so that smaller
// workgroups get the larger register budget.
using BatchKernel = void (*)(BatchTopo, BatchJob);
template <typename T, int MODE>
BatchKernel batch_kernel_t(int block) {
    if (block <= 256) return k_batch<T, MODE, 256>;
    if (block <= 512) return k_batch<T, MODE, 512>;
    return k_batch<T, MODE, 1024>;
}
inline BatchKernel batch_kernel(bool mixed, int mode, int block, bool levels) {
    if (levels && mode == 1) return mixed ? k_batch<float, 1, 1024, true> : k_batch<double, 1, 1024, true>;
    if (levels && mode == 0) return mixed ? k_batch<float, 0, 1024, true> : k_batch<double, 0, 1024, true>;
    if (mixed)
        return mode == 2 ? batch_kernel_t<float, 2>(block)
                         : mode == 1 ? batch_kernel_t<float, 1>(block) : batch_kernel_t<float, 0>(block);
    return mode == 2 ? batch_kernel_t<double, 2>(block)
                     : mode == 1 ? batch_kernel_t<double, 1>(block) : batch_kernel_t<double, 0>(block);
}

// Starting state of scenario s (one workgroup each) from row s of a device
// array of network outputs, de-normalised as the inference's outputs are.
__global__ void k_start_from_rows(const float *Y, long long ld, int v_col, int th_col, const float *mu,
                                  const float *sd, const long long *off, int n_scen, long long total, double *V0,
                                  double *T0) {
    const int s = (int)blockIdx.x;
    const long long o = off[s], nb = (s + 1 < n_scen ? off[s + 1] : total) - o;
    const float *row = Y + (long long)s * ld;
    for (long long i = threadIdx.x; i < nb; i += blockDim.x) {
        V0[o + i] = (double)(row[v_col + i] * sd[v_col + i] + mu[v_col + i]);
        T0[o + i] = (double)(row[th_col + i] * sd[th_col + i] + mu[th_col + i]);
    }
}

}  // namespace pf

// ======================================================================== host

namespace {
#define BHIP(expr)                                                                 \
    do {                                                                           \
        hipError_t e_ = (expr);                                                    \
        if (e_ != hipSuccess) {                                                    \
            pf::set_last_error(std::string(#expr) + ": " + hipGetErrorString(e_));     \
            return PF_DEVICE_ERROR;                                                \
        }                                                                          \
    } while (0)
#define BCHK(expr)                  \
    do {                            \
        pf_status s_ = (expr);      \
        if (s_ != PF_OK) return s_; \
    } while (0)
// Largest working set held in LDS (MODE 2): two workgroups of it, with the
// kernel's static LDS, share the 160 KiB of a CU.  118 buses in FP64 take
// 71 KiB: 333 scenarios 411 us there, 475 us at the best MODE 1 shape.  A
// set that leaves one workgroup per CU gains nothing: 236 buses in FP32
// (80 KiB) 1,740 us in LDS, 1,140 us in MODE 1.
constexpr long long kLdsLimit = 75 * 1024;
// Sets up to here take no other placement; the larger ones do on request.
constexpr long long kLdsOnly = 64 * 1024;
}  // namespace

// LDS bytes of k_solve_wg for a network, 0 where it does not run (the working
// set beyond the device's LDS, or a dense top past its staging)
long long pf::solve_wg_lds(const pf_network &net, const Symbolic &s, bool mixed, long long max_lds) {
    const long long b = mixed ? work_bytes<float>(net.nB, s.n, net.nPV, s.nblk())
                              : work_bytes<double>(net.nB, s.n, net.nPV, s.nblk());
    return b <= max_lds && s.ch_m <= kBatchChain ? b : 0;
}

pf_status pf::solve_wg_allow(bool mixed, long long bytes) {
    BHIP(hipFuncSetAttribute(mixed ? (const void *)k_solve_wg<float> : (const void *)k_solve_wg<double>,
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    return PF_OK;
}

pf_status pf::launch_solve_wg(const DevNet &N, const DevSym &Y, const DevState &S, int nblk, const pf_options &opt,
                              bool mixed, long long lds, Ctl *out, hipStream_t st) {
    BatchTopo tp{};
    tp.N = N;
    tp.Y = Y;
    tp.nslot = Y.nslot;
    tp.nblk = nblk;
    BatchJob J{};
    J.max_iter = opt.no_max_iter;
    J.lim = opt.lim_inj_reat ? 1 : 0;
    J.refine = mixed ? opt.refine_steps : 0;
    J.tol = opt.tolerancia;
    J.diverge = 0;   // run to max_iter, as the kernels across the GPU do
    if (mixed) k_solve_wg<float><<<1, 512, (size_t)lds, st>>>(tp, J, S, out);
    else k_solve_wg<double><<<1, 512, (size_t)lds, st>>>(tp, J, S, out);
    BHIP(hipGetLastError());
    return PF_OK;
}

namespace {
std::mutex g_scratch_mu;
char *g_scratch_ptr[64] = {};   // address of `scratch` on each device

// once per device, with that device current: the device address of the
// fixed scratch array
pf_status noalloc_setup(int device) {
    if (device < 0 || device >= 64) return PF_INVALID_ARG;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return PF_OK;
    void *p = nullptr;
    BHIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[device] = (char *)p;
    return PF_OK;
}
}  // namespace

struct BatchNet {
    pf_network net;
    YPattern yp;
    Symbolic sym;
    BatchTopo tp{};
    bool lds = false;          // the whole working set fits in LDS (MODE 2)
    long long partial = 0;     // MODE 1 LDS bytes, 0 if it does not fit
    int mode = 0;              // k_batch MODE
    long long shm = 0;         // dynamic LDS bytes
    int block = 256;
    int grid = 0;
    int per_cu = 1;            // workgroups per CU the grid is sized for
    int occ[3][17] = {};       // workgroups per CU by mode and block / 64, 0: not asked for yet
    long long ws = 0;
    std::vector<int> scen;
    // device
    int *d_scen = nullptr;
    char *d_ws = nullptr;
    size_t ws_cap = 0;         // bytes allocated at d_ws
};

struct pf_batch {
    int device = 0;
    pf_options opt;
    std::vector<std::unique_ptr<BatchNet>> nets;
    std::vector<void *> allocs;
    hipStream_t st[2] = {nullptr, nullptr};
    hipEvent_t ev_fork = nullptr, ev_mid = nullptr, ev_join = nullptr, t0 = nullptr, t1 = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    int n_scen = 0;
    long long total = 0;
    std::vector<long long> off, pv_off;
    std::vector<int> net_of;
    long long total_pv = 0;
    double *d_P = nullptr, *d_Q = nullptr, *d_L = nullptr, *d_V0 = nullptr, *d_T0 = nullptr;
    double *warm_V0 = nullptr, *warm_T0 = nullptr;
    double *d_V = nullptr, *d_T = nullptr, *d_mm = nullptr;
    int *d_it = nullptr, *d_cv = nullptr, *d_counter = nullptr, *d_fl = nullptr;
    long long *d_off = nullptr, *d_pvoff = nullptr;
    unsigned char *d_lq = nullptr;
    int cus = 0;
    PinnedSlots slots;

    template <typename T>
    pf_status alloc(T **p, size_t n) {
        void *q = nullptr;
        BHIP(hipMalloc(&q, sizeof(T) * std::max<size_t>(n, 1)));
        allocs.push_back(q);
        *p = (T *)q;
        return PF_OK;
    }
    template <typename T>
    pf_status upload(T **p, const std::vector<T> &v) {
        BCHK(alloc(p, v.size()));
        if (!v.empty()) BHIP(hipMemcpy(*p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
        return PF_OK;
    }
    PackedUploads plan;   // a network's small arrays, until add_net copies them
    template <typename T>
    pf_status plan_array(T **p, const std::vector<T> &v) {
        if (!PackedUploads::small(v)) return upload(p, v);
        plan.add(p, v);
        return PF_OK;
    }
    ~pf_batch() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        for (hipEvent_t e : {ev_fork, ev_mid, ev_join, t0, t1})
            if (e) (void)hipEventDestroy(e);
        for (void *p : allocs) (void)hipFree(p);
        for (auto &nb : nets)
            if (nb->d_ws) (void)hipFree(nb->d_ws);
        for (auto s : st)
            if (s) (void)hipStreamDestroy(s);
    }
    pf_status add_net(const pf_network &net);
    pf_status launch_net(size_t i, hipStream_t s);
    pf_status launch_all();
    pf_status configure(BatchNet &nb, int mode, int block, int per_cu);
    long long shm_bytes(const BatchNet &nb, int mode, int block) const;
    pf_status occupancy(BatchNet &nb, int mode, int block, int *per_cu);
    pf_status default_shape(BatchNet &nb, int nscen, int *block, int *per_cu);
    void drop_graph() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        gexec = nullptr;
        graph = nullptr;
    }
};

pf_status pf_batch::add_net(const pf_network &src) {
    auto b = std::make_unique<BatchNet>();
    int max_lds_i = 0;
    BHIP(hipDeviceGetAttribute(&max_lds_i, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
    const long long max_lds = max_lds_i - 8192;   // room for the kernel's static LDS
    b->net = src;
    b->yp = build_ypattern(src);
    // tail_start: the first level of the narrow top (fewer than kWideLevel
    // nodes per level up to the dense block)
    b->sym = analyze(src, b->yp, kWideLevel - 1, opt.lu_blocked ? kBatchChain : 0, 16);
    {   // a working set beyond LDS runs in MODE 1 / 0, whose kernels take a wider dense top
        const bool mx = opt.precision != PF_FP64;
        const long long w0 = mx ? work_bytes<float>(src.nB, b->sym.n, src.nPV, b->sym.nblk())
                                : work_bytes<double>(src.nB, b->sym.n, src.nPV, b->sym.nblk());
        if (w0 > kLdsLimit && opt.lu_blocked)
            dense_top(b->sym, kBatchChainWide, 64);
    }
    chunk_tail(b->sym, kBatchChunkPairs);
    if (!b->sym.level_ordered()) {
        pf::set_last_error("symbolic analysis: nodes not numbered level by level");
        return PF_INVALID_ARG;
    }
    const pf_network &net = b->net;
    const YPattern &yp = b->yp;
    const Symbolic &sym = b->sym;
    const int nB = net.nB, n = sym.n, sl = net.slack;
    std::vector<int> node_of_bus(nB, -1), pv_of_bus(nB, -1);
    for (int k = 0; k < nB; k++)
        if (k != sl) node_of_bus[k] = sym.iperm[k - (k > sl)];
    for (int i = 0; i < net.nPV; i++) pv_of_bus[net.pv[i]] = i;
    DevNet &N = b->tp.N;
    DevSym &Y = b->tp.Y;
    N.nB = nB; N.nL = net.nL; N.slack = sl; N.nPV = net.nPV; N.n = n;
    BCHK(plan_array((int **)&N.rowptr, yp.rowptr));
    BCHK(plan_array((int **)&N.colind, yp.colind));
    BCHK(plan_array((int **)&N.coorow, yp.coorow));
    BCHK(plan_array((int **)&N.ydiag, yp.diag));
    BCHK(plan_array((int **)&N.yc_ptr, yp.contrib_ptr));
    BCHK(plan_array((int **)&N.yc, yp.contrib));
    BCHK(plan_array((double **)&N.br_r, net.r));
    BCHK(plan_array((double **)&N.br_x, net.x));
    BCHK(plan_array((double **)&N.br_b, net.bch));
    BCHK(plan_array((double **)&N.br_tr, net.tap_re));
    BCHK(plan_array((double **)&N.br_ti, net.tap_im));
    BCHK(plan_array((double **)&N.gsh, net.gsh));
    BCHK(plan_array((double **)&N.bsh, net.bsh));
    BCHK(alloc(&N.y, yp.nnz));
    BCHK(plan_array((int **)&N.node_of_bus, node_of_bus));
    N.bus_of_node = nullptr;
    BCHK(plan_array((int **)&N.pv_bus, net.pv));
    BCHK(plan_array((int **)&N.pv_of_bus, pv_of_bus));
    BCHK(plan_array((double **)&N.qmin, net.Qmin));
    BCHK(plan_array((double **)&N.qmax, net.Qmax));
    BCHK(plan_array((double **)&N.vset, net.Vset));
    Y.n = n; Y.nnzL = sym.nnzL; Y.nslot = sym.nslot(); Y.nlev = sym.nlev;
    Y.ch_m = sym.ch_m; Y.ch_c0 = sym.ch_c0; Y.nlev_s = sym.nlev_s; Y.di0 = sym.di0();
    BCHK(plan_array((int **)&Y.ch_split, sym.ch_split));
    BCHK(plan_array((int **)&Y.colptr, sym.colptr));
    BCHK(plan_array((int **)&Y.rowind, sym.rowind));
    Y.pcol = nullptr;
    BCHK(plan_array((int **)&Y.lvl_ptr, sym.lvl_ptr));
    BCHK(plan_array((int **)&Y.lvl_nodes, sym.lvl_nodes));
    BCHK(plan_array((int **)&Y.fd_ptr, sym.fd_ptr));
    BCHK(plan_array((int **)&Y.fc_ptr, sym.fc_ptr));
    BCHK(plan_array((int **)&Y.fc_a, sym.fc_a));
    BCHK(plan_array((int **)&Y.fc_b, sym.fc_b));
    BCHK(plan_array((int **)&Y.rs_ptr, sym.rs_ptr));
    BCHK(plan_array((int **)&Y.rs_k, sym.rs_k));
    BCHK(plan_array((int **)&Y.rs_p, sym.rs_p));
    BCHK(plan_array((int **)&Y.lr_pos, sym.lr_pos));
    BCHK(plan_array((int **)&Y.slot_e, sym.slot_e));
    BCHK(plan_array((int **)&Y.ld_ptr, sym.ld_ptr));
    BCHK(plan_array((int **)&Y.ld_node, sym.ld_node));
    BCHK(plan_array((int **)&Y.ld_d, sym.ld_d));
    Y.tail_start = sym.tail_start;
    Y.te0 = sym.ld_ptr[sym.tail_start];
    Y.ck_lvl = Y.ck_q0 = Y.ck_q1 = Y.te_node = Y.te_p = Y.te_ck = nullptr;
    if (opt.lu_blocked && sym.ck_max <= kBatchMaxChunks && !sym.ck_q0.empty()) {
        BCHK(plan_array((int **)&Y.ck_lvl, sym.ck_lvl));
        BCHK(plan_array((int **)&Y.ck_q0, sym.ck_q0));
        BCHK(plan_array((int **)&Y.ck_q1, sym.ck_q1));
        BCHK(plan_array((int **)&Y.te_node, sym.te_node));
        BCHK(plan_array((int **)&Y.te_p, sym.te_p));
        BCHK(plan_array((int **)&Y.te_ck, sym.te_ck));
    }
    // the factorisation as flat pair lists, its products in the step vectors
    // x and r (4 n doubles, free during the factorisation): from the first
    // level, wide levels cut into steps whose products fit there, unless
    // that takes over half as many steps again as there are levels (a step
    // costs two barriers and a round of loads), else from the narrow top,
    // uncut.  1,888 buses in FP32, 38 steps for 33 levels, 100 scenarios:
    // 2,040 us; level by level below the top 2,360
    b->tp.F = DevFlat{};
    if (opt.lu_blocked && sym.tail_start < sym.nlev_s) {
        const bool mx = opt.precision != PF_FP64;
        auto need = [&](const FlatTail &f) {
            return mx ? flat_tail_lds<float>(f.max_pairs, f.max_col) : flat_tail_lds<double>(f.max_pairs, f.max_col);
        };
        const int step_blocks = (int)(32LL * sym.n / (mx ? 16 : 32));
        FlatTail ft = flat_tail(sym, 0, false, step_blocks);
        if (need(ft) > 32LL * sym.n || 2 * ft.fl_ptr.size() > 3 * (size_t)sym.nlev_s + 2)
            ft = flat_tail(sym, sym.tail_start, false, INT_MAX);
        if (need(ft) <= 32LL * sym.n) {
            DevFlat &F = b->tp.F;
            F.lv0 = ft.lv0;
            F.nsteps = (int)ft.fl_ptr.size() - 1;
            F.max_pairs = ft.max_pairs;
            F.max_col = ft.max_col;
            F.de_sentinel = ft.de_ptr.back();
            BCHK(plan_array((int **)&F.fl_ptr, ft.fl_ptr));
            BCHK(plan_array((int **)&F.fl_split, ft.fl_split));
            BCHK(plan_array((int **)&F.fl_a, ft.fl_a));
            BCHK(plan_array((int **)&F.fl_b, ft.fl_b));
            BCHK(plan_array((int **)&F.fl_s, ft.fl_s));
            BCHK(plan_array((int **)&F.fl_w, ft.fl_w));
            BCHK(plan_array((int **)&F.de_ptr, ft.de_ptr));
            BCHK(plan_array((int **)&F.de_node, ft.de_node));
            BCHK(plan_array((int **)&F.de_p, ft.de_p));
            BCHK(plan_array((int **)&F.de_q0, ft.de_q0));
            BCHK(plan_array((int **)&F.de_ext, ft.de_ext));
            BCHK(plan_array((int **)&F.de_lo, ft.de_lo));
            BCHK(plan_array((int **)&F.de_hi, ft.de_hi));
            BCHK(plan_array((int **)&F.de_dlo, ft.de_dlo));
            BCHK(plan_array((int **)&F.de_dhi, ft.de_dhi));
            BCHK(plan_array((int **)&F.de_lr, ft.de_lr));
            BCHK(plan_array((int **)&F.st_g, ft.st_g));
        }
    }
    BCHK(plan_array((double **)&b->tp.V0flat, net.V));
    BCHK(plan_array((double **)&b->tp.th0flat, net.theta));
    {   // from here on the pointers are set
        char *d = nullptr;
        BCHK(alloc(&d, plan.bytes()));
        BHIP(plan.copy_to(d));
    }
    b->tp.ck_max = Y.ck_lvl && !b->tp.F.fl_ptr ? sym.ck_max : 0;
    b->tp.nslot = sym.nslot();
    b->tp.nblk = sym.nblk();
    k_ybus<<<(yp.nnz + 255) / 256, 256, 0, st[0]>>>(N, yp.nnz);
    BHIP(hipGetLastError());
    BHIP(hipStreamSynchronize(st[0]));
    const bool mixed = opt.precision != PF_FP64;
    b->ws = mixed ? work_bytes<float>(nB, n, net.nPV, sym.nblk())
                  : work_bytes<double>(nB, n, net.nPV, sym.nblk());
    b->lds = b->ws <= kLdsLimit;
    if (b->lds)
        for (int blk : {256, 512, 1024})
            BHIP(hipFuncSetAttribute((const void *)batch_kernel(mixed, 2, blk, true),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsLimit));
    b->block = b->lds ? 256 : 1024;
    if (b->lds) {
        b->mode = 2;
        b->shm = b->ws;
    }
    if (b->ws > kLdsOnly) {
        long long pb = mixed ? partial_lds_bytes<float>(n, sym.nlev) : partial_lds_bytes<double>(n, sym.nlev);
        hipError_t e = hipSuccess;
        if (pb <= max_lds)
            for (int blk : {256, 512, 1024})
                if (e == hipSuccess)
                    e = hipFuncSetAttribute((const void *)batch_kernel(mixed, 1, blk, b->lds),
                                            hipFuncAttributeMaxDynamicSharedMemorySize,
                                            (int)(blk > 512 || b->lds ? pb : max_lds));
        if (e != hipSuccess) (void)hipGetLastError();
        b->partial = pb <= max_lds && e == hipSuccess ? pb : 0;
        if (!b->lds) {
            b->mode = b->partial ? 1 : 0;
            b->shm = b->partial;
        }
    }
    nets.push_back(std::move(b));
    return PF_OK;
}

// dynamic LDS of k_batch<T, mode> at this block size
long long pf_batch::shm_bytes(const BatchNet &nb, int mode, int block) const {
    if (mode != 1) return mode == 2 ? nb.ws : 0;
    if (block > 512 || nb.lds) return nb.partial;
    const Symbolic &y = nb.sym;
    const int ck = nb.tp.ck_max;
    return opt.precision != PF_FP64 ? LeanLds<float>(y.n, y.nnzL, y.nlev, y.ch_m, ck).bytes
                                    : LeanLds<double>(y.n, y.nnzL, y.nlev, y.ch_m, ck).bytes;
}

// resident workgroups per CU of k_batch<T, mode> at this block size
pf_status pf_batch::occupancy(BatchNet &nb, int mode, int block, int *per_cu) {
    int &known = nb.occ[mode][block / 64];
    if (known) {
        *per_cu = known;
        return PF_OK;
    }
    const bool mixed = opt.precision != PF_FP64;
    const size_t shm = (size_t)shm_bytes(nb, mode, block);
    int pc = 0;
    BHIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&pc, (const void *)batch_kernel(mixed, mode, block, nb.lds), block,
                                                      shm));
    *per_cu = known = pc;
    return PF_OK;
}

// The launch shape of nscen scenarios when none was chosen.  A scenario alone
// on its CU is fastest in a wide workgroup; with more scenarios than CUs it
// pays to keep several narrow ones resident, whose barriers and loads
// overlap, as long as they fit (118 buses, FP64: 24 scenarios 320 us at 512
// threads, 373 at 256; 333 scenarios 601 at 512 and one per CU, 411 at 256
// and two per CU).
//   LDS (MODE 2): 512 threads up to one scenario per CU, 256 above; up to 64
//   nodes and more scenarios than fit at once, 128 (57 buses, FP32, 1,500
//   scenarios: 463 -> 339 us).
//   MODE 1 / 0: 1024 threads, one per CU, up to one scenario per CU.  With
//   more, in MODE 1, two of 512 as long as a slice of global workspace stays
//   within kSlicePair: beyond, 512 of them are so far out of the 256 MB
//   Infinity Cache that nothing is gained (1,024 scenarios, FP32: 472 buses
//   2,410 -> 1,690 us, 944 4,580 -> 3,550, 1,416 5,920 -> 5,190, 1,888 (716 KB)
//   7,800 -> 7,640; FP64: 708 buses 3,740 -> 3,260, 1,180 6,920 -> 6,780, 1,416
//   8,740 -> 8,860); with more than two per CU, four of 256 where they fit,
//   up to kSliceQuad (FP32: 354 buses 1,390 -> 1,070, 708 2,160 -> 1,970, 944
//   3,550 -> 3,650; FP64: 354 buses 1,650 -> 1,420, 472 2,190 -> 2,100).
constexpr long long kSlicePair = 768 * 1024, kSliceQuad = 320 * 1024;
pf_status pf_batch::default_shape(BatchNet &nb, int nscen, int *block, int *per_cu) {
    int occ = 0;
    if (nb.mode == 2) {
        *block = nscen <= cus ? 512 : 256;
        BCHK(occupancy(nb, 2, *block, &occ));
        if (nscen > occ * cus && nscen > cus && nb.sym.n <= 64) {
            *block = 128;
            BCHK(occupancy(nb, 2, *block, &occ));
        }
        *per_cu = occ;
        return PF_OK;
    }
    *block = 1024;
    *per_cu = 1;
    if (nb.mode != 1 || nscen <= cus) return PF_OK;
    if (nscen > 2 * cus && nb.ws <= kSliceQuad) {
        BCHK(occupancy(nb, 1, 256, &occ));
        if (occ >= 4) {
            *block = 256;
            *per_cu = 4;
            return PF_OK;
        }
    }
    if (nb.ws <= kSlicePair) {
        BCHK(occupancy(nb, 1, 512, &occ));
        if (occ >= 2) {
            *block = 512;
            *per_cu = 2;
        }
    }
    return PF_OK;
}

// launch shape of one topology: mode, workgroup size and workgroups per CU
// (capped by occupancy); a larger global workspace replaces the one before,
// with the streams idle and the graph that names it dropped by the caller.
pf_status pf_batch::configure(BatchNet &nb, int mode, int block, int per_cu) {
    auto refuse = [&](const char *why) {
        pf::set_last_error(std::string("batch launch shape (mode ") + std::to_string(mode) + ", block " +
                           std::to_string(block) + "): " + why);
        return PF_INVALID_ARG;
    };
    if (mode == 2 && !nb.lds) return refuse("the working set does not fit in LDS");
    if (mode != 2 && nb.ws <= kLdsOnly) return refuse("a working set up to 64 KiB takes LDS only: use mode 2");
    if (mode == 1 && nb.partial == 0) return refuse("mode 1 is for working sets whose step vectors fit in LDS");
    if (block < 64 || block > 1024 || block % 64) return refuse("block must be a multiple of 64 up to 1024");
    // the sweeps of modes 1 and 0 give each node of a narrow level its own 16 lanes
    if (mode != 2 && block < GL * kSweepGroupLevel) return refuse("modes 1 and 0 take at least 256 threads");
    int occ = 0;
    BCHK(occupancy(nb, mode, block, &occ));
    if (occ < 1) return refuse("no workgroup fits on a CU (registers or LDS)");
    per_cu = per_cu <= 0 ? occ : std::min(per_cu, occ);
    const int grid = std::max(1, std::min<int>((int)nb.scen.size(), per_cu * cus));
    if (mode != 2) {   // before anything changes: on failure the shape stays as it was
        const size_t need = (size_t)grid * (size_t)nb.ws;
        if (need > nb.ws_cap) {
            void *p = nullptr;
            BHIP(hipMalloc(&p, need));
            if (nb.d_ws) (void)hipFree(nb.d_ws);
            nb.d_ws = (char *)p;
            nb.ws_cap = need;
        }
    }
    nb.mode = mode;
    nb.block = block;
    nb.per_cu = per_cu;
    nb.shm = shm_bytes(nb, mode, block);
    nb.grid = grid;
    return PF_OK;
}

pf_status pf_batch::launch_net(size_t i, hipStream_t s) {
    const bool mixed = opt.precision != PF_FP64;
    {
        BatchNet &b = *nets[i];
        if (b.scen.empty()) return PF_OK;
        BatchJob J{};
        J.nscen = (int)b.scen.size();
        J.scen = b.d_scen;
        J.off = d_off;
        J.Pliq = d_P; J.Qliq = d_Q; J.Qload = d_L;
        J.V0 = d_V0; J.th0 = d_T0;
        J.Vout = d_V; J.thout = d_T;
        J.iters = d_it; J.conv = d_cv; J.maxmis = d_mm;
        J.pv_off = d_pvoff; J.limQout = d_lq; J.flips = d_fl;
        J.counter = d_counter + i;
        J.gws = b.d_ws;
        J.ws_bytes = b.ws;
        J.max_iter = opt.no_max_iter;
        J.lim = opt.lim_inj_reat ? 1 : 0;
        J.refine = mixed ? opt.refine_steps : 0;
        J.tol = opt.tolerancia;
        J.diverge = 1e6;
        const size_t shm = (size_t)b.shm;
        BatchTopo tp = b.tp;
        void *args[] = {&tp, &J};
        BHIP(hipLaunchKernel((const void *)batch_kernel(mixed, b.mode, b.block, b.lds), dim3(b.grid), dim3(b.block), args,
                             b.mode == 0 ? 0 : shm, s));
    }
    return PF_OK;
}

pf_status pf_batch::launch_all() {
    BHIP(hipEventRecord(ev_fork, st[0]));
    BHIP(hipStreamWaitEvent(st[1], ev_fork, 0));
    k_zero_int<<<1, 64, 0, st[0]>>>(d_counter, (int)nets.size());
    BHIP(hipEventRecord(ev_mid, st[0]));
    BHIP(hipStreamWaitEvent(st[1], ev_mid, 0));
    // the largest topology first: its few long-running workgroups take their
    // CUs before the small topology's many short ones fill the rest, so the
    // two launches overlap instead of the long one waiting for a full GPU
    std::vector<size_t> order(nets.size());
    for (size_t i = 0; i < order.size(); i++) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t c) { return nets[a]->net.nB > nets[c]->net.nB; });
    for (size_t r = 0; r < order.size(); r++) BCHK(launch_net(order[r], st[r & 1]));
    BHIP(hipEventRecord(ev_join, st[1]));
    BHIP(hipStreamWaitEvent(st[0], ev_join, 0));
    return PF_OK;
}

pf_status pf::batch_start_from_rows(pf_batch *b, int device, int rows, const float *Y, long long ld, int v_col,
                                    int th_col, const float *mu, const float *sd, void *stream) {
    if (!b || !b->n_scen || !Y || !mu || !sd || v_col < 0 || th_col < 0) return PF_INVALID_ARG;
    if (device != b->device) {
        pf::set_last_error("warm start: the network and the batch are on different GPUs");
        return PF_INVALID_ARG;
    }
    if (rows != b->n_scen) {
        pf::set_last_error("warm start: one row per batch scenario");
        return PF_INVALID_ARG;
    }
    int nbmax = 0;
    for (int s : b->net_of) nbmax = std::max(nbmax, b->nets[s]->net.nB);
    if ((long long)v_col + nbmax > ld || (long long)th_col + nbmax > ld) {
        pf::set_last_error("warm start: a row holds fewer outputs than a scenario's buses");
        return PF_INVALID_ARG;
    }
    BHIP(hipSetDevice(b->device));
    const size_t tot = (size_t)b->total;
    if (!b->warm_V0) {
        BCHK(b->alloc(&b->warm_V0, tot));
        BCHK(b->alloc(&b->warm_T0, tot));
    }
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    k_start_from_rows<<<b->n_scen, 256, 0, st>>>(Y, ld, v_col, th_col, mu, sd, b->d_off, b->n_scen, b->total,
                                                b->warm_V0, b->warm_T0);
    BHIP(hipGetLastError());
    BHIP(hipStreamSynchronize(st));
    const bool had_warm = b->d_V0 != nullptr;
    b->d_V0 = b->warm_V0;
    b->d_T0 = b->warm_T0;
    if (!had_warm) b->drop_graph();   // kernel arguments change: capture again
    return PF_OK;
}

extern "C" {

pf_status pf_batch_create(const pf_network *const *nets, int n_nets, const pf_options *opt, int device,
                          pf_batch **out) {
    if (!nets || n_nets <= 0 || n_nets > 64 || !opt || !out) return PF_INVALID_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return PF_DEVICE_ERROR;
    auto b = std::make_unique<pf_batch>();
    b->device = device;
    b->opt = *opt;
    BHIP(hipSetDevice(device));
    for (auto &s : b->st) BHIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    BHIP(hipEventCreateWithFlags(&b->ev_fork, hipEventDisableTiming));
    BHIP(hipEventCreateWithFlags(&b->ev_mid, hipEventDisableTiming));
    BHIP(hipEventCreateWithFlags(&b->ev_join, hipEventDisableTiming));
    BHIP(hipEventCreate(&b->t0));
    BHIP(hipEventCreate(&b->t1));
    BHIP(hipDeviceGetAttribute(&b->cus, hipDeviceAttributeMultiprocessorCount, device));
    BHIP(b->slots.reserve());   // not at the first results
    BCHK(noalloc_setup(device));
    for (int i = 0; i < n_nets; i++) {
        if (!nets[i] || nets[i]->nB < 2 || nets[i]->slack < 0) return PF_INVALID_ARG;
        BCHK(b->add_net(*nets[i]));
    }
    BCHK(b->alloc(&b->d_counter, 64));
    *out = b.release();
    return PF_OK;
}

void pf_batch_destroy(pf_batch *b) {
    if (!b) return;
    (void)hipSetDevice(b->device);
    delete b;
}

pf_status pf_batch_set_scenarios(pf_batch *b, int n_scen, const int *net_of, const double *Pliq,
                                 const double *Qliq, const double *Qload, const double *V0,
                                 const double *theta0) {
    if (!b || n_scen <= 0 || !net_of || !Pliq || !Qliq || !Qload || ((V0 == nullptr) != (theta0 == nullptr)))
        return PF_INVALID_ARG;
    BHIP(hipSetDevice(b->device));
    const bool first = b->n_scen == 0;
    if (!first) {
        // a later call refreshes the data of the same scenario layout
        if (n_scen != b->n_scen || !std::equal(net_of, net_of + n_scen, b->net_of.begin())) {
            pf::set_last_error("pf_batch_set_scenarios: a later call must keep the first call's layout");
            return PF_INVALID_ARG;
        }
    } else {
        b->n_scen = n_scen;
        b->net_of.assign(net_of, net_of + n_scen);
        b->off.resize(n_scen);
        b->pv_off.resize(n_scen);
        long long tot = 0, tot_pv = 0;
        for (auto &nb : b->nets) nb->scen.clear();
        for (int s = 0; s < n_scen; s++) {
            if (net_of[s] < 0 || net_of[s] >= (int)b->nets.size()) {
                b->n_scen = 0;
                pf::set_last_error("pf_batch_set_scenarios: net_of holds an index outside the batch's networks");
                return PF_INVALID_ARG;
            }
            b->off[s] = tot;
            b->pv_off[s] = tot_pv;
            tot += b->nets[net_of[s]]->net.nB;
            tot_pv += b->nets[net_of[s]]->net.nPV;
            b->nets[net_of[s]]->scen.push_back(s);
        }
        b->total = tot;
        b->total_pv = tot_pv;
        BCHK(b->alloc(&b->d_P, tot));
        BCHK(b->alloc(&b->d_Q, tot));
        BCHK(b->alloc(&b->d_L, tot));
        BCHK(b->alloc(&b->d_V, tot));
        BCHK(b->alloc(&b->d_T, tot));
        BCHK(b->alloc(&b->d_mm, n_scen));
        BCHK(b->alloc(&b->d_it, n_scen));
        BCHK(b->alloc(&b->d_cv, n_scen));
        BCHK(b->alloc(&b->d_fl, n_scen));
        BCHK(b->alloc(&b->d_lq, tot_pv));
        BCHK(b->upload(&b->d_off, b->off));
        BCHK(b->upload(&b->d_pvoff, b->pv_off));
        for (auto &nbp : b->nets) {
            BatchNet &nb = *nbp;
            if (nb.scen.empty()) continue;
            BCHK(b->upload(&nb.d_scen, nb.scen));
            // default shape from the scenario count (pf_batch_autotune refines it)
            int block = 0, per_cu = 0;
            BCHK(b->default_shape(nb, (int)nb.scen.size(), &block, &per_cu));
            BCHK(b->configure(nb, nb.mode, block, per_cu));
        }
    }
    const size_t tot = (size_t)b->total;
    const CopyPiece in[3] = {{(void *)Pliq, b->d_P, sizeof(double) * tot},
                             {(void *)Qliq, b->d_Q, sizeof(double) * tot},
                             {(void *)Qload, b->d_L, sizeof(double) * tot}};
    BHIP(b->slots.send(in, 3, b->st[0]));
    const bool had_warm = b->d_V0 != nullptr;
    if (V0) {
        if (!b->warm_V0) {
            BCHK(b->alloc(&b->warm_V0, tot));
            BCHK(b->alloc(&b->warm_T0, tot));
        }
        BHIP(hipMemcpy(b->warm_V0, V0, sizeof(double) * tot, hipMemcpyHostToDevice));
        BHIP(hipMemcpy(b->warm_T0, theta0, sizeof(double) * tot, hipMemcpyHostToDevice));
        b->d_V0 = b->warm_V0;
        b->d_T0 = b->warm_T0;
    } else {
        b->d_V0 = b->d_T0 = nullptr;
    }
    if (had_warm != (b->d_V0 != nullptr)) b->drop_graph();   // kernel arguments change: capture again
    return PF_OK;
}

pf_status pf_batch_solve(pf_batch *b, double *elapsed_ms) {
    if (!b || !b->n_scen) return PF_INVALID_ARG;
    BHIP(hipSetDevice(b->device));
    if (!b->gexec) {
        BHIP(hipStreamBeginCapture(b->st[0], hipStreamCaptureModeThreadLocal));
        pf_status s = b->launch_all();
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(b->st[0], &g);
        if (s != PF_OK) return s;
        BHIP(e);
        b->graph = g;
        BHIP(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
    }
    BHIP(hipEventRecord(b->t0, b->st[0]));
    BHIP(hipGraphLaunch(b->gexec, b->st[0]));
    BHIP(hipEventRecord(b->t1, b->st[0]));
    BHIP(hipEventSynchronize(b->t1));
    float ms = 0;
    BHIP(hipEventElapsedTime(&ms, b->t0, b->t1));
    if (elapsed_ms) *elapsed_ms = ms;
    return PF_OK;
}

// ------------------------------------------------------------- autotuner
// For every topology of the current scenario set: time one launch of its
// persistent kernel (alone, HIP events on one stream) for each candidate
// launch shape -- kernel MODE (working set in LDS / partly in LDS / global),
// workgroup size, and for LDS topologies the resident workgroups per CU --
// keep the fastest, and remember it in a text cache keyed by the device, the
// kernels' version, the topology's sizes, the numeric options and the scenario
// count, so later runs apply it without measuring.
}  // extern "C"

namespace {

// of k_batch's timing: goes up with a change that may move the fastest shape
constexpr int kTuneVersion = 2;

std::string tune_key(const pf_batch &b, const BatchNet &nb, const char *arch) {
    char k[512];
    std::snprintf(k, sizeof k,
                  "%s kernels=%d cus=%d nB=%d n=%d nnzL=%d nlev=%d nPV=%d prec=%d refine=%d lim=%d maxit=%d nscen=%zu",
                  arch, kTuneVersion, b.cus, nb.net.nB, nb.sym.n, nb.sym.nnzL, nb.sym.nlev, nb.net.nPV,
                  (int)b.opt.precision, b.opt.refine_steps, b.opt.lim_inj_reat ? 1 : 0, b.opt.no_max_iter,
                  nb.scen.size());
    return k;
}

bool cache_lookup(const char *path, const std::string &key, int *mode, int *block, int *per_cu) {
    if (!path) return false;
    FILE *f = std::fopen(path, "r");
    if (!f) return false;
    char line[1024];
    bool found = false;
    while (std::fgets(line, sizeof line, f)) {
        char *tab = std::strchr(line, '\t');
        if (!tab) continue;
        *tab = 0;
        int m, bl, pc;
        if (key == line && std::sscanf(tab + 1, "%d %d %d", &m, &bl, &pc) == 3) {
            *mode = m; *block = bl; *per_cu = pc;
            found = true;   // the last entry for a key wins
        }
    }
    std::fclose(f);
    return found;
}

void cache_store(const char *path, const std::string &key, int mode, int block, int per_cu, float ms) {
    if (!path) return;
    FILE *f = std::fopen(path, "a");
    if (!f) return;
    std::fprintf(f, "%s\t%d %d %d %.4f\n", key.c_str(), mode, block, per_cu, ms);
    std::fclose(f);
}

}  // namespace

extern "C" {

pf_status pf_batch_autotune(pf_batch *b, const char *cache_path, int reps, int *n_measured) {
    if (!b || !b->n_scen || reps < 0) return PF_INVALID_ARG;
    BHIP(hipSetDevice(b->device));
    BHIP(hipStreamSynchronize(b->st[0]));
    BHIP(hipStreamSynchronize(b->st[1]));
    hipDeviceProp_t prop;
    BHIP(hipGetDeviceProperties(&prop, b->device));
    const int nrep = std::max(1, reps);
    int measured = 0;
    b->drop_graph();
    for (size_t i = 0; i < b->nets.size(); i++) {
        BatchNet &nb = *b->nets[i];
        if (nb.scen.empty()) continue;
        const std::string key = tune_key(*b, nb, prop.gcnArchName);
        int m = 0, bl = 0, pc = 0;
        if (cache_lookup(cache_path, key, &m, &bl, &pc) && b->configure(nb, m, bl, pc) == PF_OK) continue;
        struct Cand { int mode, block, per_cu; };
        std::vector<Cand> cands;
        if (nb.lds) {
            for (int block : {64, 128, 256, 512, 1024}) {
                int occ = 0;
                if (b->occupancy(nb, 2, block, &occ) != PF_OK || occ < 1) continue;
                cands.push_back({2, block, occ});
                if (occ > 2) cands.push_back({2, block, occ / 2});
            }
        } else {
            for (int mode : {1, 0}) {
                if (mode == 1 && nb.partial == 0) continue;
                for (int block : {256, 512, 1024}) {
                    int occ = 0;
                    if (b->occupancy(nb, mode, block, &occ) != PF_OK || occ < 1) continue;
                    cands.push_back({mode, block, 1});
                    if (occ >= 2) cands.push_back({mode, block, 2});
                    if (occ >= 4) cands.push_back({mode, block, 4});
                }
            }
        }
        float best = 1e30f;
        Cand pick{nb.mode, nb.block, nb.per_cu};
        for (const Cand &c : cands) {
            BCHK(b->configure(nb, c.mode, c.block, c.per_cu));
            float t = 1e30f;
            for (int r = 0; r <= nrep; r++) {   // the first launch is a warm-up
                k_zero_int<<<1, 64, 0, b->st[0]>>>(b->d_counter, (int)b->nets.size());
                BHIP(hipEventRecord(b->t0, b->st[0]));
                BCHK(b->launch_net(i, b->st[0]));
                BHIP(hipEventRecord(b->t1, b->st[0]));
                BHIP(hipEventSynchronize(b->t1));
                float ms = 0;
                BHIP(hipEventElapsedTime(&ms, b->t0, b->t1));
                if (r > 0) t = std::min(t, ms);
            }
            measured++;
            if (t < best) {
                best = t;
                pick = c;
            }
        }
        BCHK(b->configure(nb, pick.mode, pick.block, pick.per_cu));
        cache_store(cache_path, key, pick.mode, pick.block, pick.per_cu, best);
    }
    b->drop_graph();   // launch shapes changed: the next solve captures again
    if (n_measured) *n_measured = measured;
    return PF_OK;
}

pf_status pf_batch_set_shape(pf_batch *b, int net, int mode, int block, int per_cu) {
    if (!b || !b->n_scen || net < 0 || net >= (int)b->nets.size()) return PF_INVALID_ARG;
    BHIP(hipSetDevice(b->device));
    BatchNet &nb = *b->nets[net];
    if (nb.scen.empty()) return PF_INVALID_ARG;
    BHIP(hipStreamSynchronize(b->st[0]));
    BHIP(hipStreamSynchronize(b->st[1]));
    BCHK(b->configure(nb, mode, block, per_cu));
    b->drop_graph();
    return PF_OK;
}

pf_status pf_batch_get_shape(pf_batch *b, int net, int *mode, int *block, int *grid, long long *lds_bytes) {
    if (!b || net < 0 || net >= (int)b->nets.size()) return PF_INVALID_ARG;
    const BatchNet &nb = *b->nets[net];
    if (mode) *mode = nb.mode;
    if (block) *block = nb.block;
    if (grid) *grid = nb.grid;
    if (lds_bytes) *lds_bytes = nb.shm;
    return PF_OK;
}

pf_status pf_batch_get(pf_batch *b, double *V, double *theta, int *iterations, int *converged,
                       double *max_mismatch) {
    if (!b || !b->n_scen) return PF_INVALID_ARG;
    BHIP(hipSetDevice(b->device));
    const size_t total = (size_t)b->total, n = (size_t)b->n_scen;
    CopyPiece out[5];
    int k = 0;
    if (V) out[k++] = {V, b->d_V, sizeof(double) * total};
    if (theta) out[k++] = {theta, b->d_T, sizeof(double) * total};
    if (iterations) out[k++] = {iterations, b->d_it, sizeof(int) * n};
    if (converged) out[k++] = {converged, b->d_cv, sizeof(int) * n};
    if (max_mismatch) out[k++] = {max_mismatch, b->d_mm, sizeof(double) * n};
    BHIP(b->slots.fetch(out, k, b->st[0]));
    return PF_OK;
}

pf_status pf_batch_get_limq(pf_batch *b, unsigned char *limQ, int *flips) {
    if (!b || !b->n_scen) return PF_INVALID_ARG;
    BHIP(hipSetDevice(b->device));
    CopyPiece out[2];
    int k = 0;
    if (limQ) out[k++] = {limQ, b->d_lq, (size_t)b->total_pv};
    if (flips) out[k++] = {flips, b->d_fl, sizeof(int) * (size_t)b->n_scen};
    BHIP(b->slots.fetch(out, k, b->st[0]));
    return PF_OK;
}

}  // extern "C"

// ------------------------------------------------- allocation-free entry

extern "C" pf_status pf_batch_solve_noalloc(pf_batch *b, int n_scen, const int *net_of, const double *Pliq,
                                            const double *Qliq, const double *Qload, const double *V0,
                                            const double *theta0, double *V, double *theta, int *iterations,
                                            int *converged, double *max_mismatch, unsigned char *limQ,
                                            int *flips, void *stream) {
    if (!b || n_scen <= 0 || !net_of || !Pliq || !Qliq || !Qload || !V || !theta || !iterations ||
        !converged || !max_mismatch || !limQ || !flips || ((V0 == nullptr) != (theta0 == nullptr)))
        return PF_INVALID_ARG;
    BHIP(hipSetDevice(b->device));
    char *base = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        base = g_scratch_ptr[b->device];
    }
    if (!base) {
        pf::set_last_error("scratch address not set up on this device");
        return PF_DEVICE_ERROR;
    }
    const int nn = (int)b->nets.size();
    // layout: header, per-scenario offsets, per-network lists, workspaces
    auto up = [](long long x) { return (x + 255) & ~255LL; };
    const long long o_off = kScratchHeader;
    const long long o_pvoff = up(o_off + 8LL * n_scen);
    const long long o_scen = up(o_pvoff + 8LL * n_scen);
    const long long o_ws = up(o_scen + 4LL * n_scen * nn);
    if (o_ws > kScratchBytes) {
        pf::set_last_error("pf_batch_solve_noalloc: too many scenarios for the fixed scratch");
        return PF_INVALID_ARG;
    }
    int n_big = 0;
    for (auto &nb : b->nets) n_big += nb->mode != 2;
    const long long share = n_big ? (kScratchBytes - o_ws) / n_big : 0;
    struct Plan { int grid, block; long long ws_off; };
    Plan plan[64];            // at most 64 networks per batch (pf_batch_create)
    long long o = o_ws;
    for (int i = 0; i < nn; i++) {
        BatchNet &nb = *b->nets[i];
        int block = nb.block, per_cu = nb.per_cu;
        if (nb.grid == 0) {   // the shape for as many scenarios as have a slice
            const long long fit = nb.mode == 2 ? n_scen : std::min<long long>(n_scen, share / nb.ws);
            BCHK(b->default_shape(nb, (int)fit, &block, &per_cu));
        }
        int grid = std::max(1, per_cu * b->cus);
        if (nb.mode != 2) {
            grid = (int)std::min<long long>(grid, share / nb.ws);
            if (grid < 1) {
                pf::set_last_error("pf_batch_solve_noalloc: a working-set slice does not fit the fixed scratch");
                return PF_INVALID_ARG;
            }
        }
        plan[i] = {grid, block, o};
        if (nb.mode != 2) o += up((long long)grid * nb.ws);
    }
    if (o > kScratchBytes) {
        pf::set_last_error("pf_batch_solve_noalloc: working sets exceed the fixed scratch");
        return PF_INVALID_ARG;
    }
    hipStream_t s = stream ? (hipStream_t)stream : b->st[0];
    int *count = (int *)base, *counter = (int *)(base + 256), *invalid = (int *)(base + 512);
    long long *off = (long long *)(base + o_off), *pvoff = (long long *)(base + o_pvoff);
    int *scen = (int *)(base + o_scen);
    NoallocNets info{};
    info.n_nets = nn;
    for (int i = 0; i < nn; i++) {
        info.nB[i] = b->nets[i]->net.nB;
        info.nPV[i] = b->nets[i]->net.nPV;
    }
    k_noalloc_tables<<<1, 1024, 0, s>>>(net_of, n_scen, info, off, pvoff, scen, count, counter, invalid);
    BHIP(hipGetLastError());
    const bool mixed = b->opt.precision != PF_FP64;
    for (int i = 0; i < nn; i++) {
        BatchNet &nb = *b->nets[i];
        BatchJob J{};
        J.nscen = 0;
        J.nscen_dev = count + i;
        J.scen = scen + (long long)i * n_scen;
        J.off = off;
        J.Pliq = Pliq; J.Qliq = Qliq; J.Qload = Qload;
        J.V0 = V0; J.th0 = theta0;
        J.Vout = V; J.thout = theta;
        J.iters = iterations; J.conv = converged; J.maxmis = max_mismatch;
        J.pv_off = pvoff; J.limQout = limQ; J.flips = flips;
        J.counter = counter + i;
        J.gws = nb.mode != 2 ? base + plan[i].ws_off : nullptr;
        J.ws_bytes = nb.ws;
        J.max_iter = b->opt.no_max_iter;
        J.lim = b->opt.lim_inj_reat ? 1 : 0;
        J.refine = mixed ? b->opt.refine_steps : 0;
        J.tol = b->opt.tolerancia;
        J.diverge = 1e6;
        BatchTopo tp = nb.tp;
        void *args[] = {&tp, &J};
        BHIP(hipLaunchKernel((const void *)batch_kernel(mixed, nb.mode, plan[i].block, nb.lds), dim3(plan[i].grid),
                             dim3(plan[i].block), args, (size_t)b->shm_bytes(nb, nb.mode, plan[i].block), s));
    }
    if (!stream) {
        BHIP(hipStreamSynchronize(s));
        int bad = 0;
        BHIP(hipMemcpy(&bad, invalid, sizeof(int), hipMemcpyDeviceToHost));
        if (bad) {
            pf::set_last_error("pf_batch_solve_noalloc: net_of holds an index outside the batch's networks");
            return PF_INVALID_ARG;
        }
    }
    return PF_OK;
}
