// Dense LU with partial pivoting of the single-network solver (metodo denso
// and hibridoB; the reference: cusolverDnDgetrf / getrs,
// GPU/newtonRaphson.cuh:507-530), FP64, column-major, up to kDenseMax
// unknowns.
//
// Right-looking in panels of NB columns, two launches a panel:
//   k_dense_panel   one workgroup factors the panel with its rows in
//                   registers, RPT of them per thread;
//   k_dense_update  a workgroup per 8 columns right of it (the right-hand
//                   side is one more column) swaps their rows, solves with
//                   the panel's unit lower triangle and subtracts L21 U12;
// then k_dense_back solves the upper triangle.  The flops (2/3 n^3) are
// small: what bounds it is the panels' chain of n pivot steps, each a search
// over the workgroup, a barrier, a division and the pivot row read by every
// wave from LDS.  234 unknowns (118 buses): 8 panels of 27 us on average, their
// updates 12.5 us each, the back substitution 19 us, 336 us in all (kernel
// trace).  Before, one workgroup did everything, a thread walking its row
// through memory for each pivot: 4,635 us.

#include "dense.hpp"
#include "kernels_impl.hpp"

namespace pf {

namespace {

// value of lane l (the same for the whole wave, constant after unrolling)
__device__ __forceinline__ double lane_value(double v, int l) {
    const unsigned long long b = double_as_u64(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return u64_as_double(((unsigned long long)hi << 32) | lo);
}

template <int CTRL>
__device__ __forceinline__ double dpp_max(double v) {
    const unsigned long long b = double_as_u64(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xF, 0xF, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, false);
    return fmax(v, u64_as_double(((unsigned long long)hi << 32) | lo));
}

// max over the wave (no lane holds a NaN): in each row of 16 lanes through
// DPP moves, then the four rows
__device__ __forceinline__ double wave_fmax(double v) {
    v = dpp_max<0xB1>(v);
    v = dpp_max<0x4E>(v);
    v = dpp_max<0x141>(v);
    v = dpp_max<0x140>(v);
    return fmax(fmax(lane_value(v, 0), lane_value(v, 16)), fmax(lane_value(v, 32), lane_value(v, 48)));
}

}  // namespace

// Columns [k0, k0 + NB) of rows [k0, n), thread t holding rows t, t + T, ...
// of the panel.  Rows do not move between threads: a swap exchanges their
// positions, and each row is written back at its last one.  Per column every
// wave leaves its largest candidate and that candidate's row in LDS, so one
// barrier serves both the search and the elimination (two buffers).  The
// pivot is the largest magnitude, ties to the lowest position; a column
// without a positive finite one raises singular and ends the factorisation.
// chg: [count, then pairs (position, where its row came from)], at most 2 NB.
template <int NB, int RPT>
__global__ void __launch_bounds__(1024) k_dense_panel(double *A, int n, int k0, int *chg, Ctl *ctl, int gate) {
    if (gate && !ctl->step) return;
    if (ctl->singular) return;
    constexpr int MW = 16;
    __shared__ double s_v[2][MW];
    __shared__ int s_p[2][MW], s_n;
    __shared__ double s_row[2][MW][NB];
    const int tid = (int)threadIdx.x, T = (int)blockDim.x, w = tid / 64, nw = T / 64;
    const int rows = n - k0, nbc = min(NB, rows);
    double a[RPT][NB];
    int pos[RPT];
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        const int i = tid + r * T;
        pos[r] = i < rows ? i : -1;
#pragma unroll
        for (int c = 0; c < NB; c++) a[r][c] = (i < rows && c < nbc) ? A[(size_t)(k0 + c) * n + k0 + i] : 0.0;
    }
    if (tid == 0) s_n = 0;
    bool ok = true;
#pragma unroll
    for (int j = 0; j < NB; j++)
        if (ok && j < nbc) {
            double v = -1.0;
            int p = INT_MAX;
#pragma unroll
            for (int r = 0; r < RPT; r++) {
                const double x = fabs(a[r][j]);
                if (pos[r] >= j && (x > v || (x == v && pos[r] < p))) {   // never a NaN
                    v = x;
                    p = pos[r];
                }
            }
            const double m = wave_fmax(v);
            const unsigned long long eq = __ballot(v == m);
            int pm = __builtin_amdgcn_readlane(p, __ffsll((long long)eq) - 1);
            if (eq & (eq - 1)) {   // a tie: the lowest position
                pm = v == m ? p : INT_MAX;
                for (int off = 32; off > 0; off >>= 1) pm = min(pm, __shfl_xor(pm, off));
            }
#pragma unroll
            for (int r = 0; r < RPT; r++)
                if (pos[r] == pm) {
#pragma unroll
                    for (int c = j; c < NB; c++) s_row[j & 1][w][c] = a[r][c];
                }
            if ((tid & 63) == 0) {
                s_v[j & 1][w] = m;
                s_p[j & 1][w] = pm;
            }
            __syncthreads();
            double best = s_v[j & 1][0];
            int bp = s_p[j & 1][0], bw = 0;
            for (int i = 1; i < nw; i++) {
                const double x = s_v[j & 1][i];
                const int y = s_p[j & 1][i];
                if (x > best || (x == best && y < bp)) {
                    best = x;
                    bp = y;
                    bw = i;
                }
            }
            ok = best > 0.0 && isfinite(best);   // the same for every thread
            const double *pr = s_row[j & 1][bw];
            const double piv = pr[j];
#pragma unroll
            for (int r = 0; r < RPT; r++) {
                if (pos[r] == bp) pos[r] = j;
                else if (pos[r] == j) pos[r] = bp;
                if (pos[r] > j) {
                    const double l = a[r][j] / piv;
                    a[r][j] = l;
#pragma unroll
                    for (int c = j + 1; c < NB; c++) a[r][c] -= l * pr[c];
                }
            }
        }
    if (!ok) {
        if (tid == 0) atomicOr(&ctl->singular, 1);
        return;
    }
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        const int i = tid + r * T;
        if (i >= rows) continue;
#pragma unroll
        for (int c = 0; c < NB; c++)
            if (c < nbc) (A + (size_t)(k0 + c) * n + k0)[(unsigned)pos[r]] = a[r][c];
        if (pos[r] != i) {
            const int e = atomicAdd(&s_n, 1);
            chg[1 + 2 * e] = k0 + pos[r];
            chg[2 + 2 * e] = k0 + i;
        }
    }
    __syncthreads();
    if (tid == 0) chg[0] = s_n;
}

// The columns right of the panel at k0 (column n: the right-hand side b), TC
// per workgroup: their rows swapped as the panel's were, U12 = L11^-1 A12
// (a wave per column, lane i holding row i of L11), A22 -= L21 U12 (a thread
// per row, U12 broadcast from LDS).
template <int NB>
__global__ void __launch_bounds__(256) k_dense_update(double *A, double *b, int n, int k0, const int *chg, Ctl *ctl,
                                                      int gate) {
    if (gate && !ctl->step) return;
    if (ctl->singular) return;
    constexpr int TC = kDenseCols;
    __shared__ double s_u[NB][TC], s_c[2 * NB][TC];
    const int tid = (int)threadIdx.x, lane = tid & 63, w = tid / 64;
    const int nbc = min(NB, n - k0), k1 = k0 + nbc, c0 = k1 + (int)blockIdx.x * TC;
    auto col = [&](int c) { return c0 + c < n ? A + (size_t)(c0 + c) * n : b; };
    const int li = lane & (NB - 1);
    double l11[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const double x = (A + (size_t)(k0 + min(j, nbc - 1)) * n + k0)[(unsigned)min(li, nbc - 1)];
        l11[j] = j < li && li < nbc ? x : 0.0;
    }
    const int nchg = chg[0];
#pragma unroll 1
    for (int q = tid; q < nchg * TC; q += 256) {
        const int e = q / TC, c = q % TC;
        if (c0 + c <= n) s_c[e][c] = col(c)[chg[2 + 2 * e]];
    }
    for (int q = tid; q < NB * TC; q += 256) {
        const int i = q / TC, c = q % TC;
        s_u[i][c] = (i < nbc && c0 + c <= n) ? col(c)[k0 + i] : 0.0;
    }
    __syncthreads();
#pragma unroll 1
    for (int q = tid; q < nchg * TC; q += 256) {
        const int e = q / TC, c = q % TC, p = chg[1 + 2 * e];
        if (c0 + c > n) continue;
        if (p < k1) s_u[p - k0][c] = s_c[e][c];
        else col(c)[p] = s_c[e][c];
    }
    __syncthreads();
#pragma unroll 1
    for (int c = w; c < TC; c += 4) {
        double u = s_u[li][c];
#pragma unroll
        for (int j = 0; j < NB - 1; j++) u -= l11[j] * lane_value(u, j);
        if (lane < NB) {
            s_u[li][c] = u;
            if (li < nbc && c0 + c <= n) col(c)[k0 + li] = u;
        }
    }
    __syncthreads();
#pragma unroll 1
    for (int i = k1 + tid; i < n; i += 256) {
        double l[NB], acc[TC];
#pragma unroll
        for (int j = 0; j < NB; j++) l[j] = (A + (size_t)(k0 + j) * n)[(unsigned)i];
#pragma unroll
        for (int c = 0; c < TC; c++) acc[c] = c0 + c <= n ? col(c)[i] : 0.0;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            if (j % 4 == 0) asm volatile("" ::: "memory");   // four rows of U12 in registers at a time, not all
#pragma unroll
            for (int c = 0; c < TC; c++) acc[c] -= l[j] * s_u[j][c];
        }
#pragma unroll
        for (int c = 0; c < TC; c++) asm volatile("" : "+v"(acc[c]));   // the sums are not sunk into the stores' branches
#pragma unroll
        for (int c = 0; c < TC; c++)
            if (c0 + c <= n) col(c)[i] = acc[c];
    }
}

// U x = b from the last panel of 32 up.  Wave p % 8 solves panel p: lane i
// holds its row i and its diagonal, loaded since the wave's last panel.  The
// threads above then subtract the panel's unknowns, their rows' entries on it
// in registers by that time, so a panel waits for its 32 dependent quotients
// and multiply-adds and two barriers, not for loads.  A quotient is the
// product with the diagonal's reciprocal, corrected by its remainder
// (Markstein 1990: the rounded quotient, where nothing over- or underflows):
// rows scaled by the reciprocal beforehand save two multiply-adds a step (234
// unknowns 16.7 us instead of 18.7) and left 1 to 4 % more error.
__global__ void __launch_bounds__(512) k_dense_back(const double *A, double *b, int n, Ctl *ctl, int gate) {
    if (gate && !ctl->step) return;
    if (ctl->singular) return;
    constexpr int NB = 32, NW = 8;
    __shared__ double s_y[kDenseMax], s_x[NB];
    const int tid = (int)threadIdx.x, lane = tid & 63, w = tid / 64, li = lane & (NB - 1);
    double d[NB], dg = 1.0, rd = 0.0;   // this wave's coming panel: row li, its diagonal and 1 / that
    auto diag = [&](int p) __attribute__((always_inline)) {
        if (p < 0) return;
        const int p0 = p * NB, nbc = min(NB, n - p0);
        const bool in = li < nbc;
        dg = in ? (A + (size_t)p0 * n + p0)[(unsigned)li * (unsigned)(n + 1)] : 1.0;
        rd = 1.0 / dg;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const double x = (A + (size_t)(p0 + min(j, nbc - 1)) * n + p0)[(unsigned)min(li, nbc - 1)];
            d[j] = in && j > li && j < nbc ? x : 0.0;
        }
    };
    const int np = (n + NB - 1) / NB;
    diag(np - 1 - ((np - 1 - w) % NW + NW) % NW);   // the highest panel p with p % NW == w
    for (int i = tid; i < n; i += 512) s_y[i] = b[i];
    __syncthreads();
    for (int p = np - 1; p >= 0; p--) {
        const int p0 = p * NB, nbc = min(NB, n - p0);
        double u[NB];
        if (tid < p0) {
#pragma unroll
            for (int j = 0; j < NB; j++) u[j] = (A + (size_t)(p0 + min(j, nbc - 1)) * n)[(unsigned)tid];
        }
        if (w == p % NW) {
            const bool in = li < nbc;
            double y = in ? s_y[p0 + li] : 0.0, x = 0.0;
            auto quotient = [&]() __attribute__((always_inline)) {
                const double q = y * rd;
                return fma(fma(-q, dg, y), rd, q);
            };
#pragma unroll
            for (int j = NB - 1; j >= 0; j--) {
                const double q = quotient();
                if (li == j) x = q;
                y -= d[j] * lane_value(q, j);
            }
            if (lane < NB) {   // zeros past the panel's columns
                s_x[li] = x;
                if (in) s_y[p0 + li] = x;
            }
            diag(p - NW);
        }
        __syncthreads();
#pragma unroll 1
        for (int i = tid; i < p0; i += 512) {
            double y = s_y[i];
            if (i != tid) {
#pragma unroll
                for (int j = 0; j < NB; j++) u[j] = (A + (size_t)(p0 + min(j, nbc - 1)) * n)[(unsigned)i];
            }
#pragma unroll
            for (int j = NB - 1; j >= 0; j--) y -= u[j] * s_x[j];
            s_y[i] = y;
        }
        __syncthreads();
    }
    for (int i = tid; i < n; i += 512) b[i] = s_y[i];
}

void launch_dense_solve(double *A, double *b, int n, int *chg, Ctl *ctl, int gate, hipStream_t st) {
    for (int k0 = 0; k0 < n;) {
        // as wide a panel as its rows' registers allow (32 doubles a thread)
        const int rows = n - k0, rpt = rows <= 1024 ? 1 : 4, nb = 32 / rpt;
        const int threads = ((rows + rpt - 1) / rpt + 63) / 64 * 64;
        if (rpt == 1) k_dense_panel<32, 1><<<1, threads, 0, st>>>(A, n, k0, chg, ctl, gate);
        else k_dense_panel<8, 4><<<1, threads, 0, st>>>(A, n, k0, chg, ctl, gate);
        const int k1 = k0 + (rows < nb ? rows : nb), tiles = (n + 1 - k1 + kDenseCols - 1) / kDenseCols;
        if (rpt == 1) k_dense_update<32><<<tiles, 256, 0, st>>>(A, b, n, k0, chg, ctl, gate);
        else k_dense_update<8><<<tiles, 256, 0, st>>>(A, b, n, k0, chg, ctl, gate);
        k0 = k1;
    }
    k_dense_back<<<1, 512, 0, st>>>(A, b, n, ctl, gate);
}

}  // namespace pf
