// tm_cg.hip -- preconditioned conjugate gradients for tetmag's demag systems.
//
// Replaces GPUSolver (GPUSolver.h:53-87, GPUSolver.cu:43-98), which runs
// AMGCL smoothed-aggregation + ILU0 + GMRES on the row-replaced stiffness
// matrices.  Those matrices are symmetric except for identity rows
// (Neumann: DemagField.cpp:204-220; Dirichlet: FEMprocessing.cpp:329-369).
// With x preset to b on the identity rows, every residual and search
// direction vanishes on those rows and the iteration only sees the free
// block, which is symmetric positive definite -- so CG applies to exactly the
// reference's systems and returns the reference's solution (same gauge for
// the Neumann problem).
//
// Each iteration is two kernels, the second of which also forms the first
// product of the next V-cycle, with no host round trip and no device-scope
// fence:
//   k_cg_spmv(k) : gamma_k, (r,r) from the partials; beta; p' = z + beta p;
//                  q = A p', with p' formed in the gathers; partial (p',q)
//   k_cg_step(k) : alpha = gamma_k / (p,q); x += alpha p; r' = r - alpha q;
//                  partial (r',r'); and on further blocks F r' = F r - alpha F q
//                  for the preconditioner's first product F
// (k_cg_update is the step without that product.)  Every block reduces the
// producer's partials itself (tm_internal.hpp), so all blocks take the same
// convergence decision; block 0 publishes the scalars.  Grids are at most
// kMaxCgBlocks blocks, which keeps the partial arrays short.  A solve of a
// single right-hand side is bound by the number of its launches (each a few
// microseconds, most of it latency), so every kernel starts with the loads of
// its rows and reduces the scalars it needs while they are in flight.  The
// host reads the state once per chunk of iterations.  With the V-cycle as one
// product per level (tm_amg.hip) an iteration of a two-level solve is three
// launches (of a four-level one eight), where separate smoothing, restriction,
// prolongation and update kernels took eight (fifteen): a cold Neumann solve
// of 71,825 nodes 1,150 -> 789 us, one FP64 evaluation at 29,760 nodes 710 ->
// 352 us, at 282,897 nodes 3.47 -> 2.89 ms (2.06 ms of it the boundary product).
#include <algorithm>
#include <cmath>

#include "tm_internal.hpp"

namespace tmh {

namespace {

// Slices handled by this block's wavefronts: s = wave_global, += total waves.
#define CG_SLICE_LOOP(A)                                                                             \
    const int lane = threadIdx.x & (kWave - 1);                                                       \
    const int nsl = ((A).n + kWave - 1) / kWave;                                                      \
    const int spb_ = ((nsl + (int)gridDim.x - 1) / (int)gridDim.x + kBlock / kWave - 1) / (kBlock / kWave) * \
                     (kBlock / kWave);                                                                \
    const int s0_ = xcd_block() * spb_, s1_ = min(nsl, s0_ + spb_);                                   \
    for (int s = s0_ + (int)threadIdx.x / kWave; s < s1_; s += kBlock / kWave)

__device__ inline void block_partials(double* part, int stride, double v0, double v1, int nv) {
    __shared__ double sp[2][kBlock / kWave];
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    v0 = wave_sum(v0);
    if (nv > 1) v1 = wave_sum(v1);
    if (lane == 0) {
        sp[0][wid] = v0;
        sp[1][wid] = v1;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0.0, b = 0.0;
        for (int k = 0; k < kBlock / kWave; ++k) {
            a += sp[0][k];
            b += sp[1][k];
        }
        part[blockIdx.x] = a;
        if (nv > 1) part[stride + blockIdx.x] = b;
    }
}

// ---- initial guesses from earlier solves ---------------------------------
// x0 = x_0 + sum_j c_j dX_j over the kept pairs (backward differences at the
// newest, least squares in the residual norm; the method is described with
// kSolveWindow in tm_internal.hpp).  Slots are ordered newest first.

// per-block partials wpart[q * G + block] of the kWinDots dots and, as the
// last row, of (b, b).  The new b goes into the head slot as it is read: when
// the window is full that slot holds the oldest pair, whose value this thread
// has already loaded.  Eight threads sum the block's values of a dot from LDS
// (a shuffle tree per dot, 29 of them, took longer than the loads).
constexpr int kWinRows = kWinDots + 1;
constexpr int kWinBlocks = 256;  // at most, so that k_cg_win_combine has few partials to read
static_assert(8 * kWinRows <= kBlock, "eight threads per sum");

__global__ __launch_bounds__(kBlock) void k_cg_win_dots(int n, const CgWindow* w, double* __restrict__ Bw,
                                                        const double* __restrict__ b, double* wpart) {
    const int cnt = w->cnt, head = w->head;
    double acc[kWinDots] = {};
    double bb = 0.0;
    const double* src[kSolveWindow];
#pragma unroll
    for (int i = 0; i < kSolveWindow; ++i) src[i] = Bw + (size_t)win_slot(head, i) * n;
    double* dst = Bw + (size_t)head * n;
    for (int e = blockIdx.x * kBlock + threadIdx.x; e < n; e += gridDim.x * kBlock) {
        double v[kSolveWindow];
#pragma unroll
        for (int i = 0; i < kSolveWindow; ++i) v[i] = i < cnt ? src[i][e] : 0.0;
        const double bi = b[e];
        const double r = bi - v[0];
        win_differences(v, cnt);
        win_accumulate(acc, v, r);
        bb += bi * bi;
        dst[e] = bi;
    }
    __shared__ double sp[kWinRows][kBlock + 8];
#pragma unroll
    for (int q = 0; q < kWinDots; ++q) sp[q][threadIdx.x] = acc[q];
    sp[kWinDots][threadIdx.x] = bb;
    __syncthreads();
    const int q = threadIdx.x >> 3, sub = threadIdx.x & 7;
    if (q >= kWinRows) return;
    double t = 0.0;
#pragma unroll 8
    for (int k = sub; k < kBlock; k += 8) t += sp[q][k];
    t = group_sum<8>(t);
    if (sub == 0) wpart[(size_t)q * gridDim.x + blockIdx.x] = t;
}

// x0 = sum_i a_i x_slot(i) (the caller's x when the window is empty), x = b on
// the fixed rows, x = 0 when b = 0.  Every block sums the partials of the dots
// and solves the small least-squares system itself, with its elements' loads in
// flight meanwhile: latency alone, 7.9 -> 5.8 us at 2,205 nodes, 23 -> 16.6 at 282,897.
__global__ __launch_bounds__(kBlock) void k_cg_win_combine(int n, int G, const CgWindow* w, const double* wpart,
                                                           const double* __restrict__ Xw,
                                                           const unsigned char* __restrict__ fixed,
                                                           const double* __restrict__ b, double* __restrict__ x) {
    __shared__ double sd[kWinRows];
    __shared__ double sa[kSolveWindow];
    const int cnt = w->cnt, head = w->head;
    const double* src[kSolveWindow];
#pragma unroll
    for (int i = 0; i < kSolveWindow; ++i) src[i] = Xw + (size_t)win_slot(head, i) * n;
    // this thread's element, on its way while the system is summed and solved
    // (slots past cnt hold no pair yet: read, and left out below)
    int e = blockIdx.x * kBlock + threadIdx.x;
    double v[kSolveWindow], be = 0.0;
    unsigned char fe = 0;
    auto load = [&]() {
#pragma unroll
        for (int i = 0; i < kSolveWindow; ++i) v[i] = src[i][e];
        be = b[e];
        fe = fixed[e];
    };
    if (e < n) load();
    const int q = threadIdx.x >> 3, sub = threadIdx.x & 7;
    double t = 0.0;
    if (q < kWinRows) {
#pragma unroll 8
        for (int g = sub; g < G; g += 8) t += wpart[(size_t)q * G + g];
    }
    t = group_sum<8>(t);
    if (q < kWinRows && sub == 0) sd[q] = t;
    __syncthreads();
    if (threadIdx.x == 0 && cnt > 0) {
        double d[kWinDots], a[kSolveWindow];
#pragma unroll
        for (int k = 0; k < kWinDots; ++k) d[k] = sd[k];
        win_coefficients(cnt, d, a);
#pragma unroll
        for (int i = 0; i < kSolveWindow; ++i) sa[i] = a[i];
    }
    __syncthreads();
    const bool zero = sd[kWinDots] == 0.0;
    double a[kSolveWindow];
#pragma unroll
    for (int i = 0; i < kSolveWindow; ++i) a[i] = i < cnt ? sa[i] : 0.0;
    while (e < n) {
        if (zero) x[e] = 0.0;
        else if (fe) x[e] = be;
        else if (cnt > 0) {
            double acc = 0.0;
#pragma unroll
            for (int i = 0; i < kSolveWindow; ++i)
                if (i < cnt) acc += a[i] * v[i];
            x[e] = acc;
        }
        e += gridDim.x * kBlock;
        if (e < n) load();
    }
}

// ---- iterations ---------------------------------------------------------------
// part layout: [0, G) bb | [G, 2G) rz | [2G, 3G) rr | [3G, 4G) pq
__global__ __launch_bounds__(kBlock) void k_cg_init_fixed(int n, const unsigned char* __restrict__ fixed,
                                                          const double* __restrict__ b, double* __restrict__ x,
                                                          double* part) {
    double v = 0.0;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const double bi = b[i];
        if (fixed[i]) x[i] = bi;
        v += bi * bi;
    }
    block_partials(part, 0, v, 0.0, 1);
}

// the state of a new solve, from the Gb partials of (b, b); b = 0 has the
// solution 0 (which k_cg_finish writes)
__device__ inline void cg_begin(const double* bbpart, int Gb, double tol, CgState* st) {
    double bb[1];
    reduce_partials_all<1>(bbpart, Gb, Gb, bb);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->bb = bb[0];
        st->tol2bb = tol * tol * bb[0];
        st->iters = 0;
        st->done = bb[0] == 0.0 ? 1 : 0;
        st->rr = 0.0;
    }
}

// r = b - A x, one lane per row (SELL)
template <bool JAC>
__global__ __launch_bounds__(kBlock) void k_cg_init_res(SellView A, const double* __restrict__ val,
                                                        const double* __restrict__ dinv,
                                                        const double* __restrict__ b, const double* __restrict__ x,
                                                        double* __restrict__ r, double* __restrict__ z,
                                                        const double* bbpart, int Gb, double* part, double tol,
                                                        CgState* st) {
    const int G = gridDim.x;
    cg_begin(bbpart, Gb, tol, st);
    double vrz = 0.0, vrr = 0.0;
    CG_SLICE_LOOP(A) {
        double acc = 0.0;
        sell_row(A, s, lane, [&](int64_t e, int c) { acc += val[e] * x[c]; });
        const int row = s * kWave + lane;
        if (row < A.n) {
            const double ri = b[row] - acc;
            r[row] = ri;
            vrr += ri * ri;
            if (JAC) {
                const double zi = dinv[row] * ri;
                z[row] = zi;
                vrz += ri * zi;
            }
        }
    }
    if (JAC) block_partials(part + G, G, vrz, vrr, 2);
    else block_partials(part + 2 * G, G, vrr, 0.0, 1);
}

// r = b - A x, LPR lanes per row
template <int LPR>
__global__ __launch_bounds__(kBlock) void k_cg_init_res_l(int n, const int* __restrict__ rp,
                                                          const int* __restrict__ ci, const double* __restrict__ v,
                                                          const double* __restrict__ b, const double* __restrict__ x,
                                                          double* __restrict__ r, const double* bbpart, int Gb,
                                                          double* part, double tol, CgState* st) {
    const int G = gridDim.x;
    const RowShare R = row_share<LPR>(n, xcd_block(), G);
    const int sub = threadIdx.x & (LPR - 1);
    int row = R.r0 + threadIdx.x / LPR;
    double s[1] = {0.0};
    if (row < R.r1) csr_row<LPR, 1>(rp, ci, v, {x}, row, sub, s);
    cg_begin(bbpart, Gb, tol, st);
    double vrr = 0.0;
    while (row < R.r1) {
        if (sub == 0) {
            const double ri = b[row] - s[0];
            r[row] = ri;
            vrr += ri * ri;
        }
        row += kBlock / LPR;
        if (row < R.r1) csr_row<LPR, 1>(rp, ci, v, {x}, row, sub, s);
    }
    block_partials(part + 2 * G, G, vrr, 0.0, 1);
}

// gamma_k, convergence on the last (r, r), beta_k; false when the solve stops
__device__ inline bool cg_beta(int k, const double* part, int G, CgState* st, double& beta) {
    double t[2];
    reduce_partials_all<2>(part + G, G, G, t);  // (r,z), (r,r)
    const double gam = t[0], rr = t[1];
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    if (!isfinite(gam) || !isfinite(rr)) {
        if (lead) st->done = 2;
        return false;
    }
    if (rr <= st->tol2bb) {
        if (lead) {
            st->done = 1;
            st->rr = rr;
            st->iters = k;
        }
        return false;
    }
    beta = k > 0 ? gam / st->gam[(k - 1) & 1] : 0.0;
    if (lead) {
        st->gam[k & 1] = gam;
        st->rr = rr;
    }
    return true;
}

// p_new = z + beta p_old, q = A p_new, partial (p_new, q); one lane per row (SELL).
// (q = A z + beta q would gather z alone, but its rounding errors add up over the
// iterations: the residual that a Jacobi solve to 1e-13 leaves grew by up to 18 %.)
__global__ __launch_bounds__(kBlock) void k_cg_spmv(SellView A, const double* __restrict__ val,
                                                    const double* __restrict__ z, const double* __restrict__ p_old,
                                                    double* __restrict__ p_new, double* __restrict__ q, int k,
                                                    double* part, CgState* st) {
    if (st->done) return;
    const int G = gridDim.x;
    double beta;
    if (!cg_beta(k, part, G, st, beta)) return;
    double v = 0.0;
    CG_SLICE_LOOP(A) {
        double acc = 0.0;
        if (k == 0) sell_row(A, s, lane, [&](int64_t e, int c) { acc += val[e] * z[c]; });
        else sell_row(A, s, lane, [&](int64_t e, int c) { acc += val[e] * (z[c] + beta * p_old[c]); });
        const int row = s * kWave + lane;
        if (row < A.n) {
            const double pi = k == 0 ? z[row] : z[row] + beta * p_old[row];
            p_new[row] = pi;
            q[row] = acc;
            v += pi * acc;
        }
    }
    block_partials(part + 3 * G, G, v, 0.0, 1);
}

// the same with LPR lanes per row; A z and A p_old are summed apart, so that the
// gathers do not wait for beta
template <int LPR>
__global__ __launch_bounds__(kBlock) void k_cg_spmv_l(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                      const double* __restrict__ v, const double* __restrict__ z,
                                                      const double* __restrict__ p_old, double* __restrict__ p_new,
                                                      double* __restrict__ q, int k, double* part, CgState* st) {
    if (st->done) return;
    const int G = gridDim.x;
    const RowShare R = row_share<LPR>(n, xcd_block(), G);
    const int sub = threadIdx.x & (LPR - 1);
    int row = R.r0 + threadIdx.x / LPR;
    double s[2] = {0.0, 0.0};
    auto sums = [&]() {
        if (k > 0) {
            csr_row<LPR, 2>(rp, ci, v, {z, p_old}, row, sub, s);
        } else {
            double s0[1];
            csr_row<LPR, 1>(rp, ci, v, {z}, row, sub, s0);
            s[0] = s0[0];
        }
    };
    if (row < R.r1) sums();
    double beta;
    if (!cg_beta(k, part, G, st, beta)) return;
    double dot = 0.0;
    while (row < R.r1) {
        if (sub == 0) {
            const double pi = k == 0 ? z[row] : z[row] + beta * p_old[row];
            const double qi = k == 0 ? s[0] : s[0] + beta * s[1];
            p_new[row] = pi;
            q[row] = qi;
            dot += pi * qi;
        }
        row += kBlock / LPR;
        if (row < R.r1) sums();
    }
    block_partials(part + 3 * G, G, dot, 0.0, 1);
}

// alpha_k from the G partials of (p, q); false on breakdown
__device__ inline bool cg_alpha(int k, const double* part, int G, CgState* st, double& alpha) {
    double t[1];
    reduce_partials_all<1>(part + 3 * G, G, G, t);
    const double pq = t[0];
    if (!(pq > 0.0) || !isfinite(pq)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) st->done = 2;
        return false;
    }
    alpha = st->gam[k & 1] / pq;
    return true;
}

template <bool JAC>
__global__ __launch_bounds__(kBlock) void k_cg_update(int n, const double* __restrict__ dinv,
                                                      const double* __restrict__ p, const double* __restrict__ q,
                                                      double* __restrict__ x, double* __restrict__ r,
                                                      double* __restrict__ z, int k, double* part, CgState* st) {
    if (st->done) return;
    const int G = gridDim.x;
    double alpha;
    if (!cg_alpha(k, part, G, st, alpha)) return;
    double vrz = 0.0, vrr = 0.0;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += G * kBlock) {
        x[i] += alpha * p[i];
        const double ri = r[i] - alpha * q[i];
        r[i] = ri;
        vrr += ri * ri;
        if (JAC) {
            const double zi = dinv[i] * ri;
            z[i] = zi;
            vrz += ri * zi;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) st->iters = k + 1;
    if (JAC) block_partials(part + G, G, vrz, vrr, 2);
    else block_partials(part + 2 * G, G, vrr, 0.0, 1);
}

// Blocks [0, G): x += alpha p, rn = r - alpha q, partial (rn, rn).  Further
// blocks: out = F rn = F r - alpha F q for the preconditioner's first product
// F, LPR lanes per row of a CSR matrix (LPR = 0: one block per row of a dense
// rows x n matrix).  r is only read (rn is another vector), so the two parts
// need no order.
template <int LPR>
__global__ __launch_bounds__(kBlock) void k_cg_step(int n, int G, const double* __restrict__ p,
                                                    const double* __restrict__ q, double* __restrict__ x,
                                                    const double* __restrict__ r, double* __restrict__ rn, int rows,
                                                    const int* __restrict__ rp, const int* __restrict__ ci,
                                                    const double* __restrict__ v, double* __restrict__ out, int k,
                                                    double* part, CgState* st) {
    if (st->done) return;
    double alpha;
    if ((int)blockIdx.x < G) {
        if (!cg_alpha(k, part, G, st, alpha)) return;
        double vrr = 0.0;
        for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += G * kBlock) {
            x[i] += alpha * p[i];
            const double ri = r[i] - alpha * q[i];
            rn[i] = ri;
            vrr += ri * ri;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) st->iters = k + 1;
        block_partials(part + 2 * G, G, vrr, 0.0, 1);
    } else if constexpr (LPR > 0) {
        const int row = ((blockIdx.x - G) * kBlock + threadIdx.x) / LPR, sub = threadIdx.x & (LPR - 1);
        double s[2] = {0.0, 0.0};
        if (row < rows) csr_row<LPR, 2>(rp, ci, v, {r, q}, row, sub, s);
        if (!cg_alpha(k, part, G, st, alpha)) return;
        if (row < rows && sub == 0) out[row] = s[0] - alpha * s[1];
    } else {
        __shared__ double sp[2][kBlock / kWave];
        const int row = blockIdx.x - G;
        const double* d = v + (size_t)row * n;
        double sr = 0.0, sq = 0.0;
        for (int j = threadIdx.x; j < n; j += kBlock) {
            const double c = d[j];
            sr += c * r[j];
            sq += c * q[j];
        }
        if (!cg_alpha(k, part, G, st, alpha)) return;
        sr = wave_sum(sr);
        sq = wave_sum(sq);
        if ((threadIdx.x & (kWave - 1)) == 0) {
            sp[0][threadIdx.x / kWave] = sr;
            sp[1][threadIdx.x / kWave] = sq;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double a = 0.0, c = 0.0;
            for (int w = 0; w < kBlock / kWave; ++w) {
                a += sp[0][w];
                c += sp[1][w];
            }
            out[row] = a - alpha * c;
        }
    }
}

// After a chunk of iterations: a residual that met the tolerance on the last
// update counts as converged (the preconditioner that would test it has not
// run).  When the solve has ended (converged, broken down, or `last`: no more
// iterations follow): b = 0 gives x = 0; with a window (w) the solution goes
// into its head slot, beside its b, and the head advances, or the window is
// emptied after a failure; fails / imax (fixed budgets): solves that missed
// the tolerance and the largest iteration count.  host: a copy of the state
// in pinned memory.  The block that arrives last at the ticket changes the
// window state, which every block has read by then.
__global__ __launch_bounds__(kBlock) void k_cg_finish(int n, int G, int last, CgWindow* w, double* __restrict__ Xw,
                                                      double* __restrict__ x, const double* part, CgState* st,
                                                      unsigned* ticket, unsigned* fails, int* imax, CgState* host) {
    double t[1];
    reduce_partials_all<1>(part + 2 * G, G, G, t);
    const int done = st->done;
    const bool conv = done == 1 || (done == 0 && t[0] <= st->tol2bb);
    const bool zero = st->bb == 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        CgState c = *st;
        if (done == 0) {
            c.rr = t[0];
            c.done = conv ? 1 : 0;
            *st = c;
        }
        if (host) *host = c;
        if (fails && last) {
            if (!conv) fails[0] += 1u;
            if (c.iters > imax[0]) imax[0] = c.iters;
        }
    }
    if (!conv && done == 0 && !last) return;
    const int head = w ? w->head : 0;
    if (zero || (w && conv))
        for (int e = blockIdx.x * kBlock + threadIdx.x; e < n; e += gridDim.x * kBlock) {
            const double xe = zero ? 0.0 : x[e];
            if (zero) x[e] = xe;
            if (w && conv) Xw[(size_t)head * n + e] = xe;
        }
    if (!w) return;
    __syncthreads();  // every thread of the block has read the window state
    if (threadIdx.x != 0 || atomicAdd(ticket, 1u) != gridDim.x - 1u) return;
    *ticket = 0u;
    if (conv) {
        w->cnt = min(w->cnt + 1, kSolveWindow);
        w->head = (head + 1) % kSolveWindow;
    } else {
        w->cnt = 0;
        w->head = 0;
    }
}

}  // namespace

// Transposed solve helpers: zero the fixed entries of the right-hand side,
// then y_j = w_j - sum_i A_ij y_i over the free rows i coupled to fixed j.
__global__ __launch_bounds__(kBlock) void k_adj_zero_fixed(int n, const unsigned char* __restrict__ fixed,
                                                           const double* __restrict__ w, double* __restrict__ out) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = fixed[i] ? 0.0 : w[i];
}

__global__ __launch_bounds__(kBlock) void k_adj_fix_rows(int nf, const int* __restrict__ idx,
                                                         const int* __restrict__ rp, const int* __restrict__ ci,
                                                         const double* __restrict__ v, const double* __restrict__ w,
                                                         double* __restrict__ y) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= nf) return;
    const int j = idx[r];
    double acc = w[j];
    for (int q = rp[r]; q < rp[r + 1]; ++q) acc -= v[q] * y[ci[q]];
    y[j] = acc;
}

CgSolver::~CgSolver() {
    if (h_st) (void)hipHostFree(h_st);
    h_st = nullptr;
}

int CgSolver::setup(int n_, const int* rowptr, const int* colidx, const double* vals, int precond_,
                    hipStream_t s) {
    if (precond_ != TM_PRECOND_JACOBI && precond_ != TM_PRECOND_AMG) return TM_ERR_BAD_ARG;
    precond = precond_;
    n = n_;
    // identity rows: a single stored nonzero on the diagonal equal to 1
    std::vector<unsigned char> fx((size_t)n, 0);
    std::vector<double> di((size_t)n, 0.0);
    nfixed = 0;
    double amax = 0.0;
    for (int i = 0; i < n; ++i) {
        for (int q = rowptr[i]; q < rowptr[i + 1]; ++q) amax = std::max(amax, std::fabs(vals[q]));
        int nz = 0;
        bool diag1 = false;
        for (int q = rowptr[i]; q < rowptr[i + 1]; ++q) {
            if (vals[q] != 0.0) {
                ++nz;
                if (colidx[q] == i && vals[q] == 1.0) diag1 = true;
            }
        }
        if (nz == 1 && diag1) {
            fx[i] = 1;
            ++nfixed;
        }
    }
    // diagonal, symmetry of the free block
    const double stol = 1e-12 * amax;
    for (int i = 0; i < n; ++i) {
        double d = 0.0;
        for (int q = rowptr[i]; q < rowptr[i + 1]; ++q) {
            const int j = colidx[q];
            if (j == i) d = vals[q];
            if (fx[i] || fx[j] || j == i) continue;
            const int* lo = colidx + rowptr[j];
            const int* hi = colidx + rowptr[j + 1];
            const int* it = std::lower_bound(lo, hi, i);
            const double aji = (it != hi && *it == i) ? vals[it - colidx] : 0.0;
            if (std::fabs(aji - vals[q]) > stol) return TM_ERR_UNSUPPORTED;
        }
        if (fx[i]) di[i] = 1.0;
        else if (d > 0.0) di[i] = 1.0 / d;
        else return TM_ERR_UNSUPPORTED;  // free block must be positive definite
    }
    // fixed-row coupling for the transposed solve
    {
        std::vector<int> fidx, frp(1, 0), fci, pos((size_t)n, -1);
        for (int i = 0; i < n; ++i)
            if (fx[i]) {
                pos[i] = (int)fidx.size();
                fidx.push_back(i);
            }
        std::vector<std::vector<std::pair<int, double>>> rows(fidx.size());
        for (int i = 0; i < n; ++i) {
            if (fx[i]) continue;
            for (int q = rowptr[i]; q < rowptr[i + 1]; ++q) {
                const int j = colidx[q];
                if (fx[j] && vals[q] != 0.0) rows[pos[j]].push_back({i, vals[q]});
            }
        }
        std::vector<double> fv;
        for (auto& r : rows) {
            for (auto& e : r) {
                fci.push_back(e.first);
                fv.push_back(e.second);
            }
            frp.push_back((int)fci.size());
        }
        if (!fidx.empty()) {
            TM_CHECK(fix_idx.upload(fidx.data(), fidx.size(), s));
            TM_CHECK(fix_rp.upload(frp.data(), frp.size(), s));
            if (!fci.empty()) {
                TM_CHECK(fix_ci.upload(fci.data(), fci.size(), s));
                TM_CHECK(fix_v.upload(fv.data(), fv.size(), s));
            }
            TM_HIP(hipStreamSynchronize(s));  // host vectors go out of scope
        }
    }
    pat.build(n, n, rowptr, colidx);
    h_val.assign(vals, vals + rowptr[n]);
    h_dinv = di;
    h_fixed = fx;
    std::vector<double> sv;
    TM_CHECK(pat.scatter(rowptr, colidx, vals, sv));
    TM_CHECK(pat.upload(s));
    TM_CHECK(val.upload(sv.data(), sv.size(), s));
    TM_CHECK(dinv.upload(di.data(), di.size(), s));
    TM_CHECK(fixed.upload(fx.data(), fx.size(), s));
    TM_CHECK(z.alloc(n));
    TM_CHECK(q.alloc(n));
    for (auto& v : p) TM_CHECK(v.alloc(n));
    lanes = precond == TM_PRECOND_AMG && n <= kLaneRows;
    if (lanes) {
        // lanes per row: what fills the chip (1,024 blocks) once, at most 16
        A.n = n;
        A.lpr = 4;
        while (A.lpr < 16 && (int64_t)2 * A.lpr * n <= (int64_t)1024 * kBlock) A.lpr *= 2;
        TM_CHECK(A.rp.upload(rowptr, (size_t)n + 1, s));
        TM_CHECK(A.ci.upload(colidx, (size_t)rowptr[n], s));
        TM_CHECK(A.v.upload(vals, (size_t)rowptr[n], s));
    }
    grid = lanes ? grid_for((int64_t)n * A.lpr) : (pat.nslices + kBlock / kWave - 1) / (kBlock / kWave);
    grid = xcd_grid(std::min(kMaxCgBlocks, grid));
    TM_CHECK(part.alloc((size_t)4 * grid));
    TM_CHECK(winX.alloc((size_t)kSolveWindow * n));
    TM_CHECK(winB.alloc((size_t)kSolveWindow * n));
    TM_CHECK(wpart.alloc((size_t)kWinRows * kWinBlocks));
    TM_CHECK(win.alloc(1));
    TM_HIP(hipMemsetAsync(win.p, 0, sizeof(CgWindow), s));
    TM_CHECK(ticket.alloc(1));
    TM_HIP(hipMemsetAsync(ticket.p, 0, sizeof(unsigned), s));
    TM_CHECK(st.alloc(1));
    TM_HIP(hipMemsetAsync(st.p, 0, sizeof(CgState), s));
    if (!h_st) TM_HIP(hipHostMalloc((void**)&h_st, sizeof(CgState), hipHostMallocDefault));
    TM_HIP(hipStreamSynchronize(s));
    if (precond == TM_PRECOND_AMG) TM_CHECK(amg.setup(n, rowptr, colidx, vals, fx, &pat, val.p, dinv.p, lanes ? A.lpr : 0, s));
    for (auto& v : rb) {
        v.release();
        TM_CHECK(v.alloc((size_t)n + (precond == TM_PRECOND_AMG ? amg.tail() : 0)));
        if (!lanes) break;  // one residual vector, updated in place
    }
    last_iters[0] = last_iters[1] = -1;
    return TM_OK;
}

// Initial guess (project: from the window, b going into its head slot) and
// residual; the convergence state.
int CgSolver::start(Seq& sq, const double* b, double* x, double tol, hipStream_t s, bool project) {
    const double* bbpart = part.p;
    int Gb = grid;
    if (project) {
        Gb = std::min(kWinBlocks, grid_for(n));
        hipLaunchKernelGGL(k_cg_win_dots, dim3(Gb), dim3(kBlock), 0, s, n, (const CgWindow*)win.p, winB.p, b, wpart.p);
        hipLaunchKernelGGL(k_cg_win_combine, dim3(std::min(grid, grid_for(n))), dim3(kBlock), 0, s, n, Gb,
                           (const CgWindow*)win.p, (const double*)wpart.p, (const double*)winX.p,
                           (const unsigned char*)fixed.p, b, x);
        bbpart = wpart.p + (size_t)kWinDots * Gb;
    } else {
        hipLaunchKernelGGL(k_cg_init_fixed, dim3(grid), dim3(kBlock), 0, s, n, fixed.p, b, x, part.p);
    }
    sq = Seq{rb[0].p, rb[1].p, p[0].p, p[1].p, false, true};
    if (lanes)
        with_lanes(A.lpr, [&](auto lpr) {
            hipLaunchKernelGGL(k_cg_init_res_l<decltype(lpr)::value>, dim3(grid), dim3(kBlock), 0, s, n, A.rp.p,
                               A.ci.p, A.v.p, b, (const double*)x, sq.rcur, bbpart, Gb, part.p, tol, st.p);
        });
    else if (precond == TM_PRECOND_JACOBI)
        hipLaunchKernelGGL(k_cg_init_res<true>, dim3(grid), dim3(kBlock), 0, s, view(pat), val.p, dinv.p, b,
                           (const double*)x, sq.rcur, z.p, bbpart, Gb, part.p, tol, st.p);
    else
        hipLaunchKernelGGL(k_cg_init_res<false>, dim3(grid), dim3(kBlock), 0, s, view(pat), val.p, dinv.p, b,
                           (const double*)x, sq.rcur, z.p, bbpart, Gb, part.p, tol, st.p);
    TM_HIP(hipGetLastError());
    return TM_OK;
}

int CgSolver::precondition(Seq& sq, hipStream_t s) {
    if (precond == TM_PRECOND_JACOBI) return TM_OK;  // z = D^-1 r comes with the update
    TM_CHECK(amg.apply(sq.rcur, z.p, part.p + grid, grid, s, st.p, sq.rr_new ? part.p + 2 * (size_t)grid : nullptr,
                       sq.first_done));
    sq.rr_new = false;
    return TM_OK;
}

// another: the preconditioner runs on the new residual, and its first product
// is formed along with the update
int CgSolver::iteration(Seq& sq, double* x, int k, bool another, hipStream_t s) {
    const int G = grid;
    const bool jac = precond == TM_PRECOND_JACOBI;
    std::swap(sq.pcur, sq.pold);
    if (lanes)
        with_lanes(A.lpr, [&](auto lpr) {
            hipLaunchKernelGGL(k_cg_spmv_l<decltype(lpr)::value>, dim3(G), dim3(kBlock), 0, s, n, A.rp.p, A.ci.p,
                               A.v.p, (const double*)z.p, (const double*)sq.pold, sq.pcur, q.p, k, part.p, st.p);
        });
    else
        hipLaunchKernelGGL(k_cg_spmv, dim3(G), dim3(kBlock), 0, s, view(pat), val.p, (const double*)z.p,
                           (const double*)sq.pold, sq.pcur, q.p, k, part.p, st.p);
    sq.first_done = lanes && another && !amg.levels.empty();
    if (sq.first_done) {
        const AmgPrecond::First F = amg.first();
        double* out = F.out ? F.out : sq.rnext + n;
        if (F.dense)
            hipLaunchKernelGGL(k_cg_step<0>, dim3(G + F.rows), dim3(kBlock), 0, s, n, G, (const double*)sq.pcur,
                               (const double*)q.p, x, (const double*)sq.rcur, sq.rnext, F.rows, (const int*)nullptr,
                               (const int*)nullptr, F.dense, out, k, part.p, st.p);
        else
            with_lanes(F.csr->lpr, [&](auto lpr) {
                constexpr int kL = decltype(lpr)::value;
                hipLaunchKernelGGL(k_cg_step<kL>, dim3(G + (F.rows + kBlock / kL - 1) / (kBlock / kL)), dim3(kBlock),
                                   0, s, n, G, (const double*)sq.pcur, (const double*)q.p, x, (const double*)sq.rcur,
                                   sq.rnext, F.rows, F.csr->rp.p, F.csr->ci.p, F.csr->v.p, out, k, part.p, st.p);
            });
        std::swap(sq.rcur, sq.rnext);
    } else if (jac) {
        hipLaunchKernelGGL(k_cg_update<true>, dim3(G), dim3(kBlock), 0, s, n, dinv.p, sq.pcur, q.p, x, sq.rcur, z.p, k,
                           part.p, st.p);
    } else {
        hipLaunchKernelGGL(k_cg_update<false>, dim3(G), dim3(kBlock), 0, s, n, dinv.p, sq.pcur, q.p, x, sq.rcur, z.p, k,
                           part.p, st.p);
    }
    sq.rr_new = true;
    TM_HIP(hipGetLastError());
    return TM_OK;
}

int CgSolver::finish(const double* x, hipStream_t s, bool project, bool last, unsigned* fails, int* imax,
                     CgState* out) {
    // few blocks: each takes a ticket, one after the other
    hipLaunchKernelGGL(k_cg_finish, dim3(std::min(64, grid_for(n, 4 * kBlock))), dim3(kBlock), 0, s, n, grid, last ? 1 : 0, project ? win.p : nullptr, winX.p,
                       const_cast<double*>(x), (const double*)part.p, st.p, ticket.p, fails, imax, out);
    TM_HIP(hipGetLastError());
    return TM_OK;
}

int CgSolver::solve(const double* b, double* x, double tol, int maxit, hipStream_t s, int* iters, double* relres,
                    bool project) {
    if (n == 0) return TM_ERR_NOT_READY;
    if (!(tol > 0.0) || maxit < 1) return TM_ERR_BAD_ARG;
    Seq sq;
    TM_CHECK(start(sq, b, x, tol, s, project));
    // The first chunk is what the last such solve needed (solves along a
    // trajectory need similar counts); no preconditioner runs after a chunk's last
    // iteration before the host has seen that another one is needed.
    int& known = last_iters[project ? 0 : 1];
    int enq = 0;
    int chunk = known < 0 ? 8 : known;
    for (int more = 2;; more = std::min(2 * more, 8)) {
        const int end = std::min(maxit, enq + chunk);
        for (; enq < end; ++enq) {
            TM_CHECK(precondition(sq, s));
            TM_CHECK(iteration(sq, x, enq, enq + 1 < end, s));
        }
        TM_CHECK(finish(x, s, project, enq >= maxit, nullptr, nullptr, h_st));
        TM_HIP(hipStreamSynchronize(s));
        if (h_st->done || enq >= maxit) break;
        chunk = more;
    }
    const CgState hs = *h_st;
    known = hs.iters;
    if (iters) *iters = hs.iters;
    if (relres) *relres = hs.bb > 0 ? std::sqrt(hs.rr / hs.bb) : 0.0;
    if (hs.done == 2) return TM_ERR_NONFINITE;
    if (hs.done == 1 || hs.bb == 0.0) return TM_OK;
    return TM_ERR_MAXITER;
}

int CgSolver::enqueue(const double* b, double* x, double tol, int budget, hipStream_t s, unsigned* fails,
                      int* imax, bool project) {
    if (n == 0) return TM_ERR_NOT_READY;
    if (!(tol > 0.0) || budget < 1 || !fails || !imax) return TM_ERR_BAD_ARG;
    Seq sq;
    TM_CHECK(start(sq, b, x, tol, s, project));
    for (int k = 0; k < budget; ++k) {
        TM_CHECK(precondition(sq, s));
        TM_CHECK(iteration(sq, x, k, k + 1 < budget, s));
    }
    return finish(x, s, project, true, fails, imax, nullptr);
}

int CgSolver::solve_transposed(const double* w, double* y, double tol, int maxit, hipStream_t s, int* iters,
                               double* relres) {
    if (n == 0) return TM_ERR_NOT_READY;
    TM_CHECK(tb.alloc(n));
    hipLaunchKernelGGL(k_adj_zero_fixed, dim3(grid_for(n)), dim3(kBlock), 0, s, n, fixed.p, w, tb.p);
    TM_HIP(hipGetLastError());
    const int st = solve(tb.p, y, tol, maxit, s, iters, relres);
    if (st != TM_OK && st != TM_ERR_MAXITER) return st;
    if (nfixed > 0) {
        hipLaunchKernelGGL(k_adj_fix_rows, dim3(grid_for(nfixed)), dim3(kBlock), 0, s, nfixed, fix_idx.p, fix_rp.p,
                           fix_ci.p, fix_v.p, w, y);
        TM_HIP(hipGetLastError());
    }
    return st;
}

}  // namespace tmh

using namespace tmh;

extern "C" {

int tm_solver_create(int n, const int* rowptr, const int* colidx, const double* vals, int precond, tm_solver** out) {
    if (!out || n <= 0 || !rowptr || !colidx || !vals) return TM_ERR_BAD_ARG;
    int nd = 0;
    TM_CHECK(tm_device_count(&nd));
    tm_solver* S = new tm_solver();
    if (hipStreamCreateWithFlags(&S->stream, hipStreamNonBlocking) != hipSuccess) {
        delete S;
        return TM_ERR_HIP;
    }
    int st = S->cg.setup(n, rowptr, colidx, vals, precond, S->stream);
    if (st == TM_OK) st = S->b.alloc(n);
    if (st == TM_OK) st = S->x.alloc(n);
    if (st == TM_OK) st = S->xt.alloc(n);
    if (st == TM_OK && hipMemsetAsync(S->x.p, 0, sizeof(double) * n, S->stream) != hipSuccess) st = TM_ERR_HIP;
    if (st == TM_OK && hipMemsetAsync(S->xt.p, 0, sizeof(double) * n, S->stream) != hipSuccess) st = TM_ERR_HIP;
    if (st == TM_OK && hipStreamSynchronize(S->stream) != hipSuccess) st = TM_ERR_HIP;
    if (st != TM_OK) {
        tm_solver_destroy(S);
        return st;
    }
    *out = S;
    return TM_OK;
}

int tm_solver_destroy(tm_solver* S) {
    if (!S) return TM_OK;
    if (S->stream) (void)hipStreamSynchronize(S->stream);
    if (S->stream) (void)hipStreamDestroy(S->stream);
    delete S;
    return TM_OK;
}

int tm_solver_solve(tm_solver* S, const double* b, int bwhere, double* x, int xwhere, double tol, int maxit,
                    int warm, int* iters, double* relres) {
    if (!S || !b || !x) return TM_ERR_BAD_ARG;
    if ((bwhere != TM_HOST && bwhere != TM_DEVICE) || (xwhere != TM_HOST && xwhere != TM_DEVICE))
        return TM_ERR_BAD_ARG;
    const int n = S->cg.n;
    const double* bd = b;
    if (bwhere == TM_HOST) {
        TM_CHECK(copy_in(S->b.p, b, TM_HOST, n, S->stream));
        bd = S->b.p;
    }
    double* xd = S->x.p;  // the solver keeps its solution between calls (GPUSolver::x_d)
    if (warm == 1) TM_CHECK(copy_in(xd, x, xwhere, n, S->stream));
    else if (warm == 0) TM_HIP(hipMemsetAsync(xd, 0, sizeof(double) * n, S->stream));
    // warm == 2 (the solver's own previous solution): start from the best
    // combination of its last solutions instead
    int st = S->cg.solve(bd, xd, tol, maxit, S->stream, iters, relres, warm == 2);
    int st2 = copy_out(x, xwhere, xd, n, S->stream);
    if (xwhere == TM_DEVICE) TM_HIP(hipStreamSynchronize(S->stream));
    return st != TM_OK ? st : st2;
}

int tm_solver_solve_transposed(tm_solver* S, const double* b, int bwhere, double* x, int xwhere, double tol,
                               int maxit, int warm, int* iters, double* relres) {
    if (!S || !b || !x) return TM_ERR_BAD_ARG;
    if ((bwhere != TM_HOST && bwhere != TM_DEVICE) || (xwhere != TM_HOST && xwhere != TM_DEVICE))
        return TM_ERR_BAD_ARG;
    const int n = S->cg.n;
    const double* bd = b;
    if (bwhere == TM_HOST) {
        TM_CHECK(copy_in(S->b.p, b, TM_HOST, n, S->stream));
        bd = S->b.p;
    }
    double* xd = S->xt.p;
    if (warm == 1) TM_CHECK(copy_in(xd, x, xwhere, n, S->stream));
    else if (warm == 0) TM_HIP(hipMemsetAsync(xd, 0, sizeof(double) * n, S->stream));
    int st = S->cg.solve_transposed(bd, xd, tol, maxit, S->stream, iters, relres);
    int st2 = copy_out(x, xwhere, xd, n, S->stream);
    if (xwhere == TM_DEVICE) TM_HIP(hipStreamSynchronize(S->stream));
    return st != TM_OK ? st : st2;
}

}  // extern "C"

namespace tmh {
int amg_info(const CgSolver& cg, int* nlevels, int* sizes, int cap) {
    if (!nlevels || (cap > 0 && !sizes)) return TM_ERR_BAD_ARG;
    if (cg.precond != TM_PRECOND_AMG) {
        *nlevels = 0;
        return TM_OK;
    }
    const int L = (int)cg.amg.levels.size();
    *nlevels = L + 1;
    for (int l = 0; l < L + 1 && l < cap; ++l) sizes[l] = l < L ? cg.amg.levels[l].n : cg.amg.nc;
    return TM_OK;
}
}  // namespace tmh

extern "C" int tm_solver_amg_info(tm_solver* s, int* nlevels, int* sizes, int cap) {
    if (!s) return TM_ERR_BAD_ARG;
    return tmh::amg_info(s->cg, nlevels, sizes, cap);
}
