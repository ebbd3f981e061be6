// tm_batch.hip -- many magnetisation samples on one mesh in one pass.
//
// The reference evaluates one magnetisation at a time (TheLLG, DemagField)
// and its hysteresis driver runs field values one after another
// (Hysteresis.cpp:43-169).  Here up to 64 samples share every operator read:
// vectors are stored node-major, sample-fastest ([node][sample]); each sparse
// product runs one wavefront per row with the samples across its lanes, so
// the row's offsets and weights (row-slot layout, below) are wavefront-uniform
// scalar loads read once for all samples and every gather is one contiguous
// access (64 FP32 samples: 16 lanes x 16 bytes per gathered row, four rows per
// load instruction).  The boundary-element product becomes a GEMM (B times the
// b x S boundary potentials) on the FP64 matrix cores.
//
// Both demag solves use the same scheme per sample:
//   outer (FP64):  x_fixed = b_fixed;  r = b - A x  (FP64 operator and vectors)
//   inner (T):     A d = r by AMG-preconditioned CG in precision T, from d = 0
//   x += d, repeat until ||b - A x|| <= tol ||b|| for every sample.
// T = double solves to the final tolerance in one outer step (the FP64
// batched form); T = float runs the inner iterations in FP32 to a relative
// 1e-5 and recovers FP64 accuracy by iterative refinement (the mixed form).
// Converged samples are frozen (their step lengths are zero); once all are,
// the iterations still queued return at once.
#define ROCBLAS_BETA_FEATURES_API  // rocblas_gemm_ex_get_solutions (the GEMM autotuner)
#include <rocblas/rocblas.h>

#include <algorithm>
#include <cstddef>
#include <cmath>
#include <exception>
#include <future>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "tm_internal.hpp"

namespace tmh {

namespace {

constexpr int kMaxS = 64;  // any_active() reads 64 flags
constexpr int kRowsPerBlock = kBlock / kWave;  // one row per wavefront


// Per-sample CG state of one inner solve.
struct BState {
    double gam[kMaxS];    // (r, z)
    double alpha[kMaxS];
    double beta[kMaxS];
    double itol2[kMaxS];  // inner tolerance^2 (absolute, on ||r||^2)
    double rr[kMaxS];
    int active[kMaxS];
    int iters[kMaxS];
};

// Per-sample outer state.
struct OState {
    double bb[kMaxS];
    double rr[kMaxS];
    int done[kMaxS];  // 0 going on, 1 at the tolerance, 2 given up: the residual is not finite
};

// Wavefront w of block b walks rows b*4 + w, then + 4*G, ...  (A contiguous
// range per XCD was measured slower for these kernels.)
#define B_ROW_LOOP(NROWS)                                                                              \
    const int lane = threadIdx.x & (kWave - 1);                                                        \
    const bool on = lane < S;                                                                          \
    [[maybe_unused]] const int lc = min(lane, S - 1); /* gather lane: in bounds for every lane */  \
    for (int row = __builtin_amdgcn_readfirstlane(blockIdx.x * kRowsPerBlock + (int)(threadIdx.x / kWave)); \
         row < (NROWS); row += gridDim.x * kRowsPerBlock)

// As B_ROW_LOOP, over XCD-contiguous eighths of the rows (blocks with equal
// blockIdx % 8 share one XCD); needs lane, on, lc declared by the caller.
#define B_ROW_LOOP_XCD(NROWS)                                                                          \
    const int xr0_ = gridDim.x % kXcd ? 0 : (int)((int64_t)(NROWS) * (blockIdx.x % kXcd) / kXcd);      \
    const int xr1_ = gridDim.x % kXcd ? (NROWS) : (int)((int64_t)(NROWS) * (blockIdx.x % kXcd + 1) / kXcd); \
    const int xlb_ = gridDim.x % kXcd ? blockIdx.x : blockIdx.x / kXcd;                                \
    const int xst_ = (gridDim.x % kXcd ? gridDim.x : gridDim.x / kXcd) * kRowsPerBlock;                \
    for (int row = __builtin_amdgcn_readfirstlane(xr0_ + xlb_ * kRowsPerBlock + (int)(threadIdx.x / kWave)); \
         row < xr1_; row += xst_)

// ---- slot layout for the solver kernels ----------------------------------
// Every operator the batched solves apply is stored in row slots of kSlot
// entries: row i owns slots sp[i] .. sp[i+1]-1 (a multiple of kSlot, padded
// with offset 0 and weight 0), each slot holding the byte offset of the
// gathered row (column * S * sizeof(element)) and the weight.  A wavefront
// reads a chunk's offsets and weights with scalar loads (16 consecutive
// dwords each: wavefront-uniform data goes to SGPRs, no lane broadcasts),
// gathers with buffer loads whose row offset is the SGPR operand (no address
// arithmetic per entry) and accumulates with the weight as the SGPR operand
// of the FMA.  Per entry that is one load and one vector instruction; the
// earlier form (indices and values in lanes, read with readlane, 64-bit
// address adds) was bound by vector-instruction issue.
constexpr int kSlot = 16;

struct SlotArgs {
    int n;            // rows
    int xbytes;       // bytes of the gathered vector (ncols * S * element)
    const int* sp;    // n + 1 slot starts
    const int* off;   // per slot: byte offset of the gathered row
    const void* w;    // per slot: weight (float or double)
    const int* gate = nullptr;  // per-sample active flags: the kernel does nothing when none is set
    int gate_n = 0;
};

typedef const int __attribute__((address_space(4)))* cint_p;

// true when any of the flags is set (or there are no flags).  The batched
// CG enqueues iterations in chunks ahead of its convergence check; once every
// sample has converged, the iterations still queued return at once.  All
// kMaxS flags are read (four 16-dword scalar loads; flags past the batch size
// stay 0 from the solver's set-up).
__device__ inline bool any_active(const int* act, int) {
    if (!act) return true;
    const cint_p a = (cint_p)act;
    int any = 0;
#pragma unroll
    for (int s = 0; s < 64; ++s) any |= a[s];
    return any != 0;
}
template <typename W>
using cw_p = const W __attribute__((address_space(4)))*;

template <typename T>
__device__ inline T buf_ld(__amdgpu_buffer_rsrc_t r, int voff, int soff);
template <>
__device__ inline float buf_ld<float>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
template <>
__device__ inline double buf_ld<double>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

// raw buffer over the gathered vector (word 3: 32-bit data format, gfx9)
__device__ inline __amdgpu_buffer_rsrc_t gather_rsrc(const void* x, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(x), (short)0, bytes, 0x00020000);
}

// acc += sum over the kSlot slots at q of w * x[row]
template <typename T, typename W>
__device__ inline T slot_chunk(cint_p off, cw_p<W> w, int q, __amdgpu_buffer_rsrc_t xr, int voff, T acc) {
    int o[kSlot];
    T xv[kSlot];
#pragma unroll
    for (int k = 0; k < kSlot; ++k) o[k] = off[q + k];
#pragma unroll
    for (int k = 0; k < kSlot; ++k) xv[k] = buf_ld<T>(xr, voff, o[k]);
#pragma unroll
    for (int k = 0; k < kSlot; ++k) acc += (T)w[q + k] * xv[k];
    return acc;
}

// rows a wavefront walks at a time: two in FP32 (2 x 32 SGPRs of offsets and
// weights), one in FP64 (the weights take twice the SGPRs)
template <typename T>
constexpr int kRowsPerStep = sizeof(T) == 4 ? 2 : 1;

// Row walk: wavefront w of block b takes rows r0 + (b/8)*4 + w, then
// + 4*G/8, ... within its XCD's eighth [r0, r1); with RPI = 2 it takes two
// rows per step and issues both rows' first-chunk gathers before consuming
// any (twice the loads in flight).
// ld(row) loads what the row's epilogue needs (issued with the gathers);
// epi(row, acc, ld(row)) finishes the row.  Lanes >= S gather lane S-1's
// element (lc) and their results are discarded by epi.
template <typename T, typename W, int RPI, typename LDF, typename EPIF>
__device__ inline void slot_walk(const SlotArgs& M, const void* x, int lc, LDF&& ld, EPIF&& epi) {
    const int n = M.n;
    const __amdgpu_buffer_rsrc_t xr = gather_rsrc(x, M.xbytes);
    const cint_p sp = (cint_p)M.sp;
    const cint_p of = (cint_p)M.off;
    const cw_p<W> w = (cw_p<W>)M.w;
    const int vo = lc * (int)sizeof(T);
    // each XCD (blocks b with equal b % 8) walks its own contiguous eighth of
    // the rows, so neighbouring rows share that XCD's L2
    int r0 = 0, r1 = n, lb = blockIdx.x, gx = gridDim.x;
    if (gridDim.x % kXcd == 0) {
        const int x = blockIdx.x % kXcd;
        gx = gridDim.x / kXcd;
        lb = blockIdx.x / kXcd;
        r0 = (int)((int64_t)n * x / kXcd);
        r1 = (int)((int64_t)n * (x + 1) / kXcd);
    }
    const int stride = gx * kRowsPerBlock;
    for (int row = __builtin_amdgcn_readfirstlane(r0 + lb * kRowsPerBlock + (int)(threadIdx.x / kWave)); row < r1;
         row += RPI * stride) {
        if constexpr (RPI == 2) {
            const int rb = row + stride;
            const bool hb = rb < r1;
            const int a0 = sp[row], a1 = sp[row + 1];
            const int b0 = hb ? sp[rb] : a0, b1 = hb ? sp[rb + 1] : a0 + kSlot;
            const auto la = ld(row);
            const auto lb = ld(hb ? rb : row);
            int oa[kSlot], ob[kSlot];
            T xa[kSlot], xb[kSlot];
#pragma unroll
            for (int k = 0; k < kSlot; ++k) {
                oa[k] = of[a0 + k];
                ob[k] = of[b0 + k];
            }
#pragma unroll
            for (int k = 0; k < kSlot; ++k) {
                xa[k] = buf_ld<T>(xr, vo, oa[k]);
                xb[k] = buf_ld<T>(xr, vo, ob[k]);
            }
            T sa = 0, sb = 0;
#pragma unroll
            for (int k = 0; k < kSlot; ++k) {
                sa += (T)w[a0 + k] * xa[k];
                sb += (T)w[b0 + k] * xb[k];
            }
            for (int q = a0 + kSlot; q < a1; q += kSlot) sa = slot_chunk<T, W>(of, w, q, xr, vo, sa);
            for (int q = b0 + kSlot; q < b1; q += kSlot) sb = slot_chunk<T, W>(of, w, q, xr, vo, sb);
            epi(row, sa, la);
            if (hb) epi(rb, sb, lb);
        } else {
            const int a0 = sp[row], a1 = sp[row + 1];
            const auto la = ld(row);
            T sa = 0;
            for (int q = a0; q < a1; q += kSlot) sa = slot_chunk<T, W>(of, w, q, xr, vo, sa);
            epi(row, sa, la);
        }
    }
}


// ---- wide gathers for 64 FP32 samples -------------------------------------
// With S = 64 in FP32 a node's row of samples is 256 B.  Lanes gather 16 B
// each (4 samples), so 16 lanes cover a row and one load instruction gathers
// four different rows: lane group g = lane / 16 takes slots 4g .. 4g+3 of
// each 16-slot chunk (their offsets and weights arrive as one 16-byte load
// each), lane j = lane % 16 holds samples 4j .. 4j+3.  The groups' partial
// sums are added across lanes at the end of the row.  Against one dword
// gather per slot this issues a quarter of the vector-memory instructions
// (the per-instruction address work of the texture path bounds the 64-lane
// dword form).
typedef float f4 __attribute__((ext_vector_type(4)));
typedef int i4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef int i2 __attribute__((ext_vector_type(2)));

__device__ inline f4 buf_ld4(__amdgpu_buffer_rsrc_t r, int voff) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
}

// the gather of a slot; where its weight is zero (padding slots) the offset
// is moved past the buffer's end, so the load returns zeros without a
// memory access (raw-buffer range check; gathered vectors are < 1 GiB, see
// SlotOp::build)
constexpr int kOutOfRange = 0x7ffffff0;
__device__ inline f4 ld4_if(__amdgpu_buffer_rsrc_t r, int voff, float w) {
    return buf_ld4(r, w != 0.f ? voff : kOutOfRange);
}

__device__ inline f4 shfl_xor4(f4 v, int m) {
    return f4{__shfl_xor(v.x, m), __shfl_xor(v.y, m), __shfl_xor(v.z, m), __shfl_xor(v.w, m)};
}

// Row walk as slot_walk (XCD-contiguous eighths).  BLK = false: one row per
// lane group, four consecutive rows per wavefront step; lane j of a group
// holds samples 4j .. 4j+3 of its row and walks all of the row's slots
// itself (per chunk of CH slots: the offsets and weights as CH/4 16-byte
// loads, then all CH gathers before any is used), so a wavefront has four
// rows' gathers in flight and no cross-group sum.  BLK = true (operators of
// long rows: the coarse levels' Galerkin products, the restrictions): one
// row per block, its 16-slot chunks dealt round-robin to the block's 4
// wavefronts (lane group g: slots q+4g .. q+4g+3 of chunk q), the groups'
// and wavefronts' sums added across lanes and in LDS.  ld(row, j) loads the
// epilogue's operands for samples 4j .. 4j+3; epi(row, j, acc, ld) runs on
// every lane of a group whose row exists (BLK = false), on lanes 0-15 of
// wavefront 0 (BLK = true).
template <bool BLK, typename LDF, typename EPIF>
__device__ inline void wide_walk(const SlotArgs& M, const void* x, LDF&& ld, EPIF&& epi) {
    constexpr int CH = kSlot;
    const int n = M.n;
    const int lane = threadIdx.x & (kWave - 1), g = lane >> 4, j = lane & 15;
    const int wv = threadIdx.x / kWave;
    const __amdgpu_buffer_rsrc_t xr = gather_rsrc(x, M.xbytes);
    const i4* __restrict__ of = (const i4*)M.off;
    const f4* __restrict__ w = (const f4*)M.w;
    const int vo = j * 16;
    int r0 = 0, r1 = n, lb = blockIdx.x, gx = gridDim.x;
    if (gridDim.x % kXcd == 0) {
        const int xi = blockIdx.x % kXcd;
        gx = gridDim.x / kXcd;
        lb = blockIdx.x / kXcd;
        r0 = (int)((int64_t)n * xi / kXcd);
        r1 = (int)((int64_t)n * (xi + 1) / kXcd);
    }
    if constexpr (!BLK) {
        const int* __restrict__ sp = M.sp;
        const int stride = gx * kRowsPerBlock * 4;
        for (int base = __builtin_amdgcn_readfirstlane(r0 + (lb * kRowsPerBlock + wv) * 4); base < r1;
             base += stride) {
            const int row = base + g;
            const bool has = row < r1;
            const int rr = has ? row : base;
            const int a0 = sp[rr], a1 = has ? sp[rr + 1] : a0;
            const auto lv = ld(rr, j);
            f4 acc = {0.f, 0.f, 0.f, 0.f};
            for (int q = a0; q < a1; q += CH) {
                i4 o[CH / 4];
                f4 ww[CH / 4];
#pragma unroll
                for (int k = 0; k < CH / 4; ++k) {
                    o[k] = of[(q >> 2) + k];
                    ww[k] = w[(q >> 2) + k];
                }
                f4 xv[CH];
#pragma unroll
                for (int k = 0; k < CH / 4; ++k) {
                    xv[4 * k] = ld4_if(xr, vo + o[k].x, ww[k].x);
                    xv[4 * k + 1] = ld4_if(xr, vo + o[k].y, ww[k].y);
                    xv[4 * k + 2] = ld4_if(xr, vo + o[k].z, ww[k].z);
                    xv[4 * k + 3] = ld4_if(xr, vo + o[k].w, ww[k].w);
                }
#pragma unroll
                for (int k = 0; k < CH / 4; ++k) {
                    acc += ww[k].x * xv[4 * k];
                    acc += ww[k].y * xv[4 * k + 1];
                    acc += ww[k].z * xv[4 * k + 2];
                    acc += ww[k].w * xv[4 * k + 3];
                }
            }
            if (has) epi(row, j, acc, lv);
        }
    } else {
        auto chunk = [&](int q, f4 acc) {  // lane group g: slots q+4g .. q+4g+3
            const i4 o = of[(q >> 2) + g];
            const f4 ww = w[(q >> 2) + g];
            const f4 x0 = ld4_if(xr, vo + o.x, ww.x), x1 = ld4_if(xr, vo + o.y, ww.y);
            const f4 x2 = ld4_if(xr, vo + o.z, ww.z), x3 = ld4_if(xr, vo + o.w, ww.w);
            acc += ww.x * x0;
            acc += ww.y * x1;
            acc += ww.z * x2;
            acc += ww.w * x3;
            return acc;
        };
        const cint_p sp = (cint_p)M.sp;
        __shared__ f4 red[kRowsPerBlock][16];
        for (int row = r0 + lb; row < r1; row += gx) {  // block-uniform
            const int a0 = sp[row], a1 = sp[row + 1];
            f4 acc = {0.f, 0.f, 0.f, 0.f};
            for (int q = a0 + CH * wv; q < a1; q += CH * kRowsPerBlock) acc = chunk(q, acc);
            acc += shfl_xor4(acc, 16);
            acc += shfl_xor4(acc, 32);
            if (g == 0) red[wv][j] = acc;
            __syncthreads();
            if (wv == 0 && g == 0) {
                const auto lv = ld(row, j);
                f4 t = red[0][j];
#pragma unroll
                for (int k = 1; k < kRowsPerBlock; ++k) t += red[k][j];
                epi(row, j, t, lv);
            }
            __syncthreads();
        }
    }
}

// part[s*G + block] for samples 4j + c, v[c] held by the lanes j, j + 16,
// j + 32, j + 48 (summed across the four lane groups first)
__device__ inline void b_partial4(double* part, const double (&vin)[4]) {
    __shared__ double sp[kRowsPerBlock][kWave];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    double v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        v[c] = vin[c] + __shfl_xor(vin[c], 16);
        v[c] += __shfl_xor(v[c], 32);
    }
    if (lane < 16)
#pragma unroll
        for (int c = 0; c < 4; ++c) sp[wv][4 * lane + c] = v[c];
    __syncthreads();
    if (wv == 0) {
        double t = 0.0;
        for (int k = 0; k < kRowsPerBlock; ++k) t += sp[k][lane];
        part[(size_t)lane * gridDim.x + blockIdx.x] = t;
    }
    __syncthreads();
}

// Writes the block's per-sample partial sum v (lane = sample) to part[s*G + block].
__device__ inline void b_partial(double* part, int S, double v) {
    __shared__ double sp[kRowsPerBlock][kWave];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    sp[wv][lane] = v;
    __syncthreads();
    if (wv == 0 && lane < S) {
        double t = 0.0;
        for (int k = 0; k < kRowsPerBlock; ++k) t += sp[k][lane];
        part[(size_t)lane * gridDim.x + blockIdx.x] = t;
    }
    __syncthreads();
}

// Sum of part[s*G .. s*G+G) for sample s = blockIdx.x, returned to thread 0.
__device__ inline double b_total(const double* part, int G) {
    __shared__ double sr[kBlock / kWave];
    const int s = blockIdx.x;
    double t = 0.0;
    for (int g = threadIdx.x; g < G; g += kBlock) t += part[(size_t)s * G + g];
    t = wave_sum(t);
    if ((threadIdx.x & (kWave - 1)) == 0) sr[threadIdx.x / kWave] = t;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int k = 0; k < kBlock / kWave; ++k) r += sr[k];
    return r;
}

// ---------------------------------------------------------------- outer --
__global__ __launch_bounds__(kBlock) void k_b_fix(int n, int S, const unsigned char* __restrict__ fixed,
                                                  const double* __restrict__ b, double* __restrict__ x) {
    const size_t tot = (size_t)n * S;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock)
        if (fixed[e / S]) x[e] = b[e];
}

// r = b - A x in FP64, stored as rT = (T) r (the inner solve's right-hand
// side), partials of (b,b) and (r,r).  A: FP64 weights, offsets of FP64 rows.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_resid(SlotArgs A, int S, const double* __restrict__ b,
                                                    const double* __restrict__ x, T* __restrict__ rT,
                                                    double* part_bb, double* part_rr) {
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < S;
    const int lc = min(lane, S - 1);
    double vb = 0.0, vr = 0.0;
    auto ld = [&](int row) { return b[(size_t)row * S + lc]; };
    auto epi = [&](int row, double acc, double bi) {
        if (on) {
            const size_t ee = (size_t)row * S + lane;
            const double ri = bi - acc;
            rT[ee] = (T)ri;
            vb += bi * bi;
            vr += ri * ri;
        }
    };
    slot_walk<double, double, 1>(A, x, lc, ld, epi);
    b_partial(part_bb, S, vb);
    b_partial(part_rr, S, vr);
}

// outer decision per sample; inner tolerance and initial inner state.  track:
// keeps the largest iteration count of the refinement step that has ended.
__global__ void k_b_outer_red(int G, int S, const double* part_bb, const double* part_rr, double tol, double itol,
                              OState* os, BState* bs, int* track) {
    const int s = blockIdx.x;
    const double bb = b_total(part_bb, G);
    __syncthreads();
    const double rr = b_total(part_rr, G);
    if (threadIdx.x == 0 && s < S) {
        os->bb[s] = bb;
        os->rr[s] = rr;
        const bool done = !(rr > tol * tol * bb) || !std::isfinite(rr);
        os->done[s] = !std::isfinite(rr) || !std::isfinite(bb) ? 2 : done ? 1 : 0;
        // inner target: the final tolerance, or a relative itol for the
        // refinement steps, whichever is looser
        const double a2 = tol * tol * bb;
        const double i2 = itol * itol * rr;
        bs->itol2[s] = std::max(a2, i2);
        bs->rr[s] = rr;
        if (track && bs->iters[s] > 0) atomicMax(track, bs->iters[s]);
        bs->active[s] = done ? 0 : 1;
        bs->iters[s] = 0;
        bs->beta[s] = 0.0;
        bs->alpha[s] = 0.0;
        bs->gam[s] = 0.0;
    }
}

__global__ __launch_bounds__(kBlock) void k_b_sum2(size_t tot, const double* __restrict__ a,
                                                   const double* __restrict__ b, double* __restrict__ c) {
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock)
        c[e] = a[e] + b[e];
}

// x += sum_k alpha_k p_k = sum_i c_i z_i of an inner solve of K iterations, from
// the kept preconditioned residuals z_i (ring of [n][S] vectors) and the
// alpha_i, beta_i of every sample (ah, bh: [i][kMaxS]).  Iterations a sample did not take have
// alpha 0 (and beta 0 after them), so c_i = 0 selects their z_i (whose
// contents may be stale) out of the sum.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_combine(size_t NS, int S, int K, const T* __restrict__ ring,
                                                      const double* __restrict__ ah, const double* __restrict__ bh,
                                                      double* __restrict__ x) {
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < NS; e += (size_t)gridDim.x * kBlock) {
        const int sm = (int)(e % S);
        double acc = 0.0;
        combination_coefficients(K, ah + sm, bh + sm, kMaxS, [&](int i, double c) {
            const T v = ring[(size_t)i * NS + e];
            acc += c != 0.0 ? c * (double)v : 0.0;
        });
        x[e] += acc;
    }
}

// c_i of k_b_combine for every sample (thread s): ch[i * kMaxS + s], i < K
__global__ void k_b_coef(int S, int K, const double* __restrict__ ah, const double* __restrict__ bh,
                         double* __restrict__ ch) {
    const int sm = threadIdx.x;
    if (sm >= S) return;
    combination_coefficients(K, ah + sm, bh + sm, kMaxS, [&](int i, double c) { ch[i * kMaxS + sm] = c; });
}

// k_b_combine for S = 64 with the c_i from k_b_coef (staged in LDS, K <=
// kCombineK): four samples per thread (vector loads of each z_i)
constexpr int kCombineK = 48;
// four consecutive elements as FP64 (one 16-byte load for float, two for double)
template <typename T>
__device__ inline void load4d(const T* p, double (&v)[4]) {
    if constexpr (sizeof(T) == 4) {
        const f4 a = *(const f4*)p;
        v[0] = a.x;
        v[1] = a.y;
        v[2] = a.z;
        v[3] = a.w;
    } else {
        typedef double d2 __attribute__((ext_vector_type(2)));
        const d2 a = ((const d2*)p)[0], b = ((const d2*)p)[1];
        v[0] = a.x;
        v[1] = a.y;
        v[2] = b.x;
        v[3] = b.y;
    }
}
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_combine4(size_t NS, int K, const T* __restrict__ ring,
                                                       const double* __restrict__ ch, double* __restrict__ x) {
    typedef double d2 __attribute__((ext_vector_type(2)));
    typedef double d4 __attribute__((ext_vector_type(4)));
    __shared__ d4 cs[kCombineK * kMaxS / 4];
    for (int t = threadIdx.x; t < K * kMaxS / 4; t += kBlock) cs[t] = ((const d4*)ch)[t];
    __syncthreads();
    const size_t N4 = NS / 4;
    for (size_t e4 = (size_t)blockIdx.x * kBlock + threadIdx.x; e4 < N4; e4 += (size_t)gridDim.x * kBlock) {
        const int q = (int)(e4 % (kMaxS / 4));  // samples 4q .. 4q+3
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        for (int i = 0; i < K; ++i) {
            double v[4];
            load4d(ring + (size_t)i * NS + 4 * e4, v);
            const d4 c = cs[i * (kMaxS / 4) + q];
            acc[0] += c.x != 0.0 ? c.x * v[0] : 0.0;
            acc[1] += c.y != 0.0 ? c.y * v[1] : 0.0;
            acc[2] += c.z != 0.0 ? c.z * v[2] : 0.0;
            acc[3] += c.w != 0.0 ? c.w * v[3] : 0.0;
        }
        d2* xp = (d2*)(x + 4 * e4);
        const d2 x0 = xp[0], x1 = xp[1];
        xp[0] = d2{x0.x + acc[0], x0.y + acc[1]};
        xp[1] = d2{x1.x + acc[2], x1.y + acc[3]};
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_zero(size_t tot, T* __restrict__ x) {
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock) x[e] = (T)0;
}

// ------------------------------------------------------------- inner CG --
// Iteration k: q_k = A p_k = A z_k + beta_k q_{k-1} in one pass (the gathers
// read z_k; q_{k-1} is the row's own entry), with the partial (z_k, q_k):
// (p_k, A p_k) = (z_k, A p_k) as p_{k-1} is A-conjugate to p_k.  The
// directions are never formed: the preconditioned residuals z_k are kept (a
// ring of vectors) with alpha_k and beta_k, and the inner solution
// sum_k alpha_k p_k = sum_i c_i z_i is added once at the end (k_b_combine),
// so no iteration reads or writes a direction or the iterate.
// k = 0: q = A z (q_{-1} not read).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_cg_spmv(SlotArgs A, int S, const T* __restrict__ z, T* __restrict__ q,
                                                      int k, const BState* bs, double* part) {
    if (!any_active(A.gate, A.gate_n)) return;
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < S;
    const int lc = min(lane, S - 1);
    const T beta = k > 0 ? (T)bs->beta[lc] : (T)0;
    double v = 0.0;
    struct ZQ {
        T z, q;
    };
    auto ld = [&](int row) {
        const size_t e = (size_t)row * S + lc;
        return ZQ{z[e], k > 0 ? q[e] : (T)0};
    };
    auto epi = [&](int row, T acc, const ZQ& o) {
        if (on) {
            const T qi = acc + beta * o.q;
            q[(size_t)row * S + lane] = qi;
            v += (double)o.z * (double)qi;
        }
    };
    slot_walk<T, T, kRowsPerStep<T>>(A, z, lc, ld, epi);
    b_partial(part, S, v);
}

// k_b_cg_spmv for 64 FP32 samples, wide gathers
__global__ __launch_bounds__(kBlock) void k_b_cg_spmv_w(SlotArgs A, const float* __restrict__ z, float* __restrict__ q,
                                                        int k, const BState* bs, double* part) {
    if (!any_active(A.gate, A.gate_n)) return;
    const int j = threadIdx.x & 15;
    const f4 beta = k > 0 ? f4{(float)bs->beta[4 * j], (float)bs->beta[4 * j + 1], (float)bs->beta[4 * j + 2],
                               (float)bs->beta[4 * j + 3]}
                          : f4{0.f, 0.f, 0.f, 0.f};
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    struct ZQ {
        f4 z, q;
    };
    auto ld = [&](int row, int jj) {
        const size_t e = (size_t)row * 64 + 4 * jj;
        return ZQ{*(const f4*)(z + e), k > 0 ? *(const f4*)(q + e) : f4{0.f, 0.f, 0.f, 0.f}};
    };
    auto epi = [&](int row, int jj, f4 acc, const ZQ& o) {
        const f4 qi = acc + beta * o.q;
        *(f4*)(q + (size_t)row * 64 + 4 * jj) = qi;
        v[0] += (double)o.z.x * (double)qi.x;
        v[1] += (double)o.z.y * (double)qi.y;
        v[2] += (double)o.z.z * (double)qi.z;
        v[3] += (double)o.z.w * (double)qi.w;
    };
    wide_walk<false>(A, z, ld, epi);
    b_partial4(part, v);
}

__global__ void k_b_red_pq(int G, int S, const double* part, BState* bs, double* ah) {
    const int s = blockIdx.x;
    const double pq = b_total(part, G);
    if (threadIdx.x == 0 && s < S) {
        const bool ok = bs->active[s] && pq > 0.0 && std::isfinite(pq);
        if (bs->active[s] && !ok) bs->active[s] = 0;  // breakdown: freeze the sample
        const double a = ok ? bs->gam[s] / pq : 0.0;
        bs->alpha[s] = a;
        ah[s] = a;
    }
}

// r -= alpha q; partial (r, r)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_cg_update(int n, int S, const T* __restrict__ q, T* __restrict__ r,
                                                        const BState* bs, double* part) {
    if (!any_active(bs->active, S)) return;
    const int ln = threadIdx.x & (kWave - 1);
    const T alpha = ln < S ? (T)bs->alpha[ln] : (T)0;
    double v = 0.0;
    B_ROW_LOOP(n) {
        if (on) {
            const size_t e = (size_t)row * S + lane;
            const T ri = r[e] - alpha * q[e];
            r[e] = ri;
            v += (double)ri * (double)ri;
        }
    }
    b_partial(part, S, v);
}

// after r -= alpha q: the iteration count and convergence on ||r||^2,
// decided before the preconditioner runs, so that a batch whose samples
// have all converged skips the V-cycle (its z would never be used: the
// correction sums alpha_k p_k over the iterations taken)
__global__ void k_b_red_rr(int G, int S, const double* part_rr, BState* bs) {
    const int s = blockIdx.x;
    const double rr = b_total(part_rr, G);
    if (threadIdx.x == 0 && s < S && bs->active[s]) {
        bs->iters[s] += 1;
        bs->rr[s] = rr;
        if (!(rr > bs->itol2[s]) || !std::isfinite(rr)) bs->active[s] = 0;
    }
}

// after z = M r: gamma and beta (bh[s]: the next iteration's slot of the
// beta history).  k < 0, the first call of an inner solve, also decides
// convergence on the outer residual's ||r||^2; later iterations decide it
// in k_b_red_rr.
__global__ void k_b_red_rz(int G, int S, const double* part_rz, int k, BState* bs, double* bh) {
    const int s = blockIdx.x;
    const double rz = b_total(part_rz, G);
    if (threadIdx.x == 0 && s < S) {
        const double r2 = bs->rr[s];
        bool act = bs->active[s] && std::isfinite(rz);
        if (k < 0) act = act && r2 > bs->itol2[s] && std::isfinite(r2);
        bs->beta[s] = (act && k >= 0 && bs->gam[s] != 0.0) ? rz / bs->gam[s] : 0.0;
        bh[s] = bs->beta[s];
        bs->gam[s] = rz;
        bs->active[s] = act ? 1 : 0;
    }
}

// --------------------------------------------------------- AMG V-cycle --
// Level 0 upwards: z = U [r | x_c] (r's tail holds the coarse correction), and
// the partial (r, z).  One product with U = [2 w D^-1 - w D^-1 A w D^-1 | Q] in
// place of the prolongation (x = w D^-1 r + P x_c, written and gathered again) and
// the post-smoothing; the levels below use the same form, so a level costs two
// launches instead of three.  Bound by the gathers from L2 and, on small meshes,
// by the launch: 24 FP64 samples at 38,025 nodes 1.54 -> 1.49 ms per evaluation.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_up(SlotArgs U, int S, const T* __restrict__ r, T* __restrict__ z,
                                                 double* part) {
    if (!any_active(U.gate, U.gate_n)) return;
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < S;
    const int lc = min(lane, S - 1);
    double v = 0.0;
    auto ld = [&](int row) { return r[(size_t)row * S + lc]; };
    auto epi = [&](int row, T acc, T ri) {
        if (on) {
            z[(size_t)row * S + lane] = acc;
            v += (double)ri * (double)acc;
        }
    };
    slot_walk<T, T, kRowsPerStep<T>>(U, r, lc, ld, epi);
    b_partial(part, S, v);
}

// k_b_up for 64 FP32 samples, wide gathers
__global__ __launch_bounds__(kBlock) void k_b_up_w(SlotArgs U, const float* __restrict__ r, float* __restrict__ z,
                                                   double* part) {
    if (!any_active(U.gate, U.gate_n)) return;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    auto ld = [&](int row, int j) { return *(const f4*)(r + (size_t)row * 64 + 4 * j); };
    auto epi = [&](int row, int j, f4 acc, f4 ri) {
        *(f4*)(z + (size_t)row * 64 + 4 * j) = acc;
        v[0] += (double)ri.x * (double)acc.x;
        v[1] += (double)ri.y * (double)acc.y;
        v[2] += (double)ri.z * (double)acc.z;
        v[3] += (double)ri.w * (double)acc.w;
    };
    wide_walk<false>(U, r, ld, epi);
    b_partial4(part, v);
}

// y = M x for 64 FP32 samples
template <bool BLK>
__global__ __launch_bounds__(kBlock) void k_b_spmm_w(SlotArgs M, const float* __restrict__ x, float* __restrict__ y) {
    if (!any_active(M.gate, M.gate_n)) return;
    auto ld = [&](int, int) { return 0; };
    auto epi = [&](int row, int j, f4 acc, int) { *(f4*)(y + (size_t)row * 64 + 4 * j) = acc; };
    wide_walk<BLK>(M, x, ld, epi);
}

// ------------------------------------------------------ fields and LLG --
// The per-node operators (exchange, grad, tGrad, curl) share the union
// pattern, stored in row slots (SlotArgs) with FP64-row offsets; the slot
// weights of each operator and the slot columns are separate arrays.  A row
// is walked in halves of 8 slots: offsets, columns and weights by scalar
// loads, gathers by buffer loads with the row offset (plus the component's
// byte offset) as the SGPR operand.  Sums run in entry order (padding slots
// have weight 0).
constexpr int kHalf = 8;

__device__ inline double buf_ld8(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

// b = sum_d tGrad_d (Js m_d) / mu0 for every sample (DemagField.cpp:124-136);
// the slot weights hold tGrad_d(i, j) Js_j / mu0 (set at batch creation)
__global__ __launch_bounds__(kBlock) void k_b_div_l2(SlotArgs P, const double* __restrict__ wty,
                                                  const double* __restrict__ wtz, int S,
                                                  const double* __restrict__ m, double* __restrict__ out) {
    const int n = P.n;
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < S;
    const int lc = min(lane, S - 1);
    const int c8 = n * S * 8;  // bytes of one component
    const __amdgpu_buffer_rsrc_t mr = gather_rsrc(m, 3 * c8);
    const cint_p sp = (cint_p)P.sp, of = (cint_p)P.off;
    const cw_p<double> wx = (cw_p<double>)P.w, wy = (cw_p<double>)wty, wz = (cw_p<double>)wtz;
    const int vo = lc * 8;
    B_ROW_LOOP_XCD(n) {
        double sx = 0, sy = 0, sz = 0;
        const int a0 = sp[row], a1 = sp[row + 1];
        for (int q = a0; q < a1; q += kHalf) {
            int o[kHalf];
            double mx[kHalf], my[kHalf], mz[kHalf];
#pragma unroll
            for (int k = 0; k < kHalf; ++k) o[k] = of[q + k];
#pragma unroll
            for (int k = 0; k < kHalf; ++k) {
                mx[k] = buf_ld8(mr, vo, o[k]);
                my[k] = buf_ld8(mr, vo, o[k] + c8);
                mz[k] = buf_ld8(mr, vo, o[k] + 2 * c8);
            }
#pragma unroll
            for (int k = 0; k < kHalf; ++k) {
                sx += wx[q + k] * mx[k];
                sy += wy[q + k] * my[k];
                sz += wz[q + k] * mz[k];
            }
        }
        if (on) out[(size_t)row * S + lane] = sx + sy + sz;
    }
}

// ---- FP64 rows of 64 samples with 16-byte lanes (k_b_eval_w) --------------
// Lane l holds samples 2j, 2j+1 (j = l % 32) and takes the even (l < 32) or
// the odd (l >= 32) slots of the row; each half-wavefront picks its slot's
// offset and weight out of the pair read as wavefront-uniform scalars.
// pair_sum adds the two halves' sums and leaves sample l of the row in lane
// l.  Measured at 282,897 nodes: the field kernel 1.01 -> 0.94 ms; the same
// form of the divergence and of the FP64 residual was slower (0.62 -> 0.65,
// 0.21 -> 0.22 ms): their time follows the L2 misses of the gathered rows,
// not the lanes the texture path processes.
typedef double d2v __attribute__((ext_vector_type(2)));

__device__ inline d2v buf_ld16d(__amdgpu_buffer_rsrc_t r, int voff) {
    return __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
}

__device__ inline double pair_sum(d2v s) {
    s.x += __shfl_xor(s.x, 32);
    s.y += __shfl_xor(s.y, 32);
    const int l = threadIdx.x & (kWave - 1);
    const double vx = __shfl(s.x, l >> 1), vy = __shfl(s.y, l >> 1);
    return (l & 1) ? vy : vx;
}

// ---- FP64 gathers from tiles in LDS -----------------------------------------
// The kernels that gather FP64 rows (divergence, fields, outer residual) moved
// every neighbour's samples from L2 once per entry of the operator, about 15
// times per node, at the rate of the L2 (11 to 12 TB/s of gathered lines at
// 282,897 nodes).  Here a block takes a unit: a tile of up to 32 rows (chosen to
// share neighbours, see TileOp) and 16 samples.  It stages the distinct nodes
// that the rows refer to, about four per row, in LDS and gathers from there.
// Lane j of a 16-lane group holds sample 16 c + j of its group's row; the
// row's slots (place in the tile, weights) are one coalesced load, lane j
// holding slot j, and slot k is handed to the group by a DPP row broadcast.
// Sixteen samples keep a gathered row one 128-byte line and leave room for
// tiles of 32 rows at two blocks per CU.  A block walks several units and is
// pipelined over them: while it computes one, the nodes of the next are on
// their way into registers, and the next's slots and the node list of the one
// after that are being read (one unit at a time, without this, every unit waits for
// four dependent loads, and the kernels were no faster than the gathers
// from L2).  64 samples at 282,897 nodes, against the gathers from L2: fields
// 1,006 -> 591 us, divergence 513 -> 282, FP64 residual 216 -> 134; 24 samples
// at 38,025 nodes 102 -> 39, 55 -> 20 and 25 -> 12.  A third of the lanes' time
// goes into vector instructions, a third into LDS.  Two (fields, divergence) and
// three (residual) blocks per CU; the residual with 2, 3 and 4 of them: 129.2,
// 129.9 and 132.7 us for 64 samples at 282,897 nodes, 10.6, 10.8 and 11.8 for 24 at 38,440.
constexpr int kTileThreads = 512;
constexpr int kTileRows = kTileThreads / 16;
constexpr int kTileS = 16;       // samples of a unit
constexpr int kTileNodes = 128;  // nodes of a tile: 64 KB of LDS with four components

struct TileRow {
    int row, q0;  // its first slot
    int more;     // chunks of kSlot slots << 16 | its own place in the tile
};

struct TileArgs {
    int nt;               // tiles
    int S, nch;           // samples, chunks of kTileS of them
    const int* row0;      // nt + 1: entries of `rows` of a tile
    const TileRow* rows;
    const int* node0;     // nt + 1: its entries of `nodes`
    const int* nodes;
    const unsigned short* loc;  // per slot: the gathered node's place in the tile (padding: the row's own)
};

// blocks of a tile kernel with `percu` of them per CU: each XCD's blocks a
// multiple of the chunks, so that a block keeps to one chunk
inline int tile_blocks(int nch, int percu) { return kXcd * (32 * percu / nch * nch); }

// A unit of work.  k counts the units of a block: XCD-contiguous tiles, the
// chunks of a tile in neighbouring blocks (they share the slots), neighbouring
// tiles next to them.  Past the end: valid = false, with the data of the last
// tile (loads need no conditions).
struct TileUnit {
    bool valid;
    int r0, nr, n0, nn;
};
__device__ inline int tile_chunk(const TileArgs& t, int samples = kTileS) {
    return (int)(blockIdx.x / kXcd) % t.nch * samples;
}
__device__ inline TileUnit tile_unit(const TileArgs& t, int k) {
    const int x = blockIdx.x % kXcd, bx = gridDim.x / kXcd / t.nch;
    const int per = (t.nt + kXcd - 1) / kXcd, in = (int)(blockIdx.x / kXcd) / t.nch + k * bx;
    const int tile = min(x * per + in, t.nt - 1);
    const cint_p r = (cint_p)t.row0, c = (cint_p)t.node0;
    const int r0 = r[tile], r1 = r[tile + 1], n0 = c[tile], n1 = c[tile + 1];
    return TileUnit{in < per && x * per + in < t.nt, r0, r1 - r0, n0, n1 - n0};
}

// the value that lane K of the 16-lane group holds
template <int K>
__device__ inline int bcast16(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + K, 0xf, 0xf, true);  // row_newbcast
}
template <int K>
__device__ inline double bcast16(double v) {
    return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + K, 0xf, 0xf, true);
}
template <int K>
__device__ inline float bcast16(float v) {
    return __builtin_bit_cast(float, bcast16<K>(__builtin_bit_cast(int, v)));
}
template <class F, int... K>
__device__ inline void each16(F&& f, std::integer_sequence<int, K...>) {
    (f(std::integral_constant<int, K>{}), ...);
}

// The element and lane layout of a walk: T, VEC samples per lane (a unit has
// 16 VEC samples: 128 bytes of a node in FP64, 256 in FP32), and whether rows of
// samples are 16-byte aligned.
template <typename T_, int VEC_, bool ALIGNED_, int NODES = kTileNodes>
struct TileType {
    using T = T_;
    static constexpr int VEC = VEC_;
    static constexpr int kSamples = 16 * VEC;
    typedef T Vec __attribute__((ext_vector_type(VEC)));
    using Lane = std::conditional_t<VEC == 1, T, Vec>;  // a lane's samples
    static constexpr int kPer = ALIGNED_ ? 16 / (int)sizeof(T) : 1;  // elements per staging load
    typedef T StageVec __attribute__((ext_vector_type(16 / sizeof(T))));
    using Stage = std::conditional_t<ALIGNED_, StageVec, T>;
    static constexpr int kLanes = kSamples / kPer;  // lanes per staged row of samples
    static constexpr int kGroups = kTileThreads / kLanes;
    static constexpr int kRounds = (NODES + kGroups - 1) / kGroups;
    static constexpr int kStaged = kRounds * kGroups;  // node places of a tile in LDS
};

// The first NP chunks of 16 slots of this group's row: lane j's place and NW
// weights of the chunk's slot j
template <class TT, int NW>
struct TileChunk {
    using T = typename TT::T;
    int loc;
    T w[NW];
    __device__ void load(const TileArgs& t, int q, const T* const (&src)[NW]) {
        q += threadIdx.x & 15;
        loc = t.loc[q];
#pragma unroll
        for (int i = 0; i < NW; ++i) w[i] = src[i][q];
    }
    // f(components gathered by slot k, its weights) for k = 0 .. 15
    template <int NC, class F>
    __device__ void each(const T* lds, F&& f) const {
        const int at = loc * (NC * TT::kSamples);
        const T* mine = lds + (threadIdx.x & 15) * TT::VEC;
        each16(
            [&](auto kk) {
                constexpr int K = decltype(kk)::value;
                const T* g = mine + bcast16<K>(at);
                typename TT::Lane v[NC];
                T ww[NW];
#pragma unroll
                for (int c = 0; c < NC; ++c) v[c] = *(const typename TT::Lane*)(g + c * TT::kSamples);
#pragma unroll
                for (int i = 0; i < NW; ++i) ww[i] = bcast16<K>(w[i]);
                f(v, ww);
            },
            std::make_integer_sequence<int, kSlot>{});
    }
};

// A unit on its way through the pipeline: first its tile's bounds, node list
// and this group's row, then the nodes (in the walk's registers) and the
// row's first slots (NP chunks).
template <class TT, int NW, int NP>
struct TileStep {
    TileUnit u;
    int id[TT::kRounds];
    TileRow row;
    TileChunk<TT, NW> chunk[NP];
    __device__ void slots(const TileArgs& t, const typename TT::T* const (&w)[NW]) {
#pragma unroll
        for (int i = 0; i < NP; ++i) chunk[i].load(t, row.q0 + (i < row.more >> 16 ? i * kSlot : 0), w);
    }
    __device__ void lists(const TileArgs& t, int k) {
        u = tile_unit(t, k);
#pragma unroll
        for (int r = 0; r < TT::kRounds; ++r)
            id[r] = t.nodes[u.n0 + min((int)threadIdx.x / TT::kLanes + r * TT::kGroups, u.nn - 1)];
        row = t.rows[u.r0 + min((int)threadIdx.x / 16, u.nr - 1)];
    }
};

// The units of this block, pipelined.  NC components of a tile's nodes in
// place [node][component][16 VEC] in LDS, component c < NC - 1 from m + c cs and
// the last from `last`.  Lanes past the last sample load the last one's data;
// groups without a row (nr < kTileRows) compute the tile's last row once more;
// neither stores.  Per unit: begin(row) loads the row's own data, add(v, w) per
// entry, end(row, lds, on) when the row is summed (on: this group's row and
// this lane's samples exist).
template <class TT, int NC, int NW, int NP = 1, class Begin, class Add, class End>
__device__ inline void tile_walk(const TileArgs& t, const typename TT::T* m, size_t cs, const typename TT::T* last,
                                 const typename TT::T* const (&w)[NW], typename TT::T* lds, Begin&& begin, Add&& add,
                                 End&& end) {
    using Step = TileStep<TT, NW, NP>;
    using V = typename TT::Stage;
    constexpr int kLanes = TT::kLanes, kGroups = TT::kGroups, kRounds = TT::kRounds, kPer = TT::kPer;
    V v[kRounds][NC];
    const int s0 = tile_chunk(t, TT::kSamples), S = t.S;
    const bool lane_on = s0 + (int)(threadIdx.x & 15) * TT::VEC < S;
    const int ks = min(s0 + (int)(threadIdx.x % kLanes) * kPer, S - kPer);
    auto load = [&](const Step& p) {
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const size_t e = (size_t)p.id[r] * S + ks;
#pragma unroll
            for (int c = 0; c < NC; ++c) v[r][c] = *(const V*)((c == NC - 1 ? last : m + c * cs) + e);
        }
    };
    auto store = [&]() {  // places past the tile's last node are not read
#pragma unroll
        for (int r = 0; r < kRounds; ++r)
#pragma unroll
            for (int c = 0; c < NC; ++c)
                *(V*)(lds + ((threadIdx.x / kLanes + r * kGroups) * NC + c) * TT::kSamples +
                      (threadIdx.x % kLanes) * kPer) = v[r][c];
    };
    Step p[3];
    p[0].lists(t, 0);
    if (!p[0].u.valid) return;  // the whole block
    load(p[0]);
    p[0].slots(t, w);
    p[1].lists(t, 1);
    store();
    __syncthreads();
    int k = 2;
    // computes unit c while c1's data are loaded and c2's lists are read; false at the end
    auto step = [&](Step& c, Step& c1, Step& c2) {
        begin(c.row);
        load(c1);
        c1.slots(t, w);
        c2.lists(t, k++);
        c.chunk[0].template each<NC>(lds, add);
#pragma unroll
        for (int i = 1; i < NP; ++i)
            if (i < c.row.more >> 16) c.chunk[i].template each<NC>(lds, add);
        for (int i = NP; i < c.row.more >> 16; ++i) {
            c.chunk[0].load(t, c.row.q0 + i * kSlot, w);
            c.chunk[0].template each<NC>(lds, add);
        }
        end(c.row, lds, lane_on && (int)threadIdx.x / 16 < c.u.nr);
        if (!c1.u.valid) return false;
        __syncthreads();
        store();
        __syncthreads();
        return true;
    };
    while (step(p[0], p[1], p[2]) && step(p[1], p[2], p[0]) && step(p[2], p[0], p[1])) {
    }
}

// the c-th of a lane's samples
template <class TT>
__device__ inline typename TT::T lane_at(const typename TT::Lane& v, int c) {
    if constexpr (TT::VEC == 1) return v;
    else return v[c];
}

// The block's sums v (a lane's samples) to part[s * gridDim.x + block], zero for
// the samples of other chunks, through the walk's LDS
template <class TT>
constexpr int kTileElems = TT::kStaged * TT::kSamples;
template <class TT>
__device__ inline void tile_partial(typename TT::T* lds, double* part, int S, const double (&v)[TT::VEC], int s0) {
    constexpr int kPerRow = TT::kSamples;
    double* red = reinterpret_cast<double*>(lds);  // [kTileRows / 2][16 VEC]
    static_assert(kTileElems<TT> * sizeof(typename TT::T) >= kTileRows / 2 * kPerRow * sizeof(double),
                  "the partial sums of two groups at a time");
    const int g = threadIdx.x / 16, j = threadIdx.x & 15;
    __syncthreads();
    double u[TT::VEC];
#pragma unroll
    for (int c = 0; c < TT::VEC; ++c) u[c] = v[c] + __shfl_xor(v[c], 16);
    if ((g & 1) == 0)
#pragma unroll
        for (int c = 0; c < TT::VEC; ++c) red[(g / 2) * kPerRow + TT::VEC * j + c] = u[c];
    __syncthreads();
    const int sm = threadIdx.x, q = sm - s0;
    if (sm >= S) return;
    double s = 0.0;
    if (q >= 0 && q < kPerRow)
#pragma unroll
        for (int k = 0; k < kTileRows / 2; ++k) s += red[k * kPerRow + q];
    part[(size_t)sm * gridDim.x + blockIdx.x] = s;
}

// b = sum_d tGrad_d (Js m_d) / mu0, as k_b_div_l2 (which gathers from L2)
constexpr int kDivPerCu = 2;
template <bool EVEN>
__global__ __launch_bounds__(kTileThreads, 2 * kDivPerCu) void k_b_div(TileArgs t, const double* __restrict__ wx,
                                                                        const double* __restrict__ wy,
                                                                        const double* __restrict__ wz, int n,
                                                                        const double* __restrict__ m,
                                                                        double* __restrict__ out) {
    __shared__ double lds[kTileNodes * 3 * kTileS];
    const size_t NS = (size_t)n * t.S;
    const int s = tile_chunk(t) + (threadIdx.x & 15);
    double sx = 0.0, sy = 0.0, sz = 0.0;
    tile_walk<TileType<double, 1, EVEN>, 3, 3>(
        t, m, NS, m + 2 * NS, {wx, wy, wz}, lds, [&](const TileRow&) { sx = sy = sz = 0.0; },
        [&](const double (&v)[3], const double (&w)[3]) {
            sx += w[0] * v[0];
            sy += w[1] * v[1];
            sz += w[2] * v[2];
        },
        [&](const TileRow& r, const double*, bool on) {
            if (on) out[(size_t)r.row * t.S + s] = sx + sy + sz;
        });
}

struct BEvalArgs {
    SlotArgs P;                        // union pattern in slots, w = exchange weights (may be null)
    const double* gx; const double* gy; const double* gz;
    const double* cx; const double* cy; const double* cz;
    int S, n;
    const double* m; const double* u;   // u = u1 + u2
    const double* invjs; const double* ku; const double* kaxis;
    const double* dmi_fac; const double* nvs;
    const double* hext;   // [3][S] per-sample uniform applied field
    const double* hfield; // 3n per-node applied field shared by every sample (or null)
    double alpha;
    int variant;
    double* dmdt; double* heff;
    double* torque;       // [S], zeroed before
    double* mnext;        // if set: the explicit Euler step m + dt dm/dt, renormalised (a buffer apart from m)
    double dt;
};

// dm/dt of one (node, sample) into a.dmdt, and the Euler step into a.mnext
// when asked for (the arithmetic of k_b_euler)
__device__ inline void b_store_llg(const BEvalArgs& a, size_t e, size_t NS, double mx, double my, double mz,
                                   double dx, double dy, double dz) {
    a.dmdt[e] = dx;
    a.dmdt[NS + e] = dy;
    a.dmdt[2 * NS + e] = dz;
    if (a.mnext) {
        const double x = mx + a.dt * dx, y = my + a.dt * dy, z = mz + a.dt * dz;
        const double l = sqrt(x * x + y * y + z * z);
        const double f = l > 0.0 ? 1.0 / l : 1.0;
        a.mnext[e] = x * f;
        a.mnext[NS + e] = y * f;
        a.mnext[2 * NS + e] = z * f;
    }
}

// Fused Heff + LLG for every (node, sample): TheLLG.cpp:238-254 and
// EffFieldGPU.cu:316-362, with the demag field -grad(u1 + u2).
template <bool DMI>
__global__ __launch_bounds__(kBlock) void k_b_eval(BEvalArgs a) {
    const int S = a.S;
    const size_t NS = (size_t)a.n * S;
    const int n = a.n;
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < S;
    const int lc = min(lane, S - 1);
    const int c8 = n * S * 8;
    const __amdgpu_buffer_rsrc_t mr = gather_rsrc(a.m, 3 * c8);
    const __amdgpu_buffer_rsrc_t ur = gather_rsrc(a.u, c8);
    const cint_p sp = (cint_p)a.P.sp, of = (cint_p)a.P.off;
    const cw_p<double> wx = (cw_p<double>)a.P.w;
    const cw_p<double> gx = (cw_p<double>)a.gx, gy = (cw_p<double>)a.gy, gz = (cw_p<double>)a.gz;
    const cw_p<double> cx = (cw_p<double>)a.cx, cy = (cw_p<double>)a.cy, cz = (cw_p<double>)a.cz;
    const bool exch = a.P.w != nullptr;
    const int vo = lc * 8;
    double tmax = 0.0;
    B_ROW_LOOP_XCD(n) {
        double ex = 0, ey = 0, ez = 0, dx = 0, dy = 0, dz = 0, cxs = 0, cys = 0, czs = 0;
        const int a0 = sp[row], a1 = sp[row + 1];
        for (int q = a0; q < a1; q += kHalf) {
            int o[kHalf];
            double mv[kHalf][3], uv[kHalf];
#pragma unroll
            for (int k = 0; k < kHalf; ++k) o[k] = of[q + k];
#pragma unroll
            for (int k = 0; k < kHalf; ++k) {
                mv[k][0] = buf_ld8(mr, vo, o[k]);
                mv[k][1] = buf_ld8(mr, vo, o[k] + c8);
                mv[k][2] = buf_ld8(mr, vo, o[k] + 2 * c8);
                uv[k] = buf_ld8(ur, vo, o[k]);
            }
#pragma unroll
            for (int k = 0; k < kHalf; ++k) {
                const double mx = mv[k][0], my = mv[k][1], mz = mv[k][2];
                if (exch) {
                    const double xc = wx[q + k];
                    ex += xc * mx;
                    ey += xc * my;
                    ez += xc * mz;
                }
                dx += gx[q + k] * uv[k];
                dy += gy[q + k] * uv[k];
                dz += gz[q + k] * uv[k];
                if (DMI) {
                    const double X = cx[q + k], Y = cy[q + k], Z = cz[q + k];
                    cxs += Y * mz - Z * my;
                    cys += Z * mx - X * mz;
                    czs += X * my - Y * mx;
                }
            }
        }
        if (!on) continue;
        const size_t e = (size_t)row * S + lane;
        const double mx = a.m[e], my = a.m[NS + e], mz = a.m[2 * NS + e];
        double hx = ex, hy = ey, hz = ez;
        if (a.ku) {
            const double kx = a.kaxis[row], ky = a.kaxis[a.n + row], kz = a.kaxis[2 * a.n + row];
            const double f = 2.0 * a.ku[row] * (kx * mx + ky * my + kz * mz);
            hx += f * kx;
            hy += f * ky;
            hz += f * kz;
        }
        if (DMI) {
            const double sx = a.nvs[row], sy = a.nvs[a.n + row], sz = a.nvs[2 * a.n + row];
            const double f = a.dmi_fac[row];
            hx += ((my * sz - mz * sy) - 2.0 * cxs) * f;
            hy += ((mz * sx - mx * sz) - 2.0 * cys) * f;
            hz += ((mx * sy - my * sx) - 2.0 * czs) * f;
        }
        const double ij = a.invjs ? a.invjs[row] : 1.0;
        hx = hx * ij + a.hext[lane] - dx;
        hy = hy * ij + a.hext[S + lane] - dy;
        hz = hz * ij + a.hext[2 * S + lane] - dz;
        if (a.hfield) {
            hx += a.hfield[row];
            hy += a.hfield[n + row];
            hz += a.hfield[2 * n + row];
        }
        if (a.heff) {
            a.heff[e] = hx;
            a.heff[NS + e] = hy;
            a.heff[2 * NS + e] = hz;
        }
        const double tx = my * hz - mz * hy, ty = mz * hx - mx * hz, tz = mx * hy - my * hx;
        const double bx = my * tz - mz * ty, by = mz * tx - mx * tz, bz = mx * ty - my * tx;
        if (a.variant == TM_LLG_NOPREC)
            b_store_llg(a, e, NS, mx, my, mz, -a.alpha * bx, -a.alpha * by, -a.alpha * bz);
        else
            b_store_llg(a, e, NS, mx, my, mz, -tx - a.alpha * bx, -ty - a.alpha * by, -tz - a.alpha * bz);
        tmax = fmax(tmax, sqrt(tx * tx + ty * ty + tz * tz));
    }
    if (!a.torque) return;
    __shared__ double st[kRowsPerBlock][kWave];
    const int ln = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    st[wv][ln] = tmax;
    __syncthreads();
    if (wv == 0 && ln < S) {
        double t = st[0][ln];
        for (int k = 1; k < kRowsPerBlock; ++k) t = fmax(t, st[k][ln]);
        atomic_max_nonneg(a.torque + ln, t);
    }
}

// k_b_eval for S = 64 (16-byte lanes, slots taken in pairs, two pairs per
// step)
template <bool DMI>
__global__ __launch_bounds__(kBlock) void k_b_eval_w(BEvalArgs a) {
    constexpr int S = kMaxS;
    constexpr int KP = 2;  // slot pairs per step
    const int n = a.n;
    const size_t NS = (size_t)n * S;
    const int lane = threadIdx.x & (kWave - 1);
    const bool odd = lane >= 32;
    const int vo = (lane & 31) * 16;
    const int c8 = n * S * 8;
    const __amdgpu_buffer_rsrc_t mr = gather_rsrc(a.m, 3 * c8);
    const __amdgpu_buffer_rsrc_t ur = gather_rsrc(a.u, c8);
    const cint_p sp = (cint_p)a.P.sp, of = (cint_p)a.P.off;
    const cw_p<double> wx = (cw_p<double>)a.P.w;
    const cw_p<double> gx = (cw_p<double>)a.gx, gy = (cw_p<double>)a.gy, gz = (cw_p<double>)a.gz;
    const cw_p<double> cx = (cw_p<double>)a.cx, cy = (cw_p<double>)a.cy, cz = (cw_p<double>)a.cz;
    const bool exch = a.P.w != nullptr;
    double tmax = 0.0;
    B_ROW_LOOP_XCD(n) {
        const d2v z2 = {0.0, 0.0};
        d2v ex = z2, ey = z2, ez = z2, dx = z2, dy = z2, dz = z2, cxs = z2, cys = z2, czs = z2;
        const int a0 = sp[row], a1 = sp[row + 1];
        for (int q = a0; q < a1; q += 2 * KP) {
            int o[KP];
#pragma unroll
            for (int k = 0; k < KP; ++k) o[k] = vo + (odd ? of[q + 2 * k + 1] : of[q + 2 * k]);
            d2v mv[KP][3], uv[KP];
#pragma unroll
            for (int k = 0; k < KP; ++k) {
                mv[k][0] = buf_ld16d(mr, o[k]);
                mv[k][1] = buf_ld16d(mr, o[k] + c8);
                mv[k][2] = buf_ld16d(mr, o[k] + 2 * c8);
                uv[k] = buf_ld16d(ur, o[k]);
            }
            // the half's weight of pair k: both read as scalars, one picked
            auto pick = [&](cw_p<double> w, int k) { return odd ? w[q + 2 * k + 1] : w[q + 2 * k]; };
#pragma unroll
            for (int k = 0; k < KP; ++k) {
                const d2v mx = mv[k][0], my = mv[k][1], mz = mv[k][2];
                if (exch) {
                    const double xc = pick(wx, k);
                    ex += xc * mx;
                    ey += xc * my;
                    ez += xc * mz;
                }
                dx += pick(gx, k) * uv[k];
                dy += pick(gy, k) * uv[k];
                dz += pick(gz, k) * uv[k];
                if (DMI) {
                    const double X = pick(cx, k), Y = pick(cy, k), Z = pick(cz, k);
                    cxs += Y * mz - Z * my;
                    cys += Z * mx - X * mz;
                    czs += X * my - Y * mx;
                }
            }
        }
        const double Ex = pair_sum(ex), Ey = pair_sum(ey), Ez = pair_sum(ez);
        const double Dx = pair_sum(dx), Dy = pair_sum(dy), Dz = pair_sum(dz);
        double Cx = 0.0, Cy = 0.0, Cz = 0.0;
        if (DMI) {
            Cx = pair_sum(cxs);
            Cy = pair_sum(cys);
            Cz = pair_sum(czs);
        }
        const size_t e = (size_t)row * S + lane;
        const double mx = a.m[e], my = a.m[NS + e], mz = a.m[2 * NS + e];
        double hx = Ex, hy = Ey, hz = Ez;
        if (a.ku) {
            const double kx = a.kaxis[row], ky = a.kaxis[n + row], kz = a.kaxis[2 * n + row];
            const double f = 2.0 * a.ku[row] * (kx * mx + ky * my + kz * mz);
            hx += f * kx;
            hy += f * ky;
            hz += f * kz;
        }
        if (DMI) {
            const double sx = a.nvs[row], sy = a.nvs[n + row], sz = a.nvs[2 * n + row];
            const double f = a.dmi_fac[row];
            hx += ((my * sz - mz * sy) - 2.0 * Cx) * f;
            hy += ((mz * sx - mx * sz) - 2.0 * Cy) * f;
            hz += ((mx * sy - my * sx) - 2.0 * Cz) * f;
        }
        const double ij = a.invjs ? a.invjs[row] : 1.0;
        hx = hx * ij + a.hext[lane] - Dx;
        hy = hy * ij + a.hext[S + lane] - Dy;
        hz = hz * ij + a.hext[2 * S + lane] - Dz;
        if (a.hfield) {
            hx += a.hfield[row];
            hy += a.hfield[n + row];
            hz += a.hfield[2 * n + row];
        }
        if (a.heff) {
            a.heff[e] = hx;
            a.heff[NS + e] = hy;
            a.heff[2 * NS + e] = hz;
        }
        const double tx = my * hz - mz * hy, ty = mz * hx - mx * hz, tz = mx * hy - my * hx;
        const double bx = my * tz - mz * ty, by = mz * tx - mx * tz, bz = mx * ty - my * tx;
        if (a.variant == TM_LLG_NOPREC)
            b_store_llg(a, e, NS, mx, my, mz, -a.alpha * bx, -a.alpha * by, -a.alpha * bz);
        else
            b_store_llg(a, e, NS, mx, my, mz, -tx - a.alpha * bx, -ty - a.alpha * by, -tz - a.alpha * bz);
        tmax = fmax(tmax, sqrt(tx * tx + ty * ty + tz * tz));
    }
    if (!a.torque) return;
    __shared__ double st[kRowsPerBlock][kWave];
    const int wv = threadIdx.x / kWave;
    st[wv][lane] = tmax;
    __syncthreads();
    if (wv == 0) {
        double t = st[0][lane];
        for (int k = 1; k < kRowsPerBlock; ++k) t = fmax(t, st[k][lane]);
        atomic_max_nonneg(a.torque + lane, t);
    }
}

// k_b_eval from tiles in LDS (xw: the exchange weights, zeros without exchange)
constexpr int kEvalPerCu = 2;
template <bool DMI, bool EVEN>
__global__ __launch_bounds__(kTileThreads, DMI && !EVEN ? 2 : 2 * kEvalPerCu) void k_b_eval_t(BEvalArgs a, const double* xw, TileArgs t) {
    __shared__ double lds[kTileNodes * 4 * kTileS];
    constexpr int NW = DMI ? 7 : 4;
    const int S = t.S, n = a.n;
    const size_t NS = (size_t)n * S;
    const int j = threadIdx.x & 15, s = tile_chunk(t) + j, sc = min(s, S - 1);
    const double* w[NW];
    w[0] = xw;
    w[1] = a.gx;
    w[2] = a.gy;
    w[3] = a.gz;
    if constexpr (DMI) {
        w[4] = a.cx;
        w[5] = a.cy;
        w[6] = a.cz;
    }
    __shared__ double hs[3][kTileS];
    if (threadIdx.x < 3 * kTileS) hs[threadIdx.x / kTileS][j] = a.hext[(threadIdx.x / kTileS) * S + sc];
    // no branch around a load of the pipeline: without anisotropy the
    // constants are any values, left out by `end`
    const double* kup = a.ku ? a.ku : a.invjs;
    const double* kap = a.ku ? a.kaxis : a.m;
    double ex, ey, ez, dx, dy, dz, cxs, cys, czs;
    double ku, kx, ky, kz, ij, sx, sy, sz, fd;
    double tmax = 0.0;
    tile_walk<TileType<double, 1, EVEN>, 4, NW>(
        t, a.m, NS, a.u, w, lds,
        [&](const TileRow& r) {
            ex = ey = ez = dx = dy = dz = cxs = cys = czs = 0.0;
            ku = kup[r.row];
            kx = kap[r.row];
            ky = kap[n + r.row];
            kz = kap[2 * n + r.row];
            ij = a.invjs[r.row];
            if constexpr (DMI) {
                sx = a.nvs[r.row];
                sy = a.nvs[n + r.row];
                sz = a.nvs[2 * n + r.row];
                fd = a.dmi_fac[r.row];
            }
        },
        [&](const double (&v)[4], const double (&ww)[NW]) {
            ex += ww[0] * v[0];
            ey += ww[0] * v[1];
            ez += ww[0] * v[2];
            dx += ww[1] * v[3];
            dy += ww[2] * v[3];
            dz += ww[3] * v[3];
            if constexpr (DMI) {
                cxs += ww[5] * v[2] - ww[6] * v[1];
                cys += ww[6] * v[0] - ww[4] * v[2];
                czs += ww[4] * v[1] - ww[5] * v[0];
            }
        },
        [&](const TileRow& r, const double* tile, bool on) {
            if (!on) return;
            const int row = r.row;
            const size_t e = (size_t)row * S + s;
            const double* own = tile + (r.more & 0xffff) * (4 * kTileS) + j;
            const double mx = own[0], my = own[kTileS], mz = own[2 * kTileS];
            double hx = ex, hy = ey, hz = ez;
            if (a.ku) {
                const double f = 2.0 * ku * (kx * mx + ky * my + kz * mz);
                hx += f * kx;
                hy += f * ky;
                hz += f * kz;
            }
            if constexpr (DMI) {
                hx += ((my * sz - mz * sy) - 2.0 * cxs) * fd;
                hy += ((mz * sx - mx * sz) - 2.0 * cys) * fd;
                hz += ((mx * sy - my * sx) - 2.0 * czs) * fd;
            }
            hx = hx * ij + hs[0][j] - dx;
            hy = hy * ij + hs[1][j] - dy;
            hz = hz * ij + hs[2][j] - dz;
            if (a.hfield) {
                hx += a.hfield[row];
                hy += a.hfield[n + row];
                hz += a.hfield[2 * n + row];
            }
            if (a.heff) {
                a.heff[e] = hx;
                a.heff[NS + e] = hy;
                a.heff[2 * NS + e] = hz;
            }
            const double tx = my * hz - mz * hy, ty = mz * hx - mx * hz, tz = mx * hy - my * hx;
            const double bx = my * tz - mz * ty, by = mz * tx - mx * tz, bz = mx * ty - my * tx;
            // -tx - alpha bx (TM_LLG_CLASSIC) or -alpha bx (TM_LLG_NOPREC)
            const bool prec = a.variant != TM_LLG_NOPREC;
            b_store_llg(a, e, NS, mx, my, mz, (prec ? -tx : 0.0) - a.alpha * bx, (prec ? -ty : 0.0) - a.alpha * by,
                        (prec ? -tz : 0.0) - a.alpha * bz);
            tmax = fmax(tmax, sqrt(tx * tx + ty * ty + tz * tz));
        });
    if (a.torque && s < S) atomic_max_nonneg(a.torque + s, tmax);
}

// k_b_resid from tiles in LDS: the block's partials as b_partial lays them out
// (zero for the samples of the other chunks)
constexpr int kResidPerCu = 3;
template <typename T, bool EVEN>
__global__ __launch_bounds__(kTileThreads, 2 * kResidPerCu) void k_b_resid_t(TileArgs t, const double* __restrict__ w,
                                                                            const double* __restrict__ b,
                                                                            const double* __restrict__ x,
                                                                            T* __restrict__ rT, double* part_bb,
                                                                            double* part_rr) {
    __shared__ double lds[kTileNodes * kTileS];
    const int j = threadIdx.x & 15, g = threadIdx.x / 16, s = tile_chunk(t) + j, sc = min(s, t.S - 1);
    double bi = 0.0, acc = 0.0, vb = 0.0, vr = 0.0;
    tile_walk<TileType<double, 1, EVEN>, 1, 1>(
        t, x, 0, x, {w}, lds,
        [&](const TileRow& r) {
            acc = 0.0;
            bi = b[(size_t)r.row * t.S + sc];
        },
        [&](const double (&v)[1], const double (&ww)[1]) { acc += ww[0] * v[0]; },
        [&](const TileRow& r, const double*, bool on) {
            if (!on) return;
            const double ri = bi - acc;
            rT[(size_t)r.row * t.S + s] = (T)ri;
            vb += bi * bi;
            vr += ri * ri;
        });
    __syncthreads();
    static_assert(kTileNodes >= 2 * kTileRows, "the tile's LDS holds the partial sums");
    lds[(2 * g) * kTileS + j] = vb;
    lds[(2 * g + 1) * kTileS + j] = vr;
    __syncthreads();
    const int q = threadIdx.x / kMaxS, sm = threadIdx.x % kMaxS;
    if (q >= 2 || sm >= t.S) return;
    double v = 0.0;
    if (sm >= s - j && sm < s - j + kTileS)
        for (int k = 0; k < kTileRows; ++k) v += lds[(2 * k + q) * kTileS + (sm - (s - j))];
    (q == 0 ? part_bb : part_rr)[(size_t)sm * gridDim.x + blockIdx.x] = v;
}

// k_b_cg_spmv and k_b_cg_spmv_w from tiles in LDS: 64 samples per unit, a float4
// per lane, for 64 FP32 samples; 16 per unit otherwise.  Gathers from L2 are bound
// by the texture unit's four lanes per cycle, these by LDS and the nodes' staging:
// 64 FP32 samples at 282,897 nodes 96 -> 55 us, at 25,785 nodes a sixth less (also
// with fewer units than two per block); 24 FP64 samples at 38,025 nodes
// 24.2 -> 12.8.  Two (float4) and three blocks per CU; at four the float4 form's
// registers spill (123 us).
template <class TT>
constexpr int kSolvePerCu = TT::VEC == 1 ? 3 : 2;
template <class TT>
__global__ __launch_bounds__(kTileThreads, 2 * kSolvePerCu<TT>) void k_b_cg_spmv_t(
    TileArgs t, const typename TT::T* __restrict__ w, const typename TT::T* __restrict__ z, typename TT::T* __restrict__ q,
    int k, const BState* bs, double* part) {
    using T = typename TT::T;
    using Lane = typename TT::Lane;
    constexpr int VEC = TT::VEC;
    __shared__ T lds[kTileElems<TT>];
    if (!any_active(bs->active, kMaxS)) return;
    const int s0 = tile_chunk(t, TT::kSamples), sc = min(s0 + VEC * (int)(threadIdx.x & 15), t.S - VEC);
    Lane beta, acc = {}, old = {};
    if constexpr (VEC == 1) {
        beta = k > 0 ? (T)bs->beta[sc] : (T)0;
    } else {
#pragma unroll
        for (int c = 0; c < VEC; ++c) beta[c] = k > 0 ? (T)bs->beta[sc + c] : (T)0;
    }
    // k = 0: q has no earlier value; z is read in its place and left out
    const T* qo = k > 0 ? q : z;
    double v[VEC] = {};
    tile_walk<TT, 1, 1>(
        t, z, 0, z, {w}, lds,
        [&](const TileRow& r) {
            acc = Lane{};
            old = *(const Lane*)(qo + (size_t)r.row * t.S + sc);
        },
        [&](const Lane (&x)[1], const T (&ww)[1]) { acc += ww[0] * x[0]; },
        [&](const TileRow& r, const T* tile, bool on) {
            if (!on) return;
            const Lane zi = *(const Lane*)(tile + (r.more & 0xffff) * TT::kSamples + VEC * (int)(threadIdx.x & 15));
            const Lane qi = k > 0 ? acc + beta * old : acc;
            *(Lane*)(q + (size_t)r.row * t.S + sc) = qi;
#pragma unroll
            for (int c = 0; c < VEC; ++c) v[c] += (double)lane_at<TT>(zi, c) * (double)lane_at<TT>(qi, c);
        });
    tile_partial<TT>(lds, part, t.S, v, s0);
}

// k_b_up and k_b_up_w from tiles in LDS (rows of about 27 entries: two chunks of
// slots; tiles of up to 192 nodes, since 128 with the coarse ones among them hold
// 26 rows and leave lanes idle): 64 FP32 samples at 282,897 nodes 83 us, where
// prolongation and post-smoothing took 58 + 91 from L2 (160 and 224 nodes: 3 per
// cent slower); at 25,785 nodes a quarter less than k_b_up_w; 24 FP64 samples at
// 38,025 nodes 41 -> 18
template <class TT>
__global__ __launch_bounds__(kTileThreads, 4) void k_b_up_t(TileArgs t, const typename TT::T* __restrict__ w,
                                                            const typename TT::T* __restrict__ r,
                                                            typename TT::T* __restrict__ z, const int* gate,
                                                            double* part) {
    using T = typename TT::T;
    using Lane = typename TT::Lane;
    constexpr int VEC = TT::VEC;
    __shared__ T lds[kTileElems<TT>];
    if (!any_active(gate, kMaxS)) return;
    const int s0 = tile_chunk(t, TT::kSamples), sc = min(s0 + VEC * (int)(threadIdx.x & 15), t.S - VEC);
    double v[VEC] = {};
    Lane acc = {};
    tile_walk<TT, 1, 1, 2>(
        t, r, 0, r, {w}, lds, [&](const TileRow&) { acc = Lane{}; },
        [&](const Lane (&g)[1], const T (&ww)[1]) { acc += ww[0] * g[0]; },
        [&](const TileRow& row, const T* tile, bool on) {
            if (!on) return;
            const Lane ri = *(const Lane*)(tile + (row.more & 0xffff) * TT::kSamples + VEC * (int)(threadIdx.x & 15));
            *(Lane*)(z + (size_t)row.row * t.S + sc) = acc;
#pragma unroll
            for (int c = 0; c < VEC; ++c) v[c] += (double)lane_at<TT>(ri, c) * (double)lane_at<TT>(acc, c);
        });
    tile_partial<TT>(lds, part, t.S, v, s0);
}
constexpr int kUpPerCu = 2;
constexpr int kUpNodes = 192;

// y = M x (the V-cycle's restrictions and its way up below level 0; any sample count
// but 64 in FP32).  A row and 16 samples per wavefront, or per block of four
// (BLK, where there are too few rows to fill the chip): its 16-slot chunks are
// dealt to the 16-lane groups, lane j reads slot j's offset and weight and
// passes them on by DPP.  The rows are long (60 to 180 entries) and few, so this is
// bound by latency: with one wavefront per row and a lane per sample a row was
// a chain of 4 to 12 chunks, and at 24 samples 40 lanes were idle.  24 FP64
// samples at 38,025 nodes: 19.5 -> 11.2 us (1,520 rows from 38,025), 20.5 -> 5.5
// (96 from 1,520), 12.3 -> 8.5 (up).
template <typename T, bool BLK>
__global__ __launch_bounds__(kBlock) void k_b_spmm(SlotArgs M, int S, const T* __restrict__ x, T* __restrict__ y) {
    if (!any_active(M.gate, M.gate_n)) return;
    constexpr int kGroups = BLK ? kBlock / 16 : kWave / 16;
    const int j = threadIdx.x & 15, g = threadIdx.x / 16 % kGroups;
    const int row = __builtin_amdgcn_readfirstlane(
        BLK ? xcd_block() : xcd_block() * kRowsPerBlock + (int)(threadIdx.x / kWave));
    const int s = blockIdx.y * 16 + j;
    if (row >= M.n) return;  // (a whole block if BLK)
    const cint_p sp = (cint_p)M.sp;
    const int a0 = sp[row], a1 = sp[row + 1];
    const char* xs = (const char*)(x + min(s, S - 1));
    const T* w = (const T*)M.w;
    T acc = 0;
    for (int q = a0 + kSlot * g; q < a1; q += kSlot * kGroups) {
        const int off = M.off[q + j];
        const T ww = w[q + j];
        T v[kSlot];
        each16([&](auto kk) { v[decltype(kk)::value] = *(const T*)(xs + bcast16<decltype(kk)::value>(off)); },
               std::make_integer_sequence<int, kSlot>{});
        each16([&](auto kk) { acc += bcast16<decltype(kk)::value>(ww) * v[decltype(kk)::value]; },
               std::make_integer_sequence<int, kSlot>{});
    }
    acc += __shfl_xor(acc, 16);
    acc += __shfl_xor(acc, 32);
    if constexpr (BLK) {
        __shared__ T red[kRowsPerBlock][16];
        if ((threadIdx.x & (kWave - 1)) < 16) red[threadIdx.x / kWave][j] = acc;
        __syncthreads();
        if (threadIdx.x >= 16) return;
        acc = red[0][j];
#pragma unroll
        for (int k = 1; k < kRowsPerBlock; ++k) acc += red[k][j];
    } else if (g != 0) {
        return;
    }
    if (s < S) y[(size_t)row * S + s] = acc;
}

// y = M x for a dense M (row-major, m columns; the V-cycle's coarsest level),
// R rows and 16 VEC samples per block: the columns are dealt in chunks of 16 to
// the block's 32 groups of 16 lanes, lane j holds M's entries of column j and
// passes them on by DPP, so that a chunk costs its 16 rows of x and one load per
// row of M; the groups' sums are added across lanes and in LDS.  Bound by the
// texture unit (17 loads per chunk) where a block per CU covers the rows, so a
// second row per block is free beyond that (R = 2 for more than 256 blocks).
// With M = C^-1 R (I - A w D^-1) (the single-sample solver's, up to 2^20 entries) it
// takes the place of the last restriction and of the product with C^-1: 24 FP64
// samples at 38,025 nodes 1.49 -> 1.36 ms per evaluation, 7 samples at 2,205
// nodes 11.1 -> 5.5 us per V-cycle.  64 FP32 samples keep the two products: the
// FP64 sums over the restriction's columns cost more there (152 x 2,216: 15.3 us)
// than the restriction in FP32 and C^-1 (10.4).
constexpr int kDmvThreads = 512;
template <typename T, int VEC, int R>
__global__ __launch_bounds__(kDmvThreads) void k_b_dmv(int rows, int m, int S, const double* __restrict__ M,
                                                       const T* __restrict__ x, T* __restrict__ y, const int* gate) {
    if (!any_active(gate, S)) return;
    typedef T Vec __attribute__((ext_vector_type(VEC)));
    using Lane = std::conditional_t<VEC == 1, T, Vec>;
    constexpr int kWaves = kDmvThreads / kWave;
    __shared__ double red[kWaves][R][16 * VEC];
    const int j = threadIdx.x & 15, g = threadIdx.x / 16;
    const int r0 = blockIdx.x * R, s = (blockIdx.y * 16 + j) * VEC, sc = min(s, S - VEC);
    double acc[R][VEC];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[r][v] = 0.0;
    for (int k0 = g * 16; k0 < m; k0 += kDmvThreads) {
        double w[R];
        Lane xv[16];
#pragma unroll
        for (int r = 0; r < R; ++r) w[r] = M[(size_t)min(r0 + r, rows - 1) * m + min(k0 + j, m - 1)];
#pragma unroll
        for (int k = 0; k < 16; ++k) xv[k] = *(const Lane*)(x + (size_t)min(k0 + k, m - 1) * S + sc);
        if (k0 + j >= m)
#pragma unroll
            for (int r = 0; r < R; ++r) w[r] = 0.0;
        each16(
            [&](auto kk) {
                constexpr int K = decltype(kk)::value;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const double ww = bcast16<K>(w[r]);
                    if constexpr (VEC == 1) acc[r][0] += ww * (double)xv[K];
                    else
#pragma unroll
                        for (int v = 0; v < VEC; ++v) acc[r][v] += ww * (double)xv[K][v];
                }
            },
            std::make_integer_sequence<int, 16>{});
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
            double a = acc[r][v];
            a += __shfl_xor(a, 16);
            a += __shfl_xor(a, 32);
            if ((threadIdx.x & (kWave - 1)) < 16) red[threadIdx.x / kWave][r][j * VEC + v] = a;
        }
    __syncthreads();
    for (int e = threadIdx.x; e < R * 16 * VEC; e += kDmvThreads) {
        const int r = e / (16 * VEC), q = e % (16 * VEC), sq = (int)blockIdx.y * 16 * VEC + q;
        double a = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) a += red[w][r][q];
        if (r0 + r < rows && sq < S) y[(size_t)(r0 + r) * S + sq] = (T)a;
    }
}

// U[j][s] = u[bn[j]][s]  (S x b column-major, ld S)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_gather(int b, int S, const int* __restrict__ bn,
                                                     const double* __restrict__ u, T* __restrict__ U) {
    const size_t tot = (size_t)b * S;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock)
        U[e] = (T)u[bn ? (size_t)bn[e / S] * S + e % S : e];
}

// out[bn[j]][s] = G[j + s b]  (G = B U^T, b x S column-major); bn null: out[j][s]
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_scatter(int b, int S, const int* __restrict__ bn,
                                                      const T* __restrict__ G, double* __restrict__ out) {
    const size_t tot = (size_t)b * S;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock)
        out[(size_t)(bn ? bn[e % b] : e % b) * S + e / b] = (double)G[e];
}

// ---- FP64 MFMA GEMM for the boundary product ---------------------------
// P[ks] (b x S, row-major: P[ks][row][j]) = B[:, K_ks] (b x |K_ks|,
// column-major, ld) * U^T[K_ks, :] with U S x b column-major (ld S), S <= 16 NT
// columns.  Block: 4 wavefronts x 16 MT rows, all columns (those past S compute
// the last one and are not stored), one K range ks of the split; U^T chunks of KGK
// rows are staged in LDS.
// v_mfma_f64_16x16x4f64 operand layout (measured): A lane l = A[l%16][l/16],
// B lane l = B[l/16][l%16], D lane l register r = C[4r + l/16][l%16].
// Software-pipelined: while the MFMAs of chunk c run, its successor's U^T rows
// are in flight into registers, stored to the other of two LDS buffers
// afterwards (one barrier per chunk), and the B values of chunks c + 1 and c + 2
// into a rotation of three register sets.  No load depends on a condition: rows
// and columns past the last load the last one, U^T past the range's end is zero.
// Bound by the FP64 matrix cores under their power limit (54 TFLOP/s is what
// the library's best kernel sustains at 40,962 boundary nodes): 64 samples, 10,242
// boundary nodes 0.258 -> 0.245 ms, 9,602 0.226 -> 0.220 against masked loads one chunk ahead.
// Fewer samples take as many column tiles as they need and are bound by reading
// B: 24 samples, 10,242 boundary nodes 204 us (the library's fastest) -> 163 (5.1
// TB/s), 7 samples, 1,122 boundary nodes 21.7 -> 5.2 + 3 for the partials' sum.
typedef double dbl4 __attribute__((ext_vector_type(4)));

template <int KGK, int MT, int NT>
__global__ __launch_bounds__(kBlock) void k_b_gemm64(int b, int ld, int S, const double* __restrict__ B,
                                                     const double* __restrict__ U, int kper,
                                                     double* __restrict__ P) {
    constexpr int kCols = 16 * NT;
    constexpr int UPT = KGK * kCols / kBlock;  // U^T values per thread per chunk
    static_assert(KGK % 4 == 0 && UPT * kBlock == KGK * kCols, "chunk shape");
    __shared__ double us[2][KGK * kCols];  // U^T chunk: us[buf][k * kCols + j]
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int m0 = (blockIdx.x * (kBlock / kWave) + wv) * 16 * MT;  // this wavefront's rows
    const int ks = blockIdx.y;
    const int kb = ks * kper, ke = min(b, kb + kper);
    const int nc = ke > kb ? (ke - kb + KGK - 1) / KGK : 0;  // chunks, uniform over the block
    const int li = lane & 15, lk = lane >> 4;
    dbl4 acc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[t][u] = dbl4{0.0, 0.0, 0.0, 0.0};
    int rr[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) rr[t] = min(m0 + 16 * t + li, b - 1);  // the A row of this lane in tile t
    typedef double Vals[MT][KGK / 4];
    double ur[UPT];
    auto load_b = [&](int c, Vals& dst) {
        const int k0 = kb + c * KGK;
#pragma unroll
        for (int q = 0; q < KGK / 4; ++q) {
            const double* col = B + (size_t)min(k0 + 4 * q + lk, b - 1) * ld;  // this lane's K column
#pragma unroll
            for (int t = 0; t < MT; ++t) dst[t][q] = col[rr[t]];
        }
    };
    auto load_u = [&](int c) {
#pragma unroll
        for (int i = 0; i < UPT; ++i) {
            const int t = threadIdx.x + i * kBlock;
            ur[i] = U[(size_t)min(kb + c * KGK + t / kCols, b - 1) * S + min(t % kCols, S - 1)];
        }
    };
    auto store_u = [&](int c) {
#pragma unroll
        for (int i = 0; i < UPT; ++i) {
            const int t = threadIdx.x + i * kBlock;
            us[c & 1][t] = kb + c * KGK + t / kCols < ke ? ur[i] : 0.0;
        }
    };
    auto mfmas = [&](const Vals& av, int buf) {
#pragma unroll
        for (int q = 0; q < KGK / 4; ++q) {
#pragma unroll
            for (int u = 0; u < NT; ++u) {
                const double bu = us[buf][(4 * q + lk) * kCols + u * 16 + li];
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    acc[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[t][q], bu, acc[t][u], 0, 0, 0);
            }
        }
    };
    Vals a[3];
    load_u(0);
    load_b(0, a[0]);
    load_b(1, a[1]);
    store_u(0);
    __syncthreads();
    // chunk c from `now`, chunk c + 2 on its way into `next2`
    auto step = [&](int c, const Vals& now, Vals& next2) {
        load_u(c + 1);
        load_b(c + 2, next2);
        mfmas(now, c & 1);
        store_u(c + 1);  // that buffer was last read in chunk c - 1
        __syncthreads();
    };
    for (int c = 0; c < nc; c += 3) {  // chunks past the last add nothing
        step(c, a[0], a[2]);
        step(c + 1, a[1], a[0]);
        step(c + 2, a[2], a[1]);
    }
    double* out = P + (size_t)ks * b * S;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + t * 16 + 4 * r + lk, col = u * 16 + li;
                if (row < b && col < S) out[(size_t)row * S + col] = acc[t][u][r];
            }
}

struct GemmShape {
    int kgk, mt;
};
constexpr GemmShape kGemmShapes[] = {{16, 2}, {32, 2}, {16, 1}, {32, 1}, {8, 2}, {16, 4}, {8, 4}};
constexpr int kNumGemmShapes = sizeof(kGemmShapes) / sizeof(kGemmShapes[0]);
// the last three for four column tiles only
inline int gemm_shapes(int S) { return S > 48 ? kNumGemmShapes : 4; }

inline int gemm_rows_per_block(int shape) { return (kBlock / kWave) * 16 * kGemmShapes[shape].mt; }

template <class F>
void gemm_dispatch(int shape, int S, F&& f) {
    auto first4 = [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        switch (shape) {
            case 0: f(k_b_gemm64<16, 2, NT>); break;
            case 1: f(k_b_gemm64<32, 2, NT>); break;
            case 2: f(k_b_gemm64<16, 1, NT>); break;
            default: f(k_b_gemm64<32, 1, NT>); break;
        }
    };
    if (S <= 16) first4(std::integral_constant<int, 1>{});
    else if (S <= 32) first4(std::integral_constant<int, 2>{});
    else if (S <= 48) first4(std::integral_constant<int, 3>{});
    else if (shape < 4) first4(std::integral_constant<int, 4>{});
    else if (shape == 4) f(k_b_gemm64<8, 2, 4>);
    else if (shape == 5) f(k_b_gemm64<16, 4, 4>);
    else f(k_b_gemm64<8, 4, 4>);
}

void launch_gemm64(int shape, dim3 g, hipStream_t s, int b, int ld, int S, const double* B, const double* U, int kper,
                   double* P) {
    gemm_dispatch(shape, S, [&](auto k) { hipLaunchKernelGGL(k, g, dim3(kBlock), 0, s, b, ld, S, B, U, kper, P); });
}

// resident blocks per CU of a tile shape (0 if the runtime cannot say)
int gemm_blocks_per_cu(int shape, int S) {
    int nb = 0;
    gemm_dispatch(shape, S, [&](auto k) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k, kBlock, 0) != hipSuccess) nb = 0;
    });
    return nb;
}

// out[bn[j]][s] = sum_ks P[ks][j][s] (FP64 split-K partials of k_b_gemm64,
// row-major); without bn: out[j][s]
__global__ __launch_bounds__(kBlock) void k_b_ksum_scatter(int b, int S, int nks, const int* __restrict__ bn,
                                                           const double* __restrict__ P, double* __restrict__ out) {
    const size_t tot = (size_t)b * S;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock) {
        double acc = 0.0;
        for (int c = 0; c < nks; ++c) acc += P[(size_t)c * tot + e];
        out[bn ? (size_t)bn[e / S] * S + e % S : e] = acc;
    }
}

// out[bn[j]][s] = sum_c P[c][j + s b] in FP64 (the split-K FP32 partials);
// bn null: out[j][s]
__global__ __launch_bounds__(kBlock) void k_b_chunk_sum(int b, int S, int nch, const int* __restrict__ bn,
                                                        const float* __restrict__ P, double* __restrict__ out) {
    const size_t tot = (size_t)b * S;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock) {
        double acc = 0.0;
        for (int c = 0; c < nch; ++c) acc += (double)P[(size_t)c * tot + e];
        out[(size_t)(bn ? bn[e % b] : e % b) * S + e / b] = acc;
    }
}

// ---- boundary product from int8 digit slices (TM_PREC_MIXED_BEMI8) -------
// Every row j of B and every sample column s of U is scaled by a power of
// two (sigma_j >= max_k |B_jk|, tau_s >= max_k |U_ks|) and written as
// base-2^7 digits in [-64, 64], five for B and six for U:
//   B_jk = sigma_j sum_p d_p 2^-(6+7p),   U_ks = tau_s sum_q e_q 2^-(6+7q).
// Digit products accumulate exactly in int32 on the int8 matrix cores
// (v_mfma_i32_16x16x64_i8); the products with p + q <= 5 are kept and
// summed per p + q, so
//   (B U^T)_js = sigma_j tau_s 2^-12 sum_{d <= 5} 2^-7d acc_d(j, s),
//   acc_d = sum_{p+q=d} sum_k d_p(j, k) e_q(k, s).
// The error is then B's own rounding to five digits (~2^-35 of the row
// maximum per entry, a fixed perturbation of B, ~1e-8 relative on the
// product); U's rounding and the dropped products are ~2^-42, so the
// product varies as smoothly as U along a trajectory.  The splitting of a
// floating-point product into exact integer products follows Ozaki et al.
// (Numer. Algorithms 59 (2012) 95) and its integer-matrix-engine forms.
// |acc_d| <= 5 * 64 * 64 * K < 2^31 for K <= 104832 columns per K range.
typedef int i32x4 __attribute__((ext_vector_type(4)));
constexpr int kI8Digits = 5;            // digits of B
constexpr int kI8DigitsU = 6;           // digits of U
constexpr int kI8MaxD = 5;              // products with p + q <= kI8MaxD
constexpr int kI8Op = 64;               // i32x4 per MFMA operand (64 lanes x 16 bytes)
constexpr int kI8MaxK = 104832;         // columns per K range without int32 overflow
// Slice layouts (16-byte operands, lane l = row/column l % 16, k block l / 16):
//   Bq: [row tile T (16 rows)][k chunk c (64)][digit p][lane l] i32x4 =
//       d_p(B)[16T + l % 16][64c + 16(l / 16) + 0..15]
//   Uq: [k chunk c][digit q (6)][column tile u (16 samples)][lane l] i32x4 =
//       e_q(U)[64c + 16(l / 16) + 0..15][16u + l % 16]

// ND digits of r, |r| <= 1, each exact (power-of-two scalings and rint)
template <int ND>
__device__ inline void i8_digits(double r, int (&d)[ND]) {
#pragma unroll
    for (int p = 0; p < ND; ++p) {
        const double w = (double)(1LL << (6 + 7 * p));
        const double t = rint(r * w);
        d[p] = (int)t;
        r -= t / w;
    }
}

// the power of two 2^e >= m (m = mantissa 2^e, mantissa in [0.5, 1)); 1 for m = 0
__device__ inline double i8_scale(double m) {
    if (m == 0.0) return 1.0;
    if (!(m > 0.0) || !std::isfinite(m)) return m;  // NaN and inf pass through (non-finite products)
    int e;
    (void)frexp(m, &e);
    return ldexp(1.0, e);
}

// per-row maxima of |B| (B column-major, ld), K split over blockIdx.y
__global__ __launch_bounds__(kBlock) void k_b_i8_rowmax(int b, int ld, const double* __restrict__ B, int kper,
                                                        double* __restrict__ rmax) {
    const int j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= b) return;
    const int k0 = blockIdx.y * kper, k1 = min(b, k0 + kper);
    double m = 0.0;
    for (int k = k0; k < k1; ++k) m = fmax(m, fabs(B[(size_t)k * ld + j]));
    atomic_max_nonneg(rmax + j, m);
}

// Bq from B (once per batch): thread = (tile T, chunk c, lane l), 16 values
__global__ __launch_bounds__(kBlock) void k_b_i8_bslice(int b, int ld, const double* __restrict__ B, int nT, int nC,
                                                        const double* __restrict__ rmax, i32x4* __restrict__ Bq) {
    const size_t tot = (size_t)nT * nC * 64;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock) {
        const int l = (int)(e & 63);
        const size_t tc = e >> 6;
        const int c = (int)(tc % nC), T = (int)(tc / nC);
        const int row = 16 * T + (l & 15), kb = 64 * c + 16 * (l >> 4);
        const double inv = row < b ? 1.0 / i8_scale(rmax[row]) : 0.0;
        i32x4 w[kI8Digits];
#pragma unroll
        for (int p = 0; p < kI8Digits; ++p) w[p] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int k = kb + j;
            const double v = (row < b && k < b) ? B[(size_t)k * ld + row] * inv : 0.0;
            int d[kI8Digits];
            i8_digits(v, d);
#pragma unroll
            for (int p = 0; p < kI8Digits; ++p) w[p][j >> 2] |= (d[p] & 0xff) << (8 * (j & 3));
        }
#pragma unroll
        for (int p = 0; p < kI8Digits; ++p) Bq[(tc * kI8Digits + p) * kI8Op + l] = w[p];
    }
}

__global__ void k_b_i8_zero(int cnt, double* __restrict__ p) {
    if ((int)threadIdx.x < cnt) p[threadIdx.x] = 0.0;
}

// per-sample maxima of |u| over the boundary nodes (lane = sample)
__global__ __launch_bounds__(kBlock) void k_b_i8_umax(int b, int S, const int* __restrict__ bn,
                                                      const double* __restrict__ u, double* __restrict__ umax) {
    const int lane = threadIdx.x & 63;
    double m = 0.0;
    if (lane < S)
        for (int k = blockIdx.x * (kBlock / 64) + (int)(threadIdx.x >> 6); k < b; k += gridDim.x * (kBlock / 64)) {
            const double v = u[(size_t)(bn ? bn[k] : k) * S + lane];
            m = fmax(m, v == v ? fabs(v) : INFINITY);  // a NaN counts as inf: the product turns non-finite
        }
    __shared__ double sm[kBlock / 64][64];
    sm[threadIdx.x >> 6][lane] = m;
    __syncthreads();
    if (threadIdx.x < 64 && (int)threadIdx.x < S) {
        double t = sm[0][lane];
        for (int w = 1; w < kBlock / 64; ++w) t = fmax(t, sm[w][lane]);
        atomic_max_nonneg(umax + lane, t);
    }
}

// Uq from the boundary values: thread = (chunk c, column tile u, lane l)
__global__ __launch_bounds__(kBlock) void k_b_i8_uslice(int b, int S, int nC, const int* __restrict__ bn,
                                                        const double* __restrict__ u,
                                                        const double* __restrict__ umax, i32x4* __restrict__ Uq) {
    const size_t tot = (size_t)nC * 4 * 64;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock) {
        const int l = (int)(e & 63), ut = (int)((e >> 6) & 3), c = (int)(e >> 8);
        const int s = 16 * ut + (l & 15), kb = 64 * c + 16 * (l >> 4);
        const double inv = s < S ? 1.0 / i8_scale(umax[s]) : 0.0;
        i32x4 w[kI8DigitsU];
#pragma unroll
        for (int q = 0; q < kI8DigitsU; ++q) w[q] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int k = kb + j;
            const double v = (s < S && k < b) ? u[(size_t)(bn ? bn[k] : k) * S + s] * inv : 0.0;
            int d[kI8DigitsU];
            i8_digits(v, d);
#pragma unroll
            for (int q = 0; q < kI8DigitsU; ++q) w[q][j >> 2] |= (d[q] & 0xff) << (8 * (j & 3));
        }
#pragma unroll
        for (int q = 0; q < kI8DigitsU; ++q) Uq[(((size_t)c * kI8DigitsU + q) * 4 + ut) * kI8Op + l] = w[q];
    }
}

// P[ks][row][col] (row-major, 64 columns) = sum_d 2^-7d acc_d over the K
// chunks [ks cper, (ks+1) cper) of the slices.  Block: NW wavefronts of 16 rows
// each; the chunk's U digits (24 KB) are staged in LDS and shared by the
// wavefronts, double-buffered: while the MFMAs of chunk c run, U's digits of
// chunk c + 1 are in flight into registers, stored to the other buffer
// afterwards, and B's digits of chunks c + 1 and c + 2 into a rotation of three
// register sets: 8 wavefronts then keep 80 KB per CU in flight, with one chunk
// ahead (40 KB) every wavefront waited for memory.  40,962 boundary nodes and 64
// samples 1,700 -> 1,440 us (up to 1,530 from box to box): B's 8.4 GB of digits at
// 5.8 TB/s, and 4.3 T operations (the 131 M MFMAs) at 2.98 POPS.  Near both limits:
// 6.5 TB/s is the best streaming read here; the operations alone take 0.86 ms at
// the nominal 5 POPS, while the instruction by itself settles at 2.86 POPS when it
// runs for long (a launch of 1.4 ms can exceed that).
// v_mfma_i32_16x16x64_i8: A lane l = row l % 16, B lane l = column l % 16,
// both the 16 k of block l / 16; D lane l register r = C[4 (l / 16) + r][l % 16].
template <int NW>
__global__ __launch_bounds__(64 * NW, 2) void k_b_gemm_i8(int b, int nT, int nC, int cper,
                                                          const i32x4* __restrict__ Bq,
                                                          const i32x4* __restrict__ Uq, double* __restrict__ P) {
    constexpr int UPT = kI8DigitsU * 4 * kI8Op / (64 * NW);  // U operands per thread per chunk
    __shared__ i32x4 us[2][kI8DigitsU * 4 * kI8Op];
    const int lane = threadIdx.x & 63;
    const int T = blockIdx.x * NW + (int)(threadIdx.x >> 6);
    const int cb = blockIdx.y * cper, ce = min(nC, cb + cper);  // (empty: cb >= nC)
    i32x4 acc[kI8MaxD + 1][4];
#pragma unroll
    for (int d = 0; d <= kI8MaxD; ++d)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[d][u] = i32x4{0, 0, 0, 0};
    // tiles and chunks past the last load the last one (the tile is not stored,
    // the chunk is multiplied with zero): no load depends on a condition
    const i32x4* src = Bq + (size_t)min(T, nT - 1) * nC * (kI8Digits * kI8Op) + lane;
    i32x4 ur[UPT];
    typedef i32x4 Ops[kI8Digits];
    auto load_a = [&](int c, Ops& dst) {
        const i32x4* s = src + (size_t)min(c, nC - 1) * (kI8Digits * kI8Op);
#pragma unroll
        for (int p = 0; p < kI8Digits; ++p) dst[p] = __builtin_nontemporal_load(s + p * kI8Op);
    };
    auto load_u = [&](int c) {
        const i32x4* s = Uq + (size_t)min(c, nC - 1) * (kI8DigitsU * 4 * kI8Op) + threadIdx.x;
#pragma unroll
        for (int i = 0; i < UPT; ++i) ur[i] = s[i * 64 * NW];
    };
    auto store_u = [&](int c) {
#pragma unroll
        for (int i = 0; i < UPT; ++i)
            us[(c - cb) & 1][threadIdx.x + i * 64 * NW] = c < ce ? ur[i] : i32x4{0, 0, 0, 0};
    };
    // U's operand of step (u, q) is read two steps ahead; the scheduling barriers keep
    // the compiler from reading all 24 at once, which spills
    auto mfmas = [&](const Ops& av, int buf) {
        const i32x4* ul = us[buf] + lane;
        auto at = [&](int i) { return ul[((i % kI8DigitsU) * 4 + i / kI8DigitsU) * kI8Op]; };
        constexpr int kSteps = 4 * kI8DigitsU;
        i32x4 bq[3];
        bq[0] = at(0);
        bq[1] = at(1);
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            if (i + 2 < kSteps) bq[(i + 2) % 3] = at(i + 2);
            const int u = i / kI8DigitsU, q = i % kI8DigitsU;
#pragma unroll
            for (int p = 0; p < kI8Digits && p + q <= kI8MaxD; ++p)
                acc[p + q][u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[p], bq[i % 3], acc[p + q][u], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    Ops a[3];
    load_u(cb);
    load_a(cb, a[0]);
    load_a(cb + 1, a[1]);
    store_u(cb);
    __syncthreads();
    // chunk c from `now`, chunk c + 2 on its way into `next2`
    auto step = [&](int c, const Ops& now, Ops& next2) {
        load_u(c + 1);
        load_a(c + 2, next2);
        mfmas(now, (c - cb) & 1);
        store_u(c + 1);  // that buffer was last read in chunk c - 1
        __syncthreads();
    };
    for (int c = cb; c < ce; c += 3) {  // chunks past ce add nothing (zero digits of U)
        step(c, a[0], a[2]);
        step(c + 1, a[1], a[0]);
        step(c + 2, a[2], a[1]);
    }
    if (T >= nT) return;
    double* out = P + (size_t)blockIdx.y * b * 64;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = T * 16 + 4 * (lane >> 4) + r;
            double v = 0.0;
#pragma unroll
            for (int d = kI8MaxD; d >= 0; --d) v = v * (1.0 / 128.0) + (double)acc[d][u][r];
            if (row < b) out[(size_t)row * 64 + u * 16 + (lane & 15)] = v;
        }
}

// out[bn[j]][s] = sigma_j tau_s 2^-12 sum_ks P[ks][j][s] (s < S); without bn: out[j][s]
__global__ __launch_bounds__(kBlock) void k_b_i8_finish(int b, int S, int nks, const int* __restrict__ bn,
                                                        const double* __restrict__ P, const double* __restrict__ rmax,
                                                        const double* __restrict__ umax, double* __restrict__ out) {
    const size_t tot = (size_t)b * 64;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock) {
        const int j = (int)(e >> 6), s = (int)(e & 63);
        if (s >= S) continue;
        double acc = 0.0;
        for (int c = 0; c < nks; ++c) acc += P[(size_t)c * tot + e];
        out[(size_t)(bn ? bn[j] : j) * S + s] = acc * i8_scale(rmax[j]) * i8_scale(umax[s]) * (1.0 / 4096.0);
    }
}

void launch_gemm_i8(int nw, dim3 g, hipStream_t s, int b, int nT, int nC, int cper, const i32x4* Bq,
                    const i32x4* Uq, double* P) {
    if (nw == 8)
        hipLaunchKernelGGL(k_b_gemm_i8<8>, g, dim3(512), 0, s, b, nT, nC, cper, Bq, Uq, P);
    else
        hipLaunchKernelGGL(k_b_gemm_i8<4>, g, dim3(256), 0, s, b, nT, nC, cper, Bq, Uq, P);
}

__global__ __launch_bounds__(kBlock) void k_b_to_float(size_t tot, const double* __restrict__ a,
                                                       float* __restrict__ o) {
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock)
        o[e] = (float)a[e];
}

// m <- normalize(m + dt dm) per (node, sample)
__global__ __launch_bounds__(kBlock) void k_b_euler(size_t NS, double* __restrict__ m, const double* __restrict__ dm,
                                                    double dt) {
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < NS; e += (size_t)gridDim.x * kBlock) {
        const double x = m[e] + dt * dm[e], y = m[NS + e] + dt * dm[NS + e], z = m[2 * NS + e] + dt * dm[2 * NS + e];
        const double l = sqrt(x * x + y * y + z * z);
        const double f = l > 0.0 ? 1.0 / l : 1.0;
        m[e] = x * f;
        m[NS + e] = y * f;
        m[2 * NS + e] = z * f;
    }
}

__global__ void k_b_zero_small(int cnt, double* p) {
    if ((int)threadIdx.x < cnt) p[threadIdx.x] = 0.0;
}

// *fail, *bad += the samples whose outer residual missed the tolerance, and those that are not finite
__global__ void k_b_count_undone(int S, const OState* os, unsigned* fail, unsigned* bad) {
    const int s = threadIdx.x;
    if (s < S && os->done[s] != 1) atomicAdd(os->done[s] == 0 ? fail : bad, 1u);
}

// every sample active with finite CG scalars (kernel timing only)
__global__ void k_b_activate(int S, BState* bs) {
    const int s = threadIdx.x;
    if (s < S) {
        bs->active[s] = 1;
        bs->gam[s] = 1.0;
        bs->alpha[s] = 0.0;
        bs->beta[s] = 0.0;
    }
}

__global__ void k_b_reset_fail(int cnt, unsigned* fail) {
    if ((int)threadIdx.x < cnt && blockIdx.x == 0) fail[threadIdx.x] = 0u;
}

__global__ __launch_bounds__(kBlock) void k_b_copy(size_t tot, const double* __restrict__ a, double* __restrict__ b) {
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock) b[e] = a[e];
}

// RK4 helpers over [3][n][S]: out = base + c k;  m = normalise(base + dt/6 (k1 + 2k2 + 2k3 + k4))
__global__ __launch_bounds__(kBlock) void k_b_axpy(size_t tot, const double* __restrict__ base,
                                                   const double* __restrict__ k, double c, double* __restrict__ out) {
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock)
        out[e] = base[e] + c * k[e];
}

__global__ __launch_bounds__(kBlock) void k_b_rk_final(size_t NS, const double* __restrict__ base,
                                                       const double* __restrict__ k1, const double* __restrict__ k2,
                                                       const double* __restrict__ k3, const double* __restrict__ k4,
                                                       double dt, double* __restrict__ m) {
    const double f = dt / 6.0;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < NS; e += (size_t)gridDim.x * kBlock) {
        double v[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const size_t q = (size_t)d * NS + e;
            v[d] = base[q] + f * (k1[q] + 2.0 * k2[q] + 2.0 * k3[q] + k4[q]);
        }
        const double l = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        const double g = l > 0.0 ? 1.0 / l : 1.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) m[(size_t)d * NS + e] = v[d] * g;
    }
}

inline int elem_grid(size_t tot) { return (int)std::min<size_t>(4096, (tot + kBlock - 1) / kBlock); }
// a multiple of the XCD count (see B_ROW_LOOP)
inline int row_grid(int rows) {
    return xcd_grid(std::min(2048, (rows + kRowsPerBlock - 1) / kRowsPerBlock));
}

}  // namespace

// ---------------------------------------------------------------------------
// Batched solver for one demag system, sharing the context solver's operator
// and AMG hierarchy.
// Host copy of a device CSR matrix (slot layouts are built on the host).
struct HostCsr {
    int n = 0;
    std::vector<int> rp, ci;
    std::vector<double> v;
};

int fetch_csr(const AmgPrecond::CsrDev& M, HostCsr& h, hipStream_t s) {
    h.n = M.n;
    h.rp.assign((size_t)M.n + 1, 0);
    TM_HIP(hipMemcpyAsync(h.rp.data(), M.rp.p, h.rp.size() * sizeof(int), hipMemcpyDeviceToHost, s));
    TM_HIP(hipStreamSynchronize(s));
    const size_t nnz = (size_t)h.rp[M.n];
    h.ci.assign(nnz, 0);
    h.v.assign(nnz, 0.0);
    if (nnz) {
        TM_HIP(hipMemcpyAsync(h.ci.data(), M.ci.p, nnz * sizeof(int), hipMemcpyDeviceToHost, s));
        TM_HIP(hipMemcpyAsync(h.v.data(), M.v.p, nnz * sizeof(double), hipMemcpyDeviceToHost, s));
        TM_HIP(hipStreamSynchronize(s));
    }
    return TM_OK;
}

// A CSR pattern in row slots (see SlotArgs): every row gets a multiple of
// kSlot slots, at least one chunk, padded with offset 0 / weight 0; byte
// offsets for gathered elements of 4 and of 8 bytes.
struct SlotOp {
    int n = 0, ncols = 0, S = 0;
    std::vector<int> h_rp, h_ci, h_sp;
    DevBuf<int> sp, off4, off8;

    int build(int rows, int cols, const int* rp, const int* ci, int S_, hipStream_t s) {
        n = rows;
        ncols = cols;
        S = S_;
        if ((int64_t)cols * S * 8 > (int64_t)INT32_MAX) return TM_ERR_UNSUPPORTED;  // 32-bit byte offsets
        h_rp.assign(rp, rp + rows + 1);
        h_ci.assign(ci, ci + rp[rows]);
        h_sp.assign((size_t)rows + 1, 0);
        for (int i = 0; i < rows; ++i) {
            const int len = rp[i + 1] - rp[i];
            h_sp[i + 1] = h_sp[i] + std::max(1, (len + kSlot - 1) / kSlot) * kSlot;
        }
        const size_t ns = (size_t)h_sp[rows];
        std::vector<int> o4(ns, 0), o8(ns, 0);
        for (int i = 0; i < rows; ++i) {
            size_t k = (size_t)h_sp[i];
            for (int q = rp[i]; q < rp[i + 1]; ++q, ++k) {
                o4[k] = ci[q] * S * 4;
                o8[k] = ci[q] * S * 8;
            }
        }
        TM_CHECK(sp.upload(h_sp.data(), h_sp.size(), s));
        TM_CHECK(off4.upload(o4.data(), ns, s));
        TM_CHECK(off8.upload(o8.data(), ns, s));
        TM_HIP(hipStreamSynchronize(s));
        return TM_OK;
    }

    // per-slot weights from CSR values v (optionally scaled by colscale[col] * w0)
    template <typename W>
    int values(const std::vector<double>& v, DevBuf<W>& out, hipStream_t s, const double* colscale = nullptr,
               double w0 = 1.0) const {
        std::vector<W> h((size_t)h_sp[n], (W)0);
        for (int i = 0; i < n; ++i) {
            size_t k = (size_t)h_sp[i];
            for (int q = h_rp[i]; q < h_rp[i + 1]; ++q)
                h[k++] = (W)(colscale ? v[q] * w0 * colscale[h_ci[q]] : v[q]);
        }
        TM_CHECK(out.upload(h.data(), h.size(), s));
        TM_HIP(hipStreamSynchronize(s));
        return TM_OK;
    }

    // long rows: more than 6 chunks of 16 on average (one block per row pays off there)
    bool long_rows() const { return n > 0 && (int64_t)h_sp[n] > (int64_t)kSlot * n * 6; }
    SlotArgs args(int ebytes, const void* w) const {
        return SlotArgs{n, ncols * S * ebytes, sp.p, ebytes == 4 ? off4.p : off8.p, w};
    }
};

// Tiles of a SlotOp's rows (see TileArgs): a tile starts at the first row that
// no tile has and takes, as long as they fit, the row that adds the fewest nodes
// among the rows that are nodes of the tile already, and the next row of the
// numbering when none of those fits: 31.7 of 32 rows per tile on the 282,897-node
// cuboid (28 without the next row, and the kernels 5 to 30 per cent slower), 4
// nodes per row where 32 consecutive rows of its Z-order numbering need 5.
// None (nt = 0) when a row alone refers to too many nodes, or below 1,024 units of
// 32 rows and 16 samples: two for each of the 512 blocks of the fields and the
// divergence, 1.3 for the 768 of the residual and of the products with 16 samples
// per unit.  The FP32 products for 64 samples take one unit per tile, 256 for 512
// blocks at the line, half of which then return at once.  An evaluation in us, from L2 / with tiles:
//   64 samples, mixed  364 units 395 / 403, 608 495 / 470, 848 595 / 545, 1,052 660 / 601
//   64 samples, FP64   364 units 429 / 417, 608 498 / 462, 848 589 / 534, 1,052 657 / 583
//   24 samples, FP64   360 units 455 / 402, 640 597 / 477, 856 698 / 549, 1,052 801 / 605
//   7 samples, mixed   383 units 525 / 429, 633 686 / 505, 878 866 / 604, 1,016 950 / 631
// So the line is on the safe side: tiles are the faster form from about 400 units on.
struct TileOp {
    int nt = 0;
    DevBuf<int> row0, node0, nodes;
    DevBuf<TileRow> rows;
    DevBuf<unsigned short> loc;

    int build(const SlotOp& op, hipStream_t s, int max_nodes = kTileNodes) {
        nt = 0;
        const int n = op.n, nc = op.ncols, nch = (op.S + kTileS - 1) / kTileS;
        if (n > nc || (int64_t)n * nch < (int64_t)1024 * kTileRows) return TM_OK;
        std::vector<int> hr{0}, hn{0}, hnode, order, place((size_t)nc, -1), deg((size_t)n, 0), have((size_t)n, 0), cand;
        std::vector<char> taken((size_t)n, 0);
        for (int i = 0; i < n; ++i) {  // a row's nodes: its columns and itself
            bool self = false;
            for (int q = op.h_rp[i]; q < op.h_rp[i + 1]; ++q) self = self || op.h_ci[q] == i;
            deg[i] = op.h_rp[i + 1] - op.h_rp[i] + (self ? 0 : 1);
            if (deg[i] > max_nodes) return TM_OK;
        }
        // rows by column: the rows that refer to a node
        std::vector<int> tp((size_t)nc + 1, 0), tr(op.h_ci.size());
        for (int c : op.h_ci) ++tp[c + 1];
        for (int i = 0; i < nc; ++i) tp[i + 1] += tp[i];
        {
            std::vector<int> fill(tp.begin(), tp.end() - 1);
            for (int i = 0; i < n; ++i)
                for (int q = op.h_rp[i]; q < op.h_rp[i + 1]; ++q) tr[fill[op.h_ci[q]]++] = i;
        }
        std::vector<unsigned short> hl((size_t)op.h_sp[n], 0);
        std::vector<TileRow> hrow((size_t)n);
        int first = 0;
        while ((int)order.size() < n) {
            while (taken[first]) ++first;
            const size_t base = hnode.size(), rbase = order.size();
            cand.clear();
            auto add_node = [&](int c) {  // counts for the rows that refer to it (have: nodes of theirs in the tile)
                if (place[c] >= 0) return;
                place[c] = (int)(hnode.size() - base);
                hnode.push_back(c);
                bool self = c >= n;
                for (int q = tp[c]; q < tp[c + 1]; ++q) {
                    ++have[tr[q]];
                    self = self || tr[q] == c;
                }
                if (!self) ++have[c];
                if (c < n && !taken[c]) cand.push_back(c);
            };
            for (int row = first; row >= 0;) {
                taken[row] = 1;
                order.push_back(row);
                add_node(row);
                for (int q = op.h_rp[row]; q < op.h_rp[row + 1]; ++q) add_node(op.h_ci[q]);
                row = -1;
                if ((int)(order.size() - rbase) == kTileRows) break;
                const int room = max_nodes - (int)(hnode.size() - base);
                int best = 0;
                size_t kept = 0;
                for (size_t k = 0; k < cand.size(); ++k) {
                    const int c = cand[k];
                    if (taken[c]) continue;
                    cand[kept++] = c;
                    const int more = deg[c] - have[c];
                    if (more <= room && (row < 0 || more < best || (more == best && c < row))) {
                        row = c;
                        best = more;
                    }
                }
                cand.resize(kept);
                if (row >= 0) continue;
                while (first < n && taken[first]) ++first;
                if (first < n && deg[first] <= room) row = first;  // no neighbour fits: the next row
            }
            for (size_t k = rbase; k < order.size(); ++k) {
                const int i = order[k];
                hrow[k] = TileRow{i, op.h_sp[i], (op.h_sp[i + 1] - op.h_sp[i]) / kSlot << 16 | place[i]};
                size_t e = (size_t)op.h_sp[i];
                for (int q = op.h_rp[i]; q < op.h_rp[i + 1]; ++q)
                    hl[e++] = (unsigned short)place[op.h_ci[q]];
                for (; e < (size_t)op.h_sp[i + 1]; ++e) hl[e] = (unsigned short)place[i];
            }
            for (size_t k = base; k < hnode.size(); ++k) {  // clean up for the next tile
                const int c = hnode[k];
                place[c] = -1;
                if (c < n) have[c] = 0;
                for (int q = tp[c]; q < tp[c + 1]; ++q) have[tr[q]] = 0;
            }
            hr.push_back((int)order.size());
            hn.push_back((int)hnode.size());
        }
        TM_CHECK(row0.upload(hr.data(), hr.size(), s));
        TM_CHECK(node0.upload(hn.data(), hn.size(), s));
        TM_CHECK(nodes.upload(hnode.data(), hnode.size(), s));
        TM_CHECK(rows.upload(hrow.data(), hrow.size(), s));
        TM_CHECK(loc.upload(hl.data(), hl.size(), s));
        TM_HIP(hipStreamSynchronize(s));
        nt = (int)hr.size() - 1;
        return TM_OK;
    }
    TileArgs args(const SlotOp& op, int samples = kTileS) const {
        return TileArgs{nt, op.S, (op.S + samples - 1) / samples, row0.p, rows.p, node0.p, nodes.p, loc.p};
    }
};

// The V-cycle's way up on one level, [2 w D^-1 - w D^-1 A w D^-1 | Q] on [b | x_c],
// from A (n rows) and down = R (I - A w D^-1), the transpose of Q = (I - w D^-1 A) P.
// Fixed rows of A (identity, no part of the hierarchy) have columns of the
// whole matrix; b is zero there.
void up_operator(int n, const int* arp, const int* aci, const std::vector<double>& av, const double* dinv, double w,
                 const HostCsr& down, HostCsr& U) {
    const int nc = (int)down.rp.size() - 1;
    std::vector<int> qp((size_t)n + 1, 0);
    for (int c : down.ci) ++qp[c + 1];
    U.n = n;
    U.rp.assign((size_t)n + 1, 0);
    for (int i = 0; i < n; ++i) U.rp[i + 1] = U.rp[i] + (arp[i + 1] - arp[i]) + qp[i + 1];
    U.ci.resize((size_t)U.rp[n]);
    U.v.resize((size_t)U.rp[n]);
    std::vector<int> fill((size_t)n);
    for (int i = 0; i < n; ++i) {
        int k = U.rp[i];
        for (int q = arp[i]; q < arp[i + 1]; ++q, ++k) {
            const int j = aci[q];
            U.ci[k] = j;
            U.v[k] = (j == i ? 2.0 * w * dinv[i] : 0.0) - w * dinv[i] * av[q] * w * dinv[j];
        }
        fill[i] = k;
    }
    for (int c = 0; c < nc; ++c)
        for (int q = down.rp[c]; q < down.rp[c + 1]; ++q) {
            const int k = fill[down.ci[q]]++;
            U.ci[k] = n + c;
            U.v[k] = down.v[q];
        }
}

// ---- initial guesses from earlier solves (successive right-hand sides) ----
// Per sample as the single-sample solver: x0 = x_0 + sum_j c_j dX_j over the
// kept pairs, dB_j / dX_j backward differences at the newest pair and c the
// least-squares fit of b - b_0 (the method is described with kSolveWindow in
// tm_internal.hpp).  Window state and the small Gram systems live on the
// device (the kernels are capturable).
struct WinState {
    int head;                            // slot the next pair goes to
    int cnt;                             // pairs held (<= kSolveWindow)
    double a[kSolveWindow][kMaxS];       // x0 = sum_i a_i x_slot(i) per sample (newest first)
};

// per-block partials part[block][q][s] of the kWinDots dots, lane = sample.  The new b goes
// into the head slot as it is read: when the window is full that slot holds
// the oldest pair, whose value this thread has already loaded.
// The k-th row read is rows[k * st] (or k * st without a list), k < nr: with
// a list, every row outside it is zero in b and in the kept b (a Dirichlet
// right-hand side off the boundary); with st > 1 the dots are those of an
// evenly spread subset of the rows (a sampled least-squares fit; the kept b
// are only ever read, and written, on that subset).
__global__ __launch_bounds__(kBlock) void k_b_win_dots(int n, int S, const WinState* ws, double* __restrict__ Bw,
                                                       const double* __restrict__ b, double* part, int nr,
                                                       const int* __restrict__ rows, int st) {
    const int cnt = ws->cnt, head = ws->head;
    const size_t NS = (size_t)n * S;
    double acc[kWinDots] = {};
    const double* src[kSolveWindow];
#pragma unroll
    for (int i = 0; i < kSolveWindow; ++i) src[i] = Bw + (size_t)win_slot(head, i) * NS;
    double* dst = Bw + (size_t)head * NS;
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < S;
    const int rstride = gridDim.x * kRowsPerBlock;
    // two rows per iteration: both rows' loads in flight together
    for (int k = __builtin_amdgcn_readfirstlane(blockIdx.x * kRowsPerBlock + (int)(threadIdx.x / kWave)); k < nr;
         k += 2 * rstride) {
        const bool two = k + rstride < nr;  // wavefront-uniform
        const int k2 = two ? k + rstride : k;
        const int row = rows ? rows[k * st] : k * st, row2 = rows ? rows[k2 * st] : k2 * st;
        if (on) {
            const size_t e1 = (size_t)row * S + lane, e2 = (size_t)row2 * S + lane;
            double v1[kSolveWindow], v2[kSolveWindow];
#pragma unroll
            for (int i = 0; i < kSolveWindow; ++i) {
                v1[i] = i < cnt ? src[i][e1] : 0.0;
                v2[i] = i < cnt ? src[i][e2] : 0.0;
            }
            const double b1 = b[e1], b2 = b[e2];
            const double r1 = b1 - v1[0], r2 = b2 - v2[0];
            win_differences(v1, cnt);
            win_accumulate(acc, v1, r1);
            if (two) {
                win_differences(v2, cnt);
                win_accumulate(acc, v2, r2);
            }
            dst[e1] = b1;  // after every load of the element (the head slot may be the oldest pair's)
            if (two) dst[e2] = b2;
        }
    }
    // the block's per-sample sums of all kWinDots dots, eight at a time
    __shared__ double sp[8][kRowsPerBlock][kWave];
    const int wv = threadIdx.x / kWave;
#pragma unroll
    for (int q0 = 0; q0 < kWinDots; q0 += 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (q0 + j < kWinDots) sp[j][wv][lane] = acc[q0 + j];
        __syncthreads();
        for (int i = threadIdx.x; i < 8 * kWave; i += kBlock) {
            const int j = i / kWave, sm = i % kWave;
            if (q0 + j < kWinDots && sm < S) {
                double t = 0.0;
#pragma unroll
                for (int k = 0; k < kRowsPerBlock; ++k) t += sp[j][k][sm];
                part[((size_t)blockIdx.x * kWinDots + q0 + j) * S + sm] = t;  // block-major: contiguous per block
            }
        }
        __syncthreads();
    }
}

// second stage of the dots: block (q, c) sums dot q over chunk c of the
// block partials, lane = sample (rows of part are contiguous in s);
// red[c][q][s]
constexpr int kWinChunks = 8;
__global__ __launch_bounds__(kBlock) void k_b_win_red(int G, int S, const double* __restrict__ part,
                                                      double* __restrict__ red) {
    constexpr int kW = kBlock / kWave;
    const int q = blockIdx.x, c = blockIdx.y;
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int sm = min(lane, S - 1);
    double v = 0.0;
    for (int g = c * kW + wv; g < G; g += kWinChunks * kW) v += part[((size_t)g * kWinDots + q) * S + sm];
    __shared__ double sr[kW][kWave];
    sr[wv][lane] = v;
    __syncthreads();
    if (wv == 0 && lane < S) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < kW; ++k) t += sr[k][lane];
        red[((size_t)c * kWinDots + q) * S + lane] = t;
    }
}

// the coefficients of sample s = blockIdx.x from the chunk sums (one wavefront)
__global__ __launch_bounds__(kWave) void k_b_win_solve(int S, WinState* ws, const double* red) {
    const int s = blockIdx.x;
    __shared__ double sd[kWinDots];
    const int q = threadIdx.x;
    if (q < kWinDots && s < S) {
        double v = 0.0;
#pragma unroll
        for (int c = 0; c < kWinChunks; ++c) v += red[((size_t)c * kWinDots + q) * S + s];
        sd[q] = v;
    }
    __syncthreads();
    const int cnt = ws->cnt;
    if (threadIdx.x != 0 || s >= S || cnt == 0) return;
    double t[kWinDots];
#pragma unroll
    for (int k = 0; k < kWinDots; ++k) t[k] = sd[k];
    double a[kSolveWindow];
    win_coefficients(cnt, t, a);
    for (int i = 0; i < kSolveWindow; ++i) ws->a[i][s] = a[i];
}

// x0 = sum_i a_i x_slot(i) (the caller's x when the window is empty), lane = sample,
// and the fixed rows' values x = b.  A start that is not finite is zero: an
// earlier right-hand side of that sample was not, and its solution is kept.
__global__ __launch_bounds__(kBlock) void k_b_win_combine(int n, int S, const WinState* ws,
                                                          const double* __restrict__ Xw,
                                                          const unsigned char* __restrict__ fixed,
                                                          const double* __restrict__ b, double* __restrict__ x) {
    const int cnt = ws->cnt;
    const size_t NS = (size_t)n * S;
    double a[kSolveWindow];
    const double* src[kSolveWindow];
    const int ln = min((int)(threadIdx.x & (kWave - 1)), S - 1);
#pragma unroll
    for (int i = 0; i < kSolveWindow; ++i) {
        a[i] = i < cnt ? ws->a[i][ln] : 0.0;
        src[i] = Xw + (size_t)win_slot(ws->head, i) * NS;
    }
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < S;
    const int rstride = gridDim.x * kRowsPerBlock;
    for (int row = __builtin_amdgcn_readfirstlane(blockIdx.x * kRowsPerBlock + (int)(threadIdx.x / kWave)); row < n;
         row += 2 * rstride) {
        const bool two = row + rstride < n;  // wavefront-uniform
        if (on) {
            const int row2 = two ? row + rstride : row;
            const size_t e1 = (size_t)row * S + lane, e2 = (size_t)row2 * S + lane;
            double acc1 = 0.0, acc2 = 0.0;
#pragma unroll
            for (int i = 0; i < kSolveWindow; ++i)
                if (i < cnt) {
                    acc1 += a[i] * src[i][e1];
                    acc2 += a[i] * src[i][e2];
                }
            if (cnt == 0) {
                acc1 = x[e1];
                acc2 = x[e2];
            }
            x[e1] = fixed[row] ? b[e1] : std::isfinite(acc1) ? acc1 : 0.0;
            if (two) x[e2] = fixed[row2] ? b[e2] : std::isfinite(acc2) ? acc2 : 0.0;
        }
    }
}

// the solution into the head slot (its b is there already)
__global__ __launch_bounds__(kBlock) void k_b_win_store(size_t NS, const WinState* ws, const double* __restrict__ x,
                                                        double* __restrict__ Xw) {
    const size_t off = (size_t)ws->head * NS;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < NS; e += (size_t)gridDim.x * kBlock)
        Xw[off + e] = x[e];
}

// keep the pair and advance the head; a failed solve (done = 0 for some
// sample) empties the window instead
__global__ void k_b_win_advance(int S, WinState* ws, const OState* os) {
    const int s = threadIdx.x;
    __shared__ int bad;
    if (s == 0) bad = 0;
    __syncthreads();
    if (s < S && !os->done[s]) atomicOr(&bad, 1);
    __syncthreads();
    if (s != 0) return;
    if (bad) {
        ws->cnt = 0;
        ws->head = 0;
        return;
    }
    ws->head = (ws->head + 1) % kSolveWindow;
    ws->cnt = min(ws->cnt + 1, kSolveWindow);
}

template <typename T>
struct BatchSolver {
    int n = 0, S = 0, G = 0;
    SlotOp sl0;                   // level-0 operator in slots
    DevBuf<T> wA0;                // its weights
    DevBuf<double> wA64;          // A in FP64 (outer residual)
    TileOp t0;                    // tiles of sl0 for the outer residual
    int Gr = 0;                   // partials per sample of the outer residual
    int Gq = 0, Gz = 0;           // of (z, q) and of (r, z)
    int gmax() const { return std::max(std::max(G, Gr), std::max(Gq, Gz)); }
    // the level-0 products of the inner solve from tiles
    bool tiled() const { return t0.nt > 0 && tu.nt > 0; }
    // f(tile type) for this batch: a float4 per lane for 64 FP32 samples
    template <int NODES, class F>
    void with_tile_type(F&& f) const {
        if constexpr (sizeof(T) == 4) {
            if (S == kMaxS) return f(TileType<T, 4, true, NODES>{});
        }
        if (S % (16 / (int)sizeof(T)) == 0) f(TileType<T, 1, true, NODES>{});
        else f(TileType<T, 1, false, NODES>{});
    }
    TileOp tu;                    // tiles of level 0's way up
    struct LvOps {
        SlotOp RA;                // R (I - A w D^-1): pre-smoothing from zero + restriction
        DevBuf<T> wRA;
        SlotOp U;                 // on [b | x_c]: prolongation + post-smoothing
        DevBuf<T> wU;
    };
    std::vector<LvOps> lo;
    // the coarsest level: its C^-1 (nc x nc), or that folded into the last
    // restriction (nc x dense_m, see k_b_dmv for the line); a copy, since a captured step holds its
    // address and the context's solvers may be set anew while this batch lives
    DevBuf<double> dense;
    int nc = 0, dense_m = 0;
    bool folded = false;
    DevBuf<unsigned char> fixed;
    DevBuf<T> rT, q;              // rT: [r | x_c]
    static constexpr int kRing = 40;  // iterations per inner solve (a longer one is cut there; the outer loop goes on)
    DevBuf<T> ring;                   // (kRing + 1) x [n][S]: the preconditioned residuals z_k
    DevBuf<double> ahist, bhist;      // (kRing + 1) x kMaxS: alpha_k, beta_k
    DevBuf<double> chist;             // kRing x kMaxS: the combination coefficients c_i
    std::vector<DevBuf<T>> bx;    // levels >= 1: [b | x_c]
    DevBuf<T> bc;                 // the coarsest right-hand side
    DevBuf<double> part;          // 4 slots x S x G
    DevBuf<OState> ost;
    DevBuf<BState> bst;
    DevBuf<double> winX, winB;        // kSolveWindow x [n][S]: solved pairs for the initial guess
    DevBuf<WinState> win;
    bool use_window = true;
    // rows outside which every right-hand side is zero (the boundary nodes
    // of the Dirichlet problem), or null: the window's dots read only these
    const int* rhs_rows = nullptr;
    int rhs_nrows = 0;
    int win_stride = 1;  // the window's fit reads every win_stride-th of those rows
    OState* h_ost = nullptr;
    BState* h_bst = nullptr;
    static constexpr int kMaxOuter = 8;
    int last_inner[kMaxOuter] = {8, 8, 8, 8, 8, 8, 8, 8};  // per refinement step

    ~BatchSolver() {
        if (h_ost) (void)hipHostFree(h_ost);
        if (h_bst) (void)hipHostFree(h_bst);
    }

    int setup(const CgSolver& solver, int S_, hipStream_t s) {
        n = solver.n;
        S = S_;
        G = row_grid(n);
        const AmgPrecond& M = solver.amg;
        const int L = (int)M.levels.size();
        nc = M.nc;
        folded = M.D.p != nullptr && !wide();
        dense_m = folded ? M.levels[L - 1].n : nc;
        TM_CHECK(dense.alloc((size_t)nc * dense_m));
        TM_HIP(hipMemcpyAsync(dense.p, folded ? M.D.p : M.Cinv.p, (size_t)nc * dense_m * sizeof(double),
                              hipMemcpyDeviceToDevice, s));
        TM_CHECK(sl0.build(n, n, solver.pat.h_rowptr.data(), solver.pat.h_csrcol.data(), S, s));
        TM_CHECK(sl0.values(solver.h_val, wA0, s));
        TM_CHECK(sl0.values(solver.h_val, wA64, s));
        TM_CHECK(t0.build(sl0, s));
        Gr = t0.nt > 0 ? tile_blocks((S + kTileS - 1) / kTileS, kResidPerCu) : G;
        lo.clear();
        lo.resize((size_t)L);
        for (int l = 0; l < L; ++l) {
            const auto& V = M.levels[l];
            const int nnext = l + 1 < L ? M.levels[l + 1].n : M.nc;
            HostCsr down, up;
            TM_CHECK(fetch_csr(V.down, down, s));
            if (l + 1 < L || !folded) {
                TM_CHECK(lo[l].RA.build(nnext, V.n, down.rp.data(), down.ci.data(), S, s));
                TM_CHECK(lo[l].RA.values(down.v, lo[l].wRA, s));
            }
            if (l == 0) {
                up_operator(n, solver.pat.h_rowptr.data(), solver.pat.h_csrcol.data(), solver.h_val,
                            solver.h_dinv.data(), V.omega, down, up);
            } else {
                TM_CHECK(fetch_csr(V.up, up, s));
            }
            TM_CHECK(lo[l].U.build(V.n, V.n + nnext, up.rp.data(), up.ci.data(), S, s));
            TM_CHECK(lo[l].U.values(up.v, lo[l].wU, s));
            if (l == 0) TM_CHECK(tu.build(lo[0].U, s, kUpNodes));
        }
        Gq = Gz = G;
        if (tiled())
            with_tile_type<kTileNodes>([&](auto tt) {
                using TT = decltype(tt);
                const int nch = (S + TT::kSamples - 1) / TT::kSamples;
                Gq = tile_blocks(nch, kSolvePerCu<TT>);
                Gz = tile_blocks(nch, kUpPerCu);
            });
        TM_CHECK(fixed.upload(solver.h_fixed.data(), n, s));
        const size_t NS = (size_t)n * S;
        TM_CHECK(rT.alloc(NS + (size_t)M.tail() * S));
        TM_CHECK(ring.alloc((size_t)(kRing + 1) * NS));
        TM_CHECK(ahist.alloc((size_t)(kRing + 1) * kMaxS));
        TM_CHECK(bhist.alloc((size_t)(kRing + 1) * kMaxS));
        TM_CHECK(chist.alloc((size_t)(kRing + 1) * kMaxS));
        TM_CHECK(q.alloc(NS));
        bx.clear();
        bx.resize((size_t)L);
        for (int l = 1; l < L; ++l)
            TM_CHECK(bx[l].alloc((size_t)(M.levels[l].n + (l + 1 < L ? M.levels[l + 1].n : M.nc)) * S));
        TM_CHECK(bc.alloc((size_t)std::max(1, M.nc) * S));
        TM_CHECK(part.alloc((size_t)std::max(4, kWinDots) * S * gmax() + (size_t)kWinDots * kWinChunks * S));
        TM_CHECK(winX.alloc((size_t)kSolveWindow * NS));
        TM_CHECK(winB.alloc((size_t)kSolveWindow * NS));
        TM_CHECK(win.alloc(1));
        TM_HIP(hipMemsetAsync(win.p, 0, sizeof(WinState), s));
        TM_CHECK(ost.alloc(1));
        TM_CHECK(bst.alloc(1));
        TM_HIP(hipMemsetAsync(bst.p, 0, sizeof(BState), s));  // flags past the batch size stay 0
        if (!h_ost) TM_HIP(hipHostMalloc((void**)&h_ost, sizeof(OState), hipHostMallocDefault));
        if (!h_bst) TM_HIP(hipHostMalloc((void**)&h_bst, sizeof(BState), hipHostMallocDefault));
        TM_HIP(hipStreamSynchronize(s));
        return TM_OK;
    }

    // z = M r (AMG V-cycle, batched) for r = [r | x_c], partial (r, z) into prz:
    // one product per level in each direction, as the single-sample solver's
    int precond(T* r, T* zout, double* prz, hipStream_t s) {
        const int L = (int)lo.size();
        if (L == 0) return TM_ERR_UNSUPPORTED;  // the batched solve needs at least one AMG level
        auto vec = [&](int l) { return l == 0 ? r : bx[l].p; };  // [b | x_c] of level l
        auto tail = [&](int l) { return vec(l) + (size_t)lo[l].U.n * S; };
        for (int l = 0; l < (folded ? L - 1 : L); ++l)
            spmm(lo[l].RA, lo[l].wRA.p, vec(l), l + 1 < L ? vec(l + 1) : bc.p, s);
        dmv(folded ? vec(L - 1) : bc.p, tail(L - 1), s);
        for (int l = L - 1; l > 0; --l) spmm(lo[l].U, lo[l].wU.p, vec(l), tail(l - 1), s);
        up0(r, zout, prz, s);
        TM_HIP(hipGetLastError());
        return TM_OK;
    }

    // y = the coarsest level's dense matrix times x
    void dmv(const T* x, T* y, hipStream_t s) {
        const int rows = nc, m = dense_m;
        const double* D = dense.p;
        auto run = [&](auto vec) {
            constexpr int VEC = decltype(vec)::value;
            const int nch = (S + 16 * VEC - 1) / (16 * VEC);
            if (rows * nch <= 256)
                hipLaunchKernelGGL((k_b_dmv<T, VEC, 1>), dim3(rows, nch), dim3(kDmvThreads), 0, s, rows, m, S, D, x, y,
                                   gate());
            else
                hipLaunchKernelGGL((k_b_dmv<T, VEC, 2>), dim3((rows + 1) / 2, nch), dim3(kDmvThreads), 0, s, rows, m,
                                   S, D, x, y, gate());
        };
        if constexpr (kWideT)
            if (wide()) return run(std::integral_constant<int, 4>{});
        run(std::integral_constant<int, 1>{});
    }

    // level 0 upwards: z = U [r | x_c], partial (r, z)
    void up0(const T* r, T* z, double* prz, hipStream_t s) {
        if (tiled()) {
            with_tile_type<kUpNodes>([&](auto tt) {
                using TT = decltype(tt);
                hipLaunchKernelGGL(k_b_up_t<TT>, dim3(Gz), dim3(kTileThreads), 0, s, tu.args(lo[0].U, TT::kSamples),
                                   (const T*)lo[0].wU.p, r, z, gate(), prz);
            });
            return;
        }
        if constexpr (kWideT) {
            if (wide()) {
                hipLaunchKernelGGL(k_b_up_w, dim3(G), dim3(kBlock), 0, s, gated(lo[0].U.args(4, lo[0].wU.p)),
                                   (const float*)r, (float*)z, prz);
                return;
            }
        }
        hipLaunchKernelGGL((k_b_up<T>), dim3(G), dim3(kBlock), 0, s, gated(lo[0].U.args((int)sizeof(T), lo[0].wU.p)),
                           S, r, z, prz);
    }

    // the per-sample active flags of the inner solve (device address)
    const int* gate() const {
        return bst.p ? (const int*)((const char*)bst.p + offsetof(BState, active)) : nullptr;
    }
    SlotArgs gated(SlotArgs a) const {
        a.gate = gate();
        a.gate_n = S;
        return a;
    }

    // V-cycle kernels; the wide-gather forms for 64 FP32 samples
    static constexpr bool kWideT = sizeof(T) == 4;
    bool wide() const { return kWideT && S == kMaxS; }
    // one block per row for long-row operators (grid: a multiple of the XCD count)
    static dim3 blk_grid(int rows) { return dim3(xcd_grid(std::min(4096, std::max(rows, 1)))); }
    // y = M x (one block per row for long rows in the wide form)
    void spmm(const SlotOp& M, const T* w, const T* x, T* y, hipStream_t s) {
        const SlotArgs a = gated(M.args((int)sizeof(T), w));
        if constexpr (kWideT)
            if (wide()) {
                const float* xf = (const float*)x;
                float* yf = (float*)y;
                if (M.long_rows()) hipLaunchKernelGGL(k_b_spmm_w<true>, blk_grid(a.n), dim3(kBlock), 0, s, a, xf, yf);
                else hipLaunchKernelGGL(k_b_spmm_w<false>, dim3(row_grid(a.n)), dim3(kBlock), 0, s, a, xf, yf);
                return;
            }
        const int nch = (S + 15) / 16;
        if ((int64_t)a.n * nch < 2048)
            hipLaunchKernelGGL((k_b_spmm<T, true>), dim3(xcd_grid(a.n), nch), dim3(kBlock), 0, s, a, S, x, y);
        else
            hipLaunchKernelGGL((k_b_spmm<T, false>), dim3(xcd_grid((a.n + kRowsPerBlock - 1) / kRowsPerBlock), nch),
                               dim3(kBlock), 0, s, a, S, x, y);
    }

    // initial guess of the solve of A x = b from the window of solved pairs;
    // b goes into the head slot
    void win_project(const double* b, double* x, hipStream_t s) {
        const int nr = ((rhs_rows ? rhs_nrows : n) + win_stride - 1) / win_stride;
        const int gw = std::min(row_grid(nr), 1024);  // fewer, longer blocks: half the partials, 1.2x faster at 283k rows
        hipLaunchKernelGGL(k_b_win_dots, dim3(gw), dim3(kBlock), 0, s, n, S, (const WinState*)win.p, winB.p, b,
                           part.p, nr, rhs_rows, win_stride);
        double* red = part.p + (size_t)kWinDots * S * gw;  // after the block partials
        hipLaunchKernelGGL(k_b_win_red, dim3(kWinDots, kWinChunks), dim3(kBlock), 0, s, gw, S, (const double*)part.p,
                           red);
        hipLaunchKernelGGL(k_b_win_solve, dim3(S), dim3(kWave), 0, s, S, win.p, (const double*)red);
        hipLaunchKernelGGL(k_b_win_combine, dim3(G), dim3(kBlock), 0, s, n, S, (const WinState*)win.p,
                           (const double*)winX.p, (const unsigned char*)fixed.p, b, x);
    }
    // the solution beside its b (after win_project); the window is emptied
    // when a sample did not converge
    void win_record(const double* x, hipStream_t s) {
        const size_t NS = (size_t)n * S;
        hipLaunchKernelGGL(k_b_win_store, dim3(elem_grid(NS)), dim3(kBlock), 0, s, NS, (const WinState*)win.p, x,
                           winX.p);
        hipLaunchKernelGGL(k_b_win_advance, dim3(1), dim3(kMaxS), 0, s, S, win.p, (const OState*)ost.p);
    }

    // r -= alpha q, partial (r, r)
    void cg_update(double* prr, hipStream_t s) {
        hipLaunchKernelGGL((k_b_cg_update<T>), dim3(G), dim3(kBlock), 0, s, n, S, (const T*)q.p, rT.p,
                           (const BState*)bst.p, prr);
    }
    // per-sample convergence after cg_update, before the preconditioner
    void conv_check(const double* prr, hipStream_t s) {
        hipLaunchKernelGGL(k_b_red_rr, dim3(S), dim3(kBlock), 0, s, G, S, prr, bst.p);
    }

    // r = b - A x in FP64 (b, x: [n][S]), rT = (T) r, partials (b, b), (r, r)
    void resid(const double* b, const double* x, double* pbb, double* prr, hipStream_t s) {
        if (t0.nt > 0) {
            const TileArgs t = t0.args(sl0);
            if (S % 2 == 0)
                hipLaunchKernelGGL((k_b_resid_t<T, true>), dim3(Gr), dim3(kTileThreads), 0, s, t,
                                   (const double*)wA64.p, b, x, rT.p, pbb, prr);
            else
                hipLaunchKernelGGL((k_b_resid_t<T, false>), dim3(Gr), dim3(kTileThreads), 0, s, t,
                                   (const double*)wA64.p, b, x, rT.p, pbb, prr);
        } else {
            hipLaunchKernelGGL((k_b_resid<T>), dim3(G), dim3(kBlock), 0, s, sl0.args(8, wA64.p), S, b, x, rT.p, pbb,
                               prr);
        }
    }

    // iteration k: q = A p_k = A z_k + beta q, partial (z_k, q)
    void cg_spmv(const T* zk, int k, double* pzq, hipStream_t s) {
        if (tiled()) {
            with_tile_type<kTileNodes>([&](auto tt) {
                using TT = decltype(tt);
                hipLaunchKernelGGL(k_b_cg_spmv_t<TT>, dim3(Gq), dim3(kTileThreads), 0, s, t0.args(sl0, TT::kSamples),
                                   (const T*)wA0.p, zk, q.p, k, (const BState*)bst.p, pzq);
            });
            return;
        }
        if constexpr (kWideT)
            if (wide()) {
                hipLaunchKernelGGL(k_b_cg_spmv_w, dim3(G), dim3(kBlock), 0, s, gated(sl0.args(4, wA0.p)),
                                   (const float*)zk, (float*)q.p, k, (const BState*)bst.p, pzq);
                return;
            }
        hipLaunchKernelGGL((k_b_cg_spmv<T>), dim3(G), dim3(kBlock), 0, s, gated(sl0.args((int)sizeof(T), wA0.p)), S,
                           zk, q.p, k, (const BState*)bst.p, pzq);
    }

    // Solves A x = b for all samples ([n][S] FP64); x is the warm start.
    int solve(const double* b, double* x, double tol, int maxit, hipStream_t s, int* outer_out, int* inner_out,
              double* maxrel) {
        if (lo.empty()) return TM_ERR_UNSUPPORTED;
        const size_t NS = (size_t)n * S;
        double* pbb = part.p;
        double* prr = part.p + (size_t)S * gmax();
        double* prz = part.p + (size_t)2 * S * gmax();
        double* pzq = part.p + (size_t)3 * S * gmax();
        const double itol = sizeof(T) == 4 ? 1e-5 : 0.0;  // FP32 inner target per refinement step
        int outer = 0, inner_total = 0;
        if (use_window) win_project(b, x, s);  // (sets the fixed rows too)
        else hipLaunchKernelGGL(k_b_fix, dim3(elem_grid(NS)), dim3(kBlock), 0, s, n, S, fixed.p, b, x);
        // Host checks: after a solve that took one refinement step (the steady
        // state along a trajectory), the next one takes its first refinement
        // step without waiting for the initial residual check and enqueues
        // exactly the inner iterations the last solve needed without waiting
        // either (and no V-cycle after the last of them, whose z would go
        // unused): one host synchronisation per solve.  A sample still short of its
        // inner target after such a step is taken up by the next refinement
        // step, checked as usual, and the solve after it checks as usual too.
        bool spec_ok = spec_next;  // this solve may skip checks
        bool short_seen = false;
        bool pending = false;      // a speculative inner solve whose counts are read at the next check
        int pend_step = 0;
        for (;;) {
            resid(b, x, pbb, prr, s);
            hipLaunchKernelGGL(k_b_outer_red, dim3(S), dim3(kBlock), 0, s, Gr, S, pbb, prr, tol, itol, ost.p, bst.p,
                               (int*)nullptr);
            if (!(outer == 0 && spec_ok && last_inner[0] > 0)) {
                TM_HIP(hipMemcpyAsync(h_ost, ost.p, sizeof(OState), hipMemcpyDeviceToHost, s));
                TM_HIP(hipStreamSynchronize(s));
                if (pending) {
                    int used = 0;  // iterations the slowest sample ran
                    bool still = false;
                    for (int k = 0; k < S; ++k) {
                        used = std::max(used, h_bst->iters[k]);
                        still = still || h_bst->active[k];
                    }
                    last_inner[pend_step] = used;
                    inner_total += used;
                    pending = false;
                    if (still) {  // the enqueued iterations fell short: check as usual from here on
                        spec_ok = false;
                        short_seen = true;
                    }
                }
                bool all = true, finite = true;
                double worst = 0.0;
                for (int k = 0; k < S; ++k) {
                    all = all && h_ost->done[k];
                    finite = finite && h_ost->done[k] != 2;
                    if (h_ost->bb[k] > 0) worst = std::max(worst, std::sqrt(h_ost->rr[k] / h_ost->bb[k]));
                }
                if (!finite) worst = NAN;
                if (maxrel) *maxrel = worst;
                if (all || outer >= 8 || inner_total >= maxit) break;
            }
            ++outer;
            // inner solve A d = rT from d = 0; x += d at the end
            TM_CHECK(precond(rT.p, ring.p, prz, s));
            hipLaunchKernelGGL(k_b_red_rz, dim3(S), dim3(kBlock), 0, s, Gz, S, prz, -1, bst.p, bhist.p);
            int enq = 0;
            const int kmax = std::min(kRing, maxit);
            // iterations enqueued before the first check: what this refinement
            // step needed last time, plus one when the host checks after them
            // (queued iterations past convergence return at once, but their
            // launches still cost); unchecked, exactly that many: a sample
            // that needs more is taken up by the next refinement step
            const int step = std::min(outer, kMaxOuter) - 1;
            const bool spec = spec_ok && last_inner[step] > 0;
            int chunk = spec ? last_inner[step] : std::max(2, last_inner[step] + 1);
            for (;;) {
                for (int c = 0; c < chunk && enq < kmax; ++c, ++enq) {
                    T* zk = ring.p + (size_t)enq * NS;
                    cg_spmv(zk, enq, pzq, s);
                    hipLaunchKernelGGL(k_b_red_pq, dim3(S), dim3(kBlock), 0, s, Gq, S, pzq, bst.p,
                                       ahist.p + (size_t)enq * kMaxS);
                    cg_update(prr, s);
                    conv_check(prr, s);
                    // no iteration follows the last one of an unchecked chunk
                    // (or of the ring): its z would go unused
                    if ((spec && c + 1 == chunk) || enq + 1 == kmax) continue;
                    TM_CHECK(precond(rT.p, zk + NS, prz, s));
                    hipLaunchKernelGGL(k_b_red_rz, dim3(S), dim3(kBlock), 0, s, Gz, S, prz, enq, bst.p,
                                       bhist.p + (size_t)(enq + 1) * kMaxS);
                }
                TM_HIP(hipGetLastError());
                // the per-sample counts (read after the next wait for the speculative step)
                TM_HIP(hipMemcpyAsync(h_bst, bst.p, sizeof(BState), hipMemcpyDeviceToHost, s));
                if (spec) break;
                TM_HIP(hipStreamSynchronize(s));
                bool any = false;
                for (int k = 0; k < S; ++k) any = any || h_bst->active[k];
                if (!any || enq >= kmax) break;
                chunk = 2;
            }
            if (spec) {
                pending = true;
                pend_step = step;
            } else {
                int used = 0;  // iterations the slowest sample ran
                for (int k = 0; k < S; ++k) used = std::max(used, h_bst->iters[k]);
                last_inner[step] = used;
                inner_total += used;
            }
            if (S == kMaxS && enq <= kCombineK) {
                hipLaunchKernelGGL(k_b_coef, dim3(1), dim3(kMaxS), 0, s, S, enq, (const double*)ahist.p,
                                   (const double*)bhist.p, chist.p);
                hipLaunchKernelGGL((k_b_combine4<T>), dim3(elem_grid(NS / 4)), dim3(kBlock), 0, s, NS, enq,
                                   (const T*)ring.p, (const double*)chist.p, x);
            } else
                hipLaunchKernelGGL((k_b_combine<T>), dim3(elem_grid(NS)), dim3(kBlock), 0, s, NS, S, enq,
                                   (const T*)ring.p, (const double*)ahist.p, (const double*)bhist.p, x);
        }
        if (use_window) win_record(x, s);
        if (outer_out) *outer_out = outer;
        if (inner_out) *inner_out = inner_total;
        last_outer = outer;
        spec_next = outer == 1 && !short_seen;
        TM_HIP(hipGetLastError());
        int st = TM_OK;
        for (int k = 0; k < S; ++k) {
            if (h_ost->done[k] == 2) return TM_ERR_NONFINITE;
            if (h_ost->done[k] == 0) st = TM_ERR_MAXITER;
        }
        return st;
    }

    int last_outer = 0;  // refinement steps of the last host-polled solve
    bool spec_next = false;  // the last solve took one refinement step: the next may skip host checks

    // Times the level-0 kernels of one inner iteration and of the outer
    // residual, each launched `reps` times alone (all samples active), and
    // appends (name, ms per launch, algorithmic bytes per launch): slot
    // offsets (4 B) and weights once, every vector read or written once.
    template <class Timer>
    int time_kernels(hipStream_t s, Timer&& timeit, std::vector<tm_batch_kernel_time>& out) {
        if (lo.empty()) return TM_ERR_UNSUPPORTED;
        const int e = (int)sizeof(T);
        const double nS = (double)n * S;
        double* pzq = part.p + (size_t)3 * S * gmax();
        double* prz = part.p + (size_t)2 * S * gmax();
        auto add = [&out](const char* nm, double ms, double bytes) {
            tm_batch_kernel_time k = {};
            std::snprintf(k.name, sizeof(k.name), "%s", nm);
            k.ms = ms;
            k.bytes = bytes;
            out.push_back(k);
        };
        auto slots = [](const SlotOp& o) { return (double)o.h_sp[o.n]; };
        hipLaunchKernelGGL(k_b_activate, dim3(1), dim3(kMaxS), 0, s, S, bst.p);
        add(tiled() ? "k_b_cg_spmv_t" : wide() ? "k_b_cg_spmv_w" : "k_b_cg_spmv",
            timeit([&] { cg_spmv(ring.p, 0, pzq, s); }), slots(sl0) * (4 + e) + 3.0 * nS * e);
        add(sizeof(T) == 4 ? "k_b_cg_update<float>" : "k_b_cg_update<double>",
            timeit([&] { cg_update(part.p + (size_t)S * gmax(), s); }), 3.0 * nS * e);
        const LvOps& O = lo[0];
        const double n1 = lo.size() > 1 ? lo[1].U.n : nc;
        if (O.RA.n > 0) {
            T* y1 = lo.size() > 1 ? bx[1].p : bc.p;
            add(O.RA.long_rows() && wide() ? "k_b_spmm_w<long> (R(I-AwD^-1), level 0)"
                                           : "k_b_spmm (R(I-AwD^-1), level 0)",
                timeit([&] { spmm(O.RA, O.wRA.p, rT.p, y1, s); }), slots(O.RA) * (4 + e) + nS * e + n1 * S * e);
        } else {
            add("k_b_dmv (C^-1 R(I-AwD^-1), level 0)",
                timeit([&] { dmv(rT.p, rT.p + (size_t)n * S, s); }), 8.0 * nc * n + nS * e + n1 * S * e);
        }
        add(tiled() ? "k_b_up_t (level 0)" : wide() ? "k_b_up_w (level 0)" : "k_b_up (level 0)",
            timeit([&] { up0(rT.p, ring.p, prz, s); }), slots(O.U) * (4 + e) + 2.0 * nS * e + n1 * S * e);
        double* pbb = part.p;
        double* prr = part.p + (size_t)S * gmax();
        const char* resid_name = t0.nt > 0 ? (sizeof(T) == 4 ? "k_b_resid_t<float>" : "k_b_resid_t<double>")
                                           : (sizeof(T) == 4 ? "k_b_resid<float>" : "k_b_resid<double>");
        add(resid_name, timeit([&] { resid(lv0_b64(), lv0_x64(), pbb, prr, s); }),
            slots(sl0) * (4 + 8) + 2.0 * nS * 8 + nS * e);
        return TM_OK;
    }
    // FP64 [n][S] operands of the outer residual for kernel timing (the
    // solver's own FP64 vectors are the caller's; ring storage is large enough)
    const double* lv0_b64() const { return (const double*)ring.p; }
    const double* lv0_x64() const { return (const double*)(ring.p + (size_t)2 * n * S * 8 / sizeof(T)); }

    // The same solve with no host synchronisation (capturable in a HIP graph):
    // exactly `nouter` refinement steps of ninner[o] inner iterations each.
    // Every solver kernel is gated on the per-sample flags, so refinement
    // steps and iterations past convergence cost only their launches, and
    // iterations a sample did not take carry alpha = beta = 0 into the
    // combination.  A final residual check adds the number of samples that
    // missed the tolerance to *fail on the device, the number of those that are
    // not finite to *bad, and track[o] keeps the largest iteration count of
    // refinement step o.
    int enqueue(const double* b, double* x, double tol, int nouter, const int* ninner, hipStream_t s,
                unsigned* fail, unsigned* bad, int* track) {
        if (lo.empty()) return TM_ERR_UNSUPPORTED;
        if (nouter < 0 || nouter > kMaxOuter || !fail || !bad || !track) return TM_ERR_BAD_ARG;
        const size_t NS = (size_t)n * S;
        double* pbb = part.p;
        double* prr = part.p + (size_t)S * gmax();
        double* prz = part.p + (size_t)2 * S * gmax();
        double* pzq = part.p + (size_t)3 * S * gmax();
        const double itol = sizeof(T) == 4 ? 1e-5 : 0.0;
        if (use_window) win_project(b, x, s);  // (sets the fixed rows too)
        else hipLaunchKernelGGL(k_b_fix, dim3(elem_grid(NS)), dim3(kBlock), 0, s, n, S, fixed.p, b, x);
        for (int o = 0;; ++o) {
            resid(b, x, pbb, prr, s);
            hipLaunchKernelGGL(k_b_outer_red, dim3(S), dim3(kBlock), 0, s, Gr, S, pbb, prr, tol, itol, ost.p, bst.p,
                               o > 0 ? track + (o - 1) : (int*)nullptr);
            if (o == nouter) break;
            TM_CHECK(precond(rT.p, ring.p, prz, s));
            hipLaunchKernelGGL(k_b_red_rz, dim3(S), dim3(kBlock), 0, s, Gz, S, prz, -1, bst.p, bhist.p);
            const int K = std::max(1, std::min(kRing, ninner[o]));
            for (int k = 0; k < K; ++k) {
                T* zk = ring.p + (size_t)k * NS;
                cg_spmv(zk, k, pzq, s);
                hipLaunchKernelGGL(k_b_red_pq, dim3(S), dim3(kBlock), 0, s, Gq, S, pzq, bst.p,
                                   ahist.p + (size_t)k * kMaxS);
                cg_update(prr, s);
                conv_check(prr, s);
                if (k + 1 == K) break;  // the last z would go unused
                TM_CHECK(precond(rT.p, zk + NS, prz, s));
                hipLaunchKernelGGL(k_b_red_rz, dim3(S), dim3(kBlock), 0, s, Gz, S, prz, k, bst.p,
                                   bhist.p + (size_t)(k + 1) * kMaxS);
            }
            if (S == kMaxS && K <= kCombineK) {
                hipLaunchKernelGGL(k_b_coef, dim3(1), dim3(kMaxS), 0, s, S, K, (const double*)ahist.p,
                                   (const double*)bhist.p, chist.p);
                hipLaunchKernelGGL((k_b_combine4<T>), dim3(elem_grid(NS / 4)), dim3(kBlock), 0, s, NS, K,
                                   (const T*)ring.p, (const double*)chist.p, x);
            } else
                hipLaunchKernelGGL((k_b_combine<T>), dim3(elem_grid(NS)), dim3(kBlock), 0, s, NS, S, K,
                                   (const T*)ring.p, (const double*)ahist.p, (const double*)bhist.p, x);
        }
        hipLaunchKernelGGL(k_b_count_undone, dim3(1), dim3(kMaxS), 0, s, S, (const OState*)ost.p, fail, bad);
        if (use_window) win_record(x, s);
        TM_HIP(hipGetLastError());
        return TM_OK;
    }
};

}  // namespace tmh

using namespace tmh;

// tm_ctx internals needed here (defined in tm_field.hip)
namespace tmh {
}  // namespace tmh

struct tm_batch {
    int n = 0, S = 0, prec = TM_PREC_FP64;
    tm_ctx* ctx = nullptr;
    hipStream_t stream = nullptr;
    rocblas_handle blas = nullptr;
    CtxView cv{};
    SlotOp eo;                         // union pattern of the per-node operators, in row slots
    TileOp et;                         // its tiles
    DevBuf<double> xw, gx, gy, gz, tx, ty, tz, cx, cy, cz;  // slot weights: exchange, grad, tGrad, curl
    bool exch = false, dmi = false;
    DevBuf<double> m, dmdt, heff, u1, u2, usum, rhsN, rhsD, U, Gm, hext, torque;
    DevBuf<double> m2;                 // the next magnetisation of tm_batch_eval_euler (swapped with m)
    DevBuf<float> Bf, Uf, Gf;          // FP32 boundary product (TM_PREC_MIXED_BEM32)
    DevBuf<float> Pf;                  // its split-K partial products (nchunk x b x S)
    int kchunk = 512, nchunk = 0;
    // int8 digit-slice boundary product (TM_PREC_MIXED_BEMI8): B's digits
    // (Bq, 5 bytes per entry), the per-call digits of U, the row and sample
    // maxima, the split-K partials, and the tuned tile rows / K split
    DevBuf<int> Bq, Uq;
    DevBuf<double> i8rmax, i8umax, i8P;
    int i8nT = 0, i8nC = 0, i8nw = 8, i8ks = 1, i8candidates = 0;
    float i8ms = 0.0f, i8ms_first = 0.0f;
    DevBuf<double> rk_k[4], rk_base;   // RK4 stages and the step's start state
    // graph-replayed RK4 steps: samples whose fixed-budget solve missed the
    // tolerance, those that were not finite, and the iterations that each
    // refinement step of the two solves took (device counters), and the budgets: refinement
    // steps and inner iterations per step of the Neumann (0) and Dirichlet (1)
    // solves
    static constexpr int kMaxBud = 8;
    static constexpr int kCounts = 2 + 2 * kMaxBud;  // missed, not finite, iterations
    DevBuf<unsigned> rk_fail;
    bool bud_set = false;
    bool m_replaced = false;  // m was set from outside since the last step
    int bud_outer[2] = {0, 0};
    int bud_inner[2][kMaxBud] = {};
    // The captured step is kept for the next call with the same arguments
    // (capturing and instantiating its few hundred nodes takes as long as two
    // replays); the key holds everything the graph has by value that can
    // change after the batch's creation, the magnetisation's buffer and the
    // context's per-node field among it.
    struct StepKey {
        double dtau = 0.0, alpha = 0.0;
        int variant = -1;
        const double* m = nullptr;
        const double* hfield = nullptr;
        int outer[2] = {0, 0};
        int inner[2][kMaxBud] = {};
        bool operator==(const StepKey& o) const {
            bool e = dtau == o.dtau && alpha == o.alpha && variant == o.variant && m == o.m && hfield == o.hfield;
            for (int w = 0; w < 2; ++w) {
                e = e && outer[w] == o.outer[w];
                for (int k = 0; k < outer[w] && e; ++k) e = inner[w][k] == o.inner[w][k];
            }
            return e;
        }
    };
    StepKey step_key;
    hipGraphExec_t step_exec = nullptr;
    void drop_step() {
        if (step_exec) (void)hipGraphExecDestroy(step_exec);
        step_exec = nullptr;
    }
    int gemm_sol = 0;                  // tuned rocBLAS solution index (0: library default)
    bool gemm_own = false;             // the MFMA kernel k_b_gemm64 won the tuning
    int gemm_shape = 0, gemm_ks = 1;   // its tile shape and K split
    int gemm_own_candidates = 0;       // (shape, K split) pairs timed
    bool own_ok = false;               // an own-kernel candidate agreed with rocBLAS (used in captured graphs)
    float own_ms = 0.0f;
    int own_shape = 0, own_ks = 1;
    DevBuf<double> Pd;                 // its split-K partials (ks x b x S)
    double gemm_own_err = 0.0;         // its largest relative difference to rocBLAS at tuning
    int gemm_candidates = 0;
    float gemm_ms_default = 0.0f, gemm_ms_best = 0.0f;
    BatchSolver<double> sN64, sD64;
    BatchSolver<float> sN32, sD32;
    bool timers = false;
    hipEvent_t ev[6] = {};
    tm_phase_times tsum = {};
    // in-pipeline event pairs around the boundary GEMM (tm_batch_gemm_live)
    static constexpr int kLivePairs = 256;
    hipEvent_t lev[2 * kLivePairs] = {};
    int lev_n = 0;
    bool lev_on = false;
    bool capturing = false;  // a step is being captured: an event recorded now could not be read
    // marks the start (0) or end (1) of a boundary GEMM launch while recording
    void live_mark(int which) {
        if (!lev_on || capturing || lev_n >= kLivePairs) return;
        (void)hipEventRecord(lev[2 * lev_n + which], stream);
        if (which == 1) ++lev_n;
    }
};

namespace {

// CSR values of an operator on the union pattern (pattern entries it lacks are 0).
int csr_on_pattern(const SellPattern& P, const std::vector<int>& rp, const std::vector<int>& col,
                   const std::vector<double>& val, std::vector<double>& out) {
    out.assign(P.h_csrcol.size(), 0.0);
    for (int i = 0; i < P.n; ++i) {
        int k = P.h_rowptr[i];
        for (int q = rp[i]; q < rp[i + 1]; ++q) {
            while (k < P.h_rowptr[i + 1] && P.h_csrcol[k] < col[q]) ++k;
            if (k >= P.h_rowptr[i + 1] || P.h_csrcol[k] != col[q]) return TM_ERR_BAD_ARG;
            out[k] += val[q];
        }
    }
    return TM_OK;
}

// Slot weights of one operator; with colscale, entry (i, j) is scaled by w0 colscale[j].
int upload_op(tm_batch* bt, int op, DevBuf<double>& dst, const double* colscale = nullptr, double w0 = 1.0) {
    std::vector<double> v;
    TM_CHECK(csr_on_pattern(*bt->cv.pat, *bt->cv.hop_rp[op], *bt->cv.hop_col[op], *bt->cv.hop_val[op], v));
    return bt->eo.values(v, dst, bt->stream, colscale, w0);
}

}  // namespace

namespace {

// The boundary GEMM G (b x S) = B (b x b) * U^T (S x b) is a tall, thin
// product; the library's default tile wastes half of a 128-wide tile on
// S = 64.  At batch creation every solution rocBLAS offers for this exact
// shape and layout is timed (HIP events, one warm-up and two timed runs) and
// the fastest is kept.
// FP32 products over K chunks of kchunk columns of B (strided-batched GEMM,
// FP32 accumulation inside a chunk only), partials left in Pf.
int gemm_split_f32(tm_batch* bt) {
    const CtxView& v = bt->cv;
    const int b = v.bnx, S = bt->S, kc = bt->kchunk;
    const int nfull = b / kc, tail = b - nfull * kc;
    const float one = 1.0f, zero = 0.0f;
    if (nfull > 0 &&
        rocblas_sgemm_strided_batched(bt->blas, rocblas_operation_none, rocblas_operation_transpose, b, S, kc, &one,
                                      bt->Bf.p, v.bld, (rocblas_stride)kc * v.bld, bt->Uf.p, S, (rocblas_stride)kc * S,
                                      &zero, bt->Pf.p, b, (rocblas_stride)b * S, nfull) != rocblas_status_success)
        return TM_ERR_HIP;
    if (tail > 0 &&
        rocblas_sgemm(bt->blas, rocblas_operation_none, rocblas_operation_transpose, b, S, tail, &one,
                      bt->Bf.p + (size_t)nfull * kc * v.bld, v.bld, bt->Uf.p + (size_t)nfull * kc * S, S, &zero,
                      bt->Pf.p + (size_t)nfull * b * S, b) != rocblas_status_success)
        return TM_ERR_HIP;
    return TM_OK;
}

int gemm_run(tm_batch* bt, int sol) {
    const CtxView& v = bt->cv;
    const int b = v.bnx, S = bt->S;
    const bool f32 = bt->prec == TM_PREC_MIXED_BEM32;
    if (f32) return gemm_split_f32(bt);
    const rocblas_datatype t = f32 ? rocblas_datatype_f32_r : rocblas_datatype_f64_r;
    const double one = 1.0, zero = 0.0;
    const float onef = 1.0f, zerof = 0.0f;
    const void* al = f32 ? (const void*)&onef : (const void*)&one;
    const void* be = f32 ? (const void*)&zerof : (const void*)&zero;
    const void* A = f32 ? (const void*)bt->Bf.p : (const void*)v.B;
    const void* U = f32 ? (const void*)bt->Uf.p : (const void*)bt->U.p;
    void* G = f32 ? (void*)bt->Gf.p : (void*)bt->Gm.p;
    const rocblas_status r =
        rocblas_gemm_ex(bt->blas, rocblas_operation_none, rocblas_operation_transpose, b, S, b, al, A, t, v.bld, U, t,
                        S, be, G, t, b, G, t, b, t, sol != 0 ? rocblas_gemm_algo_solution_index : rocblas_gemm_algo_standard,
                        sol, 0);
    return r == rocblas_status_success ? TM_OK : TM_ERR_HIP;
}

__global__ __launch_bounds__(kBlock) void k_b_fill_pattern(size_t n, double* __restrict__ x) {
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < n; e += (size_t)gridDim.x * kBlock)
        x[e] = sin(0.37 * (double)(e % 100003)) + 0.25;
}

// out[0] = max |own - ref|, out[1] = max |ref| (both zero before) for own b x S
// row-major and ref column-major; a difference that is not a number is infinite
__global__ __launch_bounds__(kBlock) void k_b_max_diff(int b, int S, const double* __restrict__ own,
                                                       const double* __restrict__ ref, double* out) {
    double d = 0.0, r = 0.0;
    const size_t tot = (size_t)b * S;
    for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < tot; e += (size_t)gridDim.x * kBlock) {
        const double x = ref[(e % S) * b + e / S], y = fabs(own[e] - x);
        d = fmax(d, y == y ? y : INFINITY);
        r = fmax(r, fabs(x));
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        d = fmax(d, __shfl_xor(d, o));
        r = fmax(r, __shfl_xor(r, o));
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        atomic_max_nonneg(out, d);
        atomic_max_nonneg(out + 1, r);
    }
}

// K splits worth timing for a tile shape: the one that gives ~1024 blocks,
// and those that fill j = 1..6 rounds of the resident block slots (all
// blocks carry the same work, so a last round that is only partly filled
// leaves CUs idle).  At most 16 partial products.
std::vector<int> gemm_ks_candidates(int b, int shape, int S, int ncu) {
    const int rows = gemm_rows_per_block(shape);
    const int grid_m = (b + rows - 1) / rows;
    std::vector<int> ks = {std::max(1, std::min(16, (1024 + grid_m - 1) / grid_m))};
    const int slots = ncu * gemm_blocks_per_cu(shape, S);
    for (int j = 1; j <= 6 && slots > 0; ++j) {
        const int k = std::max(1, std::min(16, j * slots / grid_m));
        if (std::find(ks.begin(), ks.end(), k) == ks.end()) ks.push_back(k);
    }
    return ks;
}

int gemm_own_run(tm_batch* bt, double* G) {
    const CtxView& v = bt->cv;
    const int b = v.bnx;
    const int rows = gemm_rows_per_block(bt->gemm_shape);
    const int kper = (b + bt->gemm_ks - 1) / bt->gemm_ks;
    launch_gemm64(bt->gemm_shape, dim3((b + rows - 1) / rows, bt->gemm_ks), bt->stream, b, v.bld,
                  bt->S, v.B, (const double*)bt->U.p, kper, bt->Pd.p);
    TM_HIP(hipGetLastError());
    if (G) {  // sum the partials into G (b x S, row-major) without scatter
        hipLaunchKernelGGL(k_b_ksum_scatter, dim3(elem_grid((size_t)b * bt->S)), dim3(kBlock), 0, bt->stream, b,
                           bt->S, bt->gemm_ks, (const int*)nullptr, (const double*)bt->Pd.p, G);
        TM_HIP(hipGetLastError());
    }
    return TM_OK;
}

int tune_gemm(tm_batch* bt) {
    const CtxView& v = bt->cv;
    const int b = v.bnx, S = bt->S;
    const bool f32 = bt->prec == TM_PREC_MIXED_BEM32;
    const rocblas_datatype t = f32 ? rocblas_datatype_f32_r : rocblas_datatype_f64_r;
    const double one = 1.0, zero = 0.0;
    const float onef = 1.0f, zerof = 0.0f;
    const void* al = f32 ? (const void*)&onef : (const void*)&one;
    const void* be = f32 ? (const void*)&zerof : (const void*)&zero;
    const void* A = f32 ? (const void*)bt->Bf.p : (const void*)v.B;
    void* U = f32 ? (void*)bt->Uf.p : (void*)bt->U.p;
    void* G = f32 ? (void*)bt->Gf.p : (void*)bt->Gm.p;
    TM_HIP(hipMemsetAsync(U, 0, (size_t)b * S * (f32 ? sizeof(float) : sizeof(double)), bt->stream));
    if (f32) return TM_OK;  // split-K FP32 product: library defaults
    // every candidate (rocBLAS and own) is timed on the same non-zero operand:
    // matrix cores multiplying zeros draw less power and clock higher, which
    // would favour whichever candidates were timed on a zero U
    hipLaunchKernelGGL(k_b_fill_pattern, dim3(elem_grid((size_t)b * S)), dim3(kBlock), 0, bt->stream, (size_t)b * S,
                       bt->U.p);
    rocblas_int nsol = 0;
    if (rocblas_gemm_ex_get_solutions(bt->blas, rocblas_operation_none, rocblas_operation_transpose, b, S, b, al, A,
                                      t, v.bld, U, t, S, be, G, t, b, G, t, b, t, rocblas_gemm_algo_solution_index, 0,
                                      nullptr, &nsol) != rocblas_status_success ||
        nsol <= 0)
        return TM_OK;  // keep the default
    std::vector<rocblas_int> sols((size_t)nsol);
    if (rocblas_gemm_ex_get_solutions(bt->blas, rocblas_operation_none, rocblas_operation_transpose, b, S, b, al, A,
                                      t, v.bld, U, t, S, be, G, t, b, G, t, b, t, rocblas_gemm_algo_solution_index, 0,
                                      sols.data(), &nsol) != rocblas_status_success)
        return TM_OK;
    hipEvent_t e0, e1;
    TM_HIP(hipEventCreate(&e0));
    TM_HIP(hipEventCreate(&e1));
    auto time_sol = [&](int sol, float* ms) -> bool {
        if (gemm_run(bt, sol) != TM_OK) return false;
        if (hipEventRecord(e0, bt->stream) != hipSuccess) return false;
        for (int k = 0; k < 2; ++k)
            if (gemm_run(bt, sol) != TM_OK) return false;
        if (hipEventRecord(e1, bt->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) return false;
        float t2 = 0.0f;
        (void)hipEventElapsedTime(&t2, e0, e1);
        *ms = 0.5f * t2;
        return true;
    };
    float best = 0.0f;
    if (!time_sol(0, &best)) best = 1e30f;
    bt->gemm_ms_default = best;
    bt->gemm_sol = 0;
    const int cap = std::min<int>((int)sols.size(), 64);
    for (int k = 0; k < cap; ++k) {
        float ms = 0.0f;
        if (time_sol(sols[k], &ms) && ms < best) {
            best = ms;
            bt->gemm_sol = sols[k];
        }
    }
    (void)hipGetLastError();  // a rejected candidate leaves no error behind
    bt->gemm_candidates = cap;
    // the MFMA kernel, each tile shape and K split: checked against the
    // library on a non-zero U, then timed
    if (!f32) {
        int dev = 0, ncu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            ncu = 0;
        std::vector<std::pair<int, int>> cand;  // (shape, ks)
        int ksmax = 1;
        for (int sh = 0; sh < gemm_shapes(S); ++sh)
            for (int k : gemm_ks_candidates(b, sh, S, ncu)) {
                cand.push_back({sh, k});
                ksmax = std::max(ksmax, k);
            }
        if (bt->Pd.alloc((size_t)ksmax * b * S) == TM_OK) {
            hipLaunchKernelGGL(k_b_fill_pattern, dim3(elem_grid((size_t)b * S)), dim3(kBlock), 0, bt->stream,
                               (size_t)b * S, bt->U.p);
            // compared on the device: copying every candidate's product back and comparing
            // it on the host was most of the tuning's time (6,000 rows, 63 samples: 30 ms)
            DevBuf<double> G2, dmax;
            const bool ok = G2.alloc((size_t)b * S) == TM_OK && dmax.alloc(2) == TM_OK &&
                            gemm_run(bt, bt->gemm_sol) == TM_OK;
            const int keep_shape = bt->gemm_shape, keep_ks = bt->gemm_ks;
            int best_shape = -1, best_ks = 1;
            for (size_t ci = 0; ok && ci < cand.size(); ++ci) {
                bt->gemm_shape = cand[ci].first;
                bt->gemm_ks = cand[ci].second;
                double m[2] = {};
                hipLaunchKernelGGL(k_b_zero_small, dim3(1), dim3(kMaxS), 0, bt->stream, 2, dmax.p);
                if (gemm_own_run(bt, G2.p) != TM_OK) break;
                hipLaunchKernelGGL(k_b_max_diff, dim3(elem_grid((size_t)b * S)), dim3(kBlock), 0, bt->stream, b, S,
                                   (const double*)G2.p, (const double*)bt->Gm.p, dmax.p);
                if (hipMemcpyAsync(m, dmax.p, sizeof(m), hipMemcpyDeviceToHost, bt->stream) != hipSuccess ||
                    hipStreamSynchronize(bt->stream) != hipSuccess)
                    break;
                const double err = m[1] > 0 ? m[0] / m[1] : m[0];
                bt->gemm_own_err = std::max(bt->gemm_own_err, err);
                if (!(err <= 1e-12)) continue;  // never choose a kernel that disagrees with the library
                float ms = 0.0f;
                bool run_ok = hipEventRecord(e0, bt->stream) == hipSuccess;
                for (int k = 0; k < 2 && run_ok; ++k) run_ok = gemm_own_run(bt, nullptr) == TM_OK;
                if (run_ok && hipEventRecord(e1, bt->stream) == hipSuccess && hipEventSynchronize(e1) == hipSuccess) {
                    (void)hipEventElapsedTime(&ms, e0, e1);
                    ms *= 0.5f;
                    if (ms < best) {
                        best = ms;
                        best_shape = bt->gemm_shape;
                        best_ks = bt->gemm_ks;
                    }
                    if (S == 64 && (!bt->own_ok || ms < bt->own_ms)) {  // the fastest verified own kernel, for graphs
                        bt->own_ok = true;
                        bt->own_ms = ms;
                        bt->own_shape = bt->gemm_shape;
                        bt->own_ks = bt->gemm_ks;
                    }
                }
            }
            bt->gemm_own_candidates = (int)cand.size();
            if (best_shape >= 0) {
                bt->gemm_own = true;
                bt->gemm_shape = best_shape;
                bt->gemm_ks = best_ks;
            } else {
                bt->gemm_shape = keep_shape;
                bt->gemm_ks = keep_ks;
            }
            TM_HIP(hipMemsetAsync(bt->U.p, 0, (size_t)b * S * sizeof(double), bt->stream));
        }
    }
    bt->gemm_ms_best = best;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return TM_OK;
}

// ---- int8 digit-slice boundary product: set-up, tuning, one product --------
inline const i32x4* i8ops(const DevBuf<int>& q) { return reinterpret_cast<const i32x4*>(q.p); }

// chunks per K range: a multiple of the kernel's three register sets
inline int i8_range(int nC, int ks) { return ((nC + ks - 1) / ks + 2) / 3 * 3; }

int i8_gemm(tm_batch* bt, int nw, int ks) {
    const int cper = i8_range(bt->i8nC, ks);
    const dim3 g((bt->i8nT + nw - 1) / nw, ks);
    launch_gemm_i8(nw, g, bt->stream, bt->cv.bnx, bt->i8nT, bt->i8nC, cper, i8ops(bt->Bq), i8ops(bt->Uq), bt->i8P.p);
    TM_HIP(hipGetLastError());
    return TM_OK;
}

// U's digits from the boundary values u[bn[k]][s] (u[k][s] without bn)
int i8_uslice(tm_batch* bt, const int* bn, const double* u) {
    const int b = bt->cv.bnx, S = bt->S;
    hipStream_t s = bt->stream;
    hipLaunchKernelGGL(k_b_i8_zero, dim3(1), dim3(64), 0, s, 64, bt->i8umax.p);
    hipLaunchKernelGGL(k_b_i8_umax, dim3(std::min(1024, (b + 3) / 4)), dim3(kBlock), 0, s, b, S, bn, u,
                       bt->i8umax.p);
    hipLaunchKernelGGL(k_b_i8_uslice, dim3(elem_grid((size_t)bt->i8nC * 256)), dim3(kBlock), 0, s, b, S, bt->i8nC,
                       bn, u, (const double*)bt->i8umax.p, reinterpret_cast<i32x4*>(bt->Uq.p));
    TM_HIP(hipGetLastError());
    return TM_OK;
}

int i8_product(tm_batch* bt, const int* bn, const double* u, double* out) {
    TM_CHECK(i8_uslice(bt, bn, u));
    bt->live_mark(0);
    TM_CHECK(i8_gemm(bt, bt->i8nw, bt->i8ks));
    bt->live_mark(1);
    hipLaunchKernelGGL(k_b_i8_finish, dim3(elem_grid((size_t)bt->cv.bnx * 64)), dim3(kBlock), 0, bt->stream,
                       bt->cv.bnx, bt->S, bt->i8ks, bn, (const double*)bt->i8P.p, (const double*)bt->i8rmax.p,
                       (const double*)bt->i8umax.p, out);
    TM_HIP(hipGetLastError());
    return TM_OK;
}

constexpr int kI8Splits[] = {1, 2, 3, 4, 5, 6, 7, 8};
constexpr int kI8MaxSplit = 8;

// B's digits (once per batch), then the block size (4 or 8 wavefronts of 16 rows) and K split by timing each candidate on the digits of a
// non-zero U
int i8_setup(tm_batch* bt) {
    const CtxView& v = bt->cv;
    const int b = v.bnx;
    hipStream_t s = bt->stream;
    bt->i8nT = (b + 15) / 16;
    bt->i8nC = (b + 63) / 64;
    const size_t nT = bt->i8nT, nC = bt->i8nC;
    TM_CHECK(bt->Bq.alloc(nT * nC * kI8Digits * kI8Op * 4));
    TM_CHECK(bt->Uq.alloc(nC * kI8DigitsU * 4 * kI8Op * 4));
    TM_CHECK(bt->i8rmax.alloc(b));
    TM_CHECK(bt->i8umax.alloc(64));
    TM_CHECK(bt->i8P.alloc((size_t)kI8MaxSplit * b * 64));
    TM_HIP(hipMemsetAsync(bt->i8rmax.p, 0, sizeof(double) * b, s));
    const int kper = 1024;
    hipLaunchKernelGGL(k_b_i8_rowmax, dim3((b + kBlock - 1) / kBlock, (b + kper - 1) / kper), dim3(kBlock), 0, s, b,
                       v.bld, v.B, kper, bt->i8rmax.p);
    hipLaunchKernelGGL(k_b_i8_bslice, dim3(elem_grid(nT * nC * 64)), dim3(kBlock), 0, s, b, v.bld, v.B, bt->i8nT,
                       bt->i8nC, (const double*)bt->i8rmax.p, reinterpret_cast<i32x4*>(bt->Bq.p));
    TM_HIP(hipGetLastError());
    // tuning operand: a non-zero pattern as the boundary values
    hipLaunchKernelGGL(k_b_fill_pattern, dim3(elem_grid((size_t)b * bt->S)), dim3(kBlock), 0, s, (size_t)b * bt->S,
                       bt->rhsN.p);
    TM_CHECK(i8_uslice(bt, nullptr, bt->rhsN.p));
    hipEvent_t e0, e1;
    TM_HIP(hipEventCreate(&e0));
    TM_HIP(hipEventCreate(&e1));
    // each candidate timed alone five times (the median counts), over two
    // rounds in which the clock has settled under the MFMA load; a single
    // launch's time varies by a few per cent
    struct Cand {
        int nw, ks;
        float ms;
        std::vector<float> t;
    };
    std::vector<Cand> cands;
    for (int nw = 4; nw <= 8; nw += 4)
        for (int ks : kI8Splits) {
            const int cper = i8_range(bt->i8nC, ks);
            if (ks > bt->i8nC || (size_t)cper * 64 > (size_t)kI8MaxK) continue;  // int32 bound per K range
            cands.push_back({nw, ks, 1e30f, {}});
        }
    const int cand = (int)cands.size();
    for (int round = 0; round < 2; ++round)
        for (Cand& c : cands)
            for (int r = 0; r < 5; ++r) {
                (void)hipEventRecord(e0, s);
                if (i8_gemm(bt, c.nw, c.ks) != TM_OK) break;
                (void)hipEventRecord(e1, s);
                if (hipEventSynchronize(e1) != hipSuccess) break;
                float ms = 0.0f;
                (void)hipEventElapsedTime(&ms, e0, e1);
                if (round == 1) c.t.push_back(ms);
            }
    (void)hipGetLastError();
    for (Cand& c : cands)
        if (!c.t.empty()) {
            std::sort(c.t.begin(), c.t.end());
            c.ms = c.t[c.t.size() / 2];
        }
    float best = 1e30f;
    for (const Cand& c : cands)
        if (c.ms < best) {
            best = c.ms;
            bt->i8nw = c.nw;
            bt->i8ks = c.ks;
        }
    if (cand > 0) bt->i8ms_first = cands[0].ms;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    bt->i8candidates = cand;
    bt->i8ms = best;
    if (cand == 0) return TM_ERR_UNSUPPORTED;  // K too long for one int32 range at any split
    TM_HIP(hipMemsetAsync(bt->rhsN.p, 0, sizeof(double) * (size_t)bt->n * bt->S, s));
    return TM_OK;
}

// out[bn[j]][s] = sum_k B[j][k] u[bn[k]][s] for every sample (bn null: the
// boundary values themselves, out[j][s] and u[k][s]), in the batch's
// precision (DemagField.cpp:145-147 for one vector).  Column-major G (b x S)
// = B (b x b, streamed in its storage order) * U^T, U = gathered boundary
// values (S x b).  FP64, except for TM_PREC_MIXED_BEM32: an FP32 copy of B,
// FP32 products accumulated in FP32 over 512-column chunks of B only, the
// chunk results summed in FP64 (FP32 accumulation over all 41k columns costs
// ~1e-5 relative field error).
int boundary_product(tm_batch* bt, const int* bn, const double* u, double* out) {
    const CtxView& v = bt->cv;
    const int b = v.bnx, S = bt->S;
    hipStream_t s = bt->stream;
    const dim3 g(elem_grid((size_t)b * S));
    if (bt->prec == TM_PREC_MIXED_BEMI8) {
        TM_CHECK(i8_product(bt, bn, u, out));
    } else if (bt->prec == TM_PREC_MIXED_BEM32) {
        hipLaunchKernelGGL(k_b_gather<float>, g, dim3(kBlock), 0, s, b, S, bn, u, bt->Uf.p);
        bt->live_mark(0);
        TM_CHECK(gemm_split_f32(bt));
        bt->live_mark(1);
        hipLaunchKernelGGL(k_b_chunk_sum, g, dim3(kBlock), 0, s, b, S, bt->nchunk, bn, (const float*)bt->Pf.p, out);
    } else {
        hipLaunchKernelGGL(k_b_gather<double>, g, dim3(kBlock), 0, s, b, S, bn, u, bt->U.p);
        if (bt->gemm_own) {
            bt->live_mark(0);
            TM_CHECK(gemm_own_run(bt, nullptr));
            bt->live_mark(1);
            hipLaunchKernelGGL(k_b_ksum_scatter, g, dim3(kBlock), 0, s, b, S, bt->gemm_ks, bn,
                               (const double*)bt->Pd.p, out);
        } else {
            bt->live_mark(0);
            TM_CHECK(gemm_run(bt, bt->gemm_sol));
            bt->live_mark(1);
            hipLaunchKernelGGL(k_b_scatter<double>, g, dim3(kBlock), 0, s, b, S, bn, (const double*)bt->Gm.p, out);
        }
    }
    TM_HIP(hipGetLastError());
    return TM_OK;
}

// b = div(Js m) of every sample into the Neumann right-hand side
void launch_div(tm_batch* bt) {
    const int n = bt->n, S = bt->S;
    if (bt->et.nt > 0) {
        const TileArgs t = bt->et.args(bt->eo);
        if (S % 2 == 0)
            hipLaunchKernelGGL(k_b_div<true>, dim3(tile_blocks(t.nch, kDivPerCu)), dim3(kTileThreads), 0, bt->stream, t,
                               (const double*)bt->tx.p, (const double*)bt->ty.p, (const double*)bt->tz.p, n,
                               (const double*)bt->m.p, bt->rhsN.p);
        else
            hipLaunchKernelGGL(k_b_div<false>, dim3(tile_blocks(t.nch, kDivPerCu)), dim3(kTileThreads), 0, bt->stream, t,
                               (const double*)bt->tx.p, (const double*)bt->ty.p, (const double*)bt->tz.p, n,
                               (const double*)bt->m.p, bt->rhsN.p);
        return;
    }
    hipLaunchKernelGGL(k_b_div_l2, dim3(row_grid(n)), dim3(kBlock), 0, bt->stream, bt->eo.args(8, bt->tx.p),
                       (const double*)bt->ty.p, (const double*)bt->tz.p, S, (const double*)bt->m.p, bt->rhsN.p);
}

// The fused field + LLG kernel of every (node, sample) on the batch
// magnetisation and the potentials in usum (TheLLG.cpp:238-254,
// EffFieldGPU.cu:316-362); with torque, the per-sample maximum torque too.
int launch_fields(tm_batch* bt, double alpha, int variant, double* dmdt, double* heff, bool torque,
                  double* mnext = nullptr, double dt = 0.0) {
    const CtxView& v = bt->cv;
    const int n = bt->n, S = bt->S;
    hipStream_t s = bt->stream;
    BEvalArgs a = {};
    a.P = bt->eo.args(8, bt->exch ? bt->xw.p : nullptr);
    a.gx = bt->gx.p;
    a.gy = bt->gy.p;
    a.gz = bt->gz.p;
    if (bt->dmi) {
        a.cx = bt->cx.p;
        a.cy = bt->cy.p;
        a.cz = bt->cz.p;
        a.dmi_fac = v.dmi_fac;
        a.nvs = v.nvs;
    }
    a.S = S;
    a.n = n;
    a.m = bt->m.p;
    a.u = bt->usum.p;
    a.invjs = v.invjs;
    a.ku = v.has_ku ? v.ku : nullptr;
    a.kaxis = v.has_ku ? v.kaxis : nullptr;
    a.hext = bt->hext.p;
    a.hfield = ctx_hext_field(bt->ctx);  // read per call: tm_ctx_set_zeeman may change it after creation
    a.alpha = alpha;
    a.variant = variant;
    a.dmdt = dmdt;
    a.heff = heff;
    a.torque = torque ? bt->torque.p : nullptr;
    a.mnext = mnext;
    a.dt = dt;
    if (torque) hipLaunchKernelGGL(k_b_zero_small, dim3(1), dim3(kMaxS), 0, s, S, bt->torque.p);
    const dim3 g(row_grid(n));
    if (bt->et.nt > 0) {
        const TileArgs t = bt->et.args(bt->eo);
        const dim3 tg(tile_blocks(t.nch, kEvalPerCu)), tb(kTileThreads);
        if (S % 2 == 0) {
            if (bt->dmi) hipLaunchKernelGGL((k_b_eval_t<true, true>), tg, tb, 0, s, a, (const double*)bt->xw.p, t);
            else hipLaunchKernelGGL((k_b_eval_t<false, true>), tg, tb, 0, s, a, (const double*)bt->xw.p, t);
        } else {
            if (bt->dmi) hipLaunchKernelGGL((k_b_eval_t<true, false>), tg, tb, 0, s, a, (const double*)bt->xw.p, t);
            else hipLaunchKernelGGL((k_b_eval_t<false, false>), tg, tb, 0, s, a, (const double*)bt->xw.p, t);
        }
    } else if (S == kMaxS) {
        if (bt->dmi) hipLaunchKernelGGL(k_b_eval_w<true>, g, dim3(kBlock), 0, s, a);
        else hipLaunchKernelGGL(k_b_eval_w<false>, g, dim3(kBlock), 0, s, a);
    } else if (bt->dmi) {
        hipLaunchKernelGGL(k_b_eval<true>, g, dim3(kBlock), 0, s, a);
    } else {
        hipLaunchKernelGGL(k_b_eval<false>, g, dim3(kBlock), 0, s, a);
    }
    TM_HIP(hipGetLastError());
    return TM_OK;
}

// One evaluation of the batch magnetisation into dmdt with fixed-budget
// solves (bt->bud_*): no host synchronisation, so it can be captured in a
// HIP graph.  Samples whose solve missed the tolerance are counted into
// bt->rk_fail on the device.
int eval_enqueue(tm_batch* bt, double alpha, int variant, double* dmdt) {
    const int n = bt->n, S = bt->S;
    const size_t NS = (size_t)n * S;
    hipStream_t s = bt->stream;
    const CtxView& v = bt->cv;
    constexpr int kMaxBud = tm_batch::kMaxBud;
    unsigned *fail = bt->rk_fail.p, *bad = fail + 1;
    int* track = reinterpret_cast<int*>(fail + 2);
    launch_div(bt);
    TM_HIP(hipGetLastError());
    if (bt->prec == TM_PREC_FP64)
        TM_CHECK(bt->sN64.enqueue(bt->rhsN.p, bt->u1.p, v.tol, bt->bud_outer[0], bt->bud_inner[0], s, fail, bad, track));
    else
        TM_CHECK(bt->sN32.enqueue(bt->rhsN.p, bt->u1.p, v.tol, bt->bud_outer[0], bt->bud_inner[0], s, fail, bad, track));
    TM_CHECK(boundary_product(bt, v.bnodes, bt->u1.p, bt->rhsD.p));
    if (bt->prec == TM_PREC_FP64)
        TM_CHECK(bt->sD64.enqueue(bt->rhsD.p, bt->u2.p, v.tol, bt->bud_outer[1], bt->bud_inner[1], s, fail, bad,
                                  track + kMaxBud));
    else
        TM_CHECK(bt->sD32.enqueue(bt->rhsD.p, bt->u2.p, v.tol, bt->bud_outer[1], bt->bud_inner[1], s, fail, bad,
                                  track + kMaxBud));
    hipLaunchKernelGGL(k_b_sum2, dim3(elem_grid(NS)), dim3(kBlock), 0, s, NS, (const double*)bt->u1.p,
                       (const double*)bt->u2.p, bt->usum.p);
    return launch_fields(bt, alpha, variant, dmdt, nullptr, false);
}

}  // namespace

namespace {

// f()'s status; no exception (out of memory) leaves it
template <class F>
int guarded(F&& f) {
    try {
        return f();
    } catch (const std::exception& e) {
        std::fprintf(stderr, "tetmag_hip: %s\n", e.what());
        return TM_ERR_HIP;
    }
}

// f on another thread with the caller's device; where none can be started, on
// this one when its status is asked for
template <class F>
std::future<int> beside(F f) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    auto run = [f, dev] {
        if (hipSetDevice(dev) != hipSuccess) return (int)TM_ERR_HIP;
        return guarded(f);
    };
    try {
        return std::async(std::launch::async, run);
    } catch (const std::exception&) {
        return std::async(std::launch::deferred, run);
    }
}

}  // namespace

extern "C" {

int tm_batch_create(tm_ctx* c, int nsamples, int precision, tm_batch** out) {
    if (!c || !out || nsamples < 1 || nsamples > kMaxS) return TM_ERR_BAD_ARG;
    if (precision != TM_PREC_FP64 && precision != TM_PREC_MIXED && precision != TM_PREC_MIXED_BEM32 &&
        precision != TM_PREC_MIXED_BEMI8)
        return TM_ERR_BAD_ARG;
    tm_batch* bt = new tm_batch();
    int st = ctx_view(c, &bt->cv);
    if (st != TM_OK) {
        delete bt;
        return st;
    }
    const CtxView& v = bt->cv;
    if (!v.cgN || !v.cgD || !v.B || !v.js || !v.hop_set[TM_OP_GRAD_X] || !v.hop_set[TM_OP_TGRAD_X]) {
        delete bt;
        return TM_ERR_NOT_READY;
    }
    // the batched kernels cover exchange, uniaxial, bulk DMI, Zeeman and
    // demag; interfacial DMI contexts are evaluated per sample
    if (v.cgN->precond != TM_PRECOND_AMG || v.cgD->precond != TM_PRECOND_AMG || v.has_idmi) {
        delete bt;
        return TM_ERR_UNSUPPORTED;
    }
    bt->ctx = c;
    bt->n = v.n;
    bt->S = nsamples;
    bt->prec = precision;
    bt->stream = v.stream;
    auto fail = [&](int s) {
        tm_batch_destroy(bt);
        return s;
    };
    if (rocblas_create_handle(&bt->blas) != rocblas_status_success) return fail(TM_ERR_HIP);
    rocblas_set_stream(bt->blas, bt->stream);
    const SellPattern& P = *v.pat;
    // the field kernels address the three components of m and the potentials
    // with 32-bit byte offsets
    if ((int64_t)3 * P.n * nsamples * 8 > (int64_t)INT32_MAX) return fail(TM_ERR_UNSUPPORTED);
    if ((st = bt->eo.build(P.n, P.n, P.h_rowptr.data(), P.h_csrcol.data(), nsamples, bt->stream)) != TM_OK)
        return fail(st);
    bt->exch = v.hop_set[TM_OP_EXCHANGE];
    int ops_ok = TM_OK;
    if (bt->exch) ops_ok |= upload_op(bt, TM_OP_EXCHANGE, bt->xw);
    ops_ok |= upload_op(bt, TM_OP_GRAD_X, bt->gx);
    ops_ok |= upload_op(bt, TM_OP_GRAD_Y, bt->gy);
    ops_ok |= upload_op(bt, TM_OP_GRAD_Z, bt->gz);
    {  // the divergence weights carry Js of their column and 1/mu0 (the Js of the context now)
        std::vector<double> jsh((size_t)P.n);
        if (hipMemcpyAsync(jsh.data(), v.js, sizeof(double) * P.n, hipMemcpyDeviceToHost, bt->stream) != hipSuccess ||
            hipStreamSynchronize(bt->stream) != hipSuccess)
            return fail(TM_ERR_HIP);
        ops_ok |= upload_op(bt, TM_OP_TGRAD_X, bt->tx, jsh.data(), 1.0 / kMu0);
        ops_ok |= upload_op(bt, TM_OP_TGRAD_Y, bt->ty, jsh.data(), 1.0 / kMu0);
        ops_ok |= upload_op(bt, TM_OP_TGRAD_Z, bt->tz, jsh.data(), 1.0 / kMu0);
    }
    bt->dmi = v.has_dmi && v.hop_set[TM_OP_CURL_X] && v.hop_set[TM_OP_CURL_Y] && v.hop_set[TM_OP_CURL_Z];
    if (bt->dmi) {
        ops_ok |= upload_op(bt, TM_OP_CURL_X, bt->cx);
        ops_ok |= upload_op(bt, TM_OP_CURL_Y, bt->cy);
        ops_ok |= upload_op(bt, TM_OP_CURL_Z, bt->cz);
    }
    if (ops_ok != TM_OK) return fail(TM_ERR_BAD_ARG);
    const size_t NS = (size_t)bt->n * nsamples;
    int a = TM_OK;
    a |= bt->m.alloc(3 * NS);
    a |= bt->dmdt.alloc(3 * NS);
    a |= bt->heff.alloc(3 * NS);
    a |= bt->u1.alloc(NS);
    a |= bt->u2.alloc(NS);
    a |= bt->usum.alloc(NS);
    a |= bt->rhsN.alloc(NS);
    a |= bt->rhsD.alloc(NS);
    if (precision == TM_PREC_MIXED_BEM32) {
        bt->nchunk = (v.bnx + bt->kchunk - 1) / bt->kchunk;
        a |= bt->Uf.alloc((size_t)v.bnx * nsamples);
        a |= bt->Gf.alloc((size_t)v.bnx * nsamples);
        a |= bt->Bf.alloc((size_t)v.bld * v.bnx);
        a |= bt->Pf.alloc((size_t)bt->nchunk * v.bnx * nsamples);
    } else if (precision != TM_PREC_MIXED_BEMI8) {
        a |= bt->U.alloc((size_t)v.bnx * nsamples);
        a |= bt->Gm.alloc((size_t)v.bnx * nsamples);
    }
    a |= bt->hext.alloc((size_t)3 * nsamples);
    a |= bt->torque.alloc(nsamples);
    if (a != TM_OK) return fail(TM_ERR_HIP);
    if (precision == TM_PREC_MIXED_BEM32) {
        const size_t tot = (size_t)v.bld * v.bnx;
        hipLaunchKernelGGL(k_b_to_float, dim3(elem_grid(tot)), dim3(kBlock), 0, bt->stream, tot, v.B, bt->Bf.p);
        if (hipGetLastError() != hipSuccess) return fail(TM_ERR_HIP);
    }
    (void)hipMemsetAsync(bt->u1.p, 0, NS * sizeof(double), bt->stream);
    (void)hipMemsetAsync(bt->u2.p, 0, NS * sizeof(double), bt->stream);
    (void)hipMemsetAsync(bt->rhsD.p, 0, NS * sizeof(double), bt->stream);
    (void)hipMemsetAsync(bt->m.p, 0, 3 * NS * sizeof(double), bt->stream);
    std::vector<double> h((size_t)3 * nsamples);
    for (int s = 0; s < nsamples; ++s)
        for (int d = 0; d < 3; ++d) h[(size_t)d * nsamples + s] = v.hext[d];
    if ((st = bt->hext.upload(h.data(), h.size(), bt->stream)) != TM_OK) return fail(st);
    // Tiles, slot lists and operators of the two solvers and of the fields: host
    // work that does not depend on each other, side by side.  282,897 nodes, 64
    // samples: one after the other 0.87 s of the 1.28 s that a batch takes to make.
    {
        std::future<int> neumann, dirichlet;
        if (precision == TM_PREC_FP64) {
            neumann = beside([&] { return bt->sN64.setup(*v.cgN, nsamples, bt->stream); });
            dirichlet = beside([&] { return bt->sD64.setup(*v.cgD, nsamples, bt->stream); });
        } else {
            neumann = beside([&] { return bt->sN32.setup(*v.cgN, nsamples, bt->stream); });
            dirichlet = beside([&] { return bt->sD32.setup(*v.cgD, nsamples, bt->stream); });
        }
        const int se = guarded([&] { return bt->et.build(bt->eo, bt->stream); });
        const int sn = neumann.get(), sd = dirichlet.get();  // before bt may go
        if ((st = se) != TM_OK || (st = sn) != TM_OK || (st = sd) != TM_OK) return fail(st);
    }
    if (!bt->exch && bt->et.nt > 0) {
        const std::vector<double> zeros((size_t)bt->eo.h_sp[P.n], 0.0);
        if ((st = bt->xw.upload(zeros.data(), zeros.size(), bt->stream)) != TM_OK) return fail(st);
        if (hipStreamSynchronize(bt->stream) != hipSuccess) return fail(TM_ERR_HIP);
    }
    // the Dirichlet right-hand side is zero off the boundary nodes (Laplace,
    // no source; the boundary product scatters into those rows only)
    bt->sD64.rhs_rows = bt->sD32.rhs_rows = v.bnodes;
    bt->sD64.rhs_nrows = bt->sD32.rhs_nrows = v.bnx;
    bt->sN64.win_stride = bt->sN32.win_stride = 8;
    bt->sD64.win_stride = bt->sD32.win_stride = 4;
    if (hipStreamSynchronize(bt->stream) != hipSuccess) return fail(TM_ERR_HIP);
    if (precision == TM_PREC_MIXED_BEMI8) {
        if ((st = i8_setup(bt)) != TM_OK) return fail(st);
    } else if ((st = tune_gemm(bt)) != TM_OK) {
        return fail(st);
    }
    if (hipStreamSynchronize(bt->stream) != hipSuccess) return fail(TM_ERR_HIP);
    *out = bt;
    return TM_OK;
}

int tm_batch_destroy(tm_batch* bt) {
    if (!bt) return TM_OK;
    if (bt->stream) (void)hipStreamSynchronize(bt->stream);
    bt->drop_step();
    if (bt->blas) rocblas_destroy_handle(bt->blas);
    for (auto& e : bt->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto& e : bt->lev)
        if (e) (void)hipEventDestroy(e);
    delete bt;
    return TM_OK;
}

int tm_batch_set_zeeman(tm_batch* bt, const double* h3s) {
    if (!bt || !h3s) return TM_ERR_BAD_ARG;
    TM_CHECK(bt->hext.upload(h3s, (size_t)3 * bt->S, bt->stream));
    TM_HIP(hipStreamSynchronize(bt->stream));
    return TM_OK;
}

int tm_batch_set_mag(tm_batch* bt, const double* m, int where) {
    if (!bt) return TM_ERR_BAD_ARG;
    bt->m_replaced = true;
    return copy_in(bt->m.p, m, where, (size_t)3 * bt->n * bt->S, bt->stream);
}

int tm_batch_get_mag(tm_batch* bt, double* m, int where) {
    if (!bt) return TM_ERR_BAD_ARG;
    return copy_out(m, where, bt->m.p, (size_t)3 * bt->n * bt->S, bt->stream);
}

int tm_batch_get_potentials(tm_batch* bt, double* u1, double* u2, int where) {
    if (!bt) return TM_ERR_BAD_ARG;
    const size_t NS = (size_t)bt->n * bt->S;
    if (u1) TM_CHECK(copy_out(u1, where, bt->u1.p, NS, bt->stream));
    if (u2) TM_CHECK(copy_out(u2, where, bt->u2.p, NS, bt->stream));
    return TM_OK;
}

int tm_batch_enable_timers(tm_batch* bt, int on) {
    if (!bt) return TM_ERR_BAD_ARG;
    if (on && !bt->ev[0])
        for (auto& e : bt->ev) TM_HIP(hipEventCreate(&e));
    bt->timers = on != 0;
    return TM_OK;
}

int tm_batch_gemm_live(tm_batch* bt, int on, double* ms_mean, int* count) {
    if (!bt || (on != 0 && on != 1)) return TM_ERR_BAD_ARG;
    if (on) {
        if (!bt->lev[0])
            for (auto& e : bt->lev) TM_HIP(hipEventCreate(&e));
        bt->lev_n = 0;
        bt->lev_on = true;
        return TM_OK;
    }
    bt->lev_on = false;
    double sum = 0.0;
    if (bt->lev_n > 0) TM_HIP(hipEventSynchronize(bt->lev[2 * bt->lev_n - 1]));
    for (int k = 0; k < bt->lev_n; ++k) {
        float ms = 0.0f;
        TM_HIP(hipEventElapsedTime(&ms, bt->lev[2 * k], bt->lev[2 * k + 1]));
        sum += ms;
    }
    if (ms_mean) *ms_mean = bt->lev_n > 0 ? sum / bt->lev_n : 0.0;
    if (count) *count = bt->lev_n;
    return TM_OK;
}

int tm_batch_get_timers(tm_batch* bt, tm_phase_times* out, int reset) {
    if (!bt || !out) return TM_ERR_BAD_ARG;
    *out = bt->tsum;
    if (reset) bt->tsum = tm_phase_times{};
    return TM_OK;
}

}  // extern "C"

namespace {

// Statuses after which every sample has its result: some may have missed the
// tolerance, some may not be finite (the others are as without them).
bool solved(int st) { return st == TM_OK || st == TM_ERR_MAXITER || st == TM_ERR_NONFINITE; }
int worse(int a, int b) {
    if (a == TM_ERR_NONFINITE || b == TM_ERR_NONFINITE) return TM_ERR_NONFINITE;
    return a != TM_OK ? a : b;
}

// tm_batch_eval_rhs; with euler_dt > 0 the field kernel also writes the
// Euler step of m into m2, which then becomes the batch's m
int batch_eval(tm_batch* bt, const double* m, int mwhere, double alpha, int variant, double* dmdt, int dwhere,
               double* heff, int hwhere, tm_batch_stats* stats, double euler_dt) {
    if (!bt || !dmdt || (variant != TM_LLG_CLASSIC && variant != TM_LLG_NOPREC)) return TM_ERR_BAD_ARG;
    if ((dwhere != TM_HOST && dwhere != TM_DEVICE) || (heff && hwhere != TM_HOST && hwhere != TM_DEVICE))
        return TM_ERR_BAD_ARG;
    const int n = bt->n, S = bt->S;
    const size_t NS = (size_t)n * S;
    hipStream_t s = bt->stream;
    const CtxView& v = bt->cv;
    if (m) {
        bt->m_replaced = true;
        TM_CHECK(copy_in(bt->m.p, m, mwhere, 3 * NS, s));
    }
    if (bt->timers) TM_HIP(hipEventRecord(bt->ev[0], s));
    // Poisson right-hand side (DemagField.cpp:124-136), all samples
    launch_div(bt);
    TM_HIP(hipGetLastError());
    if (bt->timers) TM_HIP(hipEventRecord(bt->ev[1], s));
    int oN = 0, iN = 0, oD = 0, iD = 0;
    double rN = 0, rD = 0;
    int stN = bt->prec == TM_PREC_FP64 ? bt->sN64.solve(bt->rhsN.p, bt->u1.p, v.tol, v.maxit, s, &oN, &iN, &rN)
                                       : bt->sN32.solve(bt->rhsN.p, bt->u1.p, v.tol, v.maxit, s, &oN, &iN, &rN);
    if (!solved(stN)) return stN;
    if (bt->timers) TM_HIP(hipEventRecord(bt->ev[2], s));
    // boundary integral (DemagField.cpp:184-201) as a GEMM: G = B U^T, U the
    // gathered boundary potentials of every sample
    TM_CHECK(boundary_product(bt, v.bnodes, bt->u1.p, bt->rhsD.p));
    if (bt->timers) TM_HIP(hipEventRecord(bt->ev[3], s));
    int stD = bt->prec == TM_PREC_FP64 ? bt->sD64.solve(bt->rhsD.p, bt->u2.p, v.tol, v.maxit, s, &oD, &iD, &rD)
                                       : bt->sD32.solve(bt->rhsD.p, bt->u2.p, v.tol, v.maxit, s, &oD, &iD, &rD);
    if (!solved(stD)) return stD;
    if (bt->timers) TM_HIP(hipEventRecord(bt->ev[4], s));
    // total potential, gathered once per entry by the field kernel
    hipLaunchKernelGGL(k_b_sum2, dim3(elem_grid(NS)), dim3(kBlock), 0, s, NS, (const double*)bt->u1.p,
                       (const double*)bt->u2.p, bt->usum.p);
    // fused fields + LLG
    double* dout = dwhere == TM_DEVICE ? dmdt : bt->dmdt.p;
    double* hout = heff ? (hwhere == TM_DEVICE ? heff : bt->heff.p) : nullptr;
    if (euler_dt > 0.0) TM_CHECK(bt->m2.alloc(3 * NS));
    TM_CHECK(launch_fields(bt, alpha, variant, dout, hout, stats != nullptr, euler_dt > 0.0 ? bt->m2.p : nullptr,
                           euler_dt));
    if (euler_dt > 0.0) std::swap(bt->m, bt->m2);
    if (bt->timers) {
        TM_HIP(hipEventRecord(bt->ev[5], s));
        TM_HIP(hipEventSynchronize(bt->ev[5]));
        float t[5];
        for (int k = 0; k < 5; ++k) TM_HIP(hipEventElapsedTime(&t[k], bt->ev[k], bt->ev[k + 1]));
        bt->tsum.div_ms += t[0];
        bt->tsum.neumann_ms += t[1];
        bt->tsum.bem_ms += t[2];
        bt->tsum.dirichlet_ms += t[3];
        bt->tsum.fields_ms += t[4];
        bt->tsum.iters_neumann += iN;
        bt->tsum.iters_dirichlet += iD;
        bt->tsum.count += 1;
    }
    if (dwhere == TM_HOST) TM_CHECK(copy_out(dmdt, TM_HOST, dout, 3 * NS, s));
    if (heff && hwhere == TM_HOST) TM_CHECK(copy_out(heff, TM_HOST, hout, 3 * NS, s));
    if (stats) {
        stats->outer_neumann = oN;
        stats->outer_dirichlet = oD;
        stats->inner_neumann = iN;
        stats->inner_dirichlet = iD;
        stats->max_relres_neumann = rN;
        stats->max_relres_dirichlet = rD;
        stats->nsamples = S;
        TM_HIP(hipMemcpyAsync(stats->max_torque, bt->torque.p, sizeof(double) * S, hipMemcpyDeviceToHost, s));
        TM_HIP(hipStreamSynchronize(s));
    }
    return worse(stN, stD);
}

}  // namespace

extern "C" {

int tm_batch_eval_rhs(tm_batch* bt, const double* m, int mwhere, double alpha, int variant, double* dmdt, int dwhere,
                      double* heff, int hwhere, tm_batch_stats* stats) {
    return batch_eval(bt, m, mwhere, alpha, variant, dmdt, dwhere, heff, hwhere, stats, 0.0);
}

int tm_batch_eval_euler(tm_batch* bt, double alpha, int variant, double dtau, double* dmdt, int dwhere,
                        tm_batch_stats* stats) {
    if (!(dtau > 0.0)) return TM_ERR_BAD_ARG;
    return batch_eval(bt, nullptr, TM_DEVICE, alpha, variant, dmdt, dwhere, nullptr, TM_DEVICE, stats, dtau);
}

int tm_batch_run_rk4(tm_batch* bt, double dtau, int nsteps, double alpha, int variant, int use_graph,
                     tm_batch_stats* last, tm_rk4_stats* rk) {
    if (!bt || nsteps < 0 || !(dtau > 0.0) || (variant != TM_LLG_CLASSIC && variant != TM_LLG_NOPREC))
        return TM_ERR_BAD_ARG;
    const size_t NS = (size_t)bt->n * bt->S, N3 = 3 * NS;
    for (auto& k : bt->rk_k) TM_CHECK(k.alloc(N3));
    TM_CHECK(bt->rk_base.alloc(N3));
    constexpr int kMaxBud = tm_batch::kMaxBud, kCount = tm_batch::kCounts;
    TM_CHECK(bt->rk_fail.alloc(kCount));
    hipStream_t s = bt->stream;
    const dim3 g(elem_grid(N3));
    const double cst[4] = {0.0, 0.5 * dtau, 0.5 * dtau, dtau};
    // graphs need kernel-only boundary products (the own GEMMs): from int8 digits
    // for any number of samples, in FP64 for 64; other batches run every step
    // host-polled.  (The FP64 kernel takes fewer samples too, and captured steps
    // with it measured faster: 7 samples at 2,205 nodes 1.29 against 1.46 ms a
    // step, 24 at 38,440 4.31 against 4.93.  Not set up: own_ok asks for 64.)
    const bool graph_ok =
        use_graph && (bt->prec == TM_PREC_MIXED_BEMI8 || (bt->prec != TM_PREC_MIXED_BEM32 && bt->own_ok));
    tm_rk4_stats R = {};
    hipEvent_t e0 = nullptr, e1 = nullptr;
    TM_HIP(hipEventCreate(&e0));
    TM_HIP(hipEventCreate(&e1));
    TM_HIP(hipEventRecord(e0, s));
    // Budgets from the last host-polled solves, one iteration per refinement
    // step more than they took.  Only a step's last stage sets them: the first
    // solves of a run start cold and take several times the iterations of
    // the later ones, and a queued iteration past convergence costs its dozen
    // launches.  After a miss (grow) every stage counts, and no budget shrinks.
    auto learn = [bt](bool grow) {
        constexpr int kMaxBud = tm_batch::kMaxBud;
        const bool f64 = bt->prec == TM_PREC_FP64;
        const int o[2] = {f64 ? bt->sN64.last_outer : bt->sN32.last_outer,
                          f64 ? bt->sD64.last_outer : bt->sD32.last_outer};
        const int* in[2] = {f64 ? bt->sN64.last_inner : bt->sN32.last_inner,
                            f64 ? bt->sD64.last_inner : bt->sD32.last_inner};
        for (int w = 0; w < 2; ++w) {
            const int had = grow ? bt->bud_outer[w] : 0;
            bt->bud_outer[w] = std::min(kMaxBud, std::max(std::max(1, o[w]), had));
            for (int k = 0; k < bt->bud_outer[w]; ++k) {
                const int now = k < o[w] ? in[w][k] + (grow ? 2 : 1) : 1;
                bt->bud_inner[w][k] = k < had ? std::max(bt->bud_inner[w][k], now) : now;
            }
        }
        bt->bud_set = true;
    };
    // What the replays needed since the last tightening: the budgets shrink to
    // it, plus one, at the end of a call and after eight replays.
    int seen[2 * kMaxBud] = {}, replays = 0;
    auto tighten = [&]() {
        constexpr int kMaxBud = tm_batch::kMaxBud;
        for (int w = 0; w < 2 && replays > 0; ++w) {
            int used = 0;
            for (int k = 0; k < bt->bud_outer[w]; ++k) {
                if (seen[w * kMaxBud + k] > 0) used = k + 1;
                bt->bud_inner[w][k] = std::min(bt->bud_inner[w][k], seen[w * kMaxBud + k] + 1);
            }
            bt->bud_outer[w] = std::max(1, used);
        }
        replays = 0;
        std::fill(seen, seen + 2 * kMaxBud, 0);
    };
    auto polled_step = [&](bool final_step, bool missed) -> int {
        int st = TM_OK;
        hipLaunchKernelGGL(k_b_copy, g, dim3(kBlock), 0, s, N3, (const double*)bt->m.p, bt->rk_base.p);
        for (int k = 0; k < 4; ++k) {
            if (k > 0)
                hipLaunchKernelGGL(k_b_axpy, g, dim3(kBlock), 0, s, N3, (const double*)bt->rk_base.p,
                                   (const double*)bt->rk_k[k - 1].p, cst[k], bt->m.p);
            tm_batch_stats es = {};
            const bool fin = final_step && k == 3;
            const int r = tm_batch_eval_rhs(bt, nullptr, TM_DEVICE, alpha, variant, bt->rk_k[k].p, TM_DEVICE, nullptr,
                                            TM_DEVICE, &es);
            if (!solved(r)) return r;
            st = worse(st, r);
            R.max_iters_neumann = std::max(R.max_iters_neumann, es.inner_neumann);
            R.max_iters_dirichlet = std::max(R.max_iters_dirichlet, es.inner_dirichlet);
            if (fin && last) *last = es;
            if (missed || k == 3) learn(missed);
        }
        hipLaunchKernelGGL(k_b_rk_final, dim3(elem_grid(NS)), dim3(kBlock), 0, s, NS, (const double*)bt->rk_base.p,
                           (const double*)bt->rk_k[0].p, (const double*)bt->rk_k[1].p, (const double*)bt->rk_k[2].p,
                           (const double*)bt->rk_k[3].p, dtau, bt->m.p);
        TM_HIP(hipGetLastError());
        R.sync_steps += 1;
        bt->m_replaced = false;
        return st;
    };
    int status = TM_OK;
    if (last) *last = tm_batch_stats{};
    for (int step = 0; step < nsteps; ++step) {
        const bool fin = step == nsteps - 1;
        bool missed = false;
        // A state from outside has nothing to do with the kept solutions or the
        // budgets: its first step is host-polled (a replay would run to its end,
        // miss the tolerance and be redone)
        if (graph_ok && bt->bud_set && !bt->m_replaced) {
            if (replays >= 8) tighten();
            tm_batch::StepKey key;
            key.dtau = dtau;
            key.alpha = alpha;
            key.variant = variant;
            key.m = bt->m.p;
            key.hfield = ctx_hext_field(bt->ctx);
            for (int w = 0; w < 2; ++w) {
                key.outer[w] = bt->bud_outer[w];
                for (int k = 0; k < kMaxBud; ++k) key.inner[w][k] = bt->bud_inner[w][k];
            }
            if (!bt->step_exec || !(key == bt->step_key)) {
                bt->drop_step();
                hipGraph_t gr = nullptr;
                // the captured boundary products use the fastest verified own kernel
                const bool k_own = bt->gemm_own;
                const int k_shape = bt->gemm_shape, k_ks = bt->gemm_ks;
                bt->gemm_own = true;
                bt->gemm_shape = bt->own_shape;
                bt->gemm_ks = bt->own_ks;
                TM_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
                bt->capturing = true;
                int r = TM_OK;
                hipLaunchKernelGGL(k_b_reset_fail, dim3(1), dim3(64), 0, s, kCount, bt->rk_fail.p);
                hipLaunchKernelGGL(k_b_copy, g, dim3(kBlock), 0, s, N3, (const double*)bt->m.p, bt->rk_base.p);
                for (int k = 0; k < 4 && r == TM_OK; ++k) {
                    if (k > 0)
                        hipLaunchKernelGGL(k_b_axpy, g, dim3(kBlock), 0, s, N3, (const double*)bt->rk_base.p,
                                           (const double*)bt->rk_k[k - 1].p, cst[k], bt->m.p);
                    r = eval_enqueue(bt, alpha, variant, bt->rk_k[k].p);
                }
                hipLaunchKernelGGL(k_b_rk_final, dim3(elem_grid(NS)), dim3(kBlock), 0, s, NS,
                                   (const double*)bt->rk_base.p, (const double*)bt->rk_k[0].p,
                                   (const double*)bt->rk_k[1].p, (const double*)bt->rk_k[2].p,
                                   (const double*)bt->rk_k[3].p, dtau, bt->m.p);
                const hipError_t ec = hipStreamEndCapture(s, &gr);
                bt->capturing = false;
                bt->gemm_own = k_own;
                bt->gemm_shape = k_shape;
                bt->gemm_ks = k_ks;
                if (r != TM_OK || ec != hipSuccess) {
                    if (gr) (void)hipGraphDestroy(gr);
                    status = r != TM_OK ? r : TM_ERR_HIP;
                    break;
                }
                const hipError_t ei = hipGraphInstantiate(&bt->step_exec, gr, nullptr, nullptr, 0);
                (void)hipGraphDestroy(gr);
                if (ei != hipSuccess) {
                    bt->step_exec = nullptr;
                    status = TM_ERR_HIP;
                    break;
                }
                bt->step_key = key;
                R.captures += 1;
            }
            unsigned counts[kCount] = {};
            if (hipGraphLaunch(bt->step_exec, s) != hipSuccess ||
                hipMemcpyAsync(counts, bt->rk_fail.p, sizeof(counts), hipMemcpyDeviceToHost, s) != hipSuccess ||
                hipStreamSynchronize(s) != hipSuccess) {
                status = TM_ERR_HIP;
                break;
            }
            for (int w = 0; w < 2; ++w) {
                const int* took = reinterpret_cast<const int*>(counts) + 2 + w * kMaxBud;
                int sum = 0;
                for (int k = 0; k < kMaxBud; ++k) sum += took[k];
                (w == 0 ? R.max_iters_neumann : R.max_iters_dirichlet) =
                    std::max(w == 0 ? R.max_iters_neumann : R.max_iters_dirichlet, sum);
                for (int k = 0; k < kMaxBud; ++k)
                    seen[w * kMaxBud + k] = std::max(seen[w * kMaxBud + k], took[k]);
            }
            ++replays;
            if (counts[0] == 0) {  // (no redo for samples that are not finite: they would end the same way)
                R.graph_steps += 1;
                if (counts[1] != 0) status = TM_ERR_NONFINITE;
                if (fin && last) last->nsamples = bt->S;
                continue;
            }
            // a sample's solve missed its tolerance within the budgets: restore
            // the step's start state and redo it with host-polled solves
            hipLaunchKernelGGL(k_b_copy, g, dim3(kBlock), 0, s, N3, (const double*)bt->rk_base.p, bt->m.p);
            R.redone_steps += 1;
            missed = true;
            replays = 0;
            std::fill(seen, seen + 2 * kMaxBud, 0);
        }
        const int r = polled_step(fin, missed);
        if (!solved(r)) {
            status = r;
            break;
        }
        status = worse(status, r);
    }
    tighten();
    for (int w = 0; w < 2; ++w) {
        int tot = 0;
        for (int k = 0; k < bt->bud_outer[w]; ++k) tot += bt->bud_inner[w][k];
        (w == 0 ? R.budget_neumann : R.budget_dirichlet) = tot;
    }
    TM_HIP(hipEventRecord(e1, s));
    TM_HIP(hipEventSynchronize(e1));
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    R.ms = ms;
    if (rk) *rk = R;
    return status;
}

int tm_batch_gemm_info(tm_batch* bt, int* solution, int* own_kernel, int* candidates, double* ms_default,
                       double* ms_tuned, int* ksplit) {
    if (!bt) return TM_ERR_BAD_ARG;
    if (bt->prec == TM_PREC_MIXED_BEMI8) {  // k_b_gemm_i8: solution = wavefronts per block
        if (solution) *solution = bt->i8nw;
        if (own_kernel) *own_kernel = 1;
        if (candidates) *candidates = bt->i8candidates;
        if (ksplit) *ksplit = bt->i8ks;
        if (ms_default) *ms_default = bt->i8ms_first;
        if (ms_tuned) *ms_tuned = bt->i8ms;
        return TM_OK;
    }
    if (solution) *solution = bt->gemm_own ? bt->gemm_shape : bt->gemm_sol;
    if (own_kernel) *own_kernel = bt->gemm_own ? 1 : 0;
    if (candidates) *candidates = bt->gemm_candidates + bt->gemm_own_candidates;
    if (ksplit) *ksplit = bt->gemm_own ? bt->gemm_ks : 1;
    if (ms_default) *ms_default = bt->gemm_ms_default;
    if (ms_tuned) *ms_tuned = bt->gemm_ms_best;
    return TM_OK;
}

int tm_batch_time_kernels(tm_batch* bt, int reps, tm_batch_kernel_time* out, int cap, int* count) {
    if (!bt || reps < 1 || !out || cap < 1 || !count) return TM_ERR_BAD_ARG;
    hipStream_t s = bt->stream;
    const int n = bt->n, S = bt->S;
    const double nS = (double)n * S;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    TM_HIP(hipEventCreate(&e0));
    TM_HIP(hipEventCreate(&e1));
    int status = TM_OK;
    auto timeit = [&](auto&& launch) -> double {
        launch();  // warm-up
        if (hipEventRecord(e0, s) != hipSuccess) status = TM_ERR_HIP;
        for (int r = 0; r < reps; ++r) launch();
        if (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) status = TM_ERR_HIP;
        float ms = 0.0f;
        (void)hipEventElapsedTime(&ms, e0, e1);
        return (double)ms / reps;
    };
    std::vector<tm_batch_kernel_time> v;
    auto add = [&v](const char* nm, double ms, double bytes) {
        tm_batch_kernel_time k = {};
        std::snprintf(k.name, sizeof(k.name), "%s", nm);
        k.ms = ms;
        k.bytes = bytes;
        v.push_back(k);
    };
    const double eslots = (double)bt->eo.h_sp[n];
    add(bt->et.nt > 0 ? "k_b_div" : "k_b_div_l2", timeit([&] {
            launch_div(bt);
        }),
        eslots * (4 + 3 * 8) + 3 * nS * 8 + nS * 8);
    const int nw = (bt->exch ? 1 : 0) + 3 + (bt->dmi ? 3 : 0);
    const double per_node = 8.0 * n * (1 + (bt->cv.has_ku ? 4 : 0) + (bt->dmi ? 4 : 0));
    const std::string eval = std::string(bt->et.nt > 0 ? "k_b_eval_t" : S == kMaxS ? "k_b_eval_w" : "k_b_eval") +
                             (bt->dmi ? "<DMI>" : "");  // as launch_fields chooses
    add(eval.c_str(), timeit([&] {
            (void)launch_fields(bt, 0.5, TM_LLG_CLASSIC, bt->dmdt.p, nullptr, false);
        }),
        eslots * (4 + 8.0 * nw) + 3 * nS * 8 + nS * 8 + 3 * nS * 8 + per_node);
    // the boundary GEMM as the batch runs it (the tuned kernel, without the
    // gather and scatter); bytes: B once plus U and the product
    if (bt->prec == TM_PREC_MIXED_BEMI8) {
        // B's digit slices once, U's digits and the FP64 partials
        const double bytes = (double)bt->i8nT * bt->i8nC * kI8Digits * 1024.0 +
                             (double)bt->i8nC * kI8DigitsU * 4 * 1024.0 + 8.0 * bt->i8ks * bt->cv.bnx * 64.0;
        add("boundary GEMM (k_b_gemm_i8, int8 digits, tuned)", timeit([&] { (void)i8_gemm(bt, bt->i8nw, bt->i8ks); }),
            bytes);
    } else if (bt->prec != TM_PREC_MIXED_BEM32) {
        const double bb = (double)bt->cv.bnx;
        add(bt->gemm_own ? "boundary GEMM (k_b_gemm64, tuned)" : "boundary GEMM (rocBLAS, tuned)", timeit([&] {
                if (bt->gemm_own) (void)gemm_own_run(bt, nullptr);
                else (void)gemm_run(bt, bt->gemm_sol);
            }),
            8.0 * bb * bb + 2.0 * 8.0 * bb * S);
    }
    int st = bt->prec == TM_PREC_FP64 ? bt->sN64.time_kernels(s, timeit, v) : bt->sN32.time_kernels(s, timeit, v);
    if (status == TM_OK) status = st;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *count = 0;
    for (size_t k = 0; k < v.size() && (int)k < cap; ++k) out[(*count)++] = v[k];
    return status;
}

int tm_batch_bem_apply(tm_batch* bt, const double* x, int xwhere, double* y, int ywhere) {
    if (!bt || !x || !y || (xwhere != TM_HOST && xwhere != TM_DEVICE) || (ywhere != TM_HOST && ywhere != TM_DEVICE))
        return TM_ERR_BAD_ARG;
    const size_t bs = (size_t)bt->cv.bnx * bt->S;
    const double* xd = x;
    if (xwhere == TM_HOST) {  // staged in rhsN (n x S >= b x S)
        TM_CHECK(copy_in(bt->rhsN.p, x, TM_HOST, bs, bt->stream));
        xd = bt->rhsN.p;
    }
    // staged in usum (rewritten by every evaluation before it is read), not
    // in rhsD: the Dirichlet right-hand side must stay zero off the boundary
    double* yd = ywhere == TM_HOST ? bt->usum.p : y;
    TM_CHECK(boundary_product(bt, nullptr, xd, yd));
    if (ywhere == TM_HOST) TM_CHECK(copy_out(y, TM_HOST, yd, bs, bt->stream));
    return TM_OK;
}

int tm_batch_step_euler(tm_batch* bt, const double* dm, int where, double dtau) {
    if (!bt) return TM_ERR_BAD_ARG;
    const size_t NS = (size_t)bt->n * bt->S;
    const double* dd = dm;
    if (where == TM_HOST) {
        TM_CHECK(copy_in(bt->heff.p, dm, TM_HOST, 3 * NS, bt->stream));
        dd = bt->heff.p;
    } else if (where != TM_DEVICE) {
        return TM_ERR_BAD_ARG;
    }
    hipLaunchKernelGGL(k_b_euler, dim3(elem_grid(NS)), dim3(kBlock), 0, bt->stream, NS, bt->m.p, dd, dtau);
    TM_HIP(hipGetLastError());
    return TM_OK;
}

}  // extern "C"
