// rowwise.hip -- row softmax and row layer norm, and the row kernels of the
// backward pass (softmax backward, cross entropy and its backward).
//
// Reference: the CPU kernels (softmax backend.rs:2102-2125, layer_norm
// backend.rs:2380-2405) and the lazy WGSL (lazy.rs:4718-4737, 4786-4806),
// which runs ONE THREAD PER ROW and reads each row three times with a 16 KiB
// stride between neighbouring threads.
//
// Here a whole wavefront owns a row: lanes read 16-byte vectors so a wave
// instruction covers 1 KiB of contiguous row, the row stays in VGPRs between
// the passes (so HBM sees exactly one read and one write per element), and
// the max / sum / mean / variance reductions are wave64 butterflies with no
// LDS and no barriers.  Rows wider than 1024 columns (all but layer norm)
// take a whole workgroup of 512 threads instead, which streams faster; see
// the row-per-workgroup section below.
//
// Per-element arithmetic is kept to a few VALU operations so the kernels stay
// bound by HBM: exp(x) is the hardware 2^x (v_exp_f32) of x*log2(e) (relative
// error ~6e-8 |x|, about 1e-6 over the softmax range), and the per-row
// division by the sum (softmax) or by the standard deviation (layer norm) is
// one IEEE reciprocal per row times a multiply per element (<= 1.5 ulp).
// The CPU kernels divide per element; both stay far inside the 1e-4 parity
// bound.
//
// Rows whose width is not a multiple of 4 (a 50257-word vocabulary), or whose
// tensors start off a 16-byte boundary, take the same kernels in their ODD
// form: the row still moves as 16-byte vectors, now at 4-byte alignment
// (which global loads and stores allow), and its last cols % 4 elements sit
// one each in the first threads.  Bound by HBM like the aligned rows:
// [1024, 50257] cross entropy 35 us and its backward 85 us (4.9 TB/s; 79 us
// at 50256 columns), against 565 and 788 us for a wave per row re-reading it
// in 4-byte loads; [4096, 8191] softmax 47 us (46 at 8192).  Only rows too
// wide for the registers (53248 columns) are read more than once.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "launch.hpp"
#include "wave.h"

namespace clove {
namespace k {

namespace {

constexpr int kRowsPerBlock = 4;  // one row per wave, 4 waves per block

typedef float cl_f4u __attribute__((ext_vector_type(4), aligned(4)));

// Vector c of a row: ODD rows start at any 4-byte address.
template <bool ODD>
__device__ __forceinline__ cl_f4 row_load(const float *row, int c) {
    if constexpr (ODD) return __builtin_nontemporal_load(reinterpret_cast<const cl_f4u *>(row) + c);
    else return __builtin_nontemporal_load(reinterpret_cast<const cl_f4 *>(row) + c);
}

template <bool ODD>
__device__ __forceinline__ void row_store(float *row, int c, cl_f4 v) {
    if constexpr (ODD) __builtin_nontemporal_store((cl_f4u)v, reinterpret_cast<cl_f4u *>(row) + c);
    else __builtin_nontemporal_store(v, reinterpret_cast<cl_f4 *>(row) + c);
}

__device__ __forceinline__ float fast_exp(float x) {
    return __builtin_amdgcn_exp2f(x * 1.44269504088896341f);
}

// exp(x) for x <= 0 to about 1.5 ulp: the rounding of x * log2(e) and the
// part of log2(e) past f32 go back in as a first-order factor.  Below -200
// (the result is 0 in f32 either way) x is held there, so -inf and the
// lowest f32 give 0 and not inf - inf; a NaN stays one.  The hardware 2^x gives
// 0 where its result would be subnormal: SUB runs it 2^32 higher from there on
// (the sum is exact), and is taken by a branch where x says so, since it is
// a third more work on rows that hold no such entry (4 x 4000000: 1125 us
// against 1337 with SUB throughout).
constexpr float kExpNormal = -86.0f;  // e^x is normal from here on
template <bool SUB>
__device__ __forceinline__ float close_exp(float x) {
    x = x < -200.0f ? -200.0f : x;
    const float t = x * 0x1.715476p+0f;
    const float lo = __builtin_fmaf(x, 0x1.4ae0cp-26f, __builtin_fmaf(x, 0x1.715476p+0f, -t));
    const float p = __builtin_amdgcn_exp2f(SUB ? t + 32.0f : t);
    const float r = __builtin_fmaf(p, lo * 0.693147180559945f, p);
    return SUB ? r * 0x1p-32f : r;
}

__device__ __forceinline__ float close_exp(float x) {
    float r = close_exp<false>(x);
    if (__builtin_expect(x < kExpNormal, 0)) {
        asm volatile("");  // (keeps this a branch)
        r = close_exp<true>(x);
    }
    return r;
}

// The softmax's exponential and final division.  Aligned rows of up to 32768
// columns: the hardware 2^x and a multiply by the row's reciprocal.  CLOSE (odd
// rows, and any past that): close_exp and the IEEE quotient (the reciprocal
// times e, corrected by one FMA remainder), no less precise than the expf and
// the division that such rows used to get; the extra operations mostly hide
// behind HBM.
template <bool CLOSE>
__device__ __forceinline__ float row_exp(float x) {
    if constexpr (CLOSE) return close_exp(x);
    else return fast_exp(x);
}

template <bool CLOSE>
__device__ __forceinline__ float row_div(float e, float s, float inv) {
    const float q = e * inv;
    if constexpr (CLOSE) return __builtin_fmaf(__builtin_fmaf(-q, s, e), inv, q);
    else return q;
}

template <bool CLOSE>
__device__ __forceinline__ cl_f4 row_exp4(cl_f4 v, float m) {
    const cl_f4 d = v - m;
    if constexpr (!CLOSE) {
        return (cl_f4){fast_exp(d.x), fast_exp(d.y), fast_exp(d.z), fast_exp(d.w)};
    } else {
        cl_f4 r;
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = close_exp<false>(d[k]);
        if (__builtin_expect(fminf(fminf(d.x, d.y), fminf(d.z, d.w)) < kExpNormal, 0)) {
            asm volatile("");
#pragma unroll
            for (int k = 0; k < 4; ++k) r[k] = close_exp(d[k]);
        }
        return r;
    }
}

template <bool CLOSE>
__device__ __forceinline__ cl_f4 row_div4(cl_f4 e, float s, float inv) {
    return (cl_f4){row_div<CLOSE>(e.x, s, inv), row_div<CLOSE>(e.y, s, inv), row_div<CLOSE>(e.z, s, inv),
                   row_div<CLOSE>(e.w, s, inv)};
}

// d / sd of the layer norm, rsd = 1 / sd: a multiply, in ODD rows corrected
// to the quotient by one FMA remainder (what their division gave).  sdc is sd,
// or 0 where sd overflowed and rsd is 0, so that the remainder stays finite.
template <bool ODD>
__device__ __forceinline__ float row_norm(float d, float sdc, float rsd) {
    const float q = d * rsd;
    if constexpr (ODD) return __builtin_fmaf(__builtin_fmaf(-q, sdc, d), rsd, q);
    else return q;
}

template <bool ODD>
__device__ __forceinline__ cl_f4 row_norm4(cl_f4 d, float sdc, float rsd) {
    return (cl_f4){row_norm<ODD>(d.x, sdc, rsd), row_norm<ODD>(d.y, sdc, rsd),
                   row_norm<ODD>(d.z, sdc, rsd), row_norm<ODD>(d.w, sdc, rsd)};
}

// exp of a whole vector, the hardware form (the losses).
__device__ __forceinline__ cl_f4 fast_exp4(cl_f4 v, float m) {
    return (cl_f4){fast_exp(v.x - m), fast_exp(v.y - m), fast_exp(v.z - m), fast_exp(v.w - m)};
}

// x / y correctly rounded, for a y shared by many x, from r = 1 / y (IEEE):
// q0 = x r, then one FMA correction of the remainder (Markstein's method).
// With r the correctly rounded reciprocal this is the IEEE quotient; checked
// against x / y for every integer y up to 70000 over 2000 random x each
// (normal range, both signs).  An infinite q0 (x infinite) is returned as is.
__device__ __forceinline__ float div_exact(float x, float y, float r) {
    const float q0 = x * r;
    const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, y, x), r, q0);
    return __builtin_isfinite(q0) ? q1 : q0;
}

template <int VPT, bool ODD>
__global__ void __launch_bounds__(256) softmax_wave_kernel(const float *__restrict__ x,
                                                           float *__restrict__ y, int rows,
                                                           int cols) {
    const int lane = threadIdx.x & 63;
    const long row = (long)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int nvec = VPT ? cols >> 2 : 0;
    const float *xr = x + row * (long)cols;
    float *yr = y + row * (long)cols;
    const bool has_tail = ODD && lane < cols - 4 * nvec;  // lane holds element 4 nvec + lane too
    cl_f4 v[VPT ? VPT : 1];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = lane + 64 * i;
        v[i] = c < nvec ? row_load<ODD>(xr, c)
                        : (cl_f4){-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
    float e = has_tail ? xr[4 * nvec + lane] : -INFINITY;
    float m = ODD ? e : -INFINITY;
#pragma unroll
    for (int i = 0; i < VPT; ++i) m = fmaxf(m, hmax4(v[i]));
    m = wave_max(m);
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        if (lane + 64 * i < nvec) {
            v[i] = row_exp4<ODD>(v[i], m);
            s += hsum4(v[i]);
        }
    }
    if (has_tail) {
        e = row_exp<ODD>(e - m);
        s += e;
    }
    s = wave_sum(s);
    const float inv = 1.0f / s;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = lane + 64 * i;
        if (c < nvec) row_store<ODD>(yr, c, row_div4<ODD>(v[i], s, inv));
    }
    if (has_tail) yr[4 * nvec + lane] = row_div<ODD>(e, s, inv);
}

// gamma and beta are staged in LDS once per workgroup (2 * cols floats):
// every row of the workgroup reads them, and fetching them from L2 per row
// costs as much traffic as the rows themselves (at 4096 columns the pair is
// 32 KiB, the size of the vector L1).  The row's own loads are issued first
// so the staging overlaps them.
template <int VPT, bool ODD>
__global__ void __launch_bounds__(256) layer_norm_wave_kernel(const float *__restrict__ x,
                                                              const float *__restrict__ gamma,
                                                              const float *__restrict__ beta,
                                                              float *__restrict__ y, int rows,
                                                              int cols, float eps) {
    extern __shared__ cl_f4 s_gb[];  // [nvec] gamma, then [nvec] beta
    const int lane = threadIdx.x & 63;
    const long row = (long)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    const bool live = row < rows;
    const int nvec = VPT ? cols >> 2 : 0;
    const float *xr = x + (live ? row : 0) * (long)cols;
    const bool has_tail = ODD && live && lane < cols - 4 * nvec;
    cl_f4 v[VPT ? VPT : 1];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = lane + 64 * i;
        v[i] = (live && c < nvec) ? row_load<ODD>(xr, c) : (cl_f4){0.f, 0.f, 0.f, 0.f};
    }
    float e = 0.0f, eg = 0.0f, eb = 0.0f;  // the tail element, its gamma and beta
    if (has_tail) {
        e = xr[4 * nvec + lane];
        eg = gamma[4 * nvec + lane];
        eb = beta[4 * nvec + lane];
    }
    using gvec = typename std::conditional<ODD, cl_f4u, cl_f4>::type;
    const gvec *g4 = reinterpret_cast<const gvec *>(gamma);
    const gvec *b4 = reinterpret_cast<const gvec *>(beta);
    if (VPT) {
        for (int c = threadIdx.x; c < nvec; c += 256) {
            s_gb[c] = g4[c];
            s_gb[nvec + c] = b4[c];
        }
        __syncthreads();
    }
    if (!live) return;
    float *yr = y + row * (long)cols;
#pragma unroll
    for (int i = 0; i < VPT; ++i) s += hsum4(v[i]);
    if (ODD) s += e;
    const float n = (float)cols;
    const float mean = wave_sum(s) / n;
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        if (lane + 64 * i < nvec) {
            const cl_f4 d = v[i] - mean;
            q += hsum4(d * d);
        }
    }
    if (has_tail) q += (e - mean) * (e - mean);
    const float var = wave_sum(q) / n;
    const float sd = sqrtf(var + eps), rsd = 1.0f / sd;
    const float sdc = rsd > 0.0f ? sd : 0.0f;  // (row_norm's divisor)
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = lane + 64 * i;
        if (c < nvec)
            row_store<ODD>(yr, c, row_norm4<ODD>(v[i] - mean, sdc, rsd) * s_gb[c] + s_gb[nvec + c]);
    }
    if (has_tail) yr[4 * nvec + lane] = row_norm<ODD>(e - mean, sdc, rsd) * eg + eb;
}

// ---- backward and loss rows ----------------------------------------------

// Softmax backward (backend.rs:2163-2183): dx = y * (dy - sum(dy * y)) per
// row, the row of y and of dy held in registers.
template <int VPT, bool ODD>
__global__ void __launch_bounds__(256) softmax_bw_wave_kernel(const float *__restrict__ y,
                                                              const float *__restrict__ dy,
                                                              float *__restrict__ dx, int rows,
                                                              int cols) {
    const int lane = threadIdx.x & 63;
    const long row = (long)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int nvec = VPT ? cols >> 2 : 0;
    const float *yr = y + row * (long)cols, *gr = dy + row * (long)cols;
    float *o = dx + row * (long)cols;
    constexpr int E = VPT ? 1 : 2;  // elements a lane holds past the vectors, 64 apart
    const int tail = ODD ? cols - 4 * nvec : 0;
    cl_f4 vy[VPT ? VPT : 1], vg[VPT ? VPT : 1];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = lane + 64 * i;
        const bool in = c < nvec;
        vy[i] = in ? row_load<ODD>(yr, c) : (cl_f4){0.f, 0.f, 0.f, 0.f};
        vg[i] = in ? row_load<ODD>(gr, c) : (cl_f4){0.f, 0.f, 0.f, 0.f};
    }
    float ey[E], eg[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const int c = lane + 64 * i;
        ey[i] = c < tail ? yr[4 * nvec + c] : 0.0f;
        eg[i] = c < tail ? gr[4 * nvec + c] : 0.0f;
    }
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) s += hsum4(vg[i] * vy[i]);
#pragma unroll
    for (int i = 0; i < E; ++i)
        if (ODD) s += eg[i] * ey[i];
    s = wave_sum(s);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = lane + 64 * i;
        if (c < nvec) row_store<ODD>(o, c, vy[i] * (vg[i] - s));
    }
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const int c = lane + 64 * i;
        if (c < tail) o[4 * nvec + c] = ey[i] * (eg[i] - s);
    }
}

// Rust's `f32 as usize` saturates: NaN and negative targets read class 0.
__device__ __forceinline__ long target_class(float v) {
    if (!(v > 0.0f)) return 0;
    return v >= 9.0e18f ? (long)9.0e18 : (long)v;
}

// Cross entropy, one wave per row (backend.rs:2661-2680): row value
// v = (l[t] - max) - ln(sum exp(l - max)); the loss is -sum(v) / rows, which
// ordered_sum (reduce.hip) adds in a fixed order.  Rows at or past `used` (no target)
// give 0; a class >= cols raises the error flag and gives 0.
// MODE 0 writes v to rowv[row].  MODE 1 is the backward (backend.rs:
// 2686-2712): grad = (exp(l - max) / sum - [j == t]) * g / rows.
template <int VPT, int MODE, bool ODD>
__global__ void __launch_bounds__(256) cross_entropy_wave_kernel(
    const float *__restrict__ logits, const float *__restrict__ targets, long used, int rows,
    int cols, const float *__restrict__ grad_loss, float *__restrict__ out, int *err_flag) {
    const int lane = threadIdx.x & 63;
    const long row = (long)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int nvec = VPT ? cols >> 2 : 0;
    float *go = MODE == 1 ? out + row * (long)cols : nullptr;
    const bool has_tail = ODD && lane < cols - 4 * nvec;
    // The row's loads go out first: read after the target (and a branch on
    // it), they would wait one memory latency per row.
    const float *lr = logits + row * (long)cols;
    cl_f4 v[VPT ? VPT : 1];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = lane + 64 * i;
        v[i] = c < nvec ? row_load<ODD>(lr, c)
                        : (cl_f4){-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
    float e = has_tail ? lr[4 * nvec + lane] : -INFINITY;
    long t = -1;
    if (row < used) {
        t = target_class(targets[row]);
        if (t >= cols) {
            if (lane == 0) atomicOr(err_flag, kErrClassRange);
            t = -1;
        }
    }
    if (t < 0) {  // no target (or a bad one): the row contributes nothing
        if (MODE == 0) {
            if (lane == 0) out[row] = 0.0f;
        } else {
            for (int c = lane; c < nvec; c += 64) row_store<ODD>(go, c, (cl_f4){0.f, 0.f, 0.f, 0.f});
            if (has_tail) go[4 * nvec + lane] = 0.0f;
        }
        return;
    }
    // l[t] from the registers of the lane that holds it (vector t/4 lives in
    // lane (t/4) % 64, slot (t/4) / 64), not from a second global load.
    float lt = 0.0f;
    if (MODE == 0) {
        const int tv = (int)(t >> 2), ts = (int)(t & 3);
#pragma unroll
        for (int i = 0; i < VPT; ++i)
            if (lane + 64 * i == tv) lt = v[i][ts];
        lt = __shfl(lt, tv & 63, 64);
        if (ODD && t >= 4l * nvec) lt = __shfl(e, (int)(t - 4l * nvec), 64);
    }
    float m = ODD ? e : -INFINITY;
#pragma unroll
    for (int i = 0; i < VPT; ++i) m = fmaxf(m, hmax4(v[i]));
    m = wave_max(m);
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        if (lane + 64 * i < nvec) {
            v[i] = fast_exp4(v[i], m);
            s += hsum4(v[i]);
        }
    }
    if (has_tail) {
        e = fast_exp(e - m);
        s += e;
    }
    s = wave_sum(s);
    if (MODE == 0) {
        if (lane == 0) out[row] = (lt - m) - logf(s);
        return;
    }
    const float inv = 1.0f / s;
    const float g = grad_loss[0];
    const float fr = (float)rows;
    const float rr = 1.0f / fr;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = lane + 64 * i;
        if (c < nvec) {
            cl_f4 p = v[i] * inv;
            const long j0 = 4l * c;
            if (t >= j0 && t < j0 + 4) p[t - j0] -= 1.0f;
            const cl_f4 x = p * g;
            row_store<ODD>(go, c, (cl_f4){div_exact(x.x, fr, rr), div_exact(x.y, fr, rr),
                                          div_exact(x.z, fr, rr), div_exact(x.w, fr, rr)});
        }
    }
    if (has_tail) {
        const float p = e * inv - (t == 4l * nvec + lane ? 1.0f : 0.0f);
        go[4 * nvec + lane] = div_exact(p * g, fr, rr);
    }
}

// ---- one row per workgroup -------------------------------------------------
//
// Rows wider than 1024 columns take a whole workgroup of kBlockThreads
// threads per row, P 16-byte vectors per thread (vector c of the row lives in
// thread c % kBlockThreads, slot c / kBlockThreads).  Measured on MI355X
// with inputs cycled so the last-level cache holds none of them, a
// [8192, 4096] softmax ran at 78.9% of HBM peak this way against 69.9% with
// one wave per row (256 threads: 76.0%), and a plain 128 MiB read at 82.4%
// against 76.3%: one 16 KiB row read by eight waves at once instead of four
// rows by four waves.  The row's reductions are wave butterflies, then the
// eight wave results added (or maxed) in wave order through LDS, so results
// stay deterministic.  Per element the arithmetic is the wave kernels'.
// Layer norm keeps one wave per row: with a row per workgroup every row
// reads gamma and beta (twice the row's bytes) from the L2, and it measured
// 65-71% (one to four rows per workgroup, all loaded at once) and 63-69%
// (4-16 rows walked in order, gamma and beta in registers, the next row
// prefetched) against the wave kernel's 75%, which stages them in LDS once
// per four rows.
constexpr int kBlockThreads = 512;
constexpr int kBlockWaves = kBlockThreads / 64;
constexpr int kSlot = 4 * kBlockThreads;  // floats from one of a thread's vectors to its next

// A row of kMaxP vectors per thread is 104 registers: held to 128 in all, two
// workgroups still share a CU, one loading or storing while the other reduces
// ([1024, 50257] cross entropy 35 us, 56 us while the row's addresses took
// registers too and one workgroup filled a CU: hence row_load's uniform base
// plus a thread offset).
constexpr int kMaxP = 26;
// (row_step keeps the compiler from running several vectors' arithmetic at
// once there, whose temporaries would spill.)
template <int P>
__device__ __forceinline__ void row_step() {
    if constexpr (P == kMaxP) __builtin_amdgcn_sched_barrier(0);
}
#define CLOVE_ROW_WAVES(P) __attribute__((amdgpu_waves_per_eu((P) == kMaxP ? 4 : 2)))

// Workgroup-wide max / sum; every thread gets the result.  Each call needs
// its own `slot` (kBlockWaves floats of LDS): a slot reused by a later
// reduction could be overwritten while a slow wave still reads it.
__device__ __forceinline__ float block_max(float v, float *slot) {
    v = wave_max(v);
    if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = slot[0];
#pragma unroll
    for (int w = 1; w < kBlockWaves; ++w) r = fmaxf(r, slot[w]);
    return r;
}

__device__ __forceinline__ float block_sum(float v, float *slot) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = slot[0];
#pragma unroll
    for (int w = 1; w < kBlockWaves; ++w) r += slot[w];
    return r;
}

template <int P, bool ODD>
__global__ void __launch_bounds__(kBlockThreads)
    CLOVE_ROW_WAVES(P) softmax_block_kernel(const float *__restrict__ x,
                                                                      float *__restrict__ y,
                                                                      int cols) {
    __shared__ float red[2][kBlockWaves];
    const long row = blockIdx.x;
    const int nvec = cols >> 2;
    const float *xr = x + row * (long)cols;
    float *yr = y + row * (long)cols;
    const bool has_tail = ODD && (int)threadIdx.x < (cols & 3);
    // ([1024, 50304] aligned: 74.5 us against 71.3 in the hardware form, whose
    // entries were up to 1.8e-6 off; here 3.0e-7)
    constexpr bool CLOSE = ODD || P == kMaxP;
    cl_f4 v[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = threadIdx.x + kBlockThreads * i;
        v[i] = c < nvec ? row_load<ODD>(xr + kSlot * i, threadIdx.x)
                        : (cl_f4){-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
    float e = has_tail ? xr[4 * nvec + threadIdx.x] : -INFINITY;
    float m = ODD ? e : -INFINITY;
#pragma unroll
    for (int i = 0; i < P; ++i) m = fmaxf(m, hmax4(v[i]));
    m = block_max(m, red[0]);
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        if (threadIdx.x + kBlockThreads * i < nvec) {
            v[i] = row_exp4<CLOSE>(v[i], m);
            s += hsum4(v[i]);
        }
        row_step<P>();
    }
    if (has_tail) {
        e = row_exp<CLOSE>(e - m);
        s += e;
    }
    s = block_sum(s, red[1]);
    const float inv = 1.0f / s;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = threadIdx.x + kBlockThreads * i;
        if (c < nvec) row_store<ODD>(yr + kSlot * i, threadIdx.x, row_div4<CLOSE>(v[i], s, inv));
        row_step<P>();
    }
    if (has_tail) yr[4 * nvec + threadIdx.x] = row_div<CLOSE>(e, s, inv);
}

// Layer norm of rows past the wave kernel's 8192 columns: the same arithmetic
// with a workgroup per row, gamma and beta from L2.
template <int P, bool ODD>
__global__ void __launch_bounds__(kBlockThreads)
    CLOVE_ROW_WAVES(P) layer_norm_block_kernel(
    const float *__restrict__ x, const float *__restrict__ gamma, const float *__restrict__ beta,
    float *__restrict__ y, int cols, float eps) {
    __shared__ float red[2][kBlockWaves];
    const long row = blockIdx.x;
    const int nvec = cols >> 2;
    const float *xr = x + row * (long)cols;
    float *yr = y + row * (long)cols;
    const bool has_tail = ODD && (int)threadIdx.x < (cols & 3);
    cl_f4 v[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = threadIdx.x + kBlockThreads * i;
        v[i] = c < nvec ? row_load<ODD>(xr + kSlot * i, threadIdx.x) : (cl_f4){0.f, 0.f, 0.f, 0.f};
    }
    const float e = has_tail ? xr[4 * nvec + threadIdx.x] : 0.0f;
    float s = ODD ? e : 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) s += hsum4(v[i]);
    const float n = (float)cols;
    const float mean = block_sum(s, red[0]) / n;
    float q = has_tail ? (e - mean) * (e - mean) : 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        if (threadIdx.x + kBlockThreads * i < nvec) {
            const cl_f4 d = v[i] - mean;
            q += hsum4(d * d);
        }
        row_step<P>();
    }
    const float var = block_sum(q, red[1]) / n;
    const float sd = sqrtf(var + eps), rsd = 1.0f / sd;
    const float sdc = rsd > 0.0f ? sd : 0.0f;
    using gvec = typename std::conditional<ODD, cl_f4u, cl_f4>::type;
    const gvec *g4 = reinterpret_cast<const gvec *>(gamma);
    const gvec *b4 = reinterpret_cast<const gvec *>(beta);
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = threadIdx.x + kBlockThreads * i;
        if (c < nvec)
            row_store<ODD>(yr + kSlot * i, threadIdx.x, row_norm4<true>(v[i] - mean, sdc, rsd) * (cl_f4)(g4 + kBlockThreads * i)[threadIdx.x] +
                                      (cl_f4)(b4 + kBlockThreads * i)[threadIdx.x]);
        row_step<P>();
    }
    if (has_tail) {
        const int j = 4 * nvec + threadIdx.x;
        yr[j] = row_norm<true>(e - mean, sdc, rsd) * gamma[j] + beta[j];
    }
}

template <int P, bool ODD>
__global__ void __launch_bounds__(kBlockThreads) softmax_bw_block_kernel(
    const float *__restrict__ y, const float *__restrict__ dy, float *__restrict__ dx, int cols) {
    __shared__ float red[kBlockWaves];
    const long row = blockIdx.x;
    const int nvec = cols >> 2;
    const float *yr = y + row * (long)cols, *gr = dy + row * (long)cols;
    float *o = dx + row * (long)cols;
    const bool has_tail = ODD && (int)threadIdx.x < (cols & 3);
    cl_f4 vy[P], vg[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = threadIdx.x + kBlockThreads * i;
        const bool in = c < nvec;
        vy[i] = in ? row_load<ODD>(yr + kSlot * i, threadIdx.x) : (cl_f4){0.f, 0.f, 0.f, 0.f};
        vg[i] = in ? row_load<ODD>(gr + kSlot * i, threadIdx.x) : (cl_f4){0.f, 0.f, 0.f, 0.f};
    }
    const float ey = has_tail ? yr[4 * nvec + threadIdx.x] : 0.0f;
    const float eg = has_tail ? gr[4 * nvec + threadIdx.x] : 0.0f;
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) s += hsum4(vg[i] * vy[i]);
    if (ODD) s += eg * ey;
    s = block_sum(s, red);
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = threadIdx.x + kBlockThreads * i;
        if (c < nvec) row_store<ODD>(o + kSlot * i, threadIdx.x, vy[i] * (vg[i] - s));
    }
    if (has_tail) o[4 * nvec + threadIdx.x] = ey * (eg - s);
}

// Cross entropy and its backward with a workgroup per row (the wave
// kernel's contract and arithmetic).  l[target] comes from the registers of
// the thread holding it, through LDS, published before the max reduction's
// barrier.
template <int P, int MODE, bool ODD>
__global__ void __launch_bounds__(kBlockThreads)
    CLOVE_ROW_WAVES(P) cross_entropy_block_kernel(
    const float *__restrict__ logits, const float *__restrict__ targets, long used, int rows,
    int cols, const float *__restrict__ grad_loss, float *__restrict__ out, int *err_flag) {
    __shared__ float red[2][kBlockWaves];
    __shared__ float s_lt;
    const long row = blockIdx.x;
    const int nvec = cols >> 2;
    const float *lr = logits + row * (long)cols;
    float *go = MODE == 1 ? out + row * (long)cols : nullptr;
    const bool has_tail = ODD && (int)threadIdx.x < (cols & 3);
    cl_f4 v[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = threadIdx.x + kBlockThreads * i;
        v[i] = c < nvec ? row_load<ODD>(lr + kSlot * i, threadIdx.x)
                        : (cl_f4){-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
    float e = has_tail ? lr[4 * nvec + threadIdx.x] : -INFINITY;
    long t = -1;  // the same for every thread of the row
    if (row < used) {
        t = target_class(targets[row]);
        if (t >= cols) {
            if (threadIdx.x == 0) atomicOr(err_flag, kErrClassRange);
            t = -1;
        }
    }
    if (t < 0) {
        if (MODE == 0) {
            if (threadIdx.x == 0) out[row] = 0.0f;
        } else {
            for (int c = threadIdx.x; c < nvec; c += kBlockThreads)
                row_store<ODD>(go, c, (cl_f4){0.f, 0.f, 0.f, 0.f});
            if (has_tail) go[4 * nvec + threadIdx.x] = 0.0f;
        }
        return;
    }
    if (MODE == 0) {
        const int tv = (int)(t >> 2), ts = (int)(t & 3);
        if (tv % kBlockThreads == (int)threadIdx.x) {
#pragma unroll
            for (int i = 0; i < P; ++i)
                if (tv < nvec && i == tv / kBlockThreads) s_lt = v[i][ts];
        }
        if (has_tail && t == 4l * nvec + threadIdx.x) s_lt = e;
    }
    float m = ODD ? e : -INFINITY;
#pragma unroll
    for (int i = 0; i < P; ++i) m = fmaxf(m, hmax4(v[i]));
    m = block_max(m, red[0]);
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        if (threadIdx.x + kBlockThreads * i < nvec) {
            v[i] = fast_exp4(v[i], m);
            s += hsum4(v[i]);
        }
    }
    if (has_tail) {
        e = fast_exp(e - m);
        s += e;
    }
    s = block_sum(s, red[1]);
    if (MODE == 0) {
        if (threadIdx.x == 0) out[row] = (s_lt - m) - logf(s);
        return;
    }
    const float inv = 1.0f / s;
    const float g = grad_loss[0];
    const float fr = (float)rows;
    const float rr = 1.0f / fr;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = threadIdx.x + kBlockThreads * i;
        if (c < nvec) {
            cl_f4 p = v[i] * inv;
            const long j0 = 4l * c;
            if (t >= j0 && t < j0 + 4) p[t - j0] -= 1.0f;
            const cl_f4 xg = p * g;
            row_store<ODD>(go + kSlot * i, threadIdx.x, (cl_f4){div_exact(xg.x, fr, rr), div_exact(xg.y, fr, rr),
                                          div_exact(xg.z, fr, rr), div_exact(xg.w, fr, rr)});
        }
    }
    if (has_tail) {
        const float p = e * inv - (t == 4l * nvec + threadIdx.x ? 1.0f : 0.0f);
        go[4 * nvec + threadIdx.x] = div_exact(p * g, fr, rr);
    }
}

// Cross entropy forward with two rows per workgroup (the block kernel's
// per-row arithmetic and reduction order, so the same bits): each thread
// holds P vectors of both rows, and the two rows' maxima and sums go through
// the same butterflies and the same two barriers.  Measured at [8192, 4096]
// with cold inputs: 21.3-21.4 us against 22.0-24.0 us for one row per
// workgroup (four rows: 23.2 us): twice the bytes in flight per workgroup at
// the same barrier count.  A row past `rows` (odd row counts) loads nothing
// and writes nothing.
template <int P>
__global__ void __launch_bounds__(kBlockThreads) cross_entropy_rows2_kernel(
    const float *__restrict__ logits, const float *__restrict__ targets, long used, int rows,
    int cols, float *__restrict__ out, int *err_flag) {
    __shared__ float red[2][2][kBlockWaves];
    __shared__ float s_lt[2];
    const long row0 = 2L * blockIdx.x;
    const int nvec = cols >> 2;
    cl_f4 v[2][P];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const bool live = row0 + r < rows;
        const cl_f4 *lr = reinterpret_cast<const cl_f4 *>(logits + (row0 + r) * (long)cols);
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const int c = threadIdx.x + kBlockThreads * i;
            v[r][i] = (live && c < nvec) ? __builtin_nontemporal_load(lr + c)
                                         : (cl_f4){-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        }
    }
    long t[2];  // the same for every thread of the row; -1: the row counts 0
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const long row = row0 + r;
        t[r] = -1;
        if (row < used && row < rows) {
            t[r] = target_class(targets[row]);
            if (t[r] >= cols) {
                if (threadIdx.x == 0) atomicOr(err_flag, kErrClassRange);
                t[r] = -1;
            }
        }
        if (t[r] >= 0) {
            const int tv = (int)(t[r] >> 2), ts = (int)(t[r] & 3);
            if (tv % kBlockThreads == (int)threadIdx.x) {
#pragma unroll
                for (int i = 0; i < P; ++i)
                    if (i == tv / kBlockThreads) s_lt[r] = v[r][i][ts];
            }
        }
    }
    float m[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        m[r] = -INFINITY;
#pragma unroll
        for (int i = 0; i < P; ++i) m[r] = fmaxf(m[r], hmax4(v[r][i]));
        m[r] = wave_max(m[r]);
        if ((threadIdx.x & 63) == 0) red[0][r][threadIdx.x >> 6] = m[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        float x = red[0][r][0];
#pragma unroll
        for (int w = 1; w < kBlockWaves; ++w) x = fmaxf(x, red[0][r][w]);
        m[r] = x;
    }
    float sm[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        sm[r] = 0.0f;
#pragma unroll
        for (int i = 0; i < P; ++i) {
            if (threadIdx.x + kBlockThreads * i < nvec) {
                const cl_f4 e = {fast_exp(v[r][i].x - m[r]), fast_exp(v[r][i].y - m[r]),
                                 fast_exp(v[r][i].z - m[r]), fast_exp(v[r][i].w - m[r])};
                sm[r] += hsum4(e);
            }
        }
        sm[r] = wave_sum(sm[r]);
        if ((threadIdx.x & 63) == 0) red[1][r][threadIdx.x >> 6] = sm[r];
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const int r = threadIdx.x;
        const long row = row0 + r;
        if (row < rows) {
            float x = red[1][r][0];
#pragma unroll
            for (int w = 1; w < kBlockWaves; ++w) x += red[1][r][w];
            out[row] = t[r] < 0 ? 0.0f : (s_lt[r] - m[r]) - logf(x);
        }
    }
}

// ---- rows past the registers ---------------------------------------------
//
// Rows of more than 4 * 512 * kMaxP columns: a workgroup per row still, its
// vectors walked kLoopVec at a time at any alignment, and the row read again
// (from the last-level cache) where its values are needed a second time.
constexpr int kLoopVec = 4;

// This thread's share of a row of `cols`: fv(j, v) for its whole vectors, the
// elements j .. j + 3, and f(j, x) for its one of the last cols % 4.
template <class FV, class F>
__device__ __forceinline__ void row_walk4(const float *row, int cols, FV fv, F f) {
    const int nvec = cols >> 2;
    for (int c0 = threadIdx.x; c0 < nvec; c0 += kLoopVec * kBlockThreads) {
        cl_f4 v[kLoopVec];
#pragma unroll
        for (int u = 0; u < kLoopVec; ++u) {
            const int c = c0 + u * kBlockThreads;
            if (c < nvec) v[u] = *(reinterpret_cast<const cl_f4u *>(row) + c);
        }
#pragma unroll
        for (int u = 0; u < kLoopVec; ++u) {
            const int c = c0 + u * kBlockThreads;
            if (c < nvec) fv(4 * c, v[u]);
        }
    }
    const int j = 4 * nvec + threadIdx.x;
    if ((int)threadIdx.x < (cols & 3)) f(j, row[j]);
}

// f(j, x) for every element of it.
template <class F>
__device__ __forceinline__ void row_walk(const float *row, int cols, F f) {
    row_walk4(
        row, cols,
        [&](int j, cl_f4 v) {
#pragma unroll
            for (int k = 0; k < 4; ++k) f(j + k, v[k]);
        },
        f);
}

// The row's max and sum of exp(x - max) in one walk: a running max and a sum
// relative to it per thread, the threads' sums then brought to the row's max.
// A max of -inf counts as 0 in the subtractions (-inf entries give 0, not
// NaN); NaN entries reach the sum.  A row of -inf alone sums to 0.  (The sum is
// 1 or more: a subnormal term is no part of it.)
__device__ __forceinline__ void row_max_sum(const float *row, int cols, float red[2][kBlockWaves],
                                            float *m_out, float *s_out) {
    float m = -INFINITY, s = 0.0f;
    row_walk(row, cols, [&](int, float x) {
        if (x > m) {
            s *= m == -INFINITY ? 1.0f : close_exp<false>(m - x);
            m = x;
        }
        s += close_exp<false>(x - (m == -INFINITY ? 0.0f : m));
    });
    const float gm = block_max(m, red[0]);
    if (m != -INFINITY) s *= close_exp<false>(m - gm);
    *m_out = gm;
    *s_out = block_sum(s, red[1]);
}

__global__ void __launch_bounds__(kBlockThreads) softmax_loop_kernel(const float *__restrict__ x,
                                                                     float *__restrict__ y,
                                                                     int cols) {
    __shared__ float red[2][kBlockWaves];
    const float *xr = x + (long)blockIdx.x * cols;
    float *yr = y + (long)blockIdx.x * cols;
    float m, s;
    row_max_sum(xr, cols, red, &m, &s);
    const float inv = 1.0f / s;
    row_walk4(
        xr, cols,
        [&](int j, cl_f4 v) {
            *reinterpret_cast<cl_f4u *>(yr + j) = row_div4<true>(row_exp4<true>(v, m), s, inv);
        },
        [&](int j, float v) { yr[j] = row_div<true>(close_exp(v - m), s, inv); });
}

__global__ void __launch_bounds__(kBlockThreads) layer_norm_loop_kernel(
    const float *__restrict__ x, const float *__restrict__ gamma, const float *__restrict__ beta,
    float *__restrict__ y, int cols, float eps) {
    __shared__ float red[2][kBlockWaves];
    const float *xr = x + (long)blockIdx.x * cols;
    float *yr = y + (long)blockIdx.x * cols;
    const float n = (float)cols;
    float s = 0.0f;
    row_walk(xr, cols, [&](int, float v) { s += v; });
    const float mean = block_sum(s, red[0]) / n;
    float q = 0.0f;
    row_walk(xr, cols, [&](int, float v) { q += (v - mean) * (v - mean); });
    const float sd = sqrtf(block_sum(q, red[1]) / n + eps), rsd = 1.0f / sd;
    const float sdc = rsd > 0.0f ? sd : 0.0f;
    row_walk(xr, cols, [&](int j, float v) {
        yr[j] = row_norm<true>(v - mean, sdc, rsd) * gamma[j] + beta[j];
    });
}

__global__ void __launch_bounds__(kBlockThreads) softmax_bw_loop_kernel(
    const float *__restrict__ y, const float *__restrict__ dy, float *__restrict__ dx, int cols) {
    __shared__ float red[kBlockWaves];
    const float *yr = y + (long)blockIdx.x * cols, *gr = dy + (long)blockIdx.x * cols;
    float *o = dx + (long)blockIdx.x * cols;
    float s = 0.0f;
    row_walk(yr, cols, [&](int j, float v) { s += gr[j] * v; });
    s = block_sum(s, red);
    row_walk(yr, cols, [&](int j, float v) { o[j] = v * (gr[j] - s); });
}

template <int MODE>
__global__ void __launch_bounds__(kBlockThreads) cross_entropy_loop_kernel(
    const float *__restrict__ logits, const float *__restrict__ targets, long used, int cols,
    float rows, const float *__restrict__ grad_loss, float *__restrict__ out, int *err_flag) {
    __shared__ float red[2][kBlockWaves];
    const long row = blockIdx.x;
    const float *lr = logits + row * (long)cols;
    float *go = MODE == 1 ? out + row * (long)cols : nullptr;
    long t = -1;  // the same for every thread of the row
    if (row < used) {
        t = target_class(targets[row]);
        if (t >= cols) {
            if (threadIdx.x == 0) atomicOr(err_flag, kErrClassRange);
            t = -1;
        }
    }
    if (t < 0) {
        if (MODE == 0) {
            if (threadIdx.x == 0) out[row] = 0.0f;
        } else {
            for (int j = threadIdx.x; j < cols; j += kBlockThreads) go[j] = 0.0f;
        }
        return;
    }
    float m, s;
    row_max_sum(lr, cols, red, &m, &s);
    if (MODE == 0) {
        if (threadIdx.x == 0) out[row] = (lr[t] - m) - logf(s);
        return;
    }
    const float inv = 1.0f / s, g = grad_loss[0], rr = 1.0f / rows;
    row_walk(lr, cols, [&](int j, float v) {
        const float p = fast_exp(v - m) * inv - (j == t ? 1.0f : 0.0f);
        go[j] = div_exact(p * g, rows, rr);
    });
}

// Vectors per thread of the row-per-workgroup kernels for this width, or 0
// for the one-wave-per-row kernels (at most 1024 columns), or -1 for a row
// that the registers do not hold.
int pick_block_p(int cols) {
    const int nvec = cols / 4;
    if (nvec <= 256) return 0;
    int p = 1;
    while (p < 16 && p * kBlockThreads < nvec) p <<= 1;
    if (p * kBlockThreads < nvec) p = kMaxP;
    return p * kBlockThreads >= nvec ? p : -1;
}

// Vectors per lane of the wave-per-row kernels, or 0 past 8192 columns.
int pick_vpt(int cols) {
    const int need = (cols / 4 + 63) / 64;
    int v = 1;
    while (v < need) v <<= 1;
    return v <= 32 ? v : 0;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// launch(first row, rows) of the row-per-workgroup kernels, whose grid holds
// under 2^32 threads: 2^23 rows and more go in several launches.
constexpr size_t kRowsPerLaunch = 1 << 22;
template <class F>
void row_runs(size_t rows, F launch) {
    for (size_t r0 = 0; r0 < rows; r0 += kRowsPerLaunch)
        launch(r0, (unsigned)std::min(kRowsPerLaunch, rows - r0));
}

// launch(P, ODD) with the constants the row-per-workgroup kernels are built
// for.
template <class F>
void with_block_p(int p, bool odd, F launch) {
    auto go = [&](auto P) {
        if (odd) launch(P, std::true_type{});
        else launch(P, std::false_type{});
    };
    switch (p) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 8: go(std::integral_constant<int, 8>{}); break;
    case 16: go(std::integral_constant<int, 16>{}); break;
    default: go(std::integral_constant<int, kMaxP>{}); break;
    }
}

// Odd rows of at most a wave's lanes move one element a lane (VPT = 0): two
// loads of a row, its vectors and its tail, cost more than they carry (softmax
// backward of [1000000, 7] 119 us against 185, of [1000000, 33] 178 against 210).
bool one_per_lane(int cols, bool odd) { return odd && cols <= 64; }
// The softmax backward, which loads two rows, takes two a lane up to here
// ([300000, 65] 44 us against 69, 61 for a plain walk of the row; 127 columns 85
// against 90).
constexpr int kTwoPerLane = 128;

// The same for the wave-per-row kernels, up to MAXV vectors per lane (0: one
// element).
template <int MAXV, class F>
void with_vpt(int v, bool odd, F launch) {
    auto go = [&](auto V) {
        if (odd) launch(V, std::true_type{});
        else launch(V, std::false_type{});
    };
    switch (v) {
    case 0: launch(std::integral_constant<int, 0>{}, std::true_type{}); return;
    case 1: go(std::integral_constant<int, 1>{}); return;
    case 2: go(std::integral_constant<int, 2>{}); return;
    case 4: go(std::integral_constant<int, 4>{}); return;
    default: break;
    }
    if constexpr (MAXV >= 32) {
        if (v == 8) go(std::integral_constant<int, 8>{});
        else if (v == 16) go(std::integral_constant<int, 16>{});
        else go(std::integral_constant<int, 32>{});
    }
}

}  // namespace

void softmax_rows(const float *x, float *y, size_t rows, size_t cols, hipStream_t s) {
    if (!rows || !cols) return;
    const unsigned grid = (unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock);
    const int r = (int)rows, c = (int)cols;
    const bool odd = c % 4 != 0 || !aligned16(x) || !aligned16(y);
    const int p = pick_block_p(c);
    if (p < 0)
        row_runs(rows, [&](size_t r0, unsigned n) {
            softmax_loop_kernel<<<n, kBlockThreads, 0, s>>>(x + r0 * cols, y + r0 * cols, c);
        });
    else if (p > 0)
        with_block_p(p, odd, [&](auto P, auto O) {
            row_runs(rows, [&](size_t r0, unsigned n) {
                softmax_block_kernel<P(), O()>
                    <<<n, kBlockThreads, 0, s>>>(x + r0 * cols, y + r0 * cols, c);
            });
        });
    else
        with_vpt<4>(one_per_lane(c, odd) ? 0 : pick_vpt(c), odd, [&](auto V, auto O) {
            softmax_wave_kernel<V(), O()><<<grid, 256, 0, s>>>(x, y, r, c);
        });
}

void layer_norm_rows(const float *x, const float *gamma, const float *beta, float *y,
                     size_t rows, size_t cols, float eps, hipStream_t s) {
    if (!rows || !cols) return;
    const unsigned grid = (unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock);
    const int r = (int)rows, c = (int)cols;
    const bool odd = c % 4 != 0 || !aligned16(x) || !aligned16(y) || !aligned16(gamma) ||
                     !aligned16(beta);
    const int vpt = pick_vpt(c), p = pick_block_p(c);
    const size_t lds = 2 * (size_t)(c / 4) * sizeof(cl_f4);
    if (vpt > 0)
        with_vpt<32>(one_per_lane(c, odd) ? 0 : vpt, odd, [&](auto V, auto O) {
            layer_norm_wave_kernel<V(), O()><<<grid, 256, lds, s>>>(x, gamma, beta, y, r, c, eps);
        });
    else if (p > 0)
        with_block_p(p, odd, [&](auto P, auto O) {
            row_runs(rows, [&](size_t r0, unsigned n) {
                layer_norm_block_kernel<P(), O()><<<n, kBlockThreads, 0, s>>>(
                    x + r0 * cols, gamma, beta, y + r0 * cols, c, eps);
            });
        });
    else
        row_runs(rows, [&](size_t r0, unsigned n) {
            layer_norm_loop_kernel<<<n, kBlockThreads, 0, s>>>(x + r0 * cols, gamma, beta,
                                                               y + r0 * cols, c, eps);
        });
}

void softmax_backward_rows(const float *y, const float *dy, float *dx, size_t rows, size_t cols,
                           hipStream_t s) {
    if (!rows || !cols) return;
    const unsigned grid = (unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock);
    const int r = (int)rows, c = (int)cols;
    const bool odd = c % 4 != 0 || !aligned16(y) || !aligned16(dy) || !aligned16(dx);
    const int p = pick_block_p(c);
    if (p < 0)
        row_runs(rows, [&](size_t r0, unsigned n) {
            softmax_bw_loop_kernel<<<n, kBlockThreads, 0, s>>>(y + r0 * cols, dy + r0 * cols,
                                                               dx + r0 * cols, c);
        });
    else if (p > 0)
        with_block_p(p, odd, [&](auto P, auto O) {
            row_runs(rows, [&](size_t r0, unsigned n) {
                softmax_bw_block_kernel<P(), O()><<<n, kBlockThreads, 0, s>>>(
                    y + r0 * cols, dy + r0 * cols, dx + r0 * cols, c);
            });
        });
    else
        with_vpt<4>(odd && c <= kTwoPerLane ? 0 : pick_vpt(c), odd, [&](auto V, auto O) {
            softmax_bw_wave_kernel<V(), O()><<<grid, 256, 0, s>>>(y, dy, dx, r, c);
        });
}

template <int MODE>
static void cross_entropy_launch(const float *logits, const float *targets, size_t used,
                                 size_t rows, size_t cols, const float *grad_loss, float *out,
                                 int *err_flag, hipStream_t s) {
    const unsigned grid = (unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock);
    const int r = (int)rows, c = (int)cols;
    const long u = (long)used;
    const bool odd = c % 4 != 0 || !aligned16(logits) || (MODE == 1 && !aligned16(out));
    const int p = pick_block_p(c);
    if (MODE == 0 && !odd && (p == 1 || p == 2)) {
        const unsigned pairs = (unsigned)((rows + 1) / 2);
        if (p == 1)
            cross_entropy_rows2_kernel<1><<<pairs, kBlockThreads, 0, s>>>(logits, targets, u, r, c, out, err_flag);
        else
            cross_entropy_rows2_kernel<2><<<pairs, kBlockThreads, 0, s>>>(logits, targets, u, r, c, out, err_flag);
        return;
    }
    if constexpr (MODE == 0) {
        // Odd rows a little past the other kernels' 1027 columns: half of a
        // workgroup of 512 would hold no vector (8192 x 1029 9.2 us against 18.7,
        // 60000 x 1101 45 against 112).
        if (odd && p > 0 && c <= 1152) {
            cross_entropy_wave_kernel<8, 0, true><<<grid, 256, 0, s>>>(logits, targets, u, r, c,
                                                                       grad_loss, out, err_flag);
            return;
        }
    }
    const size_t out_row = MODE == 0 ? 1 : cols;  // floats of `out` per row
    if (p < 0)
        row_runs(rows, [&](size_t r0, unsigned n) {
            cross_entropy_loop_kernel<MODE><<<n, kBlockThreads, 0, s>>>(
                logits + r0 * cols, targets + r0, u - (long)r0, c, (float)r, grad_loss,
                out + r0 * out_row, err_flag);
        });
    else if (p > 0)
        with_block_p(p, odd, [&](auto P, auto O) {
            row_runs(rows, [&](size_t r0, unsigned n) {
                cross_entropy_block_kernel<P(), MODE, O()><<<n, kBlockThreads, 0, s>>>(
                    logits + r0 * cols, targets + r0, u - (long)r0, r, c, grad_loss,
                    out + r0 * out_row, err_flag);
            });
        });
    else
        with_vpt<4>(one_per_lane(c, odd) ? 0 : pick_vpt(c), odd, [&](auto V, auto O) {
            cross_entropy_wave_kernel<V(), MODE, O()><<<grid, 256, 0, s>>>(
                logits, targets, u, r, c, grad_loss, out, err_flag);
        });
}

void cross_entropy_rows(const float *logits, const float *targets, size_t used, size_t rows,
                        size_t cols, float *row_values, int *err_flag, hipStream_t s) {
    if (!rows || !cols) return;
    cross_entropy_launch<0>(logits, targets, used, rows, cols, nullptr, row_values, err_flag, s);
}

void cross_entropy_backward_rows(const float *logits, const float *targets, size_t used,
                                 size_t rows, size_t cols, const float *grad_loss, float *grad,
                                 int *err_flag, hipStream_t s) {
    if (!rows || !cols) return;
    cross_entropy_launch<1>(logits, targets, used, rows, cols, grad_loss, grad, err_flag, s);
}

}  // namespace k
}  // namespace clove
