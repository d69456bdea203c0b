// gemm_bf16x3.hip -- C = A.B in f32 on the bf16 matrix cores, every f32 value
// carried whole as three bf16 pieces.
//
// v_mfma_f32_32x32x16_bf16 does the multiply-adds of eight
// v_mfma_f32_32x32x2_f32 in half the cycles of one: an f32 product as six bf16
// products still runs at 2.6 times the FP32 MFMA's rate.
// The pieces (bf16x3.h) hold every bit of an operand, so a product with a
// one-hot or power-of-two operand is exact, as in f32; the MFMAs accumulate in
// f32.
// Error against float64 (normal data, 4096 x K x 4096, relative 2-norm): K =
// 64 1.13e-7, 512 3.5e-7, 1024 4.8e-7, 4096 1.02e-6 -- the FP32 MFMA kernel
// 1.44e-7, 4.1e-7, 5.7e-7, 1.15e-6.
//
// Operands go in as 2^24 x (bf16x3.h), which holds every value below 2^103.  One
// past that, an infinity, a NaN or a sum past 2^79 is not for this scheme: the
// workgroup that meets one computes its tile again from the f32 values on the
// FP32 MFMA (redo below), so the result is then what f32 arithmetic gives, and
// the tile takes 2.6 times as long (4096^3 with an infinity in every tile row
// 1701 us against 645, 948 on the FP32 tiles).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "bf16x3.h"
#include "gemm_common.h"
#include "launch.hpp"

namespace clove {
namespace k {

namespace {

constexpr uint32_t kOutside = 0x80000000u;     // past the end of both operands (each under 2 GiB)
// One operand's share of a thread: OCT octets (eight consecutive k of one row
// of A, or of one column of B) of a slab of R rows.  KC: the operand's k are
// consecutive in memory (A, or B given transposed): an octet is two 16-byte
// loads.  Otherwise its rows are (B, or A given transposed): lanes 0-31 of a
// wave take 32 consecutive rows of octet 0 and lanes 32-63 of octet 1, each
// load 128 bytes of two k.
// In LDS a piece of a slab is [R][BK] bf16, octet o of row r in slot o ^ ((r >>
// 4) & 1) at BK = 16, o ^ ((r >> 2) & 3) at BK = 32: a wave's fragment read
// (lane l: row l % 32, octet 2 step + l / 32) then touches every bank group
// once per phase, and so do the KC = false stores.
template <int R, int BK, int T, bool KC, bool FUSED>
struct Operand {
    static constexpr int OPR = BK / 8;  // octets per row
    static constexpr int OCT = R * OPR / T;
    static constexpr int kPiece = R * BK * 2;  // bytes of one piece of a slab
    static_assert(OCT >= 1 && R * OPR % T == 0, "whole octets per thread");
    static __device__ __forceinline__ int slot(int r, int o) {
        return r * (BK * 2) + ((o ^ (BK == 16 ? (r >> 4) & 1 : (r >> 2) & 3)) << 4);
    }
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off[OCT];   // byte offset of the octet's first value at k = 0, or kOutside
    int dst[OCT];        // its byte offset in each piece of a stage
    int row[OCT], oct[OCT];
    uint32_t ld;         // bytes from one k to the next (KC = false)
    float x[OCT][8];

    __device__ __forceinline__ void init(const float *base, int rows, int K, int r0) {
        rsrc = make_rsrc(base, (uint32_t)((size_t)rows * K * 4));
        ld = (uint32_t)rows * 4u;
#pragma unroll
        for (int u = 0; u < OCT; ++u) {
            const int p = u * T + (int)threadIdx.x;
            const int r = KC ? p / OPR : p / (32 * OPR) * 32 + (p & 31);
            const int o = KC ? p % OPR : (p >> 5) % OPR;
            row[u] = r;
            oct[u] = o;
            dst[u] = slot(r, o);
            off[u] = r0 + r >= rows ? kOutside
                     : KC           ? ((uint32_t)(r0 + r) * (uint32_t)K + 8u * o) * 4u
                                    : 8u * o * ld + (uint32_t)(r0 + r) * 4u;
        }
    }
    // slab of k0 .. k0 + BK - 1, all below k_end
    __device__ __forceinline__ void load(int k0) {
#pragma unroll
        for (int u = 0; u < OCT; ++u) load_octet(u, k0);
    }
    __device__ __forceinline__ void load_octet(int u, int k0) {
        {
            if constexpr (KC) {
                const f4 v0 = __builtin_bit_cast(
                    f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off[u], k0 * 4, 0));
                const f4 v1 = __builtin_bit_cast(
                    f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off[u] + 16, k0 * 4, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[u][e] = v0[e];
                    x[u][4 + e] = v1[e];
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    x[u][e] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)off[u],
                                                                    (int)((uint32_t)(k0 + e) * ld), 0));
            }
        }
    }
    // a last slab that K (or the split) ends inside: k at or past k_end are 0
    __device__ __forceinline__ void load_tail(int k0, int k_end) {
#pragma unroll
        for (int u = 0; u < OCT; ++u)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t step = KC ? (uint32_t)(k0 + e) * 4u : (uint32_t)(k0 + e) * ld;
                const uint32_t o =
                    off[u] != kOutside && k0 + 8 * oct[u] + e < k_end ? off[u] + step : kOutside;
                x[u][e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)o, 0, 0));
            }
    }
    // the pieces of the loaded slab into `stage` (piece p at p * kPiece)
    __device__ __forceinline__ void store(char *stage) const {
#pragma unroll
        for (int u = 0; u < OCT; ++u) store_octet(u, stage);
    }
    __device__ __forceinline__ void store_octet(int u, char *stage) const {
        {
            u4 p[3];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                unsigned a, b, c;
                split_pair<true, FUSED>(x[u][2 * e], x[u][2 * e + 1], &a, &b, &c);
                p[0][e] = a;
                p[1][e] = b;
                p[2][e] = c;
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<u4 *>(stage + q * kPiece + dst[u]) = p[q];
        }
    }
    // the f32 values themselves, rows of kPitch floats (the redo path)
    static constexpr int kPitch = BK + 4;
    __device__ __forceinline__ void store_f32(float *s) const {
#pragma unroll
        for (int u = 0; u < OCT; ++u) {
            f4 *d = reinterpret_cast<f4 *>(s + row[u] * kPitch + 8 * oct[u]);
            d[0] = (f4){x[u][0], x[u][1], x[u][2], x[u][3]};
            d[1] = (f4){x[u][4], x[u][5], x[u][6], x[u][7]};
        }
    }
};

// A workgroup of T / 64 waves, each WM x WN of a BM x BN tile, walking slabs of
// BK k.  While slab s multiplies out of one LDS stage, slab s + 1 (in
// registers) is split into the other and the f32 values of slab s + 2 set out;
// one barrier per slab.  The split's operations are laid between the MFMAs,
// block row by block row: written before them they ran first and the matrix
// cores waited (a lone 256 x 128 workgroup per CU: 1.4 against 1.07 us per
// slab; 128 x 128 x 32 with eight waves 0.8 against 0.56 per 16 k).
//
// What bounds it: large products run at the card's power limit (4096^3 in 256
// x 128 tiles, two workgroups per CU: 607-645 us by box against 944-1010 for
// the FP32 MFMA kernel, 213-226 TFLOP/s of f32, 1360 of bf16; the MFMA pipe 78%
// busy under the counters, the clock 1.74 GHz of 2.39 in an unprofiled run, where
// the same launch on zeros keeps 2.39 and takes 435; a large bf16 library product
// reaches 1321 TFLOP/s on the
// same card).  Waves of 128 x 64 keep LDS reads at half its rate; 64 x 64
// waves (128 x 128 tiles, three workgroups per CU) take 738 us there but fill
// the chip from smaller products; eight 64 x 32 waves on one 128 x 128 tile
// with 32-deep slabs are quickest where a CU gets a single tile (256 x 4096 x
// 4096: 56 us against 80).
template <int BM, int BN, int BK, int WM, int WN, int T, int MINW, bool EPI, bool TA, bool TB>
__global__ void __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(MINW)))
gemm_bf16x3_kernel(GemmArgs g) {
    // (128-row tiles take the split's remainder as an FMA: 128 x 4096 x 16384 115
    // against 119 us, 65536 x 1024 x 256 193 against 198; 4096 x 256 x 16384 the
    // other way, 206 against 194)
    using OpA = Operand<BM, BK, T, !TA, BM == 128>;
    using OpB = Operand<BN, BK, T, TB, BM == 128>;
    constexpr int SA = 3 * OpA::kPiece, STAGE = SA + 3 * OpB::kPiece;  // bytes
    constexpr int IB = WM / 32, JB = WN / 32, WNS = BN / WN;
    static_assert((BM / WM) * (BN / WN) * 64 == T, "the waves cover the tile");
    static_assert((BM + BN) * OpA::kPitch * 4 <= 2 * STAGE, "the redo path's slab fits");
    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];
    int tile;
    if (!gemm_tile(g, &tile)) return;  // padding of the grid (before any barrier)
    const int M = g.M, N = g.N;
    const int split = blockIdx.y;
    const int m0 = (tile / g.tiles_n) * BM, n0 = (tile % g.tiles_n) * BN;
    const int k_begin = split * g.k_per_split;
    const int k_end = min(g.K, k_begin + g.k_per_split);
    const int slabs = (k_end - k_begin + BK - 1) / BK;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    const int wm0 = (wave / WNS) * WM, wn0 = (wave % WNS) * WN;
    OpA a;
    OpB b;
    a.init(g.A, M, g.K, m0);
    b.init(g.B, N, g.K, n0);
    auto load = [&](int s) {
        const int k0 = k_begin + s * BK;
        if (k0 + BK <= k_end) {
            a.load(k0);
            b.load(k0);
        } else {
            a.load_tail(k0, k_end);
            b.load_tail(k0, k_end);
        }
    };
    f16v acc[IB][JB];
    auto clear = [&] {
#pragma unroll
        for (int i = 0; i < IB; ++i)
#pragma unroll
            for (int j = 0; j < JB; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    };
    clear();
    auto store = [&](int s) {
        char *st = smem + (s & 1) * STAGE;
        a.store(st);
        b.store(st + SA);
    };
    // this lane's octet of each MFMA step in a 32-row block
    int rd[BK / 16];
#pragma unroll
    for (int t = 0; t < BK / 16; ++t) rd[t] = OpA::slot(l32, 2 * t + h);
    // Slab s out of its stage; with NEXT, slab s + 1 (in registers) is split
    // into the other stage, and with LOAD, slab s + 2 sets out.
    auto step = [&](int s, auto next, auto load_more) {
        const char *st = smem + (s & 1) * STAGE;
        char *nst = smem + ((s + 1) & 1) * STAGE;
        const int k2 = k_begin + (s + 2) * BK;
        bf8 fb[JB][3], fa[2][3];
        auto read_a = [&](int r) {
#pragma unroll
            for (int q = 0; q < 3; ++q)
                fa[r & 1][q] = *reinterpret_cast<const bf8 *>(
                    st + q * OpA::kPiece + (wm0 + 32 * (r % IB)) * (BK * 2) + rd[r / IB]);
        };
        constexpr int REG = IB * (BK / 16), UNITS = OpA::OCT + OpB::OCT;
#pragma unroll
        for (int r = 0; r < REG; ++r) {
            if (r % IB == 0) {
#pragma unroll
                for (int j = 0; j < JB; ++j)
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        fb[j][q] = *reinterpret_cast<const bf8 *>(
                            st + SA + q * OpB::kPiece + (wn0 + 32 * j) * (BK * 2) + rd[r / IB]);
                read_a(r);
            }
            if ((r + 1) % IB != 0) read_a(r + 1);
#pragma unroll
            for (int p = 0; p < 6; ++p)
#pragma unroll
                for (int j = 0; j < JB; ++j)
                    acc[r % IB][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        fa[r & 1][kPieceA[p]], fb[j][kPieceB[p]], acc[r % IB][j], 0, 0, 0);
#pragma unroll
            for (int u = r * UNITS / REG; u < (r + 1) * UNITS / REG; ++u) {
                if constexpr (decltype(next)::value) {
                    if (u < OpA::OCT) a.store_octet(u, nst);
                    else b.store_octet(u - OpA::OCT, nst + SA);
                }
                if constexpr (decltype(load_more)::value) {
                    if (u < OpA::OCT) a.load_octet(u, k2);
                    else b.load_octet(u - OpA::OCT, k2);
                }
            }
            // the largest tile: one MFMA, then seven of the split's operations
            // (what its 32 cycles leave room for), region by region
            if constexpr (BM == 256 && decltype(next)::value) {
#pragma unroll
                for (int n = 0; n < 6 * JB; ++n) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 7, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        lds_barrier();
    };
    using Yes = std::true_type;
    using No = std::false_type;
    load(0);
    store(0);
    if (slabs > 1) load(1);
    lds_barrier();
    // whole slabs are loaded without a branch in the step
    const int whole = (k_end - k_begin) / BK;
    int s = 0;
    for (; s + 2 < whole; ++s) step(s, Yes{}, Yes{});
    for (; s + 1 < slabs; ++s) {
        const bool tail = s + 2 < slabs;  // (then s + 2 is the partial slab)
        step(s, Yes{}, No{});
        if (tail) load(s + 2);
    }
    step(s, No{}, No{});

    // Out of the pieces' range?  An infinite or NaN operand, or one that rounds to
    // infinity in bf16, always gives a sum that is not finite, and 0 times that is
    // NaN: one FMA a sum, between the last slab's MFMAs.
    float zero[IB];
#pragma unroll
    for (int i = 0; i < IB; ++i) {
        zero[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < JB; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) zero[i] = __builtin_fmaf(acc[i][j][e], 0.0f, zero[i]);
    }
    bool bad = false;
#pragma unroll
    for (int i = 0; i < IB; ++i) bad = bad || zero[i] != 0.0f;
    float unscale = kSumUnscale;
    if (__builtin_expect(__syncthreads_or(bad), 0)) {
        unscale = 1.0f;
        // redo: the same tile from the f32 values on v_mfma_f32_32x32x2_f32,
        // one slab in LDS at a time.
        clear();
        float *sA = reinterpret_cast<float *>(smem), *sB = sA + BM * OpA::kPitch;
        load(0);
        for (int s = 0; s < slabs; ++s) {
            a.store_f32(sA);
            b.store_f32(sB);
            __syncthreads();
            if (s + 1 < slabs) load(s + 1);
#pragma unroll 1
            for (int gk = 0; gk < BK / 8; ++gk) {
                f4 va[IB], vb[JB];
#pragma unroll
                for (int i = 0; i < IB; ++i)
                    va[i] = *reinterpret_cast<const f4 *>(sA + (wm0 + 32 * i + l32) * OpA::kPitch +
                                                          8 * gk + 4 * h);
#pragma unroll
                for (int j = 0; j < JB; ++j)
                    vb[j] = *reinterpret_cast<const f4 *>(sB + (wn0 + 32 * j + l32) * OpA::kPitch +
                                                          8 * gk + 4 * h);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int i = 0; i < IB; ++i)
#pragma unroll
                        for (int j = 0; j < JB; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[i][t], vb[j][t],
                                                                             acc[i][j], 0, 0, 0);
            }
            __syncthreads();
        }
    }

    // Accumulator element e of block (i, j) is tile element (r, c) with
    // r = wm0 + 32*i + 8*(e/4) + 4*h + e%4 and c = wn0 + 32*j + l%32.
    // A row of blocks is unscaled in its registers before its first store (a
    // product next to each store shares one register, which makes the stores wait
    // on one another).
    auto unscale_row = [&](int i) {
#pragma unroll
        for (int j = 0; j < JB; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] *= unscale;
                asm volatile("" : "+v"(acc[i][j][e]));
            }
    };
    if (g.splits == 1) {
        float bc[JB];  // per-column bias, loaded before any store
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            const int col = n0 + wn0 + 32 * j + l32;
            bc[j] = EPI && g.epi.bias_mode == GEMM_BIAS_COL && col < N ? g.epi.bias[col] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < IB; ++i) {
            unscale_row(i);
#pragma unroll
            for (int e = 0; e < 16; ++e)
#pragma unroll
                for (int j = 0; j < JB; ++j) {
                    const int row = m0 + wm0 + 32 * i + 8 * (e / 4) + 4 * h + (e % 4);
                    const int col = n0 + wn0 + 32 * j + l32;
                    float v = acc[i][j][e];
                    if constexpr (EPI) v = epilogue(g.epi, v, row, col, N, &bc[j]);
                    if (row < M && col < N) g.C[(size_t)row * N + col] = v;
                }
        }
        return;
    }
    float *part = g.ws + ((size_t)split * g.tiles + tile) * (BM * BN);
#pragma unroll
    for (int i = 0; i < IB; ++i) {
        unscale_row(i);
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
            for (int j = 0; j < JB; ++j)
                part[(wm0 + 32 * i + 8 * (e / 4) + 4 * h + (e % 4)) * BN + wn0 + 32 * j + l32] =
                    acc[i][j][e];
    }
}

template <int BM, int BN, int BK, int WM, int WN, int T, int MINW>
void launch(const GemmPlan &p, const GemmArgs &g, bool ta, bool tb, hipStream_t s) {
    const dim3 grid((unsigned)(g.per_xcd * 8), (unsigned)p.splits);
    const bool epi = p.splits == 1 &&
                     (g.epi.bias_mode != GEMM_BIAS_NONE || g.epi.act != GEMM_ACT_NONE);
    if (ta)
        gemm_bf16x3_kernel<BM, BN, BK, WM, WN, T, MINW, false, true, false><<<grid, T, 0, s>>>(g);
    else if (tb)
        gemm_bf16x3_kernel<BM, BN, BK, WM, WN, T, MINW, false, false, true><<<grid, T, 0, s>>>(g);
    else if (epi)
        gemm_bf16x3_kernel<BM, BN, BK, WM, WN, T, MINW, true, false, false><<<grid, T, 0, s>>>(g);
    else
        gemm_bf16x3_kernel<BM, BN, BK, WM, WN, T, MINW, false, false, false><<<grid, T, 0, s>>>(g);
}

}  // namespace

void gemm_bf16x3(const GemmPlan &p, const GemmArgs &g, bool ta, bool tb, hipStream_t s) {
    if (p.x3 == GEMM_X3_256x128) launch<256, 128, 16, 128, 64, 256, 2>(p, g, ta, tb, s);
    else if (p.x3 == GEMM_X3_128x128) launch<128, 128, 16, 64, 64, 256, 2>(p, g, ta, tb, s);
    else launch<128, 128, 32, 64, 32, 512, 2>(p, g, ta, tb, s);
}

}  // namespace k
}  // namespace clove
