// flash_attention.hip -- attention prefill (FlashAttention) and RoPE on CDNA4.
//
// Reference: the fused FlashAttention step of the lazy path (pattern
// MatMul -> Softmax -> MatMul with RoPE / ScalarMul on q and k, lazy.rs:
// 1621-1690; kernel lazy.rs:4821-4909) and the rope op (backend.rs:
// 2797-2826).  The WGSL runs one thread per query row of a single head,
// always applies RoPE and a causal mask, uses (1 + x/8)^8 for exp and keeps
// the key tile in a 1024-float array (so head_dim > 32 overflows it).  Here:
// batched, multi-head, causal and RoPE as flags, an exact exp, any length.
//
// Head dims up to 128 that are multiples of 8 run attention_x3_kernel below, on
// the bf16 matrix cores with every f32 value as three bf16 pieces (bf16x3.h);
// every other head dim, and calls that attention_x3_plan prices as faster there
// (short ones above all), run attention16_kernel (attention_general.hip),
// 16-query waves on the FP32 MFMA.  Key blocks of 32 are staged through LDS
// (double-buffered, one barrier per block).  k is rotated before the kernel,
// once per element (a rotation inside it would be repeated by every query block
// that stages the same keys).  The products run in TRANSPOSED form:
//   S^T = K . Q^T   (A = K tile from LDS, B = the wave's Q^T in registers)
//   O^T += V^T . P^T (A = V^T from LDS, B = P^T straight from S^T's registers)
// so lane l always works for query l%32: its S^T accumulator holds that
// query's scores for 16 of the block's 32 keys (the other 16 sit in lane
// l^32), and its O^T accumulator holds that query's output for 16 of every
// 32 head dimensions.  The online-softmax statistics (running max and sum)
// and the rescale of O are therefore per-lane scalars: a row reduction is
// 15 in-register ops plus one shuffle with lane l^32, and P never goes
// through LDS.
//
// Work order: workgroup L takes query block nqb-1 - L/(B*H) of (batch, head)
// L % (B*H).  Under the causal mask a query block's cost grows with its
// index, so this starts the heaviest blocks of every head first (a
// longest-first list schedule: with 64 slots per XCD at S = 4096, H = 32 its
// makespan is the ideal 33 block-units, where walking one head after another
// took 49).  Workgroups are dealt to the 8 XCDs round-robin (L % 8), so when
// B*H is a multiple of 8 each XCD serves a fixed set of heads and their K
// and V stay in its L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "attention16.h"
#include "bf16x3.h"
#include "launch.hpp"
#include "wave.h"

namespace clove {
namespace k {

namespace {

typedef float f16v __attribute__((ext_vector_type(16)));

// Writes a lane's query: o[j][e] = O[query][32j + 8(e/4) + 4hh + e%4], four
// consecutive dims per e/4; the output itself, or with the keys split over
// workgroups the unnormalised sum and (m, lsum) for attention_merge_kernel.
// unscale: the factor that o is to be brought back by.
template <int D, int kJ>
__device__ __forceinline__ void attn_store(const AttnArgs &a, int b, int h, int query, int split,
                                           int hh, const f16v (&o)[kJ], float m, float lsum,
                                           float unscale) {
    const size_t row = (size_t)b * a.S + query;
    float inv = unscale, *orow = a.out + (row * a.H + h) * a.D;
    if (a.splits > 1) {
        const size_t rows = (size_t)a.B * a.S * a.H, at = (size_t)split * rows + row * a.H + h;
        orow = a.part + at * a.D;
        if (hh == 0) {
            float *st = a.part + (size_t)a.splits * rows * a.D + 2 * at;
            st[0] = m;
            st[1] = lsum;
        }
    } else {
        inv = lsum > 0.0f ? unscale / lsum : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int d = 32 * j + 8 * u + 4 * hh;
            const cl_f4 r = {o[j][4 * u] * inv, o[j][4 * u + 1] * inv, o[j][4 * u + 2] * inv,
                             o[j][4 * u + 3] * inv};
            if (d < a.D) *reinterpret_cast<cl_f4 *>(orow + d) = r;
        }
}

// The workgroup's queries from q0 on, 32 per wave, over key blocks [blk0, blk1),
// on the FP32 MFMA (the redo path of attention_x3_kernel); smem holds
// attn_f32_floats<D> floats.  D is the size the tiles are laid out for, a.D (a
// multiple of 8) the head dim: dims past it load as zero.
template <int D>
constexpr int attn_f32_floats() { return 2 * kBK * (2 * D + 12); }
template <int D, bool CAUSAL, int T>
__device__ __forceinline__ void attention_f32(const AttnArgs &a, const int q0, const int bh,
                                              const int split, const int blk0, const int blk1,
                                              float *smem) {
    constexpr int kPK = D + 4;  // K tile pitch (16-byte reads by 32 rows: no conflicts)
    constexpr int kPV = D + 8;  // V tile pitch (rows r and r+4 land 32 banks apart)
    constexpr int kG = D / 8;   // K-groups of 8 dims
    constexpr int kJ = D / 32;  // 32-dim blocks of O^T
    constexpr int kVec = (kBK * D / 4 + T - 1) / T;  // 16-byte tile loads per thread (K and V each)
    float *const sK = smem, *const sV = smem + 2 * kBK * kPK;  // two buffers each
    const int h = bh % a.H, b = bh / a.H;

    const int DD = a.D, HD = a.H * DD;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, hh = lane >> 5;
    const int query = q0 + wave * 32 + l32;
    const bool q_ok = query < a.S;
    const float *qrow = a.q + ((size_t)b * a.S + (q_ok ? query : 0)) * HD + (size_t)h * DD;

    // this wave's Q^T fragment: dims 8g + 4hh .. +3 of its query, times the
    // softmax scale.  Scaling here also makes the Q loads complete before the
    // key loop: first used inside it, they would make the compiler wait for
    // every outstanding load (the next tile's included) at each block.
    // With RoPE, q's pairs (dims 8g + 4hh + {0,1} and {2,3}, whole pairs in
    // this lane) are rotated here, with the arithmetic of the RoPE pass
    // (rope_rows_kernel), before the scale: the same values that pass would
    // have stored, without its read and write of q.
    const float2 *trow = a.rope_tab && q_ok
                             ? a.rope_tab + (size_t)(query + a.q_pos - a.tab_pos0) * (DD / 2)
                             : nullptr;
    // Scores are kept in base-2 units: q carries scale * log2(e), so a
    // softmax weight is exp2(s - m) with no multiply per score.
    const float qscale = a.scale * 1.44269504088896341f;
    cl_f4 qf[kG];
#pragma unroll
    for (int g = 0; g < kG; ++g) {
        const bool in = 8 * g < DD;
        cl_f4 v = q_ok && in ? *reinterpret_cast<const cl_f4 *>(qrow + 8 * g + 4 * hh)
                             : (cl_f4){0.f, 0.f, 0.f, 0.f};
        if (trow && in) {
            const float2 t0 = trow[4 * g + 2 * hh], t1 = trow[4 * g + 2 * hh + 1];
            cl_f4 r;
            r.x = v.x * t0.x - v.y * t0.y;
            r.y = v.x * t0.y + v.y * t0.x;
            r.z = v.z * t1.x - v.w * t1.y;
            r.w = v.z * t1.y + v.w * t1.x;
            v = r;
        }
        qf[g] = v * qscale;
    }

    // keys this wave's queries can see (whole blocks past them are skipped)
    int k_wave = a.Sk;
    if (CAUSAL) k_wave = min(k_wave, min(q0 + wave * 32 + 31, a.S - 1) + a.q_pos - a.k_pos + 1);
    // this lane's query sees keys t < lim
    const int lim = q_ok ? (CAUSAL ? min(a.Sk, query + a.q_pos - a.k_pos + 1) : a.Sk) : 0;

    // K and V tiles come through buffer loads over this batch's [Sk, H*D]
    // rows: a key past Sk gets an offset past the end and reads as zeros.  A
    // guarded ordinary load would become a branch that the compiler closes
    // with a wait for all loads, which exposes the whole load latency of
    // every block instead of overlapping it with the block before.
    constexpr uint32_t kOutside = 0x80000000u;  // the host keeps Sk*H*D*4 < 2^31
    const uint32_t kv_bytes = (uint32_t)a.Sk * (uint32_t)HD * 4u;
    const __amdgpu_buffer_rsrc_t rsrc_k = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.k + (size_t)b * a.Sk * HD), (short)0, (int)kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_v = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.v + (size_t)b * a.Sk * HD), (short)0, (int)kv_bytes, 0x00020000);
    cl_f4 rk[kVec], rv[kVec];
    // Each load's offset within the tile (key and dims) is fixed per lane;
    // the block's first key enters as the scalar offset, so a block of keys
    // all below Sk costs no per-lane arithmetic.  (kb < Sk always, and the
    // host keeps Sk * H * D * 4 < 2^31, so the scalar offset cannot carry
    // kOutside round.)
    uint32_t toff[kVec];
    int tkey[kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const int idx = threadIdx.x + T * i;
        const int key = idx / (D / 4), dq = idx % (D / 4);
        tkey[i] = key;
        const bool in = 4 * dq < DD && (kBK * D / 4 % T == 0 || idx < kBK * D / 4);
        toff[i] = in ? ((uint32_t)key * (uint32_t)HD + (uint32_t)(h * DD + 4 * dq)) * 4u : kOutside;
    }
    auto load_tile = [&](int kb) {
        const int soff = kb * HD * 4;
        uint32_t off[kVec];
#pragma unroll
        for (int i = 0; i < kVec; ++i) off[i] = toff[i];
        if (kb + kBK > a.Sk) {  // the last block: keys past Sk read as zeros
            asm volatile("");   // (keeps this a branch, not selects every block pays for)
#pragma unroll
            for (int i = 0; i < kVec; ++i) off[i] = kb + tkey[i] < a.Sk ? toff[i] : kOutside;
        }
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            rk[i] = __builtin_bit_cast(cl_f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_k, (int)off[i], soff, 0));
            rv[i] = __builtin_bit_cast(cl_f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_v, (int)off[i], soff, 0));
        }
    };
    auto store_tile = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            const int idx = threadIdx.x + T * i;
            if (kBK * D / 4 % T != 0 && idx >= kBK * D / 4) continue;
            const int key = idx / (D / 4), dq = idx % (D / 4);
            *reinterpret_cast<cl_f4 *>(sK + buf * kBK * kPK + key * kPK + 4 * dq) = rk[i];
            *reinterpret_cast<cl_f4 *>(sV + buf * kBK * kPV + key * kPV + 4 * dq) = rv[i];
        }
    };

    float m = -INFINITY, lsum = 0.0f;
    f16v o[kJ];
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[j][e] = 0.f;

    if (blk0 < blk1) {
        load_tile(blk0 * kBK);
        store_tile(blk0 & 1);
    }
    __syncthreads();
    for (int blk = blk0; blk < blk1; ++blk) {
        const int kb = blk * kBK;
        const int cur = blk & 1;
        const bool more = blk + 1 < blk1;
        if (more) load_tile(kb + kBK);

        if (kb < k_wave) {
            const float *K = sK + cur * kBK * kPK;
            const float *V = sV + cur * kBK * kPV;
            // S^T = K . Q^T: s[i] is the score of key kb + 8(i/4) + 4hh + i%4
            // (in base-2 units).  One accumulator: splitting the chain over
            // two measured the same and cost 16 adds per block.
            f16v s;
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = 0.f;
            // Raised wave priority over the two MFMA blocks (QK and PV): a
            // wave issuing MFMAs keeps the arbiter while the other waves on
            // its SIMD do their softmax VALU work, tile loads and stores in
            // the gaps (S = 4096, H = 32, D = 128: 116.2 -> 124.9 TFLOP/s,
            // same results bit for bit).
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int g = 0; g < kG; ++g) {
                const cl_f4 kf = *reinterpret_cast<const cl_f4 *>(K + l32 * kPK + 8 * g + 4 * hh);
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[t], qf[g][t], s, 0, 0, 0);
            }
            __builtin_amdgcn_s_setprio(0);
            // A block the whole wave sees (every key < Sk and, under the causal
            // mask, at or before the wave's first query) skips the mask.
            // The empty asm statement keeps the mask a branch: without it the
            // compiler turns it into selects that every block pays for.
            const int qw0 = q0 + wave * 32;
            bool full = kb + kBK <= a.Sk && qw0 + 32 <= a.S;
            if (CAUSAL) full = full && kb + kBK - 1 + a.k_pos <= qw0 + a.q_pos;
            if (!full) {
                asm volatile("");
                const int vis = lim - kb - 4 * hh;  // s[i] visible iff 8(i/4) + i%4 < vis
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = 8 * (i / 4) + (i % 4) < vis ? s[i] : -INFINITY;
            }
            float mloc = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; ++i) mloc = fmaxf(mloc, s[i]);
            mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
            // Lazy rescale: the running max m moves only when some query of the
            // wave sees a score more than kSlack above it.  Scores up to
            // m + kSlack give weights up to 2^kSlack, harmless in f32, and the
            // numerator O and the denominator lsum share m, so the result is
            // the same; the 16*kJ-multiply rescale of O is skipped on most
            // blocks.  (m = -inf, no visible key yet, always updates.)
            constexpr float kSlack = 8.0f;
            const bool grow = __any(mloc > m + kSlack);
            if (grow) {
                const float m_new = fmaxf(m, mloc);
                const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
                lsum *= alpha;
#pragma unroll
                for (int j = 0; j < kJ; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) o[j][e] *= alpha;
                m = m_new;
            }
            // exp2(-inf) is 0, so masked scores need no test; only a lane
            // with no visible key yet (m = -inf, every score of the block
            // -inf) takes 0 as its max so that -inf - m is not NaN.
            const float mz = m == -INFINITY ? 0.0f : m;
            float ps = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] = __builtin_amdgcn_exp2f(s[i] - mz);
                ps += s[i];
            }
            ps += __shfl_xor(ps, 32, 64);
            lsum += ps;
            // O^T += V^T . P^T (step i pairs key 8(i/4)+i%4 of half 0 with key
            // 8(i/4)+4+i%4 of half 1, as S^T's layout holds them)
            // the kJ output blocks are independent accumulators: consecutive
            // MFMAs alternate between them
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = 8 * (i / 4) + 4 * hh + (i % 4);
#pragma unroll
                for (int j = 0; j < kJ; ++j) {
                    const float vv = V[key * kPV + 32 * j + l32];
                    o[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, s[i], o[j], 0, 0, 0);
                }
                // bound how far the V reads are hoisted (all 64 at once cost 64
                // registers and an occupancy step)
                if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if (more) store_tile(cur ^ 1);
        __syncthreads();
    }

    if (q_ok) attn_store<D, kJ>(a, b, h, query, split, hh, o, m, lsum, 1.0f);
}

// Head dims up to 128 that are multiples of 8, on the bf16 matrix cores, f32
// values as three bf16 pieces (bf16x3.h): the same transposed scheme on v_mfma_f32_32x32x16_bf16,
//   S^T = K . Q^T    (A = K pieces from LDS, B = the wave's Q^T pieces in registers)
//   O^T += V^T . P^T (A = V^T pieces from LDS, B = P^T split in registers)
// with lane l again on query l % 32: the accumulators have the layout of the
// f32 MFMA's.  The k order of a product is free as long as both operands agree,
// so PV's step s gives lane half h the keys 16s + 4h + {0..3, 8..11}: those
// whose scores the lane already holds, and the order V is stored in.
//  * K and V tiles of 32 keys are split once per workgroup on their way into
//    LDS: K as [key][D], V transposed as [dim][32 keys], in 16-byte octets
//    whose slots are XOR-permuted against bank conflicts in a wave's fragment
//    reads (0.4 conflict cycles per LDS instruction are left, reads and stores
//    together).  Tile n + 1 (in registers) is split while tile n multiplies,
//    its octet stores laid between the MFMAs, and tile n + 2 sets out.
//  * NW waves share a tile: eight (256 queries) at D = 128, where the split of
//    a tile is a third of the VALU work of four waves; four below.
//  * The keys of a query block may be split over workgroups (attention_x3_plan);
//    attention_merge_kernel then adds the parts.
// What bounds it: at 4096 queries, 32 heads of 128, the matrix cores at the clock
// that the load leaves them (2.0 GHz of 2.39 unprofiled, 65% busy under the
// counters: non-causal 1170-1220 us, 1350-1410 TFLOP/s of bf16; causal with RoPE
// 670-690 us with k's pass, against 1066 for the FP32 MFMA kernel; D = 64 391
// against 555, D = 96 and 104 two thirds of theirs); below that, one workgroup's chain per key
// block (3.9 us at D = 128 alone on its CU, 1.8 at D = 64), hence the splits.
// Error against float64 is below that kernel's (2.9e-7 against 3.7e-7 at 377
// keys, 5.9e-7 at 1031 keys unsplit, less split).
//  * q (times scale * log2(e)), k, the weights and v go in as 2^24 x; a score's
//    factor of 2^48 comes off in the exponent's FMA, the output's at the end.
//    (The weights' factor has to be a product: taken into the exponent, 24 more
//    there costs the subtraction before it five bits, an error of 2e-7 against
//    8e-8.)  A workgroup that ends with a sum that is not finite (an infinity, a
//    NaN, a value of 2^103, a score of 2^79, a v around 2^65 over many keys)
//    computes its queries again with attention_f32 (4096 causal queries with an
//    infinity in every head's v 1615 us against 644).
template <int D, bool CAUSAL, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
attention_x3_kernel(AttnArgs a) {
    constexpr int T = 64 * NW, QB = 32 * NW;
    constexpr int ST = D / 16;                 // QK steps
    constexpr int kJ = D / 32;                 // 32-dim blocks of O^T
    constexpr int KP = 32 * D * 2;             // bytes of one piece of K's tile, and of V's
    constexpr int STAGE = 6 * KP;
    constexpr int OCTS = 32 * D / 8;           // octets of a tile, K and V each
    constexpr int U = (OCTS + T - 1) / T;      // of a thread (whole waves go without)
    constexpr int kSmem = 2 * STAGE > attn_f32_floats<D>() * 4 ? 2 * STAGE : attn_f32_floats<D>() * 4;
    __shared__ __attribute__((aligned(16))) char smem[kSmem];

    // heaviest query blocks first, heads interleaved (see the file comment)
    const int BH = a.B * a.H;
    const int L = blockIdx.x, r = L % (BH * a.splits);
    const int bh = r % BH, split = r / BH;
    const int q0 = (a.nqb - 1 - L / (BH * a.splits)) * QB;
    const int h = bh % a.H, b = bh / a.H;
    const int DD = a.D, HD = a.H * DD;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, hh = lane >> 5;
    const int qw0 = q0 + wave * 32;
    const int query = qw0 + l32;
    const bool q_ok = query < a.S;

    // this wave's Q^T pieces: step g, slots 0..7 of lane half hh are dims 16g +
    // 8hh .. +7 of its query, rotated (with RoPE) and times 2^24 scale * log2(e),
    // in f32 as in attention_f32, before the split
    const float *qrow = a.q + ((size_t)b * a.S + (q_ok ? query : 0)) * HD + (size_t)h * DD;
    const float2 *trow = a.rope_tab && q_ok
                             ? a.rope_tab + (size_t)(query + a.q_pos - a.tab_pos0) * (DD / 2)
                             : nullptr;
    const float qscale = a.scale * 1.44269504088896341f * kPieceScale;
    bf8 qf[ST][3];
#pragma unroll
    for (int g = 0; g < ST; ++g) {
        u4 p[3];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int d0 = 16 * g + 8 * hh + 4 * c;
            const bool in = d0 < DD;
            cl_f4 v = q_ok && in ? *reinterpret_cast<const cl_f4 *>(qrow + d0)
                                 : (cl_f4){0.f, 0.f, 0.f, 0.f};
            if (trow && in) {
                const float2 t0 = trow[d0 / 2], t1 = trow[d0 / 2 + 1];
                cl_f4 r;
                r.x = v.x * t0.x - v.y * t0.y;
                r.y = v.x * t0.y + v.y * t0.x;
                r.z = v.z * t1.x - v.w * t1.y;
                r.w = v.z * t1.y + v.w * t1.x;
                v = r;
            }
            v = v * qscale;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                unsigned x, y, z;
                split_pair<false>(v[2 * e], v[2 * e + 1], &x, &y, &z);
                p[0][2 * c + e] = x;
                p[1][2 * c + e] = y;
                p[2][2 * c + e] = z;
            }
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) qf[g][q] = __builtin_bit_cast(bf8, p[q]);
    }

    int k_end = a.Sk, k_wave = a.Sk;  // keys some query of the workgroup / wave sees
    if (CAUSAL) {
        k_end = min(k_end, min(q0 + QB - 1, a.S - 1) + a.q_pos - a.k_pos + 1);
        k_wave = min(k_wave, min(qw0 + 31, a.S - 1) + a.q_pos - a.k_pos + 1);
    }
    if (qw0 >= a.S) k_wave = 0;
    // this workgroup's share of the key blocks
    const int all = k_end > 0 ? (k_end + kBK - 1) / kBK : 0;
    const int blk0 = (int)((int64_t)split * all / a.splits);
    const int blk1 = (int)((int64_t)(split + 1) * all / a.splits);
    // this lane's query sees keys t < lim
    const int lim = q_ok ? (CAUSAL ? min(a.Sk, query + a.q_pos - a.k_pos + 1) : a.Sk) : 0;

    // Tile loads through buffer descriptors over this batch's rows, as in
    // attention_f32: a key past Sk gets an offset past the end and reads 0.
    constexpr uint32_t kOutside = 0x80000000u;  // the host keeps Sk*H*D*4 < 2^31
    const uint32_t kv_bytes = (uint32_t)a.Sk * (uint32_t)HD * 4u;
    const __amdgpu_buffer_rsrc_t rsrc_k = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.k + (size_t)b * a.Sk * HD), (short)0, (int)kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_v = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.v + (size_t)b * a.Sk * HD), (short)0, (int)kv_bytes, 0x00020000);
    // K octet: key, dims 8o .. 8o + 7.  V octet: dim, keys vkey + {0..3, 8..11}.
    // A row of K's tile has D / 8 octets: the permutation spreads the 16 rows of
    // a read phase over all 16 slots of 256 bytes.
    auto k_slot = [](int key, int o) {
        return o ^ (D == 128 ? key & 15 : D == 64 ? (key >> 1) & 7 : (key >> 2) & 3);
    };
    uint32_t koff[U], voff[U];
    int kkey[U], kdst[U], vkey[U], vdst[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int p = u * T + (int)threadIdx.x;
        const int key = p / (D / 8), o = p % (D / 8);
        kkey[u] = key;
        koff[u] = 8 * o < DD ? ((uint32_t)key * (uint32_t)HD + (uint32_t)(h * DD + 8 * o)) * 4u : kOutside;
        kdst[u] = key * (D * 2) + (k_slot(key, o) << 4);
        const int dim = p / 128 * 32 + (p & 31), oct = (p >> 5) & 3;  // oct = 2 step + half
        vkey[u] = 16 * (oct >> 1) + 4 * (oct & 1);
        voff[u] = dim < DD ? ((uint32_t)vkey[u] * (uint32_t)HD + (uint32_t)(h * DD + dim)) * 4u : kOutside;
        vdst[u] = 3 * KP + dim * 64 + ((oct ^ ((dim >> 2) & 3)) << 4);
    }
    float xk[U][8], xv[U][8];
    using Yes = std::true_type;
    using No = std::false_type;
    // (whole: every key of the tile is below Sk)
    auto load_k = [&](int kb, auto whole) {
        const int soff = kb * HD * 4;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint32_t off = koff[u];
            if constexpr (!decltype(whole)::value) off = kb + kkey[u] < a.Sk ? off : kOutside;
            if (U * T != OCTS && u * T + (int)threadIdx.x >= OCTS) off = kOutside;
            const cl_f4 v0 = __builtin_bit_cast(cl_f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_k, (int)off, soff, 0));
            const cl_f4 v1 = __builtin_bit_cast(cl_f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_k, (int)(off + 16u), soff, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                xk[u][e] = v0[e];
                xk[u][4 + e] = v1[e];
            }
        }
    };
    // (in a tile that Sk ends inside the scalar offset stops at the last row: past it
    // every lane is outside, and for k and v near 2 GiB the row's offset would pass
    // 2^31.  Adding the row to the lanes' offsets instead spilled registers.)
    auto load_v = [&](int kb, auto whole) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int ke = (e & 3) + 8 * (e >> 2);
                uint32_t off = voff[u];
                int row = kb + ke;
                if constexpr (!decltype(whole)::value) {
                    off = row + vkey[u] < a.Sk ? off : kOutside;
                    row = min(row, a.Sk - 1);
                }
                xv[u][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc_v, (int)off, row * HD * 4, 0));
            }
    };
    auto split_octet = [&](const float *x, char *dst) {
        u4 p[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            unsigned x1, x2, x3;
            split_pair<true>(x[2 * e], x[2 * e + 1], &x1, &x2, &x3);
            p[0][e] = x1;
            p[1][e] = x2;
            p[2][e] = x3;
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<u4 *>(dst + q * KP) = p[q];
    };
    auto store_k = [&](int buf) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (U * T == OCTS || u * T + (int)threadIdx.x < OCTS)
                split_octet(xk[u], smem + buf * STAGE + kdst[u]);
    };
    auto store_v = [&](int buf) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (U * T == OCTS || u * T + (int)threadIdx.x < OCTS)
                split_octet(xv[u], smem + buf * STAGE + vdst[u]);
    };

    float m = -INFINITY, lsum = 0.0f;
    f16v o[kJ];
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[j][e] = 0.f;
    if (blk0 < blk1) {
        load_k(blk0 * kBK, No{});
        load_v(blk0 * kBK, No{});
        store_k(blk0 & 1);
        store_v(blk0 & 1);
        if (blk0 + 1 < blk1) {
            load_k((blk0 + 1) * kBK, No{});
            load_v((blk0 + 1) * kBK, No{});
        }
    }
    lds_barrier();
    // One block of keys.  Steady blocks (every query of the workgroup sees all
    // of it, and tile n + 2 is whole) have no branch around the staging, so the
    // splits run between the MFMAs of the same basic block.
    auto block = [&](int blk, auto steady) {
        constexpr bool kSteady = decltype(steady)::value;
        const int kb = blk * kBK;
        const int cur = blk & 1;
        const bool more = kSteady || blk + 1 < blk1, more2 = kSteady || blk + 2 < blk1;
        const char *st = smem + cur * STAGE;
        auto stage_k = [&] {
            if (more) {
                store_k(cur ^ 1);
                if (more2) load_k(kb + 2 * kBK, steady);
            }
        };
        auto stage_v = [&] {
            if (more) {
                store_v(cur ^ 1);
                if (more2) load_v(kb + 2 * kBK, steady);
            }
        };
        if (!kSteady && kb >= k_wave) {  // no query of the wave sees the block
            stage_k();
            stage_v();
            lds_barrier();
            return;
        }
        f16v s;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
        for (int g = 0; g < ST; ++g) {
            bf8 kf[3];
            const int slot = k_slot(l32, 2 * g + hh);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                kf[q] = *reinterpret_cast<const bf8 *>(st + q * KP + l32 * (D * 2) + (slot << 4));
#pragma unroll
            for (int p = 0; p < 6; ++p)
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kPieceA[p]], qf[g][kPieceB[p]], s, 0, 0,
                                                            0);
            if (g == 0) stage_k();
        }
        // s[i] is the score of key kb + 8(i/4) + 4hh + i%4 (base-2 units, times 2^48)
        if constexpr (!kSteady) {
            bool full = kb + kBK <= a.Sk && qw0 + 32 <= a.S;
            if (CAUSAL) full = full && kb + kBK - 1 + a.k_pos <= qw0 + a.q_pos;
            if (!full) {
                asm volatile("");  // (keeps the mask a branch)
                const int vis = lim - kb - 4 * hh;
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = 8 * (i / 4) + (i % 4) < vis ? s[i] : -INFINITY;
            }
        }
        float mloc = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) mloc = fmaxf(mloc, s[i]);
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64)) * kSumUnscale;
        // lazy rescale, as in attention_f32
        constexpr float kSlack = 8.0f;
        if (__any(mloc > m + kSlack)) {
            const float m_new = fmaxf(m, mloc);
            const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
            lsum *= alpha;
#pragma unroll
            for (int j = 0; j < kJ; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[j][e] *= alpha;
            m = m_new;
        }
        const float mz = m == -INFINITY ? 0.0f : m;
        float ps = 0.0f;
        // step t's weights, then its products; step 1's exponentials and splits
        // fall between step 0's MFMAs
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            bf8 pf[3];
            u4 pw[3];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float w0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * t + 2 * e], kSumUnscale, -mz));
                const float w1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * t + 2 * e + 1], kSumUnscale, -mz));
                ps += w0;
                ps += w1;
                unsigned x1, x2, x3;
                split_pair<true>(w0, w1, &x1, &x2, &x3);
                pw[0][e] = x1;
                pw[1][e] = x2;
                pw[2][e] = x3;
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) pf[q] = __builtin_bit_cast(bf8, pw[q]);
#pragma unroll
            for (int j = 0; j < kJ; ++j) {
                bf8 vf[3];
                const int slot = (2 * t + hh) ^ ((l32 >> 2) & 3);
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    vf[q] = *reinterpret_cast<const bf8 *>(st + 3 * KP + q * KP + (32 * j + l32) * 64 +
                                                           (slot << 4));
#pragma unroll
                for (int p = 0; p < 6; ++p)
                    o[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[kPieceA[p]], pf[kPieceB[p]], o[j],
                                                                   0, 0, 0);
                if (t == 0 && j == 0) stage_v();
            }
        }
        ps += __shfl_xor(ps, 32, 64);
        lsum += ps;
        lds_barrier();
    };
    // blocks before which every query of the workgroup sees all, and two more
    // whole tiles follow
    int steady = a.Sk / kBK - 2;
    if (CAUSAL) steady = min(steady, max(0, q0 + a.q_pos - a.k_pos + 1) / kBK);
    steady = min(steady, blk1 - 2);
    int blk = blk0;
    for (; blk < steady; ++blk) block(blk, Yes{});
    for (; blk < blk1; ++blk) block(blk, No{});

    bool bad = !(lsum < INFINITY);
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) bad = bad || !(__builtin_fabsf(o[j][e]) < INFINITY);
    if (__builtin_expect(__syncthreads_or(bad), 0)) {
        attention_f32<D, CAUSAL, T>(a, q0, bh, split, blk0, blk1, reinterpret_cast<float *>(smem));
        return;
    }
    if (q_ok) attn_store<D, kJ>(a, b, h, query, split, hh, o, m, lsum, kSumUnscale);
}

// Adds the key splits of every (row, head): O = sum O_p 2^(m_p - M) / sum l_p
// 2^(m_p - M), in split order; a split that saw no key of the query has m_p =
// -inf.  One thread per four dims, the splits' loads issued before any is used.
__global__ void __launch_bounds__(256) attention_merge_kernel(const float *__restrict__ part,
                                                              float *__restrict__ out,
                                                              int64_t rows, int D, int splits) {
    const int nv = D / 4;
    const float *stat = part + (size_t)splits * rows * D;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < rows * nv;
         i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / nv;
        const int c = 4 * (int)(i % nv);
        float M = -INFINITY;
#pragma unroll 4
        for (int p = 0; p < splits; ++p) M = fmaxf(M, stat[2 * (p * rows + row)]);
        cl_f4 o = {0.f, 0.f, 0.f, 0.f};
        float L = 0.0f;
#pragma unroll 4
        for (int p = 0; p < splits; ++p) {
            const float mp = stat[2 * (p * rows + row)], lp = stat[2 * (p * rows + row) + 1];
            const cl_f4 v = *reinterpret_cast<const cl_f4 *>(part + (p * rows + row) * D + c);
            const float w = mp == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mp - M);
            L += lp * w;
            o += v * w;
        }
        *reinterpret_cast<cl_f4 *>(out + row * D + c) = o * (L > 0.0f ? 1.0f / L : 0.0f);
    }
}

template <int D, int NW>
void launch_x3(const AttnArgs &a, bool causal, hipStream_t s) {
    const unsigned grid = (unsigned)(a.B * a.H * a.nqb * a.splits);
    if (causal) attention_x3_kernel<D, true, NW><<<grid, 64 * NW, 0, s>>>(a);
    else attention_x3_kernel<D, false, NW><<<grid, 64 * NW, 0, s>>>(a);
}

// RoPE table: tab[p][j] = (cos, sin) of theta = (pos0 + p) / div[j], the
// angle of pair j (dims 2j, 2j+1) at position pos0 + p (backend.rs:2818).
// Built once per call, so each (position, pair) pays one sincosf however
// many heads and rows use it.
__global__ void __launch_bounds__(256) rope_table_kernel(float2 *__restrict__ tab, int pos0,
                                                         int npos, int pairs, AttnFreq f) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= npos * pairs) return;
    const int p = i / pairs, j = i % pairs;
    const float theta = (float)(pos0 + p) / f.div[j];
    float s, c;
    sincosf(theta, &s, &c);
    tab[i] = make_float2(c, s);
}

// backend.rs:2797-2826: x1' = x1 cos - x2 sin, x2' = x1 sin + x2 cos per pair
// of every whole head; dims past the last whole head are written as 0.
// One workgroup of kRopeThreads threads per row (grid-stride over rows): the
// row's position and its table row are computed once, each thread then
// rotates 16-byte vectors (two pairs), issuing up to kRopeVec vector loads
// before any arithmetic.  512 threads x 2 vectors (a 4096-float row in one
// pass) streamed faster than 256 x 4 with inputs the last-level cache does
// not hold.
constexpr int kRopeThreads = 512, kRopeVec = 2;
// HD4 (head_dim % 4 == 0): a vector's two pairs are table entries 2m and
// 2m + 1 of one row, adjacent and 16-byte aligned, fetched with one 16-byte
// load issued with the row's loads; the whole-head bound then covers both
// pairs of a vector alike.
template <bool HD4>
__global__ void __launch_bounds__(kRopeThreads) rope_rows_kernel(const float *__restrict__ x,
                                                                 float *__restrict__ out,
                                                                 uint64_t rows, int seq,
                                                                 int hidden, int head_dim,
                                                                 int pos_offset, const float2 *tab,
                                                                 int tab_pos0) {
#pragma clang fp contract(off)
    const int nv = hidden / 4;
    const int pairs = head_dim / 2;
    const int whole = (hidden / head_dim) * head_dim;
    for (uint64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int p = (int)(r % (uint64_t)seq) + pos_offset - tab_pos0;
        const float2 *trow = tab + (size_t)p * pairs;
        const float *xr = x + r * (uint64_t)hidden;
        float *orow = out + r * (uint64_t)hidden;
        for (int v0 = threadIdx.x; v0 < nv; v0 += kRopeVec * kRopeThreads) {
            cl_f4 xv[kRopeVec], tv[kRopeVec];
#pragma unroll
            for (int u = 0; u < kRopeVec; ++u) {
                const int v = v0 + kRopeThreads * u;
                if (v < nv) {
                    xv[u] = __builtin_nontemporal_load(reinterpret_cast<const cl_f4 *>(xr) + v);
                    if (HD4 && 4 * v < whole)
                        tv[u] = *reinterpret_cast<const cl_f4 *>(trow + ((4 * v) % head_dim) / 2);
                }
            }
#pragma unroll
            for (int u = 0; u < kRopeVec; ++u) {
                const int v = v0 + kRopeThreads * u;
                if (v >= nv) continue;
                const int c0 = 4 * v;
                cl_f4 o = {0.f, 0.f, 0.f, 0.f};
                if (HD4) {
                    if (c0 < whole) {
                        o.x = xv[u].x * tv[u].x - xv[u].y * tv[u].y;
                        o.y = xv[u].x * tv[u].y + xv[u].y * tv[u].x;
                        o.z = xv[u].z * tv[u].z - xv[u].w * tv[u].w;
                        o.w = xv[u].z * tv[u].w + xv[u].w * tv[u].z;
                    }
                } else {
                    if (c0 < whole) {
                        const float2 t0 = trow[(c0 % head_dim) / 2];
                        o.x = xv[u].x * t0.x - xv[u].y * t0.y;
                        o.y = xv[u].x * t0.y + xv[u].y * t0.x;
                    }
                    if (c0 + 2 < whole) {
                        const float2 t1 = trow[((c0 + 2) % head_dim) / 2];
                        o.z = xv[u].z * t1.x - xv[u].w * t1.y;
                        o.w = xv[u].z * t1.y + xv[u].w * t1.x;
                    }
                }
                __builtin_nontemporal_store(o, reinterpret_cast<cl_f4 *>(orow) + v);
            }
        }
    }
}

// Pair-at-a-time form for rows whose vectors are not 16-byte aligned.
__global__ void __launch_bounds__(256) rope_pairs_kernel(const float *__restrict__ x,
                                                         float *__restrict__ out, uint64_t rows,
                                                         int seq, int hidden, int head_dim,
                                                         int pos_offset, const float2 *tab,
                                                         int tab_pos0) {
#pragma clang fp contract(off)
    const int pairs = head_dim / 2;
    const int whole = (hidden / head_dim) * head_dim;
    for (uint64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int p = (int)(r % (uint64_t)seq) + pos_offset - tab_pos0;
        const float2 *trow = tab + (size_t)p * pairs;
        const uint64_t base = r * (uint64_t)hidden;
        for (int c0 = 2 * threadIdx.x; c0 < hidden; c0 += 2 * 256) {
            float o0 = 0.0f, o1 = 0.0f;
            if (c0 < whole) {
                const float2 t = trow[(c0 % head_dim) / 2];
                const float x1 = x[base + c0], x2 = x[base + c0 + 1];
                o0 = x1 * t.x - x2 * t.y;
                o1 = x1 * t.y + x2 * t.x;
            }
            out[base + c0] = o0;
            out[base + c0 + 1] = o1;
        }
    }
}

}  // namespace

bool attention_supported(int head_dim) { return head_dim >= 1 && head_dim <= kAttnMaxHeadDim; }

// Tile size, query blocks and key splits of the bf16x3 kernel; qb = 0: the FP32
// MFMA kernel's call.
//
// Splitting the keys of a query block over workgroups pays where the blocks
// alone leave CUs idle or one long block finishes last (64 queries over 2064
// keys, 16 heads of 128: 42 us against 247 unsplit; 2048 causal queries, 16
// heads of 128: 133 against 251).  The cost of a split is priced as the longer of
// its longest workgroup (lone us per 32-key block) and all of them spread over
// the slots (full us per block and slot), a workgroup's prologue counted as
// three blocks, plus the partial results' traffic and the merge launch.  lone
// and full are measured (lone: one query block per CU or fewer; full: 4096
// queries, 32 heads).
struct AttnX3Plan {
    int dp, qb, splits;
};

// 32-key blocks of one head's query blocks of qb queries: their sum, and the
// longest's.
struct AttnBlocks {
    double sum;
    int most, nqb;
};
static AttnBlocks attention_blocks(int S, int Sk, int q_pos, int k_pos, bool causal, int qb) {
    AttnBlocks r{0.0, 0, (S + qb - 1) / qb};
    for (int i = 0; i < r.nqb; ++i) {
        int64_t end = Sk;
        if (causal)
            end = std::min<int64_t>(end, std::min<int64_t>((int64_t)(i + 1) * qb, S) + q_pos - k_pos);
        const int n = end > 0 ? (int)((end + kBK - 1) / kBK) : 0;
        r.sum += n;
        r.most = std::max(r.most, n);
    }
    return r;
}

// A whole call's time in us on a kernel that holds per_cu workgroups on a CU: the
// longer of its longest workgroup (lone us per key block alone on its CU, up to
// 1 + share times that beside others) and of all of them over the slots (full us
// per block and slot), pro blocks of prologue each.
struct AttnPrice {
    double lone, full, base, pro, share;
    int per_cu;
};
static double attention_us(const AttnPrice &k, double heads, double sum, double wgs, int longest,
                           int num_cus) {
    const double beside = std::min(std::max(wgs * heads / num_cus - 1.0, 0.0), k.per_cu - 1.0);
    return k.base + std::max((longest + k.pro) * k.lone * (1.0 + k.share * beside),
                             heads * (sum + k.pro * wgs) / (k.per_cu * num_cus) * k.full);
}

// Up to 64 queries over up to 64 keys, a workgroup to a CU, the split of the
// operands costs more than the faster products give, and the FP32 MFMA kernel takes the call (with RoPE, FP32 first:
// 64 queries of 12 heads of 80 13.2 against 15.6 us, of 8 of 64 11.0 against
// 12.7, of 16 of 96 14.5 against 15.8; 100 queries 18.2 against 16.1, 15.0
// against 13.7, 20.4 against 17.1).
constexpr int kShort = 64;
static AttnX3Plan attention_x3_plan(int B, int S, int Sk, int H, int D, int q_pos, int k_pos,
                                    bool causal, int num_cus) {
    AttnX3Plan p{0, 0, 1};
    if (D % 8 != 0 || D > 128) return p;
    if (S <= kShort && Sk <= kShort && (int64_t)B * H <= num_cus) return p;
    static const float lone[] = {1.25f, 1.8f, 2.6f, 3.9f}, full[] = {1.8f, 2.9f, 4.3f, 4.8f};
    static const int per_cu[] = {4, 2, 2, 1};
    const int c = (D + 31) / 32 - 1;
    p.dp = 32 * (c + 1);
    p.qb = p.dp == 128 ? 256 : 128;
    const AttnBlocks n = attention_blocks(S, Sk, q_pos, k_pos, causal, p.qb);
    const double heads = (double)B * H, slots = (double)per_cu[c] * num_cus;
    const double merge = 2.0 * heads * S * D * 4.0 / 5e6;  // us per split
    double best = 0.0;
    for (int sp = 1; sp <= 64 && (sp == 1 || sp <= n.most); sp += sp < 8 ? 1 : sp < 16 ? 2 : 8) {
        const double longest = (double)((n.most + sp - 1) / sp + 3) * lone[c];
        const double all = heads * (n.sum + 3.0 * sp * n.nqb) / slots * full[c];
        const double t = std::max(longest, all) + (sp > 1 ? 3.0 + merge * sp : 0.0);
        if (sp == 1 || t < best) {
            best = t;
            p.splits = sp;
        }
    }

    // The FP32 MFMA kernel keeps the calls where it is still the faster: short
    // queries of many heads at D past 96, whose 256-query workgroups have a CU
    // each (4096 x 32 heads of 128 over one key 2.6 against 4.3 ms, 64 x 32 of 128
    // queries 136 against 170 us), and D well under a multiple of 32, whose zero
    // dims cost as much as others here but less than 16 there (64 x 32 heads of 16,
    // 512 causal queries 197 against 227 us; 128 queries of 48 51 against 62).
    // Both are priced, by figures fitted to 2976 calls of every D, 32 to 2048
    // heads, 1 to 512 queries (each model within 10% as a rule): of the 735 that
    // were slower here than there by 4% and 0.3 us, 33 still are, and 26 became
    // slower by as much.  Queries under half a workgroup leave waves idle, which
    // speeds the others up.
    static const AttnPrice x3[] = {{1.4, 2.9, 3.0, 0.8, 0.15, 4},
                                   {1.75, 3.05, 3.0, 0.8, 0.15, 2},
                                   {2.6, 4.6, 3.0, 0.8, 0.15, 2},
                                   {4.4, 5.1, 3.0, 0.8, 0.15, 1}};
    static const AttnPrice fp32[] = {
        {0.73, 1.22, 1.8, 1.2, 0.85, 2}, {1.46, 2.3, 1.8, 0.45, 0.85, 2},
        {2.05, 3.2, 1.8, 0.45, 0.85, 2}, {2.2, 4.0, 1.8, 1.2, 0.85, 2},
        {3.2, 5.4, 1.8, 0.45, 0.85, 2},  {3.65, 6.25, 1.8, 0.45, 0.85, 2},
        {4.2, 7.2, 1.8, 0.45, 0.85, 2},  {4.75, 8.2, 1.8, 0.45, 0.85, 2}};
    const double used = std::min(1.0, (double)((S + 31) / 32 * 32) / p.qb);
    const double sp = p.splits, active = 1.0 - 0.22 * (1.0 - used);
    AttnPrice kx = x3[c];
    kx.lone *= active;
    kx.full *= active;
    const double here = attention_us(kx, heads, n.sum + kx.pro * (sp - 1) * n.nqb, n.nqb,
                                     (n.most + p.splits - 1) / p.splits, num_cus) +
                        (p.splits > 1 ? 3.0 + merge * sp : 0.0);
    const AttnBlocks n16 = attention_blocks(S, Sk, q_pos, k_pos, causal, kBQ);
    const double there =
        attention_us(fp32[(D + 15) / 16 - 1], heads, n16.sum, n16.nqb, n16.most, num_cus);
    // (past 112 dims and up to a head per CU the price of a lone workgroup here is
    // too high: 256 heads of 128, 100 queries over 200 keys 32 us against 38)
    const bool lone_heads = D > 112 && heads <= num_cus;
    if (there < 0.97 * here && !lone_heads) p = AttnX3Plan{0, 0, 1};
    return p;
}

size_t attention_workspace_floats(int B, int S, int Sk, int H, int D, int q_pos, int k_pos,
                                  bool causal, int num_cus) {
    if (B <= 0 || S <= 0 || H <= 0) return 0;
    const AttnX3Plan p = attention_x3_plan(B, S, Sk, H, D, q_pos, k_pos, causal, num_cus);
    return p.splits > 1 ? (size_t)p.splits * B * S * H * (D + 2) : 0;
}

void attention_prefill(const float *q, const float *k, const float *v, float *out, int B, int S,
                       int Sk, int H, int D, int q_pos, int k_pos, bool causal, float scale,
                       const float *q_rope_tab, int tab_pos0, float *ws, int num_cus,
                       hipStream_t s) {
    if (B <= 0 || S <= 0 || H <= 0) return;
    const AttnX3Plan p = attention_x3_plan(B, S, Sk, H, D, q_pos, k_pos, causal, num_cus);
    AttnArgs a{q, k, v, out, B, S, Sk, H, q_pos, k_pos, scale, 0,
               reinterpret_cast<const float2 *>(q_rope_tab), tab_pos0, D, p.splits, ws};
    const int qb = p.qb ? p.qb : kBQ, threads = !p.qb ? 512 : p.dp == 128 ? 512 : 256;
    a.nqb = (S + qb - 1) / qb;
    // A grid holds under 2^32 threads: more heads than that go in several launches
    // of whole batch entries (one entry's heads and queries always fit: past 2^23
    // workgroups of it, q alone would exceed the memory).
    const int64_t entry = (int64_t)H * a.nqb * p.splits * threads;
    const int per_launch =
        (int)std::min<int64_t>(B, std::max<int64_t>(1, ((1ll << 32) - 1) / entry));
    for (int b0 = 0; b0 < B; b0 += per_launch) {
        const size_t qo = (size_t)b0 * S * H * D, ko = (size_t)b0 * Sk * H * D;
        a.B = std::min(per_launch, B - b0);
        a.q = q + qo;
        a.k = k + ko;
        a.v = v + ko;
        a.out = out + qo;
        if (!p.qb) {
            attention_prefill_general(a, causal, (unsigned)((int64_t)a.B * H * a.nqb), s);
            continue;
        }
        if (p.dp == 32) launch_x3<32, 4>(a, causal, s);
        else if (p.dp == 64) launch_x3<64, 4>(a, causal, s);
        else if (p.dp == 96) launch_x3<96, 4>(a, causal, s);
        else launch_x3<128, 8>(a, causal, s);
        if (p.splits > 1) {
            const int64_t rows = (int64_t)a.B * S * H, blocks = (rows * (D / 4) + 255) / 256;
            attention_merge_kernel<<<(unsigned)std::min<int64_t>(blocks, 32 * num_cus), 256, 0, s>>>(
                ws, a.out, rows, D, p.splits);
        }
    }
}

void rope_table(float *tab, int pos0, int npos, int head_dim, const AttnFreq &freq,
                hipStream_t s) {
    const int n = npos * (head_dim / 2);
    if (n <= 0) return;
    rope_table_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(
        reinterpret_cast<float2 *>(tab), pos0, npos, head_dim / 2, freq);
}

void rope_apply(const float *x, float *out, size_t rows, int seq, int hidden, int head_dim,
                int pos_offset, const float *tab, int tab_pos0, hipStream_t s) {
    if (rows == 0 || hidden <= 0) return;
    const bool vec = hidden % 4 == 0 &&
                     ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    // one workgroup per row, at most 64 per CU's worth of rows in flight
    const unsigned grid = (unsigned)(rows < 16384 ? rows : 16384);
    const float2 *t = reinterpret_cast<const float2 *>(tab);
    if (vec && head_dim % 4 == 0)
        rope_rows_kernel<true><<<grid, kRopeThreads, 0, s>>>(x, out, rows, seq, hidden, head_dim,
                                                             pos_offset, t, tab_pos0);
    else if (vec)
        rope_rows_kernel<false><<<grid, kRopeThreads, 0, s>>>(x, out, rows, seq, hidden, head_dim,
                                                              pos_offset, t, tab_pos0);
    else
        rope_pairs_kernel<<<grid, 256, 0, s>>>(x, out, rows, seq, hidden, head_dim, pos_offset, t,
                                               tab_pos0);
}

}  // namespace k
}  // namespace clove
