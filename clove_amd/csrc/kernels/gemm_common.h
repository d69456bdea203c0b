// gemm_common.h -- what the GEMM kernels share: buffer descriptors, the
// kernel arguments, the XCD-aware tile order and the fused epilogue
// (gemm_f32.hip, gemm_bf16x3.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "launch.hpp"

namespace clove {
namespace k {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

// Raw buffer resource over [base, base + bytes): stride 0, word 3 = 32-bit
// data format (DATA_FORMAT = 4 in bits 15..18), the gfx9-family setting.
// Reads at offsets >= bytes return 0 (and a DMA lane past the end writes 0
// to LDS).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes,
                                             0x00020000);
}

struct GemmArgs {
    const float *A, *B;
    float *C;
    float *ws;        // split-K partial tiles [splits][tiles][BM*BN]
    int M, N, K, tiles_n, k_per_split, splits;
    GemmEpilogue epi;
    int tiles;        // tiles of C (the grid's x dimension is padded to 8 * per_xcd)
    int per_xcd;      // ceil(tiles / 8)
};

// Tile order.  Workgroups are dealt to the 8 XCDs round-robin (workgroup L
// runs on XCD L % 8), each with its own L2.  Workgroup L takes position
// L / 8 of its XCD's range of a grouped order, so each XCD walks one
// contiguous eighth of it (all eighths alike to one tile); the grouped order visits kGroupM tile rows column
// by column.  At 4096^3 (32 x 16 tiles of 128 x 256) an XCD then owns an
// 8 x 8 block of tiles whose concurrently running workgroups share A and B
// slabs in its L2 (the plain row-major order gave each XCD 2 tile columns
// and all 32 tile rows, so every A slab was fetched for just two tiles).
constexpr int kGroupM = 8;
__device__ __forceinline__ bool gemm_tile(const GemmArgs &g, int *tile) {
    const int L = blockIdx.x, xcd = L % 8;
    const int V = (int)((int64_t)xcd * g.tiles / 8) + L / 8;
    if (V >= (int)((int64_t)(xcd + 1) * g.tiles / 8)) return false;
    const int tiles_m = g.tiles / g.tiles_n;
    const int group_size = kGroupM * g.tiles_n;
    const int first = (V / group_size) * kGroupM;
    const int rows = min(kGroupM, tiles_m - first);
    const int r = V % group_size;
    *tile = (first + r % rows) * g.tiles_n + r / rows;
    return true;
}

// Epilogue: C = act(acc + bias[(row*N + col) % bias_n]), each step rounded
// in f32 exactly as Clove's separate Add (backend.rs:1489) and ReLU
// (:1823) / GELU (:1924) passes round it.
// bcol: bias[col] when the caller has loaded it already (GEMM_BIAS_COL), so
// that the load is not repeated after every store to C, which may alias it.
__device__ __forceinline__ float epilogue(const GemmEpilogue &e, float v, int row, int col, int N,
                                          const float *bcol = nullptr) {
#pragma clang fp contract(off)
    if (e.bias_mode == GEMM_BIAS_COL) v = v + (bcol ? *bcol : e.bias[col]);
    else if (e.bias_mode == GEMM_BIAS_SCALAR) v = v + e.bias[0];
    else if (e.bias_mode == GEMM_BIAS_MOD) v = v + e.bias[((uint64_t)row * N + col) % e.bias_n];
    if (e.act == GEMM_ACT_RELU) {
        v = v > 0.0f ? v : 0.0f;
    } else if (e.act == GEMM_ACT_GELU) {
        const float k = 0x1.988452p-1f;  // (2/pi).sqrt() in f32, backend.rs:1924
        const float x3 = (v * v) * v;
        v = 0.5f * v * (1.0f + tanhf(k * (v + 0.044715f * x3)));
    }
    return v;
}

// gemm_bf16x3.hip: launches p (p.x3 set) on A or A^T (ta) and B or B^T (tb, at
// most one of the two), any 4-byte alignment; a split product's partial tiles
// go to g.ws.
void gemm_bf16x3(const GemmPlan &p, const GemmArgs &g, bool ta, bool tb, hipStream_t s);

}  // namespace k
}  // namespace clove
