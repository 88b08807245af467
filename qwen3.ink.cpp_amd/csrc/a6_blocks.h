// A6, the block-scaled kernel's rows (gemm_fp6_a81w41.hip), as the kernels that make them write it: per (32-row panel, 32-block) the high
// pieces of the panel's int8, then the low ones, in fp6 patterns, each with the block's parameters.
#pragma once
#include "a81w41_kernels.h"
#include "quantize_common.h"

namespace a81w41 {
namespace fp6 {

constexpr int kPanelA = 2048;  // bytes per (32-row panel, 32-block)

// fp6 pattern of an integer in [-15, 15]
__host__ __device__ __forceinline__ uint32_t fp6_of_int(int v) { return v < 0 ? (0x20u | (uint32_t)(-v)) : (uint32_t)v; }

// x as two bf16 pieces, hi | lo << 16: hi = bf16(x), lo = bf16(x - hi), both rounded to nearest even.
__host__ __device__ __forceinline__ uint32_t bf16_rne_bits(float x) {
    union { float f; uint32_t u; } v = {x};
    return (v.u + 0x7fffu + ((v.u >> 16) & 1u)) >> 16;
}
__host__ __device__ __forceinline__ uint32_t split_bf16x2(float x) {
    const uint32_t hi = bf16_rne_bits(x);
    union { uint32_t u; float f; } h = {hi << 16};
    return hi | (bf16_rne_bits(x - h.f) << 16);  // the subtraction is exact
}
// x as three bf16 pieces hi + mid + lo = x exactly (24 significant bits): hi | mid << 16 in .x, lo in .y
__host__ __device__ __forceinline__ uint2 split_bf16x3(float x) {
    const uint32_t hi = bf16_rne_bits(x);
    union { uint32_t u; float f; } h = {hi << 16};
    const float r1 = x - h.f;  // exact
    const uint32_t mid = bf16_rne_bits(r1);
    union { uint32_t u; float f; } m = {mid << 16};
    return make_uint2(hi | (mid << 16), bf16_rne_bits(r1 - m.f));  // what is left has at most 8 significant bits
}

// Six dwords of 32 six-bit patterns from the eight 24-bit pieces (4 patterns each) the lanes of a
// group of 8 hold: dword d = bits [32 d, 32 d + 32) of the 192-bit string sum(piece_j << 24 j).
__device__ __forceinline__ void gather_fp6_dwords(uint32_t piece, int lane, uint32_t (&dw)[6]) {
    uint32_t p[8];
    const int base = lane & ~7;
#pragma unroll
    for (int j = 0; j < 8; j++) p[j] = (uint32_t)__shfl((int)piece, base + j, 64);
    dw[0] = p[0] | (p[1] << 24);
    dw[1] = (p[1] >> 8) | (p[2] << 16);
    dw[2] = (p[2] >> 16) | (p[3] << 8);
    dw[3] = p[4] | (p[5] << 24);
    dw[4] = (p[5] >> 8) | (p[6] << 16);
    dw[5] = (p[6] >> 16) | (p[7] << 8);
}

__device__ __forceinline__ uint32_t fp6_piece_of_bytes(uint32_t packed_q, bool high) {
    uint32_t piece = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int q = (int)(int8_t)(packed_q >> (8 * i));
        const int v = high ? (q >> 4) : (q & 15);
        piece |= fp6_of_int(v) << (6 * i);
    }
    return piece;
}

// Which float4 of the rows a thread takes (workgroups of 256, a multiple of eight rows of n4 float4s): a wave has one 32-block of eight
// rows, eight lanes a row, so that its 16-byte pieces fill lines of 128 bytes.  With a wave along a row a line came in eight parts,
// from eight workgroups on as many XCDs: silu * up of 322 x 12288 13.0 us, so 11.1; a call of 1500 rows, 8000 x 2048, 82.5 and 80.6 us.
struct RowQuad {
    int row, j;
};
__device__ __forceinline__ RowQuad row_quad(int n4) {
    const unsigned unit = blockIdx.x * 4 + (threadIdx.x >> 6), blocks = n4 >> 3, rows8 = unit / blocks;
    const int lane = threadIdx.x & 63;
    return {(int)(rows8 * 8) + (lane >> 3), (int)(unit - rows8 * blocks) * 8 + (lane & 7)};
}
inline unsigned row_quad_grid(int rows_padded, int n4) { return (unsigned)(((long long)(rows_padded / 8) * (n4 / 8) + 3) / 4); }

// Stores one 32-block of one row into A6.  The 8 lanes of the group each hold 4 of the block's int8 (packed);
// lanes 0..3 write the four 16-byte chunks (piece = lane >> 1, chunk = lane & 1).
__device__ __forceinline__ void store_a6_block(uint8_t* __restrict__ a6, int row, int blk, int nb, uint32_t packed_q, float d,
                                               float ssum, int lane) {
    uint32_t hi[6], lo[6];
    gather_fp6_dwords(fp6_piece_of_bytes(packed_q, true), lane, hi);
    gather_fp6_dwords(fp6_piece_of_bytes(packed_q, false), lane, lo);
    const int j = lane & 7;
    if (j < 4) {
        const int piece = j >> 1, chunk = j & 1;
        const uint32_t* dw = piece ? lo : hi;
        uint4 v;
        if (chunk == 0) {
            v = make_uint4(dw[0], dw[1], dw[2], dw[3]);
        } else {
            // the scaled sum as three bf16 pieces, as the contraction multiplies them: hi | hi in the high piece's copy, mid | lo in
            // the low piece's
            const uint2 s3 = split_bf16x3(ssum);
            v = make_uint4(dw[4], dw[5], __float_as_uint(d), piece == 0 ? __builtin_amdgcn_perm(s3.x, s3.x, 0x01000100u) : s3.x >> 16 | s3.y << 16);
        }
        uint8_t* dst = a6 + ((size_t)(row >> 5) * nb + blk) * kPanelA + piece * 1024 + chunk * 512 + (row & 31) * 16;
        *reinterpret_cast<uint4*>(dst) = v;
    }
}

}  // namespace fp6
}  // namespace a81w41
