// mfma_layout.hpp -- operand layouts shared by the matrix-core kernels of
// attention.hip and gqa.hip (gfx950, wave64).
//
// v_mfma_f32_32x32x16_f16 and _bf16 take A / B operands
// with lane l holding row (A) or column (B) l % 32 and the inner-dimension
// slice l / 32; the 32 x 32 result leaves lane l with column l % 32 and, in
// register r, row 8 (r / 4) + 4 (l / 32) + r % 4.  The key orders below
// choose which key each result row holds so that a lane's registers come
// out in the operand layout of the next product.
#ifndef RUSTLLM_MFMA_LAYOUT_HPP
#define RUSTLLM_MFMA_LAYOUT_HPP

#include "common.hpp"

namespace rl {
namespace {

typedef half_t h8 __attribute__((ext_vector_type(8)));
typedef half_t h4 __attribute__((ext_vector_type(4)));
typedef half_t h2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// f16: row i of a 32-key S^T tile holds key perm32(i), bits 2 and 3 of i
// swapped; register r of lane l then holds key 16 (r / 8) + 8 (l / 32) +
// r % 8 -- eight consecutive keys per lane half, the B operand layout of
// the P V product over 16 keys.
__device__ inline uint32_t perm32(uint32_t i) {
    return (i & ~12u) | ((i & 4u) << 1) | ((i & 8u) >> 1);
}

// Row stride (halves) of V in LDS for the transpose reads: the 32 lanes one
// LDS cycle serves read 4 rows x 2 runs of 16 bytes; with 64 banks of 4
// bytes those land on distinct banks when the stride in dwords is 16 or 48
// modulo 64.  Smallest such stride >= D (in steps of 8 halves).
__host__ __device__ constexpr int v_stride_tr(int d) {
    int s = d;
    while ((s / 2) % 64 != 16 && (s / 2) % 64 != 48) s += 8;
    return s;
}

// Chunk order of the unpadded LDS rows the attention and f32 kernels use: 16-byte
// chunk c of row r sits at chunk c ^ lds_swizzle(r) of that row.  The MFMA
// operand reads of K (16 rows x one chunk per 16 lanes) and the transpose
// reads of V (4 rows x 4 chunks per 32 lanes) then each fall on 64 distinct
// banks (64 banks of 4 bytes; a row is D / 8 chunks).
template <int NT>
__device__ inline uint32_t lds_swizzle(uint32_t r) {
    static_assert(NT == 1 || NT == 2 || NT == 4 || NT == 8, "rows of 4, 8, 16 or 32 chunks");
    if constexpr (NT == 1) return (r >> 2) & 3u;
    else if constexpr (NT == 2) return ((r & 2u) << 1) | ((r >> 2) & 3u);
    else return ((r & 3u) << 2) | ((r >> 2) & 3u);
}

// ds_read_b64_tr_b16: in each group of 16 lanes, lanes 4j .. 4j + 3 read 8
// bytes each (row j of a 4 x 16 block of halves); lane i of the group
// receives column i of that block, one half from each row.
__device__ inline h4 lds_read_transposed(const half_t* p) {
    const s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(p));
    return __builtin_bit_cast(h4, r);
}

// f32 products on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16, 16 times
// the rate of the f32 ones).  An f32 value is the sum of three bf16 parts, each
// the rounding of what the parts before it leave (8 + 8 + 8 bits, and their
// signs: nothing is left of a normal value); of the nine products of two such
// values the six of order 2^-18 and above are added, the three dropped are below
// 2^-26 of the product.  Both operands of an instruction, and their layout,
// are those of v_mfma_f32_32x32x16_f16.
// Values are scaled by kPartScale first: every f32 value, subnormals included,
// is a multiple of 2^-149, so its parts are then multiples of 2^-125 and none
// falls below bf16's normal range.  Values of 2^104 and above (infinities too)
// have no such parts (inf - inf), and sums past the scaled range are infinite:
// a result that is not finite has to be computed unsplit.
constexpr float kPartScale = 0x1p24f;
constexpr float kProductUnscale = 0x1p-48f;  // of a sum of products of two scaled values
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

struct Bf16x3 {
    b8 part[3];  // high, middle, low
};

__device__ inline Bf16x3 split_bf16(f32x8 x) {
    Bf16x3 r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const b2 w = __builtin_convertvector((f32x2{x[e], x[e + 1]}), b2);
            r.part[i][e] = w[0];
            r.part[i][e + 1] = w[1];
            x[e] -= float(w[0]);
            x[e + 1] -= float(w[1]);
        }
    return r;
}

// acc += the five smaller products of a b, smallest first
__device__ inline f32x16 mfma_bf16x3_low(const Bf16x3& a, const Bf16x3& b, f32x16 acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[2], b.part[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[0], b.part[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[1], b.part[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[1], b.part[0], acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[0], b.part[1], acc, 0, 0, 0);
}
// acc += a b
__device__ inline f32x16 mfma_bf16x3(const Bf16x3& a, const Bf16x3& b, f32x16 acc) {
    acc = mfma_bf16x3_low(a, b, acc);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.part[0], b.part[0], acc, 0, 0, 0);
}

}  // namespace
}  // namespace rl

#endif
