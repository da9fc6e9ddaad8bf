// 20-state (amino-acid) steps of the clustered marginal pass (tt_cluster.hip)
// on FP32 MFMA.
//
// A row times a branch matrix is 20 x 20 multiply-adds per pattern.  The
// instruction is v_mfma_f32_4x4x1 with 16 blocks: each block multiplies a
// column of 4 by a row of 4, lane l = 4 b + j supplies A[j] and B[j] of block b
// and holds column j of the block's result, its 4 rows in 4 registers.  With
// the patterns as columns a lane owns one pattern, its 20 states in 20
// registers as 5 groups of 4: no state is padding (the 32 x 32 shape pads 20
// to 32 and needs 1280 cycles for 64 patterns; this one 800), nothing is
// exchanged between lanes, and the step's other arithmetic is that of the
// small alphabets (tt_device.h).
//
// The matrix is the A operand, the same for all blocks.  A register holds 16
// of the 100 (input state, group) columns of 4, one per block, and the
// instruction broadcasts one block's (cbsz 4, abid): column t = 5 k + g of
// M[k][4 g + i] is element 4 t + i, so register q is M[64 q + lane], 7
// coalesced loads a matrix.
//
// All 64 lanes take part, whatever the number of patterns (the instruction
// ignores the lane mask): lanes past the last pattern repeat it and store the
// same values.
#pragma once
#include <utility>

#include "tt_cluster.h"
#include "tt_device.h"

namespace ttd {

constexpr int kAA = 20;
// rows waiting at once: k only in a cluster of at least 2^(k + 1) - 1 nodes
constexpr int kSlots20 = 3;
constexpr int kLut20 = 64;  // character codes whose profile rows are staged in LDS

typedef float v4f __attribute__((ext_vector_type(4)));

struct Mat20 {
    float a[7];
};

// out_i = sum_k x_k M[k][i]
__device__ __forceinline__ void load_in20(const float TT_G *M, int lane, Mat20 &A) {
#pragma unroll
    for (int q = 0; q < 6; ++q) A.a[q] = M[64 * q + lane];
    A.a[6] = M[384 + (lane & 15)];
}

// out_i = sum_k M[i][k] x_k: column t = 5 k + g holds M[4 g + i][k]
__device__ __forceinline__ void offsets_out20(int lane, int (&o)[7]) {
#pragma unroll
    for (int q = 0; q < 7; ++q) {
        const int t = min(16 * q + (lane >> 2), 99);
        o[q] = (4 * (t % 5) + (lane & 3)) * kAA + t / 5;
    }
}
__device__ __forceinline__ void load_out20(const float TT_G *M, const int (&o)[7], Mat20 &A) {
#pragma unroll
    for (int q = 0; q < 7; ++q) A.a[q] = M[o[q]];
}

template <int... T>
__device__ __forceinline__ void contract20(const Mat20 &A, const float (&x)[kAA], v4f (&acc)[5],
                                           std::integer_sequence<int, T...>) {
    ((acc[T % 5] = __builtin_amdgcn_mfma_f32_4x4x1f32(A.a[T / 16], x[T / 5], acc[T % 5], 4, T % 16, 0)), ...);
}
__device__ __forceinline__ void contract20(const Mat20 &A, const float (&x)[kAA], float (&out)[kAA]) {
    v4f acc[5];
#pragma unroll
    for (int g = 0; g < 5; ++g) acc[g] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    contract20(A, x, acc, std::make_integer_sequence<int, 100>{});
#pragma unroll
    for (int i = 0; i < kAA; ++i) out[i] = acc[i / 4][i % 4];
}

// A wave's LDS rows: 5 float4 planes a row.
struct Slots20 {
    static constexpr int kRow = kAA * TT_WAVE;
    float *base;
    int lane;
    __device__ __forceinline__ void put(int s, const float (&r)[kAA]) const {
        float4 *d = reinterpret_cast<float4 *>(base + s * kRow) + lane;
#pragma unroll
        for (int g = 0; g < 5; ++g) d[g * TT_WAVE] = make_float4(r[4 * g], r[4 * g + 1], r[4 * g + 2], r[4 * g + 3]);
    }
    __device__ __forceinline__ void get(int s, float (&r)[kAA]) const {
        const float4 *d = reinterpret_cast<const float4 *>(base + s * kRow) + lane;
#pragma unroll
        for (int g = 0; g < 5; ++g) {
            const float4 x = d[g * TT_WAVE];
            r[4 * g] = x.x;
            r[4 * g + 1] = x.y;
            r[4 * g + 2] = x.z;
            r[4 * g + 3] = x.w;
        }
    }
};

// The profile row of a character code: from LDS, or from the table where it has more codes.
struct Lut20 {
    const float *lds;
    const float TT_C *mem;
    bool staged;
    __device__ __forceinline__ void row(int code, float (&r)[kAA]) const {
        if (staged) {
            const float4 *s = reinterpret_cast<const float4 *>(lds + code * kAA);
#pragma unroll
            for (int g = 0; g < 5; ++g) {
                const float4 x = s[g];
                r[4 * g] = x.x;
                r[4 * g + 1] = x.y;
                r[4 * g + 2] = x.z;
                r[4 * g + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < kAA; ++i) r[i] = mem[code * kAA + i];
        }
    }
};

}  // namespace ttd
