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
constexpr int kSlots20 = kClusterSlots20;
constexpr int kLut20 = 64;  // character codes whose profile rows are staged in LDS

typedef float v4f __attribute__((ext_vector_type(4)));

// A branch matrix (7 registers used), or a tip's table: the deficits of every
// character code's profile down its branch (kTab20 floats; T.tiptab).
struct Mat20 {
    float a[kTab20 / TT_WAVE];
    __device__ __forceinline__ void arrive() {
#pragma unroll
        for (int q = 0; q < kTab20 / TT_WAVE; ++q) asm volatile("" : "+v"(a[q]));
    }
};

// for out_i = sum_k x_k M[k][i]; the tables are padded to whole registers
__device__ __forceinline__ void load_mat20(const float TT_G *M, int lane, Mat20 &A) {
#pragma unroll
    for (int q = 0; q < kTab20 / TT_WAVE; ++q) A.a[q] = M[TT_WAVE * q + lane];
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

// A wave's LDS: rows waiting for another step, and one row region through
// which rows change between memory and lanes.  In memory a
// pattern's row is 80 bytes; 16-byte accesses at that stride take the address
// unit four times the cycles of contiguous ones, so a wave reads and writes
// its 64 rows as 5 contiguous kilobytes and exchanges them here (lane-major
// 16-byte accesses at a stride of 20 words are free of bank conflicts).
struct Rows20 {
    static constexpr int kRow = kAA * TT_WAVE;
    float *base;
    int lane, valid;     // patterns of this tile
    uint32_t row_bytes;  // of a row of all patterns
    uint32_t off[5];     // of this lane's pieces in it

    __device__ __forceinline__ Rows20(float *b, int l, int tile, int P)
        : base(b), lane(l), valid(min(TT_WAVE, P - tile * TT_WAVE)), row_bytes((uint32_t)P * kAA * 4) {
#pragma unroll
        for (int q = 0; q < 5; ++q) off[q] = ((uint32_t)tile * TT_WAVE * 5 + min(q * TT_WAVE + l, valid * 5 - 1)) * 16;
    }
    __device__ __forceinline__ v4f *swap() const { return reinterpret_cast<v4f *>(base + kSlots20 * kRow); }
    // where this lane's row of slot s is, and the one laid out last
    __device__ __forceinline__ const float *slot(int s) const { return base + s * kRow + lane * kAA; }
    __device__ __forceinline__ const float *laid() const {  // lanes past the last pattern repeat it
        return base + kSlots20 * kRow + min(lane, valid - 1) * kAA;
    }

    __device__ __forceinline__ void put(int s, const float (&r)[kAA]) const {
        v4f *d = reinterpret_cast<v4f *>(base + s * kRow) + 5 * lane;
#pragma unroll
        for (int g = 0; g < 5; ++g) d[g] = v4f{r[4 * g], r[4 * g + 1], r[4 * g + 2], r[4 * g + 3]};
    }
    static __device__ __forceinline__ void get(const float *from, float (&r)[kAA]) {
        const v4f *d = reinterpret_cast<const v4f *>(from);
#pragma unroll
        for (int g = 0; g < 5; ++g) {
            const v4f x = d[g];
#pragma unroll
            for (int k = 0; k < 4; ++k) r[4 * g + k] = x[k];
        }
    }
    // exchanges within the wave: its LDS accesses complete in order
    static __device__ __forceinline__ void order() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    }

    // this lane's pieces of a row (use = 0: one line, unused)
    __device__ __forceinline__ void request(const float TT_G *rows, int row, bool use, v4f (&v)[5]) const {
        const char TT_G *b = reinterpret_cast<const char TT_G *>(rows) + (uint64_t)(uint32_t)row * row_bytes;
#pragma unroll
        for (int q = 0; q < 5; ++q) v[q] = *reinterpret_cast<const v4f TT_G *>(b + (use ? off[q] : 0u));
    }
    // a tip's table, for every lane to read its code's deficits from
    __device__ __forceinline__ const float *spread(const Mat20 &A) const {
        float *x = base + kSlots20 * kRow;
        order();
#pragma unroll
        for (int q = 0; q < kTab20 / TT_WAVE; ++q) x[q * TT_WAVE + lane] = A.a[q];
        order();
        return x;
    }
    // lay out a requested row
    __device__ __forceinline__ void lay(const v4f (&v)[5]) const {
        v4f *x = swap();
        order();
#pragma unroll
        for (int q = 0; q < 5; ++q) x[q * TT_WAVE + lane] = v[q];
        order();
    }
    __device__ __forceinline__ void store(float TT_G *rows, int row, const float (&r)[kAA]) const {
        v4f *x = swap();
        order();
#pragma unroll
        for (int g = 0; g < 5; ++g) x[5 * lane + g] = v4f{r[4 * g], r[4 * g + 1], r[4 * g + 2], r[4 * g + 3]};
        order();
        char TT_G *b = reinterpret_cast<char TT_G *>(rows) + (uint64_t)(uint32_t)row * row_bytes;
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const v4f v = x[q * TT_WAVE + lane];
            if (q * TT_WAVE + lane < valid * 5) *reinterpret_cast<v4f TT_G *>(b + off[q]) = v;
        }
    }
};

// The profile rows of the character codes in use (T.lut_c): in LDS, or in the
// table where there are more than kLut20.
struct Lut20 {
    const float *lds;
    const float TT_C *mem;
    bool staged;
};

// A tip's child message is its code's row of its branch's table, formed at the
// start of a pass: at most 25 codes are 25 products instead of one for every
// pattern (leaf stage up, 1000 tips x 4534 patterns: 152 -> 131 us, the tables 8).
__device__ __forceinline__ void tip_tables20(const TreeDev &T, const ClusterDev &C, int group) {
    const int n = T.n_cc * kAA, tips = min(kTableTips, T.n_tips - group * kTableTips);
    for (int e = threadIdx.x; e < tips * n; e += blockDim.x) {
        const int tip = group * kTableTips + e / n, c = e % n / kAA, j = e % kAA;
        const float TT_C *D = T.D32 + (size_t)C.tip_nodes[tip] * (kAA * kAA);
        float a = 0.0f;
#pragma unroll
        for (int i = 0; i < kAA; ++i) a = fmaf(T.lut_c[c * kAA + i], D[i * kAA + j], a);
        T.tiptab[(size_t)tip * kTab20 + e % n] = a;
    }
}

}  // namespace ttd
