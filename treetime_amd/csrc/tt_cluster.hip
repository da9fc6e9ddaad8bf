// Clustered passes (shared model): marginal, log-likelihood and, up to 5
// states, joint reconstruction of one tree or of many; marginal and
// log-likelihood of 20 states too (tt_cluster20.h).
//
// A tree is cut into connected clusters of up to 64 internal nodes, 256 where
// it is a chain (tt_cluster_plan.hip): the subtrees of at most that size first, then the
// same on what is left, up to the cluster that holds the root.  One wave
// walks a cluster's nodes in depth-first order for 64 patterns.  A row is
// consumed from registers by the next step or waits in one of five LDS slots,
// so inside a cluster no row is read back from memory, there is no barrier,
// and all of a step's loads (descriptor, P(t), tip characters, rows of other
// clusters) have addresses known in advance and are issued a step ahead.
// A pass is one launch per stage of clusters up and down the tree (5 to 7 for
// thousands of tips) instead of one per level.
//
// What bounds it: HBM for large inputs.  Per internal node and pattern, n = 4,
// the marginal pass writes the subtree row (16 B), reads it once on the way
// down, writes profile and state (17 B) and reads about one tip character:
// 50 B, where walking the levels reads every row again for its parent and
// every parent's profile for its children (90 B).  Below that the steps'
// arithmetic, about 160 vector instructions up and 70 down per 64 patterns: of
// 256 trees' 100 GB a pass the leaf stage down moves 61 at 4.2 TB/s (a
// streaming copy: 4.9), the leaf stage up 32 at 3.3.
//
// Measured (start of the pass to its end, against a launch per level, or the
// persistent kernel for the batch): marginal, 5000 tips x 2637 patterns, n = 4:
// 500 -> 305 us; joint of the same: 487 -> 320 us; marginal of 20 uneven trees
// (1.2e8 internal nodes x patterns): 3430 -> 1750 us, joint 3450 -> 1445 us;
// marginal, n = 20, 1000 tips x 4534 patterns: 710 -> 490 us.
//
// The per-(node, pattern) arithmetic is shared with the one-launch pass
// (tt_device.h), so profiles, rows and states are bit-identical to its.
#include "tt_cluster.h"

#include "tt_cluster20.h"
#include "tt_device.h"

namespace {
using namespace ttd;

constexpr int kWaves = TT_BLOCK / TT_WAVE;

// Element p of row `row` of an array of P entries of B bytes a row: a scalar
// base and a 32-bit lane offset, so the access needs no vector address
// arithmetic.  off: p * B, or 0 for every lane of an access whose value is not
// used (one line instead of a row).
template <class V, class T0>
__device__ __forceinline__ const V TT_G *at_row(const T0 TT_G *base, int row, uint32_t row_bytes, uint32_t off) {
    const char TT_G *b = reinterpret_cast<const char TT_G *>(base) + (uint64_t)(uint32_t)row * row_bytes;
    return reinterpret_cast<const V TT_G *>(b + off);
}

template <int N>
__device__ __forceinline__ void read_row(const float TT_G *base, int row, uint32_t row_bytes, uint32_t off, float (&r)[N]) {
    const float TT_G *q = at_row<float>(base, row, row_bytes, off);
    load_rowf<N>(q, r);
}

template <int N>
__device__ __forceinline__ void write_row(float TT_G *base, int row, uint32_t row_bytes, uint32_t off, const float (&r)[N]) {
    store_row<N>(const_cast<float TT_G *>(at_row<float>(base, row, row_bytes, off)), r);
}

// One wave's LDS slots: rows of N floats per lane.
template <int N>
struct Slots {
    static constexpr int kRow = N * TT_WAVE;
    float *base;  // this wave's region
    int lane;
    __device__ __forceinline__ void put(int s, const float (&r)[N]) const {
        float *d = base + s * kRow;
        if constexpr (N == 4) {
            reinterpret_cast<float4 *>(d)[lane] = make_float4(r[0], r[1], r[2], r[3]);
        } else {
#pragma unroll
            for (int i = 0; i < N; ++i) d[i * TT_WAVE + lane] = r[i];
        }
    }
    // the row of tip character `code` from lut, or of slot src & 0xff
    __device__ __forceinline__ void get(int src, int code, const float *lut, float (&r)[N]) const {
        if constexpr (N == 4) {  // one read either way
            const float *d = src < 0 ? lut + code * N : base + (src & 0xff) * kRow + lane * N;
            const float4 x = *reinterpret_cast<const float4 *>(d);
            r[0] = x.x;
            r[1] = x.y;
            r[2] = x.z;
            r[3] = x.w;
        } else if (src < 0) {
#pragma unroll
            for (int i = 0; i < N; ++i) r[i] = lut[code * N + i];
        } else {
            const float *d = base + (src & 0xff) * kRow;
#pragma unroll
            for (int i = 0; i < N; ++i) r[i] = d[i * TT_WAVE + lane];
        }
    }
};

template <int K>
__device__ __forceinline__ void load_matrix(const float TT_C *m, int node, float (&r)[K]) {
#pragma unroll
    for (int i = 0; i < K; ++i) r[i] = m[(size_t)node * K + i];
}

struct UpStep {
    int v, s0, s1, n0, n1, dst, end, vn;  // as ClusterPlan::post; dst & 0xff: slot + 1, bit 8: not binary
    int c0, c1;                            // only with rows of other clusters
};
template <bool MEM>
__device__ __forceinline__ UpStep load_up(const int32_t TT_C *q) {
    return UpStep{q[0], q[1], q[2], q[3], q[4], q[5], q[6], q[7], MEM ? q[8] : 0, MEM ? q[9] : 0};
}
struct DownStep {
    int c, ir, tr, src, par, dst;
};
__device__ __forceinline__ DownStep load_down(const int32_t TT_C *q) {
    return DownStep{q[0], q[1], q[2], q[3], q[4], q[5]};
}

__device__ __forceinline__ bool from_memory(int src) { return src >= 0 && src < kSrcSlot; }

// What a postorder step needs from memory.  Every load is issued for every
// step (of one line, unused, where the step has no such child), so that the
// loads of a step go straight into registers a step ahead and nothing
// waits for them before their use.
template <int N, bool MEM>
struct UpRaw {
    int code[2];
    float row[MEM ? 2 : 1][MEM ? N : 1];
    double off[MEM ? 2 : 1];
};

template <int N, bool MEM, bool PART>
__device__ __forceinline__ void up_fetch(const uint8_t TT_G *codes, const float TT_G *rows, const double TT_G *part,
                                         int P, const UpStep &q, int p, UpRaw<N, MEM> &R) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int s = c ? q.s1 : q.s0;
        const bool tip = s < 0;
        R.code[c] = *at_row<uint8_t>(codes, tip ? -s - 1 : 0, (uint32_t)P, tip ? (uint32_t)p : 0u);
        if constexpr (MEM) {
            const bool m = from_memory(s);
            read_row<N>(rows, m ? s : 0, (uint32_t)P * N * 4, m ? (uint32_t)p * N * 4 : 0u, R.row[c]);
            if constexpr (PART) R.off[c] = *at_row<double>(part, m ? (c ? q.c1 : q.c0) : 0, (uint32_t)P * 8, m ? (uint32_t)p * 8 : 0u);
        }
    }
}

// Rows of a step's children that are in LDS (tip characters, slots).
template <int N, bool MEM>
__device__ __forceinline__ void up_lds(const UpStep &q, const UpRaw<N, MEM> &R, const Slots<N> &slots, const float *lut,
                                       float (&r)[2][N]) {
    slots.get(q.s0 < 0 ? q.s0 : q.s0 >= kSrcSlot ? q.s0 : 0, R.code[0], lut, r[0]);
    if (q.s1 < 0) slots.get(q.s1, R.code[1], lut, r[1]);  // else the row just before, or from memory
}

// The marginal postorder steps [0, n) of a program for pattern p; row holds
// the last row, off the log normalisers of its subtree.  MEM: some steps read
// rows of other clusters.
//
// The next step's branch matrices (scalar registers) and its children's rows
// in LDS are requested as soon as a step is done, ahead of the address
// arithmetic of the fetch.
template <int N, bool MEM>
__device__ __forceinline__ void up_marginal(const TreeDev &T, const ClusterDev &C, const int32_t TT_C *prog, int n, int p,
                                            const float *s_lut, const Slots<N> &slots, float (&row)[N], double &off) {
    constexpr int NN = N * N;
    const auto codes = (const uint8_t TT_G *)T.tip_codes;
    const auto sub = T.sub;
    const auto part = C.part;
    const auto D32 = T.D32;
    const auto offs = T.offs;
    const int P = T.P;
    const uint32_t rb = (uint32_t)P * N * 4, ro = (uint32_t)p * N * 4;
    LogAcc acc;
    off = 0.0;
    float D0[NN], D1[NN];   // branch matrices of the step at hand
    float lds[2][N];        // its rows from LDS
    auto step = [&](const UpStep &q, const UpRaw<N, MEM> &R) {
        if (!(q.dst & 0x100)) {
            float r0[N], r1[N];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                r0[i] = lds[0][i];
                r1[i] = q.s1 < 0 ? lds[1][i] : row[i];
            }
            if constexpr (MEM) {
                const bool m0 = from_memory(q.s0), m1 = from_memory(q.s1);
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    r0[i] = m0 ? R.row[0][i] : r0[i];
                    r1[i] = m1 ? R.row[1][i] : r1[i];
                }
                off += (m0 ? R.off[0] : 0.0) + (m1 ? R.off[1] : 0.0);
            }
            const double f = bin_row<N>(r0, r1, (const float *)D0, (const float *)D1, row);
            acc.mul(f);
            if (offs) offs[(size_t)q.v * P + p] = log(f);
            write_row<N>(sub, q.v, rb, ro, row);
        } else {
            if constexpr (MEM) {
                const int e0 = T.child_ptr[q.v], e1 = T.child_ptr[q.v + 1];
                for (int e = e0; e < e1; ++e) {
                    const int c = C.edge_cluster[e];
                    if (c >= 0) off += part[(size_t)c * P + p];
                }
            }
            post_node_f<N>(T, q.v, p, s_lut, acc, [&](int cref, float (&r)[N]) { child_row<N>(T, cref, p, s_lut, r); },
                           [](int e) { return wave_uniform(e); }, row);
        }
        if (q.dst & 0xff) slots.put((q.dst & 0xff) - 1, row);
        if (q.end >= 0) {
            off += acc.log_value();
            part[(size_t)q.end * P + p] = off;
        }
    };
    auto reset = [&](int ended) {  // the next step opens another cluster
        if (ended >= 0) {
            acc = LogAcc();
            off = 0.0;
        }
    };
    auto at = [&](int k) { return load_up<MEM>(prog + (size_t)kClPost * min(k, n - 1)); };
    auto fetch = [&](const UpStep &q, UpRaw<N, MEM> &R) { up_fetch<N, MEM, true>(codes, sub, part, P, q, p, R); };
    auto ready = [&](const UpStep &q, const UpRaw<N, MEM> &R) {
        load_matrix<NN>(D32, q.n0, D0);
        load_matrix<NN>(D32, q.n1, D1);
        up_lds<N, MEM>(q, R, slots, s_lut, lds);
    };
    // two steps to an iteration, each with its own registers; the matrices
    // are not carried around the loop (they would leave the scalar registers)
    UpStep a = at(0), nb = at(1);
    UpRaw<N, MEM> A, B;
    fetch(a, A);
    int ended = -1;
    for (int k = 0;;) {
        ready(a, A);
        reset(ended);
        const UpStep b = nb;
        fetch(b, B);
        const UpStep na = at(k + 2);
        step(a, A);
        if (++k == n) break;
        ready(b, B);
        reset(a.end);
        a = na;
        fetch(a, A);
        nb = at(k + 2);
        step(b, B);
        if (++k == n) break;
        ended = b.end;
    }
}

template <int N>
struct DownRaw {
    float pp[N], sub[N];
    int code;
};

// The marginal preorder steps [0, n) of a program; row: the root's profile
// when the program starts at the root.  Loads as in up_marginal.
template <int N, bool TIPS>
__device__ __forceinline__ void down_marginal(const TreeDev &T, const int32_t TT_C *prog, int n, int p,
                                              const float *s_lut, const Slots<N> &slots, float (&row)[N]) {
    constexpr int NN = N * N;
    const auto codes = (const uint8_t TT_G *)T.tip_codes;
    const auto sub = T.sub;
    const auto prof = T.prof;
    const auto states = T.states;
    const auto P32 = T.P32;
    const int P = T.P;
    const uint32_t rb = (uint32_t)P * N * 4, ro = (uint32_t)p * N * 4;
    auto step = [&](const DownStep &q, const DownRaw<N> &R, const float (&M)[NN]) {
        if (q.src >= 0) {
            float pp[N], sb[N], out[N];
            if (q.src >= kSrcAcc) {
#pragma unroll
                for (int i = 0; i < N; ++i) pp[i] = row[i];
            } else if (q.src >= kSrcSlot) {
                slots.get(q.src, 0, s_lut, pp);
            } else {
#pragma unroll
                for (int i = 0; i < N; ++i) pp[i] = R.pp[i];
            }
#pragma unroll
            for (int i = 0; i < N; ++i) sb[i] = R.sub[i];
            if constexpr (TIPS)
                if (q.ir < 0) {
#pragma unroll
                    for (int i = 0; i < N; ++i) sb[i] = s_lut[R.code * N + i];
                }
            const int jm = pre_row<N>(pp, sb, M, out);
            write_row<N>(prof, q.c, rb, ro, out);
            *const_cast<uint8_t TT_G *>(at_row<uint8_t>(states, q.c, (uint32_t)P, (uint32_t)p)) = (uint8_t)jm;
            if (!TIPS || q.ir >= 0) {
#pragma unroll
                for (int i = 0; i < N; ++i) row[i] = out[i];
            }
        }
        if (q.dst >= 0) slots.put(q.dst, row);
    };
    auto at = [&](int k) { return load_down(prog + (size_t)kClPre * min(k, n - 1)); };
    auto fetch = [&](const DownStep &q, DownRaw<N> &R) {
        const bool m = from_memory(q.src);
        read_row<N>(prof, q.par, rb, m ? ro : 0u, R.pp);
        read_row<N>(sub, max(q.ir, 0), rb, q.ir >= 0 ? ro : 0u, R.sub);
        if constexpr (TIPS)
            R.code = *at_row<uint8_t>(codes, max(q.tr, 0), (uint32_t)P, q.ir < 0 ? (uint32_t)p : 0u);
    };
    DownStep a = at(0), nb = at(1);
    DownRaw<N> A, B;
    fetch(a, A);
    for (int k = 0;;) {  // as in up_marginal
        float MA[NN], MB[NN];
        load_matrix<NN>(P32, a.c, MA);
        const DownStep b = nb;
        fetch(b, B);
        const DownStep na = at(k + 2);
        step(a, A, MA);
        if (++k == n) break;
        load_matrix<NN>(P32, b.c, MB);
        a = na;
        fetch(a, A);
        nb = at(k + 2);
        step(b, B, MB);
        if (++k == n) break;
    }
}

// ---- 20 states (tt_cluster20.h) --------------------------------------------
// As up_marginal and down_marginal, with the branch matrices in vector
// registers, requested a step ahead like everything else: one wave has a SIMD
// nearly to itself (232 registers in the leaf stage up, 332 in the middle ones;
// 16.6 KB of LDS), so nothing else covers a wait.

template <bool MEM>
struct Up20 {
    int code[2];
    v4f row[MEM ? 2 : 1][MEM ? 5 : 1];
    double off[MEM ? 2 : 1];
    Mat20 D[2];
    // wait here for the loads of a step without rows from memory
    __device__ __forceinline__ void arrive() {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            asm volatile("" : "+v"(code[c]));
            D[c].arrive();
        }
    }
};

template <bool MEM>
__device__ __forceinline__ void up_marginal20(const TreeDev &T, const ClusterDev &C, const int32_t TT_C *prog, int n,
                                              int p, const Lut20 &lut, const Rows20 &rows, float (&row)[kAA],
                                              double &off) {
    const auto codes = (const uint8_t TT_G *)T.tip_cc;
    const auto D32 = (const float TT_G *)T.D32;
    const float TT_G *tab = T.tiptab;
    const auto sub = T.sub;
    const auto part = C.part;
    const auto offs = T.offs;
    const int P = T.P, lane = rows.lane;
    LogAcc acc;
    off = 0.0;
    auto at = [&](int k) { return load_up<MEM>(prog + (size_t)kClPost * min(k, n - 1)); };
    auto fetch = [&](const UpStep &q, Up20<MEM> &R) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int s = c ? q.s1 : q.s0;
            const bool tip = s < 0;
            R.code[c] = *at_row<uint8_t>(codes, tip ? -s - 1 : 0, (uint32_t)P, tip ? (uint32_t)p : 0u);
            load_mat20(tip && tab ? tab + (size_t)(-s - 1) * kTab20 : D32 + (size_t)(c ? q.n1 : q.n0) * (kAA * kAA), lane,
                       R.D[c]);
            if constexpr (MEM) {
                const bool m = from_memory(s);
                rows.request(sub, m ? s : 0, m, R.row[c]);
                R.off[c] = *at_row<double>(part, m ? (c ? q.c1 : q.c0) : 0, (uint32_t)P * 8, m ? (uint32_t)p * 8 : 0u);
            }
        }
    };
    auto step = [&](const UpStep &q, const Up20<MEM> &R, Up20<MEM> &next) {
        if (!(q.dst & 0x100)) {
            float r[2][kAA], d[2][kAA];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int s = c ? q.s1 : q.s0;
                const float *from = s < 0 ? lut.lds + (lut.staged ? R.code[c] : 0) * kAA : rows.slot(s & 1);
                if constexpr (MEM) {
                    const bool m = from_memory(s);
                    rows.lay(R.row[c]);
                    from = m ? rows.laid() : from;
                    off += m ? R.off[c] : 0.0;
                }
                rows.get(from, r[c]);
#pragma unroll
                for (int i = 0; i < kAA; ++i) r[c][i] = s >= kSrcAcc ? row[i] : r[c][i];
                if (s < 0 && !lut.staged)
#pragma unroll
                    for (int i = 0; i < kAA; ++i) r[c][i] = lut.mem[R.code[c] * kAA + i];
                if (s < 0 && tab)
                    rows.get(rows.spread(R.D[c]) + R.code[c] * kAA, d[c]);
                else
                    contract20(R.D[c], r[c], d[c]);
            }
            const double f = bin_row_d<kAA>(r[0], d[0], r[1], d[1], row);
            acc.mul(f);
            // the next step's loads, ahead of the stores: a wait for them later
            // would wait for these stores as well (leaf stage up, 1000 tips x
            // 4534 patterns: 131 -> 126 us; the other kernels' steps are too
            // short for their loads to have arrived)
            if constexpr (!MEM) next.arrive();
            if (offs) offs[(size_t)q.v * P + p] = log(f);
            rows.store(sub, q.v, row);
        } else {
            if constexpr (MEM) {
                const int e0 = T.child_ptr[q.v], e1 = T.child_ptr[q.v + 1];
                for (int e = e0; e < e1; ++e) {
                    const int c = C.edge_cluster[e];
                    if (c >= 0) off += part[(size_t)c * P + p];
                }
            }
            post_node_d<kAA>(
                T, q.v, p, acc,
                [&](int ref, float (&r)[kAA]) {
                    if (ref < 0) {
                        const int code = T.tip_codes[(size_t)(-ref - 1) * P + p];
#pragma unroll
                        for (int i = 0; i < kAA; ++i) r[i] = T.lut[code * kAA + i];
                    } else {
                        load_rowf<kAA>(sub + ((size_t)ref * P + p) * kAA, r);
                    }
                },
                [](int e) { return wave_uniform(e); },
                [&](int node, const float (&r)[kAA], float (&d)[kAA]) {
                    Mat20 A;
                    load_mat20(D32 + (size_t)node * (kAA * kAA), lane, A);
                    contract20(A, r, d);
                },
                row);
        }
        if (q.dst & 0xff) rows.put((q.dst & 0xff) - 1, row);
        if (q.end >= 0) {
            off += acc.log_value();
            part[(size_t)q.end * P + p] = off;
        }
    };
    UpStep a = at(0), nb = at(1);
    Up20<MEM> A, B;
    fetch(a, A);
    int ended = -1;
    auto reset = [&](int e) {  // the next step opens another cluster
        if (e >= 0) {
            acc = LogAcc();
            off = 0.0;
        }
    };
    for (int k = 0;;) {
        reset(ended);
        const UpStep b = nb;
        fetch(b, B);
        const UpStep na = at(k + 2);
        step(a, A, B);
        if (++k == n) break;
        reset(a.end);
        a = na;
        fetch(a, A);
        nb = at(k + 2);
        step(b, B, A);
        if (++k == n) break;
        ended = b.end;
    }
}

struct Down20 {
    v4f pp[5], sub[5];
    int code;
    Mat20 in, out;
};

template <bool TIPS>
__device__ __forceinline__ void down_marginal20(const TreeDev &T, const int32_t TT_C *prog, int n, int p,
                                                const Lut20 &lut, const Rows20 &rows, float (&row)[kAA]) {
    const auto codes = (const uint8_t TT_G *)T.tip_cc;
    const auto P32 = (const float TT_G *)T.P32, PT32 = (const float TT_G *)T.PT32;
    const auto sub = T.sub;
    const auto prof = T.prof;
    const auto states = T.states;
    const int P = T.P, lane = rows.lane;
    auto at = [&](int k) { return load_down(prog + (size_t)kClPre * min(k, n - 1)); };
    auto fetch = [&](const DownStep &q, Down20 &R) {
        const bool m = from_memory(q.src);
        rows.request(prof, q.par, m, R.pp);
        rows.request(sub, max(q.ir, 0), q.ir >= 0, R.sub);
        if constexpr (TIPS)
            R.code = *at_row<uint8_t>(codes, max(q.tr, 0), (uint32_t)P, q.ir < 0 ? (uint32_t)p : 0u);
        load_mat20(P32 + (size_t)q.c * (kAA * kAA), lane, R.in);
        load_mat20(PT32 + (size_t)q.c * (kAA * kAA), lane, R.out);
    };
    auto step = [&](const DownStep &q, const Down20 &R) {
        if (q.src >= 0) {
            float x[kAA], sb[kAA], m[kAA];
            rows.lay(R.pp);
            rows.get(from_memory(q.src) ? rows.laid() : rows.slot(q.src & 1), x);
#pragma unroll
            for (int i = 0; i < kAA; ++i) x[i] = q.src >= kSrcAcc ? row[i] : x[i];
            rows.lay(R.sub);
            const float *from = rows.laid();
            if constexpr (TIPS) from = q.ir < 0 ? lut.lds + (lut.staged ? R.code : 0) * kAA : from;
            rows.get(from, sb);
            if constexpr (TIPS)
                if (q.ir < 0 && !lut.staged)
#pragma unroll
                    for (int i = 0; i < kAA; ++i) sb[i] = lut.mem[R.code * kAA + i];
            contract20(R.in, sb, m);
            // the outgroup message by division, evolved down the branch (pre_row)
#pragma unroll
            for (int i = 0; i < kAA; ++i) x[i] = fmaxf((float)TT_TINY, x[i]) * __builtin_amdgcn_rcpf(m[i]);
            contract20(R.out, x, m);
            float xs[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // short chains: less rounding
#pragma unroll
            for (int i = 0; i < kAA; ++i) {
                m[i] *= sb[i];
                xs[i % 4] += m[i];
            }
            const int jm = argmax_first<kAA>(m);
            const float xi = __builtin_amdgcn_rcpf((xs[0] + xs[1]) + (xs[2] + xs[3]));
#pragma unroll
            for (int i = 0; i < kAA; ++i) x[i] = m[i] * xi;
            rows.store(prof, q.c, x);
            *const_cast<uint8_t TT_G *>(at_row<uint8_t>(states, q.c, (uint32_t)P, (uint32_t)p)) = (uint8_t)jm;
            if (!TIPS || q.ir >= 0) {
#pragma unroll
                for (int i = 0; i < kAA; ++i) row[i] = x[i];
            }
        }
        if (q.dst >= 0) rows.put(q.dst, row);
    };
    DownStep a = at(0), nb = at(1);
    Down20 A, B;
    fetch(a, A);
    for (int k = 0;;) {
        const DownStep b = nb;
        fetch(b, B);
        const DownStep na = at(k + 2);
        step(a, A);
        if (++k == n) break;
        a = na;
        fetch(a, A);
        nb = at(k + 2);
        step(b, B);
        if (++k == n) break;
    }
}

__device__ __forceinline__ double wave_add(double x) {
#pragma unroll
    for (int off = TT_WAVE / 2; off > 0; off >>= 1) x += __shfl_xor(x, off, TT_WAVE);
    return x;
}

// Sum of the tree's 64-pattern partials into its total.
__device__ __forceinline__ void tree_total(const TreeDev &T, const ClusterDev &C) {
    const int tiles = (T.P + TT_WAVE - 1) / TT_WAVE;
    double a = 0.0;
    for (int i = threadIdx.x; i < tiles; i += TT_BLOCK) a += C.bpart[i];
    a = block_sum(a);
    if (threadIdx.x == 0) {
        T.total[0] = a;
        if (C.out) C.out[0] = a;
    }
}

// mode bit 0: tips reconstructed; bit 1: no preorder.  One kernel per role:
// the leaf stage (most of the work) keeps no registers for rows of other
// clusters on the way up, and none of the postorder's on the way down.
template <int N, ClusterRole ROLE, bool TIPS>
__device__ __forceinline__ void marginal_item(const TreeDev &T, const ClusterDev &C, const ClusterItem TT_C &it, int mode) {
    constexpr bool kUp = ROLE != kRoleDown, kLut = kUp || TIPS;
    if constexpr (ROLE == kRoleTable) {
        if constexpr (N == kAA) tip_tables20(T, C, it.group);
        return;
    }
    if constexpr (ROLE == kRoleDown)
        if (it.kind == kClTotal) {
            tree_total(T, C);
            return;
        }
    constexpr int kCodes = N == kAA ? kLut20 : 256, kSlots = N == kAA ? kSlots20 + 1 : kClusterSlots;
    __shared__ float s_lut[kLut ? kCodes * N : 1];
    __shared__ float s_slot[kWaves][kSlots * N * TT_WAVE];
    const int lane = threadIdx.x & (TT_WAVE - 1), w = wave_uniform(threadIdx.x / TT_WAVE);
    if constexpr (kLut) {
        const int n_codes = N == kAA ? T.n_cc : T.n_codes;
        const float TT_C *lut = N == kAA ? T.lut_c : T.lut;
        if (n_codes <= kCodes)
            for (int i = threadIdx.x; i < n_codes * N; i += TT_BLOCK) s_lut[i] = lut[i];
        __syncthreads();
    }
    const int tile = it.group * kWaves + w, at = tile * TT_WAVE + lane;
    if (tile * TT_WAVE >= T.P) return;
    constexpr bool kMid = ROLE == kRoleMid;
    const int32_t TT_C *post = C.post + (size_t)kClPost * it.post0, *pre = C.pre[TIPS] + (size_t)kClPre * it.pre0;
    float row[N];
    if constexpr (N == kAA) {
        const int p = min(at, T.P - 1);
        const Rows20 rows(s_slot[w], lane, tile, T.P);
        const Lut20 lut{s_lut, T.lut_c, T.n_cc <= kCodes};
        if (kUp && it.kind != kClDown) {
            double off;
            up_marginal20<kMid>(T, C, post, it.post_n, p, lut, rows, row, off);
            if (!kMid || it.kind != kClTop) return;
            const double lh = root_row<N>(T, p, off, row);  // by all lanes: the way down stores what each holds
            const double contrib = wave_add(at < T.P ? lh : 0.0);
            if (lane == 0) C.bpart[tile] = contrib;
            if (mode & 2) return;
        }
        if constexpr (ROLE != kRoleLeaf) down_marginal20<TIPS>(T, pre, it.pre_n, p, lut, rows, row);
    } else {
        const int p = at;
        const Slots<N> slots{s_slot[w], lane};
        if (kUp && it.kind != kClDown) {
            double contrib = 0.0;
            if (p < T.P) {
                double off;
                up_marginal<N, kMid>(T, C, post, it.post_n, p, s_lut, slots, row, off);
                if (kMid && it.kind == kClTop) contrib = root_row<N>(T, p, off, row);
            }
            if (!kMid || it.kind != kClTop) return;
            contrib = wave_add(contrib);
            if (lane == 0) C.bpart[tile] = contrib;
            if (mode & 2) return;
        }
        if constexpr (ROLE != kRoleLeaf)
            if (p < T.P) down_marginal<N, TIPS>(T, pre, it.pre_n, p, s_lut, slots, row);
    }
}

// ---- joint (max-product) reconstruction ------------------------------------

// max_i PJ_ij tl_i of a tip for every parent state j; the first argmax too
// when its row is kept.
template <int N>
__device__ __forceinline__ void tip_best(const TreeDev &T, const JR<N> (&PJ)[N * N], const JR<N> *tl, int node, int p,
                                         int tips, JR<N> (&msg)[N]) {
    using R = JR<N>;
    R t[N];
#pragma unroll
    for (int i = 0; i < N; ++i) t[i] = tl[i];
    if (tips) {
        int cx[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            R best = PJ[j] * t[0];
            int bi = 0;
#pragma unroll
            for (int i = 1; i < N; ++i) {
                const R val = PJ[i * N + j] * t[i];
                if (val > best) {
                    best = val;
                    bi = i;
                }
            }
            msg[j] *= best;
            cx[j] = bi;
        }
        cx_store<N>(T, node, p, cx);
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            R best = PJ[j] * t[0];
#pragma unroll
            for (int i = 1; i < N; ++i) {
                const R val = PJ[i * N + j] * t[i];
                best = val > best ? val : best;
            }
            msg[j] *= best;
        }
    }
}

template <int K, class R>
__device__ __forceinline__ void load_joint(const R TT_C *m, int node, R (&r)[K]) {
#pragma unroll
    for (int i = 0; i < K; ++i) r[i] = m[(size_t)node * K + i];
}

// The postorder steps of a joint program; returns the root's state when the
// program ends at the root, else -1.
template <int N, bool MEM>
__device__ __forceinline__ int up_joint(const TreeDev &T, const ClusterDev &C, const int32_t TT_C *prog, int n, int p,
                                        const JR<N> *s_lut, const Slots<N> &slots, int tips) {
    using R = JR<N>;
    constexpr int NN = N * N;
    const auto codes = (const uint8_t TT_G *)T.tip_codes;
    const auto Lx = T.Lx;
    const auto PJ = joint_P<N>(T);
    const int P = T.P, root_row = T.root_row;
    const uint32_t rb = (uint32_t)P * N * 4, ro = (uint32_t)p * N * 4;
    float row[N];
    int root_state = -1;
    R J0[NN], J1[NN], JV[NN];  // the children's matrices (tips) and the row's own
    auto load_J = [&](const UpStep &q) {
        load_joint<NN>(PJ, q.n0, J0);
        load_joint<NN>(PJ, q.n1, J1);
    };
    auto step = [&](const UpStep &q, const UpRaw<N, MEM> &W) {
        R msg[N];
        load_joint<NN>(PJ, q.vn, JV);
        if (!(q.dst & 0x100)) {
#pragma unroll
            for (int i = 0; i < N; ++i) msg[i] = R(1);
            auto mul = [&](const float (&r)[N]) {
#pragma unroll
                for (int i = 0; i < N; ++i) msg[i] *= (R)r[i];
            };
            if (q.s0 < 0) {
                tip_best<N>(T, J0, s_lut + W.code[0] * N, q.n0, p, tips, msg);
            } else if (q.s0 >= kSrcSlot) {
                float r[N];
                slots.get(q.s0, 0, nullptr, r);
                mul(r);
            } else if constexpr (MEM) {
                mul(W.row[0]);
            }
            if (q.s1 < 0)
                tip_best<N>(T, J1, s_lut + W.code[1] * N, q.n1, p, tips, msg);
            else if (q.s1 >= kSrcSlot)
                mul(row);
            else if constexpr (MEM)
                mul(W.row[1]);
        } else {
            joint_children<N>(T, q.v, p, msg, tips);
        }
        if (q.v == root_row) {
            root_state = root_joint_row<N>(T, p, msg);
            return;
        }
        int cx[N];
        joint_row<N>(JV, msg, row, cx);
        write_row<N>(Lx, q.v, rb, ro, row);
        cx_store<N>(T, q.vn, p, cx);
        if (q.dst & 0xff) slots.put((q.dst & 0xff) - 1, row);
    };
    auto at = [&](int k) { return load_up<false>(prog + (size_t)kClPost * min(k, n - 1)); };
    auto fetch = [&](const UpStep &q, UpRaw<N, MEM> &W) {
        up_fetch<N, MEM, false>(codes, Lx, nullptr, P, q, p, W);
    };
    UpStep a = at(0), nb = at(1);
    UpRaw<N, MEM> A, B;
    fetch(a, A);
    for (int k = 0;;) {  // as in up_marginal
        load_J(a);
        const UpStep b = nb;
        fetch(b, B);
        const UpStep na = at(k + 2);
        step(a, A);
        if (++k == n) break;
        load_J(b);
        a = na;
        fetch(a, A);
        nb = at(k + 2);
        step(b, B);
        if (++k == n) break;
    }
    return root_state;
}

struct BackRaw {
    int ps, cx, code;
};

// A branch's score term on its way: its log P entry (an internal child), or
// those of its parent's state's column (a tip, joint_tip_term).
template <int N>
struct BackTerm {
    double v[N] = {};
    int code = 0;
    bool tip = false;
};

// The backtrack steps (treeanc.py:1048-1063) and the FP64 score of the
// decoded states of the program's branches; state: the root's when the
// program starts there.  Loads as in up_marginal.  The entries of a branch's
// term can be asked for only when its parent's state is known; the term is
// added two steps later, so that no step waits for them.
template <int N>
__device__ __forceinline__ double back_joint(const TreeDev &T, const int32_t TT_C *prog, int n, int p,
                                             const double *s_ll, int *s_state, int lane, int state, int tips) {
    const auto codes = (const uint8_t TT_G *)T.tip_codes;
    const auto states = T.states;
    const auto cxw = cx_words<N>(T);
    const auto logP = (const double TT_G *)T.logP64;
    const int P = T.P;
    double sc = 0.0;
    auto settle = [&](const BackTerm<N> &t) {
        double b = t.v[0];
        if (t.tip) {
            b = -DBL_MAX;
#pragma unroll
            for (int i = 0; i < N; ++i) b = fmax(b, t.v[i] + s_ll[t.code * N + i]);
        }
        sc += b;
    };
    // term: the one of two steps before, then this step's
    auto step = [&](const DownStep &q, const BackRaw &R, BackTerm<N> &term) {
        settle(term);
        term.tip = false;
        term.v[0] = 0.0;
        if (q.src >= 0) {
            const int ps = q.src >= kSrcAcc ? state : q.src >= kSrcSlot ? s_state[(q.src & 0xff) * TT_WAVE + lane] : R.ps;
            const int cs = cx_unpack<N>(R.cx, ps);
            const bool inner = q.ir >= 0;
            if (inner || tips)
                *const_cast<uint8_t TT_G *>(at_row<uint8_t>(states, q.c, (uint32_t)P, (uint32_t)p)) = (uint8_t)cs;
            const double TT_G *e = logP + (size_t)q.c * (N * N);
            if (inner) {
                term.v[0] = e[(uint32_t)(cs * N + ps)];
                state = cs;
            } else {
                term.tip = true;
                term.code = R.code;
#pragma unroll
                for (int i = 0; i < N; ++i) term.v[i] = e[(uint32_t)(i * N + ps)];
            }
        }
        if (q.dst >= 0) s_state[q.dst * TT_WAVE + lane] = state;
    };
    auto at = [&](int k) { return load_down(prog + (size_t)kClPre * min(k, n - 1)); };
    auto fetch = [&](const DownStep &q, BackRaw &R) {
        const bool m = from_memory(q.src), c = q.ir >= 0 || tips;
        R.ps = *at_row<uint8_t>(states, q.par, (uint32_t)P, m ? (uint32_t)p : 0u);
        R.cx = *at_row<CxWord<N>>(cxw, q.c, (uint32_t)(P * sizeof(CxWord<N>)), c ? (uint32_t)(p * sizeof(CxWord<N>)) : 0u);
        R.code = *at_row<uint8_t>(codes, max(q.tr, 0), (uint32_t)P, q.ir < 0 ? (uint32_t)p : 0u);
    };
    DownStep a = at(0), nb = at(1);
    BackRaw A, B;
    BackTerm<N> TA, TB;
    fetch(a, A);
    for (int k = 0;;) {
        const DownStep b = nb;
        fetch(b, B);
        const DownStep na = at(k + 2);
        step(a, A, TA);
        if (++k == n) {
            settle(TB);
            settle(TA);
            return sc;
        }
        a = na;
        fetch(a, A);
        nb = at(k + 2);
        step(b, B, TB);
        if (++k == n) {
            settle(TA);
            settle(TB);
            return sc;
        }
    }
}

// Log-likelihood of the decoded states of 64 patterns: the tasks' score rows,
// every fourth to a wave, in task order.
template <int N>
__device__ __forceinline__ void joint_sum(const TreeDev &T, const ClusterDev &C, int tile) {
    __shared__ double s_sum[kWaves][TT_WAVE];
    const int lane = threadIdx.x & (TT_WAVE - 1), w = threadIdx.x / TT_WAVE;
    const int p = tile * TT_WAVE + lane;
    double a = 0.0;
    if (p < T.P) {
#pragma unroll 8
        for (int r = w; r < C.n_tasks; r += kWaves) a += C.score[(size_t)r * T.P + p];
    }
    s_sum[w][lane] = a;
    __syncthreads();
    if (w > 0) return;
    double contrib = 0.0;
    if (p < T.P) {
        double lp = log(T.pi[T.states[(size_t)T.root * T.P + p]]);
#pragma unroll
        for (int q = 0; q < kWaves; ++q) lp += s_sum[q][lane];
        T.jseqlh[p] = lp;
        contrib = T.mult[p] * lp;
    }
    contrib = wave_add(contrib);
    if (lane == 0) C.bpart[tile] = contrib;
}

// mode bit 0: tips reconstructed; bit 1: the root states are given
template <int N, ClusterRole ROLE>
__device__ __forceinline__ void joint_item(const TreeDev &T, const ClusterDev &C, const ClusterItem TT_C &it, int mode) {
    if constexpr (ROLE == kRoleTotal) {
        tree_total(T, C);
    } else if constexpr (ROLE == kRoleFinal) {
        joint_sum<N>(T, C, it.group);
    } else {
        using R = JR<N>;
        constexpr bool kUp = ROLE != kRoleDown, kBack = ROLE != kRoleLeaf;
        __shared__ R s_lut[kUp ? 256 * N : 1];
        __shared__ double s_ll[kBack ? 256 * N : 1];
        // slots: rows on the way up, one state per lane on the way down
        __shared__ float s_slot[kWaves][kClusterSlots * (kUp ? N : 1) * TT_WAVE];
        const int lane = threadIdx.x & (TT_WAVE - 1), w = wave_uniform(threadIdx.x / TT_WAVE);
        const int tips = mode & 1;
        for (int i = threadIdx.x; i < T.n_codes * N; i += TT_BLOCK) {
            if constexpr (kUp) s_lut[i] = joint_lut<N>(T)[i];
            if constexpr (kBack) s_ll[i] = T.loglut[i];
        }
        __syncthreads();
        const int tile = it.group * kWaves + w, p = tile * TT_WAVE + lane;
        if (p >= T.P) return;
        int state = -1;
        if constexpr (kUp)
            if (it.kind != kClDown) {
                if (ROLE == kRoleMid && (mode & 2))
                    state = T.states[(size_t)T.root * T.P + p];
                else
                    state = up_joint<N, ROLE == kRoleMid>(T, C, C.post + (size_t)kClPost * it.post0, it.post_n, p, s_lut,
                                                          Slots<N>{s_slot[w], lane}, tips);
                if (ROLE == kRoleLeaf || it.kind != kClTop) return;
            }
        // the score needs every branch, so the program with the tips
        if constexpr (kBack)
            C.score[(size_t)it.task * T.P + p] =
                back_joint<N>(T, C.pre[1] + (size_t)kClPre * it.pre0, it.pre_n, p, s_ll,
                              reinterpret_cast<int *>(s_slot[w]), lane, state, tips);
    }
}

// One tree, or the trees of a batch.
template <int N, ClusterRole ROLE, bool TIPS>
__global__ __launch_bounds__(TT_BLOCK) void k_cluster_marginal(TreeDev T, ClusterDev C, const ClusterItem *items, int mode) {
    marginal_item<N, ROLE, TIPS>(T, C, ((const ClusterItem TT_C *)items)[blockIdx.x], mode);
}
template <int N, ClusterRole ROLE>
__global__ __launch_bounds__(TT_BLOCK) void k_cluster_joint(TreeDev T, ClusterDev C, const ClusterItem *items, int mode) {
    joint_item<N, ROLE>(T, C, ((const ClusterItem TT_C *)items)[blockIdx.x], mode);
}
template <int N, ClusterRole ROLE, bool TIPS>
__global__ __launch_bounds__(TT_BLOCK) void k_pool_marginal(const BatchTreeDev *trees, const ClusterDev *cl,
                                                            const ClusterItem *items, int mode) {
    const ClusterItem TT_C &it = ((const ClusterItem TT_C *)items)[blockIdx.x];
    marginal_item<N, ROLE, TIPS>(((const BatchTreeDev TT_C *)trees)[it.tree].T, ((const ClusterDev TT_C *)cl)[it.tree], it,
                                 mode);
}
template <int N, ClusterRole ROLE>
__global__ __launch_bounds__(TT_BLOCK) void k_pool_joint(const BatchTreeDev *trees, const ClusterDev *cl,
                                                         const ClusterItem *items, int mode) {
    const ClusterItem TT_C &it = ((const ClusterItem TT_C *)items)[blockIdx.x];
    joint_item<N, ROLE>(((const BatchTreeDev TT_C *)trees)[it.tree].T, ((const ClusterDev TT_C *)cl)[it.tree], it, mode);
}

#define TT_CLUSTER_DISPATCH(n, CALL)                     \
    switch (n) {                                         \
        case 2: { constexpr int N_ = 2; CALL; } break;   \
        case 3: { constexpr int N_ = 3; CALL; } break;   \
        case 4: { constexpr int N_ = 4; CALL; } break;   \
        case 5: { constexpr int N_ = 5; CALL; } break;   \
        default: return hipErrorInvalidValue;            \
    }

#define TT_CLUSTER_DISPATCH20(n, CALL)                   \
    if (n == kAA) {                                      \
        constexpr int N_ = kAA;                          \
        CALL;                                            \
    } else                                               \
        TT_CLUSTER_DISPATCH(n, CALL)

// kernel mode of a pass (bit 1: no way down, or given root states)
int cluster_mode(int what, bool tips) { return (tips ? 1 : 0) | (what == kClLoglik || what == kClFromRoot ? 2 : 0); }

// f(role, tips) as compile-time values
template <class F>
void with_role(ClusterRole role, bool joint, bool tips, F f) {
    using Y = std::true_type;
    using X = std::false_type;
    switch (role) {
        case kRoleLeaf: f(std::integral_constant<ClusterRole, kRoleLeaf>{}, X{}); break;
        case kRoleMid:
            tips && !joint ? f(std::integral_constant<ClusterRole, kRoleMid>{}, Y{})
                           : f(std::integral_constant<ClusterRole, kRoleMid>{}, X{});
            break;
        case kRoleDown:
            tips && !joint ? f(std::integral_constant<ClusterRole, kRoleDown>{}, Y{})
                           : f(std::integral_constant<ClusterRole, kRoleDown>{}, X{});
            break;
        case kRoleTable: f(std::integral_constant<ClusterRole, kRoleTable>{}, X{}); break;
        case kRoleFinal: f(std::integral_constant<ClusterRole, kRoleFinal>{}, X{}); break;
        case kRoleTotal: f(std::integral_constant<ClusterRole, kRoleTotal>{}, X{}); break;
    }
}

}  // namespace

namespace ttk {

bool cluster_states(int n, bool joint) {
    return (n >= 2 && n <= 5) || (n == kAA && !joint && mfma_enabled());
}

hipError_t cluster_launch(const TreeDev &T, const ClusterDev &C, const ClusterItem *items, int n_items, ClusterRole role,
                          int what, bool tips, hipStream_t s) {
    if (n_items <= 0) return hipSuccess;
    const int mode = cluster_mode(what, tips);
    const dim3 grid((unsigned)n_items), block(TT_BLOCK);
    if (what == kClJoint || what == kClFromRoot) {
        TT_CLUSTER_DISPATCH(T.n, with_role(role, true, tips, [&](auto r, auto) {
            if constexpr (r() != kRoleTable) hipLaunchKernelGGL((k_cluster_joint<N_, r()>), grid, block, 0, s, T, C, items, mode);
        }));
    } else {
        TT_CLUSTER_DISPATCH20(T.n, with_role(role, false, tips, [&](auto r, auto t) {
            if constexpr (r() <= kRoleDown || (r() == kRoleTable && N_ == kAA))
                hipLaunchKernelGGL((k_cluster_marginal<N_, r(), t()>), grid, block, 0, s, T, C, items, mode);
        }));
    }
    return hipGetLastError();
}

hipError_t pool_launch(int n, const BatchTreeDev *trees, const ClusterDev *cl, const ClusterItem *items, int n_items,
                       ClusterRole role, int what, bool tips, hipStream_t s) {
    if (n_items <= 0) return hipSuccess;
    const int mode = cluster_mode(what, tips);
    const dim3 grid((unsigned)n_items), block(TT_BLOCK);
    if (what == kClJoint) {
        TT_CLUSTER_DISPATCH(n, with_role(role, true, tips, [&](auto r, auto) {
            if constexpr (r() != kRoleTable) hipLaunchKernelGGL((k_pool_joint<N_, r()>), grid, block, 0, s, trees, cl, items, mode);
        }));
    } else {
        TT_CLUSTER_DISPATCH20(n, with_role(role, false, tips, [&](auto r, auto t) {
            if constexpr (r() <= kRoleDown || (r() == kRoleTable && N_ == kAA))
                hipLaunchKernelGGL((k_pool_marginal<N_, r(), t()>), grid, block, 0, s, trees, cl, items, mode);
        }));
    }
    return hipGetLastError();
}

}  // namespace ttk
