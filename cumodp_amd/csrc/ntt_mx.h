// ntt_mx.h -- number-theoretic transforms on the matrix cores of gfx950.
//
// A radix-16 step of a transform is a 16 x 16 matrix product mod p, and
// v_mfma_i32_16x16x64_i8 takes it exactly.  A 32-bit word x is four bytes
// x_a, so
//     y_k = sum_j w^(jk) x_j = sum_(j,a) (w^(jk) 2^(8a) mod p) x_(j,a),
// a contraction over 64 bytes.  Each constant w^(jk) 2^(8a) 2^32 mod p is
// taken in (-p/2, p/2] and written as four signed bytes c_b 256^b, which
// gives four matrices and four 32-bit sums out_b with |out_b| <= 2^20, and
//     T_k = out_0 + 2^8 out_1 + 2^16 out_2 + 2^24 out_3
// is y_k 2^32 mod p.  The instruction's bytes are signed: x ^ 0x80808080
// holds x_a - 128, and the term 128 sum_(j,a) ... that this leaves out is a
// constant per k, added through the accumulator's initial value, which also
// keeps T non-negative.  T < 2^45, so one Montgomery step returns a word below
// p + 4200 for any odd p < 2^31 and any 32-bit input words: nothing is reduced
// between rounds.
//
// Cost per element and radix-16 round: one xor, two shift-adds, one
// multiply-add to join T, two instructions of Montgomery reduction, and three
// for the twiddle of the next round: about ten against 17 to 20 for four
// stages of radix-2 butterflies, with four matrix instructions per 256
// elements running beside them.
//
// Lane layout (64 lanes, lane = 16 g + n): a set is 16 vectors of 16
// elements; lane (n, g) holds elements 4g .. 4g+3 of vector n, both before
// and after the step.  A lane holds V sets (V = 1, 2, 4 or 8).
//
// A tile is W words in LDS holding rows of L = 2^LOGL words (or, LOGC > 0,
// 2^LOGC columns of 2^LOGL words, column index fastest).  Round j works on
// vectors whose 16 elements lie S' = 2^(LOGL-4(j+1)+LOGC) words apart, and is
// followed by the twiddles w_M^(k v), M = 16 S, v the position below the
// digit.  Row lengths that are no power of 16 end with a round that applies
// 16 / 2^t transforms of length 2^t to 16 adjacent words.  Every thread
// writes a round's outputs where it read the inputs, so one barrier separates
// two rounds, and none where both rounds of a wave stay inside the wave's own
// 256 V words: a row of up to 4096 V words has one barrier per direction.
//
// Outputs of the forward transform stand in digit-reversed order; the inverse
// is its exact mirror, so products never permute data.
#pragma once

#include "internal.h"
#include "modarith.h"

#define CM_DEV __device__ __forceinline__

namespace cm {

typedef int mx_v4i __attribute__((ext_vector_type(4)));

// Table of one root family (plan.cpp): matrices of 5 x 64 lanes x 16 bytes
// (four byte matrices, then the initial values of out_0).
enum : int {
    kMxFwd = 0,        // + t: DFT_16 (t = 0) or 16 / 2^t DFTs of length 2^t
    kMxInv = 4,        // + t: inverse of kMxFwd + t, times 1/radix
    kMxInvFirst = 8,   // + t: the same times 2^32
    kMxInvPair = 12,   // kMxInvFirst + 0 times 1/2 (after a radix-2 step in the lanes)
    kMxMats = 13,
};
constexpr int kMxMatWords = 5 * 64;   // 16-byte words per matrix
// |out_b| <= 64 128 128 = 2^20 and the top digits are at most 65, so
// |out_0 + 256 out_1| <= 2^28 + 2^20: an initial value of out_0 at or above
// that makes the low half of T non-negative.  |out_2 + 256 out_3| <= 2^20 +
// 256 64 65 128 < 2^27.04: 2^16 times that is above -2^32 kMxHigh.
constexpr u32 kMxBias = (1u << 28) + (1u << 20);
constexpr u32 kMxHigh = 2100;

// What a kernel needs of a family: matrices, twiddles w_M^(k v) of level M at
// tf[M + k S + v] (M = 16 S, k < 16; inverse powers at ti), the modulus,
// 2^32 mod p, and 2^16 as a run-time value (the compiler turns a multiply-add
// by the literal into three 64-bit shifts and adds).
struct MxCtx {
    const mx_v4i *mat;
    const u32 *tf, *ti;
    u32 p, np, r1, c16;
};

static inline MxCtx mx_ctx(const Family *fam) {
    return MxCtx{(const mx_v4i *)fam->mx_mat, fam->mx_tf, fam->mx_ti, fam->p, fam->np,
                 cm_host_r1(fam->p), 1u << 16};
}

struct MxMat {
    mx_v4i a0, a1, a2, a3, clo;
};

CM_DEV MxMat mx_load_mat(const MxCtx &cx, int which) {
    const mx_v4i *m = cx.mat + which * kMxMatWords + (threadIdx.x & 63);
    return MxMat{m[0], m[64], m[128], m[192], m[256]};
}

// Keeps the scheduler from running several steps of a lane with many sets at
// once: it would exceed 128 registers and spill.
template <int V>
CM_DEV void mx_fence() {
    if constexpr (V >= 2) __builtin_amdgcn_sched_barrier(0);
}

// x <- the radix-16 step of V sets; any 32-bit words in, [0, p + 2 kMxHigh) out
template <int V>
CM_DEV void mx_dft(u32 (&x)[V][4], const MxMat &m, const MxCtx &cx) {
    typedef u32 v2 __attribute__((ext_vector_type(2)));
    const mx_v4i zero = {0, 0, 0, 0};
    // the 64-bit addend {lo, kMxHigh}: its high word stays in its register
    // from set to set (the empty asm hides that it is a constant), so only lo
    // is written
    v2 pair[2] = {{0u, kMxHigh}, {0u, kMxHigh}};
    asm("" : "+v"(pair[0]), "+v"(pair[1]));
#pragma unroll
    for (int s = 0; s < V; ++s) {
        mx_v4i b;
#pragma unroll
        for (int r = 0; r < 4; ++r) b[r] = (int)(x[s][r] ^ 0x80808080u);
        const mx_v4i d0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(m.a0, b, m.clo, 0, 0, 0);
        const mx_v4i d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(m.a1, b, zero, 0, 0, 0);
        const mx_v4i d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(m.a2, b, zero, 0, 0, 0);
        const mx_v4i d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(m.a3, b, zero, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int hi = (int)((u32)d2[r] + ((u32)d3[r] << 8));
            pair[r & 1].x = (u32)d0[r] + ((u32)d1[r] << 8);
            asm("" : "+v"(pair[r & 1]));
            const u64 t = (u64)((int64_t)hi * (int)cx.c16) + __builtin_bit_cast(u64, pair[r & 1]);
            const u32 q = (u32)t * cx.np;
            x[s][r] = (u32)(((u64)q * cx.p + t) >> 32);
        }
        mx_fence<V>();
    }
}

// canonical residue of a word that left mx_dft (below p + 4200; for p < 8192 a
// Montgomery product by one comes first)
CM_DEV u32 mx_canon(u32 v, const MxCtx &cx) {
    if (cx.p < 8192) v = cm_mont_lazy(v, cx.r1, cx.p, cx.np);
    return cm_reduce2p(v, cx.p);
}

constexpr int mx_log2(int v) { return v <= 1 ? 0 : 1 + mx_log2(v >> 1); }

// LDS word of tile word x: four pad words after every 64, so that the 128-bit
// accesses of 16 consecutive lanes fall into distinct banks in every round,
// and offsets inside a round are compile-time constants.
constexpr int mx_phys(int x) { return x + 4 * (x >> 6); }
CM_DEV int mx_phys_d(int x) { return x + 4 * (x >> 6); }
constexpr int mx_lds_words(int w) { return w + (w >> 4); }

// Where lane (n, g) of wave `wave` finds word (s, r) -- set s, element 4g + r
// -- of a round with vectors of stride 2^LOGS: base() + off(s, r).
template <int LOGS, int V>
struct MxMap {
    static constexpr int S = 1 << LOGS;
    static constexpr int RUN = LOGS == 0 ? 4 : (S < V ? S : V);   // contiguous words
    static CM_DEV int base() {
        const int n = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if constexpr (LOGS == 0) {
            return (wave * (16 * V) + n) * 16 + 4 * g;
        } else {
            const int u0 = wave * (16 * V) + V * n;
            return ((u0 >> LOGS) << (LOGS + 4)) + ((4 * g) << LOGS) + (u0 & (S - 1));
        }
    }
    static constexpr int off(int s, int r) {
        return LOGS == 0 ? 256 * s + r
                         : ((s >> LOGS) << (LOGS + 4)) + (r << LOGS) + (s & (S - 1));
    }
    static CM_DEV void load(const u32 *lds, u32 (&x)[V][4]) {
        const u32 *q = lds + mx_phys_d(base());
        if constexpr (LOGS == 0) {
#pragma unroll
            for (int s = 0; s < V; ++s) {
                const uint4 v = *(const uint4 *)(q + mx_phys(off(s, 0)));
                x[s][0] = v.x; x[s][1] = v.y; x[s][2] = v.z; x[s][3] = v.w;
            }
        } else if constexpr (RUN >= 4) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int s = 0; s < V; s += 4) {
                    const uint4 v = *(const uint4 *)(q + mx_phys(off(s, r)));
                    x[s][r] = v.x; x[s + 1][r] = v.y; x[s + 2][r] = v.z; x[s + 3][r] = v.w;
                }
        } else if constexpr (RUN == 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int s = 0; s < V; s += 2) {
                    const uint2 v = *(const uint2 *)(q + mx_phys(off(s, r)));
                    x[s][r] = v.x; x[s + 1][r] = v.y;
                }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int s = 0; s < V; ++s) x[s][r] = q[mx_phys(off(s, r))];
        }
    }
    static CM_DEV void store(u32 *lds, const u32 (&x)[V][4]) {
        u32 *q = lds + mx_phys_d(base());
        if constexpr (LOGS == 0) {
#pragma unroll
            for (int s = 0; s < V; ++s)
                *(uint4 *)(q + mx_phys(off(s, 0))) = make_uint4(x[s][0], x[s][1], x[s][2], x[s][3]);
        } else if constexpr (RUN >= 4) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int s = 0; s < V; s += 4)
                    *(uint4 *)(q + mx_phys(off(s, r))) =
                        make_uint4(x[s][r], x[s + 1][r], x[s + 2][r], x[s + 3][r]);
        } else if constexpr (RUN == 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int s = 0; s < V; s += 2)
                    *(uint2 *)(q + mx_phys(off(s, r))) = make_uint2(x[s][r], x[s + 1][r]);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int s = 0; s < V; ++s) q[mx_phys(off(s, r))] = x[s][r];
        }
    }
};

// Rounds of a length-2^LOGL transform over 2^LOGC interleaved columns.  A
// lane with two or more sets of a row holds both words of the radix-2 step
// that ends a length of 4q + 1 bits, so that step needs no round (PAIR).
template <int LOGL, int LOGC = 0, int V = 1>
struct MxPlan {
    static constexpr int NF = LOGL / 4, T = LOGL % 4;
    static constexpr bool PAIR = LOGC == 0 && T == 1 && V >= 2 && NF >= 1;
    static constexpr int NR = NF + (T && !PAIR ? 1 : 0);
    // log2 of the digit stride (without columns) of round j
    static constexpr int logs(int j) { return j < NF ? LOGL - 4 * (j + 1) : 0; }
    static constexpr int words(int j) { return logs(j) + LOGC; }   // in tile words
};

// A round of stride 2^LOGS words mixes waves when its blocks of 16 S words
// exceed the 256 V words of a wave.
template <int LOGS, int V>
CM_DEV void mx_sync() {
    if constexpr (LOGS > 4 + mx_log2(V)) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// Twiddles w_M^(k v) of the words a lane holds in a round of digit stride
// 2^LOGS over 2^LOGC columns, M = 2^(LOGS+4).
template <int LOGS, int LOGC, int V>
CM_DEV void mx_load_tw(u32 (&tw)[V][4], const u32 *tab) {
    const int n = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int LW = LOGS + LOGC;                       // vector id bits below the block
    static_assert(LOGS > 0, "no twiddles follow the last digit");
    const int u0 = wave * (16 * V) + V * n;
    const int v = (u0 & ((1 << LW) - 1)) >> LOGC;
    const u32 at = (u32)((16 << LOGS) + ((4 * g) << LOGS) + v);
    const u32 *q = (const u32 *)((const char *)tab + (at << 2));
    if constexpr (LOGC >= 2 || (LOGC > 0 && (1 << LOGC) >= V)) {
        // the V columns of a lane share their twiddle
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const u32 w = q[r << LOGS];
#pragma unroll
            for (int s = 0; s < V; ++s) tw[s][r] = w;
        }
    } else if constexpr (LOGC == 1 && V == 4) {
        // two positions of two columns
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint2 w = *(const uint2 *)(q + (r << LOGS));
            tw[0][r] = tw[1][r] = w.x;
            tw[2][r] = tw[3][r] = w.y;
        }
    } else if constexpr (V == 4 && LOGS >= 2) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint4 w = *(const uint4 *)(q + (r << LOGS));
            tw[0][r] = w.x; tw[1][r] = w.y; tw[2][r] = w.z; tw[3][r] = w.w;
        }
    } else if constexpr (V >= 2 && LOGS >= 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int s = 0; s < V; s += 2) {
                const uint2 w = *(const uint2 *)(q + (r << LOGS) + (s & ((1 << LOGS) - 1)));
                tw[s][r] = w.x; tw[s + 1][r] = w.y;
            }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) tw[0][r] = q[r << LOGS];
    }
}

template <int V>
CM_DEV void mx_mul(u32 (&x)[V][4], const u32 (&tw)[V][4], const MxCtx &cx) {
#pragma unroll
    for (int s = 0; s < V; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[s][r] = cm_mont_lazy(x[s][r], tw[s][r], cx.p, cx.np);
    mx_fence<V>();
}

// Radix-2 steps between the words of positions v = 0 and 1 that a lane holds
// after a round of stride 2 (twiddles w_32^k, k = 4g + r, on v = 1), canonical
// out; and the inverse step (times 2) with its twiddles, words below 2p out.
template <int V>
CM_DEV void mx_pair_fwd(u32 (&x)[V][4], const u32 (&w)[4], const MxCtx &cx) {
#pragma unroll
    for (int s = 0; s < V; s += 2)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const u32 a = mx_canon(x[s][r], cx);
            const u32 b = cm_mul_tw(x[s + 1][r], w[r], cx.p, cx.np);
            x[s][r] = cm_add(a, b, cx.p);
            x[s + 1][r] = cm_sub(a, b, cx.p);
        }
    mx_fence<V>();
}

template <int V>
CM_DEV void mx_pair_inv(u32 (&x)[V][4], const u32 (&w)[4], const MxCtx &cx) {
#pragma unroll
    for (int s = 0; s < V; s += 2)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const u32 a = cm_reduce2p(x[s][r], cx.p), b = cm_reduce2p(x[s + 1][r], cx.p);
            x[s][r] = cm_add(a, b, cx.p);
            x[s + 1][r] = cm_mont_lazy(cm_sub(a, b, cx.p), w[r], cx.p, cx.np);
        }
    mx_fence<V>();
}

// w_32^k (k = 4g + r) of a table of levels
CM_DEV void mx_pair_tw(u32 (&w)[4], const u32 *tab) {
    const int g = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = tab[32 + 2 * (4 * g + r) + 1];
}

// Forward rounds J .. NR-1 of NV tiles whose round-J words are in x; leaves
// the last round's outputs in x (in its map).  m: the radix-16 matrix, kept
// through all full rounds; tw: round J's twiddles (unused in the last round).
// Table loads are issued a round ahead, before the exchange that separates
// the rounds.
template <int LOGL, int LOGC, int V, int J, int NV>
CM_DEV void mx_forward(u32 (&x)[NV][V][4], u32 *const (&lds)[NV], const MxCtx &cx, MxMat &m,
                       u32 (&tw)[V][4]) {
    using P = MxPlan<LOGL, LOGC, V>;
    constexpr bool last = J == P::NR - 1;
    u32 w[4];
    if constexpr (last && P::PAIR) mx_pair_tw(w, cx.tf);
#pragma unroll
    for (int a = 0; a < NV; ++a) mx_dft<V>(x[a], m, cx);
    if constexpr (last && P::PAIR) {
#pragma unroll
        for (int a = 0; a < NV; ++a) mx_pair_fwd<V>(x[a], w, cx);
    }
    if constexpr (!last) {
#pragma unroll
        for (int a = 0; a < NV; ++a) {
            mx_mul<V>(x[a], tw, cx);
            MxMap<P::words(J), V>::store(lds[a], x[a]);
        }
        if constexpr (J + 1 == P::NR - 1) {
            if constexpr (P::T != 0 && !P::PAIR) m = mx_load_mat(cx, kMxFwd + P::T);
        } else {
            mx_load_tw<P::logs(J + 1), LOGC, V>(tw, cx.tf);
        }
        mx_sync<P::words(J), V>();
#pragma unroll
        for (int a = 0; a < NV; ++a) MxMap<P::words(J + 1), V>::load(lds[a], x[a]);
        mx_forward<LOGL, LOGC, V, J + 1, NV>(x, lds, cx, m, tw);
    }
}

// What the first forward round needs, loaded before its words arrive.
template <int LOGL, int LOGC, int V>
CM_DEV void mx_forward_begin(MxMat &m, u32 (&tw)[V][4], const MxCtx &cx) {
    using P = MxPlan<LOGL, LOGC, V>;
    m = mx_load_mat(cx, kMxFwd + (P::NF == 0 ? P::T : 0));
    if constexpr (P::NR > 1) mx_load_tw<P::logs(0), LOGC, V>(tw, cx.tf);
}

// Inverse rounds J, J-1 .. 0 of one tile: x holds round J's words, with
// J = NR - 1 the first one.  Leaves round 0's outputs (natural order, times
// 1/L) in x, words in [0, p + 4200).  m: round J's matrix; tw: its twiddles
// (none in the first round).
template <int LOGL, int LOGC, int V, int J>
CM_DEV void mx_inverse(u32 (&x)[V][4], u32 *lds, const MxCtx &cx, MxMat &m, u32 (&tw)[V][4]) {
    using P = MxPlan<LOGL, LOGC, V>;
    constexpr bool first = J == P::NR - 1;
    if constexpr (!first) mx_mul<V>(x, tw, cx);
    mx_dft<V>(x, m, cx);
    if constexpr (J > 0) {
        MxMap<P::words(J), V>::store(lds, x);
        if constexpr (first) m = mx_load_mat(cx, kMxInv);
        mx_load_tw<P::logs(J - 1), LOGC, V>(tw, cx.ti);
        mx_sync<P::words(J - 1), V>();
        MxMap<P::words(J - 1), V>::load(lds, x);
        mx_inverse<LOGL, LOGC, V, J - 1>(x, lds, cx, m, tw);
    }
}

// Whole multiply of tiles whose round-0 words are in x[0] (F) and x[1] (G),
// m and tw from mx_forward_begin; the product's round-0 words (below
// p + 4200) are left in x[0].
template <int LOGL, int V>
CM_DEV void mx_tile_multiply(u32 (&x)[2][V][4], u32 *A, u32 *B, const MxCtx &cx, MxMat &m,
                             u32 (&tw)[V][4]) {
    using P = MxPlan<LOGL, 0, V>;
    if constexpr (V >= 4) {
        // one operand after the other: both at once would exceed 128
        // registers.  The words that wait are in LDS where this thread put
        // them, so no barrier is needed to take them back.
        u32 *const ta[1] = {A}, *const tb[1] = {B};
        MxMap<P::words(0), V>::store(B, x[1]);
        mx_fence<V>();
        mx_forward<LOGL, 0, V, 0, 1>(reinterpret_cast<u32 (&)[1][V][4]>(x[0]), ta, cx, m, tw);
        MxMap<P::words(P::NR - 1), V>::store(A, x[0]);
        mx_forward_begin<LOGL, 0, V>(m, tw, cx);
        MxMap<P::words(0), V>::load(B, x[1]);
        mx_forward<LOGL, 0, V, 0, 1>(reinterpret_cast<u32 (&)[1][V][4]>(x[1]), tb, cx, m, tw);
        MxMap<P::words(P::NR - 1), V>::load(A, x[0]);
    } else {
        u32 *const ab[2] = {A, B};
        mx_forward<LOGL, 0, V, 0, 2>(x, ab, cx, m, tw);
    }
    // the pointwise product leaves 2^-32, which the first inverse matrix undoes
    m = mx_load_mat(cx, P::PAIR ? kMxInvPair : kMxInvFirst + P::T);
    u32 w[4];
    if constexpr (P::PAIR) mx_pair_tw(w, cx.ti);
    mx_mul<V>(x[0], x[1], cx);
    if constexpr (P::PAIR) mx_pair_inv<V>(x[0], w, cx);
    mx_inverse<LOGL, 0, V, P::NR - 1>(x[0], A, cx, m, tw);
}

// Frequency held by position r of a forward transform of 2^logl points: the
// first digit (the top four bits of r) is the lowest of the frequency.
CM_DEV int mx_freq(int r, int logl) {
    int k = 0, shift = 0;
    for (; logl >= 4; logl -= 4, shift += 4) k |= ((r >> (logl - 4)) & 15) << shift;
    return k | ((r & ((1 << logl) - 1)) << shift);
}

// Position that holds frequency f (inverse of mx_freq).
CM_DEV int mx_pos(int f, int logl) {
    int r = 0;
    for (; logl >= 4; logl -= 4, f >>= 4) r |= (f & 15) << (logl - 4);
    return r | f;
}

// four consecutive words at a 4-byte aligned address
struct __attribute__((packed, aligned(4))) MxQuad {
    u32 v[4];
};

// Round-0 words of one row set from global memory: word (s, r) of a lane is
// element idx of the row that row(s) names; idx at or beyond its length reads
// as zero.  ROWS(s) -> {const u32 *base, int len}.
template <int LOGL, int V, class RowFn>
CM_DEV void mx_load_rows(u32 (&x)[V][4], RowFn &&row) {
    constexpr int LOGS = MxPlan<LOGL>::words(0);
    using Map = MxMap<LOGS, V>;
    const int i0 = Map::base() & ((1 << LOGL) - 1);
    if constexpr (LOGS >= 2 && V == 4) {
        const u32 *q;
        int len;
        row(0, q, len);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i0 + (r << LOGS);
            if (i + 4 <= len) {
                const MxQuad v = *(const MxQuad *)(q + i);
#pragma unroll
                for (int s = 0; s < 4; ++s) x[s][r] = v.v[s];
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s) x[s][r] = i + s < len ? q[i + s] : 0u;
            }
        }
    } else {
#pragma unroll
        for (int s = 0; s < V; ++s) {
            const u32 *q;
            int len;
            row(s, q, len);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = i0 + (Map::off(s, r) & ((1 << LOGL) - 1));
                x[s][r] = i < len ? q[i] : 0u;
            }
        }
    }
}

// the same for canonical stores; FROM: words below `from` are not stored
template <int LOGL, int V, bool FROM = false, class RowFn>
CM_DEV void mx_store_rows(const u32 (&x)[V][4], RowFn &&row, const MxCtx &cx, int from = 0) {
    constexpr int LOGS = MxPlan<LOGL>::words(0);
    using Map = MxMap<LOGS, V>;
    const int i0 = Map::base() & ((1 << LOGL) - 1);
    if constexpr (LOGS >= 2 && V == 4) {
        u32 *q;
        int len;
        row(0, q, len);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i0 + (r << LOGS);
            MxQuad v;
#pragma unroll
            for (int s = 0; s < 4; ++s) v.v[s] = mx_canon(x[s][r], cx);
            if (i + 4 <= len && (!FROM || i >= from)) {
                *(MxQuad *)(q + i) = v;
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    if (i + s < len && (!FROM || i + s >= from)) q[i + s] = v.v[s];
            }
        }
    } else {
#pragma unroll
        for (int s = 0; s < V; ++s) {
            u32 *q;
            int len;
            row(s, q, len);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = i0 + (Map::off(s, r) & ((1 << LOGL) - 1));
                if (i < len && (!FROM || i >= from)) q[i] = mx_canon(x[s][r], cx);
            }
        }
    }
}

}  // namespace cm
