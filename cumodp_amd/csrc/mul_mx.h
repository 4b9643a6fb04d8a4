// mul_mx.h -- the passes of the matrix-core four-step multiply (ntt_mx.h) as
// device functions: columns of a 2^k1 x 2^k2 array and its rows.
#pragma once

#include "ntt_mx.h"

namespace cm {

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous range of logical blocks so that neighbouring column tiles (which
// share 128-byte lines) meet in the same L2.
CM_DEV int mx_xcd(int b, int nb) { return nb & 7 ? b : (b & 7) * (nb >> 3) + (b >> 3); }

// Outer twiddle tables of one size (struct Outer of internal.h).
struct MxOuter {
    const u32 *rb_f, *rc_f, *rb_i, *rc_i;
};

static inline MxOuter mx_outer_of(const Outer *o) {
    return MxOuter{o->rb_f, o->rc_f, o->rb_i, o->rc_i};
}

template <int LOGL, int LOGC>
constexpr int mx_col_lds() {
    return MxPlan<LOGL, LOGC>::NR > 1 ? mx_lds_words(1 << (LOGL + LOGC)) : 4;
}

// The forward pass of 2^24 points (2^11 rows, 8 columns per tile) takes 82 us
// and the inverse 39 us, where the same addresses copied without a transform
// take 52 and 40 us: one workgroup of 16 waves fits a CU (86 registers), so a
// tile's loads, rounds and stores follow each other (k_cols_loop of mul_mx.hip
// overlaps them: 74 us).  16 columns of 2^10 rows (64-byte segments) take 71 and
// 34 us but leave rows of 2^14.
//
// Forward transforms of 2^LOGC columns: rows straight from global memory into
// the first round (words at or beyond lim, relative to X, are zero), the last
// round's rows straight to Y (digit-reversed rows, words below p + 4200).
// X and Y point at the tile's first column; rows are 2^logn2 words apart.
template <int LOGL, int LOGC, int V>
CM_DEV void mx_col_fwd(u32 *lds, const u32 *X, int lim, u32 *Y, int logn2, const MxCtx &cx) {
    constexpr int C = 1 << LOGC;
    static_assert((C >= V || (C == 2 && V == 4)) && LOGL >= 4 && (C << LOGL) >= 256 * V,
                  "a wave's 256 V words lie inside the tile");
    using P = MxPlan<LOGL, LOGC>;
    MxMat m;
    u32 x[1][V][4], tw[V][4];
    mx_forward_begin<LOGL, LOGC, V>(m, tw, cx);
    {
        const int b = MxMap<P::words(0), V>::base();
        const u32 off = ((u32)(b >> LOGC) << logn2) + (b & (C - 1));
        const u32 row = 1u << (logn2 + P::logs(0));   // words between the elements of a digit
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = (int)(off + r * row);
            if constexpr (C < V) {
                // two columns of two rows
#pragma unroll
                for (int s = 0; s < V; ++s) {
                    const int i = e + ((s >> LOGC) << logn2) + (s & (C - 1));
                    x[0][s][r] = i < lim ? X[i] : 0u;
                }
                continue;
            }
            if (V == 4 && e + V <= lim) {
                const MxQuad v = *(const MxQuad *)(X + e);
#pragma unroll
                for (int s = 0; s < V; ++s) x[0][s][r] = v.v[s];
            } else {
#pragma unroll
                for (int s = 0; s < V; ++s) x[0][s][r] = e + s < lim ? X[e + s] : 0u;
            }
        }
    }
    u32 *const t[1] = {lds};
    mx_forward<LOGL, LOGC, V, 0, 1>(x, t, cx, m, tw);
    const int b = MxMap<LOGC, V>::base();
    u32 *q = Y + (((u32)(b >> LOGC) << logn2) + (b & (C - 1)));
#pragma unroll
    for (int r = 0; r < 4; ++r, q += (size_t)1 << logn2) {
        if constexpr (C < V) {
            // two columns of rows r and r + 16
            *(uint2 *)q = make_uint2(x[0][0][r], x[0][1][r]);
            *(uint2 *)(q + ((size_t)16 << logn2)) = make_uint2(x[0][2][r], x[0][3][r]);
        } else if constexpr (V == 4) {
            *(uint4 *)q = make_uint4(x[0][0][r], x[0][1][r], x[0][2][r], x[0][3][r]);
        } else {
#pragma unroll
            for (int s = 0; s < V; ++s) q[s] = x[0][s][r];
        }
    }
}

// The mirror: digit-reversed rows in, natural rows out (canonical, words at or
// beyond lim, relative to Y, not stored).  EDGES: words below `from` are not
// stored either, and word `fix` is stored less one (tests that cost the plain
// form 7%); neg negates all.
template <int LOGL, int LOGC, int V, bool EDGES>
CM_DEV void mx_col_inv(u32 *lds, const u32 *X, u32 *Y, int from, int lim, int fix, bool neg,
                       int logn2, const MxCtx &cx) {
    constexpr int C = 1 << LOGC;
    static_assert((C >= V || (C == 2 && V == 4)) && LOGL >= 4 && (C << LOGL) >= 256 * V,
                  "a wave's 256 V words lie inside the tile");
    using P = MxPlan<LOGL, LOGC>;
    u32 x[V][4], tw[V][4];
    MxMat m = mx_load_mat(cx, kMxInv + P::T);
    {
        const int b = MxMap<LOGC, V>::base();
        const u32 *q = X + (((u32)(b >> LOGC) << logn2) + (b & (C - 1)));
#pragma unroll
        for (int r = 0; r < 4; ++r, q += (size_t)1 << logn2) {
            if constexpr (C < V) {
                const uint2 v = *(const uint2 *)q, w = *(const uint2 *)(q + ((size_t)16 << logn2));
                x[0][r] = v.x; x[1][r] = v.y; x[2][r] = w.x; x[3][r] = w.y;
            } else if constexpr (V == 4) {
                const uint4 v = *(const uint4 *)q;
                x[0][r] = v.x; x[1][r] = v.y; x[2][r] = v.z; x[3][r] = v.w;
            } else {
#pragma unroll
                for (int s = 0; s < V; ++s) x[s][r] = q[s];
            }
        }
    }
    mx_inverse<LOGL, LOGC, V, P::NR - 1>(x, lds, cx, m, tw);
    const int b = MxMap<P::words(0), V>::base();
    const u32 off = ((u32)(b >> LOGC) << logn2) + (b & (C - 1));
    const u32 row = 1u << (logn2 + P::logs(0));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int e = (int)(off + r * row);
        auto at = [&](int s) { return C < V ? e + ((s >> LOGC) << logn2) + (s & (C - 1)) : e + s; };
#pragma unroll
        for (int s = 0; s < V; ++s) {
            x[s][r] = mx_canon(x[s][r], cx);
            if (EDGES && at(s) == fix) x[s][r] = cm_sub(x[s][r], 1u, cx.p);
            if (EDGES && neg) x[s][r] = cm_sub(0u, x[s][r], cx.p);
        }
        if constexpr (V == 4 && C >= V) {
            if ((!EDGES || e >= from) && e + V <= lim) {
                *(MxQuad *)(Y + e) = MxQuad{{x[0][r], x[1][r], x[2][r], x[3][r]}};
                continue;
            }
        }
#pragma unroll
        for (int s = 0; s < V; ++s)
            if ((!EDGES || at(s) >= from) && at(s) < lim) Y[at(s)] = x[s][r];
    }
}

// The same passes over many tiles, one workgroup per CU for all of them
// (mul_mx.hip, k_cols_loop): what a tile needs besides its words is loaded
// once, so that the words of the next tile can be in flight during the rounds of
// this one: the twiddles, which the columns of a tile and all tiles share, into
// registers, the two matrices into LDS (both in registers would spill).
template <int LOGL, int LOGC>
struct MxCols4 {
    static constexpr int V = 4, C = 1 << LOGC;
    using P = MxPlan<LOGL, LOGC>;
    static_assert(P::NR >= 2 && P::NR <= 3 && LOGC >= 2, "rounds");
    static constexpr int kMats = 2 * kMxMatWords * 4;   // words of `mats`
    const mx_v4i *mats;     // radix-16, and the last digit's
    u32 tw[P::NR - 1][4];

    CM_DEV void begin(bool inverse, u32 *lds_mats, const MxCtx &cx) {
        mx_v4i *dst = (mx_v4i *)lds_mats;
        const mx_v4i *src = cx.mat + (inverse ? kMxInv : kMxFwd) * kMxMatWords;
        for (int i = threadIdx.x; i < kMxMatWords; i += blockDim.x) {
            dst[i] = src[i];
            dst[kMxMatWords + i] = src[P::T * kMxMatWords + i];
        }
        mats = dst + (threadIdx.x & 63);
        __syncthreads();
        const u32 *tab = inverse ? cx.ti : cx.tf;
        u32 t[V][4];
        mx_load_tw<P::logs(0), LOGC, V>(t, tab);
#pragma unroll
        for (int r = 0; r < 4; ++r) tw[0][r] = t[0][r];
        if constexpr (P::NR == 3) {
            mx_load_tw<P::logs(1), LOGC, V>(t, tab);
#pragma unroll
            for (int r = 0; r < 4; ++r) tw[1][r] = t[0][r];
        }
    }
    CM_DEV MxMat mat(bool last) const {
        const mx_v4i *q = mats + (last && P::T ? kMxMatWords : 0);
        return MxMat{q[0], q[64], q[128], q[192], q[256]};
    }
    CM_DEV static void mul(u32 (&x)[V][4], const u32 (&w)[4], const MxCtx &cx) {
#pragma unroll
        for (int s = 0; s < V; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) x[s][r] = cm_mont_lazy(x[s][r], w[r], cx.p, cx.np);
        mx_fence<V>();
    }
    template <int J>
    CM_DEV void forward(u32 (&x)[V][4], u32 *lds, const MxCtx &cx) const {
        mx_dft<V>(x, mat(J == P::NR - 1), cx);
        if constexpr (J < P::NR - 1) {
            mul(x, tw[J], cx);
            MxMap<P::words(J), V>::store(lds, x);
            mx_sync<P::words(J), V>();
            MxMap<P::words(J + 1), V>::load(lds, x);
            forward<J + 1>(x, lds, cx);
        }
    }
    template <int J>
    CM_DEV void inverse(u32 (&x)[V][4], u32 *lds, const MxCtx &cx) const {
        if constexpr (J < P::NR - 1) mul(x, tw[J], cx);
        mx_dft<V>(x, mat(J == P::NR - 1), cx);
        if constexpr (J > 0) {
            MxMap<P::words(J), V>::store(lds, x);
            mx_sync<P::words(J - 1), V>();
            MxMap<P::words(J - 1), V>::load(lds, x);
            inverse<J - 1>(x, lds, cx);
        }
    }
    // natural rows (round 0's words; at or beyond lim: zero, or not stored).
    // Quads beyond lim (none straddles it) are read at `safe` and cleared by
    // clear_nat when the words are used: a branch here would wait for the
    // loads before it.
    CM_DEV static void load_nat(u32 (&x)[V][4], const u32 *X, const u32 *safe, int lim, int logn2) {
        const int b = MxMap<P::words(0), V>::base();
        const u32 off = ((u32)(b >> LOGC) << logn2) + (b & (C - 1));
        const u32 row = 1u << (logn2 + P::logs(0));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = (int)(off + r * row);
            const MxQuad v = *(const MxQuad *)(e + V <= lim ? X + e : safe);
#pragma unroll
            for (int s = 0; s < V; ++s) x[s][r] = v.v[s];
        }
    }
    CM_DEV static void clear_nat(u32 (&x)[V][4], int lim, int logn2) {
        const int b = MxMap<P::words(0), V>::base();
        const u32 off = ((u32)(b >> LOGC) << logn2) + (b & (C - 1));
        const u32 row = 1u << (logn2 + P::logs(0));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool in = (int)(off + r * row) + V <= lim;
#pragma unroll
            for (int s = 0; s < V; ++s) x[s][r] = in ? x[s][r] : 0u;
        }
    }
    CM_DEV static void store_nat(u32 (&x)[V][4], u32 *Y, int lim, int logn2, const MxCtx &cx) {
        const int b = MxMap<P::words(0), V>::base();
        const u32 off = ((u32)(b >> LOGC) << logn2) + (b & (C - 1));
        const u32 row = 1u << (logn2 + P::logs(0));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = (int)(off + r * row);
            MxQuad v;
#pragma unroll
            for (int s = 0; s < V; ++s) v.v[s] = mx_canon(x[s][r], cx);
            if (e + V <= lim) {
                *(MxQuad *)(Y + e) = v;
            } else {
#pragma unroll
                for (int s = 0; s < V; ++s)
                    if (e + s < lim) Y[e + s] = v.v[s];
            }
        }
    }
    // digit-reversed rows
    CM_DEV static u32 rev_offset(int logn2) {
        const int b = MxMap<LOGC, V>::base();
        return ((u32)(b >> LOGC) << logn2) + (b & (C - 1));
    }
    CM_DEV static void load_rev(u32 (&x)[V][4], const u32 *X, int logn2) {
        const u32 *q = X + rev_offset(logn2);
#pragma unroll
        for (int r = 0; r < 4; ++r, q += (size_t)1 << logn2) {
            const uint4 v = *(const uint4 *)q;
            x[0][r] = v.x; x[1][r] = v.y; x[2][r] = v.z; x[3][r] = v.w;
        }
    }
    CM_DEV static void store_rev(const u32 (&x)[V][4], u32 *Y, int logn2) {
        u32 *q = Y + rev_offset(logn2);
#pragma unroll
        for (int r = 0; r < 4; ++r, q += (size_t)1 << logn2)
            *(uint4 *)q = make_uint4(x[0][r], x[1][r], x[2][r], x[3][r]);
    }
};

// Words of a row tile: at least the 256 V words of a wave.
template <int LOGL, int V>
constexpr int mx_row_logw() { return LOGL > 8 + mx_log2(V) ? LOGL : 8 + mx_log2(V); }

// Outer twiddles of a lane's words in the row of frequency f: w_n^(f i) =
// rb[f T + v] rc[16 f + d], i = d T + v, T = 2^LOGL / 16.
template <int LOGL, int V>
CM_DEV void mx_outer(u32 (&tw)[V][4], const u32 *rb, const u32 *rc, int f, const MxCtx &cx) {
    constexpr int LT = LOGL - 4;
    const int i = MxMap<LT, V>::base() & ((1 << LOGL) - 1), v = i & ((1 << LT) - 1), d = i >> LT;
    const u32 *pb = rb + ((int64_t)f << LT) + v;
    const uint4 c = *(const uint4 *)(rc + 16 * f + d);
    u32 b[V];
    if constexpr (V == 4) {
        const uint4 q = *(const uint4 *)pb;
        b[0] = q.x; b[1] = q.y; b[2] = q.z; b[3] = q.w;
    } else {
#pragma unroll
        for (int s = 0; s < V; ++s) b[s] = pb[s];
    }
    const u32 cc[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
    for (int s = 0; s < V; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) tw[s][r] = cm_mont_lazy(cc[r], b[s], cx.p, cx.np);
}

// Bound by vector issue: transforms and twiddles take 2.1 of its 2.3 G lane
// instructions at 2^24 points; 2^11 rows of 2^13 points take 87 us at four
// sets per lane (operands one after the other, 116 registers, no spills),
// 100 us at two, 121 us with both operands in registers at four (168 bytes of
// scratch), and 115 us as radix-2 butterflies.
//
// One tile of rows of F and G (row0: its first row; the row at position
// r mod 2^k1 holds frequency f = mx_freq(r mod 2^k1)): times the outer
// twiddles, the multiply in LDS, and the inverse outer twiddles on the way
// out.  In place on F.
template <int LOGL, int V>
CM_DEV void mx_row(u32 *lds, u32 *F, const u32 *G, int row0, int k1, const MxOuter &o,
                   const MxCtx &cx) {
    static_assert(LOGL - 4 >= mx_log2(V), "row");
    using Map = MxMap<LOGL - 4, V>;
    const int b = Map::base();
    u32 *Fr = F + b;
    const u32 *Gr = G + b;
    const int f = mx_freq((row0 + (b >> LOGL)) & ((1 << k1) - 1), k1);
    MxMat m;
    u32 x[2][V][4], tw[V][4], ow[V][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if constexpr (V == 4) {
            const uint4 u = *(const uint4 *)(Fr + Map::off(0, r));
            const uint4 w = *(const uint4 *)(Gr + Map::off(0, r));
            x[0][0][r] = u.x; x[0][1][r] = u.y; x[0][2][r] = u.z; x[0][3][r] = u.w;
            x[1][0][r] = w.x; x[1][1][r] = w.y; x[1][2][r] = w.z; x[1][3][r] = w.w;
        } else {
#pragma unroll
            for (int s = 0; s < V; ++s) {
                x[0][s][r] = Fr[Map::off(s, r)];
                x[1][s][r] = Gr[Map::off(s, r)];
            }
        }
    }
    mx_outer<LOGL, V>(ow, o.rb_f, o.rc_f, f, cx);
    mx_mul<V>(x[0], ow, cx);
    mx_mul<V>(x[1], ow, cx);
    mx_forward_begin<LOGL, 0, V>(m, tw, cx);
    mx_tile_multiply<LOGL, V>(x, lds, lds + mx_lds_words(1 << mx_row_logw<LOGL, V>()), cx, m, tw);
    mx_outer<LOGL, V>(ow, o.rb_i, o.rc_i, f, cx);
    mx_mul<V>(x[0], ow, cx);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if constexpr (V == 4) {
            *(uint4 *)(Fr + Map::off(0, r)) =
                make_uint4(x[0][0][r], x[0][1][r], x[0][2][r], x[0][3][r]);
        } else {
#pragma unroll
            for (int s = 0; s < V; ++s) Fr[Map::off(s, r)] = x[0][s][r];
        }
    }
}

// Forward column transforms of cnt arrays of n = 2^(k1+k2) words, X -> Y
// (mul_mx.hip).
hipError_t launch_cols_out(int k1, const u32 *X, u32 *Y, int64_t n, int cnt, int k2,
                           const MxCtx &cx, hipStream_t s);

}  // namespace cm
