// mul_mx.hip -- whole multiplies in one workgroup on the matrix cores.
#include <algorithm>

#include "internal.h"
#include "ntt_mx.h"

namespace cm {

// A single product is bound by its serial chain (load, rounds, exchanges), many
// products by vector issue.  One 2048-point product mod 469762049, back to
// back: 4.8 us per call with one set per lane (512 threads), 8.1 us with the
// radix-2 butterflies of 16 words per thread that this replaces (128 threads).
//
// A tile of 2^LOGW words holds 2^(LOGW-LOGL) products of 2^LOGL points; the
// F and G tiles are transformed together (shared matrices and twiddles),
// multiplied in registers and the product transformed back (ntt_mx.h).
// DESC: descriptors from `descs` (or the by-value `one` when descs is null);
// otherwise product d reads F + d * one.f, G + d * one.g (one.lf / one.lg
// words) and writes H + d * one.h (one.lh words).  H may alias F or G: a
// product's words are all loaded before any of its words is stored, by the
// same wave or on the other side of a barrier.
template <int LOGL, int LOGW, int V, bool DESC>
__global__ __launch_bounds__((1 << LOGW) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_mul_mx(
    const u32 *F, const u32 *G, u32 *H, const MulDesc *__restrict__ descs, int ndesc, MulDesc one,
    MxCtx cx) {
    static_assert(LOGW >= LOGL && (1 << LOGW) >= 256 * V, "tile");
    constexpr int W = 1 << LOGW, LW = mx_lds_words(W), C = 1 << (LOGW - LOGL);
    __shared__ __align__(16) u32 lds[2 * LW];
    using Map = MxMap<MxPlan<LOGL>::words(0), V>;
    // product of word (s, .) of this lane
    const int row0 = Map::base() >> LOGL;
    auto desc = [&](int s) {
        const int d = blockIdx.x * C + row0 + (Map::off(s, 0) >> LOGL);
        MulDesc m{};
        if (d < ndesc) {
            if (DESC) {
                m = descs ? descs[d] : one;
            } else {
                m = one;
                m.f = (int64_t)d * one.f; m.g = (int64_t)d * one.g; m.h = (int64_t)d * one.h;
            }
        }
        return m;
    };
    MxMat m;
    u32 x[2][V][4], tw[V][4];
    mx_forward_begin<LOGL, 0, V>(m, tw, cx);
    mx_load_rows<LOGL, V>(x[0], [&](int s, const u32 *&q, int &len) {
        const MulDesc m = desc(s);
        q = F + m.f;
        len = m.lf;
    });
    mx_load_rows<LOGL, V>(x[1], [&](int s, const u32 *&q, int &len) {
        const MulDesc m = desc(s);
        q = G + m.g;
        len = m.lg;
    });
    mx_tile_multiply<LOGL, V>(x, lds, lds + LW, cx, m, tw);
    mx_store_rows<LOGL, V>(
        x[0],
        [&](int s, u32 *&q, int &len) {
            const MulDesc m = desc(s);
            q = H + m.h;
            len = std::min(m.lh, 1 << LOGL);
        },
        cx);
    // words beyond the transform size (lh > L) are zero
    for (int c = 0; c < C; ++c) {
        const int d = blockIdx.x * C + c;
        if (d >= ndesc) break;
        const MulDesc m = DESC && descs ? descs[d] : one;
        const int64_t h = DESC ? m.h : (int64_t)d * one.h;
        for (int i = (1 << LOGL) + threadIdx.x; i < m.lh; i += blockDim.x) H[h + i] = 0u;
    }
}

// Below 2^19 words in all, four sets per lane would leave the 1024 SIMDs fewer
// than one wave for every two; products then spread over four times the
// threads (one set per lane; two for 2^13 points, whose 2048 threads would not
// fit a workgroup).
constexpr int64_t kMxSpreadWords = (int64_t)1 << 19;

template <int LOGL, int V, bool DESC>
static hipError_t mul_mx_v(const u32 *F, const u32 *G, u32 *H, const MulDesc *descs, int ndesc,
                           const MulDesc &one, const Family *fam, hipStream_t s) {
    constexpr int LOGW = std::max(LOGL, 8 + mx_log2(V));
    constexpr int C = 1 << (LOGW - LOGL);
    ProfScope ps(kProfMulLds, s);
    hipLaunchKernelGGL((k_mul_mx<LOGL, LOGW, V, DESC>), dim3((ndesc + C - 1) / C),
                       dim3((1 << LOGW) / (4 * V)), 0, s, F, G, H, descs, ndesc, one, mx_ctx(fam));
    return hipGetLastError();
}

template <int LOGL, bool DESC>
static hipError_t mul_mx_t(const u32 *F, const u32 *G, u32 *H, const MulDesc *descs, int ndesc,
                           const MulDesc &one, const Family *fam, hipStream_t s) {
    const int64_t words = (int64_t)ndesc << LOGL;
    if constexpr (LOGL <= 12) {
        if (words < kMxSpreadWords)
            return mul_mx_v<LOGL, 1, DESC>(F, G, H, descs, ndesc, one, fam, s);
    } else if constexpr (LOGL == 13) {
        if (words < kMxSpreadWords)
            return mul_mx_v<LOGL, 2, DESC>(F, G, H, descs, ndesc, one, fam, s);
    }
    return mul_mx_v<LOGL, 4, DESC>(F, G, H, descs, ndesc, one, fam, s);
}

hipError_t launch_mul_lds_one(int logn, const u32 *F, const u32 *G, u32 *H,
                              const MulDesc *d_descs, int ndesc, const MulDesc &one,
                              const Family *fam, hipStream_t s) {
    if (ndesc <= 0) return hipSuccess;
    switch (logn) {
#define CM_CASE(K) case K: return mul_mx_t<K, true>(F, G, H, d_descs, ndesc, one, fam, s);
        CM_CASE(4) CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8) CM_CASE(9) CM_CASE(10)
        CM_CASE(11) CM_CASE(12) CM_CASE(13) CM_CASE(14)
#undef CM_CASE
    }
    return hipErrorInvalidValue;
}

hipError_t launch_mul_lds(int logn, const u32 *F, const u32 *G, u32 *H, const MulDesc *d_descs,
                          int ndesc, const Family *fam, hipStream_t s) {
    return launch_mul_lds_one(logn, F, G, H, d_descs, ndesc, MulDesc{}, fam, s);
}

hipError_t launch_mul_lds_strided(int logn, const u32 *F, const u32 *G, u32 *H, const MulDesc &sd,
                                  int count, const Family *fam, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    switch (logn) {
#define CM_CASE(K) case K: return mul_mx_t<K, false>(F, G, H, nullptr, count, sd, fam, s);
        CM_CASE(4) CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8) CM_CASE(9) CM_CASE(10)
        CM_CASE(11) CM_CASE(12) CM_CASE(13)
#undef CM_CASE
    }
    return hipErrorInvalidValue;
}


// ---------------------------------------------------------------------------
// four-step multiply: an n-word array viewed as 2^k1 rows x 2^k2 columns
// ---------------------------------------------------------------------------
// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous range of logical blocks so that neighbouring column tiles (which
// share 128-byte lines) meet in the same L2.
CM_DEV int mx_xcd(int b, int nb) { return nb & 7 ? b : (b & 7) * (nb >> 3) + (b >> 3); }

// One set of arrays of the column passes: array a reads in[a in_stride + e]
// for e < in_len (zero beyond) and writes out[a out_stride + e], e < out_len.
struct MxCols {
    const u32 *in;
    u32 *out;
    int64_t in_stride, in_len, out_stride, out_len;
};

// The forward pass of 2^24 points (2^11 rows, 8 columns per tile) takes 82 us
// and the inverse 39 us, where the same addresses copied without a transform
// take 36 and 26 us: one workgroup of 16 waves fits a CU (86 registers), so a
// tile's loads, rounds and stores follow each other.  16 columns of 2^10 rows
// (64-byte segments) take 71 and 34 us but leave rows of 2^14.
//
// Forward column transforms of 2^LOGC columns per workgroup: rows straight
// from global memory into the first round, the last round's rows straight
// back (digit-reversed rows, words below p + 4200).  grid.y: arrays, the
// first cnt0 from set s0, the rest from s1.
template <int LOGL, int LOGC, int V>
__global__ __launch_bounds__((1 << (LOGL + LOGC)) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_col_fwd_mx(MxCols s0, MxCols s1, int cnt0,
                                                             int logn2, MxCtx cx) {
    static_assert((1 << LOGC) >= V && LOGL >= 4 && (1 << (LOGL + LOGC)) >= 256 * V,
                  "a wave's 256 V words lie inside the tile");
    using P = MxPlan<LOGL, LOGC>;
    constexpr int W = 1 << (LOGL + LOGC), C = 1 << LOGC;
    __shared__ __align__(16) u32 lds[P::NR > 1 ? mx_lds_words(W) : 4];
    const int y = blockIdx.y;
    const MxCols &S = y < cnt0 ? s0 : s1;
    const int64_t a = y < cnt0 ? y : y - cnt0;
    const int c0 = mx_xcd(blockIdx.x, gridDim.x) * C;
    const u32 *X = S.in + a * S.in_stride + c0;
    u32 *Y = S.out + a * S.out_stride + c0;
    MxMat m;
    u32 x[1][V][4], tw[V][4];
    mx_forward_begin<LOGL, LOGC, V>(m, tw, cx);
    {
        using Map = MxMap<P::words(0), V>;
        const int b = Map::base();
        const int lim = (int)(S.in_len - c0);
        const u32 off = ((u32)(b >> LOGC) << logn2) + (b & (C - 1));
        const u32 row = 1u << (logn2 + P::logs(0));   // words between the elements of a digit
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = (int)(off + r * row);
            if (e + V <= lim) {
                const u32 *q = X + e;
                if constexpr (V >= 4) {
#pragma unroll
                    for (int s = 0; s < V; s += 4) {
                        const MxQuad v = *(const MxQuad *)(q + s);
#pragma unroll
                        for (int j = 0; j < 4; ++j) x[0][s + j][r] = v.v[j];
                    }
                } else {
#pragma unroll
                    for (int s = 0; s < V; ++s) x[0][s][r] = q[s];
                }
            } else {
#pragma unroll
                for (int s = 0; s < V; ++s) x[0][s][r] = e + s < lim ? X[e + s] : 0u;
            }
        }
    }
    u32 *const t[1] = {lds};
    mx_forward<LOGL, LOGC, V, 0, 1>(x, t, cx, m, tw);
    {
        using Map = MxMap<LOGC, V>;
        const int b = Map::base();
        u32 *q = Y + (((u32)(b >> LOGC) << logn2) + (b & (C - 1)));
#pragma unroll
        for (int r = 0; r < 4; ++r, q += (size_t)1 << logn2) {
            if constexpr (V >= 4) {
#pragma unroll
                for (int s = 0; s < V; s += 4)
                    *(uint4 *)(q + s) =
                        make_uint4(x[0][s][r], x[0][s + 1][r], x[0][s + 2][r], x[0][s + 3][r]);
            } else {
#pragma unroll
                for (int s = 0; s < V; ++s) q[s] = x[0][s][r];
            }
        }
    }
}

// Inverse column transforms, the mirror: digit-reversed rows in, natural rows
// out (canonical, truncated to out_len).
template <int LOGL, int LOGC, int V>
__global__ __launch_bounds__((1 << (LOGL + LOGC)) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_col_inv_mx(MxCols S, int logn2, MxCtx cx) {
    static_assert((1 << LOGC) >= V && LOGL >= 4 && (1 << (LOGL + LOGC)) >= 256 * V,
                  "a wave's 256 V words lie inside the tile");
    using P = MxPlan<LOGL, LOGC>;
    constexpr int W = 1 << (LOGL + LOGC), C = 1 << LOGC;
    __shared__ __align__(16) u32 lds[P::NR > 1 ? mx_lds_words(W) : 4];
    const int64_t a = blockIdx.y;
    const int c0 = mx_xcd(blockIdx.x, gridDim.x) * C;
    const u32 *X = S.in + a * S.in_stride + c0;
    u32 *Y = S.out + a * S.out_stride + c0;
    u32 x[V][4], tw[V][4];
    MxMat m = mx_load_mat(cx, kMxInv + P::T);
    {
        using Map = MxMap<LOGC, V>;
        const int b = Map::base();
        const u32 *q = X + (((u32)(b >> LOGC) << logn2) + (b & (C - 1)));
#pragma unroll
        for (int r = 0; r < 4; ++r, q += (size_t)1 << logn2) {
            if constexpr (V >= 4) {
#pragma unroll
                for (int s = 0; s < V; s += 4) {
                    const uint4 v = *(const uint4 *)(q + s);
                    x[s][r] = v.x; x[s + 1][r] = v.y; x[s + 2][r] = v.z; x[s + 3][r] = v.w;
                }
            } else {
#pragma unroll
                for (int s = 0; s < V; ++s) x[s][r] = q[s];
            }
        }
    }
    mx_inverse<LOGL, LOGC, V, P::NR - 1>(x, lds, cx, m, tw);
    {
        using Map = MxMap<P::words(0), V>;
        const int b = Map::base();
        const int lim = (int)(S.out_len - c0);
        const u32 off = ((u32)(b >> LOGC) << logn2) + (b & (C - 1));
        const u32 row = 1u << (logn2 + P::logs(0));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = (int)(off + r * row);
#pragma unroll
            for (int s = 0; s < V; ++s) x[s][r] = mx_canon(x[s][r], cx);
            if (V >= 4 && e + V <= lim) {
#pragma unroll
                for (int s = 0; s + 3 < V; s += 4)
                    *(MxQuad *)(Y + e + s) =
                        MxQuad{{x[s][r], x[s + 1][r], x[s + 2][r], x[s + 3][r]}};
            } else {
#pragma unroll
                for (int s = 0; s < V; ++s)
                    if (e + s < lim) Y[e + s] = x[s][r];
            }
        }
    }
}

// Bound by vector issue: 2.1 G of its 2.3 G lane instructions of 2^24 points
// are transforms and twiddles; 2^11 rows of 2^13 points take 87 us at four
// sets per lane (operands one after the other, 116 registers, no spills),
// 100 us at two, 121 us with both operands in registers at four (168 bytes of
// scratch), and 115 us as radix-2 butterflies.
// Row pass: row r (array r >> k1, position r mod 2^k1 holding frequency
// f = mx_freq(r mod 2^k1)) of F and G times the outer twiddles w_n^(f i) =
// rb[f T + v] rc[16 f + d] (i = d T + v, T = 2^LOGL / 16), the multiply in
// LDS, and the inverse outer twiddles on the way out.  In place on F.
template <int LOGL, int V>
constexpr int mx_row_logw() { return LOGL > 8 + mx_log2(V) ? LOGL : 8 + mx_log2(V); }

template <int LOGL, int V>
CM_DEV void mx_outer(u32 (&tw)[V][4], const u32 *rb, const u32 *rc, int f, const MxCtx &cx) {
    constexpr int LT = LOGL - 4;
    using Map = MxMap<LT, V>;
    const int i = Map::base() & ((1 << LOGL) - 1), v = i & ((1 << LT) - 1), d = i >> LT;
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

template <int LOGL, int V>
__global__ __launch_bounds__((1 << mx_row_logw<LOGL, V>()) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_row_mx(u32 *F, const u32 *__restrict__ G, int k1,
                                                         const u32 *__restrict__ rb,
                                                         const u32 *__restrict__ rc,
                                                         const u32 *__restrict__ rbi,
                                                         const u32 *__restrict__ rci, MxCtx cx) {
    static_assert(LOGL - 4 >= mx_log2(V), "row");
    constexpr int LOGW = mx_row_logw<LOGL, V>(), W = 1 << LOGW, LW = mx_lds_words(W);
    __shared__ __align__(16) u32 lds[2 * LW];
    using Map = MxMap<LOGL - 4, V>;
    const int b = Map::base();
    const int64_t t0 = (int64_t)blockIdx.x << LOGW;
    u32 *Fr = F + t0 + b;
    const u32 *Gr = G + t0 + b;
    const int row = (int)(blockIdx.x << (LOGW - LOGL)) + (b >> LOGL);
    const int f = mx_freq(row & ((1 << k1) - 1), k1);
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
    mx_outer<LOGL, V>(ow, rb, rc, f, cx);
    mx_mul<V>(x[0], ow, cx);
    mx_mul<V>(x[1], ow, cx);
    mx_forward_begin<LOGL, 0, V>(m, tw, cx);
    mx_tile_multiply<LOGL, V>(x, lds, lds + LW, cx, m, tw);
    mx_outer<LOGL, V>(ow, rbi, rci, f, cx);
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

template <int LOGL, int LOGC, int V>
static hipError_t cols_t(bool inverse, const MxCols &s0, const MxCols &s1, int cnt0, int cnt1,
                         int k2, const MxCtx &cx, hipStream_t s) {
    constexpr int T = (1 << (LOGL + LOGC)) / (4 * V);
    ProfScope ps(inverse ? kProfColInv : kProfColFwd, s);
    const dim3 g(1u << (k2 - LOGC), cnt0 + cnt1);
    if (inverse)
        hipLaunchKernelGGL((k_col_inv_mx<LOGL, LOGC, V>), g, dim3(T), 0, s, s0, k2, cx);
    else
        hipLaunchKernelGGL((k_col_fwd_mx<LOGL, LOGC, V>), g, dim3(T), 0, s, s0, s1, cnt0, k2, cx);
    return hipGetLastError();
}

// Columns of 2^k1 words.  Up to 2^20 words in all (kMxSmallWords) the pass is
// bound by latency: one set per lane and tiles of 512 to 4096 words keep the
// most SIMDs busy.  Above, four sets per lane share a twiddle, and tiles of 16
// columns make 64-byte row segments as long as the tile fits 16384 words (8
// and 4 columns for 2^11 and 2^12 rows).  Measured over all splits, tiles and
// sets of 2^14 .. 2^24 points; 2^17: 10.8 us per multiply against 20.6 with
// the tiles of 16384 words that all sizes had before, 2^20: 20.7 us.
constexpr int64_t kMxSmallWords = (int64_t)1 << 20;

// Words per column tile of the large passes: 16384, or 8192 (half the columns
// per tile for columns of 2^9 words and more); a tuned choice.
static int g_col_words = 16384;

bool set_col_tile_words(int words) {
    if (words != 8192 && words != 16384) return false;
    g_col_words = words;
    return true;
}

int col_tile_words() { return g_col_words; }

static hipError_t launch_cols(int k1, bool inverse, const MxCols &s0, const MxCols &s1, int cnt0,
                              int cnt1, int k2, bool small, const Family *fam, hipStream_t s) {
    const MxCtx cx = mx_ctx(fam);
#define CM_COL(LC, V) return cols_t<K, LC, V>(inverse, s0, s1, cnt0, cnt1, k2, cx, s)
#define CM_COLS(KK, LS, VS, LB)                       \
    case KK: {                                        \
        constexpr int K = KK;                         \
        if (small) CM_COL(LS, VS);                    \
        CM_COL(LB, 4);                                \
    }
#define CM_COLB(KK, LB)                               \
    case KK: {                                        \
        constexpr int K = KK;                         \
        if (g_col_words == 8192) CM_COL(LB - 1, 4);   \
        CM_COL(LB, 4);                                \
    }
    switch (k1) {
        CM_COLS(4, 4, 1, 6)
        CM_COLS(5, 4, 1, 5)
        CM_COLS(6, 3, 1, 4)
        CM_COLS(7, 4, 1, 4)
        CM_COLS(8, 3, 1, 4)
        CM_COLB(9, 4)
        CM_COLB(10, 4)
        CM_COLB(11, 3)
    case 12: {
        constexpr int K = 12;
        CM_COL(2, 4);
    }
    }
#undef CM_COLB
#undef CM_COLS
#undef CM_COL
    return hipErrorInvalidValue;
}

template <int LOGL, int V>
static hipError_t rows_t(const FourStepIO &io, const Outer *o, const Family *fam, hipStream_t s) {
    constexpr int LOGW = mx_row_logw<LOGL, V>();
    ProfScope ps(kProfRowMul, s);
    const int64_t words = (int64_t)io.cnt << o->k;
    hipLaunchKernelGGL((k_row_mx<LOGL, V>), dim3((unsigned)(words >> LOGW)),
                       dim3((1 << LOGW) / (4 * V)), 0, s, io.f_ws, io.g_ws, o->k1, o->rb_f,
                       o->rc_f, o->rb_i, o->rc_i, mx_ctx(fam));
    return hipGetLastError();
}

// Sets per lane of the row pass: one while the pass is bound by latency, two
// up to 2^22 words, four above (2^14-word rows always: 1024 threads).
static hipError_t launch_rows(const FourStepIO &io, const Outer *o, const Family *fam,
                              hipStream_t s) {
    const int64_t words = (int64_t)io.cnt << o->k;
    const int v = words <= kMxSmallWords ? 1 : (words <= 4 * kMxSmallWords ? 2 : 4);
#define CM_ROWS(K)                                        \
    case K:                                               \
        if (v == 1) return rows_t<K, 1>(io, o, fam, s);   \
        if (v == 2) return rows_t<K, 2>(io, o, fam, s);   \
        return rows_t<K, 4>(io, o, fam, s);
    switch (o->k2) {
        CM_ROWS(8) CM_ROWS(9) CM_ROWS(10) CM_ROWS(11) CM_ROWS(12)
    case 13:
        return v <= 2 ? rows_t<13, 2>(io, o, fam, s) : rows_t<13, 4>(io, o, fam, s);
    case 14:
        return rows_t<14, 4>(io, o, fam, s);
    }
#undef CM_ROWS
    return hipErrorInvalidValue;
}

hipError_t launch_mul_four_step_with(const FourStepIO &io, const Family *fam, const Outer *o,
                                     hipStream_t s) {
    if (!o || o->k > fam->K || o->k <= kMaxLdsLog) return hipErrorInvalidValue;
    const int64_t n = (int64_t)1 << o->k;
    const MxCols sf{io.f_in, io.f_ws, io.in_stride, io.f_len, n, n};
    const MxCols sg{io.g_in, io.g_ws, io.g_stride < 0 ? io.in_stride : io.g_stride, io.g_len, n, n};
    const bool small = n * io.cnt <= kMxSmallWords;
    hipError_t e = launch_cols(o->k1, false, sf, sg, io.cnt, io.cnt, o->k2, small, fam, s);
    if (e == hipSuccess) e = launch_rows(io, o, fam, s);
    if (e != hipSuccess) return e;
    const MxCols sh{io.f_ws, io.h_out, n, n, io.out_stride, io.h_len};
    return launch_cols(o->k1, true, sh, sh, io.cnt, 0, o->k2, small, fam, s);
}

hipError_t launch_mul_four_step(int k, const FourStepIO &io, const Family *fam, hipStream_t s) {
    if (k <= kMaxLdsLog || k > kMaxLog || k > fam->K) return hipErrorInvalidValue;
    const Outer *o = outer_for(fam, k);
    if (!o) return hipErrorOutOfMemory;
    return launch_mul_four_step_with(io, fam, o, s);
}

}  // namespace cm
