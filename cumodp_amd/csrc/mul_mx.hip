// mul_mx.hip -- multiplies on the matrix cores: whole products of up to 2^13 points
// in one workgroup, and the column and row passes of the four-step ones above.
#include <algorithm>

#include "internal.h"
#include "mul_mx.h"
#include "ntt_core.h"

namespace cm {

enum : int { kStrided = 0, kDesc = 1, kMonic = 2, kMiddle = 3 };

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
// words) and writes H + d * one.h (one.lh words); kMonic: the same with monic
// operands of 2^LOGL / 2 + 1 words, whose product's leading term wraps onto word
// 0 and is put into word 2^LOGL; kMiddle: product d of G array d >> 1 goes to
// output d ^ 1, from word one.logn on.  H may alias F or G: a
// product's words are all loaded before any of its words is stored, by the
// same wave or on the other side of a barrier.
template <int LOGL, int LOGW, int V, int DESC>
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
            if (DESC == kDesc) {
                m = descs ? descs[d] : one;
            } else {
                m = one;
                m.f = (int64_t)d * one.f;
                m.g = (int64_t)(DESC == kMiddle ? d >> 1 : d) * one.g;
                m.h = (int64_t)(DESC == kMiddle ? d ^ 1 : d) * one.h;
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
    if constexpr (DESC == kMonic) {
        // word 0 of a row: set s, r = 0 of the lane that holds its start
#pragma unroll
        for (int s = 0; s < V; ++s)
            if (((Map::base() + Map::off(s, 0)) & ((1 << LOGL) - 1)) == 0)
                x[0][s][0] = cm_sub(mx_canon(x[0][s][0], cx), 1u, cx.p);
    }
    mx_store_rows<LOGL, V, DESC == kMiddle>(
        x[0],
        [&](int s, u32 *&q, int &len) {
            const MulDesc m = desc(s);
            q = H + m.h;
            len = std::min(m.lh, 1 << LOGL);
        },
        cx, one.logn);
    if (DESC == kMiddle) return;
    // words beyond the transform size (lh > L) are zero, or the leading 1
    for (int c = 0; c < C; ++c) {
        const int d = blockIdx.x * C + c;
        if (d >= ndesc) break;
        const MulDesc m = DESC == kDesc && descs ? descs[d] : one;
        const int64_t h = DESC == kDesc ? m.h : (int64_t)d * one.h;
        for (int i = (1 << LOGL) + threadIdx.x; i < m.lh; i += blockDim.x)
            H[h + i] = DESC == kMonic ? 1u : 0u;
    }
}

// Below 2^19 words in all, four sets per lane would leave the 1024 SIMDs fewer
// than one wave for every two; products then spread over four times the
// threads (one set per lane; two for 2^13 points, whose 2048 threads would not
// fit a workgroup).
constexpr int64_t kMxSpreadWords = (int64_t)1 << 19;

template <int LOGL, int V, int DESC>
static hipError_t mul_mx_v(const u32 *F, const u32 *G, u32 *H, const MulDesc *descs, int ndesc,
                           const MulDesc &one, const Family *fam, hipStream_t s) {
    constexpr int LOGW = std::max(LOGL, 8 + mx_log2(V));
    constexpr int C = 1 << (LOGW - LOGL);
    ProfScope ps(kProfMulLds, s);
    hipLaunchKernelGGL((k_mul_mx<LOGL, LOGW, V, DESC>), dim3((ndesc + C - 1) / C),
                       dim3((1 << LOGW) / (4 * V)), 0, s, F, G, H, descs, ndesc, one, mx_ctx(fam));
    return hipGetLastError();
}

template <int LOGL, int DESC>
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
#define CM_CASE(K) case K: return mul_mx_t<K, kDesc>(F, G, H, d_descs, ndesc, one, fam, s);
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
#define CM_CASE(K) case K: return mul_mx_t<K, kStrided>(F, G, H, nullptr, count, sd, fam, s);
        CM_CASE(4) CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8) CM_CASE(9) CM_CASE(10)
        CM_CASE(11) CM_CASE(12) CM_CASE(13)
#undef CM_CASE
    }
    return hipErrorInvalidValue;
}

// 2 to 32 products of 2^13 points leave most of the chip idle as one workgroup
// each (15 us): as four-step multiplies on 2^5 x 2^8 words they take three
// launches of 3.5 us.  Trees of 2^14, 2^16 and 2^18 points: 58.7, 81.3 and 122.8
// us with workgroups, 52.2, 76.2 and 119.8 so; at 64 products both take the
// same and at 128 the workgroups win.  A single product, queued from the host,
// waits for three launches instead of one: 12.2 us either way.
static bool four_step_13(int logn, int64_t count) {
    return logn == kMaxLdsLog && count >= 2 && count <= 32;
}

hipError_t launch_tree_level(int i, const u32 *prev, u32 *cur, int64_t nodes, const Family *fam,
                             hipStream_t s) {
    const int64_t h = (int64_t)1 << (i - 1), n = 2 * h;
    if (nodes <= 0 || nodes > INT32_MAX) return hipErrorInvalidValue;
    const MulDesc sd{2 * (h + 1), 2 * (h + 1), n + 1, (int)(h + 1), (int)(h + 1), (int)(n + 1), i};
    switch (four_step_13(i, nodes) ? 0 : i) {
#define CM_CASE(K)                                                                        \
    case K:                                                                               \
        return mul_mx_t<K, kMonic>(prev, prev + (h + 1), cur, nullptr, (int)nodes, sd, fam, s);
        CM_CASE(9) CM_CASE(10) CM_CASE(11) CM_CASE(12) CM_CASE(13)
#undef CM_CASE
    }
    // four-step straight from and into the tree, in chunks whose two slabs
    // stay within 1 GiB each
    const int64_t chunk = std::max<int64_t>(1, ((int64_t)1 << 28) / n);
    for (int64_t c0 = 0; c0 < nodes; c0 += chunk) {
        const int cnt = (int)std::min<int64_t>(chunk, nodes - c0);
        u32 *sf = (u32 *)workspace(5, sizeof(u32) * (size_t)(n * cnt), s);
        u32 *sg = (u32 *)workspace(6, sizeof(u32) * (size_t)(n * cnt), s);
        if (!sf || !sg) return hipErrorOutOfMemory;
        const u32 *f = prev + c0 * 2 * (h + 1);
        FourStepIO io{f, f + (h + 1), h + 1, h + 1, 2 * (h + 1), sf, sg, cur + c0 * (n + 1),
                      n, n + 1, cnt};
        io.monic = 1;
        const hipError_t e = launch_mul_four_step(i, io, fam, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_mul_middle(int logn, const MidProduct &q, const Family *fam, hipStream_t s) {
    const int64_t n = (int64_t)1 << logn;
    if (q.cnt < 1 || q.from < 0 || q.from + q.len > n || (q.cnt > 1 && (q.cnt & 1)))
        return hipErrorInvalidValue;
    u32 *h = q.h - q.from;
    const MulDesc sd{q.fs, q.gs, q.hs, (int)q.lf, (int)q.lg, (int)(q.from + q.len), (int)q.from};
    switch (four_step_13(logn, q.cnt) ? 0 : logn) {
#define CM_CASE(K) \
    case K: return q.neg ? hipErrorInvalidValue \
                         : mul_mx_t<K, kMiddle>(q.f, q.g, h, nullptr, q.cnt, sd, fam, s);
        CM_CASE(9) CM_CASE(10) CM_CASE(11) CM_CASE(12) CM_CASE(13)
#undef CM_CASE
    }
    // four-step, in chunks whose two slabs stay within 1 GiB each
    const int64_t chunk = std::max<int64_t>(2, ((int64_t)1 << 28) / n);
    for (int64_t c0 = 0; c0 < q.cnt; c0 += chunk) {
        const int cnt = (int)std::min<int64_t>(chunk, q.cnt - c0), pairs = cnt > 1;
        u32 *sf = (u32 *)workspace(5, sizeof(u32) * (size_t)(n * cnt), s);
        u32 *sg = (u32 *)workspace(6, sizeof(u32) * (size_t)(n * (cnt >> pairs)), s);
        if (!sf || !sg) return hipErrorOutOfMemory;
        FourStepIO io{q.f + c0 * q.fs, q.g + (c0 >> 1) * q.gs, q.lf, q.lg, q.fs, sf, sg,
                      h + c0 * q.hs, q.from + q.len, q.hs, cnt};
        io.g_stride = q.gs;
        io.g_shift = io.out_xor = pairs;
        io.out_from = (int)q.from;
        io.neg = q.neg;
        const hipError_t e = launch_mul_four_step(logn, io, fam, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// ---------------------------------------------------------------------------
// four-step multiply: an n-word array viewed as 2^k1 rows x 2^k2 columns
// ---------------------------------------------------------------------------
// One set of arrays of the column passes: array a reads in[a in_stride + e]
// for e < in_len (zero beyond) and writes out[(a ^ out_xor) out_stride + e] for
// out_from <= e < out_len.  monic: the product of two monic polynomials of
// half the length, whose x^n wrapped onto word 0: that word less one, and a
// leading 1 in word n.  neg: outputs negated.
struct MxCols {
    const u32 *in;
    u32 *out;
    int64_t in_stride, in_len, out_stride, out_len;
    int out_from = 0, out_xor = 0, monic = 0, neg = 0;
};

// Forward column transforms of 2^LOGC columns per workgroup (mx_col_fwd).
// grid.y: arrays, the first cnt0 from set s0, the rest from s1.
template <int LOGL, int LOGC, int V>
__global__ __launch_bounds__((1 << (LOGL + LOGC)) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_col_fwd_mx(MxCols s0, MxCols s1, int cnt0,
                                                             int logn2, MxCtx cx) {
    __shared__ __align__(16) u32 lds[mx_col_lds<LOGL, LOGC>()];
    const int y = blockIdx.y;
    const MxCols &S = y < cnt0 ? s0 : s1;
    const int64_t a = y < cnt0 ? y : y - cnt0;
    const int c0 = mx_xcd(blockIdx.x, gridDim.x) << LOGC;
    mx_col_fwd<LOGL, LOGC, V>(lds, S.in + a * S.in_stride + c0, (int)(S.in_len - c0),
                              S.out + a * S.out_stride + c0, logn2, cx);
}

// Inverse column transforms (mx_col_inv), truncated to out_len.  EDGES: sets
// with out_from, out_xor, monic or neg.
template <int LOGL, int LOGC, int V, bool EDGES>
__global__ __launch_bounds__((1 << (LOGL + LOGC)) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_col_inv_mx(MxCols S, int logn2, MxCtx cx) {
    __shared__ __align__(16) u32 lds[mx_col_lds<LOGL, LOGC>()];
    const int64_t a = blockIdx.y;
    const int c0 = mx_xcd(blockIdx.x, gridDim.x) << LOGC;
    u32 *Y = S.out + (EDGES ? a ^ S.out_xor : a) * S.out_stride + c0;
    mx_col_inv<LOGL, LOGC, V, EDGES>(lds, S.in + a * S.in_stride + c0, Y, S.out_from - c0,
                                     (int)(S.out_len - c0), S.monic ? -c0 : INT32_MIN, S.neg, logn2, cx);
    if (EDGES && S.monic && c0 == 0 && threadIdx.x == 0)
        Y[(int64_t)1 << (LOGL + logn2)] = 1u;
}

// Both passes for arrays of many tiles: one workgroup per CU takes every
// gridDim.x-th tile, in two LDS buffers, so a tile costs one barrier (a wave that
// stores tile t + 2 has passed tile t + 1's barrier, which every wave reaches
// after its loads of tile t).
template <int LOGL, int LOGC, bool INV>
__global__ __launch_bounds__((1 << (LOGL + LOGC)) / 16) __attribute__((amdgpu_waves_per_eu(4, 4)))
void k_cols_loop(MxCols s0, MxCols s1, int cnt0, int ntiles, int logn2, MxCtx cx) {
    using K = MxCols4<LOGL, LOGC>;
    __shared__ __align__(16) u32 lds[2][mx_col_lds<LOGL, LOGC>()], mats[K::kMats];
    const int lx = logn2 - LOGC;    // log2 of the tiles of an array
    K k;
    k.begin(INV, mats, cx);
    u32 x[4][4], next[4][4];
    auto load = [&](u32 (&y)[4][4], int t) {
        const int a0 = t >> lx, c0 = (t & ((1 << lx) - 1)) << LOGC;
        const MxCols &S = a0 < cnt0 ? s0 : s1;
        const int64_t a = a0 < cnt0 ? a0 : a0 - cnt0;
        const u32 *X = S.in + a * S.in_stride + c0;
        if constexpr (INV) K::load_rev(y, X, logn2);
        else K::load_nat(y, X, S.in + a * S.in_stride, (int)(S.in_len - c0), logn2);
    };
    int t = mx_xcd(blockIdx.x, gridDim.x);
    if (t < ntiles) load(next, t);
    for (int b = 0; t < ntiles; t += gridDim.x, b ^= 1) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) x[s][r] = next[s][r];
        if (t + (int)gridDim.x < ntiles) load(next, t + gridDim.x);
        mx_fence<4>();
        const int a0 = t >> lx, c0 = (t & ((1 << lx) - 1)) << LOGC;
        const MxCols &S = a0 < cnt0 ? s0 : s1;
        const int64_t a = a0 < cnt0 ? a0 : a0 - cnt0;
        u32 *Y = S.out + a * S.out_stride + c0;
        if constexpr (INV) {
            k.template inverse<K::P::NR - 1>(x, lds[b], cx);
            K::store_nat(x, Y, (int)(S.out_len - c0), logn2, cx);
        } else {
            K::clear_nat(x, (int)(S.in_len - c0), logn2);
            k.template forward<0>(x, lds[b], cx);
            K::store_rev(x, Y, logn2);
        }
    }
}

// Row pass (mx_row) over all rows of the arrays of F, in place.
template <int LOGL, int V>
__global__ __launch_bounds__((1 << mx_row_logw<LOGL, V>()) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_row_mx(u32 *F, const u32 *__restrict__ G, int k1,
                                                         int g_shift, MxOuter o, MxCtx cx) {
    constexpr int LOGW = mx_row_logw<LOGL, V>();
    __shared__ __align__(16) u32 lds[2 * mx_lds_words(1 << LOGW)];
    // array a of F meets array a >> g_shift of G
    const int la = k1 + LOGL - LOGW;   // log2 of the tiles per array
    const int64_t t0 = (int64_t)blockIdx.x << LOGW;
    const int64_t ga = (int64_t)(blockIdx.x >> la) >> g_shift;
    const int64_t tg = ((ga << la) + (blockIdx.x & ((1u << la) - 1))) << LOGW;
    mx_row<LOGL, V>(lds, F + t0, G + tg, (int)(blockIdx.x << (LOGW - LOGL)), k1, o, cx);
}

// Tiles of 16384 words that run as kLoopWgs workgroups, one per CU: two to eight
// tiles for each, the inverse (of one array) two to four, so products of 2^22
// points loop the forward pass only.  Back to back, 2^22, 2^23 and 2^24 points:
// 53.1, 101.1 and 203.1 us on one pair of operands and 51.5, 106.0 and 213.3 on six
// in turn with a workgroup per tile; 50.9, 95.2, 194.1 and 48.9, 97.9, 207.6 us so;
// at 2^25, beyond the last-level cache, 466 us without it and 475 with.
// Operands whose last quad of words is not whole take a workgroup per tile.
constexpr int64_t kLoopMin = 512, kLoopMax = 2048;
constexpr unsigned kLoopWgs = 256;   // CUs of the whole device; any number is correct

template <int LOGL, int LOGC, int V>
static hipError_t cols_t(bool inverse, const MxCols &s0, const MxCols &s1, int cnt0, int cnt1,
                         int k2, const MxCtx &cx, hipStream_t s) {
    constexpr int T = (1 << (LOGL + LOGC)) / (4 * V);
    ProfScope ps(inverse ? kProfColInv : kProfColFwd, s);
    const dim3 g(1u << (k2 - LOGC), cnt0 + cnt1);
    if constexpr (V == 4 && LOGL + LOGC == 14 && LOGL >= 9 && LOGC >= 2) {
        const int64_t tiles = (int64_t)g.x * g.y;
        const bool edges = s0.out_from || s0.out_xor || s0.monic || s0.neg;
        const bool whole = inverse || (s0.in_len % 4 == 0 && s1.in_len % 4 == 0);
        if (tiles >= kLoopMin && tiles <= (inverse ? kLoopMax / 2 : kLoopMax) && !edges && whole) {
            if (inverse)
                hipLaunchKernelGGL((k_cols_loop<LOGL, LOGC, true>), dim3(kLoopWgs), dim3(T), 0, s,
                                   s0, s1, cnt0, (int)tiles, k2, cx);
            else
                hipLaunchKernelGGL((k_cols_loop<LOGL, LOGC, false>), dim3(kLoopWgs), dim3(T), 0, s,
                                   s0, s1, cnt0, (int)tiles, k2, cx);
            return hipGetLastError();
        }
    }
    if (inverse && (s0.out_from || s0.out_xor || s0.monic || s0.neg))
        hipLaunchKernelGGL((k_col_inv_mx<LOGL, LOGC, V, true>), g, dim3(T), 0, s, s0, k2, cx);
    else if (inverse)
        hipLaunchKernelGGL((k_col_inv_mx<LOGL, LOGC, V, false>), g, dim3(T), 0, s, s0, k2, cx);
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
                              int cnt1, int k2, bool small, const MxCtx &cx, hipStream_t s) {
#define CM_COL(LC, V) return cols_t<K, LC, V>(inverse, s0, s1, cnt0, cnt1, k2, cx, s)
#define CM_COLS(KK, LS, VS, LB)                       \
    case KK: {                                        \
        constexpr int K = KK;                         \
        if (small) CM_COL(LS, VS);                    \
        CM_COL(LB, 4);                                \
    }
#define CM_COLB(KK, LB, LS)                           \
    case KK: {                                        \
        constexpr int K = KK;                         \
        if (small) CM_COL(LS, 1);                     \
        if (g_col_words == 8192) CM_COL(LB - 1, 4);   \
        CM_COL(LB, 4);                                \
    }
    switch (k1) {
        CM_COLS(4, 4, 1, 6)
        CM_COLS(5, 4, 1, 5)
        CM_COLS(6, 3, 1, 4)
        CM_COLS(7, 4, 1, 4)
        CM_COLS(8, 3, 1, 4)
        CM_COLB(9, 4, 3)
        CM_COLB(10, 4, 2)
    case 11: {
        constexpr int K = 11;
        if (g_col_words == 8192) CM_COL(2, 4);
        CM_COL(3, 4);
    }
    case 12: {
        constexpr int K = 12;
        if (g_col_words == 8192) CM_COL(1, 2);
        CM_COL(2, 4);
    }
    case 13: {
        constexpr int K = 13;
        CM_COL(1, 4);
    }
    }
#undef CM_COLB
#undef CM_COLS
#undef CM_COL
    return hipErrorInvalidValue;
}

hipError_t launch_cols_out(int k1, const u32 *X, u32 *Y, int64_t n, int cnt, int k2,
                           const MxCtx &cx, hipStream_t s) {
    const MxCols c{X, Y, n, n, n, n};
    return launch_cols(k1, false, c, c, cnt, 0, k2, n * cnt <= kMxSmallWords, cx, s);
}

// Columns of 2, 4 and 8 words, which only named splits have: a thread takes a
// column, as radix-2 butterflies in registers (a radix-16 step would be mostly
// zeros).  A wave's loads and stores are 64 words of a row.  Both directions are
// decimation in frequency with the root's or the inverse root's levels; position
// r holds frequency r.  Input words are any 32 bits.
template <int LOGL, bool INV>
__global__ __launch_bounds__(256) void k_col_short(MxCols s0, MxCols s1, int cnt0, int logn2,
                                                   const u32 *__restrict__ lv, Mod md, u32 r1,
                                                   u32 sc) {
    constexpr int L = 1 << LOGL;
    const int y = blockIdx.y;
    const MxCols &S = y < cnt0 ? s0 : s1;
    const int64_t a = y < cnt0 ? y : y - cnt0;
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const u32 *X = S.in + a * S.in_stride;
    u32 *Y = S.out + (INV ? a ^ S.out_xor : a) * S.out_stride;
    u32 v[1][L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int64_t e = ((int64_t)i << logn2) + c;
        v[0][i] = e < S.in_len ? X[e] : 0u;
    }
#pragma unroll
    for (int i = 0; i < L; ++i) v[0][i] = cm_mul_tw(v[0][i], r1, md.p, md.np);
    cm_dif_stages<LOGL, LOGL, 0, 0, 1>(v, 0, lv, md);
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int64_t e = ((int64_t)i << logn2) + c;
        u32 w = v[0][cm_brev((u32)i, LOGL)];
        if (!INV) {
            Y[e] = w;
            continue;
        }
        w = cm_mul_tw(w, sc, md.p, md.np);
        if (S.monic && e == 0) w = cm_sub(w, 1u, md.p);
        if (S.neg) w = cm_sub(0u, w, md.p);
        if (e >= S.out_from && e < S.out_len) Y[e] = w;
    }
    if (INV && S.monic && c == 0) Y[(int64_t)1 << (LOGL + logn2)] = 1u;
}

template <int LOGL>
static hipError_t cols_short_t(bool inverse, const MxCols &s0, const MxCols &s1, int cnt0,
                               int cnt1, int k2, const Family *fam, hipStream_t s) {
    const Mod md{fam->p, fam->np};
    const dim3 g(1u << (k2 - 8), cnt0 + cnt1);
    const u32 r1 = cm_host_r1(fam->p),
              sc = cm_host_mont(cm_host_inv((1u << LOGL) % fam->p, fam->p), fam->p);
    ProfScope ps(inverse ? kProfColInv : kProfColFwd, s);
    if (inverse)
        hipLaunchKernelGGL((k_col_short<LOGL, true>), g, dim3(256), 0, s, s0, s1, cnt0, k2,
                           fam->lvi, md, r1, sc);
    else
        hipLaunchKernelGGL((k_col_short<LOGL, false>), g, dim3(256), 0, s, s0, s1, cnt0, k2,
                           fam->lv, md, r1, sc);
    return hipGetLastError();
}

// The columns of any split that cumodp_tune_set_split takes.
static hipError_t launch_cols_any(int k1, bool inverse, const MxCols &s0, const MxCols &s1,
                                  int cnt0, int cnt1, int k2, bool small, const Family *fam,
                                  hipStream_t s) {
    switch (k1) {
    case 1: return cols_short_t<1>(inverse, s0, s1, cnt0, cnt1, k2, fam, s);
    case 2: return cols_short_t<2>(inverse, s0, s1, cnt0, cnt1, k2, fam, s);
    case 3: return cols_short_t<3>(inverse, s0, s1, cnt0, cnt1, k2, fam, s);
    }
    return launch_cols(k1, inverse, s0, s1, cnt0, cnt1, k2, small, mx_ctx(fam), s);
}

template <int LOGL, int V>
static hipError_t rows_t(const FourStepIO &io, const Outer *o, const Family *fam, hipStream_t s) {
    constexpr int LOGW = mx_row_logw<LOGL, V>();
    ProfScope ps(kProfRowMul, s);
    const int64_t words = (int64_t)io.cnt << o->k;
    hipLaunchKernelGGL((k_row_mx<LOGL, V>), dim3((unsigned)(words >> LOGW)),
                       dim3((1 << LOGW) / (4 * V)), 0, s, io.f_ws, io.g_ws, o->k1, io.g_shift,
                       mx_outer_of(o), mx_ctx(fam));
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
    if (!o || o->k > fam->K || o->k < kMaxLdsLog) return hipErrorInvalidValue;
    const int64_t n = (int64_t)1 << o->k;
    const MxCols sf{io.f_in, io.f_ws, io.in_stride, io.f_len, n, n};
    const MxCols sg{io.g_in, io.g_ws, io.g_stride < 0 ? io.in_stride : io.g_stride, io.g_len, n, n};
    const bool small = n * io.cnt <= kMxSmallWords;
    hipError_t e =
        launch_cols_any(o->k1, false, sf, sg, io.cnt, io.cnt >> io.g_shift, o->k2, small, fam, s);
    if (e == hipSuccess) e = launch_rows(io, o, fam, s);
    if (e != hipSuccess) return e;
    const MxCols sh{io.f_ws, io.h_out, n, n, io.out_stride, io.h_len,
                    io.out_from, io.out_xor, io.monic, io.neg};
    return launch_cols_any(o->k1, true, sh, sh, io.cnt, 0, o->k2, small, fam, s);
}

hipError_t launch_mul_four_step(int k, const FourStepIO &io, const Family *fam, hipStream_t s) {
    if (k < kMaxLdsLog || k > kMaxLog || k > fam->K) return hipErrorInvalidValue;
    const Outer *o = outer_for(fam, k);
    if (!o) return hipErrorOutOfMemory;
    return launch_mul_four_step_with(io, fam, o, s);
}

}  // namespace cm
