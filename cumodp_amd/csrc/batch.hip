// batch.hip -- one call multiplying many pairs of uneven degree mod p.
//
// The reference has no list multiply for uneven degrees: list_stockham_dev
// (src/list_stockham.cu:595-630) transforms m rows of one length, and the
// unbuilt draft src/.list_fft_poly_mul.cu:15-53 multiplies equal-length
// pairs.  Here products are binned by transform size 2^e:
//   * e <= 15, and every schoolbook product: one launch of tasks in LDS
//     (k_list_persistent);
//   * e >= 16: per size, the inputs are gathered into zero-padded slabs,
//     multiplied by the batched four-step kernels and scattered back.
// A tuned choice, the per-class form (g_list_persistent = false), takes instead
//   * 2^e <= W (W = 2048, 4096 or 8192 words, a tuned choice): one fused
//     launch for every such product.  Each workgroup takes a W-word tile
//     holding W / 2^e products of one size and runs the whole multiply in
//     LDS; the tile's size selects the code path at run time, so one launch
//     covers all sizes;
//   * 2^e <= 2^13 above W: one launch of the 8192-point workgroup multiply;
//   * e >= 14: as above (many products of 2^14 points in LDS).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "accum.h"
#include "internal.h"
#include "ntt_core.h"
#include "ntt_mx.h"

namespace cm {

struct TileDesc {
    int32_t first;   // first descriptor of the tile
    int32_t count;   // products in the tile (<= 4096 >> logn)
    int32_t logn;
    int32_t pad;
};

// Mixed-size tile variants (words per tile, 16 per thread); the
// tuner picks one per process (cumodp_tune_set_list_tile).  Products of
// 2^logn <= words points go to the mixed kernel, words / 2^logn per tile.
constexpr int kMixVariants = 3;
constexpr int kMixWordsOf[kMixVariants] = {2048, 4096, 8192};
int g_mix_variant = 2;   // 8192 words, 512 threads: measured default (4096 uneven pairs)

struct Scales {
    u32 v[16];
};

template <int LOGL, int W, int T>
using MixTile = Tile<LOGL, (W >> LOGL), false, T>;

template <int LOGL, int W, int T, class MD>
CM_DEV void mul_tile(u32 *A, u32 *B, const u32 *F, const u32 *G, u32 *H, const MulDesc *d,
                     int cnt, const u32 *lv, const u32 *lvi, MD md, u32 sc) {
    using TL = MixTile<LOGL, W, T>;
    constexpr int L = TL::L;
    constexpr int kMixT = T;
    // element idx of the tile: vector c = idx >> LOGL, position i; all loads
    // of a thread are issued before the first LDS store
    constexpr int PER = TL::WORDS / kMixT;
    u32 fa[PER], ga[PER];
    if constexpr (Round<TL, 0>::R == 4 && Round<TL, 0>::GPT == 1 && TL::NR >= 2) {
        // thread t loads its group of the first forward and the last inverse
        // round (product c, elements gi + r 2^(LOGL-4)), which run on the
        // registers
        constexpr int S = LOGL - 4;
        const int c = threadIdx.x >> S, gi = threadIdx.x & ((1 << S) - 1);
        const bool live = c < cnt;
        const MulDesc dc = live ? d[c] : MulDesc{};
#pragma unroll
        for (int r = 0; r < PER; ++r) {
            const int i = gi + (r << S);
            fa[r] = live && i < dc.lf ? F[dc.f + i] : 0u;
            ga[r] = live && i < dc.lg ? G[dc.g + i] : 0u;
        }
        cm_row_multiply<TL>(A, B, fa, ga, lv, lvi, md, sc);
#pragma unroll
        for (int r = 0; r < PER; ++r) {
            const int i = gi + (r << S);
            if (live && i < dc.lh) H[dc.h + i] = cm_canon(fa[r], md);
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = threadIdx.x + r * kMixT, c = idx >> LOGL, i = idx & (L - 1);
        u32 f = 0, g = 0;
        if (c < cnt) {
            if (i < d[c].lf) f = F[d[c].f + i];
            if (i < d[c].lg) g = G[d[c].g + i];
        }
        fa[r] = f;
        ga[r] = g;
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = threadIdx.x + r * kMixT, c = idx >> LOGL, i = idx & (L - 1);
        A[TL::addr(c, i)] = fa[r];
        B[TL::addr(c, i)] = ga[r];
    }
    __syncthreads();
    cm_tile_multiply<TL>(A, B, lv, lvi, md, sc);
    for (int idx = threadIdx.x; idx < TL::WORDS; idx += kMixT) {
        const int c = idx >> LOGL, i = idx & (L - 1);
        if (c < cnt && i < d[c].lh) H[d[c].h + i] = cm_canon(A[TL::addr(c, i)], md);
    }
}

template <int W, int T, class MD>
__global__ __launch_bounds__(T) void k_mul_mixed(
    const u32 *__restrict__ F, const u32 *__restrict__ G, u32 *__restrict__ H,
    const MulDesc *__restrict__ descs, const TileDesc *__restrict__ tiles,
    const u32 *__restrict__ lv, const u32 *__restrict__ lvi, MD md, Scales scales) {
    constexpr int LW = W + (W >> 4);
    __shared__ u32 lds[2 * LW];
    u32 *A = lds, *B = lds + LW;
    const TileDesc t = tiles[blockIdx.x];
    const MulDesc *d = descs + t.first;
    const u32 sc = scales.v[t.logn];
#define CM_MIX(K)                                                                        \
    case K:                                                                              \
        if constexpr ((1 << K) <= W && (W >> K) * (1 << K) / T >= 16)                    \
            mul_tile<K, W, T>(A, B, F, G, H, d, t.count, lv, lvi, md, sc);               \
        break;
    switch (t.logn) {
        CM_MIX(4) CM_MIX(5) CM_MIX(6) CM_MIX(7) CM_MIX(8) CM_MIX(9) CM_MIX(10) CM_MIX(11)
        CM_MIX(12) CM_MIX(13)
    default: break;
    }
#undef CM_MIX
}

// zero-padded copy of operand `which` (0: F, 1: G) of descriptor row y into
// row y of a slab of n-word rows
// Row y of the slab (stride n words) gets the first m words of operand y,
// zero-padded: m is the longest operand of the batch, and the column pass
// reads no further.
__global__ void k_gather(u32 *__restrict__ slab, int64_t n, int64_t m,
                         const u32 *__restrict__ src, const MulDesc *__restrict__ d, int which) {
    const MulDesc dd = d[blockIdx.y];
    const int64_t off = which ? dd.g : dd.f;
    const int len = which ? dd.lg : dd.lf;
    u32 *row = slab + (int64_t)blockIdx.y * n;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m;
         i += (int64_t)gridDim.x * blockDim.x)
        row[i] = i < len ? src[off + i] : 0u;
}

__global__ void k_scatter(u32 *__restrict__ H, const u32 *__restrict__ slab, int64_t n,
                          const MulDesc *__restrict__ d) {
    const MulDesc dd = d[blockIdx.y];
    const u32 *row = slab + (int64_t)blockIdx.y * n;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < dd.lh;
         i += (int64_t)gridDim.x * blockDim.x)
        H[dd.h + i] = row[i];
}

// ---- one launch for the whole list ------------------------------------------
// One launch for every product of a list call up to 2^15 points, schoolbook
// and NTT alike: one workgroup of 512 threads and 68 KiB of LDS per task, so
// that two run on a CU and one's loads and stores go on under the other's
// transforms, or of 1024 threads and 136 KiB (list_log).  Each workgroup takes
// its task from a list in descending order of estimated cost through an atomic
// counter, so the tasks start largest first whatever order the hardware
// dispatches workgroups in (figures for 512 threads, W = 8192 words; twice that
// for 1024):
//   * tile: W words of products of one size 2^logn <= W (W >> logn products),
//     multiplied in LDS;
//   * big: a product of 2^14 or 2^15 points, modulo 2 to 4 factors x^8192 -
//     omega one after the other (omega = 1, -1, i, -i; 3 reach 24576 words), or
//     one of them when whole products would be too long for the chip; then a
//     short kernel recombines them after the launch.  With 1024 threads: one of
//     the two halves of a 2^15-point product, modulo x^16384 - 1 and + 1;
//   * plain: 2048 consecutive outputs of one schoolbook product (8 waves of
//     256 outputs, each wave on its own, the arithmetic of k_plain_mul).
// Bound by issue and the chains inside a wave: 59.9 M vector and 3.8 M matrix
// instructions take 58% and 15% of the SIMDs' cycles with four waves on each,
// and the CUs are busy 83% of the time.  4096 pairs of degrees 32 .. 16384: 187 us per
// call against 226 us with 1024 threads and 16384-word tiles, one workgroup per
// CU, 2^15 points as two halves; a product of up to 12288 words as 8192 + 4096
// points takes 5 us of that.  2^24 points in all of 2^13-point products take 96
// us, of 2^14 117 us (twists and two reads of the operands), of 2^15 142 us in
// four pieces and 100 us in three.
// Largest tasks first keeps the tail short; the counter starts at zero in
// every call's uploaded descriptor blob.  (A loop over tasks in fewer
// workgroups was measured slower: inlined into the loop, the task bodies'
// thread-index arithmetic is hoisted out of it and spills, and called out of
// line they take their uniform pointers in vector registers.)
// All of this on W = 2^LOG words, LOG = 13 or 14 (list_log chooses).
template <int LOG>
struct ListGeo {
    static constexpr int W = 1 << LOG;               // words per product tile
    static constexpr int T = W / 16;                 // threads
    static constexpr int PlainOut = T / 64 * 256;    // outputs of a plain task
    static constexpr int Pieces = LOG == 13 ? 4 : 2; // of the largest product
};
constexpr int kBigLog = 15;                  // largest product of the launch
constexpr int kPlainJT = 512;                // B coefficients per pass of a plain task

enum : uint32_t { kTaskTile = 0, kTaskBig = 1, kTaskPlain = 2 };

// Eight bytes, since a call uploads its tasks and descriptors and an upload
// above 16 KiB takes about 12 us longer: 300 products of 2^13 points take 31.6 us
// so and 45.4 us with tasks of 16 bytes.
struct ListTask {
    int32_t first;   // tile: first descriptor; else the descriptor
    uint32_t what;   // bits 0-1: kind; bits 2-6, sub: tile: transform size; big: kBigAll,
                     // kBigShort, or which piece goes to the scratch; the rest, count: tile:
                     // products; big, all: pieces; plain: outputs before the task, in
                     // PlainOut
};

static ListTask list_task(uint32_t kind, int64_t first, uint32_t sub, int64_t count) {
    return ListTask{(int32_t)first, kind | sub << 2 | (uint32_t)count << 7};
}

constexpr uint32_t kBigAll = 4;     // every piece of a product, one after the other
constexpr uint32_t kBigShort = 5;   // a product of up to 3/2 W words

// Pieces modulo x^W - omega that a product of `words` words needs.
template <int LOG>
CM_HD int big_pieces(int words) { return (words + ListGeo<LOG>::W - 1) >> LOG; }

// x[0] <- (canonical, natural order) the product d modulo x^W - omega, omega =
// 1, -1, i, -i for q = 0 .. 3 (i = w_4): the operands' chunks of W words are
// folded by powers of omega, twisted by psi^j (psi^W = omega: w_2M, w_4M or
// its inverse, M = W; entries of the level tables) and untwisted after the
// cyclic product.
template <int LOG>
CM_DEV void big_piece(int q, u32 (&x)[2][4][4], u32 *lds, const u32 *F, const u32 *G,
                      const MulDesc &d, const u32 *lv, const u32 *lvi, const MxCtx &cx) {
    constexpr int V = 4, M = ListGeo<LOG>::W;
    using Map = MxMap<LOG - 4, V>;
    const int i0 = Map::base();
    const u32 p = cx.p;
    const int lev = q == 1 ? M - 1 : 2 * M - 1;
    const u32 *const tw_f = (q == 3 ? lvi : lv) + lev, *const tw_i = (q == 3 ? lv : lvi) + lev;
    auto operand = [&](u32 (&y)[V][4], const u32 *src, int len) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i0 + Map::off(0, r);
            auto chunk = [&](int c) {
                MxQuad v;
                const int k = c * M + i;
                if (k + 4 <= len) {
                    v = *(const MxQuad *)(src + k);
                } else {
#pragma unroll
                    for (int s = 0; s < 4; ++s) v.v[s] = k + s < len ? src[k + s] : 0u;
                }
                return v;
            };
            MxQuad a = chunk(0), b = chunk(1);
            if (ListGeo<LOG>::Pieces > 2 && len > 2 * M) {
                const MxQuad c = chunk(2), e = chunk(3);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    a.v[s] = cm_add(a.v[s], q < 2 ? c.v[s] : cm_sub(0u, c.v[s], p), p);
                    b.v[s] = cm_add(b.v[s], q < 2 ? e.v[s] : cm_sub(0u, e.v[s], p), p);
                }
            }
            if (ListGeo<LOG>::Pieces == 2 || q < 2) {
#pragma unroll
                for (int s = 0; s < 4; ++s) y[s][r] = a.v[s] + (q ? p - b.v[s] : b.v[s]);
            } else {   // omega psi^j = psi^(j + M)
                const MxQuad w = *(const MxQuad *)(tw_f + i), w1 = *(const MxQuad *)(tw_f + M + i);
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    y[s][r] = cm_mul_tw(a.v[s], w.v[s], p, cx.np) +
                              cm_mul_tw(b.v[s], w1.v[s], p, cx.np);
            }
        }
        if (q == 1) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const MxQuad w = *(const MxQuad *)(tw_f + i0 + Map::off(0, r));
#pragma unroll
                for (int s = 0; s < 4; ++s) y[s][r] = cm_mont_lazy(y[s][r], w.v[s], p, cx.np);
            }
        }
        mx_fence<V>();
    };
    operand(x[0], F + d.f, d.lf);
    operand(x[1], G + d.g, d.lg);
    MxMat m;
    u32 tw[V][4];
    mx_forward_begin<LOG, 0, V>(m, tw, cx);
    mx_tile_multiply<LOG, V>(x, lds, lds + mx_lds_words(M), cx, m, tw);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (q == 0) {
#pragma unroll
            for (int s = 0; s < 4; ++s) x[0][s][r] = mx_canon(x[0][s][r], cx);
        } else {
            const MxQuad w = *(const MxQuad *)(tw_i + i0 + Map::off(0, r));
#pragma unroll
            for (int s = 0; s < 4; ++s) x[0][s][r] = cm_mul_tw(x[0][s][r], w.v[s], p, cx.np);
        }
    }
}

// The chunks h[c] (h = sum_c h[c] x^(c W)) from its residues a[q] modulo
// x^W - omega_q, np = 2, 3 or 4 of them (h[3] = 0 for 3).
CM_DEV void big_recombine(u32 (&a)[4], int np, u32 w4, u32 w4i, const MxCtx &cx) {
    const u32 p = cx.p;
    auto half = [&](u32 v) { return (v + (v & 1 ? p : 0u)) >> 1; };
    const u32 s = half(cm_add(a[0], a[1], p)), d = half(cm_sub(a[0], a[1], p));
    if (np == 2) {          // h0 + h2 = s, h1 + h3 = d
        a[0] = s;
        a[1] = d;
        return;
    }
    u32 t, v;               // t = h0 - h2, v = h1 - h3
    if (np == 3) {
        v = d;
        t = cm_sub(a[2], cm_mul_tw(d, w4, p, cx.np), p);
    } else {
        t = half(cm_add(a[2], a[3], p));
        v = cm_mul_tw(half(cm_sub(a[2], a[3], p)), w4i, p, cx.np);
    }
    a[0] = half(cm_add(s, t, p));
    a[2] = half(cm_sub(s, t, p));
    a[1] = half(cm_add(d, v, p));
    a[3] = half(cm_sub(d, v, p));
}

// Pieces q0 .. q1 - 1 of one product.  With S, a piece goes there; else all but
// the last wait in the output (which has more than (q1 - 1) W words), each
// word where this lane put it, and the last recombines them.
CM_DEV void task_big(u32 *lds, const u32 *F, const u32 *G, u32 *H, const MulDesc *dp, int q0,
                     int q1, u32 *S, const u32 *lv, const u32 *lvi, const MxCtx &cx) {
    constexpr int LOG = 13, W = 1 << LOG;
    using Map = MxMap<LOG - 4, 4>;
    const MulDesc d = *dp;
    u32 x[2][4][4];
    u32 *h = H + d.h;
    const int i0 = Map::base();
    for (int q = q0;; ++q) {
        big_piece<LOG>(q, x, lds, F, G, d, lv, lvi, cx);
        if (q == q1 - 1 && !S) break;
        u32 *out = S ? S : h + q * W;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *(MxQuad *)(out + i0 + Map::off(0, r)) =
                MxQuad{{x[0][0][r], x[0][1][r], x[0][2][r], x[0][3][r]}};
        if (S) return;
        __syncthreads();    // the next piece writes LDS words that others still read
    }
    const u32 w4 = lv[2], w4i = lvi[2];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = i0 + Map::off(0, r);
        MxQuad c[3] = {};
#pragma unroll
        for (int q = 0; q < 3; ++q)
            if (q < q1 - 1) c[q] = *(const MxQuad *)(h + q * W + i);
        MxQuad o[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const u32 l = x[0][s][r];
            u32 a[4] = {c[0].v[s], q1 == 2 ? l : c[1].v[s], q1 == 3 ? l : c[2].v[s], l};
            big_recombine(a, q1, w4, w4i, cx);
#pragma unroll
            for (int q = 0; q < 4; ++q) o[q].v[s] = a[q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (q >= q1) break;
            const int k = q * W + i;
            if (k + 4 <= d.lh) {
                *(MxQuad *)(h + k) = o[q];
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    if (k + s < d.lh) h[k + s] = o[q].v[s];
            }
        }
    }
}

// Half Q of a 2^15-point product, modulo x^W - 1 or x^W + 1 (W = 2^14), to S.
template <int Q>
CM_DEV void task_half(u32 *lds, const u32 *F, const u32 *G, const MulDesc *dp, u32 *S,
                      const u32 *lv, const u32 *lvi, const MxCtx &cx) {
    using Map = MxMap<14 - 4, 4>;
    u32 x[2][4][4];
    big_piece<14>(Q, x, lds, F, G, *dp, lv, lvi, cx);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        *(MxQuad *)(S + Map::base() + Map::off(0, r)) =
            MxQuad{{x[0][0][r], x[0][1][r], x[0][2][r], x[0][3][r]}};
}

// A product of W < words <= 3/2 W (W = 2^13), with M = W / 2: A = H mod x^(2M) - 1 = (H0
// + H2) + H1 x^M, then B = H mod x^M - i = H0 + i H1 - H2 on M points, which
// leaves H2 = (A_lo + i A_hi - B) / 2.  A waits in the output.
CM_DEV void task_big_short(u32 *lds, const u32 *F, const u32 *G, u32 *H, const MulDesc *dp,
                           const u32 *lv, const u32 *lvi, const MxCtx &cx) {
    constexpr int LOG = 13, V = 2, L = LOG - 1, M = 1 << L;
    using Map = MxMap<L - 4, V>;
    const MulDesc d = *dp;
    const u32 p = cx.p;
    u32 *h = H + d.h;
    {
        using Map4 = MxMap<LOG - 4, 4>;
        u32 x[2][4][4];
        big_piece<LOG>(0, x, lds, F, G, d, lv, lvi, cx);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *(MxQuad *)(h + Map4::base() + Map4::off(0, r)) =
                MxQuad{{x[0][0][r], x[0][1][r], x[0][2][r], x[0][3][r]}};
    }
    __syncthreads();        // A is read by other lanes, and so is the LDS
    u32 x[2][V][4], tw[V][4];
    MxMat m;
    const int i0 = Map::base();
    const u32 *const wf = lv + 2 * M - 1, *const wi = lvi + 2 * M - 1;   // psi^j, psi = w_4M
    auto operand = [&](u32 (&y)[V][4], const u32 *q, int len) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int s = 0; s < V; ++s) {
                const int j = i0 + Map::off(s, r);
                const u32 a = j < len ? q[j] : 0u, b = M + j < len ? q[M + j] : 0u,
                          c = 2 * M + j < len ? q[2 * M + j] : 0u;
                y[s][r] = cm_mul_tw(cm_sub(a, c, p), wf[j], p, cx.np) +
                          cm_mul_tw(b, wf[M + j], p, cx.np);
            }
    };
    operand(x[0], F + d.f, d.lf);
    operand(x[1], G + d.g, d.lg);
    mx_forward_begin<L, 0, V>(m, tw, cx);
    mx_tile_multiply<L, V>(x, lds, lds + mx_lds_words(M), cx, m, tw);
    const u32 w4 = lv[2];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int s = 0; s < V; ++s) {
            const int j = i0 + Map::off(s, r);
            const u32 lo = h[j], hi = cm_mul_tw(h[M + j], w4, p, cx.np),
                      b = cm_mul_tw(x[0][s][r], wi[j], p, cx.np);
            const u32 e = cm_sub(cm_add(lo, hi, p), b, p), h2 = (e + (e & 1 ? p : 0u)) >> 1;
            h[j] = cm_sub(lo, h2, p);
            if (2 * M + j < d.lh) h[2 * M + j] = h2;
        }
}

// The pieces of the products descs[0 .. count) (slot j at S + j Pieces W) put
// together.
template <int LOG>
__global__ void k_big_combine(u32 *__restrict__ H, const MulDesc *__restrict__ descs,
                              const u32 *__restrict__ S, const u32 *__restrict__ lv,
                              const u32 *__restrict__ lvi, MxCtx cx) {
    const MulDesc d = descs[blockIdx.y];
    constexpr int W = ListGeo<LOG>::W, NP = ListGeo<LOG>::Pieces;
    const u32 *Sp = S + (int64_t)blockIdx.y * (NP * W);
    const int np = big_pieces<LOG>(d.lf + d.lg - 1);
    const u32 w4 = lv[2], w4i = lvi[2];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < W; i += gridDim.x * blockDim.x) {
        u32 a[4] = {};
#pragma unroll
        for (int q = 0; q < NP; ++q) a[q] = q < np ? Sp[q * W + i] : 0u;
        big_recombine(a, NP == 2 ? 2 : np, w4, w4i, cx);
#pragma unroll
        for (int q = 0; q < NP; ++q)
            if (q < np && q * W + i < d.lh) H[d.h + q * W + i] = a[q];
    }
}

// Outputs c0 .. c0 + PlainOut - 1 of the schoolbook product d: wave w computes the
// 256 outputs from c0 + 256 w on its own (its own LDS region, no workgroup
// barrier; a wave past the end of the product leaves at once), lane t four of
// them, with the arithmetic of k_plain_mul.  LDS operations of one wavefront
// complete in order, so a wave reads back what its lanes just stored.
constexpr int kPlainWaveWords = 256 + kPlainJT + 8 + kPlainJT;   // A window + B slice

CM_DEV void task_plain(u32 *lds, const u32 *F, const u32 *G, u32 *H, const MulDesc *dp, int c0,
                       PlainMod m) {
    const MulDesc d = *dp;
    const bool sw = d.logn != 0;
    const u32 *A = sw ? G + d.g : F + d.f;
    const u32 *B = sw ? F + d.f : G + d.g;
    const int la = sw ? d.lg : d.lf, lb = sw ? d.lf : d.lg;
    const int t = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int cw = c0 + 256 * wv;
    if (cw >= d.lh) return;
    u32 *sa = lds + wv * kPlainWaveWords, *sb = sa + 256 + kPlainJT + 8;
    // terms j of output c need 0 <= c - j < la and 0 <= j < lb
    int j_lo = cw - (la - 1);
    j_lo = j_lo < 0 ? 0 : j_lo & ~3;
    int j_hi = cw + 255;
    j_hi = j_hi < lb - 1 ? j_hi : lb - 1;
    u64 acc[4] = {0, 0, 0, 0};
    for (int js = j_lo; js <= j_hi; js += kPlainJT) {
        const int nj = (j_hi - js + 1 + 3) & ~3;
        const int jn = nj < kPlainJT ? nj : kPlainJT;
        const int je = js + jn;
        // sa[x] = A[cw - je + x] (zero outside [0, la)), x < 256 + jn;
        // sb[k] = B[js + k] (zero beyond lb)
        const int a_lo = cw - je;
        __builtin_amdgcn_wave_barrier();
        for (int x = t; x < 256 + jn; x += 64) {
            const int i = a_lo + x;
            sa[x] = (i >= 0 && i < la) ? A[i] : 0u;
        }
        for (int k = t; k < jn; k += 64) {
            const int j = js + k;
            sb[k] = j < lb ? B[j] : 0u;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const u32 *sw4 = sa + 4 * t;
        uint4 w = *(const uint4 *)(sw4 + jn);
        for (int k = 0; k < jn; k += 4) {
            const uint4 nw = *(const uint4 *)(sw4 + jn - k - 4);
            const uint4 bv = *(const uint4 *)(sb + k);
            const u32 x[8] = {nw.x, nw.y, nw.z, nw.w, w.x, w.y, w.z, w.w};
            const u32 b[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] += (u64)x[4 + r - s] * b[s];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = plain_fold(acc[r], m.c32);
            w = nw;
        }
    }
    u32 *Hc = H + d.h;
    const int c = cw + 4 * t;
    if (c + 4 <= d.lh) {
        uint4 o;
        o.x = plain_reduce(acc[0], m);
        o.y = plain_reduce(acc[1], m);
        o.z = plain_reduce(acc[2], m);
        o.w = plain_reduce(acc[3], m);
        if (((uintptr_t)(Hc + c) & 15) == 0) {
            *(uint4 *)(Hc + c) = o;
        } else {
            Hc[c] = o.x; Hc[c + 1] = o.y; Hc[c + 2] = o.z; Hc[c + 3] = o.w;
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (c + r < d.lh) Hc[c + r] = plain_reduce(acc[r], m);
    }
}

// One tile of products of 2^K points (W >> K of them).
template <int K, int LOG>
CM_DEV void task_tile(u32 *lds, const u32 *F, const u32 *G, u32 *H, const MulDesc *d, int cnt,
                      const MxCtx &cx) {
    constexpr int V = 4;
    using Map = MxMap<MxPlan<K>::words(0), V>;
    const int row0 = Map::base() >> K;
    auto desc = [&](int s) {
        const int c = row0 + (Map::off(s, 0) >> K);
        return c < cnt ? d[c] : MulDesc{};
    };
    MxMat m;
    u32 x[2][V][4], tw[V][4];
    mx_forward_begin<K, 0, V>(m, tw, cx);
    mx_load_rows<K, V>(x[0], [&](int s, const u32 *&q, int &len) {
        const MulDesc e = desc(s);
        q = F + e.f;
        len = e.lf;
    });
    mx_load_rows<K, V>(x[1], [&](int s, const u32 *&q, int &len) {
        const MulDesc e = desc(s);
        q = G + e.g;
        len = e.lg;
    });
    mx_tile_multiply<K, V>(x, lds, lds + mx_lds_words(ListGeo<LOG>::W), cx, m, tw);
    mx_store_rows<K, V>(
        x[0],
        [&](int s, u32 *&q, int &len) {
            const MulDesc e = desc(s);
            q = H + e.h;
            len = e.lh;
        },
        cx);
}

template <int LOG>
__global__ __launch_bounds__(ListGeo<LOG>::T)
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_list_persistent(
    const u32 *__restrict__ F, const u32 *__restrict__ G, u32 *__restrict__ H,
    const MulDesc *__restrict__ descs, const ListTask *__restrict__ tasks, int ntasks,
    int *__restrict__ counter, u32 *__restrict__ big_s, int big0, const u32 *__restrict__ lv,
    const u32 *__restrict__ lvi, MxCtx cx, PlainMod pm) {
    using Geo = ListGeo<LOG>;
    __shared__ __align__(16) u32 lds[2 * mx_lds_words(Geo::W)];
    __shared__ int s_next;
    static_assert(sizeof(lds) / 4 >= Geo::T / 64 * kPlainWaveWords, "schoolbook tasks");
    if (threadIdx.x == 0) s_next = atomicAdd(counter, 1);
    __syncthreads();
    // uniform: the task and its descriptor load through the scalar unit
    const int ti = __builtin_amdgcn_readfirstlane(s_next);
    if (ti >= ntasks) return;   // one workgroup per task: never taken
    const ListTask t = tasks[ti];
    const uint32_t kind = t.what & 3, sub = t.what >> 2 & 31;
    const int count = (int)(t.what >> 7);
    if (kind == kTaskPlain) {
        task_plain(lds, F, G, H, descs + t.first, count * Geo::PlainOut, pm);
    } else if (kind == kTaskBig) {
        const MulDesc *d = descs + t.first;
        u32 *S = big_s + ((int64_t)(t.first - big0) * Geo::Pieces + sub) * Geo::W;
        if constexpr (LOG == 14) {
            // the omega as a constant: as a variable it spills 47 registers
            if (sub == 0) task_half<0>(lds, F, G, d, S, lv, lvi, cx);
            else task_half<1>(lds, F, G, d, S, lv, lvi, cx);
        } else if (sub == kBigShort) {
            task_big_short(lds, F, G, H, d, lv, lvi, cx);
        } else {
            const bool all = sub == kBigAll;
            const int q = (int)sub;
            task_big(lds, F, G, H, d, all ? 0 : q, all ? count : q + 1, all ? nullptr : S, lv, lvi,
                     cx);
        }
    } else {
        const MulDesc *d = descs + t.first;
#define CM_PMIX(K)                                       \
    case K:                                              \
        if constexpr (K <= LOG)                          \
            task_tile<K, LOG>(lds, F, G, H, d, count, cx); \
        break;
        switch (sub) {
            CM_PMIX(4) CM_PMIX(5) CM_PMIX(6) CM_PMIX(7) CM_PMIX(8) CM_PMIX(9) CM_PMIX(10)
            CM_PMIX(11) CM_PMIX(12) CM_PMIX(13) CM_PMIX(14)
        default: break;
        }
#undef CM_PMIX
    }
}

namespace {

// pointwise constants of the 2^e-point products, e = 0 .. 15 (those of the
// last modulus are kept; callers hold the API lock)
Scales scale_table(const Family *fam) {
    static u32 last_p = 0;
    static Scales t;
    if (last_p != fam->p) {
        for (int e = 0; e < 16; ++e) t.v[e] = mul_scale(e, fam->p);
        last_p = fam->p;
    }
    return t;
}

}  // namespace

bool set_list_tile_words(int words) {
    for (int v = 0; v < kMixVariants; ++v)
        if (kMixWordsOf[v] == words) {
            g_mix_variant = v;
            return true;
        }
    return false;
}

int list_tile_words() { return kMixWordsOf[g_mix_variant]; }

// Products whose shorter operand has at most this many coefficients run on
// the schoolbook kernel (plain.hip) in list multiplies: there the la * lb
// products cost less than three transforms of 2^ceil(log2(la + lb - 1))
// points.  0 sends everything to the NTT.  The tuner sets it.  Measured on
// the 4096 uneven pairs: 32 in the one-launch form (0.204 ms per call with a wait
// after each few, 0.207 at 0, 0.229 at 64 and 0.274 at 256), 256 in the
// per-class form.
int g_plain_cutoff = 32;

bool set_list_plain_cutoff(int c) {
    if (c < 0 || c > 1024) return false;
    g_plain_cutoff = c;
    return true;
}

int list_plain_cutoff() { return g_plain_cutoff; }

// The strided multiplies of tree and evaluation levels (equal shapes) take
// the schoolbook kernel up to this shorter-operand length: the measured
// crossover of equal-length pairs (plain faster up to 256 coefficients).
int strided_plain_cutoff() { return 256; }

// smallest class of 2^14-point products that runs in LDS (one workgroup per
// CU at a time, so it needs a few per CU to pay)
constexpr int64_t kLds14MinCount = 512;

// mixed-size tiles of mv = 0, 1, 2 (2048, 4096, 8192 words)
template <class MD>
static hipError_t launch_mixed(int mv, dim3 g, const u32 *F, const u32 *G, u32 *H,
                               const MulDesc *d_descs, const TileDesc *d_tiles, const Family *fam,
                               MD md, const Scales &sc, hipStream_t s) {
    if (mv == 0)
        hipLaunchKernelGGL((k_mul_mixed<2048, 128, MD>), g, dim3(128), 0, s, F, G, H, d_descs,
                           d_tiles, fam->lv, fam->lvi, md, sc);
    else if (mv == 1)
        hipLaunchKernelGGL((k_mul_mixed<4096, 256, MD>), g, dim3(256), 0, s, F, G, H, d_descs,
                           d_tiles, fam->lv, fam->lvi, md, sc);
    else
        hipLaunchKernelGGL((k_mul_mixed<8192, 512, MD>), g, dim3(512), 0, s, F, G, H, d_descs,
                           d_tiles, fam->lv, fam->lvi, md, sc);
    return hipGetLastError();
}

static hipError_t launch_list_mul_ntt(const MulDesc *descs, int64_t count, const u32 *F,
                                      const u32 *G, u32 *H, const Family *fam, hipStream_t s);
static hipError_t launch_list_persistent(const MulDesc *descs, int64_t count, const u32 *F,
                                         const u32 *G, u32 *H, const Family *fam, hipStream_t s);

// 1: the persistent launch (default); 0: one launch per size class
int g_list_persistent = [] {
    const char *e = getenv("CUMODP_LIST_PERSISTENT");
    return (e && *e == '0') ? 0 : 1;
}();

bool set_list_persistent(int on) {
    if (on != 0 && on != 1) return false;
    g_list_persistent = on;
    return true;
}

int list_persistent() { return g_list_persistent; }

hipError_t launch_list_mul(const MulDesc *descs, int64_t count, const u32 *F, const u32 *G,
                           u32 *H, const Family *fam, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    if (g_list_persistent) return launch_list_persistent(descs, count, F, G, H, fam, s);
    if (g_plain_cutoff <= 0) return launch_list_mul_ntt(descs, count, F, G, H, fam, s);
    std::vector<MulDesc> plain, rest;
    for (int64_t i = 0; i < count; ++i) {
        const MulDesc &d = descs[i];
        if (std::min(d.lf, d.lg) <= g_plain_cutoff) {
            MulDesc q = d;
            q.logn = d.lg > d.lf ? 1 : 0;   // sweep the shorter operand
            plain.push_back(q);
        } else {
            rest.push_back(d);
        }
    }
    if (!plain.empty()) {
        hipError_t e = launch_plain_list(plain.data(), (int64_t)plain.size(), F, G, H, fam->p, s);
        if (e != hipSuccess) return e;
    }
    return launch_list_mul_ntt(rest.data(), (int64_t)rest.size(), F, G, H, fam, s);
}

static hipError_t run_four_step_classes(const MulDesc *sorted, int64_t count,
                                        const MulDesc *d_descs, const u32 *F, const u32 *G,
                                        u32 *H, const Family *fam, hipStream_t s);

static hipError_t launch_list_mul_ntt(const MulDesc *descs, int64_t count, const u32 *F,
                                      const u32 *G, u32 *H, const Family *fam, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    // order: small sizes (tiled), then 2^13, then four-step classes by size
    // (a stable counting sort on logn)
    std::vector<MulDesc> sorted((size_t)count);
    {
        int64_t pos[34] = {0};
        for (int64_t i = 0; i < count; ++i) ++pos[descs[i].logn + 1];
        for (int c = 1; c < 34; ++c) pos[c] += pos[c - 1];
        for (int64_t i = 0; i < count; ++i) sorted[(size_t)pos[descs[i].logn]++] = descs[i];
    }
    // The tuned tile suits large batches.  A batch whose small products fill
    // fewer than two tiles per CU gets smaller tiles (more workgroups), down
    // to 2048 words; tile sizes below the largest small product are skipped.
    int mv = g_mix_variant;
    {
        int64_t small_words = 0;
        int max_small = 0;
        for (int64_t q = 0; q < count && sorted[(size_t)q].logn <= 13; ++q) {
            small_words += (int64_t)1 << sorted[(size_t)q].logn;
            max_small = std::max(max_small, (int)sorted[(size_t)q].logn);
        }
        while (mv > 0 && small_words / kMixWordsOf[mv] < 2 * 256 &&
               (1 << max_small) <= kMixWordsOf[mv - 1])
            --mv;
    }
    const int mix_words = kMixWordsOf[mv];
    std::vector<TileDesc> tiles;
    int64_t i = 0;
    while (i < count && ((int64_t)1 << sorted[(size_t)i].logn) <= mix_words) {
        const int lg = sorted[(size_t)i].logn;
        const int per = mix_words >> lg;
        int64_t j = i;
        while (j < count && sorted[(size_t)j].logn == lg && j - i < per) ++j;
        tiles.push_back(TileDesc{(int32_t)i, (int32_t)(j - i), lg, 0});
        i = j;
    }
    const int64_t n_small_end = i;
    int64_t n13_end = n_small_end;   // end of the one-product-per-workgroup sizes
    while (n13_end < count && sorted[(size_t)n13_end].logn <= kMaxLdsLog) ++n13_end;
    // a class of 2^14-point products large enough to fill the chip runs one
    // product per 1024-thread workgroup too (F and G tiles take 128 KiB of
    // LDS): no gather/scatter slabs and one launch instead of three
    {
        int64_t e14 = n13_end;
        while (e14 < count && sorted[(size_t)e14].logn == kMaxLdsLog + 1) ++e14;
        if (e14 - n13_end >= kLds14MinCount) n13_end = e14;
    }

    const size_t desc_bytes = sizeof(MulDesc) * (size_t)count;
    const size_t tile_bytes = sizeof(TileDesc) * tiles.size();
    std::vector<char> blob(desc_bytes + tile_bytes);
    memcpy(blob.data(), sorted.data(), desc_bytes);
    if (tile_bytes) memcpy(blob.data() + desc_bytes, tiles.data(), tile_bytes);
    char *dblob = (char *)workspace(7, blob.size(), s);
    if (!dblob) return hipErrorOutOfMemory;
    hipError_t e = stage_upload(blob.data(), blob.size(), dblob, s);
    if (e != hipSuccess) return e;
    const MulDesc *d_descs = (const MulDesc *)dblob;
    const TileDesc *d_tiles = (const TileDesc *)(dblob + desc_bytes);

    if (!tiles.empty()) {
        ProfScope ps(kProfMulMixed, s);
        const Scales sc = scale_table(fam);
        const dim3 g((unsigned)tiles.size());
        // values in [0, 2p) between butterflies when p < 2^30
        if (fam->p < (1u << 30))
            e = launch_mixed(mv, g, F, G, H, d_descs, d_tiles, fam, ModLazy{fam->p, fam->np}, sc, s);
        else
            e = launch_mixed(mv, g, F, G, H, d_descs, d_tiles, fam, Mod{fam->p, fam->np}, sc, s);
        if (e != hipSuccess) return e;
    }
    for (int64_t a = n_small_end; a < n13_end;) {
        const int lg = sorted[(size_t)a].logn;
        int64_t b = a;
        while (b < n13_end && sorted[(size_t)b].logn == lg) ++b;
        e = launch_mul_lds(lg, F, G, H, d_descs + a, (int)(b - a), fam, s);
        if (e != hipSuccess) return e;
        a = b;
    }
    return run_four_step_classes(sorted.data() + n13_end, count - n13_end, d_descs + n13_end, F,
                                 G, H, fam, s);
}

// The products sorted[0 .. count) (ascending logn, every logn > 13; their
// descriptors also at d_descs[0 .. count)) through batched four-step
// multiplies: per size, operands gathered into zero-padded slabs and products
// scattered back.
static hipError_t run_four_step_classes(const MulDesc *sorted, int64_t count,
                                        const MulDesc *d_descs, const u32 *F, const u32 *G,
                                        u32 *H, const Family *fam, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int64_t a = 0; a < count;) {
        const int lg = sorted[(size_t)a].logn;
        int64_t b = a;
        while (b < count && sorted[(size_t)b].logn == lg) ++b;
        const int64_t n = (int64_t)1 << lg;
        // process the class in chunks that keep the slabs within 1 GiB each
        const int64_t chunk = std::max<int64_t>(1, ((int64_t)1 << 28) / n);
        for (int64_t c0 = a; c0 < b; c0 += chunk) {
            const int cnt = (int)std::min<int64_t>(chunk, b - c0);
            u32 *sf = (u32 *)workspace(5, sizeof(u32) * (size_t)(n * cnt), s);
            u32 *sg = (u32 *)workspace(6, sizeof(u32) * (size_t)(n * cnt), s);
            if (!sf || !sg) return hipErrorOutOfMemory;
            // the slabs hold only the longest operand of each side (the
            // column pass zero-pads the rest, and skips the zero upper half
            // when both fit in n/2); the inverse pass stores the longest output
            int64_t mf = 1, mg = 1, mh = 1;
            for (int64_t q = c0; q < c0 + cnt; ++q) {
                mf = std::max<int64_t>(mf, sorted[(size_t)q].lf);
                mg = std::max<int64_t>(mg, sorted[(size_t)q].lg);
                mh = std::max<int64_t>(mh, sorted[(size_t)q].lh);
            }
            const unsigned gx = (unsigned)std::min<int64_t>(n / 1024, 64);
            {
            ProfScope ps(kProfGatherScatter, s);
            hipLaunchKernelGGL(k_gather, dim3(gx, cnt), dim3(1024), 0, s, sf, n, mf, F,
                               d_descs + c0, 0);
            hipLaunchKernelGGL(k_gather, dim3(gx, cnt), dim3(1024), 0, s, sg, n, mg, G,
                               d_descs + c0, 1);
            }
            e = hipGetLastError();
            FourStepIO io{sf, sg, mf, mg, n, sf, sg, sf, mh, n, cnt};
            if (e == hipSuccess) e = launch_mul_four_step(lg, io, fam, s);
            if (e != hipSuccess) return e;
            {
            ProfScope ps(kProfGatherScatter, s);
            hipLaunchKernelGGL(k_scatter, dim3(gx, cnt), dim3(1024), 0, s, H, sf, n,
                               d_descs + c0);
            }
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        a = b;
    }
    return hipSuccess;
}

// CUs of the current device.
static int device_cus() {
    static int cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cached[dev]) {
        int c = 0;
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            c <= 0)
            c = 256;
        cached[dev] = c;
    }
    return cached[dev];
}

// floor(log2(x)) of a cost, 0 .. 63: the exponent field of the double
// (a library ilogb call per task cost a few microseconds per list call)
static int cost_bucket(double x) {
    if (!(x >= 1.0)) return 0;
    uint64_t u;
    memcpy(&u, &x, sizeof u);
    const int b = (int)((u >> 52) & 0x7ff) - 1023;
    return b > 63 ? 63 : b;
}

// What the products of a list call are, in one pass over them: a pass of its own
// for each figure mispredicts its branches again (20000 pairs of degrees 16 .. 300:
// 227 us per call with three such passes, 156 us so).
struct ListCount {
    int64_t cls[33] = {0};   // products by class: 0 schoolbook, e 2^e points
    int64_t plain = 0;       // small tasks of the schoolbook products
    int64_t pieces = 0;      // small tasks of the 2^15-point products
    int cut;                 // class 0: a side of at most cut words

    bool is_plain(const MulDesc &d) const { return std::min(d.lf, d.lg) <= cut; }
    static int64_t tasks(const MulDesc &d, int words) {
        return (uint32_t)(d.lh + words - 1) / (uint32_t)words;
    }
    ListCount(const MulDesc *descs, int64_t count) : cut(g_plain_cutoff) {
        int64_t pl = 0, pc = 0;
        for (int64_t i = 0; i < count; ++i) {
            const MulDesc &d = descs[i];
            if (is_plain(d)) {
                ++cls[0];
                pl += tasks(d, ListGeo<13>::PlainOut);
            } else {
                ++cls[d.logn];
                pc += tasks(d, ListGeo<13>::W) & -(int64_t)(d.logn == kBigLog);
            }
        }
        plain = pl;
        pieces = pc;
    }
};

// tiles of 2^log words that the classes 2^4 .. 2^log fill
static int64_t list_tiles(const int64_t (&ncls)[33], int log) {
    int64_t n = 0;
    for (int e = 4; e <= log; ++e) n += (ncls[e] + (1 << (log - e)) - 1) >> (log - e);
    return n;
}

// Tasks of 2^13 words with 512 threads, two to a CU, or of 2^14 words with 1024,
// one to a CU.  A 2^14-point product is two pieces of the small tasks (each reads
// the operands, and a pass recombines them) and one large task, so the large
// ones win where they fill the chip once and the small ones would fill it
// more than half (150 products of 2^14 points: 32 us as large tasks, 44 as
// small ones, 35 as radix-2 butterflies of 1024 threads), and where 2^14-point
// products hold half the words and the small tasks either run in pieces or
// have whole products of 2^15 points, four pieces long, at the end (400
// products of 2^14 points: 71 us and 84; 700 with 116 of 2^15 and as many words
// of 2^13 and 2^11: 174 and 196).  The other lists take small tasks (4096 pairs
// of degrees 32 .. 16384: 187 us).  Measured over 220 mixes of sizes.  Schoolbook
// products alone take large tasks, which are fewer (16 products of 20 by 50000
// coefficients: 13.0 us, 15.0 as small ones); many of up to 3/2 small tasks, which
// leave most waves of a large one idle, keep their list to small tasks (the kernel
// of 20000 pairs of degrees 16 .. 300: 119 us, 138 with large ones).
static int list_log(const ListCount &n) {
    const int64_t (&ncls)[33] = n.cls, pieces = n.pieces;
    const int64_t tiles = list_tiles(ncls, 13), n14 = ncls[14], n15 = ncls[15];
    const int64_t large = list_tiles(ncls, 14) + 2 * n15;
    const bool shorts = 2 * n.plain < 3 * ncls[0];
    if (large == 0) return shorts ? 13 : 14;
    const int64_t cus = device_cus();
    if (shorts && n.plain > cus) return 13;
    if (large <= cus) return tiles + 2 * n14 + pieces > cus ? 14 : 13;
    const bool half = 2 * n14 >= tiles + 4 * n15;
    return half && large <= 8 * cus && (tiles + n14 + n15 < 4 * cus || n15 > 0) ? 14 : 13;
}

template <int LOG>
static hipError_t list_persistent_t(const MulDesc *descs, int64_t count, const ListCount &nl,
                                    const u32 *F, const u32 *G, u32 *H, const Family *fam,
                                    hipStream_t s) {
    using Geo = ListGeo<LOG>;
    const int64_t (&ncls)[33] = nl.cls;
    int64_t off[34];
    off[0] = 0;
    for (int c = 0; c < 33; ++c) off[c + 1] = off[c] + ncls[c];
    int64_t nbig = 0, ntasks = list_tiles(ncls, LOG);
    for (int e = LOG + 1; e <= kBigLog; ++e) nbig += ncls[e];
    ntasks += nbig + (LOG == 13 ? nl.plain : 0);
    for (int64_t i = 0; LOG == 14 && ncls[0] && i < count; ++i)
        if (nl.is_plain(descs[i])) ntasks += nl.tasks(descs[i], Geo::PlainOut);
    // Small tasks: below four per CU (two rounds of workgroups), or with products of
    // 2^15 points below 3 1/2 rounds of pieces, a whole product would leave the
    // chip waiting at the end, so every piece is a task, at the price of a
    // recombining pass over scratch (whose allocation a capture does without).
    // 40 pairs of degrees 32 .. 16384: 26 us, 56 with whole products; 42 products
    // of 2^15 points, 256 of 2^14 and as many words of sizes below: 107 us and 135.
    // Large tasks always take a 2^15-point product as two.
    auto split = [&] {
        if (LOG == 14 || stream_capturing(s)) return LOG == 14;
        const int64_t cus = device_cus();
        return ntasks < 4 * cus ||
               (ncls[kBigLog] > 0 &&
                list_tiles(ncls, 13) + 2 * ncls[14] + nl.pieces < 7 * cus);
    };
    u32 *big_s = nullptr;
    if (nbig > 0 && split()) {
        big_s = (u32 *)workspace(20, sizeof(u32) * (size_t)(nbig * Geo::Pieces * Geo::W), s);
        if (!big_s) (void)hipGetLastError();   // whole products need no scratch
    }
    if (LOG == 14 && nbig > 0 && !big_s)
        return list_persistent_t<13>(descs, count, nl, F, G, H, fam, s);
    if (big_s) ntasks += (LOG == 13 ? 2 * ncls[14] + nl.pieces : 2 * nbig) - nbig;
    if (ntasks > INT32_MAX) return hipErrorInvalidValue;

    // blob: the task counter (16 bytes), the sorted descriptors, the tasks;
    // written straight into the pinned staging buffer
    const size_t desc_off = 16;
    const size_t task_off = desc_off + sizeof(MulDesc) * (size_t)count;
    // whole 16-byte words, or the copy takes about 1 us longer
    const size_t bytes = (task_off + sizeof(ListTask) * (size_t)ntasks + 15) & ~(size_t)15;
    std::vector<MulDesc> tail;   // host copy of the four-step classes' descriptors
    char *dblob = (char *)workspace(7, bytes, s);
    if (!dblob) return hipErrorOutOfMemory;
    hipError_t e = stage_upload_fill(bytes, dblob, s, [&](char *blob) {
        memset(blob, 0, desc_off);   // the task counter starts at 0
        MulDesc *sorted = (MulDesc *)(blob + desc_off);
        ListTask *tasks = (ListTask *)(blob + task_off);
        int64_t pos[33];
        for (int c = 0; c < 33; ++c) pos[c] = off[c];
        for (int64_t i = 0; i < count; ++i) {
            MulDesc q = descs[i];
            if (nl.is_plain(q)) {
                q.logn = q.lg > q.lf ? 1 : 0;   // sweep the shorter operand
                sorted[pos[0]++] = q;
            } else {
                sorted[pos[q.logn]++] = q;
            }
        }
        // the tasks with their costs (butterflies; a schoolbook term costs
        // about an eighth of one), ordered by descending power-of-two cost
        // bucket: one pass counts the buckets, the second places the tasks
        auto each_task = [&](auto &&emit) {
            for (int64_t i = off[0]; i < off[1]; ++i) {
                const MulDesc &d = sorted[i];
                const int lb = std::min(d.lf, d.lg);
                for (int c0 = 0; c0 < d.lh; c0 += Geo::PlainOut) {
                    const int outs = std::min(Geo::PlainOut, d.lh - c0);
                    emit(list_task(kTaskPlain, i, 0, c0 / Geo::PlainOut), (double)outs * lb / 8.0);
                }
            }
            for (int e2 = 4; e2 <= LOG; ++e2) {
                const int per = Geo::W >> e2;
                for (int64_t i = off[e2]; i < off[e2 + 1]; i += per) {
                    const int cnt = (int)std::min<int64_t>(per, off[e2 + 1] - i);
                    emit(list_task(kTaskTile, i, (uint32_t)e2, cnt),
                         3.0 * e2 * (double)cnt * (1 << (e2 - 1)));
                }
            }
            for (int64_t i = off[LOG + 1]; i < off[kBigLog + 1]; ++i) {
                const int np = big_pieces<LOG>(sorted[i].lf + sorted[i].lg - 1);
                const double piece = 3.0 * LOG * (1 << (LOG - 1));
                if (!big_s) {
                    const bool sh = sorted[i].lf + sorted[i].lg - 1 <= Geo::W / 2 * 3;
                    emit(list_task(kTaskBig, i, sh ? kBigShort : kBigAll, np),
                         (sh ? 1.5 : np) * piece);
                }
                for (int q = 0; big_s && q < np; ++q)
                    emit(list_task(kTaskBig, i, (uint32_t)q, 0), piece);
            }
        };
        int64_t nb[64] = {0};
        each_task([&](const ListTask &, double c) { ++nb[cost_bucket(c)]; });
        int64_t at[64];
        int64_t acc = 0;
        for (int b = 63; b >= 0; --b) {
            at[b] = acc;
            acc += nb[b];
        }
        each_task([&](const ListTask &t, double c) { tasks[at[cost_bucket(c)]++] = t; });
        tail.assign(sorted + off[kBigLog + 1], sorted + count);
    });
    if (e != hipSuccess) return e;
    int *d_counter = (int *)dblob;
    const MulDesc *d_descs = (const MulDesc *)(dblob + desc_off);
    const ListTask *d_tasks = (const ListTask *)(dblob + task_off);
    if (ntasks > 0) {
        ProfScope ps(kProfListPersistent, s);
        const dim3 grid((unsigned)ntasks);
        hipLaunchKernelGGL(k_list_persistent<LOG>, grid, dim3(Geo::T), 0, s, F, G, H, d_descs,
                           d_tasks, (int)ntasks, d_counter, big_s, (int)off[LOG + 1], fam->lv,
                           fam->lvi, mx_ctx(fam), plain_mod(fam->p));
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (big_s) {
        ProfScope ps(kProfListPersistent, s);
        hipLaunchKernelGGL(k_big_combine<LOG>, dim3(Geo::W / 1024, (unsigned)nbig), dim3(1024), 0, s,
                           H, d_descs + off[LOG + 1], big_s, fam->lv, fam->lvi, mx_ctx(fam));
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    // 2^16 points and more: batched four-step multiplies
    return run_four_step_classes(tail.data(), (int64_t)tail.size(), d_descs + off[kBigLog + 1], F,
                                 G, H, fam, s);
}

static hipError_t launch_list_persistent(const MulDesc *descs, int64_t count, const u32 *F,
                                         const u32 *G, u32 *H, const Family *fam, hipStream_t s) {
    if (count > INT32_MAX / 4) return hipErrorInvalidValue;
    // descriptor order: the schoolbook products, then the transform sizes
    // ascending
    const ListCount n(descs, count);
    const auto run = list_log(n) == 14 ? list_persistent_t<14> : list_persistent_t<13>;
    return run(descs, count, n, F, G, H, fam, s);
}

}  // namespace cm
