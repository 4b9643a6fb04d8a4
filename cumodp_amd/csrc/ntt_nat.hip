// ntt_nat.hip -- stand-alone natural-order transforms on the matrix cores.
//
// Y_j = sum_i X_i w^(ij) in place for rows of 2^k words.  The rounds are those
// of ntt_mx.h up to the last one, which takes its vectors in the order of the
// frequencies they hold: lanes then hold consecutive outputs for every value of
// the last digit, and rows are stored in natural order straight from the
// registers, with no bit-reversal pass.  The inverse transform is the same with
// the matrices and twiddles of the inverse root; its matrices carry 1/radix,
// so it comes out scaled by 2^-k.
//
// Up to 2^13 words one workgroup transforms whole rows.  Longer ones take two
// launches: column transforms X -> Y, then tiles of rows with consecutive
// frequencies, transformed and stored transposed into X (rows of 2^k2 words
// whose position-r row holds frequency f give X[f + 2^k1 j]); no copy back.
#include <algorithm>

#include "internal.h"
#include "mul_mx.h"

namespace cm {

// Rounds J .. NR-2 of a row tile and the exchange into the last round, whose
// words are left in x: set s of lane (n, g) holds elements 4g .. 4g+3 of vector
// id = 16 V wave + V n + s.  ROWS: id = u 2^LOGR + row, else row L/16 + u,
// where u numbers a row's vectors by the frequencies below the last digit.
template <int LOGL, int LOGW, int V, bool ROWS, int J>
CM_DEV void nat_rounds(u32 (&x)[V][4], u32 *lds, const MxCtx &cx, MxMat &m) {
    using P = MxPlan<LOGL, 0, 1>;
    static_assert(P::NR >= 2, "one round needs no exchange");
    u32 tw[V][4];
    mx_load_tw<P::logs(J), 0, V>(tw, cx.tf);
    mx_dft<V>(x, m, cx);
    mx_mul<V>(x, tw, cx);
    MxMap<P::logs(J), V>::store(lds, x);
    if constexpr (J + 1 < P::NR - 1) {
        mx_sync<P::logs(J), V>();
        MxMap<P::logs(J + 1), V>::load(lds, x);
        nat_rounds<LOGL, LOGW, V, ROWS, J + 1>(x, lds, cx, m);
    } else {
        if constexpr (P::T != 0) m = mx_load_mat(cx, kMxFwd + P::T);
        __syncthreads();
        constexpr int LQ = 4 * (P::NF - 1), LU = LOGL - 4, LOGR = LOGW - LOGL;
        const int n = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
        const int id0 = (int)(threadIdx.x >> 6) * (16 * V) + V * n;
#pragma unroll
        for (int s = 0; s < V; ++s) {
            const int id = id0 + s;
            const int u = ROWS ? id >> LOGR : id & ((1 << LU) - 1);
            const int row = ROWS ? id & ((1 << LOGR) - 1) : id >> LU;
            // digits of u from the lowest: the digit below the top of the
            // position first; what is left (c) numbers the 16-word groups
            int at = (row << LOGL) + ((u >> LQ) << 4) + 4 * g;
#pragma unroll
            for (int i = 0; i < P::NF - 1; ++i) at += ((u >> (4 * i)) & 15) << (LOGL - 4 * (i + 1));
            const uint4 v = *(const uint4 *)(lds + mx_phys_d(at));
            x[s][0] = v.x; x[s][1] = v.y; x[s][2] = v.z; x[s][3] = v.w;
        }
    }
}

// Output index of element e16 of vector u after the last round.
template <int LOGL>
CM_DEV int nat_index(int u, int e16) {
    using P = MxPlan<LOGL, 0, 1>;
    constexpr int LQ = 4 * (P::NF - 1);
    if constexpr (P::T == 0) {
        return u + (e16 << LQ);
    } else {
        const int low = u & ((1 << LQ) - 1), c = u >> LQ;
        return low + ((((c << (4 - P::T)) + (e16 >> P::T)) + ((e16 & ((1 << P::T) - 1)) << 4)) << LQ);
    }
}

// Rows of 2^LOGL words, 2^(LOGW-LOGL) per workgroup, in place.
//
// Many rows are bound by memory.  A lane's words lie 2^(LOGL-4) words apart, and
// so do its outputs: pieces of 4 to 16 bytes for rows up to 2^7 words (STAGE),
// whose tile, one wave's 256 V words, therefore goes through LDS in both
// directions and through memory in quads of consecutive lanes.  2^25 words as
// rows of 2^4, 2^5, 2^6 and 2^7: 44.5, 47.6, 47.7 and 47.6 us; straight from and to the
// registers 92, 127, 101 and 100 us.
template <int LOGL, int LOGW, int V>
__global__ __launch_bounds__((1 << LOGW) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_ntt_mx(u32 *__restrict__ X, int64_t m, MxCtx cx) {
    static_assert(LOGW >= LOGL && (1 << LOGW) >= 256 * V, "tile");
    using P = MxPlan<LOGL, 0, 1>;
    using Map = MxMap<P::logs(0), V>;
    constexpr int LU = LOGL - 4;
    __shared__ __align__(16) u32 lds[P::NR > 1 ? mx_lds_words(1 << LOGW) : 4];
    const int64_t r0 = (int64_t)blockIdx.x << (LOGW - LOGL);
    const int row0 = Map::base() >> LOGL;
    MxMat mat = mx_load_mat(cx, kMxFwd + (P::NF == 0 ? P::T : 0));
    u32 x[V][4];
    constexpr bool STAGE = LOGL <= 7 && V == 4;
    using Flat = MxMap<0, V>;       // quads in the order of the lanes
    if constexpr (STAGE) {
        static_assert((1 << LOGW) == 256 * V, "a tile is one wave's words");
#pragma unroll
        for (int s = 0; s < V; ++s) {
            const int i = Flat::base() + Flat::off(s, 0);
            MxQuad v{};
            if (r0 + (i >> LOGL) < m) v = *(const MxQuad *)(X + (r0 << LOGL) + i);
#pragma unroll
            for (int r = 0; r < 4; ++r) x[s][r] = v.v[r];
        }
        if constexpr (P::NR > 1) {
            Flat::store(lds, x);
            mx_sync<0, V>();
            Map::load(lds, x);
        }
    } else {
        mx_load_rows<LOGL, V>(x, [&](int s, const u32 *&q, int &len) {
            const int64_t row = r0 + row0 + (Map::off(s, 0) >> LOGL);
            q = X + (row << LOGL);
            len = row < m ? 1 << LOGL : 0;
        });
    }
    if constexpr (STAGE) {
        if constexpr (P::NR > 1) nat_rounds<LOGL, LOGW, V, false, 0>(x, lds, cx, mat);
        mx_dft<V>(x, mat, cx);
        if constexpr (P::NR > 1) {
            const int n = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
            mx_sync<0, V>();
#pragma unroll
            for (int s = 0; s < V; ++s)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int id = V * n + s;
                    lds[mx_phys_d(((id >> LU) << LOGL) +
                                  nat_index<LOGL>(id & ((1 << LU) - 1), 4 * g + r))] = x[s][r];
                }
            mx_sync<0, V>();
            Flat::load(lds, x);
        }
#pragma unroll
        for (int s = 0; s < V; ++s) {
            const int i = Flat::base() + Flat::off(s, 0);
            if (r0 + (i >> LOGL) < m)
                *(MxQuad *)(X + (r0 << LOGL) + i) =
                    MxQuad{{mx_canon(x[s][0], cx), mx_canon(x[s][1], cx), mx_canon(x[s][2], cx),
                            mx_canon(x[s][3], cx)}};
        }
    } else if constexpr (P::NR == 1) {
        mx_dft<V>(x, mat, cx);
        mx_store_rows<LOGL, V>(
            x,
            [&](int s, u32 *&q, int &len) {
                const int64_t row = r0 + row0 + (Map::off(s, 0) >> LOGL);
                q = X + (row << LOGL);
                len = row < m ? 1 << LOGL : 0;
            },
            cx);
    } else {
        nat_rounds<LOGL, LOGW, V, false, 0>(x, lds, cx, mat);
        mx_dft<V>(x, mat, cx);
        const int n = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
        const int id0 = (int)(threadIdx.x >> 6) * (16 * V) + V * n;
        if constexpr (V == 4 && P::NF >= 2) {
            // four consecutive outputs per digit value
            const int64_t row = r0 + (id0 >> LU);
            if (row < m) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    *(MxQuad *)(X + (row << LOGL) +
                                nat_index<LOGL>(id0 & ((1 << LU) - 1), 4 * g + r)) =
                        MxQuad{{mx_canon(x[0][r], cx), mx_canon(x[1][r], cx),
                                mx_canon(x[2][r], cx), mx_canon(x[3][r], cx)}};
            }
        } else {
#pragma unroll
            for (int s = 0; s < V; ++s) {
                const int64_t row = r0 + ((id0 + s) >> LU);
                if (row < m) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        X[(row << LOGL) + nat_index<LOGL>((id0 + s) & ((1 << LU) - 1), 4 * g + r)] =
                            mx_canon(x[s][r], cx);
                }
            }
        }
    }
}

// 2^LOGR rows of consecutive frequencies f0 .. of an array after its column
// pass (Y, rows of 2^LOGL words, grid.y arrays 2^(k1+LOGL) words apart): outer
// twiddles, row transforms, X[f + 2^k1 j].
template <int LOGL, int LOGR, int V>
__global__ __launch_bounds__((1 << (LOGL + LOGR)) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_row_nat(const u32 *__restrict__ Y0,
                                                          u32 *__restrict__ X0, int k1, MxOuter o,
                                                          MxCtx cx) {
    constexpr int LOGW = LOGL + LOGR;
    static_assert((1 << LOGW) >= 256 * V && LOGL >= 8, "tile");
    using P = MxPlan<LOGL, 0, 1>;
    using Map = MxMap<P::logs(0), V>;
    __shared__ __align__(16) u32 lds[mx_lds_words(1 << LOGW)];
    const int64_t array = (int64_t)blockIdx.y << (k1 + LOGL);
    const int f0 = mx_xcd(blockIdx.x, gridDim.x) << LOGR;
    const int b = Map::base(), f = f0 + (b >> LOGL);
    const u32 *q = Y0 + array + ((int64_t)mx_pos(f, k1) << LOGL) + (b & ((1 << LOGL) - 1));
    MxMat mat = mx_load_mat(cx, kMxFwd);
    u32 x[V][4], ow[V][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if constexpr (V == 4) {
            const uint4 u = *(const uint4 *)(q + Map::off(0, r));
            x[0][r] = u.x; x[1][r] = u.y; x[2][r] = u.z; x[3][r] = u.w;
        } else {
#pragma unroll
            for (int s = 0; s < V; ++s) x[s][r] = q[Map::off(s, r)];
        }
    }
    mx_outer<LOGL, V>(ow, o.rb_f, o.rc_f, f, cx);
    mx_mul<V>(x, ow, cx);
    nat_rounds<LOGL, LOGW, V, true, 0>(x, lds, cx, mat);
    mx_dft<V>(x, mat, cx);
    const int n = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
    const int id0 = (int)(threadIdx.x >> 6) * (16 * V) + V * n;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if constexpr (V == 4 && LOGR >= 2) {
            u32 *w = X0 + array + f0 + (id0 & ((1 << LOGR) - 1)) +
                     ((int64_t)nat_index<LOGL>(id0 >> LOGR, 4 * g + r) << k1);
            *(MxQuad *)w = MxQuad{{mx_canon(x[0][r], cx), mx_canon(x[1][r], cx),
                                   mx_canon(x[2][r], cx), mx_canon(x[3][r], cx)}};
        } else {
#pragma unroll
            for (int s = 0; s < V; ++s)
                X0[array + f0 + ((id0 + s) & ((1 << LOGR) - 1)) +
                   ((int64_t)nat_index<LOGL>((id0 + s) >> LOGR, 4 * g + r) << k1)] =
                    mx_canon(x[s][r], cx);
        }
    }
}

// The tables of a direction: the inverse transform is the forward one with the
// inverse root's matrices (times 1/radix) and twiddles.
static MxCtx nat_ctx(const Family *fam, bool inverse) {
    MxCtx cx = mx_ctx(fam);
    if (inverse) {
        cx.mat += kMxInv * kMxMatWords;
        cx.tf = cx.ti;
    }
    return cx;
}

template <int LOGL, int V>
static hipError_t ntt_rows_v(u32 *X, int64_t m, const MxCtx &cx, hipStream_t s) {
    constexpr int LOGW = std::max(LOGL, 8 + mx_log2(V)), C = 1 << (LOGW - LOGL);
    ProfScope ps(kProfNttLds, s);
    hipLaunchKernelGGL((k_ntt_mx<LOGL, LOGW, V>), dim3((unsigned)((m + C - 1) / C)),
                       dim3((1 << LOGW) / (4 * V)), 0, s, X, m, cx);
    return hipGetLastError();
}

// Few words: one set per lane (latency); more: four (fewer table loads).
constexpr int64_t kNatSmallWords = (int64_t)1 << 19;

template <int LOGL>
static hipError_t ntt_rows_t(u32 *X, int64_t m, const MxCtx &cx, hipStream_t s) {
    if ((m << LOGL) < kNatSmallWords) return ntt_rows_v<LOGL, LOGL == 13 ? 2 : 1>(X, m, cx, s);
    return ntt_rows_v<LOGL, 4>(X, m, cx, s);
}

hipError_t launch_ntt_lds(int k, u32 *X, int64_t m, bool inverse, const Family *fam,
                          hipStream_t s) {
    if (m <= 0) return hipSuccess;
    const MxCtx cx = nat_ctx(fam, inverse);
    switch (k) {
#define CM_CASE(K) case K: return ntt_rows_t<K>(X, m, cx, s);
        CM_CASE(4) CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8) CM_CASE(9) CM_CASE(10)
        CM_CASE(11) CM_CASE(12) CM_CASE(13)
#undef CM_CASE
    }
    return hipErrorInvalidValue;
}

template <int LOGL, int LOGR, int V>
static hipError_t row_nat_t(const u32 *Y, u32 *X, int cnt, int k1, const MxOuter &o,
                            const MxCtx &cx, hipStream_t s) {
    ProfScope ps(kProfRowOut, s);
    hipLaunchKernelGGL((k_row_nat<LOGL, LOGR, V>), dim3(1u << (k1 - LOGR), cnt),
                       dim3((1 << (LOGL + LOGR)) / (4 * V)), 0, s, Y, X, k1, o, cx);
    return hipGetLastError();
}

// Split of a stand-alone transform: rows and columns about equal, so that both
// the column tiles' rows and the row tiles' transposed stores are segments of
// 16 to 64 bytes.
static void ntt_split(int k, int &k1, int &k2) {
    k2 = k <= 16 ? 8 : (k <= 20 ? 10 : (k <= 22 ? 11 : (k <= 24 ? 12 : k - 12)));
    k1 = k - k2;
}

hipError_t launch_ntt_four_step(int k, u32 *X, u32 *Y, int cnt, bool inverse, const Family *fam,
                                hipStream_t s) {
    if (k <= kMaxLdsLog || k > kMaxLog || k > fam->K) return hipErrorInvalidValue;
    // both passes take their arrays in grid.y
    for (; cnt > 65535; cnt -= 65535, X += (int64_t)65535 << k, Y += (int64_t)65535 << k) {
        const hipError_t e = launch_ntt_four_step(k, X, Y, 65535, inverse, fam, s);
        if (e != hipSuccess) return e;
    }
    int k1, k2;
    ntt_split(k, k1, k2);
    const Outer *o = outer_for_split(fam, k, k1, k2);
    if (!o) return hipErrorOutOfMemory;
    const MxCtx cx = nat_ctx(fam, inverse);
    MxOuter t = mx_outer_of(o);
    if (inverse) {
        t.rb_f = t.rb_i;
        t.rc_f = t.rc_i;
    }
    const int64_t n = (int64_t)1 << k;
    hipError_t e = launch_cols_out(k1, X, Y, n, cnt, k2, cx, s);
    if (e != hipSuccess) return e;
    const bool small = n * cnt <= ((int64_t)1 << 20);
    switch (k2) {
    case 8: return small ? row_nat_t<8, 3, 1>(Y, X, cnt, k1, t, cx, s)
                         : row_nat_t<8, 4, 4>(Y, X, cnt, k1, t, cx, s);
    case 10: return small ? row_nat_t<10, 2, 1>(Y, X, cnt, k1, t, cx, s)
                          : row_nat_t<10, 4, 4>(Y, X, cnt, k1, t, cx, s);
    case 11: return row_nat_t<11, 3, 4>(Y, X, cnt, k1, t, cx, s);
    case 12: return row_nat_t<12, 2, 4>(Y, X, cnt, k1, t, cx, s);
    case 13: return row_nat_t<13, 1, 4>(Y, X, cnt, k1, t, cx, s);
    case 14: return row_nat_t<14, 0, 4>(Y, X, cnt, k1, t, cx, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace cm
