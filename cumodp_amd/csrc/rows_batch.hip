// rows_batch.hip -- cyclic products of many rows of several lengths and moduli
// in a few launches.
//
// The integer multiply needs, for each class of products and each CRT prime,
// the products of many contiguous rows.  One launch sequence per class and
// prime leaves the chip idle (a class of a serving batch has one to six
// products) and costs several microseconds per launch.  Here the rows of every
// class and prime form segments of one list:
//   * rows up to 2^12 words: one launch, 4096 words of one segment per
//     workgroup, the size selected at run time; rows of 2^13: one launch;
//   * 2^14 .. 2^20: the four-step passes (mul_mx.h), one launch per column
//     length and direction and one per row length, grid.y over all rows of
//     those segments;
//   * longer rows (and splits that the tuner forced): segment by segment.
// The rows of 96 integer requests (32 classes) take 11 launches and 0.25 ms.
// Up to three segments of one length (a single product) travel as kernel
// arguments, more as a table in device memory.
#include <algorithm>
#include <vector>

#include "internal.h"
#include "mul_mx.h"

namespace cm {

namespace {

struct MxSeg {
    u32 *f, *g;         // row j at + j 2^e
    int first;          // number of its first row in the list
    int e, flen, glen;  // words that may be nonzero in a row of f, of g
    MxOuter o;
    MxCtx cx;
};

// Segments as kernel arguments: s[i] has `per` rows and `tiles` tiles.
struct SegVal {
    MxSeg s[3];
    int per, tiles, span;   // span: rows per tile
    CM_DEV const MxSeg &array(int a, int &row) const {
        row = a % per;
        return s[a / per];
    }
    CM_DEV const MxSeg &tile(int b, int &row, int &cnt) const {
        row = (b % tiles) * span;
        cnt = per - row;
        return s[b / tiles];
    }
};

// Segments as tables: the segment of each row, and of each tile with its
// first row and row count.
struct TileRef {
    int seg, row, cnt, pad;
};
struct SegTab {
    const MxSeg *s;
    const int *arr;
    const TileRef *tiles;
    CM_DEV const MxSeg &array(int a, int &row) const {
        const MxSeg &S = s[__builtin_amdgcn_readfirstlane(arr[a])];
        row = a - S.first;
        return S;
    }
    CM_DEV const MxSeg &tile(int b, int &row, int &cnt) const {
        row = tiles[b].row;
        cnt = tiles[b].cnt;
        return s[__builtin_amdgcn_readfirstlane(tiles[b].seg)];
    }
};

// rows of 2^K words, one tile of 2^LOGW words
template <int K, int LOGW, int V>
CM_DEV void rows_tile(u32 *lds, const MxSeg &S, int row, int cnt) {
    using Map = MxMap<MxPlan<K>::words(0), V>;
    const int row0 = Map::base() >> K;
    u32 *f = S.f + ((int64_t)row << K), *g = S.g + ((int64_t)row << K);
    const MxCtx cx = S.cx;
    MxMat m;
    u32 x[2][V][4], tw[V][4];
    mx_forward_begin<K, 0, V>(m, tw, cx);
    auto at = [&](int s, u32 *base, int len, u32 *&q, int &n) {
        const int c = row0 + (Map::off(s, 0) >> K);
        q = base + ((int64_t)c << K);
        n = c < cnt ? len : 0;
    };
    auto from = [&](u32 *base, int len) {
        return [=](int s, const u32 *&q, int &n) {
            u32 *p;
            at(s, base, len, p, n);
            q = p;
        };
    };
    mx_load_rows<K, V>(x[0], from(f, S.flen));
    mx_load_rows<K, V>(x[1], from(g, S.glen));
    mx_tile_multiply<K, V>(x, lds, lds + mx_lds_words(1 << LOGW), cx, m, tw);
    mx_store_rows<K, V>(x[0], [&](int s, u32 *&q, int &n) { at(s, f, 1 << K, q, n); }, cx);
}

template <class SRC, int LOGW, int V>
__global__ __launch_bounds__((1 << LOGW) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_rows_lds(SRC src) {
    __shared__ __align__(16) u32 lds[2 * mx_lds_words(1 << LOGW)];
    int row, cnt;
    const MxSeg &S = src.tile(blockIdx.x, row, cnt);
    if constexpr (LOGW == 13) {
        rows_tile<13, 13, V>(lds, S, row, cnt);
    } else {
        switch (S.e) {
#define CM_CASE(K) case K: rows_tile<K, LOGW, V>(lds, S, row, cnt); break;
            CM_CASE(4) CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8) CM_CASE(9) CM_CASE(10)
            CM_CASE(11) CM_CASE(12)
#undef CM_CASE
        }
    }
}

// Column passes in place; grid.x: tiles of the longest row, grid.y: rows of
// the list from a0, grid.z (forward): operand.
template <class SRC, int LOGL, int LOGC, int V>
__global__ __launch_bounds__((1 << (LOGL + LOGC)) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_rows_col_fwd(SRC src, int a0) {
    __shared__ __align__(16) u32 lds[mx_col_lds<LOGL, LOGC>()];
    int row;
    const MxSeg &S = src.array(a0 + blockIdx.y, row);
    const int logn2 = S.e - LOGL, tiles = 1 << (logn2 - LOGC);
    if ((int)blockIdx.x >= tiles) return;
    const int c0 = mx_xcd(blockIdx.x, tiles) << LOGC;
    u32 *X = (blockIdx.z ? S.g : S.f) + ((int64_t)row << S.e) + c0;
    const MxCtx cx = S.cx;
    mx_col_fwd<LOGL, LOGC, V>(lds, X, (blockIdx.z ? S.glen : S.flen) - c0, X, logn2, cx);
}

template <class SRC, int LOGL, int LOGC, int V>
__global__ __launch_bounds__((1 << (LOGL + LOGC)) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_rows_col_inv(SRC src, int a0) {
    __shared__ __align__(16) u32 lds[mx_col_lds<LOGL, LOGC>()];
    int row;
    const MxSeg &S = src.array(a0 + blockIdx.y, row);
    const int logn2 = S.e - LOGL, tiles = 1 << (logn2 - LOGC);
    if ((int)blockIdx.x >= tiles) return;
    const int c0 = mx_xcd(blockIdx.x, tiles) << LOGC;
    u32 *X = S.f + ((int64_t)row << S.e) + c0;
    const MxCtx cx = S.cx;
    mx_col_inv<LOGL, LOGC, V, false>(lds, X, X, 0, (1 << S.e) - c0, 0, false, logn2, cx);
}

template <class SRC, int LOGL, int V>
__global__ __launch_bounds__((1 << mx_row_logw<LOGL, V>()) / (4 * V))
__attribute__((amdgpu_waves_per_eu(4, 8))) void k_rows_row(SRC src, int a0) {
    constexpr int LOGW = mx_row_logw<LOGL, V>();
    __shared__ __align__(16) u32 lds[2 * mx_lds_words(1 << LOGW)];
    int row;
    const MxSeg &S = src.array(a0 + blockIdx.y, row);
    if ((int)blockIdx.x >= 1 << (S.e - LOGW)) return;
    const int64_t t0 = ((int64_t)row << S.e) + ((int64_t)blockIdx.x << LOGW);
    const MxCtx cx = S.cx;
    const MxOuter o = S.o;
    mx_row<LOGL, V>(lds, S.f + t0, S.g + t0, (int)(blockIdx.x << (LOGW - LOGL)), S.e - LOGL, o,
                    cx);
}

template <class SRC, int LOGL, int LOGC, int V>
hipError_t col_t(bool inverse, const SRC &src, int a0, int cnt, int e, hipStream_t s) {
    constexpr int T = (1 << (LOGL + LOGC)) / (4 * V);
    const unsigned tiles = 1u << (e - LOGL - LOGC);
    ProfScope ps(inverse ? kProfColInv : kProfColFwd, s);
    for (int at = 0; at < cnt; at += 65535) {
        const unsigned y = std::min(cnt - at, 65535);
        if (inverse)
            hipLaunchKernelGGL((k_rows_col_inv<SRC, LOGL, LOGC, V>), dim3(tiles, y), dim3(T), 0, s,
                               src, a0 + at);
        else
            hipLaunchKernelGGL((k_rows_col_fwd<SRC, LOGL, LOGC, V>), dim3(tiles, y, 2), dim3(T), 0,
                               s, src, a0 + at);
    }
    return hipGetLastError();
}

template <class SRC>
hipError_t cols(bool inverse, const SRC &src, int k1, bool small, int a0, int cnt, int e,
                hipStream_t s) {
    switch (k1) {
    case 6: return small ? col_t<SRC, 6, 3, 1>(inverse, src, a0, cnt, e, s)
                         : col_t<SRC, 6, 4, 4>(inverse, src, a0, cnt, e, s);
    case 7: return small ? col_t<SRC, 7, 4, 1>(inverse, src, a0, cnt, e, s)
                         : col_t<SRC, 7, 4, 4>(inverse, src, a0, cnt, e, s);
    case 8: return small ? col_t<SRC, 8, 3, 1>(inverse, src, a0, cnt, e, s)
                         : col_t<SRC, 8, 4, 4>(inverse, src, a0, cnt, e, s);
    }
    return hipErrorInvalidValue;
}

template <class SRC, int LOGL, int V>
hipError_t row_t(const SRC &src, int a0, int cnt, int e, hipStream_t s) {
    constexpr int LOGW = mx_row_logw<LOGL, V>();
    ProfScope ps(kProfRowMul, s);
    for (int at = 0; at < cnt; at += 65535)
        hipLaunchKernelGGL((k_rows_row<SRC, LOGL, V>),
                           dim3(1u << (e - LOGW), std::min(cnt - at, 65535)),
                           dim3((1 << LOGW) / (4 * V)), 0, s, src, a0 + at);
    return hipGetLastError();
}

template <class SRC>
hipError_t rows(const SRC &src, int k2, bool small, int a0, int cnt, int e, hipStream_t s) {
    switch (k2) {
#define CM_CASE(K)                                                       \
    case K:                                                              \
        return small ? row_t<SRC, K, 1>(src, a0, cnt, e, s)              \
                     : row_t<SRC, K, 4>(src, a0, cnt, e, s);
        CM_CASE(8) CM_CASE(9) CM_CASE(10) CM_CASE(11) CM_CASE(12)
#undef CM_CASE
    }
    return hipErrorInvalidValue;
}

constexpr int kBatchMaxLog = 20;

bool batched(const RowSeg &r, const Outer *o) {
    return r.e <= kBatchMaxLog && o->k1 >= 6 && o->k1 <= 8 && o->k2 >= 8 && o->k2 <= 12;
}

// the launches of the four-step segments segs[i0 .. i1) (e ascending)
template <class SRC>
hipError_t four_step(const SRC &src, const std::vector<RowSeg> &segs,
                     const std::vector<const Outer *> &outer, const std::vector<int> &first,
                     size_t i0, size_t i1, bool small, hipStream_t s) {
    hipError_t err = hipSuccess;
    // runs of equal column (row) length are contiguous: k1 and k2 do not
    // decrease both ways, so equal neighbours are grouped
    auto each = [&](auto &&key, auto &&run) {
        for (size_t i = i0; i < i1 && err == hipSuccess;) {
            size_t j = i;
            while (j < i1 && key(j) == key(i)) ++j;
            const int a0 = first[i], a1 = first[j - 1] + segs[j - 1].rows;
            err = run(key(i), a0, a1 - a0, segs[j - 1].e);
            i = j;
        }
    };
    auto k1 = [&](size_t i) { return outer[i]->k1; };
    auto k2 = [&](size_t i) { return outer[i]->k2; };
    each(k1, [&](int k, int a0, int n, int e) { return cols(false, src, k, small, a0, n, e, s); });
    each(k2, [&](int k, int a0, int n, int e) { return rows(src, k, small, a0, n, e, s); });
    each(k1, [&](int k, int a0, int n, int e) { return cols(true, src, k, small, a0, n, e, s); });
    return err;
}

// Latency-bound lists spread over four times the threads, as in mul_mx.hip.
constexpr int64_t kRowsSmallWords = (int64_t)1 << 20;

template <class SRC>
hipError_t lds_rows(const SRC &src, bool e13, bool small, unsigned tiles, hipStream_t s) {
    ProfScope ps(kProfMulLds, s);
    if (e13 && small)
        hipLaunchKernelGGL((k_rows_lds<SRC, 13, 2>), dim3(tiles), dim3(1024), 0, s, src);
    else if (e13)
        hipLaunchKernelGGL((k_rows_lds<SRC, 13, 4>), dim3(tiles), dim3(512), 0, s, src);
    else if (small)
        hipLaunchKernelGGL((k_rows_lds<SRC, 12, 1>), dim3(tiles), dim3(1024), 0, s, src);
    else
        hipLaunchKernelGGL((k_rows_lds<SRC, 12, 4>), dim3(tiles), dim3(256), 0, s, src);
    return hipGetLastError();
}

int tile_rows(int e) { return e == 13 ? 1 : 1 << (12 - e); }

}  // namespace

hipError_t launch_rows_batch(std::vector<RowSeg> segs, hipStream_t s) {
    if (segs.empty()) return hipSuccess;
    std::stable_sort(segs.begin(), segs.end(),
                     [](const RowSeg &a, const RowSeg &b) { return a.e < b.e; });
    const size_t n = segs.size();
    std::vector<const Outer *> outer(n, nullptr);
    std::vector<int> first(n);
    std::vector<MxSeg> dev(n);
    int64_t total = 0, words = 0;
    size_t nbatch = 0;      // leading segments that the list covers
    for (size_t i = 0; i < n; ++i) {
        const RowSeg &r = segs[i];
        if (r.e > kMaxLdsLog) {
            outer[i] = outer_for(r.fam, r.e);
            if (!outer[i]) return hipErrorOutOfMemory;
        }
        if (nbatch < i || (r.e > kMaxLdsLog && !batched(r, outer[i]))) continue;
        nbatch = i + 1;
        first[i] = (int)total;
        total += r.rows;
        words += (int64_t)r.rows << r.e;
        if (total > INT32_MAX / 2) return hipErrorInvalidValue;
        dev[i] = MxSeg{r.f, r.g, first[i], r.e, r.flen, r.glen,
                       outer[i] ? mx_outer_of(outer[i]) : MxOuter{}, mx_ctx(r.fam)};
    }
    const bool small = words <= kRowsSmallWords;
    hipError_t e = hipSuccess;
    bool uniform = nbatch >= 1 && nbatch <= 3;
    for (size_t i = 1; i < nbatch; ++i)
        uniform = uniform && segs[i].e == segs[0].e && segs[i].rows == segs[0].rows;
    if (uniform) {
        SegVal v{};
        for (size_t i = 0; i < nbatch; ++i) v.s[i] = dev[i];
        v.per = segs[0].rows;
        if (segs[0].e <= kMaxLdsLog) {
            v.span = tile_rows(segs[0].e);
            v.tiles = (v.per + v.span - 1) / v.span;
            e = lds_rows(v, segs[0].e == 13, small, (unsigned)(v.tiles * (int)nbatch), s);
        } else {
            e = four_step(v, segs, outer, first, 0, nbatch, small, s);
        }
    } else if (nbatch) {
        // one blob: segments, the segment of each row, the tiles
        std::vector<int> arr((size_t)total);
        std::vector<TileRef> tiles;
        size_t n12 = 0, n13 = 0, i4 = nbatch;   // tiles of each kind, first four-step segment
        for (size_t i = 0; i < nbatch; ++i) {
            const RowSeg &r = segs[i];
            std::fill(arr.begin() + first[i], arr.begin() + first[i] + r.rows, (int)i);
            if (r.e > kMaxLdsLog) {
                i4 = std::min(i4, i);
                continue;
            }
            const int span = tile_rows(r.e);
            for (int row = 0; row < r.rows; row += span) {
                tiles.push_back(TileRef{(int)i, row, std::min(span, r.rows - row), 0});
                ++(r.e == 13 ? n13 : n12);
            }
        }
        const size_t b0 = sizeof(MxSeg) * nbatch, b1 = sizeof(TileRef) * tiles.size(),
                     b2 = sizeof(int) * arr.size();
        char *d = (char *)workspace(21, b0 + b1 + b2, s);
        if (!d) return hipErrorOutOfMemory;
        e = stage_upload_fill(b0 + b1 + b2, d, s, [&](char *h) {
            std::copy_n((const char *)dev.data(), b0, h);
            std::copy_n((const char *)tiles.data(), b1, h + b0);
            std::copy_n((const char *)arr.data(), b2, h + b0 + b1);
        });
        if (e != hipSuccess) return e;
        SegTab t{(const MxSeg *)d, (const int *)(d + b0 + b1), (const TileRef *)(d + b0)};
        // the four-step rows first: they are the larger part
        if (i4 < nbatch) e = four_step(t, segs, outer, first, i4, nbatch, small, s);
        if (e == hipSuccess && n13) {
            SegTab u = t;
            u.tiles += n12;
            e = lds_rows(u, true, small, (unsigned)n13, s);
        }
        if (e == hipSuccess && n12) e = lds_rows(t, false, small, (unsigned)n12, s);
    }
    for (size_t i = nbatch; i < n && e == hipSuccess; ++i) {
        const RowSeg &r = segs[i];
        const int64_t len = (int64_t)1 << r.e;
        FourStepIO io{r.f, r.g, r.flen, r.glen, len, r.f, r.g, r.f, len, len, r.rows};
        e = launch_mul_four_step_with(io, r.fam, outer[i], s);
    }
    return e;
}

}  // namespace cm
