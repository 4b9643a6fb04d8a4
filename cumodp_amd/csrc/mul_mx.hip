// mul_mx.hip -- whole multiplies in one workgroup on the matrix cores.
#include <algorithm>

#include "internal.h"
#include "ntt_mx.h"

namespace cm {

// A single product is bound by its serial chain (load, rounds, exchanges), many
// products by vector issue.  One 2048-point product mod 469762049, back to
// back: 5.6 us per call with one set per lane (512 threads), 8.1 us with the
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
    u32 x[2][V][4];
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
    mx_tile_multiply<LOGL, V>(x, lds, lds + LW, cx);
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

static MxCtx ctx_of(const Family *fam) {
    return MxCtx{(const mx_v4i *)fam->mx_mat, fam->mx_tf, fam->mx_ti, fam->p, fam->np,
                 cm_host_r1(fam->p), 1u << 16};
}

template <int LOGL, int V, bool DESC>
static hipError_t mul_mx_v(const u32 *F, const u32 *G, u32 *H, const MulDesc *descs, int ndesc,
                           const MulDesc &one, const Family *fam, hipStream_t s) {
    constexpr int LOGW = std::max(LOGL, 8 + mx_log2(V));
    constexpr int C = 1 << (LOGW - LOGL);
    ProfScope ps(kProfMulLds, s);
    hipLaunchKernelGGL((k_mul_mx<LOGL, LOGW, V, DESC>), dim3((ndesc + C - 1) / C),
                       dim3((1 << LOGW) / (4 * V)), 0, s, F, G, H, descs, ndesc, one, ctx_of(fam));
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

}  // namespace cm
